// Weight gradients of the norms and bias gradients of the gates that wait for one launch while a step driver's backward runs
// (omx_defer_weight_sums); forgotten where it ends early.
#pragma once
#include <cstdint>

#include "ojas_mi355x.h"

struct WaitingSums {
  omx_ctx* ctx;
  bool formed = false;
  WaitingSums(omx_ctx* c, uint32_t count) : ctx(c) { (void)omx_defer_weight_sums(ctx, count); }
  ~WaitingSums() {
    if (!formed) (void)omx_form_weight_sums(ctx, 0);
  }
  WaitingSums(const WaitingSums&) = delete;
  WaitingSums& operator=(const WaitingSums&) = delete;
  int32_t form() {
    formed = true;
    return omx_form_weight_sums(ctx, 1);
  }
};
