// What the reversible MLP's translation units share.
#pragma once

#include "nf_common.h"

namespace nf {

inline int rev_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
    if (cus <= 0) cus = 256;
  }
  return cus;
}

// The backward of all couplings (reversible_bwd.hip) on checked arguments.  workspace of rev_bwd_bytes(): the gradients are written in
// `type`; NULL: they are float32 accumulators and added to with atomics.
struct RevBwdCall {
  const uint16_t *y, *dy;
  uint16_t *dx, *x_rec;
  int64_t y_stride, dy_stride, dx_stride, x_stride, rows;
  const uint16_t *w1, *b1, *w2, *b2;
  void *dw1, *db1, *dw2, *db2;  // db1, db2 may be NULL
  int half, blocks, act, type;
  void* workspace;
};
size_t rev_bwd_bytes(int64_t rows, int half, int blocks);
int rev_bwd(const RevBwdCall& c, int dtype, hipStream_t s);

}  // namespace nf
