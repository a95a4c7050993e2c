// Declarations shared by the fused-MLP translation units.
#pragma once

#include "mlp_tile.h"

namespace nf {

struct MlpArgs {
  const uint16_t* x;
  int64_t x_stride;
  uint16_t* y;
  int64_t y_stride;
  const uint16_t* dy;
  int64_t dy_stride;
  uint16_t* dx;
  int64_t dx_stride;
  const uint16_t *w_in, *b_in, *w_hid, *b_hid, *w_out, *b_out;
  float *dw_in, *db_in, *dw_hid, *db_hid, *dw_out, *db_out;
  int64_t rows;
  int d_in, d_hidden, d_out, depth, act;
  int x_vec, y_vec, dy_vec, dx_vec;
  int waves;  // waves per workgroup
  int in_act; // activation applied to x as it is loaded (x holds pre-activations of a layer in front); dx = d/dx of that
  int x_conv; // 0: x / dx stored like the weights; 1: stored as float16 (weights bfloat16); 2: stored as bfloat16 (weights float16)
  // eight-wave backward only: non-NULL = every workgroup stores its sums into partials + blockIdx.x * partial_stride
  // ([dw_in | dw_hid | dw_out | db_in | db_hid | db_out], float32) instead of adding them to dw_* / db_*
  float* partials;
  int64_t partial_stride;
  // whole-network backward only: bit l set = the pre-activations that linear layer l gives are rounded to 16 bit, as where
  // nf_mlp_bwd hands them from one launch to the next
  uint32_t handover;
};

constexpr int FRAG_ELEMS = 64 * 8;  // 16-bit elements per fragment (1 KiB)
constexpr int TPITCH = 40;          // 16-bit elements per feature row of a transposed 32-row panel (80 B)

// Fragment of 8 values stored in the other 16-bit type -> the compute type (what a cast kernel in front would do).
__device__ __forceinline__ Frag convert_frag(Frag f, int x_conv) {
  if (x_conv == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f.w[i] = pack2<BF16>(unpack_lo<F16>(f.w[i]), unpack_hi<F16>(f.w[i]));
  } else if (x_conv == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f.w[i] = pack2<F16>(unpack_lo<BF16>(f.w[i]), unpack_hi<BF16>(f.w[i]));
  }
  return f;
}

template <typename T>
__device__ __forceinline__ void stage_bias(float* dst, const uint16_t* b, int n_valid, int n_pad, int tid, int nthreads) {
  for (int i = tid; i < n_pad; i += nthreads) dst[i] = (b != nullptr && i < n_valid) ? T::to_f32(b[i]) : 0.0f;
}

// All weights of a network into LDS as A fragments, [w_in | w_hid | w_out], and its biases behind them.  The layers are one list of
// fragments, several to a wave under way together, and the biases are asked for first: layer by layer, every matrix and every bias waited for the
// one in front.  Rows move in 16-byte pieces, which are the order of the first layer's products and two halves of a fragment each in
// that of the others (8-byte pieces keep the L1 busy twice as long, a clock per lane).  Loads carry no condition of their own
// (addresses are held inside their matrix, what is outside is zeroed on its way to LDS), as a branch would be waited for at its end, and what a
// fragment is, is worked out once per wave.  Two layers alone have little to wait for (32 -> 64 -> 16, 2^18 rows 6.9 us, as a list 7.6).  IN_CHAIN: the first layer's products are in chain order, too.
// first_rows asks for the wave's first rows, behind the first weights: loads come back in order, and rows from HBM in front of the weights held up the
// barrier (one-hidden-layer ReLU networks over inputs that no cache holds, rows first / weights first: 32 -> 64 -> 64 -> 16, 2^20 rows 23.9 / 19.4 us,
// 64 -> 64 -> 64 -> 64, 2^18 14.6 / 13.8; eight hidden layers, 2^18 rows 35.3 / 34.5).
// PIECE: bytes that w_hid and w_out lie on.  16, or 8 (views into a flat buffer): the same list in two pieces of 8 bytes each; a first or, of 8 bytes, a last matrix
// off those is staged by itself behind the list.  0 (w_hid off 8 bytes, no hidden matrix): layer by layer.  Matrices 8 bytes off, us, layer by layer / as a list: 64 x 10 ReLU
// 1000 rows 17.1 / 8.7, 2^18 42.6 / 36.6; 32 -> 64 x 3 -> 16 SiLU 1000 7.7 / 5.2, 2^16 9.9 / 8.1; 32 -> 64 -> 64 -> 16 2^18 8.6 / 7.6.  The two lists are
// chosen between in front of this function: as a choice inside it the loops' wave-uniform branches became masks (32 -> 64 -> 64 -> 16, 2^18 rows 9.2 -> 10.3).
// NTHREADS: as for stage_weight_frags().
template <typename T, int KIN, int HP, int OUTP, int PIECE, bool IN_CHAIN, int NTHREADS = 0, typename FirstRows>
__device__ __forceinline__ void stage_network(uint16_t* frags, float* bias, const MlpArgs& a, int tid, int nthreads, FirstRows first_rows) {
  constexpr int KC_IN = KIN / 32, KC_H = HP / 32, MT_H = HP / 16, MT_O = OUTP / 16, AT_ONCE = NTHREADS > 0 ? 4 : 6;
  constexpr int F_IN = MT_H * KC_IN, F_HID = MT_H * KC_H, F_OUT = MT_O * KC_H;
  const int H = a.d_hidden, n_hid = a.depth - 1, hidden = n_hid * F_HID;
  if constexpr (PIECE == 0) {
    first_rows();
    stage_weight_frags<IN_CHAIN, false, NTHREADS>(frags, a.w_in, H, a.d_in, MT_H, KC_IN, tid, nthreads);
    for (int k = 0; k < n_hid; ++k) {
      stage_weight_frags<true, false, NTHREADS>(frags + (size_t)(F_IN + k * F_HID) * FRAG_ELEMS, a.w_hid + (size_t)k * H * H, H, H, MT_H, KC_H, tid, nthreads);
      stage_bias<T>(bias + (k + 1) * HP, a.b_hid ? a.b_hid + (size_t)k * H : nullptr, H, HP, tid, nthreads);
    }
    stage_weight_frags<true, false, NTHREADS>(frags + (size_t)(F_IN + hidden) * FRAG_ELEMS, a.w_out, a.d_out, H, MT_O, KC_H, tid, nthreads);
    stage_bias<T>(bias, a.b_in, H, HP, tid, nthreads);
    stage_bias<T>(bias + (n_hid + 1) * HP, a.b_out, a.d_out, OUTP, tid, nthreads);
    return;
  }
  const int n_bias = HP + n_hid * HP + OUTP;
  const auto bias_at = [&](int i, bool& valid) {
    const bool out = i >= HP + n_hid * HP;
    const int layer = i / HP, f = out ? i - (HP + n_hid * HP) : i % HP;
    const uint16_t* b = out ? a.b_out : layer == 0 ? a.b_in : a.b_hid;
    valid = b != nullptr && f < (out ? a.d_out : H);
    return valid ? b + (out || layer == 0 ? f : (layer - 1) * H + f) : a.w_out;
  };
  bool first_valid;
  const uint16_t first_bias = *bias_at(tid < n_bias ? tid : 0, first_valid);
  const bool in_listed = a.d_in % 8 == 0 && (uintptr_t)a.w_in % (PIECE == 16 ? 16 : 8) == 0, out_listed = PIECE == 16 || (uintptr_t)a.w_out % 8 == 0;
  const int lane = tid & 63, m = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = nthreads >> 6;
  const int all = F_IN + hidden + (out_listed ? F_OUT : 0);
  for (int f0 = (in_listed ? 0 : F_IN) + wave, round = 0; f0 < all || round == 0; f0 += AT_ONCE * nwaves, ++round) {
    uint4 v[AT_ONCE];
    bool there[AT_ONCE];
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      const int f = f0 + i * nwaves;
      if (f >= all) break;  // (the same for the whole wave)
      const bool in = f < F_IN, out = f >= F_IN + hidden;
      const uint32_t p = (uint32_t)(in ? f : out ? f - F_IN - hidden : f - F_IN), layer = in || out ? 0u : p / F_HID, frag = p - layer * F_HID;
      const int mt = (int)(in ? frag / KC_IN : frag / KC_H), kc = (int)(in ? frag % KC_IN : frag % KC_H);
      const int rows = out ? a.d_out : H, cols = in ? a.d_in : H, row = 16 * mt + m, k = 32 * kc + 8 * g;
      const uint16_t* w = in ? a.w_in : out ? a.w_out : a.w_hid + (size_t)layer * H * H;
      there[i] = row < rows && k < cols;
      w += __umul24((uint32_t)(row < rows ? row : 0), (uint32_t)cols) + (k < cols ? k : 0);
      if constexpr (PIECE == 16) {
        v[i] = *reinterpret_cast<const uint4*>(w);
      } else {
        const uint2 lo = *reinterpret_cast<const uint2*>(w), hi = *reinterpret_cast<const uint2*>(w + 4);
        v[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
    }
    if (round == 0) first_rows();
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      const int f = f0 + i * nwaves;
      if (f >= all) break;
      uint16_t* dst = frags + (size_t)f * FRAG_ELEMS;
      if (!there[i]) v[i] = make_uint4(0u, 0u, 0u, 0u);
      if (!IN_CHAIN && f < F_IN) {
        *reinterpret_cast<uint4*>(dst + lane * 8) = v[i];
      } else {
        put_chain(dst, m, g, v[i]);
      }
    }
  }
  if (!in_listed) stage_weight_frags<IN_CHAIN, false, NTHREADS>(frags, a.w_in, H, a.d_in, MT_H, KC_IN, tid, nthreads);
  if (!out_listed) stage_weight_frags<true, false, NTHREADS>(frags + (size_t)(F_IN + hidden) * FRAG_ELEMS, a.w_out, a.d_out, H, MT_O, KC_H, tid, nthreads);
  if (tid < n_bias) bias[tid] = first_valid ? T::to_f32(first_bias) : 0.0f;
  for (int i = tid + nthreads; i < n_bias; i += nthreads) {
    bool valid;
    const uint16_t b = *bias_at(i, valid);
    bias[i] = valid ? T::to_f32(b) : 0.0f;
  }
}

// acc[nt][mt] = bias + W(frags) * in[nt][kc]; K chunks outermost, so that the products into one accumulator tile are
// NT * MT instructions apart
template <typename T, int MT, int KC, int NT>
__device__ __forceinline__ void layer_mma(f32x4_t (&acc)[NT][4], const Frag (&in)[NT][2], const uint16_t* frags,
                                          const float* bias, int lane) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const f32x4_t b4 = *reinterpret_cast<const f32x4_t*>(bias + 16 * mt + 4 * (lane >> 4));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = b4;
  }
#pragma unroll
  for (int kc = 0; kc < KC; ++kc)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const Frag a = lds_frag(frags, mt * KC + kc, lane);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = mfma16<T>(a, in[nt][kc], acc[nt][mt]);
    }
}

// Park an accumulator-layout tile (lane (n,g): features 16*mt + 4*g + r of row 16*nt + n) into a
// transposed panel panel[feature][row].
__device__ __forceinline__ void park_tile_T(uint16_t* panel, int mt, int nt, int lane, uint32_t p01, uint32_t p23) {
  const int n = (lane & 15) + 16 * nt;
  const int f = 16 * mt + 4 * (lane >> 4);
  panel[(f + 0) * TPITCH + n] = (uint16_t)(p01 & 0xffffu);
  panel[(f + 1) * TPITCH + n] = (uint16_t)(p01 >> 16);
  panel[(f + 2) * TPITCH + n] = (uint16_t)(p23 & 0xffffu);
  panel[(f + 3) * TPITCH + n] = (uint16_t)(p23 >> 16);
}
// Park a natural-order fragment (lane (n,g): features 32*kc + 8*g + j of row 16*nt + n).
__device__ __forceinline__ void park_frag_T(uint16_t* panel, int kc, int nt, int lane, const Frag& f) {
  const int n = (lane & 15) + 16 * nt;
  const int c = 32 * kc + 8 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    panel[(c + 2 * j) * TPITCH + n] = (uint16_t)(f.w[j] & 0xffffu);
    panel[(c + 2 * j + 1) * TPITCH + n] = (uint16_t)(f.w[j] >> 16);
  }
}
// Operand of a K = 32-rows product: lane (i, g) reads rows 8*g .. 8*g+7 of feature 16*t + i.
__device__ __forceinline__ Frag panel_frag(const uint16_t* panel, int t, int lane) {
  Frag f;
  f.u = *reinterpret_cast<const uint4*>(panel + (16 * t + (lane & 15)) * TPITCH + 8 * (lane >> 4));
  return f;
}

// dW tile (mt over output features, nt over input features): lane (n, g) reg r is
// dW[16*mt + 4*g + r][16*nt + n].
// store: plain stores (the tile belongs to this workgroup alone) instead of atomic adds.
__device__ __forceinline__ void flush_dw_tile(float* dw, int out_dim, int in_dim, int mt, int nt, int lane, f32x4_t v,
                                              bool store = false) {
  const int c = 16 * nt + (lane & 15);
  const int r0 = 16 * mt + 4 * (lane >> 4);
  if (c >= in_dim) return;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (r0 + r < out_dim) {
      if (store) dw[(size_t)(r0 + r) * in_dim + c] = v[r];
      else unsafeAtomicAdd(dw + (size_t)(r0 + r) * in_dim + c, v[r]);
    }
}

// Compute units of the current device.  The count is cached per device ordinal (written once with the same value by
// whichever thread asks first); besides the thread-local error text this is the only state the library keeps.
inline int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    hipDeviceProp_t p;
    int n = 0;
    if (hipGetDeviceProperties(&p, dev) == hipSuccess) n = p.multiProcessorCount;
    cus[dev] = n > 0 ? n : 256;
  }
  return cus[dev];
}

constexpr size_t LDS_LIMIT = 160 * 1024;


// Specialised backward for exactly one hidden layer (fused_mlp_bwd2.hip), bias gradients included.
// *handled = false: shape not covered, nothing was launched.
int launch_mlp_bwd2(const MlpArgs& a, int dtype, hipStream_t s, bool* handled);
// The same for two or three hidden-to-hidden layers of width 64 with ReLU (fused_mlp_bwdn.hip).
int launch_mlp_bwdn(const MlpArgs& a, int dtype, hipStream_t s, bool* handled);
// The benchmark shape of launch_mlp_bwd2 (d_in <= 32, d_hidden = 64, d_out <= 16, ReLU, aligned rows, extents below
// 2^31 bytes) on eight waves per workgroup (fused_mlp_bwd2_w8.hip).  *handled = false: not that shape.
int launch_mlp_bwd2_w8(const MlpArgs& a, int dtype, hipStream_t s, bool* handled);
// The same with the weight and bias gradients summed in a fixed order and written, rounded to `dtype`, into out[6]
// (dw_in, db_in, dw_hid, db_hid, dw_out, db_out; NULL entries skipped); workspace: mlp_bwd2_w8_rounded_bytes().
// Also covers the shapes of launch_mlp_bwd2_ws.
size_t mlp_bwd2_w8_rounded_bytes(int d_in, int d_hidden, int d_out);
int launch_mlp_bwd2_w8_rounded(const MlpArgs& a, int dtype, int grad_dtype, void* const out[6], void* workspace, hipStream_t s, bool* handled);


// One hidden layer, width 64, ReLU, with d_in > 32 or d_out > 16 (aligned rows, extents below 2^31 bytes): chain and
// gradient waves (fused_mlp_bwd2_ws.hip).  *handled = false: not such a call, nothing was launched.
int launch_mlp_bwd2_ws(const MlpArgs& a, int dtype, hipStream_t s, bool* handled, int* blocks_out = nullptr);

// A whole network of up to nine hidden layers in one launch, any activation, widths and row alignment (fused_mlp_bwd_roles.hip);
// gradients written to out[6] (dw_in, db_in, dw_hid, db_hid, dw_out, db_out; NULL entries skipped) in grad_dtype.  The workspace
// holds mlp_bwd_roles_bytes() (0: too deep).
size_t mlp_bwd_roles_bytes(int64_t rows, int d_hidden, int depth, int act);
int launch_mlp_bwd_roles(const MlpArgs& a, int dtype, int grad_dtype, void* const out[6], void* workspace, hipStream_t s);

// The forward of one-hidden-layer ReLU networks of width 64 with aligned rows (fused_mlp_fwd2.hip).  *handled = false: not that shape, nothing was launched.
bool mlp_fwd2_takes(const MlpArgs& a, int dtype);  // whether launch_mlp_fwd2 would handle it
int launch_mlp_fwd2(const MlpArgs& a, int dtype, hipStream_t s, bool* handled);

// float32 storage and float32 products (fused_mlp_f32.hip).  The backward needs mlp32_bwd_workspace_bytes of scratch; write: see nf_mlp_bwd_f32.
size_t mlp32_bwd_workspace_bytes(int64_t rows, int d_hidden, int depth);
int mlp32_fwd(const float* x, int64_t x_stride, float* y, int64_t y_stride, const float* w_in, const float* b_in,
              const float* w_hid, const float* b_hid, const float* w_out, const float* b_out, int64_t rows, int d_in,
              int d_hidden, int d_out, int depth, int act, hipStream_t s);
int mlp32_bwd(const float* x, int64_t x_stride, const float* dy, int64_t dy_stride, float* dx, int64_t dx_stride,
              const float* w_in, const float* b_in, const float* w_hid, const float* b_hid, const float* w_out, float* dw_in,
              float* db_in, float* dw_hid, float* db_hid, float* dw_out, float* db_out, int64_t rows, int d_in, int d_hidden,
              int d_out, int depth, int act, bool write, void* workspace, int64_t workspace_bytes, hipStream_t s);

}  // namespace nf
