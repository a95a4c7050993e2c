// The forward of one-hidden-layer ReLU networks of width 64 (d_in <= 64, d_out <= 64; the decoder / benchmark shape
// 32 -> 64 -> 64 -> 16 and the 64-wide shapes of the reference's own benchmark), 8-byte aligned rows, as a kernel of
// its own per (input, output) width class: twelve waves per workgroup, the chunk body one basic block (no
// run-time tests of activation, depth, alignment or row count inside it), rows addressed through buffer descriptors
// (reads past the end return zero, stores past it are dropped), the next chunk's rows requested before this one's
// products.  Everything else stays on mlp_fwd_k (fused_mlp.hip), which loops over a run-time depth.
#include "fused_mlp_bwd2_kernels.h"

namespace nf {

// Workgroups per CU of the launch (15 KB of LDS and under 128 registers each: the grid, not the chip, sets it).
#ifndef NF_FWD2_WG_PER_CU
#define NF_FWD2_WG_PER_CU 1
#endif

#ifndef NF_FWD2_WAVES
#define NF_FWD2_WAVES 12
#endif

// XC: how x is stored (MlpArgs::x_conv); KIN / OUTP: d_in / d_out rounded up to 32 or 64 / 16 or 64.
// Twelve waves where the weight fragments (held in registers across chunks) leave room for three waves per SIMD,
// eight for the 64-wide inputs / outputs.
constexpr int fwd2_waves(int kin, int outp) { return (kin == 32 && outp == 16) ? NF_FWD2_WAVES : 8; }

// XW / YW: rows of x / y move in whole 16-byte pieces (16-byte aligned rows of a multiple of eight values) that are exchanged
// between the lane groups, instead of 8-byte pieces.  A tile access has no two neighbouring lanes on one line and the L1 takes
// a lane a clock, so 8-byte pieces are 64 clocks per 512 bytes: 30 of the 34 us that 64 -> 64 -> 64 -> 64 took at 2^19 rows, 25 now
// (2^20 rows 59 -> 47, 32 -> 64 -> 64 -> 64 41 -> 36, 64 -> 64 -> 64 -> 16 36 -> 30).  The decoder shape moves a third of that and is
// held by memory (2^20 rows 21 us either way): 8-byte pieces there.
// LIST8: the hidden matrix lies on 8 bytes and it or the output matrix not on 16.  With all ways of staging in one kernel 2^18 rows of the decoder shape take 9.4 us, with
// those of 16 bytes alone in one 8.75 (2^16 5.66; 64 -> 64 -> 64 -> 64, 2^19 rows 27.4), so 8.6 (5.5; 27.1).
template <typename T, int XC, int KIN, int OUTP, bool XW, bool YW, bool LIST8>
__global__ __launch_bounds__(64 * fwd2_waves(KIN, OUTP)) void mlp_fwd2_k(MlpArgs a) {
  constexpr int HP = 64, NT = 2, WAVES = fwd2_waves(KIN, OUTP);
  constexpr int KC_IN = KIN / 32, KC_H = HP / 32, MT_H = HP / 16, MT_O = OUTP / 16;
  constexpr int ROWS = 16 * NT;
  constexpr int nthreads = 64 * WAVES;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n_chunks = (a.rows + ROWS - 1) / ROWS;
  const int64_t wave_stride = (int64_t)gridDim.x * WAVES;
  const int64_t first_chunk = (int64_t)blockIdx.x * WAVES + wave;
  const __amdgpu_buffer_rsrc_t rs_x = rows_rsrc(a.x, a.rows, a.x_stride), rs_y = rows_rsrc(a.y, a.rows, a.y_stride);
  uint32_t off_x[KC_IN][2];
#pragma unroll
  for (int kc = 0; kc < KC_IN; ++kc)
#pragma unroll
    for (int h = 0; h < 2; ++h) off_x[kc][h] = piece_offset(lane & 15, XW ? 32 * kc + 8 * (lane >> 4) : 32 * kc + 16 * h + 4 * (lane >> 4), a.d_in, a.x_stride);
  uint32_t off_y[MT_O];
#pragma unroll
  for (int mt = 0; mt < MT_O; ++mt) {
    if (YW && MT_O > 1) off_y[mt] = piece_offset(lane & 15, 32 * (mt >> 1) + 8 * (lane >> 4), a.d_out, a.y_stride);
    else off_y[mt] = piece_offset(lane & 15, 16 * mt + 4 * (lane >> 4), a.d_out, a.y_stride);
  }
  auto load_x = [&](int64_t chunk, int nt, int kc) {  // XW: in natural order until it is used
    const uint32_t at = (uint32_t)((chunk * ROWS + 16 * nt) * a.x_stride * 2);
    if constexpr (XW) {
      Frag f;
      f.u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs_x, off_x[kc][0] + at, 0, 0));
      return f;
    }
    const buf_v2u lo = __builtin_amdgcn_raw_buffer_load_b64(rs_x, off_x[kc][0] + at, 0, 0);
    const buf_v2u hi = __builtin_amdgcn_raw_buffer_load_b64(rs_x, off_x[kc][1] + at, 0, 0);
    Frag f;
    f.w[0] = lo[0]; f.w[1] = lo[1]; f.w[2] = hi[0]; f.w[3] = hi[1];
    return f;
  };
  // rows in flight per wave: the next chunk, and for 64-wide inputs (eight waves, 4 KB per chunk) the one behind it too (64 -> 64 -> 16: 45.8 -> 40.9 us per 2^20 rows)
  constexpr bool DEEP = KIN > 32;
  Frag nx[NT][KC_IN], nnx[NT][KC_IN];
  auto first_rows = [&] {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int kc = 0; kc < KC_IN; ++kc) {
        nx[nt][kc] = load_x(first_chunk, nt, kc);
        if constexpr (DEEP) nnx[nt][kc] = load_x(first_chunk + wave_stride, nt, kc);
      }
  };

  uint16_t* f_in = reinterpret_cast<uint16_t*>(smem);   // W_in  [MT_H][KC_IN]
  uint16_t* f_hid = f_in + MT_H * KC_IN * FRAG_ELEMS;   // W_hid [MT_H][KC_H]
  uint16_t* f_out = f_hid + MT_H * KC_H * FRAG_ELEMS;   // W_out [MT_O][KC_H]
  float* bias_in = reinterpret_cast<float*>(f_out + MT_O * KC_H * FRAG_ELEMS);
  float* bias_hid = bias_in + HP;
  float* bias_out = bias_hid + HP;
  // (us over inputs that no cache holds, matrix by matrix in 8-byte pieces / this: 32 -> 64 -> 64 -> 16 2^18 rows 9.3 / 7.5, 2^20 22.5 / 19.4;
  // 64 -> 64 -> 64 -> 64 2^18 15.6 / 13.8, 2^19 30.0 / 28.3)
  if constexpr (LIST8) stage_network<T, KIN, HP, OUTP, 8, true, nthreads>(f_in, bias_in, a, tid, nthreads, first_rows);
  else if (((uintptr_t)a.w_hid | (uintptr_t)a.w_out) % 16 == 0) stage_network<T, KIN, HP, OUTP, 16, true, nthreads>(f_in, bias_in, a, tid, nthreads, first_rows);
  else stage_network<T, KIN, HP, OUTP, 0, true, nthreads>(f_in, bias_in, a, tid, nthreads, first_rows);
  __syncthreads();

  for (int64_t chunk = first_chunk; chunk < n_chunks; chunk += wave_stride) {
    Frag in[NT][2], h[NT][2];
    f32x4_t acc[NT][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int kc = 0; kc < KC_IN; ++kc) {
        in[nt][kc] = XC == 0 ? nx[nt][kc] : convert_frag(nx[nt][kc], XC);
        if constexpr (XW) in[nt][kc] = nat_to_chain(in[nt][kc]);
        if constexpr (DEEP) {
          nx[nt][kc] = nnx[nt][kc];
          nnx[nt][kc] = load_x(chunk + 2 * wave_stride, nt, kc);
        } else {
          nx[nt][kc] = load_x(chunk + wave_stride, nt, kc);
        }
      }
    layer_nt<T, NT, MT_H, KC_IN, 1>(acc, in, f_in, bias_in, lane);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT_H; ++mt) {
        h[nt][mt >> 1].w[2 * (mt & 1)] = relu_pk(pack2<T>(acc[nt][mt][0], acc[nt][mt][1]));
        h[nt][mt >> 1].w[2 * (mt & 1) + 1] = relu_pk(pack2<T>(acc[nt][mt][2], acc[nt][mt][3]));
      }
    layer_nt<T, NT, MT_H, KC_H, 1>(acc, h, f_hid, bias_hid, lane);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT_H; ++mt) {
        h[nt][mt >> 1].w[2 * (mt & 1)] = relu_pk(pack2<T>(acc[nt][mt][0], acc[nt][mt][1]));
        h[nt][mt >> 1].w[2 * (mt & 1) + 1] = relu_pk(pack2<T>(acc[nt][mt][2], acc[nt][mt][3]));
      }
    layer_nt<T, NT, MT_O, KC_H, 1>(acc, h, f_out, bias_out, lane);
    uint32_t out[NT][MT_O][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT_O; ++mt) {
        out[nt][mt][0] = pack2<T>(acc[nt][mt][0], acc[nt][mt][1]);
        out[nt][mt][1] = pack2<T>(acc[nt][mt][2], acc[nt][mt][3]);
      }
    auto at = [&](int nt) { return (uint32_t)((chunk * ROWS + 16 * nt) * a.y_stride * 2); };
    if constexpr (YW && MT_O > 1) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT_O; mt += 2) {
          Frag f;
          f.w[0] = out[nt][mt][0]; f.w[1] = out[nt][mt][1]; f.w[2] = out[nt][mt + 1][0]; f.w[3] = out[nt][mt + 1][1];
          f = chain_to_nat(f);
          const buf_v4u o = {f.w[0], f.w[1], f.w[2], f.w[3]};
          __builtin_amdgcn_raw_buffer_store_b128(o, rs_y, off_y[mt] + at(nt), 0, 0);
        }
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT_O; ++mt) {
          const buf_v2u o = {out[nt][mt][0], out[nt][mt][1]};
          __builtin_amdgcn_raw_buffer_store_b64(o, rs_y, off_y[mt] + at(nt), 0, 0);
        }
    }
  }
}

template <typename T, int KIN, int OUTP>
static int launch_fwd2(const MlpArgs& a0, hipStream_t s) {
  MlpArgs a = a0;
  constexpr int WAVES = fwd2_waves(KIN, OUTP), ROWS = 32;
  constexpr size_t LDS = ((size_t)4 * (KIN / 32) + 4 * 2 + (OUTP / 16) * 2) * 1024 + (size_t)(64 + 64 + OUTP) * 4;
  a.waves = WAVES;
  const int64_t chunks = (a.rows + ROWS - 1) / ROWS;
  int64_t blocks = (chunks + WAVES - 1) / WAVES;
  const int64_t cap = (int64_t)device_cus() * NF_FWD2_WG_PER_CU;
  if (blocks > cap) blocks = cap;
  constexpr int XC_OTHER = T::code == NF_BF16 ? 1 : 2;
  const bool list8 = (uintptr_t)a.w_hid % 8 == 0 && ((uintptr_t)a.w_hid | (uintptr_t)a.w_out) % 16 != 0;
  const auto pick = [&](auto xw_c, auto yw_c) -> const void* {
    constexpr bool XW = decltype(xw_c)::value, YW = decltype(yw_c)::value;
    if (list8) return a.x_conv == 0 ? (const void*)mlp_fwd2_k<T, 0, KIN, OUTP, XW, YW, true> : (const void*)mlp_fwd2_k<T, XC_OTHER, KIN, OUTP, XW, YW, true>;
    return a.x_conv == 0 ? (const void*)mlp_fwd2_k<T, 0, KIN, OUTP, XW, YW, false> : (const void*)mlp_fwd2_k<T, XC_OTHER, KIN, OUTP, XW, YW, false>;
  };
  const void* kern = pick(std::false_type{}, std::false_type{});
  if constexpr (KIN > 32 || OUTP > 16) {
    const bool xw = vec_load_ok(a.x, a.x_stride, a.d_in), yw = xw && OUTP > 16 && vec_load_ok(a.y, a.y_stride, a.d_out);
    if (yw) kern = pick(std::true_type{}, std::bool_constant<OUTP != 16>{});
    else if (xw) kern = pick(std::true_type{}, std::false_type{});
  }
  void* args[] = {(void*)&a};
  const hipError_t e = hipLaunchKernel(kern, dim3((unsigned)blocks), dim3(64 * WAVES), args, LDS, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(mlp_fwd2): %s", hipGetErrorString(e));
  return check_launch("mlp_fwd2");
}

bool mlp_fwd2_takes(const MlpArgs& a, int dtype) {
  const int xc_other = dtype == NF_BF16 ? 1 : 2;
  const auto rows8 = [](const void* p, int64_t stride) { return (uintptr_t)p % 8 == 0 && stride % 4 == 0; };
  const bool shape = a.depth == 2 && a.d_hidden == 64 && a.d_in <= 64 && a.d_out <= 64 && a.act == NF_ACT_RELU && a.in_act == NF_ACT_NONE &&
                     (a.x_conv == 0 || a.x_conv == xc_other);
  const bool aligned = a.d_in % 4 == 0 && a.d_out % 4 == 0 && rows8(a.x, a.x_stride) && rows8(a.y, a.y_stride);
  const bool in_reach = rows_in_reach(a.rows, a.x_stride) && rows_in_reach(a.rows, a.y_stride);
  return shape && aligned && in_reach;
}

int launch_mlp_fwd2(const MlpArgs& a, int dtype, hipStream_t s, bool* handled) {
  *handled = mlp_fwd2_takes(a, dtype);
  if (!*handled) return 0;
  const bool wide_in = a.d_in > 32, wide_out = a.d_out > 16;
#define NF_FWD2_DISPATCH(T)                                          \
  (wide_in ? (wide_out ? launch_fwd2<T, 64, 64>(a, s) : launch_fwd2<T, 64, 16>(a, s)) \
           : (wide_out ? launch_fwd2<T, 32, 64>(a, s) : launch_fwd2<T, 32, 16>(a, s)))
  return dtype == NF_BF16 ? NF_FWD2_DISPATCH(BF16) : NF_FWD2_DISPATCH(F16);
#undef NF_FWD2_DISPATCH
}

}  // namespace nf
