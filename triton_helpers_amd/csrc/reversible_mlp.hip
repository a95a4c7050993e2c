// Reversible (additive-coupling) fused MLP for gfx950, 16-bit storage, MFMA 16x16x32.
//
//   block k:  y1 = x1 + F_k(x2),  y2 = x2 + G_k(y1),   F/G(u) = act(u W1^T + b1) W2^T + b2
//
// Forward: one launch runs up to FWD_GROUP coupling blocks with all their weights resident
// in LDS; the two halves of the residual stream stay in float32 registers between blocks.
// Backward: reversible_bwd.hip.
//
// There is no counterpart in the reference; the layer math is that of its fused MLP
// (triton_helpers/layers/fully_fused_mlp/kernel.py:17-74).
#include "mlp_tile.h"
#include "reversible.h"

namespace nf {

constexpr int RFRAG = 64 * 8;
constexpr int FWD_GROUP = 4;   // coupling blocks per forward launch (LDS: 32 KiB of weights per block at H = 64)

struct RevArgs {
  const uint16_t* in;
  int64_t in_stride;
  uint16_t* out;
  int64_t out_stride;
  const uint16_t *w1, *b1, *w2, *b2;  // of the launch's first coupling
  int64_t rows;
  int half, nblocks, act;
  int vec_in, vec_out;
};

// accumulator-layout load: lane (n,g) gets features 16*mt + 4*g + r of row row0 + n as two packed dwords
__device__ __forceinline__ uint2 load_tile_packed(const uint16_t* base, int64_t stride, int64_t row0, int64_t rows, int col0,
                                                  int width, int mt, int lane, bool vec_ok) {
  uint2 v = make_uint2(0u, 0u);
  const int64_t r = row0 + (lane & 15);
  const int c = 16 * mt + 4 * (lane >> 4);
  if (r < rows && c < width) {
    const uint16_t* p = base + r * stride + col0 + c;
    if (vec_ok && c + 4 <= width) {
      v = *reinterpret_cast<const uint2*>(p);
    } else {
      uint16_t t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) t[i] = (c + i < width) ? p[i] : (uint16_t)0;
      v.x = (uint32_t)t[0] | ((uint32_t)t[1] << 16);
      v.y = (uint32_t)t[2] | ((uint32_t)t[3] << 16);
    }
  }
  return v;
}
__device__ __forceinline__ void store_tile_packed(uint16_t* base, int64_t stride, int64_t row0, int64_t rows, int col0,
                                                  int width, int mt, int lane, uint2 v, bool vec_ok) {
  const int64_t r = row0 + (lane & 15);
  const int c = 16 * mt + 4 * (lane >> 4);
  if (r >= rows || c >= width) return;
  uint16_t* p = base + r * stride + col0 + c;
  if (vec_ok && c + 4 <= width) {
    *reinterpret_cast<uint2*>(p) = v;
  } else {
    const uint16_t t[4] = {(uint16_t)(v.x & 0xffffu), (uint16_t)(v.x >> 16), (uint16_t)(v.y & 0xffffu), (uint16_t)(v.y >> 16)};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c + i < width) p[i] = t[i];
  }
}

// The same tiles when the caller knows that H is the padded width, that every row allows 8-byte accesses and that
// no chunk is ragged: one address per (tensor, row tile), the column part is an immediate offset.
template <bool FAST>
__device__ __forceinline__ uint2 ld_tile(const uint16_t* base, int64_t stride, int64_t row0, int64_t rows, int col0,
                                         int width, int mt, int lane, bool vec_ok) {
  if (FAST) return *reinterpret_cast<const uint2*>(base + (row0 + (lane & 15)) * stride + 4 * (lane >> 4) + col0 + 16 * mt);
  return load_tile_packed(base, stride, row0, rows, col0, width, mt, lane, vec_ok);
}
template <bool FAST>
__device__ __forceinline__ void st_tile(uint16_t* base, int64_t stride, int64_t row0, int64_t rows, int col0, int width,
                                        int mt, int lane, uint2 v, bool vec_ok) {
  if (FAST) {
    *reinterpret_cast<uint2*>(base + (row0 + (lane & 15)) * stride + 4 * (lane >> 4) + col0 + 16 * mt) = v;
    return;
  }
  store_tile_packed(base, stride, row0, rows, col0, width, mt, lane, v, vec_ok);
}

template <typename T>
__device__ __forceinline__ f32x4_t unpack4(uint2 v) {
  f32x4_t o = {unpack_lo<T>(v.x), unpack_hi<T>(v.x), unpack_lo<T>(v.y), unpack_hi<T>(v.y)};
  return o;
}
template <typename T>
__device__ __forceinline__ uint2 pack4(f32x4_t v) {
  return make_uint2(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]));
}

// packed accumulator-layout tiles P[nt][mt] -> B fragments (chain order) F[nt][kc]
template <int MT>
__device__ __forceinline__ void tiles_to_frags(const uint2 (&p)[2][4], Frag (&f)[2][2]) {
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f[nt][mt >> 1].w[2 * (mt & 1)] = p[nt][mt].x;
      f[nt][mt >> 1].w[2 * (mt & 1) + 1] = p[nt][mt].y;
    }
}

// K chunks outermost: the two products into one accumulator tile are MT * 2 instructions apart.
template <typename T, int MT, int KC>
__device__ __forceinline__ void rev_layer(f32x4_t (&acc)[2][4], const Frag (&in)[2][2], const uint16_t* frags, const float* bias,
                                          int lane) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    f32x4_t b4 = {0.0f, 0.0f, 0.0f, 0.0f};
    if (bias != nullptr) b4 = *reinterpret_cast<const f32x4_t*>(bias + 16 * mt + 4 * (lane >> 4));
    acc[0][mt] = b4;
    acc[1][mt] = b4;
  }
#pragma unroll
  for (int kc = 0; kc < KC; ++kc)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const Frag a = lds_frag(frags, mt * KC + kc, lane);
      acc[0][mt] = mfma16<T>(a, in[0][kc], acc[0][mt]);
      acc[1][mt] = mfma16<T>(a, in[1][kc], acc[1][mt]);
    }
}

template <typename T>
__device__ __forceinline__ void stage_bias_row(float* dst, const uint16_t* b, int n_valid, int n_pad, int tid, int nthreads) {
  for (int i = tid; i < n_pad; i += nthreads) {
    dst[i] = (b != nullptr && i < n_valid) ? T::to_f32(b[i]) : 0.0f;
  }
}

// ---------------------------------------------------------------------------------------
// Forward: up to FWD_GROUP blocks per launch
// ---------------------------------------------------------------------------------------
// ACT >= 0 fixes the activation at compile time (no per-element selection); -1 reads it from the arguments.
template <typename T, int HP, int ACT, bool FAST>
__global__ __launch_bounds__(768) void rev_fwd_k(RevArgs a) {
  constexpr int MT = HP / 16, KC = HP / 32, LAYER = MT * KC * RFRAG;
  const int act = ACT >= 0 ? ACT : a.act;
  const int nwaves = (int)(blockDim.x >> 6);
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, nthreads = blockDim.x, lane = tid & 63, wave = tid >> 6;
  uint16_t* frags = reinterpret_cast<uint16_t*>(smem);  // [nblocks][F.w1, F.w2, G.w1, G.w2][LAYER]
  float* bias = reinterpret_cast<float*>(frags + (size_t)a.nblocks * 4 * LAYER);  // [nblocks][4][HP]
  const int H = FAST ? HP : a.half;
  if constexpr (FAST) {
    // The biases are asked for first, then all layers as one list of 16-byte pieces, several in flight per thread: half as many
    // accesses as 8-byte ones, a clock each.  (Layer by layer sixteen rounds of loads waited for one another, and so did the biases, row by row.
    // Four GELU couplings, us, layer by layer / 8-byte pieces and bias rows / this: 1600 rows 32 / 21 / 16; 4096 rows 21.5 / 16.6 for the last two, 2^16
    // 35.5 / 26.5, 2^18 77 / 68.5; 32-wide 4096 rows 10.4 / 8.2.)
    const int n_bias = a.nblocks * 4 * HP;
    const auto bias_at = [&](int i) {  // [coupling][F.b1, F.b2, G.b1, G.b2][HP]
      const uint16_t* b = i / HP & 1 ? a.b2 : a.b1;
      return b != nullptr ? b + (size_t)(i / (2 * HP)) * HP + i % HP : a.w1;
    };
    const auto has_bias = [&](int i) { return (i / HP & 1 ? a.b2 : a.b1) != nullptr; };
    const int second = tid + nthreads;
    const uint16_t b0 = *bias_at(tid < n_bias ? tid : 0), b1 = *bias_at(second < n_bias ? second : 0);
    constexpr int PIECES = MT * KC * 64, AT_ONCE = 6;
    const int all = a.nblocks * 4 * PIECES;
    auto stage = [&](auto wide_c) {
      for (int u0 = tid; u0 < all; u0 += AT_ONCE * nthreads) {
        uint4 v[AT_ONCE];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
          const int u = u0 + i * nthreads;
          if (u - lane >= all) break;  // (the same for the whole wave: a matrix is whole waves' pieces)
          const int layer = u / PIECES, piece = u % PIECES, mt = (piece >> 6) / KC, kc = (piece >> 6) % KC;
          const uint16_t* w = (layer & 1 ? a.w2 : a.w1) + (size_t)(layer >> 1) * HP * HP + (16 * mt + (lane & 15)) * HP + 32 * kc + 8 * (lane >> 4);
          if constexpr (decltype(wide_c)::value) {
            v[i] = *reinterpret_cast<const uint4*>(w);
          } else {
            const uint2 lo = *reinterpret_cast<const uint2*>(w), hi = *reinterpret_cast<const uint2*>(w + 4);
            v[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
          }
        }
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
          const int u = u0 + i * nthreads;
          if (u - lane >= all) break;
          put_chain(frags + (size_t)(u - lane) * 8, lane & 15, lane >> 4, v[i]);
        }
      }
    };
    if (((uintptr_t)a.w1 | (uintptr_t)a.w2) % 16 == 0) stage(std::true_type{});
    else stage(std::false_type{});
    if (tid < n_bias) bias[tid] = has_bias(tid) ? T::to_f32(b0) : 0.0f;
    if (second < n_bias) bias[second] = has_bias(second) ? T::to_f32(b1) : 0.0f;
    for (int i = second + nthreads; i < n_bias; i += nthreads) bias[i] = has_bias(i) ? T::to_f32(*bias_at(i)) : 0.0f;
  } else {
    for (int k = 0; k < a.nblocks; ++k)
      for (int s = 0; s < 2; ++s) {
        const size_t sub = (size_t)(2 * k + s);
        stage_weight_frags<true, false>(frags + ((size_t)k * 4 + 2 * s) * LAYER, a.w1 + sub * H * H, H, H, MT, KC, tid, nthreads);
        stage_weight_frags<true, false>(frags + ((size_t)k * 4 + 2 * s + 1) * LAYER, a.w2 + sub * H * H, H, H, MT, KC, tid, nthreads);
        stage_bias_row<T>(bias + ((size_t)k * 4 + 2 * s) * HP, a.b1 ? a.b1 + sub * H : nullptr, H, HP, tid, nthreads);
        stage_bias_row<T>(bias + ((size_t)k * 4 + 2 * s + 1) * HP, a.b2 ? a.b2 + sub * H : nullptr, H, HP, tid, nthreads);
      }
  }
  __syncthreads();

  const int64_t n_chunks = (a.rows + 31) / 32;
  // Chunks to workgroups in turn, then to their waves: every unit has as many (262144 rows of four couplings, a workgroup's waves side by
  // side: 87 us, so 76), and few chunks spread over the units, where a wave has a SIMD to itself.
  for (int64_t chunk = (int64_t)wave * gridDim.x + blockIdx.x; chunk < n_chunks; chunk += (int64_t)gridDim.x * nwaves) {
    const int64_t row0 = chunk * 32;
    f32x4_t s1[2][4], s2[2][4];  // the two halves of the residual stream, float32
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        s1[nt][mt] = unpack4<T>(ld_tile<FAST>(a.in, a.in_stride, row0 + 16 * nt, a.rows, 0, H, mt, lane, a.vec_in));
        s2[nt][mt] = unpack4<T>(ld_tile<FAST>(a.in, a.in_stride, row0 + 16 * nt, a.rows, H, H, mt, lane, a.vec_in));
      }
    for (int k = 0; k < a.nblocks; ++k) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        // s == 0: s1 += F(s2) ; s == 1: s2 += G(s1)
        f32x4_t(&src)[2][4] = s == 0 ? s2 : s1;
        f32x4_t(&dst)[2][4] = s == 0 ? s1 : s2;
        const uint16_t* fw1 = frags + ((size_t)k * 4 + 2 * s) * LAYER;
        const float* bb1 = bias + ((size_t)k * 4 + 2 * s) * HP;
        uint2 p[2][4];
        Frag u[2][2], t[2][2];
        f32x4_t acc[2][4];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) p[nt][mt] = pack4<T>(src[nt][mt]);
        tiles_to_frags<MT>(p, u);
        rev_layer<T, MT, KC>(acc, u, fw1, bb1, lane);
        with_act(act, [&](auto act_c) {
          constexpr int A = decltype(act_c)::value;
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              f32x4_t z = acc[nt][mt];
#pragma unroll
              for (int r = 0; r < 4; ++r) z[r] = act_fwd(z[r], A);
              p[nt][mt] = pack4<T>(z);
            }
        });
        tiles_to_frags<MT>(p, t);
        rev_layer<T, MT, KC>(acc, t, fw1 + LAYER, bb1 + HP, lane);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) dst[nt][mt] += acc[nt][mt];
      }
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        st_tile<FAST>(a.out, a.out_stride, row0 + 16 * nt, a.rows, 0, H, mt, lane, pack4<T>(s1[nt][mt]), a.vec_out);
        st_tile<FAST>(a.out, a.out_stride, row0 + 16 * nt, a.rows, H, H, mt, lane, pack4<T>(s2[nt][mt]), a.vec_out);
      }
  }
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------
static int rev_validate(int64_t rows, int half, int blocks, int act, int dtype) {
  NF_REQUIRE(rows >= 0, NF_EINVAL, "rows negative");
  NF_REQUIRE(half >= 1 && half <= 64, NF_EINVAL, "half=%d outside 1..64", half);
  NF_REQUIRE(blocks >= 1, NF_EINVAL, "blocks=%d must be >= 1", blocks);
  NF_REQUIRE(act >= NF_ACT_NONE && act <= NF_ACT_GELU, NF_EINVAL, "unknown activation %d", act);
  NF_REQUIRE(dtype == NF_F16 || dtype == NF_BF16, NF_EUNSUPPORTED,
             "dtype code %d: the reversible MLP kernels take float16 or bfloat16 storage", dtype);
  return 0;
}

constexpr int64_t SPLIT_MIN_ROWS = 4096;  // from here on a ragged end is worth a launch of its own

static bool vec8_ok(const void* p, int64_t stride, int half) {
  return ((uintptr_t)p % 8 == 0) && (stride % 4 == 0) && (half % 4 == 0);
}
template <typename T, int HP>
static int launch_rev_fwd(RevArgs a, hipStream_t s) {
  constexpr int LAYER = (HP / 16) * (HP / 32) * RFRAG;
  const size_t lds = (size_t)a.nblocks * 4 * LAYER * 2 + (size_t)a.nblocks * 4 * HP * 4;
  const int64_t chunks = (a.rows + 31) / 32;
  // weights of several blocks leave room for one workgroup per CU only: give it 12 waves to keep three per SIMD
  const int waves = lds > 80 * 1024 ? 12 : 4;
  const int64_t cap = (int64_t)rev_cus() * (lds > 80 * 1024 ? 1 : 2);
  int64_t blocks = (chunks + waves - 1) / waves;
  if (blocks > cap) blocks = cap;
  if (blocks < rev_cus()) blocks = chunks < rev_cus() ? chunks : rev_cus();
  // full-width, aligned, unragged calls of GELU, ReLU and SiLU take the variants without per-tile checks
  const bool fast = a.half == HP && a.rows % 32 == 0 && a.vec_in && a.vec_out && (uintptr_t)a.w1 % 8 == 0 && (uintptr_t)a.w2 % 8 == 0;
  const void* kern = a.act == NF_ACT_GELU   ? (fast ? (const void*)rev_fwd_k<T, HP, NF_ACT_GELU, true>
                                                    : (const void*)rev_fwd_k<T, HP, NF_ACT_GELU, false>)
                     : a.act == NF_ACT_RELU ? (fast ? (const void*)rev_fwd_k<T, HP, NF_ACT_RELU, true>
                                                    : (const void*)rev_fwd_k<T, HP, NF_ACT_RELU, false>)
                     : (a.act == NF_ACT_SILU && fast) ? (const void*)rev_fwd_k<T, HP, NF_ACT_SILU, true>
                                            : (const void*)rev_fwd_k<T, HP, -1, false>;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  void* args[] = {(void*)&a};
  const hipError_t e = hipLaunchKernel(kern, dim3((unsigned)blocks), dim3(64 * waves), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(rev_fwd): %s", hipGetErrorString(e));
  return check_launch("rev_fwd");
}

}  // namespace nf

using namespace nf;

extern "C" int nf_revmlp_fwd(const void* x, int64_t x_stride, void* y, int64_t y_stride, const void* w1, const void* b1,
                             const void* w2, const void* b2, int64_t rows, int half, int blocks, int act, int dtype,
                             void* stream) {
  if (int rc = rev_validate(rows, half, blocks, act, dtype)) return rc;
  if (rows == 0) return 0;
  NF_REQUIRE(x && y && w1 && w2, NF_EINVAL, "NULL pointer argument");
  NF_REQUIRE(x_stride >= 2 * half && y_stride >= 2 * half, NF_EINVAL, "row stride smaller than 2*half");
  // Rows are independent: a large batch with a ragged end runs as its multiple of 32 rows (the variants without per-tile
  // checks, where the rest of the call allows them) plus a call of its own for the last rows.
  if (rows >= SPLIT_MIN_ROWS && rows % 32 != 0) {
    const int64_t main_rows = rows - rows % 32;
    if (int rc = nf_revmlp_fwd(x, x_stride, y, y_stride, w1, b1, w2, b2, main_rows, half, blocks, act, dtype, stream)) return rc;
    return nf_revmlp_fwd((const uint16_t*)x + main_rows * x_stride, x_stride, (uint16_t*)y + main_rows * y_stride, y_stride, w1, b1, w2, b2,
                         rows - main_rows, half, blocks, act, dtype, stream);
  }
  hipStream_t s = (hipStream_t)stream;
  const int es = 2;
  for (int k0 = 0; k0 < blocks; k0 += FWD_GROUP) {
    RevArgs a = {};
    // the first group reads x; later groups continue in place on y (a wave reads its rows before it writes them)
    a.in = (const uint16_t*)(k0 == 0 ? x : y);
    a.in_stride = k0 == 0 ? x_stride : y_stride;
    a.out = (uint16_t*)y;
    a.out_stride = y_stride;
    a.w1 = (const uint16_t*)w1 + (size_t)2 * k0 * half * half;
    a.w2 = (const uint16_t*)w2 + (size_t)2 * k0 * half * half;
    a.b1 = b1 ? (const uint16_t*)b1 + (size_t)2 * k0 * half : nullptr;
    a.b2 = b2 ? (const uint16_t*)b2 + (size_t)2 * k0 * half : nullptr;
    a.rows = rows;
    a.half = half;
    a.nblocks = blocks - k0 < FWD_GROUP ? blocks - k0 : FWD_GROUP;
    a.act = act;
    a.vec_in = vec8_ok(a.in, a.in_stride, half);
    a.vec_out = vec8_ok(a.out, a.out_stride, half);
    (void)es;
    int rc;
    if (half <= 32)
      rc = dtype == NF_BF16 ? launch_rev_fwd<BF16, 32>(a, s) : launch_rev_fwd<F16, 32>(a, s);
    else
      rc = dtype == NF_BF16 ? launch_rev_fwd<BF16, 64>(a, s) : launch_rev_fwd<F16, 64>(a, s);
    if (rc) return rc;
  }
  return 0;
}

extern "C" int64_t nf_revmlp_bwd_workspace_bytes(int64_t rows, int half, int blocks) {
  if (rows <= 0 || half < 1 || half > 64 || blocks < 1) return 0;
  return (int64_t)rev_bwd_bytes(rows, half, blocks);
}

extern "C" int nf_revmlp_bwd_summed(const void* y, int64_t y_stride, const void* dy, int64_t dy_stride, void* dx, int64_t dx_stride, void* x_rec,
                                    int64_t x_rec_stride, const void* w1, const void* b1, const void* w2, const void* b2, void* dw1, void* db1,
                                    void* dw2, void* db2, int64_t rows, int half, int blocks, int act, int dtype, int grad_dtype,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = rev_validate(rows, half, blocks, act, dtype)) return rc;
  NF_REQUIRE(grad_dtype == dtype || grad_dtype == NF_F32, NF_EINVAL, "gradients come back in the storage dtype or in float32");
  NF_REQUIRE(rows > 0, NF_EINVAL, "no rows: the gradients would be left unwritten");
  NF_REQUIRE(y && dy && dx && x_rec && w1 && w2 && dw1 && dw2 && workspace, NF_EINVAL,
             "NULL pointer argument (x_rec is required: it carries the reconstructed input between blocks)");
  NF_REQUIRE(y_stride >= 2 * half && dy_stride >= 2 * half && dx_stride >= 2 * half && x_rec_stride >= 2 * half, NF_EINVAL,
             "row stride smaller than 2*half");
  const int64_t need = nf_revmlp_bwd_workspace_bytes(rows, half, blocks);
  NF_REQUIRE(workspace_bytes >= need && (uintptr_t)workspace % 16 == 0, NF_EINVAL, "a 16-byte aligned workspace of %lld bytes is needed", (long long)need);
  const RevBwdCall c = {(const uint16_t*)y, (const uint16_t*)dy, (uint16_t*)dx, (uint16_t*)x_rec, y_stride, dy_stride, dx_stride, x_rec_stride, rows,
                        (const uint16_t*)w1, (const uint16_t*)b1, (const uint16_t*)w2, (const uint16_t*)b2, dw1, db1, dw2, db2, half, blocks, act,
                        grad_dtype, workspace};
  return rev_bwd(c, dtype, (hipStream_t)stream);
}

extern "C" int nf_revmlp_bwd(const void* y, int64_t y_stride, const void* dy, int64_t dy_stride, void* dx, int64_t dx_stride,
                             void* x_rec, int64_t x_rec_stride, const void* w1, const void* b1, const void* w2,
                             const void* b2, float* dw1, float* db1, float* dw2, float* db2, int64_t rows, int half,
                             int blocks, int act, int dtype, void* stream) {
  if (int rc = rev_validate(rows, half, blocks, act, dtype)) return rc;
  if (rows == 0) return 0;
  NF_REQUIRE(y && dy && dx && x_rec && w1 && w2 && dw1 && dw2, NF_EINVAL,
             "NULL pointer argument (x_rec is required: it carries the reconstructed input between blocks)");
  NF_REQUIRE(y_stride >= 2 * half && dy_stride >= 2 * half && dx_stride >= 2 * half && x_rec_stride >= 2 * half, NF_EINVAL,
             "row stride smaller than 2*half");
  const RevBwdCall c = {(const uint16_t*)y, (const uint16_t*)dy, (uint16_t*)dx, (uint16_t*)x_rec, y_stride, dy_stride, dx_stride, x_rec_stride, rows,
                        (const uint16_t*)w1, (const uint16_t*)b1, (const uint16_t*)w2, (const uint16_t*)b2, dw1, db1, dw2, db2, half, blocks, act,
                        NF_F32, nullptr};
  return rev_bwd(c, dtype, (hipStream_t)stream);
}
