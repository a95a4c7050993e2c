// Backward of the reversible MLP (reversible_mlp.hip), workgroups split by role (role_split.h).
//
//   block k:  y1 = x1 + F_k(x2),  y2 = x2 + G_k(y1),   F/G(u) = act(u W1^T + b1) W2^T + b2
//
// From a block's output (y, dy) a chain wave rebuilds the block's input (x2 = y2 - G(y1), x1 = y1 - F(x2)) while it propagates the
// gradient back, sixteen rows at a time with everything in registers, and carries (x, dx), rounded to 16 bit, into the block below.  The
// four gradient waves hold the weight gradients of the couplings of a pass (CPL: two of 64-wide halves = 128 of a wave's 168
// registers, four of 32-wide ones) over all rows; the operands of dW reach them through LDS, four sections per coupling.  A pass keeps
// its couplings' weights in LDS; the next pass, CPL couplings further down, reads (x, dx) of its own rows from where this one wrote
// them, so no workgroup waits for another.  No forward activation is stored.
//
// The stream's features are contracted in natural order and produced in "wide order" (wide_feature()), so a lane's row pieces are 16
// bytes; the columns of W1 and the rows of W2 lie permuted accordingly in LDS, and the gradients' tiles are put back when they leave.
//
// What it replaces: one wave per SIMD held a coupling's four gradients next to the chain (512 registers, matrix-core transposes for
// their operands, both forms of the weights in LDS), issued vector and matrix instructions in turn and moved (y, dy) -> (x, dx) once per
// coupling: 4.4 GB of 2^20 rows and four couplings.  Four GELU couplings in bfloat16, us: 64-wide, 1000 rows 112 -> 35, 2^16 141 -> 84, 2^18
// 324 -> 237, 2^20 1110 -> 865; 48-wide (each coupling was a launch) 96 -> 35, 174 -> 88, 461 -> 231, 1712 -> 836; 32-wide 48 -> 18, 54 -> 43,
// 129 -> 98, 500 -> 362.  What bounds it now: the chain's vector instructions (half of the time, a third of them the activation's) and what a
// chain wave waits for between its products, with two of them on a SIMD.
#include "reversible.h"
#include "role_split.h"

namespace nf {

struct RevBwdArgs {
  const uint16_t *in, *dy;  // of the topmost coupling
  uint16_t *out, *dx;       // x_rec, dx: also the input of every pass but the first
  int64_t in_stride, dy_stride, out_stride, dx_stride, rows;
  const uint16_t *w1, *b1, *w2, *b2;
  float *dw1, *db1, *dw2, *db2;  // accumulators of a call without slots
  float* slots;                  // [workgroup][couplings] sums of the weight gradients, or NULL
  int64_t slot_stride;
  int half, nblocks;
  int vec_top, vec_below;  // rows of (in, dy, out, dx) / of (out, dx) are whole 16-byte aligned pieces
};

typedef const RevBwdArgs __attribute__((address_space(4))) * RevArgsPtr;
__device__ __forceinline__ RevArgsPtr fresh_rev_args() {  // the arguments, read again where they are used (see opaque())
  RevArgsPtr p = (RevArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// The lane's number, counted again where it is used: kept, it and what depends on it would take registers for the whole kernel.
__device__ __forceinline__ int fresh_lane() {
  uint32_t all = ~0u;
  asm volatile("" : "+s"(all));
  return (int)__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u));
}

__device__ __forceinline__ float lane_xor(float v, int lane, int m) {  // (as __shfl_xor, which would keep its own lane number)
  return __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ m) << 2, __float_as_int(v)));
}

// An LDS address the optimiser takes as it is: reads around it use their instruction's offset instead of a register each.
__device__ __forceinline__ const char* lds_base(const char* p) {
  auto q = (const __attribute__((address_space(3))) char*)p;
  asm("" : "+v"(q));
  return (const char*)q;
}

// Activation and its derivative from one pre-activation (GELU shares the exponential between the two).
template <int ACT>
__device__ __forceinline__ void act_both(float z, float& h, float& g) {
  if (ACT == NF_ACT_GELU) {
    float pdf;
    const float cdf = normal_cdf_pdf3(z, &pdf);
    h = z * cdf;
    g = cdf + z * pdf;
  } else if (ACT == NF_ACT_RELU) {
    h = fmaxf(z, 0.0f);
    g = z > 0.0f ? 1.0f : 0.0f;
  } else {
    h = act_fwd(z, ACT);
    g = act_grad(z, ACT);
  }
}

// A workgroup's sums of a coupling's weight gradients: accumulator tiles [MT][MT][F.w1, F.w2, G.w1, G.w2] of 64 lanes x 4, then bias
// gradients [MT][F.b1, F.b2, G.b1, G.b2] of 16.
template <int HP>
struct RevSlot {
  static constexpr int MT = HP / 16, TILES = MT * MT * 4, FLOATS = TILES * 256 + 4 * HP;
};
constexpr int rev_couplings(int hp) { return hp == 64 ? 2 : 4; }  // couplings of a pass
constexpr size_t rev_bwd_lds(int hp, int cw) {
  return (size_t)rev_couplings(hp) * 4 * (hp * ROLES_PITCH + 64 * 4) + 4 * 64 * 4 + (size_t)4 * 16 * cw * ROLES_PITCH + 64 * 4;
}

// The weights of couplings k0 .. k0 + n - 1 as LDS matrices of HP rows, [coupling][F.w1, F.w2, G.w1, G.w2]: 8-byte piece 8kc + 4e + g of a row
// of w1 holds the features 32kc + 8g + 4e .., row 16t + m of w2 belongs to feature wide_feature(t, m); and their biases alike.
template <typename T, int HP, int N>
__device__ __forceinline__ void stage_couplings(char* w, float* bias, const RevBwdArgs& a, int k0, int n, int tid) {
  constexpr int DEEP = 8;
  const int H = a.half, units = n * 4 * HP * 16;
  const bool vec = H % 4 == 0 && ((uintptr_t)a.w1 | (uintptr_t)a.w2) % 8 == 0;
  if (H == HP && ((uintptr_t)a.w1 | (uintptr_t)a.w2) % 16 == 0) {
    // Full matrices in 16-byte pieces, two 8-byte ones each: half the accesses, a clock each for the L1, and no load under a condition (four GELU
    // couplings, us, 8-byte pieces / this: 64-wide 1024 rows 37.0 / 35.0, 2^16 86.6 / 83.5, 32-wide 4096 21.0 / 19.5, 2^18 with SiLU 92 / 88).
    constexpr int AT_ONCE = 6;
    const int wide = n * 4 * HP * (HP / 8);
    for (int u0 = tid; u0 < wide; u0 += N * AT_ONCE) {
      uint4 v[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int u = u0 + i * N;
        if (u >= wide) break;  // (the same for the whole wave)
        const int m = u / (HP * HP / 8), row = u / (HP / 8) % HP, c = 8 * (u % (HP / 8));
        const int r = m & 1 ? wide_feature(row >> 4, row & 15) : row;
        v[i] = *reinterpret_cast<const uint4*>((m & 1 ? a.w2 : a.w1) + ((size_t)(2 * k0 + (m >> 1)) * HP + r) * HP + c);
      }
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int u = u0 + i * N;
        if (u >= wide) break;
        const int m = u / (HP * HP / 8), row = u / (HP / 8) % HP, q = u % (HP / 8);
        // columns 8q .. are the pieces 2q and 2q + 1 of a second layer, 8 (q / 4) + q % 4 and the fourth behind it of a first
        const int p = m & 1 ? 2 * q : (q & 4) << 1 | (q & 3), p1 = m & 1 ? p + 1 : p + 4;
        char* dst = w + (m * HP + row) * ROLES_PITCH;
        *reinterpret_cast<uint2*>(dst + ((p ^ swizzle(row)) << 3)) = make_uint2(v[i].x, v[i].y);
        *reinterpret_cast<uint2*>(dst + ((p1 ^ swizzle(row)) << 3)) = make_uint2(v[i].z, v[i].w);
      }
    }
  } else {
    for (int u0 = tid; u0 < units; u0 += N * DEEP) {
      uint2 v[DEEP];
#pragma unroll
      for (int i = 0; i < DEEP; ++i) {
        const int u = u0 + i * N, m = u / (HP * 16), row = (u >> 4) & (HP - 1), p = u & 15;
        const bool second = m & 1;
        const int r = second ? wide_feature(row >> 4, row & 15) : row;
        const int c = 4 * (second ? p : (p & 8) | ((p & 3) << 1) | ((p >> 2) & 1));
        v[i] = make_uint2(0u, 0u);
        if (u < units && r < H && c < H) {
          const uint16_t* q = (second ? a.w2 : a.w1) + ((size_t)(2 * k0 + (m >> 1)) * H + r) * H + c;
          if (vec) {
            v[i] = *reinterpret_cast<const uint2*>(q);
          } else {
            uint16_t t[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) t[j] = c + j < H ? q[j] : (uint16_t)0;
            v[i].x = (uint32_t)t[0] | ((uint32_t)t[1] << 16);
            v[i].y = (uint32_t)t[2] | ((uint32_t)t[3] << 16);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < DEEP; ++i) {
        const int u = u0 + i * N, row = u >> 4;
        if (u < units) *reinterpret_cast<uint2*>(w + row * ROLES_PITCH + (((u & 15) ^ swizzle(row)) << 3)) = v[i];
      }
    }
  }
  for (int i = tid; i < n * 4 * 64; i += N) {
    const int m = i >> 6, q = i & 63, f = m & 1 ? wide_feature(q >> 4, q & 15) : q;
    const uint16_t* b = m & 1 ? a.b2 : a.b1;
    bias[i] = b != nullptr && f < H ? T::to_f32(b[(size_t)(2 * k0 + (m >> 1)) * H + f]) : 0.0f;
  }
}

// CW: chain waves; OCC: waves per SIMD the kernel is compiled for.
template <typename T, int HP, int ACT, int CW, int OCC>
__global__ __launch_bounds__(64 * (CW + 4), OCC) void rev_bwd_k(RevBwdArgs a) {
  constexpr int MT = HP / 16, KC = HP / 32, TW = HP / 32, CPL = rev_couplings(HP), ROWS = 16 * CW, THREADS = 64 * (CW + 4);
  constexpr int MATRIX = HP * ROLES_PITCH, PANEL = ROWS * ROLES_PITCH, AREA = 2 * PANEL;
  extern __shared__ __align__(16) char rev_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* weights = rev_smem;                                        // [CPL][F.w1, F.w2, G.w1, G.w2][HP][128]
  float* bias = reinterpret_cast<float*>(weights + CPL * 4 * MATRIX);  // [CPL][4][64]
  // Rows past the batch's end run the couplings too.  Their gradient is zero, but what the biases alone drive beyond the 16-bit range
  // would reach dW as 0 * inf, within one coupling already.  They read zeros as biases: nothing but zeros goes through them then.
  float* no_bias = bias + CPL * 4 * 64;                            // [4][64] zeros
  char* areas = reinterpret_cast<char*>(no_bias + 4 * 64);         // [2][gradient rows | input rows][ROWS][128]
  Sections<CW> sections = {reinterpret_cast<int*>(areas + 2 * AREA), 0};
  if (threadIdx.x < 32) sections.flags[threadIdx.x] = 0;
  if (threadIdx.x < 4 * 64) no_bias[threadIdx.x] = 0.0f;
  const int64_t per_round = (int64_t)gridDim.x * ROWS, rounds = (a.rows + per_round - 1) / per_round;
  const f32x4_t zero4 = {0.0f, 0.0f, 0.0f, 0.0f};

  for (int top = a.nblocks; top > 0; top -= CPL) {  // couplings top - 1 .. top - count
    const int count = top < CPL ? top : CPL, k0 = top - count, lane = fresh_lane(), n = lane & 15, g = lane >> 4;
    const int tr0 = tr_offset(n, g);
    stage_couplings<T, HP, THREADS>(weights, bias, a, k0, count, 64 * wave + fresh_lane());
    // (the rows this wave wrote in the pass before have to be in memory before it reads them)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (wave < CW) {
      // ------------------------------------------------------------------ chain waves
      const int chain0 = chain_offset(n, g);
      const int64_t row0 = (int64_t)blockIdx.x * ROWS + wave * 16 + n;  // a lane's row of the first round
      char* mine = areas + wave * 16 * ROLES_PITCH;  // this wave's rows of the first area
      // an operand of a layer's dW: panel 0 the gradient of its output, panel 1 its input
      auto park = [&](const Frag (&f)[KC], int area, int panel) {
        char* p = mine + area * AREA + panel * PANEL;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) write_pieces(p + (chain0 ^ 64 * kc), p + (chain0 ^ 64 * kc ^ 32), f[kc]);
      };
      const bool first = opaque(top) == a.nblocks;
      Frag y1[KC], y2[KC], d1[KC], d2[KC];  // the stream and its gradient, lane group g: features 32 kc + 8 g ..
      // The pieces p of a half of the stream and q of the other half's gradient.  Rows of whole pieces: of a
      // row that is there and from within it, zeroed when they are used, so that no load has a condition of its own.
      auto load_half = [&](Frag (&p)[KC], Frag (&q)[KC], bool second, int64_t r) {
        const RevArgsPtr k = fresh_rev_args();
        const int H = k->half;
        const int64_t is = first ? k->in_stride : k->out_stride, ds = first ? k->dy_stride : k->dx_stride;
        const uint16_t *in = (first ? k->in : k->out) + (second ? H : 0), *dy = (first ? k->dy : k->dx) + (second ? 0 : H);
        if ((first ? k->vec_top : k->vec_below) != 0) {
          const int64_t row = r < k->rows ? r : k->rows - 1;
          in += row * is;
          dy += row * ds;
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) {
            const int c = 32 * kc + 8 * g < H ? 32 * kc + 8 * g : H - 8;
            p[kc].u = *reinterpret_cast<const uint4*>(in + c);
            q[kc].u = *reinterpret_cast<const uint4*>(dy + c);
          }
          return;
        }
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          p[kc] = load_row8(in, is, r, k->rows, H, 32 * kc + 8 * g, false);
          q[kc] = load_row8(dy, ds, r, k->rows, H, 32 * kc + 8 * g, false);
        }
      };
      auto store_half = [&](const Frag (&p)[KC], const Frag (&q)[KC], bool second, int64_t r) {
        const RevArgsPtr k = fresh_rev_args();
        const int H = k->half;
        uint16_t *out = k->out + (second ? H : 0), *dx = k->dx + (second ? 0 : H);
        if (k->vec_below != 0) {
          if (r >= k->rows) return;
          out += r * k->out_stride;
          dx += r * k->dx_stride;
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) {
            const int c = 32 * kc + 8 * g;
            if (c >= H) continue;
            *reinterpret_cast<uint4*>(out + c) = p[kc].u;
            *reinterpret_cast<uint4*>(dx + c) = q[kc].u;
          }
          return;
        }
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          store_row8(out, k->out_stride, r, k->rows, H, 32 * kc + 8 * g, p[kc], false);
          store_row8(dx, k->dx_stride, r, k->rows, H, 32 * kc + 8 * g, q[kc], false);
        }
      };
      // Back through  v = v' + S(u):  v' = v - S(u), e += (dS/du)^T d, with the operands of S's two weight gradients parked on the way.
      // between(0), between(1): behind the first and the second of them.
      auto sub = [&](const char* w, const float* b, const Frag (&u)[KC], const Frag (&d)[KC], Frag (&v)[KC], Frag (&e)[KC], auto&& between) {
        f32x4_t acc[MT];
        Frag t[KC], gate[KC], dz[KC];
        auto product = [&](const char* m, const float* bb, const Frag (&x)[KC]) {  // acc = bb + M x
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = *reinterpret_cast<const f32x4_t*>(bb + 16 * mt + 4 * g);
#pragma unroll
          for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              const char* p = m + mt * 2048;
              acc[mt] = mfma16<T>(read_pieces(p + (chain0 ^ 64 * kc), p + (chain0 ^ 64 * kc ^ 32)), x[kc], acc[mt]);
            }
        };
        auto product_tr = [&](const char* m, const Frag (&x)[KC]) {  // acc = M^T x
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = zero4;
#pragma unroll
          for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              const char* p = m + kc * 32 * ROLES_PITCH + (tr0 ^ 32 * mt);
              acc[mt] = mfma16<T>(read_pieces_tr(p, p + 2048), x[kc], acc[mt]);
            }
        };
        product(w, b, u);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float hv[4], gv[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) act_both<ACT>(acc[mt][r], hv[r], gv[r]);
          t[mt >> 1].w[2 * (mt & 1)] = pack2<T>(hv[0], hv[1]);
          t[mt >> 1].w[2 * (mt & 1) + 1] = pack2<T>(hv[2], hv[3]);
          gate[mt >> 1].w[2 * (mt & 1)] = pack2<T>(gv[0], gv[1]);
          gate[mt >> 1].w[2 * (mt & 1) + 1] = pack2<T>(gv[2], gv[3]);
        }
        sections.room(lane);
        park(d, 0, 0);
        park(t, 0, 1);
        sections.parked(wave);
        between(0);
        product(w + MATRIX, b + 64, t);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          uint32_t* q = &v[mt >> 1].w[2 * (mt & 1)];
          const uint32_t lo = q[0], hi = q[1];
          q[0] = pack2<T>(unpack_lo<T>(lo) - acc[mt][0], unpack_hi<T>(lo) - acc[mt][1]);
          q[1] = pack2<T>(unpack_lo<T>(hi) - acc[mt][2], unpack_hi<T>(hi) - acc[mt][3]);
        }
        product_tr(w + MATRIX, d);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          gate_apply<T, false>(acc[mt], gate[mt >> 1].w[2 * (mt & 1)], gate[mt >> 1].w[2 * (mt & 1) + 1], dz[mt >> 1].w[2 * (mt & 1)],
                               dz[mt >> 1].w[2 * (mt & 1) + 1]);
        sections.room(lane);
        park(dz, 1, 0);
        park(u, 1, 1);
        sections.parked(wave);
        between(1);
        product_tr(w, dz);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          uint32_t* q = &e[mt >> 1].w[2 * (mt & 1)];
          const uint32_t lo = q[0], hi = q[1];
          q[0] = pack2<T>(unpack_lo<T>(lo) + acc[mt][0], unpack_hi<T>(lo) + acc[mt][1]);
          q[1] = pack2<T>(unpack_lo<T>(hi) + acc[mt][2], unpack_hi<T>(hi) + acc[mt][3]);
        }
      };
      Frag n1[KC], n2[KC], e1[KC], e2[KC];  // the next round's rows
      load_half(n1, e2, false, row0);
      load_half(n2, e1, true, row0);
      for (int64_t round = 0; round < rounds; ++round) {
        const int64_t r = row0 + round * per_round;
        const bool there = r < fresh_rev_args()->rows;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          y1[kc] = n1[kc];
          y2[kc] = n2[kc];
          d1[kc] = e1[kc];
          d2[kc] = e2[kc];
          if (!there || 32 * kc + 8 * g >= fresh_rev_args()->half)
            y1[kc].u = y2[kc].u = d1[kc].u = d2[kc].u = make_uint4(0u, 0u, 0u, 0u);
        }
        // A wave's sixteen accesses to its rows keep the CU's address unit busy for 1000 clocks, and issued together the waves stand still for
        // them; so they are spread over the round (2^20 rows without an activation: 787 -> 697 us).
#pragma unroll 1
        for (int c = count - 1; c >= 0; --c) {
          const char* w = weights + c * 4 * MATRIX;
          const float* b = there ? bias + c * 4 * 64 : no_bias;
          // G: y2 becomes x2, d1 the gradient of x1
          sub(w + 2 * MATRIX, b + 2 * 64, y1, d2, y2, d1, [&](int s) {
            if (c != count - 1) return;
            if (s == 0) load_half(n1, e2, false, r + per_round);
            else load_half(n2, e1, true, r + per_round);
          });
          // F: y1 becomes x1, d2 the gradient of x2
          sub(w, b, y2, d1, y1, d2, [&](int s) {
            if (c == 0 && s == 0) store_half(y2, d1, true, r);
          });
        }
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          arrived(n1[kc]);
          arrived(n2[kc]);
          arrived(e1[kc]);
          arrived(e2[kc]);
        }
        store_half(y1, d2, false, r);
      }
    } else {
      // ------------------------------------------------------------------ gradient waves
      const int qm = ((wave - CW) >> 1) & 1, qn = (wave - CW) & 1;  // tile rows qm, qm + 2 and tile columns qn, qn + 2 of every dW
      // A wave begins with tile row qm + 2 qn, and has its bias sums; the other row's belong to the wave with the same qm.
      // coupling j counts from the top; sections in the order of the chain: G.w2, G.w1, F.w2, F.w1
      f32x4_t dw[CPL][4][TW][TW];
      float db[CPL][4];
#pragma unroll
      for (int j = 0; j < CPL; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          db[j][s] = 0.0f;
#pragma unroll
          for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int k = 0; k < TW; ++k) dw[j][s][i][k] = zero4;
        }
      const int trm = tr0 ^ (qm << 5) ^ (TW == 2 ? qn << 6 : 0);
      const char* pd0 = lds_base(areas + trm);
      const char* pd1 = lds_base(areas + (trm ^ 64));
      const char* ph0 = lds_base(areas + PANEL + (tr0 ^ (qn << 5)));
      const char* ph1 = lds_base(areas + PANEL + (tr0 ^ (qn << 5) ^ 64));
      auto operand = [&](const char* p) { return read_pieces_tr(p, p + 2048); };
      for (int64_t round = 0; round < rounds; ++round)
        each_layer<CPL>([&](auto step) {
          constexpr int j = decltype(step)::value;
          if (j >= opaque(count)) return;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            sections.begin(lane);
            const int o = (s & 1) * AREA;
#pragma unroll
            for (int q = 0; q < ROWS / 32; ++q) {
              __builtin_amdgcn_sched_barrier(0);  // (no registers for two chunks' operands at once)
              Frag hb[TW], da[TW];
#pragma unroll
              for (int k = 0; k < TW; ++k) hb[k] = operand((k == 0 ? ph0 : ph1) + o + q * 4096);
#pragma unroll
              for (int i = 0; i < TW; ++i) da[i] = operand((i == 0 ? pd0 : pd1) + o + q * 4096);
#pragma unroll
              for (int i = 0; i < TW; ++i)
#pragma unroll
                for (int k = 0; k < TW; ++k) dw[j][s][i][k] = mfma16<T>(da[i], hb[k], dw[j][s][i][k]);
#pragma unroll
              for (int p = 0; p < 4; ++p) db[j][s] = dot2_ones<T>(da[0].w[p], db[j][s]);
            }
            sections.done(wave);
          }
        });
      // to this workgroup's slot, or into the accumulators
      each_layer<CPL>([&](auto step) {
        constexpr int j = decltype(step)::value;
        if (j >= opaque(count)) return;
        const RevArgsPtr a = fresh_rev_args();
        const int kb = top - 1 - j, H = a->half, lane = fresh_lane(), n = lane & 15, g = lane >> 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int m = 3 - s;  // F.w1, F.w2, G.w1, G.w2
          const bool second = m & 1;
          float sum = db[j][s];
          sum += lane_xor(sum, lane, 16);
          sum += lane_xor(sum, lane, 32);
#pragma unroll
          for (int i = 0; i < TW; ++i) {
            const bool sums = TW == 2 ? i == 0 : qn == 0;
            const int ti = TW == 2 ? qm + 2 * (qn ^ i) : qm;
            if (a->slots != nullptr) {
              float* slot = a->slots + blockIdx.x * a->slot_stride + (size_t)kb * RevSlot<HP>::FLOATS;
#pragma unroll
              for (int k = 0; k < TW; ++k)
                *reinterpret_cast<f32x4_t*>(slot + (((ti * MT + qn + 2 * k) * 4 + m) * 64 + lane) * 4) = dw[j][s][i][k];
              if (sums && lane < 16) slot[RevSlot<HP>::TILES * 256 + 64 * ti + 16 * m + lane] = sum;
            } else {
              // first layers have their columns in wide order, second layers their rows
              const size_t sub = 2 * kb + (m >> 1);
              float* dst = (second ? a->dw2 : a->dw1) + sub * H * H;
              const int r0 = second ? wide_feature(ti, 4 * g) : 16 * ti + 4 * g;
#pragma unroll
              for (int k = 0; k < TW; ++k) {
                const int tk = qn + 2 * k, c = second ? 16 * tk + n : wide_feature(tk, n);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  if (c < H && r0 + r < H) unsafeAtomicAdd(dst + (size_t)(r0 + r) * H + c, dw[j][s][i][k][r]);
              }
              float* b = second ? a->db2 : a->db1;
              const int f = second ? wide_feature(ti, n) : 16 * ti + n;
              if (b != nullptr && sums && lane < 16 && f < H) unsafeAtomicAdd(b + sub * H + f, sum);
            }
          }
        }
      });
    }
    __syncthreads();  // the weights and the areas are written again
  }
}

// The slots of all workgroups in a fixed order, to where the gradients belong: SUM_PIECES pieces of four values per workgroup, SUM_RUNS
// interleaved runs over the slots, then a fixed tree.  With 64 pieces and 16 runs the 32-wide gradients were 17 workgroups per coupling;
// this is four times as many (four couplings of 256 slots: 32-wide, 17 MB, 9.2 -> 7.1 us; 64-wide, 68 MB, 13.3 -> 12.3 us).
struct RevGrads {
  void *dw1, *db1, *dw2, *db2;
  int half, n_slots, type;
};
constexpr int SUM_PIECES = 16, SUM_RUNS = 64;
template <int HP>
__global__ __launch_bounds__(SUM_PIECES* SUM_RUNS) void rev_sum_k(const float* slots, int64_t slot_stride, RevGrads o) {
  typedef RevSlot<HP> S;
  static_assert(S::FLOATS % (4 * SUM_PIECES) == 0, "whole workgroups");
  __shared__ f32x4_t part[SUM_RUNS][SUM_PIECES];
  const int tx = threadIdx.x % SUM_PIECES, ty = threadIdx.x / SUM_PIECES, H = o.half;
  const int coupling = blockIdx.y, piece = blockIdx.x * SUM_PIECES + tx;
  const float* src = slots + (int64_t)coupling * S::FLOATS + piece * 4;
  f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
  int sl = ty;
  for (; sl + 3 * SUM_RUNS < o.n_slots; sl += 4 * SUM_RUNS) {
    f32x4_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4_t*>(src + (int64_t)(sl + SUM_RUNS * k) * slot_stride);
#pragma unroll
    for (int k = 0; k < 4; ++k) sum += v[k];
  }
  for (; sl < o.n_slots; sl += SUM_RUNS) sum += *reinterpret_cast<const f32x4_t*>(src + (int64_t)sl * slot_stride);
  part[ty][tx] = sum;
  __syncthreads();
  if (threadIdx.x >= 64) return;
  // the first wave: four lanes of a piece take sixteen runs each
  f32x4_t total = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < SUM_RUNS / 4; q += 4) {
    const int r = ty * (SUM_RUNS / 4) + q;
    total += (part[r][tx] + part[r + 1][tx]) + (part[r + 2][tx] + part[r + 3][tx]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    total[r] += __shfl_xor(total[r], 16);
    total[r] += __shfl_xor(total[r], 32);
  }
  if (ty != 0) return;
  auto put = [&](void* base, int64_t at, float v) {
    if (o.type == NF_F32) reinterpret_cast<float*>(base)[at] = v;
    else if (o.type == NF_F16) reinterpret_cast<uint16_t*>(base)[at] = F16::from_f32(v);
    else reinterpret_cast<uint16_t*>(base)[at] = BF16::from_f32(v);
  };
  if (piece < S::TILES * 64) {
    const int lane = piece & 63, tile = piece >> 6, m = tile & 3, mt = (tile >> 2) / S::MT, nt = (tile >> 2) % S::MT;
    // first layers have their columns in wide order, second layers their rows
    const int c = m & 1 ? 16 * nt + (lane & 15) : wide_feature(nt, lane & 15);
    const int r0 = m & 1 ? wide_feature(mt, 4 * (lane >> 4)) : 16 * mt + 4 * (lane >> 4);
    void* base = m & 1 ? o.dw2 : o.dw1;
    if (c >= H) return;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r0 + r < H) put(base, ((int64_t)(2 * coupling + (m >> 1)) * H + r0 + r) * H + c, total[r]);
  } else {
    const int at = piece * 4 - S::TILES * 256, m = (at >> 4) & 3, mt = at >> 6;
    void* base = m & 1 ? o.db2 : o.db1;
    if (base == nullptr) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = (at & 15) + r, f = m & 1 ? wide_feature(mt, n) : 16 * mt + n;
      if (f < H) put(base, (int64_t)(2 * coupling + (m >> 1)) * H + f, total[r]);
    }
  }
}

// Chain waves of a workgroup, and the workgroups.  With more rows than four chain waves per unit take in one round, eight hide each other's
// latencies (four 64-wide couplings, us, four / eight chain waves: 1000 rows 35 / 45, 16384 54 / 54, 30000 67 / 65, 2^18 289 / 260).
struct RevPlan {
  int cw;
  int64_t blocks;
};
static RevPlan rev_plan(int64_t rows) {
  RevPlan p = {rows > 64 * (int64_t)rev_cus() ? 8 : 4, 0};
  const int64_t n = 16 * p.cw, total = (rows + n - 1) / n, cap = rev_cus();
  const int64_t rounds = (total + cap - 1) / cap;  // every workgroup takes this many or one less
  p.blocks = (total + rounds - 1) / rounds;
  return p;
}

size_t rev_bwd_bytes(int64_t rows, int half, int blocks) {
  const size_t slot = half <= 32 ? RevSlot<32>::FLOATS : RevSlot<64>::FLOATS;
  return (size_t)rev_plan(rows).blocks * blocks * slot * sizeof(float);
}

template <typename T, int HP, int ACT>
static int launch_rev_bwd(const RevBwdArgs& a, const RevPlan& p, hipStream_t s) {
  const void* kern = p.cw == 8 ? (const void*)rev_bwd_k<T, HP, ACT, 8, 3> : (const void*)rev_bwd_k<T, HP, ACT, 4, 2>;
  const size_t lds = rev_bwd_lds(HP, p.cw);
  const hipError_t ea = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (ea != hipSuccess) return fail((int)ea, "hipFuncSetAttribute: %s", hipGetErrorString(ea));
  void* args[] = {(void*)&a};
  const hipError_t e = hipLaunchKernel(kern, dim3((unsigned)p.blocks), dim3(64 * (p.cw + 4)), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(rev_bwd): %s", hipGetErrorString(e));
  return check_launch("rev_bwd");
}

template <typename T, int HP>
static int rev_bwd_run(const RevBwdCall& c, hipStream_t s) {
  const auto vec16 = [&](const void* p, int64_t stride) { return (uintptr_t)p % 16 == 0 && stride % 8 == 0 && c.half % 8 == 0; };
  const RevPlan plan = rev_plan(c.rows);
  RevBwdArgs a = {};
  a.in = c.y; a.in_stride = c.y_stride; a.dy = c.dy; a.dy_stride = c.dy_stride;
  a.out = c.x_rec; a.out_stride = c.x_stride; a.dx = c.dx; a.dx_stride = c.dx_stride;
  a.rows = c.rows;
  a.w1 = c.w1; a.b1 = c.b1; a.w2 = c.w2; a.b2 = c.b2;
  a.half = c.half; a.nblocks = c.blocks;
  a.vec_below = vec16(a.out, a.out_stride) && vec16(a.dx, a.dx_stride);
  a.vec_top = vec16(a.in, a.in_stride) && vec16(a.dy, a.dy_stride);
  a.slots = (float*)c.workspace;
  a.slot_stride = (int64_t)c.blocks * RevSlot<HP>::FLOATS;
  if (c.workspace == nullptr) {
    a.dw1 = (float*)c.dw1; a.db1 = (float*)c.db1; a.dw2 = (float*)c.dw2; a.db2 = (float*)c.db2;
  }
  int rc;
  switch (c.act) {
    case NF_ACT_GELU: rc = launch_rev_bwd<T, HP, NF_ACT_GELU>(a, plan, s); break;
    case NF_ACT_SILU: rc = launch_rev_bwd<T, HP, NF_ACT_SILU>(a, plan, s); break;
    case NF_ACT_RELU: rc = launch_rev_bwd<T, HP, NF_ACT_RELU>(a, plan, s); break;
    case NF_ACT_RELU2: rc = launch_rev_bwd<T, HP, NF_ACT_RELU2>(a, plan, s); break;
    default: rc = launch_rev_bwd<T, HP, NF_ACT_NONE>(a, plan, s); break;
  }
  if (rc != 0 || c.workspace == nullptr) return rc;
  const RevGrads grads = {c.dw1, c.db1, c.dw2, c.db2, c.half, (int)plan.blocks, c.type};
  hipLaunchKernelGGL((rev_sum_k<HP>), dim3(RevSlot<HP>::FLOATS / 4 / SUM_PIECES, (unsigned)c.blocks), dim3(SUM_PIECES * SUM_RUNS), 0, s, a.slots,
                     a.slot_stride, grads);
  return check_launch("rev_sum");
}

int rev_bwd(const RevBwdCall& c, int dtype, hipStream_t s) {
  if (c.half <= 32) return dtype == NF_BF16 ? rev_bwd_run<BF16, 32>(c, s) : rev_bwd_run<F16, 32>(c, s);
  return dtype == NF_BF16 ? rev_bwd_run<BF16, 64>(c, s) : rev_bwd_run<F16, 64>(c, s);
}

}  // namespace nf
