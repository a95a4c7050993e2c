// Backward of a whole network in one launch: 16-bit tensors, any activation, one to nine hidden layers of width 16 .. 64,
// any input and output width up to 64, rows of any alignment.  Weight gradients leave through one slot per workgroup.
//
// A workgroup is eight, twelve or sixteen waves, split by role (a wave's vector instructions do not start while one of its own
// matrix products is in flight, so the two units of a SIMD overlap across waves only):
//   * four, eight or twelve chain waves own 16 rows of a round each.  A chain wave recomputes the forward with every layer's activations
//     left in its registers (and, but for ReLU, the activation's derivative beside them), carries the gradient back
//     through the layers, and per layer parks the two operands of dW = dz^T h in LDS, row-major;
//   * four gradient waves own every other tile row and every other tile column of every layer's dW each and keep
//     them in registers over the whole launch (160 of a wave's 256 at nine 64-wide hidden layers).  They read the parked
//     operands back with the rows along K (ds_read_b64_tr_b16) while the chain waves work on the layer below.
// The roles hand a layer over at one barrier (four chain waves) or by flags in LDS (more of them); the parked operands have two areas used
// in turn, so an area is written again when its readers are a layer further.  No tile is owned twice, so nothing is summed across waves at the end.
//
// LDS holds one copy of the weights, row-major in rows of 128 bytes: a product with W reads its fragments as rows, a
// product with W^T reads the same bytes through the transposing reads, so ten 64-wide layers and the operand areas fit
// 150 KB and the staging is a plain copy (role_split.h).
//
// What it replaces for most calls is up to five layers per launch, a replayed forward between launches, dW through LDS
// transposes of 2-byte stores or matrix-core transposes, and atomics of all workgroups into cleared sums that a cast kernel
// rounds.  Backward through autograd's host side, bfloat16, us before -> now at 2^11 / 2^16 / 2^18 rows: 64 -> 64 x 9 -> 64
// ReLU 91 -> 20 / 168 -> 55 / 269 -> 145, 32 -> 64 x 4 -> 16 SiLU 47 -> 14 / 81 -> 39 / 168 -> 101, 35 -> 64 x 2 -> 3 ReLU
// 20 -> 11 / 48 -> 22 / 76 -> 45, 32 -> 32 x 2 -> 16 ReLU 15 -> 10 / 31 -> 15 / 42 -> 26.
// What bounds it: up to 2^16 rows the weights' staging, one chain of dependent layers per round and the slots (170 KB a
// workgroup at nine layers): there its waves wait in 54 % of their clocks, LDS is busy 31 %, vector issue 27 %, the matrix cores 16 % (64 ->
// 64 x 9 -> 64, 2^16 rows).  With many rows LDS (48 % busy with four layers and 2^18 rows, vector issue 40 %, matrix cores 23 %; weight
// fragments are read once per 16 rows, as two tiles a wave need more registers than are left), and the rows' accesses at
// one lane a clock.  Measured without the gradient waves' products it is 5 - 10 % quicker.  The nine-layer ReLU form has no register to spare:
// its time moves by up to 5 % with what the allocation makes of any change to its source.
#pragma once

#include "fused_mlp_bwd2_kernels.h"
#include "role_split.h"

namespace nf {

constexpr int ROLES_MAX_DEPTH = 9;               // hidden layers (MlpArgs::depth) of one launch
// hidden layers of the kernels that leave registers for more waves (but for ReLU a layer's derivatives take as much room as its activations)
constexpr int roles_shallow(int act) { return act == NF_ACT_RELU ? 4 : 3; }
// A layer in a slot: the 16 x 16 tiles of its dW (hidden width 64: 4 x 4; narrower: 2 x 4, the output layer's 4 x 2; whether it has them all or not),
// then its bias sums in the place of another tile.  Nine layers are 44 MB (256 workgroups), narrow ones 47 MB (512).
constexpr int roles_tiles(int hp) { return hp == 64 ? 16 : 8; }
constexpr int roles_columns_log2(int hp, bool output) { return hp == 64 || !output ? 2 : 1; }  // tiles of a tile row
constexpr int roles_layer_floats(int hp) { return (roles_tiles(hp) + 1) * 256; }
constexpr int roles_slot_floats(int hp, int depth) { return (depth + 1) * roles_layer_floats(hp); }
constexpr size_t roles_lds(int hp, int depth, int rows) {
  return (size_t)(depth * hp + 64) * ROLES_PITCH + (size_t)depth * 64 * 4 + (size_t)4 * rows * ROLES_PITCH + 32 * 4;
}
static_assert(roles_lds(64, ROLES_MAX_DEPTH, 64) <= 160 * 1024, "LDS budget");

// rows of `w` [layers * nr][nc] (row-contiguous) -> LDS rows of 128 bytes, swizzled; layer l's rows start at LDS row l * pad, rows
// nr .. pad - 1 and columns nc .. 63 are zero
template <int N>
__device__ __forceinline__ void stage_rows(char* dst, const uint16_t* w, int layers, int nr, int pad, int nc, int tid) {
  const bool vec = nc % 4 == 0 && (uintptr_t)w % 8 == 0;
  const int pad_log2 = pad == 32 ? 5 : 6;
  const int units = layers * pad * 16;
  constexpr int DEEP = 8;  // loads in flight per thread
  for (int u0 = tid; u0 < units; u0 += N * DEEP) {
    uint2 v[DEEP];
#pragma unroll
    for (int i = 0; i < DEEP; ++i) {
      const int u = u0 + i * N, row = u >> 4, c = 4 * (u & 15), l = row >> pad_log2, r = row & (pad - 1);
      v[i] = make_uint2(0u, 0u);
      if (u < units && r < nr && c < nc) {
        const uint16_t* p = w + ((size_t)l * nr + r) * nc + c;
        if (vec) {
          v[i] = *reinterpret_cast<const uint2*>(p);
        } else {
          uint16_t t[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] = c + j < nc ? p[j] : (uint16_t)0;
          v[i].x = (uint32_t)t[0] | ((uint32_t)t[1] << 16);
          v[i].y = (uint32_t)t[2] | ((uint32_t)t[3] << 16);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < DEEP; ++i) {
      const int u = u0 + i * N, row = u >> 4;
      if (u < units) *reinterpret_cast<uint2*>(dst + row * ROLES_PITCH + (((u & 15) ^ swizzle(row)) << 3)) = v[i];
    }
  }
}

// Whether the matrices come in 16-byte pieces.  64-wide kernels are compiled for either, narrow ones for both: with the other way of staging in it a 64-wide
// kernel takes longer over its rows, and a narrow one is allocated the better for it (us, forward and backward, 2^20 rows, both ways in one / one each: 16 -> 64
// -> 20 ReLU 104.9 / 101.3, 32 -> 64 -> 20 107.2 / 103.3, 32 -> 64 x 4 -> 16 205.6 / 201.9; 64 -> 64 x 9 -> 64, 2^16 off 16 bytes 69.2 / 68.0; but 32 -> 32 -> 33 121.7 / 126.8).
enum class WholePieces { NO, YES, ANY };
__host__ __device__ __forceinline__ bool whole_pieces(const MlpArgs& a) {
  return a.d_in % 8 == 0 && a.d_hidden % 8 == 0 && ((uintptr_t)a.w_in | (uintptr_t)a.w_hid | (uintptr_t)a.w_out) % 16 == 0;
}

// All matrices and hidden biases of a network as one list of 16-byte pieces, laid out as stage_rows() does, with several of a thread's under way
// together and first_rows(), which asks for the wave's first rows, behind them.  The biases are asked for first.  Matrix by matrix in 8-byte pieces, a
// clock each for the L1, each waited for the one in front and all for the rows (us with the sum of the gradients, before / this: 32 -> 64 -> 64 -> 16
// 1000 rows 9.8 / 9.2, 2^16 19.5 / 18.7; 64 -> 64 x 8 -> 64, 2^16 51 / 47.6; three layers of SiLU, 2^18 69.2 / 67.1).
// WHOLE: whether the matrices are such pieces (else they are staged one by one behind the rows), or ANY for both ways in one kernel.
template <typename T, int HP, int N, WholePieces WHOLE, typename FirstRows>
__device__ __forceinline__ void stage_pieces(char* dst, float* bias, const MlpArgs& a, int tid, FirstRows first_rows) {
  constexpr int AT_ONCE = 6, HP_LOG2 = HP == 32 ? 5 : 6;
  const bool pieces = WHOLE == WholePieces::ANY ? whole_pieces(a) : WHOLE == WholePieces::YES;
  const int lane = tid & 63, first = __builtin_amdgcn_readfirstlane(tid - lane), H = a.d_hidden, units = pieces ? (a.depth * HP + 64) * 8 : 0;
  const auto bias_at = [&](int i, bool& there) {
    const int l = i >> 6, f = i & 63;
    const uint16_t* b = l == 0 ? a.b_in : a.b_hid != nullptr ? a.b_hid + (size_t)(l - 1) * H : nullptr;
    there = b != nullptr && f < H;
    return there ? b + f : a.w_in;
  };
  bool there;
  const uint16_t b0 = *bias_at(tid < a.depth * 64 ? tid : 0, there);
  for (int u0 = first; u0 < units || u0 == first; u0 += N * AT_ONCE) {  // (a wave's pieces are eight rows of one matrix)
    uint4 v[AT_ONCE];
    bool inside[AT_ONCE];
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      const int u = u0 + i * N;
      if (u >= units) break;
      const int row = (u >> 3) + (lane >> 3), c = 8 * (lane & 7), l = u >> (3 + HP_LOG2);  // l == depth and on: the output's 64 rows
      const bool out = l >= a.depth;
      const int r = out ? row - a.depth * HP : row & (HP - 1), nr = out ? a.d_out : H, nc = l == 0 ? a.d_in : H;
      const uint16_t* w = out ? a.w_out : l == 0 ? a.w_in : a.w_hid + (size_t)(l - 1) * H * H;
      inside[i] = r < nr && c < nc;
      v[i] = *reinterpret_cast<const uint4*>(w + (r < nr ? r : 0) * nc + (c < nc ? c : 0));
    }
    if (u0 == first) first_rows();
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      const int u = u0 + i * N;
      if (u >= units) break;
      const int row = (u >> 3) + (lane >> 3);
      if (!inside[i]) v[i] = make_uint4(0u, 0u, 0u, 0u);
      char* d = dst + row * ROLES_PITCH;
      *reinterpret_cast<uint2*>(d + (((2 * (lane & 7)) ^ swizzle(row)) << 3)) = make_uint2(v[i].x, v[i].y);
      *reinterpret_cast<uint2*>(d + (((2 * (lane & 7) + 1) ^ swizzle(row)) << 3)) = make_uint2(v[i].z, v[i].w);
    }
  }
  if (tid < a.depth * 64) bias[tid] = there ? T::to_f32(b0) : 0.0f;
  for (int i = tid + N; i < a.depth * 64; i += N) {
    const uint16_t b = *bias_at(i, there);
    bias[i] = there ? T::to_f32(b) : 0.0f;
  }
  if (pieces) return;
  stage_rows<N>(dst, a.w_in, 1, H, HP, a.d_in, tid);
  if (a.depth > 1) stage_rows<N>(dst + HP * ROLES_PITCH, a.w_hid, a.depth - 1, H, HP, H, tid);
  stage_rows<N>(dst + a.depth * HP * ROLES_PITCH, a.w_out, 1, a.d_out, 64, H, tid);
}

// The launch's arguments, read again where they are used (see opaque()).
typedef const MlpArgs __attribute__((address_space(4))) * ArgsPtr;
__device__ __forceinline__ ArgsPtr fresh_args() {
  ArgsPtr p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// MAXD: most hidden layers (fewer leave registers for more waves); CW: chain waves; OCC: waves per SIMD the kernel is compiled for; WHOLE: see stage_pieces().
template <typename T, int HP, int ACT, int MAXD, int CW, int OCC, WholePieces WHOLE>
__global__ __launch_bounds__(64 * (CW + 4), OCC) void mlp_bwd_roles_k(MlpArgs a) {
  constexpr int MT = HP / 16, KC = HP / 32, ROWS = 16 * CW, THREADS = 64 * (CW + 4);  // rows of a round
  constexpr bool RELU = ACT == NF_ACT_RELU;
  constexpr int TW = HP == 64 ? 2 : 1;  // tile rows / columns of a hidden layer's dW that a gradient wave owns
  extern __shared__ __align__(16) char roles_smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int depth = a.depth;

  char* w_in = roles_smem;                                     // [HP][128]
  char* w_hid = w_in + HP * ROLES_PITCH;                       // [depth - 1][HP][128]
  char* w_out = w_hid + (size_t)(depth - 1) * HP * ROLES_PITCH;  // [64][128]
  float* bias = reinterpret_cast<float*>(w_out + 64 * ROLES_PITCH);  // [depth][64]
  char* areas = reinterpret_cast<char*>(bias + depth * 64);    // [2][dz rows | input rows][ROWS][128]
  constexpr int PANEL = ROWS * ROLES_PITCH, AREA = 2 * PANEL;
  Sections<CW> sections = {reinterpret_cast<int*>(areas + 2 * AREA), 0};
  if (tid < 32) sections.flags[tid] = 0;

  const int64_t rounds = (a.rows + (int64_t)gridDim.x * ROWS - 1) / ((int64_t)gridDim.x * ROWS);
  const bool chain = wave < CW;
  const bool two_in = a.d_in > 32, two_out = a.d_out > 32;

  const int64_t row0 = (int64_t)blockIdx.x * ROWS + wave * 16 + n;  // a lane's row of the first round
  Frag nx[2], ndy[2];  // the next round's rows, lane group g columns 32 kc + 8 g .. (natural order)
  auto load_rows = [&](int64_t r) {
    const ArgsPtr k = fresh_args();
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      nx[kc].u = ndy[kc].u = make_uint4(0u, 0u, 0u, 0u);
      if (kc == 0 || two_in) nx[kc] = load_row8(k->x, k->x_stride, r, k->rows, k->d_in, 32 * kc + 8 * g, k->x_vec != 0);
      if (kc == 0 || two_out) ndy[kc] = load_row8(k->dy, k->dy_stride, r, k->rows, k->d_out, 32 * kc + 8 * g, k->dy_vec != 0);
    }
  };
  stage_pieces<T, HP, THREADS, WHOLE>(w_in, bias, a, tid, [&] {
    if (chain) load_rows(row0);
  });
  __syncthreads();

  const int chain0 = chain_offset(n, g), nat0 = natural_offset(n, g), tr0 = tr_offset(n, g);
  const f32x4_t zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  int area = 0;

  if (chain) {
    // ------------------------------------------------------------------ chain waves
    char* mine = areas + wave * 16 * ROLES_PITCH;  // this wave's rows of the first area
    // an operand of a layer's dW: panel 0 its dz (or dy) rows, panel 1 its input rows
    auto park = [&](const Frag (&f)[2], int panel, bool natural, bool two) {
      char* p = mine + area * AREA + panel * PANEL;
      const int o0 = natural ? nat0 : chain0, o1 = natural ? nat0 ^ 8 : chain0 ^ 32;
      write_pieces(p + o0, p + o1, f[0]);
      if (two) write_pieces(p + (o0 ^ 64), p + (o1 ^ 64), f[1]);
    };
    auto room = [&] { sections.room(lane); };
    auto announce = [&] {
      sections.parked(wave);
      area ^= 1;
    };
    for (int64_t round = 0; round < rounds; ++round) {
      const int64_t r = row0 + round * gridDim.x * ROWS;
      Frag h[MAXD][2], gate[RELU ? 1 : MAXD][2], x[2], cur[2], dz[2];  // h[0]: the last hidden layer
      f32x4_t acc[4];
      const ArgsPtr k = fresh_args();
      if (r >= k->rows) {  // past the batch's end x's last row again (REPEAT of load_rows_frag()).  Asked for ahead like the others it cost 4 % of nine layers
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
          if (kc == 0 || two_in) nx[kc] = load_row8(k->x, k->x_stride, k->rows - 1, k->rows, k->d_in, 32 * kc + 8 * g, k->x_vec != 0);
      }
      const bool convert = k->x_conv != 0;
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        x[kc] = convert ? convert_frag(nx[kc], T::code == NF_BF16 ? 1 : 2) : nx[kc];
        if constexpr (HP == 64) x[kc] = nat_to_chain(x[kc]);  // (narrow networks: natural order; each as the kernels of nf_mlp_bwd)
        dz[kc] = nat_to_chain(ndy[kc]);
        cur[kc] = x[kc];
      }
      // acc = b + W cur of linear layer l
      auto layer = [&](int l, bool natural) {
        const char* w = l == 0 ? w_in : w_hid + (l - 1) * HP * ROLES_PITCH;
        const int o0 = natural ? nat0 : chain0, o1 = natural ? nat0 ^ 8 : chain0 ^ 32;
        const float* b = bias + l * 64 + 4 * g;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = *reinterpret_cast<const f32x4_t*>(b + 16 * mt);
        auto chunk = [&](int kc) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma16<T>(read_pieces(w + mt * 2048 + (o0 ^ 64 * kc), w + mt * 2048 + (o1 ^ 64 * kc)), cur[kc], acc[mt]);
        };
        chunk(0);
        if (KC == 2 || (l == 0 && two_in)) chunk(1);
      };
      // ---- forward ----
      // ReLU at 64 wide with more than five linear layers: nf_mlp_bwd runs these as two launches, the second one behind a
      // replay by the forward kernel, whose layer 0 takes x in natural order; a unit within rounding of zero opens or closes
      // with the order of a sum.  To give the same gradients the layers behind the boundary are computed from a second run
      // over the first `split` hidden layers.
      constexpr bool SPLIT = RELU && HP == 64 && MAXD > 4;
      const int split = SPLIT && a.handover != 0 ? __builtin_ctz(a.handover) : depth;
      int hi = depth, lo = depth - split;
#pragma unroll 1
      for (;;) {
        each_layer<MAXD>([&](auto step) {
          constexpr int j = MAXD - 1 - decltype(step)::value;
          const int l = opaque(a.depth) - 1 - j;  // the linear layer in front of hidden layer j
          if (SPLIT ? j >= opaque(hi) || j < opaque(lo) : l < 0) return;
          layer(l, HP == 32 && l == 0);
          const bool handover = (a.handover >> l) & 1;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            uint32_t p01 = 0u, p23 = 0u;
            if constexpr (RELU) {
              p01 = relu_pk(pack2<T>(acc[mt][0], acc[mt][1]));
              p23 = relu_pk(pack2<T>(acc[mt][2], acc[mt][3]));
            } else {
              if (handover) {
                p01 = pack2<T>(acc[mt][0], acc[mt][1]);
                p23 = pack2<T>(acc[mt][2], acc[mt][3]);
                acc[mt] = f32x4_t{unpack_lo<T>(p01), unpack_hi<T>(p01), unpack_lo<T>(p23), unpack_hi<T>(p23)};
              }
              uint32_t g01 = p01, g23 = p23;
              act_pack<T, false>(acc[mt], ACT, p01, p23);
              if (!handover) gate_pack<T, false>(acc[mt], ACT, p01, p23, g01, g23);
              gate[j][mt >> 1].w[2 * (mt & 1)] = g01;  // behind a handover: the pre-activation itself
              gate[j][mt >> 1].w[2 * (mt & 1) + 1] = g23;
            }
            h[j][mt >> 1].w[2 * (mt & 1)] = p01;
            h[j][mt >> 1].w[2 * (mt & 1) + 1] = p23;
          }
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) cur[kc] = h[j][kc];
        });
        if (!SPLIT || lo == 0) break;
        hi = lo;
        lo = 0;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) cur[kc] = chain_to_nat(x[kc]);
#pragma unroll 1
        for (int l = 0; l < split; ++l) {
          layer(l, l == 0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            cur[mt >> 1].w[2 * (mt & 1)] = relu_pk(pack2<T>(acc[mt][0], acc[mt][1]));
            cur[mt >> 1].w[2 * (mt & 1) + 1] = relu_pk(pack2<T>(acc[mt][2], acc[mt][3]));
          }
        }
      }
      // ---- output layer: dW_out = dy^T h, dh = W_out^T dy ----
      room();
      park(dz, 0, false, two_out);
      park(h[0], 1, false, KC == 2);
      announce();
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = zero4;
      auto out_chunk = [&](int kc) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const char* p = w_out + kc * 32 * ROLES_PITCH + (tr0 ^ 32 * mt);
          acc[mt] = mfma16<T>(read_pieces_tr(p, p + 2048), dz[kc], acc[mt]);
        }
      };
      out_chunk(0);
      if (two_out) out_chunk(1);
      // ---- hidden layers, last to first: dz = dh * act'(z), dW = dz^T (input), dh = W^T dz ----
      each_layer<MAXD>([&](auto step) {
        constexpr int j = decltype(step)::value;
        const int depth = opaque(a.depth);
        if (j >= depth) return;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          uint32_t p01, p23;
          if constexpr (RELU) {
            p01 = relu_gate_pk(pack2<T>(acc[mt][0], acc[mt][1]), h[j][mt >> 1].w[2 * (mt & 1)]);
            p23 = relu_gate_pk(pack2<T>(acc[mt][2], acc[mt][3]), h[j][mt >> 1].w[2 * (mt & 1) + 1]);
          } else {
            const uint32_t g01 = gate[j][mt >> 1].w[2 * (mt & 1)], g23 = gate[j][mt >> 1].w[2 * (mt & 1) + 1];
            if ((a.handover >> (depth - 1 - j)) & 1) {
              const f32x4_t v = acc[mt], z = {unpack_lo<T>(g01), unpack_hi<T>(g01), unpack_lo<T>(g23), unpack_hi<T>(g23)};
              p01 = pack2<T>(v[0] * act_grad(z[0], ACT), v[1] * act_grad(z[1], ACT));
              p23 = pack2<T>(v[2] * act_grad(z[2], ACT), v[3] * act_grad(z[3], ACT));
            } else {
              gate_apply<T, false>(acc[mt], g01, g23, p01, p23);
            }
          }
          dz[mt >> 1].w[2 * (mt & 1)] = p01;
          dz[mt >> 1].w[2 * (mt & 1) + 1] = p23;
        }
        if constexpr (j + 1 < MAXD) {
          if (j == depth - 1) return;  // the input layer follows below
          room();
          park(dz, 0, false, KC == 2);
          park(h[j + 1], 1, false, KC == 2);
          announce();
          const char* w = w_hid + (depth - 2 - j) * HP * ROLES_PITCH;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = zero4;
#pragma unroll
          for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              const char* p = w + kc * 32 * ROLES_PITCH + (tr0 ^ 32 * mt);
              acc[mt] = mfma16<T>(read_pieces_tr(p, p + 2048), dz[kc], acc[mt]);
            }
        }
      });
      // ---- input layer: dW_in = dz^T x, dx = W_in^T dz ----
      room();
      park(dz, 0, false, KC == 2);
      park(x, 1, HP == 32, two_in);
      load_rows(r + (int64_t)gridDim.x * ROWS);
      announce();
      const ArgsPtr kx = fresh_args();
      if (kx->dx != nullptr) {
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
          if (kc == 1 && !two_in) continue;
          Frag o;
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            f32x4_t v = zero4;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
              const char* p = w_in + c * 32 * ROLES_PITCH + (tr0 ^ 64 * kc ^ 32 * t);
              v = mfma16<T>(read_pieces_tr(p, p + 2048), dz[c], v);
            }
            typedef typename std::conditional<T::code == NF_BF16, F16, BF16>::type Other;
            o.w[2 * t] = convert ? pack2<Other>(v[0], v[1]) : pack2<T>(v[0], v[1]);
            o.w[2 * t + 1] = convert ? pack2<Other>(v[2], v[3]) : pack2<T>(v[2], v[3]);
          }
          store_row8(kx->dx, kx->dx_stride, r, kx->rows, kx->d_in, 32 * kc + 8 * g, chain_to_nat(o), kx->dx_vec != 0);
        }
      }
    }
    return;
  }
  // -------------------------------------------------------------------- gradient waves
  const int qm = ((wave - CW) >> 1) & 1, qn = (wave - CW) & 1;  // tile rows qm, qm + 2 and tile columns qn, qn + 2 of every dW
  f32x4_t dw_out[2][TW], dw[MAXD][TW][TW], dw_in2 = zero4;  // dw_in2: the input layer's second tile column at HP = 32
  float db_out[2], db[MAXD][TW];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    db_out[i] = 0.0f;
#pragma unroll
    for (int k = 0; k < TW; ++k) dw_out[i][k] = zero4;
  }
#pragma unroll
  for (int j = 0; j < MAXD; ++j)
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      db[j][i] = 0.0f;
#pragma unroll
      for (int k = 0; k < TW; ++k) dw[j][i][k] = zero4;
    }
  const int trm = tr0 ^ (qm << 5), trk = tr0 ^ (qn << 5);
  auto operand = [&](const char* p) { return read_pieces_tr(p, p + 2048); };
  auto done = [&] {
    sections.done(wave);
    area ^= 1;
  };
  for (int64_t round = 0; round < rounds; ++round) {
    // ---- output layer ----
    sections.begin(lane);
    if (16 * qm < a.d_out) {
      const char* pd = areas + area * AREA;
      const char* ph = areas + area * AREA + PANEL;
#pragma unroll
      for (int s = 0; s < ROWS / 32; ++s) {
        Frag hb[TW];
#pragma unroll
        for (int k = 0; k < TW; ++k) hb[k] = operand(ph + s * 4096 + (trk ^ 64 * k));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (i == 1 && !two_out) continue;
          const Frag da = operand(pd + s * 4096 + (trm ^ 64 * i));
#pragma unroll
          for (int k = 0; k < TW; ++k) dw_out[i][k] = mfma16<T>(da, hb[k], dw_out[i][k]);
#pragma unroll
          for (int q = 0; q < 4; ++q) db_out[i] = dot2_ones<T>(da.w[q], db_out[i]);
        }
      }
    }
    done();
    // ---- hidden layers and the input layer (j = depth - 1) ----
    each_layer<MAXD>([&](auto step) {
      constexpr int j = decltype(step)::value;
      const int depth = opaque(a.depth);
      if (j >= depth) return;
      sections.begin(lane);
      const char* pd = areas + area * AREA;
      const char* ph = areas + area * AREA + PANEL;
      // COLS: tile columns of this layer's dW that this wave owns
      auto section = [&](auto cols_c) {
        constexpr int COLS = decltype(cols_c)::value;
#pragma unroll
        for (int s = 0; s < ROWS / 32; ++s) {
          Frag hb[COLS], da[TW];
#pragma unroll
          for (int k = 0; k < COLS; ++k) hb[k] = operand(ph + s * 4096 + (trk ^ 64 * k));
#pragma unroll
          for (int i = 0; i < TW; ++i) da[i] = operand(pd + s * 4096 + (trm ^ 64 * i));
#pragma unroll
          for (int i = 0; i < TW; ++i) {
#pragma unroll
            for (int k = 0; k < COLS; ++k) {
              if constexpr (HP == 32) {
                f32x4_t& v = k == 0 ? dw[j][i][0] : dw_in2;
                v = mfma16<T>(da[i], hb[k], v);
              } else {
                dw[j][i][k] = mfma16<T>(da[i], hb[k], dw[j][i][k]);
              }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) db[j][i] = dot2_ones<T>(da[i].w[q], db[j][i]);
          }
        }
      };
      if (HP == 32 && j == depth - 1 && two_in) section(std::integral_constant<int, 2>{});  // the input layer, wider than the others
      else section(std::integral_constant<int, TW>{});
      done();
    });
  }

  // ---- this workgroup's slot: per layer (input first) tile (mt, nt) as the registers hold it, then the bias sums ----
  float* slot = a.partials + (size_t)blockIdx.x * a.partial_stride;
  auto put = [&](int layer, int mt, int nt, f32x4_t v) {
    const int tile = (mt << roles_columns_log2(HP, layer == depth)) + nt;
    *reinterpret_cast<f32x4_t*>(slot + (size_t)layer * roles_layer_floats(HP) + (tile * 64 + lane) * 4) = v;
  };
  auto put_bias = [&](int layer, int mt, float v) {
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (qn == 0 && lane < 16) slot[(size_t)layer * roles_layer_floats(HP) + roles_tiles(HP) * 256 + 16 * mt + lane] = v;
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (i == 1 && !two_out) continue;
#pragma unroll
    for (int k = 0; k < TW; ++k) put(depth, qm + 2 * i, qn + 2 * k, dw_out[i][k]);
    put_bias(depth, qm + 2 * i, db_out[i]);
  }
  each_layer<MAXD>([&](auto step) {
    constexpr int j = decltype(step)::value;
    const int depth = opaque(a.depth);
    if (j >= depth) return;
    const int layer = depth - 1 - j;
#pragma unroll
    for (int i = 0; i < TW; ++i) {
#pragma unroll
      for (int k = 0; k < TW; ++k) put(layer, qm + 2 * i, qn + 2 * k, dw[j][i][k]);
      put_bias(layer, qm + 2 * i, db[j][i]);
    }
  });
  if constexpr (HP == 32) {
    if (two_in) put(0, qm, qn + 2, dw_in2);
  }
}

}  // namespace nf
