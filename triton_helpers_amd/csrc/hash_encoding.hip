// Multiresolution hash encoding for gfx950: forward gather, backward scatter-add,
// and an index/weight dump used for bit-exact index checks.
//
// Arithmetic contract (follows the PyTorch path of the reference,
// triton_helpers/layers/hash_encoding/kernel.py:448-479):
//   pos   = fp32(x / scale) * fp32(N_l)          one rounding per operation, no FMA
//   cell  = floor(pos),  frac = pos - floor(pos)
//   dense level  ((N_l+1)^D <= T):  row = sum_d (cell_d + bit_d) * N_l^d
//   hashed level:                   row = (xor_d (cell_d + bit_d) * pi_d) mod T_l   (64-bit products)
//   weight_j = prod_d (bit_d ? frac_d : 1 - frac_d),   out = sum_j weight_j * table[row_j]
// The file is compiled with -ffp-contract=off so that none of this is fused.
#include "hash_common.h"

namespace nf {

// ---------------------------------------------------------------------------
// Generic path: one thread per (point, level); any D <= 6, any F, any dtype mix.
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ Cell<D> locate(const void* coords, int cdt, int64_t sn, int64_t sd, int64_t n, float scale,
                                          int res) {
  float x[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    x[d] = load_as_f32(coords, n * sn + d * sd, cdt);
    if (scale != 1.0f) x[d] = x[d] / scale;
  }
  return locate_cell<D>(x, res);
}

template <int D>
__device__ __forceinline__ void load_primes(const int64_t* primes, uint64_t* pi) {
#pragma unroll
  for (int d = 0; d < D; ++d) pi[d] = (uint64_t)primes[d];
}

// V = features per load: rows whose width, base and output allow it are read V features (4, 8 or 16 bytes) at a time,
// every feature summed over the corners in the same order as with V = 1
template <int D, typename TT, int V = 1>
__global__ __launch_bounds__(256) void hash_fwd_generic_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                          const typename TT::storage* table,
                                                          typename TT::storage* out, int64_t out_stride, int64_t N,
                                                          DevGeom g, const int64_t* primes, float scale) {
  typedef typename TT::storage S;
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (n >= N) return;
  uint64_t pi[D];
  load_primes<D>(primes, pi);
  const bool hashed = l >= g.first_hash;
  const Cell<D> cell = locate<D>(coords, cdt, csn, csd, n, scale, g.res[l]);
  const S* tab = table + g.row_offset[l] * g.feat;
  uint64_t rows[1 << D];
  float w[1 << D];
#pragma unroll
  for (int j = 0; j < (1 << D); ++j) {
    rows[j] = corner_row<D>(cell, j, hashed, (uint32_t)g.res[l], g.rows[l], pi);
    w[j] = corner_weight<D>(cell, j);
  }
  if constexpr (V == 1) {
    for (int f = 0; f < g.feat; ++f) {
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < (1 << D); ++j) acc = acc + w[j] * TT::to_f32(tab[rows[j] * g.feat + f]);
      out[n * out_stride + (int64_t)l * g.feat + f] = TT::from_f32(acc);
    }
  } else {
    struct alignas(V * sizeof(S)) Piece { S v[V]; };
    for (int f = 0; f < g.feat; f += V) {
      float acc[V];
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = 0.0f;
      Piece q[1 << D];
#pragma unroll
      for (int j = 0; j < (1 << D); ++j) q[j] = *reinterpret_cast<const Piece*>(tab + rows[j] * g.feat + f);
#pragma unroll
      for (int j = 0; j < (1 << D); ++j)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = acc[e] + w[j] * TT::to_f32(q[j].v[e]);
      Piece r;
#pragma unroll
      for (int e = 0; e < V; ++e) r.v[e] = TT::from_f32(acc[e]);
      *reinterpret_cast<Piece*>(out + n * out_stride + (int64_t)l * g.feat + f) = r;
    }
  }
}

template <int D>
__global__ __launch_bounds__(256) void hash_bwd_generic_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                          const void* dout, int ddt, int64_t dout_stride,
                                                          float* dtable, int64_t N, DevGeom g, const int64_t* primes,
                                                          float scale) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (n >= N) return;
  uint64_t pi[D];
  load_primes<D>(primes, pi);
  const bool hashed = l >= g.first_hash;
  const Cell<D> cell = locate<D>(coords, cdt, csn, csd, n, scale, g.res[l]);
  float* tab = dtable + g.row_offset[l] * g.feat;
  for (int f = 0; f < g.feat; ++f) {
    const float go = load_as_f32(dout, n * dout_stride + (int64_t)l * g.feat + f, ddt);
#pragma unroll
    for (int j = 0; j < (1 << D); ++j) {
      const uint64_t row = corner_row<D>(cell, j, hashed, (uint32_t)g.res[l], g.rows[l], pi);
      unsafeAtomicAdd(tab + row * g.feat + f, corner_weight<D>(cell, j) * go);
    }
  }
}

template <int D>
__global__ __launch_bounds__(256) void hash_indices_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                      int64_t* out_rows, float* out_w, int64_t N, DevGeom g,
                                                      const int64_t* primes, float scale) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (n >= N) return;
  uint64_t pi[D];
  load_primes<D>(primes, pi);
  const bool hashed = l >= g.first_hash;
  const Cell<D> cell = locate<D>(coords, cdt, csn, csd, n, scale, g.res[l]);
  const int64_t base = (n * g.levels + l) * (1 << D);
#pragma unroll
  for (int j = 0; j < (1 << D); ++j) {
    out_rows[base + j] = (int64_t)corner_row<D>(cell, j, hashed, (uint32_t)g.res[l], g.rows[l], pi);
    if (out_w) out_w[base + j] = corner_weight<D>(cell, j);
  }
}

// The same table through the index arithmetic of the fast kernels (sweep, tiled, binned backward): cells from
// cell_index(), rows from rows_d3() / rows_d2() in 32-bit wrap-around arithmetic with the level's mask, weights from
// weights_d3() / weights_d2() -- the very inline functions those kernels call, here with their results written out.
template <int D>
__global__ __launch_bounds__(256) void hash_indices_fast_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                           int64_t* out_rows, float* out_w, int64_t N, DevGeom g,
                                                           const int64_t* primes, float scale) {
  static_assert(D == 2 || D == 3, "the fast kernels cover two and three dimensions");
  constexpr int CN = 1 << D;
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (n >= N) return;
  uint32_t pi[3] = {0u, 0u, 0u};
#pragma unroll
  for (int d = 0; d < D; ++d) pi[d] = (uint32_t)primes[d];
  float x[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    x[d] = load_as_f32(coords, n * csn + d * csd, cdt);
    if (scale != 1.0f) x[d] = x[d] / scale;
  }
  const bool hashed = l >= g.first_hash;
  const uint32_t res = (uint32_t)g.res[l];
  const float fres = (float)g.res[l];
  const uint32_t mask = g.rows[l] - 1;
  uint32_t c[3] = {0u, 0u, 0u};
  float fr[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const float pos = x[d] * fres;
    const float fl = floorf(pos);
    c[d] = cell_index(fl, fres);
    fr[d] = pos - fl;
  }
  const Corner8 r = D == 3 ? rows_d3(c, hashed, res, mask, pi) : rows_d2(c, hashed, res, mask, pi);
  float w[8];
  if (D == 3) weights_d3(fr, w);
  else weights_d2(fr, w);
  const int64_t base = (n * g.levels + l) * CN;
#pragma unroll
  for (int j = 0; j < CN; ++j) {
    out_rows[base + j] = (int64_t)r.row[j];
    if (out_w) out_w[base + j] = w[j];
  }
}

// ---------------------------------------------------------------------------
// Tiled path: D = 3, F = 2, 16-bit tables (one table row = one dword), L % 4 == 0.
//
// A workgroup of 256 threads owns P = 256*PPT consecutive points and walks the
// levels in order, so that the workgroups resident on an XCD touch the same
// one or two level tables at a time and those stay in that XCD's L2.  Results
// are staged in LDS as stage[level][point] (row stride P+2 dwords) and leave
// as full 16-byte pieces of contiguous output rows; the backward stages the
// incoming gradient rows the same way before scattering.
// ---------------------------------------------------------------------------
// FW: 32-bit words (feature pairs) per table row; a corner's FW words share a cache line, so the pairs after the
// first cost no further line fetch.
template <typename TT, int PPT, int FW>
__global__ __launch_bounds__(TILE_THREADS) void hash_fwd_tiled_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                 const uint32_t* table, uint16_t* out,
                                                                 int64_t out_stride, int64_t N, DevGeom g,
                                                                 const int64_t* primes, float scale) {
  constexpr int P = TILE_THREADS * PPT;
  constexpr int LD = P + 2;
  extern __shared__ uint32_t stage[];
  const int t = threadIdx.x;
  const int64_t p0 = (int64_t)blockIdx.x * P;
  const int L = g.levels;

  float x[PPT][3];
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    int64_t n = p0 + t + TILE_THREADS * i;
    if (n >= N) n = N - 1;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      float v = load_as_f32(coords, n * csn + d * csd, cdt);
      x[i][d] = scale != 1.0f ? v / scale : v;
    }
  }
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], (uint32_t)primes[2]};

  for (int l = 0; l < L; ++l) {
    const uint32_t res = (uint32_t)g.res[l];
    const float fres = (float)g.res[l];
    const bool hashed = l >= g.first_hash;
    const uint32_t mask = g.rows[l] - 1;
    const uint32_t* tab = table + g.row_offset[l] * FW;
    uint32_t v[PPT][8][FW];
    float w[PPT][8];
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      uint32_t c[3];
      float fr[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const float pos = x[i][d] * fres;
        const float fl = floorf(pos);
        c[d] = cell_index(fl, fres);
        fr[d] = pos - fl;
      }
      const Corner8 r = rows_d3(c, hashed, res, mask, pi);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (FW == 1) {
          v[i][j][0] = tab[r.row[j]];
        } else if (FW == 2) {
          const uint2 q = *reinterpret_cast<const uint2*>(tab + (size_t)r.row[j] * 2);
          v[i][j][0] = q.x;
          v[i][j][FW > 1 ? 1 : 0] = q.y;
        } else if (FW == 4) {
          const uint4 q = *reinterpret_cast<const uint4*>(tab + (size_t)r.row[j] * 4);
          v[i][j][0] = q.x;
          v[i][j][FW > 1 ? 1 : 0] = q.y;
          v[i][j][FW > 2 ? 2 : 0] = q.z;
          v[i][j][FW > 3 ? 3 : 0] = q.w;
        } else {
#pragma unroll
          for (int f = 0; f < FW; ++f) v[i][j][f] = tab[(size_t)r.row[j] * FW + f];
        }
      }
      weights_d3(fr, w[i]);
    }
#pragma unroll
    for (int i = 0; i < PPT; ++i)
#pragma unroll
      for (int f = 0; f < FW; ++f) {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a0 = a0 + w[i][j] * TT::to_f32((uint16_t)(v[i][j][f] & 0xffffu));
          a1 = a1 + w[i][j] * TT::to_f32((uint16_t)(v[i][j][f] >> 16));
        }
        stage[(l * FW + f) * LD + t + TILE_THREADS * i] = TT::pack(a0, a1);
      }
  }
  __syncthreads();

  // Each point's L*FW*4 bytes leave as pieces of 16 bytes; consecutive lanes take
  // consecutive pieces, so a wave writes 1 KiB of contiguous output per instruction.
  const int pieces = (L * FW) >> 2;
  const int total = P * pieces;
  for (int c = t; c < total; c += TILE_THREADS) {
    const int p = c / pieces, q = c - p * pieces;
    const int64_t n = p0 + p;
    if (n < N) {
      uint4 val;
      val.x = stage[(4 * q + 0) * LD + p];
      val.y = stage[(4 * q + 1) * LD + p];
      val.z = stage[(4 * q + 2) * LD + p];
      val.w = stage[(4 * q + 3) * LD + p];
      *reinterpret_cast<uint4*>(out + n * out_stride + 8 * q) = val;
    }
  }
}

// The points of this wave in a sweep: `per` consecutive ones, fewer (perhaps none) at the end.  Every wave of a launch gets as many,
// so that all take the same number of gather rounds per level and stay at the same level: with the points dealt to workgroups evenly
// but to their waves in turn (64 points to the first, the next 64 to the second, ...) some waves had one round per level and
// some two, the first ran ahead and the tables of more levels than an L2 holds were in use at once (304800 points: 169 against 120 us).
constexpr int LEVELS_THREADS = 1024, LEVELS_LDS = 128 * 1024, LEVELS_XCDS = 8;  // of the kernel that copies whole levels to LDS
template <int WAVES = TILE_THREADS / 64>
struct SweepPart {
  int64_t first;
  int count;
  __device__ __forceinline__ SweepPart(int64_t N, int per) {
    first = ((int64_t)blockIdx.x * WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * per;
    const int64_t left = N - first;
    count = left < per ? (left > 0 ? (int)left : 0) : per;
    if (count == 0) first = N - 1;
  }
  // lanes past the end repeat the last point (their result is not stored)
  __device__ __forceinline__ int64_t point(int k) const { return first + (k < count ? k : count > 0 ? count - 1 : 0); }
};

// Level sweep: the same work with (nearly) the whole grid resident at once.  A thread keeps the packed results of all
// its PPT points' levels in registers and stores finished 64-byte rows at the end; nothing is staged in LDS, so three
// or four workgroups fit a CU and a million points take little more than one round of workgroups.  Workgroups
// that start together and do the same work per level stay together: at any moment an XCD's L2 serves the gathers of
// a few level tables, not of all of them (a workgroup that runs ahead fetches cold lines and falls back, one
// that lags finds them warm and catches up).  With workgroups that start at different times, as in the staged
// kernel's several rounds, every level's table competes for L2 at once.  (Perfect lock-step is not the aim: one
// workgroup per CU, all in the same phase of the same level, lets the memory pipeline drain at every level.)
template <typename TT, int PPT, int D, bool LDS0 = false>
__global__ __launch_bounds__(TILE_THREADS) void hash_fwd_sweep_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                 const uint32_t* table, uint16_t* out, int64_t out_stride,
                                                                 int64_t N, int per, DevGeom g, const int64_t* primes, float scale) {
  constexpr int LMAX = 16;
  const int t = threadIdx.x, lane = t & 63;
  const SweepPart<> part(N, per);
  const int L = g.levels;
  float x[PPT][3];
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    const int64_t n = part.point(lane + 64 * i);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      float v = load_as_f32(coords, n * csn + d * csd, cdt);
      x[i][d] = scale != 1.0f ? v / scale : v;
    }
  }
  // LDS0: the rows of level 0 (dense, a few thousand) are copied to LDS once per workgroup and gathered from there
  extern __shared__ uint32_t level0_rows[];
  if constexpr (LDS0) {
    const uint32_t* src = table + g.row_offset[0];
    for (uint32_t i = t; i < g.rows[0]; i += TILE_THREADS) level0_rows[i] = src[i];
    __syncthreads();
  }
  constexpr int CN = 1 << D;  // corners of a cell
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], D > 2 ? (uint32_t)primes[D > 2 ? 2 : 0] : 0u};
  uint32_t enc[PPT][LMAX];
#pragma unroll
  for (int l = 0; l < LMAX; ++l) {
    if (l < L) {
      const uint32_t res = (uint32_t)g.res[l];
      const float fres = (float)g.res[l];
      const bool hashed = l >= g.first_hash;
      const uint32_t mask = g.rows[l] - 1;
      const uint32_t* tab = table + g.row_offset[l];
#pragma unroll
      for (int i0 = 0; i0 < PPT; i0 += 2) {
        constexpr int AT_ONCE = PPT > 1 ? 2 : 1;
        uint32_t v[AT_ONCE][8];
        float w[AT_ONCE][8];
#pragma unroll
        for (int i = 0; i < AT_ONCE && i0 + i < PPT; ++i) {
          uint32_t c[3];
          float fr[3];
#pragma unroll
          for (int d = 0; d < D; ++d) {
            const float pos = x[i0 + i][d] * fres;
            const float fl = floorf(pos);
            c[d] = cell_index(fl, fres);
            fr[d] = pos - fl;
          }
          const Corner8 r = D == 3 ? rows_d3(c, hashed, res, mask, pi) : rows_d2(c, hashed, res, mask, pi);
          // four points to a thread: each point's eight together are better than the pair's sixteen (327 and 334 us; three points: 119 and 116)
          if constexpr (D == 3 && PPT == 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < CN; ++j) v[i][j] = (LDS0 && l == 0) ? level0_rows[r.row[j]] : tab[r.row[j]];
          if constexpr (D == 3 && PPT == 4) __builtin_amdgcn_sched_barrier(0);
          if (D == 3) weights_d3(fr, w[i]);
          else weights_d2(fr, w[i]);
        }
        // the gathers leave together, ahead of the sums: left to itself the compiler puts the second point's between the
        // first point's additions, and they leave one by one (2^20 points: 410 us)
        if constexpr (D == 3 && PPT < 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < AT_ONCE && i0 + i < PPT; ++i) {
          float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
          for (int j = 0; j < CN; ++j) {
            a0 = a0 + w[i][j] * TT::to_f32((uint16_t)(v[i][j] & 0xffffu));
            a1 = a1 + w[i][j] * TT::to_f32((uint16_t)(v[i][j] >> 16));
          }
          enc[i0 + i][l] = TT::pack(a0, a1);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < PPT; ++i) enc[i][l] = 0u;
    }
  }
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    if (lane + 64 * i >= part.count) continue;
    uint4* dst = reinterpret_cast<uint4*>(out + (part.first + lane + 64 * i) * out_stride);
#pragma unroll
    for (int q = 0; q < LMAX / 4; ++q)
      if (4 * q < L) dst[q] = make_uint4(enc[i][4 * q], enc[i][4 * q + 1], enc[i][4 * q + 2], enc[i][4 * q + 3]);
  }
}

// The level sweep for float32 tables (a row is one 8-byte pair, an output row 32 floats): same walk, same operation
// order as the per-(point, level) kernel, the results of a thread's PPT points held as float pairs.
template <int PPT>
__global__ __launch_bounds__(TILE_THREADS) void hash_fwd_sweep32_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                   const float2* table, float* out, int64_t out_stride,
                                                                   int64_t N, int per, DevGeom g, const int64_t* primes, float scale) {
  constexpr int LMAX = 16;
  const int lane = threadIdx.x & 63;
  const SweepPart<> part(N, per);
  const int L = g.levels;
  float x[PPT][3];
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    const int64_t n = part.point(lane + 64 * i);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      float v = load_as_f32(coords, n * csn + d * csd, cdt);
      x[i][d] = scale != 1.0f ? v / scale : v;
    }
  }
  if (part.count == 0) return;
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], (uint32_t)primes[2]};
  float2 enc[PPT][LMAX];
#pragma unroll
  for (int l = 0; l < LMAX; ++l) {
    if (l < L) {
      const uint32_t res = (uint32_t)g.res[l];
      const float fres = (float)g.res[l];
      const bool hashed = l >= g.first_hash;
      const uint32_t mask = g.rows[l] - 1;
      const float2* tab = table + g.row_offset[l];
      float2 v[PPT][8];
      float w[PPT][8];
#pragma unroll
      for (int i = 0; i < PPT; ++i) {
        uint32_t c[3];
        float fr[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const float pos = x[i][d] * fres;
          const float fl = floorf(pos);
          c[d] = cell_index(fl, fres);
          fr[d] = pos - fl;
        }
        const Corner8 r = rows_d3(c, hashed, res, mask, pi);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = tab[r.row[j]];
        weights_d3(fr, w[i]);
      }
#pragma unroll
      for (int i = 0; i < PPT; ++i) {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a0 = a0 + w[i][j] * v[i][j].x;
          a1 = a1 + w[i][j] * v[i][j].y;
        }
        enc[i][l] = make_float2(a0, a1);
      }
    } else {
#pragma unroll
      for (int i = 0; i < PPT; ++i) enc[i][l] = make_float2(0.0f, 0.0f);
    }
  }
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    if (lane + 64 * i >= part.count) continue;
    float4* dst = reinterpret_cast<float4*>(out + (part.first + lane + 64 * i) * out_stride);
#pragma unroll
    for (int q = 0; q < LMAX / 2; ++q)
      if (2 * q < L) dst[q] = make_float4(enc[i][2 * q].x, enc[i][2 * q].y, enc[i][2 * q + 1].x, enc[i][2 * q + 1].y);
  }
}

// Levels in LDS: where the largest level of the table fits (2^14 rows, the reference's default, are 64 KiB of 16-bit pairs and 128 KiB of
// float32 ones), a workgroup copies one level, or two, into LDS and takes its share of the points through them.  A gather from
// memory costs a unit's L1 about one and a half cycles per lane and the waves wait for it; one from LDS a fraction of
// one, and what is left is the vector arithmetic of the cell and the weights (about 105 instructions per point and level; 2^20 points
// of 16 levels are 50 us of it).  Nothing is kept over the levels, so a thread needs 32 to 47 registers.  A row of the output is
// written in 4- or 8-byte pieces by the workgroups of its levels: they sit on one XCD and go through the same points at the same
// time, so the pieces meet in that XCD's L2 and leave it as whole lines.
// Before -> after (sweep and per-(point, level) kernels, us): float32 2^14 rows, 2^18 points 80 -> 33, 2^20 307 -> 105; fp16 2^14
// rows 2^18 54 -> 22, 2^20 184 -> 71; fp16 2^15 rows 2^20 234 -> 101; two dimensions fp16 2^20 97 -> 47; bf16 rows of four
// features 2^20 256 -> 108; float32 2^16 points 25 -> 12.
template <typename TT, int D, int FEAT, int LW>
__global__ __launch_bounds__(LEVELS_THREADS) void hash_fwd_levels_k(const void* coords, int cdt, int64_t csn, int64_t csd, const uint32_t* table,
                                                                    typename TT::storage* out, int64_t out_stride, int64_t N, int sets, int64_t share,
                                                                    DevGeom g, const int64_t* primes, float scale) {
  typedef typename TT::storage S;
  constexpr int RW = FEAT * (int)sizeof(S) / 4, CN = 1 << D;  // words of a row, corners of a cell
  typedef uint32_t Piece __attribute__((ext_vector_type(4), aligned(4)));  // a level begins wherever the one before it ends
  extern __shared__ __align__(16) uint32_t level_rows[];
  const int tid = threadIdx.x;
  const int set = (int)(blockIdx.x / LEVELS_XCDS) % sets, part = (int)(blockIdx.x / (LEVELS_XCDS * sets)) * LEVELS_XCDS + (int)(blockIdx.x % LEVELS_XCDS);
  const int64_t n_begin = (int64_t)part * share, n_end = n_begin + share < N ? n_begin + share : N;
  if (n_begin >= n_end) return;
  const int l0 = set * LW;
  uint32_t base[LW];  // first word of the level in LDS
  uint32_t at = 0;
#pragma unroll
  for (int k = 0; k < LW; ++k) {
    base[k] = at;
    if (l0 + k < g.levels) {
      const uint32_t* src = table + g.row_offset[l0 + k] * RW;
      const uint32_t words = g.rows[l0 + k] * RW, whole = words & ~3u;
#pragma unroll 4
      for (uint32_t i = tid * 4; i < whole; i += LEVELS_THREADS * 4) {
        const Piece v = *reinterpret_cast<const Piece*>(src + i);
        *reinterpret_cast<uint4*>(level_rows + at + i) = make_uint4(v[0], v[1], v[2], v[3]);
      }
      if (whole + tid < words) level_rows[at + whole + tid] = src[whole + tid];
      at += (words + 3u) & ~3u;
    }
  }
  __syncthreads();
  uint32_t pi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) pi[d] = d < D ? (uint32_t)primes[d < D ? d : 0] * (RW * 4) : 0u;
  auto load_point = [&](int64_t n, float (&x)[3]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const float v = load_as_f32(coords, n * csn + d * csd, cdt);
      x[d] = scale != 1.0f ? v / scale : v;
    }
  };
  float x[3], ahead[3] = {0.0f, 0.0f, 0.0f};
  load_point(n_begin + tid < n_end ? n_begin + tid : n_end - 1, ahead);
  for (int64_t n = n_begin + tid; n - tid < n_end; n += LEVELS_THREADS) {
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = ahead[d];
    load_point(n + LEVELS_THREADS < n_end ? n + LEVELS_THREADS : n_end - 1, ahead);
    uint32_t enc[LW * RW];
#pragma unroll
    for (int k = 0; k < LW; ++k) {
      const int l = l0 + k < g.levels ? l0 + k : l0;
      const uint32_t res = (uint32_t)g.res[l];
      const float fres = (float)g.res[l];
      uint32_t c[3];
      float fr[3], w[8];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const float pos = x[d] * fres;
        const float fl = floorf(pos);
        c[d] = cell_index(fl, fres);
        fr[d] = pos - fl;
      }
      // rows as byte offsets in the level: a hashed level's primes and mask carry the size of a row
      Corner8 r;
      if (l >= g.first_hash) {
        const uint32_t mask = (g.rows[l] - 1) * (RW * 4);
        r = D == 3 ? rows_d3(c, true, res, mask, pi) : rows_d2(c, true, res, mask, pi);
      } else {
        r = D == 3 ? rows_d3(c, false, res, g.rows[l] - 1, pi) : rows_d2(c, false, res, g.rows[l] - 1, pi);
#pragma unroll
        for (int j = 0; j < CN; ++j) r.row[j] *= RW * 4;
      }
      if (D == 3) weights_d3(fr, w);
      else weights_d2(fr, w);
      uint32_t v[CN][RW];
#pragma unroll
      for (int j = 0; j < CN; ++j) {
        const uint32_t* row = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(level_rows + base[k]) + r.row[j]);
        if constexpr (RW == 2) {
          const uint2 q = *reinterpret_cast<const uint2*>(row);
          v[j][0] = q.x;
          v[j][1] = q.y;
        } else {
          v[j][0] = *row;
        }
      }
      float a[FEAT];
#pragma unroll
      for (int f = 0; f < FEAT; ++f) a[f] = 0.0f;
#pragma unroll
      for (int j = 0; j < CN; ++j)
#pragma unroll
        for (int f = 0; f < FEAT; ++f) {
          if constexpr (sizeof(S) == 4) a[f] = a[f] + w[j] * __uint_as_float(v[j][f]);
          else a[f] = a[f] + w[j] * TT::to_f32((uint16_t)(f & 1 ? v[j][f / 2] >> 16 : v[j][f / 2] & 0xffffu));
        }
#pragma unroll
      for (int q = 0; q < RW; ++q) {
        if constexpr (sizeof(S) == 4) enc[k * RW + q] = __float_as_uint(a[q]);
        else enc[k * RW + q] = TT::pack(a[2 * q], a[2 * q + 1]);
      }
    }
    if (n < n_end) {
      uint32_t* dst = reinterpret_cast<uint32_t*>(out + n * out_stride + l0 * FEAT);
      if constexpr (LW * RW == 1) *dst = enc[0];
      else if (LW == 1 || l0 + 1 < g.levels) *reinterpret_cast<uint2*>(dst) = make_uint2(enc[0], enc[1]);
      else *dst = enc[0];
    }
  }
}

// Small batches: one thread per (point, level).  A thread per point walks its levels one after the other, and a batch of a few thousand
// points is then a handful of workgroups that wait out sixteen rounds of memory latency while most of the chip idles.  Same arithmetic, in
// the same order, as the kernels above.
// A workgroup's 256 points of one level are a unit of work, and the units stand level by level.  BY_XCD: every XCD takes `share` of them in
// a row (two levels of sixteen), so that a level's table is read into one L2 or two and not into all eight.
template <typename TT, int D, int FEAT, bool BY_XCD>
__global__ __launch_bounds__(TILE_THREADS) void hash_fwd_level_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                 const uint32_t* table, typename TT::storage* out, int64_t out_stride,
                                                                 int64_t N, uint32_t chunks, uint32_t share, DevGeom g, const int64_t* primes,
                                                                 float scale) {
  constexpr int RW = FEAT * (int)sizeof(typename TT::storage) / 4;  // words of a row
  typedef uint32_t Row __attribute__((ext_vector_type(RW)));
  typedef Row TableRow __attribute__((aligned(RW == 1 ? sizeof(typename TT::storage) : 4 * RW)));
  int l = (int)blockIdx.y;
  int64_t n = (int64_t)blockIdx.x * TILE_THREADS + threadIdx.x;
  if constexpr (BY_XCD) {
    const uint32_t unit = blockIdx.x % LEVELS_XCDS * share + blockIdx.x / LEVELS_XCDS;
    l = (int)(unit / chunks);
    n = (int64_t)(unit - (uint32_t)l * chunks) * TILE_THREADS + threadIdx.x;
    if (l >= g.levels) return;
  }
  if (n >= N) return;
  constexpr int CN = 1 << D;
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], D > 2 ? (uint32_t)primes[D > 2 ? 2 : 0] : 0u};
  const uint32_t res = (uint32_t)g.res[l];
  const float fres = (float)g.res[l];
  const TableRow* tab = reinterpret_cast<const TableRow*>(table) + g.row_offset[l];
  uint32_t c[3];
  float fr[3];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    float v = load_as_f32(coords, n * csn + d * csd, cdt);
    v = scale != 1.0f ? v / scale : v;
    const float pos = v * fres;
    const float fl = floorf(pos);
    c[d] = cell_index(fl, fres);
    fr[d] = pos - fl;
  }
  const Corner8 r = D == 3 ? rows_d3(c, l >= g.first_hash, res, g.rows[l] - 1, pi) : rows_d2(c, l >= g.first_hash, res, g.rows[l] - 1, pi);
  Row v[CN];
#pragma unroll
  for (int j = 0; j < CN; ++j) v[j] = tab[r.row[j]];
  float w[8];
  if (D == 3) weights_d3(fr, w);
  else weights_d2(fr, w);
  Row sum;
#pragma unroll
  for (int e = 0; e < RW; ++e) {
    if constexpr (sizeof(typename TT::storage) == 4) {
      float a = 0.0f;
#pragma unroll
      for (int j = 0; j < CN; ++j) a = a + w[j] * __uint_as_float(v[j][e]);
      sum[e] = __float_as_uint(a);
    } else {
      float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
      for (int j = 0; j < CN; ++j) {
        a0 = a0 + w[j] * TT::to_f32((uint16_t)(v[j][e] & 0xffffu));
        a1 = a1 + w[j] * TT::to_f32((uint16_t)(v[j][e] >> 16));
      }
      sum[e] = TT::pack(a0, a1);
    }
  }
  *reinterpret_cast<Row*>(out + n * out_stride + FEAT * l) = sum;
}

// Backward of small batches: one lane per (point, level, corner, feature).  What it costs are the atomics' requests, one per 64 bytes
// that a wave's instruction touches: with the features of a row, and the mostly adjacent rows of an x-pair of corners, in neighbouring
// lanes, an instruction of 64 adds is about twenty requests, where a lane that goes through the corners of its own point makes
// 64.  The cell is worked out once per lane, which costs next to nothing in comparison.
// 4096 points, 16 levels of 2^19 rows: 55 -> 19 us.
template <typename GT, int D, int FEAT>
__global__ __launch_bounds__(TILE_THREADS) void hash_bwd_level_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                 const typename GT::storage* dout, int64_t dout_stride, float* dtable,
                                                                 int64_t N, DevGeom g, const int64_t* primes, float scale) {
  constexpr int LANES = FEAT << D;  // of a point: corner, then feature
  const int l = blockIdx.y;
  const int64_t n = ((int64_t)blockIdx.x * TILE_THREADS + threadIdx.x) / LANES;
  if (n >= N) return;
  const int f = (int)(threadIdx.x % FEAT), j = (int)(threadIdx.x % LANES) / FEAT;
  const float grad = GT::to_f32(dout[n * dout_stride + l * FEAT + f]);
  if (grad == 0.0f) return;
  const uint32_t mask = g.rows[l] - 1, res = (uint32_t)g.res[l];
  const float fres = (float)g.res[l];
  const bool hashed = l >= g.first_hash;
  uint32_t row = 0u, unit = 1u;
  float w = 1.0f;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    float v = load_as_f32(coords, n * csn + d * csd, cdt);
    v = scale != 1.0f ? v / scale : v;
    const float pos = v * fres;
    const float fl = floorf(pos), fr = pos - fl;
    const uint32_t side = (uint32_t)(j >> d) & 1u, c = cell_index(fl, fres) + side;
    const float wd = side ? fr : 1.0f - fr;
    w = d == 0 ? wd : w * wd;
    row = hashed ? row ^ c * (uint32_t)primes[d] : row + c * unit;
    unit *= res;
  }
  row = hashed ? row & mask : row < mask ? row : mask;  // (x == scale in two dimensions, see rows_d2())
  unsafeAtomicAdd(dtable + (g.row_offset[l] + (int64_t)row) * FEAT + f, w * grad);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// below this many points the scattered-atomic kernels are faster than planning + scanning
constexpr int64_t SCAN_MIN_POINTS = 32768;
constexpr int SWEEP_PPT = 4;
// Batches from which the sweeps run.  In three dimensions with 16-bit tables the staged kernel's 512 points per workgroup are one
// workgroup per unit up to 2^17 points (51 us, the sweep 56) and two beyond (150000 points: 97 us, the sweep 67); the other kinds have
// the per-(point, level) kernels below them (two dimensions, 10^5 points: 36 us, the sweep 25; float32: 79 and 63 us).
constexpr int64_t SWEEP_MIN_POINTS = ((int64_t)1 << 17) + 1;
constexpr int64_t SWEEP_MIN_POINTS_D2 = (int64_t)1 << 16;
constexpr int64_t SWEEP_MIN_POINTS_F32 = (int64_t)1 << 16;
constexpr int64_t L2_BYTES = 4 << 20;
static int64_t largest_level(const nf_hash_geom* g, int es) {
  int64_t rows = 0;
  for (int l = 0; l < g->levels; ++l) rows = g->rows[l] > rows ? g->rows[l] : rows;
  return rows * g->feat * es;
}
// Units of a level on one XCD (hash_fwd_level_k): where a level fits an L2 and the table does not, in batches that every XCD would read most of
// it for.  2^15 points on 16 levels of 2^19 rows touch most of a table's lines from every XCD, 150 MB in all (us, dealt out in turn / by XCD,
// uniform and rays): fp16 2^15 points 26 / 21 and 21 / 20, 2^16 43 / 35 and 35 / 34; float32 60000 56 / 43 and 48 / 43; four features
// 2^16 57 / 48 and 49 / 47; but 8192 points along rays 9.2 / 10.4, a table of 3 MB 2^16 28 / 32, levels of 8 MiB 61 / 61, two dimensions
// (most levels dense, their rows in order) 2^16 19 / 25, 2^18 points 246 / 276; and, each XCD reading a table of 13 MB often enough to be worth
// its misses, 2^15 points 18 / 18 along rays, 2^16 30 / 32.  Two thirds of the levels have to be hashed: dense ones take a fraction of the time, above all along
// rays, and the XCDs that have those wait for the others (hashed levels of all, 2^15 points along rays, uniform): 2 of 16 (2^20 rows, 8 .. 128) 8.6 / 14 and
// 17 / 21; 8 of 16 (2^19 rows, 16 .. 400) 15.0 / 17.8 and 21 / 20; 10 of 16 (.. 1500) 19.2 / 19.6; 12 of 16 (.. 7006) 21 / 20.  With 11 or more of 16 1.1 times as
// fast along rays and 1.3 times uniform, on average over 29 tables at 16384 to 50000 points; the worst, a table of 50 MB at 16384 points along rays, 14.7 / 15.6.
static bool level_by_xcd(const nf_hash_geom* g, int table_dt, int64_t n_points) {
  if (g->dims != 3 || n_points < 16384 || 3 * (g->levels - g->first_hash_level) < 2 * g->levels) return false;
  const int es = table_dt == NF_F32 ? 4 : 2;
  int64_t rows = 0;
  for (int l = 0; l < g->levels; ++l) rows += g->rows[l];
  const int64_t bytes = rows * g->feat * es;
  return n_points * 320 <= bytes && largest_level(g, es) <= L2_BYTES && bytes > 2 * L2_BYTES;
}
// The forward per (point, level) serves batches up to this where the staged kernel is the alternative, which takes sixteen rounds of latency for any
// batch up to 2^17 points (us, level / staged: two features 2^16 points 35 / 51, 2^17 62 / 51; four 1000 4 / 54, 2^15 27 / 58, 2^16
// 48 / 59, 100000 72 / 63).  Rows of four features in levels beyond an L2: 8 MiB 2^15 37 / 59, 2^16 68 / 64.  Rows of eight in any: levels of 1 MiB 50000 points
// 28.4 / 28.2 along rays, 2^16 uniform 40 / 35, of 4 MiB 50000 51 / 46, of 8 MiB 2^15 39 / 42, 2^16 72 / 62; but by XCD 50000 points of 2 MiB 30 / 38 and, rays,
// 29 / 32, 2^16 36 / 41 and 35 / 34.
constexpr int64_t LEVEL_POINTS = 40960;  // taken whatever the rows
static int64_t level_max_points(const nf_hash_geom* g, int table_dt, int64_t n_points) {
  if (n_points <= LEVEL_POINTS) return LEVEL_POINTS;  // (the loops over the levels are 0.05 us of a call of 5.4)
  if (g->feat == 8) return level_by_xcd(g, table_dt, n_points) ? 53248 : LEVEL_POINTS;
  return g->feat > 2 && largest_level(g, 2) > L2_BYTES ? LEVEL_POINTS : 65536;
}

// How a sweep's points are dealt out.  A compute unit works its gathers off at a rate of its own (one workgroup on a unit runs
// at the rate of three: 1024 points take 83 us either way, because the unit's L1 takes about three lanes in four clocks
// whatever waits behind it), so the time is that of the unit with the most points.  A launch therefore takes whole multiples of
// one workgroup per unit, all of the same number of points, instead of full workgroups and a remainder that a few units
// run alone (304800 points, full workgroups of 1024: 298 workgroups, twice the time of 256).
constexpr int64_t COMPUTE_UNITS = 256;

// Levels in LDS: batches from which the copying pays.  Under that the per-(point, level) kernels run (16-bit pairs: 5.3 and 5.8 us
// at 8192 points, 8.5 and 6.3 at 2^14; float32: 5.1 and 5.0 us at 4096, 6.2 and 5.5 at 8192).
constexpr int64_t LEVELS_MIN_POINTS_16 = 16384, LEVELS_MIN_POINTS_F32 = 4096;

// points per wave, at most `most`, four waves to a workgroup
static int sweep_wave_points(int64_t n, int most) {
  const int64_t waves = 4 * COMPUTE_UNITS * ((n + 4 * COMPUTE_UNITS * most - 1) / (4 * COMPUTE_UNITS * most));
  return (int)((n + waves - 1) / waves);
}

// the sweep for waves of `per` points: as many per thread as that takes
template <typename TT, int PPT = SWEEP_PPT>
static const void* sweep_kernel(int per, int dims, bool lds0) {
  if constexpr (PPT > 1)
    if (per <= 64 * (PPT - 1)) return sweep_kernel<TT, PPT - 1>(per, dims, lds0);
  if (dims == 2) return (const void*)hash_fwd_sweep_k<TT, PPT, 2>;
  return lds0 ? (const void*)hash_fwd_sweep_k<TT, PPT, 3, true> : (const void*)hash_fwd_sweep_k<TT, PPT, 3>;
}

static unsigned sweep_groups(int64_t n, int per) { return (unsigned)((n + 4 * per - 1) / (4 * per)); }

static bool tiled_ok(const nf_hash_geom* g, int table_dt, const void* rows_ptr, int64_t row_stride, int feat = 2, int dims = 3) {
  if (g->dims != dims || g->feat != feat || table_dt == NF_F32) return false;
  if ((g->levels * (feat / 2)) % 4 != 0 || g->levels > 16) return false;
  for (int l = g->first_hash_level; l < g->levels; ++l) {
    if (l < 0) return false;
    const int64_t r = g->rows[l];
    if ((r & (r - 1)) != 0) return false;
  }
  if (((uintptr_t)rows_ptr & 15u) != 0 || (row_stride * 2) % 16 != 0) return false;
  return true;
}

// the per-(point, level) kernel: three dimensions, or two and two features (four 65535 points 29 us, the generic kernel 28), hashed levels of a
// power of two of rows, rows of 4, 8 or 16 bytes that can be written as one piece, and read as one (4 bytes from any address: a table of 2^19
// rows a level, a value into its buffer, 1000 / 2^16 points 5 / 35 us here and 51 / 53 staged)
static bool level_ok(const nf_hash_geom* g, int table_dt, const void* table, const void* rows_ptr, int64_t row_stride) {
  const int es = table_dt == NF_F32 ? 4 : 2, row = g->feat * es;
  if (!(g->dims == 3 || (g->dims == 2 && g->feat == 2)) || !(g->feat == 2 || g->feat == 4 || (g->feat == 8 && es == 2))) return false;
  for (int l = g->first_hash_level; l < g->levels; ++l) {
    if (l < 0) return false;
    const int64_t r = g->rows[l];
    if ((r & (r - 1)) != 0) return false;
  }
  return (row == 4 || (uintptr_t)table % row == 0) && (uintptr_t)rows_ptr % row == 0 && row_stride * es % row == 0;
}

// whether every level fits LDS and the rows can be read and written in words; pair: two levels fit together
static bool levels_ok(const nf_hash_geom* g, int table_dt, const void* table, const void* out, int64_t out_stride, bool* pair) {
  const int es = table_dt == NF_F32 ? 4 : 2, row = g->feat * es;
  if ((g->dims != 2 && g->dims != 3) || g->levels > 16 || !(g->feat == 2 || (g->feat == 4 && es == 2))) return false;
  int64_t most = 0;
  for (int l = 0; l < g->levels; ++l) {
    if (g->rows[l] * row > LEVELS_LDS) return false;
    if (l >= g->first_hash_level && (g->rows[l] & (g->rows[l] - 1)) != 0) return false;
    most = g->rows[l] > most ? g->rows[l] : most;
  }
  *pair = row == 4 && most * row <= LEVELS_LDS / 2;
  const int piece = row == 4 && !*pair ? 4 : 8;
  return ((uintptr_t)table & 3u) == 0 && ((uintptr_t)out % piece) == 0 && (out_stride * es) % piece == 0;
}

static int launch_fwd_levels(const void* coords, int cdt, int64_t csn, int64_t csd, const void* table, int table_dt, void* out, int64_t out_stride,
                             int64_t N, const DevGeom& g, const int64_t* primes, float scale, bool pair, hipStream_t s) {
  auto pick = [&](auto tt) -> const void* {
    typedef decltype(tt) TT;
    if constexpr (sizeof(typename TT::storage) == 4) return g.dims == 3 ? (const void*)hash_fwd_levels_k<TT, 3, 2, 1> : (const void*)hash_fwd_levels_k<TT, 2, 2, 1>;
    else if (g.feat == 4) return g.dims == 3 ? (const void*)hash_fwd_levels_k<TT, 3, 4, 1> : (const void*)hash_fwd_levels_k<TT, 2, 4, 1>;
    else if (pair) return g.dims == 3 ? (const void*)hash_fwd_levels_k<TT, 3, 2, 2> : (const void*)hash_fwd_levels_k<TT, 2, 2, 2>;
    else return g.dims == 3 ? (const void*)hash_fwd_levels_k<TT, 3, 2, 1> : (const void*)hash_fwd_levels_k<TT, 2, 2, 1>;
  };
  const void* kern = table_dt == NF_F32 ? pick(F32{}) : table_dt == NF_F16 ? pick(F16{}) : pick(BF16{});
  const int lw = pair ? 2 : 1, row = g.feat * (table_dt == NF_F32 ? 4 : 2);
  int sets = (g.levels + lw - 1) / lw;
  size_t lds = 0;
  for (int l = 0; l < g.levels; l += lw) {
    size_t bytes = 0;
    for (int k = l; k < l + lw && k < g.levels; ++k) bytes += ((size_t)g.rows[k] * row + 15) / 16 * 16;
    lds = bytes > lds ? bytes : lds;
  }
  hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  // one workgroup per unit: the points in parts, a multiple of the XCDs of them, and of at least a turn of the workgroup
  int64_t parts = COMPUTE_UNITS / (LEVELS_XCDS * sets);
  const int64_t most = (N + LEVELS_XCDS * LEVELS_THREADS - 1) / (LEVELS_XCDS * LEVELS_THREADS);
  parts = LEVELS_XCDS * (most < parts ? most : parts);
  int64_t share = (N + parts - 1) / parts;
  const uint32_t* tab = (const uint32_t*)table;
  DevGeom gg = g;
  void* args[] = {(void*)&coords, (void*)&cdt, (void*)&csn, (void*)&csd, (void*)&tab, (void*)&out, (void*)&out_stride, (void*)&N, (void*)&sets, (void*)&share, (void*)&gg, (void*)&primes, (void*)&scale};
  e = hipLaunchKernel(kern, dim3((unsigned)(parts * sets)), dim3(LEVELS_THREADS), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(hash_fwd_levels): %s", hipGetErrorString(e));
  return check_launch("hash_fwd_levels");
}

static bool sweep32_ok(const nf_hash_geom* g, const void* table, const void* rows_ptr, int64_t row_stride) {
  if (g->dims != 3 || g->feat != 2 || g->levels % 2 != 0 || g->levels > 16) return false;
  for (int l = g->first_hash_level; l < g->levels; ++l) {
    if (l < 0) return false;
    const int64_t r = g->rows[l];
    if ((r & (r - 1)) != 0) return false;
  }
  return ((uintptr_t)table & 7u) == 0 && ((uintptr_t)rows_ptr & 15u) == 0 && row_stride % 4 == 0;
}

template <int D, typename TT>
static void launch_fwd_generic(const void* coords, int cdt, int64_t csn, int64_t csd, const void* table, void* out,
                               int64_t out_stride, int64_t N, const DevGeom& g, const int64_t* primes, float scale, bool vec,
                               hipStream_t s) {
  typedef typename TT::storage S;
  dim3 grid((unsigned)((N + 255) / 256), (unsigned)g.levels);
  // the widest piece of 16, 8 or 4 bytes that divides a row and keeps every row of the table and of the output aligned
  int v = 1;
  if (vec && D <= 4)
    for (int bytes = 16; bytes > (int)sizeof(S); bytes >>= 1) {
      const int c = bytes / (int)sizeof(S);
      if (g.feat % c == 0 && out_stride % c == 0 && (uintptr_t)table % bytes == 0 && (uintptr_t)out % bytes == 0) {
        v = c;
        break;
      }
    }
  const void* kern = (const void*)hash_fwd_generic_k<D, TT, 1>;
  if constexpr (D <= 4) {
    if (v == 2) kern = (const void*)hash_fwd_generic_k<D, TT, 2>;
    if (v == 4) kern = (const void*)hash_fwd_generic_k<D, TT, 4>;
    if constexpr (sizeof(S) == 2)
      if (v == 8) kern = (const void*)hash_fwd_generic_k<D, TT, 8>;
  }
  const S* tab = (const S*)table;
  S* o = (S*)out;
  DevGeom gg = g;
  void* args[] = {&coords, &cdt, &csn, &csd, &tab, &o, &out_stride, &N, &gg, &primes, &scale};
  (void)hipLaunchKernel(kern, grid, dim3(256), args, 0, s);  // the caller reads the launch status
}

template <int D>
static int dispatch_fwd_generic(int table_dt, const void* coords, int cdt, int64_t csn, int64_t csd, const void* table,
                                void* out, int64_t out_stride, int64_t N, const DevGeom& g, const int64_t* primes,
                                float scale, bool vec, hipStream_t s) {
  switch (table_dt) {
    case NF_F32: launch_fwd_generic<D, F32>(coords, cdt, csn, csd, table, out, out_stride, N, g, primes, scale, vec, s); break;
    case NF_F16: launch_fwd_generic<D, F16>(coords, cdt, csn, csd, table, out, out_stride, N, g, primes, scale, vec, s); break;
    default: launch_fwd_generic<D, BF16>(coords, cdt, csn, csd, table, out, out_stride, N, g, primes, scale, vec, s); break;
  }
  return check_launch("hash_fwd_generic");
}

static int launch_fwd_level(int table_dt, const void* coords, int cdt, int64_t csn, int64_t csd, const void* table, void* out, int64_t out_stride,
                            int64_t N, const DevGeom& g, const int64_t* primes, float scale, bool by_xcd, hipStream_t s) {
  auto pick = [&](auto tt) -> const void* {
    typedef decltype(tt) TT;
    auto dims = [&](auto f_c) -> const void* {
      constexpr int F = decltype(f_c)::value;
      if constexpr (F == 2)
        if (g.dims == 2) return (const void*)hash_fwd_level_k<TT, 2, F, false>;
      return by_xcd ? (const void*)hash_fwd_level_k<TT, 3, F, true> : (const void*)hash_fwd_level_k<TT, 3, F, false>;
    };
    if constexpr (sizeof(typename TT::storage) == 2)
      if (g.feat == 8) return dims(std::integral_constant<int, 8>{});
    return g.feat == 4 ? dims(std::integral_constant<int, 4>{}) : dims(std::integral_constant<int, 2>{});
  };
  const void* kern = table_dt == NF_F32 ? pick(F32{}) : table_dt == NF_F16 ? pick(F16{}) : pick(BF16{});
  // launches of at most 2^26 points: units stay inside 32 bits
  constexpr int64_t part = (int64_t)1 << 26;
  const int row = g.feat * (table_dt == NF_F32 ? 4 : 2);
  for (int64_t n0 = 0; n0 < N; n0 += part) {
    int64_t n = N - n0 < part ? N - n0 : part;
    uint32_t chunks = (uint32_t)((n + TILE_THREADS - 1) / TILE_THREADS), share = by_xcd ? (chunks * (uint32_t)g.levels + LEVELS_XCDS - 1) / LEVELS_XCDS : 0u;
    const void* c = (const char*)coords + n0 * csn * dtype_size(cdt);
    void* o = (char*)out + n0 * out_stride * (row / g.feat);
    DevGeom gg = g;
    void* args[] = {(void*)&c, (void*)&cdt, (void*)&csn, (void*)&csd, (void*)&table, (void*)&o, (void*)&out_stride, (void*)&n, (void*)&chunks, (void*)&share, (void*)&gg, (void*)&primes, (void*)&scale};
    const hipError_t e = hipLaunchKernel(kern, by_xcd ? dim3(share * LEVELS_XCDS) : dim3(chunks, (unsigned)g.levels), dim3(TILE_THREADS), args, 0, s);
    if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(hash_fwd_level): %s", hipGetErrorString(e));
  }
  return check_launch("hash_fwd_level");
}

template <int FW>
static int launch_fwd_tiled_wide(int table_dtype, const void* coords, int coords_dtype, int64_t csn, int64_t csd, const void* table,
                                 void* out, int64_t out_stride_n, int64_t n_points, const DevGeom& g, const int64_t* primes,
                                 float scale, hipStream_t s) {
  constexpr int PPT = FW <= 2 ? 2 : 1;
  constexpr int P = TILE_THREADS * PPT;
  const size_t lds = (size_t)g.levels * FW * (P + 2) * sizeof(uint32_t);
  dim3 grid((unsigned)((n_points + P - 1) / P));
  const void* kern = table_dtype == NF_F16 ? (const void*)hash_fwd_tiled_k<F16, PPT, FW> : (const void*)hash_fwd_tiled_k<BF16, PPT, FW>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  const uint32_t* tab = (const uint32_t*)table;
  uint16_t* o = (uint16_t*)out;
  void* args[] = {(void*)&coords, (void*)&coords_dtype, (void*)&csn, (void*)&csd, (void*)&tab, (void*)&o,
                  (void*)&out_stride_n, (void*)&n_points, (void*)&g, (void*)&primes, (void*)&scale};
  const hipError_t e = hipLaunchKernel(kern, grid, dim3(TILE_THREADS), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(hash_fwd_tiled): %s", hipGetErrorString(e));
  return check_launch("hash_fwd_tiled");
}

}  // namespace nf

using namespace nf;

extern "C" int nf_hash_encode_fwd(const void* coords, int coords_dtype, int64_t csn, int64_t csd, const void* table,
                                  int table_dtype, void* out, int64_t out_stride_n, int64_t n_points,
                                  const nf_hash_geom* geom, const int64_t* primes, float scale, int flags,
                                  void* stream) {
  DevGeom g;
  if (int rc = make_dev_geom(geom, &g)) return rc;
  NF_REQUIRE(dtype_ok(coords_dtype) && dtype_ok(table_dtype), NF_EINVAL, "unknown dtype code");
  NF_REQUIRE(n_points >= 0, NF_EINVAL, "n_points negative");
  NF_REQUIRE(out_stride_n >= (int64_t)g.levels * g.feat, NF_EINVAL, "out_stride_n=%lld < levels*feat",
             (long long)out_stride_n);
  NF_REQUIRE(scale > 0.0f, NF_EINVAL, "scale must be positive");
  if (n_points == 0) return 0;
  NF_REQUIRE(coords && table && out && primes, NF_EINVAL, "NULL pointer argument");
  NF_REQUIRE(n_points <= ((int64_t)1 << 31) * 256 - 1, NF_EINVAL, "n_points too large");
  hipStream_t s = (hipStream_t)stream;

  // More than sixteen levels: the fast kernels keep a point's results of up to sixteen levels in registers, and the
  // levels are independent, so the call runs as one call per sixteen levels on its own columns of the output
  // (2^20 points, 32 levels: 1.03 -> 0.73 ms).
  if (g.levels > 16 && !(flags & NF_HASH_FORCE_GENERIC)) {
    for (int l0 = 0; l0 < g.levels; l0 += 16) {
      nf_hash_geom part = *geom;
      part.levels = g.levels - l0 < 16 ? g.levels - l0 : 16;
      const int fh = geom->first_hash_level - l0;
      part.first_hash_level = fh < 0 ? 0 : (fh > part.levels ? part.levels : fh);
      for (int l = 0; l < part.levels; ++l) {
        part.res[l] = geom->res[l0 + l];
        part.rows[l] = geom->rows[l0 + l];
        part.row_offset[l] = geom->row_offset[l0 + l];
      }
      void* cols = (char*)out + (size_t)l0 * g.feat * dtype_size(table_dtype);
      if (int rc = nf_hash_encode_fwd(coords, coords_dtype, csn, csd, table, table_dtype, cols, out_stride_n, n_points, &part, primes, scale,
                                      flags, stream))
        return rc;
    }
    return 0;
  }

  bool level_pairs;
  if (!(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FWD_STAGED)) &&
      n_points >= (table_dtype == NF_F32 ? LEVELS_MIN_POINTS_F32 : geom->feat == 2 ? LEVELS_MIN_POINTS_16 : 1) &&
      levels_ok(geom, table_dtype, table, out, out_stride_n, &level_pairs))
    return launch_fwd_levels(coords, coords_dtype, csn, csd, table, table_dtype, out, out_stride_n, n_points, g, primes, scale, level_pairs, s);
  // float32 tables: the same sweep on 8-byte rows
  if (!(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FWD_STAGED)) && n_points >= SWEEP_MIN_POINTS_F32 && table_dtype == NF_F32 &&
      sweep32_ok(geom, table, out, out_stride_n)) {
    constexpr int PPT = 2;
    // launches of up to 1024 workgroups (2^19 points), for the reason given at the 16-bit sweep below
    // (2^20 points: 663 -> 613 us, 2^22 points: 3514 -> 2687 us)
    constexpr int64_t chunk = (int64_t)1 << 19;
    for (int64_t n0 = 0; n0 < n_points; n0 += chunk) {
      const int64_t n = n_points - n0 < chunk ? n_points - n0 : chunk;
      const int per = sweep_wave_points(n, 64 * PPT);
      const void* c = (const char*)coords + n0 * csn * dtype_size(coords_dtype);
      hipLaunchKernelGGL((hash_fwd_sweep32_k<PPT>), dim3(sweep_groups(n, per)), dim3(TILE_THREADS), 0, s, c, coords_dtype, csn,
                         csd, (const float2*)table, (float*)out + n0 * out_stride_n, out_stride_n, n, per, g, primes, scale);
    }
    return check_launch("hash_fwd_sweep32");
  }
  // 16-bit tables in three dimensions, and over four corners in two
  if (!(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FWD_STAGED)) && n_points >= (g.dims == 2 ? SWEEP_MIN_POINTS_D2 : SWEEP_MIN_POINTS) &&
      tiled_ok(geom, table_dtype, out, out_stride_n, 2, g.dims == 2 ? 2 : 3)) {
    // level 0 in LDS where it is dense and small (19.6 KB at resolution 16): worth about 1 % (its rows mostly hit L1 anyway)
    const bool lds0 = g.dims == 3 && geom->first_hash_level > 0 && geom->rows[0] * 4 <= 32 * 1024;
    const size_t lds = lds0 ? (size_t)geom->rows[0] * 4 : 0;
    const uint32_t* tab = (const uint32_t*)table;
    // Launches of at most 2^20 points: the workgroups of one launch are (nearly) all resident and walk the levels
    // together; in one launch of 2^22 points later rounds of workgroups meet earlier ones at other levels and the
    // tables compete for L2 (1545 us against 1324 us in four launches; 677 against 661 us at 2^21).
    constexpr int64_t chunk = (int64_t)1 << 20;
    for (int64_t n0 = 0; n0 < n_points; n0 += chunk) {
      int64_t n = n_points - n0 < chunk ? n_points - n0 : chunk;
      int per = sweep_wave_points(n, 64 * SWEEP_PPT);
      const void* kern = table_dtype == NF_F16 ? sweep_kernel<F16>(per, g.dims, lds0) : sweep_kernel<BF16>(per, g.dims, lds0);
      const void* c = (const char*)coords + n0 * csn * dtype_size(coords_dtype);
      uint16_t* o = (uint16_t*)out + n0 * out_stride_n;
      void* args[] = {(void*)&c, (void*)&coords_dtype, (void*)&csn, (void*)&csd, (void*)&tab, (void*)&o, (void*)&out_stride_n,
                      (void*)&n, (void*)&per, (void*)&g, (void*)&primes, (void*)&scale};
      const hipError_t e = hipLaunchKernel(kern, dim3(sweep_groups(n, per)), dim3(TILE_THREADS), args, lds, s);
      if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(hash_fwd_sweep): %s", hipGetErrorString(e));
    }
    return check_launch("hash_fwd_sweep");
  }
  // batches below the sweep's minimum, and rows that neither sweep nor staged kernel takes: a thread per (point, level)
  if (!(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FWD_STAGED)) && level_ok(geom, table_dtype, table, out, out_stride_n) &&
      (n_points <= level_max_points(geom, table_dtype, n_points) || !tiled_ok(geom, table_dtype, out, out_stride_n, geom->feat)))
    return launch_fwd_level(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale,
                            level_by_xcd(geom, table_dtype, n_points), s);
  if (!(flags & NF_HASH_FORCE_GENERIC) && tiled_ok(geom, table_dtype, out, out_stride_n)) {
    constexpr int PPT = 2;
    constexpr int P = TILE_THREADS * PPT;
    const size_t lds = (size_t)g.levels * (P + 2) * sizeof(uint32_t);
    dim3 grid((unsigned)((n_points + P - 1) / P));
    if (table_dtype == NF_F16)
      hipLaunchKernelGGL((hash_fwd_tiled_k<F16, PPT, 1>), grid, dim3(TILE_THREADS), lds, s, coords, coords_dtype, csn,
                         csd, (const uint32_t*)table, (uint16_t*)out, out_stride_n, n_points, g, primes, scale);
    else
      hipLaunchKernelGGL((hash_fwd_tiled_k<BF16, PPT, 1>), grid, dim3(TILE_THREADS), lds, s, coords, coords_dtype, csn,
                         csd, (const uint32_t*)table, (uint16_t*)out, out_stride_n, n_points, g, primes, scale);
    return check_launch("hash_fwd_tiled");
  }
  // 16-bit rows of 4 or 8 features: the staged kernel with 8- or 16-byte gathers
  if (!(flags & NF_HASH_FORCE_GENERIC) && (geom->feat == 4 || geom->feat == 8) && tiled_ok(geom, table_dtype, out, out_stride_n, geom->feat) &&
      ((uintptr_t)table % (2 * geom->feat) == 0)) {
    return geom->feat == 4 ? launch_fwd_tiled_wide<2>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, s)
                           : launch_fwd_tiled_wide<4>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, s);
  }
  const bool vec = !(flags & NF_HASH_FORCE_GENERIC);  // the flag keeps the scalar form as the other kernels' bit-exact check
  switch (g.dims) {
    case 1: return dispatch_fwd_generic<1>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
    case 2: return dispatch_fwd_generic<2>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
    case 3: return dispatch_fwd_generic<3>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
    case 4: return dispatch_fwd_generic<4>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
    case 5: return dispatch_fwd_generic<5>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
    default: return dispatch_fwd_generic<6>(table_dtype, coords, coords_dtype, csn, csd, table, out, out_stride_n, n_points, g, primes, scale, vec, s);
  }
}

// whether a batch is large enough for one of the backward's LDS-tile variants
static bool bwd_tiles_apply(int64_t n_points, const nf_hash_geom* geom, int flags) {
  if (flags & NF_HASH_FORCE_PLANES) return n_points >= SCAN_MIN_POINTS;
  return n_points >= bwd_records_min(geom, flags) || bwd_walk_applies(n_points, geom, flags);
}

int64_t nf::bwd_workspace_bytes(int64_t n_points, const nf_hash_geom* geom, int dout_dtype, int flags, bool whole) {
  if (geom == nullptr || (flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FORCE_ATOMIC))) return 0;
  if (!bwd_tiles_apply(n_points, geom, flags)) return 0;
  const int64_t scan = n_points >= SCAN_MIN_POINTS ? bwd_scan_workspace_bytes(n_points, geom, dout_dtype) : 0;
  if (flags & NF_HASH_FORCE_PLANES) return scan;
  const int64_t bin = bwd_bin_workspace_bytes(n_points, geom, dout_dtype, flags, whole);
  return bin > 0 ? bin : scan;  // the bit-planes are what runs where the other kernels do not cover the geometry
}

extern "C" int64_t nf_hash_encode_bwd_workspace_bytes(int64_t n_points, const nf_hash_geom* geom, int dout_dtype, int flags) {
  return bwd_workspace_bytes(n_points, geom, dout_dtype, flags, true);
}

extern "C" int nf_hash_encode_bwd(const void* coords, int coords_dtype, int64_t csn, int64_t csd, const void* dout,
                                  int dout_dtype, int64_t dout_stride_n, float* dtable, int64_t n_points,
                                  const nf_hash_geom* geom, const int64_t* primes, float scale, void* workspace,
                                  int64_t workspace_bytes, int flags, void* stream) {
  DevGeom g;
  if (int rc = make_dev_geom(geom, &g)) return rc;
  NF_REQUIRE(dtype_ok(coords_dtype) && dtype_ok(dout_dtype), NF_EINVAL, "unknown dtype code");
  NF_REQUIRE(n_points >= 0, NF_EINVAL, "n_points negative");
  NF_REQUIRE(dout_stride_n >= (int64_t)g.levels * g.feat, NF_EINVAL, "dout_stride_n=%lld < levels*feat",
             (long long)dout_stride_n);
  NF_REQUIRE(scale > 0.0f, NF_EINVAL, "scale must be positive");
  if (n_points == 0) return 0;
  NF_REQUIRE(coords && dout && dtable && primes, NF_EINVAL, "NULL pointer argument");
  NF_REQUIRE(n_points <= ((int64_t)1 << 31) * 256 - 1, NF_EINVAL, "n_points too large");
  hipStream_t s = (hipStream_t)stream;

  // large batches: accumulate in LDS tiles (needs the caller's workspace for the sorted records or the bit-planes)
  if (!(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FORCE_ATOMIC)) && workspace != nullptr &&
      bwd_tiles_apply(n_points, geom, flags) &&
      ((uintptr_t)dout % (dout_dtype == NF_F32 ? 8 : 4) == 0) && (dout_stride_n % 2 == 0) && ((uintptr_t)workspace % 4 == 0)) {
    const int64_t need_bin = bwd_bin_workspace_bytes(n_points, geom, dout_dtype, flags, false);
    if (!(flags & NF_HASH_FORCE_PLANES) && need_bin > 0 && workspace_bytes >= need_bin && ((uintptr_t)workspace % 16 == 0))
      return launch_bwd_bin(coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, geom, g, primes,
                            scale, workspace, workspace_bytes, flags, s);
    const int64_t need = n_points >= SCAN_MIN_POINTS ? bwd_scan_workspace_bytes(n_points, geom, dout_dtype) : 0;
    if (need > 0 && workspace_bytes >= need)
      return launch_bwd_scan(coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, geom, g,
                             primes, scale, workspace, s);
  }
  if (!(flags & NF_HASH_FORCE_GENERIC) && bwd_level_ok(geom)) {
    auto pick = [&](auto gt) -> const void* {
      typedef decltype(gt) GT;
      return g.feat == 2 ? (g.dims == 3 ? (const void*)hash_bwd_level_k<GT, 3, 2> : (const void*)hash_bwd_level_k<GT, 2, 2>)
                         : (g.dims == 3 ? (const void*)hash_bwd_level_k<GT, 3, 4> : (const void*)hash_bwd_level_k<GT, 2, 4>);
    };
    const void* kern = dout_dtype == NF_F32 ? pick(F32{}) : dout_dtype == NF_F16 ? pick(F16{}) : pick(BF16{});
    // a launch has less than 2^32 threads: parts of 2^26 points, which with 32 lanes each are 2^31
    constexpr int64_t part = (int64_t)1 << 26;
    for (int64_t n0 = 0; n0 < n_points; n0 += part) {
      int64_t n = n_points - n0 < part ? n_points - n0 : part;
      const void* c = (const char*)coords + n0 * csn * dtype_size(coords_dtype);
      const void* d = (const char*)dout + n0 * dout_stride_n * dtype_size(dout_dtype);
      const int64_t lanes = n * (g.feat << g.dims);
      dim3 grid((unsigned)((lanes + TILE_THREADS - 1) / TILE_THREADS), (unsigned)g.levels);
      void* args[] = {&c, &coords_dtype, &csn, &csd, &d, &dout_stride_n, &dtable, &n, &g, &primes, &scale};
      const hipError_t e = hipLaunchKernel(kern, grid, dim3(TILE_THREADS), args, 0, s);
      if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(hash_bwd_level): %s", hipGetErrorString(e));
    }
    return check_launch("hash_bwd_level");
  }
  dim3 grid((unsigned)((n_points + 255) / 256), (unsigned)g.levels);
  switch (g.dims) {
    case 1: hipLaunchKernelGGL((hash_bwd_generic_k<1>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
    case 2: hipLaunchKernelGGL((hash_bwd_generic_k<2>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
    case 3: hipLaunchKernelGGL((hash_bwd_generic_k<3>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
    case 4: hipLaunchKernelGGL((hash_bwd_generic_k<4>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
    case 5: hipLaunchKernelGGL((hash_bwd_generic_k<5>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
    default: hipLaunchKernelGGL((hash_bwd_generic_k<6>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, n_points, g, primes, scale); break;
  }
  return check_launch("hash_bwd_generic");
}

extern "C" int nf_hash_encode_bwd_write(const void* coords, int coords_dtype, int64_t csn, int64_t csd, const void* dout, int dout_dtype,
                                        int64_t dout_stride_n, void* dtable, int table_dtype, int64_t n_points, const nf_hash_geom* geom,
                                        const int64_t* primes, float scale, void* workspace, int64_t workspace_bytes, int flags,
                                        void* stream) {
  DevGeom g;
  if (int rc = make_dev_geom(geom, &g)) return rc;
  NF_REQUIRE(dtype_ok(coords_dtype) && dtype_ok(dout_dtype) && dtype_ok(table_dtype), NF_EINVAL, "unknown dtype code");
  NF_REQUIRE(dout_stride_n >= (int64_t)g.levels * g.feat, NF_EINVAL, "dout_stride_n=%lld < levels*feat", (long long)dout_stride_n);
  NF_REQUIRE(scale > 0.0f, NF_EINVAL, "scale must be positive");
  NF_REQUIRE(bwd_write_applies(n_points, geom, flags) &&
                 !(flags & (NF_HASH_FORCE_GENERIC | NF_HASH_FORCE_ATOMIC | NF_HASH_FORCE_PLANES)),
             NF_EUNSUPPORTED, "no kernel that writes this gradient in one go (nothing was launched; use nf_hash_encode_bwd)");
  NF_REQUIRE(coords && dout && dtable && primes && workspace, NF_EINVAL, "NULL pointer argument");
  const int64_t need = bwd_bin_workspace_bytes(n_points, geom, dout_dtype, flags, false);
  NF_REQUIRE(need > 0 && (uintptr_t)dout % (dout_dtype == NF_F32 ? 8 : 4) == 0 && dout_stride_n % 2 == 0, NF_EUNSUPPORTED,
             "shape or alignment outside the sorted-record kernels (nothing was launched; use nf_hash_encode_bwd)");
  NF_REQUIRE(workspace_bytes >= need && (uintptr_t)workspace % 16 == 0, NF_EINVAL, "a 16-byte aligned workspace of %lld bytes is needed", (long long)need);
  return launch_bwd_write(coords, coords_dtype, csn, csd, dout, dout_dtype, dout_stride_n, dtable, table_dtype, n_points, geom, g, primes, scale,
                          workspace, workspace_bytes, flags, (hipStream_t)stream);
}

extern "C" int nf_hash_encode_indices_fast(const void* coords, int coords_dtype, int64_t csn, int64_t csd,
                                           int64_t* out_rows, float* out_w, int64_t n_points, const nf_hash_geom* geom,
                                           const int64_t* primes, float scale, void* stream) {
  DevGeom g;
  if (int rc = make_dev_geom(geom, &g)) return rc;
  NF_REQUIRE(dtype_ok(coords_dtype), NF_EINVAL, "unknown dtype code");
  NF_REQUIRE(n_points >= 0, NF_EINVAL, "n_points negative");
  NF_REQUIRE(scale > 0.0f, NF_EINVAL, "scale must be positive");
  NF_REQUIRE(g.dims == 2 || g.dims == 3, NF_EUNSUPPORTED, "the 32-bit index form covers 2 and 3 dimensions, got %d", g.dims);
  for (int l = g.first_hash < 0 ? 0 : g.first_hash; l < g.levels; ++l)
    NF_REQUIRE((g.rows[l] & (g.rows[l] - 1u)) == 0u, NF_EUNSUPPORTED,
               "the 32-bit index form needs power-of-two hashed levels (level %d has %u rows)", l, g.rows[l]);
  if (n_points == 0) return 0;
  NF_REQUIRE(coords && out_rows && primes, NF_EINVAL, "NULL pointer argument");
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)((n_points + 255) / 256), (unsigned)g.levels);
  if (g.dims == 3) hipLaunchKernelGGL((hash_indices_fast_k<3>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale);
  else hipLaunchKernelGGL((hash_indices_fast_k<2>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale);
  return check_launch("hash_indices_fast");
}

extern "C" int nf_hash_encode_indices(const void* coords, int coords_dtype, int64_t csn, int64_t csd,
                                      int64_t* out_rows, float* out_w, int64_t n_points, const nf_hash_geom* geom,
                                      const int64_t* primes, float scale, void* stream) {
  DevGeom g;
  if (int rc = make_dev_geom(geom, &g)) return rc;
  NF_REQUIRE(dtype_ok(coords_dtype), NF_EINVAL, "unknown dtype code");
  NF_REQUIRE(n_points >= 0, NF_EINVAL, "n_points negative");
  NF_REQUIRE(scale > 0.0f, NF_EINVAL, "scale must be positive");
  if (n_points == 0) return 0;
  NF_REQUIRE(coords && out_rows && primes, NF_EINVAL, "NULL pointer argument");
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)((n_points + 255) / 256), (unsigned)g.levels);
  switch (g.dims) {
    case 1: hipLaunchKernelGGL((hash_indices_k<1>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
    case 2: hipLaunchKernelGGL((hash_indices_k<2>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
    case 3: hipLaunchKernelGGL((hash_indices_k<3>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
    case 4: hipLaunchKernelGGL((hash_indices_k<4>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
    case 5: hipLaunchKernelGGL((hash_indices_k<5>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
    default: hipLaunchKernelGGL((hash_indices_k<6>), grid, dim3(256), 0, s, coords, coords_dtype, csn, csd, out_rows, out_w, n_points, g, primes, scale); break;
  }
  return check_launch("hash_indices");
}
