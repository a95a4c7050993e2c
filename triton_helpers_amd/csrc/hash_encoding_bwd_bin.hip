// Hash-encoding backward by binning (D = 2 or 3, and 4 to 6 as passes of the 3-D pipeline; features taken two at a time, the last
// one alone when their number is odd), and the walk without records for small tables and batches.
//
// Every (point, level, corner) contributes  w * dout[n, 2l .. 2l+1]  to one table row.  Scattering these with
// global atomics is bound by the chip's atomic request rate; accumulating them in LDS needs the contributions to
// one stretch of the table together.  So the contributions are first sorted by table bin (BIN_ROWS rows):
//
//   fill    : every workgroup takes some hundred consecutive points and a few levels (in the largest batches all) and, level by level, sorts their records by bin
//             in LDS and writes them out as one contiguous block, with the place of every bin inside the block
//   totals  : the number of records of every bin
//   accum   : a workgroup per compute unit takes task after task, a task being a bin (or, where a bin holds many more records
//             than others, a share of its blocks): the bin's rows live in LDS as two 64-bit integers
//             each and every contribution is one integer LDS atomic per feature (float LDS atomics and
//             compare-and-swap loops are an order of magnitude slower once a few thousand adds are in flight on
//             a tile); the tile is then converted and written to, or added to, the gradient table -- or to a slot of its
//             own where the bin has several tasks
//   reduce  : the slots of every bin with several tasks, summed in a fixed order, into the gradient table
//
// A block is self-contained: no pass counts the records beforehand, nothing is reserved with atomics and the blocks leave as
// whole lines.  (With records in one run per bin for the whole batch, a count pass over all points and two global atomics per
// workgroup and bin cost 50 us at 2^20 points and the fill wrote scattered pieces.)
//
// A record is the pair of corners that differ in x only: 12 bytes {row0 | row1 << 13 inside the bin, w0 and w1 in
// 19-bit fixed point (rounded to nearest: each contribution is off by at most 2^-20 |dout|), packed 16-bit gradient
// pair}.  The records are written once and read once, 4 bytes less per record are worth more than the last bits of
// a weight.  The two rows of a pair share the bin: on a dense level they are
// neighbours, on a hashed level the x prime is 1 and  (x+1) ^ a  differs from  x ^ a  only below the lowest zero
// bit of x.  When they do not (bin border, 13 trailing ones in x) the pair becomes two records with one zero weight
// each.
//
// Dense levels whose cells span less than a bin (3-D, 16-bit gradients) take ONE record per point and level instead
// of four: {row of corner 0 relative to the bin, the three cell fractions in 18 / 16 / 16-bit fixed point, gradient
// pair}, still 12 bytes.  All eight corners lie within  res^2 + res + 1  rows of the first, so they fall into one bin
// or two neighbouring ones; a cell on a bin border is sent to both, and each accumulation takes the corners inside its
// own bin.  The accumulation rebuilds the eight trilinear weights from the fractions (each off by at most 2^-17).
//
// Integer accumulation: fill also finds max |dout| per level; with 2^e the power of two above it, a contribution
// w * g is accumulated as round(w * g * 2^(30 - e)), below 2^30 in magnitude, so a task's records cannot
// overflow 64 bits, the rounding is 2^-30 of the level's largest gradient per contribution, and a task's sum does
// not depend on the order of its records.  The tasks of a split bin are added in their order: a gradient has the same bits in
// every run.  A level whose gradient holds an inf or a nan gets nan in every row it touches.
//
// One MI355X, 16 levels of 2^19 rows, fp16, uniform points, gradient of the table in its own type (us): 2^14 points 47, 2^16 62, 2^17 79, 2^18 112,
// 2^20 350, 2^21 648; along rays 2^18 127, 2^20 402.  (Before the levels were dealt to fill workgroups and the accumulation asked for the next
// chunk's records ahead of the finished tile's way out: 100, 108, 114, 144, 379, 680; 158, 436.)
//
// Arithmetic (cell, corner rows, weights) is the forward's, see hash_encoding.hip.
#include "hash_common.h"

namespace nf {

constexpr int BIN_ROWS_LOG2 = 13;
constexpr int BIN_ROWS = 1 << BIN_ROWS_LOG2;  // rows per bin (two 64-bit sums each: 128 KiB of LDS in the accumulation)
constexpr uint32_t BIN_MASK = BIN_ROWS - 1;
constexpr int W_BITS = 19;
constexpr uint32_t W_MAX = (1u << W_BITS) - 1u;
// A fill workgroup (a block of records per level): small ones leave four to a unit, each covering the others' barriers.  With
// more than FILL_WIDE_BINS bins on a level the runs of a bin inside a block get short, and a wide workgroup makes them longer;
// a batch of less than FILL_WIDE_POINTS would leave half of the chip without one.
constexpr int FILL_THREADS = 512, FILL_WIDE_THREADS = 1024;
constexpr int fill_points(bool wide) { return wide ? 2 * FILL_WIDE_THREADS : FILL_THREADS; }
constexpr int FILL_WIDE_BINS = 128;
constexpr int64_t FILL_WIDE_POINTS = (int64_t)1 << 18;
constexpr int64_t FILL_ROWS_BYTES = (int64_t)224 << 20;
constexpr int ACC_THREADS = 1024;             // of sixteen waves
constexpr int ACC_INFLIGHT = 2;               // records in flight per thread
constexpr int GROUP = 16;                     // records named by one entry of a task's list
constexpr int LIST = 5760;                    // entries of the list that LDS holds at a time
constexpr int LIST_PAD = 2 * ACC_THREADS * ACC_INFLIGHT / GROUP;  // empty entries behind it
constexpr int SPLIT_MAX_BINS = 1536;          // bins whose tasks LDS has a table for: those of the coarse levels, where points meet
// Of the bins behind them only those of LATE_SHARES shares and more are split, listed one by one: all levels together come to 768 shares, and
// of sixteen levels at most nine are behind, so LATE_MAX takes them (beyond it the shares grow).
// Points in one cell and in a cube of 0.003, 16 levels of 2^21 rows, fp16 (us; these bins unsplit, this): 2^18 points 1690 and 1110, 800 and 575;
// 2^20 points 5960 and 1720, 1710 and 1245; uniform points 311 -> 317 and 506 -> 508.
constexpr uint32_t LATE_SHARES = 2;
constexpr int LATE_MAX = 256;
constexpr uint32_t CELL_COST = 4;             // a cell record is sixteen LDS adds against an x-pair record's four
constexpr int MAX_BINS_PER_LEVEL = 2048;        // 2^24 rows
struct BinPlan {
  int n_levels;
  int nbins[NF_MAX_LEVELS];
  int binbase[NF_MAX_LEVELS + 1];  // first global bin of the level
  int cell_levels;                 // leading levels whose records are cells (one per point) instead of x-pairs
  int split_bins;                  // bins of the leading levels whose tasks LDS has a table for
  int64_t record_base[NF_MAX_LEVELS];  // first record of the level's blocks
  int block_records[NF_MAX_LEVELS];    // room of one block
};

// cell record = {u | qx << 14,  qy | qz << 16,  packed gradient pair}: u = row of corner 0 minus the bin's first row,
// plus BIN_ROWS (the cell may start in the bin below); q* = the cell fractions in 18 / 16 / 16-bit fixed point
constexpr float CELL_QX = 262143.0f, CELL_QYZ = 65535.0f;
__device__ __forceinline__ uint3 make_cell_record(int32_t rel_row, const float (&fr)[3], uint32_t packed) {
  const uint32_t qx = (uint32_t)(fr[0] * CELL_QX + 0.5f), qy = (uint32_t)(fr[1] * CELL_QYZ + 0.5f), qz = (uint32_t)(fr[2] * CELL_QYZ + 0.5f);
  return make_uint3((uint32_t)(rel_row + BIN_ROWS) | qx << 14, qy | qz << 16, packed);
}

struct BinHeader {  // cleared by the fill kernel's first workgroup for the kernels behind it
  uint32_t next_task, n_splits, pad[2];
  uint32_t gmax[NF_MAX_LEVELS];  // largest |dout| bit pattern of every level
};

// A bin cut into several tasks, each leaving its sums in a slot (of BIN_ROWS rows of two) of its own.
struct BinSplit {
  uint32_t bin, slot, n, pad;
};

struct BinWs {
  BinHeader* header;
  uint32_t* totals;     // records of every bin (cleared with the header)
  uint32_t* block_max;  // [levels][blocks] largest |dout| bit pattern
  BinSplit* splits;
  uint16_t* starts;     // [blocks][start_stride]: place of every bin inside the block, one more per level for its end
  void* slots;          // of 64-bit fixed point (`whole_slots`) or of floats
  uint32_t* records;    // 3 words per record (16-bit gradient) or 4 (float32 gradient)
  uint32_t max_slots, split_cost;
  int start_stride, blocks, whole_slots;
};

// record = {row0 | row1 << 13 | w1[18:13] << 26,  w0 | w1[12:0] << 19,  packed gradient pair}
__device__ __forceinline__ uint3 make_record(uint32_t row0, uint32_t row1, float w0, float w1, uint32_t packed) {
  const uint32_t q0 = (uint32_t)(w0 * (float)W_MAX + 0.5f), q1 = (uint32_t)(w1 * (float)W_MAX + 0.5f);
  return make_uint3(row0 | row1 << BIN_ROWS_LOG2 | (q1 >> 13) << 26, q0 | (q1 & 0x1fffu) << W_BITS, packed);
}

struct Located3 {
  uint32_t c[3];
  float fr[3];
};
template <int VD>
__device__ __forceinline__ Located3 locate(const float (&v)[VD], float fres) {
  Located3 r;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float pos = v[d] * fres;
    const float fl = floorf(pos);
    r.c[d] = cell_index(fl, fres);
    r.fr[d] = pos - fl;
  }
  return r;
}
__device__ __forceinline__ void load_point(const void* coords, int cdt, int64_t csn, int64_t csd, int64_t n, float scale,
                                           float (&v)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    v[d] = load_as_f32(coords, n * csn + d * csd, cdt);
    if (scale != 1.0f) v[d] = v[d] / scale;
  }
}

// Dimensions beyond the third (sorted-record kernels, 4-D to 6-D points): a 4-D cell is its 3-D cell twice, once per
// corner of the fourth coordinate, so the 3-D pipeline runs once per such corner (`hi`, one bit per extra dimension).  The
// extra coordinates enter a pass as one term of the hash (xor), one of the dense index (add) and one factor of the weights.
struct ExtraDims {
  uint32_t hx;     // xor term of the 32-bit hash (hashed levels of a power of two of rows)
  uint64_t hx64;   // the same in 64 bits (hashed levels of any other size)
  uint32_t add;    // term of the dense index
  float w;         // factor of every corner weight
};
template <int DX, int VD>
__device__ __forceinline__ ExtraDims extra_dims(const float (&v)[VD], float fres, uint32_t res, int hi, const int64_t* primes) {
  static_assert(VD >= 3 + DX, "coordinate array too short");
  ExtraDims e = {0u, 0ull, 0u, 1.0f};
  uint32_t stride = res * res * res;
#pragma unroll
  for (int d = 0; d < DX; ++d) {
    const float pos = v[3 + d] * fres;
    const float fl = floorf(pos);
    const uint32_t bit = (uint32_t)(hi >> d) & 1u;
    const uint32_t c = cell_index(fl, fres) + bit;
    const float fr = pos - fl;
    e.hx ^= c * (uint32_t)primes[3 + d];
    e.hx64 ^= (uint64_t)c * (uint64_t)primes[3 + d];
    e.add += c * stride;
    stride *= res;
    const float wd = bit ? fr : 1.0f - fr;
    e.w = d == 0 ? wd : e.w * wd;
  }
  return e;
}

// Table rows (and trilinear / bilinear weights) of the 2^D corners of a point's cell, corner j = bit pattern of its
// offsets with x in bit 0, so that corners 2c and 2c+1 are an x-pair.  D = 3 or 2.
// A hashed level whose size is not a power of two takes the exact remainder of the 64-bit hash (the reference's
// CPU form) instead of the 32-bit wrap-around and mask.
template <int D, int VD>
__device__ __forceinline__ void cell_rows(const float (&v)[VD], float fres, bool hashed, uint32_t res, uint32_t mask,
                                          const uint32_t (&pi)[3], const int64_t* primes, uint32_t (&row)[1 << D], float* w,
                                          const ExtraDims* ex = nullptr) {
  const uint32_t n_rows = mask + 1u;
  if constexpr (D != 2 && D != 3) {
    // one, or more than three dimensions (the walk without records only): the per-(point, level) kernels' exact forms
    static_assert(VD >= D, "coordinate array too short");
    uint64_t p64[D];
#pragma unroll
    for (int d = 0; d < D; ++d) p64[d] = (uint64_t)primes[d];
    const Cell<D> cell = locate_cell<D>(v, (int)res);
#pragma unroll
    for (int j = 0; j < (1 << D); ++j) {
      const uint32_t r = (uint32_t)corner_row<D>(cell, j, hashed, res, n_rows, p64);
      row[j] = r < n_rows ? r : mask;  // (every row is inside its level; the tile that takes it is sized by the level)
      if (w != nullptr) w[j] = corner_weight<D>(cell, j);
    }
    return;
  } else {
  if (hashed && (n_rows & mask) != 0u) {
    uint32_t c[D];
    float fr[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const float pos = v[d] * fres;
      const float fl = floorf(pos);
      c[d] = cell_index(fl, fres);
      fr[d] = pos - fl;
    }
#pragma unroll
    for (int j = 0; j < (1 << D); ++j) {
      uint64_t h = 0;
#pragma unroll
      for (int d = 0; d < D; ++d) h ^= (uint64_t)(c[d] + ((j >> d) & 1)) * (uint64_t)primes[d];
      if (ex != nullptr) h ^= ex->hx64;
      row[j] = (uint32_t)(h % (uint64_t)n_rows);
    }
    if (w != nullptr) {
      if (D == 3) {
        weights_d3(fr, w);
        if (ex != nullptr)
#pragma unroll
          for (int j = 0; j < 8; ++j) w[j] = w[j] * ex->w;
      } else {
        const float gx = 1.0f - fr[0], gy = 1.0f - fr[1];
        w[0] = gx * gy;
        w[1] = fr[0] * gy;
        w[2] = gx * fr[1];
        w[3] = fr[0] * fr[1];
      }
    }
    return;
  }
  if (D == 3) {
    const Located3 q = locate(v, fres);
    const Corner8 r = rows_d3(q.c, hashed, res, mask, pi);
#pragma unroll
    for (int j = 0; j < (1 << D); ++j) row[j] = r.row[j];
    if (w != nullptr) weights_d3(q.fr, w);
    if (ex != nullptr) {
      // (a & m) ^ (b & m) == (a ^ b) & m: the extra xor term joins the masked rows; dense rows take the extra index term
      const uint32_t hx = ex->hx & mask;
#pragma unroll
      for (int j = 0; j < (1 << D); ++j) row[j] = hashed ? (row[j] ^ hx) : row[j] + ex->add;
      if (w != nullptr)
#pragma unroll
        for (int j = 0; j < (1 << D); ++j) w[j] = w[j] * ex->w;
    }
  } else {
    uint32_t c[2];
    float fr[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const float pos = v[d] * fres;
      const float fl = floorf(pos);
      c[d] = cell_index(fl, fres);
      fr[d] = pos - fl;
    }
    if (hashed) {
      const uint32_t x0 = c[0] * pi[0], x1 = x0 + pi[0], y0 = c[1] * pi[1], y1 = y0 + pi[1];
      row[0] = (x0 ^ y0) & mask;
      row[1] = (x1 ^ y0) & mask;
      row[2] = (x0 ^ y1) & mask;
      row[3] = (x1 ^ y1) & mask;
    } else {
      const uint32_t b = c[0] + c[1] * res;
      row[0] = b;
      row[1] = b + 1;
      row[2] = b + res;
      row[3] = min(b + res + 1, mask);  // as in rows_d2: the zero-weight corner of x == scale stays inside the level
    }
    if (w != nullptr) {
      const float gx = 1.0f - fr[0], gy = 1.0f - fr[1];
      w[0] = gx * gy;
      w[1] = fr[0] * gy;
      w[2] = gx * fr[1];
      w[3] = fr[0] * fr[1];
    }
  }
  }
}
template <int D, int VD>
__device__ __forceinline__ void load_point_d(const void* coords, int cdt, int64_t csn, int64_t csd, int64_t n, float scale,
                                             float (&v)[VD]) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    v[d] = load_as_f32(coords, n * csn + d * csd, cdt);
    if (scale != 1.0f) v[d] = v[d] / scale;
  }
}

// Largest value of a wave, valid in lane 63: prefix maxima inside each row of 16 lanes, then lane 15 of rows 0 / 2 into
// rows 1 / 3 and lane 31 into rows 2 / 3 (data-parallel primitives of the vector ALU; nothing goes through LDS).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t m) {
  auto step = [](uint32_t v, uint32_t shifted) { return shifted > v ? shifted : v; };
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x111, 0xf, 0xf, false));  // row_shr:1
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x112, 0xf, 0xf, false));  // row_shr:2
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x114, 0xf, 0xf, false));  // row_shr:4
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x118, 0xf, 0xf, false));  // row_shr:8
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x142, 0xa, 0xf, false));  // row_bcast:15 -> rows 1, 3
  m = step(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x143, 0xc, 0xf, false));  // row_bcast:31 -> rows 2, 3
  return m;
}

// ---------------------------------------------------------------------------------------
// fill
// ---------------------------------------------------------------------------------------
// A workgroup takes some of the levels (blockIdx.y), or all of them: a batch that leaves a unit one workgroup pays every level's barriers in turn (44 us for
// sixteen levels at 2^14 to 2^17 points), several groups of levels cover each other's.
// A level goes through three barriers: ranks inside the bins (LDS adds on one counter per bin), an exclusive scan of the
// counters by one wave, the records into the stage in sorted order, and the stage out to the block.  The copy-out of a level runs
// beside the hashing of the next one, and two or three workgroups per unit cover each other's barriers.
// 16-bit upstream gradient: 12-byte records {.., .., packed pair}; float32 (G32): 16-byte records {.., .., g0, g1}.
// A stage holds a little more than the usual number of records; the rare ones behind it (pairs split over two bins) go
// straight to their place.
// DX: dimensions beyond the third (D == 3 then); hi: which corner of them this pass covers
constexpr int stage_records(int D, bool wide) { return fill_points(wide) * (D == 3 ? 4 : 2) + 256; }

typedef uint32_t Words4 __attribute__((ext_vector_type(4)));

template <bool WIDE, bool G32, int D, int DX = 0>
__global__ __launch_bounds__(WIDE ? FILL_WIDE_THREADS : FILL_THREADS, WIDE || G32 || DX ? 4 : 8) void hash_bwd_bin_fill_k(const void* coords, int cdt, int64_t csn, int64_t csd,
                                                                    const void* dout_v, int64_t dout_stride, int64_t N, int points,
                                                                    DevGeom g, BinPlan bp, const int64_t* primes, float scale,
                                                                    BinWs ws, int max_nb, int feat, int f0, int hi, int step) {
  extern __shared__ __align__(16) uint32_t fill_smem[];
  constexpr int RW = G32 ? 4 : 3;  // words of a record
  constexpr int THREADS = WIDE ? FILL_WIDE_THREADS : FILL_THREADS, POINTS = fill_points(WIDE), PPT = POINTS / THREADS;
  constexpr uint32_t ROOM = stage_records(D, WIDE);
  constexpr int PAIRS = 1 << (D - 1);
  uint32_t* stage = fill_smem;               // [ROOM][RW], sorted by bin
  uint32_t* cnt0 = stage + ROOM * RW;        // [2][max_nb] records per bin of this level and of the next one
  uint32_t* start = cnt0 + 2 * max_nb;       // [max_nb + 1] first record of every bin
  uint32_t* lmax = start + max_nb + 1;       // [levels] largest |dout| pattern
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n0 = (int64_t)blockIdx.x * points;
  const int here = N - n0 < points ? (int)(N - n0) : points;
  const int l_first = (int)blockIdx.y * step, l_end = min(l_first + step, bp.n_levels);  // the levels of this workgroup
  if (blockIdx.x == 0 && blockIdx.y == 0)  // the header and the totals behind it
    for (int i = tid; i < (int)(sizeof(BinHeader) / 4) + bp.binbase[bp.n_levels]; i += THREADS) reinterpret_cast<uint32_t*>(ws.header)[i] = 0u;
  for (int i = tid; i < 2 * max_nb; i += THREADS) cnt0[i] = 0u;
  if (tid < NF_MAX_LEVELS) lmax[tid] = 0u;
  float v[PPT][3 + DX] = {};
  bool valid[PPT];
  int64_t n[PPT];
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    // neighbouring lanes take points sixteen apart: along a ray neighbours share a cell, and the accumulation's lanes, which follow
    // the order of the records, would add to the same few rows (64 adds to one address one after the other)
    const int k = lane * (POINTS / 64) + wave * PPT + i;
    valid[i] = k < here;
    n[i] = n0 + (valid[i] ? k : 0);
    load_point_d<D + DX>(coords, cdt, csn, csd, n[i], scale, v[i]);
  }
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], D > 2 ? (uint32_t)primes[D > 2 ? 2 : 0] : 0u};
  // The gradient pairs (features f0, f0 + 1) of four levels are read together: rows of 2, 4 or 8 features in 16-byte pieces where
  // they are aligned, pair by pair otherwise.
  const bool row_vec = !G32 && (feat == 2 || feat == 4 || feat == 8) && (bp.n_levels & 3) == 0 && ((uintptr_t)dout_v & 15u) == 0 && (dout_stride & 7) == 0;
  const bool row_vec32 = G32 && feat == 2 && (bp.n_levels & 3) == 0 && ((uintptr_t)dout_v & 15u) == 0 && (dout_stride & 3) == 0;
  const int pair_in_level = f0 >> 1;
  auto word = [](const uint4& q, int c) { return c == 0 ? q.x : c == 1 ? q.y : c == 2 ? q.z : q.w; };
  uint32_t quad[PPT][4][G32 ? 2 : 1];
  auto load_quad = [&](int l0) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      if constexpr (G32) {
        const float* row = reinterpret_cast<const float*>(dout_v) + n[i] * dout_stride;
        if (row_vec32) {
          const uint4 a = *reinterpret_cast<const uint4*>(row + 2 * l0), b = *reinterpret_cast<const uint4*>(row + 2 * l0 + 4);
          quad[i][0][0] = a.x; quad[i][0][1] = a.y; quad[i][1][0] = a.z; quad[i][1][1] = a.w;
          quad[i][2][0] = b.x; quad[i][2][1] = b.y; quad[i][3][0] = b.z; quad[i][3][1] = b.w;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int e = (l0 + q) * feat + f0;
            const bool in = l0 + q < bp.n_levels;
            quad[i][q][0] = in ? __float_as_uint(row[e]) : 0u;
            quad[i][q][1] = in && f0 + 1 < feat ? __float_as_uint(row[e + 1]) : 0u;  // an odd feature count: the last has no partner
          }
        }
      } else {
        const uint16_t* row = reinterpret_cast<const uint16_t*>(dout_v) + n[i] * dout_stride;
        if (row_vec) {
          const uint4* g4 = reinterpret_cast<const uint4*>(row);
          uint4 t;
          const int q0 = l0 >> 2;
          if (feat == 2) {
            t = g4[q0];
          } else if (feat == 4) {
            const uint4 a = g4[2 * q0], b = g4[2 * q0 + 1];
            t = pair_in_level ? make_uint4(a.y, a.w, b.y, b.w) : make_uint4(a.x, a.z, b.x, b.z);
          } else {
            t = make_uint4(word(g4[4 * q0], pair_in_level), word(g4[4 * q0 + 1], pair_in_level), word(g4[4 * q0 + 2], pair_in_level),
                           word(g4[4 * q0 + 3], pair_in_level));
          }
          quad[i][0][0] = t.x; quad[i][1][0] = t.y; quad[i][2][0] = t.z; quad[i][3][0] = t.w;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int e = (l0 + q) * feat + f0;
            uint32_t packed = 0u;
            if (l0 + q < bp.n_levels) {
              packed = row[e];
              if (f0 + 1 < feat) packed |= (uint32_t)row[e + 1] << 16;
            }
            quad[i][q][0] = packed;
          }
        }
      }
    }
  };
  lds_barrier();

  for (int l = l_first; l < l_end; ++l) {
    const int nb = bp.nbins[l];
    uint32_t* cnt = cnt0 + (l & 1) * max_nb;
    if (l == l_first || (l & 3) == 0) load_quad(l & ~3);
    uint32_t gp[PPT][G32 ? 2 : 1], m = 0u;
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
#pragma unroll
      for (int e = 0; e < (G32 ? 2 : 1); ++e) {
        const int q = l & 3;
        gp[i][e] = q == 0 ? quad[i][0][e] : q == 1 ? quad[i][1][e] : q == 2 ? quad[i][2][e] : quad[i][3][e];
      }
      if (!valid[i]) continue;
      // largest |g| of the level: positive float patterns order like integers
      if constexpr (G32) {
        m = max(m, max(gp[i][0] & 0x7fffffffu, gp[i][1] & 0x7fffffffu));
      } else {
        const uint32_t pk = gp[i][0] & 0x7fff7fffu;
        m = max(m, max(pk & 0xffffu, pk >> 16));
      }
    }
    m = wave_max_u32(m);
    if (lane == 63 && m) atomicMax(lmax + l, m);

    // the records, and their ranks inside the bins: {bin, rank << 12}; ~0 where a pair does not reach into a second bin
    uint32_t rx[PPT][PAIRS], ry[PPT][PAIRS], at[PAIRS * PPT], at2[PAIRS * PPT];
    bool cells = false;
    if constexpr (D == 3 && !G32 && DX == 0) cells = l < bp.cell_levels;
    const int per_point = cells ? 1 : PAIRS;
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      if (cells) {
        if constexpr (D == 3 && !G32 && DX == 0) {
          const uint32_t res = (uint32_t)g.res[l];
          const Located3 q = locate(v[i], (float)g.res[l]);
          const uint32_t b = q.c[0] + q.c[1] * res + q.c[2] * res * res;
          const uint32_t k0 = b >> BIN_ROWS_LOG2, k1 = (b + res * res + res + 1u) >> BIN_ROWS_LOG2;
          const uint3 rec = make_cell_record((int32_t)(b - (k0 << BIN_ROWS_LOG2)), q.fr, 0u);
          rx[i][0] = rec.x;
          ry[i][0] = rec.y;
          at[i * PAIRS] = k0;
          at2[i * PAIRS] = valid[i] && k1 != k0 ? k1 : ~0u;
        }
      } else {
        uint32_t row[1 << D];
        float w[1 << D];
        if constexpr (DX > 0) {
          const ExtraDims ex = extra_dims<DX>(v[i], (float)g.res[l], (uint32_t)g.res[l], hi, primes);
          cell_rows<D>(v[i], (float)g.res[l], l >= g.first_hash, (uint32_t)g.res[l], g.rows[l] - 1u, pi, primes, row, w, &ex);
        } else {
          cell_rows<D>(v[i], (float)g.res[l], l >= g.first_hash, (uint32_t)g.res[l], g.rows[l] - 1u, pi, primes, row, w);
        }
#pragma unroll
        for (int c = 0; c < PAIRS; ++c) {
          const uint32_t r0 = row[2 * c], r1 = row[2 * c + 1], k0 = r0 >> BIN_ROWS_LOG2, k1 = r1 >> BIN_ROWS_LOG2;
          const uint3 rec = make_record(r0 & BIN_MASK, r1 & BIN_MASK, w[2 * c], w[2 * c + 1], 0u);
          rx[i][c] = rec.x;
          ry[i][c] = rec.y;
          at[i * PAIRS + c] = k0;
          at2[i * PAIRS + c] = valid[i] && k1 != k0 ? k1 : ~0u;
        }
      }
    }
    // all ranks of the thread asked for together: a wave waits for LDS once per level
    if (nb > 1) {
      uint32_t rank[PAIRS * PPT];
#pragma unroll
      for (int k = 0; k < PAIRS * PPT; ++k)
        rank[k] = valid[k / PAIRS] && k % PAIRS < per_point ? atomicAdd(cnt + at[k], 1u) : 0u;
#pragma unroll
      for (int k = 0; k < PAIRS * PPT; ++k) at[k] |= rank[k] << 12;
      bool more = false;
#pragma unroll
      for (int k = 0; k < PAIRS * PPT; ++k) more = more || (k % PAIRS < per_point && at2[k] != ~0u);
      if (__any(more)) {
#pragma unroll
        for (int k = 0; k < PAIRS * PPT; ++k)
          if (k % PAIRS < per_point && at2[k] != ~0u) at2[k] |= atomicAdd(cnt + at2[k], 1u) << 12;
      }
    } else {
#pragma unroll
      for (int k = 0; k < PAIRS * PPT; ++k) {
        const int i = k / PAIRS;  // a full block in the order of the threads, a ragged one in the order of its points
        const int p = here == POINTS ? tid + THREADS * i : lane * (POINTS / 64) + wave * PPT + i;
        at[k] = (uint32_t)(p * per_point + k % PAIRS) << 12;
      }
    }
    lds_barrier();
    // exclusive scan of the counters: into LDS for this workgroup, and out for the plan; the other waves clear the next
    // level's counters
    uint16_t* out_start = ws.starts + (int64_t)blockIdx.x * ws.start_stride + bp.binbase[l] + l;
    if (wave == 0) {
      if (nb == 1) {
        if (lane == 0) {
          start[0] = 0u;
          start[1] = (uint32_t)(here * per_point);
          out_start[0] = 0;
          out_start[1] = (uint16_t)(here * per_point);
        }
      } else {
        uint32_t run = 0;
        for (int b0 = 0; b0 < nb; b0 += 64) {
          const int b = b0 + lane;
          const uint32_t c = b < nb ? cnt[b] : 0u;
          uint32_t incl = c;
#pragma unroll
          for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
            if (lane >= d) incl += y;
          }
          const uint32_t excl = run + incl - c;
          if (b < nb) {
            start[b] = excl;
            out_start[b] = (uint16_t)excl;
          }
          run += (uint32_t)__shfl((int)incl, 63);
        }
        if (lane == 0) {
          start[nb] = run;
          out_start[nb] = (uint16_t)run;
        }
      }
    } else {
      uint32_t* other = cnt0 + ((l + 1) & 1) * max_nb;
      for (int i = tid - 64; i < max_nb; i += THREADS - 64) other[i] = 0u;
    }
    lds_barrier();
    const uint32_t room = (uint32_t)bp.block_records[l];
    uint32_t* block = ws.records + (bp.record_base[l] + (int64_t)blockIdx.x * room) * RW;
    auto put = [&](uint32_t pos, uint32_t x, uint32_t y, int i) {
      if (pos < ROOM) {
        stage[pos * RW] = x;
        stage[pos * RW + 1] = y;
        stage[pos * RW + 2] = gp[i][0];
        if constexpr (G32) stage[pos * RW + 3] = gp[i][1];
      } else {
        block[pos * RW] = x;
        block[pos * RW + 1] = y;
        block[pos * RW + 2] = gp[i][0];
        if constexpr (G32) block[pos * RW + 3] = gp[i][1];
      }
    };
    bool more = false;
#pragma unroll
    for (int k = 0; k < PAIRS * PPT; ++k) {
      const int i = k / PAIRS, c = k % PAIRS;
      if (!valid[i] || c >= per_point) continue;
      const bool split = at2[k] != ~0u;
      more = more || split;
      uint32_t x = rx[i][c], y = ry[i][c];
      if (split && !cells) {  // the second corner leaves as a record of its own
        x = (x & BIN_MASK) | (x & BIN_MASK) << BIN_ROWS_LOG2;
        y &= W_MAX;
      }
      put(start[at[k] & 0xfffu] + (at[k] >> 12), x, y, i);
    }
    if (__any(more)) {
#pragma unroll
      for (int k = 0; k < PAIRS * PPT; ++k) {
        const int i = k / PAIRS, c = k % PAIRS;
        if (!valid[i] || c >= per_point || at2[k] == ~0u) continue;
        const uint32_t x = rx[i][c], y = ry[i][c];
        const uint32_t pos = start[at2[k] & 0xfffu] + (at2[k] >> 12);
        if (cells) {
          put(pos, x - (((at2[k] & 0xfffu) - (at[k] & 0xfffu)) << BIN_ROWS_LOG2), y, i);  // the same cell seen from the next bin
        } else {
          const uint32_t r1 = (x >> BIN_ROWS_LOG2) & BIN_MASK, w1 = (x >> 26) << 13 | y >> W_BITS;
          put(pos, r1 | r1 << BIN_ROWS_LOG2, w1, i);
        }
      }
    }
    lds_barrier();
    // The stage leaves as it is: whole 16-byte pieces, the last one perhaps with words of no meaning behind the end; past the caches,
    // which the records of a batch overflow anyway (fill 199 -> 180 us and accum 212 -> 189 us at 2^20 points).
    const uint32_t pieces = (min(start[nb], ROOM) * RW + 3u) / 4u;
    for (uint32_t i = tid; i < pieces; i += THREADS) __builtin_nontemporal_store(reinterpret_cast<const Words4*>(stage)[i], reinterpret_cast<Words4*>(block) + i);
  }
  if (tid >= l_first && tid < l_end) ws.block_max[(int64_t)tid * ws.blocks + blockIdx.x] = lmax[tid];
}

// ---------------------------------------------------------------------------------------
// totals: a workgroup adds up 64 bins of some blocks (and takes the largest |dout| of the level)
// ---------------------------------------------------------------------------------------
// Bound by the latency of its loads, so a wave reads few blocks; and by the atomics of the workgroups, so those take many blocks.  A wave alone
// with 64 blocks 10 us at 2^20 points (each with 8 of them 38), this 6.
constexpr int TOTALS_WAVES = 16, TOTALS_ROWS = 16, TOTALS_BLOCKS = TOTALS_WAVES * TOTALS_ROWS;
typedef uint32_t TwoStarts __attribute__((aligned(2)));  // places of two neighbouring bins in a block: first | second << 16
__global__ __launch_bounds__(64 * TOTALS_WAVES) void hash_bwd_bin_totals_k(BinWs ws, BinPlan bp) {
  __shared__ uint32_t part[TOTALS_WAVES][64], largest[TOTALS_WAVES];
  int first = blockIdx.x, l = 0;  // blockIdx.x counts pieces of 64 bins over all levels
  for (;; ++l) {
    const int pieces = (bp.nbins[l] + 63) / 64;
    if (first < pieces) break;
    first -= pieces;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int w0 = blockIdx.y * TOTALS_BLOCKS + wave * TOTALS_ROWS, w1 = min(w0 + TOTALS_ROWS, ws.blocks);
  const int b = first * 64 + lane;
  uint32_t sum = 0;
  if (b < bp.nbins[l]) {
    const uint16_t* mine = ws.starts + (int64_t)w0 * ws.start_stride + bp.binbase[l] + l + b;
#pragma unroll TOTALS_ROWS
    for (int w = w0; w < w1; ++w, mine += ws.start_stride) {
      const uint32_t two = *reinterpret_cast<const TwoStarts*>(mine);
      sum += (two >> 16) - (two & 0xffffu);
    }
  }
  part[wave][lane] = sum;
  if (first == 0) {
    const uint32_t m = wave_max_u32(lane < w1 - w0 ? ws.block_max[(int64_t)l * ws.blocks + w0 + lane] : 0u);
    if (lane == 63) largest[wave] = m;
  }
  lds_barrier();
  if (wave == 0) {
    sum = 0;
#pragma unroll
    for (int w = 0; w < TOTALS_WAVES; ++w) sum += part[w][lane];
    if (sum) atomicAdd(ws.totals + bp.binbase[l] + b, sum);
    if (first == 0) {
      const uint32_t m = wave_max_u32(lane < TOTALS_WAVES ? largest[lane] : 0u);
      if (lane == 63 && m) atomicMax(ws.header->gmax + l, m);
    }
  }
}

// Sums of the lanes up to each one, inside rows of 16 and over the whole wave (the moves of wave_max_u32).
__device__ __forceinline__ uint32_t row_scan_u32(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
  return x;
}
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t x) {
  x = row_scan_u32(x);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
  return x;
}

// Sum of the threads in front of this one, of a workgroup of sixteen waves: one barrier.  `sums` alternates between two arrays from one
// call to the next, so that a wave may still read one while another writes the other.
constexpr int ACC_WAVES = 16;
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t x, uint32_t* sums, uint32_t* total) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t incl = wave_scan_u32(x);
  if (lane == 63) sums[wave] = incl;
  lds_barrier();
  const uint32_t up_to = row_scan_u32(sums[lane & (ACC_WAVES - 1)]);
  *total = (uint32_t)__builtin_amdgcn_readlane((int)up_to, ACC_WAVES - 1);
  return (wave ? (uint32_t)__builtin_amdgcn_readlane((int)up_to, wave - 1) : 0u) + incl - x;
}

// ---------------------------------------------------------------------------------------
// accumulate
// ---------------------------------------------------------------------------------------
// record type and gradient decode per upstream-gradient dtype
template <typename GT>
struct BinRec {
  typedef uint3 type;
  __device__ static __forceinline__ type zero() { return make_uint3(0u, 0u, 0u); }
  __device__ static __forceinline__ float g0(const type& q) { return GT::to_f32((uint16_t)(q.z & 0xffffu)); }
  __device__ static __forceinline__ float g1(const type& q) { return GT::to_f32((uint16_t)(q.z >> 16)); }
  __device__ static __forceinline__ float level_max(uint32_t pattern) { return GT::to_f32((uint16_t)pattern); }
};
template <>
struct BinRec<F32> {
  typedef uint4 type;
  __device__ static __forceinline__ type zero() { return make_uint4(0u, 0u, 0u, 0u); }
  __device__ static __forceinline__ float g0(const type& q) { return __uint_as_float(q.z); }
  __device__ static __forceinline__ float g1(const type& q) { return __uint_as_float(q.w); }
  __device__ static __forceinline__ float level_max(uint32_t pattern) { return __uint_as_float(pattern); }
};

// Nearest integer (halves upwards) of |x| < 2^31, in one instruction; __float2int_rn() takes two.
__device__ __forceinline__ int32_t round_to_int(float x) {
  int32_t r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// Fixed-point scale 2^se of a level whose largest |gradient| is gm:  |w * g| * 2^se < 2^30.  A level with an inf or a nan has none.
struct FixedPoint {
  int se;
  bool nonfinite;
  __device__ __forceinline__ explicit FixedPoint(float gm) : se(0), nonfinite(!(gm <= 3.0e38f)) {
    if (nonfinite || !(gm > 0.0f)) return;
    int ex;
    frexpf(gm, &ex);
    se = 30 - ex;
    se = se > 120 ? 120 : se;
  }
  // A sum a of these: |a| <= 2^30 * 2^21 points < 2^53, exact in double, and so is its quotient by 2^se: one rounding, to float, at the end
  struct ToFloat {
    double lo, hi;
    bool nonfinite;
    __device__ __forceinline__ float operator()(long long a) const {
      const float x = (float)((double)(int)(a >> 32) * hi + (double)(uint32_t)a * lo);
      return nonfinite && a != 0 ? __uint_as_float(0x7fc00000u) : x;
    }
  };
  __device__ __forceinline__ ToFloat to_float() const { return {ldexp(1.0, -se), ldexp(1.0, 32 - se), nonfinite}; }
};

// How a sum reaches the gradient table.
enum TableMode { TABLE_ADD = 0, TABLE_F32 = 1, TABLE_F16 = 2, TABLE_BF16 = 3 };  // added to float32, or written in a type of its own
template <int MODE>
__device__ __forceinline__ void store_table(void* table, int64_t i, float x) {
  if constexpr (MODE == TABLE_ADD || MODE == TABLE_F32) reinterpret_cast<float*>(table)[i] = x;
  else if constexpr (MODE == TABLE_F16) reinterpret_cast<uint16_t*>(table)[i] = F16::from_f32(x);
  else reinterpret_cast<uint16_t*>(table)[i] = BF16::from_f32(x);
}

// two features of a row (one if not `pair`); whole: the row is these two (one access)
template <int MODE>
__device__ __forceinline__ void store_pair(void* table, int64_t i, float x, float y, bool whole, bool pair) {
  if (whole) {
    if constexpr (MODE == TABLE_F32) *reinterpret_cast<float2*>(reinterpret_cast<float*>(table) + i) = make_float2(x, y);
    else if constexpr (MODE == TABLE_F16) *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(table) + i) = F16::pack(x, y);
    else *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(table) + i) = BF16::pack(x, y);
  } else {
    store_table<MODE>(table, i, x);
    if (pair) store_table<MODE>(table, i + 1, y);
  }
}

template <int MODE>
__device__ __forceinline__ void add_or_store_pair(void* table, int64_t i, float x, float y, bool whole, bool pair) {
  if constexpr (MODE == TABLE_ADD) {
    float* cell = reinterpret_cast<float*>(table) + i;
    if (x != 0.0f) cell[0] += x;
    if (pair && y != 0.0f) cell[1] += y;
  } else {
    store_pair<MODE>(table, i, x, y, whole, pair);
  }
}

// body(integral_constant) for the mode in use
template <typename Body>
__host__ __device__ __forceinline__ auto with_mode(int mode, Body&& body) {
  switch (mode) {
    case TABLE_ADD: return body(std::integral_constant<int, TABLE_ADD>{});
    case TABLE_F32: return body(std::integral_constant<int, TABLE_F32>{});
    case TABLE_F16: return body(std::integral_constant<int, TABLE_F16>{});
    default: return body(std::integral_constant<int, TABLE_BF16>{});
  }
}

// What bounds it: 2^20 points, 64-bit adds (108 us of the LDS pipe at the 4.6 lanes a clock and unit that random rows reach) next to 800 MB of
// records (130 us); what came on top were the phases of a task, one after the other.  A workgroup planned for 10 - 14 us before its first record (scans
// through LDS, an answer of the task counter, a search of the levels per bin; now 6 - 8), made a task's list in 3 - 5 us and waited for
// its first records behind that.  Now the next chunk's list is made when the last add is done and its records come while the tile leaves:
// 2^14 points 46 -> 26 us, 2^17 57 -> 42, 2^18 along rays added to float32 104 -> 87, 2^20 212 -> 190.  (Cells and pairs mixed, as cells keep the LDS pipe busy and
// pairs the memory: 2^20 uniform 351 instead of 356 us for the whole chain, 2^21 690 instead of 660, 2^17 along rays 109 instead of 96.)
// TWO: rows of two features have kernels of their own, which the addresses of other rows cost nine registers and 3 us at 2^18 points
template <typename GT, int MODE, bool TWO>
__global__ __launch_bounds__(ACC_THREADS) void hash_bwd_bin_accum_k(BinWs ws, void* table, DevGeom g, BinPlan bp, int row_feat, int f0) {
  typedef typename BinRec<GT>::type Rec;
  // Fixed-point sums, one plane of BIN_ROWS 64-bit cells per feature: the 64 lanes of an add go to random rows of one
  // feature, and with 8-byte cells those spread over all 64 banks (interleaved features would leave them half).
  extern __shared__ __align__(16) unsigned long long acc_tile[];
  uint32_t* list = reinterpret_cast<uint32_t*>(acc_tile + 2 * BIN_ROWS);  // [LIST + LIST_PAD] first word of up to GROUP records in the level | their number << 27
  uint32_t* first_task = list + LIST + LIST_PAD;                          // [SB + 1] first task of a bin | its first slot << 16
  __shared__ uint32_t next_task, wave_sums[2][ACC_WAVES], level_max[NF_MAX_LEVELS];
  const int tid = threadIdx.x, lane = tid & 63, feat = TWO ? 2 : row_feat;
  const int NB = bp.binbase[bp.n_levels], SB = bp.split_bins, cell_bins = bp.binbase[bp.cell_levels];
  // What has to come from memory is asked for first: the number of a second task, and the bins' totals
  // (An address that is the same in all lanes would have the compiler broadcast the counter's answer, that is, wait for it and for every load
  // in front of it: 0.7 - 2 us a task.)
  uint32_t lane_zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(lane_zero));
  uint32_t* const counter = &ws.header->next_task + lane_zero;
  uint32_t ticket = 0u;
  if (tid == 0) ticket = atomicAdd(counter, 1u);
  const uint32_t first_total = ws.totals[min(tid, NB - 1)], first_max = ws.header->gmax[min(tid, NF_MAX_LEVELS - 1)];
  const int level_base = lane < bp.n_levels ? bp.binbase[lane] : NB;  // of the lane's level
  uint32_t* late = first_task + SB + 1;  // [n_late + 1] heavy bins behind those: bin, its first further share | its first slot << 16
  static_assert(__alignof__(acc_tile) >= alignof(uint4), "the tile is cleared in 16-byte pieces");
  for (uint32_t i = tid; i < BIN_ROWS; i += ACC_THREADS) reinterpret_cast<uint4*>(acc_tile)[i] = make_uint4(0u, 0u, 0u, 0u);
  if (tid < NF_MAX_LEVELS) level_max[tid] = first_max;
  // The tasks, worked out by every workgroup for itself: one per bin of the leading levels, several for a bin of more than one and a half
  // shares; the further shares of heavy bins behind those; and one per bin behind them, which takes a heavy bin's first share.  Where
  // the slots (or the list of heavy bins) do not reach, larger shares.
  uint32_t split_tasks, late_tasks, n_late, turn = 0;
  const auto scan = [&](uint32_t x, uint32_t* total) { return block_exclusive_scan(x, wave_sums[turn++ & 1u], total); };
  const auto cost_of = [&](int b, uint32_t total) { return total * (b < cell_bins ? CELL_COST : 1u); };
  for (uint32_t share = ws.split_cost;; share += share / 4u) {
    const auto parts_of = [&](uint32_t cost) { return min((cost + share - 1u) / share, (uint32_t)ws.blocks); };
    uint32_t slots = 0, total;
    split_tasks = 0;
    for (int b0 = 0; b0 < SB; b0 += ACC_THREADS) {
      const int b = b0 + tid;
      uint32_t n = 0;
      if (b < SB) {
        const uint32_t cost = cost_of(b, b0 == 0 ? first_total : ws.totals[b]);
        n = cost <= share + share / 2 ? 1u : parts_of(cost);
        if (cost == 0u && MODE == TABLE_ADD) n = 0u;  // nothing to add (a table that is written gets its zeros)
      }
      // tasks and slots in one scan: neither comes to 2^16 (all levels together are at most 8 * 192 shares)
      const uint32_t before = scan(n | (n > 1u ? n : 0u) << 16, &total);
      if (b < SB) first_task[b] = (before & 0xffffu) + split_tasks | ((before >> 16) + slots) << 16;
      split_tasks += total & 0xffffu;
      slots += total >> 16;
    }
    n_late = late_tasks = 0u;
    if (SB < NB) {
      uint32_t heavy = 0, parts = 0;
      const auto each_heavy = [&](auto&& body) {
        for (int b = SB + tid; b < NB; b += ACC_THREADS) {
          const uint32_t cost = cost_of(b, ws.totals[b]);
          if (cost >= LATE_SHARES * ws.split_cost && cost > share + share / 2 && ws.blocks > 1) body(b, parts_of(cost));
        }
      };
      each_heavy([&](int, uint32_t n) {
        ++heavy;
        parts += n;
      });
      uint32_t at = scan(heavy, &n_late);
      uint32_t slot = slots + scan(parts, &total), first = slot - slots - at;
      slots += total;
      late_tasks = total - n_late;
      if (heavy && n_late <= (uint32_t)LATE_MAX)
        each_heavy([&](int b, uint32_t n) {
          late[2u * at] = (uint32_t)b;
          late[2u * at + 1u] = first | slot << 16;
          ++at;
          first += n - 1u;
          slot += n;
        });
    }
    if (slots <= ws.max_slots && n_late <= (uint32_t)LATE_MAX) break;
  }
  if (tid == 0) {
    first_task[SB] = split_tasks;
    late[2u * n_late + 1u] = late_tasks;
    next_task = gridDim.x + ticket;
  }
  lds_barrier();
  const uint32_t n_tasks = split_tasks + late_tasks + (uint32_t)(NB - SB);
  if (blockIdx.x >= n_tasks) return;
  // What a task needs, the same for all threads.
  struct Task {
    int bin, level, block0, block1;
    uint32_t slot;
  };
  auto task_of = [&](uint32_t t) {
    Task k = {SB + (int)(t - split_tasks - late_tasks), 0, 0, ws.blocks, ~0u};
    // share `which` of n: its blocks, and its slot
    auto share = [&](uint32_t which, uint32_t n, uint32_t slot) {
      if (n <= 1u) return;
      k.slot = slot + which;
      k.block0 = (int)((uint32_t)ws.blocks * which / n);  // (at most 4096 blocks, and no more shares than those)
      k.block1 = (int)((uint32_t)ws.blocks * (which + 1u) / n);
    };
    if (t < split_tasks) {
      // the bin whose first task is the last one not behind t (a bin without tasks shares it with the one behind it), found
      // in two looks of 64 lanes each
      const int step = (SB + 63) / 64;
      auto not_behind = [&](int b) { return __builtin_popcountll(__ballot(b < SB && (first_task[b] & 0xffffu) <= t)); };
      const int seg = (not_behind(lane * step) - 1) * step;
      k.bin = seg + not_behind(lane < step ? seg + lane : SB) - 1;
      const uint32_t at = first_task[k.bin], t0 = at & 0xffffu;
      share(t - t0, (first_task[k.bin + 1] & 0xffffu) - t0, at >> 16);
    } else if (n_late > 0u) {
      // the heavy bin that a further share belongs to, or the one that the bin of this place is
      const bool further = t < split_tasks + late_tasks;
      uint32_t found = 0;
      for (uint32_t i0 = 0; i0 < n_late; i0 += 64u) {
        const uint32_t i = i0 + (uint32_t)lane;
        const uint64_t m = __ballot(i < n_late && (further ? (late[2u * i + 1u] & 0xffffu) <= t - split_tasks : late[2u * i] == (uint32_t)k.bin));
        found += further ? (uint32_t)__builtin_popcountll(m) : m ? i0 + (uint32_t)__builtin_ctzll(m) + 1u : 0u;
      }
      if (found > 0u) {
        const uint32_t i = found - 1u, at = late[2u * i + 1u], e0 = at & 0xffffu;
        k.bin = (int)late[2u * i];
        share(further ? t - split_tasks - e0 + 1u : 0u, (late[2u * i + 3u] & 0xffffu) - e0 + 1u, at >> 16);
      }
    }
    k.level = __builtin_popcountll(__ballot(lane < bp.n_levels && level_base <= k.bin)) - 1;
    k.bin = __builtin_amdgcn_readfirstlane(k.bin);
    k.level = __builtin_amdgcn_readfirstlane(k.level);
    k.block0 = __builtin_amdgcn_readfirstlane(k.block0);
    k.block1 = __builtin_amdgcn_readfirstlane(k.block1);
    k.slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)k.slot);
    return k;
  };
  // an odd feature count leaves the last pass with one feature: plane 1 then has no column in the table
  const bool has_pair = TWO || f0 + 1 < feat;
  constexpr uint32_t RW = sizeof(Rec) / 4;
  // A task's blocks, ACC_THREADS at a time, and where this thread's block has the bin's records: first | end << 16 (asked for without a
  // branch, at the end of which they would be waited for).
  struct Chunk {
    Task task;
    int w0;
    bool valid, last;
    uint32_t part;
  };
  auto chunk_of = [&](const Task& k, int w0) {
    const int w = min(w0 + tid, k.block1 - 1);
    const uint32_t part = *reinterpret_cast<const TwoStarts*>(ws.starts + (int64_t)w * ws.start_stride + k.bin + k.level);
    return Chunk{k, w0, true, w0 + ACC_THREADS >= k.block1, part};
  };
  // Places in the sequence come from a counter, fetched a task ahead, and so are the places of the next chunk's records: neither is
  // waited for.  Every workgroup leaves as soon as the counter has passed the last task.
  uint32_t t_next = (uint32_t)__builtin_amdgcn_readfirstlane((int)next_task);
  bool taken = false;  // the next place has been asked for
  auto chunk_behind = [&](const Chunk& c) {
    if (!c.last) return chunk_of(c.task, c.w0 + ACC_THREADS);
    if (t_next >= n_tasks) return Chunk{c.task, c.task.block1, false, true, 0u};
    if (tid == 0) ticket = atomicAdd(counter, 1u);
    taken = true;
    const Task k = task_of(t_next);
    return chunk_of(k, k.block0);
  };
  // The level's records behind a buffer descriptor: a lane without a record asks for one past the end and gets zeros (zero
  // weights), so the loop carries no bounds tests.
  auto records_of = [&](int l) {
    return __builtin_amdgcn_make_buffer_rsrc(ws.records + bp.record_base[l] * (int64_t)RW, 0,
                                             (int)((uint32_t)ws.blocks * (uint32_t)bp.block_records[l] * (uint32_t)sizeof(Rec)), 0x00020000);
  };
  // The chunk's records as a list of groups, up to LIST of them at a time.
  struct Groups {
    uint32_t at, c, mine, before, all;
  };
  auto groups_of = [&](const Chunk& k) {  // (one barrier)
    Groups s;
    s.at = ((uint32_t)(k.w0 + tid) * (uint32_t)bp.block_records[k.task.level] + (k.part & 0xffffu)) * RW;
    s.c = k.w0 + tid < k.task.block1 ? (k.part >> 16) - (k.part & 0xffffu) : 0u;
    s.mine = (s.c + GROUP - 1u) / GROUP;
    s.before = scan(s.mine, &s.all);
    return s;
  };
  auto write_list = [&](const Groups& s, uint32_t e0) {  // entries e0 .. e0 + LIST; returns how many there are
    for (uint32_t e = s.before < e0 ? e0 : s.before; e < s.before + s.mine && e < e0 + LIST; ++e) {
      const uint32_t k = (e - s.before) * GROUP;
      list[e - e0] = (s.at + k * RW) | min(s.c - k, (uint32_t)GROUP) << 27;
    }
    const uint32_t now = min(s.all - e0, (uint32_t)LIST);
    for (uint32_t e = now + tid; e < now + LIST_PAD; e += ACC_THREADS) list[e] = 0u;
    return now;
  };
  const uint32_t in_group = (uint32_t)tid % GROUP;
  auto load_rec = [&](const __amdgpu_buffer_rsrc_t& rs, uint32_t entry) {
    const uint32_t at = in_group < entry >> 27 ? (entry & 0x7ffffffu) * 4u + in_group * (uint32_t)sizeof(Rec) : 0xf0000000u;
    Rec r;
    if constexpr (sizeof(Rec) == 12) {
      typedef unsigned int v3u __attribute__((ext_vector_type(3)));
      const v3u v = __builtin_amdgcn_raw_buffer_load_b96(rs, at, 0, 0);
      r.x = v[0]; r.y = v[1]; r.z = v[2];
    } else {
      typedef unsigned int v4u __attribute__((ext_vector_type(4)));
      const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0);
      r.x = v[0]; r.y = v[1]; r.z = v[2]; r.w = v[3];
    }
    return r;
  };
  constexpr uint32_t ROUND = ACC_THREADS * ACC_INFLIGHT;
  Rec q[ACC_INFLIGHT];  // the records of a round, a round ahead of their adds
  const uint32_t* mine = list + (uint32_t)tid / GROUP;
  auto load_round = [&](const __amdgpu_buffer_rsrc_t& rs, uint32_t e) {
#pragma unroll
    for (int k = 0; k < ACC_INFLIGHT; ++k) q[k] = load_rec(rs, mine[e + k * (ACC_THREADS / GROUP)]);
  };
  const Task first_of_all = task_of(blockIdx.x);
  Chunk now = chunk_of(first_of_all, first_of_all.block0);
  if (blockIdx.x == 0) {  // for the kernel behind this one
    const auto split = [&](uint32_t b, uint32_t slot, uint32_t n) {
      if (n > 1u) ws.splits[atomicAdd(&ws.header->n_splits, 1u)] = BinSplit{b, slot, n, 0u};
    };
    for (int b = tid; b < SB; b += ACC_THREADS) split((uint32_t)b, first_task[b] >> 16, (first_task[b + 1] & 0xffffu) - (first_task[b] & 0xffffu));
    for (uint32_t i = tid; i < n_late; i += ACC_THREADS) split(late[2u * i], late[2u * i + 1u] >> 16, (late[2u * i + 3u] & 0xffffu) - (late[2u * i + 1u] & 0xffffu) + 1u);
  }
  Groups groups = groups_of(now);
  uint32_t entries = write_list(groups, 0);
  lds_barrier();
  load_round(records_of(now.task.level), 0);
  Chunk next = chunk_behind(now);
  for (;;) {
    const Task& task = now.task;
    const int l = task.level;
    const FixedPoint fixed(BinRec<GT>::level_max(level_max[l]));
    const bool nonfinite = fixed.nonfinite;
    const float scale = nonfinite ? 0.0f : ldexpf(1.0f, fixed.se);  // |g| * 2^se < 2^30, and |se| stays inside float's exponents
    const float scale_w = scale * (1.0f / (float)W_MAX);      // with the decoding of the pair records' weights
    const __amdgpu_buffer_rsrc_t rs = records_of(l);
    // a lane without a record, and a record without a gradient, add nothing
    auto live = [](const Rec& r) {
      if constexpr (sizeof(Rec) == 12) return (r.z & 0x7fff7fffu) != 0u;
      else return ((r.z | r.w) & 0x7fffffffu) != 0u;
    };
    auto add_to = [&](uint32_t at, int32_t v) { atomicAdd(acc_tile + at, (unsigned long long)(long long)v); };
    // The next round's records are loaded before this round's adds (the list goes on with empty entries for two rounds); a level with an inf
    // or a nan in its gradient only marks the rows it touches (its own copy of the loop, so that the usual one has no test per record).
    auto rounds = [&](auto add) {
      for (uint32_t e = 0; e < entries; e += ROUND / GROUP) add(q, [&] { load_round(rs, e + ROUND / GROUP); });
    };
    auto add_pairs = [&](auto nonfinite_c) {
      constexpr bool NONFINITE = decltype(nonfinite_c)::value;
      return [&](Rec (&q)[ACC_INFLIGHT], auto load_next) {
        uint32_t slot[ACC_INFLIGHT][2];
        int32_t f[ACC_INFLIGHT][4];
        bool on[ACC_INFLIGHT];
#pragma unroll
        for (int k = 0; k < ACC_INFLIGHT; ++k) {
          const float g0 = BinRec<GT>::g0(q[k]) * scale_w, g1 = BinRec<GT>::g1(q[k]) * scale_w;
          const float w0 = (float)(q[k].y & W_MAX), w1 = (float)((q[k].x >> 26) << 13 | q[k].y >> W_BITS);
          slot[k][0] = q[k].x & BIN_MASK;
          slot[k][1] = (q[k].x >> BIN_ROWS_LOG2) & BIN_MASK;
          on[k] = live(q[k]);
          if constexpr (NONFINITE) {
            f[k][0] = w0 != 0.0f;
            f[k][2] = w1 != 0.0f;
            f[k][1] = has_pair && f[k][0];
            f[k][3] = has_pair && f[k][2];
          } else {
            f[k][0] = round_to_int(w0 * g0);
            f[k][1] = round_to_int(w0 * g1);
            f[k][2] = round_to_int(w1 * g0);
            f[k][3] = round_to_int(w1 * g1);
          }
        }
        load_next();
#pragma unroll
        for (int k = 0; k < ACC_INFLIGHT; ++k)
          if (on[k]) {
#pragma unroll
            for (int j = 0; j < 4; ++j) add_to((uint32_t)(j & 1) * BIN_ROWS + slot[k][j >> 1], f[k][j]);
          }
      };
    };
    // cell records (dense levels): the eight corners' rows and weights are rebuilt from the record; a corner outside this
    // bin belongs to the copy of the record in the neighbouring bin
    auto add_cells = [&](auto nonfinite_c) {
      constexpr bool NONFINITE = decltype(nonfinite_c)::value;
      return [&](Rec (&q)[ACC_INFLIGHT], auto load_next) {
        const uint32_t res = (uint32_t)g.res[l], r2 = res * res;
        Rec cur[ACC_INFLIGHT];
#pragma unroll
        for (int k = 0; k < ACC_INFLIGHT; ++k) cur[k] = q[k];
        load_next();
#pragma unroll
        for (int k = 0; k < ACC_INFLIGHT; ++k) {
          if (!live(cur[k])) continue;
          const int32_t rel = (int32_t)(cur[k].x & 0x3fffu) - BIN_ROWS;
          const float fx = (float)(cur[k].x >> 14) * (1.0f / CELL_QX), fy = (float)(cur[k].y & 0xffffu) * (1.0f / CELL_QYZ),
                      fz = (float)(cur[k].y >> 16) * (1.0f / CELL_QYZ);
          const float fr[3] = {fx, fy, fz};
          float w[8];
          weights_d3(fr, w);
          const float g0 = BinRec<GT>::g0(cur[k]) * scale, g1 = BinRec<GT>::g1(cur[k]) * scale;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const uint32_t slot = (uint32_t)(rel + (j & 1) + ((j >> 1) & 1) * (int32_t)res + (j >> 2) * (int32_t)r2);
            if (slot >= (uint32_t)BIN_ROWS) continue;
            if constexpr (NONFINITE) {
              if (w[j] == 0.0f) continue;
              add_to(slot, 1);
              if (has_pair) add_to((uint32_t)BIN_ROWS + slot, 1);
            } else {
              add_to(slot, round_to_int(w[j] * g0));
              add_to((uint32_t)BIN_ROWS + slot, round_to_int(w[j] * g1));
            }
          }
        }
      };
    };
    bool cells = false;
    if constexpr (sizeof(Rec) == 12) cells = l < bp.cell_levels;
    auto add_list = [&] {
      if (cells) {
        if (nonfinite) rounds(add_cells(std::true_type{}));
        else rounds(add_cells(std::false_type{}));
      } else if (nonfinite) rounds(add_pairs(std::true_type{}));
      else rounds(add_pairs(std::false_type{}));
    };
    add_list();
    for (uint32_t e0 = LIST; e0 < groups.all; e0 += LIST) {  // (a bin of very many records)
      lds_barrier();
      entries = write_list(groups, e0);
      lds_barrier();
      load_round(rs, 0);
      add_list();
    }
    // The next chunk's list takes the place of this one's and its first records are asked for; then, under way with those, the
    // finished tile leaves.
    if (tid == 0 && taken) next_task = gridDim.x + ticket;
    groups = groups_of(next);
    if (taken) t_next = (uint32_t)__builtin_amdgcn_readfirstlane((int)next_task);
    taken = false;
    const bool done = now.last;
    Chunk behind = next;
    if (next.valid) {
      entries = write_list(groups, 0);
      lds_barrier();
      load_round(records_of(next.task.level), 0);
      behind = chunk_behind(next);
    }
    if (!done) {
      now = next;
      next = behind;
      continue;
    }
    const uint32_t row0 = (uint32_t)(task.bin - bp.binbase[l]) << BIN_ROWS_LOG2;
    const uint32_t left = g.rows[l] - row0;
    const uint32_t nrows = left < (uint32_t)BIN_ROWS ? left : (uint32_t)BIN_ROWS;
    // the tile to the table (or the task's slot), and back to zero for the next task
    const int64_t first = (g.row_offset[l] + (int64_t)row0) * feat + f0;  // features f0, f0 + 1 of the bin's rows
    const FixedPoint::ToFloat to_float = fixed.to_float();
    auto take = [&](uint32_t i) {
      const long long a = (long long)acc_tile[i];
      acc_tile[i] = 0ull;
      return a;
    };
    constexpr int U = MODE == TABLE_ADD ? 4 : 8;  // rows of a thread that are under way together
    const bool whole_slot = task.slot != ~0u && ws.whole_slots;
    if (whole_slot) {
      longlong2* dst = reinterpret_cast<longlong2*>(ws.slots) + (int64_t)task.slot * BIN_ROWS;
#pragma unroll 4
      for (uint32_t r = tid; r < nrows; r += ACC_THREADS) {
        const long long x = take(r), y = take(BIN_ROWS + r);
        dst[r] = make_longlong2(x, y);
      }
    }
    for (uint32_t r0 = whole_slot ? nrows : tid; r0 < nrows; r0 += ACC_THREADS * U) {
      float x[U], y[U];
      float2 old[MODE == TABLE_ADD ? U : 1];
      // Added: the old values of all these rows are asked for before any is needed (rows of an even number of features pair by pair).  Rows
      // of other than two features, 16 levels of 2^19 rows, one / four / eight rows of a thread under way (us): 10^5 points F = 1 81 / 79 / 77,
      // F = 3 195 / 189 / 188, F = 4 204 / 201 / 200, F = 8 567 / 580 / 566; 5 * 10^5 points 198 / 192 / 188, 483 / 468 / 467, 503 / 492 / 492,
      // 1181 / 1191 / 1179: what takes the time is the traffic of rows half used per pass.
      if constexpr (MODE == TABLE_ADD)
        if (task.slot == ~0u) {
          const float* src = reinterpret_cast<const float*>(table) + first;
          if constexpr (TWO) {
#pragma unroll
            for (int u = 0; u < U; ++u) old[u] = reinterpret_cast<const float2*>(src)[min(r0 + u * ACC_THREADS, nrows - 1u)];
          } else if ((feat & 1) == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) old[u] = *reinterpret_cast<const float2*>(src + (int64_t)min(r0 + u * ACC_THREADS, nrows - 1u) * feat);
          } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const float* cell = src + (int64_t)min(r0 + u * ACC_THREADS, nrows - 1u) * feat;
              old[u] = make_float2(cell[0], has_pair ? cell[1] : 0.0f);
            }
          }
        }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t r = r0 + u * ACC_THREADS;
        x[u] = r < nrows ? to_float(take(r)) : 0.0f;
        y[u] = r < nrows ? to_float(take(BIN_ROWS + r)) : 0.0f;
      }
      if (task.slot != ~0u) {
        float2* dst = reinterpret_cast<float2*>(ws.slots) + (int64_t)task.slot * BIN_ROWS;
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (r0 + u * ACC_THREADS < nrows) dst[r0 + u * ACC_THREADS] = make_float2(x[u], y[u]);
      } else {
        if constexpr (MODE == TABLE_ADD) {
          float* dst = reinterpret_cast<float*>(table) + first;
          if constexpr (TWO) {
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (x[u] != 0.0f || y[u] != 0.0f) reinterpret_cast<float2*>(dst)[r0 + u * ACC_THREADS] = make_float2(old[u].x + x[u], old[u].y + y[u]);
          } else if ((feat & 1) == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (x[u] != 0.0f || y[u] != 0.0f)
                *reinterpret_cast<float2*>(dst + (int64_t)(r0 + u * ACC_THREADS) * feat) = make_float2(old[u].x + x[u], old[u].y + y[u]);
          } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              float* cell = dst + (int64_t)(r0 + u * ACC_THREADS) * feat;
              if (x[u] != 0.0f) cell[0] = old[u].x + x[u];
              if (has_pair && y[u] != 0.0f) cell[1] = old[u].y + y[u];
            }
          }
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t r = r0 + u * ACC_THREADS;
            if (r < nrows) store_pair<MODE>(table, first + (int64_t)r * feat, x[u], y[u], TWO, has_pair);
          }
        }
      }
    }
    if (!next.valid) return;
    lds_barrier();  // the tile is clear
    now = next;
    next = behind;
  }
}

// ---------------------------------------------------------------------------------------
// reduce: the slots of a bin with several tasks
// ---------------------------------------------------------------------------------------
constexpr int REDUCE_THREADS = 256, REDUCE_VALUES = 256;
template <int MODE>
__global__ __launch_bounds__(REDUCE_THREADS) void hash_bwd_bin_reduce_k(BinWs ws, void* table, DevGeom g, BinPlan bp, int feat, int f0, int ddt) {
  if (blockIdx.y >= ws.header->n_splits) return;
  const BinSplit sp = ws.splits[blockIdx.y];
  int l = 0;
  while (l + 1 < bp.n_levels && (int)sp.bin >= bp.binbase[l + 1]) ++l;
  const uint32_t row0 = (sp.bin - (uint32_t)bp.binbase[l]) << BIN_ROWS_LOG2;
  const uint32_t left = g.rows[l] - row0, nvals = 2u * (left < (uint32_t)BIN_ROWS ? left : (uint32_t)BIN_ROWS);
  const int64_t first = (g.row_offset[l] + (int64_t)row0) * feat + f0;
  const uint32_t pattern = ws.header->gmax[l];
  const FixedPoint::ToFloat to_float = FixedPoint(ddt == NF_F32 ? BinRec<F32>::level_max(pattern) : ddt == NF_F16 ? BinRec<F16>::level_max(pattern) : BinRec<BF16>::level_max(pattern)).to_float();
  const auto total = [&](auto* slots, uint32_t i) {
    const auto* src = slots + (int64_t)sp.slot * (2 * BIN_ROWS) + i;
    std::remove_reference_t<decltype(*slots)> sum = 0;
#pragma unroll 8
    for (uint32_t k = 0; k < sp.n; ++k) sum += src[(int64_t)k * (2 * BIN_ROWS)];
    return sum;
  };
  for (uint32_t i = blockIdx.x * REDUCE_VALUES + threadIdx.x; i < min(nvals, (blockIdx.x + 1u) * REDUCE_VALUES); i += REDUCE_THREADS) {
    const float x = ws.whole_slots ? to_float(total(reinterpret_cast<long long*>(ws.slots), i)) : total(reinterpret_cast<float*>(ws.slots), i);
    if ((i & 1u) && f0 + 1 >= feat) continue;
    const int64_t to = first + (int64_t)(i >> 1) * feat + (i & 1u);
    if constexpr (MODE == TABLE_ADD) {
      if (x != 0.0f) reinterpret_cast<float*>(table)[to] += x;
    } else {
      store_table<MODE>(table, to, x);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Small batches, and levels of a few bins: no records
// ---------------------------------------------------------------------------------------
// Where points times bins are few, sorting costs more than hashing a point once per bin: a task is one bin of a level and a slice of
// the points; its workgroup walks the slice, hashes each point's corners and adds those inside its bin to the same 64-bit
// fixed-point LDS tile as the record kernels.  The upstream gradient is transposed first into level-major pairs, so that a
// task's walk reads 4 (float32: 8) contiguous bytes per point instead of touching a whole row; the same pass takes the maxima that
// set the fixed-point scales.  A bin of one slice goes from the tile to the table; slices leave their sums in slots, which a last
// pass adds in their order: a gradient has the same bits in every run.
// Before (two rounds of workgroups that waited for each point, scattered adds of the tiles, zeros and rounding of the table as passes of
// their own) -> now: 2^14 rows float32, 2^18 points 145 -> 63 us, of which the walk 91 -> 42; fp16 2^16 rows, 8192 points 80 -> 28 (was: records).
constexpr int WALK_THREADS = 1024;
constexpr int WALK_PREP_THREADS = 256;
constexpr int WALK_STRIDE = 16;  // points between neighbouring lanes of a walk
constexpr int PREP_PITCH = 9;    // 16-byte pieces between the rows that hash_bwd_walk_prep_k turns in LDS

struct WalkPlan {
  int n_levels, n_tasks, prep_blocks;
  int bins[NF_MAX_LEVELS], slices[NF_MAX_LEVELS];
  int first[NF_MAX_LEVELS + 1];  // first task of a level; task first + which * slices + slice
};
// What a task's tile holds.  A level of one bin: both features of the pair.  A level of two bins: one of the features, of all the
// level's rows; either way every corner of a point lands in the tile, so the walk has no test per corner and its LDS adds
// run with all lanes.  A level of more bins: both features of one bin's rows.
enum WalkKind { WALK_LEVEL = 0, WALK_FEATURE = 1, WALK_BIN = 2 };

struct WalkWs {
  uint32_t* block_max;  // [levels][ceil(feat / 2)][prep_blocks] largest |gradient| pattern of a block of points
  float* points;        // [dims][N] coordinates, divided by the scale
  uint32_t* pairs;      // [levels][ceil(feat / 2)][N] gradient pairs (a missing partner is zero)
  float* slots;         // [n_tasks][2 * BIN_ROWS], where any level has more than one slice
};

// Gradient pairs level by level and coordinates dimension by dimension, both in the order of the walk: neighbouring lanes of a walk take
// points WALK_STRIDE apart, because along a ray neighbouring points share cells and their adds to one row would wait for each other
// (T = 2^14, 2^18 points along rays: 258 us without, 85 with).  Rows of whole 16-byte pieces (VEC) come in as they lie, 512 bytes of four
// neighbouring points to 32 lanes, up to 128 bytes of a row at once, and are turned to a row per lane in LDS: read a row per lane from memory,
// the lines of a unit's lanes are ten times its L1 and every piece fetched its line again.  A thread's pieces are all of the same planes, so the
// maxima are taken before the turn (one per plane and row behind it: 72.9 us).  The chain of a float32 table of 2^14 rows, 2^18 points 66.0 -> 63.3 us
// (this kernel 20.0 -> 16.6, 67 MB), 4096 points 21.8 -> 19.9; fp16 2^18 61.6 -> 59.3, rows of four features 2^17 77.5 -> 73.3.  Other rows
// have a kernel of their own, as one for both needs the registers of eight pieces (one feature, 8 levels of 2^15 rows, 425718 points 18.4 -> 16.7).
template <bool G32, int D, bool VEC>
__global__ __launch_bounds__(WALK_PREP_THREADS) void hash_bwd_walk_prep_k(const void* coords, int cdt, int64_t csn, int64_t csd, float scale,
                                                                          const void* dout_v, int64_t dout_stride, int64_t N, int levels, int feat,
                                                                          WalkWs ws) {
  extern __shared__ __align__(16) uint32_t plane_max[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int np = (feat + 1) / 2, planes = levels * np;
  for (int i = tid; i < planes; i += WALK_PREP_THREADS) plane_max[i] = 0u;
  __syncthreads();
  const int64_t at = (int64_t)blockIdx.x * WALK_PREP_THREADS + tid;  // position in the walk's order
  const bool valid = at < N;
  constexpr int CHUNK = 64 * WALK_STRIDE;
  const int64_t chunk = at / CHUNK * CHUNK;
  const int in_chunk = (int)(at - chunk);
  const bool whole = chunk + CHUNK <= N;  // (the same for the workgroup)
  const int64_t n = !valid ? 0 : whole ? chunk + (in_chunk & 63) * WALK_STRIDE + (in_chunk >> 6) : at;
  float v[D];
  load_point_d<D>(coords, cdt, csn, csd, n, scale, v);
  const uint16_t* row16 = reinterpret_cast<const uint16_t*>(dout_v) + n * dout_stride;
  const float* row32 = reinterpret_cast<const float*>(dout_v) + n * dout_stride;
  static_assert(WALK_PREP_THREADS == 4 * 64, "a workgroup's positions are four points of each of a chunk's groups");
  auto put = [&](int plane, uint32_t x, uint32_t y) {
    if (!valid) return;
    if (G32) reinterpret_cast<uint2*>(ws.pairs)[(int64_t)plane * N + at] = make_uint2(x, y);
    else ws.pairs[(int64_t)plane * N + at] = x;
  };
  auto pair_max = [&](uint32_t x, uint32_t y) { return G32 ? max(x & 0x7fffffffu, y & 0x7fffffffu) : max(x & 0x7fffu, (x >> 16) & 0x7fffu); };
  if constexpr (VEC) {
    constexpr int PER = G32 ? 2 : 4;  // planes of a piece
    uint4* tile = reinterpret_cast<uint4*>(plane_max + (planes + 3) / 4 * 4);  // [position][PREP_PITCH]
    const int pieces = planes / PER;
    auto block = [&](int q0, auto width_c) {  // pieces q0 .. of the rows
      constexpr int W = decltype(width_c)::value;
      uint4 v[W];
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const int u = tid + i * WALK_PREP_THREADS, row = u / W, q = q0 + u % W;
        const int64_t first = chunk + in_chunk / WALK_PREP_THREADS * (WALK_PREP_THREADS / 64);
        int64_t r = whole ? first + row / 4 * WALK_STRIDE + row % 4 : (int64_t)blockIdx.x * WALK_PREP_THREADS + row;
        r = r < N ? r : N - 1;
        const char* p = reinterpret_cast<const char*>(dout_v) + r * dout_stride * (G32 ? 4 : 2);
        v[i] = reinterpret_cast<const uint4*>(p)[q < pieces ? q : pieces - 1];
      }
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const int u = tid + i * WALK_PREP_THREADS, row = u / W, slot = whole ? row % 4 * 64 + row / 4 : row;
        tile[slot * PREP_PITCH + u % W] = v[i];
      }
      // a thread's pieces are of the same planes, and so are those of every W-th lane
      uint32_t m[PER] = {};
#pragma unroll
      for (int i = 0; i < W; ++i) {
        if constexpr (G32) {
          m[0] = max(m[0], pair_max(v[i].x, v[i].y));
          m[1] = max(m[1], pair_max(v[i].z, v[i].w));
        } else {
          m[0] = max(m[0], pair_max(v[i].x, 0u));
          m[1] = max(m[1], pair_max(v[i].y, 0u));
          m[2] = max(m[2], pair_max(v[i].z, 0u));
          m[3] = max(m[3], pair_max(v[i].w, 0u));
        }
      }
#pragma unroll
      for (int k = 0; k < PER; ++k) {
#pragma unroll
        for (int d = W; d < 64; d *= 2) m[k] = max(m[k], (uint32_t)__shfl_xor((int)m[k], d));
        if (lane < W && q0 + lane < pieces) atomicMax(plane_max + (q0 + lane) * PER + k, m[k]);
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < W; ++i)
        if (q0 + i < pieces) {
          const uint4 q = tile[tid * PREP_PITCH + i];
          const int plane = (q0 + i) * PER;
          if constexpr (G32) {
            put(plane, q.x, q.y);
            put(plane + 1, q.z, q.w);
          } else {
            put(plane, q.x, 0u);
            put(plane + 1, q.y, 0u);
            put(plane + 2, q.z, 0u);
            put(plane + 3, q.w, 0u);
          }
        }
      __syncthreads();
    };
    int q0 = 0;
    for (; pieces - q0 > 4; q0 += 8) block(q0, std::integral_constant<int, 8>{});
    if (q0 < pieces) block(q0, std::integral_constant<int, 4>{});
  } else {
    for (int plane = 0; plane < planes; ++plane) {
      const int e0 = plane / np * feat + 2 * (plane % np);
      const bool two = 2 * (plane % np) + 1 < feat;
      const uint32_t x = G32 ? __float_as_uint(row32[e0]) : (uint32_t)row16[e0] | (two ? (uint32_t)row16[e0 + 1] << 16 : 0u);
      const uint32_t y = G32 && two ? __float_as_uint(row32[e0 + 1]) : 0u;
      put(plane, x, y);
      const uint32_t m = wave_max_u32(valid ? pair_max(x, y) : 0u);
      if (lane == 63 && m) atomicMax(plane_max + plane, m);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (valid) ws.points[d * N + at] = v[d];
  __syncthreads();
  for (int i = tid; i < planes; i += WALK_PREP_THREADS) ws.block_max[(int64_t)i * gridDim.x + blockIdx.x] = plane_max[i];
}

template <typename GT, int D>
__global__ __launch_bounds__(WALK_THREADS) void hash_bwd_walk_k(WalkWs ws, int64_t N, DevGeom g, WalkPlan wp, const int64_t* primes, void* table, int mode,
                                                                int feat, int p) {
  constexpr bool G32 = sizeof(typename BinRec<GT>::type) == 16;
  constexpr int CN = 1 << D, VD = D > 3 ? D : 3;
  extern __shared__ __align__(16) unsigned long long acc_tile[];  // 2 * BIN_ROWS sums
  __shared__ uint32_t level_max, hit;
  const int tid = threadIdx.x, lane = tid & 63;
  const int np = (feat + 1) / 2, f0 = 2 * p;
  const bool has_pair = f0 + 1 < feat;
  const uint32_t pi[3] = {(uint32_t)primes[0], (uint32_t)primes[1], D > 2 ? (uint32_t)primes[D > 2 ? 2 : 0] : 0u};
  for (uint32_t i = tid; i < 2u * BIN_ROWS; i += WALK_THREADS) acc_tile[i] = 0ull;
  if (tid == 0) level_max = hit = 0u;
  for (int t = (int)blockIdx.x; t < wp.n_tasks; t += (int)gridDim.x) {
    int l = 0;
    while (l + 1 < wp.n_levels && t >= wp.first[l + 1]) ++l;
    const int slices = wp.slices[l], which = (t - wp.first[l]) / slices, slice = (t - wp.first[l]) % slices;
    const WalkKind kind = wp.bins[l] == 1 ? WALK_LEVEL : wp.bins[l] == 2 ? WALK_FEATURE : WALK_BIN;
    if (kind == WALK_FEATURE && which == 1 && !has_pair) continue;  // an odd feature count: the last pair has one feature
    const uint32_t row0 = kind == WALK_BIN ? (uint32_t)which << BIN_ROWS_LOG2 : 0u;
    const uint32_t left = g.rows[l] - row0, nrows = kind == WALK_BIN && left > (uint32_t)BIN_ROWS ? (uint32_t)BIN_ROWS : left;
    // fixed-point scale 2^se of the pair on this level, as in the record kernels:  |w * g| * 2^se < 2^30
    uint32_t m = 0u;
    for (int i = tid; i < wp.prep_blocks; i += WALK_THREADS) m = max(m, ws.block_max[((int64_t)l * np + p) * wp.prep_blocks + i]);
    m = wave_max_u32(m);
    __syncthreads();  // the tile is clear, and nobody reads the maximum of the task before
    if (lane == 63 && m) atomicMax(&level_max, m);
    __syncthreads();
    const float gm = BinRec<GT>::level_max(level_max);
    const bool nonfinite = !(gm <= 3.0e38f);
    int se = 0;
    if (!nonfinite && gm > 0.0f) {
      int ex;
      frexpf(gm, &ex);
      se = 30 - ex;
      se = se > 120 ? 120 : se;
    }
    // |g| * 2^se < 2^30: the scaled gradient is a float (the two steps are exact powers of two inside float range)
    const float s_lo = nonfinite ? 0.0f : ldexpf(1.0f, se / 2), s_hi = ldexpf(1.0f, se - se / 2);
    const bool hashed = l >= g.first_hash;
    const float fres = (float)g.res[l];
    const uint32_t res = (uint32_t)g.res[l], mask = g.rows[l] - 1u;
    const uint32_t* level_pairs = ws.pairs + (((int64_t)l * np + p) * N) * (G32 ? 2 : 1);
    const int64_t n_begin = N * slice / slices, n_end = N * (slice + 1) / slices;
    struct Point {
      float v[VD];
      typename BinRec<GT>::type rec;
    };
    auto load = [&](int64_t n) {
      Point q = {{}, BinRec<GT>::zero()};
#pragma unroll
      for (int d = 0; d < D; ++d) q.v[d] = ws.points[d * N + n];
      if constexpr (G32) {
        const uint2 pair = reinterpret_cast<const uint2*>(level_pairs)[n];
        q.rec.z = pair.x;
        q.rec.w = pair.y;
      } else {
        q.rec.z = level_pairs[n];
      }
      return q;
    };
    // One point per thread and turn, the next one under way.  The loop exists in six copies, by the kind of tile and for levels with an
    // inf or a nan in their gradient (which only mark the rows they touch), so that it carries no branch.
    auto walk = [&](auto kind_c, auto nonfinite_c) {
      constexpr WalkKind KIND = decltype(kind_c)::value;
      constexpr bool NONFINITE = decltype(nonfinite_c)::value;
      auto fixed = [&](float w, float gs) { return NONFINITE ? (int32_t)(w != 0.0f) : round_to_int(w * gs); };
      auto add_to = [&](uint32_t at, int32_t f) { atomicAdd(acc_tile + at, (unsigned long long)(long long)f); };
      if (n_begin + tid >= n_end) return;
      Point next = load(n_begin + tid);
      for (int64_t n = n_begin + tid; n < n_end; n += WALK_THREADS) {
        const Point q = next;
        next = load(n + WALK_THREADS < n_end ? n + WALK_THREADS : n);
        uint32_t row[CN];
        float w[CN];
        cell_rows<D>(q.v, fres, hashed, res, mask, pi, primes, row, w);
        const float g0 = BinRec<GT>::g0(q.rec) * s_lo * s_hi, g1 = BinRec<GT>::g1(q.rec) * s_lo * s_hi;
        const float gs = which ? g1 : g0;
        if constexpr (KIND == WALK_BIN) {
#pragma unroll
          for (int j = 0; j < CN; j += 2) {
            const uint32_t a = row[j] - row0, b = row[j + 1] - row0;
            if (a < (uint32_t)BIN_ROWS || b < (uint32_t)BIN_ROWS) {
              hit = 1u;
              if (a < (uint32_t)BIN_ROWS) {
                add_to(a, fixed(w[j], g0));
                if (has_pair) add_to((uint32_t)BIN_ROWS + a, fixed(w[j], g1));
              }
              if (b < (uint32_t)BIN_ROWS) {
                add_to(b, fixed(w[j + 1], g0));
                if (has_pair) add_to((uint32_t)BIN_ROWS + b, fixed(w[j + 1], g1));
              }
            }
          }
        } else {
          // zero contributions are rare here: the adds carry no test
#pragma unroll
          for (int j = 0; j < CN; ++j) {
            if constexpr (KIND == WALK_FEATURE) {
              add_to(row[j], fixed(w[j], gs));
            } else {
              add_to(row[j], fixed(w[j], g0));
              add_to((uint32_t)BIN_ROWS + row[j], has_pair ? fixed(w[j], g1) : 0);
            }
          }
        }
      }
      if constexpr (KIND != WALK_BIN) hit = 1u;
    };
    auto walk_kind = [&](auto kind_c) {
      if (nonfinite) walk(kind_c, std::true_type{});
      else walk(kind_c, std::false_type{});
    };
    if (kind == WALK_LEVEL) walk_kind(std::integral_constant<WalkKind, WALK_LEVEL>{});
    else if (kind == WALK_FEATURE) walk_kind(std::integral_constant<WalkKind, WALK_FEATURE>{});
    else walk_kind(std::integral_constant<WalkKind, WALK_BIN>{});
    lds_barrier();
    // the tile to the slot or the table, and back to zero for the next task; a tile that nothing was added to is zeros already
    const bool touched = hit != 0u;
    const float qnan = __uint_as_float(0x7fc00000u);
    const double unscale = ldexp(1.0, -se), unscale_hi = ldexp(1.0, 32 - se);
    auto value = [&](uint32_t i) {
      if (!touched) return 0.0f;
      const long long a = (long long)acc_tile[i];
      acc_tile[i] = 0ull;
      const float x = (float)((double)(int)(a >> 32) * unscale_hi + (double)(uint32_t)a * unscale);
      return nonfinite && a != 0 ? qnan : x;
    };
    const int64_t first = (g.row_offset[l] + (int64_t)row0) * feat + f0;
    const bool pairs = kind != WALK_FEATURE;
    if (ws.slots != nullptr) {
      float* slot = ws.slots + (int64_t)t * (2 * BIN_ROWS);
      for (uint32_t r = tid; r < nrows; r += WALK_THREADS) {
        slot[r] = value(r);
        if (pairs) slot[BIN_ROWS + r] = value(BIN_ROWS + r);
      }
    } else if (touched || mode != TABLE_ADD) {
      auto flush = [&](auto mode_c) {
        constexpr int MODE = decltype(mode_c)::value;
#pragma unroll 4
        for (uint32_t r = tid; r < nrows; r += WALK_THREADS) {
          if (pairs) {
            const float x = value(r), y = value(BIN_ROWS + r);
            add_or_store_pair<MODE>(table, first + (int64_t)r * feat, x, y, feat == 2, has_pair);
          } else {
            const int64_t at = first + which + (int64_t)r * feat;
            const float x = value(r);
            if constexpr (MODE == TABLE_ADD) {
              if (x != 0.0f) reinterpret_cast<float*>(table)[at] += x;
            } else {
              store_table<MODE>(table, at, x);
            }
          }
        }
      };
      with_mode(mode, flush);
    }
    lds_barrier();
    if (tid == 0) level_max = hit = 0u;
  }
}

// the slots of every bin, in the order of their slices: a thread takes four rows of a level
template <int MODE>
__global__ __launch_bounds__(REDUCE_THREADS) void hash_bwd_walk_reduce_k(WalkWs ws, void* table, DevGeom g, WalkPlan wp, int feat, int f0) {
  const int l = (int)blockIdx.y;
  const uint32_t r = (blockIdx.x * REDUCE_THREADS + threadIdx.x) * 4u;
  if (r >= g.rows[l]) return;
  const int slices = wp.slices[l];
  const bool by_feature = wp.bins[l] == 2, has_pair = f0 + 1 < feat;
  const int64_t task = wp.first[l] + (by_feature ? 0 : (int64_t)(r >> BIN_ROWS_LOG2) * slices);
  const float* src0 = ws.slots + task * (2 * BIN_ROWS) + (by_feature ? r : r & BIN_MASK);
  const float* src1 = src0 + (by_feature ? (int64_t)slices * (2 * BIN_ROWS) : (int64_t)BIN_ROWS);
  float x[4] = {}, y[4] = {};
#pragma unroll 4
  for (int s = 0; s < slices; ++s) {
    const float4 a = *reinterpret_cast<const float4*>(src0 + (int64_t)s * (2 * BIN_ROWS));
    x[0] += a.x; x[1] += a.y; x[2] += a.z; x[3] += a.w;
    if (has_pair) {
      const float4 b = *reinterpret_cast<const float4*>(src1 + (int64_t)s * (2 * BIN_ROWS));
      y[0] += b.x; y[1] += b.y; y[2] += b.z; y[3] += b.w;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (r + e < g.rows[l]) add_or_store_pair<MODE>(table, (g.row_offset[l] + r + e) * feat + f0, x[e], y[e], feat == 2, has_pair);
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------
// cells: dense 3-D levels whose eight corners span less than a bin take one record per point (16-bit gradients)
static bool bin_plan(int64_t N, int points, const nf_hash_geom* geom, BinPlan* bp, int64_t* records, bool cells) {
  // features are taken two at a time (one pass of fill + accumulate per pair; the last feature of an odd count alone)
  if (geom->dims < 2 || geom->dims > NF_MAX_DIMS || geom->feat < 1 || N <= 0) return false;
  bp->n_levels = geom->levels;
  bp->cell_levels = bp->split_bins = 0;
  const int64_t blocks = (N + points - 1) / points;
  int nb_total = 0;
  int64_t R = 0;
  for (int l = 0; l < geom->levels; ++l) {
    const int64_t r = geom->rows[l];
    const int64_t nb = (r + BIN_ROWS - 1) / BIN_ROWS;
    if (nb > MAX_BINS_PER_LEVEL) return false;
    bp->nbins[l] = (int)nb;
    bp->binbase[l] = nb_total;
    const int64_t res = geom->res[l];
    const bool cell = cells && geom->dims == 3 && l < geom->first_hash_level && res * res + res + 1 < BIN_ROWS && bp->cell_levels == l;
    if (cell) bp->cell_levels = l + 1;
    // a cell level leaves at most two records per point; an x-pair level has room for every pair to be split in two
    // (normally half of it is used); more than three dimensions run as passes of the 3-D pipeline
    bp->block_records[l] = points * (cell ? 2 : geom->dims >= 3 ? 8 : 4);
    bp->record_base[l] = R;
    R += blocks * bp->block_records[l];
    nb_total += (int)nb;
    if (nb_total <= SPLIT_MAX_BINS) bp->split_bins = nb_total;
  }
  bp->binbase[geom->levels] = nb_total;
  *records = R;
  return true;
}

// points of a block (a multiple of four keeps the blocks of records on 16-byte boundaries)
static bool wide_blocks(int64_t n_points, const nf_hash_geom* geom) {
  if (n_points < FILL_WIDE_POINTS) return false;
  for (int l = 0; l < geom->levels; ++l)
    if (geom->rows[l] > (int64_t)FILL_WIDE_BINS * BIN_ROWS) return true;
  return false;
}

// Cost (x-pair records) of a share of a split bin: a third of what a compute unit gets of them on every level, and no less than pays for the
// slot that the share is summed in.  16 levels of 2^19 rows, fp16, whole backward (us), least share 8192 / 16384 / 32768: along rays 2^14 points
// 52 / 60 / 73, 2^16 76 / 73 / 88, 2^17 91 / 87 / 97; uniform 2^18 115 / 115 / 111, added to float32 129 / 128 / 124.
// Shares of fewer than SPLIT_FLOAT_COST records leave their sums as they are, in 64-bit fixed point: a bin of that many records that was one task,
// rounded once, is several then, and float sums of their floats would be rounded for each (2.5e-8 -> 5e-8 of a row at four shares).  The slots
// are twice as large, 1 us of the chain at 2^17 points along rays; in the larger batches, cut no finer, it would be 3 to 7 us.
// A workspace without room for them (`whole` false) gets shares of SPLIT_FLOAT_COST records and slots of floats, whatever the batch.
constexpr int64_t SPLIT_FLOAT_COST = 32768;
static int64_t split_cost(int64_t N, int levels, bool whole) {
  const int64_t third = N * levels / 192, small = N < 32768 ? 8192 : N < 65536 ? N / 4 : 16384, large = N < 262144 ? N / 8 : SPLIT_FLOAT_COST;
  const int64_t least = !whole ? SPLIT_FLOAT_COST : small > large ? small : large;
  return third > least ? third : least;
}

static int64_t bin_ws(void* workspace, const BinPlan& bp, int64_t N, int points, int64_t R, int rec_words, bool whole, BinWs* ws) {
  char* p = (char*)workspace;
  const int NB = bp.binbase[bp.n_levels];
  const int64_t blocks = (N + points - 1) / points;
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    char* at = p + o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  ws->blocks = (int)blocks;
  ws->start_stride = (NB + bp.n_levels + 1) & ~1;
  ws->split_cost = (uint32_t)split_cost(N, bp.n_levels, whole);
  ws->max_slots = (uint32_t)(16 + N / 1024);
  ws->whole_slots = ws->split_cost < SPLIT_FLOAT_COST;
  ws->header = (BinHeader*)take(sizeof(BinHeader) + NB * 4);
  ws->totals = (uint32_t*)(ws->header + 1);
  ws->block_max = (uint32_t*)take(blocks * NF_MAX_LEVELS * 4);
  ws->splits = (BinSplit*)take((int64_t)ws->max_slots * sizeof(BinSplit));
  ws->starts = (uint16_t*)take(blocks * ws->start_stride * 2);
  ws->slots = take((int64_t)ws->max_slots * 2 * BIN_ROWS * (ws->whole_slots ? 8 : 4));
  ws->records = (uint32_t*)take((int64_t)rec_words * R * 4);
  return o;
}

// Batches above this many points go through the pipeline in pieces of this size, one after the other on the stream:
// the scratch stays at 2.8 GB (4.4 GB with a float32 upstream gradient) whatever the batch, and record positions stay
// inside 32 bits.  The gradient table accumulates across the pieces.  (Pieces of 2^20 points would halve the scratch
// and cost 2.5 % of a 2^21-point training step: every piece pays the fixed part of the pipeline again.)
constexpr int64_t BIN_CHUNK_POINTS = (int64_t)1 << 21;

// The walk without records hashes every point once per bin of a level; the records pay a fill and an accumulate pass per level
// whatever its size.  So the walk takes tables whose levels are all at most two bins (2^14 rows, the reference's default), where it has no
// test per corner, and of the others those with a bin or less per unit (a second round of tiles costs what the whole walk does), in
// batches of few points times bins (three bins a level cost the walk what they cost the records).  16 levels of fp16, uniform points
// and rays, walk and records: 2^15 rows 262144 points 106, 136 and 221, 238 us; 2^16 rows 131072 points 101, 130 and 121, 141; 2^17 rows
// 32768 points 62, 95 and 98, 115, 65536 points 112, 172 and 100, 120.  Under WALK_MIN_POINTS the atomics of hash_bwd_level_k are
// quicker, where they apply: 2^16 rows 4096 points 19 and 31, 8192 points 38 and 35, in every feature pair.
constexpr int WALK_FREE_BINS = 2, WALK_MAX_BINS = 256;
constexpr int64_t WALK_MAX_POINT_BINS = (int64_t)13 << 19;
constexpr int WALK_MAX_DIMS = 4;  // the walk is built for 1 to 4 dimensions (the sorted records for 2 to 6)
constexpr int64_t WALK_MIN_POINTS = 6144, WALK_MIN_POINTS_FREE = 4096, WALK_MIN_POINTS_GENERIC = 1024;
static bool walk_ok(int64_t n_points, const nf_hash_geom* geom, int flags) {
  if (flags & NF_HASH_BWD_RECORDS) return false;
  if (geom->dims < 1 || geom->dims > WALK_MAX_DIMS) return false;
  int64_t bins = 0, most = 0;
  for (int l = 0; l < geom->levels; ++l) {
    const int64_t nb = (geom->rows[l] + BIN_ROWS - 1) / BIN_ROWS;
    bins += nb;
    most = nb > most ? nb : most;
  }
  const bool free = most <= WALK_FREE_BINS;
  if (n_points < (!bwd_level_ok(geom) ? WALK_MIN_POINTS_GENERIC : free ? WALK_MIN_POINTS_FREE : WALK_MIN_POINTS * ((geom->feat + 1) / 2))) return false;
  return free || (quick_rows(geom) && bins <= WALK_MAX_BINS && n_points * (bins - 3 * geom->levels) <= WALK_MAX_POINT_BINS);
}
bool bwd_walk_applies(int64_t n_points, const nf_hash_geom* geom, int flags) {
  return walk_ok(n_points < BIN_CHUNK_POINTS ? n_points : BIN_CHUNK_POINTS, geom, flags);
}

static int compute_units() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
    if (cus <= 0) cus = 256;
  }
  return cus;
}

// One task at a time fits a unit (the tile is 128 KiB of LDS), so the points are sliced until there is about one task per unit; a
// task of both features of a level costs one and a half of the others.  Slices of at least two turns of the workgroup.
static WalkPlan walk_plan(int64_t N, const nf_hash_geom* geom) {
  WalkPlan wp = {};
  wp.n_levels = geom->levels;
  wp.prep_blocks = (int)((N + WALK_PREP_THREADS - 1) / WALK_PREP_THREADS);
  int64_t total = 0;
  auto cost = [&](int l) { return wp.bins[l] == 1 ? 3 : 2; };
  for (int l = 0; l < geom->levels; ++l) {
    wp.bins[l] = (int)((geom->rows[l] + BIN_ROWS - 1) / BIN_ROWS);
    total += wp.bins[l] * cost(l);
  }
  const int64_t most = N / (2 * WALK_THREADS);
  for (int l = 0; l < geom->levels; ++l) {
    int64_t slices = (int64_t)compute_units() * cost(l) / total;
    slices = slices > most ? most : slices;
    wp.slices[l] = (int)(slices < 1 ? 1 : slices);
    wp.first[l + 1] = wp.first[l] + wp.bins[l] * wp.slices[l];
  }
  wp.n_tasks = wp.first[wp.n_levels];
  return wp;
}
static bool walk_sliced(const WalkPlan& wp) {
  for (int l = 0; l < wp.n_levels; ++l)
    if (wp.slices[l] > 1) return true;
  return false;
}
static int64_t walk_ws(void* workspace, const WalkPlan& wp, int64_t N, int dims, int feat, int dout_dtype, WalkWs* ws) {
  char* p = (char*)workspace;
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    char* at = p + o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  ws->block_max = (uint32_t*)take((int64_t)wp.n_levels * ((feat + 1) / 2) * wp.prep_blocks * 4);
  ws->points = (float*)take((int64_t)dims * N * 4);
  ws->pairs = (uint32_t*)take((int64_t)wp.n_levels * ((feat + 1) / 2) * N * (dout_dtype == NF_F32 ? 8 : 4));
  ws->slots = walk_sliced(wp) ? (float*)take((int64_t)wp.n_tasks * 2 * BIN_ROWS * 4) : nullptr;
  return o;
}

int64_t bwd_bin_workspace_bytes(int64_t n_points, const nf_hash_geom* geom, int dout_dtype, int flags, bool whole) {
  if (n_points > BIN_CHUNK_POINTS) n_points = BIN_CHUNK_POINTS;
  if (walk_ok(n_points, geom, flags)) {
    WalkWs ws;
    return walk_ws(nullptr, walk_plan(n_points, geom), n_points, geom->dims, geom->feat, dout_dtype, &ws);
  }
  auto bytes = [&](int64_t n, bool wide) -> int64_t {
    BinPlan bp;
    BinWs ws;
    int64_t R;
    const int points = fill_points(wide);
    return bin_plan(n, points, geom, &bp, &R, dout_dtype != NF_F32) ? bin_ws(nullptr, bp, n, points, R, dout_dtype == NF_F32 ? 4 : 3, whole, &ws) : 0;
  };
  if (!wide_blocks(n_points, geom)) return bytes(n_points, false);
  // room for every smaller batch too: many small blocks have more starts than fewer wide ones
  const int64_t wide = bytes(n_points, true), small = bytes(FILL_WIDE_POINTS - 1, false);
  return wide > small ? wide : small;
}

static int launch_bwd_bin_piece(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride,
                                void* table, int mode, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                                void* workspace, int64_t workspace_bytes, hipStream_t s);

static int launch_bwd_walk(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride,
                           void* table, int mode, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                           void* workspace, hipStream_t s);

int launch_bwd_bin(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride,
                   float* dtable, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                   void* workspace, int64_t workspace_bytes, int flags, hipStream_t s) {
  // the choice is made once, on the size the workspace was asked for: every piece then fits it
  const bool walk = bwd_walk_applies(N, geom, flags);
  for (int64_t n0 = 0; n0 < N; n0 += BIN_CHUNK_POINTS) {
    const int64_t n = N - n0 < BIN_CHUNK_POINTS ? N - n0 : BIN_CHUNK_POINTS;
    const char* c = (const char*)coords + n0 * csn * dtype_size(cdt);
    const char* d = (const char*)dout + n0 * dout_stride * dtype_size(ddt);
    const int rc = walk ? launch_bwd_walk(c, cdt, csn, csd, d, ddt, dout_stride, dtable, TABLE_ADD, n, geom, g, primes, scale, workspace, s)
                        : launch_bwd_bin_piece(c, cdt, csn, csd, d, ddt, dout_stride, dtable, TABLE_ADD, n, geom, g, primes, scale, workspace, workspace_bytes, s);
    if (rc) return rc;
  }
  return 0;
}

bool bwd_write_applies(int64_t n_points, const nf_hash_geom* geom, int flags) {
  // one pass over the points that leaves every row's whole sum in one place
  if (n_points > BIN_CHUNK_POINTS) return false;
  return walk_ok(n_points, geom, flags) || (n_points >= bwd_records_min(geom, flags) && (geom->dims == 2 || geom->dims == 3));
}

int launch_bwd_write(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride, void* table,
                     int table_dtype, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                     void* workspace, int64_t workspace_bytes, int flags, hipStream_t s) {
  const int mode = table_dtype == NF_F32 ? TABLE_F32 : table_dtype == NF_F16 ? TABLE_F16 : TABLE_BF16;
  return walk_ok(N, geom, flags) ? launch_bwd_walk(coords, cdt, csn, csd, dout, ddt, dout_stride, table, mode, N, geom, g, primes, scale, workspace, s)
                                 : launch_bwd_bin_piece(coords, cdt, csn, csd, dout, ddt, dout_stride, table, mode, N, geom, g, primes, scale, workspace, workspace_bytes, s);
}

static int launch_large(const char* what, const void* kern, dim3 grid, int threads, void** args, size_t lds, hipStream_t s) {
  hipError_t e = hipSuccess;
  if (lds > 64 * 1024) e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  e = hipLaunchKernel(kern, grid, dim3((unsigned)threads), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(%s): %s", what, hipGetErrorString(e));
  return check_launch(what);
}

static int launch_bwd_walk(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride,
                           void* table, int mode, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                           void* workspace, hipStream_t s) {
  NF_REQUIRE(((uintptr_t)workspace & 15u) == 0, NF_EALIGN, "workspace must be 16-byte aligned");
  WalkPlan wp = walk_plan(N, geom);
  WalkWs ws;
  walk_ws(workspace, wp, N, geom->dims, geom->feat, ddt, &ws);
  int levels = geom->levels, feat = geom->feat;
  const void *prep, *walk;
  const int planes = levels * ((feat + 1) / 2);
  const bool vec = feat % 2 == 0 && planes % (ddt == NF_F32 ? 2 : 4) == 0 && (uintptr_t)dout % 16 == 0 && dout_stride % (ddt == NF_F32 ? 4 : 8) == 0;
  auto pick = [&](auto d_c) {
    constexpr int DD = decltype(d_c)::value;
    prep = ddt == NF_F32 ? (vec ? (const void*)hash_bwd_walk_prep_k<true, DD, true> : (const void*)hash_bwd_walk_prep_k<true, DD, false>)
                         : (vec ? (const void*)hash_bwd_walk_prep_k<false, DD, true> : (const void*)hash_bwd_walk_prep_k<false, DD, false>);
    walk = ddt == NF_F32 ? (const void*)hash_bwd_walk_k<F32, DD> : ddt == NF_BF16 ? (const void*)hash_bwd_walk_k<BF16, DD> : (const void*)hash_bwd_walk_k<F16, DD>;
  };
  if (g.dims == 3) pick(std::integral_constant<int, 3>{});
  else if (g.dims == 2) pick(std::integral_constant<int, 2>{});
  else if (g.dims == 1) pick(std::integral_constant<int, 1>{});
  else pick(std::integral_constant<int, 4>{});
  void* prep_args[] = {(void*)&coords, (void*)&cdt, (void*)&csn, (void*)&csd, (void*)&scale, (void*)&dout, (void*)&dout_stride, (void*)&N, (void*)&levels, (void*)&feat, (void*)&ws};
  const size_t prep_lds = (size_t)(planes + 3) / 4 * 16 + (vec ? (size_t)WALK_PREP_THREADS * PREP_PITCH * 16 : 0);
  if (int rc = launch_large("hash_bwd_walk_prep", prep, dim3((unsigned)wp.prep_blocks), WALK_PREP_THREADS, prep_args, prep_lds, s)) return rc;
  const void* reduce = with_mode(mode, [](auto mode_c) { return (const void*)hash_bwd_walk_reduce_k<decltype(mode_c)::value>; });
  const unsigned units = (unsigned)compute_units(), groups = (unsigned)wp.n_tasks < units ? (unsigned)wp.n_tasks : units;
  int64_t most_rows = 0;
  for (int l = 0; l < levels; ++l) most_rows = geom->rows[l] > most_rows ? geom->rows[l] : most_rows;
  DevGeom gg = g;
  for (int p = 0; p < (feat + 1) / 2; ++p) {
    int f0 = 2 * p;
    void* args[] = {(void*)&ws, (void*)&N, (void*)&gg, (void*)&wp, (void*)&primes, (void*)&table, (void*)&mode, (void*)&feat, (void*)&p};
    if (int rc = launch_large("hash_bwd_walk", walk, dim3(groups), WALK_THREADS, args, (size_t)2 * BIN_ROWS * 8, s)) return rc;
    if (ws.slots == nullptr) continue;
    void* reduce_args[] = {(void*)&ws, (void*)&table, (void*)&gg, (void*)&wp, (void*)&feat, (void*)&f0};
    const dim3 grid((unsigned)((most_rows + REDUCE_THREADS * 4 - 1) / (REDUCE_THREADS * 4)), (unsigned)levels);
    if (int rc = launch_large("hash_bwd_walk_reduce", reduce, grid, REDUCE_THREADS, reduce_args, 0, s)) return rc;
  }
  return 0;
}

static int launch_bwd_bin_piece(const void* coords, int cdt, int64_t csn, int64_t csd, const void* dout, int ddt, int64_t dout_stride,
                                void* table, int mode, int64_t N, const nf_hash_geom* geom, const DevGeom& g, const int64_t* primes, float scale,
                                void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const bool g32 = ddt == NF_F32;
  BinPlan bp;
  int64_t R;
  const bool wide = wide_blocks(N, geom);
  int points = fill_points(wide);
  NF_REQUIRE(bin_plan(N, points, geom, &bp, &R, !g32), NF_EUNSUPPORTED, "binned backward does not cover this geometry");
  NF_REQUIRE(((uintptr_t)workspace & 15u) == 0, NF_EALIGN, "workspace must be 16-byte aligned");
  BinWs ws;
  if (bin_ws(workspace, bp, N, points, R, g32 ? 4 : 3, true, &ws) > workspace_bytes) bin_ws(workspace, bp, N, points, R, g32 ? 4 : 3, false, &ws);
  const int NB = bp.binbase[bp.n_levels];
  int max_nb = 1, bin_pieces = 0;
  for (int l = 0; l < bp.n_levels; ++l) {
    max_nb = bp.nbins[l] > max_nb ? bp.nbins[l] : max_nb;
    bin_pieces += (bp.nbins[l] + 63) / 64;
  }
  const int feat = geom->feat, D = g.dims == 2 ? 2 : 3;
  auto pick_fill = [&](auto wide_c, auto g32_c) -> const void* {
    constexpr bool W = decltype(wide_c)::value, G = decltype(g32_c)::value;
    return g.dims == 6   ? (const void*)hash_bwd_bin_fill_k<W, G, 3, 3>
           : g.dims == 5 ? (const void*)hash_bwd_bin_fill_k<W, G, 3, 2>
           : g.dims == 4 ? (const void*)hash_bwd_bin_fill_k<W, G, 3, 1>
           : g.dims == 3 ? (const void*)hash_bwd_bin_fill_k<W, G, 3>
                         : (const void*)hash_bwd_bin_fill_k<W, G, 2>;
  };
  const void* fill = wide ? (g32 ? pick_fill(std::true_type{}, std::true_type{}) : pick_fill(std::true_type{}, std::false_type{}))
                          : (g32 ? pick_fill(std::false_type{}, std::true_type{}) : pick_fill(std::false_type{}, std::false_type{}));
  const void* accum = with_mode(mode, [&](auto mode_c) -> const void* {
    constexpr int M = decltype(mode_c)::value;
    auto kernel = [&](auto two_c) -> const void* {
      constexpr bool TWO = decltype(two_c)::value;
      return ddt == NF_F16    ? (const void*)hash_bwd_bin_accum_k<F16, M, TWO>
             : ddt == NF_BF16 ? (const void*)hash_bwd_bin_accum_k<BF16, M, TWO>
                              : (const void*)hash_bwd_bin_accum_k<F32, M, TWO>;
    };
    return feat == 2 ? kernel(std::true_type{}) : kernel(std::false_type{});
  });
  const void* reduce = with_mode(mode, [](auto mode_c) { return (const void*)hash_bwd_bin_reduce_k<decltype(mode_c)::value>; });
  const size_t fill_lds = ((size_t)stage_records(D, wide) * (g32 ? 4 : 3) + 3 * (size_t)max_nb + 1 + NF_MAX_LEVELS) * 4;
  const size_t acc_lds = (size_t)BIN_ROWS * 2 * sizeof(unsigned long long) + ((size_t)LIST + LIST_PAD + (NB < SPLIT_MAX_BINS ? NB : SPLIT_MAX_BINS) + 1 + (NB > SPLIT_MAX_BINS ? 2 * LATE_MAX : 0) + 2) * 4;
  auto launch = [&](const char* what, const void* kern, dim3 grid, int threads, void** args, size_t lds) { return launch_large(what, kern, grid, threads, args, lds, s); };
  const unsigned units = (unsigned)compute_units();
  // Levels of a fill workgroup: four, whose gradients are one 16-byte piece of a row, or fewer where that leaves less than two workgroups a
  // unit.  16 levels of 2^19 rows, fp16, uniform points, whole backward (us) with 16 / 4 / 2 / 1 levels to a workgroup: 2^14 points 100 / 72 /
  // 67 / 66, 2^15 104 / 76 / 72 / 73, 2^16 108 / 83 / 84 / 84, 2^17 114 / 93 / 95 / 100, 2^18 145 / 134 / 136 / 147, 2^20 378 / 374 / 418 / 530.
  // All levels where the gradient rows do not stay in the memory-side cache (256 MB) from one workgroup's four levels to the next's: fill of one
  // pass (us), several workgroups / one to a row: 134 MB, fp16 2^21 points 352 / 356; 190 MB, float32 390 / 398, fp16 rows of four 290 / 297; 268 MB, float32 2^21
  // 630 / 538, fp16 rows of four 487 / 417, of eight 240 / 234.  (The workgroups of a row next to each other on one XCD: 574 and 438 there, but 173 -> 216 at fp16 2^20.)
  int step = N * bp.n_levels * feat * (g32 ? 4 : 2) > FILL_ROWS_BYTES ? bp.n_levels : 4;
  while (step > 1 && (int64_t)ws.blocks * ((bp.n_levels + step - 1) / step) < 2 * (int64_t)units) step /= 2;
  // more than three dimensions: the whole pipeline once per corner of the extra coordinates (`hi`), see ExtraDims
  const int passes = g.dims > 3 ? 1 << (g.dims - 3) : 1;
  for (int hi = 0; hi < passes; ++hi)
    for (int f0 = 0; f0 < feat; f0 += 2) {
      DevGeom gg = g;
      void* fill_args[] = {(void*)&coords, (void*)&cdt, (void*)&csn, (void*)&csd, (void*)&dout, (void*)&dout_stride, (void*)&N, (void*)&points,
                           (void*)&gg, (void*)&bp, (void*)&primes, (void*)&scale, (void*)&ws, (void*)&max_nb, (void*)&feat, (void*)&f0, (void*)&hi, (void*)&step};
      if (int rc = launch("hash_bwd_bin_fill", fill, dim3((unsigned)ws.blocks, (unsigned)((bp.n_levels + step - 1) / step)), wide ? FILL_WIDE_THREADS : FILL_THREADS, fill_args, fill_lds)) return rc;
      void* totals_args[] = {(void*)&ws, (void*)&bp};
      const unsigned pieces = (unsigned)((ws.blocks + TOTALS_BLOCKS - 1) / TOTALS_BLOCKS);
      if (int rc = launch("hash_bwd_bin_totals", (const void*)hash_bwd_bin_totals_k, dim3((unsigned)bin_pieces, pieces), 64 * TOTALS_WAVES, totals_args, 0)) return rc;
      void* acc_args[] = {(void*)&ws, (void*)&table, (void*)&gg, (void*)&bp, (void*)&feat, (void*)&f0};
      if (int rc = launch("hash_bwd_bin_accum", accum, dim3(units), ACC_THREADS, acc_args, acc_lds)) return rc;
      void* reduce_args[] = {(void*)&ws, (void*)&table, (void*)&gg, (void*)&bp, (void*)&feat, (void*)&f0, (void*)&ddt};
      const unsigned max_splits = (unsigned)NB < ws.max_slots / 2 ? (unsigned)NB : ws.max_slots / 2;
      if (int rc = launch("hash_bwd_bin_reduce", reduce, dim3(2 * BIN_ROWS / REDUCE_VALUES, max_splits), REDUCE_THREADS, reduce_args, 0)) return rc;
    }
  return 0;
}

}  // namespace nf
