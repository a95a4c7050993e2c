// Building blocks of the backward kernels whose workgroups are split by role (fused_mlp_bwd_roles.h, reversible_bwd.hip): chain waves
// that carry rows through the layers and back, and gradient waves that hold the weight gradients.
//
// Weights and the rows that the roles exchange lie in LDS row-major, in rows of 128 bytes.  A product with W reads its fragments
// as rows, a product with W^T (or over the rows of an exchanged panel) reads the same bytes through ds_read_b64_tr_b16.
#pragma once

#include "mlp_tile.h"

namespace nf {

constexpr int ROLES_PITCH = 128;  // bytes of a row in LDS

// xor on the number of an 8-byte piece of row r.  LDS serves half a wave at a time from 64 banks, two rows wide: the sixteen rows and two lane
// groups of a row fragment (pieces g), and the eight rows and four pieces of a transposing read, then fall on 64 different ones.  (With an
// xor over eight pieces only, half the banks were used: 2.26 against 1.27 clocks of the kernel's timer per read of 512 bytes.)
__device__ __forceinline__ int swizzle(int r) { return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 3) | (((r >> 3) & 1) * 3); }

// A lane's byte offsets: n = lane % 16, g = lane / 16.  A tile row (16 rows) is 2048 bytes further; a K-chunk of 32 columns: ^ 64.
// columns 4g .. of row n (chain order); the four 16 columns on: ^ 32
__device__ __forceinline__ int chain_offset(int n, int g) { return n * ROLES_PITCH + ((g ^ swizzle(n)) << 3); }
// columns 8g .. of row n (natural order); the four behind them: ^ 8
__device__ __forceinline__ int natural_offset(int n, int g) { return n * ROLES_PITCH + (((2 * g) ^ swizzle(n)) << 3); }
// transposing reads: this lane supplies row 4g + n / 4, columns 4 (n % 4) ..; tile column t: ^ 32 t; rows + 16: 2048
__device__ __forceinline__ int tr_offset(int n, int g) { return (4 * g + (n >> 2)) * ROLES_PITCH + (((n & 3) ^ swizzle(4 * g + (n >> 2))) << 3); }

// Eight 16-bit values of row r from column c0 on, zero beyond `width` and `rows`.  vec: rows of whole 16-byte aligned pieces.
// Otherwise a row's last piece is read as the eight values that end with the row and shifted, so that no access leaves the row.
__device__ __forceinline__ Frag load_row8(const uint16_t* base, int64_t stride, int64_t r, int64_t rows, int width, int c0, bool vec) {
  Frag f;
  f.u = make_uint4(0u, 0u, 0u, 0u);
  if (r >= rows || c0 >= width) return f;
  const uint16_t* p = base + r * stride;
  if (vec) {
    f.u = *reinterpret_cast<const uint4*>(p + c0);
  } else if (width >= 8) {
    const int start = c0 < width - 8 ? c0 : width - 8, skip = c0 - start;  // values of the window in front of c0
    uint4 v;
    __builtin_memcpy(&v, p + start, 16);
    if (skip & 4) v = make_uint4(v.z, v.w, 0u, 0u);
    if (skip & 2) v = make_uint4(v.y, v.z, v.w, 0u);
    if (skip & 1) v = make_uint4((v.x >> 16) | (v.y << 16), (v.y >> 16) | (v.z << 16), (v.z >> 16) | (v.w << 16), v.w >> 16);
    f.u = v;
  } else {  // a row of less than eight values: c0 == 0
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (j < width) f.w[j >> 1] |= (uint32_t)p[j] << (16 * (j & 1));
  }
  return f;
}

// The same eight values back.
__device__ __forceinline__ void store_row8(uint16_t* base, int64_t stride, int64_t r, int64_t rows, int width, int c0, const Frag& f, bool vec) {
  if (r >= rows || c0 >= width) return;
  uint16_t* p = base + r * stride + c0;
  if (vec) {
    *reinterpret_cast<uint4*>(p) = f.u;
  } else if (c0 + 8 <= width) {
    __builtin_memcpy(p, &f.u, 16);
  } else {
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (c0 + j < width) p[j] = (uint16_t)(f.w[j >> 1] >> (16 * (j & 1)));
  }
}

// two 8-byte pieces -> fragment
__device__ __forceinline__ Frag read_pieces(const char* p0, const char* p1) {
  const uint2 a = *reinterpret_cast<const uint2*>(p0), b = *reinterpret_cast<const uint2*>(p1);
  Frag f;
  f.w[0] = a.x; f.w[1] = a.y; f.w[2] = b.x; f.w[3] = b.y;
  return f;
}
__device__ __forceinline__ Frag read_pieces_tr(const char* p0, const char* p1) {
  typedef tr_v4i16 __attribute__((address_space(3))) * lds_ptr;
  const uint2 a = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p0));
  const uint2 b = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p1));
  Frag f;
  f.w[0] = a.x; f.w[1] = a.y; f.w[2] = b.x; f.w[3] = b.y;
  return f;
}
__device__ __forceinline__ void write_pieces(char* p0, char* p1, const Frag& f) {
  *reinterpret_cast<uint2*>(p0) = make_uint2(f.w[0], f.w[1]);
  *reinterpret_cast<uint2*>(p1) = make_uint2(f.w[2], f.w[3]);
}

// Waits for what is on its way into f, here: behind stores that not every path issues, the compiler could only wait for those as well.
__device__ __forceinline__ void arrived(Frag& f) { asm volatile("" : "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.w[2]), "+v"(f.w[3])); }

// Workgroup barrier that waits for this wave's LDS traffic only: global loads and the dx stores stay in flight across it.
__device__ __forceinline__ void roles_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// body(integral_constant<0 .. N - 1>): a loop over layers whose register arrays are indexed by constants whatever its size
template <int N, int I = 0, typename Body>
__device__ __forceinline__ void each_layer(Body&& body) {
  if constexpr (I < N) {
    body(std::integral_constant<int, I>{});
    each_layer<N, I + 1>(body);
  }
}
// Hand-over between waves without a barrier: a wave writes how far it is into its flag, others read the flags of N waves.  A wave's LDS
// operations complete in order, so what it wrote before its flag is there when the flag is seen.
__device__ __forceinline__ void post(int* flag, int count) {
  auto p = (__attribute__((address_space(3))) int*)flag;
  uint64_t all;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_mov_b64 %0, exec\n\ts_mov_b64 exec, 1\n\tds_write_b32 %1, %2\n\ts_mov_b64 exec, %0"  // by one lane
               : "=&s"(all)
               : "v"(p), "v"(count)
               : "memory");
}
template <int N>  // waits until all of flags[0 .. N) have reached count
__device__ __forceinline__ void await(const int* flags, int lane, int count) {
  auto p = (const __attribute__((address_space(3))) int*)flags + (lane < N ? lane : N - 1);
  int v;  // (one statement: a loop the compiler sees would cut its register allocation in two)
  asm volatile(
      "0:\n\tds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)\n\tv_cmp_gt_i32_e32 vcc, %2, %0\n\ts_cbranch_vccz 1f\n\ts_sleep 1\n\ts_branch 0b\n1:"
      : "=&v"(v)
      : "v"(p), "s"(count)
      : "vcc", "memory");
}
// How the roles of a workgroup of CW chain waves pass a section's panels on; `section` counts a wave's sections, areas alternate.  Several
// chain waves on a SIMD go by flags: with barriers they would be in step and all want the same unit at a time (64 -> 64 with three hidden
// SiLU layers, 2^21 rows, us: 518, so 465; 64-wide reversible couplings 6 %).  A chain wave that has its SIMD to itself is better off with
// barriers, which are quicker (64 -> 64 with nine hidden ReLU layers, 2^19 rows: 268, with flags 286).
template <int CW>
struct Sections {
  static constexpr bool FLAGS = CW > 4;
  int* flags;  // LDS, 32 zeros: sections parked by each chain wave, + 16: read by each gradient wave
  int section;

  // chain waves: an area is free when the gradient waves have read the section before the last
  __device__ __forceinline__ void room(int lane) const {
    if constexpr (FLAGS) await<4>(flags + 16, lane, section - 1);
  }
  __device__ __forceinline__ void parked(int wave) {
    ++section;
    if constexpr (FLAGS) post(flags + wave, section);
    else roles_barrier();
  }
  // gradient waves
  __device__ __forceinline__ void begin(int lane) {
    ++section;
    if constexpr (FLAGS) {
      await<CW>(flags, lane, section);
      __builtin_amdgcn_s_setprio(3);  // what the chain waves wait for goes first (four 64-wide couplings, 2^20 rows: 957 -> 903 us)
    } else {
      roles_barrier();
    }
  }
  __device__ __forceinline__ void done(int wave) const {
    if constexpr (FLAGS) {
      post(flags + 16 + wave - CW, section);
      __builtin_amdgcn_s_setprio(0);
    }
  }
};

// A uniform value the optimiser knows nothing about: what is derived from it is worked out where it is used instead of being
// kept for all layers at once (the comparisons and addresses of nine layers do not fit the scalar registers).
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

}  // namespace nf
