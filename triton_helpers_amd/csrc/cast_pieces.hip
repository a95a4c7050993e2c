// The parameters of a network cast to float16 in one launch (mixed-precision training keeps them in float32): up to eight
// tensors of a few thousand values, so that what a launch per tensor costs is the launch (2 us each on the GPU, more on the host).
#include "nf_common.h"

namespace nf {

constexpr int MAX_PIECES = 8;

struct CastPieces {
  const float* src[MAX_PIECES];
  int64_t first[MAX_PIECES + 1];  // first destination element of each piece, a multiple of 8
  int64_t count[MAX_PIECES];
  int n;
};

__global__ __launch_bounds__(256) void cast_pieces_k(CastPieces pc, uint16_t* dst) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pc.first[pc.n]) return;
  int k = 0;
  while (k + 1 < pc.n && i >= pc.first[k + 1]) ++k;
  const int64_t e = i - pc.first[k];
  if (e < pc.count[k]) dst[i] = F16::from_f32(pc.src[k][e]);
}

}  // namespace nf

using namespace nf;

extern "C" int nf_cast_pieces_f16(const float* const* src, const int64_t* count, int n, void* dst, void* stream) {
  NF_REQUIRE(n >= 0 && n <= MAX_PIECES, NF_EINVAL, "%d pieces outside 0..%d", n, MAX_PIECES);
  CastPieces pc = {};
  pc.n = n;
  for (int k = 0; k < n; ++k) {
    NF_REQUIRE(count[k] >= 0 && (src[k] != nullptr || count[k] == 0), NF_EINVAL, "piece %d: NULL or a negative count", k);
    pc.src[k] = src[k];
    pc.count[k] = count[k];
    pc.first[k + 1] = pc.first[k] + (count[k] + 7) / 8 * 8;
  }
  if (pc.first[n] == 0) return 0;
  NF_REQUIRE(dst != nullptr && (uintptr_t)dst % 2 == 0, NF_EINVAL, "destination is NULL or misaligned");
  hipLaunchKernelGGL(cast_pieces_k, dim3((unsigned)((pc.first[n] + 255) / 256)), dim3(256), 0, (hipStream_t)stream, pc, (uint16_t*)dst);
  return check_launch("cast_pieces");
}
