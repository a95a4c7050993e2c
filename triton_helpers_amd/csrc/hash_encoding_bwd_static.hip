// nf_hash_encode_bwd_static: the hash-encoding backward for callers that cannot allocate device memory (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).  It is nf_hash_encode_bwd with the
// scratch of its sort-and-accumulate kernels taken from a device array that lives in this library instead of a
// caller's workspace: nothing is allocated or freed, on the device or on the host.
//
// The array is NF_HASH_BWD_STATIC_BYTES large on every GPU the library is loaded on and stays until the process ends.
// Its device address differs per GPU and is asked for once per device (hipGetSymbolAddress with that device
// current); host code never uses the array's name for anything else.  All calls on one GPU share the array: calls that
// overlap in time on one GPU (two streams, two threads) race on it.  The kernels clear what they need cleared
// themselves (with a fill kernel, not a memset node), so the previous call's contents do not matter.
#include <atomic>

#include "hash_common.h"

namespace nf {

static __device__ __attribute__((used)) __align__(256) unsigned char scratch[NF_HASH_BWD_STATIC_BYTES];

// scratch's address on the current device (cached per device ordinal; racing first calls ask twice and agree)
static int static_scratch(void** out) {
  static std::atomic<void*> cached[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail((int)e, "hipGetDevice: %s", hipGetErrorString(e));
  NF_REQUIRE(dev >= 0 && dev < 64, NF_EUNSUPPORTED, "device ordinal %d beyond the 64 this entry point keeps addresses for", dev);
  void* p = cached[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) return fail(e != hipSuccess ? (int)e : NF_EINVAL, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    cached[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return 0;
}

}  // namespace nf

using namespace nf;

extern "C" int64_t nf_hash_encode_bwd_static_bytes(void) { return (int64_t)NF_HASH_BWD_STATIC_BYTES; }

extern "C" int nf_hash_encode_bwd_static(const void* coords, int coords_dtype, int64_t csn, int64_t csd, const void* dout,
                                         int dout_dtype, int64_t dout_stride_n, float* dtable, int64_t n_points,
                                         const nf_hash_geom* geom, const int64_t* primes, float scale, int flags, void* stream) {
  NF_REQUIRE(geom != nullptr, NF_EINVAL, "geom is NULL");
  NF_REQUIRE(n_points >= 0, NF_EINVAL, "n_points negative");
  // Which variant's least scratch fits: the sorted records (~1.3 KB per point; float32 ~2.1) or the walk without them (~0.1 to 0.2 KB) of the
  // whole batch; else of its largest part that fits, the rest being a call of its own; else the bit-planes (~110 B per point, 16-bit
  // gradients of 3-D points only), which also run where the rest would need a second pass of records: 16 levels of 2^19 rows, float16,
  // 107000 points as 100864 and a rest for the atomics 146 us, with the bit-planes 180; 107000 as two halves 228; 2^14 rows, 2^21 points
  // 370 us in two parts, with the bit-planes 1620.  A call that would need none of these (small batches and shapes that scatter with
  // atomics) needs no scratch at all.
  const int64_t limit = (int64_t)NF_HASH_BWD_STATIC_BYTES;
  auto need_of = [&](int64_t n, int f) { return bwd_workspace_bytes(n, geom, dout_dtype, f, false); };
  const int64_t need_bin = need_of(n_points, flags & ~NF_HASH_FORCE_PLANES), need_planes = need_of(n_points, flags | NF_HASH_FORCE_PLANES);
  int64_t piece = n_points;
  int use_flags = flags;
  if (need_bin > limit || (flags & NF_HASH_FORCE_PLANES)) {
    const bool planes = need_planes > 0 && need_planes <= limit;
    int64_t part = (n_points + 1) / 2, beyond = n_points;  // part fits, beyond does not
    bool parts = !(flags & NF_HASH_FORCE_PLANES) && need_of(part, flags) <= limit;
    while (parts && beyond - part > 1) {
      const int64_t mid = part + (beyond - part) / 2;
      (need_of(mid, flags) <= limit ? part : beyond) = mid;
    }
    const int64_t rest = n_points - part;
    parts = parts && need_of(rest, flags) <= limit;
    if (parts && (!planes || bwd_walk_applies(part, geom, flags) || rest < bwd_records_min(geom, flags))) {
      piece = part;
    } else {
      NF_REQUIRE(planes, NF_EINVAL,
                 "n_points=%lld needs %lld bytes of scratch (%lld with the bit-plane variant, 0 = not applicable to this call); "
                 "the static scratch holds %lld: split the batch or call nf_hash_encode_bwd with a workspace",
                 (long long)n_points, (long long)need_bin, (long long)need_planes, (long long)limit);
      use_flags |= NF_HASH_FORCE_PLANES;
    }
  }
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  int64_t n0 = 0;
  do {  // (an empty batch too: its arguments are checked)
    const int64_t n = n_points - n0 < piece ? n_points - n0 : piece;
    const char* c = (const char*)coords + n0 * csn * (dtype_ok(coords_dtype) ? dtype_size(coords_dtype) : 0);
    const char* d = (const char*)dout + n0 * dout_stride_n * (dtype_ok(dout_dtype) ? dtype_size(dout_dtype) : 0);
    if (int rc = nf_hash_encode_bwd(c, coords_dtype, csn, csd, d, dout_dtype, dout_stride_n, dtable, n, geom, primes, scale, ws, limit, use_flags, stream))
      return rc;
    n0 += n;
  } while (n0 < n_points);
  return 0;
}
