// Host side of the role-split backward of whole networks (fused_mlp_bwd_roles.h), the sum over its slots, and the entry point.
#include "fused_mlp_bwd_roles.h"

namespace nf {

struct RolesGrads {
  void *dw_in, *dw_hid, *dw_out, *db_in, *db_hid, *db_out;  // NULL: not wanted
  int d_in, d_hidden, d_out, depth;
};

// gradients = the slots' sums in a fixed order (the same bits on every run), rounded once to G.  A workgroup takes one tile or
// one layer's bias sums: sixteen interleaved runs over the slots (16 bytes per lane, four loads in flight), then a tree.
template <typename G>
__global__ __launch_bounds__(1024) void mlp_sum_roles_k(const float* partials, int n_slots, int64_t slot_stride, RolesGrads p) {
  __shared__ f32x4_t part[16][64];
  const int hp = p.d_hidden <= 32 ? 32 : 64, layer = blockIdx.y, tile = blockIdx.x;
  const int columns_log2 = roles_columns_log2(hp, layer == p.depth), mt = tile >> columns_log2, nt = tile & ((1 << columns_log2) - 1);
  const int out_dim = layer == p.depth ? p.d_out : p.d_hidden, in_dim = layer == 0 ? p.d_in : p.d_hidden;
  const bool bias = tile == roles_tiles(hp);
  const size_t hid = (size_t)(layer - 1) * p.d_hidden;  // rows of the hidden layers in front (layers 1 .. depth - 1)
  typedef typename G::storage S;
  S* dst;
  if (bias) dst = layer == 0 ? (S*)p.db_in : layer == p.depth ? (S*)p.db_out : p.db_hid ? (S*)p.db_hid + hid : nullptr;
  else dst = layer == 0 ? (S*)p.dw_in : layer == p.depth ? (S*)p.dw_out : p.dw_hid ? (S*)p.dw_hid + hid * p.d_hidden : nullptr;
  if (dst == nullptr || (!bias && (16 * mt >= out_dim || 16 * nt >= in_dim))) return;
  const int lane = threadIdx.x & 63, ty = threadIdx.x >> 6;
  f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
  if (!bias || 4 * lane < (out_dim + 15) / 16 * 16) {  // a bias block holds whole 16-value tiles of its layer
    const float* src = partials + (size_t)layer * roles_layer_floats(hp) + tile * 256 + lane * 4;
    int sl = ty;
    for (; sl + 48 < n_slots; sl += 64) {
      f32x4_t v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4_t*>(src + (size_t)(sl + 16 * k) * slot_stride);
#pragma unroll
      for (int k = 0; k < 4; ++k) sum += v[k];
    }
    for (; sl < n_slots; sl += 16) sum += *reinterpret_cast<const f32x4_t*>(src + (size_t)sl * slot_stride);
  }
  part[ty][lane] = sum;
  __syncthreads();
  if (ty != 0) return;
  f32x4_t total = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < 16; q += 4) total += (part[q][lane] + part[q + 1][lane]) + (part[q + 2][lane] + part[q + 3][lane]);
  if (bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * lane + r < out_dim) dst[4 * lane + r] = G::from_f32(total[r]);
    return;
  }
  const int c = 16 * nt + (lane & 15), r0 = 16 * mt + 4 * (lane >> 4);
  if (c >= in_dim) return;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (r0 + r < out_dim) dst[(size_t)(r0 + r) * in_dim + c] = G::from_f32(total[r]);
}

// How a network runs: chain waves of a workgroup, workgroups per compute unit, workgroups of the launch.  With more rows than
// a workgroup of four chain waves per unit takes in one round, twice or three times the chain waves hide each other's
// latencies (2^18 rows, us with 4 / with more: 64 -> 64 x 2 -> 64 SiLU 73 / 59, 32 -> 32 x 2 -> 16 ReLU 31 / 27); below, they
// only stage and wait (2^11 rows: 12.2 / 13.9).
struct RolesPlan {
  int cw, wgs;
  int64_t blocks;
};
static RolesPlan roles_plan(int64_t rows, int d_hidden, int depth, int act) {
  const int hp = d_hidden <= 32 ? 32 : 64;
  const bool shallow = depth <= roles_shallow(act);
  RolesPlan p = {4, 1, 0};
  if (shallow && rows > 64 * (int64_t)device_cus()) p.cw = hp == 64 ? 8 : 12;
  if (!shallow && hp == 32 && act == NF_ACT_RELU && 2 * roles_lds(32, depth, 64) <= LDS_LIMIT) p.wgs = 2;
  const int64_t n = 16 * p.cw, total = (rows + n - 1) / n, cap = (int64_t)device_cus() * p.wgs;
  const int64_t rounds = (total + cap - 1) / cap;  // every workgroup takes this many or one less
  p.blocks = (total + rounds - 1) / rounds;
  return p;
}

template <typename T, int HP, int ACT>
static int launch_roles(const MlpArgs& a, const RolesPlan& p, hipStream_t s) {
  constexpr int SH = roles_shallow(ACT), MANY = HP == 64 ? 8 : 12;
  const size_t lds = roles_lds(HP, a.depth, 16 * p.cw);
  const auto pick = [&](auto whole_c) -> const void* {
    constexpr WholePieces WHOLE = decltype(whole_c)::value;
    return a.depth > SH   ? (const void*)mlp_bwd_roles_k<T, HP, ACT, ROLES_MAX_DEPTH, 4, HP == 32 && ACT == NF_ACT_RELU ? 4 : 2, WHOLE>
           : p.cw == MANY ? (const void*)mlp_bwd_roles_k<T, HP, ACT, SH, MANY, MANY / 4 + 1, WHOLE>
                          : (const void*)mlp_bwd_roles_k<T, HP, ACT, SH, 4, 2, WHOLE>;
  };
  const void* kern;
  if constexpr (HP == 32) kern = pick(std::integral_constant<WholePieces, WholePieces::ANY>{});
  else kern = whole_pieces(a) ? pick(std::integral_constant<WholePieces, WholePieces::YES>{}) : pick(std::integral_constant<WholePieces, WholePieces::NO>{});
  const hipError_t ea = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (ea != hipSuccess) return fail((int)ea, "hipFuncSetAttribute: %s", hipGetErrorString(ea));
  void* args[] = {(void*)&a};
  const hipError_t e = hipLaunchKernel(kern, dim3((unsigned)p.blocks), dim3(64 * (p.cw + 4)), args, lds, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(mlp_bwd_roles): %s", hipGetErrorString(e));
  return check_launch("mlp_bwd_roles");
}

template <typename T, int HP>
static int dispatch_act(const MlpArgs& a, const RolesPlan& p, hipStream_t s) {
  switch (a.act) {
    case NF_ACT_RELU: return launch_roles<T, HP, NF_ACT_RELU>(a, p, s);
    case NF_ACT_SILU: return launch_roles<T, HP, NF_ACT_SILU>(a, p, s);
    case NF_ACT_RELU2: return launch_roles<T, HP, NF_ACT_RELU2>(a, p, s);
    case NF_ACT_GELU: return launch_roles<T, HP, NF_ACT_GELU>(a, p, s);
    default: return launch_roles<T, HP, NF_ACT_NONE>(a, p, s);
  }
}

size_t mlp_bwd_roles_bytes(int64_t rows, int d_hidden, int depth, int act) {
  if (rows <= 0 || depth < 1 || depth > ROLES_MAX_DEPTH) return 0;
  return (size_t)roles_plan(rows, d_hidden, depth, act).blocks * roles_slot_floats(d_hidden <= 32 ? 32 : 64, depth) * sizeof(float);
}

int launch_mlp_bwd_roles(const MlpArgs& a0, int dtype, int grad_dtype, void* const out[6], void* workspace, hipStream_t s) {
  MlpArgs a = a0;
  const RolesPlan plan = roles_plan(a.rows, a.d_hidden, a.depth, a.act);
  if (a.dx != nullptr) a.dx_vec = vec_load_ok(a.dx, a.dx_stride, a.d_in);  // stored 16 bytes at a time
  a.partials = reinterpret_cast<float*>(workspace);
  const int hp = a.d_hidden <= 32 ? 32 : 64;
  a.partial_stride = roles_slot_floats(hp, a.depth);
  int rc;
  if (a.d_hidden <= 32) rc = dtype == NF_BF16 ? dispatch_act<BF16, 32>(a, plan, s) : dispatch_act<F16, 32>(a, plan, s);
  else rc = dtype == NF_BF16 ? dispatch_act<BF16, 64>(a, plan, s) : dispatch_act<F16, 64>(a, plan, s);
  if (rc != 0) return rc;
  RolesGrads grads = {out[0], out[2], out[4], out[1], out[3], out[5], a.d_in, a.d_hidden, a.d_out, a.depth};
  const float* part = a.partials;
  int n = (int)plan.blocks;
  int64_t st = a.partial_stride;
  void* args[] = {(void*)&part, (void*)&n, (void*)&st, (void*)&grads};
  const void* kern = grad_dtype == NF_F32    ? (const void*)mlp_sum_roles_k<F32>
                     : grad_dtype == NF_BF16 ? (const void*)mlp_sum_roles_k<BF16>
                                             : (const void*)mlp_sum_roles_k<F16>;
  const hipError_t e = hipLaunchKernel(kern, dim3((unsigned)roles_tiles(hp) + 1, (unsigned)a.depth + 1), dim3(1024), args, 0, s);
  if (e != hipSuccess) return fail((int)e, "hipLaunchKernel(mlp_sum_roles): %s", hipGetErrorString(e));
  return check_launch("mlp_sum_roles");
}

}  // namespace nf
