// Fused MLP on float32 tensors with float32 products: v_mfma_f32_16x16x4_f32, float32 storage, operands and
// accumulation, so values keep the float32 range and 24-bit mantissa.  (The reference multiplies float32 tensors in
// TF32, fully_fused_mlp/kernel.py:17-47: the same range with a 10-bit mantissa.)  The 16-bit kernels are the fast
// path; this one is bound by the float32 matrix rate (157 TFLOP/s) and, beyond two hidden layers, by its activations'
// round trip in the backward.
//
// Forward: one launch for any depth.  A wave carries 32 rows (two groups of 16), in small batches 16, through all layers in registers.
// The product is formed transposed, out^T = W * h^T, so that the 16x16 result tile of a layer (lane (r, g), register v:
// feature 16*mt + 4*g + v of row r) is already the K operand of the next layer when K is walked in the order
// 16*t + 4*g + v; the weights are read from LDS in that order (one ds_read_b128 per four products).  Weights of all
// layers stay in LDS when they fit (up to eight layers), else each layer is staged in turn.
// Backward of one or two hidden layers: one launch, see mlp32_bwd_k.  Of more: the forward is replayed keeping every hidden
// layer's pre-activation in the caller's workspace ([depth][rows][d_hidden] float32), then one launch per layer, last to
// first, forms dW += dz^T h, db += sum dz and overwrites the pre-activation of the layer in front with its gradient.  A
// workgroup sums its waves' dW in LDS and stores one partial; a small second kernel adds the partials into the caller's
// accumulators (at most 32 adds per address: thousands of waves adding into the same 16 KB of dW directly cost more than
// the products).
#include "fused_mlp.h"

namespace nf {

constexpr int W32_STRIDE = 68;                           // floats per staged weight row (64 + 4)
constexpr int W32_LAYER = 64 * W32_STRIDE + 64;          // floats per staged layer: weights, then the bias
constexpr int W32_RESIDENT_MAX = 8;                      // layers kept in LDS at once
constexpr int T32_STRIDE = 80;                           // floats per row of a wave's 16-row transposing panel
constexpr int PART32 = 64 * 64 + 64;                     // floats of one workgroup's partial dW (64 x 64) and db (64)
constexpr int SLOTS32 = 512;                             // most workgroups of a backward launch

struct Mlp32Args {
  const float* x;
  int64_t x_stride;
  float* y;
  int64_t y_stride;
  const float *w_in, *b_in, *w_hid, *b_hid, *w_out, *b_out;
  float* z;  // [depth][rows][d_hidden] pre-activations, or NULL
  int64_t rows;
  int d_in, d_hidden, d_out, depth, act;
  int resident;  // 1: every layer's weights staged once per workgroup
  int n_layers;  // linear layers computed: depth + 1, or depth when only the pre-activations are wanted
  int block_step, wave_step;  // chunks of the forward between neighbouring workgroups, and between the waves of one
};

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Rows x columns tile in "chain order": lane (r, g) holds columns 16*t + 4*g + v, v = 0..3, of row r.
__device__ __forceinline__ f32x4_t load_chain(const float* base, int64_t stride, int64_t row, int64_t rows, int col, int width,
                                              bool vec) {
  f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (row >= rows) return v;
  const float* p = base + row * stride + col;
  if (vec && col + 3 < width) return *reinterpret_cast<const f32x4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (col + i < width) v[i] = p[i];
  return v;
}

__device__ __forceinline__ void store_chain(float* base, int64_t stride, int64_t row, int64_t rows, int col, int width, bool vec,
                                            f32x4_t v) {
  if (row >= rows) return;
  float* p = base + row * stride + col;
  if (vec && col + 3 < width) {
    *reinterpret_cast<f32x4_t*>(p) = v;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (col + i < width) p[i] = v[i];
}

// Four values of a row of a padded 64 x 64 weight matrix, n_out x n_in in memory
__device__ __forceinline__ f32x4_t load_weights32(const float* w, int n_out, int n_in, bool vec, int o, int c) {
  f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (o >= n_out) return v;
  const float* row = w + (size_t)o * n_in;
  if (vec) {
    if (c < n_in) v = *reinterpret_cast<const f32x4_t*>(row + c);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < n_in) v[e] = row[c + e];
  }
  return v;
}

// A matrix over the workgroup's threads: fetch() and, where it is used, put(o, c, v).  Its loads leave together: one after the other
// they cost a layer 4 us, a third of a launch on 10^5 rows.
template <int THREADS>
struct Layer32 {
  static constexpr int PER = 1024 / THREADS, ROWS = THREADS / 16;
  f32x4_t v[PER];
  __device__ __forceinline__ void fetch(const float* w, int n_out, int n_in, int tid) {
    const bool vec = n_in % 4 == 0 && (uintptr_t)w % 16 == 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = load_weights32(w, n_out, n_in, vec, (tid >> 4) + ROWS * k, 4 * (tid & 15));
  }
  template <typename Put>
  __device__ __forceinline__ void spread(int tid, Put&& put) const {
#pragma unroll
    for (int k = 0; k < PER; ++k) put((tid >> 4) + ROWS * k, 4 * (tid & 15), v[k]);
  }
};
template <int THREADS = 256, typename Put>
__device__ __forceinline__ void read_layer32(const float* w, int n_out, int n_in, int tid, Put&& put) {
  Layer32<THREADS> m;
  m.fetch(w, n_out, n_in, tid);
  m.spread(tid, put);
}

__device__ __forceinline__ void stage_layer32(float* dst, const float* w, const float* b, int n_out, int n_in, int tid) {
  read_layer32(w, n_out, n_in, tid, [&](int o, int c, f32x4_t v) { *reinterpret_cast<f32x4_t*>(dst + o * W32_STRIDE + c) = v; });
  if (tid < 64) dst[64 * W32_STRIDE + tid] = (b != nullptr && tid < n_out) ? b[tid] : 0.0f;
}

// Forward.  NT: 16-row groups that a wave carries at once (fwd32()).  PIECES: rows of x and y are whole 16-byte aligned pieces, which are read and
// written without a test per value.  Bound by the float32 products (157 TFLOP/s) from about 2^18 rows; below by what a workgroup waits for before
// its first one.  Layers staged one after the other, rows asked for when the chunk in front was done, 128 rows to a workgroup -> this, us: 32 -> 64 ->
// 64 -> 16, 4096 rows 11.4 -> 7.4, 100003 28.7 -> 23.6 (1.4 GFLOP), 2^18 47.9 -> 46.0; eight hidden layers of 64, 2^15 42.9 -> 35.4; 64 -> 64 -> 64 ->
// 64, 2^20 265 -> 249.
template <int ACT, int NT, bool PIECES>
__global__ __launch_bounds__(256, 2) void mlp32_fwd_k(Mlp32Args a) {
  extern __shared__ float lds32[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int H = a.d_hidden, last = a.depth;
  auto layer_w = [&](int l) { return l == 0 ? a.w_in : l == last ? a.w_out : a.w_hid + (size_t)(l - 1) * H * H; };
  auto layer_b = [&](int l) -> const float* {
    return l == 0 ? a.b_in : l == last ? a.b_out : (a.b_hid ? a.b_hid + (size_t)(l - 1) * H : nullptr);
  };
  auto n_in = [&](int l) { return l == 0 ? a.d_in : H; };
  auto n_out = [&](int l) { return l == last ? a.d_out : H; };
  const bool x_vec = ((uintptr_t)a.x % 16 == 0) && (a.x_stride % 4 == 0);
  const bool y_vec = a.y != nullptr && ((uintptr_t)a.y % 16 == 0) && (a.y_stride % 4 == 0);
  const int kt_in = (a.d_in + 15) / 16;
  // The next chunk's rows are requested before this one's products.
  const int64_t n_chunks = (a.rows + 16 * NT - 1) / (16 * NT), per_round = (int64_t)gridDim.x * 4;
  const int64_t first_of_workgroup = (int64_t)blockIdx.x * a.block_step, first_chunk = first_of_workgroup + (int64_t)wave * a.wave_step;
  f32x4_t nx[NT][4];  // (PIECES)
  auto load_rows = [&](int64_t chunk) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int64_t row = chunk * (16 * NT) + 16 * nt + r;
      const float* p = a.x + (row < a.rows ? row : a.rows - 1) * a.x_stride;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= kt_in) break;
        const int col = 16 * t + 4 * g;
        nx[nt][t] = *reinterpret_cast<const f32x4_t*>(p + (col < a.d_in ? col : 0));
      }
    }
  };
  if (a.resident) {
    // The layers are staged LAYERS at a time, their loads under way together and the first rows' behind them; layer by layer each waited
    // for the one in front.
    constexpr int LAYERS = 3, PER = 1024 / 256;
    for (int l0 = 0; l0 < a.n_layers; l0 += LAYERS) {
      f32x4_t v[LAYERS][PER];
      // a wave takes the bias of a layer
      const int bl = l0 + wave;
      const float* b = wave < LAYERS && bl < a.n_layers ? layer_b(bl) : nullptr;
      const bool has_bias = b != nullptr && lane < n_out(bl);
      const float bias = *(has_bias ? b + lane : a.w_in);
#pragma unroll
      for (int k = 0; k < LAYERS; ++k) {
        const int l = l0 + k;
        if (l >= a.n_layers) break;
        const float* w = layer_w(l);
        const int rows = n_out(l), cols = n_in(l);
        if (cols % 4 != 0 || (uintptr_t)w % 16 != 0) continue;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          if (16 * i >= rows) break;  // no tile reads these (32 -> 32 x 4 -> 1, 56000 rows, with them 13.9 us, without 13.0)
          const int o = (tid >> 4) + 16 * i, c = 4 * (tid & 15);
          v[k][i] = *reinterpret_cast<const f32x4_t*>(w + (o < rows ? o : 0) * cols + (c < cols ? c : 0));
        }
      }
      if (PIECES && l0 == 0) load_rows(first_chunk);
#pragma unroll
      for (int k = 0; k < LAYERS; ++k) {
        const int l = l0 + k;
        if (l >= a.n_layers) break;
        float* dst = lds32 + l * W32_LAYER;
        const float* w = layer_w(l);
        const int rows = n_out(l), cols = n_in(l);
        if (cols % 4 != 0 || (uintptr_t)w % 16 != 0) {
          read_layer32(w, rows, cols, tid, [&](int o, int c, f32x4_t x) { *reinterpret_cast<f32x4_t*>(dst + o * W32_STRIDE + c) = x; });
          continue;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          if (16 * i >= rows) break;
          const int o = (tid >> 4) + 16 * i, c = 4 * (tid & 15);
          *reinterpret_cast<f32x4_t*>(dst + o * W32_STRIDE + c) = o < rows && c < cols ? v[k][i] : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      if (wave < LAYERS && bl < a.n_layers) lds32[bl * W32_LAYER + 64 * W32_STRIDE + lane] = has_bias ? bias : 0.0f;
    }
    __syncthreads();
  } else if (PIECES) {
    load_rows(first_chunk);
  }
  for (int64_t done = 0; first_of_workgroup + done < n_chunks; done += per_round) {  // (the same for the workgroup)
    const int64_t chunk = first_chunk + done;
    if (a.resident && chunk >= n_chunks) break;
    const int64_t row0 = chunk * (16 * NT) + r;
    f32x4_t h[NT][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (PIECES) {
          if (t >= kt_in) break;
          h[nt][t] = 16 * t + 4 * g >= a.d_in ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : nx[nt][t];
        } else {
          h[nt][t] = t < kt_in ? load_chain(a.x, a.x_stride, row0 + 16 * nt, a.rows, 16 * t + 4 * g, a.d_in, x_vec) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
    if (PIECES) load_rows(chunk + per_round);
    for (int l = 0; l < a.n_layers; ++l) {
      const float* wl = lds32;
      if (a.resident) {
        wl = lds32 + l * W32_LAYER;
      } else {
        __syncthreads();  // every wave is done with the layer before
        stage_layer32(lds32, layer_w(l), layer_b(l), n_out(l), n_in(l), tid);
        __syncthreads();
      }
      const int kt = (n_in(l) + 15) / 16, mt_n = (n_out(l) + 15) / 16;
      f32x4_t acc[NT][4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const f32x4_t b4 = *reinterpret_cast<const f32x4_t*>(wl + 64 * W32_STRIDE + 16 * mt + 4 * g);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = b4;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= kt) break;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          if (mt >= mt_n) break;
          const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(wl + (16 * mt + r) * W32_STRIDE + 16 * t + 4 * g);
#pragma unroll
          for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = mfma4(w4[v], h[nt][t][v], acc[nt][mt]);
        }
      }
      if (l == last) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < 4; ++mt)
            if (mt < mt_n) {
              const int64_t row = row0 + 16 * nt;
              const int col = 16 * mt + 4 * g;
              if constexpr (!PIECES) store_chain(a.y, a.y_stride, row, a.rows, col, a.d_out, y_vec, acc[nt][mt]);
              else if (row < a.rows && col < a.d_out) *reinterpret_cast<f32x4_t*>(a.y + row * a.y_stride + col) = acc[nt][mt];
            }
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) {
            if (a.z != nullptr && mt < mt_n)
              store_chain(a.z + (size_t)l * a.rows * H, H, row0 + 16 * nt, a.rows, 16 * mt + 4 * g, H, true, acc[nt][mt]);
#pragma unroll
            for (int v = 0; v < 4; ++v) h[nt][mt][v] = mt < mt_n ? act_fwd(acc[nt][mt][v], ACT) : 0.0f;
          }
      }
    }
  }
}

struct Lin32BwdArgs {
  const float* dz;  // gradient at this layer's output (before the activation behind it), rows x n_out
  int64_t dz_stride;
  const float* src;  // this layer's input before its activation (rows x n_in): the layer in front's pre-activation, or x
  int64_t src_stride;
  float* dsrc;  // gradient at src (may be src itself, may be NULL)
  int64_t dsrc_stride;
  const float* w;  // n_out x n_in
  float* part;  // [gridDim.x][PART32] partial dW (row stride 64) and db of every workgroup
  int64_t rows;
  int n_out, n_in;
};

// One linear layer of the backward: partial dW = dz^T act(src), partial db = column sums of dz,
// dsrc = (dz W) * act'(src).
template <int ACT>
__global__ __launch_bounds__(256) void lin32_bwd_k(Lin32BwdArgs a) {
  extern __shared__ float lds32[];
  float* wt = lds32;  // wt[in][out], W32_STRIDE floats per row
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  float* pdz = lds32 + 64 * W32_STRIDE + wave * (2 * 16 * T32_STRIDE);  // this wave's dz rows
  float* ph = pdz + 16 * T32_STRIDE;                                    // this wave's act(src) rows
  read_layer32(a.w, a.n_out, a.n_in, tid, [&](int o, int c, f32x4_t v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) wt[(c + e) * W32_STRIDE + o] = v[e];
  });
  __syncthreads();
  const int mt_n = (a.n_out + 15) / 16, kt = (a.n_in + 15) / 16;
  const bool dz_vec = ((uintptr_t)a.dz % 16 == 0) && (a.dz_stride % 4 == 0);
  const bool src_vec = ((uintptr_t)a.src % 16 == 0) && (a.src_stride % 4 == 0);
  const bool dsrc_vec = a.dsrc != nullptr && ((uintptr_t)a.dsrc % 16 == 0) && (a.dsrc_stride % 4 == 0);
  f32x4_t dw[4][4];
  f32x4_t dbs[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    dbs[mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) dw[mt][nt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const int64_t n_groups = (a.rows + 15) / 16;
  // the rows of the group after this one are asked for before this one's products (dsrc may be src itself: a group's
  // rows are read here before they are written, and no other wave touches them)
  auto load_group = [&](int64_t grp, f32x4_t (&dz)[4], f32x4_t (&z)[4]) {
    const int64_t row = grp * 16 + r;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      dz[t] = t < mt_n ? load_chain(a.dz, a.dz_stride, row, a.rows, 16 * t + 4 * g, a.n_out, dz_vec) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      z[t] = t < kt ? load_chain(a.src, a.src_stride, row, a.rows, 16 * t + 4 * g, a.n_in, src_vec) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  const int64_t step = (int64_t)gridDim.x * 4;
  int64_t grp = (int64_t)blockIdx.x * 4 + wave;
  f32x4_t dz_next[4], z_next[4];
  if (grp < n_groups) load_group(grp, dz_next, z_next);
  for (; grp < n_groups; grp += step) {
    const int64_t row = grp * 16 + r;
    f32x4_t dz[4], z[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      dz[t] = dz_next[t];
      z[t] = z_next[t];
    }
    if (grp + step < n_groups) load_group(grp + step, dz_next, z_next);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      dbs[t] += dz[t];
      f32x4_t hv;
#pragma unroll
      for (int v = 0; v < 4; ++v) hv[v] = act_fwd(z[t][v], ACT);
      *reinterpret_cast<f32x4_t*>(pdz + r * T32_STRIDE + 16 * t + 4 * g) = dz[t];
      *reinterpret_cast<f32x4_t*>(ph + r * T32_STRIDE + 16 * t + 4 * g) = hv;
    }
    if (a.dsrc != nullptr) {
      // dsrc^T = W^T dz^T: rows of wt (input features) against the upstream gradient in chain order
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        if (nt >= kt) break;
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (t >= mt_n) break;
          const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(wt + (16 * nt + r) * W32_STRIDE + 16 * t + 4 * g);
#pragma unroll
          for (int v = 0; v < 4; ++v) acc = mfma4(w4[v], dz[t][v], acc);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] *= act_grad(z[nt][v], ACT);
        store_chain(a.dsrc, a.dsrc_stride, row, a.rows, 16 * nt + 4 * g, a.n_in, dsrc_vec, acc);
      }
    }
    // dW += dz^T h over this group's 16 rows, four rows per product; lane (i, k) reads row 4*s + k, column 16*tile + i
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float bh[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) bh[nt] = nt < kt ? ph[(4 * s + g) * T32_STRIDE + 16 * nt + r] : 0.0f;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        if (mt >= mt_n) break;
        const float av = pdz[(4 * s + g) * T32_STRIDE + 16 * mt + r];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
          if (nt < kt) dw[mt][nt] = mfma4(av, bh[nt], dw[mt][nt]);
      }
    }
  }
  // the workgroup's four partial sums, added in wave order (the same result on every run), then one store
  __syncthreads();
  float* red = lds32;
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            float* p = red + (16 * mt + 4 * g + v) * 64 + 16 * nt + r;
            *p = w == 0 ? dw[mt][nt][v] : *p + dw[mt][nt][v];
          }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float sum = dbs[mt][v];
          sum += __shfl_xor(sum, 1);
          sum += __shfl_xor(sum, 2);
          sum += __shfl_xor(sum, 4);
          sum += __shfl_xor(sum, 8);
          float* p = red + 64 * 64 + 16 * mt + 4 * g + v;
          if (r == 0) *p = w == 0 ? sum : *p + sum;
        }
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < PART32; i += 256) a.part[(size_t)blockIdx.x * PART32 + i] = red[i];
}

// dw += sum of the partial dW, db += sum of the partial db; blockIdx.y takes a share of the partials.
__global__ __launch_bounds__(256) void reduce32_k(const float* part, int n_slots, float* dw, float* db, int n_out, int n_in) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= PART32) return;
  const int per = (n_slots + gridDim.y - 1) / gridDim.y;
  const int s0 = blockIdx.y * per, s1 = min(n_slots, s0 + per);
  float sum = 0.0f;
  for (int sl = s0; sl < s1; ++sl) sum += part[(size_t)sl * PART32 + i];
  if (s0 >= s1) return;
  if (i < 64 * 64) {
    const int o = i >> 6, c = i & 63;
    if (o < n_out && c < n_in) unsafeAtomicAdd(dw + (size_t)o * n_in + c, sum);
  } else if (db != nullptr && i - 64 * 64 < n_out) {
    unsafeAtomicAdd(db + (i - 64 * 64), sum);
  }
}

// ---------------------------------------------------------------------------------------
// Backward of one or two hidden layers in one launch
// ---------------------------------------------------------------------------------------
// A wave takes sixteen rows through the hidden layers and back with everything in registers; the weights stay in LDS, as they are for the
// way forth and transposed for the way back, and nothing but x, dy and dx passes through memory (layer by layer with the
// pre-activations in memory, 100003 rows of 32-64-64-16: 160 us, so 63).  A product's operand with the rows along K comes from a panel
// of the wave's own in LDS.  All weights and the first rows are under way together, and the waves' sums meet in two turns (32-64-64-16, one
// matrix and one wave after the other: 16 rows 22.7 -> 17.7 us, 100003 rows 63.3 -> 58.8).  TI, TO: 16-column tiles of the input and the output; the hidden layers have four,
// narrower ones zeros.
constexpr int fused32_tiles(int TI, int TO, int DEPTH) { return TO * 4 + (DEPTH - 1) * 16 + 4 * TI; }
constexpr int fused32_waves(int TI, int TO, int DEPTH) { return fused32_tiles(TI, TO, DEPTH) <= 28 ? 8 : 4; }  // more gradients take the registers of two waves
constexpr int fused32_sums(int TI, int TO, int DEPTH) { return fused32_tiles(TI, TO, DEPTH) * 256 + 3 * 64; }
constexpr int fused32_stride(int tiles) { return 16 * tiles + 4; }  // floats per staged row of so many tiles
constexpr size_t fused32_lds(int TI, int TO, int DEPTH) {
  const int weights = 64 * fused32_stride(TI) + 16 * TI * W32_STRIDE + (DEPTH - 1) * 2 * 64 * W32_STRIDE + 64 * fused32_stride(TO) + 128;
  const int all = weights + fused32_waves(TI, TO, DEPTH) * 2 * 16 * T32_STRIDE, sums = fused32_waves(TI, TO, DEPTH) / 2 * fused32_sums(TI, TO, DEPTH);
  return (size_t)(all > sums ? all : sums) * sizeof(float);
}

struct Fused32Args {
  const float *x, *dy;
  float* dx;
  int64_t x_stride, dy_stride, dx_stride, rows;
  const float *w_in, *b_in, *w_hid, *b_hid, *w_out;
  float* slots;  // [workgroup][fused32_sums()]
  int d_in, d_hidden, d_out, act;
};

// acc += W h, W's rows of S floats in LDS; the products into one tile are `MT` instructions apart
template <int KT, int MT, int S>
__device__ __forceinline__ void product32(f32x4_t (&acc)[4], const float* w, const f32x4_t (&h)[4], int r, int g) {
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    f32x4_t w4[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) w4[mt] = *reinterpret_cast<const f32x4_t*>(w + (16 * mt + r) * S + 16 * t + 4 * g);
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma4(w4[mt][v], h[t][v], acc[mt]);
  }
}

template <int TI, int TO, int DEPTH>
__global__ __launch_bounds__(64 * fused32_waves(TI, TO, DEPTH)) void mlp32_bwd_k(Fused32Args a) {
  constexpr int WAVES = fused32_waves(TI, TO, DEPTH), THREADS = 64 * WAVES, SI = fused32_stride(TI), SH = W32_STRIDE, SO = fused32_stride(TO);
  constexpr bool DEEP = DEPTH == 2;
  extern __shared__ __align__(16) float lds32[];
  float* w1 = lds32;               // [hidden][in]
  float* w1t = w1 + 64 * SI;       // [in][hidden]
  float* wot = w1t + 16 * TI * SH;  // [hidden][out]
  float* w2 = wot + 64 * SO;       // [hidden][hidden]
  float* w2t = w2 + (DEEP ? 64 * SH : 0);
  float* bias = w2t + (DEEP ? 64 * SH : 0);  // two layers of 64
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4, H = a.d_hidden;
  float* pdz = bias + 128 + wave * (2 * 16 * T32_STRIDE);  // this wave's rows of a gradient,
  float* ph = pdz + 16 * T32_STRIDE;                       // and of the input of that layer
  const bool x_vec = ((uintptr_t)a.x % 16 == 0) && (a.x_stride % 4 == 0);
  const bool dy_vec = ((uintptr_t)a.dy % 16 == 0) && (a.dy_stride % 4 == 0);
  const bool dx_vec = a.dx != nullptr && ((uintptr_t)a.dx % 16 == 0) && (a.dx_stride % 4 == 0);
  const int64_t n_groups = (a.rows + 15) / 16, step = (int64_t)gridDim.x * WAVES;
  f32x4_t x_next[4];
  auto load_group = [&](int64_t grp) {
    const int64_t row = grp * 16 + r < a.rows ? grp * 16 + r : a.rows - 1;  // past the end the last row again, not zeros: see load_rows_frag()
#pragma unroll
    for (int t = 0; t < TI; ++t) x_next[t] = load_chain(a.x, a.x_stride, row, a.rows, 16 * t + 4 * g, a.d_in, x_vec);
  };
  // groups to the workgroups in turn, then to their waves: every unit has as many
  int64_t grp = (int64_t)wave * gridDim.x + blockIdx.x;
  Layer32<THREADS> m_in, m_hid, m_out;
  m_in.fetch(a.w_in, H, a.d_in, tid);
  if constexpr (DEEP) m_hid.fetch(a.w_hid, H, H, tid);
  m_out.fetch(a.w_out, a.d_out, H, tid);
  if (grp < n_groups) load_group(grp);
  m_in.spread(tid, [&](int o, int c, f32x4_t v) {
    if (c >= 16 * TI) return;
    *reinterpret_cast<f32x4_t*>(w1 + o * SI + c) = v;
#pragma unroll
    for (int e = 0; e < 4; ++e) w1t[(c + e) * SH + o] = v[e];
  });
  if constexpr (DEEP)
    m_hid.spread(tid, [&](int o, int c, f32x4_t v) {
      *reinterpret_cast<f32x4_t*>(w2 + o * SH + c) = v;
#pragma unroll
      for (int e = 0; e < 4; ++e) w2t[(c + e) * SH + o] = v[e];
    });
  m_out.spread(tid, [&](int o, int c, f32x4_t v) {
    if (o < 16 * TO)
#pragma unroll
      for (int e = 0; e < 4; ++e) wot[(c + e) * SO + o] = v[e];
  });
  if (tid < 64) {
    bias[tid] = a.b_in != nullptr && tid < H ? a.b_in[tid] : 0.0f;
    bias[64 + tid] = DEEP && a.b_hid != nullptr && tid < H ? a.b_hid[tid] : 0.0f;
  }
  __syncthreads();
  const f32x4_t zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4_t dw1[4][TI], dw2[4][DEEP ? 4 : 1], dwo[TO][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < TI; ++j) dw1[i][j] = zero4;
#pragma unroll
    for (int j = 0; j < (DEEP ? 4 : 1); ++j) dw2[i][j] = zero4;
#pragma unroll
    for (int j = 0; j < TO; ++j) dwo[j][i] = zero4;
  }
  float db1 = 0.0f, db2 = 0.0f, dbo = 0.0f;  // of feature `lane`
  auto put_panel = [&](float* panel, const f32x4_t (&v)[4], int n) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (t < n) *reinterpret_cast<f32x4_t*>(panel + r * T32_STRIDE + 16 * t + 4 * g) = v[t];
  };
  auto activated = [&](const f32x4_t (&z)[4], f32x4_t (&h)[4]) {
    with_act(a.act, [&](auto act_c) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) h[t][v] = act_fwd(z[t][v], decltype(act_c)::value);
    });
  };
  auto gated = [&](f32x4_t (&d)[4], const f32x4_t (&z)[4]) {
    with_act(a.act, [&](auto act_c) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) d[t][v] *= act_grad(z[t][v], decltype(act_c)::value);
    });
  };
  // dW += dz^T h over the sixteen rows of the panels, four rows per product; lane (i, k) reads row 4*s + k, column 16*tile + i
  auto gradient = [&](auto& dw, auto mt_c, auto nt_c) {
    constexpr int MT = decltype(mt_c)::value, NT = decltype(nt_c)::value;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float av[MT], bh[NT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) av[mt] = pdz[(4 * s + g) * T32_STRIDE + 16 * mt + r];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) bh[nt] = ph[(4 * s + g) * T32_STRIDE + 16 * nt + r];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) dw[mt][nt] = mfma4(av[mt], bh[nt], dw[mt][nt]);
    }
  };
  auto column_sum = [&](int width) {
    float sum = 0.0f;
    if (lane < width)
#pragma unroll
      for (int k = 0; k < 16; ++k) sum += pdz[k * T32_STRIDE + lane];
    return sum;
  };
  for (; grp < n_groups; grp += step) {
    const int64_t row = grp * 16 + r;
    f32x4_t x[4], d[4], z1[4], z2[4], h[4], acc[4];
#pragma unroll
    for (int t = 0; t < TI; ++t) x[t] = x_next[t];
#pragma unroll
    for (int t = 0; t < TO; ++t) d[t] = load_chain(a.dy, a.dy_stride, row, a.rows, 16 * t + 4 * g, a.d_out, dy_vec);  // used after the way forth
    if (grp + step < n_groups) load_group(grp + step);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) z1[mt] = *reinterpret_cast<const f32x4_t*>(bias + 16 * mt + 4 * g);
    product32<TI, 4, SI>(z1, w1, x, r, g);
    activated(z1, h);
    if constexpr (DEEP) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) z2[mt] = *reinterpret_cast<const f32x4_t*>(bias + 64 + 16 * mt + 4 * g);
      product32<4, 4, SH>(z2, w2, h, r, g);
      activated(z2, h);
    }
    // output layer
    put_panel(pdz, d, TO);
    put_panel(ph, h, 4);
    dbo += column_sum(16 * TO);
    gradient(dwo, std::integral_constant<int, TO>{}, std::integral_constant<int, 4>{});
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = zero4;
    product32<TO, 4, SO>(acc, wot, d, r, g);
    if constexpr (DEEP) {
      gated(acc, z2);
      activated(z1, h);
      put_panel(pdz, acc, 4);
      put_panel(ph, h, 4);
      db2 += column_sum(64);
      gradient(dw2, std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] = zero4;
      product32<4, 4, SH>(d, w2t, acc, r, g);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] = acc[t];
    }
    gated(d, z1);
    put_panel(pdz, d, 4);
    put_panel(ph, x, TI);
    db1 += column_sum(64);
    gradient(dw1, std::integral_constant<int, 4>{}, std::integral_constant<int, TI>{});
    if (a.dx != nullptr) {
#pragma unroll
      for (int t = 0; t < TI; ++t) acc[t] = zero4;
      product32<4, TI, SH>(acc, w1t, d, r, g);
#pragma unroll
      for (int t = 0; t < TI; ++t) store_chain(a.dx, a.dx_stride, row, a.rows, 16 * t + 4 * g, a.d_in, dx_vec, acc[t]);
    }
  }
  // The waves' sums to the workgroup's slot, in a fixed order (the same result on every run): the upper half of the waves lay theirs down, the
  // lower half add theirs, then all threads add the areas.  (A wave after the other took eight turns.)
  constexpr int SUMS = fused32_sums(TI, TO, DEPTH), AREAS = WAVES / 2;
  for (int turn = 1; turn >= 0; --turn) {
    __syncthreads();
    if (wave / AREAS != turn) continue;
    float* area = lds32 + (wave % AREAS) * SUMS;
    f32x4_t* red = reinterpret_cast<f32x4_t*>(area) + lane;
    float* redb = area + fused32_tiles(TI, TO, DEPTH) * 256 + lane;
    int at = 0;
    auto add = [&](f32x4_t v) {
      red[64 * at] = turn == 1 ? v : red[64 * at] + v;
      ++at;
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < TI; ++j) add(dw1[i][j]);
    if constexpr (DEEP) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) add(dw2[i][j]);
    }
#pragma unroll
    for (int i = 0; i < TO; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) add(dwo[i][j]);
    redb[0] = turn == 1 ? db1 : redb[0] + db1;
    redb[64] = turn == 1 ? db2 : redb[64] + db2;
    redb[128] = turn == 1 ? dbo : redb[128] + dbo;
  }
  __syncthreads();
  f32x4_t* slot = reinterpret_cast<f32x4_t*>(a.slots + (size_t)blockIdx.x * SUMS);
  for (int i = tid; i < SUMS / 4; i += THREADS) {
    f32x4_t sum = reinterpret_cast<const f32x4_t*>(lds32)[i];
#pragma unroll
    for (int k = 1; k < AREAS; ++k) sum += reinterpret_cast<const f32x4_t*>(lds32 + k * SUMS)[i];
    slot[i] = sum;
  }
}

// The slots of the workgroups in a fixed order into the caller's accumulators: sixteen interleaved runs, then a fixed tree.
struct Fused32Sums {
  float *dw_in, *db_in, *dw_hid, *db_hid, *dw_out, *db_out;
  int ti, to, depth, d_in, d_hidden, d_out, n_slots, sums;
  int write;  // the sums replace what is there instead of being added to it
};
__global__ __launch_bounds__(1024) void mlp32_sum_k(const float* slots, Fused32Sums o) {
  __shared__ float part[16][64];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6, i = blockIdx.x * 64 + tx;
  float sum = 0.0f;
  if (i < o.sums) {
#pragma unroll 4
    for (int sl = ty; sl < o.n_slots; sl += 16) sum += slots[(size_t)sl * o.sums + i];
  }
  part[ty][tx] = sum;
  __syncthreads();
  if (ty != 0 || i >= o.sums) return;
  float total = 0.0f;
#pragma unroll
  for (int q = 0; q < 16; q += 4) total += (part[q][tx] + part[q + 1][tx]) + (part[q + 2][tx] + part[q + 3][tx]);
  const int hid = o.depth == 2 ? 16 : 0, tiles = 4 * o.ti + hid + 4 * o.to;
  if (i >= tiles * 256) {
    const int k = (i - tiles * 256) >> 6, f = i & 63;
    float* db = k == 0 ? o.db_in : k == 1 ? o.db_hid : o.db_out;
    if (db != nullptr && f < (k == 2 ? o.d_out : o.d_hidden) && (k != 1 || o.depth == 2)) db[f] = (o.write ? 0.0f : db[f]) + total;
    return;
  }
  int tile = i >> 8;
  float* dw = o.dw_in;
  int nt = o.ti, n_out = o.d_hidden, n_in = o.d_in;
  if (tile >= 4 * o.ti) {
    tile -= 4 * o.ti;
    nt = 4;
    n_in = o.d_hidden;
    dw = o.dw_hid;
    if (tile >= hid) {
      tile -= hid;
      dw = o.dw_out;
      n_out = o.d_out;
    }
  }
  const int ln = (i & 255) >> 2, row = 16 * (tile / nt) + 4 * (ln >> 4) + (i & 3), col = 16 * (tile % nt) + (ln & 15);
  if (row < n_out && col < n_in) {
    float* p = dw + (size_t)row * n_in + col;
    *p = (o.write ? 0.0f : *p) + total;
  }
}

template <typename Args>
static int launch32(const void* kern, const Args& a, int64_t blocks, size_t lds, hipStream_t s, const char* what, int threads = 256) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  void* args[] = {(void*)&a};
  const hipError_t le = hipLaunchKernel(kern, dim3((unsigned)blocks), dim3((unsigned)threads), args, lds, s);
  if (le != hipSuccess) return fail((int)le, "hipLaunchKernel(%s): %s", what, hipGetErrorString(le));
  return 0;
}

static int fwd32(Mlp32Args a, hipStream_t s) {
  a.n_layers = a.y != nullptr ? a.depth + 1 : a.depth;
  a.resident = a.n_layers <= W32_RESIDENT_MAX;
  const size_t lds = (size_t)(a.resident ? a.n_layers : 1) * W32_LAYER * sizeof(float);
  const int64_t cap = (int64_t)device_cus() * (lds > 76 * 1024 ? 1 : 2);
  // One group of sixteen rows to a wave where there is a wave for every group, or, with the layers in LDS, where a SIMD's share of groups is a tenth less than
  // that of pairs.  Layers that pass through LDS are staged once more for every round of chunks, and half as many rows to a round are up to twice the rounds.
  // us, one / two: 32 -> 64 -> 64 -> 16, 4096 rows 7.6 / 10.4, 40000 13.0 / 15.3, 100003 22.9 / 25.3, 2^18 47.0 / 45.5; 64 -> 64 -> 64 -> 64, 2^20 259 / 249;
  // 32 -> 64 x 6 -> 16 (a workgroup to a unit), 16384 rows 16.1 / 23.9, 20000 26.0 / 24.2; 32 -> 64 x 9 -> 16 (in turn), 2^15 31.4 / 37.8, 36000 53.3 / 51.0, 100003 110 / 98.7.
  const int64_t simds = (int64_t)device_cus() * 4, ones = (a.rows + 15) / 16, twos = (a.rows + 31) / 32;
  const auto share = [&](int64_t units) { return (units + simds - 1) / simds; };
  const bool single = ones <= 4 * cap || (a.resident && 10 * share(ones) < 9 * 2 * share(twos));
  const int64_t chunks = single ? ones : twos, full = (chunks + 3) / 4;
  int64_t blocks = full < cap ? full : cap;
  if (blocks < device_cus()) blocks = chunks < device_cus() ? chunks : device_cus();
  // The chunks of a batch that leaves waves without one go to the workgroups in turn, then to their waves; of a larger one, four at a time to a workgroup:
  // what the last round has left is then a chunk for every SIMD of some units.  A wave of every workgroup came down on one SIMD of every unit, and
  // where the layers do not stay in LDS all workgroups went through that round (us, so / this: 32 -> 64 x 3 -> 16, 88000 rows 34.9 / 28.2; 64 x 11, 216000 256 / 236).
  const bool spread = chunks <= 4 * blocks - 4;
  a.block_step = spread ? 1 : 4;
  a.wave_step = spread ? (int)blocks : 1;
  const auto pieces = [](const float* p, int64_t stride, int width) { return (uintptr_t)p % 16 == 0 && stride % 4 == 0 && width % 4 == 0; };
  const bool whole = pieces(a.x, a.x_stride, a.d_in) && (a.y == nullptr || pieces(a.y, a.y_stride, a.d_out));
  auto pick = [&](auto nt_c, auto whole_c) -> const void* {
    constexpr int NT = decltype(nt_c)::value;
    constexpr bool PIECES = decltype(whole_c)::value;
    switch (a.act) {
      case NF_ACT_RELU: return (const void*)mlp32_fwd_k<NF_ACT_RELU, NT, PIECES>;
      case NF_ACT_SILU: return (const void*)mlp32_fwd_k<NF_ACT_SILU, NT, PIECES>;
      case NF_ACT_RELU2: return (const void*)mlp32_fwd_k<NF_ACT_RELU2, NT, PIECES>;
      case NF_ACT_GELU: return (const void*)mlp32_fwd_k<NF_ACT_GELU, NT, PIECES>;
      default: return (const void*)mlp32_fwd_k<NF_ACT_NONE, NT, PIECES>;
    }
  };
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 2> two;
  // Pairs of groups in whole pieces for ReLU alone: with the next rows in its registers, the kernel of another activation has 186 of them and is slower than
  // with rows read value by value where they are needed (135), the more so the narrower the network (50200 rows, us, pieces / values: 32 -> 16 -> 16
  // ReLU2 8.4 / 6.7, 32 -> 64 x 3 -> 4 SiLU 23.0 / 21.4, 64 -> 64 -> 64 ReLU2 18.3 / 16.0; ReLU, 149 registers value by value: 16 -> 32 -> 4 7.1 / 7.8, 32 -> 64 x 3 -> 4 20.3 / 20.5).
  const void* kern = single ? (whole ? pick(one, std::true_type{}) : pick(one, std::false_type{}))
                     : whole && a.act == NF_ACT_RELU ? (const void*)mlp32_fwd_k<NF_ACT_RELU, 2, true>
                                                     : pick(two, std::false_type{});
  return launch32(kern, a, blocks, lds, s, "mlp32_fwd");
}

static int lin_bwd32(const Lin32BwdArgs& a, int act, float* dw, float* db, hipStream_t s) {
  const size_t lds = (size_t)(64 * W32_STRIDE + 4 * 2 * 16 * T32_STRIDE) * sizeof(float);
  const int64_t groups = (a.rows + 15) / 16;
  const int64_t want = (groups + 3) / 4;
  int64_t cap = (int64_t)device_cus() * 2;
  if (cap > SLOTS32) cap = SLOTS32;
  const int64_t blocks = want < cap ? want : cap;
  const void* kern = nullptr;
  switch (act) {
    case NF_ACT_RELU: kern = (const void*)lin32_bwd_k<NF_ACT_RELU>; break;
    case NF_ACT_SILU: kern = (const void*)lin32_bwd_k<NF_ACT_SILU>; break;
    case NF_ACT_RELU2: kern = (const void*)lin32_bwd_k<NF_ACT_RELU2>; break;
    case NF_ACT_GELU: kern = (const void*)lin32_bwd_k<NF_ACT_GELU>; break;
    default: kern = (const void*)lin32_bwd_k<NF_ACT_NONE>; break;
  }
  if (int rc = launch32(kern, a, blocks, lds, s, "lin32_bwd")) return rc;
  const float* part = a.part;
  int n_slots = (int)blocks, n_out = a.n_out, n_in = a.n_in;
  void* args[] = {(void*)&part, (void*)&n_slots, (void*)&dw, (void*)&db, (void*)&n_out, (void*)&n_in};
  const hipError_t le = hipLaunchKernel((const void*)reduce32_k, dim3((PART32 + 255) / 256, 32), dim3(256), args, 0, s);
  if (le != hipSuccess) return fail((int)le, "hipLaunchKernel(reduce32): %s", hipGetErrorString(le));
  return 0;
}

static size_t z32_bytes(int64_t rows, int d_hidden, int depth) {
  return ((size_t)depth * (size_t)rows * d_hidden * sizeof(float) + 255) / 256 * 256;
}

template <int TI, int TO, int DEPTH>
static int bwd32_fused(const Fused32Args& a, Fused32Sums o, size_t slot_bytes, hipStream_t s) {
  const int64_t groups = (a.rows + 15) / 16, slots = (int64_t)(slot_bytes / (fused32_sums(TI, TO, DEPTH) * sizeof(float)));
  int64_t blocks = groups < device_cus() ? groups : device_cus();
  if (blocks > slots) blocks = slots;  // (few rows of a wide network: the workspace is the layered kernels')
  if (int rc = launch32((const void*)mlp32_bwd_k<TI, TO, DEPTH>, a, blocks, fused32_lds(TI, TO, DEPTH), s, "mlp32_bwd", 64 * fused32_waves(TI, TO, DEPTH))) return rc;
  o.ti = TI;
  o.to = TO;
  o.depth = DEPTH;
  o.n_slots = (int)blocks;
  o.sums = fused32_sums(TI, TO, DEPTH);
  const float* sums = a.slots;
  void* args[] = {(void*)&sums, (void*)&o};
  const hipError_t le = hipLaunchKernel((const void*)mlp32_sum_k, dim3((unsigned)((o.sums + 63) / 64)), dim3(1024), args, 0, s);
  if (le != hipSuccess) return fail((int)le, "hipLaunchKernel(mlp32_sum): %s", hipGetErrorString(le));
  return 0;
}


size_t mlp32_bwd_workspace_bytes(int64_t rows, int d_hidden, int depth) {
  return z32_bytes(rows, d_hidden, depth) + (size_t)SLOTS32 * PART32 * sizeof(float);
}

int mlp32_fwd(const float* x, int64_t x_stride, float* y, int64_t y_stride, const float* w_in, const float* b_in,
              const float* w_hid, const float* b_hid, const float* w_out, const float* b_out, int64_t rows, int d_in,
              int d_hidden, int d_out, int depth, int act, hipStream_t s) {
  Mlp32Args a = {};
  a.x = x; a.x_stride = x_stride; a.y = y; a.y_stride = y_stride;
  a.w_in = w_in; a.b_in = b_in; a.w_hid = w_hid; a.b_hid = b_hid; a.w_out = w_out; a.b_out = b_out;
  a.rows = rows; a.d_in = d_in; a.d_hidden = d_hidden; a.d_out = d_out; a.depth = depth; a.act = act;
  return fwd32(a, s);
}

int mlp32_bwd(const float* x, int64_t x_stride, const float* dy, int64_t dy_stride, float* dx, int64_t dx_stride,
              const float* w_in, const float* b_in, const float* w_hid, const float* b_hid, const float* w_out, float* dw_in,
              float* db_in, float* dw_hid, float* db_hid, float* dw_out, float* db_out, int64_t rows, int d_in, int d_hidden,
              int d_out, int depth, int act, bool write, void* workspace, int64_t workspace_bytes, hipStream_t s) {
  NF_REQUIRE(!write || depth <= 2, NF_EUNSUPPORTED, "float32 gradients are written for one and two hidden layers (depth=%d)", depth);
  const size_t need = mlp32_bwd_workspace_bytes(rows, d_hidden, depth);
  NF_REQUIRE(workspace != nullptr && workspace_bytes >= (int64_t)need, NF_EINVAL,
             "float32 backward keeps %d pre-activations of %lld x %d float32 and partial weight gradients: it needs a "
             "workspace of %zu bytes (nf_mlp_workspace_bytes)", depth, (long long)rows, d_hidden, need);
  NF_REQUIRE((uintptr_t)workspace % 16 == 0, NF_EINVAL, "workspace must be 16-byte aligned");
  if (depth <= 2) {
    Fused32Args a = {x, dy, dx, x_stride, dy_stride, dx_stride, rows, w_in, b_in, w_hid, b_hid, w_out, (float*)workspace, d_in, d_hidden, d_out, act};
    Fused32Sums o = {dw_in, db_in, dw_hid, db_hid, dw_out, db_out, 0, 0, 0, d_in, d_hidden, d_out, 0, 0, write};
    const bool narrow = d_in <= 32, small = d_out <= 16;
    if (depth == 2)
      return narrow ? (small ? bwd32_fused<2, 1, 2>(a, o, need, s) : bwd32_fused<2, 4, 2>(a, o, need, s))
                    : (small ? bwd32_fused<4, 1, 2>(a, o, need, s) : bwd32_fused<4, 4, 2>(a, o, need, s));
    return narrow ? (small ? bwd32_fused<2, 1, 1>(a, o, need, s) : bwd32_fused<2, 4, 1>(a, o, need, s))
                  : (small ? bwd32_fused<4, 1, 1>(a, o, need, s) : bwd32_fused<4, 4, 1>(a, o, need, s));
  }
  float* z = (float*)workspace;
  float* part = (float*)((char*)workspace + z32_bytes(rows, d_hidden, depth));
  const int H = d_hidden;
  Mlp32Args f = {};
  f.x = x; f.x_stride = x_stride; f.y = nullptr; f.y_stride = 0;
  f.w_in = w_in; f.b_in = b_in; f.w_hid = w_hid; f.b_hid = b_hid; f.w_out = w_out; f.b_out = nullptr;
  f.z = z;
  f.rows = rows; f.d_in = d_in; f.d_hidden = H; f.d_out = d_out; f.depth = depth; f.act = act;
  if (int rc = fwd32(f, s)) return rc;
  auto zl = [&](int l) { return z + (size_t)l * rows * H; };  // pre-activation of linear layer l, l < depth
  for (int l = depth; l >= 0; --l) {
    Lin32BwdArgs b = {};
    b.dz = l == depth ? dy : zl(l);
    b.dz_stride = l == depth ? dy_stride : H;
    b.src = l == 0 ? x : zl(l - 1);
    b.src_stride = l == 0 ? x_stride : H;
    b.dsrc = l == 0 ? dx : zl(l - 1);
    b.dsrc_stride = l == 0 ? dx_stride : H;
    b.w = l == 0 ? w_in : l == depth ? w_out : w_hid + (size_t)(l - 1) * H * H;
    float* dw = l == 0 ? dw_in : l == depth ? dw_out : dw_hid + (size_t)(l - 1) * H * H;
    float* db = l == 0 ? db_in : l == depth ? db_out : (db_hid ? db_hid + (size_t)(l - 1) * H : nullptr);
    b.part = part;
    b.rows = rows;
    b.n_out = l == depth ? d_out : H;
    b.n_in = l == 0 ? d_in : H;
    if (int rc = lin_bwd32(b, l == 0 ? NF_ACT_NONE : act, dw, db, s)) return rc;
  }
  return 0;
}

}  // namespace nf
