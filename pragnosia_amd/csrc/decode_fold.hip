// The weights of the batched decode step's dense layers as decode_gemm.hip reads them, from the model's parameters:
// the layer's row blocks (up to five tensors of K columns, stacked) tiled as
//     Wt[((t KS + s) 64 + l) 4 + e] = W'[16 t + l % 16][16 s + 4 (l / 16) + e]
// (column tile t of 16 rows, 16-wide step s of KS = K / 16, lane l; rows past N zero) with W' = W diag(col_scale): a
// LayerNorm's weight (K) or a per-head RMSNorm's (G, repeated), and for a folded LayerNorm the row sums of W' (csum)
// and bias + W ln_bias, both summed in fp64.
//
// A decoder folds its whole model at the start of every generation (the parameters may have changed), so this is a
// copy bound by memory, and by launches if each layer had its own: one launch takes a table of layers. One workgroup a
// column tile, wave w the steps w, w + 4, ...; a lane reads 16 bytes of its row (a 64-byte piece of each of 16 rows a
// load) and writes 16 of a contiguous KiB, and adds its row's sums on the way. 92M parameters (d 768, 12 layers, 49
// dense layers), host and device time: 2.8 ms as torch calls (concatenation, scaling, transposes, fp64 sums and
// products, then copies into the step's buffers), 1.05 ms as 49 launches, 0.46 ms as one.
#include "common.h"

namespace {

// One layer of the table (PRAGNOSIA_FOLD_ENTRIES int64)
struct Layer {
  const float* w[5];
  int64_t end[5];  // rows up to and including block b
  int64_t K;
  const float* cs;
  int64_t G;
  const float* lb;
  const float* bias;
  float* Wt;
  float* csum;
  float* bout;
  int64_t first;  // the layer's first workgroup
};
static_assert(sizeof(Layer) == PRAGNOSIA_FOLD_ENTRIES * sizeof(int64_t), "the header's entry count");

__global__ __launch_bounds__(256) void decode_fold(const Layer* __restrict__ table, int n) {
  __shared__ double red[4][2][16];
  int lo = 0, hi = n - 1;  // the last layer whose first workgroup is not past this one
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (table[mid].first <= (int64_t)blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const Layer& b = table[lo];
  const int64_t tile = blockIdx.x - b.first, N = b.end[4], K = b.K, G = b.G;
  const float *cs = b.cs, *lb = b.lb, *bias = b.bias;
  float *Wt = b.Wt, *csum = b.csum, *bout = b.bout;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, r = l & 15, g = l >> 4;
  const int64_t n_ = tile * 16 + r, KS = K / 16;
  const float* row = nullptr;
  int64_t first = 0;
#pragma unroll
  for (int u = 0; u < 5; ++u) {
    if (row == nullptr && n_ < b.end[u]) row = b.w[u] + (n_ - first) * K;
    first = b.end[u];
  }
  double s = 0., d = 0.;
  for (int64_t st = w; st < KS; st += 4) {
    const int64_t k = 16 * st + 4 * g;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y;
    if (row != nullptr) x = *reinterpret_cast<const f32x4*>(row + k);
    y = x;
    if (cs != nullptr) y *= *reinterpret_cast<const f32x4*>(cs + k % G);
    *reinterpret_cast<f32x4*>(Wt + ((tile * KS + st) * 64 + l) * 4) = y;
    if (csum != nullptr) s += ((double)y[0] + (double)y[1]) + ((double)y[2] + (double)y[3]);
    if (lb != nullptr) {
      const f32x4 z = *reinterpret_cast<const f32x4*>(lb + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) d += (double)x[e] * (double)z[e];
    }
  }
  if (csum == nullptr && bout == nullptr) return;
  s += __shfl_xor(s, 16);
  d += __shfl_xor(d, 16);
  s += __shfl_xor(s, 32);
  d += __shfl_xor(d, 32);
  if (g == 0) {
    red[w][0][r] = s;
    red[w][1][r] = d;
  }
  __syncthreads();
  if (threadIdx.x < 16 && n_ < N) {
    if (csum != nullptr) csum[n_] = (float)((red[0][0][r] + red[1][0][r]) + (red[2][0][r] + red[3][0][r]));
    if (bout != nullptr)
      bout[n_] = (float)((bias != nullptr ? (double)bias[n_] : 0.) +
                        ((red[0][1][r] + red[1][1][r]) + (red[2][1][r] + red[3][1][r])));
  }
}

}  // namespace

extern "C" int pragnosia_decode_fold(const int64_t* table, const int64_t* device_table, int64_t n, void* stream) {
  PGN_CHECK_ARG(table && device_table && n > 0 && n < (1 << 20) && ((uintptr_t)device_table & 7) == 0);
  const Layer* t = reinterpret_cast<const Layer*>(table);
  int64_t wgs = 0;
  for (int64_t i = 0; i < n; ++i) {
    const Layer& b = t[i];
    PGN_CHECK_ARG(b.K > 0 && b.K % 16 == 0 && b.K < ((int64_t)1 << 24) && b.Wt && ((uintptr_t)b.Wt & 15) == 0);
    PGN_CHECK_ARG(b.cs == nullptr || (b.G > 0 && b.G % 4 == 0 && b.K % b.G == 0 && ((uintptr_t)b.cs & 15) == 0));
    PGN_CHECK_ARG(((uintptr_t)b.lb & 15) == 0 && b.first == wgs);
    int64_t N = 0;
    for (int u = 0; u < 5; ++u) {
      PGN_CHECK_ARG(b.end[u] >= N && b.end[u] < ((int64_t)1 << 31));
      PGN_CHECK_ARG(b.end[u] == N || (b.w[u] && ((uintptr_t)b.w[u] & 15) == 0));
      N = b.end[u];
    }
    PGN_CHECK_ARG(N > 0);
    wgs += (N + 15) / 16;
  }
  PGN_CHECK_ARG(wgs < ((int64_t)1 << 31));
  hipLaunchKernelGGL(decode_fold, dim3((unsigned)wgs), dim3(256), 0, (hipStream_t)stream,
                     reinterpret_cast<const Layer*>(device_table), (int)n);
  PGN_RETURN_LAUNCH();
}
