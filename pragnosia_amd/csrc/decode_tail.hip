// The end of one greedy decode step, in one kernel: what the reference's graphed generate does between the head and
// the next step's first layer (`src/bench.py:241-317`: argmax of the logits, the token appended, the position advanced
// modulo the position table, the next input x = tok_emb[tok] + pos_emb[pos]), plus this build's per-step device state
// (the generated-token buffer and its row counter, the carried states' position offsets reset to 1).
//
// One workgroup of 1024 threads per sequence b:
//   tok = argmax_v logits[b][v] (the first index among equal maxima, NaN above every number: torch.argmax's rule),
//   out[c][b] = tok (c = *ctr_in, row c of the generated-token buffer, skipped past its n_rows), tok_out[b] = tok,
//   p = (*pos_in + 1) mod ctx, h[b] = emb[tok] + pemb[p] (fp32, one add per element as torch's),
//   recorded logits (optional): lrec[c][b] = logits[b];
// workgroup 0 also writes *pos_out = p, *ctr_out = c + 1 and p0s[0 .. L - 1] = 1. The counter and the position are
// read from one buffer and written to another (the caller alternates the pair from step to step), so no workgroup
// reads a value another has already advanced, and a captured graph of an even number of steps replays where the last
// replay ended.
//
// Bound by its serial chain: one round trip for the logits, the reduction, one for the token's embedding. The
// candidates are compared as unsigned keys (order_key) and reduced by lane moves in the vector unit, the waves' 16 keys
// by every wave for itself after one barrier. Through the LDS permute unit, with float comparisons and one thread
// walking the 16 candidates, the reduction took longer than both round trips. us a launch, before / now: 1 sequence of
// 8192 logits 7.9 / 3.7, 64 of them 8.3 / 4.2, 4 of 50257 19.0 / 9.8.
#include "common.h"

namespace {

// A logit as an unsigned number in torch.argmax's order: NaN (any) above every number, -0 equal to +0. Above 0 always.
PGN_DEVICE unsigned order_key(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  if (x != x) return 0xffffffffu;
  if (u == 0x80000000u) return 0x80000000u;  // -0 as +0
  return u >> 31 ? ~u : u | 0x80000000u;
}

// (order key, ~index) as one 64-bit number: the larger is the better logit, the smaller index among equals
struct Key {
  unsigned hi, lo;
};
PGN_DEVICE Key max_key(const Key& a, const Key& b) {
  return a.hi > b.hi || (a.hi == b.hi && a.lo > b.lo) ? a : b;
}
template <int CTRL>
PGN_DEVICE Key max_dpp(const Key& k) {
  return max_key(k, Key{(unsigned)__builtin_amdgcn_update_dpp(0, (int)k.hi, CTRL, 0xf, 0xf, true),
                        (unsigned)__builtin_amdgcn_update_dpp(0, (int)k.lo, CTRL, 0xf, 0xf, true)});
}
// Over each row of 16 lanes, in all of them (group_sum's exchanges)
PGN_DEVICE Key max_row(Key k) {
  k = max_dpp<0xB1>(k);    // quad_perm [1, 0, 3, 2]
  k = max_dpp<0x4E>(k);    // quad_perm [2, 3, 0, 1]
  k = max_dpp<0x141>(k);   // row_half_mirror
  return max_dpp<0x140>(k);  // row_mirror
}
// Over the wave's 64 lanes, in all of them: a swap of a register with itself leaves the two halves' values side by side
PGN_DEVICE Key max_wave(Key k) {
  k = max_row(k);
  {
    const auto h = __builtin_amdgcn_permlane16_swap(k.hi, k.hi, false, false);
    const auto l = __builtin_amdgcn_permlane16_swap(k.lo, k.lo, false, false);
    k = max_key(Key{h[0], l[0]}, Key{h[1], l[1]});
  }
  const auto h = __builtin_amdgcn_permlane32_swap(k.hi, k.hi, false, false);
  const auto l = __builtin_amdgcn_permlane32_swap(k.lo, k.lo, false, false);
  return max_key(Key{h[0], l[0]}, Key{h[1], l[1]});
}

constexpr int kTailThreads = 1024;
constexpr int kTailLoads = 8;  // logits a thread loads before it compares any: one memory round trip per 8192

__global__ __launch_bounds__(kTailThreads) void decode_tail(const float* __restrict__ logits, int V,
                                                            const float* __restrict__ emb,
                                                            const float* __restrict__ pemb, int d, int ctx,
                                                            const int64_t* __restrict__ ctr_in,
                                                            int64_t* __restrict__ ctr_out,
                                                            const int64_t* __restrict__ pos_in,
                                                            int64_t* __restrict__ pos_out, int64_t* __restrict__ out,
                                                            int64_t n_rows, int64_t* __restrict__ tok_out,
                                                            float* __restrict__ h, float* __restrict__ p0s, int L,
                                                            float* __restrict__ lrec, int B) {
  constexpr int NW = kTailThreads / 64;
  static_assert(NW == 16, "the waves' keys are reduced in a row of 16 lanes");
  __shared__ Key key_s[NW];
  const int b = blockIdx.x, tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  const float* row = logits + (size_t)b * V;
  const int64_t c = *ctr_in;
  const bool rec = lrec && c < n_rows;
  // the next position and its embedding entry do not depend on the argmax: loaded with the logits, so only the token
  // embedding's load follows the reduction
  const int64_t next = *pos_in + 1;
  const int p = (int)((uint64_t)next < (uint64_t)ctx ? next : next % ctx);  // the 64-bit division only at the wrap
  const float* pr = pemb + (size_t)p * d;
  const float pr0 = tid < d ? pr[tid] : 0.f;
  unsigned bk = 0u;
  int bi = -1;
  // kTailLoads logits a thread (v = v0 + tid + kTailThreads u), all loaded before any comparison, so a pass over
  // kTailThreads kTailLoads logits costs one memory round trip; each thread keeps the better of its values
  for (int v0 = 0; v0 < V; v0 += kTailThreads * kTailLoads) {
    float xs[kTailLoads];
#pragma unroll
    for (int u = 0; u < kTailLoads; ++u) {
      const int v = v0 + tid + kTailThreads * u;
      xs[u] = v < V ? row[v] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kTailLoads; ++u) {
      const int v = v0 + tid + kTailThreads * u;
      if (v < V) {
        const unsigned key = order_key(xs[u]);
        if (key > bk) {  // v ascends, so the first index among equals stays
          bk = key;
          bi = v;
        }
        if (rec) lrec[((size_t)c * B + b) * V + v] = xs[u];
      }
    }
  }
  const Key wk = max_wave(Key{bk, ~(unsigned)bi});
  if (l == 0) key_s[w] = wk;
  __syncthreads();
  const int t = (int)~(unsigned)__builtin_amdgcn_readfirstlane((int)max_row(key_s[l & 15]).lo);
  if (tid == 0) {
    tok_out[b] = t;
    if (c < n_rows) out[c * B + b] = t;
  }
  const float* er = emb + (size_t)t * d;
  float* hr = h + (size_t)b * d;
  if (tid < d) hr[tid] = er[tid] + pr0;
  for (int k = tid + kTailThreads; k < d; k += kTailThreads) hr[k] = er[k] + pr[k];
  if (b == 0) {
    if (tid == 0) {
      *pos_out = p;
      *ctr_out = c + 1;
    }
    for (int k = tid; k < L; k += kTailThreads) p0s[k] = 1.f;
  }
}

}  // namespace

extern "C" int pragnosia_decode_tail(const float* logits, int64_t B, int64_t V, const float* emb, const float* pemb,
                                     int64_t d, int64_t ctx, const int64_t* ctr_in, int64_t* ctr_out,
                                     const int64_t* pos_in, int64_t* pos_out, int64_t* out, int64_t n_rows,
                                     int64_t* tok, float* h, float* p0s, int64_t L, float* logits_rec, void* stream) {
  PGN_CHECK_ARG(logits && emb && pemb && ctr_in && ctr_out && pos_in && pos_out && out && tok && h);
  PGN_CHECK_ARG(B > 0 && V > 0 && d > 0 && ctx > 0 && n_rows > 0 && L >= 0 && (L == 0 || p0s));
  PGN_CHECK_ARG(B < (1 << 20) && V < ((int64_t)1 << 30) && d < (1 << 30) && ctx < (1 << 30) && L < (1 << 30));
  PGN_CHECK_ARG(B * V < ((int64_t)1 << 40) && n_rows * B * V < ((int64_t)1 << 62));
  PGN_CHECK_ARG(ctr_in != ctr_out && pos_in != pos_out);
  hipLaunchKernelGGL(decode_tail, dim3((unsigned)B), dim3(kTailThreads), 0, (hipStream_t)stream, logits, (int)V, emb,
                     pemb, (int)d, (int)ctx, ctr_in, ctr_out, pos_in, pos_out, out, n_rows, tok, h, p0s, (int)L,
                     logits_rec, (int)B);
  PGN_RETURN_LAUNCH();
}
