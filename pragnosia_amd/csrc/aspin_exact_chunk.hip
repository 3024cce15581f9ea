// The exact scan (fp32 operands, fp32 accumulation) in chunked form on the fp32 matrix cores: plain and delta write
// rules, forward and backward, any value width, key widths up to 384 (the delta rule) or any (the plain rule).
//
// The function is aspin_exact.hip's, for sequences long enough to fill chunks: with chunks of 64 tokens, L the
// cumulative log-decay inside a chunk, D_ts = e^(L_t - L_s) (t >= s), w_s = e^(L_last - L_s) and S the state entering
// the chunk,
//     A = tril(Q K^T o D),   M = strict_tril(K K^T o D),   X = (I + M diag(beta))^-1          (per chunk, parallel)
//     R = X V - X (e^L o K) S,   U = beta o R   (plain: U = V)                                (along the chunks)
//     S <- e^(L_last) S + (w o K)^T U
//     O = e^L o (Q S) + A U                                                                   (per chunk, parallel)
// and backward, with G the gradient on the state a chunk leaves,
//     dU = A^T dO + w o (K G),   dY = X^T (beta o dU)   (plain: dV = dU; delta: dV = dY)
//     G <- e^(L_last) G + Q^T (e^L o dO) - K^T (e^L o dY)                                     (along the chunks)
//     dQ = e^L o (dO S^T) + (dO U^T o D) K
//     dK = (dO U^T o D)^T Q + w o (U G^T) - e^L o (dY S^T) + (P + P^T) K,   P = -strict_tril(dY R^T o D) diag(beta)
//     dbeta_s = R_s . dU_s - sum_t (dY R^T)_ts M_ts
//     dla_t = sum_{r >= t > s} (dO U^T o A + P o K K^T)_rs + sum_{r >= t} (q_r . (dQ's state term)_r
//             - k_r . (e^L o dY S^T)_r) + sum_{s < t} k_s . (w o U G^T)_s + e^(L_last) <G, S>.
// Only the state's recurrence runs along the chunks. The delta rule's is kept to two products a chunk by forming
// W = X (e^L o K) (forward) and W' = X^T (beta o w o K) (backward) beforehand: R = X V - W S, dY = Y1 + W' G.
//
// Why this form: token by token (aspin_exact.hip) a step is a few multiply-adds a lane behind two cross-lane sums, with
// one workgroup a (batch, head) and value block and a checkpoint of the state every 8 tokens, so it is bound by the
// length of its serial chain. Chunked, a head-token costs 4 D (64 + D) dense flops on the matrix cores, one state per
// 64 tokens reaches memory, and everything but the state's own walk is parallel over chunks. B4 H4 T2048 D176 plain,
// forward and backward: 283 ms token by token (in two key and two value blocks), 0.33 ms here; B2 H4 T1000 D192 delta:
// 32 ms, 0.31 ms here; a forward and backward of 32 tokens (B1 H12 D64): 282 and 40 us plain, 297 and 68 us delta.
// Against 64 bits the worst output is closer than the recurrence's, whose state takes T roundings instead of T / 64:
// relative error 8.7e-7 against 9.7e-6 plain, 6.9e-7 against 2.7e-6 delta at those shapes.
//
// Decays: L is summed in fp64 and only differences (<= 0) are exponentiated, in fp32, so a long or steep run of decays
// loses nothing to cancellation; log-decays below -1e4 (e^-1e4 = 0 in fp32) are taken as -1e4, which keeps the
// differences finite for -inf.
//
// Infinities and NaN stay in the tokens that the recurrence takes them to: outputs before such a token, and gradients
// that do not come past it, are what they are without it. Entries above a score matrix's diagonal are selected to zero,
// not multiplied; a product with a triangular operand, whose zeros meet the other operand's later (transposed: earlier)
// tokens, has its non-finite results formed again over their own tokens (`own_tokens`); a log-decay of NaN or +inf is
// left out of L and makes NaN of the differences that span it (`Decays`); and dla sums what lies on either side of its
// token, with no term added that another takes away again.
//
// Products: v_mfma_f32_16x16x4f32 (A[r][k] in lane r + 16 k, B[k][c] in lane c + 16 k, D[4 g + e][c] in lane c + 16 g).
// Four of them cover a 16-wide contraction with lane group g holding k = 4 g + e in the e-th, so an operand whose
// contraction index is contiguous is one 16-byte read a lane, and an accumulator tile is the next product's B operand
// (contracted over its rows) as it stands.
#include "mfma_tile.h"

using pgn::sum16;
using pgn::wave_idx;
using pgn::WaveIdx;
using pgn::zero4;

namespace {

constexpr int CT = 64;               // tokens a chunk
constexpr int KS = 32;               // contraction slice staged at a time
constexpr int PK = KS + 4;           // pitch of a slice whose contraction index is contiguous (64 rows)
constexpr int PR = 64 + 4;           // pitch of a slice whose outer index is contiguous (KS rows), and of 64 x 64 tiles
constexpr int kSlice = 64 * PK;      // floats of a staged slice (>= KS * PR)
constexpr int kMaxDkDelta = 384;
constexpr double kLaMin = -1e4;

PGN_DEVICE f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

PGN_DEVICE f32x4 mfma16(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = mfma4(a[e], b[e], c);
  return c;
}

// An operand of a 64 x 64 product: outer index o (the product's row or column), contraction index k. kRows: element
// p[o * ld + k] (the contraction index contiguous); kCols: p[k * ld + o]. Zero past n_outer and n_k.
enum Kind { kRows, kCols };
struct Src {
  const float* p;
  int ld, n_outer, n_k;
};

// A 64 x KS slice at k0, two 16-byte pieces a thread; scaled by ks[k] when given. VEC: 16-byte loads (ld, n_outer or
// n_k multiples of 4 and p 16-byte aligned, so a piece is whole or absent); otherwise four guarded 4-byte loads.
template <int KIND, bool VEC>
PGN_DEVICE void fetch(f32x4 (&r)[2], const Src& s, int k0, int tid, const float* ks) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int x = tid + 256 * h;
    const int o = KIND == kRows ? x >> 3 : 4 * (x & 15);
    const int k = k0 + (KIND == kRows ? 4 * (x & 7) : x >> 4);
    const float* p = s.p + (KIND == kRows ? (size_t)o * s.ld + k : (size_t)k * s.ld + o);
    f32x4 v = zero4();
    if constexpr (VEC) {
      if (o < s.n_outer && k < s.n_k) v = *reinterpret_cast<const f32x4*>(p);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (o + (KIND == kRows ? 0 : e) < s.n_outer && k + (KIND == kRows ? e : 0) < s.n_k) v[e] = p[e];
    }
    if (ks != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= ks[k + (KIND == kRows ? e : 0)];
    }
    r[h] = v;
  }
}

template <int KIND>
PGN_DEVICE void put(float* t, const f32x4 (&r)[2], int tid) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int x = tid + 256 * h;
    float* p = KIND == kRows ? t + (x >> 3) * PK + 4 * (x & 7) : t + (x >> 4) * PR + 4 * (x & 15);
    *reinterpret_cast<f32x4*>(p) = r[h];
  }
}

// Outer indices o .. o + 15, contraction 16 kk .. 16 kk + 15 of a staged slice (or of a 64 x 64 tile of pitch PR,
// kCols).
template <int KIND>
PGN_DEVICE f32x4 frag(const float* t, int o, int kk, const WaveIdx& x) {
  if constexpr (KIND == kRows) {
    return *reinterpret_cast<const f32x4*>(t + (o + x.i) * PK + 16 * kk + 4 * x.g);
  } else {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = t[(16 * kk + 4 * x.g + e) * PR + o + x.i];
    return v;
  }
}

// acc += A B over a 64 x 64 output in four waves of 32 x 32 (wave w: rows 32 (w >> 1), columns 32 (w & 1)), the
// contraction in slices of KS double-buffered in `lds` (4 kSlice floats): a slice's loads are in flight while the one
// before it is multiplied, one barrier a slice. 16-blocks past the operands' outer extents are skipped. `buf` carries
// the buffer in turn from one call to the next, so calls follow each other without a barrier between.
template <int KA, int KB, bool VA, bool VB>
PGN_DEVICE void product(f32x4 (&acc)[2][2], const Src& A, const Src& B, int K, float* lds, int& buf, const WaveIdx& x,
                        const float* ks = nullptr) {
  const int tid = threadIdx.x, r0 = 32 * (x.w >> 1), c0 = 32 * (x.w & 1);
  f32x4 ra[2], rb[2];
  fetch<KA, VA>(ra, A, 0, tid, ks);
  fetch<KB, VB>(rb, B, 0, tid, nullptr);
  for (int k0 = 0; k0 < K; k0 += KS) {
    float *ta = lds + 2 * kSlice * buf, *tb = ta + kSlice;
    put<KA>(ta, ra, tid);
    put<KB>(tb, rb, tid);
    if (k0 + KS < K) {
      fetch<KA, VA>(ra, A, k0 + KS, tid, ks);
      fetch<KB, VB>(rb, B, k0 + KS, tid, nullptr);
    }
    __syncthreads();
    if (r0 < A.n_outer && c0 < B.n_outer) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (k0 + 16 * kk < K) {
          const f32x4 a0 = frag<KA>(ta, r0, kk, x), a1 = frag<KA>(ta, r0 + 16, kk, x);
          const f32x4 b0 = frag<KB>(tb, c0, kk, x), b1 = frag<KB>(tb, c0 + 16, kk, x);
          acc[0][0] = mfma16(a0, b0, acc[0][0]);
          if (r0 + 16 < A.n_outer) acc[1][0] = mfma16(a1, b0, acc[1][0]);
          if (c0 + 16 < B.n_outer) {
            acc[0][1] = mfma16(a0, b1, acc[0][1]);
            if (r0 + 16 < A.n_outer) acc[1][1] = mfma16(a1, b1, acc[1][1]);
          }
        }
      }
    }
    buf ^= 1;
  }
}

PGN_DEVICE void clear(f32x4 (&a)[2][2]) { a[0][0] = a[0][1] = a[1][0] = a[1][1] = zero4(); }

// f(row, column, value) for every element of the wave's 32 x 32 block
template <class F>
PGN_DEVICE void each(f32x4 (&acc)[2][2], const WaveIdx& x, F&& f) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        f(32 * (x.w >> 1) + 16 * i + 4 * x.g + e, 32 * (x.w & 1) + 16 * j + x.i, acc[i][j][e]);
}

// Row t of acc times sc[t]
PGN_DEVICE void scale_rows(f32x4 (&acc)[2][2], const float* __restrict__ sc, const WaveIdx& x) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const f32x4 s = *reinterpret_cast<const f32x4*>(sc + 32 * (x.w >> 1) + 16 * i + 4 * x.g);
    acc[i][0] *= s;
    acc[i][1] *= s;
  }
}

PGN_DEVICE void store_tile(f32x4 (&acc)[2][2], float* p, int ld, int nrows, int ncols, const WaveIdx& x) {
  each(acc, x, [&](int r, int c, float v) {
    if (r < nrows && c < ncols) p[(size_t)r * ld + c] = v;
  });
}

// Where acc, the 64 x 64 product of a(r, k), zero unless k <= r (LOWER) or k >= r, with b(k, c) over k < K, holds
// anything non-finite: those entries again as sums over k's own range only, since 0 times an infinity or a NaN is NaN.
// nc: columns that b has. Costs a comparison an entry where there is none.
template <bool LOWER, class FA, class FB>
PGN_DEVICE void own_tokens(f32x4 (&acc)[2][2], int K, int nc, const WaveIdx& x, FA&& a, FB&& b) {
  bool bad = false;
  each(acc, x, [&](int, int, float v) { bad |= !(fabsf(v) < INFINITY); });
  if (!__any(bad)) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = 32 * (x.w >> 1) + 16 * i + 4 * x.g, c = min(32 * (x.w & 1) + 16 * j + x.i, nc - 1);
      f32x4 s = zero4();
      for (int k = 0; k < K; ++k) {
        const float bk = b(k, c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (LOWER ? k <= r + e : k >= r + e) s[e] += a(r + e, k) * bk;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!(fabsf(acc[i][j][e]) < INFINITY)) acc[i][j][e] = s[e];
    }
}

PGN_DEVICE void add(f32x4 (&a)[2][2], const f32x4 (&b)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) a[i][j] += b[i][j];
}

// out[row] = acc's row . X's row over the wave's 32 columns (X: rows of ld floats, nrows x ncols valid)
PGN_DEVICE void row_dots(f32x4 (&acc)[2][2], const float* __restrict__ X, int ld, int nrows, int ncols, float* out,
                         const WaveIdx& x) {
  const int r0 = 32 * (x.w >> 1), c0 = 32 * (x.w & 1) + x.i;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = r0 + 16 * i + 4 * x.g + e;
      const float* p = X + (size_t)r * ld;
      float s = 0.f;
      if (r < nrows && c0 < ncols) s = acc[i][0][e] * p[c0];
      if (r < nrows && c0 + 16 < ncols) s += acc[i][1][e] * p[c0 + 16];
      s = sum16(s);
      if (x.i == 0) out[r] = s;
    }
}

// Cumulative log-decays of a chunk's n tokens (zero decay past them) in fp64, by the first wave, without those that are
// NaN or +inf (`bad`, a bit a token)
struct Decays {
  double L[CT];
  unsigned long long bad;
};
PGN_DEVICE void decay_sums(const float* __restrict__ la, int n, Decays& d) {
  const int t = threadIdx.x;
  if (t < CT) {
    const float f = t < n ? la[t] : 0.f;
    const bool ok = f < INFINITY;
    double v = ok ? ((double)f < kLaMin ? kLaMin : (double)f) : 0.;
#pragma unroll
    for (int s = 1; s < CT; s <<= 1) {
      const double y = __shfl_up(v, s);
      if (t >= s) v += y;
    }
    d.L[t] = v;
    const unsigned long long b = __ballot(!ok);
    if (t == 0) d.bad = b;
  }
}

// The decay from after token s to token t >= s, and from the chunk's start to token t
PGN_DEVICE float decay(const Decays& d, int t, int s) {
  const float v = expf((float)(d.L[t] - d.L[s]));
  return d.bad != 0 && (d.bad >> s >> 1 & ((1ull << (t - s)) - 1)) != 0 ? NAN : v;
}
PGN_DEVICE float decay_from_start(const Decays& d, int t) {
  const float v = expf((float)d.L[t]);
  return (d.bad & (~0ull >> (63 - t))) != 0 ? NAN : v;
}

struct Shape {
  // NC chunks of each sequence, from chunk c0 on; nkt, nvt: 64-wide key and value tiles; DkP: Dk rounded up to 16
  int BH, T, Dk, Dv, NC, DkP, nkt, nvt, c0;
  PGN_DEVICE int token(int c) const { return (c0 + c) * CT; }  // the first of the c-th chunk
};

// Work items numbered so that a group's items run on one XCD (workgroup i runs on XCD i mod 8) and share its L2:
// item = 8 (group / 8 * per + sub) + group % 8.
struct Item {
  int group, sub;
};
PGN_DEVICE Item item_of(int idx, int per) {
  const int x = idx & 7, r = idx >> 3;
  return Item{(r / per) * 8 + x, r % per};
}
inline unsigned items(int groups, int per) { return (unsigned)((groups + 7) / 8 * 8 * per); }

// ------------------------------------------------------------------------------------------------------------------
// Per chunk: A = tril(Q K^T o D), the decay vectors, and for the delta rule M and X. One workgroup a chunk.
template <bool DELTA, bool VEC>
__global__ __launch_bounds__(256) void exact_scores(const float* __restrict__ q, const float* __restrict__ k,
                                                    const float* __restrict__ la, const float* __restrict__ beta,
                                                    float* __restrict__ A, float* __restrict__ eL,
                                                    float* __restrict__ wt, float* __restrict__ M,
                                                    float* __restrict__ X, Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  __shared__ Decays Ls;
  __shared__ float bes[CT];
  const WaveIdx x = wave_idx();
  const int tid = threadIdx.x, bh = blockIdx.x / s.NC, c = blockIdx.x - bh * s.NC;
  const int t0 = s.token(c), n = min(CT, s.T - t0);
  const size_t row0 = (size_t)bh * s.T + t0, ch = (size_t)bh * s.NC + c;
  decay_sums(la + row0, n, Ls);
  if (DELTA && tid < CT) bes[tid] = tid < n ? beta[row0 + tid] : 0.f;
  const Src Q{q + row0 * s.Dk, s.Dk, n, s.Dk}, K{k + row0 * s.Dk, s.Dk, n, s.Dk};
  const int r0 = 32 * (x.w >> 1), c0 = 32 * (x.w & 1);
  f32x4 aq[2][2], ak[2][2];
  clear(aq);
  clear(ak);
  f32x4 rq[2], rk[2];
  fetch<kRows, VEC>(rq, Q, 0, tid, nullptr);
  fetch<kRows, VEC>(rk, K, 0, tid, nullptr);
  int buf = 0;
  for (int k0 = 0; k0 < s.Dk; k0 += KS) {
    float *tq = lds + 2 * kSlice * buf, *tk = tq + kSlice;
    put<kRows>(tq, rq, tid);
    put<kRows>(tk, rk, tid);
    if (k0 + KS < s.Dk) {
      fetch<kRows, VEC>(rq, Q, k0 + KS, tid, nullptr);
      fetch<kRows, VEC>(rk, K, k0 + KS, tid, nullptr);
    }
    __syncthreads();
    if (r0 >= c0) {  // the upper right block is masked
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const f32x4 b0 = frag<kRows>(tk, c0, kk, x), b1 = frag<kRows>(tk, c0 + 16, kk, x);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const f32x4 a = frag<kRows>(tq, r0 + 16 * i, kk, x);
          aq[i][0] = mfma16(a, b0, aq[i][0]);
          aq[i][1] = mfma16(a, b1, aq[i][1]);
          if constexpr (DELTA) {
            const f32x4 a2 = frag<kRows>(tk, r0 + 16 * i, kk, x);
            ak[i][0] = mfma16(a2, b0, ak[i][0]);
            ak[i][1] = mfma16(a2, b1, ak[i][1]);
          }
        }
      }
    }
    buf ^= 1;
  }
  __syncthreads();
  if (tid < CT) {
    eL[ch * CT + tid] = decay_from_start(Ls, tid);
    wt[ch * CT + tid] = decay(Ls, CT - 1, tid);
  }
  float* Ac = A + ch * CT * CT;
  each(aq, x, [&](int t, int u, float v) { Ac[t * CT + u] = t >= u ? v * decay(Ls, t, u) : 0.f; });
  if constexpr (DELTA) {
    float *Nt = lds, *Xt = lds + CT * PR;
    float* Mc = M + ch * CT * CT;
    each(ak, x, [&](int t, int u, float v) {
      const float m = t > u ? v * decay(Ls, t, u) : 0.f;
      Mc[t * CT + u] = m;
      Nt[t * PR + u] = t > u ? m * bes[u] : 0.f;
      Xt[t * PR + u] = 0.f;
    });
    __syncthreads();
    // the 16 x 16 diagonal blocks by forward substitution, block w on wave w, one column a lane
    {
      const int b = 16 * x.w;
      float v[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) v[t] = t == x.i ? 1.f : 0.f;
#pragma unroll
      for (int t = 1; t < 16; ++t) {
        f32x4 nr[4];
#pragma unroll
        for (int m = 0; 4 * m < t; ++m) nr[m] = *reinterpret_cast<const f32x4*>(Nt + (b + t) * PR + b + 4 * m);
#pragma unroll
        for (int u = 0; u < t; ++u) v[t] -= (u >= x.i ? nr[u >> 2][u & 3] : 0.f) * v[u];  // v[u] = 0 above the diagonal
      }
      if (x.l < 16) {
#pragma unroll
        for (int t = 0; t < 16; ++t) Xt[(b + t) * PR + b + x.i] = v[t];
      }
    }
    __syncthreads();
    // the blocks below them a level d at a time: X_ij = -X_ii sum_{m=j}^{i-1} N_im X_mj, i = j + d, block j on wave j
    auto rows16 = [&](const float* t, int o, int kc) {
      return *reinterpret_cast<const f32x4*>(t + (16 * o + x.i) * PR + 16 * kc + 4 * x.g);
    };
    for (int d = 1; d < 4; ++d) {
      const int j = x.w, i = j + d;
      if (i < 4) {
        f32x4 t = zero4();
        for (int m = j; m < i; ++m) t = mfma16(rows16(Nt, i, m), frag<kCols>(Xt + 16 * m * PR, 16 * j, 0, x), t);
        bool bad = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= !(fabsf(t[e]) < INFINITY);
        const bool careful = __any(bad);  // own_tokens for the blocks' triangular operands, X_jj and X_ii
        if (careful) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float f = 0.f;
            for (int u = 16 * j + x.i; u < 16 * i; ++u)
              f += Nt[(16 * i + 4 * x.g + e) * PR + u] * Xt[u * PR + 16 * j + x.i];
            t[e] = f;
          }
        }
        f32x4 y = mfma16(rows16(Xt, i, i), t, zero4());
        bool bady = careful;
#pragma unroll
        for (int e = 0; e < 4; ++e) bady |= !(fabsf(y[e]) < INFINITY);
        if (__any(bady)) {
          y = zero4();
#pragma unroll
          for (int u = 0; u < 16; ++u) {
            const float tu = __shfl(t[u & 3], x.i + 16 * (u >> 2));
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (u <= 4 * x.g + e) y[e] += Xt[(16 * i + 4 * x.g + e) * PR + 16 * i + u] * tu;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) Xt[(16 * i + 4 * x.g + e) * PR + 16 * j + x.i] = -y[e];
      }
      __syncthreads();
    }
    float* Xc = X + ch * CT * CT;
    for (int p = tid; p < CT * CT / 4; p += 256)
      *reinterpret_cast<f32x4*>(Xc + 4 * p) = *reinterpret_cast<const f32x4*>(Xt + (p >> 4) * PR + 4 * (p & 15));
  }
}

// ------------------------------------------------------------------------------------------------------------------
// Delta forward, per chunk and 64 columns: R <- X V (tiles of the value columns), W = X (e^L o K) (of the keys).
template <bool VEC>
__global__ __launch_bounds__(256) void exact_wy_fwd(const float* __restrict__ k, const float* __restrict__ v,
                                                    const float* __restrict__ X, const float* __restrict__ eL,
                                                    float* __restrict__ R, float* __restrict__ W, Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, s.nvt + s.nkt);
  if (it.group >= s.BH * s.NC) return;
  const int bh = it.group / s.NC, c = it.group - bh * s.NC, t0 = s.token(c), n = min(CT, s.T - t0);
  const size_t row0 = (size_t)bh * s.T + t0, ch = it.group;
  const bool val = it.sub < s.nvt;
  const int n0 = 64 * (val ? it.sub : it.sub - s.nvt), D = val ? s.Dv : s.Dk;
  f32x4 acc[2][2];
  clear(acc);
  int buf = 0;
  product<kRows, kCols, true, VEC>(acc, Src{X + ch * CT * CT, CT, CT, CT},
                                   Src{(val ? v : k) + row0 * D + n0, D, D - n0, n}, n, lds, buf, x,
                                   val ? nullptr : eL + ch * CT);
  {
    const float *Xc = X + ch * CT * CT, *vk = (val ? v : k) + row0 * D + n0, *el = eL + ch * CT;
    own_tokens<true>(
        acc, n, D - n0, x, [&](int r, int m) { return Xc[r * CT + m]; },
        [&](int m, int cc) { return (val ? 1.f : el[m]) * vk[(size_t)m * D + cc]; });
  }
  if (val)
    store_tile(acc, R + ch * CT * D + n0, D, CT, D - n0, x);  // a short last chunk's rows end in zeros
  else
    store_tile(acc, W + ch * CT * s.DkP + n0, s.DkP, CT, s.DkP - n0, x);
}

// ------------------------------------------------------------------------------------------------------------------
// Range-checked views for the state's walk: a load past one reads zero and a store there is dropped, so neither needs a
// branch, and offsets are 32-bit. Byte offset kNone is past every view.
constexpr unsigned kNone = 0x40000000u;
PGN_DEVICE __amdgpu_buffer_rsrc_t view(const float* p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, n * (int)sizeof(float), 0x00020000);
}
PGN_DEVICE float bload(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
PGN_DEVICE void bstore(__amdgpu_buffer_rsrc_t r, unsigned off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), r, (int)off, 0, 0);
}
// A value the compiler cannot derive others from across a chunk: the dozens of load addresses built on it are then a
// few additions a chunk instead of as many registers held through the walk (174 -> 92 for the delta rule's forward with
// one key tile a wave).
PGN_DEVICE unsigned fresh(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}
// Byte offset of token row 4 g, column c of a chunk's rows (4 bytes each, ld4 a row)
PGN_DEVICE unsigned row_base(const WaveIdx& x, int ld4, int c, bool ok) { return ok ? 4u * x.g * ld4 + 4u * c : kNone; }
// ... and of row 16 (p / 4) + p % 4 past it: with it, load p of a lane is the B (or transposed A) operand's k = p-th
PGN_DEVICE unsigned row_step(int p, int ld4) { return (unsigned)((16 * (p >> 2) + (p & 3)) * ld4); }

// The state along the chunks, plain rule: S <- a S + X^T (f o Y) for 64 key rows and 16 value columns a workgroup
// (key rows and value columns are independent here), X = K, Y = V, f = w forward; X = Q, Y = dO, f = e^L and S the
// state's gradient, chunks in reverse, backward (which also leaves a <G, S_c>, one partial a wave, in hs). The state
// entering (backward: the gradient leaving) every chunk goes to `states`. No LDS and no barrier: a wave's operands come
// from memory two chunks ahead.
template <bool BWD>
__global__ __launch_bounds__(256) void exact_chain_plain(const float* __restrict__ xk, const float* __restrict__ yv,
                                                         const float* __restrict__ f, const float* __restrict__ eL,
                                                         const float* init, float* __restrict__ states,
                                                         float* last, const float* __restrict__ Sc,
                                                         float* __restrict__ hs, int nvb, int nkb, Shape s) {
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, nvb * nkb);
  if (it.group >= s.BH) return;
  const int bh = it.group, vb = it.sub % nvb, kb = it.sub / nvb;
  const int col = 16 * vb + x.i, kd4 = 4 * s.Dk, vd4 = 4 * s.Dv, sn = s.Dk * s.Dv;
  const bool cok = col < s.Dv;
  const int key = 64 * kb + 16 * x.w;  // the wave's 16 key rows
  const unsigned kbase = row_base(x, kd4, key + x.i, key + x.i < s.Dk), vbase = row_base(x, vd4, col, cok);
  // rows past Dk lie past the state's end
  const unsigned sbase = cok ? (unsigned)(key + 4 * x.g) * vd4 + 4u * col : kNone;
  f32x4 S;
  {
    const __amdgpu_buffer_rsrc_t r = view(init == nullptr ? xk : init + (size_t)bh * sn, init == nullptr ? 0 : sn);
#pragma unroll
    for (int e = 0; e < 4; ++e) S[e] = bload(r, sbase + e * vd4);
  }
  struct Set {
    float k[16], v[16];
    f32x4 f[4], z;
    float a;
  };
  auto load = [&](Set& u, int c) {
    if (c < 0 || c >= s.NC) return;
    const int t0 = s.token(c), n = min(CT, s.T - t0);
    const size_t row0 = (size_t)bh * s.T + t0, ch = (size_t)bh * s.NC + c;
    const __amdgpu_buffer_rsrc_t kr = view(xk + row0 * s.Dk, n * s.Dk), vr = view(yv + row0 * s.Dv, n * s.Dv);
    const unsigned vo = fresh(vbase);
#pragma unroll
    for (int p = 0; p < 16; ++p) u.v[p] = bload(vr, vo + row_step(p, vd4));
    const unsigned ko = fresh(kbase);
#pragma unroll
    for (int p = 0; p < 16; ++p) u.k[p] = bload(kr, ko + row_step(p, kd4));
#pragma unroll
    for (int b = 0; b < 4; ++b) u.f[b] = *reinterpret_cast<const f32x4*>(f + ch * CT + 16 * b + 4 * x.g);
    u.a = eL[ch * CT + CT - 1];
    if constexpr (BWD) {
      const __amdgpu_buffer_rsrc_t zr = view(Sc + ch * sn, sn);
#pragma unroll
      for (int e = 0; e < 4; ++e) u.z[e] = bload(zr, sbase + e * vd4);
    }
  };
  auto step = [&](Set& u, int c) {
    const size_t ch = (size_t)bh * s.NC + c;
    const __amdgpu_buffer_rsrc_t out = view(states + ch * sn, sn);
#pragma unroll
    for (int e = 0; e < 4; ++e) bstore(out, sbase + e * vd4, S[e]);
    if constexpr (BWD) {
      float h = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) h += S[e] * u.z[e];
      h = pgn::wave_sum(h * u.a);
      if (x.l == 0) hs[(ch * nvb * nkb + it.sub) * 4 + x.w] = h;
    }
    S *= u.a;
#pragma unroll
    for (int p = 0; p < 16; ++p) S = mfma4(u.k[p], u.v[p] * u.f[p >> 2][p & 3], S);
  };
  const int first = BWD ? s.NC - 1 : 0, dir = BWD ? -1 : 1;
  Set u0, u1;
  load(u0, first);
  load(u1, first + dir);
  for (int i = 0; i < s.NC; i += 2) {
    const int c = first + dir * i;
    step(u0, c);
    load(u0, c + 2 * dir);
    if (i + 1 < s.NC) {
      step(u1, c + dir);
      load(u1, c + 3 * dir);
    }
  }
  if (last != nullptr) {
    const __amdgpu_buffer_rsrc_t r = view(last + (size_t)bh * sn, sn);
#pragma unroll
    for (int e = 0; e < 4; ++e) bstore(r, sbase + e * vd4, S[e]);
  }
}

// The state along the chunks, delta rule, 16 value columns and all key rows a workgroup. Wave w holds key tiles w, w +
// 4, ... (KT of 16 rows) of the state as accumulators, which are the B operands of the products contracted over keys:
// each wave forms its share of W S (64 x 16), the four shares meet in LDS, wave w finishes token rows 16 w .. 16 w + 15
// and hands them to the others through LDS (as the B operand of the state update), two barriers a chunk. Operands
// come straight from memory, each reloaded for the next chunk as soon as its product has taken it, so half a chunk's
// work covers the loads.
//   forward:  R <- R - W S (R = X V on entry), U = beta o R, S <- a S + K^T (w o U)
//   backward: dY <- dY + W G (dY = Y1 on entry), G <- a G + Q^T (e^L o dO) - K^T (e^L o dY); a <G, S_c> to hs
template <int KT, bool BWD>
__global__ __launch_bounds__(256, KT == 1 || (KT <= 3 && !BWD) ? 2 : 1) void exact_chain_delta(
    const float* __restrict__ k, const float* __restrict__ q, const float* __restrict__ dO,
    const float* __restrict__ beta, const float* __restrict__ eL, const float* __restrict__ wt,
    const float* __restrict__ W, float* __restrict__ y, float* __restrict__ U, const float* init,
    float* __restrict__ states, float* last, const float* __restrict__ Sc, float* __restrict__ hs,
    int nvb, Shape s) {
  __shared__ f32x4 part[4][4][64];
  __shared__ f32x4 us[4][64];
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, nvb);
  if (it.group >= s.BH) return;
  const int bh = it.group, vb = it.sub, col = 16 * vb + x.i;
  const int kd4 = 4 * s.Dk, vd4 = 4 * s.Dv, wd4 = 4 * s.DkP, sn = s.Dk * s.Dv;
  const bool cok = col < s.Dv;
  unsigned kbase[KT], sbase[KT], wbase[KT];
#pragma unroll
  for (int m = 0; m < KT; ++m) {
    const int key = 16 * (x.w + 4 * m);
    kbase[m] = row_base(x, kd4, key + x.i, key + x.i < s.Dk);
    sbase[m] = cok ? (unsigned)(key + 4 * x.g) * vd4 + 4u * col : kNone;  // rows past Dk lie past the state's end
    wbase[m] = key < s.DkP ? (unsigned)x.i * wd4 + 4u * (key + 4 * x.g) : kNone;
  }
  const unsigned vbase = row_base(x, vd4, col, cok), ybase = vbase + (cok ? 16u * x.w * vd4 : 0u);
  f32x4 S[KT];
  {
    const __amdgpu_buffer_rsrc_t r = view(init == nullptr ? k : init + (size_t)bh * sn, init == nullptr ? 0 : sn);
#pragma unroll
    for (int m = 0; m < KT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[m][e] = bload(r, sbase[m] + e * vd4);
  }
  f32x4 wf[KT][4], f[4], yo, bo;
  float kf[KT][16], qf[BWD ? KT : 1][16], df[BWD ? 16 : 1], z[BWD ? KT : 1][4], a = 0.f;
  auto load_w = [&](int c) {
    const __amdgpu_buffer_rsrc_t r = view(W + ((size_t)bh * s.NC + c) * CT * s.DkP, CT * s.DkP);
#pragma unroll
    for (int m = 0; m < KT; ++m) {
      const unsigned o = fresh(wbase[m]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        wf[m][t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(o + 16 * t * wd4), 0, 0));
    }
  };
  auto load_y = [&](int c) {
    const int t0 = s.token(c), n = min(CT, s.T - t0);
    const size_t row0 = (size_t)bh * s.T + t0, yrow = BWD ? row0 : ((size_t)bh * s.NC + c) * CT;
    const __amdgpu_buffer_rsrc_t r = view(y + yrow * s.Dv, (BWD ? n : CT) * s.Dv);
    const __amdgpu_buffer_rsrc_t br = view(BWD ? wt : beta + row0, BWD ? 0 : n);
    const unsigned o = fresh(ybase);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      yo[e] = bload(r, o + e * vd4);
      if constexpr (!BWD) bo[e] = bload(br, 4u * (16 * x.w + 4 * x.g + e));
    }
  };
  auto load_k = [&](int c) {
    const int t0 = s.token(c), n = min(CT, s.T - t0);
    const size_t row0 = (size_t)bh * s.T + t0, ch = (size_t)bh * s.NC + c;
    const __amdgpu_buffer_rsrc_t kr = view(k + row0 * s.Dk, n * s.Dk);
#pragma unroll
    for (int m = 0; m < KT; ++m) {
      const unsigned o = fresh(kbase[m]);
#pragma unroll
      for (int p = 0; p < 16; ++p) kf[m][p] = bload(kr, o + row_step(p, kd4));
    }
    if constexpr (BWD) {
      const __amdgpu_buffer_rsrc_t qr = view(q + row0 * s.Dk, n * s.Dk), dr = view(dO + row0 * s.Dv, n * s.Dv);
      const __amdgpu_buffer_rsrc_t zr = view(Sc + ch * sn, sn);
      const unsigned vo = fresh(vbase);
#pragma unroll
      for (int p = 0; p < 16; ++p) df[p] = bload(dr, vo + row_step(p, vd4));
#pragma unroll
      for (int m = 0; m < KT; ++m) {
        const unsigned o = fresh(kbase[m]);
#pragma unroll
        for (int p = 0; p < 16; ++p) qf[m][p] = bload(qr, o + row_step(p, kd4));
#pragma unroll
        for (int e = 0; e < 4; ++e) z[m][e] = bload(zr, sbase[m] + e * vd4);
      }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
      f[b] = *reinterpret_cast<const f32x4*>((BWD ? eL : wt) + ch * CT + 16 * b + 4 * x.g);
    a = eL[ch * CT + CT - 1];
  };
  const int first = BWD ? s.NC - 1 : 0, dir = BWD ? -1 : 1;
  load_w(first);
  load_y(first);
  load_k(first);
  for (int i = 0; i < s.NC; ++i) {
    const int c = first + dir * i;
    const bool more = i + 1 < s.NC;
    const int t0 = s.token(c), n = min(CT, s.T - t0);
    const size_t row0 = (size_t)bh * s.T + t0, ch = (size_t)bh * s.NC + c;
    f32x4 P[4] = {zero4(), zero4(), zero4(), zero4()};
#pragma unroll
    for (int m = 0; m < KT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) P[r] = mfma16(wf[m][r], S[m], P[r]);
    if (more) load_w(c + dir);
#pragma unroll
    for (int r = 0; r < 4; ++r) part[x.w][r][x.l] = P[r];
    {
      const __amdgpu_buffer_rsrc_t out = view(states + ch * sn, sn);
#pragma unroll
      for (int m = 0; m < KT; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) bstore(out, sbase[m] + e * vd4, S[m][e]);
    }
    __syncthreads();
    {
      const f32x4 sum = (part[0][x.w][x.l] + part[1][x.w][x.l]) + (part[2][x.w][x.l] + part[3][x.w][x.l]);
      const f32x4 v = BWD ? yo + sum : yo - sum;
      const __amdgpu_buffer_rsrc_t yr = view(y + (BWD ? row0 : ch * CT) * s.Dv, (BWD ? n : CT) * s.Dv);
      const unsigned o = fresh(ybase);
#pragma unroll
      for (int e = 0; e < 4; ++e) bstore(yr, o + e * vd4, v[e]);
      if constexpr (BWD) {
        us[x.w][x.l] = v;
      } else {
        const f32x4 u = v * bo;
        const __amdgpu_buffer_rsrc_t ur = view(U + ch * CT * s.Dv, CT * s.Dv);
#pragma unroll
        for (int e = 0; e < 4; ++e) bstore(ur, o + e * vd4, u[e]);
        us[x.w][x.l] = u;
      }
    }
    if (more) load_y(c + dir);
    if constexpr (BWD) {
      float h = 0.f;
#pragma unroll
      for (int m = 0; m < KT; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) h += S[m][e] * z[m][e];
      h = pgn::wave_sum(h * a);
      if (x.l == 0) hs[(ch * nvb + vb) * 4 + x.w] = h;
    }
#pragma unroll
    for (int m = 0; m < KT; ++m) S[m] *= a;
    if constexpr (BWD) {  // the part of the update that needs no dY, before the barrier
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const float b = df[p] * f[p >> 2][p & 3];
#pragma unroll
        for (int m = 0; m < KT; ++m) S[m] = mfma4(qf[m][p], b, S[m]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int p4 = 0; p4 < 4; ++p4) {
      const f32x4 b = BWD ? -(us[p4][x.l] * f[p4]) : us[p4][x.l] * f[p4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < KT; ++m) S[m] = mfma4(kf[m][4 * p4 + e], b[e], S[m]);
    }
    if (more) load_k(c + dir);
  }
  if (last != nullptr) {
    const __amdgpu_buffer_rsrc_t r = view(last + (size_t)bh * sn, sn);
#pragma unroll
    for (int m = 0; m < KT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) bstore(r, sbase[m] + e * vd4, S[m][e]);
  }
}

// ------------------------------------------------------------------------------------------------------------------
// Outputs, per chunk and 64 value columns: O = e^L o (Q S) + A U (delta: u = U, a chunk's rows together; else V).
template <bool VEC>
__global__ __launch_bounds__(256) void exact_out(const float* __restrict__ q, const float* __restrict__ u,
                                                 const float* __restrict__ A, const float* __restrict__ eL,
                                                 const float* __restrict__ Sc, float* __restrict__ o, bool delta,
                                                 Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, s.nvt);
  if (it.group >= s.BH * s.NC) return;
  const int bh = it.group / s.NC, c = it.group - bh * s.NC, t0 = s.token(c), n = min(CT, s.T - t0), n0 = 64 * it.sub;
  const size_t row0 = (size_t)bh * s.T + t0, ch = it.group;
  f32x4 acc[2][2];
  clear(acc);
  int buf = 0;
  product<kRows, kCols, VEC, VEC>(acc, Src{q + row0 * s.Dk, s.Dk, n, s.Dk},
                                  Src{Sc + ch * s.Dk * s.Dv + n0, s.Dv, s.Dv - n0, s.Dk}, s.Dk, lds, buf, x);
  scale_rows(acc, eL + ch * CT, x);
  const float *Ac = A + ch * CT * CT, *uc = u + (delta ? ch * CT : row0) * s.Dv + n0;
  f32x4 au[2][2];
  clear(au);
  product<kRows, kCols, true, VEC>(au, Src{Ac, CT, n, CT}, Src{uc, s.Dv, s.Dv - n0, n}, n, lds, buf, x);
  own_tokens<true>(
      au, n, s.Dv - n0, x, [&](int r, int m) { return Ac[r * CT + m]; },
      [&](int m, int cc) { return uc[(size_t)m * s.Dv + cc]; });
  add(acc, au);
  store_tile(acc, o + row0 * s.Dv + n0, s.Dv, n, s.Dv - n0, x);
}

// ------------------------------------------------------------------------------------------------------------------
// Delta backward, per chunk and 64 columns: Y1 = X^T (beta o (A^T dO)) (tiles of the value columns, into dv) and
// W' = X^T (beta o w o K) (of the keys).
template <bool VEC>
__global__ __launch_bounds__(256) void exact_wy_bwd(const float* __restrict__ k, const float* __restrict__ dO,
                                                    const float* __restrict__ beta, const float* __restrict__ A,
                                                    const float* __restrict__ X, const float* __restrict__ wt,
                                                    float* __restrict__ y, float* __restrict__ W, Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  __shared__ __align__(16) float tile[CT * PR];
  __shared__ __align__(16) float sc[CT];
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, s.nvt + s.nkt);
  if (it.group >= s.BH * s.NC) return;
  const int bh = it.group / s.NC, c = it.group - bh * s.NC, t0 = c * CT, n = min(CT, s.T - t0), tid = threadIdx.x;
  const size_t row0 = (size_t)bh * s.T + t0, ch = it.group;
  const bool val = it.sub < s.nvt;
  const int n0 = 64 * (val ? it.sub : it.sub - s.nvt);
  if (tid < CT) sc[tid] = tid < n ? beta[row0 + tid] * (val ? 1.f : wt[ch * CT + tid]) : 0.f;
  __syncthreads();
  const Src Xt{X + ch * CT * CT, CT, CT, CT};
  f32x4 acc[2][2];
  clear(acc);
  int buf = 0;
  if (!val) {
    const float* kc = k + row0 * s.Dk + n0;
    product<kCols, kCols, true, VEC>(acc, Xt, Src{kc, s.Dk, s.Dk - n0, n}, n, lds, buf, x, sc);
    own_tokens<false>(
        acc, n, s.Dk - n0, x, [&](int r, int m) { return Xt.p[m * CT + r]; },
        [&](int m, int cc) { return sc[m] * kc[(size_t)m * s.Dk + cc]; });
    store_tile(acc, W + ch * CT * s.DkP + n0, s.DkP, CT, s.DkP - n0, x);
    return;
  }
  const int nc = s.Dv - n0;
  const float *Ac = A + ch * CT * CT, *doc = dO + row0 * s.Dv + n0;
  product<kCols, kCols, true, VEC>(acc, Src{Ac, CT, CT, n}, Src{doc, s.Dv, nc, n}, n, lds, buf, x);
  own_tokens<false>(
      acc, n, nc, x, [&](int r, int m) { return Ac[m * CT + r]; },
      [&](int m, int cc) { return doc[(size_t)m * s.Dv + cc]; });
  scale_rows(acc, sc, x);
  each(acc, x, [&](int r, int cc, float v) { tile[r * PR + cc] = v; });
  f32x4 rx[2];
  __syncthreads();  // every wave is done with the slices of the product above
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    fetch<kCols, true>(rx, Xt, KS * h, tid, nullptr);
    put<kCols>(lds + kSlice * h, rx, tid);
  }
  __syncthreads();
  clear(acc);
  const int r0 = 32 * (x.w >> 1), c0 = 32 * (x.w & 1);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const float* ta = lds + kSlice * (kk >> 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4 a = frag<kCols>(ta, r0 + 16 * i, kk & 1, x);
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma16(a, frag<kCols>(tile, c0 + 16 * j, kk, x), acc[i][j]);
    }
  }
  own_tokens<false>(
      acc, CT, nc, x, [&](int r, int m) { return Xt.p[m * CT + r]; },
      [&](int m, int cc) { return tile[m * PR + cc]; });
  store_tile(acc, y + row0 * s.Dv + n0, s.Dv, n, nc, x);
}

// ------------------------------------------------------------------------------------------------------------------
// Backward, per chunk: dA = tril(dO U^T o D) (before D: its products with A give the decay gradient's sums over the
// pairs of tokens on either side of each, into rc), and for the delta rule P + P^T, Z's sums and dbeta's second term
// (into db).
template <bool DELTA, bool VEC>
__global__ __launch_bounds__(256) void exact_scores_bwd(const float* __restrict__ dO, const float* __restrict__ u,
                                                        const float* __restrict__ dY, const float* __restrict__ R,
                                                        const float* __restrict__ la, const float* __restrict__ beta,
                                                        const float* __restrict__ A, const float* __restrict__ M,
                                                        float* __restrict__ dA, float* __restrict__ Psym,
                                                        float* __restrict__ rc, float* __restrict__ db, Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  __shared__ Decays Ls;
  __shared__ float bes[CT];
  const WaveIdx x = wave_idx();
  const int tid = threadIdx.x, bh = blockIdx.x / s.NC, c = blockIdx.x - bh * s.NC;
  const int t0 = c * CT, n = min(CT, s.T - t0);
  const size_t row0 = (size_t)bh * s.T + t0, ch = (size_t)bh * s.NC + c, urow = DELTA ? ch * CT : row0;
  decay_sums(la + row0, n, Ls);
  if (DELTA && tid < CT) bes[tid] = tid < n ? beta[row0 + tid] : 0.f;
  f32x4 a1[2][2], a2[2][2];
  clear(a1);
  clear(a2);
  int buf = 0;
  product<kRows, kRows, VEC, VEC>(a1, Src{dO + row0 * s.Dv, s.Dv, n, s.Dv}, Src{u + urow * s.Dv, s.Dv, n, s.Dv}, s.Dv,
                                  lds, buf, x);
  if constexpr (DELTA)
    product<kRows, kRows, VEC, VEC>(a2, Src{dY + row0 * s.Dv, s.Dv, n, s.Dv}, Src{R + urow * s.Dv, s.Dv, n, s.Dv},
                                    s.Dv, lds, buf, x);
  __syncthreads();
  float *E = lds, *F = lds + CT * PR;  // the decay gradient's matrix; dY R^T o M
  const float *Ac = A + ch * CT * CT, *Mc = DELTA ? M + ch * CT * CT : nullptr;
  float* dAc = dA + ch * CT * CT;
  each(a1, x, [&](int t, int v, float g) {
    dAc[t * CT + v] = t >= v ? g * decay(Ls, t, v) : 0.f;
    E[t * PR + v] = t > v ? g * Ac[t * CT + v] : 0.f;
  });
  if constexpr (DELTA) {
    each(a2, x, [&](int t, int v, float g) {
      const float z = t > v ? g * Mc[t * CT + v] : 0.f;
      F[t * PR + v] = z;
      E[t * PR + v] -= z * bes[v];
    });
  }
  __syncthreads();
  {
    const int r = tid >> 2, m = tid & 3;
    // row r's sums up to, not including, each column: within the thread's 16, then over the four threads of the row
    f32x4 v[4];
    float run = 0.f, cf = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(E + r * PR + 16 * m + 4 * e);
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        v[e][z] = run;
        run += w[z];
      }
    }
    float before = 0.f;
#pragma unroll
    for (int z = 1; z < 4; ++z) {
      const float y = __shfl_up(run, z);
      if (m >= z) before += y;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) *reinterpret_cast<f32x4*>(E + r * PR + 16 * m + 4 * e) = v[e] + before;
    __syncthreads();
    float d = 0.f;  // column r, the rows from r on
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if (4 * e + m >= r) d += E[(4 * e + m) * PR + r];
      if (DELTA) cf += F[(4 * e + m) * PR + r];
    }
    d = group_sum<4>(d);
    cf = group_sum<4>(cf);
    if (m == 0) {
      rc[ch * CT + r] = d;
      if (DELTA) db[ch * CT + r] = -cf;
    }
  }
  if constexpr (DELTA) {
    __syncthreads();
    each(a2, x, [&](int t, int v, float g) { E[t * PR + v] = t > v ? -g * decay(Ls, t, v) * bes[v] : 0.f; });
    __syncthreads();
    float* Pc = Psym + ch * CT * CT;
    for (int p = tid; p < CT * CT; p += 256) {
      const int t = p >> 6, v = p & 63;
      Pc[p] = E[t * PR + v] + E[v * PR + t];
    }
  }
}

// Gradients, per chunk and 64 columns, the tiles of dV (delta: dU, only for its row products with R), dQ and dK.
// Partial sums, one a (tile, wave column): q . dQ's state term, k . (w o U G^T), k . (e^L o dY S^T), R . dU.
template <bool DELTA, bool VEC>
__global__ __launch_bounds__(256, DELTA ? 3 : 4) void exact_grads(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ u,
    const float* __restrict__ R, const float* __restrict__ dO, const float* __restrict__ dY,
    const float* __restrict__ A, const float* __restrict__ dA, const float* __restrict__ Psym,
    const float* __restrict__ eL, const float* __restrict__ wt, const float* __restrict__ Sc,
    const float* __restrict__ G, float* __restrict__ dq, float* __restrict__ dk, float* __restrict__ dv,
    float* __restrict__ pq, float* __restrict__ pk, float* __restrict__ py, float* __restrict__ pb, Shape s) {
  __shared__ __align__(16) float lds[4 * kSlice];
  const WaveIdx x = wave_idx();
  const Item it = item_of(blockIdx.x, s.nvt + 2 * s.nkt);
  if (it.group >= s.BH * s.NC) return;
  const int bh = it.group / s.NC, c = it.group - bh * s.NC, t0 = c * CT, n = min(CT, s.T - t0);
  const size_t row0 = (size_t)bh * s.T + t0, ch = it.group, tot = (size_t)s.BH * s.NC * CT;
  const size_t urow = DELTA ? ch * CT : row0;
  const float *Sp = Sc + ch * s.Dk * s.Dv, *Gp = G + ch * s.Dk * s.Dv;
  const float *Ac = A + ch * CT * CT, *dAc = dA + ch * CT * CT;
  f32x4 acc[2][2], tri[2][2];
  clear(acc);
  clear(tri);
  int buf = 0;
  if (it.sub >= 2 * s.nkt) {
    const int tile = it.sub - 2 * s.nkt, n0 = 64 * tile, nc = s.Dv - n0;
    product<kRows, kCols, VEC, VEC>(acc, Src{k + row0 * s.Dk, s.Dk, n, s.Dk}, Src{Gp + n0, s.Dv, nc, s.Dk}, s.Dk, lds,
                                    buf, x);
    scale_rows(acc, wt + ch * CT, x);
    const float* doc = dO + row0 * s.Dv + n0;
    product<kCols, kCols, true, VEC>(tri, Src{Ac, CT, CT, n}, Src{doc, s.Dv, nc, n}, n, lds, buf, x);
    own_tokens<false>(
        tri, n, nc, x, [&](int r, int m) { return Ac[m * CT + r]; },
        [&](int m, int cc) { return doc[(size_t)m * s.Dv + cc]; });
    add(acc, tri);
    if constexpr (DELTA)
      row_dots(acc, R + urow * s.Dv + n0, s.Dv, n, nc, pb + (size_t)(2 * tile + (x.w & 1)) * tot + ch * CT, x);
    else
      store_tile(acc, dv + row0 * s.Dv + n0, s.Dv, n, nc, x);
    return;
  }
  const bool isq = it.sub < s.nkt;
  const int tile = isq ? it.sub : it.sub - s.nkt, n0 = 64 * tile, nc = s.Dk - n0;
  const size_t slot = (size_t)(2 * tile + (x.w & 1)) * tot + ch * CT;
  const float* kt = k + row0 * s.Dk + n0;
  if (isq) {
    const float* qt = q + row0 * s.Dk + n0;
    product<kRows, kRows, VEC, VEC>(acc, Src{dO + row0 * s.Dv, s.Dv, n, s.Dv},
                                    Src{Sp + (size_t)n0 * s.Dv, s.Dv, nc, s.Dv}, s.Dv, lds, buf, x);
    scale_rows(acc, eL + ch * CT, x);
    row_dots(acc, qt, s.Dk, n, nc, pq + slot, x);
    product<kRows, kCols, true, VEC>(tri, Src{dAc, CT, n, CT}, Src{kt, s.Dk, nc, n}, n, lds, buf, x);
    own_tokens<true>(
        tri, n, nc, x, [&](int r, int m) { return dAc[r * CT + m]; },
        [&](int m, int cc) { return kt[(size_t)m * s.Dk + cc]; });
    add(acc, tri);
    store_tile(acc, dq + row0 * s.Dk + n0, s.Dk, n, nc, x);
    return;
  }
  product<kRows, kRows, VEC, VEC>(acc, Src{u + urow * s.Dv, s.Dv, n, s.Dv},
                                  Src{Gp + (size_t)n0 * s.Dv, s.Dv, nc, s.Dv}, s.Dv, lds, buf, x);
  scale_rows(acc, wt + ch * CT, x);
  row_dots(acc, kt, s.Dk, n, nc, pk + slot, x);
  if constexpr (DELTA) {
    f32x4 ay[2][2];
    clear(ay);
    product<kRows, kRows, VEC, VEC>(ay, Src{dY + row0 * s.Dv, s.Dv, n, s.Dv},
                                    Src{Sp + (size_t)n0 * s.Dv, s.Dv, nc, s.Dv}, s.Dv, lds, buf, x);
    scale_rows(ay, eL + ch * CT, x);
    row_dots(ay, kt, s.Dk, n, nc, py + slot, x);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] -= ay[i][j];
    product<kRows, kCols, true, VEC>(acc, Src{Psym + ch * CT * CT, CT, CT, CT}, Src{kt, s.Dk, nc, n}, n, lds, buf, x);
  }
  const float* qt = q + row0 * s.Dk + n0;
  product<kCols, kCols, true, VEC>(tri, Src{dAc, CT, CT, n}, Src{qt, s.Dk, nc, n}, n, lds, buf, x);
  own_tokens<false>(
      tri, n, nc, x, [&](int r, int m) { return dAc[m * CT + r]; },
      [&](int m, int cc) { return qt[(size_t)m * s.Dk + cc]; });
  add(acc, tri);
  store_tile(acc, dk + row0 * s.Dk + n0, s.Dk, n, nc, x);
}

// dla and dbeta from the partial sums, one wave a chunk; the sums from each token on and before it in fp64.
template <bool DELTA>
__global__ __launch_bounds__(64) void exact_gates_bwd(const float* __restrict__ rc, const float* __restrict__ db,
                                                      const float* __restrict__ pq, const float* __restrict__ pk,
                                                      const float* __restrict__ py, const float* __restrict__ pb,
                                                      const float* __restrict__ hs, int nhs, float* __restrict__ dla,
                                                      float* __restrict__ dbeta, Shape s) {
  const int t = threadIdx.x, bh = blockIdx.x / s.NC, c = blockIdx.x - bh * s.NC, n = min(CT, s.T - c * CT);
  const size_t ch = blockIdx.x, tot = (size_t)s.BH * s.NC * CT, at = ch * CT + t;
  double from = 0., before = 0., b = DELTA ? db[at] : 0., end = 0.;
  for (int m = 0; m < 2 * s.nkt; ++m) {
    from += pq[m * tot + at];
    before += pk[m * tot + at];
    if (DELTA) from -= py[m * tot + at];
  }
  if (DELTA)
    for (int m = 0; m < 2 * s.nvt; ++m) b += pb[m * tot + at];
  for (int m = t; m < nhs; m += 64) end += hs[ch * nhs + m];
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) end += __shfl_xor(end, m);
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const double y = __shfl_down(from, m), z = __shfl_up(before, m);
    if (t + m < 64) from += y;
    if (t >= m) before += z;
  }
  before = __shfl_up(before, 1);
  if (t == 0) before = 0.;
  if (t < n) {
    const size_t row = (size_t)bh * s.T + c * CT + t;
    dla[row] = (float)((double)rc[at] + (from + before) + end);
    if (DELTA) dbeta[row] = (float)b;
  }
}

// ------------------------------------------------------------------------------------------------------------------

bool chunk_shape_ok(int64_t B, int64_t H, int64_t T, int64_t Dk, int64_t Dv, bool delta) {
  if (B <= 0 || H <= 0 || T <= 0 || Dk <= 0 || Dv <= 0) return false;
  if (delta && Dk > kMaxDkDelta) return false;
  if (Dk > 4096 || Dv > 4096 || T >= ((int64_t)1 << 28) || B * H >= ((int64_t)1 << 24)) return false;
  const int64_t nc = (T + CT - 1) / CT, tiles = 2 * ((Dk + 63) / 64) + (Dv + 63) / 64;
  return (B * H * nc + 8) * tiles < ((int64_t)1 << 31) &&
         (B * H + 8) * ((Dv + 15) / 16) * ((Dk + 63) / 64) < ((int64_t)1 << 31);
}

Shape shape_of(int64_t B, int64_t H, int64_t T, int64_t Dk, int64_t Dv) {
  Shape s;
  s.BH = (int)(B * H);
  s.T = (int)T;
  s.Dk = (int)Dk;
  s.Dv = (int)Dv;
  s.NC = (int)((T + CT - 1) / CT);
  s.DkP = (int)((Dk + 15) / 16 * 16);
  s.nkt = (int)((Dk + 63) / 64);
  s.nvt = (int)((Dv + 63) / 64);
  s.c0 = 0;
  return s;
}

bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (((uintptr_t)p & 15) != 0) return false;
  return true;
}

int tiles_a_wave(int Dk) { return ((Dk + 15) / 16 + 3) / 4; }

// Offsets (floats) of the backward's workspace.
struct BwdWs {
  size_t G, dA, P, W, hs, rc, db, pq, pk, py, pb, total;
};
BwdWs bwd_ws(const Shape& s, bool delta) {
  const size_t chunks = (size_t)s.BH * s.NC, tot = chunks * CT, nvb = (s.Dv + 15) / 16, nkb = delta ? 1 : s.nkt;
  BwdWs w;
  size_t at = 0;
  auto take = [&](size_t n) {
    const size_t p = at;
    at += (n + 3) / 4 * 4;
    return p;
  };
  w.G = take(chunks * s.Dk * s.Dv);
  w.dA = take(chunks * CT * CT);
  w.P = take(delta ? chunks * CT * CT : 0);
  w.W = take(delta ? chunks * CT * s.DkP : 0);
  w.hs = take(chunks * nvb * nkb * 4);
  w.rc = take(tot);
  w.db = take(delta ? tot : 0);
  w.pq = take(2 * s.nkt * tot);
  w.pk = take(2 * s.nkt * tot);
  w.py = take(delta ? 2 * s.nkt * tot : 0);
  w.pb = take(delta ? 2 * s.nvt * tot : 0);
  w.total = at;
  return w;
}

#define PGN_LAUNCHED()                             \
  do {                                             \
    const hipError_t e_ = hipGetLastError();       \
    if (e_ != hipSuccess) return (int)e_;          \
  } while (0)

template <bool BWD>
int launch_chain_delta(const float* k, const float* q, const float* dO, const float* beta, const float* eL,
                       const float* wt, const float* W, float* y, float* U, const float* init, float* states,
                       float* last, const float* Sc, float* hs, const Shape& s, hipStream_t st) {
  const int nvb = (s.Dv + 15) / 16;
  const dim3 grid(items(s.BH, nvb)), blk(256);
#define PGN_CHAIN(KT)                                                                                             \
  case KT:                                                                                                        \
    hipLaunchKernelGGL((exact_chain_delta<KT, BWD>), grid, blk, 0, st, k, q, dO, beta, eL, wt, W, y, U, init,      \
                       states, last, Sc, hs, nvb, s);                                                             \
    break
  switch (tiles_a_wave(s.Dk)) {
    PGN_CHAIN(1);
    PGN_CHAIN(2);
    PGN_CHAIN(3);
    PGN_CHAIN(4);
    PGN_CHAIN(5);
    PGN_CHAIN(6);
    default: return PRAGNOSIA_ERR_UNSUPPORTED;
  }
#undef PGN_CHAIN
  PGN_LAUNCHED();
  return PRAGNOSIA_OK;
}

template <bool DELTA, bool VEC>
int chunk_fwd(const float* q, const float* k, const float* v, const float* la, const float* beta, const float* S0,
              float* o, float* Sfin, float* Sc, float* A, float* gates, float* M, float* X, float* R, float* U,
              float* W, const Shape& s, hipStream_t st) {
  const unsigned chunks = (unsigned)(s.BH * s.NC);
  float *eL = gates, *wt = gates + (size_t)chunks * CT;
  hipLaunchKernelGGL((exact_scores<DELTA, VEC>), dim3(chunks), dim3(256), 0, st, q, k, la, beta, A, eL, wt, M, X, s);
  PGN_LAUNCHED();
  if constexpr (DELTA) {
    hipLaunchKernelGGL((exact_wy_fwd<VEC>), dim3(items(chunks, s.nvt + s.nkt)), dim3(256), 0, st, k, v, X, eL, R, W, s);
    PGN_LAUNCHED();
    const int e = launch_chain_delta<false>(k, nullptr, nullptr, beta, eL, wt, W, R, U, S0, Sc, Sfin, nullptr,
                                            nullptr, s, st);
    if (e != PRAGNOSIA_OK) return e;
  } else {
    const int nvb = (s.Dv + 15) / 16;
    hipLaunchKernelGGL((exact_chain_plain<false>), dim3(items(s.BH, nvb * s.nkt)), dim3(256), 0, st, k, v, wt, eL,
                       S0, Sc, Sfin, nullptr, nullptr, nvb, s.nkt, s);
    PGN_LAUNCHED();
  }
  hipLaunchKernelGGL((exact_out<VEC>), dim3(items(chunks, s.nvt)), dim3(256), 0, st, q, DELTA ? U : v, A, eL, Sc, o,
                     DELTA, s);
  PGN_LAUNCHED();
  return PRAGNOSIA_OK;
}

template <bool DELTA, bool VEC>
int chunk_bwd(const float* q, const float* k, const float* v, const float* la, const float* beta, const float* Sc,
              const float* A, const float* gates, const float* M, const float* X, const float* R, const float* U,
              const float* dO, const float* dSfin, float* dq, float* dk, float* dv, float* dla, float* dbeta,
              float* dS0, float* ws, const Shape& s, hipStream_t st) {
  const unsigned chunks = (unsigned)(s.BH * s.NC);
  const float *eL = gates, *wt = gates + (size_t)chunks * CT;
  const BwdWs w = bwd_ws(s, DELTA);
  float *G = ws + w.G, *dA = ws + w.dA, *P = ws + w.P, *W = ws + w.W, *hs = ws + w.hs, *rc = ws + w.rc;
  float *db = ws + w.db, *pq = ws + w.pq, *pk = ws + w.pk, *py = ws + w.py, *pb = ws + w.pb;
  const int nvb = (s.Dv + 15) / 16;
  const float* u = DELTA ? U : v;
  if constexpr (DELTA) {
    hipLaunchKernelGGL((exact_wy_bwd<VEC>), dim3(items(chunks, s.nvt + s.nkt)), dim3(256), 0, st, k, dO, beta, A, X,
                       wt, dv, W, s);
    PGN_LAUNCHED();
    const int e = launch_chain_delta<true>(k, q, dO, beta, eL, wt, W, dv, nullptr, dSfin, G, dS0, Sc, hs, s, st);
    if (e != PRAGNOSIA_OK) return e;
  } else {
    hipLaunchKernelGGL((exact_chain_plain<true>), dim3(items(s.BH, nvb * s.nkt)), dim3(256), 0, st, q, dO, eL, eL,
                       dSfin, G, dS0, Sc, hs, nvb, s.nkt, s);
    PGN_LAUNCHED();
  }
  hipLaunchKernelGGL((exact_scores_bwd<DELTA, VEC>), dim3(chunks), dim3(256), 0, st, dO, u, dv, R, la, beta, A, M, dA,
                     P, rc, db, s);
  PGN_LAUNCHED();
  hipLaunchKernelGGL((exact_grads<DELTA, VEC>), dim3(items(chunks, s.nvt + 2 * s.nkt)), dim3(256), 0, st, q, k, u, R,
                     dO, dv, A, dA, P, eL, wt, Sc, G, dq, dk, dv, pq, pk, py, pb, s);
  PGN_LAUNCHED();
  hipLaunchKernelGGL((exact_gates_bwd<DELTA>), dim3(chunks), dim3(64), 0, st, rc, db, pq, pk, py, pb, hs,
                     nvb * (DELTA ? 1 : s.nkt) * 4, dla, dbeta, s);
  PGN_LAUNCHED();
  return PRAGNOSIA_OK;
}

}  // namespace

extern "C" int64_t pragnosia_aspin_exact_chunk_bwd_workspace_bytes(int64_t B, int64_t H, int64_t T, int64_t Dk,
                                                                   int64_t Dv, int delta) {
  if (!chunk_shape_ok(B, H, T, Dk, Dv, delta != 0)) return -1;
  return (int64_t)(bwd_ws(shape_of(B, H, T, Dk, Dv), delta != 0).total * sizeof(float));
}

extern "C" int pragnosia_aspin_exact_chunk_fwd(const float* q, const float* k, const float* v, const float* la,
                                               const float* beta, const float* S0, float* o, float* S_final,
                                               float* states, float* scores, float* gates, float* M, float* X,
                                               float* R, float* U, float* W, int64_t B, int64_t H, int64_t T,
                                               int64_t Dk, int64_t Dv, int64_t first, int64_t chunks, void* stream) {
  const bool delta = beta != nullptr;
  PGN_CHECK_ARG(chunk_shape_ok(B, H, T, Dk, Dv, delta));
  PGN_CHECK_ARG(first >= 0 && chunks > 0 && first <= (T + CT - 1) / CT - chunks);
  PGN_CHECK_ARG(q && k && v && la && o && S_final && states && scores && gates);
  PGN_CHECK_ARG(aligned16({scores, gates}));
  if (delta) PGN_CHECK_ARG(M && X && R && U && W && aligned16({M, X, W}));
  Shape s = shape_of(B, H, T, Dk, Dv);
  s.c0 = (int)first;
  s.NC = (int)chunks;
  hipStream_t st = (hipStream_t)stream;
  // 16-byte loads where every row starts on one
  const bool vec = Dk % 4 == 0 && Dv % 4 == 0 && aligned16({q, k, v, states, U});
#define PGN_FWD(D, V) \
  return chunk_fwd<D, V>(q, k, v, la, beta, S0, o, S_final, states, scores, gates, M, X, R, U, W, s, st)
  if (delta) {
    if (vec) PGN_FWD(true, true);
    PGN_FWD(true, false);
  }
  if (vec) PGN_FWD(false, true);
  PGN_FWD(false, false);
#undef PGN_FWD
}

extern "C" int pragnosia_aspin_exact_chunk_bwd(const float* q, const float* k, const float* v, const float* la,
                                               const float* beta, const float* states, const float* scores,
                                               const float* gates, const float* M, const float* X, const float* R,
                                               const float* U, const float* dO, const float* dS_final, float* dq,
                                               float* dk, float* dv, float* dla, float* dbeta, float* dS0,
                                               float* workspace, int64_t workspace_bytes, int64_t B, int64_t H,
                                               int64_t T, int64_t Dk, int64_t Dv, void* stream) {
  const bool delta = beta != nullptr;
  PGN_CHECK_ARG(chunk_shape_ok(B, H, T, Dk, Dv, delta));
  PGN_CHECK_ARG(q && k && v && la && states && scores && gates && dO && dq && dk && dv && dla && workspace);
  PGN_CHECK_ARG(aligned16({scores, gates, workspace}));
  if (delta) PGN_CHECK_ARG(M && X && R && U && dbeta && aligned16({M, X}));
  const Shape s = shape_of(B, H, T, Dk, Dv);
  PGN_CHECK_ARG(workspace_bytes >= (int64_t)(bwd_ws(s, delta).total * sizeof(float)));
  hipStream_t st = (hipStream_t)stream;
  const bool vec = Dk % 4 == 0 && Dv % 4 == 0 && aligned16({q, k, v, states, R, U, dO, dv});
#define PGN_BWD(D, V)                                                                                              \
  return chunk_bwd<D, V>(q, k, v, la, beta, states, scores, gates, M, X, R, U, dO, dS_final, dq, dk, dv, dla, dbeta, \
                         dS0, workspace, s, st)
  if (delta) {
    if (vec) PGN_BWD(true, true);
    PGN_BWD(true, false);
  }
  if (vec) PGN_BWD(false, true);
  PGN_BWD(false, false);
#undef PGN_BWD
}
