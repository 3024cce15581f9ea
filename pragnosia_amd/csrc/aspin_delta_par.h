// The delta rule's scan with only the state's own recurrence along the chunks, for few heads over many chunks. Included
// by aspin_delta.hip inside its namespace, whose inverse, chunk-local backward and slot sums it shares.
//
// The one-workgroup-per-scan kernels of aspin_delta.hip walk a chunk in 3 to 6 us (its inverse, scores, outputs or
// gradients beside the state), so 44 heads of 32 chunks take 105 us forward and 160 backward on 44 of 256 compute
// units. Here everything that does not need the running state is formed for all chunks at once, and the walk itself,
// independent per value column given X, is spread over four workgroups a scan, 16 columns each:
//     forward   X (aspin_delta_inv);  walk: U = K S, rhs = beta o (V - e^L o U), W = X rhs, S <- a S + K^T (w o W)
//               (delta_walk);  O = A W + e^L o (Q S) (delta_out)
//     backward  Y = A^T dO, F = (Q o e^L)^T dO (delta_bwd_pre);  walk: dW = Y + w o (K G), drhs = X^T dW,
//               G <- a G + F - K^T (beta e^L o drhs) (delta_bwd_walk);  the row sums of drhs (delta_bwd_rsum);
//               aspin_delta_bwd_local
// with the operations, roundings and sums of the one-workgroup kernels: outputs, states, W and X are theirs bit for
// bit, and so are the gradients at head dim 128, whose one-workgroup backward is the same two kernels' work. At head
// dim 64 that backward is one fused kernel that rounds the same operands but sums some gradients in another order; they
// agree to bf16 rounding. Y, F and drhs pass through memory in fp32.
//
// A walking workgroup is bound by what one compute unit draws from memory (about 37 bytes a ns): a wave per 16 columns
// with the scan's four in one workgroup moved 56 KB a chunk and took 1.5 us over it whatever the arithmetic. One wave
// walks, four copy K, X and V's 16 columns of the next chunks to LDS through registers loaded walk_ahead chunks before
// their use; 22 KB a chunk (K and X from the L2 that the scan's other workgroups share). One barrier a chunk. A chunk
// takes 0.7 us, of which the copies alone 0.55; the walking wave is next, bound by its own issue.
// B4 H11 T2048 D64: forward 105 -> 55 us, backward 161 -> 82; B2 H12 T8192: 392 -> 137, 627 -> 215; B3 H6 T1000 D128:
// 52 -> 41, 86 -> 74. Carried windows (B2 H12 T8192, 16 of 512): 158 us as affine maps of all windows and their prefix
// (pragnosia_aspin_delta_window_maps / _prefix) -> 139; B16 H12 T1024, 2 of 512: 152 -> 94; with few heads and long
// sequences the maps are the faster ones (4 heads of 131072 in windows of 2048: 335 against 1502).

// In workgroup numbering, the sub-items (value quarters, halves) of a head or (head, chunk) lie 8 apart: workgroup i
// runs on XCD i mod 8, so they share one L2.
struct Sub {
  int item, sub;
};
PGN_DEVICE Sub sub_of(int idx, int per) {
  const int r = idx >> 3;
  return Sub{(r / per) * 8 + (idx & 7), r % per};
}
inline unsigned sub_grid(int64_t n, int per) { return (unsigned)((n + 7) / 8 * 8 * per); }

constexpr int VP = 20;  // pitch of V's 16 columns in LDS
constexpr int kParVals = 16 * 64 * 4;  // floats of Y or drhs of a (scan, chunk): [quarter][token block][lane][4]
template <int KH, bool BWD>
constexpr int walk_elems() { return (KH + 1) * TILE + (BWD ? 0 : 64 * VP); }
template <int KH, bool BWD>
constexpr int walk_bytes() { return walk_elems<KH, BWD>() * 2 + 4 * C * 4 + (BWD ? (KH + 1) * 4096 : 0); }
// (the tiles, then L, e^L, w, beta, and backward Y's and F's 16 columns)
template <int KH, bool BWD>
constexpr int walk_out_bytes() { return 2 * KH * 1024 + (BWD ? 0 : 4096); }  // the state as operands, W as accumulators
template <int KH, bool BWD>
constexpr int walk_lds() { return 2 * (walk_bytes<KH, BWD>() + walk_out_bytes<KH, BWD>()); }
template <int KH>
constexpr int walk_ahead() { return KH == 1 ? 6 : 4; }

// The copying waves (thread b of 256): chunk `it` of the walk into LDS buffer it & 1 in the turn before the walking
// wave uses it, from the register set loaded walk_ahead turns earlier; and the state and W that it left in the turn
// before from LDS to memory (wave b / 64 key block and token block b / 64), which it would otherwise spend a third of
// its issue slots on. Barriers: one before the walk, then one a turn, the turns rounded up to whole rounds of the sets
// (spare ones copy the last chunk again and store nothing): with no condition inside a turn, each copy waits for its
// own set's loads only.
template <int KH, bool BWD>
PGN_DEVICE void walk_copies(const __bf16* __restrict__ k, const __bf16* __restrict__ v, const __bf16* __restrict__ X,
                            const float* __restrict__ la, const float* __restrict__ be, __bf16* __restrict__ states,
                            __bf16* __restrict__ W, const float* yb, const float* __restrict__ fb,
                            unsigned char* smem, const DeltaRows<KH>& R, int qt, int T, int NC, int b,
                            const WaveIdx& x) {
  constexpr int DKEY = 64 * KH, A = walk_ahead<KH>();
  struct Set {
    bf16x8 k[KH][2], x[2], v;
    f32x4 y, f[KH];
    float la, be;
  } r[A];
  auto load = [&](Set& s, int it) {
    const int c = BWD ? max(NC - 1 - it, 0) : min(it, NC - 1), t0 = c * C, nr = min(C, T - t0);
#pragma unroll
    for (int h = 0; h < KH; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        s.k[h][u] = load_seg(k + R.rows(T) + (size_t)t0 * DKEY + 64 * h, nr, b + 256 * u, DKEY);
#pragma unroll
    for (int u = 0; u < 2; ++u) s.x[u] = load_seg(X + ((size_t)R.hw * NC + c) * C * C, C, b + 256 * u);
    if constexpr (!BWD) {  // row b / 2, 16-byte half b % 2 of the 16 columns (threads 128 apart copy the same)
      const __amdgpu_buffer_rsrc_t vr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(v + R.vals(T) + (size_t)t0 * DKEY), (short)0,
                                            nr * DKEY * (int)sizeof(__bf16), 0x00020000);
      const int at = (((b & 127) >> 1) * DKEY + 16 * qt + 8 * (b & 1)) * (int)sizeof(__bf16);
      s.v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(vr, at, 0, 0));
    }
    if constexpr (BWD) {
      s.y = *reinterpret_cast<const f32x4*>(yb + (size_t)c * kParVals + 4 * b);
#pragma unroll
      for (int h = 0; h < KH; ++h)
        s.f[h] = *reinterpret_cast<const f32x4*>(fb + (size_t)c * (KH * kParVals) + 1024 * h + 4 * b);
    }
    s.la = load_f32_lane(la + R.tok(T) + t0, nr, x.l);
    s.be = load_f32_lane(be + R.tok(T) + t0, nr, x.l);
  };
  auto put = [&](const Set& s, int it) {
    __bf16* tiles = reinterpret_cast<__bf16*>(smem + (it & 1) * walk_bytes<KH, BWD>());
    float* vec = reinterpret_cast<float*>(tiles + walk_elems<KH, BWD>());
#pragma unroll
    for (int h = 0; h < KH; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u) put_seg(tiles + h * TILE, s.k[h][u], b + 256 * u);
#pragma unroll
    for (int u = 0; u < 2; ++u) put_seg(tiles + KH * TILE, s.x[u], b + 256 * u);
    if constexpr (!BWD) {
      __bf16* p = tiles + (KH + 1) * TILE + ((b & 127) >> 1) * VP + 8 * (b & 1);
      *reinterpret_cast<bf16x4*>(p) = __builtin_shufflevector(s.v, s.v, 0, 1, 2, 3);
      *reinterpret_cast<bf16x4*>(p + 4) = __builtin_shufflevector(s.v, s.v, 4, 5, 6, 7);
    }
    if constexpr (BWD) {
      f32x4* yf = reinterpret_cast<f32x4*>(vec + 4 * C) + b;
      yf[0] = s.y;
#pragma unroll
      for (int h = 0; h < KH; ++h) yf[256 * (h + 1)] = s.f[h];
    }
    // every copying wave forms the same decays (no branch in a turn)
    chunk_decays(s.la, x.l, vec, vec + C, vec + 2 * C);
    vec[3 * C + x.l] = s.be;
  };
  const int cw = x.w - 1;
  auto drain = [&](int it) {  // what turn `it` left (nothing where there is no such turn: empty ranges)
    const bool ok = it >= 0 && it < NC;
    const int c = BWD ? NC - 1 - it : it, t0 = ok ? c * C : 0;
    const unsigned char* out = smem + 2 * walk_bytes<KH, BWD>() + (it & 1) * walk_out_bytes<KH, BWD>();
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        states + R.stateT(NC, ok ? c : 0), (short)0, ok ? DK * DKEY * (int)sizeof(__bf16) : 0, 0x00020000);
#pragma unroll
    for (int h = 0; h < KH; ++h) {
      const int db = 4 * h + cw;
      const i32x2 sv = *reinterpret_cast<const i32x2*>(out + (db >> 1) * 1024 + 16 * x.l + 8 * (db & 1));
      // row j holds key rows d contiguously
      const int at = ((16 * qt + x.i) * DKEY + 16 * db + 4 * x.g) * (int)sizeof(__bf16);
      __builtin_amdgcn_raw_buffer_store_b64(sv, sr, at, 0, 0);
    }
    if constexpr (!BWD) {
      const f32x4 wv = *reinterpret_cast<const f32x4*>(out + 2 * KH * 1024 + cw * 1024 + 16 * x.l);
      const __amdgpu_buffer_rsrc_t wr =
          __builtin_amdgcn_make_buffer_rsrc(W + R.vals(T) + (size_t)t0 * DKEY, (short)0,
                                            ok ? min(C, T - t0) * DKEY * (int)sizeof(__bf16) : 0, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, quad_rows(wv, x.i)), wr,
                                            ((16 * cw + 4 * x.g + (x.i & 3)) * DKEY + 16 * qt + 4 * (x.i >> 2)) *
                                                (int)sizeof(__bf16), 0, 0);
    }
  };
#pragma unroll
  for (int a = 0; a < A; ++a) load(r[a], a);
  put(r[0], 0);
  load(r[0], A);
  __syncthreads();
  for (int it0 = 0; it0 <= NC; it0 += A) {
#pragma unroll
    for (int a = 0; a < A; ++a) {  // turn it0 + a copies the next chunk, held by set (a + 1) % A
      drain(it0 + a - 1);
      put(r[(a + 1) % A], it0 + a + 1);
      load(r[(a + 1) % A], it0 + a + 1 + A);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);  // a later turn's decays are not formed (and their loads awaited) in this one
    }
  }
}
// The walking wave's share of the spare turns' barriers (at least one: the last chunk's state and W are stored in it)
template <int KH>
PGN_DEVICE void spare_turns(int n) {
  for (int it = n; it == n || it % walk_ahead<KH>() != 0; ++it) __syncthreads();
}
// The values, loaded by now: a load still in flight at a loop's entry would be waited for in every iteration
template <int N>
PGN_DEVICE void settle(f32x4 (&v)[N]) {
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[n][e] = pin_use(v[n][e]);
}

// ------------------------------------------------------------------------------------------------------------------
// forward, walk: 5 waves per (scan, 16 value columns). WIN: the state is rebased by -shift theta (key-row pairs
// rotated) after every `per` chunks but the last (carried windows).
template <int KH, bool WIN>
__global__ __launch_bounds__(320) void delta_walk(const __bf16* __restrict__ k, const __bf16* __restrict__ v,
                                                  const float* __restrict__ la, const float* __restrict__ be,
                                                  const __bf16* __restrict__ X, const float* __restrict__ S0,
                                                  __bf16* __restrict__ W, __bf16* __restrict__ sent,
                                                  float* __restrict__ Sfin, const float* __restrict__ theta,
                                                  float shift, int per, int H, int T, int NC, int heads) {
  constexpr int DKEY = 64 * KH;
  extern __shared__ __align__(16) unsigned char smem[];
  const WaveIdx x = wave_idx();
  const int g = x.g, i = x.i;
  const Sub u = sub_of(blockIdx.x, 4 * KH);
  if (u.item >= heads) return;  // grid padding (uniform over the workgroup, before any barrier)
  const int qt = u.sub & 3;
  const DeltaRows<KH> R(u.item * KH + (u.sub >> 2));
  if (x.w > 0) {
    walk_copies<KH, false>(k, v, X, la, be, sent, W, nullptr, nullptr, smem, R, qt, T, NC, threadIdx.x - 64, x);
    return;
  }
  const int j = 16 * qt + i;
  f32x4 S[4 * KH];
  {
    const __amdgpu_buffer_rsrc_t sv = f32_view(S0 ? S0 + R.state() : nullptr, DKEY * DKEY);
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[db][r] = load_f32(sv, (16 * db + 4 * g + r) * DKEY + j);
  }
  float cs[WIN ? 8 * KH : 1], sn[WIN ? 8 * KH : 1];
  if constexpr (WIN) {
#pragma unroll
    for (int p = 0; p < 8 * KH; ++p)
      sincosf(-shift * theta[(R.hw % H) * (DKEY / 2) + 8 * (p >> 1) + 2 * g + (p & 1)], &sn[p], &cs[p]);
  }
  settle(S);
  __syncthreads();
  int left = per;  // chunks to the window's end
  for (int c = 0; c < NC; ++c) {
    const int t0 = c * C;
    const __bf16* Ks = reinterpret_cast<const __bf16*>(smem + (c & 1) * walk_bytes<KH, false>());
    const __bf16 *Xs = Ks + KH * TILE, *Vs = Xs + TILE;
    const float* vec = reinterpret_cast<const float*>(Ks + walk_elems<KH, false>());
    const float *Ls = vec, *eLs = vec + C, *ws = vec + 2 * C, *bs = vec + 3 * C;
    // the turn's LDS operands in two bursts, each ahead of the products that it feeds, so the latency is paid once a
    // burst (backward walk, B4 H11 T2048: 32 us with the reads beside their products, 25 so)
    bf16x8 kf[4][2 * KH], xf[4][2];
    f32x4 vv[4], bv[4], ev[4], wv[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
#pragma unroll
      for (int m = 0; m < 2 * KH; ++m) kf[tb][m] = frag(Ks + (m >> 1) * TILE, 16 * tb + i, m & 1, g);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      vv[tb] = to_f32x4(ds_read_tr(Vs + (16 * tb + 4 * g + (i >> 2)) * VP + 4 * (i & 3)));
      bv[tb] = *reinterpret_cast<const f32x4*>(bs + 16 * tb + 4 * g);
      ev[tb] = *reinterpret_cast<const f32x4*>(eLs + 16 * tb + 4 * g);
    }
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      xf[tb][0] = frag(Xs, 16 * tb + i, 0, g);
      if (tb >= 2) xf[tb][1] = frag(Xs, 16 * tb + i, 1, g);
      wv[tb] = *reinterpret_cast<const f32x4*>(ws + 16 * tb + 4 * g);
    }
    const float a_c = __expf(Ls[C - 1]);
    bf16x8 sp[2 * KH];  // the state as operands: key rows 32 m .. 32 m + 31
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) sp[m] = pack(S[2 * m], S[2 * m + 1]);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 rhs[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      f32x4 U = zero4();
#pragma unroll
      for (int m = 0; m < 2 * KH; ++m) U = pgn_mfma(kf[tb][m], sp[m], U);
#pragma unroll
      for (int r = 0; r < 4; ++r) rhs[tb][r] = bv[tb][r] * (vv[tb][r] - ev[tb][r] * U[r]);
    }
    const bf16x8 r01 = pack(rhs[0], rhs[1]), r23 = pack(rhs[2], rhs[3]);
    bf16x8 kt[4 * KH][2];
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
      for (int m = 0; m < 2; ++m) kt[db][m] = frag_tr(Ks + (db >> 2) * TILE, 16 * (db & 3), m, g, i);
    unsigned char* out = smem + 2 * walk_bytes<KH, false>() + (c & 1) * walk_out_bytes<KH, false>() + 16 * x.l;
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) *reinterpret_cast<bf16x8*>(out + m * 1024) = sp[m];
    __builtin_amdgcn_sched_barrier(0);
    f32x4 Wt[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      Wt[tb] = pgn_mfma(xf[tb][0], r01, zero4());
      if (tb >= 2) Wt[tb] = pgn_mfma(xf[tb][1], r23, Wt[tb]);
    }
    bf16x8 ww[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) ww[m] = pack(Wt[2 * m] * wv[2 * m], Wt[2 * m + 1] * wv[2 * m + 1]);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) *reinterpret_cast<f32x4*>(out + 2 * KH * 1024 + tb * 1024) = Wt[tb];
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db) {
      S[db] = S[db] * a_c;
      S[db] = pgn_mfma(kt[db][0], ww[0], S[db]);
      S[db] = pgn_mfma(kt[db][1], ww[1], S[db]);
    }
    if constexpr (WIN) {
      if (--left == 0 && c + 1 < NC) {  // uniform
        left = per;
#pragma unroll
        for (int p = 0; p < 8 * KH; ++p) {
          const int r = 2 * (p & 1);
          const float s0 = S[p >> 1][r], s1 = S[p >> 1][r + 1];
          S[p >> 1][r] = s0 * cs[p] - s1 * sn[p];
          S[p >> 1][r + 1] = s0 * sn[p] + s1 * cs[p];
        }
      }
    }
    __syncthreads();
  }
  spare_turns<KH>(NC);
#pragma unroll
  for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) Sfin[R.state() + (size_t)(16 * db + 4 * g + r) * DKEY + j] = S[db][r];
}

// ------------------------------------------------------------------------------------------------------------------
// forward, finish: four waves per (scan, chunk); the scores by token block, then 16 value columns a wave
template <int KH>
__global__ __launch_bounds__(256) void delta_out(const __bf16* __restrict__ q, const __bf16* __restrict__ k,
                                                     const float* __restrict__ la, const __bf16* __restrict__ W,
                                                     const __bf16* __restrict__ sent, __bf16* __restrict__ o, int T,
                                                     int NC, int nhc) {
  constexpr int DKEY = 64 * KH, NT = 3 * KH + 1;
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* tiles = reinterpret_cast<__bf16*>(smem);
  const __bf16 *Qs = tiles, *Ks = tiles + KH * TILE, *Ss = tiles + 2 * KH * TILE, *Ws = tiles + 3 * KH * TILE;
  __bf16* As = tiles + NT * TILE;
  float *Ls = reinterpret_cast<float*>(As + TILE), *eLs = Ls + C, *ws = eLs + C;
  const WaveIdx x = wave_idx();
  const int w = x.w, g = x.g, i = x.i, tid = threadIdx.x;
  const Sub u_ = sub_of(blockIdx.x, KH);
  const int hc = u_.item, vh = u_.sub;
  if (hc >= nhc) return;
  const int hw = hc / NC, c = hc - hw * NC, t0 = c * C, nr = min(C, T - t0);
  const DeltaRows<KH> R(hw * KH + vh);
  const size_t roff = R.rows(T) + (size_t)t0 * DKEY, voff = R.vals(T) + (size_t)t0 * DKEY, toff = R.stateT(NC, c);
  bf16x8 sg[NT][2];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const __bf16* src = u < KH       ? q + roff + 64 * u
                        : u < 2 * KH ? k + roff + 64 * (u - KH)
                        : u < 3 * KH ? sent + toff + 64 * (u - 2 * KH)
                                     : W + voff;
    const int rows = (u >= 2 * KH && u < 3 * KH) ? DK : nr;
    sg[u][0] = load_seg(src, rows, tid, DKEY);
    sg[u][1] = load_seg(src, rows, tid + 256, DKEY);
  }
  const float lav = load_f32_lane(la + R.tok(T) + t0, nr, x.l);
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    put_seg(tiles + u * TILE, sg[u][0], tid);
    put_seg(tiles + u * TILE, sg[u][1], tid + 256);
  }
  if (w == 0) chunk_decays(lav, x.l, Ls, eLs, ws);
  __syncthreads();
  {
    const int t = 16 * w + i;
    bf16x8 qf[2 * KH];
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) qf[m] = frag(Qs + (m >> 1) * TILE, t, m & 1, g);
    const float Lt = Ls[t];
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      f32x4 sc = zero4();
      if (sb <= w) {  // uniform
#pragma unroll
        for (int m = 0; m < 2 * KH; ++m) sc = pgn_mfma(frag(Ks + (m >> 1) * TILE, 16 * sb + i, m & 1, g), qf[m], sc);
        const f32x4 Lsv = *reinterpret_cast<const f32x4*>(Ls + 16 * sb + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[r] *= masked_decay(Lt - Lsv[r], 16 * sb + 4 * g + r <= t);
      }
      store_T(As, 16 * w, 16 * sb, g, i, sc);
    }
  }
  __syncthreads();
  const __amdgpu_buffer_rsrc_t o_out =
      __builtin_amdgcn_make_buffer_rsrc(o + voff, (short)0, nr * DKEY * (int)sizeof(__bf16), 0x00020000);
  const bf16x8 w01 = frag_tr(Ws, 16 * w, 0, g, i), w23 = frag_tr(Ws, 16 * w, 1, g, i);
  bf16x8 sp[2 * KH];
#pragma unroll
  for (int m = 0; m < 2 * KH; ++m) sp[m] = frag(Ss + (m >> 1) * TILE, 16 * w + i, m & 1, g);
#pragma unroll
  for (int tb = 0; tb < 4; ++tb) {
    const int tl = 16 * tb + i;
    f32x4 acc = pgn_mfma(w01, frag(As, tl, 0, g), zero4());
    if (tb >= 2) acc = pgn_mfma(w23, frag(As, tl, 1, g), acc);
    f32x4 qs = zero4();
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) qs = pgn_mfma(sp[m], frag(Qs + (m >> 1) * TILE, tl, m & 1, g), qs);
    acc += eLs[tl] * qs;
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, to_bf16x4(acc)), o_out,
                                          (tl * DKEY + 16 * w + 4 * g) * (int)sizeof(__bf16), 0, 0);
  }
}
template <int KH>
constexpr size_t out_smem() { return (3 * KH + 2) * TILE * sizeof(__bf16) + 3 * C * sizeof(float); }

// ------------------------------------------------------------------------------------------------------------------
// backward, prepare: four waves per (head, chunk). A^T as in aspin_delta_bwd_chain.
template <int KH>
__global__ __launch_bounds__(256) void delta_bwd_pre(const __bf16* __restrict__ q, const __bf16* __restrict__ k,
                                                        const float* __restrict__ la, const __bf16* __restrict__ dO,
                                                     float* __restrict__ y, float* __restrict__ F, int T, int NC) {
  constexpr int DKEY = 64 * KH, NT = 3 * KH;
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* tiles = reinterpret_cast<__bf16*>(smem);
  const __bf16 *Qs = tiles, *Ks = tiles + KH * TILE, *Os = tiles + 2 * KH * TILE;
  __bf16* AT = tiles + NT * TILE;
  float *Ls = reinterpret_cast<float*>(AT + TILE), *eLs = Ls + C, *ws = eLs + C;
  const WaveIdx x = wave_idx();
  const int w = x.w, g = x.g, i = x.i, tid = threadIdx.x;
  const int hw = blockIdx.x / NC, c = blockIdx.x - hw * NC, t0 = c * C, nr = min(C, T - t0);
  const size_t row0 = (size_t)hw * T + t0;
  bf16x8 sg[NT][2];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const __bf16* src = u < KH       ? q + row0 * DKEY + 64 * u
                        : u < 2 * KH ? k + row0 * DKEY + 64 * (u - KH)
                                     : dO + row0 * DKEY + 64 * (u - 2 * KH);
    sg[u][0] = load_seg(src, nr, tid, DKEY);
    sg[u][1] = load_seg(src, nr, tid + 256, DKEY);
  }
  const float lav = load_f32_lane(la + row0, nr, x.l);
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    put_seg(tiles + u * TILE, sg[u][0], tid);
    put_seg(tiles + u * TILE, sg[u][1], tid + 256);
  }
  if (w == 0) chunk_decays(lav, x.l, Ls, eLs, ws);
  __syncthreads();
  {
    const int t = 16 * w + i;
    bf16x8 kf[2 * KH];
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) kf[m] = frag(Ks + (m >> 1) * TILE, t, m & 1, g);
    const float Lt = Ls[t];
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      f32x4 sc = zero4();
      if (sb >= w) {  // uniform
#pragma unroll
        for (int m = 0; m < 2 * KH; ++m) sc = pgn_mfma(frag(Qs + (m >> 1) * TILE, 16 * sb + i, m & 1, g), kf[m], sc);
        const f32x4 Lsv = *reinterpret_cast<const f32x4*>(Ls + 16 * sb + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[e] *= masked_decay(Lsv[e] - Lt, 16 * sb + 4 * g + e >= t);
      }
      store_T(AT, 16 * w, 16 * sb, g, i, sc);
    }
  }
  __syncthreads();  // A^T complete
#pragma unroll
  for (int vh = 0; vh < KH; ++vh) {
    const size_t sc = (size_t)(hw * KH + vh) * NC + c;
    const bf16x8 oc0 = frag_tr(Os + vh * TILE, 16 * w, 0, g, i), oc1 = frag_tr(Os + vh * TILE, 16 * w, 1, g, i);
    float* yo = y + sc * kParVals + w * 1024 + 4 * x.l;
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      f32x4 acc = zero4();
      if (tb < 2) acc = pgn_mfma(frag(AT, 16 * tb + i, 0, g), oc0, acc);
      acc = pgn_mfma(frag(AT, 16 * tb + i, 1, g), oc1, acc);
      *reinterpret_cast<f32x4*>(yo + tb * 256) = acc;
    }
    const bf16x8 oe0 = scale_frag_k(oc0, *reinterpret_cast<const f32x4*>(eLs + 4 * g),
                                    *reinterpret_cast<const f32x4*>(eLs + 16 + 4 * g));
    const bf16x8 oe1 = scale_frag_k(oc1, *reinterpret_cast<const f32x4*>(eLs + 32 + 4 * g),
                                    *reinterpret_cast<const f32x4*>(eLs + 48 + 4 * g));
    float* fo = F + (sc * 4 + w) * (KH * 1024) + 4 * x.l;
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db) {
      const __bf16* Qh = Qs + (db >> 2) * TILE;
      f32x4 acc = pgn_mfma(frag_tr(Qh, 16 * (db & 3), 0, g, i), oe0, zero4());
      acc = pgn_mfma(frag_tr(Qh, 16 * (db & 3), 1, g, i), oe1, acc);
      *reinterpret_cast<f32x4*>(fo + db * 256) = acc;
    }
  }
}
template <int KH>
constexpr size_t bwd_pre_smem() { return (3 * KH + 1) * TILE * sizeof(__bf16) + 3 * C * sizeof(float); }

// backward, walk: as the forward's, chunks in reverse. drhs replaces Y in place (fp32); the state gradients leave as
// bf16, transposed, as the chunk-local kernel reads them.
template <int KH>
__global__ __launch_bounds__(320) void delta_bwd_walk(const __bf16* __restrict__ k, const float* __restrict__ la,
                                                      const float* __restrict__ be, const __bf16* __restrict__ X,
                                                      float* y, const float* __restrict__ F,
                                                      const float* __restrict__ dSfin, __bf16* __restrict__ dSc,
                                                      float* __restrict__ dS0, int T, int NC, int heads) {
  constexpr int DKEY = 64 * KH;
  extern __shared__ __align__(16) unsigned char smem[];
  const WaveIdx x = wave_idx();
  const int g = x.g, i = x.i;
  const Sub u = sub_of(blockIdx.x, 4 * KH);
  if (u.item >= heads) return;  // grid padding (uniform over the workgroup, before any barrier)
  const int qt = u.sub & 3, bh = u.item * KH + (u.sub >> 2);
  const DeltaRows<KH> R(bh);
  float* yb = y + (size_t)bh * NC * kParVals + qt * 1024;
  if (x.w > 0) {
    walk_copies<KH, true>(k, nullptr, X, la, be, dSc, nullptr, yb, F + ((size_t)bh * NC * 4 + qt) * (KH * 1024), smem,
                          R, qt, T, NC, threadIdx.x - 64, x);
    return;
  }
  const int j = 16 * qt + i;
  f32x4 G[4 * KH];
  {
    const __amdgpu_buffer_rsrc_t gv = f32_view(dSfin ? dSfin + R.state() : nullptr, DKEY * DKEY);
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) G[db][r] = load_f32(gv, (16 * db + 4 * g + r) * DKEY + j);
  }
  settle(G);
  __syncthreads();
  for (int it = 0; it < NC; ++it) {
    const int c = NC - 1 - it;
    const __bf16* Ks = reinterpret_cast<const __bf16*>(smem + (it & 1) * walk_bytes<KH, true>());
    const __bf16* Xs = Ks + KH * TILE;
    const float* vec = reinterpret_cast<const float*>(Ks + walk_elems<KH, true>());
    const float *Ls = vec, *eLs = vec + C, *ws = vec + 2 * C, *bs = vec + 3 * C;
    const f32x4* yf = reinterpret_cast<const f32x4*>(vec + 4 * C) + x.l;
    bf16x8 kf[4][2 * KH], xf[4][2];
    f32x4 wv[4], ev[4], bv[4], yv[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
#pragma unroll
      for (int m = 0; m < 2 * KH; ++m) kf[tb][m] = frag(Ks + (m >> 1) * TILE, 16 * tb + i, m & 1, g);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      wv[tb] = *reinterpret_cast<const f32x4*>(ws + 16 * tb + 4 * g);
      yv[tb] = yf[64 * tb];
      if (tb < 2) xf[tb][0] = frag_tr(Xs, 16 * tb, 0, g, i);
      xf[tb][1] = frag_tr(Xs, 16 * tb, 1, g, i);
    }
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      bv[tb] = *reinterpret_cast<const f32x4*>(bs + 16 * tb + 4 * g);
      ev[tb] = *reinterpret_cast<const f32x4*>(eLs + 16 * tb + 4 * g);
    }
    const float a_c = __expf(Ls[C - 1]);
    bf16x8 gp[2 * KH];
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) gp[m] = pack(G[2 * m], G[2 * m + 1]);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 dW[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      f32x4 p = zero4();
#pragma unroll
      for (int m = 0; m < 2 * KH; ++m) p = pgn_mfma(kf[tb][m], gp[m], p);
      dW[tb] = yv[tb] + wv[tb] * p;
    }
    const bf16x8 w01 = pack(dW[0], dW[1]), w23 = pack(dW[2], dW[3]);
    bf16x8 kt[4 * KH][2];
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
      for (int m = 0; m < 2; ++m) kt[db][m] = frag_tr(Ks + (db >> 2) * TILE, 16 * (db & 3), m, g, i);
    unsigned char* out = smem + 2 * walk_bytes<KH, true>() + (it & 1) * walk_out_bytes<KH, true>() + 16 * x.l;
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) *reinterpret_cast<bf16x8*>(out + m * 1024) = gp[m];
    __builtin_amdgcn_sched_barrier(0);
    f32x4 dU[4], dr[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      f32x4 acc = zero4();
      if (tb < 2) acc = pgn_mfma(xf[tb][0], w01, acc);
      acc = pgn_mfma(xf[tb][1], w23, acc);
      dr[tb] = acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) dU[tb][r] = -bv[tb][r] * ev[tb][r] * acc[r];
    }
    const bf16x8 u01 = pack(dU[0], dU[1]), u23 = pack(dU[2], dU[3]);
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db) {
      f32x4 acc = G[db] * a_c + yf[256 + 64 * db];
      acc = pgn_mfma(kt[db][0], u01, acc);
      G[db] = pgn_mfma(kt[db][1], u23, acc);
    }
    float* yo = yb + (size_t)c * kParVals + 4 * x.l;
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) *reinterpret_cast<f32x4*>(yo + tb * 256) = dr[tb];
    __syncthreads();
  }
  spare_turns<KH>(NC);
  if (dS0) {
#pragma unroll
    for (int db = 0; db < 4 * KH; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) dS0[R.state() + (size_t)(16 * db + 4 * g + r) * DKEY + j] = G[db][r];
  }
}

// backward, the row sums that the decay and strength gradients need, from drhs in fp32 (sum_j drhs (V - e^L U) and
// -beta sum_j drhs U with U = K S_c, as aspin_delta_bwd_chain forms them), and drhs as bf16 rows for the chunk-local
// kernel. Four waves per (scan, chunk), 16 value columns a wave.
template <int KH>
__global__ __launch_bounds__(256) void delta_bwd_rsum(const __bf16* __restrict__ k, const __bf16* __restrict__ v,
                                                      const float* __restrict__ la, const float* __restrict__ be,
                                                      const __bf16* __restrict__ sent, const float* __restrict__ y,
                                                      __bf16* __restrict__ drhs, float* __restrict__ rsum, int T,
                                                      int NC, int nhc) {
  constexpr int DKEY = 64 * KH, NT = 2 * KH + 1;
  __shared__ __align__(16) __bf16 tiles[NT * TILE];
  __shared__ __align__(16) float Ls[C], eLs[C], ws[C], redV[4 * C], redU[4 * C];
  const __bf16 *Ks = tiles, *Ss = tiles + KH * TILE, *Vs = tiles + 2 * KH * TILE;
  const WaveIdx x = wave_idx();
  const int w = x.w, g = x.g, i = x.i, tid = threadIdx.x;
  const Sub u_ = sub_of(blockIdx.x, KH);
  const int hc = u_.item, vh = u_.sub;
  if (hc >= nhc) return;
  const int hw = hc / NC, c = hc - hw * NC, t0 = c * C, nr = min(C, T - t0), scan = hw * KH + vh;
  const DeltaRows<KH> R(scan);
  const size_t roff = R.rows(T) + (size_t)t0 * DKEY, voff = R.vals(T) + (size_t)t0 * DKEY, toff = R.stateT(NC, c);
  bf16x8 sg[NT][2];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const __bf16* src = u < KH ? k + roff + 64 * u : u < 2 * KH ? sent + toff + 64 * (u - KH) : v + voff;
    const int rows = (u >= KH && u < 2 * KH) ? DK : nr;
    sg[u][0] = load_seg(src, rows, tid, DKEY);
    sg[u][1] = load_seg(src, rows, tid + 256, DKEY);
  }
  const float* yb = y + ((size_t)scan * NC + c) * kParVals + w * 1024 + 4 * x.l;
  f32x4 dr[4];
#pragma unroll
  for (int tb = 0; tb < 4; ++tb) dr[tb] = *reinterpret_cast<const f32x4*>(yb + tb * 256);
  const float lav = load_f32_lane(la + R.tok(T) + t0, nr, x.l), bev = load_f32_lane(be + R.tok(T) + t0, nr, x.l);
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    put_seg(tiles + u * TILE, sg[u][0], tid);
    put_seg(tiles + u * TILE, sg[u][1], tid + 256);
  }
  if (w == 0) chunk_decays(lav, x.l, Ls, eLs, ws);
  const __amdgpu_buffer_rsrc_t out =
      __builtin_amdgcn_make_buffer_rsrc(drhs + voff, (short)0, nr * DKEY * (int)sizeof(__bf16), 0x00020000);
#pragma unroll
  for (int tb = 0; tb < 4; ++tb)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, quad_rows(dr[tb], i)), out,
                                          ((16 * tb + 4 * g + (i & 3)) * DKEY + 16 * w + 4 * (i >> 2)) *
                                              (int)sizeof(__bf16), 0, 0);
  __syncthreads();
  bf16x8 sf[2 * KH];
#pragma unroll
  for (int m = 0; m < 2 * KH; ++m) sf[m] = frag(Ss + (m >> 1) * TILE, 16 * w + i, m & 1, g);
#pragma unroll
  for (int tb = 0; tb < 4; ++tb) {
    f32x4 U = zero4();
#pragma unroll
    for (int m = 0; m < 2 * KH; ++m) U = pgn_mfma(frag(Ks + (m >> 1) * TILE, 16 * tb + i, m & 1, g), sf[m], U);
    const f32x4 vv = to_f32x4(ds_read_tr(Vs + (16 * tb + 4 * g + (i >> 2)) * kPitch + 16 * w + 4 * (i & 3)));
    float pr[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pr[e] = dr[tb][e] * vv[e];
      pr[4 + e] = dr[tb][e] * U[e];
    }
    const float tot = row_totals16x8(pr, i);
    ((i & 8) ? redU : redV)[w * C + 16 * tb + 4 * g + ((i >> 1) & 3)] = tot;
  }
  __syncthreads();
  if (w == 0) {
    const int t = x.l;
    const float pv = redV[t] + redV[C + t] + redV[2 * C + t] + redV[3 * C + t];
    const float pu = redU[t] + redU[C + t] + redU[2 * C + t] + redU[3 * C + t];
    if (t < nr) {
      rsum[((size_t)scan * T + t0 + t) * 2 + 0] = pv - eLs[t] * pu;
      rsum[((size_t)scan * T + t0 + t) * 2 + 1] = -bev * pu;
    }
  }
}
