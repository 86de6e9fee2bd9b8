// Block-mask composition into the row bitmask (FS_MASK_WORDS words per row)
// (reference: attn_src/fft_attn/my_attn_v7.py:542-550 prior, :558-560 last
// row, :588-612 stripe/diffuse dynamic mask, :256-294 qk top-k, :623-641
// columns; attn_src/fix_mask_attn/my_attn.py:39-79 for the fixed mask).
//
// One launch serves every head.  Each workgroup (8 waves) decides from diag_var
// which heads are stripe and which diffuse, and takes its share of their rows.
// N <= 8192.
//
// Stripe / fixed rows (Nk <= 4096) are built word-parallel: a lane forms the
// 64-bit membership mask of 64 key blocks (range masks for the prior, columns
// and causal limit; a funnel-shifted window of the bit-reversed lag mask for
// the lag diagonals) and stores it as word w of the row.
//
// A diffuse head's rows are taken panel_rows at a time (16 at N <= 1024): the
// workgroup forms
// the scores S[rows][0 .. last row] with MFMA tiles of 16 keys x 16 query rows
// (v_mfma_f32_16x16x32 for 16-bit inputs, v_mfma_f32_16x16x4 for fp32, so
// products and sums are fp32 as in a scalar dot product), stores them in LDS
// as order-preserving keys, and each wave then finds the k_i-th largest key
// of a row by bisection: ballot counts over the row's keys, held in registers
// at N <= 1024, ending as soon as a candidate splits off exactly k_i keys
// (about 20 of the 32 steps; only a tie at the threshold takes all 32).
// What bounds it: the bisection's compares (16 per step and row at N = 1024)
// and the latency of one load round.  64 KiB of LDS, two workgroups per CU.
// The scalar form before it (each thread one key block, 2-byte loads of a row
// per thread, 64 rows per workgroup in serial passes, 32 steps re-reading
// LDS) took 481, 841 and 3498 us for 8 diffuse heads of 32 at N = 64, 256 and
// 1024 (bf16, D = 128), and 444 us for one of 4 at N = 64 in fp32; this one 13,
// 16, 41 and 13 us.
#include <algorithm>

#include "common.h"

namespace fs {

constexpr int kSelThreads = 512;
constexpr int kSelWaves = kSelThreads / 64;
constexpr int kMaxWords = 64;                       // word-parallel path: Nk <= 4096
constexpr int kSelMaxN = 8192;
constexpr int kHeadGroup = 64;                      // heads per row of the grid: their decisions fit one lane mask
constexpr int kMaxGrid = 512;                       // workgroups per head group: two (64 KiB each) on each of 256 CUs
constexpr int kPanelRows = 16;                      // an MFMA tile's query rows: the most a panel holds
constexpr int kPanelWords = 16 * 1024;              // keys of a panel: 64 KiB, the default LDS limit of a launch
constexpr int kRegWords = 16;                       // 64-key words of a row held in registers (N <= 1024)

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// acc += A B^T of a 16-byte chunk per lane: lane l holds row l & 15 of both
// operands, chunk l >> 4 of the step's four
template <typename T> struct PanelMma;
template <> struct PanelMma<bf16_t> {
  static __device__ __forceinline__ f32x4_t go(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
};
template <> struct PanelMma<f16_t> {
  static __device__ __forceinline__ f32x4_t go(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
  }
};
template <> struct PanelMma<float> {
  // element e of every lane's chunk is one K = 4 step (the dims are added in another order)
  static __device__ __forceinline__ f32x4_t go(uint4 a, uint4 b, f32x4_t c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
  }
};

// elements d .. d + 16 / sizeof(T) - 1 of a row of D (0 past D, or when !ok); the
// row itself is readable either way.  WIDE: rows are 16-byte aligned and D a
// multiple of the chunk; the load is unconditional (clamped), so that the
// loads of several chunks are in flight together.
template <typename T, bool WIDE>
__device__ __forceinline__ uint4 row_chunk(const T* row, int d, int D, bool ok) {
  constexpr int V = 16 / sizeof(T);
  if constexpr (WIDE) {
    uint4 v = *reinterpret_cast<const uint4*>(row + (d < D ? d : 0));
    const uint32_t keep = ok && d < D ? ~0u : 0u;
    return make_uint4(v.x & keep, v.y & keep, v.z & keep, v.w & keep);
  } else {
    T e[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const T v = row[d + i < D ? d + i : 0];
      e[i] = ok && d + i < D ? v : T{0};
    }
    return __builtin_bit_cast(uint4, e);
  }
}

// Score panel of a diffuse head's rows r0 .. r0 + nrows - 1 (nrows <= 16) against keys 0 .. r0 + nrows - 1:
// S[i][j] = (q_b[i] . k_b[j]) * (1/sqrt(D)) (:234-249), as order-preserving keys.  Key j of row rr is word
// (chunk j / 4, swizzled by the row) of the row's `stride` words: the 16 rows' chunk stores of one tile fall
// on different banks, a row's 64 consecutive keys on 64 different ones.
template <typename T, bool WIDE>
__device__ __forceinline__ void score_panel(const T* qb, const T* kb, int D, int r0, int nrows, float inv_sqrt_d,
                                            uint32_t* panel, int stride, int lane) {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int kSteps = 128 / (4 * V);            // MFMA steps per 128 dims (dims past D are zero)
  constexpr int kTiles = !WIDE ? 1 : (sizeof(T) == 2 ? 4 : 2);   // key tiles in flight per wave
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int jmax = r0 + nrows, ntile = (jmax + 15) >> 4;
  const bool qok = l16 < nrows;
  const T* qrow = qb + (int64_t)(r0 + (qok ? l16 : 0)) * D;
  for (int t0 = wave * kTiles; t0 < ntile; t0 += kSelWaves * kTiles) {
    f32x4_t acc[kTiles];
#pragma unroll
    for (int u = 0; u < kTiles; ++u) acc[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int d0 = 0; d0 < D; d0 += 128) {
      uint4 qv[kSteps], kv[kTiles][kSteps];
#pragma unroll
      for (int st = 0; st < kSteps; ++st) qv[st] = row_chunk<T, WIDE>(qrow, d0 + (4 * st + g) * V, D, qok);
#pragma unroll
      for (int u = 0; u < kTiles; ++u) {
        const int j = (t0 + u) * 16 + l16;
        const T* krow = kb + (int64_t)min(j, jmax - 1) * D;   // keys past the last row: read, never counted
#pragma unroll
        for (int st = 0; st < kSteps; ++st) kv[u][st] = row_chunk<T, WIDE>(krow, d0 + (4 * st + g) * V, D, true);
      }
      // the query chunks are whole before the chains start: selected between the
      // MFMAs, they made the register allocator move an accumulator mid-chain
#pragma unroll
      for (int st = 0; st < kSteps; ++st) asm volatile("" : "+v"(qv[st].x), "+v"(qv[st].y), "+v"(qv[st].z), "+v"(qv[st].w));
#pragma unroll
      for (int st = 0; st < kSteps; ++st)
#pragma unroll
        for (int u = 0; u < kTiles; ++u) acc[u] = PanelMma<T>::go(kv[u][st], qv[st], acc[u]);
    }
    // a fixed wait between the chain and the first read of its results, whatever path leads here
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // lane: keys 16 t + 4 g .. + 3 of query row l16
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      const int c = (t0 + u) * 4 + g;              // 4-key chunk of the row
      if (t0 + u < ntile && qok) {
        uint32_t w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = order_key(acc[u][r] * inv_sqrt_d);
        *reinterpret_cast<uint4*>(panel + l16 * stride + (c ^ l16) * 4) = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  }
}

// LDS of the word-parallel path (the start of the launch's dynamic LDS)
struct WordRowsLds {
  uint64_t rkw[2 * kMaxWords + 2];                  // bit x: keep_tau[N-1-x] (x < N), 0 beyond
  uint64_t colw[kMaxWords], lastw[kMaxWords];
  uint32_t fk[4096 / 4], fc[4096 / 4], fl[4096 / 4];   // the staged flag bytes
};

// bits of word w (blocks 64w .. 64w+63) that lie in [lo, hi)
__device__ __forceinline__ uint64_t range_bits(int w, int lo, int hi) {
  const int b0 = max(lo - 64 * w, 0), b1 = min(hi - 64 * w, 64);
  if (b1 <= b0) return 0;
  const uint64_t upto = b1 == 64 ? ~0ull : ((1ull << b1) - 1);
  return upto & ~((1ull << b0) - 1);
}

// Rows r0 .. r0 + RPW - 1 of a stripe head or of a fixed mask (every thread of the workgroup).
__device__ void stripe_rows_of(const fs_select_args& a, int h, int r0, int RPW, unsigned char* sel_lds) {
  const int N = a.N, Nk = a.Nk;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));                    // keeps the lane's addresses out of the item loop's preheader
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NW = (Nk + 63) >> 6;
  const bool words = NW <= kMaxWords;              // built word-parallel
  const bool use_lags = a.dyn_mode == 1, use_cols = a.col_mode != 0;
  // The word-parallel path stages the head's lag / column / last-row flags:
  // bytes j = 4 w .. 4 w + 3 of word w = tid + 512 u, every load before the first wait.
  constexpr int kFlagWords = 4096 / 4 / kSelThreads;
  uint32_t fkr[kFlagWords], fcr[kFlagWords], flr[kFlagWords];
  const int nw4 = (N + 3) >> 2;
  if (words) {
    const int64_t hb = (int64_t)h * N;
    const bool v4 = (N & 3) == 0;                  // row starts 4-byte aligned (buffers are)
#pragma unroll
    for (int u = 0; u < kFlagWords; ++u) {
      const int w4 = tid + u * kSelThreads;
      fkr[u] = fcr[u] = flr[u] = 0;
      if (w4 >= nw4) continue;
      if (v4) {
        if (a.keep_tau) fkr[u] = reinterpret_cast<const uint32_t*>(a.keep_tau + hb)[w4];
        if (a.col_sel) fcr[u] = reinterpret_cast<const uint32_t*>(a.col_sel + hb)[w4];
        if (a.last_sel) flr[u] = reinterpret_cast<const uint32_t*>(a.last_sel + hb)[w4];
      } else {
        for (int b = 0; b < 4 && 4 * w4 + b < N; ++b) {
          const int64_t j = hb + 4 * w4 + b;
          if (a.keep_tau) fkr[u] |= (uint32_t)a.keep_tau[j] << (8 * b);
          if (a.col_sel) fcr[u] |= (uint32_t)a.col_sel[j] << (8 * b);
          if (a.last_sel) flr[u] |= (uint32_t)a.last_sel[j] << (8 * b);
        }
      }
    }
  }

  const int lw = a.local_window;
  const bool has_last = a.last_sel != nullptr;
  if (words) {
    // ---- word-parallel rows: lane (row g, word w) builds the membership of
    // blocks 64w .. 64w+63 of its row as a 64-bit mask from per-head masks
    // staged in LDS and stores it as word w of the row; the row's count is
    // the sum of its words' popcounts.
    WordRowsLds& wl = *reinterpret_cast<WordRowsLds*>(sel_lds);
    uint64_t* rkw = wl.rkw;
    uint64_t* colw = wl.colw;
    uint64_t* lastw = wl.lastw;
    uint32_t* fk = wl.fk;
    uint32_t* fc = wl.fc;
    uint32_t* fl = wl.fl;
#pragma unroll
    for (int u = 0; u < kFlagWords; ++u) {
      const int w4 = tid + u * kSelThreads;
      if (w4 < nw4) {
        fk[w4] = fkr[u];
        fc[w4] = fcr[u];
        fl[w4] = flr[u];
      }
    }
    __syncthreads();
    auto flag = [](const uint32_t* f, int j) { return ((f[j >> 2] >> (8 * (j & 3))) & 255u) != 0; };
    for (int q = wave; q < 2 * NW + 2; q += kSelWaves) {
      const int x = 64 * q + lane;
      const bool kb = use_lags && x < N && flag(fk, N - 1 - x);
      const uint64_t m = __ballot(kb);
      if (lane == 0) rkw[q] = m;
      if (q < NW) {
        const bool cb = use_cols && x < N && flag(fc, x);
        const bool lb = has_last && x < N && flag(fl, x);
        const uint64_t mc = __ballot(cb), ml = __ballot(lb);
        if (lane == 0) {
          colw[q] = mc;
          lastw[q] = ml;
        }
      }
    }
    __syncthreads();
    int lpr = 1;                                   // lanes per row (power of two >= NW)
    while (lpr < NW) lpr <<= 1;
    const int rpi = 64 / lpr;                      // rows per wave pass
    const int w = lane & (lpr - 1), g = lane / lpr;
    for (int rr0 = wave * rpi; rr0 < RPW; rr0 += kSelWaves * rpi) {
      const int rr = rr0 + g;
      const int i = r0 + rr;
      const bool row_ok = rr < RPW && i < N;
      uint64_t m = 0;
      if (row_ok && w < NW) {
        const int jlim = a.mask_causal ? min(i + 1, Nk) : Nk;
        // prior (:83-95): sink | recent | local window
        m = range_bits(w, 0, a.keep_sink) | range_bits(w, Nk - a.keep_recent, Nk);
        if (lw > 0) m |= range_bits(w, i - lw, i + lw + 1);
        if (has_last && i == N - 1) m |= lastw[w];
        if (use_lags) {
          // bit b <-> lag t = i - 64w - b <-> rkw bit p0 + b, p0 = N-1-i+64w >= 0
          const int p0 = N - 1 - i + 64 * w;
          const int qw = p0 >> 6, sh = p0 & 63;
          uint64_t win = rkw[qw] >> sh;
          if (sh) win |= rkw[qw + 1] << (64 - sh);
          m |= win & range_bits(w, a.keep_sink, i - a.remote_start + 1);   // t >= rs, j >= keep_sink
        }
        if (use_cols) m |= colw[w] & range_bits(w, 0, i + 1);
        m &= range_bits(w, 0, jlim);
      }
      int c = __popcll(m);
      for (int o = lpr >> 1; o > 0; o >>= 1) c += __shfl_xor(c, o, lpr);
      if (row_ok) {
        if (w < NW) a.blk_bits[((int64_t)h * N + i) * NW + w] = m;
        if (w == 0) a.blk_cnt[(int64_t)h * N + i] = c;
      }
    }
    return;
  }
  // ---- per-head lag / column / last-row flags, staged in LDS (bit 0 lag, 1 column, 2 last row)
  uint8_t* flags = sel_lds;
  for (int j = tid; j < N; j += kSelThreads) {
    uint8_t f = 0;
    if (a.keep_tau && a.keep_tau[(int64_t)h * N + j]) f |= 1;
    if (a.col_sel && a.col_sel[(int64_t)h * N + j]) f |= 2;
    if (a.last_sel && a.last_sel[(int64_t)h * N + j]) f |= 4;
    flags[j] = f;
  }
  __syncthreads();
  const int nrows = min(RPW, N - r0);
  for (int rr = wave; rr < nrows; rr += kSelWaves) {
    const int i = r0 + rr;
    const int jlim = a.mask_causal ? min(i + 1, Nk) : Nk;
    // ---- membership in ascending block order, one word per 64 blocks
    uint64_t* out = a.blk_bits + ((int64_t)h * N + i) * NW;
    int cnt = 0;
    for (int j0 = 0; j0 < jlim; j0 += 64) {
      const int j = j0 + lane;
      bool in = false;
      if (j < jlim) {
        // prior (:83-95): sink | recent | local window
        in = j < a.keep_sink || j >= Nk - a.keep_recent || (lw > 0 && abs(i - j) <= lw);
        const uint8_t fj = j < N ? flags[j] : 0;
        if (has_last && i == N - 1 && (fj & 4)) in = true;
        if (use_lags) {
          const int t = i - j;
          if (t >= a.remote_start && j >= a.keep_sink && (flags[t] & 1)) in = true;
        }
        if (use_cols && j <= i && (fj & 2)) in = true;
      }
      const uint64_t m = __ballot(in);
      if (lane == 0) out[j0 >> 6] = m;
      cnt += __popcll(m);
    }
    for (int w = ((jlim + 63) >> 6) + lane; w < NW; w += 64) out[w] = 0ull;   // words past the causal limit
    if (lane == 0) a.blk_cnt[(int64_t)h * N + i] = cnt;
  }
}

// Rows r0 .. r0 + panel_rows - 1 of a diffuse head (every thread of the workgroup).
template <typename T>
__device__ void diffuse_rows(const fs_select_args& a, int h, int r0, int panel_rows, float inv_sqrt_d,
                             uint32_t* panel) {
  const int N = a.N, Nk = a.Nk, D = a.D, hk = h / (a.Hq / a.Hk);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));                   // keeps the lane's addresses out of the item loop's preheader
  const int NW = (Nk + 63) >> 6;
  const int lw = a.local_window;
  const bool has_last = a.last_sel != nullptr, use_cols = a.col_mode == 2;
  const int stride = (N + 63) & ~63;
  const int nrows = min(panel_rows, N - r0);
  const T* qb = static_cast<const T*>(a.q_b) + (int64_t)h * N * D;
  const T* kb = static_cast<const T*>(a.k_b) + (int64_t)hk * N * D;
  if (D % (16 / (int)sizeof(T)) == 0 && (((uintptr_t)a.q_b | (uintptr_t)a.k_b) & 15) == 0)
    score_panel<T, true>(qb, kb, D, r0, nrows, inv_sqrt_d, panel, stride, lane);
  else
    score_panel<T, false>(qb, kb, D, r0, nrows, inv_sqrt_d, panel, stride, lane);
  __syncthreads();
  for (int rr = wave; rr < nrows; rr += kSelWaves) {
    const int i = r0 + rr, n = i + 1, nw = (n + 63) >> 6;
    const uint32_t* srow = panel + rr * stride;
    auto key_at = [&](int j) -> uint32_t { return srow[((j >> 2) ^ rr) * 4 + (j & 3)]; };   // j < n rounded up to 64
    // ---- the k_i-th largest of S[i][0..i] (:271-276).  Keys past the row are 0, below every candidate.
    int k = (int)((float)n * a.qk_topk_ratio);
    k = min(max(k, 1), n);
    uint32_t x[kRegWords];
    const bool held = nw <= kRegWords;
    if (held) {
#pragma unroll
      for (int u = 0; u < kRegWords; ++u) x[u] = 64 * u + lane < n ? key_at(64 * u + lane) : 0u;
    }
    // keys >= cand (cand > 0), over whole groups of four words
    auto count_ge = [&](uint32_t cand) -> int {
      int c = 0;
      if (held) {
#pragma unroll
        for (int q = 0; q < kRegWords / 4; ++q) {
          if (4 * q >= nw) break;
#pragma unroll
          for (int u = 4 * q; u < 4 * q + 4; ++u) c += wave_count(x[u] >= cand);
        }
      } else {
        const int full = n >> 6;                   // words with every key in the row
        int u0 = 0;
        for (; u0 + 8 <= full; u0 += 8) {          // eight reads in flight
          uint32_t y[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) y[u] = key_at(64 * (u0 + u) + lane);
#pragma unroll
          for (int u = 0; u < 8; ++u) c += wave_count(y[u] >= cand);
        }
        for (; u0 < full; ++u0) c += wave_count(key_at(64 * u0 + lane) >= cand);
        if (full < nw) c += wave_count(64 * full + lane < n && key_at(64 * full + lane) >= cand);
      }
      return c;
    };
    // thr: every larger key is selected, and the first `need` keys equal to it
    uint32_t thr = 0;
    int need = 0;
    bool split = false;                            // a candidate split off exactly k keys: no ties to rank
    for (int b = 31; b >= 0 && !split; --b) {
      const uint32_t cand = thr | (1u << b);
      const int c = count_ge(cand);
      if (c >= k) thr = cand;
      split = c == k;
    }
    if (split) thr -= 1;
    else need = k - (thr == 0xffffffffu ? 0 : count_ge(thr + 1));
    // ---- the row's words, word w0 + l kept by lane l: the top-k ballots, then (word-parallel) the prior
    // (:83-95), the last row's and the columns' words
    const int jlim = a.mask_causal ? min(n, Nk) : Nk;
    uint64_t* out = a.blk_bits + ((int64_t)h * N + i) * NW;
    const bool extra = use_cols || (has_last && i == N - 1);
    int cnt = 0, eq_seen = 0;
    for (int w0 = 0; w0 < NW; w0 += 64) {
      uint32_t mlo = 0, mhi = 0;
      auto put = [&](int w, uint64_t m) {          // |= m in lane w - w0
        if (lane == w - w0) {
          mlo |= (uint32_t)m;
          mhi |= (uint32_t)(m >> 32);
        }
      };
      for (int w = w0; w < min(nw, w0 + 64); ++w) {
        const int j = 64 * w + lane;
        const uint32_t key = j < n ? key_at(j) : 0u;
        bool in = key > thr;
        if (need > 0) {
          const bool eq = j < n && key == thr;
          const uint64_t me = __ballot(eq);
          in = in || (eq && eq_seen + rank_below(me) < need);
          eq_seen += __popcll(me);
        }
        put(w, __ballot(in));
      }
      if (extra) {
        for (int w = w0; w < min(NW, w0 + 64); ++w) {
          const int j = 64 * w + lane;
          bool in = has_last && i == N - 1 && j < N && a.last_sel[(int64_t)h * N + j] != 0;
          if (use_cols && j < n) in = in || a.col_sel[(int64_t)h * N + j] != 0;
          put(w, __ballot(in));
        }
      }
      const int w = w0 + lane;
      uint64_t m = (uint64_t)mhi << 32 | mlo;
      m |= range_bits(w, 0, a.keep_sink) | range_bits(w, Nk - a.keep_recent, Nk);
      if (lw > 0) m |= range_bits(w, i - lw, i + lw + 1);
      m &= range_bits(w, 0, jlim);
      if (w < NW) {
        out[w] = m;
        cnt += __popcll(m);
      }
    }
    cnt = wave_sum_i(cnt);
    if (lane == 0) a.blk_cnt[(int64_t)h * N + i] = cnt;
  }
}

// The head group's work, dealt to the launch's workgroups.  blockIdx.y: heads
// 64 blockIdx.y ..; every workgroup decides its group's heads (each wave some of
// them), so the items -- panel_rows rows of a diffuse head, the latest rows (the
// longest) first, then stripe_rows rows of a stripe or fixed head -- are
// enumerated without a list in memory, and workgroup b takes items b, b +
// gridDim.x, ..  (One workgroup per panel_rows rows of every head instead, the
// stripe heads' spare ones returning: 21.6 against 10.1 us on 32 stripe heads of
// 1024 blocks, the 64 KiB workgroups going through four rounds.)
// Dynamic LDS (all there is, so that the panel's 64 KiB are a whole default
// launch): the decisions, then WordRowsLds (word-parallel rows), the head's flag
// bytes [N] (other stripe rows), or the panel [panel_rows][N rounded up to 64] of keys.
template <typename T>
__global__ __launch_bounds__(kSelThreads) __attribute__((amdgpu_waves_per_eu(4))) void select_kernel(
    fs_select_args a, int stripe_rows, int panel_rows, float inv_sqrt_d) {
  extern __shared__ __attribute__((aligned(16))) unsigned char sel_lds[];
  uint8_t* is_diffuse = sel_lds;                   // [kHeadGroup], before the first item
  const int N = a.N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: what follows from it branches on scalars
  const int h0 = blockIdx.y * kHeadGroup, nh = min(kHeadGroup, a.Hq - h0);

  // ---- stripe / diffuse decisions (:359-363): wave w takes heads w, w + 8, .., four at a time
  uint64_t dmask = 0;                              // bit e: head h0 + e is diffuse
  if (a.dyn_mode == 1) {
    for (int e0 = wave; e0 < nh; e0 += 4 * kSelWaves) {
      float s[4] = {0.f, 0.f, 0.f, 0.f};
      if (!a.stripe_all_diffuse) {
        for (int i = lane; i < a.n_samples; i += 64) {
          float d[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            d[u] = a.diag_var[(int64_t)(h0 + min(e0 + u * kSelWaves, nh - 1)) * a.n_samples + i];
#pragma unroll
          for (int u = 0; u < 4; ++u) s[u] += d[u];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = e0 + u * kSelWaves;
        s[u] = wave_sum(s[u]);
        const float mv = a.stripe_all_diffuse ? INFINITY : s[u] / (float)a.n_samples;
        const bool stripe = mv <= a.stripe_threshold && !a.stripe_all_diffuse;   // false for nan
        if (lane == 0 && e < nh) {
          is_diffuse[e] = stripe ? 0 : 1;
          if (blockIdx.x == 0) {
            if (a.mean_var) a.mean_var[h0 + e] = mv;
            if (a.is_stripe) a.is_stripe[h0 + e] = stripe ? 1 : 0;
          }
        }
      }
    }
    __syncthreads();
    dmask = __ballot(lane < nh && is_diffuse[lane] != 0);
    __syncthreads();                               // read before the items overwrite it
  }
  const uint64_t hmask = nh == 64 ? ~0ull : (1ull << nh) - 1;
  const int nd = __popcll(dmask), ns = nh - nd;
  const int dchunks = (N + panel_rows - 1) / panel_rows, schunks = (N + stripe_rows - 1) / stripe_rows;
  const int ditems = nd * dchunks, items = ditems + ns * schunks;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    if (item != (int)blockIdx.x) __syncthreads();  // the previous item's LDS is read
    // The arguments are read anew for each item: held over the loop they cost 77
    // spilled scalar registers and scratch memory (stripe heads only, 32 of 256
    // blocks 5.8 -> 5.6 us, 512 6.6 -> 5.8; fp32, 1 diffuse head of 4 of 64 16.0 -> 12.9)
    typedef const __attribute__((address_space(4))) fs_select_args* argp;
    argp ap = (argp)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ap));
    const fs_select_args b = *(const fs_select_args*)ap;
    if (item < ditems) {
      diffuse_rows<T>(b, h0 + nth_set_bit(dmask, item % nd), (dchunks - 1 - item / nd) * panel_rows, panel_rows,
                      inv_sqrt_d, reinterpret_cast<uint32_t*>(sel_lds));
    } else {
      const int it = item - ditems, e = it / schunks;
      stripe_rows_of(b, h0 + nth_set_bit(hmask & ~dmask, e), (it - e * schunks) * stripe_rows, stripe_rows, sel_lds);
    }
  }
}

template <typename T>
static int launch_select(const fs_select_args& a, dim3 grid, size_t smem, int stripe_rows, int panel_rows,
                         float inv_sqrt_d, hipStream_t s) {
  if (int rc = fs_host::allow_dynamic_lds(select_kernel<T>, smem, "fs_select")) return rc;
  select_kernel<T><<<grid, kSelThreads, smem, s>>>(a, stripe_rows, panel_rows, inv_sqrt_d);
  return 0;
}

}  // namespace fs

using namespace fs;

extern "C" int fs_select(const fs_select_args* a, void* stream) {
  FS_CHECK_ARG(a != nullptr, "fs_select: null args");
  FS_CHECK_ARG(a->blk_cnt && a->blk_bits, "fs_select: null output");
  FS_CHECK_ARG(((uintptr_t)a->blk_bits & 7) == 0, "fs_select: blk_bits must be 8-byte aligned");
  FS_CHECK_ARG(a->Hq > 0 && a->Hk > 0 && a->Hq % a->Hk == 0, "fs_select: bad head counts");
  FS_CHECK_ARG(a->N >= 1 && a->Nk >= 1 && a->Nk <= 65535, "fs_select: bad block counts");
  FS_CHECK_ARG(a->dyn_mode == 0 || a->dyn_mode == 1, "fs_select: bad dyn_mode");
  FS_CHECK_ARG(a->col_mode >= 0 && a->col_mode <= 2, "fs_select: bad col_mode");
  FS_CHECK_ARG(a->dyn_mode == 0 || (a->q_b && a->k_b && a->keep_tau &&
                                    (a->stripe_all_diffuse || (a->diag_var && a->n_samples > 0))),
               "fs_select: dynamic mask inputs missing");
  FS_CHECK_ARG(a->col_mode == 0 || a->col_sel, "fs_select: col_sel missing");
  FS_CHECK_ARG(a->col_mode != 1 || a->dyn_mode == 1, "fs_select: col_mode 1 needs dyn_mode 1");
  FS_CHECK_ARG((a->dyn_mode == 0 && a->col_mode == 0 && a->last_sel == nullptr) || a->N == a->Nk,
               "fs_select: dynamic, column and last-row masks need N == Nk");
  FS_CHECK_SUPPORTED(a->N <= kSelMaxN && (a->dyn_mode == 0 || a->D <= 256), "fs_select: N=%d > %d or D=%d > 256",
                     a->N, kSelMaxN, a->D);
  // Rows of a stripe or fixed head's work item: 64 word-parallel rows of <= 1024
  // blocks (four rows per wave pass of 16 lanes each), fewer for longer rows; one
  // per wave on the per-row path.  Rows of a diffuse head's: what a 64 KiB panel
  // holds, at most one MFMA tile's 16.
  const int NW = (a->Nk + 63) / 64;
  const int stripe_rows = NW <= 16 ? 64 : (NW <= 32 ? 32 : (NW <= kMaxWords ? 16 : kSelWaves));
  int panel_rows = stripe_rows;
  size_t smem = ((size_t)a->N + 15) & ~(size_t)15;
  if (a->dyn_mode == 1) {
    const int stride = (a->N + 63) & ~63;
    panel_rows = kPanelRows;
    while (panel_rows * stride > kPanelWords) panel_rows >>= 1;   // 2 at N = 8192
    smem = std::max(smem, (size_t)panel_rows * stride * sizeof(uint32_t));
  }
  if (NW <= kMaxWords) smem = std::max(smem, sizeof(WordRowsLds));
  // the most items a head group can have: every head diffuse
  const int64_t items = (int64_t)std::min(a->Hq, kHeadGroup) * ((a->N + panel_rows - 1) / panel_rows);
  const dim3 grid((unsigned)std::min<int64_t>(items, kMaxGrid), (unsigned)((a->Hq + kHeadGroup - 1) / kHeadGroup));
  const float inv_sqrt_d = a->D > 0 ? 1.0f / (float)sqrt((double)a->D) : 1.0f;
  hipStream_t s = (hipStream_t)stream;
  const int dt = a->dyn_mode == 1 ? a->dtype : FS_DTYPE_F32;
  int rc = 0;
  fs_select_args k = *a;
  k.local_window = std::min(a->local_window, std::max(a->N, a->Nk));   // wider ones reach no further, and i + window overflows
  switch (dt) {
    case FS_DTYPE_F32: rc = launch_select<float>(k, grid, smem, stripe_rows, panel_rows, inv_sqrt_d, s); break;
    case FS_DTYPE_BF16: rc = launch_select<bf16_t>(k, grid, smem, stripe_rows, panel_rows, inv_sqrt_d, s); break;
    case FS_DTYPE_F16: rc = launch_select<f16_t>(k, grid, smem, stripe_rows, panel_rows, inv_sqrt_d, s); break;
    default: fs_host::set_error("fs_select: dtype %d unsupported", a->dtype); return FS_ERR_UNSUPPORTED;
  }
  if (rc) return rc;
  return fs_host::launch_status("fs_select");
}
