// Incremental decoding on a persistent moment state: what makes Fastmax generation O(1) per token.
//
// The causal kernel of the reference keeps running sums over the keys and adds one key per query
// (fastmax_cuda_forward.cu:160-276: the first nk - nq keys are summed before the first query, then one
// more per query).  Kept between calls, those sums are the whole memory of the sequence: a decoding step
// adds the new token's key and value to them and reads them out with the new query, without touching any
// earlier key (the reference's generation loop, transformer/eval.py:8-32, runs the whole context through the
// model for every new token).
//
// State of one batch*head, fp32, with k' = k * inv_tau and R = 1 + D (+ D (D + 1) / 2 for order 2) moment rows:
//     num [R][D]   row 0: sum v        rows 1 + m: sum k'_m v        rows 1 + D + pair(m, l): sum k'_m k'_l v,  m <= l
//     den [R]      the same sums with v replaced by 1 (row 0: the number of keys)
// The order-2 sums are symmetric in (m, l), so only the pairs m <= l are kept (2 080 of 4 096 rows at D = 64: a step
// reads and writes the state once, and this halves it), in row-major order of the upper triangle.
// Readout for a query q:  F = a0 num[0] + a1 sum_m q_m num[1+m] + a2 sum_{m<=l} w_ml q_m q_l num[1+D+pair(m,l)] with
// w_ml = 1 on the diagonal and 2 off it; g likewise from den, o = F / g.
//
// k_decode: grid (D / 4, bh), 512 threads, ONE launch per step.  A workgroup owns four value columns of every moment
// row (a contiguous [R][4] block of the state, 16-byte loads and stores) and a copy of the denominator column, so the
// sums over the rows that the readout needs (F of its four columns, and g) never leave the workgroup: no partial
// results in memory, no second launch, no fence.  A thread keeps its rows (every 512th) in registers, adds the new
// tokens one after the other (their k' and the four v columns staged through LDS), writes the rows back and, when a
// query is given (one new token), the workgroup adds up its part of the readout in a fixed order and stores its four
// outputs.  Bandwidth and latency bound: a step reads and writes the state once (the denominators once per
// workgroup: 5 floats per row and workgroup instead of 4).
//
// k_decode_absorb_mma, k_decode_absorb_f32 (further down): the same sums for a whole prompt with matrix instructions, one launch.
#pragma once
#include <type_traits>
#include "fm_kernels.h"

static constexpr int FM_DEC_ROWS = 64;      // the moment rows of a state are padded to a multiple of this
static constexpr int FM_DEC_THREADS = 512;  // eight wavefronts per workgroup: five rows per thread at D = 64, order 2 (per token: 256 threads 9.3 us, 384 7.7, 512 and 768 7.4, 1024 7.7)
constexpr int64_t fm_decode_rows(int d, bool quad) { return 1 + int64_t(d) + (quad ? int64_t(d) * (d + 1) / 2 : 0); }
constexpr int fm_decode_blocks(int d, bool quad) { return int((fm_decode_rows(d, quad) + FM_DEC_ROWS - 1) / FM_DEC_ROWS); }
// floats of one batch*head's state: per group of four value columns num [Rp][4] then den [Rp], Rp = R rounded up to whole blocks
constexpr int64_t fm_decode_rows_padded(int d, bool quad) { return int64_t(fm_decode_blocks(d, quad)) * FM_DEC_ROWS; }
inline int64_t fm_decode_state_floats(int d, bool quad) { return fm_decode_rows_padded(d, quad) * 5 * (d / 4); }

// the two key features a moment row multiplies (index DH stands for the constant 1) and how often the row counts in
// a readout (an order-2 row off the diagonal stands for the pairs (m, l) and (l, m))
template <int DH> FM_DEVICE void fm_decode_row(int r, bool quad, int& m, int& l, bool& live, float& mult) {
  live = true; mult = 1.0f;
  if (r == 0) { m = DH; l = DH; }
  else if (r <= DH) { m = r - 1; l = DH; }
  else if (quad && r < 1 + DH + DH * (DH + 1) / 2) {
    // pair index p -> (m, l), m <= l, rows of the upper triangle one after the other: row m starts at m D - m (m - 1) / 2
    // (m from the root of the quadratic, then one step either way against rounding)
    const int p = r - 1 - DH;
    m = int(0.5f * (float(2 * DH + 1) - fm_sqrtf(float((2 * DH + 1) * (2 * DH + 1) - 8 * p))));
    if (m < 0) m = 0;
    if (m > DH - 1) m = DH - 1;
    if (m * DH - m * (m - 1) / 2 > p) --m;
    else if (m + 1 < DH && (m + 1) * DH - (m + 1) * m / 2 <= p) ++m;
    l = m + (p - (m * DH - m * (m - 1) / 2));
    if (l != m) mult = 2.0f;
  } else { m = DH; l = DH; live = false; }
}

// A thread's rows of a workgroup's [R][4] block (every 512th) in registers, and the tokens added to them one after the other.
template <typename TIO, int DH> struct DecRows {
  static constexpr int TB = 16;                          // new tokens staged at a time
  static constexpr int NI = (int(fm_decode_rows(DH, true)) + FM_DEC_THREADS - 1) / FM_DEC_THREADS;   // rows per thread at most
  fm_f32x4 acc[NI];
  float dsum[NI], rmult[NI];
  int rm[NI], rl[NI];
  bool rlive[NI];
  FM_DEVICE void load(const float* num, const float* den, int R, bool quad, bool fresh, int tid) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = tid + FM_DEC_THREADS * i;
      rlive[i] = false; rm[i] = DH; rl[i] = DH; rmult[i] = 1.0f; dsum[i] = 0.f;
      acc[i] = fm_f32x4{0.f, 0.f, 0.f, 0.f};
      if (r < R) {
        if (!fresh) {
          acc[i] = *reinterpret_cast<const fm_f32x4*>(num + int64_t(r) * 4);
          dsum[i] = den[r];
        }
        fm_decode_row<DH>(r, quad, rm[i], rl[i], rlive[i], rmult[i]);
      }
    }
  }
  // ks: k' of the staged tokens, [DH] = 1; vs: their four value columns (16-byte aligned).  Begins with a barrier.
  FM_DEVICE void add(const TRef<const TIO>& k, const TRef<const TIO>& v, int bh, int c4, int n_new, float inv_tau, float (*ks)[DH + 1],
                     float (*vs)[4], int tid) {
    for (int t0 = 0; t0 < n_new; t0 += TB) {
      FM_SYNC();
      for (int i = tid; i < TB * (DH + 1); i += FM_DEC_THREADS) {
        const int t = i / (DH + 1), f = i % (DH + 1);
        float x = 0.f;
        if (t0 + t < n_new) x = f < DH ? IO<TIO>::ld(k.base(bh) + int64_t(t0 + t) * k.s_n + f) * inv_tau : 1.0f;
        ks[t][f] = x;
      }
      if (tid < TB * 4) {
        const int t = tid / 4, f = tid % 4;
        vs[t][f] = (t0 + t < n_new) ? IO<TIO>::ld(v.base(bh) + int64_t(t0 + t) * v.s_n + c4 + f) : 0.f;
      }
      FM_SYNC();
      const int nt = n_new - t0 < TB ? n_new - t0 : TB;
      for (int t = 0; t < nt; ++t) {
        const fm_f32x4 vc = *reinterpret_cast<const fm_f32x4*>(&vs[t][0]);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const float w = rlive[i] ? ks[t][rm[i]] * ks[t][rl[i]] : 0.f;
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] += w * vc[j];
          dsum[i] += w;
        }
      }
    }
  }
  FM_DEVICE void store(float* num, float* den, int R, int64_t Rp, bool fresh, int tid) const {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = tid + FM_DEC_THREADS * i;
      if (r < R) {
        *reinterpret_cast<fm_f32x4*>(num + int64_t(r) * 4) = acc[i];
        den[r] = dsum[i];
      }
    }
    if (fresh) {                                         // the padding behind the last row
      for (int64_t r = R + tid; r < Rp; r += FM_DEC_THREADS) {
        *reinterpret_cast<fm_f32x4*>(num + r * 4) = fm_f32x4{0.f, 0.f, 0.f, 0.f};
        den[r] = 0.f;
      }
    }
  }
};

template <typename TIO, int DH>
FM_GLOBAL void FM_LAUNCH_BOUNDS(FM_DEC_THREADS)
k_decode(TRef<const TIO> k, TRef<const TIO> v, TRef<const TIO> q, int n_new, int quad, float inv_tau, float a0,
         float a1, float a2, float* FM_RESTRICT state, TRef<TIO> o, TRef<float> g, int has_q, int fresh) {
  typedef DecRows<TIO, DH> W;
  FM_SHARED float ks[W::TB][DH + 1];
  FM_SHARED __attribute__((aligned(16))) float vs[W::TB][4];
  FM_SHARED float qs[DH + 1];
  FM_SHARED float red[FM_DEC_THREADS / 64][5];
  const int tid = FM_TID_X, cb = FM_BID_X, bh = FM_BID_Y, c4 = 4 * cb;
  const int R = int(fm_decode_rows(DH, quad != 0));
  const int64_t Rp = fm_decode_rows_padded(DH, quad != 0);
  float* num = state + (int64_t(bh) * (DH / 4) + cb) * Rp * 5;
  float* den = num + Rp * 4;
  W w;
  // the query travels with the state's rows (one memory latency for both)
  float qreg = 1.0f;
  if (has_q && tid < DH) qreg = IO<TIO>::ld(q.base(bh) + tid);
  w.load(num, den, R, quad != 0, fresh != 0, tid);
  if (has_q && tid <= DH) qs[tid] = qreg;             // read after the barriers of the token loop
  w.add(k, v, bh, c4, n_new, inv_tau, ks, vs, tid);
  w.store(num, den, R, Rp, fresh != 0, tid);
  if (!has_q) return;
  // readout of the new token's query: the thread's rows, then the wavefront (a butterfly: every lane ends with the
  // same sum), then the wavefronts in order
  if (n_new <= 0) FM_SYNC();                           // (no token: qs has not met a barrier yet)
  float f[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < W::NI; ++i) {
    const int r = tid + FM_DEC_THREADS * i;
    const float coef = r == 0 ? a0 : (r <= DH ? a1 : a2);
    const float x = w.rlive[i] ? coef * w.rmult[i] * qs[w.rm[i]] * qs[w.rl[i]] : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] += x * w.acc[i][j];
    f[4] += x * w.dsum[i];
  }
#pragma unroll
  for (int j = 0; j < 5; ++j) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) f[j] += fm_shfl_xor(f[j], m);
  }
  if ((tid & 63) == 0) {
#pragma unroll
    for (int j = 0; j < 5; ++j) red[tid >> 6][j] = f[j];
  }
  FM_SYNC();
  if (tid < 4) {
    // each of the four output threads adds its column and the denominator itself (one barrier less than a shared sum)
    float sum = 0.f, gs = 0.f;
#pragma unroll
    for (int i = 0; i < FM_DEC_THREADS / 64; ++i) { sum += red[i][tid]; gs += red[i][4]; }
    IO<TIO>::st(o.base(bh) + c4 + tid, sum / gs);
    if (tid == 0 && cb == 0) g.base(bh)[0] = gs;
  }
}

// ------------------------------------------------------------------------------
// Prompts: their keys and values added to the state with matrix instructions.  k_decode adds tokens one after the other on the
// vector units: 2 145 rows x 4 columns of multiply-adds per token and workgroup, 1.7 ms for 4 096 tokens at 16 batch*heads.
//
// grid (D / 4, bh), 512 threads: the workgroup owns the same [R][4] block of the state as in k_decode.  Two groups of four
// wavefronts take every other tile of tokens, wavefront w of a group the value column c = 4 cb + w: the slice
// sum_t v_tc k'_ta k'_tb of its column on the 32 x 32 tiles on and above the diagonal (it is symmetric in a, b).  What all four
// columns share is dealt by k-step: the denominators' order-2 sums, and the rows 0 .. D of numerators and denominators in one go
// as  sum_t z_tn' x_tn  with z = (k', then the rows of x) and x = (the four value columns, ones, zeros).  At the end the wavefronts'
// parts meet in LDS and are added in a fixed order, and every sum goes to the state in memory, added to what is there or (fresh) in
// its place: each address by exactly one lane, no atomics, the same bits every run.
//   k_decode_absorb_mma  bf16 tensors, D = 64, order 2: operands rounded to _Float16 (k', and the products v k'), fp32 sums
//   k_decode_absorb_f32  everything else: fp32 products (v_mfma_f32_32x32x2_f32)
// ------------------------------------------------------------------------------
static constexpr int FM_ABS_GROUPS = 2, FM_ABS_THREADS = FM_ABS_GROUPS * 256, FM_ABS_XR = 8;   // XR: rows of x
template <int DH, bool QUAD> struct AbsSums {
  static constexpr int NT = DH / 32;
  static constexpr int NP = QUAD ? NT * (NT + 1) / 2 : 0;        // pair tiles (a <= b): (0,0) or (0,0), (0,1), (1,1)
  static constexpr int NSH = NP + NT + 1;                        // shared: denominators of the pairs, rows 1 .. D, row 0
  // Tiles that meet in LDS at a time: few enough that LDS does not keep a second workgroup off a CU whose registers have room for it
  // (three everywhere: 98 KB; order 2, 128 heads of 32: 64 tokens 28.9 us, so 21.0, 128 tokens 36.6, so 28.6)
  static constexpr int RT = DH == 64 ? (QUAD ? 3 : 2) : 1;
  static constexpr size_t red_bytes() { return size_t(4) * FM_ABS_GROUPS * RT * 16 * 64 * 4; }
  static constexpr int pa(int i) { return i == 2 ? 1 : 0; }      // row tile and column tile of pair tile i
  static constexpr int pb(int i) { return i == 0 ? 0 : 1; }
};
// N elements of a caller's row as they lie in memory, in whole registers: loads that travel while other work is done wait for nothing
template <typename TIO, int N> struct Raw {
  static constexpr int NW = N * int(sizeof(TIO)) / 4;
  uint32_t w[NW];
  FM_DEVICE void zero() {
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = 0u;
  }
  FM_DEVICE void ld(const TIO* p) { __builtin_memcpy(w, p, sizeof(w)); }
  FM_DEVICE float get(int i) const {
    if (sizeof(TIO) == 4) return fm_bits_f32(w[i % NW]);
    return fm_bits_f32((i & 1) ? (w[i / 2] & 0xffff0000u) : (w[i / 2] << 16));
  }
};

// Everything accumulated -> state.  col: the wavefront's pair tiles, sh: its part of the shared sums; all LDS from red on is free.
template <int DH, bool QUAD, bool FRESH>
FM_DEVICE void fm_absorb_finish(const fm_f32x16* col, const fm_f32x16* sh, float* red, float* num, float* den) {
  typedef AbsSums<DH, QUAD> C;
  constexpr int NP = C::NP, NSH = C::NSH, NW = 4 * FM_ABS_GROUPS;
  const int lane = FM_TID_X & 63, lr = lane & 31, lh = lane >> 5;
  const int wave8 = FM_UNIFORM(FM_TID_X >> 6), wave = wave8 & 3, grp = wave8 >> 2;
  auto pair_row = [&](int a, int b) { return 1 + DH + a * DH - a * (a - 1) / 2 + (b - a); };
  // the value columns: entries (a, b) with a <= b go to their pair rows; group 0 writes accumulator entries 0 .. 7 of its
  // column's tiles, group 1 entries 8 .. 15 (16 rows further down), each with the other group's part from LDS.  Every state entry
  // is read before the first is written: as read-modify-writes one after the other they were up to 72 memory latencies in a row.
  if constexpr (NP > 0) {
    float old[NP][8];
    float* at[NP][8];
    bool live[NP][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ra = fm_acc_row(e, lh) + 16 * grp;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        live[i][e] = C::pa(i) != C::pb(i) || ra <= lr;
        at[i][e] = num + (live[i][e] ? int64_t(pair_row(32 * C::pa(i) + ra, 32 * C::pb(i) + lr)) * 4 + wave : wave);
        old[i][e] = FRESH ? 0.f : *at[i][e];
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) red[((wave8 * NP + i) * 8 + e) * 64 + lane] = grp ? col[i][e] : col[i][8 + e];
    FM_SYNC();
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float other = red[(((wave8 ^ 4) * NP + i) * 8 + e) * 64 + lane];
        if (live[i][e]) *at[i][e] = old[i][e] + ((grp ? other : col[i][e]) + (grp ? col[i][8 + e] : other));
      }
  }
  // the shared sums: the eight parts through LDS, RT tiles at a time; wavefront w adds entries 2 w and 2 w + 1 of every
  // tile in the order of the wavefronts
  constexpr int RT = C::RT, EPW = 16 / NW;
  float* sat[NSH][EPW];                                  // where they go; null: nowhere
  float sold[NSH][EPW];
#pragma unroll
  for (int i = 0; i < NSH; ++i)
#pragma unroll
    for (int x = 0; x < EPW; ++x) {
      const int ra = fm_acc_row(EPW * wave8 + x, lh);
      float* p = nullptr;
      if (i < NP) {                                      // denominators of the pair rows
        if (C::pa(i) != C::pb(i) || ra <= lr) p = den + pair_row(32 * C::pa(i) + ra, 32 * C::pb(i) + lr);
      } else if (i < NSH - 1) {                          // rows 1 + a: column n < 4 a numerator, n = 4 the denominator
        const int a = 32 * (i - NP) + ra;
        if (lr < 4) p = num + int64_t(1 + a) * 4 + lr;
        else if (lr == 4) p = den + 1 + a;
      } else if (ra == 4) {                              // row 0: the ones row of z against the columns of x
        if (lr < 4) p = num + lr;
        else if (lr == 4) p = den;
      }
      sat[i][x] = p;
      sold[i][x] = FRESH ? 0.f : *(p ? p : den);
    }
  if (FRESH) {
    // the padding behind the last row
    constexpr int R = int(fm_decode_rows(DH, QUAD)), RP = int(fm_decode_rows_padded(DH, QUAD));
    for (int r = R + FM_TID_X; r < RP; r += FM_ABS_THREADS) {
      *reinterpret_cast<fm_f32x4*>(num + int64_t(r) * 4) = fm_f32x4{0.f, 0.f, 0.f, 0.f};
      den[r] = 0.f;
    }
  }
#pragma unroll
  for (int i0 = 0; i0 < NSH; i0 += RT) {
    FM_SYNC();                                           // what lay there has been read
#pragma unroll
    for (int i = 0; i < RT; ++i)
      if (i0 + i < NSH) {
#pragma unroll
        for (int e = 0; e < 16; ++e) red[((wave8 * RT + i) * 16 + e) * 64 + lane] = sh[i0 + i][e];
      }
    FM_SYNC();
#pragma unroll
    for (int i = 0; i < RT; ++i)
      if (i0 + i < NSH) {
#pragma unroll
        for (int x = 0; x < EPW; ++x) {
          float sum = 0.f;
#pragma unroll
          for (int w = 0; w < NW; ++w) sum += red[((w * RT + i) * 16 + EPW * wave8 + x) * 64 + lane];
          float* p = sat[i0 + i][x];
          if (p) *p = sold[i0 + i][x] + sum;
        }
      }
  }
}

// Per tile of 128 tokens the keys (times inv_tau, as _Float16) are staged row-major and the four value columns, a row of ones (zero
// past the end of the prompt) and three rows of zeros as rows over the tokens.  Per k-step of 16 tokens a wavefront reads the two key
// fragments with transposing LDS reads and uses them as B operand and, times its value column's fragment, as A operand.
//
// What bounds it is latency: 16 batch*heads are one workgroup per CU, each a chain over the tiles (fetch, LDS, products); two groups
// halve it (LDS and 256 registers per lane leave no room for more).  The rows on their way to LDS wait in registers as they came:
// converted as they were loaded, they made every tile wait for its loads.
template <int DH> struct DecAbsCfg {
  typedef Mma<fm_half> M;
  static constexpr int TT = 128;                       // tokens per tile
  static constexpr int PQ = DH + M::PAD;               // pitch of the key rows
  static constexpr int XP = TT + M::PAD;
  static constexpr int TILE_E = TT * PQ + FM_ABS_XR * XP;
  static constexpr size_t lds_bytes() {
    const size_t st = size_t(FM_ABS_GROUPS) * 2 * TILE_E * 2, red = AbsSums<DH, true>::red_bytes();
    return st > red ? st : red;
  }
};

template <typename TIO, int DH, bool FRESH>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(FM_ABS_THREADS, 2)
k_decode_absorb_mma(TRef<const TIO> k, TRef<const TIO> v, int n_new, float inv_tau, float* FM_RESTRICT state) {
  static_assert(DH == 64, "two 32-row tiles per feature axis");
  typedef fm_half E;
  typedef Mma<E> M;
  typedef typename M::frag frag;
  typedef DecAbsCfg<DH> C;
  typedef AbsSums<DH, true> S;
  constexpr int TT = C::TT, PQ = C::PQ, XP = C::XP, NSTEP = TT / M::KSTEP, XR = FM_ABS_XR, NG = FM_ABS_GROUPS;
  FM_DYN_SMEM(smem);
  const int lane = FM_TID_X & 63, lr = lane & 31, lh = lane >> 5;
  const int wave8 = FM_UNIFORM(FM_TID_X >> 6), wave = wave8 & 3, grp = wave8 >> 2;
  const int tid = FM_TID_X & 255;                        // within the group
  E* const buf0 = reinterpret_cast<E*>(smem) + grp * 2 * C::TILE_E;
  E* const buf1 = buf0 + C::TILE_E;
  // the sixteen workgroups of a batch*head read the same keys: behind one L2 (145 -> 28 MB fetched for 4 096 tokens at 16 heads, 0.125 -> 0.097 ms)
  int cb, bh;
  fm_xcd_map(FM_GDIM_X, FM_GDIM_Y, cb, bh);
  const int c4 = 4 * cb;
  const int64_t Rp = fm_decode_rows_padded(DH, true);
  float* num = state + (int64_t(bh) * (DH / 4) + cb) * Rp * 5;
  float* den = num + Rp * 4;
  const TIO* kb = k.base(bh);
  const TIO* vb = v.base(bh);

  // global memory -> registers: a thread's four pieces of the key rows, and (threads below TT) a token's four values
  constexpr int CPR = DH / 8, NK = TT * CPR / 256;
  Raw<TIO, 8> kreg[NK];
  Raw<TIO, 4> vreg;
  auto fetch = [&](int t0) FM_ALWAYS_INLINE {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c = tid + 256 * i, row = t0 + c / CPR, f0 = (c % CPR) * 8;
      if (row < n_new) kreg[i].ld(kb + int64_t(row) * k.s_n + f0);
      else kreg[i].zero();
    }
    if (tid < TT) {
      if (t0 + tid < n_new) vreg.ld(vb + int64_t(t0 + tid) * v.s_n + c4);
      else vreg.zero();
    }
  };
  auto put = [&](E* b, int t0) FM_ALWAYS_INLINE {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c = tid + 256 * i;
      float sc[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sc[j] = kreg[i].get(j) * inv_tau;
      CE<E>::st8(b + (c / CPR) * PQ + (c % CPR) * 8, sc);
    }
    if (tid < TT) {
      E* x = b + TT * PQ + tid;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j * XP] = E(vreg.get(j));
      x[4 * XP] = E(t0 + tid < n_new ? 1.0f : 0.0f);
    }
  };
  const int g0 = grp * TT;                               // tiles past the end of the prompt are zeros
  fetch(g0);
  // rows 5 .. 7 of both buffers: zeros, written once
  for (int i = tid; i < 2 * 3 * XP; i += 256) {
    E* b = i < 3 * XP ? buf0 : buf1;
    b[TT * PQ + 5 * XP + (i % (3 * XP))] = E(0.0f);
  }

  fm_f32x16 col[S::NP], sh[S::NSH];                      // the wavefront's value column; its part of the shared sums
#pragma unroll
  for (int i = 0; i < S::NP; ++i) col[i] = fm_zero16();
#pragma unroll
  for (int i = 0; i < S::NSH; ++i) sh[i] = fm_zero16();

  put(buf0, g0);
  if (NG * TT < n_new) fetch(NG * TT + g0);
  FM_SYNC_LDS();
  int par = 0;
  for (int tb = 0; tb < n_new; tb += NG * TT) {
    const E* cbuf = par ? buf1 : buf0;
    const E* xt = cbuf + TT * PQ;
    if (tb + NG * TT < n_new) {
      put(par ? buf0 : buf1, tb + NG * TT + g0);
      if (tb + 2 * NG * TT < n_new) fetch(tb + 2 * NG * TT + g0);
    }
    if (tb + g0 < n_new) {
      // the wavefront's own quarter of the k-steps first (no branch around the shared sums); the fragments of the next k-step are
      // on their way while one is multiplied
      frag k0, k1, xv;
      auto load = [&](int j) FM_ALWAYS_INLINE {
        const int u = (j + NSTEP / 4 * wave) % NSTEP;
        const E* kt = cbuf + 16 * u * PQ;
        k0 = M::load_tr(kt, PQ, 0, 0, lane); k1 = M::load_tr(kt, PQ, 0, 32, lane);
        xv = M::load_nat_perm(xt + wave * XP, u, lh);
      };
      load(0);
#pragma unroll
      for (int j = 0; j < NSTEP; ++j) {
        const frag c0 = k0, c1 = k1, f0 = k0 * xv, f1 = k1 * xv;
        if (j + 1 < NSTEP) load(j + 1);
        FM_SCHED_FENCE();
        col[0] = M::mma(f0, c0, col[0]);
        col[1] = M::mma(f0, c1, col[1]);
        col[2] = M::mma(f1, c1, col[2]);
        if (j < NSTEP / 4) {
          const frag xs = M::load_nat_perm(xt + (lr < XR ? lr : XR - 1) * XP, (j + NSTEP / 4 * wave) % NSTEP, lh);   // rows past the eighth: zeros
          sh[0] = M::mma(c0, c0, sh[0]);
          sh[1] = M::mma(c0, c1, sh[1]);
          sh[2] = M::mma(c1, c1, sh[2]);
          sh[3] = M::mma(c0, xs, sh[3]);
          sh[4] = M::mma(c1, xs, sh[4]);
          sh[5] = M::mma(xs, xs, sh[5]);
        }
      }
    }
    FM_SYNC_LDS();
    par ^= 1;
  }
  // the staging buffers are spent: the loop ended on a barrier
  fm_absorb_finish<DH, true, FRESH>(col, sh, reinterpret_cast<float*>(smem), num, den);
}

// The same sums from fp32 products, for fp32 tensors, order 1 and heads of 32.  A matrix instruction takes two tokens; its operands
// are single floats of the staged rows (key rows [token][feature], x rows [token][8]), read across the lanes without conflicts.
// The matrix pipe bounds it: 4.5 instructions of 64 cycles per two tokens, wavefront and order-2 problem at D = 64.
//
// Its order-2 terms are (k'_a v) k'_b, those of k_decode (k'_a k'_b) v.  A product k'_a v that overflows leaves a sum that is not
// finite (infinity times a feature of zero is not a number); a workgroup that finds one adds its tokens one after the other
// after all.  (That code costs 3 of 237 us at 16 heads of 3001 tokens; looking at every product took 73.)  One below 2^-126 is off by
// at most 2^-150, times k'_b.
template <int DH, bool QUAD> struct DecAbsF32Cfg {
  static constexpr int TT = 64;                        // tokens per tile
  static constexpr int PQ = DH + 4;
  static constexpr int TILE = TT * PQ + TT * FM_ABS_XR;
  static constexpr size_t lds_bytes() {
    const size_t st = size_t(FM_ABS_GROUPS) * 2 * TILE * 4, red = AbsSums<DH, QUAD>::red_bytes();
    return st > red ? st : red;
  }
};
template <typename TIO, int DH, bool QUAD, bool FRESH>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(FM_ABS_THREADS, 2)
k_decode_absorb_f32(TRef<const TIO> k, TRef<const TIO> v, int n_new, float inv_tau, float* FM_RESTRICT state) {
  typedef Mma<float> M;
  typedef DecAbsF32Cfg<DH, QUAD> C;
  typedef AbsSums<DH, QUAD> S;
  constexpr int TT = C::TT, PQ = C::PQ, XR = FM_ABS_XR, NT = DH / 32, NG = FM_ABS_GROUPS;
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  if (QUAD && FM_TID_X == 0) bad = 0;
  const int lane = FM_TID_X & 63, lr = lane & 31, lh = lane >> 5;
  const int wave8 = FM_UNIFORM(FM_TID_X >> 6), wave = wave8 & 3, grp = wave8 >> 2;
  const int tid = FM_TID_X & 255;
  float* const buf0 = reinterpret_cast<float*>(smem) + grp * 2 * C::TILE;
  int cb, bh;
  fm_xcd_map(FM_GDIM_X, FM_GDIM_Y, cb, bh);
  const int c4 = 4 * cb;
  const int64_t Rp = fm_decode_rows_padded(DH, QUAD);
  float* num = state + (int64_t(bh) * (DH / 4) + cb) * Rp * 5;
  float* den = num + Rp * 4;
  const TIO* kb = k.base(bh);
  const TIO* vb = v.base(bh);
  constexpr int CPR = DH / 8, NK = TT * CPR / 256;
  static_assert(TT * CPR % 256 == 0, "whole pieces per thread");
  Raw<TIO, 8> kreg[NK];
  Raw<TIO, 4> vreg;
  auto fetch = [&](int t0) FM_ALWAYS_INLINE {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c = tid + 256 * i, row = t0 + c / CPR, f0 = (c % CPR) * 8;
      if (row < n_new) kreg[i].ld(kb + int64_t(row) * k.s_n + f0);
      else kreg[i].zero();
    }
    if (tid < TT) {
      if (t0 + tid < n_new) vreg.ld(vb + int64_t(t0 + tid) * v.s_n + c4);
      else vreg.zero();
    }
  };
  auto put = [&](float* b, int t0) FM_ALWAYS_INLINE {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c = tid + 256 * i;
      float sc[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sc[j] = kreg[i].get(j) * inv_tau;
      CE<float>::st8(b + (c / CPR) * PQ + (c % CPR) * 8, sc);
    }
    if (tid < TT) {
      const float x[8] = {vreg.get(0), vreg.get(1), vreg.get(2), vreg.get(3), t0 + tid < n_new ? 1.0f : 0.0f, 0.f, 0.f, 0.f};
      CE<float>::st8(b + TT * PQ + tid * XR, x);
    }
  };
  fm_f32x16 col[S::NP > 0 ? S::NP : 1], sh[S::NSH];
#pragma unroll
  for (int i = 0; i < S::NP; ++i) col[i] = fm_zero16();
#pragma unroll
  for (int i = 0; i < S::NSH; ++i) sh[i] = fm_zero16();
  const int g0 = grp * TT;
  fetch(g0);
  put(buf0, g0);
  if (NG * TT < n_new) fetch(NG * TT + g0);
  FM_SYNC_LDS();
  int par = 0;
  for (int tb = 0; tb < n_new; tb += NG * TT) {
    const float* kt = buf0 + par * C::TILE;
    const float* xt = kt + TT * PQ;
    if (tb + NG * TT < n_new) {
      put(buf0 + (par ^ 1) * C::TILE, tb + NG * TT + g0);
      if (tb + 2 * NG * TT < n_new) fetch(tb + 2 * NG * TT + g0);
    }
    if (tb + g0 < n_new) {
      constexpr int NU = TT / 2;
      auto step = [&](int j, auto shared_tag) FM_ALWAYS_INLINE {
        const int t = 2 * ((j + NU / 4 * wave) % NU) + lh;   // the wavefront's own quarter of the steps first
        float kf[NT], f[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) kf[i] = kt[t * PQ + 32 * i + lr];
        if constexpr (QUAD) {
          const float x = xt[t * XR + wave];
#pragma unroll
          for (int i = 0; i < NT; ++i) f[i] = kf[i] * x;
#pragma unroll
          for (int i = 0; i < S::NP; ++i) col[i] = M::mma(f[S::pa(i)], kf[S::pb(i)], col[i]);
        }
        if constexpr (decltype(shared_tag)::value) {
          const float xr = xt[t * XR + (lr & (XR - 1))], xs = lr < XR ? xr : 0.f;
#pragma unroll
          for (int i = 0; i < S::NP; ++i) sh[i] = M::mma(kf[S::pa(i)], kf[S::pb(i)], sh[i]);
#pragma unroll
          for (int i = 0; i < NT; ++i) sh[S::NP + i] = M::mma(kf[i], xs, sh[S::NP + i]);
          sh[S::NSH - 1] = M::mma(xs, xs, sh[S::NSH - 1]);
        }
      };
#pragma unroll
      for (int j = 0; j < NU / 4; ++j) step(j, std::true_type());
      if constexpr (QUAD) {
#pragma unroll 8
        for (int j = NU / 4; j < NU; ++j) step(j, std::false_type());
      }
    }
    FM_SYNC_LDS();
    par ^= 1;
  }
  if constexpr (QUAD) {
    float top = 0.f;
#pragma unroll
    for (int i = 0; i < S::NP; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) top += fm_absf(col[i][e]);
    if (!(top < 0x1p127f)) bad = 1;
    FM_SYNC_LDS();
    if (__builtin_expect(FM_UNIFORM(bad) != 0, 0)) {
      typedef DecRows<TIO, DH> W;
      static_assert(FM_ABS_THREADS == FM_DEC_THREADS && sizeof(float[W::TB][DH + 1]) % 16 == 0, "the threads and the LDS of k_decode");
      float (*ks)[DH + 1] = reinterpret_cast<float (*)[DH + 1]>(smem);
      float (*vs)[4] = reinterpret_cast<float (*)[4]>(smem + sizeof(float[W::TB][DH + 1]));
      constexpr int R = int(fm_decode_rows(DH, true));
      W w;
      w.load(num, den, R, true, FRESH, FM_TID_X);
      w.add(k, v, bh, c4, n_new, inv_tau, ks, vs, FM_TID_X);
      w.store(num, den, R, Rp, FRESH, FM_TID_X);
      return;
    }
  }
  fm_absorb_finish<DH, QUAD, FRESH>(col, sh, reinterpret_cast<float*>(smem), num, den);
}

// Prompts from this many tokens on are summed with matrix instructions.  Into a state that is there, order 2, microseconds with k_decode
// and with k_decode_absorb_f32: D = 64, 8 heads 64 tokens 27.1 and 15.6, 80 32.7 and 19.8; 64 heads 64 tokens 61.8 and 61.4, 80 73.8
// and 78.1, 96 86 and 78; D = 32, 128 heads 64 tokens 19.9 and 21.0, 80 23.3 and 28.5, 128 35.2 and 28.6.  A second tile hardly
// begun on a full chip is the one place k_decode wins; no rule for it, since at 33 heads it loses there too (65.6 and 57.2).
static constexpr int FM_DEC_MMA_MIN = 64;
// FRESH: a new state.  (With a branch on it at run time, and the addresses of a state's entries made ahead of all their loads, 64 bf16
// tokens at 64 heads took 47.6 us, so 44.2.)
template <typename TIO, int DH, bool QUAD, bool FRESH>
int fm_absorb_launch(const FastmaxDesc* d, const TRef<const TIO>& kr, const TRef<const TIO>& vr, int n_new, float* state, fm_stream_t stream) {
  const fm_dim3 grid(DH / 4, d->bh);
  if constexpr (sizeof(TIO) == 2 && DH == 64 && QUAD) {
    const size_t lds = DecAbsCfg<DH>::lds_bytes();
    fm_allow_lds(reinterpret_cast<const void*>(&k_decode_absorb_mma<TIO, DH, FRESH>), lds);
    FM_KERNEL_LAUNCH((k_decode_absorb_mma<TIO, DH, FRESH>), grid, fm_dim3(FM_ABS_THREADS), lds, stream, kr, vr, n_new, d->inv_tau, state);
  } else {
    const size_t lds = DecAbsF32Cfg<DH, QUAD>::lds_bytes();
    fm_allow_lds(reinterpret_cast<const void*>(&k_decode_absorb_f32<TIO, DH, QUAD, FRESH>), lds);
    FM_KERNEL_LAUNCH((k_decode_absorb_f32<TIO, DH, QUAD, FRESH>), grid, fm_dim3(FM_ABS_THREADS), lds, stream, kr, vr, n_new, d->inv_tau, state);
  }
  return fm_after_launch() ? FASTMAX_ERR_LAUNCH : FASTMAX_OK;
}

template <typename TIO, int DH>
int fm_decode_run(const FastmaxDesc* d, const void* q, const void* k, const void* v, int n_new, float* state, void* o,
                  float* g, float* scratch, fm_stream_t stream) {
  const bool quad = d->p == 2 && d->a2 != 0.0f;
  const TRef<const TIO> kr = fm_ref<const TIO>(static_cast<const TIO*>(k), d->sk), vr = fm_ref<const TIO>(static_cast<const TIO*>(v), d->sv);
  const TRef<const TIO> qr = q ? fm_ref<const TIO>(static_cast<const TIO*>(q), d->sq) : kr;
  (void)scratch;
  const bool fresh = !q && (d->flags & FASTMAX_FLAG_NEW_STATE);
  if (!q && n_new >= FM_DEC_MMA_MIN) {
    if (quad) return fresh ? fm_absorb_launch<TIO, DH, true, true>(d, kr, vr, n_new, state, stream)
                           : fm_absorb_launch<TIO, DH, true, false>(d, kr, vr, n_new, state, stream);
    return fresh ? fm_absorb_launch<TIO, DH, false, true>(d, kr, vr, n_new, state, stream)
                 : fm_absorb_launch<TIO, DH, false, false>(d, kr, vr, n_new, state, stream);
  }
  const TRef<TIO> orf = q ? fm_ref<TIO>(static_cast<TIO*>(o), d->so) : TRef<TIO>{};
  const TRef<float> grf = q ? fm_ref<float>(g, d->sg) : TRef<float>{};
  FM_KERNEL_LAUNCH((k_decode<TIO, DH>), fm_dim3(DH / 4, d->bh), fm_dim3(FM_DEC_THREADS), 0, stream, kr, vr, qr, n_new, quad ? 1 : 0,
                   d->inv_tau, d->a0, d->a1, quad ? d->a2 : 0.0f, state, orf, grf, q ? 1 : 0, fresh ? 1 : 0);
  return fm_after_launch() ? FASTMAX_ERR_LAUNCH : FASTMAX_OK;
}

inline int fm_decode_dispatch(const FastmaxDesc* d, const void* q, const void* k, const void* v, int n_new, float* state,
                              void* o, float* g, float* scratch, fm_stream_t stream) {
  if (d->dtype == FASTMAX_BF16)
    return d->d == 64 ? fm_decode_run<fm_bf16, 64>(d, q, k, v, n_new, state, o, g, scratch, stream)
                      : fm_decode_run<fm_bf16, 32>(d, q, k, v, n_new, state, o, g, scratch, stream);
  return d->d == 64 ? fm_decode_run<float, 64>(d, q, k, v, n_new, state, o, g, scratch, stream)
                    : fm_decode_run<float, 32>(d, q, k, v, n_new, state, o, g, scratch, stream);
}
