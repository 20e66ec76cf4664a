// Sequences of at most 64 queries and 64 keys: a whole batch*head is one workgroup's work, forward one launch, backward
// (dQ, dK and dV) one launch, the max-norm normalisation of q and k and its Jacobian inside both.
//
// Such problems (an image classifier: thousands of heads of 50 tokens) are bound by their bytes and by launches; the general
// kernels padded 50 tokens to blocks of 128 and 256, read every tensor two to four times and took a launch each for the
// norms, dQ, dK + dV and the Jacobian's row.  Here every tensor is read once and every result written once.
// fp32 tensors: products of three bf16 planes (fm_x3.h).  bf16 tensors: the operands are the caller's numbers themselves (one
// plane, exact), every factor (temperature, norms, 1 / g) is applied in fp32 to what the products give, and the weights
// are split in two planes (16 bits; the general kernels' _Float16 weights have 11), or in three (FULL, all 24 bits) where
// the caller asked for fp32 arithmetic or the weights may cancel; no range but fp32's applies here.  As in fm_x3.h the operands
// carry a power of two, so that the planes of the smallest numbers stay normal ones (dO always, the rest but for two planes).  Wavefront (i, j) of the four works on the 32 x 32 tile of query tile i and key tile j; two sums per
// result meet in LDS.  The backward forms the scores twice, keys along the accumulator rows for dQ and queries along
// them for dK and dV: each is then the operand of the product that follows, without a transposition.
// B*H = 1024, 50 tokens, D = 32, normalised (26 MB forward, 53 MB backward): fp32 forward with its norms 23 -> 11.3 us, backward
// with its Jacobian 77 -> 24.6 (160 in six launches before fm_x3.h), bf16 73 -> 30 in all; 1024 heads of 64 x 64, bf16: 82 -> 44.
// The kernels run once through straight code, so its length counts: half of the bf16 code was rounding spelt out in integer
// arithmetic, and taking it out brought forward and backward of the last shape from 56 to 44 us.
#pragma once
#include "fm_x3.h"

static constexpr int FM_SMALL_TOKENS = 64;

template <typename TIO> struct SmallArgs {
  TRef<const TIO> q, k, v, o, d_o;
  TRef<float> g;
  TRef<TIO> out, dk, dv;                // out: o | dq
  fm_half* out_resid; const fm_half* ores; int npad_q;   // see TokArgs
  int nq, nk, causal;
  float a0, a1, a2, sc;
  int plain;                            // see fm_x3_coef_lost
  int norm_q, norm_k, jac; float lim;   // max-norm scaling of q / k; jac: gradients with respect to the raw tensors
};

template <typename TIO, int DH, bool FULL> struct SmallCfg {
  static constexpr bool RAW = sizeof(TIO) == 2;        // operands are the caller's numbers
  static constexpr int PP = RAW && !FULL ? 2 : 3;      // planes of a weight
  static constexpr int PL = RAW ? 1 : 3;        // planes of an operand in LDS
  static constexpr int N = DH / 32;                    // eight-feature items of a tensor per thread
  static constexpr int PQ = PL * DH + 8, TILE = 64 * PQ, OP = DH + 4;
  static constexpr int PF = DH + 1;                    // PLAIN: pitch of a row of floats (fp32 tensors)
  static_assert(RAW || 2 * PF <= PQ, "a row of floats fits a row of planes");
  // factors on q, k and v, on dO, and on the weights
  static constexpr float UQ = FULL ? 0x1p24f : 1.0f, UG = 0x1p24f, UW = UQ;
  static constexpr size_t OS = size_t(2) * 64 * OP * 4;            // one result's two parts
  static constexpr size_t fwd_lds() { const size_t a = size_t(3) * TILE * 2, b = OS + 2 * 64 * 4; return a > b ? a : b; }
  static constexpr size_t bwd_lds() { const size_t a = size_t(4) * TILE * 2 + 2 * 64 * 4; return a > OS ? a : OS; }
};

template <typename TIO, int DH>
FM_DEVICE void fm_small_load(const TRef<const TIO>& t, int bh, int n, int tid, float (*r)[8]) {
#pragma unroll
  for (int i = 0; i < DH / 32; ++i) {
    const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
    fm_ld8_row<TIO>(t.base(bh), t.s_n, row, n, col, r[i]);
  }
}
// PLAIN, here and below: the second pass of a workgroup whose sums came out non-finite (the lower planes of a weight are
// zero or of either sign, so an infinite factor makes NaN or the other infinity of them; and see fm_x3_look): rows as
// floats (bf16 tensors: their own rows) and sums on the vector units, term by term, over the keys a query sees.
template <typename TIO, int DH, bool FULL, bool PLAIN> FM_DEVICE void fm_small_stage(uint16_t* tile, const float (*r)[8], const float* f, float up, int tid) {
  typedef SmallCfg<TIO, DH, FULL> C;
#pragma unroll
  for (int i = 0; i < DH / 32; ++i) {
    const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
    uint16_t* p = tile + row * C::PQ + col;
    if constexpr (C::RAW) {
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = r[i][j] * up;
      IO<fm_bf16>::st8(p, w);                    // exact: they came from bf16
    } else if constexpr (PLAIN) {
      float* q = reinterpret_cast<float*>(tile) + row * C::PF + col;
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = r[i][j] * (f[i] * up);
    } else {
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = r[i][j] * (f[i] * up);
      X3Row<DH>::store(p, fm_x3_split(w));
    }
  }
}
// largest squared row norm of the thread's wavefront with its row, as in k_maxnorm_keys: the first row among equal norms,
// a row whose norm is NaN left out
template <int DH> FM_DEVICE unsigned long long fm_small_norm_key(const float (*r)[8], int n, int tid) {
  unsigned long long key = 0;
#pragma unroll
  for (int i = 0; i < DH / 32; ++i) {
    const int row = (tid + 256 * i) / (DH / 8);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s += r[i][j] * r[i][j];
    s = fm_group_sum<DH / 8>(s);
    uint32_t bits;
    __builtin_memcpy(&bits, &s, 4);
    const unsigned long long k = row < n && s == s ? (static_cast<unsigned long long>(bits) << 32) | uint32_t(~row) : 0ull;
    key = k > key ? k : key;
  }
#pragma unroll
  for (int m = DH / 8; m < 64; m <<= 1) { const unsigned long long o = fm_shfl_xor_u64(key, m); key = o > key ? o : key; }
  return key;
}
// factor lim / norm, squared norm and its row from the four wavefronts' keys
FM_DEVICE float fm_small_factor(const unsigned long long* keys, bool on, float lim, float& m2, int& nstar) {
  m2 = 0.f; nstar = -1;
  if (!on) return 1.0f;
  unsigned long long k = keys[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) k = keys[w] > k ? keys[w] : k;
  m2 = fm_bits_f32(uint32_t(k >> 32));
  nstar = int(~uint32_t(k));
  return m2 > FM_MAXNORM_FLOOR ? lim * fm_rsqrtf(m2) : 0.0f;
}

template <typename TIO, int DH, bool FULL> FM_DEVICE float fm_small_at(const uint16_t* tile, int row, int col) {   // PLAIN
  typedef SmallCfg<TIO, DH, FULL> C;
  if constexpr (C::RAW) return fm_bf16_to_f32(tile[row * C::PQ + col]);
  else return reinterpret_cast<const float*>(tile)[row * C::PF + col];
}
template <typename TIO, int DH, bool FULL> FM_DEVICE float fm_small_dot(const uint16_t* a, int ra, const uint16_t* b, int rb) {
  float s = 0.f;
#pragma unroll 1
  for (int f = 0; f < DH; ++f) s += fm_small_at<TIO, DH, FULL>(a, ra, f) * fm_small_at<TIO, DH, FULL>(b, rb, f);
  return s;
}
template <typename TIO, int DH, bool FULL> FM_DEVICE void fm_small_add8(float v[8], float w, const uint16_t* tile, int row, int col) {
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] += w * fm_small_at<TIO, DH, FULL>(tile, row, col + j);
}

// 32 x 32 tile of rows `a` and columns `b` (tiles of 32 rows in LDS)
template <typename TIO, int DH, bool FULL> FM_DEVICE fm_f32x16 fm_small_tile(const uint16_t* a, const uint16_t* b, int lr, int lh) {
  typedef SmallCfg<TIO, DH, FULL> C;
  fm_f32x16 s = fm_zero16();
#pragma unroll
  for (int ks = 0; ks < DH / 16; ++ks) {
    const uint16_t *pa = a + lr * C::PQ + 16 * ks + 8 * lh, *pb = b + lr * C::PQ + 16 * ks + 8 * lh;
    if constexpr (C::RAW) s = fm_mfma_bf16(*reinterpret_cast<const fm_u16x8*>(pa), *reinterpret_cast<const fm_u16x8*>(pb), s);
    else s = fm_x3_mma(X3Row<DH>::load(pa), X3Row<DH>::load(pb), s);
  }
  return s;
}
// acc (rows = features, column = the lane's token) += sum over the 32 rows r of tile: tile[r][.] p[r]
template <typename TIO, int DH, bool FULL> FM_DEVICE void fm_small_acc(fm_f32x16* acc, const uint16_t* tile, const fm_f32x16& p, int lane) {
  typedef SmallCfg<TIO, DH, FULL> C;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const X3 pb = fm_x3_split_acc(p, h);
#pragma unroll
    for (int ct = 0; ct < DH / 32; ++ct) {
      if constexpr (C::RAW) {
        const fm_u16x8 t = fm_bf16_load_tr(tile, C::PQ, 16 * h, 32 * ct, lane);
        if constexpr (C::PP == 3) acc[ct] = fm_mfma_bf16(t, pb.p[2], acc[ct]);   // (else the optimiser drops its making)
        acc[ct] = fm_mfma_bf16(t, pb.p[1], acc[ct]);
        acc[ct] = fm_mfma_bf16(t, pb.p[0], acc[ct]);
      } else {
        acc[ct] = fm_x3_mma(X3Row<DH>::load_tr(tile, 16 * h, 32 * ct, lane), pb, acc[ct]);
      }
    }
  }
}

// bad: one flag in LDS, see fm_x3_look; keys: two times four, in LDS
template <typename TIO, int DH, bool FULL, bool PLAIN>
FM_DEVICE void fm_small_fwd(const SmallArgs<TIO>& A, unsigned char* smem, unsigned long long (*keys)[4], int* bad, const int tid) {
  typedef SmallCfg<TIO, DH, FULL> C;
  constexpr int NT = DH / 32, N = C::N;
  constexpr float UQ = PLAIN ? 1.0f : C::UQ, UW = PLAIN ? 1.0f : C::UW;
  uint16_t* Q = reinterpret_cast<uint16_t*>(smem);
  uint16_t* K = Q + C::TILE;
  uint16_t* V = K + C::TILE;
  const int lane = tid & 63, lr = lane & 31, lh = lane >> 5, bh = FM_BID_Y;
  const int wave = FM_UNIFORM(tid >> 6), ti = wave >> 1, tj = wave & 1, off = A.nk - A.nq;
  const float a0 = A.a0 * UW, a1 = A.a1 * (UW / (UQ * UQ)), a2 = A.a2 * (UW / (UQ * UQ * UQ * UQ));   // on scores that carry UQ^2
  float rq[N][8], rk[N][8], rv[N][8];
  fm_small_load<TIO, DH>(A.q, bh, A.nq, tid, rq);
  fm_small_load<TIO, DH>(A.k, bh, A.nk, tid, rk);
  fm_small_load<TIO, DH>(A.v, bh, A.nk, tid, rv);
  float fq = A.sc, fk = A.sc;
  if (A.norm_q | A.norm_k) {
    const unsigned long long a = fm_small_norm_key<DH>(rq, A.nq, tid), b = fm_small_norm_key<DH>(rk, A.nk, tid);
    if (lane == 0) { keys[0][wave] = a; keys[1][wave] = b; }
    FM_SYNC();
    float m2; int ns;
    fq *= fm_small_factor(keys[0], A.norm_q != 0, A.lim, m2, ns);
    fk *= fm_small_factor(keys[1], A.norm_k != 0, A.lim, m2, ns);
  }
  const float sq[2] = {fq, fq}, sk[2] = {fk, fk}, one[2] = {1.0f, 1.0f};
  fm_small_stage<TIO, DH, FULL, PLAIN>(Q, rq, sq, UQ, tid);
  fm_small_stage<TIO, DH, FULL, PLAIN>(K, rk, sk, UQ, tid);
  fm_small_stage<TIO, DH, FULL, PLAIN>(V, rv, one, UQ, tid);
  FM_SYNC();
  const float ss = C::RAW ? fq * fk : 1.0f;
  float* Os = reinterpret_cast<float*>(smem);
  float* Gs = Os + 2 * 64 * C::OP;
  if constexpr (!PLAIN) {
    fm_f32x16 acc[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_zero16();
    float gs = 0.f;
    if (32 * ti < A.nq && 32 * tj < A.nk && !(A.causal && 32 * tj > 32 * ti + 31 + off)) {
      fm_f32x16 s = fm_small_tile<TIO, DH, FULL>(K + 32 * tj * C::PQ, Q + 32 * ti * C::PQ, lr, lh);
      int last = A.nk - 1 - 32 * tj;                     // last key row the lane's query sees
      if (A.causal) { const int l = 32 * ti + lr + off - 32 * tj; last = l < last ? l : last; }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float x = C::RAW ? s[e] * ss : s[e], p = a0 + x * (a1 + a2 * x);
        s[e] = fm_acc_row(e, lh) <= last ? p : 0.f;
        gs += s[e];
      }
      fm_small_acc<TIO, DH, FULL>(acc, V + 32 * tj * C::PQ, s, lane);
    }
    FM_SYNC();
    fm_x3_put<DH, 64>(acc, Os, tj, 32 * ti + lr, lh);
    gs += fm_shfl_xor(gs, 32);
    if (lh == 0) Gs[tj * 64 + 32 * ti + lr] = gs;
    FM_SYNC();
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
    if (row >= A.nq) continue;
    float v[8], gt = 0.f;
    if constexpr (PLAIN) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = 0.f;
      const int ke = A.causal && row + off + 1 < A.nk ? row + off + 1 : A.nk;
#pragma unroll 1
      for (int t = 0; t < ke; ++t) {
        const float x = fm_small_dot<TIO, DH, FULL>(Q, row, K, t) * ss, p = a0 + x * (a1 + a2 * x);
        gt += p;
        fm_small_add8<TIO, DH, FULL>(v, p, V, t, col);
      }
    } else {
      fm_x3_sum8<DH, 64, 2>(Os, row, col, v);
      gt = Gs[row] + Gs[64 + row];
      fm_x3_look(bad, v, gt);
    }
    gt *= 1.0f / UW;
    const float gi = 1.0f / gt;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = v[j] * (1.0f / (UW * UQ)) * gi;
    IO<TIO>::st8(A.out.base(bh) + int64_t(row) * A.out.s_n + col, v);
    if (A.out_resid) {
      float sv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sv[j] = fm_as_stored<TIO>(v[j]);
      fm_store_resid8(A.out_resid + (int64_t(bh) * A.npad_q + row) * DH + col, v, sv);
    }
    if (col == 0) A.g.base(bh)[int64_t(row) * A.g.s_n] = gt;
  }
}
// grid (1, bh), 256 threads
template <typename TIO, int DH, bool FULL>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(256, 2) k_small_fwd(SmallArgs<TIO> A) {
  FM_DYN_SMEM(smem);
  FM_SHARED unsigned long long keys[2][4];
  FM_SHARED int bad;
  if (FM_TID_X == 0) bad = 0;
  if (!A.plain) {
    fm_small_fwd<TIO, DH, FULL, false>(A, smem, keys, &bad, FM_TID_X);
    if (!fm_x3_again(&bad)) FM_END();
  }
  fm_small_fwd<TIO, DH, FULL, true>(FM_ARGS_AGAIN(A), smem, keys, &bad, FM_TID_X + FM_OPAQUE_ZERO());
}

// one result's rows: the two parts summed, multiplied by down and by scale; returns the thread's share of sum value * raw
// (Os null: the sums are in v)
template <int DH> FM_DEVICE float fm_small_result(const float* Os, float down, float scale, const float (*raw)[8], int tid, float (*v)[8]) {
  float b = 0.f;
#pragma unroll
  for (int i = 0; i < DH / 32; ++i) {
    const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
    if (Os) fm_x3_sum8<DH, 64, 2>(Os, row, col, v[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) { v[i][j] = v[i][j] * down * scale; b += v[i][j] * raw[i][j]; }
  }
  return b;
}
// stores it, less the Jacobian's rank-one term in row nstar (see k_norm_fix)
template <typename TIO, int DH>
FM_DEVICE void fm_small_store(const TRef<TIO>& t, int bh, int n, int nstar, float coef, const float (*raw)[8], int tid, float (*v)[8]) {
#pragma unroll
  for (int i = 0; i < DH / 32; ++i) {
    const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
    if (row >= n) continue;
    if (row == nstar) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] -= coef * raw[i][j];
    }
    IO<TIO>::st8(t.base(bh) + int64_t(row) * t.s_n + col, v[i]);
  }
}

// bsum: two times four floats in LDS
template <typename TIO, int DH, bool FULL, bool PLAIN>
FM_DEVICE void fm_small_bwd(const SmallArgs<TIO>& A, unsigned char* smem, unsigned long long (*keys)[4], float (*bsum)[4], int* bad,
                            const int tid) {
  typedef SmallCfg<TIO, DH, FULL> C;
  constexpr int NT = DH / 32, N = C::N;
  constexpr float UQ = PLAIN ? 1.0f : C::UQ, UW = PLAIN ? 1.0f : C::UW;
  float ug = C::UG, down = 1.0f;                       // factor on dO; what takes it out again
  uint16_t* Q = reinterpret_cast<uint16_t*>(smem);
  uint16_t* K = Q + C::TILE;
  uint16_t* V = K + C::TILE;
  uint16_t* G = V + C::TILE;                           // gh = dO / g (bf16 tensors: dO)
  float* cs = reinterpret_cast<float*>(G + C::TILE);   // c = gh . o
  float* gr = cs + 64;                                 // 1 / g
  const int lane = tid & 63, lr = lane & 31, lh = lane >> 5, bh = FM_BID_Y;
  const int wave = FM_UNIFORM(tid >> 6), ti = wave >> 1, tj = wave & 1, off = A.nk - A.nq;
  float rq[N][8], rk[N][8];
  float fq = 1.0f, fk = 1.0f, m2q = 0.f, m2k = 0.f;
  int nsq = -1, nsk = -1;
  {
    float rv[N][8], ro[N][8], rd[N][8], gi[N];
    fm_small_load<TIO, DH>(A.q, bh, A.nq, tid, rq);
    fm_small_load<TIO, DH>(A.k, bh, A.nk, tid, rk);
    fm_small_load<TIO, DH>(A.v, bh, A.nk, tid, rv);
    fm_small_load<TIO, DH>(A.o, bh, A.nq, tid, ro);
    fm_small_load<TIO, DH>(A.d_o, bh, A.nq, tid, rd);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
      gi[i] = row < A.nq ? 1.0f / A.g.base(bh)[int64_t(row) * A.g.s_n] : 0.f;
      if (A.ores && row < A.nq) {
        const fm_half8 rs = *reinterpret_cast<const fm_half8*>(A.ores + (int64_t(bh) * A.npad_q + row) * DH + col);
#pragma unroll
        for (int j = 0; j < 8; ++j) ro[i][j] += float(rs[j]);
      }
    }
    if constexpr (PLAIN) {
      // dO of any size: its largest finite entry between 1 and 2 (a sum of products with dO itself may overflow else)
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float x = fm_absf(rd[i][j]); m = x < 0x1p127f * 1.9999999f && x > m ? x : m; }
#pragma unroll
      for (int w = 1; w < 64; w <<= 1) m = fm_fmaxf(m, fm_shfl_xor(m, w));
      if (lane == 0) bsum[0][wave] = m;
      FM_SYNC();
      m = fm_fmaxf(fm_fmaxf(bsum[0][0], bsum[0][1]), fm_fmaxf(bsum[0][2], bsum[0][3]));
      uint32_t e;
      __builtin_memcpy(&e, &m, 4);
      e >>= 23;
      e = e < 1 ? 1 : e > 253 ? 253 : e;
      ug = fm_bits_f32((254 - e) << 23);
      down = fm_bits_f32(e << 23);
      FM_SYNC();
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) rd[i][j] *= ug;
    if (A.norm_q | A.norm_k) {
      const unsigned long long a = fm_small_norm_key<DH>(rq, A.nq, tid), b = fm_small_norm_key<DH>(rk, A.nk, tid);
      if (lane == 0) { keys[0][wave] = a; keys[1][wave] = b; }
      FM_SYNC();
      fq = fm_small_factor(keys[0], A.norm_q != 0, A.lim, m2q, nsq);
      fk = fm_small_factor(keys[1], A.norm_k != 0, A.lim, m2k, nsk);
    }
    const float sq[2] = {A.sc * fq, A.sc * fq}, sk[2] = {A.sc * fk, A.sc * fk}, one[2] = {1.0f, 1.0f};
    fm_small_stage<TIO, DH, FULL, PLAIN>(Q, rq, sq, UQ, tid);
    fm_small_stage<TIO, DH, FULL, PLAIN>(K, rk, sk, UQ, tid);
    fm_small_stage<TIO, DH, FULL, PLAIN>(V, rv, one, UQ, tid);
    fm_small_stage<TIO, DH, FULL, PLAIN>(G, rd, gi, 1.0f, tid);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + 256 * i;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += rd[i][j] * ro[i][j];
      s = fm_group_sum<DH / 8>(s * gi[i] * UQ);        // carries UQ UG, as dO . v
      if (c % (DH / 8) == 0) { cs[c / (DH / 8)] = s; gr[c / (DH / 8)] = gi[i]; }
    }
  }
  FM_SYNC();
  const float ss = C::RAW ? A.sc * A.sc * fq * fk : 1.0f;
  // on scores that carry UQ^2; dS carries UG
  const float d1 = A.a1 * (1.0f / UQ), d2 = 2.0f * A.a2 * (1.0f / (UQ * UQ * UQ));
  const float a0 = A.a0 * UW, a1 = A.a1 * (UW / (UQ * UQ)), a2 = A.a2 * (UW / (UQ * UQ * UQ * UQ));
  const float scale_q = A.sc * (A.jac ? fq : 1.0f) * (C::RAW ? A.sc * fk : 1.0f), scale_k = A.sc * (A.jac ? fk : 1.0f) * (C::RAW ? A.sc * fq : 1.0f);
  float vq[N][8], vk[N][8], vv[N][8];
  float bq, bk;
  if constexpr (PLAIN) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + 256 * i, row = c / (DH / 8), col = (c % (DH / 8)) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) { vq[i][j] = 0.f; vk[i][j] = 0.f; vv[i][j] = 0.f; }
      const int ke = row >= A.nq ? 0 : A.causal && row + off + 1 < A.nk ? row + off + 1 : A.nk;
#pragma unroll 1
      for (int t = 0; t < ke; ++t) {
        const float x = fm_small_dot<TIO, DH, FULL>(Q, row, K, t) * ss, dp = fm_small_dot<TIO, DH, FULL>(G, row, V, t) * (C::RAW ? gr[row] : 1.0f);
        fm_small_add8<TIO, DH, FULL>(vq[i], (d1 + d2 * x) * (dp - cs[row]), K, t, col);
      }
      const int qb = A.causal && row > off ? row - off : 0;
#pragma unroll 1
      for (int t = row < A.nk ? qb : A.nq; t < A.nq; ++t) {
        const float gi = C::RAW ? gr[t] : 1.0f, x = fm_small_dot<TIO, DH, FULL>(Q, t, K, row) * ss, dp = fm_small_dot<TIO, DH, FULL>(G, t, V, row) * gi;
        fm_small_add8<TIO, DH, FULL>(vk[i], (d1 + d2 * x) * (dp - cs[t]), Q, t, col);
        fm_small_add8<TIO, DH, FULL>(vv[i], (a0 + x * (a1 + a2 * x)) * gi, G, t, col);
      }
    }
    bq = fm_small_result<DH>(nullptr, scale_q, down, rq, tid, vq);
    bk = fm_small_result<DH>(nullptr, scale_k, down, rk, tid, vk);
    (void)fm_small_result<DH>(nullptr, 1.0f, down, rk, tid, vv);
  } else {
    fm_f32x16 aq[NT], ak[NT], av[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) { aq[ct] = fm_zero16(); ak[ct] = fm_zero16(); av[ct] = fm_zero16(); }
    if (32 * ti < A.nq && 32 * tj < A.nk && !(A.causal && 32 * tj > 32 * ti + 31 + off)) {
      const uint16_t *Qt = Q + 32 * ti * C::PQ, *Kt = K + 32 * tj * C::PQ, *Vt = V + 32 * tj * C::PQ, *Gt = G + 32 * ti * C::PQ;
      const int diag = 32 * (ti - tj) + off;             // query row r sees key rows 0 .. r + diag
      {
        // rows = keys, column = the lane's query
        fm_f32x16 s = fm_small_tile<TIO, DH, FULL>(Kt, Qt, lr, lh);
        const fm_f32x16 dp = fm_small_tile<TIO, DH, FULL>(Vt, Gt, lr, lh);
        const float c = cs[32 * ti + lr], gi = C::RAW ? gr[32 * ti + lr] : 1.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float ds = (d1 + d2 * (s[e] * ss)) * (dp[e] * gi - c);
          s[e] = A.causal && fm_acc_row(e, lh) > lr + diag ? 0.f : ds;
        }
        fm_small_acc<TIO, DH, FULL>(aq, Kt, s, lane);
      }
      {
        // rows = queries, column = the lane's key (rows past the last query: gh = c = 0, they add nothing)
        fm_f32x16 s = fm_small_tile<TIO, DH, FULL>(Qt, Kt, lr, lh);
        fm_f32x16 dp = fm_small_tile<TIO, DH, FULL>(Gt, Vt, lr, lh);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = fm_acc_row(e, lh);
          const float gi = C::RAW ? gr[32 * ti + r] : 1.0f, x = s[e] * ss;
          const float ds = (d1 + d2 * x) * (dp[e] * gi - cs[32 * ti + r]), p = (a0 + x * (a1 + a2 * x)) * gi;
          const bool hid = A.causal && lr > r + diag;
          dp[e] = hid ? 0.f : ds;
          s[e] = hid ? 0.f : p;
        }
        fm_small_acc<TIO, DH, FULL>(ak, Qt, dp, lane);
        fm_small_acc<TIO, DH, FULL>(av, Gt, s, lane);
      }
    }
    // the three results in turn through one region (two parts each), so that two to four workgroups share a CU (fp32 rows of 64:
    // one, with 103 KB)
    float* Os = reinterpret_cast<float*>(smem);
    FM_SYNC();
    fm_x3_put<DH, 64>(aq, Os, tj, 32 * ti + lr, lh);
    FM_SYNC();
    bq = fm_small_result<DH>(Os, 1.0f / (C::UG * UQ), scale_q, rq, tid, vq);
    FM_SYNC();
    fm_x3_put<DH, 64>(ak, Os, ti, 32 * tj + lr, lh);
    FM_SYNC();
    bk = fm_small_result<DH>(Os, 1.0f / (C::UG * UQ), scale_k, rk, tid, vk);
    FM_SYNC();
    fm_x3_put<DH, 64>(av, Os, ti, 32 * tj + lr, lh);
    FM_SYNC();
    // a sum that is not finite makes its b that, whatever the row it is multiplied by
    const float bv = fm_small_result<DH>(Os, 1.0f / (C::UG * UW), 1.0f, rk, tid, vv);
    if (!(fm_absf(bq) + fm_absf(bk) + fm_absf(bv) < 0x1p127f)) *bad = 1;
  }
  float cq = 0.f, ck = 0.f;
  if (A.jac) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) { bq += fm_shfl_xor(bq, m); bk += fm_shfl_xor(bk, m); }
    if (lane == 0) { bsum[0][wave] = bq; bsum[1][wave] = bk; }
    FM_SYNC();
    if (m2q > FM_MAXNORM_FLOOR) cq = ((bsum[0][0] + bsum[0][1]) + (bsum[0][2] + bsum[0][3])) / m2q;
    if (m2k > FM_MAXNORM_FLOOR) ck = ((bsum[1][0] + bsum[1][1]) + (bsum[1][2] + bsum[1][3])) / m2k;
  }
  fm_small_store<TIO, DH>(A.out, bh, A.nq, cq != 0.f ? nsq : -1, cq, rq, tid, vq);
  fm_small_store<TIO, DH>(A.dk, bh, A.nk, ck != 0.f ? nsk : -1, ck, rk, tid, vk);
  fm_small_store<TIO, DH>(A.dv, bh, A.nk, -1, 0.f, rk, tid, vv);
}
// grid (1, bh), 256 threads
template <typename TIO, int DH, bool FULL>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(256, (DH == 64 ? (sizeof(TIO) == 4 ? 1 : 2) : (sizeof(TIO) == 4 ? 2 : 3))) k_small_bwd(SmallArgs<TIO> A) {
  FM_DYN_SMEM(smem);
  FM_SHARED unsigned long long keys[2][4];
  FM_SHARED float bsum[2][4];
  FM_SHARED int bad;
  if (FM_TID_X == 0) bad = 0;
  if (!A.plain) {
    fm_small_bwd<TIO, DH, FULL, false>(A, smem, keys, bsum, &bad, FM_TID_X);
    if (!fm_x3_again(&bad)) FM_END();
  }
  fm_small_bwd<TIO, DH, FULL, true>(FM_ARGS_AGAIN(A), smem, keys, bsum, &bad, FM_TID_X + FM_OPAQUE_ZERO());
}
