// Dense fp32 attention on the _Float16 matrix pipes, at fp32 accuracy: two planes per number where its tensor's range allows it.
//
// A number x of a tensor that has been brought to a largest entry in [2^14, 2^15) is taken as h + l: h is x rounded to 11 bits, l
// the rest (formed exactly in fp32) rounded to 11 bits.  |x - h - l| <= max(2^-23 |x|, 2^-25), about one fp32 rounding of x for the
// numbers down to 2^-17 of the tensor's largest.  A product is taken as h h + (h l + l h), three v_mfma_f32_32x32x16_f16 with fp32
// accumulation; what is left out, l l, is below 2^-22 of |x y| and below 2^-24 of it on average.  fm_x3.h takes six products of
// bf16 planes, whose exponents fit every number; its sums are rounded twice as often.
//
// 4 x 8 heads of 4096 tokens, D = 64, causal, fm_x3.h and here: relative error of o, dq, dk, dv against 64-bit results 3.6e-7, 4.3e-7, 4.3e-7, 3.6e-7
// and 1.5e-7, 3.1e-7, 3.1e-7, 2.6e-7 (the forward has the registers for sums of the small terms apart: 3.0e-7 in one sum); forward 349
// and 220 us (24 of them k_x2_range), backward 1106 and 650 (16).  A few hundred terms give the sums too few roundings for
// that (see x2_pays), and such problems stay with fm_x3.h.
// What bounds these kernels is power: the forward keeps the matrix pipe 52 % busy at 1.9 GHz.  Copying ready-made planes to LDS past the
// registers, without bank conflicts, took 14 % of its cycles away and gave them back as a clock of 1.75 GHz.
//
// What the powers of two are taken from.
//   own rows     the row's largest entry (the lane holds the row)
//   stream rows  the largest entry of the batch*head (k, v, q) or of what a block of keys sees (gh = dO / g, which falls like the
//                reciprocal of the token index): partial maxima per 64 tokens, written by k_x2_range and joined by every workgroup
//   weights      f(s) as it is, times the power of two that brings a0 to [1, 2); dS times 2^-19 (of products of two scaled rows), less
//                where scores are large (fm_x2_ds_exp)
// The powers are taken out of the polynomials' coefficients and of the sums, exactly.
//
// Which problems these kernels may take is decided in two places.  x2_coefficients (host): a0 > 0, a1 of its
// size and weights that do not change their sign.  k_x2_range and its readers, per batch*head: the largest entry of every row and every column of
// a block of 64 tokens that is not zero is at least 2^-14 of the tensor's largest, and so is held to 2^-25 of itself.  (gh: whole rows
// and blocks may be smaller, they add little to sums over rows; a column may not lie in them alone.)  A workgroup whose tensors do not
// keep to that, one whose weights may pass 65504 (fm_x2_weights) and one with a sum that is not finite make their rows as fm_x3.h does (and so,
// where those sums are not finite either, with fp32 matrix products).  What that costs, forward and backward, us, v's first row 1e-9 of the others, and
// the same problem on fm_x3.h's own launches: 32 heads of 4096 tokens 368 and 1169, 365 and 1243, 12 of 4096 205 and 632, 170 and 543, 4 of 2100 75 and 205,
// 53 and 153, unmasked 16 of 1024 48 and 122, 35 and 100.
#pragma once
#include "fm_x3.h"
#include <cmath>

struct X2 { fm_half8 h, l; };                          // eight numbers as two _Float16 planes

// a - b, a and the numbers it is near given as floats and halves: one instruction that reads the half where it lies
FM_DEVICE float fm_x2_minus(float a, fm_half b) {
#if defined(FM_HOSTSIM)
  return a - float(b);
#else
  uint32_t u = 0xbc00bc00u;                            // -1: as a constant it would become a conversion and a subtraction
  asm("" : "+s"(u));
  fm_half2 m;
  __builtin_memcpy(&m, &u, 4);
  return __builtin_fmaf(float(b), float(m[0]), a);     // v_fma_mix_f32; rounded to half v_fma_mixlo_f16
#endif
}
FM_DEVICE X2 fm_x2_split(const float v[8]) {
  X2 r;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const fm_f32x2 a = {v[i], v[i + 1]};
    const fm_half2 h = __builtin_convertvector(a, fm_half2);
    r.h[i] = h[0]; r.h[i + 1] = h[1];
    r.l[i] = fm_half(fm_x2_minus(a[0], h[0])); r.l[i + 1] = fm_half(fm_x2_minus(a[1], h[1]));
  }
  return r;
}
FM_DEVICE X2 fm_x2_split_acc(const fm_f32x16& s, int half) {
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = s[8 * half + i];
  return fm_x2_split(v);
}

// Rows of two planes: see X3Row.
template <int DH> struct X2Row {
  static constexpr int PQ = 2 * DH + 24;               // pitch of a staged row: two planes and 48 bytes, rows 12 banks apart
  static constexpr int NOWN = DH / 16, NT = DH / 32;
  struct Own { X2 f[NOWN]; };
  static FM_DEVICE X2 load(const fm_half* p) {
    X2 f;
    f.h = *reinterpret_cast<const fm_half8*>(p);
    f.l = *reinterpret_cast<const fm_half8*>(p + DH);
    return f;
  }
  static FM_DEVICE X2 load_tr(const fm_half* tile, int tok0, int col0, int lane) {
    X2 f;
    f.h = Mma<fm_half>::load_tr(tile, PQ, tok0, col0, lane);
    f.l = Mma<fm_half>::load_tr(tile + DH, PQ, tok0, col0, lane);
    return f;
  }
  static FM_DEVICE void put8(fm_half* tile, int row, int col, const float w[8]) {
    const X2 f = fm_x2_split(w);
    fm_half* p = tile + row * PQ + col;
    *reinterpret_cast<fm_half8*>(p) = f.h;
    *reinterpret_cast<fm_half8*>(p + DH) = f.l;
  }
  // small terms first
  static FM_DEVICE void score(const fm_half* X, int row, int lh, const Own& of, fm_f32x16& s) {
#pragma unroll
    for (int ks = 0; ks < NOWN; ++ks) {
      const X2 x = load(X + row * PQ + 16 * ks + 8 * lh);
      s = fm_mfma_f16(x.l, of.f[ks].h, s);
      s = fm_mfma_f16(x.h, of.f[ks].l, s);
      s = fm_mfma_f16(x.h, of.f[ks].h, s);
    }
  }
  static FM_DEVICE void score2(const fm_half* X, const fm_half* Y, int row, int lh, const Own& of, const Own& of2, fm_f32x16& s,
                               fm_f32x16& dp) {
#pragma unroll
    for (int ks = 0; ks < NOWN; ++ks) {
      const X2 x = load(X + row * PQ + 16 * ks + 8 * lh), y = load(Y + row * PQ + 16 * ks + 8 * lh);
      s = fm_mfma_f16(x.l, of.f[ks].h, s);
      dp = fm_mfma_f16(y.l, of2.f[ks].h, dp);
      s = fm_mfma_f16(x.h, of.f[ks].l, s);
      dp = fm_mfma_f16(y.h, of2.f[ks].l, dp);
      s = fm_mfma_f16(x.h, of.f[ks].h, s);
      dp = fm_mfma_f16(y.h, of2.f[ks].h, dp);
    }
  }
  // small: where the sums of the small terms go (acc itself, or sums of their own: a third of acc's roundings then)
  static FM_DEVICE void accum(fm_f32x16* acc, fm_f32x16* small, const fm_half* Y, int tok0, const fm_f32x16& s, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const X2 pb = fm_x2_split_acc(s, h);
      X2 z[NT];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) z[ct] = load_tr(Y, tok0 + 16 * h, 32 * ct, lane);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) small[ct] = fm_mfma_f16(z[ct].l, pb.h, small[ct]);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) small[ct] = fm_mfma_f16(z[ct].h, pb.l, small[ct]);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_mfma_f16(z[ct].h, pb.h, acc[ct]);
    }
  }
};

// ---- ranges ----------------------------------------------------------------------------------
static constexpr int FM_X2_TOKENS = 64;                // rows of a partial maximum; the last takes the rest (up to 127)
FM_DEVICE int fm_x2_block(int row, int nblk) { return row / FM_X2_TOKENS < nblk ? row / FM_X2_TOKENS : nblk - 1; }
inline int fm_x2_blocks(int n) { return n < FM_X2_TOKENS ? 1 : n / FM_X2_TOKENS; }
struct X2Job { TRef<const float> x; TRef<float> g; float *part, *least, *norm, *tail; unsigned long long* cols; int n, nblk, divide; };   // [bh][nblk] each

// part: largest |x| (divide: |x / g|) of a block of rows.  least: the smallest largest entry of its rows and columns that are not zero.  Where
// rows are divided their sizes are left out of that (a small row adds little to sums over rows, and its own workgroup scales it by itself), but
// a key that sees the sequence's end alone must not find it small: tail is the largest entry of the block's last row that is not zero.
// cols: one bit per column that is not zero (see fm_x2_columns).  norm: the largest Euclidean norm of a row.
// grid (blocks, bh, jobs), 256 threads.  Reads its tensors once: three of 4 x 8 heads of 4096 x 64 (101 MB).
template <int DH>
FM_GLOBAL void FM_LAUNCH_BOUNDS(256) k_x2_range(X2Job j0, X2Job j1, X2Job j2, X2Job j3) {
  constexpr int CPR = DH / 8, RPP = 256 / CPR;         // threads of a row, rows of a pass
  FM_SHARED float cm[4][DH], wr[4], wn[4];
  FM_SHARED unsigned long long wt[4];
  const X2Job& J = FM_BID_Z == 0 ? j0 : FM_BID_Z == 1 ? j1 : FM_BID_Z == 2 ? j2 : j3;
  const int tid = FM_TID_X, bh = FM_BID_Y, blk = FM_BID_X;
  if (blk >= J.nblk) return;
  const int r0 = blk * FM_X2_TOKENS, r1 = blk == J.nblk - 1 ? J.n : r0 + FM_X2_TOKENS, col = (tid % CPR) * 8;
  float c[8], rmin = 0x1p127f, n2 = 0.f;
  unsigned long long last = 0;                         // row and bits of its largest entry
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = 0.f;
  const float* base = J.x.base(bh);
  for (int p0 = r0; p0 < r1; p0 += 2 * RPP) {          // two rows in flight
    float v[2][8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = p0 + u * RPP + tid / CPR, rr = row < r1 ? row : r1 - 1;   // (a row twice: the same maxima)
      IO<float>::ld8(base + int64_t(rr) * J.x.s_n + col, v[u]);
      if (J.divide) {
        const float gi = J.g.base(bh)[int64_t(rr) * J.g.s_n];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[u][i] = v[u][i] / gi;
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float m = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) { const float a = fm_absf(v[u][i]); c[i] = fm_fmaxf(c[i], a); m = fm_fmaxf(m, a); q += a * a; }
      m = fm_lanes_max<1, CPR>(m);
      n2 = fm_fmaxf(n2, fm_group_sum<CPR>(q));
      if (m > 0.f && m < rmin) rmin = m;
      uint32_t b;
      __builtin_memcpy(&b, &m, 4);
      const int row = p0 + u * RPP + tid / CPR;
      if (m > 0.f && row < r1) last = (static_cast<unsigned long long>(uint32_t(row)) << 32) | b;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = fm_lanes_max<CPR, 64>(c[i]);
  rmin = -fm_lanes_max<CPR, 64>(-rmin);
  n2 = fm_lanes_max<CPR, 64>(n2);
  if (J.tail) {
#pragma unroll
    for (int s = CPR; s < 64; s <<= 1) {
      const unsigned long long l = fm_shfl_xor_u64(last, s);
      last = l > last ? l : last;
    }
  }
  const int wave = tid >> 6, lane = tid & 63;
  if (lane < CPR) {
#pragma unroll
    for (int i = 0; i < 8; ++i) cm[wave][col + i] = c[i];
  }
  if (lane == 0) { wr[wave] = rmin; wn[wave] = n2; wt[wave] = last; }
  FM_SYNC();
  if (tid >= 64) return;
  float m = 0.f;
  if (tid < DH) m = fm_fmaxf(fm_fmaxf(cm[0][tid], cm[1][tid]), fm_fmaxf(cm[2][tid], cm[3][tid]));
  float all = m, least = m > 0.f ? m : 0x1p127f;
  unsigned long long bits = m > 0.f ? 1ull << tid : 0ull;
  all = fm_lanes_max<1, 64>(all);
  least = -fm_lanes_max<1, 64>(-least);
  if (J.cols) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) bits |= fm_shfl_xor_u64(bits, s);
  }
  if (tid == 0) {
    for (int w = 0; w < 4; ++w) {
      if (!J.divide) least = wr[w] < least ? wr[w] : least;
      last = wt[w] > last ? wt[w] : last;
    }
    if (J.norm) J.norm[int64_t(bh) * J.nblk + blk] = fm_sqrtf(fm_fmaxf(fm_fmaxf(wn[0], wn[1]), fm_fmaxf(wn[2], wn[3])));
    if (J.tail) J.tail[int64_t(bh) * J.nblk + blk] = fm_bits_f32(uint32_t(last));
    if (J.cols) J.cols[int64_t(bh) * J.nblk + blk] = bits;
    J.part[int64_t(bh) * J.nblk + blk] = all;
    J.least[int64_t(bh) * J.nblk + blk] = least;
  }
}

// Largest of the partial maxima of blocks b0 .. nblk - 1, and whether what is not zero there reaches FM_X2_SPREAD of it.  (Whole wavefronts.)
static constexpr float FM_X2_SPREAD = 0x1p-14f;
struct X2Max { float mx, least; bool ok; };
FM_DEVICE X2Max fm_x2_join(const float* part, const float* small, int b0, int nblk, int lane) {
  float m = 0.f, least = 0x1p127f;
  for (int i = b0 + lane; i < nblk; i += 64) {
    const float x = part[i], y = small[i];
    m = fm_fmaxf(m, x);
    least = y < least ? y : least;
  }
  m = fm_lanes_max<1, 64>(m);
  least = -fm_lanes_max<1, 64>(-least);
  const X2Max r = {m, least, least >= m * FM_X2_SPREAD};
  return r;
}
// Largest of the norms.
FM_DEVICE float fm_x2_longest(const float* norm, int nblk, int lane) {
  float m = 0.f;
  for (int i = lane; i < nblk; i += 64) m = fm_fmaxf(m, norm[i]);
  return fm_lanes_max<1, 64>(m);
}
// Whether every column of blocks b0 .. nblk - 1 that is not zero reaches that part of mx (one block has all of them so), where not every block does.
FM_DEVICE bool fm_x2_columns(const float* small, const unsigned long long* cols, int b0, int nblk, float mx, int lane) {
  unsigned long long all = 0;
  for (int i = b0 + lane; i < nblk; i += 64) all |= cols[i];
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) all |= fm_shfl_xor_u64(all, s);
  unsigned long long one = 0;
  for (int i = b0 + lane; i < nblk; i += 64) one |= small[i] >= mx * FM_X2_SPREAD && cols[i] == all ? 1 : 0;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) one |= fm_shfl_xor_u64(one, s);
  return one != 0;
}
// Exponent e that brings m to [2^14, 2^15): m 2^e (0 for m = 0); ok cleared where that power or its inverse would leave fp32's
// normal numbers.
FM_DEVICE int fm_x2_exp(float m, bool& ok) {
  uint32_t b;
  __builtin_memcpy(&b, &m, 4);
  if (m > 0.f && !(m > 0x1p-100f && m < 0x1p100f)) ok = false;
  return m > 0x1p-100f && m < 0x1p100f ? 14 + 127 - int(b >> 23) : 0;
}
FM_DEVICE float fm_x2_pow(int e) { return fm_bits_f32(uint32_t(127 + e) << 23); }       // 2^e, |e| <= 126
FM_DEVICE float fm_x2_scalb(float x, int e) {
#if defined(FM_HOSTSIM)
  return std::ldexp(x, e);
#else
  return __builtin_amdgcn_ldexpf(x, e);
#endif
}
// Own rows that only form scores: no more than leaves the coefficients their range (a smaller score has no bits beside a0).  A row that has no
// exponent is a workgroup for fm_x3.h, but for one so small that its scores are (64 products with numbers below 2^(15 - stream): 2^-60).
FM_DEVICE int fm_x2_row_exp(float m, int stream, int* bad) {
  bool ok = true;
  const int e = fm_x2_exp(m, ok);
  if (!ok && (m > 1.0f || stream < -18)) *bad = 1;
  return e + stream > 56 ? 56 - stream : e;
}

#if defined(FM_HOSTSIM)
// Workgroups of these kernels whose rows fm_x3.h made: without a walk, and after one.
inline int fm_hostsim_x2_left[2] = {0, 0};
FM_DEVICE bool fm_x2_leave(int walked) { if (FM_TID_X == 0) ++fm_hostsim_x2_left[walked]; return true; }
#else
FM_DEVICE bool fm_x2_leave(int) { return true; }
#endif

static constexpr int FM_X2_DS = -19;                   // dS's power of two, see fm_x2_ds_exp
struct X2Args : X3Args<float> {
  const float *mq, *mk, *mv, *mg;       // partial maxima, least entries, gh's tails and columns: see k_x2_range
  const float *sq, *sk, *sv, *sg, *tg;
  const unsigned long long* cg;
  const float *lq, *lk;                 // largest norms of q and k rows per block
  int nbq, nbk;
  int ew;                               // exponent of the weights' factor (a0 2^ew in [1, 2))
};
// A score is at most the product of its rows' norms: b, the lane's own row with the longest stream row.
//   weights      one beyond _Float16 would be infinite: the workgroup leaves them to fm_x3.h before it makes any
//   dS           large derivatives take their size out of dS's power of two (an ordinary product of rows leaves them a factor of 8)
FM_DEVICE void fm_x2_weights(const X2Args& A, float b, int* bad) {
  const float w = fm_absf(A.a0) + b * (fm_absf(A.a1) + b * fm_absf(A.a2));
  if (!(fm_x2_scalb(w, A.ew) < 65000.0f)) *bad = 1;
}
FM_DEVICE int fm_x2_ds_exp(const X2Args& A, float b) {
  const float w = fm_x2_scalb(fm_absf(A.a1) + 2.0f * b * fm_absf(A.a2), A.ew);
  uint32_t u;
  __builtin_memcpy(&u, &w, 4);
  const int over = int(u >> 23) - 127 - 2;
  return FM_X2_DS - (over > 0 ? over : 0);
}
// The polynomials' coefficients: f(s) 2^ew, and f'(s) 2^(ew + ds), s = score 2^-es.
FM_DEVICE X3Coef fm_x2_coef(float a0, float a1, float a2, int ew, int es) {
  const X3Coef c = {fm_x2_scalb(a0, ew), fm_x2_scalb(a1, ew - es), fm_x2_scalb(a2, ew - 2 * es)};
  return c;
}
FM_DEVICE X3Coef fm_x2_dcoef(float a1, float a2, int ew, int ds, int es) {
  const X3Coef c = {0.f, fm_x2_scalb(a1, ew + ds), fm_x2_scalb(2.0f * a2, ew + ds - es)};
  return c;
}
// Coefficients that these kernels take; ew as above.  A score too small to be seen beside a0 is the whole of f'(s) where a1 is zero.  And f(s) is
// to stay away from zero (a0 / 2 at least: a1^2 <= 2 a0 a2, as the Taylor weights have it): weights of both signs cancel in the denominators and
// leave the roundings of the scores, which are two planes' there.  (Order 1, q and k with a common component that takes weights through zero,
// 176 heads of 780 tokens: o off by 9e-5, three planes 1.3e-5; 32 of 7000, D = 32, 3e-4 and 5e-5.)  So a2 is at least a0 / 512, and fm_x3.h's planes, which
// make what these kernels leave, do not lose it (see fm_x3_coef_lost).
inline bool x2_coefficients(float a0, float a1, float a2, int& ew) {
  const float b1 = std::fabs(a1), big = b1 > a2 ? b1 : a2;
  ew = 0;
  if (!(a0 > 0x1p-40f && a0 < 0x1p40f) || !(big <= 16.0f * a0) || !(b1 >= a0 * 0.0625f) || !(b1 * b1 <= 2.0f * a0 * a2)) return false;
  int e;
  std::frexp(a0, &e);
  ew = 1 - e;
  return true;
}

template <int DH, int NW, int SPLIT> struct X2Cfg {
  static constexpr int NTH = 64 * NW, OT = NW / SPLIT, QW = 32 * OT, KT = 32 * SPLIT, PQ = X2Row<DH>::PQ;
  static constexpr int STAGE = 2 * KT * PQ, NBUF = 2, SLOTS = NW == 8 ? 1 : 2;   // SLOTS: see fm_snake_rank
  // kind 0: forward, dQ; 1: dK + dV
  static constexpr size_t lds(int kind) {
    const size_t a = size_t(NBUF) * STAGE * 2 + (kind ? size_t(NBUF) * KT * 4 : 0), o = X3Cfg<DH, NW, SPLIT>::lds(kind);
    return a > o ? a : o;
  }
};

// Stage of ROWS stream rows of two tensors: caller's rows -> registers -> LDS planes.
template <int DH, int ROWS, int NTH> struct X2Stage {
  static constexpr int CPR = DH / 8, PER = ROWS * CPR, TOT = 2 * PER, N = (TOT + NTH - 1) / NTH;
  float r[N][8], gi[N];
  // Rows outside the tensor are its first or last one: whatever they give is masked (see fm_tile_edge) or not read.
  FM_DEVICE void load(const TRef<const float>& x, const TRef<const float>& y, const TRef<float>* g, int bh, int row0, int n, int tid) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + NTH * i;
      if (TOT % NTH != 0 && c >= TOT) break;
      const bool second = c >= PER;                    // the same for a whole wavefront: PER is a multiple of 64
      const int cc = second ? c - PER : c, r_ = row0 + cc / CPR, row = r_ < 0 ? 0 : r_ < n ? r_ : n - 1, col = (cc % CPR) * 8;
      const TRef<const float>& t = second ? y : x;
      IO<float>::ld8(t.base(bh) + int64_t(row) * t.s_n + col, r[i]);
      if (g) gi[i] = second ? g->base(bh)[int64_t(row) * g->s_n] : 1.0f;
    }
  }
  // rows of x times xs, rows of y times ys (div: times ys / g)
  FM_DEVICE void store(fm_half* X, fm_half* Y, float xs, float ys, bool div, int tid) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + NTH * i;
      if (TOT % NTH != 0 && c >= TOT) break;
      const bool second = c >= PER;
      const int cc = second ? c - PER : c;
      const float f = second ? (div ? ys * fm_rcpf(gi[i]) : ys) : xs;
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = r[i][j] * f;
      X2Row<DH>::put8(second ? Y : X, cc / CPR, (cc % CPR) * 8, w);
    }
  }
};

// The lane's own row, 8 features from 16 c + 8 lh in chunk c of DH / 16: times f.
template <int DH> FM_DEVICE void fm_x2_own(const TRef<const float>& t, int bh, int64_t row, bool in, int lh, float f, float (*v)[8]) {
  const float* p = t.base(bh) + row * t.s_n + 8 * lh;
#pragma unroll
  for (int c = 0; c < DH / 16; ++c) {
    IO<float>::ld8(p + 16 * c, v[c]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[c][i] = in ? v[c][i] * f : 0.f;
  }
}
template <int DH> FM_DEVICE float fm_x2_norm(const float (*v)[8]) {
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < DH / 16; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) q += v[c][i] * v[c][i];
  return fm_sqrtf(q + fm_shfl_xor(q, 32));
}
template <int DH> FM_DEVICE float fm_x2_largest(const float (*v)[8]) {
  float m = 0.f;
#pragma unroll
  for (int c = 0; c < DH / 16; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fm_fmaxf(m, fm_absf(v[c][i]));
  return fm_fmaxf(m, fm_shfl_xor(m, 32));
}
// Own rows, times f.  A quarter of the numbers lie half way between two that the planes hold, and what rounding does to an own row is the same
// for every stream token: it does not average out where the tokens have something in common.  So of the wavefronts that share an own tile every
// other one (other) rounds such numbers the other way, and what is left meets its opposite in the sums.
template <int DH> FM_DEVICE void fm_x2_set(typename X2Row<DH>::Own& o, const float (*v)[8], float f, bool other) {
#pragma unroll
  for (int c = 0; c < DH / 16; ++c) {
    float w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = v[c][i] * f;
    o.f[c] = fm_x2_split(w);
    if (other) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float l = fm_x2_minus(w[i], o.f[c].h[i]);
        o.f[c].l[i] = fm_half(l + (l - float(o.f[c].l[i])));
      }
    }
  }
}

// ------------------------------------------------------------------------------
// forward.  grid (ceil(nq / QW), bh).  Returns whether the workgroup's rows are to be made by fm_x3.h's products.
// ------------------------------------------------------------------------------
template <int DH, int SPLIT, int NW>
FM_DEVICE bool fm_x2_fwd(const X2Args& A, fm_half* st, int* bad) {
  typedef X2Cfg<DH, NW, SPLIT> C;
  typedef X2Row<DH> R;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  const int tid = FM_TID_X, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(causal, A.first != 0, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const int send = causal && t0 + QW < A.nk ? t0 + QW : A.nk;
  if (A.first && blk == 0) return fm_x2_leave(0);      // see fm_x2_dq
  typedef X2Stage<DH, KT, C::NTH> Stage;
  Stage sg;
  sg.load(A.k, A.v, nullptr, bh, 0, A.nk, tid);
  const float kf = A.sc * fm_norm_factor(A.k_fold, bh, lane), qs = A.sc * fm_norm_factor(A.q_fold, bh, lane);
  const X2Max xk = fm_x2_join(A.mk + int64_t(bh) * A.nbk, A.sk + int64_t(bh) * A.nbk, 0, A.nbk, lane), xv = fm_x2_join(A.mv + int64_t(bh) * A.nbk, A.sv + int64_t(bh) * A.nbk, 0, A.nbk, lane);
  bool ok = xk.ok && xv.ok;
  const int ek = FM_UNIFORM(fm_x2_exp(xk.mx * kf, ok)), ev = FM_UNIFORM(fm_x2_exp(xv.mx, ok));
  if (!ok) return fm_x2_leave(0);                      // the same for all of the batch*head
  const float ks_ = kf * fm_x2_pow(ek), vs = fm_x2_pow(ev), kn = kf * fm_x2_longest(A.lk + int64_t(bh) * A.nbk, A.nbk, lane);
  typename R::Own of;
  X3Coef cf;
  {
    float v[DH / 16][8];
    const bool in = lo + lr < A.nq;
    fm_x2_own<DH>(A.q, bh, in ? lo + lr : A.nq - 1, in, lh, qs, v);
    const int eq = fm_x2_row_exp(fm_x2_largest<DH>(v), ek, bad);
    fm_x2_set<DH>(of, v, fm_x2_scalb(1.0f, eq), SPLIT > 1 && (sub & 1));
    cf = fm_x2_coef(A.a0, A.a1, A.a2, A.ew, eq + ek);
    fm_x2_weights(A, kn * fm_x2_norm<DH>(v), bad);
  }
  // One accumulator over thousands of tokens rounds a sum of its own size at every product; at D = 64 there are registers to begin a new one
  // every 1024 (8192 tokens, a component that all tokens share: o 3.4e-7 off, states 1.6 - 2.6e-7, so 1.1e-7; the same time).
  constexpr bool FOLD = DH == 64;
  fm_f32x16 acc[NT], small[NT], total[FOLD ? NT : 1];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    acc[ct] = fm_zero16(); small[ct] = fm_zero16();
    if (FOLD) total[ct] = fm_zero16();
  }
  X3Sum gsum = {0.f, 0.f};
  int buf = 0;
  sg.store(st, st + KT * PQ, ks_, vs, false, tid);
  sg.load(A.k, A.v, nullptr, bh, KT, A.nk, tid);
  if (fm_x3_again(bad)) return fm_x2_leave(0);         // (the first stage's barrier)
  for (int s0 = 0; s0 < send; s0 += KT) {
    const fm_half* X = st + buf * C::STAGE;
    const fm_half* Y = X + KT * PQ;
    if (s0 > 0) FM_SYNC();
    const int ss0 = s0 + 32 * sub;
    if (ss0 < A.nk && !(causal && ss0 > lo + 31)) {
      fm_f32x16 s = fm_zero16();
      R::score(X, 32 * sub + lr, lh, of, s);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = cf.a0 + s[e] * (cf.a1 + cf.a2 * s[e]);
      if (fm_tile_edge<FM_OWN_Q>(causal, ss0, lo, A.nk)) { FM_KEEP_BRANCH(); fm_x3_window<FM_OWN_Q>(s, causal, ss0, lo, lr, lh, A.nk); }
      gsum.add(s);
      R::accum(acc, small, Y, 32 * sub, s, lane);
    }
    if (FOLD && ((s0 + KT) & (1024 * SPLIT - 1)) == 0) {
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) { total[FOLD ? ct : 0] += acc[ct]; acc[ct] = fm_zero16(); }
    }
    buf ^= 1;
    if (s0 + KT < send) {
      sg.store(st + buf * C::STAGE, st + buf * C::STAGE + KT * PQ, ks_, vs, false, tid);
      sg.load(A.k, A.v, nullptr, bh, s0 + 2 * KT, A.nk, tid);
    }
  }
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    acc[ct] += small[ct];
    if (FOLD) acc[ct] += total[FOLD ? ct : 0];
  }
  float* Os = reinterpret_cast<float*>(st);
  FM_SYNC();
  fm_x3_put<DH, QW>(acc, Os, sub, 32 * own + lr, lh);
  fm_x3_put_sum<DH, QW>(gsum, Os, sub, 32 * own + lr, lh);
  FM_SYNC();
  for (int c = tid; c < QW * (DH / 8); c += C::NTH) {
    const int r = c / (DH / 8), col = (c % (DH / 8)) * 8, qi = t0 + r;
    if (qi >= A.nq) continue;
    float v[8];
    fm_x3_sum8<DH, QW, SPLIT>(Os, r, col, v);
    const float gt = fm_x3_sum<DH, QW, SPLIT>(Os, r);
    fm_x3_look(bad, v, gt);
    const float gi = 1.0f / gt;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * gi * fm_x2_pow(-ev);
    IO<float>::st8(A.out.base(bh) + int64_t(qi) * A.out.s_n + col, v);
    if (col == 0) A.g.base(bh)[int64_t(qi) * A.g.s_n] = fm_x2_scalb(gt, -A.ew);
  }
  return fm_x3_again(bad) && fm_x2_leave(1);
}
template <int DH, int SPLIT, int NW>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(64 * NW, (DH == 32 && SPLIT == 2 ? 4 : 2)) k_x2_fwd(X2Args A) {   // (28 heads of 2200 tokens, unmasked, 78 us, with 133 registers 85)
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();                                           // (the flag is set before the first barrier of the walk)
  if (!fm_x2_fwd<DH, SPLIT, NW>(A, reinterpret_cast<fm_half*>(smem), &bad)) FM_END();
  FM_SYNC();
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();
  fm_x3_fwd<float, DH, SPLIT, X3Row<DH>, NW, true>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
  if (!fm_x3_again(&bad)) FM_END();
  fm_x3_fwd<float, DH, SPLIT, F32Row<DH>, NW, true>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
}

// ------------------------------------------------------------------------------
// dQ.  grid (ceil(nq / QW), bh).  dS = (a1 + 2 a2 s) (gh . v - c), gh = dO / g, c = gh . o.
// ------------------------------------------------------------------------------
template <int DH, int SPLIT, int NW>
FM_DEVICE bool fm_x2_dq(const X2Args& A, fm_half* st, int* bad) {
  typedef X2Cfg<DH, NW, SPLIT> C;
  typedef X2Row<DH> R;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  const int tid = FM_TID_X, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(causal, A.first != 0, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const int send = causal && t0 + QW < A.nk ? t0 + QW : A.nk;
  // Causal: the first queries have most of dq and, seen by the first keys, of dk, in few terms, which are as well rounded as their operands: gh . (v - o)
  // is small beside both factors there.  The first block of queries is short work, so it keeps three planes, forward and here, and starts first.
  // Without a temperature, errors of dq, dk, dv and three planes': 4 heads of 4096 tokens 3.1, 3.3, 2.8e-7, 2.7, 2.8, 2.6e-7, now 2.5, 2.6, 2.4e-7, 64 of
  // 2000 3.8, 5.1, 3.4e-7, 4.0, 4.0, 3.3e-7, now 3.5, 3.7, 3.0e-7.  Not where one wavefront sums 4096 tokens and more, whose roundings hide it (32 heads of
  // 4096: 3.8, 3.9, 3.7e-7, three planes 4.5, 4.4, 4.1e-7; step 866 us, with the block 881).
  if (A.first && blk == 0) return fm_x2_leave(0);
  typedef X2Stage<DH, KT, C::NTH> Stage;
  Stage sg;
  sg.load(A.k, A.v, nullptr, bh, 0, A.nk, tid);
  const float kf = A.sc * fm_norm_factor(A.k_fold, bh, lane), qf = fm_norm_factor(A.q_fold, bh, lane);
  const X2Max xk = fm_x2_join(A.mk + int64_t(bh) * A.nbk, A.sk + int64_t(bh) * A.nbk, 0, A.nbk, lane), xv = fm_x2_join(A.mv + int64_t(bh) * A.nbk, A.sv + int64_t(bh) * A.nbk, 0, A.nbk, lane);
  bool ok = xk.ok && xv.ok;
  const int ek = FM_UNIFORM(fm_x2_exp(xk.mx * kf, ok)), ev = FM_UNIFORM(fm_x2_exp(xv.mx, ok));
  if (!ok) return fm_x2_leave(0);
  const float ks_ = kf * fm_x2_pow(ek), vs = fm_x2_pow(ev), kn = kf * fm_x2_longest(A.lk + int64_t(bh) * A.nbk, A.nbk, lane);
  typename R::Own of, of2;
  X3Coef cf;
  float cs = 0.f;
  fm_f32x16 seed;                                      // gh . v starts from -c
  int eout;
  {
    const bool in = lo + lr < A.nq;
    const int64_t row = in ? lo + lr : A.nq - 1;
    float v[DH / 16][8];
    fm_x2_own<DH>(A.q, bh, row, in, lh, A.sc * qf, v);
    const int eq = fm_x2_row_exp(fm_x2_largest<DH>(v), ek, bad);
    fm_x2_set<DH>(of, v, fm_x2_scalb(1.0f, eq), SPLIT > 1 && (sub & 1));
    const int ds = fm_x2_ds_exp(A, kn * fm_x2_norm<DH>(v));
    if (causal) {
      // What that costs the small entries of dS is taken from the spread that v's rows may have, where the query sees none but small ones:
      // the largest of the blocks before its own, or the smallest of all.
      const float first = fm_x2_join(A.mv + int64_t(bh) * A.nbk, A.sv + int64_t(bh) * A.nbk, 0, fm_x2_block(t0, A.nbk), lane).mx;
      if (ds < FM_X2_DS && fm_fmaxf(first, xv.least) < xv.mx * fm_x2_scalb(FM_X2_SPREAD, FM_X2_DS - ds)) *bad = 1;
    }
    fm_x2_own<DH>(A.d_o, bh, row, in, lh, in ? 1.0f / A.g.base(bh)[row * A.g.s_n] : 0.f, v);
    const float* po = A.o.base(bh) + row * A.o.s_n + 8 * lh;
#pragma unroll
    for (int c = 0; c < DH / 16; ++c) {
      float o[8];
      IO<float>::ld8(po + 16 * c, o);
#pragma unroll
      for (int i = 0; i < 8; ++i) cs += v[c][i] * o[i];
    }
    bool fine = true;
    const int eg = fm_x2_exp(fm_x2_largest<DH>(v), fine);
    if (!fine) *bad = 1;
    fm_x2_set<DH>(of2, v, fm_x2_pow(eg), SPLIT > 1 && (sub & 1));
    cs += fm_shfl_xor(cs, 32);
    if (sub == 0 && lh == 0 && in) A.cv[int64_t(bh) * A.npad_q + row] = cs;
    cs = fm_x2_scalb(cs, eg + ev);                     // as gh . v
#pragma unroll
    for (int e = 0; e < 16; ++e) seed[e] = -cs;
    cf = fm_x2_dcoef(A.a1, A.a2, A.ew, ds, eq + ek);
    eout = -(eg + ev + ek + A.ew + ds);
  }
  fm_f32x16 acc[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_zero16();
  int buf = 0;
  sg.store(st, st + KT * PQ, ks_, vs, false, tid);
  sg.load(A.k, A.v, nullptr, bh, KT, A.nk, tid);
  if (fm_x3_again(bad)) return fm_x2_leave(0);         // (the first stage's barrier)
  for (int s0 = 0; s0 < send; s0 += KT) {
    const fm_half* X = st + buf * C::STAGE;
    const fm_half* Y = X + KT * PQ;
    if (s0 > 0) FM_SYNC();
    const int ss0 = s0 + 32 * sub;
    if (ss0 < A.nk && !(causal && ss0 > lo + 31)) {
      fm_f32x16 s = fm_zero16(), dp = seed;
      R::score2(X, Y, 32 * sub + lr, lh, of, of2, s, dp);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = (cf.a1 + cf.a2 * s[e]) * dp[e];
      if (fm_tile_edge<FM_OWN_Q>(causal, ss0, lo, A.nk)) { FM_KEEP_BRANCH(); fm_x3_window<FM_OWN_Q>(s, causal, ss0, lo, lr, lh, A.nk); }
      R::accum(acc, acc, X, 32 * sub, s, lane);
    }
    buf ^= 1;
    if (s0 + KT < send) {
      sg.store(st + buf * C::STAGE, st + buf * C::STAGE + KT * PQ, ks_, vs, false, tid);
      sg.load(A.k, A.v, nullptr, bh, s0 + 2 * KT, A.nk, tid);
    }
  }
#pragma unroll
  for (int ct = 0; ct < NT; ++ct)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[ct][e] = fm_x2_scalb(acc[ct][e], eout);
  fm_x3_store<float, DH, QW, SPLIT, C::NTH, true>(acc, reinterpret_cast<float*>(st), sub, 32 * own + lr, lh, 1.0f, A.sc * (A.bpart ? qf : 1.0f), A.out,
                                          bh, t0, A.nq, tid, A.q, A.bpart ? A.bpart + int64_t(bh) * FM_GDIM_X + blk : nullptr, bad);
  return fm_x3_again(bad) && fm_x2_leave(1);
}
template <int DH, int SPLIT, int NW>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(64 * NW, 2) k_x2_dq(X2Args A) {
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();                                           // (see k_x2_fwd)
  if (!fm_x2_dq<DH, SPLIT, NW>(A, reinterpret_cast<fm_half*>(smem), &bad)) FM_END();
  FM_SYNC();
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();
  fm_x3_dq<float, DH, SPLIT, X3Row<DH>, NW, true>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
  if (!fm_x3_again(&bad)) FM_END();
  fm_x3_dq<float, DH, SPLIT, F32Row<DH>, NW, true>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
}

// ------------------------------------------------------------------------------
// dK and dV.  grid (ceil(nk / QW), bh), 512 threads: eight wavefronts share the staged queries; own k and v in registers.
// ------------------------------------------------------------------------------
template <int DH, int SPLIT>
FM_DEVICE bool fm_x2_dkv(const X2Args& A, fm_half* st, int* bad) {
  typedef X2Cfg<DH, 8, SPLIT> C;
  typedef X2Row<DH> R;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  float* cst = reinterpret_cast<float*>(st + C::NBUF * C::STAGE);   // c of the staged queries [NBUF][KT]
  const int tid = FM_TID_X, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(false, false, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const int sbeg = causal ? t0 : 0, nst = (A.nq - sbeg + KT - 1) / KT;
  const int s_last = sbeg + (nst - 1) * KT;            // the stream is walked from its end: see k_ds
  typedef X2Stage<DH, KT, C::NTH> Stage;
  Stage sg;
  float creg = 0.f;
  const float* cvb = A.cv + int64_t(bh) * A.npad_q;
  auto fetch = [&](int s) FM_ALWAYS_INLINE {
    sg.load(A.q, A.d_o, &A.g, bh, s, A.nq, tid);
    const int r = s + tid % KT;
    creg = r >= 0 && r < A.nq ? cvb[r] : 0.f;
  };
  fetch(s_last);
  const float kf = fm_norm_factor(A.k_fold, bh, lane), qf = A.sc * fm_norm_factor(A.q_fold, bh, lane);
  const X2Max xq = fm_x2_join(A.mq + int64_t(bh) * A.nbq, A.sq + int64_t(bh) * A.nbq, 0, A.nbq, lane), xv = fm_x2_join(A.mv + int64_t(bh) * A.nbk, A.sv + int64_t(bh) * A.nbk, 0, A.nbk, lane);
  // gh: of the queries that the block's keys see
  const float *mg = A.mg + int64_t(bh) * A.nbq, *sg_ = A.sg + int64_t(bh) * A.nbq;
  const int b0 = causal ? fm_x2_block(t0, A.nbq) : 0;
  const X2Max xg = fm_x2_join(mg, sg_, b0, A.nbq, lane);
  bool ok = xq.ok && xv.ok && (xg.ok || fm_x2_columns(sg_, A.cg + int64_t(bh) * A.nbq, b0, A.nbq, xg.mx, lane));
  const int eq = FM_UNIFORM(fm_x2_exp(xq.mx * qf, ok)), ev = FM_UNIFORM(fm_x2_exp(xv.mx, ok)), eg = FM_UNIFORM(fm_x2_exp(xg.mx, ok));
  if (!ok) return fm_x2_leave(0);
  const float qs = qf * fm_x2_pow(eq), gsc = fm_x2_pow(eg), cl = fm_x2_scalb(1.0f, eg + ev), qn = qf * fm_x2_longest(A.lq + int64_t(bh) * A.nbq, A.nbq, lane);
  auto put = [&](int b) FM_ALWAYS_INLINE {
    fm_half* X = st + b * C::STAGE;
    sg.store(X, X + KT * PQ, qs, gsc, true, tid);
    if (tid < KT) cst[b * KT + tid] = -(creg * cl);
  };
  typename R::Own of, of2;
  X3Coef cp, cd;
  int ds;
  {
    const bool in = lo + lr < A.nk;
    const int64_t row = in ? lo + lr : A.nk - 1;
    float v[DH / 16][8];
    fm_x2_own<DH>(A.k, bh, row, in, lh, A.sc * kf, v);
    const int ek = fm_x2_row_exp(fm_x2_largest<DH>(v), eq, bad);
    fm_x2_set<DH>(of, v, fm_x2_scalb(1.0f, ek), SPLIT > 1 && (sub & 1));
    const float b = qn * fm_x2_norm<DH>(v);
    fm_x2_weights(A, b, bad);
    ds = fm_x2_ds_exp(A, b);
    if (causal) {
      // What the wavefront's keys see of gh falls like 1 / i: the power of two of what its first key sees.  What its last key sees has to be
      // within the range of that: the blocks of 64 behind its own, or, where those are zero, the last row of its own that is not (the row
      // before that it may not see).  As dS, 2^-11 less what its scores take (with 2^-14 and tau = 1, where g falls from one query to the next by any
      // factor: keys 16 - 63 of a head 9e-7 off, 2.3e-7 so); as gh by itself, the range of every tensor.
      const int last = (lo + 31 < A.nk ? lo + 31 : A.nk - 1), bl = fm_x2_block(last, A.nbq);
      const X2Max xw = fm_x2_join(mg, sg_, fm_x2_block(lo < last ? lo : last, A.nbq), A.nbq, lane), xl = fm_x2_join(mg, sg_, bl + 1, A.nbq, lane);
      const float seen = xl.mx > 0.f ? xl.mx : A.tg[int64_t(bh) * A.nbq + bl];
      if (seen > 0.f && (seen < xw.mx * fm_x2_scalb(0x1p-11f, FM_X2_DS - ds) || seen < xg.mx * FM_X2_SPREAD)) *bad = 1;
      bool fine = true;
      const int ew = fm_x2_exp(xw.mx, fine);
      if (xw.mx > 0.f && fine) ds += ew - eg;
    }
    fm_x2_own<DH>(A.v, bh, row, in, lh, fm_x2_pow(ev), v);
    fm_x2_set<DH>(of2, v, 1.0f, SPLIT > 1 && (sub & 1));
    cp = fm_x2_coef(A.a0, A.a1, A.a2, A.ew, ek + eq);
    cd = fm_x2_dcoef(A.a1, A.a2, A.ew, ds, ek + eq);
  }
  fm_f32x16 acc[NT], av[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) { acc[ct] = fm_zero16(); av[ct] = fm_zero16(); }
  int buf = 0;
  put(0);
  fetch(s_last - KT);
  if (fm_x3_again(bad)) return fm_x2_leave(0);         // (the first stage's barrier)
  for (int s0 = s_last; s0 >= sbeg; s0 -= KT) {
    const fm_half* X = st + buf * C::STAGE;
    const fm_half* Y = X + KT * PQ;
    if (s0 < s_last) FM_SYNC();
    const int ss0 = s0 + 32 * sub;
    if (ss0 < A.nq && !(causal && ss0 + 31 < lo)) {
      fm_f32x16 s = fm_zero16(), dp;                   // gh . v starts from -c
      const float* cf = cst + buf * KT + 32 * sub + 4 * lh;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const fm_f32x4 c4 = *reinterpret_cast<const fm_f32x4*>(cf + 8 * g4);
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[4 * g4 + i] = c4[i];
      }
      R::score2(X, Y, 32 * sub + lr, lh, of, of2, s, dp);
      // dp becomes dS, s becomes P
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float x = s[e];
        dp[e] *= cd.a1 + cd.a2 * x;
        s[e] = cp.a0 + x * (cp.a1 + cp.a2 * x);
      }
      if (fm_tile_edge<FM_OWN_K>(causal, ss0, lo, A.nq)) {
        FM_KEEP_BRANCH();
        fm_x3_window<FM_OWN_K>(s, causal, ss0, lo, lr, lh, A.nq);
        fm_x3_window<FM_OWN_K>(dp, causal, ss0, lo, lr, lh, A.nq);
      }
      R::accum(av, av, Y, 32 * sub, s, lane);
      R::accum(acc, acc, X, 32 * sub, dp, lane);
    }
    buf ^= 1;
    if (s0 - KT >= sbeg) { put(buf); fetch(s0 - 2 * KT); }
  }
  const int edk = -(eg + ev + eq + A.ew + ds), edv = -(eg + A.ew);
#pragma unroll
  for (int ct = 0; ct < NT; ++ct)
#pragma unroll
    for (int e = 0; e < 16; ++e) { acc[ct][e] = fm_x2_scalb(acc[ct][e], edk); av[ct][e] = fm_x2_scalb(av[ct][e], edv); }
  float* Os = reinterpret_cast<float*>(st);
  fm_x3_store<float, DH, QW, SPLIT, C::NTH, true>(acc, Os, sub, 32 * own + lr, lh, 1.0f, A.sc * (A.bpart ? kf : 1.0f), A.out, bh, t0, A.nk, tid, A.k,
                                          A.bpart ? A.bpart + int64_t(bh) * FM_GDIM_X + blk : nullptr, bad);
  fm_x3_store<float, DH, QW, SPLIT, C::NTH, true>(av, Os, sub, 32 * own + lr, lh, 1.0f, 1.0f, A.out2, bh, t0, A.nk, tid, A.k, nullptr, bad);
  return fm_x3_again(bad) && fm_x2_leave(1);
}
template <int DH, int SPLIT>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(512, 2) k_x2_dkv(X2Args A) {
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();                                           // (see k_x2_fwd)
  if (!fm_x2_dkv<DH, SPLIT>(A, reinterpret_cast<fm_half*>(smem), &bad)) FM_END();
  FM_SYNC();
  if (FM_TID_X == 0) bad = 0;
  FM_SYNC();
  fm_x3_dkv<float, DH, SPLIT, X3Row<DH>>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
  if (!fm_x3_again(&bad)) FM_END();
  fm_x3_dkv<float, DH, SPLIT, F32Row<DH>>(FM_ARGS_AGAIN(A), reinterpret_cast<uint16_t*>(smem), &bad, FM_TID_X + FM_OPAQUE_ZERO());
}
