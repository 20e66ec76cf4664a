// Dense fp32 attention on the bf16 matrix pipes, at fp32 accuracy.
//
// An fp32 number is the exact sum of three bfloat16 numbers, x = h + m + l: h is x rounded to 8 bits, m what is left
// rounded to 8 bits, l the rest (24 significant bits in all, each remainder formed exactly in fp32; bf16 has fp32's
// exponents).  A product of two such numbers is taken as
//     h h + (h m + m h) + (m m + h l + l h),
// six v_mfma_f32_32x32x16_bf16 with fp32 accumulation; the three products left out are below 2^-26 of |x y|, less than
// the 2^-24 of one fp32 rounding, and the pipe's rate is 16 / 6 of the fp32 instruction's.  N = 4096, D = 64, causal,
// relative error of o, dq, dk, dv against 64-bit results: v_mfma_f32_32x32x2_f32 3.9e-7, 4.7e-7, 4.8e-7, 4.0e-7; here 3.6e-7,
// 4.4e-7, 3.4e-7, 2.8e-7 (a sixth of the accumulator's roundings are fp32-sized, sixteen products to each).  Times at
// B*H = 32: forward 711 -> 370 us, dQ 1040 -> 520, dK and dV 1760 (two launches) -> 780, and the copies of 80 us are gone.
// The matrix instruction takes a bf16 number under 2^-126 for zero, which would cost a number below 2^-103 its lowest plane.
// So every operand, the weights and score gradients among them, is multiplied by UP = 2^24 before it is split: every fp32
// number, the subnormal ones included, then keeps all its bits.  The powers are taken out of the polynomials'
// coefficients and of the sums, all exactly: results are what they are without, bit for bit, wherever those keep 24 bits.
// At the other end an operand beyond 2^104 or a sum beyond 2^79 overflows; such workgroups work in fp32 (see fm_x3_look).
//
// Three kernels for problems without moment states: the forward, dQ (which first makes c = (dO / g) . o of its queries
// and leaves it for the next), dK and dV in one pass.  All read the caller's tensors; rows are scaled and split into
// the three planes on their way from registers to LDS, so nothing is converted in memory beforehand.
//
// A wavefront holds a tile of 32 own tokens (its fragments split once, in registers) and multiplies it with 32-token
// tiles of the other side staged in LDS as rows of three planes; transposed fragments come from transposing LDS reads.
// SPLIT: how many wavefronts share an own tile, each taking every SPLIT-th stream tile of a stage; their sums meet in
// LDS in a fixed order.  1 gives the fewest bytes per product, 2 and 4 spread a problem with few own tiles over more
// workgroups and wavefronts (see x3_split).
// What bounds them is the matrix pipe and the vector work beside it: per 32 x 32 tile pair and wavefront (D = 64) the
// forward issues 48 matrix instructions (1536 cycles) and about 140 vector instructions for the weights and their split.
// Long fp32 problems whose numbers two _Float16 planes hold are fm_x2.h's; short ones, bf16 tensors computed in fp32, unusual
// coefficients and the numbers that fm_x2.h refuses are made here.
#pragma once
#include "fm_kernels.h"
#include "fm_tok.h"

struct X3 { fm_u16x8 p[3]; };                          // eight numbers as three bf16 planes: h, m, l

// Splits eight floats (or eight accumulator entries).
FM_DEVICE X3 fm_x3_split(const float v[8]) {
  fm_u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      const uint32_t u = fm_cvt_pk_bf16(a, b);
      w[pl][i] = u;
      a -= fm_bits_f32(u << 16);
      b -= fm_bits_f32(u & 0xffff0000u);
    }
  }
  X3 r;
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) __builtin_memcpy(&r.p[pl], &w[pl], 16);
  return r;
}
FM_DEVICE X3 fm_x3_split_acc(const fm_f32x16& s, int half) {
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = s[8 * half + i];
  return fm_x3_split(v);
}
// small terms first
static constexpr int FM_X3_TERMS = 6;
FM_DEVICE constexpr int fm_x3_pa(int t) { return t == 0 ? 2 : t == 1 ? 0 : t == 2 ? 1 : t == 3 ? 1 : 0; }
FM_DEVICE constexpr int fm_x3_pb(int t) { return t == 0 ? 0 : t == 1 ? 2 : t == 2 ? 1 : t == 3 ? 0 : t == 4 ? 1 : 0; }
FM_DEVICE fm_f32x16 fm_x3_mma(const X3& a, const X3& b, fm_f32x16 c) {
#pragma unroll
  for (int t = 0; t < FM_X3_TERMS; ++t) c = fm_mfma_bf16(a.p[fm_x3_pa(t)], b.p[fm_x3_pb(t)], c);
  return c;
}

// transposed fragment of a row tile of 16-bit numbers: see Mma<fm_half>::load_tr
FM_DEVICE fm_u16x8 fm_bf16_load_tr(const uint16_t* tile, int pitch, int tok0, int col0, int lane) {
  const int lh = lane >> 5, half16 = (lane >> 4) & 1, s = (lane & 15) >> 2, q = lane & 3;
  const uint16_t* p = tile + (tok0 + 4 * lh + s) * pitch + col0 + 16 * half16 + 4 * q;
  const fm_u16x4 lo = fm_lds_tr4(p), hi = fm_lds_tr4(p + 8 * pitch);
  fm_u16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return r;
}

// How a kernel holds and multiplies its rows.  X3Row: three planes, the products above.  F32Row: fp32 rows and
// v_mfma_f32_32x32x2_f32, for the workgroups whose sums came out non-finite (see fm_x3_look).
//   Own              the lane's own token: CH features from feat(c, lh) in chunk c of NOWN
//   score, score2    score tile (rows = stream tokens, column = own token), and the second one beside it
//   accum, accum2    acc (rows = features) += rows of a stream tile times a weight tile, one product and two
template <int DH> struct X3Row {
  static constexpr int PQ = 3 * DH + 8;                // pitch of a staged row: three planes and 16 bytes of padding
  static constexpr float UP = 0x1p24f;                 // factor on every operand
  static constexpr bool PIPE = true;                   // the next stage is loaded while one is multiplied
  static constexpr int CH = 8, NOWN = DH / 16, NT = DH / 32;
  struct Own { X3 f[NOWN]; };
  static FM_DEVICE int feat(int c, int lh) { return 16 * c + 8 * lh; }
  template <typename TIO> static FM_DEVICE void ld(const TIO* p, float v[CH]) { IO<TIO>::ld8(p, v); }
  static FM_DEVICE void add_half(const fm_half* p, float v[CH]) {
    const fm_half8 h = *reinterpret_cast<const fm_half8*>(p);
#pragma unroll
    for (int i = 0; i < CH; ++i) v[i] += float(h[i]);
  }
  static FM_DEVICE void set(Own& o, int c, const float v[CH]) { o.f[c] = fm_x3_split(v); }
  static FM_DEVICE void fence(int) {}
  static FM_DEVICE X3 load(const uint16_t* p) {        // fragment of a row tile (p: the lane's row and features)
    X3 f;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) f.p[pl] = *reinterpret_cast<const fm_u16x8*>(p + pl * DH);
    return f;
  }
  static FM_DEVICE X3 load_tr(const uint16_t* tile, int tok0, int col0, int lane) {
    X3 f;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) f.p[pl] = fm_bf16_load_tr(tile + pl * DH, PQ, tok0, col0, lane);
    return f;
  }
  static FM_DEVICE void store(uint16_t* p, const X3& f) {
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<fm_u16x8*>(p + pl * DH) = f.p[pl];
  }
  static FM_DEVICE void put8(uint16_t* tile, int row, int col, const float w[8]) { store(tile + row * PQ + col, fm_x3_split(w)); }
  static FM_DEVICE void score(const uint16_t* X, int row, int lh, const Own& of, fm_f32x16& s) {
#pragma unroll
    for (int ks = 0; ks < NOWN; ++ks) s = fm_x3_mma(load(X + row * PQ + feat(ks, lh)), of.f[ks], s);
  }
  static FM_DEVICE void score2(const uint16_t* X, const uint16_t* Y, int row, int lh, const Own& of, const Own& of2, fm_f32x16& s,
                               fm_f32x16& dp) {
#pragma unroll
    for (int ks = 0; ks < NOWN; ++ks) terms2(load(X + row * PQ + feat(ks, lh)), of.f[ks], load(Y + row * PQ + feat(ks, lh)), of2.f[ks], s, dp);
  }
  // the second own row in LDS
  static FM_DEVICE void score2(const uint16_t* X, const uint16_t* Y, int row, int lh, const Own& of, const uint16_t* V, int vrow,
                               fm_f32x16& s, fm_f32x16& dp) {
#pragma unroll
    for (int ks = 0; ks < NOWN; ++ks)
      terms2(load(X + row * PQ + feat(ks, lh)), of.f[ks], load(Y + row * PQ + feat(ks, lh)), load(V + vrow * PQ + feat(ks, lh)), s, dp);
  }
  static FM_DEVICE void terms2(const X3& xf, const X3& of, const X3& yf, const X3& of2, fm_f32x16& s, fm_f32x16& dp) {
#pragma unroll
    for (int t = 0; t < FM_X3_TERMS; ++t) {
      s = fm_mfma_bf16(xf.p[fm_x3_pa(t)], of.p[fm_x3_pb(t)], s);
      dp = fm_mfma_bf16(yf.p[fm_x3_pa(t)], of2.p[fm_x3_pb(t)], dp);
    }
  }
  static FM_DEVICE void accum(fm_f32x16* acc, const uint16_t* Y, int tok0, const fm_f32x16& s, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const X3 pb = fm_x3_split_acc(s, h);
      X3 zf[NT];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) zf[ct] = load_tr(Y, tok0 + 16 * h, 32 * ct, lane);
#pragma unroll
      for (int t = 0; t < FM_X3_TERMS; ++t)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_mfma_bf16(zf[ct].p[fm_x3_pa(t)], pb.p[fm_x3_pb(t)], acc[ct]);
    }
  }
  // av += Y s, ak += X dp
  static FM_DEVICE void accum2(fm_f32x16* av, const uint16_t* Y, const fm_f32x16& s, fm_f32x16* ak, const uint16_t* X, const fm_f32x16& dp,
                               int tok0, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const X3 pb = fm_x3_split_acc(s, h), db = fm_x3_split_acc(dp, h);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        const X3 yt = load_tr(Y, tok0 + 16 * h, 32 * ct, lane), xt = load_tr(X, tok0 + 16 * h, 32 * ct, lane);
#pragma unroll
        for (int t = 0; t < FM_X3_TERMS; ++t) {
          av[ct] = fm_mfma_bf16(yt.p[fm_x3_pa(t)], pb.p[fm_x3_pb(t)], av[ct]);
          ak[ct] = fm_mfma_bf16(xt.p[fm_x3_pa(t)], db.p[fm_x3_pb(t)], ak[ct]);
        }
      }
    }
  }
};
template <int DH> struct F32Row {
  static constexpr int PQ = X3Row<DH>::PQ;             // the tiles lie where the planes lay
  static constexpr int PF = DH + 1;                    // a row in floats
  static_assert(2 * PF <= PQ, "a row of floats fits a row of planes");
  static constexpr float UP = 1.0f;
  static constexpr bool PIPE = false;                  // few registers: this code shares the allocation of the one above
  static constexpr int CH = 1, NOWN = DH / 2, NT = DH / 32;
  struct Own { float f[NOWN]; };
  static FM_DEVICE int feat(int c, int lh) { return 2 * c + lh; }
  template <typename TIO> static FM_DEVICE void ld(const TIO* p, float v[CH]) { v[0] = IO<TIO>::ld(p); }
  static FM_DEVICE void add_half(const fm_half* p, float v[CH]) { v[0] += float(*p); }
  static FM_DEVICE void set(Own& o, int c, const float v[CH]) { o.f[c] = v[0]; }
  static FM_DEVICE void fence(int c) { if (c % 4 == 0) FM_SCHED_FENCE(); }
  static FM_DEVICE const float* at(const uint16_t* tile, int row) { return reinterpret_cast<const float*>(tile) + row * PF; }
  static FM_DEVICE void put8(uint16_t* tile, int row, int col, const float w[8]) {
    float* p = reinterpret_cast<float*>(tile) + row * PF + col;
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = w[i];
  }
  static FM_DEVICE void score(const uint16_t* X, int row, int lh, const Own& of, fm_f32x16& s) {
    const float* x = at(X, row) + lh;
#pragma unroll
    for (int c = 0; c < NOWN; ++c) {
      fence(c);
      s = fm_mfma_f32(x[2 * c], of.f[c], s);
    }
  }
  static FM_DEVICE void score2(const uint16_t* X, const uint16_t* Y, int row, int lh, const Own& of, const Own& of2, fm_f32x16& s,
                               fm_f32x16& dp) {
    score(X, row, lh, of, s);
    score(Y, row, lh, of2, dp);
  }
  static FM_DEVICE void score2(const uint16_t* X, const uint16_t* Y, int row, int lh, const Own& of, const uint16_t* V, int vrow,
                               fm_f32x16& s, fm_f32x16& dp) {
    score(X, row, lh, of, s);
    const float *y = at(Y, row) + lh, *v = at(V, vrow) + lh;
#pragma unroll
    for (int c = 0; c < NOWN; ++c) {
      fence(c);
      dp = fm_mfma_f32(y[2 * c], v[2 * c], dp);
    }
  }
  static FM_DEVICE void accum(fm_f32x16* acc, const uint16_t* Y, int tok0, const fm_f32x16& s, int lane) {
    const float* y = at(Y, tok0) + (lane & 31);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      fence(e);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_mfma_f32(y[fm_acc_row(e, lane >> 5) * PF + 32 * ct], s[e], acc[ct]);
    }
  }
  static FM_DEVICE void accum2(fm_f32x16* av, const uint16_t* Y, const fm_f32x16& s, fm_f32x16* ak, const uint16_t* X, const fm_f32x16& dp,
                               int tok0, int lane) {
    accum(av, Y, tok0, s, lane);
    accum(ak, X, tok0, dp, lane);
  }
};

// An infinity, a NaN or a number that UP takes beyond bf16's largest comes out of the split as infinity and NaN, and
// whatever sum it enters as NaN.  So a thread looks at the
// sums it stores and, if one of the workgroup's is not finite, the workgroup makes its rows again with fp32 matrix products,
// over what it stored: an infinite value then gives the infinities and NaN that fp32 arithmetic gives.  bad: one flag in
// LDS, cleared at the kernel's start.  (A call of 8 us is bound by the length of its straight code: eight additions per
// eight sums and a barrier that does not wait for the stores.)
FM_DEVICE void fm_x3_look(int* bad, const float v[8], float g) {
  float z = fm_absf(g);
#pragma unroll
  for (int i = 0; i < 8; ++i) z += fm_absf(v[i]);
  if (!(z < 0x1p127f)) *bad = 1;
}
FM_DEVICE bool fm_x3_again(const int* bad) { FM_SYNC_LDS(); return __builtin_expect(FM_UNIFORM(*bad) != 0, 0); }

// The polynomials' coefficients where the score carries UP^2 and the result is to carry UP.
struct X3Coef { float a0, a1, a2; };                   // f(s) = a0 + s (a1 + a2 s)
template <typename R> FM_DEVICE X3Coef fm_x3_coef(float a0, float a1, float a2) {
  const X3Coef c = {a0 * R::UP, a1 / R::UP, a2 / (R::UP * R::UP * R::UP)};
  return c;
}
// A coefficient that this would take under fp32's normal numbers: fp32 matrix products from the start (X3Args::plain).
inline bool fm_x3_coef_lost(float a1, float a2) {
  typedef X3Row<64> R;
  const float least = 0x1p-126f, b1 = (a1 < 0 ? -a1 : a1) / R::UP, b2 = (a2 < 0 ? -a2 : a2) / (R::UP * R::UP * R::UP);
  return (a1 != 0.0f && b1 < least) || (a2 != 0.0f && b2 < least);
}

template <typename TIO> struct X3Args {
  TRef<const TIO> q, k, v, o, d_o;
  TRef<float> g;                        // written by the forward, read by the backward
  TRef<TIO> out, out2;                  // o | dq | dk and dv
  float* cv;                            // [bh][npad_q] c per query: written by dQ, read by dK + dV
  fm_half* out_resid; const fm_half* ores;   // bf16 tensors computed in fp32: what rounding takes from o (see TokArgs)
  int nq, nk, npad_q, causal;
  float a0, a1, a2, sc;                 // sc = sqrt(1/tau), on q and on k
  int plain;                            // see fm_x3_coef_lost
  int first;                            // causal, own queries: block 0 starts first, on three planes (see fm_x2_dq)
  NormFold q_fold, k_fold;
  float* bpart;                         // the Jacobian's partial sums (see TokArgs::bpart), or null
};

// Stage of ROWS stream rows of two tensors: caller's rows -> registers -> LDS planes.
template <typename TIO, int DH, typename R, int ROWS, int NTH> struct X3Stage {
  static constexpr int CPR = DH / 8, PER = ROWS * CPR, TOT = 2 * PER, N = (TOT + NTH - 1) / NTH;
  float r[N][8], gi[N];
  // gb: y rows are divided by g (null: not)
  FM_DEVICE void load(const TRef<const TIO>& x, const TRef<const TIO>& y, const TRef<float>* g, int bh, int row0, int n, int tid) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + NTH * i;
      if (TOT % NTH != 0 && c >= TOT) break;
      const bool second = c >= PER;                    // the same for a whole wavefront: PER is a multiple of 64
      const int cc = second ? c - PER : c, row = row0 + cc / CPR, col = (cc % CPR) * 8;
      gi[i] = 1.0f;
      if (row >= 0 && row < n) {
        const TRef<const TIO>& t = second ? y : x;
        IO<TIO>::ld8(t.base(bh) + int64_t(row) * t.s_n + col, r[i]);
        if (g && second) gi[i] = g->base(bh)[int64_t(row) * g->s_n];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) r[i][j] = 0.f;
      }
    }
  }
  FM_DEVICE void store(uint16_t* X, uint16_t* Y, float xs, bool div, int tid) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = tid + NTH * i;
      if (TOT % NTH != 0 && c >= TOT) break;
      const bool second = c >= PER;
      const int cc = second ? c - PER : c;
      const float f = second ? (div ? R::UP / gi[i] : R::UP) : xs;   // (xs has the factor already)
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = r[i][j] * f;
      R::put8(second ? Y : X, cc / CPR, (cc % CPR) * 8, w);
    }
  }
  // both steps at once, one piece after the other (few registers)
  static FM_DEVICE void copy(uint16_t* X, uint16_t* Y, const TRef<const TIO>& x, const TRef<const TIO>& y, const TRef<float>* g, int bh,
                             int row0, int n, float xs, int tid) {
#pragma unroll 1
    for (int c = tid; c < TOT; c += NTH) {
      const bool second = c >= PER;
      const int cc = second ? c - PER : c, row = row0 + cc / CPR, col = (cc % CPR) * 8;
      float w[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (row >= 0 && row < n) {
        const TRef<const TIO>& t = second ? y : x;
        IO<TIO>::ld8(t.base(bh) + int64_t(row) * t.s_n + col, w);
        const float f = second ? (g ? R::UP / g->base(bh)[int64_t(row) * g->s_n] : R::UP) : xs;
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] *= f;
      }
      R::put8(second ? Y : X, cc / CPR, col, w);
    }
  }
};

// Block of own tokens and batch*head of a workgroup: heaviest blocks first (late queries, early keys under the causal
// mask); with a multiple of eight batch*heads all blocks of one run behind one L2, dealt as in TokGeom.
FM_DEVICE void fm_x3_place(bool late_first, bool zero_first, int slots, int& blk, int& bh) {
  const int nblk = FM_GDIM_X, nbh = FM_GDIM_Y, id = FM_BID_X + nblk * FM_BID_Y;
  int unit;
  if ((nbh & 7) == 0) {
    const int nb = nbh >> 3, rank = fm_snake_rank(id >> 3, nblk * nb, slots);
    unit = rank / nb;
    bh = (id & 7) + 8 * (rank % nb);
  } else {
    unit = id / nbh;
    bh = id % nbh;
  }
  blk = !late_first ? unit : !zero_first ? nblk - 1 - unit : unit == 0 ? 0 : nblk - unit;
}

// rows of the stream tile (starting at s0) that the lane's own token (lo + lr) may see
template <int OWN> FM_DEVICE void fm_x3_window(fm_f32x16& p, bool causal, int s0, int lo, int lr, int lh, int n_str) {
  int wlo, whi;
  fm_tile_window<OWN>(causal, s0, lo, lr, n_str, wlo, whi);
#pragma unroll
  for (int e = 0; e < 16; ++e) { const int r = fm_acc_row(e, lh); if (r < wlo || r > whi) p[e] = 0.f; }
}

// Sum of many weights: a tile's sixteen as a tree, the tiles with the rounding of each addition carried on.  Denominators of 4096 weights are
// off by 2.3e-8 so, which is the rounding of the result; one weight after the other by 3.9e-7, a tree without the carry by 1.0e-7.
struct X3Sum {
  float s, c;
  FM_DEVICE void add(const fm_f32x16& w) {
    float t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = w[i] + w[i + 8];
#pragma unroll
    for (int n = 4; n > 0; n >>= 1)
#pragma unroll
      for (int i = 0; i < n; ++i) t[i] += t[i + n];
    const float y = t[0] - c, z = s + y;
    const float r = (z - s) - y;
    c = fm_absf(z) < 0x1p127f ? r : 0.f;               // a sum past fp32 stays what it is
    s = z;
  }
};
// The sums of a row's two lanes and SPLIT parts meet in the four floats behind Os's rows, added in 64 bits: what is rounded is g itself.
template <int DH, int QW> FM_DEVICE void fm_x3_put_sum(const X3Sum& w, float* Os, int sub, int row, int lh) {
  float* p = Os + (sub * QW + row) * (DH + 4) + DH + 2 * lh;
  p[0] = w.s; p[1] = w.c;
}
template <int DH, int QW, int SPLIT> FM_DEVICE float fm_x3_sum(const float* Os, int row) {
  double s = 0.0;
  float c = 0.f;
#pragma unroll
  for (int i = 0; i < SPLIT; ++i) {
    const fm_f32x4 w = *reinterpret_cast<const fm_f32x4*>(Os + (i * QW + row) * (DH + 4) + DH);
    s += double(w[0]) + double(w[2]);
    c += w[1] + w[3];
  }
  return float(s - double(c));
}

// Accumulators of all wavefronts -> Os [SPLIT][QW][DH + 4], rows summed over the SPLIT parts by fm_x3_sum8.
template <int DH, int QW>
FM_DEVICE void fm_x3_put(const fm_f32x16* acc, float* Os, int sub, int row, int lh) {
  constexpr int OP = DH + 4;
#pragma unroll
  for (int ct = 0; ct < DH / 32; ++ct)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const fm_f32x4 w = {acc[ct][4 * g], acc[ct][4 * g + 1], acc[ct][4 * g + 2], acc[ct][4 * g + 3]};
      *reinterpret_cast<fm_f32x4*>(Os + (sub * QW + row) * OP + 32 * ct + fm_acc_row(4 * g, lh)) = w;
    }
}
template <int DH, int QW, int SPLIT> FM_DEVICE void fm_x3_sum8(const float* Os, int row, int col, float v[8]) {
  constexpr int OP = DH + 4;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = 0.f;
#pragma unroll
  for (int s = 0; s < SPLIT; ++s) {
    const float* p = Os + (s * QW + row) * OP + col;
    const fm_f32x4 a = *reinterpret_cast<const fm_f32x4*>(p), b = *reinterpret_cast<const fm_f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] += a[i]; v[4 + i] += b[i]; }
  }
}
// Gradient rows of the workgroup -> caller's tensor, times scale.  bout: the sum of stored value times raw row (the
// normalisation's B: stored = fac dy, y = fac x, so dy . y = stored . x), one float per workgroup, or null.  unscale: takes a power
// of two out of the sums first.  LOOK, bad: see fm_x3_look.
template <typename TIO, int DH, int QW, int SPLIT, int NTH, bool LOOK>
FM_DEVICE void fm_x3_store(const fm_f32x16* acc, float* Os, int sub, int row, int lh, float unscale, float scale, const TRef<TIO>& out,
                           int bh, int t0, int n, int tid, const TRef<const TIO>& raw, float* bout, int* bad) {
  FM_SYNC();                                           // whatever lay there has been read
  fm_x3_put<DH, QW>(acc, Os, sub, row, lh);
  FM_SYNC();
  float bsum = 0.f;
  for (int c = tid; c < QW * (DH / 8); c += NTH) {
    const int r = c / (DH / 8), col = (c % (DH / 8)) * 8;
    if (t0 + r >= n) continue;
    float v[8];
    fm_x3_sum8<DH, QW, SPLIT>(Os, r, col, v);
    if (LOOK) fm_x3_look(bad, v, 0.f);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * unscale * scale;
    if (bout) {
      float x[8];
      IO<TIO>::ld8(raw.base(bh) + int64_t(t0 + r) * raw.s_n + col, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) bsum += v[i] * x[i];
    }
    IO<TIO>::st8(out.base(bh) + int64_t(t0 + r) * out.s_n + col, v);
  }
  if (bout) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) bsum += fm_shfl_xor(bsum, m);
    FM_SYNC();
    if ((tid & 63) == 0) Os[tid >> 6] = bsum;
    FM_SYNC();
    if (tid == 0) {
      float b = 0.f;
      for (int w = 0; w < NTH / 64; ++w) b += Os[w];
      *bout = b;
    }
  }
}

template <int DH, int NW, int SPLIT> struct X3Cfg {
  static constexpr int NTH = 64 * NW, OT = NW / SPLIT, QW = 32 * OT, KT = 32 * SPLIT, PQ = X3Row<DH>::PQ;
  static constexpr int STAGE = 2 * KT * PQ;            // u16 elements of one stage buffer
  static constexpr int NBUF = 2 * STAGE * 2 <= 112 * 1024 ? 2 : 1;
  static constexpr size_t OS = size_t(SPLIT) * QW * (DH + 4) * 4;
  // kind 0: forward, dQ; 1: dK + dV (own v rows and the stages' c values as well)
  static constexpr size_t lds(int kind) {
    const size_t a = size_t(NBUF) * STAGE * 2 + (kind ? size_t(QW) * PQ * 2 + size_t(NBUF) * KT * 4 : 0);
    return a > OS ? a : OS;
  }
  static constexpr int SLOTS = NW == 8 ? 1 : 2;        // workgroups of a CU, see fm_snake_rank
  static constexpr int OCC = NW == 8 || NBUF == 1 || 2 * (NBUF * STAGE * 2) > 150 * 1024 ? NW / 4 : DH == 32 && SPLIT == 1 ? 3 : 2;   // wavefronts per SIMD
};

// ------------------------------------------------------------------------------
// forward.  grid (ceil(nq / QW), bh).
// ------------------------------------------------------------------------------
// FIRST: called by a kernel of fm_x2.h, whose order of blocks A.first names.
template <typename TIO, int DH, int SPLIT, typename R, int NW, bool FIRST = false>
FM_DEVICE void fm_x3_fwd(const X3Args<TIO>& A, uint16_t* st, int* bad, const int tid) {
  typedef X3Cfg<DH, NW, SPLIT> C;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  const int lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(causal, FIRST && A.first != 0, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const float qs = A.sc * fm_norm_factor(A.q_fold, bh, lane) * R::UP, ks_ = A.sc * fm_norm_factor(A.k_fold, bh, lane) * R::UP;
  const X3Coef cf = fm_x3_coef<R>(A.a0, A.a1, A.a2);
  const int send = causal && t0 + QW < A.nk ? t0 + QW : A.nk;
  typedef X3Stage<TIO, DH, R, KT, C::NTH> Stage;
  Stage sg;
  if (R::PIPE) sg.load(A.k, A.v, nullptr, bh, 0, A.nk, tid);
  typename R::Own of;
  {
    const bool in = lo + lr < A.nq;
    const TIO* qr = A.q.base(bh) + int64_t(in ? lo + lr : A.nq - 1) * A.q.s_n;
#pragma unroll
    for (int c = 0; c < R::NOWN; ++c) {
      R::fence(c);
      float v[R::CH];
      R::ld(qr + R::feat(c, lh), v);
#pragma unroll
      for (int i = 0; i < R::CH; ++i) v[i] = in ? v[i] * qs : 0.f;
      R::set(of, c, v);
    }
  }
  fm_f32x16 acc[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_zero16();
  X3Sum gsum = {0.f, 0.f};
  constexpr bool TWO = R::PIPE && C::NBUF == 2;
  // Shared own tiles are short problems, bound by their straight code: there the walk starts one stage early, for that stage's
  // store alone, and the code of a store is there once (570 of 3090 instructions; 256 tokens, D = 32, B*H = 2, whole call 8.98 ->
  // 8.65 us).  A long walk is about 1 % faster with a first store of its own (headline forward, over the same kernel without
  // its second pass in turn on one box: 1.006 with the early start, 0.997 without).
  constexpr bool EARLY = TWO && SPLIT > 1;
  int buf = EARLY ? 1 : 0;
  if (TWO && !EARLY) {
    sg.store(st, st + KT * PQ, ks_, false, tid);
    sg.load(A.k, A.v, nullptr, bh, KT, A.nk, tid);
  }
  for (int s0 = EARLY ? -KT : 0; s0 < send; s0 += KT) {
    uint16_t* X = st + buf * C::STAGE;
    uint16_t* Y = X + KT * PQ;
    if (!R::PIPE) Stage::copy(X, Y, A.k, A.v, nullptr, bh, s0, A.nk, ks_, tid);
    else if (!TWO) sg.store(X, Y, ks_, false, tid);
    if (!EARLY || s0 >= 0) FM_SYNC();
    if (R::PIPE && !TWO) sg.load(A.k, A.v, nullptr, bh, s0 + KT, A.nk, tid);
    const int ss0 = s0 + 32 * sub;
    if ((!EARLY || s0 >= 0) && ss0 < A.nk && !(causal && ss0 > lo + 31)) {
      fm_f32x16 s = fm_zero16();
      R::score(X, 32 * sub + lr, lh, of, s);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = cf.a0 + s[e] * (cf.a1 + cf.a2 * s[e]);
      if (fm_tile_edge<FM_OWN_Q>(causal, ss0, lo, A.nk)) { FM_KEEP_BRANCH(); fm_x3_window<FM_OWN_Q>(s, causal, ss0, lo, lr, lh, A.nk); }
      gsum.add(s);
      R::accum(acc, Y, 32 * sub, s, lane);
    }
    if (TWO) {
      buf ^= 1;
      if (s0 + KT < send) {
        sg.store(st + buf * C::STAGE, st + buf * C::STAGE + KT * PQ, ks_, false, tid);
        sg.load(A.k, A.v, nullptr, bh, s0 + 2 * KT, A.nk, tid);
      }
    } else FM_SYNC();
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
    float gt = fm_x3_sum<DH, QW, SPLIT>(Os, r);
    if (R::PIPE) fm_x3_look(bad, v, gt);
    gt *= 1.0f / R::UP;
    const float gi = 1.0f / gt;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * (1.0f / (R::UP * R::UP)) * gi;
    IO<TIO>::st8(A.out.base(bh) + int64_t(qi) * A.out.s_n + col, v);
    if (A.out_resid) {
      float sv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[i] = fm_as_stored<TIO>(v[i]);
      fm_store_resid8(A.out_resid + (int64_t(bh) * A.npad_q + qi) * DH + col, v, sv);
    }
    if (col == 0) A.g.base(bh)[int64_t(qi) * A.g.s_n] = gt;
  }
}
template <typename TIO, int DH, int SPLIT, int NW>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(64 * NW, (X3Cfg<DH, NW, SPLIT>::OCC)) k_x3_fwd(X3Args<TIO> A) {
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  uint16_t* st = reinterpret_cast<uint16_t*>(smem);
  if (FM_TID_X == 0) bad = 0;
  if (!A.plain) {
    fm_x3_fwd<TIO, DH, SPLIT, X3Row<DH>, NW>(A, st, &bad, FM_TID_X);
    if (!fm_x3_again(&bad)) FM_END();
  }
  fm_x3_fwd<TIO, DH, SPLIT, F32Row<DH>, NW>(FM_ARGS_AGAIN(A), st, &bad, FM_TID_X + FM_OPAQUE_ZERO());
}

// ------------------------------------------------------------------------------
// dQ.  grid (ceil(nq / QW), bh).  dS = (a1 + 2 a2 s) (gh . v - c), gh = dO / g, c = gh . o.
// ------------------------------------------------------------------------------
template <typename TIO, int DH, int SPLIT, typename R, int NW, bool FIRST = false>
FM_DEVICE void fm_x3_dq(const X3Args<TIO>& A, uint16_t* st, int* bad, const int tid) {
  typedef X3Cfg<DH, NW, SPLIT> C;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  const int lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(causal, FIRST && A.first != 0, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const float qf = fm_norm_factor(A.q_fold, bh, lane), qs = A.sc * qf * R::UP, ks_ = A.sc * fm_norm_factor(A.k_fold, bh, lane) * R::UP;
  const int send = causal && t0 + QW < A.nk ? t0 + QW : A.nk;
  typedef X3Stage<TIO, DH, R, KT, C::NTH> Stage;
  Stage sg;
  if (R::PIPE) sg.load(A.k, A.v, nullptr, bh, 0, A.nk, tid);
  typename R::Own of, of2;
  float cs = 0.f;
  {
    const bool in = lo + lr < A.nq;
    const int64_t row = in ? lo + lr : A.nq - 1;
    const float ginv = in ? R::UP / A.g.base(bh)[row * A.g.s_n] : 0.f;
#pragma unroll
    for (int c = 0; c < R::NOWN; ++c) {
      R::fence(c);
      const int f = R::feat(c, lh);
      float v[R::CH], w[R::CH], o[R::CH];
      R::ld(A.q.base(bh) + row * A.q.s_n + f, v);
      R::ld(A.d_o.base(bh) + row * A.d_o.s_n + f, w);
      R::ld(A.o.base(bh) + row * A.o.s_n + f, o);
      if (A.ores) R::add_half(A.ores + (int64_t(bh) * A.npad_q + row) * DH + f, o);
#pragma unroll
      for (int i = 0; i < R::CH; ++i) { v[i] = in ? v[i] * qs : 0.f; w[i] = in ? w[i] * ginv : 0.f; cs += w[i] * o[i]; }
      R::set(of, c, v);
      R::set(of2, c, w);
    }
    cs += fm_shfl_xor(cs, 32);
    if (sub == 0 && lh == 0 && in) A.cv[int64_t(bh) * A.npad_q + row] = cs * (1.0f / R::UP);
    cs *= R::UP;                                       // as gh . v
  }
  const X3Coef cf = fm_x3_coef<R>(0.0f, A.a1, 2.0f * A.a2);
  fm_f32x16 acc[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) acc[ct] = fm_zero16();
  constexpr bool TWO = R::PIPE && C::NBUF == 2;
  int buf = 0;
  if (TWO) {
    sg.store(st, st + KT * PQ, ks_, false, tid);
    sg.load(A.k, A.v, nullptr, bh, KT, A.nk, tid);
  }
  for (int s0 = 0; s0 < send; s0 += KT) {
    uint16_t* X = st + buf * C::STAGE;
    uint16_t* Y = X + KT * PQ;
    if (!R::PIPE) Stage::copy(X, Y, A.k, A.v, nullptr, bh, s0, A.nk, ks_, tid);
    else if (!TWO) sg.store(X, Y, ks_, false, tid);
    FM_SYNC();
    if (R::PIPE && !TWO) sg.load(A.k, A.v, nullptr, bh, s0 + KT, A.nk, tid);
    const int ss0 = s0 + 32 * sub;
    if (ss0 < A.nk && !(causal && ss0 > lo + 31)) {
      fm_f32x16 s = fm_zero16(), dp = fm_zero16();
      R::score2(X, Y, 32 * sub + lr, lh, of, of2, s, dp);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = (cf.a1 + cf.a2 * s[e]) * (dp[e] - cs);
      if (fm_tile_edge<FM_OWN_Q>(causal, ss0, lo, A.nk)) { FM_KEEP_BRANCH(); fm_x3_window<FM_OWN_Q>(s, causal, ss0, lo, lr, lh, A.nk); }
      R::accum(acc, X, 32 * sub, s, lane);
    }
    if (TWO) {
      buf ^= 1;
      if (s0 + KT < send) {
        sg.store(st + buf * C::STAGE, st + buf * C::STAGE + KT * PQ, ks_, false, tid);
        sg.load(A.k, A.v, nullptr, bh, s0 + 2 * KT, A.nk, tid);
      }
    } else FM_SYNC();
  }
  fm_x3_store<TIO, DH, QW, SPLIT, C::NTH, R::PIPE>(acc, reinterpret_cast<float*>(st), sub, 32 * own + lr, lh, 1.0f / (R::UP * R::UP), A.sc * (A.bpart ? qf : 1.0f), A.out,
                                          bh, t0, A.nq, tid, A.q, A.bpart ? A.bpart + int64_t(bh) * FM_GDIM_X + blk : nullptr, bad);
}
template <typename TIO, int DH, int SPLIT, int NW>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(64 * NW, (X3Cfg<DH, NW, SPLIT>::OCC)) k_x3_dq(X3Args<TIO> A) {
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  uint16_t* st = reinterpret_cast<uint16_t*>(smem);
  if (FM_TID_X == 0) bad = 0;
  if (!A.plain) {
    fm_x3_dq<TIO, DH, SPLIT, X3Row<DH>, NW>(A, st, &bad, FM_TID_X);
    if (!fm_x3_again(&bad)) FM_END();
  }
  fm_x3_dq<TIO, DH, SPLIT, F32Row<DH>, NW>(FM_ARGS_AGAIN(A), st, &bad, FM_TID_X + FM_OPAQUE_ZERO());
}

// ------------------------------------------------------------------------------
// dK and dV.  grid (ceil(nk / QW), bh), 512 threads: eight wavefronts share the staged queries, so that two per SIMD
// leave 256 registers each; own k in registers, own v (read once per tile) in LDS.
// ------------------------------------------------------------------------------
template <typename TIO, int DH, int SPLIT, typename R>
FM_DEVICE void fm_x3_dkv(const X3Args<TIO>& A, uint16_t* Vs, int* bad, const int tid) {
  typedef X3Cfg<DH, 8, SPLIT> C;
  constexpr int NT = DH / 32, PQ = C::PQ, KT = C::KT, QW = C::QW;
  uint16_t* st = Vs + QW * PQ;                         // Vs: own v rows [QW][PQ]
  float* cst = reinterpret_cast<float*>(st + C::NBUF * C::STAGE);   // c of the staged queries [NBUF][KT]
  const int lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = FM_UNIFORM(tid >> 6), own = wave / SPLIT, sub = wave % SPLIT;
  const bool causal = A.causal != 0;
  int blk, bh;
  fm_x3_place(false, false, C::SLOTS, blk, bh);
  const int t0 = blk * QW, lo = t0 + 32 * own;
  const float kf = fm_norm_factor(A.k_fold, bh, lane), ks_ = A.sc * kf * R::UP, qs = A.sc * fm_norm_factor(A.q_fold, bh, lane) * R::UP;
  const int sbeg = causal ? t0 : 0, nst = (A.nq - sbeg + KT - 1) / KT;
  const int s_last = sbeg + (nst - 1) * KT;            // the stream is walked from its end: see k_ds
  typedef X3Stage<TIO, DH, R, KT, C::NTH> Stage;
  Stage sg;
  float creg = 0.f;
  const float* cvb = A.cv + int64_t(bh) * A.npad_q;
  auto fetch = [&](int s) FM_ALWAYS_INLINE {
    sg.load(A.q, A.d_o, &A.g, bh, s, A.nq, tid);
    const int r = s + tid % KT;
    creg = r >= 0 && r < A.nq ? cvb[r] : 0.f;
  };
  auto put = [&](int b) FM_ALWAYS_INLINE {
    uint16_t* X = st + b * C::STAGE;
    sg.store(X, X + KT * PQ, qs, true, tid);
    if (tid < KT) cst[b * KT + tid] = creg * (R::UP * R::UP);
  };
  if (R::PIPE) fetch(s_last);
  for (int c = tid; c < QW * (DH / 8); c += C::NTH) {
    const int r = c / (DH / 8), col = (c % (DH / 8)) * 8, row = t0 + r;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (row < A.nk) IO<TIO>::ld8(A.v.base(bh) + int64_t(row) * A.v.s_n + col, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= R::UP;
    R::put8(Vs, r, col, v);
  }
  typename R::Own of;
  {
    const bool in = lo + lr < A.nk;
    const TIO* kr = A.k.base(bh) + int64_t(in ? lo + lr : A.nk - 1) * A.k.s_n;
#pragma unroll
    for (int c = 0; c < R::NOWN; ++c) {
      R::fence(c);
      float v[R::CH];
      R::ld(kr + R::feat(c, lh), v);
#pragma unroll
      for (int i = 0; i < R::CH; ++i) v[i] = in ? v[i] * ks_ : 0.f;
      R::set(of, c, v);
    }
  }
  const X3Coef cp = fm_x3_coef<R>(A.a0, A.a1, A.a2), cd = fm_x3_coef<R>(0.0f, A.a1, 2.0f * A.a2);
  fm_f32x16 acc[NT], av[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) { acc[ct] = fm_zero16(); av[ct] = fm_zero16(); }
  constexpr bool TWO = R::PIPE && C::NBUF == 2;
  int buf = 0;
  if (TWO) { put(0); fetch(s_last - KT); }
  for (int s0 = s_last; s0 >= sbeg; s0 -= KT) {
    uint16_t* X = st + buf * C::STAGE;
    uint16_t* Y = X + KT * PQ;
    if (!R::PIPE) {
      Stage::copy(X, Y, A.q, A.d_o, &A.g, bh, s0, A.nq, qs, tid);
      if (tid < KT) cst[tid] = s0 + tid < A.nq ? cvb[s0 + tid] : 0.f;
    } else if (!TWO) put(0);
    FM_SYNC();
    if (R::PIPE && !TWO) fetch(s0 - KT);
    const int ss0 = s0 + 32 * sub;
    if (ss0 < A.nq && !(causal && ss0 + 31 < lo)) {
      fm_f32x16 s = fm_zero16(), dp = fm_zero16();
      R::score2(X, Y, 32 * sub + lr, lh, of, Vs, 32 * own + lr, s, dp);
      const float* cf = cst + buf * KT + 32 * sub + 4 * lh;
      // dp becomes dS, s becomes P
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const fm_f32x4 c4 = *reinterpret_cast<const fm_f32x4*>(cf + 8 * g4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 4 * g4 + i;
          const float x = s[e];
          dp[e] = (cd.a1 + cd.a2 * x) * (dp[e] - c4[i]);
          s[e] = cp.a0 + x * (cp.a1 + cp.a2 * x);
        }
      }
      if (fm_tile_edge<FM_OWN_K>(causal, ss0, lo, A.nq)) {
        FM_KEEP_BRANCH();
        fm_x3_window<FM_OWN_K>(s, causal, ss0, lo, lr, lh, A.nq);
        fm_x3_window<FM_OWN_K>(dp, causal, ss0, lo, lr, lh, A.nq);
      }
      R::accum2(av, Y, s, acc, X, dp, 32 * sub, lane);
    }
    if (TWO) {
      buf ^= 1;
      if (s0 - KT >= sbeg) { put(buf); fetch(s0 - 2 * KT); }
    } else FM_SYNC();
  }
  float* Os = reinterpret_cast<float*>(Vs);
  fm_x3_store<TIO, DH, QW, SPLIT, C::NTH, R::PIPE>(acc, Os, sub, 32 * own + lr, lh, 1.0f / (R::UP * R::UP), A.sc * (A.bpart ? kf : 1.0f), A.out, bh, t0, A.nk, tid, A.k,
                                          A.bpart ? A.bpart + int64_t(bh) * FM_GDIM_X + blk : nullptr, bad);
  fm_x3_store<TIO, DH, QW, SPLIT, C::NTH, R::PIPE>(av, Os, sub, 32 * own + lr, lh, 1.0f / (R::UP * R::UP), 1.0f, A.out2, bh, t0, A.nk, tid, A.k, nullptr, bad);
}
template <typename TIO, int DH, int SPLIT>
FM_GLOBAL void FM_LAUNCH_BOUNDS2(512, 2) k_x3_dkv(X3Args<TIO> A) {
  FM_DYN_SMEM(smem);
  FM_SHARED int bad;
  uint16_t* st = reinterpret_cast<uint16_t*>(smem);
  if (FM_TID_X == 0) bad = 0;
  if (!A.plain) {
    fm_x3_dkv<TIO, DH, SPLIT, X3Row<DH>>(A, st, &bad, FM_TID_X);
    if (!fm_x3_again(&bad)) FM_END();
  }
  fm_x3_dkv<TIO, DH, SPLIT, F32Row<DH>>(FM_ARGS_AGAIN(A), st, &bad, FM_TID_X + FM_OPAQUE_ZERO());
}
