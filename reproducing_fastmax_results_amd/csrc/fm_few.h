// Forward of a few queries against many keys: a decoding step over cached keys and values (one query, causal, every
// key visible; reference eval.generate_text, transformer/eval.py:8-32, and the nk > nq alignment of
// fastmax_cuda_forward.cu:161-172) and short blocks of new tokens.
//
// Bound by one read of k and v.  The general route has a 128-query tile per workgroup: with one query it ran one
// workgroup per batch*head over all keys, after copying k and v to the compute type, in two parts and a merge (six
// launches).  Here the keys are split over the grid and taken straight from the caller's tensors with fp32
// arithmetic on the vector units: LPR = DH / 8 lanes hold one key row (eight features, one 16-byte load of bf16),
// a wavefront 64 / LPR rows; a score is eight multiply-adds and log2(LPR) lane exchanges, and the same lane
// already holds the eight features of v that it multiplies by the weight.  No LDS in the loop, no barrier.
// B*H = 32, one query on 4097 cached keys, D = 64, bf16 (33.6 MB): 73.9 -> 11.5 us, two launches.
#pragma once
#include "fm_kernels.h"

static constexpr int FM_FEW_MAX_SPLITS = 64;
// queries that share one pass over the keys: registers 16 per query
inline int fm_few_group(int nq) { return nq >= 4 ? 4 : nq; }
inline int fm_few_groups(int nq) { return (nq + fm_few_group(nq) - 1) / fm_few_group(nq); }
// Queries the route takes.  Its work per key grows with the query groups while the general route's does not until 128
// queries, but the general route has one workgroup per batch*head.  bf16, D = 64, general route and this one, microseconds:
//   B*H = 32, 4097 keys:    1 query 73.9, 11.5;   16 queries 74.1, 27.7
//   B*H = 64, 16384 keys:   1 query 657, 43 (6.2 TB/s);   16 queries 657, 146
//   B*H = 8, 1024 keys:     64 queries 30, 14.7;     B*H = 16, 16384 keys:   64 queries 186, 139;   B*H = 32, 4097 keys:   74, 77
// So up to 64 queries while there are few batch*heads, and otherwise, on _Float16 arithmetic (`half`), what pays on a full chip:
// up to eight queries, and up to sixteen where the general route walks moment states or, under the mask, runs in two parts on
// few keys.  Times there of this route over the general one's (whole calls, B*H = 128 .. 4096, 17 .. 16384 keys): 1 to 4 queries
// 0.07 .. 0.9; 8 queries 0.15 .. 0.99; 16 queries on dense tiles 1.05 .. 1.5 (D = 32, B*H = 128: 0.83 .. 0.91, 12 queries there
// 0.92 .. 1.08), on states 0.26 .. 0.9, under the mask 0.35 .. 1.0 up to 1024 groups or 300 keys and 1.1 .. 1.2 beyond, 12 queries
// 0.7 .. 0.96 up to 1024 keys and 1.09 at
// 4096.  Up to 64 keys (`tiny`) the general route is fm_small.h, one launch: more than one group up to 1024 groups
// (B*H = 4096, 16 queries on 17 keys, D = 32: 117 us here, 12 there).
// fp32 arithmetic takes the route up to sixteen queries everywhere.
inline bool fm_few_pays(int bh, int nq, int nk, int d, bool half, bool tiny, bool split, bool states) {
  if (nq > 16 || !half) return nq <= 16 || (nq <= 64 && !tiny && bh * nq <= 1024);
  const int groups = fm_few_groups(nq);
  if (groups == 1) return true;
  if (tiny) return bh * groups <= 1024;
  if (groups == 2) return true;
  if (split) return bh * groups <= 1024 || nk <= (groups == 3 ? 2048 : 512);
  return states || bh * nq <= (d == 32 && groups == 4 ? 2048 : 1024);
}
// Parts the keys of a batch*head are cut into: enough workgroups for four per CU, about 64 keys or more in each (a count is
// rounded up: 577 keys may go in 16 parts of 37), and no more than one wavefront of the merge reads in one go.
inline int fm_few_splits(int bh, int nq, int nk) {
  const int groups = fm_few_groups(nq);
  int s = (1024 + bh * groups - 1) / (bh * groups);
  const int most = (nk + 63) / 64;
  if (s > most) s = most;
  // a power of two or a multiple of the eight XCDs: the groups that read the same keys then run behind one L2, or two (see
  // k_few's grid; B*H = 64, 12 queries on 1024 keys, whole call: 6 parts 28.1 us, 8 parts 23.4); up to eight parts not at
  // the price of shorter ones (300 keys: 5 parts 15.7 us, 8 parts 19.6)
  const int even = s > 4 ? (s + 7) / 8 * 8 : s == 3 ? 4 : s;
  if (s > 8 || even <= most) s = even;
  if (s > FM_FEW_MAX_SPLITS) s = FM_FEW_MAX_SPLITS;
  return s < 1 ? 1 : s;
}

template <typename TIO> struct FewArgs {
  TRef<const TIO> q, k, v;
  TRef<TIO> o; TRef<float> g;
  float* part;                  // [bh][nq][splits][DH + 1]: sums of f v and of f; null: one part, results written at once
  int nq, nk, causal;
  float a0, a1, a2, inv_tau;
  NormFold q_fold, k_fold;
};

// grid (splits * query groups, bh), 256 threads.  The groups that read the same keys lie nsplit workgroups apart: behind
// one L2 when nsplit is a multiple of the eight XCDs, and at about the same time.
template <typename TIO, int DH, int NQ>
FM_GLOBAL void FM_LAUNCH_BOUNDS(FM_THREADS) k_few(FewArgs<TIO> A, int nsplit) {
  constexpr int LPR = DH / 8, RPW = 64 / LPR;          // lanes per key row, rows per wavefront and load
  constexpr int U = NQ >= 3 ? 2 : 4;                   // rows in flight per lane; more queries leave fewer registers
  FM_SHARED float red[4][NQ][DH + 1];
  const int tid = FM_TID_X, lane = tid & 63, part = lane % LPR, row = lane / LPR, d0 = part * 8;
  const int wave = FM_UNIFORM(tid >> 6);
  const int split = FM_BID_X % nsplit, bh = FM_BID_Y, q0 = (FM_BID_X / nsplit) * NQ;
  const int per = (A.nk + nsplit - 1) / nsplit;
  const int kb = split * per, ke = kb + per < A.nk ? kb + per : A.nk;
  const float sc = A.inv_tau * fm_norm_factor(A.q_fold, bh, lane) * fm_norm_factor(A.k_fold, bh, lane);
  float qv[NQ][8], acc[NQ][8], gs[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int qi = q0 + i < A.nq ? q0 + i : A.nq - 1;
    IO<TIO>::ld8(A.q.base(bh) + int64_t(qi) * A.q.s_n + d0, qv[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) { qv[i][j] *= sc; acc[i][j] = 0.f; }
    gs[i] = 0.f;
  }
  const TIO* kp = A.k.base(bh) + d0;
  const TIO* vp = A.v.base(bh) + d0;
  const int see = A.causal ? A.nk - A.nq + q0 : A.nk;  // last key of query q0 + i: see + i
  for (int b = kb + wave * (RPW * U); b < ke; b += 4 * RPW * U) {
    float kx[U][8], vx[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = b + u * RPW + row, tc = t < ke ? t : ke - 1;
      IO<TIO>::ld8(kp + int64_t(tc) * A.k.s_n, kx[u]);
      IO<TIO>::ld8(vp + int64_t(tc) * A.v.s_n, vx[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = b + u * RPW + row;
      if (t >= ke) {                                   // past the part's end: zero times an infinite entry would be NaN
#pragma unroll
        for (int j = 0; j < 8; ++j) vx[u][j] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) s += qv[i][j] * kx[u][j];
        s = fm_group_sum<LPR>(s);
        float f = A.a0 + s * (A.a1 + A.a2 * s);
        if (t >= ke || t > see + i) f = 0.f;
        gs[i] += f;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] += f * vx[u][j];
      }
    }
  }
  // rows of the wavefront, then the four wavefronts
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
#pragma unroll
    for (int m = LPR; m < 64; m <<= 1) {
      gs[i] += fm_shfl_xor(gs[i], m);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] += fm_shfl_xor(acc[i][j], m);
    }
    if (row == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) red[wave][i][d0 + j] = acc[i][j];
      if (part == 0) red[wave][i][DH] = gs[i];
    }
  }
  FM_SYNC();
  for (int c = tid; c < NQ * (DH + 1); c += FM_THREADS) {
    const int i = c / (DH + 1), f = c % (DH + 1), qi = q0 + i;
    if (qi >= A.nq) continue;
    const float x = (red[0][i][f] + red[1][i][f]) + (red[2][i][f] + red[3][i][f]);
    if (A.part) {
      A.part[((int64_t(bh) * A.nq + qi) * nsplit + split) * (DH + 1) + f] = x;
    } else {
      const float gt = (red[0][i][DH] + red[1][i][DH]) + (red[2][i][DH] + red[3][i][DH]);
      if (f == DH) A.g.base(bh)[int64_t(qi) * A.g.s_n] = gt;
      else IO<TIO>::st(A.o.base(bh) + int64_t(qi) * A.o.s_n + f, x / gt);
    }
  }
}

// Sums the parts of one query in a fixed order and divides.  grid (nq, bh), 256 threads: 256 / DH groups of
// DH lanes, a lane one feature of every 256 / DH-th part.
template <typename TIO, int DH>
FM_GLOBAL void FM_LAUNCH_BOUNDS(256) k_few_merge(FewArgs<TIO> A, int nsplit) {
  constexpr int NG = 256 / DH;                         // groups of lanes, each sums every NG-th part
  FM_SHARED float red[NG][DH], redg[NG];
  const int tid = FM_TID_X, f = tid % DH, grp = tid / DH, qi = FM_BID_X, bh = FM_BID_Y;
  const float* p = A.part + (int64_t(bh) * A.nq + qi) * nsplit * (DH + 1);
  constexpr int U = FM_FEW_MAX_SPLITS / NG;            // every load of a thread is issued before the first sum
  float x[U], y[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int s = grp + u * NG;
    x[u] = s < nsplit ? p[s * (DH + 1) + f] : 0.f;
    y[u] = s < nsplit ? p[s * (DH + 1) + DH] : 0.f;
  }
  float a = 0.f, b = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) { a += x[u]; b += y[u]; }
  red[grp][f] = a;
  if (f == 0) redg[grp] = b;
  FM_SYNC();
  if (grp != 0) return;
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int i = 0; i < NG; ++i) { num += red[i][f]; den += redg[i]; }
  IO<TIO>::st(A.o.base(bh) + int64_t(qi) * A.o.s_n + f, num / den);
  if (f == 0) A.g.base(bh)[int64_t(qi) * A.g.s_n] = den;
}
