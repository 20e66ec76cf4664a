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

// Queries the route takes.  Its work per key grows with the queries while the general route's does not until 128, but
// the general route has one workgroup per batch*head.  bf16, D = 64, general route and this one, microseconds:
//   B*H = 32, 4097 keys:    1 query 73.9, 11.5;   16 queries 74.1, 27.7
//   B*H = 64, 16384 keys:   1 query 657, 43 (6.2 TB/s);   16 queries 657, 146
//   B*H = 1024, 300 keys, D = 32:   1 query 51, 10;   16 queries 50, 46
//   B*H = 8, 1024 keys:     64 queries 30, 14.7;     B*H = 16, 16384 keys:   64 queries 186, 139;   B*H = 32, 4097 keys:   74, 77
// so sixteen queries everywhere, and up to 64 while there are few batch*heads.
inline bool fm_few_pays(int bh, int nq) { return nq <= 16 || (nq <= 64 && bh * nq <= 1024); }
static constexpr int FM_FEW_MAX_SPLITS = 64;
// queries that share one pass over the keys: registers 16 per query
inline int fm_few_group(int nq) { return nq >= 4 ? 4 : nq; }
// Parts the keys of a batch*head are cut into: enough workgroups for four per CU, none with less than 64 keys, and
// no more than one wavefront of the merge reads in one go.
inline int fm_few_splits(int bh, int nq, int nk) {
  const int g = fm_few_group(nq), groups = (nq + g - 1) / g;
  int s = (1024 + bh * groups - 1) / (bh * groups);
  const int most = (nk + 63) / 64;
  if (s > most) s = most;
  if (s > 8) s = (s + 7) / 8 * 8;                       // a multiple of the XCDs: see k_few's grid
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
    IO<TIO>::ld8(A.q.base(bh) + int64_t(qi) * A.q.s_n + d0, A.q.vec != 0, qv[i]);
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
      IO<TIO>::ld8(kp + int64_t(tc) * A.k.s_n, A.k.vec != 0, kx[u]);
      IO<TIO>::ld8(vp + int64_t(tc) * A.v.s_n, A.v.vec != 0, vx[u]);
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

// Sums the parts of one query in a fixed order and divides.  grid (nq, bh), 64 threads x (DH / 64 or fewer lanes busy).
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
