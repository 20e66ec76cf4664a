// The two element-wise steps of the reference's forward_cuda that it ships switched off, as passes a caller
// can switch on:
//   * relative-position rows added to the keys after the temperature division
//     (apply_rpe_and_temp, fastmax_cuda_forward.cu:282-292; the addition at :289 is commented out there):
//       k[l][i][m] = k[l][i][m] / tau + rpe[(l + nk) % (2 nk - 1)][m]
//     Here the operator divides by tau inside its loads, so the pass writes k + tau * rpe.
//   * multiplicative noise on the output (apply_dropout, fastmax_cuda_forward.cu:340-349; called with
//     scale 0 at :443):  o[l][i][m] *= 1 + scale * noise[l][i][m].  The same pass applied to dO is its
//     backward.
// Both read one tensor (plus the table / the noise) and write one: HBM-bound, 16-byte accesses where the
// strides allow, 64 * FM_NORM_NP tokens of one batch*head per workgroup.
#pragma once
#include "fm_norm.h"

struct PointwiseArgs {
  int n;               // tokens
  int mode;            // 0: key RPE, 1: output noise
  float factor;        // tau (mode 0) or the noise scale (mode 1)
  const float* table;  // mode 0: (2 n - 1, d) contiguous fp32 rows
};

template <typename TIO, int DH>
FM_GLOBAL void FM_LAUNCH_BOUNDS(256) k_pointwise(TRef<const TIO> x, TRef<const TIO> noise, TRef<TIO> y, PointwiseArgs a) {
  constexpr int EPT = DH / 4, NP = FM_NORM_NP;
  const int tid = FM_TID_X, bh = FM_BID_Y;
  const int tok0 = FM_BID_X * 64 * NP + (tid >> 2), d0 = (tid & 3) * EPT;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int tok = tok0 + 64 * p;
    if (tok >= a.n) continue;
    float v[EPT], w[EPT];
    fm_norm_load<TIO, DH>(x.base(bh) + int64_t(tok) * x.s_n, d0, v);
    if (a.mode == 0) {
      const float* row = a.table + int64_t((tok + a.n) % (2 * a.n - 1)) * DH + d0;
#pragma unroll
      for (int j = 0; j < EPT; ++j) v[j] += a.factor * row[j];
    } else {
      fm_norm_load<TIO, DH>(noise.base(bh) + int64_t(tok) * noise.s_n, d0, w);
#pragma unroll
      for (int j = 0; j < EPT; ++j) v[j] *= 1.0f + a.factor * w[j];
    }
#pragma unroll
    for (int j = 0; j < EPT; j += 8) IO<TIO>::st8(y.base(bh) + int64_t(tok) * y.s_n + d0 + j, &v[j]);
  }
}

template <typename TIO, int DH>
int fm_pointwise_run(const FastmaxNormDesc* d, const void* x, const void* noise, void* y, const PointwiseArgs& a,
                     fm_stream_t stream) {
  const TRef<const TIO> xr = fm_ref<const TIO>(static_cast<const TIO*>(x), d->sx);
  const TRef<const TIO> nr = fm_ref<const TIO>(static_cast<const TIO*>(noise ? noise : x), d->sx);
  const TRef<TIO> yr = fm_ref<TIO>(static_cast<TIO*>(y), d->sy);
  const fm_dim3 grid(fm_norm_blocks(d->n), d->bh);
  FM_KERNEL_LAUNCH((k_pointwise<TIO, DH>), grid, fm_dim3(256), 0, stream, xr, nr, yr, a);
  return fm_after_launch() ? FASTMAX_ERR_LAUNCH : FASTMAX_OK;
}

inline int fm_pointwise_dispatch(const FastmaxNormDesc* d, const void* x, const void* noise, void* y, const PointwiseArgs& a,
                                 fm_stream_t stream) {
  if (!d || !x || !y) return FASTMAX_ERR_NULL;
  if (a.mode == 0 ? !a.table : !noise) return FASTMAX_ERR_NULL;
  if (d->dtype != FASTMAX_F32 && d->dtype != FASTMAX_BF16) return FASTMAX_ERR_DTYPE;
  if (d->bh <= 0 || d->n <= 0 || d->bh > 65535 || d->n > (1 << 30)) return FASTMAX_ERR_SHAPE;
  if (d->d != 32 && d->d != 64) return FASTMAX_ERR_UNSUPPORTED;
  if (d->sx.n < d->d || d->sy.n < d->d) return FASTMAX_ERR_SHAPE;
  if (d->dtype == FASTMAX_F32)
    return d->d == 64 ? fm_pointwise_run<float, 64>(d, x, noise, y, a, stream) : fm_pointwise_run<float, 32>(d, x, noise, y, a, stream);
  return d->d == 64 ? fm_pointwise_run<fm_bf16, 64>(d, x, noise, y, a, stream) : fm_pointwise_run<fm_bf16, 32>(d, x, noise, y, a, stream);
}

// Rows of d elements to zero-padded rows of dpad (a head size the kernels have), up to FM_PAD_JOBS tensors in one launch: a thread
// writes eight elements.  A call with heads of 48 pads q, k and v ahead of the forward and dO ahead of the backward; as a fill and a
// copy per tensor the eight tensors of a normalised step were sixteen launches of 3.4 to 3.7 us (the score-function front's step, 15
// heads of 48, 777 tokens, fp32, with the normalisation in common launches (fm_norm.h): 244 -> 160 us).  E: an unsigned type of the element's size.
static constexpr int FM_PAD_JOBS = 3;
template <typename E> struct PadJob { TRef<const E> src; TRef<E> dst; int n; };
template <typename E> struct PadJobs { PadJob<E> j[FM_PAD_JOBS]; };
template <typename E> FM_GLOBAL void FM_LAUNCH_BOUNDS(256) k_pad(PadJobs<E> jobs, int d, int dpad) {
  const PadJob<E> J = FM_BID_Z == 0 ? jobs.j[0] : FM_BID_Z == 1 ? jobs.j[1] : jobs.j[2];
  const int bh = FM_BID_Y, sh = dpad == 32 ? 2 : dpad == 64 ? 3 : 4;   // 2^sh octets per row (a shift: dividing took longer than the copy)
  const int64_t c = int64_t(FM_BID_X) * 256 + FM_TID_X, row = c >> sh;
  const int col = int(c & ((1 << sh) - 1)) * 8;
  if (row >= J.n) return;
  const E* s = J.src.base(bh) + row * J.src.s_n + col;
  struct Oct { E e[8]; } v;
  if (col + 8 <= d) {
    __builtin_memcpy(&v, s, sizeof(v));
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v.e[i] = col + i < d ? s[i] : E(0);
  }
  __builtin_memcpy(J.dst.base(bh) + row * J.dst.s_n + col, &v, sizeof(v));
}
template <typename E>
int fm_pad_run(const FastmaxNormDesc* const* d, const void* const* x, void* const* y, int count, int dpad, fm_stream_t stream) {
  PadJobs<E> jobs{};
  int nmax = 0;
  for (int i = 0; i < count; ++i) {
    jobs.j[i] = PadJob<E>{fm_ref<const E>(static_cast<const E*>(x[i]), d[i]->sx), fm_ref<E>(static_cast<E*>(y[i]), d[i]->sy), d[i]->n};
    nmax = d[i]->n > nmax ? d[i]->n : nmax;
  }
  const int64_t octets = int64_t(nmax) * (dpad / 8);
  FM_KERNEL_LAUNCH((k_pad<E>), fm_dim3(unsigned((octets + 255) / 256), d[0]->bh, count), fm_dim3(256), 0, stream, jobs, d[0]->d, dpad);
  return fm_after_launch() ? FASTMAX_ERR_LAUNCH : FASTMAX_OK;
}
inline int fm_pad_dispatch(const FastmaxNormDesc* const* d, const void* const* x, void* const* y, int count, int dpad, fm_stream_t stream) {
  if (!d || !x || !y) return FASTMAX_ERR_NULL;
  if (count < 1 || count > FM_PAD_JOBS || (dpad != 32 && dpad != 64 && dpad != 128)) return FASTMAX_ERR_UNSUPPORTED;
  for (int i = 0; i < count; ++i) {
    if (!d[i] || !x[i] || !y[i]) return FASTMAX_ERR_NULL;
    if (d[i]->dtype != FASTMAX_F32 && d[i]->dtype != FASTMAX_BF16) return FASTMAX_ERR_DTYPE;
    if (d[i]->bh <= 0 || d[i]->n <= 0 || d[i]->bh > 65535 || d[i]->n > (1 << 30) || d[i]->d <= 0 || d[i]->d >= dpad || d[i]->sy.n < dpad)
      return FASTMAX_ERR_SHAPE;
    if (d[i]->bh != d[0]->bh || d[i]->d != d[0]->d || d[i]->dtype != d[0]->dtype) return FASTMAX_ERR_SHAPE;
  }
  return d[0]->dtype == FASTMAX_F32 ? fm_pad_run<uint32_t>(d, x, y, count, dpad, stream) : fm_pad_run<uint16_t>(d, x, y, count, dpad, stream);
}
