// Driver for the CPU build of the kernel sources (host simulator) under AddressSanitizer: a few shapes through the
// C ABI, forward and backward; the simulator keeps LDS and all tensors on the heap, so an index out of bounds in a
// kernel is reported.  Built and run by tests/test_hostsim.py when FASTMAX_HOSTSIM_ASAN=1.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include <cmath>
#include "fastmax_hip.h"
static uint16_t bf16(float x) { uint32_t u; memcpy(&u, &x, 4); return uint16_t((u + 0x7fff + ((u >> 16) & 1)) >> 16); }
static float frand() { return float(rand()) / RAND_MAX * 2.f - 1.f; }
// nk 0: as many keys as queries.  norm: q and k max-normalised by the kernels themselves, gradients of the raw tensors.
// inf: an infinite value, which sends the dense fp32 kernels and the short sequences through their second pass.
struct Opt { int nk = 0, mask = 1, flags = 0, norm = 0, inf = 0, backward = 1; };
static int run(int bh, int n, int d, int p, int chunk, int dtype, int save, Opt x = Opt()) {
  const int nk = x.nk ? x.nk : n;
  FastmaxDesc D; memset(&D, 0, sizeof D);
  D.bh = bh; D.nq = n; D.nk = nk; D.d = d; D.dtype = dtype; D.mask = x.mask; D.p = p; D.a0 = 1; D.a1 = 1; D.a2 = .5f;
  D.inv_tau = 1.f / (2.f * std::sqrt(float(d))); D.chunk = chunk; D.flags = x.flags | (save ? FASTMAX_FLAG_SAVE_FOR_BACKWARD : 0);
  if (x.norm) { D.flags |= FASTMAX_FLAG_NORM_SELF; D.norm.lim = 1.5f; D.norm.grad = 1; }
  FastmaxStrides sq = {int64_t(n) * d, d, 0, 0}, sk = {int64_t(nk) * d, d, 0, 0};
  D.sq = D.so = D.sdo = D.sdq = sq;
  D.sk = D.sv = D.sdk = D.sdv = sk;
  D.sg.bh = n; D.sg.n = 1;
  size_t fb, bb; int st = fastmax_workspace_bytes(&D, &fb, &bb); if (st) return st;
  const size_t esz = dtype == FASTMAX_BF16 ? 2 : 4, ne = size_t(bh) * n * d, nke = size_t(bh) * nk * d;
  std::vector<char> q(ne * esz), k(nke * esz), v(nke * esz), go(ne * esz), o(ne * esz), dq(ne * esz), dk(nke * esz), dv(nke * esz);
  std::vector<float> g(size_t(bh) * n);
  for (std::vector<char>* b : {&q, &k, &v, &go})
    for (size_t i = 0; i < b->size() / esz; ++i) {
      const float r = frand();
      if (esz == 2) reinterpret_cast<uint16_t*>(b->data())[i] = bf16(r); else reinterpret_cast<float*>(b->data())[i] = r;
    }
  if (x.inf) { if (esz == 2) reinterpret_cast<uint16_t*>(v.data())[3] = 0x7f80; else reinterpret_cast<float*>(v.data())[3] = INFINITY; }
  // exactly the bytes the library names (a multiple of the alignment)
  void* fws = aligned_alloc(256, (fb + 255) / 256 * 256); void* bws = aligned_alloc(256, (bb + 255) / 256 * 256);
  st = fastmax_forward(&D, q.data(), k.data(), v.data(), o.data(), g.data(), fws, fb, nullptr);
  if (!st && x.backward) st = save ? fastmax_backward_saved(&D, q.data(), k.data(), v.data(), o.data(), g.data(), go.data(), dq.data(), dk.data(), dv.data(), fws, fb, bws, bb, nullptr)
                     : fastmax_backward(&D, q.data(), k.data(), v.data(), o.data(), g.data(), go.data(), dq.data(), dk.data(), dv.data(), bws, bb, nullptr);
  free(fws); free(bws);
  double sum = 0; for (float y : g) sum += y;
  printf("bh=%d n=%d nk=%d d=%d p=%d mask=%d chunk=%d dtype=%d save=%d flags=%d norm=%d inf=%d -> status %d, sum g %.3f\n", bh, n, nk, d, p,
         x.mask, chunk, dtype, save, x.flags, x.norm, x.inf, st, sum);
  fflush(stdout);
  return st;
}
static Opt opt(int nk, int mask, int flags = 0, int norm = 0, int inf = 0, int backward = 1) {
  Opt x; x.nk = nk; x.mask = mask; x.flags = flags; x.norm = norm; x.inf = inf; x.backward = backward; return x;
}
// the two element-wise passes (key RPE, output noise) on a ragged shape, in place
static int run_pointwise(int bh, int n, int d, int dtype) {
  FastmaxNormDesc N{};
  N.bh = bh; N.n = n; N.d = d; N.dtype = dtype;
  N.sx.bh = int64_t(n) * d; N.sx.n = d; N.sy = N.sx;
  const size_t esz = dtype == FASTMAX_BF16 ? 2 : 4;
  std::vector<unsigned char> x(size_t(bh) * n * d * esz, 0), noise(x.size(), 0);
  std::vector<float> rpe(size_t(2 * n - 1) * d, 0.25f);
  int st = fastmax_key_rpe(&N, x.data(), rpe.data(), x.data(), 2.0f, nullptr);
  if (!st) st = fastmax_output_noise(&N, x.data(), noise.data(), x.data(), 0.5f, nullptr);
  printf("pointwise bh=%d n=%d d=%d dtype=%d -> status %d\n", bh, n, d, dtype, st);
  return st;
}
// the decoding state: a prompt absorbed, then single-token steps (buffers of exactly the sizes the library names)
// fresh: into memory full of NaN that is said to be a new state.  big: a value beside which k' v overflows.
static int run_decode(int bh, int d, int p, int prompt, int steps, int dtype, int fresh = 0, int big = 0) {
  FastmaxDesc D; memset(&D, 0, sizeof D);
  D.bh = bh; D.nq = 1; D.nk = prompt; D.d = d; D.dtype = dtype; D.mask = 1; D.p = p; D.a0 = 1; D.a1 = 1; D.a2 = .5f;
  D.inv_tau = 1.f / (2.f * std::sqrt(float(d)));
  FastmaxStrides s = {int64_t(prompt) * d, d, 0, 0}, s1 = {int64_t(d), d, 0, 0};
  D.sq = s1; D.sk = D.sv = s; D.so = s1; D.sg.bh = 1; D.sg.n = 1;
  const size_t esz = dtype == FASTMAX_BF16 ? 2 : 4, ne = size_t(bh) * prompt * d;
  std::vector<char> k(ne * esz), v(ne * esz), q1(size_t(bh) * d * esz), k1(q1.size()), v1(q1.size()), o1(q1.size());
  auto fill = [&](std::vector<char>& b) {
    for (size_t i = 0; i < b.size() / esz; ++i) {
      const float x = frand();
      if (esz == 2) reinterpret_cast<uint16_t*>(b.data())[i] = bf16(x); else reinterpret_cast<float*>(b.data())[i] = x;
    }
  };
  fill(k); fill(v); fill(q1); fill(k1); fill(v1);
  if (big) { reinterpret_cast<float*>(v.data())[5] = 1e38f; reinterpret_cast<float*>(k.data())[1] = 1e3f; }
  const size_t sb = fastmax_decode_state_bytes(&D), cb = fastmax_decode_scratch_bytes(&D);
  if (!sb || !cb) return 99;
  float* state = static_cast<float*>(aligned_alloc(256, (sb + 255) / 256 * 256));
  memset(state, fresh ? 0xff : 0, sb);
  if (fresh) D.flags = FASTMAX_FLAG_NEW_STATE;
  float* scratch = static_cast<float*>(aligned_alloc(256, (cb + 255) / 256 * 256));
  std::vector<float> g(bh);
  int st = fastmax_decode_absorb(&D, k.data(), v.data(), state, nullptr);
  D.sk = D.sv = s1;
  for (int i = 0; i < steps && !st; ++i)
    st = fastmax_decode_step(&D, q1.data(), k1.data(), v1.data(), state, o1.data(), g.data(), scratch, nullptr);
  free(state); free(scratch);
  printf("decode bh=%d d=%d p=%d prompt=%d steps=%d dtype=%d fresh=%d big=%d -> status %d, g[0] %.3f\n", bh, d, p, prompt, steps, dtype,
         fresh, big, st, g[0]);
  fflush(stdout);
  return st;
}
// heads of d features to rows of dpad: up to three tensors of their own lengths in one launch
static int run_pad(int bh, int d, int dpad, int dtype, int count) {
  const size_t esz = dtype == FASTMAX_BF16 ? 2 : 4;
  const int ns[3] = {1, 70, 33};
  FastmaxNormDesc N[3];
  const FastmaxNormDesc* D[3];
  std::vector<unsigned char> x[3], y[3];
  const void* xp[3]; void* yp[3];
  for (int i = 0; i < count; ++i) {
    N[i] = FastmaxNormDesc();
    N[i].bh = bh; N[i].n = ns[i]; N[i].d = d; N[i].dtype = dtype;
    N[i].sx.bh = int64_t(ns[i]) * d; N[i].sx.n = d; N[i].sy.bh = int64_t(ns[i]) * dpad; N[i].sy.n = dpad;
    x[i].assign(size_t(bh) * ns[i] * d * esz, 1); y[i].assign(size_t(bh) * ns[i] * dpad * esz, 7);
    D[i] = &N[i]; xp[i] = x[i].data(); yp[i] = y[i].data();
  }
  const int st = fastmax_pad_features(D, xp, yp, count, dpad, nullptr);
  printf("pad bh=%d d=%d dpad=%d dtype=%d count=%d -> status %d\n", bh, d, dpad, dtype, count, st);
  fflush(stdout);
  return st;
}
// two tensors of different lengths through the normalisation passes in common launches
static int run_norm_pair(int bh, int n0, int n1, int d, int dtype, int centre) {
  const size_t esz = dtype == FASTMAX_BF16 ? 2 : 4;
  FastmaxNormDesc N[2];
  std::vector<unsigned char> x[2], dy[2], y[2];
  float* stats[2];
  const int ns[2] = {n0, n1};
  int st = 0;
  for (int back = 0; back < 2 && !st; ++back) {
    for (int i = 0; i < 2; ++i) {
      N[i] = FastmaxNormDesc();
      N[i].bh = bh; N[i].n = ns[i]; N[i].d = d; N[i].dtype = dtype; N[i].centre = centre; N[i].max_norm = 1; N[i].scale = 1.5f;
      N[i].sx.bh = int64_t(ns[i]) * d; N[i].sx.n = d; N[i].sy = N[i].sx;
      x[i].assign(size_t(bh) * ns[i] * d * esz, 0); dy[i] = x[i]; y[i] = x[i];
      for (std::vector<unsigned char>* b : {&x[i], &dy[i]})
        for (size_t j = 0; j < b->size() / esz; ++j) {
          const float r = frand();
          if (esz == 2) reinterpret_cast<uint16_t*>(b->data())[j] = bf16(r); else reinterpret_cast<float*>(b->data())[j] = r;
        }
      stats[i] = static_cast<float*>(malloc(back ? fastmax_normalize_backward_stats_bytes(&N[i]) : fastmax_normalize_stats_bytes(&N[i])));
    }
    st = back ? fastmax_normalize_backward_pair(&N[0], x[0].data(), dy[0].data(), y[0].data(), stats[0], &N[1], x[1].data(), dy[1].data(),
                                                y[1].data(), stats[1], nullptr)
              : fastmax_normalize_pair(&N[0], x[0].data(), y[0].data(), stats[0], &N[1], x[1].data(), y[1].data(), stats[1], nullptr);
    free(stats[0]); free(stats[1]);
  }
  printf("norm pair bh=%d n=%d,%d d=%d dtype=%d centre=%d -> status %d\n", bh, n0, n1, d, dtype, centre, st);
  fflush(stdout);
  return st;
}
extern "C" void fastmax_hostsim_one_group(int on);
extern "C" void fastmax_hostsim_x2(int split);
int main() {
  int bad = 0;
  bad |= run_pointwise(3, 333, 64, FASTMAX_BF16);
  bad |= run_pointwise(2, 70, 32, FASTMAX_F32);
  bad |= run_decode(2, 64, 2, 37, 2, FASTMAX_BF16);
  bad |= run_decode(3, 32, 1, 5, 2, FASTMAX_F32);
  bad |= run_decode(1, 64, 2, 150, 1, FASTMAX_BF16);  // a prompt summed with matrix instructions (two tiles, the second ragged)
  // prompts in fp32 products: one and several tiles, ragged, both orders, a new state, a sum that overflows
  bad |= run_decode(1, 64, 2, 64, 1, FASTMAX_F32);
  bad |= run_decode(1, 64, 2, 150, 1, FASTMAX_F32, 1);
  bad |= run_decode(2, 32, 2, 129, 1, FASTMAX_F32, 1);
  bad |= run_decode(1, 32, 2, 70, 1, FASTMAX_BF16, 1);
  bad |= run_decode(1, 64, 1, 195, 1, FASTMAX_BF16, 1);
  bad |= run_decode(1, 32, 2, 70, 1, FASTMAX_F32, 1, 1);
  bad |= run_decode(1, 64, 2, 150, 1, FASTMAX_BF16, 1);
  bad |= run_decode(1, 64, 2, 20, 1, FASTMAX_F32, 1);
  bad |= run_pad(3, 48, 64, FASTMAX_F32, 3);
  bad |= run_pad(2, 1, 32, FASTMAX_BF16, 3);
  bad |= run_pad(2, 127, 128, FASTMAX_BF16, 2);
  bad |= run_norm_pair(2, 70, 300, 64, FASTMAX_F32, 2);
  bad |= run_norm_pair(1, 257, 1, 32, FASTMAX_BF16, 2);
  bad |= run_norm_pair(1, 64, 129, 64, FASTMAX_BF16, 1);
  // one segment in one group of wavefronts per workgroup, as launches of many workgroups run (further down: in two)
  fastmax_hostsim_one_group(1);
  bad |= run(2, 200, 64, 2, 0, FASTMAX_BF16, 1);
  bad |= run(1, 130, 32, 2, 0, FASTMAX_BF16, 0);
  bad |= run(1, 70, 64, 1, 0, FASTMAX_BF16, 1, opt(75, 0, FASTMAX_FLAG_FORCE_DENSE));
  bad |= run(1, 200, 128, 2, 0, FASTMAX_BF16, 1);
  bad |= run(1, 75, 128, 1, 0, FASTMAX_BF16, 0, opt(70, 0));
  fastmax_hostsim_one_group(0);
  bad |= run(1, 300, 64, 2, 256, FASTMAX_BF16, 1);    // order-2 walk held per value column (two segments), saved and rebuilt
  bad |= run(1, 300, 64, 2, 256, FASTMAX_BF16, 0);
  bad |= run(1, 600, 32, 2, 256, FASTMAX_BF16, 1);    // order-2 walk (a CU to itself: two buffers), both walks
  bad |= run(1, 600, 32, 2, 256, FASTMAX_BF16, 0);
  bad |= run(1, 520, 64, 2, 256, FASTMAX_BF16, 1);
  bad |= run(1, 1100, 32, 1, 0, FASTMAX_BF16, 1);     // order-1 runs of segments
  bad |= run(3, 1300, 64, 1, 0, FASTMAX_BF16, 0);
  bad |= run(2, 200, 64, 2, 0, FASTMAX_BF16, 1);      // one segment, dense kernels
  bad |= run(1, 200, 128, 2, 0, FASTMAX_BF16, 1);     // heads of 128: four accumulator tiles per feature axis
  bad |= run(1, 150, 128, 1, 0, FASTMAX_BF16, 0);
  bad |= run(1, 300, 32, 2, 256, FASTMAX_F32, 1);
  // fp32 on dense tiles (fm_x3.h): square and not, saved and not, bf16 tensors computed in fp32, the second pass
  bad |= run(1, 70, 64, 2, 0, FASTMAX_F32, 1);
  bad |= run(1, 130, 32, 2, 0, FASTMAX_F32, 0);
  bad |= run(1, 40, 64, 1, 0, FASTMAX_F32, 0, opt(75, 0));
  bad |= run(1, 75, 32, 2, 0, FASTMAX_F32, 0, opt(40, 0));
  bad |= run(1, 70, 64, 2, 0, FASTMAX_BF16, 1, opt(0, 1, FASTMAX_FLAG_F32_COMPUTE));
  bad |= run(1, 70, 64, 2, 0, FASTMAX_F32, 1, opt(0, 1, 0, 0, 1));
  bad |= run(1, 70, 32, 2, 0, FASTMAX_F32, 0, opt(0, 0, 0, 0, 1));
  // fp32 on two planes (fm_x2.h): one, two and four wavefronts to a tile, square and not, saved and not, refused
  for (int split : {1, 2, 4}) {
    fastmax_hostsim_x2(split);
    bad |= run(1, 130, 64, 2, 0, FASTMAX_F32, 1, opt(0, 1, FASTMAX_FLAG_FORCE_DENSE));
    bad |= run(2, 70, 32, 2, 0, FASTMAX_F32, 0, opt(97, 0, FASTMAX_FLAG_FORCE_DENSE));
    bad |= run(1, 97, 64, 2, 0, FASTMAX_F32, 0, opt(0, 1, FASTMAX_FLAG_FORCE_DENSE));
    bad |= run(1, 70, 32, 2, 0, FASTMAX_F32, 1, opt(0, 0, FASTMAX_FLAG_FORCE_DENSE, 0, 1));
  }
  fastmax_hostsim_x2(0);
  // at most 64 tokens (fm_small.h): normalised by the kernels, causal with more keys, fp32 arithmetic, the second pass
  for (int dtype : {FASTMAX_F32, FASTMAX_BF16})
    for (int n : {1, 33, 50, 64}) bad |= run(2, n, n == 50 ? 32 : 64, 2, 0, dtype, 1, opt(0, 0, 0, 1));
  bad |= run(1, 17, 64, 2, 0, FASTMAX_F32, 0, opt(64, 1));
  bad |= run(1, 17, 32, 2, 0, FASTMAX_BF16, 0, opt(64, 1));
  bad |= run(1, 50, 64, 2, 0, FASTMAX_BF16, 1, opt(0, 1, FASTMAX_FLAG_F32_COMPUTE, 0, 1));
  bad |= run(1, 33, 32, 2, 0, FASTMAX_BF16, 1, opt(0, 1, 0, 1, 1));
  bad |= run(1, 33, 64, 2, 0, FASTMAX_F32, 0, opt(20, 0, 0, 1, 1));
  // a few queries (fm_few.h): forward alone
  for (int dtype : {FASTMAX_F32, FASTMAX_BF16}) {
    bad |= run(2, 1, 64, 2, 0, dtype, 0, opt(65, 1, 0, 0, 0, 0));
    bad |= run(1, 6, 32, 2, 0, dtype, 0, opt(577, 1, 0, 0, 0, 0));
    bad |= run(1, 3, 64, 1, 0, dtype, 0, opt(30, 0, 0, 0, 0, 0));
  }
  return bad;
}
