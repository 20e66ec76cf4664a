// Thin portability layer between the kernels and what runs them.
//
// The kernels are written once against the names below.  The normal build is
// hipcc for gfx950.  A second, test-only build (-DFM_HOSTSIM, plain C++) maps
// the same names onto a host-thread simulator so that indexing and lane layouts
// can be checked without a GPU; the shipped library never defines FM_HOSTSIM.
#pragma once
#include <functional>
#include <mutex>
#include <unordered_map>
#include <cstddef>
#include <cstdint>

typedef _Float16 fm_half;
typedef _Float16 fm_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 fm_half4 __attribute__((ext_vector_type(4)));
typedef _Float16 fm_half8 __attribute__((ext_vector_type(8)));
typedef float fm_f32x2 __attribute__((ext_vector_type(2)));
typedef float fm_f32x4 __attribute__((ext_vector_type(4)));
typedef float fm_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t fm_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t fm_u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t fm_bf16;  // raw storage of a bfloat16
typedef uint16_t fm_u16x8 __attribute__((ext_vector_type(8)));   // eight of them: one matrix operand of a lane
typedef uint16_t fm_u16x4 __attribute__((ext_vector_type(4)));

#if defined(FM_HOSTSIM)
// ------------------------------------------------------------------ host simulator
#include <cmath>
#include "hostsim.h"
#define FM_GLOBAL
#define FM_DEVICE inline
#define FM_ALWAYS_INLINE __attribute__((always_inline))
#define FM_HOST_DEVICE
#define FM_LAUNCH_BOUNDS(n)
#define FM_LAUNCH_BOUNDS2(n, m)
#define FM_RESTRICT
#define FM_UNIFORM(x) (x)
#define FM_OPAQUE_ZERO() 0
#define FM_ARGS_AGAIN(a) (a)
#define FM_END() return
#define FM_SCHED_FENCE()
#define FM_SCHED_MFMA_DS(n)
#define FM_KEEP_BRANCH()
#define FM_WAIT_GLOBAL_LOADS()
typedef void* fm_stream_t;
typedef hostsim::Dim3 fm_dim3;
#define FM_TID_X (int(hostsim::g_t.tid.x))
#define FM_BID_X (int(hostsim::g_t.bid.x))
#define FM_BID_Y (int(hostsim::g_t.bid.y))
#define FM_BID_Z (int(hostsim::g_t.bid.z))
#define FM_GDIM_X (int(hostsim::g_t.gdim.x))
#define FM_GDIM_Y (int(hostsim::g_t.gdim.y))
#define FM_GDIM_Z (int(hostsim::g_t.gdim.z))
#define FM_SYNC() hostsim::syncthreads()
#define FM_SYNC_LDS() hostsim::syncthreads()
#define FM_DYN_SMEM(name) unsigned char* name = hostsim::g_t.blk->dyn_smem
#define FM_KERNEL_LAUNCH(kern, grid, block, smem, stream, ...) \
  hostsim::launch((grid), (block), (smem), [=]() { kern(__VA_ARGS__); })
inline int fm_after_launch() { return 0; }

FM_DEVICE fm_f32x16 fm_mfma_f16(fm_half8 a, fm_half8 b, fm_f32x16 c) {
  fm_half av[8], bv[8]; float cv[16];
  for (int i = 0; i < 8; ++i) { av[i] = a[i]; bv[i] = b[i]; }
  for (int i = 0; i < 16; ++i) cv[i] = c[i];
  hostsim::mfma_32x32<fm_half, 8>(av, bv, cv);
  for (int i = 0; i < 16; ++i) c[i] = cv[i];
  return c;
}
FM_DEVICE fm_f32x16 fm_mfma_f32(float a, float b, fm_f32x16 c) {
  float cv[16];
  for (int i = 0; i < 16; ++i) cv[i] = c[i];
  hostsim::mfma_32x32<float, 1>(&a, &b, cv);
  for (int i = 0; i < 16; ++i) c[i] = cv[i];
  return c;
}
struct fm_host_bf16 {
  uint16_t u;
  // (the instruction takes subnormal operands for zero)
  operator float() const { const uint32_t w = (u & 0x7f80) ? uint32_t(u) << 16 : 0u; float f; __builtin_memcpy(&f, &w, 4); return f; }
};
FM_DEVICE fm_f32x16 fm_mfma_bf16(fm_u16x8 a, fm_u16x8 b, fm_f32x16 c) {
  fm_host_bf16 av[8], bv[8]; float cv[16];
  for (int i = 0; i < 8; ++i) { av[i].u = a[i]; bv[i].u = b[i]; }
  for (int i = 0; i < 16; ++i) cv[i] = c[i];
  hostsim::mfma_32x32<fm_host_bf16, 8>(av, bv, cv);
  for (int i = 0; i < 16; ++i) c[i] = cv[i];
  return c;
}
FM_DEVICE float fm_shfl_xor(float v, int m) { return hostsim::shfl(v, hostsim::g_t.lane ^ m); }
FM_DEVICE int fm_shfl_xor_i(int v, int m) { return hostsim::shfl(v, hostsim::g_t.lane ^ m); }
template <int N> FM_DEVICE float fm_group_sum(float v) {
  for (int m = 1; m < N; m <<= 1) v += hostsim::shfl(v, hostsim::g_t.lane ^ m);
  return v;
}
FM_DEVICE float fm_dot2(fm_half2 a, fm_half2 b, float c) { return float(a[0]) * float(b[0]) + float(a[1]) * float(b[1]) + c; }
// Transposing LDS read (ds_read_b64_tr_b16): every lane names four consecutive halves; inside each
// group of 16 lanes, lane i receives element i % 4 of the words named by lanes i/4, 4 + i/4,
// 8 + i/4 and 12 + i/4 (layout read off the instruction on an MI355X by a probe kernel).
template <typename V4, typename T> inline V4 fm_lds_tr4_any(const T* p) {
  V4 w;
  __builtin_memcpy(&w, p, 8);
  const int lane = hostsim::g_t.lane, g = lane & ~15, i = lane & 15;
  V4 r;
  for (int t = 0; t < 4; ++t) {
    const V4 o = hostsim::shfl(w, g + 4 * t + i / 4);
    r[t] = o[i % 4];
  }
  return r;
}
FM_DEVICE fm_half4 fm_lds_tr4(const fm_half* p) { return fm_lds_tr4_any<fm_half4>(p); }
FM_DEVICE fm_u16x4 fm_lds_tr4(const uint16_t* p) { return fm_lds_tr4_any<fm_u16x4>(p); }
// the upper 32 lanes' a and the lower 32 lanes' b change places
FM_DEVICE void fm_swap_halves(uint32_t& a, uint32_t& b) {
  const int l = hostsim::g_t.lane;
  const uint32_t oa = hostsim::shfl(a, l ^ 32), ob = hostsim::shfl(b, l ^ 32);
  if (l < 32) b = oa; else a = ob;
}
FM_DEVICE float fm_fmaxf(float a, float b) { return a != a ? b : (b != b ? a : (a > b ? a : b)); }   // drops a NaN, like fmaxf
template <int FROM, int TO> FM_DEVICE float fm_lanes_max(float v) {
  for (int m = FROM; m < TO; m <<= 1) v = fm_fmaxf(v, fm_shfl_xor(v, m));
  return v;
}
FM_DEVICE float fm_absf(float x) { return __builtin_fabsf(x); }
FM_DEVICE float fm_clampf(float x, float lim) { return x > lim ? lim : (x < -lim ? -lim : x); }
FM_DEVICE float fm_rsqrtf(float a) { return 1.0f / std::sqrt(a); }
FM_DEVICE float fm_sqrtf(float a) { return std::sqrt(a); }
FM_DEVICE float fm_rcpf(float a) { return 1.0f / a; }

#else
// ------------------------------------------------------------------ gfx950
#include <hip/hip_runtime.h>
#define FM_GLOBAL __global__
#define FM_DEVICE __device__ __forceinline__
#define FM_ALWAYS_INLINE __attribute__((always_inline))
#define FM_HOST_DEVICE __host__ __device__
#define FM_LAUNCH_BOUNDS(n) __launch_bounds__(n)
#define FM_LAUNCH_BOUNDS2(n, m) __launch_bounds__(n, m)
#define FM_RESTRICT __restrict__
// a value that is the same in every lane of the wavefront, moved to a scalar register so that
// branches on it are scalar branches
#define FM_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
// A zero the optimiser cannot see through: added to an LDS offset it keeps two reads of the
// same tile apart, so the second is a fresh read instead of 16 more live registers.
static __device__ __forceinline__ int fm_opaque_zero() { int z = 0; asm volatile("" : "+v"(z)); return z; }
#define FM_OPAQUE_ZERO() fm_opaque_zero()
// A kernel's only argument, read from memory again: what a rarely taken second pass needs of it stays out of the registers
// of the first (as FM_TID_X + FM_OPAQUE_ZERO() keeps out what is made from the thread index).
template <typename T> static __device__ __forceinline__ const T& fm_args_again(const T&) {
  const __attribute__((address_space(4))) void* p = (const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const T*)p;
}
#define FM_ARGS_AGAIN(a) fm_args_again(a)
// The kernel ends here.  (A return ahead of a second pass is a jump over its code, to a line that is fetched for it: 0.4 us.)
#define FM_END() __builtin_amdgcn_endpgm()
// Nothing is scheduled across this point (keeps the live ranges of one phase out of the next).
#define FM_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
// Asks the instruction scheduler to interleave the LDS reads of this block with its matrix
// instructions (strategy 0: small products, 1: one wavefront's view); it changes the order of
// instructions only.  On MI355X the dense stages run 1 to 2 % faster with it.
#define FM_SCHED_MFMA_DS(n) __builtin_amdgcn_iglp_opt(n)
// Inside a rarely taken wavefront-uniform branch: keeps it a branch (the optimiser would
// otherwise run its body on every pass and select the result).
#define FM_KEEP_BRANCH() asm volatile("")
// Waits for every global load of the wavefront that is still in flight (s_waitcnt vmcnt(0), the other counters left
// alone).  Ahead of a software-pipelined loop it tells the compiler that nothing is pending on entry, so the loop
// head does not inherit a full wait from the prologue's loads on every iteration.
#define FM_WAIT_GLOBAL_LOADS() __builtin_amdgcn_s_waitcnt(0x0F70)
typedef hipStream_t fm_stream_t;
typedef dim3 fm_dim3;
#define FM_TID_X (int(threadIdx.x))
#define FM_BID_X (int(blockIdx.x))
#define FM_BID_Y (int(blockIdx.y))
#define FM_BID_Z (int(blockIdx.z))
#define FM_GDIM_X (int(gridDim.x))
#define FM_GDIM_Y (int(gridDim.y))
#define FM_GDIM_Z (int(gridDim.z))
#define FM_SYNC() __syncthreads()
// A barrier for what lies in LDS alone: stores to memory that are on their way are not waited for.
#define FM_SYNC_LDS() do { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); __builtin_amdgcn_s_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); } while (0)
#define FM_DYN_SMEM(name) extern __shared__ __align__(16) unsigned char name[]
// A launch the runtime refuses leaves its error as the calling thread's last error.  Only an error that
// appears across the launch is this library's: it is taken (cleared) and remembered until
// fm_after_launch() asks; an error some other library left pending before the launch stays where its
// owner will look for it and is not blamed on the launch.
inline thread_local int fm_launch_refused = 0;
#define FM_KERNEL_LAUNCH(kern, grid, block, smem, stream, ...)                                      \
  do {                                                                                              \
    const bool fm_clean_ = hipPeekAtLastError() == hipSuccess;                                      \
    hipLaunchKernelGGL(kern, (grid), (block), (smem), (stream), __VA_ARGS__);                       \
    if (fm_clean_ && hipPeekAtLastError() != hipSuccess) { (void)hipGetLastError(); fm_launch_refused = 1; } \
  } while (0)
// 0, or non-zero when a launch since the last call was refused
inline int fm_after_launch() { const int r = fm_launch_refused; fm_launch_refused = 0; return r; }

FM_DEVICE fm_f32x16 fm_mfma_f16(fm_half8 a, fm_half8 b, fm_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
FM_DEVICE fm_f32x16 fm_mfma_f32(float a, float b, fm_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
FM_DEVICE fm_f32x16 fm_mfma_bf16(fm_u16x8 a, fm_u16x8 b, fm_f32x16 c) {
  typedef __bf16 fm_bf16x8 __attribute__((ext_vector_type(8)));
  fm_bf16x8 av, bv;
  __builtin_memcpy(&av, &a, 16); __builtin_memcpy(&bv, &b, 16);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, c, 0, 0, 0);
}
FM_DEVICE float fm_shfl_xor(float v, int m) { return __shfl_xor(v, m, 64); }
FM_DEVICE int fm_shfl_xor_i(int v, int m) { return __shfl_xor(v, m, 64); }
// Sum over groups of N = 4 or 8 consecutive lanes, in every lane of the group: data-parallel-primitive adds (a lane
// exchange through the LDS pipe, what __shfl_xor compiles to, costs its latency each time).
template <int N> FM_DEVICE float fm_group_sum(float v) {
  static_assert(N == 4 || N == 8, "groups of four or eight lanes");
#define FM_DPP_ADD(ctrl) \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (ctrl), 0xf, 0xf, true))
  FM_DPP_ADD(0xB1);                  // quad_perm [1,0,3,2]
  FM_DPP_ADD(0x4E);                  // quad_perm [2,3,0,1]
  if (N == 8) FM_DPP_ADD(0x141);     // row_half_mirror: the other quad of the eight
#undef FM_DPP_ADD
  return v;
}
FM_DEVICE float fm_dot2(fm_half2 a, fm_half2 b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }
// Transposing LDS read (ds_read_b64_tr_b16): every lane names four consecutive halves; inside each
// group of 16 lanes, lane i receives element i % 4 of the words named by lanes i/4, 4 + i/4,
// 8 + i/4 and 12 + i/4 (layout read off the instruction on an MI355X by a probe kernel).
FM_DEVICE fm_half4 fm_lds_tr4(const fm_half* p) {
  typedef short fm_s16x4 __attribute__((ext_vector_type(4)));
  const fm_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fm_s16x4*)(p));
  fm_half4 r;
  __builtin_memcpy(&r, &v, 8);
  return r;
}
FM_DEVICE fm_u16x4 fm_lds_tr4(const uint16_t* p) {
  typedef short fm_s16x4 __attribute__((ext_vector_type(4)));
  const fm_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fm_s16x4*)(p));
  fm_u16x4 r;
  __builtin_memcpy(&r, &v, 8);
  return r;
}
// the upper 32 lanes' a and the lower 32 lanes' b change places (v_permlane32_swap_b32)
FM_DEVICE void fm_swap_halves(uint32_t& a, uint32_t& b) {
  typedef uint32_t fm_u2 __attribute__((ext_vector_type(2)));
  const fm_u2 r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
FM_DEVICE float fm_fmaxf(float a, float b) { return fmaxf(a, b); }
// Largest of the values of the lanes that differ in the bits FROM .. TO / 2 of their number, in each of them, without the LDS pipe but for
// bit 2 alone: data-parallel primitives inside rows of 16, then rows and halves exchanged.
template <int FROM, int TO> FM_DEVICE float fm_lanes_max(float v) {
  typedef uint32_t fm_u2 __attribute__((ext_vector_type(2)));
#define FM_DPP_MAX(ctrl) v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (ctrl), 0xf, 0xf, true)))
  if (FROM <= 1 && TO > 1) FM_DPP_MAX(0xB1);           // quad_perm [1,0,3,2]
  if (FROM <= 2 && TO > 2) FM_DPP_MAX(0x4E);           // quad_perm [2,3,0,1]
  if (FROM == 1 && TO > 4) FM_DPP_MAX(0x141);          // row_half_mirror: the other quad
  else if (FROM <= 4 && TO > 4) v = fmaxf(v, fm_shfl_xor(v, 4));
  if (FROM <= 8 && TO > 8) FM_DPP_MAX(0x128);          // row_ror:8
#undef FM_DPP_MAX
  if (FROM <= 16 && TO > 16) {
    const fm_u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if (FROM <= 32 && TO > 32) {
    const fm_u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}
FM_DEVICE float fm_absf(float x) { return __builtin_fabsf(x); }
// clamp to [-lim, lim] in one instruction (v_med3_f32)
FM_DEVICE float fm_clampf(float x, float lim) { return __builtin_amdgcn_fmed3f(x, -lim, lim); }
FM_DEVICE float fm_rsqrtf(float a) { return rsqrtf(a); }
FM_DEVICE float fm_sqrtf(float a) { return sqrtf(a); }
// 1 / a for an ordinary a, to within a rounding of it (one correction of the instruction's result)
FM_DEVICE float fm_rcpf(float a) { const float r = __builtin_amdgcn_rcpf(a); return __builtin_fmaf(r, __builtin_fmaf(-a, r, 1.0f), r); }
#endif

// ---- bf16 <-> f32 (round to nearest even), usable on both builds -------------
FM_DEVICE float fm_bf16_to_f32(fm_bf16 v) {
  uint32_t u = uint32_t(v) << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}
#if defined(FM_HOSTSIM)
FM_DEVICE fm_bf16 fm_f32_to_bf16(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return fm_bf16((u >> 16) | 0x40u);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return fm_bf16(u >> 16);
}
#endif
// two floats -> two bfloat16 in one register, the first in the low half
FM_DEVICE uint32_t fm_cvt_pk_bf16(float a, float b) {
#if defined(FM_HOSTSIM)
  return uint32_t(fm_f32_to_bf16(a)) | (uint32_t(fm_f32_to_bf16(b)) << 16);
#else
  typedef __bf16 fm_bf16x2 __attribute__((ext_vector_type(2)));
  const fm_f32x2 v = {a, b};
  const fm_bf16x2 h = __builtin_convertvector(v, fm_bf16x2);   // v_cvt_pk_bf16_f32
  uint32_t u;
  __builtin_memcpy(&u, &h, 4);
  return u;
#endif
}
#if !defined(FM_HOSTSIM)
// (the conversion instruction: rounding spelt out in integer arithmetic was five instructions per element and up to half of
// the code of the kernels that store bf16)
FM_DEVICE fm_bf16 fm_f32_to_bf16(float f) { return fm_bf16(fm_cvt_pk_bf16(f, f)); }
#endif
FM_DEVICE float fm_bits_f32(uint32_t u) { float f; __builtin_memcpy(&f, &u, 4); return f; }

#if defined(FM_HOSTSIM)
static inline void fm_allow_lds(const void*, size_t) {}
#else
// Dynamic LDS above the 64 KiB default has to be allowed once per kernel function (and device); the
// attribute call costs microseconds of host time, so it is made the first time a kernel asks for more
// than it has been granted so far and skipped afterwards.
static inline void fm_allow_lds(const void* fn, size_t bytes) {
  if (bytes <= 64 * 1024) return;
  struct Key { const void* fn; int dev; bool operator==(const Key& o) const { return fn == o.fn && dev == o.dev; } };
  struct Hash { size_t operator()(const Key& k) const { return std::hash<const void*>()(k.fn) ^ (size_t(k.dev) * 0x9e3779b97f4a7c15ull); } };
  static std::mutex mu;
  static std::unordered_map<Key, size_t, Hash> granted;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  std::lock_guard<std::mutex> lock(mu);
  size_t& have = granted[Key{fn, dev}];
  if (bytes <= have) return;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)) == hipSuccess) have = bytes;
}
#endif
