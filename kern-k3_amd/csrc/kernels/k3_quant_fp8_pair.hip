// Modules k3_quant_fp8_pair / k3_quant_fp8_pair_v2: per-tensor bf16 -> e4m3.
//
//   v1: kern_quant_fp8_amax(x, n, partials)                   (k3_quant_fp8_pair.cu:18)
//       kern_quant_fp8_apply(x, y, n, partials, nb, scale_out) (k3_quant_fp8_pair.cu:32)
//   v2: kern_quant_fp8_amax_v2 / kern_quant_fp8_apply_v2 with the same
//       parameters (k3_quant_fp8_pair_v2.cu:42, 63; manifest op quant_fp8_tensor,
//       k3-tp4-prefill-16k.json:407194)
//   grid (nb, 1, 1) with nb = 2048 in the manifest, block (256, 1, 1), both launches.
//
// amax:  partials[b] = max |x| over block b's slice of a grid-stride partition.
//        v1 partitions elements (element i belongs to block (i / 256) % nb) and
//        takes an f32 max (NaN ignored); v2 partitions 16-byte vectors (vector i
//        to block (i / 256) % nb), takes the max of the |bf16| bit patterns
//        (NaN patterns included) and folds the n % 8 tail into block 0.  The
//        partials are outputs, so the slices follow those partitions exactly;
//        only the order inside a slice is free (the max is order-independent).
// apply: amax = max(partials[0..nb)), scale = amax > 0 ? amax / 448 : 1 (IEEE
//        division), scale_out[0] = scale, y = e4m3(x * (1 / scale)) with RNE and
//        saturation to +-448.  |x| * (1 / scale) exceeds 448 by rounding only,
//        which the RNE conversion maps back to 448.
// Cache policy: the amax pass reads x with cacheable loads, so that x (235 MB
// at 16384 x 7168) stays in the 256 MB MALL and the apply pass, which sweeps
// it in the same front-to-back order, reads it from there; the apply pass's
// own loads and stores are non-temporal (measured at that shape: 99.4 -> 90.5
// us after a clean 512 MB flush, 96.0 -> 87.8 us back to back over four
// rotating input / output sets, identical outputs; after a dirty 512 MB flush
// the amax pass pays the write-back of the lines it evicts, 97 -> 131 us).
#include "../common/k3_dev.h"

#define QT 256

// Block max of a non-negative u32 (four waves: wave butterfly, then LDS).
K3_DEV uint32_t k3_block_max_u32(uint32_t m) {
  __shared__ uint32_t s[QT / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t p = (uint32_t)__shfl_xor((int)m, o, 64);
    m = m > p ? m : p;
  }
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
  __syncthreads();
  uint32_t r = s[0];
#pragma unroll
  for (int w = 1; w < QT / 64; ++w) r = r > s[w] ? r : s[w];
  return r;
}

// |bf16| magnitude key for the f32-max form: NaN patterns are ignored (0).
K3_DEV uint32_t k3_mag_f32max(uint32_t h) {
  const uint32_t a = h & 0x7fffu;
  return a > 0x7f80u ? 0u : a;
}

#ifndef K3_QUANT_V2
extern "C" __global__ void __launch_bounds__(QT) kern_quant_fp8_amax(
    const uint16_t* __restrict__ x, int n, float* __restrict__ partials) {
  // block b owns the 256-element chunks b, b + nb, b + 2 nb, ...; a 256-thread
  // step covers eight chunks with one 16-byte vector per thread (32 per chunk).
  const long long nb = gridDim.x;
  const int sub = threadIdx.x >> 5, lane = threadIdx.x & 31;
  uint32_t m = 0;
  for (long long c = blockIdx.x + sub * nb; c * 256 < n; c += 8 * nb) {
    const long long e0 = c * 256 + lane * 8;
    if (e0 + 8 <= n) {
      const k3_u4 v = k3_ld16(x + e0);  // cacheable: kept in the MALL for the apply pass
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = k3_mag_f32max(v[j] & 0xffffu), hi = k3_mag_f32max(v[j] >> 16);
        m = m > lo ? m : lo;
        m = m > hi ? m : hi;
      }
    } else {
      for (long long e = e0; e < n; ++e) {
        const uint32_t a = k3_mag_f32max(x[e]);
        m = m > a ? m : a;
      }
    }
  }
  m = k3_block_max_u32(m);
  if (threadIdx.x == 0) partials[blockIdx.x] = __uint_as_float(m << 16);
}
#define K3_APPLY_NAME kern_quant_fp8_apply
#else
extern "C" __global__ void __launch_bounds__(QT) kern_quant_fp8_amax_v2(
    const uint16_t* __restrict__ x, int n, float* __restrict__ partials) {
  const long long nv = n >> 3;
  uint32_t m = 0;
  for (long long i = (long long)blockIdx.x * QT + threadIdx.x; i < nv; i += (long long)gridDim.x * QT) {
    const k3_u4 v = k3_ld16(x + i * 8);  // cacheable: kept in the MALL for the apply pass
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t a = v[j] & 0x7fff7fffu;
      const uint32_t lo = a & 0xffffu, hi = a >> 16;
      m = m > lo ? m : lo;
      m = m > hi ? m : hi;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < (n & 7)) {
    const uint32_t a = x[nv * 8 + threadIdx.x] & 0x7fffu;
    m = m > a ? m : a;
  }
  m = k3_block_max_u32(m);
  if (threadIdx.x == 0) partials[blockIdx.x] = __uint_as_float(m << 16);
}
#define K3_APPLY_NAME kern_quant_fp8_apply_v2
#endif

extern "C" __global__ void __launch_bounds__(QT) K3_APPLY_NAME(
    const uint16_t* __restrict__ x, uint8_t* __restrict__ y, int n,
    const float* __restrict__ partials, int nb, float* __restrict__ scale_out) {
  __shared__ float s[QT / 64];
  float m = 0.0f;
  for (int b = threadIdx.x; b < nb; b += QT) m = fmaxf(m, partials[b]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
  __syncthreads();
  float amax = s[0];
#pragma unroll
  for (int w = 1; w < QT / 64; ++w) amax = fmaxf(amax, s[w]);
  const float scale = amax > 0.0f ? amax / 448.0f : 1.0f;
  if (blockIdx.x == 0 && threadIdx.x == 0 && scale_out) *scale_out = scale;
  const float inv = 1.0f / scale;

  const long long nv = n >> 3;
  for (long long i = (long long)blockIdx.x * QT + threadIdx.x; i < nv; i += (long long)gridDim.x * QT) {
    const k3_u4 v = k3_ld16_nt(x + i * 8);
    k3_u2 o;
    o[0] = k3_pack_e4m3x4(k3_bf_lo(v[0]) * inv, k3_bf_hi(v[0]) * inv, k3_bf_lo(v[1]) * inv,
                          k3_bf_hi(v[1]) * inv);
    o[1] = k3_pack_e4m3x4(k3_bf_lo(v[2]) * inv, k3_bf_hi(v[2]) * inv, k3_bf_lo(v[3]) * inv,
                          k3_bf_hi(v[3]) * inv);
    k3_st8_nt(y + i * 8, o);
  }
  if (blockIdx.x == 0 && threadIdx.x < (n & 7)) {
    const long long e = nv * 8 + threadIdx.x;
    y[e] = (uint8_t)(k3_pack_e4m3x2(k3_bf(x[e]) * inv, 0.0f) & 0xffu);
  }
}

#ifdef K3_QUANT_V2
// One pass over HBM for large tensors: k3h_quant_fp8_mark, then k3h_quant_fp8_once, with
// the outputs of the pair at nb = 2048 bit for bit (partials included).  The pair reads
// x twice, and although the second pass comes from the MALL it costs as much as the
// first.  Here one persistent launch (256 workgroups of 1024 threads, one per CU) keeps
// the last 24 of a thread's vectors on the chip (15 in registers, 9 in LDS: 100.7 MB of
// x in all), meets at the partials, and quantises what it holds; only the vectors before
// those are read again, from the MALL.  Quarter s of workgroup g plays the pair's blocks
// 8 g + s and 8 g + 4 + s, so a thread's m-th vector is vector
// (8 g + 4 (m & 1) + s + 2048 (m >> 1)) * 256 + t and the chip sweeps x front to back.
// Measured over three rotating sets: n = 117 M 87.2 -> 74.8 us, 59 M 44.9 -> 33.7, 34 M
// 26.5 -> 21.2, 25 M 20.8 -> 18.7, 21 M 18.0 -> 17.8 (mark, dispatch and the meeting cost
// about 13 us): the host takes it for n >= 24 << 20.  At 117 M a workgroup spends 36 us
// reading (6.5 TB/s), 4 us meeting and 20 us on the second pass.
// A workgroup fills its CU, so another stream's kernel on one CU (one wave will do) keeps
// one of the 256 out until the others end: n = 117 M beside such a wave 120 us (the pair 97),
// 25 M 55 us (25); beside a large copy or GEMM both streams together take as long as with
// the pair.
// Requires n >= 8.
#define QO_NB 2048
#define QO_REG 15           // vectors a thread keeps in registers
#define QO_LDS 9            // and in LDS
#define QO_HELD (QO_REG + QO_LDS)
#define QO_UNSET 0xffffffffu  // a partial is a non-negative bf16 pattern << 16

extern "C" __global__ void __launch_bounds__(1024) k3h_quant_fp8_mark(uint32_t* __restrict__ partials) {
  partials[blockIdx.x * 1024 + threadIdx.x] = QO_UNSET;
}

K3_DEV uint32_t k3_qo_max(uint32_t m, k3_u4 v) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t a = v[j] & 0x7fff7fffu;
    const uint32_t lo = a & 0xffffu, hi = a >> 16;
    m = m > lo ? m : lo;
    m = m > hi ? m : hi;
  }
  return m;
}
K3_DEV k3_u2 k3_qo_codes(k3_u4 v, float inv) {
  k3_u2 o;
  o[0] = k3_pack_e4m3x4(k3_bf_lo(v[0]) * inv, k3_bf_hi(v[0]) * inv, k3_bf_lo(v[1]) * inv,
                        k3_bf_hi(v[1]) * inv);
  o[1] = k3_pack_e4m3x4(k3_bf_lo(v[2]) * inv, k3_bf_hi(v[2]) * inv, k3_bf_lo(v[3]) * inv,
                        k3_bf_hi(v[3]) * inv);
  return o;
}
K3_DEV uint32_t k3_qo_wave_max(uint32_t m) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t p = (uint32_t)__shfl_xor((int)m, o, 64);
    m = m > p ? m : p;
  }
  return m;
}

extern "C" __global__ void __launch_bounds__(1024) k3h_quant_fp8_once(
    const uint16_t* __restrict__ x, uint8_t* __restrict__ y, int n, uint32_t* __restrict__ partials,
    float* __restrict__ scale_out, int spin_ticks) {
  __shared__ k3_u4 held[QO_LDS][1024];
  __shared__ uint32_t red[2][16];
  const int tid = threadIdx.x, t = tid & 255, s = tid >> 8, wave = tid >> 6;
  const int b0 = 8 * (int)blockIdx.x + s;
  const long long nv = n >> 3;
  const k3_u4 zero = {0, 0, 0, 0};
  // slot m's vector of this thread (n < 2^31, so an index fits 32 bits); slots past
  // the end read the last vector and count as zero
  const uint32_t last = (uint32_t)nv - 1;
  auto vec = [&](int m) -> uint32_t {
    return (8u * blockIdx.x + 4u * (uint32_t)(m & 1) + (uint32_t)QO_NB * (uint32_t)(m >> 1)) * 256u +
           (uint32_t)tid;
  };
  auto at = [&](uint32_t i) { return (const k3_u4*)((const uint8_t*)x + 16u * (size_t)i); };
  auto hold = [&](int m) {
    const uint32_t i = vec(m);
    return __builtin_nontemporal_load(at(i < last ? i : last));
  };
  auto live = [&](int m, k3_u4 v) { return vec(m) <= last ? v : zero; };
  auto put = [&](uint32_t i, k3_u4 v, float inv) { k3_st8_nt(y + 8u * (size_t)i, k3_qo_codes(v, inv)); };
  const int steps = (int)((nv + (long long)QO_NB * 256 - 1) / ((long long)QO_NB * 256));
  const int M = 2 * steps;                             // vector slots (the last two may be past the end)
  const int S = M > QO_HELD ? M - QO_HELD : 0;         // the first S are read again
  uint32_t mx0 = 0, mx1 = 0;
  // S is even (M and QO_HELD are)
  // the slots read again (cacheable, so that they stay in the MALL), four by four with
  // the next four in flight; slots past S repeat the last pair
  auto again = [&](int m) { return vec(m < S ? m : S - 2 + (m & 1)); };
  k3_u4 v[2][4];
  if (S > 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[0][k] = *at(again(k));
    for (int m = 0; m < S; m += 8) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[1 - half][k] = *at(again(m + 4 * half + 4 + k));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
          mx0 = k3_qo_max(mx0, v[half][k]);
          mx1 = k3_qo_max(mx1, v[half][k + 1]);
        }
      }
    }
  }
  {
    k3_u4 l[QO_LDS];
#pragma unroll
    for (int k = 0; k < QO_LDS; ++k) {
      l[k] = hold(S + k);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < QO_LDS; ++k) {
      l[k] = live(S + k, l[k]);
      if (k & 1) mx1 = k3_qo_max(mx1, l[k]);
      else mx0 = k3_qo_max(mx0, l[k]);
      held[k][tid] = l[k];
    }
  }
  k3_u4 r[QO_REG];
#pragma unroll
  for (int k = 0; k < QO_REG; ++k) {
    r[k] = hold(S + QO_LDS + k);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < QO_REG; ++k) {
    r[k] = live(S + QO_LDS + k, r[k]);
    if ((QO_LDS + k) & 1) mx1 = k3_qo_max(mx1, r[k]);
    else mx0 = k3_qo_max(mx0, r[k]);
  }
  if (b0 == 0 && t < (n & 7)) {  // the n % 8 tail belongs to block 0
    const uint32_t a = x[nv * 8 + t] & 0x7fffu;
    mx0 = mx0 > a ? mx0 : a;
  }
  mx0 = k3_qo_wave_max(mx0);
  mx1 = k3_qo_wave_max(mx1);
  if ((tid & 63) == 0) {
    red[0][wave] = mx0;
    red[1][wave] = mx1;
  }
  __syncthreads();
  if (tid < 8) {
    const uint32_t* q = &red[tid >> 2][4 * (tid & 3)];
    uint32_t b = q[0];
#pragma unroll
    for (int k = 1; k < 4; ++k) b = b > q[k] ? b : q[k];
    __hip_atomic_store(partials + 8 * blockIdx.x + tid, b << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  // the first slots read again are requested before the wait
  if (S > 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[0][k] = __builtin_nontemporal_load(at(again(k)));
  }
  // every block's partial (slots tid and 1024 + tid): poll until it is set, for spin_ticks
  // (10 ns each) at most
  auto poll = [&](int slot) -> uint32_t {
    return __hip_atomic_load(partials + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  uint32_t p0, p1;
  {
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
      p0 = poll(tid);
      p1 = poll(1024 + tid);
      if (__ballot(p0 == QO_UNSET || p1 == QO_UNSET) == 0) break;
      if ((uint64_t)__builtin_amdgcn_s_memrealtime() - t0 >= (uint64_t)spin_ticks) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
  // the max over the partials that are not NaN patterns (those compare as bits in
  // `partials`, and the scale ignores them)
  auto fold = [&](float f, uint32_t p) { return p == QO_UNSET ? f : __builtin_fmaxf(f, __uint_as_float(p)); };
  __shared__ float fred[16];
  __shared__ int short_of[16];
  auto wave_fold = [&]() {
    float f = fold(fold(0.0f, p0), p1);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) f = __builtin_fmaxf(f, __shfl_xor(f, o, 64));
    if ((tid & 63) == 0) fred[wave] = f;
  };
  wave_fold();
  {
    const bool miss = __ballot(p0 == QO_UNSET || p1 == QO_UNSET) != 0;
    if ((tid & 63) == 0) short_of[wave] = miss;
  }
  __syncthreads();
  float amax = 0.0f;
  bool any = false;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    amax = __builtin_fmaxf(amax, fred[k]);
    any |= short_of[k] != 0;
  }
  if (any) {
    // A workgroup that is not resident yet cannot have set its partials (another stream's
    // kernel holds its CU): the waiting ones take the missing blocks' maxima themselves, one
    // block a turn, spread over the missing ones by workgroup, storing what they find for
    // the others and looking again what those have found.  No workgroup ever depends on
    // another one running, and a turn sets at least one of its partials, so this ends.
    __shared__ uint64_t missing[32];  // bit i of [k]: block 64 k + i
    for (;;) {
      const uint64_t m0 = __ballot(p0 == QO_UNSET), m1 = __ballot(p1 == QO_UNSET);
      if ((tid & 63) == 0) {
        missing[wave] = m0;
        missing[16 + wave] = m1;
      }
      __syncthreads();
      uint32_t left = 0;
      for (int k = 0; k < 32; ++k) left += (uint32_t)__popcll(missing[k]);
      if (left == 0) break;
      // the workgroup's pick among the `left` missing blocks, the same in every thread
      uint32_t pick = (blockIdx.x * left) / gridDim.x;
      int b = 0;
      for (int k = 0; k < 32; ++k) {
        uint64_t m = missing[k];
        const uint32_t c = (uint32_t)__popcll(m);
        if (pick < c) {
          for (; pick > 0; --pick) m &= m - 1;
          b = 64 * k + __builtin_ctzll(m);
          break;
        }
        pick -= c;
      }
      uint32_t bm = 0;
#pragma unroll 1
      for (uint32_t i = (uint32_t)(b + QO_NB * s) * 256u + (uint32_t)t; i <= last; i += 4u * QO_NB * 256u)
        bm = k3_qo_max(bm, *at(i));
      if (b == 0 && tid < (n & 7)) {
        const uint32_t a = x[nv * 8 + tid] & 0x7fffu;
        bm = bm > a ? bm : a;
      }
      bm = k3_qo_wave_max(bm);
      if ((tid & 63) == 0) red[0][wave] = bm;
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 16; ++k) bm = bm > red[0][k] ? bm : red[0][k];
      const uint32_t p = bm << 16;
      if (tid == 0)
        __hip_atomic_store(partials + b, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (p0 == QO_UNSET) p0 = b == tid ? p : poll(tid);
      if (p1 == QO_UNSET) p1 = b == 1024 + tid ? p : poll(1024 + tid);
    }
    wave_fold();
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) amax = __builtin_fmaxf(amax, fred[k]);
  }
  const float scale = amax > 0.0f ? amax / 448.0f : 1.0f;
  if (blockIdx.x == 0 && tid == 0 && scale_out) *scale_out = scale;
  const float inv = 1.0f / scale;
  uint32_t tid2 = (uint32_t)tid;
  asm volatile("" : "+v"(tid2));  // no address is kept across the wait
  auto vec2 = [&](int m) { return vec(m) - (uint32_t)tid + tid2; };

  // the held vectors, then the ones read again
#pragma unroll
  for (int k = 0; k < QO_REG; ++k) {
    const uint32_t i = vec2(S + QO_LDS + k);
    if (i <= last) put(i, r[k], inv);
  }
#pragma unroll
  for (int k = 0; k < QO_LDS; ++k) {
    const uint32_t i = vec2(S + k);
    if (i <= last) put(i, held[k][tid], inv);
  }
  for (int m = 0; m < S; m += 8) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[1 - half][k] = __builtin_nontemporal_load(at(again(m + 4 * half + 4 + k)));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (m + 4 * half + k < S) put(vec(m + 4 * half + k), v[half][k], inv);
    }
  }
  if (b0 == 0 && t < (n & 7)) {
    const long long e = nv * 8 + t;
    y[e] = (uint8_t)(k3_pack_e4m3x2(k3_bf(x[e]) * inv, 0.0f) & 0xffu);
  }
}
#endif  // K3_QUANT_V2
