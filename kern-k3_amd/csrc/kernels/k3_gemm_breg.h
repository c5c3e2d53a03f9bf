// Register-weight items for the MoE expert GEMMs (module k3h_moe_gemm, included by
// k3h_moe_gemm.hip after the 256-column kernels and k3_gemm_wide.h, whose layouts,
// item split and helpers it shares).  Entries kern_k3h_moe_gemm3_situ_mx (fc1),
// kern_k3h_moe_gemm3_acc (its tiling with f32 output) and kern_k3h_moe_gemm3_bf16 (fc2 over
// few tiles, by k3h_moe_gemm_mx's rule): the same products as the 256-column kernels bit for bit (the same MFMA
// sequence per output element), for 512 <= K <= 3584, K % 256 == 0.
//
// Work item: route tile t (128 rows) x one 256-column block, one 256-thread
// workgroup, two workgroups per CU.  Wave w owns all the rows and the columns
// 64 w .. + 64 (an up and a gate tile: one MX block of each row), so a weight
// operand is used by one wave only and is loaded straight into its registers; only
// the A rows, which all four waves read, go through LDS.  Against waves of 64 x 128
// with both operands in LDS the same operand reads come out of LDS, but half the
// direct-to-LDS writes go in (16 instead of 32 KB per workgroup and step), the A ring
// holds four steps in the LDS that held two, and the operands wait on counted
// vector-memory waits instead of a full one per step: fc1 over 548 tiles (16,384
// tokens, top-16) 1217-1242 -> 1160-1184 us, over 161 tiles 395 -> 369 us.
//
// Few rows per tile (short chunks): HBM streams each live expert's weights once and
// the padded rows' MFMAs, A rows and activations are what is left to save.  The
// routing tables pad a tile by repeating a row index, so every row past the last
// distinct index has the last one's results: a tile that needs at most 32 (64) rows
// runs one (two) m tiles and stores the last computed row for the rest (37 tokens,
// top-8, 39 tiles: 127 -> 91 us; 720 tokens, 56 tiles: 163 -> 127 us; the weights
// alone stream in 65 / 95 us in that order of loads).  Its free registers hold weights
// six steps ahead instead of two, and its free LDS the A rows eight (six) steps ahead
// (39 tiles 95.6 us at four / five steps, 91.2 at six; 56 tiles 133.4 -> 127; eight
// steps no faster).
//
// Without a row list (fc2) every row is computed.  Finding the repeated rows by comparing
// them on the way reads them all the same and gains nothing (39 tiles 71.9 against 72.0 us;
// with the rows known it would be 60: the routing's cta_limit holds them, but the call has no
// parameter for it).
//
// Cache policy: up to 1.25 tiles per expert the weights are loaded non-temporally (one
// tile reads them: 101 -> 94 us at 39 tiles, 143 -> 132 at 56, 184 -> 178 at 63); above, the
// L2s serve an expert's second tile, full (548 tiles: 1174 against 1430 us non-temporal) or
// thin (4000 tokens top-8, 91-99 tiles with thin last ones: 235 us where those loaded
// non-temporally, 221 now; 6000 tokens 285 and 282).
//
// Measured and not kept: the persistent form of these items (two workgroups per CU, the
// next item's A stages and scales requested during the current one's last steps): fc1
// 1412-1490 us, fc2 668 us over 548 tiles.  Its extra state spills at every item boundary,
// and the second workgroup of the CU already covers an item's start.
#pragma once

#define K3B_STAGES 4
#define K3B_STAGE_BYTES 16384
#define K3B_SAT_OFF (K3B_STAGES * K3B_STAGE_BYTES)
#define K3B_KGM 112  // A-scale table bytes per row: K <= 3584
#define K3B_LDS_BYTES (K3B_SAT_OFF + 128 * K3G_SAT_ROW(K3B_KGM))
static_assert(2 * K3B_LDS_BYTES <= 163840, "two workgroups per CU");

#define K3B_EP_ROW 144  // fc1 epilogue: a row's 128 code bytes in LDS, padded

K3_DEV uint8_t* k3b_smem() {
  __shared__ __attribute__((aligned(16))) uint8_t smem[K3B_LDS_BYTES];
  return smem;
}

// Memory operations stay on their side (the counted waits below rely on the
// issue order of the vector-memory operations).
#define K3B_FENCE()                       \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    asm volatile("" ::: "memory");        \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

typedef __attribute__((address_space(1))) k3_u4 k3b_gu4;
typedef __attribute__((address_space(1))) uint32_t k3b_gu1;

// The value that lane 31 + 32 h (row 31 of an m tile, this half-wave's columns) holds.
K3_DEV uint32_t k3b_last(uint32_t v, int h) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
  return h ? hi : lo;
}

// f(0), f(1), .. f(N - 1), the index a compile-time constant.
template <int N, int I = 0, class F>
K3_DEV void k3b_each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    k3b_each<N, I + 1>(f);
  }
}

// The K loop of one item over the tile's first 32 MT rows, for the wave's 64 columns.
// NB: weight buffers (a step's weights are requested NB steps ahead); PA: stages the A
// rows are requested ahead (ring of RS stages); NTW: weights loaded non-temporally.
template <int MT, int NB, int PA, int RS, bool NTW>
K3_DEV void k3b_loop(k3_v16f (&acc)[MT][2], const uint8_t* __restrict__ a,
                     const uint8_t* __restrict__ a_sf, int v0, int v1,
                     const uint8_t* wb0, const uint8_t* wb1, const uint8_t* sbu, int K, int w,
                     int lane) {
  constexpr int STG = MT * 4096;  // stage bytes: 32 MT rows x 128
  constexpr int P = 5 + MT;       // vector-memory operations a wave issues per step
  constexpr int LK = MT < 2 ? 1 : 2;  // units the A operands are read ahead
  static_assert(RS * STG <= K3B_SAT_OFF && (RS & (RS - 1)) == 0 && RS > PA, "A ring");
  static_assert(2 * MT * NB % 4 == 0, "the A operand buffers' turn");
  static_assert(NB * P < 64, "the vector-memory counter");
  static_assert(PA + 1 >= NB, "every A stage is requested before the last KS % NB steps");
  const int h = lane >> 5, j = lane & 31;
  const int KG = K / 32, KS = K / K3G_KSTEP;
  uint8_t* lds = k3b_smem();
  uint8_t* sat = lds + K3B_SAT_OFF;
  uint32_t lo16 = 16u * (uint32_t)lane, lo8 = 8u * (uint32_t)lane;

  // scalar-base loads: the step's wave-uniform address is held in scalar registers and
  // the lane's offset added last; requests past the last step repeat it, so that every
  // step of the counted loop issues the same operations (the use after the loop keeps
  // those whose data no step reads)
  k3_u4 bv[NB][2][2];  // [buffer][substep][n tile]
  uint32_t sb[NB];
  auto load_b = [&](auto bi_c, auto s_c, int k) {
    constexpr int BI = decltype(bi_c)::value, s = decltype(s_c)::value;
    k = k < KS ? k : KS - 1;
    const uint8_t *p0 = wb0 + (size_t)k * 2048 + s * 1024, *p1 = wb1 + (size_t)k * 2048 + s * 1024;
    asm volatile("" : "+s"(p0), "+s"(p1));
    const k3b_gu4 *q0 = (const k3b_gu4*)((k3g_gu8*)p0 + lo16), *q1 = (const k3b_gu4*)((k3g_gu8*)p1 + lo16);
    bv[BI][s][0] = NTW ? __builtin_nontemporal_load(q0) : *q0;
    bv[BI][s][1] = NTW ? __builtin_nontemporal_load(q1) : *q1;
  };
  auto load_sb = [&](int k) -> uint32_t {
    k = k < KS ? k : KS - 1;
    const uint8_t* p = sbu + (size_t)k * 512;
    asm volatile("" : "+s"(p));
    return *(const k3b_gu1*)((k3g_gu8*)p + lo8);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  k3b_each<NB>([&](auto i) {
    load_b(i, I0{}, i);
    load_b(i, I1{}, i);
    sb[i] = load_sb(i);
  });
  K3B_FENCE();
  // this wave's A loads: row slices 8 q .. + 8, q = MT w + b
  uint32_t arow[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    const int r = 8 * (MT * w + b) + (lane >> 3);  // r / 64 is wave-uniform
    arow[b] = (uint32_t)__shfl(MT < 4 || w < 2 ? v0 : v1, r & 63, 64) * (uint32_t)K +
              16u * (uint32_t)((lane & 7) ^ (lane >> 3) ^ ((MT * w + b) & 1));
  }
  auto issue_a = [&](int k) {
    uint8_t* st = lds + (k & (RS - 1)) * STG;
    const uint8_t* ak = a + (size_t)(k < KS ? k : KS - 1) * K3G_KSTEP;
    asm volatile("" : "+s"(ak));
#pragma unroll
    for (int b = 0; b < MT; ++b)
      __builtin_amdgcn_global_load_lds((k3g_gu8*)ak + arow[b],
                                       (k3g_lds_t*)(st + (MT * w + b) * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int k = 0; k < PA; ++k) issue_a(k);
  {
    // All of a row's scales in flight at once, C dwords per thread.  A row that fills the
    // table (K = 3584) gives each thread C consecutive ones, in wide loads (548 tiles 1164
    // us, dword by dword 1167-1183); a shorter one repeats its last (K = 3072: 67 us over
    // 39 tiles, 69 with a loop over the dwords).
    constexpr int TPR = 8 / MT, C = (K3B_KGM / 4 + TPR - 1) / TPR;  // threads per A-scale row
    const int row = threadIdx.x / TPR, part = threadIdx.x % TPR, KGd = KG / 4;
    const uint32_t src = (uint32_t)__shfl(MT < 4 || w < 2 ? v0 : v1, row & 63, 64);
    const uint32_t* sr = (const uint32_t*)(a_sf + (size_t)src * KG);
    uint32_t* dr = (uint32_t*)(sat + row * K3G_SAT_ROW(K3B_KGM));
    uint32_t x[C];
    if (KGd == TPR * C) {
#pragma unroll
      for (int c = 0; c < C; ++c) x[c] = sr[C * part + c];
#pragma unroll
      for (int c = 0; c < C; ++c) dr[C * part + c] = x[c];
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) x[c] = sr[min(part + TPR * c, KGd - 1)];
#pragma unroll
      for (int c = 0; c < C; ++c) dr[min(part + TPR * c, KGd - 1)] = x[c];
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[mt][nt][q] = 0.0f;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // A operand of unit (s, mt): the lane's row 32 mt + j, chunks 4 s + h and 4 s + 2 + h;
  // the swizzle depends on r % 16 only
  uint32_t ao[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    ao[s][0] = 16u * (uint32_t)k3g_aslot(j, 4 * s + h);
    ao[s][1] = 16u * (uint32_t)k3g_aslot(j, 4 * s + 2 + h);
  }
  k3_v8i ab[4];
  auto rd_a = [&](const uint8_t* st, int s, int mt) -> k3_v8i {
    const k3_u4 lo = *(const k3_u4*)(st + ao[s][0] + 4096 * mt);
    const k3_u4 hi = *(const k3_u4*)(st + ao[s][1] + 4096 * mt);
    return (k3_v8i){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
                    (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
  };
  const uint8_t* satl = sat + j * K3G_SAT_ROW(K3B_KGM);
  auto rd_sa = [&](int ks, int mt) -> uint32_t {
    return *(const uint32_t*)(satl + 32 * mt * K3G_SAT_ROW(K3B_KGM) + 4 * ks) >> (8 * h);
  };
  uint32_t sa[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) sa[mt] = rd_sa(0, mt);
#pragma unroll
  for (int u = 0; u < LK; ++u) ab[u] = rd_a(lds, u / MT, u % MT);

  auto pin = [&]() {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) asm volatile("" : "+v"(acc[mt][nt]));
  };
  // One K step with weights in buffer BI.  TAIL: everything it reads has landed and no
  // later step needs more, so it requests nothing and waits for nothing.
  auto step = [&](int ks, auto bi_c, auto tail_c) {
    constexpr int BI = decltype(bi_c)::value;
    constexpr bool TAIL = decltype(tail_c)::value;
#pragma unroll
    for (int b = 0; b < MT; ++b) asm volatile("" : "+v"(arow[b]));
    asm volatile("" : "+v"(lo16), "+v"(lo8));
    const uint8_t* st = lds + (ks & (RS - 1)) * STG;
    const uint8_t* sn = lds + ((ks + 1) & (RS - 1)) * STG;
    auto half = [&](auto s_c) {
      constexpr int s = decltype(s_c)::value;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        constexpr int U0 = 2 * MT * BI;
        const int u = s * MT + mt, ahead = u + LK;
        const int cur = (U0 + u) & 3, nxt = (U0 + ahead) & 3;
        if (ahead < 2 * MT) ab[nxt] = rd_a(st, ahead / MT, ahead % MT);
        else ab[nxt] = rd_a(sn, 0, ahead - 2 * MT);
        const k3_u4 &b0 = bv[BI][s][0], &b1 = bv[BI][s][1];
        const k3_v8i w0 = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], 0, 0, 0, 0};
        const k3_v8i w1 = {(int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3], 0, 0, 0, 0};
        acc[mt][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            w0, ab[cur], acc[mt][0], 4, 0, s, (int)sb[BI], 2 * s, (int)sa[mt]);
        acc[mt][1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            w1, ab[cur], acc[mt][1], 4, 0, 2 + s, (int)sb[BI], 2 * s, (int)sa[mt]);
      }
#pragma unroll
      for (int u = 0; u < MT; ++u) {
        __builtin_amdgcn_sched_group_barrier(K3G_SG_DS_READ, 2, 0);
        __builtin_amdgcn_sched_group_barrier(K3G_SG_MFMA, 2, 0);
      }
    };
    // the step's first weights and scales have landed (left to itself the compiler
    // would wait here for every load in flight)
    if constexpr (!TAIL) __builtin_amdgcn_s_waitcnt(K3W_VMCNT(2 + (NB - 1) * P));
    half(I0{});
    uint32_t san[MT];
    pin();
    K3B_FENCE();
    if constexpr (!TAIL) {
      load_b(bi_c, I0{}, ks + NB);
      K3B_FENCE();
      // this step's second weights and the A rows of step ks + 1 have landed
      constexpr int WB = 2 + (NB - 1) * P, WA = 5 + (PA - 2) * P;
      __builtin_amdgcn_s_waitcnt(K3W_VMCNT(WA < WB ? WA : WB));
      __builtin_amdgcn_s_barrier();
      K3B_FENCE();
      issue_a(ks + PA);
      K3B_FENCE();
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) san[mt] = rd_sa(ks + 1, mt);
    half(I1{});
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) sa[mt] = san[mt];
    pin();
    K3B_FENCE();
    if constexpr (!TAIL) {
      sb[BI] = load_sb(ks + NB);
      K3B_FENCE();
      load_b(bi_c, I1{}, ks + NB);
      K3B_FENCE();
    }
  };
  int ks = 0;  // KS is even
  for (; ks + NB <= KS; ks += NB)
    k3b_each<NB>([&](auto i) { step(ks + i, i, std::false_type{}); });
  K3B_FENCE();
  __builtin_amdgcn_s_waitcnt(0);  // no load into LDS outlives the workgroup
  if constexpr (NB > 2) {         // the last KS % NB: every wave's requests have landed
    if (ks < KS) {
      __builtin_amdgcn_s_barrier();
      K3B_FENCE();
      k3b_each<NB - 1>([&](auto i) {
        if (ks + i < KS) step(ks + i, i, std::true_type{});
      });
    }
  }
  // the counted waits of the last turn include loads past the last step: they stay
#pragma unroll
  for (int i = 0; i < NB; ++i)
    asm volatile("" ::"v"(bv[i][0][0]), "v"(bv[i][0][1]), "v"(bv[i][1][0]), "v"(bv[i][1][1]),
                 "v"(sb[i]));
}

template <class Epi>
K3_DEV void k3b_run(const uint8_t* __restrict__ a, const uint8_t* __restrict__ a_sf,
                    const int* __restrict__ a_rows, const uint8_t* __restrict__ wt,
                    const uint16_t* __restrict__ wsf, const int* __restrict__ num_tiles,
                    const int* __restrict__ cta_batch, int E, int N, int K, int max_tiles,
                    Epi&& epi) {
  int tile, cb;
  if (!k3g_item(num_tiles, max_tiles, tile, cb)) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int lane = threadIdx.x & 63;
  // source rows of the tile's rows lane and 64 + lane (requested beside the expert)
  int v0 = tile * K3G_TILE_M + lane, v1 = v0 + 64;
  if (a_rows) {
    v0 = a_rows[v0];
    v1 = a_rows[v1];
  }
  const int e = cta_batch[tile];
  if (e < 0 || e >= E) return;
  const int KT = K / 64, KS = K / K3G_KSTEP, NT = N / 32;
  const uint8_t* wb0 = wt + ((size_t)e * NT + cb * (K3G_TILE_N / 32) + 2 * w) * KT * 1024;
  const uint8_t* wb1 = wb0 + (size_t)KT * 1024;
  const uint8_t* sbu = (const uint8_t*)wsf +
                       ((size_t)e * (NT / 4) + cb * (K3G_TILE_N / 128) + (w >> 1)) * KS * 512 +
                       4 * (w & 1);
  asm volatile("" : "+s"(wb0), "+s"(wb1), "+s"(sbu));
  // rows past the last distinct source row repeat its results
  const int lastv = __builtin_amdgcn_readlane(v1, 63);
  const uint64_t d1 = __ballot(v1 != lastv), d0 = __ballot(v0 != lastv);
  const int need = d1 ? 128 : d0 ? 65 - __builtin_clzll(d0) : 1;  // rows to compute
  v0 = v0 < 0 ? 0 : v0;
  v1 = v1 < 0 ? 0 : v1;
  // About one tile per expert: no other tile reads these weights, and non-temporal loads
  // stream them faster; with more, the L2s serve the second tile.
  const int live = *num_tiles;
  const bool once = live <= E + E / 4;
  auto item = [&](auto mt_c, auto nb_c, auto pa_c, auto rs_c) {
    constexpr int MT = decltype(mt_c)::value, NB = decltype(nb_c)::value;
    constexpr int PA = decltype(pa_c)::value, RS = decltype(rs_c)::value;
    k3_v16f acc[MT][2];
    if (once) k3b_loop<MT, NB, PA, RS, true>(acc, a, a_sf, v0, v1, wb0, wb1, sbu, K, w, lane);
    else k3b_loop<MT, NB, PA, RS, false>(acc, a, a_sf, v0, v1, wb0, wb1, sbu, K, w, lane);
    epi(acc, mt_c, tile, cb, e, w, lane);
  };
  using std::integral_constant;
  if (need <= 32)
    item(integral_constant<int, 1>{}, integral_constant<int, 6>{}, integral_constant<int, 8>{},
         integral_constant<int, 16>{});
  else if (need <= 64)
    item(integral_constant<int, 2>{}, integral_constant<int, 6>{}, integral_constant<int, 6>{},
         integral_constant<int, 8>{});
  else
    item(integral_constant<int, 4>{}, integral_constant<int, 2>{}, integral_constant<int, 3>{},
         integral_constant<int, 4>{});
}

// bf16 out, stored as by k3w_gemm_bf16.
K3_DEV void k3b_gemm_bf16(K3G_PARAMS, uint16_t* __restrict__ out) {
  k3b_run(a, a_sf, a_rows, wt, wsf, num_tiles, cta_batch, E, N, K, max_tiles,
          [&](auto& acc, auto mt_c, int tile, int cb, int, int w, int lane) {
    constexpr int MT = decltype(mt_c)::value;
    const int h = lane >> 5, j = lane & 31, p = lane & 1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        uint32_t d[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) d[k] = k3_pack_bf2(acc[mt][nt][2 * k], acc[mt][nt][2 * k + 1]);
        k3g_swap(d[0], d[4]);
        k3g_swap(d[1], d[5]);
        k3g_swap(d[2], d[6]);
        k3g_swap(d[3], d[7]);
        const k3_u4 X = {d[0], d[1], d[4], d[5]}, Y = {d[2], d[3], d[6], d[7]};
        const k3_u4 snd = p ? X : Y;
        k3_u4 rcv;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          rcv[c] = (uint32_t)__builtin_amdgcn_mov_dpp((int)snd[c], K3_DPP_QP_1032, 0xf, 0xf, false);
        const size_t row = (size_t)tile * K3G_TILE_M + 32 * mt + j;
        uint16_t* o = out + (row & ~(size_t)1) * N + cb * K3G_TILE_N + 64 * w + 32 * nt +
                      8 * (2 * h + p);
        k3_st16(o, p ? rcv : X);
        k3_st16(o + N, p ? Y : rcv);
        if constexpr (MT < 4) {
          if (mt == MT - 1) {  // rows past the computed ones: row 32 MT - 1's chunks
            k3_u4 bx, by;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              bx[c] = k3b_last(X[c], h);
              by[c] = k3b_last(Y[c], h);
            }
#pragma unroll
            for (int m = MT; m < 4; ++m) {
              uint16_t* ob = out + ((size_t)tile * K3G_TILE_M + 32 * m + j) * N + cb * K3G_TILE_N +
                             64 * w + 32 * nt + 16 * h;
              k3_st16(ob, bx);
              k3_st16(ob + 8, by);
            }
          }
        }
      }
  });
}

K3_DEV void k3b_gemm_situ_mx(K3G_PARAMS, uint8_t* __restrict__ out_q, uint8_t* __restrict__ out_sf,
                             const float* __restrict__ alpha, const float* __restrict__ beta) {
  k3b_run(a, a_sf, a_rows, wt, wsf, num_tiles, cta_batch, E, N, K, max_tiles,
          [&](auto& acc, auto mt_c, int tile, int cb, int e, int w, int lane) {
    constexpr int MT = decltype(mt_c)::value;
    const int h = lane >> 5, j = lane & 31;
    const float al = alpha[e], be = beta[e];
    const float ial = 1.0f / al, ibe = 1.0f / be;
    const int form = al == 4.0f ? (be == 25.0f ? 0 : 1) : 2;
    const int NA = N / 2;
    // The codes and scale bytes go through LDS (free once every wave has left the K
    // loop), so that the stores write whole 128-byte lines: the item's 4 blocks of a row.
    uint8_t* lq = k3b_smem();
    uint8_t* lsf = lq + K3G_TILE_M * K3B_EP_ROW;
    __syncthreads();
    auto blocks = [&](auto form_c) {
      constexpr int FORM = decltype(form_c)::value;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int r = 32 * mt + j;
        k3_u4 q;
        const uint32_t sf = k3g_situ_codes<FORM>(acc[mt][0], acc[mt][1], al, ial, be, ibe, q);
        k3_st16(lq + r * K3B_EP_ROW + 32 * w + 16 * h, q);
        if (h == 0) lsf[4 * r + w] = (uint8_t)sf;
      }
    };
    if (form == 0) blocks(std::integral_constant<int, 0>{});
    else if (form == 1) blocks(std::integral_constant<int, 1>{});
    else blocks(std::integral_constant<int, 2>{});
    __syncthreads();
    const size_t row0 = (size_t)tile * K3G_TILE_M;
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // rows past the computed ones: the last computed row's
      const int r = 32 * i + (threadIdx.x >> 3), c = threadIdx.x & 7;
      const int rs = i < MT ? r : 32 * MT - 1;
      k3_st16(out_q + (row0 + r) * NA + 128 * cb + 16 * c,
              *(const k3_u4*)(lq + rs * K3B_EP_ROW + 16 * c));
    }
    if (threadIdx.x < K3G_TILE_M) {
      const int r = threadIdx.x, rs = r < 32 * MT ? r : 32 * MT - 1;
      const uint32_t sf4 = *(const uint32_t*)(lsf + 4 * rs);
      uint8_t* o = out_sf + (row0 + r) * (NA / 32) + 4 * cb;
      if (((uintptr_t)out_sf & 3) == 0) {
        *(uint32_t*)o = sf4;
      } else {  // 2-byte aligned
        ((uint16_t*)o)[0] = (uint16_t)sf4;
        ((uint16_t*)o)[1] = (uint16_t)(sf4 >> 16);
      }
    }
  });
}

K3_DEV void k3b_gemm_acc(K3G_PARAMS, float* __restrict__ out) {
  k3b_run(a, a_sf, a_rows, wt, wsf, num_tiles, cta_batch, E, N, K, max_tiles,
          [&](auto& acc, auto mt_c, int tile, int cb, int, int w, int lane) {
    constexpr int MT = decltype(mt_c)::value;
    const int h = lane >> 5, j = lane & 31;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float* orow = out + ((size_t)tile * K3G_TILE_M + 32 * mt + j) * N + cb * K3G_TILE_N + 64 * w;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *(k3_u4*)(orow + 32 * nt + 4 * h + 8 * g) =
              (k3_u4){__float_as_uint(acc[mt][nt][4 * g]), __float_as_uint(acc[mt][nt][4 * g + 1]),
                      __float_as_uint(acc[mt][nt][4 * g + 2]), __float_as_uint(acc[mt][nt][4 * g + 3])};
    }
    if constexpr (MT < 4) {  // rows past the computed ones: row 32 MT - 1's values
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          k3_u4 b;
#pragma unroll
          for (int c = 0; c < 4; ++c) b[c] = k3b_last(__float_as_uint(acc[MT - 1][nt][4 * g + c]), h);
          for (int m = MT; m < 4; ++m)
            *(k3_u4*)(out + ((size_t)tile * K3G_TILE_M + 32 * m + j) * N + cb * K3G_TILE_N + 64 * w +
                      32 * nt + 4 * h + 8 * g) = b;
        }
    }
  });
}

#define K3B_ENTRIES                                                                              \
  extern "C" __global__ void __launch_bounds__(256, 2)                                           \
      kern_k3h_moe_gemm3_acc(K3G_PARAMS, float* __restrict__ out) {                              \
    k3b_gemm_acc(K3G_ARGS, out);                                                                 \
  }                                                                                              \
  extern "C" __global__ void __launch_bounds__(256, 2)                                           \
      kern_k3h_moe_gemm3_bf16(K3G_PARAMS, uint16_t* __restrict__ out) {                          \
    k3b_gemm_bf16(K3G_ARGS, out);                                                                \
  }                                                                                              \
  extern "C" __global__ void __launch_bounds__(256, 2)                                           \
      kern_k3h_moe_gemm3_situ_mx(K3G_PARAMS, uint8_t* __restrict__ out_q,                        \
                                 uint8_t* __restrict__ out_sf, const float* __restrict__ alpha,  \
                                 const float* __restrict__ beta) {                               \
    k3b_gemm_situ_mx(K3G_ARGS, out_q, out_sf, alpha, beta);                                      \
  }
