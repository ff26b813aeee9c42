// gemm_mid_kernel: bf16 MFMA GEMMs whose whole output is one round of small
// tiles (SigLIP and the prefix at one request, the batched action expert).
//
//   acc[m][n] = sum_k A[m][k] * B[n][k]      A: activations, B: nn.Linear weight
//
// With one workgroup per CU nothing but the workgroup itself can hide a slab's
// barrier, LDS and MFMA latency, so it has 8 waves (two per SIMD): either all of
// them share one tile of BM x BN (KG = 1), or two groups of four each compute
// the whole tile over every other 64-wide K slab (KG = 2), which halves the
// steps of the K loop, and add their accumulators through the LDS at the end.
// A step moves KG slabs through an NST-deep LDS ring (LDS DMA, one barrier per
// step, the loads of step s + NST - 1 between the MFMAs of step s).
//
// Blocks are 32 x 32 with the weight rows as the MFMA's A operand, so that a lane
// ends with one output row; v_permlane32_swap joins the half-waves' runs of 4
// columns to chunks of 8.  With KG = 2 group g finishes chunk g of every block.
// The epilogue's operands are read before the K loop: nothing after it waits for
// memory but the stores.
#include "gemm_epilogue.h"

namespace fvx {

template <int RB, int JN, int WGM, int WGN, int KG, int NST>
struct MidCfg {
  static constexpr int BM = 32 * RB * WGM, BN = 32 * JN * WGN;
  static constexpr int NW = 8 / KG;                 // waves per K group
  static constexpr int SLAB = (BM + BN) * 128, STAGE = KG * SLAB;
  static constexpr int LA = BM / (8 * NW), LB = BN / (8 * NW), LPW = LA + LB;
  static constexpr int AC = RB * JN == 1 ? 2 : 1;   // accumulators per block (k-steps alternate)
  static_assert(WGM * WGN == NW && BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "waves");
  static_assert(NST >= 3 && NST * STAGE <= 152 * 1024, "LDS");
  // the K groups' exchange reuses the ring
  static_assert(8 * RB * JN * 2048 + 2 * 8 * RB * 128 <= NST * STAGE, "exchange");
};

// XF bit 0: the row sums of squares are handed over (ss_in); bit 1: they are
// taken in the K loop; bit 2: the output's are handed on (ss_out); bit 3, PLAIN:
// the plain epilogue (plain_epilogue_ok).
template <int MODE, int RB, int JN, int WGM, int WGN, int KG, int NST, int XF>
__global__ __launch_bounds__(512, 1) void gemm_mid_kernel(GemmArgs p, int m_tiles, int n_tiles) {
  typedef MidCfg<RB, JN, WGM, WGN, KG, NST> C;
  constexpr int LA = C::LA, LB = C::LB, LPW = C::LPW, AC = C::AC, NW = C::NW;
  constexpr int BM = C::BM, BN = C::BN, STAGE = C::STAGE, SLAB = C::SLAB;
  constexpr int NB = MODE == FVX_GEMM_GEGLU ? 2 : 1, JO = JN / NB;  // output blocks
  constexpr bool RPX = (XF & 1) != 0, SUMX = (XF & 2) != 0, HOX = (XF & 4) != 0;
  constexpr bool SP = (XF & 8) != 0 && MODE == FVX_GEMM_PLAIN;
  constexpr int HN = 2 / KG;  // chunks per block that a lane finishes
  __shared__ __align__(16) char smem[NST * STAGE];
  warm_kernargs<sizeof(GemmArgs) + 16>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / NW, w = wave % NW, wm = w / WGN, wn = w % WGN;
  const int fr = lane & 31, hk = lane >> 5, sw = (lane >> 1) & 7;
  const int bid = xcd_remap(blockIdx.x, m_tiles * n_tiles);
  const int nt = bid / m_tiles, mt = bid - nt * m_tiles;
  const int M = (int)p.m, N = (int)p.n, K = (int)p.k;
  const int steps = ((K + 63) / 64 + KG - 1) / KG;
  const int m0 = mt * BM, n0 = nt * (BN / NB);

  // DMA of this wave's 8 LA rows of A and 8 LB rows of B of its group's slab
  // (GEGLU: gate rows, then up rows), 8 rows of 128 bytes per load; lane l
  // fetches row l / 8, 16-byte chunk (l % 8) ^ ((row >> 1) & 7).  Rows past the
  // operand and chunks past K read as zeros.
  const int lr = lane >> 3, lc = lane & 7;
  const int ra = m0 + 8 * LA * w, br = 8 * LB * w;
  const bool up = NB == 2 && br >= BN / 2;
  const int rb = n0 + (up ? br - BN / 2 : br);
  auto rows_in = [](int left, int most) { return left <= 0 ? 0 : (left < most ? left : most); };
  const uint32_t lda2 = (uint32_t)p.lda * 2, ldb2 = (uint32_t)p.ldb * 2;
  const i32x4_t rA = make_rsrc4((const bf16_t*)p.a + (int64_t)ra * p.lda,
                                (uint32_t)rows_in(M - ra, 8 * LA) * lda2);
  const i32x4_t rB = make_rsrc4((const bf16_t*)(up ? p.b2 : p.b) + (int64_t)rb * p.ldb,
                                (uint32_t)rows_in(N - rb, 8 * LB) * ldb2);
  static_assert(LA % 2 == 0 && LB % 2 == 0, "a load's chunk parity is its index's");
  const int c0 = lc ^ (lr >> 1);
  const uint32_t la0 =
      __builtin_amdgcn_readfirstlane(lds_addr(smem) + kg * SLAB + w * LA * 1024);
  const uint32_t lb0 =
      __builtin_amdgcn_readfirstlane(lds_addr(smem) + kg * SLAB + BM * 128 + w * LB * 1024);
  // load x (A's LA, then B's LB) of step s's slab into ring stage sg
  auto issue1 = [&](int s, int sg, int x) {
    const bool isa = x < LA;
    const int i = isa ? x : x - LA, t = s * KG + kg, ch = c0 ^ (4 * (i & 1));
    const uint32_t ld2 = isa ? lda2 : ldb2;
    const uint32_t off = 64 * t + 8 * ch < K ? (uint32_t)lr * ld2 + 16u * (uint32_t)ch : kOOB;
    load_lds16_so(isa ? rA : rB,
                  __builtin_amdgcn_readfirstlane((isa ? la0 : lb0) + sg * STAGE + i * 1024),
                  off + (uint32_t)(8 * i) * ld2, (uint32_t)__builtin_amdgcn_readfirstlane(t * 128));
  };

#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
#pragma unroll
    for (int x = 0; x < LPW; ++x) issue1(s, s, x);

  // output chunk (i, j, h): row m_of(i), columns n_of(j, h) .. + 7
  auto m_of = [&](int i) { return m0 + 32 * (RB * wm + i) + fr; };
  auto n_of = [&](int j, int h) {
    return n0 + 32 * (JO * wn + j) + 16 * (KG == 2 ? kg : h) + 8 * hk;
  };
  const EpiViews V = epi_views<MODE, SP>(p, m0);
  EpiIn in[RB][JO][HN];
  // the epilogue's operands and the handed-over row sums, behind the first slabs
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < JO; ++j)
#pragma unroll
      for (int h = 0; h < HN; ++h) {
        epi_load_col<MODE>(V, n_of(j, h), true, in[i][j][h]);
        epi_load_row<MODE, SP>(p, V, m_of(i), n_of(j, h), true, 8, in[i][j][h]);
      }
  constexpr int PR = RPX ? 16 : 1;
  float prt[RB][PR];
  const __amdgpu_buffer_rsrc_t rq =
      make_rsrc(p.ss_in, RPX ? rec_bytes((int64_t)p.ss_parts * p.ss_ld * 4) : 0u);
  auto part = [&](int i, int q) {  // the half-waves take every other part
    const int m = m_of(i), qq = 2 * q + hk;
    return bload1f(rq, m < M && qq < p.ss_parts
                           ? ((uint32_t)qq * (uint32_t)p.ss_ld + (uint32_t)m) * 4u : kOOB);
  };
  if constexpr (RPX) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int q = 0; q < PR; ++q) prt[i][q] = part(i, q);
  }

  f32x16_t acc[RB][JN][AC];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int a = 0; a < AC; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][a][r] = 0.f;
  float ss[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) ss[i] = 0.f;
  const char* sA = smem + kg * SLAB + (32 * RB * wm + fr) * 128;
  auto brow = [&](int j) {
    return NB == 2 ? (j < JO ? 32 * (JO * wn + j) : BN / 2 + 32 * (JO * wn + j - JO))
                   : 32 * (JN * wn + j);
  };
  const char* sB = smem + kg * SLAB + (BM + fr) * 128;
  for (int s0 = 0; s0 < steps; s0 += NST) {
#pragma unroll
    for (int sg = 0; sg < NST; ++sg) {
      const int s = s0 + sg;
      if (s >= steps) break;
      wait_vmcnt<LPW*(NST - 2)>();  // this wave's loads of step s landed
      __syncthreads();              // everyone's, and step s - 1 is consumed
      // k-step ks + 1's fragments are read ahead of step ks's MFMAs
      bf16x8 af[2][RB], bf[2][JN];
      auto rd = [&](int ks, int b) {
        const int cpos = sg * STAGE + ((2 * ks + hk) ^ sw) * 16;
#pragma unroll
        for (int j = 0; j < JN; ++j) bf[b][j] = *(const bf16x8*)(sB + brow(j) * 128 + cpos);
#pragma unroll
        for (int i = 0; i < RB; ++i) af[b][i] = *(const bf16x8*)(sA + 32 * i * 128 + cpos);
      };
      rd(0, 0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int b = ks & 1;
        if (ks < 3) rd(ks + 1, b ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < LPW; ++x)
          if (x * 4 / LPW == ks) issue1(s + NST - 1, (sg + NST - 1) % NST, x);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
#pragma unroll
          for (int j = 0; j < JN; ++j)
            acc[i][j][ks % AC] = mfma32x32x16(bf[b][j], af[b][i], acc[i][j][ks % AC]);
          if (SUMX) ss[i] += sumsq8(af[b][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  wait_vmcnt<0>();

  // row factors
  float rf[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    rf[i] = 1.f;
    if constexpr (RPX) {
      float a = 0.f;
#pragma unroll
      for (int q = 0; q < PR; ++q) {
        asm volatile("" : "+v"(prt[i][q]));  // the adds stay behind the K loop
        a += prt[i][q];
      }
      for (int q = PR; 2 * q < p.ss_parts; ++q) a += part(i, q);
      rf[i] = rsqrtf(half_pair_sum(a) / (float)K + p.rownorm_eps);
    }
    if constexpr (SUMX) ss[i] = half_pair_sum(ss[i]);
  }
  if (AC == 2)
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][0][r] += acc[i][j][AC - 1][r];
  __syncthreads();  // the ring is free

  // this lane's chunks: 8 accumulators each, added over the K groups
  float v[RB][JN][HN][8];
  float* sum_ex = (float*)(smem + 8 * RB * JN * 2048);
  float* hand_ex = sum_ex + 8 * RB * 32;
  if constexpr (KG == 2) {
    f32x4_t* mine = (f32x4_t*)(smem + (kg * NW + w) * RB * JN * 2048);
    const f32x4_t* other = (const f32x4_t*)(smem + ((1 - kg) * NW + w) * RB * JN * 2048);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        const f32x16_t& a = acc[i][j][0];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // chunk 1 - kg goes to the other group
            o[e] = kg ? a[4 * u + e] : a[8 + 4 * u + e];
            v[i][j][0][4 * u + e] = kg ? a[8 + 4 * u + e] : a[4 * u + e];
          }
          mine[((i * JN + j) * 2 + u) * 64 + lane] = o;
        }
      }
    if constexpr (SUMX) {
#pragma unroll
      for (int i = 0; i < RB; ++i) sum_ex[((kg * NW + w) * RB + i) * 32 + fr] = ss[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4_t o = other[((i * JN + j) * 2 + u) * 64 + lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][j][0][4 * u + e] += o[e];
        }
      if constexpr (SUMX) ss[i] += sum_ex[(((1 - kg) * NW + w) * RB + i) * 32 + fr];
    }
  } else {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int h = 0; h < HN; ++h)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][j][h][e] = acc[i][j][0][(8 * h + e) & 15];
  }
  if constexpr (SUMX) {
#pragma unroll
    for (int i = 0; i < RB; ++i) rf[i] = rsqrtf(ss[i] / (float)K + p.rownorm_eps);
  }
  // columns 4 hk .. + 3 and 8 + 4 hk .. of a chunk pair -> 8 hk .. + 7
  auto join = [](float* x) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[e]),
                                                      __float_as_uint(x[4 + e]), false, false);
      x[e] = __uint_as_float(s[0]);
      x[4 + e] = __uint_as_float(s[1]);
    }
  };
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = m_of(i);
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < JO; ++j)
#pragma unroll
      for (int h = 0; h < HN; ++h) {
        float* a = v[i][j][h];
        float* u = v[i][NB == 2 ? j + JO : j][h];
        join(a);
        if (NB == 2) join(u);
        const int n = n_of(j, h);
        if (m < M && n < N) {
          float xo[8];
          epi_store<MODE, false, SP>(p, m, n, true, 8, a, u, rf[i], in[i][j][h], HOX, xo);
          if constexpr (HOX) {
#pragma unroll
            for (int e = 0; e < 8; ++e) q += xo[e] * xo[e];
          }
        }
      }
    if constexpr (HOX) {
      // the row's sum over the wave's 64 columns (JN = 2), over both groups
      static_assert(!HOX || (JN == 2 && RB == 1), "one 64-column block per wave");
      q = half_pair_sum(q);
      if (KG == 2) {
        hand_ex[(kg * NW + w) * 32 + fr] = q;
        __syncthreads();
        q += hand_ex[((1 - kg) * NW + w) * 32 + fr];
      }
      const int blk = (n0 + 64 * wn) >> 6;
      if (kg == 0 && hk == 0 && m < M && 64 * blk < N)
        p.ss_out[(int64_t)blk * p.ss_ld + m] = q;
    }
  }
}

static bool mid_ok(const GemmArgs& d) {
  if (d.b_fp8 || d.a8_out || d.ln_csum || a_grouped(d) || d.split_k > 1 || d.c_frag ||
      d.gu_out || !epi_vec_ok(d) || d.n % 8 || d.n < 64 || d.m <= 64 || d.m >= (1 << 24) ||
      d.n >= (1 << 24) || d.lda >= ((int64_t)1 << 22) ||
      d.ldb >= ((int64_t)1 << 22))
    return false;
  return d.mode == FVX_GEMM_PLAIN || d.mode == FVX_GEMM_GEGLU || d.mode == FVX_GEMM_QKV_ROPE;
}

// Where one round of a configuration's tiles (at most one per CU) serves d:
//   2: 128 x 128 (GEGLU: 64 columns of each weight), 8 waves on one tile, once
//      the 64 x 128 tiles of gemm_tile_kernel number more than 256 (two rounds or
//      two workgroups per CU there).  Measured (us, tile kernel -> this): SigLIP
//      Q|K|V 768 x 3456 x 1152 14.4 -> 11.8, fc1 768 x 4304 x 1152 15.9 -> 13.7;
//      prefix Q|K|V 816 x 2560 x 2048 23.3 -> 18.6; O 1400 x 2048 x 2048 22.4 ->
//      18.5; expert gate/up 408 x 2 x 4096 x 1024 15.1 -> 12.3.  Past one round
//      the gain goes (1536 x 4304 x 1152 23.1 -> 24.9).
//   1: 64 x 128, two K groups, for the longer epilogues (Q|K|V, row sums handed
//      on): prefix O 816 x 2048 x 2048 16.1 -> 14.3, expert Q|K|V 408 x 2560 x
//      1024 12.6 -> 9.6.  Not for the plain one: 1536 x 1152 x 1152 10.1 -> 10.4,
//      1632 x 1024 x 4096 21.4 -> 23.0.
//   0: 64 x 64, two K groups: expert O 408 x 1024 x 2048 9.6 -> 8.4, down 408 x
//      1024 x 4096 15.2 -> 14.1, SigLIP o 768 x 1152 x 1152 7.4 -> 7.2, fc2 768 x
//      1152 x 4304 22.9 -> 22.6 (68.7 MB fetched for 16.5 MB of operands: an XCD's
//      27 tiles cover all 12 tile rows, so all of A passes through each of 8 L2s).
// From K = 8192 on the wide kernel's K ranges are faster (prefix down 816 x 2048 x
// 16384: 78 us against about 84).
int plan_mid(const GemmArgs& d) {
  if (!mid_ok(d) || d.k >= 8192) return -1;
  const int64_t cus = device_cus();
  const bool gg = d.mode == FVX_GEMM_GEGLU;
  auto tiles = [&](int bm, int bn) {
    return ((d.m + bm - 1) / bm) * ((d.n + bn - 1) / bn);
  };
  const int64_t tile_kernel = tiles(64, gg ? 64 : 128);
  if (tile_kernel > 256) return tiles(128, gg ? 64 : 128) <= cus ? 2 : -1;
  if (gg) return -1;
  if (tiles(64, 128) >= 128 || d.ss_out)  // (ss_out: whole 64-column blocks per wave)
    return (d.mode == FVX_GEMM_QKV_ROPE || d.ss_out) && tiles(64, 128) <= cus ? 1 : -1;
  return tiles(64, 64) <= cus ? 0 : -1;
}

template <int MODE, int RB, int JN, int WGM, int WGN, int KG, int NST>
static void launch_mid(const GemmArgs& d, hipStream_t s) {
  typedef MidCfg<RB, JN, WGM, WGN, KG, NST> C;
  const int nb = MODE == FVX_GEMM_GEGLU ? 2 : 1;
  const int m_tiles = (int)((d.m + C::BM - 1) / C::BM);
  const int n_tiles = (int)((d.n + C::BN / nb - 1) / (C::BN / nb));
  const dim3 grid((unsigned)(m_tiles * n_tiles)), blk(512);
  const int xf = (d.rownorm ? (d.ss_in ? 1 : 2) : 0) | (d.ss_out ? 4 : 0) |
                 (plain_epilogue_ok(d) ? 8 : 0);
#define FVX_MID(XF_)                                                                      \
  case XF_:                                                                               \
    hipLaunchKernelGGL((gemm_mid_kernel<MODE, RB, JN, WGM, WGN, KG, NST, XF_>), grid, blk, 0, \
                       s, d, m_tiles, n_tiles);                                           \
    break
  switch (xf) {
    FVX_MID(0);
    FVX_MID(1);
    FVX_MID(2);
  }
  if constexpr (MODE == FVX_GEMM_PLAIN) {
    switch (xf) {
      FVX_MID(8);
      FVX_MID(9);
      FVX_MID(10);
    }
    if constexpr (JN == 2) {  // a wave's columns are one 64-column block
      switch (xf) {
        FVX_MID(4);
        FVX_MID(5);
        FVX_MID(6);
        FVX_MID(12);
        FVX_MID(13);
        FVX_MID(14);
      }
    }
  }
#undef FVX_MID
}

int run_mid(const GemmArgs& d, int cfg, hipStream_t s) {
  if (d.mode == FVX_GEMM_GEGLU) {
    launch_mid<FVX_GEMM_GEGLU, 1, 2, 4, 2, 1, 4>(d, s);
  } else if (d.mode == FVX_GEMM_QKV_ROPE) {
    if (cfg == 0) launch_mid<FVX_GEMM_QKV_ROPE, 1, 1, 2, 2, 2, 4>(d, s);
    else if (cfg == 1) launch_mid<FVX_GEMM_QKV_ROPE, 1, 2, 2, 2, 2, 3>(d, s);
    else launch_mid<FVX_GEMM_QKV_ROPE, 1, 2, 4, 2, 1, 4>(d, s);
  } else {
    if (cfg == 0) launch_mid<FVX_GEMM_PLAIN, 1, 1, 2, 2, 2, 4>(d, s);
    else if (cfg == 1) launch_mid<FVX_GEMM_PLAIN, 1, 2, 2, 2, 2, 3>(d, s);
    else launch_mid<FVX_GEMM_PLAIN, 1, 2, 4, 2, 1, 4>(d, s);
  }
  return launch_status("gemm(mid)");
}

}  // namespace fvx
