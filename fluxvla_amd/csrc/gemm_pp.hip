// gemm_pp_kernel: bf16 MFMA GEMMs of a few hundred rows and more (bf16 weights,
// or e4m3 weights made bf16 on the way from the LDS to the matrix cores), 8
// waves per workgroup in two groups that take turns on the matrix cores.
//
//   acc[m][n] = sum_k A[m][k] * B[n][k]      A: activations, B: nn.Linear weight
//
// A workgroup owns a BM x BN tile, WGM x WGN waves of RB x JN blocks of 32 x 32
// (v_mfma_f32_32x32x16_bf16, the weight rows as the A operand, so that a lane
// ends with ONE output row and runs of 4 columns of it).  K moves in 64-wide
// slabs through an NST-deep LDS ring filled by LDS DMA.  Waves w and w + 4
// share a SIMD; waves 0-3 and 4-7 run half a phase apart: while one group reads
// its next fragments from the LDS and issues its share of the DMA, the other
// one's MFMAs keep the SIMD's matrix core busy, and a barrier swaps them.  A
// phase is KPH k-steps of 16, chosen so that its MFMAs (8 or more) cover the
// other group's LDS reads.  Slab t + NST - 1 goes into the stage of slab t - 1
// once both groups have read that; before a wave leaves slab t it waits for its
// own loads of slab t + 1 only (s_waitcnt vmcnt counts the rest).
//
// The epilogue needs no LDS: v_permlane32_swap joins the two half-waves' runs
// of 4 columns to chunks of 8, the row's RMS factor is one value per lane, and
// every operand and result moves as 16 bytes per lane.
#include "gemm_epilogue.h"

namespace fvx {

__device__ __forceinline__ void pp_bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int RB, int JN, int WGM, int WGN, int NST, bool F8>
struct PpCfg {
  static constexpr int BM = 32 * RB * WGM, BN = 32 * JN * WGN;
  static constexpr int STAGE = BM * 128 + BN * (F8 ? 64 : 128);
  // DMA loads per wave and slab (8 rows of 128 bytes or 16 of 64 each)
  static constexpr int LA = BM / 64, LB = BN / (F8 ? 128 : 64), LPW = LA + LB;
  // k-steps per phase: at least 8 MFMAs (or the whole slab)
  static constexpr int KPH = RB * JN >= 8 ? 1 : (RB * JN >= 4 ? 2 : 4), PH = 4 / KPH;
  // phases over which a slab's loads are issued: two stages leave them only
  // until the end of the slab to land, so they go into its first half
  static constexpr int LPH = NST == 2 && PH > 1 ? PH / 2 : PH;
  static_assert(WGM * WGN == 8 && BM % 64 == 0 && BN % (F8 ? 128 : 64) == 0, "whole loads");
  static_assert(NST * STAGE <= 160 * 1024, "LDS");
};

// XF bit 0: the row sums of squares are handed over (ss_in); bit 1: they are
// taken in the K loop; bit 2: the output's are handed on (ss_out).
// F8 (W8A16): e4m3 weights; a lane's 32 weight bytes of a slab become the four
// bf16 fragments of k = 32 hk + 8 c + 0..7, whose A fragments are chunks 4 hk + c.
template <int MODE, int RB, int JN, int WGM, int WGN, int NST, int XF, bool F8>
__global__ __launch_bounds__(512, 1) void gemm_pp_kernel(GemmArgs p, int m_tiles, int n_tiles,
                                                         int row_block) {
  typedef PpCfg<RB, JN, WGM, WGN, NST, F8> C;
  constexpr int NB = MODE == FVX_GEMM_GEGLU ? 2 : 1, JO = JN / NB;  // output blocks
  constexpr int LA = C::LA, LB = C::LB, LPW = C::LPW, KPH = C::KPH, PH = C::PH;
  constexpr int STAGE = C::STAGE, BM = C::BM, BN = C::BN;
  constexpr bool RPX = (XF & 1) != 0, SUMX = (XF & 2) != 0, HOX = (XF & 4) != 0;
  constexpr bool SP = MODE == FVX_GEMM_PLAIN;
  __shared__ __align__(16) char smem[NST * STAGE];
  warm_kernargs<sizeof(GemmArgs) + 16>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;
  const int wm = wave / WGN, wn = wave % WGN;
  const int fr = lane & 31, hk = lane >> 5, sw = (lane >> 1) & 7;
  int mt, nt;
  tile_order(xcd_remap(blockIdx.x, m_tiles * n_tiles), m_tiles, n_tiles, row_block, mt, nt);
  const int M = (int)p.m, N = (int)p.n, K = (int)p.k, nk = (K + 63) / 64;
  const int m0 = mt * BM, n0 = nt * (BN / NB);

  // DMA: this wave's 8 LA rows of A and 8 LB rows of B, 8 rows of 128 bytes
  // per load; lane l fetches row l / 8, chunk (l % 8) ^ ((row >> 1) & 7) of 16
  // bytes, so the fragment reads are conflict-free.  Rows past the operand are
  // outside the view, chunks past K get an offset outside it: zeros.
  const int lr = lane >> 3, lc = lane & 7;
  // (GEGLU: the gate rows, then the up rows; F8: 16 rows of 64 bytes per load,
  // lane l row l / 4, chunk (l % 4) ^ ((row >> 2) & 3))
  const int ra = m0 + 8 * LA * wave, brow0 = (F8 ? 16 : 8) * LB * wave;
  const bool up = NB == 2 && brow0 >= BN / 2;
  const int rb = n0 + (up ? brow0 - BN / 2 : brow0);
  auto rows_in = [](int left, int most) { return left <= 0 ? 0 : (left < most ? left : most); };
  const uint32_t lda2 = (uint32_t)p.lda * 2, ldb2 = (uint32_t)p.ldb * (F8 ? 1 : 2);
  const i32x4_t rA = make_rsrc4((const bf16_t*)p.a + (int64_t)ra * p.lda,
                                (uint32_t)rows_in(M - ra, 8 * LA) * lda2);
  const i32x4_t rB = make_rsrc4((const char*)(up ? p.b2 : p.b) + (int64_t)rb * ldb2,
                                (uint32_t)rows_in(N - rb, (F8 ? 16 : 8) * LB) * ldb2);
  // load i: chunk parity (first 8-row unit + i) & 1
  const int c0 = lc ^ (lr >> 1), pa = (LA * wave) & 1, pb = (LB * wave) & 1;
  const int ca0 = c0 ^ (4 * pa), cb0 = c0 ^ (4 * pb);
  const uint32_t la0 = __builtin_amdgcn_readfirstlane(lds_addr(smem) + wave * LA * 1024);
  const uint32_t lb0 = __builtin_amdgcn_readfirstlane(lds_addr(smem) + BM * 128 + wave * LB * 1024);
  // load x (A's LA, then B's LB) of slab t into stage s
  auto issue1 = [&](int t, int s, int x) {
    const bool isa = x < LA;
    const int i = isa ? x : x - LA;
    if (F8 && !isa) {
      const int r = lane >> 2, c = (lane & 3) ^ ((lane >> 4) & 3);
      const uint32_t off = 64 * t < K ? (uint32_t)r * ldb2 + 16u * (uint32_t)c : kOOB;
      load_lds16_so(rB, __builtin_amdgcn_readfirstlane(lb0 + s * STAGE + i * 1024),
                    off + (uint32_t)(16 * i) * ldb2,
                    (uint32_t)__builtin_amdgcn_readfirstlane(t * 64));
      return;
    }
    const int ch = (isa ? ca0 : cb0) ^ (4 * (i & 1));
    const uint32_t ld2 = isa ? lda2 : ldb2;
    const uint32_t off = 64 * t + 8 * ch < K ? (uint32_t)lr * ld2 + 16u * (uint32_t)ch : kOOB;
    load_lds16_so(isa ? rA : rB,
                  __builtin_amdgcn_readfirstlane((isa ? la0 : lb0) + s * STAGE + i * 1024),
                  off + (uint32_t)(8 * i) * ld2, (uint32_t)__builtin_amdgcn_readfirstlane(t * 128));
  };

  f32x16_t acc[RB][JN];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
#pragma unroll
    for (int x = 0; x < LPW; ++x) issue1(s, s, x);

  // each lane's row factors (row 32 i + fr of the wave)
  float rf[RB], ss[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    rf[i] = 1.f;
    ss[i] = 0.f;
  }
  if constexpr (RPX) {
    // the handed-over sums: the half-waves take every other part
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(p.ss_in, rec_bytes((int64_t)p.ss_parts * p.ss_ld * 4));
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int m = m0 + 32 * (RB * wm + i) + fr;
      float a = 0.f;
      for (int q0 = 0; q0 < p.ss_parts; q0 += 32) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int q = q0 + 2 * u + hk;
          v[u] = bload1f(rq, m < M && q < p.ss_parts
                                 ? ((uint32_t)q * (uint32_t)p.ss_ld + (uint32_t)m) * 4u : kOOB);
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) a += v[u];
      }
      rf[i] = rsqrtf(half_pair_sum(a) / (float)K + p.rownorm_eps);
    }
  }

  const char* sA = smem + (32 * RB * wm + fr) * 128;
  // LDS row of B block j of this wave (GEGLU: gate blocks, then up)
  auto brow = [&](int j) {
    return NB == 2 ? (j < JO ? 32 * (JO * wn + j) : BN / 2 + 32 * (JO * wn + j - JO))
                   : 32 * (JN * wn + j);
  };
  const char* sB = smem + BM * 128 + fr * (F8 ? 64 : 128);
  const int sw8 = (fr >> 2) & 3;
  wait_vmcnt<(NST - 2) * LPW>();
  pp_bar();
  if (grp) pp_bar();  // half a phase behind the first group
  int st = 0, sn = NST - 1;
  for (int t = 0; t < nk; ++t) {
    bf16x8 b8[F8 ? JN : 1];  // F8: 16 weight bytes, two k-steps' worth
#pragma unroll
    for (int ph = 0; ph < PH; ++ph) {
      bf16x8 af[KPH][RB], bf[KPH][F8 ? 1 : JN], c8[F8 ? KPH : 1][F8 ? JN : 1];
#pragma unroll
      for (int kk = 0; kk < KPH; ++kk) {
        const int ks = ph * KPH + kk;
        const int cpos = st * STAGE + ((F8 ? 4 * hk + ks : 2 * ks + hk) ^ sw) * 16;
        if constexpr (F8) {
          if (ks % 2 == 0)
#pragma unroll
            for (int j = 0; j < JN; ++j)
              b8[j] = *(const bf16x8*)(sB + brow(j) * 64 + st * STAGE +
                                       (((2 * hk + ks / 2) ^ sw8) * 16));
#pragma unroll
          for (int j = 0; j < JN; ++j) c8[kk][j] = b8[j];
        } else {
#pragma unroll
          for (int j = 0; j < JN; ++j) bf[kk][j] = *(const bf16x8*)(sB + brow(j) * 128 + cpos);
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) af[kk][i] = *(const bf16x8*)(sA + 32 * i * 128 + cpos);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < LPW; ++x)
        if (x * C::LPH / LPW == ph) issue1(t + NST - 1, sn, x);
      // the reads are complete before the barrier that lets the others on
      __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
      if (ph == PH - 1 && grp) wait_vmcnt<(NST - 2) * LPW>();
      __builtin_amdgcn_sched_barrier(0);
      pp_bar();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < KPH; ++kk) {
#pragma unroll
        for (int j = 0; j < JN; ++j) {
          bf16x8 b;
          if constexpr (F8) {
            const int hf = 2 * ((ph * KPH + kk) & 1);  // the bytes' half
            b = e4m3x8_to_bf16(c8[kk][j].w[hf], c8[kk][j].w[hf + 1]);
          } else {
            b = bf[kk][j];
          }
#pragma unroll
          for (int i = 0; i < RB; ++i) acc[i][j] = mfma32x32x16(b, af[kk][i], acc[i][j]);
        }
        if (SUMX)
#pragma unroll
          for (int i = 0; i < RB; ++i) ss[i] += sumsq8(af[kk][i]);
      }
      __builtin_amdgcn_s_setprio(0);
      if (ph == PH - 1 && !grp) wait_vmcnt<(NST - 2) * LPW>();
      __builtin_amdgcn_sched_barrier(0);
      pp_bar();
      __builtin_amdgcn_sched_barrier(0);
    }
    st = st + 1 == NST ? 0 : st + 1;
    sn = sn + 1 == NST ? 0 : sn + 1;
  }
  if (!grp) pp_bar();
  wait_vmcnt<0>();
  if constexpr (SUMX) {
#pragma unroll
    for (int i = 0; i < RB; ++i) rf[i] = rsqrtf(half_pair_sum(ss[i]) / (float)K + p.rownorm_eps);
  }

  // Epilogue: block (i, j) of lane (fr, hk) holds row 32 i + fr, columns 8 (r
  // >> 2) + 4 hk + (r & 3) of 32 j; chunk h of it, columns 16 h + 8 hk .. + 7,
  // after the half-waves swap.  N % 8 == 0 and 16-byte operands (the host
  // checks): every chunk with columns left moves whole.
  const EpiViews V = epi_views<MODE, SP>(p, m0);
  const __amdgpu_buffer_rsrc_t rs0 = make_rsrc(p.b_scale, F8 ? rec_bytes(p.n * 4) : 0u);
  const __amdgpu_buffer_rsrc_t rs1 =
      make_rsrc(p.b2_scale, F8 && NB == 2 ? rec_bytes(p.n * 4) : 0u);
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = m0 + 32 * (RB * wm + i) + fr;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < JO; ++j) {
      const int nb = n0 + 32 * (JO * wn + j) + 8 * hk;
      EpiIn in[2];
      float ws[2][NB][8];  // F8: the columns' weight scales
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        epi_load_col<MODE>(V, nb + 16 * h, true, in[h]);
        epi_load_row<MODE, SP>(p, V, m, nb + 16 * h, true, 8, in[h]);
        if constexpr (F8) {
          bl_f8(rs0, (uint32_t)(nb + 16 * h) * 4u, true, ws[h][0]);
          if constexpr (NB == 2) bl_f8(rs1, (uint32_t)(nb + 16 * h) * 4u, true, ws[h][NB - 1]);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = nb + 16 * h;
        float v[NB][8];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const auto s = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(acc[i][j + b * JO][8 * h + e]),
                __float_as_uint(acc[i][j + b * JO][8 * h + 4 + e]), false, false);
            v[b][e] = __uint_as_float(s[0]);
            v[b][4 + e] = __uint_as_float(s[1]);
          }
          if constexpr (F8) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[b][e] *= ws[h][b][e];
          }
        }
        if (m < M && n < N) {
          float xo[8];
          epi_store<MODE, false, SP>(p, m, n, true, 8, v[0], v[NB - 1], rf[i], in[h], HOX, xo);
          if constexpr (HOX) {
#pragma unroll
            for (int e = 0; e < 8; ++e) q += xo[e] * xo[e];
          }
        }
      }
      if constexpr (HOX) {
        // the row's sum over a 64-column block (two 32-column blocks)
        if (j & 1) {
          const float t = half_pair_sum(q);
          const int blk = (n0 + 32 * (JN * wn + j - 1)) >> 6;
          if (hk == 0 && m < M && 64 * blk < N) p.ss_out[(int64_t)blk * p.ss_ld + m] = t;
          q = 0.f;
        }
      }
    }
  }
}

// Tile configurations and what a tile costs on a full chip (us, measured on
// MI355X at K = 1152 ... 16384): `slab` per 64-wide K slab plus `fixed`
// (prologue, first loads, epilogue), with bf16 and with e4m3 weights (half the
// weight bytes, so three stages of 256 x 256 fit the LDS; 0: no such build --
// a wave loads its rows of e4m3 16 at a time, and 256 x 320 and 192 columns are
// no multiple of 128, while 128 x 256 moves more of the bf16 side).
struct PpTile {
  int bm, bn;
  float slab, fixed, slab8, fixed8;
};
static const PpTile kPpTile[] = {{256, 256, 1.6f, 8.f, 1.45f, 10.f},
                                 {256, 320, 2.1f, 5.f, 0.f, 0.f},
                                 {256, 192, 1.4f, 4.f, 0.f, 0.f},
                                 {256, 128, 0.9f, 8.f, 0.88f, 9.f},
                                 {128, 256, 0.9f, 9.f, 0.f, 0.f}};
constexpr int kPpCfgs = 5;

static bool pp_ok(const GemmArgs& d) {
  if ((d.b_fp8 && d.fp8_act) || d.a8_out || d.ln_csum || a_grouped(d) || d.split_k > 1 ||
      d.c_frag || d.gu_out || !epi_vec_ok(d) || d.n % 8 || d.k < 64 || d.m <= 64 ||
      d.n >= (1 << 24) || d.k >= ((int64_t)1 << 24) || d.lda >= ((int64_t)1 << 22) ||
      d.ldb >= ((int64_t)1 << 22))
    return false;
  if (d.mode == FVX_GEMM_GEGLU) return d.b_fp8 != 0;
  return d.mode == FVX_GEMM_QKV_ROPE ? !d.ss_out : plain_epilogue_ok(d);
}

// The configuration whose rounds of tiles over the CUs cost least, or -1 where
// the 64 x 128 tiles of gemm_tile_kernel (about 1.6 ns per tile and slab, two
// workgroups per CU) are expected to be faster: with few rows the larger tiles
// leave CUs idle.  Measured (us, this kernel / the tile or wide kernel): prefix
// Q|K|V 6528 x 2560 x 2048 75 / 102 (256 x 320: one round of 208 tiles), O 6528
// x 2048 x 2048 60 / 71, down 6528 x 2048 x 16384 400 / 403; SigLIP Q|K|V 6144 x
// 3456 x 1152 62 / 74, fc2 6144 x 1152 x 4304 75 / 115, 24576 rows 279 / 456;
// 1536 x 4304 x 1152 24 / 29, but 768 x 3456 x 1152 20 / 15 and 1632 x 1024 x
// 2048 30 / 16.  With e4m3 weights: gate|up 22144 x 2 x 16384 x 2048 2596 / 2822,
// 6528 rows 760 / 853, 816 109 / 130, 300 60 / 74; O 22144 x 2048 x 2048 198 /
// 262, 6528 rows 59 / 85; Q|K|V 22144 x 2560 x 2048 247 / 316; down 22144 x 2048
// x 16384 1247 / 1327, 4152 rows 298 / 387; but Q|K|V 6528 rows 117 / 97 (260
// tiles: a second round of four), down 816 rows 221 / 74 (split K) and the
// expert's gate|up 400 x 2 x 4096 x 1024 29 / 15.  bf16 gate|up stays with the
// wide kernel, which moves 128 x 128 per wave: 6528 rows 754 / 750, 816 118 / 115.
// Below 8 slabs the tiles' epilogue, one per CU and not behind another workgroup's K
// loop, is most of the time, and CUs without a tile are lost to it: at least 176 of 256
// must have one (us, this / tile kernel: 140 to 169 tiles 5582 x 1280 x 80 15.7 / 14.4, 2609
// x 2560 x 136 17.1 / 16.1, 1641 x 4096 x 432 21.3 / 19.7, 6961 x 1024 x 272 18.8 / 17.2;
// 184 to 234 tiles 1978 x 4304 x 136 16.6 / 18.4, 4653 x 2048 x 72 16.7 / 17.9, 5309 x 3456
// x 416 34.4 / 42.0; but 195 tiles 3801 x 4096 x 112 26.9 / 24.2).
int plan_pp(const GemmArgs& d) {
  if (!pp_ok(d)) return -1;
  const int cus = device_cus();
  const float slabs = (float)((d.k + 63) / 64);
  const bool gg = d.mode == FVX_GEMM_GEGLU;
  const int nb = gg ? 2 : 1;
  const int64_t old_tiles = ((d.m + 63) / 64) * ((d.n * nb + 127) / 128);
  float best = (1.6e-3f * (float)old_tiles * slabs + 5.f) * 0.97f;
  int cfg = -1;
  for (int c = 0; c < kPpCfgs; ++c) {
    const PpTile& t = kPpTile[c];
    // row sums are handed on per 64 columns: whole blocks per wave; GEGLU is
    // built for 256 x 2 x 128 only
    if ((d.ss_out && (c == 1 || c == 2)) || (gg && c) || (d.b_fp8 && t.slab8 == 0.f)) continue;
    const int64_t tiles = ((d.m + t.bm - 1) / t.bm) * ((d.n * nb + t.bn - 1) / t.bn);
    if (slabs < 8.f && 16 * tiles < 11 * cus) continue;
    const float us = (float)((tiles + cus - 1) / cus) *
                     (d.b_fp8 ? slabs * t.slab8 + t.fixed8 : slabs * t.slab + t.fixed);
    if (us < best) {
      best = us;
      cfg = c;
    }
  }
  return cfg;
}

template <int MODE, int RB, int JN, int WGM, int WGN, int NST, bool F8>
static void launch_pp(const GemmArgs& d, int row_block, hipStream_t s) {
  typedef PpCfg<RB, JN, WGM, WGN, NST, F8> C;
  const int bn = C::BN / (MODE == FVX_GEMM_GEGLU ? 2 : 1);
  const int m_tiles = (int)((d.m + C::BM - 1) / C::BM), n_tiles = (int)((d.n + bn - 1) / bn);
  const dim3 grid((unsigned)(m_tiles * n_tiles)), blk(512);
  const int xf = d.rownorm ? (d.ss_in ? 1 : 2) : 0;
#define FVX_PP(XF_)                                                                          \
  hipLaunchKernelGGL((gemm_pp_kernel<MODE, RB, JN, WGM, WGN, NST, XF_, F8>), grid, blk, 0, s, \
                     d, m_tiles, n_tiles, row_block)
  if constexpr (MODE == FVX_GEMM_PLAIN && JN % 2 == 0) {
    if (d.ss_out) {
      if (xf == 1) FVX_PP(5); else if (xf == 2) FVX_PP(6); else FVX_PP(4);
      return;
    }
  }
  if (xf == 1) FVX_PP(1); else if (xf == 2) FVX_PP(2); else FVX_PP(0);
#undef FVX_PP
}

int run_pp(const GemmArgs& d, int cfg, hipStream_t s) {
  // the tile order's blocks: 2048 rows
  const int rows = 2048 / kPpTile[cfg].bm;
#define FVX_PP8(MODE)                                                   \
  if (cfg == 0) launch_pp<MODE, 2, 4, 4, 2, 3, true>(d, rows, s);       \
  else launch_pp<MODE, 2, 2, 4, 2, 3, true>(d, rows, s)
#define FVX_PPL(MODE)                                                   \
  switch (cfg) {                                                        \
    case 0: launch_pp<MODE, 2, 4, 4, 2, 2, false>(d, rows, s); break;   \
    case 1: launch_pp<MODE, 2, 5, 4, 2, 2, false>(d, rows, s); break;   \
    case 2: launch_pp<MODE, 2, 3, 4, 2, 2, false>(d, rows, s); break;   \
    case 3: launch_pp<MODE, 2, 2, 4, 2, 3, false>(d, rows, s); break;   \
    default: launch_pp<MODE, 2, 2, 2, 4, 3, false>(d, rows, s); break;  \
  }
  if (d.mode == FVX_GEMM_GEGLU) {
    launch_pp<FVX_GEMM_GEGLU, 2, 4, 4, 2, 3, true>(d, rows, s);
  } else if (d.mode == FVX_GEMM_QKV_ROPE) {
    if (d.b_fp8) {
      FVX_PP8(FVX_GEMM_QKV_ROPE);
    } else {
      FVX_PPL(FVX_GEMM_QKV_ROPE)
    }
  } else if (d.b_fp8) {
    FVX_PP8(FVX_GEMM_PLAIN);
  } else {
    FVX_PPL(FVX_GEMM_PLAIN)
  }
#undef FVX_PPL
#undef FVX_PP8
  return launch_status("gemm(pp)");
}

}  // namespace fvx
