// attn_encoder_kernel: unmasked attention with one query head per problem and
// row-major values (SigLIP: 16 heads of dim 72 over 256 patches per image).
//
// A workgroup is 4 waves of RG x 16 query rows and walks the keys in tiles of 64:
//
//   S^T(64 keys x 16 rows) = K(64 x d) . Q^T(d x 16)
//   O^T(d x 16 rows)      += V^T(d x 64) . P^T(64 x 16)
//
// on v_mfma_f32_16x16x32_bf16: both leave a lane with values of ONE query row
// (lane % 16), so that the running maximum, its rescaling and the division are
// per lane, the probabilities are P^T's operand as they are, and a lane stores 4
// consecutive dims.  With every key visible a score costs a maximum, an fma, an
// exp2 and an add; the sums of a row's 4 lanes meet once, after the last tile.
//
// At these head dims the vector ALU and the LDS bound it, not the matrix cores
// (64 keys x 16 rows: 22 MFMAs, 22 KB of fragments): RG = 2 reads every K and V
// fragment once for two row groups.  K and V pass through registers into a ring
// of two tiles (one barrier per tile, the loads of tile t + 2 behind tile t);
// V is turned in pairs of keys, so that the transposed tile is written as words.
#include <math.h>

#include "capi_util.h"
#include "common.h"

namespace fvx {

constexpr int kEncKT = 64;                        // keys per tile
constexpr int kEncLDK = 96 + 8, kEncLDV = 64 + 8;  // LDS row lengths (elements)
constexpr int kEncND = 5, kEncNS = 3;             // 16-dim blocks of O, 32-dim steps of QK^T
constexpr int kEncK = kEncKT * kEncLDK, kEncV = 16 * kEncND * kEncLDV;

// the values of lanes l and l ^ 16 (half_pair: l and l ^ 32)
__device__ __forceinline__ void enc_pair16(float v, float& a, float& b) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  a = __uint_as_float(s[0]);
  b = __uint_as_float(s[1]);
}

template <int RG>
__global__ __launch_bounds__(256) void attn_encoder_kernel(fvx_attn_desc p, int n_row_blocks,
                                                           uint32_t chunk_magic) {
  __shared__ __align__(16) bf16_t tiles[2 * (kEncK + kEncV)];
  warm_kernargs<sizeof(fvx_attn_desc) + 8>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4;
  // the row blocks of a problem, and neighbouring heads, on one XCD
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int z = bid / n_row_blocks, rb = bid - z * n_row_blocks;
  const int HD = (int)p.head_dim, sq = (int)p.sq, sk = (int)p.sk;
  const int64_t zb = (uint32_t)z / (uint32_t)p.zdiv, zh = (uint32_t)z % (uint32_t)p.zdiv;
  const bf16_t* Q = (const bf16_t*)p.q + zb * p.q_zs1 + zh * p.q_zs2;
  const bf16_t* K = (const bf16_t*)p.k + zb * p.k_zs1 + zh * p.k_zs2;
  const bf16_t* V = (const bf16_t*)p.v + zb * p.v_zs1 + zh * p.v_zs2;
  bf16_t* O = (bf16_t*)p.o + zb * p.o_zs1 + zh * p.o_zs2;

  // This thread's chunks of a tile.  K: 16 bytes of key i / (HD / 8) for i = tid,
  // tid + 256, ..; V: 16 bytes of both keys of pair i % 32, dims 8 (i / 32) .. + 7.
  constexpr int CK = 3, CV = 2;
  const int kch = HD / 8;
  const uint32_t kts2 = (uint32_t)p.k_tok_stride * 2u, vts2 = (uint32_t)p.v_tok_stride * 2u;
  const auto rq = make_rsrc(Q, (uint32_t)(((p.sq - 1) * p.q_tok_stride + HD) * 2));
  const auto rk = make_rsrc(K, (uint32_t)sk * kts2);
  const auto rv = make_rsrc(V, (uint32_t)sk * vts2);
  uint32_t koff[CK], voff[CV];
  int kl[CK], vl[CV];
  bool kin[CK], vin[CV];
#pragma unroll
  for (int c = 0; c < CK; ++c) {
    const int i = tid + 256 * c;
    kin[c] = i < kEncKT * kch;
    const int kr = (int)(((uint32_t)i * chunk_magic) >> 16), kc = i - kr * kch;
    koff[c] = (uint32_t)kr * kts2 + (uint32_t)kc * 16u;
    kl[c] = kr * kEncLDK + kc * 8;
  }
#pragma unroll
  for (int c = 0; c < CV; ++c) {
    const int i = tid + 256 * c, pr = i & 31, dc = i >> 5;
    vin[c] = dc < kch;
    voff[c] = (uint32_t)(2 * pr) * vts2 + (uint32_t)dc * 16u;
    vl[c] = 8 * dc * kEncLDV + 2 * pr;
  }
  bf16x8 rgk[CK], rgv[CV][2];
  auto load = [&](int t) {
    const uint32_t kb = (uint32_t)(t * kEncKT) * kts2, vb = (uint32_t)(t * kEncKT) * vts2;
#pragma unroll
    for (int c = 0; c < CK; ++c) rgk[c] = bload8(rk, kin[c] ? kb + koff[c] : kOOB);
#pragma unroll
    for (int c = 0; c < CV; ++c) {
      rgv[c][0] = bload8(rv, vin[c] ? vb + voff[c] : kOOB);
      rgv[c][1] = bload8(rv, vin[c] ? vb + voff[c] + vts2 : kOOB);
    }
  };
  auto store = [&](int b) {
    bf16_t* sK = tiles + b * (kEncK + kEncV);
    bf16_t* sV = sK + kEncK;
#pragma unroll
    for (int c = 0; c < CK; ++c)
      if (kin[c]) st8(&sK[kl[c]], rgk[c]);
#pragma unroll
    for (int c = 0; c < CV; ++c)
      if (vin[c]) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t a = rgv[c][0].w[w], d = rgv[c][1].w[w];
          *(uint32_t*)&sV[vl[c] + 2 * w * kEncLDV] = __builtin_amdgcn_perm(d, a, 0x05040100u);
          *(uint32_t*)&sV[vl[c] + (2 * w + 1) * kEncLDV] =
              __builtin_amdgcn_perm(d, a, 0x07060302u);
        }
      }
  };
  load(0);

  bf16x8 qf[RG][kEncNS];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    const int row = rb * (64 * RG) + (wave * RG + r) * 16 + fr;
#pragma unroll
    for (int s = 0; s < kEncNS; ++s) {
      const int d = 32 * s + 8 * g;
      qf[r][s] = bload8(rq, row < sq && d < HD
                                ? ((uint32_t)row * (uint32_t)p.q_tok_stride + (uint32_t)d) * 2u
                                : kOOB);
    }
  }
  // zeros in the dims HD .. 95 of both K tiles, which QK^T reads
  for (int i = tid; i < 2 * kEncKT * (12 - kch); i += 256) {
    const int key = i & (kEncKT - 1), b = (i >> 6) & 1, c = kch + (i >> 7);
    st8(&tiles[b * (kEncK + kEncV) + key * kEncLDK + 8 * c], zero8());
  }

  const float sc = p.scale * 1.4426950408889634f;
  float m_run[RG], l_run[RG];
  f32x4_t o[RG][kEncND];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    m_run[r] = -INFINITY;
    l_run[r] = 0.f;
#pragma unroll
    for (int i = 0; i < kEncND; ++i) o[r][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const int nt = sk / kEncKT;
  store(0);
  if (nt > 1) load(1);
  for (int t = 0; t < nt; ++t) {
    __syncthreads();  // tile t is written, tile t - 1 is read
    const bf16_t* sK = tiles + (t & 1) * (kEncK + kEncV);
    const bf16_t* sV = sK + kEncK;
    // lane: scores of keys 16 kf + 4 g + e with its row
    f32x4_t s[RG][4];
#pragma unroll
    for (int kf = 0; kf < 4; ++kf) {
#pragma unroll
      for (int r = 0; r < RG; ++r) s[r][kf] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ss = 0; ss < kEncNS; ++ss) {
        const bf16x8 kf8 = ld8(&sK[(kf * 16 + fr) * kEncLDK + ss * 32 + 8 * g]);
#pragma unroll
        for (int r = 0; r < RG; ++r) s[r][kf] = mfma16x16x32(kf8, qf[r][ss], s[r][kf]);
      }
    }
    bf16x8 pa[RG][2];
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      float mx = s[r][0][0], a, b;
#pragma unroll
      for (int kf = 0; kf < 4; ++kf)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[r][kf][e]);
      enc_pair16(mx, a, b);
      mx = fmaxf(a, b);
      mx = half_pair_max(mx);
      const float m_new = fmaxf(m_run[r], mx * sc);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run[r] - m_ref);
      m_run[r] = m_new;
      l_run[r] *= alpha;
#pragma unroll
      for (int c = 0; c < 2; ++c) {  // keys 32 c + {4 g + e, 16 + 4 g + e}
        float pf[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pf[e] = __builtin_amdgcn_exp2f(fmaf(s[r][2 * c + (e >> 2)][e & 3], sc, -m_ref));
          l_run[r] += pf[e];
        }
        pa[r][c] = pack8(pf);
      }
#pragma unroll
      for (int df = 0; df < kEncND; ++df)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[r][df][j] *= alpha;
    }
#pragma unroll
    for (int df = 0; df < kEncND; ++df)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const bf16_t* vt = &sV[(df * 16 + fr) * kEncLDV + 32 * c + 4 * g];
        const uint2 lo = *(const uint2*)vt, hi = *(const uint2*)(vt + 16);
        bf16x8 vb;
        vb.w[0] = lo.x;
        vb.w[1] = lo.y;
        vb.w[2] = hi.x;
        vb.w[3] = hi.y;
#pragma unroll
        for (int r = 0; r < RG; ++r) o[r][df] = mfma16x16x32(vb, pa[r][c], o[r][df]);
      }
    if (t + 1 < nt) {
      store((t + 1) & 1);
      if (t + 2 < nt) load(t + 2);
    }
  }

#pragma unroll
  for (int r = 0; r < RG; ++r) {
    float a, b;
    enc_pair16(l_run[r], a, b);
    const float l = half_pair_sum(a + b), inv = l > 0.f ? 1.f / l : 0.f;
    const int row = rb * (64 * RG) + (wave * RG + r) * 16 + fr;
    if (row < sq) {
      bf16_t* orow = O + (int64_t)row * p.o_tok_stride + 4 * g;
#pragma unroll
      for (int df = 0; df < kEncND; ++df)
        if (16 * df + 4 * g < HD)
          *(uint2*)(orow + 16 * df) = uint2{f2bf2(o[r][df][0] * inv, o[r][df][1] * inv),
                                            f2bf2(o[r][df][2] * inv, o[r][df][3] * inv)};
    }
  }
}

// One query head per problem, every key visible, whole key tiles and one key
// range, head dim <= 80, 8-byte output rows, operand views below 2 GiB, fewer than
// 2^32 threads (a launch's limit; the general kernel's grid has three axes); the scale
// is positive, so that the largest score is the largest product, and at most 1 in
// base 2, so that scaling cannot overflow.
bool encoder_attn_ok(const fvx_attn_desc& d) {
  const int64_t lim = (int64_t)1 << 30;
  const float sc = d.scale * 1.4426950408889634f;
  return d.heads == 1 && !d.kgrp && d.v_d_stride == 0 && d.head_dim <= 80 && d.o &&
         d.kv_splits <= 1 && d.sk % kEncKT == 0 && d.sq < lim && d.sk < lim && sc > 0.f &&
         sc <= 1.f && d.q_tok_stride >= 0 && d.sq * d.q_tok_stride + 80 < lim &&
         d.k_tok_stride >= d.head_dim && d.v_tok_stride >= d.head_dim &&
         (d.sk + 2 * kEncKT) * d.k_tok_stride < lim &&
         (d.sk + 2 * kEncKT) * d.v_tok_stride < lim && ((uintptr_t)d.o & 7u) == 0 &&
         d.o_tok_stride % 4 == 0 && d.o_zs1 % 4 == 0 && d.o_zs2 % 4 == 0 &&
         d.n_problems * ((d.sq + 63) / 64) < ((int64_t)1 << 24);
}

// 128 rows per workgroup once blocks of 64 number more than the CUs and two of them
// share a problem, 64 else.
// Measured (us per call, images of 256 patches, 16 heads of 72: attn_kernel / 64
// rows / 128 rows): 1 image 11.7 / 7.2 / 9.3, 3 images 13.9 / 7.4 / 9.5, 5 images
// 18.0 / 9.9 / 9.8, 24 images 44.8 / 27.1 / 23.4, 96 images 148 / 90 / 74 (390
// TFLOP/s).  4000 problems of 64 rows x 512 keys 164 / 140 / 170: half of 128 rows are
// absent there.  Two groups of 4 waves with every other tile each were no faster at 1 to
// 3 images (7.4 to 7.7).
int run_encoder_attn(const fvx_attn_desc& d, hipStream_t s) {
  const uint32_t kch = (uint32_t)(d.head_dim / 8);
  const uint32_t magic = (65536u + kch - 1) / kch;  // i / kch for i < 768
  const int64_t n64 = (d.sq + 63) / 64, n128 = (d.sq + 127) / 128;
  if (d.n_problems * n64 <= device_cus() || n64 == n128)
    hipLaunchKernelGGL((attn_encoder_kernel<1>), dim3((unsigned)(d.n_problems * n64)), dim3(256),
                       0, s, d, (int)n64, magic);
  else
    hipLaunchKernelGGL((attn_encoder_kernel<2>), dim3((unsigned)(d.n_problems * n128)), dim3(256),
                       0, s, d, (int)n128, magic);
  return launch_status("attention(encoder)");
}

}  // namespace fvx
