// Shared by the GEMM kernels: the descriptor, the fused epilogue on chunks of
// 8 columns (operand reads, arithmetic, stores, hand-over outputs) and the
// host-side checks of what an epilogue build covers.
#pragma once

#include "capi_util.h"
#include "common.h"

namespace fvx {

typedef fvx_gemm_desc GemmArgs;

// The largest number of product rows that one workgroup's epilogue covers
constexpr int64_t kEpiRows = 256;

// The first kCounterBytes of a GEMM workspace hold the per-column-tile
// arrival counters of the split-K skinny kernel; fp32 partials follow.
constexpr int kCounterBytes = 4096;
constexpr int kMaxSkinnyTiles = kCounterBytes / 4;

// Tile rows per block of the tile order (tile_order): about 1024 rows of the 64 x 128
// and wide tiles (the tile kernel's 128- and 256-row tiles: 2048 and 4096).  One
// block of all rows against this, us (MI355X, weights from HBM): prefix down
// 6528 x 2048 x 16384 538 -> 428 (all 26 tile rows on every XCD streamed A
// eight times), gate/up 6528 x 2 x 16384 x 2048 775 -> 750, Q|K|V 107 -> 98;
// SigLIP fc1 6144 x 4304 x 1152 97 -> 89, Q|K|V 81 -> 75, fc2 120 -> 114; fp8
// gate/up at 22144 rows 2970 -> 2850.  Blocks of 2048 rows: gate/up 785.
constexpr int kTileRowBlock = 16;  // of the tile kernel
constexpr int kWideRowBlock = 4;   // of 256 rows

// Row indices and the epilogue's periods (row_group, gate_group,
// pos_period, rtc_period) are below 2^31 (the host checks), so quotients and
// remainders take the 32-bit unsigned divide: the 64-bit one is a long
// software sequence per lane.
__device__ __forceinline__ uint32_t udiv32(int64_t a, int64_t b) {
  return (uint32_t)a / (uint32_t)b;
}
__device__ __forceinline__ uint32_t umod32(int64_t a, int64_t b) {
  return (uint32_t)a % (uint32_t)b;
}

__device__ __forceinline__ int64_t out_row(const GemmArgs& p, int64_t m) {
  if (p.row_group <= 0) return m;
  const uint32_t q = udiv32(m, p.row_group);
  return (int64_t)q * p.row_group_stride + ((uint32_t)m - q * (uint32_t)p.row_group);
}

// sum of squares of 8 bf16 values: four v_dot2c_f32_bf16 (fp32 accumulate)
__device__ __forceinline__ float sumsq8(const bf16x8& v) {
  typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bf16x2v h = __builtin_bit_cast(bf16x2v, v.w[i]);
    s = __builtin_amdgcn_fdot2_f32_bf16(h, h, s, false);
  }
  return s;
}

// sum of 8 bf16 values: four dot products with (1, 1) (exact products)
__device__ __forceinline__ float sum8(const bf16x8& v) {
  typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
  const bf16x2v one = {(__bf16)1.0f, (__bf16)1.0f};
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2v, v.w[i]), one, s, false);
  return s;
}

// ---------------------------------------------------------------------------
// Row-chunk epilogue: output columns n .. n + 7 of one row m.
//
// epi_load_col and epi_load_row issue every global read the epilogue needs
// (the column operands: bias, fp32 biases, the RTC lock; the row operands:
// residual, gate, position table, Euler state, RoPE table) and epi_store
// computes and writes.  Callers issue the reads for all of their chunks
// before the first epi_store: an in-place operand (residual == c, xt) may
// alias the output, so a read issued after a store would wait for a full
// memory round trip per element.  A lane of the tile and wide kernels keeps
// one column chunk in every item, so those kernels read the column operands
// once per lane.  `vec`: the chunk holds 8 columns and every operand is
// 16-byte aligned, so each operand moves as one 16-byte (fp32: two) access;
// otherwise `cnt` columns are handled one by one.
// ---------------------------------------------------------------------------
struct EpiIn {
  bf16x8 res, gate, pos, bias;
  float f0[8];    // bias_f32 (PLAIN, EULER) or RoPE (cos, sin) x 4 (QKV_ROPE)
  float xt[8];    // EULER state
  float prev[8];  // EULER with RTC: the previous chunk's actions
  float cw;       // EULER with RTC guidance: the row's correction weight
  float cs[8];    // PLAIN with a folded LayerNorm: the weight's column sums
  bool locked;    // PLAIN, EULER: the row is in the RTC locked prefix
};

__device__ __forceinline__ void st_b8(bf16_t* dst, const float* x, bool vec,
                                      int cnt) {
  if (vec) {
    st8(dst, pack8(x));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < cnt) dst[e] = f2bf(x[e]);
  }
}

__device__ __forceinline__ void st_f8(float* dst, const float* x, bool vec,
                                      int cnt) {
  if (vec) {
    *(f32x4_t*)dst = f32x4_t{x[0], x[1], x[2], x[3]};
    *(f32x4_t*)(dst + 4) = f32x4_t{x[4], x[5], x[6], x[7]};
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < cnt) dst[e] = x[e];
  }
}

// Buffer-view reads for the epilogue: a NULL operand gets an empty view (all
// reads return zero) and no load sits behind a branch, so the compiler can
// keep every load of a batch in flight (a branch around a load makes it
// wait for that load at the join).
__device__ __forceinline__ uint32_t rec_bytes(int64_t b) {
  return b > 0x7fffffff ? 0x7fffffffu : (uint32_t)b;
}

__device__ __forceinline__ bf16x8 bl_b8(__amdgpu_buffer_rsrc_t r, uint32_t off,
                                        bool vec) {
  if (vec) return bload8(r, off);
  bf16x8 v;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v.w[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, off + 4 * i, 0, 0) |
             ((uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, off + 4 * i + 2, 0, 0) << 16);
  return v;
}

__device__ __forceinline__ void bl_f8(__amdgpu_buffer_rsrc_t r, uint32_t off,
                                      bool vec, float* d) {
  if (vec) {
    const f32x4_t a = bload4f(r, off), b = bload4f(r, off + 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d[e] = a[e];
      d[4 + e] = b[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] = bload1f(r, off + 4 * e);
  }
}

// Buffer views of the epilogue's operands: uniform, built once per wave
// outside the item loops (an absent operand gets an empty view, whose reads
// return zeros).  A view holds less than 2 GiB and its offsets have 32 bits, so
// the row operands' views begin at the caller's first row m0 (m0, and below its
// output and gate rows) and cover up to kEpiRows rows from there: operands of
// any size are read right while those rows span less than 2 GiB (validate).
struct EpiViews {
  uint32_t m0, orow0, grow0;  // (offsets from them are taken modulo 2^32)
  __amdgpu_buffer_rsrc_t bias, bf32, gate, res, pos, xt, prev, cw, rope, positions, csum;
};

// (SP: the plain-epilogue build -- PLAIN with bias, fp32 bias, activation,
// a per-row gate, residual and the fragment-major copy only; the host
// checks that the call uses nothing else)
template <int MODE, bool SP = false>
__device__ __forceinline__ EpiViews epi_views(const GemmArgs& p, int64_t m0) {
  EpiViews V;
  const int64_t N = p.n, ml = p.m - m0;
  V.m0 = V.orow0 = V.grow0 = (uint32_t)m0;
  V.bias = V.bf32 = V.gate = V.res = V.pos = V.xt = V.prev = V.cw = V.rope = V.positions =
      V.csum = make_rsrc(nullptr, 0u);
  if constexpr (SP) {
    V.bias = make_rsrc(p.bias, p.bias ? rec_bytes(N * 2) : 0u);
    V.bf32 = make_rsrc(p.bias_f32, p.bias_f32 ? rec_bytes(N * 4) : 0u);
    V.res = make_rsrc((const bf16_t*)p.residual + m0 * p.ldr,
                      p.residual ? rec_bytes(ml * p.ldr * 2) : 0u);
    V.gate = make_rsrc((const bf16_t*)p.gate + m0 * p.ldg,
                       p.gate ? rec_bytes(ml * p.ldg * 2) : 0u);
    return V;
  }
  if (MODE == FVX_GEMM_QKV_ROPE) {
    V.positions = make_rsrc(p.positions + m0, rec_bytes(ml * 4));
    V.rope = make_rsrc(p.rope, 0x7fffffffu);
  }
  if (MODE == FVX_GEMM_PLAIN || MODE == FVX_GEMM_EULER) {
    V.bias = make_rsrc(p.bias, p.bias ? rec_bytes(N * 2) : 0u);
    V.bf32 = make_rsrc(p.bias_f32, p.bias_f32 ? rec_bytes(N * 4) : 0u);
  }
  if (MODE == FVX_GEMM_EULER) {
    V.xt = make_rsrc(p.xt + m0 * p.ldx, rec_bytes(ml * p.ldx * 4));
    V.prev = make_rsrc(p.rtc_prev + m0 * p.ld_prev,
                       p.rtc_prev ? rec_bytes(ml * p.ld_prev * 4) : 0u);
    V.cw = make_rsrc(p.rtc_cw, p.rtc_cw ? rec_bytes(p.rtc_period * 4) : 0u);
  }
  if (MODE == FVX_GEMM_PLAIN) {
    V.csum = make_rsrc(p.ln_csum, p.ln_csum ? rec_bytes(N * 4) : 0u);
    const bool gdiv = p.gate_group > 1;
    const int64_t grows = gdiv ? udiv32(p.m + p.gate_group - 1, p.gate_group) : p.m;
    if (gdiv) V.grow0 = udiv32(m0, p.gate_group);
    V.gate = make_rsrc((const bf16_t*)p.gate + V.grow0 * p.ldg,
                       p.gate ? rec_bytes((grows - V.grow0) * p.ldg * 2) : 0u);
    // (from the start of m0's group: no row of the tile lies before it)
    const int64_t orow0 =
        p.row_group > 0 ? (int64_t)udiv32(m0, p.row_group) * p.row_group_stride : m0;
    V.orow0 = (uint32_t)orow0;
    V.res = make_rsrc((const bf16_t*)p.residual + orow0 * p.ldr,
                      p.residual ? rec_bytes((out_row(p, p.m - 1) + 1 - orow0) * p.ldr * 2) : 0u);
    const int64_t pp = p.pos_period > 0 ? p.pos_period : 1;
    V.pos = make_rsrc(p.pos, p.pos ? rec_bytes(pp * p.ldp * 2) : 0u);
  }
  return V;
}

// the column operands of columns n .. n + 7 (bias_f32: the unlocked rows')
// (LN: the kernel build with the folded LayerNorm, which reads ln_csum)
template <int MODE, bool LN = false>
__device__ __forceinline__ void epi_load_col(const EpiViews& V, int64_t n, bool vec,
                                             EpiIn& in) {
  if (MODE != FVX_GEMM_PLAIN && MODE != FVX_GEMM_EULER) return;
  in.bias = bl_b8(V.bias, (uint32_t)(n * 2), vec);
  bl_f8(V.bf32, (uint32_t)(n * 4), vec, in.f0);
  if (MODE == FVX_GEMM_PLAIN && LN) bl_f8(V.csum, (uint32_t)(n * 4), vec, in.cs);
}

// the row operands of row m, columns n .. n + 7
template <int MODE, bool SP = false>
__device__ __forceinline__ void epi_load_row(const GemmArgs& p, const EpiViews& V, int64_t m,
                                             int64_t n, bool vec, int cnt, EpiIn& in) {
  if (MODE == FVX_GEMM_GEGLU) return;
  if constexpr (SP) {
    const uint32_t ml = (uint32_t)m - V.m0;
    in.res = bl_b8(V.res, (ml * (uint32_t)p.ldr + (uint32_t)n) * 2u, vec);
    in.gate = bl_b8(V.gate, (ml * (uint32_t)p.ldg + (uint32_t)n) * 2u, vec);
    return;
  }
  if (MODE == FVX_GEMM_QKV_ROPE) {
    const int hd = p.head_dim;
    const bool rot = n < (int64_t)(p.n_q_heads + 1) * hd;
    const int64_t pos =
        (int32_t)__builtin_amdgcn_raw_buffer_load_b32(V.positions, ((uint32_t)m - V.m0) * 4u, 0,
                                                      0);
    bl_f8(V.rope, rot ? (uint32_t)((pos * (hd >> 1) + (umod32(n, hd) >> 1)) * 8) : kOOB, vec,
          in.f0);
    return;
  }
  // real-time chunking: the row's position within its chunk and the locked
  // prefix (*rtc_lock: one scalar load, which waits for no vector load)
  const int rr = p.rtc_period > 0 ? (int)umod32(m, p.rtc_period) : 0;
  in.locked = false;
  if (p.rtc_lock) in.locked = rr < *(const __attribute__((address_space(4))) int32_t*)p.rtc_lock;
  if (p.bias_f32_locked) {  // (f0 holds the unlocked rows' bias: epi_load_col)
    float fl[8];
    bl_f8(make_rsrc(p.bias_f32_locked, rec_bytes(p.n * 4)), (uint32_t)(n * 4), vec, fl);
#pragma unroll
    for (int e = 0; e < 8; ++e) in.f0[e] = in.locked ? fl[e] : in.f0[e];
  }
  if (MODE == FVX_GEMM_EULER) {
    const uint32_t ml = (uint32_t)m - V.m0;
    bl_f8(V.xt, (ml * (uint32_t)p.ldx + (uint32_t)n) * 4u, vec, in.xt);
    bl_f8(V.prev, (ml * (uint32_t)p.ld_prev + (uint32_t)n) * 4u, vec, in.prev);
    in.cw = bload1f(V.cw, (uint32_t)(rr * 4));
    return;
  }
  const uint32_t grow = (p.gate_group > 1 ? udiv32(m, p.gate_group) : (uint32_t)m) - V.grow0;
  in.gate = bl_b8(V.gate, (grow * (uint32_t)p.ldg + (uint32_t)n) * 2u, vec);
  const uint32_t orow = (uint32_t)out_row(p, m) - V.orow0;
  in.res = bl_b8(V.res, (orow * (uint32_t)p.ldr + (uint32_t)n) * 2u, vec);
  in.pos = bl_b8(V.pos,
                 (uint32_t)(((p.pos_period > 1 ? umod32(m, p.pos_period) : 0) * p.ldp + n) * 2),
                 vec);
}

template <int MODE>
__device__ __forceinline__ void epi_load(const GemmArgs& p, const EpiViews& V, int64_t m,
                                         int64_t n, bool vec, int cnt, EpiIn& in) {
  epi_load_col<MODE>(V, n, vec, in);
  epi_load_row<MODE>(p, V, m, n, vec, cnt, in);
}

// v: main accumulators, u: GEGLU up accumulators, r: RMS factor of row m
// (LN build with a folded LayerNorm: its rsqrt(var + eps), with mr =
// mean * r).  want_xo (PLAIN, GEGLU): xo receives the 8 values as stored
// (bf16-rounded unless out_f32), for the hand-over outputs (epi_handoff).
template <int MODE, bool LN = false, bool SP = false>
__device__ __forceinline__ void epi_store(const GemmArgs& p, int64_t m,
                                          int64_t n, bool vec, int cnt,
                                          const float* v, const float* u,
                                          float r, const EpiIn& in,
                                          bool want_xo, float* xo, float mr = 0.f) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = v[e] * r;
  if constexpr (SP && MODE == FVX_GEMM_PLAIN) {
    // the same operations in the same order as below, with 32-bit row
    // offsets (the host keeps m * ldc below 2^31)
    float t[8];
    unpack8(in.bias, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] += t[e] + in.f0[e];
    if (p.act == FVX_ACT_SILU) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = silu(x[e]);
    } else if (p.act == FVX_ACT_GELU_TANH) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = gelu_tanh(x[e]);
    }
    if (p.gate) {
      unpack8(in.gate, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= t[e];
    }
    if (p.residual) {
      unpack8(in.res, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] += t[e];
    }
    st_b8((bf16_t*)p.c + ((uint32_t)m * (uint32_t)p.ldc + (uint32_t)n), x, vec, cnt);
    if (p.c_frag) st8((bf16_t*)p.c_frag + frag_offset(m, n), pack8(x));
    if (want_xo) unpack8(pack8(x), xo);
    return;
  }
  if (MODE == FVX_GEMM_PLAIN && LN && p.ln_csum)
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = fmaf(-mr, in.cs[e], x[e]);
  if (MODE == FVX_GEMM_GEGLU) {
    if (p.gu_out) {
      // the pre-activations the product is taken from (gate | up)
      float uu[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) uu[e] = u[e] * r;
      bf16_t* g = (bf16_t*)p.gu_out + out_row(p, m) * p.ld_gu + n;
      st_b8(g, x, vec, cnt);
      st_b8(g + p.n, uu, vec, cnt);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = gelu_tanh(x[e]) * (u[e] * r);
    st_b8((bf16_t*)p.c + out_row(p, m) * p.ldc + n, x, vec, cnt);
    if (p.c_frag) st8((bf16_t*)p.c_frag + frag_offset(m, n), pack8(x));
    if (want_xo) unpack8(pack8(x), xo);
    return;
  }
  if (MODE == FVX_GEMM_QKV_ROPE) {
    const int hd = p.head_dim;
    const int64_t qcols = (int64_t)p.n_q_heads * hd;
    if (n < qcols + hd) {
      // pair (2i, 2i+1) = (x_i, x_{i+hd/2}) rotated by (cos, sin)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = x[2 * i], b = x[2 * i + 1];
        const float c = in.f0[2 * i], s = in.f0[2 * i + 1];
        x[2 * i] = a * c - b * s;
        x[2 * i + 1] = b * c + a * s;
      }
      if (n < qcols) {
        st_b8((bf16_t*)p.q_out + m * p.ldq + n, x, vec, cnt);
      } else {
        st_b8((bf16_t*)p.k_out + out_row(p, m) * p.ldk + (n - qcols), x, vec,
              cnt);
        if (p.k_t_out) {
          // the keys transposed as well ([group][head_dim][ld_kt])
          const int64_t b = p.row_group > 0 ? udiv32(m, p.row_group) : 0;
          const int64_t t = p.row_group > 0 ? umod32(m, p.row_group) : m;
          bf16_t* dst = (bf16_t*)p.k_t_out + (b * hd + (n - qcols)) * p.ld_kt + t;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < cnt) dst[e * p.ld_kt] = f2bf(x[e]);
        }
      }
    } else if (p.v_transposed) {
      // V^T cache: [group][head_dim][ldv], tokens contiguous
      const int64_t b = p.row_group > 0 ? udiv32(m, p.row_group) : 0;
      const int64_t t = p.row_group > 0 ? umod32(m, p.row_group) : m;
      bf16_t* dst = (bf16_t*)p.v_out + (b * hd + (n - qcols - hd)) * p.ldv + t;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < cnt) dst[e * p.ldv] = f2bf(x[e]);
      if (p.v_rows_out)  // the values row-major as well
        st_b8((bf16_t*)p.v_rows_out + out_row(p, m) * p.ld_vr + (n - qcols - hd), x, vec,
              cnt);
    } else {
      st_b8((bf16_t*)p.v_out + out_row(p, m) * p.ldv + (n - qcols - hd), x,
            vec, cnt);
    }
    return;
  }
  float t[8];
  unpack8(in.bias, t);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] += t[e] + in.f0[e];
  if (MODE == FVX_GEMM_EULER) {
    float nx[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) nx[e] = in.xt[e] + p.dt * x[e];
    if (p.rtc_cw) {
      // guidance: x_1 = xt - omt * v is the predicted clean chunk; the
      // velocity is corrected by gw * w_r * (prev - x_1)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        nx[e] += in.cw * (in.prev[e] - in.xt[e] + p.rtc_omt * x[e]);
    }
    if (in.locked && p.rtc_prev) {
#pragma unroll
      for (int e = 0; e < 8; ++e) nx[e] = in.prev[e];
    }
    st_f8(p.xt + m * p.ldx + n, nx, vec, cnt);
    if (p.xt_bf16) st_b8((bf16_t*)p.xt_bf16 + m * p.ldxb + n, nx, vec, cnt);
    return;
  }
  if (p.act == FVX_ACT_SILU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = silu(x[e]);
  } else if (p.act == FVX_ACT_GELU_TANH) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = gelu_tanh(x[e]);
  }
  if (p.gate) {
    unpack8(in.gate, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= t[e];
  }
  if (p.residual) {
    unpack8(in.res, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] += t[e];
  }
  if (p.pos) {
    unpack8(in.pos, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] += t[e];
  }
  const int64_t orow = out_row(p, m);
  if (p.out_f32)
    st_f8((float*)p.c + orow * p.ldc + n, x, vec, cnt);
  else
    st_b8((bf16_t*)p.c + orow * p.ldc + n, x, vec, cnt);
  if (p.c_frag) st8((bf16_t*)p.c_frag + frag_offset(m, n), pack8(x));
  if (want_xo) {
    if (p.out_f32) {
#pragma unroll
      for (int e = 0; e < 8; ++e) xo[e] = x[e];
    } else {
      unpack8(pack8(x), xo);
    }
  }
}

// Hand-over outputs of one row's 64-column block, held as 8-column chunks
// n .. n + 7 by 8 consecutive lanes (every lane runs the shuffles; `valid`:
// this lane's chunk exists; the block's first lane stores): the row's sum of
// squares of the stored values (ss_out) and the e4m3 copy with the block's
// E8M0 exponent (a8_out), quantized exactly as quant_fp8x32 quantizes an A
// block.
__device__ __forceinline__ void epi_handoff(const GemmArgs& p, bool valid, int64_t m,
                                            int64_t n, int cnt, const float* xo) {
  const bool lead = ((n >> 3) & 7) == 0;
  if (p.ss_out) {
    float q = 0.f;
    if (valid)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < cnt) q += xo[e] * xo[e];
    q += __shfl_xor(q, 1, 64);
    q += __shfl_xor(q, 2, 64);
    q += __shfl_xor(q, 4, 64);
    if (lead && valid) p.ss_out[(n / 64) * p.ss_ld + m] = q;
  }
  if (p.a8_out) {
    const bf16x8 b = pack8(xo);
    uint32_t mx = 0;
    if (valid)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w = b.w[j] & 0x7fff7fffu;
        const uint32_t lo = 2 * j < cnt ? (w & 0xffffu) : 0u;
        const uint32_t hi = 2 * j + 1 < cnt ? (w >> 16) : 0u;
        mx = lo > mx ? lo : mx;
        mx = hi > mx ? hi : mx;
      }
#pragma unroll
    for (int sh = 1; sh <= 4; sh <<= 1) {
      const uint32_t o = (uint32_t)__shfl_xor((int)mx, sh, 64);
      mx = o > mx ? o : mx;
    }
    const int e = e8m0_for_amax(mx);
    if (valid) {
      const float scale = __uint_as_float((uint32_t)e << 23);
      uint32_t q[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        i16x2_t r = {0, 0};
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(
            r, __builtin_bit_cast(bf16x2_t, b.w[2 * j]), scale, false);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(
            r, __builtin_bit_cast(bf16x2_t, b.w[2 * j + 1]), scale, true);
        q[j] = __builtin_bit_cast(uint32_t, r);
      }
      unsigned char* dst = (unsigned char*)p.a8_out + m * p.a8_out_ld + n;
      if (cnt == 8) {
        *(uint2*)dst = uint2{q[0], q[1]};
      } else {
#pragma unroll
        for (int x = 0; x < 8; ++x)
          if (x < cnt) dst[x] = (unsigned char)(q[x >> 2] >> (8 * (x & 3)));
      }
      if (lead) ((unsigned char*)p.a8_out_scale)[(n / 64) * p.a8_out_sld + m] = (unsigned char)e;
    }
  }
}

// The handed-over sums of squares (`parts`: ss_in) of rows m0 .. m0 + R - 1,
// with every thread of an NT-thread workgroup: thread t loads parts
// t / R, t / R + NT / R, ... of row t % R, all loads in flight (up to 64
// parts per row; more take a loop), and thread t < R receives its row's
// total, added in a fixed order.  A loop over the parts in one thread per row
// waited for a memory round trip per 8 parts before its wave could start
// the K loop.  Every thread must call it (two barriers); sTmp: NT floats
// of LDS.
template <int R, int NT>
__device__ float rows_parts_sum(const GemmArgs& p, const float* parts, int64_t m0, int64_t M,
                                float* sTmp) {
  static_assert(NT % R == 0, "whole rows per thread group");
  constexpr int STEP = NT / R, MAXL = (64 + STEP - 1) / STEP;
  const int tid = threadIdx.x, row = tid % R, j0 = tid / R;
  const int64_t m = m0 + row;
  const bool mv = m < M;
  const __amdgpu_buffer_rsrc_t rs =
      make_rsrc(parts, rec_bytes((int64_t)p.ss_parts * p.ss_ld * 4));
  float acc = 0.f;
  if (p.ss_parts <= STEP * MAXL) {
    float t[MAXL];
#pragma unroll
    for (int u = 0; u < MAXL; ++u) {
      const int q = j0 + STEP * u;
      t[u] = bload1f(rs, (mv && q < p.ss_parts) ? (uint32_t)(((int64_t)q * p.ss_ld + m) * 4)
                                                : kOOB);
    }
#pragma unroll
    for (int u = 0; u < MAXL; ++u) acc += t[u];
  } else {
    for (int q = j0; q < p.ss_parts; q += STEP)
      acc += bload1f(rs, mv ? (uint32_t)(((int64_t)q * p.ss_ld + m) * 4) : kOOB);
  }
  sTmp[tid] = acc;
  __syncthreads();
  float tot = 0.f;
  if (tid < R)
#pragma unroll
    for (int j = 0; j < STEP; ++j) tot += sTmp[j * R + tid];
  __syncthreads();  // sTmp may be reused
  return tot;
}

// The tile kernel's handed-over row sums of squares (ss_in) of rows m0 ..
// m0 + R - 1, split in two so that no wait sits in front of the K loop:
// issue() puts every load in flight ahead of the first slabs (thread t takes
// parts t / R, t / R + NT / R, ... of row t % R, up to STEP * L parts per row
// in registers), finish() adds them after the K loop, when they have long
// landed; rows with more parts are loaded by finish() itself.  Thread t < R
// receives its row's total, added in a fixed order.  Every thread calls
// finish() (one barrier); sTmp: NT floats of LDS, not to be rewritten before
// the caller's next barrier.
template <int R, int NT>
struct RowParts {
  static_assert(NT % R == 0, "whole rows per thread group");
  static constexpr int STEP = NT / R, L = STEP >= 4 ? (48 + STEP - 1) / STEP : 12;
  float q[L];

  __device__ __forceinline__ bool in_regs(const GemmArgs& p) const {
    return p.ss_parts <= STEP * L;
  }
  // byte offset of part qi of row m (the host keeps the array below 2^31
  // bytes); kOOB (a zero) past the parts or the rows
  __device__ __forceinline__ static uint32_t off(uint32_t row4, uint32_t ld4, int qi, int parts,
                                                 bool mv) {
    const uint32_t o = row4 + (uint32_t)qi * ld4;
    return (mv && qi < parts) ? o : kOOB;
  }
  __device__ __forceinline__ void issue(const GemmArgs& p, int64_t m0, int64_t M) {
    const int tid = threadIdx.x, j0 = tid / R, parts = p.ss_parts;
    const int64_t m = m0 + tid % R;
    const bool mv = m < M && in_regs(p);
    const uint32_t row4 = (uint32_t)m * 4u, ld4 = (uint32_t)p.ss_ld * 4u;
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(p.ss_in, rec_bytes((int64_t)parts * p.ss_ld * 4));
#pragma unroll
    for (int u = 0; u < L; ++u) q[u] = bload1f(rq, off(row4, ld4, j0 + STEP * u, parts, mv));
  }
  __device__ __forceinline__ float finish(const GemmArgs& p, int64_t m0, int64_t M,
                                          float* sTmp) {
    const int tid = threadIdx.x, j0 = tid / R, parts = p.ss_parts;
    const int64_t m = m0 + tid % R;
    float aq = 0.f;
    if (in_regs(p)) {
      // the sum starts here, after the K loop, not where the loads were
      // issued (an add hoisted there would wait for them)
#pragma unroll
      for (int u = 0; u < L; ++u) {
        asm volatile("" : "+v"(q[u]));
        aq += q[u];
      }
    } else {
      const uint32_t row4 = (uint32_t)m * 4u, ld4 = (uint32_t)p.ss_ld * 4u;
      const __amdgpu_buffer_rsrc_t rq =
          make_rsrc(p.ss_in, rec_bytes((int64_t)parts * p.ss_ld * 4));
      for (int qi = j0; qi < parts; qi += STEP) aq += bload1f(rq, off(row4, ld4, qi, parts, m < M));
    }
    sTmp[tid] = aq;
    __syncthreads();
    float tq = 0.f;
    if (tid < R)
#pragma unroll
      for (int j = 0; j < STEP; ++j) tq += sTmp[j * R + tid];
    return tq;
  }
};

// Host check: may the chunk epilogue use 16-byte accesses for full chunks?
static bool epi_vec_ok(const GemmArgs& d) {
  auto al = [](const void* q) { return ((uintptr_t)q & 15u) == 0; };
  switch (d.mode) {
    case FVX_GEMM_GEGLU:
      return al(d.c) && d.ldc % 8 == 0;
    case FVX_GEMM_QKV_ROPE:
      return d.head_dim % 8 == 0 && al(d.rope) && al(d.q_out) &&
             d.ldq % 8 == 0 && al(d.k_out) && d.ldk % 8 == 0 &&
             (d.v_transposed || (al(d.v_out) && d.ldv % 8 == 0));
    case FVX_GEMM_EULER:
      return al(d.bias) && al(d.bias_f32) && al(d.bias_f32_locked) && al(d.xt) &&
             d.ldx % 4 == 0 && (!d.xt_bf16 || (al(d.xt_bf16) && d.ldxb % 8 == 0)) &&
             (!d.rtc_prev || (al(d.rtc_prev) && d.ld_prev % 4 == 0));
    default:
      return al(d.c) && d.ldc % (d.out_f32 ? 4 : 8) == 0 && al(d.bias) &&
             al(d.bias_f32) && al(d.bias_f32_locked) &&
             (!d.gate || (al(d.gate) && d.ldg % 8 == 0)) &&
             (!d.residual || (al(d.residual) && d.ldr % 8 == 0)) &&
             (!d.pos || (al(d.pos) && d.ldp % 8 == 0));
  }
}

// May a PLAIN GEMM's epilogue take the plain-epilogue build (the tile
// kernel's XF bit 3, the skinny kernel's and the split-K reduce's SP)?
// Bias, fp32 bias, activation, a per-row gate, residual, the fragment-major
// copy, the fused RMSNorm and the hand-overs only, bf16 output rows below
// 2^31 elements from the start of c.
static bool plain_epilogue_ok(const GemmArgs& d) {
  return d.mode == FVX_GEMM_PLAIN && !d.pos && !d.out_f32 && d.row_group == 0 && !d.rtc_lock &&
         !d.bias_f32_locked && !d.ln_csum && d.m * d.ldc < ((int64_t)1 << 31) &&
         (!d.gate || d.gate_group <= 1);
}

// A's rows in groups with gaps between them (fvx_gemm_desc.a_row_group)
static bool a_grouped(const GemmArgs& d) { return d.a_row_group > 0 && d.m > d.a_row_group; }

// gemm_pp.hip: the configuration of gemm_pp_kernel for d (-1: the other kernels
// serve it better or only they can) and its launch
int plan_pp(const GemmArgs& d);
int run_pp(const GemmArgs& d, int cfg, hipStream_t s);
// gemm_mid.hip: the same for gemm_mid_kernel
int plan_mid(const GemmArgs& d);
int run_mid(const GemmArgs& d, int cfg, hipStream_t s);

}  // namespace fvx
