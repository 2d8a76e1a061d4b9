// The value-independent part of the chunked delta rule, shared by the kernel that walks a
// head's chunks (gdn_chunk.hip) and the one that forms all chunks at once (gdn_split.hip):
// conv + SiLU of a 64-token chunk, gating, A, Tm = (I - A)^-1 and the masked q.k decay, in LDS.
// (The mathematics and the arithmetic are described at the top of gdn_chunk.hip.)  SM is the
// kernel's LDS struct; every function is called by the whole 256-thread workgroup, and the
// caller puts the barriers between them.
#pragma once

#include "gdn_common.h"

namespace lollm {

constexpr int GC_C = 64;     // tokens per chunk
constexpr int GC_PW = 136;   // bf16 pitch of 128-wide rows
constexpr int GC_PN = 72;    // bf16 pitch of 64-wide rows
constexpr int GC_PF = 68;    // fp32 pitch of 64-wide rows
constexpr int GC_PO = 132;   // fp32 pitch of the output rows

typedef float gc_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 gc_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gc_bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float gc_bf(uint16_t x) { return __uint_as_float((uint32_t)x << 16); }

__device__ __forceinline__ gc_f32x4 gc_mma(gc_bf16x8 a, gc_bf16x8 b, gc_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ gc_f32x4 gc_mma4(float a, float b, gc_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ gc_bf16x8 gc_ld8(const uint16_t* p) {
  return __builtin_bit_cast(gc_bf16x8, *reinterpret_cast<const u32x4_t*>(p));
}

// k slots 0..3 from p0, 4..7 from p1 (the accumulator row order)
__device__ __forceinline__ gc_bf16x8 gc_ld44(const uint16_t* p0, const uint16_t* p1) {
  const uint2 x = *reinterpret_cast<const uint2*>(p0), y = *reinterpret_cast<const uint2*>(p1);
  return __builtin_bit_cast(gc_bf16x8, u32x4_t{x.x, x.y, y.x, y.y});
}

// hi/lo bf16 of the 8 values p[0..3], q[0..3]
__device__ __forceinline__ void gc_split(gc_f32x4 p, gc_f32x4 q, gc_bf16x8& hi, gc_bf16x8& lo) {
  gc_bf16x8 h, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const __bf16 a = (__bf16)p[j], c = (__bf16)q[j];
    h[j] = a;
    h[j + 4] = c;
    l[j] = (__bf16)(p[j] - (float)a);
    l[j + 4] = (__bf16)(q[j] - (float)c);
  }
  hi = h;
  lo = l;
}

__device__ __forceinline__ uint16_t gc_bits(__bf16 x) { return __builtin_bit_cast(uint16_t, x); }

__device__ __forceinline__ float gc_rbf(float x) { return (float)(__bf16)x; }   // round to bf16

// 16-lane row sum in every lane of the row (DPP: quad xor 1, xor 2, half-row and row
// mirrors)
template <int CTRL> __device__ __forceinline__ float gc_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float gc_row16_sum(float v) {
  v += gc_dpp<0xB1>(v);
  v += gc_dpp<0x4E>(v);
  v += gc_dpp<0x141>(v);
  v += gc_dpp<0x140>(v);
  return v;
}

__device__ __forceinline__ uint32_t gc_pack(float lo, float hi) {
  return (uint32_t)gc_bits((__bf16)lo) | ((uint32_t)gc_bits((__bf16)hi) << 16);
}

// projection column of local channel lc (0..127 q, 128..255 k, 256..383 v) of head h
__device__ __forceinline__ int gc_chan(const GdnLayerArgs& a, int hk, int h, int lc) {
  return lc < GL_DK ? hk * GL_DK + lc
                    : (lc < 2 * GL_DK ? a.key_dim + hk * GL_DK + (lc - GL_DK)
                                      : 2 * a.key_dim + h * GL_DK + (lc - 2 * GL_DK));
}

// Conv work of a chunk: item n of thread tid = (8-channel vector cv of the 48, 4-token
// group tq of the 16) with it = tid + 256 n; its 7 input rows (3 history + 4) are
// loaded ahead of use.  Chunks after the first read the projection through a buffer
// descriptor over this sequence's rows: a row past the call reads as zero (it only
// feeds outputs of tokens past the call), no address is clamped, and a load costs one
// 32-bit add.  The loads are issued unconditionally and nothing touches the loaded
// values before their use, so no wait is placed at the loads and a later wait never
// drains loads issued after these.
constexpr int GC_ITEMS = 3;

__device__ __forceinline__ u32x4_t gc_bload(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}

// The NB blocks T_(j+d, j), d = 4 - NB, of Tm's block diagonal d (64 x 64, 16 x 16 blocks).
template <int NB>
__device__ __forceinline__ void gc_off_diagonal(float (*am)[GC_PF], float (*tf)[GC_PF], int r16, int g4) {
  constexpr int d = 4 - NB;
  gc_f32x4 p[NB], t[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    p[n] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
    t[n] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int kb = 0; kb < d; ++kb)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n = 0; n < NB; ++n)
        p[n] = gc_mma4(am[16 * (n + d) + r16][16 * (n + kb) + 4 * s + g4],
                       tf[16 * (n + kb) + 4 * s + g4][16 * n + r16], p[n]);
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int n = 0; n < NB; ++n)
      t[n] = gc_mma4(tf[16 * (n + d) + r16][16 * (n + d) + 4 * g4 + s], p[n][s], t[n]);
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) tf[16 * (n + d) + 4 * g4 + j][16 * n + r16] = t[n][j];
}

// Conv + SiLU of the chunk at t0 from the raw rows in registers, the L2-norm factors, and (wave
// 0) beta, g and cumsum(g).
template <class SM>
__device__ __forceinline__ void gc_conv_gating(SM& sh, const u32x4_t (&raw)[GC_ITEMS][7], uint16_t braw,
                                               uint16_t araw, float a_log, float dtb, int t0, int T,
                                               int tid, int wave, int lane) {
  // ================= conv + SiLU, L2-norm factors; beta, g, cumsum(g) =================
  // (every reader of the chunk buffers passed the barrier before the previous norm)
#pragma unroll
  for (int n = 0; n < GC_ITEMS; ++n) {
    const int it = tid + 256 * n, cv = it % 48, tq = it / 48;
    const int nvalid = T - (t0 + 4 * tq);   // tokens of the group inside the call
    // the 4-tap conv as two bf16 dot products per output: weights (tap 0, 1) and
    // (tap 2, 3) of a channel are consecutive bf16 pairs; the inputs are paired
    // (row r, row r + 1) per channel with a byte permute
    const u32x4_t* cwp = reinterpret_cast<const u32x4_t*>(&sh.cw[8 * cv][0]);
    uint32_t w01[8], w23[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4_t cw = cwp[q];
      w01[2 * q] = cw[0]; w23[2 * q] = cw[1]; w01[2 * q + 1] = cw[2]; w23[2 * q + 1] = cw[3];
    }
    uint32_t prs[6][8];   // (row r, row r + 1) of channel e
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        prs[r][2 * p] = __builtin_amdgcn_perm(raw[n][r + 1][p], raw[n][r][p], 0x05040100u);
        prs[r][2 * p + 1] = __builtin_amdgcn_perm(raw[n][r + 1][p], raw[n][r][p], 0x07060302u);
      }
    uint32_t pk[4][4];   // token r: bf16 pairs (channels 2p, 2p + 1)
    float ssq[4];        // token r: sum of squares over the 8 channels
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ssq[r] = 0.f;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        float o2[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int ee = 2 * p + u;
          float acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(gc_bf16x2, prs[r][ee]),
                                                      __builtin_bit_cast(gc_bf16x2, w01[ee]), 0.f, false);
          acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(gc_bf16x2, prs[r + 2][ee]),
                                                __builtin_bit_cast(gc_bf16x2, w23[ee]), acc, false);
          o2[u] = silu_g(gc_rbf(acc));
        }
        const uint32_t pv = gc_pack(o2[0], o2[1]);
        pk[r][p] = r < nvalid ? pv : 0u;
        // the two squares in one bf16 dot product (exact products, fp32 sum)
        ssq[r] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(gc_bf16x2, pk[r][p]),
                                                 __builtin_bit_cast(gc_bf16x2, pk[r][p]), ssq[r], false);
      }
    }
    // the 16 lanes of a DPP row hold the 16 channel vectors of one kind (q, k or v)
    // for the same 4 tokens: the row sum is the squared norm over 128 channels
#pragma unroll
    for (int r = 0; r < 4; ++r) ssq[r] = gc_row16_sum(ssq[r]);
    const int kind = cv >> 4, col = (cv & 15) * 8;   // 0 q, 1 k, 2 v
    if (kind < 2 && (cv & 15) == 0) {
      float* dstv = kind == 0 ? sh.rqv : sh.rkv;
#pragma unroll
      for (int r = 0; r < 4; ++r) dstv[4 * tq + r] = rsqrtf(ssq[r] + 1e-6f);
    }
    if (kind < 2) {
      uint16_t* dst = kind == 0 ? &sh.qc[0][0] : &sh.r1.kc[0][0];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<u32x4_t*>(dst + (4 * tq + r) * GC_PW + col) =
            u32x4_t{pk[r][0], pk[r][1], pk[r][2], pk[r][3]};
    }
    if (kind > 0) {
      uint16_t* dst = kind == 1 ? &sh.kt[0][0] : &sh.vt[0][0];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint32_t c[2];   // channel e of tokens (2 r2, 2 r2 + 1)
#pragma unroll
        for (int r2 = 0; r2 < 2; ++r2)
          c[r2] = __builtin_amdgcn_perm(pk[2 * r2 + 1][e >> 1], pk[2 * r2][e >> 1],
                                        e & 1 ? 0x07060302u : 0x05040100u);
        *reinterpret_cast<uint2*>(dst + (col + e) * GC_PN + 4 * tq) = make_uint2(c[0], c[1]);
      }
    }
  }
  if (wave == 0) {   // lane = token
    float gg = 0.f, bb = 0.f;
    if (t0 + lane < T) {
      const float x = gc_bf(araw) + dtb;   // softplus with torch's linear range above 20
      gg = -__expf(a_log) * (x > 20.f ? x : __logf(1.f + __expf(x)));
      bb = gc_rbf(__builtin_amdgcn_rcpf(1.f + __expf(-gc_bf(braw))));
    }
    // cumsum(g) over the chunk as an inclusive lane scan
    float gc = gg;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const float up = __shfl_up(gc, d, 64);
      gc += lane >= d ? up : 0.f;
    }
    sh.btv[lane] = bb;
    sh.gcv[lane] = gc;
    sh.egv[lane] = __expf(gc);
  }
}

// A = -(beta_i k_i.k_j) exp(gc_i - gc_j), j < i, and the scale vectors of W and the state update.
template <class SM>
__device__ __forceinline__ void gc_form_a(SM& sh, int tid, int wave, int r16, int g4) {
  if (tid < GC_C) {
    sh.fwv[tid] = sh.rkv[tid] * sh.btv[tid] * sh.egv[tid];
    sh.f7v[tid] = sh.rkv[tid] * __expf(sh.gcv[GC_C - 1] - sh.gcv[tid]);
  }
  // ================= A = -(beta_i k_i.k_j) exp(gc_i - gc_j), j < i =================
  // the 10 lower 16 x 16 tiles (ti >= tj), dealt to the waves
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    const int q = wave + 4 * n;
    if (q < 10) {
      const int ti = q < 1 ? 0 : (q < 3 ? 1 : (q < 6 ? 2 : 3));
      const int tj = q - ti * (ti + 1) / 2;
      gc_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc = gc_mma(gc_ld8(&sh.r1.kc[16 * ti + r16][32 * s + 8 * g4]),
                     gc_ld8(&sh.r1.kc[16 * tj + r16][32 * s + 8 * g4]), acc);
      const int i0 = 16 * ti + 4 * g4, jj = 16 * tj + r16;
      const float4 bt = *reinterpret_cast<const float4*>(&sh.btv[i0]);
      const float4 rk = *reinterpret_cast<const float4*>(&sh.rkv[i0]);
      const float4 gi = *reinterpret_cast<const float4*>(&sh.gcv[i0]);
      const float bta[4] = {bt.x, bt.y, bt.z, bt.w}, rka[4] = {rk.x, rk.y, rk.z, rk.w};
      const float gia[4] = {gi.x, gi.y, gi.z, gi.w};
      const float rkj = sh.rkv[jj], gj = sh.gcv[jj];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sh.r2.s.am[i0 + j][jj] = jj < i0 + j ? -bta[j] * (acc[j] * rka[j] * rkj) * __expf(gia[j] - gj) : 0.f;
    }
  }
}

// Wave 0: Tm; waves 1..3: their masked s q.k decay tiles, in registers.
template <class SM>
__device__ __forceinline__ void gc_solve(SM& sh, gc_f32x4 (&qk)[4], float qscale, int wave, int lane, int r16,
                                         int g4) {
  // ======== Tm = (I - A)^-1 (wave 0) | masked s q.k decay (waves 1..3) ========
  if (wave == 0) {
    // diagonal blocks: lane = 16 blk + column; rows broadcast from LDS per block
    {
      const int base = 16 * (lane >> 4), c = lane & 15;
      float col[16];
#pragma unroll
      for (int m = 0; m < 16; ++m) col[m] = sh.r2.s.am[base + m][base + c];
#pragma unroll
      for (int i = 1; i < 16; ++i) {
        float acc = 0.f;
#pragma unroll
        for (int m4 = 0; m4 < i; m4 += 4) {
          const float4 rowv = *reinterpret_cast<const float4*>(&sh.r2.s.am[base + i][base + m4]);
          const float rv[4] = {rowv.x, rowv.y, rowv.z, rowv.w};
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (m4 + u < i) acc = fmaf(rv[u], col[m4 + u], acc);
        }
        col[i] += acc;
      }
#pragma unroll
      for (int m = 0; m < 16; ++m) sh.r2.s.tf[base + m][base + c] = col[m] + (m == c ? 1.f : 0.f);
    }
    // off-diagonal blocks by block diagonals, T_ij = T_ii sum_{k=j}^{i-1} A_ik T_kj; the
    // blocks of one diagonal are independent (their product chains interleave) and are
    // stored together before the next diagonal reads them.  fp32 MFMA 16x16x4: in step
    // s lane group g carries k = 4s + g of the sum, and k = 4g + s of the T_ii product,
    // whose B operand is then the accumulator element s of the same lane.
    gc_off_diagonal<3>(sh.r2.s.am, sh.r2.s.tf, r16, g4);
    gc_off_diagonal<2>(sh.r2.s.am, sh.r2.s.tf, r16, g4);
    gc_off_diagonal<1>(sh.r2.s.am, sh.r2.s.tf, r16, g4);
  } else {
    // tiles (ti >= tj) of (q_i . k_j): wave 1 takes 0, 3, 6, 9; wave 2 1, 4, 7; wave 3 2, 5, 8
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int q = wave - 1 + 3 * n;
      qk[n] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
      if (q < 10) {
        const int ti = q < 1 ? 0 : (q < 3 ? 1 : (q < 6 ? 2 : 3));
        const int tj = q - ti * (ti + 1) / 2;
        gc_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
          acc = gc_mma(gc_ld8(&sh.qc[16 * ti + r16][32 * s + 8 * g4]),
                       gc_ld8(&sh.r1.kc[16 * tj + r16][32 * s + 8 * g4]), acc);
        const int i0 = 16 * ti + 4 * g4, jj = 16 * tj + r16;
        const float4 rq = *reinterpret_cast<const float4*>(&sh.rqv[i0]);
        const float4 gi = *reinterpret_cast<const float4*>(&sh.gcv[i0]);
        const float rqa[4] = {rq.x, rq.y, rq.z, rq.w}, gia[4] = {gi.x, gi.y, gi.z, gi.w};
        const float rkj = sh.rkv[jj], gj = sh.gcv[jj];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          qk[n][j] = jj <= i0 + j ? (acc[j] * rqa[j] * rkj) * qscale * __expf(gia[j] - gj) : 0.f;
      }
    }
  }
}

// The decay tiles to LDS as hi / lo (over k's rows, consumed).
template <class SM>
__device__ __forceinline__ void gc_store_decay(SM& sh, const gc_f32x4 (&qk)[4], int wave, int lane, int r16,
                                               int g4) {
  if (wave > 0) {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int q = wave - 1 + 3 * n;
      if (q < 10) {
        const int ti = q < 1 ? 0 : (q < 3 ? 1 : (q < 6 ? 2 : 3));
        const int tj = q - ti * (ti + 1) / 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const __bf16 hi = (__bf16)qk[n][j];
          sh.r1.in[0][16 * ti + 4 * g4 + j][16 * tj + r16] = gc_bits(hi);
          sh.r1.in[1][16 * ti + 4 * g4 + j][16 * tj + r16] = gc_bits((__bf16)(qk[n][j] - (float)hi));
        }
      }
    }
    // upper tiles (0, 1) and (2, 3) fall inside the 32-wide k steps of the O product
    if (wave == 1) {
      const int tr = lane < 32 ? 0 : 2, rr = (lane & 31) >> 1, half = lane & 1;
      const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        *reinterpret_cast<u32x4_t*>(&sh.r1.in[p][16 * tr + rr][16 * (tr + 1) + 8 * half]) = z;
      }
    }
  }
}

// Tm scaled two ways, hi / lo.
template <class SM>
__device__ __forceinline__ void gc_scale_tm(SM& sh, int tid) {
  // Tm diag(rk beta e^gc) and Tm diag(beta), hi / lo (thread = row, 16 columns)
  {
    const int i = tid >> 2, cb = tid & 3, c0 = 16 * cb;
    const bool live = cb <= (i >> 4);
    float tv[16];
#pragma unroll
    for (int c4 = 0; c4 < 16; c4 += 4) {
      const float4 f = live ? *reinterpret_cast<const float4*>(&sh.r2.s.tf[i][c0 + c4])
                            : make_float4(0.f, 0.f, 0.f, 0.f);
      tv[c4] = f.x; tv[c4 + 1] = f.y; tv[c4 + 2] = f.z; tv[c4 + 3] = f.w;
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const float* f = m == 0 ? sh.fwv : sh.btv;
#pragma unroll
      for (int c8 = 0; c8 < 16; c8 += 8) {
        const gc_f32x4 fa = *reinterpret_cast<const gc_f32x4*>(f + c0 + c8);
        const gc_f32x4 fb = *reinterpret_cast<const gc_f32x4*>(f + c0 + c8 + 4);
        gc_f32x4 p, q;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          p[j] = tv[c8 + j] * fa[j];
          q[j] = tv[c8 + 4 + j] * fb[j];
        }
        gc_bf16x8 hi, lo;
        gc_split(p, q, hi, lo);
        *reinterpret_cast<gc_bf16x8*>(&sh.r3.tm[2 * m][i][c0 + c8]) = hi;
        *reinterpret_cast<gc_bf16x8*>(&sh.r3.tm[2 * m + 1][i][c0 + c8]) = lo;
      }
    }
  }
}

}  // namespace lollm
