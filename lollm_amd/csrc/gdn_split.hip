// Chunked Gated DeltaNet prefill with the chunks of a head spread over the chip, gfx950: the
// layer of gdn_chunk.hip (same mathematics, arithmetic and state placement), for calls with
// few (sequence, head) pairs, which leave most CUs idle when one workgroup walks a head.
//
// Everything in a chunk but the state recurrence is independent of the other chunks.  Three
// kernels share the work:
//   gdn_split_prep   one workgroup per (sequence, v-head, chunk): conv, gating, A, Tm, the q.k
//                    decay; leaves W, U = Tm diag(beta) V, the decay, q and k^T in memory in
//                    MFMA-operand order (each later load is one coalesced 1 KB)
//   gdn_split_scan   one workgroup per (sequence, v-head, 16 or 32 value columns): the recurrence
//                    V' = U - W S,  O = diag(rq s e^gc) Q S + decay V',
//                    S <- e^gc_63 S + K^T diag(rk e^(gc_63 - gc)) V'
//                    -- 68 MFMAs per wave and chunk (32 columns) against ~1370 of the whole chunk
//   gdn_split_norm   gated RMSNorm of the core output, in place
// The scan is a chain of chunks, so its step is kept short: the four waves split the 64 tokens
// (16 each) for V' and O and the 128 keys (32 each) for the state update, every operand but S
// and V' comes straight from memory to registers one chunk ahead, S and V' pass through LDS
// as hi / lo bf16 with two barriers per chunk, and a wave keeps its part of S in fp32
// registers.
//
// What bounds it (1 x 1847 tokens, 32 heads: 543 us walked, 130 here): prep 67 us, 18 us per
// item at one workgroup per CU (149 KB of LDS) over 3.6 rounds, its barriers and the serial
// solve; the scan about 58 us, 2 us per chunk of dependent reads, products and barriers; the
// norm 9 us, bandwidth.
#include "gdn_chunk_common.h"

namespace lollm {

// Workspace of one (sequence, v-head, chunk) item and of one (sequence, qk-head, chunk) item.
constexpr int GS_W = 0;                    // -W hi, lo: [2][token block 4][key step 4][lane] 16 B
constexpr int GS_U = GS_W + 2 * 16384;     // U fp32: [column group 4][token block 4][tile 2][lane] 16 B
constexpr int GS_IN = GS_U + 32768;        // decay hi, lo: [2][token block 4][token step 2][lane] 16 B
constexpr int GS_SC = GS_IN + 16384;       // rq s e^gc (64), rk e^(gc_63 - gc) (64), e^gc_63
constexpr int GS_ITEM = GS_SC + 1024;
constexpr int GS_Q = 0;                    // q: [token block 4][key step 4][lane] 16 B
constexpr int GS_KT = 16384;               // k^T: [key block 8][token step 2][lane] 16 B
constexpr int GS_QK_ITEM = 2 * 16384;

struct GsSmem {
  union {
    uint16_t kc[GC_C][GC_PW];
    uint16_t in[2][GC_C][GC_PN];
  } r1;
  uint16_t kt[GL_DK][GC_PN];
  uint16_t qc[GC_C][GC_PW];
  uint16_t vt[GL_DK][GC_PN];
  struct {
    struct {
      float am[GC_C][GC_PF];
      float tf[GC_C][GC_PF];
    } s;
  } r2;
  struct {
    uint16_t tm[4][GC_C][GC_PN];
  } r3;
  float gcv[GC_C], egv[GC_C], btv[GC_C], rqv[GC_C], rkv[GC_C];
  float fwv[GC_C], f7v[GC_C];
  uint16_t cw[GL_CH][4];
};
static_assert(sizeof(GsSmem) <= 160 * 1024, "LDS budget");

struct GsArgs {
  GdnLayerArgs g;
  uint8_t* ws;      // items of the segment: (b, h, chunk)
  uint8_t* wsqk;    // (b, hk, chunk)
  int c0, nc;       // first chunk and chunks of the segment
};

__global__ __launch_bounds__(256) void gdn_split_prep_kernel(GsArgs s) {
  __shared__ GsSmem sh;
  const GdnLayerArgs& a = s.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int item = blockIdx.x, ci = item % s.nc, bh = item / s.nc;
  const int b = bh / a.Hv, h = bh % a.Hv;
  const int vpk = a.Hv / a.Hk, hk = h / vpk;
  const bool write_qk = (h % vpk) == 0;
  const int t0 = (s.c0 + ci) * GC_C;
  const int Km1 = a.K - 1;   // == 3 on this path
  int off = a.conv_off[b];
  off = off < 0 ? 0 : (off > 2 * a.W - Km1 ? 2 * a.W - Km1 : off);
  const int wbase = off >= a.W ? 0 : a.W;
  const size_t win_b = (size_t)b * 2 * a.W;
  const float a_log = a.A_log[h], dtb = a.dt_bias[h];

  // the raw rows of the conv items: from the projection through a descriptor over the
  // sequence's rows (past the call: zeros), the first chunk's 3 history rows from the window
  const uint16_t* projb = a.proj + (size_t)b * a.T * a.P;
  const uint32_t P2 = (uint32_t)a.P * 2u;
  const __amdgpu_buffer_rsrc_t prs = buf_rsrc(projb, (uint32_t)a.T * P2);
  u32x4_t raw[GC_ITEMS][7];
#pragma unroll
  for (int n = 0; n < GC_ITEMS; ++n) {
    const int c0n = gc_chan(a, hk, h, 8 * ((tid + 256 * n) % 48)), t4 = 4 * ((tid + 256 * n) / 48);
#pragma unroll
    for (int r = 0; r < 7; ++r) {
      const int t = t0 + t4 - 3 + r;
      raw[n][r] = gc_bload(prs, (uint32_t)max(t, 0) * P2 + 2u * (uint32_t)c0n);
      if (t < 0) raw[n][r] = *reinterpret_cast<const u32x4_t*>(a.win + (win_b + off + 3 + t) * a.C + c0n);
    }
  }
  const uint32_t boff = (uint32_t)(t0 + lane) * P2 + 2u * (uint32_t)(a.C + a.value_dim + h);
  const uint16_t braw = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(prs, boff, 0, 0);
  const uint16_t araw = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(prs, boff + 2u * a.Hv, 0, 0);
  if (tid < GL_CH / 2)
    *reinterpret_cast<u32x4_t*>(&sh.cw[2 * tid][0]) =
        *reinterpret_cast<const u32x4_t*>(a.conv_w + (size_t)gc_chan(a, hk, h, 2 * tid) * 4);
  __syncthreads();
  gc_conv_gating(sh, raw, braw, araw, a_log, dtb, t0, a.T, tid, wave, lane);
  __syncthreads();
  uint8_t* ws = s.ws + (size_t)item * GS_ITEM;
  if (write_qk) {
    uint8_t* wq = s.wsqk + ((size_t)(b * a.Hk + hk) * s.nc + ci) * GS_QK_ITEM;
#pragma unroll
    for (int n = 0; n < 4; ++n) {   // wave w: token block w of q, key blocks 2 w, 2 w + 1 of k^T
      *reinterpret_cast<u32x4_t*>(wq + GS_Q + ((wave * 4 + n) * 64 + lane) * 16) =
          *reinterpret_cast<const u32x4_t*>(&sh.qc[16 * wave + r16][32 * n + 8 * g4]);
      *reinterpret_cast<u32x4_t*>(wq + GS_KT + ((wave * 4 + n) * 64 + lane) * 16) =
          *reinterpret_cast<const u32x4_t*>(&sh.kt[32 * wave + 16 * (n >> 1) + r16][32 * (n & 1) + 8 * g4]);
    }
  }
  gc_form_a(sh, tid, wave, r16, g4);
  __syncthreads();
  gc_f32x4 qk[4];
  const float qscale = rsqrtf((float)GL_DK);
  gc_solve(sh, qk, qscale, wave, lane, r16, g4);
  __syncthreads();   // A, k (row layout) consumed; Tm complete
  gc_store_decay(sh, qk, wave, lane, r16, g4);
  gc_scale_tm(sh, tid);
  if (tid < GC_C) {
    float* sc = reinterpret_cast<float*>(ws + GS_SC);
    sc[tid] = sh.rqv[tid] * qscale * sh.egv[tid];
    sc[GC_C + tid] = sh.f7v[tid];
    if (tid == GC_C - 1) sc[2 * GC_C] = sh.egv[tid];
  }
  __syncthreads();
  // the decay: wave w copies token block w (token steps past the diagonal are never read)
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
      if (s2 <= (wave >> 1))
        *reinterpret_cast<u32x4_t*>(ws + GS_IN + (((p * 4 + wave) * 2 + s2) * 64 + lane) * 16) =
            *reinterpret_cast<const u32x4_t*>(&sh.r1.in[p][16 * wave + r16][32 * s2 + 8 * g4]);
  // -W^T = -K^T (Tm diag(rk beta e^gc))^T: wave w keys 32 w .. 32 w + 31, all tokens
  {
    gc_f32x4 acc[2][4];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) acc[c][ib] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int k2 = 0; k2 <= (ib >> 1); ++k2) {
        const gc_bf16x8 bh = gc_ld8(&sh.r3.tm[0][16 * ib + r16][32 * k2 + 8 * g4]);
        const gc_bf16x8 bl = gc_ld8(&sh.r3.tm[1][16 * ib + r16][32 * k2 + 8 * g4]);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const gc_bf16x8 av = gc_ld8(&sh.kt[32 * wave + 16 * c + r16][32 * k2 + 8 * g4]);
          acc[c][ib] = gc_mma(av, bh, acc[c][ib]);
          acc[c][ib] = gc_mma(av, bl, acc[c][ib]);
        }
      }
    // keys 32 w + 16 c + 4 g4 + j of token 16 ib + r16: operand lane 16 (2 c + g4 / 2) + r16 of
    // key step w, its half g4 % 2
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        uint16_t hb[4], lb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = -acc[c][ib][j];
          const __bf16 hi = (__bf16)x;
          hb[j] = gc_bits(hi);
          lb[j] = gc_bits((__bf16)(x - (float)hi));
        }
        uint8_t* dst = ws + GS_W + ((ib * 4 + wave) * 64 + 16 * (2 * c + (g4 >> 1)) + r16) * 16 + 8 * (g4 & 1);
        *reinterpret_cast<uint2*>(dst) =
            make_uint2(hb[0] | ((uint32_t)hb[1] << 16), hb[2] | ((uint32_t)hb[3] << 16));
        *reinterpret_cast<uint2*>(dst + 16384) =
            make_uint2(lb[0] | ((uint32_t)lb[1] << 16), lb[2] | ((uint32_t)lb[3] << 16));
      }
  }
  // U = Tm diag(beta) V: wave w value columns 32 w .. 32 w + 31, all tokens
  {
    gc_bf16x8 vb[2][2];
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int u = 0; u < 2; ++u) vb[k2][u] = gc_ld8(&sh.vt[32 * wave + 16 * u + r16][32 * k2 + 8 * g4]);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      gc_f32x4 un[2] = {gc_f32x4{0.f, 0.f, 0.f, 0.f}, gc_f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int k2 = 0; k2 <= (tb >> 1); ++k2) {
        const gc_bf16x8 ah = gc_ld8(&sh.r3.tm[2][16 * tb + r16][32 * k2 + 8 * g4]);
        const gc_bf16x8 al = gc_ld8(&sh.r3.tm[3][16 * tb + r16][32 * k2 + 8 * g4]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          un[u] = gc_mma(ah, vb[k2][u], un[u]);
          un[u] = gc_mma(al, vb[k2][u], un[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
        *reinterpret_cast<gc_f32x4*>(ws + GS_U + (((wave * 4 + tb) * 2 + u) * 64 + lane) * 16) = un[u];
    }
  }
  // the call's last K-1 raw inputs to the window half being written
  if (t0 + GC_C >= a.T)
    for (int i = tid; i < Km1 * GL_CH; i += 256) {
      const int r = i / GL_CH, lc = i % GL_CH;
      if (lc >= 2 * GL_DK || write_qk) {
        const int c = gc_chan(a, hk, h, lc);
        a.win[(win_b + wbase + r) * a.C + c] = a.proj[((size_t)b * a.T + a.T - Km1 + r) * a.P + c];
      }
    }
}

// NU 16-column tiles per workgroup.
template <int NU>
__global__ __launch_bounds__(256, 2) void gdn_split_scan_kernel(GsArgs s, int heads) {
  constexpr int GS_COLS = 16 * NU, GROUPS = GL_DK / GS_COLS;
  __shared__ uint16_t sS[2][GS_COLS][GC_PW];   // S hi, lo [column][key]
  __shared__ uint16_t sV[4][GS_COLS][GC_PN];   // V' hi, lo, diag(rk e^..) V' hi, lo [column][token]
  const GdnLayerArgs& a = s.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  // the column groups of a head on one XCD (its L2 then serves all but the first of their
  // reads of W, q, k^T and the decay)
  const int i = blockIdx.x;
  const int bh = heads % 8 == 0 ? (i / (8 * GROUPS)) * 8 + i % 8 : i / GROUPS;
  const int cg = heads % 8 == 0 ? (i / 8) % GROUPS : i % GROUPS;
  const int b = bh / a.Hv, h = bh % a.Hv, hk = h / (a.Hv / a.Hk);
  constexpr size_t SS = (size_t)GL_DK * GL_DK;
  float* st_io = a.rec + ((size_t)(b * 2 + ((a.rec_half[b] & 1) ^ 1)) * a.Hv + h) * SS;
  const uint8_t* ws = s.ws + (size_t)bh * s.nc * GS_ITEM;
  const uint8_t* wq = s.wsqk + (size_t)(b * a.Hk + hk) * s.nc * GS_QK_ITEM;

  gc_f32x4 st[2][NU];   // keys 32 w + 16 c + 4 g4 + j, column 32 cg + 16 u + r16
  const bool zero = a.fresh && s.c0 == 0;
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = st_io[(size_t)(32 * wave + 16 * c + 4 * g4 + j) * GL_DK + GS_COLS * cg + 16 * u + r16];
        st[c][u][j] = zero ? 0.f : x;
      }
  // four values as hi / lo bf16, 8 bytes each
  auto split4 = [](gc_f32x4 x, uint16_t* hi, uint16_t* lo) {
    uint16_t hb[4], lb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const __bf16 t = (__bf16)x[j];
      hb[j] = gc_bits(t);
      lb[j] = gc_bits((__bf16)(x[j] - (float)t));
    }
    *reinterpret_cast<uint2*>(hi) = make_uint2(hb[0] | ((uint32_t)hb[1] << 16), hb[2] | ((uint32_t)hb[3] << 16));
    *reinterpret_cast<uint2*>(lo) = make_uint2(lb[0] | ((uint32_t)lb[1] << 16), lb[2] | ((uint32_t)lb[3] << 16));
  };
  auto put_state = [&]() {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int u = 0; u < NU; ++u)
        split4(st[c][u], &sS[0][16 * u + r16][32 * wave + 16 * c + 4 * g4],
               &sS[1][16 * u + r16][32 * wave + 16 * c + 4 * g4]);
  };
  put_state();

  // operands of a chunk, loaded one chunk before their use (two made no difference)
  struct {   // W, U, q and the scale of V'
    gc_bf16x8 wh[4], wl[4], qr[4];
    gc_f32x4 un[NU], f7;
  } f;
  struct {   // k^T, the decay, the scales of O and S
    gc_bf16x8 kr[2][2], ih[2], il[2];
    gc_f32x4 rs;
    float eg;
  } g;
  auto load_first = [&](int c) {
    const uint8_t* w = ws + (size_t)c * GS_ITEM;
    const uint8_t* q = wq + (size_t)c * GS_QK_ITEM;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f.wh[k] = gc_ld8((const uint16_t*)(w + GS_W + ((wave * 4 + k) * 64 + lane) * 16));
      f.wl[k] = gc_ld8((const uint16_t*)(w + GS_W + 16384 + ((wave * 4 + k) * 64 + lane) * 16));
      f.qr[k] = gc_ld8((const uint16_t*)(q + GS_Q + ((wave * 4 + k) * 64 + lane) * 16));
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
      f.un[u] = *reinterpret_cast<const gc_f32x4*>(w + GS_U + (((cg * NU / 2 * 4 + wave) * 2 + (cg * NU + u) % 2) * 64 + lane) * 16);
    f.f7 = *reinterpret_cast<const gc_f32x4*>(w + GS_SC + 4 * (GC_C + 16 * wave + 4 * g4));
  };
  auto load_second = [&](int c) {
    const uint8_t* w = ws + (size_t)c * GS_ITEM;
    const uint8_t* q = wq + (size_t)c * GS_QK_ITEM;
#pragma unroll
    for (int n = 0; n < 4; ++n)
      g.kr[n >> 1][n & 1] = gc_ld8((const uint16_t*)(q + GS_KT + ((wave * 4 + n) * 64 + lane) * 16));
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {   // (the step past the diagonal of waves 0 and 1 is not used)
      const int k2 = s2 <= (wave >> 1) ? s2 : 0;
      g.ih[s2] = gc_ld8((const uint16_t*)(w + GS_IN + ((wave * 2 + k2) * 64 + lane) * 16));
      g.il[s2] = gc_ld8((const uint16_t*)(w + GS_IN + (((4 + wave) * 2 + k2) * 64 + lane) * 16));
    }
    g.rs = *reinterpret_cast<const gc_f32x4*>(w + GS_SC + 4 * (16 * wave + 4 * g4));
    g.eg = *reinterpret_cast<const float*>(w + GS_SC + 4 * 2 * GC_C);
  };
  load_first(0);
  load_second(0);

  uint16_t* outp = a.out + (size_t)b * a.T * a.value_dim + (size_t)h * GL_DK + GS_COLS * cg + r16;
  for (int c = 0; c < s.nc; ++c) {
    const int cn = min(c + 1, s.nc - 1);
    lds_only_barrier();   // S of this chunk written (and V' of the last one read)
    gc_f32x4 vn[3][NU], ov[2][NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      vn[0][u] = f.un[u];
      vn[1][u] = vn[2][u] = ov[0][u] = ov[1][u] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const gc_bf16x8 sh = gc_ld8(&sS[0][16 * u + r16][32 * k + 8 * g4]);
        const gc_bf16x8 sl = gc_ld8(&sS[1][16 * u + r16][32 * k + 8 * g4]);
        vn[0][u] = gc_mma(f.wh[k], sh, vn[0][u]);
        vn[1][u] = gc_mma(f.wh[k], sl, vn[1][u]);
        vn[2][u] = gc_mma(f.wl[k], sh, vn[2][u]);
        ov[0][u] = gc_mma(f.qr[k], sh, ov[0][u]);
        ov[1][u] = gc_mma(f.qr[k], sl, ov[1][u]);
      }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const gc_f32x4 v = vn[0][u] + (vn[1][u] + vn[2][u]);
      const int col = 16 * u + r16, tok = 16 * wave + 4 * g4;
      split4(v, &sV[0][col][tok], &sV[1][col][tok]);
      split4(v * f.f7, &sV[2][col][tok], &sV[3][col][tok]);
    }
    load_first(cn);
    lds_only_barrier();   // V' written; every wave is done with S
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int u = 0; u < NU; ++u) st[cc][u] *= g.eg;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const gc_bf16x8 qh = gc_ld8(&sV[2][16 * u + r16][32 * s2 + 8 * g4]);
        const gc_bf16x8 ql = gc_ld8(&sV[3][16 * u + r16][32 * s2 + 8 * g4]);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
          st[cc][u] = gc_mma(g.kr[cc][s2], qh, st[cc][u]);
          st[cc][u] = gc_mma(g.kr[cc][s2], ql, st[cc][u]);
        }
      }
    put_state();
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      ov[0][u] = (ov[0][u] + ov[1][u]) * g.rs;
      ov[1][u] = gc_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
      if (s2 <= (wave >> 1)) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const gc_bf16x8 vh = gc_ld8(&sV[0][16 * u + r16][32 * s2 + 8 * g4]);
          const gc_bf16x8 vl = gc_ld8(&sV[1][16 * u + r16][32 * s2 + 8 * g4]);
          ov[0][u] = gc_mma(g.ih[s2], vh, ov[0][u]);
          ov[1][u] = gc_mma(g.ih[s2], vl, ov[1][u]);
          ov[0][u] = gc_mma(g.il[s2], vh, ov[0][u]);
        }
      }
    load_second(cn);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = (s.c0 + c) * GC_C + 16 * wave + 4 * g4 + j;
      if (t < a.T) {
#pragma unroll
        for (int u = 0; u < NU; ++u)
          outp[(size_t)t * a.value_dim + 16 * u] = gc_bits((__bf16)(ov[0][u][j] + ov[1][u][j]));
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        st_io[(size_t)(32 * wave + 16 * c + 4 * g4 + j) * GL_DK + GS_COLS * cg + 16 * u + r16] = st[c][u][j];
}

// Gated RMSNorm of the core output in place: 16 lanes per (token, head), 8 columns each.
__global__ __launch_bounds__(256) void gdn_split_norm_kernel(GdnLayerArgs a) {
  const size_t bt = blockIdx.x;
  const int h = blockIdx.y * 16 + (threadIdx.x >> 4), part = threadIdx.x & 15;
  if (h >= a.Hv) return;   // whole 16-lane rows
  uint16_t* op = a.out + bt * a.value_dim + (size_t)h * GL_DK + part * 8;
  const u32x4_t ov = *reinterpret_cast<const u32x4_t*>(op);
  const u32x4_t zd = *reinterpret_cast<const u32x4_t*>(a.proj + bt * a.P + a.C + h * GL_DK + part * 8);
  const u32x4_t nw = *reinterpret_cast<const u32x4_t*>(a.norm_w + part * 8);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t w = ov[e];   // (a bit cast straight from a vector element reads element 0)
    const gc_bf16x2 p = __builtin_bit_cast(gc_bf16x2, w);
    ss = __builtin_amdgcn_fdot2_f32_bf16(p, p, ss, false);
  }
  ss = gc_row16_sum(ss);
  const float rr = rsqrtf(ss / (float)GL_DK + a.eps);
  u32x4_t od;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float y2[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float o = __uint_as_float(u ? ov[e] & 0xffff0000u : ov[e] << 16);
      const float z = __uint_as_float(u ? zd[e] & 0xffff0000u : zd[e] << 16);
      const float w = __uint_as_float(u ? nw[e] & 0xffff0000u : nw[e] << 16);
      y2[u] = gc_rbf(w * gc_rbf(o * rr)) * silu_g(z);
    }
    od[e] = gc_pack(y2[0], y2[1]);
  }
  *reinterpret_cast<u32x4_t*>(op) = od;
}

// Chunks per segment: the workspace holds one segment's items, at most GS_MAX_ITEMS unless one
// chunk of every head is more (a prompt of any length then needs the same memory).
constexpr long long GS_MAX_ITEMS = 4096;
static int gs_segment(int B, int T, int Hv) {
  const int nch = (T + GC_C - 1) / GC_C;
  long long seg = GS_MAX_ITEMS / ((long long)B * Hv);
  seg = seg < 1 ? 1 : (seg > nch ? nch : seg);
  const int n = (int)((nch + seg - 1) / seg);
  return (nch + n - 1) / n;   // even segments
}

}  // namespace lollm

using namespace lollm;

LOLLM_API long long lollm_gdn_split_workspace_bytes(int B, int T, int Hk, int Hv) {
  if (B <= 0 || T <= 0 || Hk <= 0 || Hv <= 0 || Hv % Hk) return -1;
  const long long seg = gs_segment(B, T, Hv);
  return B * seg * ((long long)Hv * GS_ITEM + (long long)Hk * GS_QK_ITEM);
}

LOLLM_API int lollm_gdn_layer_split(const void* proj, long long proj_stride, const void* conv_w,
                                    const float* A_log, const float* dt_bias, const void* norm_w,
                                    void* win, const int32_t* conv_off, int win_rows, float* rec,
                                    const int32_t* rec_half, void* rep, const int32_t* replay,
                                    int slots, int fresh, void* out, void* workspace,
                                    long long workspace_bytes, int B, int T, int Hk, int Hv, int Dk,
                                    int Dv, int conv_kernel, float eps, void* stream) {
  GsArgs s;
  if (!workspace || workspace_bytes < lollm_gdn_split_workspace_bytes(B, T, Hk, Hv)) return LOLLM_EINVAL;
  int rc = gdn_long_call_args(s.g, proj, proj_stride, conv_w, A_log, dt_bias, norm_w, win, conv_off, win_rows, rec,
                              rec_half, rep, replay, slots, fresh, out, B, T, Hk, Hv, Dk, Dv, conv_kernel, eps);
  if (rc != LOLLM_OK) return rc;
  const hipStream_t st = (hipStream_t)stream;
  if ((rc = gdn_long_call_prologue(s.g, B, st)) != LOLLM_OK) return rc;
  const int nch = (T + GC_C - 1) / GC_C, seg = gs_segment(B, T, Hv), heads = B * Hv;
  s.ws = (uint8_t*)workspace;
  s.wsqk = s.ws + (size_t)heads * seg * GS_ITEM;
  for (s.c0 = 0; s.c0 < nch; s.c0 += seg) {
    s.nc = nch - s.c0 < seg ? nch - s.c0 : seg;
    hipLaunchKernelGGL(gdn_split_prep_kernel, dim3(heads * s.nc), dim3(256), 0, st, s);
    if ((rc = launch_status())) return rc;
    // 16 columns a workgroup where that is still one workgroup per CU (us of the call, 16 / 32
    // columns: 32 heads x 29 chunks 130 / 145, 16 heads 92 / 107; 64 heads x 24 171 / 170, 96
    // heads 290 / 273, where the repeated reads of W, q and k^T cost more than the shorter step
    // gives)
    if (heads <= 32)
      hipLaunchKernelGGL(gdn_split_scan_kernel<1>, dim3(heads * 8), dim3(256), 0, st, s, heads);
    else
      hipLaunchKernelGGL(gdn_split_scan_kernel<2>, dim3(heads * 4), dim3(256), 0, st, s, heads);
    if ((rc = launch_status())) return rc;
  }
  hipLaunchKernelGGL(gdn_split_norm_kernel, dim3(B * T, (Hv + 15) / 16), dim3(256), 0, st, s.g);
  return launch_status();
}
