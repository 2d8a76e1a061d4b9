// Gated GQA attention of a long call (prefill: many new positions per sequence), gfx950.
//
// Same math and operands as attn_verify.hip (src/qwen3_5/blocks.py:226-235 +
// src/attention.py:43-51: offset-causal GQA over the cache, output o * sigmoid(gate)),
// for calls whose query rows alone fill the chip, where splitting keys between workgroups
// (and the fp32 pieces and the second launch that go with it) buys nothing.
//
// Tile.  A workgroup owns 128 RG query rows of one (sequence, KV head): the n_rep query
// heads x QB consecutive positions, packed position-major (row r = position r / n_rep,
// head r % n_rep), so every K / V byte staged serves all the heads that share it and a
// tile's causal edge is only QB positions wide.  It walks the keys in blocks of 32: K and
// V rows arrive by LDS DMA (three sets each, K three and V two blocks ahead, one barrier
// per block) and are read by all four waves; wave w owns rows 32 RG w .. of the tile with
// its Q in registers and its O^T in accumulator registers.
//
// Precision.  One running maximum serves a row where the split-K kernels have one per wave and
// piece, whose largest weights are 1 and lose nothing as bf16; so weights enter the product with
// V as hi + lo bf16 (16 bits) and the row sum as they are, fp32.  Relative error against 64 bits
// (2 x 1999 tokens, normal q, k, v): split-K 2.07e-3, weights in bf16 here 2.12e-3, hi + lo
// 1.66e-3, which is the output's own rounding to bf16.  It costs a third of the products: 185 ->
// 221 us.
//
// What bounds it: operand reads and the softmax beside the products.  A 32x32x16 MFMA
// (32 cycles) takes a 1 KB operand from LDS, and the four waves of a CU then need 128 B per
// cycle, the LDS peak.  With RG = 2 a wave reuses each K / V operand for two row groups and
// needs half of that, at one wave per SIMD: O^T of 64 rows takes all 256 accumulator
// registers, Q half of the vector registers.  A lone wave overlaps nothing by itself, so the
// exponentials of block j + 1 are placed between the products of V with block j.
//
// Measured (us, causal, T = kv length, split-K kernels / RG = 1 / RG = 2): 2 x 1999,
// 32 q / 4 kv heads 1020 / 247 / 222 (591 TFLOP/s); 1 x 4096 1822 / 407 / 372 (740 TFLOP/s);
// 3 x 1500 1110 / 216 / 217; 32 x 128 over 1128 keys 903 / 260 / 244.
//
// Rows of K and V are 512 bytes in LDS with no padding (the DMA writes 1 KB runs); the
// 16-byte chunk c of row r sits at c ^ (r & 15) for K and c ^ (2 (r & 7)) for V, so the
// operand reads (32 rows at one chunk; 8 rows x 4 chunks for the transposing V read) touch
// every bank equally.
#include "attn_common.h"

namespace lollm {

constexpr int AP_WAVES = 4;
constexpr int AP_MIN_T = 16;                   // new positions per sequence
constexpr int AP_FEW_ROWS = 64;                // tokens of a call that keeps the split-K kernels
constexpr int AP_KEYS = 32;                    // keys per block
constexpr int AP_AHEAD = 3;                    // operands read ahead of their products
constexpr int AP_SET = AP_KEYS * AT_D * 2;     // 16 KB: K or V rows of a block

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct ApArgs {
  const uint16_t* q;       // (B, T, Hq, D)
  const uint16_t* kc;      // K cache
  const uint16_t* vc;      // V cache
  const int32_t* kv_len;   // (B) keys per sequence, the T new ones included
  const uint16_t* gate;    // (B, T, Hq * D) or null
  uint16_t* out;           // (B, T, Hq * D)
  long long seq_stride, head_stride;
  int B, T, Hq, Hkv, n_rep, QB, qtiles, max_len;
  uint32_t rep_mul;        // ceil(2^16 / n_rep): r / n_rep = r * rep_mul >> 16 for r < 256
  float cl2;
};

// S += K Q^T with S in vector registers.  O of 64 rows takes all 256 accumulator registers,
// and the compiler, which gives every MFMA of a kernel one register class, would move parts of
// O out and back for each S.  (The nop: a VALU write may precede; the matrix pipe is busy for
// longer than that with the previous product.)
__device__ __forceinline__ void ap_mfma_first(f32x16& s, bf16x8 k, bf16x8 q) {
  asm("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "v"(q));
}
__device__ __forceinline__ void ap_mfma(f32x16& s, bf16x8 k, bf16x8 q) {
  asm("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "v"(q));
}
// the wait states between the last product and the first VALU access of its result
__device__ __forceinline__ void ap_mfma_done(f32x16& s) { asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s)); }

// A pair of fp32 weights as bf16 hi and lo, x = hi + lo to 16 bits.  hi is cut and not rounded, so
// that lo is never negative, and lo is at least 2^-126 where hi is not 0: an infinite V then takes
// the sum of both products to infinity as a single product does, not to infinity - infinity or
// 0 x infinity.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void ap_split(float x, float y, uint32_t& hi, uint32_t& lo) {
  const uint32_t xb = __float_as_uint(x), yb = __float_as_uint(y);
  hi = __builtin_amdgcn_perm(yb, xb, 0x07060302u);   // the upper halves
  const bf16x2 l = {(__bf16)(x - __uint_as_float(xb & 0xffff0000u)), (__bf16)(y - __uint_as_float(yb & 0xffff0000u))};
  const u16x2 least = __builtin_elementwise_min(__builtin_bit_cast(u16x2, hi), u16x2{0x0080, 0x0080});
  lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, l), least));
}
__device__ __forceinline__ int ap_div(int r, uint32_t mul) { return (int)(((uint32_t)r * mul) >> 16); }

template <int RG>
__global__ __launch_bounds__(64 * AP_WAVES, 1) void attn_prefill_kernel(ApArgs a) {
  // separate arrays, so that the reads of one set are not ordered after the DMA into another
  __shared__ __attribute__((aligned(16))) unsigned char ks0[AP_SET], ks1[AP_SET], ks2[AP_SET];
  __shared__ __attribute__((aligned(16))) unsigned char vs0[AP_SET], vs1[AP_SET], vs2[AP_SET];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  // the longest tiles first (they end last), (sequence, KV head) fastest: with a multiple of
  // 8 pairs, one pair's tiles all run on one XCD and share its L2
  const int pairs = a.B * a.Hkv;
  const int qt = a.qtiles - 1 - blockIdx.x / pairs, pair = blockIdx.x % pairs;
  const int b = pair / a.Hkv, kvh = pair % a.Hkv;
  const int q0 = qt * a.QB, QB = min(a.QB, a.T - q0);
  const int L = min(max(a.kv_len[b], 0), a.max_len);
  const int p0 = L - a.T + q0;                       // position of the tile's first query
  const int keys = min(max(p0 + QB, 0), L);          // keys any row of the tile sees
  const int nblk = (keys + AP_KEYS - 1) / AP_KEYS;

  // Loads of a block: wave w brings rows 8 w .. 8 w + 7 of K and of V, two rows (1 KB) per
  // instruction; the lane's source chunk undoes the swizzle of the place it writes.  Rows
  // past the sequence's end touch no memory.
  constexpr int WR = AP_KEYS / AP_WAVES;
  static_assert(WR == 8, "the swizzles below take the row of the wave's 8");
  const size_t cbase = (size_t)b * a.seq_stride + (size_t)kvh * a.head_stride;
  const __amdgpu_buffer_rsrc_t krs = buf_rsrc(a.kc + cbase, (uint32_t)L * (AT_D * 2));
  const __amdgpu_buffer_rsrc_t vrs = buf_rsrc(a.vc + cbase, (uint32_t)L * (AT_D * 2));
  // (row = 8 w + 2 i + h: its swizzle is the lane's part ^ that of 2 i; one register per cache,
  // the rest formed per load -- registers are what this kernel is short of)
  const uint32_t rl = (uint32_t)(WR * wave + h) * (AT_D * 2);
  const uint32_t kl = 16u * (l32 ^ (8 * (wave & 1) + h)), vl = 16u * (l32 ^ (2 * h));
  auto issue_k = [&](unsigned char* kd, int j) {
    uint32_t x = kl;
    asm volatile("" : "+v"(x));
    const uint32_t blk = (uint32_t)(j * AP_KEYS) * (AT_D * 2) + rl;
#pragma unroll
    for (int i = 0; i < WR / 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lds_void_t*)(kd + 512 * WR * wave + 1024 * i), 16,
                                               blk + 1024u * i + (x ^ (32u * i)), 0, 0, 0);
  };
  auto issue_v = [&](unsigned char* vd, int j) {
    uint32_t x = vl;
    asm volatile("" : "+v"(x));
    const uint32_t blk = (uint32_t)(j * AP_KEYS) * (AT_D * 2) + rl;
#pragma unroll
    for (int i = 0; i < WR / 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lds_void_t*)(vd + 512 * WR * wave + 1024 * i), 16,
                                               blk + 1024u * i + (x ^ (64u * i)), 0, 0, 0);
  };
  // this wave's loads up to the last N have landed and its LDS accesses are complete, then
  // every wave's
#define AP_BARRIER(N) asm volatile("s_waitcnt vmcnt(" #N ") lgkmcnt(0)\n\ts_barrier" ::: "memory")

  // Finite contents everywhere: rows past a sequence's end are never loaded, and P = 0
  // multiplies what they hold.
  for (int i = tid; i < AP_SET / 16; i += 64 * AP_WAVES) {
    *reinterpret_cast<uint4*>(vs0 + 16 * i) = make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(vs1 + 16 * i) = make_uint4(0, 0, 0, 0);
    *reinterpret_cast<uint4*>(vs2 + 16 * i) = make_uint4(0, 0, 0, 0);
  }
  // this lane's rows: position q0 + qi, query head kvh n_rep + hr
  int qpos[RG];
  bf16x8 Q[RG][16];
#pragma unroll
  for (int rg = 0; rg < RG; ++rg) {
    const int r = 32 * (RG * wave + rg) + l32, qi = ap_div(r, a.rep_mul), hr = r - qi * a.n_rep;
    const bool live = qi < QB;
    qpos[rg] = live ? p0 + qi : -1;
    const uint16_t* src = a.q + (((size_t)b * a.T + q0 + (live ? qi : 0)) * a.Hq + kvh * a.n_rep + hr) * AT_D + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks)
      Q[rg][ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4_t*>(src + 16 * ks));
  }
  AP_BARRIER(0);   // the zeroed sets, before any DMA into them (and Q: the counts below are the DMA's)
  issue_k(ks0, 0);
  issue_k(ks1, 1);
  issue_v(vs0, 0);
  issue_k(ks2, 2);
  issue_v(vs1, 1);

  // the positions this wave's rows span: the key blocks it sees, and which need a mask
  const int wq0 = ap_div(32 * RG * wave, a.rep_mul);
  const int wq1 = min(ap_div(32 * RG * wave + 32 * RG - 1, a.rep_mul), QB - 1);
  const int wmin = p0 + wq0, wmax = wq0 < QB ? p0 + wq1 : -1;
  const int wblk = wmax < 0 ? 0 : wmax / AP_KEYS + 1;

  // LDS offsets of the operand reads: K row l32 at chunk 2 ks + h, V row x = 4 h + (lane % 16) / 4
  // at chunk 4 dt + 2 ((lane / 16) % 2) + (lane % 4) / 2; the k-step and the column tile
  // enter by xor
  const int ko = l32 * (AT_D * 2) + 16 * (h ^ (l32 & 15));
  const int vxr = 4 * h + ((lane & 15) >> 2);
  const int vo = vxr * (AT_D * 2) + 16 * ((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ (2 * vxr)) + 8 * (lane & 1);

  f32x16 O[RG][8];   // O^T: 32 columns x 32 rows per tile; lane's row = l32
  float m_ref[RG], l_s[RG];
  bf16x8 P[RG][2], Pl[RG][2];   // exp of the block whose V comes next, hi and lo
#pragma unroll
  for (int rg = 0; rg < RG; ++rg) {
    m_ref[rg] = -INFINITY;
    l_s[rg] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[rg][dt][r] = 0.f;
  }

  f32x16 S[RG];
  float base[RG], alpha[RG];
  bool moved;
  // S^T (32 keys x 32 rows) = K Q^T of block j, masked, and the row maxima
  auto scores = [&](const unsigned char* kset, int j) {
    int kof = ko;
    asm volatile("" : "+v"(kof));
    bf16x8 kf[AP_AHEAD];
#pragma unroll
    for (int i = 0; i < AP_AHEAD; ++i)
      kf[i] = *reinterpret_cast<const bf16x8*>(kset + (kof ^ (32 * (i & 7))) + 256 * (i >> 3));
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
        if (ks == 0) ap_mfma_first(S[rg], kf[0], Q[rg][0]); else ap_mfma(S[rg], kf[ks % AP_AHEAD], Q[rg][ks]);
      const int kn = ks + AP_AHEAD;
      if (kn < 16)
        kf[ks % AP_AHEAD] = *reinterpret_cast<const bf16x8*>(kset + (kof ^ (32 * (kn & 7))) + 256 * (kn >> 3));
      __builtin_amdgcn_sched_barrier(0);   // no more operands ahead than the registers hold
    }
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) ap_mfma_done(S[rg]);
    const int key0 = j * AP_KEYS;
    if (key0 + AP_KEYS - 1 > wmin) {   // acc r holds key 8 (r / 4) + 4 h + r % 4 of the block
#pragma unroll
      for (int rg = 0; rg < RG; ++rg) {
        const int lim = qpos[rg] - key0 - 4 * h;
#pragma unroll
        for (int r = 0; r < 16; ++r) S[rg][r] = 8 * (r >> 2) + (r & 3) <= lim ? S[rg][r] : -INFINITY;
      }
    }
    bool any = false;
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
      float bm = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) bm = fmaxf(bm, S[rg][r]);
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(bm), __float_as_uint(bm), false, false);
      bm = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      // the reference max moves (and l, O are rescaled) only when a row's block max exceeds it
      // by more than 16 in the exponent: attn_verify's rule, each row's own decision
      const bool big = (bm - m_ref[rg]) * a.cl2 > 16.f;
      const float mn = big ? fmaxf(m_ref[rg], bm) : m_ref[rg];
      alpha[rg] = (!big || mn == -INFINITY) ? 1.f : fast_exp2((m_ref[rg] - mn) * a.cl2);
      m_ref[rg] = mn;
      l_s[rg] *= alpha[rg];
      base[rg] = mn == -INFINITY ? 0.f : mn * a.cl2;
      any = any || big;
    }
    moved = __builtin_amdgcn_readfirstlane((int)(__ballot(any) != 0)) != 0;
  };
  auto rescale = [&]() {
    if (moved) {
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          // (O stays in accumulator registers but for the tile at hand: without the pins the
          // compiler copies all of it to vector registers around this branch)
          asm volatile("" : "+a"(O[rg][dt]));
          O[rg][dt] *= alpha[rg];
          asm volatile("" : "+a"(O[rg][dt]));
          __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) asm volatile("" : "+a"(O[rg][dt]));
  };
  // One block: scores of block j + 1, then O^T += V^T P^T of block j with the exponentials of
  // block j + 1 between its products (the matrix pipe is busy 32 cycles per product, the
  // wave's VALU work of one product about as long).  Past the wave's last block the scores
  // are all masked.
  auto step = [&](const unsigned char* knext, const unsigned char* vset, int j) {
    if (j >= wblk) return;
    scores(knext, j + 1);
    int vof = vo;
    asm volatile("" : "+v"(vof));
    auto read_v = [&](int n) {   // operand n = 2 dt + k2, by transposing reads (attn_verify's key order)
      const int dt = n >> 1, k2 = n & 1;
      const unsigned char* vp = vset + (vof ^ (64 * (dt & 3))) + 256 * (dt >> 2) + 16 * (AT_D * 2) * k2;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)vp);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vp + 8 * (AT_D * 2)));
      const u32x2_t w0 = __builtin_bit_cast(u32x2_t, v0), w1 = __builtin_bit_cast(u32x2_t, v1);
      return __builtin_bit_cast(bf16x8, u32x4_t{w0.x, w0.y, w1.x, w1.y});
    };
    bf16x8 vf[AP_AHEAD];
    u32x4_t Pn[RG][2], Pm[RG][2];
    float pe[RG];
#pragma unroll
    for (int i = 0; i < AP_AHEAD; ++i) vf[i] = read_v(i);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
        O[rg][n >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[n % AP_AHEAD], P[rg][n & 1], O[rg][n >> 1], 0, 0, 0);
#pragma unroll
      for (int rg = 0; rg < RG; ++rg)
        O[rg][n >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[n % AP_AHEAD], Pl[rg][n & 1], O[rg][n >> 1], 0, 0, 0);
      if (n + AP_AHEAD < 16) vf[n % AP_AHEAD] = read_v(n + AP_AHEAD);
#pragma unroll
      for (int rg = 0; rg < RG; ++rg) {
        const float p = fast_exp2(__builtin_fmaf(S[rg][n], a.cl2, -base[rg]));
        if (n & 1) {   // (pinned here: the compiler would sink them all past the rescale)
          uint32_t hi, lo;
          ap_split(pe[rg], p, hi, lo);
          l_s[rg] += pe[rg] + p;
          asm volatile("" : "+v"(hi), "+v"(lo), "+v"(l_s[rg]));
          Pn[rg][n >> 3][(n & 7) >> 1] = hi;
          Pm[rg][n >> 3][(n & 7) >> 1] = lo;
        } else {
          pe[rg] = p;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int rg = 0; rg < RG; ++rg)
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        P[rg][k2] = __builtin_bit_cast(bf16x8, Pn[rg][k2]);
        Pl[rg][k2] = __builtin_bit_cast(bf16x8, Pm[rg][k2]);
      }
    rescale();
  };

  AP_BARRIER(16);   // block 0 of K, the first 4 of the 20 loads
  if (wblk > 0) {
    scores(ks0, 0);
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
      u32x4_t Pn[2], Pm[2];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = fast_exp2(__builtin_fmaf(S[rg][r], a.cl2, -base[rg]));
        const float p1 = fast_exp2(__builtin_fmaf(S[rg][r + 1], a.cl2, -base[rg]));
        uint32_t hi, lo;
        ap_split(p0, p1, hi, lo);
        l_s[rg] += p0 + p1;
        Pn[r >> 3][(r & 7) >> 1] = hi;
        Pm[r >> 3][(r & 7) >> 1] = lo;
      }
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        P[rg][k2] = __builtin_bit_cast(bf16x8, Pn[k2]);
        Pl[rg][k2] = __builtin_bit_cast(bf16x8, Pm[k2]);
      }
    }
    rescale();
  }
  // Barrier before step j: blocks j + 1 of K and j of V have landed (the 8 loads after them may
  // be in flight), and every wave is done with K of block j and V of block j - 1, whose sets
  // the loads of blocks j + 3 and j + 2 take.
  for (int j = 0; j < nblk; j += 3) {
    AP_BARRIER(8);
    issue_k(ks0, j + 3);
    issue_v(vs2, j + 2);
    step(ks1, vs0, j);
    AP_BARRIER(8);
    issue_k(ks1, j + 4);
    issue_v(vs0, j + 3);
    step(ks2, vs1, j + 1);
    AP_BARRIER(8);
    issue_k(ks2, j + 5);
    issue_v(vs1, j + 4);
    step(ks0, vs2, j + 2);
  }
  AP_BARRIER(0);   // no load in flight, every wave done with the sets: the dumps take them
#undef AP_BARRIER

  // Epilogue in two halves of the columns: O / l through the wave's own 16 KB (fp32, chunk c
  // of row r at c ^ (r & 15)), then whole half rows with the gate: 8 columns per lane,
  // 16-byte loads and stores.
  unsigned char* dump = wave == 0 ? ks0 : (wave == 1 ? ks1 : (wave == 2 ? ks2 : vs0));
#pragma unroll
  for (int rg = 0; rg < RG; ++rg) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_s[rg]), __float_as_uint(l_s[rg]), false, false);
    const float l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    const float inv = l == 0.f ? 0.f : 1.f / l;   // no key seen: zeros
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // this lane's 8 half rows 4 it + lane / 16, columns 8 (lane % 16) ..; gates first
      const int c8 = lane & 15;
      u32x4_t g[8];
      size_t oo[8];
      bool live[8];
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int r = 32 * (RG * wave + rg) + 4 * it + (lane >> 4), qi = ap_div(r, a.rep_mul), hr = r - qi * a.n_rep;
        live[it] = qi < QB;
        oo[it] = (((size_t)b * a.T + q0 + (live[it] ? qi : 0)) * a.Hq + kvh * a.n_rep + hr) * AT_D + 128 * half + 8 * c8;
        if (a.gate) g[it] = *reinterpret_cast<const u32x4_t*>(a.gate + oo[it]);
      }
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = (8 * dt + 2 * q + h) ^ (l32 & 15);
          const f32x16& o = O[rg][4 * half + dt];
          *reinterpret_cast<float4*>(dump + l32 * 512 + 16 * c) =
              make_float4(o[4 * q] * inv, o[4 * q + 1] * inv, o[4 * q + 2] * inv, o[4 * q + 3] * inv);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own dump, read by the wave only
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int rr = 4 * it + (lane >> 4);
        float y[8];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float4 f = *reinterpret_cast<const float4*>(dump + rr * 512 + 16 * ((2 * c8 + u) ^ (rr & 15)));
          y[4 * u] = f.x; y[4 * u + 1] = f.y; y[4 * u + 2] = f.z; y[4 * u + 3] = f.w;
        }
        if (a.gate) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y[2 * e] *= sigmoidf_(__uint_as_float(g[it][e] << 16));
            y[2 * e + 1] *= sigmoidf_(__uint_as_float(g[it][e] & 0xffff0000u));
          }
        }
        u32x4_t w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bf16x2 t = {(__bf16)y[2 * e], (__bf16)y[2 * e + 1]};
          w[e] = __builtin_bit_cast(uint32_t, t);
        }
        if (live[it]) *reinterpret_cast<u32x4_t*>(a.out + oo[it]) = w;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the next half's dump
    }
  }
}

int attn_prefill_groups(int B, int T, int Hkv, int n_rep, int cus) {
  // A sequence's numbers do not depend on how its tokens are divided into calls of up to 64 (the
  // few-row GEMMs' limit): those keep the split-K kernels, whose rows do not depend on T.  Nor do
  // they depend on the cache's capacity, so the lines below go by the queries alone.
  if (T < AP_MIN_T || (long long)B * T <= AP_FEW_ROWS) return 0;
  const long long rows = (long long)T * n_rep, pairs = (long long)B * Hkv;
  // 256-row tiles cost 1.7 of a 128-row tile's time; worth it from one and a half rounds of them
  // (us, RG = 1 / 2: 384 tiles of 3072 keys 256 / 242, 400 of 1600 161 / 150, 512 of 4096 407 /
  // 372; 128 tiles of 8256 keys 368 / 521)
  if (2 * pairs * ((rows + 255) / 256) >= 3LL * cus) return 2;
  // A lone tile walks its keys at 0.038 us each; the split kernels take 0.00048 us per key and
  // tile: from 80 tiles on this kernel is the faster one whatever the length (us, long / split:
  // 128 tiles of 500 keys 33 / 75; 64 of 1024 51 / 54, of 2000 84 / 83, of 4000 153 / 124; 56
  // of 4000 153 / 110)
  if (16 * pairs * ((rows + 127) / 128) >= 5LL * cus) return 1;
  return 0;
}

int attn_prefill_launch(const AttnArgs& v, int rg, hipStream_t st) {
  ApArgs a;
  a.q = v.q; a.kc = v.kc; a.vc = v.vc; a.kv_len = v.kv_len; a.gate = v.gate; a.out = v.out;
  a.seq_stride = v.seq_stride; a.head_stride = v.head_stride;
  a.B = v.B; a.T = v.T; a.Hq = v.Hq; a.Hkv = v.Hkv; a.n_rep = v.n_rep; a.max_len = v.max_len;
  a.cl2 = v.cl2;
  a.rep_mul = (uint32_t)((65536 + v.n_rep - 1) / v.n_rep);
  a.QB = 128 * rg / v.n_rep < v.T ? 128 * rg / v.n_rep : v.T;
  a.qtiles = (v.T + a.QB - 1) / a.QB;
  const long long n = (long long)a.qtiles * v.B * v.Hkv;
  if (n > 0x7fffffffLL) return LOLLM_EUNSUPPORTED;
  if (rg == 2)
    hipLaunchKernelGGL(attn_prefill_kernel<2>, dim3((unsigned)n), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(attn_prefill_kernel<1>, dim3((unsigned)n), dim3(256), 0, st, a);
  return launch_status();
}

}  // namespace lollm
