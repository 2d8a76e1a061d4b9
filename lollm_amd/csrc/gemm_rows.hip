// C = A W^T for many rows (prefill), gfx950 bf16 MFMA, W in the tiled layout of
// lollm_gemm_tile_weights: 1 KB blocks of 16 rows x 32 k in MFMA-operand order.
//
// A workgroup of four waves (2 x 2) owns a (64 MT) x (64 NT) tile of C (rows x columns), a wave
// (32 MT) x (32 NT) of it in 16x16 accumulators.  K runs in steps of 32 through LDS buffers
// filled by DMA two to three steps ahead (W per step, four buffers; A per pair of steps, so that
// a load takes whole 128-byte lines, two buffers), one barrier per step, and the steps of a
// workgroup's next tile follow without a break: its first loads are issued in the last steps of
// the current one and land during the epilogue.  Four waves and not eight: an operand is then
// read by half as many waves, and LDS (128 B per cycle) stays under half busy.  A lone wave per
// SIMD overlaps nothing by itself, so the operands of a step are read during the step before
// and the order is fixed: a read or a DMA every few products.  Every output adds its products
// in k order, whatever the tile: unless K is cut into parts (chosen from M), a row's bits depend
// on neither M nor the tile.
//
// What bounds it: power.  4096 x 4096 x 12288 runs at 1876 TFLOP/s on zeros and 1600 on random
// values.  Measured steps (us at 3998 x 4096 x 12288): 32x32x16 products 292 (an accumulator is
// read and written once per 16 k), 16x16x32 276 (once per 32 k), tiles without a break 265, A
// in whole lines 257; reads and DMA moved to the first half of the step 270.
#include "common.h"

namespace lollm {

typedef __bf16 gr_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gr_bf16x2 __attribute__((ext_vector_type(2)));
typedef float gr_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int gr_u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void gr_lds_t;

constexpr int GR_THREADS = 256;

struct GrArgs {
  const uint16_t* A;    // (M, K), row stride lda
  const uint16_t* Wt;   // tiled weight
  uint16_t* C;          // (M, oc), row stride ldc
  long long lda, ldc;
  int M, N, K;
  int mt, nt;           // tiles
  float* part;          // split K: (splits, M, N) fp32
  int splits;
};

__device__ __forceinline__ float gr_round(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ float gr_silu_bf16(float g) {   // lollm_gemm's SwiGLU arithmetic
  const float gr = gr_round(g);
  return gr_round(gr / (1.f + __expf(-gr)));
}
__device__ __forceinline__ uint32_t gr_pack(float a, float b) {
  const gr_bf16x2 t = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, t);
}

// This wave's loads and stores up to the last N are done and its LDS reads complete, then every
// wave's.
template <int N> struct GrInt { static constexpr int value = N; };
template <int N> __device__ __forceinline__ void gr_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// gr_wait<N> or, when more != 0, gr_wait<MORE>, without a branch for the compiler to split the
// step's registers around
template <int N, int MORE> __device__ __forceinline__ void gr_wait_if(int more) {
  asm volatile("s_cmp_eq_u32 %0, 0\n\ts_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%2)\n\ts_branch 2f\n"
               "1:\n\ts_waitcnt vmcnt(%1)\n2:\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier"
               ::"s"(more), "n"(N), "n"(MORE) : "memory", "scc");
}

// keeps an accumulator in the accumulator registers
__device__ __forceinline__ void gr_pin(gr_f32x4& v) { asm volatile("" : "+a"(v)); }

// SPLIT: K in a.splits equal parts, a (tile, part) to a workgroup, fp32 sums to a.part.
template <int MT, int NT, bool SWIGLU, bool SPLIT>
__device__ __forceinline__ void gr_tiles(const GrArgs& a) {
  constexpr int BM = 64 * MT, BN = 64 * NT;
  constexpr int ABYTES = BM * 128, BBYTES = BN * 64;   // rows of a k64 pair, columns of a k32 step
  // one array per buffer: the reads of one are not ordered after the DMA into another
  __shared__ __attribute__((aligned(16))) unsigned char a0[ABYTES], a1[ABYTES];
  __shared__ __attribute__((aligned(16))) unsigned char b0[BBYTES], b1[BBYTES], b2[BBYTES], b3[BBYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  const int ntiles = a.mt * a.nt * (SPLIT ? a.splits : 1);

  // Tile number v = blockIdx.x + i gridDim.x: an XCD (workgroups i, i + 8, ..) takes a
  // contiguous run of the tiles, ordered in bands of 8 row tiles, so that the 32 tiles it works
  // on at a time share rows and columns in its L2.
  auto locate = [&](int v, int& m0, int& n0, int& part) {
    const int x = v & 7, u = x * (ntiles / 8) + min(x, ntiles % 8) + (v >> 3);
    // (the row tiles of a column tile's part next to each other: they read the same W)
    const int tiles = a.mt * a.nt, t = SPLIT ? u % tiles : u;
    part = SPLIT ? u / tiles : 0;
    const int band = t / (8 * a.nt), r = t - band * 8 * a.nt, hb = min(8, a.mt - 8 * band);
    m0 = (8 * band + r % hb) * BM;
    n0 = (r / hb) * BN;
  };
  // descriptors of a tile's rows of A and blocks of W: what lies past M or N reads as zero
  const int kpart = SPLIT ? a.K / a.splits : a.K;   // k of a part: a multiple of 128
  auto rsrc_a = [&](int m0, int part, bool live) {
    return buf_rsrc(a.A + (live ? (size_t)m0 * a.lda + (size_t)part * kpart : 0),
                    live ? (uint32_t)(min(BM, a.M - m0) - 1) * (uint32_t)(2 * a.lda) + 2u * kpart : 0u);
  };
  auto rsrc_b = [&](int n0, int part, bool live) {
    return buf_rsrc(a.Wt + (live ? (size_t)n0 * a.K + (size_t)part * kpart * 16 : 0),
                    live ? (uint32_t)(min(BN, a.N - n0) / 16 - 1) * (32u * a.K) + 32u * kpart : 0u);
  };
  // Loads: A for a pair of steps, 8 rows of 128 bytes (whole cache lines) per instruction (lane:
  // row lane / 8, chunk lane % 8 of the place written, whose source chunk undoes the swizzle);
  // W one block per instruction.
  constexpr int AI = 2 * MT, BI = NT;   // instructions per wave: of a pair, of a step
  uint32_t aoff[AI], boff[BI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int row = 8 * (AI * wave + i) + (lane >> 3);
    aoff[i] = (uint32_t)row * (uint32_t)(2 * a.lda) + 16u * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < BI; ++i) boff[i] = (uint32_t)(BI * wave + i) * (32u * a.K) + 16u * lane;
  auto dma_a = [&](unsigned char* s, __amdgpu_buffer_rsrc_t rs, int i, uint32_t kb) {   // kb: bytes into a row
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (gr_lds_t*)(s + 1024 * (AI * wave + i)), 16, aoff[i], kb, 0, 0);
  };
  auto dma_b = [&](unsigned char* s, __amdgpu_buffer_rsrc_t rs, int i, uint32_t kb) {   // a 1 KB block per step
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (gr_lds_t*)(s + 1024 * (BI * wave + i)), 16, boff[i], 16 * kb, 0, 0);
  };
  // operand reads: A rows 16 i + r16, chunk 4 (step % 2) + g4 (swizzled); W block 2 NT wn + j
  const int ar = (32 * MT * wm + r16) * 128 + 16 * (g4 ^ ((r16 >> 1) & 7));
  const int br = 2 * NT * wn * 1024 + 16 * lane;
  auto read_a = [&](const unsigned char* s, int i, int odd) {
    return *reinterpret_cast<const gr_bf16x8*>(s + (ar ^ (64 * odd)) + 2048 * i);
  };
  auto read_b = [&](const unsigned char* s, int j) { return *reinterpret_cast<const gr_bf16x8*>(s + br + 1024 * j); };

  const int steps = kpart / 32;   // a multiple of 4
  int v = blockIdx.x, m0, n0, part;
  locate(v, m0, n0, part);
  __amdgpu_buffer_rsrc_t ars = rsrc_a(m0, part, true), brs = rsrc_b(n0, part, true);
  auto fill_a = [&](unsigned char* s, int k) {
#pragma unroll
    for (int i = 0; i < AI; ++i) dma_a(s, ars, i, 64u * k);
  };
  auto fill_b = [&](unsigned char* s, int k) {
#pragma unroll
    for (int i = 0; i < BI; ++i) dma_b(s, brs, i, 64u * k);
  };
  fill_a(a0, 0);
  fill_b(b0, 0);
  fill_b(b1, 1);
  fill_a(a1, 2);
  fill_b(b2, 2);
  gr_wait<AI + 2 * BI>();   // step 0 landed
  constexpr int AF = 2 * MT, BF = 2 * NT;   // operands of a step
  gr_bf16x8 fa[2][AF], fb[2][BF];
#pragma unroll
  for (int i = 0; i < AF; ++i) fa[0][i] = read_a(a0, i, 0);
#pragma unroll
  for (int j = 0; j < BF; ++j) fb[0][j] = read_b(b0, j);

  constexpr int OC = SWIGLU ? 16 * NT : 32 * NT;     // output columns of a wave
  constexpr int PER = OC / 8;                        // 16-byte chunks per row of it
  constexpr int STORES = SPLIT ? AF * BF : MT * (32 * PER / 64);   // store instructions of a wave's epilogue
  static_assert(AI + BI + STORES <= 63, "vmcnt");
  int after = 0;   // a tile came before this one

  for (;; after = 1) {
    // the next tile, whose first steps follow this one's last
    const int vn = v + (int)gridDim.x;
    const bool more = vn < ntiles;
    int m1 = 0, n1 = 0, part1 = 0;
    if (more) locate(vn, m1, n1, part1);
    const __amdgpu_buffer_rsrc_t arn = rsrc_a(m1, part1, more), brn = rsrc_b(n1, part1, more);

    gr_f32x4 acc[BF][AF];
#pragma unroll
    for (int j = 0; j < BF; ++j)
#pragma unroll
      for (int i = 0; i < AF; ++i) {
        acc[j][i] = gr_f32x4{0.f, 0.f, 0.f, 0.f};
        gr_pin(acc[j][i]);
      }

    // One step: barrier (the next step's data has landed, every wave holds this one's operands),
    // then AF x BF products; between them the operand reads of the next step, the DMA of W for
    // the third after this one and, in odd steps, of A for that one and the fourth.  So in flight
    // past the next step's data: W of one step and, before even steps, a pair of A.  The first
    // two barriers after an epilogue leave its stores in flight.
    auto step = [&](auto par, const unsigned char* an, const unsigned char* bn, unsigned char* ad, unsigned char* bd,
                    int k) {
      constexpr int P = decltype(par)::value, p = P & 1;
      constexpr int FLY = BI + (p ? 0 : AI), DM = BI + (p ? AI : 0);
      if (P < 2) gr_wait_if<FLY, FLY + STORES>(after & (int)(k < 2));
      else gr_wait<FLY>();
      const bool over = k + 3 >= steps;
      const __amdgpu_buffer_rsrc_t ra = over ? arn : ars, rb = over ? brn : brs;
      const uint32_t kb = 64u * (uint32_t)(over ? k + 3 - steps : k + 3);
#pragma unroll
      for (int n = 0; n < AF * BF; ++n) {
        const int j = n / AF, i = j & 1 ? AF - 1 - n % AF : n % AF;
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[p][j], fa[p][i], acc[j][i], 0, 0, 0);
        constexpr int GAP = AF * BF / (AF + BF), DG = AF * BF / DM;
        if (n % GAP == 0 && n / GAP < AF + BF) {
          const int r = n / GAP;
          if (r < BF) fb[p ^ 1][r] = read_b(bn, r);
          else fa[p ^ 1][r - BF] = read_a(an, r - BF, p ^ 1);
        }
        if (n % DG == DG / 2 && n / DG < DM) {
          const int r = n / DG;
          if (r < DM - BI) dma_a(ad, ra, r, kb);
          else dma_b(bd, rb, r - (DM - BI), kb);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for (int k = 0; k < steps; k += 4) {
      step(GrInt<0>{}, a0, b1, a0, b3, k);
      step(GrInt<1>{}, a1, b2, a0, b0, k + 1);
      step(GrInt<2>{}, a1, b3, a0, b1, k + 2);
      step(GrInt<3>{}, a0, b0, a1, b2, k + 3);
    }

#pragma unroll
    for (int j = 0; j < BF; ++j)
#pragma unroll
      for (int i = 0; i < AF; ++i) gr_pin(acc[j][i]);

    if constexpr (SPLIT) {
      // the part's sums as they are: 4 columns of a row per lane
      int elane = lane;
      asm volatile("" : "+v"(elane));
      const int er16 = elane & 15, eg4 = elane >> 4;
      const __amdgpu_buffer_rsrc_t prs = buf_rsrc(a.part + ((size_t)part * a.M + m0) * a.N,
                                                  (uint32_t)min(BM, a.M - m0) * (uint32_t)(4 * a.N));
#pragma unroll
      for (int i = 0; i < AF; ++i)
#pragma unroll
        for (int j = 0; j < BF; ++j) {
          const int row = 32 * MT * wm + 16 * i + er16, col = n0 + 32 * NT * wn + 16 * j + 4 * eg4;
          const uint32_t off = col < a.N ? (uint32_t)row * (uint32_t)(4 * a.N) + 4u * col : 0xfffffff0u;
          const gr_f32x4 t = acc[j][i];
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, t), prs, off, 0, 0);
        }
    } else {
      // Epilogue per SR rows: the accumulators (lane: row r16, columns 16 j + 4 g4 + e) through the
      // wave's quarter of b3 (free: its last data was read before the last barrier, and the next
      // DMA into it follows the next one) as bf16, 16-byte chunk c of row r at c ^ (r & XM), then
      // 16-byte stores along the rows, dropped past M and N by the descriptor (every store is
      // issued: the waits above count them).
      constexpr int PITCH = 2 * OC, SR = SWIGLU ? 32 : 16;   // rows staged at a time
      constexpr int XM = PER % 8 == 0 ? 7 : (PER % 4 == 0 ? 3 : 1);
      static_assert(SR * PITCH <= BBYTES / 4, "staging");
      unsigned char* st = b3 + wave * (BBYTES / 4);
      const int nout = SWIGLU ? a.N / 2 : a.N, c0 = (SWIGLU ? n0 / 2 : n0) + OC * wn;
      const __amdgpu_buffer_rsrc_t crs = buf_rsrc(
          a.C + (size_t)m0 * a.ldc, (uint32_t)(min(BM, a.M - m0) - 1) * (uint32_t)(2 * a.ldc) + 2u * nout);
      // (from an opaque copy of the lane, so that no address is kept through the products)
      int elane = lane;
      asm volatile("" : "+v"(elane));
      const int er16 = elane & 15, eg4 = elane >> 4;
#pragma unroll
      for (int i = 0; i < 32 * MT / SR; ++i) {
#pragma unroll
        for (int u = 0; u < SR / 16; ++u)
#pragma unroll
          for (int j = 0; j < BF; j += SWIGLU ? 2 : 1) {
            gr_f32x4 y = acc[j][SR / 16 * i + u];
            int col = 16 * j + 4 * eg4;
            if constexpr (SWIGLU) {
              // a block holds 8 gate rows, then their 8 up rows, lanes 32 apart: the swap gives the
              // lower lanes block j's pairs and the upper ones block j + 1's
              const gr_f32x4 t = acc[j + 1][SR / 16 * i + u];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[e]), __float_as_uint(t[e]), false, false);
                y[e] = gr_silu_bf16(__uint_as_float(sw[0])) * gr_round(__uint_as_float(sw[1]));
              }
              col = 8 * (j + (eg4 >> 1)) + 4 * (eg4 & 1);
            }
            *reinterpret_cast<gr_u32x2*>(st + (16 * u + er16) * PITCH + ((2 * col) ^ (16 * (er16 & XM)))) =
                gr_u32x2{gr_pack(y[0], y[1]), gr_pack(y[2], y[3])};
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own staging
#pragma unroll
        for (int n = 0; n < SR * PER / 64; ++n) {
          const int c = 64 * n + elane, r = c / PER, cc = c % PER;
          const int row = 32 * MT * wm + SR * i + r, col = c0 + 8 * cc;
          const u32x4_t w = *reinterpret_cast<const u32x4_t*>(st + r * PITCH + 16 * (cc ^ (r & XM)));
          const uint32_t off = col < nout ? (uint32_t)row * (uint32_t)(2 * a.ldc) + 2u * col : 0xfffffff0u;
          __builtin_amdgcn_raw_buffer_store_b128(w, crs, off, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    }
    if (!more) break;
    v = vn;
    m0 = m1;
    n0 = n1;
    part = part1;
    ars = arn;
    brs = brn;
  }
  // (the loads issued for a tile that does not follow moved nothing but count until they return)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int MT, int NT, bool SWIGLU, bool SPLIT>
__global__ __launch_bounds__(GR_THREADS, 1) void gemm_rows_kernel(GrArgs a) {
  gr_tiles<MT, NT, SWIGLU, SPLIT>(a);   // (a device function: the host pass drops the kernel's stub otherwise)
}

// C from the parts, added in k order: 8 columns of C per thread.
template <bool SWIGLU>
__global__ __launch_bounds__(256) void gemm_rows_reduce_kernel(GrArgs a) {
  const int per = (SWIGLU ? a.N / 2 : a.N) / 8;
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= (long long)a.M * per) return;
  const int row = (int)(c / per), cc = (int)(c % per);
  const float* p = a.part + (size_t)row * a.N + (SWIGLU ? 16 : 8) * cc;
  constexpr int Q = SWIGLU ? 4 : 2;
  gr_f32x4 s[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) s[q] = reinterpret_cast<const gr_f32x4*>(p)[q];
  for (int n = 1; n < a.splits; ++n) {
    p += (size_t)a.M * a.N;
#pragma unroll
    for (int q = 0; q < Q; ++q) s[q] += reinterpret_cast<const gr_f32x4*>(p)[q];
  }
  u32x4_t w;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int q = e >> 1, l = 2 * (e & 1);
    if (SWIGLU)   // 8 gate columns, then their 8 up columns
      w[e] = gr_pack(gr_silu_bf16(s[q][l]) * gr_round(s[2 + q][l]), gr_silu_bf16(s[q][l + 1]) * gr_round(s[2 + q][l + 1]));
    else
      w[e] = gr_pack(s[q][l], s[q][l + 1]);
  }
  *reinterpret_cast<u32x4_t*>(a.C + (size_t)row * a.ldc + 8 * cc) = w;
}

template <bool SWIGLU>
static int gr_launch(GrArgs& a, int tile, int cus, hipStream_t st) {
  const int MT = tile / 10, NT = tile % 10;
  a.mt = (a.M + 64 * MT - 1) / (64 * MT);
  a.nt = (a.N + 64 * NT - 1) / (64 * NT);
  const long long n = (long long)a.mt * a.nt;
  if (n > 0x3fffffff) return LOLLM_EUNSUPPORTED;
  const dim3 g((unsigned)(n < cus ? n : cus)), b(GR_THREADS);
  if (a.splits > 1) {
    const long long u = n * a.splits, chunks = (long long)a.M * (SWIGLU ? a.N / 2 : a.N) / 8;
    hipLaunchKernelGGL((gemm_rows_kernel<2, 4, false, true>), dim3((unsigned)(u < cus ? u : cus)), b, 0, st, a);
    const int rc = launch_status();
    if (rc) return rc;
    hipLaunchKernelGGL(gemm_rows_reduce_kernel<SWIGLU>, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st, a);
    return launch_status();
  }
  switch (tile) {
    case 44: hipLaunchKernelGGL((gemm_rows_kernel<4, 4, SWIGLU, false>), g, b, 0, st, a); break;
    case 34: hipLaunchKernelGGL((gemm_rows_kernel<3, 4, SWIGLU, false>), g, b, 0, st, a); break;
    case 43: hipLaunchKernelGGL((gemm_rows_kernel<4, 3, SWIGLU, false>), g, b, 0, st, a); break;
    case 24: hipLaunchKernelGGL((gemm_rows_kernel<2, 4, SWIGLU, false>), g, b, 0, st, a); break;
    default: return LOLLM_EINVAL;
  }
  return launch_status();
}

}  // namespace lollm

using namespace lollm;

LOLLM_API int lollm_gemm_rows(const void* A, long long lda, const void* Wt, void* C, long long ldc, int M, int N,
                              int K, int epilogue, int tile, int splits, void* workspace,
                              long long workspace_bytes, void* stream) {
  if (!A || !Wt || !C) return LOLLM_EINVAL;
  if (M <= 0 || N <= 0 || K <= 0 || lda < K || epilogue < 0 || epilogue > 1) return LOLLM_EINVAL;
  if (N % 64 || K % 128 || lda % 8 || ldc % 8 || ldc < (epilogue ? N / 2 : N)) return LOLLM_EINVAL;
  if (((uintptr_t)A | (uintptr_t)Wt | (uintptr_t)C | (uintptr_t)workspace) % 16) return LOLLM_EINVAL;
  if (splits < 1 || K / 128 % splits || (splits > 1 && tile != 24)) return LOLLM_EINVAL;
  if (splits > 1 && (!workspace || workspace_bytes < 4LL * splits * M * N)) return LOLLM_EINVAL;
  // 32-bit byte offsets inside a tile
  if (256LL * 2 * lda >= (1LL << 31) || 256LL * 2 * ldc >= (1LL << 31) || 256LL * 2 * K >= (1LL << 31) ||
      256LL * 4 * N >= (1LL << 31))
    return LOLLM_EUNSUPPORTED;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return LOLLM_EUNSUPPORTED;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return LOLLM_EUNSUPPORTED;
  GrArgs a;
  a.A = (const uint16_t*)A; a.Wt = (const uint16_t*)Wt; a.C = (uint16_t*)C;
  a.lda = lda; a.ldc = ldc; a.M = M; a.N = N; a.K = K;
  a.part = (float*)workspace; a.splits = splits;
  return epilogue ? gr_launch<true>(a, tile, cus, (hipStream_t)stream)
                  : gr_launch<false>(a, tile, cus, (hipStream_t)stream);
}
