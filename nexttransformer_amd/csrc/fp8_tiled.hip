// Grouped expert GEMM on e4m3 operands for segments of many rows (fp8 prefill).
//
// The same products as fp8_grouped_gemm_kernel (fp8.hip), bit for bit, on weights packed by
// pack_fp8_kernel; that kernel streams a segment's weights once per 32 rows, which is right for a
// few rows per expert and reads the weights eight times where an expert has 256. Here a workgroup
// takes up to 256 rows against 128 packed weight rows.
//
// What bounds it: the CU's vector-memory path (about 64 bytes a clock) and the matrix cores. A
// 128-wide K step of a full tile copies 32 KB of token rows into LDS and streams 16 KB of weights
// into registers for 64 MFMA pairs (1024 matrix-core cycles a SIMD), the same 48 bytes per clock
// as the packed bf16 kernel's tile.
//   * Wave w owns the tile's packed 32-row weight block w against all of its token blocks (up to
//     8 accumulators); the weights are private to the wave, so they skip LDS (1 KB loads, one
//     step ahead; two steps ahead in tiles of 64 to 192 rows, which have the registers to spare:
//     at 224 rows five would spill).
//   * Token rows go through LDS in a ring of two steps (direct-to-LDS loads, 16-byte chunks
//     XOR-swizzled by row as in the packed bf16 kernel), one barrier per step.
//   * The scale of a 128 x 128 weight block is an fp32 number, not a power of two, so each step's
//     product goes into a zeroed fragment that is scaled and added to the fp32 accumulator (16
//     FMAs per 128 matrix-core cycles, in the shadow of the CU's other wave).
//   * The outputs are transposed through the LDS of the token stages, so every store instruction
//     writes whole 256-byte (SwiGLU 128-byte) row segments.
// Two workgroups per CU: one's barriers, start and stores run under the other's products. A
// segment's rows are dealt evenly to its tiles in multiples of 32, so a segment of 260 rows is
// two tiles of 128 and 132 and not 256 and 4.
// The tile is instantiated for each number of 32-row blocks: with 1, 2, 4, 6 and 8 only (and two
// steps ahead up to 4) a tile of 9 / 2 blocks multiplied a sixth for padding, 4096 tokens below
// 569 / 350 us against 536 / 342, the forward 1110 against 1082.
//
// Measured, us up / down projection, that kernel -> this one (128 experts, top-8, d 4096, H 1536;
// outputs bit-identical): 4096 tokens (256 rows per expert) 2285 / 1265 -> 536 / 342 (1540 / 1200
// TFLOP/s), 1024 tokens 677 / 390 -> 300 / 194, 256 tokens 279 / 183 -> 278 / 163, 64 tokens 260 /
// 156 -> 268 / 154. At 1024 tokens and fewer the time is the weight stream's.
#include <math.h>

#include "common.h"

namespace ntmoe {
namespace {

typedef __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

constexpr int kKB = 128;           // K per step (one scale block)
constexpr int kMaxRows = 256;      // token rows per tile
constexpr int kBlockBytes = 4096;  // packed weight block: 32 rows x 128 K
constexpr int kTileBlocks = 4;     // packed blocks per tile (one per wave)
constexpr int kStageBytes = kMaxRows * kKB;
constexpr int kMaxK = 64 * kKB;    // a wave's lanes hold the K steps' scales

__device__ __forceinline__ int swz8(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

__device__ __forceinline__ float fp8_silu_mul(float g, float u) {
  return g * u * __builtin_amdgcn_rcpf(1.f + __expf(-g));
}

struct F8Args {
  const uint8_t* a;
  int64_t ld_a, a_rows;
  const float* a_scale;
  const int32_t* src_row;
  const int32_t* seg_offsets;
  int S, total_rows;
  const uint8_t* w;
  const float* w_scale;
  int K, n_out;
  uint16_t* c;
};

// One tile: rows [m0, m_end) (at most 32 NJ) of segment s against packed blocks 4 nt .. 4 nt + 3.
template <int EPI, int NJ>
__device__ __forceinline__ void fp8_tile(const F8Args& p, unsigned char* smem, int s, int nt,
                                         int m0, int m_end) {
  constexpr int D = NJ == 1 || NJ >= 7 ? 1 : 2;  // weight steps in flight beyond the current one
  constexpr int kStage = NJ * 32 * kKB;
  constexpr bool SW = EPI == NT_MOE_EPI_SWIGLU;
  const int lane = lane_id(), wave = wave_id();
  const int li = lane & 31, half = lane >> 5;
  const int w_rows = SW ? 2 * p.n_out : p.n_out;
  const int NB = w_rows / 32;
  const int nk = p.K / kKB;
  const int nb = nt * kTileBlocks + wave;  // R % 128 == 0: every wave of a tile has its block
  // scales of K step l in lane l, for the rows of accumulator elements 0-7 and 8-15
  const int row_lo = SW ? nb * 16 : nb * 32, row_hi = SW ? p.n_out + nb * 16 : nb * 32;
  const int64_t srow0 = (int64_t)s * ((w_rows + 127) / 128);
  const int lk = lane < nk ? lane : nk - 1;
  const int vs_lo = __builtin_bit_cast(int, p.w_scale[(srow0 + row_lo / 128) * nk + lk]);
  const int vs_hi = __builtin_bit_cast(int, p.w_scale[(srow0 + row_hi / 128) * nk + lk]);

  // this lane's token-row chunk in each of the wave's NJ copy instructions (8 rows of 128 bytes)
  uint32_t aoff[NJ];
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    const int row = (wave * NJ + q) * 8 + (lane >> 3);
    const int tok = m0 + row < m_end ? m0 + row : m_end - 1;
    int64_t r = p.src_row ? (int64_t)p.src_row[tok] : (int64_t)tok;
    r = r < 0 ? 0 : (r >= p.a_rows ? p.a_rows - 1 : r);
    aoff[q] = (uint32_t)(r * p.ld_a) + (uint32_t)(swz8(row, lane & 7) << 4);
  }
  const uint8_t* wbase = p.w + ((int64_t)s * NB + nb) * (int64_t)nk * kBlockBytes;
  const uint32_t b_lane = lane * 16;
  auto load_a = [&](int kb, int q) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds(
        (gvoid*)(p.a + (int64_t)(kb < nk ? kb : nk - 1) * kKB + aoff[q]),
        (lvoid*)(smem + (kb & 1) * kStage + (wave * NJ + q) * 1024), 16, 0, 0);
  };
  // Inline assembly, as in the packed bf16 kernel: the compiler adds no waits of its own, and the
  // wait before a step's products names the registers.
  auto load_b = [&](int kb, auto i_c, u32x4 (&b)[4]) __attribute__((always_inline)) {
    constexpr int i = decltype(i_c)::value;
    const uint8_t* blk = wbase + (int64_t)(kb < nk ? kb : nk - 1) * kBlockBytes;
    const uint32_t off = b_lane;
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3"
                 : "=v"(b[i])
                 : "v"(off), "s"(blk), "n"(i * 1024)
                 : "memory");
  };
  // Token fragment of block j, 64-wide half st: bytes [32 half, +32) of row 32 j + li.
  int frag_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    frag_off[q] = li * kKB + (swz8(li, (q >> 1) * 4 + half * 2 + (q & 1)) << 4);

  floatx16 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = floatx16{};
  u32x4 wq[D + 1][4];

  static_for<0, NJ>([&](auto q_c) { load_a(0, decltype(q_c)::value); });
  static_for<0, D>([&](auto j_c) {
    static_for<0, 4>([&](auto i_c) { load_b(decltype(j_c)::value, i_c, wq[decltype(j_c)::value]); });
  });
  // step 0's rows and weights have landed (the second step's weights may be in flight)
  auto wait_for = [&](u32x4 (&b)[4]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%4)"
                 : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3])
                 : "n"(4 * (D - 1))
                 : "memory");
  };
  wait_for(wq[0]);

  // K step kb: products with bc, the weights D steps ahead into bl, bn landed at its end. A TAIL
  // step's later weights have all landed: it copies token rows only.
  auto step = [&](auto tail_c, int kb, u32x4 (&bc)[4], u32x4 (&bl)[4], u32x4 (&bn)[4])
                  __attribute__((always_inline)) {
    constexpr bool TAIL = decltype(tail_c)::value;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    {
      const unsigned char* st = smem + (kb & 1) * kStage;
      const float s_lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vs_lo, kb));
      const float s_hi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vs_hi, kb));
      const i32x8 w0 = {(int)bc[0][0], (int)bc[0][1], (int)bc[0][2], (int)bc[0][3],
                        (int)bc[1][0], (int)bc[1][1], (int)bc[1][2], (int)bc[1][3]};
      const i32x8 w1 = {(int)bc[2][0], (int)bc[2][1], (int)bc[2][2], (int)bc[2][3],
                        (int)bc[3][0], (int)bc[3][1], (int)bc[3][2], (int)bc[3][3]};
      auto frag = [&](int j, int q) __attribute__((always_inline)) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(st + j * 32 * kKB + frag_off[2 * q]);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(st + j * 32 * kKB + frag_off[2 * q + 1]);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
                     (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      };
      // The step's copies, spread over the token blocks: the next step's rows, then the weights
      // D steps ahead (that order: the wait below leaves only the last 4 (D - 1) outstanding).
      constexpr int kItems = NJ + (TAIL ? 0 : 4);
      auto item = [&](auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < NJ) {
          load_a(kb + 1, i);  // (past the last step: a re-read into the free slot)
        } else {
          load_b(kb + D, std::integral_constant<int, i - NJ>(), bl);
        }
      };
      constexpr int kOver = NJ > 2 ? NJ - 1 : NJ;  // token blocks the copies are spread over
      i32x8 f[2][2];
      f[0][0] = frag(0, 0);
      f[0][1] = frag(0, 1);
      floatx16 part[2];
      static_for<0, NJ>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
        if constexpr (j + 1 < NJ) {
          f[(j + 1) & 1][0] = frag(j + 1, 0);
          f[(j + 1) & 1][1] = frag(j + 1, 1);
        }
        floatx16 z = {};
        z = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w0, f[j & 1][0], z, 0, 0, 0, 0, 0, 0);
        part[j & 1] =
            __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w1, f[j & 1][1], z, 0, 0, 0, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, kItems>([&](auto i_c) __attribute__((always_inline)) {
          constexpr int i = decltype(i_c)::value;
          if constexpr (i * kOver / kItems == j) item(i_c);
        });
        if constexpr (j > 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            acc[j - 1][i] = fmaf(part[(j - 1) & 1][i], i < 8 ? s_lo : s_hi, acc[j - 1][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int i = 0; i < 16; ++i)
        acc[NJ - 1][i] = fmaf(part[(NJ - 1) & 1][i], i < 8 ? s_lo : s_hi, acc[NJ - 1][i]);
    }
    if constexpr (TAIL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else wait_for(bn);
  };
  // Whole turns of the register ring, a wait for all of it (every load's register is named by a
  // wait before it can be reused), then the remaining steps, whose weights that wait landed.
  constexpr std::false_type kBody{};
  constexpr std::true_type kTail{};
  int kb = 0;
  if constexpr (D == 1) {
    for (; kb + 2 <= nk; kb += 2) {
      step(kBody, kb, wq[0], wq[1], wq[1]);
      step(kBody, kb + 1, wq[1], wq[0], wq[0]);
    }
    if (kb < nk) step(kTail, kb, wq[0], wq[1], wq[1]);
  } else {
    for (; kb + 3 <= nk; kb += 3) {
      step(kBody, kb, wq[0], wq[2], wq[1]);
      step(kBody, kb + 1, wq[1], wq[0], wq[2]);
      step(kBody, kb + 2, wq[2], wq[1], wq[0]);
    }
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(wq[0][0]), "+v"(wq[0][1]), "+v"(wq[0][2]), "+v"(wq[0][3]),
                   "+v"(wq[1][0]), "+v"(wq[1][1]), "+v"(wq[1][2]), "+v"(wq[1][3])
                 :
                 : "memory");
    if (kb < nk) {
      step(kTail, kb, wq[0], wq[2], wq[1]);
      if (kb + 1 < nk) step(kTail, kb + 1, wq[1], wq[0], wq[2]);
    }
  }
  // all copies landed and every wave past its last fragment read: the stages' LDS is free
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // Output tile [32 NJ][kCols] bf16 in LDS, 16-byte chunks XOR-swizzled by row.
  constexpr int kCols = SW ? 64 : 128;
  constexpr int kChunks = kCols / 8;
  auto ooff = [](int r, int c) {
    return r * kCols * 2 + ((c ^ (SW ? (r >> 1) & 7 : r & 15)) << 4);
  };
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int r = 32 * j + li;
    const int tok = m0 + r < m_end ? m0 + r : m_end - 1;
    int64_t ar = p.src_row ? (int64_t)p.src_row[tok] : (int64_t)tok;
    ar = ar < 0 ? 0 : (ar >= p.a_rows ? p.a_rows - 1 : ar);
    const float as = p.a_scale[ar];
#pragma unroll
    for (int g = 0; g < (SW ? 2 : 4); ++g) {
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (SW) {
          o[i] = fp8_silu_mul(as * acc[j][4 * g + i], as * acc[j][4 * (g + 2) + i]);
        } else {
          float v = as * acc[j][4 * g + i];
          if (EPI == NT_MOE_EPI_RELU2) v = v > 0.f ? v * v : 0.f;
          o[i] = v;
        }
      }
      u32x2 v;
      v[0] = pack_bf16x2(o[0], o[1]);
      v[1] = pack_bf16x2(o[2], o[3]);
      *reinterpret_cast<u32x2*>(smem + ooff(r, wave * (SW ? 2 : 4) + g) + half * 8) = v;
    }
  }
  __syncthreads();
  const int col0 = nt * kCols;
#pragma unroll 4
  for (int i = threadIdx.x; i < NJ * 32 * kChunks; i += 256) {
    const int r = i / kChunks, ch = i % kChunks;
    const u32x4 v = *reinterpret_cast<const u32x4*>(smem + ooff(r, ch));
    if (m0 + r < m_end)
      *reinterpret_cast<u32x4*>(p.c + (int64_t)(m0 + r) * p.n_out + col0 + ch * 8) = v;
  }
}

// Workgroup b runs on XCD b mod 8 and takes tile number (the XCD's contiguous share of the tile
// list, in order), so the tiles of a segment, which read the same rows and weights, run at about
// the same time behind one L2. The tile list (segment, m, n; n fastest) is found from
// seg_offsets by every wave with shuffles; workgroups past it leave.
template <int EPI>
__global__ __launch_bounds__(256, 2) void fp8_tiled_gemm_kernel(F8Args p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = lane_id();
  const int n_tiles = (EPI == NT_MOE_EPI_SWIGLU ? 2 * p.n_out : p.n_out) / 32 / kTileBlocks;
  // rows [lo, hi) of segment base + lane (clamped) and its m tiles
  auto segs = [&](int base, int& lo, int& hi, int& mt) {
    const int i = base + lane;
    auto off = [&](int k) {
      const int o = p.seg_offsets[k < p.S ? k : p.S];
      return o < 0 ? 0 : (o > p.total_rows ? p.total_rows : o);
    };
    lo = off(i);
    hi = off(i + 1);
    hi = hi > lo ? hi : lo;
    mt = (hi - lo + kMaxRows - 1) / kMaxRows;
  };
  int total = 0;
  for (int base = 0; base < p.S; base += 64) {
    int lo, hi, mt;
    segs(base, lo, hi, mt);
    for (int w = 32; w >= 1; w >>= 1) mt += __shfl_xor(mt, w);
    total += mt;
  }
  total = __builtin_amdgcn_readfirstlane(total);
  const int64_t n = (int64_t)total * n_tiles;
  const int xcd = blockIdx.x % 8;
  const int64_t tile = n * xcd / 8 + blockIdx.x / 8;
  if (tile >= n * (xcd + 1) / 8) return;
  const int mi = (int)(tile / n_tiles), nt = (int)(tile - (int64_t)mi * n_tiles);
  int s = 0, m0 = 0, m_end = 0, before = 0;
  for (int base = 0; base < p.S; base += 64) {
    int lo, hi, mt;
    segs(base, lo, hi, mt);
    int incl = mt;  // m tiles of segments base .. base + lane
    for (int w = 1; w < 64; w <<= 1) {
      const int u = __shfl_up(incl, w);
      if (lane >= w) incl += u;
    }
    const uint64_t mask = __ballot(mi < before + incl);
    if (mask) {
      const int l = __ffsll((unsigned long long)mask) - 1;
      const int m_tiles = __shfl(mt, l), first = before + __shfl(incl, l) - m_tiles;
      const int slo = __shfl(lo, l), shi = __shfl(hi, l);
      // the segment's 32-row blocks dealt evenly to its tiles
      const int blocks = (shi - slo + 31) / 32, t = mi - first;
      const int b0 = (int)((int64_t)blocks * t / m_tiles);
      const int b1 = (int)((int64_t)blocks * (t + 1) / m_tiles);
      s = base + l;
      m0 = slo + 32 * b0;
      m_end = slo + 32 * b1 < shi ? slo + 32 * b1 : shi;
      break;
    }
    before += __shfl(incl, 63);
  }
  s = __builtin_amdgcn_readfirstlane(s);
  m0 = __builtin_amdgcn_readfirstlane(m0);
  m_end = __builtin_amdgcn_readfirstlane(m_end);
  const int rows = m_end - m0;
  if (rows > 224) fp8_tile<EPI, 8>(p, smem, s, nt, m0, m_end);
  else if (rows > 192) fp8_tile<EPI, 7>(p, smem, s, nt, m0, m_end);
  else if (rows > 160) fp8_tile<EPI, 6>(p, smem, s, nt, m0, m_end);
  else if (rows > 128) fp8_tile<EPI, 5>(p, smem, s, nt, m0, m_end);
  else if (rows > 96) fp8_tile<EPI, 4>(p, smem, s, nt, m0, m_end);
  else if (rows > 64) fp8_tile<EPI, 3>(p, smem, s, nt, m0, m_end);
  else if (rows > 32) fp8_tile<EPI, 2>(p, smem, s, nt, m0, m_end);
  else fp8_tile<EPI, 1>(p, smem, s, nt, m0, m_end);
}

}  // namespace

bool fp8_tiled_supported(int64_t ld_a, int64_t a_rows, int64_t total_rows, int K,
                         const uint16_t* c) {
  return K <= kMaxK && a_rows * ld_a < ((int64_t)1 << 32) && total_rows < ((int64_t)1 << 30) &&
         (reinterpret_cast<uintptr_t>(c) & 15) == 0;
}

hipError_t launch_grouped_gemm_fp8_tiled(const uint8_t* a, int64_t ld_a, int64_t a_rows,
                                         const float* a_scale, const int32_t* src_row,
                                         const int32_t* seg_offsets, int num_segments,
                                         int64_t total_rows, const uint8_t* w,
                                         const float* w_scale, int K, int n_out, int epilogue,
                                         uint16_t* c, hipStream_t stream) {
  const int n_tiles =
      (epilogue == NT_MOE_EPI_SWIGLU ? 2 * n_out : n_out) / 32 / kTileBlocks;
  const int64_t upper = (total_rows / kMaxRows + num_segments) * n_tiles;
  const unsigned grid = (unsigned)((upper + 7) / 8 * 8);
  const F8Args p{a, ld_a, a_rows, a_scale, src_row, seg_offsets, num_segments, (int)total_rows,
                 w, w_scale, K, n_out, c};
  auto kern = epilogue == NT_MOE_EPI_SWIGLU ? fp8_tiled_gemm_kernel<NT_MOE_EPI_SWIGLU>
              : epilogue == NT_MOE_EPI_RELU2 ? fp8_tiled_gemm_kernel<NT_MOE_EPI_RELU2>
                                             : fp8_tiled_gemm_kernel<NT_MOE_EPI_NONE>;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 2 * kStageBytes, stream, p);
  return hipGetLastError();
}

}  // namespace ntmoe
