// Grouped expert GEMM, packed bf16 weights, few rows per segment (decode batches and short
// prompts), with the shared expert's product in the same launch.
//
// The products of grouped_gemm_packed.hip bit for bit (same packed layout, K slices and epilogue
// arithmetic). That kernel's tile of 128 rows x 256 weight rows on persistent workgroups is made
// for full row tiles; with a few rows per expert the time is the weight stream's, and there it
// had one K step of weights in flight per wave, eight or sixteen workgroups in all for one token
// or for the shared expert alone, and a tile list to scan before the first load. Here:
//   * one workgroup per (segment, 128 packed weight rows): it reads two offsets and leaves if the
//     segment is empty; nothing is scanned. A segment of more than 128 rows is dealt, in even
//     chunks of whole 32-row blocks, to the kSplitM workgroups of its weight rows;
//   * wave w streams packed block w of the tile (4 KB per 64-wide K step) into a register ring,
//     D steps ahead: 6, 4 or 2 for chunks of 32, 64 and 128 rows, as the accumulators allow;
//   * the chunk's token rows go through LDS in a ring of the same depth (direct-to-LDS copies,
//     16-byte chunks XOR-swizzled by row), one barrier per step;
//   * the outputs are transposed through that LDS, so stores write whole row segments.
// The shared expert is one more range of workgroups ahead of the routed ones (its rows are the
// batch, no gather; its widths may differ), so its few tiles overlap the routed weight stream
// instead of taking two launches on a few CUs.
//
// Measured, us up / down, that kernel -> this one (weights not in any cache): T3 cell (256
// experts, d 1280, H 320) 48 tokens 43 / 35 -> 31 / 29, 512 tokens 46 / 51 -> 40 / 40; 128 experts
// d 2048 H 768, 48 tokens 146 / 75 -> 134 / 69 (6.0 TB/s), 777 tokens 153 / 87 -> 146 / 85; 32
// experts d 1024 H 512, 48 tokens 18 / 12 -> 14 / 9. Whole forward at 48 tokens, T3 cell: see the
// dispatch rule (few_rows).
#include <math.h>

#include "common.h"

namespace ntmoe {
namespace {

typedef __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

constexpr int kBK = 64;                // K per step
constexpr int kRowBytes = kBK * 2;     // staged bytes per token row
constexpr int kBlockElems = 32 * kBK;  // packed weight block
constexpr int kTileBlocks = 4;         // packed blocks per workgroup (one per wave)
constexpr int kMaxRows = 128;          // token rows per chunk

template <int NJ>
constexpr int depth() { return NJ == 1 ? 6 : (NJ == 2 ? 4 : 2); }

__device__ __forceinline__ int swz8(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// Rows m0 .. m_end - 1 (at most 32 NJ) of one segment against packed blocks 4 nt .. 4 nt + 3 of
// its weights w (NB blocks).
template <int EPI, bool KEEP, int NJ>
__device__ __forceinline__ void few_tile(const FewPart& p, const uint16_t* w, unsigned char* smem,
                                         int nt, int m0, int m_end) {
  constexpr int D = depth<NJ>();
  constexpr int R = D + 1;
  constexpr int kStage = NJ * 32 * kRowBytes;
  constexpr bool SW = EPI == NT_MOE_EPI_SWIGLU;
  const int lane = lane_id(), wave = wave_id();
  const int li = lane & 31, half = lane >> 5;
  const int NB = (SW ? 2 * p.n_out : p.n_out) / 32;
  const int nk = p.K / kBK;
  const int nb = nt * kTileBlocks + wave;
  const bool live = nb < NB;  // a wave past the last block copies rows and takes the barriers
  const char* abase = reinterpret_cast<const char*>(p.a);

  uint32_t aoff[NJ];
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    const int row = (wave * NJ + q) * 8 + (lane >> 3);
    const int tok = m0 + row < m_end ? m0 + row : m_end - 1;
    int64_t r = p.src_row ? (int64_t)p.src_row[tok] : (int64_t)tok;
    r = r < 0 ? 0 : (r >= p.a_rows ? p.a_rows - 1 : r);
    aoff[q] = (uint32_t)(r * p.ld_a * 2) + (uint32_t)(swz8(row, lane & 7) << 4);
  }
  const uint16_t* wbase = w + (int64_t)(live ? nb : NB - 1) * nk * kBlockElems;
  const uint32_t b_lane = lane * 16;
  // Every step issues the same NJ row copies and 4 weight loads (past the last step re-reads of
  // it), so a wait counts a fixed number of operations.
  auto load = [&](int kb, int slot, u32x4 (&b)[4]) __attribute__((always_inline)) {
    const int kc = kb < nk ? kb : nk - 1;
#pragma unroll
    for (int q = 0; q < NJ; ++q)
      __builtin_amdgcn_global_load_lds(
          (gvoid*)(abase + (int64_t)kc * kRowBytes + aoff[q]),
          (lvoid*)(smem + slot * kStage + (wave * NJ + q) * 1024), 16, 0, 0);
    const uint16_t* blk = wbase + (int64_t)kc * kBlockElems;
    asm volatile("global_load_dwordx4 %0, %4, %5\n\t"
                 "global_load_dwordx4 %1, %4, %5 offset:1024\n\t"
                 "global_load_dwordx4 %2, %4, %5 offset:2048\n\t"
                 "global_load_dwordx4 %3, %4, %5 offset:3072"
                 : "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
                 : "v"(b_lane), "s"(blk)
                 : "memory");
  };
  // Waits for a step's rows and weights (the later steps' may stay in flight), naming its
  // weight registers.
  auto wait_for = [&](u32x4 (&b)[4]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%4)"
                 : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3])
                 : "n"((D - 1) * (NJ + 4))
                 : "memory");
  };
  int frag_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) frag_off[q] = li * kRowBytes + (swz8(li, 4 * half + q) << 4);

  floatx16 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = floatx16{};
  u32x4 wq[R][4];
  static_for<0, D>([&](auto i_c) __attribute__((always_inline)) {
    load(decltype(i_c)::value, decltype(i_c)::value, wq[decltype(i_c)::value]);
  });
  wait_for(wq[0]);

  // The products of K step kb from LDS slot `slot` and weights bc.
  auto multiply = [&](int slot, const u32x4 (&bc)[4]) __attribute__((always_inline)) {
    const unsigned char* st = smem + slot * kStage;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const bf16x8 f = *reinterpret_cast<const bf16x8*>(st + j * 32 * kRowBytes + frag_off[q]);
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bc[q]), f,
                                                         acc[j], 0, 0, 0);
      }
  };
  // Barrier: every wave's copies of this step have landed (its own wait) and its reads of the
  // slot that is refilled next are complete.
  auto meet = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  int kb = 0;
  for (; kb + R <= nk; kb += R)
    static_for<0, R>([&](auto u_c) __attribute__((always_inline)) {
      constexpr int u = decltype(u_c)::value;
      meet();
      load(kb + u + D, (u + D) % R, wq[(u + D) % R]);
      multiply(u, wq[u]);
      wait_for(wq[(u + 1) % R]);
    });
  // All loads land and their registers are named; the steps left (fewer than R) are in the ring.
  static_for<0, R>([&](auto u_c) __attribute__((always_inline)) {
    u32x4(&b)[4] = wq[decltype(u_c)::value];
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3])
                 :
                 : "memory");
  });
  meet();
  static_for<0, D>([&](auto u_c) __attribute__((always_inline)) {
    constexpr int u = decltype(u_c)::value;
    if (kb + u < nk) multiply(u, wq[u]);
  });
  meet();  // the ring's LDS is free

  // Lane (token li, half h) holds 8 consecutive output columns in elements 0-7 and (SwiGLU: the
  // value half of the same columns) in 8-15; the tile's outputs are laid row-major in LDS, 16-byte
  // chunks XOR-swizzled by row.
  constexpr int kCols = SW ? 64 : 128;
  constexpr int kChunks = kCols / 8;
  auto ooff = [](int r, int c) {
    return r * kCols * 2 + ((c ^ (SW ? (r >> 1) & 7 : r & 15)) << 4);
  };
  if (live) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = 32 * j + li;
#pragma unroll
      for (int st = 0; st < (SW ? 1 : 2); ++st) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if constexpr (SW) {
            const float a = acc[j][i], u = acc[j][8 + i];
            v[i] = a * u * __builtin_amdgcn_rcpf(1.f + __expf(-a));
          } else {
            const float a = acc[j][8 * st + i];
            v[i] = EPI == NT_MOE_EPI_RELU2 ? (a > 0.f ? a * a : 0.f) : a;
          }
        }
        *reinterpret_cast<u32x4*>(smem + ooff(r, SW ? wave * 2 + half : wave * 4 + st * 2 + half)) =
            u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                  pack_bf16x2(v[6], v[7])};
        if constexpr (KEEP) {  // the fc1 pre-activations, straight from the accumulators
          if (m0 + r < m_end) {
            const int col = SW ? nb * 16 + 8 * half : nb * 32 + 16 * st + 8 * half;
            uint16_t* prow = p.pre + (int64_t)(m0 + r) * (SW ? 2 : 1) * p.n_out + col;
#pragma unroll
            for (int h = 0; h < (SW ? 2 : 1); ++h) {
              const int e0 = SW ? 8 * h : 8 * st;
              *reinterpret_cast<u32x4*>(prow + h * p.n_out) =
                  u32x4{pack_bf16x2(acc[j][e0], acc[j][e0 + 1]),
                        pack_bf16x2(acc[j][e0 + 2], acc[j][e0 + 3]),
                        pack_bf16x2(acc[j][e0 + 4], acc[j][e0 + 5]),
                        pack_bf16x2(acc[j][e0 + 6], acc[j][e0 + 7])};
            }
          }
        }
      }
    }
  }
  __syncthreads();
  const int col0 = nt * kCols;
  for (int i = threadIdx.x; i < NJ * 32 * kChunks; i += 256) {
    const int r = i / kChunks, ch = i % kChunks;
    const u32x4 v = *reinterpret_cast<const u32x4*>(smem + ooff(r, ch));
    if (m0 + r < m_end && col0 + ch * 8 < p.n_out)
      *reinterpret_cast<u32x4*>(p.c + (int64_t)(m0 + r) * p.n_out + col0 + ch * 8) = v;
  }
}

__host__ __device__ inline int few_n_tiles(int n_out, int epilogue) {
  return ((epilogue == NT_MOE_EPI_SWIGLU ? 2 * n_out : n_out) / 32 + kTileBlocks - 1) / kTileBlocks;
}

// Workgroup b runs on XCD b mod 8. With spread = 8 (8 segments and more) segment s is XCD s mod
// 8's, so the workgroups that read the same token rows share an L2 (777 tokens over 128 experts:
// up 186 -> 146 us, down 108 -> 85 us); with fewer segments spread = 1: the whole chip takes
// each one's weight rows.
template <int EPI, bool KEEP>
__global__ __launch_bounds__(256, 3) void few_gemm_kernel(FewPart routed,
                                                          const int32_t* __restrict__ seg_offsets,
                                                          int S, int total_rows, int split_m,
                                                          int spread,
                                                          FewPart shared, int shared_rows,
                                                          int shared_blocks) {
  extern __shared__ __align__(16) unsigned char smem[];
  int b = blockIdx.x;
  const bool is_shared = b < shared_blocks;
  const FewPart& p = is_shared ? shared : routed;
  const int n_tiles = few_n_tiles(p.n_out, EPI);
  const uint16_t* w = p.w;
  int lo, hi, chunk, chunks_by;  // rows, this workgroup's first chunk and its step
  if (is_shared) {
    lo = 0;
    hi = shared_rows;
    chunk = b / n_tiles;
    chunks_by = shared_blocks / n_tiles;
  } else {
    b -= shared_blocks;
    const int first = b % spread;
    b /= spread;
    const int sc = b / n_tiles, s = sc / split_m * spread + first;
    if (s >= S) return;
    chunk = sc % split_m;
    chunks_by = split_m;
    lo = seg_offsets[s];
    hi = seg_offsets[s + 1];
    lo = lo < 0 ? 0 : (lo > total_rows ? total_rows : lo);
    hi = hi < lo ? lo : (hi > total_rows ? total_rows : hi);
    w += (int64_t)s * (EPI == NT_MOE_EPI_SWIGLU ? 2 : 1) * p.n_out * p.K;
  }
  const int nt = b % n_tiles;
  const int blocks = (hi - lo + 31) / 32, chunks = (hi - lo + kMaxRows - 1) / kMaxRows;
  for (; chunk < chunks; chunk += chunks_by) {
    const int m0 = lo + 32 * (int)((int64_t)blocks * chunk / chunks);
    const int end = lo + 32 * (int)((int64_t)blocks * (chunk + 1) / chunks);
    const int m_end = end < hi ? end : hi;
    const int rows = m_end - m0;
    if (rows > 64) few_tile<EPI, KEEP, 4>(p, w, smem, nt, m0, m_end);
    else if (rows > 32) few_tile<EPI, KEEP, 2>(p, w, smem, nt, m0, m_end);
    else few_tile<EPI, KEEP, 1>(p, w, smem, nt, m0, m_end);
    __syncthreads();  // the next chunk's copies reuse the LDS
  }
}

constexpr size_t few_lds() {
  return (size_t)kRowBytes * 32 * (4 * (depth<4>() + 1) > 2 * (depth<2>() + 1) ? 4 * (depth<4>() + 1)
                                                                              : 2 * (depth<2>() + 1));
}
static_assert(few_lds() >= (size_t)kMaxRows * 256 && few_lds() >= 32u * kRowBytes * (depth<1>() + 1),
              "rings and the output tile fit");

template <int EPI, bool KEEP>
hipError_t launch_few(const FewPart& routed, const int32_t* seg_offsets, int S, int64_t total_rows,
                      const FewPart* shared, int64_t shared_rows, hipStream_t stream) {
  // Workgroups per (segment, weight rows): enough for a segment of four times the mean.
  const int64_t mean = (total_rows + S - 1) / S;
  const int64_t want = (4 * mean + kMaxRows - 1) / kMaxRows;
  const int split_m = (int)(want > 4 ? 4 : want);
  const int64_t sh = shared && shared_rows > 0
                         ? (shared_rows + kMaxRows - 1) / kMaxRows * few_n_tiles(shared->n_out, EPI)
                         : 0;
  const int spread = S >= 8 ? 8 : 1;
  const int64_t grid =
      sh + ((int64_t)S + spread - 1) / spread * spread * few_n_tiles(routed.n_out, EPI) * split_m;
  if (grid >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  auto kern = few_gemm_kernel<EPI, KEEP>;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), few_lds(), stream, routed, seg_offsets,
                     S, (int)total_rows, split_m, spread, shared ? *shared : routed, (int)shared_rows, (int)sh);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_grouped_gemm_bf16_few(const FewPart& routed, const int32_t* seg_offsets,
                                        int num_segments, int64_t total_rows,
                                        const FewPart* shared, int64_t shared_rows, int epilogue,
                                        hipStream_t stream) {
  const bool keep = routed.pre != nullptr;
  switch (epilogue) {
    case NT_MOE_EPI_SWIGLU:
      return keep ? launch_few<NT_MOE_EPI_SWIGLU, true>(routed, seg_offsets, num_segments,
                                                        total_rows, shared, shared_rows, stream)
                  : launch_few<NT_MOE_EPI_SWIGLU, false>(routed, seg_offsets, num_segments,
                                                         total_rows, shared, shared_rows, stream);
    case NT_MOE_EPI_RELU2:
      return keep ? launch_few<NT_MOE_EPI_RELU2, true>(routed, seg_offsets, num_segments,
                                                       total_rows, shared, shared_rows, stream)
                  : launch_few<NT_MOE_EPI_RELU2, false>(routed, seg_offsets, num_segments,
                                                        total_rows, shared, shared_rows, stream);
    default:
      return launch_few<NT_MOE_EPI_NONE, false>(routed, seg_offsets, num_segments, total_rows,
                                                shared, shared_rows, stream);
  }
}

}  // namespace ntmoe
