// Grouped expert GEMM, packed bf16 weights, few rows per segment (decode batches and short
// prompts), with the shared expert's product in the same launch.
//
// The products of grouped_gemm_packed.hip bit for bit (same packed layout, K slices and epilogue
// arithmetic). That kernel's tile of 128 rows x 256 weight rows on persistent workgroups is made
// for full row tiles; with a few rows per expert the time is the weight stream's, and there it
// had one K step of weights in flight per wave, eight or sixteen workgroups in all for one token
// or for the shared expert alone, and a tile list to scan before the first load. Here:
//   * one workgroup per (segment, 128 packed weight rows): it reads two offsets and leaves if the
//     segment is empty; nothing is scanned. A segment of more than 128 rows is cut into even chunks
//     of whole 32-row blocks: its workgroup takes the first one, and the others have workgroups of
//     their own, which find theirs by a scan of the offsets;
//   * wave w streams packed block w of the tile (4 KB per 64-wide K step) into a register ring,
//     D steps ahead: 6, 4 or 2 for chunks of 32, 64 and 128 rows, as the accumulators allow;
//   * the chunk's token rows go through LDS in a ring of the same depth (direct-to-LDS copies,
//     16-byte chunks XOR-swizzled by row), one barrier per step;
//   * the outputs are transposed through that LDS, so stores write whole row segments.
// The shared expert is one more range of workgroups ahead of the segments' (its rows are the
// batch, no gather; its widths may differ), so its few tiles overlap the routed weight stream
// instead of taking two launches on a few CUs.
//
// Measured, us up / down, that kernel -> this one (weights not in any cache): T3 cell (256
// experts, d 1280, H 320) 48 tokens 43 / 35 -> 31 / 29, 512 tokens 46 / 51 -> 40 / 40; 128 experts
// d 2048 H 768, 48 tokens 146 / 75 -> 134 / 69 (6.0 TB/s), 777 tokens 153 / 87 -> 146 / 85; 32
// experts d 1024 H 512, 48 tokens 18 / 12 -> 14 / 9. Whole forward at 48 tokens, T3 cell (with the
// shared expert in the same launches): 185 -> 104 us of GPU time.
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
// tail_blocks workgroups each take one chunk past the first of a segment that has more than one
// (routing that favours a few experts), weight rows fastest, an eighth of that list per XCD; without
// such segments they read the offsets and leave. With the segment's own workgroups walking those
// chunks, 8192 rows of one of 256 experts (K 1280, 320 outputs) took 775 us and 8 x 1024 rows 102;
// this way both take 21 (the tiled kernel 27), and 32 rows of every expert 46 (45; tiled 54). One
// chunk each and no loop: the state of a loop around the tile spills. The first kFront of them lead
// the grid, so long segments start at once (at its end 32 experts, K 1024, 4 x 256 rows take 17.5 us,
// in front 14.0, tiled 16.3; 128 experts, K 2048, lognormal rows 180, 171 and 171); the others end
// it: all in front would keep the even case's workgroups out of the CUs for an offset read (777
// tokens of 128 experts, 576 and 768 of them, 287.8 -> 291.2 us a forward).
constexpr int kFront = 256;

template <int EPI, bool KEEP>
__global__ __launch_bounds__(256, 3) void few_gemm_kernel(FewPart routed,
                                                          const int32_t* __restrict__ seg_offsets,
                                                          int S, int total_rows, int spread,
                                                          FewPart shared, int shared_rows,
                                                          int shared_blocks, int tail_blocks) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int front = tail_blocks < kFront ? tail_blocks : kFront;
  const int own = (int)gridDim.x - tail_blocks;  // workgroups of the shared expert and the segments
  int b = (int)blockIdx.x - front;
  const int tail = b < 0 ? (int)blockIdx.x : (b < own ? -1 : (int)blockIdx.x - own);
  const bool is_shared = tail < 0 && b < shared_blocks;
  const FewPart& p = is_shared ? shared : routed;
  const int n_tiles = few_n_tiles(p.n_out, EPI);
  auto clamped = [&](int o) { return o < 0 ? 0 : (o > total_rows ? total_rows : o); };
  int s = 0, lo = 0, hi = shared_rows, chunk = 0, chunks, nt;
  if (is_shared) {
    chunk = b / n_tiles;
    nt = b % n_tiles;
    chunks = (hi + kMaxRows - 1) / kMaxRows;
  } else if (tail < 0) {
    b -= shared_blocks;
    const int first = b % spread;
    b /= spread;
    s = b / n_tiles * spread + first;
    nt = b % n_tiles;
    if (s >= S) return;
    lo = clamped(seg_offsets[s]);
    hi = clamped(seg_offsets[s + 1]);
    if (hi <= lo) return;
    chunks = (hi - lo + kMaxRows - 1) / kMaxRows;
  } else {
    // Lane l holds segments per l .. per l + per - 1: their chunks past the first, added up over
    // the lanes; the lane whose share holds the item's chunk finds it among its segments.
    constexpr int kPer = (NT_MOE_MAX_SEGMENTS + 63) / 64;
    const int per = (S + 63) / 64, lane = lane_id();
    int off[kPer + 1], sum = 0;
#pragma unroll
    for (int i = 0; i <= kPer; ++i) {
      const int at = lane * per + i;
      off[i] = i <= per ? clamped(seg_offsets[at < S ? at : S]) : 0;
    }
    auto later = [&](int i) {
      return i < per && off[i + 1] > off[i] ? (off[i + 1] - off[i] - 1) / kMaxRows : 0;
    };
#pragma unroll
    for (int i = 0; i < kPer; ++i) sum += later(i);
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o);
      if (lane >= o) incl += u;
    }
    const int64_t all = (int64_t)__builtin_amdgcn_readlane(incl, 63) * n_tiles;
    const int64_t item = all * (tail % 8) / 8 + tail / 8;
    if (item >= all * (tail % 8 + 1) / 8) return;
    const int at = (int)(item / n_tiles);
    nt = (int)(item % n_tiles);
    const int k = __builtin_ctzll(__ballot(at < incl));
    int r = at - (incl - sum), fs = 0, fl = 0, fh = 0, fc = 0, fn = 1;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int n = later(i);
      if (r >= 0 && r < n) {
        fs = lane * per + i;
        fl = off[i];
        fh = off[i + 1];
        fc = r + 1;
        fn = n + 1;
      }
      r -= n;
    }
    s = __builtin_amdgcn_readlane(fs, k);
    lo = __builtin_amdgcn_readlane(fl, k);
    hi = __builtin_amdgcn_readlane(fh, k);
    chunk = __builtin_amdgcn_readlane(fc, k);
    chunks = __builtin_amdgcn_readlane(fn, k);
  }
  const uint16_t* w = p.w + (int64_t)s * (EPI == NT_MOE_EPI_SWIGLU ? 2 : 1) * p.n_out * p.K;
  const int blocks = (hi - lo + 31) / 32;
  const int m0 = lo + 32 * (int)((int64_t)blocks * chunk / chunks);
  const int end = lo + 32 * (int)((int64_t)blocks * (chunk + 1) / chunks);
  const int m_end = end < hi ? end : hi;
  const int rows = m_end - m0;
  if (rows > 64) few_tile<EPI, KEEP, 4>(p, w, smem, nt, m0, m_end);
  else if (rows > 32) few_tile<EPI, KEEP, 2>(p, w, smem, nt, m0, m_end);
  else few_tile<EPI, KEEP, 1>(p, w, smem, nt, m0, m_end);
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
  const int n_tiles = few_n_tiles(routed.n_out, EPI);
  const int64_t sh = shared && shared_rows > 0
                         ? (shared_rows + kMaxRows - 1) / kMaxRows * few_n_tiles(shared->n_out, EPI)
                         : 0;
  const int spread = S >= 8 ? 8 : 1;
  // A workgroup for every chunk past the first that there can be (the segments' rows are not known
  // here): n segments of r rows in all have at most (r - 1) / kMaxRows of them.
  const int64_t tail = ((total_rows - 1) / kMaxRows * n_tiles + 7) / 8 * 8;
  const int64_t grid = sh + ((int64_t)S + spread - 1) / spread * spread * n_tiles + tail;
  if (grid >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  auto kern = few_gemm_kernel<EPI, KEEP>;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), few_lds(), stream, routed, seg_offsets,
                     S, (int)total_rows, spread, shared ? *shared : routed, (int)shared_rows,
                     (int)sh, (int)tail);
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
