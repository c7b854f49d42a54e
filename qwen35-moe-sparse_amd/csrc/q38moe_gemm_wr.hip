// Grouped down-form GEMM with the weights in registers (R7, R9; e4m3: R14): Y[r, c] = bf16(A[r] . W[c])
// over each group's sorted rows, for rows of 256 to 512 bytes (K of 128 to 256 bf16 or 256 to 512 e4m3
// values). Such a product is bound by writing Y (2 N bytes per row): the kernel's work is to keep the
// stores streaming.
//
// A workgroup (8 waves, one per CU) takes 512 columns of one group; each wave keeps 64 of their weight
// rows, all of K, in MFMA operand registers (128 VGPRs at 512 bytes) and multiplies every row tile by
// them. Row tiles of 64 rows go through an LDS ring, copied whole rows at a time (2 KB of 512-byte rows
// per wave and instruction pair) three tiles ahead, so per tile there are one barrier, 32 fragment reads
// per wave for 128 MFMAs, and 8 stores of whole 128-byte lines. grouped_gemm_kernel<MODE_DOWN> copies
// both operands of every 256 x 256 unit in 64-byte pieces behind a barrier per 32 K, which takes 66 of
// its 72 us at configuration 2 even with every operand in L2.
//
// Work: the (group, 512-column block, 64-row tile) units in that order, cut into one equal run per
// workgroup, so there is no partial last round; a run that crosses into the next (group, column block)
// reloads the weights through the ring. Runs are spread over the XCDs contiguously, so that the
// workgroups that share a group's rows and weights share an L2.
//
// Measured (launched alone): h = 1024, I = 256, 16384 tokens top-5 of 64 + shared 75 -> 61 us (3.3 TB/s of
// Y; with the stores taken out 51 us, the MFMAs at the clock the chip holds under them about 35), e4m3
// h = 2048, I = 512, 32768 tokens 277-286 -> 220 us (174 us without stores; the weights, loaded once per
// run and group, 26). Output through lane swaps instead of the LDS staging measured the same to 3 us
// slower, storing the second wave of each SIMD half a tile late the same (e4m3 10 us slower).
#include "q38moe_common.h"
#include "q38moe_kernels.h"

namespace q38 {
namespace {

constexpr int WR_WAVES = 8;
constexpr int WR_THREADS = 64 * WR_WAVES;
constexpr int WR_ROWS = 64;                  // rows per tile
constexpr int WR_NCW = 64;                   // columns per wave
constexpr int WR_NC = WR_NCW * WR_WAVES;     // columns per workgroup
constexpr int WR_NS = 4;                     // ring slots: copies run three tiles ahead
constexpr int WR_STORES = 8;                 // store instructions per wave and tile
constexpr int WR_GROUPS = 65;                // 64 experts and the shared expert

struct WrParams {
  const uint8_t* A;           // rows of KB bytes
  const int4* tiles;          // {group (E = shared expert), row0, rows, -} (group -1: unused); nullptr = M rows
  const int32_t* ntiles_dev;  // used entries of tiles
  int max_mtiles;             // entries that tiles holds
  int64_t M;
  const uint8_t* W;           // [E, N, K]
  const uint8_t* Ws;          // shared expert [N, K]
  uint16_t* C;                // [*, N]
  int N, E;
  const float* a_scale;       // e4m3: per row
  const float* w_scale;       // e4m3: [E, N]
  const float* ws_scale;      // e4m3: shared expert [N]
};

// Asynchronous copies from inline asm (M0 = the wave's LDS base; lane l lands at + 16 l or + 4 l): the
// compiler does not see them, and the explicit waits below order them.
__device__ __forceinline__ uint32_t wr_lds(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p);
}
__device__ __forceinline__ void wr_dma16(const void* gsrc, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(gsrc)
               : "memory", "m0");
}
__device__ __forceinline__ void wr_dma4(const void* gsrc, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 1\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(gsrc)
               : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wr_wait() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's LDS reads and writes
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wr_barrier() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ f32x4_t wr_mfma_fp8(i32x8_t a, i32x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// Position of 16-byte chunk c of row r: the 16 rows of a fragment read cover the 64 banks once. Rows a
// multiple of 256 bytes apart differ in the low four bits of their chunk, rows an odd multiple of 128
// apart in three (their parity does the rest).
template <int KB>
__device__ __forceinline__ int wr_swz(int r) {
  return KB % 256 == 0 ? r & 15 : (r >> 1) & 7;
}

// KS: 64-byte steps of K (32 bf16 or 64 e4m3 values).
template <bool FP8, int KS>
__global__ __launch_bounds__(WR_THREADS, 2) void gemm_wr_kernel(WrParams p) {
  constexpr int KB = 64 * KS;                                 // bytes per row
  constexpr int SLOT = WR_ROWS * KB;
  constexpr int CP = SLOT / 16 / WR_THREADS + (FP8 ? 1 : 0);  // copies per wave and tile (e4m3: + row scales)
  constexpr int AHEAD = WR_NS - 1;
  static_assert(KS % 2 == 0 && SLOT % (16 * WR_THREADS) == 0, "whole copies per wave");
  __shared__ __attribute__((aligned(16))) uint8_t ring[WR_NS * SLOT];
  __shared__ __attribute__((aligned(16))) uint8_t stage_all[WR_WAVES][16 * 128];
  __shared__ __attribute__((aligned(16))) float sc_all[FP8 ? WR_WAVES : 1][FP8 ? WR_NS : 1][WR_ROWS];
  __shared__ int g_row0[WR_GROUPS], g_rows[WR_GROUPS], g_pre[WR_GROUPS + 1];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, E = p.E;

  // Each group's rows from the tile table (a group's tiles cover one contiguous run of rows).
  if (tid < WR_GROUPS) {
    const bool dense = tid == E && p.tiles == nullptr;
    g_row0[tid] = dense ? 0 : 0x7fffffff;
    g_rows[tid] = dense ? (int)p.M : 0;
  }
  __syncthreads();
  if (p.tiles != nullptr) {
    const int used = load_uniform(p.ntiles_dev);  // its round trip overlaps the entries'
    for (int i = tid; i < p.max_mtiles; i += WR_THREADS) {
      const int4 t = p.tiles[i];
      if (i < used && t.x >= 0 && t.x <= E) {
        atomicMin(&g_row0[t.x], t.y);
        atomicAdd(&g_rows[t.x], t.z);
      }
    }
    __syncthreads();
  }
  const int ncb = (N + WR_NC - 1) / WR_NC;
  if (wave == 0) {
    // Exclusive prefix sums of the groups' units.
    const int n = (lane <= E ? (g_rows[lane] + WR_ROWS - 1) / WR_ROWS : 0) * ncb;
    int s = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(s, o);
      if (lane >= o) s += v;
    }
    g_pre[lane] = s - n;
    if (lane == 63) {
      g_pre[64] = s;
      g_pre[65] = s + (E == 64 ? (g_rows[64] + WR_ROWS - 1) / WR_ROWS * ncb : 0);
    }
  }
  __syncthreads();
  const int G = (int)gridDim.x, b = (int)blockIdx.x;
  const int wslot = (G & 7) == 0 ? (b & 7) * (G >> 3) + (b >> 3) : b;
  const int64_t total = g_pre[WR_GROUPS];
  int pos = __builtin_amdgcn_readfirstlane((int)(total * wslot / G));
  const int end = __builtin_amdgcn_readfirstlane((int)(total * (wslot + 1) / G));

  uint8_t* const stage = stage_all[wave];
  const uint32_t ring_lds = wr_lds(ring);
  // Per-lane fragment offsets in a slot (or weight half): chunk 4 s + lq of row 16 f + lr lies at
  // fo[s % FOP] + 64 FOP (s / FOP) + 16 KB f, since the swizzle only touches the chunk's low bits.
  constexpr int FOP = KB % 256 == 0 ? 4 : 2;
  uint32_t fo[FOP];
#pragma unroll
  for (int i = 0; i < FOP; ++i) fo[i] = lr * KB + (((4 * i + lq) ^ wr_swz<KB>(lr)) << 4);

  while (pos < end) {
    // The pair holding `pos`: the last group that starts at or before it (a group without rows starts
    // where its successor does, so it is never the last).
    int g = __builtin_popcountll(ballot64(g_pre[lane] <= pos)) - 1;
    if (g_pre[64] <= pos) g = 64;
    g = __builtin_amdgcn_readfirstlane(g);
    const int row0 = __builtin_amdgcn_readfirstlane(g_row0[g]);
    const int rows = __builtin_amdgcn_readfirstlane(g_rows[g]);
    const int ntile = (rows + WR_ROWS - 1) / WR_ROWS;
    const int off = pos - __builtin_amdgcn_readfirstlane(g_pre[g]);
    const int cb = off / ntile, t0 = off - cb * ntile;
    const int t1 = min(ntile, t0 + end - pos);
    pos += t1 - t0;
    const int n0 = cb * WR_NC + wave * WR_NCW;  // this wave's first column
    const bool active = n0 < N;                 // N is a multiple of 64

    // This wave's 64 weight rows, 16 at a time (one fragment row each) through the two halves of its
    // eighth of the ring (the previous run's copies were waited for before the barrier that ended it).
    u32x4_t wf[4][KS];
    f32x4_t sw[FP8 ? 4 : 1];
    if (active) {
      constexpr int QI = 16 * KB / 1024;  // copies per quarter
      static_assert(WR_NS * SLOT / WR_WAVES == 2 * 16 * KB, "two quarters fill an eighth of the ring");
      const uint8_t* wsrc = (g < E ? p.W + (int64_t)g * N * KB : p.Ws) + (int64_t)n0 * KB;
      const int mine = wave * (WR_NS * SLOT / WR_WAVES);
      auto fetch = [&](int q) {
#pragma unroll
        for (int i = 0; i < QI; ++i) {
          const int id = 64 * i + lane, r = id / (KB / 16), c = (id % (KB / 16)) ^ wr_swz<KB>(r);
          wr_dma16(wsrc + (int64_t)(16 * q + r) * KB + 16 * c, ring_lds + mine + (q & 1) * 16 * KB + 1024 * i);
        }
      };
      fetch(0);
      fetch(1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < 3) wr_wait<QI>();
        else wr_wait<0>();
#pragma unroll
        for (int s = 0; s < KS; ++s)
          wf[q][s] = ld16(ring + mine + (q & 1) * 16 * KB + fo[s % FOP] + 64 * FOP * (s / FOP));
        if (q < 2) {
          __builtin_amdgcn_s_waitcnt(0xC07F);  // read before the next copies land
          fetch(q + 2);
        }
      }
      if constexpr (FP8) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const float* src = (g < E ? p.w_scale + (int64_t)g * N : p.ws_scale) + n0 + 16 * n + 4 * lq;
          sw[n] = *reinterpret_cast<const f32x4_t*>(src);
        }
      }
      wr_wait<0>();
    } else {
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int s = 0; s < KS; ++s) wf[n][s] = u32x4_t{0, 0, 0, 0};
    }
    wr_barrier();

    // Copies of row tile t: rows past the group's end copy its last row. Past the run's end the last
    // tile is copied again, so that every step issues the same copies and waits with one constant.
    auto issue = [&](int t) {
      const int tt = min(t, t1 - 1), slot = (t - t0) & (WR_NS - 1);
      const uint8_t* base = p.A + (int64_t)(row0 + WR_ROWS * tt) * KB;
      const int last = rows - 1 - WR_ROWS * tt;
#pragma unroll
      for (int i = 0; i < SLOT / 16 / WR_THREADS; ++i) {
        const int id = i * WR_THREADS + tid, r = id / (KB / 16), c = (id % (KB / 16)) ^ wr_swz<KB>(r);
        wr_dma16(base + (uint32_t)(min(r, last) * KB + 16 * c),
                 ring_lds + slot * SLOT + 16 * (i * WR_THREADS + 64 * wave));
      }
      if constexpr (FP8)
        wr_dma4(p.a_scale + row0 + WR_ROWS * tt + min(lane, last), wr_lds(&sc_all[wave][slot][0]));
    };
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) issue(t0 + t);

    // A half tile's products (32 rows), and its way out: lane l of block (f, n) holds row 16 f + l % 16,
    // columns 16 n + 4 (l / 16) .. + 3; 16 rows x 64 columns at a time go through the wave's staging area
    // (chunk c of row r at c ^ ((r >> 1) & 7)) and leave as two stores of 8 rows x 128 bytes each,
    // streamed (the combine reads Y once). Rows past the group's end repeat its last row, values and
    // address, so every half tile issues WR_STORES / 2 stores.
    f32x4_t acc[2][4];
    float sa[2];
    auto multiply = [&](int t, int h) {
      const int slot = (t - t0) & (WR_NS - 1);
      const uint8_t* const rows_lds = ring + slot * SLOT + 32 * KB * h;
      constexpr int SPF = FP8 ? 2 : 1;  // 64-byte steps per MFMA
      constexpr int FH = 2 * KS / SPF;  // fragments (step, 16-row block), read WIN ahead of their MFMAs
      constexpr int WIN = 2;
      u32x4_t win[WIN][SPF];
      auto read = [&](int i) {
#pragma unroll
        for (int j = 0; j < SPF; ++j) {
          const int s = (i >> 1) * SPF + j;
          win[i % WIN][j] = ld16(rows_lds + fo[s % FOP] + 64 * FOP * (s / FOP) + 16 * KB * (i & 1));
        }
      };
#pragma unroll
      for (int i = 0; i < WIN; ++i) read(i);
      if constexpr (FP8) {
#pragma unroll
        for (int f = 0; f < 2; ++f) sa[f] = sc_all[wave][slot][32 * h + 16 * f + lr];
      }
      __builtin_amdgcn_sched_group_barrier(0x100, WIN * SPF + (FP8 ? 2 : 0), 0);
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[f][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < FH; ++i) {
        const int f = i & 1, s = (i >> 1) * SPF;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          // e4m3: one 128-byte step per MFMA, a lane taking 16 bytes of each half in both operands.
          if constexpr (FP8)
            acc[f][n] = wr_mfma_fp8(cat8(wf[n][s], wf[n][s + SPF - 1]), cat8(win[i % WIN][0], win[i % WIN][SPF - 1]), acc[f][n]);
          else
            acc[f][n] = mfma16x16x32(wf[n][s], win[i % WIN][0], acc[f][n]);
        }
        if (i + WIN < FH) read(i + WIN);
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);  // a fragment's MFMAs, then the window's read
        if (i + WIN < FH) __builtin_amdgcn_sched_group_barrier(0x100, SPF, 0);
      }
    };
    auto leave = [&](int t, int h) {
      const int last = rows - 1 - WR_ROWS * t;
      uint8_t* const cbase = reinterpret_cast<uint8_t*>(p.C + (int64_t)(row0 + WR_ROWS * t) * N + n0);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          f32x4_t v = acc[f][n];
          if constexpr (FP8) v = v * (sw[n] * sa[f]);
          const int ch = 2 * n + (lq >> 1);
          *reinterpret_cast<uint2*>(stage + lr * 128 + ((ch ^ ((lr >> 1) & 7)) << 4) + 8 * (lq & 1)) =
              make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int r = 8 * j + (lane >> 3), ch = lane & 7;
          const u32x4_t d = ld16(stage + r * 128 + ((ch ^ ((r >> 1) & 7)) << 4));
          st16_stream(cbase + ((uint32_t)min(32 * h + 16 * f + r, last) * (uint32_t)(2 * N) + 16 * ch), d);
        }
      }
    };

    for (int t = t0; t < t1; ++t) {
      // Tile t's copies of this wave are done when at most what it issued after them is outstanding:
      // the stores of the AHEAD tiles before t and the copies of the AHEAD - 1 tiles after it (the
      // first tiles have fewer stores behind them). The barrier publishes every wave's copies and
      // retires the slot that tile t + AHEAD refills.
      constexpr int C2 = (AHEAD - 1) * CP;
      if (!active || t == t0) wr_wait<C2>();
      else if (t == t0 + 1) wr_wait<C2 + WR_STORES>();
      else if (t == t0 + 2) wr_wait<C2 + 2 * WR_STORES>();
      else wr_wait<C2 + AHEAD * WR_STORES>();
      wr_barrier();
      issue(t + AHEAD);
      if (!active) continue;
      multiply(t, 0);
      leave(t, 0);
      multiply(t, 1);
      leave(t, 1);
    }
    // The copies past the run's end have landed (the last tile's stores follow them) and every wave has
    // read its tiles before the ring is reused (or released).
    if (active) wr_wait<WR_STORES>();
    else wr_wait<0>();
    wr_barrier();
  }
}

template <bool FP8>
hipError_t launch_wr(const WrParams& p, int kb, hipStream_t stream) {
  const dim3 grid((unsigned)device_cus()), block(WR_THREADS);
  switch (kb) {
    case 256: hipLaunchKernelGGL((gemm_wr_kernel<FP8, 4>), grid, block, 0, stream, p); break;
    case 384: hipLaunchKernelGGL((gemm_wr_kernel<FP8, 6>), grid, block, 0, stream, p); break;
    case 512: hipLaunchKernelGGL((gemm_wr_kernel<FP8, 8>), grid, block, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

bool gemm_wr_supported(int kb) { return kb == 256 || kb == 384 || kb == 512; }

hipError_t launch_down_wr(const void* A, const int4* tiles, const int32_t* ntiles_dev, int max_mtiles,
                          int64_t M_dense, const void* W, const void* Ws, uint16_t* C, int N, int kb, int E,
                          const float* a_scale, const float* w_scale, const float* ws_scale, hipStream_t stream) {
  if (E > WR_GROUPS - 1 || N % 64 != 0) return hipErrorInvalidValue;
  const WrParams p{static_cast<const uint8_t*>(A), tiles, ntiles_dev, max_mtiles, M_dense,
                   static_cast<const uint8_t*>(W), static_cast<const uint8_t*>(Ws), C, N, E, a_scale, w_scale, ws_scale};
  return a_scale != nullptr ? launch_wr<true>(p, kb, stream) : launch_wr<false>(p, kb, stream);
}

}  // namespace q38
