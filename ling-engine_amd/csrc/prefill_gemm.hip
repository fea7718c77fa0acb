// Block-scaled FP8 prefill GEMM on gfx950 MFMA, and the 1x128 FP8 activation quantizer that feeds it.
//
//   y[m][n] = bf16( sum_kb (sum_{k in kb} e4m3(xq[m][k]) * e4m3(wq[n][k])) * xs[m][kb] * ws[n/128][kb] )
//
// xq: FP8 E4M3 activations [M][K] (row-major) with one FP32 scale per 1x128 group, xs [M][K/128];
// wq: FP8 E4M3 weights in the tiled layout the skinny GEMMs stream (reference
// src/core/stream_gemm.cu:705-738), with one FP32 scale per 128x128 block, ws [N/128][K/128].
//
// Design:
//  * One v_mfma_f32_16x16x128_f8f6f4 per 16x16 output tile per 128-value K block: an MFMA covers exactly one
//    scale block, so its FP32 result is scaled once and added to the accumulator (one FMA per output per
//    block). Any permutation of K inside the block is harmless, since A and B use the same one.
//  * Weights are the A operand (rows n) and activations the B operand (columns m). A workgroup (8 waves, 2 per
//    SIMD: 2 along the weights x 4 along the tokens) computes 256 weight rows x 256 tokens; each wave 128 x 64
//    (8 x 4 MFMA tiles, 128 accumulator registers). A wave's 128 weight rows are one weight scale block, so
//    the block scale is a scalar and each lane's scale is that scalar times its token's activation scale.
//  * Operands reach LDS without passing through registers: buffer loads with the LDS flag write each lane's
//    16 bytes at the next 16 bytes of a 1 KB run, and the lane-to-source map implements the layout: a K
//    block of a 256-row operand is [row][8 x 16-byte units] with the unit index XOR-swizzled by the row, so
//    the fragment reads are bank-conflict free. The block's activation scales come along the same way.
//  * Two LDS stages (65 KB each): while a K block is computed from one, the next block's loads fill the
//    other. The waits are explicit: the compiler cannot see which LDS bytes a load-to-LDS writes.
//  * Tile order: each XCD works through a contiguous range of a grouped raster (kGroupN weight tiles x every
//    token tile per group), so the workgroups running at once on an XCD share the K slices of both operands
//    in its L2 instead of re-streaming the whole activation matrix per weight tile.
//  * That is prefill_fp8_kernel, for products of many tiles (a last round of few tiles is split along K, the parts
//    exchanged as FP32 partials). prefill_tile_kernel computes products whose 256 x 256 tiles would leave CUs without
//    work, in tiles of 64 x 64 to 128 x 128 with two to four LDS stages; choose_tile picks.
#include "lq_common.hpp"
#include "lq_prefill_offsets.hpp"
#include "lq_workspace.hpp"

#include <algorithm>
#include <limits>
#include <string>
#include <type_traits>

namespace lq {
namespace {

constexpr int kBN = 256;  // weight rows per workgroup
constexpr int kBM = 256;  // tokens per workgroup
constexpr int kThreads = 512;
constexpr int kGroupN = 8;                       // weight tiles per raster group (config 4: 2-6 % faster than 2, 4 or 16)
constexpr int kMaxSplit = 4;                     // K parts of a tail tile
constexpr int kRowBytes = 128;                   // one K block of one row (FP8)
constexpr int kOpBytes = 256 * kRowBytes;        // one operand's K block in LDS: 32 KB
constexpr int kStage = 2 * kOpBytes + kBM * 4;   // weights, activations, activation scales: 65 KB

// The place of 16-byte unit u of row `row` in an LDS operand tile: units are XOR-swizzled by the row, so that the 16-byte
// fragment reads (lane (r, t): row r, a unit that depends on t) are free of bank conflicts. What the counters of several
// swizzles agree on is that the LDS serves such a read 16 lanes at a time, lanes 0-3, 12-15, 20-23 and 24-27 of each 32 and
// then the others: rows 0-3 and 12-15 of one t with rows 4-11 of the next. So swz serves reads of unit 2t or 2t + 1, swz_w those of
// unit t or 4 + t, each with no conflict, and also if 8 or 16 lanes in a row were served together; reads of unit t under
// swz are two-way conflicts, as those of unit 2t under a swizzle by row / 2 are (half of all LDS cycles). Weights under
// swz_w are faster in the 256 x 256 tile (1000 x 5120 x 17408 110.2 -> 108.1 us, 2048 x 7168 x 5120 82.7 -> 81.8), under swz in the
// smaller ones, where the conflicts are hidden and swz_w costs more than it saves, in its loads (428 x 7168 x 5120 28.7, 29.2
// us, 1500 x 2048 x 4096 22.0, 23.2; three more swizzles without conflicts likewise).
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }
__device__ __forceinline__ int swz_w(int row) {
  return ((((row >> 2) ^ (row >> 3)) & 1) << 2) | (((row >> 3) & 1) << 1) | ((row >> 1) & 1);
}
__device__ __forceinline__ int lds_off(int row, int unit) { return row * kRowBytes + (unit << 4); }

// The fragment of row `row` for lanes with K 32 t .. + 32 of a block: units 2t, 2t + 1 of an activation row, units t,
// 4 + t of a weight row. A weight row's units are kept in the order of the tiled block (16-byte pieces t of its first half,
// then of its second): four lanes of a load then read one run of 64 bytes, where units in K order made them read two runs
// of 32, at half the rate (512 x 5120 x 5120 in 128 x 128 tiles 35.0 -> 30.8 us, 200 x 7168 x 5120 22.3 -> 21.0).
__device__ __forceinline__ i32x8 fragment(const uint8_t* op, int row, int u0, int u1) {
  const u32x4 lo = *reinterpret_cast<const u32x4*>(op + lds_off(row, u0));
  const u32x4 hi = *reinterpret_cast<const u32x4*>(op + lds_off(row, u1));
  return i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}
// sw: the weights' swizzle of the row, swz_w (256 x 256 tile) or swz.
__device__ __forceinline__ i32x8 fragment_w(const uint8_t* op, int row, int t, int sw) {
  return fragment(op, row, t ^ sw, (4 + t) ^ sw);
}
__device__ __forceinline__ i32x8 fragment_x(const uint8_t* op, int row, int t) {
  return fragment(op, row, (2 * t) ^ swz(row), (2 * t + 1) ^ swz(row));
}

struct PrefillArgs {
  const uint8_t* xq;
  const float* xs;  // block-scaled: activation group scales [M][K/128]
  const uint8_t* w;
  const float* ws;  // block-scaled: weight block scales [N/128][K/128]
  float alpha;      // per-tensor: the one scale (input scale x weight scale)
  void* y;          // BF16 or FP32 [M][ldy]
  int ldy, M, N, K, KB;
  int tiles_m, tiles_n;
  // Tail split: tiles [full, full + rem) of the logical order are each computed by S workgroups over
  // consecutive K ranges; their FP32 partials meet in part[(rt * S + p) * kBN * kBM] and the last part to
  // arrive (counter cnt[rt]) adds them in part order and writes the tile.
  int full, rem, S;
  float* part;
  int* cnt;
};

// Output of a prefill GEMM: BF16, FP32, or FP32 added to what y holds.
enum PrefillOut { kOutBf16 = 0, kOutF32 = 1, kOutF32Acc = 2 };

typedef __attribute__((address_space(3))) void* lds_ptr;

// soff is uniform over the wave; saying so keeps it in an SGPR (held in a VGPR, the compiler wraps every load in a
// loop over the lanes' distinct values).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds), 16, voff, __builtin_amdgcn_readfirstlane(soff), 0, 0);
}
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds), 4, voff, __builtin_amdgcn_readfirstlane(soff), 0, 0);
}
// s_waitcnt with only vmcnt / lgkmcnt constrained (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8])
#define LQ_WAIT_VM0() __builtin_amdgcn_s_waitcnt(0x0f70)
#define LQ_WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(0xc07f)

// Four outputs of one token, columns n .. n + 3.
template <bool BLOCK, int OUT>
__device__ __forceinline__ void put_out(const PrefillArgs& a, int m, int n, f32x4 v) {
  if constexpr (!BLOCK) v = f32x4{v[0] * a.alpha, v[1] * a.alpha, v[2] * a.alpha, v[3] * a.alpha};
  const size_t o = static_cast<size_t>(m) * a.ldy + n;
  if constexpr (OUT == kOutBf16) {
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + o) =
        u32x2{f32_to_bf16(v[0]) | (uint32_t(f32_to_bf16(v[1])) << 16),
              f32_to_bf16(v[2]) | (uint32_t(f32_to_bf16(v[3])) << 16)};
  } else {
    f32x4* dst = reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + o);
    if constexpr (OUT == kOutF32Acc) {
      const f32x4 old = *dst;
      v = f32x4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
    }
    *dst = v;
  }
}

// A weight block's scale as a scalar load: `p` is uniform over the wave and constant during the launch. (As a vector
// load it is counted with the loads to LDS, in order: its use waits for every operand load issued before it.)
__device__ __forceinline__ float scalar_load(const float* p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) float*>(reinterpret_cast<uintptr_t>(p));
}

// BLOCK: the block-scaled form (each 128-value block's product scaled by its activation and weight scales and
// folded into the accumulators); else one scale for the whole product, applied at the end, and the MFMAs
// accumulate across K themselves.
template <bool BLOCK, int OUT>
__global__ void __launch_bounds__(kThreads) prefill_fp8_kernel(const PrefillArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, t = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;  // the wave's 128-row weight half and 64-token quarter

  // Tile order. The hardware places block b on XCD b % 8; each XCD takes a contiguous range of the logical
  // tile order, in which tiles come in groups of kGroupN weight tiles x all token tiles, token tile slowest
  // within a group.
  // Split workgroups come after the whole tiles (the hardware dispatches in order, so they fill the last,
  // partial round); the S parts of a tile are on one XCD (same blockIdx % 8), sharing its L2.
  const int b = blockIdx.x;
  int tile = b, kb0 = 0, kb1 = a.KB, part = -1, rt = 0;
  if (b < a.full) {
    if ((a.full & 7) == 0) tile = (b & 7) * (a.full >> 3) + (b >> 3);
  } else {
    const int sidx = b - a.full, q = sidx >> 3;
    rt = (q / a.S) * 8 + (sidx & 7);
    part = q % a.S;
    if (rt >= a.rem) return;
    tile = a.full + rt;
    kb0 = part * a.KB / a.S;
    kb1 = (part + 1) * a.KB / a.S;
  }
  const int grp = tile / (kGroupN * a.tiles_m), rem = tile % (kGroupN * a.tiles_m);
  const int gsize = min(kGroupN, a.tiles_n - grp * kGroupN);
  const int tn = grp * kGroupN + rem % gsize, tm = rem / gsize;
  const int n0 = tn * kBN, m0 = tm * kBM;

  // Buffer resources sized to the operands: loads past the end (rows past N or M) return nothing.
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.w), 0, a.N * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.xq), 0, a.M * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t sr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.xs), 0, a.M * a.KB * 4, 0x00020000);

  // Load-to-LDS plan: load i (0..3) of wave w writes LDS bytes [((i * 8 + w) * 64 + lane) * 16, +16) of an
  // operand tile: row = (i * 8 + w) * 8 + lane / 8, swizzled unit lane % 8, i.e. source unit lane % 8 ^ swz(row)
  // (the same for every i, as i moves the row by 64, a multiple of 16). The per-i and per-block steps go in the scalar
  // offset, which stays within the operands (lq_prefill_offsets.hpp; choose_tile gives ones of fewer than kWholeRows rows to
  // the other tiles).
  const int row0 = wave * 8 + (lane >> 3), uw = (lane & 7) ^ swz_w(row0), ux = (lane & 7) ^ swz(row0);
  const unsigned wsrc = weight_unit_offset(n0 + row0, uw, a.KB), xsrc = activation_unit_offset(m0 + row0, ux, a.K);
  const unsigned step = 64u * static_cast<unsigned>(a.K);  // 64 rows, of either operand
  const unsigned xlast = last_load_offset(a.M, step);
  // activation scales: waves 0-3 load one token's scale per lane
  const int srow = wave * 64 + lane;
  const int ssrc = (wave < 4 && m0 + srow < a.M) ? (m0 + srow) * a.KB * 4 : static_cast<int>(0x80000000u);

  // A block's loads come in 5 parts (weights 0-1, 2-3, activations 0-1, 2-3, scales), issued one per tile
  // rather than in one burst, which would stall the waves on a full memory queue.
  auto issue_part = [&](int st, int kb, int part) {
    uint8_t* base = smem + st * kStage;
    if (part < 2) {
#pragma unroll
      for (int i = 2 * part; i < 2 * part + 2; ++i)
        dma16(wr, base + (i * 8 + wave) * 1024, wsrc, kb * kTileBytesFp8 + i * step);
    } else if (part < 4) {
#pragma unroll
      for (int i = 2 * (part - 2); i < 2 * (part - 2) + 2; ++i)
        dma16(xr, base + kOpBytes + (i * 8 + wave) * 1024, xsrc, kb * kRowBytes + (i < 3 ? i * step : xlast));
    } else if (BLOCK && wave < 4) {
      dma4(sr, base + 2 * kOpBytes + wave * 256, ssrc, kb * 4);
    }
  };
  auto issue = [&](int st, int kb) {
#pragma unroll
    for (int part = 0; part < 5; ++part) issue_part(st, kb, part);
  };

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // (a weight half past the end takes the last one's scales: its outputs are never stored)
  const float* wsrow = BLOCK ? a.ws + static_cast<size_t>(min((n0 >> 7) + wn, (a.N >> 7) - 1)) * a.KB : nullptr;

  // Fragment reads from an LDS stage: weight tile i (rows wn*128 + 16i + r) and token tile j (rows wm*64 + 16j
  // + r), 32 bytes at K 32t each.
  i32x8 bf[4], af;
  float sc[4];
  f32x4 pr[4];
  // B fragments, the lane's four block scales and the first A fragment of K block kb (stage st)
  float wnext = 0.f;  // the next block's weight scale, loaded a block ahead
  auto block_start = [&](int st) {
    const uint8_t* sa = smem + st * kStage;
    const float* sxs = reinterpret_cast<const float*>(sa + 2 * kOpBytes);
    af = fragment_w(sa, wn * 128 + r, t, swz_w(r));
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[j] = fragment_x(sa + kOpBytes, wm * 64 + 16 * j + r, t);
    if constexpr (BLOCK) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sc[j] = sxs[wm * 64 + 16 * j + r] * wnext;
    }
  };
  auto fold = [&](f32x4 (&dst)[4], const f32x4 (&p)[4], const float (&s)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[j][v] = __builtin_fmaf(p[j][v], s[j], dst[j][v]);
  };

  issue(0, kb0);
  LQ_WAIT_VM0();
  __builtin_amdgcn_s_barrier();
  if (BLOCK) wnext = scalar_load(wsrow + kb0);
  block_start(0);
  // Per K block and weight tile: the tile's four MFMAs, then the next tile's fragment read, then the fold of
  // the four results into the accumulators (the other wave on the SIMD issues its MFMAs meanwhile). The one
  // barrier per block sits after tile 7's MFMAs are issued: it publishes the next block's loads and frees this
  // block's stage for its refill. Empty volatile statements pin this order (the compiler would otherwise sink
  // the MFMAs to their use, hoist the reads and defer the folds, and run out of registers).
  for (int kb = kb0; kb < kb1; ++kb) {
    const int st = (kb - kb0) & 1;
    const uint8_t* sa = smem + st * kStage;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < 5 && kb + 1 < kb1) issue_part(st ^ 1, kb + 1, i);
      if (BLOCK && i == 0) wnext = scalar_load(wsrow + min(kb + 1, a.KB - 1));
      // the tile's MFMAs at raised issue priority: the SIMD's other wave gets the slots between them for its
      // folds and fragment reads (measured 1-2 % faster than equal priority)
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // (scales that are the constant 0 select the unscaled instruction, which needs no scale load before it: 2 % faster)
        if constexpr (BLOCK)
          pr[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[j], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0,
                                                                  0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[j], acc[i][j], 0, 0, 0, 0, 0, 0);
      }
      if constexpr (BLOCK)
        asm volatile("" ::"v"(pr[0]), "v"(pr[1]), "v"(pr[2]), "v"(pr[3]) : "memory");
      else
        asm volatile("" ::"v"(acc[i][0]), "v"(acc[i][1]), "v"(acc[i][2]), "v"(acc[i][3]) : "memory");
      __builtin_amdgcn_s_setprio(0);
      if (i < 7) {
        af = fragment_w(sa, wn * 128 + 16 * (i + 1) + r, t, swz_w(r));
      } else {
        // every wave's reads of this stage have returned and its loads of the next block have landed
        LQ_WAIT_LGKM0();
        LQ_WAIT_VM0();
        __builtin_amdgcn_s_barrier();
      }
      if constexpr (BLOCK) {
        asm volatile("" ::: "memory");
        fold(acc[i], pr, sc);
        asm volatile("" ::"v"(acc[i][0]), "v"(acc[i][1]), "v"(acc[i][2]), "v"(acc[i][3]));
      }
    }
    if (kb + 1 < kb1) block_start(st ^ 1);
  }

  if (part >= 0) {
    // A split tile: publish this part (agent-coherent stores: vector v = i * 4 + j of thread tid at
    // (v * kThreads + tid) * 16 bytes), count the arrival; the last part adds all parts in order.
    __shared__ int last_part;
    constexpr int kTileBytes = kBN * kBM * 4;
    const __amdgpu_buffer_rsrc_t pr_rs =
        __builtin_amdgcn_make_buffer_rsrc(a.part + static_cast<size_t>(rt) * a.S * (kBN * kBM), 0, a.S * kTileBytes,
                                          0x00020000);
    const int own = part * kTileBytes + static_cast<int>(threadIdx.x) * 16;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(acc[i][j], pr_rs, own + (i * 4 + j) * kThreads * 16, 0, 16 /* sc1 */);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(a.cnt + rt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_part = old == a.S - 1;
      if (last_part) __hip_atomic_store(a.cnt + rt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last_part) return;
    // sum over parts 0 .. S-1 in order, one weight tile (4 vectors x S parts) per batch of loads; this
    // workgroup's own part is in its registers
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f32x4 pv[kMaxSplit][4];
#pragma unroll
      for (int p = 0; p < kMaxSplit; ++p)
        if (p < a.S && p != part)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            pv[p][j] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                           pr_rs, p * kTileBytes + static_cast<int>(threadIdx.x) * 16 + (i * 4 + j) * kThreads * 16,
                           0, 16 /* sc1 */));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 sum = part == 0 ? acc[i][j] : pv[0][j];
#pragma unroll
        for (int p = 1; p < kMaxSplit; ++p)
          if (p < a.S) sum = sum + (p == part ? acc[i][j] : pv[p][j]);
        acc[i][j] = sum;
      }
    }
  }

  // epilogue: lane holds rows n = n0 + wn*128 + 16i + 4t + v, token m = m0 + wm*64 + 16j + r
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + wm * 64 + 16 * j + r;
    if (m >= a.M) continue;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int n = n0 + wn * 128 + 16 * i + 4 * t;
      if (n >= a.N) continue;
      put_out<BLOCK, OUT>(a, m, n, acc[i][j]);
    }
  }
}

// The smaller tiles: WN x WM waves of NI x NJ MFMA tiles each (a tile of TN = 16 NI WN weight rows x TM = 16 NJ WM
// tokens), for products whose 256 x 256 tiles would leave CUs without work. The arithmetic of an output is the same (its
// K blocks in order, each folded once), so which tile a shape gets changes no bit of an unsplit result.
//
// What bounds these is the way of the operands to the CU, not the MFMAs: with the loads to LDS taken out (and wrong
// results) 200 x 7168 x 5120 in 128 x 64 tiles takes 13.8 us instead of 21.1, without MFMAs 21.1, without the LDS reads
// 20.8. So the K loop is built around loads in flight: S stages of direct loads to LDS, of which S - 1 are on their way
// while one is multiplied. The fragments of block kb + 1 are read from LDS while block kb is multiplied (two register
// sets), spread with the loads over the block's weight tiles: issued in one burst ahead of the MFMAs they delayed them
// (26.5 us at 512 x 5120 x 5120 in 128 x 128 tiles, 32.6 with the bursts).
template <int NI, int NJ, int WN, int WM>
struct TileShape {
  static constexpr int kTN = 16 * NI * WN, kTM = 16 * NJ * WM, kNW = WN * WM;
  static constexpr int kLW = kTN * 8 / (64 * kNW), kLX = kTM * 8 / (64 * kNW);  // 16-byte loads per lane and stage
  static constexpr int kScale = (kTM > 64 * kNW ? kTM / 64 : kNW) * 256;  // a 256-byte run per wave
  static constexpr int kStageB = (kTN + kTM) * kRowBytes + kScale;
  static_assert(kLW * 64 * kNW == kTN * 8 && kLX * 64 * kNW == kTM * 8, "whole loads per wave");
  static_assert(128 % (16 * NI) == 0, "a wave's weight rows lie in one scale block");
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt holds at most 63");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

template <bool BLOCK, int OUT, int NI, int NJ, int WN, int WM, int S>
__global__ void __launch_bounds__(64 * WN * WM) prefill_tile_kernel(const PrefillArgs a) {
  using Sh = TileShape<NI, NJ, WN, WM>;
  constexpr int TN = Sh::kTN, TM = Sh::kTM, NW = Sh::kNW, LW = Sh::kLW, LX = Sh::kLX, STG = Sh::kStageB;
  constexpr int kVm = LW + LX + (BLOCK ? 1 : 0);  // loads per lane and stage (the scales': waves past TM tokens load none)
  static_assert(TM <= 64 * NW, "one scale per lane");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, t = lane >> 4;
  const int wn = wave % WN, wm = wave / WN;

  // Tile order: XCD b % 8 takes a contiguous range of the tiles; groups of kGroupN weight tiles x every token tile,
  // weight tiles fastest, so that a weight tile's readers run on one XCD, a little after one another.
  const int nb = gridDim.x, b = blockIdx.x, x = b & 7;
  const int tile = x * (nb >> 3) + min(x, nb & 7) + (b >> 3);
  const int grp = tile / (kGroupN * a.tiles_m), rem = tile % (kGroupN * a.tiles_m);
  const int gsize = min(kGroupN, a.tiles_n - grp * kGroupN);
  const int tn = grp * kGroupN + rem % gsize, tm = rem / gsize;
  const int n0 = tn * TN, m0 = tm * TM;

  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.w), 0, a.N * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.xq), 0, a.M * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t sr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.xs), 0, a.M * a.KB * 4, 0x00020000);

  // Load-to-LDS plan as in prefill_fp8_kernel: load i of wave w fills 8 rows from (i * NW + w) * 8. A row past the
  // operand gets an offset that is out of range by itself.
  unsigned wsrc[LW], xsrc[LX], ssrc = kLoadNothing;
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (i * NW + wave) * 8 + (lane >> 3), u = (lane & 7) ^ swz(row), n = n0 + row;
    wsrc[i] = n < a.N ? weight_unit_offset(n, u, a.KB) : kLoadNothing;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (i * NW + wave) * 8 + (lane >> 3), u = (lane & 7) ^ swz(row), m = m0 + row;
    xsrc[i] = m < a.M ? activation_unit_offset(m, u, a.K) : kLoadNothing;
  }
  if constexpr (BLOCK) {
    const int row = wave * 64 + lane;
    if (row < TM && m0 + row < a.M) ssrc = static_cast<unsigned>((m0 + row) * a.KB * 4);
  }
  // Loads [v0, v1) of a stage's kVm. (A block past the end is issued out of range: every wait count then holds on
  // every path.)
  auto issue_some = [&](int st, int kb, int v0, int v1) {
    const unsigned oob = kb < a.KB ? 0u : kLoadNothing;
    uint8_t* base = smem + st * STG;
#pragma unroll
    for (int v = v0; v < v1; ++v) {
      if (v < LW) dma16(wr, base + (v * NW + wave) * 1024, wsrc[v] | oob, block_offset(kb, a.KB, kTileBytesFp8));
      else if (v < LW + LX)
        dma16(xr, base + TN * kRowBytes + ((v - LW) * NW + wave) * 1024, xsrc[v - LW] | oob,
              block_offset(kb, a.KB, kRowBytes));
      else dma4(sr, base + (TN + TM) * kRowBytes + wave * 256, ssrc | oob, block_offset(kb, a.KB, 4));
    }
  };
  // all loads but those of the newest KEEP stages have landed
  auto wait_stages = [&](auto keep) {
    wait_vm<decltype(keep)::value * kVm>();
  };

  f32x4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nrow = n0 + wn * NI * 16;
  const float* wsrow = BLOCK ? a.ws + static_cast<size_t>(min(nrow, a.N - 1) >> 7) * a.KB : nullptr;
  struct Frags {
    i32x8 a[NI], b[NJ];
    float xs[NJ], ws;
  };
  // share i of NI of a block's fragment reads
  auto read_some = [&](Frags& f, int st, int kb, int i) {
    const uint8_t* sa = smem + st * STG;
    if constexpr (BLOCK) {
      if (i == 0) {
        const float* sxs = reinterpret_cast<const float*>(sa + (TN + TM) * kRowBytes);
#pragma unroll
        for (int j = 0; j < NJ; ++j) f.xs[j] = sxs[wm * NJ * 16 + 16 * j + r];
        f.ws = scalar_load(wsrow + min(kb, a.KB - 1));
      }
    }
    f.a[i] = fragment_w(sa, wn * NI * 16 + 16 * i + r, t, swz(r));
#pragma unroll
    for (int j = i * NJ / NI; j < (i + 1) * NJ / NI; ++j) f.b[j] = fragment_x(sa + TN * kRowBytes, wm * NJ * 16 + 16 * j + r, t);
  };

#pragma unroll
  for (int s = 0; s < S; ++s) issue_some(s, s, 0, kVm);
  Frags f0, f1;
  wait_stages(std::integral_constant<int, S - 1>{});
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NI; ++i) read_some(f0, 0, 0, i);
  // A block's products, one weight tile at a time; before(i) is issued ahead of tile i's MFMAs and tile i - 1's fold
  // behind them.
  auto multiply = [&](const Frags& cur, auto&& before) {
    float sc[NJ];
    f32x4 pr[2][NJ];
    if constexpr (BLOCK) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) sc[j] = cur.xs[j] * cur.ws;
    }
    auto fold = [&](int i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = __builtin_fmaf(pr[i & 1][j][v], sc[j], acc[i][j][v]);
    };
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      before(i);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if constexpr (BLOCK)
          pr[i & 1][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(cur.a[i], cur.b[j], f32x4{0.f, 0.f, 0.f, 0.f}, 0,
                                                                          0, 0, 0, 0, 0);
        else
          acc[i][j] =
              __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(cur.a[i], cur.b[j], acc[i][j], 0, 0, 0, 0, 0, 0);
      }
      if (BLOCK && i > 0) fold(i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (BLOCK) fold(NI - 1);
  };
  int st = 0;
  auto step = [&](Frags& cur, Frags& nxt, int kb) {
    const int st1 = st + 1 == S ? 0 : st + 1;
    // block kb + 1 has landed, and this wave has read its fragments of block kb; past the barrier every wave has,
    // so stage st takes block kb + S (the empty statements keep the reads on their side of the barrier)
    asm volatile("" ::: "memory");
    wait_stages(std::integral_constant<int, S - 2>{});
    LQ_WAIT_LGKM0();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(cur, [&](int i) {
      read_some(nxt, st1, kb + 1, i);
      issue_some(st, kb + S, i * kVm / NI, (i + 1) * kVm / NI);
    });
    st = st1;
  };
  // (two whole steps per round, the odd block after them: a branch between a block's instructions would part them)
  int kb = 0;
  for (; kb + 2 <= a.KB; kb += 2) {
    step(f0, f1, kb);
    step(f1, f0, kb + 1);
  }
  if (kb < a.KB) multiply(f0, [](int) {});
  LQ_WAIT_VM0();  // no load to LDS outlives the workgroup

#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int m = m0 + wm * NJ * 16 + 16 * j + r;
    if (m >= a.M) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = nrow + 16 * i + 4 * t;
      if (n < a.N) put_out<BLOCK, OUT>(a, m, n, acc[i][j]);
    }
  }
}

// 1x128 FP8 activation quantizer: 16 lanes per (row, 128-value group), eight values (16 bytes) per lane, so a
// wave covers four groups with 16-byte loads and 8-byte stores; s = amax / 448 (1 for an all-zero group),
// q = E4M3(x * (1 / s)) rounded to nearest even, the product and the reciprocal each rounded to FP32 (the
// reference's activation quantizer multiplies by the reciprocal of its scale too, src/core/prefill_gemm.cu:496-511;
// eight divisions per lane made this kernel VALU-bound: 19.4 against 15.5 us at 4096 x 5120). |x / s| <= 448 up
// to that rounding; clamped, which is the saturating conversion.
__global__ void __launch_bounds__(256) quant_fp8_g128_kernel(const uint16_t* __restrict__ x, int M, int K,
                                                             uint8_t* __restrict__ q, float* __restrict__ scale) {
  // blockIdx.x: 16 groups of a row; blockIdx.y + k gridDim.y: the rows (no integer division per thread)
  const int KB = K / 128;
  const int kb = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  const bool ok = kb < KB;  // the 16 lanes of a group agree
  for (int m = blockIdx.y; m < M; m += gridDim.y) {
    const size_t base = static_cast<size_t>(m) * K + static_cast<size_t>(kb) * 128 + 8 * sub;
    u32x4 raw = u32x4{0u, 0u, 0u, 0u};
    if (ok) raw = *reinterpret_cast<const u32x4*>(x + base);
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf16_to_f32(raw[i] & 0xffff);
      v[2 * i + 1] = bf16_to_f32(raw[i] >> 16);
    }
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[i]));
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    const float s = mx > 0.f ? mx / 448.f : 1.f;
    const float rs = 1.f / s;
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float a[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = fminf(fmaxf(v[4 * h + i] * rs, -448.f), 448.f);
      const uint32_t lo = __builtin_amdgcn_cvt_pk_fp8_f32(a[0], a[1], 0, false);
      w[h] = __builtin_amdgcn_cvt_pk_fp8_f32(a[2], a[3], lo, true);
    }
    if (ok) {
      *reinterpret_cast<u32x2*>(q + base) = u32x2{w[0], w[1]};
      if (sub == 0) scale[static_cast<size_t>(m) * KB + kb] = s;
    }
  }
}

// Per-tensor FP8 activation quantizer (reference src/core/prefill_gemm.cu:496-511): each value rounded to BF16
// first (production's activations are BF16), times 1 / input_scale, then E4M3 with saturation to +-448 (NaN
// stays NaN). Four values per thread.
// BF16IN: x holds BF16 values (reference quant_act_fp8_bf16in, prefill_gemm.cu:626-630): the same bytes as from the
// FP32 values they were rounded from.
template <bool BF16IN>
__global__ void __launch_bounds__(256) quant_fp8_pt_kernel(const void* __restrict__ x, size_t quads, float inv_scale,
                                                           uint8_t* __restrict__ q) {
  for (size_t i = blockIdx.x * static_cast<size_t>(256) + threadIdx.x; i < quads; i += static_cast<size_t>(gridDim.x) * 256) {
    float f[4];
    if constexpr (BF16IN) {
      const u32x2 h = reinterpret_cast<const u32x2*>(x)[i];
      f[0] = __uint_as_float(h.x << 16);
      f[1] = __uint_as_float(h.x & 0xffff0000u);
      f[2] = __uint_as_float(h.y << 16);
      f[3] = __uint_as_float(h.y & 0xffff0000u);
    } else {
      const f32x4 v4 = reinterpret_cast<const f32x4*>(x)[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = bf16_to_f32(f32_to_bf16(v4[k]));
    }
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float b = f[k] * inv_scale;
      v[k] = isnan(b) ? b : fminf(fmaxf(b, -448.f), 448.f);
    }
    const uint32_t lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
    const uint32_t w = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
    reinterpret_cast<uint32_t*>(q)[i] = w;
  }
}

template <bool BLOCK, int OUT, int NI, int NJ, int WN, int WM, int S>
int tile_launch(PrefillArgs a, const char* name, hipStream_t s) {
  using Sh = TileShape<NI, NJ, WN, WM>;
  a.tiles_m = cdiv(a.M, Sh::kTM);
  a.tiles_n = cdiv(a.N, Sh::kTN);
  constexpr int lds = S * Sh::kStageB;
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_tile_kernel<BLOCK, OUT, NI, NJ, WN, WM, S>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return fail(LQ_ERR_LAUNCH, std::string(name) + ": " + hipGetErrorString(attr));
  hipLaunchKernelGGL((prefill_tile_kernel<BLOCK, OUT, NI, NJ, WN, WM, S>),
                     dim3(static_cast<unsigned>(a.tiles_m) * static_cast<unsigned>(a.tiles_n)), dim3(64 * WN * WM), lds, s, a);
  return check_launch(name);
}

// The tile of a product, by an estimate of its time. `single` is what a K block of a tile costs on a CU that has one
// (microseconds, weights from memory), `pair` what one of two resident tiles' costs together; the larger the tile, the
// less each output costs, but tiles come in whole numbers per CU, so a product with few of them is done sooner in
// smaller ones. A launch costs 4 us; a split last round of 256 x 256 tiles 10 us more and 0.07 us per part, for the
// exchange. The smallest sum wins, the 256 x 256 tile unless another is 5 % better or an operand has too few rows for its
// loads' offsets (kWholeRows). Measured, block-scaled (M x N x K,
// us, rotating over 500 MB of weights): 200 x 2048 x 4096 32 -> 12 (64 x 64), 200 x 7168 x 5120 42 -> 22 (128 x 64),
// 300 x 5120 x 17408 83 -> 72 (128 x 64), 512 x 5120 x 5120 45 -> 34 (128 x 128), 1500 x 5120 x 17408 238 -> 153 (128 x 128
// x2); 1000 x 5120 x 17408 stays at 114 (133 in 128 x 128 x2) and 500 x 17408 x 5120 at 83 (80 in 128 x 128 x2).
//
// The constants are the block-scaled form's. The estimates are 0.8-1.3 of what was measured (per tensor, which has no
// folds, 0.6-1.1), but the order is what counts: over nine matrices and M = 200 .. 4096 the tile taken is on average 1.0 %
// (per tensor 1.8 %) slower than the fastest of the five, at worst 20 % (256 x 4224 x 7552: 35.5 in 128 x 64, 29.6 in 64 x 64),
// and never slower than 256 x 256. 64 x 128 (15 % faster at 300 x 5120 x 17408, 10 % slower elsewhere) and 128 x 256 (7 %
// faster at 777 x 5120 x 6144, 9 % slower at 256 x 17408 x 5120) were not worth their kernels.
enum PrefillTile { kT256x256, kT64x64, kT128x64, kT128x128, kT128x128x2 };  // x2: two stages, two tiles per CU
PrefillTile choose_tile(const PrefillArgs& a, long long cus) {
  constexpr double kLaunch = 4., kSplit = 10., kPart = 0.07, kBig = 1.72;
  double best = kLaunch + a.KB * kBig * static_cast<double>((a.full + cus - 1) / cus);
  if (a.rem) best += kBig * a.KB / a.S + kSplit + kPart * a.rem * a.S;
  best *= 0.95;
  if (a.M < kWholeRows || a.N < 256) best = std::numeric_limits<double>::infinity();
  PrefillTile tile = kT256x256;
  struct Kind {
    PrefillTile tile;
    int tn, tm;
    double single, pair;
  };
  for (const Kind& k : {Kind{kT64x64, 64, 64, 0.275, 0.52}, Kind{kT128x64, 128, 64, 0.44, 0.74},
                        Kind{kT128x128, 128, 128, 0.65, 1.3}, Kind{kT128x128x2, 128, 128, 0.85, 1.02}}) {
    const long long n = (static_cast<long long>(cdiv(a.N, k.tn)) * cdiv(a.M, k.tm) + cus - 1) / cus;
    const double us = kLaunch + a.KB * (static_cast<double>(n / 2) * k.pair + static_cast<double>(n % 2) * k.single);
    if (us < best) {
      best = us;
      tile = k.tile;
    }
  }
  return tile;
}

// The 256 x 256 tiles of a product: when they leave the last round of one-tile-per-CU workgroups at most a third full, the
// tiles of that round are each split along K into S parts (S <= #CUs / rem, each part >= 8 K blocks, S <= 4).
// Measured on config 4: down (64 of 256 CUs busy in the last round, S = 4) gains 8%; a half-full last round
// (gate|up, S would be 2) loses 4% to the partial traffic, as the clock rises when CUs idle.
void split_last_round(PrefillArgs& a, long long cus) {
  a.KB = a.K / 128;
  a.tiles_m = cdiv(a.M, kBM);
  a.tiles_n = cdiv(a.N, kBN);
  const long long tiles = static_cast<long long>(a.tiles_m) * a.tiles_n;
  a.rem = static_cast<int>(tiles % cus);
  a.S = a.rem ? static_cast<int>(std::min<long long>({cus / a.rem, a.KB / 8, kMaxSplit})) : 1;
  if (a.S < 3) {
    a.S = 1;
    a.rem = 0;
  }
  a.full = static_cast<int>(tiles - a.rem);
}

template <bool BLOCK, int OUT>
int prefill_launch(PrefillArgs a, const char* name, hipStream_t s) {
  const std::string nm(name);
  if (a.N <= 0 || a.K <= 0 || a.N % 128 != 0 || a.K % 128 != 0)
    return fail(LQ_ERR_SHAPE, "prefill_gemm: N % 128 and K % 128 must be 0");
  if (a.M < 1) return LQ_OK;  // nothing to do (the reference returns silently)
  if (a.ldy < a.N || a.ldy % 4 != 0) return fail(LQ_ERR_SHAPE, nm + ": ldy must be >= N and a multiple of 4");
  // operand byte offsets are 32-bit
  if (static_cast<long long>(a.N) * a.K >= (1LL << 31) || static_cast<long long>(a.M) * a.K >= (1LL << 31))
    return fail(LQ_ERR_SHAPE, nm + ": N * K and M * K must be below 2^31");
  if (!a.xq || !a.w || !a.y || (BLOCK && (!a.xs || !a.ws))) return fail(LQ_ERR_ARG, nm + ": null pointer");
  if (reinterpret_cast<uintptr_t>(a.y) % (OUT == kOutBf16 ? 8 : 16) != 0)
    return fail(LQ_ERR_ARG, nm + ": y must be 8-byte (BF16) or 16-byte (FP32) aligned");
  int dev = 0;
  (void)hipGetDevice(&dev);
  const long long P = device_cus(dev);
  split_last_round(a, P);
  switch (choose_tile(a, P)) {
    case kT64x64: return tile_launch<BLOCK, OUT, 2, 2, 2, 2, 4>(a, name, s);
    case kT128x64: return tile_launch<BLOCK, OUT, 4, 2, 2, 2, 3>(a, name, s);
    case kT128x128: return tile_launch<BLOCK, OUT, 4, 4, 2, 2, 4>(a, name, s);
    case kT128x128x2: return tile_launch<BLOCK, OUT, 4, 4, 2, 2, 2>(a, name, s);
    default: break;
  }
  const long long blocks = a.full + (a.rem ? 8LL * cdiv(a.rem, 8) * a.S : 0);
  if (a.rem) {
    // rem * S <= P partial tiles: the bound is reserved once per device (lq_init, or here on first use) and never
    // reallocated, so a graph captured with these pointers stays valid whatever shapes run later
    Workspace* ws = workspace_for_current_device();
    if (!ws) return LQ_ERR_DEVICE;
    const int rc = reserve_prefill_scratch(ws);
    if (rc) return rc;
    a.part = ws->pf_partials;
    a.cnt = ws->pf_counters;
  }
  // 130 KB of dynamic LDS is above the default per-launch limit; raise it (once per instantiation).
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_fp8_kernel<BLOCK, OUT>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kStage);
  if (attr != hipSuccess) return fail(LQ_ERR_LAUNCH, nm + ": " + hipGetErrorString(attr));
  hipLaunchKernelGGL((prefill_fp8_kernel<BLOCK, OUT>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 2 * kStage,
                     s, a);
  return check_launch(name);
}

}  // namespace

int reserve_prefill_scratch(Workspace* ws) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  const size_t P = static_cast<size_t>(device_cus(dev));
  return ws->reserve_prefill(P * kBN * kBM * sizeof(float), P);
}

}  // namespace lq

using namespace lq;

extern "C" {

// Test hook (not part of the interface): the tile of a product on `cus` CUs, 8 * PrefillTile + the parts along K of a tile
// of the last round (1: not split).
int lq_debug_prefill_fp8_tile(int M, int N, int K, int cus) {
  PrefillArgs a{};
  a.M = M;
  a.N = N;
  a.K = K;
  split_last_round(a, cus);
  const PrefillTile tile = choose_tile(a, cus);
  return 8 * tile + (tile == kT256x256 ? a.S : 1);
}

int lq_quant_act_fp8_g128(const uint16_t* x, int M, int K, uint8_t* q, float* scale, void* stream) {
  if (M < 1 || K <= 0 || K % 128 != 0) return fail(LQ_ERR_SHAPE, "quant_act_fp8_g128: M >= 1 and K % 128 == 0");
  if (!x || !q || !scale) return fail(LQ_ERR_ARG, "quant_act_fp8_g128: null pointer");
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(q) % 8 != 0)
    return fail(LQ_ERR_ARG, "quant_act_fp8_g128: x must be 16-byte and q 8-byte aligned");
  const unsigned rows = static_cast<unsigned>(std::min(M, 65535));
  hipLaunchKernelGGL(quant_fp8_g128_kernel, dim3(static_cast<unsigned>((K / 128 + 15) / 16), rows), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, M, K, q, scale);
  return check_launch("quant_act_fp8_g128");
}

int lq_prefill_fp8_block(const uint8_t* xq, const float* xs, int M, const uint8_t* w, const float* ws, uint16_t* y,
                         int ldy, int N, int K, void* stream) {
  PrefillArgs a{};
  a.xq = xq;
  a.xs = xs;
  a.w = w;
  a.ws = ws;
  a.y = y;
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  return prefill_launch<true, kOutBf16>(a, "prefill_gemm", static_cast<hipStream_t>(stream));
}

int lq_quant_act_fp8(const float* x, int M, int K, float input_scale, uint8_t* q, void* stream) {
  if (M < 1 || K <= 0 || K % 4 != 0) return fail(LQ_ERR_SHAPE, "quant_act_fp8: M >= 1 and K % 4 == 0");
  if (!x || !q) return fail(LQ_ERR_ARG, "quant_act_fp8: null pointer");
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(q) % 4 != 0)
    return fail(LQ_ERR_ARG, "quant_act_fp8: x must be 16-byte and q 4-byte aligned");
  const size_t quads = static_cast<size_t>(M) * K / 4;
  const unsigned grid = static_cast<unsigned>(std::min<size_t>((quads + 255) / 256, 256 * 64));
  hipLaunchKernelGGL(quant_fp8_pt_kernel<false>, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream), x, quads,
                     1.f / input_scale, q);
  return check_launch("quant_act_fp8");
}

int lq_quant_act_fp8_bf16in(const uint16_t* x, int M, int K, float input_scale, uint8_t* q, void* stream) {
  if (M < 1 || K <= 0 || K % 4 != 0) return fail(LQ_ERR_SHAPE, "quant_act_fp8_bf16in: M >= 1 and K % 4 == 0");
  if (!x || !q) return fail(LQ_ERR_ARG, "quant_act_fp8_bf16in: null pointer");
  if (reinterpret_cast<uintptr_t>(x) % 8 != 0 || reinterpret_cast<uintptr_t>(q) % 4 != 0)
    return fail(LQ_ERR_ARG, "quant_act_fp8_bf16in: x must be 8-byte and q 4-byte aligned");
  const size_t quads = static_cast<size_t>(M) * K / 4;
  const unsigned grid = static_cast<unsigned>(std::min<size_t>((quads + 255) / 256, 256 * 64));
  hipLaunchKernelGGL(quant_fp8_pt_kernel<true>, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream), x, quads,
                     1.f / input_scale, q);
  return check_launch("quant_act_fp8_bf16in");
}

int lq_prefill_gemm_fp8(const uint8_t* xq, int M, const uint8_t* w, float alpha, float* y, int ldy, int N, int K,
                        int accumulate, void* stream) {
  PrefillArgs a{};
  a.xq = xq;
  a.w = w;
  a.alpha = alpha;
  a.y = y;
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return accumulate ? prefill_launch<false, kOutF32Acc>(a, "prefill_gemm_fp8", s)
                    : prefill_launch<false, kOutF32>(a, "prefill_gemm_fp8", s);
}

int lq_prefill_gemm_fp8_bf16out(const uint8_t* xq, int M, const uint8_t* w, float alpha, uint16_t* y, int ldy, int N,
                                int K, void* stream) {
  PrefillArgs a{};
  a.xq = xq;
  a.w = w;
  a.alpha = alpha;
  a.y = y;
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  return prefill_launch<false, kOutBf16>(a, "prefill_gemm_fp8_bf16out", static_cast<hipStream_t>(stream));
}

}  // extern "C"
