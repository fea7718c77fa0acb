// NVFP4 prefill GEMMs on gfx950 (reference prefill_gemm_nvfp4 / prefill_swiglu_nvfp4, src/core/prefill_gemm.cu:
// 269-342, 593-704):
//
//   y[m][n] = alpha * sum_k (e2m1(xq[m][k]) * e4m3(xs[m][k/16])) * (e2m1(w[n][k]) * e4m3(ws[n][k/16]))   (+= y)
//
// and the FFN's gate|up form, whose output goes straight into the down projection's NVFP4 encoding:
//   v = BF16(silu(alpha_g * G) * (alpha_u * U)), then NVFP4 blocks of 16 output columns (as quant_act_nvfp4).
//
// CDNA4 has no MFMA that takes E4M3 scales per 16 values (its block-scaled MFMAs take E8M0 per 32), so both
// operands are dequantized in registers to FP16 - exact: an E2M1 value times an E4M3 scale has at most 6
// significant bits and lies in [2^-10, 2688] - and multiplied on v_mfma_f32_16x16x32_f16 with FP32
// accumulation across all of K; alpha is applied at the end.
//
//  * A wave computes 128 weight rows x 64 tokens (8 x 4 MFMA tiles, 128 accumulator registers; SwiGLU: 64 gate rows and
//    the same 64 up rows; NI = 4: 64 rows, for calls with few tiles). Per 128-value chunk a lane holds the raw 16 bytes
//    (32 E2M1 values) and the 2 scales of its row for each of its 8 weight tiles and 4 token tiles, and dequantizes one
//    8-value step at a time: lane (r, t) supplies K 32t + 8s .. +8 at step s for both operands (a permutation of K
//    inside the chunk, harmless as both operands use it; the weights' tiled layout holds exactly these 16 bytes per
//    (row, t), slot r * 4 + t).
//  * The 8 waves of a workgroup are WM (1 or 2) along the tokens x WK = 8 / WM along K, so a tile is 64 WM tokens high and a
//    prompt of a few hundred tokens still gives every CU two waves per SIMD, at the wave tile's ratio of dequantization
//    to MFMAs. Wave k of a K group takes chunks k, k + WK, ..; the group's FP32 sums meet in LDS at the end and are added
//    in wave order.
//  * Nothing is shared while a wave computes, so there are no barriers: each wave streams its own operands to its own
//    13.5 KB of LDS by direct loads, takes a landed chunk into registers (60 of them) and at once has the next one loaded
//    over it, which then has the whole chunk's 128 MFMAs to arrive.
//  * LDS of a wave (NI = 8): [weight values 128 x 64 B][weight scales 128 x 8][token values 64 x 64][token scales 64 x 8]. The
//    16-byte units of a 64-byte row are XOR-swizzled by swz4(row); four lanes of a load read one run of 64 bytes.
//
// What bounds it: the dequantization and the MFMAs share the SIMD's issue (3 VALU instructions per MFMA). Tiles of 256 x
// 256 over 8 waves, which read a step's word from LDS just ahead of its use, took 430 us at 300 x 5120 x 17408 (40 tiles
// on 256 CUs), 447 at 2048 x 5120 x 17408 and 760 for SwiGLU at 2048 x 17408 x 5120: now 63, 312 and 637.
#include "lq_common.hpp"

#include <string>

namespace lq {
namespace {

constexpr int kThreads = 512;
constexpr int wave_off_x(int ni) { return ni * 16 * 72; }  // a wave's LDS: 16 ni weight rows, then 64 tokens
constexpr int kRedWave = 16 * 1024;  // a wave's sums of four weight tiles x four token tiles
static_assert(kRedWave >= wave_off_x(8) + 64 * 72, "the reduction takes the larger part of LDS");

// Lane (r, t) reads unit t of row r, 16 bytes. 16 lanes of one t have no bank conflict, but the LDS serves rows 0-3 and 12-15 of
// one t with rows 4-11 of the next, where every read is a two-way one (3-5 % of the CUs' cycles). They are hidden: a swizzle
// without any (units of rows 0-3, 4-7, 8-11, 12-15 by 0, 2, 3, 1; counted 0) took 63.9 us at 300 x 5120 x 17408, this one 63.6,
// and the same at 2048 x 17408 x 5120 SwiGLU.
__device__ __forceinline__ int swz4(int row) { return ((row >> 1) & 3) ^ ((row >> 3) & 1); }
__device__ __forceinline__ int val_off(int row, int u) { return row * 64 + ((u ^ swz4(row)) << 4); }

struct Nvfp4Args {
  const uint8_t* xq;  // [M][K/2]
  const uint8_t* xs;  // [M][K/16]
  const uint8_t* w;   // tiled NVFP4 (raw 1152 B blocks, or coded 1024 B value blocks with wsf)
  const uint8_t* wsf; // coded blob's raw scales (128 B per block) or null
  const uint8_t* w2;  // SwiGLU: the up matrix (gate in w)
  const uint8_t* wsf2;
  float alpha, alpha2;
  float* y;
  int ldy, M, N, K, C;
  int accumulate;
  float gscale_out;  // SwiGLU: 1 / out_input_scale
  uint8_t* q_out;    // [M][N/2]
  uint8_t* sf_out;   // [M][N/16]
  int tiles_m, tiles_n;
};

typedef __attribute__((address_space(3))) void* lds_ptr;
// soff is uniform over the wave; saying so keeps it in an SGPR (held in a VGPR, the compiler wraps every load in a
// loop over the lanes' distinct values).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds), 16, voff, __builtin_amdgcn_readfirstlane(soff), 0, 0);
}
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds), 4, voff, __builtin_amdgcn_readfirstlane(soff), 0, 0);
}

// A lane's two E4M3 block scales of a chunk as FP16 (exact): one conversion per row and chunk.
__device__ __forceinline__ f16x2 scale_pair(uint32_t sc) { return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(sc, 1.0f, false); }

// Step s of a lane's raw chunk (word d = 8 E2M1 codes of its 16 bytes, its scale pair): 8 FP16 values e2m1 * scale
// (exact); steps 0, 1 use the first scale (K 32t .. +16), steps 2, 3 the second.
__device__ __forceinline__ u32x4 deq_word(uint32_t d, f16x2 sc, int s) {
  const f16x2 scv = f16x2{sc[s >> 1], sc[s >> 1]};
  const f16x2 e0 = fp4x2_to_f16x2<0>(d) * scv, e1 = fp4x2_to_f16x2<1>(d) * scv;
  const f16x2 e2 = fp4x2_to_f16x2<2>(d) * scv, e3 = fp4x2_to_f16x2<3>(d) * scv;
  return u32x4{__builtin_bit_cast(uint32_t, e0), __builtin_bit_cast(uint32_t, e1), __builtin_bit_cast(uint32_t, e2),
               __builtin_bit_cast(uint32_t, e3)};
}

#define LQ_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")

// Four outputs of one token, columns n .. n + 3.
__device__ __forceinline__ void put_out(const Nvfp4Args& a, int m, int n, f32x4 acc) {
  f32x4 v = f32x4{acc[0] * a.alpha, acc[1] * a.alpha, acc[2] * a.alpha, acc[3] * a.alpha};
  f32x4* dst = reinterpret_cast<f32x4*>(a.y + static_cast<size_t>(m) * a.ldy + n);
  if (a.accumulate) {
    const f32x4 o = *dst;
    v = f32x4{o[0] + v[0], o[1] + v[1], o[2] + v[2], o[3] + v[3]};
  }
  *dst = v;
}

// SwiGLU: the lane's four values of the 16-column output block from column ncol, token m (every lane of the wave calls
// it: a block's values are in lanes r, r + 16, r + 32, r + 48). up: alpha_up already applied.
__device__ __forceinline__ void put_swiglu(const Nvfp4Args& a, int m, int ncol, int t, f32x4 gate, f32x4 up) {
  float v[4], amax = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float gv = gate[e] * a.alpha;
    v[e] = bf16_to_f32(f32_to_bf16((gv / (1.f + __expf(-gv))) * up[e]));
    amax = fmaxf(amax, fabsf(v[e]));
  }
  amax = fmaxf(amax, __shfl_xor(amax, 16));
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  const float sraw = a.gscale_out * (amax * (1.f / 6.f));
  const uint32_t sc = __builtin_amdgcn_cvt_pk_fp8_f32(fminf(sraw, 448.f), 0.f, 0, false) & 0xffu;
  const float sv = e4m3_to_f32(sc);
  const float os = sv != 0.f ? 1.f / (sv * (1.f / a.gscale_out)) : 0.f;
  if (m < a.M && ncol < a.N) {
    uint8_t* qr = a.q_out + static_cast<size_t>(m) * (a.N / 2) + ncol / 2 + 2 * t;
    const uint32_t b0 = e2m1x2_rne(v[0] * os, v[1] * os);
    const uint32_t b1 = e2m1x2_rne(v[2] * os, v[3] * os);
    *reinterpret_cast<uint16_t*>(qr) = static_cast<uint16_t>(b0 | (b1 << 8));
    if (t == 0) a.sf_out[static_cast<size_t>(m) * (a.N / 16) + ncol / 16] = static_cast<uint8_t>(sc);
  }
}

template <bool SWIGLU, int NI, int WM>
__global__ void __launch_bounds__(kThreads) prefill_nvfp4_kernel(const Nvfp4Args a) {
  constexpr int WK = 8 / WM, TN = SWIGLU ? 64 : 16 * NI, TM = 64 * WM;
  constexpr int kOffS = NI * 1024, kOffX = wave_off_x(NI);
  static_assert(NI == 8 || (NI == 4 && !SWIGLU), "weight tiles of a wave");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, t = lane >> 4;
  const int wk = wave % WK, wm = wave / WK;

  // Tile order: XCD b % 8 takes a contiguous range of the tiles; groups of 8 weight tiles x every token tile, weight
  // tiles fastest.
  constexpr int kGroup = 8;
  const int nb = gridDim.x, b = blockIdx.x, x = b & 7;
  const int tile = x * (nb >> 3) + min(x, nb & 7) + (b >> 3);
  const int grp = tile / (kGroup * a.tiles_m), rem = tile % (kGroup * a.tiles_m);
  const int gsize = min(kGroup, a.tiles_n - grp * kGroup);
  const int n0 = (grp * kGroup + rem % gsize) * TN, m0 = (rem / gsize) * TM + wm * 64;

  const int blkb = a.wsf ? kValueBytesFp4 : kTileBytesFp4;
  const int nbytes = (a.N / 16) * a.C * blkb, sbytes = a.wsf ? (a.N / 16) * a.C * 128 : nbytes;
  auto rsrc = [](const uint8_t* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, bytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t wr1 = rsrc(a.w, nbytes), wr2 = rsrc(SWIGLU ? a.w2 : a.w, nbytes);
  const __amdgpu_buffer_rsrc_t sr1 = rsrc(a.wsf ? a.wsf : a.w, sbytes);
  const __amdgpu_buffer_rsrc_t sr2 = rsrc(SWIGLU ? (a.wsf2 ? a.wsf2 : a.w2) : (a.wsf ? a.wsf : a.w), sbytes);
  const __amdgpu_buffer_rsrc_t xr = rsrc(a.xq, a.M * (a.K / 2)), xsr = rsrc(a.xs, a.M * (a.K / 16));

  // Weight rows are whole tiles of a matrix with N % 128 == 0: always in range. Weight tile i of the wave is
  // 16-row tile n0 / 16 + i (SwiGLU: + i % 4, the up matrix from i = 4); a lane loads unit lane % 4 of row lane / 4 of a
  // tile's values, 4 bytes of two tiles' scales.
  const int srow = lane >> 2, su = (lane & 3) ^ swz4(srow);
  const int wsrc = srow * 64 + su * 16, tstep = a.C * blkb, wbase = (n0 >> 4) * tstep;
  const int sblk = a.wsf ? 128 : blkb, sstep = a.C * sblk;
  const int ssrc = (lane >> 5) * sstep + (a.wsf ? 0 : 1024) + (lane & 31) * 4, sbase = (n0 >> 4) * sstep;
  constexpr unsigned kOob = 0x80000000u;
  unsigned xsrc[4], xssrc[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + 16 * j + srow;
    xsrc[j] = m < a.M ? static_cast<unsigned>(m * (a.K / 2) + su * 16) : kOob;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = m0 + 32 * j + (lane >> 1);
    xssrc[j] = m < a.M ? static_cast<unsigned>(m * (a.K / 16) + (lane & 1) * 4) : kOob;
  }
  uint8_t* lds = smem + wave * (kOffX + 64 * 72);
  // load v of a chunk's
  constexpr int kW = NI, kWS = kW + NI / 2, kX = kWS + 4, kLoads = kX + 2;
  auto issue_one = [&](int c, int v) {
    if (v < kW) {
      if (SWIGLU && v >= 4) dma16(wr2, lds + v * 1024, wsrc, wbase + (v - 4) * tstep + c * blkb);
      else dma16(wr1, lds + v * 1024, wsrc, wbase + v * tstep + c * blkb);
    } else if (v < kWS) {
      const int p = v - kW;
      if (SWIGLU && p >= 2) dma4(sr2, lds + kOffS + p * 256, ssrc, sbase + 2 * (p - 2) * sstep + c * sblk);
      else dma4(sr1, lds + kOffS + p * 256, ssrc, sbase + 2 * p * sstep + c * sblk);
    } else if (v < kX) {
      dma16(xr, lds + kOffX + (v - kWS) * 1024, xsrc[v - kWS], c * 64);
    } else {
      dma4(xsr, lds + kOffX + 64 * 64 + (v - kX) * 256, xssrc[v - kX], c * 8);
    }
  };

  f32x4 acc[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int last = a.C - 1;
#pragma unroll
  for (int v = 0; v < kLoads; ++v) issue_one(min(wk, last), v);
  // A SIMD's two waves at different issue priority: one multiplies while the other takes in its next chunk, where equals
  // drift into doing the same at once (300 x 5120 x 17408 62.1 -> 60.2 us, 300 x 17408 x 5120 SwiGLU 139 -> 134, 2048 x
  // 17408 x 5120 level).
  if (wave >= 4) __builtin_amdgcn_s_setprio(1);
  for (int c = wk; c < a.C; c += WK) {
    LQ_WAIT_VM(0);
    u32x4 aw[NI], bw[4];
    f16x2 as[NI], bs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bw[j] = *reinterpret_cast<const u32x4*>(lds + kOffX + val_off(16 * j + r, t));
      bs[j] = scale_pair(*reinterpret_cast<const uint16_t*>(lds + kOffX + 64 * 64 + (16 * j + r) * 8 + t * 2));
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      aw[i] = *reinterpret_cast<const u32x4*>(lds + val_off(16 * i + r, t));
      as[i] = scale_pair(*reinterpret_cast<const uint16_t*>(lds + kOffS + (16 * i + r) * 8 + t * 2));
    }
    // every read has returned before the next chunk's loads go over them (past the end the last chunk again, never read)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int next = min(c + WK, last);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4 bf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) bf[j] = deq_word(bw[j][s], bs[j], s);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        // (one of the loads per weight tile: a burst would hold the wave up)
        if (s * NI + i < kLoads) issue_one(next, s * NI + i);
        const u32x4 af = deq_word(aw[i][s], as[i], s);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma16x16x32(af, bf[j], acc[i][j], true);
      }
    }
  }
  LQ_WAIT_VM(0);  // no load to LDS is on its way when the sums go there
  __builtin_amdgcn_s_setprio(0);

  // The sums, four weight tiles at a time (SwiGLU: two gate tiles and the up tiles of the same columns): sum (ii, j) of a
  // wave at (ii * 4 + j) KB of its 16 KB; unit q = wk, wk + WK, .. of 8 is two weight tiles of token tile q % 4.
#pragma unroll
  for (int half = 0; half < NI / 4; ++half) {
    __syncthreads();
    uint8_t* mine = smem + wave * kRedWave + lane * 16;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int i = SWIGLU ? (ii & 1) * 4 + half * 2 + (ii >> 1) : half * 4 + ii;
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4*>(mine + (ii * 4 + j) * 1024) = acc[i][j];
    }
    __syncthreads();
#pragma unroll
    for (int q0 = 0; q0 < 8; q0 += WK) {
      const int q = q0 + wk, pair = q >> 2, j = q & 3;
      f32x4 sum[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint8_t* from = smem + wm * WK * kRedWave + ((2 * pair + h) * 4 + j) * 1024 + lane * 16;
        sum[h] = *reinterpret_cast<const f32x4*>(from);
#pragma unroll
        for (int k = 1; k < WK; ++k) sum[h] = sum[h] + *reinterpret_cast<const f32x4*>(from + k * kRedWave);
      }
      const int m = m0 + 16 * j + r;
      if constexpr (SWIGLU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[1][e] *= a.alpha2;
        put_swiglu(a, m, n0 + 16 * (half * 2 + pair), t, sum[0], sum[1]);
      } else if (m < a.M) {
#pragma unroll
        for (int h = 0; h < 2; ++h) put_out(a, m, n0 + 16 * (half * 4 + 2 * pair + h) + 4 * t, sum[h]);
      }
    }
  }
}

template <bool SWIGLU, int NI, int WM>
int tile_launch(Nvfp4Args a, const char* name, hipStream_t s) {
  a.tiles_m = cdiv(a.M, 64 * WM);
  a.tiles_n = a.N / (SWIGLU ? 64 : 16 * NI);
  constexpr int lds = 8 * kRedWave;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_nvfp4_kernel<SWIGLU, NI, WM>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return fail(LQ_ERR_LAUNCH, std::string(name) + ": " + hipGetErrorString(attr));
  hipLaunchKernelGGL((prefill_nvfp4_kernel<SWIGLU, NI, WM>),
                     dim3(static_cast<unsigned>(a.tiles_m) * static_cast<unsigned>(a.tiles_n)), dim3(kThreads), lds, s, a);
  return check_launch(name);
}

// The tile, by an estimate of the time: rounds of one tile per CU, each of which takes every wave through its share of the
// chunks and then the sums. A wave tile of half the weight rows (NI = 4) dequantizes more per MFMA, and pays where whole ones
// leave half the CUs without work (us at NI = 8 and 4, WM = 1: 128 x 5120 x 5120 22.1, 15.3; 300 x 5120 x 5120 24.3, 27.6;
// 128 x 5120 x 17408 58, 42; 500 x 2048 x 4096 19.4, 13.9).
//
// How many waves share K (8 / WM) is a matter of the matrix alone: the FP32 sums are then taken in one order whatever the
// number of tokens, and a row's result has the same bits in every call. Eight waves leave the fewest CUs idle, four pay a
// tile's closing sums half as often; taken is what is faster over prompts of 128 to 4096 tokens, by the product of the
// ratios. Measured at M = 128, 512, 2048, 4096, eight and four: SwiGLU 17408 x 5120 70 81, 201 188, 719 637, 1409 1280;
// 6144 x 2048 14 20, 37 38, 140 115, 274 239 and N = 34816, K = 5120 69 81, 201 187 (M = 500), 730 657, 1439 1297 (four);
// SwiGLU 5120 x 5120 26 40, 66 74, 221 194, 425 394; N = 7168, K = 5120 16 35, 45 40 (M = 500), 162 151, 309 274 and N = 5120,
// K = 17408 42 106, 111 103 (M = 500), 312 325, 628 591 (eight). Over 33 matrices and M = 81 .. 4096 the rule is 5 % from
// the faster of the two at each M. (Two waves along K at M >= 1500 and short K: up to 20 % less than eight, not worth
// results that depend on how a prompt is cut. NI = 4 with WM = 2 was never ahead by more than 2 %.)
struct TileKind {
  int ni, wm;
  double chunk, tile;  // microseconds
};
constexpr TileKind kWhole{8, 1, 3.45, 5.}, kHalf{4, 1, 2.15, 4.}, kFour{8, 2, 3.2, 5.};

TileKind choose_tile(bool swiglu, int M, int N, int C, long long cus) {
  auto us = [&](const TileKind& k, int m) {
    const long long tiles = static_cast<long long>(N / (swiglu ? 64 : 16 * k.ni)) * cdiv(m, 64 * k.wm);
    return static_cast<double>((tiles + cus - 1) / cus) * (cdiv(C, 8 / k.wm) * k.chunk + k.tile);
  };
  auto eight = [&](int m) { return !swiglu && us(kHalf, m) < us(kWhole, m) ? kHalf : kWhole; };
  double ratio = 1.;
  for (int m = 128; m <= 4096; m *= 2) ratio *= us(eight(m), m) / us(kFour, m);
  return ratio > 1. ? kFour : eight(M);
}

template <bool SWIGLU>
int nvfp4_launch(Nvfp4Args a, const char* name, hipStream_t s) {
  const std::string nm(name);
  if (a.N <= 0 || a.K <= 0 || a.N % 128 != 0 || a.K % 128 != 0)
    return fail(LQ_ERR_SHAPE, nm + ": N % 128 and K % 128 must be 0");
  if (a.M < 1) return LQ_OK;
  if (!SWIGLU && (a.ldy < a.N || a.ldy % 4 != 0)) return fail(LQ_ERR_SHAPE, nm + ": ldy must be >= N and a multiple of 4");
  const long long wb = static_cast<long long>(a.N / 16) * (a.K / 128) * kTileBytesFp4;
  if (wb >= (1LL << 31) || static_cast<long long>(a.M) * (a.K / 2) >= (1LL << 31))
    return fail(LQ_ERR_SHAPE, nm + ": operands must be below 2^31 bytes");
  if (!a.xq || !a.xs || !a.w || (SWIGLU ? (!a.w2 || !a.q_out || !a.sf_out) : !a.y))
    return fail(LQ_ERR_ARG, nm + ": null pointer");
  if (!SWIGLU && reinterpret_cast<uintptr_t>(a.y) % 16 != 0) return fail(LQ_ERR_ARG, nm + ": y must be 16-byte aligned");
  a.C = a.K / 128;
  int dev = 0;
  (void)hipGetDevice(&dev);
  const TileKind k = choose_tile(SWIGLU, a.M, a.N, a.C, device_cus(dev));
  if constexpr (!SWIGLU)
    if (k.ni == 4) return tile_launch<SWIGLU, 4, 1>(a, name, s);
  return k.wm == 1 ? tile_launch<SWIGLU, 8, 1>(a, name, s) : tile_launch<SWIGLU, 8, 2>(a, name, s);
}

}  // namespace
}  // namespace lq

using namespace lq;

extern "C" {

// Test hook (not part of the interface): the tile of a product on `cus` CUs, 16 * NI + WM.
int lq_debug_prefill_nvfp4_tile(int swiglu, int M, int N, int K, int cus) {
  const TileKind k = choose_tile(swiglu != 0, M, N, K / 128, cus);
  return 16 * k.ni + k.wm;
}

int lq_prefill_gemm_nvfp4(const uint8_t* xq, const uint8_t* xs, int M, const uint8_t* w, float alpha, float* y, int ldy,
                          int N, int K, int accumulate, void* stream, const uint8_t* wsf) {
  Nvfp4Args a{};
  a.xq = xq;
  a.xs = xs;
  a.w = w;
  a.wsf = wsf;
  a.alpha = alpha;
  a.y = y;
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  a.accumulate = accumulate;
  return nvfp4_launch<false>(a, "prefill_gemm_nvfp4", static_cast<hipStream_t>(stream));
}

int lq_prefill_swiglu_nvfp4(const uint8_t* xq, const uint8_t* xs, int M, const uint8_t* gate, float alpha_gate,
                            const uint8_t* up, float alpha_up, int N, int K, float out_input_scale, uint8_t* q_out,
                            uint8_t* sf_out, void* stream, const uint8_t* gate_sf, const uint8_t* up_sf) {
  if ((gate_sf == nullptr) != (up_sf == nullptr))
    return fail(LQ_ERR_ARG, "prefill_swiglu_nvfp4: gate and up must both be raw or both coded");
  Nvfp4Args a{};
  a.xq = xq;
  a.xs = xs;
  a.w = gate;
  a.wsf = gate_sf;
  a.w2 = up;
  a.wsf2 = up_sf;
  a.alpha = alpha_gate;
  a.alpha2 = alpha_up;
  a.M = M;
  a.N = N;
  a.K = K;
  a.gscale_out = 1.f / out_input_scale;
  a.q_out = q_out;
  a.sf_out = sf_out;
  return nvfp4_launch<true>(a, "prefill_swiglu_nvfp4", static_cast<hipStream_t>(stream));
}

}  // extern "C"
