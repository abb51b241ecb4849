// Affine-4-bit GEMMs of a prefill batch on the matrix cores (dense projections, the MoE experts over
// chunks of their slots), with the bits of the dot-product GEMV (mtpx_device.h: exact integer block
// sums, an ordered float combine per block).
//
// Arithmetic.  The 24-bit fixed-point block values are split into their three bytes (limbs 0 and 1
// unsigned, limb 2 signed); each limb times 2^(E-19) of its block is an exact bf16, and a nibble n
// shifted to bits 3-6 is the bf16 denormal n * 2^-130.  v_mfma_f32_16x16x32_bf16 multiplies them
// exactly, and the sums of one 32-element block are integers below 2^24 times 2^(E-149), so the three
// f32 results d0, d1, d2 are exact in any order.  Then
//   low = fma(d1, 256, d0)      the low 16 bits' sum, rounded once, times p = 2^(E-149)
//   t   = fma(d2, 65536, low)   DXraw * p
//   acc = fma(b, SX, fma(s, t, acc))
// are the dot-product path's float operations with the block scale (a power of two) carried through:
// four VALU operations per (token, row, block), where four i8 limbs and their integer recombination
// need about nine.  A block exponent above XL_EMAX (|x| >= 4096) would overflow a limb's bf16: such a
// block is stored with the scale of XL_EMAX and a factor r = 2^(E - XL_EMAX), and a tile that holds
// such a token walks with t * r.
//
// Chains.  Block j joins chain j % L (L = lanes_for_blocks(K/32)).  A wave owns the chains = c mod C of
// RT tiles of 16 rows against 16 tokens, with all its L/C chains per value in registers, so K is walked
// in memory order and every weight line is read once; the last log2(C) butterfly levels go through LDS.
//
// What bounds it.  A 16x16x32 MFMA issues no VALU instruction beside it (16.8 cycles against 2.5 per
// VALU instruction, four waves per SIMD), so a tile of 16 rows x 16 tokens x one block costs about
// 3 * 16.8 + 28 * 2.5 = 120 cycles of a SIMD; the rest is the operands' way: two workgroups of eight
// waves per CU (128 registers), each with its next segments in flight (LDS-direct loads, the wait
// counted so that the later ones stay in flight).  Measured against the i8 batch GEMM and the slot walk
// it replaced, 512 tokens, group size 64: GDN in-projection 431 -> 190 us, K = 6144 projections 236 ->
// 127, mixer down and inject 94 -> 43 (and their layout pass), mixer up 71 -> 22, expert gate|up 1000 ->
// 340 (HBM floor about 200), expert down 213 -> 160.  On the way (in-projection): segments through
// registers 423 us, one segment ahead 313, a token's limbs in four 16-byte runs instead of one of 64
// bytes 246, limb reads with bank conflicts 232, a register for every rotation of sx (spilled ones make
// the walk wait for all loads) 202.  K = 6144 with eight classes of 64 rows, one segment ahead and spills:
// 1003 tokens 219 us, with four classes and two ahead 158.  One workgroup of 16 waves per CU, twice the rows
// per limb byte: 490 us where two of eight waves take 400 (they all wait at its barrier).
#include <algorithm>
#include <type_traits>

#include "mtpx_kernels.h"

namespace mtpx {

constexpr int GT_THREADS = 512;  // eight waves

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// The limb form of a batch (XlBatch), from x [M][K]: xl [M][nb][3][32] bf16, sx and xr [M][nb], big
// [M][XL_FLAGS] (nonzero somewhere in a token's if any of its blocks is above XL_EMAX).  One workgroup per
// token and part.  (One workgroup per token: 17 us at 75 tokens of K = 10240.)
__global__ __launch_bounds__(256) void k_xlimb(const bf16* __restrict__ x, int nb, uint32_t* __restrict__ xl,
                                               float* __restrict__ sx, float* __restrict__ xr,
                                               uint8_t* __restrict__ big) {
  const size_t t = blockIdx.x;
  x += t * nb * 32;
  xl += t * nb * 48;
  sx += t * nb;
  xr += t * nb;
  const int i = threadIdx.x & 31;
  const int part = blockIdx.y, end = min(nb, (part + 1) * XL_PART);
  int any = 0;
  for (int j = part * XL_PART + (int)(threadIdx.x >> 5); j < end; j += 8) {
    any |= xlimb_lanes(x[(size_t)j * 32 + i], i, xl + (size_t)j * 48, sx + j, xr + j);
  }
  xl_flag(big, t, part, gridDim.y, __syncthreads_or(any));
}

size_t xl_bytes(int M, int K) {
  const size_t nb = K / 32;
  return (size_t)M * nb * (192 + 8) + (size_t)M * XL_FLAGS + 1024;
}

XlBatch xl_carve(void* ws, int M, int K) {
  const size_t n = (size_t)M * (K / 32);
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  char* p = static_cast<char*>(ws);
  XlBatch b;
  b.xl = reinterpret_cast<uint4*>(p);
  p += up(n * 192);
  b.sx = reinterpret_cast<float*>(p);
  p += up(n * 4);
  b.xr = reinterpret_cast<float*>(p);
  p += up(n * 4);
  b.big = reinterpret_cast<uint8_t*>(p);
  return b;
}

hipError_t launch_xlimb(const bf16* x, int M, int K, const XlBatch& b, hipStream_t st) {
  const int parts = (K / 32 + XL_PART - 1) / XL_PART;
  if (parts > XL_FLAGS) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_xlimb, dim3(M, parts), dim3(256), 0, st, x, K / 32, reinterpret_cast<uint32_t*>(b.xl), b.sx, b.xr,
                     b.big);
  return hipGetLastError();
}

// butterfly levels S, S/2, .., 1 over v[0..2S-1]
template <int S, int NV>
__device__ __forceinline__ void gt_fold(float (&v)[NV]) {
  if constexpr (S >= 1) {
#pragma unroll
    for (int u = 0; u < S; ++u) v[u] = v[u] + v[u + S];
    gt_fold<S / 2>(v);
  }
}

// a ? x : y of values (the conditional operator of two variables is one of them, by address)
template <typename T>
__device__ __forceinline__ T sel(bool a, T x, T y) {
  return a ? x : y;
}

template <int N>
__device__ __forceinline__ void wait_vm() {  // s_waitcnt vmcnt(N)
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// One matrix of a dense launch; a launch takes up to two with the same K (a mixer's down and inject rows).
struct GemmMat {
  const uint32_t* w;
  const bf16 *s, *b;
  bf16* y;
  float* yf;
  int N;
};

struct GemmArgs {
  GemmMat mat[2];
  XlBatch x;
  uint32_t xl_len;               // bytes of x.xl
  int M;
  int rblocks1, rblocks, tiles;  // row blocks of mat[0], of both; token tiles
};

// The MoE chunk launches: the batch's slots in expert order (m.gorder) cut into chunks of at most
// MQ_CHUNK slots of one expert (m.chunks), x in limb form per token (gate|up) or per slot (down).
struct MoeGemmArgs {
  MoeArgs m;
  XlBatch x;
  uint32_t xl_len;
};
static_assert(MQ_CHUNK == 16, "a chunk is a token tile");

constexpr int GT_DENSE = 0, GT_GATE_UP = 1, GT_DOWN = 2;  // k_gemm modes

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
}
#endif

// NST stages of LDS (NST - 1 segments in flight); MINW waves per SIMD (two or three workgroups per CU).
template <int MODE, int L, int IT, int C, int RT, bool GS32, int NST, int MINW>
__global__ __launch_bounds__(GT_THREADS, MINW) void k_gemm(std::conditional_t<MODE == GT_DENSE, GemmArgs, MoeGemmArgs> a) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer resources exist on the device only
  constexpr int NB = L * IT, LC = L / C, RG = 8 / C, NT = RG * RT, R = NT * 16;
  constexpr int SEG = C;            // blocks per segment: one of each class
  constexpr int NSEG = NB / SEG;
  constexpr bool WHOLE = NB % 16 != 0;  // scales of the whole K at once, else of 16 blocks
  constexpr int GB = WHOLE ? NB : 16, SPS = WHOLE ? NSEG : 16 / SEG;  // blocks and segments per scale granule
  constexpr int SH = GS32 ? 1 : 2;      // blocks per group
  constexpr int ROWB = NB * 16, ng = NB / SH, GW = GB / SH;  // weight row bytes, groups per row and per granule
  // a stage's 16-byte units: limbs [SEG][3][16 tokens][4], weights [R][SEG slots]
  constexpr int AI = SEG * 3, WI = SEG * R / 64, NI = AI + WI, STU = NI * 64;  // wave loads
  constexpr int PER_W = (NI + 7) / 8;
  // a scale granule's: s [R][GW] bf16, b likewise, sx [16 tokens][GB] f32
  constexpr int SU = R * GW * 2 / 16, SI = (SU + 63) / 64;  // units, wave loads of one of s, b
  constexpr int XI = WHOLE ? (GB * 16 + 63) / 64 : 1;       // wave loads of sx (4-byte ones for the whole K)
  constexpr int SCU = 2 * SI * 64 + (WHOLE ? XI * 16 : 64);
  static_assert(NSEG * SEG == NB && NSEG % LC == 0 && (R * GW * 2) % 16 == 0 && SEG % 2 == 0, "whole loads");
  static_assert(MODE != GT_GATE_UP || !WHOLE, "gate and up scales by granule");
  __shared__ uint4 st0[STU], st1[STU], st2[NST > 2 ? STU : 1];
  __shared__ uint4 sc0[SCU], sc1[WHOLE ? 1 : SCU];

  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // uniform: offsets in scalar registers
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int c = wave % C, rg = wave / C;

  // ---- the unit: a row block (gate|up: half of its tiles from each matrix) and up to 16 tokens ----
  const uint32_t *w0, *w1;
  const bf16 *s0, *b0, *s1, *b1;
  int row0, rows_w, cnt;
  uint32_t xrow_n, yrow_n;  // x row and output row of token n
  bf16* yp;
  float* yfp = nullptr;
  if constexpr (MODE == GT_DENSE) {
    // tiles in groups of four, a row block's tiles of one group side by side; contiguous units on one
    // XCD, whose L2 then holds the group's activations while the row blocks stream through
    const int n_units = a.rblocks * a.tiles, per = (n_units + 7) / 8;
    const int unit = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= per || unit >= n_units) return;
    const int gsz = a.rblocks * 4, tg = unit / gsz, rem = unit - tg * gsz, tw = min(4, a.tiles - tg * 4);
    const int rb = rem / tw, tile = tg * 4 + rem % tw;
    const GemmMat& m = rb < a.rblocks1 ? a.mat[0] : a.mat[1];
    row0 = (rb < a.rblocks1 ? rb : rb - a.rblocks1) * R;
    w0 = w1 = m.w;
    s0 = s1 = m.s;
    b0 = b1 = m.b;
    rows_w = m.N;
    yp = m.y;
    yfp = m.yf;
    cnt = min(16, a.M - tile * 16);
    xrow_n = yrow_n = tile * 16 + min(n, cnt - 1);
  } else {
    const MoeArgs& m = a.m;
    // units of one chunk side by side on one XCD
    const int fb = MODE == GT_GATE_UP ? m.F / (R / 2) : (m.H + R - 1) / R;  // row blocks
    const int n_units = min(*m.chunk_n, m.max_chunks) * fb, per = (n_units + 7) / 8;
    const int unit = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= per || unit >= n_units) return;
    const int ch = unit / fb;
    row0 = (unit - ch * fb) * (MODE == GT_GATE_UP ? R / 2 : R);
    const int pos = m.chunks[2 * ch], info = m.chunks[2 * ch + 1];
    cnt = min(max(info & 0xffff, 1), 16);
    const int e1 = min(max(info >> 16, 0), m.E);  // 0: the shared expert
    rows_w = MODE == GT_GATE_UP ? m.F : m.H;
    const size_t r = e1 ? (size_t)(e1 - 1) * rows_w : 0;
    if constexpr (MODE == GT_GATE_UP) {
      w0 = (e1 ? m.gate_w : m.sh_gate_w) + r * (ROWB / 4);
      s0 = (e1 ? m.gate_s : m.sh_gate_s) + r * ng;
      b0 = (e1 ? m.gate_b : m.sh_gate_b) + r * ng;
      w1 = (e1 ? m.up_w : m.sh_up_w) + r * (ROWB / 4);
      s1 = (e1 ? m.up_s : m.sh_up_s) + r * ng;
      b1 = (e1 ? m.up_b : m.sh_up_b) + r * ng;
    } else {
      w0 = w1 = (e1 ? m.down_w : m.sh_down_w) + r * (ROWB / 4);
      s0 = s1 = (e1 ? m.down_s : m.sh_down_s) + r * ng;
      b0 = b1 = (e1 ? m.down_b : m.sh_down_b) + r * ng;
    }
    yp = MODE == GT_GATE_UP ? m.act : m.r;
    // order entry -> slot (m * K + k routed, M * K + m shared) -> token
    const int slots = m.M * (m.K + 1);
    const int sl = min(m.gorder[min(pos + min(n, cnt - 1), slots - 1)] & 0xffff, slots - 1);
    yrow_n = sl;
    if (MODE == GT_DOWN) {
      xrow_n = sl;
    } else {
      xrow_n = sl >= m.M * m.K ? sl - m.M * m.K : sl / m.K;
    }
  }
  auto xrow_at = [&](int t) -> uint32_t { return __shfl((int)xrow_n, t, 64); };
  const uint32_t xrow_l = xrow_at(lane >> 2), xoff = (xrow_l * NB + ((lane & 3) ^ g) * 4) * 4;
  // The weight and scale resources start at the unit's first row, so that offsets are of 32 bits whatever the matrix holds.
  const int rows_u = min(rows_w - row0, MODE == GT_GATE_UP ? R / 2 : R);
  w0 += (size_t)row0 * (ROWB / 4);
  w1 += (size_t)row0 * (ROWB / 4);
  s0 += (size_t)row0 * ng;
  b0 += (size_t)row0 * ng;
  s1 += (size_t)row0 * ng;
  b1 += (size_t)row0 * ng;
  // unit row of row-in-block r, clamped: rows past the end repeat the last one (computed, not stored)
  auto lrow = [&](int r) { return min(MODE == GT_GATE_UP && r >= R / 2 ? r - R / 2 : r, rows_u - 1); };
  auto my_tile = [&](int rt) {  // row tile of this wave's tile rt
    return MODE == GT_GATE_UP ? (rt / (RT / 2)) * (NT / 2) + rg * (RT / 2) + rt % (RT / 2) : rg * RT + rt;
  };
  // the block slot of a weight row is rotated so that 16 rows of one block fall on different banks
  auto slot = [](int row, int blk) {
    return blk ^ (SEG == 4 ? (row >> 2) & 3 : SEG == 8 ? (row >> 1) & 7 : (row >> 3) & (SEG - 1));
  };
  const auto rA = make_rsrc(a.x.xl, a.xl_len), rX = make_rsrc(a.x.sx, a.xl_len / 48);
  // One weight and one scale resource per wave.  gate|up: the stage loads are 12 of limbs and 8 of weights, so
  // waves 4-7 load the gate's row tiles and waves 0-3 the up's; scale load i (s: i < SI, then b) is wave i's.
  static_assert(MODE != GT_GATE_UP || (AI == 12 && WI == 8), "the waves' weight loads");
  const auto rW = make_rsrc(sel(MODE == GT_GATE_UP && wave < 4, w1, w0), (size_t)rows_u * ROWB);
  static_assert(WHOLE || 2 * SI <= 8, "a scale load per wave and granule");
  const bool cup = MODE == GT_GATE_UP && wave % SI >= SI / 2;
  const auto rC = make_rsrc(sel(wave < SI, sel(cup, s1, s0), sel(cup, b1, b0)), (size_t)rows_u * ng * 2);

  // ---- staging: this wave's loads i = wave, wave + 8, ..: limbs i < AI, then weights ----
  uint32_t off[PER_W];
#pragma unroll
  for (int k = 0; k < PER_W; ++k) {
    const int i = wave + 8 * k;
    if (i < AI) {
      // lane l: token l / 4, word group (l & 3) rotated by the token: 64-byte runs per token, and the
      // 16 tokens of one word group on different banks in every phase of a 16-byte LDS read
      off[k] = xrow_l * (NB * 192) + (uint32_t)((lane & 3) ^ ((4 - (lane >> 4)) & 3)) * 16 + (i / 3) * 192 + (i % 3) * 64;
    } else {
      const int u = (min(i, NI - 1) - AI) * 64 + lane, r = u / SEG;
      off[k] = (uint32_t)lrow(r) * ROWB + (uint32_t)slot(r, u % SEG) * 16;
    }
  }
  auto stage_load = [&](uint4* d, int seg) {
#pragma unroll
    for (int k = 0; k < PER_W; ++k) {
      const int i = wave + 8 * k;  // uniform
      if (8 * k + 7 < NI || i < NI) {
        if (8 * k + 7 < AI || (8 * k < AI && i < AI))
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void_t*)(d + i * 64), 16, off[k], seg * (SEG * 192), 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rW, (lds_void_t*)(d + i * 64), 16, off[k], seg * (SEG * 16), 0, 0);
      }
    }
  };
  // The scale granules' loads: wave i < 2 SI part i of s, then b; wave 2 SI % 8 also sx.  The whole K at
  // once: s, b and sx parts shared over the waves (the block's scale rows are contiguous).
  const uint32_t coff = WHOLE ? 0u : (uint32_t)lrow(((wave % SI) * 64 + lane) / (GW / 8 ? GW / 8 : 1)) * (ng * 2) +
                                         (uint32_t)(lane % (GW / 8 ? GW / 8 : 1)) * 16;
  const uint32_t soff = 2 * SI < 8 ? sel(wave == 2 * SI, xoff, coff) : xoff;  // one register where a wave loads one
  auto scale_load = [&](uint4* d, int q) {
    if constexpr (WHOLE) {
#pragma unroll
      for (int k = 0; k < (2 * SI + XI + 7) / 8; ++k) {
        const int i = wave + 8 * k;
        if (i < 2 * SI) {
          const auto r = make_rsrc(sel(i < SI, s0, b0), (size_t)rows_u * ng * 2);  // past the end: zeros
          __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)(d + i * 64), 16,
                                                   (uint32_t)((i % SI) * 64 + lane) * 16, 0, 0, 0);
        } else if (i < 2 * SI + XI) {
          const int j = i - 2 * SI, u = j * 64 + lane;
          const uint32_t o = (xrow_at(min(u / GB, 15)) * NB + u % GB) * 4;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rX, (lds_void_t*)(d + 2 * SI * 64 + j * 16), 4, o, 0, 0, 0);
        }
      }
    } else {
      if (wave < 2 * SI)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rC, (lds_void_t*)(d + wave * 64), 16, 2 * SI < 8 ? soff : coff, q * (GW * 2), 0, 0);
      if (wave == 2 * SI % 8)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rX, (lds_void_t*)(d + 2 * SI * 64), 16,
                                                 soff, q * 64, 0, 0);
    }
  };
  static_assert(XL_FLAGS == 16, "a token's flags in one load");
  const uint4 bigs = reinterpret_cast<const uint4*>(a.x.big)[xrow_n];
  const bool big = __any((bigs.x | bigs.y | bigs.z | bigs.w) != 0u);
  float acc[RT][4][LC];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int u = 0; u < LC; ++u) acc[rt][i][u] = 0.0f;

  // ---- one block of this wave's class against its row tiles ----
  const int al = n * 4 + (g ^ ((4 - (n >> 2)) & 3));  // limb unit of token n, word group g
  const int wl = (n * SEG + slot(n, c)) * 4 + g;      // weight word of row n (the slot depends on the row mod 16)
  const int sl = n * GW + c / SH;
  const int xl0 = g * 68 + (c & 3);  // sx of token 4 g: its four words rotated by g
  auto step = [&](auto bigc, int u, const uint4* d, const uint4* ds, int sseg, int seg) {
    constexpr bool BIG = decltype(bigc)::value;
    bf16x8_t av3[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const uint4 v = d[(c * 3 + m) * 64 + al];
      __builtin_memcpy(&av3[m], &v, 16);
    }
    const uint32_t* dw = reinterpret_cast<const uint32_t*>(d + AI * 64);
    const uint16_t* dh = reinterpret_cast<const uint16_t*>(ds);
    const float* dx = reinterpret_cast<const float*>(ds + 2 * SI * 64);
    int xa = xl0;
    asm volatile("" : "+v"(xa));  // one register, not one per rotation
    float sx4[4], r4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sx4[i] = WHOLE ? dx[(4 * g + i) * GB + sseg * SEG + c]
                     : dx[(xa ^ ((sseg * SEG + c) >> 2) * 4) + i * 16];
    if constexpr (BIG) {
#pragma unroll
      for (int i = 0; i < 4; ++i) r4[i] = a.x.xr[(size_t)xrow_at(4 * g + i) * NB + seg * SEG + c];
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int rr = my_tile(rt) * 16;
      const uint32_t w = dw[wl + rr * SEG * 4];
      const float sc = __uint_as_float((uint32_t)dh[sl + rr * GW + sseg * SEG / SH] << 16);
      const float bi = __uint_as_float((uint32_t)dh[SI * 512 + sl + rr * GW + sseg * SEG / SH] << 16);
      const uint4 bw = make_uint4((w << 3) & 0x00780078u, (w >> 1) & 0x00780078u, (w >> 5) & 0x00780078u,
                                  (w >> 9) & 0x00780078u);
      bf16x8_t bop;
      __builtin_memcpy(&bop, &bw, 16);
      const f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
      const f32x4_t d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av3[0], bop, z, 0, 0, 0);
      const f32x4_t d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av3[1], bop, z, 0, 0, 0);
      const f32x4_t d2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av3[2], bop, z, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float t = __builtin_fmaf(d2[i], 65536.0f, __builtin_fmaf(d1[i], 256.0f, d0[i]));
        if constexpr (BIG) t = t * r4[i];
        acc[rt][i][u] = __builtin_fmaf(bi, sx4[i], __builtin_fmaf(sc, t, acc[rt][i][u]));
      }
      // one tile's values at a time (the walk would otherwise keep every tile's products live)
      asm volatile("" : "+v"(acc[rt][0][u]), "+v"(acc[rt][1][u]), "+v"(acc[rt][2][u]), "+v"(acc[rt][3][u]) : : "memory");
    }
  };
  auto fence = [] { asm volatile("" ::: "memory"); };
  auto sync = [&] {
    __builtin_amdgcn_s_barrier();
    fence();
  };
  if (!big) {
    // Every wave issues at least NI / 8 loads per stage, so with at most (NST - 2) * (NI / 8) of them
    // outstanding the older stages, and the scale granules issued before them, have landed.
    auto stage = [&](int i) -> uint4* { return i == 0 ? st0 : i == 1 ? st1 : st2; };
    scale_load(sc0, 0);
#pragma unroll
    for (int p = 0; p < NST - 1; ++p) stage_load(stage(p), p);
    wait_vm<(NST - 2) * (NI / 8)>();
    sync();
#pragma unroll
    for (int seg = 0; seg < NSEG; ++seg) {
      const int q = seg / SPS;
      if (!WHOLE && seg % SPS == 0 && (q + 1) * 16 < NB) scale_load(q & 1 ? sc0 : sc1, q + 1);
      if (seg + NST - 1 < NSEG) stage_load(stage((seg + NST - 1) % NST), seg + NST - 1);
      fence();
      step(std::false_type{}, seg % LC, stage(seg % NST), q & 1 ? sc1 : sc0, seg % SPS, seg);
      fence();
      if (seg + 1 < NSEG) {
        if (NST > 2 && seg + 2 < NSEG)
          wait_vm<(NST - 2) * (NI / 8)>();
        else
          wait_vm<0>();
        sync();
      }
    }
  } else {  // rare: one stage at a time
    if constexpr (WHOLE) scale_load(sc0, 0);
#pragma unroll 1
    for (int seg0 = 0; seg0 < NSEG; seg0 += LC) {
#pragma unroll
      for (int u = 0; u < LC; ++u) {
        const int seg = seg0 + u;
        stage_load(st0, seg);
        if (!WHOLE && seg % SPS == 0) scale_load(sc0, seg / SPS);
        wait_vm<0>();
        sync();
        step(std::true_type{}, u, st0, sc0, seg % SPS, seg);
        fence();
        sync();
      }
    }
  }
  // ---- butterfly levels L/2 .. C in the wave, then the classes' levels through LDS, two row tiles a round ----
  float* part0 = reinterpret_cast<float*>(st0);  // [wave][i][lane]
  float* part1 = reinterpret_cast<float*>(st1);
  static_assert(STU * 16 >= 8 * 4 * 64 * 4 && RT % 2 == 0, "the partials of a row tile");
  __syncthreads();
#pragma unroll
  for (int p = 0; p < RT / 2; ++p) {
    const int ra = MODE == GT_GATE_UP ? p : 2 * p, rb = MODE == GT_GATE_UP ? RT / 2 + p : 2 * p + 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      gt_fold<LC / 2>(acc[ra][i]);
      gt_fold<LC / 2>(acc[rb][i]);
      part0[(wave * 4 + i) * 64 + lane] = acc[ra][i][0];
      part1[(wave * 4 + i) * 64 + lane] = acc[rb][i][0];
    }
    __syncthreads();
    constexpr int PER = 256 / C;  // values per wave and tile
    for (int q0 = 0; q0 < PER; q0 += 64) {
      const int q = q0 + lane, v = c * PER + (q < PER ? q : 0), i = v >> 6, l = v & 63, tok = 4 * (l >> 4) + i;
      float va[C], vb[C];
#pragma unroll
      for (int k = 0; k < C; ++k) {
        va[k] = part0[((rg * C + k) * 4 + i) * 64 + l];
        vb[k] = part1[((rg * C + k) * 4 + i) * 64 + l];
      }
      gt_fold<C / 2>(va);
      gt_fold<C / 2>(vb);
      const uint32_t yr = __shfl((int)yrow_n, tok, 64);
      if (q >= PER || tok >= cnt) continue;
      if constexpr (MODE == GT_GATE_UP) {
        yp[(size_t)yr * rows_w + row0 + my_tile(ra) * 16 + (l & 15)] = f2bf(silu_bf16(round_bf(va[0])) * round_bf(vb[0]));
      } else {
        const int r0 = row0 + my_tile(ra) * 16 + (l & 15), r1 = row0 + my_tile(rb) * 16 + (l & 15);
        if (r0 < rows_w) {
          yp[(size_t)yr * rows_w + r0] = f2bf(va[0]);
          if (MODE == GT_DENSE && yfp) yfp[(size_t)yr * rows_w + r0] = va[0];
        }
        if (r1 < rows_w) {
          yp[(size_t)yr * rows_w + r1] = f2bf(vb[0]);
          if (MODE == GT_DENSE && yfp) yfp[(size_t)yr * rows_w + r1] = vb[0];
        }
      }
    }
    if (p + 1 < RT / 2) __syncthreads();
  }
#endif
}

static bool mat_ok(const uint32_t* w, const bf16* s, const bf16* b) {
  return w && s && b && ((uintptr_t)w & 15) == 0 && word_aligned(s) && word_aligned(b);
}

// ---- dense ----
template <int L, int IT, int C, int RT, int NST, int MINW>
static hipError_t dense_li(GemmArgs a, bool gs32, hipStream_t st) {
  constexpr int R = 8 / C * RT * 16;  // gemm_rows
  a.rblocks1 = (a.mat[0].N + R - 1) / R;
  a.rblocks = a.rblocks1 + (a.mat[1].w ? (a.mat[1].N + R - 1) / R : 0);
  a.tiles = (a.M + 15) / 16;
  const int grid = (a.rblocks * a.tiles + 7) / 8 * 8;
  if (gs32)
    hipLaunchKernelGGL((k_gemm<GT_DENSE, L, IT, C, RT, true, NST, MINW>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((k_gemm<GT_DENSE, L, IT, C, RT, false, NST, MINW>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  return hipGetLastError();
}

static int gemm_shape(int K) {
  const int nb = K / 32, L = lanes_for_blocks(nb);
  return nb % L == 0 ? L * 16 + nb / L : 0;
}

// Rows of a unit of the dense launch, 0 where it has no instance.
static int gemm_rows(int K) {
  switch (gemm_shape(K)) {
    case 16 * 16 + 5: return 128;
    case 32 * 16 + 6: return 64;
    case 64 * 16 + 5: case 64 * 16 + 4: return 32;
    case 2 * 16 + 5: return 256;
    default: return 0;
  }
}

// Scales are loaded by the dword: an odd count of them (K = 320 at group size 64 with an odd N) is not taken.  A grid has
// less than 2^32 threads, the limb form less than 2^31 bytes.
bool gemm_takes(const uint32_t* w, const bf16* s, const bf16* b, int64_t N, int K, int gs, int M) {
  const int R = gemm_rows(K);
  if (!R || M <= MAX_TOKENS || !mat_ok(w, s, b) || N * (K / gs) % 2 != 0 || (int64_t)M * K * 6 >= ((int64_t)1 << 31)) return false;
  return ((N + R - 1) / R * ((M + 15) / 16) + 8) * GT_THREADS < ((int64_t)1 << 32);
}

// A launch takes the walk of one unit over K (23 us at K = 2560, 30 at 10240), whatever it holds, until the units
// fill the chip; the GEMV's windows take about 10 us and grow with the tokens and with tokens times rows.  So windows up
// to a number of each per depth, read off both sides at 8 .. 5120 rows and 9 .. 1024 tokens (us by windows / by the
// GEMM: 324 x 10240, 9 tokens 10 / 30, 64: 26 / 36, 96: 44 / 39; 640 x 6144, 64: 24 / 28, 96: 34 / 30; 160 x 8192, 48:
// 27 / 28, 64: 33 / 30; 8 x 2560, 256: 22 / 24, 512: 36 / 27; 640 x 2560, 128: 20 / 25, 192: 27 / 26; 2560 x 2560, 48:
// 19 / 24, 64: 25 / 24), with and without packed scale rows alike.  Above 5120 rows the GEMM (16480 x 2560, 9 tokens: 24).
// K = 320: equal (10 us) where both prepare x; on blocks that are there the windows save a launch (10240 rows: 9
// tokens 7 / 10, 24: 10 / 10).  The windows of two matrices pay their tokens twice: half as many, and none at K = 2560
// (a mixer's 64 + 4 rows: 9 tokens 18 + 16 / 21, 300 24 + 23 / 22).
bool gemm_faster(int64_t N, int K, int M, bool xp_ready, int mats) {
  int tokens, product;
  switch (gemm_shape(K)) {
    case 16 * 16 + 5: tokens = mats > 1 ? 0 : 300, product = 125000; break;
    case 32 * 16 + 6: tokens = 256, product = 41000; break;
    case 64 * 16 + 4: tokens = 128, product = 10200; break;
    case 64 * 16 + 5: tokens = 256, product = 26000; break;
    default: return !xp_ready || M * N >= 250000;
  }
  return N > 5120 || M * mats > tokens || M * N > product;
}

hipError_t launch_gemm_pair(const uint32_t* w1, const bf16* s1, const bf16* b1, int N1, bf16* y1, float* yf1,
                            const uint32_t* w2, const bf16* s2, const bf16* b2, int N2, bf16* y2, int K, int gs,
                            const XlBatch& x, int M, hipStream_t st) {
  GemmArgs a;
  a.mat[0] = {w1, s1, b1, y1, yf1, N1};
  a.mat[1] = {w2, s2, b2, y2, nullptr, N2};
  a.x = x;
  a.xl_len = (uint32_t)((size_t)M * K * 6);
  a.M = M;
  const bool g32 = gs == 32;
  switch (gemm_shape(K)) {
    case 16 * 16 + 5: return dense_li<16, 5, 4, 4, 3, 4>(a, g32, st);
    case 32 * 16 + 6: return dense_li<32, 6, 4, 2, 3, 4>(a, g32, st);
    case 64 * 16 + 5: return dense_li<64, 5, 8, 2, 2, 4>(a, g32, st);
    case 64 * 16 + 4: return dense_li<64, 4, 8, 2, 2, 4>(a, g32, st);
    case 2 * 16 + 5: return dense_li<2, 5, 2, 4, 2, 4>(a, g32, st);
    default: return hipErrorNotSupported;
  }
}

// ---- MoE ----
// The model's expert width, at any hidden size (1024 wide, 512 experts top-10, 256 tokens: by slots 157 us, by chunks 64 + 9).
bool moe_gemm_down_ok(const MoeArgs& a) {
  return gemm_shape(a.F) == 4 * 16 + 5 && a.M * (a.K + 1) < 65536 && mat_ok(a.down_w, a.down_s, a.down_b) &&
         mat_ok(a.sh_down_w, a.sh_down_s, a.sh_down_b);
}

// The model's hidden size and expert width.
bool moe_gemm_gate_up_ok(const MoeArgs& a) {
  return gemm_shape(a.H) == 16 * 16 + 5 && gemm_shape(a.F) == 4 * 16 + 5 && a.M * (a.K + 1) < 65536 &&
         mat_ok(a.gate_w, a.gate_s, a.gate_b) && mat_ok(a.up_w, a.up_s, a.up_b) &&
         mat_ok(a.sh_gate_w, a.sh_gate_s, a.sh_gate_b) && mat_ok(a.sh_up_w, a.sh_up_s, a.sh_up_b);
}

hipError_t launch_moe_gemm_gate_up(const MoeArgs& m, const XlBatch& x, hipStream_t st) {
  if (!moe_gemm_gate_up_ok(m) || !m.gorder || !m.chunks || !m.chunk_n) return hipErrorInvalidValue;
  const MoeGemmArgs a{m, x, (uint32_t)((size_t)m.M * m.H * 6)};
  const int grid = (m.max_chunks * (m.F / 64) + 7) / 8 * 8;
  if (m.gs == 32)
    hipLaunchKernelGGL((k_gemm<GT_GATE_UP, 16, 5, 4, 4, true, 3, 4>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((k_gemm<GT_GATE_UP, 16, 5, 4, 4, false, 3, 4>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_moe_gemm_down(const MoeArgs& m, const XlBatch& x, hipStream_t st) {
  if (!moe_gemm_down_ok(m) || !m.gorder || !m.chunks || !m.chunk_n) return hipErrorInvalidValue;
  const MoeGemmArgs a{m, x, (uint32_t)((size_t)m.M * (m.K + 1) * m.F * 6)};
  const int grid = (m.max_chunks * ((m.H + 127) / 128) + 7) / 8 * 8;
  if (m.gs == 32)
    hipLaunchKernelGGL((k_gemm<GT_DOWN, 4, 5, 4, 4, true, 2, 6>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((k_gemm<GT_DOWN, 4, 5, 4, 4, false, 2, 6>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  return hipGetLastError();
}

}  // namespace mtpx
