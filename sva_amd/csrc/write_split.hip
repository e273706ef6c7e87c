// Bulk write path for head_dim = rank = 64 (2x256, 4x64 and 1x256 codes): the
// projection on fp32 MFMA, the assignment by split half-precision scores with
// the rows that those cannot decide taken again in fp32.
//
// Why: the nearest-codeword products are 8 of the path's 9 multiply-adds, and
// on fp32 MFMA they alone bound it (262144 rows, nine heads, 2x256: 97 GFLOP
// at the 154 TFLOP/s a large fp32 product reaches, 0.63 of 1.05 ms).  With x
// and c as sums of two halves, x = xh + xl, three half products (xh ch, xl ch,
// xh cl) cost three sixteenths of that, and the codes stay those of the fp32
// distances: a codeword wins outright when its score
//   v[c] = x.c - |c|^2 / 2   (largest = nearest)
// leads the second largest by more than twice the bound E of either score's
// distance from the fp32 one; the other rows (3 or 4 in 1000 of a subspace
// here) are collected and take the same fp32 MFMA chain, distance order and
// first-index rule as write_encode_persistent_kernel.  One half product alone
// left 6 in 100 to the fp32 chain, which then took 306 of 649 us.
//
// E, in units of the scaled values (x and c times a power of two that puts
// the codebook's largest entry in [64, 128), exact in fp32), with |x|, |c|
// the norms and n = 64 / S <= 64 entries a subspace.  Every fp32 addition and
// product below is taken to be off by an ulp, 2^-23 of its result, whichever
// way the matrix unit rounds:
//   the halves   round to 11 bits: x - xh - xl is within 2^-22 |x|, likewise
//                c, and xl cl is left out, 3 * 2^-22 |x| |c| in all;
//   their sums   start at -|c|^2 / 2; the 2 n small products (2^-10 |x| |c| at
//                most) come first, so 3 n + 1 additions round sums of up to
//                |c|^2 / 2 and n those of up to |x| |c|: n = 64, the largest,
//                2^-17 |x| |c| and 193 * 2^-24 |c|^2;
//   the number   of the lane's codeword in the low six bits of a score:
//                2^-17 (|x| |c| + |c|^2 / 2);
//   |c|^2        n additions: n 2^-24 |c|^2 of its half;
//   the fp32 distances  decided against: n 2^-23 |x| |c| of the product sum
//                and 2^-22 (|x| + |c|)^2 of the two that follow, and 2^-117
//                unscaled where their products fall below fp32's normal range;
//   half subnormals  are off by 2^-25 an entry.
// At n = 64 that is 2.4e-5 |x| |c| + 1.9e-5 |c|^2 and the terms of (|x| + |c|);
// E takes 2^-15 = 3.05e-5 for both and more than the others need.  A row beyond the
// halves' range, or with an infinity or NaN, has no finite lead and is taken
// in fp32.
//
// Layout: a wave works alone, 32 rows at a time, and never meets the others
// after the codebooks are in LDS.  Its rows pass through its own LDS slice
// to the MFMA's k order and meet the map (A operand) there; each lane ends the projection with 16 columns of one row, which are already a B
// operand of the half product once the codebook (A) is stored in the same k
// order, so neither the scores' input nor the scores leave registers.  The
// two 16-row tiles share each codebook read: at 2 KB of LDS a block and 16
// waves that read, not the MFMA, would otherwise be the limit.
#include <algorithm>
#include <type_traits>

#include "capi_internal.h"
#include "common.cuh"
#include "summon.h"
#include "write_few.cuh"

namespace sva {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));

// Threads of the one workgroup a CU holds: as many waves as the registers
// allow (three a SIMD at up to 168) share the map and the codebooks' halves;
// two a SIMD with fp32 keys, whose staging is twice as large.  (Two
// workgroups of six waves left a CU with one: a second six do not fit beside
// the first on the two SIMDs both start from, and half the time was lost.)
template <bool KF32>
constexpr int sp_threads() { return KF32 ? 512 : 768; }
constexpr int SP_TR = 2;              // 16-row tiles a wave takes at once
constexpr int SP_ROWS = 16 * SP_TR;
constexpr int SP_LIST = 96;           // undecided rows a wave keeps per subspace
constexpr int SP_STEPS = 65536 / SP_ROWS;  // tiles whose rows 16 bits number

// LDS row of a staged key row in bytes, two banks past the row.
template <bool KF32>
constexpr int stage_row() { return KF32 ? 64 * 4 + 8 : 64 * 2 + 8; }

template <int S, int SUB, int C, bool KF32>
struct SplitLds {
  float w[64 * 64];           // the map
  _Float16 cbf[2][S * C * SUB];  // high and low halves, fragment-major: ((s * NB + b) * NK + k) * 64 lanes * 8 (4) halves
  float cn[S * C];            // |c|^2 in torch's order
  float cnh[S * C];           // -|c|^2 / 2, scaled
  float scale[S], cmax[S];    // the power of two and the largest scaled codeword norm
  uint32_t red[S][2];
  uint16_t list[sp_threads<KF32>() / WAVE][S][SP_LIST];
  int32_t left[sp_threads<KF32>() / WAVE][S];  // the waves' last undecided rows
  __attribute__((aligned(16))) unsigned char stage[sp_threads<KF32>() / WAVE][SP_ROWS * stage_row<KF32>()];
};

// |x|^2 of the row whose entries k = 4 j + lk lane (lr, lk) holds, in torch's
// sum order (torch_order_dot): eight partial sums over the entries of equal
// k mod 8, four interleaved accumulators each, then the partials in order.
template <int SUB>
SVA_DEV float row_norm(const float (&x)[SUB / 4]) {
#pragma clang fp contract(off)
  const int lr = lane_id() & 15;
  float part[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {  // k mod 8 = lk, 4 + lk
    float a[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      a[v] = 0.0f;
#pragma unroll
      for (int j = 2 * v + o; j < SUB / 4; j += 8) a[v] = a[v] + x[j] * x[j];
    }
    part[o] = ((a[0] + a[1]) + a[2]) + a[3];
  }
  float total = 0.0f;
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int q = 0; q < 4; ++q) total = total + __shfl(part[o], lr + 16 * q);
  return total;
}

// The codes of n <= 16 rows of subspace s in fp32: lane (lr, lk) gives row lr
// (the last one again past n) and holds its k = 4 j + lk entries.
template <int S, int SUB, int C>
SVA_DEV void exact_rows(const WriteParams& p, const float* cb, const float* cn, const float* klow, int64_t code0, int s,
                        int64_t row, int n) {
#pragma clang fp contract(off)
  constexpr int XJ = SUB / 4, NB = C / 16;
  const int l = lane_id(), lr = l & 15, lk = l >> 4;
  const float* x = klow + row * 64 + s * SUB;
  float xb[XJ];
#pragma unroll
  for (int j = 0; j < XJ; ++j) xb[j] = x[4 * j + lk];
  const float xx = row_norm<SUB>(xb);
  float best = INFINITY;
  int arg = 0;
#pragma unroll 1
  for (int b = 0; b < NB; b += 4) {
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < XJ; ++j)
#pragma unroll
      for (int m = 0; m < 4; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(cb[(int64_t)(16 * (b + m) + lr) * SUB + 4 * j + lk], xb[j], acc[m],
                                                      0, 0, 0);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * (b + m) + 4 * lk + i;
        // (xx - 2 x.c) + |c|^2; 2 x.c is exact, so the fma rounds like the subtraction
        const float dist = __builtin_fmaf(-2.0f, acc[m][i], xx) + cn[c];
        if (dist < best) {
          best = dist;
          arg = c;
        }
      }
  }
#pragma unroll
  for (int o = 16; o < WAVE; o <<= 1) {
    const float ob = __shfl_xor(best, o);
    const int oa = __shfl_xor(arg, o);
    if (ob < best || (ob == best && oa < arg)) {
      best = ob;
      arg = oa;
    }
  }
  if (lk == 0 && lr < n) store_code(p.codes, code0 + row * S + s, p.ctype, arg);
}

template <int S, int SUB, int C, bool KF32, bool U8>
__global__ void __launch_bounds__(sp_threads<KF32>(), KF32 ? 2 : 3) write_split_kernel(WriteParams p) {
#pragma clang fp contract(off)
  static_assert(S * SUB == 64 && C % 64 == 0 && (SUB == 16 || SUB % 32 == 0), "shape");
  constexpr int SP_WT = sp_threads<KF32>(), SP_NW = SP_WT / WAVE;
  constexpr int NB = C / 16;               // codeword blocks of a subspace
  constexpr int NK = SUB >= 32 ? SUB / 32 : 1;  // products a block
  constexpr int FE = SUB >= 32 ? 8 : 4;    // halves a lane and product
  constexpr int CM = SUB / 16;             // projection column blocks of a subspace
  constexpr int RS = stage_row<KF32>();
  __shared__ SplitLds<S, SUB, C, KF32> L;
  const int h = blockIdx.y;
  const int g = h / (p.H / p.G);
  const int t = threadIdx.x, l = lane_id(), lr = l & 15, lk = l >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(t / WAVE);  // tiles, rows and lists by scalar arithmetic
  const float* CB = p.codebooks + (int64_t)h * S * C * SUB;
  float* klow = p.k_low + (int64_t)h * p.klow_hs;
  const int64_t code0 = (int64_t)h * p.code_hs;

  // the map in LDS: the A operand of the projection, one read a product for
  // both tiles (64 registers of it a lane would spill the scores')
  for (int i = t; i < 1024; i += SP_WT)
    reinterpret_cast<float4*>(L.w)[i] = reinterpret_cast<const float4*>(p.k_proj + (int64_t)h * 4096)[i];
  // the codebooks: norms, scale, then halves in fragment order
  if (t < S) {
    L.red[t][0] = 0u;
    L.red[t][1] = 0u;
  }
  __syncthreads();
  for (int c = t; c < S * C; c += SP_WT) {
    const float* row = CB + (int64_t)c * SUB;
    const float n = torch_order_dot(row, row, SUB);
    L.cn[c] = n;
    float mx = 0.0f;
    for (int j = 0; j < SUB; ++j) {
      const float a = fabsf(row[j]);
      mx = a <= mx ? mx : a;  // a NaN is kept
    }
    // as unsigned keys: NaN above infinity above every number
    atomicMax(&L.red[c / C][0], __float_as_uint(mx) & 0x7FFFFFFFu);
    atomicMax(&L.red[c / C][1], __float_as_uint(n) & 0x7FFFFFFFu);
  }
  __syncthreads();
  if (t < S) {
    const float mx = __uint_as_float(L.red[t][0]), n2 = __uint_as_float(L.red[t][1]);
    // 2^k with mx 2^k in [64, 128); all-zero and non-finite codebooks (no row is decided by the latter) take 1
    const int ex = (int)(L.red[t][0] >> 23) - 127;
    const int k = mx > 0.0f && mx < INFINITY ? min(max(6 - ex, -100), 100) : 0;
    const float sc = __uint_as_float((uint32_t)(127 + k) << 23);
    L.scale[t] = sc;
    L.cmax[t] = sqrtf(n2) * sc * 1.0001f;  // infinity or NaN: E is not finite, every row goes to fp32
  }
  __syncthreads();
  for (int f = t; f < S * NB * NK * WAVE; f += SP_WT) {
    const int fl = f & 63, fk = (f >> 6) % NK, fb = (f >> 6) / NK % NB, s = (f >> 6) / NK / NB;
    const float* row = CB + ((int64_t)s * C + 16 * fb + (fl & 15)) * SUB;
    const float sc = L.scale[s];
    // a lane's k order: its four columns of each 16-column block, the projection's accumulator order
#pragma unroll
    for (int e = 0; e < FE; ++e) {
      const float v = row[32 * fk + 16 * (e >> 2) + 4 * (fl >> 4) + (e & 3)] * sc;
      const _Float16 hi = (_Float16)v;
      L.cbf[0][f * FE + e] = hi;
      L.cbf[1][f * FE + e] = (_Float16)(v - (float)hi);
    }
  }
  for (int c = t; c < S * C; c += SP_WT) L.cnh[c] = -0.5f * L.cn[c] * L.scale[c / C] * L.scale[c / C];
  __syncthreads();

  const int64_t n_tiles = (p.n_rows + SP_ROWS - 1) / SP_ROWS;
  const int64_t stride = (int64_t)gridDim.x * SP_NW;
  constexpr int CH = KF32 ? 8 : 4;  // 16-byte pieces a lane and tile; a row is 16 (8) of them
  constexpr int CPR = KF32 ? 16 : 8;
  const unsigned char* kbytes = (const unsigned char*)p.keys;
  constexpr int ES = KF32 ? 4 : 2;
  uint4 pre[CH];
  // a tile's address is scalar; a lane adds a 32-bit offset (write_split_eligible bounds the row stride)
  const uint32_t rsb = (uint32_t)(p.kv_rs * ES);
  const unsigned char* kbase = kbytes + ((int64_t)g * p.kv_hs + p.row0 * p.kv_rs) * ES;
  auto last_of = [&](int64_t tile) { return (int)min(p.n_rows - tile * SP_ROWS, (int64_t)SP_ROWS) - 1; };
  auto load_tile = [&](int64_t tile) {
    const unsigned char* src = kbase + tile * SP_ROWS * p.kv_rs * ES;
    const int last = last_of(tile);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int q = l + c * WAVE;
      // past the last row: that row again
      pre[c] = *reinterpret_cast<const uint4*>(src + ((uint32_t)min(q / CPR, last) * rsb + 16u * (uint32_t)(q % CPR)));
    }
  };
  unsigned char* st = L.stage[wid];
  auto stage_tile = [&]() {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int q = l + c * WAVE;
      uint2* dst = reinterpret_cast<uint2*>(st + (q / CPR) * RS + 16 * (q % CPR));
      dst[0] = uint2{pre[c].x, pre[c].y};
      dst[1] = uint2{pre[c].z, pre[c].w};
    }
  };
  uint64_t nlist = 0ull;  // undecided rows held, 16 bits a subspace (uniform)
  int64_t tile = (int64_t)blockIdx.x * SP_NW + wid;
  int64_t tile0 = tile;  // of step 0
  int step = 0;
  auto row_of = [&](int id) { return (tile0 + (id >> 5) * stride) * SP_ROWS + (id & 31); };
  static_assert(SP_ROWS == 32, "row numbers of a step");
  // every undecided row held so far (stored by this wave before)
  auto decide = [&](int least) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll 1
    for (int s = 0; s < S; ++s) {
      int n = (int)((nlist >> (16 * s)) & 0xFFFFull);
#pragma unroll 1
      while (n >= least) {
        const int m = min(n, 16);
        n -= m;
        nlist -= (uint64_t)m << (16 * s);
        exact_rows<S, SUB, C>(p, CB + (int64_t)s * C * SUB, L.cn + s * C, klow, code0, s,
                              p.row0 + row_of(L.list[wid][s][n + min(lr, m - 1)]), m);
      }
    }
  };
  load_tile(min(tile, n_tiles - 1));
  stage_tile();
  // Loads and stores are unconditional (past the end the last tile and row again): the next
  // tile's loads are issued before them and awaited behind them in one straight
  // line, so that with their number known the wait leaves the stores in flight.  Under conditions the compiler
  // waits for every store at each tile: a store's way to memory a tile.
#pragma unroll 1
  for (; tile < n_tiles; tile += stride, ++step) {
    load_tile(min(tile + stride, n_tiles - 1));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_wave_barrier();
    // projection: lane (lr, lk) ends with columns 16 m + 4 lk + i of row lr of each tile
    f32x4 acc[SP_TR][4];
#pragma unroll
    for (int r = 0; r < SP_TR; ++r)
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[r][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      float a[4], b[SP_TR];
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = L.w[(4 * j + lk) * 64 + 16 * m + lr];
#pragma unroll
      for (int r = 0; r < SP_TR; ++r) {
        const unsigned char* src = st + (16 * r + lr) * RS + (4 * j + lk) * ES;
        if (KF32) {
          b[r] = *reinterpret_cast<const float*>(src);
        } else {
          const uint16_t v = *reinterpret_cast<const uint16_t*>(src);
          b[r] = p.kv_dtype == BF16 ? __uint_as_float((uint32_t)v << 16) : __half2float(__ushort_as_half(v));
        }
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < SP_TR; ++r) acc[r][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], b[r], acc[r][m], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
    const int64_t r0 = tile * SP_ROWS;
    const int last = last_of(tile);
    float* klt = klow + (p.row0 + r0) * 64;
    uint32_t row[SP_TR];  // of the tile
#pragma unroll
    for (int r = 0; r < SP_TR; ++r) {
      row[r] = (uint32_t)min(16 * r + lr, last);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        *reinterpret_cast<f32x4*>(reinterpret_cast<char*>(klt) + (256u * row[r] + 16u * (uint32_t)lk + 64u * m)) = acc[r][m];
    }
    uint32_t code[SP_TR];  // u8 codes of the row, one byte a subspace
#pragma unroll
    for (int r = 0; r < SP_TR; ++r) code[r] = 0u;
    // scores of each subspace; the lead of the best over the second decides
    auto subspace = [&](auto sub_index) {
      constexpr int s = decltype(sub_index)::value;
      const float sc = L.scale[s], cm = L.cmax[s];
      half8 xh[SP_TR][NK], xl[SP_TR][NK];
      float x2[SP_TR];
#pragma unroll
      for (int r = 0; r < SP_TR; ++r) {
        x2[r] = 0.0f;
#pragma unroll
        for (int m = 0; m < CM; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = acc[r][s * CM + m][i] * sc;
            x2[r] = __builtin_fmaf(v, v, x2[r]);
            const _Float16 hi = (_Float16)v;
            xh[r][m >> 1][4 * (m & 1) + i] = hi;
            xl[r][m >> 1][4 * (m & 1) + i] = (_Float16)(v - (float)hi);
          }
        x2[r] += __shfl_xor(x2[r], 16);
        x2[r] += __shfl_xor(x2[r], 32);
      }
      float m1[SP_TR], m2[SP_TR];
#pragma unroll
      for (int r = 0; r < SP_TR; ++r) m1[r] = m2[r] = -INFINITY;
      const _Float16* cf = L.cbf[0] + (s * NB * NK * WAVE + l) * FE;
      const float* ch = L.cnh + s * C + 4 * lk;
      // unrolled, the mask in a register: a score takes its number by one and-or
      uint32_t mask = ~63u;
      asm volatile("" : "+s"(mask));
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f32x4 c0 = *reinterpret_cast<const f32x4*>(ch + 16 * b);
        f32x4 v[SP_TR];
        constexpr int LO = S * C * SUB;  // from a high half to its low half
        if constexpr (SUB == 16) {
          const half4 ah = *reinterpret_cast<const half4*>(cf + b * WAVE * FE);
          const half4 al = *reinterpret_cast<const half4*>(cf + b * WAVE * FE + LO);
#pragma unroll
          for (int r = 0; r < SP_TR; ++r) {
            const half4 h = __builtin_shufflevector(xh[r][0], xh[r][0], 0, 1, 2, 3);
            const half4 l = __builtin_shufflevector(xl[r][0], xl[r][0], 0, 1, 2, 3);
            v[r] = __builtin_amdgcn_mfma_f32_16x16x16f16(ah, l, c0, 0, 0, 0);
            v[r] = __builtin_amdgcn_mfma_f32_16x16x16f16(al, h, v[r], 0, 0, 0);
            v[r] = __builtin_amdgcn_mfma_f32_16x16x16f16(ah, h, v[r], 0, 0, 0);
          }
        } else {
          // the small products of every k first, so that only the high ones'
          // additions round sums of the full size (the bound at the top)
          half8 ah[NK];
#pragma unroll
          for (int k = 0; k < NK; ++k) {
            ah[k] = *reinterpret_cast<const half8*>(cf + (b * NK + k) * WAVE * FE);
            const half8 al = *reinterpret_cast<const half8*>(cf + (b * NK + k) * WAVE * FE + LO);
#pragma unroll
            for (int r = 0; r < SP_TR; ++r) v[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[k], xl[r][k], k == 0 ? c0 : v[r], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < SP_TR; ++r) v[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, xh[r][k], v[r], 0, 0, 0);
          }
#pragma unroll
          for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int r = 0; r < SP_TR; ++r) v[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[k], xh[r][k], v[r], 0, 0, 0);
        }
        // the lane's codeword number (4 b + i) in the low bits, then the two largest
#pragma unroll
        for (int r = 0; r < SP_TR; ++r)
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            const float q0 = __uint_as_float((__float_as_uint(v[r][i]) & mask) | (uint32_t)(4 * b + i));
            const float q1 = __uint_as_float((__float_as_uint(v[r][i + 1]) & mask) | (uint32_t)(4 * b + i + 1));
            m2[r] = fmaxf(m2[r], __builtin_amdgcn_fmed3f(m1[r], q0, q1));
            m1[r] = fmaxf(fmaxf(m1[r], q0), q1);
          }
      }
#pragma unroll
      for (int r = 0; r < SP_TR; ++r) {
        const uint32_t id = __float_as_uint(m1[r]) & 63u;
        int arg = (int)(16 * (id >> 2) + 4 * lk + (id & 3u));
#pragma unroll
        for (int o = 16; o < WAVE; o <<= 1) {
          const float o1 = __shfl_xor(m1[r], o), o2 = __shfl_xor(m2[r], o);
          const int oa = __shfl_xor(arg, o);
          m2[r] = fmaxf(fminf(m1[r], o1), fmaxf(m2[r], o2));
          arg = o1 > m1[r] ? oa : arg;
          m1[r] = fmaxf(m1[r], o1);
        }
        const float xn = __builtin_amdgcn_sqrtf(x2[r]) * 1.0001f;
        const float E = (xn * cm + cm * cm) * 0x1p-15f + (xn + cm) * (xn + cm) * 0x1p-21f + (xn + cm) * 0x1p-20f +
                        sc * sc * 0x1p-117f;
        const bool clear = xn < 60000.0f && m1[r] - m2[r] > 2.0f * E;  // false for a NaN anywhere
        // (an undecided row's code is replaced later)
        if (U8) code[r] |= (uint32_t)arg << (8 * s);
        else if (lk == 0) store_code(p.codes, code0 + (p.row0 + r0 + row[r]) * S + s, p.ctype, arg);
        const uint64_t open = __builtin_amdgcn_ballot_w64(l <= min(last - 16 * r, 15) && !clear);
        if (open != 0ull) {
          if ((open >> l) & 1ull)
            L.list[wid][s][((nlist >> (16 * s)) & 0xFFFFull) + __popcll(open & ((1ull << l) - 1ull))] =
                (uint16_t)(SP_ROWS * step + 16 * r + lr);
          nlist += (uint64_t)__popcll(open) << (16 * s);
        }
      }
    };
    subspace(std::integral_constant<int, 0>{});
    if constexpr (S > 1) subspace(std::integral_constant<int, 1>{});
    if constexpr (S > 2) subspace(std::integral_constant<int, 2>{});
    if constexpr (S > 3) subspace(std::integral_constant<int, 3>{});
    if (U8) {
      // all four lanes of a row hold its codes (codes lie at any address)
#pragma unroll
      for (int r = 0; r < SP_TR; ++r) {
        uint8_t* dst = (uint8_t*)p.codes + code0 + (p.row0 + r0) * S + row[r] * (uint32_t)S;
        if constexpr (S == 1) *dst = (uint8_t)code[r];
        if constexpr (S == 2) *reinterpret_cast<u16_any*>(dst) = (uint16_t)code[r];
        if constexpr (S == 4) *reinterpret_cast<u32_any*>(dst) = code[r];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    stage_tile();  // the next tile; this one's rows were last read by the projection
    __builtin_amdgcn_wave_barrier();
    bool full = step == SP_STEPS - 1;
#pragma unroll
    for (int s = 0; s < S; ++s) full = full || ((nlist >> (16 * s)) & 0xFFFFull) > (uint64_t)(SP_LIST - SP_ROWS);
    if (full) {  // uniform
      decide(step == SP_STEPS - 1 ? 1 : 16);
      if (step == SP_STEPS - 1) {
        tile0 = tile + stride;
        step = -1;
      }
    }
  }
  // the waves' last undecided rows together, a batch of 16 a wave in turn
  if (l < S) L.left[wid][l] = (int32_t)((nlist >> (16 * l)) & 0xFFFFull);
  __syncthreads();
  int batch = 0;
#pragma unroll 1
  for (int s = 0; s < S; ++s) {
    int32_t* all = reinterpret_cast<int32_t*>(L.stage[0]);  // the staging is done with
    int total = 0;
    for (int v = 0; v < SP_NW; ++v) {
      const int n = L.left[v][s];
      if (v == wid)
        for (int i = l; i < n; i += WAVE) all[total + i] = (int32_t)row_of(L.list[v][s][i]);
      total += n;
    }
    __syncthreads();
#pragma unroll 1
    for (int a = 0; a < total; a += 16, ++batch)
      if (batch % SP_NW == wid)
        exact_rows<S, SUB, C>(p, CB + (int64_t)s * C * SUB, L.cn + s * C, klow, code0, s,
                              p.row0 + all[min(a + lr, total - 1)], min(16, total - a));
    __syncthreads();
  }
}

template <int S, int SUB, int C, bool KF32, bool U8>
int launch_split_u(const WriteParams& p, hipStream_t stream) {
  constexpr int SP_WT = sp_threads<KF32>(), SP_NW = SP_WT / WAVE;
  static_assert(sizeof(SplitLds<S, SUB, C, KF32>) <= (size_t)kMaxLds, "LDS");
  const int64_t tiles = (p.n_rows + SP_ROWS * SP_NW - 1) / (SP_ROWS * SP_NW);
  const int64_t slots = device_cu_count();
  const int64_t per_head = std::max<int64_t>(1, std::min<int64_t>(tiles, slots / p.H));
  hipLaunchKernelGGL((write_split_kernel<S, SUB, C, KF32, U8>), dim3((unsigned)per_head, (unsigned)p.H), dim3(SP_WT), 0,
                     stream, p);
  SVA_CHECK_LAUNCH("write_split_kernel");
  return SVA_OK;
}

template <int S, int SUB, int C, bool KF32>
int launch_split(const WriteParams& p, hipStream_t stream) {
  return p.ctype == CODE_U8 ? launch_split_u<S, SUB, C, KF32, true>(p, stream)
                            : launch_split_u<S, SUB, C, KF32, false>(p, stream);
}

template <bool KF32>
int launch_split_s(const WriteParams& p, hipStream_t stream) {
  if (p.S == 1) return launch_split<1, 64, 256, KF32>(p, stream);
  if (p.S == 2) return launch_split<2, 32, 256, KF32>(p, stream);
  return launch_split<4, 16, 64, KF32>(p, stream);
}

}  // namespace

bool write_split_eligible(const WriteParams& p) {
  if (p.D != 64 || p.R != 64 || p.codes == nullptr || p.n_rows >= (1ll << 31)) return false;
  // below, the per-workgroup set-up (map, norms, halves: about 35 us) is what
  // counts: nine heads of 4096 rows 44 us here and 43 in fp32, 8192 rows 48
  // and 59, 262144 rows 468 and 1052 (timed calls; 540 under the profiler)
  if (p.n_rows * p.H < 49152) return false;
  if (p.kv_rs < 0 || p.kv_rs > (1ll << 24)) return false;  // 32 rows by 32-bit offsets
  return (p.S == 1 && p.C == 256) || (p.S == 2 && p.C == 256) || (p.S == 4 && p.C == 64);
}

int write_split_launch(const WriteParams& p, hipStream_t stream) {
  return p.kv_dtype == F32 ? launch_split_s<true>(p, stream) : launch_split_s<false>(p, stream);
}

}  // namespace sva
