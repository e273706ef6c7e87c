// Long-context summon of several tokens or sequences: the scan and the finish
// of the one-token path over every (sequence, head, token) item, with each
// item's floor sampled here.
#include "summon_wide.cuh"

namespace sva {
namespace wide {
namespace {

// An item's sampled floor (the query kernels sample for one token of one
// sequence only): the blocks, histogram and rank of summon.h over the item's
// own keys, one workgroup an item; writes the items' [lo, hi, floor, 0], a NaN
// for the floor where the item is not scanned.  Latency bound: one round of
// loads (table and code words), a histogram in LDS and one scan, 6.4 us for 36
// items of 262144 keys.
constexpr int MFB = 512;

template <int S>
__global__ void __launch_bounds__(MFB) multi_floor_kernel(WideArgs a, float* range) {
#pragma clang fp contract(off)
  __shared__ float tab[S * 256];
  __shared__ uint32_t hist[SAMPLE_BINS], scratch[MFB / WAVE + 1], found;
  const SummonParams& p = a.p;
  const int item = blockIdx.x, t = threadIdx.x;
  const ItemAt it = item_at<true>(a, item);
  const float lo = p.range[4 * item], hi = p.range[4 * item + 1];
  auto unsampled = [&](bool scanned) {
    if (t < 4) range[4 * item + t] = t == 0 ? lo : t == 1 ? hi : t == 2 ? (scanned ? -INFINITY : NAN) : 0.0f;
  };
  // an item that its lists would not hold is not scanned for candidates, nor
  // one whose bounds are not finite (infinities or NaN in the table): every
  // key is selected over.  (Exits uniform; the bounds are waited for behind
  // the code words' requests.)
  const int nb = sample_blocks(it.n, S);
  const int rank = multi_floor_rank(it.n, S, p.L);
  const bool fits = it.n >= a.scan_min || it.n <= KL_CAP;
  if (!fits || rank == 0) {
    unsampled(fits && fabsf(lo) < INFINITY && fabsf(hi) < INFINITY);
    return;
  }
  const uint32_t k = (uint32_t)rank;
  const uint8_t* codes = item_codes(p, it);
  constexpr int WPB = SAMPLE_KEYS * S / 16;                                  // code words per block
  constexpr int NWD = (SAMPLE_MAX_BYTES / 16 + MFB - 1) / MFB;               // words per thread at most
  constexpr int KPW = 16 / S;
  const int words = nb * WPB;
  u32x4 w[NWD];
#pragma unroll
  for (int i = 0; i < NWD; ++i) {
    const int g = min(t + i * MFB, words - 1);
    const int64_t n0 = ((int64_t)(g / WPB) * (it.n - SAMPLE_KEYS) / (nb - 1)) & ~(int64_t)15;
    w[i] = code_word(codes + n0 * S + 16 * (g % WPB));
  }
  if (!(hi > lo) || !(fabsf(lo) < INFINITY && fabsf(hi) < INFINITY)) {
    unsampled(fabsf(lo) < INFINITY && fabsf(hi) < INFINITY);
    return;
  }
  const int C = p.C;
  for (int e = t; e < S * C; e += MFB) tab[e] = p.lut[(int64_t)item * S * C + e];
  for (int e = t; e < SAMPLE_BINS; e += MFB) hist[e] = 0u;
  if (t == 0) found = 0u;
  __syncthreads();
  const float inv_w = (float)SAMPLE_BINS / (hi - lo);
#pragma unroll
  for (int i = 0; i < NWD; ++i) {
    if (t + i * MFB < words) {
#pragma unroll
      for (int j = 0; j < KPW; ++j) {
        float acc = 0.0f;
#pragma unroll
        for (int s = 0; s < S; ++s) acc = acc + tab[s * C + min((int)byte_of(w[i], j * S + s), C - 1)];
        const int bin = (int)((acc - lo) * inv_w);
        atomicAdd(&hist[bin < 0 ? 0 : (bin >= SAMPLE_BINS ? SAMPLE_BINS - 1 : bin)], 1u);
      }
    }
  }
  __syncthreads();
  constexpr int BPT = SAMPLE_BINS / MFB;  // bins per thread, from the top
  uint32_t c[BPT], mine = 0u;
#pragma unroll
  for (int j = 0; j < BPT; ++j) {
    c[j] = hist[SAMPLE_BINS - 1 - (BPT * t + j)];
    mine += c[j];
  }
  uint32_t above = block_excl_scan<MFB>(mine, scratch, nullptr);
#pragma unroll
  for (int j = 0; j < BPT; ++j) {
    if (above < k && above + c[j] >= k) found = (uint32_t)(SAMPLE_BINS - 1 - (BPT * t + j));
    above += c[j];
  }
  __syncthreads();
  if (t < 4) range[4 * item + t] = t == 0 ? lo : t == 1 ? hi : t == 2 ? lo + (float)found / inv_w : 0.0f;
}

}  // namespace

int launch_multi_floor(const WideArgs& a, int64_t items, float* range, hipStream_t stream) {
  const dim3 grid((unsigned)items), block(MFB);
  switch (a.p.S) {
    case 1: hipLaunchKernelGGL(multi_floor_kernel<1>, grid, block, 0, stream, a, range); break;
    case 2: hipLaunchKernelGGL(multi_floor_kernel<2>, grid, block, 0, stream, a, range); break;
    case 4: hipLaunchKernelGGL(multi_floor_kernel<4>, grid, block, 0, stream, a, range); break;
    default: hipLaunchKernelGGL(multi_floor_kernel<8>, grid, block, 0, stream, a, range); break;
  }
  SVA_CHECK_LAUNCH("multi_floor_kernel");
  return SVA_OK;
}

int launch_multi_scan(const WideArgs& a, int64_t items, int kp, hipStream_t stream) {
  switch (a.p.S) {
    case 1: return launch_wide_s<1, true>(a, items, false, kp, stream);
    case 2: return launch_wide_s<2, true>(a, items, false, kp, stream);
    case 4: return launch_wide_s<4, true>(a, items, false, kp, stream);
    default: return launch_wide_s<8, true>(a, items, false, kp, stream);
  }
}

int launch_multi_finish(const WideArgs& a, int64_t items, hipStream_t stream) {
  return launch_finish<0, F32, true>(a, items, stream);
}

}  // namespace wide
}  // namespace sva
