// Residual output adapter of the late-layer socket
// (experiments/sva_late4_logit_distill.py:37-51): for every token,
//   x    = [hidden_states, attn_output]                  (2 * hidden, fp32)
//   corr = up(gelu(down(x))) * scale                     (fp32; exact erf GELU)
//   out  = attn_output + corr.to(attn dtype)             (in the attn dtype)
// down [rank, 2 * hidden] and up [hidden, rank] are fp32 (nn.Linear weights).
//
// One workgroup of 16 waves per NT tokens, their inputs staged in LDS as fp32.
// Down: a wave per output o, its lanes along the 2 * hidden inputs (coalesced
// weight rows, each read once for the NT tokens), then one wave sum a token.
// Up: a thread per output j over the rank's GELU values; its first weights are
// requested at entry and wait through the down projection.  A decode step's
// few tokens are bound by the latency of weights that miss the L2 (the layer
// runs once a step): a workgroup a token takes 8 tokens, hidden 576, rank 16 in
// 15.1 us (most of it the call), where one workgroup for all of them, a sequential chain of 1152
// a thread, took 33.5.  Many tokens share a workgroup's weight reads (NT up to
// 8) once the chip is full.
#include <algorithm>
#include <cmath>

#include "capi_internal.h"
#include "common.cuh"
#include "summon.h"

using namespace sva;

namespace {

constexpr int AB = 1024;         // threads per workgroup
constexpr int MAX_RANK = 64;
constexpr int MAX_TOK = 8;
constexpr int UPF = 16;          // up weights a thread requests at entry

struct AdapterParams {
  const void* hidden;
  int h_dtype;
  int64_t h_rs;
  const void* attn;
  int a_dtype;
  int64_t a_rs;
  const float* down;  // [rank, 2 * H]
  const float* up;    // [H, rank]
  float scale;
  int64_t T;
  int H, rank;
  void* out;
  int o_dtype;
  int64_t o_rs;
};

// The value a float takes after a cast to dtype (round to nearest even).
SVA_DEV float round_to(float v, int dtype) {
  if (dtype == F32) return v;
  if (dtype == BF16) {
    uint32_t u = __float_as_uint(v);
    if ((u & 0x7F800000u) == 0x7F800000u) return v;  // inf and nan pass through
    u += 0x7FFFu + ((u >> 16) & 1u);                 // as store_elem rounds
    return __uint_as_float(u & 0xFFFF0000u);
  }
  return __half2float(__float2half_rn(v));
}

// Floats of a staged token: whole rounds of a wave's float4s, the last one's
// tail zeros.  A lane past the last input multiplies a zero weight by such a
// zero (by an input it would make a NaN of an infinity there).
__host__ __device__ inline int adapter_row(int H) { return (2 * H + 4 * WAVE - 1) / (4 * WAVE) * (4 * WAVE); }

template <int NT>
__global__ void __launch_bounds__(AB) residual_adapter_kernel(AdapterParams p) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) float xs[];  // [NT][adapter_row], then z [NT][MAX_RANK]
  const int H = p.H, H2 = 2 * H, XS = adapter_row(H), rank = p.rank;
  float* z = xs + NT * XS;
  const int64_t t0 = (int64_t)blockIdx.x * NT;
  const int nt = (int)min((int64_t)NT, p.T - t0);
  const int t = threadIdx.x, lane = lane_id();
  const int wid = __builtin_amdgcn_readfirstlane(t / WAVE);
  const bool vec_up = ((uintptr_t)p.up & 15u) == 0 && rank % 4 == 0;
  const bool vec_down = ((uintptr_t)p.down & 15u) == 0 && H2 % 4 == 0;
  // up: the first weights of output j = t (clamped; used where vec_up)
  float4 uw[UPF / 4];
  {
    const float4* row = reinterpret_cast<const float4*>(p.up + (vec_up ? (int64_t)min(t, H - 1) * rank : 0));
#pragma unroll
    for (int u = 0; u < UPF / 4; ++u) uw[u] = vec_up ? row[min(u, rank / 4 - 1)] : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  {
    // the inputs, SU elements a thread per batch: raw bits requested first
    // (indices clamped, every load unconditional), converted at the store
    constexpr int SU = 4;
    const int total = nt * H2;
    for (int e0 = t; e0 < total; e0 += SU * AB) {
      uint32_t bits[SU];
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const int e = min(e0 + u * AB, total - 1);
        const int q = e / H2, k = e - q * H2;
        const bool hid = k < H;
        bits[u] = load_elem_bits(hid ? p.hidden : p.attn, hid ? (t0 + q) * p.h_rs + k : (t0 + q) * p.a_rs + (k - H),
                                 hid ? p.h_dtype : p.a_dtype);
      }
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const int e = e0 + u * AB;
        if (e < total) {
          const int q = e / H2, k = e - q * H2;
          xs[q * XS + k] = elem_from_bits(bits[u], k < H ? p.h_dtype : p.a_dtype);
        }
      }
    }
    // tokens past the last one and the padding: zeros (their results are not stored)
    for (int e = t; e < NT * (XS - H2); e += AB) xs[(e / (XS - H2)) * XS + H2 + e % (XS - H2)] = 0.0f;
    for (int e = nt * XS + t; e < NT * XS; e += AB) xs[e] = 0.0f;
  }
  // down: this wave's first output's weights requested ahead of the barrier
  constexpr int V = 8;  // float4s a lane holds: 2048 inputs a round
  float4 dw[V];
  auto load_row = [&](int o, int k0) {
    const float4* row = reinterpret_cast<const float4*>(p.down + (int64_t)o * H2);
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const int q = k0 / 4 + lane + WAVE * u;
      dw[u] = q < H2 / 4 ? row[q] : float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  if (vec_down && wid < rank) load_row(wid, 0);
  __syncthreads();
  for (int o = wid; o < rank; o += AB / WAVE) {
    float acc[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = 0.0f;
    if (vec_down) {
      for (int k0 = 0; k0 < H2; k0 += 4 * WAVE * V) {
        if (o != wid || k0 > 0) load_row(o, k0);
#pragma unroll
        for (int u = 0; u < V; ++u) {
          const int k = k0 + 4 * (lane + WAVE * u);
          if (k0 + 4 * WAVE * u < H2) {  // uniform
#pragma unroll
            for (int q = 0; q < NT; ++q) {
              const float4 x = *reinterpret_cast<const float4*>(xs + q * XS + k);
              acc[q] = __builtin_fmaf(x.x, dw[u].x, acc[q]);
              acc[q] = __builtin_fmaf(x.y, dw[u].y, acc[q]);
              acc[q] = __builtin_fmaf(x.z, dw[u].z, acc[q]);
              acc[q] = __builtin_fmaf(x.w, dw[u].w, acc[q]);
            }
          }
        }
      }
    } else {
      const float* row = p.down + (int64_t)o * H2;
      for (int k = lane; k < H2; k += WAVE) {
        const float w = row[k];
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[q] = __builtin_fmaf(xs[q * XS + k], w, acc[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const float v = wave_sum(acc[q]);
      if (lane == q) z[q * MAX_RANK + o] = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));  // F.gelu (erf form)
    }
  }
  __syncthreads();
  for (int j = t; j < H; j += AB) {
    const float* w = p.up + (int64_t)j * rank;
    float acc[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = 0.0f;
    if (vec_up) {
      for (int o = 0; o < rank; o += UPF) {
        if (j != t || o > 0) {
#pragma unroll
          for (int u = 0; u < UPF / 4; ++u)
            uw[u] = reinterpret_cast<const float4*>(w)[min(o / 4 + u, rank / 4 - 1)];
        }
#pragma unroll
        for (int u = 0; u < UPF / 4; ++u) {
          if (o + 4 * u < rank) {  // uniform
#pragma unroll
            for (int q = 0; q < NT; ++q) {
              const float4 zz = *reinterpret_cast<const float4*>(z + q * MAX_RANK + o + 4 * u);
              acc[q] = __builtin_fmaf(zz.x, uw[u].x, acc[q]);
              acc[q] = __builtin_fmaf(zz.y, uw[u].y, acc[q]);
              acc[q] = __builtin_fmaf(zz.z, uw[u].z, acc[q]);
              acc[q] = __builtin_fmaf(zz.w, uw[u].w, acc[q]);
            }
          }
        }
      }
    } else {
      for (int o = 0; o < rank; ++o) {
        const float wv = w[o];
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[q] = __builtin_fmaf(z[q * MAX_RANK + o], wv, acc[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      if (q < nt) {  // uniform
        const float corr = round_to(acc[q] * p.scale, p.a_dtype);
        store_elem(p.out, (t0 + q) * p.o_rs + j, p.o_dtype, xs[q * XS + H + j] + corr);
      }
    }
  }
}

template <int NT>
int launch_adapter(const AdapterParams& p, hipStream_t stream) {
  const int64_t blocks = (p.T + NT - 1) / NT;
  SVA_REQUIRE(blocks < (1ll << 31), "sva_residual_adapter: too many tokens");
  const size_t lds = sizeof(float) * (size_t)NT * (size_t)(adapter_row(p.H) + MAX_RANK);
  SVA_SET_MAX_LDS_ONCE(residual_adapter_kernel<NT>, sva::kMaxLds, "hipFuncSetAttribute(residual_adapter_kernel)");
  hipLaunchKernelGGL(residual_adapter_kernel<NT>, dim3((unsigned)blocks), dim3(AB), lds, stream, p);
  SVA_CHECK_LAUNCH("residual_adapter_kernel");
  return SVA_OK;
}

}  // namespace

extern "C" int sva_residual_adapter(const void* hidden, int hidden_dtype, int64_t hidden_row_stride, const void* attn,
                                    int attn_dtype, int64_t attn_row_stride, const float* down_w, const float* up_w,
                                    float scale, int64_t n_tokens, int64_t hidden_size, int64_t rank, void* out,
                                    int out_dtype, int64_t out_row_stride, void* stream) {
  sva::clear_error();
  SVA_REQUIRE(hidden && attn && down_w && up_w && out, "sva_residual_adapter: null pointer");
  SVA_REQUIRE(n_tokens >= 0 && hidden_size > 0 && hidden_size <= 8192, "sva_residual_adapter: bad sizes");
  SVA_UNSUPPORTED(rank > 0 && rank <= MAX_RANK, "sva_residual_adapter: rank %lld (at most %d)", (long long)rank,
                  MAX_RANK);
  SVA_REQUIRE(hidden_dtype >= 0 && hidden_dtype <= 2 && attn_dtype >= 0 && attn_dtype <= 2 && out_dtype >= 0 &&
                  out_dtype <= 2,
              "sva_residual_adapter: bad dtype");
  if (n_tokens == 0) return SVA_OK;
  AdapterParams p;
  p.hidden = hidden;
  p.h_dtype = hidden_dtype;
  p.h_rs = hidden_row_stride;
  p.attn = attn;
  p.a_dtype = attn_dtype;
  p.a_rs = attn_row_stride;
  p.down = down_w;
  p.up = up_w;
  p.scale = scale;
  p.T = n_tokens;
  p.H = (int)hidden_size;
  p.rank = (int)rank;
  p.out = out;
  p.o_dtype = out_dtype;
  p.o_rs = out_row_stride;
  // tokens a workgroup shares its weight reads over: one until every CU has a
  // workgroup, then more, while two workgroups' inputs fit a CU's LDS
  const int64_t room = (72 * 1024) / (int64_t)(sizeof(float) * (adapter_row(p.H) + MAX_RANK));
  const int64_t want = std::min<int64_t>({(n_tokens + 255) / 256, room, MAX_TOK});
  if (want >= 8) return launch_adapter<8>(p, (hipStream_t)stream);
  if (want >= 4) return launch_adapter<4>(p, (hipStream_t)stream);
  if (want >= 2) return launch_adapter<2>(p, (hipStream_t)stream);
  return launch_adapter<1>(p, (hipStream_t)stream);
}
