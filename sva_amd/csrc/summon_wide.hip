// Host side of the long-context summon: eligibility, workspace layout and the
// launches (device code in summon_wide.cuh, kernels in summon_wide_*.hip).
#include "summon_wide.cuh"

namespace sva {

using namespace wide;

namespace {

int launch_finish_any(const WideArgs& a, int64_t items, hipStream_t stream) {
  if (a.fv.out == nullptr) return launch_finish_nov(a, items, stream);
  const int kv = a.fv.kv_dtype;
  if (a.fv.D == 64) {
    if (kv == BF16) return launch_finish_v64_bf16(a, items, stream);
    if (kv == F16) return launch_finish_v64_f16(a, items, stream);
    return launch_finish_v64_f32(a, items, stream);
  }
  if (kv == BF16) return launch_finish_v128_bf16(a, items, stream);
  if (kv == F16) return launch_finish_v128_f16(a, items, stream);
  return launch_finish_v128_f32(a, items, stream);
}

}  // namespace

bool summon_wide_eligible(const SummonParams& p, int64_t items) {
  if (p.Q != 1 || p.offs != nullptr || p.ctype != CODE_U8 || p.C > 256) return false;
  if (p.S != 1 && p.S != 2 && p.S != 4 && p.S != 8) return false;
  if (p.R != 64 || p.N < kWideMinKeys || p.N >= (1ll << 30) || items > kMaxWideItems) return false;
  if (p.L > FIN_MAX_L) return false;
  if (((uintptr_t)p.k_low & 15u) != 0 || p.klow_hs % 4 != 0 || ((uintptr_t)p.q_low & 15u) != 0) return false;
  if (p.mask_type != MASK_NONE && p.mask_type != MASK_BOOL && p.mask == nullptr) return false;
  return true;
}

namespace {

// Caches that one workgroup an item holds in LDS (up to about 36000 keys): the
// wide path where its lists are dense enough to be quick and no denser.  Nine
// heads, us a lookup, wide / item: 2x256 at 16385 keys L 512 17 / 33, L 2048 24
// / 38, L 4096 (no floor, or more candidates than the fast finish holds) 57 /
// 39, a float mask (chunks of 8192 keys) and L 2048 96 / 39; 8x32
// (the same chunks) L 2048 90 / 60 at 16385 keys, 75 / 79 at 24576.  By code class (one subspace) the time grows
// with L, the item form's with the keys: L 2048 54 / 42 at 16385, 45 / 50 at
// 24576; under a mask 52 / 38 and L 512.
bool wide_beats_item(const SummonParams& p, int64_t items, bool verify) {
  const bool masked = p.mask_type == MASK_F32 || p.mask_type == MASK_BF16 || p.mask_type == MASK_F16;
  if (summon_class_eligible(p, items)) return !masked && (verify ? 9 : 11) * (int64_t)p.L <= p.N;
  const int kp = scan_keys_per_thread(items, p.N, p.S, masked);
  const int cap = wg_cap((int)((p.N + WB * kp - 1) / (WB * kp)));
  const int ns = sample_blocks(p.N, p.S) * SAMPLE_KEYS, k = sample_floor_rank(p.L, p.N, ns);
  if (k == 0) return false;
  const double all = (double)k * (double)p.N / ns, list = (double)k * (WB * kp) / ns;  // candidates expected
  return all * (1.0 + 2.0 / sqrt((double)k)) <= FAST_M && list <= (masked && p.S < 8 ? 0.7 : 1.4) * cap;
}

}  // namespace

bool summon_wide_taken(const SummonParams& p, int64_t items, bool verify) {
  if (!summon_wide_eligible(p, items)) return false;
  if (p.N >= 32768 && ((uintptr_t)p.codes & 15u) == 0 && p.code_hs % 16 == 0) return true;
  return !item_keys_in_lds(p) || wide_beats_item(p, items, verify);
}

namespace {

size_t wide_bytes(int64_t items, int64_t n_keys, int64_t L) {
  // the largest over the chunk sizes a call may take (scan_keys_per_thread)
  size_t most = 0;
  for (int kp = 8; kp <= MAX_KP; kp *= 2) {
    const int64_t W = (n_keys + WB * kp - 1) / (WB * kp);
    most = std::max(most, counters_bytes(items, W) + lists_bytes(items, W, kp));
  }
  return most + over_bytes(items, std::max<int64_t>(L, 1));
}

}  // namespace

size_t summon_wide_workspace_bytes(int64_t n_seq, int64_t H, int64_t Q, int64_t n_keys, int64_t L) {
  const int64_t items = n_seq * H * Q;
  if (n_keys < kWideMinKeys) return 256;
  // (a packed batch of one sequence and token is a multi call with these sizes too)
  const size_t multi = summon_multi_workspace_bytes(items, n_keys, L);
  if (n_seq != 1 || Q != 1 || items > kMaxWideItems) return multi;
  return std::max(multi, wide_bytes(items, n_keys, L));
}

// Where it replaces one workgroup per item: caches past the register path's
// 16384 keys (below, an item's keys sit in one workgroup's registers), uint8
// codes, no value mask, and shortlists whose usual 2 L candidates the fast
// finish holds.  Four tokens over 262144 keys (4x64, 2048 / 512): 2860 us an
// item a workgroup, 53 here.
bool summon_multi_eligible(const SummonParams& p, int64_t items) {
  if (p.ctype != CODE_U8 || p.C > 256 || p.R != 64) return false;
  if (p.S != 1 && p.S != 2 && p.S != 4 && p.S != 8) return false;
  if (p.N < kWideMinKeys || p.N > kMultiMaxKeys || items > kMultiMaxItems) return false;
  if (2 * p.L > FAST_M || p.sl_idx == nullptr) return false;
  if (((uintptr_t)p.k_low & 15u) != 0 || p.klow_hs % 4 != 0 || ((uintptr_t)p.q_low & 15u) != 0) return false;
  return p.mask_type == MASK_NONE || p.mask_type == MASK_BOOL;
}

namespace {

struct MultiShape {
  int kp, W, cap;
};
MultiShape multi_shape(int64_t items, int64_t n_keys, int S, int L) {
  MultiShape m;
  m.kp = scan_keys_per_thread(items, n_keys, S, false);
  m.W = (int)((n_keys + WB * m.kp - 1) / (WB * m.kp));
  m.cap = 16 * multi_list_expects((int)n_keys, S, L, WB * m.kp) > 11 * MULTI_CAP ? MULTI_CAP_DENSE : MULTI_CAP;
  return m;
}

// Bytes of an item's counts, compact lists and one slice of the all-keys
// select, and what a call needs besides (bounds, more slices of few items,
// alignment).  Both grow with W and L.
int64_t multi_item_bytes(int64_t W, int64_t cap, int64_t L) { return 8 * W + 12 * W * cap + 8 + 8 * L; }
int64_t multi_fixed_bytes(int64_t items, int64_t L) { return 16 * items + kOverGrid * (4 + 8 * L) + 8 * 256; }

// Items a launch may take in `bytes` of workspace (at least 64, or all of
// them, of the size that summon_multi_workspace_bytes gives); 0: too few.
int64_t multi_group(int64_t items, const MultiShape& m, int64_t L, size_t bytes) {
  const int64_t room = ((int64_t)bytes - multi_fixed_bytes(items, L)) / multi_item_bytes(m.W, m.cap, L);
  if (room < std::min<int64_t>(items, 64)) return 0;
  const int64_t groups = (items + room - 1) / room;
  return (items + groups - 1) / groups;
}
size_t multi_lists_bytes(int64_t group, int64_t W, int cap) {
  return align256((size_t)(2 * group * W) * sizeof(uint32_t)) +
         align256((size_t)(group * W * cap) * (sizeof(uint64_t) + sizeof(float)));
}

}  // namespace

// Grows with the key count: lists of the smallest chunks and the largest
// capacity, all items' or MULTI_BYTES of them (64 items' if those take more).
// Where the path ends (kMultiMaxKeys) the size stays: the buffer of a longer
// cache serves shorter ones.
size_t summon_multi_workspace_bytes(int64_t items, int64_t n_keys, int64_t L) {
  if (n_keys < kWideMinKeys || items > kMultiMaxItems || 2 * L > FAST_M) return 256;
  const int64_t W = (std::min(n_keys, kMultiMaxKeys) + 8 * WB - 1) / (8 * WB);
  const int64_t one = multi_item_bytes(W, MULTI_CAP_DENSE, L);
  return (size_t)(multi_fixed_bytes(items, L) + std::min(items * one, std::max<int64_t>(MULTI_BYTES, 64 * one)));
}

// Whether the path is the better one and has room: the longest item's lists
// expect at most eleven sixteenths of what they hold, and MULTI_MOST.  An item
// that outgrows its lists costs an all-keys select of one workgroup: up to
// twice the one-workgroup form while that holds its keys in LDS (up to about
// 36000 keys; 2304 items of 16400 keys, 2x256, 3584 kept: 771 us against 385),
// a quarter of it past that, where every select pass scores every key again
// (65536 keys: 1107 us against 4614).
bool summon_multi_taken(const SummonParams& p, int64_t items, const void* workspace, size_t workspace_bytes) {
  if (!summon_multi_eligible(p, items) || workspace == nullptr || ((uintptr_t)workspace & 255u) != 0) return false;
  const MultiShape m = multi_shape(items, p.N, p.S, p.L);
  const int at_most = std::min(11 * m.cap / 16, MULTI_MOST);
  if (!multi_fits((int)p.N, p.S, p.L, WB * m.kp, at_most) && item_keys_in_lds(p)) return false;
  return multi_group(items, m, p.L, workspace_bytes) > 0;
}

size_t summon_call_workspace_bytes(int64_t items, int64_t n_keys, int64_t R, int64_t S, int64_t C, int64_t L,
                                   int code_type, int mask_type, bool one_token) {
  if (n_keys < kWideMinKeys || code_type != CODE_U8 || C > 256 || R != 64) return 256;
  if (S != 1 && S != 2 && S != 4 && S != 8) return 256;
  if (one_token) return items <= kMaxWideItems && L <= FIN_MAX_L ? wide_bytes(items, n_keys, L) : 256;
  if (mask_type != MASK_NONE && mask_type != MASK_BOOL) return 256;
  return summon_multi_workspace_bytes(items, n_keys, L);
}

int summon_multi_path(const SummonParams& p, int64_t items, void* workspace, size_t workspace_bytes,
                      hipStream_t stream) {
  const MultiShape m = multi_shape(items, p.N, p.S, p.L);
  const int kp = m.kp;
  WideArgs a{};
  a.p = p;
  a.W = m.W;
  a.cap = m.cap;
  a.span_log2 = __builtin_ctz((unsigned)list_span(a.W));
  a.wave_keys = WAVE * kp;
  // (three quarters of a list: the tokens of a call at the route's line, of
  // eleven sixteenths, differ by a few keys)
  a.scan_min = multi_scan_min((int)p.N, p.S, p.L, WB * kp, 3 * m.cap / 4);
  const int64_t group = multi_group(items, m, p.L, workspace_bytes);
  SVA_REQUIRE(group > 0, "summon_multi_path: workspace of %zu bytes is too small", workspace_bytes);
  char* ws = (char*)workspace;
  float* range = (float*)ws;  // the items' bounds and floors
  ws += align256((size_t)(4 * items) * sizeof(float));
  a.wg_count = (uint32_t*)ws;
  a.wg_cand = (uint64_t*)(ws + align256((size_t)(2 * group * a.W) * sizeof(uint32_t)));
  a.wg_rank = (float*)(a.wg_cand + group * a.W * a.cap);
  a.K = over_slices(group);
  char* over = ws + multi_lists_bytes(group, a.W, a.cap);
  a.arrive = (uint32_t*)over;
  a.slice_n = (uint32_t*)(over + align256((size_t)group * sizeof(uint32_t)));
  a.slice_list = (uint64_t*)(over + align256((size_t)group * sizeof(uint32_t)) +
                             align256((size_t)(group * a.K) * sizeof(uint32_t)));
  int rc = launch_multi_floor(a, items, range, stream);
  for (int64_t g = 0; rc == SVA_OK && g < items; g += group) {
    const int64_t n = std::min(group, items - g);
    a.item0 = (int)g;
    a.items = (int)n;
    a.p.lut = p.lut + g * p.S * p.C;
    a.p.range = range + 4 * g;
    a.p.q_low = p.q_low + g * p.R;
    a.p.sl_idx = p.sl_idx + g * p.L;
    a.p.sl_rank = p.sl_rank + g * p.L;
    a.p.sl_count = p.sl_count + g;
    if (p.B > 0) {
      a.p.fin_idx = p.fin_idx + g * p.B;
      a.p.fin_count = p.fin_count + g;
    }
    rc = launch_multi_scan(a, n, kp, stream);
    if (rc == SVA_OK) rc = launch_multi_finish(a, n, stream);
  }
  return rc;
}

bool summon_class_eligible(const SummonParams& p, int64_t items) {
  if (!summon_wide_eligible(p, items) || !class_shape(p.S, p.C, p.L)) return false;
  return (p.N + CLASS_CHUNK - 1) / CLASS_CHUNK <= CLASS_MAX_W;
}

int summon_class_path(const SummonParams& p, void* workspace, size_t workspace_bytes, hipStream_t stream,
                      const FusedVerify* fv, int32_t* overshoot, const QueryLaunch* query) {
  const int64_t items = (int64_t)p.H;  // one sequence, q = 1
  const int64_t W = (p.N + CLASS_CHUNK - 1) / CLASS_CHUNK;
  const size_t counts = align256((size_t)(items * W * 256) * sizeof(uint32_t));
  const size_t bound = align256((size_t)(items * 4) * sizeof(uint32_t));
  const size_t need = counts + bound + align256((size_t)(items * W * 2) * sizeof(uint32_t));
  SVA_REQUIRE(workspace != nullptr && workspace_bytes >= need && ((uintptr_t)workspace & 255u) == 0,
              "sva_summon: workspace of %zu bytes (256-byte aligned) required, got %zu", need, workspace_bytes);
  ClassArgs a;
  a.p = p;
  a.W = (int)W;
  a.overshoot = overshoot;
  a.fv = FusedVerify{};
  a.fv.out = nullptr;
  if (fv != nullptr) {
    SVA_REQUIRE(fused_verify_eligible(p, items, *fv), "summon_class_path: the fused verifier does not fit these sizes");
    a.fv = *fv;
  }
  char* ws = (char*)workspace;
  a.counts = (uint32_t*)ws;
  a.bound = (uint32_t*)(ws + counts);
  a.woff = (uint32_t*)(ws + counts + bound);
  const bool masked = p.mask_type == MASK_F32 || p.mask_type == MASK_BF16 || p.mask_type == MASK_F16;
  return launch_class(a, items, masked, query, stream);
}

bool fused_verify_eligible(const SummonParams& p, int64_t items, const FusedVerify& fv) {
  if (!summon_wide_eligible(p, items) || p.offs != nullptr || items != p.H || p.B <= 0) return false;
  if (fv.D != 64 && fv.D != 128) return false;
  if (fv.G <= 0 || p.H % fv.G != 0) return false;
  if (fv.q_dtype < 0 || fv.q_dtype > 2 || fv.kv_dtype < 0 || fv.kv_dtype > 2 || fv.out_dtype < 0 || fv.out_dtype > 2)
    return false;
  return verify_item_lds(p.B, fv.D) <= kFinLds;
}

int summon_wide_path(const SummonParams& p, void* workspace, size_t workspace_bytes, hipStream_t stream,
                     const FusedVerify* fv, int32_t* overshoot) {
  const int64_t items = (int64_t)p.H;  // one sequence, q = 1
  const size_t need = wide_bytes(items, p.N, p.L);
  SVA_REQUIRE(workspace != nullptr && workspace_bytes >= need && ((uintptr_t)workspace & 255u) == 0,
              "sva_summon: workspace of %zu bytes (256-byte aligned) required, got %zu", need, workspace_bytes);
  // a bool mask allows every key (the reference's `mask > -1e4` rule)
  const bool masked = p.mask_type == MASK_F32 || p.mask_type == MASK_BF16 || p.mask_type == MASK_F16;
  const int kp = scan_keys_per_thread(items, p.N, p.S, masked);
  WideArgs a{};
  a.p = p;
  a.W = (int)((p.N + WB * kp - 1) / (WB * kp));
  a.cap = wg_cap(a.W);
  a.span_log2 = __builtin_ctz((unsigned)list_span(a.W));
  a.wave_keys = WAVE * kp;
  a.overshoot = overshoot;
  a.fv = FusedVerify{};
  a.fv.out = nullptr;
  if (fv != nullptr) {
    SVA_REQUIRE(fused_verify_eligible(p, items, *fv), "summon_wide_path: the fused verifier does not fit these sizes");
    a.fv = *fv;
  }
  char* ws = (char*)workspace;
  a.ncand = (uint32_t*)ws;
  a.nallow = a.ncand + items * a.W * NW;
  a.wg_count = (uint32_t*)(ws + align256((size_t)(2 * items * a.W * NW) * sizeof(uint32_t)));
  a.wg_cand = (uint64_t*)((char*)a.wg_count + align256((size_t)(2 * items * a.W) * sizeof(uint32_t)));
  a.wg_rank = (float*)(a.wg_cand + items * a.W * a.cap);
  a.cand = (uint64_t*)(ws + counters_bytes(items, a.W));
  a.cand_rank = (float*)(a.cand + items * a.W * NW * a.wave_keys);
  a.items = (int)items;
  a.K = over_slices(items);
  a.groups = a.fv.out != nullptr && finish_grouped((int)items, a.fv.G, a.K) ? a.fv.G : 0;
  a.per = a.groups > 0 ? (int)items / a.groups : 0;
  char* over = ws + counters_bytes(items, a.W) + lists_bytes(items, a.W, kp);
  a.arrive = (uint32_t*)over;
  a.slice_n = (uint32_t*)(over + align256((size_t)items * sizeof(uint32_t)));
  a.slice_list = (uint64_t*)(over + align256((size_t)items * sizeof(uint32_t)) +
                             align256((size_t)(items * a.K) * sizeof(uint32_t)));
  const int rc = launch_scan(a, items, masked, kp, stream);
  if (rc != SVA_OK) return rc;
  return launch_finish_any(a, items, stream);
}

}  // namespace sva
