// C ABI of the ring-attention block-step library: argument validation (host only, before
// any HIP call) and dispatch to the gfx950 kernels.
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "ra_launch.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(RA_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The kernels reach the rows that one wave moves (up to 16 of them) through an unsigned 32-bit byte
// offset per lane from the wave's first row: rows may not overlap and the row stride stays below 2^27.
constexpr int64_t kMaxRowStride = RA_MAX_ROW_STRIDE;

int check_tensor(const char* name, const ra_tensor& t, int D) {
  if (!t.ptr) return fail(RA_ERR_NULL, "%s.ptr is NULL", name);
  if (!aligned16(t.ptr)) return fail(RA_ERR_ALIGN, "%s.ptr is not 16-byte aligned", name);
  if ((t.stride_b % 8) || (t.stride_h % 8) || (t.stride_l % 8))
    return fail(RA_ERR_ALIGN, "%s strides must be multiples of 8 elements (16 bytes)", name);
  if (t.stride_l < D || t.stride_l > kMaxRowStride)
    return fail(RA_ERR_SHAPE, "%s.stride_l = %lld: the row stride must lie in [D, 2^27] elements", name,
                (long long)t.stride_l);
  return RA_OK;
}

// Token positions (offset + index) stay below 2^30 - 2^16 and the window is clamped to 2^30: every
// position difference, with a window and a tile added, then fits 32 bits in the kernels.
constexpr int64_t kMaxPos = ((int64_t)1 << 30) - (1 << 16);
constexpr int kMaxWindow = 1 << 30;  // wider than any position difference: masks nothing more
constexpr int kMaxLen = 1 << 24;
constexpr int kMaxSegLen = 65536;  // tile-list capacity of the kernels (1024 tiles x 64)

// any_dim: the calls on whole sequences, which take every multiple of 32
int check_dims(int B, int H, int Lq, int Lk, int D, bool any_dim = false) {
  if (B <= 0 || H <= 0 || Lq <= 0 || Lk <= 0)
    return fail(RA_ERR_SHAPE, "B, H, Lq, Lk must be positive (got %d, %d, %d, %d)", B, H, Lq, Lk);
  if (Lq > kMaxLen || Lk > kMaxLen)
    return fail(RA_ERR_SHAPE, "shard length above %d tokens", kMaxLen);
  if ((int64_t)B * H > (1 << 20)) return fail(RA_ERR_SHAPE, "B*H too large");
  // the smallest tile any kernel hands to a workgroup is 128 tokens: the flat grid of the launch
  // must fit the 31 bits of a grid dimension
  const int64_t tiles = ((int64_t)(Lq > Lk ? Lq : Lk) + 127) / 128;
  if ((int64_t)B * H * tiles > 0x7fffffffll)
    return fail(RA_ERR_SHAPE, "B*H*ceil(L/128) = %lld workgroups exceed the grid limit of 2^31-1",
                (long long)((int64_t)B * H * tiles));
  if (any_dim ? (D < 32 || D > 128 || D % 32) : (D != 64 && D != 128))
    return fail(RA_ERR_HEAD_DIM, any_dim ? "head dim %d unsupported (32, 64, 96 or 128)" : "head dim %d unsupported (64 or 128)", D);
  return RA_OK;
}

int check_bias(const ra_bias& b, int Lq, int Lk) {
  const int known = RA_BIAS_CAUSAL | RA_BIAS_WINDOW | RA_BIAS_SEGMENT | RA_BIAS_PREFIX | RA_BIAS_ALIBI |
                    RA_BIAS_DENSE;
  if (b.flags & ~known) return fail(RA_ERR_BIAS, "unknown bias flag bits 0x%x", b.flags & ~known);
  if ((b.flags & RA_BIAS_WINDOW) && b.window <= 0)
    return fail(RA_ERR_BIAS, "window must be positive (got %d)", b.window);
  if ((b.flags & RA_BIAS_CAUSAL) && (b.flags & RA_BIAS_PREFIX))
    return fail(RA_ERR_BIAS, "causal attention does not support a prefix mask");
  if ((b.flags & RA_BIAS_SEGMENT) && (!b.q_segment_ids || !b.kv_segment_ids))
    return fail(RA_ERR_NULL, "segment bias needs q_segment_ids and kv_segment_ids");
  if ((b.flags & RA_BIAS_SEGMENT) && (Lq > kMaxSegLen || Lk > kMaxSegLen))
    return fail(RA_ERR_SHAPE, "segment bias supports shards of at most %d tokens", kMaxSegLen);
  if ((b.flags & RA_BIAS_PREFIX) && (!b.q_prefix || !b.kv_prefix))
    return fail(RA_ERR_NULL, "prefix bias needs q_prefix and kv_prefix");
  if ((b.flags & RA_BIAS_ALIBI) && !b.alibi_slopes)
    return fail(RA_ERR_NULL, "ALiBi bias needs alibi_slopes");
  if (b.flags & RA_BIAS_DENSE) {
    if (!b.dense_bias) return fail(RA_ERR_NULL, "dense bias needs dense_bias");
    if (((uintptr_t)b.dense_bias & 3) != 0) return fail(RA_ERR_ALIGN, "dense_bias is not 4-byte aligned");
    if (b.dense_stride_q < Lk || b.dense_stride_b < 0 || b.dense_stride_h < 0)
      return fail(RA_ERR_BIAS, "dense bias strides: stride_q must be at least Lk, stride_b / stride_h "
                               "non-negative (0 broadcasts)");
    if (b.dense_map && (Lq > kMaxSegLen || Lk > kMaxSegLen))
      return fail(RA_ERR_SHAPE, "a dense bias with its summary supports shards of at most %d tokens", kMaxSegLen);
  }
  if (b.q_offset < 0 || b.kv_offset < 0 || b.q_offset + Lq > kMaxPos || b.kv_offset + Lk > kMaxPos)
    return fail(RA_ERR_BIAS, "token positions (offset + index) must lie in [0, 2^30 - 2^16)");
  return RA_OK;
}

ra::TensorArg to_arg(const ra_tensor& t) {
  return ra::TensorArg{(const ra::bf16_t*)t.ptr, t.stride_b, t.stride_h, t.stride_l};
}

ra::BiasArgs to_bias(const ra_bias& b) {
  ra::BiasArgs r;
  r.flags = b.flags;
  r.window = b.window < kMaxWindow ? b.window : kMaxWindow;
  r.q_off = (int)b.q_offset;
  r.kv_off = (int)b.kv_offset;
  r.q_seg = b.q_segment_ids;
  r.kv_seg = b.kv_segment_ids;
  r.q_seg_sb = b.q_segment_stride_b;
  r.kv_seg_sb = b.kv_segment_stride_b;
  r.q_pre = b.q_prefix;
  r.kv_pre = b.kv_prefix;
  r.q_pre_sb = b.q_prefix_stride_b;
  r.kv_pre_sb = b.kv_prefix_stride_b;
  r.slopes = b.alibi_slopes;
  r.dense = b.dense_bias;
  r.dense_sb = b.dense_stride_b;
  r.dense_sh = b.dense_stride_h;
  r.dense_sq = b.dense_stride_q;
  r.dense_map = (b.flags & RA_BIAS_DENSE) ? b.dense_map : nullptr;
  r.plain_rule = 0;
  return r;
}

// kernel variant: 0 = causal / window only, 1 = per-tile terms, 2 = with a dense bias block
int kernel_mode(int flags) {
  if (flags & RA_BIAS_DENSE) return 2;
  return (flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX | RA_BIAS_ALIBI)) != 0 ? 1 : 0;
}

constexpr float kLog2eHost = 1.4426950408889634f;

ra::FwdArgs to_fwd_args(const ra_fwd_step_params& p) {
  ra::FwdArgs a;
  a.q = to_arg(p.q);
  a.k = to_arg(p.k);
  a.v = to_arg(p.v);
  a.o = p.o;
  a.m = p.m;
  a.l = p.l;
  a.B = p.B;
  a.H = p.H;
  a.Lq = p.Lq;
  a.Lk = p.Lk;
  a.scale2 = p.sm_scale * kLog2eHost;
  a.bias = to_bias(p.bias);
  return a;
}

ra::BwdArgs to_bwd_args(const ra_bwd_step_params& p) {
  ra::BwdArgs a;
  a.q = to_arg(p.q);
  a.k = to_arg(p.k);
  a.v = to_arg(p.v);
  a.dout = to_arg(p.dout);
  a.lse = p.lse;
  a.delta = p.delta;
  a.dq = p.dq;
  a.dk = p.dk;
  a.dv = p.dv;
  a.B = p.B;
  a.H = p.H;
  a.Lq = p.Lq;
  a.Lk = p.Lk;
  a.scale2 = p.sm_scale * kLog2eHost;
  int e2 = 0;
  const float mant = frexpf(a.scale2, &e2);  // scale2 = mant * 2^e2, mant in [0.5, 1)
  a.scale_p2 = ldexpf(1.0f, e2 - 1);
  a.scale_res = mant * 2.0f;
  a.sm_scale = p.sm_scale;
  a.bias = to_bias(p.bias);
  return a;
}

bool same_dims(const ra_bwd_step_params& p, const ra_bwd_step_params& f) {
  return p.B == f.B && p.H == f.H && p.Lq == f.Lq && p.Lk == f.Lk && p.D == f.D && p.sm_scale == f.sm_scale;
}

bool same_strides(const ra_tensor& x, const ra_tensor& y) {
  return x.stride_b == y.stride_b && x.stride_h == y.stride_h && x.stride_l == y.stride_l;
}

// everything of a bias description that belongs to the launch or to the query shard
bool same_q_side(const ra_bias& x, const ra_bias& y) {
  return x.flags == y.flags && x.window == y.window && x.q_offset == y.q_offset &&
         x.q_segment_ids == y.q_segment_ids && x.q_segment_stride_b == y.q_segment_stride_b &&
         x.kv_segment_stride_b == y.kv_segment_stride_b && x.q_prefix == y.q_prefix &&
         x.q_prefix_stride_b == y.q_prefix_stride_b && x.kv_prefix_stride_b == y.kv_prefix_stride_b &&
         x.alibi_slopes == y.alibi_slopes && x.dense_stride_b == y.dense_stride_b &&
         x.dense_stride_h == y.dense_stride_h && x.dense_stride_q == y.dense_stride_q;
}

// ... and to the key/value shard
bool same_kv_side(const ra_bias& x, const ra_bias& y) {
  return x.flags == y.flags && x.window == y.window && x.kv_offset == y.kv_offset &&
         x.kv_segment_ids == y.kv_segment_ids && x.q_segment_stride_b == y.q_segment_stride_b &&
         x.kv_segment_stride_b == y.kv_segment_stride_b && x.kv_prefix == y.kv_prefix &&
         x.q_prefix_stride_b == y.q_prefix_stride_b && x.kv_prefix_stride_b == y.kv_prefix_stride_b &&
         x.alibi_slopes == y.alibi_slopes && x.dense_stride_b == y.dense_stride_b &&
         x.dense_stride_h == y.dense_stride_h && x.dense_stride_q == y.dense_stride_q;
}

// ---- launches that walk several shards, and several ring passes per launch ------------------------
// The travelling side of a step, as the shared table of a ring launch holds it.
struct KvEntry {
  const void* k; const void* v; int64_t off; const int32_t* seg; const int32_t* pre; const float* dense;
  bool operator==(const KvEntry& o) const {
    return k == o.k && v == o.v && off == o.off && seg == o.seg && pre == o.pre && dense == o.dense;
  }
};
struct QEntry {
  const void* q; const void* dout; const float* lse; const float* delta; int64_t off; const int32_t* seg;
  const int32_t* pre; const float* dense;
  bool operator==(const QEntry& o) const {
    return q == o.q && dout == o.dout && lse == o.lse && delta == o.delta && off == o.off && seg == o.seg &&
           pre == o.pre && dense == o.dense;
  }
};
KvEntry kv_entry(const ra_tensor& k, const ra_tensor& v, const ra_bias& b) {
  return KvEntry{k.ptr, v.ptr, b.kv_offset, b.kv_segment_ids, b.kv_prefix, b.dense_bias};
}
QEntry q_entry(const ra_bwd_step_params& p) {
  return QEntry{p.q.ptr, p.dout.ptr, p.lse, p.delta, p.bias.q_offset, p.bias.q_segment_ids, p.bias.q_prefix,
                p.bias.dense_bias};
}
void put(ra::KvShardList& t, int i, const KvEntry& e) {
  t.kv_off[i] = (int)e.off;
  t.k[i] = (const ra::bf16_t*)e.k;
  t.v[i] = (const ra::bf16_t*)e.v;
  t.kv_seg[i] = e.seg;
  t.kv_pre[i] = e.pre;
  t.dense[i] = e.dense;
}
void put(ra::QShardList& t, int i, const QEntry& e) {
  t.q_off[i] = (int)e.off;
  t.q[i] = (const ra::bf16_t*)e.q;
  t.dout[i] = (const ra::bf16_t*)e.dout;
  t.lse[i] = e.lse;
  t.delta[i] = e.delta;
  t.q_seg[i] = e.seg;
  t.q_pre[i] = e.pre;
  t.dense[i] = e.dense;
}

// Plans the launches of `n_passes` ring passes whose live steps (entries of the travelling side)
// are entries[first[p] .. first[p + 1]).  If every pass has at most kMaxShards live steps, there
// are at most kMaxPasses passes and the passes draw from at most kMaxShards distinct shards, ONE
// launch covers them all (heaviest pass first: it is dispatched first); otherwise every pass gets
// its own launches of at most kMaxShards steps each.  Ring is KvRing or QRing, `set_pass(ring,
// slot, p)` fills the resident side of pass p into slot `slot`, `launch(ring)` enqueues.
// `whole`: a whole-ring launch - passes without a live step take part too (their results are
// still to be written), and what does not fit one launch is refused (RA_ERR_TOO_LARGE, nothing
// launched): split into several launches a pass would need its intermediate state in memory.
template <typename Ring, typename Table, typename Entry, typename SetPass, typename Launch>
int run_passes(Table Ring::*table, const std::vector<Entry>& entries, const std::vector<int>& first, int n_passes,
               SetPass set_pass, Launch launch, bool whole = false) {
  std::vector<Entry> distinct;
  std::vector<int> index(entries.size());
  bool one_launch = n_passes <= ra::kMaxPasses;
  for (size_t i = 0; i < entries.size() && one_launch; ++i) {
    size_t j = 0;
    while (j < distinct.size() && !(distinct[j] == entries[i])) ++j;
    if (j == distinct.size()) {
      if ((int)distinct.size() == ra::kMaxShards) one_launch = false;
      else distinct.push_back(entries[i]);
    }
    index[i] = (int)j;
  }
  for (int p = 0; p < n_passes && one_launch; ++p) one_launch = first[p + 1] - first[p] <= ra::kMaxShards;
  Ring ring;
  memset(&ring, 0, sizeof(ring));
  if (one_launch) {
    for (size_t j = 0; j < distinct.size(); ++j) put(ring.*table, (int)j, distinct[j]);
    (ring.*table).n = (int)distinct.size();
    std::vector<int> by_weight;
    for (int p = 0; p < n_passes; ++p)
      if (whole || first[p + 1] > first[p]) by_weight.push_back(p);
    std::stable_sort(by_weight.begin(), by_weight.end(),
                     [&](int x, int y) { return first[x + 1] - first[x] > first[y + 1] - first[y]; });
    if (by_weight.empty()) return RA_OK;
    ring.n_pass = (int)by_weight.size();
    for (int slot = 0; slot < ring.n_pass; ++slot) {
      const int p = by_weight[slot];
      ring.count[slot] = (unsigned char)(first[p + 1] - first[p]);
      for (int i = first[p]; i < first[p + 1]; ++i) ring.order[slot][i - first[p]] = (unsigned char)index[i];
      set_pass(ring, slot, p);
    }
    return launch(ring);
  }
  if (whole)
    return fail(RA_ERR_TOO_LARGE, "a whole-ring launch takes at most %d passes that draw from at most %d distinct "
                                  "travelling shards; use the *_passes entry points", ra::kMaxPasses, ra::kMaxShards);
  for (int p = 0; p < n_passes; ++p) {
    for (int i0 = first[p]; i0 < first[p + 1]; i0 += ra::kMaxShards) {
      const int cnt = std::min(ra::kMaxShards, first[p + 1] - i0);
      memset(&ring, 0, sizeof(ring));
      for (int i = 0; i < cnt; ++i) {
        put(ring.*table, i, entries[i0 + i]);
        ring.order[0][i] = (unsigned char)i;
      }
      (ring.*table).n = cnt;
      ring.n_pass = 1;
      ring.count[0] = (unsigned char)cnt;
      set_pass(ring, 0, p);
      int rc = launch(ring);
      if (rc) return rc;
    }
  }
  return RA_OK;
}

// the fields of a bias description that every step of a launch must share
bool same_bias_shape(const ra_bias& x, const ra_bias& y) {
  return x.flags == y.flags && x.window == y.window && x.q_segment_stride_b == y.q_segment_stride_b &&
         x.kv_segment_stride_b == y.kv_segment_stride_b && x.q_prefix_stride_b == y.q_prefix_stride_b &&
         x.kv_prefix_stride_b == y.kv_prefix_stride_b && x.alibi_slopes == y.alibi_slopes &&
         x.dense_stride_b == y.dense_stride_b && x.dense_stride_h == y.dense_stride_h &&
         x.dense_stride_q == y.dense_stride_q;
}

// Where a whole-ring launch stores what it finished: pass p at `base + p * stride_pass` elements
// (second array for dV), element size `esize`, strides in elements.
struct RingResult {
  void* base;
  void* base2;
  float* lse;
  int dtype;  // RA_DTYPE_*
  int64_t stride_pass, stride_b, stride_h, stride_l;
  bool via_bf16 = false;  // gradients: rounded to bf16 before the conversion
};

int check_ring_result(const char* what, const RingResult& r, bool f16 = false) {
  if (!r.base) return fail(RA_ERR_NULL, "%s: NULL result pointer", what);
  if (r.dtype != RA_DTYPE_BF16 && r.dtype != RA_DTYPE_F32 && !(f16 && r.dtype == RA_DTYPE_F16)) return fail(RA_ERR_DTYPE, "unknown out_dtype %d", r.dtype);
  if ((r.stride_pass % 4) || (r.stride_b % 4) || (r.stride_h % 4) || (r.stride_l % 4))
    return fail(RA_ERR_ALIGN, "%s: result strides must be multiples of 4 elements", what);
  // the kernels store four elements at a time: 8 bytes of bf16 or 16 bytes of fp32
  const unsigned al = r.dtype == RA_DTYPE_F32 ? 16u : 8u;
  if (reinterpret_cast<uintptr_t>(r.base) % al || reinterpret_cast<uintptr_t>(r.base2) % al)
    return fail(RA_ERR_ALIGN, "%s: results must be aligned to four elements (%u bytes)", what, al);
  return RA_OK;
}

int gradient_flags(const RingResult& r) {
  const int kind = r.dtype == RA_DTYPE_F32 ? ra::kFlagWholeF32 : r.dtype == RA_DTYPE_F16 ? ra::kFlagWholeF16 : ra::kFlagWholeBf16;
  return kind | (r.via_bf16 ? ra::kFlagViaBf16 : 0);
}

char* pass_slice(void* base, const RingResult& r, int p) {
  return (char*)base + (int64_t)p * r.stride_pass * (r.dtype == RA_DTYPE_F32 ? 4 : 2);
}

int check_pass_counts(const int32_t* steps_per_pass, int32_t n_passes, std::vector<int>& first) {
  if (n_passes < 0) return fail(RA_ERR_SHAPE, "n_passes is negative");
  if (n_passes > 0 && !steps_per_pass) return fail(RA_ERR_NULL, "steps_per_pass is NULL");
  first.assign(1, 0);
  for (int p = 0; p < n_passes; ++p) {
    if (steps_per_pass[p] < 0) return fail(RA_ERR_SHAPE, "steps_per_pass[%d] is negative", p);
    first.push_back(first.back() + steps_per_pass[p]);
  }
  return RA_OK;
}

// ---- steps on a dense block: the kernels of ra_pair.hip, one launch per step ----------------------------
// What bounds such a step is the block's elementwise term (one fp32 read and add per score), which the long-stretch kernels pay
// in generic iterations, one workgroup per compute unit with nothing beside it; the pair kernels have a second workgroup
// there, and leave a carry or accumulator alone whose tiles are all masked.  Forward + backward, long-stretch kernels -> these:
// document masks (-inf / 0, with their summary) 32768 in 4 shards, H=16, D=128: 18.8 -> 16.0 ms, 5001 in 3, H=16, D=64: 3.42 ->
// 3.00, 4096, B=4, H=32, D=96: 6.69 -> 4.33, 16384 in 8, H=4: 9.3 -> 8.3; blocks of values (every tile evaluated)
// 8192, H=32, D=128: 16.7 -> 10.5 ms, 16384 in 4, H=16: 34.6 -> 23.6, 4096, B=2, H=16, D=64: 3.11 -> 2.51; 512 and 2000 tokens in 8
// shards (host bound): 8.16 -> 8.22 and 8.15 -> 8.23, within the spread of one side (3 %), 810 in 3, H=4: 1.55 -> 1.62 (spread
// 5 to 11 %; several small steps kept in one launch of the long-stretch kernels made no difference: 1.62).
// What a block's summary says is told to each wave for its own 32 rows or keys and each 32 x 32 block of scores: values are read and
// added where there are some, and a block that is -inf throughout is not read.  By workgroup and tile | by wave and block, with the
// pair kernels' shorter steps, us, forward / dQ / dK and dV: documents of 300 in 8192, H=16, D=128 157 / 153 / 233 | 103 / 113 / 175; of 2000
// 478 / 502 / 633 | 306 / 350 / 488; values 1264 / 1365 / 1949 | 905 / 980 / 1475.
bool dense_steps_on_pair(const ra_bias& b) { return b.flags & RA_BIAS_DENSE; }
// dK and dV only where their slabs are more than one per compute unit: a lone workgroup has nothing beside it there, and
// dkdv_kernel the longer pipeline.  dkdv_kernel | dkdv_pair_kernel, us, at 256 slabs (2048, H=16), D=64: a causal mask 53 | 85, zeros
// 49 | 86, documents of 300 125 | 102, values 169 | 145; D=128 72 | 104, 79 | 110, 149 | 126, 192 | 169; at 512 (2048, H=32), D=64: values
// 329 | 217, documents 115 | 74, a causal mask 95 | 104.  (Both launched, with the block's content deciding as below, would cost the
// plain ones a launch, a tenth of these.)
int64_t key_slabs(const ra_bwd_step_params& p) { return (int64_t)p.B * p.H * ((p.Lk + 127) / 128); }
bool dkdv_on_pair(const ra_bwd_step_params& p) { return key_slabs(p) > 256; }
// Four and more steps of a single tile of rows and keys stay one launch of the long-stretch kernels, which keep their
// state in registers from step to step: launching is what such steps cost.  One launch | one per step: ra_fwd_steps, 8 steps of
// 64 x 64, H=4, D=64: 60 | 76 us, of 128 x 128 80 | 93, of 192 x 192 124 | 118; ra_bwd_dq_steps 64 | 80, 85 | 97, 128 | 122.
// 4 steps of 128 x 128: 44 | 47, 2 of them 26 | 24.
template <typename P>
bool one_tile_steps(const P& p, int n_steps) { return n_steps >= 4 && p.Lq <= 128 && p.Lk <= 128; }
// dK and dV of blocks of 8192 and more a side (of 4096 too while all slabs have their place at once) that are zeros over whole
// rows, tiles without a term to evaluate, are what dkdv_kernel is faster at, and dkdv_pair_kernel at all others: there both are
// launched and the block's summary, if it comes with one, says in every workgroup which of them runs (see mostly_plain).  Its one_in:
// of a causal mask's cells one in 64 is of another kind at 4096 tokens, one in 128 at 8192; documents are told by the last row
// of cells, which one of them hardly ever fills.  dkdv_kernel | dkdv_pair_kernel, us, H=16: all zeros 8192, D=64 570 | 698, D=128 981 |
// 1070, a causal mask 352 | 343 and 569 | 603, of 4096 115 | 157 and 165 | 208; documents of 6000 in 8192 1021 | 845 and 827 | 696, of 2000
// in 4096, D=128, 454 | 349, of 300 in 8192, D=64, 181 | 96.
// The forward takes fwd_pair_kernel throughout (fwd_step_kernel | fwd_pair_kernel, D=128: all zeros 8192 658 | 667, a causal mask 386 | 382,
// documents of 6000 in 16384, H=8, 2191 | 912), and so does dQ.
constexpr int kDkdvPlain = 50;
bool choose_by_content(const ra_bias& b, int64_t slabs, int Lq, int Lk) {
  const int side = std::min(Lq, Lk);
  return b.dense_map && (side >= 8192 || (side >= 4096 && slabs <= 512));
}
constexpr int kHeadGroup = 4;  // heads of an XCD that the pair kernels take together (see pair_decode)
constexpr int kWholeRow = 1 << 30;  // chunk_tiles of rows that are not shared

int fwd_step_on_pair(const ra_fwd_step_params& p, void* stream) {
  if (ra_step_is_skippable(&p.bias, p.Lq, p.Lk)) return RA_OK;  // identity on the carry
  ra::PairFwdArgs a;
  memset(&a, 0, sizeof(a));
  a.q = to_arg(p.q);
  a.k = to_arg(p.k);
  a.v = to_arg(p.v);
  a.B = p.B;
  a.H = p.H;
  a.Lq = p.Lq;
  a.Lk = p.Lk;
  a.scale2 = p.sm_scale * kLog2eHost;
  a.bias = to_bias(p.bias);
  a.n_split = 1;
  a.chunk_tiles = kWholeRow;
  a.group = kHeadGroup;
  a.o = p.o;
  a.m = p.m;
  a.l = p.l;
  hipError_t e = ra::launch_fwd_pair(a, p.D, kernel_mode(p.bias.flags), (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "forward step launch");
}

// parts: 1 = dK and dV, 2 = dQ
int bwd_step_on_pair(const ra_bwd_step_params& p, int parts, void* stream) {
  if (ra_step_is_skippable(&p.bias, p.Lq, p.Lk)) return RA_OK;  // contributes nothing
  ra::PairBwdArgs dq;
  memset(&dq, 0, sizeof(dq));
  dq.a = to_bwd_args(p);
  dq.n_split = 1;
  dq.chunk_tiles = kWholeRow;
  dq.group = kHeadGroup;
  ra::PairBwdArgs dkdv = dq;
  dq.acc = p.dq;
  dkdv.acc = p.dk;
  dkdv.acc2 = p.dv;
  const int mode = kernel_mode(p.bias.flags);
  const bool pair = (parts & 1) && dkdv_on_pair(p), other = (parts & 1) && !pair;
  const int rule = pair && choose_by_content(p.bias, key_slabs(p), p.Lq, p.Lk) ? kDkdvPlain : 0;
  dkdv.a.bias.plain_rule = -rule;
  hipError_t e = hipSuccess;
  if (pair || (parts & 2)) e = ra::launch_bwd_pair(pair ? &dkdv : nullptr, (parts & 2) ? &dq : nullptr, p.D, mode, (hipStream_t)stream);
  dkdv.a.bias.plain_rule = rule;
  if (e == hipSuccess && (other || rule)) e = ra::launch_bwd_step(dkdv.a, p.D, mode, 1, (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "backward step launch");
}

// The steps of a single pass on dense blocks, one launch each.  The several-step entry points evaluate whole blocks: only the blocks of
// a launch differ from step to step, a summary that travels with them describes one of them at most.
template <typename P, typename Step>
int steps_on_pair(const P* steps, int n_steps, Step step) {
  int rc = RA_OK;
  for (int i = 0; i < n_steps && !rc; ++i) {
    P p = steps[i];
    p.bias.dense_map = nullptr;
    rc = step(p);
  }
  return rc;
}

int fwd_passes(const ra_fwd_step_params* steps, const std::vector<int>& first, int n_passes, void* stream,
               const RingResult* whole = nullptr) {
  const int total = first.back();
  if (total == 0) return RA_OK;
  if (!steps) return fail(RA_ERR_NULL, "steps is NULL");
  const ra_fwd_step_params& f = steps[0];
  for (int p = 0; p < n_passes; ++p) {
    for (int i = first[p]; i < first[p + 1]; ++i) {
      const ra_fwd_step_params& s = steps[i];
      const ra_fwd_step_params& h = steps[first[p]];  // head of the pass
      ra_fwd_step_params c = s;
      if (whole) c.o = c.m = c.l = reinterpret_cast<float*>(uintptr_t(16));  // not used: there is no carry
      int rc = ra_fwd_step_check(&c);
      if (rc) return rc;
      const bool shape = s.B == f.B && s.H == f.H && s.Lq == f.Lq && s.Lk == f.Lk && s.D == f.D &&
                         s.sm_scale == f.sm_scale && same_strides(s.q, f.q) && same_strides(s.k, f.k) &&
                         same_strides(s.v, f.v) && same_bias_shape(s.bias, f.bias);
      const bool pass = !memcmp(&s.q, &h.q, sizeof(ra_tensor)) &&
                        (whole || (s.o == h.o && s.m == h.m && s.l == h.l)) && same_q_side(s.bias, h.bias);
      if (!shape || !pass)
        return fail(RA_ERR_SHAPE, "steps[%d] differs from the first step of its pass in more than its key/value shard "
                                  "(k.ptr, v.ptr, kv_offset, kv_segment_ids, kv_prefix, dense_bias), or from "
                                  "steps[0] in shape, strides or bias terms", i);
    }
  }
  if (!whole && n_passes == 1 && dense_steps_on_pair(f.bias) && !one_tile_steps(f, total))
    return steps_on_pair(steps, total, [&](const ra_fwd_step_params& p) { return fwd_step_on_pair(p, stream); });
  ra::FwdArgs a = to_fwd_args(f);
  if (whole) {
    a.bias.flags |= whole->dtype == RA_DTYPE_F32 ? ra::kFlagWholeF32 : ra::kFlagWholeBf16;
    a.out_sb = whole->stride_b;  // in the slots of the carry pointers, which have no use here
    a.out_sh = whole->stride_h;
    a.out_sl = whole->stride_l;
  }
  // live steps only: a masked step is an identity on the carry
  std::vector<KvEntry> entries;
  std::vector<int> live_first(1, 0), head(n_passes, 0);
  for (int p = 0; p < n_passes; ++p) {
    head[p] = first[p];
    for (int i = first[p]; i < first[p + 1]; ++i)
      if (!ra_step_is_skippable(&steps[i].bias, steps[i].Lq, steps[i].Lk))
        entries.push_back(kv_entry(steps[i].k, steps[i].v, steps[i].bias));
    live_first.push_back((int)entries.size());
  }
  auto set_pass = [&](ra::KvRing& r, int slot, int p) {
    const ra_fwd_step_params& h = steps[head[p]];
    r.q_off[slot] = (int)h.bias.q_offset;
    r.q[slot] = (const ra::bf16_t*)h.q.ptr;
    r.x0[slot] = h.o;
    r.x1[slot] = h.m;
    r.x2[slot] = h.l;
    if (whole) {
      r.x0[slot] = reinterpret_cast<float*>(pass_slice(whole->base, *whole, p));
      r.x1[slot] = whole->lse + (int64_t)p * f.B * f.H * f.Lq;
      r.x2[slot] = nullptr;
    }
    r.q_seg[slot] = h.bias.q_segment_ids;
    r.q_pre[slot] = h.bias.q_prefix;
  };
  auto launch = [&](const ra::KvRing& r) -> int {
    hipError_t e = ra::launch_fwd_steps(a, r, f.D, kernel_mode(f.bias.flags), (hipStream_t)stream);
    return e == hipSuccess ? RA_OK : hip_fail(e, "forward ring launch");
  };
  return run_passes<ra::KvRing>(&ra::KvRing::kv, entries, live_first, n_passes, set_pass, launch, whole != nullptr);
}

int bwd_dq_passes(const ra_bwd_step_params* steps, const std::vector<int>& first, int n_passes, void* stream,
                  const RingResult* whole = nullptr) {
  const int total = first.back();
  if (total == 0) return RA_OK;
  if (!steps) return fail(RA_ERR_NULL, "steps is NULL");
  const ra_bwd_step_params& f = steps[0];
  for (int p = 0; p < n_passes; ++p) {
    for (int i = first[p]; i < first[p + 1]; ++i) {
      const ra_bwd_step_params& s = steps[i];
      const ra_bwd_step_params& h = steps[first[p]];
      ra_bwd_step_params c = s;
      if (whole) c.dq = c.dk = c.dv = reinterpret_cast<float*>(uintptr_t(16));  // not used: no accumulators
      int rc = ra_bwd_step_check(&c);
      if (rc) return rc;
      const bool shape = same_dims(s, f) && same_strides(s.q, f.q) && same_strides(s.dout, f.dout) &&
                         same_strides(s.k, f.k) && same_strides(s.v, f.v) && same_bias_shape(s.bias, f.bias);
      const bool pass = !memcmp(&s.q, &h.q, sizeof(ra_tensor)) && !memcmp(&s.dout, &h.dout, sizeof(ra_tensor)) &&
                        s.lse == h.lse && s.delta == h.delta && (whole || s.dq == h.dq) && same_q_side(s.bias, h.bias);
      if (!shape || !pass)
        return fail(RA_ERR_SHAPE, "steps[%d] differs from the first step of its pass in more than its key/value shard "
                                  "(k.ptr, v.ptr, dk, dv, kv_offset, kv_segment_ids, kv_prefix, dense_bias), or from "
                                  "steps[0] in shape, strides or bias terms", i);
    }
  }
  if (!whole && n_passes == 1 && dense_steps_on_pair(f.bias) && !one_tile_steps(f, total))
    return steps_on_pair(steps, total, [&](const ra_bwd_step_params& p) { return bwd_step_on_pair(p, 2, stream); });
  ra::BwdArgs a = to_bwd_args(f);
  if (whole) {
    a.bias.flags |= gradient_flags(*whole);
    a.out_sb = whole->stride_b;  // in the slots of the accumulator pointers, which have no use here
    a.out_sh = whole->stride_h;
    a.out_sl = whole->stride_l;
  }
  std::vector<KvEntry> entries;
  std::vector<int> live_first(1, 0);
  for (int p = 0; p < n_passes; ++p) {
    for (int i = first[p]; i < first[p + 1]; ++i)
      if (!ra_step_is_skippable(&steps[i].bias, steps[i].Lq, steps[i].Lk))  // contributes nothing
        entries.push_back(kv_entry(steps[i].k, steps[i].v, steps[i].bias));
    live_first.push_back((int)entries.size());
  }
  auto set_pass = [&](ra::KvRing& r, int slot, int p) {
    const ra_bwd_step_params& h = steps[first[p]];
    r.q_off[slot] = (int)h.bias.q_offset;
    r.q[slot] = (const ra::bf16_t*)h.q.ptr;
    r.dout[slot] = (const ra::bf16_t*)h.dout.ptr;
    r.x0[slot] = whole ? reinterpret_cast<float*>(pass_slice(whole->base, *whole, p)) : h.dq;
    r.x1[slot] = const_cast<float*>(h.lse);
    r.x2[slot] = const_cast<float*>(h.delta);
    r.q_seg[slot] = h.bias.q_segment_ids;
    r.q_pre[slot] = h.bias.q_prefix;
  };
  auto launch = [&](const ra::KvRing& r) -> int {
    hipError_t e = ra::launch_bwd_dq_steps(a, r, f.D, kernel_mode(f.bias.flags), (hipStream_t)stream);
    return e == hipSuccess ? RA_OK : hip_fail(e, "dQ ring launch");
  };
  return run_passes<ra::KvRing>(&ra::KvRing::kv, entries, live_first, n_passes, set_pass, launch, whole != nullptr);
}

int bwd_dkdv_passes(const ra_bwd_step_params* steps, const std::vector<int>& first, int n_passes, void* stream,
                    const RingResult* whole = nullptr) {
  const int total = first.back();
  if (total == 0) return RA_OK;
  if (!steps) return fail(RA_ERR_NULL, "steps is NULL");
  const ra_bwd_step_params& f = steps[0];
  for (int p = 0; p < n_passes; ++p) {
    for (int i = first[p]; i < first[p + 1]; ++i) {
      const ra_bwd_step_params& s = steps[i];
      const ra_bwd_step_params& h = steps[first[p]];
      ra_bwd_step_params c = s;
      if (whole) c.dq = c.dk = c.dv = reinterpret_cast<float*>(uintptr_t(16));  // not used: no accumulators
      int rc = ra_bwd_step_check(&c);
      if (rc) return rc;
      const bool shape = same_dims(s, f) && same_strides(s.q, f.q) && same_strides(s.dout, f.dout) &&
                         same_strides(s.k, f.k) && same_strides(s.v, f.v) && same_bias_shape(s.bias, f.bias);
      const bool pass = !memcmp(&s.k, &h.k, sizeof(ra_tensor)) && !memcmp(&s.v, &h.v, sizeof(ra_tensor)) &&
                        (whole || (s.dk == h.dk && s.dv == h.dv)) && same_kv_side(s.bias, h.bias);
      if (!shape || !pass)
        return fail(RA_ERR_SHAPE, "steps[%d] differs from the first step of its pass in more than its query shard (q.ptr, "
                                  "dout.ptr, lse, delta, dq, q_offset, q_segment_ids, q_prefix, dense_bias), or from "
                                  "steps[0] in shape, strides or bias terms", i);
    }
  }
  // (few slabs stay one launch: 8 steps of 512 x 512, H=32, D=128: 388 us | 498 on dkdv_pair_kernel; 1024 x 1024, H=64: 1496 | 1149)
  if (!whole && n_passes == 1 && dense_steps_on_pair(f.bias) && dkdv_on_pair(f))
    return steps_on_pair(steps, total, [&](const ra_bwd_step_params& p) { return bwd_step_on_pair(p, 1, stream); });
  ra::BwdArgs a = to_bwd_args(f);
  if (whole) {
    a.bias.flags |= gradient_flags(*whole);
    a.out_sb = whole->stride_b;  // in the slots of the accumulator pointers, which have no use here
    a.out_sh = whole->stride_h;
    a.out_sl = whole->stride_l;
  }
  std::vector<QEntry> entries;
  std::vector<int> live_first(1, 0);
  for (int p = 0; p < n_passes; ++p) {
    for (int i = first[p]; i < first[p + 1]; ++i)
      if (!ra_step_is_skippable(&steps[i].bias, steps[i].Lq, steps[i].Lk))  // contributes nothing
        entries.push_back(q_entry(steps[i]));
    live_first.push_back((int)entries.size());
  }
  auto set_pass = [&](ra::QRing& r, int slot, int p) {
    const ra_bwd_step_params& h = steps[first[p]];
    r.kv_off[slot] = (int)h.bias.kv_offset;
    r.k[slot] = (const ra::bf16_t*)h.k.ptr;
    r.v[slot] = (const ra::bf16_t*)h.v.ptr;
    r.dk[slot] = whole ? reinterpret_cast<float*>(pass_slice(whole->base, *whole, p)) : h.dk;
    r.dv[slot] = whole ? reinterpret_cast<float*>(pass_slice(whole->base2, *whole, p)) : h.dv;
    r.kv_seg[slot] = h.bias.kv_segment_ids;
    r.kv_pre[slot] = h.bias.kv_prefix;
  };
  auto launch = [&](const ra::QRing& r) -> int {
    hipError_t e = ra::launch_bwd_dkdv_steps(a, r, f.D, kernel_mode(f.bias.flags), (hipStream_t)stream);
    return e == hipSuccess ? RA_OK : hip_fail(e, "dK/dV ring launch");
  };
  return run_passes<ra::QRing>(&ra::QRing::q, entries, live_first, n_passes, set_pass, launch, whole != nullptr);
}

// ---- one pair of sequences: which kernels, and how many workgroups share a row's keys --------------
constexpr int kPairSlots = 512;  // workgroups of ra_pair.hip that the chip holds at once: two per compute unit
constexpr int kPairRowsHost = 128, kPairKeysHost = 64;

struct PairPlan {
  bool pair;        // the kernels of ra_pair.hip
  int n_split;      // most workgroups that share a row's keys ...
  int chunk_tiles;  // ... each of about this many tiles
  int group;        // heads of an XCD that are taken together (see pair_decode)
};

// Key tiles that one head's query tiles visit (positional terms only): their sum, and the most.
// live: the query tiles that visit any.
void count_key_tiles(const ra_bias& bias, int Lq, int Lk, int64_t& total, int& most, int* live = nullptr) {
  const int ntiles = (Lk + kPairKeysHost - 1) / kPairKeysHost;
  const ra::BiasArgs b = to_bias(bias);
  total = 0;
  most = 0;
  if (live) *live = 0;
  for (int q0 = 0; q0 < Lq; q0 += kPairRowsHost) {
    int lo, hi;
    ra::key_tile_range(b.flags, b.window, b.q_off + q0, b.q_off + std::min(q0 + kPairRowsHost, Lq) - 1, b.kv_off, ntiles,
                       kPairKeysHost, lo, hi);
    total += hi - lo;
    most = std::max(most, hi - lo);
    if (live) *live += hi > lo;
  }
}

// Whether the kernels of ra_fwd.hip / ra_bwd.hip, which hold twice the rows or keys per compute unit and hide all
// vector work in straight-line stretches, are the faster ones: nothing but positions and ALiBi masks, D = 128, a
// grid that fills the chip, and at least `tiles` tiles per workgroup on average.  With a list of tiles (documents,
// prefix, dense block) or D = 64 those of ra_pair.hip are (documents + ALiBi, 32768, H=16: forward 1.1 ms against 1.4,
// dQ 1.25 against 1.53, dK/dV 1.87 against 1.88; causal documents of mean 1024, 8192, B=2, H=16: 0.29 / 0.22 / 0.30
// against 0.39 / 0.35 / 0.42; prefix-LM 16384, H=16: 5.6 ms in total against 18; D=64, 32768 causal, H=16: 2.34 / 2.79 /
// 3.75 against 2.39 / 3.15 / 3.92).
bool long_stretches(const ra_bias& bias, int D, int64_t wgs, int64_t total, int64_t rows, int tiles) {
  const bool lists = bias.flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX | RA_BIAS_DENSE);
  return D == 128 && !lists && wgs > kPairSlots && total >= tiles * rows;
}

// The forward kernels, in 64-key tiles per 128 rows (causal or window, H * B heads; fwd_step_kernel | fwd_pair_kernel):
// 17 of them (64 heads of 2048) 0.118 | 0.096 ms, 65 (32 of 8192) 0.52 | 0.53, 64 (64 of 4096 x 4096) 0.50 | 0.53, 129 (32 of
// 16384) 1.92 | 2.10, 257 (32 of 32768) 7.4 | 8.7; with ALiBi, 129 (16 of 16384): 1.18 | 1.21.
// A grid below 512 workgroups leaves places on the chip empty: the keys of a row are then shared.
// Under a mask that leaves all rows about the same number of keys a count of time says in how many shares
// (plan_split); under a causal mask a share is 1.5 times the mean work of a place, so that the short
// rows stay whole (B=1, D=128, causal, unsplit -> split: H=8, 2048: 46 -> 34 us; H=4, 4096: 85 -> 42 us; H=8,
// 4096: 88 -> 63 us; H=4, 16384: 375 -> 340 us).  At most kMaxSplit shares, and none under kMinChunk tiles, which
// cost more in partial results (528 bytes per row and share) than they gain.
constexpr int kMinChunk = 6, kMaxSplit = 64;
bool has_lists(const ra_bias& b) { return b.flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX | RA_BIAS_DENSE); }
// Whether all of a head's resident tiles have about the same work.
bool even_rows(int64_t total, int most, int64_t rows) { return total * 20 >= (int64_t)most * rows * 17; }
// Whether the pair kernels take an XCD's heads one after the other (see pair_decode): rows that meet about the same number of tiles,
// without a list - unmasked ones, and a few queries behind a long context under a causal mask, ALiBi included.  (Not under a
// window: D=64, 2048 of 16384, 32 heads, 1.23 ms a pass over all heads, 1.27 one by one.)
bool one_by_one(const ra_bias& b, int64_t total, int most, int64_t rows) {
  return even_rows(total, most, rows) && !has_lists(b) && !(b.flags & RA_BIAS_WINDOW);
}
// How the workgroups of one kind of a head's resident tiles, which meet `total` tiles of the other side (`most` at most), share their
// work (see above).  share: bytes of one share of every row.  beside: the other gradient's workgroups run in the same launch.
// Rows of about the same length take the number of shares k that a count of time finds best, in tiles of a workgroup (1.4 us at D = 128):
// the rounds of the fullest compute unit, two workgroups of which are 1.2 times as fast as one (1.4 where a tile has more vector
// work: ALiBi, lists) - or, beside the other kind, which fills what a round leaves, the mean and a quarter - and the shares written and
// read, 4 TB/s.  As many shares as places | by this count, us, forward, then backward: unmasked, D=128, 4096, H=8 94 | 93, 256 | 217;
// 2000, H=4 34 | 30, 71 | 59; 10000, H=4 296 | 247, 795 | 774; 1024, B=2, H=16 47 | 35, 99 | 71; window 1000 of 8192, H=4 46 | 37, 108 | 75;
// 128 x 32768, H=8 63 | 49, 119 | 108; D=80, 864 x 1024, H=32 44 | 39, 82 | 60; ALiBi 4096, H=8 109 | 107, 273 | 237.
// Rows of different lengths on more than half of the places are shared only if they are long and the places not nearly full, causal,
// D=128, shared | not: 14 heads of 4096 (448 workgroups) 104 | 100, 264 | 256; 12 of 4096 (384) 91 | 96, 225 | 230; 24 of 2048 (384) 59 | 54,
// 156 | 150; 3 of 16384 (384) 284 | 326, 736 | 776; 48 of 758 33 | 27, 86 | 81.  Under a list of tiles the lengths are not known: up to half of the
// places as many shares as places, and beyond that long rows of the forward by the count (documents of 3000 in 10000, H=5, D=64, 253
// | 184; short ones lose: documents of 1500 in 4096, H=12, 107 | 121, and so does the backward: prefix 20000, H=3, 1103 | 1202).
void plan_split(PairPlan& r, int64_t heads, int64_t rows, int64_t total, int most, int min_chunk, int64_t share, const ra_bias& bias,
                bool beside) {
  const int64_t wgs = heads * rows;
  if (wgs > kPairSlots || most <= min_chunk) return;
  const bool even = even_rows(total, most, rows), few = wgs <= kPairSlots / 2, lists = has_lists(bias);
  int64_t chunk = even ? (most + kPairSlots / wgs - 1) / (kPairSlots / wgs) : heads * total * 3 / (2 * kPairSlots);
  if (!even && !few && (wgs > kPairSlots * 3 / 4 || most < 8 * min_chunk)) return;
  if (even && lists && !few && (beside || most < 16 * min_chunk)) return;
  if (even && !(lists && few)) {
    const double pair_rate = lists || (bias.flags & RA_BIAS_ALIBI) ? 1.4 : 1.2;
    double least = 0;
    for (int k = 1; k <= std::min(kMaxSplit, (most + min_chunk - 1) / min_chunk); ++k) {
      const int64_t n = (beside ? 2 : 1) * wgs * k, c = std::max((most + k - 1) / k, min_chunk);
      const double rounds = beside ? std::max(1.0, n / (kPairSlots / 2.0) + (n > kPairSlots / 2 ? 0.25 : 0.0)) : (double)((n + kPairSlots / 2 - 1) / (kPairSlots / 2));
      const double cost = rounds * c / (n > kPairSlots / 2 ? pair_rate : 1.0) + (k > 1 ? k * (share * 3.6e-7 + 0.1) + 1 : 0);
      if (k > 1 && cost >= least) continue;
      least = cost;
      chunk = c;
    }
  }
  r.chunk_tiles = (int)std::min<int64_t>(most, std::max<int64_t>({chunk, min_chunk, (most + kMaxSplit - 1) / kMaxSplit}));
  r.n_split = (most + r.chunk_tiles - 1) / r.chunk_tiles;
}
// Whether a single step, into a carry or an accumulator, runs on fwd_pair_kernel (dq_pair_kernel) as well: nothing is shared there.  Under
// a list of tiles always.  At D = 64 always in dQ; in the forward but for even rows of fewer than 192 tiles on more than a workgroup per
// compute unit.  At D = 128 up to a workgroup per compute unit, with uneven rows up to two, and beyond where the rows that see a key
// meet fewer than 56 tiles on average.  fwd_step_kernel | fwd_pair_kernel, then dq_kernel |
// dq_pair_kernel, us: D=128, a causal diagonal of 1024, H=8, 38 | 25 and 44 | 28, of 2048, H=16, 64 | 46 and 72 | 50, of 4096, H=16, 108 | 96 and 132 | 115,
// H=32, 189 | 158 and 239 | 194, of 8192, H=16, 273 | 295 and 353 | 367; unmasked 2048, H=16, 61 | 48 and 72 | 55, 4096, H=16, 132 | 142 and 173 | 176;
// D=64, a diagonal of 4096, H=16, 83 | 68 and 89 | 71, unmasked 85 | 90 and 104 | 102, 8192 314 | 317 and 385 | 373, 16384 1221 | 1215 and 1501 | 1432.
bool step_on_pair(const ra_bias& bias, int B, int H, int Lq, int Lk, int D, bool forward) {
  if (bias.flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX | RA_BIAS_DENSE)) return true;
  int64_t total;
  int most, live;
  count_key_tiles(bias, Lq, Lk, total, most, &live);
  const int64_t rows = (Lq + kPairRowsHost - 1) / kPairRowsHost, wgs = (int64_t)B * H * rows;
  const bool even = even_rows(total, most, rows);
  if (D == 64) return !(forward && even && wgs > kPairSlots / 2 && total < 192 * rows);
  if (wgs <= kPairSlots / 2) return true;
  return wgs <= kPairSlots ? !even : total < 56 * (int64_t)live;
}
PairPlan plan_fwd_pair(const ra_fwd_step_params& p) {
  const int rows = (p.Lq + kPairRowsHost - 1) / kPairRowsHost;
  const int64_t heads = (int64_t)p.B * p.H, wgs = heads * rows;
  int64_t total;
  int most;
  count_key_tiles(p.bias, p.Lq, p.Lk, total, most);
  PairPlan r{true, 1, std::max(most, 1), kHeadGroup};
  // (with ALiBi from 192 tiles on: 65 of them, 32 heads of 8192, 0.70 | 0.63 ms, 129, 16 of 16384, 1.19 | 1.16, 257 4.48 | 4.74; and not
  // uneven rows that fill the chip less than one and a quarter times: 8 heads of 10240, 0.275 | 0.250)
  const bool even = even_rows(total, most, rows), quarter_more = wgs <= kPairSlots * 5 / 4;
  const bool nearly_one = wgs <= (even ? kPairSlots * 3 / 2 : kPairSlots * 5 / 4);
  if (!nearly_one && long_stretches(p.bias, p.D, wgs, total, rows, (p.bias.flags & RA_BIAS_ALIBI) ? 192 : 56)) r.pair = false;
  // Even rows that need up to a quarter more places than there are leave most of the chip empty in their second round: halved if they
  // are long enough for the halves' partial results.  fwd_step_kernel (D = 128) or fwd_pair_kernel unshared | in two shares, us, unmasked: 9 heads
  // of 8192, D=128 429 | 369, D=64 232 | 215, D=96 339 | 303; 18 of 4096 232 | 202, 123 | 119, 180 | 171; 5 of 16384, D=128 826 | 717; not 36 of 2048
  // (32 tiles) 113 | 127, 12 of 8192 (768 workgroups) 436 | 461; nor uneven rows, 18 of 4096, causal, 105 | 116.  Up to one and a half times
  // the places fwd_pair_kernel is the faster one: 24 of 4096 237 | 224, 12 of 8192 439 | 436.
  if (even && wgs > kPairSlots && quarter_more && most >= 56 && !has_lists(p.bias)) {
    r.chunk_tiles = (most + 1) / 2;
    r.n_split = 2;
  }
  if (r.pair) plan_split(r, heads, rows, total, most, kMinChunk, 4 * heads * p.Lq * p.D, p.bias, false);
  if (one_by_one(p.bias, total, most, rows)) r.group = 1;
  return r;
}
// Tiles of the other side that a head's resident tiles of one kind meet: their sum, and the most.
struct TileCount {
  int64_t heads, rows, total;  // rows: resident tiles of a head
  int most;
  bool even;  // (even_rows)
};
// dQ, likewise (dq_kernel | dq_pair_kernel): 65 tiles (32 heads of 8192) 0.70 | 0.66 ms, 66 (window 4096 of 65536, H=8) 1.36 |
// 1.33, 129 (16 of 16384) 1.31 | 1.30, 128 (16 of 8192 x 8192) 0.64 | 0.66, 257 (32 of 32768) 10.1 | 10.4; ALiBi, 129: 1.41 | 1.32.
// beside: dK and dV run in the same launch, if that is what comes out (plan_bwd_pair).
PairPlan plan_dq_pair(const ra_bwd_step_params& p, const TileCount& c, bool beside) {
  PairPlan r{true, 1, std::max(c.most, 1), kHeadGroup};
  if (long_stretches(p.bias, p.D, c.heads * c.rows, c.total, c.rows, 160)) r.pair = false;
  else plan_split(r, c.heads, c.rows, c.total, c.most, kMinChunk, 4 * c.heads * p.Lq * p.D, p.bias, beside);
  if (one_by_one(p.bias, c.total, c.most, c.rows)) r.group = 1;
  return r;
}
// dK / dV, in 32-query tiles per 128 keys (dkdv_kernel | dkdv_pair_kernel): uneven rows 65 of them (64 heads of 4096) 0.55 | 0.50 ms,
// 130 (32 of 8192) 1.08 | 1.04, 258 (32 of 16384) 3.42 | 3.48; even ones 128 (64 of 4096 x 4096) 0.89 | 0.90, 256 (16 of 8192 x 8192) 0.84 |
// 0.89; ALiBi 130 1.03 | 0.95, 258 1.83 | 1.79, 514 7.05 | 7.05.  Between one and two and a half slabs per compute unit dkdv_pair_kernel would
// hold them all at once, the longest one deciding: alone, uneven rows take dkdv_kernel there (16 heads of 4096: 0.13 | 0.16; 12: 0.11 | 0.13; 4
// of 16384: 0.44 | 0.56), even ones if they are long (16 heads of 4096, unmasked 0.230 | 0.233, of 3072 0.158 | 0.153, window of 1024 0.080 |
// 0.070).  With dQ's workgroups beside them in one launch, which fill what the long slabs leave, they are faster: dkdv_kernel, then dQ | both in
// one launch, us: causal 16 heads of 4096 269 | 232, 32 of 2048 174 | 136, 4 of 16384 909 | 844, 8 of 8192 478 | 430, with ALiBi 16 of 4096
// 295 | 246, 17 of 4096 291 | 256, 20 321 | 295, 70 of 1024 124 | 101, 9 of 8192 533 | 498, 5 of 16384 1078 | 1056, 3 of 24000 1463 | 1467, with ALiBi
// 18 of 4096 337 | 272; even rows too, but for long ones that all have a place: unmasked 18 heads of 4096 574 | 486, 9 of 8192 1089 | 958, with ALiBi 1206 |
// 990, 10 of 8192 1112 | 1045, 16 of 4096 435 | 416, window 4096 of 8192, 8 heads 392 | 358; 8 of 8192 796 | 805, 4 of 16384 1560 | 1620.
// Fewer slabs are shared (12 heads of 2048: 0.056 | 0.050).  beside: as for dQ.
PairPlan plan_dkdv_pair(const ra_bwd_step_params& p, const TileCount& c, bool beside) {
  PairPlan r{true, 1, std::max(c.most, 1), kHeadGroup};
  const int64_t wgs = c.heads * c.rows;
  const bool one_round = wgs > kPairSlots / 2 && wgs <= kPairSlots * 5 / 4;
  int tiles = one_round ? (c.even ? 112 : 0) : (p.bias.flags & RA_BIAS_ALIBI) ? 448 : c.even ? 112 : 192;
  if (one_round && beside) tiles = c.even && wgs <= kPairSlots ? 224 : kWholeRow;
  if (long_stretches(p.bias, p.D, one_round ? kPairSlots + 1 : wgs, c.total, c.rows, tiles)) r.pair = false;
  else if (c.heads * p.Lq + 31 >= (int64_t)1 << 30) r.pair = false;  // one 32-bit byte offset reaches both statistics of a tile's 32 rows
  else plan_split(r, c.heads, c.rows, c.total, c.most, 2 * kMinChunk, 8 * c.heads * p.Lk * p.D, p.bias, beside);
  if (one_by_one(p.bias, c.total, c.most, c.rows)) r.group = 1;
  return r;
}
struct BwdPlan {
  PairPlan dq, dkdv;
  bool one_launch;  // of both gradients' workgroups
};
// Both gradients: in one launch where both are on the pair kernels and their workgroups take eight rounds at most; the second kind fills
// the places that the first one's last round leaves empty.  Two launches | one, us: causal, D=128, 512, H=4 46 | 30, 1000, H=8 57 | 41, 640, H=40
// 72 | 55, 6000, H=16 493 | 488, 4096, H=8 180 | 163; window 1000 of 8192, H=4 88 | 74, 300 of 4096, H=2 48 | 31; D=64 causal 2048, B=2, H=16 112 |
// 97, unmasked 512, H=4 33 | 23, 2000, H=8 69 | 56, 3000, H=16 156 | 134, 16384, H=1 266 | 253, 128 x 8192, H=8 39 | 32; D=32, 8192, H=16 338 | 312;
// documents of 500 in 32768, H=8 838 | 793, of 3500 in 10112, causal, H=4, D=80 352 | 278; prefix 4096, B=2, H=16 586 | 576; unmasked 3000,
// H=24 441 | 370.  Past eight rounds (at D <= 64 of 768 workgroups: documents of 2000 in 48128, causal, B=2, H=4, 7.8 of them, a pass
// 1409 | 1296) the last one is a few per cent, and the one launch draws more power
// without a pause (documents of 1200 + ALiBi, 29696, 24 heads: a pass 3.86 | 4.00 ms).
BwdPlan plan_bwd_pair(const ra_bwd_step_params& p) {
  const int64_t heads = (int64_t)p.B * p.H;
  TileCount q{heads, (p.Lq + kPairRowsHost - 1) / kPairRowsHost, 0, 0, false}, k{heads, (p.Lk + kPairRowsHost - 1) / kPairRowsHost, 0, 0, false};
  count_key_tiles(p.bias, p.Lq, p.Lk, q.total, q.most);
  const int ntiles = (p.Lq + 31) / 32;
  const ra::BiasArgs b = to_bias(p.bias);
  for (int k0 = 0; k0 < p.Lk; k0 += kPairRowsHost) {
    int lo, hi;
    ra::query_tile_range(b.flags, b.window, b.kv_off + k0, b.kv_off + std::min(k0 + kPairRowsHost, p.Lk) - 1, b.q_off, ntiles, 32, lo, hi);
    k.total += hi - lo;
    k.most = std::max(k.most, hi - lo);
  }
  q.even = even_rows(q.total, q.most, q.rows);
  k.even = even_rows(k.total, k.most, k.rows);
  const BwdPlan r{plan_dq_pair(p, q, true), plan_dkdv_pair(p, k, true), true};
  const int64_t wgs = heads * (q.rows * r.dq.n_split + k.rows * r.dkdv.n_split);
  if (r.dq.pair && r.dkdv.pair && wgs <= (p.D <= 64 ? 12 : 8) * kPairSlots) return r;
  return {plan_dq_pair(p, q, false), plan_dkdv_pair(p, k, false), false};
}
// The workspace of ra_bwd_pair: the rows' statistics, then the shares of dQ and of dK and dV.
struct BwdSpace {
  int64_t delta, stat, dq_part, dq_n, dkdv_part, dkdv_n, total;  // byte offsets (16-byte aligned) and the size
};
BwdSpace bwd_space(const ra_bwd_step_params& p, const PairPlan& dq, const PairPlan& dkdv) {
  BwdSpace s;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 15) & ~(int64_t)15;
    return here;
  };
  auto tiles = [](int L) { return (int64_t)(L + kPairRowsHost - 1) / kPairRowsHost; };
  const int64_t heads = (int64_t)p.B * p.H, q_rows = heads * p.Lq, k_rows = heads * p.Lk;
  s.delta = take(4 * q_rows);
  s.stat = take(8 * q_rows);
  s.dq_part = take(dq.n_split > 1 ? 4 * dq.n_split * q_rows * p.D : 0);
  s.dq_n = take(dq.n_split > 1 ? 4 * heads * tiles(p.Lq) : 0);
  s.dkdv_part = take(dkdv.n_split > 1 ? 8 * dkdv.n_split * k_rows * p.D : 0);
  s.dkdv_n = take(dkdv.n_split > 1 ? 4 * heads * tiles(p.Lk) : 0);
  s.total = at;
  return s;
}
int64_t fwd_part_rows(const ra_fwd_step_params& p, int n_split) { return (int64_t)n_split * p.B * p.H * p.Lq; }
int64_t fwd_part_bytes(const ra_fwd_step_params& p, int n_split) {
  return 4 * (fwd_part_rows(p, n_split) * (p.D + 4) + (int64_t)p.B * p.H * ((p.Lq + kPairRowsHost - 1) / kPairRowsHost));
}

}  // namespace

extern "C" {

int ra_version(void) { return 1009; }

static int64_t fwd_pair_workspace(const ra_fwd_step_params* p, bool any_dim) {
  if (!p || check_dims(p->B, p->H, p->Lq, p->Lk, p->D, any_dim)) return 0;
  const int n = plan_fwd_pair(*p).n_split;
  return n > 1 ? fwd_part_bytes(*p, n) : 0;
}

// A head dim that only the kernels of ra_pair.hip have, and those without a dense block.
static bool narrow(int D) { return D != 64 && D != 128; }
static int check_whole_call(const char* what, int D, const ra_bias& bias) {
  if (narrow(D) && (bias.flags & RA_BIAS_DENSE))
    return fail(RA_ERR_HEAD_DIM, "%s: head dim %d with a dense block (64 or 128)", what, D);
  return RA_OK;
}
static int check_fwd_step(const ra_fwd_step_params* p, bool any_dim);
static int check_bwd_step(const ra_bwd_step_params* p, bool any_dim);

// The conversions that go before a call, which has been checked by then: nothing is launched for one that is refused.
struct Before {
  const ra_rows* items;
  int32_t n;
  int launch(void* stream) const { return n ? ra_convert(items, n, stream) : RA_OK; }
};

static int fwd_pair(const Before& before, const ra_fwd_step_params* p, bool any_dim, void* out, int32_t out_dtype, int64_t out_stride_b,
                    int64_t out_stride_h, int64_t out_stride_l, float* lse, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!p) return fail(RA_ERR_NULL, "params is NULL");
  ra_fwd_step_params c = *p;
  c.o = c.m = c.l = reinterpret_cast<float*>(uintptr_t(16));  // not used: there is no carry
  int rc = check_fwd_step(&c, any_dim);
  if (rc || (rc = check_whole_call("ra_fwd_whole", c.D, c.bias))) return rc;
  if (!lse) return fail(RA_ERR_NULL, "ra_fwd_pair: lse is NULL");
  const RingResult r{out, nullptr, lse, out_dtype, 0, out_stride_b, out_stride_h, out_stride_l};
  if ((rc = check_ring_result("ra_fwd_pair", r))) return rc;
  const PairPlan plan = plan_fwd_pair(*p);
  if (!plan.pair) return (rc = before.launch(stream)) ? rc : fwd_passes(p, std::vector<int>{0, 1}, 1, stream, &r);
  ra::PairFwdArgs a;
  memset(&a, 0, sizeof(a));
  a.q = to_arg(p->q);
  a.k = to_arg(p->k);
  a.v = to_arg(p->v);
  a.B = p->B;
  a.H = p->H;
  a.Lq = p->Lq;
  a.Lk = p->Lk;
  a.scale2 = p->sm_scale * kLog2eHost;
  a.bias = to_bias(p->bias);
  a.n_split = plan.n_split;
  a.chunk_tiles = plan.chunk_tiles;
  a.group = plan.group;
  a.out = out;
  a.out_f32 = out_dtype == RA_DTYPE_F32;
  a.out_sb = out_stride_b;
  a.out_sh = out_stride_h;
  a.out_sl = out_stride_l;
  a.lse = lse;
  if (plan.n_split > 1) {
    const int64_t rows = fwd_part_rows(*p, plan.n_split);
    if (!workspace || !aligned16(workspace)) return fail(RA_ERR_ALIGN, "ra_fwd_pair: the workspace must be 16-byte aligned");
    if (workspace_bytes < fwd_part_bytes(*p, plan.n_split))
      return fail(RA_ERR_SHAPE, "ra_fwd_pair: the workspace is smaller than ra_fwd_pair_workspace()");
    a.part_o = (float*)workspace;
    a.part_s = a.part_o + rows * p->D;
    a.part_n = (int*)(a.part_s + rows * 4);
  }
  if ((rc = before.launch(stream))) return rc;
  hipError_t e = ra::launch_fwd_pair(a, p->D, kernel_mode(p->bias.flags), (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_fwd_pair launch");
}

int64_t ra_fwd_pair_workspace(const ra_fwd_step_params* p) { return fwd_pair_workspace(p, false); }
int64_t ra_fwd_whole_workspace(const ra_fwd_step_params* p) { return fwd_pair_workspace(p, true); }

int ra_fwd_pair(const ra_fwd_step_params* p, void* out, int32_t out_dtype, int64_t out_stride_b, int64_t out_stride_h,
                int64_t out_stride_l, float* lse, void* workspace, int64_t workspace_bytes, void* stream) {
  return fwd_pair({}, p, false, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, lse, workspace, workspace_bytes, stream);
}
int ra_fwd_whole(const ra_fwd_step_params* p, void* out, int32_t out_dtype, int64_t out_stride_b, int64_t out_stride_h,
                 int64_t out_stride_l, float* lse, void* workspace, int64_t workspace_bytes, void* stream) {
  return fwd_pair({}, p, true, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, lse, workspace, workspace_bytes, stream);
}

const char* ra_last_error(void) { return g_err; }

int ra_step_is_skippable(const ra_bias* bias, int32_t Lq, int32_t Lk) {
  if (!bias || Lq <= 0 || Lk <= 0) return 0;
  if (bias->flags & RA_BIAS_PREFIX) return 0;
  const int64_t qlo = bias->q_offset, qhi = bias->q_offset + Lq - 1;
  const int64_t klo = bias->kv_offset, khi = bias->kv_offset + Lk - 1;
  if ((bias->flags & RA_BIAS_CAUSAL) && klo > qhi) return 1;
  if (bias->flags & RA_BIAS_WINDOW) {
    if (qlo - khi >= bias->window) return 1;
    if (!(bias->flags & RA_BIAS_CAUSAL) && klo - qhi >= bias->window) return 1;
  }
  return 0;
}

static int check_fwd_step(const ra_fwd_step_params* p, bool any_dim) {
  if (!p) return fail(RA_ERR_NULL, "params is NULL");
  int rc = check_dims(p->B, p->H, p->Lq, p->Lk, p->D, any_dim);
  if (rc) return rc;
  if ((rc = check_tensor("q", p->q, p->D))) return rc;
  if ((rc = check_tensor("k", p->k, p->D))) return rc;
  if ((rc = check_tensor("v", p->v, p->D))) return rc;
  if (!p->o || !p->m || !p->l) return fail(RA_ERR_NULL, "carry pointer (o, m or l) is NULL");
  if (!aligned16(p->o)) return fail(RA_ERR_ALIGN, "o is not 16-byte aligned");
  if (!(p->sm_scale > 0.f) || p->sm_scale > 3.0e38f)
    return fail(RA_ERR_SHAPE, "sm_scale must be a positive finite number");
  return check_bias(p->bias, p->Lq, p->Lk);
}

static int check_bwd_step(const ra_bwd_step_params* p, bool any_dim) {
  if (!p) return fail(RA_ERR_NULL, "params is NULL");
  int rc = check_dims(p->B, p->H, p->Lq, p->Lk, p->D, any_dim);
  if (rc) return rc;
  if ((rc = check_tensor("q", p->q, p->D))) return rc;
  if ((rc = check_tensor("k", p->k, p->D))) return rc;
  if ((rc = check_tensor("v", p->v, p->D))) return rc;
  if ((rc = check_tensor("dout", p->dout, p->D))) return rc;
  if (!p->lse || !p->delta) return fail(RA_ERR_NULL, "lse or delta is NULL");
  if (!p->dq || !p->dk || !p->dv) return fail(RA_ERR_NULL, "gradient accumulator (dq, dk or dv) is NULL");
  if (!aligned16(p->dq) || !aligned16(p->dk) || !aligned16(p->dv))
    return fail(RA_ERR_ALIGN, "gradient accumulators must be 16-byte aligned");
  if (!(p->sm_scale > 0.f) || p->sm_scale > 3.0e38f)
    return fail(RA_ERR_SHAPE, "sm_scale must be a positive finite number");
  return check_bias(p->bias, p->Lq, p->Lk);
}

int ra_fwd_step_check(const ra_fwd_step_params* p) { return check_fwd_step(p, false); }
int ra_bwd_step_check(const ra_bwd_step_params* p) { return check_bwd_step(p, false); }

int ra_fwd_init(float* o, float* m, float* l, int32_t B, int32_t H, int32_t Lq, int32_t D, void* stream) {
  if (!o || !m || !l) return fail(RA_ERR_NULL, "carry pointer (o, m or l) is NULL");
  int rc = check_dims(B, H, Lq, 1, D);
  if (rc) return rc;
  hipError_t e = ra::launch_fwd_init(o, m, l, (long long)B * H * Lq, D, (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_fwd_init launch");
}

int64_t ra_dense_map_bytes(int64_t stride_b, int64_t stride_h, int32_t B, int32_t H, int32_t Lq, int32_t Lk) {
  if (B <= 0 || H <= 0 || Lq <= 0 || Lk <= 0) return 0;
  const int64_t cells = (int64_t)((Lq + 31) / 32) * ((Lk + 31) / 32);
  return (stride_b ? B : 1) * (int64_t)(stride_h ? H : 1) * cells;
}

int ra_dense_map(const float* dense_bias, int64_t stride_b, int64_t stride_h, int64_t stride_q, int32_t B,
                 int32_t H, int32_t Lq, int32_t Lk, uint8_t* map, void* stream) {
  if (!dense_bias || !map) return fail(RA_ERR_NULL, "ra_dense_map: NULL pointer");
  if (B <= 0 || H <= 0 || Lq <= 0 || Lk <= 0)
    return fail(RA_ERR_SHAPE, "ra_dense_map: bad shape B=%d H=%d Lq=%d Lk=%d", B, H, Lq, Lk);
  if (Lq > kMaxSegLen || Lk > kMaxSegLen)
    return fail(RA_ERR_SHAPE, "ra_dense_map: shards of at most %d tokens", kMaxSegLen);
  if (((uintptr_t)dense_bias & 3) != 0) return fail(RA_ERR_ALIGN, "dense_bias is not 4-byte aligned");
  if (stride_q < Lk || stride_b < 0 || stride_h < 0)
    return fail(RA_ERR_BIAS, "dense bias strides: stride_q must be at least Lk, stride_b / stride_h "
                             "non-negative (0 broadcasts)");
  const int nb = stride_b ? B : 1, nh = stride_h ? H : 1;
  if ((int64_t)nb * nh > 65535) return fail(RA_ERR_SHAPE, "ra_dense_map: more than 65535 (batch, head) blocks");
  hipError_t e = ra::launch_dense_map(dense_bias, stride_b, stride_h, stride_q, nb, nh, Lq, Lk, map,
                                      (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_dense_map launch");
}

int ra_fwd_step(const ra_fwd_step_params* p, void* stream) {
  int rc = ra_fwd_step_check(p);
  if (rc) return rc;
  if (ra_step_is_skippable(&p->bias, p->Lq, p->Lk)) return RA_OK;  // identity on the carry
  if (step_on_pair(p->bias, p->B, p->H, p->Lq, p->Lk, p->D, true)) return fwd_step_on_pair(*p, stream);
  const ra::FwdArgs a = to_fwd_args(*p);
  hipError_t e = ra::launch_fwd_step(a, p->D, kernel_mode(p->bias.flags), (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_fwd_step launch");
}

int ra_fwd_steps(const ra_fwd_step_params* steps, int32_t n_steps, void* stream) {
  if (n_steps < 0) return fail(RA_ERR_SHAPE, "n_steps is negative");
  return fwd_passes(steps, std::vector<int>{0, n_steps}, 1, stream);
}

int ra_fwd_passes(const ra_fwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes, void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  return rc ? rc : fwd_passes(steps, first, n_passes, stream);
}

int ra_fwd_finalize_passes(const float* o, const float* m, const float* l, void* out, int32_t out_dtype,
                           int64_t out_stride_pass, int64_t out_stride_b, int64_t out_stride_h,
                           int64_t out_stride_l, float* lse, int32_t n_passes, int32_t B, int32_t H, int32_t Lq,
                           int32_t D, void* stream) {
  if (!o || !m || !l || !out || !lse) return fail(RA_ERR_NULL, "ra_fwd_finalize: NULL pointer");
  if (n_passes <= 0 || n_passes > (1 << 16)) return fail(RA_ERR_SHAPE, "n_passes must lie in [1, 65536]");
  int rc = check_dims(B, H, Lq, 1, D);
  if (rc) return rc;
  if ((int64_t)n_passes * B * H > (1 << 20)) return fail(RA_ERR_SHAPE, "n_passes*B*H too large");
  if (out_dtype != RA_DTYPE_BF16 && out_dtype != RA_DTYPE_F32)
    return fail(RA_ERR_DTYPE, "unknown out_dtype %d", out_dtype);
  if ((out_stride_pass % 4) || (out_stride_b % 4) || (out_stride_h % 4) || (out_stride_l % 4))
    return fail(RA_ERR_ALIGN, "out strides must be multiples of 4 elements");
  // the kernel stores four elements at a time: 8 bytes of bf16 or 16 bytes of fp32
  if (reinterpret_cast<uintptr_t>(out) % (out_dtype == RA_DTYPE_F32 ? 16u : 8u))
    return fail(RA_ERR_ALIGN, "out must be aligned to four elements (%d bytes)", out_dtype == RA_DTYPE_F32 ? 16 : 8);
  if (!aligned16(o)) return fail(RA_ERR_ALIGN, "o is not 16-byte aligned");
  hipError_t e = ra::launch_fwd_finalize(o, m, l, out, out_dtype == RA_DTYPE_F32, out_stride_pass, out_stride_b,
                                         out_stride_h, out_stride_l, lse, n_passes, B, H, Lq, D,
                                         (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_fwd_finalize launch");
}

int ra_fwd_finalize(const float* o, const float* m, const float* l, void* out, int32_t out_dtype,
                    int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_l, float* lse,
                    int32_t B, int32_t H, int32_t Lq, int32_t D, void* stream) {
  return ra_fwd_finalize_passes(o, m, l, out, out_dtype, 0, out_stride_b, out_stride_h, out_stride_l, lse, 1, B, H,
                                Lq, D, stream);
}

int ra_bwd_delta_passes(const void* out, int32_t out_dtype, int64_t out_stride_pass, int64_t out_stride_b,
                        int64_t out_stride_h, int64_t out_stride_l, const ra_tensor* dout,
                        int64_t dout_stride_pass, float* delta, int32_t n_passes, int32_t B, int32_t H,
                        int32_t Lq, int32_t D, void* stream) {
  if (!out || !dout || !delta) return fail(RA_ERR_NULL, "ra_bwd_delta: NULL pointer");
  if (n_passes <= 0 || n_passes > (1 << 16)) return fail(RA_ERR_SHAPE, "n_passes must lie in [1, 65536]");
  int rc = check_dims(B, H, Lq, 1, D);
  if (rc) return rc;
  if ((int64_t)n_passes * B * H > (1 << 20)) return fail(RA_ERR_SHAPE, "n_passes*B*H too large");
  if ((rc = check_tensor("dout", *dout, D))) return rc;
  if (out_dtype != RA_DTYPE_BF16 && out_dtype != RA_DTYPE_F32)
    return fail(RA_ERR_DTYPE, "unknown out_dtype %d", out_dtype);
  if (!aligned16(out) || (out_stride_pass % 8) || (out_stride_b % 8) || (out_stride_h % 8) || (out_stride_l % 8) ||
      (dout_stride_pass % 8))
    return fail(RA_ERR_ALIGN, "out must be 16-byte aligned with strides that are multiples of 8");
  hipError_t e = ra::launch_bwd_delta(out, out_dtype == RA_DTYPE_F32, out_stride_pass, out_stride_b, out_stride_h,
                                      out_stride_l, to_arg(*dout), dout_stride_pass, delta, n_passes, B, H, Lq, D,
                                      (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_bwd_delta launch");
}

int ra_bwd_delta(const void* out, int32_t out_dtype, int64_t out_stride_b, int64_t out_stride_h,
                 int64_t out_stride_l, const ra_tensor* dout, float* delta, int32_t B, int32_t H,
                 int32_t Lq, int32_t D, void* stream) {
  return ra_bwd_delta_passes(out, out_dtype, 0, out_stride_b, out_stride_h, out_stride_l, dout, 0, delta, 1, B, H, Lq,
                             D, stream);
}

int ra_bwd_step(const ra_bwd_step_params* p, void* stream) { return ra_bwd_step_parts(p, 3, stream); }

int ra_bwd_step_parts(const ra_bwd_step_params* p, int32_t parts, void* stream) {
  int rc = ra_bwd_step_check(p);
  if (rc) return rc;
  if (parts < 1 || parts > 3) return fail(RA_ERR_SHAPE, "parts must be 1, 2 or 3 (got %d)", parts);
  if (dense_steps_on_pair(p->bias)) return bwd_step_on_pair(*p, parts, stream);
  if (ra_step_is_skippable(&p->bias, p->Lq, p->Lk)) return RA_OK;  // contributes nothing
  if ((parts & 2) && step_on_pair(p->bias, p->B, p->H, p->Lq, p->Lk, p->D, false)) {
    if ((rc = bwd_step_on_pair(*p, 2, stream))) return rc;
    if (!(parts &= 1)) return RA_OK;
  }
  const ra::BwdArgs a = to_bwd_args(*p);
  hipError_t e = ra::launch_bwd_step(a, p->D, kernel_mode(p->bias.flags), parts, (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_bwd_step launch");
}

int ra_bwd_dq_steps(const ra_bwd_step_params* steps, int32_t n_steps, void* stream) {
  if (n_steps < 0) return fail(RA_ERR_SHAPE, "n_steps is negative");
  return bwd_dq_passes(steps, std::vector<int>{0, n_steps}, 1, stream);
}

int ra_bwd_dkdv_steps(const ra_bwd_step_params* steps, int32_t n_steps, void* stream) {
  if (n_steps < 0) return fail(RA_ERR_SHAPE, "n_steps is negative");
  return bwd_dkdv_passes(steps, std::vector<int>{0, n_steps}, 1, stream);
}

int ra_bwd_dq_passes(const ra_bwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes,
                     void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  return rc ? rc : bwd_dq_passes(steps, first, n_passes, stream);
}

int ra_bwd_dkdv_passes(const ra_bwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes,
                       void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  return rc ? rc : bwd_dkdv_passes(steps, first, n_passes, stream);
}

// every pass of a whole-ring launch needs a head block to take its resident side from
static int check_whole(const std::vector<int>& first, int n_passes) {
  for (int p = 0; p < n_passes; ++p)
    if (first[p + 1] == first[p]) return fail(RA_ERR_SHAPE, "pass %d has no block", p);
  return RA_OK;
}

int ra_fwd_ring(const ra_fwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes, void* out,
                int32_t out_dtype, int64_t out_stride_pass, int64_t out_stride_b, int64_t out_stride_h,
                int64_t out_stride_l, float* lse, void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  if (rc || (rc = check_whole(first, n_passes))) return rc;
  if (!lse) return fail(RA_ERR_NULL, "ra_fwd_ring: lse is NULL");
  const RingResult r{out, nullptr, lse, out_dtype, out_stride_pass, out_stride_b, out_stride_h, out_stride_l};
  if ((rc = check_ring_result("ra_fwd_ring", r))) return rc;
  return fwd_passes(steps, first, n_passes, stream, &r);
}

int ra_bwd_dq_ring(const ra_bwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes, void* dq,
                   int64_t stride_pass, int64_t stride_b, int64_t stride_h, int64_t stride_l, void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  if (rc || (rc = check_whole(first, n_passes))) return rc;
  const RingResult r{dq, nullptr, nullptr, RA_DTYPE_BF16, stride_pass, stride_b, stride_h, stride_l};
  if ((rc = check_ring_result("ra_bwd_dq_ring", r))) return rc;
  return bwd_dq_passes(steps, first, n_passes, stream, &r);
}

int ra_bwd_dkdv_ring(const ra_bwd_step_params* steps, const int32_t* steps_per_pass, int32_t n_passes, void* dk,
                     void* dv, int64_t stride_pass, int64_t stride_b, int64_t stride_h, int64_t stride_l,
                     void* stream) {
  std::vector<int> first;
  int rc = check_pass_counts(steps_per_pass, n_passes, first);
  if (rc || (rc = check_whole(first, n_passes))) return rc;
  if (!dv) return fail(RA_ERR_NULL, "ra_bwd_dkdv_ring: dv is NULL");
  const RingResult r{dk, dv, nullptr, RA_DTYPE_BF16, stride_pass, stride_b, stride_h, stride_l};
  if ((rc = check_ring_result("ra_bwd_dkdv_ring", r))) return rc;
  return bwd_dkdv_passes(steps, first, n_passes, stream, &r);
}

static int convert_args(const ra_rows* items, int32_t n_items, ra::ConvertArgs& a) {
  if (n_items < 1 || n_items > ra::kMaxConvert) return fail(RA_ERR_SHAPE, "ra_convert: 1 to %d arrays (got %d)", ra::kMaxConvert, n_items);
  if (!items) return fail(RA_ERR_NULL, "ra_convert: items is NULL");
  memset(&a, 0, sizeof(a));
  for (int i = 0; i < n_items; ++i) {
    const ra_rows& r = items[i];
    if (!r.src || !r.dst) return fail(RA_ERR_NULL, "ra_convert: NULL pointer");
    if (r.B <= 0 || r.L <= 0 || r.H <= 0 || r.src_d <= 0 || r.dst_d <= 0)
      return fail(RA_ERR_SHAPE, "ra_convert: bad shape B=%d L=%d H=%d d=%d -> %d", r.B, r.L, r.H, r.src_d, r.dst_d);
    if (r.src_d > 128 || r.dst_d > 128) return fail(RA_ERR_HEAD_DIM, "ra_convert: head dims of at most 128");
    if (r.B > 65535 || (int64_t)r.H * 16 >= ((int64_t)1 << 31) || (int64_t)r.L * (r.H * 16) >= ((int64_t)1 << 31))
      return fail(RA_ERR_TOO_LARGE, "ra_convert: too many rows for one launch");
    for (int dt : {r.src_dtype, r.dst_dtype})
      if (dt != RA_DTYPE_BF16 && dt != RA_DTYPE_F32 && dt != RA_DTYPE_F16) return fail(RA_ERR_DTYPE, "unknown dtype %d", dt);
    // eight elements at a time where every chunk of a row starts on a multiple of 16 bytes
    auto on_chunks = [](const void* p, int dtype, int64_t sb, int64_t sl, int64_t sh) {
      const int64_t mask = dtype == RA_DTYPE_F32 ? 3 : 7;
      return aligned16(p) && !((sb | sl | sh) & mask);
    };
    if (reinterpret_cast<uintptr_t>(r.src) % (r.src_dtype == RA_DTYPE_F32 ? 4 : 2) ||
        reinterpret_cast<uintptr_t>(r.dst) % (r.dst_dtype == RA_DTYPE_F32 ? 4 : 2))
      return fail(RA_ERR_ALIGN, "ra_convert: arrays must be aligned to their elements");
    a.item[i] = ra::ConvertItem{r.src, r.dst, r.src_dtype, r.dst_dtype, r.src_d, r.dst_d, r.B, r.L, r.H,
                                on_chunks(r.src, r.src_dtype, r.src_stride_b, r.src_stride_l, r.src_stride_h),
                                on_chunks(r.dst, r.dst_dtype, r.dst_stride_b, r.dst_stride_l, r.dst_stride_h),
                                r.src_stride_b, r.src_stride_l, r.src_stride_h, r.dst_stride_b, r.dst_stride_l, r.dst_stride_h};
  }
  return RA_OK;
}

static int64_t bwd_pair_workspace(const ra_bwd_step_params* p, bool any_dim) {
  if (!p || check_dims(p->B, p->H, p->Lq, p->Lk, p->D, any_dim)) return 0;
  const BwdPlan plan = plan_bwd_pair(*p);
  return bwd_space(*p, plan.dq, plan.dkdv).total;
}

static int bwd_pair(const Before& before, const ra_bwd_step_params* p, bool any_dim, int grad_dtype, const void* out, int32_t out_dtype, int64_t out_stride_b,
                int64_t out_stride_h, int64_t out_stride_l, void* dq, int64_t dq_stride_b, int64_t dq_stride_h,
                int64_t dq_stride_l, void* dk, void* dv, int64_t dkv_stride_b, int64_t dkv_stride_h,
                int64_t dkv_stride_l, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!p) return fail(RA_ERR_NULL, "params is NULL");
  ra_bwd_step_params c = *p;
  c.delta = c.dq = c.dk = c.dv = reinterpret_cast<float*>(uintptr_t(16));  // not used: no accumulators
  int rc = check_bwd_step(&c, any_dim);
  if (rc || (rc = check_whole_call("ra_bwd_whole", c.D, c.bias))) return rc;
  const bool via_bf16 = grad_dtype & RA_DTYPE_VIA_BF16;
  grad_dtype &= ~RA_DTYPE_VIA_BF16;
  const RingResult rq{dq, nullptr, nullptr, grad_dtype, 0, dq_stride_b, dq_stride_h, dq_stride_l, via_bf16};
  const RingResult rk{dk, dv, nullptr, grad_dtype, 0, dkv_stride_b, dkv_stride_h, dkv_stride_l, via_bf16};
  if ((rc = check_ring_result("ra_bwd_pair", rq, true)) || (rc = check_ring_result("ra_bwd_pair", rk, true))) return rc;
  if (!dv) return fail(RA_ERR_NULL, "ra_bwd_pair: dv is NULL");
  const BwdPlan plan = plan_bwd_pair(*p);
  const PairPlan &plan_q = plan.dq, &plan_k = plan.dkdv;
  if (!plan_k.pair && narrow(c.D)) return fail(RA_ERR_TOO_LARGE, "ra_bwd_whole: too many rows");
  const BwdSpace sp = bwd_space(*p, plan_q, plan_k);
  if (!workspace || !aligned16(workspace)) return fail(RA_ERR_ALIGN, "ra_bwd_pair: the workspace must be 16-byte aligned");
  if (workspace_bytes < sp.total) return fail(RA_ERR_SHAPE, "ra_bwd_pair: the workspace is smaller than ra_bwd_pair_workspace()");
  if (!out || !aligned16(out) || (out_stride_b % 8) || (out_stride_h % 8) || (out_stride_l % 8))
    return fail(RA_ERR_ALIGN, "ra_bwd_pair: out must be 16-byte aligned with strides that are multiples of 8");
  if (out_dtype != RA_DTYPE_BF16 && out_dtype != RA_DTYPE_F32) return fail(RA_ERR_DTYPE, "unknown out_dtype %d", out_dtype);
  char* const ws = (char*)workspace;
  c.delta = (float*)(ws + sp.delta);
  ra::PairBwdArgs a;
  memset(&a, 0, sizeof(a));
  a.a = to_bwd_args(c);
  a.stat = (const float*)(ws + sp.stat);
  ra::StatArgs st;
  memset(&st, 0, sizeof(st));
  st.out = out;
  st.sb = out_stride_b;
  st.sh = out_stride_h;
  st.sl = out_stride_l;
  st.dout = c.dout.ptr;
  st.dsb = c.dout.stride_b;
  st.dsh = c.dout.stride_h;
  st.dsl = c.dout.stride_l;
  st.dout_d = c.D;
  st.dout_vec = 1;
  st.lse = c.lse;
  st.inv_res = 1.0f / a.a.scale_res;
  st.stat = (float*)(ws + sp.stat);
  st.delta = (float*)(ws + sp.delta);
  st.B = c.B;
  st.H = c.H;
  st.L = c.Lq;
  int dout_dtype = RA_DTYPE_BF16;
  // A conversion that makes dO, row after row, is left to the statistics, which read it anyway.
  ra::ConvertArgs conv;
  const bool made = before.n == 1 && before.items && before.items[0].dst == c.dout.ptr;
  if (made && (rc = convert_args(before.items, 1, conv))) return rc;
  const ra::ConvertItem& it = conv.item[0];
  if (made && it.dst_dtype == RA_DTYPE_BF16 && it.dst_d == c.D && it.B == c.B && it.L == c.Lq && it.H == c.H && it.dst_sh == c.D &&
      it.dst_sl == (int64_t)c.H * c.D && it.dst_sb == (int64_t)c.Lq * c.H * c.D && c.dout.stride_h == it.dst_sh && c.dout.stride_l == it.dst_sl &&
      c.dout.stride_b == it.dst_sb) {
    st.dout = it.src;
    st.dsb = it.src_sb;
    st.dsh = it.src_sh;
    st.dsl = it.src_sl;
    st.dout_d = it.src_d;
    st.dout_vec = it.src_vec;
    st.copy = (ra::bf16_t*)it.dst;
    dout_dtype = it.src_dtype;
  } else if ((rc = before.launch(stream))) {
    return rc;
  }
  hipError_t e = ra::launch_pair_stat(st, out_dtype == RA_DTYPE_F32, dout_dtype, c.D, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "ra_bwd_pair launch");
  const std::vector<int> one{0, 1};
  const int mode = kernel_mode(c.bias.flags);
  auto share = [&](const PairPlan& plan, int64_t part, int64_t n, const RingResult& r) {
    ra::PairBwdArgs x = a;
    x.n_split = plan.n_split;
    x.chunk_tiles = plan.chunk_tiles;
    x.group = plan.group;
    x.part = plan.n_split > 1 ? (float*)(ws + part) : nullptr;
    x.part_n = plan.n_split > 1 ? (int*)(ws + n) : nullptr;
    x.out = r.base;
    x.out2 = r.base2;
    x.out_dtype = r.dtype;
    x.via_bf16 = r.via_bf16;
    x.out_sb = r.stride_b;
    x.out_sh = r.stride_h;
    x.out_sl = r.stride_l;
    return x;
  };
  const ra::PairBwdArgs dkdv = share(plan_k, sp.dkdv_part, sp.dkdv_n, rk), dq_args = share(plan_q, sp.dq_part, sp.dq_n, rq);
  auto on_pair = [&](const ra::PairBwdArgs* kv, const ra::PairBwdArgs* q) -> int {
    hipError_t err = ra::launch_bwd_pair(kv, q, c.D, mode, (hipStream_t)stream);
    return err == hipSuccess ? RA_OK : hip_fail(err, "ra_bwd_pair launch");
  };
  if (plan.one_launch) return on_pair(&dkdv, &dq_args);
  // fp32 gradients that lie as the accumulators of a step do are stored by its kernels, which know one pair only and are faster
  // (dK and dV of a causal diagonal and a full pair of 4096, H=16, D=128: 430 us on the several-shard ones, 417 on
  // these; 32768 in two shards 5.21 | 5.15 ms and dQ 2.60 | 2.54)
  auto as_accumulator = [&](const RingResult& r, int L) {
    return r.dtype == RA_DTYPE_F32 && !r.via_bf16 && aligned16(r.base) && aligned16(r.base2) && r.stride_l == c.D && r.stride_h == (int64_t)L * c.D &&
           r.stride_b == (int64_t)c.H * L * c.D && mode != 2;
  };
  auto one_step = [&](int part) -> int {
    ra::BwdArgs s = a.a;
    s.dq = (float*)rq.base;
    s.dk = (float*)rk.base;
    s.dv = (float*)rk.base2;
    s.bias.flags |= ra::kFlagWholeF32;
    hipError_t err = ra::launch_bwd_step(s, c.D, mode, part, (hipStream_t)stream);
    return err == hipSuccess ? RA_OK : hip_fail(err, "ra_bwd_pair launch");
  };
  if ((rc = plan_k.pair ? on_pair(&dkdv, nullptr) : as_accumulator(rk, c.Lk) ? one_step(1) : bwd_dkdv_passes(&c, one, 1, stream, &rk)))
    return rc;
  return plan_q.pair ? on_pair(nullptr, &dq_args) : as_accumulator(rq, c.Lq) ? one_step(2) : bwd_dq_passes(&c, one, 1, stream, &rq);
}

int64_t ra_bwd_pair_workspace(const ra_bwd_step_params* p) { return bwd_pair_workspace(p, false); }
int64_t ra_bwd_whole_workspace(const ra_bwd_step_params* p) { return bwd_pair_workspace(p, true); }

int ra_bwd_pair(const ra_bwd_step_params* p, const void* out, int32_t out_dtype, int64_t out_stride_b,
                int64_t out_stride_h, int64_t out_stride_l, void* dq, int64_t dq_stride_b, int64_t dq_stride_h,
                int64_t dq_stride_l, void* dk, void* dv, int64_t dkv_stride_b, int64_t dkv_stride_h,
                int64_t dkv_stride_l, void* workspace, int64_t workspace_bytes, void* stream) {
  return bwd_pair({}, p, false, RA_DTYPE_BF16, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, dq, dq_stride_b, dq_stride_h, dq_stride_l, dk, dv, dkv_stride_b,
                  dkv_stride_h, dkv_stride_l, workspace, workspace_bytes, stream);
}
int ra_bwd_whole(const ra_bwd_step_params* p, const void* out, int32_t out_dtype, int64_t out_stride_b,
                int64_t out_stride_h, int64_t out_stride_l, int32_t grad_dtype, void* dq, int64_t dq_stride_b, int64_t dq_stride_h,
                int64_t dq_stride_l, void* dk, void* dv, int64_t dkv_stride_b, int64_t dkv_stride_h,
                int64_t dkv_stride_l, void* workspace, int64_t workspace_bytes, void* stream) {
  return bwd_pair({}, p, true, grad_dtype, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, dq, dq_stride_b, dq_stride_h, dq_stride_l, dk, dv, dkv_stride_b,
                  dkv_stride_h, dkv_stride_l, workspace, workspace_bytes, stream);
}

int ra_convert(const ra_rows* items, int32_t n_items, void* stream) {
  ra::ConvertArgs a;
  if (int rc = convert_args(items, n_items, a)) return rc;
  hipError_t e = ra::launch_convert(a, n_items, (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_convert launch");
}

int ra_fwd_call(const ra_rows* before, int32_t n_before, const ra_fwd_step_params* p, void* out, int32_t out_dtype, int64_t out_stride_b,
                int64_t out_stride_h, int64_t out_stride_l, float* lse, void* workspace, int64_t workspace_bytes, void* stream) {
  return fwd_pair({before, n_before}, p, true, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, lse, workspace, workspace_bytes, stream);
}

int ra_bwd_call(const ra_rows* before, int32_t n_before, const ra_bwd_step_params* p, const void* out, int32_t out_dtype,
                int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_l, int32_t grad_dtype, void* dq, int64_t dq_stride_b,
                int64_t dq_stride_h, int64_t dq_stride_l, void* dk, void* dv, int64_t dkv_stride_b, int64_t dkv_stride_h,
                int64_t dkv_stride_l, void* workspace, int64_t workspace_bytes, void* stream) {
  return bwd_pair({before, n_before}, p, true, grad_dtype, out, out_dtype, out_stride_b, out_stride_h, out_stride_l, dq, dq_stride_b, dq_stride_h,
                  dq_stride_l, dk, dv, dkv_stride_b, dkv_stride_h, dkv_stride_l, workspace, workspace_bytes, stream);
}

int ra_bwd_finalize_passes(const float* acc, void* out, int64_t out_stride_pass, int64_t out_stride_b,
                           int64_t out_stride_h, int64_t out_stride_l, int32_t n_passes, int32_t B, int32_t H,
                           int32_t L, int32_t D, void* stream) {
  if (!acc || !out) return fail(RA_ERR_NULL, "ra_bwd_finalize: NULL pointer");
  if (n_passes <= 0 || n_passes > (1 << 16)) return fail(RA_ERR_SHAPE, "n_passes must lie in [1, 65536]");
  int rc = check_dims(B, H, L, 1, D);
  if (rc) return rc;
  if ((int64_t)n_passes * B * H > (1 << 20)) return fail(RA_ERR_SHAPE, "n_passes*B*H too large");
  if ((out_stride_pass % 4) || (out_stride_b % 4) || (out_stride_h % 4) || (out_stride_l % 4))
    return fail(RA_ERR_ALIGN, "out strides must be multiples of 4 elements");
  // the kernel loads 16 bytes of fp32 and stores 8 bytes of bf16 at a time
  if (reinterpret_cast<uintptr_t>(out) % 8u) return fail(RA_ERR_ALIGN, "out must be 8-byte aligned");
  if (!aligned16(acc)) return fail(RA_ERR_ALIGN, "acc is not 16-byte aligned");
  hipError_t e = ra::launch_bwd_finalize(acc, out, out_stride_pass, out_stride_b, out_stride_h, out_stride_l,
                                         n_passes, B, H, L, D, (hipStream_t)stream);
  return e == hipSuccess ? RA_OK : hip_fail(e, "ra_bwd_finalize launch");
}

int ra_bwd_finalize(const float* acc, void* out, int64_t out_stride_b, int64_t out_stride_h,
                    int64_t out_stride_l, int32_t B, int32_t H, int32_t L, int32_t D, void* stream) {
  return ra_bwd_finalize_passes(acc, out, 0, out_stride_b, out_stride_h, out_stride_l, 1, B, H, L, D, stream);
}

}  // extern "C"
