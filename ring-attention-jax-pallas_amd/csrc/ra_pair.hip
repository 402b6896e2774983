// Kernels for one (query sequence, key sequence) pair that is short, irregular or too small to fill
// the chip with the long-sequence kernels of ra_fwd.hip / ra_bwd.hip.
//
// Those hold 256 query rows per workgroup, one workgroup per compute unit, and hide everything but
// the matrix instructions inside hand-ordered straight-line stretches; every tile outside a stretch
// (masked by element, first, last) costs them 2 to 3 times as much, and a grid below 256 workgroups
// leaves compute units idle.  The kernels here take 128 rows per workgroup (4 waves x 32), need half
// of a compute unit's registers and LDS - two independent workgroups per compute unit, one's vector
// work under the other's matrix work - and treat every tile alike, masks included.  The streamed
// side of a pair can be split over several workgroups whose partial results a second kernel
// combines.
#include <type_traits>

#include "ra_launch.h"

namespace ra {

constexpr int kPairThreads = 256;
constexpr int kPairRows = 128;  // query rows per workgroup
constexpr int kPairKeys = 64;   // keys per LDS tile
constexpr int kPairListTiles = 1024;

// what a listed tile must evaluate element by element (bits of a list entry, above the tile index)
constexpr int kTestShift = 10;
constexpr int kTestSegment = 1, kTestPrefix = 2, kTestDense = 4;

// Rows and keys of a workgroup's rectangle as the prefix term sees them: 0 = untouched by the mask,
// 1 = some score may be masked, 2 = every score is.
RA_DEV int prefix_class(int qlo, int qhi, int klo, int khi, bool q_any, bool q_all, bool k_any, bool k_all) {
  if (khi <= qlo || (q_all && k_all)) return 0;
  return (klo > qhi && !(q_any && k_any)) ? 2 : 1;
}

// Flat workgroup id -> (batch * head, piece, tile).  Workgroups are handed to the 8 XCDs round-robin:
// where the heads divide by eight, all of a head's workgroups run on one XCD and share its L2.
// Tiles in descending order over all heads: under a causal mask the longest ones start first.  The
// pieces go last: the workgroups of an XCD are dealt to its shader engines in turn, so that a
// pattern of working and empty workgroups of a small even period would leave some of them idle
// (B=1, H=8, window 1024 of 16384 tokens, 4 pieces of which 3 are empty: 270 us with the pieces
// next to each other, 99 without the empty ones).
RA_DEV void pair_decode(int bid, int BH, int ntile, int& hh, int& piece, int& tile) {
  const bool spread = (BH & 7) == 0;
  const int slot = spread ? bid >> 3 : bid, heads = spread ? BH >> 3 : BH;
  const int t = slot / heads, hl = slot % heads;
  piece = t / ntile;
  tile = ntile - 1 - t % ntile;
  hh = spread ? hl * 8 + (bid & 7) : hl;
}

// S^T orientation as in fwd_step_kernel: a lane owns one query row and 16 keys of a 32-key block.
// D is the row pitch of the LDS tiles (64 or 128 elements).
template <int D, int MODE>
__global__ __launch_bounds__(kPairThreads, 2) void fwd_pair_kernel(const PairFwdArgs a) {
  constexpr bool GENERAL = MODE != 0;
  constexpr bool DENSE = MODE == 2;
  constexpr int KS = D / 16, DB = D / 32;
  constexpr int ROWB = D * 2;
  constexpr int TILE_BYTES = kPairKeys * ROWB;
  __shared__ __attribute__((aligned(16))) char s_k[2][TILE_BYTES];
  __shared__ __attribute__((aligned(16))) char s_v[2][TILE_BYTES];
  __shared__ __attribute__((aligned(16))) int s_seg[GENERAL ? 2 : 1][kPairKeys];
  __shared__ __attribute__((aligned(16))) int s_pre[GENERAL ? 2 : 1][kPairKeys];
  __shared__ unsigned short s_list[GENERAL ? kPairListTiles : 1];
  __shared__ unsigned char s_flag[GENERAL ? kPairListTiles : 1];
  __shared__ int s_red[20];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int nqt = (a.Lq + kPairRows - 1) / kPairRows;
  int hh, split, qt;
  pair_decode(blockIdx.x, a.B * a.H, nqt, hh, split, qt);
  const int b = hh / a.H, h = hh % a.H;
  const int q0 = qt * kPairRows;
  const int qw = q0 + wave * 32;
  const int qi = qw + l32;
  const bool q_valid = qi < a.Lq;
  const int qi_c = min(qi, a.Lq - 1);
  const BiasArgs& bs = a.bias;
  const int flags = bs.flags;
  const int q_off = bs.q_off, kv_off = bs.kv_off;

  // ---- the key tiles of this workgroup ----------------------------------------------------------
  const int ntiles = (a.Lk + kPairKeys - 1) / kPairKeys;
  const int q_hi = min(q0 + kPairRows, a.Lq) - 1;
  int j_lo, j_hi;
  key_tile_range(flags, bs.window, q_off + q0, q_off + q_hi, kv_off, ntiles, kPairKeys, j_lo, j_hi);
  int n = j_hi - j_lo;
  // A row's tiles are shared by as many workgroups as there are pieces of chunk_tiles in them; this
  // one takes piece `split`.
  if (split > 0 && split * a.chunk_tiles >= n) return;

  bf16x8 qf[KS];
  {
    const bf16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh + (long long)qi_c * a.q.sl + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *(const bf16x8*)(qp + 16 * s);
  }
  int q_seg = 0, q_pre = 0;
  float slope2 = 0.f;
  const int* kv_seg = nullptr;
  const int* kv_pre = nullptr;
  if constexpr (GENERAL) {
    if (flags & RA_BIAS_SEGMENT) {
      q_seg = bs.q_seg[b * bs.q_seg_sb + qi_c];
      kv_seg = bs.kv_seg + b * bs.kv_seg_sb;
    }
    if (flags & RA_BIAS_PREFIX) {
      q_pre = bs.q_pre[b * bs.q_pre_sb + qi_c];
      kv_pre = bs.kv_pre + b * bs.kv_pre_sb;
    }
    if (flags & RA_BIAS_ALIBI) slope2 = bs.slopes[h] * kLog2e / a.scale2;
  }

  bool use_list = false;
  const unsigned char* dmap = nullptr;
  if constexpr (DENSE) {
    if (bs.dense_map) dmap = dense_map_of(bs, b, h, a.H, a.Lq, a.Lk);
  }
  if constexpr (GENERAL) {
    // tiles that one or the other term rules out are dropped, the others carry the terms that they
    // have to be tested for
    const bool seg_on = flags & RA_BIAS_SEGMENT, pre_on = flags & RA_BIAS_PREFIX;
    use_list = ntiles <= kPairListTiles && (seg_on || pre_on || dmap != nullptr);
    if (use_list) {
      const int smin = wave_min(q_valid ? q_seg : 0x7fffffff), smax = wave_max(q_valid ? q_seg : (int)0x80000000);
      const int any = __any(q_valid && q_pre != 0), all = __all(!q_valid || q_pre != 0);
      if (lane == 0) {
        s_red[wave] = smin;
        s_red[4 + wave] = smax;
        s_red[8 + wave] = any;
        s_red[12 + wave] = all;
      }
      __syncthreads();
      const int qmin = min(min(s_red[0], s_red[1]), min(s_red[2], s_red[3]));
      const int qmax = max(max(s_red[4], s_red[5]), max(s_red[6], s_red[7]));
      const bool q_any = s_red[8] | s_red[9] | s_red[10] | s_red[11], q_all = s_red[12] & s_red[13] & s_red[14] & s_red[15];
      for (int j = j_lo + tid; j < j_hi; j += kPairThreads) {
        int f = 0x80;  // listed
        if (seg_on) {
          int kmin, kmax;
          tile_id_range<kPairKeys>(kv_seg, j, a.Lk, kmin, kmax);
          if (kmax < qmin || kmin > qmax) f = 0;
          else if (kmin != kmax || qmin != qmax) f |= kTestSegment;
        }
        if (pre_on && f) {
          const int klo = kv_off + j * kPairKeys, khi = kv_off + min((j + 1) * kPairKeys, a.Lk) - 1;
          if (khi > q_off + q0) {
            bool k_any, k_all;
            tile_flag_range<kPairKeys>(kv_pre, j, a.Lk, k_any, k_all);
            const int c = prefix_class(q_off + q0, q_off + q_hi, klo, khi, q_any, q_all, k_any, k_all);
            if (c == 2) f = 0;
            else if (c == 1) f |= kTestPrefix;
          }
        }
        if constexpr (DENSE) {
          if (dmap != nullptr && f) {
            const int bits = dense_map_or(dmap, a.Lk, q0, q_hi, j * kPairKeys, min((j + 1) * kPairKeys, a.Lk) - 1);
            if (!(bits & kMapLive)) f = 0;
            else if (bits & kMapNonZero) f |= kTestDense;
          }
        }
        s_flag[j - j_lo] = (unsigned char)f;
      }
      __syncthreads();
      if (wave == 0) {
        int cnt = 0;
        for (int base = 0; base < n; base += 64) {
          const int i = base + lane;
          const int f = (i < n) ? s_flag[i] : 0;
          const unsigned long long mask = __ballot(f != 0);
          if (f) s_list[cnt + __popcll(mask & ((1ull << lane) - 1ull))] = (unsigned short)((j_lo + i) | ((f & 7) << kTestShift));
          cnt += __popcll(mask);
        }
        if (lane == 0) s_red[16] = cnt;
      }
      __syncthreads();
      n = s_red[16];
    }
  }
  n = __builtin_amdgcn_readfirstlane(n);
  j_lo = __builtin_amdgcn_readfirstlane(j_lo);
  const int n_piece = max(1, min(a.n_split, (n + a.chunk_tiles - 1) / a.chunk_tiles));
  if (split >= n_piece) return;
  const int i_lo = n * split / n_piece, i_hi = n * (split + 1) / n_piece;

  // terms that a tile must be tested for if there is no list to say so
  int every_test = 0;
  if constexpr (GENERAL) {
    if (!use_list) {
      if (flags & RA_BIAS_PREFIX) every_test |= kTestPrefix;
    }
    if ((flags & RA_BIAS_DENSE) && dmap == nullptr) every_test |= kTestDense;
  }
  auto tile_at = [&](int i, int& tests) -> int {
    if (GENERAL && use_list) {
      const int e = __builtin_amdgcn_readfirstlane((int)s_list[i]);
      tests = (e >> kTestShift) | every_test;
      return e & ((1 << kTestShift) - 1);
    }
    tests = every_test;
    return j_lo + i;
  };

  // ---- global -> LDS: a wave moves 16 of a tile's 64 rows, 1 KiB per instruction -----------------
  constexpr int CPR = D / 8;         // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;      // rows per load instruction
  constexpr int NLD = 16 / RPI;      // load instructions per wave and tile
  const bf16_t* kbase = a.k.ptr + b * a.k.sb + h * a.k.sh;
  const bf16_t* vbase = a.v.ptr + b * a.v.sb + h * a.v.sh;
  // Complete tiles go through a wave-uniform base and per-lane byte offsets from the wave's first row.
  unsigned k_voff[NLD], v_voff[NLD];
#pragma unroll
  for (int t = 0; t < NLD; ++t) {
    const int row = lane / CPR + RPI * t;
    const int lc = (tile_off<D>(row, lane % CPR) - row * ROWB) >> 4;  // logical chunk stored at this lane's place
    k_voff[t] = (unsigned)(((long long)row * a.k.sl + lc * 8) * 2);
    v_voff[t] = (unsigned)(((long long)row * a.v.sl + lc * 8) * 2);
  }
  auto issue = [&](const bf16_t* base, const unsigned (&voff)[NLD], long long sl, int k0, unsigned dst) {
    if (k0 + kPairKeys <= a.Lk) {
      const bf16_t* sb = base + (long long)(k0 + 16 * wave) * sl;
#pragma unroll
      for (int t = 0; t < NLD; ++t) global_to_lds16_s(sb, voff[t], dst + (16 * wave + RPI * t) * ROWB);
    } else {  // last, partial tile: rows past the end repeat the last row (masked later)
#pragma unroll
      for (int t = 0; t < NLD; ++t) {
        const int row = 16 * wave + RPI * t + lane / CPR;
        const int lc = (tile_off<D>(row, lane % CPR) - row * ROWB) >> 4;
        global_to_lds16(base + (long long)min(k0 + row, a.Lk - 1) * sl + lc * 8, dst + (16 * wave + RPI * t) * ROWB);
      }
    }
  };
  auto issue_tile = [&](int j, int buf) {
    const int k0 = j * kPairKeys;
    issue(kbase, k_voff, a.k.sl, k0, RA_LDS_ADDR(&s_k[0][0]) + buf * TILE_BYTES);
    issue(vbase, v_voff, a.v.sl, k0, RA_LDS_ADDR(&s_v[0][0]) + buf * TILE_BYTES);
    if constexpr (GENERAL) {
      const int kk = min(k0 + lane, a.Lk - 1);
      if (kv_seg && wave == 0) global_to_lds4(kv_seg + kk, RA_LDS_ADDR(&s_seg[0][0]) + buf * (kPairKeys * 4));
      if (kv_pre && wave == 1) global_to_lds4(kv_pre + kk, RA_LDS_ADDR(&s_pre[0][0]) + buf * (kPairKeys * 4));
    }
  };

  float m_run = RA_NEG_INF;  // exponent reference (log2 domain), moves lazily
  float m_true = RA_NEG_INF;
  float l_run = 0.f, lr_run = 0.f;  // row sums of the fp32 and of the rounded probabilities (see fwd_step_kernel)
  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
  bf16x2 ones2;
  ones2[0] = (bf16_t)1.0f;
  ones2[1] = (bf16_t)1.0f;

  int koff[KS];
#pragma unroll
  for (int ss = 0; ss < KS; ++ss) koff[ss] = tile_off<D>(l32, 2 * ss + g);
  int voff[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const int j = lane & 15;
      const int vrow = 4 * g + (j >> 2) + 8 * h2;
      const int vcol = 32 * db + 16 * ((lane >> 4) & 1) + 4 * (j & 3);
      voff[db][h2] = tile_off<D>(vrow, vcol >> 3) + ((vcol & 4) << 1);
    }

  const bool wave_on = qw < a.Lq;
  const bool alibi_on = GENERAL && (flags & RA_BIAS_ALIBI);
  const int qlo_w = q_off + qw, qhi_w = q_off + qw + 31;

  auto step = [&](auto buffer, int i) {
    constexpr int BUF = decltype(buffer)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's share of tile i is in LDS
    __syncthreads();                     // everyone's is, and nobody reads the other buffer any more
    int tests;
    const int kt0 = tile_at(i, tests) * kPairKeys;
    if (i + 1 < i_hi) {
      int t1;
      issue_tile(tile_at(i + 1, t1), BUF ^ 1);
    }
    if (!wave_on) return;
    const int klo = kv_off + kt0, khi = klo + kPairKeys - 1;
    const int cls = classify_pos(flags, bs.window, qlo_w, qhi_w, klo, khi);
    if (cls & 1) return;
    f32x16 S[2];
    bool alibi_left = alibi_on;  // ALiBi still to be added element by element
#pragma unroll
    for (int r = 0; r < 16; ++r) S[0][r] = S[1][r] = 0.f;
    if (alibi_on && (khi <= qlo_w || klo >= qhi_w)) {
      // one side of the diagonal: -slope |q - k| is linear in both positions and enters through the
      // matrix unit as the accumulators' initial value, split into bf16 words (see fwd_step_kernel)
      alibi_left = false;
      const float s = khi <= qlo_w ? slope2 : -slope2;
      const float c = -s * (float)(q_off + qi - klo);
      bf16x8 bq;
      bq[0] = (bf16_t)s;
      bq[1] = (bf16_t)(s - (float)bq[0]);
      bq[2] = (bf16_t)c;
      bq[3] = (bf16_t)(c - (float)bq[2]);
      bq[4] = (bf16_t)((c - (float)bq[2]) - (float)bq[3]);
      bq[5] = bq[6] = bq[7] = (bf16_t)0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        bf16x8 rf;
#pragma unroll
        for (int e = 0; e < 8; ++e) rf[e] = (bf16_t)0.f;
        rf[0] = rf[1] = (bf16_t)(g == 0 ? (float)(32 * kb + l32) : 0.f);
        rf[2] = rf[3] = rf[4] = (bf16_t)(g == 0 ? 1.0f : 0.f);
        S[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rf, bq, S[kb], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ss = 0; ss < KS; ++ss)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        S[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(s_k[BUF] + 32 * kb * ROWB + koff[ss]), qf[ss], S[kb], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    if ((cls & 2) || kt0 + kPairKeys > a.Lk || (GENERAL && (tests || alibi_left))) {
      TileBias tb;
      tb.flags = (cls & 2) ? (flags & (RA_BIAS_CAUSAL | RA_BIAS_WINDOW)) : 0;
      if constexpr (GENERAL) {
        if (tests & kTestSegment) tb.flags |= RA_BIAS_SEGMENT;
        if (tests & kTestPrefix) tb.flags |= RA_BIAS_PREFIX;
        if (tests & kTestDense) tb.flags |= RA_BIAS_DENSE;
        if (alibi_left) tb.flags |= RA_BIAS_ALIBI;
      }
      tb.window = bs.window;
      tb.slope2 = slope2;
      tb.dense_mul = kLog2e / a.scale2;
      tb.dense = nullptr;
      tb.dense_vs = 1;
      tb.dense_vec = 0;
      const float* head = nullptr;
      if (DENSE) {
        head = bs.dense + b * bs.dense_sb + h * bs.dense_sh;
        tb.dense_vec = kt0 + kPairKeys <= a.Lk && ((((uintptr_t)head) | ((uintptr_t)bs.dense_sq << 2)) & 15) == 0;
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int var0 = kt0 + 32 * kb + 4 * g;
        tb.var_limit = a.Lk - var0;
        if (DENSE) tb.dense = head + (long long)qi_c * bs.dense_sq + var0;
        apply_bias<true, DENSE, GENERAL>(S[kb], tb, (q_off + qi) - (kv_off + var0), q_seg, q_pre,
                                         &s_seg[GENERAL ? BUF : 0][32 * kb + 4 * g], &s_pre[GENERAL ? BUF : 0][32 * kb + 4 * g]);
      }
    }
    float mx0 = RA_NEG_INF, mx1 = RA_NEG_INF;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      mx0 = fmaxf(fmaxf(mx0, S[0][r]), S[0][r + 1]);
      mx1 = fmaxf(fmaxf(mx1, S[1][r]), S[1][r + 1]);
    }
    const float mx = half_max(fmaxf(mx0, mx1)) * a.scale2;
    m_true = fmaxf(m_true, mx);
    if (__any(mx > m_run + 8.0f)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = fast_exp2(m_run - ((m_new == RA_NEG_INF) ? 0.f : m_new));
      m_run = m_new;
      l_run *= corr;
      lr_run *= corr;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= corr;
    }
    const float neg_m = (m_run == RA_NEG_INF) ? 0.f : -m_run;
    // The 32 scores of a lane go through exp2 in four groups of eight, one group per 16 keys of the
    // output product: group ks + 1 is worked on while the matrix unit multiplies with group ks.
    bf16x8 pf[4];
    float rs0 = 0.f, rs1 = 0.f;
    auto soft = [&](int ks, int e) {  // elements e, e + 1 of group ks
      const int r = 8 * (ks & 1) + e;
      const float p0 = fast_exp2(fmaf(S[ks >> 1][r], a.scale2, neg_m));
      const float p1 = fast_exp2(fmaf(S[ks >> 1][r + 1], a.scale2, neg_m));
      rs0 += p0;
      rs1 += p1;
      bf16x2 pr;
      pr[0] = (bf16_t)p0;
      pr[1] = (bf16_t)p1;
      unsigned pw = __builtin_bit_cast(unsigned, pr);
      asm volatile("" : "+v"(pw), "+v"(rs0), "+v"(rs1));
      pr = __builtin_bit_cast(bf16x2, pw);
      pf[ks][e] = pr[0];
      pf[ks][e + 1] = pr[1];
    };
    auto v_frag = [&](int op) {
      const int ks = op / DB, db = op % DB;
      const lds_char* p0 = (const lds_char*)(s_v[BUF] + 16 * ks * ROWB + voff[db][0]);
      const lds_char* p1 = (const lds_char*)(s_v[BUF] + 16 * ks * ROWB + voff[db][1]);
      const bf16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p0);
      const bf16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p1);
      return __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    constexpr int PF = 3;  // V fragments fetched ahead of the matrix instruction that uses them
    bf16x8 fr[4 * DB];
#pragma unroll
    for (int op = 0; op < PF; ++op) fr[op] = v_frag(op);
#pragma unroll
    for (int e = 0; e < 8; e += 2) soft(0, e);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int op = 0; op < 4 * DB; ++op) {
      const int ks = op / DB, db = op % DB;
      if (op + PF < 4 * DB) fr[op + PF] = v_frag(op + PF);
      oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], pf[ks], oacc[db], 0, 0, 0);
      if (ks < 3) {
#pragma unroll
        for (int e = 0; e < 8 / DB; e += 2) soft(ks + 1, db * (8 / DB) + e);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += rs0 + rs1;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        bf16x2 pr;
        pr[0] = pf[ks][e];
        pr[1] = pf[ks][e + 1];
        lr_run = __builtin_amdgcn_fdot2_f32_bf16(pr, ones2, lr_run, false);
      }
  };

  if (i_lo < i_hi) {
    int t0;
    issue_tile(tile_at(i_lo, t0), 0);
    for (int i = i_lo; i < i_hi; i += 2) {
      step(std::integral_constant<int, 0>{}, i);
      if (i + 1 < i_hi) step(std::integral_constant<int, 1>{}, i + 1);
    }
  }

  const float l_step = half_sum(l_run), lr_step = half_sum(lr_run);
  if (a.part_n != nullptr && split == 0 && tid == 0) a.part_n[hh * nqt + qt] = n_piece;
  if (!q_valid) return;
  const long long row = (long long)hh * a.Lq + qi;
  if (n_piece > 1) {
    // a share of the row's keys: combined by pair_combine_kernel
    const long long prow = (long long)split * ((long long)a.B * a.H * a.Lq) + row;
    float* op = a.part_o + prow * D + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        f32x4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = oacc[db][4 * bb + c];
        *(f32x4*)(op + 32 * db + 8 * bb) = t;
      }
    if (g == 0) *(f32x4*)(a.part_s + 4 * prow) = (f32x4){m_run, l_step, lr_step, 0.f};
  } else if (a.o != nullptr) {
    // merge into the carry (see fwd_step_kernel)
    const float m_in = a.m[row] * kLog2e, l_in = a.l[row];
    const float m_out = fmaxf(m_true, m_in), m_safe = (m_out == RA_NEG_INF) ? 0.f : m_out;
    const float f_in = fast_exp2(m_in - m_safe);
    const float f_step = (l_step > 0.f) ? fast_exp2(m_run - m_safe) : 0.f;
    const float f_o = f_step * ((lr_step > 0.f) ? l_step / lr_step : 1.f);
    float* op = a.o + row * D + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        f32x4 t = *(const f32x4*)(op + 32 * db + 8 * bb);
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = t[c] * f_in + oacc[db][4 * bb + c] * f_o;
        *(f32x4*)(op + 32 * db + 8 * bb) = t;
      }
    if (g == 0) {
      a.m[row] = m_out * kLn2;
      a.l[row] = l_in * f_in + l_step * f_step;
    }
  } else {
    const float inv = 1.0f / lr_step;
    const long long at = b * a.out_sb + h * a.out_sh + (long long)qi * a.out_sl + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        f32x4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = oacc[db][4 * bb + c] * inv;
        store4(a.out, a.out_f32, at + 32 * db + 8 * bb, t);
      }
    if (g == 0) a.lse[row] = (l_step > 0.f) ? (m_run + __log2f(l_step)) * kLn2 : RA_NEG_INF;
  }
}

// out and lse of rows whose keys were split: sum of the shares, each taken from its own exponent
// reference to the common one.  HBM bound: a share is D + 4 fp32 words per row.
template <int D>
__global__ __launch_bounds__(256) void pair_combine_kernel(const PairFwdArgs a) {
  constexpr int CPR = D / 4;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long rows = (long long)a.B * a.H * a.Lq;
  const long long row = i / CPR;
  if (row >= rows) return;
  const int c = (int)(i % CPR);
  const int li = (int)(row % a.Lq);
  const long long hh = row / a.Lq;
  const int n_piece = a.part_n[hh * ((a.Lq + kPairRows - 1) / kPairRows) + li / kPairRows];
  if (n_piece <= 1) return;  // written by its only workgroup
  float m = RA_NEG_INF;
  for (int s = 0; s < n_piece; ++s) m = fmaxf(m, a.part_s[4 * (s * rows + row)]);
  const float m_safe = (m == RA_NEG_INF) ? 0.f : m;
  float l = 0.f, lr = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < n_piece; ++s) {
    const f32x4 st = *(const f32x4*)(a.part_s + 4 * (s * rows + row));
    const f32x4 x = *(const f32x4*)(a.part_o + (s * rows + row) * D + 4 * c);
    const float w = fast_exp2(st[0] - m_safe);
    l += w * st[1];
    lr += w * st[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += w * x[e];
  }
  const float inv = 1.0f / lr;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] *= inv;
  store4(a.out, a.out_f32, (hh / a.H) * a.out_sb + (hh % a.H) * a.out_sh + (long long)li * a.out_sl + 4 * c, o);
  if (c == 0) a.lse[row] = (l > 0.f) ? (m + __log2f(l)) * kLn2 : RA_NEG_INF;
}

template <int D>
static hipError_t launch_fwd_pair_d(const PairFwdArgs& a, int mode, hipStream_t stream) {
  const int nqt = (a.Lq + kPairRows - 1) / kPairRows;
  dim3 grid((unsigned)(a.B * a.H * a.n_split * nqt)), block(kPairThreads);
  if (mode == 2) hipLaunchKernelGGL((fwd_pair_kernel<D, 2>), grid, block, 0, stream, a);
  else if (mode == 1) hipLaunchKernelGGL((fwd_pair_kernel<D, 1>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((fwd_pair_kernel<D, 0>), grid, block, 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.part_o == nullptr) return e;
  const long long n = (long long)a.B * a.H * a.Lq * (D / 4);
  hipLaunchKernelGGL((pair_combine_kernel<D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_fwd_pair(const PairFwdArgs& a, int D, int mode, hipStream_t stream) {
  return D == 128 ? launch_fwd_pair_d<128>(a, mode, stream) : launch_fwd_pair_d<64>(a, mode, stream);
}

}  // namespace ra
