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
//
// What bounds them is the latency of a wave's step through a tile, with two to four waves per SIMD to cover it: of
// the wave cycles of documents + ALiBi (D = 128) 37 to 41 % issue an instruction, 28 to 30 % wait at the barrier or for operands and 29
// to 34 % for the issue port, and a forward tile takes 7.2 vector and 2.8 scalar instructions per matrix instruction (9 and
// 3.6 before what follows) where the softmax needs 6.  Hence everything around the matrix instructions is kept short: what a wave does with
// a tile follows from a few ranges of tile indexes (WaveTiles) and from the wave's own ids (wave_tests), not the
// workgroup's; the terms of a masked block are passes of their own (apply_terms); a tile's loads share one base
// (TileLoader); and nothing that can be computed again stays in a register (opaque_lane, kernel_args), so that no
// variant spills a vector register or goes to scratch.  (Scalar registers in vector lanes: 2 to 24 in the general variants, 20 to 98 in
// those with a dense block.)  Before | after, us: documents of 2048 + ALiBi, 32768, H=16, D=128: forward 1787 | 1590, dQ 1916 | 1755, dK/dV
// 2770 | 2410; causal documents of 2175 in 48128, B=2, H=4, D=64: 443 | 325, 476 | 350, 495 | 427; prefix-LM 4096, B=2, H=16, D=128,
// forward 229 | 194; steps on dense blocks (documents of 2048 in 32768, 4 shards) 10.2 ms | 7.8 a pass.
#include <algorithm>
#include <type_traits>

#include "ra_launch.h"

namespace ra {

constexpr int kPairThreads = 256;
constexpr int kPairRows = 128;  // query rows per workgroup
constexpr int kPairKeys = 64;   // keys per LDS tile
constexpr int kPairListTiles = 1024;

// what a listed tile must evaluate element by element (bits of a list entry, above the tile index)
constexpr int kTestShift = 11;
constexpr int kTestSegment = 1, kTestPrefix = 2, kTestDense = 4;
constexpr int kTestPos = 8, kTestAlibi = 16, kTestDead = 32;  // (not in a list: from the wave's own rows)
// ... and under a dense block what its summary says about the tile, two bits (kMapLive, kMapNonZero) per wave and block of
// 32 x 32 scores, above them
constexpr int kCellShift = 16;
template <bool DENSE>
using ListEntry = std::conditional_t<DENSE, unsigned, unsigned short>;

// Rows and keys of a workgroup's rectangle as the prefix term sees them: 0 = untouched by the mask,
// 1 = some score may be masked, 2 = every score is.
RA_DEV int prefix_class(int qlo, int qhi, int klo, int khi, bool q_any, bool q_all, bool k_any, bool k_all) {
  if (khi <= qlo || (q_all && k_all)) return 0;
  return (klo > qhi && !(q_any && k_any)) ? 2 : 1;
}

// Flat workgroup id -> (batch * head, piece, tile).  Workgroups are handed to the 8 XCDs round-robin:
// where the heads divide by eight, all of a head's workgroups run on one XCD and share its L2.
// An XCD takes its heads in groups, the tiles of a group in descending order over all its heads: under a causal mask the longest ones
// start first.  Rows of even length need no order, and there a group is one head: as many workgroups as possible then read the same
// keys at the same time (128 heads of 12709 x 21941, D=96, forward 21.3 ms over all sixteen heads of an XCD, 15.7 one by one).  Else a group is four heads of an XCD (32 heads where they
// do not divide by eight): over all sixteen | four by four, 128 heads of 16384 causal, D=96, forward 9.1 | 7.3 ms, dQ 10.3 | 8.5, dK/dV
// 13.0 | 11.6; of 8192, D=64, a pass 5.86 | 5.61.  The
// pieces go last: the workgroups of an XCD are dealt to its shader engines in turn, so that a
// pattern of working and empty workgroups of a small even period would leave some of them idle
// (B=1, H=8, window 1024 of 16384 tokens, 4 pieces of which 3 are empty: 270 us with the pieces
// next to each other, 99 without the empty ones).
RA_DEV void pair_decode(int bid, int BH, int ntile, int pieces, int group, int& hh, int& piece, int& tile) {
  const bool spread = (BH & 7) == 0;
  const int slot = spread ? bid >> 3 : bid, heads = spread ? BH >> 3 : BH;
  const int size = min(spread || group == 1 ? group : 8 * group, heads), of_group = size * pieces * ntile, first = slot / of_group;
  const int here = min(size, heads - first * size), r = slot - first * of_group;
  const int t = r / here, hl = first * size + r % here;
  piece = t / ntile;
  tile = ntile - 1 - t % ntile;
  hh = spread ? hl * 8 + (bid & 7) : hl;
}

// The lane number, not known to the compiler as such: what is computed from it inside a loop is computed
// there, where it is needed, instead of sitting in a register (or in scratch: a reload waits for the tile
// loads in flight) through the loop.
RA_DEV int opaque_lane(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// Moves ROWS-row tiles of one [L][D] matrix from memory to LDS: each of the four waves takes a quarter of
// a tile's rows, 1 KiB per instruction.  Lane l fills the l-th 16 bytes of the kilobyte; the permuted
// layout (tile_off) is obtained by letting it fetch the chunk that belongs there.  A tile costs one scalar
// base and one LDS address for up to four instructions: the instruction's offset (1 KiB, 2 KiB, ..)
// moves both addresses, and what the rows are further apart in memory than in LDS is in the lanes' offsets,
// a register per instruction.  (With a base and an LDS address of its own per instruction a tile took 50 scalar
// instructions of a wave's 120.)
// LIVE: the elements of a row that there are to move; the lanes of the rest of the pitch D fetch a chunk that another lane moves
// too, which nothing reads.
template <int D, int ROWS, int LIVE = D>
struct TileLoader {
  static constexpr int CPR = D / 8;            // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;         // rows per load instruction
  static constexpr int RPW = ROWS / 4;         // rows per wave
  static constexpr int NLD = RPW / RPI;        // load instructions per wave and tile
  static constexpr int NV = NLD < 16 / RPI ? NLD : 16 / RPI;  // of which so many share a base: 16 rows, whose offsets fit
                                                              // 32 bits and after which the permutation repeats
  static constexpr int kBack = 1024 * (NV - 1);  // the base lies this far before the rows: the lanes' offsets are unsigned, and
                                                 // rows may be closer together in memory than in LDS
  const char* base;  // this wave's first row of the first tile
  unsigned rowb;     // bytes from row to row
  int left;          // rows from there on
  unsigned voff[NV];
  RA_DEV void init(const bf16_t* base_, long long sl, int L, int wave, int lane) {
    rowb = (unsigned)sl * 2;
    base = (const char*)base_ + (unsigned long long)(RPW * wave) * rowb;
    left = L - RPW * wave;
#pragma unroll
    for (int t = 0; t < NV; ++t)
      voff[t] = (unsigned)(lane / CPR + RPI * t) * rowb + (kBack - 1024 * t) + chunk(RPW * wave + RPI * t, lane);
  }
  // byte offset inside its row of the chunk that a lane moves with the instruction that starts at `row` of a tile
  static RA_DEV unsigned chunk(int row, int lane) {
    const int r = row + lane / CPR;
    const unsigned c = (unsigned)(tile_off<D>(r, lane % CPR) - r * (D * 2));
    return LIVE < D && c >= LIVE * 2 ? c - (D - LIVE) * 2 : c;
  }
  // tile of the rows from row0 on, to the LDS address dst of the whole tile
  RA_DEV void issue(int row0, unsigned dst, int wave, int lane) const {
    dst += RPW * wave * (D * 2);
    if (row0 + RPW <= left) {
      const char* sb = base + (unsigned long long)(unsigned)row0 * rowb - kBack;  // wave-uniform: scalar registers
#pragma unroll
      for (int t = 0; t < NLD; t += NV) {
        if constexpr (NV == 4) global_to_lds16_s4(sb, voff[0], voff[1], voff[2], voff[3], dst + RPI * t * (D * 2));
        else if constexpr (NV == 2) global_to_lds16_s_x2(sb, voff[0], voff[1], dst + RPI * t * (D * 2));
        else global_to_lds16_s(sb, voff[0], dst + RPI * t * (D * 2));
        sb += (unsigned long long)(RPI * NV) * rowb;
      }
    } else {  // past the end: the last row again (masked later)
      lane = opaque_lane(lane);
#pragma unroll
      for (int t = 0; t < NLD; ++t) {
        const int row = min(row0 + RPI * t + lane / CPR, left - 1);
        global_to_lds16(base + (long long)row * (long long)rowb + chunk(RPW * wave + RPI * t, lane), dst + RPI * t * (D * 2));
      }
    }
  }
};

// Per-lane LDS byte offsets of the operand fetches inside a block of 32 rows.  The permutation of a
// row's chunks is an XOR, and so is the step from one operand to the next: two registers and an XOR
// per fetch instead of a register per operand, which these kernels do not have.
template <int D>
struct FragOffsets {
  int n0, t0;
  RA_DEV explicit FragOffsets(int lane) {
    const int l32 = lane & 31, g = lane >> 5, j = lane & 15;
    n0 = tile_off<D>(l32, g);
    const int col = 16 * ((lane >> 4) & 1) + 4 * (j & 3);
    t0 = tile_off<D>(4 * g + (j >> 2), col >> 3) + ((col & 4) << 1);
  }
  RA_DEV FragOffsets opaque() const {  // not to be hoisted out of the loop it is used in
    FragOffsets r = *this;
    asm volatile("" : "+v"(r.n0), "+v"(r.t0));
    return r;
  }
  // row l32, head-dim elements 16 ss + 8 g ..: chunk 2 ss + g
  RA_DEV int nat(int ss) const { return n0 ^ (ss << 5); }
  // rows 8 h2 + 4 g + j / 4, columns 32 db + ...: chunk 4 db + ...; eight rows further the row's
  // permutation differs in one bit (D = 128: bit 1, D = 64: bit 2 of the chunk)
  RA_DEV int tr(int db, int h2) const { return (t0 ^ (db << 6) ^ (h2 * (D == 128 ? 32 : 64))) + h2 * 8 * (D * 2); }
};

// Smallest and largest value of N neighbouring lanes (8 or 16), in all of them.
template <int CTRL>
RA_DEV int dpp(int x) {
  return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false);
}
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e, kDppMirror8 = 0x141, kDppMirror16 = 0x140;
template <int N = 16>
RA_DEV int row_min(int x) {
  x = min(x, dpp<kDppXor1>(x));
  x = min(x, dpp<kDppXor2>(x));
  x = min(x, dpp<kDppMirror8>(x));
  return N == 16 ? min(x, dpp<kDppMirror16>(x)) : x;
}
template <int N = 16>
RA_DEV int row_max(int x) {
  x = max(x, dpp<kDppXor1>(x));
  x = max(x, dpp<kDppXor2>(x));
  x = max(x, dpp<kDppMirror8>(x));
  return N == 16 ? max(x, dpp<kDppMirror16>(x)) : x;
}

// The segment ids and prefix flags of a wave's 32 rows, as uniform values.
struct WaveIds {
  int lo, hi;     // smallest and largest segment id of the wave's rows
  bool any, all;  // some / every row carries the prefix flag
  RA_DEV void init(bool valid, int seg, int pre) {
    const int mn = row_min(valid ? seg : 0x7fffffff), mx = row_max(valid ? seg : (int)0x80000000);  // (both halves of the wave hold the rows)
    lo = min(__builtin_amdgcn_readlane(mn, 0), __builtin_amdgcn_readlane(mn, 16));
    hi = max(__builtin_amdgcn_readlane(mx, 0), __builtin_amdgcn_readlane(mx, 16));
    any = __any(valid && pre != 0);
    all = __all(!valid || pre != 0);
  }
};

// Calls put(i, smallest, largest) for the ids of tiles j_lo + i, i in [i_lo, n), of T tokens, of an array of L, or for its flags as 0 and 1; all
// four waves.  A lane takes four neighbouring tokens and T / 4 lanes a tile: a load instruction reads a kilobyte in one piece.  (A lane per tile
// reads 64 lines per instruction.  Documents of 16 in 32768, H=16, which are little but lists, so | like this, us, forward, backward:
// D=128 206 | 191, 534 | 501; D=64 127 | 111, 331 | 294; documents of 100, D=128 238 | 226, 628 | 606.)
template <int T, bool FLAGS, typename Put>
RA_DEV void tile_ranges(const int* ids, int j_lo, int i_lo, int n, int L, int wave, int lane, Put put) {
  constexpr int LPT = T / 4, TPL = 64 / LPT, U = 8;  // lanes per tile, tiles per load, loads in flight
  const bool aligned = ((uintptr_t)ids & 15) == 0;
  for (int base = i_lo + wave * (U * TPL); base < n; base += 4 * U * TPL) {
    i32x4 x[U];
    const int first = (j_lo + base) * T + 4 * lane;  // of this lane's tokens in the first load
    if (aligned && (j_lo + base + U * TPL) * T <= L) {
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = *(const i32x4*)(ids + first + u * 256);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c) x[u][c] = ids[min(first + u * 256 + c, L - 1)];  // (repeats of the last one change nothing)
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (FLAGS) {
#pragma unroll
        for (int c = 0; c < 4; ++c) x[u][c] = x[u][c] != 0;
      }
      const int lo = row_min<LPT>(min(min(x[u][0], x[u][1]), min(x[u][2], x[u][3])));
      const int hi = row_max<LPT>(max(max(x[u][0], x[u][1]), max(x[u][2], x[u][3])));
      const int i = base + u * TPL + lane / LPT;
      if (lane % LPT == 0 && i < n) put(i, lo, hi);
    }
  }
}

// The entries of the n tiles from j_lo on whose flag is set, in order; returns their number.  A thread takes PER neighbouring flags.
// cells: the list holds the tiles' cells.
template <bool DENSE, int PER>
RA_DEV int compact_list(int j_lo, int n, bool cells, int* s_red, const unsigned char* s_flag, ListEntry<DENSE>* s_list) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i0 = threadIdx.x * PER;
  unsigned entry[PER];
  int mine = 0;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int f = i0 + p < n ? s_flag[i0 + p] : 0;
    entry[p] = f ? (j_lo + i0 + p) | ((f & 7) << kTestShift) | 0x80000000u : 0u;
    if constexpr (DENSE) {
      if (f) entry[p] = (entry[p] & 0xffff) | (cells ? s_list[i0 + p] : 0xffffu) << kCellShift;
    }
    mine += f != 0;
  }
  int before = 0, all = 0;
#pragma unroll
  for (int bit = 1; bit <= PER; bit <<= 1) {
    const unsigned long long mask = __ballot(mine & bit);
    before += bit * __popcll(mask & ((1ull << lane) - 1ull));
    all += bit * __popcll(mask);
  }
  if (lane == 0) s_red[wave] = all;
  __syncthreads();  // (the cells have been read, too)
  const int n0 = s_red[0], n1 = s_red[1], n2 = s_red[2], n3 = s_red[3];
  int at = before + (wave > 0 ? n0 : 0) + (wave > 1 ? n1 : 0) + (wave > 2 ? n2 : 0);
#pragma unroll
  for (int p = 0; p < PER; ++p)
    if (entry[p]) s_list[at++] = (ListEntry<DENSE>)entry[p];
  __syncthreads();
  return n0 + n1 + n2 + n3;
}

// The list of key tiles that the workgroup's rows [q0, q_hi] have to visit, of the n from j_lo on:
// tiles that one or the other term rules out are dropped, the others carry the terms that they
// have to be tested for.  Returns their number.  Called by all four waves.
template <bool DENSE>
RA_DEV int list_key_tiles(int Lq, int Lk, const BiasArgs& bs, const int* kv_seg, const int* kv_pre, const unsigned char* dmap,
                          int q0, int q_hi, const WaveIds& w, int j_lo, int n, int* s_red,
                          unsigned char* s_flag, ListEntry<DENSE>* s_list) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool seg_on = kv_seg != nullptr, pre_on = kv_pre != nullptr;
  if (lane == 0) {
    s_red[wave] = w.lo;
    s_red[4 + wave] = w.hi;
    s_red[8 + wave] = w.any;
    s_red[12 + wave] = w.all;
  }
  __syncthreads();
  const int qmin = min(min(s_red[0], s_red[1]), min(s_red[2], s_red[3]));
  const int qmax = max(max(s_red[4], s_red[5]), max(s_red[6], s_red[7]));
  const bool q_any = s_red[8] | s_red[9] | s_red[10] | s_red[11], q_all = s_red[12] & s_red[13] & s_red[14] & s_red[15];
  if (seg_on) {
    tile_ranges<kPairKeys, false>(kv_seg, j_lo, 0, n, Lk, wave, lane, [&](int i, int kmin, int kmax) {
      s_flag[i] = (kmax < qmin || kmin > qmax) ? 0 : (kmin != kmax || qmin != qmax) ? 0x80 | kTestSegment : 0x80;  // 0x80: listed
    });
  } else {
    for (int i = tid; i < n; i += kPairThreads) s_flag[i] = 0x80;
  }
  if (pre_on) {
    __syncthreads();
    // from the first tile on with a key behind the first row's position
    const int i_lo = max(0, floor_div(bs.q_off + q0 - bs.kv_off + 1, kPairKeys) - j_lo);
    tile_ranges<kPairKeys, true>(kv_pre, j_lo, i_lo, n, Lk, wave, lane, [&](int i, int all, int any) {
      const int klo = bs.kv_off + (j_lo + i) * kPairKeys, khi = bs.kv_off + min((j_lo + i + 1) * kPairKeys, Lk) - 1;
      const int c = prefix_class(bs.q_off + q0, bs.q_off + q_hi, klo, khi, q_any, q_all, any, all);
      const int f = s_flag[i];
      if (f && c) s_flag[i] = c == 2 ? 0 : f | kTestPrefix;
    });
  }
  if constexpr (DENSE) {
    if (dmap != nullptr) {
      __syncthreads();
      for (int i = tid; i < n; i += kPairThreads) {
        // the summary's cells of the four waves' rows, two bits each, first and second key block of the tile
        const int ncols = (Lk + kMapCell - 1) / kMapCell;
        unsigned cells = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int r = q0 / kMapCell + c / 2, col = 2 * (j_lo + i) + c % 2;
          if (r * kMapCell <= q_hi && col < ncols) cells |= (dmap[(long long)r * ncols + col] & 3u) << (2 * c);
        }
        if (!(cells & 0x5555)) s_flag[i] = 0;
        else if ((cells & 0xaaaa) && s_flag[i]) s_flag[i] |= kTestDense;
        s_list[i] = cells;  // (until the entries are written)
      }
    }
  }
  __syncthreads();
  return compact_list<DENSE, kPairListTiles / kPairThreads>(j_lo, n, dmap != nullptr, s_red, s_flag, s_list);
}

// ALiBi on one side of the diagonal: -slope |q - k| = s (j - rel), with s = +-slope, rel the distance of this lane's
// row from the tile's first position and j the index in the tile.  s j enters through the matrix unit as the
// accumulator's initial value, exactly: an fp32 product of depth two, [j, 1] x [s, c].  The constant -s rel, which
// far from the diagonal is larger than anything else by orders of magnitude, goes into the exponent where the lane owns the row
// (forward, dQ): in the accumulator it would cost every score its last bits (logsumexp at a bias of 6200: off by
// 3.4e-3, and by 6e-4 so).  Under dK / dV it is c, on top of -logsumexp, which it cancels.  (Split into
// bf16 words for the bf16 product, s and c took 20 vector instructions a tile, of the 200 of a forward tile.)
// `j`: alibi_index of the block.
// The initial value is the same in every tile on one side: the forward keeps it in the 16 registers that it has free, dQ in LDS; one product
// per tile | kept, us, D=64 4096, B=2, H=16, causal 121 | 114 and the backward 276 | 268; 8192, H=16 381 | 366 and 918 | 899; D=128 8192, H=16
// 599 | 580 and 1585 | 1574; documents of 2000 in 32768, H=16 1735 | 1716 and 4489 | 4452.
RA_DEV float alibi_index(int first, int l32, int g) { return g == 0 ? (float)(first + l32) : 1.0f; }
// -slope rel log2(e), and what that lacks of the product to twice the bits
RA_DEV float alibi_far(float slope, int rel, float& rest) {
  constexpr float hi = kLog2e, lo = (float)(1.4426950408889634074 - (double)hi);
  const float r = (float)rel, x = -slope * r, y = x * hi;
  rest = fmaf(x, lo, fmaf(x, hi, -y)) + fmaf(-slope, r, -x) * hi;
  return y;
}
RA_DEV f32x16 alibi_one_side(const f32x16& init, float j, float s, float c, int g) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(j, g == 0 ? s : c, init, 0, 0, 0);
}

// What the 32 rows of a wave need done for a tile of the streamed side, as ranges of tile indexes: outside of `live`
// the positional terms mask every score, inside of `plain` none (and the tile is whole); ALiBi is linear
// for tiles below `past` and from `future` on.
struct WaveTiles {
  int live_lo, live_n, plain_lo, plain_n, past, future;
  template <int T>
  RA_DEV void sides(int lo, int hi, int off) {  // of rows at positions [lo, hi]; tile 0 starts at position off
    past = floor_div(lo - off - (T - 1), T) + 1;
    future = ceil_div(hi - off, T);
  }
  RA_DEV bool live(int j) const { return (unsigned)(j - live_lo) < (unsigned)live_n; }
  RA_DEV bool plain(int j) const { return (unsigned)(j - plain_lo) < (unsigned)plain_n; }
};
RA_DEV WaveTiles wave_key_tiles(const BiasArgs& bs, int qlo, int qhi, int Lk) {
  WaveTiles w;
  const int flags = bs.flags & ~RA_BIAS_PREFIX;  // (tested for by itself)
  const int n = (Lk + kPairKeys - 1) / kPairKeys;
  int hi;
  key_tile_range(flags, bs.window, qlo, qhi, bs.kv_off, n, kPairKeys, w.live_lo, hi);
  w.live_n = hi - w.live_lo;
  key_tile_plain_range(flags, bs.window, qlo, qhi, bs.kv_off, Lk / kPairKeys, kPairKeys, w.plain_lo, hi);
  w.plain_n = hi - w.plain_lo;
  w.sides<kPairKeys>(qlo, qhi, bs.kv_off);
  return w;
}

// Drops the tests of a tile that hold for none or all of the wave's scores; true: every score is masked.
// ids, flags: the tile's, one per lane (of a tile of 32 twice).  before: the keys of the tile and the wave's queries (or the other
// way round) are in causal order throughout; after: none of them is.
RA_DEV bool wave_tests(int& tests, const WaveIds& w, const int* ids, const int* flags, bool before, bool after, int lane) {
  lane = opaque_lane(lane);
  if (tests & kTestSegment) {
    const int id = ids[lane];
    if (!__any(id >= w.lo && id <= w.hi)) return true;
    if (w.lo == w.hi && __all(id == w.lo)) tests &= ~kTestSegment;
  }
  if (tests & kTestPrefix) {
    if (before) {
      tests &= ~kTestPrefix;
    } else {
      const bool f = flags[lane] != 0;
      if (w.all && __all(f)) tests &= ~kTestPrefix;
      else if (after && !(w.any && __any(f))) return true;
    }
  }
  return false;
}

// What the summary says about a block, as tests: nothing to do, values to add, or every score masked.
RA_DEV int cell_tests(int tests, unsigned cell) {
  if (!(tests & kTestDense) || cell == (kMapLive | kMapNonZero)) return tests;
  return (tests & ~kTestDense) | ((cell & kMapLive) ? 0 : kTestDead);
}

// The terms `todo` (kTest..., kTestPos, kTestAlibi, kTestDead) on one 32x32 block: see apply_bias, whose interval test, id test,
// prefix test and ALiBi are here one pass over the elements each, taken where the block needs it - most
// blocks that need one need no other, and a pass is two to four instructions per element where the common
// form takes five and a scalar one.
template <bool QFIXED, bool DENSE, bool GENERAL>
RA_DEV void apply_terms(f32x16& t, int todo, const TileBias& tb, int rel0, int fixed_seg, int fixed_pre, const int* var_seg,
                        const int* var_pre) {
  if constexpr (DENSE) {
    if (todo & kTestDead) {
#pragma unroll
      for (int r = 0; r < 16; ++r) t[r] = RA_NEG_INF;
      return;
    }
  }
  if constexpr (GENERAL) {
    if (todo & kTestAlibi) {
      const float slope = -tb.slope2, relf0 = (float)rel0;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float off = (float)(8 * (r / 4) + r % 4);
        t[r] = fmaf(fabsf(QFIXED ? relf0 - off : relf0 + off), slope, t[r]);
      }
    }
    if constexpr (DENSE) {
      if (todo & kTestDense) {
        const bool vec = __builtin_amdgcn_readfirstlane(tb.dense_vec);
        if (QFIXED && vec) {
          // a lane's four keys are 16 contiguous bytes of its row
          f32x4 dn[4];
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) dn[bb] = *(const f32x4*)(tb.dense + 8 * bb);
#pragma unroll
          for (int r = 0; r < 16; ++r) t[r] = fmaf(dn[r / 4][r % 4], tb.dense_mul, t[r]);
        } else if (QFIXED) {
          float dn[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int off = 8 * (r / 4) + r % 4;
            dn[r] = 0.f;
            if (off < tb.var_limit) dn[r] = tb.dense[off];
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) t[r] = fmaf(dn[r], tb.dense_mul, t[r]);
        } else if (vec) {
          // a row of the block is scalar, in it and between the wave's halves a lane has one offset.  (An address per lane and row, each
          // under a range test: 11 registers of dkdv_pair_kernel<128, 2> went to scratch inside the loop.)
          float dn[16];
          const char* row = (const char*)tb.dense;
          const unsigned at = tb.dense_lane;
#pragma unroll
          for (int r = 0; r < 16; ++r) dn[r] = *(const float*)(row + (8 * (r / 4) + r % 4) * tb.dense_vs * 4 + at);
#pragma unroll
          for (int r = 0; r < 16; ++r) t[r] = fmaf(dn[r], tb.dense_mul, t[r]);
        } else {
          // rows past the end read the last one again (masked below); four at a time, for want of registers
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) {
            float dn[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) dn[c] = tb.dense[max(min(8 * bb + c, tb.var_limit - 1), 0) * tb.dense_vs + tb.dense_lane];
#pragma unroll
            for (int c = 0; c < 4; ++c) t[4 * bb + c] = fmaf(dn[c], tb.dense_mul, t[4 * bb + c]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
    if (todo & kTestSegment) {
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const i32x4 vs = *(const i32x4*)(var_seg + 8 * bb);
#pragma unroll
        for (int c = 0; c < 4; ++c) t[4 * bb + c] = vs[c] != fixed_seg ? RA_NEG_INF : t[4 * bb + c];
      }
    }
    if (todo & kTestPrefix) {
      // masked where the key is behind the query's position, unless both carry the flag
      constexpr int kFar = 1 << 30;
      const int edge = QFIXED ? rel0 : -rel0, free = fixed_pre != 0 ? (QFIXED ? kFar : -kFar) : edge;
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const i32x4 vp = *(const i32x4*)(var_pre + 8 * bb);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int off = 8 * bb + c, e = vp[c] != 0 ? free : edge;
          t[4 * bb + c] = (QFIXED ? off > e : off < e) ? RA_NEG_INF : t[4 * bb + c];
        }
      }
    }
  }
  if (todo & kTestPos) {
    // range limit, causal and window terms: an interval of the element's offset on the varying side
    const bool causal = tb.flags & RA_BIAS_CAUSAL, window = tb.flags & RA_BIAS_WINDOW;
    int lo = 0, hi = tb.var_limit - 1;
    if (QFIXED) {
      if (causal) hi = min(hi, rel0);
      if (window) lo = max(lo, rel0 - tb.window + 1);
      if (window && !causal) hi = min(hi, rel0 + tb.window - 1);
    } else {
      if (causal) lo = max(lo, -rel0);
      if (window) hi = min(hi, tb.window - 1 - rel0);
      if (window && !causal) lo = max(lo, 1 - rel0 - tb.window);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 8 * (r / 4) + r % 4 > hi ? RA_NEG_INF : t[r];
    if (window || (!QFIXED && causal)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) t[r] = 8 * (r / 4) + r % 4 < lo ? RA_NEG_INF : t[r];
    }
  }
}

// The tiles of a workgroup one after another: entries of its list, or consecutive ones.  An entry is read two tiles
// ahead, so that the address of the next tile is there when it is requested.
template <bool DENSE>
struct TileWalk {
  typedef __attribute__((address_space(3))) const ListEntry<DENSE> lds_entry;
  lds_entry* list;
  bool listed;  // (else consecutive tiles)
  int j_lo, i_hi, every_test, mask;
  int now, ahead;  // the entry of the current tile (uniform); one of the next tile, as it came from LDS
  RA_DEV int entry(int i) const {
    i = min(i, i_hi - 1);
    return listed ? (int)list[i] : j_lo + i;
  }
  RA_DEV void start(bool listed_, const ListEntry<DENSE>* list_, int j_lo_, int i_lo, int i_hi_, int every_test_) {
    listed = listed_;
    list = (lds_entry*)list_;
    j_lo = j_lo_;
    i_hi = i_hi_;
    every_test = every_test_;
    mask = listed_ ? (1 << kTestShift) - 1 : 0x7fffffff;
    now = __builtin_amdgcn_readfirstlane(entry(i_lo));
    ahead = entry(i_lo + 1);
  }
  RA_DEV int tile() const { return now & mask; }
  RA_DEV int tests() const { return ((now & ~mask & 0xffff) >> kTestShift) | every_test; }
  RA_DEV unsigned cells() const { return listed ? (unsigned)now >> kCellShift : 0xffffu; }
  RA_DEV void next(int i) {  // i: ordinal of the tile that becomes the current one
    now = __builtin_amdgcn_readfirstlane(ahead);
    ahead = entry(i + 1);
  }
};

// S^T orientation as in fwd_step_kernel: a lane owns one query row and 16 keys of a 32-key block.
// DL is the head dim, a multiple of 32; the LDS tiles keep a row pitch D of 64 or 128 elements, whose layout both operand
// fetches know, and what lies beyond DL is neither multiplied nor stored.  Padded to 64 or 128 | in the head dim itself, whole training
// calls: D=96, 32768 causal, H=16 15.2 | 13.4 ms (padded on the long-stretch kernels), window 4096 4.32 | 3.47, causal 4096, B=2,
// H=16 659 | 496 us, unmasked 8192 x 16384 3.79 | 3.47 ms; D=32, 32768 causal, H=16 8.2 | 6.0 ms; fp16, D=96, 1047 x 4791, B=2, H=8 283 |
// 229 us, conversions included.
template <int DL, int MODE>
__global__ __launch_bounds__(kPairThreads, 2) void fwd_pair_kernel(const PairFwdArgs a) {
  constexpr bool GENERAL = MODE != 0;
  constexpr bool DENSE = MODE == 2;
  constexpr int D = DL <= 64 ? 64 : 128;  // row pitch of the LDS tiles
  constexpr int KS = DL / 16, DB = DL / 32;
  constexpr int ROWB = D * 2;
  constexpr int TILE_BYTES = kPairKeys * ROWB;
  __shared__ __attribute__((aligned(16))) char s_k[2][TILE_BYTES];
  __shared__ __attribute__((aligned(16))) char s_v[2][TILE_BYTES];
  __shared__ __attribute__((aligned(16))) int s_seg[GENERAL ? 2 : 1][kPairKeys];
  __shared__ __attribute__((aligned(16))) int s_pre[GENERAL ? 2 : 1][kPairKeys];
  __shared__ ListEntry<DENSE> s_list[GENERAL ? kPairListTiles : 1];
  __shared__ unsigned char s_flag[GENERAL ? kPairListTiles : 1];
  __shared__ int s_red[20];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int nqt = (a.Lq + kPairRows - 1) / kPairRows;
  int hh, split, qt;
  pair_decode(blockIdx.x, a.B * a.H, nqt, a.n_split, a.group, hh, split, qt);
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
  auto load_rows = [&]() {
    const bf16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh + (long long)qi_c * a.q.sl + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *(const bf16x8*)(qp + 16 * s);
  };
  // (A dense block may leave these rows nothing, as ring steps on masks often do: there the list comes first.  Blocks of 8192 x 8192, H=16,
  // that are masked throughout, rows first | list first, us: forward 15 | 9, both gradients 44 | 20.)
  if (!DENSE) load_rows();
  int q_seg = 0, q_pre = 0;
  float slope = 0.f, slope2 = 0.f;  // slope2: in the units of the scores
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
    if (flags & RA_BIAS_ALIBI) {
      slope = bs.slopes[h];
      slope2 = slope * kLog2e / a.scale2;
    }
  }

  WaveIds ids;
  if constexpr (GENERAL) ids.init(q_valid, q_seg, q_pre);
  bool use_list = false;
  const unsigned char* dmap = nullptr;
  if constexpr (DENSE) {
    if (bs.dense_map) dmap = dense_map_of(bs, b, h, a.H, a.Lq, a.Lk);
  }
  if constexpr (GENERAL) {
    use_list = ntiles <= kPairListTiles && ((flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX)) || dmap != nullptr);
    if (use_list)
      n = list_key_tiles<DENSE>(a.Lq, a.Lk, bs, kv_seg, kv_pre, dmap, q0, q_hi, ids, j_lo, n, s_red, s_flag, s_list);
  }
  n = __builtin_amdgcn_readfirstlane(n);
  j_lo = __builtin_amdgcn_readfirstlane(j_lo);
  if (n == 0 && a.o != nullptr) return;  // identity on the carry
  if (DENSE) load_rows();
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

  TileLoader<D, kPairKeys, DL> ldk, ldv;
  ldk.init(a.k.ptr + b * a.k.sb + h * a.k.sh, a.k.sl, a.Lk, wave, lane);
  ldv.init(a.v.ptr + b * a.v.sb + h * a.v.sh, a.v.sl, a.Lk, wave, lane);
  auto issue_tile = [&](int j, int buf) {
    const int k0 = j * kPairKeys;
    ldk.issue(k0, RA_LDS_ADDR(&s_k[0][0]) + buf * TILE_BYTES, wave, lane);
    ldv.issue(k0, RA_LDS_ADDR(&s_v[0][0]) + buf * TILE_BYTES, wave, lane);
    if constexpr (GENERAL) {
      const int kk = min(k0 + lane, a.Lk - 1);
      if (kv_seg && wave == 0) global_to_lds4(kv_seg + kk, RA_LDS_ADDR(&s_seg[0][0]) + buf * (kPairKeys * 4));
      if (kv_pre && wave == 1) global_to_lds4(kv_pre + kk, RA_LDS_ADDR(&s_pre[0][0]) + buf * (kPairKeys * 4));
    }
  };

  float m_run = RA_NEG_INF;  // exponent reference (log2 domain), moves lazily
  float m_true = RA_NEG_INF;
  float l_run = 0.f;  // row sum of the probabilities ...
  // ... and, in the first element, of the rounded ones (see fwd_step_kernel): by dot products, or, where vector issue binds and the matrix
  // pipe has room, as matrix products of four ones and a lane's own four values (a column of a 4x4 block is one lane).  us, forward, dot
  // products | matrix products: D=64 causal + ALiBi 4096, B=2, H=16 118 | 111, unmasked 8192, H=16 322 | 320; D=32 causal 8192, H=16 143 |
  // 137; D=128 causal 4096, H=16 95 | 98, documents + ALiBi 32768 1694 | 1703.
  constexpr bool SUM_MFMA = DL <= 64;
  f32x4 lr_acc = {0.f, 0.f, 0.f, 0.f};
  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
  const i16x4 ones4 = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
  const bf16x2 ones2 = {(bf16_t)1.0f, (bf16_t)1.0f};

  const FragOffsets<D> fo(lane);
  const bool wave_on = qw < a.Lq;
  const bool alibi_on = GENERAL && (flags & RA_BIAS_ALIBI);
  const WaveTiles wt = wave_key_tiles(bs, q_off + qw, q_off + qw + 31, a.Lk);
  TileWalk<DENSE> walk;
  f32x16 ramp;  // ALiBi's initial value of the scores (alibi_one_side), the same in every tile on one side of the diagonal
  bool ramp_past = false;
#pragma unroll
  for (int r = 0; r < 16; ++r) ramp[r] = 0.f;
  if (alibi_on) {
    const f32x16 none = ramp;
    ramp = alibi_one_side(none, alibi_index(0, l32, g), -slope2, 0.f, g);
  }

  auto step = [&](auto buffer, int i) {
    constexpr int BUF = decltype(buffer)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's share of tile i is in LDS
    __syncthreads();                     // everyone's is, and nobody reads the other buffer any more
    const FragOffsets<D> fr_off = fo.opaque();
    // K operands in the order of use, both key blocks of 16 head-dim elements in turn; the first ones
    // are on their way while the next tile is requested
    constexpr int PFK = 4 < 2 * KS ? 4 : 2 * KS;
    bf16x8 kf[2 * KS];
    auto k_frag = [&](int op) { return *(const bf16x8*)(s_k[BUF] + 32 * (op & 1) * ROWB + fr_off.nat(op >> 1)); };
#pragma unroll
    for (int op = 0; op < PFK; ++op) kf[op] = k_frag(op);
    __builtin_amdgcn_sched_barrier(0);
    const int j = walk.tile(), kt0 = j * kPairKeys;
    int tests = walk.tests();
    bool dead = !wave_on || !wt.live(j);
    unsigned cells = 0;
    if constexpr (DENSE) {
      if (tests & kTestDense) {
        cells = walk.cells() >> (4 * wave);
        dead = dead || !(cells & 5);
        if ((cells & 15) == 5) tests &= ~kTestDense;
      }
    }
    if (i + 1 < i_hi) {
      walk.next(i + 1);
      issue_tile(walk.tile(), BUF ^ 1);
    }
    if (dead) return;
    const bool one_side = alibi_on && (j < wt.past || j >= wt.future);
    if constexpr (GENERAL) {
      if (tests && wave_tests(tests, ids, s_seg[BUF], s_pre[BUF], j < wt.past, j > wt.future, lane)) return;
      if (alibi_on && !one_side) tests |= kTestAlibi;
    }
    if (!wt.plain(j)) tests |= kTestPos;
    f32x16 S[2], zero;
    float beyond = 0.f, far = 0.f, far_rest = 0.f;  // what the scores of the second key block, and the exponents of all, lack
#pragma unroll
    for (int r = 0; r < 16; ++r) zero[r] = 0.f;
    __builtin_amdgcn_s_setprio(1);
    if (one_side) {
      const int at = opaque_lane(lane), l = at & 31, half = at >> 5;
      // one initial value for both key blocks: the second one's is 32 slopes further, added to its exponents
      const bool past = j < wt.past;
      const float s = past ? slope2 : -slope2;
      if (past != ramp_past) {
        ramp = alibi_one_side(zero, alibi_index(0, l, half), s, 0.f, half);
        ramp_past = past;
      }
      beyond = 32.f * s;
      far = alibi_far(j < wt.past ? slope : -slope, q_off + qw + l - (kv_off + kt0), far_rest);
      S[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[0], ramp, 0, 0, 0);
      S[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[0], ramp, 0, 0, 0);
    } else {
      S[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[0], zero, 0, 0, 0);
      S[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[0], zero, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PFK < 2 * KS) {
      kf[PFK] = k_frag(PFK);
      kf[PFK + 1] = k_frag(PFK + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int op = 2; op < 2 * KS; ++op) {
      if (op + PFK < 2 * KS) kf[op + PFK] = k_frag(op + PFK);
      S[op & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[op], qf[op >> 1], S[op & 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    if (tests) {
      const int at = opaque_lane(lane), g = at >> 5, qi = qw + (at & 31);
      TileBias tb;
      tb.flags = flags;
      tb.window = bs.window;
      tb.slope2 = slope2;
      tb.dense_mul = kLog2e / a.scale2;
      const float* head = nullptr;
      if (DENSE) {
        head = bs.dense + b * bs.dense_sb + h * bs.dense_sh;
        tb.dense_vec = kt0 + kPairKeys <= a.Lk && ((((uintptr_t)head) | ((uintptr_t)bs.dense_sq << 2)) & 15) == 0;
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int var0 = kt0 + 32 * kb + 4 * g;
        tb.var_limit = a.Lk - var0;
        if (DENSE) tb.dense = head + (long long)min(qi, a.Lq - 1) * bs.dense_sq + var0;
        apply_terms<true, DENSE, GENERAL>(S[kb], DENSE ? cell_tests(tests, (cells >> (2 * kb)) & 3) : tests, tb,
                                          (q_off + qi) - (kv_off + var0), q_seg, q_pre, &s_seg[GENERAL ? BUF : 0][32 * kb + 4 * g],
                                          &s_pre[GENERAL ? BUF : 0][32 * kb + 4 * g]);
      }
    }
    float mx0 = RA_NEG_INF, mx1 = RA_NEG_INF;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      mx0 = fmaxf(fmaxf(mx0, S[0][r]), S[0][r + 1]);
      mx1 = fmaxf(fmaxf(mx1, S[1][r]), S[1][r + 1]);
    }
    const float mx = GENERAL ? fmaf(half_max(fmaxf(mx0, mx1 + beyond)), a.scale2, far) : half_max(fmaxf(mx0, mx1)) * a.scale2;
    m_true = fmaxf(m_true, mx);
    if (__any(mx > m_run + 8.0f)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = fast_exp2(m_run - ((m_new == RA_NEG_INF) ? 0.f : m_new));
      m_run = m_new;
      l_run *= corr;
      if constexpr (SUM_MFMA) lr_acc *= corr;
      else lr_acc[0] *= corr;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= corr;
    }
    const float neg_ref = (m_run == RA_NEG_INF) ? 0.f : -m_run, neg_m = GENERAL ? (neg_ref + far) + far_rest : neg_ref;
    const float neg_m1 = GENERAL ? fmaf(beyond, a.scale2, neg_m) : neg_m;
    // The 32 scores of a lane go through exp2 in four groups of eight, one group per 16 keys of the
    // output product: group ks + 1 is worked on while the matrix unit multiplies with group ks.
    bf16x8 pf[4];
    float rs0 = 0.f, rs1 = 0.f;
    auto soft = [&](int ks, int e) {  // elements e, e + 1 of group ks
      const int r = 8 * (ks & 1) + e;
      const float p0 = fast_exp2(fmaf(S[ks >> 1][r], a.scale2, ks < 2 ? neg_m : neg_m1));
      const float p1 = fast_exp2(fmaf(S[ks >> 1][r + 1], a.scale2, ks < 2 ? neg_m : neg_m1));
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
      const lds_char* p0 = (const lds_char*)(s_v[BUF] + 16 * ks * ROWB + fr_off.tr(db, 0));
      const lds_char* p1 = (const lds_char*)(s_v[BUF] + 16 * ks * ROWB + fr_off.tr(db, 1));
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
        for (int e = 4 * db / DB; e < 4 * (db + 1) / DB; ++e) soft(ks + 1, 2 * e);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += rs0 + rs1;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const bf16x4 pr = {pf[ks][e], pf[ks][e + 1], pf[ks][e + 2], pf[ks][e + 3]};
        if constexpr (SUM_MFMA) {
          lr_acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones4, __builtin_bit_cast(i16x4, pr), lr_acc, 0, 0, 0);
        } else {
          lr_acc[0] = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){pr[0], pr[1]}, ones2, lr_acc[0], false);
          lr_acc[0] = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){pr[2], pr[3]}, ones2, lr_acc[0], false);
        }
      }
  };

  if (i_lo < i_hi) {
    walk.start(GENERAL && use_list, s_list, j_lo, i_lo, i_hi, every_test);
    issue_tile(walk.tile(), 0);
    for (int i = i_lo; i < i_hi; i += 2) {
      step(std::integral_constant<int, 0>{}, i);
      if (i + 1 < i_hi) step(std::integral_constant<int, 1>{}, i + 1);
    }
  }

  const auto* e = kernel_args<PairFwdArgs>();
  // a wave without a live score leaves its rows of the carry as they are, unread (m would come back through
  // two unit conversions, a last bit off)
  const float lr_run = lr_acc[0];
  if (e->o != nullptr && __all(l_run == 0.f && lr_run == 0.f)) return;
  const float l_step = half_sum(l_run), lr_step = half_sum(lr_run);
  if (e->part_n != nullptr && split == 0 && tid == 0) e->part_n[hh * nqt + qt] = n_piece;
  if (!q_valid) return;
  const long long row = (long long)hh * e->Lq + qi;
  if (n_piece > 1) {
    // a share of the row's keys: combined by pair_combine_kernel
    const long long prow = (long long)split * ((long long)e->B * e->H * e->Lq) + row;
    float* op = e->part_o + prow * DL + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        f32x4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = oacc[db][4 * bb + c];
        *(f32x4*)(op + 32 * db + 8 * bb) = t;
      }
    if (g == 0) *(f32x4*)(e->part_s + 4 * prow) = (f32x4){m_run, l_step, lr_step, 0.f};
  } else if (e->o != nullptr) {
    // merge into the carry (see fwd_step_kernel)
    const float m_in = e->m[row] * kLog2e, l_in = e->l[row];
    const float m_out = fmaxf(m_true, m_in), m_safe = (m_out == RA_NEG_INF) ? 0.f : m_out;
    const float f_in = fast_exp2(m_in - m_safe);
    const float f_step = (l_step > 0.f) ? fast_exp2(m_run - m_safe) : 0.f;
    const float f_o = f_step * ((lr_step > 0.f) ? l_step / lr_step : 1.f);
    float* op = e->o + row * DL + 4 * g;
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
      e->m[row] = m_out * kLn2;
      e->l[row] = l_in * f_in + l_step * f_step;
    }
  } else {
    const float inv = 1.0f / lr_step;
    const long long at = b * e->out_sb + h * e->out_sh + (long long)qi * e->out_sl + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        f32x4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = oacc[db][4 * bb + c] * inv;
        store4(e->out, e->out_f32, at + 32 * db + 8 * bb, t);
      }
    if (g == 0) e->lse[row] = (l_step > 0.f) ? (m_run + __log2f(l_step)) * kLn2 : RA_NEG_INF;
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

// ------------------------------------------------------------------------------------------------
// dQ
// ------------------------------------------------------------------------------------------------
// The same split: 128 query rows per workgroup (Q and dO in registers), 64-key tiles of K and V in two
// LDS buffers, scores transposed (S^T = K Q^T, dP^T = V dO^T) so that dS^T is the B operand of
// dQ^T = K^T dS^T, whose A operand comes from the K tile through the transposing read.
// (What the loop reads lies within the 64 KB that an LDS instruction's own offset reaches: with the tiles first, what lay behind them took
// registers for its addresses, and dkdv_pair_kernel<128, 2> reloaded 11 from scratch in its loop: diagonal blocks of documents of
// 2000, 8192 x 8192, H=16, 946 and 736 us for both gradients, 818 and 693 so.)
template <int DL, int MODE>
struct DqLds {
  static constexpr int TILE_BYTES = kPairKeys * (DL <= 64 ? 64 : 128) * 2;
  __attribute__((aligned(16))) float ramp[MODE ? 2 : 1][kPairKeys];  // ALiBi on either side of the diagonal: +-slope j of a tile's keys j
  __attribute__((aligned(16))) int seg[MODE ? 2 : 1][kPairKeys];
  __attribute__((aligned(16))) int pre[MODE ? 2 : 1][kPairKeys];
  __attribute__((aligned(16))) char k[2][TILE_BYTES];
  __attribute__((aligned(16))) char v[2][TILE_BYTES];
  ListEntry<MODE == 2> list[MODE ? kPairListTiles : 1];
  unsigned char flag[MODE ? kPairListTiles : 1];
  int red[20];
};
// args_at: where p lies in the kernel's arguments
template <int DL, int MODE>
RA_DEV void dq_pair(const PairBwdArgs& p, int bid, DqLds<DL, MODE>& lds, int args_at) {
  constexpr bool GENERAL = MODE != 0;
  constexpr bool DENSE = MODE == 2;
  constexpr int D = DL <= 64 ? 64 : 128;  // row pitch of the LDS tiles
  constexpr int KS = DL / 16, DB = DL / 32;
  constexpr int ROWB = D * 2;
  constexpr int TILE_BYTES = kPairKeys * ROWB;
  const BwdArgs& a = p.a;
  auto &s_k = lds.k, &s_v = lds.v;
  auto &s_seg = lds.seg, &s_pre = lds.pre;
  auto& s_list = lds.list;
  auto& s_flag = lds.flag;
  auto& s_red = lds.red;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int nqt = (a.Lq + kPairRows - 1) / kPairRows;
  int hh, split, qt;
  pair_decode(bid, a.B * a.H, nqt, p.n_split, p.group, hh, split, qt);
  const int b = hh / a.H, h = hh % a.H;
  const int q0 = qt * kPairRows;
  const int qw = q0 + wave * 32;
  const int qi = qw + l32;
  const bool q_valid = qi < a.Lq;
  const int qi_c = min(qi, a.Lq - 1);
  const BiasArgs& bs = a.bias;
  const int flags = bs.flags;
  const int q_off = bs.q_off, kv_off = bs.kv_off;

  const int ntiles = (a.Lk + kPairKeys - 1) / kPairKeys;
  const int q_hi = min(q0 + kPairRows, a.Lq) - 1;
  int j_lo, j_hi;
  key_tile_range(flags, bs.window, q_off + q0, q_off + q_hi, kv_off, ntiles, kPairKeys, j_lo, j_hi);
  int n = j_hi - j_lo;
  if (split > 0 && split * p.chunk_tiles >= n) return;

  // Q carries the power of two below sm_scale * log2(e) (exact in bf16), the residual factor is
  // applied to the fp32 score (see dkdv_kernel)
  bf16x8 qf[KS], dof[KS];
  float neg_lse, neg_lse2, neg_delta;
  const long long row = (long long)hh * a.Lq + qi_c;
  auto load_rows = [&]() {
    const bf16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh + (long long)qi_c * a.q.sl + 8 * g;
    const bf16_t* dp = a.dout.ptr + b * a.dout.sb + h * a.dout.sh + (long long)qi_c * a.dout.sl + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 qr = *(const bf16x8*)(qp + 16 * s);
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[s][e] = (bf16_t)((float)qr[e] * a.scale_p2);
      dof[s] = *(const bf16x8*)(dp + 16 * s);
    }
    const float Lraw = a.lse[row];
    neg_lse = (Lraw == RA_NEG_INF) ? RA_NEG_INF : -Lraw;  // fully masked row: P = 0
    neg_lse2 = neg_lse * kLog2e;
    neg_delta = -a.delta[row];
  };
  if (!DENSE) load_rows();
  int q_seg = 0, q_pre = 0;
  float slope = 0.f, slope2 = 0.f;  // slope2: in the units of the scores
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
    if (flags & RA_BIAS_ALIBI) {
      slope = bs.slopes[h];
      slope2 = slope * kLog2e / a.scale_res;
    }
  }
  WaveIds ids;
  if constexpr (GENERAL) ids.init(q_valid, q_seg, q_pre);
  bool use_list = false;
  const unsigned char* dmap = nullptr;
  if constexpr (DENSE) {
    if (bs.dense_map) dmap = dense_map_of(bs, b, h, a.H, a.Lq, a.Lk);
  }
  if constexpr (GENERAL) {
    use_list = ntiles <= kPairListTiles && ((flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX)) || dmap != nullptr);
    if (use_list)
      n = list_key_tiles<DENSE>(a.Lq, a.Lk, bs, kv_seg, kv_pre, dmap, q0, q_hi, ids, j_lo, n, s_red, s_flag, s_list);
  }
  n = __builtin_amdgcn_readfirstlane(n);
  j_lo = __builtin_amdgcn_readfirstlane(j_lo);
  if (n == 0 && p.acc != nullptr) return;  // contributes nothing
  if (DENSE) load_rows();
  const int n_piece = max(1, min(p.n_split, (n + p.chunk_tiles - 1) / p.chunk_tiles));
  if (split >= n_piece) return;
  const int i_lo = n * split / n_piece, i_hi = n * (split + 1) / n_piece;
  int every_test = 0;
  if constexpr (GENERAL) {
    if ((flags & RA_BIAS_ALIBI) && wave == 0) {
      lds.ramp[0][lane] = slope2 * (float)lane;
      lds.ramp[GENERAL][lane] = -slope2 * (float)lane;
    }
    if (!use_list && (flags & RA_BIAS_PREFIX)) every_test |= kTestPrefix;
    if ((flags & RA_BIAS_DENSE) && dmap == nullptr) every_test |= kTestDense;
  }
  TileLoader<D, kPairKeys, DL> ldk, ldv;
  ldk.init(a.k.ptr + b * a.k.sb + h * a.k.sh, a.k.sl, a.Lk, wave, lane);
  ldv.init(a.v.ptr + b * a.v.sb + h * a.v.sh, a.v.sl, a.Lk, wave, lane);
  auto issue_tile = [&](int j, int buf) {
    const int k0 = j * kPairKeys;
    ldk.issue(k0, RA_LDS_ADDR(&s_k[0][0]) + buf * TILE_BYTES, wave, lane);
    ldv.issue(k0, RA_LDS_ADDR(&s_v[0][0]) + buf * TILE_BYTES, wave, lane);
    if constexpr (GENERAL) {
      const int kk = min(k0 + lane, a.Lk - 1);
      if (kv_seg && wave == 0) global_to_lds4(kv_seg + kk, RA_LDS_ADDR(&s_seg[0][0]) + buf * (kPairKeys * 4));
      if (kv_pre && wave == 1) global_to_lds4(kv_pre + kk, RA_LDS_ADDR(&s_pre[0][0]) + buf * (kPairKeys * 4));
    }
  };

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
  const FragOffsets<D> fo(lane);
  const bool wave_on = qw < a.Lq;
  const bool alibi_on = GENERAL && (flags & RA_BIAS_ALIBI);
  const WaveTiles wt = wave_key_tiles(bs, q_off + qw, q_off + qw + 31, a.Lk);
  TileWalk<DENSE> walk;

  auto step = [&](auto buffer, int i) {
    constexpr int BUF = decltype(buffer)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's share of tile i is in LDS
    __syncthreads();                     // everyone's is, and nobody reads the other buffer any more
    const FragOffsets<D> fr_off = fo.opaque();
    const int j = walk.tile(), kt0 = j * kPairKeys;
    int tests = walk.tests();
    bool dead = !wave_on || !wt.live(j);
    unsigned cells = 0;
    if constexpr (DENSE) {
      if (tests & kTestDense) {
        cells = walk.cells() >> (4 * wave);
        dead = dead || !(cells & 5);
        if ((cells & 15) == 5) tests &= ~kTestDense;
      }
    }
    if (i + 1 < i_hi) {
      walk.next(i + 1);
      issue_tile(walk.tile(), BUF ^ 1);
    }
    if (dead) return;
    const bool one_side = alibi_on && (j < wt.past || j >= wt.future);
    if constexpr (GENERAL) {
      if (tests && wave_tests(tests, ids, s_seg[BUF], s_pre[BUF], j < wt.past, j > wt.future, lane)) return;
      if (alibi_on && !one_side) tests |= kTestAlibi;
    }
    if (!wt.plain(j)) tests |= kTestPos;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      // S^T first, then dP^T with the exp2 of S in its shadow: dP^T takes no registers while the terms
      // of a biased tile are evaluated
      constexpr int PF = KS < 3 ? KS : 3;  // operand fetches in flight ahead of the matrix instruction that uses them
      f32x16 S, zero;
      float neg_row = neg_lse2;  // added to the scores in the exponent
#pragma unroll
      for (int r = 0; r < 16; ++r) zero[r] = 0.f;
      auto nat_frag = [&](const char* tile, int ss) { return *(const bf16x8*)(tile + 32 * kb * ROWB + fr_off.nat(ss)); };
      __builtin_amdgcn_s_setprio(1);
      {
        bf16x8 fr[KS];
#pragma unroll
        for (int op = 0; op < PF; ++op) fr[op] = nat_frag(s_k[BUF], op);
        __builtin_amdgcn_sched_barrier(0);
        if (one_side) {
          const int at = opaque_lane(lane), l = at & 31, half = at >> 5;
          const float* ramp = lds.ramp[GENERAL && j >= wt.past] + 32 * kb + 4 * half;
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) {
            const f32x4 t = *(const f32x4*)(ramp + 8 * bb);
#pragma unroll
            for (int c = 0; c < 4; ++c) S[4 * bb + c] = t[c];
          }
          // (the bias and the logsumexp cancel before they are scaled)
          neg_row = fmaf(j < wt.past ? -slope : slope, (float)(q_off + qw + l - (kv_off + kt0)), neg_lse) * kLog2e;
          S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[0], qf[0], S, 0, 0, 0);
        } else {
          S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[0], qf[0], zero, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (PF < KS) {
          fr[PF] = nat_frag(s_k[BUF], PF);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int op = 1; op < KS; ++op) {
          if (op + PF < KS) fr[op + PF] = nat_frag(s_k[BUF], op + PF);
          S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], qf[op], S, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      if (tests) {
        const int at = opaque_lane(lane), g = at >> 5, qi = qw + (at & 31);
        TileBias tb;
        tb.flags = flags;
        tb.window = bs.window;
        tb.slope2 = slope2;
        tb.dense_mul = kLog2e / a.scale_res;
        const int var0 = kt0 + 32 * kb + 4 * g;
        tb.var_limit = a.Lk - var0;
        if (DENSE) {
          const float* head = bs.dense + b * bs.dense_sb + h * bs.dense_sh;
          tb.dense_vec = kt0 + kPairKeys <= a.Lk && ((((uintptr_t)head) | ((uintptr_t)bs.dense_sq << 2)) & 15) == 0;
          tb.dense = head + (long long)min(qi, a.Lq - 1) * bs.dense_sq + var0;
        }
        apply_terms<true, DENSE, GENERAL>(S, DENSE ? cell_tests(tests, (cells >> (2 * kb)) & 3) : tests, tb,
                                          (q_off + qi) - (kv_off + var0), q_seg, q_pre, &s_seg[GENERAL ? BUF : 0][32 * kb + 4 * g],
                                          &s_pre[GENERAL ? BUF : 0][32 * kb + 4 * g]);
      }
      f32x16 P;
#pragma unroll
      for (int r = 0; r < 16; ++r) P[r] = neg_delta;
      {
        bf16x8 fr[KS];
#pragma unroll
        for (int op = 0; op < PF; ++op) fr[op] = nat_frag(s_v[BUF], op);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int op = 0; op < KS; ++op) {
          if (op + PF < KS) fr[op + PF] = nat_frag(s_v[BUF], op + PF);
          P = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], dof[op], P, 0, 0, 0);
#pragma unroll
          for (int e = 16 * op / KS; e < 16 * (op + 1) / KS; ++e) {
            float x = fast_exp2(fmaf(S[e], a.scale_res, GENERAL ? neg_row : neg_lse2));
            asm volatile("" : "+v"(x));
            S[e] = x;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // dS in two groups of eight keys per lane: the second one is worked on while the matrix unit
      // multiplies with the first
      bf16x8 dsf[2];
      auto grad = [&](int ks, int e) {  // elements e, e + 1 of group ks
        bf16x2 pr;
        pr[0] = (bf16_t)(S[8 * ks + e] * P[8 * ks + e]);
        pr[1] = (bf16_t)(S[8 * ks + e + 1] * P[8 * ks + e + 1]);
        unsigned pw = __builtin_bit_cast(unsigned, pr);
        asm volatile("" : "+v"(pw));
        pr = __builtin_bit_cast(bf16x2, pw);
        dsf[ks][e] = pr[0];
        dsf[ks][e + 1] = pr[1];
      };
      auto k_frag = [&](int op) {
        const int ks = op / DB, db = op % DB;
        const lds_char* p0 = (const lds_char*)(s_k[BUF] + (32 * kb + 16 * ks) * ROWB + fr_off.tr(db, 0));
        const lds_char* p1 = (const lds_char*)(s_k[BUF] + (32 * kb + 16 * ks) * ROWB + fr_off.tr(db, 1));
        const bf16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p0);
        const bf16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p1);
        return __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
      };
      bf16x8 fr[2 * DB];
#pragma unroll
      for (int op = 0; op < (PF < 2 * DB ? PF : 2 * DB); ++op) fr[op] = k_frag(op);
#pragma unroll
      for (int e = 0; e < 8; e += 2) grad(0, e);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int op = 0; op < 2 * DB; ++op) {
        const int ks = op / DB, db = op % DB;
        if (op + PF < 2 * DB) fr[op + PF] = k_frag(op + PF);
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], dsf[ks], acc[db], 0, 0, 0);
        if (ks < 1) {
#pragma unroll
          for (int e = 4 * db / DB; e < 4 * (db + 1) / DB; ++e) grad(1, 2 * e);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (i_lo < i_hi) {
    walk.start(GENERAL && use_list, s_list, j_lo, i_lo, i_hi, every_test);
    issue_tile(walk.tile(), 0);
    for (int i = i_lo; i < i_hi; i += 2) {
      step(std::integral_constant<int, 0>{}, i);
      if (i + 1 < i_hi) step(std::integral_constant<int, 1>{}, i + 1);
    }
  }

  const auto* e = kernel_args<PairBwdArgs>(args_at);
  if (e->part_n != nullptr && split == 0 && tid == 0) e->part_n[hh * nqt + qt] = n_piece;
  if (!q_valid) return;
  float* fp = nullptr;  // fp32 destination: a share of the sum, or an accumulator
  if (n_piece > 1) fp = e->part + ((long long)split * ((long long)e->a.B * e->a.H * e->a.Lq) + row) * DL;
  else if (e->acc != nullptr) fp = e->acc + row * DL;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) {
      const int d0 = 32 * db + 8 * bb + 4 * g;
      f32x4 t;
#pragma unroll
      for (int c = 0; c < 4; ++c) t[c] = acc[db][4 * bb + c] * e->a.sm_scale;
      if (fp != nullptr) {
        if (n_piece == 1) t += *(const f32x4*)(fp + d0);
        *(f32x4*)(fp + d0) = t;
      } else {
        store4(e->out, e->out_dtype, b * e->out_sb + h * e->out_sh + (long long)qi * e->out_sl + d0, round_via(t, e->via_bf16));
      }
    }
}

// ------------------------------------------------------------------------------------------------
// dK / dV
// ------------------------------------------------------------------------------------------------
constexpr int kPairSlab = 128;      // keys per workgroup: 4 waves x 32
constexpr int kPairQueries = 32;    // queries per LDS tile
constexpr int kPairQListTiles = 2048;

// The query-side twin of list_key_tiles: the 32-query tiles that the workgroup's keys [k0, k_hi] meet.
template <bool DENSE>
RA_DEV int list_query_tiles(int Lq, int Lk, const BiasArgs& bs, const int* q_seg, const int* q_pre, const unsigned char* dmap,
                            int k0, int k_hi, const WaveIds& w, int j_lo, int n, int* s_red,
                            unsigned char* s_flag, ListEntry<DENSE>* s_list) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool seg_on = q_seg != nullptr, pre_on = q_pre != nullptr;
  if (lane == 0) {
    s_red[wave] = w.lo;
    s_red[4 + wave] = w.hi;
    s_red[8 + wave] = w.any;
    s_red[12 + wave] = w.all;
  }
  __syncthreads();
  const int kmin = min(min(s_red[0], s_red[1]), min(s_red[2], s_red[3]));
  const int kmax = max(max(s_red[4], s_red[5]), max(s_red[6], s_red[7]));
  const bool k_any = s_red[8] | s_red[9] | s_red[10] | s_red[11], k_all = s_red[12] & s_red[13] & s_red[14] & s_red[15];
  if (seg_on) {
    tile_ranges<kPairQueries, false>(q_seg, j_lo, 0, n, Lq, wave, lane, [&](int i, int qmin, int qmax) {
      s_flag[i] = (qmax < kmin || qmin > kmax) ? 0 : (qmin != qmax || kmin != kmax) ? 0x80 | kTestSegment : 0x80;  // 0x80: listed
    });
  } else {
    for (int i = tid; i < n; i += kPairThreads) s_flag[i] = 0x80;
  }
  if (pre_on) {
    __syncthreads();
    // up to the last tile with a query before the last key's position
    const int i_hi = min(n, floor_div(bs.kv_off + k_hi - 1 - bs.q_off, kPairQueries) + 1 - j_lo);
    tile_ranges<kPairQueries, true>(q_pre, j_lo, 0, i_hi, Lq, wave, lane, [&](int i, int all, int any) {
      const int qlo = bs.q_off + (j_lo + i) * kPairQueries, qhi = bs.q_off + min((j_lo + i + 1) * kPairQueries, Lq) - 1;
      const int c = prefix_class(qlo, qhi, bs.kv_off + k0, bs.kv_off + k_hi, any, all, k_any, k_all);
      const int f = s_flag[i];
      if (f && c) s_flag[i] = c == 2 ? 0 : f | kTestPrefix;
    });
  }
  if constexpr (DENSE) {
    if (dmap != nullptr) {
      __syncthreads();
      for (int i = tid; i < n; i += kPairThreads) {
        // the summary's cells of the four waves' keys, two bits each
        const int ncols = (Lk + kMapCell - 1) / kMapCell;
        unsigned cells = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int col = k0 / kMapCell + c;
          if (col * kMapCell <= k_hi) cells |= (dmap[(long long)(j_lo + i) * ncols + col] & 3u) << (2 * c);
        }
        if (!(cells & 0x55)) s_flag[i] = 0;
        else if ((cells & 0xaa) && s_flag[i]) s_flag[i] |= kTestDense;
        s_list[i] = cells;  // (until the entries are written)
      }
    }
  }
  __syncthreads();
  return compact_list<DENSE, kPairQListTiles / kPairThreads>(j_lo, n, dmap != nullptr, s_red, s_flag, s_list);
}

// 128 keys per workgroup, 32 per wave, two workgroups per compute unit: K operands and the dK / dV
// accumulators in registers; V, which a second (D = 128) or third (D = 64) wave per SIMD leaves no registers
// for, in LDS; 32-query tiles of Q and dO in two LDS buffers.  S = Q K^T: a lane owns one key and 16 queries, so
// that P and dS are the A operands of dV = P^T dO and dK = dS^T Q.  The rows' statistics (stat:
// -lse log2(e) / scale_res, then -delta, from pair_stat_kernel) are the accumulators' initial values.
// Three workgroups per compute unit at D = 64: 168 registers hold everything once V is in LDS.  With V in registers too 5
// (MODE 0) and 12 (MODE 1) of them spill, and a reload inside the loop waits for the tile loads that were just issued:
// causal + ALiBi, 4096, B=2, H=16, 240 us against 189; causal documents of 2175 in 48128, B=2, H=4, 636 against 531.
template <int DL, int MODE>
struct DkdvLds {
  static constexpr int ROWB = (DL <= 64 ? 64 : 128) * 2, TILE_BYTES = kPairQueries * ROWB;
  __attribute__((aligned(16))) float stat[2][2][MODE == 2 ? 64 : kPairQueries];  // (a 64-lane load writes 64 words)
  __attribute__((aligned(16))) int seg[MODE ? 2 : 1][64];
  __attribute__((aligned(16))) int pre[MODE ? 2 : 1][64];
  __attribute__((aligned(16))) char q[2][TILE_BYTES];
  __attribute__((aligned(16))) char dout[2][TILE_BYTES];
  __attribute__((aligned(16))) char v[kPairSlab * ROWB];
  ListEntry<MODE == 2> list[MODE ? kPairQListTiles : 1];
  unsigned char flag[MODE ? kPairQListTiles : 1];
  int red[20];
};
template <int DL, int MODE>
RA_DEV void dkdv_pair(const PairBwdArgs& p, int bid, DkdvLds<DL, MODE>& lds, int args_at) {
  constexpr bool GENERAL = MODE != 0;
  constexpr bool DENSE = MODE == 2;
  constexpr int D = DL <= 64 ? 64 : 128;  // row pitch of the LDS tiles
  constexpr int KS = DL / 16, DB = DL / 32;
  constexpr int ROWB = D * 2;
  constexpr int TILE_BYTES = kPairQueries * ROWB;
  const BwdArgs& a = p.a;
  auto &s_q = lds.q, &s_do = lds.dout;
  auto& s_v = lds.v;
  auto& s_stat = lds.stat;
  auto &s_seg = lds.seg, &s_pre = lds.pre;
  auto& s_list = lds.list;
  auto& s_flag = lds.flag;
  auto& s_red = lds.red;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int nkt = (a.Lk + kPairSlab - 1) / kPairSlab;
  int hh, split, kt;
  pair_decode(bid, a.B * a.H, nkt, p.n_split, p.group, hh, split, kt);
  kt = nkt - 1 - kt;  // under a causal mask the first keys have the most work
  const int b = hh / a.H, h = hh % a.H;
  const int k0 = kt * kPairSlab;
  const int kw = k0 + wave * 32;
  const int ki = kw + l32;
  const bool k_valid = ki < a.Lk;
  const int ki_c = min(ki, a.Lk - 1);
  const BiasArgs& bs = a.bias;
  const int flags = bs.flags;
  if constexpr (DENSE) {
    if (left_to_the_other<kPairThreads>(bs, b, h, a.H, a.Lq, a.Lk, s_red)) return;
  }
  const int q_off = bs.q_off, kv_off = bs.kv_off;

  const int ntiles = (a.Lq + kPairQueries - 1) / kPairQueries;
  const int k_hi = min(k0 + kPairSlab, a.Lk) - 1;
  int j_lo, j_hi;
  query_tile_range(flags, bs.window, kv_off + k0, kv_off + k_hi, q_off, ntiles, kPairQueries, j_lo, j_hi);
  int n = j_hi - j_lo;
  if (split > 0 && split * p.chunk_tiles >= n) return;

  bf16x8 kf[KS];
  auto load_rows = [&]() {
    const bf16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh + (long long)ki_c * a.k.sl + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 kr = *(const bf16x8*)(kp + 16 * s);
#pragma unroll
      for (int e = 0; e < 8; ++e) kf[s][e] = (bf16_t)((float)kr[e] * a.scale_p2);
    }
  };
  if (!DENSE) load_rows();
  int k_seg = 0, k_pre = 0;
  float slope2 = 0.f;
  const int* q_seg = nullptr;
  const int* q_pre = nullptr;
  if constexpr (GENERAL) {
    if (flags & RA_BIAS_SEGMENT) {
      k_seg = bs.kv_seg[b * bs.kv_seg_sb + ki_c];
      q_seg = bs.q_seg + b * bs.q_seg_sb;
    }
    if (flags & RA_BIAS_PREFIX) {
      k_pre = bs.kv_pre[b * bs.kv_pre_sb + ki_c];
      q_pre = bs.q_pre + b * bs.q_pre_sb;
    }
    if (flags & RA_BIAS_ALIBI) slope2 = bs.slopes[h] * kLog2e / a.scale_res;
  }
  WaveIds ids;
  if constexpr (GENERAL) ids.init(k_valid, k_seg, k_pre);
  bool use_list = false;
  const unsigned char* dmap = nullptr;
  if constexpr (DENSE) {
    if (bs.dense_map) dmap = dense_map_of(bs, b, h, a.H, a.Lq, a.Lk);
  }
  if constexpr (GENERAL) {
    use_list = ntiles <= kPairQListTiles && ((flags & (RA_BIAS_SEGMENT | RA_BIAS_PREFIX)) || dmap != nullptr);
    if (use_list)
      n = list_query_tiles<DENSE>(a.Lq, a.Lk, bs, q_seg, q_pre, dmap, k0, k_hi, ids, j_lo, n, s_red, s_flag, s_list);
  }
  n = __builtin_amdgcn_readfirstlane(n);
  j_lo = __builtin_amdgcn_readfirstlane(j_lo);
  if (n == 0 && p.acc != nullptr) return;  // contributes nothing
  if (DENSE) load_rows();
  const int n_piece = max(1, min(p.n_split, (n + p.chunk_tiles - 1) / p.chunk_tiles));
  if (split >= n_piece) return;
  const int i_lo = n * split / n_piece, i_hi = n * (split + 1) / n_piece;
  int every_test = 0;
  if constexpr (GENERAL) {
    if (!use_list && (flags & RA_BIAS_PREFIX)) every_test |= kTestPrefix;
    if ((flags & RA_BIAS_DENSE) && dmap == nullptr) every_test |= kTestDense;
  }
  TileLoader<D, kPairQueries, DL> ldq, ldo;
  ldq.init(a.q.ptr + b * a.q.sb + h * a.q.sh, a.q.sl, a.Lq, wave, lane);
  ldo.init(a.dout.ptr + b * a.dout.sb + h * a.dout.sh, a.dout.sl, a.Lq, wave, lane);
  // lanes 0..31 move -lse of a tile's rows, lanes 32..63 -delta; under a dense block two waves move one each
  const bool raw_stat = DENSE && p.stat == nullptr;  // a single step, which has no room for them: from lse and delta, per tile
  const float* stat = (raw_stat ? a.lse : p.stat) + (long long)hh * a.Lq;
  const float* stat_delta = raw_stat ? a.delta + (long long)hh * a.Lq : stat + (long long)a.B * a.H * a.Lq;
  const unsigned to_delta = (unsigned)(a.B * a.H) * (unsigned)a.Lq * 4;  // (with a row's 124 bytes below 2^32: plan_dkdv_pair)
  auto issue_tile = [&](int j, int buf) {
    const int r0 = j * kPairQueries;
    ldq.issue(r0, RA_LDS_ADDR(&s_q[0][0]) + buf * TILE_BYTES, wave, lane);
    ldo.issue(r0, RA_LDS_ADDR(&s_do[0][0]) + buf * TILE_BYTES, wave, lane);
    const int row = min(opaque_lane(lane) & 31, a.Lq - 1 - r0);
    if constexpr (DENSE) {
      if (wave == 0) global_to_lds4_s(stat + r0, 4 * row, RA_LDS_ADDR(&s_stat[0][0][0]) + buf * 512);
      if (wave == 3) global_to_lds4_s(stat_delta + r0, 4 * row, RA_LDS_ADDR(&s_stat[0][1][0]) + buf * 512);
    } else if (wave == 0) {
      global_to_lds4_s(stat + r0, 4 * row + (lane >= 32 ? to_delta : 0u), RA_LDS_ADDR(&s_stat[0][0][0]) + buf * (2 * kPairQueries * 4));
    }
    if constexpr (GENERAL) {
      if (q_seg && wave == 1) global_to_lds4_s(q_seg + r0, 4 * row, RA_LDS_ADDR(&s_seg[0][0]) + buf * 256);
      if (q_pre && wave == 2) global_to_lds4_s(q_pre + r0, 4 * row, RA_LDS_ADDR(&s_pre[0][0]) + buf * 256);
    }
  };

  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[db][r] = dv[db][r] = 0.f;
  const FragOffsets<D> fo(lane);
  const bool wave_on = kw < a.Lk;
  const bool alibi_on = GENERAL && (flags & RA_BIAS_ALIBI);
  const float lse_mul = -kLog2e / a.scale_res;
  WaveTiles wt;
  {
    const int klo_w = kv_off + kw, khi_w = kv_off + kw + 31, pos_flags = flags & ~RA_BIAS_PREFIX;  // (prefix: tested for by itself)
    int hi;
    query_tile_range(pos_flags, bs.window, klo_w, khi_w, q_off, ntiles, kPairQueries, wt.live_lo, hi);
    wt.live_n = hi - wt.live_lo;
    query_tile_plain_range(pos_flags, bs.window, klo_w, khi_w, q_off, a.Lq / kPairQueries, kPairQueries, wt.plain_lo, hi);
    wt.plain_n = hi - wt.plain_lo;
    wt.sides<kPairQueries>(klo_w, khi_w, q_off);
  }
  TileWalk<DENSE> walk;

  auto step = [&](auto buffer, int i) {
    constexpr int BUF = decltype(buffer)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's share of tile i is in LDS
    __syncthreads();                     // everyone's is, and nobody reads the other buffer any more
    const FragOffsets<D> fr_off = fo.opaque();
    const int j = walk.tile(), qt0 = j * kPairQueries;
    int tests = walk.tests();
    bool dead = !wave_on || !wt.live(j);
    if constexpr (DENSE) {
      if (tests & kTestDense) {
        const unsigned cell = (walk.cells() >> (2 * wave)) & 3;
        dead = dead || !(cell & kMapLive);
        if (cell == kMapLive) tests &= ~kTestDense;
      }
    }
    if (i + 1 < i_hi) {
      walk.next(i + 1);
      issue_tile(walk.tile(), BUF ^ 1);
    }
    if (dead) return;
    const bool one_side = alibi_on && (j < wt.past || j >= wt.future);
    if constexpr (GENERAL) {
      if (tests && wave_tests(tests, ids, s_seg[BUF], s_pre[BUF], j >= wt.future, j < wt.past - 1, lane)) return;
      if (alibi_on && !one_side) tests |= kTestAlibi;
    }
    if (!wt.plain(j)) tests |= kTestPos;
    constexpr int PF = KS < 3 ? KS : 3;  // operand fetches in flight ahead of the matrix instruction that uses them
    f32x16 S;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) {
      const f32x4 t = *(const f32x4*)&s_stat[BUF][0][8 * bb + 4 * g];
#pragma unroll
      for (int c = 0; c < 4; ++c) S[4 * bb + c] = t[c];
    }
    if (raw_stat) {
#pragma unroll
      for (int r = 0; r < 16; ++r) S[r] = (S[r] == RA_NEG_INF) ? RA_NEG_INF : S[r] * lse_mul;
    }
    if (one_side) {
      const int at = opaque_lane(lane), l = at & 31;
      const float s = j < wt.past ? slope2 : -slope2;
      S = alibi_one_side(S, alibi_index(0, l, at >> 5), s, -s * (float)((kv_off + kw + l) - (q_off + qt0)), at >> 5);
    }
    auto nat_frag = [&](const char* tile, int ss) { return *(const bf16x8*)(tile + fr_off.nat(ss)); };
    __builtin_amdgcn_s_setprio(1);
    {
      bf16x8 fr[KS];
#pragma unroll
      for (int op = 0; op < PF; ++op) fr[op] = nat_frag(s_q[BUF], op);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int op = 0; op < KS; ++op) {
        if (op + PF < KS) fr[op + PF] = nat_frag(s_q[BUF], op + PF);
        S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], kf[op], S, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if (tests) {
      const int at = opaque_lane(lane), g = at >> 5, ki = kw + (at & 31);
      TileBias tb;
      tb.flags = flags;
      tb.window = bs.window;
      tb.slope2 = slope2;
      tb.dense_mul = kLog2e / a.scale_res;
      tb.var_limit = a.Lq - (qt0 + 4 * g);
      if (DENSE) {
        // whole tiles whose lanes' offsets (four rows at most) fit 32 bits; else, in elements, from the lane's own first row on
        const int key = min(ki, a.Lk - 1);
        tb.dense = bs.dense + b * bs.dense_sb + h * bs.dense_sh + (long long)qt0 * bs.dense_sq;
        tb.dense_vs = bs.dense_sq;
        tb.dense_vec = qt0 + kPairQueries <= a.Lq && bs.dense_sq < (1 << 27);
        tb.dense_lane = tb.dense_vec ? 4 * (4 * g * (unsigned)bs.dense_sq + key) : key;
        if (!tb.dense_vec) tb.dense += (long long)(g && qt0 + 4 < a.Lq ? 4 : 0) * bs.dense_sq;
      }
      apply_terms<false, DENSE, GENERAL>(S, tests, tb, (q_off + qt0 + 4 * g) - (kv_off + ki), k_seg, k_pre,
                                         &s_seg[GENERAL ? BUF : 0][4 * g], &s_pre[GENERAL ? BUF : 0][4 * g]);
    }
    // dP with exp2(S) in its shadow
    bf16x8 pf[2], dsf[2];
    f32x16 P;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) {
      const f32x4 t = *(const f32x4*)&s_stat[BUF][1][8 * bb + 4 * g];
#pragma unroll
      for (int c = 0; c < 4; ++c) P[4 * bb + c] = t[c];
    }
    if (raw_stat) {
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const f32x4 t = *(const f32x4*)&s_stat[BUF][0][8 * bb + 4 * g];
#pragma unroll
        for (int c = 0; c < 4; ++c) P[4 * bb + c] = (t[c] == RA_NEG_INF) ? 0.f : -P[4 * bb + c];
      }
    }
    {
      bf16x8 fr[KS], vr[KS];
      auto v_op = [&](int op) { return *(const bf16x8*)(s_v + 32 * wave * ROWB + fr_off.nat(op)); };
      constexpr int PFV = 2;
#pragma unroll
      for (int op = 0; op < PFV; ++op) {
        fr[op] = nat_frag(s_do[BUF], op);
        vr[op] = v_op(op);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int op = 0; op < KS; ++op) {
        if (op + PFV < KS) {
          fr[op + PFV] = nat_frag(s_do[BUF], op + PFV);
          vr[op + PFV] = v_op(op + PFV);
        }
        P = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[op], vr[op], P, 0, 0, 0);
#pragma unroll
        for (int e = 8 * op / KS; e < 8 * (op + 1) / KS; ++e) {
          const int r = 2 * e;
          float x0 = fast_exp2(S[r] * a.scale_res), x1 = fast_exp2(S[r + 1] * a.scale_res);
          bf16x2 pr;
          pr[0] = (bf16_t)x0;
          pr[1] = (bf16_t)x1;
          unsigned pw = __builtin_bit_cast(unsigned, pr);
          asm volatile("" : "+v"(x0), "+v"(x1), "+v"(pw));
          pr = __builtin_bit_cast(bf16x2, pw);
          S[r] = x0;
          S[r + 1] = x1;
          pf[r >> 3][r & 7] = pr[0];
          pf[r >> 3][(r & 7) + 1] = pr[1];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    auto tr_frag = [&](const char* tile, int op) {
      const int ks = op / DB, db = op % DB;
      const lds_char* p0 = (const lds_char*)(tile + 16 * ks * ROWB + fr_off.tr(db, 0));
      const lds_char* p1 = (const lds_char*)(tile + 16 * ks * ROWB + fr_off.tr(db, 1));
      const bf16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p0);
      const bf16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p1);
      return __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    // dV with dS = P (dP - delta) in its shadow, then dK
    {
      constexpr int NOP = 4 * DB;  // the dV products, then the dK products
      bf16x8 fr[NOP];
      auto t_op = [&](int op) { return tr_frag(op < 2 * DB ? s_do[BUF] : s_q[BUF], op % (2 * DB)); };
#pragma unroll
      for (int op = 0; op < PF; ++op) fr[op] = t_op(op);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int op = 0; op < NOP; ++op) {
        if (op + PF < NOP) fr[op + PF] = t_op(op + PF);
        const int o = op % (2 * DB), ks = o / DB, db = o % DB;
        if (op < 2 * DB) {
          dv[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pf[ks], fr[op], dv[db], 0, 0, 0);
#pragma unroll
          for (int e = 8 * op / (2 * DB); e < 8 * (op + 1) / (2 * DB); ++e) {
            const int r = 2 * e;
            bf16x2 pr;
            pr[0] = (bf16_t)(S[r] * P[r]);
            pr[1] = (bf16_t)(S[r + 1] * P[r + 1]);
            unsigned pw = __builtin_bit_cast(unsigned, pr);
            asm volatile("" : "+v"(pw));
            pr = __builtin_bit_cast(bf16x2, pw);
            dsf[r >> 3][r & 7] = pr[0];
            dsf[r >> 3][(r & 7) + 1] = pr[1];
          }
        } else {
          dk[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dsf[ks], fr[op], dk[db], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (i_lo < i_hi) {
    TileLoader<D, kPairSlab, DL> ldv;
    ldv.init(a.v.ptr + b * a.v.sb + h * a.v.sh, a.v.sl, a.Lk, wave, lane);
    ldv.issue(k0, RA_LDS_ADDR(&s_v[0]), wave, lane);
    walk.start(GENERAL && use_list, s_list, j_lo, i_lo, i_hi, every_test);
    issue_tile(walk.tile(), 0);
    for (int i = i_lo; i < i_hi; i += 2) {
      step(std::integral_constant<int, 0>{}, i);
      if (i + 1 < i_hi) step(std::integral_constant<int, 1>{}, i + 1);
    }
  }

  const auto* e = kernel_args<PairBwdArgs>(args_at);
  if (e->part_n != nullptr && split == 0 && tid == 0) e->part_n[hh * nkt + kt] = n_piece;
  // lane l32 holds column 32 db + l32 of rows kw + 4 g + 8 (r / 4) + r % 4
  const long long rows = (long long)e->a.B * e->a.H * e->a.Lk;
  if (n_piece == 1 && e->acc != nullptr) {
    // All loads of an array are issued before the first value is needed (see dkdv_kernel): a block of values, L=256, H=8, D=128,
    // 64.7 us with a load - add - store chain per element, 35.6 without; L=128, H=2, D=64, 36.4 and 19.8.
    auto add_to = [&](float* acc, const f32x16 (&x)[DB], float mul) {
      float* const at = acc + ((long long)hh * e->a.Lk + kw + 4 * g) * DL + l32;
      if (kw + 32 <= e->a.Lk) {  // (wave-uniform)
        float old[DB][16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int db = 0; db < DB; ++db) old[db][r] = at[(8 * (r / 4) + r % 4) * DL + 32 * db];
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int db = 0; db < DB; ++db) at[(8 * (r / 4) + r % 4) * DL + 32 * db] = fmaf(x[db][r], mul, old[db][r]);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = 8 * (r / 4) + r % 4;
          if (kw + 4 * g + row >= e->a.Lk) continue;
#pragma unroll
          for (int db = 0; db < DB; ++db) at[row * DL + 32 * db] += x[db][r] * mul;
        }
      }
    };
    add_to(e->acc, dk, e->a.sm_scale);
    add_to(e->acc2, dv, 1.0f);
    return;
  }
  if (n_piece > 1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = kw + 4 * g + 8 * (r / 4) + (r % 4);
      if (key >= e->a.Lk) continue;
      float* fp = e->part + ((long long)split * 2 * rows + (long long)hh * e->a.Lk + key) * DL + l32;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        fp[32 * db] = dk[db][r] * e->a.sm_scale;
        fp[rows * DL + 32 * db] = dv[db][r];
      }
    }
    return;
  }
  auto store = [&](auto like) {
    using T = decltype(like);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = kw + 4 * g + 8 * (r / 4) + (r % 4);
      if (key >= e->a.Lk) continue;
      const long long at = b * e->out_sb + h * e->out_sh + (long long)key * e->out_sl + l32;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        ((T*)e->out)[at + 32 * db] = (T)round_via(dk[db][r] * e->a.sm_scale, e->via_bf16);
        ((T*)e->out2)[at + 32 * db] = (T)round_via(dv[db][r], e->via_bf16);
      }
    }
  };
  if (e->out_dtype == RA_DTYPE_F32) store(float{});
  else if (e->out_dtype == RA_DTYPE_F16) store(_Float16{});
  else store(bf16_t{});
}

template <int DL, int MODE>
__global__ __launch_bounds__(kPairThreads, DL <= 64 ? 3 : 2) void dq_pair_kernel(const PairBwdArgs p) {
  __shared__ DqLds<DL, MODE> lds;
  dq_pair<DL, MODE>(p, blockIdx.x, lds, 0);
}
template <int DL, int MODE>
__global__ __launch_bounds__(kPairThreads, DL <= 64 ? 3 : 2) void dkdv_pair_kernel(const PairBwdArgs p) {
  __shared__ DkdvLds<DL, MODE> lds;
  dkdv_pair<DL, MODE>(p, blockIdx.x, lds, 0);
}
// Both in one launch, the kind with the longer workgroups first.
struct BothBwdArgs {
  PairBwdArgs dkdv, dq;
  int n_first;  // workgroups of the first kind; a multiple of eight where a head stays on its XCD (see pair_decode), for the second's too
  int dq_first;
};
template <int DL, int MODE>
__global__ __launch_bounds__(kPairThreads, DL <= 64 ? 3 : 2) void bwd_pair_kernel(const BothBwdArgs p) {
  __shared__ union Lds {
    DqLds<DL, MODE> dq;
    DkdvLds<DL, MODE> dkdv;
  } lds;
  const bool second = (int)blockIdx.x >= p.n_first;
  const int bid = second ? blockIdx.x - p.n_first : blockIdx.x;
  if (second == (p.dq_first != 0)) dkdv_pair<DL, MODE>(p.dkdv, bid, lds.dkdv, offsetof(BothBwdArgs, dkdv));
  else dq_pair<DL, MODE>(p.dq, bid, lds.dq, offsetof(BothBwdArgs, dq));
}

// What the dK / dV kernel adds to a row's scores: stat[row] = -lse log2(e) / scale_res (-inf for a row without
// any key: P = 0) and stat[rows + row] = -delta (0 there: its output, and delta with it, is NaN), with
// delta = rowsum(out * dout).  A dO that has to be converted (StatArgs::copy) is rounded and stored on the way.
// HBM bound.  A wave takes rows that lie next to each other: the heads of a token where heads are neighbours, tokens of a head
// else, up to four such loads in flight; the results are turned round in LDS.  A row after the other of one head, conversion by itself | so,
// us: 8192, B=2, H=16, D=128 40 | 33 (134 MB, 4.1 TB/s), 32768, H=16 71 | 66; fp32 2048, B=2, H=4, D=64 3.7 + 3.1 | 4.3, fp16 1047, B=2, H=8,
// D=96 5 + 4.1 | 5.8, D=80, 4096, H=5 4.3 + 4.3 | 5.2, and a launch less.
template <typename OutT, typename DoT, int D>
__global__ __launch_bounds__(256) void pair_stat_kernel(const StatArgs a) {
  constexpr int CPR = D == 96 ? 16 : D / 8;  // lanes per row (a power of two)
  constexpr int RW = 64 / CPR, P = 4;        // rows per wave and load, loads
  __shared__ float s_delta[4 * P * RW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.heads, lw = RW / G, LB = 4 * a.loads * lw;  // heads and tokens per wave and load, tokens per workgroup (powers of two)
  const int lb = blockIdx.x % a.n_l, rest = blockIdx.x / a.n_l, h0 = rest % a.n_h * G, b = rest / a.n_h;
  const int c = lane % CPR, hl = lane / CPR & (G - 1), lsub = lane / CPR / G, h = h0 + hl;
  typedef __attribute__((ext_vector_type(8))) DoT do8;
  typedef __attribute__((ext_vector_type(8))) OutT out8;
  const bool whole = a.dout_vec && a.dout_d % 8 == 0;  // a chunk of dO is there or not
  const int n = a.dout_d - 8 * c;                      // elements of this lane's
  const int co = min(c, D / 8 - 1), cd = min(c, max(a.dout_d / 8 - 1, 0));
  const OutT* op = (const OutT*)a.out + b * a.sb + h * a.sh + 8 * co;
  const DoT* dp = (const DoT*)a.dout + b * a.dsb + h * a.dsh;
  const long long first = ((long long)b * a.H + h0) * a.L;
  const int mine = lb * LB + threadIdx.x % LB;  // the token whose results this thread writes
  const long long row = first + (long long)(threadIdx.x / LB) * a.L + mine;
  const bool writes = (int)threadIdx.x < G * LB && mine < a.L;
  const float lse = writes ? a.lse[row] : 0.f;
  // (all loads first: what lies behind the end reads the last row again)
  do8 x[P];
  out8 y[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p >= a.loads) break;
    const long long l = min(lb * LB + (4 * p + wave) * lw + lsub, a.L - 1);
    if (whole) {
      x[p] = *(const do8*)(dp + l * a.dsl + 8 * cd);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[p][e] = dp[l * a.dsl + min(8 * c + e, a.dout_d - 1)];
    }
    y[p] = *(const out8*)(op + l * a.sl);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p >= a.loads) break;
    const int at = (4 * p + wave) * lw + lsub, li = lb * LB + at;
    bf16x8 dv;
#pragma unroll
    for (int e = 0; e < 8; ++e) dv[e] = (bf16_t)(e < n ? (float)x[p][e] : 0.f);
    if (a.copy != nullptr && li < a.L && c < D / 8) *(bf16x8*)(a.copy + (((long long)b * a.L + li) * a.H + h) * D + 8 * c) = dv;
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc += (float)y[p][e] * (float)dv[e];
    if (c >= D / 8) acc = 0.f;
#pragma unroll
    for (int o = CPR / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (c == 0) s_delta[hl * LB + at] = acc;
  }
  __syncthreads();
  if (!writes) return;
  const float delta = s_delta[threadIdx.x];
  const bool dead = lse == RA_NEG_INF;
  a.delta[row] = delta;
  a.stat[row] = dead ? RA_NEG_INF : -lse * kLog2e * a.inv_res;
  a.stat[(long long)a.B * a.H * a.L + row] = dead ? 0.f : -delta;
}

// Sum of the shares of rows that were split, stored in the gradient's dtype.  Grid dimension y, from `first` on: dK and dV, whose
// rows lie one after another in a share, then dQ.
template <int D>
__global__ __launch_bounds__(256) void pair_sum_kernel(const BothBwdArgs both, int first) {
  constexpr int CPR = D / 4;
  static_assert(kPairSlab == kPairRows, "shares of as many rows");
  const int which = blockIdx.y + first;
  const PairBwdArgs& p = which < 2 ? both.dkdv : both.dq;
  const int H = p.a.H, L = which < 2 ? p.a.Lk : p.a.Lq, n_out = which < 2 ? 2 : 1;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long rows = (long long)p.a.B * H * L, row = i / CPR;
  if (row >= rows) return;
  const int c = (int)(i % CPR), li = (int)(row % L);
  const long long hh = row / L;
  const int n_piece = p.part_n[hh * ((L + kPairRows - 1) / kPairRows) + li / kPairRows];
  if (n_piece <= 1) return;  // written by its only workgroup
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < n_piece; ++s) x += *(const f32x4*)(p.part + (((long long)s * n_out + (which & 1)) * rows + row) * D + 4 * c);
  store4(which == 1 ? p.out2 : p.out, p.out_dtype, (hh / H) * p.out_sb + (hh % H) * p.out_sh + (long long)li * p.out_sl + 4 * c,
         round_via(x, p.via_bf16));
}

// The kernels of a head dim: a multiple of 32, dense blocks at 64 and 128 only.
template <typename Launch>
static hipError_t with_dim(int D, int mode, Launch launch) {
  if (mode < 0 || mode > 2 || (mode == 2 && D != 64 && D != 128)) return hipErrorInvalidValue;
  switch (D) {
    case 32: return launch(std::integral_constant<int, 32>{});
    case 64: return launch(std::integral_constant<int, 64>{});
    case 96: return launch(std::integral_constant<int, 96>{});
    case 128: return launch(std::integral_constant<int, 128>{});
  }
  return hipErrorInvalidValue;
}

// dkdv, dq: nullptr for none
template <int D, int MODE>
static hipError_t launch_bwd_pair_dm(const PairBwdArgs* dkdv, const PairBwdArgs* dq, hipStream_t stream) {
  auto tiles = [](int L) { return (L + kPairRows - 1) / kPairRows; };
  const int n_dkdv = dkdv ? dkdv->a.B * dkdv->a.H * dkdv->n_split * tiles(dkdv->a.Lk) : 0;
  const int n_dq = dq ? dq->a.B * dq->a.H * dq->n_split * tiles(dq->a.Lq) : 0;
  const dim3 block(kPairThreads);
  if (dkdv && dq) {
    const bool dq_first = dq->chunk_tiles > dkdv->chunk_tiles;
    const BothBwdArgs p{*dkdv, *dq, dq_first ? n_dq : n_dkdv, dq_first};
    hipLaunchKernelGGL((bwd_pair_kernel<D, MODE>), dim3((unsigned)(n_dkdv + n_dq)), block, 0, stream, p);
  } else if (dkdv) {
    hipLaunchKernelGGL((dkdv_pair_kernel<D, MODE>), dim3((unsigned)n_dkdv), block, 0, stream, *dkdv);
  } else {
    hipLaunchKernelGGL((dq_pair_kernel<D, MODE>), dim3((unsigned)n_dq), block, 0, stream, *dq);
  }
  hipError_t e = hipGetLastError();
  const bool sum_dkdv = dkdv && dkdv->n_split > 1, sum_dq = dq && dq->n_split > 1;
  if (e != hipSuccess || !(sum_dkdv || sum_dq)) return e;
  const PairBwdArgs& any = dkdv ? *dkdv : *dq;
  const long long n = (long long)any.a.B * any.a.H * std::max(sum_dkdv ? any.a.Lk : 0, sum_dq ? any.a.Lq : 0) * (D / 4);
  const BothBwdArgs p{sum_dkdv ? *dkdv : *dq, sum_dq ? *dq : *dkdv, 0, 0};
  hipLaunchKernelGGL((pair_sum_kernel<D>), dim3((unsigned)((n + 255) / 256), (unsigned)(2 * sum_dkdv + sum_dq)), block, 0, stream, p,
                     sum_dkdv ? 0 : 2);
  return hipGetLastError();
}

hipError_t launch_bwd_pair(const PairBwdArgs* dkdv, const PairBwdArgs* dq, int D, int mode, hipStream_t stream) {
  return with_dim(D, mode, [&](auto d) {
    if (mode == 2) {
      if constexpr (d.value == 64 || d.value == 128) return launch_bwd_pair_dm<d.value, 2>(dkdv, dq, stream);
    }
    return mode == 1 ? launch_bwd_pair_dm<d.value, 1>(dkdv, dq, stream) : launch_bwd_pair_dm<d.value, 0>(dkdv, dq, stream);
  });
}

template <typename OutT, typename DoT, int D>
static hipError_t launch_pair_stat_d(StatArgs a, hipStream_t stream) {
  constexpr int RW = 64 / (D == 96 ? 16 : D / 8);
  a.heads = 1;
  while (a.sh < a.sl && 2 * a.heads <= RW && a.H % (2 * a.heads) == 0) a.heads *= 2;
  // (four loads a wave where that still gives every compute unit two workgroups)
  a.loads = (long long)a.B * a.H * a.L >= 512 * 16 * RW ? 4 : 1;
  const int tokens = 4 * a.loads * RW / a.heads;
  a.n_l = (a.L + tokens - 1) / tokens;
  a.n_h = a.H / a.heads;
  hipLaunchKernelGGL((pair_stat_kernel<OutT, DoT, D>), dim3((unsigned)((long long)a.B * a.n_h * a.n_l)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_pair_stat(const StatArgs& a, int out_f32, int dout_dtype, int D, hipStream_t stream) {
  return with_dim(D, 0, [&](auto d) {
    auto with_out = [&](auto out) {
      using OutT = decltype(out);
      if (dout_dtype == RA_DTYPE_F32) return launch_pair_stat_d<OutT, float, d.value>(a, stream);
      if (dout_dtype == RA_DTYPE_F16) return launch_pair_stat_d<OutT, _Float16, d.value>(a, stream);
      return launch_pair_stat_d<OutT, bf16_t, d.value>(a, stream);
    };
    return out_f32 ? with_out(float{}) : with_out(bf16_t{});
  });
}

template <int D>
static hipError_t launch_fwd_pair_d(const PairFwdArgs& a, int mode, hipStream_t stream) {
  const int nqt = (a.Lq + kPairRows - 1) / kPairRows;
  dim3 grid((unsigned)(a.B * a.H * a.n_split * nqt)), block(kPairThreads);
  if (mode == 2) {
    if constexpr (D == 64 || D == 128) hipLaunchKernelGGL((fwd_pair_kernel<D, 2>), grid, block, 0, stream, a);
  } else if (mode == 1) {
    hipLaunchKernelGGL((fwd_pair_kernel<D, 1>), grid, block, 0, stream, a);
  } else {
    hipLaunchKernelGGL((fwd_pair_kernel<D, 0>), grid, block, 0, stream, a);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.part_o == nullptr) return e;
  const long long n = (long long)a.B * a.H * a.Lq * (D / 4);
  hipLaunchKernelGGL((pair_combine_kernel<D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_fwd_pair(const PairFwdArgs& a, int D, int mode, hipStream_t stream) {
  return with_dim(D, mode, [&](auto d) { return launch_fwd_pair_d<d.value>(a, mode, stream); });
}

}  // namespace ra
