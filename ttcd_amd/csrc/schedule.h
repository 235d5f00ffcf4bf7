// schedule.h - tile/phase schedule of the dual-window attention kernels.
//
// Shared verbatim by the gfx950 kernels (attn.hip) and by the host-side
// replay ttcd_attn_schedule_coverage (api.hip), so the CPU test suite proves
// the exact iteration logic the GPU runs: every (query, key) pair inside a
// window is folded into that window's output exactly once.
//
// Geometry. A workgroup has 4 wavefronts; each wavefront owns R consecutive
// query rows (r0..r0+R-1), R = Schedule::rows: 32 rows of one query head, or,
// for an even GQA group, 16 rows of each of two query heads of the group (the
// 32 columns of one score MFMA; both heads read the same K/V, so every MFMA
// operand is shared). A workgroup owns 4R tokens. Keys are swept in tiles of
// kBlockN = 64, tile n covering keys [64n - kshift, 64n - kshift + 63], from
// the tile holding the workgroup's last diagonal downward (the same
// backward-from-diagonal order as profiling/fused_dual_attn.py:91,119,151,
// 176,191); every wave of the workgroup steps through the same tiles.
//
// Phases. A band {lo, hi} selects keys with lo <= i - j < hi. The dual kernel
// runs phase 1 = student band {0, ws} and then phase 2 = far band {ws, wt}
// on ONE online-softmax accumulator: when a wave finishes phase 1 it writes
// the student output from the accumulator and keeps going, so the teacher
// output is the same accumulator after phase 2. This replaces the two
// accumulators of the reference kernel (fused_dual_attn.py:68-73) and its
// five segments A-E (:90-232) with a schedule that never needs a second
// output accumulator in registers.
//
// The single-accumulator order needs every wave's "mixed" keys (keys that
// are student-visible for some of its rows and far for others: the R-1 keys
// [r0-ws+1, r0+R-1-ws]) to sit in one tile, so that all phase-1 tiles of a
// wave precede all of its phase-2-only tiles. With r0 a multiple of R this
// holds iff tile starts are congruent to (1 - ws) or (-ws) modulo R, so
// kshift = ws mod 32 serves both geometries (0 for single-band calls). It
// also makes the waves of each aligned 64-row run share their mixed tile:
// one repeated tile per 16-row-wave workgroup (two for 32-row waves) when
// ws mod 64 < 32. The tile boundaries, and with them every row's order of
// accumulation, are the same in both geometries.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define TTCD_HD __host__ __device__ __forceinline__
#else
#define TTCD_HD inline
#endif

namespace ttcd {

constexpr int kBlockN = 64;    // keys per K/V tile
constexpr int kWaveRows = 32;  // query columns per wavefront (score MFMA columns)
constexpr int kWaves = 4;      // wavefronts per workgroup
constexpr int kBlockM = kWaveRows * kWaves;  // query tokens per workgroup, one head per wave

struct Band {
  int lo;  // inclusive lower bound of i - j
  int hi;  // exclusive upper bound of i - j
};

// Floor division for b > 0 and any a (C++ '/' truncates toward zero).
TTCD_HD int floordiv(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

struct Schedule {
  int T;       // sequence length (queries == keys)
  int dual;    // 1: phase 1 = student, phase 2 = far band; 0: phase 1 only
  Band p1;     // phase-1 band
  Band p2;     // phase-2 band (dual only; empty when lo == hi)
  int kshift;  // tile n starts at key 64n - kshift
  int rows;    // query rows (tokens) per wavefront: 32, or 16 of each of two heads

  TTCD_HD int tile_of(int j) const { return floordiv(j + kshift, kBlockN); }
  TTCD_HD int tile_start(int n) const { return n * kBlockN - kshift; }

  // Tile range [n_lo, n_hi] swept by the workgroup owning tokens t0..t_last.
  // Returns false when no row of the workgroup has a key in any band.
  TTCD_HD bool wg_range(int t0, int t_last, int* n_hi, int* n_lo) const {
    const int top = t_last - p1.lo;  // phase 1 always has the smallest lo
    const int widest = (dual && p2.lo < p2.hi) ? p2.hi : p1.hi;
    int bottom = t0 - widest + 1;
    if (bottom < 0) bottom = 0;
    if (top < 0 || top < bottom) return false;
    *n_hi = tile_of(top);
    *n_lo = tile_of(bottom);
    return true;
  }
};

// Does tile [j0, j0+63] hold a key of band b for some row of the wave r0..r0+R-1?
TTCD_HD bool wave_touches(int r0, int R, Band b, int j0) {
  return b.lo < b.hi && j0 + kBlockN - 1 >= r0 - b.hi + 1 && j0 <= r0 + R - 1 - b.lo;
}

// Is every (row, key) pair of the tile inside band b (no mask needed)?
TTCD_HD bool wave_full(int r0, int R, Band b, int j0) {
  return j0 >= 0 && r0 - (j0 + kBlockN - 1) >= b.lo && r0 + R - 1 - j0 < b.hi;
}

// Is this the wave's last tile of band b in the backward sweep?
TTCD_HD bool wave_last(int r0, Band b, int j0) {
  return j0 <= r0 - b.hi + 1 || j0 <= 0;
}

// Per-element visibility used by masked tiles.
TTCD_HD bool visible(int i, int j, Band b, int T) {
  const int d = i - j;
  return d >= b.lo && d < b.hi && j >= 0 && j < T;
}

// Slots. A workgroup sweeps a sequence of slots, one tile per slot. For the
// dual kernel each distinct "mixed" tile of its waves (a tile holding both
// student and far keys of a wave, at most one per wave) appears twice in a
// row: in the first slot its waves fold the student keys and then write the
// student output; in the repeated slot they fold the far keys. Waves whose
// mixed tile it is not skip the repeated slot. Every wave therefore carries
// one accumulator and one pending P^T between phases, as in the band kernel.
constexpr int kMaxDup = kWaves;
constexpr int kNoTile = -0x7fffffff - 1;

// All loops below have compile-time trip counts and static indices, so on the
// GPU the plan lives in scalar registers (no scratch memory).
struct SlotPlan {
  int n_hi;            // first (highest) tile
  int count;           // tiles n_hi .. n_hi - count + 1
  int ndup;            // repeated (mixed) tiles
  int dup[kMaxDup];    // their tile indices, descending, among unused entries (kNoTile)

  TTCD_HD int slots() const { return count + ndup; }

  // Tile of slot k and whether it is a repeat.
  TTCD_HD int tile(int k, bool* repeat) const {
    int n = n_hi - k;
    int before = 0;       // repeats already placed
    int rep_tile = kNoTile;
#pragma unroll
    for (int i = 0; i < kMaxDup; ++i) {
      if (dup[i] != kNoTile) {
        const int first = n_hi - dup[i] + before;  // slot of dup[i]'s first pass
        if (k == first + 1) rep_tile = dup[i];
        if (k > first + 1) n += 1;
        before += 1;
      }
    }
    *repeat = rep_tile != kNoTile;
    return *repeat ? rep_tile : n;
  }
};

// The wave's mixed tile, or kNoTile when it has none.
TTCD_HD int wave_mixed_tile(const Schedule& sc, int r0) {
  if (!sc.dual) return kNoTile;
  int lowest = r0 - sc.p1.hi + 1;  // lowest student key of the wave
  if (lowest < 0) lowest = 0;
  const int n = sc.tile_of(lowest);
  const int j0 = sc.tile_start(n);
  return (wave_touches(r0, sc.rows, sc.p1, j0) && wave_touches(r0, sc.rows, sc.p2, j0)) ? n
                                                                                   : kNoTile;
}

// Slot plan of a workgroup whose wave w starts at row r0_of_wave(w), rising
// with w (rows >= T are idle waves), and whose tiles are n_hi down to n_lo.
// A later wave's mixed tile is never a lower one, and the waves without one
// (no far key yet, or no row) are the first or the last of the workgroup: the
// last wave's tile first, equal neighbours dropped, is the descending list.
template <typename R0>
TTCD_HD SlotPlan make_slot_plan(const Schedule& sc, R0 r0_of_wave, int n_hi, int n_lo) {
  SlotPlan sp;
  sp.n_hi = n_hi;
  sp.count = n_hi - n_lo + 1;
  sp.ndup = 0;
  int prev = kNoTile;
#pragma unroll
  for (int i = 0; i < kMaxDup; ++i) {
    const int r0 = r0_of_wave(kMaxDup - 1 - i);
    int n = r0 < sc.T ? wave_mixed_tile(sc, r0) : kNoTile;
    n = (n >= n_lo && n <= n_hi) ? n : kNoTile;
    sp.dup[i] = (n == prev) ? kNoTile : n;
    prev = n;
    sp.ndup += sp.dup[i] != kNoTile;
  }
  return sp;
}

// What a wave folds in a slot: nothing, one band (mask chosen by wave_full),
// the student part of its mixed tile (then writes the student output) or the
// far part (repeat slot).
enum SlotAction { kSkip = 0, kBand1 = 1, kBand2 = 2, kStudentLast = 3, kFar = 4 };

TTCD_HD int slot_action(const Schedule& sc, int r0, int j0, bool repeat) {
  const bool in1 = wave_touches(r0, sc.rows, sc.p1, j0);
  const bool in2 = sc.dual && wave_touches(r0, sc.rows, sc.p2, j0);
  if (repeat) return (in1 && in2) ? kFar : kSkip;
  if (in1 && (in2 || (sc.dual && wave_last(r0, sc.p1, j0)))) return kStudentLast;
  return in1 ? kBand1 : (in2 ? kBand2 : kSkip);
}

// Per-wave slot actions in closed form: the tile-index ranges behind
// slot_action() and wave_full(), computed once per wave so that each slot
// costs a few branch-free scalar compares. Must agree with those functions
// on every tile of the sweep (checked by ttcd_attn_schedule_coverage).
struct WaveSlots {
  int n1a, n1b;  // tiles touched by phase 1 (empty: n1a > n1b)
  int n2a, n2b;  // tiles touched by phase 2 (dual kernel)
  int nl;        // tiles n <= nl end the student phase (wave_last)
  int f1a, f1b;  // tiles fully inside band 1
  int f2a, f2b;  // tiles fully inside band 2
  int dual;

  TTCD_HD WaveSlots(const Schedule& sc, int r0) : dual(sc.dual) {
    const int big = 0x3fffffff;
    auto range = [&](Band b, int* a, int* z) {
      if (b.lo < b.hi) {
        *a = sc.tile_of(r0 - b.hi + 1);
        *z = sc.tile_of(r0 + sc.rows - 1 - b.lo);
      } else {
        *a = big;
        *z = -big;
      }
    };
    range(sc.p1, &n1a, &n1b);
    if (sc.dual) {
      range(sc.p2, &n2a, &n2b);
    } else {
      n2a = big;
      n2b = -big;
    }
    const int lowest = r0 - sc.p1.hi + 1;
    nl = sc.tile_of(lowest > 0 ? lowest : 0);
    const int nz = sc.kshift > 0 ? 1 : 0;  // first tile with j0 >= 0
    auto full = [&](Band b, int* a, int* z) {
      const int lo_t = sc.tile_of(r0 + sc.rows + kBlockN - 1 - b.hi);  // j0 > r0 + R-1 - hi
      *a = lo_t > nz ? lo_t : nz;
      *z = sc.tile_of(r0 - (kBlockN - 1) - b.lo);                      // j0 <= r0 - 63 - lo
    };
    full(sc.p1, &f1a, &f1b);
    full(sc.p2, &f2a, &f2b);
  }

  // slot_action(sc, r0, tile_start(n), repeat), branch-free.
  TTCD_HD int act(int n, bool repeat) const {
    const bool in1 = (n >= n1a) & (n <= n1b);
    const bool in2 = (n >= n2a) & (n <= n2b);
    const int normal = in1 ? ((in2 | ((dual != 0) & (n <= nl))) ? kStudentLast : kBand1)
                           : (in2 ? kBand2 : kSkip);
    return repeat ? ((in1 & in2) ? kFar : kSkip) : normal;
  }
  // !wave_full(r0, band of action a, tile_start(n)) for an action that is not kSkip.
  TTCD_HD bool mask(int n, int a) const {
    const bool far = (a == kBand2) | (a == kFar);
    const int fa = far ? f2a : f1a, fz = far ? f2b : f1b;
    return !((n >= fa) & (n <= fz));
  }
};

// Slot words: everything the slot loop needs about slot k for one wave, in
// one 32-bit word. The kernel computes 64 consecutive slots at once (slot
// base + lane in each lane) and reads one word per slot back with
// v_readlane, so a slot costs a few scalar bit tests instead of evaluating
// the plan, the actions and the load bounds. Bits 0-5 are flags; bits 6+
// hold the tile index, so (word & ~63) is the tile's first key + kshift.
enum SlotWordBits : uint32_t {
  kWordLoad = 1u,      // slot exists: its K and V tiles are loaded
  kWordInterior = 2u,  // tile keys all inside [0, T): unclamped loads
  kWordActive = 4u,    // this wave folds keys (action != kSkip)
  kWordFar = 8u,       // ... of phase 2 (kBand2 or kFar), else of phase 1
  kWordLast = 16u,     // ... and it is kStudentLast (student output follows)
  kWordMask = 32u,     // ... and the scores need masking
};
constexpr int kWordTileShift = 6;
static_assert((1 << kWordTileShift) == kBlockN, "word & ~63 is the tile's key offset");

// The load part of the word of a slot over tile n (keys [0, T)).
TTCD_HD uint32_t slot_load_word(const Schedule& sc, int n, int T) {
  const int j0 = sc.tile_start(n);
  return (uint32_t)n << kWordTileShift | kWordLoad |
         (((j0 >= 0) & (j0 + kBlockN <= T)) ? kWordInterior : 0u);
}

// Word of slot k of plan sp (nslot slots) for the wave described by ws
// (wave_valid false: a wave without rows, which only loads), keys [0, T).
TTCD_HD uint32_t slot_word(const Schedule& sc, const SlotPlan& sp, const WaveSlots& ws,
                           int nslot, bool wave_valid, int T, int k) {
  bool repeat;
  int n = sp.tile(k, &repeat);
  const bool load = (k >= 0) & (k < nslot);
  n = load ? n : 0;
  const int act = (load & wave_valid) ? ws.act(n, repeat) : (int)kSkip;
  const bool far = (act == kBand2) | (act == kFar);
  uint32_t w = load ? slot_load_word(sc, n, T) : 0u;
  w |= act != kSkip ? kWordActive : 0u;
  w |= far ? kWordFar : 0u;
  w |= act == kStudentLast ? kWordLast : 0u;
  w |= (act != kSkip && ws.mask(n, act)) ? kWordMask : 0u;
  return w;
}

TTCD_HD int word_tile(uint32_t w) { return (int)(w >> kWordTileShift); }
TTCD_HD int word_j0(const Schedule& sc, uint32_t w) { return (int)(w & ~63u) - sc.kshift; }
TTCD_HD Band word_band(const Schedule& sc, uint32_t w) { return (w & kWordFar) ? sc.p2 : sc.p1; }

// Workgroup ids -> query blocks.
//
// The hardware deals consecutive workgroup ids round-robin to the kXcd XCDs
// (each with its own L2) and, inside an XCD, to its kXcdCus CUs, so id g is
// the (g / 8)-th workgroup of XCD g % 8, and the ones 32 apart there share a
// CU while every place is free. A call has npair = B * Hkv K/V heads, each
// with nqb query blocks (block nqb - 1 sweeps the most keys of a causal
// sequence) of ngrp workgroups. The blocks of a K/V head are cut into levels
// of seg consecutive blocks, the heaviest first, and the (level, head) items
// are dealt to the XCDs level by level: every XCD gets the same share of
// every level of every head (of every packed sequence too), while the
// workgroups of an item, which sweep nearly the same keys, share one L2.
// With npair a multiple of 8 the deal leaves an XCD whole heads; where these are
// not alike (sequences of a packed call, parts of a split one) it starts one
// XCD later every round. With another npair it runs forth and back, so that no
// XCD always gets the heavier items.
//
// Why: one contiguous run of (head, block) per XCD leaves the XCDs unequal
// when a head's run is split between them (causal heads, npair not a multiple
// of 8) or when packed sequences differ in length; the call then waits for
// one XCD. Where all workgroups sweep alike, or each has a CU to itself, a run
// per XCD is even to one workgroup, and items are not: such calls take runs
// when the deal would leave an XCD too many.
//
// Within an XCD the workgroups start heaviest first, except that the second
// one of each CU is taken so that a CU's two add up to about the same sweep:
// when all of them start at once nothing else evens the CUs out.
constexpr int kXcd = 8;
constexpr int kXcdCus = 32;

// n / d for 0 <= n < 2^31 by one 64-bit product: with m = ceil(2^(31+s) / d),
// 2^s >= d, n * m / 2^(31+s) rounds down to the quotient (Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994).
// A workgroup's start is a chain of scalar operations with nothing to hide
// it, and a division by a kernel argument is ~30 of them.
struct FastDiv {
  uint32_t d, m;
  int sh;

  TTCD_HD int quot(int n) const { return (int)(((uint64_t)(uint32_t)n * m) >> sh); }
};

TTCD_HD FastDiv make_fast_div(int d) {
  FastDiv f;
  int s = 0;
  while ((int64_t(1) << s) < d) ++s;
  f.d = (uint32_t)d;
  f.sh = 31 + s;
  f.m = (uint32_t)(((uint64_t(1) << f.sh) + d - 1) / d);
  return f;
}

// How the items go to the XCDs: always in the same direction, forth and back, or
// from one XCD later every round (a mask of the round). Or no items: one run of
// workgroups per XCD.
enum BlockDeal : int { kDealForth = 0, kDealSnake = 1, kDealTurn = 7 << 1, kDealRuns = 16 };

struct BlockMap {
  int nqb;               // query blocks per K/V head
  FastDiv npair, ngrp;   // K/V heads, workgroups per block
  FastDiv per;           // workgroups per item (runs: nqb)
  int seg;               // blocks per item (runs: workgroups per run)
  int items;             // (levels) * npair (runs: the XCDs whose run has one more)
  int rounds;            // items per XCD, rounded up (runs: workgroups, rounded up)
  int deal;

  TTCD_HD int per_xcd() const { return deal == kDealRuns ? rounds : rounds * (int)per.d; }
  TTCD_HD int launched() const { return kXcd * per_xcd(); }

  // Position in the heaviest-first order of an XCD's n workgroups of its
  // i-th started one.
  TTCD_HD int rank(int i) const {
    const int n = per_xcd();
    if (n <= kXcdCus) return i;
    const int both = n < 2 * kXcdCus ? n - kXcdCus : kXcdCus;  // CUs that start with two
    if (i >= kXcdCus) return i < kXcdCus + both ? kXcdCus + both - 1 - (i - kXcdCus) : i;
    // the CUs that start with two take the lighter of the first kXcdCus
    return i < both ? kXcdCus - both + i : i - both;
  }

  // The K/V head, query block and workgroup of the block that id g takes;
  // false when it takes none.
  TTCD_HD bool locate(int g, int* pair, int* qb, int* grp) const {
    const int x = g % kXcd;
    if (deal == kDealRuns) {
      const int i = g / kXcd, at = x * seg + (x < items ? x : items) + i;
      const int row = ngrp.quot(at);
      *grp = at - row * (int)ngrp.d;
      *pair = per.quot(row);
      *qb = nqb - 1 - (row - *pair * nqb);
      return i < seg + (x < items ? 1 : 0);
    }
    const int r = rank(g / kXcd);
    const int round = per.quot(r), in = r - round * (int)per.d;
    const int at = ((x + (round & deal >> 1)) & (kXcd - 1)) ^ (-(deal & round & 1) & (kXcd - 1));
    const int item = round * kXcd + at;
    const int level = npair.quot(item);
    const int blk = ngrp.quot(in);
    *pair = item - level * (int)npair.d;
    *grp = in - blk * (int)ngrp.d;
    *qb = nqb - 1 - (level * seg + blk);
    return item < items && *qb >= 0;
  }
};

// Blocks per item. A fixed-length call whose heads (alike of them in a row sweep
// alike: all, the ones of a sequence, or of a part) are a multiple of the XCDs
// gives each XCD whole heads. Otherwise: when every workgroup starts at once
// on a CU of its own, a run per XCD (the sweep of the heaviest workgroup is
// then the call, and it is fastest when the workgroups beside it fetch the same
// tiles); when they queue, 8 items per XCD of at least 4 blocks (whose
// workgroups share nearly all of their tiles) and at most 32 (about what an XCD
// runs at once). even: all blocks sweep about as many tiles.
//
// Measured against one contiguous run per XCD (us, kernel time): packed
// 12345 tokens in 9 sequences, 15/5 heads of 64, 153 -> 88; causal T = 8192,
// 15/5 heads of 64, 230 -> 162, T = 4500 80.7 -> 67.9; 16/8 heads of 128,
// T = 8192, 282 -> 271 and T = 4096 92.3 -> 87.2 (the order within an XCD
// alone); 4/2 heads of 64, T = 4096, with 64 items instead of 8 50.6 -> 54.1.
// Parts dealt from one XCD later every round instead of a part to an XCD (us, call
// time, full windows of cached keys): 2048 queries, 15/5 heads of 64, window 8192
// 111 -> 92; 4096, 4/2 heads, 80 -> 60.
//
// Runs also where the items leave a CU one workgroup more than it has to have, or
// an XCD 3 % more than its share (us, items / runs): 1900 queries on 2047 cached keys,
// 15/5 heads of 64, window 2048 (240 workgroups, 48 of them on one XCD) 44 / 32;
// causal, 4/4 heads of 128, T = 8192 (256 workgroups, the heavy ones on 4 XCDs
// beside each other) 134 / 129; windows 512 / 256, 15/5 heads of 64, T = 13000
// 64 / 59, 2 x 18432 155 / 148. 4/2 heads, T = 33000, windows 1024 / 512, has 2 %
// more and stays with items (53; with equal counts 61: its extra workgroups are
// the short first ones).
TTCD_HD BlockMap make_block_map(int npair, int alike, int nqb, int ngrp, bool packed,
                                bool even) {
  BlockMap m;
  m.nqb = nqb;
  m.npair = make_fast_div(npair);
  m.ngrp = make_fast_div(ngrp);
  const int64_t nwg = (int64_t)npair * nqb * ngrp, cus = kXcd * kXcdCus;
  const bool queued = nwg > cus;
  int seg = 32;
  auto few = [&](int items) { return (int64_t)npair * ((nqb + seg - 1) / seg) < items; };
  while (seg > 1 && few(seg > 4 ? 8 * kXcd : kXcd)) seg /= 2;
  const bool whole = !packed && alike % kXcd == 0;
  if (whole) seg = nqb;
  const int levels = (nqb + seg - 1) / seg;
  m.seg = (nqb + levels - 1) / levels;
  m.per = make_fast_div(m.seg * ngrp);
  m.items = levels * npair;
  m.rounds = (m.items + kXcd - 1) / kXcd;
  m.deal = npair % kXcd != 0 ? kDealSnake : alike % kXcd != 0 ? kDealTurn : kDealForth;
  // the workgroups of the fullest XCD, by items and by runs
  int dealt = 0;
  const int run = (int)((nwg + kXcd - 1) / kXcd);
  if (even && nwg <= 32 * cus) {
    int count[kXcd] = {};
    for (int i = 0; i < m.items; ++i) {
      const int round = i / kXcd, left = nqb - i / npair * m.seg;
      const int x = ((i ^ (-(m.deal & round & 1) & (kXcd - 1))) - (round & m.deal >> 1)) & (kXcd - 1);
      count[x] += (left < m.seg ? left : m.seg) * ngrp;
      dealt = count[x] > dealt ? count[x] : dealt;
    }
  }
  auto cu = [](int n) { return (n + kXcdCus - 1) / kXcdCus; };
  if ((!queued && !whole) || cu(dealt) > cu(run) || dealt > run + run / 32) {
    m.deal = kDealRuns;
    m.per = make_fast_div(nqb);
    m.seg = (int)(nwg / kXcd);
    m.items = (int)(nwg % kXcd);
    m.rounds = m.seg + (m.items > 0);
  }
  return m;
}

// Whether the rows q_off .. T - 1 have (nearly) their whole window of hi keys, so
// that every block sweeps about as many tiles: 5 % of the keys are missing at most.
TTCD_HD bool even_rows(int T, int q_off, int hi) {
  const int64_t first = q_off + 1, last = hi - 1;  // histories shorter than hi
  return first > last ||
         (last - first + 1) * (2 * (int64_t)hi - first - last) * 10 <= (int64_t)(T - q_off) * hi;
}

// Query rows per wavefront for a GQA group size (see Geometry): 16 rows of
// each of two heads for an even group, else 32 rows of one head.
#ifndef TTCD_PAIR_WAVES
#define TTCD_PAIR_WAVES 1
#endif
TTCD_HD int wave_rows(int gqa_group) {
  return (TTCD_PAIR_WAVES && gqa_group % 2 == 0) ? kWaveRows / 2 : kWaveRows;
}

// Query tokens swept by one workgroup.
TTCD_HD int wg_span_tokens(int gqa_group) { return kWaves * wave_rows(gqa_group); }

// Schedules built by the C ABI entry points (windows already validated), for
// wavefronts of `rows` query rows.
TTCD_HD Schedule make_dual_schedule(int T, int ws, int wt, int rows) {
  if (wt > T) wt = T;
  if (ws > wt) ws = wt;
  Schedule s;
  s.T = T;
  s.dual = 1;
  s.p1.lo = 0;
  s.p1.hi = ws;
  s.p2.lo = ws;
  s.p2.hi = wt;
  s.kshift = ws % kWaveRows;
  s.rows = rows;
  return s;
}

TTCD_HD Schedule make_band_schedule(int T, int lo, int hi, int rows) {
  if (hi > T) hi = T;
  if (lo > hi) lo = hi;
  Schedule s;
  s.T = T;
  s.dual = 0;
  s.p1.lo = lo;
  s.p1.hi = hi;
  s.p2.lo = hi;
  s.p2.hi = hi;
  s.kshift = 0;
  s.rows = rows;
  return s;
}

}  // namespace ttcd
