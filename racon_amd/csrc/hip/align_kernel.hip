// Global (NW) edit-distance alignment of racon overlaps on gfx950.
//
// Reproduces the alignment path racon gets from edlib (EDLIB_MODE_NW,
// EDLIB_TASK_PATH; src/overlap.cpp:205-224). The path is defined by a
// recursion on the target: a subproblem (query span, target span, score)
// whose stored columns would take (2*8+4) * ceil(|q|/64) * |t| < 1 MiB is
// traced back directly from its last cell, preferring up (insertion), then
// left (deletion), then the diagonal; a larger one is split at column
// |t|/2 at the first query row x where the forward score D(q[..x], t[..|t|/2))
// plus the reverse score of the rest equals the subproblem score (then x = -1,
// then x = |q|-1), and the two halves are solved in order.
//
// Scores are computed in a diagonal band (Band below) that starts from a
// guess of the distance and doubles until the banded distance fits it; every
// score on an optimal path is then exact, which gives edlib's path: banding
// only drops cells whose score cannot be on an optimal path, and every choice
// above reads cells on optimal paths.
//
// Myers' bit-vector recurrence runs on 64-row blocks, one block per lane, in
// an anti-diagonal pipeline along the band (see "banded runs" below): the
// recursion goes level by level, and the runs of a level share the lanes of
// the wave (or of a team of eight waves, for few long pairs). Bands too wide
// for the lanes are processed in strips of 64 blocks whose bottom carries
// pass through the slot. A persistent grid takes overlaps from a work queue
// ordered by size.
//
// Bound by the vector instructions of the steps. 12,000 pairs of 8 +- 4 kbp
// at 12% error: 404 M wave steps of 59 instructions and 81 ms in the strip
// form, 145 M steps of 34 and 36 ms in one-wave pairs, 16 ms with the longest
// in teams beside them; 61 pairs of 30 +- 9 kbp at 20% (teams): 140 -> 13.3
// ms; one pair of 1 kbp: 0.89 -> 0.40 ms.
#include <hip/hip_runtime.h>

#include "align_types.hpp"

namespace rh {

namespace {

constexpr int kWave = 64;
typedef uint64_t Word;

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// Orders this wave's memory operations: what its lanes wrote before, every
// lane of the wave reads after (waits for the outstanding ones).
__device__ __forceinline__ void wave_done() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

typedef uint32_t U4 __attribute__((ext_vector_type(4)));

// One Myers/Hyyro block step with horizontal input hin in {-1, 0, +1};
// *hp: the horizontal +1 deltas of the column.
__device__ __forceinline__ int block_step(Word& P, Word& M, Word eq, int hin, Word* hp) {
  const Word hin_neg = hin < 0 ? Word(1) : Word(0);
  const Word xv = eq | M;
  eq |= hin_neg;
  const Word xh = (((eq & P) + P) ^ P) | eq;
  Word ph = M | ~(xh | P);
  Word mh = P & xh;
  *hp = ph;
  int hout = 0;
  if (ph >> 63) hout = 1;
  if (mh >> 63) hout = -1;
  ph <<= 1;
  mh <<= 1;
  mh |= hin_neg;
  ph |= hin > 0 ? Word(1) : Word(0);
  P = mh | ~(xv | ph);
  M = ph & xv;
  return hout;
}

struct Seg {
  const uint8_t* q;  // query span
  const uint8_t* t;  // target span
  int ql;
  int tl;
  bool rev;  // read both spans from the end
  __device__ uint8_t qc(int i) const { return rev ? q[ql - 1 - i] : q[i]; }
  __device__ uint8_t tc(int j) const { return rev ? t[tl - 1 - j] : t[j]; }
};

// Match words of one block: for each of A, C, G, T the rows holding it (or
// past the query end, pad, which match everything), the rows holding N, and
// pad. A target A/C/G/T byte picks its word with two selects on its 2-bit
// code; other bytes take the N word or an exact byte compare (rare_eq).
struct Peq {
  Word a, c, g, t;  // match words of A, C, G, T (pad included)
  Word n;           // rows holding N
  Word pad;         // rows beyond the query
};

// 2-bit code of A, C, G, T (0..3) from the byte's bits 1 and 2; any byte
// maps to some code, so is_acgt checks the byte against the code's letter.
__device__ __forceinline__ int code2(int c) { return ((c >> 1) ^ (c >> 2)) & 3; }
__device__ __forceinline__ bool is_acgt(int c, int code) {
  return static_cast<int>((0x54474341u >> (8 * code)) & 0xffu) == c;  // "ACGT"
}

__device__ Peq build_peq(const Seg& g, int block) {
  Peq p{0, 0, 0, 0, 0, 0};
  Word lo = 0, hi = 0, acgt = 0;
  const int r0 = block * 64;
  for (int i = 0; i < 64; ++i) {
    const int r = r0 + i;
    const Word bit = Word(1) << i;
    if (r >= g.ql) {
      p.pad |= bit;
      continue;
    }
    const int c = g.qc(r);
    const int code = code2(c);
    if (is_acgt(c, code)) {
      acgt |= bit;
      if (code & 1) lo |= bit;
      if (code & 2) hi |= bit;
    } else if (c == 'N') {
      p.n |= bit;
    }
  }
  p.a = (acgt & ~lo & ~hi) | p.pad;
  p.c = (acgt & lo & ~hi) | p.pad;
  p.g = (acgt & ~lo & hi) | p.pad;
  p.t = (acgt & lo & hi) | p.pad;
  return p;
}

// Match word of an A/C/G/T byte from its 2-bit code.
__device__ __forceinline__ Word acgt_eq(const Peq& p, int code) {
  const Word e01 = (code & 1) ? p.c : p.a;
  const Word e23 = (code & 1) ? p.t : p.g;
  return (code & 2) ? e23 : e01;
}

// Match word for a target byte outside A/C/G/T/N (exact byte compare).
__device__ Word rare_eq(const Seg& g, int block, uint8_t c, Word pad) {
  Word w = pad;
  const int r0 = block * 64;
  for (int i = 0; i < 64; ++i) {
    const int r = r0 + i;
    if (r < g.ql && g.qc(r) == c) w |= Word(1) << i;
  }
  return w;
}

// Diagonal band of a (sub)problem: the cells (i, j) with lo <= i - j <= hi.
// A path through (i, j) costs at least |i - j| + |(ql - tl) - (i - j)|, so
// with d >= the subproblem's distance every optimal path lies inside
// band_for(ql, tl, d). Cells outside are not computed: a strip of blocks
// runs only over the columns where its rows meet the band, a strip that
// starts past column 0 begins from upper bounds (vertical deltas of +1 from
// max(row + 1, column + 1)), and a column the strip above did not compute
// feeds it a horizontal delta of +1. Every computed score is then an upper
// bound of the exact one, equal to it on every cell of an optimal path,
// which is all that the traceback and the split search read (a cell they
// look up outside the computed columns reads as kFar).
struct Band {
  int lo, hi;
};
constexpr int32_t kFar = 1 << 28;

__device__ __forceinline__ Band band_for(int ql, int tl, int d) {
  const int delta = ql - tl;
  const int ad = delta < 0 ? -delta : delta;
  const int slack = d >= ad ? (d - ad) / 2 : 0;
  return Band{min(0, delta) - slack, max(0, delta) + slack};
}

// The band of the reversed segment (row ql-1-i, column tl-1-j).
__device__ __forceinline__ Band band_reversed(Band b, int ql, int tl) {
  return Band{(ql - tl) - b.hi, (ql - tl) - b.lo};
}

// Columns [cs, ce] that strip k (rows k * 4096 .. + 64 * nbs - 1) computes.
__device__ __forceinline__ void strip_columns(const Seg& g, Band bd, int k, int nbs, int* cs,
                                              int* ce) {
  const int row_lo = k * kWave * 64;
  const int row_hi = min(g.ql, (k * kWave + nbs) * 64) - 1;
  *cs = max(0, row_lo - bd.hi);
  *ce = min(g.tl - 1, row_hi - bd.lo);
}

// Runs the bit-vector DP of seg over the columns of band bd in strips of 64
// blocks, one wave; for bands wider than the cyclic runs below hold. With stop >= 0
// (which must be the last column, tl - 1: the only column the recursion asks
// for), writes the scores of that column for rows 0..ql-1 into col, from each
// block's state after its last step (kFar for rows of a strip that does not
// reach it). With store, keeps the vertical and horizontal +1 deltas of every
// computed (column, block) for the traceback. Returns the score of the last
// cell (row ql-1, column tl-1) when stop < 0. *steps counts the wave's steps.
__device__ __noinline__ int forward(const Seg& g, int stop, int32_t* col, bool store,
                                    int8_t* carry, U4* columns, Band bd, uint32_t* steps_done) {
  const int lane = lane_id();
  const int nb = (g.ql + 63) / 64;
  const int strips = (nb + kWave - 1) / kWave;
  int last_score = kFar;
  int prev_cs = 1, prev_ce = 0;  // columns whose bottom carries the strip above stored
  // the last row of the strip above at the column before this strip's first
  // (join_col): this strip's first column continues it by +1 per row
  int join_score = 0;
  int join_col = -1;
  for (int k = 0; k < strips; ++k) {
    const int b = k * kWave + lane;
    const int nbs = min(kWave, nb - k * kWave);  // blocks in this strip
    const bool active_lane = lane < nbs;
    int cs, ce;
    strip_columns(g, bd, k, nbs, &cs, &ce);
    cs = uniform(cs);
    ce = uniform(ce);
    // where the next strip starts (its join column is the one before)
    int next_cs = 0, next_ce = -1;
    if (k + 1 < strips) {
      strip_columns(g, bd, k + 1, min(kWave, nb - (k + 1) * kWave), &next_cs, &next_ce);
    }
    const int next_join = uniform(next_cs) - 1;
    if (cs > ce) {
      // the band misses every row of this strip
      if (stop >= 0 && active_lane) {
        for (int i = 0; i < 64; ++i) {
          const int r = b * 64 + i;
          if (r < g.ql) col[r] = kFar;
        }
      }
      prev_cs = 1;
      prev_ce = 0;
      join_col = -1;
      wave_done();
      continue;
    }
    Peq peq{0, 0, 0, 0, 0, 0};
    if (active_lane) {
      peq = build_peq(g, b);
    }
    Word P = ~Word(0), M = 0;
    // D at the block's last row before column cs, with vertical deltas of +1
    // down the column: exact at column -1; further right, +1 per row from the
    // strip above's last row at column cs - 1 (an upper bound, and a column
    // whose deltas join the carries of the strip above), or from the bound
    // max(row, column) + 1 when the strip above computed nothing
    int score;
    if (cs == 0) {
      score = (b + 1) * 64;
    } else {
      const int top = join_col == cs - 1 ? join_score : max(k * kWave * 64, cs);
      score = top + (lane + 1) * 64;
    }
    int joined = 0;  // (the carry lane: its score at the next strip's join column)
    const int steps = ce + nbs;  // lane 0 runs columns cs..ce, the last lane ends nbs - 1 later
    *steps_done += static_cast<uint32_t>(steps - cs);
    const uint64_t store_base = static_cast<uint64_t>(k) * (g.tl + 63) * 64;
    // Lane b works on column c = st - b, the column lane b - 1 had one step
    // earlier: each lane hands its target byte and its bottom carry (hout + 1
    // in bits 8..9) to the next lane with one DPP wave shift. Lane 0 takes
    // its byte (and, below the first strip, its carry from the strip above)
    // from 64-column chunks that every lane loads one chunk ahead.
    auto t_at = [&](int j) -> int { return j < g.tl ? g.tc(j) : 0; };
    // (a column the strip above did not compute: +1, an upper bound)
    auto carry_at = [&](int j) -> int {
      return k == 0 ? 1 : (j >= prev_cs && j <= prev_ce ? static_cast<int>(carry[j]) : 1);
    };
    // (an outer loop per chunk: a loaded chunk is only read in the chunk
    // after the one that issued its load, and no loaded value is carried
    // through the step loop, which would make every step wait for memory)
    const int st_begin = cs & ~(kWave - 1);
    int t_next = t_at(st_begin + lane);
    int c_next = carry_at(st_begin + lane);
    const bool carry_lane = lane == nbs - 1 && k + 1 < strips;
    bool prev_acgt = true;  // (no columns before the first chunk)
    int fwd = 1 << 8;  // (byte, hout + 1) of this lane's last step
    for (int st0 = st_begin; st0 < steps; st0 += kWave) {
     const int t_cur = t_next, c_cur = c_next;
     // this chunk's bytes and carries (loaded a chunk ago) are waited for
     // here, once, before the next chunk's loads go out
     asm volatile("" ::"v"(t_cur), "v"(c_cur));
     // lanes work on columns st0 - 63 .. st0 + 63 in this chunk: when those
     // are all A/C/G/T and every active lane's column is inside the matrix
     // on every step, the steps run without the range and byte checks
     const bool mine_acgt = st0 + lane >= g.tl || is_acgt(t_cur, code2(t_cur));
     const bool chunk_acgt = __all(mine_acgt);
     const int st_end = min(steps, st0 + kWave);
     const bool fast = chunk_acgt && prev_acgt && st0 >= cs + nbs - 1 && st_end - 1 <= ce;
     prev_acgt = chunk_acgt;
     t_next = t_at(st0 + kWave + lane);
     c_next = carry_at(st0 + kWave + lane);
     if (fast) {
      for (int st = st0; st < st_end; ++st) {
       const int c = st - lane;
       const int up = __builtin_amdgcn_update_dpp(0, fwd, 0x138, 0xf, 0xf, false);
       const int t0 = __builtin_amdgcn_readlane(t_cur, st & (kWave - 1));
       const int h0 = __builtin_amdgcn_readlane(c_cur, st & (kWave - 1));
       const uint8_t tc = static_cast<uint8_t>(lane == 0 ? t0 : (up & 0xff));
       const int hin = lane == 0 ? h0 : (up >> 8) - 1;
       // (lanes past the strip compute unused values; they store nothing and
       // feed only lanes past the strip)
       const Word eq = acgt_eq(peq, code2(tc));
       Word hp;
       const int hout = block_step(P, M, eq, hin, &hp);
       score += hout;
       if (store && active_lane) {
         const uint64_t idx = store_base + static_cast<uint64_t>(st) * nbs + lane;
         columns[idx] = U4{static_cast<uint32_t>(P), static_cast<uint32_t>(P >> 32),
                            static_cast<uint32_t>(hp), static_cast<uint32_t>(hp >> 32)};
       }
       if (carry_lane) {
         carry[c] = static_cast<int8_t>(hout);
         if (c == next_join) joined = score;
       }
       fwd = static_cast<int>(tc) | ((hout + 1) << 8);
      }
      continue;
     }
     for (int st = st0; st < st_end; ++st) {
      const int c = st - lane;
      const int up = __builtin_amdgcn_update_dpp(0, fwd, 0x138, 0xf, 0xf, false);
      // lane 0's inputs are uniform reads; selected, not branched to
      const int t0 = __builtin_amdgcn_readlane(t_cur, st & (kWave - 1));
      const int h0 = __builtin_amdgcn_readlane(c_cur, st & (kWave - 1));
      const uint8_t tc = static_cast<uint8_t>(lane == 0 ? t0 : (up & 0xff));
      const int hin = lane == 0 ? h0 : (up >> 8) - 1;
      int hout = 0;
      if (active_lane && c >= cs && c <= ce) {
        // rows equal to the target byte (exact byte equality, as edlib's
        // alphabet without equalities)
        const int code = code2(tc);
        Word eq = acgt_eq(peq, code);
        if (!is_acgt(tc, code)) {
          eq = tc == 'N' ? (peq.n | peq.pad) : rare_eq(g, b, tc, peq.pad);
        }
        Word hp;
        hout = block_step(P, M, eq, hin, &hp);
        score += hout;
        if (store) {
          const uint64_t idx = store_base + static_cast<uint64_t>(st) * nbs + lane;
          columns[idx] = U4{static_cast<uint32_t>(P), static_cast<uint32_t>(P >> 32),
                            static_cast<uint32_t>(hp), static_cast<uint32_t>(hp >> 32)};
        }
        if (carry_lane) {
          carry[c] = static_cast<int8_t>(hout);
          if (c == next_join) joined = score;
        }
      }
      fwd = static_cast<int>(tc) | ((hout + 1) << 8);
     }
    }
    const bool reaches_end = ce == g.tl - 1;
    if (stop >= 0 && active_lane) {
      // this block's rows at the last column
      int v = score;
      for (int i = 63; i >= 0; --i) {
        const int r = b * 64 + i;
        if (r < g.ql) col[r] = reaches_end ? v : kFar;
        if ((P >> i) & 1) v -= 1;
        if ((M >> i) & 1) v += 1;
      }
    }
    // score of the last row (in the last strip's last block)
    if (k == strips - 1 && reaches_end) {
      const int last_block = nb - 1;
      const int last_bit = (g.ql - 1) % 64;
      int v = score;
      for (int i = 63; i > last_bit; --i) {
        if ((P >> i) & 1) v -= 1;
        if ((M >> i) & 1) v += 1;
      }
      last_score = __shfl(v, last_block - k * kWave, kWave);
    }
    prev_cs = cs;
    prev_ce = ce;
    join_col = next_join >= cs && next_join <= ce ? next_join : -1;
    join_score = __shfl(joined, nbs - 1, kWave);
    wave_done();  // carries and stored columns visible to every lane
  }
  return last_score;
}

// Inclusive scans over the 64 lanes.
__device__ __forceinline__ int32_t lane_scan_add(int32_t x) {
  const int lane = lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int32_t y = __shfl_up(x, d, kWave);
    if (lane >= d) x += y;
  }
  return x;
}
__device__ __forceinline__ int32_t lane_scan_max(int32_t x) {
  const int lane = lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int32_t y = __shfl_up(x, d, kWave);
    if (lane >= d) x = max(x, y);
  }
  return x;
}

// A task of another lane (uniform or per lane), and as a uniform value.
__device__ __forceinline__ void read_task(const AlignTask& t, int l, AlignTask* w) {
  *w = AlignTask{__builtin_amdgcn_readlane(t.q0, l), __builtin_amdgcn_readlane(t.ql, l),
                 __builtin_amdgcn_readlane(t.t0, l), __builtin_amdgcn_readlane(t.tl, l),
                 __builtin_amdgcn_readlane(t.score, l)};
}
__device__ __forceinline__ void shuffle_task(const AlignTask& t, int l, AlignTask* w) {
  *w = AlignTask{__shfl(t.q0, l, kWave), __shfl(t.ql, l, kWave),    __shfl(t.t0, l, kWave),
                 __shfl(t.tl, l, kWave), __shfl(t.score, l, kWave)};
}
__device__ __forceinline__ AlignTask uniform_task(const AlignTask& t) {
  return AlignTask{uniform(t.q0), uniform(t.ql), uniform(t.t0), uniform(t.tl),
                   uniform(t.score)};
}

// Position of the n-th set bit.
__device__ __forceinline__ int nth_bit(unsigned long long m, int n) {
  for (int i = 0; i < n; ++i) m &= m - 1;
  return __ffsll(static_cast<long long>(m)) - 1;
}

// ---- banded runs: blocks on lanes, cyclically along the band ----
//
// A run is one bit-vector DP of a (sub)problem over its diagonal band: the
// forward half or the reversed half of a split, or a whole leaf whose columns
// are kept for the traceback. Block b (64 query rows) is active over the
// columns where its rows meet the band, about 64 + band width of them, and
// starts 64 columns after block b - 1, so only band / 65 blocks are active at
// a time. A group of G lanes takes blocks l, l + G, l + 2G, ... in turn, in
// an anti-diagonal pipeline: at step s block b works on column s - b, and its
// bottom row's horizontal delta reaches block b + 1 (the next lane of the
// group, cyclically) one step later through a lane rotation. A run takes
// about (columns + blocks) steps whatever its band, and 64 / G runs share the
// wave: the two halves of a split, and the subproblems of one recursion
// level, run side by side. With the lanes fixed to the 64 blocks of a strip
// instead, an 8 kbp pair at 12% error took 34,000 steps; here it takes 8,200.
//
// Block b's state when it starts right of column 0 continues the last row of
// block b - 1 at the column before by +1 per row, and a column that block
// b - 1 did not compute feeds it a horizontal delta of +1: upper bounds, as
// Band above requires. Activity starts and ends on chunks of 16 steps
// (columns before and after the band are computed as well), so that the steps
// of a chunk need no activity checks; an inactive lane computes a block whose
// column is flat and matches nothing, which passes +1 on for the 16 steps
// of a chunk. Chunks at the first or last column, or with target bytes other
// than A, C, G, T and N, take the checked steps.
//
// A step is about 34 vector instructions on 32-bit halves (59 in the strip
// form): the four match words of a block live in LDS, one 8-byte read per
// step picked by the target byte's code; the deltas of the block above come
// from its raw high words (bit 31), which the shift by one takes in with
// v_alignbit; the score is counted once per chunk from the collected bits.

constexpr int kChunk = 16;
constexpr int kCodeN = 4;      // table entry of N
constexpr int kCodeNone = 5;   // matches nothing
constexpr int kCodeRare = 6;   // other bytes: compared exactly in checked steps
constexpr int kEqEntries = 6;
constexpr int kTeamWaves = static_cast<int>(kAlignTeamWaves);
constexpr int kTeamGroup = 256;  // lanes of a run that spans half a team

typedef __attribute__((address_space(3))) uint64_t LdsWord;
// Query bit planes of 64 rows: code bits, A/C/G/T rows, N rows.
struct PlaneWord {
  Word lo, hi, acgt, n;
};

// One run, as every lane of its group sees it.
struct Run {
  int q0, ql;          // query rows
  int t0, tl;          // target columns
  bool rev;            // both read from the end
  Band band;           // in the run's own orientation
  uint64_t store;      // first entry of its columns (leaf runs)
};

// Lanes a run needs: its blocks and one idle lane, or enough that block
// b + G starts after block b + 1 has ended (their starts are 65 steps apart,
// their lives 64 + width columns, both rounded to chunks).
__device__ __forceinline__ int run_lanes(int ql, int width) {
  return min((ql + 63) / 64 + 1, (width + 160 + 64) / 65);
}

// First and last step of block b, the columns it covers, and whether its
// state at the last column is needed.
struct BlockSpan {
  int first;   // chunk it becomes active in (a multiple of kChunk)
  int last;    // first chunk in which it is no longer active
  int skew;    // its column at step s is s - skew
  bool edge;   // starts at column 0
  bool final;  // its rows meet the band at the last column
  bool any;    // it meets the band at all
};

template <int G>
__device__ __forceinline__ BlockSpan block_span(const Run& r, int nb, int b) {
  BlockSpan s;
  // (a run over several waves hands deltas on by whole chunks: 16 steps
  // between the last block of a wave and the first of the next)
  s.skew = G > kWave ? b + (kChunk - 1) * (b >> 6) : b;
  const int cs = max(0, 64 * b - r.band.hi);
  const int reach = 64 * b + 63 - r.band.lo;
  const int ce = min(r.tl - 1, reach);
  s.any = b < nb && cs <= r.tl - 1 && ce >= 0;
  s.final = reach >= r.tl - 1;
  s.first = (cs + s.skew) & ~(kChunk - 1);
  s.edge = cs == 0 || s.first < s.skew;
  if (s.edge) s.first = s.skew & ~(kChunk - 1);
  // (one column more than the band asks for: a lane that becomes inactive
  // loses its last step's delta)
  s.last = (ce + s.skew + 1 + kChunk) & ~(kChunk - 1);
  return s;
}

// Index of the last block of a run that meets the band.
__device__ __forceinline__ int last_block(const Run& r, int nb) {
  return min(nb - 1, (r.tl - 1 + r.band.hi) / 64);
}

// Lane position in its group and the group's number. Groups of 8 and 32
// lanes are interleaved in pairs, so that one step to the next lane of a
// group is a rotation by two of a row or of the wave.
template <int G>
__device__ __forceinline__ void lane_group(int lane, int* group, int* pos) {
  if (G == 8) {
    *group = (lane >> 4) * 2 + (lane & 1);
    *pos = (lane & 15) >> 1;
  } else if (G == 16) {
    *group = lane >> 4;
    *pos = lane & 15;
  } else if (G == 32) {
    *group = lane & 1;
    *pos = lane >> 1;
  } else {
    *group = 0;
    *pos = lane;
  }
}

// x of the group's previous lane, cyclically.
template <int G>
__device__ __forceinline__ uint32_t group_prev(uint32_t x) {
  const int v = static_cast<int>(x);
  if (G == 8) return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(v, 0x122, 0xf, 0xf, false));
  if (G == 16) return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(v, 0x121, 0xf, 0xf, false));
  const int once = __builtin_amdgcn_mov_dpp(v, 0x13c, 0xf, 0xf, false);  // wave_ror:1
  if (G == 32) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(once, 0x13c, 0xf, 0xf, false));
  }
  return static_cast<uint32_t>(once);
}

__device__ __forceinline__ uint32_t shl1(uint32_t x, uint32_t below) {
  return __builtin_amdgcn_alignbit(x, below, 31);  // (x << 1) | (below >> 31)
}

// State of a lane's block: vertical deltas, and the raw high words of the
// last step's horizontal deltas (bit 31: the block's bottom row).
struct BlockState {
  uint32_t pl, ph, ml, mh;
  uint32_t out_p, out_m;
};

// One step on 32-bit halves; up_p / up_m: bit 31 holds the delta from above.
// hp receives the horizontal positive deltas of the column.
__device__ __forceinline__ void half_step(BlockState& s, uint32_t eql, uint32_t eqh, uint32_t up_p,
                                          uint32_t up_m, uint32_t* hpl, uint32_t* hph) {
  const uint32_t neg = up_m >> 31;
  const uint32_t xvl = eql | s.ml, xvh = eqh | s.mh;
  eql |= neg;
  const Word p = static_cast<Word>(s.ph) << 32 | s.pl;
  const Word sum = (static_cast<Word>(eqh & s.ph) << 32 | (eql & s.pl)) + p;
  const uint32_t xhl = (static_cast<uint32_t>(sum) ^ s.pl) | eql;
  const uint32_t xhh = (static_cast<uint32_t>(sum >> 32) ^ s.ph) | eqh;
  const uint32_t pl = s.ml | ~(xhl | s.pl), ph = s.mh | ~(xhh | s.ph);
  const uint32_t ml = s.pl & xhl, mh = s.ph & xhh;
  const uint32_t spl = shl1(pl, up_p), sph = shl1(ph, pl);
  const uint32_t sml = (ml << 1) | neg, smh = shl1(mh, ml);
  s.pl = sml | ~(xvl | spl);
  s.ph = smh | ~(xvh | sph);
  s.ml = spl & xvl;
  s.mh = sph & xvh;
  s.out_p = ph;
  s.out_m = mh;
  *hpl = pl;
  *hph = ph;
}

// What a run leaves in a lane: the state of its final block.
struct FinalState {
  uint32_t pl, ph, ml, mh;
  int score;
  int block;  // -1: none
};

// Per-team view of one pair.
struct PairView {
  const uint8_t* Q;
  const uint8_t* T;
  const PlaneWord* planes;  // word w: rows 64 (w - 1) .. (one guard word in front)
  U4* store;                // this wave's leaf columns
  int32_t* col_left;
  int32_t* col_right;
  uint8_t* tmp;             // ops in place (see leaf_walk)
};

// 64 plane bits from absolute row p (>= -63) on.
__device__ __forceinline__ Word plane_bits(Word a, Word b, int sh) {
  return sh == 0 ? a : (a >> sh) | (b << (64 - sh));
}

// Match words of block b of the run into the lane's table entries.
__device__ __forceinline__ void load_block(const PairView& v, const Run& r, int b, LdsWord* table) {
  const int p = r.rev ? r.q0 + r.ql - 64 * (b + 1) : r.q0 + 64 * b;
  const PlaneWord* w = v.planes + ((p + 64) >> 6);
  const int sh = p & 63;
  const PlaneWord a = w[0], c = w[1];
  Word lo = plane_bits(a.lo, c.lo, sh), hi = plane_bits(a.hi, c.hi, sh);
  Word acgt = plane_bits(a.acgt, c.acgt, sh), n = plane_bits(a.n, c.n, sh);
  if (r.rev) {
    lo = __builtin_bitreverse64(lo);
    hi = __builtin_bitreverse64(hi);
    acgt = __builtin_bitreverse64(acgt);
    n = __builtin_bitreverse64(n);
  }
  const int rows = r.ql - 64 * b;
  // rows past the query match everything
  const Word pad = rows >= 64 ? Word(0) : ~Word(0) << rows;
  table[0 * kWave] = (acgt & ~lo & ~hi) | pad;
  table[1 * kWave] = (acgt & lo & ~hi) | pad;
  table[2 * kWave] = (acgt & ~lo & hi) | pad;
  table[3 * kWave] = (acgt & lo & hi) | pad;
  table[kCodeN * kWave] = n | pad;
}

// The 16 target bytes of columns c0 .. c0 + 15 of the run (clamped to the
// target; *at: the first column they hold, ascending).
__device__ __forceinline__ U4 load_target(const PairView& v, const Run& r, int c0, int* at) {
  const uint8_t* t = v.T + r.t0;
  if (r.tl >= kChunk) {
    const int a = min(max(c0, 0), r.tl - kChunk);
    *at = a;
    const uint8_t* src = r.rev ? t + (r.tl - kChunk - a) : t + a;
    U4 x;
    __builtin_memcpy(&x, src, 16);
    return x;
  }
  // a target shorter than a chunk: byte by byte
  *at = 0;
  uint32_t w[4] = {0};
  for (int i = 0; i < r.tl; ++i) {
    const uint32_t c = t[i];
    const int k = r.rev ? kChunk - r.tl + i : i;  // (rev: the bytes end at position 15)
    w[k >> 2] |= c << (8 * (k & 3));
  }
  return U4{w[0], w[1], w[2], w[3]};
}

// Rows equal to a target byte outside A/C/G/T/N, compared one by one.
__device__ Word rare_rows(const PairView& v, const Run& r, int b, uint8_t c) {
  Word w = 0;
  for (int i = 0; i < 64; ++i) {
    const int row = 64 * b + i;
    if (row >= r.ql) {
      w |= Word(1) << i;
    } else if (v.Q[r.rev ? r.q0 + r.ql - 1 - row : r.q0 + row] == c) {
      w |= Word(1) << i;
    }
  }
  return w;
}

// Runs the group's run `r` (have: the lane's group has one). G = kTeamGroup:
// one run over four waves of a team (pos_base: the wave's first lane in it),
// all of them in step, with mail the team's mailbox. kStore keeps (vertical,
// horizontal) positive deltas of every column for the traceback, entry
// store + step * stride + lane. n_chunks is the same for every lane that
// shares a barrier. Returns the lane's final state.
template <int G, bool kStore>
__device__ __forceinline__ FinalState run_band(const PairView& v, const Run& r, bool have,
                                               int n_chunks, int pos_base, LdsWord* eq_table,
                                               uint32_t* mail) {
  const int lane = threadIdx.x & (kWave - 1);
  int group, pos;
  lane_group<G>(lane, &group, &pos);
  if (G > kWave) pos += pos_base;
  const int nb = (r.ql + 63) / 64;
  LdsWord* table = eq_table + lane;
  table[kCodeNone * kWave] = 0;
  const uint32_t table_at = static_cast<uint32_t>((size_t)table);
  FinalState fin{0, 0, 0, 0, 0, -1};
  BlockState st{0, 0, 0, 0, 0x80000000u, 0};
  int score = 0, score_before = 0;
  int b = pos;
  BlockSpan span = block_span<G>(r, nb, b);
  bool pending = have && span.any, active = false;
  if (pending) load_block(v, r, b, table);
  const int stride = min(G, nb);
  U4 raw = U4{0};
  int raw_at = 0;
  const uint32_t fwd_sel = 0x03020100u, rev_sel = 0x04050607u;
  const uint32_t byte_sel = r.rev ? rev_sel : fwd_sel;
  for (int chunk = 0; chunk < n_chunks; ++chunk) {
    const int S = chunk * kChunk;
    if (__any((active && S >= span.last) || (pending && S >= span.first))) {
      // the score of the block above at the column before this one's first
      const int hout = static_cast<int>(st.out_p >> 31) - static_cast<int>(st.out_m >> 31);
      int above = static_cast<int>(group_prev<G>(static_cast<uint32_t>(score - hout)));
      if (G > kWave && lane == 0) above = static_cast<int>(mail[3 * (threadIdx.x >> 6) + 2]);
      if (active && S >= span.last) {
        if (span.final) fin = FinalState{st.pl, st.ph, st.ml, st.mh, score, b};
        active = false;
        b += G;
        span = block_span<G>(r, nb, b);
        pending = span.any;
        if (pending) load_block(v, r, b, table);
      }
      if (pending && S >= span.first) {
        pending = false;
        active = true;
        st.pl = st.ph = ~0u;
        st.ml = st.mh = 0;
        st.out_p = 0x80000000u;
        st.out_m = 0;
        score = (span.edge ? 64 * b : above) + 64;
        raw = load_target(v, r, S - span.skew, &raw_at);
      }
    }
    const int c0 = S - span.skew;
    // the chunk's target bytes in column order, as 4-bit codes
    const U4 now = raw;
    const int shift = 4 * (c0 - raw_at);
    if (active) raw = load_target(v, r, c0 + kChunk, &raw_at);
    uint32_t x[4], y[4];
    x[0] = __builtin_amdgcn_perm(now.w, now.x, byte_sel);
    x[1] = __builtin_amdgcn_perm(now.z, now.y, byte_sel);
    x[2] = __builtin_amdgcn_perm(now.y, now.z, byte_sel);
    x[3] = __builtin_amdgcn_perm(now.x, now.w, byte_sel);
    uint32_t odd = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      y[k] = ((x[k] >> 1) ^ (x[k] >> 2)) & 0x03030303u;
      odd |= __builtin_amdgcn_perm(0u, 0x54474341u, y[k]) ^ x[k];
      y[k] |= y[k] >> 4;
    }
    Word codes = static_cast<Word>(__builtin_amdgcn_perm(y[3], y[2], 0x06040200u)) << 32 |
                 __builtin_amdgcn_perm(y[1], y[0], 0x06040200u);
    const int c_lo = max(0, -c0), c_hi = min(kChunk, r.tl - c0);  // valid steps of the chunk
    bool rare = false;
    if (__any(active && odd != 0)) {
      // N and other bytes
      codes = 0;
#pragma unroll 1
      for (int k = 0; k < kChunk; ++k) {
        const uint32_t w = k < 8 ? (k < 4 ? x[0] : x[1]) : (k < 12 ? x[2] : x[3]);
        const int c = static_cast<int>((w >> (8 * (k & 3))) & 0xffu);
        const int two = code2(c);
        const int code = is_acgt(c, two) ? two : (c == 'N' ? kCodeN : kCodeRare);
        codes |= static_cast<Word>(code) << (4 * k);
        const int i = k - (shift >> 2);  // its step
        rare |= code == kCodeRare && i >= c_lo && i < c_hi;
      }
    }
    if (shift != 0) {
      codes = shift > 0 ? (shift < 64 ? codes >> shift : 0) : (shift > -64 ? codes << -shift : 0);
    }
    if (!active) {
      codes = 0x5555555555555555ull;
      st.pl = st.ph = st.ml = st.mh = 0;
      st.out_p = 0x80000000u;
      st.out_m = 0;
    }
    uint32_t acc_p = 0, acc_m = 0;
    const bool keep = kStore && active && pos < stride;
    U4* const at = kStore ? v.store + r.store + static_cast<uint64_t>(S) * stride + pos : nullptr;
    uint32_t in_p = 0, in_m = 0;  // lane 0 of a wave in a team run: the deltas from above
    if (G > kWave) {
      in_p = mail[3 * (threadIdx.x >> 6)];
      in_m = mail[3 * (threadIdx.x >> 6) + 1];
    }
    const bool plain = !active || (c_lo == 0 && c_hi == kChunk && !rare);
    if (__all(plain)) {
#pragma unroll
      for (int i = 0; i < kChunk; ++i) {
        uint32_t up_p, up_m;
        if (G > kWave) {
          up_p = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
              static_cast<int>(in_p << (16 + i)), static_cast<int>(st.out_p), 0x138, 0xf, 0xf, false));
          up_m = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
              static_cast<int>(in_m << (16 + i)), static_cast<int>(st.out_m), 0x138, 0xf, 0xf, false));
        } else {
          up_p = group_prev<G>(st.out_p);
          up_m = group_prev<G>(st.out_m);
        }
        const uint32_t half = i < 8 ? static_cast<uint32_t>(codes) : static_cast<uint32_t>(codes >> 32);
        const uint32_t code = (half >> (4 * (i & 7))) & 15u;
        const Word eq = *(LdsWord*)(size_t)(table_at + (code << 9));
        uint32_t hl, hh;
        half_step(st, static_cast<uint32_t>(eq), static_cast<uint32_t>(eq >> 32), up_p, up_m, &hl, &hh);
        acc_p = shl1(acc_p, st.out_p);
        acc_m = shl1(acc_m, st.out_m);
        if (kStore && keep) at[static_cast<uint64_t>(i) * stride] = U4{st.pl, st.ph, hl, hh};
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < kChunk; ++i) {
        uint32_t up_p, up_m;
        if (G > kWave) {
          up_p = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
              static_cast<int>(in_p << (16 + i)), static_cast<int>(st.out_p), 0x138, 0xf, 0xf, false));
          up_m = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
              static_cast<int>(in_m << (16 + i)), static_cast<int>(st.out_m), 0x138, 0xf, 0xf, false));
        } else {
          up_p = group_prev<G>(st.out_p);
          up_m = group_prev<G>(st.out_m);
        }
        const int code = static_cast<int>(codes >> (4 * i)) & 15;
        uint32_t p1 = 0, m1 = 0;  // this step's deltas for the score
        if (!active || (i >= c_lo && i < c_hi)) {
          Word eq;
          if (active && code == kCodeRare) {
            const int c = c0 + i;
            eq = rare_rows(v, r, b, v.T[r.t0 + (r.rev ? r.tl - 1 - c : c)]);
          } else {
            eq = *(LdsWord*)(size_t)(table_at + (static_cast<uint32_t>(code) << 9));
          }
          uint32_t hl, hh;
          half_step(st, static_cast<uint32_t>(eq), static_cast<uint32_t>(eq >> 32), up_p, up_m, &hl, &hh);
          p1 = st.out_p;
          m1 = st.out_m;
          if (kStore && keep) at[static_cast<uint64_t>(i) * stride] = U4{st.pl, st.ph, hl, hh};
        } else {
          st.out_p = 0x80000000u;
          st.out_m = 0;
        }
        acc_p = shl1(acc_p, p1);
        acc_m = shl1(acc_m, m1);
      }
    }
    score_before = score;
    score += __popc(acc_p) - __popc(acc_m);
    if (G > kWave) {
      // hand lane 63's deltas and score to the next wave of the run
      __syncthreads();
      if (lane == kWave - 1) {
        const int w = threadIdx.x >> 6;
        const int next = (w & ~3) | ((w + 1) & 3);
        // (an inactive lane passes +1)
        mail[3 * next] = active ? acc_p : 0xffffu;
        mail[3 * next + 1] = active ? acc_m : 0u;
        mail[3 * next + 2] = static_cast<uint32_t>(score_before);
      }
      __syncthreads();
    }
  }
  if (active && span.final) fin = FinalState{st.pl, st.ph, st.ml, st.mh, score, b};
  return fin;
}

// Scores of the run's last column from the lanes' final states, row r at
// col[r].
__device__ __forceinline__ void dump_column(const Run& r, const FinalState& f, int32_t* col) {
  if (f.block < 0) return;
  int32_t* at = col + 64 * f.block;
  const int rows = min(64, r.ql - 64 * f.block);
  int v = f.score;
#pragma unroll 1
  for (int j = 15; j >= 0; --j) {
    const uint32_t p = (j >= 8 ? f.ph : f.pl) >> (4 * (j & 7));
    const uint32_t m = (j >= 8 ? f.mh : f.ml) >> (4 * (j & 7));
    int x[4];
#pragma unroll
    for (int u = 3; u >= 0; --u) {
      x[u] = v;
      v += static_cast<int>((m >> u) & 1u) - static_cast<int>((p >> u) & 1u);
    }
    if (4 * j + 3 < rows) {
      const int4 q = make_int4(x[0], x[1], x[2], x[3]);
      __builtin_memcpy(at + 4 * j, &q, 16);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (4 * j + u < rows) at[4 * j + u] = x[u];
      }
    }
  }
}

// Rows of a banded run whose last-column scores dump_column writes.
__device__ __forceinline__ void column_rows(const Run& r, int* first, int* last) {
  const int from = r.tl - 1 + r.band.lo - 63;  // 64 b >= from
  const int b0 = from <= 0 ? 0 : (from + 63) / 64;
  const int b1 = last_block(r, (r.ql + 63) / 64);
  *first = 64 * b0;
  *last = min(r.ql, 64 * (b1 + 1)) - 1;
}

// A leaf whose columns are stored.
struct Leaf {
  int q0, ql, t0, tl;
  uint64_t store;
  int group;  // lanes of its run; 0: strips of 64 blocks
};

// Entry of column c and the block of a row; nb: blocks of the leaf, stride:
// entries of a step in a group's run.
__device__ __forceinline__ uint64_t leaf_entry(const Leaf& f, int nb, int stride, int row, int c) {
  const int b = row >> 6;
  if (f.group == 0) {
    const int k = b / kWave, lb = b % kWave;
    const int nbs = min(kWave, nb - k * kWave);
    return f.store + static_cast<uint64_t>(k) * (f.tl + 63) * 64 +
           static_cast<uint64_t>(c + lb) * nbs + lb;
  }
  return f.store + static_cast<uint64_t>(c + b) * stride + (b & (f.group - 1));
}

// Traceback of one leaf by one lane, from its last cell: up (insertion) where
// the vertical delta is +1, else left (deletion) where the horizontal delta
// is, else the diagonal, a match where the bytes are equal. (On an optimal
// path's cells the deltas are exact, and a neighbour one below is on an
// optimal path itself, so it was computed.) Ops go to the end of the leaf's
// own q0 + t0 .. room of tmp, last op last. The next four cells down the
// diagonal are loaded together: most moves are diagonal, and each round trip
// to the stored columns costs several hundred cycles.
__device__ __forceinline__ void leaf_walk(const PairView& v, const Leaf& f) {
  const int nb = (f.ql + 63) / 64;
  const int stride = min(f.group, nb);
  int r = f.ql - 1, c = f.tl - 1;
  uint8_t* out = v.tmp + f.q0 + f.t0 + f.ql + f.tl;  // one past the next op
  const uint8_t* q = v.Q + f.q0;
  const uint8_t* t = v.T + f.t0;
  constexpr int kAhead = 4;
  while (r >= 0 && c >= 0) {
    U4 e[kAhead];
    uint8_t qb[kAhead], tb[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      // (clamped cells past the edge are not used)
      const int rr = max(r - k, 0), cc = max(c - k, 0);
      const int d = min(r - rr, c - cc);
      e[k] = v.store[leaf_entry(f, nb, stride, r - d, c - d)];
      qb[k] = q[r - d];
      tb[k] = t[c - d];
    }
    bool straight = true;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      if (straight && r >= 0 && c >= 0) {
        const bool high = (r & 32) != 0;
        const uint32_t p = high ? e[k].y : e[k].x, h = high ? e[k].w : e[k].z;
        const uint32_t up = (p >> (r & 31)) & 1u, left = (h >> (r & 31)) & 1u;
        const uint8_t op = up ? 1 : (left ? 2 : (qb[k] == tb[k] ? 0 : 3));
        *--out = op;
        r -= op != 2;
        c -= op != 1;
        straight = op == 0 || op == 3;
      }
    }
  }
  while (c >= 0) {
    *--out = 2;
    --c;
  }
  while (r >= 0) {
    *--out = 1;
    --r;
  }
}

// leaf_walk for a leaf of far more rows than columns or the other way round,
// whose path is mostly gaps: an insertion goes up as far as the column's
// deltas in the block lead, and after two deletions the next four cells to
// the left are loaded together. (Every op of a gap is a round trip in
// leaf_walk: 500 pairs of 8,000 x 1,500 bases took 5.7 ms, of 8,000 x 200 6.2
// and of 200 x 8,000 6.4; now 2.9, 0.6 and 3.7. On other leaves this form
// is 4% slower.)
__device__ __forceinline__ void leaf_walk_gaps(const U4* store, const uint8_t* q, const uint8_t* t,
                                               uint8_t* out, int ql, int tl, int group) {
  const Leaf f{0, ql, 0, tl, 0, group};
  const int nb = (ql + 63) / 64;
  const int stride = min(group, nb);
  int r = ql - 1, c = tl - 1;
  constexpr int kAhead = 4;
  int lefts = 0;  // deletions since the last other op
  while (r >= 0 && c >= 0) {
    U4 e[kAhead];
    uint8_t qb[kAhead], tb[kAhead];
    const bool sideways = lefts >= 2;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      // (clamped cells past the edge are not used)
      const int d = min(k, sideways ? c : min(r, c));
      const int row = sideways ? r : r - d;
      e[k] = store[leaf_entry(f, nb, stride, row, c - d)];
      qb[k] = q[row];
      tb[k] = t[c - d];
    }
    bool straight = true;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      if (straight && r >= 0 && c >= 0) {
        const Word p = static_cast<Word>(e[k].y) << 32 | e[k].x;
        const Word h = static_cast<Word>(e[k].w) << 32 | e[k].z;
        const Word above = p << (63 - (r & 63));  // the row's delta on top
        if (above >> 63) {
          // (the zeroes shifted in end the run at the block's first row)
          const int n = __clzll(static_cast<long long>(~above));
          for (int i = 0; i < n; ++i) *--out = 1;
          r -= n;
          lefts = 0;
          straight = false;
        } else {
          const bool left = (h >> (r & 63)) & 1u;
          *--out = left ? 2 : (qb[k] == tb[k] ? 0 : 3);
          if (!left) --r;
          --c;
          lefts = left ? lefts + 1 : 0;
          straight = left == sideways;
        }
      }
    }
  }
  for (; c >= 0; --c) *--out = 2;
  for (; r >= 0; --r) *--out = 1;
}

__device__ __noinline__ void leaf_walk_gaps_call(const U4* store, const uint8_t* q,
                                                 const uint8_t* t, uint8_t* out, int ql, int tl,
                                                 int group) {
  leaf_walk_gaps(store, q, t, out, ql, tl, group);
}

// Query bit planes of the pair (word 0 is a guard), 64 rows per ballot.
__device__ __forceinline__ void build_planes(const uint8_t* Q, int QL, PlaneWord* planes, int wave,
                                             int waves) {
  const int lane = threadIdx.x & (kWave - 1);
  const int words = (QL + 63) / 64 + 3;
  for (int w = wave; w < words; w += waves) {
    const int row = 64 * (w - 1) + lane;
    const int c = row >= 0 && row < QL ? Q[row] : 0;
    const int code = code2(c);
    const bool plain = is_acgt(c, code);
    const Word lo = __ballot(plain && (code & 1) != 0), hi = __ballot(plain && (code & 2) != 0);
    const Word acgt = __ballot(plain), n = __ballot(c == 'N');
    if (lane < 4) {
      reinterpret_cast<Word*>(planes + w)[lane] =
          lane == 0 ? lo : (lane == 1 ? hi : (lane == 2 ? acgt : n));
    }
  }
}

enum : int { kTaskTrivial = 0, kTaskLeaf = 1, kTaskSplit = 2 };

__device__ __forceinline__ bool is_leaf(int ql, int tl) {
  const uint64_t nb = (static_cast<uint64_t>(ql) + 63) / 64;
  return 20ull * nb * static_cast<uint64_t>(tl) < kLeafBytes;
}

__device__ __forceinline__ int band_width(Band b) { return b.hi - b.lo; }

// The run of one side of a split task (0: forward over the left half, 1:
// reversed over the right half), and of a leaf.
__device__ __forceinline__ Run split_run(const AlignTask& t, int side, int d) {
  const Band bd = band_for(t.ql, t.tl, d);
  const int lw = t.tl / 2;
  if (side == 0) return Run{t.q0, t.ql, t.t0, lw, false, bd, 0};
  return Run{t.q0, t.ql, t.t0 + lw, t.tl - lw, true, band_reversed(bd, t.ql, t.tl), 0};
}

template <int G>
__device__ __forceinline__ int run_chunks(const Run& r) {
  const int nb = (r.ql + 63) / 64;
  return block_span<G>(r, nb, last_block(r, nb)).last / kChunk;
}

// Up to 64 / G runs of the wave, group g's one in lane g of the task arrays.
template <int G, bool kStore>
__device__ __forceinline__ FinalState run_groups(const PairView& v, const Run& r, bool have,
                                                 LdsWord* eq, uint32_t* steps) {
  int n = have ? run_chunks<G>(r) : 0;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) n = max(n, __shfl_xor(n, d, kWave));
  n = uniform(n);
  *steps += static_cast<uint32_t>(n * kChunk);
  return run_band<G, kStore>(v, r, have, n, 0, eq, nullptr);
}

template <bool kStore>
__device__ __noinline__ FinalState run_wave(const PairView& v, const Run& r, bool have, int G,
                                            LdsWord* eq, uint32_t* steps) {
  if (G == 8) return run_groups<8, kStore>(v, r, have, eq, steps);
  if (G == 16) return run_groups<16, kStore>(v, r, have, eq, steps);
  if (G == 32) return run_groups<32, kStore>(v, r, have, eq, steps);
  return run_groups<64, kStore>(v, r, have, eq, steps);
}

// Lane's group and position for a group size known at run time.
__device__ __forceinline__ int group_of(int G, int lane) {
  int group = 0, pos = 0;
  if (G == 8) lane_group<8>(lane, &group, &pos);
  else if (G == 16) lane_group<16>(lane, &group, &pos);
  else if (G == 32) lane_group<32>(lane, &group, &pos);
  return group;
}

__device__ __forceinline__ int group_size(int lanes) {
  return lanes <= 8 ? 8 : lanes <= 16 ? 16 : lanes <= 32 ? 32 : 64;
}

// One pair by a workgroup of kWaves waves. The recursion runs level by level:
// every split of a level first (both halves, side by side in the waves), then
// the split rows, which give the next level's tasks, then the leaves with
// their tracebacks. Ops are written in place (see leaf_walk) and packed at the
// end.
template <int kWaves>
__device__ __forceinline__ void align_pair(const AlignParams& A, const AlignPair& pr, AlignResult& R) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform(static_cast<int>(threadIdx.x) >> 6);
  __shared__ __attribute__((aligned(16))) uint64_t eq_tables[kWaves][kEqEntries * kWave];
  __shared__ uint32_t mail[3 * kWaves];
  __shared__ int team_next, team_error, team_min, team_ops[kWaves];
  __shared__ uint32_t team_steps;
  LdsWord* eq = (LdsWord*)eq_tables[wave];
  uint8_t* slot = A.scratch + static_cast<uint64_t>(blockIdx.x) * A.slot_bytes;
  PlaneWord* planes = reinterpret_cast<PlaneWord*>(slot + A.layout.planes);
  AlignTask* cur = reinterpret_cast<AlignTask*>(slot + A.layout.tasks);
  AlignTask* next = cur + A.caps.tasks;
  const int QL = static_cast<int>(pr.q_len), TL = static_cast<int>(pr.t_len);
  uint8_t* out = A.ops + pr.out_off;
  if (QL > static_cast<int>(A.caps.q) || TL > static_cast<int>(A.caps.t)) {
    R.status = kAlignScratch;
    return;
  }
  if (QL == 0 || TL == 0) {
    for (int i = threadIdx.x; i < QL + TL; i += kWaves * kWave) out[i] = QL == 0 ? 2 : 1;
    R.n_ops = static_cast<uint32_t>(QL + TL);
    R.edit_distance = QL > TL ? QL : TL;
    R.status = kAlignOk;
    return;
  }
  PairView v;
  v.Q = A.arena + pr.q_off;
  v.T = A.arena + pr.t_off;
  v.planes = planes;
  v.store = reinterpret_cast<U4*>(slot + A.layout.store) + static_cast<uint64_t>(wave) * A.caps.store_words;
  v.col_left = reinterpret_cast<int32_t*>(slot + A.layout.col_left);
  v.col_right = reinterpret_cast<int32_t*>(slot + A.layout.col_right);
  v.tmp = slot + A.layout.ops_tmp;
  // (one carry array per wave; a strip run is one wave's)
  int8_t* carry = reinterpret_cast<int8_t*>(slot + A.layout.carry) +
                  static_cast<uint64_t>(wave) * A.layout.carry_bytes;
  uint32_t steps = 0;

  build_planes(v.Q, QL, planes, wave, kWaves);
  // no op yet anywhere
  for (int i = threadIdx.x * 16; i < QL + TL; i += kWaves * kWave * 16) {
    *reinterpret_cast<U4*>(v.tmp + i) = U4{~0u, ~0u, ~0u, ~0u};
  }
  // The whole pair's distance is not known: its band starts from a guess k
  // (the batch's band width, else |delta| + max(|q|, |t|) / 5) and doubles
  // until the banded distance is at most k (then it is exact: with k >= the
  // true distance every optimal path lies inside the band) or the band holds
  // the whole matrix. Every subproblem below knows its score, and its band is
  // the tightest one for it.
  const int delta_top = QL > TL ? QL - TL : TL - QL;
  int k_top = A.band0 > 0 ? max(static_cast<int>(A.band0), delta_top)
                          : delta_top + max(QL, TL) / 5 + 64;
  auto full_band = [](Band b, int ql, int tl) { return b.lo <= -(tl - 1) && b.hi >= ql - 1; };
  if (threadIdx.x == 0) {
    team_next = 0;
    team_error = 0;
    team_steps = 0;
    cur[0] = AlignTask{0, QL, 0, TL, -1};
  }
  __syncthreads();
  int n_cur = 1;
  int best = -1;

  // a whole leaf by this wave: columns, then (with walk) the ops
  auto wide_leaf = [&](const AlignTask& t, Band bd) -> int {
    Seg g{v.Q + t.q0, v.T + t.t0, t.ql, t.tl, false};
    return forward(g, -1, nullptr, true, carry, v.store, bd, &steps);
  };

  while (n_cur > 0) {
    // ---- splits: both halves of every task ----
    int serial = 0;  // batches, dealt to the waves in turn
    for (int base = 0; base < n_cur; base += kWave) {
      AlignTask t{0, 0, 0, 0, 0};
      int kind = -1, need = 0;
      if (base + lane < n_cur) {
        t = cur[base + lane];
        if (t.ql == 0 || t.tl == 0) {
          kind = kTaskTrivial;
        } else {
          kind = is_leaf(t.ql, t.tl) ? kTaskLeaf : kTaskSplit;
          const int d = t.score >= 0 ? t.score : k_top;
          need = run_lanes(t.ql, band_width(band_for(t.ql, t.tl, d)));
        }
      }
      unsigned long long todo = __ballot(kind == kTaskSplit);
      while (todo != 0) {
        const int first = __ffsll(static_cast<long long>(todo)) - 1;
        const int lanes = __builtin_amdgcn_readlane(need, first);
        if (lanes > kWave) {
          todo &= todo - 1;
          AlignTask w;
          read_task(t, first, &w);
          const int d = w.score >= 0 ? w.score : k_top;
          if (kWaves == kTeamWaves && lanes <= kTeamGroup) {
            if constexpr (kWaves == kTeamWaves) {
              // both halves at once, four waves each
              const Run r = split_run(w, wave >> 2, d);
              const int n = max(run_chunks<kTeamGroup>(split_run(w, 0, d)),
                                run_chunks<kTeamGroup>(split_run(w, 1, d)));
              __syncthreads();
              if (threadIdx.x < 3 * kWaves) mail[threadIdx.x] = threadIdx.x % 3 == 0 ? 0xffffu : 0u;
              __syncthreads();
              const FinalState f =
                  run_band<kTeamGroup, false>(v, r, true, n, (wave & 3) * kWave, eq, mail);
              steps += static_cast<uint32_t>(n * kChunk);
              dump_column(r, f, (r.rev ? v.col_right : v.col_left) + r.q0);
            }
          } else {
            // wider than the lanes: strips of 64 blocks
            for (int side = 0; side < 2; ++side) {
              if (serial++ % kWaves != wave) continue;
              const Run r = split_run(w, side, d);
              Seg g{v.Q + r.q0, v.T + r.t0, r.ql, r.tl, r.rev};
              forward(g, r.tl - 1, (side ? v.col_right : v.col_left) + r.q0, false, carry, v.store,
                      r.band, &steps);
            }
          }
          continue;
        }
        const int G = group_size(lanes);
        const int fits = G == 64 ? 1 : (kWave / G) / 2;  // tasks per batch
        unsigned long long take = 0;
        int taken = 0;
        for (unsigned long long m = todo; m != 0 && taken < fits; m &= m - 1) {
          const int k = __ffsll(static_cast<long long>(m)) - 1;
          if (__builtin_amdgcn_readlane(need, k) <= G) {
            take |= 1ull << k;
            ++taken;
          }
        }
        todo &= ~take;
        const int group = group_of(G, lane);
        for (int half = 0; half < (G == 64 ? 2 : 1); ++half) {
          if (serial++ % kWaves != wave) continue;
          // group g: task number g / 2 of the batch, side g % 2
          const int number = G == 64 ? 0 : group >> 1;
          const int side = G == 64 ? half : group & 1;
          const bool have = number < taken;
          AlignTask w;
          shuffle_task(t, nth_bit(take, have ? number : 0), &w);
          const Run r = split_run(w, side, w.score >= 0 ? w.score : k_top);
          const FinalState f = run_wave<false>(v, r, have, G, eq, &steps);
          if (have) dump_column(r, f, (r.rev ? v.col_right : v.col_left) + r.q0);
        }
      }
    }
    __syncthreads();
    // ---- split rows ----
    int number = 0;
    for (int i = 0; i < n_cur; ++i) {
      const AlignTask t = uniform_task(cur[i]);
      if (t.ql == 0 || t.tl == 0 || is_leaf(t.ql, t.tl)) continue;
      if (number++ % kWaves != wave) continue;
      const int d = t.score >= 0 ? t.score : k_top;
      const Band bd = band_for(t.ql, t.tl, d);
      const int lanes = run_lanes(t.ql, band_width(bd));
      const int lw = t.tl / 2, rw = t.tl - lw;
      const int32_t* left = v.col_left + t.q0;
      const int32_t* right = v.col_right + t.q0;
      int l0 = 0, l1 = t.ql - 1, r0 = 0, r1 = t.ql - 1;  // rows with a score
      if (lanes <= kWave || (kWaves == kTeamWaves && lanes <= kTeamGroup)) {
        column_rows(split_run(t, 0, d), &l0, &l1);
        column_rows(split_run(t, 1, d), &r0, &r1);
      }
      // interior split rows x: left row x and right row ql - 2 - x
      const int x0 = max(max(0, l0), t.ql - 2 - r1), x1 = min(min(t.ql - 2, l1), t.ql - 2 - r0);
      const int at_top = r1 == t.ql - 1 ? lw + uniform(right[t.ql - 1]) : kFar;       // x = -1
      const int at_end = l1 == t.ql - 1 ? uniform(left[t.ql - 1]) + rw : kFar;        // x = ql - 1
      int score = t.score;
      if (score < 0) {
        // the distance of the whole pair: the minimum over all split rows
        int m = min(at_top, at_end);
        for (int x = x0 + lane; x <= x1; x += kWave) m = min(m, left[x] + right[t.ql - 2 - x]);
        for (int s = 1; s < kWave; s <<= 1) m = min(m, __shfl_xor(m, s, kWave));
        score = uniform(m);
        if (lane == 0) team_min = score;
      }
      if (t.score >= 0 || score <= k_top || full_band(bd, t.ql, t.tl)) {
        int split = -2;
        constexpr int kRows = 4;  // rounds of 64 rows loaded together
        for (int x = x0; x <= x1 && split == -2; x += kRows * kWave) {
          unsigned long long hit[kRows];
#pragma unroll
          for (int u = 0; u < kRows; ++u) {
            const int at = x + u * kWave + lane;
            const int sum = at <= x1 ? left[at] + right[t.ql - 2 - at] : -1;
            hit[u] = __ballot(sum == score);
          }
#pragma unroll
          for (int u = kRows - 1; u >= 0; --u) {
            if (hit[u] != 0) split = x + u * kWave + __ffsll(static_cast<long long>(hit[u])) - 1;
          }
        }
        int ls = 0, rs = 0;
        bool found = true;
        if (split != -2) {
          ls = uniform(left[split]);
          rs = uniform(right[t.ql - 2 - split]);
        } else if (at_top == score) {
          split = -1;
          ls = lw;
          rs = at_top - lw;
        } else if (at_end == score) {
          split = t.ql - 1;
          ls = at_end - rw;
          rs = rw;
        } else {
          found = false;
          if (lane == 0) team_error = kAlignNoSplit;
        }
        if (found && lane == 0) {
          const int at = atomicAdd(&team_next, 2);
          if (at + 2 > static_cast<int>(A.caps.tasks)) {
            team_error = kAlignStack;
          } else {
            next[at] = AlignTask{t.q0, split + 1, t.t0, lw, ls};
            next[at + 1] = AlignTask{t.q0 + split + 1, t.ql - split - 1, t.t0 + lw, rw, rs};
          }
        }
      }
    }
    __syncthreads();
    const AlignTask top = uniform_task(cur[0]);
    const bool unknown = top.score < 0;
    if (unknown && !is_leaf(top.ql, top.tl)) {
      const int m = uniform(team_min);
      if (m > k_top && !full_band(band_for(top.ql, top.tl, k_top), top.ql, top.tl)) {
        // outside the guess: nothing was added to the next level
        k_top *= 2;
        __syncthreads();
        continue;
      }
      best = m;
    }
    if (uniform(team_error) != 0) {
      R.status = uniform(team_error);
      return;
    }
    // ---- leaves: columns, then the tracebacks of a batch side by side ----
    serial = 0;
    for (int base = 0; base < n_cur; base += kWave) {
      AlignTask t{0, 0, 0, 0, 0};
      int kind = -1, need = 0;
      if (base + lane < n_cur) {
        t = cur[base + lane];
        if (t.ql == 0 || t.tl == 0) {
          kind = kTaskTrivial;
        } else if (is_leaf(t.ql, t.tl)) {
          kind = kTaskLeaf;
          const int d = t.score >= 0 ? t.score : k_top;
          need = run_lanes(t.ql, band_width(band_for(t.ql, t.tl, d)));
        }
      }
      for (unsigned long long m = __ballot(kind == kTaskTrivial); m != 0; m &= m - 1) {
        AlignTask w;
        read_task(t, __ffsll(static_cast<long long>(m)) - 1, &w);
        for (int i = threadIdx.x; i < w.ql + w.tl; i += kWaves * kWave) {
          v.tmp[w.q0 + w.t0 + i] = w.ql == 0 ? 2 : 1;
        }
      }
      unsigned long long todo = __ballot(kind == kTaskLeaf);
      while (todo != 0) {
        const int first = __ffsll(static_cast<long long>(todo)) - 1;
        const int lanes = __builtin_amdgcn_readlane(need, first);
        const int G = lanes > kWave ? 0 : group_size(lanes);
        const int fits = G == 0 ? 1 : kWave / G;
        unsigned long long take = 0;
        int taken = 0;
        uint64_t room = 0;       // entries taken
        uint64_t my_store = 0;   // (lane k: of the batch's task k)
        for (unsigned long long m = todo; m != 0 && taken < fits; m &= m - 1) {
          const int k = __ffsll(static_cast<long long>(m)) - 1;
          if (__builtin_amdgcn_readlane(need, k) > max(G, lanes)) continue;
          const int ql = __builtin_amdgcn_readlane(t.ql, k), tl = __builtin_amdgcn_readlane(t.tl, k);
          const int nb = (ql + 63) / 64;
          const uint64_t entries =
              G == 0 ? 0 : static_cast<uint64_t>(tl + nb) * min(G, nb);
          if (taken > 0 && room + entries > A.caps.store_words) continue;
          if (lane == taken) my_store = room;
          room += entries;
          take |= 1ull << k;
          ++taken;
        }
        todo &= ~take;
        if (serial++ % kWaves != wave) continue;
        AlignTask w;
        const int group = group_of(G, lane);
        const bool have = group < taken;
        shuffle_task(t, nth_bit(take, have ? group : 0), &w);
        uint64_t store = __shfl(my_store, have ? group : 0, kWave);
        int k_leaf = k_top;
        while (true) {
          const int d = w.score >= 0 ? w.score : k_leaf;
          const Band bd = band_for(w.ql, w.tl, d);
          int distance = kFar;
          int used = G;
          if (unknown) {
            // (the guess may have grown past the group)
            const int lanes_now = run_lanes(w.ql, band_width(bd));
            used = lanes_now > kWave ? 0 : group_size(lanes_now);
            store = 0;
          }
          if (used == 0) {
            distance = wide_leaf(uniform_task(w), bd);
          } else {
            const bool mine = unknown ? group_of(used, lane) == 0 : have;
            const Run r{w.q0, w.ql, w.t0, w.tl, false, bd, store};
            const FinalState f = run_wave<true>(v, r, mine, used, eq, &steps);
            if (unknown) {
              // the last cell, in the last block's state
              const int last = (w.ql - 1) >> 6, bits = (w.ql - 1) & 63;
              int x = kFar;
              if (f.block == last) {
                const Word p = static_cast<Word>(f.ph) << 32 | f.pl;
                const Word m = static_cast<Word>(f.mh) << 32 | f.ml;
                const Word mask = bits == 63 ? Word(0) : ~Word(0) << (bits + 1);
                x = f.score - __popcll(p & mask) + __popcll(m & mask);
              }
              for (int s = 1; s < kWave; s <<= 1) x = min(x, __shfl_xor(x, s, kWave));
              distance = uniform(x);
            }
          }
          if (!unknown) break;
          best = distance;
          if (distance <= k_leaf || full_band(bd, w.ql, w.tl)) {
            if (lane == 0) team_min = used;  // (the walk below follows this layout)
            break;
          }
          k_leaf *= 2;
        }
        wave_done();
        int used = G;
        if (unknown) used = uniform(team_min);
        // one lane per leaf follows its path
        AlignTask mine;
        shuffle_task(t, nth_bit(take, lane < taken ? lane : 0), &mine);
        // (the path has at least `net` gap ops. Where they are half of it,
        // unrelated bases 1:2, they come one or two at a time and leaf_walk is
        // 6% faster; at 1:5 it takes 1.2 to 2 times as long. One form for all
        // leaves of the wave: one after the other they cost 12% where it has
        // both kinds. Teams call it per leaf: in their kernel the code in
        // line costs every pair 3%.)
        const int net = mine.ql > mine.tl ? mine.ql - mine.tl : mine.tl - mine.ql;
        bool gaps = net > 16 + max(mine.ql, mine.tl) * 5 / 8;
        if (kWaves == 1) gaps = __any(gaps);
        if (lane < taken) {
          const Leaf leaf{mine.q0, mine.ql, mine.t0, mine.tl, unknown ? 0 : my_store, used};
          if (!gaps) {
            leaf_walk(v, leaf);
          } else {
            const U4* store = v.store + leaf.store;
            const uint8_t* q = v.Q + leaf.q0;
            const uint8_t* t = v.T + leaf.t0;
            uint8_t* end = v.tmp + leaf.q0 + leaf.t0 + leaf.ql + leaf.tl;
            if constexpr (kWaves == 1) {
              leaf_walk_gaps(store, q, t, end, leaf.ql, leaf.tl, used);
            } else {
              leaf_walk_gaps_call(store, q, t, end, leaf.ql, leaf.tl, used);
            }
          }
        }
        wave_done();
      }
    }
    __syncthreads();
    n_cur = uniform(team_next);
    AlignTask* x = cur;
    cur = next;
    next = x;
    __syncthreads();
    if (threadIdx.x == 0) team_next = 0;
    __syncthreads();
  }
  // ---- pack the ops ----
  const int total = QL + TL;
  const int share = ((total + kWaves - 1) / kWaves + 1023) / 1024 * 1024;
  const int from = wave * share, to = min(total, from + share);
  auto valid_mask = [&](const U4& x, int at) -> uint32_t {
    uint32_t m = 0;
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // top bit of each byte set: no op
      const uint32_t b = ~w[k] & 0x80808080u;
      m |= ((b >> 7 | b >> 14 | b >> 21 | b >> 28) & 15u) << (4 * k);
    }
    const int n = to - at;
    return n >= 16 ? m : (n > 0 ? m & ((1u << n) - 1u) : 0u);
  };
  int count = 0;
  if (kWaves > 1) {
    int c = 0;
    for (int i = from + lane * 16; i < to; i += kWave * 16) {
      c += __popc(valid_mask(*reinterpret_cast<const U4*>(v.tmp + i), i));
    }
    for (int s = 1; s < kWave; s <<= 1) c += __shfl_xor(c, s, kWave);
    if (lane == 0) team_ops[wave] = c;
    __syncthreads();
    for (int w = 0; w < wave; ++w) count += team_ops[w];
  }
  for (int i0 = from; i0 < to; i0 += kWave * 16) {
    const int i = i0 + lane * 16;
    U4 x{~0u, ~0u, ~0u, ~0u};
    uint32_t m = 0;
    if (i < to) {
      x = *reinterpret_cast<const U4*>(v.tmp + i);
      m = valid_mask(x, i);
    }
    const int c = __popc(m);
    const int incl = lane_scan_add(c);
    uint8_t* dst = out + count + incl - c;
    if (m == 0xffffu) {
      __builtin_memcpy(dst, &x, 16);
    } else if (m != 0) {
      const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if ((m >> k) & 1u) *dst++ = static_cast<uint8_t>(w[k >> 2] >> (8 * (k & 3)));
      }
    }
    count += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  if (kWaves > 1) {
    if (wave == kWaves - 1 && lane == 0) team_next = count;
    if (lane == 0) atomicAdd(&team_steps, steps);
    __syncthreads();
    count = uniform(team_next);
    steps = uniform(static_cast<int>(team_steps));
  }
  R.n_ops = static_cast<uint32_t>(count);
  R.edit_distance = best;
  R.status = kAlignOk;
  R.pad = steps;
}
}  // namespace

// kWaves = 1: one wave per pair, for batches that fill the device; kTeamWaves:
// a workgroup of eight waves per pair, for few long pairs.
template <int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(5))) void align_batch_kernel(
    AlignParams A) {
  __shared__ uint32_t next;
  while (true) {
    if (threadIdx.x == 0) {
      next = atomicAdd(A.queue_head, 1u);
    }
    __syncthreads();
    const uint32_t q = next;
    __syncthreads();
    if (q >= A.n_order) {
      break;
    }
    const uint32_t i = A.order != nullptr ? A.order[q] : q;
    AlignResult res{0, -1, kAlignNotRun, 0};
    align_pair<kWaves>(A, A.pairs[i], res);
    __syncthreads();
    if (threadIdx.x == 0) {
      A.results[i] = res;
    }
    __syncthreads();
  }
}

hipError_t launch_align_batch(const AlignParams& params, uint32_t grid, hipStream_t stream) {
  if (params.waves == kTeamWaves) {
    hipLaunchKernelGGL(align_batch_kernel<kTeamWaves>, dim3(grid), dim3(64 * kTeamWaves), 0, stream,
                       params);
  } else {
    hipLaunchKernelGGL(align_batch_kernel<1>, dim3(grid), dim3(64), 0, stream, params);
  }
  return hipGetLastError();
}

// Clears the work-queue counter with a kernel store (no memset node, so the
// sequence can sit inside a captured graph).
__global__ void clear_counter_kernel(uint32_t* counter) {
  if (threadIdx.x == 0) *counter = 0;
}

hipError_t launch_align_batch_cleared(const AlignParams& params, uint32_t grid,
                                      hipStream_t stream) {
  hipLaunchKernelGGL(clear_counter_kernel, dim3(1), dim3(64), 0, stream, params.queue_head);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_align_batch(params, grid, stream);
}

// Breaking points of every aligned pair (racon overlap.cpp:226-292, the walk
// over edlib's CIGAR), from the edit operations the batch kernel left in
// device memory. A match or mismatch advances target and query, an insertion
// the query, a deletion the target; the first match of a window and the
// position after its last match are emitted as a pair when the target
// position reaches the window's last base (k * W - 1 for the multiples of W
// inside (t_begin, t_end), then t_end - 1). counts[i] is the number of points
// (2 per window with a match), or 0xffffffff when they would outgrow the
// pair's room.
//
// One wave per pair walks the ops 256 at a time (4 per lane, adjacent bytes
// across lanes): prefix sums of the target and query advances give every
// op's positions, a prefix max the last match so far (matches advance the
// target, so the last one has the largest position), and windows follow
// from target positions: window w covers (end(w - 1), end(w)]. A match whose
// window differs from the previous match's opens that window's entry (first
// match); an op that reaches end(w) closes it when the last match so far lies
// in w. Entry e of a pair is points 4e..4e+3 of its room: windows with a
// match, in order.
__global__ __launch_bounds__(256) void breaking_points_kernel(
    const AlignPair* __restrict__ pairs, const AlignResult* __restrict__ results,
    const uint8_t* __restrict__ ops, const BreakSpan* __restrict__ spans, uint32_t n,
    uint32_t window_length, uint32_t* __restrict__ points, uint32_t* __restrict__ counts) {
  const uint32_t i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (i >= n) return;  // (uniform over the wave)
  const BreakSpan sp = spans[i];
  if (results[i].status != kAlignOk) {
    if (lane == 0) counts[i] = 0xfffffffeu;  // not aligned on the device
    return;
  }
  const uint8_t* op = ops + pairs[i].out_off;
  const uint32_t n_ops = results[i].n_ops;
  const int64_t W = window_length;
  // windows: ends m0 - 1, m0 + W - 1, ... for the nm multiples of W in
  // (t_begin, t_end), then t_end - 1 (window nm)
  const int64_t t_end = sp.t_end;
  const int64_t m0_wide = (static_cast<int64_t>(sp.t_begin) / W + 1) * W;
  const uint32_t nm = m0_wide < t_end ? static_cast<uint32_t>((t_end - 1 - m0_wide) / W + 1) : 0;
  const uint32_t m0 = nm ? static_cast<uint32_t>(m0_wide) : 0;  // < t_end when used
  const uint32_t Wn = window_length;
  // (target positions here are in [0, t_end), so 32-bit arithmetic holds)
  auto window_of = [&](int64_t t) -> uint32_t {
    const uint32_t tt = static_cast<uint32_t>(t);
    const uint32_t w = (nm == 0 || tt < m0) ? 0 : (tt - m0) / Wn + 1;
    return w < nm ? w : nm;
  };
  auto window_end = [&](uint32_t w) -> int64_t {
    return w < nm ? static_cast<int64_t>(m0) + static_cast<int64_t>(w) * W - 1 : t_end - 1;
  };
  uint32_t* out = points + 2 * sp.out;
  const int64_t cap_entries = sp.cap / 2;  // entries that fit the pair's room
  // carried over chunks (uniform)
  int64_t t_base = static_cast<int64_t>(sp.t_begin) - 1;
  int64_t q_base = static_cast<int64_t>(sp.q_first) - 1;
  int64_t last_t = -1, last_q = -1;  // last match so far (t, q after the op)
  int64_t opened = 0;                // entries opened so far
  int64_t closed = 0;                // entries closed so far
  for (uint32_t c0 = 0; c0 < n_ops; c0 += 4 * kWave) {
    uint32_t o[4];
    int32_t dt = 0, dq = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t k = c0 + 4 * lane + u;
      o[u] = k < n_ops ? (op[k] & 3u) : 4u;  // 4: past the end (no op)
      dt += (o[u] != 1u && o[u] != 4u);
      dq += (o[u] != 2u && o[u] != 4u);
    }
    const int32_t st = lane_scan_add(dt), sq = lane_scan_add(dq);
    int64_t t = t_base + (st - dt), q = q_base + (sq - dq);
    // positions after each of the lane's ops, and the lane's last match
    int64_t ta[4], qa[4];
    int32_t lm_t = -1, lm_q = -1;  // relative to t_base / q_base + 1
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (o[u] != 1u && o[u] != 4u) ++t;
      if (o[u] != 2u && o[u] != 4u) ++q;
      ta[u] = t;
      qa[u] = q;
      if (o[u] == 0u || o[u] == 3u) {
        lm_t = static_cast<int32_t>(t - t_base);
        lm_q = static_cast<int32_t>(q - q_base);
      }
    }
    // last match before the lane (exclusive max over lanes, then the carry)
    const int32_t mt = lane_scan_max(lm_t), mq = lane_scan_max(lm_q);
    const int32_t pt = __shfl_up(mt, 1, kWave), pq = __shfl_up(mq, 1, kWave);
    int64_t prev_t = last_t, prev_q = last_q;
    if (lane > 0 && pt >= 0) {
      prev_t = t_base + pt;
      prev_q = q_base + pq;
    }
    // windows of the lane's target advances (-1: none), and of the last
    // match before each op
    int64_t wa[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) wa[u] = (o[u] != 1u && o[u] != 4u) ? window_of(ta[u]) : -1;
    const int64_t pw0 = prev_t >= 0 ? window_of(prev_t) : -1;
    // entries the lane opens, then their numbers
    int32_t n_open = 0;
    {
      int64_t pw = pw0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (o[u] == 0u || o[u] == 3u) {
          if (wa[u] != pw) ++n_open;
          pw = wa[u];
        }
      }
    }
    const int32_t so = lane_scan_add(n_open);
    int64_t e_open = opened + (so - n_open);  // entries opened before this lane
    int32_t n_close = 0;
    int64_t pw = pw0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (o[u] == 0u || o[u] == 3u) {
        if (wa[u] != pw) {
          // first match of window w: entry e_open
          if (e_open < cap_entries) {
            out[4 * e_open] = static_cast<uint32_t>(ta[u]);
            out[4 * e_open + 1] = static_cast<uint32_t>(qa[u]);
          }
          ++e_open;
        }
        prev_t = ta[u];
        prev_q = qa[u];
        pw = wa[u];
      }
      if (wa[u] >= 0) {
        if (ta[u] == window_end(static_cast<uint32_t>(wa[u])) && pw == wa[u]) {
          // the op reaches the window's last base with a match in the window:
          // close its entry (the last one opened)
          const int64_t e = e_open - 1;
          if (e < cap_entries) {
            out[4 * e + 2] = static_cast<uint32_t>(prev_t + 1);
            out[4 * e + 3] = static_cast<uint32_t>(prev_q + 1);
          }
          ++n_close;
        }
      }
    }
    const int32_t sc = lane_scan_add(n_close);
    // carry to the next chunk (from the last lane)
    const int32_t all_t = __shfl(st, kWave - 1, kWave), all_q = __shfl(sq, kWave - 1, kWave);
    const int32_t all_mt = __shfl(mt, kWave - 1, kWave), all_mq = __shfl(mq, kWave - 1, kWave);
    if (all_mt >= 0) {
      last_t = t_base + all_mt;
      last_q = q_base + all_mq;
    }
    t_base += all_t;
    q_base += all_q;
    opened += __shfl(so, kWave - 1, kWave);
    closed += __shfl(sc, kWave - 1, kWave);
  }
  if (lane == 0) {
    counts[i] = 2 * closed > sp.cap ? 0xffffffffu : static_cast<uint32_t>(2 * closed);
  }
}

hipError_t launch_breaking_points(const AlignPair* pairs, const AlignResult* results,
                                  const uint8_t* ops, const BreakSpan* spans, uint32_t n,
                                  uint32_t window_length, uint32_t* points, uint32_t* counts,
                                  hipStream_t stream) {
  // one wave per pair, four pairs per workgroup
  hipLaunchKernelGGL(breaking_points_kernel, dim3((n + 3) / 4), dim3(256), 0, stream, pairs,
                     results, ops, spans, n, window_length, points, counts);
  return hipGetLastError();
}

hipError_t align_occupancy(int* blocks_per_cu, uint32_t waves) {
  if (waves == kTeamWaves) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks_per_cu, align_batch_kernel<kTeamWaves>, 64 * kTeamWaves, 0);
  }
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, align_batch_kernel<1>, 64, 0);
}

}  // namespace rh
