// Partial-order alignment consensus of racon windows on gfx950.
//
// One 64-lane wave owns one window at a time (a "slot" of device scratch).
// Per layer, in racon's order (window.cpp:89-113):
//   1. the subgraph the layer is aligned to: nodes reached backwards from
//      node `end` through in-edges and aligned links without passing below
//      node id `begin` (whole graph when the layer spans the window);
//   2. its DFS topological order (roots in increasing node id, predecessors
//      then aligned nodes pushed, an aligned set emitted right after the
//      node that reached it first);
//   3. linear-gap NW of the layer against that order: lanes own strips of
//      4 to 20 columns of each DP row, predecessor rows come from LDS, the
//      horizontal gap chain is a wave prefix-max, and each cell records the
//      first matching move (diagonal over predecessors in in-edge order,
//      then vertical, then horizontal);
//   4. the traceback from the first sink row with the highest last-column
//      score, following the recorded moves;
//   5. insertion of the layer into the graph (edge weight = w[i-1] + w[i],
//      w = phred - 33 or 1) and a new topological order.
// After the last layer: heaviest-bundle path with branch completion,
// per-position coverage and racon's trimming (window.cpp:115-139).
//
// The subgraph closure, the row tables, the insertion and the new order work on
// 64 ranks, rows or layer positions at a time. What is sequential by nature
// (the walk along the recorded moves, the exact DFS order where a tie asks for
// it, the insertion of a path whose nodes share an aligned set, the consensus
// path) the wave runs lane-uniformly: every lane executes the same loads and
// branches, so no lane-0 divergence or broadcast is needed. Parallelism comes
// from thousands of windows in flight (persistent kernel over a size-ordered
// queue) and from the 64-lane DP rows.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "poa_types.hpp"

namespace rh {

namespace {

constexpr int kWave = 64;
// Launch-invariant data (parameters, slot layout, window and layer tables)
// is read through constant-address-space references: uniform scalar loads
// that no store of the kernel can clobber, hoisted and kept in scalar
// registers.
typedef __attribute__((address_space(1))) uint8_t GByte;
// Device buffers named by the parameters, as global-memory pointers (they
// are loaded from memory, so the compiler cannot infer their address space).
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* global(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}
typedef const __attribute__((address_space(4))) PoaParams CParams;
typedef const __attribute__((address_space(4))) PoaSlotLayout CLayout;
typedef const __attribute__((address_space(4))) PoaSlotCaps CCaps;
typedef const __attribute__((address_space(4))) PoaWindow CWindow;
typedef const __attribute__((address_space(4))) PoaLayer CLayer;

// Resident waves per SIMD the kernel is register-allocated for (168 VGPRs
// at 3, 128 at 4).
#ifndef RH_POA_WAVES_PER_EU
#define RH_POA_WAVES_PER_EU 4
#endif

// Aligned-set entries kept per node. The default build keeps kMaxAligned;
// poa_kernel_wide.hip compiles this file again with kMaxAlignedWide (and
// "_wide" kernel and launcher names) for the windows whose columns hold more
// distinct bytes (IUPAC codes), which the host reruns there.
#ifndef RH_POA_ALIGNED
#define RH_POA_ALIGNED kMaxAligned
#endif
#ifdef RH_POA_WIDE
#define RH_POA_SYM(name) name##_wide
#else
#define RH_POA_SYM(name) name
#endif
constexpr uint32_t kAligned = RH_POA_ALIGNED;

constexpr int kStrip = 4;                  // DP columns per lane per tile
constexpr int kTile = kWave * kStrip;      // 256 columns per tile
constexpr int32_t kNegInf = -(1 << 29);
// Move codes (16 bits per DP cell): bits 15-14 the move (diagonal,
// vertical, horizontal); for diagonal and vertical moves bits 12-0 are the
// index of the predecessor in the row's in-edge list.
constexpr uint16_t kCodeDiag = 0x0000;
constexpr uint16_t kCodeVert = 0x4000;
constexpr uint16_t kCodeHorz = 0x8000;
constexpr uint32_t kCodePayload = 0x1fff;
// Bits 16..22 of a row's meta word: the row's entry in the slot's pool of
// global score rows (a row that found no LDS slot, in a pass with a pool).
constexpr int kRowMetaGShift = 16;
constexpr int kRowMetaGMask = 127;
static_assert(kPoaHPoolRows <= kRowMetaGMask + 1, "pool entries fit the meta bits");
// Bits 24..26: the number of predecessors, at most 7.
constexpr int kRowMetaPredShift = 24;
constexpr int kRowMetaPredMask = 7;

__device__ __forceinline__ int lane_id() { return threadIdx.x; }

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// v_writelane: `old` with lane `lane` set to the uniform `value` (the
// intrinsic has no clang builtin here, so it is bound by name)
extern "C" __device__ int32_t rh_amdgcn_writelane(int32_t value, int32_t lane, int32_t old) __asm(
    "llvm.amdgcn.writelane.i32");
__device__ __forceinline__ int lane_write(int value, int lane, int old) {
  return rh_amdgcn_writelane(value, lane, old);
}

__device__ __forceinline__ void wave_sync() { __syncthreads(); }

// Phase clock: accumulates device constant-clock ticks into R.phase[k].
struct PhaseClock {
  uint64_t t;
  __device__ PhaseClock() : t(wall_clock64()) {}
  __device__ void lap(PoaResult& R, int k) {
    const uint64_t now = wall_clock64();
    R.phase[k] += now - t;
    t = now;
  }
};

// Views of one slot's arrays: one base pointer plus the layout's offsets
// (kernel arguments), so the array addresses are rebuilt where used instead of
// occupying registers.
struct Slot {
  GByte* p;  // slot base (global memory)
  CLayout* L;
  __device__ uint8_t* base() const { return (uint8_t*)(p + L->base); }
  __device__ int32_t* in_head() const { return (int32_t*)(p + L->in_head); }
  __device__ int32_t* out_head() const { return (int32_t*)(p + L->out_head); }
  __device__ int32_t* in_tail() const { return (int32_t*)(p + L->in_tail); }
  __device__ int32_t* out_tail() const { return (int32_t*)(p + L->out_tail); }
  __device__ uint8_t* n_aligned() const { return (uint8_t*)(p + L->n_aligned); }
  __device__ int32_t* aligned() const { return (int32_t*)(p + L->aligned); }
  __device__ int32_t* cov() const { return (int32_t*)(p + L->cov); }
  __device__ int32_t* last_label() const { return (int32_t*)(p + L->last_label); }
  __device__ int32_t* e_tail() const { return (int32_t*)(p + L->e_tail); }
  __device__ int32_t* e_head() const { return (int32_t*)(p + L->e_head); }
  __device__ int32_t* e_weight() const { return (int32_t*)(p + L->e_weight); }
  __device__ int32_t* e_next_in() const { return (int32_t*)(p + L->e_next_in); }
  __device__ int32_t* e_next_out() const { return (int32_t*)(p + L->e_next_out); }
  __device__ int32_t* rank_to_node() const { return (int32_t*)(p + L->rank_to_node); }
  __device__ int32_t* node_rank() const { return (int32_t*)(p + L->node_rank); }
  __device__ uint8_t* mark() const { return (uint8_t*)(p + L->mark); }
  __device__ uint8_t* lead() const { return (uint8_t*)(p + L->lead); }
  __device__ int32_t* stack() const { return (int32_t*)(p + L->stack); }
  __device__ uint8_t* in_sub() const { return (uint8_t*)(p + L->in_sub); }
  __device__ int32_t* row_of() const { return (int32_t*)(p + L->row_of); }
  __device__ int32_t* sub_order() const { return (int32_t*)(p + L->sub_order); }
  __device__ int32_t* pred_off() const { return (int32_t*)(p + L->pred_off); }
  __device__ int32_t* pred_rows() const { return (int32_t*)(p + L->pred_rows); }
  __device__ int32_t* row_meta() const { return (int32_t*)(p + L->row_meta); }
  __device__ int32_t* H() const { return (int32_t*)(p + L->H); }
  // global score row of DP row `row` (meta: its row meta word): its pool
  // entry when the slot keeps a pool, else row `row` of the matrix
  __device__ int32_t* H_row(int row, int meta, int pitch) const {
    const int64_t at = L->hpool != 0 ? ((meta >> kRowMetaGShift) & kRowMetaGMask) : row;
    return H() + at * pitch;
  }
  __device__ int32_t* H_row(int row, int pitch) const {
    return L->hpool != 0 ? H_row(row, __builtin_amdgcn_readfirstlane(row_meta()[row - 1]), pitch)
                         : H() + static_cast<int64_t>(row) * pitch;
  }
  __device__ uint16_t* code() const { return (uint16_t*)(p + L->code); }
  __device__ int64_t* scores() const { return (int64_t*)(p + L->scores); }
  __device__ int32_t* preds() const { return (int32_t*)(p + L->preds); }
  __device__ int32_t* path() const { return (int32_t*)(p + L->path); }
  __device__ uint8_t* seq() const { return (uint8_t*)(p + L->seq); }
  __device__ int32_t* qual() const { return (int32_t*)(p + L->qual); }
  __device__ int32_t* anchor() const { return (int32_t*)(p + L->anchor); }
  __device__ int32_t* lpath() const { return (int32_t*)(p + L->lpath); }
  __device__ int32_t* sink_score() const { return (int32_t*)(p + L->sink_score); }
  __device__ int32_t* tie_mark() const { return (int32_t*)(p + L->tie_mark); }
  // per node: base | in-edge count << 8, and the tails of the first eight
  // in-edges (two quads)
  __device__ uint32_t* node_info() const { return (uint32_t*)(p + L->node_info); }
  __device__ int4* node_in() const { return (int4*)(p + L->node_in); }
  // the in-edge that node_info has counted `info >> 8` of before
  __device__ void add_in(int node, uint32_t info, int tail) const {
    const uint32_t n = info >> 8;
    if (n < 8) ((int32_t*)(p + L->node_in))[8 * node + n] = tail;
    node_info()[node] = info + 256u;
  }
  __device__ uint4* row_rec() const { return (uint4*)(p + L->row_rec); }

  int32_t n_nodes;
  int32_t n_edges;
  int32_t n_seqs;
  bool overflow;
};

__device__ __forceinline__ Slot carve(GByte* p, CLayout& l) {
  Slot s;
  s.p = p;
  s.L = &l;
  s.n_nodes = 0;
  s.n_edges = 0;
  s.n_seqs = 0;
  s.overflow = false;
  return s;
}

// ---- graph construction (lane-uniform) ----

__device__ __forceinline__ void touch(Slot& s, int node, int label) {
  if (s.last_label()[node] != label) {
    s.last_label()[node] = label;
    s.cov()[node] = s.cov()[node] + 1;
  }
}

__device__ __forceinline__ int add_node(Slot& s, CCaps& caps, uint8_t base) {
  if (s.n_nodes >= static_cast<int>(caps.nodes)) {
    s.overflow = true;
    return 0;
  }
  const int v = s.n_nodes++;
  s.base()[v] = base;
  s.node_info()[v] = base;
  s.in_head()[v] = -1;
  s.out_head()[v] = -1;
  s.in_tail()[v] = -1;
  s.out_tail()[v] = -1;
  s.n_aligned()[v] = 0;
  s.cov()[v] = 0;
  s.last_label()[v] = -1;
  return v;
}

__device__ __forceinline__ void add_edge(Slot& s, CCaps& caps, int tail, int head, int weight) {
  for (int e = s.out_head()[tail]; e != -1; e = s.e_next_out()[e]) {
    if (s.e_head()[e] == head) {
      s.e_weight()[e] = s.e_weight()[e] + weight;
      touch(s, tail, s.n_seqs);
      touch(s, head, s.n_seqs);
      return;
    }
  }
  if (s.n_edges >= static_cast<int>(caps.edges)) {
    s.overflow = true;
    return;
  }
  const int e = s.n_edges++;
  s.e_tail()[e] = tail;
  s.e_head()[e] = head;
  s.e_weight()[e] = weight;
  s.e_next_in()[e] = -1;
  s.e_next_out()[e] = -1;
  if (s.out_tail()[tail] == -1) {
    s.out_head()[tail] = e;
  } else {
    s.e_next_out()[s.out_tail()[tail]] = e;
  }
  s.out_tail()[tail] = e;
  if (s.in_tail()[head] == -1) {
    s.in_head()[head] = e;
  } else {
    s.e_next_in()[s.in_tail()[head]] = e;
  }
  s.in_tail()[head] = e;
  s.add_in(head, s.node_info()[head], tail);
  touch(s, tail, s.n_seqs);
  touch(s, head, s.n_seqs);
}

// DFS topological order over nodes with keep[v] (all nodes when keep is
// null); writes node ids in rank order to out, returns how many.
__device__ __forceinline__ int topo_sort(Slot& s, const uint8_t* keep, int32_t* out, int stack_cap) {
  const int n = s.n_nodes;
  for (int v = lane_id(); v < n; v += kWave) {
    s.mark()[v] = 0;
    s.lead()[v] = 1;
  }
  wave_sync();
  int count = 0;
  for (int root = 0; root < n; ++root) {
    if (keep != nullptr && keep[root] == 0) {
      continue;
    }
    if (s.mark()[root] != 0) {
      continue;
    }
    int top = 0;
    s.stack()[top++] = root;
    while (top > 0) {
      const int v = uniform(s.stack()[top - 1]);
      bool ready = true;
      if (s.mark()[v] != 2) {
        for (int e = uniform(s.in_head()[v]); e != -1; e = uniform(s.e_next_in()[e])) {
          const int u = uniform(s.e_tail()[e]);
          if (keep != nullptr && keep[u] == 0) {
            continue;
          }
          if (s.mark()[u] != 2) {
            if (top >= stack_cap) {
              s.overflow = true;
              return count;
            }
            s.stack()[top++] = u;
            ready = false;
          }
        }
        if (s.lead()[v] != 0) {
          const int na = s.n_aligned()[v];
          for (int k = 0; k < na; ++k) {
            const int a = uniform(s.aligned()[v * kAligned + k]);
            if (keep != nullptr && keep[a] == 0) {
              continue;
            }
            if (s.mark()[a] != 2) {
              if (top >= stack_cap) {
                s.overflow = true;
                return count;
              }
              s.stack()[top++] = a;
              s.lead()[a] = 0;
              ready = false;
            }
          }
        }
        if (ready) {
          s.mark()[v] = 2;
          if (s.lead()[v] != 0) {
            if (count + 1 + s.n_aligned()[v] > n) {
              s.overflow = true;
              return count;
            }
            out[count++] = v;
            const int na = s.n_aligned()[v];
            for (int k = 0; k < na; ++k) {
              const int a = uniform(s.aligned()[v * kAligned + k]);
              if (keep == nullptr || keep[a] != 0) {
                out[count++] = a;
              }
            }
          }
        } else {
          s.mark()[v] = 1;
        }
      }
      if (ready) {
        --top;
      }
    }
  }
  return count;
}

// ---- DP ----

// Inclusive prefix max over the 64 lanes with DPP row shifts and row
// broadcasts (no LDS crossbar traffic).

__device__ __forceinline__ int32_t wave_prefix_max(int32_t x) {
  // within rows of 16 lanes: shifts 1, 2, 4, 8 (lanes shifted in from
  // outside the row keep the identity). INT32_MIN, the identity of max, lets
  // each move fold into one v_max_i32 with a DPP source.
  constexpr int32_t kId = INT32_MIN;
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x111, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x112, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x114, 0xf, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x118, 0xf, 0xf, false));
  // across rows: lane 15 into rows 1 and 3, lane 31 into rows 2 and 3
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x142, 0xa, 0xf, false));
  x = max(x, __builtin_amdgcn_update_dpp(kId, x, 0x143, 0xc, 0xf, false));
  return x;
}

// Value of the previous lane (lane 0 gets `first`), via DPP wave shift.
__device__ __forceinline__ int32_t wave_shift_right(int32_t x, int32_t first) {
  return __builtin_amdgcn_update_dpp(first, x, 0x138, 0xf, 0xf, false);
}

// Wavefront-scope ordering of LDS/global traffic between lanes of this wave
// (a single-wave workgroup needs no s_barrier; the fence keeps the compiler
// from moving memory operations across it).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Waits for this wave's outstanding global stores (vmcnt(0)).
__device__ __forceinline__ void wait_stores() { __builtin_amdgcn_s_waitcnt(0x0F70); }

constexpr int kRowMetaSink = 0x100;
// Bits 10..14 of a row's meta word: where the row's scores live while later
// rows need them. Slots 0..kMaxLdsSlots-1 are LDS rows; kSlotGlobal rows go
// through the slot's global H matrix; kSlotNone rows are read by no later row.
constexpr int kRowMetaSlotShift = 10;
constexpr int kSlotGlobal = 30;
constexpr int kSlotNone = 31;
constexpr int kMaxLdsSlots = 30;
// Predecessor list entries: DP row in the low 24 bits, its slot above.
constexpr int kPredRowBits = 24;
constexpr int kPredRowMask = (1 << kPredRowBits) - 1;

// LDS score rows keep column j at element j + kColShift, so that the four
// columns of a lane's strip (j0 = 1 + 4k) start on an aligned quad.
constexpr int kColShift = 3;

// Code matrix index of column j inside a row: columns 1..L at j - 1 (aligned
// quads per strip), column 0 at the row's last element (pitch >= L + 9).
__device__ __forceinline__ int code_index(int j, int pitch) { return j == 0 ? pitch - 1 : j - 1; }

template <typename T>
struct Quad;

template <>
struct Quad<int16_t> {
  static __device__ __forceinline__ void load(const int16_t* p, int32_t* v) {
    const uint2 q = *reinterpret_cast<const uint2*>(p);
    v[0] = static_cast<int16_t>(q.x & 0xffffu);
    v[1] = static_cast<int32_t>(q.x) >> 16;
    v[2] = static_cast<int16_t>(q.y & 0xffffu);
    v[3] = static_cast<int32_t>(q.y) >> 16;
  }
  static __device__ __forceinline__ void store(int16_t* p, const int32_t* v) {
    uint2 q;
    q.x = (static_cast<uint32_t>(v[0]) & 0xffffu) | (static_cast<uint32_t>(v[1]) << 16);
    q.y = (static_cast<uint32_t>(v[2]) & 0xffffu) | (static_cast<uint32_t>(v[3]) << 16);
    *reinterpret_cast<uint2*>(p) = q;
  }
};

template <>
struct Quad<int32_t> {
  static __device__ __forceinline__ void load(const int32_t* p, int32_t* v) {
    const int4 q = *reinterpret_cast<const int4*>(p);
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    v[3] = q.w;
  }
  static __device__ __forceinline__ void store(int32_t* p, const int32_t* v) {
    *reinterpret_cast<int4*>(p) = make_int4(v[0], v[1], v[2], v[3]);
  }
};

// All DP rows of one layer. Lanes own 4-column strips of 256-column tiles;
// predecessor rows come from their LDS slots (the global H matrix for rows
// that found no free slot); the horizontal gap chain is a wave prefix-max;
// every cell stores the first move that reproduces its score (diagonal,
// then vertical, each over predecessors in in-edge order, then horizontal).
// Returns the DP row of the end cell: the first sink row with the highest
// score in column L.
//
// The global-H branch waits for its own loads before leaving the branch, so
// the common LDS path never waits on vector memory (on gfx9 the vector memory
// counter also counts the traceback-code stores of earlier rows). Strips
// that start past column L are idle; the columns past L inside the last
// strip are computed from padding and never read back.
// General DP (any score width, layer length and in-degree).
template <typename T>
__device__ __forceinline__ int dp_layer(CParams& P, const Slot& s, uint8_t* lds, int V, int L,
                        int* best_score, bool* tied) {
  static_assert(kStrip == 4, "strips are loaded and stored as quads");
  const int lane = lane_id();
  const int pitch = static_cast<int>(P.caps.cols);
  // scores as uniform registers (a select between two parameter fields
  // would otherwise become a per-lane load from the selected address)
  const int32_t gap = uniform(P.gap);
  const int32_t match = uniform(P.match);
  const int32_t mismatch = uniform(P.mismatch);
  T* ring = reinterpret_cast<T*>(lds);
  const uint8_t* seq = lds + align_up(static_cast<uint64_t>(P.ring_rows) * pitch * 2, 16);
  int32_t best = kNegInf;
  int best_row = 0;
  int ties = 0;
  const int total_preds = uniform(s.pred_off()[V]);
  // rows are processed in chunks of 64: lane k holds the metadata of row
  // r0 + k and a 128-entry window of the predecessor list, broadcast per row
  for (int r0 = 1; r0 <= V; r0 += kWave) {
  const int rk = r0 + lane;
  int off_v = 0, end_v = 0, meta_v = 0;
  if (rk <= V) {
    off_v = s.pred_off()[rk - 1];
    end_v = s.pred_off()[rk];
    meta_v = s.row_meta()[rk - 1];
  }
  const int base = __builtin_amdgcn_readlane(off_v, 0);
  const int pr0 = base + lane < total_preds ? s.pred_rows()[base + lane] : 0;
  const int pr1 = base + kWave + lane < total_preds ? s.pred_rows()[base + kWave + lane] : 0;
  // (up to four entries per row of the chunk without a reload)
  const int pr2 =
      base + 2 * kWave + lane < total_preds ? s.pred_rows()[base + 2 * kWave + lane] : 0;
  const int pr3 =
      base + 3 * kWave + lane < total_preds ? s.pred_rows()[base + 3 * kWave + lane] : 0;
  // complete the chunk's loads here: otherwise the row loop below would wait
  // for them (and for every code store before them) on each row
  wait_stores();
  const int chunk = min(kWave, V - r0 + 1);
  for (int rr = 0; rr < chunk; ++rr) {
    const int r = r0 + rr;
    const int off = __builtin_amdgcn_readlane(off_v, rr);
    const int np = __builtin_amdgcn_readlane(end_v, rr) - off;
    const int meta = __builtin_amdgcn_readlane(meta_v, rr);
    auto pred_at = [&](int k) -> int {
      const int idx = off + k - base;
      if (idx < kWave) return __builtin_amdgcn_readlane(pr0, idx);
      if (idx < 2 * kWave) return __builtin_amdgcn_readlane(pr1, idx - kWave);
      if (idx < 3 * kWave) return __builtin_amdgcn_readlane(pr2, idx - 2 * kWave);
      if (idx < 4 * kWave) return __builtin_amdgcn_readlane(pr3, idx - 3 * kWave);
      const int e = uniform(s.pred_rows()[off + k]);
      wait_stores();
      return e;
    };
    const uint32_t b = static_cast<uint32_t>(meta & 0xff);
    const int own = (meta >> kRowMetaSlotShift) & 31;
    T* Hr = ring + (own < kSlotGlobal ? own : 0) * pitch;
    int32_t* Hg = s.H_row(r, meta, pitch);
    uint16_t* Cr = s.code() + static_cast<int64_t>(r) * pitch;

    // column 0: max over predecessors of their column 0, plus gap
    int32_t c0 = kNegInf;
    int k0 = 0;
    for (int k = 0; k < np; ++k) {
      const int e = pred_at(k);
      const int p = e & kPredRowMask;
      const int sl = static_cast<unsigned>(e) >> kPredRowBits;
      int32_t h0;
      if (p == 0) {
        h0 = 0;
      } else if (sl < kSlotGlobal) {
        h0 = ring[sl * pitch + kColShift];
      } else {
        h0 = uniform(s.H_row(p, pitch)[0]);
        wait_stores();
      }
      if (h0 + gap > c0) {
        c0 = h0 + gap;
        k0 = k;
      }
    }
    if (lane == 0) {
      if (own < kSlotGlobal) Hr[kColShift] = static_cast<T>(c0);
      if (own == kSlotGlobal) Hg[0] = c0;
      Cr[pitch - 1] = kCodeVert | static_cast<uint16_t>(k0);
    }
    int32_t carry = c0;
    int32_t h_last = kNegInf;

    for (int t0 = 1; t0 <= L; t0 += kTile) {
      const int j0 = t0 + lane * kStrip;
      const bool live = j0 <= L;
      const int jr = live ? j0 : 1;  // idle strips read column 0..4 (in bounds)
      const uint32_t w4 = *reinterpret_cast<const uint32_t*>(seq + (jr - 1));
      int32_t sc[kStrip];
      bool in[kStrip];
#pragma unroll
      for (int u = 0; u < kStrip; ++u) {
        sc[u] = ((w4 >> (8 * u)) & 0xffu) == b ? match : mismatch;
        in[u] = j0 + u <= L;
      }
      int32_t bd[kStrip], bv[kStrip];
      uint32_t kk[kStrip];  // diagonal k (low 16 bits), vertical k (high 16 bits)
#pragma unroll
      for (int u = 0; u < kStrip; ++u) {
        bd[u] = kNegInf;
        bv[u] = kNegInf;
        kk[u] = 0;
      }
      for (int k = 0; k < np; ++k) {
        const int e = pred_at(k);
        const int p = e & kPredRowMask;
        const int sl = static_cast<unsigned>(e) >> kPredRowBits;
        int32_t hp[kStrip + 1];
        if (p == 0) {
#pragma unroll
          for (int u = 0; u <= kStrip; ++u) hp[u] = (j0 - 1 + u) * gap;
        } else if (sl < kSlotGlobal) {
          const T* row = ring + sl * pitch + kColShift;
          hp[0] = row[jr - 1];
          Quad<T>::load(row + jr, hp + 1);
        } else {
          const int32_t* row = s.H_row(p, pitch);
#pragma unroll
          for (int u = 0; u <= kStrip; ++u) {
            const int j = j0 - 1 + u;
            hp[u] = j <= L ? row[j] : kNegInf;
          }
          wait_stores();
        }
#pragma unroll
        for (int u = 0; u < kStrip; ++u) {
          const int32_t d = hp[u] + sc[u];
          const int32_t v = hp[u + 1] + gap;
          const bool dg = d > bd[u];
          const bool vg = v > bv[u];
          bd[u] = dg ? d : bd[u];
          bv[u] = vg ? v : bv[u];
          kk[u] = dg ? ((kk[u] & 0xffff0000u) | static_cast<uint32_t>(k)) : kk[u];
          kk[u] = vg ? ((kk[u] & 0xffffu) | (static_cast<uint32_t>(k) << 16)) : kk[u];
        }
      }
      // horizontal chain: H[j] = j*g + max_{k<=j} (t_k - k*g)
      int32_t pm = kNegInf;
      int32_t pre[kStrip];
#pragma unroll
      for (int u = 0; u < kStrip; ++u) {
        const int j = j0 + u;
        const int32_t t = max(bd[u], bv[u]);
        pre[u] = in[u] ? t - j * gap : kNegInf;
        pm = max(pm, pre[u]);
        pre[u] = pm;
      }
      const int32_t incl = wave_prefix_max(pm);
      const int32_t excl = wave_shift_right(incl, kNegInf);
      const int32_t in_carry = max(excl, carry - (t0 - 1) * gap);
      int32_t h[kStrip];
      uint32_t cd[kStrip];
#pragma unroll
      for (int u = 0; u < kStrip; ++u) {
        h[u] = max(pre[u], in_carry) + (j0 + u) * gap;
        const uint32_t c_diag = kCodeDiag | (kk[u] & 0xffffu);
        const uint32_t c_vert = kCodeVert | (kk[u] >> 16);
        cd[u] = bd[u] == h[u] ? c_diag : (bv[u] == h[u] ? c_vert : kCodeHorz);
      }
      if (live) {
        uint2 q;
        q.x = cd[0] | (cd[1] << 16);
        q.y = cd[2] | (cd[3] << 16);
        *reinterpret_cast<uint2*>(Cr + (j0 - 1)) = q;
        if (own < kSlotGlobal) {
          Quad<T>::store(Hr + kColShift + j0, h);
        }
      }
      if (own == kSlotGlobal) {
#pragma unroll
        for (int u = 0; u < kStrip; ++u) {
          if (in[u]) Hg[j0 + u] = h[u];
        }
      }
      // value of the tile's last column: carry into the next tile and, in
      // the last tile, the end-cell candidate
      const int last_col = min(L, t0 + kTile - 1);
      const int owner = (last_col - t0) / kStrip;
      const int last_u = (last_col - t0) % kStrip;
      int32_t lv = h[0];
#pragma unroll
      for (int u = 1; u < kStrip; ++u) {
        if (u == last_u) lv = h[u];
      }
      carry = __builtin_amdgcn_readlane(lv, owner);
      h_last = carry;
    }
    if ((meta & kRowMetaSink) != 0) {
      if (lane == 0) {
        s.sink_score()[r] = h_last;
      }
      if (h_last > best) {
        best = h_last;
        best_row = r;
        ties = 0;
      } else if (h_last == best) {
        ++ties;
      }
    }
    if (own == kSlotGlobal) {
      wait_stores();
    }
    wave_fence();
  }
  }
  *best_score = best;
  *tied = ties > 0;
  return best_row;
}

// ---- packed 16-bit pairs: two DP columns per 32-bit register ----

typedef unsigned short __attribute__((ext_vector_type(2))) U16x2;

__device__ __forceinline__ U16x2 as_u16x2(uint32_t x) { return __builtin_bit_cast(U16x2, x); }
__device__ __forceinline__ uint32_t pk_bits(U16x2 x) { return __builtin_bit_cast(uint32_t, x); }
// per-half wrapping add / subtract, unsigned min, multiply-add
__device__ __forceinline__ uint32_t pk_add(uint32_t a, uint32_t b) {
  return pk_bits(as_u16x2(a) + as_u16x2(b));
}
__device__ __forceinline__ uint32_t pk_sub(uint32_t a, uint32_t b) {
  return pk_bits(as_u16x2(a) - as_u16x2(b));
}
__device__ __forceinline__ uint32_t pk_min_u(uint32_t a, uint32_t b) {
  return pk_bits(__builtin_elementwise_min(as_u16x2(a), as_u16x2(b)));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
  return pk_bits(as_u16x2(a) * as_u16x2(b) + as_u16x2(c));
}
// unsigned max; of a with the high half of b; inclusive prefix max inside the
// pair; saturating subtract
__device__ __forceinline__ uint32_t pk_max_u(uint32_t a, uint32_t b) {
  return pk_bits(__builtin_elementwise_max(as_u16x2(a), as_u16x2(b)));
}
__device__ __forceinline__ uint32_t pk_max_hi_u(uint32_t a, uint32_t b) {
  const U16x2 v = as_u16x2(b);
  return pk_bits(__builtin_elementwise_max(as_u16x2(a), __builtin_shufflevector(v, v, 1, 1)));
}
__device__ __forceinline__ uint32_t pk_scan_u(uint32_t a) {
  const U16x2 v = as_u16x2(a);
  return pk_bits(__builtin_elementwise_max(v, __builtin_shufflevector(v, v, 0, 0)));
}
__device__ __forceinline__ uint32_t pk_sub_sat(uint32_t a, uint32_t b) {
  return pk_bits(__builtin_elementwise_sub_sat(as_u16x2(a), as_u16x2(b)));
}
__device__ __forceinline__ uint32_t pk_splat(int32_t v) {
  return (static_cast<uint32_t>(v) & 0xffffu) * 0x10001u;
}

// ---- packed DP rows (dp_rows) ----
//
// One pass of the wave per DP row: lane k owns columns kW .. kW + W - 1 of
// columns 0..L (column 0 is lane 0's first), two columns per register. Every
// value is kept as G = H - j * gap + bias in unsigned 16 bits: a horizontal
// move keeps G, a vertical one adds gap, a diagonal one s - gap, so the
// horizontal chain is a plain prefix max and column 0 is an ordinary column
// (the diagonal into it comes from column -1, a value below every other).
// G falls by |gap| per row at most and rises by max(s) - gap per column, so
// the rows fit 16 bits while |gap| (V + 2) + (max(s) - gap)(L + 1) does
// (rows_fit_16).
//
// A row's scores live in its LDS slot, column j at element j; a lane reads
// only what it wrote itself, so rows need no ordering between lanes. The row's
// base selects the substitution scores with one byte permute per pair: the
// pair's letters are kept as selectors into an eight-byte table (low bytes of
// s - gap for A, C, G, T, then the high bytes) that is built per row in scalar
// registers.
//
// What a row stores for the traceback: per column a move kind (bit 1: the
// diagonal reaches the cell's score, bit 0: the vertical does; diagonal is
// taken before vertical before horizontal) and, for rows with two to four
// predecessors, the index of the first predecessor with the column's best
// score (2 bits each): the diagonal into column j takes the one of column
// j - 1, the vertical the one of column j, which is spoa's choice. Rows of
// more than four predecessors or of the virtual start row store 16-bit codes,
// column j at element j. They take the general form of the DP, and so do rows
// that live in global memory or read one that does; these keep move records,
// because a 16-bit code costs the traceback a round trip per move: with two
// LDS rows 3,000 windows of 500 bp at 20 layers spent 22.7 wave-seconds in it
// and 3.7 with records. A row of a letter other than A, C, G and T compares it
// with the layer's letters and goes the way of the others from there: those
// windows in lower case take 19.7 wave-seconds of DP, 11.1 in upper case and
// 36.6 in the general form.
//
// The rows are bound by their instructions: a wave alone issues one about
// every 8 cycles, and 4 waves per SIMD share the issue slots. A row whose one
// predecessor is the row before takes 93 instructions at W = 8, 22 of them
// scalar (the form with per-row predecessor lists, a separate column 0 and
// 16-bit codes took 212 over all rows; the one that prepared each row's
// scores at its own start, with no-ops in the gaps of the chain, 122). One
// 500 bp window at 30 layers: DP 17.5 -> 8.5 -> 6.8 ms; 9,980 windows of
// 500 bp at 52 layers: DP 521 -> 291 -> 252 wave-seconds.

// Row descriptor: number of predecessors (0: the general form), 8 x the code
// of the row's base, own slot, slots of up to four predecessors, whether the
// single predecessor is the row before, and the sink flag. A row of another
// letter has kRecOther and no number and code (the number is in its meta
// word); the general form has the sink flag and kRecMoves, set when the row
// keeps a move record (also with kRecOther).
constexpr uint32_t kRecPreds = 7u;
constexpr uint32_t kRecMoves = 8u;
constexpr uint32_t kRecOther = 16u;
constexpr uint32_t kRecBase = 0x18u;
constexpr int kRecOwnShift = 5;
constexpr int kRecPredShift = 10;
constexpr uint32_t kRecChain = 1u << 30;
constexpr uint32_t kRecSink = 1u << 31;
constexpr uint32_t kRecMaxPreds = 4;

// Layout of a row's move record: per lane row_record_bytes(W) bytes, the kinds in
// the first half and the predecessor indices in the second; in each half the
// even columns' fields are followed by the odd columns', the first column in
// the highest bits (groups of eight column pairs for W > 16).
__device__ __forceinline__ int row_record_bytes(int W) { return W == 4 ? 2 : W == 8 ? 4 : W <= 16 ? 8 : 16; }

// 16-bit rows hold every value of the layer (see above), with room for the
// sums formed on the way. bias: the value of G = 0.
__device__ __forceinline__ bool rows_fit_16(int match, int mismatch, int gap, int V, int L,
                                            int* bias) {
  const int top = max(match, mismatch);
  const int max_abs = max(max(abs(match), abs(mismatch)), abs(gap));
  if (gap > 0 || max_abs > 1024) return false;
  const int m = 2 * max_abs;
  const int64_t low = static_cast<int64_t>(-gap) * (V + 2) + 4 * m;
  const int64_t high = static_cast<int64_t>(max(top - gap, 0)) * (L + 1) + 2 * m;
  *bias = static_cast<int>(low);
  return low + high <= 65535;
}

// Lane-private LDS bytes of a row slot (an LDS address).
typedef __attribute__((address_space(3))) uint8_t LByte;
typedef __attribute__((address_space(3))) uint32_t LWord;
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) U32x4 LQuad;
typedef __attribute__((address_space(3))) U32x2 LPair;

template <int W>
__device__ __forceinline__ void lds_row_load(uint32_t at, uint32_t* v) {
  if constexpr (W % 8 == 0) {
#pragma unroll
    for (int q = 0; q < W / 8; ++q) {
      const U32x4 x = ((const LQuad*)(size_t)at)[q];
      v[4 * q] = x.x;
      v[4 * q + 1] = x.y;
      v[4 * q + 2] = x.z;
      v[4 * q + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < W / 4; ++q) {
      const U32x2 x = ((const LPair*)(size_t)at)[q];
      v[2 * q] = x.x;
      v[2 * q + 1] = x.y;
    }
  }
}

template <int W>
__device__ __forceinline__ void lds_row_store(uint32_t at, const uint32_t* v) {
  if constexpr (W % 8 == 0) {
#pragma unroll
    for (int q = 0; q < W / 8; ++q) {
      ((LQuad*)(size_t)at)[q] = U32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    }
  } else {
#pragma unroll
    for (int q = 0; q < W / 4; ++q) ((LPair*)(size_t)at)[q] = U32x2{v[2 * q], v[2 * q + 1]};
  }
}

// Inclusive prefix max over the lanes of unsigned words (0 is the identity,
// which lanes without a source read).
// fill(x, k), k = 0..5, is called after each step.
template <typename Fill>
__device__ __forceinline__ uint32_t wave_prefix_max_u(uint32_t x, Fill fill) {
  const auto step = [](uint32_t v, auto ctrl, auto rows) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        0, static_cast<int>(v), decltype(ctrl)::value, decltype(rows)::value, 0xf, false));
  };
  x = max(x, step(x, std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{}));
  fill(x, 0);
  x = max(x, step(x, std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{}));
  fill(x, 1);
  x = max(x, step(x, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{}));
  fill(x, 2);
  x = max(x, step(x, std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{}));
  fill(x, 3);
  x = max(x, step(x, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}));
  fill(x, 4);
  x = max(x, step(x, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{}));
  fill(x, 5);
  return x;
}
__device__ __forceinline__ uint32_t wave_prefix_max_u(uint32_t x) {
  return wave_prefix_max_u(x, [](uint32_t&, int) {});
}

// x of the previous lane; lane 0 keeps its value of `old` (a register that
// is passed from row to row, so that lane 0's constant costs nothing).
__device__ __forceinline__ uint32_t shift_into(uint32_t old, uint32_t x) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
      static_cast<int>(old), static_cast<int>(x), 0x138, 0xf, 0xf, false));
}

// Ties a value to its place among the other pinned ones (no instruction).
__device__ __forceinline__ void pin(uint32_t& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin_scalar(uint32_t& x) { asm volatile("" : "+s"(x)); }

// x of the previous lane, 0 in lane 0.
__device__ __forceinline__ uint32_t shift_lanes(uint32_t x) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0x138, 0xf, 0xf, true));
}

// One row from its best predecessor scores in h: diagonal (scores sub from
// the letters; lane 0's column 0 has no letter: its first half is 0, which
// keeps the diagonal below every score) and vertical candidates, horizontal
// chain, scores into h.
//
// A packed instruction's result is read by the second instruction after it at
// the earliest, a lane's by a DPP read in the third: the pairs go through each
// step together, and fill(k), k = 0..8, issues a part of the next row's work
// (one or two instructions, free of this row's results) in the gaps of the
// chain and of the prefix max, which would be no-ops otherwise.
template <int W, typename Fill>
__device__ __forceinline__ void row_scores(uint32_t* h, const uint32_t* sub, uint32_t gap_pair,
                                           uint32_t* bd, uint32_t* bv, Fill fill) {
  constexpr int H2 = W / 2;
  const uint32_t prev = shift_lanes(h[H2 - 1]);
  uint32_t pre[H2];
#pragma unroll
  for (int q = 0; q < H2; ++q) bv[q] = pk_add(h[q], gap_pair);
#pragma unroll
  for (int q = 0; q < H2; ++q) {
    // G[p][j - 1] of the pair
    pre[q] = __builtin_amdgcn_alignbit(h[q], q == 0 ? prev : h[q - 1], 16);
  }
#pragma unroll
  for (int q = 0; q < H2; ++q) bd[q] = pk_add(pre[q], sub[q]);
#pragma unroll
  for (int q = 0; q < H2; ++q) pre[q] = pk_max_u(bd[q], bv[q]);
#pragma unroll
  for (int q = 0; q < H2; ++q) pre[q] = pk_scan_u(pre[q]);
#pragma unroll
  for (int q = 0; q < H2; ++q) pin(pre[q]);
#pragma unroll
  for (int q = 1; q < H2; ++q) {
    pre[q] = pk_max_hi_u(pre[q], pre[q - 1]);
    pin(pre[q]);
    if (q >= H2 - 3) fill(q - H2 + 3);
  }
  // (the whole word goes through the scan: its high half, the strip's
  // maximum, decides)
  const uint32_t excl = shift_lanes(
      wave_prefix_max_u(pre[H2 - 1], [&](uint32_t& x, int k) {
        pin(x);
        fill(3 + k);
      }));
#pragma unroll
  for (int q = 0; q < H2; ++q) h[q] = pk_max_hi_u(pre[q], excl);
}

template <int W>
__device__ __forceinline__ void row_kinds(const uint32_t* h, const uint32_t* bd,
                                          const uint32_t* bv, uint32_t* acc) {
  constexpr int H2 = W / 2;
#pragma unroll
  for (int q = 0; q < H2; ++q) {
    // 1 where the candidate reaches the score (it is never above it)
    const uint32_t below = pk_sub(h[q], 0x00010001u);
    const uint32_t kind = (pk_sub_sat(bd[q], below) << 1) | pk_sub_sat(bv[q], below);
    acc[q / 8] = (q % 8) == 0 ? kind : (acc[q / 8] << 2) | kind;
  }
}

// Scores of a pair whose letters are not all A, C, G or T: those match no row
// of these four (a row of another letter compares letters).
constexpr uint32_t kOddLetter = 0x0d0du;  // their selector
__device__ __forceinline__ uint32_t odd_letters(uint32_t sub, uint32_t sel, uint32_t miss) {
  const uint32_t m = ((sel >> 3) & sel & 0x00010001u) * 0xffffu;
  return (sub & ~m) | (miss & m);
}

// One DP layer in packed rows; the end cell as dp_layer. W: 4, 8, 12, 16 or
// 20 with 64 W > L. kPlain: the layer holds A, C, G and T only (functions of
// their own: a test per row cost 2%).
template <int W, bool kPlain>
__device__ __forceinline__ int dp_rows(CParams& P, const Slot& s, uint32_t lds, int V, int L,
                                       int bias, int* best_score, bool* tied) {
  constexpr int H2 = W / 2;
  constexpr int NA = (H2 + 7) / 8;
  const int lane = lane_id();
  const int pitch = static_cast<int>(P.caps.cols);
  const int32_t gap = uniform(P.gap);
  const int32_t match = uniform(P.match);
  const int32_t mismatch = uniform(P.mismatch);
  const uint32_t row_bytes = static_cast<uint32_t>(pitch) * 2;
  const LByte* seq = (const LByte*)(size_t)(
      lds + static_cast<uint32_t>(align_up(static_cast<uint64_t>(P.ring_rows) * row_bytes, 16)));
  // Lanes past the last column run along (every lane's registers stay whole for
  // the row loop's readlanes): their scores and moves go to the row's columns
  // past L, those that find no room there to its last ones (a row has at least
  // L + 24 columns, so these are past L as well).
  const bool live = lane < (L + W) / W;
  const uint32_t strip =
      lds + min(static_cast<uint32_t>(lane) * (2 * W), row_bytes - 2 * W);
  // letters of the strip (column j holds letter j - 1) as table selectors
  uint32_t sel[H2];
#pragma unroll
  for (int q = 0; q < H2; ++q) {
    uint32_t x = 0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int idx = lane * W + 2 * q + u - 1;
      const int c = idx >= 0 && idx < L ? static_cast<int>(seq[idx]) : 'A';
      const int code = ((c >> 1) ^ (c >> 2)) & 3;
      const bool is_base = static_cast<int>((0x54474341u >> (8 * code)) & 0xffu) == c;
      // (a selector byte of 0x0c gives 0: column 0)
      x |= (idx < 0    ? 0x0c0cu
            : !kPlain && !is_base ? kOddLetter
                       : static_cast<uint32_t>(code) * 0x0101u + 0x0400u)
           << (16 * u);
    }
    sel[q] = x;
  }
  const uint32_t gap_pair = pk_splat(gap);
  // score tables: s - gap of a mismatch in every byte pair, and the change
  // to the match in the pair of code 0
  const uint32_t miss = static_cast<uint32_t>(mismatch - gap) & 0xffffu;
  const uint32_t flip = (static_cast<uint32_t>(match - gap) & 0xffffu) ^ miss;
  const uint64_t table0 = static_cast<uint64_t>((miss >> 8) * 0x01010101u) << 32 |
                          (miss & 0xffu) * 0x01010101u;
  const uint64_t table1 = static_cast<uint64_t>(flip >> 8) << 32 | (flip & 0xffu);
  // 1 in both halves, opaque to the optimizer (a visible 1 turns min(x, 1)
  // into compares and selects per half)
  uint32_t one = 0x00010001u;
  asm volatile("" : "+s"(one));
  const int end_lane = L / W, end_u = L % W;
  int32_t best = kNegInf;
  int best_row = 0;
  int ties = 0;
  const int total_preds = uniform(s.pred_off()[V]);
  uint32_t cur[H2];  // the scores of the row before
#pragma unroll
  for (int q = 0; q < H2; ++q) cur[q] = 0;
  // position in seq of the letter of the strip's first column (-1: column 0
  // has none; lanes past the last column read the bytes behind the layer)
  [[maybe_unused]] const int letters = min(lane * W, pitch - W) - 1;
  GByte* const codes = (GByte*)s.code();
  uint32_t rec_lane = min(static_cast<uint32_t>(lane * row_record_bytes(W)),
                          row_bytes - static_cast<uint32_t>(row_record_bytes(W)));
  // (chunks of 63 rows: the last lane's descriptor is 0 and ends the row loop)
  constexpr int kChunk = kWave - 1;
  for (int r0 = 1; r0 <= V; r0 += kChunk) {
    const int rk = r0 + lane;
    uint32_t desc_v = 0;
    if (lane < kChunk && rk <= V) desc_v = s.row_rec()[rk - 1].x;
    const int chunk = uniform(min(kChunk, V - r0 + 1));
    // what the rows of the general form need of this chunk
    int off_v = 0, end_v = 0, meta_v = 0, base = 0, pr0 = 0, pr1 = 0;
    if (__any(lane < kChunk && rk <= V && (desc_v & kRecPreds) == 0)) {
      if (rk <= V) {
        off_v = s.pred_off()[rk - 1];
        end_v = s.pred_off()[rk];
        meta_v = s.row_meta()[rk - 1];
      }
      base = __builtin_amdgcn_readlane(off_v, 0);
      pr0 = base + lane < total_preds ? s.pred_rows()[base + lane] : 0;
      pr1 = base + kWave + lane < total_preds ? s.pred_rows()[base + kWave + lane] : 0;
    }
    // complete the chunk's loads here: otherwise the row loop would wait for
    // them (and for every store issued before them) on each row
    wait_stores();
    GByte* record = codes + static_cast<int64_t>(r0 - 1) * row_bytes;  // of the row before
    // the next row's descriptor and substitution scores, a piece at a time
    uint32_t d = 0, d_next = 0;
    uint64_t table = 0;
    uint32_t sub[H2];
    const auto next_desc = [&](int rr) {
      d_next = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(desc_v), rr));
      pin_scalar(d_next);
    };
    const auto next_table = [&]() {
      table = table0 ^ (table1 << (d_next & kRecBase));
      asm volatile("" : "+s"(table));
    };
    const auto next_sub = [&](int q) {
      sub[q] = __builtin_amdgcn_perm(static_cast<uint32_t>(table >> 32),
                                     static_cast<uint32_t>(table), sel[q]);
      pin(sub[q]);
    };
    const auto next_odd = [&]() {
      if constexpr (!kPlain) {
#pragma unroll
        for (int q = 0; q < H2; ++q) {
          uint32_t letters = sel[q];
          pin(letters);  // (its masks are not kept in registers)
          sub[q] = odd_letters(sub[q], letters, miss * 0x10001u);
        }
      }
    };
    const auto next_row = [&](int rr) {
      next_desc(rr);
      next_table();
#pragma unroll
      for (int q = 0; q < H2; ++q) next_sub(q);
      next_odd();
      d = d_next;
    };
    const auto sink_row = [&](int r) {
      uint32_t last = cur[0];
#pragma unroll
      for (int q = 1; q < H2; ++q) {
        uint32_t v = cur[q];
        asm volatile("" : "+v"(v));  // (selected, not indexed through a stack copy)
        if (q == (end_u >> 1)) last = v;
      }
      const uint32_t g = static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(last), end_lane));
      const int32_t h_last =
          static_cast<int32_t>((end_u & 1) ? g >> 16 : g & 0xffffu) - bias + L * gap;
      if (lane == 0) s.sink_score()[r] = h_last;
      if (h_last > best) {
        best = h_last;
        best_row = r;
        ties = 0;
      } else if (h_last == best) {
        ++ties;
      }
    };
    const auto store_moves = [&](const uint32_t* acc, const uint32_t* ack) {
      pin(rec_lane);  // (stays a 32-bit offset to the uniform row address)
      GByte* at = record + rec_lane;
      if constexpr (W == 4) {
        const uint32_t a = (acc[0] | (acc[0] >> 12)) & 0xffu;
        const uint32_t k = (ack[0] | (ack[0] >> 12)) & 0xffu;
        *(__attribute__((address_space(1))) uint16_t*)at = static_cast<uint16_t>(a | (k << 8));
      } else if constexpr (W == 8) {
        *(__attribute__((address_space(1))) uint32_t*)at =
            __builtin_amdgcn_perm(ack[0], acc[0], 0x06040200u);
      } else if constexpr (NA == 1) {
        *(__attribute__((address_space(1))) U32x2*)at = U32x2{acc[0], ack[0]};
      } else {
        *(__attribute__((address_space(1))) U32x4*)at = U32x4{acc[0], acc[1], ack[0], ack[1]};
      }
    };
    // scores of the strip's letters against a row's of any letter: from the
    // table in a plain layer, letter by letter in another
    const auto letter_scores = [&](uint32_t meta, uint32_t* out) {
      const uint32_t letter = meta & 0xffu;
      if constexpr (kPlain) {
        const uint32_t code = ((letter >> 1) ^ (letter >> 2)) & 3u;
        const bool base = ((0x54474341u >> (8 * code)) & 0xffu) == letter;
        const uint64_t t = base ? table0 ^ (table1 << (8 * code)) : table0;
#pragma unroll
        for (int q = 0; q < H2; ++q) {
          out[q] = __builtin_amdgcn_perm(static_cast<uint32_t>(t >> 32),
                                         static_cast<uint32_t>(t), sel[q]);
        }
      } else {
        const uint32_t hit = miss ^ flip;
#pragma unroll
        for (int q = 0; q < H2; ++q) {
          // (column 0's position is before the first)
          const uint32_t a = seq[q == 0 ? max(letters, 0) : letters + 2 * q];
          const uint32_t b = seq[letters + 2 * q + 1];
          const uint32_t differ = pk_min_u((a | b << 16) ^ letter * 0x10001u, one);
          out[q] = pk_mad(differ, pk_sub(miss * 0x10001u, hit * 0x10001u), hit * 0x10001u);
        }
        if (lane == 0) out[0] &= 0xffff0000u;  // column 0 has no letter
      }
    };
    next_row(0);
    int rr = 0;
    uint32_t np = d & kRecPreds;
    for (;;) {
      // rows of up to four predecessors (a loop of their own: the common
      // ones go through without a taken branch)
      uint32_t np_next = 0;
      while (np != 0) {
        const auto slot_at = [&](int k) {
          return strip + ((d >> (kRecPredShift + 5 * k)) & 31u) * row_bytes;
        };
        uint32_t bd[H2], bv[H2], acc[NA], ack[NA];
#pragma unroll
        for (int a = 0; a < NA; ++a) ack[a] = 0;
        if ((d & kRecChain) == 0) lds_row_load<W>(slot_at(0), cur);
        if (np > 1) {
          // best predecessor score of each column and the first
          // predecessor reaching it (a later one only when better)
          uint32_t kx[H2], p1[H2];
          lds_row_load<W>(slot_at(1), p1);
#pragma unroll
          for (int q = 0; q < H2; ++q) {
            kx[q] = pk_min_u(pk_sub_sat(p1[q], cur[q]), one);
            cur[q] = pk_max_u(cur[q], p1[q]);
          }
          if (np > 2) {
            lds_row_load<W>(slot_at(2), p1);
#pragma unroll
            for (int q = 0; q < H2; ++q) {
              const uint32_t g = pk_min_u(pk_sub_sat(p1[q], cur[q]), one);
              kx[q] = pk_max_u(kx[q], g << 1);
              cur[q] = pk_max_u(cur[q], p1[q]);
            }
            if (np > 3) {
              lds_row_load<W>(slot_at(3), p1);
#pragma unroll
              for (int q = 0; q < H2; ++q) {
                const uint32_t g = pk_min_u(pk_sub_sat(p1[q], cur[q]), one);
                kx[q] = pk_max_u(kx[q], pk_mad(g, 0x00030003u, 0u));
                cur[q] = pk_max_u(cur[q], p1[q]);
              }
            }
          }
#pragma unroll
          for (int q = 0; q < H2; ++q) {
            ack[q / 8] = (q % 8) == 0 ? kx[q] : (ack[q / 8] << 2) | kx[q];
          }
        }
        const uint32_t own = (d >> kRecOwnShift) & 31u;
        uint32_t own_at = 0;
        row_scores<W>(cur, sub, gap_pair, bd, bv, [&](int k) {
          if (k == (H2 == 2 ? 2 : 1)) next_desc(rr + 1);
          if (k == 2) next_table();
          if (k == 3) {
            own_at = strip + own * row_bytes;
            pin(own_at);
          }
          constexpr int kShare = (H2 + 2) / 3;  // pairs per gap
          if (k >= 4 && k < 7) {
#pragma unroll
            for (int q = (k - 4) * kShare; q < min(H2, (k - 3) * kShare); ++q) next_sub(q);
          }
          if (k == 7) {
            record += row_bytes;
            asm volatile("" : "+s"(record));
          }
          if (k == 8) {
            np_next = d_next & kRecPreds;
            pin_scalar(np_next);
            next_odd();
          }
        });
        if (own != static_cast<uint32_t>(kSlotNone)) lds_row_store<W>(own_at, cur);
        row_kinds<W>(cur, bd, bv, acc);
        store_moves(acc, ack);
        if (__builtin_expect((d & kRecSink) != 0, 0)) sink_row(r0 + rr);
        ++rr;
        d = d_next;
        np = np_next;
      }
      if (rr >= chunk) break;
      if ((d & (kRecPreds | kRecOther)) == kRecOther) {
        // a row of another letter: it goes through the loop above with its
        // own scores
        const uint32_t meta = static_cast<uint32_t>(__builtin_amdgcn_readlane(meta_v, rr));
        np = (meta >> kRowMetaPredShift) & kRowMetaPredMask;
        letter_scores(meta, sub);
        continue;
      }
      record += row_bytes;
      {
        uint32_t bd[H2], bv[H2];
        // the general form: any number of predecessors, in LDS, in global
        // memory or the virtual start row; any letters; 16-bit codes
        const int r = r0 + rr;
        const int off = __builtin_amdgcn_readlane(off_v, rr);
        const int n_preds = __builtin_amdgcn_readlane(end_v, rr) - off;
        const int meta = __builtin_amdgcn_readlane(meta_v, rr);
        const int own = (meta >> kRowMetaSlotShift) & 31;
        const int j0 = lane * W;
        uint32_t mx[H2], kx[H2];
#pragma unroll
        for (int q = 0; q < H2; ++q) mx[q] = kx[q] = 0;
        for (int k = 0; k < n_preds; ++k) {
          const int idx = off + k - base;
          int e;
          if (idx < kWave) {
            e = __builtin_amdgcn_readlane(pr0, idx);
          } else if (idx < 2 * kWave) {
            e = __builtin_amdgcn_readlane(pr1, idx - kWave);
          } else {
            e = uniform(s.pred_rows()[off + k]);
          }
          const int p = e & kPredRowMask;
          const int sl = static_cast<int>(static_cast<unsigned>(e) >> kPredRowBits);
          uint32_t pp[H2];
          if (p == 0) {
#pragma unroll
            for (int q = 0; q < H2; ++q) pp[q] = pk_splat(bias);
          } else if (sl == kSlotNone) {
            // the row before, kept in registers only
#pragma unroll
            for (int q = 0; q < H2; ++q) pp[q] = cur[q];
          } else if (sl < kSlotGlobal) {
            lds_row_load<W>(strip + static_cast<uint32_t>(sl) * row_bytes, pp);
          } else {
            const int32_t* row = s.H_row(p, pitch);
#pragma unroll
            for (int q = 0; q < H2; ++q) {
              // (columns past L are never stored: any value does)
              const int ja = min(j0 + 2 * q, L), jb = min(j0 + 2 * q + 1, L);
              pp[q] = (static_cast<uint32_t>(row[ja]) & 0xffffu) |
                      (static_cast<uint32_t>(row[jb]) << 16);
            }
          }
          const uint32_t ks = static_cast<uint32_t>(k) * 0x10001u;
#pragma unroll
          for (int q = 0; q < H2; ++q) {
            const uint32_t g = pk_min_u(pk_sub_sat(pp[q], mx[q]), one);
            kx[q] = pk_mad(g, pk_sub(ks, kx[q]), kx[q]);
            mx[q] = pk_max_u(mx[q], pp[q]);
          }
        }
#pragma unroll
        for (int q = 0; q < H2; ++q) {
          // (a move, so that mx and cur need not share registers)
          asm volatile("v_mov_b32 %0, %1" : "=v"(cur[q]) : "v"(mx[q]));
        }
        letter_scores(static_cast<uint32_t>(meta), sub);
        row_scores<W>(cur, sub, gap_pair, bd, bv, [](int) {});
        if (own < kSlotGlobal) {
          lds_row_store<W>(strip + static_cast<uint32_t>(own) * row_bytes, cur);
        } else if (own == kSlotGlobal) {
          int32_t* Hg = s.H_row(r, meta, pitch);
#pragma unroll
          for (int u = 0; u < W; ++u) {
            if (j0 + u <= L) Hg[j0 + u] = static_cast<int32_t>((cur[u / 2] >> (16 * (u & 1))) & 0xffffu);
          }
        }
        if ((d & kRecMoves) != 0) {
          uint32_t acc[NA], ack[NA];
          row_kinds<W>(cur, bd, bv, acc);
#pragma unroll
          for (int q = 0; q < H2; ++q) {
            ack[q / 8] = (q % 8) == 0 ? kx[q] : (ack[q / 8] << 2) | kx[q];
          }
          store_moves(acc, ack);
        } else {
          // 16-bit codes
          uint32_t kprev = shift_into(0u, kx[H2 - 1]);
          uint16_t* Cr = s.code() + static_cast<int64_t>(r) * pitch;
#pragma unroll
          for (int q = 0; q < H2; ++q) {
            const uint32_t kd = __builtin_amdgcn_alignbit(kx[q], q == 0 ? kprev : kx[q - 1], 16);
            uint32_t code = 0;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const uint32_t hu = (cur[q] >> (16 * u)) & 0xffffu;
              const bool dg = ((bd[q] >> (16 * u)) & 0xffffu) == hu;
              const bool vt = ((bv[q] >> (16 * u)) & 0xffffu) == hu;
              const uint32_t kdu = (kd >> (16 * u)) & 0xffffu, kvu = (kx[q] >> (16 * u)) & 0xffffu;
              const uint32_t c = dg ? (kCodeDiag | kdu)
                                    : (vt ? (kCodeVert | kvu) : kCodeHorz);
              code |= c << (16 * u);
            }
            if (live) *reinterpret_cast<uint32_t*>(Cr + j0 + 2 * q) = code;
          }
        }
        if ((d & kRecSink) != 0) sink_row(r);
      }
      ++rr;
      next_row(rr);
      np = d & kRecPreds;
    }
  }
  *best_score = best;
  *tied = ties > 0;
  return best_row;
}

// ---- banded rows: the opt-in approximation of racon -b ----
//
// Each DP row r (1..V) computes only 256 columns, 4 per lane: columns
// lo(r) + 1 .. lo(r) + 256, where lo(r) follows the diagonal of the V x L
// matrix (centred on column r L / V, a multiple of 4, inside [0, L + 3]).
// lo never decreases with r, so a predecessor p < r holds row r's lane k in
// its lane k + (lo(r) - lo(p)) / 4. Values outside a row's band read as
// kBandNeg; a window whose traceback would leave the band is rerun unbanded
// (kPoaBandMiss). Used for layers longer than 256 only, and only while scores
// fit signed 16 bits (kBandNeg sits below every value they hold).
//
// The rows work as dp_rows' with 4 columns per lane (unsigned halves, the
// bias is 32768): one descriptor per row, scores by byte permute, move
// records. An LDS row holds column lo's value (column 0's when lo is 0, else
// kBandNeg) in front of the lanes' strips, so the value left of the first
// lane is one read whatever the shift. Records are kept by column as if column
// j were j + 3, so that a lane's four columns are one record; a row with
// several predecessors also keeps the index chosen at column lo, which the
// diagonal into its first column takes. Rows of one wave alone are bound by
// their instructions: 611 windows of 1,000 bp at 30 layers take 61 ms, where
// band rows with a predecessor list per row, letters reloaded per row and a
// traceback in blocks of 16 rows took about 90.
constexpr int kBandW = 4;
constexpr int kBand = kWave * kBandW;  // 256 columns
constexpr uint32_t kBandNeg = 64;      // -32768 + 64, with the bias
constexpr uint32_t kBandBias = 0x8000;
constexpr int kBandColumn = 3;         // record column of column j: j + 3

__device__ __forceinline__ int band_lo(int r, int V, int L) {
  // (single-precision r * (L / V): monotone in r, the same in the DP and the
  // traceback)
  const int c = static_cast<int>(static_cast<float>(r) * (static_cast<float>(L) /
                                                           static_cast<float>(V))) - kBand / 2;
  const int top = (L - kBand + 3) & ~3;
  return min(max(c, 0) & ~3, top);
}

// Predecessor row in the LDS row at `row` (its data after 8 bytes), seen
// `shift` lanes further right; *left: the value left of the first lane.
__device__ __forceinline__ void band_load(uint32_t row, int lane, int shift, uint32_t* pp,
                                          uint32_t* left) {
  constexpr uint32_t neg = kBandNeg * 0x10001u;
  if (shift > kWave) {
    pp[0] = pp[1] = neg;
    *left = kBandNeg;
    return;
  }
  const int src = lane + shift;
  const U32x2 v = *(const LPair*)(size_t)(row + 8 + 8 * static_cast<uint32_t>(min(src, kWave - 1)));
  typedef __attribute__((address_space(3))) uint16_t LHalf;
  *left = *(const LHalf*)(size_t)(row + 8 * static_cast<uint32_t>(shift) + 6);
  pp[0] = src < kWave ? v.x : neg;
  pp[1] = src < kWave ? v.y : neg;
}

// The rest of a band row: moves, chain, scores (cur), from the best
// predecessor scores pp and the value left of the first lane.
__device__ __forceinline__ void band_scores(const uint32_t* pp, uint32_t left, const uint32_t* sub,
                                            uint32_t gap_pair, int lane, int lo, uint32_t& excl,
                                            uint32_t* cur, uint32_t* cur_left, uint32_t* bd,
                                            uint32_t* bv) {
  constexpr uint32_t neg = kBandNeg * 0x10001u;
  const uint32_t prev = shift_into(left << 16, pp[1]);
  // column 0 heads the chain of a band that starts there
  const uint32_t h0 = lo == 0 ? (left + gap_pair) & 0xffffu : kBandNeg;
  uint32_t carry = lane == 0 ? h0 << 16 : 0u;
  uint32_t pre[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t d = __builtin_amdgcn_alignbit(pp[q], q == 0 ? prev : pp[0], 16);
    bd[q] = pk_add(d, sub[q]);
    bv[q] = pk_add(pp[q], gap_pair);
    carry = pk_max_hi_u(pk_scan_u(pk_max_u(bd[q], bv[q])), carry);
    pre[q] = carry;
  }
  excl = shift_into(excl, wave_prefix_max_u(carry));
#pragma unroll
  for (int q = 0; q < 2; ++q) cur[q] = pk_max_u(pk_max_hi_u(pre[q], excl), neg);
  *cur_left = h0;
}

// DP rows of one layer in band rows (layers longer than 256, 16-bit form).
__device__ __forceinline__ int dp_band(CParams& P, const Slot& s, uint32_t lds, int V, int L,
                                       int* best_score, bool* tied) {
  const int lane = lane_id();
  const int pitch = static_cast<int>(P.caps.cols);
  const int32_t gap = uniform(P.gap);
  const int32_t match = uniform(P.match);
  const int32_t mismatch = uniform(P.mismatch);
  const uint32_t row_bytes = static_cast<uint32_t>(pitch) * 2;
  const uint32_t seq_at =
      lds + static_cast<uint32_t>(align_up(static_cast<uint64_t>(P.ring_rows) * row_bytes, 16));
  const LByte* seq = (const LByte*)(size_t)seq_at;
  typedef __attribute__((address_space(3))) uint16_t LHalf;
  typedef __attribute__((address_space(1))) uint16_t GHalf;
  const uint32_t gap_pair = pk_splat(gap);
  const uint32_t miss = static_cast<uint32_t>(mismatch - gap) & 0xffffu;
  const uint32_t flip = (static_cast<uint32_t>(match - gap) & 0xffffu) ^ miss;
  const uint64_t table0 = static_cast<uint64_t>((miss >> 8) * 0x01010101u) << 32 |
                          (miss & 0xffu) * 0x01010101u;
  const uint64_t table1 = static_cast<uint64_t>(flip >> 8) << 32 | (flip & 0xffu);
  uint32_t one = 0x00010001u;  // (opaque, as in dp_rows)
  asm volatile("" : "+s"(one));
  bool plain = true;
  for (int j = lane; j < L; j += kWave) {
    const int c = seq[j];
    plain &= static_cast<int>((0x54474341u >> (8 * (((c >> 1) ^ (c >> 2)) & 3))) & 0xffu) == c;
  }
  const bool layer_plain = __all(plain);
  uint32_t excl = 0;  // lane 0: nothing to its left
  int32_t best = kNegInf;
  int best_row = 0;
  int ties = 0;
  const int total_preds = uniform(s.pred_off()[V]);
  uint32_t cur[2] = {0u, 0u}, cur_left = 0u;  // the row before
  uint32_t sel[2] = {0u, 0u};
  int sel_lo = -1;
  GByte* const codes = (GByte*)s.code();
  for (int r0 = 1; r0 <= V; r0 += kWave) {
    const int rk = r0 + lane;
    uint32_t desc_v = 0, shift_v = 0;
    const int lo_v = band_lo(min(rk, V), V, L);
    if (rk <= V) {
      const uint4 rec = s.row_rec()[rk - 1];
      desc_v = rec.x;
      const uint32_t d[4] = {rec.z & 0xffffu, rec.z >> 16, rec.w & 0xffffu, rec.w >> 16};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int by = (lo_v - band_lo(rk - static_cast<int>(d[k]), V, L)) >> 2;
        shift_v |= static_cast<uint32_t>(min(max(by, 0), kWave + 1)) << (8 * k);
      }
    }
    const int chunk = uniform(min(kWave, V - r0 + 1));
    int off_v = 0, end_v = 0, meta_v = 0, base = 0, pr0 = 0, pr1 = 0;
    if (__any(rk <= V && (desc_v & kRecPreds) == 0)) {
      if (rk <= V) {
        off_v = s.pred_off()[rk - 1];
        end_v = s.pred_off()[rk];
        meta_v = s.row_meta()[rk - 1];
      }
      base = __builtin_amdgcn_readlane(off_v, 0);
      pr0 = base + lane < total_preds ? s.pred_rows()[base + lane] : 0;
      pr1 = base + kWave + lane < total_preds ? s.pred_rows()[base + kWave + lane] : 0;
    }
    wait_stores();  // (the chunk's loads, as in dp_rows)
    GByte* record = codes + static_cast<int64_t>(r0) * row_bytes;
    const auto store_moves = [&](uint32_t acc, uint32_t ack, int lo) {
      const uint32_t a = (acc | (acc >> 12)) & 0xffu;
      const uint32_t k = (ack | (ack >> 12)) & 0xffu;
      *(GHalf*)(record + ((lo >> 2) + 1 + lane) * 2) = static_cast<uint16_t>(a | (k << 8));
    };
    for (int rr = 0; rr < chunk; ++rr) {
      const int r = r0 + rr;
      const uint32_t d = static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(desc_v), rr));
      const int lo = __builtin_amdgcn_readlane(lo_v, rr);
      uint32_t np = d & kRecPreds;
      uint32_t bd[2], bv[2], sub[2];
      bool general = false;
      if (np != 0) {
        if (lo != sel_lo) {
          // letters of columns lo + 1 + 4 lane .. (bytes past the layer are
          // never read back)
          const uint32_t w = *(const LWord*)(size_t)(seq_at + static_cast<uint32_t>(lo + kBandW * lane));
          const uint32_t c = ((w >> 1) ^ (w >> 2)) & 0x03030303u;
          sel[0] = __builtin_amdgcn_perm(0u, c, 0x01010000u) + 0x04000400u;
          sel[1] = __builtin_amdgcn_perm(0u, c, 0x03030202u) + 0x04000400u;
          if (!layer_plain) {
            const uint32_t other = __builtin_amdgcn_perm(0u, 0x54474341u, c) ^ w;
#pragma unroll
            for (int u = 0; u < kBandW; ++u) {
              if (((other >> (8 * u)) & 0xffu) != 0) {
                sel[u / 2] = (sel[u / 2] & (0xffffu << (16 * (~u & 1)))) | kOddLetter << (16 * (u & 1));
              }
            }
          }
          sel_lo = lo;
        }
        const uint64_t table = table0 ^ (table1 << (d & kRecBase));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          sub[q] = __builtin_amdgcn_perm(static_cast<uint32_t>(table >> 32),
                                         static_cast<uint32_t>(table), sel[q]);
        }
        if (!layer_plain) {
          sub[0] = odd_letters(sub[0], sel[0], miss * 0x10001u);
          sub[1] = odd_letters(sub[1], sel[1], miss * 0x10001u);
        }
      } else if ((d & kRecOther) != 0) {
        // a row of another letter
        const uint32_t meta = static_cast<uint32_t>(__builtin_amdgcn_readlane(meta_v, rr));
        np = (meta >> kRowMetaPredShift) & kRowMetaPredMask;
        const uint32_t w = *(const LWord*)(size_t)(seq_at + static_cast<uint32_t>(lo + kBandW * lane));
        const uint32_t hit = miss ^ flip;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint32_t pair = __builtin_amdgcn_perm(0u, w, q == 0 ? 0x0c010c00u : 0x0c030c02u);
          const uint32_t differ = pk_min_u(pair ^ (meta & 0xffu) * 0x10001u, one);
          sub[q] = pk_mad(differ, pk_sub(miss * 0x10001u, hit * 0x10001u), hit * 0x10001u);
        }
      } else {
        general = true;
      }
      if (!general) {
        const uint32_t shifts = static_cast<uint32_t>(
            __builtin_amdgcn_readlane(static_cast<int>(shift_v), rr));
        const auto row_at = [&](int k) {
          return lds + ((d >> (kRecPredShift + 5 * k)) & 31u) * row_bytes;
        };
        uint32_t mx[2], left;
        uint32_t ack = 0, k_left = 0;
        if ((d & kRecChain) != 0 && (shifts & 0xffu) == 0) {
          mx[0] = cur[0];
          mx[1] = cur[1];
          left = cur_left;
        } else {
          band_load(row_at(0), lane, static_cast<int>(shifts & 0xffu), mx, &left);
        }
        if (np > 1) {
          uint32_t kx[2] = {0u, 0u};
#pragma unroll
          for (int k = 1; k < static_cast<int>(kRecMaxPreds); ++k) {
            if (k < static_cast<int>(np)) {
              uint32_t pp[2], l1;
              band_load(row_at(k), lane, static_cast<int>((shifts >> (8 * k)) & 0xffu), pp, &l1);
#pragma unroll
              for (int q = 0; q < 2; ++q) {
                const uint32_t g = pk_min_u(pk_sub_sat(pp[q], mx[q]), one);
                kx[q] = pk_max_u(kx[q], pk_mad(g, static_cast<uint32_t>(k) * 0x10001u, 0u));
                mx[q] = pk_max_u(mx[q], pp[q]);
              }
              k_left = l1 > left ? static_cast<uint32_t>(k) : k_left;
              left = max(left, l1);
            }
          }
          ack = (kx[0] << 2) | kx[1];
        }
        band_scores(mx, left, sub, gap_pair, lane, lo, excl, cur, &cur_left, bd, bv);
        const uint32_t own = (d >> kRecOwnShift) & 31u;
        if (own != static_cast<uint32_t>(kSlotNone)) {
          const uint32_t at = lds + own * row_bytes;
          *(LPair*)(size_t)(at + 8 + 8 * static_cast<uint32_t>(lane)) = U32x2{cur[0], cur[1]};
          if (lane == 0) *(LHalf*)(size_t)(at + 6) = static_cast<uint16_t>(cur_left);
        }
        uint32_t acc[1];
        row_kinds<kBandW>(cur, bd, bv, acc);
        store_moves(acc[0], ack, lo);
        if (np > 1 && lane == 0) record[(lo >> 2) * 2 + 1] = static_cast<uint8_t>(k_left << 4);
      } else {
        // the general form, as in dp_rows
        const int off = __builtin_amdgcn_readlane(off_v, rr);
        const int n_preds = __builtin_amdgcn_readlane(end_v, rr) - off;
        const int meta = __builtin_amdgcn_readlane(meta_v, rr);
        const int own = (meta >> kRowMetaSlotShift) & 31;
        const int j0 = lo + 1 + kBandW * lane;
        uint32_t mx[2] = {0u, 0u}, kx[2] = {0u, 0u}, left = 0u, k_left = 0u;
        for (int k = 0; k < n_preds; ++k) {
          const int idx = off + k - base;
          int e;
          if (idx < kWave) {
            e = __builtin_amdgcn_readlane(pr0, idx);
          } else if (idx < 2 * kWave) {
            e = __builtin_amdgcn_readlane(pr1, idx - kWave);
          } else {
            e = uniform(s.pred_rows()[off + k]);
          }
          const int p = e & kPredRowMask;
          const int sl = static_cast<int>(static_cast<unsigned>(e) >> kPredRowBits);
          uint32_t pp[2], l1;
          if (p == 0) {
            pp[0] = pp[1] = kBandBias * 0x10001u;
            l1 = kBandBias;
          } else {
            const int lo_p = band_lo(p, V, L);
            if (sl < kSlotGlobal) {
              band_load(lds + static_cast<uint32_t>(sl) * row_bytes, lane,
                        min(max(lo - lo_p, 0) >> 2, kWave + 1), pp, &l1);
            } else {
              // a row kept in the slot's global matrix (absolute columns)
              const int32_t* row = s.H_row(p, pitch);
              uint32_t v[kBandW + 1];
#pragma unroll
              for (int u = 0; u <= kBandW; ++u) {
                const int j = j0 - 1 + u;
                const bool valid = (j > lo_p && j <= lo_p + kBand && j <= L) || (j == 0 && lo_p == 0);
                v[u] = valid ? static_cast<uint32_t>(row[j]) & 0xffffu : kBandNeg;
              }
              wait_stores();
              pp[0] = v[1] | v[2] << 16;
              pp[1] = v[3] | v[4] << 16;
              l1 = __builtin_amdgcn_readlane(static_cast<int>(v[0]), 0);
            }
          }
          const uint32_t ks = static_cast<uint32_t>(k) * 0x10001u;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const uint32_t g = pk_min_u(pk_sub_sat(pp[q], mx[q]), one);
            kx[q] = pk_mad(g, pk_sub(ks, kx[q]), kx[q]);
            mx[q] = pk_max_u(mx[q], pp[q]);
          }
          k_left = l1 > left ? static_cast<uint32_t>(k) : k_left;
          left = max(left, l1);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          uint32_t x = 0;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int idx = j0 + 2 * q + u - 1;
            const bool same = idx < L && static_cast<int>(seq[idx]) == (meta & 0xff);
            x |= (static_cast<uint32_t>((same ? match : mismatch) - gap) & 0xffffu) << (16 * u);
          }
          sub[q] = x;
        }
        band_scores(mx, left, sub, gap_pair, lane, lo, excl, cur, &cur_left, bd, bv);
        if (own < kSlotGlobal) {
          const uint32_t at = lds + static_cast<uint32_t>(own) * row_bytes;
          *(LPair*)(size_t)(at + 8 + 8 * static_cast<uint32_t>(lane)) = U32x2{cur[0], cur[1]};
          if (lane == 0) *(LHalf*)(size_t)(at + 6) = static_cast<uint16_t>(cur_left);
        } else if (own == kSlotGlobal) {
          int32_t* Hg = s.H_row(r, meta, pitch);
#pragma unroll
          for (int u = 0; u < kBandW; ++u) {
            if (j0 + u <= L) Hg[j0 + u] = static_cast<int32_t>((cur[u / 2] >> (16 * (u & 1))) & 0xffffu);
          }
          if (lane == 0) Hg[0] = static_cast<int32_t>(cur_left);
          wait_stores();
          wave_fence();
        }
        if ((d & kRecMoves) != 0) {
          uint32_t acc[1];
          row_kinds<kBandW>(cur, bd, bv, acc);
          store_moves(acc[0], (kx[0] << 2) | kx[1], lo);
          if (n_preds > 1 && lane == 0) {
            record[(lo >> 2) * 2 + 1] = static_cast<uint8_t>(k_left << 4);
          }
        } else {
          // 16-bit codes, column j at element j + 3
          const uint32_t kprev = shift_into(k_left << 16, kx[1]);
          uint16_t* Cr = s.code() + static_cast<int64_t>(r) * pitch;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const uint32_t kd = __builtin_amdgcn_alignbit(kx[q], q == 0 ? kprev : kx[0], 16);
            uint32_t code = 0;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const uint32_t hu = (cur[q] >> (16 * u)) & 0xffffu;
              const bool dg = ((bd[q] >> (16 * u)) & 0xffffu) == hu;
              const bool vt = ((bv[q] >> (16 * u)) & 0xffffu) == hu;
              const uint32_t kdu = (kd >> (16 * u)) & 0xffffu, kvu = (kx[q] >> (16 * u)) & 0xffffu;
              uint32_t c = vt ? (kCodeVert | kvu) : kCodeHorz;
              if (dg) c = kCodeDiag | kdu;
              pin(c);  // (without it the compiler's loop of the common rows takes 3% longer)
              code |= c << (16 * u);
            }
            *reinterpret_cast<uint32_t*>(Cr + j0 + kBandColumn + 2 * q) = code;
          }
          if (lane == 0 && lo == 0) {
            Cr[kBandColumn] = static_cast<uint16_t>(kCodeVert | k_left);
          }
        }
      }
      if ((d & kRecSink) != 0) {
        const int e = L - 1 - lo;  // column L in the band: lane e / 4, column e % 4
        int32_t h_last = kNegInf;
        if (e >= 0 && e < kBand) {
          const uint32_t w = (e & 2) != 0 ? cur[1] : cur[0];
          const uint32_t g = static_cast<uint32_t>(
              __builtin_amdgcn_readlane(static_cast<int>(w), e / kBandW));
          h_last = static_cast<int32_t>((e & 1) ? g >> 16 : g & 0xffffu) -
                   static_cast<int32_t>(kBandBias) + L * gap;
        }
        if (lane == 0) s.sink_score()[r] = h_last;
        if (h_last > best) {
          best = h_last;
          best_row = r;
          ties = 0;
        } else if (h_last == best) {
          ++ties;
        }
      }
      record += row_bytes;
      wave_fence();  // (a lane reads what another lane wrote)
    }
  }
  *best_score = best;
  *tied = ties > 0 && best > kNegInf;
  return best == kNegInf ? 0 : best_row;
}

// Uniform copy of a pointer (both halves read from the first active lane).
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return (T*)((static_cast<uint64_t>(hi) << 32) | lo);
}

enum DpKind : int {
  kDpRows4,
  kDpRows8,
  kDpRows12,
  kDpRows16,
  kDpRows20,
  kDpGeneric16,
  kDpGeneric32,
  kDpBand4
};

// The DP of one layer as an out-of-line call: its loops get a register
// allocation of their own instead of sharing one with the rest of the window
// loop. Arguments arrive in vector registers and are made uniform again on
// entry. Returns the end-cell row, its score and whether sinks tied.
template <int kKind, bool kPlain = true>
__device__ __noinline__ uint64_t dp_layer_call(CParams* params, GByte* base, CLayout* layout,
                                               uint32_t lds_addr, int V, int L, int bias) {
  CParams& P = *uniform_ptr(params);
  Slot s = carve(uniform_ptr(base), *uniform_ptr(layout));
  V = uniform(V);
  L = uniform(L);
  bias = uniform(bias);
  // the wave's LDS as a local-memory pointer from the caller (no lookup of
  // the dynamic LDS offset inside the loops)
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  [[maybe_unused]] uint8_t* lds = (uint8_t*)(LByte*)(size_t)lds_addr;
  int best_score = 0;
  bool tied = false;
  int row;
  if constexpr (kKind == kDpRows4) {
    row = dp_rows<4, kPlain>(P, s, lds_addr, V, L, bias, &best_score, &tied);
  } else if constexpr (kKind == kDpRows8) {
    row = dp_rows<8, kPlain>(P, s, lds_addr, V, L, bias, &best_score, &tied);
  } else if constexpr (kKind == kDpRows12) {
    row = dp_rows<12, kPlain>(P, s, lds_addr, V, L, bias, &best_score, &tied);
  } else if constexpr (kKind == kDpRows16) {
    row = dp_rows<16, kPlain>(P, s, lds_addr, V, L, bias, &best_score, &tied);
  } else if constexpr (kKind == kDpRows20) {
    row = dp_rows<20, kPlain>(P, s, lds_addr, V, L, bias, &best_score, &tied);
  } else if constexpr (kKind == kDpBand4) {
    row = dp_band(P, s, lds_addr, V, L, &best_score, &tied);
  } else if constexpr (kKind == kDpGeneric16) {
    row = dp_layer<int16_t>(P, s, lds, V, L, &best_score, &tied);
  } else {
    row = dp_layer<int32_t>(P, s, lds, V, L, &best_score, &tied);
  }
  return (static_cast<uint64_t>(static_cast<uint32_t>(best_score)) << 32) |
         (static_cast<uint32_t>(row) & 0x7fffffffu) | (tied ? 0x80000000u : 0u);
}

// Graph insertion of one layer (spoa add_alignment), position by position,
// lane-uniform, from the aligned node of every layer position (pos_node,
// -1 for an insertion). New nodes record their anchor rank for the
// incremental order. (Rare: two path nodes share an aligned set. Out of
// line; returns the slot with its updated counters.)
__device__ __noinline__ Slot insert_sequential(Slot s, CCaps& caps, int L, bool* order_ok_out,
                                              int* n_path_out) {
  bool order_ok = true;
  bool aligned_full = false;
  int n_path = 0;
  const int32_t* pos_node = s.path();
  const int before = s.n_nodes;
  int head = -1;
  int prev_w = 0;
  int head_anchor = -1;  // anchor of the previous path node when it is new
  for (int pos = 0; pos < L && !s.overflow; ++pos) {
    const int node = uniform(pos_node[pos]);
    const uint8_t letter = s.seq()[pos];
    int nv;
    if (node == -1) {
      nv = add_node(s, caps, letter);
    } else if (s.base()[node] == letter) {
      nv = node;
    } else {
      int same = -1;
      const int cnt = s.n_aligned()[node];
      for (int k = 0; k < cnt; ++k) {
        const int a = uniform(s.aligned()[node * kAligned + k]);
        if (s.base()[a] == letter) {
          same = a;
          break;
        }
      }
      if (same == -1) {
        nv = add_node(s, caps, letter);
        if (!s.overflow && cnt + 1 > static_cast<int>(kAligned)) {
          aligned_full = true;
          s.overflow = true;
        }
        if (s.overflow) break;
        for (int k = 0; k < cnt; ++k) {
          const int a = uniform(s.aligned()[node * kAligned + k]);
          const int ca = s.n_aligned()[a];
          s.aligned()[nv * kAligned + k] = a;
          s.aligned()[a * kAligned + ca] = nv;
          s.n_aligned()[a] = static_cast<uint8_t>(ca + 1);
        }
        s.aligned()[nv * kAligned + cnt] = node;
        s.n_aligned()[nv] = static_cast<uint8_t>(cnt + 1);
        s.aligned()[node * kAligned + cnt] = nv;
        s.n_aligned()[node] = static_cast<uint8_t>(cnt + 1);
      } else {
        nv = same;
      }
    }
    if (nv >= before) {
      // a new node: placed after its path predecessor's aligned set
      // (mismatch nodes: after the aligned set they join)
      int anchor;
      if (node != -1) {
        anchor = s.node_rank()[node];
        const int cnt = s.n_aligned()[node];
        for (int k = 0; k < cnt; ++k) {
          const int a = uniform(s.aligned()[node * kAligned + k]);
          if (a < before) anchor = max(anchor, s.node_rank()[a]);
        }
      } else if (head == -1) {
        anchor = -1;
      } else if (head >= before) {
        anchor = head_anchor;
      } else {
        anchor = s.node_rank()[head];
        const int cnt = s.n_aligned()[head];
        for (int k = 0; k < cnt; ++k) {
          const int a = uniform(s.aligned()[head * kAligned + k]);
          if (a < before) anchor = max(anchor, s.node_rank()[a]);
        }
      }
      const int k_new = nv - before;
      if (k_new > 0 && anchor < s.anchor()[k_new - 1]) {
        order_ok = false;
      }
      s.anchor()[k_new] = anchor;
      head_anchor = anchor;
    }
    s.lpath()[n_path++] = nv;
    if (head != -1) {
      add_edge(s, caps, head, nv, prev_w + s.qual()[pos]);
    }
    head = nv;
    prev_w = s.qual()[pos];
  }
  s.n_seqs = s.n_seqs + 1;
  *order_ok_out = order_ok;
  *n_path_out = aligned_full ? -1 : n_path;  // -1: an aligned set was full
  return s;
}

// Graph insertion of one layer, one lane per layer position. A global
// alignment covers every layer position once (positions 0..L-1 in order), so
// the path is the whole layer and its graph nodes are distinct. When no two
// of them share an aligned set, every position reads and writes only its own
// node, aligned set, in-edge list and out-edge list, and the result equals
// the position-by-position insertion: node ids and edge ids are handed out
// in position order with wave prefix counts, and the anchor of an insertion
// (the rank bound of the last non-insertion position before it) is a wave
// prefix scan. The same independence lets each pass load what kU chunks of
// 64 positions read before any of their writes, so those loads are in
// flight together. Status 1 when two path nodes share an aligned set
// (nothing in the graph has changed then), 0 when inserted (with the new
// node and edge counts), or a negative status. Out of line, for a register
// allocation of its own.
struct InsertResult {
  int32_t status;
  int32_t n_nodes;
  int32_t n_edges;
  int32_t order_ok;
};

__device__ __noinline__ InsertResult insert_parallel(GByte* slot_base, CLayout* layout,
                                                     uint32_t lseq_addr, int L, int n_nodes,
                                                     int n_edges, int n_seqs, int cap_nodes,
                                                     int cap_edges) {
  constexpr int kU = 4;   // chunks per round in the edge and label passes
  constexpr int kUA = 2;  // in the passes that hold aligned sets
  constexpr int kA = static_cast<int>(kAligned);
  const Slot s = carve(uniform_ptr(slot_base), *uniform_ptr(layout));
  const uint8_t* lseq = (const uint8_t*)(LByte*)(size_t)uniform(static_cast<int>(lseq_addr));
  L = uniform(L);
  n_nodes = uniform(n_nodes);
  n_edges = uniform(n_edges);
  n_seqs = uniform(n_seqs);
  cap_nodes = uniform(cap_nodes);
  cap_edges = uniform(cap_edges);
  InsertResult res;
  res.status = 0;
  res.n_nodes = n_nodes;
  res.n_edges = n_edges;
  res.order_ok = 1;
  const int lane = lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  const int32_t* pnode = s.path();  // aligned graph node of each layer position (-1: none)
  int32_t* pnv = s.lpath();         // graph node of each layer position after insertion
  uint8_t* stamp = s.in_sub();      // 2 on the path's nodes (the DP no longer needs it)
  uint8_t* base = s.base();
  uint8_t* n_aligned = s.n_aligned();
  int32_t* aligned = s.aligned();
  int32_t* node_rank = s.node_rank();
  for (int p = lane; p < L; p += kWave) {
    const int v = pnode[p];
    if (v != -1) stamp[v] = 2;
  }
  wave_sync();
  // existing node per position (match, or an aligned node with the letter)
  bool conflict = false, full = false;
  int n_new = 0;
  for (int p0 = 0; p0 < L; p0 += kUA * kWave) {
    int v[kUA], cnt[kUA], nv[kUA], letter[kUA], al[kUA][kA];
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      const int p = p0 + i * kWave + lane;
      v[i] = p < L ? pnode[p] : -1;
      letter[i] = p < L ? static_cast<int>(lseq[p]) : 0;
    }
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      cnt[i] = v[i] != -1 ? static_cast<int>(n_aligned[v[i]]) : 0;
      nv[i] = v[i] != -1 && static_cast<int>(base[v[i]]) == letter[i] ? v[i] : -1;
#pragma unroll
      for (int k = 0; k < kA; ++k) al[i][k] = v[i] != -1 ? aligned[v[i] * kA + k] : 0;
    }
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      int st[kA], ba[kA];
#pragma unroll
      for (int k = 0; k < kA; ++k) {
        st[k] = k < cnt[i] ? static_cast<int>(stamp[al[i][k]]) : 0;
        ba[k] = k < cnt[i] ? static_cast<int>(base[al[i][k]]) : -1;
      }
#pragma unroll
      for (int k = 0; k < kA; ++k) {
        conflict |= st[k] == 2;
        if (nv[i] == -1 && ba[k] == letter[i]) nv[i] = al[i][k];
      }
      full |= v[i] != -1 && nv[i] == -1 && cnt[i] + 1 > kA;
      const int p = p0 + i * kWave + lane;
      if (p < L) pnv[p] = nv[i];
      n_new += __popcll(__ballot(p < L && nv[i] == -1));
    }
  }
  if (__ballot(conflict) != 0) {
    res.status = 1;
    return res;
  }
  if (__ballot(full) != 0) {
    res.status = kPoaAlignedFull;  // a column with more distinct bytes than kAligned + 1
    return res;
  }
  if (n_nodes + n_new > cap_nodes) {
    res.status = kPoaNodeOverflow;
    return res;
  }
  wave_sync();
  // new nodes (ids in position order), aligned sets, anchors
  const int before = n_nodes;
  int next_id = before;
  int carry = -1;  // rank bound of the last non-insertion position so far
  for (int p0 = 0; p0 < L; p0 += kUA * kWave) {
    int v[kUA], nv[kUA], cnt[kUA], bound[kUA], al[kUA][kA];
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      const int p = p0 + i * kWave + lane;
      v[i] = p < L ? pnode[p] : -1;
      nv[i] = p < L ? pnv[p] : 0;
    }
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      cnt[i] = v[i] != -1 ? static_cast<int>(n_aligned[v[i]]) : 0;
      bound[i] = v[i] != -1 ? node_rank[v[i]] : -1;
#pragma unroll
      for (int k = 0; k < kA; ++k) al[i][k] = v[i] != -1 ? aligned[v[i] * kA + k] : 0;
    }
    int nal[kUA][kA];  // aligned-set sizes of the members (read before any write)
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      int rk[kA];
#pragma unroll
      for (int k = 0; k < kA; ++k) {
        rk[k] = k < cnt[i] ? node_rank[al[i][k]] : -1;
        nal[i][k] = k < cnt[i] ? static_cast<int>(n_aligned[al[i][k]]) : 0;
      }
#pragma unroll
      for (int k = 0; k < kA; ++k) bound[i] = max(bound[i], rk[k]);  // highest rank in v's set
    }
#pragma unroll
    for (int i = 0; i < kUA; ++i) {
      const int p = p0 + i * kWave + lane;
      const bool in = p < L;
      const bool isnew = in && nv[i] == -1;
      const unsigned long long m = __ballot(isnew);
      if (isnew) nv[i] = next_id + __popcll(m & below);
      next_id += __popcll(m);
      const int incl = wave_prefix_max(v[i] != -1 ? lane : -1);
      const int excl = wave_shift_right(incl, -1);
      const int from_lane = __shfl(bound[i], max(excl, 0), kWave);
      const int prev_bound = excl >= 0 ? from_lane : carry;
      if (isnew) {
        const int id = nv[i];
        s.anchor()[id - before] = v[i] != -1 ? bound[i] : prev_bound;
        base[id] = lseq[p];
        s.node_info()[id] = lseq[p];
        s.in_head()[id] = -1;
        s.out_head()[id] = -1;
        s.in_tail()[id] = -1;
        s.out_tail()[id] = -1;
        n_aligned[id] = 0;
        s.cov()[id] = 0;
        s.last_label()[id] = -1;
        if (v[i] != -1) {
          // the mismatch node joins v's aligned set
          const int c = cnt[i];
#pragma unroll
          for (int k = 0; k < kA; ++k) {
            if (k < c) {
              const int a = al[i][k];
              const int ca = nal[i][k];
              aligned[id * kA + k] = a;
              aligned[a * kA + ca] = id;
              n_aligned[a] = static_cast<uint8_t>(ca + 1);
            }
          }
          aligned[id * kA + c] = v[i];
          n_aligned[id] = static_cast<uint8_t>(c + 1);
          aligned[v[i] * kA + c] = id;
          n_aligned[v[i]] = static_cast<uint8_t>(c + 1);
        }
      }
      if (in) pnv[p] = nv[i];
      const int last = __builtin_amdgcn_readlane(incl, kWave - 1);
      if (last >= 0) carry = __builtin_amdgcn_readlane(bound[i], last);
    }
  }
  res.n_nodes = next_id;
  wave_sync();
  // anchors of the new nodes must be non-decreasing for the merged order
  bool bad = false;
  for (int k = 1 + lane; k < n_new; k += kWave) {
    bad |= s.anchor()[k] < s.anchor()[k - 1];
  }
  res.order_ok = __ballot(bad) == 0 ? 1 : 0;
  // edges between consecutive positions: weight w[p-1] + w[p]
  int32_t* e_tail = s.e_tail();
  int32_t* e_head = s.e_head();
  int32_t* e_weight = s.e_weight();
  int32_t* e_next_in = s.e_next_in();
  int32_t* e_next_out = s.e_next_out();
  int32_t* out_head = s.out_head();
  int32_t* out_tail = s.out_tail();
  int32_t* in_head = s.in_head();
  int32_t* in_tail = s.in_tail();
  for (int p0 = 1; p0 < L; p0 += kU * kWave) {
    int tail[kU], head[kU], w[kU], found[kU], e[kU];
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int p = p0 + i * kWave + lane;
      const bool in = p < L;
      tail[i] = in ? pnv[p - 1] : 0;
      head[i] = in ? pnv[p] : 0;
      w[i] = in ? s.qual()[p - 1] + s.qual()[p] : 0;
      found[i] = -1;
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int p = p0 + i * kWave + lane;
      e[i] = p < L ? out_head[tail[i]] : -1;
    }
    // out-edge lists of the kU tails in lockstep
    for (;;) {
      bool act = false;
#pragma unroll
      for (int i = 0; i < kU; ++i) act = act || e[i] != -1;
      if (__ballot(act) == 0) break;
      int h[kU], nx[kU];
#pragma unroll
      for (int i = 0; i < kU; ++i) {
        h[i] = -1;
        nx[i] = -1;
        if (e[i] != -1) {
          h[i] = e_head[e[i]];
          nx[i] = e_next_out[e[i]];
        }
      }
#pragma unroll
      for (int i = 0; i < kU; ++i) {
        if (e[i] != -1 && h[i] == head[i]) {
          found[i] = e[i];
          nx[i] = -1;
        }
        e[i] = nx[i];
      }
    }
    int ot[kU], it[kU];
    uint32_t info[kU];
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int p = p0 + i * kWave + lane;
      const bool need = p < L && found[i] == -1;
      ot[i] = need ? out_tail[tail[i]] : -1;
      it[i] = need ? in_tail[head[i]] : -1;
      info[i] = need ? s.node_info()[head[i]] : 0u;
      if (found[i] != -1) e_weight[found[i]] = e_weight[found[i]] + w[i];
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int p = p0 + i * kWave + lane;
      const bool need = p < L && found[i] == -1;
      const unsigned long long m = __ballot(need);
      if (n_edges + __popcll(m) > cap_edges) {
        res.status = kPoaNodeOverflow;
        return res;
      }
      if (need) {
        const int ne = n_edges + __popcll(m & below);
        e_tail[ne] = tail[i];
        e_head[ne] = head[i];
        e_weight[ne] = w[i];
        e_next_in[ne] = -1;
        e_next_out[ne] = -1;
        if (ot[i] == -1) {
          out_head[tail[i]] = ne;
        } else {
          e_next_out[ot[i]] = ne;
        }
        out_tail[tail[i]] = ne;
        if (it[i] == -1) {
          in_head[head[i]] = ne;
        } else {
          e_next_in[it[i]] = ne;
        }
        in_tail[head[i]] = ne;
        s.add_in(head[i], info[i], tail[i]);
      }
      n_edges += __popcll(m);
    }
  }
  res.n_edges = n_edges;
  // every node of the layer has an incident edge of this sequence when L > 1
  if (L > 1) {
    const int label = n_seqs;
    int32_t* last_label = s.last_label();
    int32_t* cov = s.cov();
    for (int p0 = 0; p0 < L; p0 += kU * kWave) {
      int v[kU], ll[kU], cv[kU];
#pragma unroll
      for (int i = 0; i < kU; ++i) {
        const int p = p0 + i * kWave + lane;
        v[i] = p < L ? pnv[p] : -1;
      }
#pragma unroll
      for (int i = 0; i < kU; ++i) {
        ll[i] = v[i] != -1 ? last_label[v[i]] : label;
        cv[i] = v[i] != -1 ? cov[v[i]] : 0;
      }
#pragma unroll
      for (int i = 0; i < kU; ++i) {
        if (ll[i] != label) {
          last_label[v[i]] = label;
          cov[v[i]] = cv[i] + 1;
        }
      }
    }
  }
  wave_sync();
  return res;
}

// Inclusive prefix sum over the 64 lanes (DPP, as wave_prefix_max; 0 is
// the identity, so each move folds into one v_add_u32 with a DPP source).
__device__ __forceinline__ int32_t wave_prefix_sum(int32_t x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

// DP rows of a layer (row r + 1 is node sub_order[r]): predecessor rows in
// in-edge order (row 0, the virtual start, for rows without one), sink flags,
// and an LDS slot for every row that a later row reads: the lowest slot whose
// previous row is no longer needed (lane k < n_slots holds the last row that
// reads slot k). row_of is 0 for nodes outside the layer's subgraph. Returns
// the largest predecessor count, or -1 when a row needs a global score row
// and the slot's pool has none free. Out of line, like the DP, for a register
// allocation of its own.
//
// Bound by the round trips to the graph's arrays (a slot's graph does not
// stay in the caches of a full device) and by the serial slot assignment. The
// first pass takes kU rows per lane per round in three round trips: the rows'
// nodes, their first eight in-edges (kept inline per node) and the in-edges'
// rows; it leaves each row's predecessor rows in its record, and the last
// reader of every row in LDS with an atomic maximum, so no out-edge list is
// walked. The second pass goes over 64 rows at a time, with the next rows
// already loaded: slots one row after the other (ten instructions each), then
// records and lists from the slots kept in LDS. With `records` (1 dp_rows, 2
// band rows) only rows of the general form get a predecessor list, and in
// dp_rows a row whose only reader is the next row, which reads nothing else,
// takes no slot (the DP still holds it in registers). Walking both edge lists of every row instead took
// 187 us a layer in a full batch of 500 bp windows at 52 layers and 79 us
// alone; this takes 146 and 67.
__device__ __noinline__ int build_rows(GByte* slot_base, CLayout* layout, int V, int n_slots,
                                       uint32_t lds_addr, int lds_bytes, int records) {
  constexpr int kU = 4;       // rows per lane per round of the first pass
  constexpr int kInline = 8;  // in-edges kept per node
  const Slot s = carve(uniform_ptr(slot_base), *uniform_ptr(layout));
  V = uniform(V);
  n_slots = uniform(n_slots);
  lds_bytes = uniform(lds_bytes);
  records = uniform(records);
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  const int lane = lane_id();
  // word r: last reader of row r + 1, then (second pass) its slot
  LWord* word = (LWord*)(size_t)lds_addr;
  const bool words = 4 * static_cast<int64_t>(V) <= lds_bytes;
  LByte* lslot = (LByte*)(size_t)lds_addr;  // without room for words: slots in bytes
  const bool bytes = V <= lds_bytes;
  const bool packed = V < 0x10000;  // predecessor rows fit 16 bits
  const int32_t* sub_order = s.sub_order();
  const int32_t* row_of = s.row_of();
  const uint32_t* node_info = s.node_info();
  const int4* node_in = s.node_in();
  const int32_t* in_head = s.in_head();
  const int32_t* e_next_in = s.e_next_in();
  const int32_t* e_tail = s.e_tail();
  int32_t* row_meta = s.row_meta();
  int32_t* pred_off = s.pred_off();
  int32_t* pred_rows = s.pred_rows();
  uint4* row_rec = s.row_rec();
  if (words) {
    for (int r = lane; r < V; r += kWave) word[r] = 0u;
    wave_fence();
  }
  auto read_by = [&](int p, int row) {
    if (words) __hip_atomic_fetch_max(&word[p - 1], static_cast<uint32_t>(row), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  int max_np = 0;
  for (int r0 = 0; r0 < V; r0 += kU * kWave) {
    int v[kU], np[kU];
    uint32_t info[kU], at[kU][kInline / 2];
    int4 in[kU];
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int r = r0 + i * kWave + lane;
      v[i] = r < V ? sub_order[r] : -1;
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      info[i] = v[i] >= 0 ? node_info[v[i]] : 0u;
      in[i] = v[i] >= 0 ? node_in[2 * v[i]] : make_int4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int n = static_cast<int>(info[i] >> 8);
      const int t[4] = {in[i].x, in[i].y, in[i].z, in[i].w};
      int row[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) row[j] = j < n ? row_of[t[j]] : 0;
      in[i] = make_int4(row[0], row[1], row[2], row[3]);
    }
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      const int r = r0 + i * kWave + lane;
      np[i] = 0;
#pragma unroll
      for (int j = 0; j < kInline / 2; ++j) at[i][j] = 0u;
      // the next predecessor of the row, in in-edge order
      auto add = [&](int p) {
        if (p <= 0) return;
        read_by(p, r + 1);
#pragma unroll
        for (int j = 0; j < kInline / 2; ++j) {
          at[i][j] |= (np[i] >> 1) == j ? static_cast<uint32_t>(p) << (16 * (np[i] & 1)) : 0u;
        }
        ++np[i];
      };
      add(in[i].x);
      add(in[i].y);
      add(in[i].z);
      add(in[i].w);
      const int n = static_cast<int>(info[i] >> 8);
      if (__any(n > 4)) {
        if (n > 4) {
          const int4 t = node_in[2 * v[i] + 1];
          const int a = row_of[t.x], b = n > 5 ? row_of[t.y] : 0;
          const int c = n > 6 ? row_of[t.z] : 0, d = n > 7 ? row_of[t.w] : 0;
          add(a);
          add(b);
          add(c);
          add(d);
        }
        if (n > kInline) {
          int k = 0;
          for (int e = in_head[v[i]]; e != -1; e = e_next_in[e], ++k) {
            if (k >= kInline) add(row_of[e_tail[e]]);
          }
        }
      }
      if (v[i] >= 0) {
        row_meta[r] = static_cast<int32_t>((info[i] & 0xffu) | static_cast<uint32_t>(min(np[i], 255)) << 8);
        row_rec[r] = make_uint4(at[i][0], at[i][1], at[i][2], at[i][3]);
        max_np = max(max_np, max(np[i], 1));  // row 0 stands in for none
      }
    }
  }
  wave_sync();
  int busy = lane < n_slots ? 0 : 0x7fffffff;
  // pooled global score rows: lane k holds the last reader of entry k
  // (pool0) and of entry 64 + k (pool1); entries past the pool never free
  const int hpool = uniform(static_cast<int>(s.L->hpool));
  int pool0 = lane < hpool ? 0 : 0x7fffffff;
  int pool1 = lane + kWave < hpool ? 0 : 0x7fffffff;
  bool pool_full = false;
  int run = 0;
  uint4 rec_next = make_uint4(0u, 0u, 0u, 0u);
  int meta_next = 0, after_next = 0, node_next = 0;
  auto fetch = [&](int r) {
    if (r < V) {
      rec_next = row_rec[r];
      meta_next = row_meta[r];
      node_next = sub_order[r];
    }
    after_next = r + 1 < V ? row_meta[r + 1] : 0;
  };
  fetch(lane);
  for (int c0 = 0; c0 < V; c0 += kWave) {
    const int r = c0 + lane;
    const bool in = r < V;
    const uint4 x = rec_next;
    const int meta0 = meta_next, after = after_next, node = node_next;
    // (the next rows' first-pass records: this chunk's writes stop before)
    fetch(r + kWave);
    const int letter = meta0 & 0xff;
    const int np = (meta0 >> 8) & 0xff;
    int last = 0;
    if (words) {
      last = in ? static_cast<int>(word[r]) : 0;
    } else if (in) {
      // no room for the last readers: from the out-edges
      for (int e = s.out_head()[node]; e != -1; e = s.e_next_out()[e]) {
        last = max(last, row_of[s.e_head()[e]]);
      }
    }
    const bool chained = records == 1 && last == r + 2 && ((after >> 8) & 0xff) == 1;
    int my_slot = kSlotNone;
    int my_pool = 0;
    for (unsigned long long need = __ballot(in && last != 0 && !chained); need != 0;
         need &= need - 1) {
      const int rr = __ffsll(static_cast<long long>(need)) - 1;
      const int l = __builtin_amdgcn_readlane(last, rr);
      const int row = c0 + rr + 1;
      const unsigned long long free_mask = __ballot(busy < row);
      if (free_mask != 0) {
        const int sl = __ffsll(static_cast<long long>(free_mask)) - 1;
        busy = lane_write(l, sl, busy);
        my_slot = lane_write(sl, rr, my_slot);
        continue;
      }
      // no LDS slot: the global matrix
      my_slot = lane_write(kSlotGlobal, rr, my_slot);
      if (hpool != 0) {
        // the lowest free pool entry (lane k of pool0 holds entry k, of
        // pool1 entry 64 + k); none free: the window reruns exactly
        const unsigned long long g0 = __ballot(pool0 < row);
        const unsigned long long g1 = __ballot(pool1 < row);
        int g = 0;
        if (g0 != 0) {
          g = __ffsll(static_cast<long long>(g0)) - 1;
          pool0 = lane_write(l, g, pool0);
        } else if (g1 != 0) {
          const int t = __ffsll(static_cast<long long>(g1)) - 1;
          pool1 = lane_write(l, t, pool1);
          g = kWave + t;
        } else {
          pool_full = true;
        }
        my_pool = lane_write(g, rr, my_pool);
      }
    }
    const bool sink = last == 0;
    if (in) {
      row_meta[r] = letter | (sink ? kRowMetaSink : 0) |
                    (my_slot << kRowMetaSlotShift) | (my_pool << kRowMetaGShift) |
                    min(np, kRowMetaPredMask) << kRowMetaPredShift;
      if (words) {
        word[r] = static_cast<uint32_t>(my_slot);
      } else if (bytes) {
        lslot[r] = static_cast<uint8_t>(my_slot);
      }
    }
    if (!words && !bytes) {
      wave_sync();  // slots are read from the row table
    } else {
      wave_fence();
    }
    auto slot_of = [&](int p) -> int {
      if (words) return static_cast<int>(word[p - 1]);
      if (bytes) return static_cast<int>(lslot[p - 1]);
      return (row_meta[p - 1] >> kRowMetaSlotShift) & 31;
    };
    // the row's descriptor, unless it takes the general form
    const int code = ((letter >> 1) ^ (letter >> 2)) & 3;
    bool fast = packed && np >= 1 && np <= static_cast<int>(kRecMaxPreds) && my_slot != kSlotGlobal;
    const bool base = static_cast<int>((0x54474341u >> (8 * code)) & 0xffu) == letter;
    uint32_t fields = (base ? static_cast<uint32_t>(np) | static_cast<uint32_t>(code << 3)
                            : kRecMoves | kRecOther) |
                      static_cast<uint32_t>(my_slot) << kRecOwnShift;
    uint64_t deltas = 0;  // row deltas of the first four predecessors (0: none or too far)
    int p[kInline], sl[kInline];
    if (in) {
      const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int j = 0; j < kInline; ++j) {
        p[j] = static_cast<int>((w[j / 2] >> (16 * (j & 1))) & 0xffffu);
        sl[j] = 0;
      }
#pragma unroll
      for (int j = 0; j < static_cast<int>(kRecMaxPreds); ++j) {
        if (j < np && packed) {
          sl[j] = slot_of(p[j]);
          // (a chained predecessor is the row before: the descriptor's flag
          // or, in the general form, kSlotNone)
          fast = fast && (sl[j] < kSlotGlobal || (sl[j] == kSlotNone && np == 1));
          fields |= static_cast<uint32_t>(sl[j] & 31) << (kRecPredShift + 5 * j);
          deltas |= static_cast<uint64_t>(static_cast<uint32_t>(r + 1 - p[j])) << (16 * j);
        }
      }
      if (np == 1 && packed && p[0] == r) fields |= kRecChain;
    }
    const bool lists = in && !(records != 0 && fast);
    int cnt = lists ? max(np, 1) : 0;
    const bool walk = lists && (!packed || np > kInline);
    if (__any(walk)) {
      if (walk) {
        // (the count was capped in the row's record)
        cnt = 0;
        for (int e = in_head[node]; e != -1; e = e_next_in[e]) cnt += row_of[e_tail[e]] > 0;
        cnt = max(cnt, 1);
      }
    }
    const int sum = wave_prefix_sum(cnt);
    const int off = run + sum - cnt;
    run += __builtin_amdgcn_readlane(sum, kWave - 1);
    if (in) pred_off[r] = off;
    if (__any(lists)) {
      if (lists && !walk) {
        if (np == 0) {
          pred_rows[off] = 0;
          deltas = static_cast<uint64_t>(r + 1 <= 0xffff ? r + 1 : 0);
        }
#pragma unroll
        for (int j = 0; j < kInline; ++j) {
          if (j < np) pred_rows[off + j] = p[j] | (slot_of(p[j]) << kPredRowBits);
        }
      } else if (walk) {
        int o = off;
        int k = 0;
        deltas = 0;
        for (int e = in_head[node]; e != -1; e = e_next_in[e]) {
          const int q = row_of[e_tail[e]];
          if (q > 0) {
            pred_rows[o++] = q | (slot_of(q) << kPredRowBits);
            const int d = r + 1 - q;
            if (k < 4 && d <= 0xffff) deltas |= static_cast<uint64_t>(d) << (16 * k);
            ++k;
          }
        }
        if (k == 0) {
          pred_rows[off] = 0;
          deltas = static_cast<uint64_t>(r + 1 <= 0xffff ? r + 1 : 0);
        }
      }
    }
    if (in) {
      // (the general form keeps a record of its moves too while four indices
      // name its predecessors)
      const bool moves = packed && np >= 1 && np <= static_cast<int>(kRecMaxPreds);
      const uint32_t desc = (sink ? kRecSink : 0u) | (fast ? fields : moves ? kRecMoves : 0u);
      row_rec[r] = make_uint4(desc, static_cast<uint32_t>(node), static_cast<uint32_t>(deltas),
                              static_cast<uint32_t>(deltas >> 32));
    }
  }
  if (lane == 0) {
    pred_off[V] = run;
  }
  if (pool_full) return -1;
  return __builtin_amdgcn_readlane(wave_prefix_max(max_np), kWave - 1);
}

// Included nodes of a layer that does not span the window (spoa
// Graph::subgraph's walk): the nodes >= begin that reach `end` backwards
// along in-edges and aligned sets through nodes >= begin. The set is a
// reachability closure, so the order in which it is found changes nothing:
// here it is found by rank, 64 ranks at a time from `end`'s down. In-edges lead
// to lower ranks and aligned sets lie side by side, so a chunk's nodes are
// decided by chunks above it and by each other. A chunk takes three round
// trips to memory (its nodes; their in-edges and aligned sets; the ranks of
// those), then closes over itself in registers: each node's readers inside the
// chunk as a 64-bit mask, and one ballot per edge of the longest chain. Edges
// that leave the chunk set the rank's bit in LDS; when one leads up to a chunk
// that is done (an aligned set across a chunk border), that chunk is taken
// again with its new nodes. Every pass over a chunk marks at least one new
// node done, so the walk ends.
//
// On 800 windows of 150 bp reads a layer takes 23 us; a walk from `end` with a
// round trip per edge of the path through the graph took 121.
//
// Writes in_sub[0..nn) for every rank's node. Returns 0, or 1 when the LDS
// (lds_bytes at lds_addr) cannot hold the bits.
__device__ __noinline__ int include_ranks(GByte* slot_base, CLayout* layout, uint32_t lds_addr,
                                          int lds_bytes, int begin, int end, int nn) {
  constexpr int kInline = 8;
  constexpr int kA = static_cast<int>(kAligned);
  constexpr int kT = kInline + kA;  // targets of a node kept in registers
  const Slot s = carve(uniform_ptr(slot_base), *uniform_ptr(layout));
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  lds_bytes = uniform(lds_bytes);
  begin = uniform(begin);
  end = uniform(end);
  nn = uniform(nn);
  const int lane = lane_id();
  const int chunks = (nn + kWave - 1) / kWave;
  // per chunk 64 reached bits and 64 done bits, then the chunk's reader masks
  typedef __attribute__((address_space(3))) unsigned long long LMask;
  if (16 * chunks + 8 * kWave > lds_bytes) return 1;
  LMask* reached = (LMask*)(size_t)lds_addr;
  LMask* done = reached + chunks;
  LMask* readers = done + chunks;
  for (int c = lane; c < 2 * chunks; c += kWave) reached[c] = 0ull;
  const int32_t* rank_to_node = s.rank_to_node();
  const int32_t* node_rank = s.node_rank();
  const uint32_t* node_info = s.node_info();
  const int32_t* node_in = (const int32_t*)s.node_in();
  const uint8_t* n_aligned = s.n_aligned();
  const int32_t* aligned = s.aligned();
  auto set_bit = [&](int rank) {
    return __hip_atomic_fetch_or(&reached[rank >> 6], 1ull << (rank & 63), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  const int rank_end = uniform(node_rank[end]);
  wave_fence();
  if (lane == 0 && end >= begin) set_bit(rank_end);
  wave_fence();
  int c = rank_end >> 6;
  int low = c;  // lowest chunk with a reached node so far
  while (c >= low) {
    const unsigned long long before = reached[c], was_done = done[c];
    const uint64_t r_lo = uniform(static_cast<int>(before)) & 0xffffffffu;
    const uint64_t r_hi = uniform(static_cast<int>(before >> 32)) & 0xffffffffu;
    unsigned long long now = r_hi << 32 | r_lo;
    const uint64_t d_lo = uniform(static_cast<int>(was_done)) & 0xffffffffu;
    const uint64_t d_hi = uniform(static_cast<int>(was_done >> 32)) & 0xffffffffu;
    const unsigned long long old = d_hi << 32 | d_lo;
    if (now == old) {
      --c;
      continue;
    }
    const int base = c * kWave;
    const int v = base + lane < nn ? rank_to_node[base + lane] : -1;
    // targets: in-edge tails, then the aligned set (-1: none or below begin)
    int t[kT];
    int n_in = 0, n_al = 0;
    if (v >= 0) {
      n_in = static_cast<int>(node_info[v] >> 8);
      n_al = n_aligned[v];
    }
    const int max_in = min(kInline, uniform(__builtin_amdgcn_readlane(wave_prefix_max(n_in), kWave - 1)));
    const int max_al = uniform(__builtin_amdgcn_readlane(wave_prefix_max(n_al), kWave - 1));
#pragma unroll
    for (int j = 0; j < kT; ++j) {
      const bool edge = j < kInline;
      const int k = edge ? j : j - kInline;
      t[j] = -1;
      if (k < (edge ? max_in : max_al)) {
        if (k < (edge ? n_in : n_al)) t[j] = edge ? node_in[kInline * v + k] : aligned[v * kA + k];
      }
    }
#pragma unroll
    for (int j = 0; j < kT; ++j) {
      const bool edge = j < kInline;
      const int k = edge ? j : j - kInline;
      if (k < (edge ? max_in : max_al)) t[j] = t[j] >= begin ? node_rank[t[j]] : -1;
    }
    readers[lane] = 0ull;
    wave_fence();
    const unsigned long long mine = 1ull << lane;
    auto inside = [&](int rank) { return rank >= base && rank < base + kWave; };
    auto add_reader = [&](int rank) {
      __hip_atomic_fetch_or(&readers[rank - base], mine, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_WAVEFRONT);
    };
#pragma unroll
    for (int j = 0; j < kT; ++j) {
      const bool edge = j < kInline;
      const int k = edge ? j : j - kInline;
      if (k < (edge ? max_in : max_al)) {
        if (t[j] >= 0 && inside(t[j])) add_reader(t[j]);
      }
    }
    // in-edges past the inline ones
    auto more = [&](auto&& f) {
      if (n_in > kInline) {
        int k = 0;
        for (int e = s.in_head()[v]; e != -1; e = s.e_next_in()[e], ++k) {
          const int u = s.e_tail()[e];
          if (k >= kInline && u >= begin) f(node_rank[u]);
        }
      }
    };
    more([&](int rank) {
      if (inside(rank)) add_reader(rank);
    });
    wave_fence();
    const unsigned long long by = readers[lane];
    for (;;) {
      const unsigned long long grown = now | __ballot((by & now) != 0);
      if (grown == now) break;
      now = grown;
    }
    // edges out of the chunk, from its new nodes
    int up = -1;
    int down = c;
    if (((now & ~old) & mine) != 0) {
      auto leave = [&](int rank) {
        if (inside(rank)) return;
        const unsigned long long seen = set_bit(rank);
        if (rank < base) {
          down = min(down, rank >> 6);
        } else if (((seen >> (rank & 63)) & 1ull) == 0) {
          up = max(up, rank >> 6);
        }
      };
#pragma unroll
      for (int j = 0; j < kT; ++j) {
        const bool edge = j < kInline;
        const int k = edge ? j : j - kInline;
        if (k < (edge ? max_in : max_al)) {
          if (t[j] >= 0) leave(t[j]);
        }
      }
      more(leave);
    }
    if (lane == 0) {
      reached[c] = now;
      done[c] = now;
    }
    wave_fence();
    low = min(low, uniform(-__builtin_amdgcn_readlane(wave_prefix_max(-down), kWave - 1)));
    up = uniform(__builtin_amdgcn_readlane(wave_prefix_max(up), kWave - 1));
    c = up >= 0 ? up : c - 1;
  }
  uint8_t* in_sub = s.in_sub();
  for (int r0 = 0; r0 < nn; r0 += kWave) {
    const int r = r0 + lane;
    if (r < nn) in_sub[rank_to_node[r]] = static_cast<uint8_t>((reached[r0 >> 6] >> lane) & 1ull);
  }
  return 0;
}

// Traceback over the move records of dp_rows, from the end cell
// (row, L) up to the virtual start row; the graph node of the diagonal move
// into column p + 1, or -1 for a horizontal one, goes to path()[p] (s.path).
// Returns the column reached in row 0, -1 when a move leads outside, or, over
// band rows (kBanded, V DP rows), -2 when one leaves the band.
//
// A tile is 64 rows, one per lane, and the columns of the last few strip
// records at and before the current one: one round trip brings every row's
// record (descriptor, node, predecessor deltas) and 16 or 32 bytes of moves.
// The lanes put their fields in column order, the current column on top, so
// that a column step is one shift of the tile and the walk reads its row's
// move with v_readlane: 29 instructions a move, most of them scalar. (Tiles of
// 16 rows x 8 columns with successor indices per cell took 66 round trips a
// layer of 490 columns instead of 20, 106 us alone and 216 us in a full
// batch.) Rows of 16-bit codes are decoded one move at a time.
template <int W, bool kBanded>
__device__ __noinline__ int trace_rows(GByte* slot_base, CLayout* layout, int pitch, int V, int L,
                                       int row) {
  static_assert(W == 4 || W == 8 || W == 12 || W == 16 || W == 20, "strip width");
  const Slot s = carve(uniform_ptr(slot_base), *uniform_ptr(layout));
  pitch = uniform(pitch);
  V = uniform(V);
  const int length = uniform(L);
  constexpr int kShift = kBanded ? kBandColumn : 0;  // record column of column j: j + kShift
  const int lane = lane_id();
  constexpr int kRecord = W == 4 ? 2 : W == 8 ? 4 : W <= 16 ? 8 : 16;  // bytes
  constexpr int kRecords = W <= 16 ? 16 / kRecord : 2;  // records of a tile
  const GByte* codes = (const GByte*)s.code();
  const uint4* row_rec = s.row_rec();
  int32_t* pos_node = s.path();
  int i = uniform(row), j = uniform(L);
  while (i > 0) {
    const int i0 = i, j0 = j;
    const int ri = i0 - lane;
    const int rc = max(ri, 1);
    const GByte* mrow = codes + static_cast<int64_t>(rc) * pitch * 2;
    const int q = (j0 + kShift) / W;
    const int first = max(0, q - (kRecords - 1));  // first record of the tile
    U32x4 w;
    [[maybe_unused]] U32x4 w_last;  // W = 20: the current column's record
    __builtin_memcpy(&w, (const uint8_t*)(mrow + first * kRecord), 16);
    if constexpr (W == 20) __builtin_memcpy(&w_last, (const uint8_t*)(mrow + q * kRecord), 16);
    const uint4 rec = row_rec[rc - 1];
    // fields of columns first * W .. in ascending order (two bits each, the
    // bits of a field swapped: 1 diagonal, 2 vertical; predecessor indices 1
    // and 2 trade places)
    uint64_t kinds, preds;
    const int at = j0 + kShift - first * W;
    if constexpr (W == 20) {
      // words: kinds of 16 and of 4 columns, then indices; 32 columns end at
      // the current one, from its record and the one before
      const auto spread = [](uint32_t x) {  // 16 bits of fields to every second field
        x = (x | x << 8) & 0x00ff00ffu;
        x = (x | x << 4) & 0x0f0f0f0fu;
        return (x | x << 2) & 0x33333333u;
      };
      const auto order = [&](uint32_t a, uint32_t b) -> uint64_t {
        a = __builtin_bitreverse32(a);
        b = __builtin_bitreverse32(b);
        const uint32_t low = spread(a >> 16) | spread(a & 0xffffu) << 2;
        const uint32_t high = spread(b >> 28) | spread((b >> 12) & 0xfu) << 2;
        return static_cast<uint64_t>(high) << 32 | low;
      };
      const int up = 62 - 2 * (j0 - q * W);  // 24..62
      const auto top = [&](uint64_t before, uint64_t last) -> uint64_t {
        before = up >= 2 * W ? before << (up - 2 * W) : before >> (2 * W - up);
        return last << up | (first < q ? before : 0);
      };
      kinds = top(order(w.x, w.y), order(w_last.x, w_last.y));
      preds = top(order(w.z, w.w), order(w_last.z, w_last.w));
    } else {
      const uint32_t r[4] = {__builtin_bitreverse32(w.x), __builtin_bitreverse32(w.y),
                             __builtin_bitreverse32(w.z), __builtin_bitreverse32(w.w)};
      if constexpr (W == 4) {
        // bytes of r: record 2m + 1's indices, its kinds, record 2m's
        // indices, its kinds; columns 1, 3, 0, 2 from the low bits up
        uint32_t y[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          y[m] = ((r[m] >> 4) & 0x03030303u) | ((r[m] & 0x03030303u) << 2) |
                 ((r[m] >> 2) & 0x30303030u) | ((r[m] & 0x0c0c0c0cu) << 4);
        }
        const auto pick = [&](uint32_t a, uint32_t b, uint32_t sel) {
          return __builtin_amdgcn_perm(b, a, sel);
        };
        kinds = static_cast<uint64_t>(pick(y[2], y[3], 0x05070103u)) << 32 | pick(y[0], y[1], 0x05070103u);
        preds = static_cast<uint64_t>(pick(y[2], y[3], 0x04060002u)) << 32 | pick(y[0], y[1], 0x04060002u);
      } else if constexpr (W == 8) {
        // bytes of r: indices of the odd columns, of the even ones, kinds of
        // the odd columns, of the even ones
        const auto spread = [](uint32_t x) {  // even bytes' fields to every second field
          x = (x | x << 4) & 0x0f0f0f0fu;
          x = (x | x << 2) & 0x33333333u;
          return (x | x >> 14) & 0xffffu;
        };
        uint32_t k[4], p[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          k[m] = spread(__builtin_amdgcn_perm(0u, r[m], 0x0c020c03u));
          p[m] = spread(__builtin_amdgcn_perm(0u, r[m], 0x0c000c01u));
        }
        kinds = static_cast<uint64_t>(k[2] | k[3] << 16) << 32 | (k[0] | k[1] << 16);
        preds = static_cast<uint64_t>(p[2] | p[3] << 16) << 32 | (p[0] | p[1] << 16);
      } else {
        // words: kinds, indices per record; after the reversal the odd
        // columns' fields are the low half, the even ones' the high half
        const auto spread = [](uint32_t x) {  // 16 bits of fields to every second field
          x = (x | x << 8) & 0x00ff00ffu;
          x = (x | x << 4) & 0x0f0f0f0fu;
          return (x | x << 2) & 0x33333333u;
        };
        const auto order = [&](uint32_t x) {
          const uint32_t even = W == 16 ? x >> 16 : x >> 20;
          const uint32_t odd = W == 16 ? x & 0xffffu : (x >> 4) & 0xfffu;
          return spread(even) | spread(odd) << 2;
        };
        kinds = static_cast<uint64_t>(order(r[2])) << (2 * W) | order(r[0]);
        preds = static_cast<uint64_t>(order(r[3])) << (2 * W) | order(r[1]);
      }
    }
    // the current column's field on top
    if constexpr (W < 20) {
      kinds <<= 62 - 2 * at;
      preds <<= 62 - 2 * at;
    }
    if (kBanded) {
      // column 0 is always vertical; records of rows with one predecessor
      // leave the index left of the band unwritten
      const int field = 62 - 2 * j0;
      if (first == 0) kinds = (kinds & ~(3ull << field)) | 2ull << field;
      if (rec.z < 0x10000u) preds = 0;
    }
    // A cell takes one move: diagonal before vertical. Its predecessor index is
    // the one kept at the column before for a diagonal, at its own column for
    // a vertical.
    kinds &= ~((kinds & 0x5555555555555555ull) << 1);
    {
      const uint64_t diagonal = (kinds & 0x5555555555555555ull) * 3;
      preds = ((preds << 2) & diagonal) | (preds & ~diagonal);
    }
    // the four row deltas as bytes, in the order of the swapped indices; 255
    // and more lead out of the tile and are made exact after the walk
    const auto clamp = [](uint32_t x) { return pk_min_u(pk_max_u(x, 0x00010001u), 0x00ff00ffu); };
    const uint32_t deltas = clamp(rec.z) | clamp(rec.w) << 8;
    // lanes that end the walk inside the tile: rows of 16-bit codes and
    // rows past the start (their node's sign bit set)
    const bool stop = ri < 1 || (rec.x & (kRecPreds | kRecMoves)) == 0;
    const int node_v = static_cast<int>(rec.y | (stop ? 0x80000000u : 0u));
    // columns the tile can step: a diagonal also reads the column before
    const int columns = first == 0 && (W < 20 || j0 < 32) ? j0 + 1 : min(at, 31);
    const int lo_v = kBanded ? band_lo(rc, V, length) : 0;
    int left_band = 0;
    int out = -1;  // lane (t - columns) mod 64: the node of position j0 - 1 - t
    // Rows and columns walked, l and t, in one word: l + 0x8000 - 64 below,
    // t + 0x8000 - columns above, so that the low bits of each half number
    // lanes and one test finds the walk at the tile's end.
    constexpr uint32_t kRow0 = 0x8000u - kWave;
    const uint32_t col0 = 0x8000u - static_cast<uint32_t>(columns);
    uint32_t c = col0 << 16 | kRow0;
    uint32_t delta = 0, index = 0;
    int node = __builtin_amdgcn_readlane(node_v, 0);
    // (no branch on the kind of move: every move reads the same lanes and
    // selects in scalar registers; a vertical move's -1 in lane t is written
    // over by the move that leaves the column)
    while (((c | (static_cast<uint32_t>(node) & 0x80000000u)) & 0x80008000u) == 0 &&
           (!kBanded || left_band == 0)) {
      uint32_t kx = static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(kinds >> 32), c & 63u));
      const uint32_t px = static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(preds >> 32), c & 63u));
      const uint32_t ds = static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(deltas), c & 63u));
      // (opaque, so that the tests below stay on one word)
      asm volatile("" : "+s"(kx));
      index = (px >> 27) & 24u;
      delta = (ds >> index) & 0xffu;
      delta = kx > 0x3fffffffu ? delta : 0u;
      out = lane_write((kx & 0x40000000u) != 0 ? node : -1, static_cast<int>(c >> 16) & 63, out);
      const bool vertical = (kx >> 31) != 0;
      const uint32_t fields = vertical ? 0u : 2u;
      c += vertical ? 0u : 0x10000u;
      c += delta;
      kinds <<= fields;
      preds <<= fields;
      node = __builtin_amdgcn_readlane(node_v, c & 63u);
      if (kBanded && (c & 0x80008000u) == 0) {
        // (rows past the start hold every column)
        const int l = static_cast<int>((c & 0xffffu) - kRow0);
        const int col = j0 - static_cast<int>((c >> 16) - col0);
        const int lo = __builtin_amdgcn_readlane(lo_v, l);
        if (static_cast<uint32_t>(col - lo - 1) >= static_cast<uint32_t>(kBand) && i0 - l > 0 &&
            !(col == 0 && lo == 0)) {
          left_band = 1;
        }
      }
    }
    const bool stopped = (c & 0x80008000u) == 0;  // at a row that ends the walk
    int l = static_cast<int>((c & 0xffffu) - kRow0);
    const int t = static_cast<int>((c >> 16) - col0);
    asm volatile("" : "+s"(delta));  // (tested here, not on every move)
    if (delta == 0xffu) {
      l -= 0xff;
      const uint32_t pair = static_cast<uint32_t>(__builtin_amdgcn_readlane(
          static_cast<int>((index & 8u) != 0 ? rec.w : rec.z), l));
      l += static_cast<int>((index & 16u) != 0 ? pair >> 16 : pair & 0xffffu);
    }
    i = i0 - l;
    j = j0 - t;
    const int mine = (lane + columns) & (kWave - 1);  // the lane's t
    if (mine < t && j0 - 1 - mine >= 0) pos_node[j0 - 1 - mine] = out;
    if (i < 0 || j < 0) return -1;
    if (kBanded && i > 0) {
      const int lo = uniform(band_lo(i, V, length));
      if (left_band != 0 || !((j > lo && j <= lo + kBand) || (j == 0 && lo == 0))) return -2;
    }
    if (i > 0 && stopped) {
      // one move of a row of 16-bit codes
      const int c = uniform(static_cast<int>(s.code()[static_cast<int64_t>(i) * pitch + j + kShift]));
      const int kind = c & 0xc000;
      if (kind == 0xc000 || (kind != kCodeVert && j == 0)) return -1;
      if (kind != kCodeVert) {
        if (lane == 0) {
          pos_node[j - 1] = kind == kCodeDiag ? uniform(static_cast<int>(row_rec[i - 1].y)) : -1;
        }
        --j;
      }
      if (kind != kCodeHorz) {
        const int k = c & static_cast<int>(kCodePayload);
        int delta = 0;
        if (k < 4) {
          const uint4 x = row_rec[i - 1];
          const uint32_t pair = k < 2 ? x.z : x.w;
          delta = uniform(static_cast<int>((pair >> (16 * (k & 1))) & 0xffffu));
        }
        if (delta == 0) {
          const int p = uniform(s.pred_rows()[uniform(s.pred_off()[i - 1]) + k]) & kPredRowMask;
          delta = i - p;
        }
        if (delta <= 0) return -1;
        i -= delta;
        if (i < 0) return -1;
      }
      if (kBanded && i > 0) {
        const int lo = uniform(band_lo(i, V, length));
        if (!((j > lo && j <= lo + kBand) || (j == 0 && lo == 0))) return -2;
      }
    }
  }
  return j;
}

// End cell among tied sinks: spoa takes the first tied sink in its DFS order
// of the (sub)graph (roots in id order; a node's predecessors first; a lead
// node pushes its aligned set and emits it after itself, in aligned-list
// order). A root's DFS reaches exactly the nodes from which it can be
// reached along edges and aligned sets, so the aligned set G of a tied sink
// is first reached in the root iteration r = the smallest id among G and
// everything reachable from G (out-edges and aligned sets). When r is itself
// in G, r leads G and G is emitted as r followed by r's aligned list. Tied
// sinks are then ordered by (r, position after r) without the DFS: this is
// exact for sets of sinks (then r is the smallest member) and for sets whose
// descendants all have larger ids. Returns the first tied sink's row, or -1
// when some tied sink's r lies outside its set or its search outgrows the
// bound (the caller then runs the DFS).
__device__ __forceinline__ int sink_tie_by_sets(const Slot& s, int V, bool full, int best,
                                                int stack_cap) {
  constexpr int kReachCap = 256;  // nodes one search may visit
  const int lane = lane_id();
  const uint8_t* in_sub = s.in_sub();
  const int32_t* sub_order = s.sub_order();
  const int32_t* row_meta = s.row_meta();
  const int32_t* sink_score = s.sink_score();
  const uint8_t* n_aligned = s.n_aligned();
  const int32_t* aligned = s.aligned();
  const int32_t* out_head = s.out_head();
  const int32_t* e_next_out = s.e_next_out();
  const int32_t* e_head = s.e_head();
  int32_t* mark = s.tie_mark();
  int32_t* stack = s.stack();
  if (stack_cap < kReachCap) {
    return -1;
  }
  auto kept = [&](int v) { return full || in_sub[v] != 0; };
  int best_key = 0x7fffffff, best_at = -1, searches = 0;
  for (int r0 = 1; r0 <= V; r0 += kWave) {
    const int row = r0 + lane;
    unsigned long long cand = __ballot(row <= V && (row_meta[row - 1] & kRowMetaSink) != 0 &&
                                       sink_score[row] == best);
    while (cand != 0) {
      // one tied sink at a time (the searches share the visit marks)
      const int l = __ffsll(static_cast<long long>(cand)) - 1;
      cand &= cand - 1;
      const int crow = r0 + l;
      const int v = uniform(sub_order[crow - 1]);
      if (++searches >= 256) return -1;
      const int tag = s.n_seqs << 8 | searches;  // unique per layer and search
      // smallest id reachable from v's aligned set (the set included)
      int top = 0, visited = 0, r = v;
      mark[v] = tag;
      stack[top++] = v;
      while (top > 0) {
        const int x = uniform(stack[--top]);
        r = min(r, x);
        if (++visited > kReachCap) return -1;
        for (int e = uniform(out_head[x]); e != -1; e = uniform(e_next_out[e])) {
          const int h = uniform(e_head[e]);
          if (kept(h) && uniform(mark[h]) != tag) {
            if (top >= kReachCap) return -1;
            mark[h] = tag;
            stack[top++] = h;
          }
        }
        const int na = n_aligned[x];
        for (int k = 0; k < na; ++k) {
          const int a = uniform(aligned[x * kAligned + k]);
          if (kept(a) && uniform(mark[a]) != tag) {
            if (top >= kReachCap) return -1;
            mark[a] = tag;
            stack[top++] = a;
          }
        }
      }
      // r must lead v's set: r == v or r in v's aligned list
      int pos = 0;
      if (r != v) {
        bool member = false;
        const int nv = n_aligned[v];
        for (int k = 0; k < nv; ++k) member |= aligned[v * kAligned + k] == r;
        if (!member) return -1;
        const int nr = n_aligned[r];
        for (int k = 0; k < nr; ++k) {
          const int a = uniform(aligned[r * kAligned + k]);
          if (!kept(a)) continue;
          ++pos;
          if (a == v) break;
        }
      }
      const int key = r * 16 + pos;
      if (key < best_key) {
        best_key = key;
        best_at = crow;
      }
    }
  }
  return best_at;
}

// Heaviest-bundle scores over a topological rank order (spoa's
// traverse_heaviest_bundle scan): a node takes the in-edge of the highest
// weight, a later in-edge of equal weight when its tail scores at least as
// much, and adds that tail's score; nodes without in-edges keep -1. The
// recurrence is sequential in rank order, but its inputs are not: each round
// loads, for 64 ranks at once, up to kE in-edges per node (tail, weight,
// tail rank) and the scores of tails from earlier rounds; the scan then runs
// on lane registers (scores of this round's ranks are written into a lane
// register as they are found). Nodes with more in-edges read the rest from
// memory. Scores are 32-bit: the caller takes this path only when every
// path weight fits (|edge weight| <= 252 per inserted position). Writes
// scores[] and preds[]; returns the first node in rank order with the top
// score, with bit 31 set when another node ties it, or kScanUnordered (and
// nothing usable) when some tail does not precede its node in node_rank.
constexpr uint32_t kScanUnordered = 0xffffffffu;

__device__ __noinline__ uint32_t bundle_scan(GByte* slot_base, CLayout* layout, int N) {
  constexpr int kE = 8;
  const Slot s = carve(uniform_ptr(slot_base), *uniform_ptr(layout));
  N = uniform(N);
  const int lane = lane_id();
  const int32_t* r2n = s.rank_to_node();
  const int32_t* in_head = s.in_head();
  const int32_t* e_next_in = s.e_next_in();
  const int32_t* e_tail = s.e_tail();
  const int32_t* e_weight = s.e_weight();
  const int32_t* node_rank = s.node_rank();
  int64_t* scores = s.scores();
  int32_t* preds = s.preds();
  int max_node = 0;
  int max_score = -1;  // the initial max_node (node 0) scores -1 until it is scanned
  bool tied = false;
  bool unordered = false;
  for (int r0 = 0; r0 < N; r0 += kWave) {
    const int r = r0 + lane;
    const int v = r < N ? r2n[r] : -1;
    int t[kE], w[kE], tr[kE], ts[kE];
    int e = v >= 0 ? in_head[v] : -1;
#pragma unroll
    for (int j = 0; j < kE; ++j) {
      t[j] = -1;
      w[j] = 0;
      if (e != -1) {
        t[j] = e_tail[e];
        w[j] = e_weight[e];
        e = e_next_in[e];
      }
    }
#pragma unroll
    for (int j = 0; j < kE; ++j) tr[j] = t[j] != -1 ? node_rank[t[j]] : r0;
#pragma unroll
    for (int j = 0; j < kE; ++j) {
      ts[j] = t[j] != -1 && tr[j] < r0 ? static_cast<int>(scores[t[j]]) : 0;
    }
    int sc = -1;  // lane k: score of rank r0 + k
    int pr = -1;  // lane k: its predecessor
    const int n = uniform(min(kWave, N - r0));
    for (int k = 0; k < n; ++k) {
      const int vk = __builtin_amdgcn_readlane(v, k);
      int sv = -1, pv = -1, spv = 0;
      auto consider = [&](int tj, int wj, int stj) {
        if (sv < wj || (sv == wj && pv != -1 && spv <= stj)) {
          sv = wj;
          pv = tj;
          spv = stj;
        }
      };
#pragma unroll
      for (int j = 0; j < kE; ++j) {
        const int tj = __builtin_amdgcn_readlane(t[j], k);
        if (tj == -1) break;
        const int trj = __builtin_amdgcn_readlane(tr[j], k);
        unordered |= trj >= r0 + k;
        const int stj = trj >= r0 ? __builtin_amdgcn_readlane(sc, (trj - r0) & (kWave - 1))
                                  : __builtin_amdgcn_readlane(ts[j], k);
        consider(tj, __builtin_amdgcn_readlane(w[j], k), stj);
      }
      for (int f = uniform(__builtin_amdgcn_readlane(e, k)); f != -1; f = uniform(e_next_in[f])) {
        const int tj = uniform(e_tail[f]);
        const int trj = uniform(node_rank[tj]);
        unordered |= trj >= r0 + k;
        const int stj = trj >= r0 ? __builtin_amdgcn_readlane(sc, (trj - r0) & (kWave - 1))
                                  : uniform(static_cast<int>(scores[tj]));
        consider(tj, uniform(e_weight[f]), stj);
      }
      const int score = pv != -1 ? sv + spv : sv;
      sc = lane_write(score, k, sc);
      pr = lane_write(pv, k, pr);
      if (vk == max_node) {
        max_score = score;
      } else if (max_score < score) {
        max_node = vk;
        max_score = score;
        tied = false;
      } else if (max_score == score) {
        tied = true;
      }
    }
    if (v >= 0) {
      scores[v] = sc;
      preds[v] = pr;
    }
  }
  if (unordered) return kScanUnordered;
  return static_cast<uint32_t>(max_node) | (tied ? 0x80000000u : 0u);
}

// ---- the window ----

__device__ __forceinline__ void process_window(CParams& P, Slot& s, uint8_t* lds, CWindow& W,
                               PoaResult& R) {
  const int lane = lane_id();
  CCaps& caps = P.caps;
  const int pitch = static_cast<int>(caps.cols);
  const GByte* arena = global(P.arena);
  const GByte* bb = arena + W.backbone_off;
  const GByte* bq = arena + W.backbone_qual;
  const int n = static_cast<int>(W.backbone_len);
  uint64_t cells = 0;
  int max_rows = 0;
  PhaseClock clk;

  // backbone chain: nodes 0..n-1, edges i-1 -> i (weights q-33), label 0
  if (n > static_cast<int>(caps.nodes) || n - 1 > static_cast<int>(caps.edges)) {
    R.status = kPoaNodeOverflow;
    return;
  }
  for (int i = lane; i < n; i += kWave) {
    s.base()[i] = bb[i];
    s.node_info()[i] = bb[i] | (i > 0 ? 256u : 0u);
    s.node_in()[2 * i] = make_int4(i - 1, 0, 0, 0);
    s.in_head()[i] = i > 0 ? i - 1 : -1;
    s.in_tail()[i] = i > 0 ? i - 1 : -1;
    s.out_head()[i] = i + 1 < n ? i : -1;
    s.out_tail()[i] = i + 1 < n ? i : -1;
    s.n_aligned()[i] = 0;
    s.cov()[i] = n >= 2 ? 1 : 0;
    s.last_label()[i] = n >= 2 ? 0 : -1;
    s.rank_to_node()[i] = i;
    s.node_rank()[i] = i;
    if (i + 1 < n) {
      s.e_tail()[i] = i;
      s.e_head()[i] = i + 1;
      s.e_weight()[i] = (static_cast<int>(bq[i]) - 33) + (static_cast<int>(bq[i + 1]) - 33);
      s.e_next_in()[i] = -1;
      s.e_next_out()[i] = -1;
    }
  }
  s.n_nodes = n;
  s.n_edges = n > 0 ? n - 1 : 0;
  s.n_seqs = 1;
  // visit marks of the tie resolution: (layer, lane) tags, none set yet
  // (node ids stay below the slot's node capacity, which may be below the
  // window's node bound)
  const int n_marks = min(static_cast<int>(W.node_bound), static_cast<int>(caps.nodes));
  for (int v = lane; v < n_marks; v += kWave) {
    s.tie_mark()[v] = 0;
  }
  wave_sync();
  clk.lap(R, kPhaseSetup);

  for (uint32_t li = 0; li < W.n_layers; ++li) {
    CLayer& Lr = ((CLayer*)P.layers)[W.layer_first + li];
    const int L = static_cast<int>(Lr.len);
    if (L + static_cast<int>(kPoaColPad) > pitch) {
      R.status = kPoaRowOverflow;
      return;
    }
    // layer bytes and weights into the slot
    uint8_t* lds_seq = lds + align_up(static_cast<uint64_t>(P.ring_rows) * pitch * 2, 16);
    bool plain = true;  // A, C, G and T only
    for (int j = lane; j < L; j += kWave) {
      const uint8_t c = arena[Lr.seq_off + j];
      s.seq()[j] = c;
      lds_seq[j] = c;
      plain &= c == 'A' || c == 'C' || c == 'G' || c == 'T';
      s.qual()[j] = Lr.qual_off == kNoQuality
                      ? 1
                      : static_cast<int>(arena[Lr.qual_off + j]) - 33;
    }
    const bool layer_plain = __all(plain);
    const bool full = Lr.begin < W.offset && Lr.end > W.backbone_len - W.offset;
    if (static_cast<int>(Lr.end) >= s.n_nodes || Lr.begin > Lr.end) {
      R.status = kPoaBadInput;
      return;
    }

    // 1. included node set (all nodes for a layer spanning the window)
    const int nn = s.n_nodes;
    int walk_rc = 1;
    if (!full) {
      uint32_t walk_lds = static_cast<uint32_t>((size_t)(LByte*)lds);
      asm volatile("" : "+v"(walk_lds));
      walk_rc = uniform(include_ranks(s.p, s.L, walk_lds, static_cast<int>(P.ring_rows) * pitch * 2,
                                      static_cast<int>(Lr.begin), static_cast<int>(Lr.end), nn));
    }
    if (walk_rc != 0) {
      for (int v = lane; v < nn; v += kWave) {
        s.in_sub()[v] = full ? 1 : 0;
      }
      wave_sync();
      if (!full) {
        int top = 0;
        s.stack()[top++] = static_cast<int>(Lr.end);
        while (top > 0) {
          const int v = uniform(s.stack()[--top]);
          if (s.in_sub()[v] == 0 && v >= static_cast<int>(Lr.begin)) {
            const int na = s.n_aligned()[v];
            int deg = na;
            for (int e = uniform(s.in_head()[v]); e != -1; e = uniform(s.e_next_in()[e])) {
              ++deg;
            }
            if (top + deg > static_cast<int>(caps.stack)) {
              R.status = kPoaNodeOverflow;
              return;
            }
            for (int e = uniform(s.in_head()[v]); e != -1; e = uniform(s.e_next_in()[e])) {
              s.stack()[top++] = s.e_tail()[e];
            }
            for (int k = 0; k < na; ++k) {
              s.stack()[top++] = s.aligned()[v * kAligned + k];
            }
            s.in_sub()[v] = 1;
          }
        }
      }
    }
    wave_sync();

    clk.lap(R, kPhaseInclude);
    // 2. DP row order: the maintained topological order restricted to the
    // included nodes (the DP values and move codes do not depend on which
    // topological order is used; spoa's exact DFS order is computed only
    // where it decides a tie)
    int V = 0;
    // (with the DP row of every included node, row_of)
    if (full) {
      V = nn;
      for (int r = lane; r < V; r += kWave) {
        const int v = s.rank_to_node()[r];
        s.sub_order()[r] = v;
        s.row_of()[v] = r + 1;
      }
    } else {
      for (int r0 = 0; r0 < nn; r0 += kWave) {
        const int r = r0 + lane;
        const int v = r < nn ? s.rank_to_node()[r] : 0;
        const bool keep = r < nn && s.in_sub()[v] != 0;
        const unsigned long long mask = __ballot(keep);
        if (keep) {
          const int at = V + __popcll(mask & ((1ull << lane) - 1ull));
          s.sub_order()[at] = v;
          s.row_of()[v] = at + 1;
        } else if (r < nn) {
          s.row_of()[v] = 0;
        }
        V += __popcll(mask);
      }
    }
    if (V + 1 > static_cast<int>(caps.rows)) {
      R.status = kPoaRowOverflow;
      return;
    }
    max_rows = max(max_rows, V + 1);
    wave_sync();
    clk.lap(R, kPhaseSubSort);

    // score width: 16-bit ring rows when every score of the layer fits
    const int32_t max_abs = max(max(abs(P.match), abs(P.mismatch)), abs(P.gap));
    const bool narrow = static_cast<int64_t>(max_abs) * (V + L + 2) < 32000;
    // the packed one-pass rows (dp_rows) hold the layer
    int bias = 0;
    const bool rows16 = L >= 1 && L < 20 * kWave &&
                        rows_fit_16(P.match, P.mismatch, P.gap, V, L, &bias);
    // (a pass for very long layers may keep no rows in LDS at all)
    const int n_slots = min(kMaxLdsSlots, narrow || rows16 ? static_cast<int>(P.ring_rows)
                                                 : static_cast<int>(P.ring_rows) / 2);

    // predecessor rows, sink flags, slots
    uint32_t rows_lds = static_cast<uint32_t>((size_t)(LByte*)lds);
    asm volatile("" : "+v"(rows_lds));
    const int ring_bytes = static_cast<int>(P.ring_rows) * pitch * 2;
    const int max_np =
        uniform(build_rows(s.p, s.L, V, n_slots, rows_lds, ring_bytes,
                           !rows16 ? 0 : P.band != 0 && L > kBand ? 2 : 1));
    wave_sync();
    if (max_np < 0) {
      R.status = kPoaRowOverflow;  // the pooled global rows ran out: rerun exactly
      return;
    }
    if (max_np > static_cast<int>(kCodePayload) + 1) {
      // a move code holds the in-edge index in 13 bits
      R.status = kPoaInDegree;
      return;
    }

    clk.lap(R, kPhaseRows);
    // 3. DP over the layer (column 0 folded into each row)
    clk.lap(R, kPhaseColumn0);
    int best_score = 0;
    bool tied = false;
    uint64_t dp;
    CParams* pp = &P;
    CLayout* ly = s.L;
    uint32_t lds_addr = static_cast<uint32_t>((size_t)(LByte*)lds);
    // opaque to the optimizer: otherwise the callee would rebuild the address
    // from the dynamic LDS symbol (a table load) inside its loops
    asm volatile("" : "+v"(lds_addr));
    // racon -b: band rows for layers longer than the band (approximation),
    // while their scores fit signed 16 bits. Which layers the band applies to
    // is part of the option's results, so the line stays at the band's width
    // although the exact rows are the faster ones below about 600 columns:
    // 4,096 windows at 30 layers take 18.7 ms exact and 21.8 banded at 300 bp,
    // 29.9 and 35.8 at 500, 58.2 and 51.9 at 700, 162 and 99.6 at 1,000.
    const bool banded = P.band != 0 && L > kBand && max_abs <= 4096 && max_np <= 255 &&
                        static_cast<int64_t>(max_abs) * (V + 2 * L + 2) < 32000;
    // columns per lane of the packed rows
    const int row_w = L < 4 * kWave ? 4 : L < 8 * kWave ? 8 : L < 12 * kWave ? 12
                      : L < 16 * kWave ? 16 : 20;
    if (banded) {
      dp = dp_layer_call<kDpBand4>(pp, s.p, ly, lds_addr, V, L, 0);
    } else if (rows16 && row_w == 4) {
      dp = layer_plain ? dp_layer_call<kDpRows4, true>(pp, s.p, ly, lds_addr, V, L, bias)
                       : dp_layer_call<kDpRows4, false>(pp, s.p, ly, lds_addr, V, L, bias);
    } else if (rows16 && row_w == 8) {
      dp = layer_plain ? dp_layer_call<kDpRows8, true>(pp, s.p, ly, lds_addr, V, L, bias)
                       : dp_layer_call<kDpRows8, false>(pp, s.p, ly, lds_addr, V, L, bias);
    } else if (rows16 && row_w == 12) {
      dp = layer_plain ? dp_layer_call<kDpRows12, true>(pp, s.p, ly, lds_addr, V, L, bias)
                       : dp_layer_call<kDpRows12, false>(pp, s.p, ly, lds_addr, V, L, bias);
    } else if (rows16 && row_w == 16) {
      dp = layer_plain ? dp_layer_call<kDpRows16, true>(pp, s.p, ly, lds_addr, V, L, bias)
                       : dp_layer_call<kDpRows16, false>(pp, s.p, ly, lds_addr, V, L, bias);
    } else if (rows16) {
      dp = layer_plain ? dp_layer_call<kDpRows20, true>(pp, s.p, ly, lds_addr, V, L, bias)
                       : dp_layer_call<kDpRows20, false>(pp, s.p, ly, lds_addr, V, L, bias);
    } else if (narrow) {
      dp = dp_layer_call<kDpGeneric16>(pp, s.p, ly, lds_addr, V, L, 0);
    } else {
      dp = dp_layer_call<kDpGeneric32>(pp, s.p, ly, lds_addr, V, L, 0);
    }
    int best_row = uniform(static_cast<int>(static_cast<uint32_t>(dp) & 0x7fffffffu));
    best_score = uniform(static_cast<int>(dp >> 32));
    tied = uniform(static_cast<int>(static_cast<uint32_t>(dp) >> 31)) != 0;
    wave_sync();
    if (banded && best_score == kNegInf) {
      R.status = kPoaBandMiss;  // no sink reaches column L inside its band
      return;
    }
    if (tied) {
      best_row = uniform(sink_tie_by_sets(s, V, full, best_score, static_cast<int>(caps.stack)));
    }
    if (tied && best_row < 0) {
      // several sinks share the best score: spoa takes the first one in its
      // DFS order of the (sub)graph
      const int cnt = topo_sort(s, full ? nullptr : s.in_sub(), s.path(),
                                static_cast<int>(caps.stack));
      if (s.overflow) {
        R.status = kPoaNodeOverflow;
        return;
      }
      wave_sync();
      int found = -1;
      for (int i0 = 0; i0 < cnt && found < 0; i0 += kWave) {
        const int i = i0 + lane;
        bool hit = false;
        int row = 0;
        if (i < cnt) {
          row = s.row_of()[s.path()[i]];
          hit = (s.row_meta()[row - 1] & kRowMetaSink) != 0 && s.sink_score()[row] == best_score;
        }
        const unsigned long long mask = __ballot(hit);
        if (mask != 0) {
          found = __shfl(row, __ffsll(static_cast<long long>(mask)) - 1, kWave);
        }
      }
      best_row = uniform(found);
    }
    cells += static_cast<uint64_t>(V) * static_cast<uint64_t>(banded ? kBand : L);
    clk.lap(R, kPhaseDp);

    // 4. traceback, from the end cell to (0, 0). The alignment of layer
    // position p (the graph node of a diagonal move into column p + 1, or -1
    // for a horizontal move) goes to pos_node[p]; vertical moves align no
    // layer position. Packed and band rows: trace_rows. The tiled rows' 16-bit
    // codes: per round trip the wave loads the 16-row x 8-column block of codes
    // at and before the current cell (the path falls about two rows per column)
    // with the node and the predecessor-delta table of each block row, and
    // every lane turns its two cells into their successor cell in the block (or
    // "leaves the block", or "needs the lists"). The walk through the block is
    // then a chase of successor indices read from lane registers; the move that
    // leaves the block (and any the table left to the predecessor lists) is
    // taken by the full single-step decoder. The block's positions are collected
    // in one register (lane t: position j0 - 1 - t) and stored together.
    if (banded || rows16) {
      const int left = uniform(
          banded        ? trace_rows<4, true>(s.p, s.L, pitch, V, L, best_row)
          : row_w == 4  ? trace_rows<4, false>(s.p, s.L, pitch, V, L, best_row)
          : row_w == 8  ? trace_rows<8, false>(s.p, s.L, pitch, V, L, best_row)
          : row_w == 12 ? trace_rows<12, false>(s.p, s.L, pitch, V, L, best_row)
          : row_w == 16 ? trace_rows<16, false>(s.p, s.L, pitch, V, L, best_row)
                        : trace_rows<20, false>(s.p, s.L, pitch, V, L, best_row));
      if (left < 0) {
        R.status = left == -2 ? kPoaBandMiss : kPoaBadInput;
        return;
      }
      // from the virtual start row only horizontal moves remain
      for (int p = lane; p < left; p += kWave) s.path()[p] = -1;
    } else {
      const uint16_t* code = s.code();
      const int32_t* pred_off = s.pred_off();
      const int32_t* pred_rows = s.pred_rows();
      const uint4* row_rec = s.row_rec();
      int32_t* pos_node = s.path();
      constexpr uint32_t kNextExit = 0xff;  // successor: the decoder takes the move
      constexpr uint32_t kDiagBit = 0x100;
      int i = best_row, j = L;
      int steps = 0;
      const int step_cap = uniform(V + L + 1);  // every move lowers i or j
      bool bad = false;
      while (i > 0 && !bad) {
        i = uniform(i);
        j = uniform(j);
        const int i0 = i, j0 = j;
        // lane l: row i0 - (l >> 2), columns j0 - 2 (l & 3) - 0..1 (two codes
        // per register); indices outside the matrix are clamped to a valid
        // cell and the value dropped, so the loads issue unconditionally
        const int di_l = lane >> 2;
        const int ri = i0 - di_l;
        const int rc = max(ri, 1);
        const int cj = j0 - 2 * (lane & 3);
        const uint16_t* crow = code + static_cast<int64_t>(rc) * pitch;
        const uint4 rec = row_rec[rc - 1];  // graph node, first four predecessor row deltas
        const uint32_t c0 = crow[code_index(max(cj, 0), pitch)];
        const uint32_t c1 = crow[code_index(max(cj - 1, 0), pitch)];
        const uint64_t d4 = static_cast<uint64_t>(rec.w) << 32 | rec.z;
        const int nrow = static_cast<int>(rec.y);  // graph node of the row
        const uint32_t cw = ri >= 1 ? ((cj >= 0 ? c0 : 0u) | ((cj >= 1 ? c1 : 0u) << 16)) : 0u;
        wait_stores();  // the block is in registers before the walk starts
        // successor of the lane's cell (di_l, dj) as di * 8 + dj, with the
        // diagonal flag; kNextExit when the move leaves the block or row 1..,
        // reaches column 0 other than vertically, or needs the lists
        auto successor = [&](uint32_t c, int dj) -> uint32_t {
          const int kind = static_cast<int>(c & 0xc000u);
          const int pay = static_cast<int>(c & kCodePayload);
          const int delta = pay < 4 ? static_cast<int>((d4 >> (16 * pay)) & 0xffffu) : 0;
          const int jj = j0 - dj;
          if (ri < 1 || jj < 0 || (kind != kCodeVert && jj == 0) || kind == 0xc000) return kNextExit;
          int ndi = di_l, ndj = dj;
          if (kind == kCodeHorz) {
            ndj = dj + 1;
          } else {
            if (delta == 0) return kNextExit;
            ndi = di_l + delta;
            if (kind == kCodeDiag) ndj = dj + 1;
          }
          if (ndi >= 16 || ndj >= 8 || i0 - ndi <= 0) return kNextExit;
          return static_cast<uint32_t>(ndi * 8 + ndj) | (kind == kCodeDiag ? kDiagBit : 0u);
        };
        const int dja = 2 * (lane & 3);
        const uint32_t ent = successor(cw & 0xffffu, dja) | (successor(cw >> 16, dja + 1) << 16);
        int out = -1;  // lane t: the node of position j0 - 1 - t
        // moves inside the block (each raises di * 8 + dj, so at most 127)
        int idx = 0;
        for (;;) {
          const uint32_t e = (__builtin_amdgcn_readlane(ent, idx >> 1) >> (16 * (idx & 1))) & 0xffffu;
          if ((e & 0xffu) == kNextExit || steps >= step_cap) break;
          ++steps;
          if ((e & kDiagBit) != 0) {
            const int node = __builtin_amdgcn_readlane(nrow, (idx >> 3) * 4);
            out = lane == (idx & 7) ? node : out;
          }
          idx = static_cast<int>(e & 0xffu);
        }
        i = i0 - (idx >> 3);
        j = j0 - (idx & 7);
        // the move out of the block: the full decoder
        {
          const int dj = idx & 7;
          const uint32_t cp = __builtin_amdgcn_readlane(cw, idx >> 1);
          const int c = static_cast<int>((cp >> (16 * (idx & 1))) & 0xffffu);
          const int kind = c & 0xc000;
          if (++steps > step_cap || (kind != kCodeVert && j == 0)) {
            bad = true;  // only vertical moves leave column 0
          } else if (kind == kCodeHorz) {
            --j;
          } else {
            if (kind == kCodeDiag) {
              const int node = __builtin_amdgcn_readlane(nrow, (idx >> 3) * 4);
              out = lane == dj ? node : out;
              --j;
            }
            const int pay = c & static_cast<int>(kCodePayload);
            // predecessor by in-edge index: the row's delta table, else the lists
            int delta = 0;
            if (pay < 4) {
              const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(d4), (idx >> 3) * 4);
              const uint32_t hi =
                  __builtin_amdgcn_readlane(static_cast<uint32_t>(d4 >> 32), (idx >> 3) * 4);
              const uint32_t w = pay < 2 ? lo : hi;
              delta = static_cast<int>((w >> (16 * (pay & 1))) & 0xffffu);
            }
            if (delta == 0) {
              delta = i - (uniform(pred_rows[uniform(pred_off[i - 1]) + pay]) & kPredRowMask);
            }
            i -= delta;
            bad = i < 0;
          }
        }
        if (lane < j0 - j) {
          pos_node[j0 - 1 - lane] = out;
        }
      }
      if (bad) {
        R.status = kPoaBadInput;
        return;
      }
      // from the virtual start row only horizontal moves remain
      for (int p = lane; p < j; p += kWave) {
        pos_node[p] = -1;
      }
    }
    wave_sync();

    clk.lap(R, kPhaseTraceback);
    // 5. insert the layer: lane-parallel over layer positions unless two
    // nodes of the path share an aligned set (then position by position)
    bool order_ok = true;
    int n_path = 0;
    const int nodes_before = s.n_nodes;
    {
      uint32_t lseq_addr = static_cast<uint32_t>((size_t)(LByte*)lds_seq);
      asm volatile("" : "+v"(lseq_addr));
      const InsertResult ir =
          insert_parallel(s.p, s.L, lseq_addr, L, s.n_nodes, s.n_edges, s.n_seqs,
                          static_cast<int>(caps.nodes), static_cast<int>(caps.edges));
      const int rc = uniform(ir.status);
      if (rc < 0) {
        R.status = rc;
        return;
      }
      if (rc == 0) {
        s.n_nodes = uniform(ir.n_nodes);
        s.n_edges = uniform(ir.n_edges);
        s.n_seqs = s.n_seqs + 1;
        order_ok = uniform(ir.order_ok) != 0;
        n_path = L;
      } else {
        s = insert_sequential(s, caps, L, &order_ok, &n_path);
      }
    }
    if (s.overflow) {
      R.status = n_path < 0 ? kPoaAlignedFull : kPoaNodeOverflow;
      return;
    }
    wave_sync();
    clk.lap(R, kPhaseInsert);
    // topological order of the grown graph: new nodes merged after their
    // anchors (old nodes keep their relative order), then checked along the
    // inserted path; any violation falls back to the exact DFS order
    {
      const int M = s.n_nodes - nodes_before;
      const int total = s.n_nodes;
      if (order_ok && M > 0) {
        // an old node of rank r moves up by the number of anchors below r
        // (anchors are non-decreasing; searched in LDS when they fit), so a
        // sweep from the top rank down reads every entry before it is
        // overwritten; ranks up to the first anchor stay
        const int32_t* anchor = s.anchor();
        LWord* la = (LWord*)(size_t)static_cast<uint32_t>((size_t)(LByte*)lds);
        const bool anchors_in_lds = M * 4 <= static_cast<int>(P.ring_rows) * pitch * 2;
        if (anchors_in_lds) {
          for (int k = lane; k < M; k += kWave) la[k] = static_cast<uint32_t>(anchor[k]);
          wave_fence();
        }
        const int first_moved = uniform(anchor[0]) + 1;
        // four chunks of 64 ranks per round, loaded before any of their
        // stores (every store lands at or above its own rank, and later
        // rounds read only below this one)
        constexpr int kMU = 4;
        for (int r0 = ((nodes_before - 1) / kWave) * kWave; r0 + kWave > first_moved;
             r0 -= kMU * kWave) {
          int r[kMU], lo[kMU], v[kMU];
          bool moves[kMU];
#pragma unroll
          for (int u = 0; u < kMU; ++u) {
            r[u] = r0 - u * kWave + lane;
            moves[u] = r[u] >= first_moved && r[u] < nodes_before;
            v[u] = moves[u] ? s.rank_to_node()[r[u]] : 0;
          }
#pragma unroll
          for (int u = 0; u < kMU; ++u) {
            int l = 1, hi = M;  // anchor[0] < r for every moved rank
            while (__ballot(moves[u] && l < hi) != 0) {
              if (moves[u] && l < hi) {
                const int mid = (l + hi) >> 1;
                const int a = anchors_in_lds ? static_cast<int>(la[mid]) : anchor[mid];
                if (a < r[u]) l = mid + 1; else hi = mid;
              }
            }
            lo[u] = l;
          }
#pragma unroll
          for (int u = 0; u < kMU; ++u) {
            if (moves[u]) {
              s.rank_to_node()[r[u] + lo[u]] = v[u];
              s.node_rank()[v[u]] = r[u] + lo[u];
            }
          }
          wave_fence();
        }
        wave_sync();
        for (int k = lane; k < M; k += kWave) {
          const int r = anchor[k] + 1 + k;
          s.rank_to_node()[r] = nodes_before + k;
          s.node_rank()[nodes_before + k] = r;
        }
        wave_sync();
      }
      bool bad = !order_ok;
      if (!bad) {
        for (int i = lane; i + 1 < n_path; i += kWave) {
          if (s.node_rank()[s.lpath()[i]] >= s.node_rank()[s.lpath()[i + 1]]) bad = true;
        }
        bad = __ballot(bad) != 0;
      }
      if (bad) {
        topo_sort(s, nullptr, s.rank_to_node(), static_cast<int>(caps.stack));
        if (s.overflow) {
          R.status = kPoaNodeOverflow;
          return;
        }
        wave_sync();
        for (int r = lane; r < total; r += kWave) {
          s.node_rank()[s.rank_to_node()[r]] = r;
        }
      }
    }
    wave_sync();
    clk.lap(R, kPhaseSort);
  }

  clk.lap(R, kPhaseSort);

  // heaviest bundle (lane-uniform). Node scores and predecessors do not
  // depend on which topological order visits the nodes; spoa's DFS order
  // decides only which of several top-scoring nodes comes first and which
  // nodes branch completion revisits. The first pass takes the maintained
  // order; when the top score is shared or its node has out-edges, spoa's
  // exact DFS order of the final graph is computed and the bundle taken
  // again. (With no layers the backbone chain is already in DFS order.)
  const int N = s.n_nodes;
  int max_node = 0;
  // 32-bit scores: every path weight is at most 252 per inserted position
  const bool fast_scan = static_cast<int64_t>(W.node_bound) * 252 < 0x7fffffffll;
  for (int pass = 0;; ++pass) {
    const bool exact = pass > 0 || W.n_layers == 0;
    if (pass > 0) {
      clk.lap(R, kPhaseConsensus);
      topo_sort(s, nullptr, s.rank_to_node(), static_cast<int>(caps.stack));
      if (s.overflow) {
        R.status = kPoaNodeOverflow;
        return;
      }
      wave_sync();
      // ranks of the new order (the scan looks tails up by rank)
      for (int r = lane; r < N; r += kWave) {
        s.node_rank()[s.rank_to_node()[r]] = r;
      }
      wave_sync();
      clk.lap(R, kPhaseSort);
    }
    max_node = 0;
    bool top_tied = false;
    uint32_t mt = kScanUnordered;
    if (fast_scan) {
      mt = static_cast<uint32_t>(uniform(static_cast<int>(bundle_scan(s.p, s.L, N))));
      max_node = static_cast<int>(mt & 0x7fffffffu);
      top_tied = (mt >> 31) != 0;
    }
    if (mt == kScanUnordered) {
    for (int v = lane; v < N; v += kWave) {
      s.scores()[v] = -1;
      s.preds()[v] = -1;
    }
    wave_sync();
    for (int r = 0; r < N; ++r) {
      const int v = uniform(s.rank_to_node()[r]);
      for (int e = uniform(s.in_head()[v]); e != -1; e = uniform(s.e_next_in()[e])) {
        const int t = uniform(s.e_tail()[e]);
        const int64_t w = s.e_weight()[e];
        const int64_t sv = s.scores()[v];
        const int pv = s.preds()[v];
        if (sv < w || (sv == w && pv != -1 && s.scores()[pv] <= s.scores()[t])) {
          s.scores()[v] = w;
          s.preds()[v] = t;
        }
      }
      const int pv = s.preds()[v];
      if (pv != -1) {
        s.scores()[v] = s.scores()[v] + s.scores()[pv];
      }
      if (s.scores()[max_node] < s.scores()[v]) {
        max_node = v;
        top_tied = false;
      } else if (v != max_node && s.scores()[max_node] == s.scores()[v]) {
        top_tied = true;
      }
    }
    }
    wave_sync();
    if (!exact && (top_tied || s.out_head()[max_node] != -1)) continue;
    if (s.out_head()[max_node] != -1) {
      for (int r = lane; r < N; r += kWave) {
        s.node_rank()[s.rank_to_node()[r]] = r;
      }
      wave_sync();
      int guard = 0;
      while (s.out_head()[max_node] != -1) {
        if (++guard > N + 1) {
          R.status = kPoaLoopLimit;
          return;
        }
        // branch completion from the rank of max_node
        const int rank = s.node_rank()[max_node];
        const int v0 = max_node;
        for (int e = uniform(s.out_head()[v0]); e != -1; e = uniform(s.e_next_out()[e])) {
          const int h = uniform(s.e_head()[e]);
          for (int f = uniform(s.in_head()[h]); f != -1; f = uniform(s.e_next_in()[f])) {
            const int t = uniform(s.e_tail()[f]);
            if (t != v0) {
              s.scores()[t] = -1;
            }
          }
        }
        int64_t best_score = 0;
        int best_node = 0;
        for (int r = rank + 1; r < N; ++r) {
          const int u = uniform(s.rank_to_node()[r]);
          s.scores()[u] = -1;
          s.preds()[u] = -1;
          for (int e = uniform(s.in_head()[u]); e != -1; e = uniform(s.e_next_in()[e])) {
            const int t = uniform(s.e_tail()[e]);
            const int64_t st = s.scores()[t];
            if (st == -1) {
              continue;
            }
            const int64_t w = s.e_weight()[e];
            const int64_t su = s.scores()[u];
            const int pu = s.preds()[u];
            if (su < w || (su == w && pu != -1 && s.scores()[pu] <= st)) {
              s.scores()[u] = w;
              s.preds()[u] = t;
            }
          }
          const int pu = s.preds()[u];
          if (pu != -1) {
            s.scores()[u] = s.scores()[u] + s.scores()[pu];
          }
          if (best_score < s.scores()[u]) {
            best_score = s.scores()[u];
            best_node = u;
          }
        }
        max_node = best_node;
      }
    }
    break;
  }
  // path back from max_node
  int plen = 0;
  {
    int v = max_node;
    while (true) {
      s.path()[plen++] = v;
      const int p = uniform(s.preds()[v]);
      if (p == -1 || plen >= N) {
        break;
      }
      v = p;
    }
  }
  wave_sync();
  // coverage and trimming (window.cpp:118-139); path is stored backwards
  int begin = 0, end = plen - 1;
  uint8_t status = kPoaPolished;
  if ((W.flags & 3u) == 3u) {
    const int threshold = static_cast<int>(W.n_layers) / 2;  // (n_seqs - 1) / 2
    auto coverage = [&](int idx) -> int {
      const int v = s.path()[plen - 1 - idx];
      int c = s.cov()[v];
      const int na2 = s.n_aligned()[v];
      for (int k = 0; k < na2; ++k) {
        c += s.cov()[s.aligned()[v * kAligned + k]];
      }
      return c;
    };
    for (; begin < plen; ++begin) {
      if (coverage(begin) >= threshold) break;
    }
    for (; end >= 0; --end) {
      if (coverage(end) >= threshold) break;
    }
    if (begin >= end) {
      status = kPoaPolishedUntrimmed;
      begin = 0;
      end = plen - 1;
    }
  }
  const int out_len = end - begin + 1;
  if (out_len > static_cast<int>(W.out_cap)) {
    R.status = kPoaOutOverflow;
    return;
  }
  for (int i = lane; i < out_len; i += kWave) {
    global(P.out)[W.out_off + i] = s.base()[s.path()[plen - 1 - (begin + i)]];
  }
  clk.lap(R, kPhaseConsensus);
  R.length = static_cast<uint32_t>(out_len);
  R.status = status;
  R.cells = cells;
  R.nodes = static_cast<uint32_t>(N);
  R.max_rows = static_cast<uint32_t>(max_rows);
}

}  // namespace

// Persistent batch kernel: each wave takes windows from the shared queue.
// The parameters stay in device memory (read-only for the whole launch) and
// are read through a restrict pointer: uniform scalar loads, and no private
// copy of the struct (a by-value kernel argument whose address is taken is
// copied to scratch, with its fields held in vector registers).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RH_POA_WAVES_PER_EU))) void RH_POA_SYM(poa_batch_kernel)(
    const PoaParams* __restrict__ params) {
  CParams& P = *(CParams*)params;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  GByte* slot_mem = global(P.scratch) + static_cast<uint64_t>(blockIdx.x) * P.slot_bytes;
  __shared__ uint32_t next;
  while (true) {
    if (threadIdx.x == 0) {
      next = atomicAdd(P.queue_head, 1u);
    }
    __syncthreads();
    const uint32_t q = next;
    __syncthreads();
    if (q >= P.n_order) {
      break;
    }
    const uint32_t w = global(P.order)[q];
    // the heaviest windows (front of the cost-ordered queue) bound the
    // kernel's length: their waves issue ahead of the other waves of their
    // SIMD while both are ready
    if (q < P.n_priority) {
      __builtin_amdgcn_s_setprio(3);
    } else {
      __builtin_amdgcn_s_setprio(0);
    }
    Slot s = carve(slot_mem, P.layout);
    // the window's result accumulates in LDS (phase ticks are read-modify-
    // written by every lane with the same value), not in registers
    __shared__ PoaResult res;
    if (threadIdx.x == 0) {
      res = PoaResult{};
      res.status = kPoaNotRun;
    }
    __syncthreads();
    process_window(P, s, lds, ((CWindow*)P.windows)[w], res);
    __syncthreads();
    if (threadIdx.x == 0) {
      P.results[w] = res;
    }
    __syncthreads();
  }
}

// Plain kernel: one launch per window (single wave, window index given).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RH_POA_WAVES_PER_EU))) void RH_POA_SYM(poa_single_kernel)(
    const PoaParams* __restrict__ params, uint32_t q) {
  CParams& P = *(CParams*)params;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t w = global(P.order)[q];
  Slot s = carve(global(P.scratch), P.layout);
  __shared__ PoaResult res;
  if (threadIdx.x == 0) {
    res = PoaResult{};
    res.status = kPoaNotRun;
  }
  __syncthreads();
  process_window(P, s, lds, ((CWindow*)P.windows)[w], res);
  __syncthreads();
  if (threadIdx.x == 0) {
    P.results[w] = res;
  }
}

// Static-grid kernel: one workgroup per window, no queue and no cost order.
// Block b takes window order[first + b] and scratch slot b; the hardware
// dispatcher starts blocks in index order as CUs free up. Kept as the
// comparison for the persistent kernel's queue.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RH_POA_WAVES_PER_EU))) void RH_POA_SYM(poa_static_kernel)(
    const PoaParams* __restrict__ params, uint32_t first) {
  CParams& P = *(CParams*)params;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t w = global(P.order)[first + blockIdx.x];
  Slot s = carve(global(P.scratch) + static_cast<uint64_t>(blockIdx.x) * P.slot_bytes, P.layout);
  __shared__ PoaResult res;
  if (threadIdx.x == 0) {
    res = PoaResult{};
    res.status = kPoaNotRun;
  }
  __syncthreads();
  process_window(P, s, lds, ((CWindow*)P.windows)[w], res);
  __syncthreads();
  if (threadIdx.x == 0) {
    P.results[w] = res;
  }
}

}  // namespace rh

namespace rh {

// Host launchers (kept in this translation unit with the kernels).
hipError_t RH_POA_SYM(launch_poa_batch)(const PoaParams* d_params, uint32_t lds_bytes,
                                        uint32_t grid, hipStream_t stream) {
  hipLaunchKernelGGL(RH_POA_SYM(poa_batch_kernel), dim3(grid), dim3(64), lds_bytes, stream,
                     d_params);
  return hipGetLastError();
}

hipError_t RH_POA_SYM(launch_poa_single)(const PoaParams* d_params, uint32_t lds_bytes,
                                         uint32_t q, hipStream_t stream) {
  hipLaunchKernelGGL(RH_POA_SYM(poa_single_kernel), dim3(1), dim3(64), lds_bytes, stream,
                     d_params, q);
  return hipGetLastError();
}

hipError_t RH_POA_SYM(launch_poa_static)(const PoaParams* d_params, uint32_t lds_bytes,
                                         uint32_t first, uint32_t count, hipStream_t stream) {
  hipLaunchKernelGGL(RH_POA_SYM(poa_static_kernel), dim3(count), dim3(64), lds_bytes, stream,
                     d_params, first);
  return hipGetLastError();
}

hipError_t RH_POA_SYM(poa_occupancy)(int* blocks_per_cu, uint32_t lds_bytes) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu,
                                                      RH_POA_SYM(poa_batch_kernel), 64,
                                                      lds_bytes);
}

}  // namespace rh
