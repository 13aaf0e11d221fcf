// nsm_tiled.hip -- mixed-precision step with tile-local force assembly.
//
// k_element_tiled: one workgroup per element tile (nsm_tiles.h), one thread
// per element.  The tile's nodes (X, u in FP64) are staged in LDS; each
// thread runs the mixed-precision element arithmetic (nsm_mixed_math.h),
// writes F and sigma, and its 24 node forces are summed per node in a fixed
// order: gathered per corner index after one barrier where no node repeats
// a corner index in the tile, else added into FP64 LDS accumulators colour
// by colour.  Tile-interior nodes then take their whole central-difference
// update here; every other node gets this tile's partial sum (FP64, stored
// in FP32).  k_boundary_update adds the partials of the remaining nodes in
// ascending tile order and updates them.  Each kernel also leaves one
// reaction partial per workgroup.
//
// The loads a tile needs are issued before its element arithmetic (one tile
// ahead for X, u and element data, two for node ids, where workgroups walk
// several tiles; at the tile's start for the flags, mass and v of its interior
// nodes) and the kinematic-condition table sits in LDS: the F and sigma stores
// issued during the arithmetic count in the same in-order vector-memory
// counter as loads, so a load issued after them would wait until all of them
// had completed.  Lean tiles (kLeanTiles) store none and load their nodes'
// state after the arithmetic, which frees the registers it would hold.
#include "nsm_mixed_math.h"
#include "nsm_node_step.h"
#include "nsm_tiled.h"
#include "nsm_tiles.h"

#include <algorithm>
#include <type_traits>

namespace nsm {
namespace {

// Sum over the workgroup in a fixed order (butterfly inside each 64-lane
// wave, then the wave sums in ascending wave order); valid in thread 0.
template <int kThreads>
__device__ __forceinline__ double block_sum(double v, double* red)
{
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
#pragma unroll
    for (int w = 0; w < kThreads / 64; w++) s += red[w];
  return s;
}

// Tile indices are uniform; readfirstlane keeps them in scalar registers, and
// the per-tile tables (read-only for the whole launch) are read through the
// constant address space, so they come in by scalar loads, which do not
// count in the vector-memory counter.
__device__ __forceinline__ int uniform(int t) { return __builtin_amdgcn_readfirstlane(t); }

template <typename T>
__device__ __forceinline__ T tile_table(const T* p, int t)
{
  return ((const __attribute__((address_space(4))) T*)p)[t];
}

// F / sigma rows go out as buffer stores: the resource covers one tile's
// block (base and size uniform), the row offset is a scalar operand and the
// lane's element offset one vector register shared by all 60 stores, so
// the stores need no per-store address arithmetic.  A store past the block
// is dropped by the range check.  0x00020000: gfx9 resource word 3 (32-bit
// data format, which untyped buffer accesses need).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(float* p, int bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00020000);
}

constexpr int kNonTemporal = 2;  // cache-policy operand: nt

// Values of points 2p and 2p+1 of one component, side by side: one 8-byte
// store per lane.
template <int kAux>
__device__ __forceinline__ void store_pair(float even, float odd, __amdgpu_buffer_rsrc_t r, int lane_off,
                                           int row_off)
{
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  const v2u d = {__builtin_bit_cast(uint32_t, even), __builtin_bit_cast(uint32_t, odd)};
  __builtin_amdgcn_raw_buffer_store_b64(d, r, lane_off, row_off, kAux);
}

// Node ids of the (at most two) tile-node slots a thread stages, with the
// slot's partial destination (kInterior for a tile-interior node).  A thread
// past the tile's last slot gets that last slot's node (so every load stays
// unconditional) with destination kAbsent.
constexpr int kInterior = -1;
constexpr int kAbsent   = -2;
struct SlotIds {
  int gid[2];
  int dst[2];
};

template <int kThreads>
__device__ __forceinline__ SlotIds load_ids(const TileArgs& ta, const TileCtx& c)
{
  const int t  = uniform(c.t);
  const int n0 = tile_table(ta.node_off, t), nn = tile_table(ta.node_off, t + 1) - n0;
  SlotIds   r;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int ln = (int)threadIdx.x + k * kThreads;
    const int sl = n0 + staged_slot(ln, nn);
    r.gid[k]     = ta.nodes[sl] + c.node_base;
    const int d  = ta.slot_dst[sl];
    r.dst[k]     = ln < nn ? (d >= 0 ? d + c.partial_base : d) : kAbsent;
  }
  return r;
}

// Element data of one thread: local connectivity (8 x uint16) and colour
// byte.  A thread past the tile's last element takes that last element (it
// recomputes it and rewrites identical F and sigma) with colour 0xff, so it
// adds no force.
struct ElemData {
  uint4 lq;
  int   cinfo;
};

template <int kThreads>
__device__ __forceinline__ ElemData load_elem(const TileArgs& ta, int t)
{
  t               = uniform(t);
  const int e0    = tile_table(ta.elem_off, t), ne = tile_table(ta.elem_off, t + 1) - e0;
  const int64_t e = e0 + (int64_t)min((int)threadIdx.x, ne - 1);
  ElemData      d;
  d.lq    = *reinterpret_cast<const uint4*>(ta.lconn + 8 * e);
  d.cinfo = (int)threadIdx.x < ne ? (int)ta.color[e] : 0xff;
  return d;
}

// LDS of the force assembly.  Colour tiles: one FP64 accumulator per node
// slot.  Gather tiles: per node slot, the element holding it at each corner
// index (kNoElement: none), and the elements' FP32 forces component-major
// (ef[3 j + c][element]: neighbouring elements in neighbouring banks, for
// the writes and for the gathers of neighbouring slots), so a slot sums its
// at most 8 contributions in ascending corner order after one barrier.
// Column kThreads of ef is zero (absent corners read it); staging a gather
// tile rewrites it, since a colour tile's accumulators overlap it.  kLean: a
// slot's elements take the place of its X once every element has read that
// (NodeRow).
constexpr uint16_t kNoElement = 0xffff;
template <int kThreads, bool kLean>
union Assembly {
  double acc[2 * kThreads][3];
  struct {
    uint16_t inv[kLean ? 1 : 2 * kThreads][8];
    float    ef[24][kThreads + 1];
  } g;
};

// X and u of a node slot side by side (48 bytes): an element reads each of
// its nodes with three 16-byte LDS reads
union NodeRow {
  double   xu[6];
  uint16_t inv[8];
};

template <int kThreads, bool kLean>
__device__ __forceinline__ uint16_t* slot_elements(NodeRow* rows, Assembly<kThreads, kLean>& as, int ln)
{
  if constexpr (kLean)
    return rows[ln].inv;
  else
    return as.g.inv[ln];
}

// Staging of one tile: its nodes' X and u into LDS, cleared assembly slots,
// and the loads of its interior nodes' flags (and v, m when the step updates
// velocities).  Values of non-interior slots are left unset: they are never
// read, and no merge of a default forces an early wait.
struct NodeState {
  int    flg[2];
  double v[2][3], m[2];
};

__device__ __forceinline__ void load_node_state(const SlotIds& ids, int x_delta, const NodeArrays& na, int update_v,
                                                NodeState& ns)
{
#pragma unroll
  for (int k = 0; k < 2; k++)
    if (ids.dst[k] == kInterior) {
      ns.flg[k] = na.flags[ids.gid[k] + x_delta];
      if (update_v) {
        load3(na.v, ids.gid[k], ns.v[k]);
        ns.m[k] = na.mass[ids.gid[k]];
      }
    }
}

template <int kThreads, bool kLean>
__device__ __forceinline__ void stage(const SlotIds& ids, int x_delta, const double (&xr)[2][3],
                                      const double (&ur)[2][3], const NodeArrays& na, int update_v,
                                      NodeRow* rows, Assembly<kThreads, kLean>& as, bool gather, NodeState& ns,
                                      bool load_state = true)
{
  if (gather && threadIdx.x < 24) as.g.ef[threadIdx.x][kThreads] = 0.0f;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int ln = (int)threadIdx.x + k * kThreads;
    if (ids.dst[k] != kAbsent) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        rows[ln].xu[c]     = xr[k][c];
        rows[ln].xu[3 + c] = ur[k][c];
      }
      if (!gather)
#pragma unroll
        for (int c = 0; c < 3; c++) as.acc[ln][c] = 0.0;
      else if (!kLean)
        *reinterpret_cast<uint4*>(as.g.inv[ln]) = make_uint4(~0u, ~0u, ~0u, ~0u);
    }
  }
  if (load_state) load_node_state(ids, x_delta, na, update_v, ns);
}

// ---- the two kinds of element-launch work (nsm_tiled.h) ----
__device__ __forceinline__ int work_count(const ModelTileWork& w) { return w.t_count; }
__device__ __forceinline__ int work_count(const EnsTileWork& w) { return w.count; }
__device__ __forceinline__ int work_count(const UqTileWork& w) { return w.count; }
__device__ __forceinline__ int work_count(const JointTileWork& w) { return w.t_count; }
__device__ __forceinline__ int work_update_v(const ModelTileWork& w) { return w.sa.update_v; }
__device__ __forceinline__ int work_update_v(const EnsTileWork& w) { return w.es.update_v; }
__device__ __forceinline__ int work_update_v(const UqTileWork& w) { return w.sa.update_v; }
__device__ __forceinline__ int work_update_v(const JointTileWork&) { return 1; }

__device__ __forceinline__ TileCtx tile_ctx(const ModelTileWork& w, int i)
{
  return TileCtx{w.t_begin + i, 0, 0, 0, 0, 0, 0};
}
__device__ __forceinline__ TileCtx tile_ctx(const EnsTileWork& w, int i)
{
  const EnsTile   et = ens_load(w.tiles, (int64_t)uniform(i));
  const EnsSample sm = ens_load(w.samples, (int64_t)uniform(et.s));
  return TileCtx{uniform(et.t), uniform(et.s), uniform(sm.node_base), uniform(sm.x_base - sm.node_base),
                 uniform(sm.partial_base), uniform(sm.bc_base), uniform(sm.kg_base)};
}

__device__ __forceinline__ TileCtx tile_ctx(const JointTileWork& w, int i)
{
  return TileCtx{w.t_begin + i, 0, 0, 0, 0, 0, 0};
}
__device__ __forceinline__ TileCtx tile_ctx(const UqTileWork& w, int i)
{
  int s = 0;
  for (; i >= w.t_count; i -= w.t_count) s++;  // a few trajectories
  return TileCtx{w.t_begin + i, s, 0, 0, s * w.num_partials, 0, s * w.num_blocks + w.first_block};
}

// Node arrays of the item's trajectory
template <typename Work>
__device__ __forceinline__ NodeArrays work_arrays(const Work&, const TileCtx&, const NodeArrays& na)
{
  return na;
}
__device__ __forceinline__ NodeArrays work_arrays(const UqTileWork& w, const TileCtx& c, const NodeArrays& na)
{
  const UqTrajectory t = ens_load(w.traj, (int64_t)c.s);
  NodeArrays         r = na;
  r.u                  = t.u;
  r.v                  = t.v;
  r.a                  = t.a;
  r.f                  = t.f;
  return r;
}
// its kinematic conditions (not ensembles, whose items carry their own)
template <typename Work>
__device__ __forceinline__ const BcEntry* item_bc(const Work&, const TileCtx&, const NodeArrays& na)
{
  return na.bc_table;
}
__device__ __forceinline__ const BcEntry* item_bc(const UqTileWork& w, const TileCtx& c, const NodeArrays& na)
{
  return c.s > 0 ? w.sample_bc : na.bc_table;
}
// whether the item stores F and sigma and sums a reaction
template <typename Work>
__device__ __forceinline__ bool item_output(const Work&, const TileCtx&)
{
  return true;
}
__device__ __forceinline__ bool item_output(const UqTileWork&, const TileCtx& c) { return c.s == 0; }

__device__ __forceinline__ const BcEntry* work_bc(const ModelTileWork&) { return nullptr; }
__device__ __forceinline__ const BcEntry* work_bc(const UqTileWork&) { return nullptr; }
__device__ __forceinline__ const BcEntry* work_bc(const JointTileWork&) { return nullptr; }
__device__ __forceinline__ const BcEntry* work_bc(const EnsTileWork& w) { return w.bc; }

// moduli of the tile's block (tiles never straddle blocks)
template <typename Work>
__device__ __forceinline__ void tile_moduli(const Work& w, const TileCtx&, int e0, float& K, float& G)
{
  const int b = uniform(block_of(w.bt, (int64_t)e0));
  K           = w.bt.K[b];
  G           = w.bt.G[b];
}
__device__ __forceinline__ void tile_moduli(const EnsTileWork& w, const TileCtx& c, int, float& K, float& G)
{
  const int b = c.kg_base + tile_table(w.tile_block, c.t);
  K           = tile_table(w.K, b);
  G           = tile_table(w.G, b);
}

__device__ __forceinline__ void tile_moduli(const UqTileWork& w, const TileCtx& c, int e0, float& K, float& G)
{
  const int b = c.kg_base + uniform(block_of(w.bt, (int64_t)e0));
  K           = tile_table(w.K, b);
  G           = tile_table(w.G, b);
}

__device__ __forceinline__ StepArgs tile_step(const ModelTileWork& w, const TileCtx&) { return w.sa; }
__device__ __forceinline__ StepArgs tile_step(const UqTileWork& w, const TileCtx&) { return w.sa; }
__device__ __forceinline__ StepArgs tile_step(const JointTileWork& w, const TileCtx&) { return w.sa; }
__device__ __forceinline__ StepArgs tile_step(const EnsTileWork& w, const TileCtx& c)
{
  return ens_step_args(w.es, c.s);
}

// index of the tile's reaction partial
__device__ __forceinline__ int tile_rx_slot(const ModelTileWork&, const TileCtx& c, int) { return c.t; }
__device__ __forceinline__ int tile_rx_slot(const UqTileWork&, const TileCtx& c, int) { return c.t; }
__device__ __forceinline__ int tile_rx_slot(const JointTileWork&, const TileCtx& c, int) { return c.t; }
__device__ __forceinline__ int tile_rx_slot(const EnsTileWork&, const TileCtx&, int i) { return i; }

// A previous step's reaction total(s): workgroup 0 sums the model's
// partials; in an ensemble every wave of the launch takes samples in turn.
template <int kThreads, typename Work>
__device__ __forceinline__ void fold_previous(const Work& w, double* fold_red)
{
  if (w.fold.n > 0 && blockIdx.x == 0) {  // uniform
    const double total = reaction_total<kThreads>(w.fold.partials, w.fold.tiles, w.fold.n, fold_red);
    if (threadIdx.x == 0) *w.fold.out = total;
  }
}
template <int kThreads>
__device__ __forceinline__ void fold_previous(const EnsTileWork& w, double*)
{
  const EnsFold& f = w.fold;
  if (f.step < 0) return;
  constexpr int kWaves = kThreads / 64;
  for (int s = (int)blockIdx.x * kWaves + (int)(threadIdx.x >> 6); s < f.num_samples;
       s += (int)gridDim.x * kWaves) {
    const int    p0    = f.ptr[s];
    const double total = wave_reaction_total(f.partials, f.idx + p0, f.ptr[s + 1] - p0);
    if ((threadIdx.x & 63) == 0) f.hist[(int64_t)s * f.hist_stride + f.step] = total;
  }
}

// Force of a boundary node: its partials [p0, p1) in ascending tile order
// from 0.0 in FP64.  Up to 8 partials are loaded at once, then added in
// ascending order (the same order as one at a time); more than 8 continue
// one by one.
__device__ __forceinline__ void sum_partials(const float* __restrict__ partials, int64_t p0, int64_t p1, double f[3])
{
  constexpr int kBatch = 8;
  float         pv[kBatch][3];
#pragma unroll
  for (int k = 0; k < kBatch; k++)
    if (p0 + k < p1)
#pragma unroll
      for (int c = 0; c < 3; c++) pv[k][c] = partials[3 * (p0 + k) + c];
  f[0] = f[1] = f[2] = 0.0;
#pragma unroll
  for (int k = 0; k < kBatch; k++)
    if (p0 + k < p1) {
      f[0] += (double)pv[k][0];
      f[1] += (double)pv[k][1];
      f[2] += (double)pv[k][2];
    }
  for (int64_t p = p0 + kBatch; p < p1; p++) {
    f[0] += (double)partials[3 * p];
    f[1] += (double)partials[3 * p + 1];
    f[2] += (double)partials[3 * p + 2];
  }
}

// Joint steps: the reaction partial of the boundary group `group` (256 shared
// nodes) of the previous step, as k_boundary_update sums it.
template <int kThreads>
__device__ __forceinline__ void joint_reaction(const JointTileWork& w, const TileArgs& ta, const NodeArrays& na,
                                               int group, double* red)
{
  for (int t0 = 0; t0 < kBoundaryNodesPerGroup; t0 += kThreads) {
    const int t = t0 + (int)threadIdx.x;
    if (t >= kBoundaryNodesPerGroup) break;  // whole waves
    const int bi = (group - ta.num_tiles) * kBoundaryNodesPerGroup + t;
    double    v  = 0.0;
    if (bi < ta.num_bnd && (na.flags[ta.bnd_base + bi] & kReactionFlag)) {
      double f[3];
      sum_partials(w.partials_in, ta.bnd_ptr[bi], ta.bnd_ptr[bi + 1], f);
      v = f[w.coord];
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
    if ((t & 63) == 0) red[t >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kBoundaryNodesPerGroup / 64; q++) s += red[q];
    w.prev_rx[group] = s;
  }
}

// Joint steps: u of the thread's slots, the shared nodes' after their
// previous step (see JointTileWork), and the flags, mass and v of its
// interior nodes (left in ns).  Every load of both slots is issued before the
// first is used, whatever kind of slot it is (an interior slot's partials are
// entry 0, not used; a slot past the tile's last loads that one's values,
// from the arrays that hold its node): a branch around them would make the
// kernel wait for one slot's chain after the other's.  table (LDS) is staged in the meantime.
template <int kThreads>
__device__ __forceinline__ void joint_nodes(const JointTileWork& w, const TileArgs& ta, const TileCtx& c,
                                            const SlotIds& ids, const NodeArrays& na, const BcEntry* table,
                                            double (&ur)[2][3], NodeState& ns)
{
  constexpr int kBatch = 8;
  const int     n0 = tile_table(ta.node_off, c.t), nn = tile_table(ta.node_off, c.t + 1) - n0;
  int2          p[2];
  float         pv[2][kBatch][3];
#pragma unroll
  for (int k = 0; k < 2; k++) p[k] = w.slot_partials[n0 + staged_slot((int)threadIdx.x + k * kThreads, nn)];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int  i      = ids.gid[k];
    const bool shared = has_boundary_row(i, ta.bnd_base);
    load3(shared ? w.bu_in : na.u, i, ur[k]);
    load3(shared ? w.bv_in : na.v, i, ns.v[k]);
    ns.flg[k] = na.flags[i];
    ns.m[k]   = na.mass[i];
  }
  if (w.kick)  // uniform
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < kBatch; j++)
#pragma unroll
        for (int cc = 0; cc < 3; cc++) pv[k][j][cc] = w.partials_in[3 * (p[k].x + max(min(j, p[k].y - 1), 0)) + cc];
  __syncthreads();  // table
  if (!w.kick) return;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    if (ids.dst[k] == kInterior || ids.dst[k] == kAbsent) continue;
    double f[3] = {0.0, 0.0, 0.0}, v[3] = {ns.v[k][0], ns.v[k][1], ns.v[k][2]}, a[3];
#pragma unroll
    for (int j = 0; j < kBatch; j++)
      if (j < p[k].y)
#pragma unroll
        for (int cc = 0; cc < 3; cc++) f[cc] += (double)pv[k][j][cc];
    for (int64_t q = p[k].x + kBatch; q < p[k].x + p[k].y; q++)
#pragma unroll
      for (int cc = 0; cc < 3; cc++) f[cc] += (double)w.partials_in[3 * q + cc];
    const int i = ids.gid[k];
    node_advance(table, ns.flg[k] & 0x7f, f, ur[k], v, a, ns.m[k], w.prev);
    if (ids.dst[k] == p[k].x) {  // the node's first tile
      store3_stream(na.f, i, f);
      store3(w.bu_out, i, ur[k]);
      store3(w.bv_out, i, v);
    }
  }
}

// Persistent workgroups, each walking every G-th tile, or (kOne) a workgroup
// per work item, which loads nothing ahead.  kThreads elements
// and at most 2*kThreads nodes per tile.  While tile t computes, X, u and
// element data of its next tile and node ids of the one after are in flight;
// the next tile is staged into LDS at the end of the iteration.
// Inside the loop every vector load and every F / sigma store is executed on
// every path (indices clamped), so at least the 120 stores of the element
// arithmetic always separate a load from its first use and the waits the
// compiler places never wait for those stores.  kStoreIp = false (ensembles
// and off-nominal UQ samples, which keep no element data) stores nothing,
// but each Gauss-point pair's stress still passes through an empty asm
// statement where its stores would be: with no such point of use the
// compiler schedules the element arithmetic with more registers than a wave
// pair has and spills.  The launch bound
// holds the kernel to two waves per SIMD (at most 256 registers): left free,
// the scheduler takes more for the gather assembly and halves occupancy.
//
// kLeanTiles: ensembles with a workgroup per item run three waves per SIMD,
// in 168 registers and a third less LDS: no next item in registers, the
// nodes' state loaded after the element arithmetic, the slots' elements where
// their X was.  With no element data to store the arithmetic's issue bounds
// them, and a third wave fills what two left idle: 64 meshes of 32^3 elements
// 8.56 -> 6.72 ms per 40 steps, 128 of 24^3 in 64-element tiles 8.94 -> 5.91.
// Kernels that store element data gain nothing from it (52^3 elements,
// 128-element tiles, 29.9 / 29.5 us, 74^3 63.4 / 69.8, 16 windows 314 / 374).
template <int kThreads, bool kOne, typename Work>
constexpr bool kLeanTiles = kOne && kThreads < 512 && std::is_same<Work, EnsTileWork>::value;

template <int kThreads, bool kStoreIp, bool kOne, typename Work>
__global__ __launch_bounds__(kThreads, (kLeanTiles<kThreads, kOne, Work> ? 3 : 2)) void k_element_tiled(
    const Work work, TileArgs ta, const double* __restrict__ X, NodeArrays na, float* __restrict__ Fip,
    float* __restrict__ sip, ReactionArgs rx, int* __restrict__ status)
{
  constexpr int  kNodes      = 2 * kThreads;
  constexpr bool kEnsemble   = std::is_same<Work, EnsTileWork>::value;
  constexpr bool kUq         = std::is_same<Work, UqTileWork>::value;
  constexpr bool kJoint      = std::is_same<Work, JointTileWork>::value;
  static_assert(!kJoint || kOne, "a joint step's grid holds every tile");
  // ensembles stage each tile's sample's kinematic-condition entries (one
  // 8-byte word per thread)
  constexpr int  kTileBcWords = kBcWords * kEnsMaxBcCodes;
  static_assert(!kEnsemble || kTileBcWords <= kThreads, "one condition word per thread");
  constexpr bool kLean       = kLeanTiles<kThreads, kOne, Work>;
  __shared__ __attribute__((aligned(16))) NodeRow rows[kNodes];
  __shared__ __attribute__((aligned(16))) Assembly<kThreads, kLean> as;
  __shared__ double  red[kThreads / 64];
  __shared__ BcEntry sbc[kEnsemble ? kEnsMaxBcCodes : kMaxBcEntries];
  __shared__ int     bad;
  __shared__ double  fold_red[256];

  unsigned block = blockIdx.x, blocks = gridDim.x;
  if constexpr (kJoint) {
    if (block < work.reaction_groups) {  // uniform
      const bool last = work.fold.n > 0 && block == work.reaction_groups - 1;
      if (last) {
        const double total = reaction_total<kThreads>(work.fold.partials, work.fold.tiles, work.fold.n, fold_red);
        if (threadIdx.x == 0) *work.fold.out = total;
      } else {
        joint_reaction<kThreads>(work, ta, na, work.groups[block], fold_red);
      }
      return;
    }
    block -= work.reaction_groups;
    blocks -= work.reaction_groups;
  } else {
    fold_previous<kThreads>(work, fold_red);
  }

  // Workgroup w (numbered so that each XCD holds a contiguous run of w)
  // processes work items w, w + G, w + 2G, ... (G workgroups): at any time
  // the grid works on one window of G consecutive tiles, so the F and sigma
  // rows are written in one narrow address range and each XCD's L2 sees
  // neighbouring tiles.
  const int G        = (int)blocks;
  const int w        = (int)xcd_tile(block, blocks);
  const int count    = work_count(work);
  const int update_v = work_update_v(work);
  const int ib       = uniform(w);
  if (ib >= count) return;  // uniform across the workgroup
  // last work item of this workgroup, and the item after i (i itself if none)
  const int  ie   = uniform(ib + ((count - 1 - ib) / G) * G + 1);
  const auto next = [&](int i) { return i + G < ie ? i + G : i; };
  const int  tid  = (int)threadIdx.x;

  // ---- prologue: stage item ib, load item ib+G's node ids
  if (tid == 0) bad = 0;
  TileCtx c_first = tile_ctx(work, ib);
  if (!kEnsemble && update_v)
    for (int b = tid; b < na.num_bc; b += kThreads) sbc[b] = item_bc(work, c_first, na)[b];
  if (kEnsemble && tid < kTileBcWords)
    reinterpret_cast<uint64_t*>(sbc)[tid] =
        reinterpret_cast<const uint64_t*>(work_bc(work) + c_first.bc_base)[tid];
  SlotIds ids      = load_ids<kThreads>(ta, c_first);
  ElemData  cur = load_elem<kThreads>(ta, c_first.t);
  NodeState ns;
  SlotIds   ids_next{};
  if (!kOne) ids_next = load_ids<kThreads>(ta, tile_ctx(work, next(ib)));
  double  xr[2][3], ur[2][3];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    load3(X, ids.gid[k] + c_first.x_delta, xr[k]);
    if (!kJoint) load3(work_arrays(work, c_first, na).u, ids.gid[k], ur[k]);
  }
  if constexpr (kJoint) joint_nodes<kThreads>(work, ta, c_first, ids, na, sbc, ur, ns);
  stage<kThreads, kLean>(ids, c_first.x_delta, xr, ur, work_arrays(work, c_first, na), update_v, rows, as,
                  tile_table(ta.gather, c_first.t) != 0, ns, !kJoint && !kLean);
  // every prologue load complete (vmcnt(0); lgkmcnt and expcnt at their
  // maximum, gfx9 encoding): the loop's waits then depend on its body only
  __builtin_amdgcn_s_waitcnt(0x0F70);

  for (int il = ib; il < ie; il += G) {
    const int     i    = uniform(il);
    const TileCtx c    = tile_ctx(work, i);
    const TileCtx cn   = tile_ctx(work, next(i));
    const int     t    = c.t;
    const int     e0   = tile_table(ta.elem_off, t);
    const int     ncol = tile_table(ta.num_colors, t);
    __syncthreads();  // tile t staged

    // ---- prefetch (clamped to this workgroup's last item): the next
    // item's nodes and elements, the node ids of the one after, and (in
    // ensembles) the next item's sample's condition entries
    ElemData el_next   = cur;
    SlotIds  ids_after = ids;
    if (!kOne) {
#pragma unroll
      for (int k = 0; k < 2; k++) {
        load3(X, ids_next.gid[k] + cn.x_delta, xr[k]);
        load3(work_arrays(work, cn, na).u, ids_next.gid[k], ur[k]);
      }
      el_next   = load_elem<kThreads>(ta, cn.t);
      ids_after = load_ids<kThreads>(ta, tile_ctx(work, next(next(i))));
    }
    uint64_t       bc_next   = 0;
    if (kEnsemble && !kOne)
      bc_next = reinterpret_cast<const uint64_t*>(work_bc(work) + cn.bc_base)[min(tid, kTileBcWords - 1)];

    // ---- element arithmetic (every thread; see load_elem)
    const int ntl = tile_table(ta.elem_off, t + 1) - e0;  // elements of tile t
    const int lcl = min(tid, ntl - 1);
    float         f[8][3];
    uint16_t      lc[8];
    lc[0] = (uint16_t)(cur.lq.x & 0xffff);
    lc[1] = (uint16_t)(cur.lq.x >> 16);
    lc[2] = (uint16_t)(cur.lq.y & 0xffff);
    lc[3] = (uint16_t)(cur.lq.y >> 16);
    lc[4] = (uint16_t)(cur.lq.z & 0xffff);
    lc[5] = (uint16_t)(cur.lq.z >> 16);
    lc[6] = (uint16_t)(cur.lq.w & 0xffff);
    lc[7] = (uint16_t)(cur.lq.w >> 16);
    {
      double Xe[8][3], ue[8][3];
#pragma unroll
      for (int j = 0; j < 8; j++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
          Xe[j][c] = rows[lc[j]].xu[c];
          ue[j][c] = rows[lc[j]].xu[3 + c];
        }
      float Kt, Gt;
      tile_moduli(work, c, e0, Kt, Gt);
      // tile-blocked F and sigma: tile t owns [72 e0, 72 (e0 + n)) and
      // [48 e0, 48 (e0 + n)), in rows (component c, point pair p) of 2n
      // values, element l's points 2p and 2p+1 side by side, so each tile
      // writes two contiguous blocks with 8-byte stores; non-temporal stores
      // (the step never reads them back) keep node data and partials in cache
      float* const Ft   = kStoreIp ? Fip + (int64_t)e0 * 72 : nullptr;
      float* const St   = kStoreIp ? sip + (int64_t)e0 * 48 : nullptr;
      // an item without element data has blocks of no bytes: its stores are
      // dropped by the range check
      const int    nst  = item_output(work, c) ? ntl : 0;
      const auto   rF   = tile_rsrc(Ft, 72 * 4 * nst);
      const auto   rS   = tile_rsrc(St, 48 * 4 * nst);
      const int    loff = 8 * lcl;
      auto store = [&](int qm, int qp, const float* Fm, const float* Sm, const float* Fp, const float* Sp) {
        const bool   m_even = qm < qp;  // qm, qp: constants after inlining
        const int    p      = (m_even ? qm : qp) / 2;
        const float* Fe     = m_even ? Fm : Fp;
        const float* Fo     = m_even ? Fp : Fm;
        const float* Se     = m_even ? Sm : Sp;
        const float* So     = m_even ? Sp : Sm;
        if (kStoreIp) {
#pragma unroll
          for (int c = 0; c < 9; c++) store_pair<kNonTemporal>(Fe[c], Fo[c], rF, loff, 8 * (c * 4 + p) * ntl);
#pragma unroll
          for (int c = 0; c < 6; c++) store_pair<kNonTemporal>(Se[c], So[c], rS, loff, 8 * (c * 4 + p) * ntl);
        } else {
          // the pair's point of use (see above); emits no instruction
#pragma unroll
          for (int c = 0; c < 6; c++) asm volatile("" ::"v"(Se[c]), "v"(So[c]));
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (!mixed::element(Xe, ue, Kt, Gt, store, f)) bad = 1;
    }

    if constexpr (kLean) load_node_state(ids, c.x_delta, work_arrays(work, c, na), update_v, ns);

    const bool gather = tile_table(ta.gather, t) != 0;  // uniform
    if (gather) {
      // ---- gather tiles: every element publishes its forces and, for each
      // corner j, itself as the slot's corner-j element (no other element of
      // the tile holds that slot at corner j)
      if constexpr (kLean) {
        __syncthreads();  // every element has read its nodes
#pragma unroll
        for (int k = 0; k < 2; k++)
          *reinterpret_cast<uint4*>(rows[tid + k * kThreads].inv) = make_uint4(~0u, ~0u, ~0u, ~0u);
        __syncthreads();
      }
      if (tid < ntl) {
#pragma unroll
        for (int j = 0; j < 8; j++) slot_elements<kThreads, kLean>(rows, as, lc[j])[j] = (uint16_t)tid;
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
          for (int c = 0; c < 3; c++) as.g.ef[3 * j + c][tid] = f[j][c];
      }
      __syncthreads();
    } else {
      // ---- colour-ordered assembly: the elements of one colour touch
      // distinct nodes.  An element's 8 nodes are distinct unless it is
      // flagged kRepeatedNode, so its 24 updates are done as one batch of
      // reads, adds and writes; a flagged element adds node by node.
      const int  col      = cur.cinfo == 0xff ? -1 : (cur.cinfo & kColorMask);
      const bool repeated = cur.cinfo != 0xff && (cur.cinfo & kRepeatedNode) != 0;
      for (int c = 0; c < ncol; c++) {
        if (col == c) {
          if (!repeated) {
            double a[8][3];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
              for (int k = 0; k < 3; k++) a[j][k] = as.acc[lc[j]][k];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
              for (int k = 0; k < 3; k++) as.acc[lc[j]][k] = a[j][k] + (double)f[j][k];
          } else {
            for (int j = 0; j < 8; j++)
              for (int k = 0; k < 3; k++) as.acc[lc[j]][k] += (double)f[j][k];
          }
        }
        __syncthreads();
      }
    }

    // ---- interior nodes: complete step; others: this tile's partial
    const StepArgs   sa  = tile_step(work, c);
    const NodeArrays nac = work_arrays(work, c, na);
    double           rxs = 0.0;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int ln = tid + k * kThreads;
      if (ids.dst[k] == kAbsent) continue;
      double fn[3];
      if (gather) {
        // the slot's contributions in ascending corner order, from 0.0
        const uint4    iv   = *reinterpret_cast<const uint4*>(slot_elements<kThreads, kLean>(rows, as, ln));
        const unsigned wd[4] = {iv.x, iv.y, iv.z, iv.w};
        fn[0] = fn[1] = fn[2] = 0.0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const unsigned e  = (wd[j >> 1] >> (16 * (j & 1))) & 0xffffu;
          const int      ec = e == kNoElement ? kThreads : (int)e;
#pragma unroll
          for (int cc = 0; cc < 3; cc++) fn[cc] += (double)as.g.ef[3 * j + cc][ec];
        }
      } else {
#pragma unroll
        for (int cc = 0; cc < 3; cc++) fn[cc] = as.acc[ln][cc];
      }
      if (ids.dst[k] == kInterior) {
        if (rx.coord >= 0 && (ns.flg[k] & kReactionFlag)) rxs += fn[rx.coord];
        double un[3] = {rows[ln].xu[3], rows[ln].xu[4], rows[ln].xu[5]};
        node_update(nac, sbc, ids.gid[k], ns.flg[k], fn, un, ns.v[k], ns.m[k], sa);
      } else {
        float* const pp = ta.partials + 3 * (int64_t)ids.dst[k];
        pp[0]           = (float)fn[0];
        pp[1]           = (float)fn[1];
        pp[2]           = (float)fn[2];
      }
    }
    if (rx.coord >= 0 && item_output(work, c)) {  // uniform across the workgroup
      const double s = block_sum<kThreads>(rxs, red);
      if (threadIdx.x == 0) rx.partials[tile_rx_slot(work, c, i)] = s;
    }
    if (kOne) break;
    __syncthreads();  // tile t's LDS reads done

    // ---- stage the next item
    ids      = ids_next;
    ids_next = ids_after;
    cur      = el_next;
    if (i + G < ie) {
      if (kEnsemble && tid < kTileBcWords) reinterpret_cast<uint64_t*>(sbc)[tid] = bc_next;
      if (kUq && update_v && (c.s > 0) != (cn.s > 0))  // the next item's conditions (once per launch)
        for (int b = tid; b < na.num_bc; b += kThreads) sbc[b] = item_bc(work, cn, na)[b];
      stage<kThreads, kLean>(ids, cn.x_delta, xr, ur, work_arrays(work, cn, na), update_v, rows, as,
                      tile_table(ta.gather, cn.t) != 0, ns);
    }
  }
  if (tid == 0 && bad) raise(status);
}

constexpr int kBndThreads = kBoundaryNodesPerGroup;

// Closure terms (UqModel::ApplyClosure, src/uq/nimble_uq.cc:327-346) with
// separate multiply and add, as k_uq_closure rounds them
__device__ __forceinline__ double closure_scale(double f, double c)
{
#pragma clang fp contract(off)
  return f * c;
}
__device__ __forceinline__ void closure_add(double f[3], const double g[3], double c)
{
#pragma clang fp contract(off)
  f[0] += g[0] * c;
  f[1] += g[1] * c;
  f[2] += g[2] * c;
}

// Boundary node bi (partials [p0, p1)) at row i, flags at row xi: its force,
// then the node update.  Returns its reaction contribution.
__device__ __forceinline__ double boundary_node(const TileArgs& ta, const NodeArrays& na, const BcEntry* table,
                                                int64_t i, int64_t xi, int64_t p0, int64_t p1, const StepArgs& sa,
                                                int rx_coord)
{
  // the node's own state is loaded first, so its latency overlaps the
  // dependent partial-sum loads
  const int flags = na.flags[xi];
  double    u[3], v[3], m = 1.0;
  if (sa.update_v) {
    load3(na.u, i, u);
    load3(na.v, i, v);
    m = na.mass[i];
  }
  double f[3];
  sum_partials(ta.partials, p0, p1, f);
  const double rxs = rx_coord >= 0 && (flags & kReactionFlag) ? f[rx_coord] : 0.0;
  node_update(na, table, i, flags, f, u, v, m, sa);
  return rxs;
}

__global__ __launch_bounds__(kBndThreads) void k_boundary_update(TileArgs ta, NodeArrays na, StepArgs sa,
                                                                 ReactionArgs rx)
{
  __shared__ double red[kBndThreads / 64];
  const unsigned    g   = xcd_tile(blockIdx.x, gridDim.x);
  const int         bi  = (int)g * kBndThreads + threadIdx.x;
  double            rxs = 0.0;
  if (bi < ta.num_bnd) {
    const int64_t i = (int64_t)ta.bnd_base + bi;
    rxs = boundary_node(ta, na, na.bc_table, i, i, ta.bnd_ptr[bi], ta.bnd_ptr[bi + 1], sa, rx.coord);
  }
  if (rx.coord < 0) return;
  const double s = block_sum<kBndThreads>(rxs, red);
  if (threadIdx.x == 0) rx.partials[ta.num_tiles + g] = s;
}

// Off-nominal ensemble, one launch for every node: workgroups [0, groups)
// take the boundary nodes, each thread its node's force and update for the
// nominal trajectory and every exact sample, the rest the interior nodes,
// whose forces the element launch stored.  With the trajectories' forces in
// registers a thread then runs the closure of the approximate samples, as
// k_uq_closure does.  One launch where a step took one boundary launch per
// trajectory and the closure: at 48^3 with two exact and five approximate
// samples 122 -> 72 us per step (element 43, this 28).
__global__ __launch_bounds__(kBndThreads) void k_uq_nodes(TileArgs ta, NodeArrays na, const BcEntry* sample_bc,
                                                          UqClosure uc, int num_partials, unsigned groups,
                                                          StepArgs sa, ReactionArgs rx)
{
  __shared__ double red[kBndThreads / 64];
  const int         ne  = uc.num_exact;
  const bool        bnd = blockIdx.x < groups;  // uniform
  const unsigned    g   = bnd ? xcd_tile(blockIdx.x, groups) : xcd_tile(blockIdx.x - groups, gridDim.x - groups);
  const int64_t     l   = (int64_t)g * kBndThreads + threadIdx.x;
  const int64_t     i   = bnd ? ta.bnd_base + l : l;
  double            rxs = 0.0;
  if (l < (bnd ? ta.num_bnd : ta.bnd_base)) {
    const int  flags = na.flags[i];
    NodeArrays ns    = na;  // a sample's arrays
    ns.bc_table      = sample_bc;
    const auto of    = [&](int s) {
      double* b = uc.state + 4 * (int64_t)s * uc.stride;
      ns.u      = b;
      ns.v      = b + uc.stride;
      ns.a      = b + 2 * uc.stride;
      ns.f      = b + 3 * uc.stride;
    };
    double fn[3], fe[kUqCachedExact][3];
    if (bnd) {
      const int64_t p0 = ta.bnd_ptr[l], p1 = ta.bnd_ptr[l + 1];
      sum_partials(ta.partials, p0, p1, fn);
      if (rx.coord >= 0 && (flags & kReactionFlag)) rxs = fn[rx.coord];
      double u[3];
      if (sa.update_v) load3(na.u, i, u);
      node_step(na, i, flags, fn, u, sa);
#pragma unroll
      for (int k = 0; k < kUqCachedExact; k++)
        if (k < ne) {
          const int64_t q = (int64_t)(k + 1) * num_partials;
          sum_partials(ta.partials, q + p0, q + p1, fe[k]);
          of(k);
          if (sa.update_v) load3(ns.u, i, u);
          node_step(ns, i, flags, fe[k], u, sa);
        }
    } else {
      load3(uc.f_nominal, i, fn);
#pragma unroll
      for (int k = 0; k < kUqCachedExact; k++)
        if (k < ne) load3(uc.state + (4 * (int64_t)k + 3) * uc.stride, i, fe[k]);
    }
    for (int s = 0; s < uc.num_approx; s++) {
      const double* c    = uc.coeff + (int64_t)s * (ne + 1);
      double        f[3] = {closure_scale(fn[0], c[0]), closure_scale(fn[1], c[0]), closure_scale(fn[2], c[0])};
#pragma unroll
      for (int k = 0; k < kUqCachedExact; k++)
        if (k < ne) closure_add(f, fe[k], c[k + 1]);
      of(ne + s);
      double u[3];
      if (sa.update_v) load3(ns.u, i, u);
      node_step(ns, i, flags, f, u, sa);
    }
  }
  if (rx.coord < 0 || !bnd) return;  // uniform
  const double s = block_sum<kBndThreads>(rxs, red);
  if (threadIdx.x == 0) rx.partials[ta.num_tiles + g] = s;
}

// Ensemble boundary nodes: group g is nodes [first, first + count) of the
// boundary nodes of sample groups[g].s.
__global__ __launch_bounds__(kBndThreads) void k_ens_boundary_update(TileArgs ta, EnsNodes en,
                                                                     const EnsRange* __restrict__ groups, EnsStep es,
                                                                     ReactionArgs rx, int rx_base)
{
  __shared__ double red[kBndThreads / 64];
  const unsigned    g   = xcd_tile(blockIdx.x, gridDim.x);
  const EnsRange    gr  = ens_load(groups, (int64_t)g);
  const EnsSample   sm  = ens_load(en.samples, (int64_t)gr.s);
  const EnsMesh     ms  = ens_load(en.meshes, (int64_t)sm.mesh);
  const StepArgs    sa  = ens_step_args(es, gr.s);
  double            rxs = 0.0;
  if ((int)threadIdx.x < gr.count) {
    const int     bi  = gr.first + (int)threadIdx.x;
    const int64_t loc = (int64_t)ms.num_interior + bi;  // mesh-local device row
    NodeArrays    na;
    na.num_nodes   = 0;
    na.slot_stride = 0;
    na.node_ptr    = nullptr;
    na.node_ent    = nullptr;
    na.mass        = en.mass;
    na.u           = en.u;
    na.v           = en.v;
    na.a           = en.a;
    na.f           = en.f;
    na.flags       = en.flags;
    na.bc_table    = en.bc;
    na.num_bc      = 0;
    const int64_t p0 = (int64_t)sm.partial_base + ta.bnd_ptr[ms.bnd_pos + bi];
    const int64_t p1 = (int64_t)sm.partial_base + ta.bnd_ptr[ms.bnd_pos + bi + 1];
    rxs = boundary_node(ta, na, en.bc + sm.bc_base, sm.node_base + loc, sm.x_base + loc, p0, p1, sa, rx.coord);
  }
  if (rx.coord < 0) return;
  const double s = block_sum<kBndThreads>(rxs, red);
  if (threadIdx.x == 0) rx.partials[rx_base + (int)g] = s;
}

}  // namespace

unsigned boundary_grid(int num_bnd) { return (unsigned)((num_bnd + kBndThreads - 1) / kBndThreads); }

template <int kThreads, bool kOne, typename Work>
void launch_tiles(unsigned grid, const Work& work, const TileArgs& ta, const double* X, const NodeArrays& na,
                  float* Fip, float* sip, ReactionArgs rx, int* status, hipStream_t s, const LaunchTimer& t)
{
  const auto launch = [&](auto kernel) {
    hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, s, t.start, t.stop, 0, work, ta, X, na, Fip, sip, rx,
                          status);
  };
  // an off-nominal ensemble's launch always holds the nominal trajectory; a
  // batched ensemble keeps no element data
  if constexpr (std::is_same<Work, EnsTileWork>::value)
    launch(k_element_tiled<kThreads, false, kOne, Work>);
  else if (std::is_same<Work, UqTileWork>::value || std::is_same<Work, JointTileWork>::value || Fip)
    launch(k_element_tiled<kThreads, true, kOne, Work>);
  else if constexpr (std::is_same<Work, ModelTileWork>::value)
    launch(k_element_tiled<kThreads, false, kOne, Work>);
}

template <bool kOne, typename Work>
void launch_grid(const Work& work, unsigned grid, const TileArgs& ta, const double* X, const NodeArrays& na,
                 float* Fip, float* sip, ReactionArgs rx, int* status, hipStream_t s, const LaunchTimer& t)
{
  switch (ta.tile_elems) {
    case 64: launch_tiles<64, kOne>(grid, work, ta, X, na, Fip, sip, rx, status, s, t); break;
    case 128: launch_tiles<128, kOne>(grid, work, ta, X, na, Fip, sip, rx, status, s, t); break;
    case 512: launch_tiles<512, kOne>(grid, work, ta, X, na, Fip, sip, rx, status, s, t); break;
    default: launch_tiles<256, kOne>(grid, work, ta, X, na, Fip, sip, rx, status, s, t);
  }
}

// One workgroup per item where the last window of a persistent grid is little
// filled.  The persistent workgroups take equally many items each, the next
// one's loads behind the current one's arithmetic, and in the last window
// most of them have run out; a workgroup per item starts as another ends, but
// waits out its loads.  us per step, persistent / per item, models of
// 256-element tiles (512 at once): 1.07 windows 37.7 / 32.4, 1.65 40.4 / 41.5,
// 2.0 42.2 / 44.3, 3.1 69.9 / 64.7, 4.2 89.9 / 84.0.  512-element tiles fill a
// CU with one workgroup, so nothing runs during those loads: 3.1 windows 70.5
// / 73.6.  Ensembles' tiles (kLeanTiles) go one per workgroup at any number:
// 1.7 windows 1597 / 1378 us per 40 steps, 5.0 3205 / 2701, 16.0 8580 / 6720.
bool last_window_partial(int64_t items, const TileArgs& ta, int tenths)
{
  const int64_t window = std::max(ta.resident_groups, 1);
  return ta.tile_elems < kTileElems && items % window != 0 && 10 * (items % window) <= tenths * window;
}

template <typename Work>
void launch_work(const Work& work, int count, const TileArgs& ta, const double* X, const NodeArrays& na, float* Fip,
                 float* sip, ReactionArgs rx, int* status, hipStream_t s, const LaunchTimer& t = LaunchTimer{})
{
  if (count <= 0) return complete_timer(t, s);
  const int window = std::max(ta.resident_groups, 1);
  const bool each  = kLeanTiles<64, true, Work> && ta.tile_elems < kTileElems;
  if (each || count <= window || last_window_partial(count, ta, 6))
    launch_grid<true>(work, (unsigned)count, ta, X, na, Fip, sip, rx, status, s, t);
  else
    launch_grid<false>(work, (unsigned)window, ta, X, na, Fip, sip, rx, status, s, t);
}

void launch_element_tiled(const BlockTable<float>& bt, const TileArgs& ta, int t_begin, int t_count,
                          const double* X, const NodeArrays& na, float* Fip, float* sip, const StepArgs& sa,
                          ReactionArgs rx, ReactionFold fold, int* status, hipStream_t s, const LaunchTimer& timer)
{
  const ModelTileWork work{bt, t_begin, t_count, sa, fold};
  launch_work(work, t_count, ta, X, na, Fip, sip, rx, status, s, timer);
}

void launch_ens_element_tiled(const EnsTileWork& work, const TileArgs& ta, const double* X, const NodeArrays& na,
                              ReactionArgs rx, int* status, hipStream_t s)
{
  launch_work(work, work.count, ta, X, na, nullptr, nullptr, rx, status, s);
}

__global__ __launch_bounds__(256) void k_slot_partials(TileArgs ta, int num_slots, int2* __restrict__ out)
{
  const int s = (int)(blockIdx.x * 256 + threadIdx.x);
  if (s >= num_slots) return;
  int2 r = make_int2(0, 0);
  if (ta.slot_dst[s] >= 0) {
    const int b = ta.nodes[s] - ta.bnd_base;
    r.x         = ta.bnd_ptr[b];
    r.y         = ta.bnd_ptr[b + 1] - r.x;
  }
  out[s] = r;
}

void launch_slot_partials(const TileArgs& ta, int num_slots, int2* out, hipStream_t s)
{
  if (num_slots <= 0) return;
  hipLaunchKernelGGL(k_slot_partials, dim3((unsigned)((num_slots + 255) / 256)), dim3(256), 0, s, ta, num_slots, out);
}

void launch_joint_element_tiled(const JointTileWork& work, const TileArgs& ta, const double* X, const NodeArrays& na,
                                float* Fip, float* sip, ReactionArgs rx, int* status, hipStream_t s)
{
  if (work.t_count <= 0) return;
  launch_grid<true>(work, work.reaction_groups + (unsigned)work.t_count, ta, X, na, Fip, sip, rx, status, s, LaunchTimer{});
}

void launch_uq_element_tiled(const UqTileWork& work, const TileArgs& ta, const double* X, const NodeArrays& na,
                             float* Fip, float* sip, ReactionArgs rx, int* status, hipStream_t s,
                             const LaunchTimer& timer)
{
  launch_work(work, work.count, ta, X, na, Fip, sip, rx, status, s, timer);
}

void launch_uq_nodes(const TileArgs& ta, const NodeArrays& na, const BcEntry* sample_bc, const UqClosure& uc,
                     int num_partials, const StepArgs& sa, ReactionArgs rx, hipStream_t s, const LaunchTimer& timer)
{
  const unsigned groups   = boundary_grid(ta.num_bnd);
  const unsigned interior = uc.num_approx > 0 ? boundary_grid(ta.bnd_base) : 0;
  if (groups + interior == 0) return complete_timer(timer, s);
  hipExtLaunchKernelGGL(k_uq_nodes, dim3(groups + interior), dim3(kBndThreads), 0, s, timer.start, timer.stop, 0, ta,
                        na, sample_bc, uc, num_partials, groups, sa, rx);
}

int element_tiled_groups_per_cu(int tile_elems)
{
  int n = 0;
  switch (tile_elems) {
    case 64:
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_element_tiled<64, true, false, ModelTileWork>, 64, 0);
      break;
    case 128:
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_element_tiled<128, true, false, ModelTileWork>, 128, 0);
      break;
    case 512:
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_element_tiled<512, true, false, ModelTileWork>, 512, 0);
      break;
    default:
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_element_tiled<256, true, false, ModelTileWork>, 256, 0);
  }
  return n;
}

void launch_boundary_update(const TileArgs& ta, const NodeArrays& na, const StepArgs& sa, ReactionArgs rx,
                            hipStream_t s, const LaunchTimer& timer)
{
  if (ta.num_bnd <= 0) return complete_timer(timer, s);
  hipExtLaunchKernelGGL(k_boundary_update, dim3(boundary_grid(ta.num_bnd)), dim3(kBndThreads), 0, s, timer.start,
                        timer.stop, 0, ta, na, sa, rx);
}

void launch_ens_boundary_update(const TileArgs& ta, const EnsNodes& en, const EnsRange* groups, int num_groups,
                                EnsStep es, ReactionArgs rx, int rx_base, hipStream_t s)
{
  if (num_groups <= 0) return;
  hipLaunchKernelGGL(k_ens_boundary_update, dim3((unsigned)num_groups), dim3(kBndThreads), 0, s, ta, en, groups, es,
                     rx, rx_base);
}

}  // namespace nsm
