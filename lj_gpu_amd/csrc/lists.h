// lists.h — neighbour lists on the device: the Verlet-list build from device
// positions (cell list, the reference's exact pair set and CSR order) and
// every layout the force kernels evaluate, derived on the device from a CSR
// list (half-to-full expansion, row ordering, ELL, LDS tiles). HIP-only
// header, used by api.hip and lists.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

#include "ljgpu_internal.h"

namespace ljgpu {

// A device allocation that only grows: reserve() reallocates (after
// synchronising `stream`) when more bytes are needed, so repeated list
// builds of similar size reuse their buffers.
struct DevMem {
  void* p = nullptr;
  size_t bytes = 0;
  size_t limit = SIZE_MAX;  // most bytes to take (ljgpu_internal_limit)
  template <class T>
  T* as() const {
    return static_cast<T*>(p);
  }
};
int dev_reserve(DevMem& m, size_t bytes, hipStream_t stream);
void dev_release(DevMem& m);

// A CSR list on the device: number_of_partners[n], pointer[n + 1] (pointer[n]
// = e when rows are stored in order), sorted_list[e].
struct DevCSR {
  int32_t n = 0;
  int64_t e = 0;
  DevMem nop, ptr, list;
  // > 0: the rows are still in the pair search's slab (ListWork::tmp), row i
  // at i * slab_stride, and `list` is not filled (dev_copy_slab).
  int32_t slab_stride = 0;
};
void dev_release(DevCSR& c);

// LDS tiling of a row-ordered full list (the layout ListView describes).
// Blocks cover consecutive slots of a particle order: slot s holds particle
// member[s], whose row occupies local[slot_ptr[s] .. slot_ptr[s+1]). In
// index order (member[s] = s) neither array is kept: the list's own
// pointer serves as slot_ptr.
struct DevTiles {
  int32_t tile_particles = 0;  // particles per block (0: no tiling)
  int32_t blocks = 0;
  int64_t staged = 0;
  int32_t max_stage = 0;
  int32_t lds_bytes = 0;
  int order = 0;               // LJGPU_TILE_ORDER_INDEX (member[s] = s) or _SPATIAL
  int32_t stage_stride = 0;    // >0: block b stages at b * stage_stride (one-pass build);
                               // 0: staging areas packed back to back
  DevMem desc, stage, local;
  DevMem member;      // int32 per slot
  DevMem slot_ptr;    // int32 per slot (+1)
  DevMem stage_slot;  // stage as slots (spatial order only)
  // Each block's staged particles are sorted by slot (by index in index
  // order), and local holds 24 * the rank of each entry's partner among them.

  // The same offsets sliced per wavefront for the streamed tile kernel of
  // sliced_lanes lanes per particle and sliced_unroll entries per lane per
  // batch (see dev_slice_tiles); sliced_lanes = 0: not built.
  DevMem sliced;      // uint16
  DevMem wave_off;    // int32 per (block, wavefront slot): start of its slice
  int32_t sliced_lanes = 0, sliced_unroll = 0, waves_per_block = 0;
  int64_t slice_elems = 0;  // entries that `sliced` has room for

  // Cutoff classes (cut): the rows of local hold their inner entries first,
  // inner[s] of them in slot s's row.
  bool cut = false;
  DevMem inner;          // int32 per slot
  // The rows in the bank-class order, and slices of them for bank_lanes and
  // bank_unroll (0: none), made on first use (dev_bank_rows, dev_bank_slices)
  // in ListWork::tmp: local itself keeps its order.
  bool bank_rows = false;
  int32_t bank_lanes = 0, bank_unroll = 0;
  int32_t longest = 0;   // longest row

  // Half lists (dev_half_tiles): see ListView. half_ready: all four belong to
  // this tiling.
  DevMem half_tile, half_first, half_at, half_part;
  bool half_ready = false;
  bool shared = false;  // half lists: dev_make_tiles found partners shared
};
void dev_release(DevTiles& t);

// Results of enqueued kernels, in pinned memory that they write: valid once
// the stream has been synchronised after the kernel.
struct ScanStats {
  int64_t total;
  int32_t lo, hi;  // smallest and largest value scanned
};
struct ListResults {
  ScanStats scan;    // of dev_scan
  ScanStats cells;   // particles per cell
  ScanStats order;   // particles per bin of the spatial tile order
  int32_t tiles[8];  // k_tile_stats
};

// Scratch buffers reused across builds.
struct ListWork {
  DevMem scan_sums;   // a 16-byte record (sum, extrema) per scan tile
  DevMem small;       // a few int64 results (totals, flags, extrema)
  DevMem cell_count;  // int32 per cell (+1)
  DevMem cell_start;  // int32 per cell (+1)
  DevMem cell_slot;   // int32 per particle: rank within its cell / fill counters
  DevMem cell_of;     // int32 per particle: cell index
  DevMem cell_sorted; // int32 per particle, cell order: cell index
  DevMem cpos;        // double4 per particle, cell order: x, y, z, index
  DevMem counts;      // int32 per row (+1)
  DevMem tmp;         // int32 per list entry; between builds see DevTiles::bank_rows
  DevMem tile_ns;     // int32 per tile (+1)
  DevMem tile_soff;   // int32 per tile (+1)
  DevMem tile_stats;  // int4 per tile
  DevMem tile_geo;    // int32 x 4 per tile: first particle, count, replica
  DevMem rep_of;      // int32 per particle: replica index
  DevMem order;       // int32 per particle: spatial tile order
  DevMem order_grid;  // OrderGrid per system
  DevMem slot_of;     // int32 per particle: its slot in the tile order
  DevCSR part;        // one replica's list during a batched build
  int32_t last_max_row = 0;  // longest row of the last device build (slab size hint)
  int32_t row_min = 0, row_max = 0;  // row lengths of the last device build
  ListResults* results = nullptr;    // pinned
  std::vector<int32_t> geo_host;     // blocks of a replicas' tiling, as uploaded
  std::vector<char> order_host;      // bins and offsets of a replicas' tile order, as uploaded
  std::vector<char> order_job;       // a tile order left for dev_makepair (else empty)
};
void dev_release(ListWork& w);

// Positions as three strided arrays (AoS: q, q+1, q+2 with stride 4; SoA:
// three arrays with stride 1).
struct PosIn {
  const double* x = nullptr;
  const double* y = nullptr;
  const double* z = nullptr;
  int stride = 4;
};

// Exclusive scan of in[0..n) into out[0..n], out[n] = total, both 16-byte
// aligned; *total receives the sum (synchronises the stream).
int dev_scan(hipStream_t s, const int32_t* in, int32_t* out, int64_t n, ListWork& w,
             int64_t* total);

// Strict check of a CSR list on the device (the rules of validate_csr);
// returns LJGPU_OK or LJGPU_ERR_BAD_LIST naming the first bad row.
int dev_validate(hipStream_t s, int32_t n, const int32_t* nop, const int32_t* ptr,
                 const int32_t* list, int64_t e, int kind, ListWork& w);

// Copy a caller's device CSR into `out` with rows stored in order.
int dev_copy_row_ordered(hipStream_t s, int32_t n, const int32_t* nop, const int32_t* ptr,
                         const int32_t* list, int64_t e, ListWork& w, DevCSR& out);

// Full list from a half list (both on the device): row i holds its lower
// partners ascending, then its own half row as stored.
int dev_expand_half(hipStream_t s, int32_t n, const int32_t* nop, const int32_t* ptr,
                    const int32_t* list, ListWork& w, DevCSR& full);

// Verlet list of `kind` from device positions: pair predicate
// r2 = (dx*dx + dy*dy) + dz*dz < search^2, unfused, minimum image for
// box > 0; rows ascending in i. With sort_rows, partners ascending (the
// reference's order); without, each row's partners come in an order fixed
// by the positions (stencil runs, cells, particle index within a cell), the
// same on every build from the same positions, and usually stay in the
// search's slab (out.slab_stride).
int dev_makepair(hipStream_t s, const PosIn& q, int32_t n, double box, double search_length,
                 int kind, ListWork& w, DevCSR& out, bool sort_rows = true);

// The rows of a list that is still in the slab, copied to its `list`.
int dev_copy_slab(hipStream_t s, ListWork& w, DevCSR& c);

// Smallest and largest of a[0..n) (synchronises); 0, 0 for n = 0.
int dev_minmax(hipStream_t s, const int32_t* a, int32_t n, ListWork& w, int32_t* mn, int32_t* mx);
// Row lengths of the half list contained in a full list with ascending rows
// (partners j > i), as min/max (synchronises).
int dev_half_row_stats(hipStream_t s, const DevCSR& full, ListWork& w, int32_t* min_np,
                       int32_t* max_np);

// ELL ("transposed") copy, entry k of row i at ell[i + k*n], width = longest
// row (at least 1), zero padded.
int dev_make_ell(hipStream_t s, const DevCSR& c, int32_t width, DevMem& ell);

// The slots of the spatial order in w.order (dev_tile_order): within each
// block of tile_particles consecutive slots (restarted at every replica
// boundary) the particles by row length, longest first, ties in the order
// given. Sets out.member, out.slot_ptr and w.slot_of.
int dev_tile_slots(hipStream_t s, const DevCSR& c, int32_t tile_particles,
                   const std::vector<int32_t>& replicas, ListWork& w, DevTiles& out);

// LDS tiling of a row-ordered full list with blocks of `tile_particles`
// consecutive particles, restarted at each replica boundary of `replicas`
// (host offsets; empty for a single system), descriptor slot 6 holding the
// block's replica. Returns LJGPU_OK with out.tile_particles = 0 when a block
// does not fit the LDS budget (the caller then halves the tile size or
// evaluates untiled). With `spatial` the blocks cover the slots of
// dev_tile_slots, else particles in index order. With `slices` (rows in list
// order, the longest known) the wavefront slices are made in the same pass
// where they can be (sliced_lanes > 0 afterwards), and local is then written
// only if wanted. A half list's (`half`) tiles write a force sum per staged
// partner: where partners are hardly shared (scattered particles of an open
// box) those are nearly as many as the pairs, and out.shared is false, with no
// tiles. The first pass over the list tells, by more than half as many staged
// partners as entries or by an eighth of the tiles with partners all over the
// list (in smaller systems every tile's fit). Install of a scattered half list of
// 62,500 particles (density 0.8) from the device: 175 us, 161 without the pass;
// with the sets of such tiles made, size after size, before they were dropped it
// took 4546, at 256,000 particles 23 ms.
struct SliceReq {
  int32_t lanes, unroll;
  int32_t longest;  // longest row
  bool local;
};
int dev_make_tiles(hipStream_t s, const DevCSR& c, int32_t tile_particles,
                   const std::vector<int32_t>& replicas, bool spatial, bool half,
                   const SliceReq* slices, ListWork& w, DevTiles& out);

// The tiles' entry offsets sliced per wavefront, for a tile kernel in
// which `lanes` consecutive lanes own one row and take entries in batches
// of lanes * unroll (entry k of a row: batch k / (lanes * unroll), slot
// (k / lanes) % unroll, lane k % lanes). Wavefront w of block b holds the
// block's rows [w * 64/lanes, (w+1) * 64/lanes) and owns the slice that
// starts at wave_off[b * waves_per_block + w]: for each of its batches
// (as many as its longest row needs) 64 * unroll offsets (scale * rank, scale
// the bytes per staged partner), slot by slot,
// each slot the 64 lanes' entries in lane order, so one offset load of the
// kernel reads 64 consecutive values. Slots past a row's end hold 0.
// Needs local, desc and the slot row starts of a built tiling of n particles; a slicing
// whose total does not fit int32 is not built (sliced_lanes stays 0). With
// bank_order, the rows of local first take the cutoff classes
// (cut_partition) of the positions in `cut`, if it has any and they have
// none yet, and the places of a row (its inner ones, then the others) are given out so
// that the lanes that read LDS together mostly read different banks
// (order_part). Without it places follow local.
struct CutHint {
  PosIn q;                        // positions in the caller's particle order
  double box = 0.0;               // single system: periodic box (<= 0 open)
  const double* rep_box = nullptr;  // replicas: (box, 1/box) per replica on the device
  double cl2 = 9.0;
};
int dev_slice_tiles(hipStream_t s, const int32_t* slot_ptr, int32_t lanes, int32_t unroll,
                    int32_t scale, bool bank_order, int32_t n, const CutHint* cut, ListWork& w,
                    DevTiles& t);

// What the tiled half-list kernel needs beyond a tiling of n particles: where
// each tile writes its staged partners' force sums, and which of them belong
// to each slot (in ascending order).
int dev_half_tiles(hipStream_t s, int32_t n, ListWork& w, DevTiles& t);

// The bank-class order (bank_class_order) of a tiling's rows, e entries, for what
// reads rows rather than slices; and slices of those rows, cut as the tiling's
// (t.sliced), for sums that depend on the order. Nothing where they are made
// already. Enqueued only, and without allocating after dev_bank_reserve, which
// leaves them without room where there is none.
int dev_bank_rows(hipStream_t s, const int32_t* slot_ptr, int64_t e, ListWork& w, DevTiles& t);
int dev_bank_slices(hipStream_t s, const int32_t* slot_ptr, int64_t e, ListWork& w, DevTiles& t);
int dev_bank_reserve(hipStream_t s, int64_t e, ListWork& w, DevTiles& t);
const uint16_t* bank_rows(const ListWork& w);
const uint16_t* bank_slices(const ListWork& w, int64_t e);

// Spatial particle order for LDS tiles, into w.order: each periodic system
// (the whole set, or every replica of `replicas` with its box) is cut into
// columns along x about 0.75 * cbrt(tile_particles / density) wide in y and
// z, each column into x bins of about one particle; particles are ordered by
// (system, z column, y column, x bin, index). Consecutive slots then hold
// compact groups of particles, so a block of them stages fewer partners than
// a block of consecutive indices. *ok = false (and no order) for an open box,
// non-finite positions or a bin of more than 256 particles.
int dev_tile_order(hipStream_t s, const PosIn& q, int32_t n, double box,
                   const std::vector<int32_t>& replicas, const std::vector<double>& boxes,
                   int32_t tile_particles, ListWork& w, bool* ok);
// The same in two steps, so that a caller's next synchronisation serves it
// too: begin enqueues it (*begun = false: no order for this box), end tells
// after that synchronisation whether the order holds. With `defer` a few
// particles' order is left in w.order_job for the dev_makepair that follows,
// which runs it beside its own binning.
int dev_tile_order_begin(hipStream_t s, const PosIn& q, int32_t n, double box,
                         const std::vector<int32_t>& replicas, const std::vector<double>& boxes,
                         int32_t tile_particles, ListWork& w, bool* begun, bool defer = false);
bool dev_tile_order_end(const ListWork& w);

// Batched replicas: lists of every replica (particles [off[r], off[r+1]),
// box boxes[r]) built on the device into one CSR with global indices.
int dev_makepair_batch(hipStream_t s, const PosIn& q, const std::vector<int32_t>& off,
                       const std::vector<double>& boxes, double search_length, int kind,
                       ListWork& w, DevCSR& out);

// LJGPU_ERR_BAD_LIST unless every entry of row i lies in i's replica.
int dev_check_replicas(hipStream_t s, const DevCSR& c, const std::vector<int32_t>& off,
                       ListWork& w);

}  // namespace ljgpu
