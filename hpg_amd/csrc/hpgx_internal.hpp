// Internal declarations shared by the C ABI (hpgx_api.cpp) and the HIP
// kernels (hpgx_kernels.hip).  Not installed; the public interface is
// include/hpgx.h.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace hpgx {

// CFArray::padding (src/hpg.hpp:655)
constexpr int cf_padding = 2;
// maximum number of CF groups (HPG_MAX_NUM_CF_GROUPS, src/CMakeLists.txt:37)
constexpr int max_cf_groups = 1000;
// grid tile edge (pixels) owned by one workgroup of the gridding kernel
constexpr int tile = 32;

// Per-group geometry of the device CF.  The device layout of group g is
// "fine-offset sliced": for every (cube, fx, fy) -- fx, fy in [-F, F] the
// visibility's fine offset on each axis, F = (os + 1) / 2 -- the sx x sy
// taps of the support are contiguous, x fastest, each with its Mueller
// elements side by side (a record reads all of them, so whole lines of its
// slice, wherever a tile border cuts the support):
//   taps[tap_offset + ((((cube * nf + fx + F) * nf + fy + F) * sx * sy
//        + Y * sx + X) * nmueller + k]
//   = CFArray(ix, iy, elem[k], cube, g), ix = (X + padding) * os + fx, iy
// likewise, which is the element the reference reaches through its 6-D layout
// (src/hpg_impl.hpp:221-281, src/hpg_core.hpp:422-446: major * os + minor).
// wsum[wsum_offset + ((cube * nmueller + k) * nf + fx + F) * nf + fy + F]
// is the FP64 sum of that element's taps of the slice.
// Planar (one polarization, supports that the tile kernels take: a record reads
// one element for a grid row): the slice's elements one after the other instead,
//   ... * nf + fy + F) * nmueller + k) * sx * sy + Y * sx + X]
// (one polarization in four grid rows of an element each, 500,000 records,
// supports of 15, FP64: 896 us side by side, 678 so; predicted 1034, 606).
// Only elements that some Mueller row names are held (CfElements, ascending;
// the rows that the kernels see count in them): a tap's neighbours in memory
// are then values that the calls read.  One polarization on a CF of 16 elements,
// 1e6 records, supports of 7: 320 us with all 16 side by side, 134 with the one.
struct GroupInfo {
  long long tap_offset;
  long long wsum_offset;
  int sx, sy;          // support 2r + 1 per axis
  int rx, ry;          // radii (src/hpg.hpp:687-694)
  int nmueller, ncube;  // held elements (the first so many of CfElements)
};

// the Mueller elements held, ascending; -1: none of the CFArray's, all zero,
// first and named by no row, where a group has none of those that rows name (so
// that every group has one: lanes without an element read it)
struct CfElements {
  int n;
  int elem[33];  // two matrices of 4 x 4, and the -1
};

struct Mueller {
  int M[4][4];   // mueller_indexes, padded with -1
  int Mc[4][4];  // conjugate_mueller_indexes, padded with -1
};

// grid / CF geometry passed by value to kernels
struct Geometry {
  int nx, ny, nr, nc;  // grid_size: x, y, mrow, cube
  double scale[2];     // grid_scale
  int os;              // CF oversampling
  int F;               // max |fine offset| = (os + 1) / 2
  int nf;              // 2F + 1
  int ngroups;
  int planar;          // the CF layout (GroupInfo)
  int ntx, nty;        // tiles per plane along x and y
};

// flags of a bin entry
constexpr unsigned short flag_pos_w = 1;
constexpr unsigned short flag_gradient = 4;

enum class GvisSource { Values, Adjoint };

// Device buffers for one gridding call (owned by the state).
struct CallBuffers {
  void* vis;            // raw VisData<N> records
  float2* gvis;         // per visibility x N
  unsigned* hist;       // per (plane, tile) key, nkeys + 1
  unsigned* offsets;    // exclusive scan of hist, nkeys + 1
  unsigned* cursor;     // scatter positions, nkeys
  size_t entries_capacity;  // entries of stream_entries
  void* scan_temp;
  size_t scan_temp_bytes;
  void* stream_entries;  // compact binned entries (Entry4), sorted by key
  unsigned* entry_vis;   // record index of entries with a phase gradient
  unsigned* off_table;   // block-local bins: per bin block, nkeys + 1 offsets
  size_t off_table_capacity;
  double2* halo;         // haloed tiles: per key, the halo's FP64 values
  unsigned* halo_set;    // per key: 1 if its halo was written by this pass
  size_t halo_capacity;  // elements of halo
  size_t halo_set_capacity;
  unsigned long long* invalid_count;
  double2* degrid_acc;   // binned degridding: per record x polarization sums
  size_t degrid_acc_capacity;
  void* tally_entries;   // launch_tally: entries in record order (Entry4)
  void* tally_keys;      // and per slot its key and a (lower key bits, slot) pair
  size_t tally_capacity; // slots of both
  unsigned* sort_bins;   // launch_tally, launch_degrid: the sort's counts, offsets
  size_t sort_capacity;  // and places, for this many records (sort_bins_entries)
  void* patch_recs;       // launch_patch: prepared records (PatchRec<N>)
  size_t patch_capacity;
  unsigned* patch_list;   // and the tiles' lists of record indexes
  size_t patch_list_capacity;
  unsigned* patch_table;  // and the workgroups' places in them (few tiles)
  size_t patch_table_capacity;
  void* patch_split;      // and the chunks of split lists: their sums and slots
  size_t patch_split_slots;
  unsigned* degrid_order; // launch_degrid: keys, the record order, (key, record)
                          // pairs, 4 order_capacity values
  void* degrid_recs;      // and its prepared records (DegridRec)
  size_t order_capacity;
};

struct DeviceCF {
  GroupInfo* groups;  // device array
  float2* taps;
  double2* wsum;
  int os, F, nf, ngroups;
  int max_sx, max_sy;
  int max_ncube;  // CF cubes of the group with the most
  int min_nm;     // Mueller elements of the group with the fewest
  bool even_nm;   // every group has an even number of them
  bool planar;    // the layout (GroupInfo)
};

// ---- launchers (hpgx_kernels.hip) -------------------------------------

hipError_t launch_cf_relayout(
  hipStream_t s, const float2* staging, const unsigned ext[4],
  const GroupInfo& gi, const CfElements& ce, int os, int F, int nf, bool planar,
  float2* taps);
hipError_t launch_cf_wsum(
  hipStream_t s, const GroupInfo& gi, int nf, bool planar, const float2* taps,
  double2* wsum);

// exclusive scan of the global bin counts (hist -> offsets, cursor)
hipError_t launch_scan(hipStream_t s, size_t nkeys, CallBuffers& cb);
size_t scan_temp_bytes(size_t nkeys);
// global bins: one Entry4 per record and plane in the bin of the tile holding the
// support corner (for launch_tile_halo with global_bins)
hipError_t launch_count(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool do_grid, CallBuffers& cb,
  double* weights);
hipError_t launch_emit(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool gvis_ready, GvisSource src, const double2* residuals,
  CallBuffers& cb);
// the whole gridding pass of a few records in one launch, on no buffers of cb
// but vis, gvis and invalid_count
bool direct_ok(size_t n, const Geometry& geo);
hipError_t launch_direct(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf, const Mueller& mu,
  bool update_weights, bool gvis_ready, GvisSource src, const double2* residuals,
  const CallBuffers& cb, double* weights, double2* grid);
// global quadrant bins (one polarization, haloed entries): the entries in their
// keys' order in cb.stream_entries, the keys' offsets in cb.offsets; n x nr slots
// of cb.tally_entries / cb.tally_keys
hipError_t launch_tally(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, double* weights);
// block-local binning (small key counts)
int bin_blocks_for(size_t n);
size_t bin_block_records();
int bin_keys_limit();
int bin_quad_keys_limit();  // with quad_keys: 4 x (plane, tile) keys
int tile_bins_limit();
hipError_t launch_bin(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, size_t block_cap, double* weights,
  bool degrid_pass = false, void* copy_records = nullptr,
  bool quad_keys = false);
// haloed tiles (one entry per record and plane; supports below tile)
size_t halo_entry_bytes();
size_t halo_pixels_per_key(int hx, int hy);
int halo_tile_limit();
size_t halo_lds_bytes(int hx, int hy, int nbins);
// acc (FP32 grids): 0 FP64 tile sums, else FP32 two-sum of (hi, lo) pairs under
// compare-and-swap
hipError_t launch_tile_halo(
  hipStream_t s, int npol, int mode, int acc, size_t n, size_t nkeys, const Geometry& geo,
  const DeviceCF& cf, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, void* grid, bool global_bins = false);
// the quadrant-key kernel (k_sub): FP32-compensated grids, supports of at
// most 8 x 8 (hx, hy <= 7), bins of launch_bin with quad_keys; ntile_keys
// (plane, tile) keys, whose offset-table rows hold 4 ntile_keys + 1 values;
// CF taps of at most 2^32 - 1 bytes
int sub_bins_limit();
bool sub_supported(int hx, int hy);
// uni: every CF group has the same support; global_bins (one polarization):
// the entries of launch_tally, cb.offsets their key offsets
hipError_t launch_tile_sub(
  hipStream_t s, int npol, size_t n, size_t ntile_keys, const Geometry& geo, const DeviceCF& cf,
  size_t taps_bytes, bool uni, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, void* grid, bool global_bins = false);
// register patches (k_patch): any number of polarizations and grid rows, any
// support and grid.  cb.hist and cb.offsets hold patch_keys + 1 values,
// cb.patch_recs patch_capacity records and cb.patch_list
// patch_tiles_per_footprint indexes for each
size_t patch_keys(const Geometry& geo);
size_t patch_rec_bytes(int npol);
// values of cb.patch_table for n records a call (0 for many tiles)
size_t patch_table_entries(const Geometry& geo, size_t n);
// slots of cb.patch_split for lists of so many entries in all, at most
// patch_slots_max, and the bytes they take
constexpr size_t patch_slots_max = 2048;
size_t patch_split_slots(size_t entries);
size_t patch_split_bytes(size_t slots);
size_t patch_tiles_per_footprint(int nr, int max_sx, int max_sy);
// the rows of a slice that one wave's pixels take have 32-bit byte offsets (not
// so from 2^32 bytes in 16 rows on: CFs of 38 GB at the least)
bool patch_offsets_fit(const GroupInfo& g);
hipError_t launch_patch(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, double* weights, int mode, bool halo_rounds, void* grid);
// binned degridding from the model's LDS tiles (entries of launch_bin with
// degrid_pass).  one_plane (every record has exactly one entry): the
// predictions are finished in the same kernel -- FP64 values to pred64, or
// values written into out_recs (residuals, and gvis in cb, when do_grid).
// Otherwise per-record sums are added into acc (zeroed beforehand) for
// launch_degrid_finish.
hipError_t launch_degrid_tiles(
  hipStream_t s, int npol, size_t n, size_t nkeys, const Geometry& geo,
  const DeviceCF& cf, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, const double2* model, double2* acc, bool one_plane, bool do_grid,
  void* out_recs, double2* pred64);
// predictions from those sums for the records at `records`: FP64 values
// to pred64, or values written into out_records when not null (residuals,
// and gvis in cb, when do_grid)
hipError_t launch_degrid_finish(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, const double2* acc, bool do_grid, const void* records,
  void* out_records, CallBuffers& cb, double2* pred64);
// slice-ordered degridding of the records at `records`: FP64 predictions to
// pred64, or predicted values (residuals, and gvis in cb, when do_grid)
// written into out_records when not null, which may be `records`.  With a
// model, cb.degrid_order, sort_bins, degrid_recs and degrid_acc hold at least n
// records.
size_t degrid_rec_bytes();
size_t sort_bins_entries(size_t n);
hipError_t launch_degrid(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, const double2* model, bool do_grid, CallBuffers& cb, double2* pred64,
  const void* records, void* out_records);

hipError_t launch_normalize(
  hipStream_t s, int mode, void* grid, const double* weights, double wfactor,
  const Geometry& geo);
hipError_t launch_scale(
  hipStream_t s, int mode, void* grid, double inv_norm, size_t count);
// the deferred finishing chain's pass before its FFT: divided by wfactor *
// the plane's weight (weights not null), times scale, and with modulate
// multiplied by (-1)^(x + y); for grids with finish_pre_fits (rows and
// planes within a launch's y and z extents)
bool finish_pre_fits(const Geometry& geo);
hipError_t launch_finish_pre(
  hipStream_t s, int mode, void* grid, const double* weights, double wfactor, double scale,
  bool modulate, const Geometry& geo);
hipError_t launch_shift(
  hipStream_t s, int mode, void* grid, void* scratch, int direction,
  const Geometry& geo);
hipError_t launch_widen(hipStream_t s, const float2* src, double2* dst, size_t count);
hipError_t launch_narrow(hipStream_t s, const double2* src, float2* dst, size_t count);

}  // namespace hpgx
