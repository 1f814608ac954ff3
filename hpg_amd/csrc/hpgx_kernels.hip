// HIP kernels of the MI355X gridding device (gfx950, wave64).
//
// Build with -ffp-contract=off: a product or sum is fused only where the code
// says so.  FP64 grids without phase gradients hold the reference's per-tap FP32
// values bit for bit, and differ from it only by the order of FP64 accumulation.
// Fused by intent: the FP32 products of k_sub (FP32 grids), the FP64 products of
// k_degrid, and cphase_taylor's reduction and series.
//
// Gridding (VisibilityGridder::kernel, src/hpg_core.hpp:1082-1253) is
// re-organized for the device in two stages: binning, then one workgroup per
// grid tile accumulating it on chip and adding it into the grid with one
// coalesced read-modify-write, so that no global atomic touches the grid.
//   k_bin + k_sub / k_tile4 + k_halo   one polarization, supports narrower
//        than a tile: records binned by the 32 x 32 tile holding their support
//        corner (block-local bins, no global atomics; grids of more than 8192
//        keys bin through global memory: k_tally + k_tally_sort, k_count +
//        k_emit); the tile kernels accumulate the tile plus a halo of
//        (support - 1) pixels in LDS, and k_halo folds each tile's halo into
//        its neighbours.
//   k_direct   the same records, FP64 grids, where they are few: one launch.
//   k_patch_prep + k_patch_list + k_patch   several polarizations, larger
//        supports: each tile's sums of all its grid rows in registers.
// Degridding (degrid_vis, src/hpg_core.hpp:579-682): k_degrid4 reads the
// model's tile and halo from LDS for binned records (one polarization, small
// supports); k_degrid takes the records in CF-slice order, several sharing
// the CF values that a wave loads.

#include "hpgx_internal.hpp"

#include <hipcub/hipcub.hpp>

#include <cmath>
#include <type_traits>

namespace hpgx {
namespace {

constexpr double c_light = 299792458.0;  // src/hpg_core.hpp:527
constexpr int wave = 64;
constexpr int block = 256;

// hpg::VisData<N> as seen by the device (src/hpg.hpp:236-311)
template <int N>
struct VisRec {
  float2 vis[N];
  float w[N];
  double freq;
  double phase;
  double uvw[3];
  unsigned grid_cube;
  unsigned cf_index[2];  // {cube, grp}
  double grad[2];
};
static_assert(sizeof(VisRec<1>) == 88, "VisData<1>");
static_assert(sizeof(VisRec<2>) == 96, "VisData<2>");
static_assert(sizeof(VisRec<3>) == 112, "VisData<3>");
static_assert(sizeof(VisRec<4>) == 120, "VisData<4>");

typedef int v2i_t __attribute__((ext_vector_type(2)));
typedef int v4i_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// complex<float> * complex<double> -> complex<double> (Kokkos mixed product)
__device__ __forceinline__ double2 cmul(float2 a, double2 b) {
  return make_double2(
    double(a.x) * b.x - double(a.y) * b.y, double(a.x) * b.y + double(a.y) * b.x);
}
// Kokkos 4.x complex division: scale by the divisor's 1-norm
__device__ __forceinline__ double2 kdiv(double2 x, double2 y) {
  const double s = fabs(y.x) + fabs(y.y);
  if (s == 0.0) return make_double2(x.x / s, x.y / s);
  const double2 xs = make_double2(x.x / s, x.y / s);
  const double2 ycs = make_double2(y.x / s, -y.y / s);
  const double yabs = ycs.x * ycs.x + ycs.y * ycs.y;
  double2 r = cmul(xs, ycs);
  r.x /= yabs;
  r.y /= yabs;
  return r;
}
__device__ __forceinline__ double2 cphase(double ph) {
  double s, c;
  sincos(ph, &s, &c);
  return make_double2(c, s);
}
__device__ __forceinline__ float2 narrow(double2 a) {
  return make_float2(float(a.x), float(a.y));
}
// gvis = fl32(vis * phasor * weight) (src/hpg_core.hpp:1172-1182)
__device__ __forceinline__ float2 prephase(float2 v, double2 phasor, float w) {
  const double2 t = cmul(v, phasor);
  return make_float2(float(t.x * double(w)), float(t.y * double(w)));
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int m = wave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, wave);
  return v;
}

// q / d for 0 <= q < 2^32 / d, with m = magic(d) (exact in that range)
__device__ __forceinline__ unsigned magic(unsigned d) {
  return d == 1u ? 0u : 0xFFFFFFFFu / d + 1u;
}
__device__ __forceinline__ unsigned div_magic(unsigned q, unsigned d, unsigned m) {
  return d == 1u ? q : __umulhi(q, m);
}

__device__ __forceinline__ int uniform(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}

// compute_vis_coord + Vis<N> ctor + all_within_grid
// (src/hpg_core.hpp:422-446, 493-550, 1070-1080)
struct Coord {
  int gx, gy;    // grid coordinate of the support corner
  int fx, fy;    // fine offsets
  bool inside;
};

__device__ __forceinline__ bool axis_coord(
  int g_size, int os, int radius, int support, double coord, double inv_lambda,
  double scale, int& corner, int& fine) {
  corner = 0;
  fine = 0;
  const double position = scale * coord * inv_lambda + g_size / 2.0;
  if (!(fabs(position) < 1.0e9)) return false;
  const double G = rint(position);
  fine = int(rint((G - position) * os));
  corner = int(G) - radius;
  return 0 <= corner && corner + support <= g_size;
}

template <int N>
__device__ __forceinline__ Coord vis_coord(
  const VisRec<N>& r, const Geometry& geo, const GroupInfo& g) {
  Coord c;
  const double inv_lambda = r.freq / c_light;
  const bool ix = axis_coord(
    geo.nx, geo.os, g.rx, g.sx, r.uvw[0], inv_lambda, geo.scale[0], c.gx, c.fx);
  const bool iy = axis_coord(
    geo.ny, geo.os, g.ry, g.sy, r.uvw[1], inv_lambda, geo.scale[1], c.gy, c.fy);
  c.inside = ix && iy;
  return c;
}

__device__ __forceinline__ int tiles_begin(int corner) { return corner / tile; }
__device__ __forceinline__ bool row_has_index(const int* row, int npol) {
  bool any = false;
  for (int v = 0; v < npol; ++v) any |= row[v] >= 0;
  return any;
}

// W_v = sum over grid rows of the degridding CF slice sums
// (degrid_vis weights, src/hpg_core.hpp:643-668): with the im factor applied
// to every tap, the sum is T[m] (w > 0) or conj(T[m]) (w <= 0).
template <int N>
__device__ __forceinline__ void degrid_norms(
  const Geometry& geo, const GroupInfo& g, const double2* wsum,
  const Mueller& mu, bool pos_w, unsigned cfcube, int fxi, int fyi,
  double2* W) {
  for (int v = 0; v < N; ++v) W[v] = make_double2(0.0, 0.0);
  for (int gpol = 0; gpol < geo.nr; ++gpol) {
    const int* row = pos_w ? mu.Mc[gpol] : mu.M[gpol];
    for (int v = 0; v < N; ++v) {
      const int m = row[v];
      if (m >= 0 && m < g.nmueller) {
        const double2 t = wsum[g.wsum_offset
                               + ((long long)(cfcube * g.nmueller + m) * geo.nf + fxi)
                                 * geo.nf + fyi];
        W[v].x += t.x;
        W[v].y += pos_w ? t.y : -t.y;
      }
    }
  }
}

// index of the first value of the CF slice (cube, fx, fy); its Mueller
// element m follows at m, tap t at t * g.nmueller, or (planar) at m * ntap, t
__device__ __forceinline__ long long slice_start(
  const GroupInfo& g, int nf, int cube, int fxi, int fyi) {
  const long long slice = ((long long)cube * nf + fxi) * nf + fyi;
  return g.tap_offset + slice * ((long long)g.sx * g.sy * g.nmueller);
}
// of its element m in the planar form
__device__ __forceinline__ long long plane_start(
  const GroupInfo& g, int nf, int cube, int m, int fxi, int fyi) {
  const long long slice = ((long long)cube * nf + fxi) * nf + fyi;
  return g.tap_offset + (slice * g.nmueller + m) * ((long long)g.sx * g.sy);
}

// ---- CF ingestion ----------------------------------------------------

__global__ void k_cf_relayout(
  const float2* __restrict__ staging, unsigned ex, unsigned ey, unsigned em, GroupInfo gi,
  CfElements ce, int os, int F, int nf, int planar, float2* __restrict__ taps, long long total,
  long long block0) {
  const long long o = (block0 + blockIdx.x) * (long long)blockDim.x + threadIdx.x;
  if (o >= total) return;
  long long q = o;
  int k = 0;
  if (!planar) {
    k = int(q % gi.nmueller);
    q /= gi.nmueller;
  }
  const int X = int(q % gi.sx);
  q /= gi.sx;
  const int Y = int(q % gi.sy);
  q /= gi.sy;
  if (planar) {
    k = int(q % gi.nmueller);
    q /= gi.nmueller;
  }
  const int m = ce.elem[k];
  const int fyi = int(q % nf);
  q /= nf;
  const int fxi = int(q % nf);
  const int c = int(q / nf);
  const long long ix = (long long)(X + cf_padding) * os + (fxi - F);
  const long long iy = (long long)(Y + cf_padding) * os + (fyi - F);
  float2 v = make_float2(0.0f, 0.0f);
  if (m >= 0 && ix >= 0 && iy >= 0 && ix < ex && iy < ey)
    v = staging[(((long long)c * em + m) * ey + iy) * ex + ix];
  taps[gi.tap_offset + o] = v;
}

// the same through LDS: one workgroup per cube, support row, fine y offset and
// xc support columns reads the columns' values of every Mueller element (runs
// of (xc - 1) os + nf values) and writes each fine x offset's taps (runs of
// xc nmueller values).  k_cf_relayout reads one value of each line at a time:
// 221 us a group of 64 with 16 elements and supports of 9 to 65 at oversampling
// 20, on average, against 58 us here.
constexpr int relayout_block = 256;
constexpr size_t relayout_lds = 40960;
__global__ __launch_bounds__(relayout_block) void k_cf_relayout_lds(
  const float2* __restrict__ staging, unsigned ex, unsigned ey, unsigned em, GroupInfo gi,
  CfElements ce, int os, int F, int nf, int planar, float2* __restrict__ taps, int xc, int nxc,
  long long block0) {
  extern __shared__ float2 win[];
  unsigned long long b = (unsigned long long)(block0 + blockIdx.x);
  const int X0 = int(b % unsigned(nxc)) * xc;
  b /= unsigned(nxc);
  const int Y = int(b % unsigned(gi.sy));
  b /= unsigned(gi.sy);
  const int fyi = int(b % unsigned(nf));
  const int c = int(b / unsigned(nf));
  const int nm = gi.nmueller;
  const int cols = min(xc, gi.sx - X0);
  const int width = (xc - 1) * os + nf;
  const long long ix0 = (long long)(X0 + cf_padding) * os - F;
  const long long iy = (long long)(Y + cf_padding) * os + (fyi - F);
  for (int m = 0; m < nm; ++m) {
    const int em_m = ce.elem[m];
    for (int k = threadIdx.x; k < width; k += relayout_block) {
      const long long ix = ix0 + k;
      float2 v = make_float2(0.0f, 0.0f);
      if (em_m >= 0 && ix >= 0 && iy >= 0 && ix < ex && iy < ey)
        v = staging[(((long long)c * em + em_m) * ey + iy) * ex + ix];
      win[m * width + k] = v;
    }
  }
  __syncthreads();
  const unsigned run = unsigned(cols) * unsigned(nm);
  for (unsigned k = threadIdx.x; k < run * unsigned(nf); k += relayout_block) {
    const int fxi = int(k / run);
    const unsigned t = k - unsigned(fxi) * run;
    const long long slice = ((long long)c * nf + fxi) * nf + fyi;
    int X, m;
    long long at;
    if (planar) {
      m = int(t / unsigned(cols));
      X = int(t) - m * cols;
      at = ((slice * nm + m) * gi.sy + Y) * gi.sx + X0 + X;
    } else {
      X = int(t / unsigned(nm));
      m = int(t - unsigned(X) * unsigned(nm));
      at = (slice * gi.sy + Y) * gi.sx * nm + (long long)X0 * nm + t;
    }
    taps[gi.tap_offset + at] = win[m * width + X * os + fxi];
  }
}

// the FP64 sum of each Mueller element's taps of each CF slice (the weights'
// normalization), one workgroup per slice (of 64 to 1024 threads by the
// slice's size: large supports have few slices): thread t sums the values t,
// t + threads, ... (coalesced reads), which with per = 2^k <= 64 elements all
// belong to element t mod per, then a fixed-order reduction.  Other numbers of
// elements, and planar slices (per = 0): one workgroup per slice and element.  FP64 sums of FP32
// taps: exact while the taps' exponents span fewer than about 29 bits, else
// within a few FP64 ulps of any other order
constexpr int wsum_block = 1024;
__global__ __launch_bounds__(wsum_block) void k_cf_wsum(
  GroupInfo gi, int nf, const float2* __restrict__ taps,
  double2* __restrict__ wsum, int per, int planar, long long block0) {
  __shared__ double2 part[wsum_block / wave][wave];
  const int nm = gi.nmueller;
  const long long ntap = (long long)gi.sx * gi.sy;
  const long long b = block0 + blockIdx.x;
  const long long slice = per ? b : b / nm;  // (cube * nf + fx) * nf + fy
  const int step = per || planar ? 1 : nm;
  const float2* t = taps + gi.tap_offset + slice * ntap * nm
    + (per ? 0 : (b % nm) * (planar ? ntap : 1));
  const int keep = per ? per : 1;  // elements of this workgroup
  double re = 0.0, im = 0.0;
  for (long long k = threadIdx.x; k < ntap * keep; k += blockDim.x) {
    const float2 c = t[k * step];
    re += double(c.x);
    im += double(c.y);
  }
  for (int d = wave / 2; d >= keep; d >>= 1) {
    re += __shfl_xor(re, d, wave);
    im += __shfl_xor(im, d, wave);
  }
  const int lane = int(threadIdx.x % wave);
  if (lane < keep) part[threadIdx.x / wave][lane] = make_double2(re, im);
  __syncthreads();
  if (int(threadIdx.x) >= keep) return;
  re = im = 0.0;
  for (int w = 0; w < int(blockDim.x) / wave; ++w) {
    re += part[w][threadIdx.x].x;
    im += part[w][threadIdx.x].y;
  }
  const int m = per ? int(threadIdx.x) : int(b % nm);
  const long long nslice = (long long)nf * nf;
  const long long c = slice / nslice;
  wsum[gi.wsum_offset + (c * nm + m) * nslice + (slice - c * nslice)] = make_double2(re, im);
}

// ---- gridding ----------------------------------------------------------

// s + e = a + b exactly, s = fl(a + b) (Knuth's two-sum)
__device__ __forceinline__ void two_sum(float a, float b, float& s, float& e) {
  s = a + b;
  const float bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

// An FP32-compensated tile pixel component is a pair (hi, lo) of floats
// packed into 64 bits (hi in the low word), updated as one unit by
// compare-and-swap where several lanes may add to it.
__device__ __forceinline__ unsigned long long pack_pair(float hi, float lo) {
  return (unsigned long long)__float_as_uint(hi)
    | ((unsigned long long)__float_as_uint(lo) << 32);
}

// the pair (hi, lo) after adding h to it: hi' = fl(hi + h), lo' = fl(lo + err)
// with err the exact rounding error of the first sum (two-sum)
__device__ __forceinline__ unsigned long long pair_plus(unsigned long long pair, float h) {
  const float hi = __uint_as_float(unsigned(pair));
  const float lo = __uint_as_float(unsigned(pair >> 32));
  float sum, err;
  two_sum(hi, h, sum, err);
  return pack_pair(sum, lo + err);
}

// compare-and-swap of the pair at a from `expect` to `desired`; on failure
// `expect` receives the value found
__device__ __forceinline__ bool pair_swap(
  unsigned long long* a, unsigned long long& expect, unsigned long long desired) {
  return __hip_atomic_compare_exchange_strong(
    a, &expect, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// retries until the update of the pair at a lands; every retry follows a
// successful update of the same pair by another lane or wave
__device__ __forceinline__ void pair_add(
  unsigned long long* a, unsigned long long expect, float h) {
  while (!pair_swap(a, expect, pair_plus(expect, h))) {
  }
}

// ---- gridding, global bins ---------------------------------------------------
//
// (and the kernels of the next two sections: one polarization)
// k_count   one thread per visibility: skip rule, weights, bin counts
// k_emit    one thread per visibility: writes one compact Entry4 per grid plane
//           -- support corner, fine offsets, CF group and cube, pre-phased
//           values -- into the bin of the tile holding the support corner, so
//           the tile kernel reads its bin as one contiguous stream instead of
//           gathering per-visibility records

// an entry under construction in k_bin
struct Entry {
  int gx, gy;
  unsigned fpk;  // fxi | fyi << 8 | flags << 16
  unsigned gpk;  // grp | cfcube << 16
  float2 g;
};

// entries of the haloed-tile pipeline (k_tile4): one per (record, plane),
// position relative to the tile that holds the support corner
struct Entry4Head {
  unsigned pos;  // lx | ly << 6 | fxi << 12 | fyi << 20 | flags << 28
  unsigned gpk;  // grp | cfcube << 16
};
struct Entry4 {
  Entry4Head h;
  float2 g;
};
constexpr unsigned e4_pos_w = 1u << 28;
constexpr unsigned e4_gradient = 1u << 29;
static_assert(sizeof(Entry4) == 16, "Entry4 layout");

// quadrant key of tile key k for a support corner (gx, gy): 4 k + the quadrant
// of the corner within its tile
__device__ __forceinline__ int quad_key(int k, int gx, int gy) {
  const int qx = (gx % tile) >= tile / 2 ? 1 : 0;
  const int qy = (gy % tile) >= tile / 2 ? 1 : 0;
  return 4 * k + (qx | (qy << 1));
}

// one entry per plane, in the bin of the tile holding the support corner
// Weights: each wave sums its records' weights per (grid cube, row), and
// for grids of at most count_planes_lds planes adds the sums into the
// workgroup's LDS, which adds into the grid weights once at its end (the
// workgroups stride over the records, so a few thousand global atomics per
// plane instead of one per wave).
constexpr int count_planes_lds = 64;
constexpr unsigned count_blocks_max = 2048;

__global__ __launch_bounds__(block) void k_count(
  const VisRec<1>* __restrict__ recs, size_t n, Geometry geo,
  const GroupInfo* __restrict__ groups, const double2* __restrict__ wsum,
  Mueller mu, int update_weights, int do_grid, unsigned* __restrict__ hist,
  double* __restrict__ weights, unsigned long long* __restrict__ invalid) {

  __shared__ double wblk[count_planes_lds];
  const int nplanes = geo.nr * geo.nc;
  const bool lds_w = update_weights && nplanes <= count_planes_lds;
  if (lds_w)
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x) wblk[k] = 0.0;
  __syncthreads();

  const size_t stride = size_t(gridDim.x) * blockDim.x;
  const size_t i0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  // every thread runs the same number of iterations (the wave reductions
  // below need all lanes)
  const size_t iters = (n + stride - 1) / stride;
  for (size_t it = 0; it < iters; ++it) {
    const size_t i = i0 + it * stride;
    bool counted = false;
    unsigned gcube = 0;
    double tw[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < n) {
      const VisRec<1>& r = recs[i];
      const unsigned grp = r.cf_index[1];
      const unsigned cfcube = r.cf_index[0];
      gcube = r.grid_cube;
      bool valid = grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc);
      if (valid) valid = cfcube < unsigned(groups[grp].ncube);
      if (!valid) {
        atomicAdd(invalid, 1ull);
      } else {
        const GroupInfo g = groups[grp];
        const Coord c = vis_coord(r, geo, g);
        const bool pos_w = r.uvw[2] > 0;
        if (c.inside && update_weights) {
          counted = true;
          const int fxi = c.fx + geo.F, fyi = c.fy + geo.F;
          for (int gpol = 0; gpol < geo.nr; ++gpol) {
            const int* row = pos_w ? mu.M[gpol] : mu.Mc[gpol];
            const int m = row[0];
            double mag = 0.0;
            if (m >= 0 && m < g.nmueller) {
              const double2 sw = wsum[g.wsum_offset
                                      + ((long long)(cfcube * g.nmueller + m) * geo.nf
                                         + fxi) * geo.nf + fyi];
              mag = hypot(sw.x, sw.y);
            }
            tw[gpol] = mag * double(r.w[0]);
          }
        }
        if (c.inside && do_grid) {
          const int ntiles = geo.ntx * geo.nty;
          const int t = tiles_begin(c.gy) * geo.ntx + tiles_begin(c.gx);
          for (int gpol = 0; gpol < geo.nr; ++gpol) {
            if (!row_has_index(pos_w ? mu.M[gpol] : mu.Mc[gpol], 1)) continue;
            const int base = int(gcube * geo.nr + gpol) * ntiles;
            atomicAdd(hist + base + t, 1u);
          }
        }
      }
    }
    if (update_weights) {
      unsigned long long active = __ballot(counted);
      const int lane = threadIdx.x % wave;
      while (active) {
        const int leader = __ffsll((long long)active) - 1;
        const unsigned cube = __shfl(gcube, leader, wave);
        const bool mine = counted && gcube == cube;
        active &= ~__ballot(mine);
        for (int gpol = 0; gpol < geo.nr; ++gpol) {
          const double sw = wave_sum(mine ? tw[gpol] : 0.0);
          if (lane == leader) {
            const size_t k = size_t(cube) * geo.nr + gpol;
            if (lds_w)
              __hip_atomic_fetch_add(wblk + k, sw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            else
              atomicAdd(weights + k, sw);
          }
        }
      }
    }
  }
  if (lds_w) {
    __syncthreads();
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x)
      if (wblk[k] != 0.0) atomicAdd(weights + k, wblk[k]);
  }
}

__global__ __launch_bounds__(block) void k_emit(
  const VisRec<1>* __restrict__ recs, size_t n, Geometry geo,
  const GroupInfo* __restrict__ groups, const double2* __restrict__ wsum,
  Mueller mu, int gvis_ready, int adjoint, const float2* __restrict__ gvis_in,
  const double2* __restrict__ residuals, unsigned* __restrict__ cursor,
  Entry4* __restrict__ entries, unsigned* __restrict__ entry_vis) {

  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const VisRec<1>& r = recs[i];
  const unsigned grp = r.cf_index[1];
  const unsigned cfcube = r.cf_index[0];
  const unsigned gcube = r.grid_cube;
  if (!(grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc))) return;
  const GroupInfo g = groups[grp];
  if (!(cfcube < unsigned(g.ncube))) return;
  const Coord c = vis_coord(r, geo, g);
  if (!c.inside) return;
  const bool pos_w = r.uvw[2] > 0;
  const bool grad = r.grad[0] != 0.0 || r.grad[1] != 0.0;
  const int fxi = c.fx + geo.F, fyi = c.fy + geo.F;

  const int tx = tiles_begin(c.gx), ty = tiles_begin(c.gy);
  // corner relative to the tile, fine offsets, flags
  Entry4 e;
  e.h.pos = unsigned(c.gx - tx * tile) | (unsigned(c.gy - ty * tile) << 6)
    | (unsigned(fxi) << 12) | (unsigned(fyi) << 20) | (pos_w ? e4_pos_w : 0u)
    | (grad ? e4_gradient : 0u);
  e.h.gpk = grp | (cfcube << 16);
  if (gvis_ready) {
    e.g = gvis_in[i];
  } else {
    const double2 phasor = cphase(r.phase);
    if (!adjoint) {
      e.g = prephase(r.vis[0], phasor, r.w[0]);
    } else {
      double2 d;
      degrid_norms<1>(geo, g, wsum, mu, pos_w, cfcube, fxi, fyi, &d);
      if (d.x == 0.0 && d.y == 0.0) d = make_double2(1.0, 0.0);
      d.y = -d.y;
      e.g = narrow(kdiv(cmul(residuals[i], phasor), d));
    }
  }
  const int ntiles = geo.ntx * geo.nty;
  for (int gpol = 0; gpol < geo.nr; ++gpol) {
    if (!row_has_index(pos_w ? mu.M[gpol] : mu.Mc[gpol], 1)) continue;
    const int base = int(gcube * geo.nr + gpol) * ntiles;
    const unsigned pos = atomicAdd(cursor + base + ty * geo.ntx + tx, 1u);
    entries[pos] = e;
    if (grad) entry_vis[pos] = unsigned(i);
  }
}

// ---- counting sort -----------------------------------------------------------
//
// 32-bit keys (~0: not sorted) in two levels: the upper bits in at most
// patch_local_keys bins, counted in LDS by the kernel that makes the keys, a
// workgroup of patch_local_threads per batch, with one global atomic per
// workgroup and bin (global counters of every key are bound by the 10 G/s of the
// chip) whose result is the workgroup's place in the bin (k_sort_place); the lower low_bits within a bin in LDS (sort_bin).  As the
// degridder's order 35 us for 1e6 records of 3e5 keys and 25 for 300,000, against
// 130 and 104 us of hipCUB's radix sort (two-polarization residuals 752 -> 649 us).

constexpr int patch_local_threads = 1024;
constexpr int patch_local_keys = 16384;
constexpr int sort_threads = 256;
constexpr int sort_loads = 8;
constexpr int sort_low_bits_max = 14;

struct SortKeys {
  int drop_bits, low_bits, bins;  // the key's bits, from the lowest
};

// block-wide exclusive scan of a[0, n) in LDS (n <= bin_quad_keys_max), returns
// the total; `part` holds blockDim.x / wave + 1 values
__device__ unsigned block_exclusive_scan(unsigned* a, int n, unsigned* part) {
  const int nt = blockDim.x;
  const int per = (n + nt - 1) / nt;
  const int beg = min(n, int(threadIdx.x) * per);
  const int end = min(n, beg + per);
  unsigned sum = 0;
  for (int k = beg; k < end; ++k) sum += a[k];
  // inclusive wave scan of the per-thread sums
  const int lane = threadIdx.x % wave;
  unsigned v = sum;
#pragma unroll
  for (int d = 1; d < wave; d <<= 1) {
    const unsigned t = __shfl_up(v, d, wave);
    if (lane >= d) v += t;
  }
  const int w = threadIdx.x / wave;
  if (lane == wave - 1) part[w] = v;
  __syncthreads();
  if (w == 0) {
    // exclusive scan of the wave totals (at most 64 waves) by one wave
    const int nw = nt / wave;
    const unsigned t = lane < nw ? part[lane] : 0u;
    unsigned incl = t;
#pragma unroll
    for (int d = 1; d < wave; d <<= 1) {
      const unsigned u = __shfl_up(incl, d, wave);
      if (lane >= d) incl += u;
    }
    if (lane < nw) part[lane] = incl - t;
    if (lane == nw - 1) part[nw] = incl;
  }
  __syncthreads();
  unsigned run = part[w] + v - sum;  // exclusive prefix of this thread
  for (int k = beg; k < end; ++k) {
    const unsigned t = a[k];
    a[k] = run;
    run += t;
  }
  const unsigned total = part[nt / wave];
  __syncthreads();
  return total;
}

__global__ __launch_bounds__(block) void k_zero(unsigned* __restrict__ p, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// (lower key bits, index) pairs by bin; order given (no lower bits): the indexes
__global__ __launch_bounds__(patch_local_threads) void k_sort_place(
  size_t n, SortKeys sk, unsigned batch, const unsigned* __restrict__ keys,
  const unsigned* __restrict__ offsets, const unsigned* __restrict__ table,
  unsigned* __restrict__ order, uint2* __restrict__ pairs) {
  __shared__ unsigned at[patch_local_keys];
  const unsigned* row = table + size_t(blockIdx.x) * sk.bins;
  for (int k = threadIdx.x; k < sk.bins; k += blockDim.x) at[k] = offsets[k] + row[k];
  __syncthreads();
  const size_t first = blockIdx.x * (size_t)batch;
  const size_t last = min(n, first + batch);
  for (size_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    const unsigned key = keys[i];
    if (key == ~0u) continue;
    const unsigned pos =
      __hip_atomic_fetch_add(at + (key >> (sk.low_bits + sk.drop_bits)), 1u, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    if (order)
      order[pos] = unsigned(i);
    else
      pairs[pos] = make_uint2((key >> sk.drop_bits) & ((1u << sk.low_bits) - 1u), unsigned(i));
  }
}

// a workgroup's bin, pairs [beg, end): scanned(counts) once each lower key's
// first place is known, then put(place, index) for every pair
template <typename S, typename F>
__device__ __forceinline__ void sort_bin(
  int low_bits, unsigned beg, unsigned end, const uint2* __restrict__ pairs, S scanned, F put) {
  extern __shared__ unsigned low[];  // 2^low_bits
  __shared__ unsigned part[sort_threads / wave + 1];
  constexpr unsigned stride = sort_threads * sort_loads;
  const int low_keys = 1 << low_bits;
  for (int k = threadIdx.x; k < low_keys; k += sort_threads) low[k] = 0u;
  __syncthreads();
  for (int pass = 0; pass < 2; ++pass) {
    for (size_t first = beg; first < end; first += stride) {
      uint2 p[sort_loads];
#pragma unroll
      for (int j = 0; j < sort_loads; ++j) {
        const size_t k = first + j * sort_threads + threadIdx.x;
        p[j] = k < end ? pairs[k] : make_uint2(~0u, 0u);
      }
#pragma unroll
      for (int j = 0; j < sort_loads; ++j) {
        if (p[j].x == ~0u) continue;
        const unsigned at = __hip_atomic_fetch_add(low + p[j].x, 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        if (pass) put(at, p[j].y);
      }
    }
    __syncthreads();
    if (!pass) {
      block_exclusive_scan(low, low_keys, part);
      __syncthreads();
      scanned(low);
      __syncthreads();
    }
  }
}

// Global quadrant bins: k_tally makes each record's entries (one per grid row
// with a Mueller index, keyed by the quadrant of the support corner) in record
// order (slot record * nr + row) and counts the keys' bins; k_sort_place and
// k_tally_sort then move the entries into their keys' ranges, whose offsets
// k_tally_sort writes.  Weights as k_count.  Bound by the passes over records
// and entries: 1e6 records on 4001 x 3750, 96 us (49, 10, 27 and two small ones),
// against 114 with a returning global atomic per entry, a device-wide scan and
// a memset; moving the entries already with k_sort_place costs there (24 us)
// what it saves.
__global__ __launch_bounds__(patch_local_threads) void k_tally(
  const VisRec<1>* __restrict__ recs, size_t n, Geometry geo,
  const GroupInfo* __restrict__ groups, const double2* __restrict__ wsum,
  Mueller mu, int update_weights, int gvis_ready, int adjoint,
  const float2* __restrict__ gvis_in, const double2* __restrict__ residuals,
  SortKeys sk, unsigned batch, unsigned* __restrict__ hist, unsigned* __restrict__ table,
  double* __restrict__ weights, unsigned long long* __restrict__ invalid,
  Entry4* __restrict__ tally, unsigned* __restrict__ tally_keys) {

  __shared__ double wblk[count_planes_lds];
  __shared__ unsigned cnt[patch_local_keys];
  for (int k = threadIdx.x; k < sk.bins; k += blockDim.x) cnt[k] = 0u;
  const int nplanes = geo.nr * geo.nc;
  const bool lds_w = update_weights && nplanes <= count_planes_lds;
  if (lds_w)
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x) wblk[k] = 0.0;
  __syncthreads();

  const size_t first = blockIdx.x * (size_t)batch;
  const size_t last = min(n, first + batch);
  const int ntiles = geo.ntx * geo.nty;
  // every thread runs the same number of iterations (the wave reductions
  // below need all lanes)
  for (size_t at = first; at < last; at += blockDim.x) {
    const size_t i = at + threadIdx.x;
    bool counted = false;
    unsigned gcube = 0;
    double tw[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < last) {
      // slots of rows without an entry say so
      for (int gpol = 0; gpol < geo.nr; ++gpol)
        tally_keys[i * geo.nr + gpol] = ~0u;
      const VisRec<1>& r = recs[i];
      const unsigned grp = r.cf_index[1];
      const unsigned cfcube = r.cf_index[0];
      gcube = r.grid_cube;
      bool valid = grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc);
      if (valid) valid = cfcube < unsigned(groups[grp].ncube);
      if (!valid) {
        atomicAdd(invalid, 1ull);
      } else {
        const GroupInfo g = groups[grp];
        const Coord c = vis_coord(r, geo, g);
        const bool pos_w = r.uvw[2] > 0;
        const int fxi = c.fx + geo.F, fyi = c.fy + geo.F;
        if (c.inside && update_weights) {
          counted = true;
          for (int gpol = 0; gpol < geo.nr; ++gpol) {
            const int* row = pos_w ? mu.M[gpol] : mu.Mc[gpol];
            const int m = row[0];
            double mag = 0.0;
            if (m >= 0 && m < g.nmueller) {
              const double2 sw = wsum[g.wsum_offset
                                      + ((long long)(cfcube * g.nmueller + m) * geo.nf
                                         + fxi) * geo.nf + fyi];
              mag = hypot(sw.x, sw.y);
            }
            tw[gpol] = mag * double(r.w[0]);
          }
        }
        if (c.inside) {
          const bool grad = r.grad[0] != 0.0 || r.grad[1] != 0.0;
          Entry4 e;
          const int tx = tiles_begin(c.gx), ty = tiles_begin(c.gy);
          e.h.pos = unsigned(c.gx - tx * tile) | (unsigned(c.gy - ty * tile) << 6)
            | (unsigned(fxi) << 12) | (unsigned(fyi) << 20) | (pos_w ? e4_pos_w : 0u)
            | (grad ? e4_gradient : 0u);
          e.h.gpk = grp | (cfcube << 16);
          if (gvis_ready) {
            e.g = gvis_in[i];
          } else {
            const double2 phasor = cphase(r.phase);
            if (!adjoint) {
              e.g = prephase(r.vis[0], phasor, r.w[0]);
            } else {
              double2 d;
              degrid_norms<1>(geo, g, wsum, mu, pos_w, cfcube, fxi, fyi, &d);
              if (d.x == 0.0 && d.y == 0.0) d = make_double2(1.0, 0.0);
              d.y = -d.y;
              e.g = narrow(kdiv(cmul(residuals[i], phasor), d));
            }
          }
          for (int gpol = 0; gpol < geo.nr; ++gpol) {
            if (!row_has_index(pos_w ? mu.M[gpol] : mu.Mc[gpol], 1)) continue;
            const int key =
              quad_key((int(gcube) * geo.nr + gpol) * ntiles + ty * geo.ntx + tx, c.gx, c.gy);
            __hip_atomic_fetch_add(cnt + (unsigned(key) >> sk.low_bits), 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            tally[i * geo.nr + gpol] = e;
            tally_keys[i * geo.nr + gpol] = unsigned(key);
          }
        }
      }
    }
    if (update_weights) {
      unsigned long long active = __ballot(counted);
      const int lane = threadIdx.x % wave;
      while (active) {
        const int leader = __ffsll((long long)active) - 1;
        const unsigned cube = __shfl(gcube, leader, wave);
        const bool mine = counted && gcube == cube;
        active &= ~__ballot(mine);
        for (int gpol = 0; gpol < geo.nr; ++gpol) {
          const double sw = wave_sum(mine ? tw[gpol] : 0.0);
          if (lane == leader) {
            const size_t k = size_t(cube) * geo.nr + gpol;
            if (lds_w)
              __hip_atomic_fetch_add(wblk + k, sw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            else
              atomicAdd(weights + k, sw);
          }
        }
      }
    }
  }
  __syncthreads();
  if (lds_w)
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x)
      if (wblk[k] != 0.0) atomicAdd(weights + k, wblk[k]);
  unsigned* row = table + size_t(blockIdx.x) * sk.bins;
  for (int k = threadIdx.x; k < sk.bins; k += blockDim.x)
    row[k] = cnt[k] ? atomicAdd(hist + k, cnt[k]) : 0u;
}

// one workgroup per bin: its entries in order of their keys, and the keys'
// offsets
__global__ __launch_bounds__(sort_threads) void k_tally_sort(
  int low_bits, size_t nkeys, int nr, const unsigned* __restrict__ bin_offsets,
  const uint2* __restrict__ pairs, const Entry4* __restrict__ tally,
  unsigned* __restrict__ offsets, Entry4* __restrict__ entries,
  unsigned* __restrict__ entry_vis) {
  const unsigned beg = bin_offsets[blockIdx.x], end = bin_offsets[blockIdx.x + 1];
  const size_t key0 = size_t(blockIdx.x) << low_bits;
  const size_t keys = min(size_t(1) << low_bits, nkeys - key0);
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) offsets[nkeys] = end;
  if (beg == end) {
    for (size_t k = threadIdx.x; k < keys; k += sort_threads) offsets[key0 + k] = beg;
    return;
  }
  sort_bin(
    low_bits, beg, end, pairs,
    [&](const unsigned* first) {
      for (size_t k = threadIdx.x; k < keys; k += sort_threads) offsets[key0 + k] = beg + first[k];
    },
    [&](unsigned at, unsigned slot) {
      const Entry4 e = tally[slot];
      entries[beg + at] = e;
      if (e.h.pos & e4_gradient) entry_vis[beg + at] = slot / unsigned(nr);
    });
}

__device__ __forceinline__ int bcast(int v, int k) {
  return __builtin_amdgcn_readlane(v, k);
}
__device__ __forceinline__ float bcast(float v, int k) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// ---- gridding, block-local bins ----------------------------------------------
//
// For grids with few (plane, tile) keys (<= bin_keys_max) the bins are built
// without any contended global atomic:
// k_bin     one workgroup per 4096 records: a histogram of the block's
//           entries over all keys in LDS, its exclusive scan, the per-block
//           offset table off[block][key] (nkeys + 1 values), then each entry
//           written at its block-local position -- one pass over the records.
//           Weights are reduced per grid plane in LDS first.

constexpr int bin_threads = 1024;
constexpr int bin_recs_per_thread = 4;
constexpr int bin_records = bin_threads * bin_recs_per_thread;  // per block
constexpr int bin_keys_max = 8192;        // (plane, tile) keys of the block-local bins
constexpr int bin_quad_keys_max = 16384;  // quadrant keys (4 per tile key): LDS histogram
constexpr int bin_planes_max = 1024;
constexpr int tile_bins_max = 2048;  // bin blocks per pass (LDS of k_tile4)
constexpr int bin_stage_bytes = 65536;  // LDS staging of k_bin's haloed entries (one
                                        // chunk for a block of one-polarization entries)

// one entry per record and plane, keyed by the tile of the support corner
__global__ __launch_bounds__(bin_threads) void k_bin(
  const VisRec<1>* __restrict__ recs, size_t n, Geometry geo,
  const GroupInfo* __restrict__ groups, const double2* __restrict__ wsum,
  Mueller mu, int update_weights, int gvis_ready, int adjoint, int degrid_pass,
  const float2* __restrict__ gvis_in, const double2* __restrict__ residuals,
  unsigned* __restrict__ off_table, void* __restrict__ entries_out,
  unsigned* __restrict__ entry_vis, size_t block_cap, double* __restrict__ weights,
  unsigned long long* __restrict__ invalid, VisRec<1>* __restrict__ copy_recs, int quad_keys) {

  __shared__ unsigned cnt[bin_quad_keys_max];
  __shared__ double wl[bin_planes_max];
  __shared__ unsigned part[bin_threads / wave + 1];

  // quad_keys: a key per 16 x 16 quadrant of each (plane, tile),
  // key = 4 * tile key + quadrant of the support corner, so that the
  // entries of one quadrant are contiguous within each bin block
  const int nkeys = geo.ntx * geo.nty * geo.nr * geo.nc * (quad_keys ? 4 : 1);
  const int nplanes = geo.nr * geo.nc;
  const bool local_w = nplanes <= bin_planes_max;
  for (int k = threadIdx.x; k < nkeys; k += bin_threads) cnt[k] = 0;
  if (local_w)
    for (int k = threadIdx.x; k < nplanes; k += bin_threads) wl[k] = 0.0;
  __syncthreads();

  const int ntiles = geo.ntx * geo.nty;
  const size_t b = blockIdx.x;
  // weights of this thread's records, per grid row, for one grid cube at a
  // time (records of another cube flush the sums first)
  int wcube = -1;
  double wacc[4] = {0.0, 0.0, 0.0, 0.0};
  auto flush_weights = [&](int cube, const double* acc) {
    for (int gpol = 0; gpol < geo.nr; ++gpol) {
      const int k = cube * geo.nr + gpol;
      if (local_w)
        __hip_atomic_fetch_add(wl + k, acc[gpol], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      else
        atomicAdd(weights + k, acc[gpol]);
    }
  };
  Entry e[bin_recs_per_thread];
  bool keep[bin_recs_per_thread];
  unsigned gc[bin_recs_per_thread];
  unsigned ninvalid = 0;

  // grid rows with an index, per sign of w (bit gpol): the Mueller rows read
  // at constant indices (kernel-argument scalars), not per record
  unsigned rows_m = 0u, rows_mc = 0u;
#pragma unroll
  for (int gp = 0; gp < 4; ++gp) {
    if (gp >= geo.nr) continue;
    rows_m |= row_has_index(mu.M[gp], 1) ? 1u << gp : 0u;
    rows_mc |= row_has_index(mu.Mc[gp], 1) ? 1u << gp : 0u;
  }
  const bool one_group = geo.ngroups == 1;
  const GroupInfo group0 = groups[0];

  // the thread's records are loaded whole, two at a time, so that two records'
  // loads are in flight at once rather than one record (and its chain of
  // dependent loads) at a time; four would spill the 128 registers a
  // 1024-thread block allows
  constexpr int words = int(sizeof(VisRec<1>) / sizeof(unsigned long long));
  static_assert(sizeof(VisRec<1>) % sizeof(unsigned long long) == 0, "8-byte record words");
  static_assert(bin_recs_per_thread % 2 == 0, "records loaded in pairs");
  VisRec<1> rc[2];
  // the place of each of this thread's entries (one per record and
  // grid row with an index; ~0u for none) within its key, from the count's
  // returned value, then (after the scan) its block-local position; the
  // entries are then written through LDS in position order
  unsigned hpos[bin_recs_per_thread][4];
#pragma unroll
  for (int j = 0; j < bin_recs_per_thread; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) hpos[j][r] = ~0u;

#pragma unroll
  for (int j = 0; j < bin_recs_per_thread; ++j) {
    if (j % 2 == 0) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const size_t i = b * bin_records + size_t(j + jj) * bin_threads + threadIdx.x;
        if (i >= n) continue;
        const unsigned long long* src = reinterpret_cast<const unsigned long long*>(recs + i);
        unsigned long long wds[words];
#pragma unroll
        for (int k = 0; k < words; ++k) wds[k] = src[k];
        __builtin_memcpy(&rc[jj], wds, sizeof(VisRec<1>));
      }
    }
    keep[j] = false;
    const size_t i = b * bin_records + size_t(j) * bin_threads + threadIdx.x;
    if (i >= n) continue;
    const VisRec<1>& r = rc[j % 2];
    // degridding that returns the batch: every record is written to the
    // returned batch here, whose values the degridding kernels then replace
    if (copy_recs) {
      const unsigned long long* src = reinterpret_cast<const unsigned long long*>(&r);
      unsigned long long* dst = reinterpret_cast<unsigned long long*>(copy_recs + i);
#pragma unroll
      for (int k = 0; k < words; ++k) dst[k] = src[k];
    }
    const unsigned grp = r.cf_index[1];
    const unsigned cfcube = r.cf_index[0];
    const unsigned gcube = r.grid_cube;
    bool valid = grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc);
    const GroupInfo g = !valid || one_group ? group0 : groups[grp];
    if (valid) valid = cfcube < unsigned(g.ncube);
    if (!valid) {
      // counted by the gridding pass only
      if (!degrid_pass) ++ninvalid;
      continue;
    }
    const Coord c = vis_coord(r, geo, g);
    if (!c.inside) continue;
    const bool pos_w = r.uvw[2] > 0;
    const bool grad = r.grad[0] != 0.0 || r.grad[1] != 0.0;
    const int fxi = c.fx + geo.F, fyi = c.fy + geo.F;
    keep[j] = true;
    gc[j] = gcube;
    e[j].gx = c.gx;
    e[j].gy = c.gy;
    e[j].fpk = unsigned(fxi) | (unsigned(fyi) << 8)
      | (unsigned((pos_w ? flag_pos_w : 0) | (grad ? flag_gradient : 0)) << 16);
    e[j].gpk = grp | (cfcube << 16);
    if (degrid_pass) {
      // degridding reads the model: entries carry no values
      e[j].g = make_float2(0.0f, 0.0f);
    } else if (gvis_ready) {
      e[j].g = gvis_in[i];
    } else {
      const double2 phasor = cphase(r.phase);
      if (!adjoint) {
        e[j].g = prephase(r.vis[0], phasor, r.w[0]);
      } else {
        double2 d;
        degrid_norms<1>(geo, g, wsum, mu, pos_w, cfcube, fxi, fyi, &d);
        if (d.x == 0.0 && d.y == 0.0) d = make_double2(1.0, 0.0);
        d.y = -d.y;
        e[j].g = narrow(kdiv(cmul(residuals[i], phasor), d));
      }
    }
    if (update_weights) {
      // twgt = |sum_XY cf'| * w (src/hpg_core.hpp:877-885); grid rows
      // unrolled, so the Mueller indices are scalars
      // and the slice-sum loads of all rows issue together
      if (int(gcube) != wcube) {
        if (wcube >= 0) flush_weights(wcube, wacc);
        wcube = int(gcube);
#pragma unroll
        for (int k = 0; k < 4; ++k) wacc[k] = 0.0;
      }
#pragma unroll
      for (int gp = 0; gp < 4; ++gp) {
        if (gp >= geo.nr) continue;
        const int m = pos_w ? mu.M[gp][0] : mu.Mc[gp][0];
        double mag = 0.0;
        if (m >= 0 && m < g.nmueller) {
          const double2 sw = wsum[g.wsum_offset
                                  + ((long long)(cfcube * g.nmueller + m) * geo.nf + fxi)
                                    * geo.nf + fyi];
          mag = hypot(sw.x, sw.y);
        }
        wacc[gp] += mag * double(r.w[0]);
      }
    }
    const int t = tiles_begin(c.gy) * geo.ntx + tiles_begin(c.gx);
    const unsigned rows = (pos_w != bool(degrid_pass)) ? rows_m : rows_mc;
    for (int gpol = 0; gpol < geo.nr; ++gpol) {
      if (!((rows >> gpol) & 1u)) continue;
      const int base = (int(gcube) * geo.nr + gpol) * ntiles;
      const unsigned place = __hip_atomic_fetch_add(
        cnt + (quad_keys ? quad_key(base + t, c.gx, c.gy) : base + t), 1u,
        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r == gpol) hpos[j][r] = place;
    }
  }
  // the threads' weight sums: one sum per (wave, grid cube) present, the
  // wave's lanes all active here
  if (update_weights) {
    const int lane = threadIdx.x % wave;
    int key = wcube;
    for (;;) {
      const unsigned long long act = __ballot(key >= 0);
      if (act == 0) break;
      const int leader = __ffsll((long long)act) - 1;
      const int lk = __shfl(key, leader, wave);
      double part_w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        part_w[k] = k < geo.nr ? wave_sum(key == lk ? wacc[k] : 0.0) : 0.0;
      if (lane == leader) flush_weights(lk, part_w);
      if (key == lk) key = -1;
    }
  }
  // invalid records: one global atomic per wave at most
  {
    unsigned long long inv = ninvalid;
#pragma unroll
    for (int m = wave / 2; m > 0; m >>= 1) inv += __shfl_xor(inv, m, wave);
    if (threadIdx.x % wave == 0 && inv) atomicAdd(invalid, inv);
  }
  __syncthreads();
  const unsigned btotal = block_exclusive_scan(cnt, nkeys, part);
  unsigned* tab = off_table + b * size_t(nkeys + 1);
  for (int k = threadIdx.x; k < nkeys; k += bin_threads) tab[k] = cnt[k];
  if (threadIdx.x == 0) tab[nkeys] = btotal;
  if (update_weights && local_w)
    for (int k = threadIdx.x; k < nplanes; k += bin_threads)
      if (wl[k] != 0.0) atomicAdd(weights + k, wl[k]);
  __syncthreads();

  unsigned* outv = entry_vis + b * block_cap;
#pragma unroll
  for (int j = 0; j < bin_recs_per_thread; ++j) {
    if (!keep[j]) continue;
    const size_t i = size_t(j) * bin_threads + threadIdx.x;
    const bool pos_w = (e[j].fpk >> 16) & flag_pos_w;
    const bool grad = (e[j].fpk >> 16) & flag_gradient;
    const int t = tiles_begin(e[j].gy) * geo.ntx + tiles_begin(e[j].gx);
    const unsigned rows = (pos_w != bool(degrid_pass)) ? rows_m : rows_mc;
    for (int gpol = 0; gpol < geo.nr; ++gpol) {
      if (!((rows >> gpol) & 1u)) continue;
      const int base = (int(gc[j]) * geo.nr + gpol) * ntiles;
      // the key's offset (cnt holds the scan now) + the entry's place
      unsigned place = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r == gpol) place = hpos[j][r];
      const unsigned pos =
        cnt[quad_keys ? quad_key(base + t, e[j].gx, e[j].gy) : base + t] + place;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r == gpol) hpos[j][r] = pos;
      if (grad || degrid_pass) outv[pos] = unsigned(b * bin_records + i);
    }
  }
  // chunks of the block's entry range: each thread puts its entries of
  // the chunk into LDS, then the block copies the chunk out contiguously
  // (scattered 16-byte stores would each write a partial line)
  constexpr unsigned ewords = unsigned(sizeof(Entry4) / sizeof(unsigned long long));
  constexpr unsigned chunk = unsigned(bin_stage_bytes / sizeof(Entry4));
  __shared__ unsigned long long stage[chunk * ewords];
  Entry4* staged = reinterpret_cast<Entry4*>(stage);
  unsigned long long* dst =
    reinterpret_cast<unsigned long long*>(static_cast<Entry4*>(entries_out) + b * block_cap);
  for (unsigned c0 = 0; c0 < btotal; c0 += chunk) {
#pragma unroll
    for (int j = 0; j < bin_recs_per_thread; ++j) {
      if (!keep[j]) continue;
      const bool pos_w = (e[j].fpk >> 16) & flag_pos_w;
      const bool grad = (e[j].fpk >> 16) & flag_gradient;
      Entry4 q;
      q.h.pos = unsigned(e[j].gx - tiles_begin(e[j].gx) * tile)
        | (unsigned(e[j].gy - tiles_begin(e[j].gy) * tile) << 6)
        | ((e[j].fpk & 0xffffu) << 12) | (pos_w ? e4_pos_w : 0u)
        | (grad ? e4_gradient : 0u);
      q.h.gpk = e[j].gpk;
      q.g = e[j].g;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (hpos[j][r] - c0 < chunk) staged[hpos[j][r] - c0] = q;
    }
    __syncthreads();
    const unsigned cw = min(chunk, btotal - c0) * ewords;
    for (unsigned k = threadIdx.x; k < cw; k += bin_threads) dst[size_t(c0) * ewords + k] = stage[k];
    __syncthreads();
  }
}

// ---- gridding, haloed tiles ---------------------------------------------
//
// k_bin writes one Entry4 per (record, plane) into the bin of the
// tile that holds the support corner.  The workgroup of a key accumulates
// the tile plus a halo of hx = max_sx - 1 columns and hy = max_sy - 1 rows on
// its high sides (R = (tile + hx) x (tile + hy) pixels in LDS), so every tap
// of an entry lands in LDS without clipping.  One lane carries one entry
// through all of its taps: per tap a CF load, the FP32 product and the LDS
// accumulation, with no cross-lane traffic.  The workgroup then adds its own
// tile into the grid (it is the only writer of those pixels during the
// kernel) and stores the halo, as FP64 values, into a per-key side buffer;
// k_halo adds each tile's neighbours' halos into it afterwards, in a fixed
// order.  Requires hx, hy < tile.

constexpr int halo_block = 256;

// The dispatcher hands workgroups to the 8 XCDs in turn (workgroup b to
// XCD b mod 8).  The keyed kernels take key xcd_key(b) instead of b, so
// that each XCD works through one contiguous run of keys: neighbouring
// keys' bin segments and offset-table entries share cache lines, which
// are then fetched into one XCD's L2 instead of several.  A bijection on
// [0, nkeys).
constexpr unsigned xcd_count = 8;
__device__ __forceinline__ unsigned xcd_key(unsigned b, unsigned nkeys) {
  const unsigned x = b % xcd_count, j = b / xcd_count;
  const unsigned q = nkeys / xcd_count, r = nkeys % xcd_count;
  return x * q + min(x, r) + j;
}
constexpr int halo_chunk = 8;     // CF taps loaded together per lane
constexpr int halo_classes = 32;  // LDS bank classes of the entry schedule
constexpr int halo_sched = 2048;  // entries per scheduling round

// pixels of the halo of one key: columns [tile, tile + hx) of rows
// [0, tile), then all columns of rows [tile, tile + hy)
__host__ __device__ inline int halo_pixels(int hx, int hy) {
  return hx * tile + (tile + hx) * hy;
}

// tile accumulation schemes of k_tile4
//   acc_f64       FP64 LDS atomics (FP64 grids; also selectable for FP32 grids)
//   acc_f32_cas   FP32 hi/lo per pixel packed into 64 bits and updated by
//                 compare-and-swap: hi' = fl(hi + p), lo' = fl(lo + err) with
//                 err the exact two-sum error, so each update is one
//                 error-free transformation on one coherent pair
constexpr int acc_f64 = 0;
constexpr int acc_f32_cas = 2;

template <int MODE, int ACC>
__global__ __launch_bounds__(halo_block) void k_tile4(
  Geometry geo, const GroupInfo* __restrict__ groups,
  const float2* __restrict__ taps, Mueller mu, const unsigned* __restrict__ off_table,
  int nbins, size_t block_cap, const Entry4* __restrict__ entries,
  const unsigned* __restrict__ entry_vis, const VisRec<1>* __restrict__ recs,
  int hx, int hy, void* __restrict__ grid, double2* __restrict__ halo,
  unsigned* __restrict__ halo_set) {
  static_assert(MODE == 1 || ACC == acc_f64, "FP64 grids accumulate in FP64");

  extern __shared__ double smem[];
  const int RX = tile + hx;
  const int RY = tile + hy;
  const int R = RX * RY;
  // LDS: accumulators (16 bytes per region pixel), then the segment tables
  double* acc64 = smem;                                // acc_f64: re[R], im[R]
  unsigned long long* pairs = reinterpret_cast<unsigned long long*>(smem);  // cas: re[R], im[R]
  unsigned* seg_pref = reinterpret_cast<unsigned*>(smem + 2 * R);
  unsigned* seg_beg = seg_pref + nbins + 1;
  unsigned* part = seg_beg + nbins;
  unsigned* cls = part + (halo_block / wave + 1);  // bank classes: counts, then cursors
  unsigned* sched = cls + halo_classes;            // entry indexes of one round

  const unsigned key = xcd_key(blockIdx.x, gridDim.x);  // one block per key
  const int nkeys = geo.ntx * geo.nty * geo.nr * geo.nc;
  for (int bb = threadIdx.x; bb < nbins; bb += halo_block) {
    const unsigned* tab = off_table + size_t(bb) * (nkeys + 1);
    const unsigned s0 = tab[key], s1 = tab[key + 1];
    seg_pref[bb] = s1 - s0;
    seg_beg[bb] = s0;
  }
  __syncthreads();
  const unsigned total = block_exclusive_scan(seg_pref, nbins, part);
  if (total == 0) {
    if (threadIdx.x == 0) halo_set[key] = 0u;
    return;
  }
  if (threadIdx.x == 0) seg_pref[nbins] = total;

  const int ntiles = geo.ntx * geo.nty;
  const unsigned plane = key / ntiles;
  const int t = int(key % ntiles);
  const int x0 = (t % geo.ntx) * tile;
  const int y0 = (t / geo.ntx) * tile;
  const int gpol = int(plane % geo.nr);

  for (int k = threadIdx.x; k < 2 * R; k += halo_block) acc64[k] = 0.0;
  __syncthreads();

  const int w = threadIdx.x / wave;
  const int lane = threadIdx.x % wave;
  constexpr int nw = halo_block / wave;

  // entry q of the key (0 <= q < total): its index in the entry array
  auto locate = [&](unsigned q) {
    int lo = 0, hi = nbins;  // seg_pref[lo] <= q < seg_pref[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (seg_pref[mid] <= q) lo = mid; else hi = mid;
    }
    return unsigned(lo) * unsigned(block_cap) + seg_beg[lo] + (q - seg_pref[lo]);
  };
  // LDS bank class of an entry's first tap; every tap of every lane adds
  // the same offset to it, so a wave whose lanes hold consecutive classes
  // spreads each of its LDS updates evenly over the banks
  auto bank_class = [&](unsigned pos) {
    return unsigned(int((pos >> 6) & 63u) * RX + int(pos & 63u)) % unsigned(halo_classes);
  };
  // rank of this lane in a wave's sample of the class-sorted round: lanes
  // l and l + 32 take neighbouring samples, so lanes 0-31 (and 32-63) hold
  // ascending classes
  const unsigned rank = unsigned((lane & 31) * 2 + (lane >> 5));

  for (unsigned r0 = 0; r0 < total; r0 += halo_sched) {
    const unsigned rn = min(unsigned(halo_sched), total - r0);
    if (rn <= wave) {  // one wave's entries: as they come
      if (threadIdx.x < rn) sched[threadIdx.x] = locate(r0 + threadIdx.x);
      __syncthreads();
    } else {
      // counting sort of the round's entries by bank class
      if (threadIdx.x < halo_classes) cls[threadIdx.x] = 0u;
      __syncthreads();
      for (unsigned q = threadIdx.x; q < rn; q += halo_block)
        __hip_atomic_fetch_add(cls + bank_class(entries[locate(r0 + q)].h.pos), 1u,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned run = 0;
        for (int c = 0; c < halo_classes; ++c) {
          const unsigned t = cls[c];
          cls[c] = run;
          run += t;
        }
      }
      __syncthreads();
      for (unsigned q = threadIdx.x; q < rn; q += halo_block) {
        const unsigned idx = locate(r0 + q);
        const unsigned slot = __hip_atomic_fetch_add(
          cls + bank_class(entries[idx].h.pos), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        sched[slot] = idx;
      }
      __syncthreads();
    }
    // batch j of the round takes sorted entries rank * nbatch + j
    const unsigned nbatch = (rn + wave - 1) / wave;
    for (unsigned j = w; j < nbatch; j += nw) {
      const unsigned sp = rank * nbatch + j;
      if (sp >= rn) continue;
      const unsigned idx = sched[sp];
      const Entry4 e = entries[idx];
      const unsigned pos = e.h.pos;
      const int lx = int(pos & 63u);
      const int ly = int((pos >> 6) & 63u);
      const int fxi = int((pos >> 12) & 255u);
      const int fyi = int((pos >> 20) & 255u);
      const bool pos_w = pos & e4_pos_w;
      const bool grad = pos & e4_gradient;
      const int grp = int(e.h.gpk & 0xffffu);
      const int cfcube = int(e.h.gpk >> 16);
      const GroupInfo g = groups[grp];
      const int sx = g.sx, sy = g.sy;
      const int* row = pos_w ? mu.M[gpol] : mu.Mc[gpol];
      const float imf = pos_w ? -1.0f : 1.0f;
      const int m = row[0];
      const bool use = m >= 0 && m < g.nmueller;
      const float2* slice = taps + plane_start(g, geo.nf, int(cfcube), use ? m : 0, fxi, fyi);
      double phi0x = 0.0, phi0y = 0.0, dphix = 0.0, dphiy = 0.0;
      if (grad) {
        const unsigned i = entry_vis[idx];
        const double gxr = recs[i].grad[0];
        const double gyr = recs[i].grad[1];
        phi0x = -gxr * ((sx / 2) * geo.os - (fxi - geo.F));
        phi0y = -gyr * ((sy / 2) * geo.os - (fyi - geo.F));
        dphix = gxr * geo.os;
        dphiy = gyr * geo.os;
      }
      // the value of one tap
      auto tap_value = [&](float2 cc, int X, int Y) {
        cc.y *= imf;
        if (grad) cc = cmul(cc, narrow(cphase((phi0x + X * dphix) + (phi0y + Y * dphiy))));
        return cmul(cc, e.g);
      };
      // adds the M taps held in the arrays to LDS pixels li[0..M) (ok[m]:
      // tap present).  The compare-and-swap form reads each pixel just
      // before its swap: the wave's LDS operations execute in order, so two
      // lanes of one wave only race on a pixel when their corners coincide;
      // failed swaps are retried after the last tap.
      auto accumulate = [&](auto m_c, const int* li, const bool* ok, const float2* p) {
        constexpr int M = decltype(m_c)::value;
        if constexpr (ACC == acc_f64) {
#pragma unroll
          for (int m = 0; m < M; ++m) {
            if (!ok[m]) continue;
            __hip_atomic_fetch_add(acc64 + li[m], double(p[m].x), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(acc64 + R + li[m], double(p[m].y), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        } else {
          // pixel li holds (H_re, L_re) at pairs[li], (H_im, L_im) at pairs[R + li]
          unsigned long long er[M], ei[M];
          bool okr[M], oki[M];
#pragma unroll
          for (int m = 0; m < M; ++m) {
            if (!ok[m]) continue;
            er[m] = pairs[li[m]];
            ei[m] = pairs[R + li[m]];
            okr[m] = pair_swap(pairs + li[m], er[m], pair_plus(er[m], p[m].x));
            oki[m] = pair_swap(pairs + R + li[m], ei[m], pair_plus(ei[m], p[m].y));
          }
#pragma unroll
          for (int m = 0; m < M; ++m) {
            if (!ok[m]) continue;
            if (!okr[m]) pair_add(pairs + li[m], er[m], p[m].x);
            if (!oki[m]) pair_add(pairs + R + li[m], ei[m], p[m].y);
          }
        }
      };
      // any support: taps in slice order (t = Y * sx + X), halo_chunk at a
      // time; full chunks are straight-line code
      auto run_chunks = [&]() {
        const int ntap = sx * sy;
        int cx = 0, cy = 0;          // (X, Y) of the chunk's first tap
        int lc = ly * RX + lx;       // its LDS pixel
        const int wrap = RX - sx;    // pixel step from a row end to the next row
        auto do_chunk = [&](auto full, int t0) {
          constexpr bool FULL = decltype(full)::value;
          bool ok[halo_chunk];
          int li[halo_chunk];
          float2 c[halo_chunk], p[halo_chunk];
          int Xk[halo_chunk], Yk[halo_chunk];
#pragma unroll
          for (int k = 0; k < halo_chunk; ++k) {
            ok[k] = FULL || t0 + k < ntap;
            Xk[k] = cx;
            Yk[k] = cy;
            li[k] = lc;
            const bool eol = ++cx == sx;
            cx = eol ? 0 : cx;
            cy += eol ? 1 : 0;
            lc += eol ? 1 + wrap : 1;
            float2 tv = make_float2(0.0f, 0.0f);
            if (ok[k]) tv = slice[t0 + k];
            c[k] = use ? tv : make_float2(0.0f, 0.0f);
          }
#pragma unroll
          for (int k = 0; k < halo_chunk; ++k)
            p[k] = tap_value(c[k], Xk[k], Yk[k]);
          accumulate(std::integral_constant<int, halo_chunk>{}, li, ok, p);
        };
        int t0 = 0;
        for (; t0 + halo_chunk <= ntap; t0 += halo_chunk) do_chunk(std::true_type{}, t0);
        if (t0 < ntap) do_chunk(std::false_type{}, t0);
      };
      run_chunks();
    }
    __syncthreads();  // the next round reuses cls and sched
  }

  const int hs = halo_pixels(hx, hy);
  double2* hk = halo + size_t(key) * hs;
  for (int k = threadIdx.x; k < R; k += halo_block) {
    const int ry = k / RX;
    const int rx = k - ry * RX;
    // tile value: FP64 sum (acc_f64) or FP32 hi + lo
    double vr, vi;
    float fr = 0.0f, fi = 0.0f, flr = 0.0f, fli = 0.0f;
    if constexpr (ACC == acc_f64) {
      vr = acc64[k];
      vi = acc64[R + k];
    } else {
      const unsigned long long pr = pairs[k], pi = pairs[R + k];
      fr = __uint_as_float(unsigned(pr));
      flr = __uint_as_float(unsigned(pr >> 32));
      fi = __uint_as_float(unsigned(pi));
      fli = __uint_as_float(unsigned(pi >> 32));
      vr = double(fr) + double(flr);
      vi = double(fi) + double(fli);
    }
    if (rx < tile && ry < tile) {
      const int xx = x0 + rx, yy = y0 + ry;
      if (xx >= geo.nx || yy >= geo.ny) continue;
      const size_t gi = (size_t(plane) * geo.ny + yy) * geo.nx + xx;
      if constexpr (MODE == 0) {
        double2* gp = static_cast<double2*>(grid) + gi;
        double2 gvl = *gp;
        gvl.x += vr;
        gvl.y += vi;
        *gp = gvl;
      } else if constexpr (ACC == acc_f64) {
        // one rounding of grid value + FP64 tile sum
        float2* gp = static_cast<float2*>(grid) + gi;
        const float2 g0 = *gp;
        *gp = make_float2(float(double(g0.x) + vr), float(double(g0.y) + vi));
      } else {
        float2* gp = static_cast<float2*>(grid) + gi;
        const float2 g0 = *gp;
        float sr, er, si, ei;
        two_sum(g0.x, fr, sr, er);
        two_sum(g0.y, fi, si, ei);
        *gp = make_float2(sr + (er + flr), si + (ei + fli));
      }
    } else {
      const int h = ry < tile ? ry * hx + (rx - tile) : tile * hx + (ry - tile) * RX + rx;
      hk[h] = make_double2(vr, vi);
    }
  }
  if (threadIdx.x == 0) halo_set[key] = 1u;
}

// adds the halos of each tile's left, upper and upper-left neighbours into
// the tile (pixels (u, v) of the tile with u < hx or v < hy), one thread per
// pixel, in that fixed order
template <typename T>
__global__ void k_halo(
  Geometry geo, int hx, int hy, const double2* __restrict__ halo,
  const unsigned* __restrict__ halo_set, size_t nkeys, T* __restrict__ grid) {
  const int zone = hy * tile + (tile - hy) * hx;
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (zone == 0 || tid >= nkeys * zone) return;
  const size_t key = tid / zone;
  const int z = int(tid - key * zone);
  int u, v;
  if (z < hy * tile) {
    v = z / tile;
    u = z - v * tile;
  } else {
    const int z2 = z - hy * tile;
    v = hy + z2 / hx;
    u = z2 - (v - hy) * hx;
  }
  const int ntiles = geo.ntx * geo.nty;
  const size_t plane = key / ntiles;
  const int t = int(key - plane * ntiles);
  const int TX = t % geo.ntx;
  const int TY = t / geo.ntx;
  const int x = TX * tile + u;
  const int y = TY * tile + v;
  if (x >= geo.nx || y >= geo.ny) return;
  const int hs = halo_pixels(hx, hy);
  const int RX = tile + hx;
  // the neighbours' flags, their halo values and the grid value load
  // together (a halo not written by this pass is read but not added)
  const bool has_l = TX > 0 && u < hx;
  const bool has_u = TY > 0 && v < hy;
  const bool has_ul = has_l && has_u;
  const unsigned set_l = has_l ? halo_set[key - 1] : 0u;
  const unsigned set_u = has_u ? halo_set[key - geo.ntx] : 0u;
  const unsigned set_ul = has_ul ? halo_set[key - geo.ntx - 1] : 0u;
  double2 h_l = make_double2(0.0, 0.0), h_u = h_l, h_ul = h_l;
  if (has_l) h_l = halo[(key - 1) * hs + v * hx + u];
  if (has_u) h_u = halo[(key - geo.ntx) * hs + tile * hx + v * RX + u];
  if (has_ul) h_ul = halo[(key - geo.ntx - 1) * hs + tile * hx + v * RX + tile + u];
  T* gp = grid + (plane * geo.ny + y) * geo.nx + x;
  T g = *gp;
  if (!(set_l | set_u | set_ul)) return;
  // added in the order left, upper, upper-left
  double sr = 0.0, si = 0.0;
  if (set_l) {
    sr += h_l.x;
    si += h_l.y;
  }
  if (set_u) {
    sr += h_u.x;
    si += h_u.y;
  }
  if (set_ul) {
    sr += h_ul.x;
    si += h_ul.y;
  }
  g.x = double(g.x) + sr;
  g.y = double(g.y) + si;
  *gp = g;
}

constexpr int quad_edge = tile / 2;  // pixels of a tile quadrant
constexpr unsigned quad_pos_w = 1u << 29;

// The flush of the quadrant kernel: the sum of the four quadrant regions
// of (hi, lo) pairs (LDS, float4 per pixel, quadrant qd at qd * QX * QY)
// over the tile and its halo.  Tile pixels are added to the FP32 grid with
// one rounding (a two-sum of the grid value and hi, then hi + (err + lo));
// halo pixels are stored as FP64 hi + lo into the key's halo values hk.
// BLOCK threads, PER pixels per thread: BLOCK * PER >= (tile + hx) * (tile + hy).
template <int BLOCK, int PER>
__device__ __forceinline__ void quad_flush_tile(
  const float4* regions, int QX, int QY, int hx, int hy, const Geometry& geo,
  unsigned plane, int x0, int y0, float2* __restrict__ grid, double2* __restrict__ hk) {
  const int Q = QX * QY;
  const int RX = tile + hx;
  const int RY = tile + hy;
  const int R = RX * RY;
  // every pixel's value first, with the grid loads of the tile's pixels
  // issued together, then the stores
  float4 val[PER];
  float2 g0[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = int(threadIdx.x) + j * BLOCK;
    val[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    g0[j] = make_float2(0.0f, 0.0f);
    if (k >= R) continue;
    const int ry = k / RX;
    const int rx = k - ry * RX;
    // (hi, lo) of the pixel: the quadrants' pairs combined by two-sum
    float fr = 0.0f, fi = 0.0f, flr = 0.0f, fli = 0.0f;
    bool first = true;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const int ux = rx - (qd & 1) * quad_edge;
      const int uy = ry - (qd >> 1) * quad_edge;
      if (ux < 0 || uy < 0 || ux >= QX || uy >= QY) continue;
      const float4 a = regions[qd * Q + uy * QX + ux];
      if (first) {
        fr = a.x;
        fi = a.y;
        flr = a.z;
        fli = a.w;
      } else {
        float sum, err;
        two_sum(fr, a.x, sum, err);
        fr = sum;
        flr = flr + (err + a.z);
        two_sum(fi, a.y, sum, err);
        fi = sum;
        fli = fli + (err + a.w);
      }
      first = false;
    }
    val[j] = make_float4(fr, fi, flr, fli);
    const int xx = x0 + rx, yy = y0 + ry;
    if (rx < tile && ry < tile && xx < geo.nx && yy < geo.ny)
      g0[j] = grid[(size_t(plane) * geo.ny + yy) * geo.nx + xx];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = int(threadIdx.x) + j * BLOCK;
    if (k >= R) continue;
    const int ry = k / RX;
    const int rx = k - ry * RX;
    const float4 v = val[j];
    if (rx < tile && ry < tile) {
      const int xx = x0 + rx, yy = y0 + ry;
      if (xx >= geo.nx || yy >= geo.ny) continue;
      float sr, er, si, ei;
      two_sum(g0[j].x, v.x, sr, er);
      two_sum(g0[j].y, v.y, si, ei);
      grid[(size_t(plane) * geo.ny + yy) * geo.nx + xx] =
        make_float2(sr + (er + v.z), si + (ei + v.w));
    } else {
      const int h = ry < tile ? ry * hx + (rx - tile) : tile * hx + (ry - tile) * RX + rx;
      hk[h] = make_double2(double(v.x) + double(v.z), double(v.y) + double(v.w));
    }
  }
}

// ---- gridding: quadrant keys, two waves per quadrant, FP32 block sums ----
//
// k_sub grids FP32-compensated tiles for supports of at most 8 x 8 pixels
// from quadrant-keyed bins (k_bin with quad_keys: quadrant q of tile key t
// is bin key 4 t + q in every bin block).  The workgroup of a (plane, tile)
// has eight waves; waves q and q + 4 own quadrant q (the entries whose
// support corner lies in it) and take its entry list alternately, 64
// entries at a time: lane j locates, loads and prepares entry j of the
// batch (CF slices, region pixel, w-sign, flags).  The wave then adds the
// batch's entries one at a time, one lane per CF tap, to its own FP32
// region of (16 + hx) x (16 + hy) pixels in LDS by a plain read-modify-write
// (an entry's taps are distinct pixels, the region is the wave's own and a
// wave's LDS operations execute in order).  The batches run in rounds,
// in step across the workgroup (two halves of 32 slots, each followed by
// its entries with a phase gradient); after every sub_fold_rounds-th round
// and the last, every wave folds (between two barriers): wave q + 4 h holds
// the
// (hi, lo) pairs of half h of quadrant q's region pixels (lane l: pixels
// l + 64 k), adds both of the quadrant's regions' FP32 sums of those pixels
// to its pairs by two-sum and clears them.  So the products of a pixel are
// summed in FP32 over at most sub_fold entries of a region, those sums are
// accumulated with compensation, and a wave keeps the pairs of half a
// region in registers.  The flush sums the four quadrants' pairs over the
// tile and halo (quad_flush_tile), as k_tile4 does, and k_halo folds the halos.
constexpr int sub_waves = 8;
constexpr int sub_block = sub_waves * wave;
constexpr int sub_bins_max = 256;  // bin blocks per pass (LDS segment tables)
constexpr int sub_fold_rounds = 4; // rounds between folds
constexpr int sub_fold = 64 * sub_fold_rounds;  // entries of a region between folds
constexpr int sub_ring = 8;        // slots whose CF taps load ahead
constexpr int sub_flush = 3;       // tile + halo pixels per thread in the flush

// lane -> CF tap (X, Y) for supports up to 8 x 8: X = lane & 7, and the
// 8-lane groups take rows 0, 4, 1, 5, 2, 6, 3, 7, so that each 16 lanes
// read two rows 4 region rows apart
__device__ __forceinline__ int sub_lane_y(int lane) {
  const int g = lane >> 3;
  return (g >> 1) + 4 * (g & 1);
}

// PK (one polarization, CF of fewer than 2^21 taps): an entry's region
// pixel, w-sign and CF slice travel in one word, read once per slot
constexpr unsigned sub_pk_flip = 1u << 10;
constexpr int sub_pk_shift = 11;
constexpr size_t sub_pk_taps = size_t(1) << (32 - sub_pk_shift);

// exp(i phi) rounded to FP32 for an FP64 phase: phi is reduced to
// [-pi, pi] in FP64 (2 pi split into a 53-bit head and its tail, exact for
// the multiples used for |phi| < 2^20), then the FP32 sine and cosine of the
// remainder.  Within 2 ulp of fl32(cos phi), fl32(sin phi) (the reference's
// cphase in FP64, rounded) -- far inside the FP32-compensated grid's 1e-6.
__device__ __forceinline__ float2 screen_f32(double phi) {
  constexpr double two_pi_hi = 6.283185307179586;       // fl64(2 pi)
  constexpr double two_pi_lo = 2.4492935982947064e-16;  // 2 pi - fl64(2 pi)
  const double k = rint(phi * 0.15915494309189535);      // phi / (2 pi)
  const double r = (phi - k * two_pi_hi) - k * two_pi_lo;
  float sn, cs;
  __sincosf(float(r), &sn, &cs);
  return make_float2(cs, sn);
}

// an entry with a phase gradient: its CF taps times the phase screen
// exp(i phi(X, Y)) (FP64 phase as the reference's, screen_f32), added by
// one wave, one lane per tap, to the wave's FP32 region
__device__ __forceinline__ void sub_gradient_entry(
  unsigned w0, unsigned slice, float2 g, unsigned ri, unsigned pos,
  const Geometry& geo, const float2* __restrict__ taps, const VisRec<1>* __restrict__ recs,
  int QX, float2* region) {
  const int lane = int(threadIdx.x % wave);
  const int base = int(w0 & 4095u);
  const int sx = int((w0 >> 12) & 63u);
  const int sy = int((w0 >> 18) & 63u);
  const float imf = (w0 & quad_pos_w) ? -1.0f : 1.0f;
  const int fxi = int((pos >> 12) & 255u);
  const int fyi = int((pos >> 20) & 255u);
  const double gxr = recs[ri].grad[0];
  const double gyr = recs[ri].grad[1];
  const double phi0x = -gxr * ((sx / 2) * geo.os - (fxi - geo.F));
  const double phi0y = -gyr * ((sy / 2) * geo.os - (fyi - geo.F));
  const double dphix = gxr * geo.os;
  const double dphiy = gyr * geo.os;
  const int X = lane & 7, Y = sub_lane_y(lane);
  if (X >= sx || Y >= sy) return;
  const int tp = Y * sx + X;
  const float2 scr = screen_f32((phi0x + X * dphix) + (phi0y + Y * dphiy));
  float2 cc = taps[size_t(slice) + size_t(tp)];
  cc.y *= imf;
  const float2 pr = cmul(cmul(cc, scr), g);
  float2* a = region + base + Y * QX + X;
  float2 t = *a;
  t.x += pr.x;
  t.y += pr.y;
  *a = t;
}

// The entry lists of tile key tkey's four quadrant keys: seg_pref[q][b] =
// entries of quadrant q in the bin blocks before b (seg_pref[q][nbins] the
// quadrant's total), seg_beg[q][b] = its first entry within block b.  GB
// (global bins, grids of more keys than one workgroup's LDS histogram
// holds): off_table is the exclusive scan of the quadrant keys' entry
// counts, each key one contiguous range from gb_beg[q] (nbins = 1).  Ends
// with a barrier; the block has at least four waves.
template <int BLOCK, bool GB>
__device__ __forceinline__ void sub_tables(
  const unsigned* __restrict__ off_table, int nbins, unsigned ntk, unsigned tkey,
  unsigned (*seg_pref)[sub_bins_max + 1], unsigned short (*seg_beg)[sub_bins_max],
  unsigned* gb_beg) {
  const unsigned tid = threadIdx.x;
  if constexpr (GB) {
    if (tid < 4) {
      const unsigned s0 = off_table[4 * size_t(tkey) + tid];
      const unsigned s1 = off_table[4 * size_t(tkey) + tid + 1];
      gb_beg[tid] = s0;
      seg_pref[tid][0] = 0u;
      seg_pref[tid][1] = s1 - s0;
    }
    __syncthreads();
  } else {
    // segment tables of the four quadrant keys, then their exclusive scans
    const size_t row = size_t(4) * ntk + 1;  // offset-table row
    for (int i = int(tid); i < 4 * nbins; i += BLOCK) {
      const int bb = i >> 2, qq = i & 3;
      const unsigned* tab = off_table + size_t(bb) * row + 4 * size_t(tkey) + qq;
      const unsigned s0 = tab[0], s1 = tab[1];
      seg_pref[qq][bb] = s1 - s0;
      seg_beg[qq][bb] = (unsigned short)s0;
    }
    __syncthreads();
    const int w = int(tid) / wave;
    const int lane = int(tid) % wave;
    if (w < 4) {
      unsigned* a = seg_pref[w];
      unsigned v[4];
      unsigned sum = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int idx = lane * 4 + k;
        v[k] = idx < nbins ? a[idx] : 0u;
        sum += v[k];
      }
      unsigned incl = sum;
#pragma unroll
      for (int d = 1; d < wave; d <<= 1) {
        const unsigned t = __shfl_up(incl, d, wave);
        if (lane >= d) incl += t;
      }
      unsigned run = incl - sum;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int idx = lane * 4 + k;
        if (idx < nbins) a[idx] = run;
        run += v[k];
      }
      if (lane == wave - 1) a[nbins] = incl;
    }
    __syncthreads();
  }
}

// entry i of quadrant q's list (sub_tables): its index in the entry array
template <bool GB>
__device__ __forceinline__ unsigned sub_locate(
  unsigned i, int q, int nbins, size_t block_cap, const unsigned (*seg_pref)[sub_bins_max + 1],
  const unsigned short (*seg_beg)[sub_bins_max], const unsigned* gb_beg) {
  if constexpr (GB) return gb_beg[q] + i;
  int lo = 0, hi = nbins;  // seg_pref[q][lo] <= i < seg_pref[q][hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (seg_pref[q][mid] <= i) lo = mid; else hi = mid;
  }
  return unsigned(lo) * unsigned(block_cap) + seg_beg[q][lo] + (i - seg_pref[q][lo]);
}

// PX: region pixels per lane; each wave's region is padded to PX * 64
// pixels (>= (16 + hx) * (16 + hy)), so a lane folds pixels lane + 64 k with
// no bounds test.  UNI: every CF group has the same support, whose lane mask
// then holds for the whole call.  PK: see sub_pk_flip.  GB: global bins
// (sub_tables).
template <int PX, bool UNI, bool PK, bool GB>
__global__ __launch_bounds__(sub_block) __attribute__((amdgpu_waves_per_eu(8)))
void k_sub(
  Geometry geo, const GroupInfo* __restrict__ groups, const float2* __restrict__ taps,
  unsigned taps_bytes, Mueller mu, const unsigned* __restrict__ off_table, int nbins,
  size_t block_cap,
  const Entry4* __restrict__ entries, const unsigned* __restrict__ entry_vis,
  const VisRec<1>* __restrict__ recs, int hx, int hy, float2* __restrict__ grid,
  double2* __restrict__ halo, unsigned* __restrict__ halo_set) {
  // eight FP32 regions of QP = PX * 64 pixels (float2); in the flush the
  // same bytes hold the four quadrants' (hi, lo) pairs (float4, Q each)
  extern __shared__ float2 sregions[];
  __shared__ unsigned seg_pref[4][sub_bins_max + 1];
  __shared__ unsigned short seg_beg[4][sub_bins_max];
  __shared__ unsigned gb_beg[4];  // GB: first entry of each quadrant key
  constexpr int QP = PX * wave;

  const int QX = quad_edge + hx;
  const int QY = quad_edge + hy;
  const int Q = QX * QY;
  const unsigned ntk = unsigned(geo.ntx) * geo.nty * geo.nr * geo.nc;
  const unsigned tkey = xcd_key(blockIdx.x, gridDim.x);  // one block per tile key
  const unsigned tid = threadIdx.x;
  const int w = int(tid) / wave;
  const int lane = int(tid) % wave;
  const int q = w & 3;
  const int half = w >> 2;

  sub_tables<sub_block, GB>(off_table, nbins, ntk, tkey, seg_pref, seg_beg, gb_beg);
  if (seg_pref[0][nbins] + seg_pref[1][nbins] + seg_pref[2][nbins] + seg_pref[3][nbins] == 0u) {
    if (tid == 0) halo_set[tkey] = 0u;
    return;
  }

  const unsigned ntiles = unsigned(geo.ntx) * geo.nty;
  const unsigned plane = tkey / ntiles;
  const int t = int(tkey % ntiles);
  const int x0 = (t % geo.ntx) * tile;
  const int y0 = (t / geo.ntx) * tile;
  const int gpol = int(plane % geo.nr);
  const int qx = q & 1, qy = q >> 1;

  float2* region = sregions + size_t(w) * QP;
#pragma unroll
  for (int k = 0; k < PX; ++k) region[lane + k * wave] = make_float2(0.0f, 0.0f);
  // the (hi, lo) pairs of this wave's share of its quadrant's pixels: wave
  // half 0 holds pixels lane + 64 k for k < PXA, half 1 the rest
  constexpr int PXA = (PX + 1) / 2;
  const int k0 = half ? PXA : 0;
  const int nk = half ? PX - PXA : PXA;
  float4 acc[PXA];
#pragma unroll
  for (int k = 0; k < PXA; ++k) acc[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float2* reg_a = sregions + size_t(q) * QP;      // the quadrant's two regions
  const float2* reg_b = sregions + size_t(q + 4) * QP;
  // the FP32 sums of both regions' pixels of this wave's share into its
  // (hi, lo) pairs, by two-sum, clearing the pixels (all waves at once,
  // between barriers)
  auto fold = [&]() {
#pragma unroll
    for (int k = 0; k < PXA; ++k) {
      if (PX % 2 == 1 && k >= nk) continue;
      const int px = lane + (k0 + k) * wave;
      const float2 pa = reg_a[px];
      const float2 pb = reg_b[px];
      const_cast<float2*>(reg_a)[px] = make_float2(0.0f, 0.0f);
      const_cast<float2*>(reg_b)[px] = make_float2(0.0f, 0.0f);
      float sum, err;
      two_sum(acc[k].x, pa.x, sum, err);
      acc[k].x = sum;
      acc[k].z += err;
      two_sum(acc[k].y, pa.y, sum, err);
      acc[k].y = sum;
      acc[k].w += err;
      two_sum(acc[k].x, pb.x, sum, err);
      acc[k].x = sum;
      acc[k].z += err;
      two_sum(acc[k].y, pb.y, sum, err);
      acc[k].y = sum;
      acc[k].w += err;
    }
  };

  const bool one_group = geo.ngroups == 1;
  const GroupInfo group0 = groups[0];
  // this plane's Mueller elements for both signs of w
  const int row_m = mu.M[gpol][0], row_mc = mu.Mc[gpol][0];
  // the quadrant's list, taken by its two waves alternately 64 entries at
  // a time (fewer partly filled batches than an even split, whose per-batch
  // costs outweigh its balance)
  const unsigned total = seg_pref[q][nbins];
  auto locate = [&](unsigned i) {
    return sub_locate<GB>(i, q, nbins, block_cap, seg_pref, seg_beg, gb_beg);
  };
  const int lane_x = lane & 7;
  const int lane_y = sub_lane_y(lane);
  // LDS byte offset of this lane's tap pixel in the wave's region, relative
  // to an entry's support corner
  const unsigned lane_addr =
    unsigned((size_t(w) * QP + size_t(lane_y * QX + lane_x)) * sizeof(float2));
  // CF taps through a buffer resource: the slice's byte offset goes in a
  // scalar register and the lane's tap offset in a 32-bit vector register;
  // reads past taps_bytes return 0
  const __amdgpu_buffer_rsrc_t tap_rsrc = __builtin_amdgcn_make_buffer_rsrc(
    const_cast<float2*>(taps), 0, int(taps_bytes), 0x00020000);
  // lanes holding a tap of a support (sx, sy), and their tap byte offset
  auto support_lanes = [&](int sx, int sy, unsigned& off) {
    const bool ok = lane_x < sx && lane_y < sy;
    off = unsigned(ok ? lane_y * sx + lane_x : 0) * unsigned(sizeof(float2));
    return ok;
  };
  unsigned tap_off = 0;
  const bool uni_ok = UNI ? support_lanes(group0.sx, group0.sy, tap_off) : true;
  int tap_key = -1;
  unsigned long long tap_lanes = 0ull;

  // rounds: in round r, wave half h takes batch 2 r + h of its quadrant's
  // list; all eight waves run every round (the folds are shared)
  const unsigned tq[4] = {seg_pref[0][nbins], seg_pref[1][nbins], seg_pref[2][nbins],
                          seg_pref[3][nbins]};
  const unsigned tmax = max(max(tq[0], tq[1]), max(tq[2], tq[3]));
  const unsigned nrounds = (tmax + 2u * wave - 1u) / (2u * wave);
  for (unsigned rd = 0; rd < nrounds; ++rd) {
    const unsigned b0 = (2u * rd + unsigned(half)) * wave;
    // entries in the round's largest batch over the workgroup (uniform)
    unsigned rmax = 0;
#pragma unroll
    for (int qq = 0; qq < 4; ++qq)
#pragma unroll
      for (unsigned hh = 0; hh < 2; ++hh) {
        const unsigned bb = (2u * rd + hh) * wave;
        rmax = max(rmax, tq[qq] > bb ? min(unsigned(wave), tq[qq] - bb) : 0u);
      }
    // lane j: entry b0 + j of the quadrant's list, prepared.  Slots that
    // add nothing here (past the list, phase gradient, no CF index) keep
    // zero values and the region's first pixel, and read a valid CF slice.
    const unsigned i = b0 + unsigned(lane);
    const bool valid = i < total;
    unsigned ei = 0;
    Entry4 e{};
    if (valid) {
      ei = locate(i);
      e = entries[ei];
    }
    // p_addr: the entry's LDS byte offset from the region origin, with the
    // w-sign flip (bit 31: conj(c) for w > 0) -- 0 for slots that add
    // nothing.  PK: the region pixel | sub_pk_flip | slice << sub_pk_shift
    unsigned p_addr = 0, p_key = 0;
    unsigned p_sl = 0u;
    float p_gx = 0.0f, p_gy = 0.0f;
    bool grad = false, normal = false;
    if (valid) {
      const unsigned pos = e.h.pos;
      const int lx = int(pos & 63u);
      const int ly = int((pos >> 6) & 63u);
      const int fxi = int((pos >> 12) & 255u);
      const int fyi = int((pos >> 20) & 255u);
      const bool pos_w = pos & e4_pos_w;
      grad = pos & e4_gradient;
      const int grp = int(e.h.gpk & 0xffffu);
      const int cfcube = int(e.h.gpk >> 16);
      const GroupInfo g = one_group ? group0 : groups[grp];
      const int m = pos_w ? row_m : row_mc;
      const bool use = m >= 0 && m < g.nmueller;
      p_sl = unsigned(plane_start(g, geo.nf, cfcube, use ? m : 0, fxi, fyi));
      if (use && !grad) {
        p_gx = e.g.x;
        p_gy = e.g.y;
      }
      const unsigned base = unsigned((ly - qy * quad_edge) * QX + (lx - qx * quad_edge));
      p_key = unsigned(g.sx) | (unsigned(g.sy) << 6);
      normal = !grad && use;
      if constexpr (PK) {
        p_addr = (p_sl << sub_pk_shift) | (normal ? base | (pos_w ? sub_pk_flip : 0u) : 0u);
      } else {
        if (normal) p_addr = base * unsigned(sizeof(float2)) | (pos_w ? 0x80000000u : 0u);
      }
      grad = grad && use;
    }
    const unsigned long long nmask = __ballot(normal);
    const unsigned long long gtodo = __ballot(valid && grad);
    // slots up to the last entry added here
    const int nslots = nmask ? 64 - __builtin_clzll(nmask) : 0;

    // CF taps of slot j: loaded sub_ring slots ahead into ring[j % sub_ring]
    // (the fetches run on the whole wave: a lane's prepared values are read
    // from it while it is active); the slot's other values are read from
    // its lane when it is added
    float2 ring[sub_ring];
    unsigned ring_pk[sub_ring];               // PK: the slot's word
    unsigned long long ring_lanes[sub_ring];  // !UNI: lanes of the slot's support
    auto fetch = [&](int j) {
      const int r = j % sub_ring;
      if constexpr (!UNI) {
        const int key_s = __builtin_amdgcn_readlane(int(p_key), j);
        if (key_s != tap_key) {
          tap_key = key_s;
          tap_lanes = __ballot(support_lanes(key_s & 63, key_s >> 6, tap_off));
        }
        ring_lanes[r] = tap_lanes;
      }
      if constexpr (PK) {
        const unsigned pk = unsigned(__builtin_amdgcn_readlane(int(p_addr), j));
        ring_pk[r] = pk;
        const v2i_t raw = __builtin_amdgcn_raw_buffer_load_b64(
          tap_rsrc, int(tap_off), int((pk >> sub_pk_shift) * unsigned(sizeof(float2))), 0);
        ring[r] = make_float2(__int_as_float(raw.x), __int_as_float(raw.y));
      } else {
        const int slv = __builtin_amdgcn_readlane(int(p_sl), j);
        const v2i_t raw = __builtin_amdgcn_raw_buffer_load_b64(
          tap_rsrc, int(tap_off), slv * int(sizeof(float2)), 0);
        ring[r] = make_float2(__int_as_float(raw.x), __int_as_float(raw.y));
      }
    };
    auto add = [&](int j) {
      const int r = j % sub_ring;
      unsigned flip, addr;
      if constexpr (PK) {
        const unsigned pk = ring_pk[r];
        flip = (pk << (31 - 10)) & 0x80000000u;
        addr = (pk & (sub_pk_flip - 1u)) * unsigned(sizeof(float2));
      } else {
        const unsigned aw = unsigned(__builtin_amdgcn_readlane(int(p_addr), j));
        flip = aw & 0x80000000u;
        addr = aw & 0x7fffffffu;
      }
      // UNI: the slot loops run on the support's lanes only
      bool on;
      if constexpr (UNI) on = true; else on = __builtin_amdgcn_inverse_ballot_w64(ring_lanes[r]);
      const unsigned ux = unsigned(__builtin_amdgcn_readlane(__float_as_int(p_gx), j));
      const unsigned uy = unsigned(__builtin_amdgcn_readlane(__float_as_int(p_gy), j));
      const float gx = __uint_as_float(ux), gy = __uint_as_float(uy);
      // conj(c) g for w > 0: c.y g.y and c.y g.x enter with the sign flipped
      const float gcx = __uint_as_float(uy ^ flip), gcy = __uint_as_float(ux ^ flip);
      // the FP32 complex product, each part as one product and one fused
      // multiply-add
      const float2 c = ring[r];
      const float pr = __builtin_fmaf(c.x, gx, -(c.y * gcx));
      const float pi = __builtin_fmaf(c.x, gy, c.y * gcy);
      if (on) {
        float2* a =
          reinterpret_cast<float2*>(reinterpret_cast<char*>(sregions) + addr + lane_addr);
        float2 tv = *a;
        tv.x += pr;
        tv.y += pi;
        *a = tv;
      }
    };
    // two halves of 32 slots, each followed by the half's entries with a
    // phase gradient; the shared fold after the last half of every
    // sub_fold_rounds-th round and of the last, so at most sub_fold entries
    // reach a region between folds.  A half without entries in any wave of
    // the workgroup is skipped
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      if (unsigned(hb * 32) >= rmax) continue;
      if (hb * 32 < nslots && uni_ok) {
#pragma unroll
        for (int j = 0; j < sub_ring; ++j) fetch(hb * 32 + j);
#pragma unroll
        for (int j = 0; j < 32; ++j) {
          add(hb * 32 + j);
          if (j + sub_ring < 32) fetch(hb * 32 + j + sub_ring);
        }
      }
      unsigned long long gl = gtodo & (hb ? 0xffffffff00000000ull : 0xffffffffull);
      const bool last_half = hb == 1 || 32u >= rmax;
      while (gl) {
        const int j = __builtin_ctzll(gl);
        gl &= gl - 1ull;
        // the entry again (a scalar load), so that the batch's raw entries
        // need not stay in registers through the loop above
        const unsigned ej = unsigned(__builtin_amdgcn_readlane(int(ei), j));
        const Entry4 ge = entries[ej];
        const unsigned gpos = ge.h.pos;
        const bool gpos_w = gpos & e4_pos_w;
        const GroupInfo gg = one_group ? group0 : groups[ge.h.gpk & 0xffffu];
        const unsigned sl =
          PK ? unsigned(__builtin_amdgcn_readlane(int(p_addr), j)) >> sub_pk_shift
             : unsigned(__builtin_amdgcn_readlane(int(p_sl), j));
        const unsigned gbase = ((gpos >> 6) & 63u) - unsigned(qy * quad_edge);
        const unsigned w0 = (gbase * unsigned(QX) + ((gpos & 63u) - unsigned(qx * quad_edge)))
          | (unsigned(gg.sx) << 12) | (unsigned(gg.sy) << 18)
          | (gpos_w ? quad_pos_w : 0u);
        sub_gradient_entry(w0, sl, ge.g, entry_vis[ej], ge.h.pos, geo, taps, recs, QX, region);
      }
      if (last_half && ((rd + 1u) % unsigned(sub_fold_rounds) == 0u || rd + 1u == nrounds)) {
        __syncthreads();
        fold();
        __syncthreads();
      }
    }
  }

  // each wave's pairs into LDS (the regions are no longer read), then flush
  float4* pairs = reinterpret_cast<float4*>(sregions);
#pragma unroll
  for (int k = 0; k < PXA; ++k) {
    if (PX % 2 == 1 && k >= nk) continue;
    const int px = lane + (k0 + k) * wave;
    if (px < Q) pairs[q * Q + px] = acc[k];
  }
  __syncthreads();
  quad_flush_tile<sub_block, sub_flush>(pairs, QX, QY, hx, hy, geo, plane, x0, y0, grid,
                                        halo + size_t(tkey) * halo_pixels(hx, hy));
  if (tid == 0) halo_set[tkey] = 1u;
}

// ---- gridding: pixel patches in registers -----------------------------------
//
// The gridder of several polarizations, and of supports beyond the other
// tile kernels'.  One workgroup owns a tile of all grid rows of one cube and
// keeps its pixels' FP64 sums in registers, so a tap costs no LDS or global
// atomic: a lane is a (pixel, grid row), a wave holds 2 x 2 patches of 64 / P
// pixels (P = lanes per pixel: 1, 2 or 4 rows), the workgroup 2 x 2 waves, or
// twice that, two waves sharing the entries of the same pixels (patch_split).
//
//   k_patch_prep  one thread per visibility: skip rule, weights, the record's
//                 prepared form (support corner, CF slice, pre-phased values)
//                 and the counts of the tiles it touches
//   k_patch_scan  the tiles' list offsets and their order (many tiles: hipCUB's
//                 scan, in grid order)
//   k_patch_list  one thread per visibility: its index into the lists of the
//                 tiles it touches
//   k_patch       one workgroup per tile: 256 list entries at a time staged in
//                 LDS; each wave tests them 64 at a time against its own
//                 pixels, and adds those that overlap one by one
//
// A slice holds its Mueller elements side by side, so the 64 lanes of a patch
// read whole runs of it (4 x 128 bytes for 16 elements), each CF byte once
// per record whatever the tile borders cut; lanes outside the support read
// past the buffer resource's end, which fetches nothing.  Small patches keep
// the lanes busy: a support S wide fills (S / (S + 3))^2 of the 4 x 4 patches
// it touches, 72% at S = 17.
//
// Bound: the CF reads from HBM for large CFs (64 groups of supports 9-65, 16
// elements, 500,000 records: 104 GB in 19.5 ms, 5.3 TB/s, against 27.7 ms for
// clipped tiles in LDS, one workgroup per plane and element-major slices;
// supports 17-129, 150,000 records: 119 GB in 19.2 ms, before 38.4 ms), vector
// issue for CFs that stay in the last-level cache (supports 9-25, 200,000
// records: 1.00 ms, before 4.31 ms by LDS compare-and-swap). Loading the next
// one to three entries' CF values ahead of their turn gained nothing there and
// cost the small supports 10%: the waves cover the loads.

// lanes per pixel for nr grid rows
constexpr int patch_lanes(int nr) { return nr <= 1 ? 1 : nr == 2 ? 2 : 4; }
// pixels of a patch, of a wave's 2 x 2 patches and of a tile along x and y
__host__ __device__ constexpr int patch_w(int P) { return P == 4 ? 4 : 8; }
__host__ __device__ constexpr int patch_h(int P) { return P == 1 ? 8 : 4; }
__host__ __device__ constexpr int patch_tile_x(int P) { return 4 * patch_w(P); }
__host__ __device__ constexpr int patch_tile_y(int P) { return 4 * patch_h(P); }
constexpr int patch_block = 4 * wave;
// waves that share the entries of the same pixels: a tile's entries run one
// after the other, so the fullest tile of a dense uv core sets the kernel's
// length. Two where a tile is 16 pixels wide (four rows: 300,000 records on
// 1024^2 1.58 -> 0.97 ms, the large CFs 2 to 5% less), four gained no more; one
// for the wider tiles, whose entries are cheap (two rows: 244 us against 312).
__host__ __device__ constexpr int patch_split(int P) { return P == 4 ? 2 : 1; }

// a record prepared for its tiles; sxy = 0: not gridded.  The support's extents
// (odd, below 2^30) are split: their lower 16 bits in sxy, and what is left of
// them above the 36 bits of an index of 8-byte values in 512 GB, which keeps the
// record at 64 bytes (two more words would cost a quarter of the staged records'
// LDS, and in DegridRec a register in the loop over the taps)
template <int N>
struct __align__(16) PatchRec {
  int gx, gy;               // support corner
  unsigned long long base;  // first value of its CF slice (element 0, tap 0)
                            // | sx >> 16 << 36 | sy >> 16 << 50
  unsigned sxy;             // low 16 bits of sx | sy << 16
  unsigned fl;              // flags | fxi << 8 | fyi << 16
  unsigned nm;              // Mueller elements of its CF group
  unsigned cube;            // grid cube
  float2 g[N];
};
static_assert(sizeof(PatchRec<1>) == 48 && sizeof(PatchRec<4>) == 64, "PatchRec layout");
// the slice's index, taken apart and made (also of DegridRec)
constexpr unsigned patch_base_hi = 0xfu;  // its bits of the upper word
__device__ __forceinline__ void patch_pack(
  long long slice, int sx, int sy, unsigned long long& base, unsigned& sxy) {
  base = (unsigned long long)slice | ((unsigned long long)(unsigned(sx) >> 16) << 36)
    | ((unsigned long long)(unsigned(sy) >> 16) << 50);
  sxy = (unsigned(sx) & 0xffffu) | (unsigned(sy) << 16);
}
__device__ __forceinline__ int patch_sx(unsigned sxy, unsigned base_hi) {
  return int((sxy & 0xffffu) | ((base_hi << 12) & 0x3fff0000u));
}
__device__ __forceinline__ int patch_sy(unsigned sxy, unsigned base_hi) {
  return int((sxy >> 16) | ((base_hi >> 2) & 0x3fff0000u));
}
// of a uniform record: supports of 65536 pixels and more by a branch, whose
// instructions would lengthen the loops' scalar chains (228 -> 231 us, two
// polarizations, 300,000 records)
__device__ __forceinline__ void patch_unpack(
  unsigned sxy, unsigned& base_hi, int& sx, int& sy) {
  sx = int(sxy & 0xffffu);
  sy = int(sxy >> 16);
  if (__builtin_expect(base_hi > patch_base_hi, 0)) {
    asm volatile("");  // kept a branch
    sx = patch_sx(sxy, base_hi);
    sy = patch_sy(sxy, base_hi);
    base_hi &= patch_base_hi;
  }
}

// record i, whose support at c is inside the grid, prepared (sxy = 0 and
// false: no row takes it), and its weight in each grid row
template <int N>
__device__ __forceinline__ bool patch_record(
  const VisRec<N>& r, size_t i, const Coord& c, const Geometry& geo, const GroupInfo& g,
  const double2* __restrict__ wsum, const Mueller& mu, int update_weights, int gvis_ready,
  int adjoint, const float2* __restrict__ gvis_in, const double2* __restrict__ residuals,
  PatchRec<N>& e, double (&tw4)[4]) {
  const bool pos_w = r.uvw[2] > 0;
  const unsigned cfcube = r.cf_index[0];
  const int fxi = c.fx + geo.F, fyi = c.fy + geo.F;
  bool any = false;
#pragma unroll
  for (int gp = 0; gp < 4; ++gp) {
    tw4[gp] = 0.0;
    if (gp >= geo.nr) continue;
    double t = 0.0;
#pragma unroll
    for (int v = 0; v < N; ++v) {
      const int m = pos_w ? mu.M[gp][v] : mu.Mc[gp][v];
      any |= m >= 0;
      if (update_weights && m >= 0 && m < g.nmueller) {
        const double2 sw = wsum[g.wsum_offset
                                + ((long long)(cfcube * g.nmueller + m) * geo.nf + fxi) * geo.nf
                                + fyi];
        t += hypot(sw.x, sw.y) * double(r.w[v]);
      }
    }
    tw4[gp] = t;
  }
  e.sxy = 0u;
  if (!any) return false;
  const bool grad = r.grad[0] != 0.0 || r.grad[1] != 0.0;
  e.gx = c.gx;
  e.gy = c.gy;
  patch_pack(slice_start(g, geo.nf, int(cfcube), fxi, fyi), g.sx, g.sy, e.base, e.sxy);
  e.fl = unsigned((pos_w ? flag_pos_w : 0) | (grad ? flag_gradient : 0)) | (unsigned(fxi) << 8)
    | (unsigned(fyi) << 16);
  e.nm = unsigned(g.nmueller);
  e.cube = r.grid_cube;
  if (gvis_ready) {
    for (int v = 0; v < N; ++v) e.g[v] = gvis_in[i * N + v];
  } else {
    const double2 phasor = cphase(r.phase);
    if (!adjoint) {
      for (int v = 0; v < N; ++v) e.g[v] = prephase(r.vis[v], phasor, r.w[v]);
    } else {
      double2 W[N];
      degrid_norms<N>(geo, g, wsum, mu, pos_w, cfcube, fxi, fyi, W);
      for (int v = 0; v < N; ++v) {
        double2 d = W[v];
        if (d.x == 0.0 && d.y == 0.0) d = make_double2(1.0, 0.0);
        d.y = -d.y;
        e.g[v] = narrow(kdiv(cmul(residuals[i * N + v], phasor), d));
      }
    }
  }
  return true;
}

// For tiles of at most patch_scan_keys: the exclusive scan of their counts, and
// their order by falling count class, so that the tiles of a dense uv core
// start first: in grid order they came in the middle, and the chip waited for
// them (200,000 records, supports 9-25: 1172 -> 1071 us, two polarizations,
// 7-17: 280 -> 244 us).  One workgroup, 11 us for 4096 tiles and 19 us for 8836,
// in place of hipCUB's scan (10 us).  order null: the scan alone.
//
// A list of two chunks or more (patch_full_chip) is split: one workgroup for each
// chunk of it, in slots next to each other (the last of a tile's to end adds up their
// sums in the slots' order), or a dense uv core would be one workgroup's serial chain.  The
// chunk is the least, from patch_chunk_min on, that leaves the launch enough slots:
// a list of two chunks or more has 1.5 slots a chunk of its entries at most.
// Two polarizations, FP64: 100,000 records of supports 5 within a few pixels 28.5 ->
// 0.41 ms (1.8 by haloed LDS tiles), 200,000 on 128^2, supports 3, 2.38 -> 0.21
// (0.37), 10,000 on 256^2 104 -> 91 us (75); least chunks of 16 and 64 are 5 and 4%
// slower there.  With a fence of the device's scope instead of stores past the L2s
// 116 us: it writes a whole L2 back for every chunk.
constexpr unsigned patch_chunk_min = 32;
// Even lists of tiles that fill the chip by themselves, two workgroups a CU and more,
// would only pay for the chunks' sums: where a quarter of the tiles are over the mean,
// lists of 1.5 times the mean and more are split (30,000 records: 384^2, four
// polarizations, FP32, 576 tiles 173 us split, 149 not; 512^2, two, 512 tiles 99, 88;
// 100,000 of a Gaussian core there stay split, 135 us for 197).
constexpr unsigned patch_full_chip = 512;
constexpr unsigned patch_none = ~0u;  // in the tiles' order: a split one
constexpr int patch_values = 8 * patch_block;
// device scope: past the XCDs' own L2s
__device__ __forceinline__ void patch_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double patch_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
struct PatchSplit {
  unsigned slots;  // of the launch; 0: no list is split
  char* base;
  // slots taken, chunk
  __host__ __device__ unsigned* ctl() const { return reinterpret_cast<unsigned*>(base); }
  // a slot's patch_values sums
  __device__ double* sums(unsigned slot) const {
    return reinterpret_cast<double*>(base + 256) + size_t(slot) * patch_values;
  }
  // (tile, chunk's number) of every slot
  __device__ uint2* items() const { return reinterpret_cast<uint2*>(sums(slots)); }
  // of a tile's first slot, for each of two k_patch launches
  __device__ unsigned* tickets() const { return reinterpret_cast<unsigned*>(items() + slots); }
};
__device__ __forceinline__ unsigned patch_chunk(unsigned total, unsigned slots) {
  return max(patch_chunk_min, unsigned(1.5 * double(total) / double(slots)) + 1u);
}
// the slots of a tile whose list has cnt entries, taken from *taken
__device__ __forceinline__ void patch_take(
  const PatchSplit& ps, unsigned chunk, unsigned key, unsigned cnt, unsigned* taken, int scope) {
  const unsigned m = (cnt + chunk - 1u) / chunk;
  const unsigned at = scope == __HIP_MEMORY_SCOPE_WORKGROUP
    ? __hip_atomic_fetch_add(taken, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)
    : atomicAdd(taken, m);
  ps.tickets()[at] = ps.tickets()[ps.slots + at] = 0u;
  for (unsigned i = 0; i < m; ++i) ps.items()[at + i] = make_uint2(key, i);
}
// the same for more tiles than k_patch_scan takes, and their order, as they come
__global__ __launch_bounds__(block) void k_patch_split(
  size_t keys, const unsigned* __restrict__ offsets, unsigned* __restrict__ order,
  PatchSplit ps) {
  const size_t k = blockIdx.x * (size_t)block + threadIdx.x;
  if (k >= keys) return;
  const unsigned chunk = patch_chunk(offsets[keys], ps.slots);
  if (k == 0) ps.ctl()[1] = chunk;
  const unsigned cnt = offsets[k + 1] - offsets[k];
  const bool split = cnt >= 2u * chunk;
  order[k] = split ? patch_none : unsigned(k);
  if (split)
    patch_take(ps, chunk, unsigned(k), cnt, ps.ctl(), __HIP_MEMORY_SCOPE_AGENT);
}

constexpr int patch_scan_threads = 1024;
constexpr int patch_scan_keys = patch_local_keys;
constexpr int patch_classes = 6;
// a: the counts in LDS, keys + 1 values, afterwards the offsets
__device__ __forceinline__ void patch_scan(
  int keys, unsigned* a, unsigned* __restrict__ offsets, unsigned* __restrict__ order,
  const PatchSplit& ps) {
  __shared__ unsigned part[patch_scan_threads / wave + 1];
  __shared__ unsigned cls[patch_classes];
  __shared__ unsigned taken;
  if (threadIdx.x == 0) taken = 0u;
  if (threadIdx.x < patch_classes) cls[threadIdx.x] = 0u;
  __syncthreads();
  const unsigned total = block_exclusive_scan(a, keys, part);
  if (threadIdx.x == 0) a[keys] = total;
  __syncthreads();
  if (!order) {
    for (int k = threadIdx.x; k <= keys; k += patch_scan_threads) offsets[k] = a[k];
    return;
  }
  const int lane = threadIdx.x % wave;
  const int rounds = (keys + patch_scan_threads - 1) / patch_scan_threads;
  const unsigned chunk = ps.slots ? patch_chunk(total, ps.slots) : 0u;
  __shared__ unsigned least;  // the shortest list that is split
  // class 0: over four times the mean, 2: over the mean, ..., the last: empty
  auto class_of = [&](int k) {
    const unsigned cnt = a[k + 1] - a[k];
    const unsigned long long c = (unsigned long long)cnt * unsigned(keys);
    return c > 4ull * total ? 0u : c > 2ull * total ? 1u : c > total ? 2u
      : 4ull * c > total ? 3u : c ? 4u : 5u;
  };
  static_assert(patch_scan_keys <= 16 * patch_scan_threads, "four bits a round in classes");
  unsigned long long classes = 0;  // of this thread's tiles, from the first pass
  for (int pass = 0; pass < 2; ++pass) {
    for (int r = 0; r < rounds; ++r) {
      const int k = r * patch_scan_threads + int(threadIdx.x);
      unsigned q = ~0u;
      if (k < keys) {
        if (pass == 0) {
          q = class_of(k);
          classes |= (unsigned long long)q << (4 * r);
          offsets[k] = a[k];
        } else {
          q = unsigned(classes >> (4 * r)) & 15u;
        }
      }
#pragma unroll
      for (int c = 0; c < patch_classes; ++c) {
        const bool mine = q == unsigned(c);
        const unsigned long long m = __ballot(mine);
        if (!m) continue;
        const int lead = __builtin_ctzll(m);
        unsigned at = 0;
        if (lane == lead)
          at = __hip_atomic_fetch_add(cls + c, unsigned(__builtin_popcountll(m)),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        at = unsigned(__builtin_amdgcn_readlane(int(at), lead));
        if (pass == 1 && mine) {
          const unsigned cnt = a[k + 1] - a[k];
          const bool split = cnt >= least;
          order[at + unsigned(__builtin_popcountll(m & ((1ull << lane) - 1ull)))] =
            split ? patch_none : unsigned(k);
          if (split)
            patch_take(ps, chunk, unsigned(k), cnt, &taken,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
    __syncthreads();
    if (pass == 0 && threadIdx.x == 0) {
      unsigned run = 0;
      for (int c = 0; c < patch_classes; ++c) {
        const unsigned t = cls[c];
        cls[c] = run;
        run += t;
      }
      const bool even = unsigned(keys) >= patch_full_chip && 4u * cls[3] >= unsigned(keys);
      least = !ps.slots ? ~0u
        : max(2u * chunk, even ? unsigned(3ull * total / (2ull * unsigned(keys))) + 1u : 0u);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    offsets[keys] = total;
    if (ps.slots) {
      ps.ctl()[0] = taken;
      ps.ctl()[1] = chunk;
    }
  }
}
__global__ __launch_bounds__(patch_scan_threads) void k_patch_scan(
  int keys, const unsigned* __restrict__ hist, unsigned* __restrict__ offsets,
  unsigned* __restrict__ order, PatchSplit ps) {
  __shared__ unsigned a[patch_scan_keys + 1];
  for (int k = threadIdx.x; k < keys; k += patch_scan_threads) a[k] = hist[k];
  patch_scan(keys, a, offsets, order, ps);
}

// f(tile) for the tiles that a prepared record touches
template <int N, typename F>
__device__ __forceinline__ void patch_tiles(
  const PatchRec<N>& e, int pty, int ptx, int tw, int th, F f) {
  const unsigned sxy = e.sxy;
  if (!sxy) return;
  const int gx = e.gx, gy = e.gy;
  const unsigned bhi = unsigned(e.base >> 32);
  const int tx0 = gx / tw, tx1 = (gx + patch_sx(sxy, bhi) - 1) / tw;
  const int ty0 = gy / th, ty1 = (gy + patch_sy(sxy, bhi) - 1) / th;
  const int cube = int(e.cube) * pty;
  for (int ty = ty0; ty <= ty1; ++ty)
    for (int tx = tx0; tx <= tx1; ++tx) f((cube + ty) * ptx + tx);
}

// Weights: each wave sums its records' weights per (grid cube, row), and
// for grids of at most count_planes_lds planes adds the sums into the
// workgroup's LDS, which adds into the grid weights once at its end (the
// workgroups stride over the records, so a few thousand global atomics per
// plane instead of one per wave).
// LOCAL (at most patch_local_keys tiles): the workgroup, of `batch` records in a
// row, counts its tiles in LDS, adds its counts to hist once per tile, and
// keeps each tile's place for it in its row of `table`, so that k_patch_list
// places the entries without global atomics (10 G/s over the chip: they were
// all of the two kernels' time: 284 + 265 us for 300,000 records of supports 9-33
// on 4096 tiles, now 48 + 19).  A single workgroup (patch_batch) does the scan and
// the lists too (offsets not null), three launches fewer: 300 records of two
// polarizations 70 -> 64 us with the call's end waited for.
template <int N, bool LOCAL>
__global__ __launch_bounds__(LOCAL ? patch_local_threads : block)
__attribute__((amdgpu_waves_per_eu(4))) void k_patch_prep(
  const VisRec<N>* __restrict__ recs, size_t n, Geometry geo,
  const GroupInfo* __restrict__ groups, const double2* __restrict__ wsum,
  Mueller mu, int update_weights, int gvis_ready, int adjoint,
  const float2* __restrict__ gvis_in, const double2* __restrict__ residuals,
  int ptx, int pty, int tw, int th, PatchRec<N>* __restrict__ out,
  unsigned* __restrict__ hist, double* __restrict__ weights,
  unsigned long long* __restrict__ invalid, unsigned batch, unsigned* __restrict__ table,
  unsigned* __restrict__ offsets, unsigned* __restrict__ order, unsigned* __restrict__ list,
  PatchSplit ps) {

  __shared__ double wblk[count_planes_lds];
  __shared__ unsigned cnt[LOCAL ? patch_local_keys + 1 : 1];
  const int keys = ptx * pty * geo.nc;
  if constexpr (LOCAL)
    for (int k = threadIdx.x; k < keys; k += blockDim.x) cnt[k] = 0u;
  const int nplanes = geo.nr * geo.nc;
  const bool lds_w = update_weights && nplanes <= count_planes_lds;
  if (lds_w)
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x) wblk[k] = 0.0;
  __syncthreads();

  const size_t stride = LOCAL ? blockDim.x : size_t(gridDim.x) * blockDim.x;
  const size_t i0 = blockIdx.x * (size_t)(LOCAL ? batch : blockDim.x) + threadIdx.x;
  // every thread runs the same number of iterations (the wave reductions
  // below need all lanes)
  const size_t iters = LOCAL ? (batch + stride - 1) / stride : (n + stride - 1) / stride;
  for (size_t it = 0; it < iters; ++it) {
    const size_t i = i0 + it * stride;
    bool counted = false;
    unsigned gcube = 0;
    double tw4[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < n) {
      const VisRec<N>& r = recs[i];
      const unsigned grp = r.cf_index[1];
      const unsigned cfcube = r.cf_index[0];
      gcube = r.grid_cube;
      bool valid = grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc);
      if (valid) valid = cfcube < unsigned(groups[grp].ncube);
      PatchRec<N> e;
      e.sxy = 0u;
      if (!valid) {
        atomicAdd(invalid, 1ull);
      } else {
        const GroupInfo g = groups[grp];
        const Coord c = vis_coord(r, geo, g);
        if (c.inside) {
          counted = update_weights != 0;
          if (patch_record<N>(r, i, c, geo, g, wsum, mu, update_weights, gvis_ready, adjoint,
                              gvis_in, residuals, e, tw4)) {
            const int tx0 = c.gx / tw, tx1 = (c.gx + g.sx - 1) / tw;
            const int ty0 = c.gy / th, ty1 = (c.gy + g.sy - 1) / th;
            for (int ty = ty0; ty <= ty1; ++ty)
              for (int tx = tx0; tx <= tx1; ++tx)
                if constexpr (LOCAL)
                  __hip_atomic_fetch_add(cnt + (int(gcube) * pty + ty) * ptx + tx, 1u,
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                else
                  atomicAdd(hist + (size_t(gcube) * pty + ty) * ptx + tx, 1u);
          }
        }
      }
      if (e.sxy) out[i] = e; else out[i].sxy = 0u;
    }
    if (update_weights) {
      unsigned long long active = __ballot(counted);
      const int lane = threadIdx.x % wave;
      while (active) {
        const int leader = __ffsll((long long)active) - 1;
        const unsigned cube = __shfl(gcube, leader, wave);
        const bool mine = counted && gcube == cube;
        active &= ~__ballot(mine);
#pragma unroll
        for (int gp = 0; gp < 4; ++gp) {
          if (gp >= geo.nr) continue;
          const double sw = wave_sum(mine ? tw4[gp] : 0.0);
          if (lane == leader) {
            const size_t k = size_t(cube) * geo.nr + gp;
            if (lds_w)
              __hip_atomic_fetch_add(wblk + k, sw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            else
              atomicAdd(weights + k, sw);
          }
        }
      }
    }
  }
  if (lds_w || LOCAL) __syncthreads();
  if (lds_w)
    for (int k = threadIdx.x; k < nplanes; k += blockDim.x)
      if (wblk[k] != 0.0) atomicAdd(weights + k, wblk[k]);
  if constexpr (LOCAL) {
    if (offsets) {
      patch_scan(keys, cnt, offsets, order, ps);
      for (size_t i = threadIdx.x; i < n; i += blockDim.x)  // its own records
        patch_tiles(out[i], pty, ptx, tw, th, [&](int key) {
          const unsigned at = __hip_atomic_fetch_add(cnt + key, 1u, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP);
          list[at] = unsigned(i);
        });
      return;
    }
    unsigned* row = table + size_t(blockIdx.x) * keys;
    for (int k = threadIdx.x; k < keys; k += blockDim.x)
      row[k] = cnt[k] ? atomicAdd(hist + k, cnt[k]) : 0u;
  }
}

// an entry's place in its tile's list: hist counts down what is left, or
// (LOCAL) the workgroup counts up from its place
template <int N, bool LOCAL>
__global__ __launch_bounds__(LOCAL ? patch_local_threads : block) void k_patch_list(
  size_t n, int nc, int ptx, int pty, int tw, int th, const PatchRec<N>* __restrict__ prs,
  unsigned* __restrict__ hist, const unsigned* __restrict__ offsets,
  unsigned* __restrict__ list, unsigned batch, const unsigned* __restrict__ table) {
  __shared__ unsigned at[LOCAL ? patch_local_keys : 1];
  const size_t first = blockIdx.x * (size_t)(LOCAL ? batch : blockDim.x);
  if constexpr (LOCAL) {
    const int keys = ptx * pty * nc;
    const unsigned* row = table + size_t(blockIdx.x) * keys;
    for (int k = threadIdx.x; k < keys; k += blockDim.x) at[k] = offsets[k] + row[k];
    __syncthreads();
  }
  const size_t last = min(n, first + (LOCAL ? size_t(batch) : size_t(blockDim.x)));
  for (size_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    patch_tiles(prs[i], pty, ptx, tw, th, [&](int key) {
      unsigned pos;
      if constexpr (LOCAL)
        pos = __hip_atomic_fetch_add(at + key, 1u, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
      else
        pos = offsets[key] + atomicSub(hist + key, 1u) - 1u;
      list[pos] = unsigned(i);
    });
  }
}

// 64 zeros and the 1152 bits of 2 / pi behind the point (computed from Machin's
// formula for pi)
__device__ const unsigned long long two_over_pi[19] = {
  0ull,
  0xa2f9836e4e441529ull, 0xfc2757d1f534ddc0ull, 0xdb6295993c439041ull,
  0xfe5163abdebbc561ull, 0xb7246e3a424dd2e0ull, 0x06492eea09d1921cull,
  0xfe1deb1cb129a73eull, 0xe88235f52ebb4484ull, 0xe99c7026b45f7e41ull,
  0x3991d639835339f4ull, 0x9c845f8bbdf9283bull, 0x1ff897ffde05980full,
  0xef2f118b5a0a6d1full, 0x6d367ecf27cb09b7ull, 0x4f463f669e5fea2dull,
  0x7527bac7ebe5f17bull, 0x3d0739f78a5292eaull, 0x6bfb5fb11f8d5d08ull};

// exp(i ph).  |ph| < 2^40: ph less the nearest multiple k of pi / 2 (pi / 2 as a
// 53-bit head, whose difference is exact, and its tail).  From there on, where
// the rounding of k itself would come to matter: Payne and Hanek's reduction
// ("Radian reduction for trigonometric functions", 1983), ph = m 2^e times the
// 128 bits of 2 / pi from the first that makes less than four quarter turns on,
// to 2^-62 of one.  Then the Taylor series of sine and cosine up to r^15 and
// r^16, |r| <= pi / 4 (remainders below 1e-16).  As cphase, whose library call
// would cost the tap loops 40 registers and with them a quarter of their waves
// (out of line still: its calling convention spills 20 to 100).
__device__ __forceinline__ double2 cphase_taylor(double ph) {
  double r;
  int q;
  if (fabs(ph) < 1099511627776.0) {
    const double k = rint(ph * 0.63661977236758134);  // 2 / pi
    r = __builtin_fma(-k, 1.5707963267948966, ph);
    r = __builtin_fma(-k, 6.123233995736766e-17, r);
    q = int(k - 4.0 * rint(0.25 * k)) & 3;  // quadrant (0 .. 3)
  } else {
    const unsigned long long b = (unsigned long long)__double_as_longlong(ph);
    const int e = int(b >> 52) & 0x7ff;  // ph = m 2^(e - 1075)
    const unsigned long long m = (b & 0xfffffffffffffull) | 0x10000000000000ull;
    // the first bit that makes less than four turns: 2^-(e - 1076) in 2 / pi
    const int at = min(e, 2046) - 1077 + 64;
    const unsigned long long* w = two_over_pi + (at >> 6);
    const int sh = at & 63;
    const unsigned long long hi = sh ? (w[0] << sh) | (w[1] >> (64 - sh)) : w[0];
    const unsigned long long lo = sh ? (w[1] << sh) | (w[2] >> (64 - sh)) : w[1];
    const unsigned long long phi = __umul64hi(m, lo) + m * hi;
    // phi: two bits of quarter turns, then their fraction, to the nearest
    const long long f = (long long)(phi << 2);
    q = int(phi >> 62) + (f < 0 ? 1 : 0);
    r = double(f) * 8.515303950216386e-20;  // pi / 2 2^-64
    if (b >> 63) {
      q = -q;
      r = -r;
    }
    q &= 3;
    if (e == 0x7ff) r = ph - ph;  // not finite
  }
  const double z = r * r;
  double s = -1.0 / 1307674368000.0;
  s = __builtin_fma(s, z, 1.0 / 6227020800.0);
  s = __builtin_fma(s, z, -1.0 / 39916800.0);
  s = __builtin_fma(s, z, 1.0 / 362880.0);
  s = __builtin_fma(s, z, -1.0 / 5040.0);
  s = __builtin_fma(s, z, 1.0 / 120.0);
  s = __builtin_fma(s, z, -1.0 / 6.0);
  s = __builtin_fma(s * z, r, r);
  double c = 1.0 / 20922789888000.0;
  c = __builtin_fma(c, z, -1.0 / 87178291200.0);
  c = __builtin_fma(c, z, 1.0 / 479001600.0);
  c = __builtin_fma(c, z, -1.0 / 3628800.0);
  c = __builtin_fma(c, z, 1.0 / 40320.0);
  c = __builtin_fma(c, z, -1.0 / 720.0);
  c = __builtin_fma(c, z, 1.0 / 24.0);
  c = __builtin_fma(c, z, -0.5);
  c = __builtin_fma(c, z, 1.0);
  const double re = q & 1 ? s : c, im = q & 1 ? c : s;
  return make_double2(q == 1 || q == 2 ? -re : re, q >= 2 ? -im : im);
}

// what a row takes of a slice (patch_kind)
constexpr int patch_any = 0;   // any of the N elements, one load each
constexpr int patch_full = 1;  // N neighbouring elements, N even, at 16-byte
                               // alignment: two elements a load
constexpr int patch_one = 2;   // at most one element
constexpr int patch_plane = 3;  // k_patch: that, of planar slices (one polarization)

// the records that a launch takes for a pixel: all, those whose support corner
// lies in the pixel's 32 x 32 tile, or the others
constexpr int patch_all = 0, patch_own = 1, patch_others = 2;

template <int N, int P, int KIND>
__global__ __launch_bounds__(patch_split(P) * patch_block)
__attribute__((amdgpu_waves_per_eu(5)))
void k_patch(
  Geometry geo, const float2* __restrict__ taps, Mueller mu, int mode, int take, int ptx, int pty,
  const unsigned* __restrict__ offsets, const unsigned* __restrict__ order,
  const unsigned* __restrict__ list, const PatchRec<N>* __restrict__ prs,
  const VisRec<N>* __restrict__ recs, void* __restrict__ grid, unsigned block0, PatchSplit ps) {

  constexpr int PW = patch_w(P), PH = patch_h(P);
  constexpr bool PLANAR = KIND == patch_plane;
  constexpr bool ONE = KIND == patch_one || PLANAR;
  constexpr int L = ONE ? 1 : N;  // elements a lane loads per tap
  constexpr int SPLIT = patch_split(P);
  constexpr unsigned stage = SPLIT * patch_block;
  __shared__ PatchRec<N> st[stage];
  __shared__ unsigned st_i[stage];

  // the slots of split lists first, then every tile
  const unsigned b = block0 + blockIdx.x;
  const bool split = b < ps.slots;
  unsigned key;
  uint2 ctl = make_uint2(0u, 0u), it = make_uint2(0u, 0u);
  if (split) {
    ctl = *reinterpret_cast<const uint2*>(ps.ctl());
    it = ps.items()[b];
    if (b >= ctl.x) return;
    key = it.x;
  } else {
    key = order ? order[b - ps.slots] : b - ps.slots;
    if (key == patch_none) return;
  }
  unsigned beg = offsets[key];
  unsigned cnt = offsets[key + 1] - beg;
  // what the end of a chunk needs, in LDS: scalar registers held through the loop
  // would spill others
  __shared__ unsigned chunk_slot, chunk_slot0, chunk_count;
  __shared__ PatchSplit chunk_ps;
  if (split) {
    if (threadIdx.x == 0) {
      chunk_slot = b;
      chunk_slot0 = b - it.y;
      chunk_count = (cnt + ctl.y - 1u) / ctl.y;
      chunk_ps = ps;
    }
    beg += it.y * ctl.y;
    cnt = min(ctl.y, cnt - it.y * ctl.y);
  }
  if (cnt == 0) return;
  const int tx = int(key % unsigned(ptx));
  const int tq = int(key / unsigned(ptx));
  const int ty = tq % pty;
  const int cube = tq / pty;

  const int w = uniform(int(threadIdx.x) / wave);
  const int part = w >> 2;  // this wave's share of its pixels' entries
  const int lane = threadIdx.x % wave;
  const int row = lane % P;
  const int px = (lane / P) % PW;
  const int py = (lane / P) / PW;
  const int bx = tx * patch_tile_x(P) + (w & 1) * 2 * PW;  // the wave's pixels
  const int by = ty * patch_tile_y(P) + ((w >> 1) & 1) * 2 * PH;

  // this lane's Mueller row for w <= 0: byte offsets of its elements within a
  // tap (~0u: none) and, for patch_one, the polarization they multiply; in
  // eo_x, vs_x what changes of them (xor) for w > 0
  unsigned eo[L], eo_x[L];
  unsigned vs = 0u, vs_x = 0u;
#pragma unroll
  for (int k = 0; k < L; ++k) {
    eo[k] = ~0u;
    eo_x[k] = ~0u;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (r >= geo.nr || r != row) continue;
#pragma unroll
    for (int v = 0; v < N; ++v) {
      const int m0 = mu.Mc[r][v], m1 = mu.M[r][v];
      constexpr unsigned es = unsigned(sizeof(float2));
      const int k = ONE ? 0 : v;
      if (m0 >= 0) {
        eo[k] = unsigned(m0) * es;
        if (ONE) vs = unsigned(v);
      }
      if (m1 >= 0) {
        eo_x[k] = unsigned(m1) * es;
        if (ONE) vs_x = unsigned(v);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < L; ++k) eo_x[k] ^= eo[k];
  vs_x ^= vs;

  double ar[4] = {0.0, 0.0, 0.0, 0.0}, ai[4] = {0.0, 0.0, 0.0, 0.0};

  for (unsigned b0 = 0; b0 < cnt; b0 += stage) {
    const unsigned m = min(stage, cnt - b0);
    __syncthreads();
    if (threadIdx.x < m) {
      const unsigned i = list[beg + b0 + threadIdx.x];
      st_i[threadIdx.x] = i;
      st[threadIdx.x] = prs[i];
    }
    __syncthreads();
    for (unsigned k0 = 0; k0 < m; k0 += wave) {
      // lane j: does entry k0 + j, of the wave's share, touch its pixels
      const unsigned je = min(k0 + unsigned(lane), m - 1u);
      const int hgx = st[je].gx, hgy = st[je].gy;
      const unsigned long long hbase = st[je].base;
      const unsigned hsxy = st[je].sxy, hfl = st[je].fl, hnm = st[je].nm;
      const unsigned hbhi = unsigned(hbase >> 32);
      const bool hit = lane % SPLIT == part && k0 + unsigned(lane) < m && hgx < bx + 2 * PW
        && hgx + patch_sx(hsxy, hbhi) > bx && hgy < by + 2 * PH
        && hgy + patch_sy(hsxy, hbhi) > by
        && (take == patch_all
            || ((hgx / tile == bx / tile && hgy / tile == by / tile) == (take == patch_own)));
      unsigned long long todo = __ballot(hit);
      while (todo) {
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        const int gx = __builtin_amdgcn_readlane(hgx, j);
        const int gy = __builtin_amdgcn_readlane(hgy, j);
        const unsigned blo = unsigned(__builtin_amdgcn_readlane(int(unsigned(hbase)), j));
        unsigned bhi = unsigned(__builtin_amdgcn_readlane(int(hbhi), j));
        const unsigned sxy = unsigned(__builtin_amdgcn_readlane(int(hsxy), j));
        const unsigned fl = unsigned(__builtin_amdgcn_readlane(int(hfl), j));
        const unsigned nm = unsigned(__builtin_amdgcn_readlane(int(hnm), j));
        const PatchRec<N>& e = st[k0 + unsigned(j)];
        int sx, sy;
        patch_unpack(sxy, bhi, sx, sy);
        const bool pos_w = fl & flag_pos_w;
        const unsigned pm = pos_w ? ~0u : 0u;
        // the slice from the first support row within the wave's pixels on,
        // at most 2 PH rows: offsets of 32 bits (patch_offsets_fit)
        const int y0 = max(by - gy, 0);
        const int rows = min(sy - y0, 2 * PH);
        const unsigned elem_bytes = nm * unsigned(sizeof(float2));
        // planar (one polarization): an element's taps lie side by side, the next
        // element `plane` taps on
        const unsigned plane = PLANAR ? unsigned(sx) * unsigned(sy) : 1u;
        const unsigned tap_bytes = PLANAR ? unsigned(sizeof(float2)) : elem_bytes;
        const unsigned row_bytes = unsigned(sx) * tap_bytes;
        const float2* first = taps
          + ((unsigned long long)blo | ((unsigned long long)bhi << 32))
          + (unsigned long long)unsigned(y0) * (unsigned(sx) * (PLANAR ? 1u : nm));
        const unsigned bytes = unsigned(rows) * row_bytes
          + (PLANAR ? (elem_bytes - unsigned(sizeof(float2))) * plane : 0u);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float2*>(first), 0, int(bytes), 0x00020000);
        const int X = bx + px - gx;
        const int Y = by + py - gy;
        const unsigned off0 = unsigned(Y - y0) * row_bytes + unsigned(X) * tap_bytes;
        float2 c[4][L];
        bool in[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int dx = (k & 1) * PW, dy = (k >> 1) * PH;
          in[k] = unsigned(X + dx) < unsigned(sx) && unsigned(Y + dy) < unsigned(sy);
          // a row without its element takes nothing, nor do lanes past the rows
          // (of three rows: whole elements of none would be read at ~0u)
          if constexpr (ONE)
            in[k] = in[k] && (eo[0] ^ (eo_x[0] & pm)) < elem_bytes;
          if constexpr (KIND == patch_full && P == 4) in[k] = in[k] && row < geo.nr;
          const unsigned off = off0 + unsigned(dy) * row_bytes + unsigned(dx) * tap_bytes;
          if constexpr (KIND == patch_full) {
            const unsigned o = in[k] ? off + (eo[0] ^ (eo_x[0] & pm)) : ~0u;
#pragma unroll
            for (int v = 0; v < N; v += 2) {
              const v4i_t q = __builtin_amdgcn_raw_buffer_load_b128(
                rsrc, int(o), v * int(sizeof(float2)), 0);
              c[k][v] = make_float2(__int_as_float(q.x), __int_as_float(q.y));
              c[k][v + 1] = make_float2(__int_as_float(q.z), __int_as_float(q.w));
            }
          } else {
#pragma unroll
            for (int v = 0; v < L; ++v) {
              const unsigned ev = eo[v] ^ (eo_x[v] & pm);
              const v2i_t q = __builtin_amdgcn_raw_buffer_load_b64(
                rsrc,
                int(in[k] && (ONE || ev < elem_bytes)
                      ? off + (PLANAR ? ev * plane : ev) : ~0u),
                0, 0);
              c[k][v] = make_float2(__int_as_float(q.x), __int_as_float(q.y));
            }
          }
        }
        // conj(c) g for w > 0: c.y g.y and c.y g.x enter with the sign
        // flipped, which rounds as conjugating c does
        float imf = pos_w ? -1.0f : 1.0f;
        if (fl & flag_gradient) {
          // the taps times the phase screen instead
          const unsigned i = st_i[k0 + unsigned(j)];
          const double gxr = recs[i].grad[0], gyr = recs[i].grad[1];
          const int fxi = int((fl >> 8) & 255u), fyi = int((fl >> 16) & 255u);
          const double phi0x = -gxr * ((sx / 2) * geo.os - (fxi - geo.F));
          const double phi0y = -gyr * ((sy / 2) * geo.os - (fyi - geo.F));
          const double dphix = gxr * geo.os;
          const double dphiy = gyr * geo.os;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int Xk = X + (k & 1) * PW, Yk = Y + (k >> 1) * PH;
            const float2 scr =
              narrow(cphase_taylor((phi0x + Xk * dphix) + (phi0y + Yk * dphiy)));
#pragma unroll
            for (int v = 0; v < L; ++v)
              c[k][v] = cmul(make_float2(c[k][v].x, imf * c[k][v].y), scr);
            // one patch at a time: the four together would hold the registers
            // of a wave
            __builtin_amdgcn_sched_barrier(0);
          }
          imf = 1.0f;
        }
        float2 g[L], gs[L];
#pragma unroll
        for (int v = 0; v < L; ++v) {
          g[v] = ONE ? e.g[vs ^ (vs_x & pm)] : e.g[v];
          gs[v] = make_float2(imf * g[v].x, imf * g[v].y);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (!in[k]) continue;
          double sr = 0.0, si = 0.0;
#pragma unroll
          for (int v = 0; v < L; ++v) {
            const float2 cc = c[k][v];
            const float pr = cc.x * g[v].x - cc.y * gs[v].y;
            const float pi = cc.x * g[v].y + cc.y * gs[v].x;
            if constexpr (KIND != patch_any) {
              sr += double(pr);
              si += double(pi);
            } else {
              const bool use = (eo[v] ^ (eo_x[v] & pm)) < elem_bytes;
              sr += use ? double(pr) : 0.0;
              si += use ? double(pi) : 0.0;
            }
          }
          ar[k] += sr;
          ai[k] += si;
        }
      }
    }
  }

  if constexpr (SPLIT > 1) {
    // the parts' sums, added by part 0 in their order
    static_assert(sizeof(st) >= size_t(SPLIT - 1) * 4 * wave * 8 * sizeof(double), "sums in st");
    double* sums = reinterpret_cast<double*>(st);
    __syncthreads();
    if (part > 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        double* q = sums + ((size_t(w - 4) * 8 + 2 * k) * wave + lane);
        q[0] = ar[k];
        q[wave] = ai[k];
      }
    }
    __syncthreads();
    for (int o = 1; o < SPLIT; ++o) {
      if (part > 0) break;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double* q = sums + ((size_t(w + 4 * (o - 1)) * 8 + 2 * k) * wave + lane);
        ar[k] += q[0];
        ai[k] += q[wave];
      }
    }
  }
  if (split) {
    const unsigned chunks = unsigned(uniform(int(chunk_count)));
    // this chunk's sums into its slot; the tile's last chunk to get here goes on
    // with those of all of them
    __shared__ unsigned ticket;
    const PatchSplit cs = chunk_ps;
    if (part == 0) {
      double* q = cs.sums(chunk_slot) + threadIdx.x;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        patch_store(q + 2 * k * patch_block, ar[k]);
        patch_store(q + (2 * k + 1) * patch_block, ai[k]);
      }
    }
    // written through to where every XCD reads them, before the ticket
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      ticket = atomicAdd(cs.tickets() + (take == patch_others ? cs.slots : 0u) + chunk_slot0, 1u);
    __syncthreads();
    if (ticket + 1u != chunks) return;
    if (part == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) ar[k] = ai[k] = 0.0;
      const double* q = cs.sums(chunk_slot0) + threadIdx.x;
#pragma unroll 1
      for (unsigned c = 0; c < chunks; ++c, q += patch_values) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = patch_load(q + k * patch_block);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          ar[k] += v[2 * k];
          ai[k] += v[2 * k + 1];
        }
      }
    }
  }

  // the tile's only writer: a plain read-modify-write of each pixel
  if (part > 0 || row >= geo.nr) return;
  const size_t plane = (size_t(cube) * geo.nr + row) * size_t(geo.ny) * geo.nx;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int x = bx + px + (k & 1) * PW, y = by + py + (k >> 1) * PH;
    if (x >= geo.nx || y >= geo.ny) continue;
    // a patch that nothing was added to stays as it is
    if (!__any(ar[k] != 0.0 || ai[k] != 0.0)) continue;
    const size_t gi = plane + size_t(y) * geo.nx + x;
    if (mode == 0) {
      double2* gp = static_cast<double2*>(grid) + gi;
      double2 v = *gp;
      v.x += ar[k];
      v.y += ai[k];
      *gp = v;
    } else {
      // one rounding of grid value + FP64 tile sum
      float2* gp = static_cast<float2*>(grid) + gi;
      const float2 v = *gp;
      *gp = make_float2(float(double(v.x) + ar[k]), float(double(v.y) + ai[k]));
    }
  }
}


// ---- gridding, few records -----------------------------------------------------
//
// One launch in place of the three or more of the binned pipelines, for batches
// whose time those launches are (one polarization, supports narrower than a
// tile): one workgroup per 32 x 32 tile looks through all records for those
// that touch it, adds the weights of those whose support corner it holds, and
// sums them in LDS (FP64 atomics; the grid rows' planes in turn), then adds the
// tile into the grid, of which it is the only writer.  A thread prepares a
// record in registers, and its wave adds its threads' records one after the
// other, a tap per lane in blocks of 8 x 8, the taps of direct_loads records
// loaded together; where it has many, a record per lane.  Bound by latencies: the
// launch, two reads of the records and what the densest tile takes.  Supports of 7
// on 512^2, uniform, back to back: 200 records 25.6 -> 9.9 us, 2000 32.3 -> 14.7; a
// register patch per wave in place of LDS sums took 0.33 us per record of the densest
// tile.

struct DirectArgs {
  const GroupInfo* groups;
  const double2* wsum;
  const float2* gvis;
  const double2* residuals;
  double* weights;
  unsigned long long* invalid;
  int update_weights, gvis_ready, adjoint;
};
constexpr int direct_block = 512;
constexpr int direct_loads = 4;
// A wave's lanes take a record each, tap by tap, where the supports have at most so
// many taps for each of its records (the time goes with the taps then, not with
// the records).  2000 records, sigma 2 pixels: supports 3 76 -> 37 us, 7 107 -> 80, 9
// 375 -> 103, 25 880 -> 450; 1500 on 128^2, supports 25 242 -> 107.  Limits of 1.5 and
// 20: 500 records of supports 25 there 122 us, 117 so.
constexpr float direct_lane_plain = 2.0f, direct_lane = 40.0f;
constexpr int direct_lane_min = 5;
constexpr int direct_lane_loads = 8;  // 4: 118 us for the 1500
// of a call (hit_i, 16 bits each); below what launches cost up to 8000: 240 tiles,
// supports of 7, binned and in one launch 2000 30.9, 15.6 us, 4000 37.0, 20.6, 8000
// 36.4, 30.9
constexpr unsigned direct_records = 2048;
constexpr int direct_row = tile + 8;  // LDS row: four rows of a block on banks of their own
constexpr int direct_plane = tile * direct_row;

__global__ __launch_bounds__(direct_block) __attribute__((amdgpu_waves_per_eu(4))) void k_direct(
  Geometry geo, const float2* __restrict__ taps, Mueller mu,
  const VisRec<1>* __restrict__ recs, unsigned n, DirectArgs da, double2* __restrict__ grid) {
  extern __shared__ double sums[];  // per grid row: re, im
  __shared__ unsigned short hit_i[direct_records];
  __shared__ unsigned hits;
  __shared__ double row_w[4];

  const unsigned key = blockIdx.x;
  const int x0 = int(key % unsigned(geo.ntx)) * tile;
  const unsigned tq = key / unsigned(geo.ntx);
  const int y0 = int(tq % unsigned(geo.nty)) * tile;
  const int cube = int(tq / unsigned(geo.nty));
  if (threadIdx.x == 0) hits = 0u;
  if (threadIdx.x < 4) row_w[threadIdx.x] = 0.0;
  __syncthreads();
  for (unsigned i = threadIdx.x; i < n; i += direct_block) {
    const VisRec<1>& r = recs[i];
    const unsigned grp = r.cf_index[1], gcube = r.grid_cube;
    bool valid = grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc);
    if (valid) valid = r.cf_index[0] < unsigned(da.groups[grp].ncube);
    if (!valid) {
      if (key == 0) atomicAdd(da.invalid, 1ull);
      continue;
    }
    if (int(gcube) != cube) continue;
    const GroupInfo& g = da.groups[grp];
    const Coord c = vis_coord(r, geo, g);
    if (c.inside && c.gx < x0 + tile && c.gx + g.sx > x0 && c.gy < y0 + tile && c.gy + g.sy > y0)
      hit_i[__hip_atomic_fetch_add(&hits, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)] =
        (unsigned short)i;
  }
  __syncthreads();
  const unsigned cnt = unsigned(uniform(int(hits)));
  if (cnt == 0) return;
  for (int k = threadIdx.x; k < geo.nr * 2 * direct_plane; k += direct_block) sums[k] = 0.0;
  __syncthreads();

  const unsigned w = unsigned(uniform(int(threadIdx.x) / wave));
  const int lane = threadIdx.x % wave;
  const int lx = lane & 7, ly = lane >> 3;
  constexpr unsigned nw = direct_block / wave;
  for (unsigned b0 = 0; b0 < cnt; b0 += direct_block) {
    // lane l: record w + l * nw of the round
    const unsigned h = b0 + w + unsigned(lane) * nw;
    const unsigned left = cnt - b0;
    const int mine = left > w ? int(min((left - w + nw - 1u) / nw, unsigned(wave))) : 0;
    PatchRec<1> e{};
    unsigned i = 0;
    if (h < cnt) {
      i = hit_i[h];
      const VisRec<1>& r = recs[i];
      const GroupInfo g = da.groups[r.cf_index[1]];
      const Coord c = vis_coord(r, geo, g);
      double tw4[4];
      patch_record<1>(r, i, c, geo, g, da.wsum, mu, da.update_weights, da.gvis_ready, da.adjoint,
                      da.gvis, da.residuals, e, tw4);
      if (da.update_weights && c.gx >= x0 && c.gy >= y0) {
#pragma unroll
        for (int gp = 0; gp < 4; ++gp)
          if (gp < geo.nr)
            __hip_atomic_fetch_add(row_w + gp, tw4[gp], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    const bool plain = int(e.sxy & 0xffffu) <= 8 && int(e.sxy >> 16) <= 8
      && !(e.fl & flag_gradient);
    const unsigned long long plain_m = __ballot(plain);
    // many records in the wave: each lane its own, tap by tap
    const float most = float(mine) * (plain_m == ~0ull ? direct_lane_plain : direct_lane);
    if (__builtin_expect(mine >= direct_lane_min, 0)
        && !__any(float(int(e.sxy & 0xffffu) * int(e.sxy >> 16)) > most)) {
      if (!e.sxy) continue;
      const int sx = int(e.sxy & 0xffffu), sy = int(e.sxy >> 16);
      const bool pos_w = e.fl & flag_pos_w, grad = e.fl & flag_gradient;
      const float imf = pos_w ? -1.0f : 1.0f;
      double gxr = 0.0, gyr = 0.0;
      if (grad) {
        gxr = recs[i].grad[0];
        gyr = recs[i].grad[1];
      }
      const double phi0x = -gxr * ((sx / 2) * geo.os - (int((e.fl >> 8) & 255u) - geo.F));
      const double phi0y = -gyr * ((sy / 2) * geo.os - (int((e.fl >> 16) & 255u) - geo.F));
      const double dphix = gxr * geo.os, dphiy = gyr * geo.os;
      // the support's part in the tile
      const int bx0 = max(x0 - e.gx, 0), bx1 = min(sx, x0 + tile - e.gx);
      const int by0 = max(y0 - e.gy, 0), by1 = min(sy, y0 + tile - e.gy);
      const int nt = (bx1 - bx0) * (by1 - by0);
      for (int gp = 0; gp < geo.nr; ++gp) {
        const int el = pos_w ? mu.M[gp][0] : mu.Mc[gp][0];
        if (el < 0 || unsigned(el) >= e.nm) continue;
        const float2* cf = taps + e.base + unsigned(el) * unsigned(sx * sy);
        double* dst = sums + gp * 2 * direct_plane;
        auto add_at = [&](int X, int Y, float2 cc) {
          const float2 pr = cmul(cc, e.g[0]);
          double* at = dst + (e.gy + Y - y0) * direct_row + e.gx + X - x0;
          __hip_atomic_fetch_add(at, double(pr.x), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
          __hip_atomic_fetch_add(at + direct_plane, double(pr.y), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        if (grad) {  // apart: its registers would be the whole kernel's
#pragma unroll 1
          for (int Y = by0; Y < by1; ++Y)
#pragma unroll 1
            for (int X = bx0; X < bx1; ++X) {
              float2 cc = cf[Y * sx + X];
              cc.y *= imf;
              add_at(X, Y, cmul(cc, narrow(cphase_taylor((phi0x + X * dphix)
                                                         + (phi0y + Y * dphiy)))));
            }
          continue;
        }
        int X = bx0, Y = by0;
        for (int t0 = 0; t0 < nt; t0 += direct_lane_loads) {
          float2 c[direct_lane_loads];
          int Xk[direct_lane_loads], Yk[direct_lane_loads];
#pragma unroll
          for (int k = 0; k < direct_lane_loads; ++k) {
            Xk[k] = X;
            Yk[k] = Y;
            c[k] = t0 + k < nt ? cf[Y * sx + X] : make_float2(0.0f, 0.0f);
            if (++X == bx1) {
              X = bx0;
              ++Y;
            }
          }
#pragma unroll
          for (int k = 0; k < direct_lane_loads; ++k) {
            if (t0 + k >= nt) continue;
            c[k].y *= imf;
            add_at(Xk[k], Yk[k], c[k]);
          }
        }
      }
      continue;
    }
    auto of = [&](int v, int j) { return __builtin_amdgcn_readlane(v, j); };
    // the tap (X, Y) of record j: its value (in: there is one in the tile)
    auto load = [&](int j, int gp, int X, int Y, bool& in, int& px) {
      const unsigned sxy = unsigned(of(int(e.sxy), j));
      const unsigned nm = unsigned(of(int(e.nm), j));
      const bool pos_w = of(int(e.fl), j) & flag_pos_w;
      const int el = pos_w ? mu.M[gp][0] : mu.Mc[gp][0];
      const int x = of(e.gx, j) + X - x0, y = of(e.gy, j) + Y - y0;
      in = X < int(sxy & 0xffffu) && Y < int(sxy >> 16) && unsigned(x) < unsigned(tile)
        && unsigned(y) < unsigned(tile) && el >= 0 && unsigned(el) < nm;
      px = y * direct_row + x;
      const float2* cf = taps
        + ((unsigned long long)unsigned(of(int(unsigned(e.base)), j))
           | ((unsigned long long)unsigned(of(int(e.base >> 32), j)) << 32));
      return in ? cf[(unsigned(el) * (sxy >> 16) + unsigned(Y)) * (sxy & 0xffffu) + unsigned(X)]
                : make_float2(0.0f, 0.0f);
    };
    auto add = [&](int j, int gp, float2 cc, bool in, int px) {
      const float2 gv = make_float2(__int_as_float(of(__float_as_int(e.g[0].x), j)),
                                    __int_as_float(of(__float_as_int(e.g[0].y), j)));
      if (!in) return;
      const float2 pr = cmul(cc, gv);
      double* dst = sums + gp * 2 * direct_plane + px;
      __hip_atomic_fetch_add(dst, double(pr.x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(dst + direct_plane, double(pr.y), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    for (int j0 = 0; j0 < mine; j0 += direct_loads) {
      constexpr unsigned long long all = (1ull << direct_loads) - 1ull;
      if (((plain_m >> j0) & all) == all) {  // lanes past the last record are plain
        for (int gp = 0; gp < geo.nr; ++gp) {
          float2 c[direct_loads];
          bool in[direct_loads];
          int px[direct_loads];
#pragma unroll
          for (int u = 0; u < direct_loads; ++u) c[u] = load(j0 + u, gp, lx, ly, in[u], px[u]);
#pragma unroll
          for (int u = 0; u < direct_loads; ++u) {
            c[u].y *= (of(int(e.fl), j0 + u) & flag_pos_w) ? -1.0f : 1.0f;
            add(j0 + u, gp, c[u], in[u], px[u]);
          }
        }
        continue;
      }
#pragma unroll 1
      for (int j = j0; j < min(j0 + direct_loads, mine); ++j) {
        const unsigned sxy = unsigned(of(int(e.sxy), j));
        const unsigned fl = unsigned(of(int(e.fl), j));
        const int sx = int(sxy & 0xffffu), sy = int(sxy >> 16);
        const float imf = (fl & flag_pos_w) ? -1.0f : 1.0f;
        double gxr = 0.0, gyr = 0.0;
        if (fl & flag_gradient) {
          const unsigned ri = unsigned(of(int(i), j));
          gxr = recs[ri].grad[0];
          gyr = recs[ri].grad[1];
        }
        const double phi0x = -gxr * ((sx / 2) * geo.os - (int((fl >> 8) & 255u) - geo.F));
        const double phi0y = -gyr * ((sy / 2) * geo.os - (int((fl >> 16) & 255u) - geo.F));
        const double dphix = gxr * geo.os, dphiy = gyr * geo.os;
        // the support's blocks in the tile
        const int gx = of(e.gx, j), gy = of(e.gy, j);
        const int bx0 = max(x0 - gx, 0), bx1 = min(sx, x0 + tile - gx);
        const int by0 = max(y0 - gy, 0), by1 = min(sy, y0 + tile - gy);
        for (int gp = 0; gp < geo.nr; ++gp)
          for (int Y = by0 + ly; Y - ly < by1; Y += 8) {
            float2 c[direct_loads];
            bool in[direct_loads];
            int px[direct_loads];
#pragma unroll
            for (int u = 0; u < direct_loads; ++u)  // at most 4 blocks in a row of them
              c[u] = load(j, gp, bx0 + lx + 8 * u, Y, in[u], px[u]);
#pragma unroll 1
            for (int u = 0; u < direct_loads; ++u) {
              if (bx0 + 8 * u >= bx1) break;
              float2 cc = u == 0 ? c[0] : u == 1 ? c[1] : u == 2 ? c[2] : c[3];
              const bool ok = u == 0 ? in[0] : u == 1 ? in[1] : u == 2 ? in[2] : in[3];
              const int at = u == 0 ? px[0] : u == 1 ? px[1] : u == 2 ? px[2] : px[3];
              cc.y *= imf;
              if (fl & flag_gradient)
                cc = cmul(cc, narrow(cphase((phi0x + (bx0 + lx + 8 * u) * dphix)
                                            + (phi0y + Y * dphiy))));
              add(j, gp, cc, ok, at);
            }
          }
      }
    }
  }
  __syncthreads();
  if (int(threadIdx.x) < geo.nr && row_w[threadIdx.x] != 0.0)
    atomicAdd(da.weights + (size_t(cube) * geo.nr + threadIdx.x), row_w[threadIdx.x]);
  for (int k = threadIdx.x; k < geo.nr * tile * tile; k += direct_block) {
    const int gp = k / (tile * tile), px = k % (tile * tile);
    const int x = x0 + px % tile, y = y0 + px / tile;
    if (x >= geo.nx || y >= geo.ny) continue;
    const double* src = sums + gp * 2 * direct_plane + (px / tile) * direct_row + px % tile;
    const double vr = src[0], vi = src[direct_plane];
    if (vr == 0.0 && vi == 0.0) continue;
    const size_t gi = ((size_t(cube) * geo.nr + gp) * geo.ny + y) * geo.nx + x;
    const double2 g0 = grid[gi];
    grid[gi] = make_double2(g0.x + vr, g0.y + vi);
  }
}

// ---- degridding --------------------------------------------------------

// The slice-ordered degridder, for several polarizations, large supports and
// large grids: k_degrid_keys prepares the records, k_sort_place and
// k_degrid_sort order them by CF slice, k_degrid sums c' x model over their
// supports and k_degrid_finish makes predictions of the sums.

// a record prepared for k_degrid; sxy = 0: not degridded
struct __align__(16) DegridRec {
  unsigned long long base;  // as PatchRec::base
  long long corner;         // model index of its support corner, grid row 0
  unsigned sxy;             // as PatchRec::sxy
  unsigned fl;              // flags | fxi << 8 | fyi << 16
  unsigned nm;              // Mueller elements of its CF group
  unsigned pad;
};

struct DegridKeys {
  unsigned slices, stride;  // of the batch, of a group
  int region_sh;
  unsigned regions_x, regions;
};

// key = the record's (grid cube, region, group, CF cube, fine offsets), ~0 for
// records that are skipped (no CF, outside the grid); region (region_sh below
// 31) the square of 2^region_sh pixels that holds the support corner.  keys
// null: prepared only
template <int N>
__global__ __launch_bounds__(patch_local_threads) void k_degrid_keys(
  size_t n, Geometry geo, const GroupInfo* __restrict__ groups,
  const VisRec<N>* __restrict__ recs, DegridKeys dk, SortKeys sk, unsigned batch,
  unsigned* __restrict__ keys,
  DegridRec* __restrict__ out, unsigned* __restrict__ hist, unsigned* __restrict__ table) {
  __shared__ unsigned cnt[patch_local_keys];
  if (keys)
    for (int k = threadIdx.x; k < sk.bins; k += blockDim.x) cnt[k] = 0u;
  __syncthreads();
  const size_t first = blockIdx.x * (size_t)batch;
  const size_t last = min(n, first + batch);
  for (size_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    const VisRec<N>& r = recs[i];
    const unsigned grp = r.cf_index[1];
    const unsigned cfcube = r.cf_index[0];
    const unsigned gcube = r.grid_cube;
    unsigned key = ~0u;
    DegridRec d{};
    if (grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc)) {
      const GroupInfo g = groups[grp];
      if (cfcube < unsigned(g.ncube)) {
        const Coord c = vis_coord(r, geo, g);
        if (c.inside) {
          const unsigned fxi = unsigned(c.fx + geo.F), fyi = unsigned(c.fy + geo.F);
          const bool grad = r.grad[0] != 0.0 || r.grad[1] != 0.0;
          const unsigned region = (unsigned(c.gy) >> dk.region_sh) * dk.regions_x
            + (unsigned(c.gx) >> dk.region_sh);
          key = (gcube * dk.regions + region) * dk.slices + grp * dk.stride
            + (cfcube * unsigned(geo.nf) + fxi) * unsigned(geo.nf) + fyi;
          patch_pack(slice_start(g, geo.nf, int(cfcube), int(fxi), int(fyi)), g.sx, g.sy,
                     d.base, d.sxy);
          d.corner = ((long long)gcube * geo.nr * geo.ny + c.gy) * geo.nx + c.gx;
          d.fl = unsigned((r.uvw[2] > 0 ? flag_pos_w : 0) | (grad ? flag_gradient : 0))
            | (fxi << 8) | (fyi << 16);
          d.nm = unsigned(g.nmueller);
          if (keys)
            __hip_atomic_fetch_add(cnt + (key >> (sk.low_bits + sk.drop_bits)), 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
    if (keys) keys[i] = key;
    out[i] = d;
  }
  if (!keys) return;
  __syncthreads();
  unsigned* row = table + size_t(blockIdx.x) * sk.bins;
  for (int k = threadIdx.x; k < sk.bins; k += blockDim.x)
    row[k] = cnt[k] ? atomicAdd(hist + k, cnt[k]) : 0u;
}

// one workgroup per bin: its records in order of their lower key bits
__global__ __launch_bounds__(sort_threads) void k_degrid_sort(
  int low_bits, const unsigned* __restrict__ offsets, const uint2* __restrict__ pairs,
  unsigned* __restrict__ order) {
  const unsigned beg = offsets[blockIdx.x], end = offsets[blockIdx.x + 1];
  if (end - beg <= 1u) {
    if (threadIdx.x == 0 && end != beg) order[beg] = pairs[beg].y;
    return;
  }
  sort_bin(low_bits, beg, end, pairs, [](const unsigned*) {},
           [&](unsigned at, unsigned i) { order[beg + at] = i; });
}

// sums val[0, V) of the lanes that differ in bits 1 .. MASK of their number.
// Each step halves the values a lane holds (it keeps one half, and adds its
// partner's values of that half) while their number is even: V - 1 adds
// instead of V log2(lanes).  Value `at` + i is in val[i] afterwards, i below
// the returned number.
template <int V, int MASK>
__device__ __forceinline__ int reduce_lanes(double* val, int lane, int& at) {
  if constexpr (MASK == 0) {
    return V;
  } else if constexpr (V % 2 == 0) {
    constexpr int H = V / 2;
    const bool up = lane & MASK;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const double keep = up ? val[i + H] : val[i];
      const double send = up ? val[i] : val[i + H];
      val[i] = keep + __shfl_xor(send, MASK, wave);
    }
    at += up ? H : 0;
    return reduce_lanes<H, MASK / 2>(val, lane, at);
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) val[i] += __shfl_xor(val[i], MASK, wave);
    return reduce_lanes<V, MASK / 2>(val, lane, at);
  }
}

// records a wave takes (eight of one element a row, or of two polarizations,
// measured slower: their registers cost a wave per SIMD)
constexpr int degrid_recs = 4;
// Rounds of loads between sums put aside, where a row uses one element and the
// supports are long: its taps then fill 16 to 64 lanes, and a sum of n taps rounds
// like sqrt(n / 2) of its last steps.  Error against 64 bits and the call: four rows,
// supports of 33 to 65, 50,000 records, 7.3e-16 in one chain of two roundings a tap
// (1170 us), 4.5e-16 by pairs of steps (k_degrid), 3.4e-16 with parts too (1190; 3.8e-16
// by 64 lanes a row); 9 to 33, 1e6 records, 3.7e-16 (3070 us) and 2.9e-16 (3062); two
// rows, 9 to 33, 100,000 records, 3.3e-16 (237) and 2.9e-16 (243).
constexpr unsigned degrid_part = 8;
// and the steps of a chain that stays whole: two rows, supports of 7 to 17 (9 steps),
// 2.7e-16 either way, the kernel 222 us whole and 233 in pairs
constexpr int degrid_whole = 16;

// One wave takes R records in a row of the order; those of one slice share
// every CF value it loads (per tap of 4 x 4 elements a record reads 64 bytes
// of model and 128 of CF: the CF reads are the larger part until four share
// them).  A lane is a (tap, grid row), 64 / P taps a step, the taps of a row in
// neighbouring lanes: their model values are neighbours too (the cache takes a
// load by lines, 16 for 64 lanes of 16 bytes so, 64 with the rows in
// neighbouring lanes: 1.2 ms against 0.97 for 300,000 records of supports 9-33
// and one element a row).  The sums over the support go to acc (record x polarization).
// order null: the records as they come, else *ordered of them.  same_rows: M and Mc are equal, so
// that records of both signs of w share CF values (the model's imaginary part
// takes the sign: sum conj(c) m = conj(sum c conj(m))).  patch_one: no two
// rows use one polarization; acc of one that no row uses is not written.
// Bound: the model gathers, from HBM for batches that are sparse on the grid
// (64 bytes per tap from anywhere in the model, 4.4 TB/s with their line ends:
// 500,000 records of supports 9-65 and 16 elements 13.8 ms, 26.8 ms one record a
// wave; 150,000 of 17-129 14.0 ms, before 27.1), from L2 in dense regions
// (launch_degrid): 1e6 records of supports 9-33 and one element a row 2.9 ms,
// before 7.3; 300,000 of 7-17, two polarizations, 222 us, before 1250 us one
// record a lane.  Two steps' loads at once where a row uses one element (3.3 ms
// one by one).  Three waves per SIMD for several: at four the sums spill
// (15.9 ms the first).
template <int N, int P, int KIND, bool LONG>
__global__ __launch_bounds__(block) __attribute__((amdgpu_waves_per_eu(KIND == patch_one ? 4 : 3)))
void k_degrid(
  size_t n, Geometry geo, const float2* __restrict__ taps, Mueller mu, int same_rows,
  const double2* __restrict__ model, int by_xcd, const DegridRec* __restrict__ drs,
  const VisRec<N>* __restrict__ recs, const unsigned* __restrict__ order,
  const unsigned* __restrict__ ordered, double* __restrict__ acc, unsigned block0) {

  constexpr int R = degrid_recs;
  constexpr int L = KIND == patch_one ? 1 : N;  // elements of a row
  constexpr int TPS = wave / P;                 // taps a step
  constexpr bool parts = KIND == patch_one && LONG;
  __shared__ double part[parts ? R * L * 2 * block : 1];

  const int w = uniform(int(threadIdx.x) / wave);
  const int lane = threadIdx.x % wave;
  const unsigned bi = block0 + (by_xcd ? xcd_key(blockIdx.x, gridDim.x) : blockIdx.x);
  const size_t p0 = (bi * (size_t)(block / wave) + w) * R;
  if (order) n = *ordered;  // the records that are not skipped
  if (p0 >= n) return;
  const int row = lane / TPS;
  const int q = lane % TPS;

  // lane r < R: record r of the wave
  DegridRec d{};
  unsigned rec_i = 0;
  if (lane < R && p0 + lane < n) {
    rec_i = order ? order[p0 + lane] : unsigned(p0 + lane);
    d = drs[rec_i];
  }
  const unsigned long long live = __ballot(d.sxy != 0u);

  // this lane's Mueller row for w <= 0 (element indexes, -1: none; for
  // patch_one in [0] only, with its polarization) and what changes of it
  // (xor) for w > 0
  int el[L], el_x[L];
  int vs = 0, vs_x = 0;
#pragma unroll
  for (int k = 0; k < L; ++k) el[k] = el_x[k] = -1;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (r >= geo.nr || r != row) continue;
#pragma unroll
    for (int v = 0; v < N; ++v) {
      // degridding uses the other Mueller matrix than gridding
      // (src/hpg_core.hpp:598-600)
      const int m0 = mu.M[r][v], m1 = mu.Mc[r][v];
      const int k = KIND == patch_one ? 0 : v;
      if (m0 >= 0) {
        el[k] = m0;
        vs = v;
      }
      if (m1 >= 0) {
        el_x[k] = m1;
        vs_x = v;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < L; ++k) el_x[k] ^= el[k];
  vs_x ^= vs;
  const long long row_off = (long long)(row < geo.nr ? row : 0) * geo.ny * geo.nx;

  auto lane_u64 = [&](unsigned long long v, int j) {
    return (unsigned long long)unsigned(__builtin_amdgcn_readlane(int(unsigned(v)), j))
      | ((unsigned long long)unsigned(__builtin_amdgcn_readlane(int(v >> 32), j)) << 32);
  };
  auto lane_u32 = [&](unsigned v, int j) {
    return unsigned(__builtin_amdgcn_readlane(int(v), j));
  };

  // the sums of RR records from record r on, which share one slice and
  // Mueller row; GRAD: one record with a phase gradient
  auto run = [&](auto rr_c, auto grad_c, int r) {
    constexpr int RR = decltype(rr_c)::value;
    constexpr bool GRAD = decltype(grad_c)::value;
    const unsigned sxy = lane_u32(d.sxy, r);
    const unsigned base_lo = lane_u32(unsigned(d.base), r);
    unsigned base_hi = lane_u32(unsigned(d.base >> 32), r);
    int sx, sy;
    patch_unpack(sxy, base_hi, sx, sy);
    const unsigned ntap = unsigned(sx) * unsigned(sy);  // of one slice: below 2^32 in 288 GB
    const unsigned nm = lane_u32(d.nm, r);
    const int pm = (lane_u32(d.fl, r) & flag_pos_w) ? -1 : 0;
    const bool planar = N == 1 && geo.planar;
    const unsigned step = planar ? 1u : nm;  // from tap to tap
    const float2* cf = taps
      + ((unsigned long long)base_lo | ((unsigned long long)base_hi << 32))
      + size_t(q) * step;  // this lane's tap
    unsigned eo[L];                                                  // its elements
    bool use[L];
#pragma unroll
    for (int v = 0; v < L; ++v) {
      const int m = el[v] ^ (el_x[v] & pm);
      use[v] = m >= 0 && m < int(nm);
      eo[v] = unsigned(use[v] ? m : 0) * (planar ? ntap : 1u);
    }
    const double2* mp[RR];
    unsigned flip[RR];  // w <= 0: the imaginary parts' sign
#pragma unroll
    for (int k = 0; k < RR; ++k) {
      mp[k] = model + (lane_u64((unsigned long long)d.corner, r + k) + row_off);
      flip[k] = (lane_u32(d.fl, r + k) & flag_pos_w) ? 0u : 0x80000000u;
    }
    double val[RR * L * 2];
#pragma unroll
    for (int k = 0; k < RR * L * 2; ++k) val[k] = 0.0;
    // the tap's (X, Y), from a float reciprocal and one correction either way
    // (exact: q < 64), and the model offset
    int Y = int(float(q) * __builtin_amdgcn_rcpf(float(sx)));
    int X = q - Y * sx;
    if (X < 0) {
      X += sx;
      --Y;
    }
    if (X >= sx) {
      X -= sx;
      ++Y;
    }
    long long off = (long long)Y * geo.nx + X;
    const int dY = sx > TPS ? 0 : TPS / sx;
    const int dX = TPS - dY * sx;
    const long long doff = (long long)dY * geo.nx + dX;
    const long long wrap = (long long)geo.nx - sx;
    double gp0 = 0.0, gdx = 0.0, gdy = 0.0, gp1 = 0.0;
    if constexpr (GRAD) {
      const unsigned fl = lane_u32(d.fl, r);
      const VisRec<N>& rc = recs[lane_u32(rec_i, r)];
      const double gxr = rc.grad[0], gyr = rc.grad[1];
      gp0 = -gxr * ((sx / 2) * geo.os - (int((fl >> 8) & 255u) - geo.F));
      gp1 = -gyr * ((sy / 2) * geo.os - (int((fl >> 16) & 255u) - geo.F));
      gdx = gxr * geo.os;
      gdy = gyr * geo.os;
    }
    // U steps, their loads issued together
    auto steps = [&](auto u_c) {
      constexpr int U = decltype(u_c)::value;
      float2 c[U][L];
      double2 m[U][RR];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (KIND == patch_full) {
#pragma unroll
          for (int v = 0; v < N; v += 2) {
            const float4 t = *reinterpret_cast<const float4*>(cf + eo[0] + v);
            c[u][v] = make_float2(t.x, t.y);
            c[u][v + 1] = make_float2(t.z, t.w);
          }
        } else {
#pragma unroll
          for (int v = 0; v < L; ++v) c[u][v] = cf[eo[v]];
        }
        cf += size_t(TPS) * step;
#pragma unroll
        for (int k = 0; k < RR; ++k) m[u][k] = mp[k][off];
        if constexpr (GRAD)
          m[u][0] = cmul(m[u][0], cphase_taylor(-(gp0 + X * gdx) - (gp1 + Y * gdy)));
        X += dX;
        Y += dY;
        off += doff;
        if (X >= sx) {
          X -= sx;
          ++Y;
          off += wrap;
        }
      }
      // LONG: the steps' products added up, then to the sums: one rounding of a sum
      // for U taps in place of two for each
#pragma unroll
      for (int k = 0; k < RR; ++k) {
#pragma unroll
        for (int v = 0; v < L; ++v) {
          if (KIND == patch_any && !use[v]) continue;
          double& a = val[(k * L + v) * 2];
          double& b = val[(k * L + v) * 2 + 1];
          double tr = LONG ? 0.0 : a, ti = LONG ? 0.0 : b;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const double mx = m[u][k].x;
            const double my = __hiloint2double(
              int(unsigned(__double2hiint(m[u][k].y)) ^ flip[k]), __double2loint(m[u][k].y));
            const double cx = double(c[u][v].x), cy = double(c[u][v].y);
            tr = u || !LONG ? __builtin_fma(cx, mx, tr) : cx * mx;
            tr = __builtin_fma(-cy, my, tr);
            ti = u || !LONG ? __builtin_fma(cx, my, ti) : cx * my;
            ti = __builtin_fma(cy, mx, ti);
          }
          a = LONG ? a + tr : tr;
          b = LONG ? b + ti : ti;
        }
      }
    };
    constexpr int U = GRAD || RR * (L + 1) > 12 ? 1 : 2;
    const unsigned full = ntap / TPS;
    unsigned s = 0;
    bool kept = false;
#pragma unroll 1
    for (; s + U <= full; s += U) {
      steps(std::integral_constant<int, U>{});
      if (parts && (s / U) % degrid_part == degrid_part - 1) {
#pragma unroll
        for (int k = 0; k < RR * L * 2; ++k) {
          double* p = part + k * block + threadIdx.x;
          *p = kept ? *p + val[k] : val[k];
          val[k] = 0.0;
        }
        kept = true;
      }
    }
    if constexpr (U > 1) {
#pragma unroll 1
      for (; s < full; ++s) steps(std::integral_constant<int, 1>{});
    }
    if (full * TPS + unsigned(q) < ntap) steps(std::integral_constant<int, 1>{});
    if (kept)
#pragma unroll
      for (int k = 0; k < RR * L * 2; ++k) val[k] += part[k * block + threadIdx.x];
    // the other sign's imaginary parts, then the sums over the taps (and,
    // but for patch_one, the rows)
#pragma unroll
    for (int k = 0; k < RR; ++k)
#pragma unroll
      for (int v = 0; v < L; ++v) {
        double& b = val[(k * L + v) * 2 + 1];
        b = flip[k] ? -b : b;
        if (KIND != patch_one && !use[v]) val[(k * L + v) * 2] = b = 0.0;
      }
    int at = 0;
    const int left =
      reduce_lanes<RR * L * 2, (KIND == patch_one ? TPS : wave) / 2>(val, lane, at);
#pragma unroll
    for (int i = 0; i < RR * L * 2; ++i) {
      if (i >= left) continue;
      const int a = at + i;
      const int k = a / (L * 2);
      const size_t ri = unsigned(__shfl(int(rec_i), r + k, wave));
      const int v = KIND == patch_one ? vs ^ (vs_x & pm) : (a / 2) % L;
      if (KIND != patch_one || use[0]) acc[(ri * N + v) * 2 + (a & 1)] = val[i];
    }
  };

  for (int r = 0; r < R;) {
    if (!((live >> r) & 1ull)) {
      ++r;
      continue;
    }
    const unsigned long long base = lane_u64(d.base, r);
    const unsigned fl = lane_u32(d.fl, r);
    const unsigned long long same = __ballot(
      d.sxy != 0u && !(d.fl & flag_gradient) && d.base == base
      && (same_rows || !((d.fl ^ fl) & flag_pos_w))) >> r;
    const int len = __builtin_ctzll(~same);  // records in a row, 0 for a gradient
    if (len >= R) {
      run(std::integral_constant<int, R>{}, std::false_type{}, r);
      r += R;
    } else if (len >= 2) {
      run(std::integral_constant<int, 2>{}, std::false_type{}, r);
      r += 2;
    } else if (len == 1) {
      run(std::integral_constant<int, 1>{}, std::false_type{}, r);
      r += 1;
    } else {
      run(std::integral_constant<int, 1>{}, std::true_type{}, r);
      r += 1;
    }
  }
}

// Binned degridding (supports below a tile): the entries of k_bin
// in degrid mode (record index beside every entry) are processed one
// workgroup per (plane, tile) key.  The workgroup loads the model's tile +
// halo region of its plane into LDS with coalesced reads, then one lane per
// entry sums c' x model over the footprint from LDS (FP64), in slice-order
// chunks whose CF loads issue together.  The per-plane sums go to acc
// (stored when one plane per record, else added atomically); k_degrid_finish
// turns them into predictions.
// model value times the phase screen exp(i ph) (FP64, the reference's
// cphase).  Not inlined: the FP64 sine and cosine would otherwise raise the
// register count of k_degrid4's tap loop, which runs them only for records
// with a phase gradient.
__device__ __noinline__ double2 degrid_screen(double2 m, double ph) {
  return cmul(m, cphase(ph));
}
// cphase out of line, for the same reason
__device__ __noinline__ double2 cphase_call(double ph) { return cphase(ph); }

__global__ __launch_bounds__(halo_block) __attribute__((amdgpu_waves_per_eu(4))) void k_degrid4(
  Geometry geo, const GroupInfo* __restrict__ groups,
  const float2* __restrict__ taps, Mueller mu, const unsigned* __restrict__ off_table,
  int nbins, size_t block_cap, const Entry4* __restrict__ entries,
  const unsigned* __restrict__ entry_vis, const VisRec<1>* recs,
  int hx, int hy, const double2* __restrict__ model, double2* __restrict__ acc,
  int one_plane, const double2* __restrict__ wsum, int do_grid, VisRec<1>* out_recs,
  float2* __restrict__ gvis, double2* __restrict__ pred64) {
  // one_plane: each record has exactly one entry, so the lane finishes the
  // prediction itself (the end of degrid_vis and the degridding branch of
  // VisibilityGridder::kernel, src/hpg_core.hpp:643-682, 1136-1169): FP64
  // predictions to pred64, or values written into out_recs when given
  // (residuals, and gvis, when do_grid); recs and out_recs may be the same
  // records, each lane reading its record's fields before writing them.
  // Otherwise the per-plane sums are added into acc for k_degrid_finish.

  extern __shared__ double smem[];
  const int RX = tile + hx;
  const int RY = tile + hy;
  const int R = RX * RY;
  double2* mreg = reinterpret_cast<double2*>(smem);
  unsigned* seg_pref = reinterpret_cast<unsigned*>(smem + 2 * R);
  unsigned* seg_beg = seg_pref + nbins + 1;
  unsigned* part = seg_beg + nbins;

  const unsigned key = xcd_key(blockIdx.x, gridDim.x);  // one block per key
  const int nkeys = geo.ntx * geo.nty * geo.nr * geo.nc;
  for (int bb = threadIdx.x; bb < nbins; bb += halo_block) {
    const unsigned* tab = off_table + size_t(bb) * (nkeys + 1);
    const unsigned s0 = tab[key], s1 = tab[key + 1];
    seg_pref[bb] = s1 - s0;
    seg_beg[bb] = s0;
  }
  __syncthreads();
  const unsigned total = block_exclusive_scan(seg_pref, nbins, part);
  if (total == 0) return;
  if (threadIdx.x == 0) seg_pref[nbins] = total;

  const int ntiles = geo.ntx * geo.nty;
  const unsigned plane = key / ntiles;
  const int t = int(key % ntiles);
  const int x0 = (t % geo.ntx) * tile;
  const int y0 = (t / geo.ntx) * tile;
  const int gpol = int(plane % geo.nr);
  const double2* mplane = model + size_t(plane) * geo.ny * size_t(geo.nx);
  for (int k = threadIdx.x; k < R; k += halo_block) {
    const int ry = k / RX;
    const int rx = k - ry * RX;
    const int xx = x0 + rx, yy = y0 + ry;
    mreg[k] = (xx < geo.nx && yy < geo.ny) ? mplane[size_t(yy) * geo.nx + xx]
                                           : make_double2(0.0, 0.0);
  }
  __syncthreads();

  const int w = threadIdx.x / wave;
  const int lane = threadIdx.x % wave;
  constexpr int nw = halo_block / wave;
  for (unsigned base = w * wave; base < total; base += nw * wave) {
    // issue priority by the passes this wave has left: near the end the
    // waves of the keys with the most entries, which set the kernel's
    // length, go first on their SIMD
    {
      const unsigned left = (total - base + unsigned(nw * wave) - 1u) / unsigned(nw * wave);
      if (left >= 3u)
        __builtin_amdgcn_s_setprio(3);
      else if (left == 2u)
        __builtin_amdgcn_s_setprio(2);
      else
        __builtin_amdgcn_s_setprio(1);
    }
    const unsigned q = base + lane;
    if (q >= total) continue;
    int lo = 0, hi = nbins;  // seg_pref[lo] <= q < seg_pref[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (seg_pref[mid] <= q) lo = mid; else hi = mid;
    }
    const unsigned idx = unsigned(lo) * unsigned(block_cap) + seg_beg[lo] + (q - seg_pref[lo]);
    const Entry4Head eh = entries[idx].h;
    const unsigned i = entry_vis[idx];
    const unsigned pos = eh.pos;
    const int lx = int(pos & 63u);
    const int ly = int((pos >> 6) & 63u);
    const int fxi = int((pos >> 12) & 255u);
    const int fyi = int((pos >> 20) & 255u);
    const bool pos_w = pos & e4_pos_w;
    const bool grad = pos & e4_gradient;
    const int grp = int(eh.gpk & 0xffffu);
    const int cfcube = int(eh.gpk >> 16);
    const GroupInfo g = groups[grp];
    const int sx = g.sx, sy = g.sy;
    // degridding uses the other Mueller matrix and the opposite conjugation
    // of gridding (src/hpg_core.hpp:598-600)
    const int* row = pos_w ? mu.Mc[gpol] : mu.M[gpol];
    const float imf = pos_w ? 1.0f : -1.0f;
    const int m = row[0];
    const bool use = m >= 0 && m < g.nmueller;
    const float2* slice = taps + plane_start(g, geo.nf, int(cfcube), use ? m : 0, fxi, fyi);
    double phi0x = 0.0, phi0y = 0.0, dphix = 0.0, dphiy = 0.0;
    if (grad) {
      const double gxr = recs[i].grad[0];
      const double gyr = recs[i].grad[1];
      phi0x = -gxr * ((sx / 2) * geo.os - (fxi - geo.F));
      phi0y = -gyr * ((sy / 2) * geo.os - (fyi - geo.F));
      dphix = gxr * geo.os;
      dphiy = gyr * geo.os;
    }
    double2 a = make_double2(0.0, 0.0);
    // c' x model for one tap, added to a
    auto add_tap = [&](float2 cc, double2 m, int X, int Y) {
      if (grad) {
        const double phX = phi0x + X * dphix;
        const double phY = phi0y + Y * dphiy;
        m = degrid_screen(m, -phX - phY);
      }
      if (use) {
        cc.y *= imf;
        const double2 p = cmul(cc, m);
        a.x += p.x;
        a.y += p.y;
      }
    };
    // any support: taps in slice order (t = Y * sx + X), halo_chunk at a
    // time, the LDS pixel carried from tap to tap
    auto run_chunks = [&]() {
      const int ntap = sx * sy;
      int cx = 0, cy = 0;          // (X, Y) of the chunk's first tap
      int lc = ly * RX + lx;       // its LDS pixel
      const int wrap = RX - sx;    // pixel step from a row end to the next row
      auto do_chunk = [&](auto full, int t0) {
        constexpr bool FULL = decltype(full)::value;
        bool ok[halo_chunk];
        int Xk[halo_chunk], Yk[halo_chunk];
        double2 mv[halo_chunk];
        float2 c[halo_chunk];
#pragma unroll
        for (int k = 0; k < halo_chunk; ++k) {
          ok[k] = FULL || t0 + k < ntap;
          Xk[k] = cx;
          Yk[k] = cy;
          mv[k] = ok[k] ? mreg[lc] : make_double2(0.0, 0.0);
          const bool eol = ++cx == sx;
          cx = eol ? 0 : cx;
          cy += eol ? 1 : 0;
          lc += eol ? 1 + wrap : 1;
          float2 tv = make_float2(0.0f, 0.0f);
          if (ok[k]) tv = slice[t0 + k];
          c[k] = tv;
        }
#pragma unroll
        for (int k = 0; k < halo_chunk; ++k)
          if (ok[k]) add_tap(c[k], mv[k], Xk[k], Yk[k]);
      };
      int t0 = 0;
      for (; t0 + halo_chunk <= ntap; t0 += halo_chunk) do_chunk(std::true_type{}, t0);
      if (t0 < ntap) do_chunk(std::false_type{}, t0);
    };
    run_chunks();
    if (!one_plane) {
      atomicAdd(&acc[i].x, a.x);
      atomicAdd(&acc[i].y, a.y);
      continue;
    }
    double2 W;
    degrid_norms<1>(geo, g, wsum, mu, pos_w, unsigned(cfcube), fxi, fyi, &W);
    const double2 phasor = cphase_call(recs[i].phase);
    const double2 conj_phasor = make_double2(phasor.x, -phasor.y);
    const double2 d = (W.x != 0.0 || W.y != 0.0) ? W : make_double2(1.0, 0.0);
    const double2 pred_d = cmul(kdiv(a, d), conj_phasor);
    if (pred64) {
      pred64[i] = pred_d;
      continue;
    }
    const float2 pred = narrow(pred_d);
    if (do_grid) {
      float2 val = recs[i].vis[0];
      val.x -= pred.x;
      val.y -= pred.y;
      const float wv = recs[i].w[0];
      if (out_recs) out_recs[i].vis[0] = val;
      gvis[i] = prephase(val, phasor, wv);
    } else if (out_recs) {
      out_recs[i].vis[0] = pred;
    }
  }
}

// predictions from the per-record sums of k_degrid and k_degrid4 (acc null: no
// model, which predicts zero) (the end of degrid_vis and of the degridding
// branch of VisibilityGridder::kernel,
// src/hpg_core.hpp:643-682, 1136-1169), one thread per record
template <int N>
__global__ __launch_bounds__(block) void k_degrid_finish(
  size_t n, Geometry geo, const GroupInfo* __restrict__ groups,
  const double2* __restrict__ wsum, Mueller mu, const double2* __restrict__ acc,
  int do_grid, const VisRec<N>* recs_in, VisRec<N>* recs, float2* __restrict__ gvis,
  double2* __restrict__ pred64) {
  // recs_in and recs may be the same records: each thread reads its
  // record's fields before writing them back; recs null: values not written
  const size_t i = blockIdx.x * (size_t)block + threadIdx.x;
  if (i >= n) return;
  const VisRec<N>& r = recs_in[i];
  const unsigned grp = r.cf_index[1];
  const unsigned cfcube = r.cf_index[0];
  const unsigned gcube = r.grid_cube;
  if (!(grp < unsigned(geo.ngroups) && gcube < unsigned(geo.nc))) return;
  const GroupInfo g = groups[grp];
  if (!(cfcube < unsigned(g.ncube))) return;
  const Coord c = vis_coord(r, geo, g);
  if (!c.inside) return;
  const bool pos_w = r.uvw[2] > 0;
  const double2 phasor = cphase(r.phase);
  double2 W[N];
  degrid_norms<N>(geo, g, wsum, mu, pos_w, cfcube, c.fx + geo.F, c.fy + geo.F, W);
  const double2 conj_phasor = make_double2(phasor.x, -phasor.y);
  float2 pred[N];
  double2 pred_d[N];
  for (int v = 0; v < N; ++v) {
    // a polarization that no row uses has no sum
    bool any = false;
    for (int gpol = 0; gpol < geo.nr; ++gpol) {
      const int m = pos_w ? mu.Mc[gpol][v] : mu.M[gpol][v];
      any |= m >= 0 && m < g.nmueller;
    }
    const double2 d = (W[v].x != 0.0 || W[v].y != 0.0) ? W[v] : make_double2(1.0, 0.0);
    const double2 a = any && acc ? acc[i * N + v] : make_double2(0.0, 0.0);
    pred_d[v] = acc ? cmul(kdiv(a, d), conj_phasor) : a;
    pred[v] = narrow(pred_d[v]);
  }
  if (pred64) {
    for (int v = 0; v < N; ++v) pred64[i * N + v] = pred_d[v];
    return;
  }
  for (int v = 0; v < N; ++v) {
    if (do_grid) {
      float2 val = r.vis[v];
      val.x -= pred[v].x;
      val.y -= pred[v].y;
      if (recs) recs[i].vis[v] = val;
      gvis[i * N + v] = prephase(val, phasor, r.w[v]);
    } else if (recs) {
      recs[i].vis[v] = pred[v];
    }
  }
}

// ---- finishing passes ------------------------------------------------------

template <typename T>
__global__ void k_normalize(
  T* __restrict__ grid, const double* __restrict__ weights, double wfactor,
  size_t plane_size, size_t count) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k >= count) return;
  const double d = wfactor * weights[k / plane_size];
  T g = grid[k];
  g.x = double(g.x) / d;
  g.y = double(g.y) / d;
  grid[k] = g;
}

// the finishing chain's one elementwise pass before its FFT: each value
// divided by wfactor * its plane's weight (when weights is given: the
// GridNormalizer's FP64 division, src/hpg_core.hpp:1849-1860), times s,
// and negated where x + y is odd (modulate: for even nx, ny the FFT of
// x (-1)^(x+y) is the FFT of x shifted by half the grid on both axes, so
// the shift that follows the FFT needs no pass of its own).  The launch
// is (x blocks, row y, plane), so no index needs a division.
template <typename T>
__global__ void k_finish_pre(
  T* __restrict__ grid, const double* __restrict__ weights, double wfactor, double s,
  int modulate, int nx, int ny) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= nx) return;
  const int y = blockIdx.y;
  const size_t plane = blockIdx.z;
  T* p = grid + (plane * size_t(ny) + size_t(y)) * size_t(nx) + x;
  T g = *p;
  double vx = double(g.x), vy = double(g.y);
  if (weights) {
    const double d = wfactor * weights[plane];
    vx /= d;
    vy /= d;
  }
  const double f = modulate && ((x + y) & 1) ? -s : s;
  g.x = vx * f;
  g.y = vy * f;
  *p = g;
}

template <typename T>
__global__ void k_scale(T* __restrict__ grid, double s, size_t count) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k >= count) return;
  T g = grid[k];
  g.x = double(g.x) * s;
  g.y = double(g.y) * s;
  grid[k] = g;
}

// even sizes: FORWARD and BACKWARD both swap (x, y) with
// ((x + nx/2) mod nx, y + ny/2) -- one thread per pair
template <typename T>
__global__ void k_shift_even(T* __restrict__ grid, int nx, int ny, size_t nplanes) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t half = size_t(nx) * (ny / 2);
  if (k >= half * nplanes) return;
  const size_t p = k / half;
  const int r = int(k % half);
  const int x = r % nx;
  const int y = r / nx;
  T* plane = grid + p * size_t(nx) * ny;
  const size_t a = size_t(y) * nx + x;
  const size_t b = size_t(y + ny / 2) * nx + (x + nx / 2) % nx;
  const T t = plane[a];
  plane[a] = plane[b];
  plane[b] = t;
}

template <typename T>
__global__ void k_shift_general(
  const T* __restrict__ src, T* __restrict__ dst, int nx, int ny, int sx, int sy,
  size_t count) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k >= count) return;
  const size_t ps = size_t(nx) * ny;
  const size_t p = k / ps;
  const int r = int(k % ps);
  const int x = r % nx;
  const int y = r / nx;
  dst[p * ps + size_t((y + sy) % ny) * nx + (x + sx) % nx] = src[k];
}

__global__ void k_widen(const float2* __restrict__ s, double2* __restrict__ d, size_t n) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k < n) d[k] = make_double2(double(s[k].x), double(s[k].y));
}
__global__ void k_narrow(const double2* __restrict__ s, float2* __restrict__ d, size_t n) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k < n) d[k] = make_float2(float(s[k].x), float(s[k].y));
}

inline unsigned blocks_for(size_t n, int b = block) {
  return unsigned((n + b - 1) / b);
}

// launch(first block, blocks) for parts of a grid of workgroups: HIP counts a
// launch's threads in 32 bits, and a launch of more runs what is left of them
// modulo 2^32
template <typename F>
hipError_t in_launches(unsigned long long blocks, int threads, F launch) {
  const unsigned long long most = 0xffffffffull / unsigned(threads);
  hipError_t e = hipSuccess;
  for (unsigned long long first = 0; first < blocks && e == hipSuccess; first += most) {
    launch(first, unsigned(std::min(most, blocks - first)));
    e = hipGetLastError();
  }
  return e;
}

}  // namespace

// ---- launchers -------------------------------------------------------------

hipError_t launch_cf_relayout(
  hipStream_t s, const float2* staging, const unsigned ext[4],
  const GroupInfo& gi, const CfElements& ce, int os, int F, int nf, bool planar,
  float2* taps) {
  const long long total =
    (long long)gi.ncube * gi.nmueller * nf * nf * gi.sx * gi.sy;
  if (total == 0) return hipSuccess;
  // support columns whose window fits LDS
  auto lds = [&](int xc) {
    return (size_t(xc - 1) * os + nf) * gi.nmueller * sizeof(float2);
  };
  int xc = std::min(gi.sx, 8);
  while (xc > 1 && lds(xc) > relayout_lds) --xc;
  const int nxc = (gi.sx + xc - 1) / xc;
  const unsigned long long blocks = (unsigned long long)nxc * gi.sy * nf * gi.ncube;
  if (lds(xc) <= relayout_lds)
    return in_launches(blocks, relayout_block, [&](unsigned long long first, unsigned nb) {
      hipLaunchKernelGGL(
        k_cf_relayout_lds, dim3(nb), dim3(relayout_block), lds(xc), s, staging, ext[0], ext[1],
        ext[2], gi, ce, os, F, nf, int(planar), taps, xc, nxc, (long long)first);
    });
  return in_launches((total + block - 1) / block, block,
                     [&](unsigned long long first, unsigned nb) {
    hipLaunchKernelGGL(
      k_cf_relayout, dim3(nb), dim3(block), 0, s, staging, ext[0], ext[1], ext[2], gi, ce, os, F,
      nf, int(planar), taps, total, (long long)first);
  });
}

hipError_t launch_cf_wsum(
  hipStream_t s, const GroupInfo& gi, int nf, bool planar, const float2* taps,
  double2* wsum) {
  const int nm = gi.nmueller;
  const int per = !planar && nm > 0 && nm <= wave && (nm & (nm - 1)) == 0 ? nm : 0;
  const long long ns = (long long)gi.ncube * (per ? 1 : nm) * nf * nf;
  if (ns == 0) return hipSuccess;
  const long long values = (long long)gi.sx * gi.sy * (per ? per : 1);
  const int threads = values <= 1024 ? wave : values <= 8192 ? 256 : wsum_block;
  return in_launches(ns, threads, [&](unsigned long long first, unsigned nb) {
    hipLaunchKernelGGL(k_cf_wsum, dim3(nb), dim3(threads), 0, s, gi, nf, taps, wsum, per,
                       int(planar), (long long)first);
  });
}

size_t scan_temp_bytes(size_t nkeys) {
  size_t bytes = 0;
  (void)hipcub::DeviceScan::ExclusiveSum(
    nullptr, bytes, static_cast<unsigned*>(nullptr),
    static_cast<unsigned*>(nullptr), int(nkeys + 1));
  return bytes;
}

hipError_t launch_scan(hipStream_t s, size_t nkeys, CallBuffers& cb) {
  size_t bytes = cb.scan_temp_bytes;
  hipError_t e = hipcub::DeviceScan::ExclusiveSum(
    cb.scan_temp, bytes, cb.hist, cb.offsets, int(nkeys + 1), s);
  if (e != hipSuccess) return e;
  return hipMemcpyAsync(
    cb.cursor, cb.offsets, nkeys * sizeof(unsigned), hipMemcpyDeviceToDevice, s);
}

hipError_t launch_count(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool do_grid, CallBuffers& cb,
  double* weights) {
  if (n == 0) return hipSuccess;
  if (npol != 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(
    k_count, dim3(std::min(unsigned(blocks_for(n)), count_blocks_max)),
    dim3(block), 0, s,
    static_cast<const VisRec<1>*>(cb.vis), n, geo, cf.groups, cf.wsum, mu,
    int(update_weights), int(do_grid), cb.hist, weights, cb.invalid_count);
  return hipGetLastError();
}

// records of a workgroup that counts in LDS: all of a small batch (which one
// workgroup then prepares whole), 1024 (a record a thread) where 2048 would leave
// most of the chip idle (10,000 records, two polarizations, 256^2: 90 -> 84 us), then
// 2048, or more so that there are at most 512 workgroups
size_t patch_batch(size_t n) {
  if (n > 2048 && n <= 16384) return 1024;
  return std::max<size_t>(2048, ((n + 511) / 512 + 1023) / 1024 * 1024);
}
// workgroups of up to n records a call at most
size_t patch_batches(size_t n) {
  return std::min<size_t>(std::max<size_t>((n + 2047) / 2048, 16), 512);
}

// Bins: at most half of the items that one workgroup counts (its global
// atomics, one for each of its bins), not fewer than 1024: the second level
// has one workgroup per bin, which of 1e6 records in 256 bins around a dense
// uv core took 58 us and of 1024 bins 16.  Keys beyond patch_local_keys bins
// of 2^sort_low_bits_max lose their lowest bits.
SortKeys sort_plan(unsigned long long keys, size_t batch) {
  const unsigned long long most =
    std::clamp<unsigned long long>(batch / 2, 1024, patch_local_keys);
  SortKeys sk{};
  auto bins = [&]() { return ((keys - 1) >> (sk.low_bits + sk.drop_bits)) + 1; };
  while (sk.low_bits < sort_low_bits_max && bins() > most) ++sk.low_bits;
  while (bins() > (unsigned long long)patch_local_keys) ++sk.drop_bits;
  sk.bins = int(bins());
  return sk;
}

size_t sort_bins_entries(size_t n) {
  return (2 + patch_batches(n)) * (patch_local_keys + 1);
}

// the bins' offsets and the pairs of n keys, from the counts in cb.sort_bins
hipError_t launch_sort_place(hipStream_t s, size_t n, size_t batch, const SortKeys& sk,
                             const CallBuffers& cb, const unsigned* keys, unsigned* order,
                             uint2* pairs) {
  unsigned* hist = cb.sort_bins;
  unsigned* offsets = hist + patch_local_keys + 1;
  const unsigned* table = offsets + patch_local_keys + 1;
  hipLaunchKernelGGL(k_patch_scan, dim3(1), dim3(patch_scan_threads), 0, s, sk.bins, hist, offsets,
                     static_cast<unsigned*>(nullptr), PatchSplit{});
  hipLaunchKernelGGL(k_sort_place, dim3(unsigned((n + batch - 1) / batch)),
                     dim3(patch_local_threads), 0, s, n, sk, unsigned(batch), keys, offsets, table,
                     order, pairs);
  return hipGetLastError();
}

hipError_t launch_tally(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, double* weights) {
  if (n == 0) return hipSuccess;
  if (npol != 1 || n * size_t(geo.nr) > cb.tally_capacity || n > cb.sort_capacity)
    return hipErrorInvalidValue;
  const size_t nkeys = 4 * size_t(geo.ntx) * geo.nty * geo.nr * geo.nc;
  const size_t batch = patch_batch(n);
  const SortKeys sk = sort_plan(nkeys, batch);
  if (sk.drop_bits) return hipErrorInvalidValue;
  unsigned* hist = cb.sort_bins;
  unsigned* offsets = hist + patch_local_keys + 1;
  unsigned* table = offsets + patch_local_keys + 1;
  uint2* pairs = static_cast<uint2*>(cb.tally_keys);
  unsigned* keys = reinterpret_cast<unsigned*>(pairs + cb.tally_capacity);
  Entry4* tally = static_cast<Entry4*>(cb.tally_entries);
  hipLaunchKernelGGL(k_zero, dim3(blocks_for(size_t(sk.bins))), dim3(block), 0, s, hist,
                     size_t(sk.bins));
  hipLaunchKernelGGL(
    k_tally, dim3(unsigned((n + batch - 1) / batch)), dim3(patch_local_threads), 0, s,
    static_cast<const VisRec<1>*>(cb.vis), n, geo, cf.groups, cf.wsum, mu,
    int(update_weights), int(gvis_ready), int(src == GvisSource::Adjoint), cb.gvis, residuals,
    sk, unsigned(batch), hist, table, weights, cb.invalid_count, tally, keys);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  e = launch_sort_place(s, n * size_t(geo.nr), batch * size_t(geo.nr), sk, cb, keys, nullptr,
                        pairs);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(
    k_tally_sort, dim3(unsigned(sk.bins)), dim3(sort_threads),
    (size_t(1) << sk.low_bits) * sizeof(unsigned), s, sk.low_bits, nkeys, geo.nr, offsets, pairs,
    tally, cb.offsets, static_cast<Entry4*>(cb.stream_entries), cb.entry_vis);
  return hipGetLastError();
}

hipError_t launch_emit(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool gvis_ready, GvisSource src, const double2* residuals,
  CallBuffers& cb) {
  if (n == 0) return hipSuccess;
  const int adj = src == GvisSource::Adjoint;
  if (npol != 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(
    k_emit, dim3(blocks_for(n)), dim3(block), 0, s,
    static_cast<const VisRec<1>*>(cb.vis), n, geo, cf.groups, cf.wsum, mu,
    int(gvis_ready), adj, cb.gvis, residuals, cb.cursor,
    static_cast<Entry4*>(cb.stream_entries), cb.entry_vis);
  return hipGetLastError();
}

int bin_blocks_for(size_t n) { return int((n + bin_records - 1) / bin_records); }
size_t bin_block_records() { return bin_records; }
int bin_keys_limit() { return bin_keys_max; }
int bin_quad_keys_limit() { return bin_quad_keys_max; }
int tile_bins_limit() { return tile_bins_max; }

hipError_t launch_bin(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, size_t block_cap, double* weights,
  bool degrid_pass, void* copy_records, bool quad_keys) {
  if (n == 0) return hipSuccess;
  if (copy_records && !degrid_pass) return hipErrorInvalidValue;
  if (quad_keys && degrid_pass) return hipErrorInvalidValue;
  const int adj = src == GvisSource::Adjoint;
  const int dg = degrid_pass;
  const unsigned nb = unsigned(bin_blocks_for(n));
  if (npol != 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(
    k_bin, dim3(nb), dim3(bin_threads), 0, s,
    static_cast<const VisRec<1>*>(cb.vis), n, geo, cf.groups, cf.wsum, mu,
    int(update_weights), int(gvis_ready), adj, dg, cb.gvis, residuals,
    cb.off_table, cb.stream_entries, cb.entry_vis, block_cap, weights,
    cb.invalid_count, static_cast<VisRec<1>*>(copy_records), int(quad_keys));
  return hipGetLastError();
}

size_t halo_entry_bytes() { return sizeof(Entry4); }
size_t halo_pixels_per_key(int hx, int hy) { return size_t(halo_pixels(hx, hy)); }
int halo_tile_limit() { return tile; }
size_t halo_lds_bytes(int hx, int hy, int nbins) {
  const size_t r = size_t(tile + hx) * (tile + hy);
  return r * 16
    + sizeof(unsigned)
      * (2 * size_t(nbins) + 1 + halo_block / wave + 1 + halo_classes + halo_sched);
}

// the halo pass after a haloed-tile kernel
hipError_t launch_halo(
  hipStream_t s, int mode, size_t nkeys, const Geometry& geo, const CallBuffers& cb,
  int hx, int hy, void* grid) {
  const size_t zone = size_t(hy) * tile + size_t(tile - hy) * hx;
  const size_t count = nkeys * zone;
  if (count == 0) return hipSuccess;
  if (mode == 0)
    hipLaunchKernelGGL(
      k_halo<double2>, dim3(blocks_for(count)), dim3(block), 0, s, geo, hx, hy,
      cb.halo, cb.halo_set, nkeys, static_cast<double2*>(grid));
  else
    hipLaunchKernelGGL(
      k_halo<float2>, dim3(blocks_for(count)), dim3(block), 0, s, geo, hx, hy,
      cb.halo, cb.halo_set, nkeys, static_cast<float2*>(grid));
  return hipGetLastError();
}

int sub_bins_limit() { return sub_bins_max; }
bool sub_supported(int hx, int hy) { return hx >= 0 && hy >= 0 && hx < 8 && hy < 8; }

hipError_t launch_tile_sub(
  hipStream_t s, int npol, size_t n, size_t ntile_keys, const Geometry& geo, const DeviceCF& cf,
  size_t taps_bytes, bool uni, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, void* grid, bool global_bins) {
  if (ntile_keys == 0 || n == 0) return hipSuccess;
  const int nb = global_bins ? 1 : bin_blocks_for(n);
  // segment starts are 16-bit offsets within a bin block; CF taps are
  // addressed by 32-bit byte offsets
  if (npol != 1 || !cf.planar || !sub_supported(hx, hy) || taps_bytes > 0xffffffffull)
    return hipErrorInvalidValue;
  if (!global_bins && (nb > sub_bins_max || block_cap > 65536)) return hipErrorInvalidValue;
  const unsigned* offs = global_bins ? cb.offsets : cb.off_table;
  const int Q = (quad_edge + hx) * (quad_edge + hy);
  const int px = (Q + wave - 1) / wave;  // 4 .. 9
  const int pxc = px <= 4 ? 4 : px <= 6 ? 6 : px <= 8 ? 8 : 9;
  const size_t dyn = size_t(sub_waves) * pxc * wave * sizeof(float2);
#define HPGX_SUB_G(PX, PK, GB)                                                 \
  hipLaunchKernelGGL(                                                          \
    uni ? (k_sub<PX, true, PK, GB>) : (k_sub<PX, false, PK, GB>),              \
    dim3(unsigned(ntile_keys)), dim3(sub_block), dyn, s,                       \
    geo, cf.groups, cf.taps, unsigned(taps_bytes), mu, offs, nb,               \
    block_cap,                                                                 \
    static_cast<const Entry4*>(cb.stream_entries), cb.entry_vis,               \
    static_cast<const VisRec<1>*>(cb.vis), hx, hy, static_cast<float2*>(grid), \
    cb.halo, cb.halo_set)
#define HPGX_SUB(PX, PK)                                                       \
  do {                                                                         \
    if (global_bins) HPGX_SUB_G(PX, PK, true);                                 \
    else HPGX_SUB_G(PX, PK, false);                                            \
  } while (0)
#define HPGX_SUB_PX(PK)                                                        \
  switch (pxc) {                                                               \
  case 4: HPGX_SUB(4, PK); break;                                              \
  case 6: HPGX_SUB(6, PK); break;                                              \
  case 8: HPGX_SUB(8, PK); break;                                              \
  default: HPGX_SUB(9, PK); break;                                             \
  }
  // one word per slot: region pixels below sub_pk_flip, slices addressed
  // by tap index below sub_pk_taps
  static_assert(9 * wave < int(sub_pk_flip), "region pixel in the packed word");
  if (taps_bytes / sizeof(float2) < sub_pk_taps) HPGX_SUB_PX(true) else HPGX_SUB_PX(false)
#undef HPGX_SUB_PX
#undef HPGX_SUB
#undef HPGX_SUB_G
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_halo(s, 1, ntile_keys, geo, cb, hx, hy, grid);
}

hipError_t launch_tile_halo(
  hipStream_t s, int npol, int mode, int acc, size_t n, size_t nkeys, const Geometry& geo,
  const DeviceCF& cf, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, void* grid, bool global_bins) {
  if (nkeys == 0 || n == 0) return hipSuccess;
  if (hx < 0 || hy < 0 || hx >= tile || hy >= tile) return hipErrorInvalidValue;
  // global bins: one contiguous range per key, read as a single bin block
  // whose offset-table row is the scanned offsets
  const int nb = global_bins ? 1 : bin_blocks_for(n);
  const unsigned* table = global_bins ? cb.offsets : cb.off_table;
  const size_t lds = halo_lds_bytes(hx, hy, nb);
  if (lds > 65536) return hipErrorInvalidValue;
#define HPGX_TILE4(MD, AC)                                                     \
  hipLaunchKernelGGL(                                                          \
    (k_tile4<MD, AC>), dim3(unsigned(nkeys)), dim3(halo_block), lds, s,                           \
    geo, cf.groups, cf.taps, mu, table, nb, block_cap,                         \
    static_cast<const Entry4*>(cb.stream_entries), cb.entry_vis,            \
    static_cast<const VisRec<1>*>(cb.vis), hx, hy, grid, cb.halo, cb.halo_set)
  if (npol != 1 || !cf.planar) return hipErrorInvalidValue;
  if (mode == 0)
    HPGX_TILE4(0, acc_f64);
  else if (acc == 0)
    HPGX_TILE4(1, acc_f64);
  else
    HPGX_TILE4(1, acc_f32_cas);
#undef HPGX_TILE4
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_halo(s, mode, nkeys, geo, cb, hx, hy, grid);
}

int patch_tiles_x(const Geometry& geo) {
  return (geo.nx + patch_tile_x(patch_lanes(geo.nr)) - 1) / patch_tile_x(patch_lanes(geo.nr));
}
int patch_tiles_y(const Geometry& geo) {
  return (geo.ny + patch_tile_y(patch_lanes(geo.nr)) - 1) / patch_tile_y(patch_lanes(geo.nr));
}
size_t patch_keys(const Geometry& geo) {
  return size_t(patch_tiles_x(geo)) * patch_tiles_y(geo) * geo.nc;
}
size_t patch_table_entries(const Geometry& geo, size_t n) {
  const size_t keys = patch_keys(geo);
  return keys <= size_t(patch_local_keys) ? patch_batches(n) * keys : 0;
}
// slots for the split lists of so many entries in all, and their memory
size_t patch_split_slots(size_t entries) {
  return std::min<size_t>(patch_slots_max, entries * 3 / (2 * patch_chunk_min));
}
size_t patch_split_bytes(size_t slots) {
  return slots * (patch_values * sizeof(double) + sizeof(uint2) + 2 * sizeof(unsigned)) + 256;
}
size_t patch_rec_bytes(int npol) {
  switch (npol) {
  case 1: return sizeof(PatchRec<1>);
  case 2: return sizeof(PatchRec<2>);
  case 3: return sizeof(PatchRec<3>);
  default: return sizeof(PatchRec<4>);
  }
}
size_t patch_tiles_per_footprint(int nr, int max_sx, int max_sy) {
  const int tw = patch_tile_x(patch_lanes(nr)), th = patch_tile_y(patch_lanes(nr));
  return size_t((max_sx - 1 + tw - 1) / tw + 1) * size_t((max_sy - 1 + th - 1) / th + 1);
}

bool patch_offsets_fit(const GroupInfo& g) {
  const size_t rows = std::min(g.sy, 2 * patch_h(1));
  return rows * size_t(g.sx) * size_t(g.nmueller) * sizeof(float2) < 0xfffffff0ull;
}

// how the rows of both signs of w take their elements of a slice
int patch_kind(int npol, const Geometry& geo, const DeviceCF& cf, const Mueller& mu) {
  bool one = true, full = npol % 2 == 0 && cf.even_nm;
  for (int s = 0; s < 2; ++s)
    for (int r = 0; r < geo.nr; ++r) {
      const int* row = s ? mu.M[r] : mu.Mc[r];
      int used = 0;
      for (int v = 0; v < npol; ++v) {
        used += row[v] >= 0;
        full = full && row[0] >= 0 && row[0] % 2 == 0 && row[v] == row[0] + v
          && row[v] < cf.min_nm;
      }
      one = one && used <= 1;
    }
  return one ? patch_one : full ? patch_full : patch_any;
}

hipError_t launch_patch(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, bool update_weights, bool gvis_ready, GvisSource src,
  const double2* residuals, CallBuffers& cb, double* weights, int mode, bool halo_rounds,
  void* grid) {
  if (n == 0) return hipSuccess;
  if (n > cb.patch_capacity) return hipErrorInvalidValue;
  const int P = patch_lanes(geo.nr);
  const int ptx = patch_tiles_x(geo), pty = patch_tiles_y(geo);
  const size_t keys = patch_keys(geo);
  const int kind = patch_kind(npol, geo, cf, mu);
  const bool local = keys <= size_t(patch_local_keys);
  PatchSplit ps{};
  ps.slots = unsigned(std::min(
    cb.patch_split_slots,
    patch_split_slots(n * patch_tiles_per_footprint(geo.nr, cf.max_sx, cf.max_sy))));
  ps.base = static_cast<char*>(cb.patch_split);
  const size_t batch = patch_batch(n);
  const unsigned nb = local ? unsigned((n + batch - 1) / batch) : 0u;
  if (local && nb * keys > cb.patch_table_capacity) return hipErrorInvalidValue;
  const bool one = local && nb == 1;  // one workgroup prepares, scans and lists
  // a kernel, not a memset: a captured graph may replay it
  if (!one)
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(keys + 1)), dim3(block), 0, s, cb.hist, keys + 1);
#define HPGX_PREP(NP)                                                          \
  hipLaunchKernelGGL(                                                          \
    local ? (k_patch_prep<NP, true>) : (k_patch_prep<NP, false>),              \
    dim3(local ? nb : std::min(blocks_for(n), count_blocks_max)),              \
    dim3(local ? patch_local_threads : block), 0, s,                           \
    static_cast<const VisRec<NP>*>(cb.vis), n, geo, cf.groups, cf.wsum, mu,    \
    int(update_weights), int(gvis_ready), int(src == GvisSource::Adjoint), cb.gvis, residuals, \
    ptx, pty, patch_tile_x(P), patch_tile_y(P), static_cast<PatchRec<NP>*>(cb.patch_recs), \
    cb.hist, weights, cb.invalid_count, unsigned(batch), cb.patch_table,       \
    one ? cb.offsets : nullptr, cb.cursor, cb.patch_list, ps)
#define HPGX_LIST(NP)                                                          \
  hipLaunchKernelGGL(                                                          \
    local ? (k_patch_list<NP, true>) : (k_patch_list<NP, false>),              \
    dim3(local ? nb : blocks_for(n)), dim3(local ? patch_local_threads : block), 0, s, n, \
    geo.nc, ptx, pty,                                                          \
    patch_tile_x(P), patch_tile_y(P), static_cast<const PatchRec<NP>*>(cb.patch_recs), \
    cb.hist, cb.offsets, cb.patch_list, unsigned(batch), cb.patch_table)
#define HPGX_PATCH_P(NP, PP, KD)                                               \
  e = in_launches(ps.slots + keys, patch_split(PP) * patch_block,              \
                  [&](unsigned long long first, unsigned blocks) {             \
    hipLaunchKernelGGL(                                                        \
      (k_patch<NP, PP, KD>), dim3(blocks), dim3(patch_split(PP) * patch_block), 0, s, \
      geo, cf.taps, mu, mode, take, ptx, pty, cb.offsets, order, cb.patch_list, \
      static_cast<const PatchRec<NP>*>(cb.patch_recs),                         \
      static_cast<const VisRec<NP>*>(cb.vis), grid, unsigned(first), ps);      \
  })
#define HPGX_PATCH_K(NP, KD)                                                   \
  do {                                                                         \
    if (P == 1) HPGX_PATCH_P(NP, 1, KD);                                       \
    else if (P == 2) HPGX_PATCH_P(NP, 2, KD);                                  \
    else HPGX_PATCH_P(NP, 4, KD);                                              \
  } while (0)
  switch (npol) {
  case 1: HPGX_PREP(1); break;
  case 2: HPGX_PREP(2); break;
  case 3: HPGX_PREP(3); break;
  case 4: HPGX_PREP(4); break;
  default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const unsigned* order = nullptr;
  if (one) {
    order = cb.cursor;
  } else if (local) {
    order = cb.cursor;
    hipLaunchKernelGGL(k_patch_scan, dim3(1), dim3(patch_scan_threads), 0, s, int(keys), cb.hist,
                       cb.offsets, cb.cursor, ps);
    e = hipGetLastError();
  } else {
    size_t bytes = cb.scan_temp_bytes;
    e = hipcub::DeviceScan::ExclusiveSum(cb.scan_temp, bytes, cb.hist, cb.offsets, int(keys + 1),
                                         s);
    if (ps.slots && e == hipSuccess) {
      hipLaunchKernelGGL(k_zero, dim3(1), dim3(block), 0, s, ps.ctl(), size_t(2));
      order = cb.cursor;
      hipLaunchKernelGGL(k_patch_split, dim3(blocks_for(keys)), dim3(block), 0, s, keys,
                         cb.offsets, cb.cursor, ps);
      e = hipGetLastError();
    }
  }
  if (e != hipSuccess) return e;
  if (!one) {
    switch (npol) {
    case 1: HPGX_LIST(1); break;
    case 2: HPGX_LIST(2); break;
    case 3: HPGX_LIST(3); break;
    default: HPGX_LIST(4); break;
    }
  }
  // FP32 grids of supports below a tile round twice a pixel, as the haloed tiles
  // do: once with the sum of the tile's records, once with its neighbours'
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  for (int take = halo_rounds ? patch_own : patch_all; take <= (halo_rounds ? patch_others : patch_all);
       ++take) {
    switch (npol) {
    case 1:
      if (cf.planar) HPGX_PATCH_K(1, patch_plane);
      else HPGX_PATCH_K(1, patch_one);
      break;
    case 2:
      if (kind == patch_one) HPGX_PATCH_K(2, patch_one);
      else if (kind == patch_full) HPGX_PATCH_K(2, patch_full);
      else HPGX_PATCH_K(2, patch_any);
      break;
    case 3:
      if (kind == patch_one) HPGX_PATCH_K(3, patch_one);
      else HPGX_PATCH_K(3, patch_any);
      break;
    default:
      if (kind == patch_one) HPGX_PATCH_K(4, patch_one);
      else if (kind == patch_full) HPGX_PATCH_K(4, patch_full);
      else HPGX_PATCH_K(4, patch_any);
      break;
    }
    if (e != hipSuccess) return e;
  }
#undef HPGX_PATCH_K
#undef HPGX_PATCH_P
#undef HPGX_LIST
#undef HPGX_PREP
  return hipSuccess;
}

// Every tile looks through all records: their product, at 2^21 still the faster
// (supports of 7, binned and in one launch: 2000 records on 1024 tiles 38.8, 35.1 us;
// 3000 42.9, 44.7).  And not where few tiles hold them all, which is even for wide
// supports (1500 of 25 on 16 tiles 106, 107 us; narrow ones would still gain: 2000 of 7
// on 4 tiles 39.7, 25.5).
bool direct_ok(size_t n, const Geometry& geo) {
  const size_t tiles = size_t(geo.ntx) * geo.nty * geo.nc;
  return n <= direct_records && n * tiles <= (size_t(1) << 21) && n <= 256 * tiles;
}

hipError_t launch_direct(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf, const Mueller& mu,
  bool update_weights, bool gvis_ready, GvisSource src, const double2* residuals,
  const CallBuffers& cb, double* weights, double2* grid) {
  if (n == 0) return hipSuccess;
  if (npol != 1 || !cf.planar || n > direct_records || geo.nr > 4) return hipErrorInvalidValue;
  const size_t lds = size_t(geo.nr) * 2 * direct_plane * sizeof(double);
  const DirectArgs args{cf.groups, cf.wsum, cb.gvis, residuals, weights, cb.invalid_count,
                        int(update_weights), int(gvis_ready), int(src == GvisSource::Adjoint)};
  hipLaunchKernelGGL(
    k_direct, dim3(unsigned(size_t(geo.ntx) * geo.nty * geo.nc)), dim3(direct_block), lds, s, geo,
    cf.taps, mu, static_cast<const VisRec<1>*>(cb.vis), unsigned(n), args, grid);
  return hipGetLastError();
}

hipError_t launch_degrid_tiles(
  hipStream_t s, int npol, size_t n, size_t nkeys, const Geometry& geo,
  const DeviceCF& cf, const Mueller& mu, const CallBuffers& cb, size_t block_cap,
  int hx, int hy, const double2* model, double2* acc, bool one_plane, bool do_grid,
  void* out_recs, double2* pred64) {
  if (nkeys == 0 || n == 0) return hipSuccess;
  if (hx < 0 || hy < 0 || hx >= tile || hy >= tile) return hipErrorInvalidValue;
  const int nb = bin_blocks_for(n);
  const size_t lds = halo_lds_bytes(hx, hy, nb);
  if (lds > 65536) return hipErrorInvalidValue;
  if (npol != 1 || !cf.planar) return hipErrorInvalidValue;
  hipLaunchKernelGGL(
    k_degrid4, dim3(unsigned(nkeys)), dim3(halo_block), lds, s, geo, cf.groups, cf.taps, mu,
    cb.off_table, nb, block_cap, static_cast<const Entry4*>(cb.stream_entries), cb.entry_vis,
    static_cast<const VisRec<1>*>(cb.vis), hx, hy, model, acc, int(one_plane), cf.wsum,
    int(do_grid), static_cast<VisRec<1>*>(out_recs), cb.gvis, pred64);
  return hipGetLastError();
}

hipError_t launch_degrid_finish(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, const double2* acc, bool do_grid, const void* records,
  void* out_records, CallBuffers& cb, double2* pred64) {
  if (n == 0) return hipSuccess;
  const void* in = records;
#define HPGX_DFIN(NP)                                                          \
  hipLaunchKernelGGL(                                                          \
    k_degrid_finish<NP>, dim3(blocks_for(n)), dim3(block), 0, s, n, geo,       \
    cf.groups, cf.wsum, mu, acc, int(do_grid),                                 \
    static_cast<const VisRec<NP>*>(in), static_cast<VisRec<NP>*>(out_records), \
    cb.gvis, pred64)
  switch (npol) {
  case 1: HPGX_DFIN(1); break;
  case 2: HPGX_DFIN(2); break;
  case 3: HPGX_DFIN(3); break;
  case 4: HPGX_DFIN(4); break;
  default: return hipErrorInvalidValue;
  }
#undef HPGX_DFIN
  return hipGetLastError();
}

size_t degrid_rec_bytes() { return sizeof(DegridRec); }

hipError_t launch_degrid(
  hipStream_t s, int npol, size_t n, const Geometry& geo, const DeviceCF& cf,
  const Mueller& mu, const double2* model, bool do_grid, CallBuffers& cb, double2* pred64,
  const void* records, void* out_records) {
  if (n == 0) return hipSuccess;
  if (!model)
    return launch_degrid_finish(s, npol, n, geo, cf, mu, nullptr, do_grid, records, out_records,
                                cb, pred64);
  if (cb.order_capacity < n || cb.sort_capacity < n || n > 0xffffffffull)
    return hipErrorInvalidValue;
  const int P = patch_lanes(geo.nr);
  int kind = patch_kind(npol, geo, cf, mu);
  bool same_rows = true;
  for (int v = 0; v < npol; ++v) {
    int used = 0, used_c = 0;
    for (int r = 0; r < geo.nr; ++r) {
      same_rows = same_rows && mu.M[r][v] == mu.Mc[r][v];
      used += mu.M[r][v] >= 0;
      used_c += mu.Mc[r][v] >= 0;
    }
    if (kind == patch_one && (used > 1 || used_c > 1)) kind = patch_any;
  }
  const unsigned* order = nullptr;
  // The records in CF-slice order; where the batch is dense, region by region,
  // whose model then stays in L2: the largest square of 2^k pixels whose model
  // (all rows, with the supports' halo) fits half of an XCD's 4 MB, each XCD
  // taking a contiguous share of the records.  Dense: a region's records read
  // its model four times over at least, and what their shorter runs of one
  // slice read more of the CF is no more than the model reads that leave HBM.
  // Degridding kernel without and with regions: 1e6 records of supports 9-33,
  // one element a row, 2048^2: 5.7 -> 2.9 ms; 300,000 on 1024^2: 1.45 -> 0.92;
  // 300,000 of 7-17, two polarizations, 2 x 1500^2: 287 -> 222 us.  (Contiguous
  // shares without regions would give the XCDs different CF groups, the large
  // supports to one: 14 -> 22 ms on 64 groups.)
  // Grid cubes one after the other while the keys fit 32 bits; no order if the
  // slices alone do not.
  const unsigned long long stride = (unsigned long long)std::max(cf.max_ncube, 1) * cf.nf * cf.nf;
  const unsigned long long slices = stride * (unsigned long long)cf.ngroups;
  constexpr unsigned long long key_limit = 0xffffffffull;
  constexpr double l2_bytes = 2.0 * (1 << 20);
  const double density = double(n) / (double(geo.nx) * geo.ny * geo.nc);
  const double support = std::max(cf.max_sx, cf.max_sy);
  int region_sh = 5;
  while (std::pow(std::ldexp(1.0, region_sh + 1) + support, 2) * geo.nr * sizeof(double2) <= l2_bytes)
    ++region_sh;
  {
    const double in_region = std::ldexp(density, 2 * region_sh);
    const double cf_bytes = double(kind == patch_one ? 1 : npol) * sizeof(float2);
    const double run = std::max(1.0, in_region / double(slices));
    const double run_all = std::max(1.0, double(n) / (double(slices) * geo.nc));
    const double edge = std::ldexp(1.0, region_sh) + support;
    if (cf_bytes / run > sizeof(double2) + cf_bytes / run_all
        || in_region * support * support < 4.0 * edge * edge
        || edge * edge * geo.nr * sizeof(double2) > l2_bytes)
      region_sh = 31;
  }
  auto count = [&](int size) { return (unsigned long long)((unsigned(size) - 1u) >> region_sh) + 1; };
  if (slices * geo.nc * count(geo.nx) * count(geo.ny) >= key_limit) region_sh = 31;
  const unsigned long long regions = count(geo.nx) * count(geo.ny);
  const bool by_cube = slices * regions * geo.nc < key_limit;
  const unsigned long long kmax = by_cube ? slices * regions * geo.nc : slices;
  // Keys beyond the sort's 2^28 lose their lowest bits: more than the records
  // of a call in practice, next to no two records have one slice.
  const bool sorted = kmax > 0 && kmax < key_limit;
  const size_t batch = patch_batch(n);
  const unsigned nb = unsigned((n + batch - 1) / batch);
  DegridKeys dk{};
  dk.slices = unsigned(slices);
  dk.stride = unsigned(stride);
  dk.region_sh = region_sh;
  dk.regions_x = unsigned(count(geo.nx));
  dk.regions = unsigned(by_cube ? regions : 0ull);
  const SortKeys sk = sorted ? sort_plan(kmax, batch) : SortKeys{};
  DegridRec* drs = static_cast<DegridRec*>(cb.degrid_recs);
  unsigned* keys = sorted ? cb.degrid_order : nullptr;
  unsigned* sorted_idx = cb.degrid_order + cb.order_capacity;
  uint2* pairs = reinterpret_cast<uint2*>(cb.degrid_order + 2 * cb.order_capacity);
  unsigned* hist = cb.sort_bins;  // counts, offsets, then the table
  unsigned* offsets = hist + patch_local_keys + 1;
  unsigned* table = offsets + patch_local_keys + 1;
  if (sorted)
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(size_t(sk.bins))), dim3(block), 0, s, hist,
                       size_t(sk.bins));
#define HPGX_DKEYS(NP)                                                         \
  hipLaunchKernelGGL(                                                          \
    k_degrid_keys<NP>, dim3(nb), dim3(patch_local_threads), 0, s, n, geo,      \
    cf.groups, static_cast<const VisRec<NP>*>(records), dk, sk,                \
    unsigned(batch), keys, drs, hist, table)
  switch (npol) {
  case 1: HPGX_DKEYS(1); break;
  case 2: HPGX_DKEYS(2); break;
  case 3: HPGX_DKEYS(3); break;
  case 4: HPGX_DKEYS(4); break;
  default: return hipErrorInvalidValue;
  }
#undef HPGX_DKEYS
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (sorted) {
    e = launch_sort_place(s, n, batch, sk, cb, keys, sk.low_bits ? nullptr : sorted_idx, pairs);
    if (e != hipSuccess) return e;
    if (sk.low_bits)
      hipLaunchKernelGGL(k_degrid_sort, dim3(unsigned(sk.bins)), dim3(sort_threads),
                         (size_t(1) << sk.low_bits) * sizeof(unsigned), s, sk.low_bits, offsets,
                         pairs, sorted_idx);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    order = sorted_idx;
  }
  const bool longer = (long long)cf.max_sx * cf.max_sy > (long long)degrid_whole * (wave / P);
#define HPGX_DEGRID_P(NP, PP, KD)                                              \
  do {                                                                         \
    constexpr size_t per = size_t(block / wave) * degrid_recs;                 \
    e = in_launches((n + per - 1) / per, block, [&](unsigned long long first, unsigned blocks) { \
      hipLaunchKernelGGL(                                                      \
        longer || KD != patch_one ? (k_degrid<NP, PP, KD, true>)               \
                                  : (k_degrid<NP, PP, KD, KD != patch_one>),   \
        dim3(blocks), dim3(block), 0, s, n, geo,                               \
        cf.taps, mu, int(same_rows), model, int(region_sh < 31), drs,          \
        static_cast<const VisRec<NP>*>(records), order, offsets + sk.bins,     \
        reinterpret_cast<double*>(cb.degrid_acc), unsigned(first));            \
    });                                                                        \
  } while (0)
#define HPGX_DEGRID_K(NP, KD)                                                  \
  do {                                                                         \
    if (P == 1) HPGX_DEGRID_P(NP, 1, KD);                                      \
    else if (P == 2) HPGX_DEGRID_P(NP, 2, KD);                                 \
    else HPGX_DEGRID_P(NP, 4, KD);                                             \
  } while (0)
  switch (npol) {
  case 1:
    if (kind == patch_one) HPGX_DEGRID_K(1, patch_one);
    else HPGX_DEGRID_K(1, patch_any);
    break;
  case 2:
    if (kind == patch_one) HPGX_DEGRID_K(2, patch_one);
    else if (kind == patch_full) HPGX_DEGRID_K(2, patch_full);
    else HPGX_DEGRID_K(2, patch_any);
    break;
  case 3:
    if (kind == patch_one) HPGX_DEGRID_K(3, patch_one);
    else HPGX_DEGRID_K(3, patch_any);
    break;
  case 4:
    if (kind == patch_one) HPGX_DEGRID_K(4, patch_one);
    else if (kind == patch_full) HPGX_DEGRID_K(4, patch_full);
    else HPGX_DEGRID_K(4, patch_any);
    break;
  default: return hipErrorInvalidValue;
  }
#undef HPGX_DEGRID_K
#undef HPGX_DEGRID_P
  if (e != hipSuccess) return e;
  return launch_degrid_finish(s, npol, n, geo, cf, mu, cb.degrid_acc, do_grid, records,
                              out_records, cb, pred64);
}

bool finish_pre_fits(const Geometry& geo) {
  return geo.ny <= 65535 && size_t(geo.nr) * geo.nc <= 65535;
}

hipError_t launch_normalize(
  hipStream_t s, int mode, void* grid, const double* weights, double wfactor,
  const Geometry& geo) {
  const size_t ps = size_t(geo.nx) * geo.ny;
  const size_t count = ps * geo.nr * geo.nc;
  if (count == 0) return hipSuccess;
  // the same FP64 division, times 1
  if (finish_pre_fits(geo))
    return launch_finish_pre(s, mode, grid, weights, wfactor, 1.0, false, geo);
  if (mode == 0)
    hipLaunchKernelGGL(
      k_normalize<double2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<double2*>(grid), weights, wfactor, ps, count);
  else
    hipLaunchKernelGGL(
      k_normalize<float2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<float2*>(grid), weights, wfactor, ps, count);
  return hipGetLastError();
}

hipError_t launch_finish_pre(
  hipStream_t s, int mode, void* grid, const double* weights, double wfactor, double scale,
  bool modulate, const Geometry& geo) {
  const size_t planes = size_t(geo.nr) * geo.nc;
  if (size_t(geo.nx) * geo.ny * planes == 0) return hipSuccess;
  // grid rows and planes index the launch's y and z
  if (!finish_pre_fits(geo)) return hipErrorInvalidValue;
  const dim3 grid_dim(unsigned((geo.nx + block - 1) / block), unsigned(geo.ny), unsigned(planes));
  if (mode == 0)
    hipLaunchKernelGGL(
      k_finish_pre<double2>, grid_dim, dim3(block), 0, s,
      static_cast<double2*>(grid), weights, wfactor, scale, int(modulate), geo.nx, geo.ny);
  else
    hipLaunchKernelGGL(
      k_finish_pre<float2>, grid_dim, dim3(block), 0, s,
      static_cast<float2*>(grid), weights, wfactor, scale, int(modulate), geo.nx, geo.ny);
  return hipGetLastError();
}

hipError_t launch_scale(
  hipStream_t s, int mode, void* grid, double inv_norm, size_t count) {
  if (count == 0) return hipSuccess;
  if (mode == 0)
    hipLaunchKernelGGL(
      k_scale<double2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<double2*>(grid), inv_norm, count);
  else
    hipLaunchKernelGGL(
      k_scale<float2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<float2*>(grid), inv_norm, count);
  return hipGetLastError();
}

hipError_t launch_shift(
  hipStream_t s, int mode, void* grid, void* scratch, int direction,
  const Geometry& geo) {
  const size_t ps = size_t(geo.nx) * geo.ny;
  const size_t nplanes = size_t(geo.nr) * geo.nc;
  const size_t count = ps * nplanes;
  if (count == 0) return hipSuccess;
  const size_t esize = mode == 0 ? sizeof(double2) : sizeof(float2);
  if (geo.nx % 2 == 0 && geo.ny % 2 == 0) {
    const size_t pairs = size_t(geo.nx) * (geo.ny / 2) * nplanes;
    if (mode == 0)
      hipLaunchKernelGGL(
        k_shift_even<double2>, dim3(blocks_for(pairs)), dim3(block), 0, s,
        static_cast<double2*>(grid), geo.nx, geo.ny, nplanes);
    else
      hipLaunchKernelGGL(
        k_shift_even<float2>, dim3(blocks_for(pairs)), dim3(block), 0, s,
        static_cast<float2*>(grid), geo.nx, geo.ny, nplanes);
    return hipGetLastError();
  }
  const int sx = direction == 0 ? geo.nx / 2 : geo.nx - geo.nx / 2;
  const int sy = direction == 0 ? geo.ny / 2 : geo.ny - geo.ny / 2;
  if (mode == 0)
    hipLaunchKernelGGL(
      k_shift_general<double2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<const double2*>(grid), static_cast<double2*>(scratch), geo.nx,
      geo.ny, sx, sy, count);
  else
    hipLaunchKernelGGL(
      k_shift_general<float2>, dim3(blocks_for(count)), dim3(block), 0, s,
      static_cast<const float2*>(grid), static_cast<float2*>(scratch), geo.nx,
      geo.ny, sx, sy, count);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return hipMemcpyAsync(grid, scratch, count * esize, hipMemcpyDeviceToDevice, s);
}

hipError_t launch_widen(hipStream_t s, const float2* src, double2* dst, size_t count) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(k_widen, dim3(blocks_for(count)), dim3(block), 0, s, src, dst, count);
  return hipGetLastError();
}

hipError_t launch_narrow(hipStream_t s, const double2* src, float2* dst, size_t count) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(k_narrow, dim3(blocks_for(count)), dim3(block), 0, s, src, dst, count);
  return hipGetLastError();
}

}  // namespace hpgx
