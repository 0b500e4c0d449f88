// Device kernels of the tessellate -> smooth -> render path for gfx950.
//
// FP64 form: every floating-point step is the reference's, in the same
// order, built with -ffp-contract=off so no multiply-add is fused; the
// results are bit-identical to the reference's FP64 arithmetic.
// FP32 form (R = float): the corner classification and the 1e-8 edge test
// stay in FP64 (topology is exact); interpolation, normals, projection,
// depth and shading run in FP32.
#include "c3d_internal.h"

#include <cfloat>
#include <type_traits>

namespace c3d {

// ----------------------------------------------------------------------
// block-wide exclusive scan of one value per thread (256 threads)

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) s_wave[wave] = x;
  __syncthreads();
  uint32_t off = 0;
  uint32_t tot = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) {
    const uint32_t s = s_wave[w];
    off += w < wave ? s : 0u;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

// ----------------------------------------------------------------------
// field access

// Field and grid pointers reach the kernels through device-side job tables,
// where the compiler cannot tell that they address global memory; read
// through gptr they become global loads (scalar base + vector offset)
// instead of flat ones, which also wait on the LDS counter.
#define C3D_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const C3D_GLOBAL T* gptr(const T* p) {
  return (const C3D_GLOBAL T*)p;
}

// a value that every lane holds, as a scalar
__device__ __forceinline__ uint32_t uniform(uint32_t x) { return uint32_t(__builtin_amdgcn_readfirstlane(int(x))); }
__device__ __forceinline__ uint64_t uniform(uint64_t x) {
  return uint64_t(uniform(uint32_t(x >> 32))) << 32 | uniform(uint32_t(x));
}
__device__ __forceinline__ double uniform(double x) {
  return __longlong_as_double(int64_t(uniform(uint64_t(__double_as_longlong(x)))));
}

// orders a wave's LDS accesses among its own lanes
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

struct CellLoc {
  uint32_t i, j, k;
  uint64_t p0;  // lattice index of corner 0
};

__device__ __forceinline__ CellLoc locate(const FieldDev& f, uint32_t c) {
  CellLoc L;
  const uint32_t jk = fdiv(c, f.div_ncx);
  L.i = c - jk * f.ncx;
  L.k = fdiv(jk, f.div_ncy);
  L.j = jk - L.k * f.ncy;
  L.p0 = (uint64_t(L.k) * f.ny + L.j) * f.nx + L.i;
  return L;
}

__device__ __forceinline__ uint64_t corner_offset(const FieldDev& f, uint32_t c) {
  // selects rather than 64-bit products: c is a corner number (0-7)
  const uint64_t nxy = uint64_t(f.nx) * f.ny;
  return uint64_t(c & 1u) + uint64_t(c & 2u ? f.nx : 0u) + (c & 4u ? nxy : 0ull);
}

template <typename R>
__device__ __forceinline__ V3<R> corner_pos(const FieldDev& f, const CellLoc& L, uint32_t c) {
  if (f.cx) {
    const uint64_t p = L.p0 + corner_offset(f, c);
    return {R(gptr(f.cx)[p]), R(gptr(f.cy)[p]), R(gptr(f.cz)[p])};
  }
  return {R(gptr(f.gx)[L.i + (c & 1u)]), R(gptr(f.gy)[L.j + ((c >> 1) & 1u)]), R(gptr(f.gz)[L.k + (c >> 2)])};
}

// ----------------------------------------------------------------------
// block-wide exclusive scan of a 64-bit value per thread (256 threads); used
// on four 16-bit counters packed in one word, one per threshold

__device__ __forceinline__ uint64_t block_excl_scan64(uint64_t v, uint64_t* s_wave, uint64_t& total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) s_wave[wave] = x;
  __syncthreads();
  uint64_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) {
    const uint64_t s = s_wave[w];
    off += w < wave ? s : 0ull;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

// the eight corner values of cell c (corner q = i + 2j + 4k offsets)
__device__ __forceinline__ void load_corners(const FieldDev& f, const CellLoc& L, double v[8]) {
  const C3D_GLOBAL double* p = gptr(f.f) + L.p0;
  const uint64_t sy = f.nx, sz = uint64_t(f.nx) * f.ny;
  v[0] = p[0];
  v[1] = p[1];
  v[2] = p[sy];
  v[3] = p[sy + 1];
  v[4] = p[sz];
  v[5] = p[sz + 1];
  v[6] = p[sz + sy];
  v[7] = p[sz + sy + 1];
}

// Topology tables, built once by upload_tables from the tetra and case
// tables of triangulate.c:145-152, 204-270:
//   c_ntri[code]            triangles of a cell with that 8-bit corner code
//   c_cslot[code * 12 + s]  triangle slot s of such a cell: bits 0-17 hold the
//                           (tail, head) cube corners of its vertices 0, 1, 2
//                           (3 + 3 bits each, reversal of triangulate.c:108-112
//                           already applied), bits 18-32 the three 5-bit
//                           cell-local edge ids (triangulate.c:23-32)
__constant__ uint8_t c_ntri[256];
__constant__ uint64_t c_cslot[256 * 12];
//   c_emask[code * 19 + e]  the slots (bit s) of such a cell whose triangle
//                           has a vertex on cell-local edge e
__constant__ uint16_t c_emask[256 * 19];

__device__ __forceinline__ uint32_t corner_code(double thr, const double v[8]) {
  uint32_t code = 0;
#pragma unroll
  for (int n = 0; n < 8; n++) code |= uint32_t(thr < v[n]) << n;
  return code;
}

// ----------------------------------------------------------------------
// tessellation tiles and work items

// the tile arithmetic of c3d_tiles.h on a field
__device__ __forceinline__ TileSpan tile_span(const FieldDev& f, uint32_t k, uint32_t col) {
  return tile_span(f.tg, f.ncx, f.ncy, f.nx, f.ny, k, col);
}

__device__ __forceinline__ uint32_t tile_corner_off(const FieldDev& f, const TileSpan&, uint32_t p) {
  return tile_corner_off(f.tg, f.ncx, f.nx, f.div_ncx, p);
}

__device__ __forceinline__ void item_range(const FieldDev& f, uint32_t item, uint32_t& col, uint32_t& k0,
                                           uint32_t& k1) {
  item_range(f.tg, f.ncz, item, col, k0, k1);
}

// the tile holding cell c of an object's field (the stored mesh's lookup)
__device__ __forceinline__ uint32_t tile_of_cell(const ObjMeta& om, uint32_t c) {
  return tile_of_cell(om.tg, om.ncx, om.ncy, om.div_ncx, om.div_ncy, c);
}

// The 4-bit code of four corners against threshold thr: bit n = thr < v[n]
// (triangulate.c:176-179).  A cell's 8-bit corner code is the code of its
// lower plane (corners 0-3) | the code of its upper plane (corners 4-7) << 4,
// and a cell's upper code is the lower code of the cell above it.
__device__ __forceinline__ uint32_t plane_code(double thr, const double v[4]) {
  uint32_t c = 0;
#pragma unroll
  for (int n = 0; n < 4; n++) c |= uint32_t(thr < v[n]) << n;
  return c;
}

// the four corners of one plane of a cell, from its corner 0 at p
__device__ __forceinline__ void load_plane4(const C3D_GLOBAL double* p, uint32_t nx, double v[4]) {
  v[0] = p[0];
  v[1] = p[1];
  v[2] = p[nx];
  v[3] = p[nx + 1];
}

// plane codes of up to four thresholds, 4 bits apart
__device__ __forceinline__ uint32_t plane_codes(const ThrSet& ts, const double v[4]) {
  uint32_t c = 0;
#pragma unroll
  for (int q = 0; q < kMaxThr; q++)
    if (q < ts.n) c |= plane_code(ts.thr[q], v) << (4 * q);
  return c;
}

// ----------------------------------------------------------------------
// the walk over work items
//
// Workgroups are dispatched round-robin over the 8 XCDs.  The work items of
// each field pass are split into 8 contiguous segments, one per XCD, so that
// every XCD gets an equal share of every pass, however unequal the passes of
// a batch are.  Work items are numbered column-fastest within a z-range, so
// the workgroups an XCD runs at once march neighbouring columns over the
// same planes (the rows they share meet in that XCD's L2).  XCD x walks
// positions 0 .. end-1: position p lies in the pass jb with
// jobs[jb].xoff <= p < jobs[jb + 1].xoff, at item x * seg + p - xoff of it
// (seg = ceil(items of the pass / 8)); the XCD's workgroups stride through
// the positions.  The grid must be a multiple of 8.
struct XcdWalk {
  uint32_t x, begin, end, step;
};

__device__ __forceinline__ XcdWalk xcd_walk(const TessJob* __restrict__ jobs, int njobs, uint32_t nitems) {
  const TessJob& last = jobs[njobs - 1];
  XcdWalk w;
  w.x = blockIdx.x % 8u;
  w.begin = blockIdx.x / 8u;
  w.end = last.xoff + (nitems - last.item0 + 7u) / 8u;
  w.step = gridDim.x / 8u;
  return w;
}

// The pass and its work item at position p of XCD x's walk; false where the
// XCD's segment of that pass is shorter than seg (the last ones).
__device__ __forceinline__ bool xcd_item(const TessJob* __restrict__ jobs, int njobs, uint32_t nitems, uint32_t x,
                                         uint32_t p, uint32_t& jb, uint32_t& item) {
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].xoff <= p) lo = mid;
    else hi = mid - 1;
  }
  jb = uint32_t(lo);
  const uint32_t t0 = jobs[lo].item0;
  const uint32_t nt = (lo + 1 < njobs ? jobs[lo + 1].item0 : nitems) - t0;
  item = x * ((nt + 7u) / 8u) + (p - jobs[lo].xoff);
  return item < nt;
}

// ----------------------------------------------------------------------
// tessellation: count pass
//
// Per work item, each thread takes column segments of R rows of the tile
// (R = 4, 2 or 1, the largest that divides the tile's rows): a segment's
// R cells share their rows of lattice points, so a plane costs 2 (R + 1)
// point loads and threshold compares for R cells instead of 4 R.  The
// cells' lower-plane codes (4 bits per threshold) stay in registers while
// the item marches up its column, so the field is read about once.  Only
// the tile totals are written, so the cells may be taken in any order.

// the bits of one lattice point: thr_q < v at bit 4q
__device__ __forceinline__ uint32_t point_bits(const ThrSet& ts, double v) {
  uint32_t b = 0;
#pragma unroll
  for (int q = 0; q < kMaxThr; q++)
    if (q < ts.n) b |= uint32_t(ts.thr[q] < v) << (4 * q);
  return b;
}

// the plane codes (plane_codes order) of the R cells of a segment whose
// top-left point is at p: points of rows 0..R, columns 0 and 1
template <int R>
__device__ __forceinline__ void segment_codes(const ThrSet& ts, const C3D_GLOBAL double* p, uint32_t nx,
                                              uint32_t out[R]) {
  double v[R + 1][2];
#pragma unroll
  for (int jj = 0; jj <= R; jj++) {
    v[jj][0] = p[uint64_t(jj) * nx];
    v[jj][1] = p[uint64_t(jj) * nx + 1];
  }
  uint32_t b0 = point_bits(ts, v[0][0]) | point_bits(ts, v[0][1]) << 1;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const uint32_t b1 = point_bits(ts, v[r + 1][0]) | point_bits(ts, v[r + 1][1]) << 1;
    out[r] = b0 | b1 << 2;
    b0 = b1;
  }
}

template <int R>
__device__ __forceinline__ void count_item(const FieldDev& f, const ThrSet& ts, const TileSpan& t, uint32_t col,
                                           uint32_t k0, uint32_t k1, const uint8_t* s_ntri, uint64_t* s_wave,
                                           uint32_t* __restrict__ cnt) {
  constexpr int M = kTileChunks / R;  // segments per thread at most (R * M = kTileCells / kThreads cells)
  const uint32_t nseg = (t.rows / R) * t.w;
  const uint64_t nxy = uint64_t(f.nx) * f.ny;
  uint32_t off[M], low[M][R];
#pragma unroll
  for (int m = 0; m < M; m++) {
    const uint32_t sg = m * kThreads + threadIdx.x;
    off[m] = 0;
#pragma unroll
    for (int r = 0; r < R; r++) low[m][r] = 0;
    if (sg < nseg) {
      // segment sg: rows R * (sg / w) .. + R - 1, column sg % w of the tile
      const uint32_t rs = R == 1 && f.tg.segs != 1 ? 0u : fdiv(sg, f.div_ncx);
      off[m] = rs * R * f.nx + (sg - rs * t.w);
      segment_codes<R>(ts, gptr(f.f) + t.l0 + off[m], f.nx, low[m]);
    }
  }
  for (uint32_t k = k0; k < k1; k++) {
    const C3D_GLOBAL double* up = gptr(f.f) + t.l0 + uint64_t(k - k0 + 1) * nxy;
    uint64_t acc = 0;
#pragma unroll
    for (int m = 0; m < M; m++) {
      const uint32_t sg = m * kThreads + threadIdx.x;
      if (sg < nseg) {
        uint32_t hi[R];
        segment_codes<R>(ts, up + off[m], f.nx, hi);
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
          for (int q = 0; q < kMaxThr; q++) {
            const uint32_t cd = ((low[m][r] >> (4 * q)) & 15u) | ((hi[r] >> (4 * q)) & 15u) << 4;
            acc += uint64_t(q < ts.n ? s_ntri[cd] : 0u) << (16 * q);
          }
          low[m][r] = hi[r];
        }
      }
    }
    uint64_t tot;
    block_excl_scan64(acc, s_wave, tot);
    const uint32_t tile = k * f.tg.cols + col;
    if (threadIdx.x < uint32_t(ts.n)) cnt[ts.boff[threadIdx.x] + tile] = uint32_t(tot >> (16 * threadIdx.x)) & 0xffffu;
  }
}

// The plane codes of every cell of tile t on the plane whose tile corner is
// at p, by column segments of R rows as in count_item, into out[cell]
// (cell = row * w + column within the tile).
template <int R>
__device__ __forceinline__ void classify_plane_r(const FieldDev& f, const ThrSet& ts, const TileSpan& t,
                                                 const C3D_GLOBAL double* p, uint16_t* out) {
  constexpr int M = kTileChunks / R;
  const uint32_t nseg = (t.rows / R) * t.w;
#pragma unroll
  for (int m = 0; m < M; m++) {
    const uint32_t sg = m * kThreads + threadIdx.x;
    if (sg < nseg) {
      const uint32_t rs = R == 1 && f.tg.segs != 1 ? 0u : fdiv(sg, f.div_ncx);
      const uint32_t c = sg - rs * t.w;
      uint32_t codes[R];
      segment_codes<R>(ts, p + rs * R * f.nx + c, f.nx, codes);
#pragma unroll
      for (int r = 0; r < R; r++) out[(rs * R + r) * t.w + c] = uint16_t(codes[r]);
    }
  }
}

__device__ __forceinline__ void classify_plane(const FieldDev& f, const ThrSet& ts, const TileSpan& t,
                                               const C3D_GLOBAL double* p, uint16_t* out) {
  if (t.rows % 4u == 0) classify_plane_r<4>(f, ts, t, p, out);
  else if (t.rows % 2u == 0) classify_plane_r<2>(f, ts, t, p, out);
  else classify_plane_r<1>(f, ts, t, p, out);
}

// seven waves per SIMD (72 VGPRs, no spill): 0.265 ms against 0.282 at six at
// 512^3 x 3 thresholds; eight spill and take 0.41 ms
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(7))) void k_count(
    const TessJob* __restrict__ jobs, int njobs, uint32_t nitems, uint32_t* __restrict__ cnt) {
  __shared__ uint64_t s_wave[kThreads / 64];
  __shared__ uint8_t s_ntri[256];
  s_ntri[threadIdx.x] = c_ntri[threadIdx.x];
  __syncthreads();
  const XcdWalk W = xcd_walk(jobs, njobs, nitems);
  for (uint32_t pp = W.begin; pp < W.end; pp += W.step) {
    uint32_t jb, item;
    if (!xcd_item(jobs, njobs, nitems, W.x, pp, jb, item)) continue;
    const FieldDev f = jobs[jb].f;
    const ThrSet ts = jobs[jb].ts;
    uint32_t col, k0, k1;
    item_range(f, item, col, k0, k1);
    const TileSpan t = tile_span(f, k0, col);
    if (t.rows % 4u == 0) count_item<4>(f, ts, t, col, k0, k1, s_ntri, s_wave, cnt);
    else if (t.rows % 2u == 0) count_item<2>(f, ts, t, col, k0, k1, s_ntri, s_wave, cnt);
    else count_item<1>(f, ts, t, col, k0, k1, s_ntri, s_wave, cnt);
  }
}

// ----------------------------------------------------------------------
// scan of tile counts into triangle starts (u64, exclusive, start[n] = total)


__global__ __launch_bounds__(kThreads) void k_scan_reduce(const uint32_t* __restrict__ cnt, uint64_t n,
                                                          uint64_t* __restrict__ tile_sum) {
  __shared__ uint64_t s[kThreads];
  const uint64_t base = uint64_t(blockIdx.x) * kScanTile;
  uint64_t acc = 0;
  for (int q = 0; q < kScanTile / kThreads; q++) {
    const uint64_t i = base + q * kThreads + threadIdx.x;
    if (i < n) acc += cnt[i];
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = s[0];
}

// single workgroup: exclusive scan of the tile sums in place
__global__ __launch_bounds__(kThreads) void k_scan_tiles(uint64_t* __restrict__ tile_sum, uint64_t ntile) {
  __shared__ uint64_t s[kThreads];
  uint64_t carry = 0;
  for (uint64_t b = 0; b < ntile; b += kThreads) {
    const uint64_t i = b + threadIdx.x;
    const uint64_t v = i < ntile ? tile_sum[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t d = 1; d < kThreads; d <<= 1) {
      const uint64_t y = threadIdx.x >= d ? s[threadIdx.x - d] : 0;
      __syncthreads();
      s[threadIdx.x] += y;
      __syncthreads();
    }
    if (i < ntile) tile_sum[i] = carry + s[threadIdx.x] - v;
    const uint64_t tot = s[kThreads - 1];
    __syncthreads();
    carry += tot;
  }
  if (threadIdx.x == 0) tile_sum[ntile] = carry;
}

__global__ __launch_bounds__(kThreads) void k_scan_apply(const uint32_t* __restrict__ cnt, uint64_t n,
                                                         const uint64_t* __restrict__ tile_off,
                                                         uint64_t* __restrict__ start) {
  __shared__ uint32_t s_wave[kThreads / 64];
  const uint64_t base = uint64_t(blockIdx.x) * kScanTile;
  uint64_t carry = tile_off[blockIdx.x];
  for (int q = 0; q < kScanTile / kThreads; q++) {
    const uint64_t i = base + q * kThreads + threadIdx.x;
    const uint32_t v = i < n ? cnt[i] : 0u;
    uint32_t tot;
    const uint32_t ex = block_excl_scan(v, s_wave, tot);
    if (i < n) start[i] = carry + ex;
    carry += tot;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) start[n] = tile_off[gridDim.x];
}

// Object bases and counts, the frame total and each image's triangle range,
// read off the tile starts on the device (so that no host round trip sits
// between counting and emitting when a frame is replayed from a graph).
template <typename R>
__global__ void k_plan(const uint64_t* __restrict__ start, uint64_t ntiles, ObjMeta* __restrict__ meta, int nobj,
                       RasterJob<R>* __restrict__ rjobs, int njobs, FrameHdr* __restrict__ hdr, uint64_t cap) {
  // objects are never empty (at least one cell), so nobj > 0 implies ntiles > 0
  for (int o = threadIdx.x; o < nobj; o += blockDim.x) {
    const uint64_t b = start[meta[o].tile_off];
    const uint64_t e = o + 1 < nobj ? start[meta[o + 1].tile_off] : start[ntiles];
    meta[o].base = b;
    meta[o].count = e - b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint64_t ntri = ntiles ? start[ntiles] : 0;
    uint64_t wk = 0;
    for (int j = 0; j < njobs; j++) {
      const uint64_t t0 = rjobs[j].obj0 < uint32_t(nobj) ? meta[rjobs[j].obj0].base : ntri;
      const uint64_t t1 = rjobs[j].obj1 < uint32_t(nobj) ? meta[rjobs[j].obj1].base : ntri;
      // each image's work starts on a workgroup boundary, so that every
      // workgroup round of the raster kernels belongs to one image
      wk = (wk + kThreads - 1) / kThreads * kThreads;
      rjobs[j].tri0 = t0;
      rjobs[j].tri1 = t1;
      rjobs[j].wk0 = wk;
      wk += t1 - t0;
    }
    hdr->ntri = ntri;
    hdr->nwork = wk;
    hdr->nfrag = 0;
    // triangles take ids 1..ntri and line fragments the ids after them, all
    // in 32 bits; a frame beyond that is flagged like one beyond `cap` (the
    // host then rejects it after its read back)
    hdr->overflow = (ntri > cap || !frame_ids_fit(ntri, hdr->nline)) ? 1u : 0u;
  }
}

// linear interpolation along a tetra edge (triangulate.c:40-73); the 1e-8
// test is on the FP64 corner values in both forms
template <typename R>
__device__ __forceinline__ V3<R> interp(double thr, V3<R> p0, double v0, V3<R> p1, double v1) {
  if (fabs(v1 - v0) < 1.e-8) return p0;
  R fct;
  if constexpr (sizeof(R) == 8) {
    fct = (thr - v0) / (v1 - v0);
  } else {
    fct = R(thr - v0) / R(v1 - v0);
  }
  return vadd(p0, vscale(fct, vsub(p1, p0)));
}

// The smoothing weight of a triangle: area * unit face normal
// (triangulate.c:75-93), formed as normal.c:39-40 forms it.  The FP32 form
// takes the cross product itself (the same vector): a triangle whose
// vertices rounded onto one point then weighs 0 instead of NaN
// (0 * (n / 0)), which would poison its neighbours' normals.
template <typename R>
__device__ __forceinline__ V3<R> smoothing_weight(const V3<R> P[3]) {
  const V3<R> n = vcross(vsub(P[1], P[0]), vsub(P[2], P[0]));
  if constexpr (sizeof(R) == 8) {
    const R area = sqrt(vdot(n, n));
    const V3<R> fn = vscale(R(1) / area, n);
    return vscale(area, fn);
  } else {
    return n;
  }
}

__device__ __forceinline__ bool interior_cell(const FieldDev& f, const CellLoc& L) {
  return L.i >= 1 && L.i + 2 <= f.ncx && L.j >= 1 && L.j + 2 <= f.ncy && L.k >= 1 && L.k + 2 <= f.ncz;
}

// ----------------------------------------------------------------------
// vertex-normal smoothing

__constant__ NbrTable c_nbr;

// the edge word of stored triangle u (in the gather record in FP64, in the
// position record in FP32)
template <typename R>
__device__ __forceinline__ uint32_t edges_of(const MeshView<R>& m, uint64_t u) {
  if constexpr (sizeof(R) == 8) return m.aux[u].edges;
  else return m.pos[u].edges;
}

template <typename R>
__device__ __forceinline__ uint64_t lower_bound_cell(const MeshAux<R>* __restrict__ aux, uint64_t lo, uint64_t hi,
                                                     uint32_t key) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (aux[mid].cell < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Unit vertex normal of a vertex on cell-local lattice edge e of cell c
// (normal.c:46-165): the sum of area * unit face normal over every triangle
// of the cells sharing the edge that has a vertex on it -- cells in
// increasing order, triangles in slot order, starting from +0 -- then
// normalised.  A cell's triangles are found from its tile's triangle range
// (triangles are stored in cell order) by binary search on the cell index.
template <typename R>
__device__ V3<R> vertex_normal(const MeshView<R>& m, const ObjMeta& om, uint32_t c, uint32_t e) {
  const int64_t sy = om.ncx, sz = int64_t(om.ncx) * om.ncy;
  V3<R> sum = {R(0), R(0), R(0)};
  const int nn = c_nbr.n[e];
  for (int q = 0; q < nn; q++) {
    const int dk = c_nbr.v[e][q][0], dj = c_nbr.v[e][q][1], di = c_nbr.v[e][q][2];
    const uint32_t want = uint32_t(c_nbr.v[e][q][3]);
    const uint32_t c2 = uint32_t(int64_t(c) + dk * sz + dj * sy + di);
    const uint32_t tl = tile_of_cell(om, c2);
    const uint64_t hi = om.bstart[tl + 1];
    for (uint64_t u = lower_bound_cell(m.aux, om.bstart[tl], hi, c2); u < hi && m.aux[u].cell == c2; u++) {
      const uint32_t eu = edges_of(m, u);
      if ((eu & 31u) == want || ((eu >> 5) & 31u) == want || ((eu >> 10) & 31u) == want)
        sum = vadd(sum, V3<R>{m.aux[u].w[0], m.aux[u].w[1], m.aux[u].w[2]});
    }
  }
  return vunit(sum);
}

// Cell starts of one object of a stored mesh, a workgroup per tile: for
// every cell c of the tile, the number of the object's triangles in the
// tile's cells before c (a tile holds at most 12 * kTileCells triangles, so
// 16 bits), from the corner codes the emit pass stored.  The triangles of
// cell c are then bstart[tile] + cstart[c] + slot, slot < c_ntri[code[c]],
// in slot order.
__global__ __launch_bounds__(kThreads) void k_cell_starts(const uint8_t* __restrict__ code,
                                                          const ObjMeta* __restrict__ meta,
                                                          uint16_t* __restrict__ cstart) {
  __shared__ uint64_t s_wave[kThreads / 64];
  __shared__ uint8_t s_ntri[256];
  s_ntri[threadIdx.x] = c_ntri[threadIdx.x];
  __syncthreads();
  const ObjMeta om = *meta;
  const uint32_t tile = blockIdx.x;
  const uint32_t k = fdiv(tile, om.tg.div_cols);
  const TileSpan t = tile_span(om.tg, om.ncx, om.ncy, om.ncx + 1u, om.ncy + 1u, k, tile - k * om.tg.cols);
  const uint8_t* cd = code + om.code_off;
  uint16_t* cs = cstart + om.code_off;
  uint32_t run = 0;
  for (uint32_t ch = 0; ch < t.n; ch += kThreads) {
    const uint32_t p = ch + threadIdx.x;
    const uint32_t n = p < t.n ? s_ntri[cd[t.c0 + p]] : 0u;
    uint64_t tot;
    const uint32_t ex = uint32_t(block_excl_scan64(n, s_wave, tot));
    if (p < t.n) cs[t.c0 + p] = uint16_t(run + ex);
    run += uint32_t(tot);
  }
}

// Compares object meshes built in two arithmetic forms, triangle by
// triangle (the topology is the same by construction, which this checks):
// out[0] topology mismatches (cell or edge ids), out[1] max |vertex
// difference| (as the bits of a non-negative double), out[2] max vertex
// normal angle in degrees (bits), out[3] sum of angles in 1e-9 degree
// units, out[4] interior vertices compared, out[5] / out[6] vertices whose
// angle exceeds 1 / 10 degrees.  Non-finite normals (zero-area
// neighbourhoods) are skipped.
template <typename RA, typename RB>
__global__ __launch_bounds__(kThreads) void k_mesh_compare(MeshView<RA> a, const ObjMeta* __restrict__ ma,
                                                           MeshView<RB> b, const ObjMeta* __restrict__ mb,
                                                           uint64_t count, unsigned long long* __restrict__ out) {
  const ObjMeta oa = *ma, ob = *mb;
  double verr = 0.0, amax = 0.0;
  unsigned long long asum = 0, nv = 0, bad = 0, over1 = 0, over10 = 0;
  for (uint64_t t = uint64_t(blockIdx.x) * kThreads + threadIdx.x; t < count; t += uint64_t(gridDim.x) * kThreads) {
    const uint64_t ga = oa.base + t, gb = ob.base + t;
    const uint32_t ea = edges_of(a, ga), eb = edges_of(b, gb);
    if (ea != eb || a.aux[ga].cell != b.aux[gb].cell) {
      bad++;
      continue;
    }
#pragma unroll
    for (int c = 0; c < 9; c++) verr = fmax(verr, fabs(double(a.pos[ga].p[c]) - double(b.pos[gb].p[c])));
    if (!((ea >> 15) & 1u)) continue;
    for (int v = 0; v < 3; v++) {
      const uint32_t e = (ea >> (5 * v)) & 31u;
      const V3<RA> na = vertex_normal<RA>(a, oa, a.aux[ga].cell, e);
      const V3<RB> nb = vertex_normal<RB>(b, ob, b.aux[gb].cell, e);
      const double d = double(na.x) * double(nb.x) + double(na.y) * double(nb.y) + double(na.z) * double(nb.z);
      if (!(d == d) || !isfinite(d)) continue;
      const double ang = acos(fmin(1.0, fmax(-1.0, d))) * (180.0 / 3.14159265358979323846);
      amax = fmax(amax, ang);
      asum += (unsigned long long)(ang * 1e9 + 0.5);
      nv++;
      over1 += ang > 1.0 ? 1u : 0u;
      over10 += ang > 10.0 ? 1u : 0u;
    }
  }
  if (bad) atomicAdd(out + 0, bad);
  atomicMax(out + 1, (unsigned long long)__double_as_longlong(verr));
  atomicMax(out + 2, (unsigned long long)__double_as_longlong(amax));
  if (asum) atomicAdd(out + 3, asum);
  if (nv) atomicAdd(out + 4, nv);
  if (over1) atomicAdd(out + 5, over1);
  if (over10) atomicAdd(out + 6, over10);
}

// ----------------------------------------------------------------------
// rasterisation

// order-preserving integer images of the depths (larger depth = nearer)
__device__ __forceinline__ uint64_t ord64(double x) {
  if (x == 0.0) x = 0.0;
  const uint64_t u = __double_as_longlong(x);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double unord64(uint64_t k) {
  const uint64_t u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
  return __longlong_as_double(u);
}
__device__ __forceinline__ uint32_t ord32(float x) {
  if (x == 0.0f) x = 0.0f;
  const uint32_t u = __float_as_uint(x);
  return (u >> 31) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float unord32(uint32_t k) {
  const uint32_t u = (k >> 31) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}

// the image owning raster work item u (the last job starting at or before
// it: images with no triangles share their successor's start)
template <typename R>
__device__ __forceinline__ int find_rjob(const RasterJob<R>* __restrict__ jobs, int n, uint64_t u) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].wk0 <= u) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// ----------------------------------------------------------------------
// raster
//
// One triangle per thread; a workgroup round takes 256 consecutive work
// items of one image, so the image's constants are uniform.  Workgroups
// stride over the rounds and load the next round's triangles while drawing
// the current ones.  In FP64 the coverage loop runs over the narrowed box
// of tight_box.
// Modes:
//   kRasterFp32     FP32: packed (depth << 32 | id) keys, one pass
//   kRasterDepth64  FP64 depth pass that keeps the fragments that may end
//                   up nearest: a key below the value read from the z-buffer
//                   can never win (keys only grow); every other one goes
//                   through atomicMax and into a workgroup list in LDS, which
//                   is flushed with one global reservation per round.  The
//                   list holds every fragment whose key equals the final
//                   value.  Overflow (LDS or global) sets bit 2 of
//                   hdr->overflow.
//   kRasterId64     FP64 id pass over the geometry: the latest serial id at
//                   each pixel's final depth; runs only when the fragment
//                   list overflowed
constexpr int kFragLds = 1024;

// Projection (project.c), the reference's box and area (render.c:60-89)
// and the narrowed box of one triangle; returns its candidate pixels (0
// when a vertex fails to project or, in FP32, the projection has no area:
// such a triangle's weights are all +-0 and its depth 1 / +-0).
template <typename R>
__device__ __forceinline__ uint32_t setup_triangle(const ViewDev<R>& v, const V3<R> wpos[3], Projected<R>& P) {
  bool vis = true;
#pragma unroll
  for (int n = 0; n < 3; n++) vis = vis && project(v, wpos[n], P.q[n]);
  if (!vis) return 0;
  if (sizeof(R) == 4 && edge_fn(P.q[0], P.q[1], P.q[2].x, P.q[2].y) == R(0)) return 0;
  // about 12 reference-box candidates of a pixel-sized triangle narrow to 3
  // (by way of the reference's box: 512^3 FP32 frame 2.89 ms instead of 2.81)
  pixel_box(v, P);
  if (P.i1 < P.i0 || P.j1 < P.j0) return 0;
  // a box lies inside one image: fewer than 2^31 pixels
  return uint32_t(P.i1 - P.i0 + 1) * uint32_t(P.j1 - P.j0 + 1);
}

__device__ __forceinline__ void atomic_max_id(uint32_t* p, uint32_t v) { atomicMax(p, v); }
__device__ __forceinline__ void atomic_max_id(uint64_t* p, uint64_t v) {
  atomicMax(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
}

// One candidate pixel (i, j) of stored triangle P (id tid1): the reference's
// barycentric test and harmonic depth (render.c:91-124), then the z-buffer
// update of `MODE`.  Depth64 puts fragments in the workgroup list s_frag
// (s_n entries).
template <typename R, int MODE>
__device__ __forceinline__ void pixel_update(const ViewDev<R>& v, uint64_t row0, const Projected<R>& P, int32_t i,
                                             int32_t j, uint32_t tid1, uint64_t* __restrict__ key,
                                             uint32_t* __restrict__ id, Frag* s_frag, uint32_t* s_n) {
  R w0, w1, w2;
  if (!pixel_weights(P, column_centre(v, i), row_centre(v, j), w0, w1, w2)) return;
  const R dep = pixel_depth(P, w0, w1, w2);
  const uint64_t px = row0 + uint64_t(j) * uint64_t(v.W) + uint64_t(i);
  if constexpr (MODE == kRasterFp32) {
    // keys only grow: a key at or below a value read from the buffer can
    // never change it and skips the atomic
    const uint64_t k = uint64_t(ord32(float(dep))) << 32 | uint64_t(tid1);
    if (k > key[px]) atomicMax(reinterpret_cast<unsigned long long*>(key + px), (unsigned long long)k);
  } else if constexpr (MODE == kRasterDepth64) {
    const uint64_t k = ord64(double(dep));
    if (k < key[px]) return;
    atomicMax(reinterpret_cast<unsigned long long*>(key + px), (unsigned long long)k);
    // every fragment whose key equals the final value is kept: its key was
    // at least the value read before its own atomic
    const uint32_t o = atomicAdd(s_n, 1u);
    if (o < uint32_t(kFragLds)) {
      Frag fr;
      fr.px = uint32_t(px);
      fr.id = tid1;
      fr.key = k;
      s_frag[o] = fr;
    }
  } else {
    if (ord64(double(dep)) == key[px]) atomic_max_id(id + px, tid1);
  }
}

// one triangle drawn by its own lane: every candidate of its box in turn
template <typename R, int MODE>
__device__ __forceinline__ void draw_triangle(const ViewDev<R>& v, uint64_t row0, const V3<R> wpos[3], uint32_t tid1,
                                              uint64_t* __restrict__ key, uint32_t* __restrict__ id, Frag* s_frag,
                                              uint32_t* s_n) {
  Projected<R> P;
  if (!setup_triangle<R>(v, wpos, P)) return;
  for (int32_t j = P.j0; j <= P.j1; j++)
    for (int32_t i = P.i0; i <= P.i1; i++)
      pixel_update<R, MODE>(v, row0, P, i, j, tid1, key, id, s_frag, s_n);
}

// registers of one raster work item, loaded a round ahead
template <typename R>
struct TriRegs {
  R p[9];
  uint32_t ed;
  uint64_t t;
  int jb;
  bool ok;
};

template <typename R>
__device__ __forceinline__ void fetch_tri(const MeshView<R>& m, const RasterJob<R>* __restrict__ rjobs, int njobs,
                                          uint64_t u0, TriRegs<R>& T) {
  T.jb = njobs > 1 ? find_rjob(rjobs, njobs, u0) : 0;
  T.t = rjobs[T.jb].tri0 + (u0 + threadIdx.x - rjobs[T.jb].wk0);
  T.ok = T.t < rjobs[T.jb].tri1;
  T.ed = 0;
  if (T.ok) {
    T.ed = edges_of(m, T.t);
#pragma unroll
    for (int n = 0; n < 9; n++) T.p[n] = m.pos[T.t].p[n];
  }
}

template <typename R, int MODE>
__global__ __launch_bounds__(kThreads) void k_raster(MeshView<R> m, const RasterJob<R>* __restrict__ rjobs, int njobs,
                                                     FrameHdr* __restrict__ hdr, uint64_t* __restrict__ key,
                                                     uint32_t* __restrict__ id, Frag* __restrict__ frags,
                                                     uint32_t cap) {
  __shared__ Frag s_frag[MODE == kRasterDepth64 ? kFragLds : 1];
  __shared__ uint32_t s_n, s_base;
  // a frame whose triangles outgrew the mesh (bit 1, set by the plan of a
  // replayed frame) has triangles that were never stored: draw nothing
  if (hdr->overflow & 1u) return;
  if (MODE == kRasterId64 && !(hdr->overflow & 2u)) return;
  const uint64_t nwork = hdr->nwork;
  const uint64_t stride = uint64_t(gridDim.x) * kThreads;
  uint64_t u0 = uint64_t(blockIdx.x) * kThreads;
  TriRegs<R> cur;
  cur.ok = false;
  if (u0 < nwork) fetch_tri(m, rjobs, njobs, u0, cur);
  for (; u0 < nwork; u0 += stride) {
    // the next round's triangle is loaded while this one is drawn
    TriRegs<R> nxt;
    nxt.ok = false;
    if (u0 + stride < nwork) fetch_tri(m, rjobs, njobs, u0 + stride, nxt);
    if (MODE == kRasterDepth64) {
      if (threadIdx.x == 0) s_n = 0;
      __syncthreads();
    }
    if (cur.ok && ((cur.ed >> 15) & 1u)) {
      const V3<R> wp[3] = {{cur.p[0], cur.p[1], cur.p[2]}, {cur.p[3], cur.p[4], cur.p[5]},
                           {cur.p[6], cur.p[7], cur.p[8]}};
      const ViewDev<R> v = rjobs[cur.jb].v;
      draw_triangle<R, MODE>(v, rjobs[cur.jb].px0, wp, uint32_t(cur.t + 1), key, id, s_frag, &s_n);
    }
    if constexpr (MODE == kRasterDepth64) {
      __syncthreads();
      const uint32_t n = s_n < uint32_t(kFragLds) ? s_n : uint32_t(kFragLds);
      if (threadIdx.x == 0) {
        s_base = n ? atomicAdd(&hdr->nfrag, n) : 0u;
        if (s_n > uint32_t(kFragLds) || (n && uint64_t(s_base) + n > cap)) atomicOr(&hdr->overflow, 2u);
      }
      __syncthreads();
      const uint32_t b0 = s_base;
      for (uint32_t e = threadIdx.x; e < n; e += kThreads) {
        if (uint64_t(b0) + e < cap) frags[b0 + e] = s_frag[e];
      }
      __syncthreads();
    }
    cur = nxt;
  }
}

// ----------------------------------------------------------------------
// frames without a stored mesh: tessellation fused with the raster
//
// Every wave works by itself, with no barrier between the waves of a
// workgroup.  It takes bricks of a field (c3d_bricks.h: up to 8 x 8 x 8
// cells, a lane per cell column), nearest groups first, from one counter per
// XCD; classifies the brick's lattice points plane by plane; lists the cells
// that a threshold cuts (about a fifth of a turbulent field's); and queues
// the triangles of the listed cells of the rendered interior, 64 cells at a
// time, as 8-byte items (cell; vertex corners, threshold, slot) in an LDS
// ring that is drained 64 at a time: every lane then computes, projects and
// draws one triangle into each image that shows its object (jimg: offsets
// per field pass into a list of the images showing any of its objects).  The
// ring carries items over rounds and bricks (within one field pass).
// Nothing is stored per triangle: ids name the object, cell and slot
// (tri_id64), and the resolve recomputes what it needs from the field.
//
// A brick that lies behind what the z-buffer holds is counted but not drawn,
// except for cells whose triangles' projections may be too small for the
// depth bound to hold (c3d_cull.h; FP64 only: with FP32's rounding the rule,
// which judges a cell by its brick's extent, holds of next to none at 512^3).
// With the bricks taken front to back, most of a dense field is behind its
// first surfaces: at 512^3, three thresholds and 1920 x 1080, 42 M of 129 M
// triangles are drawn.
//
// What bounds it: vector-ALU issue (1000 instructions per 64 triangles in
// FP32 before the pixel box was formed directly, divisions by view constants
// became products and corners were selected by masks: 512^3 FP32 frame 3.15
// -> 2.81 ms, 1024^3 19.1 -> 16.9 ms), and the latency of each brick's chain
// of reads.  Letting every lane walk to its next covered pixel before any of
// them forms a depth was no faster on small triangles and slower on large
// ones (close-up 1.65 -> 2.51 ms).  The 512^3 FP64 frame's kernel took 4.50
// ms as a tessellation of whole rows with a queue and barriers per workgroup,
// no z-test and no order; 3.61 ms in bricks taken front to back by
// workgroups; 2.2 ms by waves, with the cut cells listed before anything is
// done with them; and 1.86 ms since (FP32, where every triangle is drawn:
// 3.41 -> 2.56 ms, besides 0.28 ms of counting passes that serial ids had
// needed).  Close-ups, where few triangles cover many pixels each, gained
// most: 301 x 187 x 223 with five thresholds 8.15 -> 1.19 ms.
//
// Every covered pixel is tested against the z-buffer as it is drawn (key:
// the depth's order key, larger is nearer); a fragment at or above the value
// read goes through atomicMax into the z-buffer and, with its id, into the
// frame's fragment list.  The list holds every fragment whose key equals the pixel's final key, and
// k_frag_ids then gives each pixel the largest id among them: "largest
// depth, then last in drawing order", the result of the reference's
// sequential >= test (render.c:125-132).  If the frame's list overflows, a
// second pass over the geometry (kFrameIds) finds the ids instead.
constexpr uint32_t kFragChunk0 = 64, kFragChunk = 1024;  // entries of the frame's fragment list that a wave
                                                         // reserves at a time: at first, and at most
static_assert(kFragChunk0 >= 64, "a reservation holds a fragment of every lane");
constexpr uint32_t kNoPixel = 0xffffffffu;               // a reserved entry that stayed empty
constexpr uint32_t kWaveRing = 128;    // queued triangles of a wave (a power of two, at least 2 * 64)
constexpr uint32_t kRing = 512;        // of a workgroup of the emit (at least 2 * kThreads)

// a queued triangle names its threshold in 2 bits (ring item bits 18-19),
// and the drains index ThrSet::thr and ::obj with it
static_assert(kMaxThr == 4, "the ring's threshold field is 2 bits wide");

// bit b of x as a mask, and a where the mask is set, else b
__device__ __forceinline__ uint32_t bit_mask(uint32_t x, int b) { return uint32_t(int32_t(x << (31 - b)) >> 31); }
__device__ __forceinline__ uint32_t pick(uint32_t m, uint32_t a, uint32_t b) { return (m & a) | (~m & b); }
__device__ __forceinline__ float pick(uint32_t m, float a, float b) {
  return __uint_as_float(pick(m, __float_as_uint(a), __float_as_uint(b)));
}
__device__ __forceinline__ uint64_t pick(uint32_t m, uint64_t a, uint64_t b) {
  return uint64_t(pick(m, uint32_t(a >> 32), uint32_t(b >> 32))) << 32 | pick(m, uint32_t(a), uint32_t(b));
}
__device__ __forceinline__ double pick(uint32_t m, double a, double b) {
  return __hiloint2double(int(pick(m, uint32_t(__double2hiint(a)), uint32_t(__double2hiint(b)))),
                          int(pick(m, uint32_t(__double2loint(a)), uint32_t(__double2loint(b)))));
}

// positions of the triangle whose vertices join the corners in `ent` (slot
// entry bits 0-17) of cell L, reading the two corner values of each
// vertex's lattice edge from the field; on a grid lattice the cell's six
// coordinates are read once.  Every load depends only on L and ent, so they
// are in flight together.  The corners' bits select by masks (v_bfi), which
// is half the instructions of compares and selects: a frame at 512^3 in FP32
// took 2.92 ms with those instead of 2.81.
template <typename R>
__device__ __forceinline__ void slot_positions_mem(const FieldDev& f, const CellLoc& L, double thr, uint32_t ent,
                                                   V3<R> P[3]) {
  const C3D_GLOBAL double* p = gptr(f.f) + L.p0;
  if (f.cx) {
#pragma unroll
    for (int vv = 0; vv < 3; vv++) {
      const uint32_t tail = (ent >> (6 * vv)) & 7u;
      const uint32_t head = (ent >> (6 * vv + 3)) & 7u;
      P[vv] = interp<R>(thr, corner_pos<R>(f, L, tail), p[corner_offset(f, tail)], corner_pos<R>(f, L, head),
                        p[corner_offset(f, head)]);
    }
    return;
  }
  const R x0 = R(gptr(f.gx)[L.i]), x1 = R(gptr(f.gx)[L.i + 1]), y0 = R(gptr(f.gy)[L.j]),
          y1 = R(gptr(f.gy)[L.j + 1]), z0 = R(gptr(f.gz)[L.k]), z1 = R(gptr(f.gz)[L.k + 1]);
  const uint64_t below = uint64_t(p), above = uint64_t(p + uint64_t(f.nx) * f.ny);  // the cell's two planes
  const auto load_at = [](uint64_t plane, uint32_t off) { return reinterpret_cast<const C3D_GLOBAL double*>(plane)[off]; };
#pragma unroll
  for (int vv = 0; vv < 3; vv++) {
    uint32_t m[6];  // the corners' bits as masks: tail x, y, z, head x, y, z
#pragma unroll
    for (int b = 0; b < 6; b++) m[b] = bit_mask(ent, 6 * vv + b);
    const V3<R> pt = {pick(m[0], x1, x0), pick(m[1], y1, y0), pick(m[2], z1, z0)};
    const V3<R> ph = {pick(m[3], x1, x0), pick(m[4], y1, y0), pick(m[5], z1, z0)};
    // a plane may hold 2^32 points and more, a row holds at most 2^30
    const uint64_t at = pick(m[2], above, below), ah = pick(m[5], above, below);
    P[vv] = interp<R>(thr, pt, load_at(at, (m[0] & 1u) + (m[1] & f.nx)), ph, load_at(ah, (m[3] & 1u) + (m[4] & f.nx)));
  }
}

// Images of a field pass for which triangles are told apart by whether they
// can reach them; a pass shown in more draws every triangle into the others.
constexpr uint32_t kMaskImages = 8;
constexpr uint32_t kAllImages = (1u << kMaskImages) - 1u;

struct FrameLds {
  uint16_t pc[kBrickPlanes + 1][64];    // plane codes of each lane's cell column
  uint16_t list[kBrickPlanes * 64];     // the brick's cut cells: plane << 6 | column
  uint32_t rc[kWaveRing];  // cell of the queued triangle
  uint32_t re[kWaveRing];  // its vertices' (tail, head) corners (slot entry bits 0-17) | threshold << 18 | slot << 20 |
                           // the images it may reach, of the pass's first kMaskImages, << 24
  // a round of 64 listed cells: their indices, codes, exclusive triangle
  // counts and irregular thresholds (bit q)
  uint32_t cell[64];
  uint16_t pref[kMaxThr][64];
  uint8_t code[kMaxThr][64];
  uint8_t irr[64];
  uint32_t fnext, fend, fchunk;  // the wave's entries of the fragment list: free ones, and the next reservation's size
};

// a lane's value, as a scalar
__device__ __forceinline__ uint32_t lane_u32(uint32_t x, int l) { return uint32_t(__builtin_amdgcn_readlane(int(x), l)); }
__device__ __forceinline__ float lane_of(float x, int l) { return __uint_as_float(lane_u32(__float_as_uint(x), l)); }
__device__ __forceinline__ uint64_t lane_of(uint64_t x, int l) {
  return uint64_t(lane_u32(uint32_t(x >> 32), l)) << 32 | lane_u32(uint32_t(x), l);
}
__device__ __forceinline__ double lane_of(double x, int l) {
  return __longlong_as_double(int64_t(lane_of(uint64_t(__double_as_longlong(x)), l)));
}

// depth keys: larger is nearer; 32-bit depths in the upper half
__device__ __forceinline__ uint64_t depth_key(double d) { return ord64(d); }
__device__ __forceinline__ uint64_t depth_key(float d) { return uint64_t(ord32(d)) << 32; }

// Appends fr to the frame's fragment list (called by any subset of the
// wave's lanes).  A wave fills entries that it reserved, and reserves twice
// as many as the last time when they run out, so the list's counter, which
// all waves share, is touched rarely whether a wave finds three fragments or
// a million.
__device__ __forceinline__ void append_frag(const Frag64& fr, FrameLds& S, Frag64* __restrict__ gfrags, uint32_t gcap,
                                            FrameHdr* __restrict__ hdr) {
  const uint64_t act = __ballot(1);
  const uint32_t lane = __lane_id(), n = uint32_t(__popcll(act));
  const int leader = __builtin_ctzll(act);
  const uint32_t rank = uint32_t(__popcll(act & ((1ull << lane) - 1ull)));
  const uint32_t at = S.fnext, room = S.fend - at;
  wave_lds_fence();
  uint32_t more = 0;
  if (n > room) {
    // the rest go to a new reservation
    const uint32_t size = S.fchunk;
    if (lane == uint32_t(leader)) {
      more = atomicAdd(&hdr->nfrag, size);
      if (uint64_t(more) + size > gcap) atomicOr(&hdr->overflow, 2u);
      S.fnext = more + (n - room);
      S.fend = more + size;
      S.fchunk = 2u * size < kFragChunk ? 2u * size : kFragChunk;
    }
    more = lane_u32(more, leader);
  } else if (lane == uint32_t(leader)) {
    S.fnext = at + n;
  }
  wave_lds_fence();
  const uint32_t g = rank < room ? at + rank : more + (rank - room);
  if (g < gcap) gfrags[g] = fr;
}

// what a drawing lane needs beside its triangle
struct DrawTo {
  uint64_t* __restrict__ key;
  uint64_t* __restrict__ id;
  Frag64* __restrict__ frags;
  uint32_t fcap;
  FrameHdr* __restrict__ hdr;
};

// One candidate pixel (i, j) of triangle P (id tid): the reference's
// barycentric test and harmonic depth (render.c:91-124), then the z-test.
template <typename R, int MODE>
__device__ __forceinline__ void frame_pixel(const ViewDev<R>& v, uint64_t row0, const Projected<R>& P, int32_t i,
                                            int32_t j, uint64_t tid, FrameLds& S, const DrawTo& D) {
  R w0, w1, w2;
  if (!pixel_weights(P, column_centre(v, i), row_centre(v, j), w0, w1, w2)) return;
  const uint64_t k = depth_key(pixel_depth(P, w0, w1, w2));
  const uint64_t px = row0 + uint64_t(j) * uint64_t(v.W) + uint64_t(i);
  // keys only grow, so a value read here, however stale, that is above k
  // means the fragment cannot be the pixel's
  const uint64_t was = D.key[px];
  if constexpr (MODE == kFrameDraw) {
    if (k < was) return;
    if (k > was) atomicMax(reinterpret_cast<unsigned long long*>(D.key + px), (unsigned long long)k);
    Frag64 fr;
    fr.key = k;
    fr.id = tid;
    fr.px = uint32_t(px);
    fr.pad = 0;
    append_frag(fr, S, D.frags, D.fcap, D.hdr);
  } else {
    if (k == was) atomic_max_id(D.id + px, tid);
  }
}

// Draws the wave's triangles (one per lane with `here`).  Each lane walks
// the box of its own triangle; a large box is walked by the whole wave, 8 x 8
// pixels at a time: one of more than kHuge pixels, or of more than kLarge and
// half the wave's average, so that one large triangle among small ones does
// not hold the other 63 lanes, and triangles that are all huge do not leave
// most lanes waiting for the longest walk.  With kLarge and four times the
// average, the rule before, frames (FP64 unless said otherwise) took
//   100^3, 1920 x 1080, deep inside     12.6 ms, now 2.3
//   64^3 blobs, FP32, close             2.2 ms, now 0.8
//   300^3, close                        3.85 ms, now 2.4
//   128^3, close                        1.80 ms, now 1.1
// and frames of small triangles the same.  Of kLarge 16, 301 x 187 x 223
// takes 1.41 ms instead of 1.37 and an uneven batch 4.21 instead of 4.10; of
// 128, 24^3 185 us instead of 157.
template <typename R, int MODE>
__device__ __forceinline__ void draw_wave(const ViewDev<R>& v, uint64_t row0, bool here, const V3<R> wpos[3],
                                          uint64_t tid, FrameLds& S, const DrawTo& D) {
  constexpr uint32_t kLarge = 64, kHuge = 256;
  Projected<R> P;
  uint32_t n = 0;
  if (here) n = setup_triangle<R>(v, wpos, P);
  bool together = n > kLarge;
  if (__ballot(together)) {
    float sum = float(n);
#pragma unroll
    for (int d = 32; d; d >>= 1) sum += __shfl_xor(sum, d, 64);
    together = n > kHuge || (together && float(n) > sum * (0.5f / 64.0f));
  }
  if (n && !together)
    for (int32_t j = P.j0; j <= P.j1; j++)
      for (int32_t i = P.i0; i <= P.i1; i++) frame_pixel<R, MODE>(v, row0, P, i, j, tid, S, D);
  for (uint64_t todo = __ballot(together); todo; todo &= todo - 1u) {
    const int l = __builtin_ctzll(todo);
    Projected<R> Q;
#pragma unroll
    for (int a = 0; a < 3; a++) Q.q[a] = {lane_of(P.q[a].x, l), lane_of(P.q[a].y, l), lane_of(P.q[a].z, l)};
    Q.ainv = lane_of(P.ainv, l);
    Q.i0 = int32_t(lane_u32(uint32_t(P.i0), l));
    Q.i1 = int32_t(lane_u32(uint32_t(P.i1), l));
    Q.j0 = int32_t(lane_u32(uint32_t(P.j0), l));
    Q.j1 = int32_t(lane_u32(uint32_t(P.j1), l));
    const uint64_t t = lane_of(tid, l);
    const int32_t li = int32_t(__lane_id() & 7u), lj = int32_t(__lane_id() >> 3);
    for (int32_t jb = Q.j0; jb <= Q.j1; jb += 8)
      for (int32_t ib = Q.i0; ib <= Q.i1; ib += 8)
        if (ib + li <= Q.i1 && jb + lj <= Q.j1) frame_pixel<R, MODE>(v, row0, Q, ib + li, jb + lj, t, S, D);
  }
}

// Marks the entries that the wave reserved and did not fill.
__device__ __forceinline__ void close_frags(FrameLds& S, Frag64* __restrict__ frags, uint32_t fcap) {
  wave_lds_fence();
  for (uint32_t g = S.fnext + __lane_id(); g < S.fend; g += 64u)
    if (g < fcap) frags[g].px = kNoPixel;
}

// Draws the n (<= 64) oldest queued triangles of field pass jb, one per
// lane.
template <typename R, int MODE>
__device__ __forceinline__ void drain_ring(FrameLds& S, uint32_t head, uint32_t n, const TessJob* __restrict__ jobs,
                                           uint32_t jb, const RasterJob<R>* __restrict__ rjobs,
                                           const uint32_t* __restrict__ jimg, const DrawTo& D) {
  V3<R> P[3];
  uint32_t obj = 0, images = 0;
  uint64_t tid = 0;
  const uint32_t lane = __lane_id();
  const bool drawn = lane < n;
  if (drawn) {
    const FieldDev f = jobs[jb].f;
    const uint32_t s = (head + lane) & (kWaveRing - 1u);
    const uint32_t cc = S.rc[s], x = S.re[s];
    const CellLoc L = locate(f, cc);
    const uint32_t q = (x >> 18) & 3u;
    // one load per lane indexed by the threshold number: fewer vector
    // instructions and spilled registers than selecting among kMaxThr
    const double thr = jobs[jb].ts.thr[q];
    obj = jobs[jb].ts.obj[q];
    slot_positions_mem<R>(f, L, thr, x & 0x3ffffu, P);
    tid = tri_id64(obj, cc, (x >> 20) & 15u);
    images = x >> 24;
  }
  // the images of this field pass (the same for every lane)
  for (uint32_t u = uniform(jimg[jb]), end = uniform(jimg[jb + 1]); u < end; u++) {
    const uint32_t k = uniform(jimg[u]);
    const bool here = drawn && obj >= rjobs[k].obj0 && obj < rjobs[k].obj1 && (images & 1u);
    images = images >> 1 | 1u << (kMaskImages - 1u);  // the images past the mask: always
    if (!__ballot(here)) continue;
    const ViewDev<R> v = rjobs[k].v;
    draw_wave<R, MODE>(v, rjobs[k].px0, here, P, tid, S, D);
  }
}

constexpr uint32_t kMaxBoxPixels = 1u << 14;  // pixels read for one brick's visibility at most

// Whether every z-buffer key of the pixel box of an image (first pixel row0,
// W pixels a row) is above `bound`: 256 pixels at a time until one is not.
// The reads go to the device's coherent level, so that they see what other
// XCDs have drawn (an older value would only be smaller).
__device__ __forceinline__ bool box_above(const uint64_t* __restrict__ key, uint64_t row0, uint32_t W,
                                          const BrickLimits& o, uint64_t bound) {
  if (o.i1 < o.i0 || o.j1 < o.j0) return true;  // no fragment falls on the image
  const uint32_t w = uint32_t(o.i1 - o.i0) + 1u, n = w * (uint32_t(o.j1 - o.j0) + 1u);
  if (n > kMaxBoxPixels) return false;
  const float rw = 1.0f / float(w);
  for (uint32_t t0 = 0; t0 < n; t0 += 256u) {
    bool below = false;
#pragma unroll
    for (uint32_t a = 0; a < 4u; a++) {
      uint32_t t = t0 + a * 64u + __lane_id();
      t = t < n ? t : n - 1u;
      // t / w for t < 2^14: the quotient's error is far below 1 / w
      const uint32_t r = uint32_t((float(t) + 0.5f) * rw);
      const uint64_t px = row0 + uint64_t(uint32_t(o.j0) + r) * W + uint32_t(o.i0) + (t - r * w);
      below = below || __hip_atomic_load(key + px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= bound;
    }
    if (__ballot(below)) return false;
  }
  return true;
}

// The images (of the pass's first kMaskImages, bit u for image jimg[u0 + u])
// that regular cells of brick B may still reach; scale gets the others'
// area scale (lane u holds image u's).  The corners' views are formed by
// lanes 0-7 (and every other eight lanes alike).
__device__ __forceinline__ uint32_t reachable_images(const FieldDev& f, BrickBox B,
                                                     const RasterJob<double>* __restrict__ rjobs,
                                                     const uint32_t* __restrict__ jimg, uint32_t u0, uint32_t u1,
                                                     const uint64_t* __restrict__ key, double& scale) {
  uint32_t seen = kAllImages;
  const uint32_t c = __lane_id() & 7u;
  const double px = gptr(f.gx)[B.i0 + (c & 1u) * (B.i1 - B.i0)], py = gptr(f.gy)[B.j0 + (c >> 1 & 1u) * (B.j1 - B.j0)],
               pz = gptr(f.gz)[B.k0 + (c >> 2) * (B.k1 - B.k0)];
  for (uint32_t u = u0; u < u1 && u - u0 < kMaskImages; u++) {
    const RasterJob<double>& J = rjobs[uniform(jimg[u])];
    CornerView cv;
    const bool ok = corner_view(J.v, px, py, pz, cv);
    if (__ballot(ok) != ~0ull) continue;
    BrickRange r = {cv.x, cv.x, cv.y, cv.y, cv.nr, cv.nr, cv.size};
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) {
      r.x0 = fmin(r.x0, __shfl_xor(r.x0, d, 64));
      r.x1 = fmax(r.x1, __shfl_xor(r.x1, d, 64));
      r.y0 = fmin(r.y0, __shfl_xor(r.y0, d, 64));
      r.y1 = fmax(r.y1, __shfl_xor(r.y1, d, 64));
      r.n0 = fmin(r.n0, __shfl_xor(r.n0, d, 64));
      r.n1 = fmax(r.n1, __shfl_xor(r.n1, d, 64));
      r.size = fmax(r.size, __shfl_xor(r.size, d, 64));
    }
    BrickLimits o;
    if (!uniform(uint32_t(brick_limits(J.v, r, o)))) continue;
    o.i0 = int32_t(uniform(uint32_t(o.i0)));
    o.i1 = int32_t(uniform(uint32_t(o.i1)));
    o.j0 = int32_t(uniform(uint32_t(o.j0)));
    o.j1 = int32_t(uniform(uint32_t(o.j1)));
    if (!box_above(key, J.px0, uint32_t(J.v.W), o, uniform(depth_key(o.bound)))) continue;
    seen &= ~(1u << (u - u0));
    scale = __lane_id() == u - u0 ? o.scale : scale;
  }
  return seen;
}

// The thresholds (bit q) at which cell (i, j, k) is cut (`cuts`) and not
// regular in one of the images its brick is hidden in: there it is drawn all
// the same.
__device__ __forceinline__ uint32_t irregular_at(const TessJob& J, uint32_t i, uint32_t j, uint32_t k, uint32_t cuts,
                                                 const RasterJob<double>* __restrict__ rjobs,
                                                 const uint32_t* __restrict__ jimg, uint32_t u0, uint32_t seen,
                                                 double scale, bool inner) {
  const FieldDev& f = J.f;
  double v[8], x0 = 0, y0 = 0, z0 = 0, hx = 1, hy = 1, hz = 1;
  if (inner) {
    const uint64_t nxy = uint64_t(f.nx) * f.ny;
    const C3D_GLOBAL double* p = gptr(f.f) + k * nxy + uint64_t(j) * f.nx + i;
    load_plane4(p, f.nx, v);
    load_plane4(p + nxy, f.nx, v + 4);
    x0 = gptr(f.gx)[i];
    y0 = gptr(f.gy)[j];
    z0 = gptr(f.gz)[k];
    hx = gptr(f.gx)[i + 1u] - x0;
    hy = gptr(f.gy)[j + 1u] - y0;
    hz = gptr(f.gz)[k + 1u] - z0;
  }
  const float fx = float(hx), fy = float(hy), fz = float(hz);
  uint32_t bad = 0;
  for (uint32_t hid = ~seen & kAllImages; hid; hid &= hid - 1u) {
    const uint32_t u = uint32_t(__builtin_ctz(hid));
    const ViewDev<double>& vw = rjobs[uniform(jimg[u0 + u])].v;
    const float volume = cell_volume(hx, hy, hz, lane_of(scale, int(u)));
    if (inner) {
      CellValues cv;
      cell_values(v, float(vw.cam[0] - x0) / fx, float(vw.cam[1] - y0) / fy, float(vw.cam[2] - z0) / fz, cv);
#pragma unroll
      for (int q = 0; q < kMaxThr; q++)
        if (((cuts >> q) & 1u) && !cell_regular(cv, float(v[0] - J.ts.thr[q]), volume)) bad |= 1u << q;
    }
  }
  return bad;
}

// Bricks are taken one by one from XCD list x, and from another list once
// that one is empty; each is asked for while the one before is worked on.
// The lists' counters are `take`, 64 words apart.  ask_brick gives lane 0 a
// position of list x; next_brick gives the wave the position asked for
// (`ahead`), or one of the first other list that still has some, in p, and
// asks for the next; false when every list is empty.
__device__ __forceinline__ uint32_t ask_brick(uint32_t* __restrict__ take, uint32_t x) {
  uint32_t p = 0;
  if (__lane_id() == 0) p = atomicAdd(take + 64u * x, 1u);
  return p;
}

__device__ __forceinline__ bool next_brick(uint32_t* __restrict__ take, uint32_t ngroups, uint32_t shift, uint32_t& x,
                                           uint32_t& ahead, uint32_t& from, uint32_t& p) {
  p = uniform(ahead);
  for (uint32_t tried = 0; p >= brick_positions(ngroups, shift, x); tried++) {
    if (tried == 16u) return false;  // a list never fills again
    const uint32_t lane = __lane_id();
    bool some = false;
    if (lane < 8u)
      some = __hip_atomic_load(take + 64u * lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
             brick_positions(ngroups, shift, lane);
    const uint32_t left = uint32_t(__ballot(some));
    if (!left) return false;
    // the first after x
    const uint32_t turned = (left >> x | left << (8u - x)) & 255u;
    x = uniform((x + uint32_t(__builtin_ctz(turned))) & 7u);
    p = uniform(ask_brick(take, x));
  }
  from = x;
  ahead = ask_brick(take, x);
  return true;
}

// Occupancy: four waves per SIMD in FP64 (128 VGPRs, no spill; five spill 120
// bytes a lane and take 2.71 ms instead of 2.34 for the 512^3 frame), six in
// FP32.
template <typename R, int MODE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 8 ? 4 : 6))) void k_frame(
    const TessJob* __restrict__ jobs, const uint2* __restrict__ order, uint32_t ngroups, uint32_t shift,
    uint32_t* __restrict__ take, const RasterJob<R>* __restrict__ rjobs, const uint32_t* __restrict__ jimg,
    FrameHdr* __restrict__ hdr, uint64_t* __restrict__ key, uint64_t* __restrict__ id, Frag64* __restrict__ frags,
    uint32_t fcap) {
  __shared__ FrameLds lds[kThreads / 64];
  __shared__ uint8_t s_ntri[256];
  // the id pass runs only after the fragment list overflowed
  if (MODE == kFrameIds && !(hdr->overflow & 2u)) return;
  const uint32_t lane = __lane_id(), wave = uniform(threadIdx.x >> 6);
  FrameLds& S = lds[wave];
  s_ntri[threadIdx.x] = c_ntri[threadIdx.x];
  if (lane == 0) {
    S.fnext = 0;
    S.fend = 0;
    S.fchunk = kFragChunk0;
  }
  __syncthreads();  // the only barrier
  const DrawTo D = {key, id, frags, fcap, hdr};
  uint32_t list = uniform(blockIdx.x & 7u), ahead = ask_brick(take, list);
  uint32_t ntri = 0;  // triangles of the cells this lane counted
  // ring state: oldest item, items queued, and the field pass they belong to
  // (the queue holds one pass at a time)
  uint32_t head = 0, npend = 0, cur = 0;
  for (bool more = true; more;) {
    uint32_t tx = 0, tp = 0;
    more = next_brick(take, ngroups, shift, list, ahead, tx, tp);
    uint32_t jb = cur, ncut = 0;  // the brick's field pass, and its cut cells
    BrickBox B = {};
    if (more) {
      const uint2 og = order[tx + 8u * (tp >> (3u * shift))];
      const uint32_t ogx = uniform(og.x), within = tp & ((1u << (3u * shift)) - 1u);
      jb = ogx & 0x1fffffffu;
      const FieldDev& f = jobs[jb].f;
      if (brick_box(jobs[jb].bg, f.ncx, f.ncy, f.ncz, uniform(og.y), within, ogx >> 29, B)) {
        const uint32_t row = fdiv(lane, jobs[jb].bg.div_bw), col = lane - row * jobs[jb].bg.bw;
        const uint32_t ci = B.i0 + col, cj = B.j0 + row;
        const bool valid = ci < B.i1 && cj < B.j1;
        // plane codes of the lane's cell column, every load independent
        const uint64_t nxy = uint64_t(f.nx) * f.ny;
        const C3D_GLOBAL double* p = gptr(f.f) + B.k0 * nxy + uint64_t(cj) * f.nx + ci;
        const uint32_t points = B.k1 - B.k0 + 1u;
        if (valid) {
          for (uint32_t z = 0; z < points; z += 3u) {
            // three planes in flight; past the last one it is read again
            double v[3][4];
            uint32_t zz[3];
#pragma unroll
            for (uint32_t u = 0; u < 3u; u++) {
              zz[u] = z + u < points ? z + u : points - 1u;
              load_plane4(p + zz[u] * nxy, f.nx, v[u]);
            }
#pragma unroll
            for (uint32_t u = 0; u < 3u; u++) S.pc[zz[u]][lane] = uint16_t(plane_codes(jobs[jb].ts, v[u]));
          }
        }
        // the cells that a threshold cuts: some corner of either kind
        uint32_t lo = valid ? S.pc[0][lane] : 0u;
        for (uint32_t z = 0; z + 1u < points; z++) {
          const uint32_t hi = valid ? S.pc[z + 1u][lane] : 0u;
          const uint32_t some = lo | hi, all = lo & hi;
          const uint32_t any = (some | some >> 1 | some >> 2 | some >> 3) & 0x1111u;
          const bool is_cut = (any & ~(all & all >> 1 & all >> 2 & all >> 3)) != 0u;
          const uint64_t m = __ballot(is_cut);
          if (is_cut) S.list[ncut + uint32_t(__popcll(m & ((1ull << lane) - 1ull)))] = uint16_t(z << 6 | lane);
          ncut += uint32_t(__popcll(m));
          lo = hi;
        }
        wave_lds_fence();
      }
    }
    uint32_t seen = kAllImages;  // the images that the brick's regular cells may reach
    bool unseen = false;         // none at all
    double scale = 0.0;
    if constexpr (sizeof(R) == 8) {
      if (ncut && jobs[jb].f.ordered) {
        const uint32_t u0 = uniform(jimg[jb]), u1 = uniform(jimg[jb + 1u]);
        seen = reachable_images(jobs[jb].f, B, rjobs, jimg, u0, u1, key, scale);
        unseen = u1 - u0 <= kMaskImages && (seen & ((1u << (u1 - u0)) - 1u)) == 0;
      }
    }
    // The pass's constants are read again around every drain, through an
    // index made opaque: the compiler then loads them (scalar loads from the
    // constant cache) instead of holding them in scalar registers across the
    // drain, where the image constants need those registers.
    const auto job = [&]() -> const TessJob& {
      uint32_t again = jb;
      asm volatile("" : "+v"(again));
      return jobs[uniform(again)];
    };
    // round 0 draws what is left of an earlier pass; then 64 listed cells a
    // round, drawing every full 64 triangles (one drain in the code: it is
    // large)
    const bool rest = npend && (!more || jb != cur);
    const uint32_t rounds = (ncut + 63u) >> 6;
    for (uint32_t round = rest ? 0u : 1u; round <= rounds; round++) {
      uint32_t qoff[kMaxThr + 1] = {};
      if (round) {
        cur = jb;
        const TessJob& J = job();
        const uint32_t at = (round - 1u) * 64u + lane;
        const bool has = at < ncut;
        const uint32_t it = S.list[has ? at : 0u], z = it >> 6, c = it & 63u;
        const uint32_t lo = S.pc[z][c], hi = S.pc[z + 1u][c];
        const uint32_t row = fdiv(c, J.bg.div_bw);
        const uint32_t i = B.i0 + c - row * J.bg.bw, j = B.j0 + row, k = B.k0 + z;
        const bool inner = has && i >= 1u && i + 2u <= J.f.ncx && j >= 1u && j + 2u <= J.f.ncy && k >= 1u &&
                           k + 2u <= J.f.ncz;
        uint64_t packed = 0;
        uint32_t cuts = 0;
#pragma unroll
        for (int q = 0; q < kMaxThr; q++) {
          // codes of thresholds past the last are 0
          const uint32_t cd = ((lo >> (4 * q)) & 15u) | ((hi >> (4 * q)) & 15u) << 4;
          const uint32_t nt = has ? s_ntri[cd] : 0u;
          S.code[q][lane] = uint8_t(cd);
          ntri += nt;
          cuts |= nt ? 1u << q : 0u;
          packed |= uint64_t(nt) << (16 * q);
        }
        uint32_t irr = 0;
        if constexpr (sizeof(R) == 8) {
          if (seen != kAllImages) {
            irr = irregular_at(J, i, j, k, cuts, rjobs, jimg, uniform(jimg[cur]), seen, scale, inner);
            // a brick hidden in every image draws only its irregular cells
            if (unseen)
#pragma unroll
              for (int q = 0; q < kMaxThr; q++)
                if (!((irr >> q) & 1u)) packed &= ~(uint64_t(0xffffu) << (16 * q));
          }
        }
        // cells outside the rendered interior are counted, not drawn
        if (!inner) packed = 0;
        if (!__ballot(packed != 0)) continue;
        uint64_t end = packed;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint64_t y = __shfl_up((unsigned long long)end, d, 64);
          if (lane >= uint32_t(d)) end += y;
        }
        const uint64_t tot = lane_of(end, 63), ex = end - packed;
#pragma unroll
        for (int q = 0; q < kMaxThr; q++) {
          qoff[q + 1] = qoff[q] + (uint32_t(tot >> (16 * q)) & 0xffffu);
          S.pref[q][lane] = uint16_t(ex >> (16 * q));
        }
        S.cell[lane] = (k * J.f.ncy + j) * J.f.ncx + i;
        S.irr[lane] = uint8_t(irr);
        wave_lds_fence();
      }
      const uint32_t total = qoff[kMaxThr];
      uint32_t pos = 0;
      do {
        // queue as many of the round's triangles as the ring holds
        const uint32_t room = kWaveRing - npend;
        const uint32_t put = total - pos < room ? total - pos : room;
        for (uint32_t e = lane; e < put; e += 64u) {
          const uint32_t item = pos + e;
          int q = 0;
#pragma unroll
          for (int z = 1; z < kMaxThr; z++) q += item >= qoff[z] ? 1 : 0;
          uint32_t qsel = 0;
#pragma unroll
          for (int z = 1; z < kMaxThr; z++) qsel = q == z ? qoff[z] : qsel;
          const uint32_t r = item - qsel;
          uint32_t l = 0;
#pragma unroll
          for (uint32_t step = 32; step; step >>= 1) l += S.pref[q][l + step] <= r ? step : 0u;
          const uint32_t sl = r - S.pref[q][l];
          const uint32_t s = (head + npend + e) & (kWaveRing - 1u);
          const uint32_t images = seen != kAllImages && !((S.irr[l] >> q) & 1u) ? seen : kAllImages;
          S.rc[s] = S.cell[l];
          S.re[s] = (uint32_t(c_cslot[S.code[q][l] * 12u + sl]) & 0x3ffffu) | uint32_t(q) << 18 | sl << 20 |
                    images << 24;
        }
        pos += put;
        npend += put;
        wave_lds_fence();
        while (npend >= 64u || (round == 0 && npend)) {
          const uint32_t n = npend < 64u ? npend : 64u;
          drain_ring<R, MODE>(S, head, n, jobs, uniform(cur), rjobs, jimg, D);
          head = (head + n) & (kWaveRing - 1u);
          npend -= n;
        }
      } while (pos < total);
    }
  }
  if constexpr (MODE == kFrameDraw) {
    close_frags(S, frags, fcap);
    // the frame's triangle count, which no count pass gives it
#pragma unroll
    for (int d = 32; d; d >>= 1) ntri += __shfl_xor(ntri, d, 64);
    if (lane == 0 && ntri)
      atomicAdd(reinterpret_cast<unsigned long long*>(&hdr->ntri), (unsigned long long)ntri);
  }
}

// Before a frame: clears its z-buffer, ids, header and brick counters, and
// (workgroup b for field pass b) lists the pass's groups of bricks, nearest
// first: a counting sort over 256 depth bins of the groups' centres, the
// depth being the reference's z key direction (nrm . (p - cam), larger is
// nearer) scaled to the lattice's range, the nearest of the images' where a
// pass is shown in several.  The order decides only how soon the z-buffer
// fills, never a result.
constexpr uint32_t kBins = 256;

template <typename R>
__device__ void order_groups(const TessJob& J, uint32_t jb, const RasterJob<R>* __restrict__ rjobs,
                             const uint32_t* __restrict__ jimg, uint2* __restrict__ order, uint32_t* s_bin,
                             uint32_t* s_wave, float (*s_range)[2]) {
  const FieldDev& f = J.f;
  const BrickGeo& g = J.bg;
  const uint32_t ng = brick_groups(g);
  const auto point = [&](uint32_t i, uint32_t j, uint32_t k) -> V3<R> {
    if (f.cx) {
      const uint64_t p = (uint64_t(k) * f.ny + j) * f.nx + i;
      return {R(gptr(f.cx)[p]), R(gptr(f.cy)[p]), R(gptr(f.cz)[p])};
    }
    return {R(gptr(f.gx)[i]), R(gptr(f.gy)[j]), R(gptr(f.gz)[k])};
  };
  const auto depth = [&](const ViewDev<R>& v, V3<R> p) {
    return v.nrm[0] * (p.x - v.cam[0]) + v.nrm[1] * (p.y - v.cam[1]) + v.nrm[2] * (p.z - v.cam[2]);
  };
  const uint32_t u0 = jimg[jb], u1 = jimg[jb + 1];
  // from which end each axis is taken inside a group: the nearer one in the
  // first image
  uint32_t flip = 0;
  if (u0 < u1) {
    const ViewDev<R>& v = rjobs[jimg[u0]].v;
    const R d0 = depth(v, point(0, 0, 0));
    flip = (depth(v, point(f.ncx, 0, 0)) > d0 ? 1u : 0u) | (depth(v, point(0, f.ncy, 0)) > d0 ? 2u : 0u) |
           (depth(v, point(0, 0, f.ncz)) > d0 ? 4u : 0u);
  }
  // depth range of the lattice's corners in each of the first kMaskImages
  // images (a pass shown in more is ordered for those)
  const uint32_t nu = u1 - u0 < kMaskImages ? u1 - u0 : kMaskImages;
  __syncthreads();
  if (threadIdx.x < nu) {
    const ViewDev<R>& v = rjobs[jimg[u0 + threadIdx.x]].v;
    R lo = R(0), hi = R(0);
    for (uint32_t c = 0; c < 8u; c++) {
      const R d = depth(v, point(c & 1u ? f.ncx : 0u, c & 2u ? f.ncy : 0u, c & 4u ? f.ncz : 0u));
      lo = c ? fmin(lo, d) : d;
      hi = c ? fmax(hi, d) : d;
    }
    s_range[threadIdx.x][0] = float(lo);
    s_range[threadIdx.x][1] = float(kBins) / float(hi - lo);
  }
  __syncthreads();
  const auto bin_of = [&](uint32_t s) {
    uint32_t x, y, z;
    group_at(g, s, x, y, z);
    const auto mid = [&](uint32_t a, uint32_t b, uint32_t n) {
      const uint32_t m = ((2u * a + 1u) << g.shift) * b / 2u;
      return m < n ? m : n;
    };
    const V3<R> p = point(mid(x, g.bw, f.ncx), mid(y, g.bh, f.ncy), mid(z, g.bz, f.ncz));
    float best = 0.0f;
    for (uint32_t u = 0; u < nu; u++)
      best = fmaxf(best, (float(depth(rjobs[jimg[u0 + u]].v, p)) - s_range[u][0]) * s_range[u][1]);
    // not a number, or outside the corners' range: an end bin
    const float t = float(kBins) - best;
    return t > 0.0f ? (t < float(kBins) ? uint32_t(t) : kBins - 1u) : 0u;
  };
  s_bin[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t s = threadIdx.x; s < ng; s += kThreads) atomicAdd(&s_bin[bin_of(s)], 1u);
  __syncthreads();
  uint32_t tot;
  const uint32_t ex = block_excl_scan(s_bin[threadIdx.x], s_wave, tot);
  s_bin[threadIdx.x] = ex;
  __syncthreads();
  for (uint32_t s = threadIdx.x; s < ng; s += kThreads)
    order[J.group0 + atomicAdd(&s_bin[bin_of(s)], 1u)] = make_uint2(jb | flip << 29, s);
}

template <typename R>
__global__ __launch_bounds__(kThreads) void k_frame_begin(const TessJob* __restrict__ jobs, uint32_t njobs,
                                                          const RasterJob<R>* __restrict__ rjobs,
                                                          const uint32_t* __restrict__ jimg,
                                                          uint2* __restrict__ order, uint32_t* __restrict__ take,
                                                          uint64_t* __restrict__ key, uint64_t* __restrict__ id,
                                                          uint64_t npx, FrameHdr* __restrict__ hdr) {
  static_assert(kBins == kThreads, "a bin per thread");
  __shared__ uint32_t s_bin[kBins], s_wave[kThreads / 64];
  __shared__ float s_range[kMaskImages][2];
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      hdr->ntri = 0;
      hdr->nfrag = 0;
      hdr->overflow = 0;
    }
    if (threadIdx.x < 16u) take[64u * threadIdx.x] = 0;
  }
  for (uint32_t jb = blockIdx.x; jb < njobs; jb += gridDim.x) {
    order_groups<R>(jobs[jb], jb, rjobs, jimg, order, s_bin, s_wave, s_range);
    __syncthreads();
  }
  const uint64_t k0 = sizeof(R) == 8 ? 0x0010000000000000ull /* ord64(-DBL_MAX) */ : 0ull;
  for (uint64_t p = uint64_t(blockIdx.x) * kThreads + threadIdx.x; p < npx; p += uint64_t(gridDim.x) * kThreads) {
    key[p] = k0;
    id[p] = 0;
  }
}

// ----------------------------------------------------------------------
// tessellation: emit pass (the stored mesh)
//
// The work-item loop of the queue kernels; every drain computes up to 256
// triangles, one per thread, into records in LDS (a position record and a
// gather record each), and the workgroup then stores those records at
// their serial positions as 8-byte words, thread q taking words q, q + 256,
// ... of each array: the drain's triangles are a few runs of consecutive
// positions (one per object in the drained chunks), so every store
// instruction writes contiguous bytes and whole lines, where one store per
// record field (14 streams) had written scattered 4- or 8-byte pieces.  The
// stores are non-temporal: the mesh streams past the caches, and the field
// planes the workgroups march through stay in L2.
//
// Every earlier vector memory operation is waited for once before the
// drain's stores, so that nothing is in flight when they issue: the
// compiler then issues the store sequence back to back, where otherwise it
// waited between stores for loads still counted ahead of them.

// The emit's triangle queue: an LDS ring of 12-byte items, drained 256 at a
// time so that every lane holds a triangle.
struct EmitLds {
  uint8_t code[kMaxThr][kThreads];
  uint16_t pref[kMaxThr][kThreads];
  uint16_t low[kTileChunks][kThreads];  // lower-plane codes of the tile's cells (cell p at [p / 256][p % 256])
  uint64_t wave[kThreads / 64];
  uint8_t ntri[256];
  uint32_t rg[kRing];  // serial position of the queued triangle
  uint32_t rc[kRing];  // its cell
  uint32_t re[kRing];  // its vertices' (tail, head) corners (slot entry bits 0-17) | threshold << 18 |
                       // slot << 20 | corner code << 24
};

// The emit's work-item loop: marches each work item's column up its planes,
// classifies each tile's cells in chunks of 256 (loading only the upper
// corners: the lower-plane codes carry over from the plane below, in LDS),
// queues the chunk's triangles in the LDS ring in serial order and calls
// drain(head, n, jb) for every full 256 items (and for the rest when the
// field pass changes and at the end).  With kPlanes each plane's upper codes
// are first computed for the whole tile by column segments (classify_plane,
// into s_hi: the cells of a segment share their rows of lattice points) and
// the chunks read them from LDS; the FP32 emit measured 1.5% faster so; the
// FP64 emit, which would lose a workgroup per CU to the extra LDS, loads
// each cell's corners itself.  Every cell's corner code of every threshold q
// is stored at codeout[code_off + q * ncells + cell]: by each cell's thread
// as bytes (kStoreCode 1) or from LDS as 4-byte words (kStoreCode 2;
// measured faster in the FP64 emit, slower in the FP32 one).  Expects S.ntri
// loaded and a barrier since.
template <int kStoreCode, bool kPlanes, typename Drain>
__device__ __forceinline__ void ring_tiles(EmitLds& S, uint16_t* s_hi, const TessJob* __restrict__ jobs, int njobs,
                                           uint32_t nitems, const uint64_t* __restrict__ start,
                                           uint8_t* __restrict__ codeout, Drain&& drain) {
  // ring state, the same in every thread: oldest item, items queued, and
  // the field pass they belong to
  uint32_t head = 0, npend = 0, cur = 0;
  const XcdWalk W = xcd_walk(jobs, njobs, nitems);
  for (uint32_t pp = W.begin; pp < W.end; pp += W.step) {
    uint32_t jb, item;
    if (!xcd_item(jobs, njobs, nitems, W.x, pp, jb, item)) continue;
    // the queue holds one field pass at a time
    while (npend && jb != cur) {
      const uint32_t n = npend < kThreads ? npend : kThreads;
      drain(head, n, cur);
      head = (head + n) & (kRing - 1u);
      npend -= n;
    }
    cur = jb;
    const auto Fd = [&]() -> const FieldDev& { return jobs[jb].f; };
    const auto Ts = [&]() -> const ThrSet& { return jobs[jb].ts; };
    uint32_t col, k0, k1;
    item_range(Fd(), item, col, k0, k1);
    // the tile's span and plane strides, recomputed from the pass
    const auto Tsp = [&]() { return tile_span(Fd(), k0, col); };
    const uint32_t nch = (Tsp().n + kThreads - 1) / kThreads;
    const auto nxy = [&]() { return uint64_t(Fd().nx) * Fd().ny; };
    const auto ncxy = [&]() { return Fd().ncx * Fd().ncy; };
    // codes of the first plane's corners: with kPlanes by column segments
    // (the cells of a segment share their rows of lattice points), else
    // each thread its own cells (reading back only what it wrote)
    if constexpr (kPlanes) {
      __syncthreads();  // the previous item's chunk loop is done with S.low
      classify_plane(Fd(), Ts(), Tsp(), gptr(Fd().f) + Tsp().l0, &S.low[0][0]);
    } else {
      for (uint32_t ch = 0; ch < nch; ch++) {
        const uint32_t p = ch * kThreads + threadIdx.x;
        if (p < Tsp().n) {
          double v[4];
          load_plane4(gptr(Fd().f) + Tsp().l0 + tile_corner_off(Fd(), Tsp(), p), Fd().nx, v);
          S.low[ch][threadIdx.x] = uint16_t(plane_codes(Ts(), v));
        }
      }
    }
    for (uint32_t k = k0; k < k1; k++) {
      const uint32_t tile = k * Fd().tg.cols + col;
      const uint32_t ctile = Tsp().c0 + (k - k0) * ncxy();
      const C3D_GLOBAL double* up = gptr(Fd().f) + Tsp().l0 + uint64_t(k - k0 + 1) * nxy();
      if constexpr (kPlanes) {
        __syncthreads();  // the previous plane's chunk loop is done with s_hi
        classify_plane(Fd(), Ts(), Tsp(), up, s_hi);
        __syncthreads();
      }
      uint64_t base[kMaxThr];
#pragma unroll
      for (int q = 0; q < kMaxThr; q++) base[q] = q < Ts().n ? start[Ts().boff[q] + tile] : 0;
      for (uint32_t ch = 0; ch < nch; ch++) {
        const uint32_t c0 = ctile + ch * kThreads;
        const uint32_t p = ch * kThreads + threadIdx.x;
        const bool valid = p < Tsp().n;
        uint32_t code[kMaxThr];
        uint64_t packed = 0;
#pragma unroll
        for (int q = 0; q < kMaxThr; q++) code[q] = 0;
        if (valid) {
          uint32_t hi;
          if constexpr (kPlanes) {
            hi = s_hi[p];
          } else {
            double v[4];
            load_plane4(up + tile_corner_off(Fd(), Tsp(), p), Fd().nx, v);
            hi = plane_codes(Ts(), v);
          }
          const uint32_t lo = S.low[ch][threadIdx.x];
          S.low[ch][threadIdx.x] = uint16_t(hi);
#pragma unroll
          for (int q = 0; q < kMaxThr; q++) {
            const uint32_t cd = ((lo >> (4 * q)) & 15u) | ((hi >> (4 * q)) & 15u) << 4;
            code[q] = q < Ts().n ? cd : 0u;
            packed |= uint64_t(S.ntri[code[q]]) << (16 * q);
          }
          if (kStoreCode == 1) {
            uint8_t* co = codeout + jobs[jb].code_off + (c0 + threadIdx.x);
#pragma unroll
            for (int q = 0; q < kMaxThr; q++)
              if (q < Ts().n) co[uint64_t(q) * Fd().ncells] = uint8_t(code[q]);
          }
        }
        uint64_t tot;
        const uint64_t ex = block_excl_scan64(packed, S.wave, tot);
        uint32_t qoff[kMaxThr + 1];
        qoff[0] = 0;
#pragma unroll
        for (int q = 0; q < kMaxThr; q++) {
          qoff[q + 1] = qoff[q] + (uint32_t(tot >> (16 * q)) & 0xffffu);
          S.pref[q][threadIdx.x] = uint16_t(ex >> (16 * q));
          if (valid) S.code[q][threadIdx.x] = uint8_t(code[q]);
        }
        __syncthreads();
        if (kStoreCode == 2) {
          // the chunk's codes of threshold q are bytes [d0, d0 + nv) of the
          // code array: whole 4-byte words inside that range are stored as
          // words, the bytes of the (at most two) words it shares with the
          // neighbouring chunks one by one
          const uint32_t nv = Tsp().n - ch * kThreads < kThreads ? Tsp().n - ch * kThreads : kThreads;
          const uint32_t nw = (kThreads + 3u) / 4u + 1u;  // words touched by 256 bytes at any alignment
          for (uint32_t w = threadIdx.x; w < uint32_t(Ts().n) * nw; w += kThreads) {
            const uint32_t q = w / nw, kw = w - q * nw;
            const uint64_t d0 = jobs[jb].code_off + uint64_t(q) * Fd().ncells + c0;
            const uint64_t a = (d0 & ~uint64_t(3)) + 4u * kw;
            const uint64_t lo = a > d0 ? a : d0, hi = a + 4u < d0 + nv ? a + 4u : d0 + nv;
            if (lo >= hi) continue;
            if (lo == a && hi == a + 4u) {
              const uint32_t l = uint32_t(a - d0);
              const uint32_t word = uint32_t(S.code[q][l]) | uint32_t(S.code[q][l + 1]) << 8 |
                                    uint32_t(S.code[q][l + 2]) << 16 | uint32_t(S.code[q][l + 3]) << 24;
              *reinterpret_cast<uint32_t*>(codeout + a) = word;
            } else {
              for (uint64_t b = lo; b < hi; b++) codeout[b] = S.code[q][uint32_t(b - d0)];
            }
          }
        }
        const uint32_t total = qoff[kMaxThr];
        for (uint32_t pos = 0; pos < total;) {
          // queue as many of the chunk's triangles as the ring holds, in
          // serial order (threshold, cell, slot)
          const uint32_t room = kRing - npend;
          const uint32_t take = total - pos < room ? total - pos : room;
          for (uint32_t e = threadIdx.x; e < take; e += kThreads) {
            const uint32_t it = pos + e;
            int q = 0;
#pragma unroll
            for (int z = 1; z < kMaxThr; z++) q += it >= qoff[z] ? 1 : 0;
            uint32_t qsel = 0;
#pragma unroll
            for (int z = 1; z < kMaxThr; z++) qsel = q == z ? qoff[z] : qsel;
            const uint32_t r = it - qsel;
            uint32_t l = 0;
#pragma unroll
            for (uint32_t step = kThreads / 2; step; step >>= 1) l += S.pref[q][l + step] <= r ? step : 0u;
            const uint32_t sl = r - S.pref[q][l];
            const uint32_t cc = c0 + l;
            const uint32_t cd = S.code[q][l];
            const uint32_t s = (head + npend + e) & (kRing - 1u);
            uint64_t bq = base[0];
#pragma unroll
            for (int z = 1; z < kMaxThr; z++) bq = q == z ? base[z] : bq;
            S.rg[s] = uint32_t(bq + r);
            S.rc[s] = cc;
            S.re[s] = (uint32_t(c_cslot[cd * 12u + sl]) & 0x3ffffu) | uint32_t(q) << 18 | sl << 20 | cd << 24;
          }
          pos += take;
          npend += take;
          __syncthreads();
          while (npend >= kThreads) {
            drain(head, kThreads, jb);
            head = (head + kThreads) & (kRing - 1u);
            npend -= kThreads;
          }
        }
        // the next chunk's triangles follow this chunk's in every object
#pragma unroll
        for (int q = 0; q < kMaxThr; q++) base[q] += qoff[q + 1] - qoff[q];
      }
    }
  }
  while (npend) {
    const uint32_t n = npend < kThreads ? npend : kThreads;
    drain(head, n, cur);
    head = (head + n) & (kRing - 1u);
    npend -= n;
  }
}

// stores n records of type Rec from LDS at the drain's serial positions
template <typename Rec>
__device__ __forceinline__ void store_drain(const EmitLds& S, const Rec* s_src, uint32_t head, uint32_t n,
                                            Rec* out, uint64_t cap) {
  constexpr uint32_t kWords = sizeof(Rec) / 8u;
  const uint64_t* src = reinterpret_cast<const uint64_t*>(s_src);
  char* dst = reinterpret_cast<char*>(out);
  for (uint32_t k = threadIdx.x; k < n * kWords; k += kThreads) {
    const uint32_t r = k / kWords;
    const uint32_t g = S.rg[(head + r) & (kRing - 1u)];
    if (g < cap)
      __builtin_nontemporal_store(src[k], reinterpret_cast<uint64_t*>(dst + uint64_t(g) * sizeof(Rec) +
                                                                     8u * (k - r * kWords)));
  }
}

template <typename R>
__device__ __forceinline__ void emit_ring(EmitLds& S, MeshPos<R>* s_pos, MeshAux<R>* s_aux, uint32_t head,
                                          uint32_t n, const TessJob* __restrict__ jobs, uint32_t jb,
                                          const MeshView<R>& m, FrameHdr* __restrict__ hdr) {
  if (threadIdx.x < n) {
    const FieldDev f = jobs[jb].f;
    const uint32_t s = (head + threadIdx.x) & (kRing - 1u);
    const uint32_t cc = S.rc[s], x = S.re[s];
    const CellLoc L = locate(f, cc);
    const uint32_t q = (x >> 18) & 3u;
    const double thr = jobs[jb].ts.thr[q];
    V3<R> P[3];
    slot_positions_mem<R>(f, L, thr, x & 0x3ffffu, P);
    const V3<R> w = smoothing_weight<R>(P);
    const uint32_t ent_edges = uint32_t(c_cslot[(x >> 24) * 12u + ((x >> 20) & 15u)] >> 18) & 0x7fffu;
    const uint32_t edges = ent_edges | uint32_t(interior_cell(f, L)) << 15;
    MeshPos<R>& rp = s_pos[threadIdx.x];
    MeshAux<R>& ra = s_aux[threadIdx.x];
#pragma unroll
    for (int vv = 0; vv < 3; vv++) {
      rp.p[3 * vv + 0] = P[vv].x;
      rp.p[3 * vv + 1] = P[vv].y;
      rp.p[3 * vv + 2] = P[vv].z;
    }
    ra.w[0] = w.x;
    ra.w[1] = w.y;
    ra.w[2] = w.z;
    ra.cell = cc;
    if constexpr (sizeof(R) == 8) ra.edges = edges;
    else rp.edges = edges;
    if (uint64_t(S.rg[s]) >= m.cap) hdr->overflow = 1u;  // capacity reserved ahead of a replayed frame was too small
  }
  __syncthreads();
  __builtin_amdgcn_s_waitcnt(0);
  store_drain(S, s_pos, head, n, m.pos, m.cap);
  store_drain(S, s_aux, head, n, m.aux, m.cap);
  __syncthreads();
}

template <typename R>
__global__ __launch_bounds__(kThreads) void k_emit(const TessJob* __restrict__ jobs, int njobs, uint32_t nitems,
                                                   const uint64_t* __restrict__ start, MeshView<R> m,
                                                   FrameHdr* __restrict__ hdr) {
  __shared__ EmitLds S;
  __shared__ MeshPos<R> s_pos[kThreads];
  __shared__ MeshAux<R> s_aux[kThreads];
  constexpr bool kPl = sizeof(R) == 4;  // the FP64 build would lose a workgroup per CU to the LDS
  __shared__ uint16_t s_hi[kPl ? kTileCells : 1];
  S.ntri[threadIdx.x] = c_ntri[threadIdx.x];
  __syncthreads();
  ring_tiles<sizeof(R) == 8 ? 2 : 1, kPl>(S, s_hi, jobs, njobs, nitems, start, m.code, [&](uint32_t head, uint32_t n, uint32_t jb) {
    emit_ring<R>(S, s_pos, s_aux, head, n, jobs, jb, m, hdr);
  });
}

// the latest triangle among the kept fragments at each pixel's final depth
template <typename FT, typename TId>
__global__ void k_frag_ids(const FT* __restrict__ frags, uint32_t cap, const FrameHdr* __restrict__ hdr,
                           const uint64_t* __restrict__ key, TId* __restrict__ id) {
  if (hdr->overflow & 2u) return;
  const uint32_t n = min(hdr->nfrag, cap);
  for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < n; f += gridDim.x * blockDim.x) {
    const FT fr = frags[f];
    if (sizeof(TId) == 8 && fr.px == kNoPixel) continue;
    if (fr.key == key[fr.px]) atomic_max_id(id + fr.px, fr.id);
  }
}

// Before a stored mesh is rendered: clears the z-buffer, the ids and the
// frame header's raster state.
__global__ void k_zinit(uint64_t* __restrict__ key, uint32_t* __restrict__ id, uint64_t npx, uint64_t k0,
                        FrameHdr* __restrict__ hdr) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    hdr->nfrag = 0;
    hdr->overflow &= 1u;
  }
  for (uint64_t p = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < npx; p += uint64_t(gridDim.x) * blockDim.x) {
    key[p] = k0;
    if (id) id[p] = 0;
  }
}

// Line fragments (pixels and depths computed on the host, in drawing
// order) take part in the same z-test; their ids follow every triangle's
// (64-bit: after every object, kLineObj; 32-bit: after the frame's ntri).
template <typename TId>
__global__ void k_line_frags(const uint32_t* __restrict__ pix, const double* __restrict__ depth,
                             const FrameHdr* __restrict__ hdr, int pass, int fp32, uint64_t* __restrict__ key,
                             TId* __restrict__ id) {
  const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= hdr->nline) return;
  const uint32_t px = pix[f];
  const TId lid = sizeof(TId) == 8 ? TId(kLineObj << 40 | f) : TId(hdr->ntri + 1 + f);
  if (sizeof(TId) == 4 && fp32) {
    // a stored FP32 mesh: one pass, the key carries the id
    const uint64_t k = uint64_t(ord32(float(depth[f]))) << 32 | uint64_t(lid);
    atomicMax(reinterpret_cast<unsigned long long*>(key + px), (unsigned long long)k);
    return;
  }
  const uint64_t k = fp32 ? depth_key(float(depth[f])) : depth_key(depth[f]);
  if (pass == 0) {
    atomicMax(reinterpret_cast<unsigned long long*>(key + px), (unsigned long long)k);
  } else if (k == __hip_atomic_load(key + px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    atomic_max_id(id + px, lid);
  }
}

// ----------------------------------------------------------------------
// resolve: the final colour of every pixel from its winning fragment
//
// A workgroup takes a 32 x 8 pixel tile of one image, in three phases:
//   1. one thread per pixel: the winning triangle, its barycentric weights
//      at the pixel centre, and the three lattice edges its vertices lie on.
//      The edges are entered in a hash table in LDS;
//   2. the tile's distinct edges are shared out over the waves, and each
//      one's smoothed vertex normal (normal.c:46-165) is formed once;
//   3. one thread per pixel again: shading (render.c:137-159) and the write,
//      in PPM row order (output.c:113-123).
// The normals of normal.c are needed only where a triangle is nearest, and
// a vertex normal depends on its lattice edge alone: the cells that share
// the edge are visited in increasing order and their triangles in slot
// order, whichever cell the vertex is seen from, so one sum serves every
// triangle with a vertex on the edge, bit for bit.
//
// What bounds it: the chain of dependent reads behind a vertex normal
// (corner values, code, slot masks, slots: 4, 2 or 1 cells per edge).  With
// one thread gathering all three normals of a pixel's triangle the chains
// ran one after the other and neighbouring pixels repeated them; a tile's
// 768 vertices are a few hundred distinct edges at a pixel per cell and a
// few dozen on a close-up.
constexpr uint32_t kTileW = 32, kTileH = kThreads / 32;  // pixels of a workgroup's tile
constexpr uint32_t kVtxSlots = 1024;                     // hash slots, at least 3 per pixel
static_assert(kTileW * kTileH == kThreads && kVtxSlots > 3 * kThreads, "the tile's vertices fit the hash table");

// The distinct vertices of a pixel tile: open addressing over vertex keys,
// each occupied slot numbered in order of entry (idx), and the numbered
// slots and their normals.
template <typename R>
struct VtxTable {
  unsigned long long key[kVtxSlots];
  uint16_t idx[kVtxSlots];
  uint16_t slot[3 * kThreads];
  R n[3 * kThreads][3];
  uint32_t count;
};

constexpr unsigned long long kNoVtx = ~0ull;

// A vertex's lattice edge as object, cell and direction: the edge runs from
// corner 0 of that cell to corner `dir` (1-7).  An interior cell's edges
// all start at corner 0 of a cell of the lattice.
__device__ __forceinline__ unsigned long long vtx_key(uint32_t obj, uint32_t cell, uint32_t dir) {
  return (unsigned long long)obj << 36 | (unsigned long long)cell << 4 | dir;
}

// the cell whose corner 0 is corner `lo` of cell c
__device__ __forceinline__ uint32_t corner_cell(uint32_t c, uint32_t lo, uint32_t ncx, uint32_t ncy) {
  return c + (lo & 1u) + (lo & 2u ? ncx : 0u) + (lo & 4u ? ncx * ncy : 0u);
}

// the lower corner and the direction of cell-local edge e
__device__ __forceinline__ void edge_lo_dir(uint32_t e, uint32_t& lo, uint32_t& dir) {
  if (e < 4u) {
    lo = 2u * e;
    dir = 1u;
  } else if (e < 8u) {
    lo = (e & 1u) | ((e - 4u) >> 1) << 2;
    dir = 2u;
  } else if (e < 12u) {
    lo = e - 8u;
    dir = 4u;
  } else if (e < 14u) {
    lo = e - 12u;
    dir = 6u;
  } else if (e < 16u) {
    lo = (e - 14u) << 1;
    dir = 5u;
  } else if (e < 18u) {
    lo = (e - 16u) << 2;
    dir = 3u;
  } else {
    lo = 0u;
    dir = 7u;
  }
}

// enters key k; returns its slot (idx and n are valid after a barrier)
template <typename R>
__device__ __forceinline__ uint32_t vtx_enter(VtxTable<R>& T, unsigned long long k) {
  uint32_t s = uint32_t((k * 0x9e3779b97f4a7c15ull) >> 54);
  static_assert(kVtxSlots == 1u << 10, "the hash keeps 10 bits");
  for (;;) {
    const unsigned long long was = atomicCAS(&T.key[s], kNoVtx, k);
    if (was == k) return s;
    if (was == kNoVtx) {
      const uint32_t u = atomicAdd(&T.count, 1u);
      T.idx[s] = uint16_t(u);
      T.slot[u] = uint16_t(s);
      return s;
    }
    s = (s + 1u) & (kVtxSlots - 1u);
  }
}

// The q-th of the n cells sharing the lattice edge from corner 0 of a cell
// in direction dir, in increasing linear order (normal.c:78-158): the edge
// starts at corner `lo` of that cell.  An axis edge is shared by four cells,
// a face diagonal by two, the body diagonal belongs to one.
__device__ __forceinline__ uint32_t sharing_corner(uint32_t dir, uint32_t q, uint32_t& n) {
  const uint32_t free = 7u ^ dir, a = free & (0u - free), b = free & (free - 1u);
  n = 1u << __popc(free);
  const uint32_t back = n - 1u - q;
  return (back & 1u ? a : 0u) | (back & 2u ? b : 0u);
}

// cell-local id of the edge from corner lo in direction dir (triangulate.c:23-32)
__device__ __forceinline__ uint32_t edge_id_at(uint32_t lo, uint32_t dir) {
  const uint32_t i = lo & 1u, j = (lo >> 1) & 1u, k = lo >> 2;
  const uint32_t by_axis = dir == 1u ? lo >> 1 : dir == 2u ? 4u + i + 2u * k : 8u + (lo & 3u);
  const uint32_t by_diag = dir == 6u ? 12u + i : dir == 5u ? 14u + j : dir == 3u ? 16u + k : 18u;
  return dir == 1u || dir == 2u || dir == 4u ? by_axis : by_diag;
}

// Vertex normals of every triangle of one object: rows of nine reals, NaN
// for triangles outside the rendered interior.  A workgroup takes 256
// consecutive triangles, enters their vertices in a table of lattice edges in
// LDS, forms each distinct vertex's normal once, a thread each, and writes
// the rows as contiguous words.
//
// A normal is the sum of vertex_normal -- cells sharing the vertex's lattice
// edge in the neighbour table's increasing order, in each the triangles with
// a vertex on the edge in slot order (c_emask of the cell's stored corner
// code), from +0 -- gathered directly: a neighbour cell's triangles start at
// bstart[its tile] + cstart[cell].  A thread's (at most four) neighbour cells
// are fetched together.  The sum depends on the edge alone, so it serves
// every triangle with a vertex there.
//
// What bounds it: the gather of each vertex's code, start and weight records
// through L1 and L2, 4 to 16 records a vertex.
// With a thread per (triangle, vertex), each vertex of a cell's triangles was
// gathered two or three times: 256^3 and two thresholds, FP64, 2 x 517 us
// then, 2 x 308 now, and 1.38 ms for the mesh built and smoothed, 1.34 with
// the rows stored non-temporally.
//
// (Measured against a thread per (triangle, vertex), the form before: one
// 32-bit cell word of code and start, the masks in LDS and a persistent grid
// were 5% slower; a workgroup per tile, tiles z-fastest along each column and
// one contiguous run per XCD (to keep the planes above and below in L2),
// 1.55-1.66x slower: the serial order streams the records and the normals in
// address order; a workgroup per tile gathering a window of cells into LDS
// 3-4x slower.)
template <typename R>
__device__ __forceinline__ V3<R> gathered_normal(const MeshView<R>& m, const ObjMeta& om, const uint8_t* cd,
                                                 const uint16_t* cs, uint32_t c, uint32_t e) {
  const int64_t sy = om.ncx, sz = int64_t(om.ncx) * om.ncy;
  const int nn = c_nbr.n[e];
  uint32_t mask[4];
  uint64_t s2[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    mask[q] = 0;
    s2[q] = 0;
    if (q < nn) {
      // an interior cell's neighbours lie inside the lattice
      const uint32_t c2 = uint32_t(int64_t(c) + c_nbr.v[e][q][0] * sz + c_nbr.v[e][q][1] * sy + c_nbr.v[e][q][2]);
      mask[q] = c_emask[uint32_t(cd[c2]) * 19u + uint32_t(c_nbr.v[e][q][3])];
      s2[q] = om.bstart[tile_of_cell(om, c2)] + cs[c2];
    }
  }
  // each neighbour's first four hits are loaded together, then added in
  // slot order (more hits, rare, follow one at a time)
  V3<R> sum = {R(0), R(0), R(0)};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    uint32_t h = mask[q];
    V3<R> wv[4];
    bool hv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint64_t u2 = s2[q] + uint32_t(__builtin_ctz(h | 0x80000000u));
      hv[r] = h != 0 && u2 < m.cap;
      wv[r] = hv[r] ? V3<R>{m.aux[u2].w[0], m.aux[u2].w[1], m.aux[u2].w[2]} : V3<R>{R(0), R(0), R(0)};
      h &= h - 1u;
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (hv[r]) sum = vadd(sum, wv[r]);
    for (; h; h &= h - 1u) {
      const uint64_t u2 = s2[q] + uint32_t(__builtin_ctz(h));
      if (u2 < m.cap) sum = vadd(sum, V3<R>{m.aux[u2].w[0], m.aux[u2].w[1], m.aux[u2].w[2]});
    }
  }
  return vunit(sum);
}

template <typename R>
__global__ __launch_bounds__(kThreads) void k_smooth(MeshView<R> m, const ObjMeta* __restrict__ meta,
                                                     const uint16_t* __restrict__ cstart, R* __restrict__ out) {
  __shared__ VtxTable<R> T;
  __shared__ uint16_t s_vtx[3 * kThreads];  // the slots of the triangles' vertices
  constexpr uint16_t kOutside = 0xffff;
  const ObjMeta om = *meta;
  const uint8_t* cd = m.code + om.code_off;
  const uint16_t* cs = cstart + om.code_off;
  const R nan = R(__longlong_as_double(0x7ff8000000000000ll));
  for (uint64_t t0 = uint64_t(blockIdx.x) * kThreads; t0 < om.count; t0 += uint64_t(gridDim.x) * kThreads) {
    for (uint32_t s = threadIdx.x; s < kVtxSlots; s += kThreads) T.key[s] = kNoVtx;
    if (threadIdx.x == 0) T.count = 0;
    __syncthreads();
    const uint32_t nt = om.count - t0 < kThreads ? uint32_t(om.count - t0) : kThreads;
    if (threadIdx.x < nt) {
      const uint64_t u = om.base + t0 + threadIdx.x;
      const uint32_t c = m.aux[u].cell, ed = edges_of(m, u);
#pragma unroll
      for (int n = 0; n < 3; n++) {
        uint32_t s = kOutside;
        if ((ed >> 15) & 1u) {
          uint32_t lo, dir;
          edge_lo_dir((ed >> (5 * n)) & 31u, lo, dir);
          s = vtx_enter(T, vtx_key(0u, corner_cell(c, lo, om.ncx, om.ncy), dir));
        }
        s_vtx[3u * threadIdx.x + n] = uint16_t(s);
      }
    }
    __syncthreads();
    for (uint32_t u = threadIdx.x; u < T.count; u += kThreads) {
      const unsigned long long key = T.key[T.slot[u]];
      const V3<R> n = gathered_normal<R>(m, om, cd, cs, uint32_t(key >> 4), edge_id_at(0u, uint32_t(key) & 7u));
      T.n[u][0] = n.x;
      T.n[u][1] = n.y;
      T.n[u][2] = n.z;
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < 9u * nt; w += kThreads) {
      const uint32_t v = w / 3u, s = s_vtx[v];
      // (the rows stream past the caches, which hold the records)
      __builtin_nontemporal_store(s == kOutside ? nan : T.n[T.idx[s]][w - 3u * v], out + 9u * t0 + w);
    }
    __syncthreads();  // the next triangles reuse the table
  }
}

// Unpacks n triangles of a stored mesh into the arrays that a host caller
// takes (null: not wanted), as doubles: positions, weights, vertex normals
// (vn: n rows of the mesh's precision), cells and edges.
//
// Bound by the copies to the host that follow it: 176 bytes a triangle over
// the bus.  Records unpacked by the host after a copy of them took 3.5 to 9
// ms for 61 x 57 x 50 turbulence built, copied and freed, by the state of the
// host allocator (8.2 beside the 1.98 this takes).
template <typename R>
__global__ __launch_bounds__(kThreads) void k_unpack(const MeshPos<R>* __restrict__ pos,
                                                     const MeshAux<R>* __restrict__ aux, const R* __restrict__ vn,
                                                     uint32_t n, double* __restrict__ opos, double* __restrict__ owfn,
                                                     double* __restrict__ ovn, uint32_t* __restrict__ ocell,
                                                     uint32_t* __restrict__ oedges) {
  for (uint32_t w = blockIdx.x * kThreads + threadIdx.x; w < 9u * n; w += gridDim.x * kThreads) {
    const uint32_t t = w / 9u, c = w - 9u * t;
    if (opos) opos[w] = double(pos[t].p[c]);
    if (ovn) ovn[w] = double(vn[w]);
    if (owfn && c < 3u) owfn[3u * t + c] = double(aux[t].w[c]);
    if (c == 0u) {
      if (ocell) ocell[t] = aux[t].cell;
      if (oedges) {
        if constexpr (sizeof(R) == 8) oedges[t] = aux[t].edges;
        else oedges[t] = pos[t].edges;
      }
    }
  }
}

// Scratch of one wave forming vertex normals: the triangles found around
// its 16 vertices (owner lane | slot << 6; an axis edge has at most 16, and
// the diagonals fewer) and the smoothing weights of 64 of them.
template <typename R>
struct WaveHits {
  uint16_t hit[256];
  R w[64][3];
};

// The winning triangle of one pixel, as phase 1 leaves it for phase 3.
template <typename R>
struct PixelTri {
  bool tri;
  uint32_t obj;
  R w0, w1, w2;
  uint32_t s[3];  // its vertices' slots
};

// barycentric weights at pixel (i, j) of a triangle with vertices p
template <typename R>
__device__ __forceinline__ void weights_at(const ViewDev<R>& v, const V3<R> p[3], int32_t i, int32_t j, PixelTri<R>& X) {
  Projected<R> P;
#pragma unroll
  for (int n = 0; n < 3; n++) project(v, p[n], P.q[n]);
  raster_box(v, P);
  pixel_weights(P, column_centre(v, i), row_centre(v, j), X.w0, X.w1, X.w2);
}

// A frame without a stored mesh: triangles are found from their ids (the
// object, cell and slot fields of tri_id64) and recomputed from the field.
template <typename R>
struct FieldSource {
  const TessJob* __restrict__ jobs;
  const ObjMeta* __restrict__ meta;
  const uint64_t* __restrict__ ids;

  // the winner at pixel p with key k: a triangle (obj, cell c, slot sl), a
  // line fragment (fi) or neither
  __device__ __forceinline__ void winner(const RasterJob<R>& J, uint64_t, uint64_t p, uint64_t k, bool& tri,
                                         bool& line, uint32_t& obj, uint32_t& c, uint32_t& sl, uint64_t& fi,
                                         double& dep) const {
    // tri_id64: (object + 1) << 40 | cell << 4 | slot
    const uint64_t id = ids[p];
    if constexpr (sizeof(R) == 8) dep = unord64(k);
    else dep = id ? double(unord32(uint32_t(k >> 32))) : -DBL_MAX;
    const uint64_t ob = id >> 40;
    line = ob == kLineObj;
    fi = id & ((uint64_t(1) << 40) - 1u);
    tri = id != 0 && !line && ob - 1u >= J.obj0 && ob - 1u < J.obj1;
    obj = uint32_t(ob - 1u);
    c = uint32_t(id >> 4);
    sl = uint32_t(id & 15u);
  }

  // phase 1 of the wave's pixels with a winning triangle (have)
  __device__ __forceinline__ void triangle(const ViewDev<R>& v, bool have, uint32_t obj, uint32_t c, uint32_t sl,
                                           int32_t i, int32_t j, VtxTable<R>& T, PixelTri<R>& X) const {
    const uint32_t job = have ? meta[obj].job : 0u;
    // one field pass of the wave's pixels at a time (usually all of them),
    // so that its constants are scalars
    for (uint64_t todo = __ballot(have); todo;) {
      const uint32_t jb = uint32_t(__builtin_amdgcn_readlane(int(job), __builtin_ctzll(todo)));
      const bool mine = have && job == jb;
      todo &= ~__ballot(mine);
      const FieldDev& f = jobs[jb].f;
      // a cell index outside the object's field or its interior, or a slot
      // outside its cell, can only come from a damaged id buffer:
      // such a pixel keeps the background rather than read out of bounds
      if (!mine || c >= f.ncells) continue;
      const double thr = jobs[jb].ts.thr[meta[obj].q & 3u];
      const CellLoc L = locate(f, c);
      if (!interior_cell(f, L)) continue;
      double cv[8];
      load_corners(f, L, cv);
      const uint32_t code = corner_code(thr, cv);
      if (sl >= c_ntri[code]) continue;
      const uint32_t ent = uint32_t(c_cslot[code * 12u + sl]);
      V3<R> wpos[3];
      // (the vertices' six values are read again, from L1: choosing them from
      // the eight in registers took 126 selects; four 1280 x 720 cameras 1.90
      // ms instead of 1.885, other frames within 0.5 %)
      slot_positions_mem<R>(f, L, thr, ent & 0x3ffffu, wpos);
      weights_at(v, wpos, i, j, X);
#pragma unroll
      for (int n = 0; n < 3; n++) {
        const uint32_t a = (ent >> (6 * n)) & 7u, b = (ent >> (6 * n + 3)) & 7u;
        X.s[n] = vtx_enter(T, vtx_key(obj, corner_cell(c, a & b, f.ncx, f.ncy), a ^ b));
      }
      X.obj = obj;
      X.tri = true;
    }
  }

  // Phase 2: the normals of the table's vertices, 16 a wave at a time.  Four
  // lanes per vertex read the (at most four) cells sharing its edge and list
  // the triangles with a vertex on it (c_emask), cell by cell and in slot
  // order; the listed triangles are then recomputed 64 at a time, one per
  // lane, and each vertex's first lane adds its own in list order, from +0,
  // and normalises: the sums of vertex_normal over a stored mesh, bit for
  // bit.  A lane that walked all of a vertex's cells and triangles itself
  // had chains four times as long, and the wave ran as many rounds as its
  // busiest lane.
  __device__ __forceinline__ void normals(VtxTable<R>& T, WaveHits<R>* scratch) const {
    const uint32_t lane = threadIdx.x & 63u, nv = T.count;
    WaveHits<R>& S = scratch[threadIdx.x >> 6];
    for (uint32_t u0 = (threadIdx.x >> 6) * 16u; u0 < nv; u0 += kThreads / 4u) {
      const uint32_t u = u0 + (lane >> 2), q = lane & 3u;
      const bool have = u < nv;
      const unsigned long long key = have ? T.key[T.slot[u]] : 0ull;
      const uint32_t obj = uint32_t(key >> 36), c = uint32_t(key >> 4), dir = uint32_t(key) & 7u;
      const uint32_t job = have ? meta[obj].job : 0u, qt = have ? meta[obj].q & 3u : 0u;
      // one field pass of the wave's vertices at a time (usually all of them)
      for (uint64_t todo = __ballot(have); todo;) {
        const uint32_t jb = uint32_t(__builtin_amdgcn_readlane(int(job), __builtin_ctzll(todo)));
        const bool mine = have && job == jb;
        todo &= ~__ballot(mine);
        const FieldDev& f = jobs[jb].f;
        uint32_t n, c2 = 0, mask = 0, code = 0;
        const uint32_t lo = sharing_corner(dir, q, n);
        if (mine && q < n) {
          c2 = c - ((lo & 1u) + (lo & 2u ? f.ncx : 0u) + (lo & 4u ? f.ncx * f.ncy : 0u));
          double v[8];
          load_corners(f, locate(f, c2), v);
          code = corner_code(jobs[jb].ts.thr[qt], v);
          mask = c_emask[code * 19u + edge_id_at(lo, dir)];
        }
        // where each lane's triangles start in the wave's list
        uint32_t end = uint32_t(__popc(mask));
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t y = __shfl_up(end, d, 64);
          if (lane >= uint32_t(d)) end += y;
        }
        uint32_t at = end - uint32_t(__popc(mask));
        const uint32_t first = at, last = uint32_t(__shfl(int(end), int(lane | 3u)));
        const uint32_t total = uint32_t(__builtin_amdgcn_readlane(int(end), 63));
        for (; mask; mask &= mask - 1u) S.hit[at++] = uint16_t(lane | uint32_t(__builtin_ctz(mask)) << 6);
        V3<R> sum = {R(0), R(0), R(0)};
        for (uint32_t h0 = 0; h0 < total; h0 += 64u) {
          wave_lds_fence();  // the list is written, and the last round's weights are added
          const uint32_t h = h0 + lane;
          const uint32_t e = S.hit[h < total ? h : total - 1u];
          const uint32_t cc = uint32_t(__shfl(int(c2), int(e & 63u)));
          const uint32_t cq = uint32_t(__shfl(int(code | qt << 8), int(e & 63u)));
          const uint32_t ent = uint32_t(c_cslot[(cq & 255u) * 12u + (e >> 6)]);
          V3<R> P[3];
          slot_positions_mem<R>(f, locate(f, cc), jobs[jb].ts.thr[cq >> 8], ent, P);
          const V3<R> w = smoothing_weight<R>(P);
          S.w[lane][0] = w.x;
          S.w[lane][1] = w.y;
          S.w[lane][2] = w.z;
          wave_lds_fence();
          if (q == 0) {
            const uint32_t a = first > h0 ? first - h0 : 0u, b = last < h0 + 64u ? last : h0 + 64u;
            for (uint32_t g = a; h0 + g < b; g++) sum = vadd(sum, V3<R>{S.w[g][0], S.w[g][1], S.w[g][2]});
          }
        }
        if (mine && q == 0) {
          const V3<R> nrm = vunit(sum);
          T.n[u][0] = nrm.x;
          T.n[u][1] = nrm.y;
          T.n[u][2] = nrm.z;
        }
        wave_lds_fence();
      }
    }
  }
};

// A stored mesh: triangles by serial id, with their records.
template <typename R>
struct MeshSource {
  MeshView<R> m;
  const ObjMeta* __restrict__ meta;
  int nobj;
  const uint32_t* __restrict__ idbuf;

  __device__ __forceinline__ void winner(const RasterJob<R>&, uint64_t ntri, uint64_t p, uint64_t k, bool& tri,
                                         bool& line, uint32_t& obj, uint32_t& c, uint32_t& sl, uint64_t& fi,
                                         double& dep) const {
    uint32_t id;
    if constexpr (sizeof(R) == 8) {
      id = idbuf[p];
      dep = unord64(k);
    } else {
      id = uint32_t(k);
      dep = id ? double(unord32(uint32_t(k >> 32))) : -DBL_MAX;
    }
    line = id > ntri;
    fi = id - ntri - 1;
    tri = id != 0 && !line;
    c = id - 1u;  // the serial position
    sl = 0;
    if (tri) {
      int lo = 0, hi = nobj - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (meta[mid].base <= c) lo = mid;
        else hi = mid - 1;
      }
      obj = uint32_t(lo);
    }
  }

  __device__ __forceinline__ void triangle(const ViewDev<R>& v, bool have, uint32_t obj, uint32_t t, uint32_t,
                                           int32_t i, int32_t j, VtxTable<R>& T, PixelTri<R>& X) const {
    if (!have) return;
    V3<R> p[3];
#pragma unroll
    for (int n = 0; n < 3; n++)
      p[n] = {m.pos[t].p[3 * n + 0], m.pos[t].p[3 * n + 1], m.pos[t].p[3 * n + 2]};
    weights_at(v, p, i, j, X);
    const uint32_t c = m.aux[t].cell, ed = edges_of(m, t);
    const uint32_t ncx = meta[obj].ncx, ncy = meta[obj].ncy;
#pragma unroll
    for (int n = 0; n < 3; n++) {
      uint32_t lo, dir;
      edge_lo_dir((ed >> (5 * n)) & 31u, lo, dir);
      X.s[n] = vtx_enter(T, vtx_key(obj, corner_cell(c, lo, ncx, ncy), dir));
    }
    X.obj = obj;
    X.tri = true;
  }

  __device__ __forceinline__ void normals(VtxTable<R>& T, WaveHits<R>*) const {
    for (uint32_t u = threadIdx.x; u < T.count; u += kThreads) {
      const unsigned long long key = T.key[T.slot[u]];
      const V3<R> n = vertex_normal<R>(m, meta[uint32_t(key >> 36)], uint32_t(key >> 4),
                                       edge_id_at(0u, uint32_t(key) & 7u));
      T.n[u][0] = n.x;
      T.n[u][1] = n.y;
      T.n[u][2] = n.z;
    }
  }
};

template <typename R, typename Source>
__device__ __forceinline__ void resolve_tile(const Source& src, VtxTable<R>& T, WaveHits<R>* hits,
                                             const RasterJob<R>* __restrict__ rjobs, int njobs, uint32_t frame_tile,
                                             const uint8_t* __restrict__ frag_rgb, uint64_t ntri,
                                             const uint64_t* __restrict__ key) {
  // the image of this tile
  int jb = 0;
  for (int hi = njobs - 1; jb < hi;) {
    const int mid = (jb + hi + 1) >> 1;
    if (rjobs[mid].tile0 <= frame_tile) jb = mid;
    else hi = mid - 1;
  }
  const RasterJob<R>& J = rjobs[jb];
  const ViewDev<R> v = J.v;
  const uint32_t tile = frame_tile - J.tile0, tw = (uint32_t(v.W) + kTileW - 1u) / kTileW;
  const uint32_t ty = tile / tw;
  const int32_t i = int32_t((tile - ty * tw) * kTileW + threadIdx.x % kTileW);
  const int32_t j = int32_t(ty * kTileH + threadIdx.x / kTileW);
  const bool inside = i < v.W && j < v.H;
  const uint64_t lp = uint64_t(j) * uint64_t(v.W) + uint64_t(i);

  bool tri = false, line = false;
  uint32_t obj = 0, c = 0, sl = 0;
  uint64_t fi = 0;
  double dep = 0;
  if (inside) src.winner(J, ntri, J.px0 + lp, key[J.px0 + lp], tri, line, obj, c, sl, fi, dep);
  PixelTri<R> X;
  X.tri = false;
  // a tile of background and lines has no vertices
  if (__syncthreads_or(tri)) {
    for (uint32_t s = threadIdx.x; s < kVtxSlots; s += kThreads) T.key[s] = kNoVtx;
    if (threadIdx.x == 0) T.count = 0;
    __syncthreads();
    src.triangle(v, tri, obj, c, sl, i, j, T, X);
    __syncthreads();
    src.normals(T, hits);
    __syncthreads();
  }
  if (!inside) return;
  uint8_t r = J.bg[0], gg = J.bg[1], b = J.bg[2];
  if (X.tri) {
    V3<R> nv3[3];
#pragma unroll
    for (int n = 0; n < 3; n++) {
      const R* q = T.n[T.idx[X.s[n]]];
      nv3[n] = {q[0], q[1], q[2]};
    }
    const V3<R> n = vunit(vadd(vscale(X.w0, nv3[0]), vadd(vscale(X.w1, nv3[1]), vscale(X.w2, nv3[2]))));
    const V3<R> light = {v.light[0], v.light[1], v.light[2]};
    const R fct = fmax(R(0.15), fabs(vdot(n, light)));
    const uint8_t* rgb = src.meta[X.obj].rgb;
    r = uint8_t(fct * R(rgb[0]));
    gg = uint8_t(fct * R(rgb[1]));
    b = uint8_t(fct * R(rgb[2]));
  } else if (line) {
    r = frag_rgb[3 * fi + 0];
    gg = frag_rgb[3 * fi + 1];
    b = frag_rgb[3 * fi + 2];
  }
  const uint64_t o = (uint64_t(v.H - 1 - j) * uint64_t(v.W) + uint64_t(i)) * 3;
  J.rgb[o + 0] = r;
  J.rgb[o + 1] = gg;
  J.rgb[o + 2] = b;
  if (J.depth) J.depth[lp] = dep;
}

// Occupancy: the FP64 table and scratch (38 KB) allow four workgroups per CU.
template <typename R, typename Source>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_resolve(
    Source src, const RasterJob<R>* __restrict__ rjobs, int njobs, uint32_t ntiles,
    const uint8_t* __restrict__ frag_rgb, const FrameHdr* __restrict__ hdr, const uint64_t* __restrict__ key,
    uint64_t max_tri) {
  // a frame of more triangles than it may hold is refused: write nothing
  if ((hdr->overflow & 1u) || hdr->ntri > max_tri) return;
  __shared__ VtxTable<R> T;
  __shared__ WaveHits<R> hits[kThreads / 64];
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    resolve_tile(src, T, hits, rjobs, njobs, tile, frag_rgb, hdr->ntri, key);
    __syncthreads();  // the next tile reuses the table
  }
}

// ----------------------------------------------------------------------
// host launchers

int persistent_blocks() {
  static int n = 0;
  if (n == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                 hipSuccess || cus <= 0)
      cus = 256;
    n = ((cus * 8 + 7) / 8) * 8;
  }
  return n;
}

static uint32_t grid8(uint64_t want, uint32_t cap) {
  uint64_t g = want < cap ? want : cap;
  if (g == 0) g = 1;
  return uint32_t((g + 7) / 8 * 8);
}

hipError_t launch_count(const TessJob* jobs, int njobs, uint32_t nitems, uint32_t* cnt, uint32_t grid,
                        hipStream_t st) {
  if (nitems == 0) return hipSuccess;
  hipLaunchKernelGGL(k_count, dim3(grid8(nitems, grid)), dim3(kThreads), 0, st, jobs, njobs, nitems, cnt);
  return hipGetLastError();
}

hipError_t launch_scan(const uint32_t* cnt, uint64_t* start, uint64_t n, uint64_t* tile_tmp, hipStream_t st) {
  const uint64_t ntile = (n + kScanTile - 1) / kScanTile;
  if (ntile == 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_scan_reduce, dim3(uint32_t(ntile)), dim3(kThreads), 0, st, cnt, n, tile_tmp);
  hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kThreads), 0, st, tile_tmp, ntile);
  hipLaunchKernelGGL(k_scan_apply, dim3(uint32_t(ntile)), dim3(kThreads), 0, st, cnt, n,
                     (const uint64_t*)tile_tmp, start);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_plan(const uint64_t* start, uint64_t ntiles, ObjMeta* meta, int nobj, RasterJob<R>* rjobs,
                       int njobs, FrameHdr* hdr, uint64_t cap, hipStream_t st) {
  hipLaunchKernelGGL(k_plan<R>, dim3(1), dim3(kThreads), 0, st, start, ntiles, meta, nobj, rjobs, njobs, hdr, cap);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_emit(const TessJob* jobs, int njobs, uint32_t nitems, const uint64_t* start, const MeshView<R>& m,
                       FrameHdr* hdr, uint32_t grid, hipStream_t st) {
  if (nitems == 0) return hipSuccess;
  hipLaunchKernelGGL(k_emit<R>, dim3(grid8(nitems, grid)), dim3(kThreads), 0, st, jobs, njobs, nitems, start, m, hdr);
  return hipGetLastError();
}

hipError_t launch_cell_starts(const uint8_t* code, const ObjMeta* meta_dev, uint32_t ntiles, uint16_t* cstart,
                              hipStream_t st) {
  if (ntiles == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_starts, dim3(ntiles), dim3(kThreads), 0, st, code, meta_dev, cstart);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_vertex_normals(const MeshView<R>& m, const ObjMeta* meta_dev, const uint16_t* cstart,
                                 uint64_t count, R* out, hipStream_t st) {
  if (count == 0) return hipSuccess;
  // one triangle per thread (the kernel strides past 2^24 workgroups)
  const uint64_t blocks = (count + kThreads - 1) / kThreads;
  const uint32_t grid = uint32_t(blocks < (uint64_t(1) << 24) ? blocks : (uint64_t(1) << 24));
  hipLaunchKernelGGL(k_smooth<R>, dim3(grid), dim3(kThreads), 0, st, m, meta_dev, cstart, out);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_unpack(const MeshPos<R>* pos, const MeshAux<R>* aux, const R* vn, uint32_t n, double* opos,
                         double* owfn, double* ovn, uint32_t* ocell, uint32_t* oedges, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_unpack<R>, dim3(grid8((9ull * n + kThreads - 1) / kThreads, 8192)), dim3(kThreads), 0, st, pos,
                     aux, vn, n, opos, owfn, ovn, ocell, oedges);
  return hipGetLastError();
}

hipError_t launch_zinit(uint64_t* key, uint32_t* id, uint64_t npx, int precision, FrameHdr* hdr, hipStream_t st) {
  const uint64_t k0 = precision == 0 ? 0x0010000000000000ull /* ord64(-DBL_MAX) */ : 0ull;
  hipLaunchKernelGGL(k_zinit, dim3(grid8((npx + 255) / 256, 4096)), dim3(256), 0, st, key, id, npx, k0, hdr);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_raster(const MeshView<R>& m, const RasterJob<R>* rjobs, int njobs, FrameHdr* hdr, int mode,
                         uint64_t* key, uint32_t* id, Frag* frags, uint32_t cap, uint32_t grid, hipStream_t st) {
  if (sizeof(R) == 4 && mode != kRasterFp32) return hipErrorInvalidValue;
  if (sizeof(R) == 8 && mode == kRasterFp32) return hipErrorInvalidValue;
  if (mode == kRasterFp32)
    hipLaunchKernelGGL((k_raster<R, kRasterFp32>), dim3(grid), dim3(kThreads), 0, st, m, rjobs, njobs, hdr, key, id,
                       frags, cap);
  else if (mode == kRasterDepth64)
    hipLaunchKernelGGL((k_raster<R, kRasterDepth64>), dim3(grid), dim3(kThreads), 0, st, m, rjobs, njobs, hdr, key,
                       id, frags, cap);
  else
    hipLaunchKernelGGL((k_raster<R, kRasterId64>), dim3(grid), dim3(kThreads), 0, st, m, rjobs, njobs, hdr, key, id,
                       frags, cap);
  return hipGetLastError();
}

hipError_t launch_frag_ids(const void* frags, bool wide, uint32_t cap, const FrameHdr* hdr, const uint64_t* key,
                           void* id, uint32_t grid, hipStream_t st) {
  if (wide)
    hipLaunchKernelGGL((k_frag_ids<Frag64, uint64_t>), dim3(grid), dim3(256), 0, st, static_cast<const Frag64*>(frags),
                       cap, hdr, key, static_cast<uint64_t*>(id));
  else
    hipLaunchKernelGGL((k_frag_ids<Frag, uint32_t>), dim3(grid), dim3(256), 0, st, static_cast<const Frag*>(frags), cap,
                       hdr, key, static_cast<uint32_t*>(id));
  return hipGetLastError();
}

hipError_t launch_line_frags(const uint32_t* pix, const double* depth, uint32_t cap, const FrameHdr* hdr, int pass,
                             int precision, uint64_t* key, void* id, bool wide, hipStream_t st) {
  if (cap == 0) return hipSuccess;
  const dim3 g((cap + 255) / 256);
  if (wide)
    hipLaunchKernelGGL(k_line_frags<uint64_t>, g, dim3(256), 0, st, pix, depth, hdr, pass, precision, key,
                       static_cast<uint64_t*>(id));
  else
    hipLaunchKernelGGL(k_line_frags<uint32_t>, g, dim3(256), 0, st, pix, depth, hdr, pass, precision, key,
                       static_cast<uint32_t*>(id));
  return hipGetLastError();
}

uint32_t resolve_tiles(uint64_t W, uint64_t H) {
  return uint32_t((W + kTileW - 1) / kTileW * ((H + kTileH - 1) / kTileH));
}

// a workgroup per tile (the kernel strides past 2^23 of them)
static dim3 resolve_grid(uint32_t ntiles) { return dim3(ntiles < (1u << 23) ? ntiles : (1u << 23)); }

template <typename R>
hipError_t launch_resolve(const MeshView<R>& m, const RasterJob<R>* rjobs, int njobs, uint32_t ntiles,
                          const ObjMeta* meta, int nobj, const uint8_t* frag_rgb, const FrameHdr* hdr,
                          const uint64_t* key, const uint32_t* id, hipStream_t st) {
  const MeshSource<R> src = {m, meta, nobj, id};
  hipLaunchKernelGGL((k_resolve<R, MeshSource<R>>), resolve_grid(ntiles), dim3(kThreads), 0, st, src, rjobs, njobs,
                     ntiles, frag_rgb, hdr, key, ~uint64_t(0));
  return hipGetLastError();
}

hipError_t launch_mesh_compare(const MeshView<double>& a, const ObjMeta* ma, const void* b, int b_fp32,
                               const ObjMeta* mb, uint64_t count, unsigned long long* out, hipStream_t st) {
  if (count == 0) return hipSuccess;
  const uint32_t grid = grid8((count + kThreads - 1) / kThreads, uint32_t(persistent_blocks()) * 4);
  if (b_fp32)
    hipLaunchKernelGGL((k_mesh_compare<double, float>), dim3(grid), dim3(kThreads), 0, st, a, ma,
                       *static_cast<const MeshView<float>*>(b), mb, count, out);
  else
    hipLaunchKernelGGL((k_mesh_compare<double, double>), dim3(grid), dim3(kThreads), 0, st, a, ma,
                       *static_cast<const MeshView<double>*>(b), mb, count, out);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_frame_begin(const TessJob* jobs, int njobs, const RasterJob<R>* rjobs, const uint32_t* jimg,
                              uint2* order, uint32_t* take, uint64_t* key, uint64_t* id, uint64_t npx, FrameHdr* hdr,
                              hipStream_t st) {
  const uint64_t want = (npx + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(k_frame_begin<R>, dim3(grid8(want > uint64_t(njobs) ? want : uint64_t(njobs), 4096)),
                     dim3(kThreads), 0, st, jobs, uint32_t(njobs), rjobs, jimg, order, take, key, id, npx, hdr);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_frame(const TessJob* jobs, const uint2* order, uint32_t ngroups, uint32_t shift, uint32_t* take,
                        const RasterJob<R>* rjobs, const uint32_t* jimg, FrameHdr* hdr, int mode, uint64_t* key,
                        uint64_t* id, Frag64* frags, uint32_t fcap, uint32_t grid, hipStream_t st) {
  if (ngroups == 0) return hipSuccess;
  const uint64_t bricks = uint64_t(ngroups) << (3 * shift);
  const dim3 g(grid8((bricks + kThreads / 64 - 1) / (kThreads / 64), grid));
  if (mode == kFrameDraw)
    hipLaunchKernelGGL((k_frame<R, kFrameDraw>), g, dim3(kThreads), 0, st, jobs, order, ngroups, shift, take, rjobs,
                       jimg, hdr, key, id, frags, fcap);
  else
    hipLaunchKernelGGL((k_frame<R, kFrameIds>), g, dim3(kThreads), 0, st, jobs, order, ngroups, shift,
                       take + 64 * 8, rjobs, jimg, hdr, key, id, frags, fcap);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_resolve_field(const TessJob* jobs, const RasterJob<R>* rjobs, int njobs, uint32_t ntiles,
                                const ObjMeta* meta, const uint8_t* frag_rgb, const FrameHdr* hdr, const uint64_t* key,
                                const uint64_t* id, uint64_t max_tri, hipStream_t st) {
  const FieldSource<R> src = {jobs, meta, id};
  hipLaunchKernelGGL((k_resolve<R, FieldSource<R>>), resolve_grid(ntiles), dim3(kThreads), 0, st, src, rjobs, njobs,
                     ntiles, frag_rgb, hdr, key, max_tri);
  return hipGetLastError();
}

template hipError_t launch_frame_begin<double>(const TessJob*, int, const RasterJob<double>*, const uint32_t*, uint2*,
                                               uint32_t*, uint64_t*, uint64_t*, uint64_t, FrameHdr*, hipStream_t);
template hipError_t launch_frame<double>(const TessJob*, const uint2*, uint32_t, uint32_t, uint32_t*,
                                         const RasterJob<double>*, const uint32_t*, FrameHdr*, int, uint64_t*, uint64_t*,
                                         Frag64*, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_resolve_field<double>(const TessJob*, const RasterJob<double>*, int, uint32_t, const ObjMeta*,
                                                 const uint8_t*, const FrameHdr*, const uint64_t*, const uint64_t*,
                                                 uint64_t, hipStream_t);
template hipError_t launch_frame_begin<float>(const TessJob*, int, const RasterJob<float>*, const uint32_t*, uint2*,
                                               uint32_t*, uint64_t*, uint64_t*, uint64_t, FrameHdr*, hipStream_t);
template hipError_t launch_frame<float>(const TessJob*, const uint2*, uint32_t, uint32_t, uint32_t*,
                                         const RasterJob<float>*, const uint32_t*, FrameHdr*, int, uint64_t*, uint64_t*,
                                         Frag64*, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_resolve_field<float>(const TessJob*, const RasterJob<float>*, int, uint32_t, const ObjMeta*,
                                                 const uint8_t*, const FrameHdr*, const uint64_t*, const uint64_t*,
                                                 uint64_t, hipStream_t);
template hipError_t launch_plan<double>(const uint64_t*, uint64_t, ObjMeta*, int, RasterJob<double>*, int, FrameHdr*,
                                        uint64_t, hipStream_t);
template hipError_t launch_plan<float>(const uint64_t*, uint64_t, ObjMeta*, int, RasterJob<float>*, int, FrameHdr*,
                                       uint64_t, hipStream_t);
template hipError_t launch_emit<double>(const TessJob*, int, uint32_t, const uint64_t*, const MeshView<double>&,
                                        FrameHdr*, uint32_t, hipStream_t);
template hipError_t launch_emit<float>(const TessJob*, int, uint32_t, const uint64_t*, const MeshView<float>&,
                                       FrameHdr*, uint32_t, hipStream_t);
template hipError_t launch_vertex_normals<double>(const MeshView<double>&, const ObjMeta*, const uint16_t*,
                                                  uint64_t, double*, hipStream_t);
template hipError_t launch_vertex_normals<float>(const MeshView<float>&, const ObjMeta*, const uint16_t*, uint64_t,
                                                 float*, hipStream_t);
template hipError_t launch_unpack<double>(const MeshPos<double>*, const MeshAux<double>*, const double*, uint32_t,
                                          double*, double*, double*, uint32_t*, uint32_t*, hipStream_t);
template hipError_t launch_unpack<float>(const MeshPos<float>*, const MeshAux<float>*, const float*, uint32_t, double*,
                                         double*, double*, uint32_t*, uint32_t*, hipStream_t);
template hipError_t launch_raster<double>(const MeshView<double>&, const RasterJob<double>*, int, FrameHdr*, int,
                                          uint64_t*, uint32_t*, Frag*, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_raster<float>(const MeshView<float>&, const RasterJob<float>*, int, FrameHdr*, int,
                                         uint64_t*, uint32_t*, Frag*, uint32_t, uint32_t, hipStream_t);
template hipError_t launch_resolve<double>(const MeshView<double>&, const RasterJob<double>*, int, uint32_t,
                                           const ObjMeta*, int, const uint8_t*, const FrameHdr*, const uint64_t*,
                                           const uint32_t*, hipStream_t);
template hipError_t launch_resolve<float>(const MeshView<float>&, const RasterJob<float>*, int, uint32_t,
                                           const ObjMeta*, int, const uint8_t*, const FrameHdr*, const uint64_t*,
                                           const uint32_t*, hipStream_t);

hipError_t upload_tables(const NbrTable& nt) {
  // case table of triangulate.c:204-270: reduced mask -> triangles as
  // (tail, head) tetra-vertex pairs
  static const int ntri[8] = {0, 1, 1, 2, 1, 2, 2, 1};
  static const int pairs[8][2][3][2] = {
      {{{0, 0}, {0, 0}, {0, 0}}, {{0, 0}, {0, 0}, {0, 0}}},
      {{{0, 1}, {0, 3}, {0, 2}}, {{0, 0}, {0, 0}, {0, 0}}},
      {{{1, 0}, {1, 2}, {1, 3}}, {{0, 0}, {0, 0}, {0, 0}}},
      {{{0, 2}, {1, 3}, {0, 3}}, {{0, 2}, {1, 2}, {1, 3}}},
      {{{2, 0}, {2, 3}, {2, 1}}, {{0, 0}, {0, 0}, {0, 0}}},
      {{{2, 1}, {0, 3}, {2, 3}}, {{2, 1}, {0, 1}, {0, 3}}},
      {{{0, 2}, {2, 3}, {1, 3}}, {{0, 2}, {1, 3}, {0, 1}}},
      {{{3, 0}, {3, 2}, {3, 1}}, {{0, 0}, {0, 0}, {0, 0}}},
  };
  static const int tet[6][4] = {{0, 7, 3, 1}, {0, 7, 1, 5}, {0, 7, 5, 4},
                                {0, 7, 4, 6}, {0, 7, 6, 2}, {0, 7, 2, 3}};
  hipError_t e;
  // per corner code: triangle count and every slot's corners and edge ids
  static uint8_t nt8[256];
  static uint64_t cs[256 * 12];
  static uint16_t em[256 * 19];
  auto eid = [](uint32_t a, uint32_t b) -> uint32_t {
    const uint32_t lo = a < b ? a : b;
    switch (a ^ b) {
      case 1: return lo >> 1;
      case 2: return 4 + (lo & 1) + 2 * (lo >> 2);
      case 4: return 8 + (lo & 3);
      case 6: return 12 + (lo & 1);
      case 5: return 14 + ((lo >> 1) & 1);
      case 3: return 16 + (lo >> 2);
      default: return 18;
    }
  };
  for (int code = 0; code < 256; code++) {
    int sl = 0;
    for (int t = 0; t < 6; t++) {
      int mk = 0;
      for (int n = 0; n < 4; n++) mk |= ((code >> tet[t][n]) & 1) << n;
      const bool rev = mk >= 8;
      const int mm = rev ? 15 - mk : mk;
      for (int s = 0; s < ntri[mm]; s++, sl++) {
        uint64_t ent = 0;
        for (int v = 0; v < 3; v++) {
          const int q = rev ? 2 - v : v;
          const uint32_t tail = uint32_t(tet[t][pairs[mm][s][q][0]]);
          const uint32_t head = uint32_t(tet[t][pairs[mm][s][q][1]]);
          ent |= uint64_t(tail | head << 3) << (6 * v);
          ent |= uint64_t(eid(tail, head)) << (18 + 5 * v);
          em[code * 19 + eid(tail, head)] |= uint16_t(1u << sl);
        }
        cs[code * 12 + sl] = ent;
      }
    }
    nt8[code] = uint8_t(sl);
  }
  e = hipMemcpyToSymbol(HIP_SYMBOL(c_ntri), nt8, sizeof(nt8));
  if (e != hipSuccess) return e;
  e = hipMemcpyToSymbol(HIP_SYMBOL(c_cslot), cs, sizeof(cs));
  if (e != hipSuccess) return e;
  e = hipMemcpyToSymbol(HIP_SYMBOL(c_emask), em, sizeof(em));
  if (e != hipSuccess) return e;
  return hipMemcpyToSymbol(HIP_SYMBOL(c_nbr), &nt, sizeof(nt));
}

NbrTable build_nbr_table() {
  // every cell within one step holding both endpoints of edge e as a
  // tetra edge, in increasing (dk, dj, di) = increasing linear order
  static const int tet[6][4] = {{0, 7, 3, 1}, {0, 7, 1, 5}, {0, 7, 5, 4},
                                {0, 7, 4, 6}, {0, 7, 6, 2}, {0, 7, 2, 3}};
  auto is_tet_edge = [&](int a, int b) {
    if (a == b) return false;
    for (int t = 0; t < 6; t++) {
      bool ha = false, hb = false;
      for (int n = 0; n < 4; n++) {
        ha |= tet[t][n] == a;
        hb |= tet[t][n] == b;
      }
      if (ha && hb) return true;
    }
    return false;
  };
  auto eid = [](int a, int b) {
    const int lo = a < b ? a : b;
    switch (a ^ b) {
      case 1: return lo >> 1;
      case 2: return 4 + (lo & 1) + 2 * (lo >> 2);
      case 4: return 8 + (lo & 3);
      case 6: return 12 + (lo & 1);
      case 5: return 14 + ((lo >> 1) & 1);
      case 3: return 16 + (lo >> 2);
      default: return 18;
    }
  };
  NbrTable nt = {};
  for (int a = 0; a < 8; a++) {
    for (int b = a + 1; b < 8; b++) {
      if (!is_tet_edge(a, b)) continue;
      const int e = eid(a, b);
      const int A[3] = {a & 1, (a >> 1) & 1, a >> 2};
      const int B[3] = {b & 1, (b >> 1) & 1, b >> 2};
      for (int dk = -1; dk <= 1; dk++)
        for (int dj = -1; dj <= 1; dj++)
          for (int di = -1; di <= 1; di++) {
            const int d[3] = {di, dj, dk};
            int la[3], lb[3];
            bool ok = true;
            for (int x = 0; x < 3; x++) {
              la[x] = A[x] - d[x];
              lb[x] = B[x] - d[x];
              ok = ok && la[x] >= 0 && la[x] <= 1 && lb[x] >= 0 && lb[x] <= 1;
            }
            if (!ok) continue;
            const int ca = la[0] + 2 * la[1] + 4 * la[2];
            const int cb = lb[0] + 2 * lb[1] + 4 * lb[2];
            if (!is_tet_edge(ca, cb)) continue;
            const int q = nt.n[e]++;
            nt.v[e][q][0] = int8_t(dk);
            nt.v[e][q][1] = int8_t(dj);
            nt.v[e][q][2] = int8_t(di);
            nt.v[e][q][3] = int8_t(eid(ca, cb));
          }
    }
  }
  return nt;
}

}  // namespace c3d
