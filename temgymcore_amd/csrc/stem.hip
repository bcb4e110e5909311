// 4D-STEM shadow-image model: forward (detector coordinates, bilinear sample
// lookup, optional 4D scatter) and the descan / geometry fit (loss + adjoint)
// over every (camera length, scan position, ray) in one launch.
//
// Model (per scan position s, ray j; see include/temgym_hip.h):
//   x_s   = sp_x + (th_x + st_x) * d                       sample plane
//   x_det = x_s + Dx + (th_x + st_x + Ddx) * L_c           detector
// with Dx = A0 . v + o_x - sp_x, Ddx = A2 . v + o_dx - st_x,
// v = (sp_x, sp_y, st_x, st_y), st = pivot * sp.  Hence
//   x_det = th_x * (d + L_c) + Bx(s, c),  y_det = th_y * (d + L_c) + By(s, c)
// (reference component bodies: Scanner components.py:279-285, propagation
// propagator.py:51-72, Descanner components.py:320-372).
//
// The fit kernel streams the f32 targets exactly once (HBM-bound).  For each
// (s, c) it reduces residual moments  sum r_x, sum r_x th_x, sum r_x th_y,
// sum r_y, sum r_y th_x, sum r_y th_y, sum |r|^2  (FP32 per lane and across
// the wavefront, FP64 across wavefronts), from which every parameter gradient
// follows exactly because the detector coordinates are affine in the slopes.
// Per-scan-position gradient rows go to a workspace that a second kernel sums
// in a fixed order (deterministic FP64 result).
#include <algorithm>
#include <cmath>
#include <mutex>

#include "tg_common.hpp"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxSide = 1024;
constexpr double kPi = 3.14159265358979323846;

typedef float f4 __attribute__((ext_vector_type(4)));

struct ScanPos {
  double spx, spy, stx, sty;
};

// Scan position of flattened scan index s: ScanGrid.pixels_to_metres with
// square pixels `step`, rotation `rot_deg`, centre 0, no flip
// (reference coordinate_transforms.py:50-101, test_component.py:356-378).
__device__ __forceinline__ ScanPos scan_position(const tg_stem_geometry& G, const double* P, int64_t s) {
  const int64_t i = s / G.scan_w, j = s % G.scan_w;
  const double step = P[16];
  const double phi = P[17] * (kPi / 180.0);
  const double u = step * ((double)i - 0.5 * (G.scan_h - 1));
  const double v = step * ((double)j - 0.5 * (G.scan_w - 1));
  double sn, cs;
  sincos(phi, &sn, &cs);
  ScanPos p;
  p.spx = -sn * u + cs * v;
  p.spy = -(cs * u + sn * v);
  p.stx = G.pivot * p.spx;
  p.sty = G.pivot * p.spy;
  return p;
}

__device__ __forceinline__ double row_dot(const double* A, int r, const ScanPos& p) {
  return A[4 * r + 0] * p.spx + A[4 * r + 1] * p.spy + A[4 * r + 2] * p.stx + A[4 * r + 3] * p.sty;
}

// Detector-coordinate offsets (Bx, By) for camera length L.
__device__ __forceinline__ void offsets_at(const tg_stem_geometry& G, const double* A, const ScanPos& p, double L,
                                           double& bx, double& by) {
  bx = p.stx * G.defocus + (row_dot(A, 0, p) + G.offsets[0]) + (row_dot(A, 2, p) + G.offsets[2]) * L;
  by = p.sty * G.defocus + (row_dot(A, 1, p) + G.offsets[1]) + (row_dot(A, 3, p) + G.offsets[3]) * L;
}

__device__ __forceinline__ float slope_of(const tg_stem_geometry& G, int k) {
  const double pitch = 2.0 * G.semi_conv / G.n_side;
  return (float)(((double)k - 0.5 * (G.n_side - 1)) * pitch);
}

// Bilinear lookup of the sample image at (x, y) metres; neighbours outside
// the image contribute zero.
// Sample-image pixel coordinates of the sample-plane position of slope
// (tx, ty) at one scan position.  The position is affine in the slope,
//   x = spx + (tx + stx) d,  y = spy + (ty + sty) d  (d = defocus),
// so (fy, fx) = origin + slope terms, with the origin and the four slope
// coefficients folded per scan position (FP64).
struct SampleMap {
  double fy0, fx0, ky_x, ky_y, kx_x, kx_y;
};

__device__ __forceinline__ SampleMap sample_map(const tg_stem_geometry& G, const ScanPos& p) {
  const double xc = p.spx + p.stx * G.defocus, yc = p.spy + p.sty * G.defocus;
  SampleMap m;
  m.fy0 = G.img_m[0] * yc + G.img_m[1] * xc + G.img_m[2];
  m.fx0 = G.img_m[3] * yc + G.img_m[4] * xc + G.img_m[5];
  m.ky_y = G.img_m[0] * G.defocus;
  m.ky_x = G.img_m[1] * G.defocus;
  m.kx_y = G.img_m[3] * G.defocus;
  m.kx_x = G.img_m[4] * G.defocus;
  return m;
}

__device__ __forceinline__ void sample_pixel(const SampleMap& m, float tx, float ty, double& fy, double& fx) {
  fy = fma(m.ky_y, (double)ty, fma(m.ky_x, (double)tx, m.fy0));
  fx = fma(m.kx_y, (double)ty, fma(m.kx_x, (double)tx, m.fx0));
}

// The sample-image region one scan position's rays read: kImgTile^2 pixels
// around the footprint centre, staged in LDS (pixels outside the image are
// never read from it: the lookup keeps the image-bounds test).
constexpr int kImgTile = 32;

// Bilinear lookup at pixel coordinates (fy, fx); neighbours outside the
// image contribute zero (the lookup is 0 when (floor fy, floor fx) is not in
// [-1, h) x [-1, w)).  The four neighbours come from the LDS tile when they
// all lie in it, else from global memory (same weights, same order).
__device__ __forceinline__ float bilinear_tiled(const tg_stem_geometry& G, const float* __restrict__ img,
                                                const float* tile, int oy, int ox, double fy, double fx) {
  const double y0d = floor(fy), x0d = floor(fx);
  if (!(y0d >= -1.0 && y0d < (double)G.img_h && x0d >= -1.0 && x0d < (double)G.img_w)) return 0.0f;
  const int y0 = (int)y0d, x0 = (int)x0d;
  const bool in_tile = y0 >= oy && y0 + 1 < oy + kImgTile && x0 >= ox && x0 + 1 < ox + kImgTile;
  const float wy = (float)(fy - y0d), wx = (float)(fx - x0d);
  float acc = 0.0f;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int yy = y0 + a, xx = x0 + b;
      if (yy < 0 || yy >= G.img_h || xx < 0 || xx >= G.img_w) continue;
      const float w = (a ? wy : 1.0f - wy) * (b ? wx : 1.0f - wx);
      const float v = in_tile ? tile[(yy - oy) * kImgTile + (xx - ox)] : img[(int64_t)yy * G.img_w + xx];
      acc = fmaf(w, v, acc);
    }
  }
  return acc;
}

// The lookup with a branch-free path for rays whose four neighbours all lie in
// a tile that is inside the image: bilinear_tiled's accumulation without its
// bounds tests.
__device__ __forceinline__ float sample_value(const tg_stem_geometry& G, const float* __restrict__ img,
                                              const float* tile, int oy, int ox, bool tile_inside, double fy,
                                              double fx) {
  const double y0d = floor(fy), x0d = floor(fx);
  // tile coordinates (clamped first: positions far off the image or NaN
  // only ever take the general path)
  const int y0 = (int)fmin(fmax(y0d, -1e8), 1e8) - oy, x0 = (int)fmin(fmax(x0d, -1e8), 1e8) - ox;
  if (tile_inside && y0 >= 0 && y0 < kImgTile - 1 && x0 >= 0 && x0 < kImgTile - 1) {
    const float wy = (float)(fy - y0d), wx = (float)(fx - x0d);
    const int t = y0 * kImgTile + x0;
    float v = fmaf((1.0f - wy) * (1.0f - wx), tile[t], 0.0f);
    v = fmaf((1.0f - wy) * wx, tile[t + 1], v);
    v = fmaf(wy * (1.0f - wx), tile[t + kImgTile], v);
    return fmaf(wy * wx, tile[t + kImgTile + 1], v);
  }
  return bilinear_tiled(G, img, tile, oy, ox, fy, fx);
}

// What all rays of a scan position share: the sample map, the origin of the
// tile x tile image (accumulator) tile around the footprint centre, and the
// constants of some camera lengths.
struct PositionSetup {
  SampleMap smap;
  float a[TG_STEM_MAX_CAM], bx[TG_STEM_MAX_CAM], by[TG_STEM_MAX_CAM];
  int oy, ox;
};

// By one wavefront for its workgroup, a lane a camera length (cam0 ..
// cam0 + n_cam - 1): about 600 instructions, f64 for the most part, that cost
// the other wavefronts as much again each when all made them.  Whole calls, all /
// one: forward of 5x5 positions, 16^2 rays 12.7 / 10.0 us, 64x64 positions, 16^2
// rays, 3 cameras 17.3 / 14.7; back-projection of 64x64 positions, 64^2 rays
// 72.4 / 69.5.
template <int TILE>
__device__ __forceinline__ void position_setup(const tg_stem_geometry& G, const double* __restrict__ P, int64_t s,
                                               int cam0, int n_cam, PositionSetup& out) {
  const int lane = threadIdx.x & 63;
  const double L = P[18 + cam0 + min(lane, n_cam - 1)];
  const ScanPos p = scan_position(G, P, s);
  const SampleMap m = sample_map(G, p);
  double bx, by;
  offsets_at(G, P, p, L, bx, by);
  if (lane < n_cam) {
    out.a[lane] = (float)(G.defocus + L);
    out.bx[lane] = (float)bx;
    out.by[lane] = (float)by;
  }
  if (lane == 0) {
    out.smap = m;
    // (origins far outside the image only send every lookup to global memory)
    out.oy = (int)fmin(fmax(floor(m.fy0) - TILE / 2, -4.0 * TILE), (double)G.img_h + 4.0 * TILE);
    out.ox = (int)fmin(fmax(floor(m.fx0) - TILE / 2, -4.0 * TILE), (double)G.img_w + 4.0 * TILE);
  }
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------
// rays per lane: a workgroup covers 4096 rays (one scan position of the
// 64x64 workload), so its set-up (slopes, scan position, camera offsets)
// is paid once per 4096 rays rather than per 1024.  Bound: HBM writes, 8 B a
// ray and camera length and 4 B a value: 16.7M rays 34 us into memory written
// just before (37.7 with a ray a lane and 8- and 4-byte stores), 41 us a call
// in a row (29 at a fill's rate: the workgroups' outputs lie 32 KB apart.
// Workgroups of 512 and 1,024 threads, closer together, took 38 and 49 us.)
constexpr int kFwdRays = 16;

__global__ __launch_bounds__(kThreads) void stem_forward_kernel(const tg_stem_geometry G, const double* __restrict__ P,
                                                                const float* __restrict__ img,
                                                                float* __restrict__ coords,
                                                                float* __restrict__ values,
                                                                float* __restrict__ image4d) {
  __shared__ __align__(8) float th[kMaxSide];
  __shared__ PositionSetup sh;
  __shared__ float tile[kImgTile * kImgTile];
  const int64_t s = blockIdx.y;
  const int64_t S = (int64_t)G.scan_h * G.scan_w;
  const int64_t J = (int64_t)G.n_side * G.n_side;
  if (threadIdx.x < 64) {
    position_setup<kImgTile>(G, P, s, 0, G.n_cam, sh);
  } else {
    for (int k = (int)threadIdx.x - 64; k < G.n_side; k += kThreads - 64) th[k] = slope_of(G, k);
  }
  __syncthreads();
  const SampleMap smap = sh.smap;
  const int oy = sh.oy, ox = sh.ox;
  if (img != nullptr) {
    // all of a thread's tile loads are issued before the first is used
    // (clamped indices, unpredicated; pixels outside the image become 0):
    // predicated loads in a loop made each one wait for the previous
    constexpr int kPerThread = kImgTile * kImgTile / kThreads;
    static_assert(kPerThread * kThreads == kImgTile * kImgTile, "tile loads per thread");
    float tv[kPerThread];
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const int k = (int)threadIdx.x + i * kThreads;
      const int yy = min(max(oy + k / kImgTile, 0), G.img_h - 1), xx = min(max(ox + k % kImgTile, 0), G.img_w - 1);
      tv[i] = img[(int64_t)yy * G.img_w + xx];
    }
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const int k = (int)threadIdx.x + i * kThreads;
      const int yy = oy + k / kImgTile, xx = ox + k % kImgTile;
      tile[k] = (yy >= 0 && yy < G.img_h && xx >= 0 && xx < G.img_w) ? tv[i] : 0.0f;
    }
  }
  __syncthreads();
  // the tile lies inside the image: lookups whose neighbours are all in the
  // tile need no image-bounds tests
  const bool tile_inside = oy >= 0 && ox >= 0 && oy + kImgTile <= G.img_h && ox + kImgTile <= G.img_w;
  const int jb = blockIdx.x * kThreads * kFwdRays;  // J <= 2^20
  // per-workgroup output bases; rays index them with 32-bit offsets
  float* __restrict__ vrow = values != nullptr ? values + s * J : nullptr;
  float2* __restrict__ crow = coords != nullptr ? (float2*)coords + s * J : nullptr;
  const int64_t cstride = S * J;  // between camera lengths, in float2
  // Rays j, j + 1 = (row iy, columns ix, ix + 1; n_side is even), stepped by
  // 2 kThreads without dividing.  Two a lane, so that they are stored together
  // where the outputs are aligned for it.
  const int n = G.n_side, drow = 2 * kThreads / n, dcol = 2 * kThreads % n;
  const int j0 = jb + 2 * (int)threadIdx.x;
  int iy = j0 / n, ix = j0 - (j0 / n) * n;
  const bool need_v = values != nullptr || image4d != nullptr;
  const bool wide_c = ((uintptr_t)coords & 15) == 0, wide_v = ((uintptr_t)values & 7) == 0;
#pragma unroll 2
  for (int u = 0; u < kFwdRays / 2; ++u, ix += dcol, iy += drow) {
    if (ix >= n) {
      ix -= n;
      ++iy;
    }
    const int j = j0 + u * 2 * kThreads;
    if (j >= (int)J) continue;
    const float2 tx = *(const float2*)(th + ix);
    const float ty = th[iy];
    float2 v = make_float2(0.0f, 0.0f);
    if (need_v) {
      double fy, fx;
      sample_pixel(smap, tx.x, ty, fy, fx);
      v.x = sample_value(G, img, tile, oy, ox, tile_inside, fy, fx);
      sample_pixel(smap, tx.y, ty, fy, fx);
      v.y = sample_value(G, img, tile, oy, ox, tile_inside, fy, fx);
      if (vrow != nullptr) {
        if (wide_v) {
          *(float2*)(vrow + j) = v;
        } else {
          vrow[j] = v.x;
          vrow[j + 1] = v.y;
        }
      }
    }
    float2* __restrict__ co = crow;
    for (int c = 0; c < G.n_cam; ++c, co += cstride) {
      const float2 xd = make_float2(fmaf(tx.x, sh.a[c], sh.bx[c]), fmaf(tx.y, sh.a[c], sh.bx[c]));
      const float yd = fmaf(ty, sh.a[c], sh.by[c]);
      if (co != nullptr) {
        if (wide_c) {
          *(f4*)(co + j) = f4{xd.x, yd, xd.y, yd};
        } else {
          co[j] = make_float2(xd.x, yd);
          co[j + 1] = make_float2(xd.y, yd);
        }
      }
      if (c == 0 && image4d != nullptr) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float x = k == 0 ? xd.x : xd.y;
          const double fy = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[0], (double)yd), __dmul_rn(G.det_m[1], (double)x)),
                                      G.det_m[2]);
          const double fx = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[3], (double)yd), __dmul_rn(G.det_m[4], (double)x)),
                                      G.det_m[5]);
          const int32_t py = tg::xla_f64_to_i32(rint(fy)), px = tg::xla_f64_to_i32(rint(fx));
          if (py >= 0 && py < G.det_h && px >= 0 && px < G.det_w)
            unsafeAtomicAdd(image4d + (s * G.det_h + py) * G.det_w + px, k == 0 ? v.x : v.y);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// simulated dataset: the 4D deposit alone, every pixel written once
// ---------------------------------------------------------------------------
// image4d[s, pixel] = sum of the sample values of scan position s's rays that
// land on the pixel (camera length 0): the positions, binning and lookup of
// stem_forward_kernel.  One workgroup walks bands of rows of one position's
// detector image: it deposits a band into LDS and writes it out, zeros
// included, so the dataset is neither cleared beforehand nor updated through
// memory.  Bound: HBM writes, 4 B a detector pixel.  A band takes 24 KB of LDS
// (four workgroups a CU, so that some store while others deposit), and only
// the ray rows that can reach the band are visited: the detector row is
// monotone in the slope row, so they are one range, found from each row's two
// end columns.  One wavefront sets the position up for all, once for all of
// the workgroup's bands (a few positions are shared by several workgroups).  64x64 positions of 256x256 pixels, 64x64 rays:
// 193 us (5.6 TB/s of writes; 379 us cleared by a fill and deposited with
// 16.7M global atomics).  The same without any rays takes 189 us: what is left
// above the 147 us of a plain fill is the set-up at the start of each round of
// workgroups and the scattered order of the writes.  Measured beside it: one
// band a workgroup 288, two 230, four 207 us; bands of 12/16/24/30 KB
// 214/210/196/198 us; a first band that differs from position to position
// 207-219 us; non-temporal stores 196 us.
// Cleared and deposited / this, whole calls: 64x64 positions of 70x201 pixels,
// 30^2 rays 62 / 50 us, of 128^2 87 / 52; 31x33 of 70x201, 40^2 rays 23 / 23.  LDS
// adds floats at half a lane a cycle (58 us for 16.7M), memory faster where every
// ray has a pixel of its own, and far slower where rays share them: 64x64
// positions, 64^2 rays on 100x130 pixels 107 / 119, 40^2 rays on 64^2 51 / 59, 64^2
// rays on 64^2 316 / 119.
constexpr int kBandFloats = 6144;

// float4s of LDS for a band of npix pixels, wherever in its first 16 bytes it begins
__host__ __device__ inline int band_quads(int npix) { return (npix + 6) / 4; }

__global__ __launch_bounds__(kThreads) void stem_dataset_kernel(const tg_stem_geometry G, const double* __restrict__ P,
                                                                const float* __restrict__ img, int band_rows,
                                                                int bands_each, float* __restrict__ image4d) {
  extern __shared__ __align__(16) float band[];  // band_quads float4s, then the slopes
  __shared__ float tile[kImgTile * kImgTile];
  __shared__ PositionSetup sh;
  __shared__ int sh_lo[2], sh_hi[2];
  const int64_t s = blockIdx.y;
  const int n = G.n_side, W = G.det_w;
  const int quads = band_quads(band_rows * W);
  float* th = band + 4 * quads;
  const int row_begin = (int)blockIdx.x * bands_each * band_rows;
  const int row_end = min(row_begin + bands_each * band_rows, G.det_h);
  if (threadIdx.x < 64) {
    position_setup<kImgTile>(G, P, s, 0, 1, sh);
    if (threadIdx.x == 0) {
      sh_lo[0] = n;
      sh_hi[0] = -1;
    }
  }
  for (int k = threadIdx.x; k < n; k += kThreads) th[k] = slope_of(G, k);
  for (int k = threadIdx.x; k < quads; k += kThreads) ((float4*)band)[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();
  const float a = sh.a[0], bx = sh.bx[0], by = sh.by[0];
  const int oy = sh.oy, ox = sh.ox;
  for (int k = threadIdx.x; k < kImgTile * kImgTile; k += kThreads) {
    const int yy = oy + k / kImgTile, xx = ox + k % kImgTile;
    const float v = img[(int64_t)min(max(yy, 0), G.img_h - 1) * G.img_w + min(max(xx, 0), G.img_w - 1)];
    tile[k] = (yy >= 0 && yy < G.img_h && xx >= 0 && xx < G.img_w) ? v : 0.0f;
  }
  const auto detector_row = [&](float xd, float yd) {
    return __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[0], (double)yd), __dmul_rn(G.det_m[1], (double)xd)), G.det_m[2]);
  };
  // the ray rows that can reach detector rows [r0, r1), into sh_lo/sh_hi[buf]
  const auto find_rows = [&](int r0, int r1, int buf) {
    const float x0 = fmaf(th[0], a, bx), x1 = fmaf(th[n - 1], a, bx);
    for (int k = threadIdx.x; k < n; k += kThreads) {
      const float yd = fmaf(th[k], a, by);
      const double f0 = detector_row(x0, yd), f1 = detector_row(x1, yd);
      // rounded rows are monotone between the ends; a row with a NaN (which
      // bins to 0) is always visited
      const bool miss = rint(fmax(f0, f1)) < (double)r0 || rint(fmin(f0, f1)) > (double)(r1 - 1);
      if (f0 != f0 || f1 != f1 || !miss) {
        atomicMin(&sh_lo[buf], k);
        atomicMax(&sh_hi[buf], k);
      }
    }
  };
  find_rows(row_begin, min(row_begin + band_rows, row_end), 0);
  __syncthreads();
  const SampleMap smap = sh.smap;
  const bool tile_inside = oy >= 0 && ox >= 0 && oy + kImgTile <= G.img_h && ox + kImgTile <= G.img_w;
  const int drow = kThreads / n, dcol = kThreads % n;
  int buf = 0;
  for (int r0 = row_begin; r0 < row_end; r0 += band_rows, buf ^= 1) {
    const int r1 = min(r0 + band_rows, row_end);
    float* __restrict__ dst = image4d + (s * G.det_h + r0) * W;
    // band pixel k lives at band[k + shift]: 16-byte aligned in LDS where it is in memory
    const int shift = (int)(((uintptr_t)dst >> 2) & 3);
    const int npix = (r1 - r0) * W;
    const int lo = sh_lo[buf], rays = (sh_hi[buf] - lo + 1) * n;  // <= 0: none
    int iy = lo + (int)threadIdx.x / n, ix = (int)threadIdx.x % n;
    for (int j = threadIdx.x; j < rays; j += kThreads) {
      const float tx = th[ix], ty = th[iy];
      const float xd = fmaf(tx, a, bx), yd = fmaf(ty, a, by);
      const double fy = detector_row(xd, yd);
      const double fx =
          __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[3], (double)yd), __dmul_rn(G.det_m[4], (double)xd)), G.det_m[5]);
      const int32_t py = tg::xla_f64_to_i32(rint(fy)), px = tg::xla_f64_to_i32(rint(fx));
      if (py >= r0 && py < r1 && px >= 0 && px < W) {
        double sy, sx;
        sample_pixel(smap, tx, ty, sy, sx);
        unsafeAtomicAdd(&band[(py - r0) * W + px + shift], sample_value(G, img, tile, oy, ox, tile_inside, sy, sx));
      }
      ix += dcol;
      iy += drow;
      if (ix >= n) {
        ix -= n;
        ++iy;
      }
    }
    if (threadIdx.x == 0) {
      sh_lo[buf ^ 1] = n;
      sh_hi[buf ^ 1] = -1;
    }
    __syncthreads();
    // out, and zero again
    for (int k = threadIdx.x; k < (npix + shift + 3) / 4; k += kThreads) {
      const f4 v = *(const f4*)(band + 4 * k);
      *(f4*)(band + 4 * k) = f4{0.f, 0.f, 0.f, 0.f};
      const int q = 4 * k - shift;  // first of four band pixels
      if (q >= 0 && q + 4 <= npix) {
        *(f4*)(dst + q) = v;
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (q + u >= 0 && q + u < npix) dst[q + u] = v[u];
      }
    }
    if (r1 < row_end) find_rows(r1, min(r1 + band_rows, row_end), buf ^ 1);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// shadow-image back-projection: the adjoint of the 4D deposit above
// ---------------------------------------------------------------------------
// image[q] += sum over rays (s, j) whose detector pixel (camera `cam`) lies on
// the detector of data4d[s, pixel] * w_q(s, j), with w_q the bilinear weight
// of sample pixel q at the ray's sample-plane position (the same weights,
// bounds and detector binning as stem_forward_kernel); weight[q] += w_q.
// One scan position's sample footprint is a few pixels across
// (defocus x semi-convergence), so each workgroup accumulates into a
// kBpTile^2 LDS tile centred on it and flushes that once; contributions
// outside the tile go to global memory directly.  FP64 accumulation.
//
// Each thread takes a kBpBlock x kBpBlock block of adjacent rays, whose
// sample positions span well under a pixel on the usual geometries: the
// block's bilinear deposits then fall in a 3 x 3 pixel window anchored at
// the floor of the block's smallest coordinates, accumulated in registers and
// added to the tile once (9 LDS atomics per 16 rays instead of 64; same-
// address LDS atomics from the lanes of a wavefront serialise, and bound the
// one-ray-at-a-time form).  A ray whose cell falls outside the window (wide
// footprints) deposits its four neighbours directly to the LDS tile (or to
// global memory outside it).
constexpr int kBpTile = 32;
constexpr int kBpBlock = 4;                        // rays per side of one thread's block
constexpr int kBpRayTile = 16 * kBpBlock;          // rays per side of one workgroup (16 x 16 blocks)
static_assert(kThreads == 256, "one workgroup = 16 x 16 ray blocks");

// Destination of a deposit to sample pixel (yy, xx): its index in the LDS
// tile, kBpGlobal for global memory, kBpSkip outside the image.  (The atomics
// stay at the call sites on the __shared__ arrays themselves, so that they
// compile to LDS atomics rather than flat ones.)
constexpr int kBpGlobal = -1, kBpSkip = -2;

__device__ __forceinline__ int bp_slot(const tg_stem_geometry& G, int oy, int ox, int yy, int xx) {
  if (yy < 0 || yy >= G.img_h || xx < 0 || xx >= G.img_w) return kBpSkip;
  const int ty_ = yy - oy, tx_ = xx - ox;
  return ty_ >= 0 && ty_ < kBpTile && tx_ >= 0 && tx_ < kBpTile ? ty_ * kBpTile + tx_ : kBpGlobal;
}

// One axis of a block's rays where sample and detector pixels are not rotated
// against the slopes: the row (column) of each ray of that axis depends on its
// own slope alone.
struct BpAxis {
  uint32_t at[kBpBlock];         // detector row (column), 0 where it is off the detector or past n
  float w[kBpBlock][3];          // window weights, 0 where the ray is out
  uint32_t hit, on_img, in_win;  // bit k: ray k lands on the detector, lies on the sample image, in the window
  int anchor;
};

// slope: the slopes from index i0; (m, m0): detector coordinate m d + m0 of the
// position d = slope a + b; (k, f0): sample coordinate k slope + f0.  Roundings
// as in the general form, whose cross terms are exact zeros.
__device__ __forceinline__ BpAxis bp_axis(const float* slope, int i0, int n, float a, float b, double m, double m0,
                                          int det, double k, double f0, int img, bool& finite) {
  BpAxis o;
  o.hit = o.on_img = o.in_win = 0;
  double f[kBpBlock];
#pragma unroll
  for (int i = 0; i < kBpBlock; ++i) {
    const float t = slope[min(i0 + i, n - 1)];
    const float d = fmaf(t, a, b);
    finite = finite && d * 0.0f == 0.0f;
    const int32_t p = tg::xla_f64_to_i32(rint(__dadd_rn(__dmul_rn(m, (double)d), m0)));
    const bool ok = (i0 + i < n) & ((uint32_t)p < (uint32_t)det);
    o.at[i] = ok ? (uint32_t)p : 0u;
    o.hit |= (uint32_t)ok << i;
    f[i] = fma(k, (double)t, f0);
  }
  const double lo = floor(fmin(f[0], f[kBpBlock - 1]));
  const bool anchored = lo > -4.0 && lo < (double)img + 4.0;
  o.anchor = anchored ? (int)lo : 0;
#pragma unroll
  for (int i = 0; i < kBpBlock; ++i) {
    const double q = floor(f[i]);
    const bool on = (q >= -1.0) & (q < (double)img);
    const float w = (float)(f[i] - q);
    const int at = (int)(on ? q : 0.0) - o.anchor;
    const bool win = on & anchored & ((unsigned)at <= 1u);
    o.on_img |= (uint32_t)on << i;
    o.in_win |= (uint32_t)win << i;
    const bool use = win & ((o.hit >> i) & 1u);
    o.w[i][0] = use & (at == 0) ? 1.0f - w : 0.0f;
    o.w[i][1] = use ? (at == 0 ? w : 1.0f - w) : 0.0f;
    o.w[i][2] = use & (at != 0) ? w : 0.0f;
  }
  return o;
}

// bit r kBpBlock + c: bit r of rows and bit c of columns
__device__ __forceinline__ uint32_t bp_outer(uint32_t rows, uint32_t cols) {
  uint32_t m = 0;
#pragma unroll
  for (int r = 0; r < kBpBlock; ++r) m |= (rows >> r) & 1u ? cols << (r * kBpBlock) : 0u;
  return m;
}

// WEIGHT: also accumulate weight[q] (the sum of w_q), else weight is unused.
// SEPARABLE: the cross terms of the sample and detector maps are zero, so that
// rows and columns are binned, looked up and weighted once each: a block's
// deposits are then sum_r wy_r (sum_c wx_c d_rc), 6 instructions a ray in place
// of about 110, and its weights (sum_r wy_r) (sum_c wx_c).  Bound: the gathered
// detector pixels (260 MB of cache lines for 16.7M rays); the general form,
// vector issue.  64x64 positions: 64^2 rays 67.6 / 49.2 us, 20^2 rays (whole
// call) 69.9 / 42.9.
template <bool WEIGHT, bool SEPARABLE>
__global__ __launch_bounds__(kThreads) void stem_backproject_kernel(const tg_stem_geometry G,
                                                                    const double* __restrict__ P,
                                                                    const float* __restrict__ data, int cam,
                                                                    double* __restrict__ image,
                                                                    double* __restrict__ weight) {
  __shared__ float th[kMaxSide];
  __shared__ double t_img[kBpTile * kBpTile];
  __shared__ double t_w[WEIGHT ? kBpTile * kBpTile : 1];
  __shared__ PositionSetup sh;
  const int64_t s = blockIdx.y;
  const int n = G.n_side;
  if (threadIdx.x < 64) {
    position_setup<kBpTile>(G, P, s, cam, 1, sh);
  } else {
    for (int k = (int)threadIdx.x - 64; k < n; k += kThreads - 64) th[k] = slope_of(G, k);
    for (int k = (int)threadIdx.x - 64; k < kBpTile * kBpTile; k += kThreads - 64) {
      t_img[k] = 0.0;
      if (WEIGHT) t_w[k] = 0.0;
    }
  }
  __syncthreads();
  const SampleMap smap = sh.smap;
  const int oy = sh.oy, ox = sh.ox;
  const float sh_a = sh.a[0], sh_bx = sh.bx[0], sh_by = sh.by[0];
  // this thread's block of rays: rows iy0.., columns ix0.. (clipped to n)
  const int ntx = (n + kBpRayTile - 1) / kBpRayTile;
  const int iy0 = (int)(blockIdx.x / ntx) * kBpRayTile + (int)(threadIdx.x / 16) * kBpBlock;
  const int ix0 = (int)(blockIdx.x % ntx) * kBpRayTile + (int)(threadIdx.x % 16) * kBpBlock;
  if (iy0 < n && ix0 < n) {
    int Y, X;  // window anchor
    uint32_t direct = 0;  // rays deposited one by one
    double acc[9], accw[WEIGHT ? 9 : 1];
#pragma unroll
    for (int k = 0; k < 9; ++k) acc[k] = 0.0;
#pragma unroll
    for (int k = 0; k < (WEIGHT ? 9 : 1); ++k) accw[k] = 0.0;
    const char* __restrict__ dimg = (const char*)(data + s * G.det_h * G.det_w);
    if constexpr (SEPARABLE) {
      bool finite = true;
      const BpAxis cols = bp_axis(th, ix0, n, sh_a, sh_bx, G.det_m[4], G.det_m[5], G.det_w, smap.kx_x, smap.fx0,
                                  G.img_w, finite);
      const BpAxis rows = bp_axis(th, iy0, n, sh_a, sh_by, G.det_m[0], G.det_m[2], G.det_h, smap.ky_y, smap.fy0,
                                  G.img_h, finite);
      Y = rows.anchor;
      X = cols.anchor;
      float dv[kBpBlock * kBpBlock];
#pragma unroll
      for (int r = 0; r < kBpBlock; ++r)
#pragma unroll
        for (int c = 0; c < kBpBlock; ++c)
          dv[r * kBpBlock + c] = *(const float*)(dimg + ((rows.at[r] * (uint32_t)G.det_w + cols.at[c]) << 2));
      __builtin_amdgcn_sched_barrier(0);  // all 16 loads in flight before the deposits
      if (finite) {
        const uint32_t use = bp_outer(rows.hit & rows.in_win, cols.hit & cols.in_win);
        direct = bp_outer(rows.hit & rows.on_img, cols.hit & cols.on_img) & ~use;
        double rx[kBpBlock][3], sx[3] = {0.0, 0.0, 0.0}, sy[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < kBpBlock; ++c)
#pragma unroll
          for (int k = 0; k < 3; ++k) sx[k] += rx[c][k] = (double)cols.w[c][k];
#pragma unroll
        for (int r = 0; r < kBpBlock; ++r) {
          double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
          for (int c = 0; c < kBpBlock; ++c) {
            const double d = (double)((use >> (r * kBpBlock + c)) & 1u ? dv[r * kBpBlock + c] : 0.0f);
#pragma unroll
            for (int k = 0; k < 3; ++k) t[k] = fma(rx[c][k], d, t[k]);
          }
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const double ry = (double)rows.w[r][i];
            sy[i] += ry;
#pragma unroll
            for (int k = 0; k < 3; ++k) acc[3 * i + k] = fma(ry, t[k], acc[3 * i + k]);
          }
        }
        if (WEIGHT) {
#pragma unroll
          for (int k = 0; k < 9; ++k) accw[k] = sy[k / 3] * sx[k % 3];
        }
      } else {
        // an infinite or NaN position: the zero cross terms turn its partner's
        // coordinate into NaN, so every ray by itself
        for (int k = 0; k < kBpBlock * kBpBlock; ++k) {
          const int iy = iy0 + k / kBpBlock, ix = ix0 + k % kBpBlock;
          if (iy >= n || ix >= n) continue;
          const float xd = fmaf(th[ix], sh_a, sh_bx), yd = fmaf(th[iy], sh_a, sh_by);
          const double dfy = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[0], (double)yd), __dmul_rn(G.det_m[1], (double)xd)),
                                       G.det_m[2]);
          const double dfx = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[3], (double)yd), __dmul_rn(G.det_m[4], (double)xd)),
                                       G.det_m[5]);
          const int32_t py = tg::xla_f64_to_i32(rint(dfy)), px = tg::xla_f64_to_i32(rint(dfx));
          double fy, fx;
          sample_pixel(smap, th[ix], th[iy], fy, fx);
          const double y0d = floor(fy), x0d = floor(fx);
          const bool on = ((uint32_t)py < (uint32_t)G.det_h) & ((uint32_t)px < (uint32_t)G.det_w) & (y0d >= -1.0) &
                          (y0d < (double)G.img_h) & (x0d >= -1.0) & (x0d < (double)G.img_w);
          direct |= (uint32_t)on << k;
        }
      }
    } else {
      // The sample position fma(ky_y, ty, fma(ky_x, tx, fy0)) (likewise fx) and
      // the detector coordinate ((m0 yd) + (m1 xd)) + m2 (likewise fx) take
      // their inner terms from the ray's column (tx, xd) or row (ty, yd) alone:
      // computed once per row and column of the block, with the same roundings
      // as the per-ray expressions of stem_forward_kernel.  Rows and columns
      // past n repeat the last one (their rays are masked out below).
      double cy[kBpBlock], cx[kBpBlock], tyd[kBpBlock];
      double ry0[kBpBlock], ry3[kBpBlock], cx1[kBpBlock], cx4[kBpBlock];
#pragma unroll
      for (int k = 0; k < kBpBlock; ++k) {
        const float tx = th[min(ix0 + k, n - 1)], ty = th[min(iy0 + k, n - 1)];
        cy[k] = fma(smap.ky_x, (double)tx, smap.fy0);
        cx[k] = fma(smap.kx_x, (double)tx, smap.fx0);
        tyd[k] = (double)ty;
        const float xd = fmaf(tx, sh_a, sh_bx), yd = fmaf(ty, sh_a, sh_by);
        ry0[k] = __dmul_rn(G.det_m[0], (double)yd);
        ry3[k] = __dmul_rn(G.det_m[3], (double)yd);
        cx1[k] = __dmul_rn(G.det_m[1], (double)xd);
        cx4[k] = __dmul_rn(G.det_m[4], (double)xd);
      }
      // window anchor: floor of the smallest sample coordinates over the
      // block's corners (the position is affine in the slopes)
      constexpr int L = kBpBlock - 1;
      const double wy0 = floor(fmin(fmin(fma(smap.ky_y, tyd[0], cy[0]), fma(smap.ky_y, tyd[0], cy[L])),
                                    fmin(fma(smap.ky_y, tyd[L], cy[0]), fma(smap.ky_y, tyd[L], cy[L]))));
      const double wx0 = floor(fmin(fmin(fma(smap.kx_y, tyd[0], cx[0]), fma(smap.kx_y, tyd[0], cx[L])),
                                    fmin(fma(smap.kx_y, tyd[L], cx[0]), fma(smap.kx_y, tyd[L], cx[L]))));
      // anchors far outside the image: every ray deposits directly (and skips)
      const bool anchored = wy0 > -4.0 && wy0 < (double)G.img_h + 4.0 && wx0 > -4.0 && wx0 < (double)G.img_w + 4.0;
      Y = anchored ? (int)wy0 : 0;
      X = anchored ? (int)wx0 : 0;
      // the block's 16 detector values, all loads issued before the first is
      // used (the position's first pixel stands in for a ray off the detector
      // or past n; `hit` says which rays are real): a load per ray behind its
      // bounds test waited for each in turn.  One scan position's detector
      // image is addressed by a 32-bit byte offset from a uniform base (the
      // host bounds det_h * det_w by 2^30).
      float dv[kBpBlock * kBpBlock];
      uint32_t hit = 0;
#pragma unroll
      for (int r = 0; r < kBpBlock; ++r) {
#pragma unroll
        for (int c = 0; c < kBpBlock; ++c) {
          const double dfy = __dadd_rn(__dadd_rn(ry0[r], cx1[c]), G.det_m[2]);
          const double dfx = __dadd_rn(__dadd_rn(ry3[r], cx4[c]), G.det_m[5]);
          const int32_t py = tg::xla_f64_to_i32(rint(dfy)), px = tg::xla_f64_to_i32(rint(dfx));
          // (& rather than &&: one straight-line test, no exec-mask branches)
          const bool ok = (iy0 + r < n) & (ix0 + c < n) & ((uint32_t)py < (uint32_t)G.det_h) &
                          ((uint32_t)px < (uint32_t)G.det_w);
          dv[r * kBpBlock + c] = *(const float*)(dimg + (ok ? (uint32_t)(py * G.det_w + px) << 2 : 0u));
          hit |= (uint32_t)ok << (r * kBpBlock + c);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // all 16 loads in flight before the deposits
      // Per ray, straight-line: the window deposit runs for every ray with its
      // weights and value selected to zero unless the ray is real, on the
      // image and inside the window.  Rays on the image outside the window
      // (wide footprints; rare) are marked in `direct` and deposited by the
      // loop below.  (Conditional blocks in this unrolled loop would let the
      // compiler sink the gathered loads into them and keep the rays' values
      // live across them.)
#pragma unroll
      for (int r = 0; r < kBpBlock; ++r) {
#pragma unroll
        for (int c = 0; c < kBpBlock; ++c) {
          const bool real = (hit >> (r * kBpBlock + c)) & 1u;
          // bilinear weights at the sample-plane position, as in bilinear_tiled()
          const double fy = fma(smap.ky_y, tyd[r], cy[c]), fx = fma(smap.kx_y, tyd[r], cx[c]);
          const double y0d = floor(fy), x0d = floor(fx);
          const bool on_img = (y0d >= -1.0) & (y0d < (double)G.img_h) & (x0d >= -1.0) & (x0d < (double)G.img_w);
          // (positions off the image, NaN included, convert a stand-in 0)
          const int y0 = (int)(on_img ? y0d : 0.0), x0 = (int)(on_img ? x0d : 0.0);
          const float wy = (float)(fy - y0d), wx = (float)(fx - x0d);
          const int dy = y0 - Y, dx = x0 - X;
          const bool win = real & on_img & anchored & ((unsigned)dy <= 1u) & ((unsigned)dx <= 1u);
          direct |= (uint32_t)(real & on_img & !win) << (r * kBpBlock + c);
          // separable weights placed in the 3 x 3 window: row i of the window
          // carries (1 - wy) at dy and wy at dy + 1, likewise columns.  rx * d
          // is exact in FP64 (two 24-bit significands), so each deposit
          // ry * rx * d is rounded once, by the FMA into the sum.
          float ry[3] = {win & (dy == 0) ? 1.0f - wy : 0.0f, win ? (dy == 0 ? wy : 1.0f - wy) : 0.0f,
                         win & (dy != 0) ? wy : 0.0f};
          float rx[3] = {win & (dx == 0) ? 1.0f - wx : 0.0f, win ? (dx == 0 ? wx : 1.0f - wx) : 0.0f,
                         win & (dx != 0) ? wx : 0.0f};
          float df = win ? dv[r * kBpBlock + c] : 0.0f;
          // (the selects stay in f32: without these empty statements the
          // compiler converts first and selects both halves of each double)
#pragma unroll
          for (int k = 0; k < 3; ++k) asm volatile("" : "+v"(ry[k]), "+v"(rx[k]));
          asm volatile("" : "+v"(df));
          const double d = (double)df;
          double rxd[3], t[3];
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            rxd[k] = (double)rx[k];
            t[k] = rxd[k] * d;
          }
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const double ryd = (double)ry[i];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              acc[3 * i + k] = fma(ryd, t[k], acc[3 * i + k]);
              if (WEIGHT) accw[3 * i + k] = fma(ryd, rxd[k], accw[3 * i + k]);
            }
          }
          // one ray at a time: instruction selection would otherwise defer
          // every ray's sums past the last ray's set-up and hold all their
          // weights live at once.  (The empty statements emit nothing; they
          // make this ray's sums complete before the next ray's begin.)
#pragma unroll
          for (int k = 0; k < 9; ++k) {
            asm volatile("" : "+v"(acc[k]));
            if (WEIGHT) asm volatile("" : "+v"(accw[k]));
          }
        }
      }
    }
    // direct deposits: the ray's position and detector value again, by the
    // same operations, then its four bilinear neighbours straight to the LDS
    // tile (or global memory outside it)
    while (direct != 0u) {
      const int k = __builtin_ctz(direct);
      direct &= direct - 1u;
      const int r = k / kBpBlock, c = k % kBpBlock;
      const float tx = th[ix0 + c], ty = th[iy0 + r];  // real rays lie inside n
      double fy, fx;
      sample_pixel(smap, tx, ty, fy, fx);
      const float xd = fmaf(tx, sh_a, sh_bx), yd = fmaf(ty, sh_a, sh_by);
      const double dfy = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[0], (double)yd), __dmul_rn(G.det_m[1], (double)xd)),
                                   G.det_m[2]);
      const double dfx = __dadd_rn(__dadd_rn(__dmul_rn(G.det_m[3], (double)yd), __dmul_rn(G.det_m[4], (double)xd)),
                                   G.det_m[5]);
      const int32_t py = tg::xla_f64_to_i32(rint(dfy)), px = tg::xla_f64_to_i32(rint(dfx));
      const double dd = (double)*(const float*)(dimg + ((uint32_t)(py * G.det_w + px) << 2));
      const double y0d = floor(fy), x0d = floor(fx);
      const int y0 = (int)y0d, x0 = (int)x0d;  // on the image: marked rays only
      const float wy = (float)(fy - y0d), wx = (float)(fx - x0d);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const double w = (double)(a ? wy : 1.0f - wy) * (double)(b ? wx : 1.0f - wx);  // exact
          const int q = bp_slot(G, oy, ox, y0 + a, x0 + b);
          if (q >= 0) {
            atomicAdd(&t_img[q], w * dd);
            if (WEIGHT) atomicAdd(&t_w[q], w);
          } else if (q == kBpGlobal) {
            const int64_t gq = (int64_t)(y0 + a) * G.img_w + (x0 + b);
            unsafeAtomicAdd(image + gq, w * dd);
            if (WEIGHT) unsafeAtomicAdd(weight + gq, w);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      // untouched window pixels hold exact zeros (as do zero deposits, which
      // change no sum)
      if (WEIGHT ? accw[k] == 0.0 : acc[k] == 0.0) continue;
      const int yy = Y + k / 3, xx = X + k % 3;
      const int q = bp_slot(G, oy, ox, yy, xx);
      if (q >= 0) {
        atomicAdd(&t_img[q], acc[k]);
        if (WEIGHT) atomicAdd(&t_w[q], accw[k]);
      } else if (q == kBpGlobal) {
        const int64_t gq = (int64_t)yy * G.img_w + xx;
        unsafeAtomicAdd(image + gq, acc[k]);
        if (WEIGHT) unsafeAtomicAdd(weight + gq, accw[k]);
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kBpTile * kBpTile; k += kThreads) {
    const int yy = oy + k / kBpTile, xx = ox + k % kBpTile;
    if (yy < 0 || yy >= G.img_h || xx < 0 || xx >= G.img_w) continue;  // never written
    const int64_t q = (int64_t)yy * G.img_w + xx;
    if (t_img[k] != 0.0) unsafeAtomicAdd(image + q, t_img[k]);
    if (WEIGHT && t_w[k] != 0.0) unsafeAtomicAdd(weight + q, t_w[k]);
  }
}

// ---------------------------------------------------------------------------
// fit: forward + adjoint
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int kMom = 7;  // sum rx, rx*tx, rx*ty, ry, ry*tx, ry*ty, |r|^2
constexpr int kPerLane = 8;
constexpr int64_t kTile = (int64_t)kThreads * kPerLane;

// Tile `it` (camera c = it / ntile, tile it % ntile) of scan position s:
// N float4 per lane, lane-strided so each load instruction of a
// wavefront covers 1 KiB of contiguous targets.  Streamed once: non-temporal.
// Indices past the row's end are clamped to its last float4 (the tile sums
// skip those pairs), so every load is issued unpredicated: predicated loads
// made the compiler wait for all outstanding loads before the first use.
template <int N>
__device__ __forceinline__ void load_tile(const f4* __restrict__ T4, int64_t S, int64_t s, int64_t npair,
                                          int64_t ntile, int64_t it, f4 (&dst)[N]) {
  const int64_t c = it / ntile, tile = it - c * ntile;
  const int64_t row = (c * S + s) * npair;
  const int64_t q0 = tile * kTile + threadIdx.x;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int64_t q = q0 + (int64_t)k * kThreads;
    dst[k] = __builtin_nontemporal_load(T4 + row + (q < npair ? q : npair - 1));
  }
}

// Per-scan-position gradient terms from the per-camera moments M[c][k]
// (FP64 sums of the wavefront partials, waves in order); thread t < np
// writes entry t of the workspace row s (the np terms of one scan position
// are contiguous: one short coalesced store per workgroup, where a column
// layout cost 27 scattered 8-byte stores and ~9 us per pass).  Every term
// is linear in the moments with coefficients affine in the camera length
// L_c, so entries 0..17 need only the camera sums of the x and y residual
// totals, plain and L-weighted; entry 18 + c takes camera c alone and the
// last entry sums |r|^2.  In two parts, so that the coefficients of thread t
// can be made while the targets are on their way.
struct FitCoef {
  double x, xl, y, yl;
};

__device__ __forceinline__ FitCoef fit_coef(const tg_stem_geometry& G, const double* __restrict__ P, const ScanPos& p,
                                            int64_t s, int t) {
  const int np = 18 + G.n_cam + 1;
  const double* A = P;
  FitCoef f = {0.0, 0.0, 0.0, 0.0};
  if (t >= np - 1) return f;
  if (t >= 18) {
    f.x = row_dot(A, 2, p) + G.offsets[2];  // dbx / dL
    f.y = row_dot(A, 3, p) + G.offsets[3];  // dby / dL
  } else if (t < 16) {
    // d/dA[r][k] of sum_c |r_c|^2: rows 0, 1 act on the offsets (x, y),
    // rows 2, 3 on the slopes (scaled by L_c); column k picks v[k]
    const int k = t & 3;
    f.x = 2.0 * (k == 0 ? p.spx : k == 1 ? p.spy : k == 2 ? p.stx : p.sty);
  } else {
    // d(Bx, By) / d(spx, spy) = a + b L_c, with st = pivot * sp
    const double d = G.defocus, kap = G.pivot;
    const double ax_x = kap * d + (A[0] + A[2] * kap), bx_x = A[8] + A[10] * kap;
    const double ax_y = A[1] + A[3] * kap, bx_y = A[9] + A[11] * kap;
    const double ay_x = A[4] + A[6] * kap, by_x = A[12] + A[14] * kap;
    const double ay_y = kap * d + (A[5] + A[7] * kap), by_y = A[13] + A[15] * kap;
    double dsx, dsy;
    if (t == 16) {
      // step: sp = step * (rotated integer pixel offsets), so d sp / d step
      // is the offsets themselves (finite at step = 0, where sp / step is 0/0)
      const int64_t i = s / G.scan_w, j = s % G.scan_w;
      const double u1 = (double)i - 0.5 * (G.scan_h - 1);
      const double v1 = (double)j - 0.5 * (G.scan_w - 1);
      double sn, cs;
      sincos(P[17] * (kPi / 180.0), &sn, &cs);
      dsx = -sn * u1 + cs * v1;
      dsy = -(cs * u1 + sn * v1);
    } else {        // rotation in degrees: d sp_x = sp_y dphi, d sp_y = -sp_x dphi
      dsx = p.spy * (kPi / 180.0);
      dsy = -p.spx * (kPi / 180.0);
    }
    f.x = ax_x * dsx + ax_y * dsy;
    f.xl = bx_x * dsx + bx_y * dsy;
    f.y = ay_x * dsx + ay_y * dsy;
    f.yl = by_x * dsx + by_y * dsy;
  }
  return f;
}

// Entry t of a scan position from its moments M [n_cam][kMom].
__device__ __forceinline__ double fit_value(const tg_stem_geometry& G, const double* __restrict__ P, const FitCoef& f,
                                            const double* M, int t) {
  const double* L = P + 18;
  double g = 0.0;
  if (t == 18 + G.n_cam) {
    for (int c = 0; c < G.n_cam; ++c) g += M[c * kMom + 6];
  } else if (t >= 18) {
    const double* m = M + (t - 18) * kMom;
    g = 2.0 * (m[1] + f.x * m[0] + m[5] + f.y * m[3]);
  } else {
    double sx = 0.0, sxl = 0.0, sy = 0.0, syl = 0.0;
    for (int c = 0; c < G.n_cam; ++c) {
      sx += M[c * kMom];
      sxl += L[c] * M[c * kMom];
      sy += M[c * kMom + 3];
      syl += L[c] * M[c * kMom + 3];
    }
    const int r = t >> 2;
    g = t < 16 ? f.x * (r == 0 ? sx : r == 1 ? sy : r == 2 ? sxl : syl)
               : 2.0 * (f.x * sx + f.xl * sxl + f.y * sy + f.yl * syl);
  }
  return g;
}

__device__ __forceinline__ void fit_epilogue(const tg_stem_geometry& G, const double* __restrict__ P,
                                             const ScanPos& p, const double (&M)[TG_STEM_MAX_CAM][kMom], int64_t s,
                                             int64_t S, double* __restrict__ partials) {
  const int np = 18 + G.n_cam + 1;
  const int t = threadIdx.x;
  if (t < np) partials[s * np + t] = fit_value(G, P, fit_coef(G, P, p, s, t), M[0], t);
}

// Camera-length constants of the residual r = th a + b - t as double-float
// splits: r = (fma(th, a_hi, -t) + b_hi) + fma(th, a_lo, b_lo) is exact to
// about one ulp of r itself (fma(th, a_hi, -t) rounds once), not to one ulp
// of the ~1e-4 m detector coordinate.
struct CamConst {
  float a_hi, a_lo, bx_hi, bx_lo, by_hi, by_lo;
};

__device__ __forceinline__ CamConst cam_const(const tg_stem_geometry& G, const double* __restrict__ P,
                                              const ScanPos& p, int c) {
  const double L = P[18 + c];
  double bx, by;
  offsets_at(G, P, p, L, bx, by);
  const double ad = G.defocus + L;
  CamConst k;
  k.a_hi = (float)ad;
  k.a_lo = (float)(ad - (double)k.a_hi);
  k.bx_hi = (float)bx;
  k.bx_lo = (float)(bx - (double)k.bx_hi);
  k.by_hi = (float)by;
  k.by_lo = (float)(by - (double)k.by_hi);
  return k;
}

// Adds the residual moments of one tile's first N pairs a lane to m[7] (per
// lane, FP32).
template <int N>
__device__ __forceinline__ void accumulate_tile(const tg_stem_geometry& G, const float* __restrict__ th,
                                                const CamConst& K, const f4 (&cur)[N], int64_t tile, int64_t npair,
                                                float (&m)[kMom]) {
  const int half = G.n_side >> 1, drow = kThreads / half, dcol = kThreads % half;
  // ray pair q = (row iy, columns 2*hc, 2*hc+1); stepped without division
  const int64_t q0 = tile * kTile + threadIdx.x;
  int iy = (int)(q0 / half), hc = (int)(q0 % half);
  if (dcol == 0 && (tile + 1) * kTile <= npair) {
    // full tile and a column count that divides the workgroup: this lane's
    // two columns are fixed, rows advance by drow per pair
    const float tx0 = th[2 * hc], tx1 = th[2 * hc + 1];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const f4 g = cur[k];
      const float ty = th[iy + k * drow];
      const float rx0 = (fmaf(tx0, K.a_hi, -g.x) + K.bx_hi) + fmaf(tx0, K.a_lo, K.bx_lo);
      const float ry0 = (fmaf(ty, K.a_hi, -g.y) + K.by_hi) + fmaf(ty, K.a_lo, K.by_lo);
      const float rx1 = (fmaf(tx1, K.a_hi, -g.z) + K.bx_hi) + fmaf(tx1, K.a_lo, K.bx_lo);
      const float ry1 = (fmaf(ty, K.a_hi, -g.w) + K.by_hi) + fmaf(ty, K.a_lo, K.by_lo);
      m[0] += rx0 + rx1;
      m[1] = fmaf(rx0, tx0, fmaf(rx1, tx1, m[1]));
      m[2] = fmaf(rx0 + rx1, ty, m[2]);
      m[3] += ry0 + ry1;
      m[4] = fmaf(ry0, tx0, fmaf(ry1, tx1, m[4]));
      m[5] = fmaf(ry0 + ry1, ty, m[5]);
      m[6] = fmaf(rx0, rx0, fmaf(ry0, ry0, fmaf(rx1, rx1, fmaf(ry1, ry1, m[6]))));
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (q0 + (int64_t)k * kThreads < npair) {
      const f4 g = cur[k];
      const float tx0 = th[2 * hc], tx1 = th[2 * hc + 1], ty = th[iy];
      const float rx0 = (fmaf(tx0, K.a_hi, -g.x) + K.bx_hi) + fmaf(tx0, K.a_lo, K.bx_lo);
      const float ry0 = (fmaf(ty, K.a_hi, -g.y) + K.by_hi) + fmaf(ty, K.a_lo, K.by_lo);
      const float rx1 = (fmaf(tx1, K.a_hi, -g.z) + K.bx_hi) + fmaf(tx1, K.a_lo, K.bx_lo);
      const float ry1 = (fmaf(ty, K.a_hi, -g.w) + K.by_hi) + fmaf(ty, K.a_lo, K.by_lo);
      m[0] += rx0 + rx1;
      m[1] = fmaf(rx0, tx0, fmaf(rx1, tx1, m[1]));
      m[2] = fmaf(rx0 + rx1, ty, m[2]);
      m[3] += ry0 + ry1;
      m[4] = fmaf(ry0, tx0, fmaf(ry1, tx1, m[4]));
      m[5] = fmaf(ry0 + ry1, ty, m[5]);
      m[6] = fmaf(rx0, rx0, fmaf(ry0, ry0, fmaf(rx1, rx1, fmaf(ry1, ry1, m[6]))));
    }
    hc += dcol;
    iy += drow;
    if (hc >= half) {
      hc -= half;
      ++iy;
    }
  }
}

// Wavefront sums of m[7] into wm[wave][k] (lane 0 writes).
__device__ __forceinline__ void wave_moments(const float (&m)[kMom], double (&wm)[kWaves][kMom]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < kMom; ++k) {
    const float v = wave_sum(m[k]);
    if (lane == 0) wm[wave][k] = v;
  }
}

__device__ __forceinline__ void fill_slopes(const tg_stem_geometry& G, float* th) {
  for (int k = threadIdx.x; k < G.n_side; k += kThreads) th[k] = slope_of(G, k);
}

// Variant "scan": one workgroup per scan position streams the tiles of every
// camera length, double-buffered across tiles and cameras.  (A persistent
// variant that also prefetched across scan positions needed 140 VGPRs, fell
// to 3 waves per SIMD and was slower.)
__global__ __launch_bounds__(kThreads) void stem_fit_kernel(const tg_stem_geometry G, const double* __restrict__ P,
                                                            const float* __restrict__ T,
                                                            double* __restrict__ partials) {
  __shared__ float th[kMaxSide];
  __shared__ double wm[TG_STEM_MAX_CAM][kWaves][kMom];
  __shared__ double M[TG_STEM_MAX_CAM][kMom];
  __shared__ double sp[18 + TG_STEM_MAX_CAM];  // the parameters, read by the set-up and the epilogue
  const int64_t S = (int64_t)G.scan_h * G.scan_w;
  const int64_t J = (int64_t)G.n_side * G.n_side;
  fill_slopes(G, th);
  if (threadIdx.x < 18 + G.n_cam) sp[threadIdx.x] = P[threadIdx.x];
  __syncthreads();
  const int64_t npair = J >> 1;  // two rays per float4 of targets (n_side even)
  const int64_t ntile = (npair + kTile - 1) / kTile;
  const int64_t nit = (int64_t)G.n_cam * ntile;
  const f4* __restrict__ T4 = (const f4*)T;
  f4 cur[kPerLane], nxt[kPerLane];
  const int64_t s = blockIdx.x;
  load_tile(T4, S, s, npair, ntile, 0, cur);
  const ScanPos p = scan_position(G, sp, s);
  CamConst K = {};
  float m[kMom];
  for (int64_t it = 0; it < nit; ++it) {
    if (it + 1 < nit) load_tile(T4, S, s, npair, ntile, it + 1, nxt);
    const int c = (int)(it / ntile);
    const int64_t tile = it - (int64_t)c * ntile;
    if (tile == 0) {
      K = cam_const(G, sp, p, c);
#pragma unroll
      for (int k = 0; k < kMom; ++k) m[k] = 0.f;
    }
    accumulate_tile(G, th, K, cur, tile, npair, m);
    if (tile == ntile - 1) wave_moments(m, wm[c]);
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) cur[k] = nxt[k];
  }
  __syncthreads();
  if (threadIdx.x < G.n_cam * kMom) {
    const int c = threadIdx.x / kMom, k = threadIdx.x % kMom;
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) acc += wm[c][w][k];
    M[c][k] = acc;
  }
  __syncthreads();
  fit_epilogue(G, sp, p, M, s, S, partials);
}

// Variant "scan" where one camera's rays are at most four pairs a lane (N): the
// instructions of the set-up and the sums then bound it, not the targets, so
// one wavefront sets the position up for all (a lane a camera, the
// coefficients of the terms beside it), no more loads are issued than the rays
// need, and the same wavefront makes the terms.  Whole fits, stem_fit_kernel /
// this one: 64x64 positions, 16^2 rays, 1 camera 30.5 / 22.4 us; 30^2, 3
// cameras 57.9 / 42.1; 32^2, 8 cameras 119.5 / 89.8; 45x50, 44^2, 8 cameras
// 82.8 / 61.9.  With eight pairs a lane its registers cost more than the set-up:
// 46^2, 3 cameras 62.3 / 71.9.
template <int N>
__global__ __launch_bounds__(kThreads) void stem_fit_small_kernel(const tg_stem_geometry G,
                                                                  const double* __restrict__ P,
                                                                  const float* __restrict__ T,
                                                                  double* __restrict__ partials) {
  __shared__ float th[kMaxSide];
  __shared__ double wm[TG_STEM_MAX_CAM][kWaves][kMom];
  __shared__ double M[TG_STEM_MAX_CAM][kMom];
  __shared__ CamConst sk[TG_STEM_MAX_CAM];
  const int64_t S = (int64_t)G.scan_h * G.scan_w, s = blockIdx.x;
  const int64_t npair = ((int64_t)G.n_side * G.n_side) >> 1;
  const f4* __restrict__ T4 = (const f4*)T;
  f4 cur[N], nxt[N];
  load_tile(T4, S, s, npair, 1, 0, cur);
  FitCoef f = {};
  if (threadIdx.x < 64) {
    const ScanPos p = scan_position(G, P, s);
    if (threadIdx.x < G.n_cam) sk[threadIdx.x] = cam_const(G, P, p, threadIdx.x);
    f = fit_coef(G, P, p, s, threadIdx.x);
  } else {
    for (int k = (int)threadIdx.x - 64; k < G.n_side; k += kThreads - 64) th[k] = slope_of(G, k);
  }
  __syncthreads();
  for (int c = 0; c < G.n_cam; ++c) {
    if (c + 1 < G.n_cam) load_tile(T4, S, s, npair, 1, c + 1, nxt);
    float m[kMom];
#pragma unroll
    for (int k = 0; k < kMom; ++k) m[k] = 0.f;
    accumulate_tile(G, th, sk[c], cur, 0, npair, m);
    wave_moments(m, wm[c]);
#pragma unroll
    for (int k = 0; k < N; ++k) cur[k] = nxt[k];
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;  // one wavefront from here
  for (int i = threadIdx.x; i < G.n_cam * kMom; i += 64) {
    const int c = i / kMom, k = i % kMom;
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) acc += wm[c][w][k];
    M[c][k] = acc;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int np = 18 + G.n_cam + 1;
  if (threadIdx.x < np) partials[s * np + threadIdx.x] = fit_value(G, P, f, M[0], threadIdx.x);
}

// Variant "camera": one workgroup per (scan position, camera length) --
// n_cam times more, shorter work items, for scans too small to fill the
// device one workgroup per position.  Each pays the per-workgroup set-up
// (slopes, scan position, camera constants) without a second tile to
// overlap it with, so on large scans it is slower than "scan".  Writes the
// camera's FP64 moments; stem_fit_sum_kernel (or stem_fit_epilogue) makes the
// terms of them with the same arithmetic as the scan variant.
// Bound: latency.  So the targets' loads come first, N of them a lane (as many
// as the rays need where they are one tile), and one wavefront makes the
// constants while the others fill the slopes.  With the terms and sums in one
// launch, whole fits before / now: 13x21 positions, 46^2 rays, 3 cameras 13.7 /
// 11.7 us; 7x13, 30^2, 3 12.4 / 9.4; 31x33, 30^2, 8 43.5 / 28.9; 5x5, 16^2, 1 11.5
// / 8.4.
template <int N>
__global__ __launch_bounds__(kThreads) void stem_fit_cam_kernel(const tg_stem_geometry G,
                                                                const double* __restrict__ P,
                                                                const float* __restrict__ T,
                                                                double* __restrict__ cam_mom) {
  __shared__ float th[kMaxSide];
  __shared__ double wm[kWaves][kMom];
  __shared__ CamConst sk;
  const int64_t S = (int64_t)G.scan_h * G.scan_w;
  const int64_t J = (int64_t)G.n_side * G.n_side;
  const int64_t npair = J >> 1;
  const int64_t ntile = N < kPerLane ? 1 : (npair + kTile - 1) / kTile;
  const f4* __restrict__ T4 = (const f4*)T;
  const int64_t s = blockIdx.x;
  const int c = blockIdx.y;
  f4 cur[N], nxt[N];
  load_tile(T4, S, s, npair, ntile, (int64_t)c * ntile, cur);
  if (threadIdx.x < 64) {
    const CamConst k = cam_const(G, P, scan_position(G, P, s), c);
    if (threadIdx.x == 0) sk = k;
  } else {
    for (int k = (int)threadIdx.x - 64; k < G.n_side; k += kThreads - 64) th[k] = slope_of(G, k);
  }
  __syncthreads();
  const CamConst K = sk;
  float m[kMom];
#pragma unroll
  for (int k = 0; k < kMom; ++k) m[k] = 0.f;
  for (int64_t tile = 0; tile < ntile; ++tile) {
    if (tile + 1 < ntile) load_tile(T4, S, s, npair, ntile, (int64_t)c * ntile + tile + 1, nxt);
    accumulate_tile(G, th, K, cur, tile, npair, m);
#pragma unroll
    for (int k = 0; k < N; ++k) cur[k] = nxt[k];
  }
  wave_moments(m, wm);
  __syncthreads();
  if (threadIdx.x < kMom) {
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) acc += wm[w][threadIdx.x];
    cam_mom[(s * G.n_cam + c) * kMom + threadIdx.x] = acc;
  }
}

__global__ __launch_bounds__(64) void stem_fit_epilogue(const tg_stem_geometry G, const double* __restrict__ P,
                                                        const double* __restrict__ cam_mom,
                                                        double* __restrict__ partials) {
  __shared__ double M[TG_STEM_MAX_CAM][kMom];
  const int64_t S = (int64_t)G.scan_h * G.scan_w;
  const int64_t s = blockIdx.x;
  for (int i = threadIdx.x; i < G.n_cam * kMom; i += 64) M[i / kMom][i % kMom] = cam_mom[s * G.n_cam * kMom + i];
  __syncthreads();
  const ScanPos p = scan_position(G, P, s);
  fit_epilogue(G, P, p, M, s, S, partials);
}

// Fixed-order FP64 column sums of the [rows, cols] workspace (one block per
// column, strided reads of the L2-resident terms, wavefront shuffles then
// one LDS step).
constexpr int kSumThreads = 1024;

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The sum of a block's values, wavefronts in order, into *out.
__device__ __forceinline__ void block_sum_store(double acc, double* __restrict__ out) {
  __shared__ double red[kSumThreads / 64];
  acc = wave_sum_f64(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x < 64) {
    double v = threadIdx.x < kSumThreads / 64 ? red[threadIdx.x] : 0.0;
    v = wave_sum_f64(v);
    if (threadIdx.x == 0) *out = v;
  }
}

__global__ __launch_bounds__(kSumThreads) void row_sum_kernel(const double* __restrict__ partials, int64_t rows,
                                                              int64_t cols, double* __restrict__ out) {
  const double* __restrict__ src = partials + blockIdx.x;  // column blockIdx.x of [rows, cols]
  double acc = 0.0;
  int64_t r = threadIdx.x;
  // four loads in flight per step (a plain loop waited for each), summed in
  // the same order as one at a time
  for (; r + 3 * kSumThreads < rows; r += 4 * kSumThreads) {
    const double a = src[r * cols], b = src[(r + kSumThreads) * cols];
    const double c = src[(r + 2 * kSumThreads) * cols], d = src[(r + 3 * kSumThreads) * cols];
    acc += a;
    acc += b;
    acc += c;
    acc += d;
  }
  for (; r < rows; r += kSumThreads) acc += src[r * cols];
  block_sum_store(acc, out + blockIdx.x);
}

// Variant "camera", the terms and their sums in one launch: block t makes entry
// t of every scan position from the cameras' moments, as stem_fit_epilogue
// does, keeps them, and sums them in row_sum_kernel's order.  For up to 2,048
// cameras' moments: each block reads all of them, a position a lane, which for
// more takes longer than the launch that it saves (whole fits in two launches /
// in three: 600 positions, 3 cameras 17.7 / 19.1 us; 992, 2 13.8 / 16.0; 440, 8
// 27.8 / 27.1; 992, 8 52.5 / 47.5).
__global__ __launch_bounds__(kSumThreads) void stem_fit_sum_kernel(const tg_stem_geometry G,
                                                                   const double* __restrict__ P,
                                                                   const double* __restrict__ cam_mom,
                                                                   double* __restrict__ partials,
                                                                   double* __restrict__ out) {
  const int64_t S = (int64_t)G.scan_h * G.scan_w;
  const int t = blockIdx.x, np = gridDim.x;
  double acc = 0.0;
  for (int64_t s = threadIdx.x; s < S; s += kSumThreads) {
    const double v = fit_value(G, P, fit_coef(G, P, scan_position(G, P, s), s, t), cam_mom + s * G.n_cam * kMom, t);
    partials[s * np + t] = v;
    acc += v;
  }
  block_sum_store(acc, out + t);
}

int validate(const tg_stem_geometry* g, const double* params) {
  TG_REQUIRE(g != nullptr && params != nullptr, "stem: NULL geometry or params");
  TG_REQUIRE(g->scan_h > 0 && g->scan_w > 0 && (int64_t)g->scan_h * g->scan_w <= 65535,
             "stem: scan grid %dx%d must have 1..65535 positions", g->scan_h, g->scan_w);
  TG_REQUIRE(g->n_side >= 2 && g->n_side <= kMaxSide && (g->n_side % 2) == 0,
             "stem: n_side %d must be even and in [2, %d]", g->n_side, kMaxSide);
  TG_REQUIRE(g->n_cam >= 1 && g->n_cam <= TG_STEM_MAX_CAM, "stem: n_cam %d out of range", g->n_cam);
  return TG_OK;
}

}  // namespace

extern "C" int32_t tg_stem_dataset_max_width(void) { return kBandFloats; }

extern "C" int tg_stem_forward(const tg_stem_geometry* g, const double* params, const float* image, float* coords,
                               float* values, float* image4d, void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  TG_REQUIRE(image != nullptr || (values == nullptr && image4d == nullptr),
             "tg_stem_forward: sample image required for values / image4d");
  TG_REQUIRE(image == nullptr || (g->img_h > 0 && g->img_w > 0), "tg_stem_forward: bad sample image shape");
  TG_REQUIRE(image4d == nullptr || (g->det_h > 0 && g->det_w > 0), "tg_stem_forward: bad detector shape");
  if (coords == nullptr && values == nullptr && image4d == nullptr) return TG_OK;
  const int64_t J = (int64_t)g->n_side * g->n_side;
  dim3 grid((unsigned)tg::cdiv(J, (int64_t)kThreads * kFwdRays), (unsigned)((int64_t)g->scan_h * g->scan_w));
  hipLaunchKernelGGL(stem_forward_kernel, grid, dim3(kThreads), 0, (hipStream_t)stream, *g, params, image, coords,
                     values, image4d);
  TG_LAUNCH_CHECK("stem_forward_kernel launch");
  return TG_OK;
}

extern "C" int tg_stem_dataset(const tg_stem_geometry* g, const double* params, const float* image, float* image4d,
                               void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  TG_REQUIRE(image != nullptr && image4d != nullptr, "tg_stem_dataset: NULL sample image or dataset");
  TG_REQUIRE(g->img_h > 0 && g->img_w > 0, "tg_stem_dataset: bad sample image shape");
  TG_REQUIRE(g->det_h > 0 && g->det_w > 0, "tg_stem_dataset: bad detector shape");
  TG_REQUIRE(g->det_w <= tg_stem_dataset_max_width(), "tg_stem_dataset: detector rows of %d pixels exceed %d", g->det_w,
             tg_stem_dataset_max_width());
  // As many workgroups a position as run at a time (five a CU): a few positions
  // are shared by several, and with many the set-up is paid once for all bands.
  const int64_t S = (int64_t)g->scan_h * g->scan_w, W = g->det_w;
  const int64_t share = std::min<int64_t>(16, std::max<int64_t>(1, 5LL * tg::cu_count() / S));
  // Even bands of whole rows, no more than LDS holds and as many for each that
  // shares them; a multiple of four rows keeps every band of an aligned image
  // aligned.
  const int64_t most = std::max<int64_t>(1, kBandFloats / W);
  const int64_t want = tg::cdiv(tg::cdiv(g->det_h, most), share) * share;
  int64_t rows = tg::cdiv(g->det_h, want);
  rows = std::min((rows + 3) / 4 * 4, most > 4 ? most / 4 * 4 : most);
  rows = std::min<int64_t>(rows, g->det_h);
  const int64_t bands = tg::cdiv(g->det_h, rows), each = tg::cdiv(bands, std::min(bands, share));
  const dim3 grid((unsigned)tg::cdiv(bands, each), (unsigned)S);
  // As much LDS as the detector and the rays take: the workgroups a CU holds at a
  // time hide the set-up's latency, which is most of a small detector's time.
  // Of workgroups with many bands no more than make the rounds even: 64x64
  // positions of 256x256 pixels 193 us four a CU, 200 five a CU.
  const int64_t own = 4608, all = 160 * 1024;  // the kernel's other LDS, a CU's
  int64_t lds = (4 * (int64_t)band_quads((int)(rows * W)) + g->n_side) * (int64_t)sizeof(float);
  const int64_t held = std::min<int64_t>(8, all / (lds + own)), cus = tg::cu_count(), count = (int64_t)grid.x * S;
  const int64_t even = std::max<int64_t>(3, tg::cdiv(count, tg::cdiv(count, held * cus) * cus));
  if (each >= 6 && even < held) lds = std::max(lds, all / (even + 1) - own + 1280);
  hipLaunchKernelGGL(stem_dataset_kernel, grid, dim3(kThreads), (size_t)lds, (hipStream_t)stream, *g, params, image,
                     (int)rows, (int)each, image4d);
  TG_LAUNCH_CHECK("stem_dataset_kernel launch");
  return TG_OK;
}

extern "C" int tg_stem_backproject(const tg_stem_geometry* g, const double* params, const float* data4d,
                                   int32_t cam, double* image, double* weight, void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  TG_REQUIRE(data4d != nullptr && image != nullptr, "tg_stem_backproject: NULL data or image");
  TG_REQUIRE(cam >= 0 && cam < g->n_cam, "tg_stem_backproject: camera %d out of range", cam);
  TG_REQUIRE(g->img_h > 0 && g->img_w > 0 && g->det_h > 0 && g->det_w > 0,
             "tg_stem_backproject: bad sample or detector shape");
  TG_REQUIRE((int64_t)g->det_h * g->det_w <= (int64_t)1 << 30,
             "tg_stem_backproject: detector of %lld pixels exceeds 2^30", (long long)g->det_h * g->det_w);
  const int64_t ntile = tg::cdiv((int64_t)g->n_side, (int64_t)kBpRayTile);
  dim3 grid((unsigned)(ntile * ntile), (unsigned)((int64_t)g->scan_h * g->scan_w));
  // grids whose axes lie along the slopes (no rotation between them)
  const bool separable = g->img_m[1] == 0.0 && g->img_m[3] == 0.0 && g->det_m[1] == 0.0 && g->det_m[3] == 0.0 &&
                         std::isfinite(g->defocus);
  auto* kernel = weight != nullptr ? (separable ? stem_backproject_kernel<true, true> : stem_backproject_kernel<true, false>)
                                   : (separable ? stem_backproject_kernel<false, true> : stem_backproject_kernel<false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, (hipStream_t)stream, *g, params, data4d, cam, image, weight);
  TG_LAUNCH_CHECK("stem_backproject_kernel launch");
  return TG_OK;
}

extern "C" int64_t tg_stem_fit_workspace(const tg_stem_geometry* g) {
  if (g == nullptr || g->scan_h <= 0 || g->scan_w <= 0 || g->n_cam < 1 || g->n_cam > TG_STEM_MAX_CAM) return 0;
  const int64_t S = (int64_t)g->scan_h * g->scan_w;
  return (int64_t)sizeof(double) * S * ((18 + g->n_cam + 1) + (int64_t)g->n_cam * kMom);
}

namespace {

// The first launch of a fit: the per-scan-position terms [S, np] at the head of
// the workspace (variant "scan"), or the cameras' moments behind them.
int fit_first(const tg_stem_geometry* g, const double* params, const float* targets, double* workspace,
              hipStream_t stream, int32_t& variant) {
  TG_REQUIRE(targets != nullptr && workspace != nullptr, "tg_stem_fit: NULL buffer");
  TG_REQUIRE(((uintptr_t)targets & 15) == 0, "tg_stem_fit: targets must be 16-byte aligned");
  const int64_t S = (int64_t)g->scan_h * g->scan_w;
  const int np = 18 + g->n_cam + 1;
  // launch variant: the autotuner's choice, else one workgroup per scan
  // position when that gives every CU several workgroups, and one per (scan
  // position, camera length) for small scans
  const int64_t key[4] = {S, (int64_t)g->n_side * g->n_side, g->n_cam, 0};
  variant = S >= 4LL * tg::cu_count() ? TG_STEM_FIT_SCAN : TG_STEM_FIT_CAMERA;
  int32_t tuned = 0;
  if (tg::tune_lookup(TG_TUNE_STEM_FIT, key, tuned)) variant = tuned;
  const int64_t npair = ((int64_t)g->n_side * g->n_side) >> 1;
  if (variant == TG_STEM_FIT_SCAN) {
    auto* kernel = npair <= 2 * kThreads   ? stem_fit_small_kernel<2>
                   : npair <= 4 * kThreads ? stem_fit_small_kernel<4>
                                           : stem_fit_kernel;
    hipLaunchKernelGGL(kernel, dim3((unsigned)S), dim3(kThreads), 0, stream, *g, params, targets, workspace);
    TG_LAUNCH_CHECK("stem_fit_kernel launch");
  } else {
    auto* kernel = npair <= 2 * kThreads   ? stem_fit_cam_kernel<2>
                   : npair <= 4 * kThreads ? stem_fit_cam_kernel<4>
                                           : stem_fit_cam_kernel<kPerLane>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)S, (unsigned)g->n_cam), dim3(kThreads), 0, stream, *g, params, targets,
                       workspace + (int64_t)np * S);
    TG_LAUNCH_CHECK("stem_fit_cam_kernel launch");
  }
  return TG_OK;
}

// tg_stem_fit with checked arguments
int fit_run(const tg_stem_geometry* g, const double* params, const float* targets, double* workspace, double* out,
            hipStream_t stream) {
  int32_t variant = 0;
  const int st = fit_first(g, params, targets, workspace, stream, variant);
  if (st != TG_OK) return st;
  const int64_t S = (int64_t)g->scan_h * g->scan_w;
  const int np = 18 + g->n_cam + 1;
  double* cam_mom = workspace + (int64_t)np * S;  // [S, n_cam, 7]
  if (variant != TG_STEM_FIT_SCAN && S * g->n_cam <= 2 * kSumThreads && S <= kSumThreads) {
    hipLaunchKernelGGL(stem_fit_sum_kernel, dim3((unsigned)np), dim3(kSumThreads), 0, stream, *g, params, cam_mom,
                       workspace, out);
    TG_LAUNCH_CHECK("stem_fit_sum_kernel launch");
    return TG_OK;
  }
  if (variant != TG_STEM_FIT_SCAN) {
    hipLaunchKernelGGL(stem_fit_epilogue, dim3((unsigned)S), dim3(64), 0, stream, *g, params, cam_mom, workspace);
    TG_LAUNCH_CHECK("stem_fit_epilogue launch");
  }
  hipLaunchKernelGGL(row_sum_kernel, dim3((unsigned)np), dim3(kSumThreads), 0, stream, workspace, S, (int64_t)np, out);
  TG_LAUNCH_CHECK("row_sum_kernel launch");
  return TG_OK;
}

}  // namespace

extern "C" int tg_stem_fit_terms(const tg_stem_geometry* g, const double* params, const float* targets,
                                 double* workspace, void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  int32_t variant = 0;
  st = fit_first(g, params, targets, workspace, (hipStream_t)stream, variant);
  if (st != TG_OK || variant == TG_STEM_FIT_SCAN) return st;
  const int64_t S = (int64_t)g->scan_h * g->scan_w;
  hipLaunchKernelGGL(stem_fit_epilogue, dim3((unsigned)S), dim3(64), 0, (hipStream_t)stream, *g, params,
                     workspace + (18 + g->n_cam + 1) * S, workspace);
  TG_LAUNCH_CHECK("stem_fit_epilogue launch");
  return TG_OK;
}

extern "C" int tg_stem_fit(const tg_stem_geometry* g, const double* params, const float* targets, double* workspace,
                           double* out, void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  TG_REQUIRE(out != nullptr, "tg_stem_fit: NULL buffer");
  return fit_run(g, params, targets, workspace, out, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// tg_stem_fit_noalloc: tg_stem_fit with its workspace in a device array of
// this code object instead of a caller buffer, for callers that cannot
// allocate (HIP graph capture, allocation-free serving loops).  Each GPU holds
// its own copy of the array until the process ends.  Host code never passes
// the array's name to a kernel (on the host it is only a stand-in for the
// symbol): the device address comes from hipGetSymbolAddress, once per
// device, with that device current.
// ---------------------------------------------------------------------------

namespace {

constexpr int64_t kNoAllocScratchBytes = 8LL << 20;  // 8 MiB per GPU
static __device__ __align__(256) double scratch[kNoAllocScratchBytes / sizeof(double)];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kScratchDevices] = {};

// Device address of this device's scratch (the current device, which must be
// the stream's device).
int scratch_address(hipStream_t stream, double** out) {
  int dev = -1;
  TG_HIP_CHECK(hipGetDevice(&dev));
  TG_REQUIRE(dev >= 0 && dev < kScratchDevices, "tg_stem_fit_noalloc: device %d out of range", dev);
  if (stream != nullptr) {
    int sdev = -1;
    TG_HIP_CHECK(hipStreamGetDevice(stream, &sdev));
    TG_REQUIRE(sdev == dev, "tg_stem_fit_noalloc: the stream belongs to device %d, the current device is %d", sdev,
               dev);
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    TG_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    TG_REQUIRE(p != nullptr, "tg_stem_fit_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return TG_OK;
}

}  // namespace

extern "C" int64_t tg_stem_fit_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int tg_stem_fit_noalloc(const tg_stem_geometry* g, const double* params, const float* targets,
                                   double* out, void* stream) {
  tg::clear_error();
  int st = validate(g, params);
  if (st != TG_OK) return st;
  TG_REQUIRE(out != nullptr, "tg_stem_fit_noalloc: NULL buffer");
  const int64_t need = tg_stem_fit_workspace(g);
  TG_REQUIRE(need > 0 && need <= kNoAllocScratchBytes,
             "tg_stem_fit_noalloc: this geometry needs %lld bytes of scratch, more than the %lld available "
             "(use tg_stem_fit with a caller workspace)",
             (long long)need, (long long)kNoAllocScratchBytes);
  double* ws = nullptr;
  st = scratch_address((hipStream_t)stream, &ws);
  if (st != TG_OK) return st;
  // every word of the workspace a launch reads is written earlier in the same
  // call (per-position rows, per-camera moments): nothing needs clearing
  return fit_run(g, params, targets, ws, out, (hipStream_t)stream);
}
