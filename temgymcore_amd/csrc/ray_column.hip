// Ray branch, columns of standard elements: drift, lens, deflector, rotator,
// scanner / descanner offsets and biprism, applied in turn to a bundle held as
// contiguous SoA arrays, optionally followed (in the same pass) by detector
// binning.
//
// Replaces the same reference code as ray_program.hip (run.py:47-116,
// propagator.py:51-72, components.py) for the models that consist of these
// elements; the host's matcher recognises them in the traced instructions, so
// the arithmetic here is that program's, operation by operation (built with
// -ffp-contract=off: one rounding each, bit-identical results).
//
// Bound: HBM, 36 B (f32) or 72 B (f64) a ray.  The register-program interpreter
// spends ~230 cycles of a wavefront on every instruction (fetch, dispatch,
// indexed register moves) and stores a long model's values between two
// programs; here the state lives in named registers and one uniform dispatch
// covers an element and the drift before it, ten operations or more.  Measured
// without binning (interpreter -> column): 4,194,301 f64 rays through 2 / 5 /
// 10 elements 81 / 176 / 400 -> 53 / 55 / 74 us (302 MB: 5.7 TB/s at 2; the
// lenses' divisions show at 10), f32 38 / 76 / 171 -> 25 / 27 / 45 us; 1,000
// rays 9.4 -> 3.4 us.
//
// Layout: a lane owns the 16 bytes of consecutive rays that one load moves
// (4 f32, 2 f64), where every array is 16-byte aligned; the host's other arrays
// take the form with one ray a lane.
#include <algorithm>

#include "ray_common.hpp"

namespace {

using namespace tgr;

static_assert(sizeof(tg_column) + sizeof(tg_bin_spec) <= 4096, "ray column exceeds the kernel-argument limit");

template <typename T, int VEC>
struct Pack {
  typedef T type __attribute__((ext_vector_type(VEC)));
};
template <typename T>
struct Pack<T, 1> {
  typedef T type;
};

template <typename T, int VEC>
__device__ __forceinline__ void load_rays(const void* p, int64_t i, int64_t n, T (&v)[VEC]) {
  const T* __restrict__ src = (const T*)p + i;
  if constexpr (VEC == 1) {
    v[0] = *src;
  } else if (i + VEC <= n) {
    const auto q = *(const typename Pack<T, VEC>::type*)src;
#pragma unroll
    for (int k = 0; k < VEC; ++k) v[k] = q[k];
  } else {
#pragma unroll
    for (int k = 0; k < VEC; ++k) v[k] = i + k < n ? src[k] : T(0);
  }
}

template <typename T, int VEC>
__device__ __forceinline__ void store_rays(void* p, int64_t i, int64_t n, const T (&v)[VEC]) {
  if (p == nullptr) return;
  T* __restrict__ dst = (T*)p + i;
  if constexpr (VEC == 1) {
    *dst = v[0];
  } else if (i + VEC <= n) {
    typename Pack<T, VEC>::type q;
#pragma unroll
    for (int k = 0; k < VEC; ++k) q[k] = v[k];
    *(typename Pack<T, VEC>::type*)dst = q;
  } else {
#pragma unroll
    for (int k = 0; k < VEC; ++k)
      if (i + k < n) dst[k] = v[k];
  }
}

// ---------------------------------------------------------------------------
// Detectors that no workgroup's LDS holds.  4.2M scattered atomics on a
// 1024x1024 image take 120-150 us however the rays fall (350 us on 512x512:
// fewer lines, more of the rays on each), so many rays are counted in two
// passes instead: the column stores each ray's pixel index, and
// bin_bands_kernel counts slices of them into bands of the image in LDS.  The
// flush then costs an atomic a cache line the slice touched, not one a ray.
// 4,194,301 f64 rays through 10 elements onto 1024x1024: 78 us with the
// indices + 20 us of counting (74 + 120 us with memory atomics); 2 elements
// onto 512x512: 347 -> 80 us.
// ---------------------------------------------------------------------------
constexpr int kBinChunk = 2048;   // rays a workgroup of the column covers; its lowest and highest index are kept
constexpr int kSliceChunks = 31;  // chunks a slice: at most kMaxRaysPerGroup rays, 16-bit counters
constexpr int64_t kBandBins = kLdsBins - 64;  // a band, beside the kernel's own few bytes of LDS
static_assert(kBinChunk * kSliceChunks <= kMaxRaysPerGroup, "a slice's counters may not carry");

struct BinWorkspace {
  int2* range;     // [chunks]: lowest and highest pixel index (highest -1: none on the detector)
  int32_t* index;  // [n]: pixel index, -1 off the detector
};

__host__ __device__ inline BinWorkspace bin_workspace(void* ws, int64_t n) {
  const int64_t chunks = (n + kBinChunk - 1) / kBinChunk;
  BinWorkspace w;
  w.range = (int2*)ws;
  w.index = (int32_t*)((char*)ws + (chunks * (int64_t)sizeof(int2) + 15) / 16 * 16);
  return w;
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return v;
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// Workgroup (blockIdx.x, blockIdx.y) counts slice blockIdx.x into every
// gridDim.y-th of the bands its indices reach.
__global__ __launch_bounds__(1024) void bin_bands_kernel(const tg_bin_spec B, void* ws, int64_t n, int band_bins) {
  extern __shared__ __align__(16) int32_t hist[];
  __shared__ int sh_lo, sh_hi;
  const BinWorkspace w = bin_workspace(ws, n);
  const int64_t chunks = (n + kBinChunk - 1) / kBinChunk, c0 = (int64_t)blockIdx.x * kSliceChunks;
  if (threadIdx.x < 64) {
    const int64_t c = c0 + threadIdx.x;
    const bool in = threadIdx.x < kSliceChunks && c < chunks;
    const int2 r = in ? w.range[c] : make_int2(0x7fffffff, -1);
    const int lo = wave_min(r.x), hi = wave_max(r.y);
    if (threadIdx.x == 0) sh_lo = lo, sh_hi = hi;
  }
  __syncthreads();
  if (sh_hi < 0) return;
  const int64_t r0 = c0 * kBinChunk;
  const int64_t r1 = r0 + kSliceChunks * kBinChunk < n ? r0 + kSliceChunks * kBinChunk : n;
  const int64_t bins = B.height * B.width;
  const int last = sh_hi / band_bins;
  for (int band = sh_lo / band_bins + (int)blockIdx.y; band <= last; band += (int)gridDim.y) {
    const int64_t b0 = (int64_t)band * band_bins;
    const int nb = (int)(bins - b0 < band_bins ? bins - b0 : band_bins);
    lds_clear<1024>(hist, nb);
    __syncthreads();
    // four loads of four indices in flight (unpredicated: past the end the last four again, masked out)
    for (int64_t r = r0 + 4 * threadIdx.x; r < r1; r += 4 * 4096) {
      int4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t q = r + u * 4096;
        v[u] = *(const int4*)(w.index + (q < r1 ? q : r));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t q = r + u * 4096;
        const int e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const unsigned p = (unsigned)(e[k] - (int)b0);
          if (q + k < r1 && e[k] >= 0 && p < (unsigned)nb) lds_deposit(hist, p);
        }
      }
    }
    __syncthreads();
    lds_flush<1024>(B, hist, b0, nb);
    __syncthreads();
  }
}

// BIN: 0 = no binning, 1 = LDS-privatised integer histogram, 2 = global
// atomics, 3 = pixel indices into the workspace (then bin_bands_kernel)
template <typename T, int VEC, int BIN, int NT>
__global__ __launch_bounds__(NT) void ray_column_kernel(const tg_column C, const tg_bin_spec B, void* ws) {
  extern __shared__ __align__(16) int32_t hist[];
  // BIN 3: a workgroup covers one chunk of consecutive rays
  const int64_t n = BIN == 3 ? ((int64_t)(blockIdx.x + 1) * kBinChunk < C.n ? (int64_t)(blockIdx.x + 1) * kBinChunk : C.n)
                             : C.n;
  int lo = 0x7fffffff, hi = -1;
  if constexpr (BIN == 1) {
    lds_clear<NT>(hist, (int)(B.height * B.width));
    __syncthreads();
  }
  constexpr int64_t kChunk = (int64_t)NT * VEC;
  const int64_t begin = (int64_t)blockIdx.x * (BIN == 3 ? (int64_t)kBinChunk : kChunk);
  const int64_t stride = BIN == 3 ? kChunk : (int64_t)gridDim.x * kChunk;
  for (int64_t base = begin; base < n; base += stride) {
    const int64_t i = base + (int64_t)threadIdx.x * VEC;
    if (i >= n) break;
    T x[VEC], y[VEC], dx[VEC], dy[VEC], pl[VEC];
    load_rays<T, VEC>(C.in[0], i, n, x);
    load_rays<T, VEC>(C.in[1], i, n, y);
    load_rays<T, VEC>(C.in[2], i, n, dx);
    load_rays<T, VEC>(C.in[3], i, n, dy);
    if (C.in[4] != nullptr) {
      load_rays<T, VEC>(C.in[4], i, n, pl);
    } else {
#pragma unroll
      for (int k = 0; k < VEC; ++k) pl[k] = (T)C.pathlength;
    }
    for (int s = 0; s < C.n_step; ++s) {
      const tg_step& S = C.step[s];
      const int flags = S.flags;
      if (flags & TG_STEP_DRIFT) {
        const T d = (T)S.d;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          x[k] = x[k] + dx[k] * d;
          y[k] = y[k] + dy[k] * d;
        }
        if (flags & TG_STEP_DRIFT_PATH) {
#pragma unroll
          for (int k = 0; k < VEC; ++k) pl[k] = pl[k] + d;
        }
      }
      const T p0 = (T)S.p[0], p1 = (T)S.p[1];
      switch (S.kind) {
        case TG_STEP_LENS:  // p0 = f, p1 = 2 f
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            dx[k] = (-x[k]) / p0 + dx[k];
            dy[k] = (-y[k]) / p0 + dy[k];
            pl[k] = pl[k] - (x[k] * x[k] + y[k] * y[k]) / p1;
          }
          break;
        case TG_STEP_DEFLECT:  // the pathlength takes the incoming slopes
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            pl[k] = (pl[k] + dx[k] * x[k]) + dy[k] * y[k];
            dx[k] = dx[k] + p0;
            dy[k] = dy[k] + p1;
          }
          break;
        case TG_STEP_ROTATE:  // p0 = cos, p1 = sin
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            const T u = x[k] * p0 - y[k] * p1, v = x[k] * p1 + y[k] * p0;
            const T du = dx[k] * p0 - dy[k] * p1, dv = dx[k] * p1 + dy[k] * p0;
            x[k] = u;
            y[k] = v;
            dx[k] = du;
            dy[k] = dv;
          }
          break;
        case TG_STEP_SHIFT: {
          const T p2 = (T)S.p[2], p3 = (T)S.p[3];
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            x[k] = x[k] + p0;
            y[k] = y[k] + p1;
            dx[k] = dx[k] + p2;
            dy[k] = dy[k] + p3;
          }
          break;
        }
        case TG_STEP_BIPRISM:  // the pathlength takes the incoming slopes
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            pl[k] = (pl[k] + dx[k] * x[k]) + dy[k] * y[k];
            dx[k] = dx[k] + sign_of<T>(x[k]) * p0;
          }
          break;
        default:  // TG_STEP_NONE: the drift alone
          break;
      }
    }
    store_rays<T, VEC>(C.out[0], i, n, x);
    store_rays<T, VEC>(C.out[1], i, n, y);
    store_rays<T, VEC>(C.out[2], i, n, dx);
    store_rays<T, VEC>(C.out[3], i, n, dy);
    store_rays<T, VEC>(C.out[4], i, n, pl);
    if constexpr (BIN == 3) {
      int32_t px[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        px[k] = VEC > 1 && i + k >= n ? -1 : (int32_t)bin_index(B, (double)y[k], (double)x[k]);
        lo = px[k] >= 0 ? min(lo, px[k]) : lo;
        hi = max(hi, px[k]);
      }
      store_rays<int32_t, VEC>(bin_workspace(ws, C.n).index, i, n, px);
    } else if constexpr (BIN != 0) {
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        if (VEC > 1 && i + k >= n) continue;
        const int64_t p = bin_index(B, (double)y[k], (double)x[k]);
        if (p < 0) continue;
        if constexpr (BIN == 1)
          lds_deposit(hist, p);
        else
          global_deposit<T>(B, p, T(1));
      }
    }
  }
  if constexpr (BIN == 1) {
    __syncthreads();
    lds_flush<NT>(B, hist, 0, (int)(B.height * B.width));
  }
  if constexpr (BIN == 3) {
    __shared__ int part[2][NT / 64];
    lo = wave_min(lo);
    hi = wave_max(hi);
    if ((threadIdx.x & 63) == 0) part[0][threadIdx.x >> 6] = lo, part[1][threadIdx.x >> 6] = hi;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 1; k < NT / 64; ++k) {
        lo = min(lo, part[0][k]);
        hi = max(hi, part[1][k]);
      }
      bin_workspace(ws, C.n).range[blockIdx.x] = make_int2(lo, hi);
    }
  }
}

template <typename T, int VEC, int BIN>
int launch(const tg_column& C, const tg_bin_spec& B, void* ws, hipStream_t stream) {
  constexpr int NT = BIN == 1 ? 1024 : 256;
  constexpr int64_t kChunk = (int64_t)NT * VEC;
  static_assert(BIN != 3 || kBinChunk % kChunk == 0, "a chunk is whole passes of the workgroup");
  const int cus = tg::cu_count();
  int64_t grid = tg::cdiv(C.n, BIN == 3 ? (int64_t)kBinChunk : kChunk);
  size_t lds = 0;
  if (BIN != 3) {
    // LDS histograms are cleared and flushed once per workgroup, so that grid
    // stays at one 1024-thread workgroup per CU; a caller (the autotuner) may override
    int64_t cap = BIN == 1 ? 1LL * cus : 32LL * cus;
    int32_t tuned = 0;
    if (B.grid_hint > 0) {
      cap = B.grid_hint;
    } else if (BIN != 0) {
      const int64_t key[4] = {C.n, B.height * B.width, C.dtype, 0};
      if (tg::tune_lookup(TG_TUNE_RAY_GRID, key, tuned) && tuned > 0) cap = tuned;
    }
    if (grid > cap) grid = cap;
  }
  if (BIN == 1) {
    const int64_t min_grid = tg::cdiv(C.n, (kMaxRaysPerGroup / kChunk) * kChunk);
    if (grid < min_grid) grid = min_grid;
    lds = (size_t)lds_words(B.height * B.width) * sizeof(int32_t);
    const int st = allow_lds((const void*)ray_column_kernel<T, VEC, BIN, NT>, lds);
    if (st != TG_OK) return st;
  }
  hipLaunchKernelGGL((ray_column_kernel<T, VEC, BIN, NT>), dim3((unsigned)grid), dim3(NT), lds, stream, C, B, ws);
  TG_LAUNCH_CHECK("ray_column_kernel launch");
  if (BIN == 3) {
    const int64_t bins = B.height * B.width;
    const int band = (int)std::min(bins, kBandBins);
    lds = (size_t)lds_words(band) * sizeof(int32_t);
    const int st = allow_lds((const void*)bin_bands_kernel, lds);
    if (st != TG_OK) return st;
    // one workgroup a CU (its LDS holds one band): the bands of a slice are
    // shared by as many workgroups as that leaves
    const int64_t slices = tg::cdiv(C.n, (int64_t)kBinChunk * kSliceChunks), bands = tg::cdiv(bins, band);
    const int64_t each = std::max<int64_t>(1, std::min<int64_t>(bands, cus / slices));
    hipLaunchKernelGGL(bin_bands_kernel, dim3((unsigned)slices, (unsigned)each), dim3(1024), lds, stream, B, ws, C.n,
                       band);
    TG_LAUNCH_CHECK("bin_bands_kernel launch");
  }
  return TG_OK;
}

template <typename T, int VEC>
int dispatch(const tg_column& C, const tg_bin_spec& B, int bin, void* ws, hipStream_t s) {
  switch (bin) {
    case 0: return launch<T, VEC, 0>(C, B, ws, s);
    case 1: return launch<T, VEC, 1>(C, B, ws, s);
    case 2: return launch<T, VEC, 2>(C, B, ws, s);
    default: return launch<T, VEC, 3>(C, B, ws, s);
  }
}

// Rays from which the two passes are taken.  They add a launch, ~10 us for
// few rays; memory atomics take 26-75 ns per 1,000 rays (1M rays on 1024x1024:
// 51 us in all against 42, on 512x512: 93 against 42; 200,000 rays: the
// launches are all that shows, 35 against 41).
constexpr int64_t kBandRays = 1 << 18;

bool by_bands(int64_t n, int64_t bins, int32_t acc_dtype) {
  return acc_dtype <= 1 && bins > kLdsBins && bins < ((int64_t)1 << 31) && n >= kBandRays && n < ((int64_t)1 << 31);
}

}  // namespace

extern "C" int64_t tg_ray_column_workspace(int64_t n, int64_t height, int64_t width, int32_t acc_dtype) {
  if (n <= 0 || height <= 0 || width <= 0 || height > ((int64_t)1 << 31) / width) return 0;
  if (!by_bands(n, height * width, acc_dtype)) return 0;
  return (char*)(bin_workspace(nullptr, n).index + (n + 3) / 4 * 4) - (char*)nullptr;
}

extern "C" int tg_ray_column_run(const tg_column* column, const tg_bin_spec* bin, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
  tg::clear_error();
  TG_REQUIRE(column != nullptr, "tg_ray_column_run: column is NULL");
  const tg_column& C = *column;
  TG_REQUIRE(C.dtype == TG_F32 || C.dtype == TG_F64, "tg_ray_column_run: bad dtype %d", C.dtype);
  TG_REQUIRE(C.n >= 0, "tg_ray_column_run: negative ray count %lld", (long long)C.n);
  TG_REQUIRE(C.n_step >= 0 && C.n_step <= TG_MAX_STEP, "tg_ray_column_run: n_step %d out of range", C.n_step);
  for (int s = 0; s < C.n_step; ++s)
    TG_REQUIRE(C.step[s].kind >= TG_STEP_NONE && C.step[s].kind <= TG_STEP_BIPRISM,
               "tg_ray_column_run: step %d has bad kind %d", s, C.step[s].kind);
  tg_bin_spec B{};
  int mode = 0;
  if (bin != nullptr && bin->enabled) {
    B = *bin;
    TG_REQUIRE(B.acc != nullptr, "tg_ray_column_run: bin accumulator is NULL");
    TG_REQUIRE(B.height > 0 && B.width > 0, "tg_ray_column_run: bad detector shape");
    TG_REQUIRE(B.acc_dtype >= 0 && B.acc_dtype <= 3, "tg_ray_column_run: bad accumulator dtype");
    TG_REQUIRE(B.w_reg < 0, "tg_ray_column_run: columns bin unit weights");
    TG_REQUIRE(B.grid_hint >= 0, "tg_ray_column_run: negative grid_hint");
    mode = B.acc_dtype <= 1 && B.height * B.width <= kLdsBins ? 1 : 2;
    const int64_t need = tg_ray_column_workspace(C.n, B.height, B.width, B.acc_dtype);
    if (need > 0 && workspace != nullptr && workspace_bytes >= need) {
      TG_REQUIRE((uintptr_t)workspace % 16 == 0, "tg_ray_column_run: workspace not 16-byte aligned");
      mode = 3;
    }
  }
  if (C.n == 0) return TG_OK;
  uintptr_t bits = 0;
  for (int k = 0; k < 5; ++k) {
    TG_REQUIRE(k == 4 || C.in[k] != nullptr, "tg_ray_column_run: input %d is NULL", k);
    bits |= (uintptr_t)C.in[k] | (uintptr_t)C.out[k];
  }
  TG_REQUIRE(bits % (C.dtype == TG_F32 ? 4 : 8) == 0, "tg_ray_column_run: misaligned array");
  const bool aligned = bits % 16 == 0;
  hipStream_t s = (hipStream_t)stream;
  if (C.dtype == TG_F32)
    return aligned ? dispatch<float, 4>(C, B, mode, workspace, s) : dispatch<float, 1>(C, B, mode, workspace, s);
  return aligned ? dispatch<double, 2>(C, B, mode, workspace, s) : dispatch<double, 1>(C, B, mode, workspace, s);
}
