// Gaussian-beamlet field sums (reference gaussian.py:225-427).
//
// Stage 1 (beamlet_coef_kernel, one lane per beamlet, f64): the reference's
// per-beamlet 2x2 complex algebra -- Q1^-1 from waist/radius/theta
// (gaussian.py:138-177), Q2^-1 = solve(A + B Q1^-1, C + D Q1^-1)
// (gaussian.py:92-96), the misalignment phases phi1, phi2, the offset term
// 2 r.f and the prefactor amp / sqrt(det(A + B Q1^-1)) (gaussian.py:276-316),
// or the input-plane Gaussian (gaussian.py:402-407) -- is folded together
// with the k*pathlength phase and the Grid's pixel->metre map into
//   Phi(px, py) = a px^2 + b px py + c py^2 + d px + e py + f   (complex),
// so that a beamlet's field at pixel (py, px) is exp(Phi).  The envelope
// exp(Re Phi) gives the culling ellipse.
//
// Stage 2 (beamlet_sum_kernel): a workgroup owns a 64x64 detector tile and a
// slice of the beamlets.  Beamlets whose cutoff ellipse overlaps the tile are
// compacted (deterministically, by wavefront ballots) into an LDS list.  Each
// lane owns a run of 16 pixels of one row; per beamlet it evaluates Phi in
// f64 at the first pixel of the run that lies inside the ellipse (phase
// reduced to revolutions in double-double), then walks the run with the
// complex multiplicative recurrence F <- F R, R <- R K (K = exp(2a)): two
// complex f32 products per pixel, no transcendental per pixel.  Partial tiles
// of the beamlet slices are summed in a fixed order by a final kernel.
//
// Backward (tg_beamlet_backward): for a real loss L of the field, with the
// cotangent g = dL/dRe(field) + i dL/dIm(field) and W = conj(g),
//   dL/dtheta = Re sum_pixels W du_b/dtheta,  u_b = amp exp(Phi'_b(px, py)),
// Phi' being Phi with unit amplitude.  One wavefront per beamlet reduces the
// six complex moments sum W exp(Phi') {1, u, v, u^2, uv, v^2} over its cutoff
// ellipse (the kernel shared with the batched fits); then, per beamlet in
// f64, the moments give G_k = sum W exp(Phi') m_k for the six monomials
// m_k = px^2, px py, py^2, px, py, 1 of Phi, and
//   dL/dtheta = Re[amp sum_k G_k dc_k/dtheta]
// with dc_k/dtheta from forward-mode dual numbers through the same
// coefficient algebra (one pass per parameter and ray-transfer entry).
#include <string.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "beamlet_common.hpp"

namespace {

using namespace tgb;

// The parameter rows of n beamlets from their 13 columns (an array each, or a
// value for all), and a matrix that the host knows: one launch in place of the
// torch operations that converted, stacked and copied them.  Bound: the launch,
// the rows' store for many beamlets (131,072: 17 MB).  A lane writes one entry,
// so that a wavefront stores 512 bytes in a row.
struct PackArgs {
  tg_beamlet_column col[TG_BEAMLET_NCOLUMN];
  double matrix[25];
};

__global__ __launch_bounds__(256) void beamlet_pack_kernel(const PackArgs a, int64_t n, double* __restrict__ out,
                                                           double* __restrict__ matrix_out) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (matrix_out != nullptr && i < 25) matrix_out[i] = a.matrix[i];
  const int c = threadIdx.x % TG_BEAMLET_NPARAM;  // the stride below is a multiple of it
  const tg_beamlet_column col = a.col[c < TG_BEAMLET_NCOLUMN ? c : 0];
  const int32_t type = c < TG_BEAMLET_NCOLUMN ? col.type : TG_COLUMN_VALUE;
  const double value = c < TG_BEAMLET_NCOLUMN ? col.value : 0.0;
  for (; i < n * TG_BEAMLET_NPARAM; i += (int64_t)gridDim.x * 256) {
    const int64_t at = i / TG_BEAMLET_NPARAM * col.stride;
    out[i] = type == TG_COLUMN_F64   ? static_cast<const double*>(col.data)[at]
             : type == TG_COLUMN_F32 ? (double)static_cast<const float*>(col.data)[at]
                                     : value;
  }
}

__global__ __launch_bounds__(256) void beamlet_coef_kernel(const double* __restrict__ params, int64_t n,
                                                           const double* __restrict__ abcd, int64_t abcd_stride,
                                                           int32_t mode, double m0, double m1, double m2, double m3,
                                                           double m4, double m5, float cut,
                                                           tg_beamlet_coef* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* p = params + i * TG_BEAMLET_NPARAM;
  const double m[6] = {m0, m1, m2, m3, m4, m5};
  const double* T = mode == TG_BEAMLET_PROPAGATED ? abcd + i * abcd_stride : nullptr;
  out[i] = make_coef(p, T, mode, m, mk(p[5], p[6]), cut);
}

// ---------------------------------------------------------------------------
// Path selection: kFlagBlocks workgroups each write whether their share of
// the beamlets holds one that is not separable (every entry rewritten per
// launch, no atomics); every tile-sum workgroup reads all of them.
// ---------------------------------------------------------------------------
constexpr int kFlagBlocks = 256;

// exp(Phi) = Ex(px) Ey(py) with bounded factors: no px*py term, an envelope
// that decays along both axes, finite coefficients.
__device__ __forceinline__ bool separable(const tg_beamlet_coef& c) {
  bool fin = true;
#pragma unroll
  for (int j = 0; j < 12; ++j) fin = fin && isfinite(c.phi[j]);
  return fin && c.phi[2] == 0.0 && c.phi[3] == 0.0 && c.phi[0] < 0.0 && c.phi[4] < 0.0;
}

// The factors of a separable beamlet (b = 0):
//   Ex = exp(ar (px - cx)^2 + i (ai px^2 + di px)),
//   Ey = exp(cr (py - cy)^2 + g0 + i (ci py^2 + ei py + fi)),
// with a = ar + i ai etc., cx = -dr / (2 ar), cy = -er / (2 cr) and
// g0 = fr - ar cx^2 - cr cy^2 (the log of the peak amplitude): |Ex| <= 1 and
// |Ey| <= the peak.  One axis is
//   exp(q2 (p - cen)^2 + g + i (q1 p^2 + l1 p + c0)).
struct SepAxis {
  float q2l, gl;  // q2 and g times log2(e)
  double q1, l1, c0, cen;
};

// The factors of n beamlets, 96 bytes each: what every tile reads (the cutoff
// ellipse cx, cy, gamma, beta, then gl and the x factor's q2l), the x
// factors (gl = c0 = 0 left out), the y factors.
struct SepTables {
  float4* cull;
  float2* peak;   // gl, q2l of x
  double* x;      // 4 a beamlet: (q2l, -), q1, l1, cen
  double* y;      // 5 a beamlet: (q2l, gl), q1, l1, c0, cen
};
constexpr int64_t kSepBytes = 96;
constexpr double kLog2e = 1.4426950408889634;

__host__ __device__ inline SepTables sep_tables(void* p, int64_t n) {
  SepTables t;
  t.cull = (float4*)p;
  t.peak = (float2*)(t.cull + n);
  t.x = (double*)(t.peak + n);
  t.y = t.x + 4 * n;
  return t;
}

__device__ __forceinline__ double two_floats(float lo, float hi) {
  return __hiloint2double(__float_as_int(hi), __float_as_int(lo));
}

__device__ __forceinline__ void store_sep(const SepTables& t, int64_t i, const tg_beamlet_coef& c) {
  const double ar = c.phi[0], cr = c.phi[4];
  const double cx = -c.phi[6] / (2.0 * ar), cy = -c.phi[8] / (2.0 * cr);
  const float qx = (float)(ar * kLog2e), qy = (float)(cr * kLog2e);
  const float gl = (float)((c.phi[10] - ar * cx * cx - cr * cy * cy) * kLog2e);
  t.cull[i] = make_float4(c.cx, c.cy, c.gamma, c.beta);
  t.peak[i] = make_float2(gl, qx);
  double* x = t.x + 4 * i;
  x[0] = two_floats(qx, 0.0f);
  x[1] = c.phi[1];
  x[2] = c.phi[7];
  x[3] = cx;
  double* y = t.y + 5 * i;
  y[0] = two_floats(qy, gl);
  y[1] = c.phi[5];
  y[2] = c.phi[9];
  y[3] = c.phi[11];
  y[4] = cy;
}

__device__ __forceinline__ SepAxis load_sep(const SepTables& t, int64_t i, bool y_axis) {
  const double* p = y_axis ? t.y + 5 * i : t.x + 4 * i;
  const double q = p[0];
  return {__int_as_float(__double2loint(q)), __int_as_float(__double2hiint(q)), p[1], p[2],
          y_axis ? p[3] : 0.0, p[y_axis ? 4 : 3]};
}

// flags[blockIdx.x]: some beamlet of this workgroup's share is not separable
// (or force_valu); tab[i]: the factors of beamlet i when it is separable.
__global__ __launch_bounds__(256) void sep_flag_kernel(const tg_beamlet_coef* __restrict__ coef, int64_t n,
                                                       int32_t force_valu, int32_t* __restrict__ flags,
                                                       SepTables tab) {
  int bad = force_valu;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n && !force_valu; i += (int64_t)gridDim.x * 256) {
    const tg_beamlet_coef& c = coef[i];
    if (separable(c))
      store_sep(tab, i, c);
    else
      bad = 1;
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) flags[blockIdx.x] = bad;
}

// True (in every thread of the workgroup) when the launch takes the
// matrix-core path.
__device__ __forceinline__ bool matrix_path(const int32_t* __restrict__ flags) {
  const int bad = threadIdx.x < kFlagBlocks ? flags[threadIdx.x] : 0;
  return !__syncthreads_or(bad);
}

template <int LPR, int RUN>
__global__ __launch_bounds__(kThreads) void beamlet_sum_kernel(const tg_beamlet_coef* __restrict__ coef, int64_t n,
                                                               int64_t H, int64_t W, int32_t ntx, int32_t ntiles,
                                                               int32_t nsplit, const int32_t* __restrict__ flags,
                                                               float2* __restrict__ ws) {
  __shared__ TileLists sh;
  if (matrix_path(flags)) return;  // beamlet_sum_sep_kernel covers this launch
  const int split = blockIdx.x % nsplit, tile = blockIdx.x / nsplit;  // slices of a tile adjacent
  const int32_t tx0 = (tile % ntx) * (LPR * RUN), ty0 = (tile / ntx) * (kThreads / LPR);
  const int64_t b_begin = n * split / nsplit, b_end = n * (split + 1) / nsplit;
  tile_sum_store<LPR, RUN>(coef, b_begin, b_end, tx0, ty0, (int32_t)H, (int32_t)W, sh, ws + (int64_t)split * H * W);
}

// ---------------------------------------------------------------------------
// Separable beamlets on the matrix cores.  A tile is the complex matrix
// product  T[m][n] = sum_k Ey_k(ty0 + m) Ex_k(tx0 + n)  over the beamlets whose
// cutoff ellipse meets it, K = beamlets.
//
// Precision.  A factor value is held as two f16, x = h + l (l the rounding of
// h, itself rounded: 22 bits, no less than the 16 phasor steps behind a value
// carry), and a real product is ah bh + ah bl + al bh in f32 accumulators (what
// is left out is below 2^-22 |a b|).  f16 has few exponents, so the factors are
// scaled: each x factor by the power of two that takes its largest value in
// the tile (its pixels on the image) to [2^14, 2^15), and the y factor,
// amplitude included, by the rest, so that no term exceeds 2^29 times
// 2^exp, the largest of the slice's terms in the tile.  What a factor has below
// 2^-25 is lost, 2^-39 of its largest value: so the halves serve a slice and
// tile all of whose terms that are to be kept lie within 2^20 of 2^exp (then no
// kept term is off by more than 2^-19 of itself), or are cut off at no less than
// 2^-25 of it (2^-14 of the weakest kept, in the mean 2^-16, where the cut leaves
// out terms of that size).  Any other -- tails without a cut, weak beamlets
// beside strong ones -- is left to the f32 products of beamlet_sum_wide_kernel.
// Against complex128, norm of the error over norm of the field, 131,072
// beamlets on 1024^2: 3.9e-6 (f32 products: 4.2e-6; both are the phasor
// recurrence's error).
//
// Rate.  12 v_mfma_f32_32x32x16_f16 take 16 beamlets of a 32x32 block, 25
// cycles a beamlet, where f32 products (three v_mfma_f32_32x32x2_f32 a pair)
// take 96.  And vector instructions run beside f16 MFMAs, which they do not
// beside f32 ones (register-only chains, two wavefronts a SIMD: 8 FMAs beside
// each MFMA cost 33 -> 44 cycles in f16, 67 -> 103 in f32).  (Three bf16 parts,
// six products, 24 bits: 3.75 ms where f16 takes 2.45.)
//
// A workgroup owns a 128x128 tile, a wave 2x2 of its 32x32 blocks: evaluating
// a factor costs about as much as its products, and a wider tile uses a value
// more often.  131,072 beamlets on 1024^2: 2.45 ms, 64x64 tiles (one block a
// wave) 3.06 ms; 20,000 on 512^2: 398 and 496 us; on images of one tile the two
// differ by less than the launch's host work, so there is one tile shape.
// 16 beamlets a chunk go through two LDS buffers, one barrier a chunk: beside
// its products of chunk c every lane evaluates one 16-pixel segment of one
// factor of chunk c + 1, a pixel between every three products (at raised
// priority: a wave between its loads would otherwise hold up the matrix cores'
// next instruction; 2.57 -> 2.45 ms), with chunk c + 2's parameters in flight.
// A lane's beamlet is k = lane & 15; lanes k and k + 1 exchange a component
// (DPP) so that the even lane packs both real parts and the odd one both
// imaginary parts: the operand layout wants consecutive beamlets side by side.
// A pixel's 16 beamlets take 32 bytes, with 64 more after every 16 pixels and
// 32 between the arrays: stores of a wavefront meet 64 banks, operand reads
// (16 bytes a lane) are contiguous.
//
// A segment's value is  exp2(q2' (p - cen)^2 + g') (cos, sin)(2 pi theta(p)),
//   theta(p0 + j) = theta0 + j A + j^2 B   (revolutions),
// theta0 being the segment start's phase reduced in double-double.  theta0,
// A and B are reduced modulo one revolution as 32-bit fixed-point fractions
// (exact whatever the size of the linear and quadratic phase terms; an f32
// sum theta0 + jA + j^2 B lost 1e-5 revolutions on strongly curved
// input-plane beamlets), and seed a unit-phasor recurrence (two transcendental
// pairs per segment instead of a sine and cosine per value).
//
// 131,072 beamlets, 1024^2, 4 sigma, the whole sum: 4.64 ms with f32 products,
// now 2.17 ms (of which the search for the range is 0.02).  Bound: vector issue
// (63% of the cycles, 520 instructions a chunk) and the matrix cores (48%)
// together, at the 1.7 to 1.9 GHz that this mix runs at.
// ---------------------------------------------------------------------------
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int kMxK = 16;           // beamlets per MFMA
constexpr int kMxSeg = 16;         // pixels per evaluated segment
constexpr int kMxBlock = 1024;     // beamlets per list build
constexpr int kMxScaleX = 14;      // x factors are held times 2^14, below 2^15
constexpr int kMxScaleY = 15;      // y factors at most 2^15 (f16 ends at 2^16)
constexpr int kMxScale = kMxScaleX + kMxScaleY;
constexpr int kMxRange = 20;       // bits from the largest term to the weakest that the halves serve
constexpr int kMxCutBits = 5;      // further bits for a term at its own cut

// A TW x TH tile, KC beamlets a chunk, BM x BN 32x32 blocks a wave: LDS layout
// and workgroup.
template <int TW_, int TH_, int KC_, int BM_, int BN_>
struct MxTile {
  static constexpr int TW = TW_, TH = TH_, KC = KC_, BM = BM_, BN = BN_;
  static constexpr int kPix = TW + TH;  // x pixels, then y pixels
  // waves side by side and one below the other; a wave's blocks lie as far apart
  static constexpr int kCols = TW / (32 * BN), kRows = TH / (32 * BM);
  static constexpr int kWaves = kCols * kRows, kThreads = 64 * kWaves;
  // dwords (two beamlets each) of one component of one split part, and of the
  // four of them for one MFMA's beamlets
  static constexpr int kPart = kPix * (kMxK / 2) + kPix / 16 * 16 + 8;
  static constexpr int kStep = 4 * kPart;
  static constexpr int kBuffer = KC / kMxK * kStep;
  static_assert(TW % (32 * BN) == 0 && TH % (32 * BM) == 0 && TW % 64 == 0 && kPart % 64 == 8 && kStep % 64 == 32,
                "whole blocks; stores of a wavefront on 64 banks");
  static_assert(KC * kPix / kMxSeg == kThreads, "one segment a lane");
};

using SepTile = MxTile<128, 128, 16, 2, 2>;

constexpr int kNoExp = -(1 << 24);  // no beamlet met yet
constexpr int kLeft = 0x7fa51e55;   // (a signalling NaN, which no sum is)

__device__ __forceinline__ int wave_max_i32(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// dword offset of a pixel's row within a part
__host__ __device__ constexpr int mx_row(int pix) { return pix * (kMxK / 2) + (pix >> 4) * 16; }

// Evaluation state of one 16-pixel segment starting at pixel p0: the
// log2-scaled envelope, evaluated directly, and the unit phasor
// z_j = exp(2 pi i theta(p0 + j)) stepped by the unit ratios
// r_j = z_{j+1} / z_j, r_{j+1} = r_j k (|z| = 1: nothing to underflow).  The
// seeds come from theta0, A and B reduced modulo one revolution as 32-bit
// fixed-point fractions (exact wrapping integer arithmetic), so the phase
// error is that of 16 f32 rotations (CPU emulation of this scheme: worst
// 1.4e-5 rad, |z| within 6e-6 of 1).  An invalid segment evaluates to zero.
struct SegGen {
  float2 z, r, k;
  float t0, q2l, gl;
};

// r (revolutions, |r| < 2^52) modulo one, in 2^-32 units, rounded to nearest:
// the low word of the fraction times 2^32 plus 1.5 2^52 (a conversion to a
// 64-bit integer takes about ten instructions)
__device__ __forceinline__ uint32_t fixed_revolutions(double r) {
  const double f = fma(r - rint(r), 4294967296.0, 6755399441055744.0);
  return (uint32_t)__double2loint(f);
}

// exp(2 pi i u 2^-32)
__device__ __forceinline__ float2 phasor(uint32_t u) {
  const float t = (float)(int32_t)u * 0x1p-32f;  // [-0.5, 0.5) revolutions
  return make_float2(__builtin_amdgcn_cosf(t), __builtin_amdgcn_sinf(t));
}

// exponent: added to the envelope's log2.  swap: the values come out as (im,
// re): z with its parts exchanged, stepped by the conjugate ratios.
__device__ __forceinline__ SegGen seg_setup(const SepAxis& v, double p0, float exponent, bool valid, bool swap) {
  // theta(p0 + j) = theta0 + j A + j^2 B  (revolutions)
  const double x = fma(fma(v.q1, p0, v.l1), p0, v.c0);
  const double hi = x * kInv2PiHi;
  const double theta0 = (hi - rint(hi)) + fma(x, kInv2PiLo, fma(x, kInv2PiHi, -hi));
  const uint32_t a = fixed_revolutions(fma(2.0 * v.q1, p0, v.l1) * kInv2PiHi);
  const uint32_t b = fixed_revolutions(v.q1 * kInv2PiHi);
  SegGen s;
  // (quarter turn minus theta: (sin, cos); minus a phase: the conjugate)
  const uint32_t flip = swap ? 0xffffffffu : 0u;
  const uint32_t t = fixed_revolutions(theta0);
  s.z = phasor(swap ? 0x40000000u - t : t);
  s.r = phasor(((a + b) ^ flip) - flip);  // theta(1) - theta(0) = A + B
  s.k = phasor(((2u * b) ^ flip) - flip);  // second difference 2 B
  s.t0 = (float)(p0 - v.cen);
  s.q2l = v.q2l;
  s.gl = valid ? v.gl + exponent : -INFINITY;
  return s;
}

// The segment's value at pixel p0 + j (j = 0, 1, ... in turn).
__device__ __forceinline__ float2 seg_next(SegGen& s, int j) {
  const float t = s.t0 + (float)j;
  const float mag = __builtin_amdgcn_exp2f(fmaf(s.q2l * t, t, s.gl));
  const float2 v = make_float2(mag * s.z.x, mag * s.z.y);
  s.z = cmulf(s.z, s.r);
  s.r = cmulf(s.r, s.k);
  return v;
}

// Two values rounded to f16, packed (first in the low half), and what the
// rounding left of them (one mixed-precision instruction each).
__device__ __forceinline__ uint32_t take_f16(float& u, float& v) {
  const f16x2 p = __builtin_convertvector((floatx2){u, v}, f16x2);
  const uint32_t w = __builtin_bit_cast(uint32_t, p);
  asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(u) : "v"(w));
  asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(v) : "v"(w));
  return w;
}

// Pixel j of a segment: lanes k (even) and k + 1 exchange their second
// components; high and low get the halves of both beamlets' real parts (even
// lane) or imaginary parts (odd lane, whose values come as (im, re)).
__device__ __forceinline__ void mx_pack(float2 v, bool odd, uint32_t& high, uint32_t& low) {
  const float got = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v.y), 0xB1, 0xF, 0xF, true));  // lane ^ 1
  float a = odd ? got : v.x, b = odd ? v.x : got;
  high = take_f16(a, b);
  low = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){a, b}, f16x2));
}

// Operands of one component: its high and low halves.
struct MxOperand {
  f16x8 h, l;
};

template <int PART>
__device__ __forceinline__ MxOperand mx_load(const uint32_t* src) {
  return {*reinterpret_cast<const f16x8*>(src), *reinterpret_cast<const f16x8*>(src + 2 * PART)};
}

__device__ __forceinline__ f16x8 mx_neg(f16x8 v) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(f16x8, __builtin_bit_cast(u32x4, v) ^ 0x80008000u);
}

// Product P of the 12 of a 32x32 block: the three of a real product (smallest
// first), for each of re += ar br, im += ai br, re -= ai bi, im += ar bi; the
// real and imaginary sums in turn.
template <int P>
__device__ __forceinline__ void mx_mfma(const MxOperand& ar, const MxOperand& ai, const MxOperand& br,
                                        const MxOperand& bi, const MxOperand& bn, floatx16& re, floatx16& im) {
  constexpr bool to_im = P & 1, second = P >= 6;
  constexpr int part = (P / 2) % 3;
  const MxOperand& a = to_im != second ? ai : ar;
  const MxOperand& b = !second ? br : to_im ? bi : bn;
  floatx16& acc = to_im ? im : re;
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(part == 0 ? a.l : a.h, part == 1 ? b.l : b.h, acc, 0, 0, 0);
}

// f(0), f(1), ... f(N - 1) with compile-time arguments
template <int N, class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

template <class M>
__global__ __launch_bounds__(M::kThreads, 2) void beamlet_sum_sep_kernel(const SepTables tab, int64_t n, int64_t H,
                                                                    int64_t W, int32_t ntx, int32_t nsplit,
                                                                    const int32_t* __restrict__ flags,
                                                                    float2* __restrict__ ws) {
  constexpr int kT = M::kThreads, kW = M::kWaves, TW = M::TW, TH = M::TH;
  __shared__ int32_t list[kMxBlock];
  __shared__ int32_t wave_cnt[kW], wave_low[kW];
  __shared__ __align__(16) uint32_t fac[2][M::kBuffer];
  if (!matrix_path(flags)) return;  // beamlet_sum_kernel covers this launch
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // the slices of one tile are consecutive workgroups: the heavy tiles near
  // the pattern's centre are spread through the dispatch order instead of
  // all ending it
  const int split = blockIdx.x % nsplit, tile = blockIdx.x / nsplit;
  const int32_t tx0 = (tile % ntx) * TW, ty0 = (tile / ntx) * TH;
  const int64_t b_begin = n * split / nsplit, b_end = n * (split + 1) / nsplit;
  // the tile's pixels on the image: nothing past them is scaled for
  const int32_t tx1 = (int32_t)min((int64_t)tx0 + TW, W) - 1, ty1 = (int32_t)min((int64_t)ty0 + TH, H) - 1;
  const float ftx0 = (float)tx0, fty0 = (float)ty0, ftx1 = (float)tx1, fty1 = (float)ty1;
  const int mb = (wave / M::kCols) * 32, nb = (wave % M::kCols) * 32;
  constexpr int kBlockX = 32 * M::kCols, kBlockY = 32 * M::kRows;  // from a wave's block to its next
  // operand reads: A[m][k] = Ey_k(ty0 + mb + m), B[k][n] = Ex_k(tx0 + nb + n); lane l holds row (column) l % 32,
  // k = 8 (l / 32) .. + 7 (v_mfma_f32_32x32x16 operand layout)
  const int a_at = mx_row(TW + mb + (lane & 31)) + 4 * (lane >> 5), b_at = mx_row(nb + (lane & 31)) + 4 * (lane >> 5);
  // this thread's segment: beamlet gk of a chunk, 16 pixels from p0 of one axis
  // (one axis a wave: TW is a multiple of a wave's pixels)
  const int gk = t % M::KC, seg = t / M::KC;
  const bool y_axis = __builtin_amdgcn_readfirstlane(seg * kMxSeg) >= TW, odd = lane & 1;
  const double p0 = (double)(y_axis ? ty0 + seg * kMxSeg - TW : tx0 + seg * kMxSeg);
  const double dtx0 = (double)tx0, dtx1 = (double)tx1;
  const int dst_at = (gk / kMxK) * M::kStep + odd * M::kPart + mx_row(seg * kMxSeg) + (gk % kMxK) / 2;
  floatx16 re[M::BM][M::BN], im[M::BM][M::BN];
#pragma unroll
  for (int i = 0; i < M::BM; ++i)
#pragma unroll
    for (int k = 0; k < M::BN; ++k)
#pragma unroll
      for (int j = 0; j < 16; ++j) re[i][k][j] = im[i][k][j] = 0.0f;
  // A separable beamlet's cutoff ellipse is axis-aligned (alpha = 0): u^2 +
  // gamma v^2 <= beta, so the tile's pixel centre nearest (cx, cy) decides,
  // exactly, whether it meets the tile -- tiles in the corners of the ellipse's
  // bounding box are skipped.
  auto meets = [&](float4 c, float& du, float& dv) {  // cx, cy, gamma, beta
    du = fmaxf(fmaxf(ftx0 - c.x, c.x - ftx1), 0.0f);
    dv = fmaxf(fmaxf(fty0 - c.y, c.y - fty1), 0.0f);
    return fmaf(c.z * dv, dv, du * du) <= c.w;
  };
  // The exponents of the slice's largest term in the tile and of the least that is to be kept.
  int exp_now = kNoExp, low = -kNoExp;
#pragma unroll 2
  for (int64_t b = b_begin + t; b < b_end; b += kT) {
    const float4 c = tab.cull[b];
    const float2 p = tab.peak[b];
    float du, dv;
    if (!meets(c, du, dv)) continue;
    // no term exceeds 2^top (the centre's f32 rounding taken off the distances)
    du = fmaxf(fmaf(-0x1p-22f, fabsf(c.x), du), 0.0f);
    dv = fmaxf(fmaf(-0x1p-22f, fabsf(c.y), dv), 0.0f);
    const float top = ceilf(fmaf(p.y, fmaf(c.z * dv, dv, du * du), p.x));
    // nor is any that is to be kept below 2^far: the pixel farthest from the centre, or the cut
    du = fmaxf(c.x - ftx0, ftx1 - c.x);
    dv = fmaxf(c.y - fty0, fty1 - c.y);
    const float far = fmaxf(fmaf(p.y, fmaf(c.z * dv, dv, du * du), p.x), fmaf(p.y, c.w, p.x) + (float)kMxCutBits);
    exp_now = max(exp_now, (int)fminf(fmaxf(top, -1e6f), 1e6f));
    low = min(low, (int)(far >= -1e6f ? fminf(floorf(far), 1e6f) : -1e6f));
  }
  exp_now = wave_max_i32(exp_now);
  low = -wave_max_i32(-low);
  if (lane == 0) wave_cnt[wave] = exp_now, wave_low[wave] = low;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    exp_now = max(exp_now, wave_cnt[w]);
    low = min(low, wave_low[w]);
  }
  exp_now = __builtin_amdgcn_readfirstlane(exp_now);
  const bool leave = exp_now != kNoExp && low < exp_now - kMxRange;  // more than the halves hold
  if (leave) {
    const int32_t x = tx0 + (t & 1) * kTileW, y = ty0 + (t >> 1) * kTileH;
    static_assert(TW == 2 * kTileW && TH == 2 * kTileH, "four tiles of beamlet_sum_wide_kernel");
    if (t < 4 && x < W && y < H)
      ws[((int64_t)split * H + y) * W + x] = make_float2(__int_as_float(kLeft), __int_as_float(exp_now));
    return;
  }
  __syncthreads();  // wave_cnt is rewritten
  // the sums are held times 2^(kMxScale - exp_now)
  for (int64_t blk = b_begin; blk < b_end; blk += kMxBlock) {
    // the beamlets of [blk, blk + kMxBlock) that meet the tile, in order
    int cnt = 0;
    for (int64_t b0 = blk; b0 < b_end && b0 < blk + kMxBlock; b0 += kT) {
      const int64_t b = b0 + t;
      float du, dv;
      const bool hit = b < b_end && meets(tab.cull[b], du, dv);
      const uint64_t mask = __ballot(hit);
      if (lane == 0) wave_cnt[wave] = __popcll(mask);
      __syncthreads();
      int off = cnt, total = 0;
#pragma unroll
      for (int w = 0; w < kW; ++w) {
        off += (w < wave) ? wave_cnt[w] : 0;
        total += wave_cnt[w];
      }
      if (hit) list[off + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)(b - blk);
      cnt += total;
      __syncthreads();  // wave_cnt is rewritten next; the list is complete after the last pass
    }
    if (cnt == 0) continue;
    const int nch = (cnt + M::KC - 1) / M::KC;
    // chunk q's beamlet for this thread (past cnt: the last one again,
    // evaluated as zero), and the power of two its factor is multiplied by: an
    // x factor's largest value in the tile goes to [2^14, 2^15) and the y
    // factor takes the rest
    float ex = 0.0f;
    auto load = [&](int q) {
      const int64_t i = blk + list[min(q * M::KC + gk, cnt - 1)];
      const SepAxis a = load_sep(tab, i, y_axis);
      const double* x = tab.x + 4 * i;
      const float qx = y_axis ? __int_as_float(__double2loint(x[0])) : a.q2l;
      const double cen = y_axis ? x[3] : a.cen;
      const float du = (float)fmax(fmax(dtx0 - cen, cen - dtx1), 0.0);
      const float top = fmaxf(floorf(qx * du * du), -1e6f);
      ex = y_axis ? (float)kMxScaleY + top - (float)exp_now : (float)kMxScaleX - top;
      return a;
    };
    SepAxis v = load(0);
    {
      SegGen sg = seg_setup(v, p0, ex, gk < cnt, odd);
      v = load(1);
      uint32_t* dst = &fac[0][dst_at];
#pragma unroll
      for (int j = 0; j < kMxSeg; ++j)
        mx_pack(seg_next(sg, j), odd, dst[j * (kMxK / 2)], dst[j * (kMxK / 2) + 2 * M::kPart]);
    }
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
      const uint32_t* cur = fac[c & 1];
      constexpr int S = M::KC / kMxK;
      MxOperand ar[S][M::BM], ai[S][M::BM], br[S][M::BN], bi[S][M::BN], bn;
#pragma unroll
      for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int i = 0; i < M::BM; ++i) {
          ar[s][i] = mx_load<M::kPart>(cur + s * M::kStep + a_at + mx_row(i * kBlockY));
          ai[s][i] = mx_load<M::kPart>(cur + s * M::kStep + M::kPart + a_at + mx_row(i * kBlockY));
        }
#pragma unroll
        for (int k = 0; k < M::BN; ++k) {
          br[s][k] = mx_load<M::kPart>(cur + s * M::kStep + b_at + mx_row(k * kBlockX));
          bi[s][k] = mx_load<M::kPart>(cur + s * M::kStep + M::kPart + b_at + mx_row(k * kBlockX));
        }
      }
      // chunk c + 1's factors (past the last chunk: zeros nobody reads), and
      // chunk c + 2's parameters in flight
      SegGen sg = seg_setup(v, p0, ex, (c + 1) * M::KC + gk < cnt, odd);
      v = load(c + 2);
      __builtin_amdgcn_s_setprio(1);
      uint32_t* dst = &fac[(c & 1) ^ 1][dst_at];
      // a pixel of the segment beside its share of the products.  (The barriers
      // keep the steps apart: left alone, the scheduler issues all products
      // first and the evaluation after them.)
      static_for<kMxSeg>([&](auto step) {
        constexpr int j = step, kMfma = 12 * M::BM * M::BN * S;
        __builtin_amdgcn_sched_barrier(0);
        static_for<(j + 1) * kMfma / kMxSeg - j * kMfma / kMxSeg>([&](auto sub) {
          constexpr int q = j * kMfma / kMxSeg + sub, P = q % 12;
          constexpr int i = q / 12 % M::BM, k = q / (12 * M::BM) % M::BN, s = q / (12 * M::BM * M::BN);
          if constexpr (P == 0 && i == 0) bn = {mx_neg(bi[s][k].h), mx_neg(bi[s][k].l)};
          mx_mfma<P>(ar[s][i], ai[s][i], br[s][k], bi[s][k], bn, re[i][k], im[i][k]);
        });
        mx_pack(seg_next(sg, j), odd, dst[j * (kMxK / 2)], dst[j * (kMxK / 2) + 2 * M::kPart]);
      });
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();  // chunk c + 1 is complete and chunk c read
    }
  }
  // accumulator j of lane l holds row 8 (j / 4) + 4 (l / 32) + j % 4, column l % 32
#pragma unroll
  for (int i = 0; i < M::BM; ++i)
#pragma unroll
    for (int k = 0; k < M::BN; ++k)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int64_t py = ty0 + mb + i * kBlockY + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
        const int64_t px = tx0 + nb + k * kBlockX + (lane & 31);
        if (py < H && px < W)
          ws[((int64_t)split * H + py) * W + px] =
              make_float2(ldexpf(re[i][k][j], exp_now - kMxScale), ldexpf(im[i][k][j], exp_now - kMxScale));
      }
}

// ---------------------------------------------------------------------------
// The same sum with f32 factors and products, for the slices and tiles that
// beamlet_sum_sep_kernel leaves (marked in the tile's first pixel: kLeft and the
// largest term's exponent), a 64x64 tile a workgroup, wave w the 32x32 block at
// rows 32 (w / 2), columns 32 (w % 2).  |Ex| <= 1 and is at least exp(-80) at a
// pixel that is to be kept; Ey, amplitude included, is taken up by the power of
// two that brings the largest term to 2^10 (no visible value of Ey then exceeds
// 2^126, as its beamlet's term is at most exp(80) below it), never down: what a
// normal f32 holds of the field is held.  One k pair of the complex product is
// three real products (Gauss): p1 += a.re b.re, p2 += a.im b.im, p3 += (a.re +
// a.im)(b.re + b.im); then Re = p1 - p2 and Im = p3 - (p1 + p2).  Vector
// instructions and f32 MFMAs of a SIMD do not execute together (their times
// add), so the evaluation's instruction count is what it costs: one segment a
// thread and chunk, a value between the products of each k pair.  (In one kernel
// with the f16 products its registers spilled theirs.)  131,072 beamlets of 100
// pixels on 1024^2, no cut: 7.98 ms; where every tile is left out, 8 us for the
// workgroups of such an image, 1 us for a small one's.
// ---------------------------------------------------------------------------
constexpr int kWideScale = 10;
constexpr int kWideBlock = 2048;          // beamlets per list build
constexpr int kWideK = 32;                // beamlets per LDS chunk (the product's K)
constexpr int kWideRow = kTileW + 1;      // LDS row pitch (float2): a bank offset per beamlet row
static_assert(kTileW == 64 && kTileH == 64 && kThreads == 256 && kWideK * 2 * (kTileW / kMxSeg) == kThreads &&
                  kMxSeg == kWideK / 2,
              "64x64 tiles, four waves, one segment per thread and one segment value per k pair");

__device__ __forceinline__ void wide_mfma(float2 a, float2 b, floatx16& p1, floatx16& p2, floatx16& p3) {
  p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, p1, 0, 0, 0);
  p2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, p2, 0, 0, 0);
  p3 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x + a.y, b.x + b.y, p3, 0, 0, 0);
}

__global__ __launch_bounds__(kThreads) void beamlet_sum_wide_kernel(const SepTables tab, int64_t n, int64_t H,
                                                                    int64_t W, int32_t ntx, int32_t nsplit,
                                                                    const int32_t* __restrict__ flags,
                                                                    float2* __restrict__ ws) {
  __shared__ int32_t list[kWideBlock];
  __shared__ int32_t wave_cnt[kWaves];
  __shared__ float2 fac[2][2][kWideK][kWideRow];  // [buffer][x: Ex_k(tx0 + n), y: Ey_k(ty0 + m)][k][pixel]
  const int split = blockIdx.x % nsplit, tile = blockIdx.x / nsplit;
  const int32_t tx0 = (tile % ntx) * kTileW, ty0 = (tile / ntx) * kTileH;
  const float2 mark = ws[((int64_t)split * H + ty0) * W + tx0];
  if (__float_as_int(mark.x) != kLeft) return;  // beamlet_sum_sep_kernel's
  if (!matrix_path(flags)) return;              // beamlet_sum_kernel covers this launch (the mark is an older one's)
  const int exp_now = __float_as_int(mark.y);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t b_begin = n * split / nsplit, b_end = n * (split + 1) / nsplit;
  const int32_t tx1 = (int32_t)min((int64_t)tx0 + kTileW, W) - 1, ty1 = (int32_t)min((int64_t)ty0 + kTileH, H) - 1;
  const float ftx0 = (float)tx0, fty0 = (float)ty0, ftx1 = (float)tx1, fty1 = (float)ty1;
  const int mb = (wave >> 1) * 32, nb = (wave & 1) * 32;
  // this thread's segment: beamlet gk of a chunk, axis (waves 0-1: x, 2-3: y), pixels p0 .. p0 + 15
  const int gk = t & (kWideK - 1), s0 = ((t >> 5) & 3) * kMxSeg;
  const bool y_axis = __builtin_amdgcn_readfirstlane(t >> 7) != 0;
  const double p0 = (double)((y_axis ? ty0 : tx0) + s0);
  const double* axis = y_axis ? tab.y : tab.x;
  const int axis_step = y_axis ? 5 : 4;
  const int scale = max(kWideScale - exp_now, 0);
  const float ex = y_axis ? (float)scale : 0.0f;
  floatx16 p1, p2, p3;
#pragma unroll
  for (int j = 0; j < 16; ++j) p1[j] = p2[j] = p3[j] = 0.0f;
  for (int64_t blk = b_begin; blk < b_end; blk += kWideBlock) {
    const int64_t end = min(b_end, blk + kWideBlock);
    int cnt = 0;
    for (int64_t b0 = blk; b0 < end; b0 += kThreads) {
      const int64_t b = b0 + t;
      bool hit = false;
      if (b < end) {
        const float4 c = tab.cull[b];  // cx, cy, gamma, beta
        const float du = fmaxf(fmaxf(ftx0 - c.x, c.x - ftx1), 0.0f);
        const float dv = fmaxf(fmaxf(fty0 - c.y, c.y - fty1), 0.0f);
        hit = fmaf(c.z * dv, dv, du * du) <= c.w;
      }
      const uint64_t mask = __ballot(hit);
      if (lane == 0) wave_cnt[wave] = __popcll(mask);
      __syncthreads();
      int off = cnt, total = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        off += (w < wave) ? wave_cnt[w] : 0;
        total += wave_cnt[w];
      }
      if (hit) list[off + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)(b - blk);
      cnt += total;
      __syncthreads();  // wave_cnt is rewritten next; the list is complete after the last pass
    }
    if (cnt == 0) continue;
    // chunk q's beamlet for this thread (past cnt: the last one again, evaluated
    // as zero): load_sep without a branch, which the loads in flight would wait at
    auto load = [&](int q) -> SepAxis {
      const double* a = axis + axis_step * (blk + list[min(q * kWideK + gk, cnt - 1)]);
      const double c0 = a[3];
      return {__int_as_float(__double2loint(a[0])), __int_as_float(__double2hiint(a[0])), a[1], a[2], y_axis ? c0 : 0.0,
              a[axis_step - 1]};
    };
    SepAxis v = load(0);
    {
      SegGen sg = seg_setup(v, p0, ex, gk < cnt, false);
      v = load(1);
      float2* dst = &fac[0][y_axis][gk][s0];
#pragma unroll
      for (int j = 0; j < kMxSeg; ++j) dst[j] = seg_next(sg, j);
    }
    __syncthreads();
    const int nch = (cnt + kWideK - 1) / kWideK;
    for (int c = 0; c < nch; ++c) {
      // A[m][k] = Ey_k(ty0 + mb + m) from lane m + 32 k, B[k][n] = Ex_k(tx0 + nb + n) from lane n + 32 k
      // (v_mfma_f32_32x32x2f32 operand layout); operands one k pair ahead, so LDS latency hides behind the products
      const float2* ea = &fac[c & 1][1][lane >> 5][mb + (lane & 31)];
      const float2* eb = &fac[c & 1][0][lane >> 5][nb + (lane & 31)];
      float2 a = ea[0], b = eb[0];
      if (c + 1 < nch) {
        // chunk c + 1's factors beside the products, and chunk c + 2's parameters in flight
        SegGen sg = seg_setup(v, p0, ex, (c + 1) * kWideK + gk < cnt, false);
        v = load(c + 2);
        // (kept here: sunk below the products, the next chunk waited a memory round trip)
        __builtin_amdgcn_sched_barrier(0);
        // (stored after the products: a store between them would order every later operand read behind it)
        float2 val[kMxSeg];
#pragma unroll
        for (int kk = 0; kk < kWideK; kk += 2) {
          float2 an = a, bn = b;
          if (kk + 2 < kWideK) {
            an = ea[(kk + 2) * kWideRow];
            bn = eb[(kk + 2) * kWideRow];
          }
          wide_mfma(a, b, p1, p2, p3);
          val[kk >> 1] = seg_next(sg, kk >> 1);
          a = an;
          b = bn;
          // issue order: products and the value's dependent vector instructions alternate
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // four VALU
          }
        }
        float2* dst = &fac[(c & 1) ^ 1][y_axis][gk][s0];
#pragma unroll
        for (int j = 0; j < kMxSeg; ++j) dst[j] = val[j];
      } else {
#pragma unroll
        for (int kk = 0; kk < kWideK; kk += 2) {
          float2 an = a, bn = b;
          if (kk + 2 < kWideK) {
            an = ea[(kk + 2) * kWideRow];
            bn = eb[(kk + 2) * kWideRow];
          }
          wide_mfma(a, b, p1, p2, p3);
          a = an;
          b = bn;
        }
      }
      __syncthreads();  // chunk c + 1 is complete and chunk c read
    }
  }
  // accumulator j of lane l holds row 8 (j / 4) + 4 (l / 32) + j % 4, column l % 32
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int64_t py = ty0 + mb + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
    const int64_t px = tx0 + nb + (lane & 31);
    if (py < H && px < W)
      ws[((int64_t)split * H + py) * W + px] =
          make_float2(ldexpf(p1[j] - p2[j], -scale), ldexpf(p3[j] - (p1[j] + p2[j]), -scale));
  }
}

// The slices' sum, in order.  Bound: reading them; four loads in flight hide
// some of the latency where a small image has too few wavefronts for that (300
// beamlets on 100^2 pixels, the whole sum in 64 slices: 34 -> 24 us; eight: 22,
// but large images lose 3%).
__global__ __launch_bounds__(256) void split_sum_kernel(const float2* __restrict__ ws, int64_t npix, int32_t nsplit,
                                                        float2* __restrict__ field) {
  constexpr int kAhead = 4;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix) return;
  double re = 0.0, im = 0.0;
  int s = 0;
  for (; s + kAhead <= nsplit; s += kAhead) {
    float2 v[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) v[k] = ws[(int64_t)(s + k) * npix + i];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) re += v[k].x, im += v[k].y;
  }
  for (; s < nsplit; ++s) {
    const float2 v = ws[(int64_t)s * npix + i];
    re += v.x;
    im += v.y;
  }
  field[i] = make_float2((float)re, (float)im);
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void beamlet_unit_kernel(const double* __restrict__ params, int64_t n,
                                                           const double* __restrict__ abcd, int64_t abcd_stride,
                                                           int32_t mode, double m0, double m1, double m2, double m3,
                                                           double m4, double m5, float cut,
                                                           tg_beamlet_coef* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* p = params + i * TG_BEAMLET_NPARAM;
  const double m[6] = {m0, m1, m2, m3, m4, m5};
  const double* T = mode == TG_BEAMLET_PROPAGATED ? abcd + i * abcd_stride : nullptr;
  out[i] = make_coef(p, T, mode, m, mk(1.0, 0.0), cut);
}

// w = conj(g) over the image, then kRun zeros of tail padding
__global__ __launch_bounds__(256) void conj_pad_kernel(const float2* __restrict__ g, int64_t npix,
                                                       float2* __restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < npix) {
    const float2 v = g[i];
    w[i] = make_float2(v.x, -v.y);
  } else if (i < npix + kRun) {
    w[i] = make_float2(0.0f, 0.0f);
  }
}

constexpr int kBeamletsPerMomentBlock = 4;  // one wavefront each

__global__ __launch_bounds__(256) void beamlet_moment_kernel(const tg_beamlet_coef* __restrict__ unit, int64_t n,
                                                             int32_t H, int32_t W, const float2* __restrict__ w,
                                                             double* __restrict__ moments) {
  const int lane = threadIdx.x & 63;
  // one beamlet per wavefront: its index and record are wave-uniform
  const int64_t b = (int64_t)blockIdx.x * kBeamletsPerMomentBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (b >= n) return;  // whole wavefronts leave; no block barrier below
  double M[kMoments];
  beamlet_moments<1>(unit[b], H, W, w, lane, M);
#pragma unroll
  for (int k = 0; k < kMoments; ++k) M[k] = wave_sum_f64(M[k]);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < kMoments; ++k) moments[b * kMoments + k] = M[k];
  }
}

__global__ __launch_bounds__(64 * kSharedWaves) void beamlet_moment_shared_kernel(
    const tg_beamlet_coef* __restrict__ unit, int32_t H, int32_t W, const float2* __restrict__ w,
    double* __restrict__ moments) {
  block_moments(unit[blockIdx.x], H, W, w, moments + (int64_t)blockIdx.x * kMoments);
}

// The chain rule of one beamlet (blockIdx.x, lane) along one direction
// (blockIdx.y): a forward-mode pass of the coefficient algebra.  Bound: the
// latency of a few thousand dependent f64 instructions (divisions, square
// roots, sincos), so the 31 directions of a beamlet run side by side: 2,048
// beamlets take 15 us, where all directions in one lane kept 32 wavefronts
// busy for 268 us.  The direction is uniform over a workgroup, so its seeds
// are scalar selects.
__global__ __launch_bounds__(64) void beamlet_grad_kernel(const double* __restrict__ params, int64_t n,
                                                          const double* __restrict__ abcd, int64_t abcd_stride,
                                                          int32_t mode, double m0, double m1, double m2, double m3,
                                                          double m4, double m5, int32_t H, int32_t W,
                                                          const tg_beamlet_coef* __restrict__ unit,
                                                          const double* __restrict__ moments,
                                                          double* __restrict__ grad_params,
                                                          double* __restrict__ grad_abcd) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* p = params + i * TG_BEAMLET_NPARAM;
  const bool prop = mode == TG_BEAMLET_PROPAGATED;
  const double* T = prop ? abcd + i * abcd_stride : nullptr;
  const double m[6] = {m0, m1, m2, m3, m4, m5};
  float fcx, fcy;
  centre_pixel(unit[i], H, W, fcx, fcy);
  const double pcx = fcx, pcy = fcy;
  const double* Mo = moments + i * kMoments;
  const cd S0 = mk(Mo[0], Mo[1]), Su = mk(Mo[2], Mo[3]), Sv = mk(Mo[4], Mo[5]);
  const cd Suu = mk(Mo[6], Mo[7]), Suv = mk(Mo[8], Mo[9]), Svv = mk(Mo[10], Mo[11]);
  // G_k = sum W exp(Phi') m_k, monomials of (px, py) = (pcx + u, pcy + v)
  cd G[6];
  G[0] = add(add(Suu, scl(Su, 2.0 * pcx)), scl(S0, pcx * pcx));
  G[1] = add(add(Suv, scl(Su, pcy)), add(scl(Sv, pcx), scl(S0, pcx * pcy)));
  G[2] = add(add(Svv, scl(Sv, 2.0 * pcy)), scl(S0, pcy * pcy));
  G[3] = add(Su, scl(S0, pcx));
  G[4] = add(Sv, scl(S0, pcy));
  G[5] = S0;
  const double ar = p[5], ai = p[6];
  double* gp = grad_params + i * TG_BEAMLET_NPARAM;
  // directions: parameter columns 0-4 and 7-12, then ray-transfer entries 0-19
  const int q = blockIdx.y;
  if (q == 0) {
    gp[5] = S0.re;   // u = amp exp(Phi'): dL/d amp_re = Re sum W exp(Phi')
    gp[6] = -S0.im;  //                    dL/d amp_im = Re(i sum W exp(Phi'))
    gp[13] = gp[14] = gp[15] = 0.0;
    if (grad_abcd) {
      for (int e = prop ? 20 : 0; e < 25; ++e) grad_abcd[i * 25 + e] = 0.0;
    }
  }
  const int col = q < 5 ? q : (q < 11 ? q + 2 : -1);
  const int ent = q < 11 ? -1 : q - 11;
  dual pd[13], Td[25];
#pragma unroll
  for (int k = 0; k < 13; ++k) pd[k] = dual(p[k], k == col ? 1.0 : 0.0);
  if (prop) {
#pragma unroll
    for (int e = 0; e < 25; ++e) Td[e] = dual(T[e], e == ent ? 1.0 : 0.0);
  }
  cx<dual> d6[6];
  phi_coefficients<dual>(pd, Td, mode, m, mk(dual(1.0), dual(0.0)), d6);
  double sr = 0.0, si = 0.0;  // sum_k G_k dc_k
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    sr += G[k].re * d6[k].re.t - G[k].im * d6[k].im.t;
    si += G[k].re * d6[k].im.t + G[k].im * d6[k].re.t;
  }
  const double g = ar * sr - ai * si;  // Re[amp sum_k G_k dc_k]
  if (col >= 0)
    gp[col] = g;
  else
    grad_abcd[i * 25 + ent] = g;
}

int splits_for(int64_t n, int64_t H, int64_t W) {
  const int64_t key[4] = {n, H, W, 0};
  int32_t tuned = 0;
  if (tg::tune_lookup(TG_TUNE_BEAMLET_SPLITS, key, tuned)) {
    int64_t s = tuned;
    if (s > 128) s = 128;
    if (s > n && n > 0) s = n;
    if (s < 1) s = 1;
    return (int)s;
  }
  const int64_t ntiles = tg::cdiv(H, kTileH) * tg::cdiv(W, kTileW);
  // Few beamlets: about six workgroups of 64x64 pixels a CU, down to where the
  // slices' own cost takes over: a start, and a partial image each, so slices of
  // sqrt(n) beamlets, and of more above 60,000 pixels.  The sum's kernels, 256
  // beamlets a slice as a rule / slices of sqrt(n) whatever the pixels / this
  // one: tilted 64 on 600 x 612 40 / 34 / 27 us, 300 on 600^2 79 / 46 / 38 (with a
  // 4-sigma cut 39 / 44 / 32), 2,048 on 500 x 612 141 / 75 / 78, 500 on 300^2
  // 257 / 38 / 42, 300 on 100^2 166 / 27 / 29; separable 30 on 1024^2 24 / 61 / 29,
  // 64 on 600 x 612 19 / 48 / 27.  (A sixth of that, from 10,000 pixels on: 2,048
  // tilted ones 120, 500 on 300^2 70.)
  // Many separable ones: whole rounds of the matrix-core kernel's tiles (two
  // workgroups a CU at a time; tiles of uneven weight want some rounds), slices
  // of at least 600.  20,000 on 512^2: 32 slices, a round, 152 us, 39 slices
  // 212; 131,072 on 1024^2: 16 / 32 / 64 / 128 slices 2.50 / 2.15 / 2.15 /
  // 2.30 ms; 50,000 on 1000 x 300 533 / 468 us.
  const double start = std::max(1.0, (double)H * (double)W / 60000.0);
  const int64_t few = std::min<int64_t>(6LL * tg::cu_count() / ntiles, (int64_t)std::sqrt((double)n / start));
  const int64_t tiles = tg::cdiv(H, (int64_t)SepTile::TH) * tg::cdiv(W, (int64_t)SepTile::TW);
  const int64_t slots = 2LL * tg::cu_count();
  const int64_t rounds = std::min<int64_t>(4, (int64_t)((double)n * (double)tiles / (600.0 * (double)slots)));
  int64_t s = std::max(few, rounds * slots / tiles);
  if (s > 128) s = 128;
  if (s < 1) s = 1;
  return (int)s;
}

int64_t sep_tiles(int64_t H, int64_t W) {
  return tg::cdiv(W, (int64_t)SepTile::TW) * tg::cdiv(H, (int64_t)SepTile::TH);
}

// The two sums of separable beamlets: the f16 halves, then the f32 products of
// what they leave.
int launch_sep_sums(const SepTables& tab, int64_t n, int64_t H, int64_t W, int nsplit, const int32_t* flags,
                    float2* ws, hipStream_t s) {
  hipLaunchKernelGGL(beamlet_sum_sep_kernel<SepTile>, dim3((unsigned)(sep_tiles(H, W) * nsplit)),
                     dim3(SepTile::kThreads), 0, s, tab, n, H, W, (int32_t)tg::cdiv(W, (int64_t)SepTile::TW),
                     (int32_t)nsplit, flags, ws);
  TG_LAUNCH_CHECK("beamlet_sum_sep_kernel launch");
  const int64_t ntx = tg::cdiv(W, (int64_t)kTileW), ntiles = ntx * tg::cdiv(H, (int64_t)kTileH);
  hipLaunchKernelGGL(beamlet_sum_wide_kernel, dim3((unsigned)(ntiles * nsplit)), dim3(kThreads), 0, s, tab, n, H, W,
                     (int32_t)ntx, (int32_t)nsplit, flags, ws);
  TG_LAUNCH_CHECK("beamlet_sum_wide_kernel launch");
  return TG_OK;
}

// The recurrence tile sum (beamlet_sum_kernel) for a tile shape
// (tg_tile_shape): one workgroup per (tile, beamlet slice).
int launch_recurrence_sum(int32_t shape, const tg_beamlet_coef* coef, int64_t n, int64_t H, int64_t W, int nsplit,
                          const int32_t* flags, float2* ws, hipStream_t s) {
  const TileDims d = tile_dims(shape);
  const int64_t ntx = tg::cdiv(W, (int64_t)d.w), ntiles = ntx * tg::cdiv(H, (int64_t)d.h);
  TG_REQUIRE(ntiles * nsplit < (int64_t)1 << 31, "tg_beamlet_sum: detector too large");
  const dim3 grid((unsigned)(ntiles * nsplit));
  switch (shape) {
    case TG_TILE_128x32_RUN16:
      hipLaunchKernelGGL((beamlet_sum_kernel<8, 16>), grid, dim3(kThreads), 0, s, coef, n, H, W, (int32_t)ntx,
                         (int32_t)ntiles, (int32_t)nsplit, flags, ws);
      break;
    case TG_TILE_32x128_RUN16:
      hipLaunchKernelGGL((beamlet_sum_kernel<2, 16>), grid, dim3(kThreads), 0, s, coef, n, H, W, (int32_t)ntx,
                         (int32_t)ntiles, (int32_t)nsplit, flags, ws);
      break;
    case TG_TILE_64x32_RUN8:
      hipLaunchKernelGGL((beamlet_sum_kernel<8, 8>), grid, dim3(kThreads), 0, s, coef, n, H, W, (int32_t)ntx,
                         (int32_t)ntiles, (int32_t)nsplit, flags, ws);
      break;
    default:
      hipLaunchKernelGGL((beamlet_sum_kernel<kLanesPerRow, kRun>), grid, dim3(kThreads), 0, s, coef, n, H, W,
                         (int32_t)ntx, (int32_t)ntiles, (int32_t)nsplit, flags, ws);
  }
  TG_LAUNCH_CHECK("beamlet_sum_kernel launch");
  return TG_OK;
}

}  // namespace

extern "C" int tg_beamlet_pack(const tg_beamlet_column* columns, int64_t n, double* params, const double* matrix,
                               double* matrix_out, void* stream) {
  tg::clear_error();
  TG_REQUIRE(n >= 0, "tg_beamlet_pack: negative count");
  TG_REQUIRE((matrix == nullptr) == (matrix_out == nullptr), "tg_beamlet_pack: matrix and matrix_out go together");
  if (n == 0 && matrix == nullptr) return TG_OK;
  TG_REQUIRE(n == 0 || (columns != nullptr && params != nullptr), "tg_beamlet_pack: NULL buffer");
  PackArgs a{};
  for (int c = 0; c < TG_BEAMLET_NCOLUMN && n > 0; ++c) {
    a.col[c] = columns[c];
    TG_REQUIRE(columns[c].type >= TG_COLUMN_VALUE && columns[c].type <= TG_COLUMN_F64,
               "tg_beamlet_pack: column %d has an unknown type %d", c, columns[c].type);
    TG_REQUIRE(columns[c].type == TG_COLUMN_VALUE || columns[c].data != nullptr, "tg_beamlet_pack: column %d is NULL",
               c);
  }
  if (matrix != nullptr) memcpy(a.matrix, matrix, sizeof(a.matrix));
  const int64_t blocks = tg::cdiv(n * TG_BEAMLET_NPARAM, 256);
  hipLaunchKernelGGL(beamlet_pack_kernel, dim3((unsigned)(blocks < 1 ? 1 : blocks > 16384 ? 16384 : blocks)),
                     dim3(256), 0, (hipStream_t)stream, a, n, params, matrix_out);
  TG_LAUNCH_CHECK("beamlet_pack_kernel launch");
  return TG_OK;
}

extern "C" int tg_beamlet_coefficients(const double* params, int64_t n, const double* abcd, int64_t abcd_stride,
                                       int32_t mode, const double* pix2m, double nsigma, tg_beamlet_coef* out,
                                       void* stream) {
  tg::clear_error();
  TG_REQUIRE(n >= 0, "tg_beamlet_coefficients: negative count");
  TG_REQUIRE(mode == TG_BEAMLET_PROPAGATED || mode == TG_BEAMLET_INPUT, "tg_beamlet_coefficients: bad mode");
  TG_REQUIRE(pix2m != nullptr, "tg_beamlet_coefficients: NULL pixel transform");
  if (n == 0) return TG_OK;
  TG_REQUIRE(params != nullptr && out != nullptr, "tg_beamlet_coefficients: NULL buffer");
  TG_REQUIRE(mode == TG_BEAMLET_INPUT || (abcd != nullptr && (abcd_stride == 0 || abcd_stride == 25)),
             "tg_beamlet_coefficients: propagated mode needs abcd with stride 0 or 25");
  const float cut = nsigma > 0.0 ? (float)(nsigma * nsigma) : 80.0f;
  hipLaunchKernelGGL(beamlet_coef_kernel, dim3((unsigned)tg::cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, params,
                     n, abcd, abcd_stride, mode, pix2m[0], pix2m[1], pix2m[2], pix2m[3], pix2m[4], pix2m[5], cut, out);
  TG_LAUNCH_CHECK("beamlet_coef_kernel launch");
  return TG_OK;
}

// Workspace of tg_beamlet_sum: [nsplit, H, W] complex64 slice tiles (padded to
// 256 bytes), the kFlagBlocks path flags, then n separable beamlets' factors.
int64_t slices_bytes(int nsplit, int64_t H, int64_t W) {
  return ((int64_t)nsplit * H * W * (int64_t)sizeof(float2) + 255) / 256 * 256;
}

int64_t sum_workspace_bytes(int nsplit, int64_t n, int64_t H, int64_t W) {
  return slices_bytes(nsplit, H, W) + kFlagBlocks * (int64_t)sizeof(int32_t) + n * kSepBytes;
}

extern "C" int64_t tg_beamlet_sum_workspace(int64_t n, int64_t height, int64_t width) {
  if (n < 0 || height <= 0 || width <= 0) return 0;
  return sum_workspace_bytes(splits_for(n, height, width), n, height, width);
}

extern "C" int tg_beamlet_sum(const tg_beamlet_coef* coef, int64_t n, int64_t height, int64_t width, float* field,
                              void* workspace, int64_t workspace_bytes, void* stream) {
  tg::clear_error();
  TG_REQUIRE(n >= 0 && height > 0 && width > 0, "tg_beamlet_sum: bad sizes");
  TG_REQUIRE(field != nullptr && workspace != nullptr, "tg_beamlet_sum: NULL buffer");
  TG_REQUIRE(n == 0 || coef != nullptr, "tg_beamlet_sum: NULL coefficients");
  TG_REQUIRE(n <= (int64_t)1 << 31, "tg_beamlet_sum: too many beamlets");
  const int nsplit = splits_for(n, height, width);
  const int64_t slices = slices_bytes(nsplit, height, width);
  const int64_t need = sum_workspace_bytes(nsplit, n, height, width);
  TG_REQUIRE(workspace_bytes >= need, "tg_beamlet_sum: workspace %lld bytes < %lld", (long long)workspace_bytes,
             (long long)need);
  int st = TG_OK;
  const int64_t ntx = tg::cdiv(width, kTileW), nty = tg::cdiv(height, kTileH);
  const int64_t ntiles = ntx * nty;
  TG_REQUIRE(ntiles * nsplit < (int64_t)1 << 31, "tg_beamlet_sum: detector too large");
  const int64_t key[4] = {n, height, width, 0};
  int32_t path = TG_BEAMLET_PATH_AUTO;
  tg::tune_lookup(TG_TUNE_BEAMLET_PATH, key, path);
  int32_t* flags = (int32_t*)((char*)workspace + slices);
  const SepTables tab = sep_tables(flags + kFlagBlocks, n);
  // which tile sum runs is decided on the device (no host round trip, so the
  // call stays graph-capturable); the other kernels' workgroups exit at once
  hipLaunchKernelGGL(sep_flag_kernel, dim3(kFlagBlocks), dim3(256), 0, (hipStream_t)stream, coef, n,
                     (int32_t)(path == TG_BEAMLET_PATH_VALU), flags, tab);
  TG_LAUNCH_CHECK("sep_flag_kernel launch");
  st = launch_sep_sums(tab, n, height, width, nsplit, flags, (float2*)workspace, (hipStream_t)stream);
  if (st != TG_OK) return st;
  int32_t shape = TG_TILE_64x64_RUN16;
  tg::tune_lookup(TG_TUNE_TILE_SHAPE, key, shape);
  st = launch_recurrence_sum(shape, coef, n, height, width, nsplit, flags, (float2*)workspace, (hipStream_t)stream);
  if (st != TG_OK) return st;
  const int64_t npix = height * width;
  hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)tg::cdiv(npix, 256)), dim3(256), 0, (hipStream_t)stream,
                     (const float2*)workspace, npix, (int32_t)nsplit, (float2*)field);
  TG_LAUNCH_CHECK("split_sum_kernel launch");
  return TG_OK;
}

extern "C" int64_t tg_beamlet_backward_workspace(int64_t n, int64_t height, int64_t width) {
  if (n < 0 || height <= 0 || width <= 0) return 0;
  auto al = [](int64_t b) { return (b + 255) & ~(int64_t)255; };
  return al(n * (int64_t)sizeof(tg_beamlet_coef)) + al((height * width + kRun) * (int64_t)sizeof(float2)) +
         al(n * kMoments * (int64_t)sizeof(double));
}

extern "C" int tg_beamlet_backward(const double* params, int64_t n, const double* abcd, int64_t abcd_stride,
                                   int32_t mode, const double* pix2m, double nsigma, int64_t height, int64_t width,
                                   const float* grad_field, double* grad_params, double* grad_abcd, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  tg::clear_error();
  TG_REQUIRE(n >= 0 && height > 0 && width > 0, "tg_beamlet_backward: bad sizes");
  TG_REQUIRE(height < ((int64_t)1 << 31) && width < ((int64_t)1 << 31) && height * width < ((int64_t)1 << 40),
             "tg_beamlet_backward: image too large");
  TG_REQUIRE(mode == TG_BEAMLET_PROPAGATED || mode == TG_BEAMLET_INPUT, "tg_beamlet_backward: bad mode");
  TG_REQUIRE(pix2m != nullptr, "tg_beamlet_backward: NULL pixel transform");
  TG_REQUIRE(grad_abcd == nullptr || mode == TG_BEAMLET_PROPAGATED,
             "tg_beamlet_backward: ray-transfer gradients need propagated mode");
  if (n == 0) return TG_OK;
  TG_REQUIRE(params != nullptr && grad_field != nullptr && grad_params != nullptr && workspace != nullptr,
             "tg_beamlet_backward: NULL buffer");
  TG_REQUIRE(mode == TG_BEAMLET_INPUT || (abcd != nullptr && (abcd_stride == 0 || abcd_stride == 25)),
             "tg_beamlet_backward: propagated mode needs abcd with stride 0 or 25");
  TG_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 256 == 0, "tg_beamlet_backward: workspace not 256-byte aligned");
  const int64_t need = tg_beamlet_backward_workspace(n, height, width);
  TG_REQUIRE(workspace_bytes >= need, "tg_beamlet_backward: workspace %lld bytes < %lld", (long long)workspace_bytes,
             (long long)need);
  auto al = [](int64_t b) { return (b + 255) & ~(int64_t)255; };
  char* ws = static_cast<char*>(workspace);
  tg_beamlet_coef* unit = reinterpret_cast<tg_beamlet_coef*>(ws);
  float2* w = reinterpret_cast<float2*>(ws + al(n * (int64_t)sizeof(tg_beamlet_coef)));
  double* moments = reinterpret_cast<double*>(reinterpret_cast<char*>(w) +
                                              al((height * width + kRun) * (int64_t)sizeof(float2)));
  const float cut = nsigma > 0.0 ? (float)(nsigma * nsigma) : 80.0f;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(beamlet_unit_kernel, dim3((unsigned)tg::cdiv(n, 256)), dim3(256), 0, s, params, n, abcd,
                     abcd_stride, mode, pix2m[0], pix2m[1], pix2m[2], pix2m[3], pix2m[4], pix2m[5], cut, unit);
  TG_LAUNCH_CHECK("beamlet_unit_kernel launch");
  const int64_t npix = height * width;
  hipLaunchKernelGGL(conj_pad_kernel, dim3((unsigned)tg::cdiv(npix + kRun, 256)), dim3(256), 0, s,
                     (const float2*)grad_field, npix, w);
  TG_LAUNCH_CHECK("conj_pad_kernel launch");
  if (share_moments(n))
    hipLaunchKernelGGL(beamlet_moment_shared_kernel, dim3((unsigned)n), dim3(64 * kSharedWaves), 0, s, unit,
                       (int32_t)height, (int32_t)width, w, moments);
  else
    hipLaunchKernelGGL(beamlet_moment_kernel, dim3((unsigned)tg::cdiv(n, kBeamletsPerMomentBlock)), dim3(256), 0, s,
                       unit, n, (int32_t)height, (int32_t)width, w, moments);
  TG_LAUNCH_CHECK("beamlet_moment_kernel launch");
  // the 20 ray-transfer directions only where their gradient is wanted
  const unsigned n_dir = grad_abcd != nullptr ? 31 : 11;
  hipLaunchKernelGGL(beamlet_grad_kernel, dim3((unsigned)tg::cdiv(n, 64), n_dir), dim3(64), 0, s, params, n, abcd,
                     abcd_stride, mode, pix2m[0], pix2m[1], pix2m[2], pix2m[3], pix2m[4], pix2m[5], (int32_t)height,
                     (int32_t)width, unit, moments, grad_params, grad_abcd);
  TG_LAUNCH_CHECK("beamlet_grad_kernel launch");
  return TG_OK;
}
