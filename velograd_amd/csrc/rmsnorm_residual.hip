// Fused RMSNorm + residual add, forward and backward, hand-written for gfx950 (CDNA4, wave64).
//
// Math (reference: python/velograd/kernels/fused.py:28-66):
//   forward   h = x + residual;  inv_rms = 1 / sqrt(mean(h^2) + eps);  y = (h * inv_rms) * w
//             (the residual-free module form, python/velograd/nn.py:338-355, first floors
//             mean(h^2) at a minimum: see floor_mean_sq)
//   backward  gw = g * w;  m = mean(gw * xhat);  dx = inv_rms * (gw - xhat * m)
//             dweight = sum over rows of g * xhat,  with xhat = h * inv_rms
// Every operation is fp32 and rounds where the NumPy reference rounds (this file is built with
// -ffp-contract=off so no multiply-add pair is fused behind the code's back); stores round to
// nearest even.  Only the order of the row sums differs from NumPy's pairwise summation.  The
// exceptions are the norm + RoPE kernels, whose walks are bound by their vector instructions:
// they fuse multiply-adds explicitly (one rounding where the reference has two).
//
// Kernels
//   fwd_vec_kernel      one row per `tpr` threads (1..16 wave64), `groups` rows per workgroup;
//                       each thread holds NV 16-byte chunks of the row in registers, so every
//                       element moves through HBM exactly once (read x, residual; write h, y).
//   bwd_vec_kernel      persistent: each row slot walks rows slot, slot + S, ... with the next
//                       row's loads in flight while the current row reduces; the weight chunk and
//                       the fp32 dweight column accumulators stay in registers for the whole walk;
//                       each slot finally writes one fp32 partial row (no atomics).
//   bwd_ring_kernel     the same walk for rows of whole 16-byte chunks (some lanes may idle;
//                       2-byte rows of 8n + 4 elements in 8-byte halves) with a ring of three
//                       row buffers (two rows in flight while one reduces) in a branch-free
//                       steady loop, 512-thread workgroups, one per CU: the backward's default
//                       where the rows suit it.
//   fwd_rope_tile_kernel  the forward with the model's interleaved RoPE on y: short tiles of
//                       consecutive positions, the rotation advanced by a recurrence in each.
//   bwd_rope_ring_kernel  its backward (grad_y rotated back, then the norm's backward) in
//                       bwd_ring_kernel's walk, one or two chunks per thread (rows of up to
//                       1024 chunks), one workgroup per CU (two of one chunk and under 512
//                       threads);
//                       bwd_vec_kernel with kRopeG where the rows or positions do not suit it.
//   dweight_reduce      stage 2: sums the partial rows in a fixed order -> dweight[dim].
//   *_generic_kernel    any dim and any alignment: the same arithmetic with scalar accesses.
// Row sums: DPP inside each 16-lane row of the wave, readlane across the four rows, LDS only
// across the waves that share a row; every order is fixed, so results are bitwise reproducible.

#include <mutex>
#include <type_traits>

#include "common.h"
#include "fp8_e4m3.h"
#include "mx_formats.h"

#define VG_VERSION_STRING "velograd_amd 0.1.0 fused-rmsnorm-residual gfx950"

namespace {

using namespace vg;
using vg_fp8::inverse_scale;
using vg_fp8::kE4M3Max;
using vg_plan::BwdPlan;
using vg_plan::kGenericBlock;
using vg_plan::kMaxNV;
using vg_plan::kMaxWavesPerRow;
using vg_plan::kWave;
using vg_plan::max_block_for_nv;
using vg_plan::RowPlan;
using vg_plan::xcd_item;

// The weight values of one activation chunk (kVec(DT) columns), kept packed in registers: one
// 16-byte vector when the weight has the activation dtype, kVec/4 vectors when it is fp32.
// No weight (NULL) reads as 1.0, which leaves (h * r) * w == h * r and g * w == g exactly.
template <int DT, int WDT>
struct WeightChunk {
  static_assert(WDT == DT || WDT == VELOGRAD_DTYPE_F32, "weight is the activation dtype or fp32");
  static constexpr int kParts = (WDT == DT) ? 1 : Codec<DT>::kVec / 4;
  u32x4 q[kParts];

  __device__ inline void load(const void* w, int64_t col0) {
    if (w == nullptr) {
      // fp32 1.0 in every slot, decoded through the fp32 codec below
#pragma unroll
      for (int i = 0; i < kParts; ++i) q[i] = u32x4{0u, 0u, 0u, 0u};
      return;
    }
#pragma unroll
    for (int i = 0; i < kParts; ++i) q[i] = load16<WDT>(w, col0 + i * Codec<WDT>::kVec);
  }
  // the same from any element of a weight that starts anywhere
  __device__ inline void load_any(const void* w, int64_t col0) {
#pragma unroll
    for (int i = 0; i < kParts; ++i)
      q[i] = load16_any<WDT>(w, col0 + i * Codec<WDT>::kVec);
  }
  __device__ inline void unpack(bool has_w, float* f) const {
    if (!has_w) {
#pragma unroll
      for (int i = 0; i < Codec<DT>::kVec; ++i) f[i] = 1.0f;
      return;
    }
#pragma unroll
    for (int i = 0; i < kParts; ++i) Codec<WDT>::unpack(q[i], f + i * Codec<WDT>::kVec);
  }
};

// Where element `elem` of a stream starts inside its 16-byte line (the generic kernels' aligned
// middle of a row, see fwd_generic_kernel).
__device__ inline uintptr_t row_offset16(const void* base, int64_t elem, int elem_bytes) {
  return (reinterpret_cast<uintptr_t>(base) + (uintptr_t)(elem * elem_bytes)) & 15u;
}

// The 16 bytes at p whatever its 2-byte alignment (`align` = p's offset in its 16-byte line, the
// same on every lane), in the widest loads that alignment allows: the generic kernels' weight
// values for a body chunk, which sits elsewhere in its line than the row's chunk.
__device__ inline u32x4 load16_unaligned(const char* p, uintptr_t align) {
  if (align == 0) return *reinterpret_cast<const u32x4*>(p);
  if ((align & 7) == 0) {
    const u32x2 lo = *reinterpret_cast<const u32x2*>(p);
    const u32x2 hi = *reinterpret_cast<const u32x2*>(p + 8);
    return u32x4{lo.x, lo.y, hi.x, hi.y};
  }
  if ((align & 3) == 0) {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    return u32x4{q[0], q[1], q[2], q[3]};
  }
  const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (uint32_t)h[2 * i] | ((uint32_t)h[2 * i + 1] << 16);
  return v;
}

// The weight values of the body chunk at element j (Codec<DT>::kVec of them) into f, for the
// generic kernels: one to four loads of 16 bytes' worth instead of one per element.  `align` is
// the weight's offset inside its 16-byte line at the row's first body element (uniform).
template <int DT, int WDT>
__device__ inline void weight_run(const void* w, int64_t j, uintptr_t align, float* f) {
  constexpr int kParts = (Codec<DT>::kVec * Codec<WDT>::kBytes) / 16;
  const char* p = static_cast<const char*>(w) + j * Codec<WDT>::kBytes;
#pragma unroll
  for (int q = 0; q < kParts; ++q)
    Codec<WDT>::unpack(load16_unaligned(p + 16 * q, align), f + q * Codec<WDT>::kVec);
}

// Largest |value| over the `tpr` threads of row group `grp`, on the bit patterns of |value|
// (sign cleared): for non-negative IEEE floats the unsigned order is the numeric order, and
// every NaN pattern lies above +inf, so a NaN anywhere in the row wins (NaN propagates).
template <int CTRL>
__device__ inline uint32_t dpp_move_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}

__device__ inline uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }

__device__ inline uint32_t row_max_abs_bits(uint32_t v, int tpr, int grp, uint32_t* red) {
  v = umax(v, dpp_move_u32<0xB1>(v));
  v = umax(v, dpp_move_u32<0x4E>(v));
  v = umax(v, dpp_move_u32<0x124>(v));
  v = umax(v, dpp_move_u32<0x128>(v));
  v = umax(umax((uint32_t)__builtin_amdgcn_readlane((int)v, 0),
                (uint32_t)__builtin_amdgcn_readlane((int)v, 16)),
           umax((uint32_t)__builtin_amdgcn_readlane((int)v, 32),
                (uint32_t)__builtin_amdgcn_readlane((int)v, 48)));
  if (tpr > kWave) {
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    const int wpr = tpr / kWave;
    const uint32_t* p = red + grp * wpr;
    uint32_t t = p[0];
    for (int i = 1; i < wpr; ++i) t = umax(t, p[i]);
    v = t;
  }
  return v;
}

// ------------------------------------------------------------------------------------------
// fp8 E4M3 codes on the device.  gfx950's v_cvt_pk_fp8_f32 converts two fp32 values to OCP
// e4m3fn with round to nearest even (one instruction per pair instead of the integer steps of
// vg_fp8::e4m3_encode, which the CPU tests pin against the oracle).  It is not saturating, and
// needs not be here: the inputs are y * (1 / scale) with |y| <= amax, so |y * inv| <=
// 448 * (1 + 2^-22), which rounds to 448 (values up to the 464 midpoint do); the exception,
// inv = 1 for a row whose scale is below the smallest normal float, has |y| < 2^-117.  NaN
// converts to a NaN code.  Build with -DVG_FP8_SOFT_ENCODE=1 to use the integer encoder.
// ------------------------------------------------------------------------------------------
#ifndef VG_FP8_SOFT_ENCODE
#define VG_FP8_SOFT_ENCODE 0
#endif

__device__ inline uint32_t e4m3x4(float a, float b, float c, float d) {
#if VG_FP8_SOFT_ENCODE
  return vg_fp8::e4m3_encode(a) | (vg_fp8::e4m3_encode(b) << 8) | (vg_fp8::e4m3_encode(c) << 16) |
         (vg_fp8::e4m3_encode(d) << 24);
#else
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, lo, true);
#endif
}

__device__ inline uint32_t e4m3x1(float a) {
#if VG_FP8_SOFT_ENCODE
  return vg_fp8::e4m3_encode(a);
#else
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, a, 0, false) & 0xffu;
#endif
}

// fp4 E2M1 nibbles on the device: gfx950's v_cvt_scalef32_pk_fp4_f32 converts two fp32 values
// divided by a scale to E2M1, round to nearest even, saturating, the first value in the low
// nibble of the selected byte (checked against the oracle's nearest-value encoder on every
// midpoint and a dense sweep at scales 0.5..4).  The block factor 2^-s is applied by an exact
// multiplication first and the instruction's scale is 1.  Build with -DVG_FP4_SOFT_ENCODE=1 to
// use vg_mx::e2m1_encode (the comparison chain the CPU tests pin) instead.
#ifndef VG_FP4_SOFT_ENCODE
#define VG_FP4_SOFT_ENCODE 0
#endif

template <int SEL>
__device__ inline uint32_t e2m1x2(uint32_t old, float a, float b) {
#if VG_FP4_SOFT_ENCODE
  return old | ((vg_mx::e2m1_encode(a) | (vg_mx::e2m1_encode(b) << 4)) << (8 * SEL));
#else
  return (uint32_t)__builtin_amdgcn_cvt_scalef32_pk_fp4_f32(old, a, b, 1.0f, SEL);
#endif
}

// The reference module's `mean_sq = max(1e-12, sum(x ** 2) / dim)` (python/velograd/nn.py:349),
// for a floor given > 0.  Python's max keeps its first argument unless the second compares
// greater, so a NaN mean square becomes the floor there, and here.  floor == 0 (the fused
// functions, which have no clamp, fused.py:41-42) leaves mean_sq untouched, NaN included.
__device__ __forceinline__ float floor_mean_sq(float mean_sq, float floor) {
  return (floor > 0.0f && !(mean_sq > floor)) ? floor : mean_sq;
}

// ------------------------------------------------------------------------------------------
// Kernel arguments.
// ------------------------------------------------------------------------------------------
struct FwdArgs {
  const void* x;
  const void* res;
  const void* w;
  void* y;          // activation dtype, or fp8 e4m3 codes (one byte each) for the fp8 epilogue
  void* h;
  float* inv_rms;
  float* y_scale;   // fp8 epilogue: per-row dequantisation scale amax(|y|) / 448
  uint8_t* mx_scale;  // MX epilogues: E8M0 scale codes, one per 32 elements of a row
  int64_t ld_mx;      // row stride of mx_scale in bytes
  int64_t rows;
  int64_t ld_x, ld_res, ld_y, ld_h;
  int32_t dim;
  int32_t tpr;
  float eps;
  float ms_floor;   // > 0: floor on mean(h^2) before eps (the reference module's clamp)
  int64_t rope_seq;       // kOutRopeI: positions per outer index (row position = row % rope_seq)
  int32_t rope_half;      // kOutRopeI: dim / 2
  int32_t run_log2;       // log2 of the workgroups of consecutive rows one XCD takes (xcd_item)
  float rope_c_hi, rope_c_lo;  // kOutRopeI: log2(base) / half as an unevaluated float sum
  double rope_log2_step, rope_ratio;  // kOutRopeI: -log2(base) / half and 2 to it
  bool rope_small_step;       // kOutRopeI: base >= 1, so a position's step is 1 radian at most
  bool rope_across;           // kOutRopeI: a tile is one position of consecutive sequences
  double rope_step_rad;       // kOutRopeI: 2 pi, or 0 across sequences
};

struct BwdArgs {
  const void* g;
  const void* saved;
  const void* w;
  const float* inv_rms;
  const void* gh;  // residual-stream gradient added to dx, or null
  void* dx;
  void* dres;
  float* partial;  // [slots, dim] fp32 or null
  int64_t rows;
  int64_t ld_g, ld_s, ld_gh, ld_dx, ld_dres;
  int32_t dim;
  int32_t tpr;
  int32_t iters;  // rows visited per slot = ceil(rows / slots)
  int64_t rope_seq;            // kRopeG: positions per outer index (row position = row % rope_seq)
  float rope_c_hi, rope_c_lo;  // kRopeG: log2(base) / half as an unevaluated float sum
  double rope_ratio;           // kRopeG: base^(-2/dim), one pair's frequency over the one before
  bool rope_back;              // the ring: a walk past a sequence's end returns to its first position
  int32_t rope_anchor;         // the ring: rows between evaluations of a rotation afresh
};

// Output modes of the forward kernels.
constexpr int kOutDtype = 0;   // y in the activation dtype
constexpr int kOutFp8Row = 1;  // y as e4m3 codes with one fp32 scale per row
constexpr int kOutMxE4M3 = 2;  // MXFP8: e4m3 codes, one E8M0 scale per 32 elements
constexpr int kOutMxE2M1 = 3;  // MXFP4: e2m1 nibbles (two per byte), one E8M0 scale per 32
constexpr int kOutRopeI = 4;   // y rotated by the reference model's interleaved RoPE
constexpr int kOutDtypeLateH = 5;  // as kOutDtype, with h stored after the row reduction
// The reference model's RoPE applied to y in registers (python/velograd/functional.py:287-315;
// models/llama.py:48-49 rotates the normalised attention input): the pair (y_2i, y_2i+1) of a
// row at position pos turns by pos * freq_i, freq_i = base^(-2i/dim) = 2^-(i * c) with
// c = log2(base) / half.  c arrives as c_hi + c_lo (from double on the host); freq_i and the
// angle pos * freq_i are formed in double, as the reference's Python floats are, and the angle is
// reduced exactly to [-1/2, 1/2] revolutions before a float32 cos and sin, so they are within
// a few float32 ulps at any position (a float32 angle would carry pos * freq_i * 2^-24 radians of
// error: 0.016 rad at position 2.6e5).
constexpr double kInv2PiD = 0.159154943091895335768883763372514362;
constexpr double kTwoPiD = 6.283185307179586476925286766559005768;
__device__ __forceinline__ double rope_freq(int i, float c_hi, float c_lo) {
  return exp2(-(double)i * ((double)c_hi + (double)c_lo));
}

// A double angle in revolutions reduced exactly to [-1/2, 1/2], and the cos and sin of such an
// angle: the quarter turn nearest to it, then the Taylor series of sin and cos over the +-1/8
// turn that is left (1.02 ulp at most against 64 bits over 20 million angles; the leading
// pi/2 in two floats).
__device__ __forceinline__ float rope_frac(double rev) { return (float)(rev - rint(rev)); }
__device__ __forceinline__ void cos_sin_turn(float rev, float& c, float& s) {
  const float t = 4.0f * rev;
  const float k = rintf(t);
  const float f = t - k;  // quarter turns, exact
  const float z = f * f;
  float ps = 0.00016044118478735975f;  // (pi/2)^n / n!, alternating
  ps = fmaf(ps, z, -0.004681754135318687f);
  ps = fmaf(ps, z, 0.07969262624616703f);
  ps = fmaf(ps, z, -0.6459640975062462f);
  ps = fmaf(ps, z, -4.371139000186241e-8f);  // pi/2 - (float)(pi/2)
  const float s0 = fmaf(f, 1.5707963267948966f, f * ps);
  float pc = -2.5202042373060596e-05f;
  pc = fmaf(pc, z, 0.0009192602748394263f);
  pc = fmaf(pc, z, -0.020863480763352957f);
  pc = fmaf(pc, z, 0.253669507901048f);
  pc = fmaf(pc, z, -1.2337005501361697f);
  const float c0 = fmaf(pc, z, 1.0f);
  const int q = (int)k;
  const bool odd = (q & 1) != 0;
  s = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, odd ? c0 : s0) ^
                                    ((uint32_t)(q & 2) << 30));
  c = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, odd ? s0 : c0) ^
                                    ((uint32_t)((q + 1) & 2) << 30));
}

// cos and sin of pair i's angle at position pos.
__device__ __forceinline__ void rope_cos_sin(int64_t pos, int i, float c_hi, float c_lo, float& c,
                                             float& s) {
  cos_sin_turn(rope_frac((double)pos * rope_freq(i, c_hi, c_lo) * kInv2PiD), c, s);
}

// The frequencies of a thread's pairs in a strided loop (pairs i0, i0 + stride, ...): the first
// from exp2, each next one the previous times base^(-2 stride / dim), in double (a few double
// ulps over a row, far below the float32 rotation's rounding), so the generic kernels pay one
// double exp2 per row and thread instead of one per pair.
struct RopeFreqWalk {
  double f, ratio;
  __device__ RopeFreqWalk(int i0, int stride, float c_hi, float c_lo) {
    const double c = (double)c_hi + (double)c_lo;
    f = exp2(-(double)i0 * c);
    ratio = exp2(-(double)stride * c);
  }
  __device__ double next() {
    const double v = f;
    f *= ratio;
    return v;
  }
};

// cos and sin at position pos of the pair whose frequency is fr (as rope_cos_sin)
__device__ __forceinline__ void rope_cos_sin_f(int64_t pos, double fr, float& c, float& s) {
  cos_sin_turn(rope_frac((double)pos * fr * kInv2PiD), c, s);
}

// cos and sin of |x| <= 1 in double by their Taylor series through x^14 and x^13 (truncation below
// 1e-12).
__device__ __forceinline__ void cos_sin_small_d(double x, double& c, double& s) {
  const double z = x * x;
  double ps = 1.0 / 6227020800.0;
  ps = fma(ps, z, -1.0 / 39916800.0);
  ps = fma(ps, z, 1.0 / 362880.0);
  ps = fma(ps, z, -1.0 / 5040.0);
  ps = fma(ps, z, 1.0 / 120.0);
  ps = fma(ps, z, -1.0 / 6.0);
  s = fma(x * z, ps, x);
  double pc = -1.0 / 87178291200.0;
  pc = fma(pc, z, 1.0 / 479001600.0);
  pc = fma(pc, z, -1.0 / 3628800.0);
  pc = fma(pc, z, 1.0 / 40320.0);
  pc = fma(pc, z, -1.0 / 720.0);
  pc = fma(pc, z, 1.0 / 24.0);
  pc = fma(pc, z, -0.5);
  c = fma(z, pc, 1.0);
}

// cos and sin of 2 pi rev in double, |rev| <= 1/2: Taylor series of an eighth of the angle
// (|x| <= pi/8: truncation below 1e-17), doubled three times.
__device__ __forceinline__ void cos_sin_turn_d(double rev, double& c, double& s) {
  const double x = rev * 0.78539816339744830961566084581987572;  // 2 pi / 8
  const double z = x * x;
  double ps = -1.0 / 1307674368000.0;
  ps = fma(ps, z, 1.0 / 6227020800.0);
  ps = fma(ps, z, -1.0 / 39916800.0);
  ps = fma(ps, z, 1.0 / 362880.0);
  ps = fma(ps, z, -1.0 / 5040.0);
  ps = fma(ps, z, 1.0 / 120.0);
  ps = fma(ps, z, -1.0 / 6.0);
  s = fma(x * z, ps, x);
  double pc = 1.0 / 20922789888000.0;  // cos x - 1
  pc = fma(pc, z, -1.0 / 87178291200.0);
  pc = fma(pc, z, 1.0 / 479001600.0);
  pc = fma(pc, z, -1.0 / 3628800.0);
  pc = fma(pc, z, 1.0 / 40320.0);
  pc = fma(pc, z, -1.0 / 720.0);
  pc = fma(pc, z, 1.0 / 24.0);
  pc = fma(pc, z, -0.5);
  pc = pc * z;
#pragma unroll
  for (int i = 0; i < 3; ++i) {  // v = cos - 1: v(2x) = 2 v (2 + v), sin(2x) = 2 sin (1 + v)
    s = 2.0 * fma(s, pc, s);
    pc = 2.0 * pc * (2.0 + pc);
  }
  c = 1.0 + pc;
}

// Largest value over aligned groups of L lanes (L = 4 or 8), on every lane of the group.
template <int L>
__device__ inline uint32_t lane_group_max(uint32_t v) {
  static_assert(L == 4 || L == 8, "MX blocks span 4 or 8 lanes");
  v = umax(v, dpp_move_u32<0xB1>(v));     // quad_perm [1,0,3,2]
  v = umax(v, dpp_move_u32<0x4E>(v));     // quad_perm [2,3,0,1]
  if constexpr (L == 8) v = umax(v, dpp_move_u32<0x141>(v));  // row_half_mirror
  return v;
}

// Quantised codes of one chunk at p: aligned to their own size, or (ANY) at any byte.
template <bool ANY, typename T>
__device__ inline void store_codes(uint8_t* p, const T v) {
  if constexpr (ANY) {
    typedef T AnyT __attribute__((aligned(1)));
    __builtin_nontemporal_store((AnyT)v, reinterpret_cast<AnyT*>(p));
  } else {
    __builtin_nontemporal_store(v, reinterpret_cast<T*>(p));
  }
}

// ------------------------------------------------------------------------------------------
// Forward, register-resident row.
// ------------------------------------------------------------------------------------------
// OUT selects the epilogue.  kOutFp8Row: y is not stored in the activation dtype; a second row
// reduction finds amax = max |y| over the row (fp32 y, before any rounding), the row's scale is
// amax / 448, and y * (1 / scale) is stored as e4m3 codes: 8 bytes per bf16/fp16 chunk, 4 per
// fp32 chunk.  kOutMxE4M3 / kOutMxE2M1: the 32 elements of an MX block are the chunks of 4
// (bf16/fp16) or 8 (fp32) consecutive lanes, whose amax is reduced with DPP inside the group.
// ANY: rows of any length from one chunk up whose streams start at any element.  The chunks start
// at the row's first 16-byte boundary of x (the MX blocks at the row's start), and the at most
// 2 V - 2 elements before and after them go one to a lane.  Streams that sit elsewhere in their
// 16-byte lines than x are read and written unaligned.
constexpr int kRowsChunks = 0;    // whole aligned 16-byte chunks
constexpr int kRowsAnyRes = 1;    // ANY, with a residual
constexpr int kRowsAnyNoRes = 2;  // ANY, without
template <int DT, int WDT, int NV, int OUT, int ROWS = kRowsChunks>
__global__ __launch_bounds__(max_block_for_nv(NV)) void fwd_vec_kernel(const FwdArgs a) {
  using C = Codec<DT>;
  constexpr int V = C::kVec;
  constexpr bool ANY = ROWS != kRowsChunks;
  __shared__ float red[kMaxWavesPerRow];

  const int tpr = a.tpr;
  const int grp = threadIdx.x / tpr;
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t row = (int64_t)xcd_item(blockIdx.x, gridDim.x, a.run_log2) * groups + grp;
  const bool row_ok = row < a.rows;
  constexpr bool MX = OUT == kOutMxE4M3 || OUT == kOutMxE2M1;
  int head = 0;
  if constexpr (ANY && !MX) {
    const int off = (int)row_offset16(a.x, row * a.ld_x, C::kBytes);
    head = min(((16 - off) & 15) / C::kBytes, a.dim);
  }
  const int nchunk = (a.dim - head) / V;
  // (known at compile time for ANY: a branch on it would put waits between the loads)
  const bool has_res = ANY ? ROWS == kRowsAnyRes : a.res != nullptr;
  const bool has_w = a.w != nullptr;
  auto col_of = [&](int c) -> int { return head + c * V; };
  auto load_chunk = [&](const void* base, int64_t e) -> u32x4 {
    if constexpr (ANY) return load16_any_stream<DT>(base, e);
    else return load16_stream<DT>(base, e);
  };
  auto store_chunk = [&](void* base, int64_t e, const u32x4 v) {
    if constexpr (ANY) store16_any_stream<DT>(base, e, v);
    else store16_stream<DT>(base, e, v);
  };

  // Only the packed 16-byte chunks stay live across the row reduction; fp32 h is formed again
  // after it (the same single fp32 add, so the same bits), which keeps VGPRs low enough for
  // up to 8 chunks per thread.
  u32x4 xv[NV], rv[NV];
  WeightChunk<DT, WDT> wc[NV];
  // ANY: the lane's element outside the chunks
  constexpr bool kAllStray = ROWS == kRowsAnyNoRes && (MX || OUT == kOutFp8Row);
  const bool own_s = ANY && row_ok && lt < a.dim - nchunk * V;
  const int j_s = lt < head ? lt : lt + nchunk * V;
  typename C::Raw x_raw{}, r_raw{};
  typename Codec<WDT>::Raw w_raw{};
  // No wait may fall between these loads (16384 x 4095 bf16 100.9 us with one, 94.2 without; two
  // chunks a thread: MXFP4 32768 x 1024 39.4 / 36.8, without a residual 16384 x 4096 48.6 / 45.1),
  // so they stand under no per-lane condition, which would merge each value with the one that the
  // other lanes keep: a lane without a chunk reads the row's last columns, a row past the end the
  // last row.
  const int64_t rw = row_ok ? row : a.rows - 1;
  if constexpr (ANY) {
    // The raw elements come first and are decoded at the row sum; what is absent is read from x.
    // Quantised outputs without a residual, short of loads, take them on every lane for the same
    // reason (16384 x 255 fp8 9.6 / 9.3 us); the others ran up to 2% slower that way (more
    // requests).
    if (kAllStray || own_s) {
      const int j = own_s ? j_s : 0;
      x_raw = static_cast<const typename C::Raw*>(a.x)[rw * a.ld_x + j];
      if (has_res) r_raw = static_cast<const typename C::Raw*>(a.res)[rw * a.ld_res + j];
      w_raw = static_cast<const typename Codec<WDT>::Raw*>(has_w ? a.w : a.x)[has_w ? j : 0];
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int col = min(col_of(lt + k * tpr), a.dim - V);
      xv[k] = load_chunk(a.x, rw * a.ld_x + col);
      if (has_res) rv[k] = load_chunk(a.res, rw * a.ld_res + col);
      if (has_w) wc[k].load_any(a.w, col);
    }
  } else {
    int col[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      col[k] = min(lt + k * tpr, nchunk - 1) * V;
      xv[k] = load_chunk(a.x, rw * a.ld_x + col[k]);
      if (has_res) rv[k] = load_chunk(a.res, rw * a.ld_res + col[k]);
    }
    auto load_w = [&]() {
      if (!has_w) return;
#pragma unroll
      for (int k = 0; k < NV; ++k) wc[k].load(a.w, col[k]);
    };
    // An fp32 weight beside 2-byte activations is twice their bytes, all from L2: with two or more
    // chunks a thread it goes out after the wait, while the row is summed (fp32 weight, with the
    // others / after, us: without a residual 8192 x 12288 82.5 / 71.9, 16384 x 4096 49.6 / 47.8, to fp8
    // 8192 x 16384 208.8 / 195.5, 16384 x 5120 101.2 / 97.3; 32768 x 1024 39.4 / 39.9).
    constexpr bool kLateW = WeightChunk<DT, WDT>::kParts > 1 && NV > 1;
    if constexpr (!kLateW) load_w();
    // one wait for all of them, before the first store of h: a wait after that, at the next
    // chunk's first use, would be for the store as well
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      forget(xv[k]);
      forget(rv[k]);
    }
    if constexpr (kLateW) load_w();
  }

  auto make_h = [&](int k, float* hf) {
    C::unpack(xv[k], hf);
    if (has_res) {
      float rf[V];
      C::unpack(rv[k], rf);
#pragma unroll
      for (int i = 0; i < V; ++i) hf[i] = hf[i] + rf[i];
    }
  };

  const bool write_h = has_res && a.h != nullptr;
  constexpr bool kLateH = OUT == kOutDtypeLateH;
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float hf[V];
    make_h(k, hf);
    const int c = lt + k * tpr;
    if constexpr (ANY) {
      float p = 0.0f;
#pragma unroll
      for (int i = 0; i < V; ++i) p += hf[i] * hf[i];
      ss += c < nchunk ? p : 0.0f;
    } else {
      float t = ss;
#pragma unroll
      for (int i = 0; i < V; ++i) t += hf[i] * hf[i];
      ss = c < nchunk ? t : ss;
    }
    if (!kLateH && write_h && row_ok && c < nchunk)
      store_chunk(a.h, row * a.ld_h + col_of(c), C::pack(hf));
  }

  float h_s = 0.0f, w_s = 1.0f;
  if constexpr (ANY) {
    asm volatile("" : "+v"(x_raw), "+v"(r_raw), "+v"(w_raw));  // no decoding before this point
    h_s = C::decode1(x_raw);
    if (has_res) h_s = h_s + C::decode1(r_raw);
    if (has_w) w_s = Codec<WDT>::decode1(w_raw);
    ss += own_s ? h_s * h_s : 0.0f;
    if (write_h && own_s) C::store1(a.h, row * a.ld_h + j_s, h_s);
  }
  ss = row_sum(ss, tpr, grp, red);
  const float mean_sq = floor_mean_sq(ss / (float)a.dim, a.ms_floor);
  const float r = 1.0f / __builtin_sqrtf(mean_sq + a.eps);
  if (row_ok && lt == 0 && a.inv_rms != nullptr) a.inv_rms[row] = r;

#pragma unroll
  for (int k = 0; k < NV; ++k) {
    forget(xv[k]);
    forget(rv[k]);
#pragma unroll
    for (int i = 0; i < WeightChunk<DT, WDT>::kParts; ++i) forget(wc[k].q[i]);
  }
  auto make_y = [&](int k, float* yf) {
    float hf[V], wf[V];
    make_h(k, hf);
    wc[k].unpack(has_w, wf);
#pragma unroll
    for (int i = 0; i < V; ++i) yf[i] = (hf[i] * r) * wf[i];
  };

  static_assert(OUT != kOutRopeI, "the RoPE output runs in fwd_rope_tile_kernel");
  if constexpr (OUT == kOutDtype || OUT == kOutDtypeLateH) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      if (row_ok && c < nchunk) {
        if (kLateH && write_h) {
          float hf[V];
          make_h(k, hf);
          store_chunk(a.h, row * a.ld_h + col_of(c), C::pack(hf));
        }
        float yf[V];
        make_y(k, yf);
        store_chunk(a.y, row * a.ld_y + col_of(c), C::pack(yf));
      }
    }
    if constexpr (ANY) {
      if (own_s) C::store1(a.y, row * a.ld_y + j_s, (h_s * r) * w_s);
    }
  } else if constexpr (MX) {
    constexpr int kEmax = OUT == kOutMxE4M3 ? vg_mx::kEmaxE4M3 : vg_mx::kEmaxE2M1;
    constexpr int kLanes = vg_mx::kBlock / V;  // lanes per MX block
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      float yf[V];
      make_y(k, yf);
      uint32_t am = 0;
#pragma unroll
      for (int i = 0; i < V; ++i) am = umax(am, __builtin_bit_cast(uint32_t, yf[i]) & 0x7fffffffu);
      am = lane_group_max<kLanes>(am);  // every lane, before any divergence
      if (row_ok && c < nchunk) {
        const bool finite = am < 0x7f800000u;
        const float f = finite ? vg_mx::inverse_scale(vg_mx::shared_exp(am, kEmax)) : 0.0f;
        uint8_t* dst = static_cast<uint8_t*>(a.y) + row * a.ld_y;
        if constexpr (OUT == kOutMxE4M3) {
          uint32_t words[V / 4];
#pragma unroll
          for (int j = 0; j < V / 4; ++j) {
            float q[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
              q[t] = __builtin_fminf(__builtin_fmaxf(yf[4 * j + t] * f, -kE4M3Max), kE4M3Max);
            words[j] = finite ? e4m3x4(q[0], q[1], q[2], q[3]) : 0u;
          }
          if constexpr (V == 8) {
            const u32x2 w2 = {words[0], words[1]};
            store_codes<ANY>(dst + (int64_t)c * V, w2);
          } else {
            store_codes<ANY>(dst + (int64_t)c * V, words[0]);
          }
        } else {
          uint32_t word = 0;
          word = e2m1x2<0>(word, yf[0] * f, yf[1] * f);
          word = e2m1x2<1>(word, yf[2] * f, yf[3] * f);
          if constexpr (V == 8) {
            word = e2m1x2<2>(word, yf[4] * f, yf[5] * f);
            word = e2m1x2<3>(word, yf[6] * f, yf[7] * f);
          }
          if (!finite) word = 0;
          if constexpr (V == 8) {
            store_codes<ANY>(dst + (int64_t)c * 4, word);
          } else {
            store_codes<ANY>(dst + (int64_t)c * 2, (uint16_t)word);
          }
        }
        if (lt % kLanes == 0)
          a.mx_scale[row * a.ld_mx + c / kLanes] = (uint8_t)vg_mx::scale_code(am, kEmax);
      }
    }
  } else {
    // y stays in registers from the amax pass to the encoding (NV * V floats).
    __shared__ uint32_t red_max[kMaxWavesPerRow];
    float yf[NV][V];
    uint32_t am = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      make_y(k, yf[k]);
      if (row_ok && c < nchunk) {
#pragma unroll
        for (int i = 0; i < V; ++i)
          am = umax(am, __builtin_bit_cast(uint32_t, yf[k][i]) & 0x7fffffffu);
      }
    }
    const float y_s = (h_s * r) * w_s;
    if constexpr (ANY) {
      if (own_s) am = umax(am, __builtin_bit_cast(uint32_t, y_s) & 0x7fffffffu);
    }
    am = row_max_abs_bits(am, tpr, grp, red_max);
    const float scale = __builtin_bit_cast(float, am) / kE4M3Max;
    const float inv = inverse_scale(scale);
    if (row_ok && lt == 0) a.y_scale[row] = scale;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      if (row_ok && c < nchunk) {
        uint32_t words[V / 4];
#pragma unroll
        for (int j = 0; j < V / 4; ++j) {
          words[j] = e4m3x4(yf[k][4 * j] * inv, yf[k][4 * j + 1] * inv, yf[k][4 * j + 2] * inv,
                            yf[k][4 * j + 3] * inv);
        }
        uint8_t* dst = static_cast<uint8_t*>(a.y) + row * a.ld_y + col_of(c);
        if constexpr (V == 8) {
          const u32x2 w2 = {words[0], words[1]};
          store_codes<ANY>(dst, w2);
        } else {
          store_codes<ANY>(dst, words[0]);
        }
      }
    }
    if constexpr (ANY) {
      if (own_s) static_cast<uint8_t*>(a.y)[row * a.ld_y + j_s] = (uint8_t)e4m3x1(y_s * inv);
    }
  }
}

// ------------------------------------------------------------------------------------------
// Forward with the model's RoPE on y (kOutRopeI): a one-shot grid of tiles.  A row group takes the R
// rows of a tile (launch_plan.h: rope_tile): consecutive positions of one sequence, or one position
// of consecutive short sequences (a row past the end re-reads the last one and stores nothing): all
// their loads are in flight at once, the rotations are formed while they
// are, one barrier serves the R row sums, and consecutive tiles run on one XCD (xcd_item).
// Angles, as the reference's Python floats form them (functional.py:302-305): pair j turns
// g_j = base^(-2j/dim) / (2 pi) revolutions per position, in double (one exp2 per chunk, its next
// pairs by the double ratio); the tile's first position times g_j in double is reduced exactly to
// [-1/2, 1/2] revolutions before a float cos and sin (cos_sin_turn), and the next positions
// advance that by the step rotation (none across sequences), at most R - 1 times: in float for bf16/fp16 outputs (3
// float32 ulps a step at most, far below their rounding), in double for fp32 ones.
// Short tiles cost trigonometry, which the vector units pay (28 instructions an element at four
// positions), long ones parallelism; a walk of 16 or 32 strided rows per workgroup instead, its
// trigonometry set up once, left most of the chip idle on short tensors and waited at every row.
// Measured (bf16 without residual, that walk / tiles, us): 64 x 4096 16.0 / 3.5, 2048 x 4096 16.7 /
// 8.1, 8192 x 4096 26.9 / 25.4, 16384 x 4096 49.8 / 45.9 (the norm alone 43.7), 16384 x 768 18.6 /
// 11.4, 8192 x 8192 52.1 / 49.9, fp32 8192 x 4096 49.4 / 49.8; with residual and h 16384 x 4096
// 97.4 / 88.2.  Rows of two chunks a thread, whose pairs were each evaluated at every row:
// 8192 x 16384 160 / 111, fp32 8192 x 8192 133 / 107.  Error against 64 bits in fp32: 8.1e-8 both.
// ANY: even rows that are not whole chunks, streams at any element: the row's last chunk begins at
// dim - V, inside the one before it; the columns it shares add nothing and are not stored (4100
// bf16, generic kernel / tiles, 8192 rows: 100 / 28.6 us; 3002 74 / 21.5; 1000, aligned, 16.8 / 7.5).
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int NV, bool RES, int R, bool ANY>
__global__ __launch_bounds__(max_block_for_nv(NV)) void fwd_rope_tile_kernel(const FwdArgs a) {
  using C = Codec<DT>;
  constexpr int V = C::kVec;
  constexpr int P = V / 2;     // pairs per chunk
  constexpr int NP = NV * P;   // pairs per thread
  constexpr int RQ = (R + 3) / 4;  // quads of rows in the second reduction step
  __shared__ float red[kMaxWavesPerRow][4 * RQ];

  const int tpr = a.tpr;
  // a row group is whole waves: its tile and rows are wave-uniform, and so scalar
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / (uint32_t)tpr);
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  // the tile: ns rows, step apart, the first at position s0
  const vg_plan::RopeTile tile =
      vg_plan::rope_tile(xcd_item(blockIdx.x, gridDim.x, a.run_log2) * groups + grp,
                         (uint32_t)a.rows, (uint32_t)a.rope_seq, R, a.rope_across);
  const bool ok = tile.ok;
  const uint32_t s0 = tile.pos;
  const int ns = tile.n;
  const int64_t row0 = tile.first, step = tile.step;
  const bool has_w = a.w != nullptr;
  const int nchunk = ANY ? (a.dim + V - 1) / V : a.dim / V;
  int col[NV];    // first column of the lane's chunks
  bool own[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = lt + k * tpr;
    own[k] = c < nchunk;
    col[k] = min(c * V, a.dim - V);
  }

  u32x4 xv[R][NV], rv[RES ? R : 1][NV];
  WeightChunk<DT, WDT> wc[NV];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t row = row0 + (u < ns ? u : ns - 1) * step;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if constexpr (ANY) {
        xv[u][k] = load16_any_stream<DT>(a.x, row * a.ld_x + col[k]);
        if constexpr (RES) rv[u][k] = load16_any_stream<DT>(a.res, row * a.ld_res + col[k]);
      } else {
        xv[u][k] = load16_stream<DT>(a.x, row * a.ld_x + col[k]);
        if constexpr (RES) rv[u][k] = load16_stream<DT>(a.res, row * a.ld_res + col[k]);
      }
    }
  }
  if (has_w) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if constexpr (ANY) wc[k].load_any(a.w, col[k]);
      else wc[k].load(a.w, col[k]);
    }
  }

  // the rotation of each pair at s0 and its step, while the loads are in flight
  using RotT = std::conditional_t<DT == VELOGRAD_DTYPE_F32, double, float>;
  RotT cr[NP], sr[NP], cs[NP], sn[NP];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double g = exp2((double)(col[k] / 2) * a.rope_log2_step) * kInv2PiD;  // revolutions a position
#pragma unroll
    for (int q = 0; q < P; ++q) {
      const int e = k * P + q;
      float c0, s0f;
      cos_sin_turn(rope_frac((double)s0 * g), c0, s0f);
      cr[e] = c0;
      sr[e] = s0f;
      if constexpr (R > 1) {
        // (a step of 0, across sequences, gives 1 and 0 exactly)
        const double turns = a.rope_small_step || !a.rope_across ? g : 0.0;
        if constexpr (DT == VELOGRAD_DTYPE_F32) {
          if (a.rope_small_step) cos_sin_small_d(g * a.rope_step_rad, cs[e], sn[e]);
          else cos_sin_turn_d(turns - rint(turns), cs[e], sn[e]);
        } else {
          if (a.rope_small_step) cos_sin_small((float)(g * a.rope_step_rad), cs[e], sn[e]);
          else cos_sin_turn(rope_frac(turns), cs[e], sn[e]);
        }
      }
      g *= a.rope_ratio;
    }
  }

  auto make_h = [&](int u, int k, float* hf) {
    C::unpack(xv[u][k], hf);
    if constexpr (RES) {
      float rf[V];
      C::unpack(rv[u][k], rf);
#pragma unroll
      for (int i = 0; i < V; ++i) hf[i] = hf[i] + rf[i];
    }
  };
  // ANY: the row's last chunk may begin inside the one before it; those columns are not its own
  auto skip_of = [&](int k) { return ANY ? (lt + k * tpr) * V - col[k] : 0; };

  // row sums: each wave's in its lane 0, then the waves' of four rows at once, one row to each
  // 16 lanes
#pragma unroll
  for (int u = 0; u < R; ++u) {
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float hf[V];
      make_h(u, k, hf);
      float p = 0.0f;
      if constexpr (ANY) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float t = i >= skip_of(k) ? hf[i] : 0.0f;
          p = __builtin_fmaf(t, t, p);
        }
      } else {
#pragma unroll
        for (int i = 0; i < V; ++i) p = __builtin_fmaf(hf[i], hf[i], p);
      }
      ss += own[k] ? p : 0.0f;
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave][u] = ss;
  }
  __syncthreads();
  float r[R];
  {
    const int lane = threadIdx.x & (kWave - 1);
    const int wpr = tpr / kWave;
    const int w = lane & 15;
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int u = 4 * q + (lane >> 4);
      float t = (w < wpr && u < R) ? red[grp * wpr + (w < wpr ? w : 0)][u] : 0.0f;
      t += dpp_move<0xB1>(t);
      t += dpp_move<0x4E>(t);
      t += dpp_move<0x124>(t);
      t += dpp_move<0x128>(t);
      const float mean = t / (float)a.dim;
      const float ir = 1.0f / __builtin_sqrtf(floor_mean_sq(mean, a.ms_floor) + a.eps);
      if (lt < kWave && w == 0 && ok && u < ns && a.inv_rms != nullptr)
        a.inv_rms[row0 + u * step] = ir;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (4 * q + j < R)
          r[4 * q + j] = __builtin_bit_cast(
              float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ir), 16 * j));
      }
    }
  }

  const bool write_h = RES && a.h != nullptr;
  float wf[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) wc[k].unpack(has_w, wf[k]);
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int64_t row = row0 + u * step;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float hf[V];
      forget(xv[u][k]);
      if constexpr (RES) forget(rv[u][k]);
      make_h(u, k, hf);
      const bool store = ok && u < ns && own[k];
      auto put = [&](void* base, int64_t ld, const u32x4 v) {
        if (!store) return;
        if constexpr (ANY) {
          const int skip = skip_of(k);
          if (skip == 0) {
            store16_any_stream<DT>(base, row * ld + col[k], v);
          } else {
#pragma unroll
            for (int i = 2; i < V; ++i) {
              if (i >= skip) {
                float f[V];
                C::unpack(v, f);
                C::store1(base, row * ld + col[k] + i, f[i]);
              }
            }
          }
        } else {
          store16_stream<DT>(base, row * ld + col[k], v);
        }
      };
      if (write_h) put(a.h, a.ld_h, C::pack(hf));
      float yf[V];
#pragma unroll
      for (int i = 0; i < V; ++i) yf[i] = (hf[i] * r[u]) * wf[k][i];
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const int e = k * P + q;
        const float c = (float)cr[e], s = (float)sr[e];
        if constexpr (R > 1) {
          if (u + 1 < R) {
            const RotT cn = __builtin_elementwise_fma(cr[e], cs[e], -(sr[e] * sn[e]));
            sr[e] = __builtin_elementwise_fma(sr[e], cs[e], cr[e] * sn[e]);
            cr[e] = cn;
          }
        }
        const float y0 = yf[2 * q], y1 = yf[2 * q + 1];
        yf[2 * q] = __builtin_fmaf(y0, c, -(y1 * s));                      // functional.py:313
        yf[2 * q + 1] = __builtin_fmaf(y0, s, y1 * c);                     // functional.py:314
      }
      put(a.y, a.ld_y, C::pack(yf));
    }
  }
}

// ------------------------------------------------------------------------------------------
// Forward, short rows of any length and alignment (kFwdElemMaxDim): one-shot rows as in
// fwd_vec_kernel, several a workgroup, with bwd_ring_elem_kernel's element-strided lanes (lane lt
// of a row group holds columns lt, lt + tpr, ..., M of them), so each of a wave's element loads
// and stores moves one contiguous run of 64 elements.  y in the activation dtype (the plain
// output) only; longer rows move in chunks (fwd_vec_kernel's ANY).
// ------------------------------------------------------------------------------------------
constexpr int64_t kFwdElemMaxDim = 64;  // the host plans it for rows of at most this length
constexpr int kFwdElemPerLane = vg_plan::elem_per_lane(kFwdElemMaxDim);

template <int DT, int WDT, int M>
__global__ __launch_bounds__(vg_plan::kRingBlock) void fwd_elem_kernel(const FwdArgs a) {
  using C = Codec<DT>;
  using Raw = std::conditional_t<C::kBytes == 2, uint16_t, uint32_t>;
  static_assert(M == 4 || M == 8, "four or eight elements a lane");
  __shared__ float red[kMaxWavesPerRow];
  const int tpr = a.tpr;
  const int grp = threadIdx.x / tpr;
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t row = (int64_t)blockIdx.x * groups + grp;
  const bool row_ok = row < a.rows;
  const int64_t rw = row_ok ? row : a.rows - 1;  // a row group past the end reads the last row
  const bool has_res = a.res != nullptr;
  const bool write_h = has_res && a.h != nullptr;
  int col[M];
  bool own[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int c = lt + m * tpr;
    own[m] = c < a.dim;
    col[m] = own[m] ? c : a.dim - 1;
  }
  auto decode = [&](uint32_t u) -> float {
    if constexpr (DT == VELOGRAD_DTYPE_BF16) {
      return __builtin_bit_cast(float, u << 16);
    } else if constexpr (DT == VELOGRAD_DTYPE_F16) {
      return (float)__builtin_bit_cast(_Float16, (uint16_t)u);
    } else {
      return __builtin_bit_cast(float, u);
    }
  };
  auto load_raw = [&](const void* base, int64_t i) -> uint32_t {
    return (uint32_t)__builtin_nontemporal_load(static_cast<const Raw*>(base) + i);
  };
  auto store_one = [&](void* base, int64_t i, float f) {
    Raw v;
    if constexpr (DT == VELOGRAD_DTYPE_BF16) v = __builtin_bit_cast(uint16_t, (__bf16)f);
    else if constexpr (DT == VELOGRAD_DTYPE_F16) v = __builtin_bit_cast(uint16_t, (_Float16)f);
    else v = __builtin_bit_cast(uint32_t, f);
    __builtin_nontemporal_store(v, static_cast<Raw*>(base) + i);
  };

  uint32_t xr[M], rr[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    xr[m] = load_raw(a.x, rw * a.ld_x + col[m]);
    rr[m] = has_res ? load_raw(a.res, rw * a.ld_res + col[m]) : 0u;
  }
  float wf[M];
#pragma unroll
  for (int m = 0; m < M; ++m) wf[m] = a.w != nullptr ? Codec<WDT>::load1(a.w, col[m]) : 1.0f;
  float hf[M];
  float ss = 0.0f;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    hf[m] = decode(xr[m]);
    if (has_res) hf[m] = hf[m] + decode(rr[m]);
    const float t = hf[m] * hf[m];
    ss += own[m] ? t : 0.0f;
  }
  ss = row_sum(ss, tpr, grp, red);
  const float mean_sq = floor_mean_sq(ss / (float)a.dim, a.ms_floor);
  const float r = 1.0f / __builtin_sqrtf(mean_sq + a.eps);
  if (row_ok && lt == 0 && a.inv_rms != nullptr) a.inv_rms[row] = r;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (row_ok && own[m]) {
      if (write_h) store_one(a.h, row * a.ld_h + col[m], hf[m]);
      store_one(a.y, row * a.ld_y + col[m], (hf[m] * r) * wf[m]);
    }
  }
}

// ------------------------------------------------------------------------------------------
// Forward, the rows that the kernels above do not take (longer than their registers hold, wide
// ragged ones without a residual (plan_any_rows), rows shorter than a chunk with a quantised or RoPE
// output, streams off their element's alignment): one row per workgroup, two passes over the row
// (the second re-reads x and residual, normally from L2, and recomputes the identical fp32 h).
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int OUT>
__global__ __launch_bounds__(kGenericBlock) void fwd_generic_kernel(const FwdArgs a) {
  using C = Codec<DT>;
  using CW = Codec<WDT>;
  __shared__ float red[kGenericBlock / kWave];
  const int64_t row = xcd_item(blockIdx.x, gridDim.x, a.run_log2);
  const bool has_res = a.res != nullptr;
  const bool has_w = a.w != nullptr;
  const bool write_h = has_res && a.h != nullptr;

  // The plain output moves the row's 16-byte-aligned middle with 16-byte accesses when every
  // stream's row starts at the same offset inside a 16-byte line (contiguous tensors of one dtype
  // whose rows are not 16-byte multiples): `head` elements up to the first boundary and the `tail`
  // past the last whole chunk go element by element.  Other layouts stay element-wise.
  int head = a.dim, nbody = 0;
  if constexpr (OUT == kOutDtype) {
    const uintptr_t mis = row_offset16(a.x, row * a.ld_x, C::kBytes);
    if (mis % C::kBytes == 0 && (!has_res || row_offset16(a.res, row * a.ld_res, C::kBytes) == mis) &&
        row_offset16(a.y, row * a.ld_y, C::kBytes) == mis &&
        (!write_h || row_offset16(a.h, row * a.ld_h, C::kBytes) == mis)) {
      head = (int)(((16 - mis) & 15) / C::kBytes);
      if (head > a.dim) head = a.dim;
      nbody = (a.dim - head) / C::kVec;
    }
  }
  const int tail = head + nbody * C::kVec;  // first element after the body
  auto scalar_j = [&](int t) { return t < head ? t : tail + (t - head); };
  const int nscalar = a.dim - nbody * C::kVec;
  // the weight at the body's chunks: where it sits in its 16-byte lines (2-byte aligned at least)
  const uintptr_t w_align = has_w ? row_offset16(a.w, head, CW::kBytes) : 0;

  // A thread's first KR body chunks stay in registers from the first pass to the second (rows
  // of up to KR * 256 chunks: 8192 bf16/fp16 or 4096 fp32 elements read once); chunks past
  // them are read again in the second pass.  That re-read finds them in L2 when the first pass
  // reads with the normal cache policy and the second non-temporally (its last use): 147.6
  // against 174.9 us the other way round at 16384 x 4100 bf16, before the registers.
  constexpr int KR = OUT == kOutDtype ? 4 : 0;
  u32x4 xk[KR > 0 ? KR : 1], rk[KR > 0 ? KR : 1];
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    const int c = threadIdx.x + k * blockDim.x;
    xk[k] = u32x4{0u, 0u, 0u, 0u};
    rk[k] = u32x4{0u, 0u, 0u, 0u};
    if (c < nbody) {
      const int64_t j = head + (int64_t)c * C::kVec;
      xk[k] = load16_stream<DT>(a.x, row * a.ld_x + j);
      if (has_res) rk[k] = load16_stream<DT>(a.res, row * a.ld_res + j);
    }
  }
  // With a body, the head and tail are fewer than two chunks' worth of elements: one per thread
  // at most, loaded with the body, so a row waits for memory once per pass.
  const bool few_scalar = KR > 0 && nbody > 0;
  int j_s = 0;
  float h_s = 0.0f, w_s = 1.0f;
  if (few_scalar && (int)threadIdx.x < nscalar) {
    j_s = scalar_j(threadIdx.x);
    h_s = C::load1(a.x, row * a.ld_x + j_s);
    if (has_res) h_s = h_s + C::load1(a.res, row * a.ld_res + j_s);
    if (has_w) w_s = CW::load1(a.w, j_s);
  }
  // h of register chunk k (the same single fp32 add as every other path)
  auto h_reg = [&](int k, float* hf) {
    C::unpack(xk[k], hf);
    if (has_res) {
      float rf[C::kVec];
      C::unpack(rk[k], rf);
#pragma unroll
      for (int i = 0; i < C::kVec; ++i) hf[i] = hf[i] + rf[i];
    }
  };
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    const int c = threadIdx.x + k * blockDim.x;
    if (c < nbody) {
      float hf[C::kVec];
      h_reg(k, hf);
      if (write_h) store16_stream<DT>(a.h, row * a.ld_h + head + (int64_t)c * C::kVec, C::pack(hf));
#pragma unroll
      for (int i = 0; i < C::kVec; ++i) ss += hf[i] * hf[i];
    }
  }
  for (int c = threadIdx.x + KR * blockDim.x; c < nbody; c += blockDim.x) {
    const int64_t j = head + (int64_t)c * C::kVec;
    float hf[C::kVec];
    C::unpack(load16<DT>(a.x, row * a.ld_x + j), hf);
    if (has_res) {
      float rf[C::kVec];
      C::unpack(load16<DT>(a.res, row * a.ld_res + j), rf);
#pragma unroll
      for (int i = 0; i < C::kVec; ++i) hf[i] = hf[i] + rf[i];
    }
    if (write_h) store16_stream<DT>(a.h, row * a.ld_h + j, C::pack(hf));
#pragma unroll
    for (int i = 0; i < C::kVec; ++i) ss += hf[i] * hf[i];
  }
  if (few_scalar) {
    if ((int)threadIdx.x < nscalar) {
      if (write_h) C::store1(a.h, row * a.ld_h + j_s, h_s);
      ss += h_s * h_s;
    }
  } else {
    for (int t = threadIdx.x; t < nscalar; t += blockDim.x) {
      const int j = scalar_j(t);
      float hx = C::load1(a.x, row * a.ld_x + j);
      if (has_res) hx = hx + C::load1(a.res, row * a.ld_res + j);
      if (write_h) C::store1(a.h, row * a.ld_h + j, hx);
      ss += hx * hx;
    }
  }
  ss = row_sum(ss, blockDim.x, 0, red);
  const float mean_sq = floor_mean_sq(ss / (float)a.dim, a.ms_floor);
  const float r = 1.0f / __builtin_sqrtf(mean_sq + a.eps);
  if (threadIdx.x == 0 && a.inv_rms != nullptr) a.inv_rms[row] = r;

  auto y_at = [&](int j) {
    float hx = C::load1(a.x, row * a.ld_x + j);
    if (has_res) hx = hx + C::load1(a.res, row * a.ld_res + j);
    const float n = hx * r;
    return has_w ? n * CW::load1(a.w, j) : n;
  };
  if constexpr (OUT == kOutDtype) {
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int c = threadIdx.x + k * blockDim.x;
      if (c < nbody) {
        const int64_t j = head + (int64_t)c * C::kVec;
        float hf[C::kVec], wf[C::kVec];
        h_reg(k, hf);
        if (has_w) weight_run<DT, WDT>(a.w, j, w_align, wf);
#pragma unroll
        for (int i = 0; i < C::kVec; ++i) {
          const float n = hf[i] * r;
          hf[i] = has_w ? n * wf[i] : n;
        }
        store16_stream<DT>(a.y, row * a.ld_y + j, C::pack(hf));
      }
    }
    // the chunks past the registers: x and the residual read again (normally from L2)
    for (int c = threadIdx.x + KR * blockDim.x; c < nbody; c += blockDim.x) {
      const int64_t j = head + (int64_t)c * C::kVec;
      float hf[C::kVec];
      C::unpack(load16_stream<DT>(a.x, row * a.ld_x + j), hf);
      if (has_res) {
        float rf[C::kVec];
        C::unpack(load16_stream<DT>(a.res, row * a.ld_res + j), rf);
#pragma unroll
        for (int i = 0; i < C::kVec; ++i) hf[i] = hf[i] + rf[i];
      }
      float wf[C::kVec];
      if (has_w) weight_run<DT, WDT>(a.w, j, w_align, wf);
#pragma unroll
      for (int i = 0; i < C::kVec; ++i) {
        const float n = hf[i] * r;
        hf[i] = has_w ? n * wf[i] : n;
      }
      store16_stream<DT>(a.y, row * a.ld_y + j, C::pack(hf));
    }
    if (few_scalar) {
      if ((int)threadIdx.x < nscalar) {
        const float n = h_s * r;  // y_at's arithmetic on the register copies
        C::store1(a.y, row * a.ld_y + j_s, has_w ? n * w_s : n);
      }
    } else {
      for (int t = threadIdx.x; t < nscalar; t += blockDim.x) {
        const int j = scalar_j(t);
        C::store1(a.y, row * a.ld_y + j, y_at(j));
      }
    }
  } else if constexpr (OUT == kOutRopeI) {
    const int64_t pos = row % a.rope_seq;
    RopeFreqWalk fw(threadIdx.x, blockDim.x, a.rope_c_hi, a.rope_c_lo);
    for (int i = threadIdx.x; i < a.rope_half; i += blockDim.x) {
      const float x0 = y_at(2 * i), x1 = y_at(2 * i + 1);
      float c, sn;
      rope_cos_sin_f(pos, fw.next(), c, sn);
      C::store1(a.y, row * a.ld_y + 2 * i, x0 * c - x1 * sn);       // functional.py:313
      C::store1(a.y, row * a.ld_y + 2 * i + 1, x0 * sn + x1 * c);   // functional.py:314
    }
  } else if constexpr (OUT == kOutMxE4M3 || OUT == kOutMxE2M1) {
    // MX epilogue (see fwd_vec_kernel): a third pass, one 32-element block per thread.
    constexpr int kEmax = OUT == kOutMxE4M3 ? vg_mx::kEmaxE4M3 : vg_mx::kEmaxE2M1;
    uint8_t* yq = static_cast<uint8_t*>(a.y) + row * a.ld_y;
    for (int b = threadIdx.x; b < a.dim / vg_mx::kBlock; b += blockDim.x) {
      const int j0 = b * vg_mx::kBlock;
      uint32_t am = 0;
      for (int i = 0; i < vg_mx::kBlock; ++i)
        am = umax(am, __builtin_bit_cast(uint32_t, y_at(j0 + i)) & 0x7fffffffu);
      const bool finite = am < 0x7f800000u;
      const float f = finite ? vg_mx::inverse_scale(vg_mx::shared_exp(am, kEmax)) : 0.0f;
      for (int i = 0; i < vg_mx::kBlock; i += 2) {
        const float v0 = y_at(j0 + i) * f, v1 = y_at(j0 + i + 1) * f;
        if constexpr (OUT == kOutMxE4M3) {
          yq[j0 + i] = finite ? (uint8_t)e4m3x1(__builtin_fminf(__builtin_fmaxf(v0, -kE4M3Max), kE4M3Max)) : 0;
          yq[j0 + i + 1] = finite ? (uint8_t)e4m3x1(__builtin_fminf(__builtin_fmaxf(v1, -kE4M3Max), kE4M3Max)) : 0;
        } else {
          yq[(j0 + i) / 2] = finite ? (uint8_t)e2m1x2<0>(0u, v0, v1) : 0;
        }
      }
      a.mx_scale[row * a.ld_mx + b] = (uint8_t)vg_mx::scale_code(am, kEmax);
    }
  } else {
    // fp8 epilogue (see fwd_vec_kernel): a third pass stores the codes.
    __shared__ uint32_t red_max[kGenericBlock / kWave];
    uint32_t am = 0;
    for (int j = threadIdx.x; j < a.dim; j += blockDim.x)
      am = umax(am, __builtin_bit_cast(uint32_t, y_at(j)) & 0x7fffffffu);
    am = row_max_abs_bits(am, blockDim.x, 0, red_max);
    const float scale = __builtin_bit_cast(float, am) / kE4M3Max;
    const float inv = inverse_scale(scale);
    if (threadIdx.x == 0) a.y_scale[row] = scale;
    uint8_t* yq = static_cast<uint8_t*>(a.y) + row * a.ld_y;
    for (int j = threadIdx.x; j < a.dim; j += blockDim.x)
      yq[j] = (uint8_t)e4m3x1(y_at(j) * inv);
  }
}

// ------------------------------------------------------------------------------------------
// Backward, register-resident row, persistent row slots.
// FLAGS: kSavedIsH (the saved tensor is h, xhat = h * inv_rms is formed in registers),
//        kGradH (a residual-stream gradient grad_h is added to dx in the same pass).
// ------------------------------------------------------------------------------------------
constexpr int kSavedIsH = 1;
constexpr int kGradH = 2;
// kRopeG: grad_y is the gradient of the interleaved-RoPE-rotated output (the model's
// F.apply_rotary_emb(attention_norm(x)), models/llama.py:48-49), rotated back in registers
// before use: the backward of the rotation (functional.py:316-345) fused into the norm's.
constexpr int kRopeG = 4;
// kRopeDirect: as kRopeG with each pair's rotation evaluated directly where g is decoded (both
// passes), no walk state and no LDS table: rows too wide for the walk's launch bound.
constexpr int kRopeDirect = 16;
// Rows of the RoPE-gradient walk between direct evaluations of the rotation state.
constexpr int kRopeAnchor = 16;

template <int DT, int WDT, int NV, int FLAGS>
__global__ __launch_bounds__((FLAGS & kRopeG) ? vg_plan::max_block_for_nv_rope(NV)
                                               : max_block_for_nv(NV)) void bwd_vec_kernel(const BwdArgs a) {
  using C = Codec<DT>;
  constexpr int V = C::kVec;
  constexpr bool SAVED_IS_H = (FLAGS & kSavedIsH) != 0;
  constexpr bool HAS_GH = (FLAGS & kGradH) != 0;
  constexpr bool ROPE = (FLAGS & kRopeG) != 0;
  constexpr bool RD = (FLAGS & kRopeDirect) != 0;
  static_assert(!(ROPE && RD), "one RoPE mode");
  constexpr int NH = HAS_GH ? NV : 1;  // grad_h chunks (a dummy slot when absent)
  constexpr int P = V / 2;             // RoPE pairs per chunk
  constexpr int NR = ROPE ? NV : 1;    // rotation state slots (a dummy slot without RoPE)
  __shared__ float red[2][kMaxWavesPerRow];
  // dim floats of dynamic LDS: with kRopeG the walk's step rotations (cos, sin per pair), then
  // (after a barrier) the combine of the row groups' dweight columns.
  extern __shared__ __align__(16) float dyn_lds[];

  const int tpr = a.tpr;
  const int grp = threadIdx.x / tpr;
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t slot = (int64_t)blockIdx.x * groups + grp;
  const int64_t nslots = (int64_t)gridDim.x * groups;
  const int nchunk = a.dim / V;
  const bool has_w = a.w != nullptr;
  const bool has_dres = a.dres != nullptr;

  // RoPE: each thread holds (cos, sin) of its pairs at the current row's position and advances
  // them by the rotation through nslots positions (the walk's row step) from the LDS table; they
  // are evaluated directly where the position wraps to a new outer index and on every
  // kRopeAnchor-th row of the walk.  Float32 state: each step adds about an ulp, so re-anchoring
  // keeps the drift under kRopeAnchor ulps however long the walk (the sequence length over the
  // slot count), far below the output rounding of bf16/fp16 and the fp32 dx tolerance.
  float rc[NR][P], rs[NR][P];
  if constexpr (ROPE) {
    for (int q = threadIdx.x; q < a.dim / 2; q += blockDim.x) {
      double sv, cv;
      sincos((double)nslots * rope_freq(q, a.rope_c_hi, a.rope_c_lo), &sv, &cv);
      dyn_lds[2 * q] = (float)cv;
      dyn_lds[2 * q + 1] = (float)sv;
    }
    __syncthreads();
  }
  auto rope_start = [&](int64_t pos) {
    if constexpr (ROPE) {
#pragma unroll
      for (int k = 0; k < NR; ++k) {
#pragma unroll
        for (int p = 0; p < P; ++p)
          rope_cos_sin(pos, (lt + k * tpr) * P + p, a.rope_c_hi, a.rope_c_lo, rc[k][p],
                       rs[k][p]);
      }
    }
  };
  auto rope_step = [&]() {
    if constexpr (ROPE) {
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const int c = lt + k * tpr;
        if (c < nchunk) {
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const float sc = dyn_lds[2 * (c * P + p)], ss = dyn_lds[2 * (c * P + p) + 1];
            const float cn = rc[k][p] * sc - rs[k][p] * ss;
            rs[k][p] = rs[k][p] * sc + rc[k][p] * ss;
            rc[k][p] = cn;
          }
        }
      }
    }
  };

  // Packed weight chunks and the fp32 dweight column accumulators live for the whole walk; the
  // row's g and saved chunks stay packed and are decoded once per pass.
  WeightChunk<DT, WDT> wc[NV];
  float acc[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = lt + k * tpr;
    wc[k].load((has_w && c < nchunk) ? a.w : nullptr, (int64_t)c * V);
#pragma unroll
    for (int i = 0; i < V; ++i) acc[k][i] = 0.0f;
  }

  // Loads of one row into (gv, sv, hv, rr); zeros outside the tensor.
  auto load_row = [&](int64_t row, u32x4* gv, u32x4* sv, u32x4* hv, float& rr) {
    const bool ok = row < a.rows;
    rr = ok ? a.inv_rms[row] : 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      gv[k] = u32x4{0u, 0u, 0u, 0u};
      sv[k] = u32x4{0u, 0u, 0u, 0u};
      if constexpr (HAS_GH) hv[k] = u32x4{0u, 0u, 0u, 0u};
      if (ok && c < nchunk) {
        gv[k] = load16_stream<DT>(a.g, row * a.ld_g + (int64_t)c * V);
        sv[k] = load16_stream<DT>(a.saved, row * a.ld_s + (int64_t)c * V);
        if constexpr (HAS_GH) hv[k] = load16_stream<DT>(a.gh, row * a.ld_gh + (int64_t)c * V);
      }
    }
  };
  // kRopeDirect: the current row's position, each chunk's first pair frequency (double) and
  // the ratio between consecutive pairs' frequencies, base^(-2/dim)
  int64_t rd_pos = 0;
  double rd_f0[RD ? NV : 1], rd_ratio = 0.0;
  if constexpr (RD) {
    const double cc = (double)a.rope_c_hi + (double)a.rope_c_lo;
    rd_ratio = exp2(-cc);
#pragma unroll
    for (int k = 0; k < NV; ++k) rd_f0[k] = exp2(-(double)((lt + k * tpr) * P) * cc);
  }
  // Decoded chunk k of the current row: g, xhat (h * inv_rms when h was saved), weight.
  auto decode = [&](const u32x4* gv, const u32x4* sv, float rr, int k, float* gf, float* xh,
                    float* wf) {
    C::unpack(gv[k], gf);
    if constexpr (RD) {
      // inverse rotation, each pair's (cos, sin) from its double angle (as rope_cos_sin)
      double f = rd_f0[k];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        float cs, sn;
        rope_cos_sin_f(rd_pos, f, cs, sn);
        f *= rd_ratio;
        const float g0 = gf[2 * p], g1 = gf[2 * p + 1];
        gf[2 * p] = g0 * cs + g1 * sn;
        gf[2 * p + 1] = g1 * cs - g0 * sn;
      }
    }
    if constexpr (ROPE) {
      // inverse rotation of each pair (y0, y1) -> (y0 c + y1 s, y1 c - y0 s)
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const float g0 = gf[2 * p], g1 = gf[2 * p + 1];
        gf[2 * p] = g0 * rc[k][p] + g1 * rs[k][p];
        gf[2 * p + 1] = g1 * rc[k][p] - g0 * rs[k][p];
      }
    }
    C::unpack(sv[k], xh);
    if constexpr (SAVED_IS_H) {
#pragma unroll
      for (int i = 0; i < V; ++i) xh[i] = xh[i] * rr;
    }
    wc[k].unpack(has_w, wf);
  };

  int64_t row = slot;
  u32x4 gv[NV], sv[NV], hv[NH];
  float rr;
  load_row(row, gv, sv, hv, rr);
  int64_t pos = ROPE ? row % a.rope_seq : 0;
  rope_start(pos);

  for (int it = 0; it < a.iters; ++it) {
    const bool ok = row < a.rows;
    if constexpr (RD) rd_pos = row % a.rope_seq;
    const int64_t nrow = row + nslots;
    u32x4 gn[NV], sn[NV], hn[NH];
    float rn = 0.0f;
    if (it + 1 < a.iters) {
      load_row(nrow, gn, sn, hn, rn);
    } else {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        gn[k] = u32x4{0u, 0u, 0u, 0u};
        sn[k] = u32x4{0u, 0u, 0u, 0u};
        if constexpr (HAS_GH) hn[k] = u32x4{0u, 0u, 0u, 0u};
      }
    }

    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float gf[V], xh[V], wf[V];
      decode(gv, sv, rr, k, gf, xh, wf);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float gw = gf[i] * wf[i];
        s += gw * xh[i];
      }
    }
    s = row_sum(s, tpr, grp, red[it & 1]);
    const float m = s / (float)a.dim;

#pragma unroll
    for (int k = 0; k < NV; ++k) {
      forget(gv[k]);
      forget(sv[k]);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      float gf[V], xh[V], wf[V];
      decode(gv, sv, rr, k, gf, xh, wf);
      if (ok && c < nchunk) {
        float d[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float gw = gf[i] * wf[i];
          d[i] = rr * (gw - xh[i] * m);
        }
        if constexpr (HAS_GH) {
          float ghf[V];
          C::unpack(hv[k], ghf);
#pragma unroll
          for (int i = 0; i < V; ++i) d[i] = d[i] + ghf[i];
        }
        const u32x4 pv = C::pack(d);
        store16_stream<DT>(a.dx, row * a.ld_dx + (int64_t)c * V, pv);
        if (has_dres) store16_stream<DT>(a.dres, row * a.ld_dres + (int64_t)c * V, pv);
      }
#pragma unroll
      for (int i = 0; i < V; ++i) acc[k][i] += gf[i] * xh[i];
    }

    if constexpr (ROPE) {
      pos += nslots;
      if (pos >= a.rope_seq) {
        pos = nrow % a.rope_seq;
        rope_start(pos);
      } else if ((it + 1) % kRopeAnchor == 0) {
        rope_start(pos);
      } else {
        rope_step();
      }
    }
    row = nrow;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      gv[k] = gn[k];
      sv[k] = sn[k];
      if constexpr (HAS_GH) hv[k] = hn[k];
    }
    rr = rn;
  }

  if (a.partial == nullptr) return;
  // One fp32 partial row per workgroup.  Row groups are added in group order through LDS
  // (dim floats of dynamic LDS), so the partial does not depend on timing.
  float* prow = a.partial + (int64_t)blockIdx.x * a.dim;
  if (groups == 1) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = lt + k * tpr;
      if (c < nchunk) {
#pragma unroll
        for (int q = 0; q < V / 4; ++q)
          store16<VELOGRAD_DTYPE_F32>(prow, (int64_t)c * V + 4 * q,
                                      Codec<VELOGRAD_DTYPE_F32>::pack(&acc[k][4 * q]));
      }
    }
    return;
  }
  float* comb = dyn_lds;
  if constexpr (ROPE) __syncthreads();  // every thread is done with the step table
  for (int gi = 0; gi < groups; ++gi) {
    if (grp == gi) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int c = lt + k * tpr;
        if (c < nchunk) {
#pragma unroll
          for (int i = 0; i < V; ++i)
            comb[c * V + i] = (gi == 0) ? acc[k][i] : comb[c * V + i] + acc[k][i];
        }
      }
    }
    __syncthreads();
  }
  for (int q = threadIdx.x; q < a.dim / 4; q += blockDim.x)
    store16<VELOGRAD_DTYPE_F32>(prow, 4 * (int64_t)q, *reinterpret_cast<const u32x4*>(comb + 4 * q));
}

// ------------------------------------------------------------------------------------------
// Backward, ring-pipelined (launch_plan.h: plan_bwd_ring).  Each row slot walks rows slot,
// slot + S, ... as in bwd_vec_kernel, but keeps a ring of PF + 1 = 3 row buffers (2 with
// grad_h): while a row reduces, the next two rows' loads are in flight.  Rows are of whole
// 16-byte chunks, dim <= NV * tpr * V (kRingTail where lanes are left idle; kRing8 for rows of
// 8-byte alignment with a half chunk at their end), and the steady loop
// covers only iterations in which every slot has a row, loading prefetch rows past the end from
// the last row instead (never used), so it is free of branches around memory operations: the
// wait for a row's data then counts exactly the later loads and stores instead of draining them,
// which a guarded loop forces.  The loop is unrolled by the ring length so the buffers are
// indexed at compile time.  kRingDres: dres is written too.
// ------------------------------------------------------------------------------------------
constexpr int kRingDres = 8;
constexpr int kRingTail = 32;
constexpr int kRing8 = 64;
constexpr int kRingAny = 128;

template <int DT, int WDT, int NV, int FLAGS>
__global__ __launch_bounds__(vg_plan::kRingBlock) void bwd_ring_kernel(const BwdArgs a) {
  using C = Codec<DT>;
  constexpr int V = C::kVec;
  constexpr bool SAVED_IS_H = (FLAGS & kSavedIsH) != 0;
  constexpr bool HAS_GH = (FLAGS & kGradH) != 0;
  constexpr bool HAS_DRES = (FLAGS & kRingDres) != 0;
  // kRingTail: rows of fewer chunks than the row group's lanes (launch_plan.h ring_eligible):
  // an idle lane loads the row's last chunk instead (no branch around the load), adds nothing
  // and stores nothing
  constexpr bool TAIL = (FLAGS & kRingTail) != 0;
  // kRing8: rows of a 2-byte dtype that start on 8-byte boundaries only, dim = n * V + V / 2
  // (hidden sizes such as 4100): each of the n whole chunks moves as two 8-byte halves, and the
  // row's last V / 2 elements form an extra half chunk that lane 0 of the row group owns; every
  // lane of the group loads those same 8 bytes (one request per wave), so no branch guards the
  // load.  The row group is laid out over the n whole chunks.
  constexpr bool X8 = (FLAGS & kRing8) != 0;
  static_assert(!X8 || C::kBytes == 2, "rows of 8-byte alignment are of a 2-byte dtype");
  // kRingAny: rows of any length from one chunk up whose streams start at any element.  Lane c of
  // the row group takes the chunk at column min(c * V, dim - V), so its columns are the same in
  // every row.  The columns that the last chunk shares with the one before it add nothing to the
  // sums and are stored by both lanes, the same bits (one store a lane and row, as everywhere: the
  // ring's waits count them; storing them element by element instead held the last wave up at
  // every row, 16384 x 4095 bf16 126 us); dx must then not be grad_h itself.
  constexpr bool ANY = (FLAGS & kRingAny) != 0;
  static_assert(!ANY || (!X8 && !TAIL), "one row layout");
  constexpr int VH = V / 2;
  constexpr int NH = HAS_GH ? NV : 1;  // grad_h chunks (a dummy slot when absent)
  // With grad_h a third stream fills the ring: one row ahead keeps it within 256 VGPRs.
  constexpr int PF = HAS_GH ? 1 : vg_plan::kRingPrefetch;
  constexpr int R = PF + 1;
  constexpr int RX = X8 ? R : 1;  // extra half-chunk buffers (a dummy slot without kRing8)
  static_assert((FLAGS & kRopeG) == 0, "the RoPE gradient runs in bwd_vec_kernel");
  __shared__ float red[2][kMaxWavesPerRow];
  extern __shared__ __align__(16) float dyn_lds[];  // dim floats: the row groups' combine

  const int tpr = a.tpr;
  const int grp = threadIdx.x / tpr;
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t slot = (int64_t)blockIdx.x * groups + grp;
  const int64_t nslots = (int64_t)gridDim.x * groups;
  const bool has_w = a.w != nullptr;
  const int64_t last = a.rows - 1;
  // chunk k of this lane (the row's last whole one for an idle lane) and whether it is its own
  const int nfull = ANY ? (a.dim + V - 1) / V : a.dim / V;
  int ccol[NV];  // its first column
  bool own[NV];
  int skip[NV];  // kRingAny: its columns that are not its own to sum
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = lt + k * tpr;
    own[k] = !(TAIL || ANY) || c < nfull;
    ccol[k] = ANY ? min(c * V, a.dim - V) : (own[k] ? c : nfull - 1) * V;
    skip[k] = ANY ? (own[k] ? c * V - ccol[k] : V) : 0;
  }
  const int64_t xcol = (int64_t)a.dim - VH;  // kRing8: the extra half chunk's first column
  const bool own_x = X8 && lt == 0;

  WeightChunk<DT, WDT> wc[NV];
  float acc[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if constexpr (ANY) {
      if (has_w) wc[k].load_any(a.w, ccol[k]);
    } else {
      wc[k].load(has_w ? a.w : nullptr, ccol[k]);
    }
#pragma unroll
    for (int i = 0; i < V; ++i) acc[k][i] = 0.0f;
  }
  float wfx[VH], accx[VH];
  if constexpr (X8) {
#pragma unroll
    for (int i = 0; i < VH; ++i) {
      wfx[i] = 1.0f;
      accx[i] = 0.0f;
    }
    if (has_w) {
      if constexpr (WDT == VELOGRAD_DTYPE_F32) {
        Codec<VELOGRAD_DTYPE_F32>::unpack(load16<VELOGRAD_DTYPE_F32>(a.w, xcol), wfx);
      } else {
        const u32x2 q = *reinterpret_cast<const u32x2*>(static_cast<const char*>(a.w) +
                                                        xcol * Codec<WDT>::kBytes);
        float t[V];
        Codec<WDT>::unpack(u32x4{q.x, q.y, 0u, 0u}, t);
#pragma unroll
        for (int i = 0; i < VH; ++i) wfx[i] = t[i];
      }
    }
  }

  u32x4 gr[R][NV], sr[R][NV], hr[R][NH];
  u32x2 gx[RX][HAS_GH ? 3 : 2];  // kRing8: the extra half chunk's g, saved (and grad_h)
  float rr[R];
  // One chunk of a stream: 16 bytes, or two 8-byte halves for kRing8 rows.
  auto load_chunk = [&](const void* base, int64_t e) -> u32x4 {
    if constexpr (X8) {
      const u32x2 lo = load8_stream<DT>(base, e);
      const u32x2 hi = load8_stream<DT>(base, e + VH);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    } else if constexpr (ANY) {
      return load16_any_stream<DT>(base, e);
    } else {
      return load16_stream<DT>(base, e);
    }
  };
  auto store_chunk = [&](void* base, int64_t e, const u32x4 v) {
    if constexpr (X8) {
      store8_stream<DT>(base, e, u32x2{v.x, v.y});
      store8_stream<DT>(base, e + VH, u32x2{v.z, v.w});
    } else if constexpr (ANY) {
      store16_any_stream<DT>(base, e, v);
    } else {
      store16_stream<DT>(base, e, v);
    }
  };
  // Row `row`'s g, saved, grad_h chunks and inv_rms; rows past the end read the last row.
  auto load_row = [&](int64_t row, u32x4* gv, u32x4* sv, u32x4* hv, float& r, u32x2* xv) {
    const int64_t rw = row < a.rows ? row : last;
    r = a.inv_rms[rw];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int64_t col = ccol[k];
      gv[k] = load_chunk(a.g, rw * a.ld_g + col);
      sv[k] = load_chunk(a.saved, rw * a.ld_s + col);
      if constexpr (HAS_GH) hv[k] = load_chunk(a.gh, rw * a.ld_gh + col);
    }
    if constexpr (X8) {
      xv[0] = load8_stream<DT>(a.g, rw * a.ld_g + xcol);
      xv[1] = load8_stream<DT>(a.saved, rw * a.ld_s + xcol);
      if constexpr (HAS_GH) xv[2] = load8_stream<DT>(a.gh, rw * a.ld_gh + xcol);
    }
  };
  auto decode = [&](const u32x4* gv, const u32x4* sv, float r, int k, float* gf, float* xh,
                    float* wf) {
    C::unpack(gv[k], gf);
    C::unpack(sv[k], xh);
    if constexpr (SAVED_IS_H) {
#pragma unroll
      for (int i = 0; i < V; ++i) xh[i] = xh[i] * r;
    }
    wc[k].unpack(has_w, wf);
  };
  // The backward of one row (as bwd_vec_kernel's loop body); `ok` = the row exists.  The row's
  // decoded g * w and xhat stay in registers across the reduction (one workgroup per CU leaves
  // 256 VGPRs a lane): decoding them again after it, as bwd_vec_kernel does to save registers,
  // ran 16384 x 4096 bf16 in 69.2 us against 68.5 and 16384 x 5120 in 92.7 against 85.1.
  auto process = [&](u32x4* gv, u32x4* sv, const u32x4* hv, float r, const u32x2* xv,
                     int64_t row, bool ok, int it) {
    float s = 0.0f;
    float gfk[NV][V], xhk[NV][V], gwk[NV][V];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float wf[V];
      decode(gv, sv, r, k, gfk[k], xhk[k], wf);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        gwk[k][i] = gfk[k][i] * wf[i];
        if constexpr (ANY) {
          const float t = gwk[k][i] * xhk[k][i];
          s += i >= skip[k] ? t : 0.0f;
        } else if constexpr (TAIL) {
          const float t = gwk[k][i] * xhk[k][i];
          s += own[k] ? t : 0.0f;
        } else {
          s += gwk[k][i] * xhk[k][i];
        }
      }
    }
    float gfx[VH], xhx[VH], gwx[VH];
    if constexpr (X8) {
      float t[V];
      C::unpack(u32x4{xv[0].x, xv[0].y, 0u, 0u}, t);
#pragma unroll
      for (int i = 0; i < VH; ++i) gfx[i] = t[i];
      C::unpack(u32x4{xv[1].x, xv[1].y, 0u, 0u}, t);
#pragma unroll
      for (int i = 0; i < VH; ++i) {
        xhx[i] = SAVED_IS_H ? t[i] * r : t[i];
        gwx[i] = gfx[i] * wfx[i];
        const float p = gwx[i] * xhx[i];
        s += own_x ? p : 0.0f;
      }
    }
    s = row_sum(s, tpr, grp, red[it & 1]);
    const float m = s / (float)a.dim;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int64_t col = ccol[k];
      const float* gf = gfk[k];
      const float* xh = xhk[k];
      float d[V];
#pragma unroll
      for (int i = 0; i < V; ++i) d[i] = r * (gwk[k][i] - xh[i] * m);
      if constexpr (HAS_GH) {
        float ghf[V];
        C::unpack(hv[k], ghf);
#pragma unroll
        for (int i = 0; i < V; ++i) d[i] = d[i] + ghf[i];
      }
      const u32x4 pv = C::pack(d);
      const bool store = (TAIL || ANY) ? ok && own[k] : ok;
      if (store) {
        store_chunk(a.dx, row * a.ld_dx + col, pv);
        if constexpr (HAS_DRES) store_chunk(a.dres, row * a.ld_dres + col, pv);
      }
#pragma unroll
      for (int i = 0; i < V; ++i) acc[k][i] += store ? gf[i] * xh[i] : 0.0f;
    }
    if constexpr (X8) {
      float d[V];
#pragma unroll
      for (int i = 0; i < VH; ++i) d[i] = r * (gwx[i] - xhx[i] * m);
#pragma unroll
      for (int i = VH; i < V; ++i) d[i] = 0.0f;
      if constexpr (HAS_GH) {
        float t[V];
        C::unpack(u32x4{xv[2].x, xv[2].y, 0u, 0u}, t);
#pragma unroll
        for (int i = 0; i < VH; ++i) d[i] = d[i] + t[i];
      }
      const u32x4 pv = C::pack(d);
      const bool sx = ok && own_x;
      if (sx) {
        store8_stream<DT>(a.dx, row * a.ld_dx + xcol, u32x2{pv.x, pv.y});
        if constexpr (HAS_DRES)
          store8_stream<DT>(a.dres, row * a.ld_dres + xcol, u32x2{pv.x, pv.y});
      }
#pragma unroll
      for (int i = 0; i < VH; ++i) accx[i] += sx ? gfx[i] * xhx[i] : 0.0f;
    }
  };

  // Row j of the walk sits in buffer j % R; processing row j first issues row j + PF's loads
  // into buffer (j + PF) % R, the one row j - 1 has just released.
  const int full = (int)(a.rows / nslots);  // iterations in which every slot has a row
#pragma unroll
  for (int j = 0; j < PF; ++j)
    load_row(slot + (int64_t)j * nslots, gr[j], sr[j], hr[j], rr[j], gx[X8 ? j : 0]);
  int it = 0;
  for (; it + R <= full; it += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int nb = (u + PF) % R;
      load_row(slot + (int64_t)(it + u + PF) * nslots, gr[nb], sr[nb], hr[nb], rr[nb],
               gx[X8 ? nb : 0]);
      process(gr[u], sr[u], hr[u], rr[u], gx[X8 ? u : 0], slot + (int64_t)(it + u) * nslots, true,
              it + u);
    }
  }
  // The last (up to R) iterations, some of whose slots may have no row.
#pragma unroll
  for (int u = 0; u < R; ++u) {
    if (it + u < a.iters) {
      const int nb = (u + PF) % R;
      if (it + u + PF < a.iters)
        load_row(slot + (int64_t)(it + u + PF) * nslots, gr[nb], sr[nb], hr[nb], rr[nb],
                 gx[X8 ? nb : 0]);
      const int64_t row = slot + (int64_t)(it + u) * nslots;
      process(gr[u], sr[u], hr[u], rr[u], gx[X8 ? u : 0], row, row < a.rows, it + u);
    }
  }

  if (a.partial == nullptr) return;
  // One fp32 partial row per workgroup; row groups added in group order through LDS.
  float* prow = a.partial + (int64_t)blockIdx.x * a.dim;
  if (groups == 1) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (!own[k]) continue;
      if constexpr (ANY) {
#pragma unroll
        for (int i = 0; i < V; ++i)
          if (i >= skip[k]) prow[ccol[k] + i] = acc[k][i];
        continue;
      }
#pragma unroll
      for (int q = 0; q < V / 4; ++q)
        store16<VELOGRAD_DTYPE_F32>(prow, ccol[k] + 4 * q,
                                    Codec<VELOGRAD_DTYPE_F32>::pack(&acc[k][4 * q]));
    }
    if constexpr (X8) {
      if (own_x) store16<VELOGRAD_DTYPE_F32>(prow, xcol, Codec<VELOGRAD_DTYPE_F32>::pack(accx));
    }
    return;
  }
  float* comb = dyn_lds;
  for (int gi = 0; gi < groups; ++gi) {
    if (grp == gi) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        if (!own[k]) continue;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const int c = ccol[k] + i;
          if (i >= skip[k]) comb[c] = (gi == 0) ? acc[k][i] : comb[c] + acc[k][i];
        }
      }
      if constexpr (X8) {
        if (own_x) {
#pragma unroll
          for (int i = 0; i < VH; ++i)
            comb[xcol + i] = (gi == 0) ? accx[i] : comb[xcol + i] + accx[i];
        }
      }
    }
    __syncthreads();
  }
  if constexpr (ANY) {
    for (int q = threadIdx.x; q < a.dim; q += blockDim.x) prow[q] = comb[q];
    return;
  }
  for (int q = threadIdx.x; q < a.dim / 4; q += blockDim.x)
    store16<VELOGRAD_DTYPE_F32>(prow, 4 * (int64_t)q, *reinterpret_cast<const u32x4*>(comb + 4 * q));
}

// ------------------------------------------------------------------------------------------
// Backward, short rows of any length and alignment (and longer ones where dx is grad_h itself), in
// bwd_ring_kernel's walk and ring
// (launch_plan.h: plan_bwd_ring_elem).  Element-strided lanes: lane lt of a row group holds
// columns lt, lt + tpr, ..., lt + (M - 1) tpr, so each element load or store of a wave moves
// one contiguous run of 64 elements; a column past the row's end loads the row's last element
// (no branch around a load) and adds and stores nothing.  Rows of M * tpr elements at most: M 4
// or 8 (106-232 VGPRs; sixteen spilled 21-258 VGPRs a lane even one row ahead), so rows of up
// to 4096 elements.
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int M, int FLAGS>
__global__ __launch_bounds__(vg_plan::kRingBlock) void bwd_ring_elem_kernel(const BwdArgs a) {
  using C = Codec<DT>;
  using Raw = std::conditional_t<C::kBytes == 2, uint16_t, uint32_t>;
  constexpr bool SAVED_IS_H = (FLAGS & kSavedIsH) != 0;
  constexpr bool HAS_GH = (FLAGS & kGradH) != 0;
  constexpr bool HAS_DRES = (FLAGS & kRingDres) != 0;
  constexpr int MH = HAS_GH ? M : 1;  // grad_h elements (a dummy slot when absent)
  constexpr int PF = HAS_GH ? 1 : vg_plan::kRingPrefetch;
  constexpr int R = PF + 1;
  static_assert((FLAGS & (kRopeG | kRingTail | kRing8)) == 0, "plain rows only");
  static_assert(M == 4 || M == 8, "sixteen elements a lane spill past 256 VGPRs");
  __shared__ float red[2][kMaxWavesPerRow];
  extern __shared__ __align__(16) float dyn_lds[];  // dim floats: the row groups' combine

  const int tpr = a.tpr;
  const int grp = threadIdx.x / tpr;
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t slot = (int64_t)blockIdx.x * groups + grp;
  const int64_t nslots = (int64_t)gridDim.x * groups;
  const bool has_w = a.w != nullptr;
  const int64_t last = a.rows - 1;
  // column m of this lane (the row's last one past its end) and whether it is the lane's own
  int col[M];
  bool own[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int c = lt + m * tpr;
    own[m] = c < a.dim;
    col[m] = own[m] ? c : a.dim - 1;
  }
  float wf[M], acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    wf[m] = has_w ? Codec<WDT>::load1(a.w, col[m]) : 1.0f;
    acc[m] = 0.0f;
  }
  auto load_raw = [&](const void* base, int64_t i) -> uint32_t {
    return (uint32_t)__builtin_nontemporal_load(static_cast<const Raw*>(base) + i);
  };
  auto decode = [&](uint32_t u) -> float {
    if constexpr (DT == VELOGRAD_DTYPE_BF16) {
      return __builtin_bit_cast(float, u << 16);
    } else if constexpr (DT == VELOGRAD_DTYPE_F16) {
      return (float)__builtin_bit_cast(_Float16, (uint16_t)u);
    } else {
      return __builtin_bit_cast(float, u);
    }
  };
  auto store_one = [&](void* base, int64_t i, float f) {
    Raw v;
    if constexpr (DT == VELOGRAD_DTYPE_BF16) v = __builtin_bit_cast(uint16_t, (__bf16)f);
    else if constexpr (DT == VELOGRAD_DTYPE_F16) v = __builtin_bit_cast(uint16_t, (_Float16)f);
    else v = __builtin_bit_cast(uint32_t, f);
    __builtin_nontemporal_store(v, static_cast<Raw*>(base) + i);
  };

  uint32_t gr[R][M], sr[R][M], hr[R][MH];
  float rr[R];
  // Row `row`'s g, saved, grad_h elements and inv_rms; rows past the end read the last row.
  auto load_row = [&](int64_t row, uint32_t* gv, uint32_t* sv, uint32_t* hv, float& r) {
    const int64_t rw = row < a.rows ? row : last;
    r = a.inv_rms[rw];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      gv[m] = load_raw(a.g, rw * a.ld_g + col[m]);
      sv[m] = load_raw(a.saved, rw * a.ld_s + col[m]);
      if constexpr (HAS_GH) hv[m] = load_raw(a.gh, rw * a.ld_gh + col[m]);
    }
  };
  // The backward of one row (bwd_ring_kernel's, element by element); `ok` = the row exists.
  auto process = [&](const uint32_t* gv, const uint32_t* sv, const uint32_t* hv, float r,
                     int64_t row, bool ok, int it) {
    float gf[M], xh[M], gw[M];
    float s = 0.0f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      gf[m] = decode(gv[m]);
      xh[m] = decode(sv[m]);
      if constexpr (SAVED_IS_H) xh[m] = xh[m] * r;
      gw[m] = gf[m] * wf[m];
      const float t = gw[m] * xh[m];
      s += own[m] ? t : 0.0f;
    }
    s = row_sum(s, tpr, grp, red[it & 1]);
    const float mean = s / (float)a.dim;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float d = r * (gw[m] - xh[m] * mean);
      if constexpr (HAS_GH) d = d + decode(hv[m]);
      const bool store = ok && own[m];
      if (store) {
        store_one(a.dx, row * a.ld_dx + col[m], d);
        if constexpr (HAS_DRES) store_one(a.dres, row * a.ld_dres + col[m], d);
      }
      acc[m] += store ? gf[m] * xh[m] : 0.0f;
    }
  };

  // The walk and ring of bwd_ring_kernel.
  const int full = (int)(a.rows / nslots);
#pragma unroll
  for (int j = 0; j < PF; ++j) load_row(slot + (int64_t)j * nslots, gr[j], sr[j], hr[j], rr[j]);
  int it = 0;
  for (; it + R <= full; it += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int nb = (u + PF) % R;
      load_row(slot + (int64_t)(it + u + PF) * nslots, gr[nb], sr[nb], hr[nb], rr[nb]);
      process(gr[u], sr[u], hr[u], rr[u], slot + (int64_t)(it + u) * nslots, true, it + u);
    }
  }
#pragma unroll
  for (int u = 0; u < R; ++u) {
    if (it + u < a.iters) {
      const int nb = (u + PF) % R;
      if (it + u + PF < a.iters)
        load_row(slot + (int64_t)(it + u + PF) * nslots, gr[nb], sr[nb], hr[nb], rr[nb]);
      const int64_t row = slot + (int64_t)(it + u) * nslots;
      process(gr[u], sr[u], hr[u], rr[u], row, row < a.rows, it + u);
    }
  }

  if (a.partial == nullptr) return;
  // One fp32 partial row per workgroup; row groups added in group order through LDS.
  float* prow = a.partial + (int64_t)blockIdx.x * a.dim;
  if (groups == 1) {
#pragma unroll
    for (int m = 0; m < M; ++m)
      if (own[m]) prow[col[m]] = acc[m];
    return;
  }
  float* comb = dyn_lds;
  for (int gi = 0; gi < groups; ++gi) {
    if (grp == gi) {
#pragma unroll
      for (int m = 0; m < M; ++m)
        if (own[m]) comb[col[m]] = (gi == 0) ? acc[m] : comb[col[m]] + acc[m];
    }
    __syncthreads();
  }
  for (int q = threadIdx.x; q < a.dim; q += blockDim.x) prow[q] = comb[q];
}

// ------------------------------------------------------------------------------------------
// Backward with the fused RoPE gradient, ring-pipelined (launch_plan.h: plan_bwd_rope_ring, and with
// ANY plan_bwd_rope_ring_any: even rows of any length, streams at any element, the row's last chunk
// overlapping the one before it): NV (1 or 2) 16-byte chunks per thread, the saved tensor h, no
// grad_h or dres (the module's backward).  The walk, ring and steady loop are bwd_ring_kernel's: slot
// s walks rows s, s + S, ... (S slots), three row buffers, rows past the end read the last row, no branch
// around a memory operation in the steady loop.  Each thread keeps the rotation (cos, sin) of
// its pairs at the current row's position in float32 and advances it by S positions per row with
// the rotation through S * freq_j (formed in double once per walk, rounded to float).  Where a
// walk crosses the end of a sequence and S is a multiple or a divisor of rope_seq (rope_walk_ok,
// a.rope_back), the position returns to the walk's first one and the rotation to its first value;
// any other crossing evaluates the angles at the new position.  A walk that goes a.rope_anchor rows
// without either evaluates its angles afresh (double angle, exact reduction, float cos and sin), so
// no state is more than that less one float steps from an exact value (about 3 * 2^-24 of the pair
// per step): 16 rows, or 4 where the general path forms every angle at its row (launch_plan.h:
// rope_ring_anchor).  fp32 rows of ANY advance in double instead: their outputs hold what float
// steps lose (dx 2.0e-7 off the 64-bit one against 0.7e-7, 4096 x 3002), and they are bound by HBM (40.7
// / 40.6 us, 8192 x 2046).  The row group is a whole number of waves, so slots, rows and positions are
// wave-uniform and the walk's bookkeeping is scalar.  The walk is bound by its vector
// instructions as much as by HBM, so the row's decoded, rotated chunks stay in registers across
// the reduction, the weight is decoded once, sums of products use fused multiply-adds, and for a
// power-of-two dim the mean is s * (1 / dim), exact.  One chunk per thread runs within 128 VGPRs
// (two workgroups of fewer than 512 threads fit a CU); two chunks per thread, one workgroup per
// CU, within 256.
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int NV, bool ANY>
__global__ __launch_bounds__(vg_plan::kRingBlock, NV == 1 ? 4 : 2) void bwd_rope_ring_kernel(
    const BwdArgs a) {
  using C = Codec<DT>;
  constexpr int V = C::kVec;
  constexpr int P = V / 2;    // RoPE pairs per chunk
  constexpr int NP = NV * P;  // RoPE pairs per thread: pair e = k * P + q of chunk lt + k * tpr
  // The rotation state and step: float, or for fp32 rows of ANY double (see above).  One chunk per
  // thread keeps its pair frequencies and first rotations in LDS; with two they would not fit 64 KiB
  // beside the step rotations, so the first rotation is evaluated afresh at a return (also where the
  // step is double), and the frequencies are formed again there, except for the 2-byte rows of ANY,
  // which evaluate often.
  constexpr bool kDoubleRot = ANY && DT == VELOGRAD_DTYPE_F32;
  constexpr bool kFreqInLds = NV == 1 || (ANY && !kDoubleRot);
  constexpr bool kFirstInLds = NV == 1 && !kDoubleRot;
  using RotT = std::conditional_t<kDoubleRot, double, float>;
  typedef RotT Rot2 __attribute__((ext_vector_type(2)));
  constexpr int PF = vg_plan::kRingPrefetch;
  constexpr int R = PF + 1;
  static_assert(NV == 1 || NV == 2, "the RoPE ring takes one or two chunks per thread");
  __shared__ float red[2][kMaxWavesPerRow];
  // Dynamic LDS, pair-major so a wave reads consecutive entries: each thread's pair frequencies
  // (doubles, kFreqInLds), its step rotations (Rot2), its first rotations (float pairs, kFirstInLds),
  // then with several row groups dim floats for their combine (plan_bwd_rope_ring's lds_bytes).
  extern __shared__ __align__(16) float dyn_lds[];

  const int tpr = a.tpr;
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / tpr);
  const int lt = threadIdx.x - grp * tpr;
  const int groups = blockDim.x / tpr;
  const int64_t slot = (int64_t)blockIdx.x * groups + grp;
  const int64_t S = (int64_t)gridDim.x * groups;
  const int64_t last = a.rows - 1;
  const int64_t seq = a.rope_seq;
  const int64_t pos0 = slot % seq;
  const int bd = blockDim.x;
  const int tid = threadIdx.x;
  double* freq_lds = reinterpret_cast<double*>(dyn_lds);  // [NP][bd], kFreqInLds
  Rot2* step_lds = reinterpret_cast<Rot2*>(kFreqInLds ? freq_lds + NP * bd : freq_lds);  // [NP][bd]
  float2* first_lds = reinterpret_cast<float2*>(step_lds + NP * bd);  // [P][bd], kFirstInLds
  float* comb = reinterpret_cast<float*>(kFirstInLds ? first_lds + P * bd : first_lds);
  // 1 / dim is exact for a power of two, so s * (1 / dim) has the bits of s / dim
  const bool dim_pow2 = (a.dim & (a.dim - 1)) == 0;
  const float inv_dim = 1.0f / (float)a.dim;
  // first column of the lane's chunk k; the columns not its own to sum, and whether it has any
  auto col_of = [&](int k) { return ANY ? min((lt + k * tpr) * V, a.dim - V) : (lt + k * tpr) * V; };
  auto skip_of = [&](int k) { return ANY ? (lt + k * tpr) * V - col_of(k) : 0; };
  auto own = [&](int k) { return !ANY || skip_of(k) < V; };
  auto load_chunk = [&](const void* base, int64_t e) {
    if constexpr (ANY) return load16_any_stream<DT>(base, e);
    else return load16_stream<DT>(base, e);
  };
  // pair e's turns a position: base^(-2i/dim) / (2 pi), i its pair index in the row
  auto turns_of = [&](int e) {
    if constexpr (kFreqInLds) return freq_lds[e * bd + tid];
    else
      return rope_freq(col_of(e / P) / 2 + e % P, a.rope_c_hi, a.rope_c_lo) * kInv2PiD;
  };

  float wf[NV][V], acc[NV][V];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    WeightChunk<DT, WDT> wc;
    if constexpr (ANY) {
      if (a.w != nullptr) wc.load_any(a.w, col_of(k));
    } else {
      wc.load(a.w, col_of(k));
    }
    wc.unpack(a.w != nullptr, wf[k]);
#pragma unroll
    for (int i = 0; i < V; ++i) acc[k][i] = 0.0f;
  }
  // one pair at a time (the walk needs the registers): its turns a position, the first of a chunk
  // from exp2, each next one by the double ratio; the rotation through S positions in double
  double g = 0.0;
#pragma unroll 1
  for (int e = 0; e < NP; ++e) {
    if (e % P == 0)
      g = vg_plan::rope_first_turns(
          col_of(e / P) / 2, ANY ? P : 1, a.rope_ratio,
          [&](int i) { return rope_freq(i, a.rope_c_hi, a.rope_c_lo) * kInv2PiD; });
    else
      g = g * a.rope_ratio;
    const double rev = (double)S * g;
    double sv, cv;
    cos_sin_turn_d(rev - rint(rev), cv, sv);
    step_lds[e * bd + tid] = Rot2{(RotT)cv, (RotT)sv};
    if constexpr (kFreqInLds) freq_lds[e * bd + tid] = g;
    if constexpr (kFirstInLds) {
      // the rotation at the walk's first position: double angle, reduced exactly, float cos and sin
      float s0, c0;
      cos_sin_turn(rope_frac((double)pos0 * g), c0, s0);
      first_lds[e * bd + tid] = float2{c0, s0};
    }
  }
  RotT cr[NP], sr[NP];
  // the rotations at position p evaluated afresh: double angle, exact reduction, float cos and sin
  auto evaluate_at = [&](int64_t p) {
#pragma unroll
    for (int e = 0; e < NP; ++e) {
      float c, sn;
      cos_sin_turn(rope_frac((double)p * turns_of(e)), c, sn);
      cr[e] = c;
      sr[e] = sn;
    }
  };
  auto restore_first = [&]() {
    if constexpr (kFirstInLds) {
#pragma unroll
      for (int e = 0; e < NP; ++e) {
        const float2 f0 = first_lds[e * bd + tid];
        cr[e] = f0.x;
        sr[e] = f0.y;
      }
    } else {
      evaluate_at(pos0);
    }
  };
  restore_first();
  int64_t pos = pos0;
  int since = 0;  // float steps taken since the state was last exact

  u32x4 gr[R][NV], hr[R][NV];
  float rr[R];
  // Row `row`'s grad_y and h chunks and inv_rms; rows past the end read the last row.
  auto load_row = [&](int64_t row, u32x4* gv, u32x4* hv, float& r) {
    const int64_t rw = row < a.rows ? row : last;
    r = a.inv_rms[rw];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      gv[k] = load_chunk(a.g, rw * a.ld_g + col_of(k));
      hv[k] = load_chunk(a.saved, rw * a.ld_s + col_of(k));
    }
  };
  // The backward of one row (bwd_vec_kernel's with kSavedIsH | kRopeG); `ok` = the row exists.
  auto process = [&](const u32x4* gv, const u32x4* hv, float r, int64_t row, bool ok, int it) {
    float gf[NV][V], xh[NV][V];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      C::unpack(gv[k], gf[k]);
      // inverse rotation of each pair (y0, y1) -> (y0 c + y1 s, y1 c - y0 s)
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const float c = (float)cr[k * P + q], sn = (float)sr[k * P + q];
        const float g0 = gf[k][2 * q], g1 = gf[k][2 * q + 1];
        gf[k][2 * q] = __builtin_fmaf(g0, c, g1 * sn);
        gf[k][2 * q + 1] = __builtin_fmaf(g1, c, -(g0 * sn));
      }
      C::unpack(hv[k], xh[k]);
#pragma unroll
      for (int i = 0; i < V; ++i) xh[k][i] = xh[k][i] * r;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float t = __builtin_fmaf(gf[k][i] * wf[k][i], xh[k][i], s);
        s = ANY && i < skip_of(k) ? s : t;
      }
    }
    s = row_sum(s, tpr, grp, red[it & 1]);
    const float m = dim_pow2 ? s * inv_dim : s / (float)a.dim;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      float d[V];
#pragma unroll
      for (int i = 0; i < V; ++i) d[i] = r * __builtin_fmaf(-xh[k][i], m, gf[k][i] * wf[k][i]);
      if (ok && own(k)) {
        if constexpr (ANY) store16_any_stream<DT>(a.dx, row * a.ld_dx + col_of(k), C::pack(d));
        else store16_stream<DT>(a.dx, row * a.ld_dx + col_of(k), C::pack(d));
      }
#pragma unroll
      for (int i = 0; i < V; ++i) {
        acc[k][i] = ok ? __builtin_fmaf(gf[k][i], xh[k][i], acc[k][i]) : acc[k][i];
        // the row's sums are done here: its g and xhat are not held into the next row
        asm volatile("" : "+v"(acc[k][i]));
      }
    }
    // the next row's angles: the walk's first position again, evaluated afresh after
    // a.rope_anchor rows, or one step of S positions on (each thread reads only the
    // LDS entries it wrote, in program order: no barrier)
    pos += S;
    ++since;
    if (pos >= seq) {
      since = 0;
      if (a.rope_back) {
        if (!ANY || pos - S != pos0) restore_first();  // (a walk that has not left it keeps it)
        pos = pos0;
      } else {
        pos = (row + S) % seq;
        evaluate_at(pos);
      }
    } else if (since == a.rope_anchor) {
      since = 0;
      evaluate_at(pos);
    } else {
#pragma unroll
      for (int e = 0; e < NP; ++e) {
        const Rot2 st = step_lds[e * bd + tid];
        const RotT cn = __builtin_elementwise_fma(cr[e], st.x, -(sr[e] * st.y));
        sr[e] = __builtin_elementwise_fma(sr[e], st.x, cr[e] * st.y);
        cr[e] = cn;
      }
    }
  };

  // Row j of the walk sits in buffer j % R; processing row j first issues row j + PF's loads
  // into buffer (j + PF) % R, the one row j - 1 has just released.
  const int full = (int)(a.rows / S);  // iterations in which every slot has a row
#pragma unroll
  for (int j = 0; j < PF; ++j) load_row(slot + (int64_t)j * S, gr[j], hr[j], rr[j]);
  int it = 0;
  for (; it + R <= full; it += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int nb = (u + PF) % R;
      load_row(slot + (int64_t)(it + u + PF) * S, gr[nb], hr[nb], rr[nb]);
      process(gr[u], hr[u], rr[u], slot + (int64_t)(it + u) * S, true, it + u);
    }
  }
  // The last (up to R) iterations, some of whose slots may have no row.
#pragma unroll
  for (int u = 0; u < R; ++u) {
    if (it + u < a.iters) {
      const int nb = (u + PF) % R;
      if (it + u + PF < a.iters)
        load_row(slot + (int64_t)(it + u + PF) * S, gr[nb], hr[nb], rr[nb]);
      const int64_t row = slot + (int64_t)(it + u) * S;
      process(gr[u], hr[u], rr[u], row, row < a.rows, it + u);
    }
  }

  if (a.partial == nullptr) return;
  // One fp32 partial row per workgroup; row groups added in group order through LDS.
  float* prow = a.partial + (int64_t)blockIdx.x * a.dim;
  if (groups == 1) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if constexpr (ANY) {
#pragma unroll
        for (int i = 0; i < V; ++i)
          if (i >= skip_of(k)) prow[col_of(k) + i] = acc[k][i];
        continue;
      }
#pragma unroll
      for (int q = 0; q < V / 4; ++q)
        store16<VELOGRAD_DTYPE_F32>(prow, col_of(k) + 4 * q,
                                    Codec<VELOGRAD_DTYPE_F32>::pack(&acc[k][4 * q]));
    }
    return;
  }
  for (int gi = 0; gi < groups; ++gi) {
    if (grp == gi) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const int c = col_of(k) + i;
          if (i >= skip_of(k)) comb[c] = (gi == 0) ? acc[k][i] : comb[c] + acc[k][i];
        }
      }
    }
    __syncthreads();
  }
  if constexpr (ANY) {
    for (int q = threadIdx.x; q < a.dim; q += blockDim.x) prow[q] = comb[q];
    return;
  }
  for (int q = threadIdx.x; q < a.dim / 4; q += blockDim.x)
    store16<VELOGRAD_DTYPE_F32>(prow, 4 * (int64_t)q, *reinterpret_cast<const u32x4*>(comb + 4 * q));
}

// ------------------------------------------------------------------------------------------
// Backward, any dim / alignment: one row slot per workgroup, two passes per row; the slot's
// dweight partial row is accumulated in place (each column owned by one thread).
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int FLAGS>
__global__ __launch_bounds__(kGenericBlock) void bwd_generic_kernel(const BwdArgs a) {
  using C = Codec<DT>;
  using CW = Codec<WDT>;
  constexpr bool SAVED_IS_H = (FLAGS & kSavedIsH) != 0;
  constexpr bool HAS_GH = (FLAGS & kGradH) != 0;
  constexpr bool ROPE = (FLAGS & kRopeG) != 0;
  __shared__ float red[2][kGenericBlock / kWave];
  // The dweight columns of the slot's rows, summed in row order: in dynamic LDS (dim floats)
  // where the launch gave it (vg_plan::generic_bwd_lds_bytes), else in the slot's partial row
  // in global memory, each column then always touched by the same thread.
  extern __shared__ __align__(16) float acc_lds[];
  const int64_t slot = blockIdx.x;
  const int64_t nslots = gridDim.x;
  const bool has_w = a.w != nullptr;
  const bool has_dres = a.dres != nullptr;
  float* prow = a.partial != nullptr ? a.partial + slot * (int64_t)a.dim : nullptr;
  const bool acc_in_lds = vg_plan::generic_bwd_lds_bytes(a.dim, prow != nullptr) != 0;
  auto accumulate = [&](int j, float p, int it) {
    if (acc_in_lds) acc_lds[j] = (it == 0) ? p : acc_lds[j] + p;
    else prow[j] = (it == 0) ? p : prow[j] + p;
  };
  // the 16-byte middle of a row (see fwd_generic_kernel) moves a column between threads from
  // row to row, so it needs the LDS sums when dweight is requested
  const bool body_allowed = !ROPE && (prow == nullptr || acc_in_lds);

  for (int it = 0; it < a.iters; ++it) {
    const int64_t row = slot + (int64_t)it * nslots;
    if (row >= a.rows) break;  // uniform across the workgroup
    const float rr = a.inv_rms[row];
    // element j's contributions given its (rotated-back) gradient gf: to the row sum, then to
    // dx, dres and the partial row
    auto xh_at = [&](int j) {
      float xh = C::load1(a.saved, row * a.ld_s + j);
      if constexpr (SAVED_IS_H) xh = xh * rr;
      return xh;
    };
    auto sum_term = [&](int j, float gf) {
      const float gw = has_w ? gf * CW::load1(a.w, j) : gf;
      return gw * xh_at(j);
    };
    auto finish = [&](int j, float gf, float m) {
      const float xh = xh_at(j);
      const float gw = has_w ? gf * CW::load1(a.w, j) : gf;
      float d = rr * (gw - xh * m);
      if constexpr (HAS_GH) d = d + C::load1(a.gh, row * a.ld_gh + j);
      C::store1(a.dx, row * a.ld_dx + j, d);
      if (has_dres) C::store1(a.dres, row * a.ld_dres + j, d);
      if (prow != nullptr) accumulate(j, gf * xh, it);
    };
    float s = 0.0f;
    if constexpr (ROPE) {
      // one rotation per pair (y0, y1) -> (y0 c + y1 s, y1 c - y0 s) and pass
      const int64_t pos = row % a.rope_seq;
      const int half = a.dim / 2;
      auto grad_pair = [&](int i, double fr, float& g0, float& g1) {
        float c, sn;
        rope_cos_sin_f(pos, fr, c, sn);
        const float y0 = C::load1(a.g, row * a.ld_g + 2 * i);
        const float y1 = C::load1(a.g, row * a.ld_g + 2 * i + 1);
        g0 = y0 * c + y1 * sn;
        g1 = y1 * c - y0 * sn;
      };
      RopeFreqWalk fw(threadIdx.x, blockDim.x, a.rope_c_hi, a.rope_c_lo);
      for (int i = threadIdx.x; i < half; i += blockDim.x) {
        float g0, g1;
        grad_pair(i, fw.next(), g0, g1);
        s += sum_term(2 * i, g0);
        s += sum_term(2 * i + 1, g1);
      }
      s = row_sum(s, blockDim.x, 0, red[it & 1]);
      const float m = s / (float)a.dim;
      RopeFreqWalk fw2(threadIdx.x, blockDim.x, a.rope_c_hi, a.rope_c_lo);
      for (int i = threadIdx.x; i < half; i += blockDim.x) {
        float g0, g1;
        grad_pair(i, fw2.next(), g0, g1);
        finish(2 * i, g0, m);
        finish(2 * i + 1, g1, m);
      }
    } else {
      int head = a.dim, nbody = 0;
      if (body_allowed) {
        const uintptr_t mis = row_offset16(a.g, row * a.ld_g, C::kBytes);
        if (mis % C::kBytes == 0 && row_offset16(a.saved, row * a.ld_s, C::kBytes) == mis &&
            row_offset16(a.dx, row * a.ld_dx, C::kBytes) == mis &&
            (!has_dres || row_offset16(a.dres, row * a.ld_dres, C::kBytes) == mis) &&
            (!HAS_GH || row_offset16(a.gh, row * a.ld_gh, C::kBytes) == mis)) {
          head = (int)(((16 - mis) & 15) / C::kBytes);
          if (head > a.dim) head = a.dim;
          nbody = (a.dim - head) / C::kVec;
        }
      }
      const int tail = head + nbody * C::kVec;
      const int nscalar = a.dim - nbody * C::kVec;
      auto scalar_j = [&](int t) { return t < head ? t : tail + (t - head); };
      const uintptr_t w_align = has_w ? row_offset16(a.w, head, CW::kBytes) : 0;
      // A thread's first KR body chunks of g and the saved tensor stay in registers from the
      // first pass to the second (rows of up to KR * 256 chunks read once); chunks past them
      // are read in the first pass with the normal cache policy and again, non-temporally,
      // in the second (normally from L2).
      constexpr int KR = 4;
      // (grad_h's register chunks too, loaded with them: its loads in the second pass, after
      // the row reduction, cost a memory wait per row)
      u32x4 gk[KR], sk[KR], hk[HAS_GH ? KR : 1];
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int c = threadIdx.x + k * blockDim.x;
        gk[k] = u32x4{0u, 0u, 0u, 0u};
        sk[k] = u32x4{0u, 0u, 0u, 0u};
        if constexpr (HAS_GH) hk[k] = u32x4{0u, 0u, 0u, 0u};
        if (c < nbody) {
          const int64_t j = head + (int64_t)c * C::kVec;
          gk[k] = load16_stream<DT>(a.g, row * a.ld_g + j);
          sk[k] = load16_stream<DT>(a.saved, row * a.ld_s + j);
          if constexpr (HAS_GH) hk[k] = load16_stream<DT>(a.gh, row * a.ld_gh + j);
        }
      }
      // With a body, the head and tail are fewer than two chunks' worth of elements (one per
      // thread at most): loaded with the body chunks, so a row waits for memory once per pass
      // instead of three times.
      const bool few_scalar = nbody > 0;
      int j_s = 0;
      float g_s = 0.0f, x_s = 0.0f, w_s = 1.0f;
      float gh_s = 0.0f;
      if (few_scalar && (int)threadIdx.x < nscalar) {
        j_s = scalar_j(threadIdx.x);
        g_s = C::load1(a.g, row * a.ld_g + j_s);
        x_s = C::load1(a.saved, row * a.ld_s + j_s);
        if (has_w) w_s = CW::load1(a.w, j_s);
        if constexpr (HAS_GH) gh_s = C::load1(a.gh, row * a.ld_gh + j_s);
        if constexpr (SAVED_IS_H) x_s = x_s * rr;
      }
      // the body chunk at element j: g and x-hat decoded, g * w formed as sum_term and finish do
      auto body_chunk = [&](const u32x4& gq, const u32x4& sq, int64_t j, float* gf, float* gw,
                            float* xh) {
        C::unpack(gq, gf);
        C::unpack(sq, xh);
        float wf[C::kVec];
        if (has_w) weight_run<DT, WDT>(a.w, j, w_align, wf);
#pragma unroll
        for (int i = 0; i < C::kVec; ++i) {
          if constexpr (SAVED_IS_H) xh[i] = xh[i] * rr;
          gw[i] = has_w ? gf[i] * wf[i] : gf[i];
        }
      };
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int c = threadIdx.x + k * blockDim.x;
        if (c < nbody) {
          float gf[C::kVec], gw[C::kVec], xh[C::kVec];
          body_chunk(gk[k], sk[k], head + (int64_t)c * C::kVec, gf, gw, xh);
#pragma unroll
          for (int i = 0; i < C::kVec; ++i) s += gw[i] * xh[i];
        }
      }
      for (int c = threadIdx.x + KR * blockDim.x; c < nbody; c += blockDim.x) {
        const int64_t j = head + (int64_t)c * C::kVec;
        float gf[C::kVec], gw[C::kVec], xh[C::kVec];
        body_chunk(load16<DT>(a.g, row * a.ld_g + j), load16<DT>(a.saved, row * a.ld_s + j), j,
                   gf, gw, xh);
#pragma unroll
        for (int i = 0; i < C::kVec; ++i) s += gw[i] * xh[i];
      }
      if (few_scalar) {
        if ((int)threadIdx.x < nscalar) s += (has_w ? g_s * w_s : g_s) * x_s;
      } else {
        for (int t = threadIdx.x; t < nscalar; t += blockDim.x) {
          const int j = scalar_j(t);
          s += sum_term(j, C::load1(a.g, row * a.ld_g + j));
        }
      }
      s = row_sum(s, blockDim.x, 0, red[it & 1]);
      const float m = s / (float)a.dim;
      // dx of a body chunk, its stores and its dweight terms
      // `ghq`: the chunk's grad_h when it is already in registers, else null (loaded here)
      auto finish_chunk = [&](int64_t j, const float* gf, const float* gw, const float* xh,
                              const u32x4* ghq) {
        float d[C::kVec];
#pragma unroll
        for (int i = 0; i < C::kVec; ++i) d[i] = rr * (gw[i] - xh[i] * m);
        if constexpr (HAS_GH) {
          float ghf[C::kVec];
          C::unpack(ghq != nullptr ? *ghq : load16_stream<DT>(a.gh, row * a.ld_gh + j), ghf);
#pragma unroll
          for (int i = 0; i < C::kVec; ++i) d[i] = d[i] + ghf[i];
        }
        const u32x4 pk = C::pack(d);
        store16_stream<DT>(a.dx, row * a.ld_dx + j, pk);
        if (has_dres) store16_stream<DT>(a.dres, row * a.ld_dres + j, pk);
        if (prow != nullptr) {
          float pv[C::kVec];
#pragma unroll
          for (int i = 0; i < C::kVec; ++i) pv[i] = gf[i] * xh[i];
          // the widest LDS accesses the chunk's first column allows: the dweight reduction costs
          // 11.9 / 13.8 / 27.0 us at 16384 x 4100 / 4102 / 4099 bf16, whose chunks start 16-byte
          // / 8-byte / any aligned in LDS; one word per element in a layout that spreads a
          // chunk's columns across lanes (no bank conflicts, 8 accesses a chunk) cost ~25 us at
          // all three
          if (acc_in_lds && (j & 3) == 0) {
            float4* a4 = reinterpret_cast<float4*>(acc_lds + j);
#pragma unroll
            for (int q = 0; q < C::kVec / 4; ++q) {
              const float4 pq = {pv[4 * q], pv[4 * q + 1], pv[4 * q + 2], pv[4 * q + 3]};
              a4[q] = (it == 0) ? pq : a4[q] + pq;
            }
          } else if (acc_in_lds && (j & 1) == 0) {
            float2* a2 = reinterpret_cast<float2*>(acc_lds + j);
#pragma unroll
            for (int q = 0; q < C::kVec / 2; ++q) {
              const float2 pq = {pv[2 * q], pv[2 * q + 1]};
              a2[q] = (it == 0) ? pq : a2[q] + pq;
            }
          } else {
#pragma unroll
            for (int i = 0; i < C::kVec; ++i) accumulate((int)j + i, pv[i], it);
          }
        }
      };
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int c = threadIdx.x + k * blockDim.x;
        if (c < nbody) {
          const int64_t j = head + (int64_t)c * C::kVec;
          float gf[C::kVec], gw[C::kVec], xh[C::kVec];
          body_chunk(gk[k], sk[k], j, gf, gw, xh);
          finish_chunk(j, gf, gw, xh, HAS_GH ? &hk[k] : nullptr);
        }
      }
      for (int c = threadIdx.x + KR * blockDim.x; c < nbody; c += blockDim.x) {
        const int64_t j = head + (int64_t)c * C::kVec;
        float gf[C::kVec], gw[C::kVec], xh[C::kVec];
        body_chunk(load16_stream<DT>(a.g, row * a.ld_g + j),
                   load16_stream<DT>(a.saved, row * a.ld_s + j), j, gf, gw, xh);
        finish_chunk(j, gf, gw, xh, nullptr);
      }
      if (few_scalar) {
        if ((int)threadIdx.x < nscalar) {
          // finish's arithmetic on the register copies
          const float gw = has_w ? g_s * w_s : g_s;
          float d = rr * (gw - x_s * m);
          if constexpr (HAS_GH) d = d + gh_s;
          C::store1(a.dx, row * a.ld_dx + j_s, d);
          if (has_dres) C::store1(a.dres, row * a.ld_dres + j_s, d);
          if (prow != nullptr) accumulate(j_s, g_s * x_s, it);
        }
      } else {
        for (int t = threadIdx.x; t < nscalar; t += blockDim.x) {
          const int j = scalar_j(t);
          finish(j, C::load1(a.g, row * a.ld_g + j), m);
        }
      }
    }
  }
  if (acc_in_lds) {
    __syncthreads();
    for (int j = threadIdx.x; j < a.dim; j += blockDim.x) prow[j] = acc_lds[j];
  }
}

// ------------------------------------------------------------------------------------------
// dweight stage 2: dweight[j] = sum over partial rows p = 0..nparts-1, in a fixed order.
// A workgroup owns 64 columns; wave w sums rows p = w, w + W, ... and the W wave sums are
// added in wave order.  The kernel is bound by the round trips to the partial rows that another
// XCD wrote, not by their bytes, so a wave's rows are read in batches of 16 loads in flight (four
// for at most 64 partial rows), the last batch filled up with the last row (read, not added): one
// round trip up to 256 partial rows.  A loop over the rows past the last whole batch waited for
// each, up to 15 times with under 256 partial rows (short tensors, several row groups a
// workgroup).  The whole backward, such a loop / batches (bf16, graph replays, us): 512 x 768 7.8 /
// 6.0, 512 x 1024 8.7 / 6.8, 128 x 4096 9.4 / 7.6, 200 x 4096 10.7 / 8.1, 512 x 4096 9.3 / 9.0.
// ------------------------------------------------------------------------------------------
constexpr int kReduceBlock = 1024;
__global__ __launch_bounds__(kReduceBlock) void dweight_reduce_kernel(const float* partial,
                                                                       int32_t nparts,
                                                                       int32_t dim,
                                                                       float* dweight) {
  constexpr int kWaves = kReduceBlock / kWave;
  __shared__ float red[kWaves][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int col = blockIdx.x * kWave + lane;
  float s = 0.0f;
  auto sum_rows = [&](auto batch) {
    constexpr int kBatch = decltype(batch)::value;
    for (int p = wave; p < nparts; p += kBatch * kWaves) {
      float v[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; ++b)
        v[b] = partial[(int64_t)min(p + b * kWaves, nparts - 1) * dim + col];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) s = p + b * kWaves < nparts ? s + v[b] : s;
    }
  };
  if (col < dim) {
    if (nparts <= 4 * kWaves) sum_rows(std::integral_constant<int, 4>{});
    else sum_rows(std::integral_constant<int, 16>{});
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && col < dim) {
    float t = red[0][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) t += red[w][lane];
    dweight[col] = t;
  }
}

// Launch-shape knobs, read once per process from the environment (for tuning sweeps; the
// defaults are the measured best on MI355X).  Results do not depend on them except through the
// dweight summation order, which stays fixed for a given setting.
struct Tuning {
  int fwd_nv;             // preferred 16-byte chunks per thread, forward (0 = automatic)
  int bwd_nv;             // same, backward
  int bwd_waves_per_cu;   // resident waves per CU targeted by the persistent backward grid
  int bwd_block;          // upper bound on backward workgroup size (row groups per workgroup)
  int bwd_ring;           // 1: the ring-pipelined backward where the rows suit it
  int ring_block;         // upper bound on the ring backward's workgroup size
  int ring_wgs_per_cu;    // ring backward workgroups per CU (1 or 2)
  int fwd_elem;           // 1: the element-strided forward where the chunked kernels cannot go
};

const Tuning& tuning() {
  static const Tuning t = {
      env_int("VELOGRAD_FWD_NV", 0, 0, kMaxNV),
      env_int("VELOGRAD_BWD_NV", 0, 0, kMaxNV),
      env_int("VELOGRAD_BWD_WAVES_PER_CU", 16, 1, 64),
      env_int("VELOGRAD_BWD_BLOCK", 1024, 64, 1024),
      env_int("VELOGRAD_BWD_RING", 1, 0, 1),
      env_int("VELOGRAD_BWD_RING_BLOCK", vg_plan::kRingBlock, 64, vg_plan::kRingBlock),
      env_int("VELOGRAD_BWD_RING_WGS_PER_CU", 1, 1, 2),
      env_int("VELOGRAD_FWD_ELEM", 1, 0, 1),
  };
  return t;
}

// `one_stream`: no residual, so the row kernel reads x and writes y only.  `epilogue`: a
// quantised output (fp8 per row, MX), whose two row reductions prefer fewer waves per row.
RowPlan plan_fwd(int64_t dim, int elem_bytes, bool aligned, bool one_stream, bool epilogue) {
  return vg_plan::plan_rows(dim, elem_bytes, aligned, tuning().fwd_nv,
                            epilogue     ? vg_plan::kFwdOrderEpilogue
                            : one_stream ? vg_plan::kFwdOrderOneStream
                                         : vg_plan::kFwdOrder);
}

// `aligned8`: every stream starts on an 8-byte boundary (the weight on a 16-byte one), the
// condition of the ring's kRing8 rows; `aligned_elem`: on their own elements' (kRingAny).
BwdPlan plan_bwd(int64_t rows, int64_t dim, int elem_bytes, bool aligned, bool aligned8,
                 bool aligned_elem, bool has_gh, bool dx_is_gh, int cus, bool rope) {
  const Tuning& t = tuning();
  if (!rope && t.bwd_ring) {
    const BwdPlan r = vg_plan::plan_bwd_ring(rows, dim, elem_bytes, aligned, cus, t.bwd_nv,
                                             t.ring_block, t.ring_wgs_per_cu);
    if (r.ring) return r;
    if (aligned8) {
      const BwdPlan r8 = vg_plan::plan_bwd_ring8(rows, dim, elem_bytes, cus, t.ring_block,
                                                 t.ring_wgs_per_cu);
      if (r8.ring) return r8;
    }
  }
  if (rope && t.bwd_ring) {
    const BwdPlan r = vg_plan::plan_bwd_rope_ring(rows, dim, elem_bytes, aligned, cus);
    if (r.ring) return r;
    const BwdPlan ra = vg_plan::plan_bwd_rope_ring_any(rows, dim, elem_bytes, cus);
    const bool whole = aligned && dim % (16 / elem_bytes) == 0;  // (bwd_vec_kernel's otherwise)
    if (ra.ring && aligned_elem &&
        (whole || !vg_plan::rope_bwd_generic_first(rows, dim, elem_bytes, cus)))
      return ra;
  }
  if (rope)
    return vg_plan::plan_bwd_rope(rows, dim, elem_bytes, aligned, cus, t.bwd_nv, t.bwd_block,
                                  t.bwd_waves_per_cu);
  const BwdPlan p = vg_plan::plan_bwd(rows, dim, elem_bytes, aligned, cus, t.bwd_nv, t.bwd_block,
                                      t.bwd_waves_per_cu);
  // Rows the chunked kernels cannot take: short ones (bwd_elem_first) in the element-strided ring,
  // the others in chunks from any element (unless dx is grad_h itself, see kRingAny), else
  // element-strided as far as that goes.  Measured on MI355X, 16384 rows, elements (generic past
  // 4096) / chunks, us: bf16 99 11.8 / 13.7, 301 18.3 / 14.8, 1001 29.6 / 23.6, 2047 48.8 / 40.1, 2050 69.1 /
  // 43.4, 3002 75.0 / 56.4, 4095 90.8 / 83.5, 8192 x 4099 68.2 / 49.5, 8192 x 8191 119 / 89; with
  // grad_h 1001 36.2 / 29.1, 3002 99.5 / 71.1, 4095 119.5 / 111.4; fp32 401 20.8 / 21.7 but with
  // grad_h 25.2 / 23.3, 1025 45.9 / 39.9, 2047 76.0 / 72.7.
  if (!p.rp.vec && t.bwd_ring) {
    if (!vg_plan::bwd_elem_first(rows, dim, elem_bytes, has_gh, cus) && aligned_elem &&
        !dx_is_gh) {
      const BwdPlan a = vg_plan::plan_bwd_ring_any(rows, dim, elem_bytes, cus);
      if (a.ring) return a;
    }
    const BwdPlan e = vg_plan::plan_bwd_ring_elem(rows, dim, elem_bytes, cus);
    if (e.elem_m > 0) return e;
  }
  return p;
}

bool ld_ok(int64_t ld, int elem_bytes) { return ((ld * elem_bytes) & 15) == 0; }
bool ld_ok8(int64_t ld, int elem_bytes) { return ((ld * elem_bytes) & 7) == 0; }
bool elem_ok_ptr(const void* p, int bytes) {
  return (reinterpret_cast<uintptr_t>(p) & (uintptr_t)(bytes - 1)) == 0;
}
bool aligned8p(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; }

// ------------------------------------------------------------------------------------------
// Typed launchers.
// ------------------------------------------------------------------------------------------
template <int DT, int WDT, int OUT>
void launch_fwd(const FwdArgs& a, const RowPlan& p, hipStream_t st) {
  if (!p.vec) {
    hipLaunchKernelGGL((fwd_generic_kernel<DT, WDT, OUT>), dim3((uint32_t)a.rows), dim3(p.block),
                       0, st, a);
    return;
  }
  if constexpr (OUT != kOutRopeI) {  // (the RoPE output's rows run in fwd_rope_tile_kernel)
    const dim3 grid((uint32_t)((a.rows + p.groups - 1) / p.groups));
    const dim3 block(p.block);
    if constexpr (OUT == kOutDtype) {
      if (vg_plan::fwd_late_h(p)) {
        switch (p.nv) {
#define VG_LATE_H(N)                                                                          \
  case N:                                                                                     \
    hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, N, kOutDtypeLateH>), grid, block, 0, st, a); \
    break;
          VG_LATE_H(1)
          VG_LATE_H(2)
          VG_LATE_H(3)
          default: VG_LATE_H(4)
#undef VG_LATE_H
        }
        return;
      }
    }
    switch (p.nv) {
      case 1: hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 1, OUT>), grid, block, 0, st, a); break;
      case 2: hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 2, OUT>), grid, block, 0, st, a); break;
      case 3: hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 3, OUT>), grid, block, 0, st, a); break;
      default: hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 4, OUT>), grid, block, 0, st, a); break;
    }
  }
}

// Rows of any length and alignment (fwd_vec_kernel's ANY), planned by plan_any_rows.
template <int DT, int WDT, int OUT, int ROWS>
void launch_fwd_any_rows(const FwdArgs& a, const RowPlan& p, hipStream_t st) {
  const dim3 grid((uint32_t)((a.rows + p.groups - 1) / p.groups)), block(p.block);
  if (p.nv == 1) {
    hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 1, OUT, ROWS>), grid, block, 0, st, a);
    return;
  }
  if constexpr (OUT == kOutDtype && ROWS == kRowsAnyRes) {
    if (vg_plan::fwd_late_h(p)) {
      hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 2, kOutDtypeLateH, ROWS>), grid, block, 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((fwd_vec_kernel<DT, WDT, 2, OUT, ROWS>), grid, block, 0, st, a);
}

template <int DT, int WDT, int OUT>
void launch_fwd_any(const FwdArgs& a, const RowPlan& p, hipStream_t st) {
  if (a.res != nullptr) launch_fwd_any_rows<DT, WDT, OUT, kRowsAnyRes>(a, p, st);
  else launch_fwd_any_rows<DT, WDT, OUT, kRowsAnyNoRes>(a, p, st);
}

// The norm + RoPE tiles (vg_plan::RopeTilePlan).
template <int DT, int WDT, int NV, bool RES, bool ANY>
void launch_rope_tile(const FwdArgs& a, const vg_plan::RopeTilePlan& p, hipStream_t st) {
  const dim3 grid((uint32_t)p.wgs), block(p.rp.block);
  constexpr int kMost = vg_plan::rope_tile_most(Codec<DT>::kBytes, NV, RES);
  if constexpr (kMost >= 4) {
    if (p.tile == 4) {
      hipLaunchKernelGGL((fwd_rope_tile_kernel<DT, WDT, NV, RES, 4, ANY>), grid, block, 0, st, a);
      return;
    }
  }
  if constexpr (kMost >= 2) {
    if (p.tile == 2) {
      hipLaunchKernelGGL((fwd_rope_tile_kernel<DT, WDT, NV, RES, 2, ANY>), grid, block, 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((fwd_rope_tile_kernel<DT, WDT, NV, RES, 1, ANY>), grid, block, 0, st, a);
}

template <int DT, int WDT>
void launch_rope_tiles(const FwdArgs& a, const vg_plan::RopeTilePlan& p, bool any, hipStream_t st) {
  const int which = (p.rp.nv == 2 ? 4 : 0) | (a.res != nullptr ? 2 : 0) | (any ? 1 : 0);
  switch (which) {
    case 0: launch_rope_tile<DT, WDT, 1, false, false>(a, p, st); break;
    case 1: launch_rope_tile<DT, WDT, 1, false, true>(a, p, st); break;
    case 2: launch_rope_tile<DT, WDT, 1, true, false>(a, p, st); break;
    case 3: launch_rope_tile<DT, WDT, 1, true, true>(a, p, st); break;
    case 4: launch_rope_tile<DT, WDT, 2, false, false>(a, p, st); break;
    case 5: launch_rope_tile<DT, WDT, 2, false, true>(a, p, st); break;
    case 6: launch_rope_tile<DT, WDT, 2, true, false>(a, p, st); break;
    default: launch_rope_tile<DT, WDT, 2, true, true>(a, p, st); break;
  }
}

// Rows of element-strided lanes (fwd_elem_kernel): `p` from plan_elem_rows.
template <int DT, int WDT>
void launch_fwd_elem(const FwdArgs& a, const RowPlan& p, hipStream_t st) {
  const dim3 grid((uint32_t)((a.rows + p.groups - 1) / p.groups)), block(p.block);
  hipLaunchKernelGGL((fwd_elem_kernel<DT, WDT, kFwdElemPerLane>), grid, block, 0, st, a);
}

template <int DT, int WDT, int F>
void launch_bwd_ring(const BwdArgs& a, const BwdPlan& b, hipStream_t st) {
  const dim3 grid((uint32_t)b.wgs), block(b.rp.block);
  if constexpr (Codec<DT>::kBytes == 2) {
    // rows of 8-byte alignment with a half chunk at their end: one chunk per thread
    if (b.x8) {
      if ((int64_t)b.rp.tpr * Codec<DT>::kVec != a.dim - Codec<DT>::kVec / 2)
        hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 1, F | kRing8 | kRingTail>), grid, block,
                           b.lds_bytes, st, a);
      else
        hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 1, F | kRing8>), grid, block, b.lds_bytes,
                           st, a);
      return;
    }
  }
  if (b.any) {
    if (b.rp.nv == 1)
      hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 1, F | kRingAny>), grid, block, b.lds_bytes, st,
                         a);
    else
      hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 2, F | kRingAny>), grid, block, b.lds_bytes, st,
                         a);
    return;
  }
  // rows of fewer chunks than the row group's lanes take the idle-lane variant
  if ((int64_t)b.rp.nv * b.rp.tpr * Codec<DT>::kVec != a.dim) {
    if (b.rp.nv == 1)
      hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 1, F | kRingTail>), grid, block, b.lds_bytes,
                         st, a);
    else
      hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 2, F | kRingTail>), grid, block, b.lds_bytes,
                         st, a);
    return;
  }
  if (b.rp.nv == 1)
    hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 1, F>), grid, block, b.lds_bytes, st, a);
  else
    hipLaunchKernelGGL((bwd_ring_kernel<DT, WDT, 2, F>), grid, block, b.lds_bytes, st, a);
}

template <int DT, int WDT, int F>
void launch_bwd_ring_elem(const BwdArgs& a, const BwdPlan& b, hipStream_t st) {
  const dim3 grid((uint32_t)b.wgs), block(b.rp.block);
  if (b.elem_m == 4)
    hipLaunchKernelGGL((bwd_ring_elem_kernel<DT, WDT, 4, F>), grid, block, b.lds_bytes, st, a);
  else
    hipLaunchKernelGGL((bwd_ring_elem_kernel<DT, WDT, 8, F>), grid, block, b.lds_bytes, st, a);
}

template <int DT, int WDT, int F>
void launch_bwd_flags(const BwdArgs& a, const BwdPlan& b, hipStream_t st) {
  const RowPlan& p = b.rp;
  const dim3 grid((uint32_t)b.wgs);
  const dim3 block(p.block);
  const size_t lds = b.lds_bytes;
  if constexpr ((F & kRopeG) == 0) {
    if (b.elem_m > 0) {
      if (a.dres != nullptr)
        launch_bwd_ring_elem<DT, WDT, F | kRingDres>(a, b, st);
      else
        launch_bwd_ring_elem<DT, WDT, F>(a, b, st);
      return;
    }
  }
  if (!p.vec) {
    hipLaunchKernelGGL((bwd_generic_kernel<DT, WDT, F>), grid, block,
                       vg_plan::generic_bwd_lds_bytes(a.dim, a.partial != nullptr), st, a);
    return;
  }
  if constexpr ((F & kRopeG) == 0) {
    if (b.ring) {
      if (a.dres != nullptr)
        launch_bwd_ring<DT, WDT, F | kRingDres>(a, b, st);
      else
        launch_bwd_ring<DT, WDT, F>(a, b, st);
      return;
    }
  }
  if constexpr ((F & kRopeG) != 0) {
    if (b.ring) {
      switch (p.nv * 2 + (b.any ? 1 : 0)) {
        case 2:
          hipLaunchKernelGGL((bwd_rope_ring_kernel<DT, WDT, 1, false>), grid, block, lds, st, a);
          break;
        case 3:
          hipLaunchKernelGGL((bwd_rope_ring_kernel<DT, WDT, 1, true>), grid, block, lds, st, a);
          break;
        case 4:
          hipLaunchKernelGGL((bwd_rope_ring_kernel<DT, WDT, 2, false>), grid, block, lds, st, a);
          break;
        default:
          hipLaunchKernelGGL((bwd_rope_ring_kernel<DT, WDT, 2, true>), grid, block, lds, st, a);
          break;
      }
      return;
    }
    if (b.rope_direct) {
      constexpr int FD = (F & ~kRopeG) | kRopeDirect;
      switch (p.nv) {
        case 1: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 1, FD>), grid, block, lds, st, a); break;
        case 2: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 2, FD>), grid, block, lds, st, a); break;
        case 3: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 3, FD>), grid, block, lds, st, a); break;
        default: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 4, FD>), grid, block, lds, st, a); break;
      }
      return;
    }
    // NV 4 is never planned with the RoPE gradient (max_block_for_nv_rope); it is not compiled
    switch (p.nv) {
      case 1: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 1, F>), grid, block, lds, st, a); break;
      case 2: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 2, F>), grid, block, lds, st, a); break;
      default: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 3, F>), grid, block, lds, st, a); break;
    }
  } else {
    switch (p.nv) {
      case 1: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 1, F>), grid, block, lds, st, a); break;
      case 2: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 2, F>), grid, block, lds, st, a); break;
      case 3: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 3, F>), grid, block, lds, st, a); break;
      default: hipLaunchKernelGGL((bwd_vec_kernel<DT, WDT, 4, F>), grid, block, lds, st, a); break;
    }
  }
}

template <int DT, int WDT>
void launch_bwd(const BwdArgs& a, bool saved_is_h, bool rope, const BwdPlan& b, hipStream_t st) {
  if (rope) {  // the module form: the saved tensor is h, no residual-stream gradient
    launch_bwd_flags<DT, WDT, kSavedIsH | kRopeG>(a, b, st);
    return;
  }
  const int flags = (saved_is_h ? kSavedIsH : 0) | (a.gh != nullptr ? kGradH : 0);
  switch (flags) {
    case 0: launch_bwd_flags<DT, WDT, 0>(a, b, st); break;
    case kSavedIsH: launch_bwd_flags<DT, WDT, kSavedIsH>(a, b, st); break;
    case kGradH: launch_bwd_flags<DT, WDT, kGradH>(a, b, st); break;
    default: launch_bwd_flags<DT, WDT, kSavedIsH | kGradH>(a, b, st); break;
  }
}

// Supported (dtype, w_dtype) pairs: weight in the activation dtype, or fp32.
bool types_ok(int32_t dt, int32_t wdt) {
  if (elem_bytes_of(dt) == 0) return false;
  return wdt == dt || wdt == VELOGRAD_DTYPE_F32;
}

#define VG_DISPATCH_TYPES(DT, WDT, CALL)                                       \
  do {                                                                         \
    if ((DT) == VELOGRAD_DTYPE_F32) {                                          \
      constexpr int kD = VELOGRAD_DTYPE_F32, kW = VELOGRAD_DTYPE_F32;          \
      CALL;                                                                    \
    } else if ((DT) == VELOGRAD_DTYPE_BF16 && (WDT) == VELOGRAD_DTYPE_BF16) {  \
      constexpr int kD = VELOGRAD_DTYPE_BF16, kW = VELOGRAD_DTYPE_BF16;        \
      CALL;                                                                    \
    } else if ((DT) == VELOGRAD_DTYPE_BF16) {                                  \
      constexpr int kD = VELOGRAD_DTYPE_BF16, kW = VELOGRAD_DTYPE_F32;         \
      CALL;                                                                    \
    } else if ((WDT) == VELOGRAD_DTYPE_F16) {                                  \
      constexpr int kD = VELOGRAD_DTYPE_F16, kW = VELOGRAD_DTYPE_F16;          \
      CALL;                                                                    \
    } else {                                                                   \
      constexpr int kD = VELOGRAD_DTYPE_F16, kW = VELOGRAD_DTYPE_F32;          \
      CALL;                                                                    \
    }                                                                          \
  } while (0)

size_t workspace_bytes_for(int64_t rows, int64_t dim, int cus) {
  const Tuning& t = tuning();
  return vg_plan::bwd_workspace_bytes(rows, dim, cus, t.bwd_nv, t.bwd_block, t.bwd_waves_per_cu,
                                      t.ring_block, t.ring_wgs_per_cu);
}

// ------------------------------------------------------------------------------------------
// Scratch of the allocation-free backward (velograd_rmsnorm_residual_bwd_noalloc): the dweight
// partial rows live in this file-scope device array instead of a caller workspace.  Each GPU
// the library runs on holds its own copy, at its own address, until the process ends.  In host
// code `scratch` names a host-side stand-in, never the device memory: the device address comes
// from hipGetSymbolAddress, once per device with that device current, and only that address is
// passed to kernels.  Nothing in it needs to start at zero (stage 1 writes every partial row it
// hands to stage 2 before stage 2 reads it), so no call clears it.  Calls that overlap on one
// GPU (two streams, or two host threads) share the array and race.
// ------------------------------------------------------------------------------------------
constexpr size_t kNoAllocScratchBytes = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

std::once_flag g_scratch_once[kMaxDevices];
void* g_scratch_ptr[kMaxDevices];
hipError_t g_scratch_err[kMaxDevices];

// Device address of `scratch` on `device` (the current device), or null with the HIP error.
void* scratch_on(int device, hipError_t* err) {
  std::call_once(g_scratch_once[device], [device] {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    g_scratch_err[device] = e;
    g_scratch_ptr[device] = (e == hipSuccess) ? p : nullptr;
  });
  *err = g_scratch_err[device];
  return g_scratch_ptr[device];
}

// Shared by the forward entry points.  `out` is the epilogue (kOut*): for kOutFp8Row y holds one
// e4m3 byte per element and y_scale one fp32 per row; for the MX modes y holds e4m3 bytes or
// e2m1 nibbles and mx_scale one E8M0 byte per 32 elements.  ld_y (and ld_mx) count bytes then.
int32_t run_fwd(const char* what, int out, const void* x, const void* residual,
                const void* weight, void* y, float* y_scale, uint8_t* mx_scale, int64_t ld_mx,
                void* h, float* inv_rms, int64_t rows, int64_t dim, int64_t ld_x,
                int64_t ld_res, int64_t ld_y, int64_t ld_h, int32_t dtype, int32_t w_dtype,
                float eps, float ms_floor, void* hip_stream, int64_t rope_seq = 0,
                float rope_theta = 0.0f) {
  const bool mx = out == kOutMxE4M3 || out == kOutMxE2M1;
  if (!types_ok(dtype, w_dtype))
    return fail(VELOGRAD_ERR_UNSUPPORTED_DTYPE,
                "%s: unsupported dtype/w_dtype pair (%d, %d): weight must be the activation "
                "dtype or fp32",
                what, (int)dtype, (int)w_dtype);
  if (rows < 0 || dim <= 0 || dim > INT32_MAX)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: invalid shape rows=%lld dim=%lld", what,
                (long long)rows, (long long)dim);
  if (!(ms_floor >= 0.0f) || !__builtin_isfinite(ms_floor))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "%s: min_mean_sq=%g must be finite and >= 0", what, (double)ms_floor);
  if (out == kOutRopeI && (dim % 2 != 0 || rope_seq < 1 || (rows > 0 && rows % rope_seq != 0) ||
                           !(rope_theta > 0.0f) || !__builtin_isfinite(rope_theta)))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "%s: RoPE needs an even dim (%lld), seq >= 1 dividing rows (seq=%lld rows=%lld) "
                "and a finite base > 0 (%g)",
                what, (long long)dim, (long long)rope_seq, (long long)rows, (double)rope_theta);
  if (mx && dim % vg_mx::kBlock != 0)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "%s: dim=%lld must be a multiple of the 32-element MX block", what,
                (long long)dim);
  if (rows == 0) {
    clear_error();
    return 0;
  }
  if (x == nullptr || y == nullptr)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: x and y must not be NULL", what);
  if (out == kOutFp8Row && y_scale == nullptr)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: y_scale must not be NULL", what);
  if (mx && mx_scale == nullptr)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: scales must not be NULL", what);
  if (residual == nullptr) h = nullptr;  // h is x itself
  const int64_t y_row = out == kOutMxE2M1 ? dim / 2 : dim;  // y row length in its own units
  if (ld_x < dim || ld_y < y_row || (residual && ld_res < dim) || (h && ld_h < dim) ||
      (mx && ld_mx < dim / vg_mx::kBlock))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "%s: row strides too small (ld_x=%lld ld_res=%lld ld_y=%lld ld_h=%lld "
                "ld_scales=%lld for dim=%lld)",
                what, (long long)ld_x, (long long)ld_res, (long long)ld_y, (long long)ld_h,
                (long long)ld_mx, (long long)dim);
  const void* extra_out = out == kOutFp8Row ? (const void*)y_scale : (const void*)mx_scale;
  if (y == x || y == residual || (h && (h == x || h == residual || h == y)) ||
      (extra_out && (extra_out == x || extra_out == residual || extra_out == y ||
                     (h && extra_out == h))))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: outputs must not alias inputs", what);
  if (rows > INT32_MAX)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: rows=%lld exceeds the grid limit", what,
                (long long)rows);

  const int eb = elem_bytes_of(dtype);
  // Bytes of y per 16-byte input chunk: 16 (activation dtype), 16 / eb (e4m3), 8 / eb (e2m1).
  bool y_aligned;
  if (out == kOutDtype || out == kOutRopeI) {
    y_aligned = aligned16(y) && ld_ok(ld_y, eb);
  } else {
    const int64_t cb = out == kOutMxE2M1 ? 8 / eb : 16 / eb;
    y_aligned = ((uintptr_t)y % (uintptr_t)cb) == 0 && ld_y % cb == 0;
  }
  const bool aligned = aligned16(x) && ld_ok(ld_x, eb) && y_aligned &&
                       (!residual || (aligned16(residual) && ld_ok(ld_res, eb))) &&
                       (!h || (aligned16(h) && ld_ok(ld_h, eb))) && (!weight || aligned16(weight));
  RowPlan p = plan_fwd(dim, eb, aligned && out != kOutRopeI, residual == nullptr,
                       out == kOutFp8Row || mx);
  // rows the chunked layout does not fit, on element boundaries
  const bool aligned_elem = elem_ok_ptr(x, eb) &&
                            ((out != kOutDtype && out != kOutRopeI) || elem_ok_ptr(y, eb)) &&
                            elem_ok_ptr(residual, eb) && elem_ok_ptr(h, eb) &&
                            elem_ok_ptr(weight, elem_bytes_of(w_dtype));
  // The shortest of them go element by element, several rows a workgroup; the others in chunks
  // from any element (plan_any_rows), longer ones than that fits in the generic kernel.  Measured
  // on MI355X, 16384 rows with a residual, the kernels before (elements up to 1024, the generic
  // kernel past them) / chunks, us: bf16 17 7.2 / 8.7, 99 10.0 / 9.8, 255 14.0 / 10.8, 1001 45.4 /
  // 24.4, 2047 59.2 / 50.6, 4095 99.7 / 94.2, 8192 x 8191 103.2 / 93.3, 8192 x 12001 146.4 / 137.2,
  // fp32 1001 57.9 / 47.5, 8192 x 4099 105.8 / 90.6; rows of 8n + 4 elements in 8-byte halves 4100
  // 93.0 / 92.4, 2052 48.4 / 48.7; without a residual 2047 41.3 / 25.8; quantised to fp8 (generic
  // kernel) 255 30.6 / 11.3, 2047 192 / 44.4, 4095 404 / 86.4.
  bool any = false;
  int elem_m = 0;
  if (!p.vec && out == kOutDtype && dim <= kFwdElemMaxDim && tuning().fwd_elem) {
    elem_m = vg_plan::elem_per_lane(dim);
    if (elem_m > 0) p = vg_plan::plan_elem_rows(dim);
  } else if (!p.vec && out != kOutRopeI && aligned_elem) {
    const RowPlan pa =
        vg_plan::plan_any_rows(rows, dim, eb, residual != nullptr, out != kOutDtype);
    if (pa.vec) {
      p = pa;
      any = true;
    }
  }
  const bool elem_ok = p.tpr % kWave == 0 && p.tpr >= kWave && p.groups >= 1 &&
                       p.block == p.tpr * p.groups && p.block <= vg_plan::kRingBlock &&
                       (int64_t)elem_m * p.tpr >= dim;
  if (elem_m > 0 ? !elem_ok : !vg_plan::row_plan_valid(p, any ? dim / (16 / eb) * (16 / eb) : dim, eb))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "%s: internal launch plan rejected (dim=%lld)",
                what, (long long)dim);

  FwdArgs a;
  a.x = x;
  a.res = residual;
  a.w = weight;
  a.y = y;
  a.h = h;
  a.inv_rms = inv_rms;
  a.y_scale = y_scale;
  a.mx_scale = mx_scale;
  a.ld_mx = ld_mx;
  a.rows = rows;
  a.ld_x = ld_x;
  a.ld_res = ld_res;
  a.ld_y = ld_y;
  a.ld_h = ld_h;
  a.dim = (int32_t)dim;
  a.tpr = p.tpr;
  a.eps = eps;
  a.ms_floor = ms_floor;
  a.rope_seq = rope_seq > 0 ? rope_seq : 1;
  a.rope_half = (int32_t)(dim / 2);
  a.run_log2 = vg_plan::xcd_run_log2(dim * eb, p.groups, !p.vec && elem_m == 0);
  const double c = (rope_theta > 0.0f && dim >= 2) ? log2((double)rope_theta) / (double)(dim / 2)
                                                   : 0.0;
  a.rope_c_hi = (float)c;
  a.rope_c_lo = (float)(c - (double)a.rope_c_hi);
  a.rope_log2_step = -c;
  a.rope_ratio = exp2(-c);
  a.rope_small_step = rope_theta >= 1.0f;
  a.rope_across = false;
  a.rope_step_rad = kTwoPiD;
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  if (out == kOutRopeI && aligned_elem) {
    const vg_plan::RopeTilePlan t =
        vg_plan::plan_rope_tiles(rows, dim, eb, rope_seq, residual != nullptr);
    if (t.rp.vec) {
      a.tpr = t.rp.tpr;
      a.rope_across = t.across;
      if (t.across) a.rope_step_rad = 0.0;
      a.run_log2 = vg_plan::xcd_run_log2(dim * eb * t.tile, t.rp.groups);
      const bool any = !aligned || dim % (16 / eb) != 0;
      VG_DISPATCH_TYPES(dtype, w_dtype, (launch_rope_tiles<kD, kW>(a, t, any, st)));
      return check_launch(what);
    }
  }
  switch (out) {
#define VG_FWD_OUT(O)                                                                  \
  case O:                                                                              \
    if (any)                                                                           \
      VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd_any<kD, kW, O>(a, p, st)));        \
    else                                                                               \
      VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd<kD, kW, O>(a, p, st)));            \
    break;
    VG_FWD_OUT(kOutFp8Row)
    VG_FWD_OUT(kOutMxE4M3)
    VG_FWD_OUT(kOutMxE2M1)
#undef VG_FWD_OUT
    case kOutRopeI: VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd<kD, kW, kOutRopeI>(a, p, st))); break;
    default:
      if (any)
        VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd_any<kD, kW, kOutDtype>(a, p, st)));
      else if (elem_m > 0)
        VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd_elem<kD, kW>(a, p, st)));
      else
        VG_DISPATCH_TYPES(dtype, w_dtype, (launch_fwd<kD, kW, kOutDtype>(a, p, st)));
      break;
  }
  return check_launch(what);
}

// The backward behind both C entry points.  rope_seq > 0: grad_y is the gradient of the
// interleaved-RoPE output (velograd_rmsnorm_rope_bwd); the saved tensor is then h.
int32_t run_bwd(const void* grad_y, const void* saved, int32_t saved_is_h, const void* weight,
                const float* inv_rms, const void* grad_h, void* dx, void* dres, float* dweight,
                void* workspace, size_t ws_bytes, int64_t rows, int64_t dim, int64_t ld_g,
                int64_t ld_saved, int64_t ld_grad_h, int64_t ld_dx, int64_t ld_dres,
                int32_t dtype, int32_t w_dtype, void* hip_stream, int64_t rope_seq = 0,
                float rope_base = 0.0f, bool static_scratch = false) {
  if (!types_ok(dtype, w_dtype))
    return fail(VELOGRAD_ERR_UNSUPPORTED_DTYPE,
                "bwd: unsupported dtype/w_dtype pair (%d, %d): weight must be the activation "
                "dtype or fp32",
                (int)dtype, (int)w_dtype);
  if (rows < 0 || dim <= 0 || dim > INT32_MAX)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "bwd: invalid shape rows=%lld dim=%lld",
                (long long)rows, (long long)dim);
  if (weight == nullptr) dweight = nullptr;  // no weight, no weight gradient (fused.py:62-65)
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  if (rows == 0) {
    // Sum over zero rows: dweight = 0, written by stage 2 with no partial rows.
    if (dweight != nullptr) {
      hipLaunchKernelGGL(dweight_reduce_kernel, dim3((uint32_t)((dim + kWave - 1) / kWave)),
                         dim3(kReduceBlock), 0, st, (const float*)nullptr, 0, (int32_t)dim,
                         dweight);
      return check_launch("velograd_rmsnorm_residual_bwd(dweight)");
    }
    clear_error();
    return 0;
  }
  if (grad_y == nullptr || saved == nullptr || inv_rms == nullptr || dx == nullptr)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "bwd: grad_y, saved, inv_rms and dx must not be NULL");
  if (ld_g < dim || ld_saved < dim || ld_dx < dim || (dres && ld_dres < dim) ||
      (grad_h && ld_grad_h < dim))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "bwd: row strides must be >= dim (ld_g=%lld ld_saved=%lld ld_grad_h=%lld "
                "ld_dx=%lld ld_dres=%lld)",
                (long long)ld_g, (long long)ld_saved, (long long)ld_grad_h, (long long)ld_dx,
                (long long)ld_dres);
  // dx may be grad_h itself (accumulating in place: each element is read before it is written
  // by the same thread); no other output may alias an input.
  if (dx == grad_y || dx == saved || dx == dres ||
      (dres && (dres == grad_y || dres == saved || dres == grad_h)))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "bwd: outputs must not alias inputs");
  if (grad_h == dx && ld_grad_h != ld_dx)
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "bwd: dx may alias grad_h only with the same row stride");

  int device = 0;
  if (hipGetDevice(&device) != hipSuccess)
    return fail(VELOGRAD_ERR_DEVICE_QUERY, "bwd: hipGetDevice failed");
  const int cus = cu_count(device);
  if (cus <= 0) return fail(VELOGRAD_ERR_DEVICE_QUERY, "bwd: cannot query the CU count");

  const int eb = elem_bytes_of(dtype);
  const bool aligned = aligned16(grad_y) && aligned16(saved) && aligned16(dx) &&
                       ld_ok(ld_g, eb) && ld_ok(ld_saved, eb) && ld_ok(ld_dx, eb) &&
                       (!dres || (aligned16(dres) && ld_ok(ld_dres, eb))) &&
                       (!grad_h || (aligned16(grad_h) && ld_ok(ld_grad_h, eb))) &&
                       (!weight || aligned16(weight));
  const bool aligned8 = aligned8p(grad_y) && aligned8p(saved) && aligned8p(dx) &&
                        ld_ok8(ld_g, eb) && ld_ok8(ld_saved, eb) && ld_ok8(ld_dx, eb) &&
                        (!dres || (aligned8p(dres) && ld_ok8(ld_dres, eb))) &&
                        (!grad_h || (aligned8p(grad_h) && ld_ok8(ld_grad_h, eb))) &&
                        (!weight || aligned16(weight));
  const bool rope = rope_seq > 0;
  const bool aligned_elem = elem_ok_ptr(grad_y, eb) && elem_ok_ptr(saved, eb) &&
                            elem_ok_ptr(dx, eb) && elem_ok_ptr(dres, eb) &&
                            elem_ok_ptr(grad_h, eb) && elem_ok_ptr(weight, elem_bytes_of(w_dtype));
  BwdPlan plan = plan_bwd(rows, dim, eb, aligned, aligned8, aligned_elem, grad_h != nullptr,
                          dx == grad_h, cus, rope);
  // the columns the row plan lays out
  const int64_t plan_dim = plan.x8    ? dim - 4
                           : plan.any ? (dim + 16 / eb - 1) / (16 / eb) * (16 / eb)
                                      : dim;
  // bwd_vec_kernel's RoPE walk keeps its step rotations (two floats per pair: dim floats) in the
  // same dynamic LDS as the group combine, one after the other.
  if (rope && plan.rp.vec && !plan.ring && !plan.rope_direct)
    plan.lds_bytes = (size_t)dim * sizeof(float);
  const bool elem_ok =
      plan.elem_m > 0 && !rope && plan.rp.tpr % kWave == 0 && plan.rp.tpr >= kWave &&
      plan.rp.groups >= 1 && plan.rp.block == plan.rp.tpr * plan.rp.groups &&
      plan.rp.block <= vg_plan::kRingBlock && (int64_t)plan.elem_m * plan.rp.tpr >= dim;
  if ((plan.elem_m > 0 ? !elem_ok : !vg_plan::row_plan_valid(plan.rp, plan_dim, eb)) ||
      plan.wgs < 1 || plan.wgs > INT32_MAX || plan.lds_bytes > 64 * 1024 ||
      (plan.ring && plan.any && (dim < 16 / eb || plan.rp.block > vg_plan::kRingBlock)) ||
      (plan.ring && !rope &&
       ((plan.any ? dim < 16 / eb || plan.rp.nv > vg_plan::kRingMaxNV
                  : !vg_plan::ring_eligible(plan.rp, plan_dim, eb)) ||
        plan.rp.block > vg_plan::kRingBlock)) ||
      (plan.x8 && (rope || !plan.ring || eb != 2 || dim % 8 != 4 || plan.rp.nv != 1 ||
                   !aligned8)) ||
      (plan.ring && rope && !plan.any && !vg_plan::rope_ring_eligible(plan.rp, dim, eb)) ||
      (rope && plan.rp.vec && !plan.ring && !plan.rope_direct &&
       plan.rp.block > vg_plan::max_block_for_nv_rope(plan.rp.nv)) ||
      (plan.rope_direct && (!rope || plan.rp.block > vg_plan::max_block_for_nv(plan.rp.nv))))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "bwd: internal launch plan rejected (dim=%lld)",
                (long long)dim);
  const int64_t slots = plan.wgs * plan.rp.groups;  // row slots walking the rows

  float* partial = nullptr;
  if (dweight != nullptr) {
    size_t need = (size_t)plan.wgs * (size_t)dim * sizeof(float);
    if (static_scratch) {
      // velograd_rmsnorm_residual_bwd_noalloc: the partial rows go to the library's own array.
      // Wide rows that the chunked kernels cannot take are held to the generic kernel's need, which
      // is never less than the plan's (it has at least one workgroup a CU or a row).
      if (plan.any && dim > vg_plan::kRingElemMaxM * vg_plan::kRingBlock)
        need = (size_t)vg_plan::plan_bwd(rows, dim, eb, false, cus, tuning().bwd_nv,
                                         tuning().bwd_block, tuning().bwd_waves_per_cu).wgs *
               (size_t)dim * sizeof(float);
      if (need > kNoAllocScratchBytes)
        return fail(VELOGRAD_ERR_WORKSPACE_TOO_SMALL,
                    "bwd_noalloc: dweight needs %zu bytes of scratch for rows=%lld dim=%lld, above "
                    "the fixed maximum of %zu bytes; pass a workspace to "
                    "velograd_rmsnorm_residual_bwd instead",
                    need, (long long)rows, (long long)dim, kNoAllocScratchBytes);
      if (device < 0 || device >= kMaxDevices)
        return fail(VELOGRAD_ERR_DEVICE_QUERY, "bwd_noalloc: device %d out of range", device);
      hipError_t e = hipSuccess;
      workspace = scratch_on(device, &e);
      if (workspace == nullptr)
        return fail((int32_t)e, "bwd_noalloc: hipGetSymbolAddress of the scratch failed: %s",
                    hipGetErrorString(e));
      ws_bytes = kNoAllocScratchBytes;
    }
    if (workspace == nullptr || ws_bytes < need)
      return fail(VELOGRAD_ERR_WORKSPACE_TOO_SMALL,
                  "bwd: workspace of %zu bytes given, %zu needed", ws_bytes, need);
    if (!aligned16(workspace))
      return fail(VELOGRAD_ERR_INVALID_ARGUMENT, "bwd: workspace must be 16-byte aligned");
    partial = static_cast<float*>(workspace);
  }

  BwdArgs a;
  a.g = grad_y;
  a.saved = saved;
  a.w = weight;
  a.inv_rms = inv_rms;
  a.gh = grad_h;
  a.dx = dx;
  a.dres = dres;
  a.partial = partial;
  a.rows = rows;
  a.ld_g = ld_g;
  a.ld_gh = ld_grad_h;
  a.ld_s = ld_saved;
  a.ld_dx = ld_dx;
  a.ld_dres = ld_dres;
  a.dim = (int32_t)dim;
  a.tpr = plan.rp.tpr;
  a.iters = (int32_t)((rows + slots - 1) / slots);
  a.rope_seq = rope ? rope_seq : 1;
  const double c = rope ? log2((double)rope_base) / (double)(dim / 2) : 0.0;
  a.rope_c_hi = (float)c;
  a.rope_c_lo = (float)(c - (double)a.rope_c_hi);
  a.rope_ratio = exp2(-c);
  a.rope_back = rope && vg_plan::rope_walk_ok(rows, slots, rope_seq);
  a.rope_anchor = vg_plan::rope_ring_anchor(plan.any && !(aligned && dim % (16 / eb) == 0));
  VG_DISPATCH_TYPES(dtype, w_dtype, (launch_bwd<kD, kW>(a, saved_is_h != 0, rope, plan, st)));
  int32_t rc = check_launch(rope ? "velograd_rmsnorm_rope_bwd" : "velograd_rmsnorm_residual_bwd");
  if (rc != 0 || dweight == nullptr) return rc;
  hipLaunchKernelGGL(dweight_reduce_kernel, dim3((uint32_t)((dim + kWave - 1) / kWave)),
                     dim3(kReduceBlock), 0, st, (const float*)partial, (int32_t)plan.wgs,
                     (int32_t)dim, dweight);
  return check_launch("velograd_rmsnorm_residual_bwd(dweight)");
}

}  // namespace

// ------------------------------------------------------------------------------------------
// C ABI.
// ------------------------------------------------------------------------------------------
extern "C" {

VELOGRAD_API const char* velograd_kernels_version(void) { return VG_VERSION_STRING; }

VELOGRAD_API const char* velograd_kernels_last_error(void) { return g_last_error; }

VELOGRAD_API size_t velograd_rmsnorm_residual_bwd_workspace_bytes(int64_t rows, int64_t dim,
                                                                  int32_t device) {
  return workspace_bytes_for(rows, dim, cu_count(device));
}

VELOGRAD_API int32_t velograd_rmsnorm_residual_fwd(const void* x, const void* residual,
                                                   const void* weight, void* y, void* h,
                                                   float* inv_rms, int64_t rows, int64_t dim,
                                                   int64_t ld_x, int64_t ld_res, int64_t ld_y,
                                                   int64_t ld_h, int32_t dtype, int32_t w_dtype,
                                                   float eps, void* hip_stream) {
  return run_fwd("velograd_rmsnorm_residual_fwd", kOutDtype, x, residual, weight, y, nullptr,
                 nullptr, 0, h, inv_rms, rows, dim, ld_x, ld_res, ld_y, ld_h, dtype, w_dtype,
                 eps, 0.0f, hip_stream);
}

VELOGRAD_API int32_t velograd_rmsnorm_fwd(const void* x, const void* residual,
                                          const void* weight, void* y, void* h, float* inv_rms,
                                          int64_t rows, int64_t dim, int64_t ld_x,
                                          int64_t ld_res, int64_t ld_y, int64_t ld_h,
                                          int32_t dtype, int32_t w_dtype, float eps,
                                          float min_mean_sq, void* hip_stream) {
  return run_fwd("velograd_rmsnorm_fwd", kOutDtype, x, residual, weight, y, nullptr, nullptr, 0,
                 h, inv_rms, rows, dim, ld_x, ld_res, ld_y, ld_h, dtype, w_dtype, eps,
                 min_mean_sq, hip_stream);
}

VELOGRAD_API int32_t velograd_rmsnorm_rope_fwd(
    const void* x, const void* residual, const void* weight, void* y, void* h, float* inv_rms,
    int64_t rows, int64_t dim, int64_t ld_x, int64_t ld_res, int64_t ld_y, int64_t ld_h,
    int64_t seq, int32_t dtype, int32_t w_dtype, float eps, float min_mean_sq, float base,
    void* hip_stream) {
  return run_fwd("velograd_rmsnorm_rope_fwd", kOutRopeI, x, residual, weight, y, nullptr,
                 nullptr, 0, h, inv_rms, rows, dim, ld_x, ld_res, ld_y, ld_h, dtype, w_dtype, eps,
                 min_mean_sq, hip_stream, seq, base);
}

VELOGRAD_API int32_t velograd_rmsnorm_residual_fwd_fp8(
    const void* x, const void* residual, const void* weight, uint8_t* y_fp8, float* y_scale,
    void* h, float* inv_rms, int64_t rows, int64_t dim, int64_t ld_x, int64_t ld_res,
    int64_t ld_y, int64_t ld_h, int32_t dtype, int32_t w_dtype, float eps, void* hip_stream) {
  return run_fwd("velograd_rmsnorm_residual_fwd_fp8", kOutFp8Row, x, residual, weight, y_fp8,
                 y_scale, nullptr, 0, h, inv_rms, rows, dim, ld_x, ld_res, ld_y, ld_h, dtype,
                 w_dtype, eps, 0.0f, hip_stream);
}

VELOGRAD_API int32_t velograd_rmsnorm_residual_fwd_mx(
    const void* x, const void* residual, const void* weight, uint8_t* y_q, uint8_t* y_scales,
    void* h, float* inv_rms, int64_t rows, int64_t dim, int64_t ld_x, int64_t ld_res,
    int64_t ld_yq, int64_t ld_scales, int64_t ld_h, int32_t dtype, int32_t w_dtype,
    int32_t mx_format, float eps, void* hip_stream) {
  if (mx_format != VELOGRAD_MX_E4M3 && mx_format != VELOGRAD_MX_E2M1)
    return fail(VELOGRAD_ERR_UNSUPPORTED_DTYPE,
                "velograd_rmsnorm_residual_fwd_mx: unsupported mx_format %d", (int)mx_format);
  return run_fwd("velograd_rmsnorm_residual_fwd_mx",
                 mx_format == VELOGRAD_MX_E4M3 ? kOutMxE4M3 : kOutMxE2M1, x, residual, weight,
                 y_q, nullptr, y_scales, ld_scales, h, inv_rms, rows, dim, ld_x, ld_res, ld_yq,
                 ld_h, dtype, w_dtype, eps, 0.0f, hip_stream);
}

VELOGRAD_API int32_t velograd_rmsnorm_residual_bwd(
    const void* grad_y, const void* saved, int32_t saved_is_h, const void* weight,
    const float* inv_rms, const void* grad_h, void* dx, void* dres, float* dweight,
    void* workspace, size_t ws_bytes, int64_t rows, int64_t dim, int64_t ld_g, int64_t ld_saved,
    int64_t ld_grad_h, int64_t ld_dx, int64_t ld_dres, int32_t dtype, int32_t w_dtype,
    void* hip_stream) {
  return run_bwd(grad_y, saved, saved_is_h, weight, inv_rms, grad_h, dx, dres, dweight, workspace,
                 ws_bytes, rows, dim, ld_g, ld_saved, ld_grad_h, ld_dx, ld_dres, dtype, w_dtype,
                 hip_stream);
}

VELOGRAD_API int32_t velograd_rmsnorm_residual_bwd_noalloc(
    const void* grad_y, const void* saved, int32_t saved_is_h, const void* weight,
    const float* inv_rms, const void* grad_h, void* dx, void* dres, float* dweight, int64_t rows,
    int64_t dim, int64_t ld_g, int64_t ld_saved, int64_t ld_grad_h, int64_t ld_dx,
    int64_t ld_dres, int32_t dtype, int32_t w_dtype, void* hip_stream) {
  return run_bwd(grad_y, saved, saved_is_h, weight, inv_rms, grad_h, dx, dres, dweight, nullptr,
                 0, rows, dim, ld_g, ld_saved, ld_grad_h, ld_dx, ld_dres, dtype, w_dtype,
                 hip_stream, 0, 0.0f, /*static_scratch=*/true);
}

VELOGRAD_API int32_t velograd_rmsnorm_rope_bwd(
    const void* grad_y, const void* h, const void* weight, const float* inv_rms, void* dx,
    float* dweight, void* workspace, size_t ws_bytes, int64_t rows, int64_t dim, int64_t ld_g,
    int64_t ld_h, int64_t ld_dx, int64_t seq, int32_t dtype, int32_t w_dtype, float base,
    void* hip_stream) {
  if (dim % 2 != 0 || seq < 1 || (rows > 0 && rows % seq != 0) || !(base > 0.0f) ||
      !__builtin_isfinite(base))
    return fail(VELOGRAD_ERR_INVALID_ARGUMENT,
                "velograd_rmsnorm_rope_bwd: RoPE needs an even dim (%lld), seq >= 1 dividing rows "
                "(seq=%lld rows=%lld) and a finite base > 0 (%g)",
                (long long)dim, (long long)seq, (long long)rows, (double)base);
  return run_bwd(grad_y, h, 1, weight, inv_rms, nullptr, dx, nullptr, dweight, workspace,
                 ws_bytes, rows, dim, ld_g, ld_h, dim, ld_dx, dim, dtype, w_dtype, hip_stream,
                 seq, base);
}

}  // extern "C"
