// pbf_math.h -- device arithmetic of the PBF step.
//
// Every file of the library is compiled with -ffp-contract=off and correctly rounded FP32
// division and square root, so each `a * b + c` below rounds twice, exactly like the CPU oracle.
// Operation order follows the reference kernels (file:line next to each helper): glm's dot is
// (x*x + y*y) + z*z, vec*scalar rounds per component, integer powers are left-to-right products.
#pragma once

#include <hip/hip_runtime.h>

#include "pbf_types.h"

namespace akua {

struct f3 {
    float x, y, z;
};

__device__ __forceinline__ f3 make3(float4 a) { return {a.x, a.y, a.z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ f3 operator/(f3 a, float s) { return {a.x / s, a.y / s, a.z / s}; }

// glm::dot for vec3 (glm/detail/func_geometric.inl:48-54)
__device__ __forceinline__ float dot3(f3 a, f3 b) {
    float tx = a.x * b.x, ty = a.y * b.y, tz = a.z * b.z;
    return (tx + ty) + tz;
}
__device__ __forceinline__ float length3(f3 a) { return sqrtf(dot3(a, a)); }

// MathUtilsCUDA::cross (MathUtilsCUDA.h:12-18)
__device__ __forceinline__ f3 cross3(f3 a, f3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// device_poly6 (SmoothingKernelsCUDA.h:16-21): cp * (h^2 - r^2)^3, 0 beyond h.
__device__ __forceinline__ float poly6(float d2, const SphParams& P) {
    if (d2 > P.h2) return 0.0f;
    float t = P.h2 - d2;
    return P.cp * ((t * t) * t);
}

// ---- correctly rounded division and square root, written out ------------------------------
// The gfx950 sequence for a correctly rounded a / b is
//   den = div_scale(b); num = div_scale(a); r = rcp(den); r = fma(fma(-den, r, 1), r, r);
//   q = num * r; t = fma(-den, q, num); q = fma(t, r, q); t = fma(-den, q, num);
//   q = div_fmas(t, r, q); q = div_fixup(q, b, a).
// For a positive divisor and a numerator of magnitude in [2^-40, 2^40] neither div_scale scales
// (exponents far from the limits, difference below 96) nor div_fixup changes anything, and
// div_fmas is a plain fma.  Two facts shorten the rest:
//  - the refined reciprocal r = fma(fma(-b, rcp(b), 1), rcp(b), rcp(b)) is RN(1/b), the correctly
//    rounded reciprocal, for every significand of b (checked exhaustively on the device; the
//    exponent only scales rcp's result in this range), and it is shared by every numerator over
//    one divisor;
//  - with y = RN(1/b), q = RN(a y) and the exact remainder t = a - b q (one fma), RN(q + t y) is
//    RN(a / b) (Markstein's theorem on the final correction of a division), so one correction
//    step instead of two gives the same quotient.
// Outside that range the '/' operator is used.  akua_selftest_arith checks the reciprocal and the
// quotient against '/' on the device.
struct Recip {
    float b, r;
};

__device__ __forceinline__ Recip recip(float b) {
    float r = __builtin_amdgcn_rcpf(b);
    const float e = fmaf(-b, r, 1.0f);
    r = fmaf(e, r, r);
    return {b, r};
}

// a / b by the shared reciprocal, valid (equal to '/') when in_div_range(a) and
// in_div_range(b).  The quotient takes a's sign bit: for b > 0 a nonzero quotient has it
// already, and a zero numerator gives a quotient of magnitude zero whose sign the fmas may
// lose (one bit insert instead of a compare and a select).
__device__ __forceinline__ float div_rn_unchecked(float a, const Recip& R) {
    float q = a * R.r;
    const float t = fmaf(-R.b, q, a);
    q = fmaf(t, R.r, q);
    return __uint_as_float((__float_as_uint(q) & 0x7FFFFFFFu) | (__float_as_uint(a) & 0x80000000u));
}

// Range tests on the bit patterns: |x| in [2^-40, 2^40] (0x2B800000 .. 0x53800000) or x == 0.
// For several numerators at once, (|bits| - 1) maps zero above every finite pattern, so one
// unsigned min and one max test them all.
constexpr uint32_t kDivLo = 0x2B800000u, kDivHi = 0x53800000u;

__device__ __forceinline__ uint32_t mag_bits(float x) { return __float_as_uint(x) & 0x7FFFFFFFu; }

// 2 (|bits| - 1) mod 2^32, one shift-and-add: the sign bit shifts out, and zero maps to
// 0xFFFFFFFE, above every finite pattern.  So low2(x) >= kDivLo2 exactly when |x| >= 2^-40 or
// x == 0, the lower half of in_div_range.
constexpr uint32_t kDivLo2 = 2u * kDivLo - 2u;
__device__ __forceinline__ uint32_t low2(float x) { return (__float_as_uint(x) << 1) - 2u; }

__device__ __forceinline__ bool in_div_range(float x) {
    const uint32_t m = mag_bits(x);
    return m - 1u >= kDivLo - 1u && m <= kDivHi;
}

// b > 0 and |b| in [2^-40, 2^40]
__device__ __forceinline__ bool divisor_ok(float b) {
    const uint32_t u = __float_as_uint(b);
    return u >= kDivLo && u <= kDivHi;
}

__device__ __forceinline__ float div_rn(float a, const Recip& R) {
    float q = div_rn_unchecked(a, R);
    if (!(in_div_range(a) && divisor_ok(R.b))) q = a / R.b;
    return q;
}

// (x, y, z) / b with one range check for the four operands.
__device__ __forceinline__ f3 div3_rn(f3 v, float b) {
    const Recip R = recip(b);
    f3 q{div_rn_unchecked(v.x, R), div_rn_unchecked(v.y, R), div_rn_unchecked(v.z, R)};
    const uint32_t mx = mag_bits(v.x), my = mag_bits(v.y), mz = mag_bits(v.z);
    const uint32_t lo = min(min(mx - 1u, my - 1u), mz - 1u);
    const uint32_t hi = max(max(mx, my), mz);
    const bool ok = divisor_ok(b) && lo >= kDivLo - 1u && hi <= kDivHi;
    if (!ok) q = {v.x / b, v.y / b, v.z / b};
    return q;
}

// Correctly rounded sqrt for x >= 2^-96 (no scaling needed there): the 1-ulp hardware root,
// corrected by the residuals of its two neighbours, as the compiler's own lowering does.  Below
// 2^-96 it returns a value below 2^-47 (not necessarily correctly rounded): callers use it only
// where every such value leads to the same branch.
__device__ __forceinline__ float sqrt_rn_unscaled(float x) {
    float s = __builtin_amdgcn_sqrtf(x);
    const float sm = __uint_as_float(__float_as_uint(s) - 1u);
    const float sp = __uint_as_float(__float_as_uint(s) + 1u);
    const float em = fmaf(-sm, s, x);
    const float ep = fmaf(-sp, s, x);
    s = (em <= 0.0f) ? sm : s;
    s = (ep > 0.0f) ? sp : s;
    return s;
}

// device_gradient_spiky (SmoothingKernelsCUDA.h:23-28): cs * (h - |r|)^2 * r / |r|.  |r| and
// the three quotients are correctly rounded (the reference's length and '/'): a squared length
// below 2^-96 gives |r| < 1e-5, the zero branch, whatever its last bits.
// grad_spiky_nonzero: the same gradient into g, or false (g untouched) where it is zero, for
// callers whose sums a zero gradient leaves unchanged.
__device__ __forceinline__ bool grad_spiky_nonzero(f3 r, const SphParams& P, f3& g) {
    const float d2 = dot3(r, r);
    const float rm = sqrt_rn_unscaled(d2);
    if (rm > P.h || rm < 1e-5f) return false;
    float t = P.h - rm;
    float s = P.cs * (t * t);
    g = div3_rn(s * r, rm);
    return true;
}

__device__ __forceinline__ f3 grad_spiky(f3 r, const SphParams& P) {
    f3 g{0.0f, 0.0f, 0.0f};
    grad_spiky_nonzero(r, P, g);
    return g;
}

// ---- the sweeps with bounded quotients (SphParams::fast) ------------------------------------------
// |r| lies in [1e-5, h] and |cs| h^3 bounds the numerators, both inside the exact-division range, so
// of the range tests only the numerators' lower bound is left; and |r| and 1 / |r| come from one
// hardware reciprocal root instead of a root, a reciprocal and their corrections (10 instead of 18
// issue slots, a transcendental taking four):
//   y = rsq(x); s0 = x y; s = fma(fma(-s0, s0, x), y / 2, s0) is RN(sqrt x) for every x, and
//   i = fma(fma(-s, y, 1), y, y) is RN(1 / s) for every x but those whose root has a significand of
//   all ones (there 1 / s lies just above the middle of two floats, and fma(-s, y, 1) is exactly 2^-24).
// Both were checked over all 2^24 significands and exponent parities on the device (the exponent
// only scales rsq here), and akua_selftest_arith checks them again.
struct RootRecip {
    float s, i;
    bool inexact;  // i may not be the correctly rounded reciprocal
};

__device__ __forceinline__ RootRecip root_recip(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float s0 = x * y;
    const float d = fmaf(-s0, s0, x);
    const float s = fmaf(d, 0.5f * y, s0);
    const float e = fmaf(-s, y, 1.0f);
    return {s, fmaf(e, y, y), e == 0x1p-24f};
}

// a / b from b's correctly rounded reciprocal where both lie in the exact-division range.  A zero
// numerator gives a zero whose sign may differ: the sweeps only add terms to sums that start at
// +0 and therefore are never -0, to which a zero of either sign is the same.
__device__ __forceinline__ float div_by(float a, float b, float recip) {
    const float q = a * recip;
    return fmaf(fmaf(-b, q, a), recip, q);
}

// poly6 for squared lengths of any size, infinite and NaN included (cp is finite here, so cp * 0 is 0).
__device__ __forceinline__ float poly6_bounded(float d2, const SphParams& P) {
    const float t = __builtin_elementwise_maximum(P.h2 - d2, 0.0f);
    return P.cp * ((t * t) * t);
}

// The gradient's quotients before their numerators' lower bound is looked at.
struct GradTerm {
    f3 n, g;      // numerators, quotients
    float rm;     // |r|
    float low;    // the smallest numerator's magnitude
    bool inexact;
};

// False where the gradient is zero (d2 = |r|^2, NaN counting as inside, as the rounded length does).
__device__ __forceinline__ bool grad_term(f3 r, float d2, const SphParams& P, GradTerm& G) {
    if (d2 > P.d2Far || d2 < P.d2Near) return false;
    const RootRecip R = root_recip(d2);
    const float t = P.h - R.s;
    G.n = (P.cs * (t * t)) * r;
    G.g = {div_by(G.n.x, R.s, R.i), div_by(G.n.y, R.s, R.i), div_by(G.n.z, R.s, R.i)};
    G.rm = R.s;
    G.low = fminf(fminf(fabsf(G.n.x), fabsf(G.n.y)), fabsf(G.n.z));
    G.inexact = R.inexact;
    return true;
}

constexpr float kDivLowest = 0x1p-40f;

// The quotients by '/' where the short form does not hold: a numerator below 2^-40 that is not zero,
// or the reciprocal's exception.  Called where G.low < kDivLowest or G.inexact (also with a zero
// numerator, whose quotient stands).
__device__ __forceinline__ void grad_by_division(GradTerm& G) {
    const uint32_t lo = min(min(low2(G.n.x), low2(G.n.y)), low2(G.n.z));
    if (G.inexact || lo < kDivLo2) G.g = G.n / G.rm;
}

// The gradient into g, or false where it is zero.
__device__ __forceinline__ bool grad_bounded(f3 r, float d2, const SphParams& P, f3& g) {
    GradTerm G;
    if (!grad_term(r, d2, P, G)) return false;
    if (__builtin_expect(G.low < kDivLowest || G.inexact, 0)) grad_by_division(G);
    g = G.g;
    return true;
}

// The kernels' forms by kFast: bounded quotients or the general ones.
template <bool kFast>
__device__ __forceinline__ float poly6_of(float d2, const SphParams& P) {
    return kFast ? poly6_bounded(d2, P) : poly6(d2, P);
}
template <bool kFast>
__device__ __forceinline__ bool grad_of(f3 r, float d2, const SphParams& P, f3& g) {
    return kFast ? grad_bounded(r, d2, P, g) : grad_spiky_nonzero(r, P, g);
}
template <bool kFast>
__device__ __forceinline__ f3 grad_or_zero(f3 r, float d2, const SphParams& P) {
    f3 g{0.0f, 0.0f, 0.0f};
    grad_of<kFast>(r, d2, P, g);
    return g;
}

// The artificial pressure's quotient w / wdq of the bounded sweeps (w is +0 or positive), before and
// after its numerator's lower bound is looked at.
__device__ __forceinline__ float corr_by_division(float w, float q, const Recip& R) {
    return low2(w) < kDivLo2 ? w / R.b : q;
}

// powf(x, n) of the artificial pressure (ConstraintSolverCUDA.cu:124): an integer n is the n-fold
// left-to-right product; any other n calls powf.
__device__ __forceinline__ float corr_pow(float x, const SphParams& P) {
    int k = P.corrNInt;
    if (k == 4) return ((x * x) * x) * x;  // the usual exponent, without the loop
    if (k < 0) return powf(x, P.corrN);
    if (k == 0) return 1.0f;
    float r = x;
    for (int i = 1; i < k; ++i) r = r * x;
    return r;
}

// float -> int with NaN -> 0 and saturation, spelled out so the result never depends on what
// the compiler assumes about an out-of-range conversion.
__device__ __forceinline__ int to_int_sat(float x) {
    if (!(x == x)) return 0;
    if (x >= 2147483648.0f) return 2147483647;
    if (x < -2147483648.0f) return (int)0x80000000u;
    return (int)x;
}

// device_discretize_position (NeighbourSearchCUDA.cu:15-21)
__device__ __forceinline__ void discretize(f3 p, float cs, int& cx, int& cy, int& cz) {
    cx = to_int_sat(floorf(p.x / cs));
    cy = to_int_sat(floorf(p.y / cs));
    cz = to_int_sat(floorf(p.z / cs));
}

// device_get_hash (NeighbourSearchCUDA.cu:23-27), with the int multiply's wrap done in uint32
// and the modulo by the scene's table size done by multiply-high (exact for every input).
__device__ __forceinline__ uint32_t cell_hash(int cx, int cy, int cz, const SceneDev& sc) {
    uint32_t a = (uint32_t)cx * 73856093u;
    uint32_t b = (uint32_t)cy * 19349663u;
    uint32_t c = (uint32_t)cz * 83492791u;
    return fast_mod(a ^ b ^ c, sc.tableSize, sc.modMagic, sc.modShift);
}

// Key of a cell of the non-parity search over h / 2 cells: the low 10 bits of each coordinate,
// packed (never kEmptyKey).  Cells less than 1024 apart along every axis get distinct keys, so no
// two cells of one 5x5x5 stencil share a bucket.
__device__ __forceinline__ uint32_t cell_key_fine(int cx, int cy, int cz) {
    return (((uint32_t)cx & 1023u) << 20) | (((uint32_t)cy & 1023u) << 10) | ((uint32_t)cz & 1023u);
}

// kernel_predict_position (IntegrationCUDA.cu:27-36): v* = v + g dt; x* = x + v* dt.
__device__ __forceinline__ f3 predict_x(f3 x, f3 v, const StepParams& S) {
    f3 g{S.g[0], S.g[1], S.g[2]};
    f3 vs = v + g * S.dt;
    return x + vs * S.dt;
}

// First slot of a hash in the scene's open-addressing cell table.
__device__ __forceinline__ uint32_t table_slot(uint32_t hash, uint32_t log2cap) {
    return (hash * 2654435761u) >> (32u - log2cap);
}

}  // namespace akua
