// The scalar functions of the elementwise operators, one definition for every kernel that applies them:
// the operators one by one (k_elem.hip) and a run of them in one pass (k_chain.hip) store the same bits.
#pragma once
#include <hip/hip_runtime.h>

#include "gorgonia_hip.h"

namespace {

template <class T> struct VecOf;
template <> struct VecOf<float> { typedef float type __attribute__((ext_vector_type(4))); static constexpr int N = 4; };
template <> struct VecOf<double> { typedef double type __attribute__((ext_vector_type(2))); static constexpr int N = 2; };

// ---- scalar functions ------------------------------------------------------

template <int FN, class T>
__device__ __forceinline__ T bin_apply(T a, T b) {
  if constexpr (FN == GH_ADD) return a + b;
  else if constexpr (FN == GH_SUB) return a - b;
  else if constexpr (FN == GH_MUL) return a * b;
  else if constexpr (FN == GH_DIV) return a / b;
  else if constexpr (FN == GH_POW) return (T)pow((double)a, (double)b);
  else if constexpr (FN == GH_LT) return a < b ? (T)1 : (T)0;
  else if constexpr (FN == GH_LTE) return a <= b ? (T)1 : (T)0;
  else if constexpr (FN == GH_GT) return a > b ? (T)1 : (T)0;
  else if constexpr (FN == GH_GTE) return a >= b ? (T)1 : (T)0;
  else if constexpr (FN == GH_EQ) return a == b ? (T)1 : (T)0;
  else if constexpr (FN == GH_MOD) return (T)fmod((double)a, (double)b);   // exact in either width
  else return a != b ? (T)1 : (T)0;
}

// exp in float64 for results that are rounded to float32 afterwards.
// Range reduction x = n ln2 + r with |r| <= ln2/2: n comes from the
// "add 1.5*2^52" trick (the integer sits in the low mantissa bits, so no
// round/convert instructions), exp(r) - 1 from a degree-10 Taylor polynomial
// (relative error below 2^-41, far under half a float32 ulp), and the scaling
// by 2^n is an integer add on the exponent field.  Valid for |x| <= 700;
// callers clamp.  Explicit fma() so the -ffp-contract=off build still gets
// fused steps here.  Conversion, reciprocal and ldexp instructions run at a
// quarter of the FMA rate on this hardware, which is why they are avoided:
// sigmoid/tanh/exp stay memory-bound.
struct ExpParts { double q; int n; };  // exp(x) = (1 + q) * 2^n

// A float64 constant pinned in a scalar register pair.  As a plain literal each
// Horner step costs an extra 64-bit vector move (the compiler materialises the
// coefficient into the accumulator of v_fmac_f64); from a scalar register the
// step is a single v_fma_f64.  The empty asm only hides the value's origin.
__device__ __forceinline__ double sconst(double v) {
  asm("" : "+s"(v));
  return v;
}

__device__ __forceinline__ ExpParts exp_parts(double x) {
  const double kShift = sconst(6755399441055744.0);  // 1.5 * 2^52
  const double t = fma(x, sconst(1.4426950408889634), kShift);
  const double n = t - kShift;
  double r = fma(-n, sconst(0.6931471803691238), x);   // ln2 high part
  r = fma(-n, sconst(1.9082149292705877e-10), r);      // ln2 low part
  double p = sconst(2.7557319223985893e-07);           // 1/10!
  p = fma(p, r, sconst(2.7557319223985888e-06));       // 1/9!
  p = fma(p, r, sconst(2.4801587301587302e-05));       // 1/8!
  p = fma(p, r, sconst(1.9841269841269841e-04));       // 1/7!
  p = fma(p, r, sconst(1.3888888888888889e-03));       // 1/6!
  p = fma(p, r, sconst(8.3333333333333332e-03));       // 1/5!
  p = fma(p, r, sconst(4.1666666666666664e-02));       // 1/4!
  p = fma(p, r, sconst(1.6666666666666666e-01));       // 1/3!
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  ExpParts e;
  e.q = p * r;
  e.n = (int)(unsigned)__double_as_longlong(t);    // low 32 bits of t hold n
  return e;
}

__device__ __forceinline__ double scale_pow2(double v, int n) {  // v * 2^n, result normal
  return __longlong_as_double(__double_as_longlong(v) + ((long long)n << 52));
}

__device__ __forceinline__ double exp_f64_fast(double x) {
  const ExpParts e = exp_parts(x);
  return scale_pow2(1.0 + e.q, e.n);
}

// 1/s in float64 to ~2^-50: hardware reciprocal estimate plus one Newton step.
__device__ __forceinline__ double rcp_f64_fast(double s) {
  const double r = __builtin_amdgcn_rcp(s);
  return fma(fma(-s, r, 1.0), r, r);
}

// exp(x) for a float32 argument, rounded once from float64.
__device__ __forceinline__ float exp_f32_via_f64(float x) {
  double xd = (double)x;
  xd = xd < -110.0 ? -110.0 : xd;  // beyond the clamps the rounded result is 0 / +inf
  xd = xd > 90.0 ? 90.0 : xd;      // (NaN fails both compares and propagates)
  return (float)exp_f64_fast(xd);
}

// tanh in float64 from one exp, branch free: with a = 2|x|,
// tanh|x| = (e^a - 1)/(e^a + 1) = em1/(em1 + 2).  For n == 0 the polynomial
// yields e^a - 1 directly (no cancellation near zero); otherwise e^a >= sqrt(2)
// and the subtraction is harmless.  Error stays far below half a float32 ulp.
__device__ __forceinline__ double tanh_f64_for_f32(double x) {
  double a = 2.0 * fabs(x);
  a = a > 44.0 ? 44.0 : a;  // tanh rounds to 1 long before; NaN propagates
  const ExpParts e = exp_parts(a);
  const double em1 = e.n == 0 ? e.q : scale_pow2(1.0 + e.q, e.n) - 1.0;
  const double r = em1 * rcp_f64_fast(em1 + 2.0);
  return copysign(r, x);
}

// ---- float32 sigmoid / tanh without float64 ---------------------------------------
// The float64 forms above are within half an ulp but cost two quarter-rate
// conversions, a float64 reciprocal and ~20 half-rate FMAs per element, which
// makes a streaming kernel ALU-bound on this part.  These stay in float32, take
// about twenty instructions each and stay within 2 ulp of the correctly rounded
// result over every float32 input (measured exhaustively; the dense sweep in the
// GPU tests repeats it against the CPU oracle): sigmoid at most 2, tanh at most 1.
// With fewer instructions the kernels stay memory-bound at the clocks a device
// holds after minutes of load as well.
//
// exp(t) = 2^n * (1 + q): n = round(t / ln2) through the 1.5*2^23 shift (the
// integer also sits in the low mantissa bits of `shifted`), Cody-Waite reduction
// with a short-mantissa ln2 high part so that n*ln2_hi is exact, and
// exp(r) - 1 = r + r^2 P(r) with a degree-4 minimax P on |r| <= ln2/2 (relative
// error of exp below 2^-28).
struct ExpF { float q; int shbits; };

constexpr unsigned kShiftBits = 0x4B400000u;   // bits of 1.5 * 2^23

__device__ __forceinline__ ExpF expf_parts(float t) {
  const float kShift = 12582912.0f;  // 1.5 * 2^23
  const float shifted = __builtin_fmaf(t, 1.44269504088896341f, kShift);
  const float nf = shifted - kShift;
  float r = __builtin_fmaf(-nf, 0.693145751953125f, t);
  r = __builtin_fmaf(-nf, 1.428606765330187e-06f, r);
  float p = 0.0013813756f;
  p = __builtin_fmaf(p, r, 0.008369124f);
  p = __builtin_fmaf(p, r, 0.041668426f);
  p = __builtin_fmaf(p, r, 0.16666517f);
  p = __builtin_fmaf(p, r, 0.49999994f);
  ExpF e;
  e.q = __builtin_fmaf(r * r, p, r);
  e.shbits = __float_as_int(shifted);
  return e;
}

// 2^(n + bias) as a float from the shifted sum's bits: one shift-and-add.
template <int BIAS>
__device__ __forceinline__ float pow2_of(int shbits) {
  return __int_as_float((shbits << 23) + (int)(((unsigned)(127 + BIAS) << 23) - (kShiftBits << 23)));
}

// sigmoid with the reference's cut-offs (math_nooptim.go:36-44).  With E = exp(|x|) =
// 2^n (1 + q), r = 1 / (1 + E) is sigmoid(-|x|) and 1 - r is sigmoid(|x|).  The sum
// 1 + E is formed scaled by 2^-64, as (2^(n-64) q + 2^-64) + 2^(n-64): two roundings
// of at most 0.9 ulp together for every n (adding the 1 to 2^n first would lose it
// from n = 24 on), and the scaling keeps the hardware reciprocal's result normal
// where r itself is subnormal (x below -87.3); the final multiply-add by 2^-64
// rounds once.  Beyond the cut-offs r is replaced by 0, which gives exactly 0 and 1.
// NaN fails the compare and propagates through r.
__device__ __forceinline__ float sigmoid_f32_fast(float x) {
  const float a = fabsf(x);
  const ExpF p = expf_parts(a);
  const float s = pow2_of<-64>(p.shbits);
  const float c = 5.421010862427522e-20f;                       // 2^-64
  const float d = __builtin_fmaf(s, p.q, c) + s;
  float rc = __builtin_amdgcn_rcpf(d);                          // 2^64 / (1 + E), within an ulp
  const float cs = copysignf(c, x);
  const float lim = __builtin_fmaf(cs, -36.5f * 18446744073709551616.0f, 51.5f);   // 15 right of zero, 88 left
  const float base = __builtin_fmaf(cs, 0.5f * 18446744073709551616.0f, 0.5f);     // 1 right of zero, 0 left
  rc = a > lim ? 0.0f : rc;
  return __builtin_fmaf(-cs, rc, base);
}

// tanh: below 0.55 an odd polynomial x + x^3 R(x^2) (R fitted on [0, 0.56^2],
// approximation error 0.07 ulp); above it 1 - 2/(e^(2|x|) + 1), where the result
// is at least 0.5 and the quotient's error (the sum's single rounding and the
// hardware reciprocal's ulp) shrinks by the factor 2/(e^(2|x|) + 1) <= 1/2.
// The exponential's argument is clamped (tanh(22) rounds to 1); the clamp drops a
// NaN, so the choice between the two forms is written to fall to the polynomial,
// which keeps it, when the compare fails.
__device__ __forceinline__ float tanh_f32_fast(float x) {
  const float ax = fabsf(x);
  const float s2 = ax * ax;
  float R = 0.0024976127315312624f;
  R = __builtin_fmaf(R, s2, -0.008506525307893753f);
  R = __builtin_fmaf(R, s2, 0.02181374467909336f);
  R = __builtin_fmaf(R, s2, -0.05396425351500511f);
  R = __builtin_fmaf(R, s2, 0.133333221077919f);
  R = __builtin_fmaf(R, s2, -0.3333333432674408f);
  const float small = __builtin_fmaf(ax * s2, R, ax);
  const float ac = fminf(ax, 22.0f);
  const ExpF p = expf_parts(ac + ac);
  const float s = pow2_of<0>(p.shbits);
  const float d = __builtin_fmaf(s, p.q, s + 1.0f);             // e^(2|x|) + 1 in one rounding (n <= 64 / ln2)
  const float rc = __builtin_amdgcn_rcpf(d);
  const float large = __builtin_fmaf(-2.0f, rc, 1.0f);
  return copysignf(ax >= 0.55f ? large : small, x);
}

template <int FN>
__device__ __forceinline__ float unary_apply(float x) {
  if constexpr (FN == GH_ABS) return fabsf(x);
  else if constexpr (FN == GH_SIGN) return (float)((x > 0.0f) - (x < 0.0f));
  else if constexpr (FN == GH_CEIL) return ceilf(x);
  else if constexpr (FN == GH_FLOOR) return floorf(x);
  else if constexpr (FN == GH_SIN) return (float)sin((double)x);
  else if constexpr (FN == GH_COS) return (float)cos((double)x);
  else if constexpr (FN == GH_EXP) return exp_f32_via_f64(x);
  else if constexpr (FN == GH_LN) return (float)log((double)x);
  else if constexpr (FN == GH_LOG2) return (float)log2((double)x);
  else if constexpr (FN == GH_NEG) return -x;
  else if constexpr (FN == GH_SQUARE) return x * x;
  else if constexpr (FN == GH_SQRT) return sqrtf(x);
  else if constexpr (FN == GH_INVERSE) return 1.0f / x;
  else if constexpr (FN == GH_INVSQRT) return 1.0f / sqrtf(x);
  else if constexpr (FN == GH_CUBE) return x * x * x;
  else if constexpr (FN == GH_TANH) return tanh_f32_fast(x);
  else if constexpr (FN == GH_SIGMOID) return sigmoid_f32_fast(x);
  else if constexpr (FN == GH_LOG1P) return (float)log1p((double)x);
  else if constexpr (FN == GH_EXPM1) return (float)expm1((double)x);
  else {  // softplus
    if (x < -103.0f) return 0.0f;
    if (x > 14.0f) return x;
    return (float)log1p(exp((double)x));
  }
}

template <int FN>
__device__ __forceinline__ double unary_apply(double x) {
  if constexpr (FN == GH_ABS) return fabs(x);
  else if constexpr (FN == GH_SIGN) return (double)((x > 0.0) - (x < 0.0));
  else if constexpr (FN == GH_CEIL) return ceil(x);
  else if constexpr (FN == GH_FLOOR) return floor(x);
  else if constexpr (FN == GH_SIN) return sin(x);
  else if constexpr (FN == GH_COS) return cos(x);
  else if constexpr (FN == GH_EXP) return exp(x);
  else if constexpr (FN == GH_LN) return log(x);
  else if constexpr (FN == GH_LOG2) return log2(x);
  else if constexpr (FN == GH_NEG) return -x;
  else if constexpr (FN == GH_SQUARE) return x * x;
  else if constexpr (FN == GH_SQRT) return sqrt(x);
  else if constexpr (FN == GH_INVERSE) return 1.0 / x;
  else if constexpr (FN == GH_INVSQRT) return 1.0 / sqrt(x);
  else if constexpr (FN == GH_CUBE) return x * x * x;
  else if constexpr (FN == GH_TANH) return tanh(x);
  else if constexpr (FN == GH_SIGMOID) {
    if (x < -709.0) return 0.0;
    if (x > 19.0) return 1.0;
    return 1.0 / (1.0 + exp(-x));
  } else if constexpr (FN == GH_LOG1P) return log1p(x);
  else if constexpr (FN == GH_EXPM1) return expm1(x);
  else {
    if (x < -708.0) return 0.0;
    if (x > 16.0) return x;
    return log1p(exp(x));
  }
}

// ---- ReLU / LeakyReLU in the reference's arithmetic form --------------------
// Rectify: x * float(x >= 0) (nn.go:136-163) - negative inputs give -0.0.
// LeakyRelu: x*(x>=0) + (x*(x<0))*alpha (nn.go:83-131).
__device__ __forceinline__ float relu_ref(float x) { return x * (x >= 0.0f ? 1.0f : 0.0f); }
__device__ __forceinline__ float leaky_ref(float x, float alpha) {
  const float pos = x * (x >= 0.0f ? 1.0f : 0.0f);
  const float neg = x * (x < 0.0f ? 1.0f : 0.0f);
  const float na = neg * alpha;
  return pos + na;
}

// STREAM: non-temporal, for operands the last-level cache cannot hold or has lost.
template <class V, bool STREAM>
__device__ __forceinline__ V ld_vec(const V* p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(p);
  else return *p;
}
template <class V, bool STREAM>
__device__ __forceinline__ void st_vec(V* p, V v) {
  if constexpr (STREAM) __builtin_nontemporal_store(v, p);
  else *p = v;
}

}  // namespace
