// Sine, cosine, arctangent and quotient for the ranges that the U(1) kernels
// meet: angles of a few turns at most and finite, non-zero quotients (the functions
// named any: those of a caller's links, which need not be wrapped).
//
// These kernels are held by vector instructions, and the library's functions
// carry the reduction of huge arguments, infinities and zeros: sincosf and
// atan2f are about 90 and 60 instructions a call against 24 and 27 here, the
// double cosine about 100 against 35.  Coefficients: minimax fits (reweighted
// least squares) of (sin r - r) / r^3 and (cos r - 1 + r^2 / 2) / r^4 over
// |r| <= pi / 4 and of (atan q - q) / q^3 over [0, 1].  Largest errors (checked on
// the host): in the first eighth of a turn 0.69 ulp (sin) and 0.88 ulp (cos), in two
// turns either way 1.5 ulp of both; arctangent 1.5 ulp; quotient half an ulp; double
// cosine (Taylor series) 1.6 2^-53.
#pragma once
#include <cmath>
#include <hip/hip_runtime.h>

namespace mesh_dev {

// (the host side serves the check of these bounds)
#define TD __host__ __device__ __forceinline__

// n / d to within an ulp, for d and 1 / d in the normal range
TD float div1(float n, float d)
{
#ifdef __HIP_DEVICE_COMPILE__
	const float r = __builtin_amdgcn_rcpf(d);
#else
	const float r = 1.f / d;
#endif
	const float q = n * r;
	return fmaf(fmaf(-q, d, n), r, q);
}

constexpr float HALF_PI_HI = 1.57079637050628662109f, HALF_PI_LO = -4.37113900018624283e-8f;

TD float sin_quarter(float r, float r2)
{
	return fmaf(r * r2,
	            fmaf(fmaf(-0.00019516977772582322f, r2, 0.008332176133990288f), r2, -0.16666655242443085f), r);
}
// (one rounding at the magnitude of 1: with 1 - r2 / 2 rounded before the rest was
// added the largest error was 1.24 ulp and cosines below 0.1 were 1e-9 low on average)
TD float cos_quarter(float r2)
{
	return fmaf(fmaf(fmaf(fmaf(2.443809171381872e-05f, r2, -0.0013887364184483886f), r2, 0.04166664555668831f), r2, -0.5f),
	            r2, 1.f);
}
// r = x - i pi / 2, |r| <= pi / 4 (the first step is exact for a few turns)
TD float quarter(float x, int &i)
{
	const float q = rintf(x * 0.63661977236758134f);
	i = (int)q;
	return fmaf(-q, HALF_PI_LO, fmaf(-q, HALF_PI_HI, x));
}

// sin and cos for |x| up to a few turns (NaN gives NaN)
TD void sincos1(float x, float &sn, float &cs)
{
	int i;
	const float r = quarter(x, i), r2 = r * r, s = sin_quarter(r, r2), c = cos_quarter(r2);
	const bool odd = i & 1;
	const auto flip = [](float v, unsigned sign) {
		return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ sign << 31);
	};
	sn = flip(odd ? c : s, (unsigned)i >> 1 & 1);
	cs = flip(odd ? s : c, (unsigned)(i + 1) >> 1 & 1);
}
// sin and cos of any x: a caller's angle may be anything, and beyond some 10^7 the
// reduction above leaves no angle at all
TD void sincos_any(float x, float &sn, float &cs)
{
	if (fabsf(x) < 32768.f)
		sincos1(x, sn, cs);
	else
		sn = sinf(x), cs = cosf(x);
}
// atan2(y, x) for finite arguments, the larger of them a normal number whose
// reciprocal is one too
TD float atan2_1(float y, float x)
{
	const float ax = fabsf(x), ay = fabsf(y);
	const float q = div1(fminf(ax, ay), fmaxf(ax, ay)), q2 = q * q;
	float p = fmaf(-0.0018272141460329294f, q2, 0.011064446531236172f);
	p = fmaf(p, q2, -0.031455714255571365f);
	p = fmaf(p, q2, 0.0582345649600029f);
	p = fmaf(p, q2, -0.0841946005821228f);
	p = fmaf(p, q2, 0.10957576334476471f);
	p = fmaf(p, q2, -0.1426524519920349f);
	p = fmaf(p, q2, 0.19998638331890106f);
	p = fmaf(p, q2, -0.33333301544189453f);
	const float a = fmaf(q * q2, p, q);
	// pi/2 -+ a where |y| > |x|, pi - a for x < 0 below that
	const bool steep = ay > ax, neg = x < 0.f;
	const float k = steep ? HALF_PI_HI : (neg ? 2.f * HALF_PI_HI : 0.f);
	const float t = fmaf(k, HALF_PI_LO / HALF_PI_HI, steep != neg ? -a : a);
	return copysignf(k + t, y);
}

// cos for |x| < 10^9, FP64
TD double cos1(double x)
{
	const double q = rint(x * 0.63661977236758134308);
	const double r = fma(-q, 6.123233995736766036e-17, fma(-q, 1.57079632679489655800, x)), r2 = r * r;
	double ps = -1.0 / 1307674368000.0;
	ps = fma(ps, r2, 1.0 / 6227020800.0);
	ps = fma(ps, r2, -1.0 / 39916800.0);
	ps = fma(ps, r2, 1.0 / 362880.0);
	ps = fma(ps, r2, -1.0 / 5040.0);
	ps = fma(ps, r2, 1.0 / 120.0);
	ps = fma(ps, r2, -1.0 / 6.0);
	const double s = fma(r * r2, ps, r);
	double pc = 1.0 / 20922789888000.0;
	pc = fma(pc, r2, -1.0 / 87178291200.0);
	pc = fma(pc, r2, 1.0 / 479001600.0);
	pc = fma(pc, r2, -1.0 / 3628800.0);
	pc = fma(pc, r2, 1.0 / 40320.0);
	pc = fma(pc, r2, -1.0 / 720.0);
	pc = fma(pc, r2, 1.0 / 24.0);
	const double c = fma(r2 * r2, pc, fma(-0.5, r2, 1.0));
	const int i = (int)q;
	const double v = i & 1 ? s : c;
	return (i + 1) & 2 ? -v : v;
}
// cos of any x, FP64
TD double cos_any(double x) { return fabs(x) < 1e9 ? cos1(x) : cos(x); }

#undef TD

} // namespace mesh_dev
