// Host check of the kernels' sine, cosine, arctangent and quotient (trig_dev.h)
// against the double and long double functions: the largest error in units in the
// last place of the result over the ranges that they are used in, against the bounds
// that the header states.  (The reciprocal in the quotients is the host's; the
// device's is within an ulp, which the correction step removes.)  Exit status 0 when
// all hold.
#include "../mesh_amd/csrc/trig_dev.h"
#include <cstdio>
#include <cstdlib>

using namespace mesh_dev;

namespace {

double ulp(double v)
{
	const float a = std::fabs((float)v);
	return (double)std::nextafter(a, INFINITY) - a;
}

int bad = 0;
void check(const char *what, double worst, double bound)
{
	std::printf("%s %.3f ulp (bound %.2f)\n", what, worst, bound);
	bad += !(worst <= bound);
}

} // namespace

int main()
{
	const long N = 4000000;
	// angles of the first octant, where the polynomials are, and of two turns either way; away
	// from a function's zeros, where the reduction's last bits (3e-15) stand out
	double s8 = 0, c8 = 0, s = 0, c = 0, abs0 = 0, lean = 0;
	for (long i = 0; i <= N; ++i)
	{
		const float x = (float)(0.78539816339744830962 * i / N), y = (float)(12.566370614359172954 * (2.0 * i / N - 1));
		float sn, cs;
		sincos1(x, sn, cs);
		if (x > 0)
			s8 = fmax(s8, std::fabs(sn - std::sin((double)x)) / ulp(std::sin((double)x)));
		c8 = fmax(c8, std::fabs(cs - std::cos((double)x)) / ulp(std::cos((double)x)));
		if (x < 0.1f)
			lean += (cs - std::cos((double)x)) / (N * 0.1 / 0.78539816339744830962);
		sincos1(y, sn, cs);
		const double S = std::sin((double)y), C = std::cos((double)y);
		s = fmax(s, std::fabs(sn - S) / fmax(ulp(S), 1e-12));
		c = fmax(c, std::fabs(cs - C) / fmax(ulp(C), 1e-12));
		abs0 = fmax(abs0, fmax(std::fabs(sn - S), std::fabs(cs - C)));
	}
	check("sine, an eighth of a turn", s8, 0.70);
	check("cosine, an eighth of a turn", c8, 0.90);
	check("sine, two turns", s, 1.50);
	check("cosine, two turns", c, 1.50);
	check("absolute, in 2^-24", abs0 * 16777216.0, 1.20);
	check("mean error of small angles' cosine, in 1e-10", std::fabs(lean) * 1e10, 1.0);
	// arctangents all round, quotients from e^-16 to e^16
	double a = 0, q = 0;
	srand(1);
	auto uniform = [] { return (rand() + 0.5) / ((double)RAND_MAX + 1.0); };
	for (long i = 0; i <= N; ++i)
	{
		const float y = (float)((uniform() * 2 - 1) * std::exp(16 * (uniform() - 0.5))),
		            x = (float)((uniform() * 2 - 1) * std::exp(16 * (uniform() - 0.5)));
		if (x == 0 || y == 0)
			continue;
		const double A = std::atan2((double)y, (double)x);
		a = fmax(a, std::fabs(atan2_1(y, x) - A) / ulp(A));
		const float n = (float)std::exp(32 * (uniform() - 0.5)), d = (float)std::exp(32 * (uniform() - 0.5));
		q = fmax(q, std::fabs(div1(n, d) - (double)n / d) / ulp((double)n / d));
	}
	check("arctangent", a, 1.55);
	check("quotient", q, 0.51);
	// double cosine: angles of a few turns and of a plaquette's sum of four
	double d1 = 0;
	for (long i = 0; i <= N; ++i)
	{
		const double x = 30.0 * (2.0 * i / N - 1);
		const long double C = std::cos((long double)x);
		d1 = fmax(d1, (double)std::fabs((long double)cos1(x) - C) * 9007199254740992.0);
	}
	check("double cosine, absolute, in 2^-53", d1, 1.60);
	std::printf("%d wrong\n", bad);
	return bad != 0;
}
