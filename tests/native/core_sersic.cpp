// The FP32 core-Sersic value, its plain form and its derivatives against FP64 on
// the CPU, over sharp and soft transitions (a from 0.3 to 60) whose powers r^a,
// rb^a, re^a and (r/rb)^-a lie far beyond FP32's range, at radii from re / 1e5 to
// 30 re.  Prints "ok <points>".
#include <hip/hip_runtime.h>

#include <cstdio>
#include <random>

using std::max;
using std::min;

#include "profile_math.h"

using namespace profit_amd;

int main()
{
	std::mt19937_64 rng(99);
	auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
	auto logu = [&](double a, double b) { return std::exp(uni(std::log(a), std::log(b))); };
	const double e = 1.2e-7;  // 2^-23
	long points = 0, bad = 0;
	for (int k = 0; k < 2000; ++k) {
		Comp c{};
		ProfileParams p;
		default_params(CORESERSIC, &p);
		p.adjust = 0;
		double *s = p.shape;
		s[0] = logu(0.5, 100);
		s[1] = s[0] * logu(0.01, 2);
		s[2] = logu(0.5, 6);
		s[3] = logu(0.3, 60);
		s[4] = k % 10 ? uni(-1, 1.9) : 0.0;
		sf::QuadState qs;
		if (setup_component(p, 0, 1, 1, 1, 1, 0, 0, &qs, &c, false) != SE_OK) return 1;
		const double re = s[0], rb = s[1], n = s[2], a = s[3], b = std::fabs(s[4]), bn = c.bn;
		for (int m = 0; m < 50; ++m) {
			const float rf = (float)(re * logu(1e-5, 30));
			const double r = rf;
			// libprofit's value from logarithms: no power overflows in FP64
			const double lu = std::log(r / rb), x = std::exp(-a * std::fabs(lu)), lq = std::log1p(x), lM = std::log(std::fmax(r, rb));
			const double lQ = lq + (lu < 0 ? -a * lu : 0), lS = a * (lM - std::log(re)) + lq, W = std::exp(lS / (n * a)), E = bn * W;
			const double v = std::exp(s[4] / a * lQ - E);
			if (!(v > 1e-30 && v < 1e30)) continue;
			++points;
			const double L = std::fabs(std::log2(r)) + std::fabs(std::log2(rb)) + std::fabs(std::log2(re));
			// the sums of the operations' rounding errors, each times the exponents behind it
			const double tol = e * (20 + 2 * b + 3 * b / a + E * (11 + 3 / n + 3 / (n * a)) + 0.5 * b * std::fabs(lu) + E * std::fabs(std::log(W)));
			const double tolf = e * (8 + 2 * b * L + 4 * b / a + E * (2 * L / n + 3 * std::fabs(std::log(W)) + 6 + 3 / (n * a)));
			const double told = 8 * (tolf + e * (2 * a * L + 8));
			bool ok = std::fabs(eval_at<float, CORESERSIC>(c, rf, 0.f) - v) <= tol * v;
			ok &= std::fabs(eval_fast<CORESERSIC>(c, rf, 0.f) - v) <= tolf * v;
			float o[9];
			sample_grad<float, CORESERSIC>(c, rf, 0.f, o);
			const double gb = lu < 0 ? 1 / (1 + x) : x / (1 + x), gr = lu < 0 ? x / (1 + x) : 1 / (1 + x), dl = (gr * std::fabs(std::log(r)) + gb * std::fabs(std::log(rb)) + std::fabs(std::log(re)));
			const double aS = a * (std::fabs(lM) + std::fabs(std::log(re))) + lq;
			const double want[6] = {E / (n * re), s[4] * gb / rb - E * gb / (n * rb), -c.dbn * W + E * lS / (n * n * a),
			                        -s[4] / (a * a) * lQ - s[4] / a * gb * lu -
			                            E * ((gr * std::log(r) + gb * std::log(rb) - std::log(re)) / (n * a) - lS / (n * a * a)),
			                        lQ / a, -s[4] * gb / r - E * gr / (n * r)};
			const double size[6] = {E / (n * re), b * gb / rb + E * gb / (n * rb), std::fabs(c.dbn) * W + E * aS / (n * n * a),
			                        b / (a * a) * lQ + b / a * gb * std::fabs(lu) + E * (dl / (n * a) + aS / (n * a * a)), lQ / a,
			                        b * gb / r + E * gr / (n * r)};
			const float got[6] = {o[4], o[5], o[6], o[7], o[8], o[1]};
			// the logarithm of 1 + x errs by the rounding of that sum, also where x is below it
			const double round1[6] = {0, 0, 2 * e * E / (n * n * a), 2 * e * (b + E / n) / (a * a), 2 * e / a, 0};
			for (int d = 0; d < 6; ++d) ok &= std::fabs(got[d] - v * want[d]) <= v * (told * size[d] + round1[d]) + 1e-35;
			if (!ok && ++bad < 5) std::printf("bad: re %g rb %g n %g a %g b %g r %g: %g, %g, FP64 %g\n", re, rb, n, a, s[4], r, eval_at<float, CORESERSIC>(c, rf, 0.f), eval_fast<CORESERSIC>(c, rf, 0.f), v);
		}
	}
	std::printf("%s %ld %ld\n", bad ? "FAIL" : "ok", points, bad);
	return bad != 0;
}
