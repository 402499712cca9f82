// The FP32 refinement test against the FP64 one on the CPU, over random
// components of a family and random cells of their sub-sampled pixels, with the
// transcendental unit's results off by up to one unit in the last place.  For
// each cell the accuracy `acc` is set to the cell's own |test - val| / val, so
// that its FP64 margin is zero: the FP32 test must leave such a cell undecided
// with half the component's guard band.  Prints "ok <family> ..." per family, and
// of a failing one the worst margin and its parameters.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <random>

#define __constant__
#define __align__(n)
#define __builtin_amdgcn_fence(...) (void)0
#define __builtin_amdgcn_wave_barrier() (void)0
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, l) (v)
struct float4 {
	float x, y, z, w;
};
static unsigned long long __ballot(bool p) { return p; }
static int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
static int __ffsll(long long m) { return __builtin_ffsll(m); }
static int __shfl_xor(int v, int) { return v; }
template <class T> static T atomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
using std::isfinite;
using std::max;
using std::min;
template <class A, class B> static long min(A a, B b) { return (long)a < (long)b ? (long)a : (long)b; }

// a correctly rounded result moved by -1, 0 or 1 ulp
static std::mt19937_64 rng(20240607);
static float nudge(float v)
{
	const unsigned k = (unsigned)(rng() >> 60) % 3u;
	return k == 0 ? std::nextafterf(v, -INFINITY) : k == 1 ? std::nextafterf(v, INFINITY) : v;
}
static float unit_log2(float x) { return nudge((float)std::log2((double)x)); }
static float unit_exp2(float x) { return nudge((float)std::exp2((double)x)); }
static float unit_sqrt(float x) { return nudge(std::sqrt(x)); }
static float unit_rcp(float x) { return nudge(1.f / x); }
#define __builtin_amdgcn_logf unit_log2
#define __builtin_amdgcn_exp2f unit_exp2
#define __builtin_amdgcn_sqrtf unit_sqrt
#define __builtin_amdgcn_rcpf unit_rcp

#include "kernel_common.h"

using namespace profit_amd;

static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static double logu(double a, double b) { return std::exp(uni(std::log(a), std::log(b))); }

template <int TYPE>
static ProfileParams draw()
{
	ProfileParams p;
	default_params(TYPE, &p);
	p.xcen = uni(0, 1);
	p.ycen = uni(0, 1);
	if (uni(0, 1) < 0.2) p.xcen = p.ycen = 0.5;
	p.ang = uni(0, 180);
	p.axrat = uni(0, 1) < 0.5 ? uni(0.2, 1) : logu(0.03, 1);
	p.box = uni(0, 1) < 0.7 ? 0.0 : uni(-1.6, 4);
	p.adjust = uni(0, 1) < 0.5;
	p.rscale_switch = logu(0.3, 2);
	p.resolution = 2 + (unsigned)(uni(0, 1) * 14.99);
	double *s = p.shape;
	switch (TYPE) {
	case SERSIC: s[0] = logu(0.5, 100); s[1] = logu(0.2, 12); break;
	case MOFFAT: s[0] = logu(0.5, 50); s[1] = logu(1.1, 1000); break;
	case FERRER: s[0] = logu(1, 200); s[1] = logu(0.1, 12); s[2] = 2 - logu(0.003, 8); break;
	case KING: s[0] = logu(0.2, 20); s[1] = s[0] * logu(0.3, 60); s[2] = logu(0.3, 12); break;
	case CORESERSIC: s[0] = logu(1, 60); s[1] = s[0] * logu(0.02, 2); s[2] = logu(0.5, 8); s[3] = logu(0.1, 30); s[4] = uni(-1, 1.95); break;
	default: s[0] = logu(0.5, 40); s[1] = logu(0.5, 40); s[2] = logu(0.5, 60); s[3] = logu(0.05, 30); break;
	}
	return p;
}

template <int TYPE>
static bool check(const char *name, int ncomp, int ncell)
{
	double worst = 0;
	long tested = 0, wrong = 0;
	ProfileParams bad{};
	for (int k = 0; k < ncomp; ++k) {
		const ProfileParams p = draw<TYPE>();
		Comp c;
		sf::QuadState qs;
		if (setup_component(p, 0, 1, 1, 1, 1, 0, 0, &qs, &c, false) != SE_OK) continue;
		for (int m = 0; m < ncell; ++m) {
			// a pixel whose centre lies inside the switch radius, then a node of
			// its tree and a cell of it
			const double r = c.rsw_r * std::sqrt(uni(0, 1)) * (uni(0, 1) < 0.3 ? uni(0, 1) : 1), th = uni(0, 6.283185307);
			const double xp = r * std::cos(th), yq = r * std::sin(th) * p.axrat;
			double x0 = std::floor(c.xc + xp * c.cos_ang - yq * c.sin_ang), y0 = std::floor(c.yc + xp * c.sin_ang + yq * c.cos_ang);
			if (uni(0, 1) < 0.1) x0 = y0 = 0;
			const double qx = x0 + .5 - c.xc, qy = y0 + .5 - c.yc;
			if (std::hypot(qx * c.cos_ang + qy * c.sin_ang, -qx * c.sin_over + qy * c.cos_over) > c.rsw_r) continue;
			double x1 = x0 + 1, y1 = y0 + 1;
			const int res = c.res, depth = (int)uni(0, 3);
			for (int d = 0; d < depth; ++d) {
				const double hx = (x1 - x0) / res / 2., hy = (y1 - y0) / res / 2.;
				int ci = (int)uni(0, res), cj = (int)uni(0, res);
				if (uni(0, 1) < 0.5) {  // towards the centre
					ci = (int)std::fmin(std::fmax((c.xc - x0) / (2 * hx), 0), res - 1);
					cj = (int)std::fmin(std::fmax((c.yc - y0) / (2 * hy), 0), res - 1);
				}
				const double cx = cell_centre(x0, hx, ci), cy = cell_centre(y0, hy, cj);
				x0 = cx - hx, x1 = cx + hx, y0 = cy - hy, y1 = cy + hy;
			}
			Node n = make_node(c, refine_limits(c), x0, x1, y0, y1, res);
			const int ci = (int)uni(0, res), cj = (int)uni(0, res);
			const double xb = (x1 - x0) / res, yb = (y1 - y0) / res;
			double X, Y, v;
			cell_pos64(c, x0, y0, xb / 2., yb / 2., ci, cj, &X, &Y);
			const double dyp = -xb * c.sin_over + yb * c.cos_over;
			refine_cell64<TYPE>(c, X, Y, dyp, &v);
			const double t = eval_at<double, TYPE>(c, std::fabs(X), std::fabs(Y) + std::fabs(dyp));
			c.acc = std::fabs(t - v) / v;
			if (!(c.acc < 10)) continue;
			c.f.acc = (float)c.acc;
			float xf, yf;
			cell_pos32(c, n.ox, n.oy, n.xbin, n.ybin, ci, cj, &xf, &yf);
			const float vf = eval_at<float, TYPE>(c, xf, yf);
			n.test.acc = c.f.acc;
			n.test.band = 0.5f * guard_band(c, guard_radius(c, 1, 1));
			const int dec = refine_cell32<TYPE>(c, xf, yf, n.test, vf);
			++tested;
			if (dec == 2 || v == 0) continue;
			++wrong;
			const float tf = eval_fast<TYPE>(c, std::fabs(xf), std::fabs(yf) + std::fabs(n.test.dyp));
			const double e = std::fabs(std::fabs(tf - vf) / vf - c.acc);
			if (e > worst) {
				worst = e;
				bad = p;
			}
		}
	}
	std::printf("%s %s %ld cells, %ld decided, worst margin %.2e", wrong ? "FAIL" : "ok", name, tested, wrong, worst);
	if (wrong) std::printf(" (shape %g %g %g %g %g axrat %g box %g)", bad.shape[0], bad.shape[1], bad.shape[2], bad.shape[3], bad.shape[4], bad.axrat, bad.box);
	std::printf("\n");
	return !wrong;
}

int main(int argc, char **argv)
{
	const int n = argc > 1 ? std::atoi(argv[1]) : 300, m = 600;
	bool ok = true;
	ok &= check<SERSIC>("sersic", n, m);
	ok &= check<MOFFAT>("moffat", n, m);
	ok &= check<FERRER>("ferrer", n, m);
	ok &= check<KING>("king", n, m);
	ok &= check<CORESERSIC>("coresersic", n, m);
	ok &= check<BROKENEXP>("brokenexp", n, m);
	return ok ? 0 : 1;
}
