// Runs the tree walk (walk_tree) on the CPU with one host thread per GPU
// thread, by a wavefront and by a block, under AddressSanitizer, and compares
// it with a plain recursion over the same cell step: the value and Jacobian
// sums, the number of leaves' total weight, and the overflow of its stack.
// Every wavefront primitive waits for the whole block, so a barrier that only
// some threads reach would hang here.  Prints "ok <case>" per case.
#include <hip/hip_runtime.h>

#include <cstdio>

#define __constant__
#define __align__(n)
#define __builtin_amdgcn_fence(...) __syncthreads()
#define __builtin_amdgcn_wave_barrier() (void)0
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, l) (v)
struct float4 {
	float x, y, z, w;
};
static unsigned char vote[1024];
static unsigned long long __ballot(bool p)
{
	vote[threadIdx.x] = p;
	__syncthreads();
	unsigned long long m = 0;
	for (int l = 0; l < 64; ++l) m |= (unsigned long long)vote[(threadIdx.x & ~63u) + l] << l;
	__syncthreads();
	return m;
}
static int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
static int __ffsll(long long m) { return __builtin_ffsll(m); }
static int __shfl_xor(int v, int m) { return (int)__shfl_xor((double)v, m); }
template <class T> static T atomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
using std::isfinite;
using std::max;
using std::min;
template <class A, class B> static long min(A a, B b) { return (long)a < (long)b ? (long)a : (long)b; }

#include "kernel_common.h"

using namespace profit_amd;

template <int TYPE>
static void recurse(const Comp &c, double x0, double x1, double y0, double y1, double w, int res, int maxrec, int level,
                    double &sum, float *gj, long &leaves)
{
	const Node n = make_node(c, refine_limits(c), x0, x1, y0, y1, res);
	const bool fuse = TYPE == SERSIC && !c.boxy && !c.grad_box;
	for (int cell = 0; cell < res * res; ++cell) {
		if (!cell_step<TYPE, true>(c, n, cell, res > 1 && level < maxrec, false, fuse, w, sum, gj)) {
			++leaves;
			continue;
		}
		const double hx = (x1 - x0) / res / 2., hy = (y1 - y0) / res / 2.;
		const double cx = cell_centre(x0, hx, cell / res), cy = cell_centre(y0, hy, cell % res);
		recurse<TYPE>(c, cx - hx, cx + hx, cy - hy, cy + hy, w * kInvCells[res], res, maxrec, level + 1, sum, gj, leaves);
	}
}

template <int TYPE, int T>
static bool check(const char *name, ProfileParams p, double px, double py, int res, int maxrec, bool overflows)
{
	Comp c;
	sf::QuadState qs;
	p.type = TYPE;
	if (setup_component(p, 0, 1, 1, 1, 1, 0, 0, &qs, &c) != SE_OK) return false;
	c.grad_box = 0;
	constexpr int W = T == 64 ? 4 : T / 64;
	// guard memory on both sides of the stack is the sanitizer's
	TreeStack<W> *S = new TreeStack<W>;
	std::vector<double> sum(T, 0.0);
	std::vector<float> gj((size_t)T * NGRAD, 0.f);
	std::vector<char> ok(T);
	hip_cpu::launch(1, T, [&] {
		const int t = threadIdx.x;
		ok[t] = walk_tree<TYPE, true, T>(c, *S, 0, t, px, px + 1, py, py + 1, res, maxrec, false, sum[t], &gj[(size_t)t * NGRAD]);
	});
	delete S;
	for (char v : ok)
		if ((bool)v == overflows) return std::printf("FAIL %s: overflow %d\n", name, !v), false;
	if (overflows) return std::printf("ok %s %d overflow\n", name, T), true;
	double ref = 0, got = 0;
	float rg[NGRAD] = {};
	long leaves = 0;
	recurse<TYPE>(c, px, px + 1, py, py + 1, kInvCells[res], res, maxrec, 0, ref, rg, leaves);
	for (double v : sum) got += v;
	// the same FP64 terms in another order: leaves * 2^-53 of a sum of positive terms
	bool good = std::fabs(got - ref) <= 2.3e-16 * (double)(leaves + T) * std::fabs(ref);
	double scale = 0;
	for (int s = 0; s < NGRAD; ++s) scale = std::max(scale, (double)std::fabs(rg[s]));
	for (int s = 0; s < NGRAD; ++s) {
		double g = 0;
		for (int t = 0; t < T; ++t) g += gj[(size_t)t * NGRAD + s];
		// FP32 sums of `leaves` terms on both sides
		good &= std::fabs(g - rg[s]) <= 1.2e-7 * (double)leaves * std::max(scale, 1e-30);
	}
	std::printf("%s %s %d leaves %ld\n", good ? "ok" : "FAIL", name, T, leaves);
	return good;
}

int main()
{
	auto par = [](int type, double s0, double s1, double s2 = 0, double acc = 0.1) {
		ProfileParams p;
		default_params(type, &p);
		p.xcen = 0.37;
		p.ycen = 0.58;
		p.ang = 33;
		p.axrat = 0.7;
		p.adjust = 0;
		p.acc = acc;
		p.shape[0] = s0;
		p.shape[1] = s1;
		if (type == FERRER || type == KING) p.shape[2] = s2;
		return p;
	};
	bool ok = true;
	const ProfileParams cusp = par(SERSIC, 3, 4), flat = par(SERSIC, 30, 0.5), all = par(SERSIC, 3, 4, 0, 0);
	// a centre tree, a leaf-only root, full refinement by every resolution's remainder, and overflows
	ok &= check<SERSIC, 256>("centre", cusp, 0, 0, 8, 10, false);
	ok &= check<SERSIC, 64>("centre", cusp, 0, 0, 8, 6, false);
	ok &= check<SERSIC, 256>("leaf", flat, 5, 5, 4, 3, false);
	ok &= check<SERSIC, 64>("leaf", flat, 5, 5, 16, 3, false);
	ok &= check<SERSIC, 256>("res1", all, 2, 1, 1, 3, false);
	ok &= check<SERSIC, 64>("full4", all, 2, 1, 4, 2, false);
	ok &= check<SERSIC, 256>("full5", all, 2, 1, 5, 2, false);
	ok &= check<SERSIC, 64>("full10", all, 2, 1, 10, 1, false);
	ok &= check<SERSIC, 256>("full16", all, 2, 1, 16, 1, false);
	ok &= check<SERSIC, 64>("full16", all, 2, 1, 16, 1, false);
	ok &= check<SERSIC, 64>("full16", all, 2, 1, 16, 2, true);
	ok &= check<SERSIC, 256>("full16", all, 2, 1, 16, 5, true);
	ok &= check<SERSIC, 768>("centre", cusp, 0, 0, 8, 10, false);
	ok &= check<SERSIC, 768>("full10", all, 2, 1, 10, 1, false);
	ok &= check<KING, 256>("king", par(KING, 0.3, 2.0, 2.0), 0, 0, 10, 3, false);
	ok &= check<FERRER, 64>("ferrer", par(FERRER, 1.3, 1.0, 0.5), 0, 1, 6, 3, false);
	return ok ? 0 : 1;
}
