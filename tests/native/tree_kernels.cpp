// Runs the sub-pixel kernels (k_subsample_root, k_subsample_tree, k_subsample_mask)
// on the CPU with one host thread per GPU thread, a barrier per wavefront for the
// wavefront's exchanges and one per block for __syncthreads, under AddressSanitizer
// with every list and buffer at its exact size, and compares each pixel's value and
// Jacobian with a plain recursion over the same cell step: entries of the heavy
// list, big and small trees, trees that overflow the stack and are walked by masks.
// Prints "ok <case>".
#include <hip/hip_runtime.h>

#include <cstdio>
#include <memory>
#include <mutex>

#undef __shared__
#define __shared__ static
#define __constant__
#define __align__(n)
struct float4 {
	float x, y, z, w;
};
static std::unique_ptr<std::barrier<>> wave_bar[16];
static void wave_wait() { wave_bar[threadIdx.x >> 6]->arrive_and_wait(); }
static double wave_d[1024];
template <class T> static T wave_read(T v, unsigned lane)
{
	double w;
	static_assert(sizeof(T) <= sizeof(double));
	wave_wait();
	std::memcpy(&wave_d[threadIdx.x], &v, sizeof(T));
	wave_wait();
	std::memcpy(&w, &wave_d[(threadIdx.x & ~63u) + lane], sizeof(T));
	T r;
	std::memcpy(&r, &w, sizeof(T));
	return r;
}
static unsigned long long wave_ballot(bool p)
{
	static unsigned char vote[1024];
	wave_wait();
	vote[threadIdx.x] = p;
	wave_wait();
	unsigned long long m = 0;
	for (int l = 0; l < 64; ++l) m |= (unsigned long long)vote[(threadIdx.x & ~63u) + l] << l;
	return m;
}
template <class T> static T wave_shfl_xor(T v, int m) { return wave_read(v, (threadIdx.x & 63u) ^ (unsigned)m); }
template <class T> static T wave_shfl(T v, int l) { return wave_read(v, (unsigned)l & 63u); }
#define __ballot wave_ballot
#define __shfl_xor wave_shfl_xor
#define __shfl wave_shfl
#define __builtin_amdgcn_fence(...) wave_wait()
#define __builtin_amdgcn_wave_barrier() wave_wait()
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_readlane(v, l) (v)
static int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
static int __ffsll(long long m) { return __builtin_ffsll(m); }
static std::mutex atomic_mu;
template <class T> static T atomicAdd(T *p, T v)
{
	std::lock_guard<std::mutex> lock(atomic_mu);
	T o = *p;
	*p += v;
	return o;
}
using std::isfinite;
using std::max;
using std::min;
template <class A, class B> static long min(A a, B b) { return (long)a < (long)b ? (long)a : (long)b; }

#include "kernel_common.h"

using namespace profit_amd;

static void launch(unsigned grid, unsigned block, const std::function<void()> &k)
{
	for (unsigned w = 0; w < block / 64; ++w) wave_bar[w].reset(new std::barrier<>(64));
	hip_cpu::launch(grid, block, k);
}

template <int TYPE>
static void recurse(const Comp &c, double x0, double x1, double y0, double y1, double w, int res, int maxrec, int level,
                    double &sum, double *g, long &leaves)
{
	const Node n = make_node(c, refine_limits(c), x0, x1, y0, y1, res);
	const bool fuse = TYPE == SERSIC && !c.boxy && !c.grad_box;
	for (int cell = 0; cell < res * res; ++cell) {
		float gj[NGRAD] = {};
		if (!cell_step<TYPE, true>(c, n, cell, res > 1 && level < maxrec, false, fuse, w, sum, gj)) {
			for (int s = 0; s < NGRAD; ++s) g[s] += gj[s];
			++leaves;
			continue;
		}
		const double hx = (x1 - x0) / res / 2., hy = (y1 - y0) / res / 2.;
		const double cx = cell_centre(x0, hx, cell / res), cy = cell_centre(y0, hy, cell % res);
		recurse<TYPE>(c, cx - hx, cx + hx, cy - hy, cy + hy, w * kInvCells[res], res, maxrec, level + 1, sum, g, leaves);
	}
}

template <int TYPE, int W>
static bool check(const char *name, const std::vector<ProfileParams> &ps, double acc, bool mark, bool overflows)
{
	constexpr int DW = 9, DH = 7, kSlots = G_S0 + n_shape(TYPE);
	GalaxyDev g{};
	g.DW = g.W = DW;
	g.DH = g.H = DH;
	g.sx = g.sy = g.img_sx = g.img_sy = 1;
	std::vector<Comp> comps;
	for (ProfileParams p : ps) {
		Comp c{};
		sf::QuadState qs;
		p.type = TYPE;
		if (setup_component(p, 0, 1, 1, 1, 1, 0, 0, &qs, &c) != SE_OK) return false;
		c.grad_box = 0;
		c.instance = 0;
		if (acc >= 0) c.acc = acc, c.f.acc = (float)acc;
		comps.push_back(c);
	}
	std::vector<float> canvas(DW * DH, 0.f);
	InstDev I{};
	I.canvas = canvas.data();
	std::vector<QEntry> light, heavy;
	for (int k = 0; k < (int)comps.size(); ++k)
		for (int p = 0; p < DW * DH; ++p) {
			const Comp &c = comps[k];
			const double x = .5 + p % DW, y = .5 + p / DW, xr = x - c.xc, yr = y - c.yc;
			if (std::hypot(xr * c.cos_ang + yr * c.sin_ang, -xr * c.sin_over + yr * c.cos_over) > c.rsw_r) continue;
			(centre_pixel(c, x, y) ? heavy : light).push_back(QEntry{k, p});
		}
	const std::vector<QEntry> heavy0 = heavy;
	std::vector<int> count(kQueueCounters, 0), deep(light.size());
	std::vector<float> ljac(light.size() * kJacStride), hjac(heavy.size() * kJacStride);
	WorkQueue wq{};
	wq.light = light.data();
	wq.heavy = heavy.data();
	for (int f = 0; f <= kFamilies; ++f) wq.lbase[f] = f <= TYPE ? 0 : (int)light.size();
	wq.hcap = (int)heavy.size();
	wq.count = count.data();
	wq.ljac = ljac.data();
	wq.hjac = hjac.data();
	wq.deep = deep.data();
	count[1] = (int)heavy.size();
	count[light_count(TYPE)] = (int)light.size();
	launch(2, 256, [&] { k_subsample_root<TYPE, true>(&g, &I, comps.data(), wq, 0); });
	launch(2, 64 * W, [&] { k_subsample_tree<TYPE, true, W>(&g, &I, comps.data(), wq, 0, mark); });
	if (mark) launch(2, 256, [&] { k_subsample_mask<TYPE, true>(&g, &I, comps.data(), wq, 0); });
	bool ok = (count[0] > 0) == overflows;
	const int nd = count[deep_count(TYPE)], nb = count[big_count(TYPE)];
	if (overflows && !mark) {
		std::printf("%s %s overflow %d\n", ok ? "ok" : "FAIL", name, count[0]);
		return ok;
	}
	for (size_t k = 0; k < heavy.size(); ++k) ok &= heavy[k].pix == heavy0[k].pix && heavy[k].comp == heavy0[k].comp;
	std::vector<double> want(DW * DH, 0.0);
	double worst = 0;
	for (int list = 0; list < 2; ++list)
		for (size_t e = 0; e < (list ? heavy : light).size(); ++e) {
			const QEntry q = (list ? heavy : light)[e];
			const Comp &c = comps[q.comp];
			double sum = 0, gr[NGRAD] = {};
			long leaves = 0;
			const int x = q.pix % DW, y = q.pix / DW, res = list ? 8 : c.res;
			recurse<TYPE>(c, x, x + 1, y, y + 1, kInvCells[res], res, list ? 10 : c.maxrec, 0, sum, gr, leaves);
			want[q.pix] += c.flux_scale * sum;
			const float *J = (list ? hjac : ljac).data() + e * kJacStride;
			double scale = 0;
			for (int s = 0; s < kSlots; ++s) scale = std::max(scale, std::fabs(gr[s]));
			// FP32 sums of up to all leaves on a thread, added in FP64
			for (int s = 0; s < kSlots; ++s) {
				const double e1 = std::fabs(J[s] - gr[s]) / (6e-8 * (double)std::min(leaves, 4000L) * scale + 1e-30);
				worst = std::max(worst, e1);
				ok &= e1 <= 1;
			}
			ok &= std::fabs(J[kJacStride - 1] - sum) <= 1e-5 * sum;
		}
	// FP32 additions of the pixel's values
	for (int p = 0; p < DW * DH; ++p) ok &= std::fabs(canvas[p] - want[p]) <= 1e-6 * std::fabs(want[p]);
	std::printf("%s %s W %d: light %zu heavy %zu small %d big %d overflowed %d, Jacobian %.2g of its bound\n", ok ? "ok" : "FAIL",
	            name, W, light.size(), heavy.size(), nd, nb, count[0], worst);
	return ok;
}

int main()
{
	std::setvbuf(stdout, nullptr, _IOLBF, 0);
	auto par = [](double x, double y, double s0, double s1, double acc, int res, unsigned rec) {
		ProfileParams p;
		default_params(SERSIC, &p);
		p.xcen = x;
		p.ycen = y;
		p.ang = 20;
		p.axrat = 0.8;
		p.shape[0] = s0;
		p.shape[1] = s1;
		p.acc = acc;
		p.mag = -10;
		p.adjust = res == 0;
		p.resolution = res ? res : 9;
		p.max_recursions = rec;
		p.rscale_switch = 1.0;
		return p;
	};
	bool ok = true;
	// centre trees (heavy list) and ordinary ones
	ok &= check<SERSIC, 4>("adjusted", {par(4.4, 3.3, 1.5, 3, 0.1, 0, 2), par(2.2, 5.1, 2, 6, 0.1, 0, 2)}, -1, true, false);
	ok &= check<SERSIC, 12>("adjusted", {par(4.4, 3.3, 1.5, 3, 0.1, 0, 2)}, -1, false, false);
	// more than 64 cells a node, odd resolutions, leaf-only entries, and a tree that overflows
	const std::vector<ProfileParams> mixed = {par(4.4, 3.3, 2, 3, 0.05, 11, 2), par(5.5, 2.1, 2, 1, 0.3, 5, 2), par(1.5, 1.5, 1, 0.6, 0.9, 3, 1)};
	ok &= check<SERSIC, 4>("resolutions", mixed, -1, false, true);
	ok &= check<SERSIC, 4>("resolutions", mixed, -1, true, true);
	// a centre tree that overflows
	ok &= check<SERSIC, 4>("centre", {par(5 - 1e-5, 4 - 1e-5, 0.9, 8, 0.1, 0, 2)}, 0.08, true, true);
	ProfileParams k = par(4.2, 3.4, 1.0, 3, 0.05, 6, 2);
	k.shape[2] = 6.0;
	ok &= check<KING, 4>("king", {k}, -1, true, true);
	return ok ? 0 : 1;
}
