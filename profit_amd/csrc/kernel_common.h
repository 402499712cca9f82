// Device code shared by the kernel translation units: block ownership,
// wave reductions, libprofit's cell positions and refinement test, and the
// templates of the sub-pixel walks and of the adjoint kernels.
// walkers_fwd.hip compiles the forward walks once per profile family and
// walkers_adj.hip the sub-pixel adjoint once per family and the adjoint render
// once per family and sum precision: a kernel's register allocation is the
// maximum over the code it holds, so one family per kernel lifts the walks
// from two to three or four waves per SIMD and the adjoint render from two
// to seven or eight.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"

namespace profit_amd {

// The instance whose block range [off[i], off[i+1]) holds block b (off: the
// n + 1 prefix sums of the instances' block counts).
__device__ inline int owner_of(const int *__restrict__ off, int n, int b)
{
	// a first guess from the mean count per instance (exact, up to the
	// rounding that the neighbour checks absorb, when every instance has the
	// same count), then the binary search if it misses
	int gs = min(n - 1, (int)((float)b * ((float)n / (float)off[n])));
	if (gs > 0 && off[gs] > b) --gs;
	else if (gs + 1 < n && off[gs + 1] <= b) ++gs;
	if (off[gs] <= b && off[gs + 1] > b) return gs;
	int lo = 0, hi = n - 1;
	while (lo < hi) {
		const int mid = (lo + hi + 1) >> 1;
		if (off[mid] <= b) lo = mid;
		else hi = mid - 1;
	}
	return lo;
}

__device__ inline double wave_sum(double v)
{
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
	return v;
}

// A 64-bit value that is the same on every lane, moved to scalar registers.
__device__ __forceinline__ unsigned long long uniform64(unsigned long long v)
{
	const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
	return (unsigned long long)hi << 32 | lo;
}

// 1 / res^2 and 1 / res for the recursion's resolutions 1 .. 16 (setup
// rejects higher ones), correctly rounded like the divisions they replace
static __constant__ double kInvCells[17] = {0.0,        1.0 / 1,   1.0 / 4,   1.0 / 9,   1.0 / 16,  1.0 / 25,
                                            1.0 / 36,   1.0 / 49,  1.0 / 64,  1.0 / 81,  1.0 / 100, 1.0 / 121,
                                            1.0 / 144,  1.0 / 169, 1.0 / 196, 1.0 / 225, 1.0 / 256};
static __constant__ float kInvRes[17] = {0.f,       1.f / 1,  1.f / 2,  1.f / 3,  1.f / 4,  1.f / 5,
                                         1.f / 6,   1.f / 7,  1.f / 8,  1.f / 9,  1.f / 10, 1.f / 11,
                                         1.f / 12,  1.f / 13, 1.f / 14, 1.f / 15, 1.f / 16};

// sersic.cpp:331-347: pixels within one image pixel of the centre of an
// nser > 1 Sersic profile are sub-sampled at resolution 8, depth 10
__device__ __forceinline__ bool centre_pixel(const Comp &c, double x, double y)
{
	return c.centre_rule && fabs(x - c.xc) < c.img_sx && fabs(y - c.yc) < c.img_sy;
}

struct WalkLevel {
	double x0, x1, y0, y1, weight;
	unsigned long long mask[4];
};

__device__ __forceinline__ double cell_centre(double lo, double half, int idx)
{
	// the same sequence of additions as libprofit's loops (radial.cpp:86-106)
	double v = lo;
	for (int t = 0; t < idx; ++t) {
		v += half;
		v += half;
	}
	return v + half;
}

// The rectangle of pixel centres a canvas tile (64 x 4 rows, at tile
// coordinates t) spans.
struct TileRect {
	double x0, x1, y0, y1;
};

__device__ __forceinline__ TileRect tile_rect(const GalaxyDev &g, int2 t, int rows)
{
	const double hx = g.sx / 2., hy = g.sy / 2.;
	const int i0 = t.x * kTileW, i1 = min(i0 + kTileW, g.DW) - 1;
	const int j0 = t.y * 4 * rows, j1 = min(j0 + 4 * rows, g.DH) - 1;
	return TileRect{hx + i0 * g.sy, hx + i1 * g.sy, hy + j0 * g.sx, hy + j1 * g.sx};
}

// What a component does on a tile: 0 nothing (every pixel beyond rscale_max),
// 2 every pixel drawn directly, 1 anything else.  The profile radius is at
// least the distance from the centre (axrat <= 1) and, being convex, largest
// at a corner; the margins of 1e-4 are far beyond the FP32 errors here and
// beyond classify32's band, so a 0 or 2 agrees with every pixel's own class.
// The render leaves dmask untouched where this is 0, and the adjoint render
// asks again before it reads dmask: both through this function.
__device__ __forceinline__ int tile_class(const Comp &c, const TileRect &r)
{
	if (!is_radial(c.type)) return 1;
	const float ax = (float)(r.x0 - c.xc), bx = (float)(r.x1 - c.xc);
	const float ay = (float)(r.y0 - c.yc), by = (float)(r.y1 - c.yc);
	const float dx = fmaxf(fmaxf(ax, -bx), 0.f), dy = fmaxf(fmaxf(ay, -by), 0.f);
	const float near2 = dx * dx + dy * dy;
	if (c.has_rmax) {
		const float lim = 1.0001f;
		const float cq = c.f.cos_ang, sq = c.f.sin_ang, q = c.f.axrat;
		// half extents of the ellipse of radius rscale_max, squared
		const float ex2 = c.f.rmax2 * (cq * cq + q * q * sq * sq), ey2 = c.f.rmax2 * (sq * sq + q * q * cq * cq);
		if (near2 > lim * c.f.rmax2 || dx * dx > lim * ex2 || dy * dy > lim * ey2) return 0;
	}
	if (!c.rough && !(near2 > 1.0001f * c.f.rsw2)) return 1;
	if (c.has_rmax) {
		float far2 = 0.f;
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			const float x = (k & 1) ? bx : ax, y = (k & 2) ? by : ay;
			const float xp = x * c.f.cos_ang + y * c.f.sin_ang, yp = -x * c.f.sin_over + y * c.f.cos_over;
			far2 = fmaxf(far2, xp * xp + yp * yp);
		}
		if (!(far2 < 0.9999f * c.f.rmax2)) return 1;
	}
	return 2;
}

// components whose tile classes a block keeps as bit masks (the ones beyond
// are taken as class 1)
constexpr int kCullWords = 64;

// d(f)/d slot of one sample in precision T, chain rule to the component
// slots, accumulated with weight wgt (FP64) into gs; returns f.  TYPE >= 0
// compiles the one profile family (see eval_at).
template <class T, int TYPE = -1>
__device__ __forceinline__ double sample_accumulate(const Comp &c, double xp, double yp, double wgt, double *gs)
{
	T o[9];
	const T fxp = (T)xp, fyp = (T)yp;
	sample_grad<T, TYPE>(c, fxp, fyp, o);
	// the rotation's chain rule with the per-component sin/q, cos/q and 1/q
	const T q = (T)c.axrat, iq = (T)c.inv_axrat;
	const T ca = (T)c.cos_ang, sa = (T)c.sin_ang;
	const T sq = (T)c.sin_over, cq = (T)c.cos_over;
	const T fx = o[1], fy = o[2];
	gs[G_XCEN] = fma(wgt, (double)(fx * -ca + fy * sq), gs[G_XCEN]);
	gs[G_YCEN] = fma(wgt, (double)(fx * -sa + fy * -cq), gs[G_YCEN]);
	gs[G_ANG] = fma(wgt, (double)((fx * (q * fyp) + fy * (-fxp * iq)) * (T(3.14159265358979323846) / T(180))), gs[G_ANG]);
	gs[G_AXRAT] = fma(wgt, (double)(fy * (-fyp * iq)), gs[G_AXRAT]);
	if (c.grad_box) gs[G_BOX] = fma(wgt, (double)o[3], gs[G_BOX]);
#pragma unroll
	for (int s = 0; s < n_shape(TYPE); ++s) gs[G_S0 + s] = fma(wgt, (double)o[4 + s], gs[G_S0 + s]);
	return (double)o[0];
}

// The same for a Sersic sample without box: the FP32 derivatives from the
// value's own logarithm and exponentials, with no powers or signs of the
// general form (and two logarithms more where d / d box is wanted).  A 500-source
// field's steep cores, every slot wanted: 2.27 -> 2.01 ms.
__device__ __forceinline__ double sersic_accumulate(const Comp &c, double xp, double yp, double wgt, double *gs)
{
#pragma clang fp contract(fast)
	const float x = (float)xp, y = (float)yp;
	float base, l2, rf;
	const float f = sersic_parts_f32(c, x, y, base, l2, rf);
	if (!(base > 0.f)) return (double)f;  // the centre: every derivative is 0
	const float bfr = c.f.bn * f * rf * c.f.inv_n;
	const float k = -bfr * c.f.inv_re2 * __builtin_amdgcn_rcpf(base);
	const float fx = k * x, fy = k * y;
	const float q = c.f.axrat, iq = c.f.inv_axrat;
	gs[G_XCEN] = fma(wgt, (double)(fx * -c.f.cos_ang + fy * c.f.sin_over), gs[G_XCEN]);
	gs[G_YCEN] = fma(wgt, (double)(fx * -c.f.sin_ang + fy * -c.f.cos_over), gs[G_YCEN]);
	gs[G_ANG] = fma(wgt, (double)((fx * (q * y) + fy * (-x * iq)) * (3.14159265358979323846f / 180.f)), gs[G_ANG]);
	gs[G_AXRAT] = fma(wgt, (double)(fy * (-y * iq)), gs[G_AXRAT]);
	if (c.grad_box) {
		// d base / dB = pu ln u + pv ln v with u = |x| / re, pu = u^2, at B = 2;
		// ln u = ln(u^2) / 2
		const float pu = (x * x) * c.f.inv_re2, pv = (y * y) * c.f.inv_re2;
		const float d2 = (pu > 0.f ? pu * log2_fast(pu) : 0.f) + (pv > 0.f ? pv * log2_fast(pv) : 0.f);
		const float half_ln2 = 0.5f * float(kLn2);
		// inv_nB (dbase_dB / base - ln(base) / B), inv_nB = inv_n / 2
		const float t = 0.5f * half_ln2 * (d2 * __builtin_amdgcn_rcpf(base) - l2);
		gs[G_BOX] = fma(wgt, (double)(-bfr * t), gs[G_BOX]);
	}
	gs[G_S0] = fma(wgt, (double)(bfr * c.f.inv_re), gs[G_S0]);
	gs[G_S1] = fma(wgt, (double)(f * (-c.f.dbn * (rf - 1.f) + c.f.bn * rf * (l2 * float(kLn2)) * c.f.inv_n * c.f.inv_2n)), gs[G_S1]);
	return (double)f;
}

// Where a King or Ferrer cell lies against its profile's cut-off (rt, rout),
// from the FP32 radii of the cell centre (x, y) and of the test point
// (ax, ay), which lies at least as far out: 0 when the centre lies beyond
// 1.01 x the cut (the value and the test are then exactly 0 in either
// precision, so the cell is a leaf of value 0); 1 when the centre lies in
// [0.97, 1.01] x the cut or the test point within 1% of it, where the value is
// a difference of nearly equal terms (King: A - C; Ferrer: 1 - t^(2-b)) whose
// FP32 relative error grows without bound and a point can fall on either side
// of the cut (the FP64 test decides, and the leaf value is FP64); -1
// otherwise, and for the other families.
template <int TYPE>
__device__ __forceinline__ int cut_zone(const Comp &c, float x, float y, float ax, float ay)
{
	if (TYPE >= 0 && TYPE != KING && TYPE != FERRER) return -1;
	const int t = TYPE >= 0 ? TYPE : c.type;
	if (t != KING && t != FERRER) return -1;
	const float cut = t == KING ? c.f.s[1] : c.f.rscale;
	const float rc = boxy_r<float>(c, x, y), rt = boxy_r<float>(c, ax, ay);
	if (rc > 1.01f * cut) return 0;
	const bool band_c = rc >= 0.97f * cut, band_t = rt >= 0.99f * cut && rt <= 1.01f * cut;
	return band_c || band_t ? 1 : -1;
}

// The component's accuracy, guard band and near radius (Comp::F32), read once per
// tree or entry: where the test may not run, or behind a barrier, the component's
// fields would be loaded again for every cell or round (root pass of 300,000 entries
// 103 -> 117 us, tree walk 167 -> 182).
struct RefineLimits {
	float acc, band, rnear;
};

__device__ __forceinline__ RefineLimits refine_limits(const Comp &c) { return RefineLimits{c.f.acc, c.f.band, c.f.rnear}; }

// What the refinement test of a node's cells needs besides a cell's value: the test
// point's offset, the limits and the squared profile radius below which a cell is
// undecided.
struct RefineTest {
	float dyp, acc, band, near2;
};

__device__ __forceinline__ RefineTest refine_test(const RefineLimits &l, float dyp, float xbin)
{
	const float near = fmaxf(0.05f * xbin, l.rnear);
	return RefineTest{dyp, l.acc, l.band, near * near};
}

// libprofit's refinement test |test - val| > acc * val (radial.cpp:92-100),
// evaluated in FP32 at FP32 cell positions: 1 refine, 0 leaf, 2 undecided.
// The decision is taken only when the FP32 margin lies outside the component's guard
// band, which covers the FP32 errors of values and positions (guard_band), so it equals
// the FP64 one.  The positions err by 6e-8 of the node, which is more than the band
// allows for next to the profile's centre: a cell within 5% of a cell of it is
// undecided, as is one so close that a box's powers underflow (RefineTest::near2).  King and
// Ferrer cells beyond their cut-off are leaves; those near it are undecided (cut_zone).
// Undecided cells take refine_cell64 at libprofit's own FP64 cell position, and its
// value if they are leaves.  Ordinary shapes have a band of 2.5e-4; one of 1e-3 for all
// sent four times the cells to FP64, half the root pass of a King family (77 of them:
// 1.64 ms, 0.80 now), with the same image errors against FP64 (the FP64 leaf values
// within 1e-3 change them by less than 1%).
template <int TYPE = -1>
__device__ __forceinline__ int refine_cell32(const Comp &c, float xp, float yp, const RefineTest &rt, float v32)
{
	const float ax = fabsf(xp), ay = fabsf(yp) + fabsf(rt.dyp);
	const int zone = cut_zone<TYPE>(c, xp, yp, ax, ay);
	if (zone == 0) return 0;
	if (zone == 1) return 2;
	const float t32 = eval_fast<TYPE>(c, ax, ay);
	const float margin = fabsf(t32 - v32) - rt.acc * v32;
	if (!(v32 > 1e-30f && isfinite(margin) && fabsf(margin) > rt.band * v32 && xp * xp + yp * yp >= rt.near2)) return 2;
	return margin > 0.f ? 1 : 0;
}

// the FP64 refinement test; *v64 receives the FP64 value
template <int TYPE = -1>
__device__ __forceinline__ bool refine_cell64(const Comp &c, double xp, double yp, double dyp, double *v64)
{
	const double v = eval_at<double, TYPE>(c, xp, yp);
	const double t = eval_at<double, TYPE>(c, fabs(xp), fabs(yp) + fabs(dyp));
	*v64 = v;
	return fabs(t - v) > c.acc * v;
}

// Profile coordinates of cell (ci, cj) in FP32: the node's lower corner
// relative to the component centre (ox, oy, formed once per node in FP64 and
// rounded) plus the cell's offset.  Relative to the distance from the centre
// the position errs by a few parts in 1e8, which moves a profile value by
// |d ln f / d ln r| times that: far inside the refinement test's guard band.
__device__ __forceinline__ void cell_pos32(const Comp &c, float ox, float oy, float fxbin, float fybin, int ci, int cj,
                                           float *xp, float *yp)
{
	const float dx = ox + ((float)ci + 0.5f) * fxbin;
	const float dy = oy + ((float)cj + 0.5f) * fybin;
	*xp = dx * c.f.cos_ang + dy * c.f.sin_ang;
	*yp = -dx * c.f.sin_over + dy * c.f.cos_over;
}

// libprofit's FP64 cell position (its sequence of additions, radial.cpp:86-106)
// in profile coordinates
__device__ __forceinline__ void cell_pos64(const Comp &c, double nx0, double ny0, double hx, double hy, int ci, int cj,
                                           double *xp, double *yp)
{
	const double x = cell_centre(nx0, hx, ci), y = cell_centre(ny0, hy, cj);
	const double xr = x - c.xc, yr = y - c.yc;
	*xp = xr * c.cos_ang + yr * c.sin_ang;
	*yp = -xr * c.sin_over + yr * c.cos_over;
}

// d(f)/d slot of one sample in FP32, chain rule to the component slots,
// accumulated with weight wgt into FP32 sums gs; returns f.
template <int TYPE>
__device__ __forceinline__ float pixel_accumulate_f32(const Comp &c, float xp, float yp, float wgt, float *gs)
{
	// FP32 derivatives only: products and sums may fuse into FMAs
#pragma clang fp contract(fast)
	float o[9];
	sample_grad<float, TYPE>(c, xp, yp, o);
	// the rotation's chain rule with the per-component sin/q, cos/q and 1/q
	const float q = c.f.axrat, iq = c.f.inv_axrat;
	const float ca = c.f.cos_ang, sa = c.f.sin_ang;
	const float sq = c.f.sin_over, cq = c.f.cos_over;
	const float fx = o[1], fy = o[2];
	gs[G_XCEN] += wgt * (fx * -ca + fy * sq);
	gs[G_YCEN] += wgt * (fx * -sa + fy * -cq);
	gs[G_ANG] += wgt * ((fx * (q * yp) + fy * (-xp * iq)) * (3.14159265358979323846f / 180.f));
	gs[G_AXRAT] += wgt * (fy * (-yp * iq));
	if (c.grad_box) gs[G_BOX] += wgt * o[3];
#pragma unroll
	for (int s = 0; s < n_shape(TYPE); ++s) gs[G_S0 + s] += wgt * o[4 + s];
	return o[0];
}

// The same for a Sersic sample without box from the intermediates of its
// value (sersic_parts_f32): f, base = (r / re)^2, l2 = log2(base), rf =
// base^(1/(2n)), so that a leaf pays no second logarithm or exponential.
__device__ __forceinline__ void sersic_jac_f32(const Comp &c, float xp, float yp, float f, float base, float l2,
                                               float rf, float wgt, float *gs)
{
#pragma clang fp contract(fast)
	if (!(base > 0.f)) return;  // the centre: every derivative is 0
	const float bn = c.f.bn, in = c.f.inv_n;
	const float bfr = bn * f * rf * in;
	// df/dxp = k xp, df/dyp = k yp with k = -bn f rf / (n re^2 base)
	const float k = -bfr * c.f.inv_re2 * __builtin_amdgcn_rcpf(base);
	const float fx = k * xp, fy = k * yp;
	const float q = c.f.axrat, iq = c.f.inv_axrat;
	gs[G_XCEN] += wgt * (fx * -c.f.cos_ang + fy * c.f.sin_over);
	gs[G_YCEN] += wgt * (fx * -c.f.sin_ang + fy * -c.f.cos_over);
	gs[G_ANG] += wgt * ((fx * (q * yp) + fy * (-xp * iq)) * (3.14159265358979323846f / 180.f));
	gs[G_AXRAT] += wgt * (fy * (-yp * iq));
	gs[G_S0] += wgt * (bfr * c.f.inv_re);
	gs[G_S1] += wgt * (f * (-c.f.dbn * (rf - 1.f) + bn * rf * (l2 * float(kLn2)) * in * c.f.inv_2n));
}

// A node of the recursion: its FP64 bounds (libprofit's), the resolution,
// and the FP32 cell size, refinement test and lower corner relative to the
// component centre that the FP32 cell positions use.
struct Node {
	double x0, x1, y0, y1;
	int res;
	float inv_res, xbin, ybin, ox, oy;
	RefineTest test;
};

__device__ __forceinline__ Node make_node(const Comp &c, const RefineLimits &lim, double x0, double x1, double y0,
                                          double y1, int res)
{
	Node n;
	n.x0 = x0;
	n.x1 = x1;
	n.y0 = y0;
	n.y1 = y1;
	n.res = res;
	n.inv_res = kInvRes[res];
	n.xbin = (float)(x1 - x0) * n.inv_res;
	n.ybin = (float)(y1 - y0) * n.inv_res;
	n.test = refine_test(lim, -n.xbin * c.f.sin_over + n.ybin * c.f.cos_over, n.xbin);
	n.ox = (float)(x0 - c.xc);
	n.oy = (float)(y0 - c.yc);
	return n;
}

// One cell of a node: its FP32 position, value and refinement test (in FP64
// at libprofit's own cell centre when the FP32 test is undecided); a leaf
// adds weight * value to sum and, with kJac, its weighted FP32 derivatives
// to gj.  `fuse`: a Sersic without box, whose derivatives reuse the value's
// logarithm and exponentials.  Returns whether the cell is to be refined.
template <int TYPE, bool kJac>
__device__ __forceinline__ bool cell_step(const Comp &c, const Node &n, int cell, bool recurse, bool fp64, bool fuse,
                                          double weight, double &sum, float *gj)
{
	// libprofit's FP64 cell size and test offset, for the cells that need an
	// FP64 position
	auto node64 = [&](double &hx, double &hy, double &dyp) {
		const double xbin = (n.x1 - n.x0) / n.res;
		const double ybin = (n.y1 - n.y0) / n.res;
		hx = xbin / 2.;
		hy = ybin / 2.;
		dyp = -xbin * c.sin_over + ybin * c.cos_over;
	};
	// cell -> (ci, cj) by an FP32 reciprocal: (cell + 0.5) / res lies at least
	// 0.5 / res from an integer, far beyond the product's rounding, so the
	// truncation is the exact quotient
	const int ci = (int)(((float)cell + 0.5f) * n.inv_res), cj = cell - ci * n.res;
	float xp, yp;
	cell_pos32(c, n.ox, n.oy, n.xbin, n.ybin, ci, cj, &xp, &yp);
	float v32, s_base = 0.f, s_l2 = 0.f, s_rf = 0.f;
	if (fuse) v32 = sersic_parts_f32(c, xp, yp, s_base, s_l2, s_rf);
	else v32 = eval_at<float, TYPE>(c, xp, yp);
	int dec = recurse ? refine_cell32<TYPE>(c, xp, yp, n.test, v32) : 0;
	double v64 = 0;
	bool have64 = false;
	if (dec == 2) {
		double hx, hy, dyp, xp64, yp64;
		node64(hx, hy, dyp);
		cell_pos64(c, n.x0, n.y0, hx, hy, ci, cj, &xp64, &yp64);
		dec = refine_cell64<TYPE>(c, xp64, yp64, dyp, &v64) ? 1 : 0;
		have64 = true;
	}
	if (dec == 1) return true;
	// leaf values in FP64 or the FP32 value already at hand
	if (!have64) {
		if (fp64) {
			double hx, hy, dyp, xp64, yp64;
			node64(hx, hy, dyp);
			cell_pos64(c, n.x0, n.y0, hx, hy, ci, cj, &xp64, &yp64);
			v64 = eval_at<double, TYPE>(c, xp64, yp64);
		}
		else {
			v64 = (double)v32;
		}
	}
	sum += v64 * weight;
	if (fuse) sersic_jac_f32(c, xp, yp, v32, s_base, s_l2, s_rf, (float)weight, gj);
	else if (kJac) pixel_accumulate_f32<TYPE>(c, xp, yp, (float)weight, gj);
	return false;
}

// Walks the recursion tree of one pixel of a TYPE profile.  Cell positions,
// values and refinement tests are FP32; libprofit's FP64 cell position is
// formed only for an undecided test and for FP64 leaf values (`fp64`).  The
// descent to a refined cell follows libprofit's FP64 node bounds, so the
// trees are its own.  Every lane returns its share of sum_s weight_s f(s) in
// `sum`; with kJac (the forward walk of a gradient evaluation) every leaf
// also adds its weighted FP32 derivatives to gj (per lane), for the pixel's
// Jacobian.
template <int TYPE, bool kJac>
__device__ __forceinline__ void walk_pixel(const Comp &c, WalkLevel *L, int lane, double x0, double x1, double y0,
                                           double y1, int res, int maxrec, bool fp64, double &sum, float *gj)
{
	// a Sersic Jacobian without box (or box derivative) from the value's
	// own logarithm and exponentials
	const bool fuse = kJac && TYPE == SERSIC && !c.boxy && !c.grad_box;
	const int ncell = res * res;
	const int nchunk = (ncell + 63) >> 6;
	// 1 / res^2 from a table (the quotient a division rounds to)
	const double inv_cells = kInvCells[res];
	int level = 0;
	double nx0 = x0, nx1 = x1, ny0 = y0, ny1 = y1;
	double weight = inv_cells;
	const RefineLimits lim = refine_limits(c);
	for (;;) {
		const bool recurse = res > 1 && level < maxrec;
		const Node n = make_node(c, lim, nx0, nx1, ny0, ny1, res);
		// the cells in chunks of 64 (one per lane); lane 0 stores each chunk's
		// refine mask with the node, and `any` gathers them.  A node with no
		// cell to refine is not stored: the search below starts under it.
		unsigned long long any = 0ull;
#pragma unroll 1
		for (int k = 0; k < nchunk; ++k) {
			const int cell = k * 64 + lane;
			const bool fail = cell < ncell && cell_step<TYPE, kJac>(c, n, cell, recurse, fp64, fuse, weight, sum, gj);
			const unsigned long long mk = __ballot(fail);
			any |= mk;
			if (lane == 0) L[level].mask[k] = mk;
		}
		if (any != 0ull) {
			if (lane == 0) {
				L[level].x0 = nx0;
				L[level].x1 = nx1;
				L[level].y0 = ny0;
				L[level].y1 = ny1;
				L[level].weight = weight;
				for (int k = nchunk; k < 4; ++k) L[level].mask[k] = 0ull;
			}
		}
		else if (level == 0) {
			break;  // a leaf-only root: the tree is done
		}
		__builtin_amdgcn_wave_barrier();
		// next node: lowest pending cell of the deepest level that has one
		int lv = any != 0ull ? level : level - 1;
		int cell = -1;
		for (;;) {
			int found = -1;
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				const unsigned long long mk = L[lv].mask[k];
				if (found < 0 && mk) {
					found = k * 64 + (__ffsll((long long)mk) - 1);
				}
			}
			if (found >= 0) {
				cell = found;
				break;
			}
			if (lv == 0) break;
			--lv;
		}
		if (cell < 0) break;
		__builtin_amdgcn_wave_barrier();
		if (lane == 0) L[lv].mask[cell >> 6] &= ~(1ull << (cell & 63));
		const double px0 = L[lv].x0, px1 = L[lv].x1, py0 = L[lv].y0, py1 = L[lv].y1;
		const double pxbin = (px1 - px0) / res, pybin = (py1 - py0) / res;
		const double phx = pxbin / 2., phy = pybin / 2.;
		const int ci = cell / res, cj = cell - ci * res;
		const double cx = cell_centre(px0, phx, ci);
		const double cy = cell_centre(py0, phy, cj);
		nx0 = cx - phx;
		nx1 = cx + phx;
		ny0 = cy - phy;
		ny1 = cy + phy;
		weight = L[lv].weight * inv_cells;
		level = lv + 1;
		__builtin_amdgcn_wave_barrier();
	}
}

// The trees that k_subsample_tree marked because they overflow its stack, one
// wavefront each, by the mask walk, whose memory is one mask per level: adds
// flux_scale * value to the canvas (or the aux canvas, or the FP64 canvas) and,
// with kJac, writes the entry's Jacobian and value to wq.ljac / hjac for
// k_adj_queue.  Entries are dealt out by index, as there, and the marks taken back.
// Held to the registers of four waves per SIMD (three for the Sersic, Moffat
// and broken-exponential walks with kJac, whose code needs more).
template <int TYPE, bool kJac>
__global__ __launch_bounds__(256, kJac && (TYPE == SERSIC || TYPE == MOFFAT || TYPE == BROKENEXP) ? 3 : 4) void k_subsample_mask(
    const GalaxyDev *__restrict__ gals, const InstDev *__restrict__ insts, const Comp *__restrict__ comps, WorkQueue wq, int split)
{
	__shared__ WalkLevel levels[4][kMaxLevels];
	// the Jacobian's slots of a pixel (with kJac) and its value: per
	// wavefront, one row of 64 lane sums per slot (rows kJacPitch floats
	// apart, so that the 16 lanes reading one quarter of each row fall on
	// distinct banks)
	constexpr int kSlots = G_S0 + n_shape(TYPE), kJacPitch = 68;
	__shared__ __align__(16) float jred[4][(kJac ? kSlots + 1 : 1) * kJacPitch];
	// the wavefront index is uniform: make that visible to the compiler so queue
	// entries and component fields are read through the scalar cache
	const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	WalkLevel *L = levels[wv];
	static_assert(TYPE >= 0 && TYPE < kFamilies, "one walker launch per profile family");
	static_assert(kSlots < kJacStride && kSlots + 1 <= 16, "Jacobian slots and the value");
	const int lb = wq.lbase[TYPE], cap = wq.lbase[TYPE + 1] - lb;
	const int nd = min(wq.count[deep_count(TYPE)], cap), nb = min(wq.count[big_count(TYPE)], cap);
	const int nh = TYPE == SERSIC ? min(wq.count[1], wq.hcap) : 0;
	// per-lane Jacobian sums
	float gj[NGRAD];
#pragma unroll
	for (int s = 0; s < NGRAD; ++s) gj[s] = 0.f;
	for (int t = blockIdx.x * 4 + wv; t < nh + nb + nd; t += gridDim.x * 4) {
		const bool heavy = t < nh;
		int e = t;  // the entry's index in its list (heavy, or the family's light list)
		QEntry q;
		if (heavy) {
			q = wq.heavy[e];
			if (q.pix >= 0) continue;
			q.pix = ~q.pix;
			__builtin_amdgcn_wave_barrier();  // every lane has read the mark
			if (lane == 0) wq.heavy[e].pix = q.pix;
		}
		else {
			e = wq.deep[lb + (t < nh + nb ? cap - 1 - (t - nh) : t - nh - nb)];
			if (e >= 0) continue;
			e = ~e;
			q = wq.light[lb + e];
		}
		{
			const Comp &c = comps[q.comp];
			if (c.type != TYPE) continue;
			const InstDev &I = insts[c.instance];
			const GalaxyDev &g = gals[I.galaxy];
			const int i = q.pix % g.DW, j = q.pix / g.DW;
			const double hx = g.sx / 2., hy = g.sy / 2.;
			const double y = hy + j * g.sx;
			const double x = hx + i * g.sy;
			int res = c.res, maxrec = c.maxrec;
			if (centre_pixel(c, x, y)) {
				res = 8;
				maxrec = 10;
			}
			double s_local = 0;
			walk_pixel<TYPE, kJac>(c, L, lane, x - hx, x + hx, y - hy, y + hy, res, maxrec, g.render_fp64 != 0, s_local,
			                       gj);
			const bool to_aux = split && !c.convolve;
			// on the FP32 canvas the value is summed through the wavefront's
			// LDS rows (as one more row of the Jacobian's), the same way with
			// and without the Jacobian, so that a pixel's value does not depend
			// on whether gradients are asked for; the FP64 canvas sums it in
			// FP64 across the wave
			const bool fold = !g.canvas64;
			double tot = 0.0;
			if (!fold) {
				tot = wave_sum(s_local);
				if (lane == 0) {
					if (!to_aux) atomicAdd(&I.canvas64[q.pix], c.flux_scale * tot);
					else atomicAdd(&I.aux[q.pix], (float)(c.flux_scale * tot));
				}
			}
			if (kJac || fold) {
				// the lane sums go to the wavefront's rows (the Jacobian's
				// slots, then the value); lane l adds quarter l >> 4 of row
				// l & 15 in FP64 and two exchanges add the quarters
				constexpr int kRows = kJac ? kSlots : 0;  // the value's row
				float *R = jred[wv];
#pragma unroll
				for (int s = 0; s < kRows; ++s) {
					R[s * kJacPitch + lane] = gj[s];
					gj[s] = 0.f;
				}
				if (fold) R[kRows * kJacPitch + lane] = (float)s_local;
				__builtin_amdgcn_wave_barrier();
				const int slot = lane & 15, qt = lane >> 4;
				double t = 0.0;
				if (slot < kRows + (fold ? 1 : 0)) {
					const float4 *row = reinterpret_cast<const float4 *>(R + slot * kJacPitch + qt * 16);
#pragma unroll
					for (int k = 0; k < 4; ++k) {
						const float4 v = row[k];
						t += ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
					}
				}
				__builtin_amdgcn_wave_barrier();
				t += __shfl_xor(t, 16);
				t += __shfl_xor(t, 32);
				float *J = nullptr;
				if (kJac) {
					J = (heavy ? wq.hjac : wq.ljac + (long)lb * kJacStride) + (long)e * kJacStride;
					if (lane < kSlots) J[lane] = (float)t;
					if (!fold && lane == 0) J[kJacStride - 1] = (float)tot;
				}
				if (fold && lane == kRows) {
					if (kJac) J[kJacStride - 1] = (float)t;
					atomicAdd(&(to_aux ? I.aux : I.canvas)[q.pix], (float)(c.flux_scale * t));
				}
			}
		}
	}
}

// The root pass of the sub-sampled pixels, one group of 2^k lanes per light
// entry of a TYPE family: the lanes share the pixel's root cells, and when none
// is to be refined (most pixels: 98% on a 400x400 bulge+disk) the group adds
// the value to the canvas and, with kJac, writes the entry's Jacobian and
// value.  An entry with a cell to refine goes to the family's deep list: to its
// front, or, from kBigTree refined cells or 64 cells a node on, to its back;
// k_subsample_tree walks those trees from the root, the front's
// with a wavefront each.
//
// Bound by VALU issue on long lists and by latency on short ones, so the group
// is as wide as the list leaves room for in kRootLanes lanes: one lane per entry
// from 524,289 entries (no exchange, 0.53 ms for the 1.3 M of a batch of 1024
// bulge+disk images), a whole wavefront up to 16,384.  At 2^18 lanes the families
// of 384 survey galaxies took 172 to 752 us, at 2^20 91 to 521; at 2^21 the 300 k
// entries of 256 likelihoods 127 us (110, 107).  Entries are dealt out by index:
// asking a counter cost 11.6 ns per wavefront (95 us for 8,192 of them, also with
// nothing to do).
constexpr int kRootLanes = 1 << 20;
constexpr int kBigTree = 8;

template <int TYPE, bool kJac>
__global__ __launch_bounds__(256) void k_subsample_root(const GalaxyDev *__restrict__ gals,
                                                         const InstDev *__restrict__ insts,
                                                         const Comp *__restrict__ comps, WorkQueue wq, int split)
{
	constexpr int kSlots = G_S0 + n_shape(TYPE);
	const int lane = threadIdx.x & 63;
	const int lb = wq.lbase[TYPE], cap = wq.lbase[TYPE + 1] - lb;
	const int nl = min(wq.count[light_count(TYPE)], cap);
	int lg = 0;
	while (lg < 6 && ((long)nl << (lg + 1)) <= kRootLanes) ++lg;
	const int grp = 1 << lg, sub = lane & (grp - 1);
	const long gtid = (long)blockIdx.x * blockDim.x + threadIdx.x, sweep = (long)gridDim.x * blockDim.x;
	// the loop's bound is the wavefront's first entry: uniform
	for (long t = gtid; ((t - lane) >> lg) < nl; t += sweep) {
		const int e = (int)min(t >> lg, (long)nl);
		int nref = 0;
		double sum = 0;
		float gj[NGRAD];
#pragma unroll
		for (int s = 0; s < NGRAD; ++s) gj[s] = 0.f;
		QEntry q{-1, 0};
		bool mine = false, wide = false;
		if (e < nl) {
			q = wq.light[lb + e];
			const Comp &c = comps[q.comp];
			const GalaxyDev &g = gals[insts[c.instance].galaxy];
			const int i = q.pix % g.DW, j = q.pix / g.DW;
			const double hx = g.sx / 2., hy = g.sy / 2.;
			const double y = hy + j * g.sx;
			const double x = hx + i * g.sy;
			mine = c.type == TYPE;
			// centre-rule pixels belong to the heavy list: any found here go
			// to the tree walk, which applies the rule
			if (mine && centre_pixel(c, x, y)) nref = kBigTree;
			else if (mine) {
				const int res = c.res, ncell = res * res;
				wide = ncell > 64;
				const bool recurse = res > 1 && c.maxrec > 0;
				const bool fuse = kJac && TYPE == SERSIC && !c.boxy && !c.grad_box;
				const Node n = make_node(c, refine_limits(c), x - hx, x + hx, y - hy, y + hy, res);
				const double weight = kInvCells[res];
				const bool fp64 = g.render_fp64 != 0;
				for (int cell = sub; cell < ncell; cell += grp)
					nref += cell_step<TYPE, kJac>(c, n, cell, recurse, fp64, fuse, weight, sum, gj) ? 1 : 0;
			}
		}
		double gd[kSlots];
		if (kJac) {
#pragma unroll
			for (int s = 0; s < kSlots; ++s) gd[s] = (double)gj[s];
		}
		for (int o = grp >> 1; o > 0; o >>= 1) {
			nref += __shfl_xor(nref, o);
			sum += __shfl_xor(sum, o);
			if (kJac) {
#pragma unroll
				for (int s = 0; s < kSlots; ++s) gd[s] += __shfl_xor(gd[s], o);
			}
		}
		const bool lead = mine && sub == 0;
		if (lead && nref == 0) {
			const Comp &c = comps[q.comp];
			const InstDev &I = insts[c.instance];
			const bool to_aux = split && !c.convolve;
			if (gals[I.galaxy].canvas64 && !to_aux) atomicAdd(&I.canvas64[q.pix], c.flux_scale * sum);
			else atomicAdd(&(to_aux ? I.aux : I.canvas)[q.pix], (float)(c.flux_scale * sum));
			if (kJac) {
				float *J = wq.ljac + (long)(lb + e) * kJacStride;
#pragma unroll
				for (int s = 0; s < kSlots; ++s) J[s] = (float)gd[s];
				J[kJacStride - 1] = (float)sum;
			}
		}
		// the deep entries appended, one atomic per wavefront and list
		const bool big = lead && nref > 0 && (wide || nref >= kBigTree), deep = lead && nref > 0 && !big;
#pragma unroll
		for (int k = 0; k < 2; ++k) {
			const unsigned long long m = __ballot(k ? big : deep);
			if (!m) continue;
			const int leader = __ffsll((long long)m) - 1;
			int at = 0;
			if (lane == leader) at = atomicAdd(&wq.count[k ? big_count(TYPE) : deep_count(TYPE)], __popcll(m));
			at = __shfl(at, leader) + __popcll(m & ((1ull << lane) - 1ull));
			if (k ? big : deep) wq.deep[lb + (k ? cap - 1 - at : at)] = e;
		}
	}
}

// ------------------------------------------------------------------ trees

// The pending nodes of the trees a block of W wavefronts walks, in LDS:
// wavefront w's share holds kTreeShare of them (its own stack while each
// wavefront walks a tree of its own; a part of the block's while the block
// walks one together).
constexpr int kTreeShare = 256;
template <int W>
struct TreeStack {
	struct Share {
		double x0[kTreeShare], x1[kTreeShare], y0[kTreeShare], y1[kTreeShare], weight[kTreeShare];
		uint8_t level[kTreeShare];
	} q[W];
	int count[2][W];  // refined cells per wavefront of a round, double-buffered
};

// Walks the recursion tree of one pixel of a TYPE profile with T threads (a
// wavefront, T = 64, or the block of W wavefronts, T = 64 W), starting from
// stack slot `base` (T = 64: the wavefront's share).  A round takes as many pending
// nodes off the stack as T threads have cells for, one cell per thread (a node
// of more cells alone, its cells T at a time); a cell to be refined pushes its
// own FP64 node bounds (libprofit's additions).  Every thread returns its share
// of sum_s weight_s f(s) in `sum` and, with kJac, of the weighted FP32
// derivatives in gj.  Returns false when the stack (cap nodes) would overflow:
// the sums are then void.
//
// `top`, `n` and `total` are equal on all T threads, so all take the same
// barriers; each round removes a node and a node's children lie one level
// deeper (at most maxrec), so the rounds end.
template <int TYPE, bool kJac, int T, int W>
__device__ __forceinline__ bool walk_tree(const Comp &c, TreeStack<W> &S, int base, int tid, double x0, double x1,
                                          double y0, double y1, int res, int maxrec, bool fp64, double &sum, float *gj)
{
	static_assert(T == 64 || T == 64 * W, "a wavefront or the block");
	constexpr int cap = (T / 64) * kTreeShare;
	const bool fuse = kJac && TYPE == SERSIC && !c.boxy && !c.grad_box;
	const int ncell = res * res, wv = tid >> 6, lane = tid & 63;
	const double inv_cells = kInvCells[res];
	const RefineLimits lim = refine_limits(c);
	// the thread's node of a round and its first cell
	const int per = ncell >= T ? 1 : T / ncell;
	const int slot = ncell >= T ? 0 : tid / ncell;
	const int cell0 = tid - slot * ncell;
	auto put = [&](int at, double a, double b, double d, double e, double w, int level) {
		typename TreeStack<W>::Share &q = S.q[(base + at) / kTreeShare];
		const int k = (base + at) % kTreeShare;
		q.x0[k] = a;
		q.x1[k] = b;
		q.y0[k] = d;
		q.y1[k] = e;
		q.weight[k] = w;
		q.level[k] = (uint8_t)level;
	};
	auto sync = [&]() {
		if constexpr (T == 64) {
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
		}
		else {
			__syncthreads();
		}
	};
	if (tid == 0) put(0, x0, x1, y0, y1, inv_cells, 0);
	sync();
	int top = 1, buf = 0;
	while (top > 0) {
		const int n = min(per, top);
		const bool on = slot < n;
		const int r = base + top - 1 - (on ? slot : 0);
		const typename TreeStack<W>::Share &Q = S.q[r / kTreeShare];
		const int k = r % kTreeShare;
		const Node node = make_node(c, lim, Q.x0[k], Q.x1[k], Q.y0[k], Q.y1[k], res);
		const double weight = Q.weight[k];
		const int level = Q.level[k];
		const bool recurse = res > 1 && level < maxrec;
		top -= n;
		bool pushed = false;
		for (int at = 0; at < ncell; at += T) {
			const int cell = cell0 + at;
			const bool fail = on && cell < ncell && cell_step<TYPE, kJac>(c, node, cell, recurse, fp64, fuse, weight, sum, gj);
			const unsigned long long m = __ballot(fail);
			int off = __popcll(m & ((1ull << lane) - 1ull)), total = __popcll(m);
			if constexpr (T > 64) {
				// every thread has read its node before a push may overwrite it
				if (lane == 0) S.count[buf][wv] = total;
				__syncthreads();
				total = 0;
				for (int w = 0; w < W; ++w) {
					const int v = S.count[buf][w];
					off += w < wv ? v : 0;
					total += v;
				}
				buf ^= 1;
			}
			if (total == 0) continue;
			if (top + total > cap) return false;
			if (fail) {
				const double hx = (node.x1 - node.x0) / res / 2., hy = (node.y1 - node.y0) / res / 2.;
				const int ci = (int)(((float)cell + 0.5f) * node.inv_res), cj = cell - ci * res;
				const double cx = cell_centre(node.x0, hx, ci), cy = cell_centre(node.y0, hy, cj);
				put(top + off, cx - hx, cx + hx, cy - hy, cy + hy, weight * inv_cells, level + 1);
			}
			top += total;
			pushed = true;
		}
		if (pushed) sync();
	}
	return true;
}

// The trees of a TYPE family: the centre pixels (heavy list, Sersic) and the
// entries with kBigTree or more refined root cells or more than 64 cells a node
// (the back of the deep list), a block each; then the other deep entries, a wavefront each.  Adds flux_scale
// * value to the canvas (or the aux canvas, or the FP64 canvas) and, with kJac,
// writes the entry's Jacobian and value.  A block takes its first big tree by index and
// the next ones from a counter, asked for while it walks (the trees differ by a factor
// of hundreds: King trees of 4,096 survey galaxies 5.7 ms by index, 4.4 so, core-Sersic
// 3.1 and 2.0); small trees are dealt out by index.  An overflowing tree is counted in count[0] and, with `mark`, its entry is marked for
// the mask walk that follows (k_subsample_mask): the pixel of a heavy entry, the index
// of a deep one, bitwise inverted.  Without it the evaluation has to be run again.
//
// A centre tree (res 8, depth 10: 160 nodes, 16 a level) is a chain of levels:
// one wavefront walking its nodes in turn took 220 to 300 us, whatever the
// batch; a core-Sersic pixel of resolution 16 is a chain of 300 nodes of 256
// cells.  W = 4 wavefronts share a tree (three blocks a CU) where there are trees
// for all blocks, W = 12 (one block a CU, the same registers) where there are
// not.
template <int TYPE, bool kJac, int W>
__global__ __launch_bounds__(64 * W, 3) void k_subsample_tree(const GalaxyDev *__restrict__ gals,
                                                           const InstDev *__restrict__ insts,
                                                           const Comp *__restrict__ comps, WorkQueue wq, int split,
                                                           int mark)
{
	constexpr int kSlots = G_S0 + n_shape(TYPE), kJacPitch = 68;
	__shared__ __align__(16) TreeStack<W> S;
	__shared__ double red[W][16];
	__shared__ int next;
	static_assert(kSlots < kJacStride && kSlots + 1 <= 16, "Jacobian slots and the value");
	static_assert(sizeof(float) * kSlots * kJacPitch <= sizeof(typename TreeStack<W>::Share), "a wavefront's rows fit its share");
	static_assert(sizeof(typename TreeStack<W>::Share) % 16 == 0, "a wavefront's rows are 16-byte aligned");
	const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int lb = wq.lbase[TYPE], cap = wq.lbase[TYPE + 1] - lb;
	const int nd = min(wq.count[deep_count(TYPE)], cap), nb = min(wq.count[big_count(TYPE)], cap);
	const int nh = TYPE == SERSIC ? min(wq.count[1], wq.hcap) : 0;
	float gj[NGRAD];
	double sum;
	// the thread's sums of its wavefront: lane s < kSlots of the wavefront
	// returns slot s, lane 15 the value (the wavefront's share as scratch:
	// the walk is over)
	auto wave_totals = [&]() {
		float *R = reinterpret_cast<float *>(&S.q[wv]);
		const double v = wave_sum(sum);
		double t = 0.0;
		if constexpr (kJac) {
#pragma unroll
			for (int s = 0; s < kSlots; ++s) R[s * kJacPitch + lane] = gj[s];
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
			const int slot = lane & 15, qt = lane >> 4;
			if (slot < kSlots) {
				const float4 *row = reinterpret_cast<const float4 *>(R + slot * kJacPitch + qt * 16);
#pragma unroll
				for (int k = 0; k < 4; ++k) {
					const float4 w = row[k];
					t += ((double)w.x + (double)w.y) + ((double)w.z + (double)w.w);
				}
			}
			t += __shfl_xor(t, 16);
			t += __shfl_xor(t, 32);
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
		}
		return lane == 15 ? v : t;
	};
	auto finish = [&](const QEntry &q, const Comp &c, const InstDev &I, const GalaxyDev &g, bool heavy, int e, double t) {
		if (kJac) {
			float *J = (heavy ? wq.hjac : wq.ljac + (long)lb * kJacStride) + (long)e * kJacStride;
			if (lane < kSlots) J[lane] = (float)t;
			if (lane == 15) J[kJacStride - 1] = (float)t;
		}
		if (lane == 15) {
			const bool to_aux = split && !c.convolve;
			if (g.canvas64 && !to_aux) atomicAdd(&I.canvas64[q.pix], c.flux_scale * t);
			else atomicAdd(&(to_aux ? I.aux : I.canvas)[q.pix], (float)(c.flux_scale * t));
		}
	};
	auto clear = [&]() {
		sum = 0;
#pragma unroll
		for (int s = 0; s < NGRAD; ++s) gj[s] = 0.f;
	};
	for (int t = blockIdx.x; t < nh + nb;) {
		if (threadIdx.x == 0) next = gridDim.x + atomicAdd(&wq.count[tree_count(TYPE)], 1);
		const bool heavy = t < nh;
		const int e = heavy ? t : wq.deep[lb + cap - 1 - (t - nh)];
		const QEntry q = heavy ? wq.heavy[e] : wq.light[lb + e];
		const Comp &c = comps[q.comp];
		const InstDev &I = insts[c.instance];
		const GalaxyDev &g = gals[I.galaxy];
		const int i = q.pix % g.DW, j = q.pix / g.DW;
		const double hx = g.sx / 2., hy = g.sy / 2.;
		const double y = hy + j * g.sx, x = hx + i * g.sy;
		const bool centre = centre_pixel(c, x, y);
		clear();
		const bool ok = walk_tree<TYPE, kJac, 64 * W>(c, S, 0, threadIdx.x, x - hx, x + hx, y - hy, y + hy,
		                                           centre ? 8 : c.res, centre ? 10 : c.maxrec, g.render_fp64 != 0, sum, gj);
		if (ok) {
			const double w = wave_totals();
			if (lane < 16) red[wv][lane] = w;
		}
		else if (threadIdx.x == 0) {
			atomicAdd(&wq.count[0], 1);
			if (mark && heavy) wq.heavy[e].pix = ~q.pix;
			else if (mark) wq.deep[lb + cap - 1 - (t - nh)] = ~e;
		}
		__syncthreads();
		const int then = next;
		if (ok && wv == 0) {
			double v = 0;
#pragma unroll
			for (int w = 0; w < W; ++w) v += red[w][lane & 15];
			finish(q, c, I, g, heavy, e, v);
		}
		__syncthreads();
		t = then;
	}
	for (int t = blockIdx.x * W + wv; t < nd; t += gridDim.x * W) {
		const int e = wq.deep[lb + t];
		const QEntry q = wq.light[lb + e];
		const Comp &c = comps[q.comp];
		const InstDev &I = insts[c.instance];
		const GalaxyDev &g = gals[I.galaxy];
		const int i = q.pix % g.DW, j = q.pix / g.DW;
		const double hx = g.sx / 2., hy = g.sy / 2.;
		const double y = hy + j * g.sx, x = hx + i * g.sy;
		clear();
		if (walk_tree<TYPE, kJac, 64>(c, S, wv * kTreeShare, lane, x - hx, x + hx, y - hy, y + hy, c.res, c.maxrec,
		                              g.render_fp64 != 0, sum, gj))
			finish(q, c, I, g, false, e, wave_totals());
		else if (lane == 0) {
			atomicAdd(&wq.count[0], 1);
			if (mark) wq.deep[lb + t] = ~e;
		}
	}
}

// The adjoint of the sub-sampled pixels from their Jacobians (written by the
// forward walk's three kernels with kJac): per entry (component c,
// pixel q), G(q) fs (J_s + dlnfs_s V) for every slot s.  Lanes take
// consecutive entries of the family's lists (the heavy list first, Sersic
// only); the lanes of one component are summed across the wave, one
// component at a time, in FP64, and added with one atomic per slot.
template <int TYPE>
__global__ __launch_bounds__(256) void k_adj_queue(const InstDev *__restrict__ insts, const Comp *__restrict__ comps,
                                                   WorkQueue wq, double *grad_acc)
{
	constexpr int kSlots = G_S0 + n_shape(TYPE);
	const int lane = threadIdx.x & 63;
	const int lb = wq.lbase[TYPE];
	const long nl = min(wq.count[light_count(TYPE)], wq.lbase[TYPE + 1] - lb);
	const long nh = TYPE == SERSIC ? min(wq.count[1], wq.hcap) : 0;
	const long total = nl + nh;
	const long stride = (long)gridDim.x * blockDim.x;
	for (long base = (long)blockIdx.x * blockDim.x + (threadIdx.x & ~63); base < total; base += stride) {
		const long e = base + lane;
		int comp = -1;
		double cs[kSlots];
#pragma unroll
		for (int s = 0; s < kSlots; ++s) cs[s] = 0;
		if (e < total) {
			const bool heavy = e < nh;
			const long ei = heavy ? e : e - nh;
			const QEntry q = heavy ? wq.heavy[ei] : wq.light[lb + ei];
			const float *J = heavy ? wq.hjac + ei * kJacStride : wq.ljac + (lb + ei) * kJacStride;
			const Comp &c = comps[q.comp];
			const float G = insts[c.instance].G[q.pix];
			if (c.type == TYPE && G != 0.f) {
				comp = q.comp;
				const double gw = (double)G * c.flux_scale, V = (double)J[kJacStride - 1];
#pragma unroll
				for (int s = 0; s < kSlots; ++s) cs[s] = gw * ((double)J[s] + c.dlnfs[s] * V);
			}
		}
		unsigned long long left = __ballot(comp >= 0);
		while (left) {
			const int leader = __ffsll((long long)left) - 1;
			const int lc = __builtin_amdgcn_readlane(comp, leader);
			const bool mine = comp == lc;
			left &= ~__ballot(mine);
#pragma unroll
			for (int s = 0; s < kSlots; ++s) {
				const double t = wave_sum(mine ? cs[s] : 0.0);
				if (lane == leader && t != 0) atomicAdd(&grad_acc[(long)lc * NGRAD + s], t);
			}
		}
	}
}

// ------------------------------------------------------------------ adjoint render

// Adjoint of the directly evaluated pixels: sum_q G(q) fs d f(q) / d slot over
// the pixels the forward render marked direct (so no classification is
// repeated), FP32 per-pixel derivatives, per-thread sums in FP32 (in FP64 for
// steep cores, G64: their centroid and shape terms cancel over many pixels,
// which FP32 sums do not survive), the flux-scale term applied once per
// component from sum_q G(q) fs f(q).  A block takes `grp` consecutive canvas
// tiles of one instance (block offsets per instance in grp_off), so that the
// per-component reduction and its atomics are paid once per grp tiles, or one
// of `parts` parts of a tile (grp = 1).  Components that do nothing on the
// block's tiles are left out through a bit mask the block forms first.
// Compiled per profile family TYPE and G64; components of other kinds are
// left to the launch made for them.
template <int TYPE, bool G64>
__global__ __launch_bounds__(256) void k_adj_render(const GalaxyDev *__restrict__ gals,
                                                    const InstDev *__restrict__ insts,
                                                    const int *__restrict__ grp_off, int ninst, int grp, int parts,
                                                    const Comp *__restrict__ comps, double *grad_acc)
{
	constexpr int kAdjRows = 4;  // rows whose masks and G a thread loads together
	__shared__ double red[4][NGRAD];
	__shared__ unsigned long long hit[kCullWords];
	const int b = blockIdx.x / parts, part = blockIdx.x - b * parts;
	const int inst = owner_of(grp_off, ninst, b);
	const InstDev I = insts[inst];
	const GalaxyDev &g = gals[I.galaxy];
	const int rows = g.conv_rows / parts;  // rows per thread
	const int t0 = (b - grp_off[inst]) * grp, t1 = min(t0 + grp, g.n_atiles);
	const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int wpr = (g.DW + 63) >> 6;
	const int nwords = (I.ncomp + 63) >> 6;
	for (int w = wv; w < min(nwords, kCullWords); w += 4) {
		const int k = w * 64 + lane;
		bool on = false;
		if (k < I.ncomp) {
			const Comp &c = comps[I.comp0 + k];
			if (c.type == TYPE && (bool)c.grad64 == G64)
				for (int ti = t0; ti < t1 && !on; ++ti) on = tile_class(c, tile_rect(g, g.atiles[ti], g.conv_rows)) != 0;
		}
		const unsigned long long m = __ballot(on);
		if (lane == 0) hit[w] = m;
	}
	__syncthreads();
	const double hx = g.sx / 2., hy = g.sy / 2.;
	// G at column i of rows j .. j + kAdjRows - 1 (n of them this thread's), 0
	// where component k did not draw the pixel directly: the loads of all rows
	// are in flight together
	auto load_rows = [&](int k, int tx, int i, int j, int n, float *Gr) {
		unsigned long long m[kAdjRows];
#pragma unroll
		for (int u = 0; u < kAdjRows; ++u) {
			const bool ok = u < n && j + u < g.DH;
			m[u] = ok ? I.dmask[((long)k * g.DH + j + u) * wpr + tx] : 0ull;
			Gr[u] = ok && i < g.DW ? I.G[i + (j + u) * g.DW] : 0.f;
		}
#pragma unroll
		for (int u = 0; u < kAdjRows; ++u) Gr[u] = (m[u] >> lane) & 1ull ? Gr[u] : 0.f;
	};
	for (int w = 0; w < nwords; ++w) {
	  for (unsigned long long left = w < kCullWords ? uniform64(hit[w]) : ~0ull; left; left &= left - 1ull) {
		const int k = w * 64 + __ffsll((long long)left) - 1;
		if (k >= I.ncomp) break;
		const Comp &c = comps[I.comp0 + k];
		if (c.type != TYPE || (bool)c.grad64 != G64) continue;
		double gl[NGRAD];
#pragma unroll
		for (int s = 0; s < NGRAD; ++s) gl[s] = 0;
		double vsum = 0;
		if (G64) {
			for (int ti = t0; ti < t1; ++ti) {
				const int2 t = g.atiles[ti];
				if (tile_class(c, tile_rect(g, t, g.conv_rows)) == 0) continue;
				const int i = t.x * kTileW + lane;
				const int j0 = t.y * 4 * g.conv_rows + (part * 4 + wv) * rows;
				const double x = hx + i * g.sy;
				for (int r0 = 0; r0 < rows; r0 += kAdjRows) {
				  float Gr[kAdjRows];
				  load_rows(k, t.x, i, j0 + r0, rows - r0, Gr);
#pragma unroll
				  for (int u = 0; u < kAdjRows; ++u) {
					const float Gq = Gr[u];
					if (Gq == 0.f) continue;
					const double y = hy + (j0 + r0 + u) * g.sx;
					const double xr = x - c.xc, yr = y - c.yc;
					const double xp = xr * c.cos_ang + yr * c.sin_ang;
					const double yp = -xr * c.sin_over + yr * c.cos_over;
					const double wq = (double)Gq * c.flux_scale;
					const double v = TYPE == SERSIC && !c.boxy ? sersic_accumulate(c, xp, yp, wq, gl)
					                                           : sample_accumulate<float, TYPE>(c, xp, yp, wq, gl);
					vsum = fma(wq, v, vsum);
				  }
				}
			}
		}
		else {
			float gf[NGRAD];
#pragma unroll
			for (int s = 0; s < NGRAD; ++s) gf[s] = 0.f;
			float vf = 0.f;
			const float fs = (float)c.flux_scale;
			// a Sersic without box (or box derivative): the derivatives from
			// the value's own logarithm and exponentials
			const bool fuse = TYPE == SERSIC && !c.boxy && !c.grad_box;
			for (int ti = t0; ti < t1; ++ti) {
				const int2 t = g.atiles[ti];
				if (tile_class(c, tile_rect(g, t, g.conv_rows)) == 0) continue;
				const int i = t.x * kTileW + lane;
				const int j0 = t.y * 4 * g.conv_rows + (part * 4 + wv) * rows;
				const double x = hx + i * g.sy;
				const float xr = (float)(x - c.xc);
				for (int r0 = 0; r0 < rows; r0 += kAdjRows) {
				  float Gr[kAdjRows];
				  load_rows(k, t.x, i, j0 + r0, rows - r0, Gr);
#pragma unroll
				  for (int u = 0; u < kAdjRows; ++u) {
					const float Gq = Gr[u];
					if (Gq == 0.f) continue;
					const double y = hy + (j0 + r0 + u) * g.sx;
					const float yr = (float)(y - c.yc);
					const float xp = xr * c.f.cos_ang + yr * c.f.sin_ang;
					const float yp = -xr * c.f.sin_over + yr * c.f.cos_over;
					const float wq = Gq * fs;
					if (fuse) {
						float base, l2, rf;
						const float v = sersic_parts_f32(c, xp, yp, base, l2, rf);
						sersic_jac_f32(c, xp, yp, v, base, l2, rf, wq, gf);
						vf += wq * v;
					}
					else {
						vf += wq * pixel_accumulate_f32<TYPE>(c, xp, yp, wq, gf);
					}
				  }
				}
			}
#pragma unroll
			for (int s = 0; s < NGRAD; ++s) gl[s] = (double)gf[s];
			vsum = (double)vf;
		}
		// flux-scale dependence: d fs / d slot = fs * dlnfs
#pragma unroll
		for (int s = 0; s < G_S0 + n_shape(TYPE); ++s) {
			const double v = wave_sum(gl[s] + vsum * c.dlnfs[s]);
			if (lane == 0) red[wv][s] = v;
		}
		__syncthreads();
		if (threadIdx.x < G_S0 + n_shape(TYPE)) {
			const int s = threadIdx.x;
			const double v = (red[0][s] + red[1][s]) + (red[2][s] + red[3][s]);
			if (v != 0) atomicAdd(&grad_acc[(long)(I.comp0 + k) * NGRAD + s], v);
		}
		__syncthreads();
	  }
	}
}

}  // namespace profit_amd
