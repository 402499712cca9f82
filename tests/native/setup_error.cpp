// Set-ups that fail must leave a component that draws nothing, with no field of
// the memory it was formed in.  Prints "ok <error>" per invalid parameter.
#include <hip/hip_runtime.h>

#include <cstdio>

using std::max;
using std::min;

#include "profile_math.h"

using namespace profit_amd;

int main()
{
	struct Case {
		int type;
		void (*spoil)(ProfileParams &);
		int error;
	};
	const Case cases[] = {
	    {SERSIC, [](ProfileParams &p) { p.axrat = 0; }, SE_AXRAT_LE0},
	    {SERSIC, [](ProfileParams &p) { p.shape[0] = -1; }, SE_RE},
	    {MOFFAT, [](ProfileParams &p) { p.axrat = 1.5; }, SE_AXRAT_GT1},
	    {FERRER, [](ProfileParams &p) { p.shape[2] = 3; }, SE_FB},
	    {KING, [](ProfileParams &p) { p.adjust = 0; p.resolution = 100; }, SE_RESOLUTION},
	    {BROKENEXP, [](ProfileParams &p) { p.adjust = 0; p.resolution = 0; }, SE_RESOLUTION},
	    {SERSIC, [](ProfileParams &p) { p.max_recursions = 31; }, SE_MAXREC},
	    {CORESERSIC, [](ProfileParams &p) { p.max_recursions = 4000000000u; }, SE_MAXREC},
	    {55, [](ProfileParams &) {}, SE_TYPE},
	};
	bool ok = true;
	for (const Case &k : cases) {
		ProfileParams p;
		default_params(k.type, &p);
		k.spoil(p);
		Comp c, want;
		std::memset(&c, 0x7f, sizeof(c));
		std::memset(&want, 0, sizeof(want));
		want.type = NULLPROF;
		want.has_rmax = 1;
		want.rmax_r = -1;
		want.f.rmax2 = -1.f;
		sf::QuadState qs;
		const int e = setup_component(p, 0, 1, 1, 1, 1, 0, 0, &qs, &c);
		const bool good = e == k.error && c.type == want.type && c.res == 0 && c.maxrec == 0 && c.has_rmax == 1 && c.rmax_r == -1 &&
		                  c.f.rmax2 == -1.f && c.flux_scale == 0 && c.f.rsw2 == 0 && c.rough == 0 && c.acc == 0 && c.xc == 0 && c.f.cos_ang == 0;
		std::printf("%s %d\n", good ? "ok" : "FAIL", e);
		ok &= good;
	}
	return !ok;
}
