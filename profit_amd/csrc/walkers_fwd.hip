// Forward recursion walk (libprofit's subsample_pixel, radial.cpp:54-134): a
// root pass, the tree walk and (for trees that overflow it) the mask walk, one
// kernel each per radial profile family; see kernel_common.h.
#include "kernel_common.h"

namespace profit_amd {

// The root pass over the light entries, then the tree walk over the heavy list
// and the entries the root pass left to it (mask: then the mask walk over the
// trees that overflowed it).  `few`: the family's big trees (four centre pixels a
// component, or the like) do not fill the GPU, so the tree walk takes blocks of
// twelve wavefronts, one a CU, and otherwise blocks of four, three a CU (one
// bulge+disk image: 53 us with four, 30 with twelve; both shapes by family and
// count: Engine::sync_aux_flags).
template <int TYPE, bool kJac>
static int fwd_launch(int nblocks, const GalaxyDev *gals, const InstDev *insts, const Comp *comps, WorkQueue wq,
                      int split, bool mask, bool few, hipStream_t st)
{
	k_subsample_root<TYPE, kJac><<<nblocks, 256, 0, st>>>(gals, insts, comps, wq, split);
	if (few) k_subsample_tree<TYPE, kJac, 12><<<(nblocks + 7) / 8, 768, 0, st>>>(gals, insts, comps, wq, split, mask);
	else k_subsample_tree<TYPE, kJac, 4><<<(nblocks * 3 + 7) / 8, 256, 0, st>>>(gals, insts, comps, wq, split, mask);
	if (mask) k_subsample_mask<TYPE, kJac><<<nblocks, 256, 0, st>>>(gals, insts, comps, wq, split);
	return (int)hipGetLastError();
}

int launch_subsample_fwd(int type, int nblocks, const GalaxyDev *gals, const InstDev *insts, const Comp *comps,
                         WorkQueue wq, int split, bool jac, bool mask, bool few, hipStream_t st)
{
	if (nblocks <= 0) return 0;
#define PA_FWD(T)                                                                                        \
	case T:                                                                                              \
		return jac ? fwd_launch<T, true>(nblocks, gals, insts, comps, wq, split, mask, few, st)               \
		           : fwd_launch<T, false>(nblocks, gals, insts, comps, wq, split, mask, few, st)
	switch (type) {
		PA_FWD(SERSIC);
		PA_FWD(MOFFAT);
		PA_FWD(FERRER);
		PA_FWD(KING);
		PA_FWD(CORESERSIC);
		PA_FWD(BROKENEXP);
	default: return (int)hipErrorInvalidValue;
	}
#undef PA_FWD
}

}  // namespace profit_amd
