// ssx_ax_f64.hip -- element operator instantiations, fields double,
// geometric factors double (template in ssx_ax.h).
#include "ssx_ax.h"

extern "C" int ssxk_ax_dispatch_f64(void *stream, int n, int v, int nel,
		int op, const void *u, void *au, const void *gf, const void *mass,
		const void *dmat, double lambda, const int *bc, int apply_mask,
		const int *done, double *part, const void *pu)
{
	if (nel <= 0)
		return SSX_OK;
	return ax_dispatch<double, double>((hipStream_t) stream, n, v, nel, op, u, au,
			gf, mass, dmat, lambda, bc, apply_mask, done, part,
			(const PUpd *) pu);
}

// 1 where launch_ax_v takes the matrix kernel for these sizes
extern "C" int ssxk_ax_matrix(int n, int nel)
{
	switch (n) {
	case 9: return axm_use<9>(nel);
	case 10: return axm_use<10>(nel);
	case 11: return axm_use<11>(nel);
	case 12: return axm_use<12>(nel);
	default: return 0;
	}
}

// The Poisson operator by the team kernel at n = 9..12, whatever the number
// of elements: the batched operator is that kernel at every size, so its
// shape is ranked by this one's time.
extern "C" int ssxk_ax_team(void *stream, int n, int v, int nel,
		const double *u, double *au, const double *gf, const double *mass,
		const double *dmat, double lambda, const int *bc, double *part)
{
	const PUpd pu = { nullptr, nullptr, nullptr, 0, -1, nullptr, 0,
		ssx_replay{} };
	if (nel <= 0)
		return SSX_OK;
	switch (n * SSX_AX_NVARIANTS + v) {
#define CASEV(NN, VV) case NN * SSX_AX_NVARIANTS + VV: \
		launch_ax1<NN, double, double, 0, VV>((hipStream_t) stream, nel, \
				SSX_OP_POISSON, u, au, gf, mass, dmat, lambda, bc, 1, \
				nullptr, part, pu); break;
#define CASE(NN) CASEV(NN, 0) CASEV(NN, 1) CASEV(NN, 2) CASEV(NN, 3) \
		CASEV(NN, 4) CASEV(NN, 5) CASEV(NN, 6) CASEV(NN, 7)
	CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
#undef CASEV
	default:
		ssx_set_error("ssxk_ax_team: n=%d variant %d unsupported", n, v);
		return SSX_EINVAL;
	}
	hipError_t e = hipGetLastError();
	if (e != hipSuccess) {
		ssx_set_error("k_ax: %s", hipGetErrorString(e));
		return SSX_EHIP;
	}
	return SSX_OK;
}
