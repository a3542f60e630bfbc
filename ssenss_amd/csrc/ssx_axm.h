// ssx_axm.h -- the FP64 element operator for 9 to 12 points per direction
// (discrete_laplace_operator, poisson.c:34-56; discrete_helmholtz_operator,
// helmholtz.c:33-49) with its contractions on the FP64 matrix instruction.
//
// One element per workgroup, one wavefront a tile of 16 lines, W = ceil(N^2 /
// 16) of them.  The six derivative products D u and D^T t (three directions,
// forward and transposed) are 16x16x4 matrix instructions with D in
// registers: a line's values are read from LDS once per direction instead of
// N times, and a lane holds neither a column of the element nor rows of D.
//
//   load     u (or the fused direction update) into LDS, every global load
//            and all six factors of the lane's nodes issued first
//   forward  D_xi u and D_eta u to LDS, D_zeta u kept by the lane
//   flux     t_a = sum_b G_ab (D_b u) at the lane's nodes (the layout in which
//            the matrix instruction leaves the zeta product), t_xi, t_eta,
//            t_zeta over the three arrays in place
//   adjoint  xi and eta products in place (a wavefront reads and writes its
//            own lines only), zeta kept; the three are added and stored
//
// Four barriers an element, against two a plane of the team kernel
// (ssx_ax.h), which holds 2N values and 2N to 4N entries of D a lane (216
// to 256 registers from N = 9, two wavefronts a SIMD) and idles a quarter of
// its lanes at N = 12.  LDS 3 N^2 (N|1) + 2 N (N|1) doubles, 47 KB at N = 12.
//
// What bounds it: HBM at N = 12 (64 B a node Poisson, 72 B Helmholtz), where
// the 16-line tiles and the 4-steps fit the order exactly and every factor
// load is four whole 128 B lines.  8000 elements, launched back to back:
// Poisson 238 -> 145-150 us (5.9-6.1 TB/s), Helmholtz 235 -> 166 us (6.0
// TB/s); in the assembled operator, with the DSS after it, the Helmholtz one
// takes 190 us (5.2 TB/s).  A Helmholtz CG iteration 475 -> 417 us.  It needs six (OP 0: seven) wavefronts a SIMD there: with
// five, the two workgroups of nine do not spread over the four SIMDs, 195 us.
// At N = 9 to 11 a fifth to a third of each tile and of the lanes is padding
// and the factor rows straddle lines: on large meshes the team kernel is the
// faster one (N = 10, 9216 elements: 135 us, here 133-155).  On small ones
// the short chain of phases counts, up to 512 elements at each of the three
// orders; us, team / here (Poisson, Helmholtz, a Helmholtz CG iteration):
//   elements       64                    512                   729
//   N =  9   7.5/6.0 7.4/6.1    9.3/8.5  9.3/8.8    10.0/10.4 10.0/14.0
//            18.6/15.6          25.7/24.7           28.1/30.9
//   N = 10  10.8/6.0 8.9/6.1   13.7/9.1 13.1/9.6    14.8/13.3 14.3/13.9
//            20.2/15.5          30.8/26.6           35.4/34.5
//   N = 11  10.3/6.3 10.7/6.4  13.8/10.8 13.6/11.8  16.1/16.4 16.5/16.8
//            22.3/16.6          34.7/30.4           41.7/38.9
// At 1000 elements it loses at N = 9 (11.9 / 18.0 Helmholtz) and 11 (19.1 /
// 21.2).  N = 13 needs 11 wavefronts and spills: 198 -> 239-278 us on a large
// mesh; 14 to 16 were not tried.
// Other lane layouts tried at N = 10 and 12: nodes in storage order in the
// flux phase with the zeta product through LDS too (N = 12 213 us).
#ifndef SSX_AXM_H
#define SSX_AXM_H
#include "ssx_ax.h"

// Where it is taken (a rule of order and size only: every launch of a level
// goes the same way).
template <int N, typename T>
static constexpr bool axm_takes = sizeof(T) == 8 && N >= 9 && N <= 12;
#define SSX_AXM_NEL 512
template <int N>
static inline bool axm_use(int nel)
{
	return N == 12 || nel <= SSX_AXM_NEL;
}

typedef double axm_v4 __attribute__((ext_vector_type(4)));

// p[i] with a uniform p: the load takes the base from scalar registers and
// a 32-bit lane offset, where p + i costs two registers an address
template <typename T>
__device__ __forceinline__ T &axm_at(T *p, unsigned i)
{
	return *(T *) ((const char *) p + i * (unsigned) sizeof(T));
}

template <bool B>
struct axm_flag {
	static constexpr bool value = B;
};

template <int N>
struct AxmShape {
	static constexpr int N2 = N * N, N3 = N2 * N;
	static constexpr int W = (N2 + 15) / 16;     // wavefronts
	static constexpr int BLOCK = 64 * W;
	static constexpr int KC = N | 1;             // odd LDS row
	static constexpr int F = N2 * KC;            // one array in LDS
	static constexpr int LDS = 3 * F + 2 * N * KC;   // and D, D of the SVV
	static constexpr int S = (N + 3) / 4;        // steps of 4 along a line
	static constexpr int R = (N + 3) / 4;        // result rows a lane may use
	static constexpr int M = (N3 + BLOCK - 1) / BLOCK;
};

// a matrix operand from LDS (rows of KC): value 4 t + kq of lane (col, kq) is
// m(col, 4 t + kq), zero outside N x N; TR: m(4 t + kq, col)
template <int N, bool TR>
__device__ __forceinline__ void axm_matrix(const double *m, int col, int kq,
		double e[(N + 3) / 4])
{
	constexpr int KC = N | 1;
	const int cc = col < N ? col : N - 1;
#pragma unroll
	for (int t = 0; t < (N + 3) / 4; ++t) {
		const int k = 4 * t + kq, kk = k < N ? k : N - 1;
		const double x = m[TR ? kk * KC + cc : cc * KC + kk];
		e[t] = col < N && k < N ? x : 0.0;
	}
}

// One workgroup's element e: the arguments of ax_team.  sm: LDS doubles.
// The element's value of sum p (A_e p) is returned in lane 0 of wavefront 0
// where `partial`.
template <int N, int OP, int PU, bool NT, typename SC>
__device__ __forceinline__ double axm_elem(size_t e, double *sm,
		const double *__restrict__ u, double *__restrict__ au,
		const double *__restrict__ gf, const double *__restrict__ mass,
		const double *__restrict__ dmat, double lambda, int ebits,
		int apply_mask, const double *__restrict__ zin,
		double *__restrict__ pio, double *__restrict__ uio, bool hc, SC &&sc,
		bool *stopped, bool partial)
{
	using S = AxmShape<N>;
	constexpr int N2 = S::N2, N3 = S::N3, KC = S::KC, R = S::R, M = S::M,
		ST = S::S;
	double *su = sm, *sx = sm + S::F, *sy = sm + 2 * S::F;
	// the SVV matrix enters the xi-forward and the eta/zeta-transposed
	// products only (helmholtz.c:41-44, deriv.c:29-66)
	double *sn = sm + 3 * S::F, *ss = OP == 1 ? sn + N * KC : sn;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int col = lane & 15, kq = lane >> 4;
	// this lane's line c of the tile and its nodes (4 r + kq, c) along zeta;
	// idle lanes and rows read the last line and row and store nothing
	const int cl = 16 * wave + col;
	const bool okc = cl < N2;
	const int c = okc ? cl : N2 - 1;
	const int cz = c / N, ci = c - cz * N;
	const size_t eoff = e * N3;
	const int bits = apply_mask ? ebits : 0;
	auto row = [&](int r) {
		return (unsigned) (4 * r + 3 < N || 4 * r + kq < N ? 4 * r + kq
				: N - 1);
	};
	auto in = [&](int r) { return okc && (4 * r + 3 < N || 4 * r + kq < N); };

	// ---- load
	double uv[M], f[R][6], ms[OP == 1 ? R : 1];
	double po[PU >= 1 ? M : 1], zz[PU >= 1 ? M : 1], uo[PU == 2 ? M : 1];
#pragma unroll
	for (int m = 0; m < M; ++m) {
		const int q = tid + m * S::BLOCK;
		const unsigned g = q < N3 ? q : N3 - 1;
		if (PU >= 1) {
			po[PU >= 1 ? m : 0] = axm_at(pio + eoff, g);
			zz[PU >= 1 ? m : 0] = axm_at(zin + eoff, g);
			if (PU == 2)
				uo[PU == 2 ? m : 0] = axm_at(uio + eoff, g);
		} else {
			uv[m] = axm_at(u + eoff, g);
		}
	}
	const double *ge = gf + e * 6 * N3;
	auto factors = [&]() {
#pragma unroll
		for (int r = 0; r < R; ++r) {
			const unsigned q = row(r) * N2 + c;
#pragma unroll
			for (int a = 0; a < 6; ++a) {
				if constexpr (NT)
					f[r][a] = __builtin_nontemporal_load(
							&axm_at(ge + a * N3, q));
				else
					f[r][a] = axm_at(ge + a * N3, q);
			}
			if (OP == 1)
				ms[OP == 1 ? r : 0] = axm_at(mass + eoff, q);
		}
	};
	// with the fused update the factors follow once its operands are used:
	// both at once cost the registers of a second workgroup a CU
	if (PU == 0)
		factors();
	constexpr int ND = OP == 1 ? 2 * N2 : N2;
	static_assert(ND <= S::BLOCK, "one entry of D a lane");
	const double dv = dmat[tid < ND ? tid : 0];
	AxScal s = {};
	if (PU >= 1) {
		s = sc();
		if (s.stop) {
			*stopped = true;
			return 0.0;
		}
	}
#pragma unroll
	for (int m = 0; m < M; ++m) {
		const int q = tid + m * S::BLOCK;
		if (PU >= 1) {
			const double pp = po[PU >= 1 ? m : 0], zq = zz[PU >= 1 ? m : 0];
			const double zv = hc ? -s.c + zq : zq;
			double v = s.b * pp + zv;
			if (bits) {
				const int k = q / N2, j = q / N - k * N, i = q % N;
				const bool mk = ((bits & 1) && i == 0)
					|| ((bits & 2) && i == N - 1) || ((bits & 4) && j == 0)
					|| ((bits & 8) && j == N - 1) || ((bits & 16) && k == 0)
					|| ((bits & 32) && k == N - 1);
				v = v * (mk ? 0.0 : 1.0);
			}
			if (q < N3) {
				if (PU == 2)
					axm_at(uio + eoff, q) = s.a * pp + uo[PU == 2 ? m : 0];
				axm_at(pio + eoff, q) = v;
			}
			uv[m] = v;
		}
		if ((m + 1) * S::BLOCK <= N3 || q < N3)
			su[KC == N ? q : q + q / N] = uv[m];
	}
	if (tid < ND)
		sn[KC == N ? tid : tid + tid / N] = dv;
	if (PU >= 1) {
		__builtin_amdgcn_sched_barrier(0);
		factors();
	}
	lds_sync();

	// ---- forward.  Operand k of line c: along xi line (z, y), eta (z, x),
	// zeta (y, x); entries past N are 0 on both sides
	auto opnd = [&](const double *w, int b, double x[ST]) {
#pragma unroll
		for (int t = 0; t < ST; ++t) {
			const int k = 4 * t + kq, kk = k < N ? k : N - 1;
			x[t] = b == 0 ? w[c * KC + kk] : b == 1
				? w[(cz * N + kk) * KC + ci] : w[(kk * N + cz) * KC + ci];
		}
		if (N % 4 != 0)
			x[ST - 1] = 4 * (ST - 1) + kq < N ? x[ST - 1] : 0.0;
	};
	// the product of direction b of `from` with m, or its transpose
	auto product = [&](int b, const double *from, const double *m, auto tr) {
		double x[ST], a[ST];
		opnd(from, b, x);
		axm_matrix<N, decltype(tr)::value>(m, col, kq, a);
		axm_v4 d = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
		for (int t = 0; t < ST; ++t)
			d = b == 0          // rows are lines, columns xi
				? __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], a[t], d, 0, 0, 0)
				: __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], x[t], d, 0, 0, 0);
		return d;
	};
	constexpr axm_flag<false> fwd{};
	constexpr axm_flag<true> adj{};
	auto store_x = [&](const axm_v4 &d) {
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			const int l = 16 * wave + 4 * r + kq;
			if (col < N && (16 * S::W == N2 || l < N2))
				sx[l * KC + col] = d[r];
		}
	};
	auto store_y = [&](const axm_v4 &d) {
#pragma unroll
		for (int r = 0; r < R; ++r)
			if (in(r))
				sy[(cz * N + 4 * r + kq) * KC + ci] = d[r];
	};
	store_x(product(0, su, ss, fwd));
	store_y(product(1, su, sn, fwd));
	const axm_v4 gz = product(2, su, sn, fwd);
	double uc[R];
	int nd[R];
#pragma unroll
	for (int r = 0; r < R; ++r) {
		nd[r] = (row(r) * N + cz) * KC + ci;
		uc[r] = su[nd[r]];
	}
	lds_sync();

	// ---- flux, over the arrays in place
#pragma unroll
	for (int r = 0; r < R; ++r) {
		const double gx = sx[nd[r]], gy = sy[nd[r]], gzr = gz[r];
		const double t0 = f[r][0] * gx + f[r][1] * gy + f[r][2] * gzr;
		const double t1 = f[r][1] * gx + f[r][3] * gy + f[r][4] * gzr;
		const double t2 = f[r][2] * gx + f[r][4] * gy + f[r][5] * gzr;
		if (in(r)) {
			sx[nd[r]] = t0;
			sy[nd[r]] = t1;
			su[nd[r]] = t2;
		}
	}
	lds_sync();

	// ---- adjoint; in place along xi and eta: a wavefront reads and writes
	// its own lines only
	store_x(product(0, sx, sn, adj));
	store_y(product(1, sy, ss, adj));
	const axm_v4 d = product(2, su, ss, adj);
	lds_sync();
	double pd = 0.0;
#pragma unroll
	for (int r = 0; r < R; ++r) {
		const int k = 4 * r + kq;
		double v = (sx[nd[r]] + sy[nd[r]]) + d[r];
		if (OP == 1)
			v += lambda * (ms[OP == 1 ? r : 0] * uc[r]);
		const bool mk = ((bits & 1) && ci == 0) || ((bits & 2) && ci == N - 1)
			|| ((bits & 4) && cz == 0) || ((bits & 8) && cz == N - 1)
			|| ((bits & 16) && k == 0) || ((bits & 32) && k == N - 1);
		v = mk ? 0.0 : v;
		if (in(r)) {
			double &o = axm_at(au + eoff, (unsigned) k * N2 + c);
			if (NT)
				__builtin_nontemporal_store(v, &o);
			else
				o = v;
			// <p, DSS(Ap)>_w as the sum over local copies (ssx_ax.h)
			pd += uc[r] * v;
		}
	}
	if (!partial)
		return 0.0;
	// a fixed tree: within the wavefront, then over the wavefronts in order
#pragma unroll
	for (int st = 32; st > 0; st >>= 1)
		pd += __shfl_down(pd, st, 64);
	if (lane == 0)
		su[wave] = pd;          // free since the adjoint's last barrier
	lds_sync();
	double t = 0.0;
	if (tid == 0)
#pragma unroll
		for (int w = 0; w < S::W; ++w)
			t += su[w];
	return t;
}

template <int N, int OP, int PU, bool NT>
__global__ void __launch_bounds__((AxmShape<N>::BLOCK),
		(N == 12 ? (OP == 0 ? 7 : 6) : 5))
k_axm(const double *__restrict__ u, double *__restrict__ au,
		const double *__restrict__ gf, const double *__restrict__ mass,
		const double *__restrict__ dmat, double lambda,
		const int *__restrict__ bc, int apply_mask,
		const int *done, double *__restrict__ part,
		const double *__restrict__ zin, double *__restrict__ pio,
		const double *__restrict__ scal, int ib, int ic,
		double *__restrict__ uio, int ia, ssx_replay rp)
{
	__shared__ double sm[AxmShape<N>::LDS];
	const bool late = ax_late(PU, rp);
	const int dn = done ? *done : 0;     // converged: no-op (as k_ax)
	if (!late && dn)
		return;
	bool stopped = false;
	const double pd = axm_elem<N, OP, PU, NT>(blockIdx.x, sm, u, au, gf, mass,
			dmat, lambda, bc[blockIdx.x], apply_mask, zin, pio, uio, ic >= 0,
			[&]() {
				AxScal s;
				const double al = PU == 2 ? scal[ia] : 0.0;
				if (rp.part) {
					s = replay_beta<AxmShape<N>::BLOCK>(rp, dn);
				} else {
					s.b = scal[ib];
					s.c = ic >= 0 ? scal[ic] : 0.0;
					s.stop = dn != 0;
				}
				s.a = al;
				return s;
			}, &stopped, part != nullptr);
	if (!stopped && part && threadIdx.x == 0)
		part[blockIdx.x] = pd;
}

template <int N, int PU, bool NT>
static void launch_axm(hipStream_t st, int nel, int op, const void *u,
		void *au, const void *gf, const void *mass, const void *dmat,
		double lambda, const int *bc, int apply_mask, const int *done,
		double *part, const PUpd &pu)
{
#define AXM(OP) hipLaunchKernelGGL((k_axm<N, OP, PU, NT>), dim3(nel), \
		dim3(AxmShape<N>::BLOCK), 0, st, (const double *) u, (double *) au, \
		(const double *) gf, (const double *) mass, (const double *) dmat, \
		lambda, bc, apply_mask, done, part, (const double *) pu.z, \
		(double *) pu.p, pu.scal, pu.ib, pu.ic, (double *) pu.u, pu.ia, pu.rp)
	if (op == SSX_OP_HELMHOLTZ)
		AXM(1);
	else
		AXM(0);
#undef AXM
}

#endif
