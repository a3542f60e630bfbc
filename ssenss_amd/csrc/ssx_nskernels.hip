// ssx_nskernels.hip -- element operators of the Navier-Stokes step around
// the elliptic solves (stokes.c, convection.c, poisson.c:58-224, time.c):
// reference-space Jacobians of fields, curl, weak divergence and gradient,
// the dealiased skew-symmetric convection operator at the convective
// resolution, face integrals, and the BDF3/EXT3 and interpolated-velocity
// combinations.  All on element-local E-vectors, node (e,k,j,i) at
// ((e*n+k)*n+j)*n+i; one thread per node unless stated.  The arithmetic
// keeps the reference's order of operations per node (products formed
// and summed in its loop order).
//
// D layout: dm[i*n+l] = D_il = l_l'(xi_i); reference derivatives
//   (D_xi u)(k,j,i)   = sum_l D_il u(k,j,l)
//   (D_eta u)(k,j,i)  = sum_l D_jl u(k,l,i)
//   (D_zeta u)(k,j,i) = sum_l D_kl u(l,j,i)          (deriv.c:29-52)
// Inverse Jacobian: ti[3*a+b] = d xi_b / d x_a (the transposed inverse
// tinv_jac, geometry.c:109-112).
#include <hip/hip_runtime.h>
#include "ssx_internal.h"
#include "ssx_device.h"

#define NS_LAUNCH(name)                                                    \
	do {                                                               \
		hipError_t e_ = hipGetLastError();                         \
		if (e_ != hipSuccess) {                                    \
			ssx_set_error("%s: %s", name, hipGetErrorString(e_)); \
			return SSX_EHIP;                                   \
		}                                                          \
	} while (0)

struct P3 { const double *p[3]; };
struct M3 { double *p[3]; };
struct P9 { const double *p[9]; };

static inline unsigned ns_blocks(size_t n)
{
	return (unsigned) ((n + 255) / 256);
}

// The curl and the weak divergence of a field a, from its Jacobian J[3a+b] =
// D_b a_a (compute_jacobian, deriv.c:68-79), in one launch:
// curl (discrete_curl_operator, stokes.c:71-92): omega_c, for c = 0..2 and
// xi-direction i = 0..2 in that loop order, += s_c (D_i u_k)(d xi_i/d x_l)
// - s_c (D_i u_l)(d xi_i/d x_k) with k = (5-c)/2, l = (2-c)/2, s = (+1, -1,
// +1); with mass, times w detJ (the test-function product of
// double_curl_operator, stokes.c:94-105).
// divergence (DIV; discrete_divergence_operator, stokes.c:52-69): sum_a sum_b
// (D_b u_a)(d xi_b/d x_a) in that loop order, times w detJ, times `scale`.
//
// Bound by the 16 values (divergence: 14) a node that it moves: n = 10, 9.2
// million nodes, 197 us at 6 TB/s.  A workgroup takes the elements that make
// about 512 nodes, or one element, with the three fields and D in LDS, so
// that a node's 9 n products read LDS; read from memory, with the Jacobian
// stored between two launches, the curl took 826 + 300 us; now 225, the
// divergence 1102 -> 221.
template <int N>
struct JacShape {
	static constexpr int N3 = N * N * N;
	static constexpr int E = N3 >= 512 ? 1 : 512 / N3;
};

template <int N, bool DIV>
__global__ void __launch_bounds__(256)
k_ns_jac(int nel, const double *__restrict__ dm, P3 a, P9 ti,
		const double *__restrict__ mass, double scale, M3 out)
{
	constexpr int N3 = JacShape<N>::N3, E = JacShape<N>::E;
	__shared__ double sa[3][E * N3], sd[N][N + 1];
	const int e0 = blockIdx.x * E;
	const int m = (nel - e0 < E ? nel - e0 : E) * N3;
	const size_t b0 = (size_t) e0 * N3;
	for (int q = threadIdx.x; q < N * N; q += 256)
		sd[q / N][q % N] = dm[q];
#pragma unroll
	for (int c = 0; c < 3; ++c)
		for (int q = threadIdx.x; q < m; q += 256)
			sa[c][q] = a.p[c][b0 + q];
	__syncthreads();
	for (int q = threadIdx.x; q < m; q += 256) {
		double tv[9];
#pragma unroll
		for (int b = 0; b < 9; ++b)
			tv[b] = ti.p[b][b0 + q];
		const double mv = mass ? mass[b0 + q] : 1.0;
		const int i = q % N, j = (q / N) % N, k = (q / (N * N)) % N;
		const int x0 = q - i, y0 = q - j * N, z0 = q - k * N * N;
		double jv[9];
#pragma unroll
		for (int b = 0; b < 9; ++b)
			jv[b] = 0.0;
#pragma unroll
		for (int l = 0; l < N; ++l) {
			const double dx = sd[i][l], dy = sd[j][l], dz = sd[k][l];
#pragma unroll
			for (int c = 0; c < 3; ++c) {
				jv[3 * c] += dx * sa[c][x0 + l];
				jv[3 * c + 1] += dy * sa[c][y0 + l * N];
				jv[3 * c + 2] += dz * sa[c][z0 + l * N * N];
			}
		}
		if (DIV) {
			double s = jv[0] * tv[0];
#pragma unroll
			for (int b = 1; b < 9; ++b)
				s = jv[b] * tv[b] + s;
			out.p[0][b0 + q] = (s * mv) * scale;
		} else {
#pragma unroll
			for (int c = 0; c < 3; ++c) {
				const int kk = (5 - c) / 2, l = (2 - c) / 2;
				const double s = c == 1 ? -1.0 : 1.0;
				double om = 0.0;
#pragma unroll
				for (int b = 0; b < 3; ++b) {
					const double t = s * jv[3 * kk + b] * tv[3 * l + b];
					om = b == 0 ? t : t + om;
					om = -s * jv[3 * l + b] * tv[3 * kk + b] + om;
				}
				out.p[c][b0 + q] = om * mv;
			}
		}
	}
}

// weak gradient (discrete_gradient_operator, stokes.c:30-50): with
// t = p w detJ and f_b = (d xi_b/d x_c) t, grad_c = -(D_xi^T f_0 +
// D_eta^T f_1 + D_zeta^T f_2) (transpose_divergence, deriv.c:54-66)
// Bound by the 14 values a node that it moves.  Laid out as k_ns_jac, one
// component's three f_b in LDS at a time; read from memory by each of the 3 n
// nodes that use it, it took 1626 us on 9.2 million nodes, n = 10; now 254.
template <int N>
__global__ void __launch_bounds__(256)
k_ns_grad(int nel, const double *__restrict__ dm, const double *__restrict__ p,
		const double *__restrict__ mass, P9 ti, M3 out)
{
	constexpr int N3 = JacShape<N>::N3, E = JacShape<N>::E;
	constexpr int R = (E * N3 + 255) / 256;
	__shared__ double sf[3][E * N3], sd[N][N + 1];
	const int e0 = blockIdx.x * E;
	const int m = (nel - e0 < E ? nel - e0 : E) * N3;
	const size_t b0 = (size_t) e0 * N3;
	for (int q = threadIdx.x; q < N * N; q += 256)
		sd[q % N][q / N] = dm[q];           // transposed: sd[i][l] = D_li
	double t[R];
#pragma unroll
	for (int r = 0; r < R; ++r) {
		const int q = threadIdx.x + 256 * r;
		t[r] = q < m ? p[b0 + q] * mass[b0 + q] : 0.0;
	}
	for (int c = 0; c < 3; ++c) {
#pragma unroll
		for (int r = 0; r < R; ++r) {
			const int q = threadIdx.x + 256 * r;
			if (q < m) {
#pragma unroll
				for (int b = 0; b < 3; ++b)
					sf[b][q] = ti.p[3 * c + b][b0 + q] * t[r];
			}
		}
		__syncthreads();
		for (int q = threadIdx.x; q < m; q += 256) {
			const int i = q % N, j = (q / N) % N, k = (q / (N * N)) % N;
			const int x0 = q - i, y0 = q - j * N, z0 = q - k * N * N;
			double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
			for (int l = 0; l < N; ++l) {
				sx += sd[i][l] * sf[0][x0 + l];
				sy += sd[j][l] * sf[1][y0 + l * N];
				sz += sd[k][l] * sf[2][z0 + l * N * N];
			}
			out.p[c][b0 + q] = -((sx + sy) + sz);
		}
		__syncthreads();
	}
}

// ---------------------------------------------------------------------
// The dealiased skew-symmetric convection operator, one workgroup per
// element (antialiased_convection_operator, convection.c:37-69): u and v
// interpolated from N to NC = 3N/2 points, half the convective form
// (u . grad) v_c (:71-93) plus half the conservative form as
// convection.c:95-127 forms it, sum_a sum_b (d xi_b/d x_a) D_b(u_b v_c),
// each times w detJ, integrated back to N points.
//
// Every contraction (interpolation, D, and their transposes) is a product
// of a small constant matrix with the element's lines, taken by the FP64
// matrix instruction 16x16x4: the constant matrix sits in registers (one
// value a lane and step of 4), the lines come from LDS once each, so LDS
// carries one read and one write per value and contraction.  The earlier
// form (one lane a node, matrix and lines read from LDS at every
// multiply-add) was LDS-bound.
//
// With C_b = sum_a u_a g_ab and T_b = sum_a g_ab, g_ab = w detJ d xi_b/d x_a
// (premultiplied at set-up), both forms together are
//   0.5 sum_b (C_b D_b v_c + T_b D_b(u_b v_c)),
// so the nine factors are read once, in the lane layout in which the
// matrix instruction leaves D_b's result (another for each direction b:
// 36 loads a lane), and the three components take them from registers;
// the directions meet in LDS.  One wavefront a tile of 16 lines, W =
// ceil(NC^2 / 16) of them (960 lanes at NC = 15); LDS 6 NC^2 (NC|1)
// doubles: one workgroup a CU at N = 10.
//
// What bounds it at N = 10: 12 short phases between barriers of the one
// workgroup a CU holds.  The matrix instructions (2050 of them an element,
// 0.5 ms on 9216 elements at their peak) keep their unit busy 38 % of the
// time and the address arithmetic its own 26 %; the factors (2.2 GB) are
// loaded during the contractions of u.  Measured per evaluation: 9216
// elements at N = 10 3.5 -> 1.47 ms, 64 elements at N = 8 48 -> 24 us.
// ---------------------------------------------------------------------
typedef double conv_v4 __attribute__((ext_vector_type(4)));

template <int N, int NC>
struct ConvShape {
	static constexpr int W = (NC * NC + 15) / 16;   // wavefronts
	static constexpr int KP = N | 1, KC = NC | 1;   // odd LDS rows
	static constexpr int REG = 3 * NC * NC * KC;    // doubles of a region
	static constexpr size_t BYTES = sizeof(double) * (2 * REG + 64);
};

// D's rows of the 16x16x4 instruction: lane l holds rows 4 r + l / 16 (r =
// 0..3) of column l % 16; A: row l % 16, k = l / 16; B: column l % 16, k =
// l / 16
#define CONV_ROW(r) (4 * (r) + kq)

// one contraction of three components: for every line l < C of component f,
// dst(f, l)[m * SM] = sum_k a[m][k] src(f, l)[k], m < M, k < K.  A
// wavefront takes its tiles of 16 lines together (all loads, then the
// matrix instructions in turn), with no branch: lines and rows past the end
// read the last line and write to `dump` (DUMP false: not at all).
template <int M, int K, int C, int SM, int W, bool DUMP, typename Src,
		typename Dst>
__device__ __forceinline__ void conv_stage(const double *a, int wave,
		int lane, double *dump, Src src, Dst dst)
{
	constexpr int KS = (K + 3) / 4, TI = ((3 * C + 15) / 16 + W - 1) / W;
	const int l = fresh(lane), col = l & 15, kq = l >> 4;
	const int klast = 4 * (KS - 1) + kq < K ? 4 * (KS - 1) + kq : K - 1;
	double b[TI][KS];
	double *o[TI];
	bool ok[TI];
	conv_v4 d[TI];
#pragma unroll
	for (int t = 0; t < TI; ++t) {
		const int q0 = 16 * (wave + t * W) + col;
		const int q = q0 < 3 * C ? q0 : 3 * C - 1;
		const int f = q / C, c = q - f * C;
		const double *p = src(f, c);
#pragma unroll
		for (int s = 0; s < KS; ++s)
			b[t][s] = p[s < KS - 1 ? 4 * s + kq : klast];
		ok[t] = q0 < 3 * C;
		o[t] = dst(f, c) + kq * SM;
	}
	// every load issued before the first is used, none behind a branch
#pragma unroll
	for (int t = 0; t < TI; ++t) {
#pragma unroll
		for (int s = 0; s < KS; ++s)
			asm volatile("" : "+v"(b[t][s]));
		if (K % 4 != 0)
			b[t][KS - 1] = 4 * (KS - 1) + kq < K ? b[t][KS - 1] : 0.0;
		d[t] = conv_v4{ 0.0, 0.0, 0.0, 0.0 };
	}
#pragma unroll
	for (int s = 0; s < KS; ++s)
#pragma unroll
		for (int t = 0; t < TI; ++t)
			d[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[t][s], d[t],
					0, 0, 0);
#pragma unroll
	for (int t = 0; t < TI; ++t)
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			if (4 * r >= M)
				continue;
			const bool in = ok[t] && (4 * r + 3 < M || CONV_ROW(r) < M);
			if (DUMP)
				*(in ? o[t] + 4 * r * SM : dump) = d[t][r];
			else if (in)
				o[t][4 * r * SM] = d[t][r];
		}
}

template <int N, int NC>
__global__ void __launch_bounds__((64 * ConvShape<N, NC>::W))
k_ns_conv(const double *__restrict__ prol, const double *__restrict__ dm,
		P3 u, P3 v, const double *__restrict__ geo, M3 out)
{
	using S = ConvShape<N, NC>;
	constexpr int W = S::W, KP = S::KP, KC = S::KC;
	constexpr int N2 = N * N, N3 = N2 * N, C2 = NC * NC, C3 = C2 * NC;
	constexpr int F3 = C2 * KC;             // one field at NC points in LDS
	constexpr int SP = (N + 3) / 4, SC = (NC + 3) / 4;
	extern __shared__ double sm[];
	double *ra = sm, *rb = sm + S::REG;
	double *dump = sm + 2 * S::REG + (threadIdx.x & 63);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int col = lane & 15, kq = lane >> 4;
	const size_t e = blockIdx.x;
	// the interpolation matrix (rows < NC, k < N), zero outside; D and the
	// transpose are loaded where they are used, to keep registers free
	double ap[SP];
#pragma unroll
	for (int s = 0; s < SP; ++s) {
		const int k = 4 * s + kq;
		const bool ok = col < NC && k < N;
		const double x = prol[ok ? k * NC + col : 0];
		ap[s] = ok ? x : 0.0;
	}
	// this wavefront's lines: line c of tile `wave` along eta (z, x), zeta
	// (y, x) by column, along xi (z, y) by row; idle lanes take line 0
	struct Line { int col, kq, c, cz, ci; bool ok; };
	auto line = [&]() {
		const int l = fresh(lane);
		Line w;
		w.col = l & 15;
		w.kq = l >> 4;
		const int cl = 16 * wave + w.col;
		w.ok = cl < C2;
		w.c = w.ok ? cl : 0;
		w.cz = w.c / NC;
		w.ci = w.c - w.cz * NC;
		return w;
	};

	// three contractions: interpolation of w (global) to NC points in ra
	// ([X][z][y], then [Y][X][z], then [Z][Y][X])
	auto interpolate = [&](const P3 &w, auto &&loads) {
		const double *w0 = w.p[0] + e * N3, *w1 = w.p[1] + e * N3,
			*w2 = w.p[2] + e * N3;
		conv_stage<NC, N, N2, N * KP, W, true>(ap, wave, lane, dump,
			[&](int f, int l) {
				return (f == 0 ? w0 : f == 1 ? w1 : w2) + l * N;
			},
			[&](int f, int l) {
				return ra + f * (NC * N * KP) + (l / N) * KP + l % N;
			});
		loads();
		lds_sync();
		conv_stage<NC, N, NC * N, NC * KP, W, true>(ap, wave, lane, dump,
			[&](int f, int l) { return ra + f * (NC * N * KP) + l * KP; },
			[&](int f, int l) {
				return rb + f * (C2 * KP) + (l / N) * KP + l % N;
			});
		lds_sync();
		conv_stage<NC, N, C2, NC * KC, W, true>(ap, wave, lane, dump,
			[&](int f, int l) { return rb + f * (C2 * KP) + l * KP; },
			[&](int f, int l) {
				return ra + f * F3 + (l / NC) * KC + l % NC;
			});
		lds_sync();
	};

	// node of this lane's result r along direction b, as line (z, y) and x:
	// along xi the rows are lines and the columns x (idle lanes: node 0)
	auto result = [&](const Line &w, int b, int r, int &zy, int &x) {
		const int m = 4 * r + w.kq;
		if (b == 0) {
			const int l = 16 * wave + m;
			const bool ok = l < C2 && w.col < NC;
			zy = ok ? l : 0;
			x = ok ? w.col : 0;
		} else {
			const int mm = w.ok && m < NC ? m : 0;
			zy = b == 1 ? w.cz * NC + mm : mm * NC + w.cz;
			x = w.ci;
		}
	};

	// the factors at those nodes, issued after u's own loads and in flight
	// during the other two contractions (the barriers order LDS only)
	double gv[3][4][3];
	const double *g = geo + e * 9 * C3;
	interpolate(u, [&]() {
#pragma unroll
		for (int b = 0; b < 3; ++b) {
			const Line w = line();
#pragma unroll
			for (int r = 0; r < 4; ++r) {
				int zy, x;
				result(w, b, r, zy, x);
				// uniform base, 32-bit lane offset
				const unsigned q = 8u * (unsigned) (zy * NC + x);
#pragma unroll
				for (int a = 0; a < 3; ++a)
					gv[b][r][a] = *(const double *) ((const char *)
							(g + (3 * a + b) * C3) + q);
			}
		}
	});
	// C_b, T_b at this lane's results, and u_b at its operands
	double cc[3][4], tt[3][4], uo[3][SC];
#pragma unroll
	for (int b = 0; b < 3; ++b) {
		const Line w = line();
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			int zy, x;
			result(w, b, r, zy, x);
			const double *q = ra + zy * KC + x;
			tt[b][r] = (gv[b][r][0] + gv[b][r][1]) + gv[b][r][2];
			cc[b][r] = q[0] * gv[b][r][0] + q[F3] * gv[b][r][1]
				+ q[2 * F3] * gv[b][r][2];
			// formed here: sunk to their use, their operands spilled
			asm volatile("" : "+v"(tt[b][r]), "+v"(cc[b][r]));
		}
	}
	// operand k of line c along each direction (clamped: a[k >= NC] is 0
	// and the value there is replaced by 0)
	auto opnd = [&](const double *f, const Line &w, int b, int s) {
		const int k = 4 * s + w.kq, kk = k < NC ? k : NC - 1;
		const double x = b == 0 ? f[w.c * KC + kk]
			: b == 1 ? f[(w.cz * NC + kk) * KC + w.ci]
			: f[(kk * NC + w.cz) * KC + w.ci];
		return k < NC ? x : 0.0;
	};
#pragma unroll
	for (int b = 0; b < 3; ++b) {
		const Line w = line();
#pragma unroll
		for (int s = 0; s < SC; ++s)
			uo[b][s] = opnd(ra + b * F3, w, b, s);
	}
#pragma unroll
	for (int b = 0; b < 3; ++b)
#pragma unroll
		for (int s = 0; s < SC; ++s)
			asm volatile("" : "+v"(uo[b][s]));
	lds_sync();

	interpolate(v, []() {});
	// the operator at NC points in rb, direction by direction
	double ad[SC];
#pragma unroll
	for (int s = 0; s < SC; ++s) {
		const int k = 4 * s + kq;
		const bool ok = col < NC && k < NC;
		const double x = dm[ok ? col * NC + k : 0];
		ad[s] = ok ? x : 0.0;
	}
#pragma unroll
	for (int b = 0; b < 3; ++b) {
		__builtin_amdgcn_sched_barrier(0);
		const Line w = line();
		const int kq = w.kq;
#pragma unroll 1
		for (int f = 0; f < 3; ++f) {
			conv_v4 d1 = { 0.0, 0.0, 0.0, 0.0 }, d2 = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
			for (int s = 0; s < SC; ++s) {
				const double x = opnd(ra + f * F3, w, b, s);
				const double y = uo[b][s] * x;
				if (b == 0) {
					d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, ad[s], d1,
							0, 0, 0);
					d2 = __builtin_amdgcn_mfma_f64_16x16x4f64(y, ad[s], d2,
							0, 0, 0);
				} else {
					d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ad[s], x, d1,
							0, 0, 0);
					d2 = __builtin_amdgcn_mfma_f64_16x16x4f64(ad[s], y, d2,
							0, 0, 0);
				}
			}
#pragma unroll
			for (int r = 0; r < 4; ++r) {
				const int m = CONV_ROW(r);
				const double x = cc[b][r] * d1[r] + tt[b][r] * d2[r];
				if (b == 0) {
					const int l = 16 * wave + m;
					if (l < C2 && w.col < NC)
						rb[f * F3 + l * KC + w.col] = x;
				} else if (w.ok && m < NC) {
					double *o = rb + f * F3 + (b == 1
						? (w.cz * NC + m) * KC + w.ci
						: (m * NC + w.cz) * KC + w.ci);
					*o = b == 1 ? *o + x : 0.5 * (*o + x);
				}
			}
		}
		lds_sync();
	}
	// integrated back to N points (the transposed contractions)
	double ar[SC];
#pragma unroll
	for (int s = 0; s < SC; ++s) {
		const int k = 4 * s + kq;
		const bool ok = col < N && k < NC;
		const double x = prol[ok ? col * NC + k : 0];
		ar[s] = ok ? x : 0.0;
	}
	// ([p][z][y], [q][p][z], then z, y, x in global memory)
	conv_stage<N, NC, C2, NC * KC, W, true>(ar, wave, lane, dump,
		[&](int f, int l) { return rb + f * F3 + l * KC; },
		[&](int f, int l) {
			return ra + f * (N * NC * KC) + (l / NC) * KC + l % NC;
		});
	lds_sync();
	conv_stage<N, NC, N * NC, N * KC, W, true>(ar, wave, lane, dump,
		[&](int f, int l) { return ra + f * (N * NC * KC) + l * KC; },
		[&](int f, int l) {
			return rb + f * (N2 * KC) + (l / NC) * KC + l % NC;
		});
	lds_sync();
	double *o0 = out.p[0] + e * N3, *o1 = out.p[1] + e * N3,
		*o2 = out.p[2] + e * N3;
	conv_stage<N, NC, N2, N2, W, false>(ar, wave, lane, nullptr,
		[&](int f, int l) { return rb + f * (N2 * KC) + l * KC; },
		[&](int f, int l) { return (f == 0 ? o0 : f == 1 ? o1 : o2) + l; });
}

// the element's LDS granted to the kernel on the current device
template <int N>
static int conv_lds(void)
{
	constexpr int NC = (3 * N) / 2;
	using S = ConvShape<N, NC>;
	if (hipFuncSetAttribute((const void *) k_ns_conv<N, NC>,
			hipFuncAttributeMaxDynamicSharedMemorySize, (int) S::BYTES)
			!= hipSuccess) {
		ssx_set_error("k_ns_conv: %zu bytes of LDS refused", S::BYTES);
		return SSX_EHIP;
	}
	return SSX_OK;
}

template <int N>
static int launch_conv(hipStream_t st, int nel, const double *prol,
		const double *dm, const P3 &u, const P3 &v, const double *geo,
		const M3 &out)
{
	constexpr int NC = (3 * N) / 2;
	using S = ConvShape<N, NC>;
	static_assert(S::W <= 16 && S::BYTES <= 160 * 1024, "element too large");
	const int rc = conv_lds<N>();
	if (rc != SSX_OK)
		return rc;
	hipLaunchKernelGGL((k_ns_conv<N, NC>), dim3(nel), dim3(64 * S::W),
			S::BYTES, st, prol, dm, u, v, geo, out);
	return SSX_OK;
}

// f += (w_b w_a) n_s g on the face nodes of every face s of an element
// whose Dirichlet bit equals `dirichlet` (add_surface_integral,
// poisson.c:145-210: all nodes of face W, then E, S, N, B, T).  One
// workgroup per element; faces in order, so edge and corner nodes take
// their additions in the reference's order.  wn[(e*6+s)*n*n + a*n+b] =
// (w_b w_a) n_s(a,b) for the normal component of the direction.
__global__ void __launch_bounds__(256)
k_ns_surf(int nel, int n, const int *__restrict__ bc, int dirichlet,
		const double *__restrict__ wn, const double *__restrict__ g,
		double *__restrict__ f)
{
	const int e = blockIdx.x;
	const int n2 = n * n, n3 = n2 * n, m = n - 1;
	const int bits = bc[e];
	const long long b0 = (long long) e * n3;
	for (int s = 0; s < 6; ++s) {
		const int isd = (bits >> s) & 1;
		if (isd == dirichlet) {
			for (int t = threadIdx.x; t < n2; t += blockDim.x) {
				const int a = t / n, b = t % n;
				int k, j, i;
				switch (s) {
				case 0: k = a; j = b; i = 0; break;
				case 1: k = a; j = b; i = m; break;
				case 2: k = a; j = 0; i = b; break;
				case 3: k = a; j = m; i = b; break;
				case 4: k = 0; j = a; i = b; break;
				default: k = m; j = a; i = b; break;
				}
				const long long q = b0 + (k * n + j) * n + i;
				f[q] += wn[((long long) e * 6 + s) * n2 + t] * g[q];
			}
		}
		__syncthreads();
	}
}

// u = 0 on the nodes of the element's Dirichlet faces
// (set_dirichlet_boundaries with the reference's zero boundary function,
// poisson.c:101-143, structs.c:67)
__global__ void __launch_bounds__(256)
k_ns_zero_dir(long long nt, int n, const int *__restrict__ bc, M3 u)
{
	const long long q = (long long) blockIdx.x * 256 + threadIdx.x;
	if (q >= nt)
		return;
	const int n3 = n * n * n, m = n - 1;
	const long long e = q / n3;
	const int r = (int) (q - e * n3);
	const int i = r % n, j = (r / n) % n, k = r / (n * n);
	const int bits = bc[e];
	const bool z = ((bits & 1) && i == 0) || ((bits & 2) && i == m)
		|| ((bits & 4) && j == 0) || ((bits & 8) && j == m)
		|| ((bits & 16) && k == 0) || ((bits & 32) && k == m);
	if (z)
		for (int c = 0; c < 3; ++c)
			u.p[c][q] = 0.0;
}

// y_c = ((a0 x0_c + y_c) + a1 x1_c) + a2 x2_c for the three components,
// a term skipped where its flag is clear (the daxpy sequences of
// stiffly_stable, time.c:51-73, and add_interpolated_velocity,
// time.c:132-152)
struct Comb {
	const double *x[3][3];    // [term][component]
	double a[3];
	int use[3];
};

__global__ void __launch_bounds__(256)
k_ns_comb(long long nt, Comb cb, M3 y)
{
	const long long q = (long long) blockIdx.x * 256 + threadIdx.x;
	if (q >= nt)
		return;
	for (int c = 0; c < 3; ++c) {
		double v = y.p[c][q];
		for (int t = 0; t < 3; ++t)
			if (cb.use[t])
				v = cb.a[t] * cb.x[t][c][q] + v;
		y.p[c][q] = v;
	}
}

// z_c = alpha x_c w + beta z_c, w shared by the components or per
// component (multiply, linalg.c:142-152); w NULL: z_c = alpha x_c +
// beta z_c
__global__ void __launch_bounds__(256)
k_ns_mul3(long long nt, double alpha, P3 x, P3 w, double beta, M3 z)
{
	const long long q = (long long) blockIdx.x * 256 + threadIdx.x;
	if (q >= nt)
		return;
	for (int c = 0; c < 3; ++c) {
		if (!z.p[c])
			continue;
		const double wv = w.p[c] ? w.p[c][q] : 1.0;
		const double old = beta != 0.0 ? beta * z.p[c][q] : 0.0;
		z.p[c][q] = alpha * x.p[c][q] * wv + old;
	}
}

// One stage of the convection RK4 (time.c:84-130), per node and component
// (blockIdx.y): a = sum of T terms co_t x_t, the velocity at the stage's time
// (from zero, in order), and with STAGE y = ut + ch (im f), the stage's
// argument, im f being the inverse mass applied to the last stage's f.
// With T alone it is any such sum; a may be one of the x.
// Bound by the T + 1 (+ 4) values it moves (T = 3 with STAGE: 311 us on 9.2
// million nodes, 5.7 TB/s).  The stage had 13 launches: three copies, three
// fills, two sums read and written in place, one DSS a component, the
// inverse mass; 2 to 5 us each on 64 elements of 8 points, 0.83 ms
// together on the 9.2 million nodes.  Now this, the operator and one DSS,
// and a velocity formed once for the stages at one time: 0.43 ms.
struct RkTerms {
	const double *x[3][3];    // [term][component]
	double co[3];
};

template <int T, bool STAGE>
__global__ void __launch_bounds__(256)
k_ns_rk_stage(long long nt, RkTerms rk, P3 ut, P3 f,
		const double *__restrict__ im, double ch, M3 a, M3 y)
{
	const long long q = (long long) blockIdx.x * 256 + threadIdx.x;
	const int c = blockIdx.y;
	if (q >= nt)
		return;
	double xv[T > 0 ? T : 1], uv = 0.0, fv = 0.0, mv = 0.0;
#pragma unroll
	for (int t = 0; t < T; ++t)
		xv[t] = rk.x[t][c][q];
	if (STAGE) {
		uv = ut.p[c][q];
		fv = f.p[c][q];
		mv = im[q];
	}
	if (T > 0) {
		double v = 0.0;
#pragma unroll
		for (int t = 0; t < T; ++t)
			v = rk.co[t] * xv[t] + v;
		a.p[c][q] = v;
	}
	if (STAGE) {
		const double g = __dmul_rn(fv, mv);
		y.p[c][q] = ch * g + uv;
	}
}

// ut += sum of the four stages, in order, the inverse mass applied to each
__global__ void __launch_bounds__(256)
k_ns_rk_end(long long nt, P3 f0, P3 f1, P3 f2, P3 f3,
		const double *__restrict__ im, double c0, double c1, M3 ut)
{
	const long long q = (long long) blockIdx.x * 256 + threadIdx.x;
	const int c = blockIdx.y;
	if (q >= nt)
		return;
	const double mv = im[q];
	const double g0 = __dmul_rn(f0.p[c][q], mv);
	const double g1 = __dmul_rn(f1.p[c][q], mv);
	const double g2 = __dmul_rn(f2.p[c][q], mv);
	const double g3 = __dmul_rn(f3.p[c][q], mv);
	double v = ut.p[c][q];
	v = c0 * g0 + v;
	v = c1 * g1 + v;
	v = c1 * g2 + v;
	ut.p[c][q] = c0 * g3 + v;
}

// dss_group on three fields: the group's list read once, the three sums of
// a copy in dss_group's order
template <int M>
__device__ __forceinline__ void dss3_group(long long G, long long g,
		const int *__restrict__ idx, M3 u)
{
	int ix[M];
	double v[3][M];
#pragma unroll
	for (int t = 0; t < M; ++t)
		ix[t] = idx[(long long) t * G + g];
#pragma unroll
	for (int c = 0; c < 3; ++c)
#pragma unroll
		for (int t = 0; t < M; ++t)
			v[c][t] = u.p[c][ix[t]];
#pragma unroll
	for (int c = 0; c < 3; ++c)
#pragma unroll
		for (int t = 0; t < M; ++t) {
			double s = v[c][t];
#pragma unroll
			for (int k = 1; k < M; ++k)
				s = s + v[c][t ^ dss_ord(M, k)];
			u.p[c][ix[t]] = s;
		}
}

// k_dss_all on three fields in one launch
__global__ void __launch_bounds__(256)
k_ns_dss3(long long G2, long long G4, long long G8,
		const int *__restrict__ i2, const int *__restrict__ i4,
		const int *__restrict__ i8, M3 u)
{
	const long long b2 = (G2 + 255) / 256, b4 = (G4 + 255) / 256;
	const long long b = blockIdx.x;
	if (b < b2) {
		const long long g = b * 256 + threadIdx.x;
		if (g < G2)
			dss3_group<2>(G2, g, i2, u);
	} else if (b < b2 + b4) {
		const long long g = (b - b2) * 256 + threadIdx.x;
		if (g < G4)
			dss3_group<4>(G4, g, i4, u);
	} else {
		const long long g = (b - b2 - b4) * 256 + threadIdx.x;
		if (g < G8)
			dss3_group<8>(G8, g, i8, u);
	}
}

// nterm 0..3 terms; f NULL: no stage argument; ncomp components
extern "C" int ssxk_ns_rk_stage(void *st, size_t nt, int ncomp, int nterm,
		const double *const x[3][3], const double co[3],
		const double *const ut[3], const double *const f[3],
		const double *im, double ch, double *const a[3], double *const y[3])
{
	RkTerms rk;
	P3 pu, pf;
	M3 pa, py;
	for (int c = 0; c < 3; ++c) {
		for (int t = 0; t < 3; ++t)
			rk.x[t][c] = t < nterm && c < ncomp ? x[t][c] : nullptr;
		pu.p[c] = f ? ut[c] : nullptr;
		pf.p[c] = f ? f[c] : nullptr;
		pa.p[c] = nterm && c < ncomp ? a[c] : nullptr;
		py.p[c] = f ? y[c] : nullptr;
		rk.co[c] = c < nterm ? co[c] : 0.0;
	}
	const dim3 grid(ns_blocks(nt), (unsigned) ncomp);
#define RKCASE(T, F)                                                         \
	case 2 * T + F:                                                      \
		hipLaunchKernelGGL((k_ns_rk_stage<T, F>), grid, dim3(256), 0,    \
				(hipStream_t) st, (long long) nt, rk, pu, pf, im, ch, \
				pa, py);                                     \
		break;
	switch (2 * nterm + (f ? 1 : 0)) {
	RKCASE(0, 1) RKCASE(1, 0) RKCASE(1, 1) RKCASE(2, 0) RKCASE(2, 1)
	RKCASE(3, 0) RKCASE(3, 1)
	default:
		break;                          // nothing asked for
	}
#undef RKCASE
	NS_LAUNCH("k_ns_rk_stage");
	return SSX_OK;
}

extern "C" int ssxk_ns_rk_end(void *st, size_t nt,
		double *const f[4][3], const double *im, double c0, double c1,
		double *const ut[3])
{
	P3 pf[4];
	for (int i = 0; i < 4; ++i)
		for (int c = 0; c < 3; ++c)
			pf[i].p[c] = f[i][c];
	M3 pu = { { ut[0], ut[1], ut[2] } };
	hipLaunchKernelGGL(k_ns_rk_end, dim3(ns_blocks(nt), 3), dim3(256), 0,
			(hipStream_t) st, (long long) nt, pf[0], pf[1], pf[2], pf[3], im,
			c0, c1, pu);
	NS_LAUNCH("k_ns_rk_end");
	return SSX_OK;
}

extern "C" int ssxk_ns_dss3(void *st, int *const grp[3],
		const long long ng[3], double *const u[3])
{
	const long long nb = ssxk_dss_blocks(ng);
	M3 pu = { { u[0], u[1], u[2] } };
	if (nb == 0)
		return SSX_OK;
	hipLaunchKernelGGL(k_ns_dss3, dim3((unsigned) nb), dim3(256), 0,
			(hipStream_t) st, ng[0], ng[1], ng[2], grp[0], grp[1], grp[2],
			pu);
	NS_LAUNCH("k_ns_dss3");
	return SSX_OK;
}

template <bool DIV>
static int launch_jac(const char *name, void *st, int nel, int n,
		const double *dm, const double *const a[3], const double *const ti[9],
		const double *mass, double scale, M3 out)
{
	P3 pa = { { a[0], a[1], a[2] } };
	P9 pt;
	for (int k = 0; k < 9; ++k)
		pt.p[k] = ti[k];
#define JCASE(N)                                                             \
	case N:                                                              \
		hipLaunchKernelGGL((k_ns_jac<N, DIV>), dim3((unsigned) ((nel     \
				+ JacShape<N>::E - 1) / JacShape<N>::E)), dim3(256), 0, \
				(hipStream_t) st, nel, dm, pa, pt, mass, scale, out); \
		break;
	switch (n) {
	JCASE(2) JCASE(3) JCASE(4) JCASE(5) JCASE(6) JCASE(7) JCASE(8)
	JCASE(9) JCASE(10)
	default:
		ssx_set_error("%s: %d points per direction (2..10)", name, n);
		return SSX_EINVAL;
	}
#undef JCASE
	NS_LAUNCH(name);
	return SSX_OK;
}

extern "C" int ssxk_ns_curl(void *st, int nel, int n, const double *dm,
		const double *const a[3], const double *const ti[9],
		const double *mass, double *const out[3])
{
	M3 po = { { out[0], out[1], out[2] } };
	return launch_jac<false>("ssxk_ns_curl", st, nel, n, dm, a, ti, mass, 1.0,
			po);
}

extern "C" int ssxk_ns_div(void *st, int nel, int n, const double *dm,
		const double *const a[3], const double *const ti[9],
		const double *mass, double scale, double *out)
{
	M3 po = { { out, nullptr, nullptr } };
	return launch_jac<true>("ssxk_ns_div", st, nel, n, dm, a, ti, mass, scale,
			po);
}

extern "C" int ssxk_ns_grad(void *st, int nel, int n, const double *dm,
		const double *p, const double *mass, const double *const ti[9],
		double *const out[3])
{
	P9 pt;
	for (int k = 0; k < 9; ++k)
		pt.p[k] = ti[k];
	M3 po = { { out[0], out[1], out[2] } };
#define GCASE(N)                                                             \
	case N:                                                              \
		hipLaunchKernelGGL(k_ns_grad<N>, dim3((unsigned) ((nel           \
				+ JacShape<N>::E - 1) / JacShape<N>::E)), dim3(256), 0, \
				(hipStream_t) st, nel, dm, p, mass, pt, po); \
		break;
	switch (n) {
	GCASE(2) GCASE(3) GCASE(4) GCASE(5) GCASE(6) GCASE(7) GCASE(8)
	GCASE(9) GCASE(10)
	default:
		ssx_set_error("ssxk_ns_grad: %d points per direction (2..10)", n);
		return SSX_EINVAL;
	}
#undef GCASE
	NS_LAUNCH("k_ns_grad");
	return SSX_OK;
}

// geo: [nel][9][nc^3], component 3a+b w detJ d xi_b / d x_a at the nc =
// 3n/2 points; n in [2, 10]
extern "C" int ssxk_ns_conv(void *stream, int nel, int n, const double *prol,
		const double *dm, const double *const u[3], const double *const v[3],
		const double *geo, double *const out[3])
{
	hipStream_t st = (hipStream_t) stream;
	const P3 pu = { { u[0], u[1], u[2] } }, pv = { { v[0], v[1], v[2] } };
	const M3 po = { { out[0], out[1], out[2] } };
	int rc;
	switch (n) {
#define CASE(NN) case NN: rc = launch_conv<NN>(st, nel, prol, dm, pu, pv, \
			geo, po); break;
	CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10)
#undef CASE
	default:
		ssx_set_error("k_ns_conv: n = %d unsupported", n);
		return SSX_EINVAL;
	}
	if (rc != SSX_OK)
		return rc;
	NS_LAUNCH("k_ns_conv");
	return SSX_OK;
}

extern "C" int ssxk_ns_surf(void *st, int nel, int n, const int *bc,
		int dirichlet, const double *wn, const double *g, double *f)
{
	hipLaunchKernelGGL(k_ns_surf, dim3(nel), dim3(256), 0, (hipStream_t) st,
			nel, n, bc, dirichlet, wn, g, f);
	NS_LAUNCH("k_ns_surf");
	return SSX_OK;
}

extern "C" int ssxk_ns_zero_dir(void *st, size_t nt, int n, const int *bc,
		double *const u[3])
{
	M3 pu = { { u[0], u[1], u[2] } };
	hipLaunchKernelGGL(k_ns_zero_dir, dim3(ns_blocks(nt)), dim3(256), 0,
			(hipStream_t) st, (long long) nt, n, bc, pu);
	NS_LAUNCH("k_ns_zero_dir");
	return SSX_OK;
}

extern "C" int ssxk_ns_comb(void *st, size_t nt, const double *const x[3][3],
		const double a[3], const int use[3], double *const y[3])
{
	Comb cb;
	for (int t = 0; t < 3; ++t) {
		cb.a[t] = a[t];
		cb.use[t] = use[t];
		for (int c = 0; c < 3; ++c)
			cb.x[t][c] = x[t][c];
	}
	M3 py = { { y[0], y[1], y[2] } };
	hipLaunchKernelGGL(k_ns_comb, dim3(ns_blocks(nt)), dim3(256), 0,
			(hipStream_t) st, (long long) nt, cb, py);
	NS_LAUNCH("k_ns_comb");
	return SSX_OK;
}

extern "C" int ssxk_ns_mul3(void *st, size_t nt, double alpha,
		const double *const x[3], const double *const w[3], double beta,
		double *const z[3])
{
	P3 px = { { x[0], x[1], x[2] } };
	P3 pw = { { w ? w[0] : nullptr, w ? w[1] : nullptr, w ? w[2] : nullptr } };
	M3 pz = { { z[0], z[1], z[2] } };
	hipLaunchKernelGGL(k_ns_mul3, dim3(ns_blocks(nt)), dim3(256), 0,
			(hipStream_t) st, (long long) nt, alpha, px, pw, beta, pz);
	NS_LAUNCH("k_ns_mul3");
	return SSX_OK;
}

// whether the current device can run the convection operator at n points: a
// workgroup's LDS (162,512 bytes at n = 10) within its limit, and granted
extern "C" int ssxk_ns_conv_ready(int n)
{
	int dev = 0, lim = 0;
	if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&lim,
			hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) {
		ssx_set_error("k_ns_conv: no device to run on");
		return SSX_EHIP;
	}
	size_t need = 0;
	int rc = SSX_OK;
	switch (n) {
#define CASE(NN) case NN: need = ConvShape<NN, (3 * NN) / 2>::BYTES; \
		rc = need <= (size_t) lim ? conv_lds<NN>() : SSX_EHIP; break;
	CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10)
#undef CASE
	default:
		ssx_set_error("k_ns_conv: n = %d unsupported", n);
		return SSX_EINVAL;
	}
	if (need > (size_t) lim)
		ssx_set_error("k_ns_conv: n = %d needs %zu bytes of LDS, the device "
				"has %d", n, need, lim);
	return rc;
}
