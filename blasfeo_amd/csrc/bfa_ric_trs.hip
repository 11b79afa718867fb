// bfa_ric_trs.hip -- batched Riccati solve (d_back_ric_trs_libstr,
// examples/example_d_riccati_recursion.c:203-267) on the factors L[0..N] of
// the backward factorisation sweep.
//
// One wavefront per instance runs both sweeps in one launch.  With
// Lxx(k) = L[k](nu[k]:, nu[k]:) and nk = nu[k] + nx[k]:
//   backward, k = N-1 .. 0 (ux[N] = rq[N]):
//     Pb[k] = Lxx(k+1) Lxx(k+1)^T b[k]                       (trmv_ltn, trmv_lnn)
//     ux[k] = rq[k] + BAbt[k] (Pb[k] + ux[k+1](nu[k+1]:))     (gemv_n)
//     ux[k] = trsv_lnn_mn(nk, ns) of L[k] on ux[k]
//   forward, k = 0 .. N-1:
//     pi[k] = ux[k+1](nu[k+1]:)                               (the backward value)
//     ux[k](0:ns) = -ux[k](0:ns); ux[k] = trsv_ltn_mn(nk, ns) of L[k]
//     ux[k+1](nu[k+1]:) = b[k] + BAbt[k]^T ux[k]              (gemv_t)
//     pi[k] += Lxx(k+1) Lxx(k+1)^T ux[k+1](nu[k+1]:)
// where ns = nu[k] on stages k >= 1 and ns = nk on stage 0 (the reference's
// full trsv and full negation there).
//
// Work is level 2 and bound by HBM: each sweep reads every factor's lower
// triangle and every BAbt once.  Lanes own rows (gemv_n, trmv_lnn, the
// forward substitution) or columns (gemv_t, trmv_ltn); the vector a lane
// multiplies by is broadcast from LDS; the backward substitution's column
// sums are wave reductions with DPP moves.  Rows and columns go up to 128
// (two per lane).
#include "bfa_common.hpp"
#include "bfa_chol_core.hpp"
#include "bfa_internal.hpp"

namespace bfa {

constexpr int TRS_MAX = 2 * WAVE;   // largest nu+nx and nx of an instance

template <int PS>
struct PmRead
{
	const double *p;
	int cn;
	__device__ __forceinline__ double operator()(int i, int j) const
	{
		return p[(i & ~(PS - 1)) * cn + j * PS + (i & (PS - 1))];
	}
};

template <int PS>
__device__ __forceinline__ PmRead<PS> pm_read(const blasfeo_dmat &d)
{
	return PmRead<PS>{d.pA, d.cn};
}

// t(j) = sum_{i >= j} A(r0+i, r0+j) x(i), j < n   (A^T x, A lower; one column per lane)
template <int PS>
__device__ __forceinline__ void trs_trmv_t(const PmRead<PS> A, int r0, int n, const double *x, int j, double &t)
{
	double acc = 0.0;
#pragma unroll 8
	for (int i = j; i < n; i++)
		acc += A(r0 + i, r0 + j) * x[i];
	t = acc;
}

// y(i) = sum_{j <= i} A(r0+i, r0+j) t(j)   (A t, A lower; one row per lane)
template <int PS>
__device__ __forceinline__ double trs_trmv_n(const PmRead<PS> A, int r0, const double *t, int i)
{
	double acc = 0.0;
#pragma unroll 8
	for (int j = 0; j <= i; j++)
		acc += A(r0 + i, r0 + j) * t[j];
	return acc;
}

// L(i, j) for the lane's rows i = lane, lane + 64 with j < i < n0, else 0
template <int PS>
__device__ __forceinline__ void trs_coef(const PmRead<PS> L, int j, int n0, double (&e)[2])
{
	const int lane = threadIdx.x;
#pragma unroll
	for (int q = 0; q < 2; q++)
	{
		const int i = lane + q * WAVE;
		e[q] = (i > j && i < n0) ? L(i, j) : 0.0;
	}
}

// 1 / L(j, j): the cached reciprocal, or formed as the reference's trsv does
template <int PS>
__device__ __forceinline__ double trs_recip(const PmRead<PS> L, const double *dA, bool cached, int j)
{
	return cached ? dA[j] : 1.0 / L(j, j);
}

// s_x: vector broadcast to the lanes, s_t: intermediate of the trmv pairs, s_p: ux[k+1]
// of the backward sweep
template <int PS>
__device__ __forceinline__ void trs_instance(const blasfeo_amd_riccati_trs_arg &a, double *s_x, double *s_t, double *s_p)
{
	const int lane = threadIdx.x;
	const int N = a.N;
	if (N < 0)
		return;
	// an instance the on-chip vectors cannot hold is left untouched (the host
	// rejects a hint above TRS_MAX)
	for (int k = 0; k <= N; k++)
		if (a.nu[k] + a.nx[k] > TRS_MAX || a.nx[k] > TRS_MAX || a.nu[k] < 0 || a.nx[k] < 0)
			return;

	// ---- backward substitution ----
	{
		const int n = a.nu[N] + a.nx[N];
		const double *rq = a.rq[N].pa;
		double *ux = a.ux[N].pa;
		for (int i = lane; i < n; i += WAVE)
		{
			const double v = rq[i];
			ux[i] = v;
			s_p[i] = v;
		}
	}
	__syncthreads();
	for (int k = N - 1; k >= 0; k--)
	{
		const int nu0 = a.nu[k], n0 = nu0 + a.nx[k];
		const int nu1 = a.nu[k + 1], nx1 = a.nx[k + 1];
		const PmRead<PS> L1 = pm_read<PS>(a.L[k + 1]);
		const PmRead<PS> B = pm_read<PS>(a.BAbt[k]);
		const double *b = a.b[k].pa;
		const double *rq = a.rq[k].pa;
		double *Pb = a.Pb[k].pa;
		double *ux = a.ux[k].pa;

		for (int i = lane; i < nx1; i += WAVE)
			s_x[i] = b[i];
		__syncthreads();
		for (int j = lane; j < nx1; j += WAVE)
			trs_trmv_t<PS>(L1, nu1, nx1, s_x, j, s_t[j]);
		__syncthreads();
		// Pb = Lxx t; the gemv_n operand w = Pb + ux[k+1](nu1:) goes to s_x
		for (int i = lane; i < nx1; i += WAVE)
		{
			const double pb = trs_trmv_n<PS>(L1, nu1, s_t, i);
			Pb[i] = pb;
			s_x[i] = pb + s_p[nu1 + i];
		}
		__syncthreads();

		// z = rq + BAbt w, rows lane and lane + 64
		double z[2];
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int i = lane + q * WAVE;
			z[q] = 0.0;
			if (i < n0)
			{
				double acc = 0.0;
#pragma unroll 8
				for (int j = 0; j < nx1; j++)
					acc += B(i, j) * s_x[j];
				z[q] = rq[i] + acc;
			}
		}

		// forward substitution with the first ns columns of L[k] (trsv_lnn_mn):
		// z(j) *= 1/L(j,j), then every later row drops L(i,j) z(j)
		const int ns = k == 0 ? n0 : nu0;
		const blasfeo_dmat *Ld = &a.L[k];
		const PmRead<PS> L0 = pm_read<PS>(*Ld);
		double *dA = Ld->dA;
		const bool cached = Ld->use_dA == 1;
		// the column's coefficients and reciprocal are loaded one column ahead,
		// off the serial chain of v_readlane broadcasts
		double e[2] = {0.0, 0.0}, d = 0.0;
		if (ns > 0)
		{
			trs_coef<PS>(L0, 0, n0, e);
			d = trs_recip<PS>(L0, dA, cached, 0);
		}
		for (int j = 0; j < ns; j++)
		{
			double en[2] = {0.0, 0.0}, dn = 0.0;
			const bool more = j + 1 < ns;
			if (more)
			{
				trs_coef<PS>(L0, j + 1, n0, en);
				dn = trs_recip<PS>(L0, dA, cached, j + 1);
			}
			const double zj = readlane(j < WAVE ? z[0] : z[1], j & (WAVE - 1)) * d;
			if (!cached && lane == 0)
				dA[j] = d;
#pragma unroll
			for (int q = 0; q < 2; q++)
			{
				const int i = lane + q * WAVE;
				if (i == j)
					z[q] = zj;
				else if (i > j && i < n0)
					z[q] -= e[q] * zj;
			}
			if (more)
			{
				e[0] = en[0];
				e[1] = en[1];
				d = dn;
			}
		}
		if (!cached && ns > 0 && n0 > 0 && lane == 0)
			a.L[k].use_dA = 1;
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int i = lane + q * WAVE;
			if (i < n0)
			{
				ux[i] = z[q];
				s_p[i] = z[q];
			}
		}
		__syncthreads();
	}

	// ---- forward substitution ----
	for (int k = 0; k < N; k++)
	{
		const int nu0 = a.nu[k], n0 = nu0 + a.nx[k];
		const int nu1 = a.nu[k + 1], nx1 = a.nx[k + 1];
		const PmRead<PS> L1 = pm_read<PS>(a.L[k + 1]);
		const PmRead<PS> B = pm_read<PS>(a.BAbt[k]);
		const double *b = a.b[k].pa;
		double *ux0 = a.ux[k].pa;
		double *ux1 = a.ux[k + 1].pa;
		double *pi = a.pi[k].pa;
		const int ns = k == 0 ? n0 : nu0;

		double pio[2], z[2];
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int i = lane + q * WAVE;
			pio[q] = i < nx1 ? ux1[nu1 + i] : 0.0;
			z[q] = i < n0 ? ux0[i] : 0.0;
			if (i < ns)
				z[q] = -z[q];
		}

		// backward substitution with the first ns columns of L[k] (trsv_ltn_mn):
		// z(j) = (z(j) - sum_{i > j} L(i,j) z(i)) / L(j,j), j = ns-1 .. 0
		const blasfeo_dmat *Ld = &a.L[k];
		const PmRead<PS> L0 = pm_read<PS>(*Ld);
		double *dA = Ld->dA;
		const bool cached = Ld->use_dA == 1;
		double e[2] = {0.0, 0.0}, d = 0.0;
		if (ns > 0)
		{
			trs_coef<PS>(L0, ns - 1, n0, e);
			d = trs_recip<PS>(L0, dA, cached, ns - 1);
		}
		for (int j = ns - 1; j >= 0; j--)
		{
			double en[2] = {0.0, 0.0}, dn = 0.0;
			const bool more = j > 0;
			if (more)
			{
				trs_coef<PS>(L0, j - 1, n0, en);
				dn = trs_recip<PS>(L0, dA, cached, j - 1);
			}
			// only rows j+1 .. n0-1 contribute (e is zero elsewhere, but a zero
			// coefficient times an Inf or NaN in an unsolved row is NaN)
			const int i0 = lane, i1 = lane + WAVE;
			const double part = (i0 > j && i0 < n0 ? e[0] * z[0] : 0.0) + (i1 > j && i1 < n0 ? e[1] * z[1] : 0.0);
			const double s = readlane(wave_sum_d(part), WAVE - 1);
			if (!cached && lane == 0)
				dA[j] = d;
#pragma unroll
			for (int q = 0; q < 2; q++)
				if (lane + q * WAVE == j)
					z[q] = (z[q] - s) * d;
			if (more)
			{
				e[0] = en[0];
				e[1] = en[1];
				d = dn;
			}
		}
		if (!cached && n0 > 0 && lane == 0)
			a.L[k].use_dA = 1;
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int i = lane + q * WAVE;
			if (i < n0)
			{
				ux0[i] = z[q];
				s_x[i] = z[q];
			}
		}
		__syncthreads();

		// x(k+1) = b + BAbt^T z (gemv_t), one column per lane
		for (int j = lane; j < nx1; j += WAVE)
		{
			double acc = 0.0;
#pragma unroll 8
			for (int i = 0; i < n0; i++)
				acc += B(i, j) * s_x[i];
			const double y = b[j] + acc;
			ux1[nu1 + j] = y;
			s_p[j] = y;
		}
		__syncthreads();
		for (int j = lane; j < nx1; j += WAVE)
			trs_trmv_t<PS>(L1, nu1, nx1, s_p, j, s_t[j]);
		__syncthreads();
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int i = lane + q * WAVE;
			if (i < nx1)
				pi[i] = pio[q] + trs_trmv_n<PS>(L1, nu1, s_t, i);
		}
		__syncthreads();
	}
}

template <int PS>
__global__ __launch_bounds__(WAVE) void k_ric_trs(const blasfeo_amd_riccati_trs_arg *__restrict__ args, int batch)
{
	__shared__ double s_x[TRS_MAX], s_t[TRS_MAX], s_p[TRS_MAX];
	const int inst = blockIdx.x;
	if (inst >= batch)
		return;
	const blasfeo_amd_riccati_trs_arg a = args[inst];
	trs_instance<PS>(a, s_x, s_t, s_p);
}

// ---------------------------------------------------------------------------
// Instances whose stages have at most TRS_SMALL rows and columns, one wavefront
// each: a chain of short steps, bound by the latency of memory when every step
// fetches its own operands (descriptors, then matrices, a column at a time).
// Here a stage's descriptors are read two stages ahead and its matrices and
// vectors one stage ahead, into registers, and a step works on LDS copies (L
// of two stages, BAbt of one).  The forward sweep's substitution drops the
// solved entries from all earlier ones (one broadcast a column) instead of a
// wave sum a column.
// Measured (MI355X; factorisation and solve, before and now): one system of nx = 8,
// nu = 3, N = 10 115 -> 78 us, of nx, nu up to 24, 6, N = 15 282 -> 248, 2048 of nx = 8
// 203 -> 120, 1024 of nx = 8..24, N = 30 846 -> 559.  A step takes 5000 cycles, most of
// it the chain of LDS exchanges between its products.
// ---------------------------------------------------------------------------
constexpr int TRS_SMALL = 32;

// What stage k of an instance holds
struct TrsStage
{
	int nu, nx;           // (scalars once trs_sizes has run)
	int n;                // nu + nx
	const BFA_GLOBAL double *L, *B;
	int Lcn, Bcn, use;    // use: the reciprocals in dA are valid
	BFA_GLOBAL double *dA;
	const BFA_GLOBAL double *b, *rq;
	BFA_GLOBAL double *Pb, *ux, *pi;
};

// (through global-memory pointers: a wait for LDS would also wait for flat loads, and
// with it for the stages ahead)
__device__ __forceinline__ TrsStage trs_stage(const blasfeo_amd_riccati_trs_arg &a, int k)
{
	typedef const BFA_GLOBAL blasfeo_dmat *mat;
	typedef const BFA_GLOBAL blasfeo_dvec *vec;
	typedef BFA_GLOBAL double *out;
	TrsStage s;
	s.nu = ((const BFA_GLOBAL int *)a.nu)[k];
	s.nx = ((const BFA_GLOBAL int *)a.nx)[k];
	s.n = 0;
	mat L = (mat)a.L + k;
	s.L = (out)L->pA;
	s.Lcn = L->cn;
	s.use = L->use_dA;
	s.dA = (out)L->dA;
	s.rq = (out)((vec)a.rq)[k].pa;
	s.ux = (out)((vec)a.ux)[k].pa;
	s.B = nullptr, s.b = nullptr, s.Pb = nullptr, s.pi = nullptr;
	s.Bcn = 0;
	if (k < a.N)
	{
		s.B = (out)((mat)a.BAbt)[k].pA;
		s.Bcn = ((mat)a.BAbt)[k].cn;
		s.b = (out)((vec)a.b)[k].pa;
		s.Pb = (out)((vec)a.Pb)[k].pa;
		s.pi = (out)((vec)a.pi)[k].pa;
	}
	return s;
}

// the sizes to scalar registers: waits for the loads, so not where they are issued
__device__ __forceinline__ void trs_sizes(TrsStage &s)
{
	s.nu = __builtin_amdgcn_readfirstlane(s.nu);
	s.n = s.nu + __builtin_amdgcn_readfirstlane(s.nx);
}

// A matrix of m x n (both at most MX) in registers and in LDS (leading dimension
// MX + 1): row lane % MX, columns (64 / MX) t + lane / MX; rows and columns past the
// end repeat the last one, so that neither loads nor stores need a mask.
template <int MX> constexpr int trs_regs() { return MX * MX / WAVE; }
template <int PS, int MX>
__device__ __forceinline__ void trs_fetch(const BFA_GLOBAL double *p, int cn, int m, int n, double (&v)[trs_regs<MX>()])
{
	const int h = threadIdx.x / MX, i = min((int)threadIdx.x % MX, m - 1);
	p += (size_t)(i & ~(PS - 1)) * cn + (i & (PS - 1));
#pragma unroll
	for (int t = 0; t < trs_regs<MX>(); t++)
		v[t] = p[min(WAVE / MX * t + h, n - 1) * PS];
}
template <int MX>
__device__ __forceinline__ void trs_put(double *lds, const double (&v)[trs_regs<MX>()])
{
#pragma unroll
	for (int t = 0; t < trs_regs<MX>(); t++)
		lds[(WAVE / MX * t + threadIdx.x / MX) * (MX + 1) + threadIdx.x % MX] = v[t];
}

// sum over i < n of A(i) x(i), i from `from` on for this lane (to `to`): eight
// elements of LDS at a time, from p + i st and x + i
__device__ __forceinline__ double trs_dot(const double *p, int st, const double *x, int n, int from, int to)
{
	double acc = 0.0;
	for (int i0 = 0; i0 < n; i0 += 8)
	{
		double v[8], y[8];
#pragma unroll
		for (int u = 0; u < 8; u++)
		{
			const int i = min(i0 + u, n - 1);
			v[u] = p[i * st];
			y[u] = x[i];
		}
#pragma unroll
		for (int u = 0; u < 8; u++)
			if (i0 + u >= from && i0 + u < to)
				acc += v[u] * y[u];
	}
	return acc;
}
// this lane's element of A^T x (A lower n x n at p, leading dimension ld; lane < n)
__device__ __forceinline__ double trs_lt(const double *p, int ld, int n, const double *x)
{
	const int j = min((int)threadIdx.x, n - 1);
	return trs_dot(p + j * ld, 1, x, n, j, n);
}
// this lane's element of A t (lane < n)
__device__ __forceinline__ double trs_ln(const double *p, int ld, int n, const double *t)
{
	const int i = min((int)threadIdx.x, n - 1);
	return trs_dot(p + i, ld, t, n, 0, i + 1);
}

template <int PS, int MX>
__global__ __launch_bounds__(WAVE) void k_ric_trs_small(const blasfeo_amd_riccati_trs_arg *__restrict__ args, int batch, int most)
{
	constexpr int ld = MX + 1;
	__shared__ double Lb[2 * MX * ld], Bb[MX * ld];   // L of even and of odd stages, BAbt
	__shared__ double s_x[TRS_MAX], s_t[TRS_MAX], s_p[TRS_MAX];
	const int inst = blockIdx.x, lane = threadIdx.x;
	if (inst >= batch)
		return;
	const blasfeo_amd_riccati_trs_arg a = args[inst];
	const int N = __builtin_amdgcn_readfirstlane(a.N);
	if (N < 0)
		return;
	bool fits = true;
	for (int k = lane; k <= N; k += WAVE)
		fits = fits && a.nu[k] >= 0 && a.nx[k] >= 0 && a.nu[k] + a.nx[k] <= most;
	if (__ballot(!fits))
		return trs_instance<PS>(a, s_x, s_t, s_p);   // larger than the bound says
	auto Ls = [&](int k) { return Lb + (k & 1) * ld * MX; };

	// ---- backward substitution ----
	double dl[trs_regs<MX>()], db[trs_regs<MX>()], vb = 0.0, vr = 0.0, vd = 0.0, z = 0.0;
	// S0: the stage at hand, S1: the one after it in time, SP and SQ: those before
	TrsStage S1 = trs_stage(a, N), S0 = trs_stage(a, max(N - 1, 0)), SP = trs_stage(a, max(N - 2, 0)), SQ;
	trs_sizes(S1);
	trs_sizes(S0);
	auto fetch_back = [&](const TrsStage &s, int n1) {
		if (s.n > 0)
		{
			trs_fetch<PS, MX>(s.L, s.Lcn, s.n, s.n, dl);
			vr = s.rq[min(lane, s.n - 1)];
			vd = s.use == 1 ? s.dA[min(lane, s.n - 1)] : 0.0;
			if (n1 > 0)
				trs_fetch<PS, MX>(s.B, s.Bcn, s.n, n1, db);
		}
		if (n1 > 0)
			vb = s.b[min(lane, n1 - 1)];
	};
	if (S1.n > 0)
	{
		trs_fetch<PS, MX>(S1.L, S1.Lcn, S1.n, S1.n, dl);
		z = lane < S1.n ? S1.rq[lane] : 0.0;
		trs_put<MX>(Ls(N), dl);
	}
	if (N > 0)
		fetch_back(S0, S1.n - S1.nu);
	// A step's results are stored a step later, ahead of the next loads: every load
	// and store has a step's time before the next wait, which cannot tell them apart.
	double pb = 0.0;
	int npb = 0;          // of Pb[k+1]
	for (int k = N - 1; k >= 0; k--)
	{
		const int n0 = S0.n, nu0 = S0.nu, nu1 = S1.nu, nx1 = S1.n - S1.nu;
		trs_sizes(SP);
		// this stage's operands to LDS and registers, the one before's on their way
		wave_sync();
		if (lane < S1.n)
			s_p[lane] = z;   // ux[k+1]
		if (n0 > 0)
		{
			trs_put<MX>(Ls(k), dl);
			if (nx1 > 0)
				trs_put<MX>(Bb, db);
		}
		if (lane < nx1)
			s_x[lane] = vb;
		const double r0 = vr, dA0 = vd;
		wave_sync();
		if (lane < S1.n)
			S1.ux[lane] = z;
		if (lane < npb)
			S1.Pb[lane] = pb;
		SQ = trs_stage(a, max(k - 2, 0));
		if (k > 0)
			fetch_back(SP, n0 - nu0);
		const double *L1 = Ls(k + 1) + nu1 * ld + nu1, *L0 = Ls(k);
		if (lane < nx1)
			s_t[lane] = trs_lt(L1, ld, nx1, s_x);
		wave_sync();
		// Pb = Lxx t; w = Pb + ux[k+1](nu1:)
		if (lane < nx1)
		{
			pb = trs_ln(L1, ld, nx1, s_t);
			s_x[lane] = pb + s_p[nu1 + lane];
		}
		wave_sync();
		z = 0.0;
		if (lane < n0)
		{
			z = r0 + trs_dot(Bb + lane, ld, s_x, nx1, 0, nx1);
		}
		// forward substitution with the first ns columns (trsv_lnn_mn)
		const int ns = k == 0 ? n0 : nu0;
		const bool cached = S0.use == 1;
		const double rd = cached ? dA0 : lane < n0 ? 1.0 / L0[lane * ld + lane] : 0.0;
		if (!cached && ns > 0)
		{
			if (lane < ns)
				S0.dA[lane] = rd;
			if (lane == 0)
				((BFA_GLOBAL blasfeo_dmat *)a.L)[k].use_dA = 1;
		}
		for (int j0 = 0; j0 < ns; j0 += 4)
		{
			double e[4];
#pragma unroll
			for (int u = 0; u < 4; u++)
				e[u] = L0[min(j0 + u, ns - 1) * ld + min(lane, MX - 1)];
#pragma unroll
			for (int u = 0; u < 4; u++)
				if (j0 + u < ns)
				{
					const int j = j0 + u;
					const double zj = readlane(z, j) * readlane(rd, j);
					z = lane == j ? zj : lane > j && lane < n0 ? z - e[u] * zj : z;
				}
		}
		npb = nx1;
		S1 = S0;
		S0 = SP;
		SP = SQ;
	}
	if (N > 0 && lane < npb)
		S1.Pb[lane] = pb;
	if (N == 0)
	{
		if (lane < S1.n)
			S1.ux[lane] = z;
		return;
	}

	// ---- forward substitution: z = ux[0] and L[0], L[1], BAbt[0] are on chip ----
	// S0, S1: the stage at hand and the next, SP and SQ: those after
	S0 = S1;
	S1 = trs_stage(a, 1);
	SP = trs_stage(a, min(2, N));
	trs_sizes(S1);
	double vu = 0.0, vp = 0.0, xu = 0.0;
	// operands of the step from stage s to s1 (BAbt[0] and L[1] are there)
	auto fetch_fwd = [&](const TrsStage &s, const TrsStage &s1, bool mats) {
		const int nx1 = s1.n - s1.nu;
		if (s.n > 0)
			vd = s.use == 1 ? s.dA[min(lane, s.n - 1)] : 0.0;
		if (s1.n > 0)
		{
			if (mats)
				trs_fetch<PS, MX>(s1.L, s1.Lcn, s1.n, s1.n, dl);
			vu = s1.ux[min(lane, s1.n - 1)];
			if (nx1 > 0)
			{
				vp = s1.ux[s1.nu + min(lane, nx1 - 1)];
				vb = s.b[min(lane, nx1 - 1)];
				if (mats && s.n > 0)
					trs_fetch<PS, MX>(s.B, s.Bcn, s.n, nx1, db);
			}
		}
	};
	// stage 0's reciprocals were formed or read by the backward sweep's last step
	S0.use = S0.n > 0 ? ((const BFA_GLOBAL blasfeo_dmat *)a.L)[0].use_dA : 0;
	fetch_fwd(S0, S1, false);
	double pv = 0.0, zv = 0.0;   // pi and ux of the step before
	int npi = 0, nux = 0;
	BFA_GLOBAL double *ppi = nullptr, *pux = nullptr;
	for (int k = 0; k < N; k++)
	{
		const int n0 = S0.n, nu0 = S0.nu, nu1 = S1.nu, nx1 = S1.n - S1.nu;
		const int ns = k == 0 ? n0 : nu0;
		trs_sizes(SP);
		wave_sync();
		if (k > 0)
		{
			if (S1.n > 0)
				trs_put<MX>(Ls(k + 1), dl);
			if (n0 > 0 && nx1 > 0)
				trs_put<MX>(Bb, db);
			// ux[k]: the inputs of the backward sweep, the state of the step before
			z = lane < nu0 ? xu : lane < n0 ? s_p[lane - nu0] : 0.0;
		}
		const double pio = vp, b0 = vb, dA0 = vd;
		xu = vu;
		if (lane < ns)
			z = -z;
		wave_sync();
		s_x[lane] = lane < n0 ? z : 0.0;
		if (lane < nux)
			pux[lane] = zv;
		if (lane < npi)
			ppi[lane] = pv;
		SQ = trs_stage(a, min(k + 3, N));
		if (k + 1 < N)
			fetch_fwd(S1, SP, true);
		wave_sync();
		// backward substitution with the first ns columns (trsv_ltn_mn): the rows
		// from ns on first, then each solved entry out of all earlier ones
		const double *L0 = Ls(k), *L1 = Ls(k + 1) + nu1 * ld + nu1;
		const bool cached = S0.use == 1;
		const double rd = cached ? dA0 : lane < n0 ? 1.0 / L0[lane * ld + lane] : 0.0;
		if (!cached && n0 > 0)
		{
			if (lane < ns)
				S0.dA[lane] = rd;
			if (lane == 0)
				((BFA_GLOBAL blasfeo_dmat *)a.L)[k].use_dA = 1;
		}
		if (ns > 0)
		{
			if (lane < ns && ns < n0)
				z -= trs_dot(L0 + lane * ld + ns, 1, s_x + ns, n0 - ns, 0, n0 - ns);
			for (int j0 = ns - 1; j0 >= 0; j0 -= 4)
			{
				double e[4];
#pragma unroll
				for (int u = 0; u < 4; u++)
					e[u] = L0[min(lane, MX - 1) * ld + max(j0 - u, 0)];
#pragma unroll
				for (int u = 0; u < 4; u++)
					if (j0 - u >= 0)
					{
						const int j = j0 - u;
						const double zj = readlane(z, j) * readlane(rd, j);
						z = lane == j ? zj : lane < j ? z - e[u] * zj : z;
					}
			}
		}
		wave_sync();
		if (lane < n0)
			s_x[lane] = z;
		zv = z, nux = n0, pux = S0.ux;
		wave_sync();
		// x(k+1): the next step's state, stored with its ux = b + BAbt^T z
		if (lane < nx1)
		{
			const double y = b0 + trs_dot(Bb + lane * ld, 1, s_x, n0, 0, n0);
			if (k + 1 == N)
				S1.ux[nu1 + lane] = y;
			s_p[lane] = y;
		}
		wave_sync();
		if (lane < nx1)
			s_t[lane] = trs_lt(L1, ld, nx1, s_p);
		wave_sync();
		if (lane < nx1)
			pv = pio + trs_ln(L1, ld, nx1, s_t);
		npi = nx1, ppi = S0.pi;
		S0 = S1;
		S1 = SP;
		SP = SQ;
	}
	if (lane < nux)
		pux[lane] = zv;
	if (lane < npi)
		ppi[lane] = pv;
}

template <int PS>
static int launch_trs(int batch, const blasfeo_amd_riccati_trs_arg *args, int most, hipStream_t st, const char *name)
{
	// above 16 rows LDS leaves five instances per CU: for batches of up to 16 per CU
	// (2048 of nx = 20..24 588 against 591 us, 8192 of nx = 4..24 1026 against 983)
	const int cus = num_cus() > 0 ? num_cus() : 256;
	if (most <= 16 || (most <= TRS_SMALL && batch <= 16 * cus))
	{
		if (most <= 16)
			hipLaunchKernelGGL((k_ric_trs_small<PS, 16>), dim3(batch), dim3(WAVE), 0, st, args, batch, most);
		else
			hipLaunchKernelGGL((k_ric_trs_small<PS, 32>), dim3(batch), dim3(WAVE), 0, st, args, batch, most);
		return check_launch(name);
	}
	hipLaunchKernelGGL(k_ric_trs<PS>, dim3(batch), dim3(WAVE), 0, st, args, batch);
	return check_launch(name);
}

} // namespace bfa

using namespace bfa;

extern "C" int blasfeo_amd_d_back_ric_trs_batched(int ps, int batch, const blasfeo_amd_riccati_trs_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t stream)
{
	const char *name = "blasfeo_amd_d_back_ric_trs_batched";
	if (batch < 0)
		return set_error(BLASFEO_AMD_EINVAL, "%s: batch=%d < 0", name, batch);
	if (batch == 0)
		return BLASFEO_AMD_OK;
	if (!args)
		return set_error(BLASFEO_AMD_EINVAL, "%s: args is NULL", name);
	if (ps != 4 && ps != 8)
		return set_error(BLASFEO_AMD_EINVAL, "%s: unsupported panel size %d", name, ps);
	if (!hint || hint->max_m <= 0)
		return set_error(BLASFEO_AMD_EINVAL, "%s: hint->max_m (largest nu[k]+nx[k]) is required", name);
	const int nxmax = hint->max_n > 0 ? hint->max_n : hint->max_m;
	if (hint->max_m > TRS_MAX || nxmax > TRS_MAX)
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: nu+nx and nx up to %d supported, got %d and %d",
		                 name, TRS_MAX, hint->max_m, nxmax);
	hipStream_t st = (hipStream_t)stream;
	const int most = hint->max_m > nxmax ? hint->max_m : nxmax;
	return ps == 4 ? launch_trs<4>(batch, args, most, st, name) : launch_trs<8>(batch, args, most, st, name);
}
