// bfa_lapack.hip -- batched factorisations for gfx950: potrf_l, potrf_l_mn,
// syrk_dpotrf_ln(_mn) and getrf_rp on panel-major matrices.
//
// potrf and syrk_dpotrf up to 256 columns: 16-row strips in registers
// (bfa_potrf_wave.hpp), getrf up to 256 rows: bfa_getrf_wg.hpp.  Above: one workgroup
// (4 waves) per instance, left-looking over 16-column panels held in LDS at full
// height (the role of the reference's 12x4 / 8x8 register blocks,
// blasfeo_hp_pm/d_lapack_lib4.c:954-985 and :2443-2634):
//   potrf: panel <- C - L(:,0:c0) L(c0:c0+16,0:c0)^T on the matrix
//          cores, then one wave factors the top 64 rows in registers (the
//          diagonal 16x16 Cholesky, broadcasting L(jj,j) with v_readlane) and
//          all waves solve the remaining rows against it;
//   getrf: panel <- rows gathered through the current row permutation, the
//          previous unit-lower panels applied block by block (unit solve of
//          the 16-row block, matrix-core update of the rows below), then one
//          wave factors the panel column by column with a wave-wide argmax
//          for the pivot (first index of the largest |x|, as idamax and
//          blasfeo_ref/x_lapack_ref.c:1275-1302), and the panel's swaps are
//          applied to the finished columns on the left.
#include "bfa_chol_core.hpp"
#include "bfa_internal.hpp"

namespace bfa {

template <typename T> struct FactArg;
template <> struct FactArg<double> { typedef blasfeo_amd_dfact_arg type; };
template <> struct FactArg<float> { typedef blasfeo_amd_sfact_arg type; };

template <typename T> struct SPArg;
template <> struct SPArg<double> { typedef blasfeo_amd_dsyrk_dpotrf_arg type; };

} // namespace bfa
#include "bfa_potrf_wave.hpp"
namespace bfa {

// potrf_l for n > 256: left-looking over 16-column LDS panels at full height,
// the earlier panels read back from D (chol_instance)
template <typename T, int PS>
__global__ __launch_bounds__(NTL) void k_potrf(const typename FactArg<T>::type *__restrict__ args, int mmax)
{
	extern __shared__ unsigned char smem_raw[];
	__shared__ T L11[PW * (PW + 1)];
	__shared__ T invs[PW];
	T *P = reinterpret_cast<T *>(smem_raw);
	const typename FactArg<T>::type &a = args[blockIdx.x];
	const int m = a.m;
	if (m <= 0 || m > mmax)
		return;
	const int LDP = (mmax + 15) / 16 * 16 + 1;
	PM<T, PS> gD = view<T, PS>(a.sD);
	chol_instance<T, PS>(P, LDP, L11, invs, m, m, 0, gD, 0, 0, gD, 0, 0,
		view<T, PS>(a.sC), a.ci, a.cj, gD, a.di, a.dj, a.sD->dA);
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? m : 0;
}

// ---------------------------------------------------------------------------
// LU with partial row pivoting (blasfeo_ref/x_lapack_ref.c:1156-1536 semantics);
// PIV = false: LU without pivoting, getrf_np (x_lapack_ref.c:880-1150): no
// pivot search, no swaps, ipiv not touched, and dA = 1/U(j,j) with no guard
// for a zero pivot (the reference divides unconditionally)
// ---------------------------------------------------------------------------
// Launch order: the plan kernel sorts the instances into buckets of 16 rows
// of max(m, n), largest first, and workgroup b of the launch takes the b-th
// instance of that order (counts/lists == nullptr: the input order), so the
// largest instances start first and the launch does not end on one of them
// running alone.
constexpr int GETRF_NB = 16;
template <typename T>
__global__ void k_getrf_plan(const typename FactArg<T>::type *__restrict__ args, int batch, int *counts, int *lists)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	int b = -1;
	if (i < batch)
	{
		const int s = max(args[i].m, args[i].n);
		b = s <= 0 ? GETRF_NB - 1 : max(0, GETRF_NB - 1 - (s - 1) / 16);
	}
	plan_bucket<GETRF_NB>(i, b, batch, counts, lists);
}

__global__ void k_zero_ints(int *p, int n)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		p[i] = 0;
}

__device__ __forceinline__ int getrf_order(int t, int batch, const int *counts, const int *lists)
{
	if (!counts)
		return t;
	for (int b = 0; b < GETRF_NB; b++)
	{
		const int c = counts[b];
		if (t < c)
			return lists[(size_t)b * batch + t];
		t -= c;
	}
	return -1;
}

} // namespace bfa
#include "bfa_getrf_wg.hpp"
namespace bfa {

// instances of more than 256 rows
template <typename T, int PS, bool PIV = true>
__global__ __launch_bounds__(NTL) __attribute__((amdgpu_waves_per_eu(4))) void k_getrf(const typename FactArg<T>::type *__restrict__ args, int mmax,
	int batch = 0, const int *__restrict__ counts = nullptr, const int *__restrict__ lists = nullptr)
{
	typedef typename Vec4<T>::type V4;
	extern __shared__ unsigned char smem_raw[];
	__shared__ T invs[PW];
	__shared__ int pivs[PW];
	__shared__ T Lb[16 * 17];   // the unit-lower block L(r0:r0+16, r0:r0+16) of the solve
	__shared__ T wbest[NTL / WAVE];   // per-wave pivot candidates
	__shared__ int widx[NTL / WAVE];
	const int LDP = (mmax + 15) / 16 * 16 + 1;
	T *P = reinterpret_cast<T *>(smem_raw);                              // [PW][LDP]
	int *perm = reinterpret_cast<int *>(smem_raw + sizeof(T) * PW * LDP);  // [mmax]

	const int inst = getrf_order(blockIdx.x, batch, counts, lists);
	if (inst < 0)
		return;
	const typename FactArg<T>::type &a = args[inst];
	const int m = a.m, n = a.n;
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? 1 : 0;
	if (m <= 0 || n <= 0 || m > mmax)
		return;
	const PM<T, PS> gC = view<T, PS>(a.sC);
	PM<T, PS> gD = view<T, PS>(a.sD);
	const int ci = a.ci, cj = a.cj, di = a.di, dj = a.dj;
	T *dD = a.sD->dA;
	int *ipiv = a.ipiv;
	const int p = min(m, n);
	const int lane = lane_id();
	const int w = wave_id();
	const int mt = (m + 15) / 16;

	for (int i = threadIdx.x; i < m; i += NTL)
		perm[i] = i;

	for (int c0 = 0; c0 < n; c0 += PW)
	{
		const int cw = min(PW, n - c0);
		__syncthreads();
		// gather the panel through the current row permutation, eight
		// elements per thread at a time (all loads issued before the stores)
		for (int e0 = threadIdx.x; e0 < PW * mt * 16; e0 += 8 * NTL)
		{
			T v[8];
#pragma unroll
			for (int u = 0; u < 8; u++)
			{
				const int e = e0 + u * NTL;
				const int c = e / (mt * 16);
				const int i = e - c * (mt * 16);
				v[u] = (e < PW * mt * 16 && i < m && c < cw) ? gC.at(ci + perm[i], cj + c0 + c) : T(0);
			}
#pragma unroll
			for (int u = 0; u < 8; u++)
			{
				const int e = e0 + u * NTL;
				const int c = e / (mt * 16);
				const int i = e - c * (mt * 16);
				if (e < PW * mt * 16)
					P[c * LDP + i] = v[u];
			}
		}
		// apply the finished unit-lower panels, 16 rows at a time
		const int rbmax = min(c0, p);
		for (int r0 = 0; r0 < rbmax; r0 += 16)
		{
			const int rh = min(16, rbmax - r0);
			// stage the strictly lower part of L(r0:r0+rh, r0:r0+rh), one
			// element per thread, so that the solve reads it from LDS
			if (threadIdx.x < 256)
			{
				const int r = threadIdx.x >> 4, l = threadIdx.x & 15;
				if (l < r && r < rh)
					Lb[r * 17 + l] = gD.at(di + r0 + r, dj + r0 + l);
			}
			__syncthreads();
			// unit-lower solve of rows r0..r0+rh: one lane per panel column
			if (w == 0 && lane < cw)
			{
				T x[16];
#pragma unroll
				for (int r = 0; r < 16; r++)
					x[r] = P[lane * LDP + r0 + r];
#pragma unroll
				for (int r = 1; r < 16; r++)
				{
					if (r < rh)
					{
						T c = x[r];
#pragma unroll
						for (int l = 0; l < r; l++)
							c -= Lb[r * 17 + l] * x[l];
						x[r] = c;
					}
				}
#pragma unroll
				for (int r = 0; r < 16; r++)
					P[lane * LDP + r0 + r] = x[r];
			}
			__syncthreads();
			// rows below: P(r0+16.., :) -= L(r0+16.., r0:r0+16) * P(r0:r0+16, :)
			const int rs = r0 + 16;
			const int ntile = (m - rs + 15) / 16;
			// the right operand (the solved rows r0..r0+16) is the same for
			// every tile: read once
			T bv[4];
#pragma unroll
			for (int u = 0; u < 4; u++)
			{
				const int kq = 4 * u + (lane >> 4);
				bv[u] = kq < rh ? P[(lane & 15) * LDP + r0 + kq] : T(0);
			}
			// up to four of the wave's row tiles at a time: all their loads
			// are issued before any product
			for (int rt0 = w; rt0 < ntile; rt0 += 4 * (NTL / WAVE))
			{
				T av[4][4];
#pragma unroll
				for (int t = 0; t < 4; t++)
				{
					const int rt = rt0 + t * (NTL / WAVE);
					const int ir = rs + rt * 16 + (lane & 15);
					const bool iok = rt < ntile && ir < m;
#pragma unroll
					for (int u = 0; u < 4; u++)
					{
						const int kq = 4 * u + (lane >> 4);
						av[t][u] = (iok && kq < rh) ? gD.at(di + ir, dj + r0 + kq) : T(0);
					}
				}
#pragma unroll
				for (int t = 0; t < 4; t++)
				{
					const int rt = rt0 + t * (NTL / WAVE);
					if (rt >= ntile)
						break;
					V4 acc = V4{0, 0, 0, 0};
#pragma unroll
					for (int u = 0; u < 4; u++)
						acc = mfma16(av[t][u], bv[u], acc);
#pragma unroll
					for (int r = 0; r < 4; r++)
					{
						const int il = rs + rt * 16 + acc_row<T>(lane, r);
						P[(lane & 15) * LDP + il] -= acc[r];
					}
				}
			}
		}
		__syncthreads();
		// factor the panel rows c0..m-1 (only columns that have a pivot row)
		const int cf = min(cw, p - c0);
		if (cf > 0 && m - c0 > WAVE)
		{
			// all waves, rows striped over the threads: per column a wave
			// argmax, the waves' winners combined through LDS (the same
			// total order, so the same pivot), the swap, then the rank-1
			// update of the rows below; three barriers per column
			for (int j = 0; j < cf; j++)
			{
				const int jr = c0 + j;
				int ip = jr;
				if (PIV)
				{
				T best = T(0);
				int bi = jr;
				for (int i = jr + threadIdx.x; i < m; i += NTL)
				{
					const T v = P[j * LDP + i];
					const T av = v > T(0) ? v : -v;
					if (av > best)
					{
						best = av;
						bi = i;
					}
				}
				wave_argmax_abs_to_last<T>(best, bi);
				if (lane == WAVE - 1)
				{
					wbest[w] = best;
					widx[w] = bi;
				}
				__syncthreads();
				T b = wbest[0];
				ip = widx[0];
				for (int ww = 1; ww < NTL / WAVE; ww++)
					if (wbest[ww] > b || (wbest[ww] == b && widx[ww] < ip))
					{
						b = wbest[ww];
						ip = widx[ww];
					}
				if (threadIdx.x == 0)
					pivs[j] = ip;
				}
				if (PIV && ip != jr)
				{
					if (threadIdx.x < PW)
					{
						const T t0 = P[threadIdx.x * LDP + jr];
						P[threadIdx.x * LDP + jr] = P[threadIdx.x * LDP + ip];
						P[threadIdx.x * LDP + ip] = t0;
					}
					if (threadIdx.x == 0)
					{
						const int t1 = perm[jr];
						perm[jr] = perm[ip];
						perm[ip] = t1;
					}
				}
				__syncthreads();
				const T piv = P[j * LDP + jr];
				const T inv = PIV ? (piv != T(0) ? T(1) / piv : T(0)) : T(1) / piv;
				if (threadIdx.x == 0)
					invs[j] = inv;
				for (int i = jr + 1 + threadIdx.x; i < m; i += NTL)
				{
					const T l = P[j * LDP + i] * inv;
					P[j * LDP + i] = l;
					for (int jj = j + 1; jj < cw; jj++)
						P[jj * LDP + i] -= l * P[jj * LDP + jr];
				}
				__syncthreads();
			}
		}
		else if (w == 0 && cf > 0)
		{
			for (int j = 0; j < cf; j++)
			{
				const int jr = c0 + j;
				int ip = jr;
				if (PIV)
				{
				// pivot: first row of largest |x| among jr..m-1, from (0, jr)
				T best = T(0);
				int bi = jr;
				for (int i = jr + lane; i < m; i += WAVE)
				{
					const T v = P[j * LDP + i];
					const T av = v > T(0) ? v : -v;
					if (av > best)
					{
						best = av;
						bi = i;
					}
				}
				ip = wave_argmax_abs<T>(best, bi);
				if (lane == 0)
					pivs[j] = ip;
				}
				if (PIV && ip != jr)
				{
					if (lane < PW)
					{
						const T t0 = P[lane * LDP + jr];
						P[lane * LDP + jr] = P[lane * LDP + ip];
						P[lane * LDP + ip] = t0;
					}
					if (lane == 0)
					{
						const int t1 = perm[jr];
						perm[jr] = perm[ip];
						perm[ip] = t1;
					}
				}
				wave_sync();
				const T piv = P[j * LDP + jr];
				const T inv = PIV ? (piv != T(0) ? T(1) / piv : T(0)) : T(1) / piv;
				if (lane == 0)
					invs[j] = inv;
				for (int i = jr + 1 + lane; i < m; i += WAVE)
				{
					const T l = P[j * LDP + i] * inv;
					P[j * LDP + i] = l;
					for (int jj = j + 1; jj < cw; jj++)
						P[jj * LDP + i] -= l * P[jj * LDP + jr];
				}
				wave_sync();
			}
		}
		__syncthreads();
		// write the panel (all rows, current order) and its pivot data
		s2g<T, PS, NTL, false>(gD, di, dj + c0, m, cw, P, LDP, 0);
		for (int j = threadIdx.x; j < cf; j += NTL)
		{
			if (PIV)
				ipiv[c0 + j] = pivs[j];
			dD[c0 + j] = invs[j];
		}
		__syncthreads();
		// this panel's swaps on the finished columns 0..c0-1 (one thread per column)
		for (int c = threadIdx.x; PIV && c < c0; c += NTL)
		{
			for (int j = 0; j < cf; j++)
			{
				const int r1 = c0 + j, r2 = pivs[j];
				if (r1 != r2)
				{
					auto &u = gD.at(di + r1, dj + c);
					auto &v = gD.at(di + r2, dj + c);
					const T t = u;
					u = v;
					v = t;
				}
			}
		}
	}
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
template <typename T>
static int fact_mmax_arg(const blasfeo_amd_hint *hint, const char *name, int *mmax)
{
	int mm = (hint && hint->max_m > 0) ? hint->max_m : 256;
	if (mm > fact_mmax<T>())
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: m up to %d supported, got %d", name, fact_mmax<T>(), mm);
	*mmax = mm;
	return BLASFEO_AMD_OK;
}

static int fact_check(int ps, int batch, const void *args, bool is_float, const char *name)
{
	if (batch < 0)
		return set_error(BLASFEO_AMD_EINVAL, "%s: batch=%d < 0", name, batch);
	if (batch > 0 && !args)
		return set_error(BLASFEO_AMD_EINVAL, "%s: args is NULL", name);
	const bool ok = is_float ? (ps == 4 || ps == 8 || ps == 16) : (ps == 4 || ps == 8);
	if (!ok)
		return set_error(BLASFEO_AMD_EINVAL, "%s: unsupported panel size %d", name, ps);
	return BLASFEO_AMD_OK;
}

// ---------------------------------------------------------------------------
// potrf_l_mn and syrk_dpotrf_ln(_mn) for m > 128: the m x n lower trapezoid
// as the n x n Cholesky of its top block (potrf_l, whose kernels store the
// reciprocal diagonal in D's dA) followed by the rows below,
// L21 = C21 L11^{-T}, solved with those reciprocals (trsm_rltn reading dA);
// syrk_dpotrf first forms C + A B^T in D (syrk_ln_mn) and then factors D in
// place.  The per-instance records of the steps are built on the device into
// the stream's workspace, so the call stays asynchronous.  This is the
// reference's own decomposition of the trapezoid
// (blasfeo_ref/x_lapack_ref.c:185-326: column j of the rows below is the
// pivot column's update times 1/L_jj).
// ---------------------------------------------------------------------------
constexpr int MN_NMAX = 256;

__global__ void k_mn_split(const blasfeo_amd_dfact_arg *__restrict__ args, int batch,
	blasfeo_amd_dfact_arg *top, blasfeo_amd_dtrsm_arg *rows)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= batch)
		return;
	const blasfeo_amd_dfact_arg a = args[i];
	const int m = a.m;
	const int n = a.n < m ? a.n : m;
	blasfeo_amd_dfact_arg t = a;
	blasfeo_amd_dtrsm_arg r;
	const bool live = m > 0 && n > 0;
	t.m = t.n = live ? n : 0;
	t.ipiv = nullptr;
	r.m = live ? m - n : 0;
	r.n = n;
	r.ai = a.di; r.aj = a.dj;
	r.bi = a.ci + n; r.bj = a.cj;
	r.di = a.di + n; r.dj = a.dj;
	r.alpha = 1.0;
	r.sA = a.sD; r.sB = a.sC; r.sD = a.sD;
	top[i] = t;
	rows[i] = r;
}

// use_dA of the trapezoid factorisations (blasfeo_hp_pm/d_lapack_lib4.c:1185,1545,1882)
__global__ void k_mn_finish(const blasfeo_amd_dfact_arg *__restrict__ args, int batch)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= batch)
		return;
	const blasfeo_amd_dfact_arg &a = args[i];
	if (a.m > 0 && a.n > 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? 1 : 0;
}

// syrk_dpotrf records -> syrk_ln_mn records (D = C + A B^T on the trapezoid)
// and trapezoid Cholesky records (in place on D)
__global__ void k_sp_split(const blasfeo_amd_dsyrk_dpotrf_arg *__restrict__ args, int batch,
	blasfeo_amd_dgemm_arg *upd, blasfeo_amd_dfact_arg *fact)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= batch)
		return;
	const blasfeo_amd_dsyrk_dpotrf_arg a = args[i];
	const int m = a.m;
	const int n = a.n < m ? a.n : m;
	const bool live = m > 0 && n > 0 && a.k >= 0;
	blasfeo_amd_dgemm_arg g;
	g.m = live ? m : 0; g.n = n; g.k = a.k;
	g.ai = a.ai; g.aj = a.aj; g.bi = a.bi; g.bj = a.bj;
	g.ci = a.ci; g.cj = a.cj; g.di = a.di; g.dj = a.dj;
	g.alpha = 1.0; g.beta = 1.0;
	g.sA = a.sA; g.sB = a.sB; g.sC = a.sC; g.sD = a.sD;
	blasfeo_amd_dfact_arg f;
	f.m = live ? m : 0; f.n = n;
	f.ci = a.di; f.cj = a.dj; f.di = a.di; f.dj = a.dj;
	f.sC = a.sD; f.sD = a.sD;
	f.ipiv = nullptr;
	upd[i] = g;
	fact[i] = f;
}

static int mn_nmax(const blasfeo_amd_hint *hint, int mmax)
{
	return (hint && hint->max_n > 0 && hint->max_n < mmax) ? hint->max_n : mmax;
}

static int launch_potrf_mn_split(int ps, int batch, const blasfeo_amd_dfact_arg *args, const blasfeo_amd_hint *hint, int mmax, hipStream_t st, const char *name)
{
	const int nmax = mn_nmax(hint, mmax);
	if (nmax > MN_NMAX)
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: n up to %d supported when m > 128, got a bound of %d", name, MN_NMAX, nmax);
	const size_t tb = ((size_t)batch * sizeof(blasfeo_amd_dfact_arg) + 255) / 256 * 256;
	unsigned char *ws = (unsigned char *)workspace(tb + (size_t)batch * sizeof(blasfeo_amd_dtrsm_arg), st);
	if (!ws)
		return set_error(BLASFEO_AMD_ENOMEM, "%s: workspace allocation failed", name);
	blasfeo_amd_dfact_arg *top = (blasfeo_amd_dfact_arg *)ws;
	blasfeo_amd_dtrsm_arg *rows = (blasfeo_amd_dtrsm_arg *)(ws + tb);
	const int nb = (batch + 255) / 256;
	hipLaunchKernelGGL(k_mn_split, dim3(nb), dim3(256), 0, st, args, batch, top, rows);
	int rc = check_launch(name);
	if (rc)
		return rc;
	blasfeo_amd_hint ht = {nmax, nmax, 0};
	if ((rc = blasfeo_amd_dpotrf_l_batched(ps, batch, top, &ht, st)))
		return rc;
	blasfeo_amd_hint hr = {mmax, nmax, 0};
	if ((rc = trsm_rltn_given_dA(ps, batch, rows, &hr, st, name)))
		return rc;
	hipLaunchKernelGGL(k_mn_finish, dim3(nb), dim3(256), 0, st, args, batch);
	return check_launch(name);
}

template <typename T, int MODE>
static int launch_potrf(int ps, int batch, const typename FactArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = fact_check(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	int mmax;
	if ((rc = fact_mmax_arg<T>(hint, name, &mmax)))
		return rc;
	if (mmax <= (MODE == 0 ? 256 : 128))
	{
		// sizes up to 128 are bounded to whole strips
		if (mmax <= 128)
			mmax = (mmax + 15) / 16 * 16;
		// One wave per instance once the batch gives every CU more than three
		// instances (four up to 64 columns, two in FP32 above), NW waves per
		// instance below: n = 64, 128 and 256 in batches of 256 take 16, 59 and 311 us
		// against 14, 41 and 114 us, in batches of 8192 88, 489 and 2715 us against
		// 106, 597 and 3431 us (MI355X); at 558 instances of 128, 256 and U{199..245}
		// 65, 354 and 334 us against 54, 315 and 266, at 1024 of the first two 72 and
		// 419 against 86 and 447; of 64 at 1024 17.8 against 17.5; FP32 of 128 at 558
		// 56 and 56, at 1024 61 and 74.  The "potrf_bw" knob forces the first (1) or
		// the second (2, 4).
		const int cus = num_cus() > 0 ? num_cus() : 256;
		const int knob = tune_value(TUNE_POTRF_BW, 0);
		const int few = mmax <= 64 ? 4 : sizeof(T) == 8 ? 3 : 2;
		const bool wave = knob == 1 || (knob == 0 && batch > few * cus);
#define BFA_POTRF(PS_, NB_, NW_)                                                                                           \
	do                                                                                                                     \
	{                                                                                                                      \
		if (wave)                                                                                                          \
			hipLaunchKernelGGL((k_potrf_wave<T, PS_, NB_>), dim3(batch), dim3(WAVE), 0, st, args, mmax, MODE == 1);        \
		else                                                                                                               \
			hipLaunchKernelGGL((k_potrf_coop<T, PS_, NW_>), dim3(batch), dim3(WAVE * NW_), 0, st, args, mmax, MODE == 1);  \
	} while (0)
#define BFA_POTRF_N(PS_)              \
	do                                \
	{                                 \
		if (mmax <= 32)               \
			BFA_POTRF(PS_, 2, 1);     \
		else if (mmax <= 64)          \
			BFA_POTRF(PS_, 4, 2);     \
		else if (mmax <= 128)         \
			BFA_POTRF(PS_, 8, 4);     \
		else                          \
			BFA_POTRF(PS_, 16, 8);    \
	} while (0)
		if (ps == 4)
			BFA_POTRF_N(4);
		else if (ps == 8)
			BFA_POTRF_N(8);
		else if constexpr (sizeof(T) == 4)
			BFA_POTRF_N(16);
#undef BFA_POTRF_N
#undef BFA_POTRF
		return check_launch(name);
	}
	if (MODE == 1)
		return launch_potrf_mn_split(ps, batch, (const blasfeo_amd_dfact_arg *)args, hint, mmax, st, name);
	const size_t shm = sizeof(T) * PW * ((mmax + 15) / 16 * 16 + 1);
	if (ps == 4)
		hipLaunchKernelGGL((k_potrf<T, 4>), dim3(batch), dim3(NTL), shm, st, args, mmax);
	else if (ps == 8)
		hipLaunchKernelGGL((k_potrf<T, 8>), dim3(batch), dim3(NTL), shm, st, args, mmax);
	else
		hipLaunchKernelGGL((k_potrf<T, 16>), dim3(batch), dim3(NTL), shm, st, args, mmax);
	return check_launch(name);
}

template <typename T, bool PIV, int NW>
static void launch_getrf_wg(int ps, int batch, const typename FactArg<T>::type *args, int mmax, const int *counts, const int *lists, hipStream_t st)
{
	constexpr size_t shm = sizeof(T) * 16 * (NW * WAVE + 1);
	if (ps == 4)
		hipLaunchKernelGGL((k_getrf_wg<T, 4, PIV, NW>), dim3(batch), dim3(NW * WAVE), shm, st, args, mmax, batch, counts, lists);
	else if (ps == 8)
		hipLaunchKernelGGL((k_getrf_wg<T, 8, PIV, NW>), dim3(batch), dim3(NW * WAVE), shm, st, args, mmax, batch, counts, lists);
	else if constexpr (sizeof(T) == 4)
		hipLaunchKernelGGL((k_getrf_wg<T, 16, PIV, NW>), dim3(batch), dim3(NW * WAVE), shm, st, args, mmax, batch, counts, lists);
}

template <typename T, bool PIV = true>
static int launch_getrf(int ps, int batch, const typename FactArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = fact_check(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	int mmax;
	if ((rc = fact_mmax_arg<T>(hint, name, &mmax)))
		return rc;
	const size_t shm = sizeof(T) * PW * ((mmax + 15) / 16 * 16 + 1) + sizeof(int) * mmax;
	// the size order (k_getrf_plan): counts (64 ints) and one list per bucket
	int *ws = (int *)workspace(sizeof(int) * (64 + (size_t)GETRF_NB * batch), st);
	if (!ws)
		return set_error(BLASFEO_AMD_ENOMEM, "%s: workspace allocation failed", name);
	int *counts = ws, *lists = ws + 64;
	hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, st, counts, 64);
	hipLaunchKernelGGL((k_getrf_plan<T>), dim3((batch + 255) / 256), dim3(256), 0, st, args, batch, counts, lists);
	if (mmax <= GLU_M)
	{
		// the waves of a workgroup by the bound of the rows, so that small instances
		// come with as many workgroups per CU as there are registers for; a launch
		// for each range of rows was no faster on mixed batches (8192 LU solves of
		// U{16..256} 3916 against 3925 us) and slower on small ones (512: 600, 806)
		if (mmax <= 64)
			launch_getrf_wg<T, PIV, 1>(ps, batch, args, mmax, counts, lists, st);
		else if (mmax <= 128)
			launch_getrf_wg<T, PIV, 2>(ps, batch, args, mmax, counts, lists, st);
		else
			launch_getrf_wg<T, PIV, 4>(ps, batch, args, mmax, counts, lists, st);
		return check_launch(name);
	}
	if (ps == 4)
		hipLaunchKernelGGL((k_getrf<T, 4, PIV>), dim3(batch), dim3(NTL), shm, st, args, mmax, batch, counts, lists);
	else if (ps == 8)
		hipLaunchKernelGGL((k_getrf<T, 8, PIV>), dim3(batch), dim3(NTL), shm, st, args, mmax, batch, counts, lists);
	else
		hipLaunchKernelGGL((k_getrf<T, 16, PIV>), dim3(batch), dim3(NTL), shm, st, args, mmax, batch, counts, lists);
	return check_launch(name);
}

static int launch_syrk_potrf(int ps, int batch, const blasfeo_amd_dsyrk_dpotrf_arg *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = fact_check(ps, batch, args, false, name);
	if (rc || batch == 0)
		return rc;
	int mmax;
	if ((rc = fact_mmax_arg<double>(hint, name, &mmax)))
		return rc;
	if (mmax > 128)
	{
		const int nmax = mn_nmax(hint, mmax);
		if (nmax > MN_NMAX)
			return set_error(BLASFEO_AMD_ETOOBIG, "%s: n up to %d supported when m > 128, got a bound of %d", name, MN_NMAX, nmax);
		const size_t gb = ((size_t)batch * sizeof(blasfeo_amd_dgemm_arg) + 255) / 256 * 256;
		const size_t fb = ((size_t)batch * sizeof(blasfeo_amd_dfact_arg) + 255) / 256 * 256;
		const size_t tb = fb;
		// layout: [gemm records][fact records][potrf_l_mn split: top records][rows]
		unsigned char *ws = (unsigned char *)workspace(gb + fb + tb + (size_t)batch * sizeof(blasfeo_amd_dtrsm_arg), st);
		if (!ws)
			return set_error(BLASFEO_AMD_ENOMEM, "%s: workspace allocation failed", name);
		blasfeo_amd_dgemm_arg *upd = (blasfeo_amd_dgemm_arg *)ws;
		blasfeo_amd_dfact_arg *fact = (blasfeo_amd_dfact_arg *)(ws + gb);
		blasfeo_amd_dfact_arg *top = (blasfeo_amd_dfact_arg *)(ws + gb + fb);
		blasfeo_amd_dtrsm_arg *rows = (blasfeo_amd_dtrsm_arg *)(ws + gb + fb + tb);
		const int nb = (batch + 255) / 256;
		hipLaunchKernelGGL(k_sp_split, dim3(nb), dim3(256), 0, st, args, batch, upd, fact);
		if ((rc = check_launch(name)))
			return rc;
		blasfeo_amd_hint hg = {mmax, nmax, hint ? hint->max_k : 0};
		if ((rc = blasfeo_amd_dsyrk_ln_mn_batched(ps, batch, upd, &hg, st)))
			return rc;
		hipLaunchKernelGGL(k_mn_split, dim3(nb), dim3(256), 0, st, fact, batch, top, rows);
		if ((rc = check_launch(name)))
			return rc;
		blasfeo_amd_hint ht = {nmax, nmax, 0};
		if ((rc = blasfeo_amd_dpotrf_l_batched(ps, batch, top, &ht, st)))
			return rc;
		blasfeo_amd_hint hr = {mmax, nmax, 0};
		if ((rc = trsm_rltn_given_dA(ps, batch, rows, &hr, st, name)))
			return rc;
		hipLaunchKernelGGL(k_mn_finish, dim3(nb), dim3(256), 0, st, fact, batch);
		return check_launch(name);
	}
	mmax = (mmax + 15) / 16 * 16;
#define BFA_SP(PS_, NW_) hipLaunchKernelGGL((k_syrk_potrf_coop<double, PS_, NW_>), dim3(batch), dim3(WAVE * NW_), 0, st, args, mmax)
#define BFA_SP_N(PS_)           \
	do                          \
	{                           \
		if (mmax <= 32)         \
			BFA_SP(PS_, 1);     \
		else if (mmax <= 64)    \
			BFA_SP(PS_, 2);     \
		else                    \
			BFA_SP(PS_, 4);     \
	} while (0)
	if (ps == 4)
		BFA_SP_N(4);
	else
		BFA_SP_N(8);
#undef BFA_SP_N
#undef BFA_SP
	return check_launch(name);
}

} // namespace bfa

using namespace bfa;

extern "C" {

int blasfeo_amd_dpotrf_l_batched(int ps, int batch, const blasfeo_amd_dfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_potrf<double, 0>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dpotrf_l_batched"); }
// Large m: the trapezoid as potrf_l of the top block plus the solve of the rows
// below (launch_potrf_mn_split).
int blasfeo_amd_dpotrf_l_mn_batched(int ps, int batch, const blasfeo_amd_dfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_potrf<double, 1>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dpotrf_l_mn_batched"); }
int blasfeo_amd_dsyrk_dpotrf_ln_batched(int ps, int batch, const blasfeo_amd_dsyrk_dpotrf_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_syrk_potrf(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dsyrk_dpotrf_ln_batched"); }
int blasfeo_amd_dgetrf_rp_batched(int ps, int batch, const blasfeo_amd_dfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_getrf<double>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dgetrf_rp_batched"); }
int blasfeo_amd_dgetrf_np_batched(int ps, int batch, const blasfeo_amd_dfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_getrf<double, false>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dgetrf_np_batched"); }
int blasfeo_amd_spotrf_l_batched(int ps, int batch, const blasfeo_amd_sfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_potrf<float, 0>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_spotrf_l_batched"); }
int blasfeo_amd_sgetrf_rp_batched(int ps, int batch, const blasfeo_amd_sfact_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_getrf<float>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_sgetrf_rp_batched"); }

} // extern "C"
