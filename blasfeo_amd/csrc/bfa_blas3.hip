// bfa_blas3.hip -- batched level-3 kernels for gfx950: gemm_nt, gemm_nn,
// syrk_ln(_mn), trmm_rlnn and trsm_rltn on panel-major matrices.
//
// Launch model: one workgroup per (instance, tile slot), `slots` slots per
// instance (tile t of an instance goes to slot t mod slots), so a batch of
// small instances uses one workgroup each and a batch of large ones spreads
// its tiles over several.  gemm and syrk: one wavefront per tile
// (bfa_gemm_wave.hpp); trmm: 64 x 64 tiles by four waves through LDS
// (bfa_gemm_core.hpp), in XCD-aware order when an instance has more than four slots
// and instance-fastest otherwise (batch_slot); trsm: bfa_trsm_strip.hpp.
#include "bfa_gemm_core.hpp"
#include "bfa_gemm_wave.hpp"
#include "bfa_chol_core.hpp"
#include "bfa_trsm_strip.hpp"
#include "bfa_internal.hpp"

namespace bfa {

// D = alpha * B * A, A lower n x n (blasfeo_ref/x_blas3_ref.c:3218-3330)
template <typename T, int PS>
__global__ __launch_bounds__(NT3) __attribute__((amdgpu_waves_per_eu(3))) void k_trmm_rlnn(const typename TrsmArg<T>::type *__restrict__ args, int batch, int slots)
{
	__shared__ T As[KC * LDT];
	__shared__ T Bs[KC * LDT];
	int inst, slot;
	batch_slot(slots > 4, batch, slots, inst, slot);
	if (inst >= batch)
		return;
	const typename TrsmArg<T>::type &a = args[inst];
	if (a.m <= 0 || a.n <= 0)
		return;
	if (threadIdx.x == 0 && slot == 0)
		a.sD->use_dA = 0;
	trmm_core<T, PS>(As, Bs, a.m, a.n, a.alpha, view<T, PS>(a.sA), a.ai, a.aj, view<T, PS>(a.sB), a.bi, a.bj,
		view<T, PS>(a.sD), a.di, a.dj, slot, slots);
}

// ---------------------------------------------------------------------------
// trsm_llnn / trsm_lltn / trsm_llnu / trsm_lunn: D = alpha * A^{-1} * B,
// alpha * A^{-T} * B with A lower, alpha * A^{-1} * B with A unit lower, or
// alpha * U^{-1} * B with U the upper triangle of A; m x m, B m x n
// (blasfeo_ref/x_blas3_ref.c:445-673, 674-900, 572-672, 920-1100).  lunn is
// lltn on the transposed view of A (U(i,k) = A^T(i,k)), so it shares lltn's
// bottom-up sweep; llnu is llnn without the reciprocal diagonal.
// A workgroup keeps a block of up to LNC columns of X = alpha*B for all m rows
// in LDS (column-major, odd leading dimension) and sweeps the 16-row blocks of
// A, top-down for llnn and bottom-up for lltn: wave 0 solves the 16x16
// diagonal triangle of the block (one column of X per lane, the 16 rows in
// registers, multiplying by the reciprocal diagonal as the reference does),
// then every thread applies the solved rows to one remaining row of X (below
// for llnn, above for lltn), reading that row's 16 elements of A once.  The
// next diagonal block is staged into the other half of a double buffer during
// the update, so each block costs two workgroup barriers.
// ---------------------------------------------------------------------------
constexpr int LNC = 16;
template <typename T> constexpr int trsml_mmax() { return sizeof(T) == 8 ? 1024 : 2048; }

enum TrsmLeftMode { TL_LLNN = 0, TL_LLTN = 1, TL_LLNU = 2, TL_LUNN = 3 };
// the sweep runs bottom-up for the transposed-lower and the upper solves
constexpr bool tl_back(int mode) { return mode == TL_LLTN || mode == TL_LUNN; }

// element (r, c) of the lower triangle the sweep works on: A itself, or A^T
// for the upper solve (its upper triangle read as a lower one)
template <typename T, int PS, int MODE>
__device__ __forceinline__ T tl_at(const PM<T, PS> gA, int ai, int aj, int r, int c)
{
	return MODE == TL_LUNN ? gA.at(ai + c, aj + r) : gA.at(ai + r, aj + c);
}

template <typename T, int PS, int MODE>
__device__ __forceinline__ void trsml_stage_diag(const PM<T, PS> gA, int ai, int aj, int r0, int rv, T *Ad)
{
	for (int e = threadIdx.x; e < 256; e += NT3)
	{
		const int r = e & 15, c = e >> 4;
		T v = T(0);
		if (r < rv && c < rv && r > c)
			v = tl_at<T, PS, MODE>(gA, ai, aj, r0 + r, r0 + c);
		Ad[r * 17 + c] = v;
	}
}

template <typename T, int PS, int MODE>
__global__ __launch_bounds__(NT3) void k_trsm_left(const typename TrsmArg<T>::type *__restrict__ args, int mmax)
{
	constexpr bool TRANS = tl_back(MODE);
	constexpr bool UNIT = MODE == TL_LLNU;
	extern __shared__ unsigned char smem_raw[];
	__shared__ T Ad[2][16 * 17];
	const int mpad = (mmax + 15) / 16 * 16;
	const int LDM = mpad + 1;
	T *Xs = reinterpret_cast<T *>(smem_raw);   // [LNC][LDM]
	T *inv_s = Xs + (size_t)LNC * LDM;           // [mpad]

	const typename TrsmArg<T>::type &a = args[blockIdx.x];
	const int m = a.m, n = a.n;
	if (m <= 0 || n <= 0 || m > mmax)
		return;
	const PM<T, PS> gA = view<T, PS>(a.sA);
	const PM<T, PS> gB = view<T, PS>(a.sB);
	PM<T, PS> gD = view<T, PS>(a.sD);
	const int ai = a.ai, aj = a.aj;
	const T alpha = a.alpha;
	const int lane = lane_id();
	const int w = wave_id();
	const int mb = (m + 15) / 16;

	if (!UNIT)
	{
		const bool cached = (ai == 0 && aj == 0 && a.sD != a.sA && a.sA->use_dA >= m);
		for (int j = threadIdx.x; j < m; j += NT3)
			inv_s[j] = cached ? a.sA->dA[j] : T(1) / gA.at(ai + j, aj + j);
	}

	for (int j0 = blockIdx.y * LNC; j0 < n; j0 += gridDim.y * LNC)
	{
		const int nc = min(LNC, n - j0);
		__syncthreads();
		g2s<T, PS, NT3, false>(gB, a.bi, a.bj + j0, mb * 16, LNC, m, nc, Xs, LDM);
		{
			const int rb0 = TRANS ? mb - 1 : 0;
			trsml_stage_diag<T, PS, MODE>(gA, ai, aj, rb0 * 16, min(16, m - rb0 * 16), Ad[0]);
		}
		__syncthreads();
		for (int e = threadIdx.x; e < LNC * LDM; e += NT3)
			Xs[e] *= alpha;
		__syncthreads();
		for (int s = 0; s < mb; s++)
		{
			const int rb = TRANS ? mb - 1 - s : s;
			const int r0 = rb * 16;
			const int rv = min(16, m - r0);
			const T *A0 = Ad[s & 1];
			// diagonal triangle: lane c owns column c of the block
			if (w == 0 && lane < nc)
			{
				T x[16];
#pragma unroll
				for (int l = 0; l < 16; l++)
					x[l] = Xs[lane * LDM + r0 + l];
				if (!TRANS)
				{
#pragma unroll
					for (int i = 0; i < 16; i++)
					{
						if (i < rv)
						{
							T c = x[i];
#pragma unroll
							for (int l = 0; l < i; l++)
								c -= A0[i * 17 + l] * x[l];
							x[i] = UNIT ? c : c * inv_s[r0 + i];
						}
					}
				}
				else
				{
#pragma unroll
					for (int i = 15; i >= 0; i--)
					{
						if (i < rv)
						{
							T c = x[i];
#pragma unroll
							for (int l = i + 1; l < 16; l++)
								c -= A0[l * 17 + i] * x[l];
							x[i] = c * inv_s[r0 + i];
						}
					}
				}
#pragma unroll
				for (int l = 0; l < 16; l++)
					if (l < rv)
						Xs[lane * LDM + r0 + l] = x[l];
			}
			__syncthreads();
			// stage the next diagonal block, then update the remaining rows
			if (s + 1 < mb)
			{
				const int rbn = TRANS ? rb - 1 : rb + 1;
				trsml_stage_diag<T, PS, MODE>(gA, ai, aj, rbn * 16, min(16, m - rbn * 16), Ad[(s + 1) & 1]);
			}
			const int ilo = TRANS ? 0 : r0 + 16;
			const int ihi = TRANS ? r0 : m;
			for (int i = ilo + threadIdx.x; i < ihi; i += NT3)
			{
				T av[16];
#pragma unroll
				for (int l = 0; l < 16; l++)
				{
					T v = T(0);
					if (l < rv)
						v = TRANS ? tl_at<T, PS, MODE>(gA, ai, aj, r0 + l, i) : tl_at<T, PS, MODE>(gA, ai, aj, i, r0 + l);
					av[l] = v;
				}
				for (int c = 0; c < nc; c++)
				{
					T acc = Xs[c * LDM + i];
#pragma unroll
					for (int l = 0; l < 16; l++)
						acc -= av[l] * Xs[c * LDM + r0 + l];
					Xs[c * LDM + i] = acc;
				}
			}
			__syncthreads();
		}
		s2g<T, PS, NT3, false>(gD, a.di, a.dj + j0, m, nc, Xs, LDM, 0);
	}
}

// ---------------------------------------------------------------------------
// The same four left-side solves for few right-hand sides (chosen when the hint
// bounds n by 4) and m <= 256: one wavefront per instance, row i of X in lane
// i % 64 (slot i / 64), four columns of X at a time in registers.  The columns j of
// the solve are taken in order (top-down for llnn and llnu, bottom-up for lltn and
// lunn): row j's values are scaled by the reciprocal diagonal and broadcast with
// v_readlane, and every row still to be solved drops its multiple of them.  No
// barriers.  The elements of A are loaded four columns at a time (a 128-byte line
// holds four columns of a panel's rows for ps = 4), the next four while the
// current ones are applied.
// Measured (MI355X, 4 right-hand sides; before: a column at a time): 8192 LU solves
// (factorisation included) of U{16..256} 3922 -> 3829 us, of U{16..64} 355 -> 326.
// ---------------------------------------------------------------------------
constexpr int THIN_RHS = 4;
constexpr int THIN_Q = 4;

template <typename T, int PS, int MODE, int Q>
__device__ __forceinline__ void trsm_thin(const typename TrsmArg<T>::type &a, int m, int nrhs, const StripView<T, PS> &vA,
	const StripView<T, PS> &vB, const StripView<T, PS> &vD)
{
	constexpr bool BACK = tl_back(MODE);
	constexpr bool UNIT = MODE == TL_LLNU;
	constexpr unsigned CS = PS * sizeof(T);
	typedef unsigned O;
	int ai = a.ai, aj = a.aj, bi = a.bi, bj = a.bj, di = a.di, dj = a.dj;
	const StripView<T, PS, O> A = vA.template block<O>(ai, aj), B = vB.template block<O>(bi, bj), D = vD.template block<O>(di, dj);
	const int lane = threadIdx.x;
	const bool cached = !UNIT && a.ai == 0 && a.aj == 0 && a.sD != a.sA && a.sA->use_dA >= m;
	const BFA_GLOBAL T *dA = (const BFA_GLOBAL T *)a.sA->dA;
	// this lane's rows of A (lltn: columns; rows past the end read the last one)
	// and their reciprocal diagonals
	O oa[Q];
	T rd[Q];
#pragma unroll
	for (int q = 0; q < Q; q++)
		if (q * WAVE < m)
		{
			const int i = min(lane + q * WAVE, m - 1);
			oa[q] = MODE == TL_LLTN ? (O)(aj + i) * CS : A.at(ai + i, aj);
			rd[q] = UNIT ? T(1) : cached ? dA[i] : T(1) / A.ld(0, A.at(ai + i, aj + i));
		}
	// columns j0 .. j0+3 of the solve, slots q0 .. q1-1
	auto coef = [&](int j0, int q0, int q1, T (&e)[Q][4]) {
#pragma unroll
		for (int q = 0; q < Q; q++)
			if (q >= q0 && q < q1 && q * WAVE < m)
#pragma unroll
				for (int t = 0; t < 4; t++)
				{
					const int j = max(0, min(j0 + t, m - 1));
					e[q][t] = A.ld(MODE == TL_LLTN ? A.at(ai + j, 0) : (O)j * CS, oa[q]);
				}
	};
	// right-hand sides in groups of THIN_RHS (one group when n <= 4)
	for (int c0 = 0; c0 < nrhs; c0 += THIN_RHS)
	{
		const int n = min(THIN_RHS, nrhs - c0);
		// (pinned, here and at the end: the rows' offsets in B and D, the same for every
		// group, would be kept in registers across the sweep)
		int lb0 = lane;
		BFA_PIN(lb0);
		T x[Q][THIN_RHS];
#pragma unroll
		for (int q = 0; q < Q; q++)
#pragma unroll
			for (int c = 0; c < THIN_RHS; c++)
			{
				const int i = lb0 + q * WAVE;
				x[q][c] = (i < m && c < n) ? a.alpha * B.ld(0, B.at(bi + i, bj + c0 + c)) : T(0);
			}
		T e[Q][4];
		coef(BACK ? (m - 1) & ~3 : 0, 0, Q, e);
		// grouped by the register slot qb = j / 64 that holds row j (unrolled, so
		// that every register index is a constant)
#pragma unroll
		for (int qq = 0; qq < Q; qq++)
		{
			const int qb = BACK ? Q - 1 - qq : qq;
#pragma unroll 1
			for (int l4 = 0; l4 < WAVE; l4 += 4)
			{
				const int lb = BACK ? WAVE - 4 - l4 : l4;   // first lane of the group
				const int j0 = qb * WAVE + lb;
				if (j0 >= m)
				{
					if (BACK)
						continue;
					break;
				}
				T en[Q][4];
				if (BACK ? j0 > 0 : j0 + 4 < m)
					coef(BACK ? j0 - 4 : j0 + 4, BACK ? 0 : qb, BACK ? qb + 1 : Q, en);
#pragma unroll
				for (int tt = 0; tt < 4; tt++)
				{
					const int t = BACK ? 3 - tt : tt;
					const int j = j0 + t;
					if (j < m)
					{
						const T d = UNIT ? T(1) : readlane(rd[qb], lb + t);
						T xj[THIN_RHS];
#pragma unroll
						for (int c = 0; c < THIN_RHS; c++)
							xj[c] = readlane(x[qb][c], lb + t) * d;
						// only the rows still to be solved take the update (a
						// solved row is never touched again, so an Inf or NaN in
						// xj cannot reach it); row j itself keeps its unscaled
						// value, scaled by its reciprocal after the sweep
						const bool open = BACK ? lane < lb + t : lane > lb + t;
#pragma unroll
						for (int q = 0; q < Q; q++)
						{
							if (BACK ? q > qb : q < qb)
								continue;
							if (q * WAVE >= m)
								continue;
#pragma unroll
							for (int c = 0; c < THIN_RHS; c++)
							{
								const T y = x[q][c] - e[q][t] * xj[c];
								x[q][c] = q != qb || open ? y : x[q][c];
							}
						}
					}
				}
#pragma unroll
				for (int q = 0; q < Q; q++)
#pragma unroll
					for (int t = 0; t < 4; t++)
						e[q][t] = en[q][t];
			}
		}
		// row i's solved value is its unscaled value times the reciprocal the
		// sweep used for column i (the same product the broadcast formed)
		int ld0 = lane;
		BFA_PIN(ld0);
#pragma unroll
		for (int q = 0; q < Q; q++)
		{
			const int i = ld0 + q * WAVE;
			if (i < m)
#pragma unroll
				for (int c = 0; c < THIN_RHS; c++)
					if (c < n)
						D.st(0, D.at(di + i, dj + c0 + c), UNIT ? x[q][c] : x[q][c] * rd[q]);
		}
	}
}

// The same with X in D, for panel strides too large for 32-bit offsets and for instances
// larger than the launch's slots.  (With 64-bit offsets the code above spills, and
// scratch costs the launches of small instances that never use it: 16384 of 24 rows
// 45 -> 66 us.)
template <typename T, int PS, int MODE>
__device__ __forceinline__ void trsm_thin_wide(const typename TrsmArg<T>::type &a, int m, int nrhs, const StripView<T, PS> &A,
	const StripView<T, PS> &B, const StripView<T, PS> &D)
{
	constexpr bool BACK = tl_back(MODE), UNIT = MODE == TL_LLNU;
	const int lane = threadIdx.x;
	const bool cached = !UNIT && a.ai == 0 && a.aj == 0 && a.sD != a.sA && a.sA->use_dA >= m;
	const BFA_GLOBAL T *dA = (const BFA_GLOBAL T *)a.sA->dA;
#pragma unroll 1
	for (int c = 0; c < nrhs; c++)
	{
#pragma unroll 1
		for (int i = lane; i < m; i += WAVE)
			D.st(0, D.at(a.di + i, a.dj + c), a.alpha * B.ld(0, B.at(a.bi + i, a.bj + c)));
		wave_sync();
#pragma unroll 1
		for (int t = 0; t < m; t++)
		{
			const int j = BACK ? m - 1 - t : t;
			const size_t oj = D.at(a.di + j, a.dj + c);
			const T d = UNIT ? T(1) : cached ? dA[j] : T(1) / A.ld(0, A.at(a.ai + j, a.aj + j));
			const T x = D.ld(0, oj) * d;
			wave_sync();   // every lane has read row j
			if (lane == 0)
				D.st(0, oj, x);
#pragma unroll 1
			for (int i = (BACK ? 0 : j + 1) + lane; i < (BACK ? j : m); i += WAVE)
			{
				const size_t o = D.at(a.di + i, a.dj + c);
				D.st(0, o, D.ld(0, o) - A.ld(0, MODE == TL_LLTN ? A.at(a.ai + j, a.aj + i) : A.at(a.ai + i, a.aj + j)) * x);
			}
			wave_sync();
		}
	}
}

// Q: the row slots that the hint's bound asks for.  Each form is compiled for as many waves
// as leave it without scratch (with four slots for every bound 16384 dtrsm_lunn of
// U{4..64} took 120 us, the column at a time before it 113, one and two slots 73).
template <typename T, int PS, int MODE, int Q>
__global__ __launch_bounds__(WAVE, Q == 4 ? 3 : 4) void k_trsm_left_thin(const typename TrsmArg<T>::type *__restrict__ args)
{
	const typename TrsmArg<T>::type &a = args[blockIdx.x];
	const int m = __builtin_amdgcn_readfirstlane(a.m), nrhs = __builtin_amdgcn_readfirstlane(a.n);
	if (m <= 0 || nrhs <= 0 || m > THIN_Q * WAVE)
		return;
	const StripView<T, PS> A = strip_view<T, PS>(a.sA), B = strip_view<T, PS>(a.sB), D = strip_view<T, PS>(a.sD);
	if (__builtin_expect(m <= Q * WAVE && strip_fits<T, PS>(max(A.cn, max(B.cn, D.cn))), 1))
		trsm_thin<T, PS, MODE, Q>(a, m, nrhs, A, B, D);
	else
		trsm_thin_wide<T, PS, MODE>(a, m, nrhs, A, B, D);
}

// Cache update after trsm_rltn / trsm_llnn / trsm_lltn, in the reference's
// order (blasfeo_hp_pm/d_blas3_lib4.c:4157-4178; blasfeo_ref/x_blas3_ref.c:
// 466-480): invalidate D's cache, then refresh A's reciprocal diagonal unless
// it was valid.  Run as its own launch so that no workgroup of the solve
// reads a dA another one is writing.  LEFT: the triangle is m x m, else n x n.
template <typename T, int PS, bool LEFT, bool UNIT = false>
__global__ void k_trsm_dA(const typename TrsmArg<T>::type *__restrict__ args)
{
	const typename TrsmArg<T>::type &a = args[blockIdx.x];
	const int n = LEFT ? a.m : a.n;
	if (a.m <= 0 || a.n <= 0)
		return;
	if (UNIT)
	{
		// trsm_llnu reads no reciprocal diagonal: only D's cache is invalidated
		if (threadIdx.x == 0)
			a.sD->use_dA = 0;
		return;
	}
	const bool zero_off = (a.ai == 0 && a.aj == 0);
	const int use0 = (a.sD == a.sA) ? 0 : a.sA->use_dA;
	__syncthreads();
	if (threadIdx.x == 0)
		a.sD->use_dA = 0;
	if (zero_off && use0 >= n)
		return;
	const PM<T, PS> gA = view<T, PS>(a.sA);
	for (int j = threadIdx.x; j < n; j += blockDim.x)
		a.sA->dA[j] = T(1) / gA.at(a.ai + j, a.aj + j);
	__syncthreads();
	if (threadIdx.x == 0)
		a.sA->use_dA = zero_off ? n : 0;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static int tiles_y(const blasfeo_amd_hint *hint, int tm, int tn)
{
	if (!hint || hint->max_m <= 0)
		return 1;
	int mt = (hint->max_m + tm - 1) / tm;
	int nt = hint->max_n > 0 ? (hint->max_n + tn - 1) / tn : 1;
	int y = mt * nt;
	int cap = tune_value(TUNE_GEMM_GRID_Y, 0);
	if (cap <= 0)
		cap = 64;
	return y < 1 ? 1 : (y > cap ? cap : y);
}

// tile slots per instance of a gemm-family launch with TE x TE tiles
template <int OP>
static int gemm_slots(const blasfeo_amd_hint *hint, int te)
{
	if (!hint || hint->max_m <= 0)
		return 1;
	const int mt = (hint->max_m + te - 1) / te;
	const int nt = OP == OP_SYRK ? mt : hint->max_n > 0 ? (hint->max_n + te - 1) / te : 1;
	int cap = tune_value(TUNE_GEMM_GRID_Y, 0);
	if (cap <= 0)
		cap = 64;
	return max(1, min(cap, gw_ntiles<OP>(mt, nt)));
}

static int check_common(int ps, int batch, const void *args, bool is_float, const char *name)
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

// threads of a launch (the CPU emulator of the kernels sets a smaller limit)
#ifndef BFA_GRID_THREADS
#define BFA_GRID_THREADS 0x7fffffffLL
#endif

// 1-D grid of batch * slots workgroups rounded up to a multiple of XCDS, for
// kernels that map their workgroup id through xcd_local_index
static int xcd_grid(int batch, int slots, int threads, dim3 *grid, const char *name)
{
	const long long wgs = ((long long)batch * slots + XCDS - 1) / XCDS * XCDS;
	if (wgs * threads > 0x7fffffffLL)
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: batch %d too large for one launch", name, batch);
	*grid = dim3((unsigned)wgs);
	return BLASFEO_AMD_OK;
}

// One wavefront per output tile, E = 4 (64 x 64) or E = 2 (32 x 32).
template <typename T, int PS, int OP, int E>
static int launch_gemm_tile(int batch, const typename GemmArg<T>::type *args, int slots, hipStream_t st, const char *name)
{
	// FP32 and few instances: their tiles over all XCDs (64 sgemm_nn of U{64..512}
	// 118 -> 81 us, of 512: 154 and 155 us; in FP64, where the operands that several
	// XCDs then read weigh more, 118 and 120, 270 and 304 us)
	const bool spread = sizeof(T) == 4 && batch <= 64;
	dim3 grid;
	int rc = xcd_grid(batch, slots, WAVE, &grid, name);
	if (rc)
		return rc;
	hipLaunchKernelGGL((k_gemm_wave<T, PS, OP, E>), grid, dim3(WAVE), 0, st, args, batch, slots, spread);
	return check_launch(name);
}
template <typename T, int PS, int OP>
static int launch_gemm_ps(int batch, const typename GemmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	// The large tile reads a quarter of the operands that the small one reads per
	// product but leaves a batch of few or uneven instances with too few waves.
	// It is taken above 256 rows or columns (64 dgemm_nn of 512: 270 us against 348,
	// 16 of them 74 against 120), and above 128 (FP32 96) where the
	// batch has 16384 of its tiles (4096 dgemm_nt + dsyrk_ln of U{16..256}: 1052
	// against 1132 us, 512 of them 219 against 180; 4096 of 128: 738 against 788, of
	// U{4..128} 260 against 229; 4096 FP32 of U{4..128} 157 against 166, of U{4..96}
	// 99 against 95).  The "gemm_wave" knob sets the small (1) or the large tile (2).
	const int knob = tune_value(TUNE_GEMM_WAVE, 0);
	const int slots = gemm_slots<OP>(hint, 64);
	const int maxm = hint ? hint->max_m : 0, maxn = OP == OP_SYRK ? maxm : hint ? hint->max_n : 0;
	// A bound missing: small tiles, and as many slots per instance as make 65536 waves of
	// the batch, 4 to 64 (dgemm_nt, us, against one slot of large tiles and the four
	// waves of the 64 x 64 LDS tile before them: one of 1024 737, 30957, 20992; one of 64
	// 5.9, 12.6, 10.2; 64 of 512 343, 4049, 2785; 512 of U{16..256} 94, 519, 409; 4096
	// 791, 1215, 1337; 2048 of 64 49, 44, 57; 65536 of U{4..32} 176, 231, 623).  Large
	// tiles with as many slots are up to 1.5 times faster on the largest and up to 5
	// times slower on the smallest.
	if (knob == 0 && (maxm <= 0 || maxn <= 0))
	{
		const int cap = tune_value(TUNE_GEMM_GRID_Y, 0);
		const int s = min(cap > 0 ? cap : 64, max(4, min(64, 65536 / batch)));
		return launch_gemm_tile<T, PS, OP, 2>(batch, args, s, st, name);
	}
	const int most = maxm > 0 && maxn > 0 ? max(maxm, maxn) : 512;
	const bool large = most > 256 || (most > (sizeof(T) == 8 ? 128 : 96) && (long long)batch * slots >= 16384);
	if (knob == 2 || (knob == 0 && large))
		return launch_gemm_tile<T, PS, OP, 4>(batch, args, slots, st, name);
	return launch_gemm_tile<T, PS, OP, 2>(batch, args, gemm_slots<OP>(hint, 32), st, name);
}

template <typename T, int OP>
static int launch_gemm(int ps, int batch, const typename GemmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = check_common(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	if (ps == 4)
		return launch_gemm_ps<T, 4, OP>(batch, args, hint, st, name);
	if (ps == 8)
		return launch_gemm_ps<T, 8, OP>(batch, args, hint, st, name);
	if constexpr (sizeof(T) == 4)
		return launch_gemm_ps<T, 16, OP>(batch, args, hint, st, name);
	return BLASFEO_AMD_EINVAL;
}

template <typename T>
static int launch_trmm(int ps, int batch, const typename TrsmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = check_common(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	const int slots = tiles_y(hint, TM, TN);
	dim3 grid;
	if ((rc = xcd_grid(batch, slots, NT3, &grid, name)))
		return rc;
	if (ps == 4)
		hipLaunchKernelGGL((k_trmm_rlnn<T, 4>), grid, dim3(NT3), 0, st, args, batch, slots);
	else if (ps == 8)
		hipLaunchKernelGGL((k_trmm_rlnn<T, 8>), grid, dim3(NT3), 0, st, args, batch, slots);
	else
		hipLaunchKernelGGL((k_trmm_rlnn<T, 16>), grid, dim3(NT3), 0, st, args, batch, slots);
	return check_launch(name);
}

// trsm_rltn: one launch per range of n, up to 64, 128 and 256 columns (the
// registers that hold a strip, and with them the waves per SIMD, go with the
// range), the largest first; a workgroup whose instance is not in its launch's
// range leaves at once.
template <typename T, int PS, int NB, bool GIVEN>
static int launch_trsm_nb(int batch, const typename TrsmArg<T>::type *args, int mmax, int nlo, int nmax, hipStream_t st, const char *name)
{
	constexpr int rows = 64 * trsm_strips<NB>();
	const int slots = mmax > 0 ? min(64, (mmax + rows - 1) / rows) : 4;
	constexpr size_t shm = trsm_lds<T, NB>();
	int rc = lds_check(reinterpret_cast<const void *>(&k_trsm_rltn<T, PS, NB, GIVEN>), shm, name);
	// a launch has fewer than BFA_GRID_THREADS threads: larger batches take several
	const int most = max(1, ((int)((long long)BFA_GRID_THREADS / NT3) - XCDS) / slots);
	for (int i = 0; i < batch && !rc; i += most)
	{
		const int part = min(most, batch - i);
		dim3 grid;
		if ((rc = xcd_grid(part, slots, NT3, &grid, name)))
			break;
		hipLaunchKernelGGL((k_trsm_rltn<T, PS, NB, GIVEN>), grid, dim3(NT3), shm, st, args + i, part, slots, nlo, nmax);
		rc = check_launch(name);
		if (batch - i <= most)
			break;   // (i + most may pass the range of an int)
	}
	return rc;
}
template <typename T, int PS, bool GIVEN = false>
static int launch_trsm_ps(int batch, const typename TrsmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	const int nmax = (hint->max_n + 15) / 16 * 16;
	int rc = 0;
	if (nmax > 128)
		rc = launch_trsm_nb<T, PS, 16, GIVEN>(batch, args, hint->max_m, 128, nmax, st, name);
	if (!rc && nmax > 64)
		rc = launch_trsm_nb<T, PS, 8, GIVEN>(batch, args, hint->max_m, 64, nmax, st, name);
	if (!rc)
		rc = launch_trsm_nb<T, PS, 4, GIVEN>(batch, args, hint->max_m, 0, nmax, st, name);
	if (rc || GIVEN)
		return rc;
	hipLaunchKernelGGL((k_trsm_dA<T, PS, false>), dim3(batch), dim3(64), 0, st, args);
	return check_launch(name);
}

// given: the solve of the rows below the diagonal block in the trapezoid
// Cholesky: reciprocals from sA->dA, no cache update (the caller sets use_dA)
template <typename T>
static int launch_trsm(int ps, int batch, const typename TrsmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name, bool given = false)
{
	int rc = check_common(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	if (!hint || hint->max_n <= 0)
		return set_error(BLASFEO_AMD_EINVAL, "%s: hint->max_n (upper bound of n) is required", name);
	if (hint->max_n > TRSM_NMAX)
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: n up to %d supported, got %d", name, TRSM_NMAX, hint->max_n);
	if constexpr (sizeof(T) == 8)
		if (given)
			return ps == 4 ? launch_trsm_ps<T, 4, true>(batch, args, hint, st, name)
			               : launch_trsm_ps<T, 8, true>(batch, args, hint, st, name);
	if (ps == 4)
		return launch_trsm_ps<T, 4>(batch, args, hint, st, name);
	if (ps == 8)
		return launch_trsm_ps<T, 8>(batch, args, hint, st, name);
	if constexpr (sizeof(T) == 4)
		return launch_trsm_ps<T, 16>(batch, args, hint, st, name);
	return BLASFEO_AMD_EINVAL;
}

template <typename T, int PS, int MODE>
static int launch_trsml_ps(int batch, const typename TrsmArg<T>::type *args, dim3 grid, size_t shm, int mmax, bool thin, hipStream_t st, const char *name)
{
	if (thin && mmax <= WAVE)
		hipLaunchKernelGGL((k_trsm_left_thin<T, PS, MODE, 1>), dim3(batch), dim3(WAVE), 0, st, args);
	else if (thin && mmax <= 2 * WAVE)
		hipLaunchKernelGGL((k_trsm_left_thin<T, PS, MODE, 2>), dim3(batch), dim3(WAVE), 0, st, args);
	else if (thin)
		hipLaunchKernelGGL((k_trsm_left_thin<T, PS, MODE, 4>), dim3(batch), dim3(WAVE), 0, st, args);
	else
		hipLaunchKernelGGL((k_trsm_left<T, PS, MODE>), grid, dim3(NT3), shm, st, args, mmax);
	int rc = check_launch(name);
	if (rc)
		return rc;
	hipLaunchKernelGGL((k_trsm_dA<T, PS, true, MODE == TL_LLNU>), dim3(batch), dim3(64), 0, st, args);
	return check_launch(name);
}

template <typename T, int MODE>
static int launch_trsml(int ps, int batch, const typename TrsmArg<T>::type *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	int rc = check_common(ps, batch, args, sizeof(T) == 4, name);
	if (rc || batch == 0)
		return rc;
	if (!hint || hint->max_m <= 0)
		return set_error(BLASFEO_AMD_EINVAL, "%s: hint->max_m (upper bound of m) is required", name);
	if (hint->max_m > trsml_mmax<T>())
		return set_error(BLASFEO_AMD_ETOOBIG, "%s: m up to %d supported, got %d", name, trsml_mmax<T>(), hint->max_m);
	const int mmax = hint->max_m;
	const int mpad = (mmax + 15) / 16 * 16;
	const size_t shm = sizeof(T) * ((size_t)LNC * (mpad + 1) + mpad);
	const int gy = hint->max_n > 0 ? min(64, (hint->max_n + LNC - 1) / LNC) : 1;
	dim3 grid(batch, gy);
	// few right-hand sides (hint->max_n <= 4), m <= 256 and a batch that fills
	// the GPU by itself (8 instances per CU): one wavefront per instance with X
	// in registers.  Smaller batches keep the four-wave block sweep, whose
	// per-instance chain is shorter (SPD solves, factorisation included, 4
	// right-hand sides: 2048 of 256 1037 us with one wavefront against 1066, 512 of
	// 256 389 against 357, 1000 of U{100..200} 332 against 300).
	// The "trsm_thin" knob forces it on (1) or off (2) where it applies.
	const int cus = num_cus() > 0 ? num_cus() : 256;
	const int knob = tune_value(TUNE_TRSM_THIN, 0);
	const bool thin = sizeof(T) == 8 && hint->max_n > 0 && hint->max_n <= THIN_RHS && mmax <= THIN_Q * WAVE
	                  && (knob == 1 || (knob == 0 && batch >= 8 * cus));
	if (ps == 4)
		return launch_trsml_ps<T, 4, MODE>(batch, args, grid, shm, mmax, thin, st, name);
	if (ps == 8)
		return launch_trsml_ps<T, 8, MODE>(batch, args, grid, shm, mmax, thin, st, name);
	return launch_trsml_ps<T, 16, MODE>(batch, args, grid, shm, mmax, thin, st, name);
}

int trsm_rltn_given_dA(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, hipStream_t st, const char *name)
{
	return launch_trsm<double>(ps, batch, args, hint, st, name, true);
}

} // namespace bfa

using namespace bfa;

extern "C" {

int blasfeo_amd_dgemm_nt_batched(int ps, int batch, const blasfeo_amd_dgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<double, OP_NT>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dgemm_nt_batched"); }
int blasfeo_amd_dgemm_nn_batched(int ps, int batch, const blasfeo_amd_dgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<double, OP_NN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dgemm_nn_batched"); }
int blasfeo_amd_dsyrk_ln_batched(int ps, int batch, const blasfeo_amd_dgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<double, OP_SYRK>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dsyrk_ln_batched"); }
int blasfeo_amd_dsyrk_ln_mn_batched(int ps, int batch, const blasfeo_amd_dgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<double, OP_SYRK_MN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dsyrk_ln_mn_batched"); }
int blasfeo_amd_dtrmm_rlnn_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trmm<double>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrmm_rlnn_batched"); }
int blasfeo_amd_dtrsm_rltn_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsm<double>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrsm_rltn_batched"); }
int blasfeo_amd_dtrsm_llnn_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsml<double, TL_LLNN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrsm_llnn_batched"); }
int blasfeo_amd_dtrsm_lltn_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsml<double, TL_LLTN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrsm_lltn_batched"); }
int blasfeo_amd_dtrsm_llnu_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsml<double, TL_LLNU>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrsm_llnu_batched"); }
int blasfeo_amd_dtrsm_lunn_batched(int ps, int batch, const blasfeo_amd_dtrsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsml<double, TL_LUNN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_dtrsm_lunn_batched"); }

int blasfeo_amd_sgemm_nt_batched(int ps, int batch, const blasfeo_amd_sgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<float, OP_NT>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_sgemm_nt_batched"); }
int blasfeo_amd_sgemm_nn_batched(int ps, int batch, const blasfeo_amd_sgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<float, OP_NN>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_sgemm_nn_batched"); }
int blasfeo_amd_ssyrk_ln_batched(int ps, int batch, const blasfeo_amd_sgemm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_gemm<float, OP_SYRK>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_ssyrk_ln_batched"); }
int blasfeo_amd_strsm_rltn_batched(int ps, int batch, const blasfeo_amd_strsm_arg *args, const blasfeo_amd_hint *hint, blasfeo_amd_stream_t s)
{ return launch_trsm<float>(ps, batch, args, hint, (hipStream_t)s, "blasfeo_amd_strsm_rltn_batched"); }

} // extern "C"
