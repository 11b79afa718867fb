// bfa_potrf_wave.hpp -- potrf_l, potrf_l_mn and syrk_dpotrf_ln(_mn) on 16-row
// strips held in registers (bfa_strip.hpp): one wavefront per instance, or a
// few that share its strips.
#pragma once
#include "bfa_strip.hpp"
#include <type_traits>

namespace bfa {

// Waves per SIMD that a kernel with NB block accumulators is compiled for.
template <typename T, int NB>
constexpr int strip_waves()
{
	return sizeof(T) * NB <= 16 ? 4 : sizeof(T) * NB <= 64 ? 3 : 2;
}

// The finished part of L that a later strip needs is kept in LDS up to 64
// columns (9 KB), read back from D above.
template <int NB> constexpr bool potrf_wave_lds() { return NB <= 4; }
// LDS values of one wave: the 4 x 4 triangles (64 a block column), and with
// potrf_wave_lds the diagonal blocks (three steps) and the blocks left of them,
// of the strips 0 .. NB - 2
template <int NB>
constexpr int potrf_wave_elems()
{
	return 64 * NB + (potrf_wave_lds<NB>() ? 192 * (NB - 1) + 256 * (NB - 1) * (NB - 2) / 2 : 0);
}

// ---------------------------------------------------------------------------
// One wavefront per instance.  The wave takes the 16-row strips J of the
// trapezoid in order; left to right, block K of the strip is C_JK minus the
// products of its finished blocks p < K with the row block L_K, solved with L_KK;
// the diagonal block takes the strip's own products and is factored.  No barrier:
// the panel chain that one wave of a workgroup ran while the others waited is
// all there is, and the other waves of the SIMD, each with an instance of its own,
// fill its latencies.  NB bounds the block columns (n <= 16 NB).
// Measured (MI355X, 8192 FP64 instances, ps = 4; before: four waves per instance,
// the trapezoid in LDS, one wave factoring the panels): n = 32 40 -> 25 us,
// n = 64 487 -> 86 us, n = 128 1932 -> 480 us, n = 256 3237 -> 2650 us.
// Bound up to 64 columns by the vector instructions of the solves and diagonal
// factorisations (3050 of them and 70 matrix-core steps per wave at n = 64),
// above by memory: the rows of L that are read back miss L2 for the most part
// (n = 128: 1.9 GB read for 0.55 GB of input).
// ---------------------------------------------------------------------------
template <typename T, int PS, int NB, typename O>
__device__ __forceinline__ void potrf_wave(int m, int n, const StripView<T, PS> vC, int ci, int cj,
	const StripView<T, PS> vD, int di, int dj, BFA_GLOBAL T *dD, T *lds)
{
	typedef typename Vec4<T>::type V4;
	constexpr bool LDSL = potrf_wave_lds<NB>();
	const StripView<T, PS, O> C = vC.template block<O>(ci, cj), D = vD.template block<O>(di, dj);
	const int lane = lane_id(), g = lane >> 4, rid = strip_row<T>(lane & 15);
	const int R = (m + 15) / 16, Cb = (n + 15) / 16;
	T *tri = lds, *ldiag = lds + 64 * NB, *ltile = ldiag + 192 * (NB - 1);
	V4 nx[NB];   // -X of the strip's finished blocks
#pragma unroll 1
	for (int J = 0; J < R; J++)
	{
		// (pinned: column and row offsets of all blocks, the same for every
		// strip, would be kept in registers across the strips)
		int gj = g, rj = rid;
		BFA_PIN(gj);
		BFA_PIN(rj);
		const int row = 16 * J + rj, rc = min(row, m - 1);
		const int kend = min(J, Cb);            // blocks left of the diagonal
		const int nblk = min(J + 1, Cb);
		const O oc = C.at(ci + rc, cj + gj), od = D.at(di + rc, dj + gj);
		V4 cn;
		strip_load<4>(C, oc, gj, 0, n, cn);
#pragma unroll 1
		for (int K = 0; K < kend; K++)
		{
			// row block L_K: its steps left of the diagonal from lp / ol
			const T *lp = ltile + 256 * (K * (K - 1) / 2) + lane;
			const O ol = LDSL ? 0 : D.at(di + min(16 * K + rj, m - 1), dj + gj);
			T lk[3], d[4], l[3][4];
			auto load_l = [&](int p, T (&v)[4]) {
				if constexpr (LDSL)
#pragma unroll
					for (int s = 0; s < 4; s++)
						v[s] = lp[256 * p + 64 * s];
				else
					strip_load_full<4>(D, ol, 16 * p, v);
			};
			if (K > 0)
				load_l(0, l[0]);
			if (K > 1)
				load_l(1, l[1]);
			V4 acc = cn;
			if constexpr (LDSL)
#pragma unroll
				for (int s = 0; s < 3; s++)
					lk[s] = ldiag[192 * K + 64 * s + lane];
			else
				strip_load<3>(D, ol, gj, 16 * K, n, lk);
			if (K + 1 < nblk)
				strip_load<4>(C, oc, gj, 16 * (K + 1), n, cn);
#pragma unroll
			for (int s = 0; s < 4; s++)
				d[s] = tri[64 * K + 16 * s + (lane & 15)];
			// two blocks of L in flight
#pragma unroll
			for (int p = 0; p < NB - 1; p++)
				if (p < K)
				{
					if (p + 2 < K)
						load_l(p + 2, l[(p + 2) % 3]);
#pragma unroll
					for (int s = 0; s < 4; s++)
						acc = mfma16(l[p % 3][s], nx[p][s], acc);
				}
			T x[4];
			strip_solve<T>(acc, lk, d, x);
			strip_store(D, od, gj, 16 * K, n, row < m, x);
			if (LDSL && J < NB - 1)
#pragma unroll
				for (int s = 0; s < 4; s++)
					ltile[256 * (J * (J - 1) / 2 + K) + 64 * s + lane] = x[s];
			V4 y;
#pragma unroll
			for (int s = 0; s < 4; s++)
				y[s] = -x[s];
			strip_set(nx, K, y);
		}
		if (J < Cb)
		{
			T l[4], iv[4];
			V4 acc = cn;
#pragma unroll
			for (int p = 0; p < NB - 1; p++)
				if (p < J)
#pragma unroll
					for (int s = 0; s < 4; s++)
						acc = mfma16(-nx[p][s], nx[p][s], acc);
			strip_chol16<T>(acc, l, iv);
			strip_put_tri<T>(tri + 64 * J, l, iv);
			if (LDSL && J < NB - 1)
#pragma unroll
				for (int s = 0; s < 3; s++)
					ldiag[192 * J + 64 * s + lane] = l[s];
			strip_store_diag(D, od, gj, rj, 16 * J, n, row < m, l, dD, iv);
		}
		// the next strips read this one's rows of D (or of LDS) and the triangle
		wave_sync();
	}
}

template <typename T, int PS, int NB>
__global__ __launch_bounds__(WAVE, (strip_waves<T, NB>())) void k_potrf_wave(const typename FactArg<T>::type *__restrict__ args,
	int mmax, bool mn)
{
	__shared__ T lds[potrf_wave_elems<NB>()];
	const typename FactArg<T>::type &a = args[blockIdx.x];
	const int m = __builtin_amdgcn_readfirstlane(a.m);
	const int n = mn ? min(m, __builtin_amdgcn_readfirstlane(a.n)) : m;
	if (m <= 0 || n <= 0 || m > mmax || n > 16 * NB)
		return;
	const StripView<T, PS> C = strip_view<T, PS>(a.sC), D = strip_view<T, PS>(a.sD);
	BFA_GLOBAL T *dD = (BFA_GLOBAL T *)a.sD->dA;
	// narrow offsets where the rows of L are read back (n = 256: 2048 of them 3 per cent)
	if (!potrf_wave_lds<NB>() && __builtin_expect(strip_fits<T, PS>(max(C.cn, D.cn)), 1))
		potrf_wave<T, PS, NB, unsigned>(m, n, C, a.ci, a.cj, D, a.di, a.dj, dD, lds);
	else
		potrf_wave<T, PS, NB, size_t>(m, n, C, a.ci, a.cj, D, a.di, a.dj, dD, lds);
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? (mn ? 1 : m) : 0;
}

// ---------------------------------------------------------------------------
// The same with NW waves per instance, the tiles in registers (chol_coop).
// SYRK: 16 columns of k at a time every wave loads its strips' rows of B, passes
// them to LDS as operand tiles and applies every tile of the chunk to its own
// strips' rows of A, which it loads itself (the same registers where A is B); the
// next chunk's loads are in flight meanwhile.  A and B are read once.
// Measured (MI355X, FP64, ps = 4, before: as above): syrk_dpotrf_ln, 8192 of
// m = k = 64 629 -> 249 us, of m = k = 128 2978 -> 892 us (863 with the sums begun at
// C, whose errors were up to 1.7 times as large); potrf_l, 256 of n = 128 113 -> 35 us,
// of n = 256 268 -> 108 us.  Bound by the chain of
// one diagonal block and one solve per block column (three instances per CU).
// ---------------------------------------------------------------------------
template <typename T, int PS, int NW, bool SYRK>
__device__ __forceinline__ void potrf_coop(int m, int n, int k, const StripView<T, PS> A, int ai, int aj,
	const StripView<T, PS> B, int bi, int bj, bool same, const StripView<T, PS> C, int ci, int cj,
	const StripView<T, PS> D, int di, int dj, BFA_GLOBAL T *dD, T *lds)
{
	typedef typename Vec4<T>::type V4;
	constexpr unsigned CS = StripView<T, PS>::CS;
	const int lane = lane_id(), g = lane >> 4, rid = strip_row<T>(lane & 15);
	const int w = __builtin_amdgcn_readfirstlane(wave_id());
	const int R = (m + 15) / 16, Cb = (n + 15) / 16;
	const int ih = R - 1 - w, il = R - 2 * NW + w;
	const int rh = min(16 * max(ih, 0) + rid, m - 1), rl = min(16 * max(il, 0) + rid, m - 1);
	V4 hi[2 * NW], lo[NW];
	if (SYRK)
	{
#pragma unroll
		for (int J = 0; J < 2 * NW; J++)
			hi[J] = V4{0, 0, 0, 0};
#pragma unroll
		for (int J = 0; J < NW; J++)
			lo[J] = V4{0, 0, 0, 0};
	}
	else
	{
		const size_t oh = C.at(ci + rh, cj + g), ol = C.at(ci + rl, cj + g);
#pragma unroll
		for (int J = 0; J < 2 * NW; J++)
			if (J <= ih && J < Cb)
				strip_load<4>(C, oh, g, 16 * J, n, hi[J]);
#pragma unroll
		for (int J = 0; J < NW; J++)
			if (J <= il && J < Cb)
				strip_load<4>(C, ol, g, 16 * J, n, lo[J]);
	}
	if (SYRK && k > 0)
	{
		// rows of B of a strip past its n rows: row n - 1 again (their columns of
		// the result are past n)
		const size_t ah = A.at(ai + rh, aj + g), al = A.at(ai + rl, aj + g);
		const size_t bh = B.at(bi + min(rh, n - 1), bj + g), bl = B.at(bi + min(rl, n - 1), bj + g);
		// the operands of columns kk .. kk+15, zero past k (nothing is read there)
		auto load = [&](const StripView<T, PS> &v, size_t o, int kk, T (&x)[4]) {
			if (kk + 16 <= k)
#pragma unroll
				for (int s = 0; s < 4; s++)
					x[s] = v.ld((size_t)(kk + 4 * s) * CS, o);
			else
#pragma unroll
				for (int s = 0; s < 4; s++)
				{
					x[s] = T(0);
					if (kk + 4 * s + g < k)
						x[s] = v.ld((size_t)(kk + 4 * s) * CS, o);
				}
		};
		T vh[4] = {}, vl[4] = {}, uh[4] = {}, ul[4] = {};   // rows of A, rows of B
		auto fetch = [&](int kk) {
			if (ih >= 0)
				load(A, ah, kk, vh);
			if (il >= 0)
				load(A, al, kk, vl);
			if (!same)
			{
				if (ih >= 0 && ih < Cb)
					load(B, bh, kk, uh);
				if (il >= 0 && il < Cb)
					load(B, bl, kk, ul);
			}
		};
		fetch(0);
#pragma unroll 1
		for (int kk = 0; kk < k; kk += 16)
		{
			T *buf = lds + ((kk >> 4) & 1) * (2 * NW * 256);
			T ch[4], cl[4];
#pragma unroll
			for (int s = 0; s < 4; s++)
			{
				ch[s] = vh[s];
				cl[s] = vl[s];
				if (ih >= 0)
					buf[256 * ih + 64 * s + lane] = same ? vh[s] : uh[s];
				if (il >= 0)
					buf[256 * il + 64 * s + lane] = same ? vl[s] : ul[s];
			}
			if (kk + 16 < k)
				fetch(kk + 16);
			__syncthreads();
#pragma unroll
			for (int J = 0; J < 2 * NW; J++)
				if (J <= ih && J < Cb)
				{
					T b[4];
#pragma unroll
					for (int s = 0; s < 4; s++)
						b[s] = buf[256 * J + 64 * s + lane];
#pragma unroll
					for (int s = 0; s < 4; s++)
						hi[J] = mfma16(b[s], ch[s], hi[J]);
					if (J < NW && J <= il)
#pragma unroll
						for (int s = 0; s < 4; s++)
							lo[J < NW ? J : 0] = mfma16(b[s], cl[s], lo[J < NW ? J : 0]);
				}
		}
	}
	if (SYRK)
	{
		// C joins last, four tiles at a time with no branch between their loads (columns
		// past n read column n - 1): sums begun at C are rounded at C's size in every
		// step, which made the factors' errors up to 1.7 times as large
		int ge = g, re = rid;
		BFA_PIN(ge);
		BFA_PIN(re);
		auto add = [&](int I, int J0, auto &acc, auto cnt) {
			constexpr int CNT = decltype(cnt)::value;
			if (J0 > I || J0 >= Cb)
				return;
			const size_t o = C.at(ci + min(16 * I + re, m - 1), cj);
			T cv[CNT][4];
#pragma unroll
			for (int t = 0; t < CNT; t++)
#pragma unroll
				for (int s = 0; s < 4; s++)
					cv[t][s] = C.ld(0, o + (size_t)((unsigned)min(16 * (J0 + t) + 4 * s + ge, n - 1) * CS));
#pragma unroll
			for (int t = 0; t < CNT; t++)
#pragma unroll
				for (int s = 0; s < 4; s++)
					acc[J0 + t][s] += cv[t][s];
		};
		typedef std::integral_constant<int, NW < 4 ? NW : 4> Cnt;
#pragma unroll
		for (int J = 0; J < 2 * NW; J += Cnt::value)
			add(ih, J, hi, Cnt());
#pragma unroll
		for (int J = 0; J < NW; J += Cnt::value)
			add(il, J, lo, Cnt());
		// the first column's tiles go to the buffer that the last chunk may still
		// be read from
		__syncthreads();
	}
	auto emit = [&](int I, int J, const T (&x)[4]) {
		int ge = g, re = rid;   // (pinned: nothing of this is kept across the columns)
		BFA_PIN(ge);
		BFA_PIN(re);
		const int row = 16 * I + re;
		strip_store(D, D.at(di + min(row, m - 1), dj + ge), ge, 16 * J, n, row < m, x);
	};
	auto emit_diag = [&](int J, const T (&l)[4], const T (&iv)[4]) {
		const int row = 16 * J + rid;
		strip_store_diag(D, D.at(di + min(row, m - 1), dj + g), g, rid, 16 * J, n, row < m, l, dD, iv);
	};
	chol_coop<T, NW>(hi, lo, ih, il, Cb, CoopRing<T, NW>{lds, lane}, emit, emit_diag);
}

// Waves per SIMD that a kernel with NW waves per instance is compiled for.
template <typename T, int NW>
constexpr int coop_waves()
{
	return sizeof(T) * NW <= 32 ? 3 : 2;
}

template <typename T, int PS, int NW>
__global__ __launch_bounds__(NW * WAVE, (coop_waves<T, NW>())) void k_potrf_coop(const typename FactArg<T>::type *__restrict__ args,
	int mmax, bool mn)
{
	__shared__ T lds[CoopRing<T, NW>::ELEMS];
	const typename FactArg<T>::type &a = args[blockIdx.x];
	const int m = __builtin_amdgcn_readfirstlane(a.m);
	const int n = mn ? min(m, __builtin_amdgcn_readfirstlane(a.n)) : m;
	if (m <= 0 || n <= 0 || m > mmax || m > 32 * NW)
		return;
	const StripView<T, PS> C = strip_view<T, PS>(a.sC), D = strip_view<T, PS>(a.sD);
	potrf_coop<T, PS, NW, false>(m, n, 0, C, 0, 0, C, 0, 0, true, C, a.ci, a.cj, D, a.di, a.dj,
		(BFA_GLOBAL T *)a.sD->dA, lds);
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? (mn ? 1 : m) : 0;
}

template <typename T, int PS, int NW>
__global__ __launch_bounds__(NW * WAVE, (coop_waves<T, NW>())) void k_syrk_potrf_coop(const typename SPArg<T>::type *__restrict__ args, int mmax)
{
	__shared__ T lds[CoopRing<T, NW>::ELEMS];
	const typename SPArg<T>::type &a = args[blockIdx.x];
	const int m = __builtin_amdgcn_readfirstlane(a.m), k = __builtin_amdgcn_readfirstlane(a.k);
	const int n = min(m, __builtin_amdgcn_readfirstlane(a.n));
	if (m <= 0 || n <= 0 || m > mmax || m > 32 * NW || k < 0)
		return;
	const bool same = a.sA == a.sB && a.ai == a.bi && a.aj == a.bj;
	potrf_coop<T, PS, NW, true>(m, n, k, strip_view<T, PS>(a.sA), a.ai, a.aj, strip_view<T, PS>(a.sB), a.bi, a.bj, same,
		strip_view<T, PS>(a.sC), a.ci, a.cj, strip_view<T, PS>(a.sD), a.di, a.dj, (BFA_GLOBAL T *)a.sD->dA, lds);
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? 1 : 0;
}

} // namespace bfa
