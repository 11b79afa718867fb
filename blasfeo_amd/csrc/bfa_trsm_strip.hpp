// bfa_trsm_strip.hpp -- trsm_rltn (D = alpha * B * A^{-T}, A lower n x n,
// blasfeo_ref/x_blas3_ref.c:1642-1752) with the 16-row strips of B in registers
// (bfa_strip.hpp).
//
// A wave holds S strips from their first block column to the last: block K is
// alpha B_K minus the products of the finished blocks with the row block A_K (summed
// before B_K is added, which keeps the rounding of the sum at the size of the
// products), then the solve with A_KK.  The four waves of a workgroup walk the block columns
// together: the tiles of row block A_K are brought to LDS once for all of them, as
// operand tiles, dealt to the waves and loaded one block column ahead (read by
// every wave for itself they came from L2 at a rate that bound the kernel).
// Per block column one barrier.
// Measured (MI355X, 8192 FP64 solves, ps = 4; before: the row block in LDS, one of
// four waves solving the diagonal blocks): m = n = 32 124 -> 56 us, 64 234 -> 169,
// 128 1608 -> 702, 256 15.3 -> 5.0 ms (27 TFLOP/s; every wave reading A for itself
// took 1.4 times as long); m, n ~ U{16..256} 4.60 -> 1.79 ms (1.69 with the sum begun at B_K,
// whose error was 2.4 times as large).  Bound by memory up to 64
// columns, then by the matrix cores and the substitution's vector instructions,
// with two waves per SIMD.
#pragma once
#include "bfa_strip.hpp"
#include "bfa_gemm_core.hpp"

namespace bfa {

constexpr int TRSM_NMAX = 256;

// Strips per wave for NB block columns: NB S block accumulators stay in registers.
template <int NB> constexpr int trsm_strips() { return NB == 8 ? 2 : 1; }
// The whole triangle of A in LDS?
template <int NB> constexpr bool trsm_whole() { return NB <= 4; }
template <typename T, int NB>
constexpr size_t trsm_lds()
{
	return sizeof(T) * 256 * (trsm_whole<NB>() ? NB * (NB + 1) / 2 : 2 * NB);
}
// Waves per SIMD that the kernel is compiled for.
template <typename T, int NB>
constexpr int trsm_waves()
{
	return NB <= 4 ? (sizeof(T) == 8 ? 4 : 5) : sizeof(T) * NB * trsm_strips<NB>() <= 64 ? 3 : 2;
}

// Workgroup (instance, slot) solves the blocks of 64 S rows slot, slot + slots, ...
// of its instance; instances with n outside (nlo, 16 NB] belong to another launch.
// DA_GIVEN: the reciprocal diagonal is read from sA->dA whatever use_dA says
// (the trapezoid Cholesky, whose diagonal block was just factored into the same
// descriptor with its reciprocals stored there).
template <typename T, int PS, int NB, bool DA_GIVEN>
__device__ __forceinline__ void trsm_rows(const typename TrsmArg<T>::type &a, int m, int n, const StripView<T, PS> &vA,
	const StripView<T, PS> &vB, const StripView<T, PS> &vD, int slot, int slots, T *tiles, T *inv_s)
{
	typedef typename Vec4<T>::type V4;
	typedef unsigned O;
	constexpr int S = trsm_strips<NB>(), NW = NT3 / WAVE, NT = NB / NW;
	int ai = a.ai, aj = a.aj;
	const StripView<T, PS, O> A = vA.template block<O>(ai, aj);
	const T alpha = a.alpha;
	// reciprocal diagonal: cached copy when valid at launch, else 1/A_jj
	// (an output aliasing A invalidates the cache first, as in the reference)
	// (through global-memory pointers: a wait for flat loads waits for LDS as well)
	const BFA_GLOBAL typename MatOf<T>::type *sA = (const BFA_GLOBAL typename MatOf<T>::type *)a.sA;
	const bool cached = DA_GIVEN || (a.ai == 0 && a.aj == 0 && a.sD != a.sA && sA->use_dA >= n);
	const BFA_GLOBAL T *dA = (const BFA_GLOBAL T *)sA->dA;
	for (int j = threadIdx.x; j < 16 * NB; j += NT3)
		inv_s[j] = j < n ? (cached ? dA[j] : T(1) / A.ld(0, A.at(ai + j, aj + j))) : T(0);
	const int w = __builtin_amdgcn_readfirstlane(wave_id());
	const int lane = lane_id(), g = lane >> 4, c = lane & 15, rid = strip_row<T>(c);
	const int nb = (n + 15) / 16;
	// where this lane's entries of the 4 x 4 triangles of A_KK (strip_solve) are
	// in the diagonal tile: entry (4 s + tr, 4 s + tc)
	const int tr = c >> 2, tc = c & 3;
	int trio[4];
#pragma unroll
	for (int s = 0; s < 4; s++)
		trio[s] = 64 * s + 16 * tc + strip_row<T>(4 * s + tr);
	if constexpr (trsm_whole<NB>())
	{
		// tile (K, p) at 256 (K (K + 1) / 2 + p), dealt round-robin to the waves
		constexpr int NTT = (NB * (NB + 1) / 2 + NW - 1) / NW;
		const int ntile = nb * (nb + 1) / 2;
		T ta[NTT][4];
#pragma unroll
		for (int t = 0; t < NTT; t++)
			if (w + NW * t < ntile)
			{
				int p = w + NW * t, K = 0;
				while (p > K)
					p -= ++K;
				strip_load<4>(A, A.at(ai + min(16 * K + rid, n - 1), aj + g), g, 16 * p, n, ta[t]);
			}
		bool first = true;
		for (int r0 = slot * 64 * S; r0 < m; r0 += slots * 64 * S)
		{
			// rows from r0 on
			int row[S], bi = a.bi + r0, bj = a.bj, di = a.di + r0, dj = a.dj;
			const int mr = m - r0;
			const StripView<T, PS, O> B = vB.template block<O>(bi, bj), D = vD.template block<O>(di, dj);
			V4 nx[S][NB];   // alpha B, then -X of the finished blocks
#pragma unroll
			for (int t = 0; t < S; t++)
			{
				row[t] = 16 * (S * w + t) + rid;
				const O ob = B.at(bi + min(row[t], mr - 1), bj + g);
#pragma unroll
				for (int K = 0; K < NB; K++)
					if (K < nb)
						strip_load<4>(B, ob, g, 16 * K, n, nx[t][K]);
			}
			if (first)
			{
#pragma unroll
				for (int t = 0; t < NTT; t++)
					if (w + NW * t < ntile)
#pragma unroll
						for (int s = 0; s < 4; s++)
							tiles[256 * (w + NW * t) + 64 * s + lane] = ta[t][s];
				__syncthreads();
				first = false;
			}
			// the waves past the last row have shared in the loads above
			if (16 * S * w >= mr)
				continue;
#pragma unroll
			for (int K = 0; K < NB; K++)
				if (K < nb)
				{
					const T *buf = tiles + 256 * (K * (K + 1) / 2);
					T lk[3], d[4];
#pragma unroll
					for (int s = 0; s < 3; s++)
						lk[s] = buf[256 * K + 64 * s + lane];
#pragma unroll
					for (int s = 0; s < 4; s++)
						d[s] = tr == tc ? inv_s[16 * K + 4 * s + tc] : buf[256 * K + trio[s]];
					V4 acc[S];
#pragma unroll
					for (int t = 0; t < S; t++)
						acc[t] = V4{0, 0, 0, 0};
#pragma unroll
					for (int p = K - 1; p >= 0; p--)
					{
						T l[4];
#pragma unroll
						for (int s = 0; s < 4; s++)
							l[s] = buf[256 * p + 64 * s + lane];
#pragma unroll
						for (int s = 0; s < 4; s++)
#pragma unroll
							for (int t = 0; t < S; t++)
								acc[t] = mfma16(l[s], nx[t][p][s], acc[t]);
					}
#pragma unroll
					for (int t = 0; t < S; t++)
						acc[t] += alpha * nx[t][K];
					T x[S][4];
					if constexpr (S == 2)
						strip_solve2<T>(acc[0], acc[1], lk, d, x[0], x[1]);
					else
						strip_solve<T>(acc[0], lk, d, x[0]);
#pragma unroll
					for (int t = 0; t < S; t++)
					{
						const O od = D.at(di + min(row[t], mr - 1), dj + g);
						strip_store(D, od, g, 16 * K, n, row[t] < mr, x[t]);
#pragma unroll
						for (int s = 0; s < 4; s++)
							nx[t][K][s] = -x[t][s];
					}
				}
		}
		return;
	}
	// tiles w, w + NW, ... of row block K, loaded into registers and, a block
	// column later, to LDS
	T st[NT][4];
	auto fetch = [&](int K) {
		const O ol = A.at(ai + min(16 * K + rid, n - 1), aj + g);
#pragma unroll
		for (int t = 0; t < NT; t++)
			if (w + NW * t <= K)
				strip_load<4>(A, ol, g, 16 * (w + NW * t), n, st[t]);
	};
	auto stage = [&](int K) {
		T *buf = tiles + (K & 1) * (NB * 256);
#pragma unroll
		for (int t = 0; t < NT; t++)
			if (w + NW * t <= K)
#pragma unroll
				for (int s = 0; s < 4; s++)
					buf[256 * (w + NW * t) + 64 * s + lane] = st[t][s];
	};
	for (int r0 = slot * 64 * S; r0 < m; r0 += slots * 64 * S)
	{
		int row[S], bi = a.bi + r0, bj = a.bj, di = a.di + r0, dj = a.dj;
		const int mr = m - r0;
		const StripView<T, PS, O> B = vB.template block<O>(bi, bj), D = vD.template block<O>(di, dj);
		O ob[S];
		V4 nx[S][NB], cn[S];
#pragma unroll
		for (int t = 0; t < S; t++)
		{
			row[t] = 16 * (S * w + t) + rid;
			ob[t] = B.at(bi + min(row[t], mr - 1), bj + g);
			strip_load<4>(B, ob[t], g, 0, n, cn[t]);
		}
		fetch(0);
		stage(0);
		__syncthreads();
#pragma unroll 1
		for (int K = 0; K < nb; K++)
		{
			const T *buf = tiles + (K & 1) * (NB * 256);
			V4 acc[S];
#pragma unroll
			for (int t = 0; t < S; t++)
				acc[t] = V4{0, 0, 0, 0};
			if (K + 1 < nb)
				fetch(K + 1);
			T lk[3], d[4];
#pragma unroll
			for (int s = 0; s < 3; s++)
				lk[s] = buf[256 * K + 64 * s + lane];
#pragma unroll
			for (int s = 0; s < 4; s++)
				d[s] = tr == tc ? inv_s[16 * K + 4 * s + tc] : buf[256 * K + trio[s]];
#pragma unroll
			for (int p = NB - 2; p >= 0; p--)
				if (p < K)
				{
					T l[4];
#pragma unroll
					for (int s = 0; s < 4; s++)
						l[s] = buf[256 * p + 64 * s + lane];
#pragma unroll
					for (int s = 0; s < 4; s++)
#pragma unroll
						for (int t = 0; t < S; t++)
							acc[t] = mfma16(l[s], nx[t][p][s], acc[t]);
				}
#pragma unroll
			for (int t = 0; t < S; t++)
			{
				acc[t] += alpha * cn[t];
				// needed after the next block column's products
				if (K + 1 < nb)
					strip_load<4>(B, ob[t], g, 16 * (K + 1), n, cn[t]);
			}
			T x[S][4];
			if constexpr (S == 2)
				strip_solve2<T>(acc[0], acc[1], lk, d, x[0], x[1]);
			else
				strip_solve<T>(acc[0], lk, d, x[0]);
#pragma unroll
			for (int t = 0; t < S; t++)
			{
				V4 y;
#pragma unroll
				for (int s = 0; s < 4; s++)
					y[s] = -x[t][s];
				strip_set(nx[t], K, y);
			}
			if (K + 1 < nb)
				stage(K + 1);
			__syncthreads();
		}
		// (pinned: the column masks of all blocks would be formed at the start
		// and kept in registers)
		int ge = g;
		BFA_PIN(ge);
#pragma unroll
		for (int t = 0; t < S; t++)
		{
			const O od = D.at(di + min(row[t], mr - 1), dj + g);
#pragma unroll
			for (int K = 0; K < NB; K++)
				if (K < nb)
					strip_store(D, od, ge, 16 * K, n, row[t] < mr, -nx[t][K]);
		}
	}
}

// The rows r0 .. r0+rows-1 and every step-th such block of an instance whose panel strides
// are too large for 32-bit offsets: a thread per row, finished columns read back
// from D.  (The code above with 64-bit offsets spills, and scratch costs the launches
// of small instances that never use it.)
template <typename T, int PS, bool DA_GIVEN>
__device__ __forceinline__ void trsm_rows_wide(const typename TrsmArg<T>::type &a, int m, int n, const StripView<T, PS> &A,
	const StripView<T, PS> &B, const StripView<T, PS> &D, int r0, int rows, int step)
{
	const bool cached = DA_GIVEN || (a.ai == 0 && a.aj == 0 && a.sD != a.sA && a.sA->use_dA >= n);
	const BFA_GLOBAL T *dA = (const BFA_GLOBAL T *)a.sA->dA;
	for (; r0 < m; r0 += step)
		for (int i = r0 + threadIdx.x; i < min(m, r0 + rows); i += NT3)
#pragma unroll 1
			for (int j = 0; j < n; j++)
			{
				T w = T(0);
#pragma unroll 1
				for (int l = 0; l < j; l++)
					w += D.ld(0, D.at(a.di + i, a.dj + l)) * A.ld(0, A.at(a.ai + j, a.aj + l));
				const T d = cached ? dA[j] : T(1) / A.ld(0, A.at(a.ai + j, a.aj + j));
				D.st(0, D.at(a.di + i, a.dj + j), (a.alpha * B.ld(0, B.at(a.bi + i, a.bj + j)) - w) * d);
			}
}

template <typename T, int PS, int NB, bool DA_GIVEN>
__global__ __launch_bounds__(NT3, (trsm_waves<T, NB>())) void k_trsm_rltn(const typename TrsmArg<T>::type *__restrict__ args,
	int batch, int slots, int nlo, int nmax)
{
	extern __shared__ unsigned char smem_raw[];
	T *tiles = reinterpret_cast<T *>(smem_raw);
	__shared__ T inv_s[16 * NB];
	int inst, slot;
	xcd_inst_slot(slots, inst, slot);
	if (inst >= batch)
		return;
	const typename TrsmArg<T>::type &a = args[inst];
	const int m = __builtin_amdgcn_readfirstlane(a.m), n = __builtin_amdgcn_readfirstlane(a.n);
	if (m <= 0 || n <= nlo || n > nmax || n > 16 * NB || slot * 64 * trsm_strips<NB>() >= m)
		return;
	const StripView<T, PS> A = strip_view<T, PS>(a.sA), B = strip_view<T, PS>(a.sB), D = strip_view<T, PS>(a.sD);
	BFA_NEED("s"(a.ai), "s"(a.aj), "s"(a.bi), "s"(a.bj), "s"(a.di), "s"(a.dj), "s"(a.alpha));
	if (__builtin_expect(strip_fits<T, PS>(max(A.cn, max(B.cn, D.cn))), 1))
		trsm_rows<T, PS, NB, DA_GIVEN>(a, m, n, A, B, D, slot, slots, tiles, inv_s);
	else
		trsm_rows_wide<T, PS, DA_GIVEN>(a, m, n, A, B, D, slot * 64 * trsm_strips<NB>(), 64 * trsm_strips<NB>(), slots * 64 * trsm_strips<NB>());
}

} // namespace bfa
