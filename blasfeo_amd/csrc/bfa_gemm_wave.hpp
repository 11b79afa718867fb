// bfa_gemm_wave.hpp -- gemm_nt / gemm_nn / syrk_ln(_mn) with one wavefront per
// output tile and no LDS: operands from global memory straight into the matrix
// cores' registers.
//
// A wave computes a tile of 64 x 64 (E = 4) or 32 x 32 (E = 2) as 16x16
// accumulators.  It forms D^T = B A^T, so that a lane's accumulators are elements of
// one row of D (lane % 16) in four consecutive columns across the lanes of a
// register: with A's rows taken VA at a time (rows VA c .. VA c + VA - 1 of a
// group of 16 VA rows by lane c, one row for each of VA tiles), A is loaded, C
// loaded and D stored in 16-byte pieces, four columns of a panel side by side
// (whole 128-byte lines for ps = 4).  Matrices whose rows do not start on a
// VA-row boundary take the same loop one element at a time.
// The operands of the next DEPTH steps of four K columns are in flight; columns
// past K read the last one and are zeroed in the tail.  Only the 16-row groups
// and 16-column blocks that the tile has are loaded and multiplied (one loop
// per shape), so that the edges cost no products beyond their last block.
// Measured (MI355X; before: 32 x 32 tiles with 8-byte loads up to 256, a 64 x 64
// tile staged through LDS by four waves above): 1024 dgemm_nn of U{64..512}, ps = 8,
// 1925 -> 1117 us (46 TFLOP/s), 256 of 512^3 1697 -> 1030 us (67 TFLOP/s, the rate of
// a large library product here), 8192 sgemm_nt + ssyrk_ln of U{16..256} 1851 -> 1141 us
// (3.3 TB/s, 60 TFLOP/s): bound by the matrix cores and the last blocks' padding.
// 32768 dgemm_nt + dsyrk_ln of U{4..128} 1943 -> 1683 us (4.3 TB/s), 16384 of 64^3
// 698 -> 648 us (4.95 TB/s, a large copy's rate): bound by memory.
#pragma once
#include "bfa_gemm_core.hpp"
#include "bfa_strip.hpp"
#include <type_traits>

namespace bfa {

// tile t of an instance -> (ti, tj); syrk walks the lower tiles column by
// column (tiles ti >= tj, tj < ntj)
template <int OP>
__device__ __forceinline__ void gw_tile(int t, int mt, int nt, int &ti, int &tj)
{
	if (OP == OP_SYRK || OP == OP_SYRK_MN)
	{
		int j = 0, rem = t;
		while (rem >= mt - j)
		{
			rem -= mt - j;
			j++;
		}
		ti = j + rem;
		tj = j;
	}
	else
	{
		ti = t % mt;
		tj = t / mt;
	}
}

template <int OP>
__host__ __device__ __forceinline__ int gw_ntiles(int mt, int nt)
{
	if (OP == OP_SYRK || OP == OP_SYRK_MN)
	{
		const int c = nt < mt ? nt : mt;
		return c * mt - c * (c - 1) / 2;
	}
	return mt * nt;
}

template <typename T, int N> struct VecN { typedef T type __attribute__((ext_vector_type(N))); };
template <typename T> struct VecN<T, 1> { typedef T type; };
template <typename T, int N>
__device__ __forceinline__ T vec_get(const typename VecN<T, N>::type &v, int e)
{
	if constexpr (N == 1)
		return v;
	else
		return v[e];
}

// K steps of operands in flight and waves per SIMD that the kernel is compiled for:
// between 2 and 6 steps and 2 and 6 waves nothing but the least (2 steps of the
// large tile) was more than a few per cent apart.
template <typename T, int E> constexpr int gw_depth() { return E == 4 ? 3 : 4; }
template <typename T, int E> constexpr int gw_waves() { return E == 4 ? (sizeof(T) == 8 ? 2 : 4) : sizeof(T) == 8 ? 5 : 8; }
// rows that a lane takes at a time in a tile of MX 16-row groups
template <typename T, int MX> constexpr int gw_rows() { return MX == 4 && sizeof(T) == 4 ? 4 : 2; }

// A tile and what is right of and below it: m rows, n columns; the views start at the
// tile (B's of gemm_nn at its columns), low is how far it lies below the diagonal.
template <typename T, int PS, typename O>
struct GwArg
{
	StripView<T, PS, O> A, B, C, D;
	int ai, aj, bi, bj, ci, cj, di, dj, m, n, k, low;
	T alpha, beta;
};

// The tile's MX 16-row groups and NY 16-column blocks; VA: rows that a lane takes at a
// time (1: any offsets).
template <typename T, int PS, int OP, int MX, int NY, int VA, int DEPTH, typename O>
__device__ __forceinline__ void gw_body(const GwArg<T, PS, O> &a)
{
	typedef typename Vec4<T>::type V4;
	typedef typename VecN<T, VA>::type VV;
	constexpr int NV = MX / VA;
	constexpr unsigned CS = PS * sizeof(T);
	constexpr bool SY = OP == OP_SYRK || OP == OP_SYRK_MN;
	// (pinned: the columns and rows of the lane's elements, the same for every tile, would
	// be kept in registers across the tiles)
	int lane = lane_id();
	BFA_PIN(lane);
	const int g = lane >> 4, c = lane & 15;
	const int m = a.m, n = a.n, k = a.k;
	const int lastv = (m - 1) & ~(VA - 1);
	auto ldv = [](const StripView<T, PS, O> &v, O o) -> VV { return *(const BFA_GLOBAL VV *)(v.p + o); };
	V4 acc[MX][NY];
#pragma unroll
	for (int x = 0; x < MX; x++)
#pragma unroll
		for (int y = 0; y < NY; y++)
			acc[x][y] = V4{0, 0, 0, 0};
	if (k > 0)
	{
		O ao[NV], bo[NY];
#pragma unroll
		for (int v = 0; v < NV; v++)
			ao[v] = a.A.at(a.ai + min(16 * VA * v + VA * c, lastv), a.aj);
#pragma unroll
		for (int y = 0; y < NY; y++)
		{
			const int j = min(16 * y + strip_row<T>(c), n - 1);
			bo[y] = OP == OP_NN ? (O)(a.bj + j) * CS : a.B.at(a.bi + j, a.bj);
		}
		const int ns = (k + 3) / 4;
		VV av[DEPTH][NV];
		T bv[DEPTH][NY];
		auto load = [&](int s, VV (&x)[NV], T (&y)[NY]) {
			s = min(s, ns - 1);
			const int kq = min(4 * s + g, k - 1);
			const O kc = (O)kq * CS;
			// gemm_nn: the rows of B from the panel of row 4 s on
			StripView<T, PS, O> B = a.B;
			O kb = kc;
			if constexpr (OP == OP_NN)
			{
				B.p += (size_t)((unsigned)(4 * s) / PS) * B.cn * CS;
				kb = B.at(a.bi + kq - ((4 * s) & ~(PS - 1)), 0);
			}
#pragma unroll
			for (int v = 0; v < NV; v++)
				x[v] = ldv(a.A, ao[v] + kc);
#pragma unroll
			for (int t = 0; t < NY; t++)
				y[t] = B.ld(0, bo[t] + kb);
		};
		auto step = [&](const VV (&x)[NV], const T (&y)[NY]) {
#pragma unroll
			for (int v = 0; v < NV; v++)
#pragma unroll
				for (int e = 0; e < VA; e++)
#pragma unroll
					for (int t = 0; t < NY; t++)
						acc[VA * v + e][t] = mfma16(y[t], vec_get<T, VA>(x[v], e), acc[VA * v + e][t]);
		};
#pragma unroll
		for (int d = 0; d < DEPTH; d++)
			load(d, av[d], bv[d]);
		int s = 0;
		for (; s + DEPTH < ns; s += DEPTH)
		{
#pragma unroll
			for (int d = 0; d < DEPTH; d++)
			{
				step(av[d], bv[d]);
				load(s + DEPTH + d, av[d], bv[d]);
			}
		}
		// the last 1 .. DEPTH steps
#pragma unroll
		for (int d = 0; d < DEPTH; d++)
			if (s + d < ns)
			{
				if (4 * (s + d) + 4 > k)
				{
					const bool in = 4 * (s + d) + g < k;
#pragma unroll
					for (int v = 0; v < NV; v++)
						av[d][v] = in ? av[d][v] : VV(0);
#pragma unroll
					for (int t = 0; t < NY; t++)
						bv[d][t] = in ? bv[d][t] : T(0);
				}
				step(av[d], bv[d]);
			}
	}
	// D = beta * C + alpha * acc, a 16-column block at a time: its elements of C are
	// all loaded before any of D is stored (C may be D)
	const bool whole = 16 * MX <= m && 16 * NY <= n && !(SY && a.low < 16 * NY - 1);
#pragma unroll
	for (int y = 0; y < NY; y++)
	{
		VV cv[NV][4];
		if (a.beta != T(0))
		{
#pragma unroll
			for (int v = 0; v < NV; v++)
			{
				const O oc = a.C.at(a.ci + min(16 * VA * v + VA * c, lastv), a.cj);
#pragma unroll
				for (int r = 0; r < 4; r++)
					cv[v][r] = ldv(a.C, oc + (O)min(16 * y + 4 * r + g, n - 1) * CS);
			}
		}
#pragma unroll
		for (int v = 0; v < NV; v++)
		{
			const int gi = 16 * VA * v + VA * c;
			const O od = a.D.at(a.di + min(gi, lastv), a.dj);
#pragma unroll
			for (int r = 0; r < 4; r++)
			{
				const int gj = 16 * y + 4 * r + g;
				const O o = od + (O)min(gj, n - 1) * CS;
				T val[VA];
				VV vv;
#pragma unroll
				for (int e = 0; e < VA; e++)
				{
					val[e] = a.alpha * acc[VA * v + e][y][r];
					if (a.beta != T(0))
						val[e] = a.beta * vec_get<T, VA>(cv[v][r], e) + val[e];
					if constexpr (VA == 1)
						vv = val[e];
					else
						vv[e] = val[e];
				}
				if (whole)
					*(BFA_GLOBAL VV *)(a.D.p + o) = vv;
				else if (gj < n)
				{
					if (gi + VA <= m && !(SY && a.low + gi < gj))
						*(BFA_GLOBAL VV *)(a.D.p + o) = vv;
					else
#pragma unroll
						for (int e = 0; e < VA; e++)
							if (gi + e < m && !(SY && a.low + gi + e < gj))
								*(BFA_GLOBAL T *)(a.D.p + o + e * (unsigned)sizeof(T)) = val[e];
				}
			}
		}
	}
}

// the loop for a tile's nb <= E column blocks
template <typename T, int PS, int OP, int MX, int E, int DEPTH>
__device__ __forceinline__ void gw_blocks(const GwArg<T, PS, unsigned> &a, int nb)
{
	constexpr int VA = gw_rows<T, MX>();
	if constexpr (E == 4)
	{
		if (nb == 4)
			return gw_body<T, PS, OP, MX, 4, VA, DEPTH>(a);
		if (nb == 3)
			return gw_body<T, PS, OP, MX, 3, VA, DEPTH>(a);
	}
	if (nb >= 2)
		return gw_body<T, PS, OP, MX, 2, VA, DEPTH>(a);
	gw_body<T, PS, OP, MX, 1, VA, DEPTH>(a);
}

// One wave per (instance, tile slot): `slots` slots per instance (the tile
// count of the hint's largest instance), a 1-D launch of batch * slots
// workgroups rounded up to a multiple of XCDS.  The slots of one instance
// map to consecutive logical indices on one XCD (xcd_local_index), so the
// tiles that re-read the same A row block or B column block run together
// on one L2; slot t >= the instance's tile count exits at once.
template <typename T, int PS, int OP, int E>
__global__ __launch_bounds__(WAVE, (gw_waves<T, E>())) void k_gemm_wave(const typename GemmArg<T>::type *__restrict__ args, int batch,
	int slots, bool spread)
{
	constexpr int TE = 16 * E, DEPTH = gw_depth<T, E>();
	int inst, slot;
	xcd_inst_slot(slots, inst, slot, spread);
	if (inst >= batch)
		return;
	const typename GemmArg<T>::type &r = args[inst];
	const int m = __builtin_amdgcn_readfirstlane(r.m), n = OP == OP_SYRK ? m : __builtin_amdgcn_readfirstlane(r.n);
	if (m <= 0 || n <= 0)
		return;
	if (threadIdx.x == 0 && slot == 0)
		r.sD->use_dA = 0;
	const int mt = (m + TE - 1) / TE, nt = (n + TE - 1) / TE;
	const int ntiles = gw_ntiles<OP>(mt, nt);
	if (slot >= ntiles)
		return;
	const StripView<T, PS> A = strip_view<T, PS>(r.sA), B = strip_view<T, PS>(r.sB), C = strip_view<T, PS>(r.sC), D = strip_view<T, PS>(r.sD);
	const int k = __builtin_amdgcn_readfirstlane(r.k);
	// the tile at (i0, j0)
	auto tile = [&](auto &a, int i0, int j0) {
		typedef typename std::remove_reference_t<decltype(a.A)>::ofs O;
		a.m = m - i0, a.n = n - j0, a.k = k, a.low = i0 - j0;
		a.ai = r.ai + i0, a.aj = r.aj;
		a.bi = OP == OP_NN ? r.bi : r.bi + j0, a.bj = OP == OP_NN ? r.bj + j0 : r.bj;
		a.ci = r.ci + i0, a.cj = r.cj + j0, a.di = r.di + i0, a.dj = r.dj + j0;
		a.A = A.template block<O>(a.ai, a.aj);
		a.B = B.template block<O>(a.bi, a.bj);
		a.C = C.template block<O>(a.ci, a.cj);
		a.D = D.template block<O>(a.di, a.dj);
		a.alpha = r.alpha;
		a.beta = r.beta;
	};
	if (__builtin_expect(!strip_fits<T, PS>(max(max(A.cn, B.cn), max(C.cn, D.cn))), 0))
	{
		// 32 x 32 at a time: 64-bit offsets of more would not leave the other form
		// its registers
		for (int t = slot; t < ntiles; t += slots)
		{
			int ti, tj;
			gw_tile<OP>(t, mt, nt, ti, tj);
#pragma unroll 1
			for (int q = 0; q < E * E / 4; q++)
			{
				const int i0 = ti * TE + 32 * (q / (E / 2)), j0 = tj * TE + 32 * (q % (E / 2));
				if (i0 < m && j0 < n)
				{
					GwArg<T, PS, size_t> a;
					tile(a, i0, j0);
					gw_body<T, PS, OP, 2, 2, 1, 2>(a);
				}
			}
		}
		return;
	}
	// rows in pieces: the matrices' rows start on a piece's boundary, in memory too
	constexpr int VA = gw_rows<T, E>();
	const unsigned long long low = (unsigned long long)(uintptr_t)A.p | (unsigned long long)(uintptr_t)C.p | (unsigned long long)(uintptr_t)D.p;
	const bool pieces = ((r.ai | r.ci | r.di) & (VA - 1)) == 0 && (low & (VA * sizeof(T) - 1)) == 0;
	for (int t = slot; t < ntiles; t += slots)
	{
		int ti, tj;
		gw_tile<OP>(t, mt, nt, ti, tj);
		const int i0 = ti * TE, j0 = tj * TE;
		GwArg<T, PS, unsigned> a;
		tile(a, i0, j0);
		const int nb = min(E, (a.n + 15) / 16);
		if (!pieces)
			gw_body<T, PS, OP, E, E, 1, 2>(a);
		else if (E == 2 || a.m <= 32)
			gw_blocks<T, PS, OP, 2, E, DEPTH>(a, nb);
		else if constexpr (E == 4)
			gw_blocks<T, PS, OP, 4, E, DEPTH>(a, nb);
	}
}

} // namespace bfa
