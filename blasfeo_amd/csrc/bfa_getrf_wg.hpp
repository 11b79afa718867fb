// bfa_getrf_wg.hpp -- LU with partial row pivoting (blasfeo_ref/x_lapack_ref.c:1156-1536
// semantics; PIV = false: x_lapack_ref.c:880-1150) of instances of up to 256 rows,
// one workgroup each: one wave up to 64 rows, two up to 128, else four.
//
// By rows and columns of 16 (Crout's order): step J forms the column panel
// C(c0:m, J) - L(c0:m, 0:c0) U(0:c0, J) and, once that is factored, the row panel
// L_JJ^{-1} (C(J, c0+16:n) - L(J, 0:c0) U(0:c0, c0+16:n)).  Both are products over
// all finished columns, so that a wave keeps its tiles in the accumulators from
// the first to the last of them, with operands straight from global memory (L2)
// and no barrier in between; the row panel's blocks are strips of U^T
// (bfa_strip.hpp), solved in the registers that the products leave them in.
// The column panel is factored by one wave with the panel in registers, NQ rows
// of 16 columns per lane.  Rows stay where they are: a row's position is an integer
// beside it, the pivot row's values are broadcast with v_readlane and put aside as a
// row of U, and each step leaves the panel one column narrower, one register
// to the left, so that the loop over the columns needs no register indexing.
// The panel's exchanges reach the finished columns as one permutation of at
// most 32 rows, all loads before the stores.
// Measured (MI355X, dgetrf_rp; before: 16-column panels brought up to date block by
// block with two barriers each, exchanges one after the other): 8192 of
// U{16..256} 3840 -> 2990 us, with the solves of 4 right-hand sides 4600 -> 3600;
// 4096 of 64 479 -> 154 us, 2048 of 128 711 -> 444, 512 of 256 982 -> 632.  The
// products are summed from zero and C joins last: sums begun at C are rounded at C's
// size in every step, and cost registers besides (3180 us of the first batch, errors
// up to 2.5 times as large).  Bound by latency: of 5550 cycles a column of panels
// took with sums begun at C (three workgroups per CU) 1760 were the panel's chain of
// search, reciprocal and broadcast, 1110 the column and 1440 the row panel's products
// and gathers, 700 the exchanges, the rest the panel's way to D and the barriers.
#pragma once
#include "bfa_strip.hpp"

namespace bfa {

constexpr int GLU_M = 256;            // most rows
// Pairs of K steps in flight: with 3 or 4 registers spilled (with the solves and sums begun
// at C 4059 -> 4322, 4437 us).
constexpr int GLU_D = 2;
constexpr int GLU_UL = 18;            // stride of the rows of U put aside

// The upper (float: all) and the lower 32 bits of |v|: the order of the values is that
// of the pairs.
__device__ __forceinline__ unsigned key_hi(double v) { return (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32) & 0x7fffffffu; }
__device__ __forceinline__ unsigned key_lo(double v) { return (unsigned)__builtin_bit_cast(unsigned long long, v); }
__device__ __forceinline__ unsigned key_hi(float v) { return __builtin_bit_cast(unsigned, v) & 0x7fffffffu; }
__device__ __forceinline__ unsigned key_lo(float v) { return 0; }

// wave-wide maximum, in a scalar register
__device__ __forceinline__ unsigned wave_max_u32(unsigned v)
{
	v = max(v, (unsigned)dpp_i<0xb1, 0xf>(0, (int)v));
	v = max(v, (unsigned)dpp_i<0x4e, 0xf>(0, (int)v));
	v = max(v, (unsigned)dpp_i<0x114, 0xf>(0, (int)v));
	v = max(v, (unsigned)dpp_i<0x118, 0xf>(0, (int)v));
	v = max(v, (unsigned)dpp_i<0x142, 0xa>(0, (int)v));
	v = max(v, (unsigned)dpp_i<0x143, 0xc>(0, (int)v));
	return (unsigned)__builtin_amdgcn_readlane((int)v, WAVE - 1);
}

// Columns j0 .. j1-1 (at most W) of the panel: x[q][c] at lane l is column j + c of
// row l + 64 q.  pos: the rows' positions (-1 past the end; < j: rows of U).
// The pivot is the largest |x| of the open rows, the first position of them, never a
// NaN, position j when no entry is larger than zero.  Its search goes over the
// upper 32 bits, one DPP maximum per step; more than one row with the largest of them
// (equal entries, or ones that agree in 20 bits) are told apart one by one.  Every lane
// takes the reciprocal of its own candidate meanwhile.
template <typename T, bool PIV, int NQ, int W>
__device__ __forceinline__ void glu_columns(T (&x)[NQ][16], int (&pos)[NQ], int j0, int j1, int c0, T *P, int ldp, T *Ub, T *invs, int *pivs)
{
	const int lane = lane_id();
#pragma unroll 1
	for (int j = j0; j < j1; j++)
	{
		unsigned long long hit[NQ];
		T xb = x[0][0];
		if (PIV)
		{
			unsigned key[NQ], kb = 0;
			bool open[NQ];
#pragma unroll
			for (int q = 0; q < NQ; q++)
			{
				open[q] = pos[q] >= j && x[q][0] == x[q][0];
				key[q] = open[q] ? key_hi(x[q][0]) : 0u;
				xb = key[q] > kb ? x[q][0] : xb;
				kb = max(kb, key[q]);
			}
			kb = wave_max_u32(kb);
			int count = 0;
#pragma unroll
			for (int q = 0; q < NQ; q++)
			{
				hit[q] = __ballot(open[q] && key[q] == kb);
				count += __builtin_popcountll(hit[q]);
			}
			if (count != 1 || kb == 0)
			{
				unsigned lo = 0;
				int first = 0x7fffffff;
#pragma unroll
				for (int q = 0; q < NQ; q++)
					for (unsigned long long b = hit[q]; b; b &= b - 1)
					{
						const int i = (int)__builtin_ctzll(b);
						const unsigned lv = (unsigned)__builtin_amdgcn_readlane((int)key_lo(x[q][0]), i);
						const int pv = __builtin_amdgcn_readlane(pos[q], i);
						if (lv > lo || (lv == lo && pv < first))
						{
							lo = lv;
							first = pv;
						}
					}
				if (kb == 0 && lo == 0)
					first = j;
#pragma unroll
				for (int q = 0; q < NQ; q++)
				{
					hit[q] = __ballot(pos[q] == first);
					xb = pos[q] == first ? x[q][0] : xb;
				}
			}
		}
		else
		{
			// row j has stayed at its place: lane j of the first slot
			hit[0] = 1ull << j;
#pragma unroll
			for (int q = 1; q < NQ; q++)
				hit[q] = 0;
		}
		const T rb = PIV ? (xb != T(0) ? T(1) / xb : T(0)) : T(1) / xb;
		// the pivot's row to all lanes and, put aside, to U
		T u[W], inv = T(0);
		int pp = j;
#pragma unroll
		for (int c = 0; c < W; c++)
			u[c] = T(0);
#pragma unroll
		for (int q = 0; q < NQ; q++)
			if (hit[q])
			{
				const int lp = (int)__builtin_ctzll(hit[q]);
#pragma unroll
				for (int c = 1; c < W; c++)
					u[c] = readlane(x[q][c], lp);
				inv = readlane(rb, lp);
				pp = __builtin_amdgcn_readlane(pos[q], lp);
				if (lane == lp)
				{
#pragma unroll
					for (int c = 0; c < W; c++)
						Ub[j * GLU_UL + c] = x[q][c];
					invs[j] = rb;
					pivs[j] = c0 + pp;
				}
			}
		// the exchange of positions j and pp, the multipliers, the update
#pragma unroll
		for (int q = 0; q < NQ; q++)
		{
			if (PIV)
				pos[q] = pos[q] == pp ? j : pos[q] == j ? pp : pos[q];
			const T l = x[q][0] * inv;
			if (pos[q] > j)
				P[j * ldp + lane + WAVE * q] = l;
#pragma unroll
			for (int c = 1; c < W; c++)
				x[q][c - 1] = x[q][c] - l * u[c];
		}
	}
}

// One wave factors the panel of R rows (at most 64 NQ) in P: cf pivots.
template <typename T, bool PIV, int NQ>
__device__ __forceinline__ void glu_panel(int R, int cf, int c0, T *P, int ldp, T *Ub, T *invs, int *pivs, int *src)
{
	const int lane = lane_id();
	T x[NQ][16];
	int pos[NQ];
#pragma unroll
	for (int q = 0; q < NQ; q++)
	{
		const int r = lane + WAVE * q;
		pos[q] = r < R ? r : -1;
#pragma unroll
		for (int c = 0; c < 16; c++)
			x[q][c] = P[c * ldp + r];
	}
	// (pinned: the loop would wait for its own stores to LDS where it waits for these)
#pragma unroll
	for (int q = 0; q < NQ; q++)
#pragma unroll
		for (int c = 0; c < 16; c++)
			BFA_PIN(x[q][c]);
	glu_columns<T, PIV, NQ, 16>(x, pos, 0, min(8, cf), c0, P, ldp, Ub, invs, pivs);
	glu_columns<T, PIV, NQ, 8>(x, pos, 8, cf, c0, P, ldp, Ub, invs, pivs);
#pragma unroll
	for (int q = 0; q < NQ; q++)
		if (pos[q] >= 0)
			src[pos[q]] = lane + WAVE * q;
}

// acc[t] = C minus the sum over k < kend (a multiple of 16) of the products of tiles
// t = 0 .. NT-1; ldc(lane, t, r): element r of C's tile t.  The sum begins at zero and C joins
// last: begun at C the sum is rounded at C's size in
// every step, which made the factors' errors 2.4 times as large.
// COLS: the tiles are 16 rows of L each (ot: the lane's row at column g) and share
// 16 columns of U (os: the lane's column at row g, rows of U being rows of panels);
// else the tiles are 16 columns of U each and share 16 rows of L.
template <typename T, int PS, int NT, bool COLS, typename O, typename LDC>
__device__ __forceinline__ void glu_products(const StripView<T, PS, O> &D, const O (&ot)[4], O os, int di, int kend,
	const LDC &ldc, typename Vec4<T>::type (&acc)[4])
{
	constexpr unsigned CS = PS * sizeof(T);
	const int g = lane_id() >> 4;
	T ta[GLU_D][NT][2], sh[GLU_D][2];
	auto load = [&](int k, T (&t)[NT][2], T (&s)[2]) {
		k = min(k, kend - 8);
#pragma unroll
		for (int u = 0; u < 2; u++)
		{
			// column of L and row of U of this step
			const O lc = (unsigned)(k + 4 * u) * CS, ur = D.at(di + k + 4 * u + g, 0);
			s[u] = COLS ? D.ld(0, os + ur) : D.ld(lc, os);
#pragma unroll
			for (int i = 0; i < NT; i++)
				t[i][u] = COLS ? D.ld(lc, ot[i]) : D.ld(0, ot[i] + ur);
		}
	};
	auto step = [&](const T (&t)[NT][2], const T (&s)[2]) {
#pragma unroll
		for (int u = 0; u < 2; u++)
#pragma unroll
			for (int i = 0; i < NT; i++)
				acc[i] = COLS ? mfma16(t[i][u], s[u], acc[i]) : mfma16(s[u], t[i][u], acc[i]);
	};
	static_assert(8 * GLU_D == 16, "kend ends on a whole number of rounds");
	if (kend > 0)
	{
#pragma unroll
		for (int d = 0; d < GLU_D; d++)
			load(8 * d, ta[d], sh[d]);
		for (int k = 0; k + 8 * GLU_D < kend; k += 8 * GLU_D)
		{
#pragma unroll
			for (int d = 0; d < GLU_D; d++)
			{
				step(ta[d], sh[d]);
				load(k + 8 * (GLU_D + d), ta[d], sh[d]);
			}
		}
#pragma unroll
		for (int d = 0; d < GLU_D; d++)
			step(ta[d], sh[d]);
	}
	// (pinned: C's places are looked up when the operands' registers are free)
	int lane = lane_id();
	BFA_PIN(lane);
	T cv[NT][4];
#pragma unroll
	for (int i = 0; i < NT; i++)
#pragma unroll
		for (int r = 0; r < 4; r++)
			cv[i][r] = ldc(lane, i, r);
#pragma unroll
	for (int i = 0; i < NT; i++)
#pragma unroll
		for (int r = 0; r < 4; r++)
			acc[i][r] = cv[i][r] - acc[i][r];
}

template <typename T, int PS, bool COLS, typename O, typename LDC>
__device__ __forceinline__ void glu_sum(int nt, const StripView<T, PS, O> &D, const O (&ot)[4], O os, int di, int kend,
	const LDC &ldc, typename Vec4<T>::type (&acc)[4])
{
	if (nt == 4)
		glu_products<T, PS, 4, COLS>(D, ot, os, di, kend, ldc, acc);
	else if (nt == 3)
		glu_products<T, PS, 3, COLS>(D, ot, os, di, kend, ldc, acc);
	else if (nt == 2)
		glu_products<T, PS, 2, COLS>(D, ot, os, di, kend, ldc, acc);
	else if (nt == 1)
		glu_products<T, PS, 1, COLS>(D, ot, os, di, kend, ldc, acc);
}

// a wave-uniform offset in a scalar register
template <typename O>
__device__ __forceinline__ O glu_uniform(size_t v)
{
	if constexpr (sizeof(O) == 8)
		return uniform_u64(v);
	else
		return (O)__builtin_amdgcn_readfirstlane((int)v);
}

// What the waves of a workgroup share besides the panel.
template <typename T, int NW>
struct GluShared
{
	T Ub[16 * GLU_UL], invs[16];
	size_t mdst[32], msrc[32];   // the moved rows' places, byte offsets
	int pivs[16], perm[NW * WAVE], src[NW * WAVE], mrow[32], mperm[32], mcount;
};

template <typename T, int PS, bool PIV, int NW, typename O>
__device__ __forceinline__ void glu_instance(const typename FactArg<T>::type &a, int m, int n, const StripView<T, PS> &vC,
	const StripView<T, PS> &vD, T *P, GluShared<T, NW> &sh)
{
	typedef typename Vec4<T>::type V4;
	constexpr int NTH = NW * WAVE, LDP = NTH + 1;   // P: [16][LDP], rows from c0 on
	constexpr unsigned CS = PS * sizeof(T);
	T *const Ub = sh.Ub, *const invs = sh.invs;
	int *const pivs = sh.pivs, *const perm = sh.perm, *const src = sh.src, *const mrow = sh.mrow, *const mperm = sh.mperm;
	int &mcount = sh.mcount;
	size_t *const mdst = sh.mdst, *const msrc = sh.msrc;
	int ci = a.ci, cj = a.cj, di = a.di, dj = a.dj;
	const StripView<T, PS, O> C = vC.template block<O>(ci, cj), D = vD.template block<O>(di, dj);
	// in place (the same elements, through whatever descriptors and offsets): the rows
	// of C still to come are exchanged too, and perm stays
	const bool inplace = C.p == D.p && ci == di && C.cn == D.cn;
	BFA_GLOBAL T *dD = (BFA_GLOBAL T *)a.sD->dA;
	BFA_GLOBAL int *ipiv = (BFA_GLOBAL int *)a.ipiv;
	const int p = min(m, n);
	const int w = __builtin_amdgcn_readfirstlane(wave_id());
	// the wave that factors the panels: another SIMD for each of a CU's workgroups
	const int fw = (int)((blockIdx.x ^ blockIdx.x >> 2 ^ blockIdx.x >> 8) & (NW - 1));

	if ((int)threadIdx.x < m)
		perm[threadIdx.x] = threadIdx.x;
	__syncthreads();
#pragma unroll 1
	for (int c0 = 0; c0 < p; c0 += 16)
	{
		const int cw = min(16, n - c0), cf = min(16, p - c0), R = m - c0;
		// (pinned, here and below: what follows from the lane would be formed ahead
		// of the loop and kept, more than the registers hold)
		int lane = lane_id();
		BFA_PIN(lane);
		{
			const int g = lane >> 4, c = lane & 15, rid = strip_row<T>(c);
			// column panel: row tiles w, w + 4, ... of 16
			const int nt = min(4, max(0, ((R + 15) / 16 - w + NW - 1) / NW));
			O ot[4];
			V4 acc[4];
#pragma unroll
			for (int t = 0; t < 4; t++)
				acc[t] = V4{0, 0, 0, 0}, ot[t] = D.at(di + min(c0 + 16 * (w + NW * t) + rid, m - 1), dj + g);
			auto ldc = [&](int l, int t, int r) {
				return C.ld(0, C.at(ci + perm[min(c0 + 16 * (w + NW * t) + 4 * r + (l >> 4), m - 1)], cj + min(c0 + (l & 15), n - 1)));
			};
			glu_sum<T, PS, true>(nt, D, ot, (O)(dj + min(c0 + c, n - 1)) * CS, di, c0, ldc, acc);
#pragma unroll
			for (int t = 0; t < 4; t++)
				if (t < nt)
#pragma unroll
					for (int r = 0; r < 4; r++)
						P[c * LDP + 16 * (w + NW * t) + 4 * r + g] = acc[t][r];
			if (w == 0 && lane == 0)
				mcount = 0;
		}
		__syncthreads();
		if (w == fw)
		{
			if (NW == 4 && R > 128)
				glu_panel<T, PIV, 4>(R, cf, c0, P, LDP, Ub, invs, pivs, src);
			else if (NW >= 2 && R > 64)
				glu_panel<T, PIV, 2>(R, cf, c0, P, LDP, Ub, invs, pivs, src);
			else
				glu_panel<T, PIV, 1>(R, cf, c0, P, LDP, Ub, invs, pivs, src);
		}
		__syncthreads();
		// element (i, j) of the factored panel, i at its position
		auto lu = [&](int i, int j) -> T {
			return i < cf && j >= i ? Ub[i * GLU_UL + j - i] : P[j * LDP + src[i]];
		};
		BFA_PIN(lane);
		{
			// the panel to D, in strips of 16 rows
			const int g = lane >> 4, c = lane & 15;
			const O oc = (O)(dj + c0 + g) * CS;
#pragma unroll
			for (int t = 0; t < 4; t++)
			{
				const int i = 16 * (w + NW * t) + c;
				if (16 * (w + NW * t) < R)
				{
					const int si = src[min(i, R - 1)];
					const O od = D.at(di + c0 + min(i, R - 1), 0) + oc;
					T v[4];
#pragma unroll
					for (int s = 0; s < 4; s++)
						v[s] = i < cf && 4 * s + g >= i ? Ub[i * GLU_UL + 4 * s + g - i] : P[(4 * s + g) * LDP + si];
#pragma unroll
					for (int s = 0; s < 4; s++)
						if (i < R && 4 * s + g < cw)
							D.st(4 * s * CS, od, v[s]);
				}
			}
		}
		const int tid = w * WAVE + lane;
		if (tid < cf)
		{
			if (PIV)
				ipiv[c0 + tid] = pivs[tid];
			dD[c0 + tid] = invs[tid];
		}
		if (PIV)
		{
			// the moved rows
			const int i = tid;
			if (i < R && src[i] != i)
			{
				const int k = atomicAdd(&mcount, 1);
				mdst[k] = D.at(di + c0 + i, 0);
				msrc[k] = D.at(di + c0 + src[i], 0);
				mrow[k] = c0 + i;
				mperm[k] = perm[c0 + src[i]];
			}
			__syncthreads();
			const int nm = __builtin_amdgcn_readfirstlane(mcount);
			if (nm > 0)
			{
				const int ncol = inplace ? c0 + max(0, n - c0 - 16) : c0;
				for (int kb = 0; kb < ncol; kb += NTH)
				{
					const int k0 = kb + tid;
					const bool in = k0 < ncol;
					const O oc = (O)(dj + (!in ? 0 : k0 < c0 ? k0 : k0 + 16)) * CS;
					T v[32];
#pragma unroll
					for (int u = 0; u < 32; u++)
						v[u] = D.ld(glu_uniform<O>(msrc[min(u, nm - 1)]), oc);
					wave_sync();   // the rows' places looked up after the loads
#pragma unroll
					for (int u = 0; u < 32; u++)
						if (u < nm)
						{
							const O od = glu_uniform<O>(mdst[u]);
							if (in)
								D.st(od, oc, v[u]);
						}
				}
				if (!inplace && tid < nm)
					perm[mrow[tid]] = mperm[tid];
			}
		}
		if (c0 + 16 < n)
		{
			__syncthreads();
			BFA_PIN(lane);
			const int g = lane >> 4, c = lane & 15, rid = strip_row<T>(c);
			const O os = D.at(di + min(c0 + rid, m - 1), dj + g);
			const int ntc = (n - c0 - 1) / 16;   // column tiles right of the panel
#pragma unroll 1
			for (int t0 = w; t0 < ntc; t0 += 4 * NW)
			{
				const int nt = min(4, (ntc - t0 + NW - 1) / NW);
				O ot[4];
				V4 acc[4];
#pragma unroll
				for (int t = 0; t < 4; t++)
					acc[t] = V4{0, 0, 0, 0}, ot[t] = (O)(dj + min(c0 + 16 * (t0 + NW * t + 1) + c, n - 1)) * CS;
				auto ldc = [&](int l, int t, int s) {
					return C.ld(0, C.at(ci + perm[min(c0 + 4 * s + (l >> 4), m - 1)], cj + min(c0 + 16 * (t0 + NW * t + 1) + (l & 15), n - 1)));
				};
				glu_sum<T, PS, false>(nt, D, ot, os, di, c0, ldc, acc);
				// the factored diagonal block for strip_solve; its 4 x 4 triangles
				// with unit reciprocals
				T l[3], d[4];
				const int tr = c >> 2, tc = c & 3;
#pragma unroll
				for (int s = 0; s < 3; s++)
					l[s] = rid > 4 * s + g && rid < cf ? lu(rid, 4 * s + g) : T(0);
#pragma unroll
				for (int s = 0; s < 4; s++)
					d[s] = tr > tc && 4 * s + tr < cf ? lu(4 * s + tr, 4 * s + tc) : T(1);
#pragma unroll
				for (int t = 0; t < 4; t++)
					if (t < nt)
					{
						T x[4];
						strip_solve<T>(acc[t], l, d, x);
						const int j = c0 + 16 * (t0 + NW * t + 1) + c;
#pragma unroll
						for (int s = 0; s < 4; s++)
							if (j < n && 4 * s + g < cf)
								D.st(0, D.at(di + c0 + 4 * s + g, dj + j), x[s]);
					}
			}
		}
		__syncthreads();
	}
}

template <typename T, int PS, bool PIV, int NW>
__global__ __launch_bounds__(NW * WAVE, sizeof(T) == 8 ? 3 : 4) void k_getrf_wg(const typename FactArg<T>::type *__restrict__ args, int mmax,
	int batch, const int *__restrict__ counts, const int *__restrict__ lists)
{
	extern __shared__ unsigned char smem_raw[];
	T *P = reinterpret_cast<T *>(smem_raw);
	__shared__ GluShared<T, NW> sh;
	const int inst = __builtin_amdgcn_readfirstlane(getrf_order(blockIdx.x, batch, counts, lists));
	if (inst < 0)
		return;
	const typename FactArg<T>::type &a = args[inst];
	const int m = __builtin_amdgcn_readfirstlane(a.m), n = __builtin_amdgcn_readfirstlane(a.n);
	if (threadIdx.x == 0)
		a.sD->use_dA = (a.di == 0 && a.dj == 0) ? 1 : 0;
	if (m <= 0 || n <= 0 || m > mmax || m > NW * WAVE)
		return;
	const StripView<T, PS> C = strip_view<T, PS>(a.sC), D = strip_view<T, PS>(a.sD);
	if (__builtin_expect(strip_fits<T, PS>(max(C.cn, D.cn)), 1))
		glu_instance<T, PS, PIV, NW, unsigned>(a, m, n, C, D, P, sh);
	else
		glu_instance<T, PS, PIV, NW, size_t>(a, m, n, C, D, P, sh);
}

} // namespace bfa
