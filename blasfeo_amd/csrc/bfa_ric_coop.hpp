// bfa_ric_coop.hpp -- the backward Riccati sweep with the stage matrix in
// registers: NW waves per instance share the 16-row strips of a stage
// (bfa_strip.hpp: chol_coop), 2 NW strips at most.
//
// Stage k, wave w with the strips ih and il:
//   W_I = BAbt_I Lxx        the strip's rows of BAbt (registers, loaded during the
//                           previous stage's Cholesky) times the previous factor
//                           (LDS tiles); the result replaces them, and goes to LDS
//                           as operand tiles for the other strips
//   M_IJ = RSQ_IJ + W_I W_J^T   summed from zero, RSQ added last: sums begun at RSQ are
//                           rounded at its size in every step
//   L = chol(M)             chol_coop; its column tiles are the LDS tiles that the
//                           next stage's product reads
// Barriers: one after W, one per block column of the Cholesky and two before
// it.  Sizes, descriptors and the BAbt strips of the next stage are loaded one
// stage ahead.  With one wave (stages of one or two strips, shorter than the
// memory latency) RSQ is too, and a factor is written to memory from its LDS tiles
// in the next stage, before its Cholesky: a load issued behind stores is waited
// for together with them (N = 20, nx = 8, nu = 3, one instance: 80 -> 68 us).
// LDS: the lower tiles of L (16 x 17), the tiles of W but the last strip's, which
// no other strip reads.
// Measured (MI355X; before: the stage matrix in LDS, its panels factored by one of
// the waves, nine launches a call): 8192 x N = 20, nx ~ U{8..64}, nu ~ U{2..16}
// 5.47 -> 4.49 ms, 2048 sv of N = 15, nx ~ U{6..40} 1.33 -> 0.93 ms, one instance
// of N = 20, nx = 8, nu = 3 203 -> 79 us (whole calls).  Bound by instruction issue (about two
// thirds of the SIMDs' cycles on the first batch: 78 cycles per matrix-core step,
// 1830 per 16 x 16 diagonal block, 560 per strip and column solve) and by the
// chain solve - diagonal block of each block column (about 5000 cycles).
#pragma once
#include "bfa_strip.hpp"

namespace bfa {

// Tiles of the factor kept by column-major 16 x 17 tiles: read as operands by the
// Cholesky and, at any row and column offset, by the next stage's product.
template <typename T>
struct CoopLower
{
	static constexpr int DSTEPS = 4;
	T *p, *t;   // tiles; 4 x 4 triangles of two diagonal blocks
	int lane;
	__device__ __forceinline__ T *tile(int I, int j) const { return p + ric_tix(I, j) * RT_SZ; }
	__device__ __forceinline__ int at(int s) const { return RT_LD * (4 * s + (lane >> 4)) + strip_row<T>(lane & 15); }
	__device__ __forceinline__ T *diag(int j) const { return tile(j, j); }
	__device__ __forceinline__ T *tri(int j) const { return t + (j & 1) * 64; }
};

// LDS values for an instance of R strips and nxt state tiles at most.  The first
// two hold a zero (the product's operand above the diagonal) and padding; then
// the 4 x 4 triangles and the reciprocal diagonal.
constexpr int RC_TRI = 2, RC_INV = RC_TRI + 128, RC_TILES = RC_INV + 128;   // (ric_beyond takes 512 of at least 530)
__host__ __device__ constexpr int ric_coop_elems(int R, int nxt)
{
	return RC_TILES + R * (R + 1) / 2 * RT_SZ + (R > 0 ? R - 1 : 0) * nxt * 256;
}

// largest of the lanes' values, in every lane
__device__ __forceinline__ int wave_max_i(int v)
{
	v = max(v, dpp_i<0xb1, 0xf>(v, v));
	v = max(v, dpp_i<0x4e, 0xf>(v, v));
	v = max(v, dpp_i<0x114, 0xf>(v, v));
	v = max(v, dpp_i<0x118, 0xf>(v, v));
	v = max(v, dpp_i<0x142, 0xa>(v, v));
	v = max(v, dpp_i<0x143, 0xc>(v, v));
	return __builtin_amdgcn_readlane(v, WAVE - 1);
}

// The fields of a record that the sweep reads, wave-uniform: read from the record
// at every use they would be loaded and waited for in every stage.
struct RicRec
{
	const int *nx, *nu;
	blasfeo_dmat *BAbt, *RSQrq, *L, *work;
};
template <typename ArgT>
__device__ __forceinline__ RicRec ric_rec(const ArgT &a)
{
	auto p = [](auto *q) { return (decltype(q))(uintptr_t)uniform_u64((unsigned long long)(uintptr_t)q); };
	return RicRec{p(a.nx), p(a.nu), p(a.BAbt), p(a.RSQrq), p(a.L), p(ric_work(a))};
}

// max(nu + nx), max(nx) over the stages and the smallest size (negative: bad),
// every lane a stage
__device__ __forceinline__ void ric_sizes(const RicRec &a, int N, int &nk, int &nx, int &least)
{
	const BFA_GLOBAL int *gx = (const BFA_GLOBAL int *)a.nx, *gu = (const BFA_GLOBAL int *)a.nu;
	int mk = 0, mx = 0, lo = 0;
	for (int k = lane_id(); k <= N; k += WAVE)
	{
		const int x = gx[k], u = k < N ? gu[k] : 0;
		mk = max(mk, x + u);
		mx = max(mx, x);
		lo = max(lo, max(-x, -u));
	}
	nk = wave_max_i(mk);
	nx = wave_max_i(mx);
	least = -wave_max_i(lo);
}

// What a stage needs of its descriptors, wave-uniform.
template <int PS>
struct RicStage
{
	int nx, nu;
	StripView<double, PS> C, R, L;   // BAbt[k], RSQrq[k], L[k]
	unsigned long long dA;           // L[k].dA
};
// The dwords of the three descriptors of stage k and its sizes, one per lane
// (BAbt[k] is not read for k = N).
__device__ __forceinline__ int ric_fetch(const RicRec &a, int N, int k)
{
	const int lane = lane_id(), q = lane >> 4, i = min(lane & 15, (int)(sizeof(blasfeo_dmat) / 4) - 1);
	const char *p;
	if (q == 0)
		p = k < N ? (const char *)(a.BAbt + k) + 4 * i : (const char *)(a.nx + k);
	else if (q == 1)
		p = (const char *)(a.RSQrq + k) + 4 * i;
	else if (q == 2)
		p = (const char *)(a.L + k) + 4 * i;
	else
		p = (lane & 15) == 1 && k < N ? (const char *)(a.nu + k) : (const char *)(a.nx + k);
	return *(const BFA_GLOBAL int *)p;
}
template <int PS>
__device__ __forceinline__ RicStage<PS> ric_stage(int raw, bool last)
{
	auto u64 = [&](int l) {
		return (unsigned long long)(unsigned)__builtin_amdgcn_readlane(raw, l) |
			((unsigned long long)(unsigned)__builtin_amdgcn_readlane(raw, l + 1) << 32);
	};
	auto view = [&](int q) {
		StripView<double, PS> v;
		v.p = (BFA_GLOBAL char *)(uintptr_t)u64(16 * q + 2);
		v.cn = (unsigned)__builtin_amdgcn_readlane(raw, 16 * q + 9);
		return v;
	};
	static_assert(offsetof(blasfeo_dmat, pA) == 8 && offsetof(blasfeo_dmat, dA) == 16 && offsetof(blasfeo_dmat, cn) == 36, "dwords of a descriptor");
	RicStage<PS> s;
	s.C = view(0);
	s.R = view(1);
	s.L = view(2);
	s.dA = u64(32 + 4);
	s.nx = __builtin_amdgcn_readlane(raw, 48);
	s.nu = last ? 0 : __builtin_amdgcn_readlane(raw, 49);
	return s;
}

// One instance.  The caller has checked that it fits: at most 2 NW strips
// (of nu + nx rows, one more with AUG), 16 NX states, lds for its largest stage.
// AUG: the augmented matrices of d_back_ric_sv_libstr (one more row, the linear
// terms), as in ric_sweep_lds.
template <int PS, int NW, int NX, bool AUG>
__device__ __forceinline__ void ric_coop(const RicRec &a, int N, int nkmax, double *lds)
{
	typedef d4_t V4;
	constexpr int XR = AUG ? 1 : 0;
	constexpr unsigned CS = StripView<double, PS>::CS;
	const int lane = lane_id(), g = lane >> 4, c = lane & 15;
	// wave 0 has the last strip, the most work: every other workgroup of a CU
	// (they come 256 apart) deals its strips to its waves in reverse, so that not
	// all of them load the same SIMD most
	const int w0 = __builtin_amdgcn_readfirstlane(wave_id());
	const int w = (blockIdx.x >> 8) & 1 ? NW - 1 - w0 : w0;
	const int Rmax = (nkmax + XR + 15) / 16;
	const CoopLower<double> lay{lds + RC_TILES, lds + RC_TRI, lane};
	double *W = lds + RC_TILES + Rmax * (Rmax + 1) / 2 * RT_SZ;   // tile (I, C) at 256 (I NX + C)
	V4 hi[2 * NW], lo[NW], bh[NX], bl[NX];

	auto strips = [&](int nk, int &R, int &ih, int &il) {
		R = (nk + XR + 15) / 16;
		ih = R - 1 - w;
		il = R - 2 * NW + w;
	};
	// the strip's rows of BAbt, columns past n1 zero
	auto load_b = [&](const StripView<double, PS> &v, int I, int m, int n1, V4 (&b)[NX]) {
		const size_t o = v.at(min(16 * I + c, m - 1), g);
#pragma unroll
		for (int C = 0; C < NX; C++)
			if (16 * C < n1)
			{
				if (16 * C + 16 <= n1)
					strip_load_full<4>(v, o, 16 * C, b[C]);
				else
#pragma unroll
					for (int s = 0; s < 4; s++)
					{
						b[C][s] = 0.0;
						if (16 * C + 4 * s + g < n1)
							b[C][s] = v.ld((size_t)(16 * C + 4 * s) * CS, o);
					}
			}
	};

	int raw = ric_fetch(a, N, N);
	RicStage<PS> st = ric_stage<PS>(raw, true);
	if (N > 0)
		raw = ric_fetch(a, N, N - 1);
	int n1 = 0, u1 = 0;   // sizes of stage k + 1
	// RSQ[k], added to the products at the end
	auto load_m = [&](const RicStage<PS> &q, V4 (&th)[2 * NW], V4 (&tl)[NW]) {
		const int nk = q.nu + q.nx, m = nk + XR;
		int R, ih, il;
		strips(nk, R, ih, il);
		if (nk <= 0)
			return;
		int gk = g, ck = c;   // (pinned: offsets of all blocks are not kept across the stages)
		BFA_PIN(gk);
		BFA_PIN(ck);
		const size_t oh = q.R.at(min(16 * max(ih, 0) + ck, m - 1), gk), ol = q.R.at(min(16 * max(il, 0) + ck, m - 1), gk);
#pragma unroll
		for (int J = 0; J < 2 * NW; J++)
			if (J <= ih && 16 * J < nk)
				strip_load<4>(q.R, oh, gk, 16 * J, nk, th[J]);
#pragma unroll
		for (int J = 0; J < NW; J++)
			if (J <= il && 16 * J < nk)
				strip_load<4>(q.R, ol, gk, 16 * J, nk, tl[J]);
	};
	// L[k] of a finished stage from its LDS tiles to memory, each wave its strips
	auto store_l = [&](const RicStage<PS> &q) {
		const int nk = q.nu + q.nx, m = nk + XR;
		int R, ih, il;
		strips(nk, R, ih, il);
		int gk = g, ck = c;
		BFA_PIN(gk);
		BFA_PIN(ck);
		auto strip = [&](int I) {
			const int row = 16 * I + ck;
			const size_t o = q.L.at(min(row, m - 1), gk);
#pragma unroll 1
			for (int J = 0; J <= I && 16 * J < nk; J++)
			{
				const double *t = lay.tile(I, J);
				double x[4];
#pragma unroll
				for (int s = 0; s < 4; s++)
					x[s] = t[lay.at(s)];
				if (J < I)
					strip_store(q.L, o, gk, 16 * J, nk, row < m, x);
				else
				{
					double iv[4];
#pragma unroll
					for (int s = 0; s < 4; s++)
						iv[s] = lds[RC_INV + 16 * J + 4 * s + gk];
					strip_store_diag(q.L, o, gk, ck, 16 * J, nk, row < m, x, (BFA_GLOBAL double *)(uintptr_t)q.dA, iv);
				}
			}
		};
		if (ih >= 0)
			strip(ih);
		if (il >= 0)
			strip(il);
	};
	// a small stage's RSQ is loaded before the previous stage's Cholesky too
	constexpr bool AHEAD = NW == 1;
	V4 ph[AHEAD ? 2 * NW : 1], pl[AHEAD ? NW : 1];
	if constexpr (AHEAD)
		load_m(st, ph, pl);
	RicStage<PS> done = st;   // (AHEAD) the finished stage whose L is still in LDS only
#pragma unroll 1
	for (int k = N; k >= 0; k--)
	{
		const int nk = st.nu + st.nx, m = nk + XR;
		int R, ih, il;
		strips(nk, R, ih, il);
		const int Cb = (nk + 15) / 16;
		if constexpr (AHEAD)
		{
#pragma unroll
			for (int J = 0; J < 2 * NW; J++)
				hi[J] = ph[J];
#pragma unroll
			for (int J = 0; J < NW; J++)
				lo[J] = pl[J];
		}
		else
			load_m(st, hi, lo);
		if (k < N && n1 > 0)
		{
			// W_I = BAbt_I Lxx, Lxx = L[k+1](u1.., u1..): column tile C from the
			// inner tiles K >= C, in place (b[C] is not needed after it)
			const int n1t = (n1 + 15) / 16;
			int gk = g, ck = c;
			BFA_PIN(gk);
			BFA_PIN(ck);
			if (ih >= 0)
			{
#pragma unroll
				for (int C = 0; C < NX; C++)
					if (C < n1t)
					{
						const int jv = 16 * C + ck, cc = u1 + min(jv, n1 - 1);
						const int hcol = (cc >> 4) * RT_SZ + (cc & 15) * RT_LD;
						V4 ah = V4{0, 0, 0, 0}, al = V4{0, 0, 0, 0};
#pragma unroll
						for (int K = C; K < NX; K++)
							if (K < n1t)
							{
								double x[4];
#pragma unroll
								for (int s = 0; s < 4; s++)
								{
									const int lk = 16 * K + 4 * s + gk, rr = u1 + min(lk, n1 - 1), r = rr >> 4;
									// lds[1] is the zero above the diagonal
									x[s] = lds[lk >= jv ? RC_TILES + r * (r + 1) / 2 * RT_SZ + (rr & 15) + hcol : 1];
								}
#pragma unroll
								for (int s = 0; s < 4; s++)
								{
									ah = mfma16(x[s], bh[K][s], ah);
									if (il >= 0)
										al = mfma16(x[s], bl[K][s], al);
								}
							}
						if (AUG && w == 0)
						{
							// the linear term's row of the previous factor (blasfeo_dgead):
							// W(nk, :) += L[k+1](u1 + n1, u1:), row nk in the last strip
							const int rr = u1 + n1;
#pragma unroll
							for (int s = 0; s < 4; s++)
							{
								const int cl = 16 * C + 4 * s + gk, cx = u1 + cl;
								if (ck == (nk & 15) && cl < n1)
									ah[s] += lds[RC_TILES + ric_tix(rr >> 4, cx >> 4) * RT_SZ + (cx & 15) * RT_LD + (rr & 15)];
							}
						}
						bh[C] = ah;
						bl[C] = al;
						if (w > 0)
#pragma unroll
							for (int s = 0; s < 4; s++)
								W[256 * (ih * NX + C) + 64 * s + lane] = ah[s];
						if (il >= 0)
#pragma unroll
							for (int s = 0; s < 4; s++)
								W[256 * (il * NX + C) + 64 * s + lane] = al[s];
					}
			}
			__syncthreads();
			// M_IJ += W_I W_J^T, a tile's products summed from zero (begun at RSQ they
			// are rounded at its size in every step)
#pragma unroll
			for (int J = 0; J < 2 * NW; J++)
				if (J <= ih && J < Cb)
				{
					V4 ah = V4{0, 0, 0, 0}, al = V4{0, 0, 0, 0};
#pragma unroll
					for (int C = 0; C < NX; C++)
						if (C < n1t)
						{
							double x[4];
							if (J == R - 1)
#pragma unroll
								for (int s = 0; s < 4; s++)
									x[s] = bh[C][s];
							else
#pragma unroll
								for (int s = 0; s < 4; s++)
									x[s] = W[256 * (J * NX + C) + 64 * s + lane];
#pragma unroll
							for (int s = 0; s < 4; s++)
								ah = mfma16(x[s], bh[C][s], ah);
							if (J < NW && J <= il)
#pragma unroll
								for (int s = 0; s < 4; s++)
									al = mfma16(x[s], bl[C][s], al);
						}
					hi[J] += ah;
					if (J < NW && J <= il)
						lo[J < NW ? J : 0] += al;
				}
		}
		// the next stage's descriptors and strips of BAbt, loaded beside the Cholesky
		const RicStage<PS> cur = st;
		if (k > 0)
		{
			st = ric_stage<PS>(raw, false);
			if (k > 1)
				raw = ric_fetch(a, N, k - 2);
			const int mn = st.nu + st.nx + XR;
			int Rn, jh, jl;
			strips(st.nu + st.nx, Rn, jh, jl);
			if (jh >= 0)
				load_b(st.C, jh, mn, cur.nx, bh);
			if (jl >= 0)
				load_b(st.C, jl, mn, cur.nx, bl);
			if constexpr (AHEAD)
				load_m(st, ph, pl);
		}
		if (AHEAD && k < N)
		{
			store_l(done);
			__syncthreads();   // its tiles are read: the Cholesky may write them
		}
		auto emit = [&](int I, int J, const double (&x)[4]) {
			if constexpr (!AHEAD)
			{
				int ge = g, ce = c;
				BFA_PIN(ge);
				BFA_PIN(ce);
				const int row = 16 * I + ce;
				strip_store(cur.L, cur.L.at(min(row, m - 1), ge), ge, 16 * J, nk, row < m, x);
			}
		};
		auto emit_diag = [&](int J, const double (&l)[4], const double (&iv)[4]) {
			int ge = g, ce = c;
			BFA_PIN(ge);
			BFA_PIN(ce);
			if constexpr (AHEAD)
			{
#pragma unroll
				for (int s = 0; s < 4; s++)
					if (ce == 0)
						lds[RC_INV + 16 * J + 4 * s + ge] = iv[s];
			}
			else
			{
				const int row = 16 * J + ce;
				strip_store_diag(cur.L, cur.L.at(min(row, m - 1), ge), ge, ce, 16 * J, nk, row < m, l,
					(BFA_GLOBAL double *)(uintptr_t)cur.dA, iv);
			}
		};
		chol_coop<double, NW>(hi, lo, ih, il, Cb, lay, emit, emit_diag);
		done = cur;
		if (threadIdx.x == 0)
		{
			// potrf_l marks the whole diagonal cached; syrk_dpotrf_ln and the
			// trapezoid forms (potrf_l_mn, syrk_dpotrf_ln_mn) one entry
			a.L[k].use_dA = (k == N && !AUG) ? nk : 1;
			if (k < N)
				a.work->use_dA = 0;
		}
		n1 = cur.nx;
		u1 = cur.nu;
	}
	if (AHEAD)
		store_l(done);
}

// An instance of up to 128 rows that does not fit a direct launch, its hint being too
// small: one wave, the stage matrix in L[k] itself, four columns of W at a time in LDS.
// What it takes does not matter, only that such an instance is factorised as the class
// launches factorise it.
template <int PS, bool AUG>
__device__ __forceinline__ void ric_beyond(const RicRec &a, int N, double *W)
{
	constexpr int XR = AUG ? 1 : 0, RW = 128;
	const int lane = lane_id();
	int n1 = 0, u1 = 0;   // sizes of stage k + 1
#pragma unroll 1
	for (int k = N; k >= 0; k--)
	{
		const int x = a.nx[k], u = k < N ? a.nu[k] : 0, nk = x + u, m = nk > 0 || AUG ? nk + XR : 0;
		const PM<double, PS> C = view<double, PS>(a.BAbt + (k < N ? k : 0)), R = view<double, PS>(a.RSQrq + k);
		const PM<double, PS> L = view<double, PS>(a.L + k), L1 = view<double, PS>(a.L + min(k + 1, N));
#pragma unroll 1
		for (int i = lane; i < m; i += WAVE)
#pragma unroll 1
			for (int j = 0; j <= min(i, nk - 1); j++)
				L.at(i, j) = R.at(i, j);
#pragma unroll 1
		for (int c = 0; k < N && c < n1; c += 4)
		{
			const int cw = min(4, n1 - c);
#pragma unroll 1
			for (int i = lane; i < m; i += WAVE)
#pragma unroll 1
				for (int q = 0; q < cw; q++)
				{
					double w = 0.0;
#pragma unroll 1
					for (int l = c + q; l < n1; l++)
						w += C.at(i, l) * L1.at(u1 + l, u1 + c + q);
					if (AUG && i == nk)
						w += L1.at(u1 + n1, u1 + c + q);
					W[q * RW + i] = w;
				}
			wave_sync();
#pragma unroll 1
			for (int i = lane; i < m; i += WAVE)
#pragma unroll 1
				for (int j = 0; j <= min(i, nk - 1); j++)
				{
					double w = 0.0;
#pragma unroll 1
					for (int q = 0; q < cw; q++)
						w += W[q * RW + i] * W[q * RW + j];
					L.at(i, j) += w;
				}
			wave_sync();
		}
#pragma unroll 1
		for (int j = 0; j < nk; j++)
		{
			double v[2] = {0.0, 0.0};   // rows lane and lane + 64 of column j
#pragma unroll
			for (int q = 0; q < 2; q++)
				if (lane + WAVE * q >= j && lane + WAVE * q < m)
				{
					double w = 0.0;
#pragma unroll 1
					for (int p = 0; p < j; p++)
						w += L.at(lane + WAVE * q, p) * L.at(j, p);
					v[q] = L.at(lane + WAVE * q, j) - w;
				}
			const double d = j < WAVE ? readlane(v[0], j) : readlane(v[1], j - WAVE);
			const double inv = d > 0.0 ? rsqrt_fast(d) : 0.0;
#pragma unroll
			for (int q = 0; q < 2; q++)
				if (lane + WAVE * q >= j && lane + WAVE * q < m)
					L.at(lane + WAVE * q, j) = v[q] * inv;
			if (lane == 0)
				a.L[k].dA[j] = inv;
			wave_sync();
		}
		if (lane == 0)
		{
			a.L[k].use_dA = (k == N && !AUG) ? nk : 1;
			if (k < N)
				a.work->use_dA = 0;
		}
		n1 = x;
		u1 = u;
	}
}

// Waves per SIMD that the kernels are compiled for.
constexpr int ric_coop_waves(int NW) { return NW == 1 ? 3 : 2; }

// DIRECT: one instance per workgroup (workgroup b takes instance b); else a persistent
// launch over a class list, the workgroups taking instances from the atomic queue
// head.  Rcap: the strips that the launch's LDS holds.  A direct launch has the plan's rule
// (ric_class) for instances larger than the hint (mmax rows): up to 64 states and 128
// rows, with AUG the augmented one among them, or up to mmax rows whatever their states
// (not with AUG) they are factorised all the same, others are left alone, as are
// negative sizes.
template <int PS, int NW, int NX, bool AUG, bool DIRECT>
__global__ __launch_bounds__(NW * WAVE, (ric_coop_waves(NW))) void k_ric_coop(const typename RicArg<AUG>::type *__restrict__ args,
	int Rcap, int mmax, const int *__restrict__ count, const int *__restrict__ list, int *head)
{
	extern __shared__ double smem_d[];
	__shared__ int qslot;
	constexpr int XR = AUG ? 1 : 0;
	const int cnt = DIRECT ? 0 : *count;
	for (;;)
	{
		int i = blockIdx.x;
		if (!DIRECT)
		{
			__syncthreads();   // every wave has left the previous instance
			if (threadIdx.x == 0)
				qslot = atomicAdd(head, 1);
			__syncthreads();
			const int t = __builtin_amdgcn_readfirstlane(qslot);
			if (t >= cnt)
				return;
			i = __builtin_amdgcn_readfirstlane(list[t]);
		}
		const RicRec a = ric_rec(args[i]);
		const int N = __builtin_amdgcn_readfirstlane(args[i].N);
		if (N >= 0)
		{
			int nk, nx, least;
			ric_sizes(a, N, nk, nx, least);
			if (least >= 0 && nx <= 16 * NX && (nk + XR + 15) / 16 <= Rcap)
			{
				if (threadIdx.x < 2)
					smem_d[threadIdx.x] = 0.0;   // read after the first barrier at the earliest
				ric_coop<PS, NW, NX, AUG>(a, N, nk, smem_d);
			}
			else if (DIRECT && least >= 0 && nk + XR <= 128 && (nx <= 64 || (!AUG && nk <= mmax)))
			{
				if (wave_id() == 0)
					ric_beyond<PS, AUG>(a, N, smem_d);
			}
		}
		if (DIRECT)
			return;
	}
}

} // namespace bfa
