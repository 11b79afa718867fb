// bfa_strip.hpp -- building blocks of the one-wavefront factorisations and
// solves: a strip of 16 rows of a matrix held in registers, with no LDS
// staging and no barriers.
//
// Strip layout.  Lane l of the wave is (g, c) = (l / 16, l % 16).  A 16 x 16
// block X (16 rows of the strip, 16 columns) is held as four values per lane,
//   x[s] at lane (g, c) = X[row(c)][4 s + g],
// row(c) = c for double and the 4 x 4 transposed index for float (strip_row).
// Read as a matrix-core operand, x[s] is step s of both operands of the
// 16x16x4 product (A: row = lane % 16, k = lane / 16; B the same of X^T), and
// because the accumulator of v_mfma_f64_16x16x4f64 holds row l/16 + 4 r of its
// column l%16 in register r, a product whose A operand is a block of rows of
// another matrix and whose B operand is the strip comes out in the strip
// layout again: the result of one product is the operand of the next
// without a transposition or a trip through LDS.  For float the accumulator
// holds row 4 (l/16) + r instead; feeding the rows in the order strip_row
// makes the two types agree.
//
// With that, X A^{-T} of a strip (the rows below a factored block, trsm_rltn)
// and the rows of a Cholesky factor are chains of products in registers:
// block column K of the strip is C_K minus the products of the finished blocks
// p < K with the row block L_K, then a triangular solve with L_KK.
#pragma once
#include "bfa_common.hpp"
#include "bfa_chol_core.hpp"

// Keeps the compiler from treating x as known (scheduling and hoisting barrier
// for what depends on it); nothing in the CPU emulator of the kernels.
#ifndef BFA_PIN
#define BFA_PIN(x) asm volatile("" : "+v"(x))
#endif

// Wants these wave-uniform values, each as "s"(x), in scalar registers here: their loads
// from the argument record are then issued together before this point, not waited for
// one by one after the next branches.
#ifndef BFA_NEED
#define BFA_NEED(...) asm volatile("" : : __VA_ARGS__)
#endif

namespace bfa {

// A panel-major matrix as the strip kernels address it: a wave-uniform base and byte
// offsets of type O.  O = size_t reaches every matrix.  With O = unsigned an access is
// one instruction with a scalar base, a 32-bit offset register and a constant
// for the column; a matrix may take 4 GiB and more, so the base is first moved to
// the block at hand (block()), and that the block's own offsets fit is asked of
// the panel stride (strip_fits).  Where registers are short, the kernel has both forms
// and takes the narrow one where it reaches (with size_t alone gemm in FP32 takes 1.12,
// trsm_rltn 1.12, getrf 1.09 times as long); the Cholesky and Riccati kernels are no
// slower with size_t.
template <typename T, int PS, typename O = size_t>
struct StripView
{
	typedef O ofs;
	static constexpr unsigned CS = PS * sizeof(T);   // bytes from one column to the next
	BFA_GLOBAL char *p;
	unsigned cn;
	// byte offset of element (i, j)
	__device__ __forceinline__ O at(int i, int j) const
	{
		return ((O)((unsigned)i / PS) * cn + (unsigned)j) * CS + ((unsigned)i & (PS - 1)) * (unsigned)sizeof(T);
	}
	// the value at a wave-uniform offset u plus this lane's offset o
	__device__ __forceinline__ T ld(O u, O o) const { return *(const BFA_GLOBAL T *)((p + u) + o); }
	__device__ __forceinline__ void st(O u, O o, T v) const { *(BFA_GLOBAL T *)((p + u) + o) = v; }
	// The matrix from the panel of row i and column j on (wave-uniform): i becomes the row
	// within that panel, j 0.
	template <typename O2>
	__device__ __forceinline__ StripView<T, PS, O2> block(int &i, int &j) const
	{
		StripView<T, PS, O2> r;
		r.p = p + ((size_t)((unsigned)i / PS) * cn + (unsigned)j) * CS;
		r.cn = cn;
		i &= PS - 1;
		j = 0;
		return r;
	}
};

// Steps 0 .. NS-1 of a strip's 16-column block that starts at column c (wave-
// uniform) of n <= 256: og is this lane's row at column g.  Columns past n read
// column n - 1.
template <int NS, typename T, int PS, typename O, typename X>
__device__ __forceinline__ void strip_load(const StripView<T, PS, O> &v, O og, int g, int c, int n, X &x)
{
	constexpr unsigned CS = PS * sizeof(T);
	if (c + 16 <= n)
	{
#pragma unroll
		for (int s = 0; s < NS; s++)
			x[s] = v.ld((unsigned)c * CS + 4 * s * CS, og);
	}
	else
	{
#pragma unroll
		for (int s = 0; s < NS; s++)
			x[s] = v.ld(0, og + (O)(ptrdiff_t)((min(c + 4 * s + g, n - 1) - g) * (int)CS));
	}
}
// The same where the block is known to be inside.
template <int NS, typename T, int PS, typename O, typename X>
__device__ __forceinline__ void strip_load_full(const StripView<T, PS, O> &v, O og, int c, X &x)
{
	constexpr unsigned CS = PS * sizeof(T);
#pragma unroll
	for (int s = 0; s < NS; s++)
		x[s] = v.ld((unsigned)c * CS + 4 * s * CS, og);
}
// Block x (columns c .. c+15 of n) to a strip's rows; ok: this lane's row is
// one of the matrix's.
template <typename T, int PS, typename O, typename X>
__device__ __forceinline__ void strip_store(const StripView<T, PS, O> &v, O og, int g, int c, int n, bool ok, const X &x)
{
	constexpr unsigned CS = PS * sizeof(T);
	if (c + 16 <= n)
	{
		if (ok)
#pragma unroll
			for (int s = 0; s < 4; s++)
				v.st((unsigned)c * CS + 4 * s * CS, og, x[s]);
	}
	else
	{
#pragma unroll
		for (int s = 0; s < 4; s++)
			if (ok && c + 4 * s + g < n)
				v.st((unsigned)c * CS + 4 * s * CS, og, x[s]);
	}
}
// The lower triangle of a factored diagonal block (columns c .. c+15 of n) to D
// and its reciprocal pivots to dD.
template <typename T, int PS, typename O>
__device__ __forceinline__ void strip_store_diag(const StripView<T, PS, O> &v, O og, int g, int rid, int c, int n, bool ok,
	const T (&l)[4], BFA_GLOBAL T *dD, const T (&iv)[4])
{
	constexpr unsigned CS = PS * sizeof(T);
#pragma unroll
	for (int s = 0; s < 4; s++)
	{
		const int cl = 4 * s + g;
		if (ok && c + cl < n && cl <= rid)
			v.st((unsigned)c * CS + 4 * s * CS, og, l[s]);
		if (rid == 0 && c + cl < n)
			dD[c + cl] = iv[s];
	}
}
__device__ __forceinline__ unsigned long long uniform_u64(unsigned long long v)
{
	const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
	const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
	return ((unsigned long long)hi << 32) | lo;
}
template <typename T, int PS>
__device__ __forceinline__ StripView<T, PS> strip_view(const typename MatOf<T>::type *s)
{
	const PM<T, PS> v = view<T, PS>(s);
	StripView<T, PS> r;
	r.p = (BFA_GLOBAL char *)(uintptr_t)uniform_u64((unsigned long long)(uintptr_t)v.p);
	r.cn = (unsigned)__builtin_amdgcn_readfirstlane(v.cn);
	return r;
}

// Do the byte offsets of a block of up to 256 rows (and a panel's remainder at either
// end) fit 32 bits, the largest panel stride being cn?
template <typename T, int PS>
__device__ __forceinline__ bool strip_fits(unsigned cn)
{
	return cn <= 0xffffffffu / ((256 + 2 * PS) * (unsigned)sizeof(T));
}

// Row (0..15) of the 16-row strip that lane position c holds, and, the map
// being its own inverse, the lane position that holds row c.
template <typename T>
__host__ __device__ constexpr int strip_row(int c)
{
	return sizeof(T) == 8 ? c : ((c & 3) << 2) | (c >> 2);
}

// The value of lane position P of the lane's own 16-lane row.
template <int P>
__device__ __forceinline__ double row_bcast(double v)
{
	return __builtin_amdgcn_update_dpp(v, v, 0x150 + P, 0xf, 0xf, true);
}
template <int P>
__device__ __forceinline__ float row_bcast(float v)
{
	return dpp_t<0x150 + P, 0xf>(v, v);
}

// The values of the four 16-lane rows at the lane's own position c, in every
// row: y[q] = v of lane (q, c).
__device__ __forceinline__ void gather4_u(unsigned v, unsigned (&y)[4])
{
	const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);          // {0,0,2,2}, {1,1,3,3}
	const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);    // {0,0,0,0}, {2,2,2,2}
	const auto o = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
	y[0] = e[0];
	y[1] = o[0];
	y[2] = e[1];
	y[3] = o[1];
}
__device__ __forceinline__ void gather4(double v, double (&y)[4])
{
	const int2 x = __builtin_bit_cast(int2, v);
	unsigned lo[4], hi[4];
	gather4_u((unsigned)x.x, lo);
	gather4_u((unsigned)x.y, hi);
#pragma unroll
	for (int q = 0; q < 4; q++)
	{
		int2 r;
		r.x = (int)lo[q];
		r.y = (int)hi[q];
		y[q] = __builtin_bit_cast(double, r);
	}
}
__device__ __forceinline__ void gather4(float v, float (&y)[4])
{
	unsigned u[4];
	gather4_u(__builtin_bit_cast(unsigned, v), u);
#pragma unroll
	for (int q = 0; q < 4; q++)
		y[q] = __builtin_bit_cast(float, u[q]);
}

// Block K (wave-uniform) of an array of blocks held in registers, read or
// written by a branch per block: register arrays cannot be indexed, and a
// select per block and register would cost more than the block's products.
template <typename V4, int NB>
__device__ __forceinline__ V4 strip_get(const V4 (&nx)[NB], int K)
{
	V4 x = nx[0];
#pragma unroll
	for (int i = 1; i < NB; i++)
		if (i == K)
		{
			x = nx[i];
			BFA_PIN(x);
		}
	return x;
}
template <typename V4, int NB>
__device__ __forceinline__ void strip_set(V4 (&nx)[NB], int K, V4 x)
{
#pragma unroll
	for (int i = 0; i < NB; i++)
		if (i == K)
		{
			nx[i] = x;
			BFA_PIN(nx[i]);
		}
}

// v[g] of the lane's row g
template <typename T>
__device__ __forceinline__ T select4(int g, T v0, T v1, T v2, T v3)
{
	const T a = (g & 1) ? v1 : v0, b = (g & 1) ? v3 : v2;
	return (g & 2) ? b : a;
}

// Cholesky of one 16 x 16 diagonal block, one wave.  acc: the block's lower
// triangle in the strip layout (element (i, j), i >= j, at the lane and
// register of X[i][j]; the others may hold anything, they reach no element
// of the lower triangle).  l: the factor, lower triangle valid, in the strip
// layout; iv[s] at lane (g, c): the reciprocal of pivot 4 s + g with the
// zero-pivot rule of chol_acc (pivot <= 0 or NaN: reciprocal 0).
// Four columns at a time: the four rows of acc that hold them are brought to
// every lane (each then has its own row's four entries), factored with row
// broadcasts, and the columns to the right take one rank-4 matrix-core
// step.  Against a row per lane with v_readlane broadcasts for all 120 updates
// this leaves 24 of them to the vector unit and keeps the scalar registers out.
template <typename T>
__device__ __forceinline__ void strip_chol16(typename Vec4<T>::type acc, T (&l)[4], T (&iv)[4])
{
	const int g = lane_id() >> 4;
#pragma unroll
	for (int s = 0; s < 4; s++)
	{
		T y[4], r[4], inv[4];
		gather4(acc[s], y);
		auto pivot = [&](T c, int q) {
			inv[q] = (c > T(0)) ? rsqrt_fast(c) : T(0);
			r[q] = y[q] * inv[q];
		};
		// the value of the lane that holds row 4 s + q
		auto bc = [&](T v, auto qc) -> T {
			constexpr int q = decltype(qc)::value;
			if (s == 0)
				return row_bcast<strip_row<T>(q)>(v);
			if (s == 1)
				return row_bcast<strip_row<T>(4 + q)>(v);
			if (s == 2)
				return row_bcast<strip_row<T>(8 + q)>(v);
			return row_bcast<strip_row<T>(12 + q)>(v);
		};
		struct Q0 { enum { value = 0 }; };
		struct Q1 { enum { value = 1 }; };
		struct Q2 { enum { value = 2 }; };
		struct Q3 { enum { value = 3 }; };
		pivot(bc(y[0], Q0{}), 0);
		y[1] -= r[0] * bc(r[0], Q1{});
		pivot(bc(y[1], Q1{}), 1);
		y[2] -= r[0] * bc(r[0], Q2{});
		y[3] -= r[0] * bc(r[0], Q3{});
		y[2] -= r[1] * bc(r[1], Q2{});
		pivot(bc(y[2], Q2{}), 2);
		y[3] -= r[1] * bc(r[1], Q3{});
		y[3] -= r[2] * bc(r[2], Q3{});
		pivot(bc(y[3], Q3{}), 3);
		l[s] = select4(g, r[0], r[1], r[2], r[3]);
		iv[s] = select4(g, inv[0], inv[1], inv[2], inv[3]);
		if (s < 3)
			acc = mfma16(-l[s], l[s], acc);
	}
}

// The 4 x 4 triangles on the diagonal of a 16 x 16 lower block as strip_solve
// takes them: d[s] at lane position c (the same in all four rows) = entry
// (4 s + c/4, 4 s + c%4) below the diagonal and the reciprocal pivot on it.
// Given the block and its reciprocals as strip_chol16 returns them, this
// lane's entry is written to tri[16 s + c'] (64 values per block).
template <typename T>
__device__ __forceinline__ void strip_put_tri(T *tri, const T (&l)[4], const T (&iv)[4])
{
	const int g = lane_id() >> 4, i = strip_row<T>(lane_id() & 15);
#pragma unroll
	for (int s = 0; s < 4; s++)
		if ((i >> 2) == s)
			tri[16 * s + 4 * (i & 3) + g] = (i & 3) == g ? iv[s] : l[s];
}

// X L^{-T} for one block of the strip: acc holds the block C minus the
// products of the finished blocks, l the diagonal block (its steps 0..2, lower
// triangle) and d its 4 x 4 triangles; x: the solved block.
// Four columns at a time: their values are brought to all four rows of lanes
// (each lane then has its row's four entries), solved by substitution with
// the reciprocal pivots in the reference's order, and applied to the columns
// to the right by one matrix-core step each.  The coefficients above the
// diagonal reach finished columns only, so an Inf or NaN of one column does not
// spread to earlier ones.
template <typename T>
__device__ __forceinline__ void strip_solve(typename Vec4<T>::type acc, const T (&l)[3], const T (&d)[4], T (&x)[4])
{
	const int g = lane_id() >> 4;
#pragma unroll
	for (int s = 0; s < 4; s++)
	{
		T y[4];
		gather4(acc[s], y);
		y[0] *= row_bcast<0>(d[s]);
		y[1] -= y[0] * row_bcast<4>(d[s]);
		y[1] *= row_bcast<5>(d[s]);
		y[2] -= y[0] * row_bcast<8>(d[s]);
		y[2] -= y[1] * row_bcast<9>(d[s]);
		y[2] *= row_bcast<10>(d[s]);
		y[3] -= y[0] * row_bcast<12>(d[s]);
		y[3] -= y[1] * row_bcast<13>(d[s]);
		y[3] -= y[2] * row_bcast<14>(d[s]);
		y[3] *= row_bcast<15>(d[s]);
		x[s] = select4(g, y[0], y[1], y[2], y[3]);
		if (s < 3)
			acc = mfma16(-l[s], x[s], acc);
	}
}

// Two strips solved with the same block: the first strip's rows in the lanes of
// the lower half, the second's in the upper half, so that the substitution is
// done once for both (36 vector instructions per four columns against 2 x 46).
__device__ __forceinline__ void pair_u(unsigned &a, unsigned &b)
{
	const auto p = __builtin_amdgcn_permlane32_swap(a, b, false, false);   // {a0,a1,b0,b1}, {a2,a3,b2,b3}
	a = p[0];
	b = p[1];
}
__device__ __forceinline__ void pair_swap(double &a, double &b)
{
	int2 x = __builtin_bit_cast(int2, a), y = __builtin_bit_cast(int2, b);
	unsigned xl = (unsigned)x.x, xh = (unsigned)x.y, yl = (unsigned)y.x, yh = (unsigned)y.y;
	pair_u(xl, yl);
	pair_u(xh, yh);
	x.x = (int)xl, x.y = (int)xh, y.x = (int)yl, y.y = (int)yh;
	a = __builtin_bit_cast(double, x);
	b = __builtin_bit_cast(double, y);
}
__device__ __forceinline__ void pair_swap(float &a, float &b)
{
	unsigned x = __builtin_bit_cast(unsigned, a), y = __builtin_bit_cast(unsigned, b);
	pair_u(x, y);
	a = __builtin_bit_cast(float, x);
	b = __builtin_bit_cast(float, y);
}
// {r0,r0,r2,r2} and {r1,r1,r3,r3} of the 16-lane rows of v
__device__ __forceinline__ void twin_u(unsigned v, unsigned &e, unsigned &o)
{
	const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
	e = p[0];
	o = p[1];
}
__device__ __forceinline__ void twin(double v, double &e, double &o)
{
	const int2 x = __builtin_bit_cast(int2, v);
	unsigned el, eh, ol, oh;
	twin_u((unsigned)x.x, el, ol);
	twin_u((unsigned)x.y, eh, oh);
	int2 r;
	r.x = (int)el, r.y = (int)eh;
	e = __builtin_bit_cast(double, r);
	r.x = (int)ol, r.y = (int)oh;
	o = __builtin_bit_cast(double, r);
}
__device__ __forceinline__ void twin(float v, float &e, float &o)
{
	unsigned ue, uo;
	twin_u(__builtin_bit_cast(unsigned, v), ue, uo);
	e = __builtin_bit_cast(float, ue);
	o = __builtin_bit_cast(float, uo);
}
template <typename T>
__device__ __forceinline__ void strip_solve2(typename Vec4<T>::type acc0, typename Vec4<T>::type acc1, const T (&l)[3],
	const T (&d)[4], T (&x0)[4], T (&x1)[4])
{
	const bool odd = (lane_id() >> 4) & 1;
#pragma unroll
	for (int s = 0; s < 4; s++)
	{
		T a = acc0[s], b = acc1[s], y[4];
		pair_swap(a, b);
		twin(a, y[0], y[1]);
		twin(b, y[2], y[3]);
		y[0] *= row_bcast<0>(d[s]);
		y[1] -= y[0] * row_bcast<4>(d[s]);
		y[1] *= row_bcast<5>(d[s]);
		y[2] -= y[0] * row_bcast<8>(d[s]);
		y[2] -= y[1] * row_bcast<9>(d[s]);
		y[2] *= row_bcast<10>(d[s]);
		y[3] -= y[0] * row_bcast<12>(d[s]);
		y[3] -= y[1] * row_bcast<13>(d[s]);
		y[3] -= y[2] * row_bcast<14>(d[s]);
		y[3] *= row_bcast<15>(d[s]);
		a = odd ? y[1] : y[0];
		b = odd ? y[3] : y[2];
		pair_swap(a, b);
		x0[s] = a;
		x1[s] = b;
		if (s < 3)
		{
			acc0 = mfma16(-l[s], a, acc0);
			acc1 = mfma16(-l[s], b, acc1);
		}
	}
}

// ---------------------------------------------------------------------------
// Cholesky of an m x n lower trapezoid (m >= n) by NW waves, its 16 x 16 tiles
// in registers.
// Strip I (rows 16 I ..) belongs to one wave; the strips are dealt from the last
// one down and back, two a wave: wave w has ih = R - 1 - w and il = R - 2 NW + w
// (none where negative), so every wave has about the same number of tiles.
// hi[J], lo[J]: the tiles (ih, J), (il, J), J <= min(I, Cb - 1), in the strip layout.
// Right-looking, one barrier per block column j: every wave solves its strips'
// tiles (I, j) with L_jj, passes them to LDS as operand tiles and, for the strip
// j + 1, applies its own tile to the diagonal one and factors it; after the
// barrier every wave applies column j to its tiles on the right.  The tiles never
// leave the registers, L goes to memory once (emit(I, j, x), emit_diag(j, l, iv))
// and no finished part of it is read again: with one wave per instance the
// finished strips are read back for every later one, which above 64 rows
// misses L2 and bounds the launch (8192 x 128 rows: 1.9 GB read for 0.55 GB of
// input).
// LAY says where in LDS the tiles are passed on: tile(I, j) the base of tile (I, j)
// of the current column, at(s) this lane's offset in it for step s, diag(j) and
// tri(j) the diagonal block and its 4 x 4 triangles.
// ---------------------------------------------------------------------------
// Two columns of operand tiles and two diagonal blocks, used in turn.
template <typename T, int NW>
struct CoopRing
{
	static constexpr int ELEMS = 2 * (2 * NW * 256 + 256);
	static constexpr int DSTEPS = 3;   // steps of a diagonal block that are passed on
	T *p;
	int lane;
	__device__ __forceinline__ T *tile(int I, int j) const { return p + (j & 1) * (2 * NW * 256) + 256 * I; }
	__device__ __forceinline__ int at(int s) const { return 64 * s + lane; }
	__device__ __forceinline__ T *diag(int j) const { return p + 2 * 2 * NW * 256 + (j & 1) * 256; }
	__device__ __forceinline__ T *tri(int j) const { return diag(j) + 192; }
};

template <typename T, int NW, typename LAY, typename EMIT, typename EMITD>
__device__ __forceinline__ void chol_coop(typename Vec4<T>::type (&hi)[2 * NW], typename Vec4<T>::type (&lo)[NW],
	int ih, int il, int Cb, const LAY &lay, const EMIT &emit, const EMITD &emit_diag)
{
	typedef typename Vec4<T>::type V4;
	const int lane = lane_id();
	// factors the diagonal tile of block column j and passes it on
	auto factor = [&](V4 acc, int j) {
		T l[4], iv[4];
		strip_chol16<T>(acc, l, iv);
		T *db = lay.diag(j);
#pragma unroll
		for (int s = 0; s < LAY::DSTEPS; s++)
			db[lay.at(s)] = l[s];
		strip_put_tri<T>(lay.tri(j), l, iv);
		emit_diag(j, l, iv);
	};
	if (Cb > 0 && ih == 0)
		factor(hi[0], 0);
	else if (Cb > 0 && il == 0)
		factor(lo[0], 0);
	__syncthreads();
#pragma unroll 1
	for (int j = 0; j < Cb; j++)
	{
		const T *db = lay.diag(j), *tb = lay.tri(j);
		V4 yh = V4{0, 0, 0, 0}, yl = V4{0, 0, 0, 0};   // -X of this column
		{
			T lk[3], d[4];
#pragma unroll
			for (int s = 0; s < 3; s++)
				lk[s] = db[lay.at(s)];
#pragma unroll
			for (int s = 0; s < 4; s++)
				d[s] = tb[16 * s + (lane & 15)];
			auto done = [&](const T (&x)[4], int I, V4 &y) {
				emit(I, j, x);
				T *t = lay.tile(I, j);
#pragma unroll
				for (int s = 0; s < 4; s++)
				{
					t[lay.at(s)] = x[s];
					y[s] = -x[s];
				}
			};
			auto next = [&](V4 acc, const V4 &y) {
#pragma unroll
				for (int s = 0; s < 4; s++)
					acc = mfma16(-y[s], y[s], acc);
				factor(acc, j + 1);
			};
			T xh[4], xl[4];
			if (il > j)
			{
				strip_solve2<T>(strip_get(hi, j), strip_get(lo, j), lk, d, xh, xl);
				done(xl, il, yl);
				done(xh, ih, yh);
			}
			else if (ih > j)
			{
				strip_solve<T>(strip_get(hi, j), lk, d, xh);
				done(xh, ih, yh);
			}
			if (j + 1 < Cb)
			{
				if (ih == j + 1)
					next(strip_get(hi, j + 1), yh);
				else if (il == j + 1)
					next(strip_get(lo, j + 1), yl);
			}
		}
		__syncthreads();
		// the tiles right of column j
#pragma unroll
		for (int J = 1; J < 2 * NW; J++)
			if (J > j && J < Cb && J <= ih)
			{
				T a[4];
#pragma unroll
				for (int s = 0; s < 4; s++)
					a[s] = lay.tile(J, j)[lay.at(s)];
#pragma unroll
				for (int s = 0; s < 4; s++)
					hi[J] = mfma16(a[s], yh[s], hi[J]);
				if (J < NW && J <= il)
#pragma unroll
					for (int s = 0; s < 4; s++)
						lo[J < NW ? J : 0] = mfma16(a[s], yl[s], lo[J < NW ? J : 0]);
			}
	}
}

} // namespace bfa
