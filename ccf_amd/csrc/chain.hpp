// FP64 Cauchy sums with shared reciprocals, and the phi chain of a row solved
// by one workgroup (weisluke/ccf include/ccf_functions.cuh:193-243 and
// ccf.cuh:979-1083): used by the single-field sweeps and small fields
// (solve.hip) and by the batched form (batch.hip).
#pragma once

#include "lens.hpp"

namespace ccf
{

// 1/x for x > 0: hardware reciprocal estimate refined by two Newton steps
// (each squares the relative error of the ~2^-23 estimate)
__device__ inline double rcp64(double x)
{
	double r = __builtin_amdgcn_rcp(x);
	double e = fma(-x, r, 1.0);
	r = fma(r, e, r);
	e = fma(-x, r, 1.0);
	return fma(r, e, r);
}

// Four Cauchy terms d_i / |d_i|^2, d_i = z - w_i, added to (ax, ay) over one
// reciprocal: with n_i = |d_i|^2 and the pair numerators d_0 n_1 + d_1 n_0
// and d_2 n_3 + d_3 n_2, their sum is
//   ((d_0 n_1 + d_1 n_0) n_2 n_3 + (d_2 n_3 + d_3 n_2) n_0 n_1) / (n_0 n_1 n_2 n_3).
// 36 FP64 instructions and one v_rcp_f64 (3.4 instructions' time) for four
// terms, against 11 (one of them v_max_f64, 1.7) and one for each term of
// its own. No numerator cancels more than the sum of the terms itself does,
// and the accumulator rounds once in four terms. NORM_FLOOR makes the term
// of the root itself (d = 0) zero; it does not reach the last bit of any
// n_i of two positions further apart than 1e-22. Products stay within range
// while every |d_i| is below 1e38; beyond it the sums are not finite and the
// slice is summed again term by term.
// Relative error of sums of 200 to 20 000 terms against 80-bit ones: 2e-16
// to 5e-16 rms, 4e-16 to 1.3e-15 term by term.
constexpr double NORM_FLOOR = 1e-60;

// 1/x from the hardware estimate r (relative error about 2^-23) as
// r (1 + e + e^2), e = 1 - x r: one third-order step, whose error e^3 is far
// below the rounding of the last multiply-add
__device__ __forceinline__ double rcp64_cubic(double x)
{
	const double r = __builtin_amdgcn_rcp(x);
	const double e = fma(-x, r, 1.0);
	return fma(r, fma(e, e, e), r);
}

// four terms as one fraction (X, Y) / P
__device__ __forceinline__ void cauchy_quad(double zx, double zy, const double2* w, double& X, double& Y, double& P)
{
	double dx[4], dy[4], n[4];
#pragma unroll
	for (int i = 0; i < 4; i++)
	{
		dx[i] = zx - w[i].x;
		dy[i] = zy - w[i].y;
		n[i] = fma(dx[i], dx[i], fma(dy[i], dy[i], NORM_FLOOR));
	}
	const double p = n[0] * n[1], q = n[2] * n[3];
	const double x01 = fma(dx[0], n[1], dx[1] * n[0]), y01 = fma(dy[0], n[1], dy[1] * n[0]);
	const double x23 = fma(dx[2], n[3], dx[3] * n[2]), y23 = fma(dy[2], n[3], dy[3] * n[2]);
	X = fma(x01, q, x23 * p);
	Y = fma(y01, q, y23 * p);
	P = p * q;
}

// the four terms times SIGN (1 or -1) added to (ax, ay)
template <int SIGN>
__device__ __forceinline__ void cauchy4(double zx, double zy, const double2 (&w)[4], double& ax, double& ay)
{
	double X, Y, P;
	cauchy_quad(zx, zy, w, X, Y, P);
	const double iv = SIGN * rcp64_cubic(P);
	ax = fma(X, iv, ax);
	ay = fma(Y, iv, ay);
}

// Eight terms over one reciprocal, two such fractions over their common
// denominator: one reciprocal, its refinement and a rounding of the
// accumulator less than in two groups of four (75 instructions' time against
// 79), and three quarters of their error. The range is |d| below 1e19; a
// product that underflows (six positions that coincide) ends as not finite
// too, and the slice is then summed again term by term. The dense sums of a
// 10 000-star run, num_phi 100: continuation 46.4 -> 44.8 ms.
template <int SIGN>
__device__ __forceinline__ void cauchy8(double zx, double zy, const double2 (&w)[8], double& ax, double& ay)
{
	double X0, Y0, P0, X1, Y1, P1;
	cauchy_quad(zx, zy, w, X0, Y0, P0);
	cauchy_quad(zx, zy, w + 4, X1, Y1, P1);
	const double iv = SIGN * rcp64_cubic(P0 * P1);
	ax = fma(fma(X0, P1, X1 * P0), iv, ax);
	ay = fma(fma(Y0, P1, Y1 * P0), iv, ay);
}

// one Cauchy term times SIGN; d = 0 gives zero
template <int SIGN>
__device__ __forceinline__ void cauchy1(double zx, double zy, double2 w, double& ax, double& ay)
{
	const double dx = zx - w.x, dy = zy - w.y;
	const double iv = SIGN * rcp64(fmax(fma(dx, dx, dy * dy), 1e-300));
	ax = fma(dx, iv, ax);
	ay = fma(dy, iv, ay);
}

// the terms of src[lo, hi) for a lane's target: every lane of the wave reads
// the same source, so the sources come through scalar loads
template <int SIGN>
__device__ __forceinline__ void cauchy_run(const double2* __restrict__ src, int lo, int hi, double zx, double zy, double& ax,
	double& ay)
{
	int q = lo;
#pragma unroll 2
	for (; q + 8 <= hi; q += 8)
	{
		const double2 w[8] = {src[q], src[q + 1], src[q + 2], src[q + 3], src[q + 4], src[q + 5], src[q + 6], src[q + 7]};
		cauchy8<SIGN>(zx, zy, w, ax, ay);
	}
	if (q + 4 <= hi)
	{
		const double2 w[4] = {src[q], src[q + 1], src[q + 2], src[q + 3]};
		cauchy4<SIGN>(zx, zy, w, ax, ay);
		q += 4;
	}
	for (; q < hi; q++) cauchy1<SIGN>(zx, zy, src[q], ax, ay);
}

// the same terms of one target, the wave's lanes over the sources (four of
// its own at a time): the lane's part of the sum
template <int SIGN>
__device__ __forceinline__ void cauchy_lanes(const double2* __restrict__ src, int lo, int hi, double zx, double zy, double& ax,
	double& ay)
{
	const int lane = threadIdx.x & 63;
	int q0 = lo;
#pragma unroll 1
	for (; q0 + 256 <= hi; q0 += 256)
	{
		const double2 w[4] = {src[q0 + lane], src[q0 + 64 + lane], src[q0 + 128 + lane], src[q0 + 192 + lane]};
		cauchy4<SIGN>(zx, zy, w, ax, ay);
	}
#pragma unroll 1
	for (int q = q0 + lane; q < hi; q += 64) cauchy1<SIGN>(zx, zy, src[q], ax, ay);
}

// The near-field sums of a root outside the tree (its node is not a leaf:
// every star of the node's ranges), by the lanes of one wave: lane l sums
// the stars l, l + 64, ... of the ranges (p2p's terms), and a butterfly of
// fixed order gives every lane the total. Every lane of the wave calls it
// with the same z and node.
__device__ inline Near wave_near(const LensView& L, int node, cd z)
{
	Near nr;
	const int lane = threadIdx.x & 63;
	const int ranges = L.nnf[node];
	for (int k = 0; k < ranges; k++)
	{
		const int2 rg = L.nf[node * MAX_NEAR_RANGES + k];
		const int e = rg.x + rg.y;
		// the lane's stars in order, two loads issued before their terms
		for (int s0 = rg.x + lane; s0 < e; s0 += 2 * 64)
		{
			double2 q[2];
			double m[2];
#pragma unroll
			for (int u = 0; u < 2; u++)
			{
				const int s = min(s0 + u * 64, e - 1);
				q[u] = L.spos[s];
				m[u] = L.smass[s];
			}
#pragma unroll
			for (int u = 0; u < 2; u++)
				if (s0 + u * 64 < e)
				{
					const cd t = cd(z.re - q[u].x, z.im - q[u].y).inv();
					nr.s0 += t;
					const cd t1 = t * m[u];
					nr.s1 += t1;
					const cd t2 = t1 * t;
					nr.s2 += t2;
					nr.s3 += t2 * t;
				}
		}
		nr.count += rg.y;
	}
	double v[8] = {nr.s0.re, nr.s0.im, nr.s1.re, nr.s1.im, nr.s2.re, nr.s2.im, nr.s3.re, nr.s3.im};
#pragma unroll
	for (int q = 0; q < 8; q++)
		for (int o = 32; o >= 1; o >>= 1) v[q] += __shfl_xor(v[q], o, 64);
	nr.s0 = cd(v[0], v[1]);
	nr.s1 = cd(v[2], v[3]);
	nr.s2 = cd(v[4], v[5]);
	nr.s3 = cd(v[6], v[7]);
	return nr;
}

// ---------------------------------------------------------------------------
// A row's sweeps in one workgroup, FP64, continuation steps. The roots start
// next to the roots of Witt's equation, where a rounding of the sums does
// not change which root an index takes, so the sums are free to be split
// over lanes by what a sweep lists.

// lanes that share the evaluation of a root when n are active: from the row,
// not from the workgroup, so that results do not depend on its size
__device__ __forceinline__ int chain_eval_lanes(int n)
{
	return n <= 128 ? 8 : (n <= 256 ? 4 : (n <= 512 ? 2 : 1));
}

// lanes that share the sums of a listed root when nf are listed and T terms
// are summed: the cheapest of 1 .. 64 for CHAIN_LANES lanes that each take a
// group of four terms in about 160 cycles and a reduction step in about 60
constexpr int CHAIN_LANES = 1024;

__device__ __forceinline__ int chain_sum_lanes(int nf, int T)
{
	int best = 1, bc = 0x7fffffff;
	for (int l = 0; l <= 6; l++)
	{
		const int rounds = ((nf << l) + CHAIN_LANES - 1) / CHAIN_LANES, quads = ((T + (1 << l) - 1) / (1 << l) + 3) / 4;
		const int c = rounds * (160 * quads + 60 * l);
		if (c < bc)
		{
			bc = c;
			best = 1 << l;
		}
	}
	return best;
}

// near-field sums of a leaf's run of stars by W lanes, lane sub the stars
// sub, sub + W, ...: the second and third only (f0 and f1 take no others)
__device__ __forceinline__ Near chain_near(const LensView& L, int node, cd z, int sub, int W)
{
	Near r;
	const int n = L.nf_cnt[node];
	const double4* __restrict__ p = L.nfs + L.nf_off[node];
	for (int t = sub; t < n; t += 4 * W)
	{
		double4 s[4];
#pragma unroll
		for (int k = 0; k < 4; k++) s[k] = p[min(t + k * W, n - 1)];
#pragma unroll
		for (int k = 0; k < 4; k++)
			if (t + k * W < n)
			{
				const cd u = cd(z.re - s[k].x, z.im - s[k].y).inv();
				const cd u2 = (u * s[k].z) * u;
				r.s2 += u2;
				r.s3 += u2 * u;
			}
	}
	for (int o = 1; o < W; o <<= 1)
	{
		r.s2 += cd(__shfl_xor(r.s2.re, o, 64), __shfl_xor(r.s2.im, o, 64));
		r.s3 += cd(__shfl_xor(r.s3.re, o, 64), __shfl_xor(r.s3.im, o, 64));
	}
	r.count = n;
	return r;
}

// SIGN times the terms of src[0, m) for a target, by W lanes, lane sub the
// terms sub, sub + W, ...: whole groups of 4 W terms, then one group that
// takes the target itself, whose term is zero, past the end. The few lanes a
// root of a sweep that lists many shares (WC = W = 1, 2, 4) are compiled in,
// so that the loads' offsets are immediate: the address arithmetic of a
// variable stride costs a fifth of the loop.
template <int SIGN, int WC>
__device__ __forceinline__ void chain_terms_w(const double2* src, int m, double2 z, int sub, int Wr, double& ax, double& ay)
{
	const int W = WC > 0 ? WC : Wr, rounds = m / (4 * W);
	const double2* p = src + sub;
#pragma unroll 1
	for (int k = 0; k < rounds; k++)
	{
		const double2 w[4] = {p[0], p[W], p[2 * W], p[3 * W]};
		p += 4 * W;
		cauchy4<SIGN>(z.x, z.y, w, ax, ay);
	}
	const int q = rounds * 4 * W + sub;
	if (rounds * 4 * W < m)
	{
		double2 w[4];
#pragma unroll
		for (int k = 0; k < 4; k++) w[k] = q + k * W < m ? src[q + k * W] : z;
		cauchy4<SIGN>(z.x, z.y, w, ax, ay);
	}
}

template <int SIGN>
__device__ __forceinline__ void chain_terms(const double2* src, int m, double2 z, int sub, int W, double& ax, double& ay)
{
	if (W == 1) chain_terms_w<SIGN, 1>(src, m, z, sub, W, ax, ay);
	else if (W == 2) chain_terms_w<SIGN, 2>(src, m, z, sub, W, ax, ay);
	else if (W == 4) chain_terms_w<SIGN, 4>(src, m, z, sub, W, ax, ay);
	else chain_terms_w<SIGN, 0>(src, m, z, sub, W, ax, ay);
}

// what a workgroup counts of its rows: full updates, early exits, converged,
// near-field stars (of updates that formed f1), sweeps
constexpr int CHAIN_COUNTS = 5;

// A batch's rows of at most this many roots run their phi chain as one
// workgroup, whose time grows with the square of its roots (400 roots: 112
// us a step; 600: 184); a step over the device takes 70 us and more.
constexpr int CHAIN_ROOTS = 480;

struct ChainLists
{
	int* la;     // ping-pong active lists
	int* lb;
	int* fl;     // listed roots
	double2* f0; // Witt function of a listed root
	double2* f1; // its derivative; then the moved root
};

// A sweep's three phases, between barriers, as in the batched form's
// solve_row (batch.hip): zc holds the row's roots, st the stars.

// Witt function and 1/mu exit of the n roots listed in cur, chain_eval_lanes
// lanes a root (a root outside the tree, whose near field is every star, by
// its whole wave); the roots that take the Cauchy sums are appended to ls.fl
// (*nf their count, zero before)
template <int BS>
__device__ __forceinline__ void chain_evaluate(const LensView& L, double cp, double sp, const double2* zc, const int* cur, int n,
	const ChainLists& ls, int* nf, int (&cnt)[CHAIN_COUNTS])
{
	const int lane = threadIdx.x & 63;
	const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
	const int W = chain_eval_lanes(n), sub = threadIdx.x & (W - 1), step = BS / W;
	// whole waves go round together (the last round's idle lanes help
	// with the roots outside the tree)
	for (int q0 = 0; q0 < n; q0 += step)
	{
		const int q = q0 + threadIdx.x / W;
		const bool valid = q < n;
		if (__ballot(valid) == 0) continue;
		const int i = valid ? cur[q] : 0;
		cd z;
		int node = 0;
		if (valid)
		{
			z = cd(zc[i].x, zc[i].y);
			node = nearest_node(L, z);
		}
		const bool outside = valid && L.nf_off[node] < 0;
		Near nr;
		for (unsigned long long m = __ballot(outside && sub == 0); m; m &= m - 1)
		{
			const int src = __ffsll(m) - 1;
			const Near t = wave_near(L, __shfl(node, src, 64), cd(__shfl(z.re, src, 64), __shfl(z.im, src, 64)));
			if ((lane & ~(W - 1)) == src) nr = t;
		}
		bool full = false;
		Witt w;
		cd f1;
		if (valid)
		{
			if (!outside) nr = chain_near(L, node, z, sub, W);
			w = witt_from(L, z, cp, sp, node, nr);
			if (!w.early) f1 = witt_f1(L, z, w);
			full = !w.early && sub == 0;
			cnt[0] += full;
			cnt[1] += w.early && sub == 0;
			cnt[2] += w.early && sub == 0;
			cnt[3] += full ? w.nr.count : 0;
		}
		const unsigned long long m = __ballot(full);
		if (m)
		{
			int base = 0;
			if (lane == 0) base = atomicAdd(nf, (int)__popcll(m));
			base = __shfl(base, 0, 64);
			if (full)
			{
				const int k = base + (int)__popcll(m & below);
				ls.fl[k] = i;
				ls.f0[k] = make_double2(w.f0.re, w.f0.im);
				ls.f1[k] = make_double2(f1.re, f1.im);
			}
		}
	}
}

// the Cauchy sums of the nf listed roots, chain_sum_lanes lanes each, and
// where they move to (in ls.f1)
template <int BS>
__device__ __forceinline__ void chain_sums(int R, int N, int circ_exact, const double2* zc, const double2* st, const ChainLists& ls, int nf)
{
	const int W = chain_sum_lanes(nf, N + R), sub = threadIdx.x & (W - 1);
	for (int g = threadIdx.x / W; g < nf; g += BS / W)
	{
		const double2 z = zc[ls.fl[g]];
		double ax = 0, ay = 0;
		chain_terms<1>(st, N, z, sub, W, ax, ay);
		ax *= 2;
		ay *= 2;
		chain_terms<-1>(zc, R, z, sub, W, ax, ay);
		if (!(isfinite(ax) && isfinite(ay)))
		{
			// out of cauchy4's range: the lane's terms one by one
			ax = ay = 0;
			for (int q = sub; q < N; q += W) cauchy1<1>(z.x, z.y, st[q], ax, ay);
			ax *= 2;
			ay *= 2;
			for (int q = sub; q < R; q += W) cauchy1<-1>(z.x, z.y, zc[q], ax, ay);
		}
		for (int o = 1; o < W; o <<= 1)
		{
			ax += __shfl_xor(ax, o, 64);
			ay += __shfl_xor(ay, o, 64);
		}
		if (sub == 0)
		{
			const double2 a0 = ls.f0[g], a1 = ls.f1[g];
			const cd zz(z.x, z.y), f0(a0.x, a0.y), f1(a1.x, a1.y);
			cd sum(ax, -ay);
			if (circ_exact) sum += 2.0 * zz.inv(); // ccf_functions.cuh:223-227
			const cd zn = zz - f0 / (f1 + f0 * sum);
			ls.f1[g] = make_double2(zn.re, zn.im);
		}
	}
}

// the nf updates written and tested, the roots that are left in nxt (*left
// their count)
template <int BS>
__device__ __forceinline__ void chain_update(const LensView& L, double2* zc, const ChainLists& ls, int nf, int* nxt, int* left,
	int (&cnt)[CHAIN_COUNTS])
{
	for (int g = threadIdx.x; g < nf; g += BS)
	{
		const int i = ls.fl[g];
		const double2 v = ls.f1[g];
		const cd dz(v.x - zc[i].x, v.y - zc[i].y);
		zc[i] = v;
		if (dz.abs() / L.theta < CONV_TOL) cnt[2]++;
		else nxt[atomicAdd(left, 1)] = i; // a non-finite step stays active
	}
}

// The sweeps of one row (at most cap) from the n active roots in ls.la (as
// written before a barrier): zc holds its roots, st the stars, ls room for
// the row's lists. s_cnt: two ints of LDS, zero.
template <int BS>
__device__ __forceinline__ void chain_row(const LensView& L, int R, int N, int circ_exact, int cap, double cp, double sp, double2* zc,
	const double2* st, const ChainLists& ls, int n, int* s_cnt, int (&cnt)[CHAIN_COUNTS])
{
	int* cur = ls.la;
	int* nxt = ls.lb;
	// s_cnt: listed this sweep, active next
	for (int it = 0; it < cap && n > 0; it++)
	{
		cnt[4] += threadIdx.x == 0;
		chain_evaluate<BS>(L, cp, sp, zc, cur, n, ls, &s_cnt[0], cnt);
		__syncthreads();
		const int nf = s_cnt[0];
		chain_sums<BS>(R, N, circ_exact, zc, st, ls, nf);
		__syncthreads();
		chain_update<BS>(L, zc, ls, nf, nxt, &s_cnt[1], cnt);
		__syncthreads();
		n = s_cnt[1];
		int* const t = cur;
		cur = nxt;
		nxt = t;
		__syncthreads();
		if (threadIdx.x == 0) s_cnt[0] = s_cnt[1] = 0;
		__syncthreads();
	}
}

} // namespace ccf
