// oz_narrow.hip -- the plain form's GEMM where its slices are narrow: the binary32 routines and the
// mixed ones of binary64 data in binary32 slices (<float,float,float>, <double,float,float>).
//
// Their slices hold b = prec - rho = floor((24 - log2 k) / 2) bits: slice s of a row or column is
// q 2^u, u = rho + tau_s - prec, with q an integer of |q| <= 2^b, and by the choice of rho a pair's
// product over k terms is an integer of at most 24 bits in units 2^(u_a + u_b) (reference
// src/cpu/ozblas_split.cpp:20-34,151-189).  So the products run on the matrix units for small
// numbers, and stay exact: INT8 with INT32 accumulators for b <= 6 (k > 1024), FP16 with FP32
// accumulators for 7 <= b <= 11 (k >= 2; |q| <= 2048 is exact in FP16, the sums stay below 2^24).
// The sum then takes P = isum 2^(u_a + u_b), exact in binary64, through the same term rounding and in
// the same order as the FP64 kernel, so every bit of the result is the same.
//
// What bounds it: at 1000 x 1100 x 1200 (8 x 8 slices) the 64 products are 169 GOP; the FP64 matrix
// units need 2.5 ms for that and the fused ordered sum walked all 64 pairs in one workgroup per
// 128 x 128 tile, 72 workgroups on 256 CUs: 14.3 ms.  Here: split 33 us, INT8 products 124 us (1.4 POP/s;
// short k, so the pipeline's fill and the int32 stores count), sum 90 us (282 MB of int32 planes, 3.1 TB/s).
#include "oz_digits.hpp"

namespace oz {

__device__ __forceinline__ double scale2(double a, int e) { return ldexp(a, e); }
__device__ __forceinline__ float scale2(float a, int e) { return ldexpf(a, e); }

// q of one slice element; the four of a thread go out as one word
template <class TO>
struct NarrowOut;
template <>
struct NarrowOut<int8_t> {
	// tiled INT8 layout (16 columns x 64 k in one KiB), the layout of i8_tile
	static __device__ int64_t offset(int j, int i, int64_t ldp) {
		return (int64_t)(j / 16) * 16 * ldp + (int64_t)(i / 64) * 1024 + (j % 16) * 64 + i % 64;
	}
	static __device__ void store(int8_t *p, const int (&q)[4]) {
		*(uint32_t *)p = (uint32_t)(q[0] & 255) | (uint32_t)(q[1] & 255) << 8 | (uint32_t)(q[2] & 255) << 16 |
		                 (uint32_t)(q[3] & 255) << 24;
	}
};
template <>
struct NarrowOut<_Float16> {
	static __device__ int64_t offset(int j, int i, int64_t ldp) { return (int64_t)j * ldp + i; }
	static __device__ void store(_Float16 *p, const int (&q)[4]) {
		typedef _Float16 h4 __attribute__((ext_vector_type(4)));
		*(h4 *)p = h4{(_Float16)(float)q[0], (_Float16)(float)q[1], (_Float16)(float)q[2], (_Float16)(float)q[3]};
	}
};

__device__ inline void narrow_max(int *p, int v) {
	if (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < v) atomicMax(p, v);
}

// The split of k_split_cols_reg (same operations in the same order, column in registers) with the
// slices stored as their integers q.  NT threads take one column: a wave for columns of up to 512 (no
// barrier), a workgroup beyond (1100 columns of 1200, one wave each: 43 us; 256 threads each 37 us, with the
// reductions on the DPP network and the maxima a cache line apart 16 us).  Each thread holds R4 groups of four
// consecutive elements, so a plane is written in words.  ue[s cols + j] = u of slice s; a level past the column's last non-zero
// remainder is not written here (k_narrow_zero).  stat: kNarrowSlots copies of four maxima from zero:
// first zero level, 1 for a column outside the integer model, kNarrowOff - min u, kNarrowOff + max u.
template <int NT, int R4, class TI, class TO>
__global__ __launch_bounds__(NT < 256 ? 256 : NT) void k_narrow_split(int m, int n, const TI *in, int64_t ldi,
                                                                     TO *planes, int64_t ldp, int64_t pstride,
                                                                     int rho, int cap, const uint16_t *J, int *ue,
                                                                     int *zcol, int *stat) {
	constexpr int BS = NT < 256 ? 256 : NT;
	__shared__ double red[2 * BS / 64];
	int par = 0;
	const int t = threadIdx.x % NT;
	const int j = blockIdx.x * (BS / NT) + threadIdx.x / NT;
	if (j >= n) return;  // a whole wave, or (NT >= 256) a whole workgroup: j < n there by the grid
	const TI *x = in + (int64_t)j * ldi;
	TI v[4 * R4];
	double mx = 0.0;
	int bad = 0;
#pragma unroll
	for (int g = 0; g < R4; g++)
#pragma unroll
		for (int u = 0; u < 4; u++) {
			const int i = 4 * (t + NT * g) + u;
			v[4 * g + u] = (i < m) ? x[i] : (TI)0;
		}
#pragma unroll
	for (int q = 0; q < 4 * R4; q++) {
		if (!isfinite(v[q])) bad = 1;
		mx = std_max(mx, fabs((double)v[q]));
	}
	auto reduce = [&](double a) { return block_max_nonneg<NT>(a, red, par); };
	mx = reduce(mx);
	const bool zcolumn = mx == 0.0;
	int s = 0, lo = 0, hi = 0;
	bool zero = false;
	for (s = 0; s < cap; s++) {
		const int tau = SplitRule<TI>::tau(mx, J);
		const TI sigma = SplitRule<TI>::sigma(rho, tau, 1);
		const int u0 = rho + tau - SplitRule<TI>::kPrec;
		// |slice| <= 2^tau, i.e. |q| <= 2^b, for the largest remainder (and so, the rounding being
		// monotone, for all); a sigma out of range fails it too
		if (!(fabs((double)(((TI)mx + sigma) - sigma)) <= ldexp(1.0, tau))) bad = 1;
		TI lm = 0;
#pragma unroll
		for (int g = 0; g < R4; g++) {
			const int i = 4 * (t + NT * g);
			int q[4];
#pragma unroll
			for (int u = 0; u < 4; u++) {
				const TI a = (v[4 * g + u] + sigma) - sigma;
				v[4 * g + u] = v[4 * g + u] - a;
				lm = max_abs(lm, v[4 * g + u]);
				q[u] = (int)scale2(a, -u0);
			}
			if (i < ldp) NarrowOut<TO>::store(planes + (int64_t)s * pstride + NarrowOut<TO>::offset(j, i, ldp), q);
		}
		if (t == 0) ue[(int64_t)s * n + j] = zcolumn ? 0 : u0;
		lo = (s == 0) ? kNarrowOff - u0 : max(lo, kNarrowOff - u0);
		hi = (s == 0) ? kNarrowOff + u0 : max(hi, kNarrowOff + u0);
		mx = reduce((double)lm);
		if (mx == 0.0) {
			zero = true;
			break;
		}
	}
	const int z = zero ? s : cap;
	int *st = stat + kNarrowSlotInts * (blockIdx.x % kNarrowSlots);
	if (t == 0) {
		zcol[j] = z;
		narrow_max(st, z);
		if (!zcolumn) {
			narrow_max(st + 2, lo);
			narrow_max(st + 3, hi);
		}
	}
	if (bad) narrow_max(st + 1, 1);
}

// zero slices [zcol[j] + 1, count) of every column (and their exponents)
template <class TO>
__global__ __launch_bounds__(64) void k_narrow_zero(int n, TO *planes, int64_t ldp, int64_t pstride, int *ue,
                                                    const int *zcol, int count) {
	const int j = blockIdx.x;
	const int q[4] = {0, 0, 0, 0};
	for (int s = zcol[j] + 1; s < count; s++) {
		for (int i = 4 * threadIdx.x; i < ldp; i += 256)
			NarrowOut<TO>::store(planes + (int64_t)s * pstride + NarrowOut<TO>::offset(j, i, ldp), q);
		if (threadIdx.x == 0) ue[(int64_t)s * n + j] = 0;
	}
}

// t = the ordered sum of np pair products (T planes of int32; pair p's term is T_p 2^(u_a + u_b)), one
// thread per row and four columns; then C = fma(alpha, t, beta C).  carry: the running sums (m x n,
// pitch m) between the launches of a product whose planes do not fit at once.  The row blocks of four columns, then
// the next four, on grid x: grid y ends at 65536, 262144 columns.
// STORE (binary32): the terms replace the int32 values, for the NearSum kernels; eight pairs a workgroup (grid y), as
// nothing orders them (one workgroup for all pairs waited for memory eight at a time: 64 pairs of 16 x 16 39 us, 8 so).
constexpr int kNarrowStep = 8;  // pairs whose loads are issued before their terms are used
template <class T, bool STORE>
__global__ __launch_bounds__(256) void k_narrow_sum(int m, int n, int32_t *P, int64_t ldt, int64_t tstride,
                                                    const int2 *pairs, int np, const int *ueA, const int *ueB,
                                                    T *carry, int first, int last, T alpha, T beta, T *C,
                                                    int64_t ldc) {
	const int rb = (m + 255) / 256;
	const int i = ((int)blockIdx.x % rb) * 256 + (int)threadIdx.x;
	const int j0 = 4 * ((int)blockIdx.x / rb);
	if (i >= m) return;
	const int nc = min(4, n - j0);
	T t[4];
#pragma unroll
	for (int c = 0; c < 4; c++) t[c] = (!STORE && !first && c < nc) ? carry[(int64_t)(j0 + c) * m + i] : (T)0;
	int32_t *p0 = P + (int64_t)j0 * ldt + i;
	constexpr int U = kNarrowStep;
	const int p1 = STORE ? min(np, U * ((int)blockIdx.y + 1)) : np;
	for (int pb = STORE ? U * (int)blockIdx.y : 0; pb < p1; pb += U) {
		int32_t v[U][4];
		int e[U][4];
#pragma unroll
		for (int u = 0; u < U; u++) {
			const int p = min(pb + u, np - 1);
			const int2 pr = pairs[p];
			const int ea = ueA[(int64_t)pr.x * m + i];
#pragma unroll
			for (int c = 0; c < 4; c++) {
				const int cc = min(c, nc - 1);
				v[u][c] = p0[(int64_t)p * tstride + (int64_t)cc * ldt];
				e[u][c] = ea + ueB[(int64_t)pr.y * n + j0 + cc];
			}
		}
#pragma unroll
		for (int u = 0; u < U; u++) {
			if (pb + u < np) {
#pragma unroll
				for (int c = 0; c < 4; c++) {
					const T term = sum_term<T>(ldexp((double)v[u][c], e[u][c]));
					if constexpr (STORE) {
						if (c < nc) *(T *)(p0 + (int64_t)(pb + u) * tstride + (int64_t)c * ldt) = term;
					} else {
						t[c] = t[c] + term;
					}
				}
			}
		}
	}
	if constexpr (STORE) return;
#pragma unroll
	for (int c = 0; c < 4; c++) {
		if (c < nc) {
			if (last) {
				T *d = C + (int64_t)(j0 + c) * ldc + i;
				*d = fma1_t(alpha, t[c], beta * *d);
			} else {
				carry[(int64_t)(j0 + c) * m + i] = t[c];
			}
		}
	}
}

template <class TI, class TO>
static void narrow_split(hipStream_t st, int m, int n, const TI *in, int64_t ldi, void *planes, int64_t ldp,
                         int64_t pstride, int rho, int cap, const uint16_t *J, int *ue, int *zcol, int *stat) {
#define OZ_NARROW(NT, R4)                                                                                    \
	hipLaunchKernelGGL((k_narrow_split<NT, R4, TI, TO>), dim3((n + (NT < 256 ? 256 / NT : 1) - 1) / (NT < 256 ? 256 / NT : 1)), \
	                   dim3(NT < 256 ? 256 : NT), 0, st, m, n, in, ldi, (TO *)planes, ldp, pstride, rho, cap, \
	                   J, ue, zcol, stat)
	if (ldp <= 256 * 2)
		OZ_NARROW(64, 2);
	else if (ldp <= 1024)
		OZ_NARROW(256, 1);
	else if (ldp <= 1024 * 2)
		OZ_NARROW(256, 2);
	else if (ldp <= 1024 * 4)
		OZ_NARROW(256, 4);
	else if (ldp <= 1024 * 8)
		OZ_NARROW(256, 8);
	else
		OZ_NARROW(1024, 8);
#undef OZ_NARROW
}

template <class TI>
static void narrow_split_any(hipStream_t st, int elem, int m, int n, const TI *in, int64_t ldi, void *planes,
                             int64_t ldp, int64_t pstride, int rho, int cap, const uint16_t *J, int *ue, int *zcol,
                             int *stat) {
	if (elem == 1)
		narrow_split<TI, int8_t>(st, m, n, in, ldi, planes, ldp, pstride, rho, cap, J, ue, zcol, stat);
	else
		narrow_split<TI, _Float16>(st, m, n, in, ldi, planes, ldp, pstride, rho, cap, J, ue, zcol, stat);
}

void launch_narrow_split(hipStream_t st, int elem, int m, int n, const double *in, int64_t ldi, void *planes,
                         int64_t ldp, int64_t pstride, int rho, int cap, const uint16_t *J, int *ue, int *zcol,
                         int *stat) {
	narrow_split_any(st, elem, m, n, in, ldi, planes, ldp, pstride, rho, cap, J, ue, zcol, stat);
}
void launch_narrow_split(hipStream_t st, int elem, int m, int n, const float *in, int64_t ldi, void *planes,
                         int64_t ldp, int64_t pstride, int rho, int cap, const uint16_t *J, int *ue, int *zcol,
                         int *stat) {
	narrow_split_any(st, elem, m, n, in, ldi, planes, ldp, pstride, rho, cap, J, ue, zcol, stat);
}

void launch_narrow_zero(hipStream_t st, int elem, int n, void *planes, int64_t ldp, int64_t pstride, int *ue,
                        const int *zcol, int count) {
	if (elem == 1)
		hipLaunchKernelGGL(k_narrow_zero<int8_t>, dim3(n), dim3(64), 0, st, n, (int8_t *)planes, ldp, pstride, ue,
		                   zcol, count);
	else
		hipLaunchKernelGGL(k_narrow_zero<_Float16>, dim3(n), dim3(64), 0, st, n, (_Float16 *)planes, ldp, pstride,
		                   ue, zcol, count);
}

static dim3 narrow_sum_grid(int m, int n) { return dim3((unsigned)((m + 255) / 256) * (unsigned)((n + 3) / 4)); }

template <class T>
static void narrow_sum(hipStream_t st, int m, int n, int32_t *P, int64_t ldt, int64_t tstride, const int2 *pairs,
                       int np, const int *ueA, const int *ueB, T *carry, int first, int last, T alpha, T beta,
                       T *C, int64_t ldc) {
	hipLaunchKernelGGL((k_narrow_sum<T, false>), narrow_sum_grid(m, n), dim3(256), 0, st, m, n, P, ldt,
	                   tstride, pairs, np, ueA, ueB, carry, first, last, alpha, beta, C, ldc);
}
void launch_narrow_sum(hipStream_t st, int m, int n, int32_t *P, int64_t ldt, int64_t tstride, const int2 *pairs,
                       int np, const int *ueA, const int *ueB, double *carry, int first, int last, double alpha,
                       double beta, double *C, int64_t ldc) {
	narrow_sum(st, m, n, P, ldt, tstride, pairs, np, ueA, ueB, carry, first, last, alpha, beta, C, ldc);
}
void launch_narrow_sum(hipStream_t st, int m, int n, int32_t *P, int64_t ldt, int64_t tstride, const int2 *pairs,
                       int np, const int *ueA, const int *ueB, float *carry, int first, int last, float alpha,
                       float beta, float *C, int64_t ldc) {
	narrow_sum(st, m, n, P, ldt, tstride, pairs, np, ueA, ueB, carry, first, last, alpha, beta, C, ldc);
}
void launch_narrow_terms_f(hipStream_t st, int m, int n, int32_t *P, int64_t ldt, int64_t tstride,
                           const int2 *pairs, int np, const int *ueA, const int *ueB) {
	dim3 g = narrow_sum_grid(m, n);
	g.y = (np + kNarrowStep - 1) / kNarrowStep;
	hipLaunchKernelGGL((k_narrow_sum<float, true>), g, dim3(256), 0, st, m, n, P, ldt,
	                   tstride, pairs, np, ueA, ueB, (float *)nullptr, 1, 1, 1.f, 0.f, (float *)nullptr, 0);
}

}  // namespace oz
