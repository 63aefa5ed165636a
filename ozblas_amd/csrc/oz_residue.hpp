// oz_residue.hpp -- device routines of the residue form shared by the single-problem kernels
// (oz_residue.hip) and the grouped batched kernels (oz_batched.hip): the balanced residues of one
// element modulo each modulus, the tiled INT8 residue-plane writer, and the Chinese-remainder
// reconstruction of one output element.  The scheme itself is described in oz_residue.hip.
#pragma once
#include "oz_digits.hpp"

namespace oz {

// ---- device: residues of one element ------------------------------------------------------
// x 2^-lo = sf 2^sh with sf a signed integer below 2^53 in magnitude and sh >= 0: sh is the exponent
// of x's last place relative to lo (clamped at 0), sf = x 2^-(lo + sh) exactly.  lo is at most the
// lowest set bit of every element of the row or column, so sf is an integer either way, and sh is at
// most the shift of x's lowest set bit (below the operand's span).  A zero x gives sf = 0, sh = 0.
struct ResElem {
	double sf;
	int sh;
};

__device__ inline ResElem res_elem(double x, int lo) {
	const int Eb = (int)((d2u(x) >> 52) & 0x7ff);  // biased exponent; 0 for zero and subnormals
	int sh = (Eb > 1 ? Eb : 1) - 1075 - lo;         // the unit of x's last place is 2^(max(Eb,1) - 1075)
	sh = sh > 0 ? sh : 0;
	return ResElem{ldexp(x, -(lo + sh)), sh};
}

// Residues by groups of three moduli: (sf 2^sh) mod P in binary64, P the group's product (< 2^24), as
// the representative nearest zero: each quotient is rounded to the nearest integer, from an estimate
// that is off by at most |v| 2^-52 / P (below 2 / P for |sf| < 2^53), so the first remainder is an
// integer of at most P / 2 + 2, its product with 2^sh mod P is exact (< 2^47), and the second remainder
// is at most P / 2 <= 2^23 in magnitude.  Every fma that forms a remainder is exact.  The sign rides on
// sf.
__device__ __forceinline__ double res_group(const ResElem &e, double P, double invP, const uint32_t *pw2) {
	double q = rint(e.sf * invP);
	const double r0 = fma(-q, P, e.sf);
	const double x = r0 * (double)pw2[e.sh];
	q = rint(x * invP);
	return fma(-q, P, x);
}

// The member residues of a group's representative rx, an integer of at most 2^23 in magnitude and so
// exact in binary32: fma(rx, RN(1/p), 1.5 2^23) rounds rx / p to the nearest integer q in one
// instruction, and its bits are those of 1.5 2^23 plus q.  q is exact: RN(1/p) is off by less than
// 2^-24 relatively, which moves rx / p by less than 2^23 2^-24 / p = 1 / (2p), and an odd p keeps rx / p
// that far from a rounding boundary; 1 / 256 is exact (a tie gives +128 or -128, one byte).  r = rx - q p
// is then the balanced residue, in [-128, 128).  Its low byte needs no more than a 24-bit
// multiply-add on the bits (0x4B400000 p is 0 modulo 2^22).
// The binary64 form of this (floor, fma, conversion, byte packing: 10.5 VALU instructions a residue
// with the group's share, against about 6) bound the writer: 0.51 ms an operand of 8192 x 8192 and 23
// moduli; with this one it takes 0.42 ms, 4.8 TB/s of reads and writes.
constexpr float kResMagic = 12582912.f;  // 1.5 2^23
__device__ __forceinline__ uint32_t res_member_byte(float rf, int ri, float invp, int negp) {
	const float t = fmaf(rf, invp, kResMagic);
	return (uint32_t)(ri + __mul24(__float_as_int(t), negp));  // the residue in the low byte
}
__device__ __forceinline__ float res_member_float(float rf, float invp, float p) {
	const float q = fmaf(rf, invp, kResMagic) - kResMagic;
	return fmaf(-q, p, rf);
}

// the per-group and per-modulus tables of the residue writers, staged in LDS by the whole workgroup
// (2^sh mod P_g only for sh below the operand's span)
struct ResLds {
	double2 g[kResMaxGroups];  // P, RN(1/P)
	float2 p[kResMaxMod];      // RN(1/p) and p
	int shs;  // row length of the shift table
};
// the shift table 2^sh mod P_g (sh below the operand's span, `shs` per group row) in the kernel's
// dynamic LDS: res_lds_bytes(nmod, shLimit) of it, so that a narrow span leaves room for more
// workgroups per CU
extern __shared__ uint32_t resPw2[];
__host__ __device__ inline size_t res_lds_bytes(int nmod, int shLimit) {
	return sizeof(uint32_t) * (size_t)((nmod + 2) / 3) * (size_t)shLimit;
}

// scaleU: the tables of op(A), whose residues carry the factors u_t (ResConst::pow2gU)
__device__ inline void res_lds_load(ResLds &T, const ResConst *rc, int nmod, int shLimit, int scaleU) {
	const int ng = (nmod + 2) / 3;
	const uint32_t(*src)[kResMaxShift] = scaleU ? rc->pow2gU : rc->pow2g;
	for (int q = threadIdx.x; q < ng * shLimit; q += blockDim.x) resPw2[q] = src[q / shLimit][q % shLimit];
	if (threadIdx.x == 0) T.shs = shLimit;
	for (int q = threadIdx.x; q < ng; q += blockDim.x) T.g[q] = make_double2(rc->Pg[q], rc->invPg[q]);
	for (int q = threadIdx.x; q < nmod; q += blockDim.x) T.p[q] = make_float2(rc->invpf[q], (float)rc->p[q]);
}

// One 256-thread workgroup: residues of the 16 columns x 64 k-bytes tile (kt, jb) of every modulus
// plane in the INT8 tiled layout (4 bytes per thread).  The blocks of 16 columns beyond n, up to the tile size of the
// product, are not written: what they hold only enters product elements outside the m x n result.
__device__ inline void res_write_tile_i8(int m, int n, const double *in, int64_t ldi, const int *colLo,
                                         int nmod, const ResLds &T, int8_t *planes, int64_t ldp,
                                         int64_t pstride, int kt, int jb) {
	const int t = threadIdx.x;
	if (kt * 64 >= m) {  // a tile of k padding only: zero residues, nothing to compute
		int8_t *dst = planes + (int64_t)jb * 16 * ldp + (int64_t)kt * 1024 + 4 * t;
		for (int s = 0; s < nmod; s++) *(uint32_t *)(dst + (int64_t)s * pstride) = 0u;
		return;
	}
	const int j = jb * 16 + t / 16;
	const int lo = (j < n) ? colLo[j] : 0;
	const double *x = in + (int64_t)(j < n ? j : 0) * ldi;
	const int q0 = kt * 64 + 4 * (t % 16);
	ResElem e[4];
#pragma unroll
	for (int u = 0; u < 4; u++) e[u] = res_elem((j < n && q0 + u < m) ? x[q0 + u] : 0.0, lo);
	int8_t *dst = planes + (int64_t)jb * 16 * ldp + (int64_t)kt * 1024 + 4 * t;
	const int ng = (nmod + 2) / 3;
	const int shs = T.shs;
	for (int gi = 0; gi < ng; gi++) {
		float rf[4];
		int ri[4];
		const double2 gp = T.g[gi];
#pragma unroll
		for (int u = 0; u < 4; u++) {
			const double rx = res_group(e[u], gp.x, gp.y, resPw2 + gi * shs);
			rf[u] = (float)rx;
			ri[u] = (int)rx;
		}
#pragma unroll
		for (int c = 0; c < 3; c++) {
			const int s = 3 * gi + c;
			if (s < nmod) {
				const float2 mp = T.p[s];
				const int negp = -(int)mp.y;
				uint32_t r[4];
#pragma unroll
				for (int u = 0; u < 4; u++) r[u] = res_member_byte(rf[u], ri[u], mp.x, negp);
				*(uint32_t *)(dst + (int64_t)s * pstride) =
				    pack_low_bytes((int)r[0], (int)r[1], (int)r[2], (int)r[3]);
			}
		}
	}
}

// v mod p for 0 <= v < 2^24 (binary32 quotient estimate off by at most one; q p with a 24-bit
// multiply: q < 2^24 / p, p <= 256)
__device__ __forceinline__ int mod_f(int v, int p, float invpf) {
	const float q = floorf((float)v * invpf);
	int r = v - (int)__umul24((uint32_t)(int)q, (uint32_t)p);
	r += (r < 0) ? p : 0;
	r -= (r >= p) ? p : 0;
	return r;
}

// an integer-valued binary64 with |d| < 2^51 as int64: d + 1.5 2^52 is exact and its fraction
// field holds d + 2^51
__device__ __forceinline__ int64_t f64_to_i64_exact(double d) {
	return (int64_t)(d2u(d + 0x1.8p52) - 0x4338000000000000ULL);
}

// a += v 2^sh (two's complement) when the bits of a at and above sh are all zero: no carries
template <int NW>
__device__ __forceinline__ void big_or_shifted(BigInt<NW> &a, int64_t v, int sh) {
	const int wi = sh >> 6, b = sh & 63;
	const uint64_t ext = (v < 0) ? ~0ULL : 0ULL;
	const uint64_t lo = (uint64_t)v << b;
	const uint64_t hi = b ? (uint64_t)(v >> (64 - b)) : ext;
#pragma unroll
	for (int q = 0; q < NW; q++) {
		if (q == wi)
			a.w[q] |= lo;
		else if (q == wi + 1)
			a.w[q] |= hi;
		else if (q > wi + 1)
			a.w[q] |= ext;
	}
}

// The four elements (i, 4g .. 4g + 3) of one product-residue word: X of each from its residues
// (nmod moduli, nchunk k-chunk planes per modulus summed modulo p), then t[e] = RN(X 2^e0[e]).
// The planes hold c_t = X u_t mod p_t < 2^8 (op(A) was written with the factors u_t);
// X = sum_t c_t M/p_t - K M is summed in binary64 chunks of 39 bits
// (every product c_t chunk < 2^47, every chunk sum of up to 49 moduli < 2^53: exact in any order),
// K = rint(sum_t c_t / p_t), and the chunks minus K M's are carried into NW 64-bit words.  The words
// of a block of moduli are loaded together (clamped indices; the surplus ones are not used).
// Rw addresses the word in plane 0; plane b is rstride bytes further.
template <int NW>
__device__ __forceinline__ void res_group_values(const uint8_t *Rw, int64_t rstride, int nchunk,
                                        const ResConst *rc, int nmod, const int *e0, double *t) {
	constexpr int NC = (64 * NW + kResChunkBits - 1) / kResChunkBits;
	if (nmod <= 0) {  // an all-zero operand: no planes
#pragma unroll
		for (int e = 0; e < 4; e++) t[e] = 0.0;
		return;
	}
	double A[4][NC];
	double S[4];
#pragma unroll
	for (int e = 0; e < 4; e++) {
		S[e] = 0.0;
#pragma unroll
		for (int c = 0; c < NC; c++) A[e][c] = 0.0;
	}
	// modulus q's residues ct[e] of the four elements enter the sums
	auto absorb = [&](int q, const double (&ct)[4]) {
		const double ipd = rc->invpd[q];
		double mp[NC];
#pragma unroll
		for (int c = 0; c < NC; c++) mp[c] = rc->Mpd[q][c];
#pragma unroll
		for (int e = 0; e < 4; e++) {
			S[e] = fma(ct[e], ipd, S[e]);
#pragma unroll
			for (int c = 0; c < NC; c++) A[e][c] = fma(ct[e], mp[c], A[e][c]);
		}
	};
	if (nchunk == 1) {
		// one k chunk: the words of QB moduli are loaded while the previous QB are absorbed, so
		// 2 QB loads per thread are in flight
		constexpr int QB = 8;
		uint32_t w[QB];
		auto load = [&](uint32_t(&d)[QB], int q0) {
#pragma unroll
			for (int j = 0; j < QB; j++) d[j] = *(const uint32_t *)(Rw + (int64_t)min(q0 + j, nmod - 1) * rstride);
		};
		load(w, 0);
		for (int q0 = 0; q0 < nmod; q0 += QB) {
			uint32_t wn[QB];
			load(wn, min(q0 + QB, nmod - 1));
#pragma unroll
			for (int j = 0; j < QB; j++) {
				if (q0 + j >= nmod) break;
				double ct[4];
#pragma unroll
				for (int e = 0; e < 4; e++) ct[e] = (double)((w[j] >> (8 * e)) & 255);
				absorb(q0 + j, ct);
			}
#pragma unroll
			for (int j = 0; j < QB; j++) w[j] = wn[j];
		}
	} else {
		// several k chunks: the chunks' residues of a modulus are summed (below 2^24) and reduced
		constexpr int QB = 4;
		for (int q0 = 0; q0 < nmod; q0 += QB) {
			int rs[QB][4];
#pragma unroll
			for (int j = 0; j < QB; j++)
#pragma unroll
				for (int e = 0; e < 4; e++) rs[j][e] = 0;
			for (int c = 0; c < nchunk; c++) {
				uint32_t w[QB];
#pragma unroll
				for (int j = 0; j < QB; j++) {
					const int q = min(q0 + j, nmod - 1);
					w[j] = *(const uint32_t *)(Rw + (int64_t)(c * nmod + q) * rstride);
				}
#pragma unroll
				for (int j = 0; j < QB; j++)
#pragma unroll
					for (int e = 0; e < 4; e++) rs[j][e] += (int)((w[j] >> (8 * e)) & 255);
			}
#pragma unroll
			for (int j = 0; j < QB; j++) {
				const int q = q0 + j;
				if (q >= nmod) break;
				const int p = rc->p[q];
				const float ipf = rc->invpf[q];
				double ct[4];
#pragma unroll
				for (int e = 0; e < 4; e++) ct[e] = (double)mod_f(rs[j][e], p, ipf);  // rs < 2^24
				absorb(q, ct);
			}
		}
	}
#pragma unroll
	for (int e = 0; e < 4; e++) {
		const double K = rint(S[e]);
		// chunk c of X is d_c = A_c - K M_c, exact: 0 <= A_c < 49 * 255 * 2^39 < 2^52.61 and
		// |K M_c| < 2^45.  The carries run in binary64: hi = floor(d_c 2^-39) (at most 2^13.61 in
		// magnitude) moves to d_(c+1), which stays below 2^53, and leaves d_c in [0, 2^39); every step
		// is exact.  The top chunk carries the sign, |d_top| < 2^51 because |X| < 2^(64 NW - 1).
		double d[NC];
#pragma unroll
		for (int c = 0; c < NC; c++) d[c] = fma(-K, rc->Md[c], A[e][c]);
#pragma unroll
		for (int c = 0; c + 1 < NC; c++) {
			const double hi = floor(d[c] * 0x1p-39);
			d[c] = fma(-hi, 0x1p39, d[c]);
			d[c + 1] += hi;
		}
		// the chunks occupy disjoint bit ranges: X is their OR
		BigInt<NW> X;
#pragma unroll
		for (int q = 0; q < NW; q++) X.w[q] = 0;
#pragma unroll
		for (int c = 0; c < NC; c++) big_or_shifted<NW>(X, f64_to_i64_exact(d[c]), kResChunkBits * c);
		t[e] = big_finish<NW>(X, e0[e]);
	}
}

// one thread per (row i, column group g) of an M x N product: C(i, 4g + e) = fma(alpha, RN(X 2^(lo_i +
// lo_j)), beta C) for the columns of the group inside N
template <int NW>
__device__ __forceinline__ void res_recon_group(int M, int N, const uint8_t *R, int64_t ldr, int64_t rstride,
                                       int nchunk, const ResConst *rc, int nmod, const int *rowLo,
                                       const int *colLo, double alpha, double beta, double *C,
                                       int64_t ldc, int i, int g) {
	int e0[4];
	const int li = rowLo[i];
#pragma unroll
	for (int e = 0; e < 4; e++) e0[e] = li + ((4 * g + e < N) ? colLo[4 * g + e] : 0);
	double t[4];
	res_group_values<NW>(R + res_word_offset(i, 4 * g, ldr), rstride, nchunk, rc, nmod, e0, t);
#pragma unroll
	for (int e = 0; e < 4; e++) {
		const int j = 4 * g + e;
		if (j < N) {
			double *c = C + (int64_t)j * ldc + i;
			*c = fma(alpha, t[e], beta * *c);
		}
	}
}

// ---- the reconstruction on the matrix units ---------------------------------------------------
// X' = sum_t c_t M/p_t is a product of the byte matrix (elements x moduli) with the digits of the
// M/p_t, so up to 32 moduli of 32 elements are one v_mfma_i32_32x32x32_i8: limb b of element e is
// sum_t (c_t - 128) w_tb, below 2^19, on accumulators that start at the limbs of 128 sum_t M/p_t.  A wave
// takes 32 rows x 4 columns: lane l loads the words (row l % 32, 4 columns) of the moduli
// 16 (l / 32) .. + 15, turns them into four MFMA operands by byte permutes, and after four MFMAs holds
// 16 of the 32 limbs of four elements; neighbouring limbs are paired and a swap of the lane halves
// leaves lane l with all limbs of two elements: row l % 32, columns (l / 32) * 2 and the next.
// In scalar binary64 (res_group_values) the sums are 6 instructions per element and modulus and the
// carry and rounding another 240: 407 VALU instructions an element at 23 moduli, which bound the kernel
// (8192 x 8192: 0.89 ms).  Here it is memory: 0.61 ms, 4.3 TB/s of residues, C in and C out.

// the instance (NL) for a product of nl words
inline int res_recon_words(int nl) { return nl <= 4 ? 4 : nl <= 6 ? 6 : 8; }

// RN(x 2^e0) for the two's-complement integer x (NL 32-bit words, least significant first).  The
// result is never subnormal and never overflows: the fast forms are taken only when every product is a
// multiple of 2^-1000 and below 2^1000 (fast_valid).
template <int NL>
__device__ __forceinline__ double res_round(uint32_t (&x)[NL], int e0) {
	const bool neg = (int32_t)x[NL - 1] < 0;
	const uint32_t sm = neg ? 0xffffffffu : 0u;
	uint32_t carry = sm & 1u;
#pragma unroll
	for (int q = 0; q < NL; q++) {
		const uint32_t v = x[q] ^ sm;
		x[q] = v + carry;
		carry = x[q] < carry ? 1u : 0u;
	}
	// zero words at the top move out, 4, 2 and 1 at a time
	int sh = 0;
#pragma unroll
	for (int s = 4; s >= 1; s /= 2) {
		if (s >= NL) continue;
		uint32_t top = 0;
#pragma unroll
		for (int q = 0; q < s; q++) top |= x[NL - 1 - q];
		const bool z = top == 0;
#pragma unroll
		for (int q = NL - 1; q >= 0; q--) x[q] = z ? (q >= s ? x[q - s] : 0u) : x[q];
		sh += z ? 32 * s : 0;
	}
	// the 64 bits from the leading one, everything below folded into the last of them: the one
	// rounding of the fma is then the rounding of x
	const int lz = x[NL - 1] ? __builtin_clz(x[NL - 1]) : 0;
	const uint64_t hi = (((uint64_t)x[NL - 1] << 32) | x[NL - 2]) << lz;
	const uint64_t lo = (((uint64_t)x[NL - 2] << 32) | x[NL - 3]) << lz;
	uint32_t rest = (uint32_t)lo;
#pragma unroll
	for (int q = 0; q < NL - 3; q++) rest |= x[q];
	const uint32_t mid = (uint32_t)(lo >> 32) | (rest ? 1u : 0u);
	const double r = fma((double)(uint32_t)(hi >> 32), 0x1p32, (double)mid);
	const double t = ldexp(r, e0 + 32 * (NL - 2) - sh - lz);
	return neg ? -t : t;
}

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// per-lane state of a wave's reconstruction: the digit operand and the accumulator start
struct ResWave {
	l2v w;
	i16v init;
	__device__ void load(const ResTab *tab) {
		const int l = threadIdx.x % 64;
		const u4v v = *(const u4v *)tab->w[l];
		w = __builtin_bit_cast(l2v, v);
#pragma unroll
		for (int r = 0; r < 16; r++) init[r] = tab->init[l / 32][r];
	}
};

// rows i0 .. i0 + 31 and columns 4g .. 4g + 3 of C by one wave; km: the table -K M in LDS
template <int NL>
__device__ __forceinline__ void res_recon_wave(const ResWave &ws, const uint32_t (*km)[8], double invM, int M,
                                               int N, const uint8_t *R, int64_t ldr, int64_t rstride, int nmod,
                                               const int *rowLo, const int *colLo, double alpha, double beta,
                                               double *C, int64_t ldc, int i0, int g) {
	const int l = threadIdx.x % 64, h = l / 32;
	const int i = i0 + l % 32;
	const bool row = i < M;
	const int ic = row ? i : M - 1;
	const uint8_t *Rw = R + res_word_offset(ic, 4 * g, ldr);
	uint32_t w[16];
#pragma unroll
	for (int j = 0; j < 16; j++)  // (a word beyond the moduli meets zero digits)
		w[j] = *(const uint32_t *)(Rw + (int64_t)min(16 * h + j, nmod - 1) * rstride);
	double *cp[2], c0[2];
	int e0[2];
	bool in[2];
	const int li = rowLo[ic];
#pragma unroll
	for (int c = 0; c < 2; c++) {
		const int j = 4 * g + 2 * h + c;
		in[c] = row && j < N;
		const int jc = j < N ? j : N - 1;
		cp[c] = C + (int64_t)jc * ldc + ic;
		c0[c] = *cp[c];
		e0[c] = li + colLo[jc];
	}
	u4v b[4];
#pragma unroll
	for (int a = 0; a < 4; a++) {
		// 4 x 4 byte transpose of the words of moduli 4a .. 4a + 3, then c_t - 128 as int8
		const uint32_t t0 = __builtin_amdgcn_perm(w[4 * a + 1], w[4 * a], 0x05010400);
		const uint32_t t1 = __builtin_amdgcn_perm(w[4 * a + 1], w[4 * a], 0x07030602);
		const uint32_t t2 = __builtin_amdgcn_perm(w[4 * a + 3], w[4 * a + 2], 0x05010400);
		const uint32_t t3 = __builtin_amdgcn_perm(w[4 * a + 3], w[4 * a + 2], 0x07030602);
		b[0][a] = __builtin_amdgcn_perm(t2, t0, 0x05040100) ^ 0x80808080u;
		b[1][a] = __builtin_amdgcn_perm(t2, t0, 0x07060302) ^ 0x80808080u;
		b[2][a] = __builtin_amdgcn_perm(t3, t1, 0x05040100) ^ 0x80808080u;
		b[3][a] = __builtin_amdgcn_perm(t3, t1, 0x07060302) ^ 0x80808080u;
	}
	int32_t p[4][8];
#pragma unroll
	for (int c = 0; c < 4; c++) {
		const i16v acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(ws.w, __builtin_bit_cast(l2v, b[c]), ws.init, 0, 0, 0);
#pragma unroll
		for (int r = 0; r < 8; r++) p[c][r] = acc[2 * r] + (acc[2 * r + 1] << 8);  // below 2^28
	}
#pragma unroll
	for (int c = 0; c < 2; c++) {
		int32_t q[16];
#pragma unroll
		for (int r = 0; r < 8; r++) {
			const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)p[c][r], (uint32_t)p[c + 2][r], false, false);
			q[r] = (int32_t)s[0];
			q[8 + r] = (int32_t)s[1];
		}
		// carries in base 2^16, two digits a word; X' is non-negative
		uint32_t x[NL];
		int32_t carry = 0;
#pragma unroll
		for (int k = 0; k < NL; k++) {
			const int32_t a = q[2 * k] + carry;
			const int32_t d = q[2 * k + 1] + (a >> 16);
			x[k] = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)a, 0x05040100);
			carry = d >> 16;
		}
		// X = X' - K M, K = rint(X' / M), with X / M at most 1/4 in magnitude: the three top words give
		// X' / M to 2^-24 for the word counts nl (ResConst) of the instance, NL - 1 and NL (M is above
		// 2^(32 (nl - 1) - 7)); NL = 4 serves every smaller count too, with all four words
		double f = fma((double)x[NL - 1], 0x1p32, (double)x[NL - 2]);
		f = fma((double)x[NL - 3], 0x1p-32, f);
		if (NL == 4) f = fma((double)x[0], 0x1p-64, f);
		const int K = (int)rint(f * invM);
		uint32_t cy = 0;
#pragma unroll
		for (int k = 0; k < NL; k++) {
			const uint64_t v = (uint64_t)x[k] + km[K][k] + cy;
			x[k] = (uint32_t)v;
			cy = (uint32_t)(v >> 32);
		}
		const double t = res_round<NL>(x, e0[c]);
		if (in[c]) *cp[c] = fma(alpha, t, beta * c0[c]);
	}
}

}  // namespace oz
