// Exact modular arithmetic in double precision for moduli q < kFpQ = 2^50
// (the double-precision class).  Residues are integers of any sign held
// exactly in doubles; every operation below is exact on them, so the results
// are the same integers mod q the integer classes compute.
//
// Why: gfx950 issues double-precision fused multiply-adds at the rate of its
// integer multiply-adds (37.7 against 35.1 T lane-ops/s measured), and an FMA
// gives the exact low part of a product in one instruction.  A product mod q
// takes 6 instructions (12 for the integer Shoup product), signed residues
// need no offset in the difference, and a twiddle is one 8-byte double
// instead of a 16-byte pair.  Measured on MI355X, split passes, 512 x 2^16
// forward and inverse 434 -> 395 us (the passes are then bound by memory:
// 5.4 TB/s; 362 with their input streamed, batch.hip stream_input), 512 x 2^14
// 119 -> 110, a single 2^16 call 23.0 -> 21.0.
#pragma once

#include "internal.h"

namespace vk {

struct FpK {
	double q, qinv;  // q and RN(1/q)
};

// Bounds are kept in units of q/1024 at compile time.  kFpLimit: |v| <= 8q
// < 2^53, so sums within it are exact.
constexpr int kFpLimit = 8 * 1024;

// y*w - c*q for an integer c near y*w/q; |w| <= q/2, |y| <= 8q.
// h = RN(yw) and l = yw - h (exact, one FMA); c = rint(RN(h * qinv)), and
// three roundings of relative size 2^-53 leave |c - yw/q| <= 1/2 +
// 3.01 * 2^-53 * |y|/2 <= 1/2 + 0.1882 |y|/q.  h - cq = (yw - cq) - l is an
// integer below 2q + 2^48 < 2^53 in magnitude, so the FMA forms it exactly,
// and so is the last sum.
__device__ __forceinline__ double fp_mulmod(double y, double w,
		const FpK &k) {
#pragma clang fp contract(off)
	const double h = y * w;
	const double l = __builtin_fma(y, w, -h);
	const double c = __builtin_rint(h * k.qinv);
	return __builtin_fma(-c, k.q, h) + l;
}

// Bound of fp_mulmod's result for |y| <= b.
__host__ __device__ constexpr int fp_mul_bound(int b) {
	return 513 + (b * 193 + 1023) / 1024;
}

// v - c*q with c = rint(v/q): |result| <= q/2 + (error of v/q) q, below
// 513/1024 q for |v| <= 8q and below q for |v| < 2^52 and any q >= 3.
constexpr int kFpReduced = 513;

__device__ __forceinline__ double fp_reduce(double v, const FpK &k) {
#pragma clang fp contract(off)
	return __builtin_fma(-__builtin_rint(v * k.qinv), k.q, v);
}

// An integer word x < 2^52 as a double: the words 0x433 << 52 | x hold
// 2^52 + x.
__device__ __forceinline__ double fp_from_word(uint64_t x) {
	return __builtin_bit_cast(double, x | 0x4330000000000000ull) -
		4503599627370496.0;
}

// The canonical word of v, |v| <= 8q: reduced below q in magnitude, q added
// to a negative value (by masking q's bits with the sign), then the mantissa
// of 2^52 + v.  (The reduced value is never -0: an exact cancellation rounds
// to +0, and c = 0 keeps v's own sign only for v != 0.)
__device__ __forceinline__ uint64_t fp_canonical(double v, const FpK &k) {
#pragma clang fp contract(off)
	const double r = fp_reduce(v, k);
	const uint64_t rb = __builtin_bit_cast(uint64_t, r);
	const uint64_t qb = __builtin_bit_cast(uint64_t, k.q);
	const uint32_t s = (uint32_t) ((int32_t) (rb >> 32) >> 31);
	const uint64_t add = (uint64_t) ((uint32_t) (qb >> 32) & s) << 32 |
		((uint32_t) qb & s);
	const double p = r + __builtin_bit_cast(double, add) + 4503599627370496.0;
	return __builtin_bit_cast(uint64_t, p) & 0x000fffffffffffffull;
}

// ---- where values are reduced, fixed at compile time ----
//
// Forward: a butterfly leaves both outputs below |x| + fp_mul_bound(|y|).
__host__ __device__ constexpr int fp_grow(int b, int stages) {
	for (int i = 0; i < stages; i++)
		b += fp_mul_bound(b);
	return b;
}

// Bound of the values a forward first pass leaves for the second: what
// three stages still fit on top of.
constexpr int kFpForwardPass = 3700;
// Bound entering an inverse round other than a transform's first.
constexpr int kFpInverseRound = 2 * 1024;

// Inverse rounds: sums double, products of differences start again near
// q/2.  Register e of a round enters below `entry`; before[d] is the set of
// registers reduced ahead of the round's stage d (so that each butterfly's
// operands sum to at most 8q), after the set reduced when the round ends (to
// leave every register below kFpInverseRound).
struct FpInvPlan {
	int before[3], after;
	int bound[8];
};

__host__ __device__ constexpr FpInvPlan fp_inv_plan(int entry, int active,
		bool last) {
	FpInvPlan p{};
	for (int e = 0; e < 8; e++)
		p.bound[e] = entry;
	for (int d = 0; d < 3; d++) {
		if (!((active >> d) & 1))
			continue;
		for (int e = 0; e < 8; e++) {
			if ((e >> d) & 1)
				continue;
			const int f = e | (1 << d);
			while (p.bound[e] + p.bound[f] > kFpLimit) {
				const int g = p.bound[e] >= p.bound[f] ? e : f;
				p.before[d] |= 1 << g;
				p.bound[g] = kFpReduced;
			}
			const int s = p.bound[e] + p.bound[f];
			p.bound[e] = s;
			p.bound[f] = fp_mul_bound(s);
		}
	}
	for (int e = 0; e < 8 && !last; e++) {
		if (p.bound[e] > kFpInverseRound) {
			p.after |= 1 << e;
			p.bound[e] = kFpReduced;
		}
	}
	return p;
}

}  // namespace vk
