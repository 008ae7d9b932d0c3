// One-pass transforms of n = 2^14 for the double-precision class (q < kFpQ)
// with 32 words per thread.  Included by ntt_fused.h.
//
// A tile of 2^14 words with eight words per thread and round (Geo) takes
// 144 KiB of LDS, so one workgroup per CU: its loads, arithmetic and stores
// follow each other with nothing beside them, and its five rounds exchange
// four times.  Here a thread keeps 32 words in registers (64 of 128 VGPRs,
// four waves per SIMD) and runs five stages between exchanges, so two
// exchanges are left, one of them inside each wave; and an exchange moves the
// low halves of all words first and the high halves after them through 66 KiB
// of LDS, so two workgroups share a CU and one's loads and stores run beside
// the other's arithmetic.
// Measured on MI355X, forward + inverse, us, against eight words per thread:
// 512 polynomials 89.5 -> 80.5, 2048 329 -> 295.  Not all of the arithmetic fits
// the 128 registers: the compiler spills 34 values of the forward (92 bytes of
// scratch per lane) and 6 of the inverse (28 bytes), and the forward's
// spilled words show as 20% more written than the result holds.
#pragma once

namespace vk {

constexpr int kWideBits = 5;  // log2 words per thread
constexpr int kWideWords = 1 << kWideBits;

// Three rounds by field position (the thread's words differ in the five index
// bits from F up): the top five bits, bits 4 to 8, bits 0 to 4.  A wave's
// words in the last two are the same 2^11 consecutive ones.
template <int LOGN>
struct Wide {
	static constexpr int THREADS = 1 << (LOGN - kWideBits);
	static constexpr int F1 = LOGN - kWideBits;
	static constexpr int F2 = F1 - kWideBits > 4 ? F1 - kWideBits : 4;
	// one padding word per 32: lanes 32 words apart (field 0) and runs of
	// sixteen lanes 512 apart (field 4) fall on different banks
	static constexpr int LDS = (1 << LOGN) + (1 << (LOGN - 5));
};

__device__ __forceinline__ constexpr uint32_t wide_pad(uint32_t i) {
	return i + (i >> 5);
}

// Index of word 0 of thread t with the field at F; word e is at + (e << F).
template <int F>
__device__ __forceinline__ uint32_t wide_base(uint32_t t) {
	return ((t >> F) << (F + kWideBits)) | (t & ((1u << F) - 1));
}

// Index of word 0 of thread t in lane order (whole waves on consecutive
// words, as global accesses take them); word e is at + 64 e.
__device__ __forceinline__ uint32_t wide_lane_base(uint32_t t) {
	return ((t >> 6) << (6 + kWideBits)) | (t & 63);
}

// A read that is not paired with its neighbour: a pair would arrive in two
// adjacent registers, the low halves of two words, and each cost a move.
__device__ __forceinline__ uint32_t wide_read(const uint32_t *p) {
	const uint32_t v = *p;
	asm volatile("" ::: "memory");
	return v;
}

// Moves the thread's words from index `from` + k * FROM to `to` + k * TO.
// CROSS: between waves.  Of the two orders one is always a wave's own 2^11
// words (see Wide), so the next exchange, which writes those, needs no barrier
// after this one, nor this one before it.  The padding is additive over the
// disjoint bit fields of a base and its steps.
template <int FROM, int TO, bool CROSS>
__device__ __forceinline__ void wide_exchange(double x[kWideWords],
		uint32_t *lds, uint32_t from, uint32_t to) {
	const uint32_t pf = wide_pad(from), pt = wide_pad(to);
	uint32_t lo[kWideWords], hi[kWideWords];
#pragma unroll
	for (int e = 0; e < kWideWords; e++) {
		const uint64_t b = __builtin_bit_cast(uint64_t, x[e]);
		lo[e] = (uint32_t) b;
		hi[e] = (uint32_t) (b >> 32);
	}
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		lds[pf + wide_pad(e * FROM)] = lo[e];
	exchange_sync<CROSS>();
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		lo[e] = wide_read(lds + pt + wide_pad(e * TO));
	exchange_sync<CROSS>();
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		lds[pf + wide_pad(e * FROM)] = hi[e];
	exchange_sync<CROSS>();
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		hi[e] = wide_read(lds + pt + wide_pad(e * TO));
	wave_sync();
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		x[e] = __builtin_bit_cast(double, (uint64_t) hi[e] << 32 | lo[e]);
}

// Twiddle of the thread's butterfly group g at stage bit F + D, `hi` the index
// bits above the field (tw_pos: the thread's groups are 2^(4 - D) consecutive
// ones from a multiple of that).
template <int LOGN, int F, int D>
__device__ __forceinline__ double wide_tw(const double *tw, uint32_t hi, int g) {
	constexpr uint32_t M = 1u << (LOGN - 1 - F - D);
	const uint32_t first = hi << (kWideBits - 1 - D);
	if constexpr (M < 4)
		return gload_tw(tw, M + first + (uint32_t) g);
	else
		return gload_tw(tw, tw_pos(M, first) + (g & 3) * (M >> 2) + (g >> 2));
}

// Forward stages D, D - 1, ..., END of the field at F.
template <int LOGN, int F, int D, int END>
__device__ __forceinline__ void wide_forward(double x[kWideWords],
		const double *tw, uint32_t hi, const FpK &k) {
#pragma clang fp contract(off)
	if constexpr (D >= END) {
#pragma unroll
		for (int g = 0; g < (kWideWords / 2 >> D); g++) {
			const double w = wide_tw<LOGN, F, D>(tw, hi, g);
#pragma unroll
			for (int l = 0; l < (1 << D); l++) {
				const int e = (g << (D + 1)) | l, f = e | (1 << D);
				const double t = fp_mulmod(x[f], w, k);
				x[f] = x[e] - t;
				x[e] = x[e] + t;
			}
		}
		wide_forward<LOGN, F, D - 1, END>(x, tw, hi, k);
	}
}

// Where the forward's rounds reduce every value first: bounds in q/1024 as
// for the eight-word rounds (canonical input below q).
template <int LOGN>
struct WideForward {
	using W = Wide<LOGN>;
	static constexpr int B1 = fp_grow(1024, kWideBits);
	static constexpr int S2 = W::F1 - W::F2;
	static constexpr bool RED2 = fp_grow(B1, S2) > kFpLimit;
	static constexpr int B2 = fp_grow(RED2 ? kFpReduced : B1, S2);
	static constexpr bool RED3 = fp_grow(B2, W::F2) > kFpLimit;
	static constexpr int B3 = fp_grow(RED3 ? kFpReduced : B2, W::F2);
	// (fp_scale_word's difference is a word below q less such a value)
	static_assert(B1 <= kFpLimit && B2 <= kFpLimit && B3 + 1024 <= kFpLimit,
			"forward values past 8q");
};

__device__ __forceinline__ void wide_reduce(double x[kWideWords],
		const FpK &k) {
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		x[e] = fp_reduce(x[e], k);
}

// FpInvPlan for 32 registers and the stages [0, STAGES) of a field (or, TOP,
// its upper STAGES): before[d] and after are masks of registers to reduce.
struct WideInvPlan {
	uint32_t before[kWideBits], after;
	int bound[kWideWords];
};

__host__ __device__ constexpr WideInvPlan wide_inv_plan(int entry, int stages,
		bool last) {
	WideInvPlan p{};
	for (int e = 0; e < kWideWords; e++)
		p.bound[e] = entry;
	for (int d = 0; d < stages; d++) {
		for (int e = 0; e < kWideWords; e++) {
			if ((e >> d) & 1)
				continue;
			const int f = e | (1 << d);
			while (p.bound[e] + p.bound[f] > kFpLimit) {
				const int g = p.bound[e] >= p.bound[f] ? e : f;
				p.before[d] |= 1u << g;
				p.bound[g] = kFpReduced;
			}
			const int s = p.bound[e] + p.bound[f];
			p.bound[e] = s;
			p.bound[f] = fp_mul_bound(s);
		}
	}
	for (int e = 0; e < kWideWords && !last; e++) {
		if (p.bound[e] > kFpInverseRound) {
			p.after |= 1u << e;
			p.bound[e] = kFpReduced;
		}
	}
	return p;
}

// Inverse stages D, D + 1, ..., STAGES - 1 of the field at F, entered below
// ENTRY; the transform's last stage has n^-1 folded in (src/vector.c:633-638).
template <int LOGN, int F, int D, int STAGES, int ENTRY>
__device__ __forceinline__ void wide_inverse(double x[kWideWords],
		const double *tw, uint32_t hi, const NttConsts &c, const FpK &k) {
#pragma clang fp contract(off)
	constexpr bool LAST = F + STAGES == LOGN;
	constexpr WideInvPlan plan = wide_inv_plan(ENTRY, STAGES, LAST);
	if constexpr (D < STAGES) {
#pragma unroll
		for (int e = 0; e < kWideWords; e++) {
			if ((plan.before[D] >> e) & 1)
				x[e] = fp_reduce(x[e], k);
		}
#pragma unroll
		for (int g = 0; g < (kWideWords / 2 >> D); g++) {
			const double w = LAST && D == STAGES - 1 ? c.fw1n
				: wide_tw<LOGN, F, D>(tw, hi, g);
#pragma unroll
			for (int l = 0; l < (1 << D); l++) {
				const int e = (g << (D + 1)) | l, f = e | (1 << D);
				const double s = x[e] + x[f], t = x[e] - x[f];
				x[e] = LAST && D == STAGES - 1 ? fp_mulmod(s, c.fninv, k) : s;
				x[f] = fp_mulmod(t, w, k);
			}
		}
		wide_inverse<LOGN, F, D + 1, STAGES, ENTRY>(x, tw, hi, c, k);
	} else {
#pragma unroll
		for (int e = 0; e < kWideWords; e++) {
			if ((plan.after >> e) & 1)
				x[e] = fp_reduce(x[e], k);
		}
	}
}

// The forward's input words as doubles and its first stage, as fp_round has
// them: words below q convert as they are; a wave holding a larger one reduces
// them all while they are below 2^52, and otherwise takes the reference's
// first stage in integers.
template <int LOGN>
__device__ __forceinline__ void wide_first(double x[kWideWords],
		uint64_t v[kWideWords], const double *tw, const ulonglong2 *pairs,
		const NttConsts &c, const FpK &k) {
#pragma clang fp contract(off)
	constexpr int H = kWideWords / 2;
	bool canon = true;
	uint32_t top = 0;
#pragma unroll
	for (int e = 0; e < kWideWords; e++) {
		canon &= v[e] < c.q;
		top |= (uint32_t) (v[e] >> 32);
	}
	if (!__all(canon) && !__all(top < (1u << 20))) {
		const ulonglong2 w1 = gload_tw(pairs, 1);
#pragma unroll
		for (int e = 0; e < H; e++)
			bf_fwd_first(v[e], v[e + H], w1, c);
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			x[e] = fp_from_word(v[e]);
		return;
	}
#pragma unroll
	for (int e = 0; e < kWideWords; e++)
		x[e] = fp_from_word(v[e]);
	if (!__all(canon))
		wide_reduce(x, k);
	const double w = gload_tw(tw, 1);
#pragma unroll
	for (int e = 0; e < H; e++) {
		const double t = fp_mulmod(x[e + H], w, k);
		x[e + H] = x[e] - t;
		x[e] = x[e] + t;
	}
}

// One workgroup per task (or per polynomial after `uniform`), as k_ntt_fused.
template <int LOGN, bool INV>
__global__ __launch_bounds__((Wide<LOGN>::THREADS))
__attribute__((amdgpu_waves_per_eu(4, 4))) void k_ntt_wide(NttTask uniform,
		const NttTask *tasks) {
	using W = Wide<LOGN>;
	__shared__ uint32_t lds[W::LDS];
	NttTask task;
	if (tasks) {
		task = tasks[blockIdx.x];
	} else {
		task = uniform;
		const uint64_t off = (uint64_t) blockIdx.x << LOGN;
		task.in += off;
		task.out += off;
		if (task.in2)
			task.in2 += off;
	}
	const NttConsts &c = task.c;
	const FpK k{c.fq, c.fqinv};
	const double *tw = tw_fp(task.tw, 1u << LOGN, INV);
	const uint32_t t = threadIdx.x;
	const uint32_t lane0 = wide_lane_base(t);
	double x[kWideWords];
	uint64_t v[kWideWords];
	if constexpr (!INV) {
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			v[e] = gload_in<0>(task.in, t + (e << W::F1));
		if (c.lift_add) {
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				v[e] = lift_word(v[e], c);
		}
		wide_first<LOGN>(x, v, tw, task.tw, c, k);
		wide_forward<LOGN, W::F1, kWideBits - 2, 0>(x, tw, 0, k);
		wide_exchange<1 << W::F1, 1 << W::F2, true>(x, lds, t,
				wide_base<W::F2>(t));
		if constexpr (WideForward<LOGN>::RED2)
			wide_reduce(x, k);
		wide_forward<LOGN, W::F2, W::F1 - W::F2 - 1, 0>(x, tw, t >> W::F2, k);
		wide_exchange<1 << W::F2, 1, false>(x, lds, wide_base<W::F2>(t),
				t << kWideBits);
		if constexpr (WideForward<LOGN>::RED3)
			wide_reduce(x, k);
		wide_forward<LOGN, 0, W::F2 - 1, 0>(x, tw, t, k);
		if (c.scale_w) {
			wide_exchange<1, 64, false>(x, lds, t << kWideBits, lane0);
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				gstore(task.out, lane0 + 64 * e, fp_scale_word(gload_in<0>(task.in2,
								lane0 + 64 * e), __builtin_bit_cast(uint64_t, x[e]), c));
		} else {
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				x[e] = __builtin_bit_cast(double, fp_canonical(x[e], k));
			wide_exchange<1, 64, false>(x, lds, t << kWideBits, lane0);
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				gstore(task.out, lane0 + 64 * e, __builtin_bit_cast(uint64_t, x[e]));
		}
	} else {
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			v[e] = gload_in<0>(task.in, lane0 + 64 * e);
		if (task.in2) {
			// the product of two canonical spectra
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				v[e] = spectra_product(v[e], gload_in<0>(task.in2, lane0 + 64 * e), c);
		}
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			x[e] = fp_from_word(v[e]);
		wide_exchange<64, 1, false>(x, lds, lane0, t << kWideBits);
		wide_inverse<LOGN, 0, 0, W::F2, 1024>(x, tw, t, c, k);
		wide_exchange<1, 1 << W::F2, false>(x, lds, t << kWideBits,
				wide_base<W::F2>(t));
		wide_inverse<LOGN, W::F2, 0, W::F1 - W::F2, kFpInverseRound>(x, tw,
				t >> W::F2, c, k);
		wide_exchange<1 << W::F2, 1 << W::F1, true>(x, lds, wide_base<W::F2>(t),
				t);
		wide_inverse<LOGN, W::F1, 0, kWideBits, kFpInverseRound>(x, tw, 0, c, k);
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			v[e] = fp_canonical(x[e], k);
		if (c.post_p) {
#pragma unroll
			for (int e = 0; e < kWideWords; e++)
				v[e] = post_center(v[e], c);
		}
#pragma unroll
		for (int e = 0; e < kWideWords; e++)
			gstore(task.out, t + (e << W::F1), v[e]);
	}
}

}  // namespace vk
