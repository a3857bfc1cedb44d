// Device helpers shared by the grouped GEMM kernels: operand addressing and the lane-held term descriptors.

#pragma once

#include <hip/hip_runtime.h>
#include "ct_internal.h"

namespace ctg {

typedef double double4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ const double* rebase(const double* base, const double* off)
{
	return (const double*)((const char*)base + (intptr_t)off);
}

// Term descriptors of a task are held one per lane (64 at a time, one vector load) and read with
// v_readlane: walking the terms costs no dependent memory round trip.
struct TermCache
{
	uint32_t w[12];   // the GemmTerm of term base + lane (12 dwords)
	int base;
};

static_assert(sizeof(GemmTerm) == 48, "GemmTerm layout");

__device__ __forceinline__ void term_cache_load(TermCache& c, const GemmTerm* __restrict__ terms, int base, int t1, int lane)
{
	c.base = base;
	const int idx = base + lane;
	if (idx < t1) {
		const uint4* src = (const uint4*)(terms + idx);
		const uint4 a = src[0], b = src[1], d = src[2];
		c.w[0] = a.x; c.w[1] = a.y; c.w[2] = a.z; c.w[3] = a.w;
		c.w[4] = b.x; c.w[5] = b.y; c.w[6] = b.z; c.w[7] = b.w;
		c.w[8] = d.x; c.w[9] = d.y; c.w[10] = d.z; c.w[11] = d.w;
	}
	else {
		#pragma unroll
		for (int i = 0; i < 12; i++) c.w[i] = 0;
	}
}

__device__ __forceinline__ uint32_t term_word(const TermCache& c, int t, int i)
{
	return (uint32_t)__builtin_amdgcn_readlane((int)c.w[i], t - c.base);
}

__device__ __forceinline__ int term_K(const TermCache& c, int t) { return (int)term_word(c, t, 6); }

__device__ __forceinline__ const double* term_ptr(const TermCache& c, int t, int i)
{
	const uint64_t lo = term_word(c, t, i), hi = term_word(c, t, i + 1);
	return (const double*)(intptr_t)(lo | (hi << 32));
}

// The fields of term t: the task's first term comes with the work item (scalar registers), later
// ones from the lane-held cache. Uniform across the wavefront.
struct TermF
{
	const double* A;
	const double* B;
	int64_t sb_batch;
	int K, sa_i, sa_k, sb_k, sb_j;
};

__device__ __forceinline__ TermF term_fields(const TermCache& c, int t, const GemmTerm& first, int t0)
{
	TermF f;
	if (t == t0) {
		f.A = first.A; f.B = first.B; f.sb_batch = first.sb_batch;
		f.K = first.K; f.sa_i = first.sa_i; f.sa_k = first.sa_k; f.sb_k = first.sb_k; f.sb_j = first.sb_j;
	}
	else {
		f.A = term_ptr(c, t, 0); f.B = term_ptr(c, t, 2); f.sb_batch = (int64_t)term_ptr(c, t, 4);
		f.K = term_K(c, t); f.sa_i = (int)term_word(c, t, 7); f.sa_k = (int)term_word(c, t, 8);
		f.sb_k = (int)term_word(c, t, 9); f.sb_j = (int)term_word(c, t, 10);
	}
	return f;
}

__device__ __forceinline__ int term_K_at(const TermCache& c, int t, const GemmTerm& first, int t0)
{
	return (t == t0) ? first.K : term_K(c, t);
}

// the cache of a task's terms: loaded (one vector load) only when the task has more than one term,
// in flight while the first term's operands are loaded
__device__ __forceinline__ void term_cache_start(TermCache& c, const GemmTerm* __restrict__ terms, const GemmTask& tk, int lane)
{
	c.base = tk.t0;
	if (tk.t1 - tk.t0 > 1) term_cache_load(c, terms, tk.t0, tk.t1, lane);
}

// identity DPP moves: the cache words get registers written by a VALU op, so that later readlanes
// wait for nothing (the wait for the cache load happens here, once)
__device__ __forceinline__ void term_cache_settle(TermCache& c)
{
	#pragma unroll
	for (int i = 0; i < 12; i++) c.w[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)c.w[i], 0xE4, 0xF, 0xF, false);
}

}  // namespace ctg
