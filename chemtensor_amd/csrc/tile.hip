// LDS-tiled grouped FP64 GEMM for gfx950: one workgroup per 64 x 64 output tile of a task, operands
// through raw buffer loads and LDS panels, 16x16x4 MFMA.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "ct_internal.h"
#include "gemm_device.h"
#include "tile_device.h"

namespace ctg {

// The descriptors are read through the constant address space: scalar loads into scalar registers.
typedef const __attribute__((address_space(4))) GemmTerm* TermPtr;
typedef const __attribute__((address_space(4))) WorkItem* ItemPtr;

struct TileTerm { const double* A; const double* B; int K, sa_i, sa_k, sb_k; };

__device__ __forceinline__ TileTerm load_term(TermPtr p)
{
	return TileTerm{ p->A, p->B, p->K, p->sa_i, p->sa_k, p->sb_k };
}

// the loads of one thread of a panel: two neighbouring entries each
struct TilePanel { double2_t a[2], b[2]; };

// One 64 x 64 tile per workgroup of four wavefronts, terms in order and k ascending in steps of four (the
// order of the wavefront forms). What bounds it: the FP64 matrix rate. A 16x16x4 MFMA holds its SIMD for
// 64 cycles; vector instructions do not run beside it and a vector memory instruction costs it 25 to 28
// cycles whatever its width (measured with four wavefronts per SIMD), so the panel loop has as few of both
// as possible: loads are 16 bytes wide at 8-byte alignment, their per-thread offsets stay the same over the
// panels of a term (the descriptor's base moves, on the scalar unit), and rows, columns and k past the
// operand read zero from the descriptor's range check instead of a select. The next panel is in flight in
// registers while the current one is multiplied from a single LDS buffer (18 KB; 76 VGPRs, 72 with DOT: six
// or seven workgroups per CU; a double buffer with one barrier per panel allows four: 172 us against 160 us
// for stage 1 of a Hubbard bond of 2000 states, 6.3 GFLOP). Now 136 us for that stage (49.6 TFLOP/s executed,
// the pipe busy 63 % of the time) and 167 us for stage 3, whose 1441 tiles are one uneven round (53 %).
// AK: A is stored k by k (sa_i 1), else row by row (sa_k 1); B is stored k by k (sb_j 1).
// DOT: udot[tile] = the sum of its entries times x at their indices in the result vector (butterfly within
// each wavefront, then the four wavefronts in order).
template <bool AK, bool DOT>
__global__ __launch_bounds__(256, 4) void k_tile_gemm_f64(const GemmTerm* __restrict__ terms, const WorkItem* __restrict__ items, GemmBases bs,
	const double* __restrict__ x, double* __restrict__ udot)
{
	__shared__ __attribute__((aligned(16))) double sa[TPANEL];
	__shared__ __attribute__((aligned(16))) double sb[TPANEL];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = uni(tid >> 6);
	const ItemPtr it = (ItemPtr)(uintptr_t)items + blockIdx.x;
	const TermPtr ct = (TermPtr)(uintptr_t)terms;
	const int m0 = it->m0, n0 = it->n0;
	const int M = it->task.M, N = it->task.N, t1 = it->task.t1;
	// a panel stored k by k: this thread loads entries 2 q, 2 q + 1 of k rows kr and kr + 8; row by row:
	// k 2 q, 2 q + 1 of rows ir and ir + 32
	const int kr = tid >> 5, kc = 2 * (tid & 31), ir = tid >> 3, iq = 2 * (tid & 7);
	int t = it->task.t0, left = 0;     // term, and its k from the next panel on
	TileTerm cur = load_term(&it->first), nxt = cur;
	TileOperand oa = { 0, 0 }, ob = { 0, 0 };
	int stepa = 0, stepb = 0, va0 = 0, va1 = 0, vb0 = 0, vb1 = 0;
	auto open_term = [&]() {
		const TileTerm& f = cur;
		left = f.K;
		oa.p = (uint64_t)(uintptr_t)rebase(bs.A, f.A);
		ob.p = (uint64_t)(uintptr_t)rebase(bs.B, f.B);
		oa.bytes = 8 * (AK ? (f.K - 1) * f.sa_k + M : (M - 1) * f.sa_i + f.K);
		ob.bytes = 8 * ((f.K - 1) * f.sb_k + N);
		stepa = AK ? 8 * TK * f.sa_k : 8 * TK;
		stepb = 8 * TK * f.sb_k;
		vb0 = n0 + kc < N ? 8 * (kr * f.sb_k + n0 + kc) : TILE_OOB;
		vb1 = vb0 + 64 * f.sb_k;
		if constexpr (AK) {
			va0 = m0 + kc < M ? 8 * (kr * f.sa_k + m0 + kc) : TILE_OOB;
			va1 = va0 + 64 * f.sa_k;
		}
		else {
			va0 = m0 + ir < M ? 8 * ((m0 + ir) * f.sa_i + iq) : TILE_OOB;
			va1 = m0 + ir + 32 < M ? 8 * ((m0 + ir + 32) * f.sa_i + iq) : TILE_OOB;
		}
	};
	// the next term with entries, from term t on (in cur); none: nothing left and every load past the end.
	// The descriptor after it is loaded ahead.
	auto seek_term = [&]() {
		while (t < t1 && cur.K <= 0) {
			cur = nxt;
			t++;
			if (t + 1 < t1) nxt = load_term(ct + t + 1);
		}
		if (t < t1) open_term();
		else { left = 0; oa.bytes = 0; ob.bytes = 0; }
	};
	if (t + 1 < t1) nxt = load_term(ct + t + 1);
	seek_term();
	const bool any = left > 0;
	// the next panel into registers; returns its k (0: none left)
	auto issue = [&](TilePanel& r) -> int {
		const __amdgpu_buffer_rsrc_t ra = oa.rsrc(), rb = ob.rsrc();
		r.b[0] = buf_load2(rb, vb0);
		r.b[1] = buf_load2(rb, vb1);
		r.a[0] = buf_load2(ra, va0);
		r.a[1] = buf_load2(ra, va1);
		const int k = min(left, TK);
		if (left > TK) {
			left -= TK;
			oa.advance(stepa);
			ob.advance(stepb);
		}
		else if (left > 0) {
			cur.K = 0;
			seek_term();
		}
		return k;
	};
	const int wk = (kr >> 2) * T_STEP + (kr & 3) * T_Q + (kc >> 5) * T_PAIR + 2 * (kc & 15) + ((kc >> 4) & 1);
	const int wi = (iq >> 2) * T_STEP + (iq & 3) * T_Q + 2 * (ir & 15) + (ir >> 4);
	auto store_panel = [&](const TilePanel& r, int k) {
		double* const pb = sb + wk;
		pb[0] = r.b[0].x;
		pb[2] = r.b[0].y;
		pb[2 * T_STEP] = r.b[1].x;
		pb[2 * T_STEP + 2] = r.b[1].y;
		if constexpr (AK) {
			double* const pa = sa + wk;
			pa[0] = r.a[0].x;
			pa[2] = r.a[0].y;
			pa[2 * T_STEP] = r.a[1].x;
			pa[2 * T_STEP + 2] = r.a[1].y;
		}
		else {
			double* const pa = sa + wi;
			double2_t a0 = r.a[0], a1 = r.a[1];
			if (k < TK) {
				// k past the term: what follows in the row form is the next row's
				if (iq >= k) { a0.x = 0; a1.x = 0; }
				if (iq + 1 >= k) { a0.y = 0; a1.y = 0; }
			}
			pa[0] = a0.x;
			pa[T_Q] = a0.y;
			pa[T_PAIR] = a1.x;
			pa[T_PAIR + T_Q] = a1.y;
		}
	};
	double4_t acc00 = { 0, 0, 0, 0 }, acc01 = acc00, acc10 = acc00, acc11 = acc00;
	const int i16 = lane & 15, kq = lane >> 4;
	// the 16 x 16 sub-tiles inside the task (nm x nn of 4 x 4) are dealt to the wavefronts: a quadrant
	// each, or, when at most two rows (columns) of sub-tiles are inside, a column (row) of them each
	const int nm = M - m0 > 48 ? 4 : (M - m0 + 15) >> 4, nn = N - n0 > 48 ? 4 : (N - n0 + 15) >> 4;
	int rb0, cb0, NMr, NNr;   // first sub-tile row and column, and how many of each
	if (nm <= 2) { rb0 = 0; cb0 = wave; NMr = nm; NNr = wave < nn ? 1 : 0; }
	else if (nn <= 2) { rb0 = wave; cb0 = 0; NMr = wave < nm ? 1 : 0; NNr = nn; }
	else { rb0 = 2 * (wave >> 1); cb0 = 2 * (wave & 1); NMr = min(2, max(0, nm - rb0)); NNr = min(2, max(0, nn - cb0)); }
	const int fa = kq * T_Q + 2 * i16 + (rb0 >> 1) * T_PAIR + (rb0 & 1);
	const int fb = kq * T_Q + 2 * i16 + (cb0 >> 1) * T_PAIR + (cb0 & 1);
	auto mainloop = [&](auto cm, auto cn) {
		constexpr int NM = decltype(cm)::value, NN = decltype(cn)::value;
		auto step = [&](const double* pa, const double* pb, int st) {
			if constexpr (NM > 0 && NN > 0) {
				double2_t a, b;
				if constexpr (NM > 1) a = *(const double2_t*)(pa + st * T_STEP); else a.x = pa[st * T_STEP];
				if constexpr (NN > 1) b = *(const double2_t*)(pb + st * T_STEP); else b.x = pb[st * T_STEP];
				acc00 = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, acc00, 0, 0, 0);
				if constexpr (NN > 1) acc01 = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, acc01, 0, 0, 0);
				if constexpr (NM > 1) acc10 = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, acc10, 0, 0, 0);
				if constexpr (NM > 1 && NN > 1) acc11 = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, acc11, 0, 0, 0);
			}
		};
		// the k-steps that hold entries
		auto compute = [&](int k) {
			const double* const pa = sa + fa;
			const double* const pb = sb + fb;
			step(pa, pb, 0);
			if (k > 4) step(pa, pb, 1);
			if (k > 8) step(pa, pb, 2);
			if (k > 12) step(pa, pb, 3);
		};
		TilePanel r;
		int k = issue(r);
		store_panel(r, k);
		__syncthreads();
		while (true) {
			const int next = issue(r);
			compute(k);
			if (next == 0) break;
			__syncthreads();
			store_panel(r, next);
			__syncthreads();
			k = next;
		}
	};
	typedef std::integral_constant<int, 0> c0;
	typedef std::integral_constant<int, 1> c1;
	typedef std::integral_constant<int, 2> c2;
	if (any) {
		if (NMr == 2 && NNr == 2) mainloop(c2(), c2());
		else if (NMr == 2 && NNr == 1) mainloop(c2(), c1());
		else if (NMr == 1 && NNr == 2) mainloop(c1(), c2());
		else if (NMr == 1 && NNr == 1) mainloop(c1(), c1());
		else mainloop(c0(), c0());
	}
	// store: register r of lane l holds D(l / 16 + 4 r, l % 16) of each sub-tile; entries outside the task
	// go past the end
	const int sc_i = it->task.sc_i;
	const TileOperand oc = { (uint64_t)(uintptr_t)rebase(bs.C, it->task.C), 8 * ((M - 1) * sc_i + N) };
	const __amdgpu_buffer_rsrc_t rc = oc.rsrc();
	const TileOperand ox = { DOT ? (uint64_t)(uintptr_t)(x + it->task.pad) : 0, DOT ? oc.bytes : 0 };
	const __amdgpu_buffer_rsrc_t rx = ox.rsrc();
	double dot = 0;
	#pragma unroll
	for (int sub = 0; sub < 4; sub++) {
		const int mi = sub >> 1, ni = sub & 1;
		if (mi >= NMr || ni >= NNr) continue;
		const double4_t acc = (sub == 0 ? acc00 : sub == 1 ? acc01 : sub == 2 ? acc10 : acc11);
		const int col = n0 + 16 * (cb0 + ni) + i16, row0 = m0 + 16 * (rb0 + mi) + kq;
		const int off = col < N ? 8 * (row0 * sc_i + col) : TILE_OOB;
		#pragma unroll
		for (int rr = 0; rr < 4; rr++) {
			const int o = row0 + 4 * rr < M ? off + 32 * rr * sc_i : TILE_OOB;
			__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, (double)acc[rr]), rc, o, 0, 0);
			if constexpr (DOT) dot += acc[rr] * __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rx, o, 0, 0));
		}
	}
	if constexpr (DOT) {
		#pragma unroll
		for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o, 64);
		__syncthreads();
		if (lane == 0) sa[wave] = dot;
		__syncthreads();
		if (tid == 0) udot[blockIdx.x] = (sa[0] + sa[1]) + (sa[2] + sa[3]);
	}
}

void launch_tile_gemm_f64(bool a_kmajor, const GemmTerm* terms, const WorkItem* items, int nitems, GemmBases b, hipStream_t s, const double* x,
	double* udot)
{
	if (nitems == 0) return;
	const dim3 grid((unsigned)nitems), block(256);
	if (udot && a_kmajor) hipLaunchKernelGGL((k_tile_gemm_f64<true, true>), grid, block, 0, s, terms, items, b, x, udot);
	else if (udot) throw HipError{ hipErrorInvalidValue, "tiled GEMM: products with x need a k-major A" };
	else if (a_kmajor) hipLaunchKernelGGL((k_tile_gemm_f64<true, false>), grid, block, 0, s, terms, items, b, x, udot);
	else hipLaunchKernelGGL((k_tile_gemm_f64<false, false>), grid, block, 0, s, terms, items, b, x, udot);
	CTG_HIP(hipGetLastError());
}

}  // namespace ctg
