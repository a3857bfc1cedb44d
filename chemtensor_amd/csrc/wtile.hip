// Stage 2 of the matvec, T2 = W_D T1, for classes whose W_D is too large for the column stream (the merged
// operators of quantum chemistry: hundreds of rows and columns, one entry in five not zero). The rows of a
// class are gathered into tiles of 64 with similar sets of non-zero columns; a tile keeps only the columns
// that some row of it uses, so neither their T1 entries are read nor the products formed.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <numeric>
#include "ct_internal.h"
#include "gemm_device.h"
#include "tile_device.h"

namespace ctg {

constexpr int WT_KMAX = 2048;    // columns of a row tile (their T1 offsets are kept in LDS, 16 KB)

typedef const __attribute__((address_space(4))) WtItem* WtItemPtr;
typedef const __attribute__((address_space(4))) uint32_t* MaskPtr;

// One workgroup per 64 rows of W_D and 64 columns (a, c) of a block pair; each wavefront takes all rows of 16
// columns. What bounds it: the operand loads (a T1 panel is read again by each row tile that uses it; molecular
// operator of 20 orbitals, 512 states: 7.1 GB in 1119 us, 6.3 TB/s) and, next, the FP64 matrix cores (busy 56 %
// of the time, 49 GFLOP for 20 GFLOP of products with entries that are not zero). W comes packed in panels of 16 kept columns in fragment order; within a tile
// the kept columns are sorted by the 16-row sub-tiles that use them, and a k-step runs the MFMAs of the
// sub-tiles in its mask only. Columns are paired within a row a (an odd dC is padded by one column that is
// computed and not stored), so that T1 loads are 16 bytes wide.
__global__ __launch_bounds__(256, 4) void k_wtile(const WtItem* __restrict__ items, const int64_t* __restrict__ kbase, const int* __restrict__ kstride,
	const int64_t* __restrict__ rbase, const int* __restrict__ rstride, const int* __restrict__ lists, const uint32_t* __restrict__ masks,
	const double* __restrict__ pack, const double* __restrict__ t1, double* __restrict__ t2)
{
	__shared__ __attribute__((aligned(16))) double sa[1024];
	__shared__ __attribute__((aligned(16))) double sb[1024];
	__shared__ int2 ko[WT_KMAX];
	__shared__ int2 ro[64];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = uni(tid >> 6);
	const WtItemPtr it = (WtItemPtr)(uintptr_t)items + blockIdx.x;
	const int np = it->np, dA = it->dA, dC = it->dC, j0 = it->j0;
	const int dCp = (dC + 1) & ~1;
	for (int i = tid; i < np * TK; i += 256) {
		const int k = lists[it->klist + i];
		const int64_t b = k >= 0 ? kbase[it->kb + k] : -1;
		int2 e;
		e.x = b >= 0 ? (int)((b - it->t1_off) * 8) : TILE_OOB;
		e.y = b >= 0 ? kstride[it->kb + k] * 8 : 0;
		ko[i] = e;
	}
	if (tid < 64) {
		const int r = lists[it->rlist + tid];
		const int64_t b = r >= 0 ? rbase[it->rb + r] : -1;
		int2 e;
		e.x = b >= 0 ? (int)((b - it->t2_off) * 8) : TILE_OOB;
		e.y = b >= 0 ? rstride[it->rb + r] * 8 : 0;
		ro[tid] = e;
	}
	// this thread's T1 entries of a panel: k rows kr and kr + 8, columns j, j + 1 (one row a, c even)
	const int kr = tid >> 5, kc = 2 * (tid & 31);
	const int j = j0 + kc, a = j / dCp, c8 = 8 * (j - a * dCp);
	const int out = a < dA ? 0 : TILE_OOB;
	const TileOperand ob = { (uint64_t)(uintptr_t)(t1 + it->t1_off), it->t1_bytes }, oc = { (uint64_t)(uintptr_t)(t2 + it->t2_off), it->t2_bytes };
	TileOperand oa = { (uint64_t)(uintptr_t)(pack + it->pack), np * TK * 64 * 8 };
	const MaskPtr mp = (MaskPtr)(uintptr_t)masks + it->mask;
	__syncthreads();
	struct Panel { double2_t a[2], b[2]; };
	auto issue = [&](Panel& r, int p) {
		const __amdgpu_buffer_rsrc_t ra = oa.rsrc(), rb = ob.rsrc();
		const int2 e0 = ko[min(p, np - 1) * TK + kr], e1 = ko[min(p, np - 1) * TK + kr + 8];
		r.b[0] = buf_load2(rb, (e0.x + a * e0.y + c8) | out);
		r.b[1] = buf_load2(rb, (e1.x + a * e1.y + c8) | out);
		r.a[0] = buf_load2(ra, 16 * tid);
		r.a[1] = buf_load2(ra, 16 * tid + 4096);
		oa.advance(8192);
	};
	// T1 panel in LDS: entry (k, 16 sub + i) at (4 (k / 4) + sub) 64 + 16 (k % 4) + i
	double* const pb = sb + ((kr >> 2) * 4 + (kc >> 4)) * 64 + (kr & 3) * 16 + (kc & 15);
	auto store = [&](const Panel& r) {
		*(double2_t*)pb = r.b[0];
		*(double2_t*)(pb + 512) = r.b[1];
		*(double2_t*)(sa + 2 * tid) = r.a[0];
		*(double2_t*)(sa + 2 * tid + 512) = r.a[1];
	};
	const int i16 = lane & 15, kq = lane >> 4;
	// the 16-column sub-tiles inside the pair (nn of 4) are dealt to the wavefronts: one each with all four
	// row sub-tiles, or, with one or two of them, a column sub-tile with one or two row sub-tiles each
	const int cols = dA * dCp - j0, nn = cols > 48 ? 4 : (cols + 15) >> 4;
	const int cw = nn > 2 ? wave : nn == 2 ? wave & 1 : 0;
	const uint32_t rm = nn > 2 ? (wave < nn ? 15u : 0u) : nn == 2 ? (wave & 2 ? 12u : 3u) : 1u << wave;
	const double* const fb = sb + cw * 64 + lane;
	const double* const fa = sa + 2 * lane;
	double4_t acc0 = { 0, 0, 0, 0 }, acc1 = acc0, acc2 = acc0, acc3 = acc0;
	Panel r;
	issue(r, 0);
	store(r);
	__syncthreads();
	for (int p = 0; ; p++) {
		const uint32_t m = mp[p];
		issue(r, p + 1);
		#pragma unroll
		for (int st = 0; st < TK / 4; st++) {
			const uint32_t q = (m >> (4 * st)) & rm;
			const double b = fb[st * 256];
			if (q & 3) {
				const double2_t f = *(const double2_t*)(fa + st * 256);
				if (q & 1) acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, b, acc0, 0, 0, 0);
				if (q & 2) acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(f.y, b, acc1, 0, 0, 0);
			}
			if (q & 12) {
				const double2_t f = *(const double2_t*)(fa + st * 256 + 128);
				if (q & 4) acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(f.x, b, acc2, 0, 0, 0);
				if (q & 8) acc3 = __builtin_amdgcn_mfma_f64_16x16x4f64(f.y, b, acc3, 0, 0, 0);
			}
		}
		if (p + 1 >= np) break;
		__syncthreads();
		store(r);
		__syncthreads();
	}
	// register r of lane l holds row l / 16 + 4 r, column l % 16 of each sub-tile
	const int js = j0 + 16 * cw + i16, as = js / dCp, cs = js - as * dCp;
	const int oj = as < dA && cs < dC ? 0 : TILE_OOB;
	const __amdgpu_buffer_rsrc_t rc = oc.rsrc();
	#pragma unroll
	for (int s = 0; s < 4; s++) {
		if (!(rm >> s & 1)) continue;
		const double4_t acc = s == 0 ? acc0 : s == 1 ? acc1 : s == 2 ? acc2 : acc3;
		#pragma unroll
		for (int rr = 0; rr < 4; rr++) {
			const int2 e = ro[16 * s + kq + 4 * rr];
			__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, (double)acc[rr]), rc, (e.x + as * e.y + 8 * cs) | oj, 0, 0);
		}
	}
}

// Groups of up to n of the column sets in 'bits' (nw words each), greedily: the largest remaining set, then
// the sets that add the fewest columns to the group (ties: that share the most with it).
static std::vector<std::vector<int>> greedy_groups(const std::vector<uint64_t>& bits, int count, int nw, int n)
{
	std::vector<int> size((size_t)count, 0), rest((size_t)count), add((size_t)count), fresh((size_t)nw);
	for (int r = 0; r < count; r++) for (int q = 0; q < nw; q++) size[(size_t)r] += __builtin_popcountll(bits[(size_t)r * nw + q]);
	std::iota(rest.begin(), rest.end(), 0);
	std::stable_sort(rest.begin(), rest.end(), [&](int x, int y) { return size[(size_t)x] > size[(size_t)y]; });
	std::vector<std::vector<int>> groups;
	while (!rest.empty()) {
		std::vector<int> g;
		std::vector<uint64_t> u((size_t)nw, 0), gain((size_t)nw, 0);
		for (const int r : rest) add[(size_t)r] = size[(size_t)r];   // columns that r would add to the group
		size_t best = 0;
		while ((int)g.size() < n && !rest.empty()) {
			if (!g.empty()) {
				int bn = INT32_MAX, bo = -1;
				for (size_t i = 0; i < rest.size(); i++) {
					const int r = rest[i], overlap = size[(size_t)r] - add[(size_t)r];
					if (add[(size_t)r] < bn || (add[(size_t)r] == bn && overlap > bo)) { bn = add[(size_t)r]; bo = overlap; best = i; }
				}
			}
			const int r = rest[best];
			g.push_back(r);
			rest.erase(rest.begin() + (ptrdiff_t)best);
			best = 0;
			// the group's new columns (words 'fresh' of 'gain') are none to add any more
			int nf = 0;
			for (int q = 0; q < nw; q++) {
				gain[(size_t)q] = bits[(size_t)r * nw + q] & ~u[(size_t)q];
				if (gain[(size_t)q]) fresh[(size_t)nf++] = q;
				u[(size_t)q] |= gain[(size_t)q];
			}
			if (nf > 0)
				for (const int i : rest) {
					const uint64_t* w = &bits[(size_t)i * nw];
					int c = 0;
					for (int k = 0; k < nf; k++) c += __builtin_popcountll(w[fresh[(size_t)k]] & gain[(size_t)fresh[(size_t)k]]);
					add[(size_t)i] -= c;
				}
		}
		groups.push_back(std::move(g));
	}
	return groups;
}

// The row tiles of one class, W_D (R x K row-major): rows in groups of 64 with similar columns (the 16 rows
// of a sub-tile are then similar as well: groups of 16 first, and these in fours, take a quarter more MFMAs on
// the molecular operator of 20 orbitals, 1.25 against 1.12 ms), a tile's columns sorted by the sub-tiles that
// use them and padded to whole panels. Appends to h.lists, h.masks and h.pack.
static void plan_row_tiles(WtHost& h, const std::vector<double>& w, int R, int K, std::vector<WtTile>& tiles)
{
	const int nw = (K + 63) / 64;
	std::vector<uint64_t> bits((size_t)R * nw, 0);
	for (int r = 0; r < R; r++)
		for (int k = 0; k < K; k++)
			if (w[(size_t)r * K + k] != 0.0) bits[(size_t)r * nw + k / 64] |= (uint64_t)1 << (k % 64);
	std::vector<uint64_t> sub((size_t)4 * nw);   // columns of the four sub-tiles
	for (std::vector<int>& rows : greedy_groups(bits, R, nw, 64)) {
		rows.resize(64, -1);
		uint64_t* const u = sub.data();
		std::fill(sub.begin(), sub.end(), 0);
		for (int i = 0; i < 64; i++)
			if (rows[(size_t)i] >= 0) for (int q = 0; q < nw; q++) u[(size_t)(i / 16) * nw + q] |= bits[(size_t)rows[(size_t)i] * nw + q];
		WtTile t;
		t.rlist = (int)h.lists.size();
		for (int i = 0; i < 64; i++) h.lists.push_back(rows[(size_t)i]);
		// the sub-tiles that use each column
		std::vector<std::pair<int, int>> cols;
		for (int k = 0; k < K; k++) {
			int m = 0;
			for (int g = 0; g < 4; g++) if (u[(size_t)g * nw + k / 64] >> (k % 64) & 1) m |= 1 << g;
			if (m) cols.emplace_back(m, k);
		}
		std::stable_sort(cols.begin(), cols.end(), [](const std::pair<int, int>& x, const std::pair<int, int>& y) { return x.first < y.first; });
		t.np = std::max<int>(1, (int)((cols.size() + TK - 1) / TK));
		t.klist = (int)h.lists.size();
		for (int i = 0; i < t.np * TK; i++) h.lists.push_back(i < (int)cols.size() ? cols[(size_t)i].second : -1);
		t.mask = (int)h.masks.size();
		t.pack = (int64_t)h.pack.size();
		h.pack.resize(h.pack.size() + (size_t)t.np * TK * 64, 0.0);
		int mfmas = 0;
		for (int p = 0; p < t.np; p++) {
			uint32_t m = 0;
			for (int q = 0; q < TK; q++) {
				const int i = p * TK + q;
				if (i >= (int)cols.size()) break;
				m |= (uint32_t)cols[(size_t)i].first << (4 * (q / 4));
				// fragment order: step q / 4, sub-tile pair, lane (q % 4) 16 + row % 16, sub-tile % 2
				for (int x = 0; x < 64; x++)
					if (rows[(size_t)x] >= 0) h.pack[(size_t)t.pack + (size_t)p * 1024 + (size_t)((((q / 4) * 2 + x / 32) * 64 + (q % 4) * 16 + x % 16) * 2 + (x / 16) % 2)] =
						w[(size_t)rows[(size_t)x] * K + cols[(size_t)i].second];
			}
			h.masks.push_back(m);
			mfmas += __builtin_popcount(m);
		}
		t.cost = mfmas + 12 * t.np + 24;   // MFMAs of a wavefront, and what a panel and a tile cost beside them
		tiles.push_back(t);
	}
}

bool plan_wtiles(WtHost& h, const WApplyHost& wa, const Meta& W, const double* w)
{
	std::vector<std::vector<WtTile>> tiles(wa.classes.size());
	std::vector<int64_t> nonzero(wa.classes.size(), 0);
	std::vector<uint8_t> acts(wa.classes.size(), 0);   // on some block pair
	for (const int ci : wa.unit_class) acts[(size_t)ci] = 1;
	// the packs of all columns: address space, of which the packs in use are touched
	size_t most = 0;
	for (size_t ci = 0; ci < wa.classes.size(); ci++)
		if (acts[ci]) most += (size_t)((wa.classes[ci].R + 63) / 64) * (size_t)((wa.classes[ci].K + TK - 1) / TK) * 64 * TK;
	h.pack.reserve(most);
	for (size_t ci = 0; ci < wa.classes.size(); ci++) {
		const WaClass& c = wa.classes[ci];
		if (c.K > WT_KMAX) return false;
		if (!acts[ci] || c.K < 1 || c.R < 1) continue;
		std::vector<double> m((size_t)c.R * c.K, 0.0);
		int r0 = 0;
		for (const auto& mq : c.rows) {
			const ct_long dM = W.block_count[0][(size_t)mq.first], dQ = W.block_count[1][(size_t)mq.second];
			int k0 = 0;
			for (const auto& pn : c.cols) {
				const ct_long dP = W.block_count[2][(size_t)pn.first], dN = W.block_count[3][(size_t)pn.second];
				const ct_long iw[4] = { mq.first, mq.second, pn.first, pn.second };
				const ct_long kw = W.flat_index(iw);
				if (W.present(kw))
					for (ct_long i = 0; i < dM * dQ; i++)
						for (ct_long k = 0; k < dP * dN; k++) m[(size_t)((r0 + i) * c.K + k0 + k)] = w[W.offset[kw] + i * dP * dN + k];
				k0 += (int)(dP * dN);
			}
			r0 += (int)(dM * dQ);
		}
		for (const double v : m) nonzero[ci] += v != 0.0;
		plan_row_tiles(h, m, c.R, c.K, tiles[ci]);
	}
	// the tiles of one column tile share its T1 panel: they go to one XCD, the column tiles dealt to the
	// eight XCDs by cost
	struct Group { int64_t cost; size_t unit; int j0; };
	std::vector<Group> groups;
	std::vector<WtItem> proto(wa.units.size());
	for (size_t ui = 0; ui < wa.units.size(); ui++) {
		const WaUnit& u = wa.units[ui];
		const std::vector<WtTile>& ts = tiles[(size_t)wa.unit_class[ui]];
		WtItem& q = proto[ui];
		q = WtItem{};
		q.kb = u.kb;
		q.rb = u.rb;
		q.dA = u.dA;
		q.dC = u.dC;
		auto span = [](const std::vector<int64_t>& base, const std::vector<int>& stride, int64_t b0, int n, int dA, int dC, int64_t& off, int64_t& bytes) {
			int64_t lo = INT64_MAX, hi = 0;
			for (int k = 0; k < n; k++) {
				const int64_t b = base[(size_t)(b0 + k)];
				if (b < 0) continue;
				lo = std::min(lo, b);
				hi = std::max(hi, b + (int64_t)(dA - 1) * stride[(size_t)(b0 + k)] + dC);
			}
			off = hi > 0 ? lo : 0;
			bytes = hi > 0 ? 8 * (hi - lo) : 0;
		};
		int64_t b1 = 0, b2 = 0;
		span(wa.kbase, wa.kstride, u.kb, u.K, u.dA, u.dC, q.t1_off, b1);
		span(wa.rbase, wa.rstride, u.rb, u.R, u.dA, u.dC, q.t2_off, b2);
		if (std::max(b1, b2) >= (int64_t)1 << 30) return false;
		q.t1_bytes = (int)b1;
		q.t2_bytes = (int)b2;
		int64_t cost = 0;
		for (const WtTile& t : ts) cost += t.cost;
		h.flops += 2.0 * (double)nonzero[(size_t)wa.unit_class[ui]] * u.dA * u.dC;
		const int cols = u.dA * ((u.dC + 1) & ~1);
		for (int j0 = 0; j0 < cols; j0 += 64) groups.push_back(Group{ cost, ui, j0 });
	}
	std::stable_sort(groups.begin(), groups.end(), [](const Group& x, const Group& y) { return x.cost > y.cost; });
	std::vector<std::vector<WtItem>> q(PR_XCDS);
	std::vector<int64_t> load(PR_XCDS, 0);
	for (const Group& g : groups) {
		const size_t x = (size_t)(std::min_element(load.begin(), load.end()) - load.begin());
		load[x] += g.cost;
		for (const WtTile& t : tiles[(size_t)wa.unit_class[g.unit]]) {
			WtItem i = proto[g.unit];
			i.j0 = g.j0;
			i.np = t.np;
			i.pack = t.pack;
			i.klist = t.klist;
			i.rlist = t.rlist;
			i.mask = t.mask;
			q[x].push_back(i);
		}
	}
	size_t longest = 0;
	for (const auto& v : q) longest = std::max(longest, v.size());
	for (size_t jj = 0; jj < longest; jj++)
		for (int x = 0; x < PR_XCDS; x++)
			if (jj < q[(size_t)x].size()) h.items.push_back(q[(size_t)x][jj]);
	return true;
}

template <typename T>
static T* upload_new(const std::vector<T>& v, hipStream_t s)
{
	T* d = (T*)dev_alloc(std::max<size_t>(1, v.size()) * sizeof(T));
	copy_h2d_async(d, v.data(), v.size() * sizeof(T), s);
	return d;
}

void WTiles::upload(const WtHost& h, hipStream_t s)
{
	release();
	items = upload_new(h.items, s);
	lists = upload_new(h.lists, s);
	masks = upload_new(h.masks, s);
	pack = upload_new(h.pack, s);
	nitems = (int)h.items.size();
	flops = h.flops;
	ok = true;
}

void WTiles::release()
{
	dev_free(items); dev_free(lists); dev_free(masks); dev_free(pack);
	items = nullptr; lists = nullptr; masks = nullptr; pack = nullptr;
	nitems = 0;
	ok = use = false;
}

void launch_wtiles(const WTiles& wt, const WApply& wa, const double* t1, double* t2, hipStream_t s)
{
	if (wt.nitems == 0) return;
	hipLaunchKernelGGL(k_wtile, dim3((unsigned)wt.nitems), dim3(256), 0, s, (const WtItem*)wt.items, (const int64_t*)wa.kbase, (const int*)wa.kstride,
		(const int64_t*)wa.rbase, (const int*)wa.rstride, (const int*)wt.lists, (const uint32_t*)wt.masks, (const double*)wt.pack, t1, t2);
	CTG_HIP(hipGetLastError());
}

}  // namespace ctg
