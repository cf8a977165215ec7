// tg_prep.hip -- a solver's list work built on the device from the device walk's lists, which
// never leave the device: the arrays prepare_work (tg_upload.cpp) builds on the host from a host
// copy of the lists, element for element.
//
// Node kinds (CC, CP; direct and Ewald), one thread per node: the entries of each kind, cut into
// chunks of <= node_chunk entries (one partial slot each; a node's slots are contiguous, its kinds
// in the order CC_d, CP_d, CC_e, CP_e).  Exclusive scans over the nodes give every offset; then
// the chunks, the slot of every entry, the node of every slot and the CP ranges expanded to
// particle indices are written, and the chunks packed into waves of <= 64 entries (a longer chunk
// is a wave alone): greedily, restarting every WAVE_SEGMENT chunks, so the segments pack in
// parallel.  The CC lists are the
// walk's own (its node-order CSR is the list order).
// Leaf kinds (PC, PP), one wave per non-empty leaf, leaves in node order: the entries, and for PP
// direct the near prefix -- the sources of ranges whose bounding box comes within the softening
// length of the sink leaf's box, the test made in FP64 with the host's operations.  Scans over
// the leaves give the offsets; the PP ranges are expanded (PP direct: near ranges first, both
// groups in list order), the items of <= 64 sinks written, and every kind's items put in the
// order of a stable sort by descending cost class (a counting sort).  The PC lists are the walk's own.
// Every kernel covers its four kinds at once and all arrays of a stage are scanned together
// (tg_scan.hpp): a small set's preparation is a matter of launches, 25 of them, and two host waits
// for the sizes.
#include <algorithm>
#include <cstring>

#include "tg_gravity.h"
#include "tg_solver.hpp"
#include "tg_devmem.hpp"
#include "tg_math.hpp"
#include "tg_scan.hpp"

namespace tg {
namespace {

// walk kinds 0..3 are the node kinds, 4..7 the leaf kinds, in these solver kinds
constexpr int NODE_KIND[4] = {CC_DIRECT, CP_DIRECT, CC_EWALD, CP_EWALD};
constexpr int LEAF_KIND[4] = {PC_DIRECT, PP_DIRECT, PC_EWALD, PP_EWALD};

__device__ __forceinline__ double pos_d(int32_t x) {
#pragma clang fp contract(off)
	return double(x) * (1.0 / 4294967296.0) + 0.5;
}

__device__ __forceinline__ int64_t wave_sum(int64_t v) {
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
	return v;
}

__device__ __forceinline__ int wave_min(int v) {
	for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
	return v;
}

__device__ __forceinline__ int wave_max(int v) {
	for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
	return v;
}

// ---- node kinds ----------------------------------------------------------------------------------

struct NodeIn {
	const int64_t* ptr[4];  // walk kinds 0..3
	const int32_t* val[4];
	int64_t nn;
	int chunk;
};

// per node and kind: entries and chunks; per node: slots.  Arrays of nn + 1 (the last zero, so an
// exclusive scan over nn + 1 ends with the total)
__global__ __launch_bounds__(256) void k_node_count(NodeIn A, int64_t* __restrict__ nent, int64_t* __restrict__ nchk,
		int64_t* __restrict__ nslot) {
	const int64_t nd = int64_t(blockIdx.x) * 256 + threadIdx.x;
	const int64_t np = A.nn + 1;
	if (nd > A.nn) return;
	if (nd == A.nn) {
		for (int q = 0; q < 4; q++) nent[q * np + nd] = nchk[q * np + nd] = 0;
		nslot[nd] = 0;
		return;
	}
	int64_t slots = 0;
	for (int q = 0; q < 4; q++) {
		const int64_t kb = A.ptr[q][nd], ke = A.ptr[q][nd + 1];
		int64_t ent = 0;
		if (q & 1) {  // CP: [begin, end) ranges
			for (int64_t j = kb; j < ke; j += 2) {
				const int64_t len = int64_t(A.val[q][j + 1]) - int64_t(A.val[q][j]);
				if (len > 0) ent += len;
			}
		} else {
			ent = ke - kb;
		}
		const int64_t nch = (ent + A.chunk - 1) / A.chunk;
		nent[q * np + nd] = ent;
		nchk[q * np + nd] = nch;
		slots += nch;
	}
	nslot[nd] = slots;
}

struct NodeOut {
	int2* chunks[4];       // per kind: [begin, end) entries of each chunk
	int* chunk_slot[4];    // per kind: the partial slot of each chunk
	int* slot_node;
};

// the chunks of every node: records, slots and the slots' node
__global__ __launch_bounds__(256) void k_node_chunks(NodeIn A, const int64_t* __restrict__ nent, const int64_t* __restrict__ oent,
		const int64_t* __restrict__ ochk, const int64_t* __restrict__ slot_ptr, NodeOut O) {
	const int64_t nd = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (nd >= A.nn) return;
	const int64_t np = A.nn + 1;
	int64_t sl = slot_ptr[nd];
	for (int q = 0; q < 4; q++) {
		const int64_t lb = oent[q * np + nd], le = lb + nent[q * np + nd];
		int64_t c = ochk[q * np + nd];
		for (int64_t b = lb; b < le; b += A.chunk, c++, sl++) {
			const int64_t e = le < b + A.chunk ? le : b + A.chunk;
			O.chunks[q][c] = make_int2(int(b), int(e));
			O.chunk_slot[q][c] = int(sl);
			O.slot_node[sl] = int(nd);
		}
	}
}

struct ChunkSet {
	const int2* chunks[4];
	const int* slot[4];
	int* owner[4];
	int64_t nch[4];
};

// The partial slot of the entries: one wave per chunk, kinds in grid.y.  The solve reads the slot of
// a wave's first 64 entries only (a longer chunk is a wave of its own), so no more are written
// unless `all` asks (0.35 ms of 1.3 GB at 2M theta 0.3 leaf 8).
__global__ __launch_bounds__(256) void k_node_owner(ChunkSet S, int all) {
	const int q = blockIdx.y;
	const int64_t c = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
	if (c >= S.nch[q]) return;
	const int2 ch = S.chunks[q][c];
	const int sl = S.slot[q][c];
	const int end = all ? ch.y : min(ch.y, ch.x + 64);
	for (int j = ch.x + int(threadIdx.x & 63); j < end; j += 64) S.owner[q][j] = sl;
}

// Greedy packing of a segment's chunks into waves of <= 64 entries (a longer chunk is a wave alone):
// a wave that starts at chunk c ends before next(c), the first chunk whose end lies more than 64
// entries past c's begin.  The waves' first chunks are the orbit of the segment's first under
// next, marked by doubling: eight tables of 2^k-fold jumps, eight rounds of marks.  (One thread walking a
// segment's 256 chunks took 37 us whatever the set's size.)
struct PackShared {
	int begin[WAVE_SEGMENT], end[WAVE_SEGMENT];
	short jump[8][WAVE_SEGMENT + 1];
	uint8_t mark[WAVE_SEGMENT + 1];
	int wsum[WAVE_SEGMENT / 64];
};
static_assert(WAVE_SEGMENT == 256, "eight doublings cover a segment");

// calls emit(rank, begin, end) in the thread of every wave's first chunk; returns the wave count
template <class F>
__device__ __forceinline__ int pack_segment(const int2* __restrict__ chunks, int64_t c0, int cnt, PackShared& S, F emit) {
	const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
	if (t < cnt) {
		const int2 c = chunks[c0 + t];
		S.begin[t] = c.x;
		S.end[t] = c.y;
	}
	S.mark[t] = t == 0;
	__syncthreads();
	if (t < cnt) {
		int lo = t + 1, hi = cnt;
		while (lo < hi) {
			const int mid = (lo + hi) >> 1;
			if (S.end[mid] - S.begin[t] > 64)
				hi = mid;
			else
				lo = mid + 1;
		}
		S.jump[0][t] = short(lo);
	} else {
		S.jump[0][t] = short(cnt);
	}
	if (t == 0) {
		for (int k = 0; k < 8; k++) S.jump[k][cnt] = short(cnt);
		S.mark[cnt] = 0;
	}
	__syncthreads();
	for (int k = 1; k < 8; k++) {
		if (t < cnt) S.jump[k][t] = S.jump[k - 1][S.jump[k - 1][t]];
		__syncthreads();
	}
	for (int k = 7; k >= 0; k--) {
		const int to = t < cnt && S.mark[t] ? int(S.jump[k][t]) : cnt;
		if (to < cnt) S.mark[to] = 1;
		__syncthreads();
	}
	const bool first = t < cnt && S.mark[t];
	const unsigned long long m = __ballot(first);
	if (lane == 0) S.wsum[wave] = __popcll(m);
	__syncthreads();
	int before = 0, all = 0;
	for (int w = 0; w < WAVE_SEGMENT / 64; w++) {
		if (w < wave) before += S.wsum[w];
		all += S.wsum[w];
	}
	if (first) emit(before + __popcll(m & (lane ? ~0ull >> (64 - lane) : 0ull)), S.begin[t], S.end[S.jump[0][t] - 1]);
	return all;
}

// waves per segment of WAVE_SEGMENT chunks, kinds in grid.y
struct PackOut {
	int64_t nseg[4];
	int64_t* nw[4];
	const int64_t* ow[4];
	int2* waves[4];
};
__global__ __launch_bounds__(WAVE_SEGMENT) void k_wave_count(ChunkSet S, PackOut O) {
	__shared__ PackShared P;
	const int q = blockIdx.y;
	const int64_t sg = blockIdx.x;
	if (sg >= O.nseg[q]) return;
	const int64_t c0 = sg * WAVE_SEGMENT;
	const int n = pack_segment(S.chunks[q], c0, int(S.nch[q] - c0 < WAVE_SEGMENT ? S.nch[q] - c0 : WAVE_SEGMENT), P, [](int, int, int) {});
	if (threadIdx.x == 0) O.nw[q][sg] = n;
}

__global__ __launch_bounds__(WAVE_SEGMENT) void k_wave_write(ChunkSet S, PackOut O) {
	__shared__ PackShared P;
	const int q = blockIdx.y;
	const int64_t sg = blockIdx.x;
	if (sg >= O.nseg[q]) return;
	const int64_t c0 = sg * WAVE_SEGMENT;
	int2* out = O.waves[q] + O.ow[q][sg];
	pack_segment(S.chunks[q], c0, int(S.nch[q] - c0 < WAVE_SEGMENT ? S.nch[q] - c0 : WAVE_SEGMENT), P,
			[&](int r, int b, int e) { out[r] = make_int2(b, e); });
}

// ---- range expansion (CP, PP) --------------------------------------------------------------------

// One wave writes the entries of the non-empty ranges of v[kb, ke) (2 ints each) that keep()
// accepts, consecutively from out: 64 ranges per round, an exclusive scan of their lengths, the
// non-empty ones moved to the first lanes; then 64 entries at a time, each finding its range from a
// mask of the entries at which ranges start (a binary search of the scan per entry took 1.6 times
// as long).  Returns the entries written.  The block is this one wave (the barriers are the wave's).
template <class Keep>
__device__ int64_t expand_ranges(const int32_t* __restrict__ v, int64_t kb, int64_t ke, Keep keep, int32_t* __restrict__ out) {
	__shared__ int s_start[64], s_off[64];
	__shared__ uint8_t s_flag[64];
	const int lane = threadIdx.x;
	const unsigned long long below = lane ? ~0ull >> (64 - lane) : 0ull;
	int64_t pos = 0;
	for (int64_t j0 = kb; j0 < ke; j0 += 128) {
		const int64_t j = j0 + 2 * lane;
		int b = 0, len = 0;
		if (j < ke) {
			b = v[j];
			const int e = v[j + 1];
			len = e > b ? e - b : 0;
			if (len > 0 && !keep(b, e, j)) len = 0;
		}
		int s = len;
		for (int o = 1; o < 64; o <<= 1) {
			const int t = __shfl_up(s, o, 64);
			if (lane >= o) s += t;
		}
		const int tot = __shfl(s, 63, 64);
		const unsigned long long some = __ballot(len > 0);
		const int nr = __popcll(some);
		if (len > 0) {
			const int r = __popcll(some & below);
			s_start[r] = s - len;
			s_off[r] = b - (s - len);
		}
		__syncthreads();
		const int start = lane < nr ? s_start[lane] : INT32_MAX;
		const int off = lane < nr ? s_off[lane] : 0;
		int r0 = 0;  // ranges that started before the 64 entries
		for (int p0 = 0; p0 < tot; p0 += 64) {
			s_flag[lane] = 0;
			__syncthreads();
			const int at = start - p0;
			if (at >= 0 && at < 64) s_flag[at] = 1;
			__syncthreads();
			const unsigned long long m = __ballot(s_flag[lane] != 0);
			const int r = r0 + __popcll(m & (below | (1ull << lane))) - 1;
			const int o = __shfl(off, r & 63, 64);
			if (p0 + lane < tot) out[pos + p0 + lane] = o + p0 + lane;
			r0 += __popcll(m);
			__syncthreads();
		}
		pos += tot;
	}
	return pos;
}

// CP ranges of every node expanded: one wave per node
__global__ __launch_bounds__(64) void k_node_expand(NodeIn A, const int64_t* __restrict__ oent, int32_t* cp_d, int32_t* cp_e) {
	const int64_t nd = blockIdx.x;
	const int64_t np = A.nn + 1;
	for (int q = 1; q < 4; q += 2) {
		const int64_t kb = A.ptr[q][nd], ke = A.ptr[q][nd + 1];
		if (ke == kb) continue;
		int32_t* out = (q == 1 ? cp_d : cp_e) + oent[q * np + nd];
		expand_ranges(A.val[q], kb, ke, [](int, int, int64_t) { return true; }, out);
	}
}

// ---- leaf kinds ----------------------------------------------------------------------------------

struct LeafIn {
	const int64_t* ptr[4];  // walk kinds 4..7: pc_d, pp_d, pc_e, pp_e
	const int32_t* val[4];
	const int4* leaf_items;  // (node, first particle, end, -)
	const int4* parts;
	const int* pleaf;        // particle -> leaf
	const int4* box;         // per node, 2 records: lowest and highest particle coordinates, first particle, end (leaves)
	uint8_t* near;           // PP direct: per range (entry pair j / 2), the near test's outcome
	int64_t nl;
	int ewald;
	double hnear;
};

// the bounding box of every non-empty leaf's particles: one wave per leaf
__global__ __launch_bounds__(64) void k_leaf_boxes(const int4* __restrict__ leaf_items, const int4* __restrict__ parts, int4* __restrict__ box) {
	const int4 li = leaf_items[blockIdx.x];
	int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
	for (int p = li.y + int(threadIdx.x); p < li.z; p += 64) {
		const int4 x = parts[p];
		lo[0] = min(lo[0], x.x);
		lo[1] = min(lo[1], x.y);
		lo[2] = min(lo[2], x.z);
		hi[0] = max(hi[0], x.x);
		hi[1] = max(hi[1], x.y);
		hi[2] = max(hi[2], x.z);
	}
	for (int d = 0; d < 3; d++) {
		lo[d] = wave_min(lo[d]);
		hi[d] = wave_max(hi[d]);
	}
	if (threadIdx.x == 0) {
		box[2 * li.x] = make_int4(lo[0], lo[1], lo[2], li.y);
		box[2 * li.x + 1] = make_int4(hi[0], hi[1], hi[2], li.z);
	}
}

// may a source of the box [lo, hi] lie within the softening length of the sink box [slo, shi]?
// The host's test (prepare_work, tg_upload.cpp) with the same FP64 operations.
__device__ bool may_be_near(int4 slo, int4 shi, int4 lo, int4 hi, int ewald, double hnear) {
#pragma clang fp contract(off)
	const int a0[3] = {slo.x, slo.y, slo.z}, a1[3] = {shi.x, shi.y, shi.z};
	const int b0[3] = {lo.x, lo.y, lo.z}, b1[3] = {hi.x, hi.y, hi.z};
	double d2 = 0.0;
	for (int d = 0; d < 3; d++) {
		const double smn = pos_d(a0[d]), smx = pos_d(a1[d]), mn = pos_d(b0[d]), mx = pos_d(b1[d]);
		const double h1 = 0.5 * (smx - smn), h2 = 0.5 * (mx - mn);
		if (ewald && h1 + h2 > 0.25) return true;
		double dc = 0.5 * (smx + smn) - 0.5 * (mx + mn);
		if (ewald) dc -= rint(dc);
		const double gap = fabs(dc) - h1 - h2;
		if (gap > 0.0) d2 += gap * gap;
	}
	return d2 <= hnear * hnear;
}

// the same decided by one axis alone where that is clear: a gap beyond the softening length by more
// than FP32's error (3e-7 of the box) on any axis, and no periodic axis near the quarter-box rule
__device__ __forceinline__ bool surely_far(int4 slo, int4 shi, int4 lo, int4 hi, int ewald, float hnear) {
	const int a0[3] = {slo.x, slo.y, slo.z}, a1[3] = {shi.x, shi.y, shi.z};
	const int b0[3] = {lo.x, lo.y, lo.z}, b1[3] = {hi.x, hi.y, hi.z};
	float gap = -1.0f, wide = 0.0f;
	for (int d = 0; d < 3; d++) {
		const float hh = (float(unsigned(a1[d]) - unsigned(a0[d])) + float(unsigned(b1[d]) - unsigned(b0[d]))) * 1.1641532182693481e-10f;  // 2^-33
		float dc = float((int64_t(a0[d]) + a1[d]) - (int64_t(b0[d]) + b1[d])) * 1.1641532182693481e-10f;
		if (ewald) dc -= rintf(dc);
		gap = fmaxf(gap, fabsf(dc) - hh);
		wide = fmaxf(wide, hh);
	}
	return gap > hnear + 1e-6f && !(ewald && wide > 0.2499f);
}

// the near test of the source range [b, e) (non-empty) for a sink leaf of box [slo, shi]: a whole
// leaf (which the walk's ranges are) takes that leaf's box, any other range its particles' box
__device__ bool range_near(const LeafIn& A, int4 slo, int4 shi, int b, int e) {
	const int lf = A.pleaf[b];
	int4 lo = A.box[2 * lf], hi = A.box[2 * lf + 1];
	if (lo.w != b || hi.w != e) {
		lo = make_int4(INT32_MAX, INT32_MAX, INT32_MAX, 0);
		hi = make_int4(INT32_MIN, INT32_MIN, INT32_MIN, 0);
		for (int p = b; p < e; p++) {
			const int4 x = A.parts[p];
			lo = make_int4(min(lo.x, x.x), min(lo.y, x.y), min(lo.z, x.z), 0);
			hi = make_int4(max(hi.x, x.x), max(hi.y, x.y), max(hi.z, x.z), 0);
		}
	}
	if (surely_far(slo, shi, lo, hi, A.ewald, float(A.hnear))) return false;
	return may_be_near(slo, shi, lo, hi, A.ewald, A.hnear);
}

// per leaf and kind: entries (list ints for PC, expanded sources for PP), near-prefix length (PP
// direct) and items; per leaf the census terms (sinks x entries, sums[q]) and the raw list
// lengths (sums[4 + q], to check that the leaves hold every entry), summed afterwards by
// reductions (one atomic per leaf on a shared total would serialise at one cache line)
__global__ __launch_bounds__(64) void k_leaf_count(LeafIn A, int64_t* __restrict__ lent, int64_t* __restrict__ lnear, int64_t* __restrict__ litem,
		int64_t* __restrict__ sums) {
	const int64_t i = blockIdx.x;
	const int lane = threadIdx.x;
	const int64_t np = A.nl + 1;
	if (i == A.nl) {
		if (lane < 4) lent[lane * np + i] = litem[lane * np + i] = 0;
		if (lane < 8) sums[lane * np + i] = 0;
		if (lane == 0) lnear[i] = 0;
		return;
	}
	const int4 li = A.leaf_items[i];
	const int lf = li.x;
	const int64_t ns = li.z - li.y;
	const int4 slo = A.box[2 * lf], shi = A.box[2 * lf + 1];
	for (int q = 0; q < 4; q++) {
		const int64_t kb = A.ptr[q][lf], ke = A.ptr[q][lf + 1];
		int64_t ent = 0, nearl = 0;
		if (q & 1) {
			for (int64_t j = kb + 2 * lane; j < ke; j += 128) {
				const int b = A.val[q][j], e = A.val[q][j + 1];
				if (e <= b) continue;
				ent += e - b;
				if (q == 1) {
					const bool nr = range_near(A, slo, shi, b, e);
					A.near[j >> 1] = nr ? 1 : 0;  // for the write pass
					if (nr) nearl += e - b;
				}
			}
			ent = wave_sum(ent);
			nearl = wave_sum(nearl);
		} else {
			ent = ke - kb;
		}
		if (lane == 0) {
			lent[q * np + i] = ent;
			litem[q * np + i] = ent > 0 ? (ns + 63) / 64 : 0;
			if (q == 1) lnear[i] = nearl;
			sums[q * np + i] = ns * ent;
			sums[(4 + q) * np + i] = ke - kb;
		}
	}
}

struct LeafOut {
	int32_t* list[4];  // PP kinds: expanded lists (PC: unused)
	int4* items[4];    // unsorted items
	uint8_t* cls[4];   // their cost classes (item_class, below CLASSES)
};
constexpr int CLASSES = 64;

// the expanded PP lists and every kind's items, in leaf order: one wave per leaf
__global__ __launch_bounds__(64) void k_leaf_write(LeafIn A, const int64_t* __restrict__ lent, const int64_t* __restrict__ olent,
		const int64_t* __restrict__ lnear, const int64_t* __restrict__ olitem, LeafOut O) {
	const int64_t i = blockIdx.x;
	const int lane = threadIdx.x;
	const int64_t np = A.nl + 1;
	const int4 li = A.leaf_items[i];
	const int lf = li.x;
	const int4 slo = A.box[2 * lf], shi = A.box[2 * lf + 1];
	for (int q = 0; q < 4; q++) {
		const int64_t ent = lent[q * np + i];
		if (ent == 0) continue;
		const int64_t kb = A.ptr[q][lf], ke = A.ptr[q][lf + 1];
		int64_t lb, le, nearl = 0;
		if (q & 1) {
			lb = olent[q * np + i];
			le = lb + ent;
			int32_t* out = O.list[q] + lb;
			if (q == 1) {
				nearl = lnear[i];
				const uint8_t* nr = A.near;
				const int64_t w = expand_ranges(A.val[q], kb, ke, [&](int, int, int64_t j) { return nr[j >> 1] != 0; }, out);
				expand_ranges(A.val[q], kb, ke, [&](int, int, int64_t j) { return nr[j >> 1] == 0; }, out + w);
			} else {
				expand_ranges(A.val[q], kb, ke, [](int, int, int64_t) { return true; }, out);
			}
		} else {
			lb = kb;
			le = ke;
		}
		const int64_t it0 = olitem[q * np + i];
		const int nblk = (li.z - li.y + 63) / 64;
		for (int k = lane; k < nblk; k += 64) {
			const int b = li.y + 64 * k;
			const int cnt = li.z - b < 64 ? li.z - b : 64;
			const int y = (q & 1) ? pp_item_y(cnt, nearl) : cnt;
			const int64_t it = it0 + k;
			O.items[q][it] = make_int4(b, y, int(lb), int(le));
			O.cls[q][it] = uint8_t(item_class(le - lb, cnt));
		}
	}
}

// Counting sort of the items by descending class, stable: tiles of SORT_TILE items, per tile the items
// of each class (hist[(CLASSES - 1 - class) tiles + tile], kinds in grid.y); a scan of those gives the
// place of each tile's first item of each class, and an item's rank among the tile's earlier ones of
// its class the rest.
constexpr int SORT_TILE = 1024;
struct SortSet {
	const int4* in[4];
	const uint8_t* cls[4];
	int4* out[4];
	int64_t* hist[4];
	const int64_t* place[4];
	int64_t n[4];
};

__global__ __launch_bounds__(SORT_TILE) void k_item_hist(SortSet S) {
	__shared__ int h[CLASSES];
	const int q = blockIdx.y;
	const int64_t tiles = (S.n[q] + SORT_TILE - 1) / SORT_TILE;
	if (int64_t(blockIdx.x) >= tiles) return;
	if (threadIdx.x < CLASSES) h[threadIdx.x] = 0;
	__syncthreads();
	const int64_t i = int64_t(blockIdx.x) * SORT_TILE + threadIdx.x;
	if (i < S.n[q]) atomicAdd(&h[S.cls[q][i]], 1);
	__syncthreads();
	if (threadIdx.x < CLASSES) S.hist[q][(CLASSES - 1 - int(threadIdx.x)) * tiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(SORT_TILE) void k_item_scatter(SortSet S) {
	__shared__ int h[SORT_TILE / 64][CLASSES];
	const int q = blockIdx.y;
	const int64_t tiles = (S.n[q] + SORT_TILE - 1) / SORT_TILE;
	if (int64_t(blockIdx.x) >= tiles) return;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	for (int k = threadIdx.x; k < SORT_TILE / 64 * CLASSES; k += SORT_TILE) h[k / CLASSES][k % CLASSES] = 0;
	__syncthreads();
	const int64_t i = int64_t(blockIdx.x) * SORT_TILE + threadIdx.x;
	const bool in = i < S.n[q];
	const int c = in ? int(S.cls[q][i]) : 0;
	// the lanes of the wave with this lane's class
	unsigned long long same = __ballot(in);
	for (int bit = 0; bit < 6; bit++) {
		const unsigned long long set = __ballot((c >> bit) & 1);
		same &= (c >> bit) & 1 ? set : ~set;
	}
	const int rank = __popcll(same & (lane ? ~0ull >> (64 - lane) : 0ull));
	if (in && rank == 0) h[wave][c] = __popcll(same);
	__syncthreads();
	if (!in) return;
	int64_t pos = S.place[q][(CLASSES - 1 - c) * tiles + blockIdx.x] + rank;
	for (int w = 0; w < wave; w++) pos += h[w][c];
	S.out[q][pos] = S.in[q][i];
}

unsigned blocks(int64_t n, int per) { return unsigned((n + per - 1) / per); }

// ---- the tree's arrays from a device-built tree ---------------------------------------------------

// particle records (x, y, z, mass bits) and the input order
__global__ __launch_bounds__(256) void k_tw_parts(const int32_t* __restrict__ pos, const float* __restrict__ mass, const int64_t* __restrict__ order,
		int64_t n, int4* __restrict__ parts, int64_t* __restrict__ order_out) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	parts[i] = make_int4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], __float_as_int(mass[i]));
	order_out[i] = order[i];
}

// per node: source multipole, centre, level, parent; flags of the non-empty leaves and their
// root-path lengths, and of every leaf, empty ones included
__global__ __launch_bounds__(256) void k_tw_nodes(const DNode* __restrict__ nodes, const DMulti* __restrict__ multi, int64_t nn,
		MultiSrc* __restrict__ multis, FoldedMulti* __restrict__ folded, int4* __restrict__ npos, int* __restrict__ level, int* __restrict__ parent, int64_t* __restrict__ lflag,
		int64_t* __restrict__ plen, int64_t* __restrict__ leaves) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= nn) return;
	const DNode nd = nodes[i];
	const DMulti& m = multi[i];
	MultiSrc ms;
	for (int q = 0; q < 17; q++) ms.m[q] = m.m[q];
	for (int d = 0; d < 3; d++) ms.x[d] = m.x[d];
	multis[i] = ms;
	FoldedMulti f;
	float qzz;
	f.m = ms.m[0];
	fold_multi(ms.m, f.q, f.o, qzz);
	for (int d = 0; d < 3; d++) f.x[d] = ms.x[d];
	folded[i] = f;
	npos[i] = make_int4(m.x[0], m.x[1], m.x[2], 0);
	level[i] = nd.level;
	parent[i] = nd.parent;
	const bool leaf = nd.c0 < 0;
	const bool use = leaf && nd.pend > nd.pbegin;
	lflag[i] = use ? 1 : 0;
	plen[i] = use ? nd.level + 1 : 0;
	leaves[i] = leaf ? 1 : 0;
}

// the non-empty leaves in node order: (node, first particle, end, root-path offset) and the paths
__global__ __launch_bounds__(256) void k_tw_leaves(const DNode* __restrict__ nodes, int64_t nn, const int64_t* __restrict__ lflag,
		const int64_t* __restrict__ loff, const int64_t* __restrict__ poff, int4* __restrict__ leaf_items, int* __restrict__ path) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= nn || !lflag[i]) return;
	const DNode nd = nodes[i];
	leaf_items[loff[i]] = make_int4(int(i), nd.pbegin, nd.pend, int(poff[i]));
	int64_t p = poff[i] + nd.level + 1;
	for (int a = int(i); a >= 0; a = nodes[a].parent) path[--p] = a;
}

// each particle's leaf: one wave per leaf
__global__ __launch_bounds__(64) void k_tw_pleaf(const int4* __restrict__ leaf_items, int* __restrict__ pleaf) {
	const int4 li = leaf_items[blockIdx.x];
	for (int p = li.y + int(threadIdx.x); p < li.z; p += 64) pleaf[p] = li.x;
}

}  // namespace

#define PCHK(call)                                                   \
	do {                                                             \
		const hipError_t e_ = (call);                                \
		if (e_ != hipSuccess) {                                      \
			err = std::string("device list work: ") + #call + ": " + hipGetErrorString(e_); \
			return e_ == hipErrorOutOfMemory ? TG_ENOMEM : TG_EHIP;  \
		}                                                            \
	} while (0)

int Solver::upload_tree_device() {
	hipStream_t s = stream;
	const DeviceTree& D = dtree;
	const int64_t nn = D.nn;
	if (D.level_begin.size() < 2 || D.level_begin.back() != nn) {
		err = "device tree work: the level ranges do not cover the nodes";
		return TG_EINVAL;
	}
	if (max_level + 1 > 64) {  // the local-expansion pass's limit
		err = "tree deeper than the local-expansion pass supports (64 levels)";
		return TG_EINVAL;
	}
	PCHK(d_parts.alloc(std::max<size_t>(size_t(n) * sizeof(int4), 16)));
	PCHK(d_multis.alloc(std::max<size_t>(size_t(nn) * sizeof(MultiSrc), 16)));
	PCHK(d_folded.alloc(std::max<size_t>(size_t(nn) * sizeof(FoldedMulti), 16)));
	PCHK(d_nodepos.alloc(std::max<size_t>(size_t(nn) * sizeof(int4), 16)));
	PCHK(d_level.alloc(std::max<size_t>(size_t(nn) * 4, 16)));
	PCHK(d_parent.alloc(std::max<size_t>(size_t(nn) * 4, 16)));
	PCHK(d_pleaf.alloc(std::max<size_t>(size_t(n) * 4, 16)));
	PCHK(d_order.alloc(std::max<size_t>(size_t(n) * 8, 16)));
	PCHK(d_Lnode.alloc(std::max<size_t>(size_t(nn) * 35 * sizeof(double), 16)));
	// scratch, freed with the build's working buffers: six columns of nn words, the scan's workspace
	void* cols = nullptr;
	void* work = nullptr;
	PCHK(dev_malloc(&cols, size_t(6 * nn + 1) * 8));
	build_later.push_back(cols);
	int64_t* flag = static_cast<int64_t*>(cols);
	int64_t *loff = flag + nn, *plen = flag + 2 * nn, *poff = flag + 3 * nn, *lall = flag + 4 * nn, *aoff = flag + 5 * nn;
	if (n > 0) {
		hipLaunchKernelGGL(k_tw_parts, dim3(blocks(n, 256)), dim3(256), 0, s, D.pos, D.mass, D.order, n, d_parts.as<int4>(), d_order.as<int64_t>());
		PCHK(hipGetLastError());
	}
	order_on_device = true;
	int64_t tot[3] = {0, 0, 0};
	if (nn > 0) {
		hipLaunchKernelGGL(k_tw_nodes, dim3(blocks(nn, 256)), dim3(256), 0, s, D.nodes, D.multi, nn, d_multis.as<MultiSrc>(), d_folded.as<FoldedMulti>(), d_nodepos.as<int4>(),
				d_level.as<int>(), d_parent.as<int>(), flag, plen, lall);
		PCHK(hipGetLastError());
		ScanSet sc;
		sc.add(flag, loff, nn);
		sc.add(plen, poff, nn);
		sc.add(lall, aoff, nn);
		PCHK(dev_malloc(&work, size_t(scan_workspace(sc) + sc.cols) * 8));
		build_later.push_back(work);
		int64_t* wt = static_cast<int64_t*>(work);
		PCHK(scan_columns(sc, wt + sc.cols, wt, s));
		PCHK(hipMemcpyAsync(tot, wt, sizeof(tot), hipMemcpyDeviceToHost, s));
		PCHK(hipStreamSynchronize(s));
	}
	if (tot[1] > int64_t(INT32_MAX)) {
		err = "root-to-leaf paths exceed 2^31 entries";
		return TG_EINVAL;
	}
	n_leaf_items = int(tot[0]);
	n_leaves = tot[2];
	path_len = tot[1];
	PCHK(d_leaf_items.alloc(std::max<size_t>(size_t(tot[0]) * sizeof(int4), 16)));
	PCHK(d_path.alloc(std::max<size_t>(size_t(tot[1]) * 4, 16)));
	if (nn > 0) {
		hipLaunchKernelGGL(k_tw_leaves, dim3(blocks(nn, 256)), dim3(256), 0, s, D.nodes, nn, flag, loff, poff, d_leaf_items.as<int4>(),
				d_path.as<int>());
		PCHK(hipGetLastError());
	}
	if (tot[0] > 0) {
		hipLaunchKernelGGL(k_tw_pleaf, dim3(unsigned(tot[0])), dim3(64), 0, s, d_leaf_items.as<const int4>(), d_pleaf.as<int>());
		PCHK(hipGetLastError());
	}
	level_begin.assign(D.level_begin.begin(), D.level_begin.end());
	return TG_OK;
}

int Solver::upload_lists_device() {
	hipStream_t s = stream;
	const DeviceLists& L = dlists;
	const int64_t nn = n_nodes;
	const int64_t nl = n_leaf_items;
	const int chunk = std::min(NODE_CHUNK_MAX, std::max(1, chunk_of()));
	if (L.nn != nn || !L.ptr_all) {
		err = "device list work: the device walk's lists do not belong to this tree";
		return TG_EINVAL;
	}
	for (int k = 0; k < 8; k++)
		if (L.len[k] > int64_t(INT32_MAX)) {
			err = "an interaction list exceeds 2^31 entries (32-bit list offsets)";
			return TG_EINVAL;
		}
	auto scratch = [&](size_t bytes) -> void* {  // freed with the build's working buffers
		void* p = nullptr;
		if (dev_malloc(&p, std::max<size_t>(bytes, 16)) != hipSuccess) return nullptr;
		build_later.push_back(p);
		return p;
	};
	auto words = [&](int64_t count) { return static_cast<int64_t*>(scratch(size_t(count) * 8)); };
	list_bytes = 0;

	// ---- sizes: node kinds per node (entries, chunks, slots), leaf kinds per leaf (entries, items, census) ----
	NodeIn ni{};
	for (int q = 0; q < 4; q++) {
		ni.ptr[q] = L.ptr(q);
		ni.val[q] = L.val[q];
	}
	ni.nn = nn;
	ni.chunk = chunk;
	const int64_t np = nn + 1, lp = nl + 1;
	int64_t* nent = words(4 * np);
	int64_t* oent = words(4 * np);
	int64_t* nchk = words(4 * np);
	int64_t* ochk = words(4 * np);
	int64_t* nslot = words(np);
	int64_t* lent = words(4 * lp);
	int64_t* olent = words(4 * lp);
	int64_t* litem = words(4 * lp);
	int64_t* olitem = words(4 * lp);
	int64_t* lnear = words(lp);
	int64_t* sums = words(8 * lp);   // per leaf, 8 columns
	int64_t* osums = words(8 * lp);  // (their totals only)
	int4* box = static_cast<int4*>(scratch(size_t(std::max<int64_t>(nn, 1)) * 2 * sizeof(int4)));
	if (!nent || !oent || !nchk || !ochk || !nslot || !lent || !olent || !litem || !olitem || !lnear || !sums || !osums || !box)
		PCHK(hipErrorOutOfMemory);
	PCHK(d_node_slot_ptr.alloc(np * 8));
	int64_t* slot_ptr = d_node_slot_ptr.as<int64_t>();
	LeafIn li{};
	for (int q = 0; q < 4; q++) {
		li.ptr[q] = L.ptr(4 + q);
		li.val[q] = L.val[4 + q];
	}
	li.leaf_items = d_leaf_items.as<int4>();
	li.parts = d_parts.as<int4>();
	li.pleaf = d_pleaf.as<int>();
	li.nl = nl;
	li.ewald = ewald;
	li.hnear = soft_len * 1.001 + 1e-9;  // the host's margin over the kernel's single-precision test
	li.box = box;
	li.near = static_cast<uint8_t*>(scratch(size_t(std::max<int64_t>(L.len[5], 2)) / 2 + 1));
	if (!li.near) PCHK(hipErrorOutOfMemory);
	hipLaunchKernelGGL(k_node_count, dim3(blocks(np, 256)), dim3(256), 0, s, ni, nent, nchk, nslot);
	PCHK(hipGetLastError());
	if (nl > 0) {
		hipLaunchKernelGGL(k_leaf_boxes, dim3(unsigned(nl)), dim3(64), 0, s, li.leaf_items, li.parts, box);
		PCHK(hipGetLastError());
	}
	hipLaunchKernelGGL(k_leaf_count, dim3(unsigned(lp)), dim3(64), 0, s, li, lent, lnear, litem, sums);
	PCHK(hipGetLastError());
	int64_t nlen[4], nch[4], nslots, llen[4], nitems[4];
	uint64_t census[8];
	{
		// two sets of columns, one wait
		ScanSet a, b;
		for (int q = 0; q < 4; q++) a.add(nent + q * np, oent + q * np, np);
		for (int q = 0; q < 4; q++) a.add(nchk + q * np, ochk + q * np, np);
		a.add(nslot, slot_ptr, np);
		for (int q = 0; q < 4; q++) b.add(lent + q * lp, olent + q * lp, lp);
		for (int q = 0; q < 4; q++) b.add(litem + q * lp, olitem + q * lp, lp);
		for (int k = 0; k < 8; k++) b.add(sums + k * lp, osums + k * lp, lp);
		int64_t* wa = words(scan_workspace(a));
		int64_t* wb = words(scan_workspace(b));
		int64_t* tot = words(32);
		if (!wa || !wb || !tot) PCHK(hipErrorOutOfMemory);
		PCHK(scan_columns(a, wa, tot, s));
		PCHK(scan_columns(b, wb, tot + a.cols, s));
		int64_t v[25];
		PCHK(hipMemcpyAsync(v, tot, sizeof(v), hipMemcpyDeviceToHost, s));
		PCHK(hipStreamSynchronize(s));
		for (int q = 0; q < 4; q++) {
			nlen[q] = v[q];
			nch[q] = v[4 + q];
			llen[q] = v[9 + q];
			nitems[q] = v[13 + q];
		}
		nslots = v[8];
		for (int k = 0; k < 8; k++) census[k] = uint64_t(v[17 + k]);
	}
	for (int q = 0; q < 4; q++) {
		if (int64_t(census[4 + q]) != L.len[4 + q]) {
			err = "device list work: leaf-kind entries outside the non-empty leaves";
			return TG_EINVAL;
		}
		if (nlen[q] > int64_t(INT32_MAX) || llen[q] > int64_t(INT32_MAX) || nitems[q] > int64_t(INT32_MAX)) {
			err = "an interaction list exceeds 2^31 entries (32-bit list offsets)";
			return TG_EINVAL;
		}
	}
	if (nslots > int64_t(INT32_MAX)) {
		err = "partial slots exceed 2^31";
		return TG_EINVAL;
	}

	// ---- node kinds ----
	n_slots = nslots;
	PCHK(d_slot_node.alloc(std::max<size_t>(size_t(nslots) * 4, 16)));
	NodeOut no{};
	no.slot_node = d_slot_node.as<int>();
	ChunkSet cs{};
	int64_t nch_max = 0;
	for (int q = 0; q < 4; q++) {
		KindWork& w = work[NODE_KIND[q]];
		// kept with the work: the slots of all entries are written from them on demand (complete_owners)
		PCHK(w.chunks.alloc(std::max<size_t>(size_t(nch[q]) * sizeof(int2), 16)));
		PCHK(w.chunk_slot.alloc(std::max<size_t>(size_t(nch[q]) * 4, 16)));
		w.nchunks = nch[q];
		no.chunks[q] = w.chunks.as<int2>();
		no.chunk_slot[q] = w.chunk_slot.as<int>();
		// lists: CC the walk's own, CP expanded
		w.list.release();
		if (q & 1) {
			PCHK(w.list.alloc(std::max<size_t>(size_t(nlen[q]) * 4, 16)));
		} else {
			w.list.p = L.val[q];
			w.list.bytes = size_t(L.len[q]) * 4;
			w.list.owned = false;
		}
		w.nlist = nlen[q];
		PCHK(w.owner.alloc(std::max<size_t>(size_t(nlen[q]) * 4, 16)));
		PCHK(w.items.alloc(std::max<size_t>(size_t(nch[q]) * sizeof(int2), 16)));  // a wave holds a chunk or more
		cs.chunks[q] = no.chunks[q];
		cs.slot[q] = no.chunk_slot[q];
		cs.owner[q] = w.owner.as<int>();
		cs.nch[q] = nch[q];
		nch_max = std::max(nch_max, nch[q]);
	}
	owners_complete = false;
	if (nn > 0) {
		hipLaunchKernelGGL(k_node_chunks, dim3(blocks(nn, 256)), dim3(256), 0, s, ni, nent, oent, ochk, slot_ptr, no);
		PCHK(hipGetLastError());
		if (L.len[1] > 0 || L.len[3] > 0) {
			hipLaunchKernelGGL(k_node_expand, dim3(unsigned(nn)), dim3(64), 0, s, ni, oent, work[CP_DIRECT].list.as<int32_t>(),
					work[CP_EWALD].list.as<int32_t>());
			PCHK(hipGetLastError());
		}
	}
	int64_t* d_nwaves = words(4);
	if (!d_nwaves) PCHK(hipErrorOutOfMemory);
	if (nch_max > 0) {
		hipLaunchKernelGGL(k_node_owner, dim3(blocks(nch_max, 4), 4), dim3(256), 0, s, cs, 0);
		PCHK(hipGetLastError());
	}
	{
		PackOut po{};
		ScanSet sc;
		int64_t nseg_max = 0;
		for (int q = 0; q < 4; q++) {
			po.nseg[q] = (nch[q] + WAVE_SEGMENT - 1) / WAVE_SEGMENT;
			po.nw[q] = words(po.nseg[q] + 1);
			int64_t* ow = words(po.nseg[q] + 1);
			if (!po.nw[q] || !ow) PCHK(hipErrorOutOfMemory);
			po.ow[q] = ow;
			po.waves[q] = work[NODE_KIND[q]].items.as<int2>();
			sc.add(po.nw[q], ow, po.nseg[q]);
			nseg_max = std::max(nseg_max, po.nseg[q]);
		}
		int64_t* ws = words(scan_workspace(sc));
		if (!ws) PCHK(hipErrorOutOfMemory);
		if (nseg_max > 0) {
			hipLaunchKernelGGL(k_wave_count, dim3(unsigned(nseg_max), 4), dim3(WAVE_SEGMENT), 0, s, cs, po);
			PCHK(hipGetLastError());
		}
		PCHK(scan_columns(sc, ws, d_nwaves, s));
		if (nseg_max > 0) {
			hipLaunchKernelGGL(k_wave_write, dim3(unsigned(nseg_max), 4), dim3(WAVE_SEGMENT), 0, s, cs, po);
			PCHK(hipGetLastError());
		}
	}

	// ---- leaf kinds ----
	LeafOut lo{};
	SortSet so{};
	int64_t tiles_max = 0;
	ScanSet sc;
	for (int q = 0; q < 4; q++) {
		KindWork& w = work[LEAF_KIND[q]];
		w.list.release();
		if (q & 1) {
			PCHK(w.list.alloc(std::max<size_t>(size_t(llen[q]) * 4, 16)));
			lo.list[q] = w.list.as<int32_t>();
		} else {
			w.list.p = L.val[4 + q];
			w.list.bytes = size_t(L.len[4 + q]) * 4;
			w.list.owned = false;
		}
		w.owner.release();
		w.nlist = llen[q];
		w.nitems = int(nitems[q]);
		PCHK(w.items.alloc(std::max<size_t>(size_t(nitems[q]) * sizeof(int4), 16)));
		list_bytes += nitems[q] * int64_t(sizeof(int4));
		lo.items[q] = static_cast<int4*>(scratch(size_t(nitems[q]) * sizeof(int4)));
		lo.cls[q] = static_cast<uint8_t*>(scratch(size_t(nitems[q])));
		const int64_t tiles = (nitems[q] + SORT_TILE - 1) / SORT_TILE;
		tiles_max = std::max(tiles_max, tiles);
		so.hist[q] = words(CLASSES * tiles);
		int64_t* place = words(CLASSES * tiles);
		if (!lo.items[q] || !lo.cls[q] || !so.hist[q] || !place) PCHK(hipErrorOutOfMemory);
		so.place[q] = place;
		so.in[q] = lo.items[q];
		so.cls[q] = lo.cls[q];
		so.out[q] = w.items.as<int4>();
		so.n[q] = nitems[q];
		sc.add(so.hist[q], place, CLASSES * tiles);
	}
	if (nl > 0) {
		hipLaunchKernelGGL(k_leaf_write, dim3(unsigned(nl)), dim3(64), 0, s, li, lent, olent, lnear, olitem, lo);
		PCHK(hipGetLastError());
	}
	if (tiles_max > 0) {
		// heaviest cost class first, leaf order within a class
		hipLaunchKernelGGL(k_item_hist, dim3(unsigned(tiles_max), 4), dim3(SORT_TILE), 0, s, so);
		PCHK(hipGetLastError());
		int64_t* ws = words(scan_workspace(sc) + 4);
		if (!ws) PCHK(hipErrorOutOfMemory);
		PCHK(scan_columns(sc, ws + 4, ws, s));
		hipLaunchKernelGGL(k_item_scatter, dim3(unsigned(tiles_max), 4), dim3(SORT_TILE), 0, s, so);
		PCHK(hipGetLastError());
	}
	int64_t nwaves[4];
	PCHK(hipMemcpyAsync(nwaves, d_nwaves, sizeof(nwaves), hipMemcpyDeviceToHost, s));
	PCHK(hipStreamSynchronize(s));
	for (int q = 0; q < 4; q++) {
		work[NODE_KIND[q]].nitems = int(nwaves[q]);
		list_bytes += nwaves[q] * int64_t(sizeof(int2)) + nlen[q] * 4;
	}
	// the census as the reference counts it (node kinds: sources; leaf kinds: sinks x sources)
	Census& C = tree.census;
	C.CC_direct = uint64_t(nlen[0]);
	C.CP_direct = uint64_t(nlen[1]);
	C.CC_ewald = uint64_t(nlen[2]);
	C.CP_ewald = uint64_t(nlen[3]);
	C.PC_direct = census[0];
	C.PP_direct = census[1];
	C.PC_ewald = census[2];
	C.PP_ewald = census[3];
	return TG_OK;
}

int Solver::complete_owners() {
	if (owners_complete) return TG_OK;
	PCHK(hipSetDevice(device));
	ChunkSet cs{};
	int64_t nch_max = 0;
	for (int q = 0; q < 4; q++) {
		KindWork& w = work[NODE_KIND[q]];
		cs.chunks[q] = w.chunks.as<int2>();
		cs.slot[q] = w.chunk_slot.as<int>();
		cs.owner[q] = w.owner.as<int>();
		cs.nch[q] = w.nchunks;
		nch_max = std::max(nch_max, w.nchunks);
	}
	if (nch_max > 0) {
		hipLaunchKernelGGL(k_node_owner, dim3(blocks(nch_max, 4), 4), dim3(256), 0, stream, cs, 1);
		PCHK(hipGetLastError());
		PCHK(hipStreamSynchronize(stream));
	}
	owners_complete = true;
	return TG_OK;
}

}  // namespace tg
