// tg_devtree.hip -- the kd-tree (tree::refine, src/tree.cpp:122-201) and its multipoles
// (tree::compute_multipoles, src/tree.cpp:203-296) on the device, bit for bit as the host
// restatement in tg_tree.cpp builds them.
//
// Split passes, one per tree level (the reference refines one level per pass, src/main.cpp:170-174):
//   * every node of the level with more than parts_per_node particles (below the depth limit) is
//     split at the midpoint of its box's longest side; its children are numbered after the level,
//     in node order (a scan over the level's split flags);
//   * the reference's in-place partition (src/part_vect.cpp:905-926: scan up from the low end, on
//     a high particle search down from the high end for a low one and swap) exchanges the k-th high
//     particle left of the split point with the k-th low particle right of it counting from the
//     high end, and moves nothing else.  So each particle's partner follows from two prefix counts
//     of the "low" flags over the particle array: every exchange is made at once, each pair by the
//     thread of its left particle.
// A set of at most SMALL_N particles is split by one work group, all levels in one launch, the
// permutation and the prefix counts in LDS; larger sets take four or five launches a level.
// Multipole passes, leaves first, then levels from the deepest up (runs of small levels by one work
// group in one launch): leaves by 16 threads each (the 16 float lanes of
// part_vect_multipole_info, src/part_vect.cpp:567-635, lane k taking particles i + k of each block
// of 16, the lanes summed in order at the end), interior nodes by one thread each.  Every
// floating-point expression keeps the host's operand order and roundings (no contraction).
#include "tg_devtree.hpp"
#include "tg_devmem.hpp"
#include "tg_math.hpp"
#include "tg_walk.hpp"

#include <hipcub/hipcub.hpp>

#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

namespace tg {

namespace {

struct SplitInfo {
	double mid;
	int32_t dim, first_child;  // first_child: -1 where the node does not split
};

__device__ __forceinline__ double d_pos_to_double(int32_t x) {
#pragma clang fp contract(off)
	return double(x) * (1.0 / 4294967296.0) + 0.5;
}

__device__ __forceinline__ int32_t d_double_to_pos(double x) {
#pragma clang fp contract(off)
	const double POS_MAX = 4294967296.0;
	const double y = x - 0.5;
	long long z = llround(y * POS_MAX);
	if (double(z) >= POS_MAX / 2.0) z -= (long long) POS_MAX;
	return int32_t(z);
}

__device__ __forceinline__ void d_box_range(uint64_t id, double* mn, double* mx) {
#pragma clang fp contract(off)
	double x[3] = {0.0, 0.0, 0.0};
	double dx[3] = {1.0, 1.0, 1.0};
	while (id != 1) {
		const double t1 = x[0], t2 = dx[0];
		x[0] = x[2];
		x[2] = x[1];
		x[1] = t1;
		dx[0] = dx[2];
		dx[2] = dx[1];
		dx[1] = t2;
		if (id & 1)
			x[0] = 0.5 * x[0] + 0.5;
		else
			x[0] = 0.5 * x[0];
		dx[0] *= 0.5;
		id >>= 1;
	}
	for (int d = 0; d < 3; d++) {
		mn[d] = x[d];
		mx[d] = x[d] + dx[d];
	}
}

__device__ __forceinline__ double d_vabs(const double* v) {
#pragma clang fp contract(off)
	return sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
}

// one particle of the build: position and input index, moved together
__global__ __launch_bounds__(256) void k_records(const int32_t* __restrict__ x, int64_t n, int4* __restrict__ rec, int32_t* __restrict__ pnode) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	rec[i] = make_int4(x[3 * i], x[3 * i + 1], x[3 * i + 2], int32_t(i));
	pnode[i] = 0;
}

// the tree-order arrays from the records, or from the input and a permutation
__global__ __launch_bounds__(256) void k_unpack(const int4* __restrict__ rec, const int32_t* __restrict__ x, const int32_t* __restrict__ perm,
		const float* __restrict__ masses, float m, int64_t n, int32_t* __restrict__ pos, float* __restrict__ mass, int64_t* __restrict__ order) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	int4 r;
	if (rec) {
		r = rec[i];
	} else {
		const int64_t j = perm[i];
		r = make_int4(x[3 * j], x[3 * j + 1], x[3 * j + 2], int32_t(j));
	}
	pos[3 * i] = r.x;
	pos[3 * i + 1] = r.y;
	pos[3 * i + 2] = r.z;
	mass[i] = masses ? masses[r.w] : m;
	order[i] = r.w;
}

// The level being split is [lev[0], lev[1]) in device memory: the host launches a level's kernels
// with grids sized by a bound on its node count and reads the counts back only every few levels.

__device__ __forceinline__ bool splits(const DNode& nd, int ppn, int max_level) { return nd.pend - nd.pbegin > ppn && nd.level < max_level; }

// the split dimension and midpoint of a splitting node (src/tree.cpp:136-157)
__device__ __forceinline__ SplitInfo split_of(const DNode& nd, int first_child) {
#pragma clang fp contract(off)
	SplitInfo si{};
	si.first_child = first_child;
	double bmin[3], bmax[3];
	d_box_range(nd.boxid, bmin, bmax);
	double max_span = 0.0;
	int max_dim = 0;
	for (int dim = 0; dim < 3; dim++) {
		const double span = bmax[dim] - bmin[dim];
		if (span > max_span) {
			max_span = span;
			max_dim = dim;
		}
	}
	si.mid = (bmax[max_dim] + bmin[max_dim]) * 0.5;
	si.dim = max_dim;
	return si;
}

// exclusive prefix of one value per thread over a block of 1,024; total in every thread
__device__ __forceinline__ int block_scan(int v, int& total) {
	__shared__ int wsum[16];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	int x = v;
	for (int o = 1; o < 64; o <<= 1) {
		const int w = __shfl_up(x, o, 64);
		if (lane >= o) x += w;
	}
	__syncthreads();  // the last call's sums are read
	if (lane == 63) wsum[wave] = x;
	__syncthreads();
	int before = 0, all = 0;
	for (int w = 0; w < 16; w++) {
		if (w < wave) before += wsum[w];
		all += wsum[w];
	}
	total = all;
	return before + x - v;
}

// a level's split records in one launch of one block (levels of up to a few thousand nodes): the
// splitting nodes numbered in node order, the records, the next level and the log
__global__ __launch_bounds__(1024) void k_level(const DNode* __restrict__ nodes, int32_t* __restrict__ lev, int ppn, int max_level,
		SplitInfo* __restrict__ info, int32_t* __restrict__ log) {
	const int lb = lev[0], le = lev[1], nl = le - lb;
	int carry = 0;
	for (int j0 = 0; j0 < nl; j0 += 1024) {
		const int j = j0 + int(threadIdx.x);
		DNode nd{};
		if (j < nl) nd = nodes[lb + j];
		const bool f = j < nl && splits(nd, ppn, max_level);
		int all;
		const int rank = carry + block_scan(f, all);
		if (j < nl) {
			SplitInfo si{};
			si.first_child = -1;
			if (f) si = split_of(nd, le + 2 * rank);
			info[j] = si;
		}
		carry += all;
	}
	if (threadIdx.x == 0) {
		// the other kernels of the level read lev as it was from the log
		log[0] = lb;
		log[1] = le;
		log[2] = carry;
		lev[0] = le;
		lev[1] = le + 2 * carry;
	}
}

// 1 for every node of the level that splits, 0 from nl up to bound (the scan's total at nl)
__global__ void k_split_flags(const DNode* __restrict__ nodes, const int32_t* __restrict__ lev, int ppn, int max_level,
		int32_t* __restrict__ flags, int bound) {
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j > bound) return;
	const int lb = lev[0], nl = lev[1] - lev[0];
	flags[j] = j < nl && splits(nodes[lb + j], ppn, max_level) ? 1 : 0;
}

// the next level: [le, le + 2 nsplit); log = (lb, le, nsplit) of the level just split
__global__ void k_next_level(int32_t* __restrict__ lev, const int32_t* __restrict__ rank, int32_t* __restrict__ log) {
	if (threadIdx.x != 0 || blockIdx.x != 0) return;
	const int32_t lb = lev[0], le = lev[1];
	const int32_t ns = rank[le - lb];
	log[0] = lb;
	log[1] = le;
	log[2] = ns;
	lev[0] = le;
	lev[1] = le + 2 * ns;
}

// the split record of every node, its children's index
__global__ void k_split_setup(const DNode* __restrict__ nodes, const int32_t* __restrict__ lev, const int32_t* __restrict__ flags,
		const int32_t* __restrict__ rank, SplitInfo* __restrict__ info) {
	const int lb = lev[0], le = lev[1], nl = le - lb;
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= nl) return;
	SplitInfo si{};
	si.first_child = -1;
	if (flags[j]) si = split_of(nodes[lb + j], le + 2 * rank[j]);
	info[j] = si;
}

// The prefix counts of the low particles (those of a splitting node of the level below that node's
// midpoint): within tiles of LOW_TILE particles (loc), the tiles' sums scanned by k_low_tops; the
// flags as bytes.  One particle past the end carries the total.
constexpr int LOW_TILE = 4096;
struct LowCount {
	const int32_t* loc;
	const int32_t* base;  // per tile
	__device__ __forceinline__ int operator()(int64_t p) const { return loc[p] + base[p / LOW_TILE]; }
};

__global__ __launch_bounds__(1024) void k_low_tiles(const int4* __restrict__ rec, const int32_t* __restrict__ pnode, int64_t n,
		const int32_t* __restrict__ log, const SplitInfo* __restrict__ info, uint8_t* __restrict__ low, int32_t* __restrict__ loc,
		int32_t* __restrict__ base, int tiles) {
	const int lb = log[0], nl = log[1] - log[0];
	const int64_t p0 = int64_t(blockIdx.x) * LOW_TILE + int64_t(threadIdx.x) * 4;
	int f[4], sum = 0;
	for (int k = 0; k < 4; k++) {
		const int64_t p = p0 + k;
		f[k] = 0;
		if (p < n) {
			const int j = pnode[p] - lb;
			if (j >= 0 && j < nl) {
				const SplitInfo si = info[j];
				if (si.first_child >= 0) f[k] = d_pos_to_double(reinterpret_cast<const int32_t*>(rec + p)[si.dim]) < si.mid ? 1 : 0;
			}
		}
		sum += f[k];
	}
	int all;
	int x = block_scan(sum, all);
	for (int k = 0; k < 4; k++) {
		if (p0 + k <= n) loc[p0 + k] = x;
		if (p0 + k < n) low[p0 + k] = uint8_t(f[k]);
		x += f[k];
	}
	if (threadIdx.x == 0) base[blockIdx.x] = tiles > 1 ? all : 0;
}

__global__ __launch_bounds__(1024) void k_low_tops(int32_t* __restrict__ base, int tiles) {
	int carry = 0;
	for (int t0 = 0; t0 < tiles; t0 += 1024) {
		const int t = t0 + int(threadIdx.x);
		const int v = t < tiles ? base[t] : 0;
		int all;
		const int x = block_scan(v, all);
		if (t < tiles) base[t] = carry + x;
		carry += all;
	}
}

// the low particles right of the split point, by rank counted from the node's high end
__global__ __launch_bounds__(256) void k_high_side_lows(const int32_t* __restrict__ pnode, int64_t n, const DNode* __restrict__ nodes,
		const uint8_t* __restrict__ low, LowCount S, int32_t* __restrict__ mr) {
	const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (p >= n || !low[p]) return;
	const DNode nd = nodes[pnode[p]];  // a low particle's node splits
	const int sb = S(nd.pbegin), se = S(nd.pend);
	if (p < nd.pbegin + (se - sb)) return;
	mr[nd.pbegin + (se - S(p) - 1)] = int32_t(p);
}

// every high particle left of the split point exchanges its record with its partner; every
// particle of a splitting node moves to its child; the first of them makes the children
// [pbegin, split) and [split, pend), the split point being where the low particles end
__global__ __launch_bounds__(256) void k_exchange(int4* __restrict__ rec, int32_t* __restrict__ pnode, int64_t n, const int32_t* __restrict__ log,
		const SplitInfo* __restrict__ info, DNode* __restrict__ nodes, const uint8_t* __restrict__ low, LowCount S,
		const int32_t* __restrict__ mr) {
	const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (p >= n) return;
	const int lb = log[0], nl = log[1] - log[0];
	const int a = pnode[p], j = a - lb;
	if (j < 0 || j >= nl) return;
	const int first_child = info[j].first_child;
	if (first_child < 0) return;
	const int b = nodes[a].pbegin, e = nodes[a].pend;
	const int sb = S(b);
	const int split = b + (S(e) - sb);
	if (p < split && !low[p]) {
		const int64_t q = mr[b + ((int32_t(p) - b) - (S(p) - sb))];
		const int4 t = rec[p];
		rec[p] = rec[q];
		rec[q] = t;
	}
	pnode[p] = p < split ? first_child : first_child + 1;
	if (p == b) {
		const DNode nd = nodes[a];
		nodes[first_child] = DNode{b, split, -1, -1, a, nd.level + 1, nd.boxid << 1};
		nodes[first_child + 1] = DNode{split, e, -1, -1, a, nd.level + 1, (nd.boxid << 1) + 1};
		nodes[a].c0 = first_child;
		nodes[a].c1 = first_child + 1;
	}
}

// All levels of a small set by one work group: the same passes with the permutation, each
// particle's node (its index in the level), the prefix counts and the exchange partners in LDS.
// Launches are all a set this small costs: 1,001 particles took 108 of them.  Tree and moments at the
// upper end, against 4,097 particles level by level: uniform, leaves of 16, 0.13 ms against 0.41; leaves of
// one 0.27 against 0.88; Plummer, leaves of one, 0.34 against 0.91.  log: (lb, le, nsplit) per
// level, the last with nsplit 0.
constexpr int SMALL_N = 4096;
__global__ __launch_bounds__(1024) void k_small_tree(const int32_t* __restrict__ x, int n, DNode* nodes, int ppn, int max_level, SplitInfo* info,
		int32_t* __restrict__ log, int32_t* __restrict__ perm_out) {
	__shared__ unsigned short perm[SMALL_N], S[SMALL_N + 1], mr[SMALL_N], pn[SMALL_N];
	constexpr unsigned short DONE = 0xffff;
	const int t = threadIdx.x;
	for (int k = 0; k < 4; k++) {
		perm[4 * t + k] = (unsigned short) (4 * t + k);
		pn[4 * t + k] = 4 * t + k < n ? 0 : DONE;
	}
	if (t == 0) nodes[0] = DNode{0, n, -1, -1, -1, 0, 1};
	int lb = 0, le = 1;
	__syncthreads();
	for (int level = 0;; level++) {
		const int nl = le - lb;
		int ns = 0;
		for (int j0 = 0; j0 < nl; j0 += 1024) {
			const int j = j0 + t;
			DNode nd{};
			if (j < nl) nd = nodes[lb + j];
			const bool f = j < nl && splits(nd, ppn, max_level);
			int all;
			const int rank = ns + block_scan(f, all);
			if (j < nl) {
				SplitInfo si{};
				si.first_child = -1;
				if (f) si = split_of(nd, le + 2 * rank);
				info[j] = si;
			}
			ns += all;
		}
		if (t == 0) {
			log[3 * level] = lb;
			log[3 * level + 1] = le;
			log[3 * level + 2] = ns;
		}
		if (ns == 0) break;
		__syncthreads();
		int f[4], child[4], sum = 0;
		for (int k = 0; k < 4; k++) {
			const int p = 4 * t + k;
			f[k] = 0;
			child[k] = -1;
			if (pn[p] != DONE) {
				const SplitInfo si = info[pn[p]];
				child[k] = si.first_child;
				if (child[k] >= 0) f[k] = d_pos_to_double(x[3 * int(perm[p]) + si.dim]) < si.mid ? 1 : 0;
			}
			sum += f[k];
		}
		int all;
		int pre = block_scan(sum, all);
		for (int k = 0; k < 4; k++) {
			S[4 * t + k] = (unsigned short) pre;
			pre += f[k];
		}
		if (t == 1023) S[SMALL_N] = (unsigned short) pre;
		__syncthreads();
		int b[4], e[4], split[4];
		for (int k = 0; k < 4; k++) {
			const int p = 4 * t + k;
			if (child[k] < 0) continue;
			const DNode& nd = nodes[lb + pn[p]];
			b[k] = nd.pbegin;
			e[k] = nd.pend;
			split[k] = b[k] + (int(S[e[k]]) - int(S[b[k]]));
			if (f[k] && p >= split[k]) mr[b[k] + (int(S[e[k]]) - int(S[p]) - 1)] = (unsigned short) p;
		}
		__syncthreads();
		for (int k = 0; k < 4; k++) {
			const int p = 4 * t + k;
			if (child[k] < 0) {
				pn[p] = DONE;
				continue;
			}
			if (!f[k] && p < split[k]) {
				const int q = mr[b[k] + ((p - b[k]) - (int(S[p]) - int(S[b[k]])))];
				const unsigned short v = perm[p];
				perm[p] = perm[q];
				perm[q] = v;
			}
			if (p == b[k]) {
				const int a = lb + pn[p];
				const DNode nd = nodes[a];
				nodes[child[k]] = DNode{b[k], split[k], -1, -1, a, nd.level + 1, nd.boxid << 1};
				nodes[child[k] + 1] = DNode{split[k], e[k], -1, -1, a, nd.level + 1, (nd.boxid << 1) + 1};
				nodes[a].c0 = child[k];
				nodes[a].c1 = child[k] + 1;
			}
			pn[p] = (unsigned short) (child[k] - le + (p < split[k] ? 0 : 1));
		}
		__syncthreads();
		lb = le;
		le += 2 * ns;
	}
	__syncthreads();
	for (int k = 0; k < 4; k++)
		if (4 * t + k < n) perm_out[4 * t + k] = perm[4 * t + k];
}

// ---- multipoles ----------------------------------------------------------------------------------
// a node without particles (src/tree.cpp:214-227)
__device__ void empty_node(const DNode& nd, DMulti& M) {
#pragma clang fp contract(off)
	double bmin[3], bmax[3];
	d_box_range(nd.boxid, bmin, bmax);
	M.N = 0;
	for (int q = 0; q < 17; q++) M.m[q] = 0.0f;
	for (int d = 0; d < 3; d++) {
		M.x[d] = d_double_to_pos(0.5 * (bmax[d] - bmin[d]));
		M.rmin[d] = bmin[d];
		M.rmax[d] = bmax[d];
	}
	M.r = 0.0f;
}

// all leaves: 16 threads per leaf, four leaves per work group
__global__ __launch_bounds__(64) void k_leaf_moments(const DNode* __restrict__ nodes, int nn, const int32_t* __restrict__ pos,
		const float* __restrict__ mass, DMulti* __restrict__ out) {
#pragma clang fp contract(off)
	__shared__ float red[4][17][16];
	__shared__ float rr[4][16];
	__shared__ double bb[4][16][6];
	const int slot = threadIdx.x >> 4;
	const int k = threadIdx.x & 15;
	const int j = blockIdx.x * 4 + slot;
	const bool active = j < nn && nodes[j].c0 < 0;
	DNode nd{};
	if (active) nd = nodes[j];
	const bool nonempty = active && nd.pend > nd.pbegin;
	float M[17];
	for (int q = 0; q < 17; q++) M[q] = 0.0f;
	double Xcom[3] = {0.0, 0.0, 0.0};
	float r = 0.0f;
	double mn[3] = {1.0, 1.0, 1.0}, mx[3] = {0.0, 0.0, 0.0};
	int32_t cx[3] = {0, 0, 0};
	if (nonempty) {
		// part_vect_center_of_mass (src/part_vect.cpp:542-565): FP64 sum in particle order
		double com[3] = {0.0, 0.0, 0.0};
		for (int64_t i = nd.pbegin; i < nd.pend; i++)
			for (int d = 0; d < 3; d++) com[d] += d_pos_to_double(pos[3 * i + d]);
		const double cnt = double(nd.pend - nd.pbegin);
		for (int d = 0; d < 3; d++) {
			cx[d] = d_double_to_pos(com[d] / cnt);
			Xcom[d] = d_pos_to_double(cx[d]);
		}
		// lane k: particles i + k of each block of 16 (padding past the end: position 0, mass 0)
		for (int64_t i = nd.pbegin; i < nd.pend; i += 16) {
			double X[3];
			float ms;
			if (i + k < nd.pend) {
				for (int d = 0; d < 3; d++) X[d] = d_pos_to_double(pos[3 * (i + k) + d]);
				ms = mass[i + k];
			} else {
				X[0] = X[1] = X[2] = 0.0;
				ms = 0.0f;
			}
			float dx[3];
			for (int d = 0; d < 3; d++) dx[d] = float(X[d] - Xcom[d]);
			M[0] += ms;
#pragma unroll
			for (int a = 0; a < 3; a++)
#pragma unroll
				for (int b = 0; b <= a; b++) {
					const float Xab = dx[a] * dx[b];
					M[M2(a, b)] += ms * Xab;
#pragma unroll
					for (int l = 0; l <= b; l++) M[M3(a, b, l)] += ms * Xab * dx[l];
				}
		}
		// radius and particle box of this lane's particles (max / min are exact in any order)
		for (int64_t i = nd.pbegin + k; i < nd.pend; i += 16) {
			double v[3];
			for (int d = 0; d < 3; d++) {
				const double xd = d_pos_to_double(pos[3 * i + d]);
				v[d] = xd - Xcom[d];
				mx[d] = mx[d] < xd ? xd : mx[d];
				mn[d] = xd < mn[d] ? xd : mn[d];
			}
			const float a = float(d_vabs(v));
			r = r < a ? a : r;
		}
	}
	for (int q = 0; q < 17; q++) red[slot][q][k] = M[q];
	rr[slot][k] = r;
	for (int d = 0; d < 3; d++) {
		bb[slot][k][d] = mn[d];
		bb[slot][k][3 + d] = mx[d];
	}
	__syncthreads();
	if (!active) return;
	DMulti& o = out[j];
	if (!nonempty) {
		if (k == 0) empty_node(nd, o);
		return;
	}
	// lanes summed in order, 0..15 (slot q by thread q, slot 16 by thread 0)
	for (int q = k; q < 17; q += 16) {
		float s = 0.0f;
		for (int l = 0; l < 16; l++) s += red[slot][q][l];
		o.m[q] = s;
	}
	if (k == 0) {
		float rm = 0.0f;
		double lo[3] = {1.0, 1.0, 1.0}, hi[3] = {0.0, 0.0, 0.0};
		for (int l = 0; l < 16; l++) {
			rm = rm < rr[slot][l] ? rr[slot][l] : rm;
			for (int d = 0; d < 3; d++) {
				lo[d] = bb[slot][l][d] < lo[d] ? bb[slot][l][d] : lo[d];
				hi[d] = hi[d] < bb[slot][l][3 + d] ? bb[slot][l][3 + d] : hi[d];
			}
		}
		o.N = uint64_t(nd.pend - nd.pbegin);
		o.r = rm;
		for (int d = 0; d < 3; d++) {
			o.x[d] = cx[d];
			o.rmin[d] = lo[d];
			o.rmax[d] = hi[d];
		}
	}
}

// multipole<float>::operator>>= (tigergrav/multipole.hpp:414-433)
__device__ __forceinline__ void d_m2m_shift(float* me, const float* Y) {
#pragma clang fp contract(off)
#pragma unroll
	for (int p = 0; p < 3; p++)
#pragma unroll
		for (int q = p; q < 3; q++)
#pragma unroll
			for (int l = q; l < 3; l++) {
				float t = me[M3(p, q, l)];
				t += me[0] * Y[p] * Y[q] * Y[l];
				t += me[M2(p, q)] * Y[l];
				t += me[M2(q, l)] * Y[p];
				t += me[M2(l, p)] * Y[q];
				me[M3(p, q, l)] = t;
			}
#pragma unroll
	for (int p = 0; p < 3; p++)
#pragma unroll
		for (int q = p; q < 3; q++) me[M2(p, q)] += me[0] * Y[p] * Y[q];
}

// an interior node (src/tree.cpp:235-288)
__device__ void interior_moments(const DNode& nd, int k, DMulti* out) {
#pragma clang fp contract(off)
	DMulti o{};
	if (nd.pend == nd.pbegin) {
		empty_node(nd, o);
		out[k] = o;
		return;
	}
	const DMulti L = out[nd.c0];
	const DMulti R = out[nd.c1];
	o.N = L.N + R.N;
	double lx[3], rx[3], x[3];
	for (int d = 0; d < 3; d++) {
		lx[d] = d_pos_to_double(L.x[d]);
		rx[d] = d_pos_to_double(R.x[d]);
		o.x[d] = d_double_to_pos((lx[d] * double(L.N) + rx[d] * double(R.N)) / double(o.N));
		x[d] = d_pos_to_double(o.x[d]);
	}
	float ml[17], mr[17], yl[3], yr[3];
	for (int q = 0; q < 17; q++) {
		ml[q] = L.m[q];
		mr[q] = R.m[q];
	}
	for (int d = 0; d < 3; d++) {
		yl[d] = float(lx[d] - x[d]);
		yr[d] = float(rx[d] - x[d]);
	}
	d_m2m_shift(ml, yl);
	d_m2m_shift(mr, yr);
	for (int q = 0; q < 17; q++) o.m[q] = ml[q] + mr[q];
	double dl[3], dr[3];
	for (int d = 0; d < 3; d++) {
		dl[d] = lx[d] - x[d];
		dr[d] = rx[d] - x[d];
	}
	if (L.N == 0) {
		o.r = R.r;
	} else if (R.N == 0) {
		o.r = L.r;
	} else {
		const double a = d_vabs(dl) + double(L.r), b = d_vabs(dr) + double(R.r);
		o.r = float(a < b ? b : a);
	}
	for (int d = 0; d < 3; d++) {
		o.rmax[d] = L.rmax[d] < R.rmax[d] ? R.rmax[d] : L.rmax[d];
		o.rmin[d] = R.rmin[d] < L.rmin[d] ? R.rmin[d] : L.rmin[d];
	}
	double rmax = 0.0;
	for (int c = 0; c < 8; c++) {  // the eight corners, in the reference's order
		const double corner[3] = {(c & 1) ? o.rmax[0] : o.rmin[0], (c & 2) ? o.rmax[1] : o.rmin[1], (c & 4) ? o.rmax[2] : o.rmin[2]};
		double v[3];
		for (int d = 0; d < 3; d++) v[d] = x[d] - corner[d];
		const double a = d_vabs(v);
		rmax = c == 0 ? a : (rmax < a ? a : rmax);
	}
	const float rf = float(rmax);
	o.r = rf < o.r ? rf : o.r;
	out[k] = o;
}

// The walk's record of a node.  sbox: per node the box of its particles (leaves) or the union of its
// non-empty children's (Tree::sink_spans); the span is its diagonal, in FP64 with the host's
// operations.
__device__ void walk_record(const DNode* nodes, const DNode& nd, int k, const DMulti* multi, double* sbox, WalkNode* wn) {
#pragma clang fp contract(off)
	const DMulti& m = multi[k];
	double mn[3] = {1.0, 1.0, 1.0}, mx[3] = {0.0, 0.0, 0.0};
	const bool empty = nd.pend == nd.pbegin;
	if (!empty) {
		if (nd.c0 < 0) {
			for (int d = 0; d < 3; d++) {
				mn[d] = m.rmin[d];
				mx[d] = m.rmax[d];
			}
		} else {
			const int ch[2] = {nd.c0, nd.c1};
			for (int c = 0; c < 2; c++) {
				if (nodes[ch[c]].pend == nodes[ch[c]].pbegin) continue;
				const double* b = sbox + 6 * int64_t(ch[c]);
				for (int d = 0; d < 3; d++) {
					mx[d] = mx[d] < b[3 + d] ? b[3 + d] : mx[d];
					mn[d] = b[d] < mn[d] ? b[d] : mn[d];
				}
			}
		}
	}
	double* o = sbox + 6 * int64_t(k);
	for (int d = 0; d < 3; d++) {
		o[d] = mn[d];
		o[3 + d] = mx[d];
	}
	float span = 0.0f;
	if (!empty) {
		double s2 = 0.0;
		for (int d = 0; d < 3; d++) s2 += (mx[d] - mn[d]) * (mx[d] - mn[d]);
		span = float(sqrt(s2));
	}
	WalkNode w;
	w.pbegin = nd.pbegin;
	w.pend = nd.pend;
	w.c0 = nd.c0;
	w.c1 = nd.c1;
	for (int d = 0; d < 3; d++) w.x[d] = m.x[d];
	w.r = m.r;
	w.rmax = span;
	wn[k] = w;
}

struct UpArgs {
	const DNode* nodes;
	DMulti* multi;
	double* sbox;
	WalkNode* wn;  // null: moments only
};

__device__ __forceinline__ void up_node(const UpArgs& A, int k) {
	const DNode nd = A.nodes[k];
	if (nd.c0 >= 0) interior_moments(nd, k, A.multi);
	if (A.wn) walk_record(A.nodes, nd, k, A.multi, A.sbox, A.wn);
}

// one level, one thread per node
__global__ __launch_bounds__(64) void k_up_level(UpArgs A, int b, int e) {
	const int k = b + int(blockIdx.x) * 64 + int(threadIdx.x);
	if (k < e) up_node(A, k);
}

// a run of small levels, the deepest first, by one work group: begin[i] is level lo + i's first node
constexpr int UP_SMALL = 512;
struct UpLevels {
	int begin[MAX_SPLIT_LEVEL + 4];
	int levels;
};
__global__ __launch_bounds__(UP_SMALL) void k_up_levels(UpArgs A, UpLevels U) {
	for (int l = U.levels - 1; l >= 0; l--) {
		const int k = U.begin[l] + int(threadIdx.x);
		if (k < U.begin[l + 1]) up_node(A, k);
		__syncthreads();
	}
}

unsigned blocks(int64_t n, int b) { return unsigned((n + b - 1) / b); }

// pinned host staging for the copy back (full-rate transfers), grown on demand and kept for the
// process; one build at a time uses it
std::mutex pinned_mtx;
void* pinned_buf = nullptr;
size_t pinned_bytes = 0;

hipError_t pinned_staging(size_t bytes, void** out) {
	if (bytes > pinned_bytes) {
		if (pinned_buf) (void) hipHostFree(pinned_buf);
		pinned_buf = nullptr;
		pinned_bytes = 0;
		const size_t want = bytes + bytes / 4;
		const hipError_t e = hipHostMalloc(&pinned_buf, want, hipHostMallocDefault);
		if (e != hipSuccess) return e;
		pinned_bytes = want;
	}
	*out = pinned_buf;
	return hipSuccess;
}

double wall() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

// device array freed with its owner
struct Buf {
	void* p = nullptr;
	size_t bytes = 0;
	std::vector<void*>& later;  // takes the array when its owner goes: the stream may still use it
	explicit Buf(std::vector<void*>& l) : later(l) {}
	~Buf() {
		if (p) later.push_back(p);
	}
	hipError_t alloc(size_t b) {
		if (b <= bytes) return hipSuccess;
		if (p) later.push_back(p);
		p = nullptr;
		bytes = 0;
		const hipError_t e = dev_malloc(&p, b < 256 ? 256 : b);
		if (e == hipSuccess) bytes = b < 256 ? 256 : b;
		return e;
	}
	template <class T>
	T* as() const {
		return static_cast<T*>(p);
	}
};

}  // namespace

void DeviceTree::release() {
	if (pos) dev_free(pos);
	if (mass) dev_free(mass);
	if (order) dev_free(order);
	if (nodes) dev_free(nodes);
	if (multi) dev_free(multi);
	if (walk) dev_free(walk);
	*this = DeviceTree();
}

hipError_t device_build_tree(Tree& T, const int32_t* x, const float* masses, int64_t n, const TreeParams& p,
		double particle_mass, int device, hipStream_t s, std::string& err, double* t_out, bool on_device, DeviceTree* keep,
		std::vector<void*>& later) {
	const double t0 = wall();
	hipError_t e = hipSuccess;
#define DTCHK(call)                                                    \
	do {                                                               \
		e = (call);                                                    \
		if (e != hipSuccess) {                                         \
			err = std::string(#call) + ": " + hipGetErrorString(e);    \
			return e;                                                  \
		}                                                              \
	} while (0)
#define DTLAUNCH(name)                                                                 \
	do {                                                                               \
		e = hipGetLastError();                                                         \
		if (e != hipSuccess) {                                                         \
			err = std::string("device tree build: launch ") + name + ": " + hipGetErrorString(e); \
			return e;                                                                  \
		}                                                                              \
	} while (0)
	(void) hipGetLastError();  // an error left by an earlier call is not the build's
	if (n > int64_t(INT32_MAX) - 1) {
		err = "device tree build: more than 2^31 - 2 particles";
		return hipErrorInvalidValue;
	}
	DTCHK(hipSetDevice(device));
	T.P = p;
	T.m = particle_mass;
	T.lists = Lists();
	T.census = Census();
	Buf dpos(later), dmass(later), dorder(later), dnodes(later), dinfo(later), dmulti(later), dlog(later), dx(later), dmin(later);
	DTCHK(dpos.alloc(size_t(3 * n) * 4));
	DTCHK(dmass.alloc(size_t(n) * 4));
	DTCHK(dorder.alloc(size_t(n) * 8));
	// the input on the device
	const int32_t* xd = x;
	const float* md = masses;
	if (!on_device && n > 0) {
		DTCHK(dx.alloc(size_t(3 * n) * 4));
		DTCHK(hipMemcpyAsync(dx.p, x, size_t(3 * n) * 4, hipMemcpyHostToDevice, s));
		xd = dx.as<const int32_t>();
		if (masses) {
			DTCHK(dmin.alloc(size_t(n) * 4));
			DTCHK(hipMemcpyAsync(dmin.p, masses, size_t(n) * 4, hipMemcpyHostToDevice, s));
			md = dmin.as<const float>();
		}
	}
	const int ppn = p.parts_per_node;
	const int64_t split_cap = n / (int64_t(std::max(1, ppn)) + 1) + 1;  // splitting nodes of a level, at most
	constexpr int DT_BATCH = 4;
	const int log_cap = MAX_SPLIT_LEVEL + 2 + DT_BATCH;
	DTCHK(dlog.alloc(size_t(3 * log_cap) * sizeof(int32_t)));
	std::vector<int> level_begin;
	int le = 1;
	if (n > 0 && n <= SMALL_N) {
		Buf dperm(later);
		DTCHK(dperm.alloc(size_t(n) * 4));
		// every level splits split_cap nodes at most, MAX_SPLIT_LEVEL levels split
		DTCHK(dnodes.alloc(size_t(1 + 2 * split_cap * MAX_SPLIT_LEVEL) * sizeof(DNode)));
		DTCHK(dinfo.alloc(size_t(2 * split_cap) * sizeof(SplitInfo)));
		hipLaunchKernelGGL(k_small_tree, dim3(1), dim3(1024), 0, s, xd, int(n), dnodes.as<DNode>(), ppn, MAX_SPLIT_LEVEL, dinfo.as<SplitInfo>(),
				dlog.as<int32_t>(), dperm.as<int32_t>());
		DTLAUNCH("k_small_tree");
		hipLaunchKernelGGL(k_unpack, dim3(blocks(n, 256)), dim3(256), 0, s, nullptr, xd, dperm.as<const int32_t>(), md, float(particle_mass), n,
				dpos.as<int32_t>(), dmass.as<float>(), dorder.as<int64_t>());
		DTLAUNCH("k_unpack");
		std::vector<int32_t> lg(size_t(3 * log_cap), 0);
		DTCHK(hipMemcpyAsync(lg.data(), dlog.p, lg.size() * 4, hipMemcpyDeviceToHost, s));
		DTCHK(hipStreamSynchronize(s));
		for (int i = 0; i < log_cap; i++) {
			level_begin.push_back(lg[size_t(3 * i)]);
			le = lg[size_t(3 * i) + 1];
			if (lg[size_t(3 * i) + 2] == 0) break;
		}
	} else {
		Buf drec(later), dpnode(later), dlow(later), dloc(later), dbase(later), dmr(later), dflags(later), drank(later), dlev(later), scan_tmp(later);
		int64_t node_cap = 4 * (n / std::max(1, ppn)) + 16;
		const int tiles = int((n + 1 + LOW_TILE - 1) / LOW_TILE);
		DTCHK(drec.alloc(size_t(n) * sizeof(int4)));
		DTCHK(dpnode.alloc(size_t(n) * 4));
		DTCHK(dlow.alloc(size_t(n)));
		DTCHK(dloc.alloc(size_t(n + 1) * 4));
		DTCHK(dbase.alloc(size_t(tiles) * 4));
		DTCHK(dmr.alloc(size_t(n) * 4));
		DTCHK(dnodes.alloc(size_t(node_cap) * sizeof(DNode)));
		if (n > 0) {
			hipLaunchKernelGGL(k_records, dim3(blocks(n, 256)), dim3(256), 0, s, xd, n, drec.as<int4>(), dpnode.as<int32_t>());
			DTLAUNCH("k_records");
		}
		const DNode root{0, int32_t(n), -1, -1, -1, 0, 1};
		DTCHK(hipMemcpyAsync(dnodes.p, &root, sizeof(root), hipMemcpyHostToDevice, s));
		// Level by level, a batch of DT_BATCH levels at a time without a host wait: a level's first kernel
		// moves its extent from dlev on to the next and logs (lb, le, nsplit), which the others read;
		// grids are sized by bounds (a level's splitting nodes hold more than ppn particles each, so there are
		// at most split_cap of them, and a level has at most twice the previous level's nodes).  After a
		// batch the host reads the log, stops at the first level that split nothing (the levels after
		// it in the batch found no nodes and did nothing), and grows the node array for the next batch.
		const int64_t lvl_max = 2 * split_cap;
		const int64_t fl_cap = lvl_max + 1;
		DTCHK(dflags.alloc(size_t(fl_cap + 1) * 4));
		DTCHK(drank.alloc(size_t(fl_cap + 1) * 4));
		DTCHK(dinfo.alloc(size_t(fl_cap) * sizeof(SplitInfo)));
		DTCHK(dlev.alloc(2 * sizeof(int32_t)));
		const int32_t lev0[2] = {0, 1};
		DTCHK(hipMemcpyAsync(dlev.p, lev0, sizeof(lev0), hipMemcpyHostToDevice, s));
		size_t level_scan_bytes = 0;
		DTCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, level_scan_bytes, dflags.as<int32_t>(), drank.as<int32_t>(), int(fl_cap), s));
		DTCHK(scan_tmp.alloc(level_scan_bytes));
		const LowCount S{dloc.as<const int32_t>(), dbase.as<const int32_t>()};
		int64_t le_h = 1;      // nodes made, as of the host's last look
		int64_t nl_bound = 1;  // the current level's nodes, at most
		int level = 0;
		bool finished = false;
		while (!finished) {
			if (level + DT_BATCH > log_cap) {
				err = "device tree build: more levels than the split limit allows";
				return hipErrorInvalidValue;
			}
			// node capacity for this batch
			int64_t add = 0;
			for (int64_t i = 0, b = nl_bound; i < DT_BATCH; i++, b = std::min(2 * b, lvl_max)) add += 2 * std::min(b, split_cap);
			if (le_h + add > INT32_MAX) {
				err = "device tree build: node count overflow";
				return hipErrorInvalidValue;
			}
			if (le_h + add > node_cap) {
				// grow the node array, keeping the nodes made so far
				int64_t cap = node_cap;
				while (cap < le_h + add) cap *= 2;
				Buf bigger(later);
				DTCHK(bigger.alloc(size_t(cap) * sizeof(DNode)));
				DTCHK(hipMemcpyAsync(bigger.p, dnodes.p, size_t(le_h) * sizeof(DNode), hipMemcpyDeviceToDevice, s));
				std::swap(dnodes.p, bigger.p);
				std::swap(dnodes.bytes, bigger.bytes);
				node_cap = cap;
			}
			const int first = level;
			for (int i = 0; i < DT_BATCH; i++, level++) {
				const int bound = int(nl_bound);
				int32_t* lg = dlog.as<int32_t>() + 3 * level;
				if (bound <= 8192) {
					// one launch; past a few thousand nodes its one work group takes longer than the four below
					hipLaunchKernelGGL(k_level, dim3(1), dim3(1024), 0, s, dnodes.as<const DNode>(), dlev.as<int32_t>(), ppn, MAX_SPLIT_LEVEL,
							dinfo.as<SplitInfo>(), lg);
					DTLAUNCH("k_level");
				} else {
					const int32_t* lev = dlev.as<const int32_t>();
					hipLaunchKernelGGL(k_split_flags, dim3(blocks(bound + 1, 256)), dim3(256), 0, s, dnodes.as<const DNode>(), lev, ppn, MAX_SPLIT_LEVEL,
							dflags.as<int32_t>(), bound);
					DTLAUNCH("k_split_flags");
					size_t have = scan_tmp.bytes;
					DTCHK(hipcub::DeviceScan::ExclusiveSum(scan_tmp.p, have, dflags.as<int32_t>(), drank.as<int32_t>(), bound + 1, s));
					hipLaunchKernelGGL(k_split_setup, dim3(blocks(bound, 256)), dim3(256), 0, s, dnodes.as<const DNode>(), lev,
							dflags.as<const int32_t>(), drank.as<const int32_t>(), dinfo.as<SplitInfo>());
					hipLaunchKernelGGL(k_next_level, dim3(1), dim3(64), 0, s, dlev.as<int32_t>(), drank.as<const int32_t>(), lg);
					DTLAUNCH("k_split_setup/k_next_level");
				}
				if (n > 0) {
					hipLaunchKernelGGL(k_low_tiles, dim3(tiles), dim3(1024), 0, s, drec.as<const int4>(), dpnode.as<const int32_t>(), n, lg,
							dinfo.as<const SplitInfo>(), dlow.as<uint8_t>(), dloc.as<int32_t>(), dbase.as<int32_t>(), tiles);
					if (tiles > 1) hipLaunchKernelGGL(k_low_tops, dim3(1), dim3(1024), 0, s, dbase.as<int32_t>(), tiles);
					DTLAUNCH("k_low_tiles/k_low_tops");
					hipLaunchKernelGGL(k_high_side_lows, dim3(blocks(n, 256)), dim3(256), 0, s, dpnode.as<const int32_t>(), n,
							dnodes.as<const DNode>(), dlow.as<const uint8_t>(), S, dmr.as<int32_t>());
					hipLaunchKernelGGL(k_exchange, dim3(blocks(n, 256)), dim3(256), 0, s, drec.as<int4>(), dpnode.as<int32_t>(), n, lg,
							dinfo.as<const SplitInfo>(), dnodes.as<DNode>(), dlow.as<const uint8_t>(), S, dmr.as<const int32_t>());
					DTLAUNCH("k_high_side_lows/k_exchange");
				}
				nl_bound = std::min(2 * nl_bound, lvl_max);
			}
			int32_t lg[3 * DT_BATCH];
			DTCHK(hipMemcpyAsync(lg, dlog.as<int32_t>() + 3 * first, sizeof(lg), hipMemcpyDeviceToHost, s));
			DTCHK(hipStreamSynchronize(s));
			for (int i = 0; i < DT_BATCH; i++) {
				const int32_t lb_i = lg[3 * i], le_i = lg[3 * i + 1], ns = lg[3 * i + 2];
				level_begin.push_back(lb_i);
				le = le_i;
				if (ns == 0) {
					finished = true;
					break;
				}
			}
			le_h = int64_t(lg[3 * DT_BATCH - 2]) + 2 * int64_t(lg[3 * DT_BATCH - 1]);
			nl_bound = std::max<int64_t>(2 * int64_t(lg[3 * DT_BATCH - 1]), 1);  // the next level's nodes, exactly
		}
		if (n > 0) {
			hipLaunchKernelGGL(k_unpack, dim3(blocks(n, 256)), dim3(256), 0, s, drec.as<const int4>(), nullptr, nullptr, md, float(particle_mass), n,
					dpos.as<int32_t>(), dmass.as<float>(), dorder.as<int64_t>());
			DTLAUNCH("k_unpack");
		}
	}
	level_begin.push_back(le);
	const int nn = le;
	const double t1 = wall();
	// multipoles: all leaves, then levels from the deepest up; with the tree kept, the walk's records too
	DTCHK(dmulti.alloc(size_t(nn) * sizeof(DMulti)));
	Buf dsbox(later), dwalk(later);
	if (keep) {
		DTCHK(dsbox.alloc(size_t(nn) * 6 * sizeof(double)));
		DTCHK(dwalk.alloc(size_t(nn) * sizeof(WalkNode)));
	}
	hipLaunchKernelGGL(k_leaf_moments, dim3(blocks(nn, 4)), dim3(64), 0, s, dnodes.as<const DNode>(), nn, dpos.as<const int32_t>(),
			dmass.as<const float>(), dmulti.as<DMulti>());
	DTLAUNCH("k_leaf_moments");
	const UpArgs up{dnodes.as<const DNode>(), dmulti.as<DMulti>(), dsbox.as<double>(), dwalk.as<WalkNode>()};
	const int levels = int(level_begin.size()) - 1;
	auto level_size = [&](int l) { return level_begin[size_t(l) + 1] - level_begin[size_t(l)]; };
	for (int l = levels - 1; l >= 0;) {
		if (level_size(l) > UP_SMALL) {
			hipLaunchKernelGGL(k_up_level, dim3(blocks(level_size(l), 64)), dim3(64), 0, s, up, level_begin[size_t(l)], level_begin[size_t(l) + 1]);
			DTLAUNCH("k_up_level");
			l--;
			continue;
		}
		int lo = l;
		while (lo > 0 && level_size(lo - 1) <= UP_SMALL) lo--;
		UpLevels U;
		U.levels = l - lo + 1;
		for (int i = 0; i <= U.levels; i++) U.begin[i] = level_begin[size_t(lo + i)];
		hipLaunchKernelGGL(k_up_levels, dim3(1), dim3(UP_SMALL), 0, s, up, U);
		DTLAUNCH("k_up_levels");
		l = lo - 1;
	}
	if (keep) {
		// everything stays on the device: the caller's DeviceTree takes the arrays
		keep->release();
		keep->n = n;
		keep->nn = nn;
		keep->level_begin = level_begin;
		keep->pos = static_cast<int32_t*>(dpos.p);
		keep->mass = static_cast<float*>(dmass.p);
		keep->order = static_cast<int64_t*>(dorder.p);
		keep->nodes = static_cast<DNode*>(dnodes.p);
		keep->multi = static_cast<DMulti*>(dmulti.p);
		keep->walk = static_cast<WalkNode*>(dwalk.p);
		dpos.p = dmass.p = dorder.p = dnodes.p = dmulti.p = dwalk.p = nullptr;
		T.pos.clear();
		T.mass.clear();
		T.order.clear();
		T.nodes.clear();
		T.leaves.clear();
		T.max_level = int(level_begin.size()) - 2;
		if (t_out) {
			t_out[0] = t1 - t0;
			t_out[1] = wall() - t1;
		}
		return hipSuccess;
	}
#undef DTLAUNCH
	{
		DeviceTree view;  // the build's arrays, still owned by the buffers above
		view.n = n;
		view.nn = nn;
		view.pos = static_cast<int32_t*>(dpos.p);
		view.mass = static_cast<float*>(dmass.p);
		view.order = static_cast<int64_t*>(dorder.p);
		view.nodes = static_cast<DNode*>(dnodes.p);
		view.multi = static_cast<DMulti*>(dmulti.p);
		e = device_tree_to_host(view, T, s, err);
		view = DeviceTree();  // not released: the buffers free them
		if (e != hipSuccess) return e;
	}
	if (t_out) {
		t_out[0] = t1 - t0;
		t_out[1] = wall() - t1;
	}
	return hipSuccess;
#undef DTCHK
}

hipError_t device_tree_to_host(const DeviceTree& D, Tree& T, hipStream_t s, std::string& err) {
	hipError_t e = hipSuccess;
#define DTCHK(call)                                                    \
	do {                                                               \
		e = (call);                                                    \
		if (e != hipSuccess) {                                         \
			err = std::string(#call) + ": " + hipGetErrorString(e);    \
			return e;                                                  \
		}                                                              \
	} while (0)
	const int64_t n = D.n;
	const int nn = int(D.nn);
	// through pinned staging
	std::lock_guard<std::mutex> lock(pinned_mtx);
	const size_t b_pos = size_t(3 * n) * 4, b_mass = size_t(n) * 4, b_order = size_t(n) * 8;
	const size_t b_nodes = size_t(nn) * sizeof(DNode), b_multi = size_t(nn) * sizeof(DMulti);
	const size_t o_mass = b_pos, o_order = o_mass + b_mass, o_nodes = (o_order + b_order + 255) / 256 * 256,
			o_multi = (o_nodes + b_nodes + 255) / 256 * 256;
	void* stage = nullptr;
	DTCHK(pinned_staging(o_multi + b_multi, &stage));
	char* st = static_cast<char*>(stage);
	if (n > 0) {
		DTCHK(hipMemcpyAsync(st, D.pos, b_pos, hipMemcpyDeviceToHost, s));
		DTCHK(hipMemcpyAsync(st + o_mass, D.mass, b_mass, hipMemcpyDeviceToHost, s));
		DTCHK(hipMemcpyAsync(st + o_order, D.order, b_order, hipMemcpyDeviceToHost, s));
	}
	DTCHK(hipMemcpyAsync(st + o_nodes, D.nodes, b_nodes, hipMemcpyDeviceToHost, s));
	DTCHK(hipMemcpyAsync(st + o_multi, D.multi, b_multi, hipMemcpyDeviceToHost, s));
	DTCHK(hipStreamSynchronize(s));
	T.pos.resize(size_t(3 * n));
	T.mass.resize(size_t(n));
	T.order.resize(size_t(n));
	const DNode* hn = reinterpret_cast<const DNode*>(st + o_nodes);
	const DMulti* hm = reinterpret_cast<const DMulti*>(st + o_multi);
	{
		// the particle arrays in parallel slices
		const int64_t chunk = 1 << 16;
		const int64_t nch = (n + chunk - 1) / chunk;
#pragma omp parallel for schedule(static)
		for (int64_t c = 0; c < nch; c++) {
			const int64_t b = c * chunk, e2 = std::min(n, b + chunk);
			std::memcpy(T.pos.data() + 3 * b, st + 12 * b, size_t(e2 - b) * 12);
			std::memcpy(T.mass.data() + b, st + o_mass + 4 * b, size_t(e2 - b) * 4);
			std::memcpy(T.order.data() + b, st + o_order + 8 * b, size_t(e2 - b) * 8);
		}
	}
	T.nodes.resize(size_t(nn));
	T.leaves.clear();
	T.max_level = 0;
#pragma omp parallel for schedule(static)
	for (int i = 0; i < nn; i++) {
		Node& o = T.nodes[size_t(i)];
		const DNode& a = hn[size_t(i)];
		const DMulti& m = hm[size_t(i)];
		o.pbegin = a.pbegin;
		o.pend = a.pend;
		o.child[0] = a.c0;
		o.child[1] = a.c1;
		o.parent = a.parent;
		o.level = a.level;
		o.boxid = boxid_t(a.boxid);
		std::memcpy(o.m, m.m, sizeof(o.m));
		o.r = m.r;
		for (int d = 0; d < 3; d++) {
			o.x[d] = m.x[d];
			o.rmin[d] = m.rmin[d];
			o.rmax[d] = m.rmax[d];
		}
		o.N = m.N;
	}
	for (int i = 0; i < nn; i++) {
		if (T.nodes[size_t(i)].leaf()) T.leaves.push_back(i);
		T.max_level = std::max(T.max_level, T.nodes[size_t(i)].level);
	}
	return hipSuccess;
#undef DTCHK
}

}  // namespace tg
