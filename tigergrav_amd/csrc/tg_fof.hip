// tg_fof.hip -- friends-of-friends groups on the device (tree::find_groups, src/tree.cpp:637-760,
// with part_vect_find_groups, src/part_vect.cpp:84-120).
//
// The reference links particles i, j when the squared int32 wrap-around separation, taken in
// uint64, is below L^2 and not zero (L = N^(-1/3) link_len (2^32 - 1), truncated to an integer),
// and relabels every linked particle with the smallest id among its links until nothing changes,
// each particle's first id being its own tree-order index.  At convergence a linked particle
// carries the smallest tree-order index of its connected component; an unlinked one keeps
// DEFAULT_GROUP.  Here the same components come from a lock-free union-find in which the larger
// root is always hooked under the smaller, so every root is its component's smallest index:
//   * candidate leaf pairs: one thread per leaf walks the tree and keeps the leaves whose particle
//     boxes come within L of its own (minimum image), counted, then written;
//   * links: one 64-lane group per candidate pair tests every particle pair with the reference's
//     integer test and unites the linked ones;
//   * labels: the root of every linked particle, DEFAULT_GROUP for the rest, in tree and in input
//     order.
// The nodes come from the device build's tree where that is current, else from the host's, whose boxes are
// then made anew from the particles (tg_solver_update_particles moves them under the tree); only the
// labels in input order cross to the host (with set_particles at 2M clustered particles, leaves of 32:
// 27.8 -> 8.7 ms; before, tree and order were copied, the nodes rebuilt and the labels permuted on
// the host).
// The candidate search only has to find a superset of the linked pairs, so its box test is in
// FP64 with a margin; the link test itself is the reference's exact integer one.
//
// Across the periodic boundary: the reference's integer test wraps, but the ranges it searches
// (range_expand / ranges_intersect, src/tree.cpp:660-670, src/range.cpp:80-116) are not
// wrapped, so a pair straddling the box edge is seen only where a kd box reaches across it, and
// then by one side only.  Here such a pair is never a friend (its coordinate difference must not
// wrap), in either boundary mode, and groups are the plain connected components; every pair away
// from the edge is treated as the reference treats it.
#include "tg_fof.hpp"
#include "tg_devmem.hpp"
#include "tg_scan.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

namespace tg {

namespace {

struct FofNode {
	int32_t pbegin, pend, c0, c1;
	double mn[3], mx[3];
};

// the smallest distance between two boxes on the unit torus (periodic) or in space, per axis
__device__ __forceinline__ double axis_gap(double amn, double amx, double bmn, double bmx, bool periodic) {
	double g = 0.0;
	const double d1 = bmn - amx, d2 = amn - bmx;
	g = d1 > g ? d1 : g;
	g = d2 > g ? d2 : g;
	if (periodic) {
		// the box shifted by one period either way
		double gp = 0.0, gm = 0.0;
		const double p1 = (bmn + 1.0) - amx, p2 = amn - (bmx + 1.0);
		gp = p1 > gp ? p1 : gp;
		gp = p2 > gp ? p2 : gp;
		const double m1 = (bmn - 1.0) - amx, m2 = amn - (bmx - 1.0);
		gm = m1 > gm ? m1 : gm;
		gm = m2 > gm ? m2 : gm;
		g = gp < g ? gp : g;
		g = gm < g ? gm : g;
	}
	return g;
}

__device__ __forceinline__ bool boxes_near(const FofNode& a, const FofNode& b, double L2, bool periodic) {
	double s = 0.0;
	for (int d = 0; d < 3; d++) {
		const double g = axis_gap(a.mn[d], a.mx[d], b.mn[d], b.mx[d], periodic);
		s += g * g;
	}
	return s <= L2;
}

// the search's record of a device-built node
__global__ __launch_bounds__(256) void k_fof_nodes(const DNode* __restrict__ nodes, const DMulti* __restrict__ multi, int64_t nn,
		FofNode* __restrict__ out) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= nn) return;
	const DNode d = nodes[i];
	FofNode o;
	o.pbegin = d.pbegin;
	o.pend = d.pend;
	o.c0 = d.c0;
	o.c1 = d.c1;
	for (int k = 0; k < 3; k++) {
		o.mn[k] = multi[i].rmin[k];
		o.mx[k] = multi[i].rmax[k];
	}
	out[i] = o;
}

constexpr int STACK = 256;

// pass 0 counts each leaf's candidates (leaves b >= a whose boxes come within L), pass 1 writes
// them at the leaf's offset
__global__ void k_fof_candidates(const FofNode* __restrict__ nodes, const int4* __restrict__ leaves, int nleaves, double L2, int periodic,
		int pass, int64_t* __restrict__ count, const int64_t* __restrict__ offset, int2* __restrict__ pairs, int* __restrict__ overflow) {
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= nleaves) return;
	const int a = leaves[k].x;
	const FofNode A = nodes[a];
	int64_t c = 0;
	if (A.pend == A.pbegin) {
		if (!pass) count[k] = 0;
		return;
	}
	int64_t o = pass ? offset[k] : 0;
	int stack[STACK];
	int sp = 0;
	stack[sp++] = 0;
	while (sp > 0) {
		const int id = stack[--sp];
		const FofNode B = nodes[id];
		if (B.pend == B.pbegin || !boxes_near(A, B, L2, periodic != 0)) continue;
		if (B.c0 < 0) {
			if (id >= a) {
				if (pass) pairs[o + c] = make_int2(a, id);
				c++;
			}
		} else {
			if (sp + 2 > STACK) {
				atomicOr(overflow, 1);
				continue;
			}
			stack[sp++] = B.c1;
			stack[sp++] = B.c0;
		}
	}
	if (!pass) count[k] = c;
}

// parents only ever decrease (parent[i] <= i, equal at roots), so the walk ends even on stale
// reads; loads are device-coherent so other groups' hooks are seen
__device__ __forceinline__ int ld(const int* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ int uf_find(int* parent, int x) {
	int p = ld(parent + x);
	while (p != x) {
		const int gp = ld(parent + p);
		if (gp != p) parent[x] = gp;  // path halving: only ever lowers a parent to an ancestor
		x = p;
		p = gp;
	}
	return x;
}

// unites the sets of a and b; returns their root as of then
__device__ int uf_union(int* parent, int a, int b) {
	for (;;) {
		a = uf_find(parent, a);
		b = uf_find(parent, b);
		if (a == b) return a;
		if (a > b) {
			const int t = a;
			a = b;
			b = t;
		}
		// hook the larger root under the smaller one
		const int old = atomicCAS(&parent[b], b, a);
		if (old == b) return a;
		b = old;
	}
}

// a node's box widened by the linking length, in positions
struct Reach {
	int lo[3], hi[3];
};

__device__ __forceinline__ Reach box_reach(const FofNode& b, double Lb) {
	Reach r;
	for (int d = 0; d < 3; d++) {
		r.lo[d] = int(fmax(floor((b.mn[d] - 0.5 - Lb) * 4294967296.0), -2147483648.0));
		r.hi[d] = int(fmin(ceil((b.mx[d] - 0.5 + Lb) * 4294967296.0), 2147483647.0));
	}
	return r;
}

__device__ __forceinline__ bool within(const Reach& r, const int4& x) {
	return x.x >= r.lo[0] && x.x <= r.hi[0] && x.y >= r.lo[1] && x.y <= r.hi[1] && x.z >= r.lo[2] && x.z <= r.hi[2];
}

// Every particle pair of each candidate leaf pair, the reference's integer test.  A linking length is
// a fraction of the spacing, so of two neighbouring leaves only the particles next to the common face
// can link: each leaf's are kept in LDS where they come within reach of the other's box (the
// candidate search's margin), then lane = (particle of A, phase), the phases splitting B's.  In a
// cluster most links join particles already in one set, which a parent equal to the last root shows
// without a walk.  Bound by its chains of loads (pair, node, particles, parents): 2M clustered
// particles, leaves of 32, 2.46 -> 1.28 ms against every pair of two leaves tested in turn.
constexpr int64_t LINK_PAIRS = 1 << 25;  // of a launch, which takes fewer than 2^32 threads
__global__ __launch_bounds__(64) void k_fof_link(const FofNode* __restrict__ nodes, const int2* __restrict__ pairs, int64_t npairs,
		const int4* __restrict__ parts, double Lb, uint64_t L2, int* parent, int* linked) {
	__shared__ int4 sa[64], sb[64];
	const int64_t q = blockIdx.x;
	if (q >= npairs) return;
	const int lane = int(threadIdx.x);
	const int2 pr = pairs[q];
	const FofNode &A = nodes[pr.x], &B = nodes[pr.y];
	const bool same = pr.x == pr.y;
	const int ae = A.pend, bb = B.pbegin, be = B.pend;
	const Reach ra = box_reach(A, Lb), rb = box_reach(B, Lb);
	const uint64_t before = (uint64_t(1) << lane) - 1;
	for (int a0 = A.pbegin; a0 < ae; a0 += 64) {
		int4 x = a0 + lane < ae ? parts[a0 + lane] : make_int4(0, 0, 0, 0);
		bool in = a0 + lane < ae && (same || within(rb, x));
		uint64_t m = __ballot(in);
		const int na = __popcll(m);
		if (na == 0) continue;
		x.w = a0 + lane;
		if (in) sa[__popcll(m & before)] = x;
		const int lg = na <= 1 ? 0 : 32 - __clz(na - 1);
		const int P = 64 >> lg, ph = lane >> lg, ia = lane & ((1 << lg) - 1);
		for (int b0 = same ? a0 : bb; b0 < be; b0 += 64) {
			x = b0 + lane < be ? parts[b0 + lane] : make_int4(0, 0, 0, 0);
			in = b0 + lane < be && (same || within(ra, x));
			m = __ballot(in);
			const int nb = __popcll(m);
			x.w = b0 + lane;
			if (in) sb[__popcll(m & before)] = x;
			__syncthreads();
			if (ia < na) {
				const int4 xi = sa[ia];
				const int i = xi.w;
				int root = -1;  // of i's set, when last looked at
				for (int k = ph; k < nb; k += P) {
					const int4 xj = sb[k];
					const int j = xj.w;
					// vect<pos_type> difference (int32 wrap), then vect<uint64_t> and its dot product; a
					// difference that wraps crosses the box edge
					const int64_t ex = int64_t(xi.x) - int64_t(xj.x), ey = int64_t(xi.y) - int64_t(xj.y), ez = int64_t(xi.z) - int64_t(xj.z);
					const bool wraps = ex != int64_t(int32_t(ex)) || ey != int64_t(int32_t(ey)) || ez != int64_t(int32_t(ez));
					const uint64_t d2 = uint64_t(int64_t(int32_t(ex)) * int32_t(ex)) + uint64_t(int64_t(int32_t(ey)) * int32_t(ey)) +
							uint64_t(int64_t(int32_t(ez)) * int32_t(ez));
					if (d2 < L2 && d2 != 0 && !wraps && (!same || j > i)) {
						// a parent that was i's root once keeps j in i's set
						if (root >= 0 && ld(parent + j) == root) {
							if (!linked[j]) linked[j] = 1;
							continue;
						}
						root = uf_union(parent, i, j);
						linked[i] = 1;
						linked[j] = 1;
					}
				}
			}
			__syncthreads();
		}
	}
}

__global__ void k_fof_init(int* parent, int* linked, int64_t n) {
	const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < n) {
		parent[i] = int(i);
		linked[i] = 0;
	}
}

// the labels in tree and in input order; the groups counted by their roots
__global__ __launch_bounds__(256) void k_fof_labels(int* parent, const int* __restrict__ linked, const int64_t* __restrict__ order, int64_t n,
		uint64_t* __restrict__ group, uint64_t* __restrict__ group_in, unsigned long long* __restrict__ ngroups) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	const uint64_t g = i < n && linked[i] ? uint64_t(uf_find(parent, int(i))) : TG_FOF_NONE;
	const int roots = __syncthreads_count(i < n && g == uint64_t(i));
	if (threadIdx.x == 0 && roots) atomicAdd(ngroups, (unsigned long long) roots);
	if (i >= n) return;
	group[i] = g;
	group_in[order[i]] = g;
}

// device memory of one call, freed once the stream has drained
struct Scratch {
	hipStream_t s;
	std::vector<void*> blocks;
	~Scratch() {
		(void) hipStreamSynchronize(s);
		for (void* p : blocks) dev_free(p);
	}
	template <class T>
	hipError_t get(T** p, size_t count) {
		void* q = nullptr;
		const hipError_t e = dev_malloc(&q, std::max<size_t>(count * sizeof(T), 16));
		if (e == hipSuccess) blocks.push_back(q);
		*p = static_cast<T*>(q);
		return e;
	}
};

}  // namespace

hipError_t fof_device(const FofSource& F, double link_len, hipStream_t s, uint64_t* group_tree, uint64_t* group_input, int64_t* n_groups,
		std::string& err) {
	const int64_t n = F.n, nn = F.nn;
	hipError_t e = hipSuccess;
#define FCHK(call)                                                 \
	do {                                                           \
		e = (call);                                                \
		if (e != hipSuccess) {                                     \
			err = std::string(#call) + ": " + hipGetErrorString(e); \
			return e;                                              \
		}                                                          \
	} while (0)
	*n_groups = 0;
	if (n == 0) return hipSuccess;
	// the reference's integer linking length (src/part_vect.cpp:86-88)
	const uint64_t L = uint64_t((std::pow(double(n), -1.0 / 3.0) * link_len) * 4294967295.0);
	const uint64_t L2 = L * L;
	// candidate boxes within the linking length, with a margin (the exact test is per pair)
	const double Lb = 1.01 * double(L) / 4294967296.0 + 1e-9;
	const int nleaves = F.n_leaf_items;
	std::vector<FofNode> hn;
	Scratch scratch{s, {}};  // drained before hn goes
	FofNode* nodes;
	int64_t *count, *offset, *work, *info;  // info: candidate pairs, overflow, groups
	int *parent, *linked;
	uint64_t* gin;
	int2* pairs;
	ScanSet sc;
	FCHK(scratch.get(&nodes, size_t(nn)));
	FCHK(scratch.get(&count, size_t(nleaves)));
	FCHK(scratch.get(&offset, size_t(nleaves)));
	FCHK(scratch.get(&info, 3));
	FCHK(scratch.get(&parent, size_t(n)));
	FCHK(scratch.get(&linked, size_t(n)));
	FCHK(scratch.get(&gin, size_t(n)));
	sc.add(count, offset, nleaves);
	FCHK(scratch.get(&work, size_t(scan_workspace(sc))));
	if (F.dtree) {
		hipLaunchKernelGGL(k_fof_nodes, dim3(unsigned((nn + 255) / 256)), dim3(256), 0, s, F.dtree->nodes, F.dtree->multi, nn, nodes);
		FCHK(hipGetLastError());
	} else {
		// the boxes of the particles where they are: those of a tree kept under moved particles are stale
		const std::vector<double> box = F.tree->particle_boxes();
		hn.resize(static_cast<size_t>(nn));
		for (int64_t i = 0; i < nn; i++) {
			const Node& d = F.tree->nodes[size_t(i)];
			FofNode& o = hn[size_t(i)];
			o.pbegin = d.pbegin;
			o.pend = d.pend;
			o.c0 = d.child[0];
			o.c1 = d.child[1];
			for (int k = 0; k < 3; k++) {
				o.mn[k] = box[6 * size_t(i) + size_t(k)];
				o.mx[k] = box[6 * size_t(i) + 3 + size_t(k)];
			}
		}
		FCHK(hipMemcpyAsync(nodes, hn.data(), hn.size() * sizeof(FofNode), hipMemcpyHostToDevice, s));
	}
	FCHK(hipMemsetAsync(info, 0, 3 * 8, s));
	const bool periodic = false;  // pairs across the box edge are not friends (above)
	const unsigned lb = unsigned((nleaves + 127) / 128), pb = unsigned((n + 255) / 256);
	int* overflow = reinterpret_cast<int*>(info + 1);
	hipLaunchKernelGGL(k_fof_init, dim3(pb), dim3(256), 0, s, parent, linked, n);
	FCHK(hipGetLastError());
	hipLaunchKernelGGL(k_fof_candidates, dim3(lb), dim3(128), 0, s, nodes, F.leaf_items, nleaves, Lb * Lb, int(periodic), 0, count, nullptr, nullptr,
			overflow);
	FCHK(hipGetLastError());
	FCHK(scan_columns(sc, work, info, s));
	int64_t v[3];
	FCHK(hipMemcpyAsync(v, info, sizeof(v), hipMemcpyDeviceToHost, s));
	FCHK(hipStreamSynchronize(s));
	const int64_t npairs = v[0];
	if (v[1]) {
		err = "friends-of-friends: tree deeper than the candidate search's stack";
		return hipErrorInvalidValue;
	}
	if (npairs > int64_t(INT32_MAX)) {
		err = "friends-of-friends: more than 2^31 candidate leaf pairs";
		return hipErrorInvalidValue;
	}
	FCHK(scratch.get(&pairs, size_t(npairs)));
	hipLaunchKernelGGL(k_fof_candidates, dim3(lb), dim3(128), 0, s, nodes, F.leaf_items, nleaves, Lb * Lb, int(periodic), 1, count, offset, pairs,
			overflow);
	FCHK(hipGetLastError());
	for (int64_t q0 = 0; q0 < npairs; q0 += LINK_PAIRS) {
		const int64_t m = std::min(npairs - q0, LINK_PAIRS);
		hipLaunchKernelGGL(k_fof_link, dim3(unsigned(m)), dim3(64), 0, s, nodes, pairs + q0, m, F.parts, Lb, L2, parent, linked);
		FCHK(hipGetLastError());
	}
	hipLaunchKernelGGL(k_fof_labels, dim3(pb), dim3(256), 0, s, parent, linked, F.order, n, group_tree, gin,
			reinterpret_cast<unsigned long long*>(info + 2));
	FCHK(hipGetLastError());
	FCHK(hipMemcpyAsync(v, info, sizeof(v), hipMemcpyDeviceToHost, s));
	FCHK(hipMemcpyAsync(group_input, gin, size_t(n) * 8, hipMemcpyDeviceToHost, s));
	FCHK(hipStreamSynchronize(s));
	*n_groups = v[2];
	return hipSuccess;
#undef FCHK
}

}  // namespace tg
