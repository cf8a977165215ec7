// tg_walk.hip -- the dual-tree walk (tree::kick_fmm's list construction, src/tree.cpp:378-635) on
// the device, producing the same lists as the host walk (Tree::walk).
//
// The recursion is flattened into steps.  A step holds work units, each one checklist pass of
// one node:
//   FIRST  (node n, direct checklist D, Ewald checklist E): the first MAC pass every non-empty
//          node makes (src/tree.cpp:424-494): far entries become CC (node) or CP (opened leaf's
//          particle range); near leaves are passed on opened, near interior nodes as their two
//          children (after all the opened leaves, as the reference appends them).  An interior
//          node's two next lists become the checklists of both children in the next step; a
//          leaf's become its drains.
//   DRAIN  (leaf n, one checklist, direct or Ewald): one round of the leaf's drain loop
//          (src/tree.cpp:530-602): opened leaves become PP ranges, far nodes PC, the rest is
//          opened or split for the next round.
// Per step, on the device, three launches: k_walk_count (one wave per unit, 64 checklist entries at a
// time) classifies every entry and counts every unit's outputs, k_walk_scan turns the counts into
// per-unit offsets (entries of each output, of the next checklists, next units) and the step's
// totals, k_walk_write (one wave per unit, from the kept categories) writes the outputs and the
// next step's units.  A step's extent lives in device memory (WalkState), so with capacities known
// from the solver's last walk every step is enqueued without a host wait; a step that would
// pass a capacity stops the walk, which is then run again with the host reading each step's totals to
// size the pools.  An entry's test is made in FP32 on integer separations and repeated in the host
// walk's FP64, without contraction, where the two sides come within 1e-5 of each other, so every
// decision is bit-identical.
// Each node's outputs are segments in step order, which is the host walk's order.  The node kinds'
// lists need no more: only first passes make them, level by level in node order, so the pools are
// the node-order CSR already.  The leaf kinds' segments (one per drain round) are put into node
// order at the end by k_walk_place.
#include "tg_walk.hpp"
#include "tg_devmem.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include <hipcub/hipcub.hpp>  // DeviceScan over the node lengths

namespace tg {
namespace {

enum { MODE_FIRST = 0, MODE_DRAIN_D = 1, MODE_DRAIN_E = 2 };

struct WalkUnit {
	int32_t node, mode, len_d, len_e;
	int64_t off_d, off_e;
	int32_t child, pad;  // a FIRST unit's sibling (0, 1): the two children of a node share their checklists
};

struct WalkParams {
	const WalkNode* nodes;
	const int4* cls;       // per node what a test needs, 16 bytes: centre, radius with the leaf flag in its sign
	const int4* rng;       // and what its outputs need: particle range, children
	const int32_t* lists;  // this step's checklists
	double theta_inv, h;
	float theta_inv_f, h_f;
	float r_ewald;
	int ewald;
};

enum { K_CC_D, K_CP_D, K_CC_E, K_CP_E, K_PC_D, K_PP_D, K_PC_E, K_PP_E, K_N };
// columns of a step's sizes: 8 outputs, next lists, next units, drain units
constexpr int COL_NEXT = K_N, COL_UNITS = K_N + 1, COL_DRAIN = K_N + 2, NCOL = K_N + 3;
constexpr int SCAN_TILE = 1024;  // units per scan block
constexpr int LOG_STEPS = 256;   // steps whose unit counts are kept for the next walk's grids

enum { WALK_OVERFLOW = 1, WALK_TOO_LONG = 2, WALK_DISAGREE = 4 };

// a step's extent and the pools' fill before it
struct WalkStep {
	int32_t nu;            // units
	int32_t pad;
	int64_t in_len;        // entries of its checklists
	int64_t base[K_N];     // entries in each output pool
	int64_t drains;        // drain records
};
struct WalkState {
	WalkStep st[2];        // by the step's parity: the running step and the next
	int32_t flags, pad;
	int64_t max_lists;
	int32_t max_units, steps;
	int32_t log_nu[LOG_STEPS];
};
struct WalkCaps {
	int64_t out[K_N], lists, units, drains;
};

// a drain round's segments for the final placement
struct DrainRec {
	int32_t node, ewald;
	int64_t src[2], fill[2];  // pool offset, offset in the node's list: PC, PP
	int64_t len[2];
};

// what a test reads of a node: the centre, and the radius' bits with the sign set for a leaf; a NaN
// for an empty node
__global__ __launch_bounds__(256) void k_walk_cls(const WalkNode* __restrict__ nodes, int64_t nn, int4* __restrict__ cls,
		int4* __restrict__ rng) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= nn) return;
	const WalkNode n = nodes[i];
	const int r = n.pend == n.pbegin ? 0x7fc00000 : (__float_as_int(n.r) & 0x7fffffff) | (n.c0 < 0 ? INT32_MIN : 0);
	cls[i] = make_int4(n.x[0], n.x[1], n.x[2], r);
	rng[i] = make_int4(n.pbegin, n.pend, n.c0, n.c1);
}

__device__ __forceinline__ double pos_d(int32_t x) {
#pragma clang fp contract(off)
	return double(x) * (1.0 / 4294967296.0) + 0.5;
}

__device__ __forceinline__ double near_sep(const double* x) {
#pragma clang fp contract(off)
	double d = 0.0;
	for (int k = 0; k < 3; k++) {
		const double ax = fabs(x[k]);
		const double o = 1.0 - ax;
		const double t = o < ax ? o : ax;
		d += t * t;
	}
	return sqrt(d);
}

// the host walk's direct_far / ewald_far (tg_tree.cpp walk_rec) for sink n (centre X) and source c
__device__ __forceinline__ bool far_test(const WalkParams& P, const WalkNode& n, const double* X, const WalkNode& c, bool ewald_kind) {
#pragma clang fp contract(off)
	double dX[3];
	for (int k = 0; k < 3; k++) dX[k] = X[k] - pos_d(c.x[k]);
	const float rsum = n.r + c.r;
	if (!ewald_kind) {
		const double dx = P.ewald ? near_sep(dX) : sqrt(dX[0] * dX[0] + dX[1] * dX[1] + dX[2] * dX[2]);
		return dx > double(rsum) * P.theta_inv && dx > double(rsum) + P.h;
	}
	const double ns = near_sep(dX);
	const double dx = 0.25 < ns ? ns : 0.25;
	if (dX[0] * dX[0] + dX[1] * dX[1] + dX[2] * dX[2] > 0.0) return dx > double(rsum) * P.theta_inv && dx > double(rsum) + P.h;
	return n.rmax < P.r_ewald;
}

// Checklist entries are classified 64 at a time by one wave, each lane one entry, in checklist
// order.  Categories: FIRST {0 cc, 1 cp range, 2 opened, 3 deferred}; DRAIN {0 pp range, 1 pc,
// 2 opened, 3 deferred}; 4: an empty node (nothing).  The count pass keeps every entry's category
// (one byte, beside the entry) for the write pass, which then places each lane's outputs by its
// rank among the lanes of the same category: the serial pass's order.  The two children of a node
// read the same checklists, so entry i keeps a category byte per child (2 i + child).
enum { CAT_SKIP = 4 };

__device__ __forceinline__ unsigned long long lanes_below(int lane) { return lane ? ~0ull >> (64 - lane) : 0ull; }

// a - b in position units as float: the wrap-around difference, or the exact one rounded once
__device__ __forceinline__ float diff_f(int a, int b, bool wrap) {
	const unsigned d = unsigned(a) - unsigned(b);
	if (wrap) return float(int(d));
	return a < b ? -float(0u - d) : float(d);
}

// The test of far_test in FP32, in position units: the squared separation against the squared
// limit.  Both carry less than 1e-6 of rounding; within 1e-5 of each other, at a zero Ewald
// separation, and where a limit is no number, the FP64 test decides (one entry in some ten
// thousand).  FP64 with its square root took twice the kernel's time.
__device__ __forceinline__ int classify(const WalkParams& P, const WalkNode& n, const int4& c, int id, bool opened, bool ewald_kind,
		bool drain) {
	const float rc = __int_as_float(c.w & 0x7fffffff);
	if (rc != rc) return CAT_SKIP;  // an empty node
	const bool leaf = c.w < 0;
	const bool wrap = P.ewald != 0 || ewald_kind;
	const float fx = diff_f(n.x[0], c.x, wrap), fy = diff_f(n.x[1], c.y, wrap), fz = diff_f(n.x[2], c.z, wrap);
	float d2 = fmaf(fz, fz, fmaf(fy, fy, fx * fx));
	bool exact = ewald_kind && d2 == 0.0f;
	if (ewald_kind) d2 = fmaxf(d2, 1152921504606846976.0f);  // a quarter box: 2^60
	const float rsum = n.r + rc;
	const float lim = fmaxf(rsum * P.theta_inv_f, rsum + P.h_f) * 4294967296.0f;
	const float l2 = lim * lim;
	bool far = d2 > l2 * 1.00001f;
	exact |= (!far && !(d2 < l2 * 0.99999f)) || !(P.theta_inv_f < 1e38f);
	if (exact) {
		const double X[3] = {pos_d(n.x[0]), pos_d(n.x[1]), pos_d(n.x[2])};
		far = far_test(P, n, X, P.nodes[id], ewald_kind);
	}
	if (drain) return opened ? 0 : far ? 1 : leaf ? 2 : 3;
	return far ? (opened ? 1 : 0) : leaf ? 2 : 3;
}

// one checklist pass of NS sinks (1, or the two children that share the list) classified and counted
// by the wave; c (4 per sink, the same in every lane) += counts
template <int NS>
__device__ __forceinline__ void count_pass(const WalkParams& P, const WalkNode* n, const int32_t* __restrict__ list, uint8_t* __restrict__ codes,
		int len, bool ewald_kind, bool drain, int (*c)[8]) {
	const int lane = threadIdx.x & 63;
	int e = lane < len ? list[lane] : 0;
	for (int b = 0; b < len; b += 64) {
		const int i = b + lane;
		const bool opened = e < 0;
		const int id = opened ? ~e : e;
		int cat[NS];
		for (int q = 0; q < NS; q++) cat[q] = CAT_SKIP;
		if (i < len) {
			const int4 cl = P.cls[id];
#pragma unroll
			for (int q = 0; q < NS; q++) cat[q] = classify(P, n[q], cl, id, opened, ewald_kind, drain);
			if (NS == 2)
				*reinterpret_cast<uint16_t*>(codes + 2 * i) = uint16_t(cat[0] | cat[NS - 1] << 8);
			else
				codes[2 * i] = uint8_t(cat[0]);
		}
		e = i + 64 < len ? list[i + 64] : 0;
#pragma unroll
		for (int q = 0; q < NS; q++)
#pragma unroll
			for (int k = 0; k < 4; k++) c[q][k] += __popcll(__ballot(cat[q] == k));
	}
}

// Four waves per work group, one unit each at a time.  The two children of a node, neighbours in the
// unit array, are classified by one wave: they read the same checklists, so an entry's node is
// gathered once for both.  Bound by the gathers and by the tests' arithmetic.
__global__ __launch_bounds__(256) void k_walk_count(WalkParams P, uint8_t* __restrict__ codes, const WalkUnit* __restrict__ units,
		const WalkStep* __restrict__ step, int32_t* __restrict__ counts) {
	const int nu = step->nu;
	const int lane = threadIdx.x & 63;
	for (int i0 = int(blockIdx.x) * 4; i0 < nu; i0 += 4 * int(gridDim.x)) {
		const int i = __builtin_amdgcn_readfirstlane(i0 + int(threadIdx.x >> 6));
		if (i >= nu) break;
		const WalkUnit u = units[i];
		int c[2][8] = {};
		bool pair = false;
		if (u.mode == MODE_FIRST) {
			// a second child is done with the unit before it where that is a first child of the same checklists
			auto shares = [](const WalkUnit& a, const WalkUnit& b) {
				return a.mode == MODE_FIRST && a.child == 0 && b.mode == MODE_FIRST && b.child == 1 && a.off_d == b.off_d && a.len_d == b.len_d &&
				       a.off_e == b.off_e && a.len_e == b.len_e;
			};
			if (i > 0 && shares(units[i - 1], u)) continue;
			WalkNode n[2];
			n[0] = P.nodes[u.node];
			if (u.child == 0 && i + 1 < nu) {
				pair = shares(u, units[i + 1]);
				if (pair) n[1] = P.nodes[units[i + 1].node];
			}
			if (pair) {
				count_pass<2>(P, n, P.lists + u.off_d, codes + 2 * u.off_d, u.len_d, false, false, c);
				int(*ce)[8] = reinterpret_cast<int(*)[8]>(&c[0][4]);
				if (P.ewald) count_pass<2>(P, n, P.lists + u.off_e, codes + 2 * u.off_e, u.len_e, true, false, ce);
			} else {
				count_pass<1>(P, n, P.lists + u.off_d, codes + 2 * u.off_d + u.child, u.len_d, false, false, c);
				int(*ce)[8] = reinterpret_cast<int(*)[8]>(&c[0][4]);
				if (P.ewald) count_pass<1>(P, n, P.lists + u.off_e, codes + 2 * u.off_e + u.child, u.len_e, true, false, ce);
			}
		} else {
			const WalkNode n = P.nodes[u.node];
			count_pass<1>(P, &n, P.lists + u.off_d, codes + 2 * u.off_d + u.child, u.len_d, u.mode == MODE_DRAIN_E, true, c);
		}
		int v = 0;
#pragma unroll
		for (int k = 0; k < 16; k++) v = lane == k ? c[k / 8][k % 8] : v;
		if (lane < (pair ? 16 : 8)) counts[8 * int64_t(i) + lane] = v;
	}
}

// One checklist pass, written by the wave from the count pass's categories: FIRST into (a: cc, b: cp)
// and next; DRAIN into (a: pp, b: pc) and next.  Next holds the opened leaves first (n_opened of
// them), then the deferred nodes' children.  Every entry writes one or two ints to its category's
// next places, so the lanes of all categories store together; the pass writes as many entries of
// each category as the count pass counted from the same bytes (the caller checks those against the
// capacities).
__device__ __forceinline__ void write_pass(const WalkParams& P, const int32_t* __restrict__ list, const uint8_t* __restrict__ codes, int len,
		bool drain, int32_t* a, int32_t* b, int32_t* next, int n_opened) {
	const int lane = threadIdx.x & 63;
	const unsigned long long below = lanes_below(lane);
	int32_t* opened = next;
	int32_t* deferred = next + n_opened;
	const int twin = drain ? 0 : 1;  // the range category: two ints an entry
	int cat_n = lane < len ? int(codes[2 * lane]) : CAT_SKIP;
	int e_n = lane < len ? list[lane] : 0;
	for (int base = 0; base < len; base += 64) {
		const int cat = cat_n, e = e_n;
		const int j = base + 64 + lane;
		cat_n = j < len ? int(codes[2 * j]) : CAT_SKIP;
		e_n = j < len ? list[j] : 0;
		const unsigned long long m0 = __ballot(cat == 0), m1 = __ballot(cat == 1), m2 = __ballot(cat == 2), m3 = __ballot(cat == 3);
		if (cat != CAT_SKIP) {
			const int id = e < 0 ? ~e : e;
			const int r = __popcll((cat == 0 ? m0 : cat == 1 ? m1 : cat == 2 ? m2 : m3) & below);
			int32_t* to = cat == 0 ? a : cat == 1 ? b : cat == 2 ? opened : deferred;
			if (cat == 3 || cat == twin) {
				const int4 g = P.rng[id];
				to += 2 * r;
				to[0] = cat == 3 ? g.z : g.x;
				to[1] = cat == 3 ? g.w : g.y;
			} else {
				to[r] = cat == 2 ? ~id : id;
			}
		}
		const int n0 = __popcll(m0), n1 = __popcll(m1);
		a += drain ? 2 * n0 : n0;
		b += drain ? n1 : 2 * n1;
		opened += __popcll(m2);
		deferred += 2 * __popcll(m3);
	}
}

// a unit's entries of each output, of its next checklists, the number of its next units, and whether
// it is a drain
__device__ __forceinline__ void unit_sizes(const int4* rng, const WalkUnit& u, const int32_t* c, int ewald, int* z) {
	for (int k = 0; k < NCOL; k++) z[k] = 0;
	const int ld = c[2] + 2 * c[3];
	if (u.mode == MODE_FIRST) {
		const int le = ewald ? c[6] + 2 * c[7] : 0;
		z[K_CC_D] = c[0];
		z[K_CP_D] = 2 * c[1];
		if (ewald) {
			z[K_CC_E] = c[4];
			z[K_CP_E] = 2 * c[5];
		}
		z[COL_NEXT] = ld + le;
		const int4 n = rng[u.node];
		if (n.z >= 0)
			z[COL_UNITS] = int(rng[n.z].y > rng[n.z].x) + int(rng[n.w].y > rng[n.w].x);
		else
			z[COL_UNITS] = int(ld > 0) + int(le > 0);
	} else {
		const bool ew = u.mode == MODE_DRAIN_E;
		z[ew ? K_PP_E : K_PP_D] = 2 * c[0];
		z[ew ? K_PC_E : K_PC_D] = c[1];
		z[COL_NEXT] = ld;
		z[COL_UNITS] = ld > 0;
		z[COL_DRAIN] = 1;
	}
}

// The tiles' sums scanned by one block, one wave per column, and the next step's extent; a step that
// would pass a capacity sets the flag and leaves no next step.
__device__ void scan_top(WalkState* S, int par, const WalkCaps& caps, int64_t* tile_base, int tiles) {
	__shared__ int64_t tot[NCOL];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const WalkStep& cur = S->st[par];
	const int nu = cur.nu;
	if (wave < NCOL) {
		int64_t carry = 0;
		for (int t0 = 0; t0 < tiles; t0 += 64) {
			const int t = t0 + lane;
			const int64_t z = t < tiles ? tile_base[int64_t(t) * NCOL + wave] : 0;
			int64_t v = z;
			for (int o = 1; o < 64; o <<= 1) {
				const int64_t w = __shfl_up(v, o, 64);
				if (lane >= o) v += w;
			}
			if (t < tiles) tile_base[int64_t(t) * NCOL + wave] = carry + v - z;
			carry += __shfl(v, 63, 64);
		}
		if (lane == 0) tot[wave] = carry;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		WalkStep nx;
		bool over = tot[COL_NEXT] > caps.lists || tot[COL_UNITS] > caps.units || cur.drains + tot[COL_DRAIN] > caps.drains;
		for (int k = 0; k < K_N; k++) {
			nx.base[k] = cur.base[k] + tot[k];
			over |= nx.base[k] > caps.out[k];
		}
		int fl = S->flags;
		if (over) fl |= WALK_OVERFLOW;
		if (tot[COL_NEXT] > INT32_MAX || tot[COL_UNITS] > INT32_MAX) fl |= WALK_TOO_LONG;
		nx.nu = fl ? 0 : int32_t(tot[COL_UNITS]);
		nx.pad = 0;
		nx.in_len = tot[COL_NEXT];
		nx.drains = cur.drains + tot[COL_DRAIN];
		S->st[1 - par] = nx;
		S->flags = fl;
		if (nu > 0) {
			if (S->steps < LOG_STEPS) S->log_nu[S->steps] = nu;
			S->steps++;
			if (nx.in_len > S->max_lists) S->max_lists = nx.in_len;
			if (nu > S->max_units) S->max_units = nu;
		}
	}
}

// Offsets of every unit's sizes, per column: within its tile of 1024 units (loc), and of every tile
// (tile_base), both exclusive.  Launched as one block, it scans the tiles' sums too; as several,
// k_walk_scan_top follows (a last-block scan behind a device-wide fence took 15 us of small steps).
__global__ __launch_bounds__(SCAN_TILE) void k_walk_scan(const int4* __restrict__ rng, const WalkUnit* __restrict__ units,
		const int32_t* __restrict__ counts, int ewald, WalkState* __restrict__ S, int par, WalkCaps caps, int32_t* __restrict__ loc,
		int64_t* __restrict__ tile_base) {
	__shared__ int wsum[NCOL][SCAN_TILE / 64];
	const int nu = S->st[par].nu;
	const int tiles = (nu + SCAN_TILE - 1) / SCAN_TILE;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
		const int i = t * SCAN_TILE + int(threadIdx.x);
		int z[NCOL], x[NCOL];
		for (int k = 0; k < NCOL; k++) z[k] = 0;
		if (i < nu) {
			int c[8];
			for (int k = 0; k < 8; k++) c[k] = counts[8 * int64_t(i) + k];
			unit_sizes(rng, units[i], c, ewald, z);
		}
#pragma unroll
		for (int k = 0; k < NCOL; k++) {
			int v = z[k];
			for (int o = 1; o < 64; o <<= 1) {
				const int w = __shfl_up(v, o, 64);
				if (lane >= o) v += w;
			}
			x[k] = v - z[k];
			if (lane == 63) wsum[k][wave] = v;
		}
		__syncthreads();
		if (threadIdx.x < NCOL) {
			int64_t a = 0;
			for (int w = 0; w < SCAN_TILE / 64; w++) {
				const int v = wsum[threadIdx.x][w];
				wsum[threadIdx.x][w] = int(a);
				a += v;
			}
			tile_base[int64_t(t) * NCOL + threadIdx.x] = a;  // the tile's sum, until the tiles are scanned
			if (a > INT32_MAX) atomicOr(&S->flags, WALK_TOO_LONG);
		}
		__syncthreads();
		if (i < nu)
			for (int k = 0; k < NCOL; k++) loc[int64_t(i) * NCOL + k] = x[k] + wsum[k][wave];
		__syncthreads();
	}
	if (gridDim.x == 1) scan_top(S, par, caps, tile_base, tiles);
}

__global__ __launch_bounds__(SCAN_TILE) void k_walk_scan_top(WalkState* __restrict__ S, int par, WalkCaps caps, int64_t* __restrict__ tile_base) {
	scan_top(S, par, caps, tile_base, (S->st[par].nu + SCAN_TILE - 1) / SCAN_TILE);
}

struct WalkPools {
	int32_t* out[K_N];   // output pools, appended step by step
	int64_t cap[K_N + 1];
	int32_t* next;       // the next step's checklists
	WalkUnit* next_units;
	int64_t units_cap;
	DrainRec* drains;
	int64_t drains_cap;
	int64_t* node_len;   // K_N x (nn + 1): entries of each node's lists so far
};

// what a unit's wave and its thread below both need of its offsets
struct UnitAt {
	const int32_t* loc;
	const int64_t* base;
	__device__ __forceinline__ UnitAt(const int32_t* l, const int64_t* b, int i) : loc(l + int64_t(i) * NCOL), base(b + int64_t(i / SCAN_TILE) * NCOL) {}
	__device__ __forceinline__ int64_t operator()(int k) const { return base[k] + loc[k]; }
};

// The first unit_blocks blocks take one unit per thread: the next step's units (an interior node's
// first pass hands its two next lists to its non-empty children, a leaf's to its drains; a drain
// round with a non-empty next list continues), and its share of its node's list lengths.  Only
// the one unit of (node, kind) with entries in a step touches that length (one first pass, one
// direct and one Ewald drain round a step at most).  The other blocks write the units' outputs and
// next checklists, four waves per block, one unit each at a time.
__global__ __launch_bounds__(256) void k_walk_write(WalkParams P, const uint8_t* __restrict__ codes, const WalkUnit* __restrict__ units,
		const int32_t* __restrict__ counts, const int32_t* __restrict__ loc, const int64_t* __restrict__ tile_base, int64_t nn,
		WalkState* __restrict__ S, int par, WalkPools W, int unit_blocks) {
	if (S->flags) return;
	const WalkStep& cur = S->st[par];
	const int nu = cur.nu;
	if (int(blockIdx.x) < unit_blocks) {
		for (int i = int(blockIdx.x) * 256 + int(threadIdx.x); i < nu; i += 256 * unit_blocks) {
			const WalkUnit u = units[i];
			const int32_t* c = counts + 8 * int64_t(i);
			const UnitAt off(loc, tile_base, i);
			const int64_t nb = off(COL_NEXT);
			int64_t q = off(COL_UNITS);
			auto emit = [&](WalkUnit w) {
				if (q < W.units_cap)
					W.next_units[q] = w;
				else
					S->flags = WALK_DISAGREE;
				q++;
			};
			const int ld = c[2] + 2 * c[3];
			if (u.mode == MODE_FIRST) {
				const int le = P.ewald ? c[6] + 2 * c[7] : 0;
				W.node_len[int64_t(K_CC_D) * (nn + 1) + u.node] = c[0];
				W.node_len[int64_t(K_CP_D) * (nn + 1) + u.node] = 2 * c[1];
				if (P.ewald) {
					W.node_len[int64_t(K_CC_E) * (nn + 1) + u.node] = c[4];
					W.node_len[int64_t(K_CP_E) * (nn + 1) + u.node] = 2 * c[5];
				}
				const int4 n = P.rng[u.node];
				if (n.z >= 0) {
					if (P.rng[n.z].y > P.rng[n.z].x) emit(WalkUnit{n.z, MODE_FIRST, ld, le, nb, nb + ld, 0, 0});
					if (P.rng[n.w].y > P.rng[n.w].x) emit(WalkUnit{n.w, MODE_FIRST, ld, le, nb, nb + ld, 1, 0});
				} else {
					if (ld > 0) emit(WalkUnit{u.node, MODE_DRAIN_D, ld, 0, nb, 0, 0, 0});
					if (le > 0) emit(WalkUnit{u.node, MODE_DRAIN_E, le, 0, nb + ld, 0, 0, 0});
				}
			} else {
				if (ld > 0) emit(WalkUnit{u.node, u.mode, ld, 0, nb, 0, 0, 0});
				const bool ew = u.mode == MODE_DRAIN_E;
				const int kc = ew ? K_PC_E : K_PC_D, kp = ew ? K_PP_E : K_PP_D;
				int64_t* lc = W.node_len + int64_t(kc) * (nn + 1) + u.node;
				int64_t* lp = W.node_len + int64_t(kp) * (nn + 1) + u.node;
				DrainRec r;
				r.node = u.node;
				r.ewald = ew;
				r.src[0] = cur.base[kc] + off(kc);
				r.src[1] = cur.base[kp] + off(kp);
				r.fill[0] = *lc;
				r.fill[1] = *lp;
				r.len[0] = c[1];
				r.len[1] = 2 * c[0];
				*lc = r.fill[0] + r.len[0];
				*lp = r.fill[1] + r.len[1];
				const int64_t d = cur.drains + off(COL_DRAIN);
				if (d < W.drains_cap)
					W.drains[d] = r;
				else
					S->flags = WALK_DISAGREE;
			}
		}
		return;
	}
	const int wave = (int(blockIdx.x) - unit_blocks) * 4 + int(threadIdx.x >> 6);
	for (int i0 = wave; i0 < nu; i0 += 4 * (int(gridDim.x) - unit_blocks)) {
		const int i = __builtin_amdgcn_readfirstlane(i0);
		const WalkUnit u = units[i];
		const int32_t* c = counts + 8 * int64_t(i);
		const UnitAt off(loc, tile_base, i);
		const int64_t nb = off(COL_NEXT);
		const int ld = c[2] + 2 * c[3];
		// the unit's runs of kind ka (na ints), kind kb (nbk ints) and next entries lie inside their buffers
		auto fits = [&](int ka, int na, int kb, int nbk, int64_t next_end) {
			const bool ok = cur.base[ka] + off(ka) + na <= W.cap[ka] && cur.base[kb] + off(kb) + nbk <= W.cap[kb] && next_end <= W.cap[K_N];
			if (!ok) S->flags = WALK_DISAGREE;
			return ok;
		};
		if (u.mode == MODE_FIRST) {
			if (fits(K_CC_D, c[0], K_CP_D, 2 * c[1], nb + ld))
				write_pass(P, P.lists + u.off_d, codes + 2 * u.off_d + u.child, u.len_d, false, W.out[K_CC_D] + cur.base[K_CC_D] + off(K_CC_D),
						W.out[K_CP_D] + cur.base[K_CP_D] + off(K_CP_D), W.next + nb, c[2]);
			if (P.ewald && fits(K_CC_E, c[4], K_CP_E, 2 * c[5], nb + ld + c[6] + 2 * int64_t(c[7])))
				write_pass(P, P.lists + u.off_e, codes + 2 * u.off_e + u.child, u.len_e, false, W.out[K_CC_E] + cur.base[K_CC_E] + off(K_CC_E),
						W.out[K_CP_E] + cur.base[K_CP_E] + off(K_CP_E), W.next + nb + ld, c[6]);
		} else {
			const bool ew = u.mode == MODE_DRAIN_E;
			const int kc = ew ? K_PC_E : K_PC_D, kp = ew ? K_PP_E : K_PP_D;
			if (fits(kp, 2 * c[0], kc, c[1], nb + ld))
				write_pass(P, P.lists + u.off_d, codes + 2 * u.off_d + u.child, u.len_d, true, W.out[kp] + cur.base[kp] + off(kp),
						W.out[kc] + cur.base[kc] + off(kc), W.next + nb, c[2]);
		}
	}
}

// the walk's start: the root's checklists, {root} for both kinds, and its first pass
__global__ __launch_bounds__(64) void k_walk_root(const WalkNode* __restrict__ nodes, int ewald, WalkState* __restrict__ S,
		WalkUnit* __restrict__ units, int32_t* __restrict__ lists) {
	int32_t* w = reinterpret_cast<int32_t*>(S);
	for (int i = threadIdx.x; i < int(sizeof(WalkState) / 4); i += 64) w[i] = 0;
	__syncthreads();
	if (threadIdx.x == 0) {
		lists[0] = lists[1] = 0;
		units[0] = WalkUnit{0, MODE_FIRST, 1, ewald ? 1 : 0, 0, 1, 0, 0};
		S->st[0].nu = nodes[0].pend > nodes[0].pbegin ? 1 : 0;
		S->st[0].in_len = 2;
	}
}

// the scan of all kinds' node lengths as one sequence, less each kind's start
__global__ __launch_bounds__(256) void k_walk_colfix(const int64_t* __restrict__ scan, int64_t np, int64_t* __restrict__ ptr) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i < K_N * np) ptr[i] = scan[i] - scan[i / np * np];
}

// the drain rounds' segments into the node-order PC and PP lists: one wave per round
__global__ __launch_bounds__(256) void k_walk_place(const DrainRec* __restrict__ recs, int64_t nrec, const int64_t* __restrict__ ptr,
		int64_t nn, WalkPools src, WalkPools dst) {
	const int lane = threadIdx.x & 63;
	for (int64_t i = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6); i < nrec; i += 4 * int64_t(gridDim.x)) {
		const DrainRec r = recs[i];
		for (int h = 0; h < 2; h++) {
			const int k = (h ? K_PP_D : K_PC_D) + (r.ewald ? K_PC_E - K_PC_D : 0);
			const int32_t* from = src.out[k] + r.src[h];
			int32_t* to = dst.out[k] + ptr[int64_t(k) * (nn + 1) + r.node] + r.fill[h];
			for (int64_t t = lane; t < r.len[h]; t += 64) to[t] = from[t];
		}
	}
}

// a device buffer that grows, keeping its contents where asked
template <class T>
struct Pool {
	T* p = nullptr;
	int64_t cap = 0;
	hipError_t reserve(int64_t n, hipStream_t s, bool keep = true) {
		if (n <= cap) return hipSuccess;
		int64_t nc = std::max<int64_t>(n, cap * 2);
		nc = std::max<int64_t>(nc, 1024);
		T* q = nullptr;
		hipError_t e = dev_malloc(&q, size_t(nc) * sizeof(T));
		if (e != hipSuccess) return e;
		if (p) {
			// the stream may still read the old buffer
			if (keep) e = hipMemcpyAsync(q, p, size_t(cap) * sizeof(T), hipMemcpyDeviceToDevice, s);
			if (e == hipSuccess) e = hipStreamSynchronize(s);
			dev_free(p);
			p = nullptr;
		}
		if (e != hipSuccess) {
			dev_free(q);
			cap = 0;
			return e;
		}
		p = q;
		cap = nc;
		return hipSuccess;
	}
	void release() {
		if (p) dev_free(p);
		p = nullptr;
		cap = 0;
	}
};

}  // namespace

static double wall() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

void DeviceLists::release() {
	if (nodes) dev_free(nodes);
	if (ptr_all) dev_free(ptr_all);
	for (auto& v : val)
		if (v) dev_free(v);
	*this = DeviceLists();
}

hipError_t device_walk(Tree& T, int device, hipStream_t s, std::string& err, double* t_out, DeviceLists* keep, WalkNode* given,
		int64_t given_nn, WalkHint* hint, std::vector<void*>& later) {
	static_assert(sizeof(WalkHint::out) / sizeof(int64_t) == K_N, "one hint per output kind");
	double tw[4] = {wall(), 0, 0, 0};
	const int64_t nn = given ? given_nn : int64_t(T.nodes.size());
	const int64_t np = nn + 1;
	hipError_t e = hipSuccess;
	WalkNode* dev_nodes = given;  // owned from here on
	int64_t* dev_ptr = nullptr;
	Pool<int4> cls, rng;
	Pool<WalkState> state;
	Pool<int64_t> node_len, node_scan, tile_base;
	Pool<int32_t> lists_in, lists_out, out[K_N], fin[K_N], counts, loc;
	Pool<uint8_t> codes, scan_tmp;  // codes: the category of every checklist entry of the step, byte 2 i + child for entry i
	Pool<WalkUnit> units_in, units_out;
	Pool<DrainRec> drains;
	hvec<WalkNode> wn;
	WalkState h{};  // host copy of the state
	WalkParams P{};
	hipError_t pending = hipSuccess;
	size_t scan_need = 0;
#define WCHK(call)                                     \
	do {                                               \
		e = (call);                                    \
		if (e != hipSuccess) {                         \
			err = std::string(#call) + ": " + hipGetErrorString(e); \
			goto done;                                 \
		}                                              \
	} while (0)
#define WLAUNCH(name)                                                                       \
	do {                                                                                    \
		e = hipGetLastError();                                                              \
		if (e != hipSuccess) {                                                              \
			err = std::string("launch ") + name + ": " + hipGetErrorString(e);              \
			if (pending != hipSuccess) err += std::string(" (pending before the walk: ") + hipGetErrorString(pending) + ")"; \
			goto done;                                                                      \
		}                                                                                   \
	} while (0)
	pending = hipGetLastError();  // an error left by an earlier call is not the walk's
	WCHK(hipSetDevice(device));
	if (!given) {
		wn.resize(size_t(std::max<int64_t>(nn, 1)));
		walk_nodes(T, wn.data());
		WCHK(dev_malloc(&dev_nodes, wn.size() * sizeof(WalkNode)));
		WCHK(hipMemcpyAsync(dev_nodes, wn.data(), wn.size() * sizeof(WalkNode), hipMemcpyHostToDevice, s));
		WCHK(hipStreamSynchronize(s));
	}
	WCHK(cls.reserve(std::max<int64_t>(nn, 1), s));
	WCHK(rng.reserve(std::max<int64_t>(nn, 1), s));
	WCHK(state.reserve(1, s));
	WCHK(node_len.reserve(K_N * np, s));
	WCHK(node_scan.reserve(K_N * np, s));
	WCHK(dev_malloc(&dev_ptr, size_t(K_N * np) * sizeof(int64_t)));
	P.nodes = dev_nodes;
	P.cls = cls.p;
	P.rng = rng.p;
	P.theta_inv = 1.0 / T.P.theta;
	P.h = T.P.soft_len;
	P.theta_inv_f = float(P.theta_inv);
	P.h_f = float(P.h);
	P.r_ewald = float(2.0 * T.P.theta * std::pow(1.0e-3 / 8.0, 1.0 / 3.0));  // src/tree.cpp:403-404
	P.ewald = T.P.ewald ? 1 : 0;
	if (nn > 0) {
		hipLaunchKernelGGL(k_walk_cls, dim3(unsigned((nn + 255) / 256)), dim3(256), 0, s, dev_nodes, nn, cls.p, rng.p);
		WLAUNCH("k_walk_cls");
	}
	tw[1] = wall();
	{
		// Enqueued whole where the last walk's sizes are known (an eighth more is allowed for), with a wait
		// per step otherwise, or again where a size was passed.
		bool sized = hint && hint->steps > 0;
		const bool any = nn > 0;
		for (int attempt = 0; any; attempt++) {
			auto room = [](int64_t v) { return v + v / 8 + 64; };
			if (hint) {
				for (int k = 0; k < K_N; k++)
					if (hint->out[k] > 0) WCHK(out[k].reserve(room(hint->out[k]), s, false));
				if (hint->lists > 0) {
					WCHK(lists_in.reserve(room(hint->lists), s, false));
					WCHK(lists_out.reserve(room(hint->lists), s, false));
				}
				if (hint->drains > 0) WCHK(drains.reserve(room(hint->drains), s, false));
			}
			const int64_t nu0 = std::max<int64_t>(hint ? room(hint->units) : 0, 1024);
			auto unit_room = [&](int64_t nu) -> hipError_t {
				hipError_t r = units_in.reserve(nu, s);
				if (r == hipSuccess) r = counts.reserve(8 * nu, s, false);
				if (r == hipSuccess) r = loc.reserve(NCOL * nu, s, false);
				if (r == hipSuccess) r = tile_base.reserve(NCOL * ((nu + SCAN_TILE - 1) / SCAN_TILE), s, false);
				return r;
			};
			WCHK(unit_room(nu0));
			WCHK(units_out.reserve(nu0, s, false));
			WCHK(lists_in.reserve(2, s, false));
			WCHK(lists_out.reserve(2, s, false));
			WCHK(drains.reserve(1, s, false));
			for (auto& o : out) WCHK(o.reserve(1, s, false));
			WCHK(codes.reserve(2 * std::max(lists_in.cap, lists_out.cap), s, false));
			WCHK(hipMemsetAsync(node_len.p, 0, size_t(K_N * np) * sizeof(int64_t), s));
			hipLaunchKernelGGL(k_walk_root, dim3(1), dim3(64), 0, s, dev_nodes, P.ewald, state.p, units_in.p, lists_in.p);
			WLAUNCH("k_walk_root");
			int par = 0;
			bool again = false;
			for (int step = 0;; step++, par = 1 - par) {
				const bool wait = !sized || step >= hint->steps;
				if (sized && step == hint->steps) {
					// the steps the last walk took are enqueued: most often nothing is left
					WCHK(hipMemcpyAsync(&h, state.p, sizeof(h), hipMemcpyDeviceToHost, s));
					WCHK(hipStreamSynchronize(s));
					if (h.flags || h.st[par].nu == 0) break;
				}
				int64_t bound = 1;
				if (wait)
					bound = step == 0 ? 1 : h.st[par].nu;
				else
					bound = room(step < LOG_STEPS ? hint->step_units[size_t(step)] : hint->units);
				P.lists = lists_in.p;
				const unsigned g = unsigned(std::min<int64_t>((bound + 3) / 4, 1 << 18));
				// up to four tiles by one block, whose last barrier saves a launch
				const unsigned gs = bound <= 4 * SCAN_TILE ? 1 : unsigned(std::min<int64_t>((bound + SCAN_TILE - 1) / SCAN_TILE, 1024));
				const unsigned gu = unsigned(std::min<int64_t>((bound + 255) / 256, 1 << 12));
				hipLaunchKernelGGL(k_walk_count, dim3(g), dim3(256), 0, s, P, codes.p, units_in.p, &state.p->st[par], counts.p);
				WLAUNCH("k_walk_count");
				WalkCaps caps;
				for (int k = 0; k < K_N; k++) caps.out[k] = wait ? INT64_MAX : out[k].cap;
				caps.lists = wait ? INT64_MAX : std::min(lists_out.cap, codes.cap / 2);
				caps.units = wait ? INT64_MAX : std::min(std::min(units_out.cap, units_in.cap), std::min(counts.cap / 8, loc.cap / NCOL));
				caps.units = wait ? INT64_MAX : std::min(caps.units, tile_base.cap / NCOL * SCAN_TILE);
				caps.drains = wait ? INT64_MAX : drains.cap;
				hipLaunchKernelGGL(k_walk_scan, dim3(gs), dim3(SCAN_TILE), 0, s, rng.p, units_in.p, counts.p, P.ewald, state.p, par, caps, loc.p,
						tile_base.p);
				WLAUNCH("k_walk_scan");
				if (gs > 1) {
					hipLaunchKernelGGL(k_walk_scan_top, dim3(1), dim3(SCAN_TILE), 0, s, state.p, par, caps, tile_base.p);
					WLAUNCH("k_walk_scan_top");
				}
				if (wait) {
					WCHK(hipMemcpyAsync(&h, state.p, sizeof(h), hipMemcpyDeviceToHost, s));
					WCHK(hipStreamSynchronize(s));
					if (h.flags) break;
					const WalkStep& nx = h.st[1 - par];
					for (int k = 0; k < K_N; k++) WCHK(out[k].reserve(std::max<int64_t>(nx.base[k], 1), s));
					WCHK(lists_out.reserve(std::max<int64_t>(nx.in_len, 1), s, false));
					WCHK(units_out.reserve(std::max<int64_t>(nx.nu, 1), s, false));
					WCHK(drains.reserve(std::max<int64_t>(nx.drains, 1), s));
				}
				WalkPools W{};
				for (int k = 0; k < K_N; k++) {
					W.out[k] = out[k].p;
					W.cap[k] = out[k].cap;
				}
				W.cap[K_N] = lists_out.cap;
				W.next = lists_out.p;
				W.next_units = units_out.p;
				W.units_cap = units_out.cap;
				W.drains = drains.p;
				W.drains_cap = drains.cap;
				W.node_len = node_len.p;
				hipLaunchKernelGGL(k_walk_write, dim3(g + gu), dim3(256), 0, s, P, codes.p, units_in.p, counts.p, loc.p, tile_base.p, nn, state.p, par, W,
						int(gu));
				WLAUNCH("k_walk_write");
				std::swap(lists_in, lists_out);
				std::swap(units_in, units_out);
				if (wait) {
					const WalkStep& nx = h.st[1 - par];
					if (nx.nu == 0) {
						par = 1 - par;
						break;
					}
					// the next step's per-unit and per-entry buffers (the last step's kernels may still read the old)
					WCHK(unit_room(nx.nu));
					WCHK(codes.reserve(2 * nx.in_len, s, false));
				}
			}
			// the write passes' own check, and the totals (a wait per step read them before the last write)
			WCHK(hipMemcpyAsync(&h, state.p, sizeof(h), hipMemcpyDeviceToHost, s));
			WCHK(hipStreamSynchronize(s));
			if (h.flags & WALK_TOO_LONG) {
				err = "walk checklists exceed 2^31 entries";
				e = hipErrorInvalidValue;
				goto done;
			}
			again = sized && (h.flags & WALK_OVERFLOW);
			if (again) {
				sized = false;
				continue;
			}
			if (h.flags) {
				err = "device walk: a write pass disagreed with its count pass";
				e = hipErrorUnknown;
				goto done;
			}
			break;
		}
	}
	tw[2] = wall();
	{
		// the fills only grow: the later of the two parities
		int64_t tot[K_N];
		for (int k = 0; k < K_N; k++) tot[k] = std::max(h.st[0].base[k], h.st[1].base[k]);
		const int64_t nrec = std::max(h.st[0].drains, h.st[1].drains);
		if (hint) {
			for (int k = 0; k < K_N; k++) hint->out[k] = tot[k];
			hint->lists = h.max_lists;
			hint->units = h.max_units;
			hint->drains = nrec;
			hint->steps = h.steps;
			hint->step_units.assign(h.log_nu, h.log_nu + std::min<int>(h.steps, LOG_STEPS));
		}
		// node-order pointers per kind, and the drain rounds' segments placed
		WCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_need, node_len.p, node_scan.p, K_N * np, s));
		WCHK(scan_tmp.reserve(int64_t(scan_need), s, false));
		if (nn == 0) WCHK(hipMemsetAsync(node_len.p, 0, size_t(K_N * np) * sizeof(int64_t), s));
		WCHK(hipcub::DeviceScan::ExclusiveSum(scan_tmp.p, scan_need, node_len.p, node_scan.p, K_N * np, s));
		hipLaunchKernelGGL(k_walk_colfix, dim3(unsigned((K_N * np + 255) / 256)), dim3(256), 0, s, node_scan.p, np, dev_ptr);
		WLAUNCH("k_walk_colfix");
		WalkPools src{}, dst{};
		for (int k = K_PC_D; k < K_N; k++) {
			WCHK(fin[k].reserve(std::max<int64_t>(tot[k], 1), s, false));
			src.out[k] = out[k].p;
			dst.out[k] = fin[k].p;
		}
		if (nrec > 0) {
			hipLaunchKernelGGL(k_walk_place, dim3(unsigned(std::min<int64_t>((nrec + 3) / 4, 1 << 18))), dim3(256), 0, s, drains.p, nrec, dev_ptr, nn,
					src, dst);
			WLAUNCH("k_walk_place");
		}
		T.lists = Lists();
		T.census = Census();
		// the caller's DeviceLists takes the arrays: the node kinds' pools as they are
		keep->release();
		keep->nn = nn;
		keep->ptr_all = dev_ptr;
		dev_ptr = nullptr;
		keep->nodes = dev_nodes;
		dev_nodes = nullptr;
		for (int k = 0; k < K_N; k++) {
			Pool<int32_t>& p = k < K_PC_D ? out[k] : fin[k];
			WCHK(p.reserve(1, s, false));
			keep->val[k] = p.p;
			keep->len[k] = tot[k];
			p.p = nullptr;
			p.cap = 0;
		}
		tw[3] = wall();
		if (t_out) {
			for (int k = 0; k < 3; k++) t_out[k] = tw[k + 1] - tw[k];
			t_out[3] = 0.0;
		}
	}
done:
#undef WCHK
#undef WLAUNCH
	// the stream may still read the working buffers: freed now after an error, by the caller otherwise
	if (e != hipSuccess) (void) hipStreamSynchronize(s);
	std::vector<void*> mine = {dev_nodes, dev_ptr, cls.p, rng.p, state.p, node_len.p, node_scan.p, tile_base.p, lists_in.p, lists_out.p, counts.p, loc.p,
			codes.p, scan_tmp.p, units_in.p, units_out.p, drains.p};
	for (auto& p : out) mine.push_back(p.p);
	for (auto& p : fin) mine.push_back(p.p);
	for (void* p : mine) {
		if (!p) continue;
		if (e != hipSuccess)
			dev_free(p);
		else
			later.push_back(p);
	}
	return e;
}

}  // namespace tg
