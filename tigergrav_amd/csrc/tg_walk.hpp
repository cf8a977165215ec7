// tg_walk.hpp -- the dual-tree walk (interaction lists) on the device.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "tg_tree.hpp"

namespace tg {

// a node as the device walk reads it
struct WalkNode {
	int32_t pbegin, pend, c0, c1;
	int32_t x[3];
	float r;
	float rmax;  // span of the node's particle box (the sink rmax of the Ewald self test)
};

// fills out[i] for every node of T (host, OpenMP; tg_upload.cpp)
void walk_nodes(const Tree& T, WalkNode* out);

// The walk's lists left in device memory: node-order CSR per kind, kinds in the order cc_d, cp_d,
// cc_e, cp_e, pc_d, pp_d, pc_e, pp_e (node kinds hold node ids or [begin, end) particle ranges as
// the host Lists do).  The table of nodes the walk read stays too.  Every array is owned here.
struct DeviceLists {
	WalkNode* nodes = nullptr;   // nn nodes
	int64_t* ptr_all = nullptr;  // 8 x (nn + 1) pointers, kind-major
	int32_t* val[8] = {};        // values per kind
	int64_t len[8] = {};         // values per kind (ints)
	int64_t nn = 0;
	const int64_t* ptr(int k) const { return ptr_all + int64_t(k) * (nn + 1); }
	void release();
};

// The sizes a walk reached, for the next one's working buffers and grids.
struct WalkHint {
	int64_t out[8] = {};    // entries of each output kind
	int64_t lists = 0;      // the longest checklist set of a step
	int64_t units = 0;      // the most units of a step
	int64_t drains = 0;     // drain rounds
	int steps = 0;          // steps (0: no walk yet)
	std::vector<int32_t> step_units;  // units of the first steps
};

// Tree::walk on the device: exactly the lists the host walk builds (same entries, same order), left
// on the device in *keep (released first); T supplies the parameters, its lists are left empty and
// its census zero.  Returns hipSuccess or the first HIP error; err names it.  t, if given,
// receives the seconds spent in set-up, the walk steps and list assembly (enqueued), and zero.
// With nodes (a device table of nn nodes, which device_walk then owns and frees or hands to keep),
// the tree itself may be on the device only.
// With hint, the walk's working buffers start at the sizes *hint holds (those the caller's last
// walk reached, which this walk writes back) and its steps are enqueued without a host wait; a walk
// that passes one of those sizes runs again, waiting for each step's (200,000 Plummer particles after
// 3,000: 3.9 ms to set, after 200,000 2.6).
// The work may still be running on s when this returns: the caller frees the blocks added to `later`
// (dev_free) once s has drained.
hipError_t device_walk(Tree& T, int device, hipStream_t s, std::string& err, double* t, DeviceLists* keep, WalkNode* nodes, int64_t nn,
		WalkHint* hint, std::vector<void*>& later);

}  // namespace tg
