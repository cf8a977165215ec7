// tg_fof.hpp -- friends-of-friends groups on the device (tg_fof.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "tg_devtree.hpp"
#include "tg_fof.h"
#include "tg_tree.hpp"

namespace tg {

// what the group search reads of a solver: the tree on the device where that is current (dtree), else
// on the host (tree); the rest is device memory (particles x, y, z, mass bits and input indices in tree
// order, non-empty leaves as (node, first particle, end, -))
struct FofSource {
	const DeviceTree* dtree = nullptr;
	const Tree* tree = nullptr;
	const int4* parts = nullptr;
	const int64_t* order = nullptr;
	const int4* leaf_items = nullptr;
	int n_leaf_items = 0;
	int64_t n = 0, nn = 0;
};

// group of every particle, the smallest tree-order index of its friends-of-friends component or
// TG_FOF_NONE for a particle linked to no other: into group_tree (device, tree order) and group_input
// (host, input order); n_groups: components of two or more
hipError_t fof_device(const FofSource& F, double link_len, hipStream_t s, uint64_t* group_tree, uint64_t* group_input, int64_t* n_groups,
		std::string& err);

// the catalog of the groups in group_tree (tg_groups.cpp): groups of at least min_n members, by id
int group_catalog(const Tree& T, const std::vector<uint64_t>& group_tree, const float* v_input, double a, int32_t min_n, tg_group* out,
		int64_t capacity, int64_t* n_out);

}  // namespace tg
