// tg_scan.hpp -- exclusive scans of several int64 arrays in one go.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// up to MAX arrays of their own lengths, scanned together
struct ScanSet {
	static constexpr int MAX = 24;
	const int64_t* in[MAX];
	int64_t* out[MAX];
	int64_t n[MAX];
	int cols = 0;
	void add(const int64_t* i, int64_t* o, int64_t len) {
		in[cols] = i;
		out[cols] = o;
		n[cols++] = len;
	}
};

// int64 words of workspace that scan_columns needs for S
int64_t scan_workspace(const ScanSet& S);

// out[c][i] = in[c][0] + ... + in[c][i - 1] for every column and its sum into tot[c] (device memory);
// in and out may not overlap.  One launch where every column fits a tile of 4,096, else three.
hipError_t scan_columns(const ScanSet& S, int64_t* work, int64_t* tot, hipStream_t s);

}  // namespace tg
