// tg_scan.hip -- exclusive scans of several int64 arrays in one go (tg_scan.hpp).
//
// The rebuild scans some thirty short arrays (a library scan is two launches each, which at a few
// thousand nodes is all they cost): here a launch covers every array, a tile of 4,096 elements per
// block, and only sets with a longer array take the two launches that add up the tiles.  Bound by
// launches below about 100,000 elements, by memory above (32 bytes an element).
#include "tg_scan.hpp"

#include <algorithm>

namespace tg {
namespace {

constexpr int TILE = 4096, THREADS = 1024, PER = TILE / THREADS;

// exclusive prefix of one value per thread over the block; total in every thread
__device__ __forceinline__ int64_t block_scan(int64_t v, int64_t& total) {
	__shared__ int64_t wsum[THREADS / 64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	int64_t x = v;
	for (int o = 1; o < 64; o <<= 1) {
		const int64_t w = __shfl_up(x, o, 64);
		if (lane >= o) x += w;
	}
	__syncthreads();  // the last call's sums are read
	if (lane == 63) wsum[wave] = x;
	__syncthreads();
	int64_t before = 0, all = 0;
	for (int w = 0; w < THREADS / 64; w++) {
		if (w < wave) before += wsum[w];
		all += wsum[w];
	}
	total = all;
	return before + x - v;
}

// tile t of column c: its own scan, its sum into work; a column of one tile is done
__global__ __launch_bounds__(THREADS) void k_scan_tiles(ScanSet S, int64_t* __restrict__ work, int64_t* __restrict__ tot, int tiles_max) {
	const int c = blockIdx.y, t = blockIdx.x;
	const int64_t n = S.n[c], tiles = (n + TILE - 1) / TILE;
	if (t >= tiles && t > 0) return;
	const int64_t i0 = int64_t(t) * TILE + int64_t(threadIdx.x) * PER;
	int64_t v[PER], sum = 0;
	for (int k = 0; k < PER; k++) {
		v[k] = i0 + k < n ? S.in[c][i0 + k] : 0;
		sum += v[k];
	}
	int64_t all;
	int64_t x = block_scan(sum, all);
	for (int k = 0; k < PER; k++) {
		if (i0 + k < n) S.out[c][i0 + k] = x;
		x += v[k];
	}
	if (threadIdx.x == 0) {
		work[int64_t(c) * tiles_max + t] = all;
		if (tiles <= 1) tot[c] = all;
	}
}

// the sums of each column's tiles scanned in place, its total
__global__ __launch_bounds__(THREADS) void k_scan_tops(ScanSet S, int64_t* __restrict__ work, int64_t* __restrict__ tot, int tiles_max) {
	const int c = blockIdx.x;
	const int64_t tiles = (S.n[c] + TILE - 1) / TILE;
	if (tiles <= 1) return;
	int64_t carry = 0;
	for (int64_t t0 = 0; t0 < tiles; t0 += THREADS) {
		const int64_t t = t0 + threadIdx.x;
		const int64_t v = t < tiles ? work[int64_t(c) * tiles_max + t] : 0;
		int64_t all;
		const int64_t x = block_scan(v, all);
		if (t < tiles) work[int64_t(c) * tiles_max + t] = carry + x;
		carry += all;
	}
	if (threadIdx.x == 0) tot[c] = carry;
}

__global__ __launch_bounds__(THREADS) void k_scan_add(ScanSet S, const int64_t* __restrict__ work, int tiles_max) {
	const int c = blockIdx.y, t = blockIdx.x;
	const int64_t n = S.n[c];
	if (t == 0 || int64_t(t) * TILE >= n) return;
	const int64_t add = work[int64_t(c) * tiles_max + t];
	for (int k = 0; k < PER; k++) {
		const int64_t i = int64_t(t) * TILE + int64_t(k) * THREADS + threadIdx.x;
		if (i < n) S.out[c][i] += add;
	}
}

int64_t tiles_of(const ScanSet& S) {
	int64_t m = 1;
	for (int c = 0; c < S.cols; c++) m = std::max(m, (S.n[c] + TILE - 1) / TILE);
	return m;
}

}  // namespace

int64_t scan_workspace(const ScanSet& S) { return std::max(1, S.cols) * tiles_of(S); }

hipError_t scan_columns(const ScanSet& S, int64_t* work, int64_t* tot, hipStream_t s) {
	if (S.cols == 0) return hipSuccess;
	const int64_t tiles = tiles_of(S);
	hipLaunchKernelGGL(k_scan_tiles, dim3(unsigned(tiles), S.cols), dim3(THREADS), 0, s, S, work, tot, int(tiles));
	if (tiles > 1) {
		hipLaunchKernelGGL(k_scan_tops, dim3(S.cols), dim3(THREADS), 0, s, S, work, tot, int(tiles));
		hipLaunchKernelGGL(k_scan_add, dim3(unsigned(tiles), S.cols), dim3(THREADS), 0, s, S, work, int(tiles));
	}
	return hipGetLastError();
}

}  // namespace tg
