// tg_leaf_waves.hpp -- several waves per leaf item: the split of an item's source list over the waves
// of a work group, and the sum of their results.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// orders a wave's accesses to its own LDS tile, which no other wave of the work group touches.  The
// LDS serves a wave's accesses in order, so with several waves only the compiler has to keep them
// apart.  The wait on the LDS and scalar counter costs little here and lets the loops behind it wait
// for each LDS read as it comes (a scalar load that may be pending makes every such wait one for
// all reads: 4% of the far-pair loop); a one-wave group's barrier is that wait.
template <int NW>
__device__ __forceinline__ void wave_lds_sync() {
	if (NW == 1) {
		__syncthreads();
	} else {
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	}
}

// Leaf kinds: NW waves share an item, each taking a contiguous run of its tiles of TILE sources;
// their sums are added in wave order.  [begin, end) of wave w's sources in the list [b, e).
template <int NW, int TILE = 64>
__device__ __forceinline__ int2 wave_share(int b, int e, int w) {
	if (NW == 1) return make_int2(b, e);
	const int tiles = (e - b + TILE - 1) / TILE;
	const int per = (tiles + NW - 1) / NW;
	const int lo = min(int64_t(e), int64_t(b) + int64_t(TILE) * per * w);
	const int hi = min(int64_t(e), int64_t(lo) + int64_t(TILE) * per);
	return make_int2(lo, hi);
}

// Waves per leaf item.  One wave's chain of tiles is serial, so few items with long lists leave the
// chip idle, and on clustered sets the longest lists set the kernel's time.  The waves are raised
// up to a target in all (four rounds of the chip: 256 CUs, 4 SIMDs each, eight waves a SIMD, for the
// uneven lists to even out), as long as each keeps two tiles or more on average.  Sets of more than
// half the target's items (2M particles: 65,000 and more) keep one wave each, whose sums need no second
// pass.
constexpr int64_t TARGET_WAVES = 32768;
inline int leaf_waves(int nitems, int64_t sources, int most) {
	const int64_t tiles = (sources / (nitems > 0 ? nitems : 1) + 63) / 64;
	int w = 1;
	while (w < most && int64_t(nitems) * (2 * w) <= TARGET_WAVES && tiles >= 4 * w) w *= 2;
	return w;
}

// The same for kinds whose turn takes one source (or as few as share the wave's lanes) through a long
// evaluation: shares of per sources or more on average, whatever the tiles.  300 multipoles on 64
// sinks: 69 us with two waves (the tiles' rule), 22 us with eight; the far multipoles of 262,144
// clustered particles (39 a leaf): 91 -> 59 us, their adjoint's (65,536) 160 -> 92 us.
inline int leaf_waves_fine(int nitems, int64_t sources, int most, int per) {
	int w = 1;
	while (w < most && int64_t(nitems) * (2 * w) <= TARGET_WAVES && sources >= int64_t(nitems) * per * (2 * w)) w *= 2;
	return w;
}

// The waves of a sink add up: the phases of each wave by cross-lane adds, then the waves in order
// (wave 0's first NSP lanes hold the sums).  Every lane of the group calls this.
template <int NW>
__device__ __forceinline__ void leaf_sums(double& dphi, double* dg, int nsp, int lane, int wave, double (*red)[4][64]) {
	for (int off = nsp; off < 64; off <<= 1) {
		dphi += __shfl_xor(dphi, off, 64);
		dg[0] += __shfl_xor(dg[0], off, 64);
		dg[1] += __shfl_xor(dg[1], off, 64);
		dg[2] += __shfl_xor(dg[2], off, 64);
	}
	if (NW == 1) return;
	if (wave > 0 && lane < nsp) {
		red[wave - 1][0][lane] = dphi;
		for (int d = 0; d < 3; d++) red[wave - 1][1 + d][lane] = dg[d];
	}
	__syncthreads();
	if (wave == 0 && lane < nsp)
		for (int w = 0; w < NW - 1; w++) {
			dphi += red[w][0][lane];
			for (int d = 0; d < 3; d++) dg[d] += red[w][1 + d][lane];
		}
}

}  // namespace tg
