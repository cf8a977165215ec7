// tg_kernels.hip -- gfx950 kernels for tigergrav's eight interaction kinds.
//
// Mapping to CDNA4:
//  * leaf kinds (PP, PC): one 64-lane wave per item; lane = (sink, phase).  A leaf of n <= 64
//    sinks is padded to the next power of two nsp and the wave runs 64/nsp phases, each phase
//    taking every (64/nsp)-th source of the tile, so small leaves still fill the wave.  Sources
//    are staged 64 at a time through LDS and read back as broadcasts.  Per-tile partial sums are
//    float, the running sum FP64 (the reference accumulates float terms in FP64 lanes,
//    src/gravity.cpp:259-261), and phases are merged with cross-lane FP64 shuffles.
//  * node kinds (CC, CP): lane = source; a wave packs the short lists of several expansion
//    centres (<= 64 entries), 35 float accumulators per lane, merged per centre in FP64 through
//    LDS by a segmented scan.
//  * Ewald kinds use tg::ewt_eval (tg_math.hpp).
#include "tg_kernels.hpp"
#include "tg_leaf_waves.hpp"
#include "tg_math.hpp"

#include <climits>
#include <cmath>
#include <mutex>
#include <vector>

namespace tg {

__constant__ const float* c_ewt;

// ---- the tabulated correction -------------------------------------------------------------
static std::mutex table_mtx;                     // guards device_table and the per-device set-up
static std::vector<const float*> device_table;  // the tabulated correction on each device

const float* ewald_table_on(int device) {
	std::lock_guard<std::mutex> lock(table_mtx);
	return device >= 0 && device < (int) device_table.size() ? device_table[size_t(device)] : nullptr;
}

hipError_t init_device_tables(int device) {
	static std::vector<int> done;
	std::lock_guard<std::mutex> lock(table_mtx);
	if ((int) done.size() <= device) done.resize(device + 1, 0);
	if (done[device]) return hipSuccess;
	hipError_t e;
	if ((e = hipSetDevice(device)) != hipSuccess) return e;
	{
		// the tabulated correction: built once per process on the host, copied to every device, and
		// kept until the process ends
		static std::vector<float> table;
		if (table.empty()) ewald_table_build(table);
		float* dt = nullptr;
		if ((e = hipMalloc(&dt, table.size() * sizeof(float))) != hipSuccess) return e;
		if ((e = hipMemcpy(dt, table.data(), table.size() * sizeof(float), hipMemcpyHostToDevice)) != hipSuccess) return e;
		const float* cdt = dt;
		if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_ewt), &cdt, sizeof(cdt))) != hipSuccess) return e;
		if ((int) device_table.size() <= device) device_table.resize(size_t(device) + 1, nullptr);
		device_table[size_t(device)] = cdt;
	}
	done[device] = 1;
	return hipSuccess;
}

// ---- separations -----------------------------------------------------------------------------
// position difference a - b in position units (2^32 per box), as float:
//   WRAP: the int32 wrap-around difference (periodic minimum image, src/gravity.cpp:221-225);
//   else: the exact 33-bit difference, rounded once (src/gravity.cpp:227-229).
template <bool WRAP>
__device__ __forceinline__ float sepu(int a, int b) {
	const unsigned d = unsigned(a) - unsigned(b);
	if (WRAP) return float(int(d));
	const bool neg = a < b;
	const float f = float(neg ? 0u - d : d);
	return neg ? -f : f;
}

__device__ __forceinline__ int ceil_log2_64(int n) { return n <= 1 ? 0 : 32 - __clz(n - 1); }


// ---- PP direct -------------------------------------------------------------------------------
// Spline-softened (GADGET-2 cubic spline, support h) potential and acceleration
// (src/gravity.cpp:231-287).  Beyond h it is Newton's 1/r.  A leaf item's source list starts with
// the sources that may come within h of its sinks (the near prefix, PP_NEAR_LEN of the item);
// tiles that reach into it run the per-lane softened branch, every later tile the straight-line
// far field.  The 64-source tile is stored phase-major in LDS, so every lane walks consecutive
// entries with a wave-uniform trip count; a partial last tile is padded with zero-weight entries.
// With equal masses (UNIFORM) the mass multiplies the sums once at the end.
template <bool USE_W, bool PHI>
__device__ __forceinline__ void pp_pair(const int4& s, float h2u, float hinvu, float hinv3u, float& ax, float& ay, float& az,
		float& pp, float fx, float fy, float fz) {
	const float r2 = fmaf(fz, fz, fmaf(fy, fy, fx * fx));
	const float w = __int_as_float(s.w);
	if (r2 > h2u) {
		const float ri = __builtin_amdgcn_rsqf(r2);
		const float wri = USE_W ? w * ri : ri;
		const float wri3 = wri * ri * ri;
		ax = fmaf(fx, wri3, ax);
		ay = fmaf(fy, wri3, ay);
		az = fmaf(fz, wri3, az);
		if (PHI) pp += wri;
	} else {
		const float ru = sqrtf(r2);
		const float q = ru * hinvu;
		float f, p;
		if (q < 0.5f) {
			const float q2 = q * q;
			f = fmaf(q2, fmaf(32.0f, q, -192.0f / 5.0f), 32.0f / 3.0f) * hinv3u;
			p = fmaf(q2, fmaf(q2, fmaf(-32.0f / 5.0f, q, 48.0f / 5.0f), -16.0f / 3.0f), 14.0f / 5.0f) * hinvu;
		} else {
			const float ri = 1.0f / ru;
			const float q3 = q * q * q;
			f = fmaf(fmaf(fmaf(fmaf(-32.0f / 3.0f, q, 192.0f / 5.0f), q, -48.0f), q, 64.0f / 3.0f), q3, -1.0f / 15.0f) *
			    (ri * ri * ri);
			p = fmaf(fmaf(fmaf(fmaf(fmaf(32.0f / 15.0f, q, -48.0f / 5.0f), q, 16.0f), q, -32.0f / 3.0f), q * q, 16.0f / 5.0f), q,
			         -1.0f / 15.0f) * ri;
		}
		const float wf = w * f;
		ax = fmaf(fx, wf, ax);
		ay = fmaf(fy, wf, ay);
		az = fmaf(fz, wf, az);
		if (PHI) pp = fmaf(w, p, pp);
	}
}

// a pair known to be at least h apart, from its exact separation (position units).  The
// separation of two distinct positions is at least one unit, so the floor of r2 changes no pair of
// the list and keeps a zero-weight pad that lands on a sink finite.
template <bool USE_W, bool PHI>
__device__ __forceinline__ void pp_far(const int4& s, float& ax, float& ay, float& az, float& pp, float fx, float fy, float fz) {
	const float r2 = fmaxf(fmaf(fz, fz, fmaf(fy, fy, fx * fx)), 1.0f);
	const float ri = __builtin_amdgcn_rsqf(r2);
	const float wri = USE_W ? __int_as_float(s.w) * ri : ri;
	const float wri3 = wri * ri * ri;
	ax = fmaf(fx, wri3, ax);
	ay = fmaf(fy, wri3, ay);
	az = fmaf(fz, wri3, az);
	if (PHI) pp += wri;
}

// the same far pair from offsets to a common centre: sink offset (ox, oy, oz) minus the source's
// offset (s.x, s.y, s.z), source weight s.w
template <bool USE_W, bool PHI>
__device__ __forceinline__ void pp_far_off(const float4& s, float ox, float oy, float oz, float& ax, float& ay, float& az,
		float& pp) {
	const float fx = ox - s.x, fy = oy - s.y, fz = oz - s.z;
	const float r2 = fmaf(fz, fz, fmaf(fy, fy, fx * fx));
	const float ri = __builtin_amdgcn_rsqf(r2);
	const float wri = USE_W ? s.w * ri : ri;
	const float wri3 = wri * ri * ri;
	ax = fmaf(fx, wri3, ax);
	ay = fmaf(fy, wri3, ay);
	az = fmaf(fz, wri3, az);
	if (PHI) pp += wri;
}

// offsets of at least 2^30 position units (a quarter box) from the item's centre: the difference
// of two offsets below it is the wrapped separation itself
__device__ __forceinline__ bool off_big(float ox, float oy, float oz) {
	return fabsf(ox) >= 1073741824.0f || fabsf(oy) >= 1073741824.0f || fabsf(oz) >= 1073741824.0f;
}

// one PP item (<= 64 sinks of a leaf against its source list), by one work group of NW waves, each
// on its own share of the list.
// Lane = (sink si, phase ph) with P = 64 / ns phases (lanes from P ns on idle), so a leaf of ns
// sinks keeps P ns of the 64 lanes busy.  A 64-source tile is staged phase-major in LDS: phase ph
// takes sources ph, ph + P, ... from K = ceil(64 / P) consecutive slots (slots no source fills hold
// zero-weight pads), so every lane walks its slots with a wave-uniform trip count.  The phases
// start an odd number of 16-byte slots apart, so the P addresses one read instruction broadcasts
// lie in different LDS banks.  Per-tile partial
// sums are float, the running sums FP64; the phases of a sink are added in phase order through LDS.
// Tiles of the near prefix take separations as exact integer differences rounded once
// (src/gravity.cpp:221-229) and the softened pair.  Far tiles take every separation as the
// difference of two float offsets from the item's first sink: a source's offset is converted
// once per tile when it is staged, so the pair costs one subtract per axis instead of an integer
// subtract and a conversion.  The offsets are integer differences rounded once, so a separation
// carries at most the rounding of the larger offset (2^-24 of it) beside its own.  Periodic tiles
// with an offset of a quarter box or more (possible only when leaves span that much) keep the
// exact form, so the wrap-around always picks the nearest image.
struct PPShared {  // one wave's
	int4 tile[128];
	float4 ftile[128];
	double red[4][64];
};

template <int NW, bool WRAP, bool PHI, bool UNIFORM>
__device__ __forceinline__ void pp_item(const LeafArgs& A, const int4 it, PPShared* SS) {
	const int lane = threadIdx.x & 63;
	const int wave = NW == 1 ? 0 : int(threadIdx.x >> 6);
	PPShared& S = SS[wave];
	const int2 share = wave_share<NW>(it.z, it.w, wave);
	const int ns = max(it.y & PP_COUNT_MASK, 1);
	const int near_len = int(unsigned(it.y) >> PP_NEAR_SHIFT);
	const int near_end = near_len == PP_NEAR_ALL ? INT_MAX : it.z + near_len;
	const int P = 64 / ns;             // phases
	const int K = (64 + P - 1) / P;    // slots per phase
	// phase stride in the tile: odd, so the phases' broadcast reads in one instruction fall on
	// different 4-bank groups of the LDS (conflict-free for up to 8 phases)
	const int KS = K | 1;
	const int ph = min(lane / ns, P - 1);
	const int si = lane - (lane / ns) * ns;
	const int4 me = A.sinks[it.x + si];
	const int4 c0 = A.sinks[it.x];     // the item's centre for the far tiles
	const float ox = sepu<WRAP>(me.x, c0.x), oy = sepu<WRAP>(me.y, c0.y), oz = sepu<WRAP>(me.z, c0.z);
	const bool item_off = !WRAP || __ballot(off_big(ox, oy, oz)) == 0ull;
	// source l of a tile goes to phase l % P, slot l / P; slots past the tile's sources are pads
	const int dst = (lane % P) * KS + lane / P;
	const int4 pad = make_int4(INT_MIN, INT_MIN, INT_MIN, 0);
	const float4 fpad = make_float4(3.0e30f, 3.0e30f, 3.0e30f, 0.0f);
	S.tile[lane] = pad;
	S.tile[lane + 64] = pad;
	S.ftile[lane] = fpad;
	S.ftile[lane + 64] = fpad;
	const int4* mine = S.tile + ph * KS;
	const float4* fmine = S.ftile + ph * KS;
	float ax = 0.f, ay = 0.f, az = 0.f, pp = 0.f;
	double dax = 0.0, day = 0.0, daz = 0.0, dpp = 0.0;
	// software pipeline: the next tile's source record (and the list index after it) are loaded
	// while the current tile is evaluated
	auto index_at = [&](int b) { return b + lane < share.y ? (A.list ? A.list[b + lane] : b + lane) : -1; };
	auto source_at = [&](int j) {
		int4 v = pad;  // zero weight
		if (j >= 0) {
			v = A.srcs[j];
			if (UNIFORM) v.w = __float_as_int(1.0f);
		}
		return v;
	};
	int next_idx0 = index_at(share.x);
	int4 next = source_at(next_idx0);
	bool next_pad = next_idx0 < 0;
	int next_idx = index_at(share.x + 64);
	for (int base = share.x; base < share.y; base += 64) {
		const int n = min(64, share.y - base);
		const bool near = base < near_end;
		// the staged source as an offset from the centre; a pad sits out of reach (r2 overflows to
		// infinity, its reciprocal root and weight are zero)
		float4 f = fpad;
		if (!next_pad) f = make_float4(sepu<WRAP>(next.x, c0.x), sepu<WRAP>(next.y, c0.y), sepu<WRAP>(next.z, c0.z),
				__int_as_float(next.w));
		const unsigned long long bigs = WRAP ? __ballot(!next_pad && off_big(f.x, f.y, f.z)) : 0ull;
		const bool use_off = item_off && !near && bigs == 0ull;
		wave_lds_sync<NW>();
		S.tile[dst] = next;
		S.ftile[dst] = f;
		wave_lds_sync<NW>();
		next_pad = next_idx < 0;
		next = source_at(next_idx);
		next_idx = index_at(base + 128);
		const int trip = n == 64 ? K : (n + P - 1) / P;
		if (near) {
			for (int j = 0; j < trip; j++) {
				const int4 s = mine[j];
				pp_pair<true, PHI>(s, A.h2u, A.hinvu, A.hinv3u, ax, ay, az, pp, sepu<WRAP>(me.x, s.x), sepu<WRAP>(me.y, s.y),
						sepu<WRAP>(me.z, s.z));
			}
		} else if (use_off) {
			// pads add exact zeros with or without their weight
#pragma unroll 8
			for (int j = 0; j < trip; j++) pp_far_off<!UNIFORM, PHI>(fmine[j], ox, oy, oz, ax, ay, az, pp);
		} else {
			for (int j = 0; j < trip; j++) {
				const int4 s = mine[j];
				pp_far<true, PHI>(s, ax, ay, az, pp, sepu<WRAP>(me.x, s.x), sepu<WRAP>(me.y, s.y), sepu<WRAP>(me.z, s.z));
			}
		}
		dax += ax;
		day += ay;
		daz += az;
		dpp += pp;
		ax = ay = az = pp = 0.f;
	}
	// the phases of each sink, added in phase order, wave after wave
	S.red[0][lane] = dax;
	S.red[1][lane] = day;
	S.red[2][lane] = daz;
	S.red[3][lane] = dpp;
	__syncthreads();
	if (wave == 0 && lane < ns) {
		for (int q = 1; q < NW * P; q++) {
			const PPShared& R = SS[NW == 1 ? 0 : q / P];
			const int l = (NW == 1 ? q : q % P) * ns + lane;
			dax += R.red[0][l];
			day += R.red[1][l];
			daz += R.red[2][l];
			dpp += R.red[3][l];
		}
		// position units: g = -sum w dx r^-3 = -2^64 sum (w du ru^-3), phi = -2^32 sum (w / ru)
		const double ms = UNIFORM ? double(A.m) : 1.0;
		double* o = A.out + 4 * (size_t) (it.x + lane);
		if (PHI) o[0] += -4294967296.0 * ms * dpp;
		o[1] += -18446744073709551616.0 * ms * dax;
		o[2] += -18446744073709551616.0 * ms * day;
		o[3] += -18446744073709551616.0 * ms * daz;
	}
}

// one work group per item; the dispatcher hands items out in array order (heaviest first)
template <int NW, bool WRAP, bool PHI, bool UNIFORM>
__global__ __launch_bounds__(64 * NW) void k_pp_direct(LeafArgs A) {
	__shared__ PPShared S[NW];
	pp_item<NW, WRAP, PHI, UNIFORM>(A, A.items[blockIdx.x], S);
}

// persistent form: work groups of as many waves in all as the machine keeps resident, each taking the
// next item from a queue counter (A.queue, zero at launch) until the items run out
template <int NW, bool WRAP, bool PHI, bool UNIFORM>
__global__ __launch_bounds__(64 * NW) void k_pp_direct_queue(LeafArgs A) {
	__shared__ PPShared S[NW];
	__shared__ int next;
	for (;;) {
		__syncthreads();
		if (threadIdx.x == 0) next = atomicAdd(A.queue, 1);
		__syncthreads();
		const int k = next;
		if (k >= A.nitems) break;
		pp_item<NW, WRAP, PHI, UNIFORM>(A, A.items[k], S);
	}
}

__global__ void k_zero_counter(int* c) {
	if (threadIdx.x == 0) c[0] = 0;
}

template <int NW, bool WRAP, bool PHI, bool UNIFORM>
static void pp_launch(const LeafArgs& a, hipStream_t s) {
	if (a.queue) {
		// the counter is cleared by a kernel (not a memset) so the launch sequence stays graph-safe
		hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, s, a.queue);
		const int most = a.resident > NW ? a.resident / NW : 1;
		const int groups = a.nitems < most ? a.nitems : most;
		hipLaunchKernelGGL((k_pp_direct_queue<NW, WRAP, PHI, UNIFORM>), dim3(groups), dim3(64 * NW), 0, s, a);
	} else {
		hipLaunchKernelGGL((k_pp_direct<NW, WRAP, PHI, UNIFORM>), dim3(a.nitems), dim3(64 * NW), 0, s, a);
	}
}

template <bool WRAP, bool PHI, bool UNIFORM>
static void pp_waves(const LeafArgs& a, hipStream_t s) {
	switch (leaf_waves(a.nitems, a.nlist, 8)) {
		case 1: pp_launch<1, WRAP, PHI, UNIFORM>(a, s); break;
		case 2: pp_launch<2, WRAP, PHI, UNIFORM>(a, s); break;
		case 4: pp_launch<4, WRAP, PHI, UNIFORM>(a, s); break;
		default: pp_launch<8, WRAP, PHI, UNIFORM>(a, s); break;
	}
}

hipError_t launch_pp_direct(const LeafArgs& a, bool do_phi, hipStream_t s) {
	if (a.nitems <= 0) return hipSuccess;
	const bool u = a.uniform != 0;
	if (a.wrap) {
		if (do_phi) { if (u) pp_waves<true, true, true>(a, s); else pp_waves<true, true, false>(a, s); }
		else { if (u) pp_waves<true, false, true>(a, s); else pp_waves<true, false, false>(a, s); }
	} else {
		if (do_phi) { if (u) pp_waves<false, true, true>(a, s); else pp_waves<false, true, false>(a, s); }
		else { if (u) pp_waves<false, false, true>(a, s); else pp_waves<false, false, false>(a, s); }
	}
	return hipGetLastError();
}

// ---- PC (multipole -> particle) ----------------------------------------------------------------
template <int NW, bool EWALD, bool WRAP>
__global__ __launch_bounds__(64 * NW) void k_pc(LeafArgs A) {
	const int4 it = A.items[blockIdx.x];
	const int lane = threadIdx.x & 63;
	const int wave = NW == 1 ? 0 : int(threadIdx.x >> 6);
	const int2 share = wave_share<NW, 4>(it.z, it.w, wave);
	const int ns = it.y & PP_COUNT_MASK;
	const int lg = ceil_log2_64(ns);
	const int nsp = 1 << lg;
	const int P = 64 >> lg;
	const int si = lane & (nsp - 1);
	const int ph = lane >> lg;
	const int4 me = A.sinks[it.x + min(si, ns - 1)];
	__shared__ float tiles[NW][64][20];
	__shared__ double red[NW > 1 ? NW - 1 : 1][4][64];
	__shared__ EwtStage<35> stages[EWALD ? NW : 1];
	float (*tile)[20] = tiles[wave];
	float phi = 0.f, g[3] = {0.f, 0.f, 0.f};
	double dphi = 0.0, dg[3] = {0.0, 0.0, 0.0};
	for (int base = share.x; base < share.y; base += 64) {
		const int n = min(64, share.y - base);
		wave_lds_sync<NW>();
		if (lane < n) {
			const float4* src = reinterpret_cast<const float4*>(A.multis + (A.list ? A.list[base + lane] : base + lane));
#pragma unroll
			for (int q = 0; q < 5; q++) {
				const float4 v = src[q];
				tile[lane][4 * q] = v.x;
				tile[lane][4 * q + 1] = v.y;
				tile[lane][4 * q + 2] = v.z;
				tile[lane][4 * q + 3] = v.w;
			}
		}
		wave_lds_sync<NW>();
		auto source = [&](int k, bool on) {
			float M[17];
#pragma unroll
			for (int q = 0; q < 17; q++) M[q] = tile[k][q];
			const float x[3] = {sepu<EWALD || WRAP>(me.x, __float_as_int(tile[k][17])) * POS_INVF,
					sepu<EWALD || WRAP>(me.y, __float_as_int(tile[k][18])) * POS_INVF,
					sepu<EWALD || WRAP>(me.z, __float_as_int(tile[k][19])) * POS_INVF};
			float D[35];
			if (EWALD)
				green_ewald_wave<35>(D, x, c_ewt, stages[EWALD ? wave : 0], lane);
			else
				green_direct(D, x);
			if (on) m2p(phi, g, M, D);
		};
		if (EWALD) {  // the whole wave takes every turn (its table rows are read together)
			for (int k0 = 0; k0 < n; k0 += P) source(min(k0 + ph, n - 1), k0 + ph < n);
		} else {
			for (int k = ph; k < n; k += P) source(k, true);
		}
		dphi += phi;
		dg[0] += g[0];
		dg[1] += g[1];
		dg[2] += g[2];
		phi = g[0] = g[1] = g[2] = 0.f;
	}
	leaf_sums<NW>(dphi, dg, nsp, lane, wave, red);
	if (wave == 0 && ph == 0 && si < ns) {
		double* o = A.out + 4 * (size_t) (it.x + si);
		o[0] += dphi;
		o[1] += dg[0];
		o[2] += dg[1];
		o[3] += dg[2];
	}
}

template <int NW>
static void pc_launch(const LeafArgs& a, bool ewald, hipStream_t s) {
	if (ewald)
		hipLaunchKernelGGL((k_pc<NW, true, true>), dim3(a.nitems), dim3(64 * NW), 0, s, a);
	else if (a.wrap)
		hipLaunchKernelGGL((k_pc<NW, false, true>), dim3(a.nitems), dim3(64 * NW), 0, s, a);
	else
		hipLaunchKernelGGL((k_pc<NW, false, false>), dim3(a.nitems), dim3(64 * NW), 0, s, a);
}

static void pc_launch8(const LeafArgs& a, hipStream_t s) {
	if (a.wrap)
		hipLaunchKernelGGL((k_pc<8, false, true>), dim3(a.nitems), dim3(512), 0, s, a);
	else
		hipLaunchKernelGGL((k_pc<8, false, false>), dim3(a.nitems), dim3(512), 0, s, a);
}

hipError_t launch_pc(const LeafArgs& a, bool ewald, hipStream_t s) {
	if (a.nitems <= 0) return hipSuccess;
	// the Ewald kind's rows and tile take 13 KB of LDS a wave
	switch (leaf_waves_fine(a.nitems, a.nlist, ewald ? 4 : 8, 8)) {
		case 1: pc_launch<1>(a, ewald, s); break;
		case 2: pc_launch<2>(a, ewald, s); break;
		case 4: pc_launch<4>(a, ewald, s); break;
		default: pc_launch8(a, s); break;
	}
	return hipGetLastError();
}

// ---- PP Ewald correction -------------------------------------------------------------------------
// The periodic correction between particle pairs (src/gravity.cpp:491-614): per pair the potential
// and gradient of the tabulated correction (ewt_eval<4>: the reference's real-space images,
// Fourier terms, n = 0 term and pi/4 in one table), weighted by the source mass; pairs closer than
// 1e-6 take the reference's constant 2.8372975 and zero force (its zmask).  Sinks and sources are
// laid out as in k_pc: 2^lg lanes per sink, the other lane bits split the tile's sources.
// Bound by the rows' way through the vector cache and LDS (8 KB a turn) beside about 150
// instructions of arithmetic, at the four waves a SIMD that the stages leave.  32,768 uniform
// particles, leaves of 64 (4.5e7 pairs): 646 -> 460 us against a row read by each lane and a 19-term
// sum per component (16 waves in 152 KB took 430; a work group keeps to 64 KB).
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_pp_ewald(LeafArgs A) {
	const int4 it = A.items[blockIdx.x];
	const int lane = threadIdx.x & 63;
	const int wave = NW == 1 ? 0 : int(threadIdx.x >> 6);
	const int2 share = wave_share<NW, 8>(it.z, it.w, wave);
	const int ns = it.y & PP_COUNT_MASK;
	const int lg = ceil_log2_64(ns);
	const int nsp = 1 << lg;
	const int P = 64 >> lg;
	const int si = lane & (nsp - 1);
	const int ph = lane >> lg;
	const int4 me = A.sinks[it.x + min(si, ns - 1)];
	// the sums' exchange at the end reuses the stages (8 waves take 64 KB with the tiles)
	__shared__ EwtStage<4> stages[NW];
	__shared__ int4 tiles[NW][64];
	static_assert(sizeof(double) * (NW - 1) * 4 * 64 <= sizeof(stages), "exchange in the stages");
	double (*red)[4][64] = reinterpret_cast<double (*)[4][64]>(stages);
	int4* tile = tiles[wave];
	double dphi = 0.0, dg[3] = {0.0, 0.0, 0.0};
	for (int base = share.x; base < share.y; base += 64) {
		const int n = min(64, share.y - base);
		wave_lds_sync<NW>();
		if (lane < n) tile[lane] = A.srcs[A.list ? A.list[base + lane] : base + lane];
		wave_lds_sync<NW>();
		float phi = 0.f, g[3] = {0.f, 0.f, 0.f};
		// the next turn's rows are on their way while this turn's are evaluated
		auto at = [&](int k0) {
			const int4 s = tile[min(k0 + ph, n - 1)];
			const float x[3] = {sepu<true>(me.x, s.x) * POS_INVF, sepu<true>(me.y, s.y) * POS_INVF, sepu<true>(me.z, s.z) * POS_INVF};
			return ewt_point(x);
		};
		EwtPoint p = at(0);
		EwtRows<4> rows;
		rows.fetch(p.row, c_ewt, stages[wave], lane);
		for (int k0 = 0; k0 < n; k0 += P) {
			float c[EwtRead<4>::F4 * 4], D[4];
			rows.take(c, stages[wave], lane);
			const EwtPoint now = p;
			const float w = k0 + ph < n ? __int_as_float(tile[min(k0 + ph, n - 1)].w) : 0.0f;
			if (k0 + P < n) {
				p = at(k0 + P);
				rows.fetch(p.row, c_ewt, stages[wave], lane);
			}
			ewt_eval<4>(D, c, now);
			phi = fmaf(w, D[0], phi);
			g[0] = fmaf(-w, D[1], g[0]);
			g[1] = fmaf(-w, D[2], g[1]);
			g[2] = fmaf(-w, D[3], g[2]);
		}
		dphi += phi;
		dg[0] += g[0];
		dg[1] += g[1];
		dg[2] += g[2];
	}
	if (NW > 1) __syncthreads();
	leaf_sums<NW>(dphi, dg, nsp, lane, wave, red);
	if (wave == 0 && ph == 0 && si < ns) {
		double* o = A.out + 4 * (size_t) (it.x + si);
		o[0] += dphi;
		o[1] += dg[0];
		o[2] += dg[1];
		o[3] += dg[2];
	}
}

hipError_t launch_pp_ewald(const LeafArgs& a, hipStream_t s) {
	if (a.nitems <= 0) return hipSuccess;
	// 64 sources a wave: a turn takes one source per sink's lane group through its rows
	switch (leaf_waves_fine(a.nitems, a.nlist, 8, 64)) {
		case 1: hipLaunchKernelGGL(k_pp_ewald<1>, dim3(a.nitems), dim3(64), 0, s, a); break;
		case 2: hipLaunchKernelGGL(k_pp_ewald<2>, dim3(a.nitems), dim3(128), 0, s, a); break;
		case 4: hipLaunchKernelGGL(k_pp_ewald<4>, dim3(a.nitems), dim3(256), 0, s, a); break;
		default: hipLaunchKernelGGL(k_pp_ewald<8>, dim3(a.nitems), dim3(512), 0, s, a); break;
	}
	return hipGetLastError();
}

// ---- node kinds ----------------------------------------------------------------------------------
// Segmented FP64 reduction of the lanes' 35 float accumulators by owner slot, through LDS.  The entries
// of one slot are consecutive: lanes 0..34 add one coefficient each over every segment.
// All 35 components are summed, though the tensor's trace is known (zero for derivatives of 1/r, a
// constant for the periodic correction): one taken from two others carries their errors, up to 1.8
// times its own against FP64.  Ten sums fewer took 0.2 ms off the 4.35 ms solve of 2M particles at
// theta 0.3.
struct NodeSums {
	float red[35][65];
	int sl[64];
};
union NodeLds {  // the Ewald kinds' rows, then the sums
	EwtStage<35> rows;
	NodeSums sums;
};
union NodeFoldLds {  // the direct kind's multipoles, then the sums
	ewt_f4 stage[256];
	NodeSums sums;
};

__device__ __forceinline__ void node_store(const float* L, int slot, int cnt, NodeSums& S, double* partial) {
	const int lane = threadIdx.x;
	__syncthreads();
#pragma unroll
	for (int c = 0; c < 35; c++) S.red[c][lane] = L[c];
	S.sl[lane] = slot;
	__syncthreads();
	// the wave's segments (runs of one slot) from a ballot of their first entries, four FP64 partial sums
	// per segment
	const bool first = lane < cnt && (lane == 0 || S.sl[lane] != S.sl[lane - 1]);
	unsigned long long starts = __ballot(first);
	if (lane >= 35) return;
	while (starts) {
		const int b = __ffsll(starts) - 1;
		starts &= starts - 1;
		const int e = starts ? __ffsll(starts) - 1 : cnt;
		double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
		int j = b;
		for (; j + 4 <= e; j += 4) {
			a0 += double(S.red[lane][j]);
			a1 += double(S.red[lane][j + 1]);
			a2 += double(S.red[lane][j + 2]);
			a3 += double(S.red[lane][j + 3]);
		}
		for (; j < e; j++) a0 += double(S.red[lane][j]);
		partial[35 * (size_t) S.sl[b] + lane] = (a0 + a1) + (a2 + a3);
	}
}

__device__ __forceinline__ void multi_floats(float* v, const float4* m) {
#pragma unroll
	for (int q = 0; q < 5; q++) {
		v[4 * q] = m[q].x;
		v[4 * q + 1] = m[q].y;
		v[4 * q + 2] = m[q].z;
		v[4 * q + 3] = m[q].w;
	}
}

// A wave takes a run of list entries: up to 64 entries of one or more partial slots (one entry per
// lane), or the entries of one slot beyond 64 (a chunk longer than a wave), which the lanes take
// 64 apart, each adding its entries' terms in order before the store.
template <bool WRAP>
__global__ __launch_bounds__(64) void k_cc(NodeArgs A) {
	__shared__ NodeSums sums;
	const int2 wv = A.waves[blockIdx.x];
	const int lane = threadIdx.x;
	float L[35];
#pragma unroll
	for (int c = 0; c < 35; c++) L[c] = 0.f;
	int slot = -1;
	int j = wv.x + lane;
	if (j < wv.y) {
		slot = A.owner ? A.owner[j] : int(blockIdx.x);  // the plain drop-in: one slot per wave, one sink
		const int4 X = A.sinkpos[A.slot_node ? A.slot_node[slot] : 0];
		for (; j < wv.y; j += 64) {
			const float4* src = reinterpret_cast<const float4*>(A.multis + (A.list ? A.list[j] : j));
			float4 f[5];
#pragma unroll
			for (int q = 0; q < 5; q++) f[q] = src[q];
			float v[20], q[5], o[7], qzz, D[35];
			multi_floats(v, f);
			const float x[3] = {sepu<WRAP>(X.x, __float_as_int(v[17])) * POS_INVF, sepu<WRAP>(X.y, __float_as_int(v[18])) * POS_INVF,
					sepu<WRAP>(X.z, __float_as_int(v[19])) * POS_INVF};
			green_direct(D, x);
			fold_multi(v, q, o, qzz);
			m2l(L, v[0], q, o, D);
		}
	}
	node_store(L, slot, min(wv.y - wv.x, 64), sums, A.partial);
}

// The same from a solver's folded multipoles, which the wave reads together: four lanes take a record,
// so a load touches 16 half lines where a record per lane touches 64, and LDS hands each lane its own
// (parts rotated so that neither side conflicts).  The next turn's records are on their way while this
// turn's are evaluated; lanes past the end carry the last entry without weight.
// Bound by FP32 arithmetic: 1.37e9 wave instructions for 3.3e8 entries (2M particles at theta 0.3), 2.10 ->
// 2.05 ms against records per lane with the weights formed per entry; at theta 0.6 (1.05e7 entries)
// 0.210 -> 0.179 ms.
template <bool WRAP>
__global__ __launch_bounds__(64) void k_cc_folded(NodeArgs A) {
	__shared__ NodeFoldLds lds;
	const int2 wv = A.waves[blockIdx.x];
	const int lane = threadIdx.x;
	float L[35];
#pragma unroll
	for (int c = 0; c < 35; c++) L[c] = 0.f;
	int slot = -1;
	int4 X = make_int4(0, 0, 0, 0);
	if (wv.x + lane < wv.y) {
		slot = A.owner[wv.x + lane];
		X = A.sinkpos[A.slot_node[slot]];
	}
	if (wv.x < wv.y) {
		const int part = (lane & 3) ^ (lane >> 4);  // of records 16 q + lane / 4, rotated by record / 4
		const unsigned at = lane >> 2, last = wv.y - 1;
		int i0, i1, i2, i3;  // the next turn's records
		ewt_f4 in0, in1, in2, in3;
		const ewt_f4* recs = reinterpret_cast<const ewt_f4*>(A.folded) + part;
#define TG_CC_INDICES(j)                     \
	i0 = A.list[min(unsigned(j) + at, last)];        \
	i1 = A.list[min(unsigned(j) + 16 + at, last)];   \
	i2 = A.list[min(unsigned(j) + 32 + at, last)];   \
	i3 = A.list[min(unsigned(j) + 48 + at, last)]
#define TG_CC_RECORDS              \
	in0 = recs[4 * size_t(i0)];    \
	in1 = recs[4 * size_t(i1)];    \
	in2 = recs[4 * size_t(i2)];    \
	in3 = recs[4 * size_t(i3)]
		TG_CC_INDICES(wv.x);
		TG_CC_RECORDS;
		TG_CC_INDICES(wv.x + 64);
		for (int j0 = wv.x; j0 < wv.y; j0 += 64) {
			__syncthreads();
			lds.stage[lane] = in0;
			lds.stage[64 + lane] = in1;
			lds.stage[128 + lane] = in2;
			lds.stage[192 + lane] = in3;
			__syncthreads();
			TG_CC_RECORDS;
			TG_CC_INDICES(j0 + 128);
			float v[16];
			static_for<4>([&](auto q_) {
				constexpr int q = decltype(q_)::value;
				const ewt_f4 f = lds.stage[4 * lane + (q ^ ((lane >> 2) & 3))];
				v[4 * q] = f.x;
				v[4 * q + 1] = f.y;
				v[4 * q + 2] = f.z;
				v[4 * q + 3] = f.w;
			});
			const float x[3] = {sepu<WRAP>(X.x, __float_as_int(v[13])) * POS_INVF, sepu<WRAP>(X.y, __float_as_int(v[14])) * POS_INVF,
					sepu<WRAP>(X.z, __float_as_int(v[15])) * POS_INVF};
			float D[35];
			green_direct(D, x);
			if (j0 + 64 > wv.y && j0 + lane >= wv.y) {
#pragma unroll
				for (int c = 0; c < 13; c++) v[c] = 0.0f;
			}
			m2l(L, v[0], v + 1, v + 6, D);
		}
	}
#undef TG_CC_INDICES
#undef TG_CC_RECORDS
	node_store(L, slot, min(wv.y - wv.x, 64), lds.sums, A.partial);
}

// The Ewald correction of the same: the whole wave takes every turn (its table rows are read
// together), lanes past the end with the last entry and no weight.  Its multipoles fold with the
// Laplacian (error against FP64 no larger than unfolded).  Bound by arithmetic (4.0e8 wave
// instructions for 3.6e7 entries, 5.2e8 with a row per lane and a 19-term sum per component) and by the
// rows' way through the vector cache and LDS, 16 KB a turn, at three waves a SIMD: 0.78 ms (2M
// particles at theta 0.3), 0.93 before; two waves with the next turn's rows in flight took an eighth
// longer.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_cc_ewald(NodeArgs A) {
	__shared__ NodeLds lds;
	const int2 wv = A.waves[blockIdx.x];
	const int lane = threadIdx.x;
	float L[35];
#pragma unroll
	for (int c = 0; c < 35; c++) L[c] = 0.f;
	int slot = -1;
	int4 X = make_int4(0, 0, 0, 0);
	if (wv.x + lane < wv.y) {
		slot = A.owner ? A.owner[wv.x + lane] : int(blockIdx.x);
		X = A.sinkpos[A.slot_node ? A.slot_node[slot] : 0];
	}
	for (int j0 = wv.x; j0 < wv.y; j0 += 64) {
		const int j = min(j0 + lane, wv.y - 1);
		const float4* src = reinterpret_cast<const float4*>(A.multis + (A.list ? A.list[j] : j));
		float4 m[5];
#pragma unroll
		for (int q = 0; q < 5; q++) m[q] = src[q];
		float v[20];
		multi_floats(v, m);
		const float x[3] = {sepu<true>(X.x, __float_as_int(v[17])) * POS_INVF, sepu<true>(X.y, __float_as_int(v[18])) * POS_INVF,
				sepu<true>(X.z, __float_as_int(v[19])) * POS_INVF};
		if (j0 + 64 > wv.y && j0 + lane >= wv.y) {
#pragma unroll
			for (int c = 0; c < 17; c++) v[c] = 0.0f;
		}
		float q[5], o[7], qzz, D[35];
		fold_multi(v, q, o, qzz);
		const EwtPoint p = ewt_point(x);
		EwtRows<35> rows;
		rows.fetch(p.row, c_ewt, lds.rows, lane);
		float c[EwtRead<35>::F4 * 4];
		rows.take(c, lds.rows, lane);
		// the folded weights wait in LDS while the tensor is evaluated: in registers they are seven too many
		// for three waves a SIMD, which the compiler keeps in scratch memory (0.86 ms)
		ewt_f4* wait = lds.rows.part;
		EwtRows<35>::settle();
		wait[lane] = ewt_f4{v[0], q[0], q[1], q[2]};
		wait[64 + lane] = ewt_f4{q[3], q[4], o[0], o[1]};
		wait[128 + lane] = ewt_f4{o[2], o[3], o[4], o[5]};
		wait[192 + lane] = ewt_f4{o[6], qzz, 0.0f, 0.0f};
		EwtRows<35>::settle();
		ewt_eval<35>(D, c, p);
		EwtRows<35>::settle();
		const ewt_f4 w0 = wait[lane], w1 = wait[64 + lane], w2 = wait[128 + lane], w3 = wait[192 + lane];
		const float qw[5] = {w0.y, w0.z, w0.w, w1.x, w1.y}, ow[7] = {w1.z, w1.w, w2.x, w2.y, w2.z, w2.w, w3.x};
		L[0] = fmaf(w3.y, p.lap, L[0]);
		m2l(L, w0.x, qw, ow, D);
	}
	node_store(L, slot, min(wv.y - wv.x, 64), lds.sums, A.partial);
}

template <bool WRAP>
__global__ __launch_bounds__(64) void k_cp(NodeArgs A) {
	__shared__ NodeSums sums;
	const int2 wv = A.waves[blockIdx.x];
	const int lane = threadIdx.x;
	float L[35];
#pragma unroll
	for (int c = 0; c < 35; c++) L[c] = 0.f;
	int slot = -1;
	int j = wv.x + lane;
	if (j < wv.y) {
		slot = A.owner ? A.owner[j] : int(blockIdx.x);  // the plain drop-in: one slot per wave, one sink
		const int4 X = A.sinkpos[A.slot_node ? A.slot_node[slot] : 0];
		for (; j < wv.y; j += 64) {
			const int4 s = A.srcs[A.list ? A.list[j] : j];
			const float x[3] = {sepu<WRAP>(X.x, s.x) * POS_INVF, sepu<WRAP>(X.y, s.y) * POS_INVF, sepu<WRAP>(X.z, s.z) * POS_INVF};
			float D[35];
			green_direct(D, x);
			p2l(L, __int_as_float(s.w), D);
		}
	}
	node_store(L, slot, min(wv.y - wv.x, 64), sums, A.partial);
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_cp_ewald(NodeArgs A) {
	__shared__ NodeLds lds;
	const int2 wv = A.waves[blockIdx.x];
	const int lane = threadIdx.x;
	float L[35];
#pragma unroll
	for (int c = 0; c < 35; c++) L[c] = 0.f;
	int slot = -1;
	int4 X = make_int4(0, 0, 0, 0);
	if (wv.x + lane < wv.y) {
		slot = A.owner ? A.owner[wv.x + lane] : int(blockIdx.x);
		X = A.sinkpos[A.slot_node ? A.slot_node[slot] : 0];
	}
	for (int j0 = wv.x; j0 < wv.y; j0 += 64) {
		const int j = min(j0 + lane, wv.y - 1);
		const int4 s = A.srcs[A.list ? A.list[j] : j];
		const float x[3] = {sepu<true>(X.x, s.x) * POS_INVF, sepu<true>(X.y, s.y) * POS_INVF, sepu<true>(X.z, s.z) * POS_INVF};
		float D[35];
		const float lap = green_ewald_wave<35>(D, x, c_ewt, lds.rows, lane);
		const float m = j0 + lane < wv.y ? __int_as_float(s.w) : 0.0f;
		p2l(L, m, D);
	}
	node_store(L, slot, min(wv.y - wv.x, 64), lds.sums, A.partial);
}

hipError_t launch_cc(const NodeArgs& a, bool ewald, hipStream_t s) {
	if (a.nwaves <= 0) return hipSuccess;
	const dim3 g(a.nwaves), b(64);
	if (ewald)
		hipLaunchKernelGGL(k_cc_ewald, g, b, 0, s, a);
	else if (a.folded && a.wrap)
		hipLaunchKernelGGL(k_cc_folded<true>, g, b, 0, s, a);
	else if (a.folded)
		hipLaunchKernelGGL(k_cc_folded<false>, g, b, 0, s, a);
	else if (a.wrap)
		hipLaunchKernelGGL(k_cc<true>, g, b, 0, s, a);
	else
		hipLaunchKernelGGL(k_cc<false>, g, b, 0, s, a);
	return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fold_multis(const MultiSrc* __restrict__ multis, int64_t nn, FoldedMulti* __restrict__ out) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= nn) return;
	const MultiSrc s = multis[i];
	FoldedMulti f;
	float qzz;
	f.m = s.m[0];
	fold_multi(s.m, f.q, f.o, qzz);
	for (int d = 0; d < 3; d++) f.x[d] = s.x[d];
	out[i] = f;
}

hipError_t launch_fold_multis(const MultiSrc* multis, int64_t nn, FoldedMulti* out, hipStream_t s) {
	if (nn <= 0) return hipSuccess;
	hipLaunchKernelGGL(k_fold_multis, dim3(unsigned((nn + 255) / 256)), dim3(256), 0, s, multis, nn, out);
	return hipGetLastError();
}

hipError_t launch_cp(const NodeArgs& a, bool ewald, hipStream_t s) {
	if (a.nwaves <= 0) return hipSuccess;
	const dim3 g(a.nwaves), b(64);
	if (ewald)
		hipLaunchKernelGGL(k_cp_ewald, g, b, 0, s, a);
	else if (a.wrap)
		hipLaunchKernelGGL(k_cp<true>, g, b, 0, s, a);
	else
		hipLaunchKernelGGL(k_cp<false>, g, b, 0, s, a);
	return hipGetLastError();
}

}  // namespace tg
