// tg_adjoint.hip -- the adjoint of the batched force solve.
//
// For a loss L = sum_i w_i . g_i of the accelerations of one solve, the gradients dL/dx_k and
// dL/dm_k, with the tree, the interaction lists and the expansion centres of that solve held
// fixed (the function tg_solver_update_particles evaluates).  The solve is linear in every
// expansion and moment, so the adjoint runs the solve's operators transposed, recomputing every
// interaction from the stored lists (nothing of the forward is kept but its expansions dL):
//   1. sinks, over the forward's leaf work items:
//      k_adj_l2p       g = -grad T_L(x - X):   dL/dx += -w^T Hess T_L,  lambda_leaf = dg/dL^T w;
//      k_adj_up        Lambda_a = sum over leaves B below a of S(X_B - X_a)^T lambda_B (L2L transposed),
//                      level by level from the children's
//      k_adj_pp(_ewald) tidal tensor J(d) = dF/dd per pair; the lists are symmetric (leaf B is in
//                      A's PP list iff A is in B's), so each particle's source-side terms are gathered
//                      from its own list: dL/dx_k += J(d_kj) (m_j w_k - m_k w_j), dL/dm_k += -w_j . F(d_kj)
//      k_adj_pc_sink   dL/dx_i += w . dg/dx_i (fifth derivatives); k_adj_pc_t (by source node c)
//                      mu_c += dg/dM_c^T w
//   2. node lists:
//      k_adj_cc_t  mu_c += M2L(., X_a - X_c)^T Lambda_a, over the CC entries sorted by source c
//      k_adj_cp_t  CP, by source leaf: dL/dm_j += Lambda_a . D(X_a - x_j), dL/dx_j += -m_j Lambda_a . grad D
//                  (fifth derivatives), no atomics
//   3. k_adj_down, level by level from the root: mu~_c = mu_c + M2M^T mu~_parent; then k_adj_moments,
//      per leaf: the transposed P2M onto the leaf's particles.
// Ewald kinds use the periodic correction's derivatives in the same places.  Per-term arithmetic is
// FP32 like the forward; sums are FP64.  The multipole adjoints mu are accumulated with FP64
// atomics (one per source node and item), so their summation order varies between runs; Lambda and
// the particle gradients are not.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>  // DeviceRadixSort of the pair keys

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "tg_adjoint_math.hpp"
#include "tg_devmem.hpp"
#include "tg_leaf_waves.hpp"
#include "tg_scan.hpp"
#include "tg_gravity.h"
#include "tg_local.hpp"
#include "tg_solver.hpp"

namespace tg {

__constant__ const float* c_adj_ewt;  // the device's tabulated correction (tg_kernels.hip)

namespace {

using adj::add;
using adj::merge;

hipError_t init_adjoint_tables(int device) {
	const float* table = ewald_table_on(device);
	if (!table) return hipErrorNotInitialized;
	return hipMemcpyToSymbol(HIP_SYMBOL(c_adj_ewt), &table, sizeof(table));
}

// ---- compile-time contraction helpers ---------------------------------------------------------
// multipole slot of expansion slot K of order 2 or 3 (the multipole has no order 1)
constexpr int mslot(int K) { return K < 10 ? 1 + (K - 4) : 7 + (K - 10); }
constexpr float mfac(int K) { return K < 10 ? ef2(K - 4) : -ef3(K - 10); }  // M2P/M2L sign and expansion factor

// forces a constant index to be folded at compile time (the slot searches are loops)
template <int V>
constexpr int cx = V;

template <int... S, class F>
__device__ __forceinline__ void for_seq(std::integer_sequence<int, S...>, F&& f) {
	(f(std::integral_constant<int, S>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_n(F&& f) {
	for_seq(std::make_integer_sequence<int, N>{}, f);
}

// M2P acceleration at offset with derivative tensor D (the forward's m2p):
//   g_a = -sum_K fac_K M_K D_{K u a}, K over {0} u order-2 u order-3 slots, fac_0 = 1
// its derivative along b adds index b; its transpose in M contracts with w.
// returns dg/dx_b contracted with w (3 values) -- needs D to order 5
__device__ __forceinline__ void m2p_sink_adjoint(float* gx, const float* M, const float* D, const float* w) {
	for_n<3>([&](auto b_) {
		constexpr int b = decltype(b_)::value;
		float acc = 0.0f;
		for_n<3>([&](auto a_) {
			constexpr int a = decltype(a_)::value;
			float t = -M[0] * D[cx<add(add(0, a), b)>];
			for_n<16>([&](auto q_) {
				constexpr int K = 4 + decltype(q_)::value;  // order-2 and order-3 slots 4..19
				constexpr float f = -mfac(K);
				t = fmaf(f * M[cx<mslot(K)>], D[cx<add(add(K, a), b)>], t);
			});
			acc = fmaf(w[a], t, acc);
		});
		gx[b] += acc;
	});
}
// mu_K += dg/dM_K^T w
__device__ __forceinline__ void m2p_source_adjoint(float* mu, const float* D, const float* w) {
	float t0 = 0.0f;
	for_n<3>([&](auto a_) {
		constexpr int a = decltype(a_)::value;
		t0 = fmaf(-w[a], D[cx<add(0, a)>], t0);
	});
	mu[0] += t0;
	for_n<16>([&](auto q_) {
		constexpr int K = 4 + decltype(q_)::value;
		float t = 0.0f;
		for_n<3>([&](auto a_) {
			constexpr int a = decltype(a_)::value;
			t = fmaf(w[a], D[cx<add(K, a)>], t);
		});
		constexpr float f = -mfac(K);
		mu[cx<mslot(K)>] += f * t;
	});
}
// M2L transposed: mu_K += sum_t Lambda_t dL_t/dM_K for the forward's m2l (L_t += sum_K fac_K M_K D_{t u K}
// over |t| + |K| <= 4, fac_0 = 1)
__device__ __forceinline__ void m2l_adjoint(float* mu, const float* Lam, const float* D) {
	float t0 = 0.0f;
	for_n<35>([&](auto t_) {
		constexpr int t = decltype(t_)::value;
		t0 = fmaf(Lam[t], D[t], t0);
	});
	mu[0] += t0;
	for_n<16>([&](auto q_) {
		constexpr int K = 4 + decltype(q_)::value;
		float acc = 0.0f;
		for_n<35>([&](auto t_) {
			constexpr int t = decltype(t_)::value;
			if constexpr (adj::order_of(t) + adj::order_of(K) <= 4) acc = fmaf(Lam[t], D[cx<merge(t, K)>], acc);
		});
		constexpr float f = mfac(K);
		mu[cx<mslot(K)>] += f * acc;
	});
}

// spline-softened pair (src/gravity.cpp:231-287) in box units: F(d) = -d f(r), and f'(r)/r
__device__ __forceinline__ void spline_f(float r2, float h, float& f, float& fr) {
	if (r2 > h * h) {
		const float ri = __builtin_amdgcn_rsqf(r2);
		const float ri2 = ri * ri;
		f = ri2 * ri;
		fr = -3.0f * f * ri2;
		return;
	}
	const float r = sqrtf(r2), hi = 1.0f / h, q = r * hi;
	if (q < 0.5f) {
		const float hi3 = hi * hi * hi;
		f = fmaf(q * q, fmaf(32.0f, q, -192.0f / 5.0f), 32.0f / 3.0f) * hi3;
		fr = fmaf(96.0f, q, -384.0f / 5.0f) * hi3 * hi * hi;
	} else {
		const float q3 = q * q * q;
		const float P = fmaf(fmaf(fmaf(fmaf(-32.0f / 3.0f, q, 192.0f / 5.0f), q, -48.0f), q, 64.0f / 3.0f), q3, -1.0f / 15.0f);
		const float dP = q * q * fmaf(fmaf(fmaf(-64.0f, q, 192.0f), q, -192.0f), q, 64.0f);
		const float ri = 1.0f / r, ri3 = ri * ri * ri;
		f = P * ri3;
		fr = (dP * hi - 3.0f * P * ri) * ri3 * ri;
	}
}

struct AdjArgs {
	const int4* parts;      // tree order (x, y, z, mass bits)
	const float4* w;        // loss weights, tree order
	const MultiSrc* multis;
	const int4* nodepos;
	const double* dL;       // the forward's per-node expansions
	const int4* leaves;     // (node, pbegin, pend, path begin)
	const int* path;
	const int* level;
	double* grad;           // 4 per particle, tree order: dL/dx, dL/dy, dL/dz, dL/dm
	double* Lam;            // 35 per node
	double* mu;             // 17 per node
	float h;                // softening, box units
	int wrap;
	int maxdepth;
};

constexpr float PINV = 1.0f / 4294967296.0f;
__device__ __forceinline__ float sepf(int a, int b, bool wrap) {
	const unsigned d = unsigned(a) - unsigned(b);
	if (wrap) return float(int(d)) * PINV;
	return float(double(a) - double(b)) * PINV;
}

// sum of row[0..n) with four partial sums (short dependency chains)
__device__ __forceinline__ double sum4(const double* row, int n) {
	double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
	int k = 0;
	for (; k + 4 <= n; k += 4) {
		a0 += row[k];
		a1 += row[k + 1];
		a2 += row[k + 2];
		a3 += row[k + 3];
	}
	for (; k < n; k++) a0 += row[k];
	return (a0 + a1) + (a2 + a3);
}

// ---- 1. leaves -------------------------------------------------------------------------------
// L2P and the shifts: per leaf, writes each sink's gradient (the first term; later kernels add)
__global__ __launch_bounds__(64) void k_adj_l2p(AdjArgs A) {
	const int4 lf = A.leaves[blockIdx.x];
	const int t = threadIdx.x;
	const int depth = A.level[lf.x] + 1;
	const int ns = lf.z - lf.y;
	extern __shared__ double lds[];  // [35][64] per-sink lambda, [35] L then lambda of the leaf, [35][maxdepth]
	double* lam64 = lds;
	double* Ls = lds + 35 * 64;
	double* sh = Ls + 35;
	const int4 c = A.nodepos[lf.x];
	// the leaf's local expansion, as the forward forms it (sum over the path of shifted dL)
	double off[3] = {0.0, 0.0, 0.0};
	if (t < depth) {
		const int a = A.path[lf.w + t];
		const int4 X = A.nodepos[a];
		off[0] = double(int64_t(c.x) - int64_t(X.x)) * POS_INV;
		off[1] = double(int64_t(c.y) - int64_t(X.y)) * POS_INV;
		off[2] = double(int64_t(c.z) - int64_t(X.z)) * POS_INV;
		double La[35], Lt[35];
#pragma unroll
		for (int q = 0; q < 35; q++) La[q] = A.dL[35 * int64_t(a) + q];
		l2l(Lt, La, off);
#pragma unroll
		for (int q = 0; q < 35; q++) sh[q * A.maxdepth + t] = Lt[q];
	}
	__syncthreads();
	if (t < 35) Ls[t] = sum4(sh + t * A.maxdepth, depth);
	__syncthreads();
	const bool sink = t < ns;
	const int pi = lf.y + min(t, ns - 1);
	const int4 me = A.parts[pi];
	const float4 wv = A.w[pi];
	const float wi[3] = {sink ? wv.x : 0.0f, sink ? wv.y : 0.0f, sink ? wv.z : 0.0f};
	double gx[3] = {0.0, 0.0, 0.0};
	{
		const double d[3] = {double(float(double(centre_offset(me.x, c.x, A.wrap)) * POS_INV)),
				double(float(double(centre_offset(me.y, c.y, A.wrap)) * POS_INV)),
				double(float(double(centre_offset(me.z, c.z, A.wrap)) * POS_INV))};
		double W[35];
		taylor_weights(W, d);
		// g_a = -sum_{|s|<=3} L_{s u a} W_s  ->  dg_a/dd_b = -sum_{|s|<=2} L_{s u a u b} W_s
		for_n<3>([&](auto a_) {
			constexpr int a = decltype(a_)::value;
			for_n<3>([&](auto b_) {
				constexpr int b = decltype(b_)::value;
				double hab = 0.0;
				for_n<10>([&](auto s_) {
					constexpr int s = decltype(s_)::value;
					hab = fma(Ls[Merge<Merge<s, 1 + a>::value, 1 + b>::value], W[s], hab);
				});
				gx[b] -= double(wi[a]) * hab;
			});
		});
		// lambda_t = dg/dL_t^T w = -sum_a w_a W_{t minus a}
		double lam[35];
#pragma unroll
		for (int q = 0; q < 35; q++) lam[q] = 0.0;
		for_n<20>([&](auto s_) {
			constexpr int s = decltype(s_)::value;
			for_n<3>([&](auto a_) {
				constexpr int a = decltype(a_)::value;
				lam[Merge<s, 1 + a>::value] -= double(wi[a]) * W[s];
			});
		});
#pragma unroll
		for (int q = 0; q < 35; q++) lam64[q * 64 + t] = lam[q];
	}
	__syncthreads();
	// lambda of the leaf; k_adj_up carries it to the ancestors
	if (t < 35) A.Lam[35 * int64_t(lf.x) + t] = sum4(lam64 + t * 64, ns);
	if (sink) {
		double* o = A.grad + 4 * int64_t(pi);
		o[0] = gx[0];
		o[1] = gx[1];
		o[2] = gx[2];
		o[3] = 0.0;
	}
}

// leaf work items of one kind (the forward's: first sink, count [| upper bits], list begin, end)
struct AdjItems {
	const int4* items;
	const int* list;
	int nitems;
};

// the lanes of an item's wave: sinks padded to a power of two nsp, the P = 64 / nsp lane groups
// (phases) splitting the sources, so leaves of 32 or fewer particles keep every lane busy; the
// NW waves of the group share the list (tg_leaf_waves.hpp)
template <int NW, int TILE = 64>
struct LeafLanes {
	int lane, wave, ns, nsp, P, si, ph, pi;
	int2 share;
	__device__ __forceinline__ LeafLanes(const int4& it) {
		lane = threadIdx.x & 63;
		wave = NW == 1 ? 0 : int(threadIdx.x >> 6);
		ns = it.y & PP_COUNT_MASK;
		const int lg = ns <= 1 ? 0 : 32 - __clz(ns - 1);
		nsp = 1 << lg;
		P = 64 >> lg;
		si = lane & (nsp - 1);
		ph = lane >> lg;
		pi = it.x + min(si, ns - 1);
		share = wave_share<NW, TILE>(it.z, it.w, wave);
	}
	// the sums of all phases and waves onto the sink's gradient
	__device__ __forceinline__ void store(double gm, double* gx, double (*red)[4][64], double* grad) {
		leaf_sums<NW>(gm, gx, nsp, lane, wave, red);
		if (wave == 0 && ph == 0 && si < ns) {
			double* o = grad + 4 * int64_t(pi);
			o[0] += gx[0];
			o[1] += gx[1];
			o[2] += gx[2];
			o[3] += gm;
		}
	}
};

// PP direct: lane = (sink, phase), sources in LDS tiles of 64 with their weights.
// The lists are symmetric, so particle k's own list carries its source-side terms as well:
//   dL/dx_k += sum_j J(d_kj) (m_j w_k - m_k w_j),  J v = -f v - (f'/r)(d.v) d,
//   dL/dm_k += sum_j f(d_kj) (d_kj . w_j)
// Bound by FP32 arithmetic (about 45 instructions a pair) where enough waves are in flight: one
// wave per item left the longest lists of clustered sets to run alone.
template <int NW, bool WRAP>
__global__ __launch_bounds__(64 * NW) void k_adj_pp(AdjArgs A, AdjItems I) {
	const int4 it = I.items[blockIdx.x];
	LeafLanes<NW> T(it);
	const int near_len = int(unsigned(it.y) >> PP_NEAR_SHIFT);
	const int near_end = near_len == PP_NEAR_ALL ? INT_MAX : it.z + near_len;
	const int4 me = A.parts[T.pi];
	const float4 wv = A.w[T.pi];
	const float wi[3] = {wv.x, wv.y, wv.z};
	const float mi = __int_as_float(me.w);
	__shared__ int4 tps[NW][64];
	__shared__ float4 tws[NW][64];
	__shared__ double red[NW > 1 ? NW - 1 : 1][4][64];
	int4* tp = tps[T.wave];
	float4* tw = tws[T.wave];
	double gx[3] = {0.0, 0.0, 0.0}, gm = 0.0;
	for (int base = T.share.x; base < T.share.y; base += 64) {
		const int n = min(64, T.share.y - base);
		wave_lds_sync<NW>();
		if (T.lane < n) {
			const int j = I.list[base + T.lane];
			tp[T.lane] = A.parts[j];
			tw[T.lane] = A.w[j];
		}
		wave_lds_sync<NW>();
		float fx[3] = {0.f, 0.f, 0.f}, fm = 0.f;
		// tiles inside the list's near prefix may hold pairs closer than h (spline); later tiles
		// hold only pairs at least h apart (the forward's split)
		const bool near = base < near_end;
		auto pair = [&](int k, bool soft) {
			const int4 s = tp[k];
			const float4 ws = tw[k];
			const float mj = __int_as_float(s.w);
			const float d[3] = {sepf(me.x, s.x, WRAP), sepf(me.y, s.y, WRAP), sepf(me.z, s.z, WRAP)};
			const float v[3] = {mj * wi[0] - mi * ws.x, mj * wi[1] - mi * ws.y, mj * wi[2] - mi * ws.z};
			const float r2 = fmaf(d[2], d[2], fmaf(d[1], d[1], d[0] * d[0]));
			float f, fr;
			if (soft) {
				spline_f(r2, A.h, f, fr);
			} else {
				const float ri = __builtin_amdgcn_rsqf(r2);
				const float ri2 = ri * ri;
				f = ri2 * ri;
				fr = -3.0f * f * ri2;
			}
			const float dv = fmaf(d[2], v[2], fmaf(d[1], v[1], d[0] * v[0]));
			const float dw = fmaf(d[2], ws.z, fmaf(d[1], ws.y, d[0] * ws.x));
			const float frdv = fr * dv;
#pragma unroll
			for (int b = 0; b < 3; b++) fx[b] = fmaf(-f, v[b], fmaf(-frdv, d[b], fx[b]));
			fm = fmaf(f, dw, fm);
		};
		if (near) {
			for (int k = T.ph; k < n; k += T.P) pair(k, true);
		} else {
#pragma unroll 4
			for (int k = T.ph; k < n; k += T.P) pair(k, false);
		}
#pragma unroll
		for (int b = 0; b < 3; b++) gx[b] += fx[b];
		gm += fm;
	}
	T.store(gm, gx, red, A.grad);
}

// PP Ewald: the correction's F = -D1, J = -D2, per pair from the tabulated correction (its
// real-space images, Fourier terms and n = 0 term together, as the forward's k_pp_ewald reads them):
//   dL/dx_k += sum_j J(d_kj) (m_j w_k - m_k w_j),  dL/dm_k += sum_j w_j . D1(d_kj)
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_adj_pp_ewald(AdjArgs A, AdjItems I) {
	const int4 it = I.items[blockIdx.x];
	LeafLanes<NW, 8> T(it);
	const int4 me = A.parts[T.pi];
	const float4 wv = A.w[T.pi];
	const float wi[3] = {wv.x, wv.y, wv.z};
	const float mi = __int_as_float(me.w);
	__shared__ int4 tps[NW][64];
	__shared__ float4 tws[NW][64];
	__shared__ double red[NW > 1 ? NW - 1 : 1][4][64];
	__shared__ EwtStage<10> stages[NW];
	int4* tp = tps[T.wave];
	float4* tw = tws[T.wave];
	double gx[3] = {0.0, 0.0, 0.0}, gm = 0.0;
	for (int base = T.share.x; base < T.share.y; base += 64) {
		const int n = min(64, T.share.y - base);
		wave_lds_sync<NW>();
		if (T.lane < n) {
			const int j = I.list[base + T.lane];
			tp[T.lane] = A.parts[j];
			tw[T.lane] = A.w[j];
		}
		wave_lds_sync<NW>();
		float fx[3] = {0.f, 0.f, 0.f}, fm = 0.f;
		// the whole wave takes every turn (its table rows are read together), the next turn's rows on
		// their way while this turn's are evaluated
		auto at = [&](int k0, bool& on) {
			const int4 s = tp[min(k0 + T.ph, n - 1)];
			const float x[3] = {sepf(me.x, s.x, true), sepf(me.y, s.y, true), sepf(me.z, s.z, true)};
			const float r2 = fmaf(x[2], x[2], fmaf(x[1], x[1], x[0] * x[0]));
			on = k0 + T.ph < n && r2 > 1e-12f;  // the reference's constant below r = 1e-6: no derivatives
			return ewt_point(x);
		};
		bool on;
		EwtPoint p = at(0, on);
		EwtRows<10> rows;
		rows.fetch(p.row, c_adj_ewt, stages[T.wave], T.lane);
		for (int k0 = 0; k0 < n; k0 += T.P) {
			float c[EwtRead<10>::F4 * 4], D[10];
			rows.take(c, stages[T.wave], T.lane);
			const EwtPoint now = p;
			const bool add_it = on;
			const int k = min(k0 + T.ph, n - 1);
			const float mj = __int_as_float(tp[k].w);
			const float4 ws = tw[k];
			if (k0 + T.P < n) {
				p = at(k0 + T.P, on);
				rows.fetch(p.row, c_adj_ewt, stages[T.wave], T.lane);
			}
			ewt_eval<10>(D, c, now);
			if (!add_it) continue;
			const float v[3] = {mj * wi[0] - mi * ws.x, mj * wi[1] - mi * ws.y, mj * wi[2] - mi * ws.z};
			for_n<3>([&](auto b_) {
				constexpr int b = decltype(b_)::value;
				float jv = 0.0f;
				for_n<3>([&](auto a_) {
					constexpr int a = decltype(a_)::value;
					jv = fmaf(-D[cx<add(add(0, a), b)>], v[a], jv);
				});
				fx[b] += jv;
			});
			fm = fmaf(ws.x, D[1], fmaf(ws.y, D[2], fmaf(ws.z, D[3], fm)));
		}
#pragma unroll
		for (int b = 0; b < 3; b++) gx[b] += fx[b];
		gm += fm;
	}
	T.store(gm, gx, red, A.grad);
}

// PC, sink side: lane = (sink, phase), over the item's multipoles, dL/dx_i += w . dg/dx_i (fifth
// derivatives)
template <int NW, bool EWALD>
__global__ __launch_bounds__(64 * NW) void k_adj_pc_sink(AdjArgs A, AdjItems I) {
	const int4 it = I.items[blockIdx.x];
	LeafLanes<NW, 4> T(it);
	__shared__ double red[NW > 1 ? NW - 1 : 1][4][64];
	__shared__ EwtStage<adj::NS5> stages[EWALD ? NW : 1];
	const int4 me = A.parts[T.pi];
	const float4 wv = A.w[T.pi];
	const float wi[3] = {wv.x, wv.y, wv.z};
	double dx[3] = {0.0, 0.0, 0.0};
	const bool wrapx = EWALD || A.wrap;
	for (int base = T.share.x; base < T.share.y; base += 64) {
		const int end = min(base + 64, T.share.y);
		float gx[3] = {0.f, 0.f, 0.f};
		for (int e0 = base; e0 < end; e0 += T.P) {
			const int e = e0 + T.ph;
			if (!EWALD && e >= end) break;
			const MultiSrc& ms = A.multis[I.list[min(e, end - 1)]];
			float M[17];
#pragma unroll
			for (int q = 0; q < 17; q++) M[q] = ms.m[q];
			const float d[3] = {sepf(me.x, ms.x[0], wrapx), sepf(me.y, ms.x[1], wrapx), sepf(me.z, ms.x[2], wrapx)};
			float D[adj::NS5];
			if (EWALD)
				green_ewald_wave<adj::NS5>(D, d, c_adj_ewt, stages[EWALD ? T.wave : 0], T.lane);
			else
				adj::green_direct_n<adj::NS5>(D, d);
			if (!EWALD || e < end) m2p_sink_adjoint(gx, M, D, wi);
		}
#pragma unroll
		for (int b = 0; b < 3; b++) dx[b] += double(gx[b]);
	}
	T.store(0.0, dx, red, A.grad);
}

// PC source side by source node: mu_c += sum over the sinks i of every leaf whose PC list holds c of
// dg_i/dM_c^T w_i.  One work group per item (node c, a run of at most 16 sink leaves); the lanes
// cover 64 / L leaves at a time, L = 2^lgL lanes per leaf (L >= the largest leaf), one sink each;
// the 17 sums are reduced over the wave once per item and added with one atomic each.
struct AdjPCArgs {
	const int4* items;   // (node c, first sink leaf, end, 0)
	const int2* leaves;  // sink leaves: (first particle, count)
	const int4* parts;
	const float4* w;
	const MultiSrc* multis;
	double* mu;
	int lgL;
	int wrap;
};

template <bool EWALD>
__global__ __launch_bounds__(64) void k_adj_pc_t(AdjPCArgs A) {
	const int4 it = A.items[blockIdx.x];
	const int t = threadIdx.x;
	const int Q = 64 >> A.lgL;         // leaves per pass
	const int qq = t >> A.lgL;         // this lane's leaf within the pass
	const int o = t & ((1 << A.lgL) - 1);  // and its sink within the leaf
	const MultiSrc& ms = A.multis[it.x];
	const int cx0 = ms.x[0], cx1 = ms.x[1], cx2 = ms.x[2];
	const bool wrapx = EWALD || A.wrap;
	float mu[17];
#pragma unroll
	for (int q = 0; q < 17; q++) mu[q] = 0.0f;
	__shared__ EwtStage<35> stage[1];
	for (int k = it.y + qq; k - qq < it.z; k += Q) {
		const int2 lf = A.leaves[min(k, it.z - 1)];
		const bool on = k < it.z && o < lf.y;
		if (!EWALD && !on) continue;
		const int pi = lf.x + (on ? o : 0);
		const int4 me = A.parts[pi];
		const float4 wv = A.w[pi];
		const float wi[3] = {wv.x, wv.y, wv.z};
		const float d[3] = {sepf(me.x, cx0, wrapx), sepf(me.y, cx1, wrapx), sepf(me.z, cx2, wrapx)};
		float D[35];
		if (EWALD)
			green_ewald_wave<35>(D, d, c_adj_ewt, stage[0], t);
		else
			adj::green_direct_n<35>(D, d);
		if (on) m2p_source_adjoint(mu, D, wi);
	}
	__shared__ float red[17][65];
#pragma unroll
	for (int q = 0; q < 17; q++) red[q][t] = mu[q];
	__syncthreads();
	if (t < 17) {
		double acc = 0.0;
		for (int k = 0; k < 64; k++) acc += double(red[t][k]);
		atomicAdd(A.mu + 17 * int64_t(it.x) + t, acc);
	}
}

// ---- 2. node lists -------------------------------------------------------------------------------
// CP by source leaf: the forward adds m_j D(X_a - x_j) to the expansion of every node a whose CP
// list holds leaf B's range, so  dL/dm_j = sum_a Lambda_a . D(X_a - x_j)  and
// dL/dx_j = -m_j sum_a Lambda_a . grad D(X_a - x_j)  (fifth derivatives).  One work group per source
// leaf (item: first particle, count, sink-node list range); lanes are the leaf's particles, and the
// P = 64 / nsp lane groups split the sink nodes, staged 64 at a time in LDS.  Every particle belongs
// to one item, so the gradient is added without atomics.
struct AdjCPArgs {
	const int4* items;
	const uint64_t* keys;  // first particle << sink_bits | sink node, ascending
	int sink_bits;
	const int4* nodepos;
	const int4* parts;
	const double* Lam;
	double* grad;
	int wrap;
};

template <int NW, bool EWALD>
__global__ __launch_bounds__(64 * NW) void k_adj_cp_t(AdjCPArgs A) {
	const int4 it = A.items[blockIdx.x];
	if (it.z == it.w) return;  // no node takes this leaf
	const int t = threadIdx.x & 63;
	const int wave = NW == 1 ? 0 : int(threadIdx.x >> 6);
	const int2 share = wave_share<NW, 4>(it.z, it.w, wave);
	const int ns = it.y;
	const int lg = ns <= 1 ? 0 : 32 - __clz(ns - 1);
	const int nsp = 1 << lg;
	const int P = 64 >> lg;
	const int si = t & (nsp - 1);
	const int ph = t >> lg;
	const int pi = it.x + min(si, ns - 1);
	const int4 me = A.parts[pi];
	const bool wrapx = EWALD || A.wrap;
	__shared__ float lams[NW][64][36];
	__shared__ int4 xss[NW][64];
	__shared__ double red[NW > 1 ? NW - 1 : 1][4][64];
	__shared__ EwtStage<adj::NS5> stages[EWALD ? NW : 1];
	float (*lam)[36] = lams[wave];
	int4* xs = xss[wave];
	double gm = 0.0, g3[3] = {0.0, 0.0, 0.0};
	for (int base = share.x; base < share.y; base += 64) {
		const int n = min(64, share.y - base);
		wave_lds_sync<NW>();
		if (t < n) {
			const int a = int(A.keys[base + t] & ((uint64_t(1) << A.sink_bits) - 1));
			xs[t] = A.nodepos[a];
#pragma unroll
			for (int q = 0; q < 35; q++) lam[t][q] = float(A.Lam[35 * int64_t(a) + q]);
		}
		wave_lds_sync<NW>();
		float fm = 0.0f, f3[3] = {0.f, 0.f, 0.f};
		for (int k0 = 0; k0 < n; k0 += P) {
			if (!EWALD && k0 + ph >= n) break;
			const int k = min(k0 + ph, n - 1);
			const int4 X = xs[k];
			const float d[3] = {sepf(X.x, me.x, wrapx), sepf(X.y, me.y, wrapx), sepf(X.z, me.z, wrapx)};
			float D[adj::NS5];
			if (EWALD)
				green_ewald_wave<adj::NS5>(D, d, c_adj_ewt, stages[EWALD ? wave : 0], t);
			else
				adj::green_direct_n<adj::NS5>(D, d);
			if (EWALD && k0 + ph >= n) continue;
			for_n<35>([&](auto t_) {
				constexpr int tt = decltype(t_)::value;
				const float l = lam[k][tt];
				fm = fmaf(l, D[tt], fm);
				for_n<3>([&](auto b_) {
					constexpr int bb = decltype(b_)::value;
					f3[bb] = fmaf(l, D[cx<add(tt, bb)>], f3[bb]);
				});
			});
		}
		gm += fm;
#pragma unroll
		for (int q = 0; q < 3; q++) g3[q] += f3[q];
	}
	leaf_sums<NW>(gm, g3, nsp, t, wave, red);
	if (wave == 0 && ph == 0 && si < ns) {
		const double mj = double(__int_as_float(me.w));
		double* o = A.grad + 4 * int64_t(pi);
		o[0] -= mj * g3[0];
		o[1] -= mj * g3[1];
		o[2] -= mj * g3[2];
		o[3] += gm;
	}
}

// CC by source: the entries (source c, sink node a) sorted by source and cut into waves of <= 64; each
// lane forms M2L(., X_a - X_c)^T Lambda_a, then 17 lanes add the wave's entries source by source and
// issue one atomic per source segment and slot
struct AdjCCArgs {
	const uint64_t* keys;  // source << sink_bits | sink node, ascending
	int64_t n;
	int sink_bits;
	const int4* nodepos;
	const MultiSrc* multis;
	const double* Lam;
	double* mu;
	int wrap;
};

template <bool EWALD>
__global__ __launch_bounds__(64) void k_adj_cc_t(AdjCCArgs A) {
	const int64_t begin = 64 * int64_t(blockIdx.x);
	const int t = threadIdx.x;
	const int64_t j = begin + t;
	const int cnt = int(A.n - begin < 64 ? A.n - begin : 64);
	__shared__ float red[17][65];
	__shared__ int sc[64];
	__shared__ EwtStage<35> stage[1];
	float mu[17];
#pragma unroll
	for (int q = 0; q < 17; q++) mu[q] = 0.0f;
	int c = -1;
	if (EWALD || j < A.n) {  // the Ewald kind's wave reads its table rows together
		const uint64_t key = A.keys[j < A.n ? j : A.n - 1];
		c = int(key >> A.sink_bits);
		const int a = int(key & ((uint64_t(1) << A.sink_bits) - 1));
		const int4 X = A.nodepos[a];
		const MultiSrc& ms = A.multis[c];
		float Lam[35];
#pragma unroll
		for (int q = 0; q < 35; q++) Lam[q] = float(A.Lam[35 * int64_t(a) + q]);
		const bool wrapx = EWALD || A.wrap;
		const float d[3] = {sepf(X.x, ms.x[0], wrapx), sepf(X.y, ms.x[1], wrapx), sepf(X.z, ms.x[2], wrapx)};
		float D[35];
		if (EWALD)
			green_ewald_wave<35>(D, d, c_adj_ewt, stage[0], t);
		else
			adj::green_direct_n<35>(D, d);
		if (j < A.n)
			m2l_adjoint(mu, Lam, D);
		else
			c = -1;
	}
#pragma unroll
	for (int q = 0; q < 17; q++) red[q][t] = mu[q];
	sc[t] = c;
	__syncthreads();
	// segments of one source from a ballot of their first entries; lanes 0..16 add one slot each
	const bool first = t < cnt && (t == 0 || sc[t] != sc[t - 1]);
	unsigned long long starts = __ballot(first);
	if (t < 17) {
		while (starts) {
			const int b = __ffsll(starts) - 1;
			starts &= starts - 1;
			const int e = starts ? __ffsll(starts) - 1 : cnt;
			double a0 = 0.0, a1 = 0.0;
			int k = b;
			for (; k + 2 <= e; k += 2) {
				a0 += double(red[t][k]);
				a1 += double(red[t][k + 1]);
			}
			if (k < e) a0 += double(red[t][k]);
			atomicAdd(A.mu + 17 * int64_t(sc[b]) + t, a0 + a1);
		}
	}
}

// ---- up-sweep of Lambda ------------------------------------------------------------------------------
// The forward gives leaf B the expansion sum_a S(X_B - X_a) dL_a over its path, so dL/d(dL_a) =
// sum over leaves B below a of S(X_B - X_a)^T lambda_B.  Shifts compose exactly
// (S(X_B - X_a) = S(X_B - X_c) S(X_c - X_a) for a child c of a on the way), hence level by level,
// deepest first:  Lambda_a = sum_children S(X_c - X_a)^T Lambda_c,  with Lambda_B = lambda_B at the
// leaves.  One lane per child of a level (nodes are numbered level by level, the children of a node
// side by side); the two children of a node sit on adjacent lanes and are added with one exchange (an
// empty child's Lambda is zero).  No atomics: every Lambda is written once.
__global__ __launch_bounds__(64) void k_adj_up(const int* __restrict__ parent, int begin, int npairs, const int4* __restrict__ nodepos,
		double* __restrict__ Lam) {
	const int j = blockIdx.x * 64 + threadIdx.x;
	const int2 pc = j < npairs ? make_int2(parent[begin + j], begin + j) : make_int2(-1, -1);
	double out[35];
#pragma unroll
	for (int q = 0; q < 35; q++) out[q] = 0.0;
	if (pc.y >= 0) {
		const int4 Xa = nodepos[pc.x], Xc = nodepos[pc.y];
		// (S^T l)_u = sum_{t u s = u} l_t W_s(X_c - X_a), W the Taylor weights of the offset
		const double off[3] = {double(int64_t(Xc.x) - int64_t(Xa.x)) * POS_INV, double(int64_t(Xc.y) - int64_t(Xa.y)) * POS_INV,
				double(int64_t(Xc.z) - int64_t(Xa.z)) * POS_INV};
		double W[35];
		taylor_weights(W, off);
		const double* lc = Lam + 35 * int64_t(pc.y);
		for_n<35>([&](auto t_) {
			constexpr int tt = decltype(t_)::value;
			const double lt = lc[tt];
			for_n<35>([&](auto s_) {
				constexpr int s = decltype(s_)::value;
				if constexpr (Merge<tt, s>::valid) out[Merge<tt, s>::value] = fma(lt, W[s], out[Merge<tt, s>::value]);
			});
		});
	}
#pragma unroll
	for (int q = 0; q < 35; q++) out[q] += __shfl_xor(out[q], 1, 64);
	if ((j & 1) == 0 && j < npairs) {
		double* dst = Lam + 35 * int64_t(pc.x);
#pragma unroll
		for (int q = 0; q < 35; q++) dst[q] = out[q];
	}
}

// ---- 3. moments ----------------------------------------------------------------------------------
// multipole<float>::operator>>= transposed (tigergrav/multipole.hpp:414-433, restated in the host
// tree): M3'_pql = M3 + M0 Y_p Y_q Y_l + M2_pq Y_l + M2_ql Y_p + M2_lp Y_q, M2'_pq = M2 + M0 Y_p Y_q
__device__ __forceinline__ void m2m_adjoint(float* mu, const float* mup, const float* Y) {
	mu[0] = mup[0];
#pragma unroll
	for (int s = 0; s < 6; s++) mu[1 + s] = mup[1 + s];
#pragma unroll
	for (int s = 0; s < 10; s++) mu[7 + s] = mup[7 + s];
#pragma unroll
	for (int s = 0; s < 6; s++) mu[0] = fmaf(mup[1 + s] * Y[T2[s].i[0]], Y[T2[s].i[1]], mu[0]);
#pragma unroll
	for (int s = 0; s < 10; s++) {
		const int p = T3[s].i[0], q = T3[s].i[1], l = T3[s].i[2];
		const float u = mup[7 + s];
		mu[0] = fmaf(u * Y[p] * Y[q], Y[l], mu[0]);
		mu[1 + s2(p, q)] = fmaf(u, Y[l], mu[1 + s2(p, q)]);
		mu[1 + s2(q, l)] = fmaf(u, Y[p], mu[1 + s2(q, l)]);
		mu[1 + s2(l, p)] = fmaf(u, Y[q], mu[1 + s2(l, p)]);
	}
}

// The forward forms a parent's moments from its children's (M2M), so the multipole adjoint of a
// node is its own mu plus the M2M transpose of its parent's:  mu~_c = mu_c + M2M(X_c - X_a)^T mu~_a,
// level by level from the root; in place.
__global__ __launch_bounds__(64) void k_adj_down(const int* __restrict__ parent, int begin, int npairs, const int4* __restrict__ nodepos,
		double* __restrict__ mu) {
	const int j = blockIdx.x * 64 + threadIdx.x;
	if (j >= npairs) return;
	const int2 pc = make_int2(parent[begin + j], begin + j);
	const int4 Xa = nodepos[pc.x], Xc = nodepos[pc.y];
	const float Y[3] = {float(double(int64_t(Xc.x) - int64_t(Xa.x)) * POS_INV), float(double(int64_t(Xc.y) - int64_t(Xa.y)) * POS_INV),
			float(double(int64_t(Xc.z) - int64_t(Xa.z)) * POS_INV)};
	float m[17], n[17];
#pragma unroll
	for (int q = 0; q < 17; q++) m[q] = float(mu[17 * int64_t(pc.x) + q]);
	m2m_adjoint(n, m, Y);
	double* dst = mu + 17 * int64_t(pc.y);
#pragma unroll
	for (int q = 0; q < 17; q++) dst[q] += double(n[q]);
}

// P2M transposed onto a leaf's particles, from the leaf's swept multipole adjoint
__global__ __launch_bounds__(64) void k_adj_moments(AdjArgs A) {
	const int4 lf = A.leaves[blockIdx.x];
	const int t = threadIdx.x;
	__shared__ float mus[17];
	if (t < 17) mus[t] = float(A.mu[17 * int64_t(lf.x) + t]);
	__syncthreads();
	const int ns = lf.z - lf.y;
	if (t >= ns) return;
	const int pi = lf.y + t;
	const int4 me = A.parts[pi];
	const int4 c = A.nodepos[lf.x];
	const float mj = __int_as_float(me.w);
	// P2M (part_vect_multipole_info): M2_pq += m d_p d_q, M3_pql += m d_p d_q d_l, d = float(x - X)
	const float d[3] = {float(double(centre_offset(me.x, c.x, A.wrap)) * POS_INV), float(double(centre_offset(me.y, c.y, A.wrap)) * POS_INV),
			float(double(centre_offset(me.z, c.z, A.wrap)) * POS_INV)};
	float gm = mus[0], g3[3] = {0.f, 0.f, 0.f};
#pragma unroll
	for (int s = 0; s < 6; s++) {
		const int p = T2[s].i[0], q = T2[s].i[1];
		const float u = mus[1 + s];
		gm = fmaf(u * d[p], d[q], gm);
		g3[p] = fmaf(u, d[q], g3[p]);
		g3[q] = fmaf(u, d[p], g3[q]);
	}
#pragma unroll
	for (int s = 0; s < 10; s++) {
		const int p = T3[s].i[0], q = T3[s].i[1], l = T3[s].i[2];
		const float u = mus[7 + s];
		gm = fmaf(u * d[p] * d[q], d[l], gm);
		g3[p] = fmaf(u * d[q], d[l], g3[p]);
		g3[q] = fmaf(u * d[p], d[l], g3[q]);
		g3[l] = fmaf(u * d[p], d[q], g3[l]);
	}
	double* o = A.grad + 4 * int64_t(pi);
	o[0] += double(mj * g3[0]);
	o[1] += double(mj * g3[1]);
	o[2] += double(mj * g3[2]);
	o[3] += double(gm);
}

__global__ void k_adj_zero(double* p, int64_t n) {
	const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < n) p[i] = 0.0;
}

// ---- set-up: the lists by source, on the device ---------------------------------------------------
// What the source-side passes read follows from the walk's node-order lists by one sort per kind of
// (source, sink) pairs packed into one word, sink in the low sink_bits.  (On the host, with the lists
// and the tree copied there, this took 195 ms at 262,144 particles and most of an autograd pass.)

struct AdjKeyArgs {
	const int64_t* ptr;     // the kind's CSR over the nodes
	const int32_t* val;
	const WalkNode* nodes;
	const int* pleaf;
	int64_t nn;
	int sink_bits;
	int64_t* flag;          // set to 1 where a range is no whole leaf, or holds more than 64 particles where that counts
};

// kinds of node entries (CC, PC): one wave per sink node
__global__ __launch_bounds__(256) void k_adj_node_keys(AdjKeyArgs A, uint64_t* __restrict__ keys) {
	const int64_t a = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
	if (a >= A.nn) return;
	for (int64_t q = A.ptr[a] + (threadIdx.x & 63); q < A.ptr[a + 1]; q += 64) keys[q] = uint64_t(uint32_t(A.val[q])) << A.sink_bits | uint64_t(a);
}

// CP: (first particle of the source leaf, sink node); an empty range sorts past every leaf
__global__ __launch_bounds__(256) void k_adj_cp_keys(AdjKeyArgs A, uint64_t empty, uint64_t* __restrict__ keys) {
	const int64_t a = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
	if (a >= A.nn) return;
	for (int64_t q = A.ptr[a] / 2 + (threadIdx.x & 63); q < A.ptr[a + 1] / 2; q += 64) {
		const int b = A.val[2 * q], e = A.val[2 * q + 1];
		uint64_t key = empty;
		if (e > b) {
			const WalkNode& n = A.nodes[A.pleaf[b]];
			if (n.pbegin != b || n.pend != e || e - b > 64) *A.flag = 1;
			key = uint64_t(uint32_t(b)) << A.sink_bits | uint64_t(a);
		}
		keys[q] = key;
	}
}

// PP, for the symmetry check: (sink leaf, source leaf) and (source leaf, sink leaf)
__global__ __launch_bounds__(256) void k_adj_pp_keys(AdjKeyArgs A, uint64_t* __restrict__ fwd, uint64_t* __restrict__ rev) {
	const int64_t a = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
	if (a >= A.nn) return;
	for (int64_t q = A.ptr[a] / 2 + (threadIdx.x & 63); q < A.ptr[a + 1] / 2; q += 64) {
		const int b = A.val[2 * q], e = A.val[2 * q + 1];
		uint64_t src = 0;
		if (e > b) {
			src = uint64_t(A.pleaf[b]);
			const WalkNode& n = A.nodes[src];
			if (n.pbegin != b || n.pend != e) *A.flag = 1;
		} else {
			*A.flag = 1;
		}
		fwd[q] = uint64_t(a) << A.sink_bits | src;
		rev[q] = src << A.sink_bits | uint64_t(a);
	}
}

__global__ __launch_bounds__(256) void k_adj_differ(const uint64_t* __restrict__ a, const uint64_t* __restrict__ b, int64_t n, int64_t* flag) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i < n && a[i] != b[i]) *flag = 1;
}

// the first of n ascending keys that is at least k
__device__ __forceinline__ int64_t lower_bound(const uint64_t* keys, int64_t n, uint64_t k) {
	int64_t lo = 0, hi = n;
	while (lo < hi) {
		const int64_t mid = (lo + hi) >> 1;
		if (keys[mid] < k)
			lo = mid + 1;
		else
			hi = mid;
	}
	return lo;
}

// CP items, one per non-empty leaf in leaf order: (first particle, count, its run of keys); the
// largest leaf
__global__ __launch_bounds__(256) void k_adj_cp_items(const int4* __restrict__ leaves, int nl, const uint64_t* __restrict__ keys, int64_t n,
		int sink_bits, int4* __restrict__ items, unsigned long long* __restrict__ maxleaf) {
	const int i = int(blockIdx.x) * 256 + int(threadIdx.x);
	if (i >= nl) return;
	const int4 lf = leaves[i];
	if (maxleaf) atomicMax(maxleaf, (unsigned long long) (lf.z - lf.y));
	items[i] = make_int4(lf.y, lf.z - lf.y, int(lower_bound(keys, n, uint64_t(uint32_t(lf.y)) << sink_bits)),
			int(lower_bound(keys, n, uint64_t(uint32_t(lf.y) + 1) << sink_bits)));
}

// PC: 1 where an item (a run of at most 16 sink leaves of one source node) starts; the sink leaves
__global__ __launch_bounds__(256) void k_adj_pc_starts(const uint64_t* __restrict__ keys, int64_t n, int sink_bits,
		const WalkNode* __restrict__ nodes, int64_t* __restrict__ starts, int2* __restrict__ leaves) {
	const int64_t q = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (q >= n) return;
	const uint64_t key = keys[q], src = key >> sink_bits;
	const WalkNode& lf = nodes[key & ((uint64_t(1) << sink_bits) - 1)];
	leaves[q] = make_int2(lf.pbegin, lf.pend - lf.pbegin);
	const bool same = q > 0 && keys[q - 1] >> sink_bits == src;
	starts[q] = !same || (q - lower_bound(keys, n, src << sink_bits)) % 16 == 0;
}

__global__ __launch_bounds__(256) void k_adj_pc_items(const uint64_t* __restrict__ keys, int64_t n, int sink_bits,
		const int64_t* __restrict__ starts, const int64_t* __restrict__ place, int4* __restrict__ items) {
	const int64_t q = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (q >= n || !starts[q]) return;
	int64_t e = q + 1;
	while (e < n && !starts[e]) e++;
	items[place[q]] = make_int4(int(keys[q] >> sink_bits), int(q), int(e), 0);
}

// ---- input and output order -----------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_adj_weights(const float* __restrict__ w, const int64_t* __restrict__ order, int64_t n,
		float4* __restrict__ out) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	const int64_t o = order[i];
	out[i] = make_float4(w[3 * o], w[3 * o + 1], w[3 * o + 2], 0.0f);
}

__global__ __launch_bounds__(256) void k_adj_output(const double* __restrict__ g, const int64_t* __restrict__ order, int64_t n,
		double* __restrict__ out) {
	const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	const int64_t o = order[i];
	for (int c = 0; c < 4; c++) out[4 * o + c] = g[4 * i + c];
}

int bits_of(int64_t v) {  // bits that hold every value up to v
	int b = 1;
	while (v >> b) b++;
	return b;
}

}  // namespace

#define ACHK(call)                                                   \
	do {                                                             \
		hipError_t e_ = (call);                                      \
		if (e_ != hipSuccess) {                                      \
			err = std::string(#call) + ": " + hipGetErrorString(e_); \
			return e_ == hipErrorOutOfMemory ? TG_ENOMEM : TG_EHIP;  \
		}                                                            \
	} while (0)

// The lists by source, and what the adjoint asks of the tree (symmetric PP lists, leaves of at most
// 64 particles), once per tree.  The walk's lists are on the device, or are copied there from a host
// walk's.
int Solver::adjoint_lists() {
	if (adj_lists_ready) return TG_OK;
	hipStream_t s = stream;
	// scratch, freed once the stream has drained
	struct Scratch {
		hipStream_t s;
		std::vector<void*> blocks;
		~Scratch() {
			(void) hipStreamSynchronize(s);
			for (void* p : blocks) dev_free(p);
		}
		void* get(size_t bytes) {
			void* p = nullptr;
			if (dev_malloc(&p, std::max<size_t>(bytes, 16)) != hipSuccess) return nullptr;
			blocks.push_back(p);
			return p;
		}
	} scratch{s, {}};
	const int64_t nn = n_nodes;
	if (!dlists.ptr_all || dlists.nn != nn) {
		// a host walk's lists
		const Lists& Ls = tree.lists;
		const hvec<int64_t>* ptrs[8] = {&Ls.cc_d_ptr, &Ls.cp_d_ptr, &Ls.cc_e_ptr, &Ls.cp_e_ptr, &Ls.pc_d_ptr, &Ls.pp_d_ptr, &Ls.pc_e_ptr, &Ls.pp_e_ptr};
		const hvec<int32_t>* vals[8] = {&Ls.cc_d, &Ls.cp_d, &Ls.cc_e, &Ls.cp_e, &Ls.pc_d, &Ls.pp_d, &Ls.pc_e, &Ls.pp_e};
		for (int k = 0; k < 8; k++)
			if (int64_t(ptrs[k]->size()) != nn + 1) {
				err = "adjoint: the interaction lists do not belong to this tree";
				return TG_EINVAL;
			}
		// built aside and taken whole: after an error the next call starts again
		struct Fresh : DeviceLists {
			~Fresh() { release(); }
		} fresh;
		fresh.nn = nn;
		hvec<WalkNode> wn(static_cast<size_t>(nn));
		walk_nodes(tree, wn.data());
		ACHK(dev_malloc(&fresh.nodes, size_t(nn) * sizeof(WalkNode)));
		ACHK(dev_malloc(&fresh.ptr_all, size_t(8 * (nn + 1)) * 8));
		for (int k = 0; k < 8; k++) {
			fresh.len[k] = int64_t(vals[k]->size());
			ACHK(dev_malloc(&fresh.val[k], std::max<size_t>(size_t(fresh.len[k]) * 4, 16)));
		}
		ACHK(hipMemcpyAsync(fresh.nodes, wn.data(), size_t(nn) * sizeof(WalkNode), hipMemcpyHostToDevice, s));
		for (int k = 0; k < 8; k++) {
			ACHK(hipMemcpyAsync(fresh.ptr_all + int64_t(k) * (nn + 1), ptrs[k]->data(), size_t(nn + 1) * 8, hipMemcpyHostToDevice, s));
			if (fresh.len[k] > 0) ACHK(hipMemcpyAsync(fresh.val[k], vals[k]->data(), size_t(fresh.len[k]) * 4, hipMemcpyHostToDevice, s));
		}
		ACHK(hipStreamSynchronize(s));
		dlists.release();
		std::swap(dlists, static_cast<DeviceLists&>(fresh));
	}
	const int sink_bits = bits_of(nn), src_bits = bits_of(std::max(nn, n + 1));
	const int key_bits = sink_bits + src_bits;
	if (key_bits > 64) {
		err = "adjoint: more nodes and particles than a 64-bit pair key holds";
		return TG_EINVAL;
	}
	// [0], [1] PP lists (direct, Ewald) not symmetric; [2] a CP range that is no leaf of at most 64; [3] the
	// largest leaf; [4], [5] PC items
	int64_t* info = static_cast<int64_t*>(scratch.get(8 * 8));
	if (!info) ACHK(hipErrorOutOfMemory);
	hipLaunchKernelGGL(k_adj_zero, dim3(1), dim3(64), 0, s, reinterpret_cast<double*>(info), int64_t(8));
	ACHK(hipGetLastError());
	void* sort_tmp = nullptr;
	size_t sort_bytes = 0;
	auto sort = [&](const uint64_t* in, uint64_t* out, int64_t m) -> hipError_t {
		size_t need = 0;
		hipError_t e = hipcub::DeviceRadixSort::SortKeys(nullptr, need, in, out, m, 0, key_bits, s);
		if (e != hipSuccess) return e;
		if (need > sort_bytes) {
			sort_bytes = need;
			sort_tmp = scratch.get(need);
			if (!sort_tmp) return hipErrorOutOfMemory;
		}
		return hipcub::DeviceRadixSort::SortKeys(sort_tmp, need, in, out, m, 0, key_bits, s);
	};
	const dim3 node_grid(unsigned((nn + 3) / 4));
	auto grid = [](int64_t m) { return dim3(unsigned((m + 255) / 256)); };
	AdjKeyArgs A{nullptr, nullptr, dlists.nodes, d_pleaf.as<int>(), nn, sink_bits, nullptr};
	auto kind = [&](int k, int64_t* flag) {
		A.ptr = dlists.ptr(k);
		A.val = dlists.val[k];
		A.flag = flag;
	};
	enum { W_CC_D, W_CP_D, W_CC_E, W_CP_E, W_PC_D, W_PP_D, W_PC_E, W_PP_E };
	ScanSet pc_scan;
	int64_t* pc_starts[2] = {nullptr, nullptr};
	for (int e = 0; e < 2; e++) {
		// PP: symmetric, leaf by leaf
		kind(e ? W_PP_E : W_PP_D, info + e);
		if (const int64_t m = dlists.len[e ? W_PP_E : W_PP_D] / 2) {
			uint64_t* f = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			uint64_t* r = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			uint64_t* fs = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			uint64_t* rs = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			if (!f || !r || !fs || !rs) ACHK(hipErrorOutOfMemory);
			hipLaunchKernelGGL(k_adj_pp_keys, node_grid, dim3(256), 0, s, A, f, r);
			ACHK(hipGetLastError());
			ACHK(sort(f, fs, m));
			ACHK(sort(r, rs, m));
			hipLaunchKernelGGL(k_adj_differ, grid(m), dim3(256), 0, s, fs, rs, m, info + e);
			ACHK(hipGetLastError());
		}
		// CC by source
		kind(e ? W_CC_E : W_CC_D, nullptr);
		adj_cct_n[e] = dlists.len[e ? W_CC_E : W_CC_D];
		ACHK(d_adj_cct_keys[e].alloc(std::max<size_t>(size_t(adj_cct_n[e]) * 8, 16)));
		if (const int64_t m = adj_cct_n[e]) {
			uint64_t* k = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			if (!k) ACHK(hipErrorOutOfMemory);
			hipLaunchKernelGGL(k_adj_node_keys, node_grid, dim3(256), 0, s, A, k);
			ACHK(hipGetLastError());
			ACHK(sort(k, d_adj_cct_keys[e].as<uint64_t>(), m));
		}
		// CP by source leaf
		kind(e ? W_CP_E : W_CP_D, info + 2);
		adj_cpt_n[e] = dlists.len[e ? W_CP_E : W_CP_D] / 2;
		ACHK(d_adj_cpt_keys[e].alloc(std::max<size_t>(size_t(adj_cpt_n[e]) * 8, 16)));
		ACHK(d_adj_cpt_items[e].alloc(std::max<size_t>(size_t(n_leaf_items) * sizeof(int4), 16)));
		if (const int64_t m = adj_cpt_n[e]) {
			uint64_t* k = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
			if (!k) ACHK(hipErrorOutOfMemory);
			hipLaunchKernelGGL(k_adj_cp_keys, node_grid, dim3(256), 0, s, A, key_bits == 64 ? ~uint64_t(0) : (uint64_t(1) << key_bits) - 1, k);
			ACHK(hipGetLastError());
			ACHK(sort(k, d_adj_cpt_keys[e].as<uint64_t>(), m));
		}
		if (n_leaf_items > 0) {
			hipLaunchKernelGGL(k_adj_cp_items, grid(n_leaf_items), dim3(256), 0, s, d_leaf_items.as<int4>(), n_leaf_items,
					d_adj_cpt_keys[e].as<uint64_t>(), adj_cpt_n[e], sink_bits, d_adj_cpt_items[e].as<int4>(),
					e == 0 ? reinterpret_cast<unsigned long long*>(info + 3) : nullptr);
			ACHK(hipGetLastError());
		}
		// PC by source node
		kind(e ? W_PC_E : W_PC_D, nullptr);
		const int64_t m = dlists.len[e ? W_PC_E : W_PC_D];
		ACHK(d_adj_pct_leaves[e].alloc(std::max<size_t>(size_t(m) * sizeof(int2), 16)));
		ACHK(d_adj_pct_items[e].alloc(std::max<size_t>(size_t(m) * sizeof(int4), 16)));
		uint64_t* k = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
		uint64_t* ks = static_cast<uint64_t*>(scratch.get(size_t(m) * 8));
		pc_starts[e] = static_cast<int64_t*>(scratch.get(size_t(m) * 8));
		int64_t* place = static_cast<int64_t*>(scratch.get(size_t(m) * 8));
		if (!k || !ks || !pc_starts[e] || !place) ACHK(hipErrorOutOfMemory);
		ScanSet sc;
		sc.add(pc_starts[e], place, m);
		int64_t* ws = static_cast<int64_t*>(scratch.get(size_t(scan_workspace(sc)) * 8));
		if (!ws) ACHK(hipErrorOutOfMemory);
		if (m > 0) {
			hipLaunchKernelGGL(k_adj_node_keys, node_grid, dim3(256), 0, s, A, k);
			ACHK(hipGetLastError());
			ACHK(sort(k, ks, m));
			hipLaunchKernelGGL(k_adj_pc_starts, grid(m), dim3(256), 0, s, ks, m, sink_bits, dlists.nodes, pc_starts[e], d_adj_pct_leaves[e].as<int2>());
			ACHK(hipGetLastError());
			ACHK(scan_columns(sc, ws, info + 4 + e, s));
			hipLaunchKernelGGL(k_adj_pc_items, grid(m), dim3(256), 0, s, ks, m, sink_bits, pc_starts[e], place, d_adj_pct_items[e].as<int4>());
			ACHK(hipGetLastError());
		}
	}
	int64_t v[8];
	ACHK(hipMemcpyAsync(v, info, sizeof(v), hipMemcpyDeviceToHost, s));
	ACHK(hipStreamSynchronize(s));
	adj_pp_symmetric = v[0] == 0 && v[1] == 0;
	adj_cp_whole = v[2] == 0;
	adj_maxleaf = int(v[3]);
	adj_pct_nitems[0] = int(v[4]);
	adj_pct_nitems[1] = int(v[5]);
	adj_sink_bits = sink_bits;
	adj_lists_ready = true;
	return TG_OK;
}

namespace {

// launch for the number of waves per group, 1, 2, 4 or 8
template <class F>
void with_waves(int waves, F launch) {
	switch (waves) {
		case 1: launch(std::integral_constant<int, 1>{}); break;
		case 2: launch(std::integral_constant<int, 2>{}); break;
		case 4: launch(std::integral_constant<int, 4>{}); break;
		default: launch(std::integral_constant<int, 8>{}); break;
	}
}

}  // namespace

int Solver::adjoint(const float* w_in, double* grad_out, float* ms) {
	if (device < 0 || n == 0 || n_nodes == 0) {
		err = "adjoint needs a device solver with particles";
		return TG_EINVAL;
	}
	if (parts_per_node > 64) {
		err = "the adjoint handles leaves of at most 64 particles";
		return TG_EINVAL;
	}
	ACHK(hipSetDevice(device));
	{
		const int rc = adjoint_lists();
		if (rc != TG_OK) return rc;
	}
	if (adj_maxleaf > 64) {
		// only more coincident particles than a leaf holds make one (the tree's depth limit)
		err = "the adjoint handles leaves of at most 64 particles; a leaf at the tree's depth limit holds more";
		return TG_EINVAL;
	}
	if (!adj_pp_symmetric) {
		err = "the adjoint needs symmetric PP lists";
		return TG_EINVAL;
	}
	if (!adj_cp_whole) {
		err = "the adjoint needs CP sources that are whole leaves of at most 64 particles";
		return TG_EINVAL;
	}
	adj_pc_lgL = 0;
	while ((1 << adj_pc_lgL) < adj_maxleaf) adj_pc_lgL++;
	static thread_local int tables_ready = -1;
	if (tables_ready != device) {
		ACHK(init_adjoint_tables(device));
		tables_ready = device;
	}
	{
		const int rc = forces_device_order();  // the input index of each tree-order particle
		if (rc != TG_OK) return rc;
	}
	const int64_t nn = n_nodes;
	ACHK(d_adj_w.alloc(std::max<size_t>(n * sizeof(float4), 16)));
	ACHK(d_adj_grad.alloc(std::max<size_t>(n * 4 * sizeof(double), 16)));
	ACHK(d_adj_out.alloc(std::max<size_t>(n * 4 * sizeof(double), 16)));
	ACHK(d_adj_lam.alloc(std::max<size_t>(nn * 35 * sizeof(double), 16)));
	ACHK(d_adj_mu.alloc(std::max<size_t>(nn * 17 * sizeof(double), 16)));
	hipStream_t s = stream;
	const dim3 part_grid(unsigned((n + 255) / 256));
	// the weights as they come (host or device memory), put into tree order there; d_adj_out holds them so long
	ACHK(hipMemcpyAsync(d_adj_out.p, w_in, size_t(n) * 12, hipMemcpyDefault, s));
	hipLaunchKernelGGL(k_adj_weights, part_grid, dim3(256), 0, s, d_adj_out.as<const float>(), d_order.as<const int64_t>(), n, d_adj_w.as<float4>());
	ACHK(hipGetLastError());
	if (!adj_ev[0]) {
		ACHK(hipEventCreate(&adj_ev[0]));
		ACHK(hipEventCreate(&adj_ev[1]));
	}
	hipEvent_t e0 = adj_ev[0], e1 = adj_ev[1];
	if (ms) ACHK(hipEventRecord(e0, s));
	hipLaunchKernelGGL(k_adj_zero, dim3(unsigned((nn * 35 + 255) / 256)), dim3(256), 0, s, d_adj_lam.as<double>(), nn * 35);
	hipLaunchKernelGGL(k_adj_zero, dim3(unsigned((nn * 17 + 255) / 256)), dim3(256), 0, s, d_adj_mu.as<double>(), nn * 17);
	ACHK(hipGetLastError());
	AdjArgs a{};
	a.parts = d_parts.as<int4>();
	a.w = d_adj_w.as<float4>();
	a.multis = d_multis.as<MultiSrc>();
	a.nodepos = d_nodepos.as<int4>();
	a.dL = d_dL.as<double>();
	a.leaves = d_leaf_items.as<int4>();
	a.path = d_path.as<int>();
	a.level = d_level.as<int>();
	a.grad = d_adj_grad.as<double>();
	a.Lam = d_adj_lam.as<double>();
	a.mu = d_adj_mu.as<double>();
	a.h = float(soft_len);
	a.wrap = ewald;
	a.maxdepth = max_level + 1;
	const size_t lds = size_t(35 * 64 + 35 + 35 * a.maxdepth) * sizeof(double);
	if (n_leaf_items > 0) {
		hipLaunchKernelGGL(k_adj_l2p, dim3(n_leaf_items), dim3(64), lds, s, a);
		ACHK(hipGetLastError());
	}
	// children of each level, the deepest first
	const int* parent = d_parent.as<int>();
	const int levels = int(level_begin.size()) - 1;
	for (int l = levels - 1; l >= 1; l--) {
		const int b = level_begin[size_t(l)], np = level_begin[size_t(l) + 1] - b;
		hipLaunchKernelGGL(k_adj_up, dim3(unsigned((np + 63) / 64)), dim3(64), 0, s, parent, b, np, d_nodepos.as<int4>(), d_adj_lam.as<double>());
		ACHK(hipGetLastError());
	}
	for (int k : {PP_DIRECT, PP_EWALD, PC_DIRECT, PC_EWALD}) {
		if (work[k].nitems <= 0) continue;
		AdjItems I{work[k].items.as<int4>(), work[k].list.as<int>(), work[k].nitems};
		const dim3 g(work[k].nitems);
		// as the forward's; the Ewald kinds' rows and tiles take up to 10 KB of LDS a wave
		const int waves = k == PP_DIRECT ? leaf_waves(work[k].nitems, work[k].nlist, 8) :
				leaf_waves_fine(work[k].nitems, work[k].nlist, k == PC_DIRECT ? 8 : 4, k == PP_EWALD ? 64 : 8);
		with_waves(waves, [&](auto nw_) {
			constexpr int NW = decltype(nw_)::value, NWE = NW < 4 ? NW : 4;
			const dim3 b(64 * NW);
			if (k == PP_DIRECT && ewald)
				hipLaunchKernelGGL((k_adj_pp<NW, true>), g, b, 0, s, a, I);
			else if (k == PP_DIRECT)
				hipLaunchKernelGGL((k_adj_pp<NW, false>), g, b, 0, s, a, I);
			else if (k == PP_EWALD)
				hipLaunchKernelGGL((k_adj_pp_ewald<NWE>), g, dim3(64 * NWE), 0, s, a, I);
			else if (k == PC_DIRECT)
				hipLaunchKernelGGL((k_adj_pc_sink<NW, false>), g, b, 0, s, a, I);
			else
				hipLaunchKernelGGL((k_adj_pc_sink<NWE, true>), g, dim3(64 * NWE), 0, s, a, I);
		});
		ACHK(hipGetLastError());
	}
	for (int e = 0; e < 2; e++) {
		if (adj_cct_n[e] <= 0) continue;
		AdjCCArgs ca{d_adj_cct_keys[e].as<uint64_t>(), adj_cct_n[e], adj_sink_bits, d_nodepos.as<int4>(), d_multis.as<MultiSrc>(),
				d_adj_lam.as<double>(), d_adj_mu.as<double>(), ewald};
		const dim3 g(unsigned((adj_cct_n[e] + 63) / 64));
		if (e)
			hipLaunchKernelGGL(k_adj_cc_t<true>, g, dim3(64), 0, s, ca);
		else
			hipLaunchKernelGGL(k_adj_cc_t<false>, g, dim3(64), 0, s, ca);
		ACHK(hipGetLastError());
	}
	for (int e = 0; e < 2; e++) {
		if (adj_pct_nitems[e] <= 0) continue;
		AdjPCArgs pa{d_adj_pct_items[e].as<int4>(), d_adj_pct_leaves[e].as<int2>(), d_parts.as<int4>(), d_adj_w.as<float4>(),
				d_multis.as<MultiSrc>(), d_adj_mu.as<double>(), adj_pc_lgL, ewald};
		if (e)
			hipLaunchKernelGGL(k_adj_pc_t<true>, dim3(adj_pct_nitems[e]), dim3(64), 0, s, pa);
		else
			hipLaunchKernelGGL(k_adj_pc_t<false>, dim3(adj_pct_nitems[e]), dim3(64), 0, s, pa);
		ACHK(hipGetLastError());
	}
	for (int e = 0; e < 2; e++) {
		if (adj_cpt_n[e] <= 0 || n_leaf_items <= 0) continue;
		AdjCPArgs pa{d_adj_cpt_items[e].as<int4>(), d_adj_cpt_keys[e].as<uint64_t>(), adj_sink_bits, d_nodepos.as<int4>(), d_parts.as<int4>(),
				d_adj_lam.as<double>(), d_adj_grad.as<double>(), ewald};
		// four waves at most, 10 KB of staged expansions each; two where the table's rows take 8 KB more
		with_waves(leaf_waves_fine(n_leaf_items, adj_cpt_n[e], e ? 2 : 4, 8), [&](auto nw_) {
			constexpr int NW = decltype(nw_)::value < 4 ? decltype(nw_)::value : 4, NWE = NW < 2 ? NW : 2;
			if (e)
				hipLaunchKernelGGL((k_adj_cp_t<NWE, true>), dim3(n_leaf_items), dim3(64 * NWE), 0, s, pa);
			else
				hipLaunchKernelGGL((k_adj_cp_t<NW, false>), dim3(n_leaf_items), dim3(64 * NW), 0, s, pa);
		});
		ACHK(hipGetLastError());
	}
	for (int l = 1; l < levels; l++) {
		const int b = level_begin[size_t(l)], np = level_begin[size_t(l) + 1] - b;
		hipLaunchKernelGGL(k_adj_down, dim3(unsigned((np + 63) / 64)), dim3(64), 0, s, parent, b, np, d_nodepos.as<int4>(), d_adj_mu.as<double>());
		ACHK(hipGetLastError());
	}
	if (n_leaf_items > 0) {
		hipLaunchKernelGGL(k_adj_moments, dim3(n_leaf_items), dim3(64), 0, s, a);
		ACHK(hipGetLastError());
	}
	if (ms) ACHK(hipEventRecord(e1, s));
	hipLaunchKernelGGL(k_adj_output, part_grid, dim3(256), 0, s, d_adj_grad.as<const double>(), d_order.as<const int64_t>(), n, d_adj_out.as<double>());
	ACHK(hipGetLastError());
	ACHK(hipMemcpyAsync(grad_out, d_adj_out.p, size_t(n) * 4 * sizeof(double), hipMemcpyDefault, s));
	ACHK(hipStreamSynchronize(s));
	if (ms) ACHK(hipEventElapsedTime(ms, e0, e1));
	return TG_OK;
}

}  // namespace tg
