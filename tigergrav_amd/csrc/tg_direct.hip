// tg_direct.hip -- FP64 direct summation: the accuracy reference for a force solve.
//
// The reference checks a solve by comparing it with a direct sum over all particles
// (--solver_test, src/main.cpp:137-164, error statistics src/output.cpp:17-51).  This is that
// direct sum, in FP64, for a sample of sink particles against all N sources:
//   open:      spline-softened Newton (src/gravity.cpp:231-287, no self-potential offset);
//   periodic:  spline-softened Newton on the nearest image plus the converged Ewald correction
//              of the periodic Green's function minus 1/r (the function tigergrav's Ewald kernels
//              truncate, tigergrav/green.hpp:189-286), with its +pi/alpha^2 constant.
// The forces' Ewald sum is split at alpha = 12: the real-space part then lives on the nearest image
// alone within r = 1/2 (every omitted term is below erfc(6) / 0.5 ~ 4e-17), and the Fourier part over
// 0 < |h|^2 <= 576 (exp(-pi^2 577 / 144) ~ 7e-18) is separable: cos(2 pi h.(x_i - x_j)) summed over the
// signs of h's components is a product of cosines, so the structure factors are the eight sums
// T = sum_j m_j {cos, sin}(a x_j) {cos, sin}(b y_j) {cos, sin}(c z_j) per octant vector (a, b, c), eight FMAs each
// from per-particle tables of {cos, sin}(2 pi k x), k <= 24.  (alpha = 6 with its 27 images and a sincos
// per vector and particle took 285 ms for 256 sinks of 2M particles.)  The gradient's sum is
// split at alpha = 6: 27 images with |n_i| <= 1 (every omitted image is >= 1.5 away, erfc(9) ~ 1e-37),
// cut off at r = 1 (erfc(6) ~ 2e-17); the Fourier part over 0 < |h|^2 <= 144 (exp(-pi^2 145 / 36) ~
// 5e-18) through structure factors of one half-space of h with a factor 2.
// Every sum has a fixed order: results are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "tg_direct.h"
#include "tg_gravity.h"

namespace {

constexpr double kAlphaF = 12.0;  // the forces' split
constexpr int kHF = 24;           // their highest Fourier index per axis
constexpr int kHF2 = kHF * kHF;
constexpr int kZG = 9;            // z indices of one structure-factor task: three tasks cover 0..26
constexpr int kTab = 3 * kZG;     // table entries per axis, zero past kHF
constexpr double kAlpha = 6.0;    // the gradient's split
constexpr int kHMax2 = 144;
constexpr int kSFChunks = 128;   // the gradient's particle chunks of the structure-factor pass
constexpr int kSrcChunks = 64;   // and source chunks of the pair pass
constexpr double kPosInv = 1.0 / 4294967296.0;

thread_local std::string g_direct_err;

__device__ __forceinline__ double sep(int ewald, int a, int b) {
	return ewald ? double(int(unsigned(a) - unsigned(b))) * kPosInv : (double(a) - double(b)) * kPosInv;
}

// spline-softened Newton: f (g = -m dx f) and p (phi = -m p), as the reference's three branches
__device__ __forceinline__ void spline64(double r, double h, double& f, double& p) {
	if (r >= h) {
		f = 1.0 / (r * r * r);
		p = 1.0 / r;
		return;
	}
	const double q = r / h, q2 = q * q, q3 = q2 * q;
	if (r < 0.5 * h) {
		f = (32.0 / 3.0 - 192.0 / 5.0 * q2 + 32.0 * q3) / (h * h * h);
		p = (14.0 / 5.0 - 16.0 / 3.0 * q2 + 48.0 / 5.0 * q2 * q2 - 32.0 / 5.0 * q3 * q2) / h;
	} else {
		f = (64.0 / 3.0 * q3 - 48.0 * q3 * q + 192.0 / 5.0 * q3 * q2 - 32.0 / 3.0 * q3 * q3 - 1.0 / 15.0) / (r * r * r);
		p = (-1.0 / 15.0 + 16.0 / 5.0 * q - 32.0 / 3.0 * q3 + 16.0 * q3 * q - 48.0 / 5.0 * q3 * q2 + 32.0 / 15.0 * q3 * q3) / r;
	}
}

// the same inside the softening length, out of line: a handful of pairs in a million, and its erf
// would hold half the registers of the loop
__device__ __attribute__((noinline)) void softened_pair64(double r, double h, double& f, double& p) {
	const double a = kAlphaF, c = 1.1283791670955126 * kAlphaF;
	const double r2 = r * r, z2 = a * a * r2;
	spline64(r, h, f, p);
	double u, d;  // erf(alpha r) / r and -(1/r) d/dr of it
	if (z2 < 0.01) {  // as series in z^2
		u = c * (1.0 + z2 * (-1.0 / 3.0 + z2 * (1.0 / 10.0 + z2 * (-1.0 / 42.0 + z2 * (1.0 / 216.0 + z2 * (-1.0 / 1320.0 + z2 / 9360.0))))));
		d = -c * a * a *
		    (-2.0 / 3.0 + z2 * (4.0 / 10.0 + z2 * (-6.0 / 42.0 + z2 * (8.0 / 216.0 + z2 * (-10.0 / 1320.0 + z2 * (12.0 / 9360.0 - z2 * 14.0 / 75600.0))))));
	} else {
		u = erf(a * r) / r;
		d = (u - c * exp(-z2)) / r2;
	}
	p -= u;
	f -= d;
}

// the periodic pair within the cut-off (nearest image at distance r): g = -m dx f, phi = -m p, the
// spline-softened Newton pair less the Gaussian-smoothed one that the Fourier part sums.  Past h
// the difference is erfc(alpha r) / r.
__device__ __forceinline__ void ewald_pair64(double r2, double h, double& f, double& p) {
	const double a = kAlphaF, c = 1.1283791670955126 * kAlphaF;  // 2 alpha / sqrt(pi)
	const double r = sqrt(r2), z2 = a * a * r2;
	if (r >= h) {
		const double ri = 1.0 / r;
		p = erfc(a * r) * ri;
		f = (p + c * exp(-z2)) * (ri * ri);
		return;
	}
	softened_pair64(r, h, f, p);
}

// the real-space correction's gradient and Hessian for one pair at nearest-image offset x:
// du = grad u, hu = the 6 distinct entries of grad grad u (xx, xy, xz, yy, yz, zz); for a radial
// psi with d_k = (r^-1 d/dr)^k psi, grad psi = d1 y, grad grad psi = d2 y y^T + d1 I
//   n = 0:  psi = erf(a r)/r,   d_k = (-1)^k (2k-1)!! r^-(2k+1) [erf - g S_k]   (series for a r < 0.1)
//   n != 0: psi = -erfc(a r)/r, d_k = -(-1)^k (2k-1)!! r^-(2k+1) [erfc + g S_k]
// with g = (2a/sqrt(pi)) exp(-a^2 r^2), S_1 = r, S_2 = r + 2 a^2 r^3 / 3
__device__ void real_space2(const double* x, double* du, double* hu) {
	const double a = kAlpha, c = 1.1283791670955126 * kAlpha;
	for (int q = 0; q < 3; q++) du[q] = 0.0;
	for (int q = 0; q < 6; q++) hu[q] = 0.0;
	for (int i = -1; i <= 1; i++)
		for (int j = -1; j <= 1; j++)
			for (int k = -1; k <= 1; k++) {
				const double y[3] = {x[0] + i, x[1] + j, x[2] + k};
				const double r2 = y[0] * y[0] + y[1] * y[1] + y[2] * y[2];
				double d1, d2;
				if (i == 0 && j == 0 && k == 0) {
					const double z2 = a * a * r2;
					if (z2 < 0.01) {
						// erf(z)/r = c sum_k (-1)^k z^2k / (k! (2k+1)): differentiate term by term in u = r^2
						double s1 = 0.0, s2 = 0.0, zp = 1.0, zq = 1.0, fact = 1.0;  // zp = z^2(q-1), zq = z^2(q-2)
						for (int q = 1; q <= 14; q++) {
							fact *= q;
							const double sg = (q & 1) ? -1.0 : 1.0;
							s1 += sg * 2.0 * q / (fact * (2 * q + 1)) * zp;
							if (q >= 2) {
								s2 += sg * 4.0 * q * (q - 1) / (fact * (2 * q + 1)) * zq;
								zq *= z2;
							}
							zp *= z2;
						}
						d1 = c * a * a * s1;
						d2 = c * a * a * a * a * s2;
					} else {
						const double r = sqrt(r2), e = erf(a * r), g = c * exp(-z2);
						d1 = -(e - g * r) / (r2 * r);
						d2 = 3.0 * (e - g * (r + 2.0 * a * a * r2 * r / 3.0)) / (r2 * r2 * r);
					}
				} else {
					if (r2 >= 1.0) continue;
					const double r = sqrt(r2), ec = erfc(a * r), g = c * exp(-a * a * r2);
					d1 = (ec + g * r) / (r2 * r);
					d2 = -3.0 * (ec + g * (r + 2.0 * a * a * r2 * r / 3.0)) / (r2 * r2 * r);
				}
				du[0] += y[0] * d1;
				du[1] += y[1] * d1;
				du[2] += y[2] * d1;
				hu[0] += d2 * y[0] * y[0] + d1;
				hu[1] += d2 * y[0] * y[1];
				hu[2] += d2 * y[0] * y[2];
				hu[3] += d2 * y[1] * y[1] + d1;
				hu[4] += d2 * y[1] * y[2];
				hu[5] += d2 * y[2] * y[2] + d1;
			}
}

// spline pair in FP64: f (F = -d f) and fr = f'(r)/r
__device__ __forceinline__ void spline64_grad(double r, double h, double& f, double& fr) {
	if (r >= h) {
		f = 1.0 / (r * r * r);
		fr = -3.0 * f / (r * r);
		return;
	}
	const double q = r / h, q2 = q * q, q3 = q2 * q;
	if (r < 0.5 * h) {
		f = (32.0 / 3.0 - 192.0 / 5.0 * q2 + 32.0 * q3) / (h * h * h);
		fr = (-384.0 / 5.0 + 96.0 * q) / (h * h * h * h * h);
	} else {
		const double P = 64.0 / 3.0 * q3 - 48.0 * q3 * q + 192.0 / 5.0 * q3 * q2 - 32.0 / 3.0 * q3 * q3 - 1.0 / 15.0;
		const double dP = 64.0 * q2 - 192.0 * q3 + 192.0 * q3 * q - 64.0 * q3 * q2;
		f = P / (r * r * r);
		fr = (dP / h - 3.0 * P / r) / (r * r * r * r);
	}
}

// The forces' structure factors: thread = task (a, b, g), the eight sums of the octant vectors
// (a, b, 9 g .. 9 g + 8); block = 256 tasks x one particle chunk.  The block makes each particle's
// tables of (cos, sin)(2 pi k x) together, 75 sincospi a particle (2 k x is exact in FP64: x carries 32
// fraction bits, so sincospi reduces exactly), and every task takes 76 FP64 operations a particle from
// them: bound by FP64 arithmetic.  64 FMAs and 9 broadcast LDS reads a particle and task: nine z
// indices a task balance the two (one index a task would read as often as it multiplies), and their
// 72 sums fit the registers.
constexpr int kSFTile = 16;  // particles staged at a time
__global__ __launch_bounds__(256) void k_structure(const int4* __restrict__ tasks, int nt, const int* __restrict__ x,
		const float* __restrict__ mass, double m, int64_t n, double* __restrict__ part) {
	__shared__ double2 tab[kSFTile][3][kTab];
	const int t = blockIdx.x * 256 + threadIdx.x;
	const int4 task = tasks[min(t, nt - 1)];
	const int64_t per = (n + gridDim.y - 1) / gridDim.y;
	const int64_t b = int64_t(blockIdx.y) * per, e = min(n, b + per);
	double acc[kZG][8];
#pragma unroll
	for (int z = 0; z < kZG; z++)
#pragma unroll
		for (int q = 0; q < 8; q++) acc[z][q] = 0.0;
	for (int64_t base = b; base < e; base += kSFTile) {
		__syncthreads();
		for (int q = threadIdx.x; q < kSFTile * 3 * kTab; q += 256) {
			const int p = q / (3 * kTab), axis = q / kTab % 3, k = q % kTab;
			const int64_t j = base + p;
			double2 v = make_double2(0.0, 0.0);
			if (j < e && k <= kHF) {
				sincospi(2.0 * k * (double(x[3 * j + axis]) * kPosInv + 0.5), &v.y, &v.x);
				if (axis == 0) {
					const double mj = mass ? double(mass[j]) : m;
					v.x *= mj;
					v.y *= mj;
				}
			}
			tab[p][axis][k] = v;
		}
		__syncthreads();
		const int cnt = int(min<int64_t>(kSFTile, e - base));
		for (int p = 0; p < cnt; p++) {
			const double2 X = tab[p][0][task.x], Y = tab[p][1][task.y];
			const double w[4] = {X.x * Y.x, X.x * Y.y, X.y * Y.x, X.y * Y.y};
			const double2* zt = &tab[p][2][kZG * task.z];
#pragma unroll
			for (int z = 0; z < kZG; z++) {
				const double2 Z = zt[z];
#pragma unroll
				for (int q = 0; q < 4; q++) {
					acc[z][2 * q] = fma(w[q], Z.x, acc[z][2 * q]);
					acc[z][2 * q + 1] = fma(w[q], Z.y, acc[z][2 * q + 1]);
				}
			}
		}
	}
	if (t < nt) {
		// element-major within the chunk, so that neighbouring tasks write neighbouring words
		double* o = part + int64_t(blockIdx.y) * nt * (8 * kZG) + t;
#pragma unroll
		for (int z = 0; z < kZG; z++)
#pragma unroll
			for (int q = 0; q < 8; q++) o[int64_t(8 * z + q) * nt] = acc[z][q];
	}
}

// the chunks added in order: cs[task][z][8]
__global__ __launch_bounds__(256) void k_structure_sum(const double* __restrict__ part, int nt, int chunks, double* __restrict__ cs) {
	const int i = blockIdx.x * 256 + threadIdx.x;
	if (i >= nt * 8 * kZG) return;
	double s = 0.0;
	for (int c = 0; c < chunks; c++) s += part[int64_t(c) * nt * (8 * kZG) + i];
	cs[int64_t(i % nt) * (8 * kZG) + i / nt] = s;
}

// Pair pass: block = one wave, 64 / P sinks x P phases of one source chunk, P a power of two that
// fills the wave where there are fewer than 64 sinks.  Periodic pairs past the cut-off (r >= 1/2,
// half of them) are done after the distance.
template <bool EWALD>
__global__ __launch_bounds__(64) void k_pairs(const int* __restrict__ x, const float* __restrict__ mass, double m, int64_t n,
		const int64_t* __restrict__ sinks, int64_t ns, int lanes, double h, double* __restrict__ part) {
	const int P = 64 / lanes, ph = threadIdx.x / lanes;
	const int64_t si = int64_t(blockIdx.x) * lanes + threadIdx.x % lanes;
	const int64_t i = sinks[min(si, ns - 1)];
	const int xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
	const int64_t per = (n + gridDim.y - 1) / gridDim.y;
	const int64_t b = int64_t(blockIdx.y) * per, e = min(n, b + per);
	const double cut2 = fmax(0.25, h * h);
	__shared__ int sx[256][3];
	__shared__ double sm[256];
	double phi = 0.0, g[3] = {0.0, 0.0, 0.0};
	for (int64_t base = b; base < e; base += 256) {
		__syncthreads();
		for (int q = threadIdx.x; q < 256; q += 64) {
			const int64_t j = base + q;
			const bool in = j < e;
			sx[q][0] = in ? x[3 * j] : 0;
			sx[q][1] = in ? x[3 * j + 1] : 0;
			sx[q][2] = in ? x[3 * j + 2] : 0;
			sm[q] = in ? (mass ? double(mass[j]) : m) : 0.0;
		}
		__syncthreads();
		const int cnt = int(min<int64_t>(256, e - base));
		for (int q = ph; q < cnt; q += P) {
			const double dx[3] = {sep(EWALD, xi[0], sx[q][0]), sep(EWALD, xi[1], sx[q][1]), sep(EWALD, xi[2], sx[q][2])};
			const double r2 = dx[0] * dx[0] + dx[1] * dx[1] + dx[2] * dx[2];
			if (EWALD && r2 >= cut2) continue;
			double f, p;
			if (EWALD)
				ewald_pair64(r2, h, f, p);
			else
				spline64(sqrt(r2), h, f, p);
			const double mj = sm[q];
			f *= mj;
			phi = fma(-mj, p, phi);
			g[0] = fma(-dx[0], f, g[0]);
			g[1] = fma(-dx[1], f, g[1]);
			g[2] = fma(-dx[2], f, g[2]);
		}
	}
	for (int o = lanes; o < 64; o <<= 1) {
		phi += __shfl_xor(phi, o, 64);
		for (int d = 0; d < 3; d++) g[d] += __shfl_xor(g[d], o, 64);
	}
	if (ph == 0 && si < ns) {
		double* o = part + 4 * (si * gridDim.y + blockIdx.y);
		o[0] = phi;
		o[1] = g[0];
		o[2] = g[1];
		o[3] = g[2];
	}
}

// Per sink (a block each at a time): pair partials, then the Fourier part over the octant vectors, thread by
// thread, and the constant.  With K = exp(-pi^2 h^2 / alpha^2) / h^2 and every sign of (a, b, c) distinct
// (half for each zero component), phi = -(8 / pi) sum K C_x C_y C_z, where C = cos_i cos_j + sin_i sin_j per axis;
// the gradient along an axis takes k (cos_i sin_j - sin_i cos_j) there.
constexpr int64_t kFinishBlocks = 1 << 20;  // a launch takes fewer than 2^32 threads
__global__ __launch_bounds__(256) void k_finish(const int* __restrict__ x, const int64_t* __restrict__ sinks, int64_t ns, int chunks,
		const double* __restrict__ part, int ewald, const int4* __restrict__ tasks, const double* __restrict__ cs, int nt,
		double mtot, double* __restrict__ out) {
	__shared__ double2 tab[3][kTab];
	__shared__ double red[4][256];
	const int t = threadIdx.x;
	for (int64_t si = blockIdx.x; si < ns; si += gridDim.x) {
		__syncthreads();  // the last sink's tables and sums are read
		double v[4] = {0.0, 0.0, 0.0, 0.0};
		for (int c = t; c < chunks; c += 256)
			for (int q = 0; q < 4; q++) v[q] += part[4 * (si * chunks + c) + q];
		if (ewald) {
			if (t < 3 * kTab) {
				const int axis = t / kTab, k = t % kTab;
				double2 w = make_double2(0.0, 0.0);
				if (k <= kHF) sincospi(2.0 * k * (double(x[3 * sinks[si] + axis]) * kPosInv + 0.5), &w.y, &w.x);
				tab[axis][k] = w;
			}
			__syncthreads();
			const double pi = 3.141592653589793;
			for (int j = t; j < nt * kZG; j += 256) {
				const int4 task = tasks[j / kZG];
				const int a = task.x, b = task.y, c = kZG * task.z + j % kZG;
				const int h2 = a * a + b * b + c * c;
				if (h2 == 0 || h2 > kHF2) continue;
				const double K = exp(-pi * pi / (kAlphaF * kAlphaF) * h2) / h2 * (a ? 2.0 : 1.0) * (b ? 2.0 : 1.0) * (c ? 2.0 : 1.0);
				const double2 X = tab[0][a], Y = tab[1][b], Z = tab[2][c];
				const double* T = cs + int64_t(j) * 8;  // (cos, sin) of x, y, z from the highest bit down
				// contract z, then y, then x: P with C, Q with the derivative's sine
				double Pz[4], Qz[4], PP[2], QP[2], PQ[2];
				for (int q = 0; q < 4; q++) {
					Pz[q] = Z.x * T[2 * q] + Z.y * T[2 * q + 1];
					Qz[q] = Z.x * T[2 * q + 1] - Z.y * T[2 * q];
				}
				for (int q = 0; q < 2; q++) {
					PP[q] = Y.x * Pz[2 * q] + Y.y * Pz[2 * q + 1];
					QP[q] = Y.x * Pz[2 * q + 1] - Y.y * Pz[2 * q];
					PQ[q] = Y.x * Qz[2 * q] + Y.y * Qz[2 * q + 1];
				}
				v[0] -= K / pi * (X.x * PP[0] + X.y * PP[1]);
				v[1] += 2.0 * K * a * (X.x * PP[1] - X.y * PP[0]);
				v[2] += 2.0 * K * b * (X.x * QP[0] + X.y * QP[1]);
				v[3] += 2.0 * K * c * (X.x * PQ[0] + X.y * PQ[1]);
			}
		}
		for (int q = 0; q < 4; q++) red[q][t] = v[q];
		for (int o = 128; o > 0; o >>= 1) {
			__syncthreads();
			if (t < o)
				for (int q = 0; q < 4; q++) red[q][t] += red[q][t + o];
		}
		__syncthreads();
		if (t < 4) out[4 * si + t] = red[t][0] + (t == 0 && ewald ? mtot * 3.141592653589793 / (kAlphaF * kAlphaF) : 0.0);
	}
}

// gradient: structure factors C, S (mass weighted) and Cw, Sw (weight weighted), 8 per h
__global__ __launch_bounds__(64) void k_structure8(const int4* __restrict__ hv, int nh, const int* __restrict__ x,
		const float* __restrict__ mass, double m, const float* __restrict__ w, int64_t n, double* __restrict__ part) {
	const int t = blockIdx.x * 64 + threadIdx.x;
	const int64_t per = (n + kSFChunks - 1) / kSFChunks;
	const int64_t b = int64_t(blockIdx.y) * per, e = min(n, b + per);
	__shared__ double sx[128][7];
	const int4 h = t < nh ? hv[t] : make_int4(0, 0, 0, 0);
	double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
	for (int64_t base = b; base < e; base += 128) {
		__syncthreads();
		for (int q = threadIdx.x; q < 128; q += 64) {
			const int64_t j = base + q;
			const bool in = j < e;
			sx[q][0] = in ? double(x[3 * j]) * kPosInv + 0.5 : 0.0;
			sx[q][1] = in ? double(x[3 * j + 1]) * kPosInv + 0.5 : 0.0;
			sx[q][2] = in ? double(x[3 * j + 2]) * kPosInv + 0.5 : 0.0;
			sx[q][3] = in ? (mass ? double(mass[j]) : m) : 0.0;
			sx[q][4] = in ? double(w[3 * j]) : 0.0;
			sx[q][5] = in ? double(w[3 * j + 1]) : 0.0;
			sx[q][6] = in ? double(w[3 * j + 2]) : 0.0;
		}
		__syncthreads();
		const int cnt = int(min<int64_t>(128, e - base));
		for (int q = 0; q < cnt; q++) {
			double sn, cs;
			sincospi(2.0 * (h.x * sx[q][0] + h.y * sx[q][1] + h.z * sx[q][2]), &sn, &cs);
			acc[0] = fma(sx[q][3], cs, acc[0]);
			acc[1] = fma(sx[q][3], sn, acc[1]);
			for (int d = 0; d < 3; d++) {
				acc[2 + d] = fma(sx[q][4 + d], cs, acc[2 + d]);
				acc[5 + d] = fma(sx[q][4 + d], sn, acc[5 + d]);
			}
		}
	}
	if (t < nh)
		for (int q = 0; q < 8; q++) part[8 * (int64_t(blockIdx.y) * nh + t) + q] = acc[q];
}

__global__ __launch_bounds__(256) void k_structure8_sum(const double* __restrict__ part, int nh, double* __restrict__ cs) {
	const int t = blockIdx.x * 256 + threadIdx.x;
	if (t >= nh) return;
	double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
	for (int c = 0; c < kSFChunks; c++)
		for (int q = 0; q < 8; q++) acc[q] += part[8 * (int64_t(c) * nh + t) + q];
	for (int q = 0; q < 8; q++) cs[8 * t + q] = acc[q];
}

// gradient pair pass: d/dx_k += J(d_kj) (m_j w_k - m_k w_j),  d/dm_k += -w_j . F(d_kj)
__global__ __launch_bounds__(64) void k_pairs_grad(const int* __restrict__ x, const float* __restrict__ mass, double m,
		const float* __restrict__ w, int64_t n, const int64_t* __restrict__ sinks, int64_t ns, int ewald, double h,
		double* __restrict__ part) {
	const int64_t si = int64_t(blockIdx.x) * 64 + threadIdx.x;
	const int64_t i = sinks[min(si, ns - 1)];
	const int xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
	const double mi = mass ? double(mass[i]) : m;
	const double wi[3] = {w[3 * i], w[3 * i + 1], w[3 * i + 2]};
	const int64_t per = (n + kSrcChunks - 1) / kSrcChunks;
	const int64_t b = int64_t(blockIdx.y) * per, e = min(n, b + per);
	__shared__ int sx[256][3];
	__shared__ double sm[256], sw[256][3];
	double g[3] = {0.0, 0.0, 0.0}, gm = 0.0;
	for (int64_t base = b; base < e; base += 256) {
		__syncthreads();
		for (int q = threadIdx.x; q < 256; q += 64) {
			const int64_t j = base + q;
			const bool in = j < e;
			sx[q][0] = in ? x[3 * j] : 0;
			sx[q][1] = in ? x[3 * j + 1] : 0;
			sx[q][2] = in ? x[3 * j + 2] : 0;
			sm[q] = in ? (mass ? double(mass[j]) : m) : 0.0;
			for (int d = 0; d < 3; d++) sw[q][d] = in ? double(w[3 * j + d]) : 0.0;
		}
		__syncthreads();
		const int cnt = int(min<int64_t>(256, e - base));
		for (int q = 0; q < cnt; q++) {
			const double dx[3] = {sep(ewald, xi[0], sx[q][0]), sep(ewald, xi[1], sx[q][1]), sep(ewald, xi[2], sx[q][2])};
			const double mj = sm[q];
			const double v[3] = {mj * wi[0] - mi * sw[q][0], mj * wi[1] - mi * sw[q][1], mj * wi[2] - mi * sw[q][2]};
			const double r = sqrt(dx[0] * dx[0] + dx[1] * dx[1] + dx[2] * dx[2]);
			double f, fr;
			spline64_grad(r, h, f, fr);
			const double dv = dx[0] * v[0] + dx[1] * v[1] + dx[2] * v[2];
			const double dw = dx[0] * sw[q][0] + dx[1] * sw[q][1] + dx[2] * sw[q][2];
			for (int d = 0; d < 3; d++) g[d] += -f * v[d] - fr * dv * dx[d];
			gm += f * dw;
			if (ewald) {
				// correction: F = -grad u, J = -grad grad u
				double du[3], hu[6];
				real_space2(dx, du, hu);
				g[0] -= hu[0] * v[0] + hu[1] * v[1] + hu[2] * v[2];
				g[1] -= hu[1] * v[0] + hu[3] * v[1] + hu[4] * v[2];
				g[2] -= hu[2] * v[0] + hu[4] * v[1] + hu[5] * v[2];
				gm += du[0] * sw[q][0] + du[1] * sw[q][1] + du[2] * sw[q][2];
			}
		}
	}
	if (si < ns) {
		double* o = part + 4 * (si * kSrcChunks + blockIdx.y);
		o[0] = g[0];
		o[1] = g[1];
		o[2] = g[2];
		o[3] = gm;
	}
}

// per sink: pair partials, then the Fourier part: with c0 = 2 exp(-pi^2 h^2/a^2)/h^2 per half-space h
//   d/dx_k += -4 pi c0 h [(h.w_k)(cos_k C + sin_k S) - m_k (cos_k h.Cw + sin_k h.Sw)]
//   d/dm_k += 2 c0 [sin_k h.Cw - cos_k h.Sw]
__global__ __launch_bounds__(64) void k_finish_grad(const int* __restrict__ x, const float* __restrict__ mass, double m,
		const float* __restrict__ w, const int64_t* __restrict__ sinks, int64_t ns, const double* __restrict__ part, int ewald,
		const int4* __restrict__ hv, const double* __restrict__ cs8, int nh, double* __restrict__ out) {
	const int64_t si = int64_t(blockIdx.x) * 64 + threadIdx.x;
	if (si >= ns) return;
	double g[4] = {0.0, 0.0, 0.0, 0.0};
	for (int c = 0; c < kSrcChunks; c++)
		for (int q = 0; q < 4; q++) g[q] += part[4 * (si * kSrcChunks + c) + q];
	if (ewald) {
		const int64_t i = sinks[si];
		const double xi[3] = {double(x[3 * i]) * kPosInv + 0.5, double(x[3 * i + 1]) * kPosInv + 0.5,
				double(x[3 * i + 2]) * kPosInv + 0.5};
		const double mi = mass ? double(mass[i]) : m;
		const double wi[3] = {w[3 * i], w[3 * i + 1], w[3 * i + 2]};
		const double pi = 3.141592653589793, a2 = kAlpha * kAlpha;
		for (int t = 0; t < nh; t++) {
			const int4 h = hv[t];
			const double hd[3] = {double(h.x), double(h.y), double(h.z)};
			const double h2 = hd[0] * hd[0] + hd[1] * hd[1] + hd[2] * hd[2];
			const double c0 = 2.0 * exp(-pi * pi * h2 / a2) / h2;
			double sn, cs;
			sincospi(2.0 * (hd[0] * xi[0] + hd[1] * xi[1] + hd[2] * xi[2]), &sn, &cs);
			const double* S8 = cs8 + 8 * t;
			const double hw = hd[0] * wi[0] + hd[1] * wi[1] + hd[2] * wi[2];
			const double hCw = hd[0] * S8[2] + hd[1] * S8[3] + hd[2] * S8[4];
			const double hSw = hd[0] * S8[5] + hd[1] * S8[6] + hd[2] * S8[7];
			// F_F(d) = -2 sum_half c0 h sin(2 pi h.d), J_F(d) = -4 pi sum_half c0 h h^T cos(2 pi h.d)
			const double coef = -4.0 * pi * c0 * (hw * (cs * S8[0] + sn * S8[1]) - mi * (cs * hCw + sn * hSw));
			for (int d = 0; d < 3; d++) g[d] += coef * hd[d];
			g[3] += 2.0 * c0 * (sn * hCw - cs * hSw);
		}
	}
	double* o = out + 4 * si;
	for (int q = 0; q < 4; q++) o[q] = g[q];
}

struct Buf {
	void* p = nullptr;
	~Buf() {
		if (p) (void) hipFree(p);
	}
};

}  // namespace

extern "C" int tg_direct_forces(const tg_params* prm, const int32_t* x, const float* mass, int64_t n, const int64_t* sinks,
		int64_t ns, tg_force* out) {
	if (!prm || !x || !sinks || !out || n <= 0 || ns <= 0 || !(prm->soft_len > 0.0)) return TG_EINVAL;
	for (int64_t k = 0; k < ns; k++)
		if (sinks[k] < 0 || sinks[k] >= n) {
			g_direct_err = "sink index out of range";
			return TG_EINVAL;
		}
	const int ewald = prm->ewald ? 1 : 0;
	double mtot = 0.0;
	if (mass)
		for (int64_t j = 0; j < n; j++) mtot += mass[j];
	else
		mtot = prm->m * double(n);
	// the structure-factor tasks: octant columns (a, b) in runs of kZG z indices that reach into the sphere
	std::vector<int4> hv;
	if (ewald)
		for (int g = 0; kZG * g <= kHF; g++)
			for (int i = 0; i <= kHF; i++)
				for (int j = 0; j <= kHF; j++)
					if (i * i + j * j + kZG * g * kZG * g <= kHF2) hv.push_back(make_int4(i, j, g, 0));
	const int nt = int(hv.size());
	// Particle chunks of the structure factors: one round of the chip (two blocks of four waves per CU by
	// its registers), a chunk of 64 particles or more.  Source chunks of the pair pass: 16,384 waves (four rounds of the chip at four
	// waves a SIMD), a chunk of 512 sources or more.
	const int sf_chunks = int(std::max<int64_t>(1, std::min<int64_t>(512 / std::max(1, (nt + 255) / 256), n / 64)));
	int lanes = 1;
	while (lanes < 64 && lanes < ns) lanes *= 2;
	const int64_t sblocks = (ns + lanes - 1) / lanes;
	const int src_chunks = int(std::max<int64_t>(1, std::min<int64_t>((16384 + sblocks - 1) / sblocks, n / 512)));
	Buf dx, dm, ds, dh, dsf, dcs, dpart, dout;
	hipStream_t st = nullptr;
	int rc = TG_OK;
#define DCHK(call)                                                   \
	do {                                                             \
		hipError_t e_ = (call);                                      \
		if (e_ != hipSuccess) {                                      \
			g_direct_err = std::string(#call) + ": " + hipGetErrorString(e_); \
			rc = e_ == hipErrorOutOfMemory ? TG_ENOMEM : TG_EHIP;    \
			goto done;                                               \
		}                                                            \
	} while (0)
	{
		DCHK(hipSetDevice(prm->device));
		DCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
		DCHK(hipMalloc(&dx.p, size_t(n) * 12));
		DCHK(hipMemcpyAsync(dx.p, x, size_t(n) * 12, hipMemcpyHostToDevice, st));
		if (mass) {
			DCHK(hipMalloc(&dm.p, size_t(n) * 4));
			DCHK(hipMemcpyAsync(dm.p, mass, size_t(n) * 4, hipMemcpyHostToDevice, st));
		}
		DCHK(hipMalloc(&ds.p, size_t(ns) * 8));
		DCHK(hipMemcpyAsync(ds.p, sinks, size_t(ns) * 8, hipMemcpyHostToDevice, st));
		if (ewald) {
			DCHK(hipMalloc(&dh.p, hv.size() * sizeof(int4)));
			DCHK(hipMemcpyAsync(dh.p, hv.data(), hv.size() * sizeof(int4), hipMemcpyHostToDevice, st));
			DCHK(hipMalloc(&dcs.p, size_t(nt) * 8 * kZG * 8));
			DCHK(hipMalloc(&dsf.p, size_t(sf_chunks) * nt * 8 * kZG * 8));
			hipLaunchKernelGGL(k_structure, dim3((nt + 255) / 256, sf_chunks), dim3(256), 0, st, static_cast<const int4*>(dh.p), nt,
					static_cast<const int*>(dx.p), static_cast<const float*>(dm.p), prm->m, n, static_cast<double*>(dsf.p));
			DCHK(hipGetLastError());
			hipLaunchKernelGGL(k_structure_sum, dim3((nt * 8 * kZG + 255) / 256), dim3(256), 0, st, static_cast<const double*>(dsf.p), nt,
					sf_chunks, static_cast<double*>(dcs.p));
			DCHK(hipGetLastError());
		}
		DCHK(hipMalloc(&dpart.p, size_t(ns) * src_chunks * 32));
		if (ewald)
			hipLaunchKernelGGL(k_pairs<true>, dim3(unsigned(sblocks), src_chunks), dim3(64), 0, st, static_cast<const int*>(dx.p),
					static_cast<const float*>(dm.p), prm->m, n, static_cast<const int64_t*>(ds.p), ns, lanes, prm->soft_len,
					static_cast<double*>(dpart.p));
		else
			hipLaunchKernelGGL(k_pairs<false>, dim3(unsigned(sblocks), src_chunks), dim3(64), 0, st, static_cast<const int*>(dx.p),
					static_cast<const float*>(dm.p), prm->m, n, static_cast<const int64_t*>(ds.p), ns, lanes, prm->soft_len,
					static_cast<double*>(dpart.p));
		DCHK(hipGetLastError());
		DCHK(hipMalloc(&dout.p, size_t(ns) * 32));
		hipLaunchKernelGGL(k_finish, dim3(unsigned(std::min(ns, kFinishBlocks))), dim3(256), 0, st, static_cast<const int*>(dx.p),
				static_cast<const int64_t*>(ds.p), ns, src_chunks, static_cast<const double*>(dpart.p), ewald, static_cast<const int4*>(dh.p),
				static_cast<const double*>(dcs.p), nt, mtot, static_cast<double*>(dout.p));
		DCHK(hipGetLastError());
		DCHK(hipMemcpyAsync(out, dout.p, size_t(ns) * 32, hipMemcpyDeviceToHost, st));
		DCHK(hipStreamSynchronize(st));
	}
done:
#undef DCHK
	if (st) (void) hipStreamDestroy(st);
	return rc;
}

extern "C" int tg_direct_gradient(const tg_params* prm, const int32_t* x, const float* mass, int64_t n, const float* w,
		const int64_t* sinks, int64_t ns, double* out) {
	if (!prm || !x || !w || !sinks || !out || n <= 0 || ns <= 0 || !(prm->soft_len > 0.0)) return TG_EINVAL;
	for (int64_t k = 0; k < ns; k++)
		if (sinks[k] < 0 || sinks[k] >= n) {
			g_direct_err = "sink index out of range";
			return TG_EINVAL;
		}
	const int ewald = prm->ewald ? 1 : 0;
	std::vector<int4> hv;
	for (int i = -12; i <= 12; i++)
		for (int j = -12; j <= 12; j++)
			for (int k = -12; k <= 12; k++) {
				const int h2 = i * i + j * j + k * k;
				if (h2 == 0 || h2 > kHMax2) continue;
				if (i < 0 || (i == 0 && (j < 0 || (j == 0 && k < 0)))) continue;
				hv.push_back(make_int4(i, j, k, 0));
			}
	const int nh = int(hv.size());
	Buf dx, dm, dw, ds, dh, dsf, dcs, dpart, dout;
	hipStream_t st = nullptr;
	int rc = TG_OK;
#define DCHK(call)                                                   \
	do {                                                             \
		hipError_t e_ = (call);                                      \
		if (e_ != hipSuccess) {                                      \
			g_direct_err = std::string(#call) + ": " + hipGetErrorString(e_); \
			rc = e_ == hipErrorOutOfMemory ? TG_ENOMEM : TG_EHIP;    \
			goto done;                                               \
		}                                                            \
	} while (0)
	{
		DCHK(hipSetDevice(prm->device));
		DCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
		DCHK(hipMalloc(&dx.p, size_t(n) * 12));
		DCHK(hipMemcpyAsync(dx.p, x, size_t(n) * 12, hipMemcpyHostToDevice, st));
		DCHK(hipMalloc(&dw.p, size_t(n) * 12));
		DCHK(hipMemcpyAsync(dw.p, w, size_t(n) * 12, hipMemcpyHostToDevice, st));
		if (mass) {
			DCHK(hipMalloc(&dm.p, size_t(n) * 4));
			DCHK(hipMemcpyAsync(dm.p, mass, size_t(n) * 4, hipMemcpyHostToDevice, st));
		}
		DCHK(hipMalloc(&ds.p, size_t(ns) * 8));
		DCHK(hipMemcpyAsync(ds.p, sinks, size_t(ns) * 8, hipMemcpyHostToDevice, st));
		DCHK(hipMalloc(&dh.p, hv.size() * sizeof(int4)));
		DCHK(hipMemcpyAsync(dh.p, hv.data(), hv.size() * sizeof(int4), hipMemcpyHostToDevice, st));
		DCHK(hipMalloc(&dcs.p, size_t(nh) * 64));
		if (ewald) {
			DCHK(hipMalloc(&dsf.p, size_t(kSFChunks) * nh * 64));
			hipLaunchKernelGGL(k_structure8, dim3((nh + 63) / 64, kSFChunks), dim3(64), 0, st, static_cast<const int4*>(dh.p), nh,
					static_cast<const int*>(dx.p), static_cast<const float*>(dm.p), prm->m, static_cast<const float*>(dw.p), n,
					static_cast<double*>(dsf.p));
			DCHK(hipGetLastError());
			hipLaunchKernelGGL(k_structure8_sum, dim3((nh + 255) / 256), dim3(256), 0, st, static_cast<const double*>(dsf.p), nh,
					static_cast<double*>(dcs.p));
			DCHK(hipGetLastError());
		}
		DCHK(hipMalloc(&dpart.p, size_t(ns) * kSrcChunks * 32));
		const unsigned sblocks = unsigned((ns + 63) / 64);
		hipLaunchKernelGGL(k_pairs_grad, dim3(sblocks, kSrcChunks), dim3(64), 0, st, static_cast<const int*>(dx.p),
				static_cast<const float*>(dm.p), prm->m, static_cast<const float*>(dw.p), n, static_cast<const int64_t*>(ds.p), ns, ewald,
				prm->soft_len, static_cast<double*>(dpart.p));
		DCHK(hipGetLastError());
		DCHK(hipMalloc(&dout.p, size_t(ns) * 32));
		hipLaunchKernelGGL(k_finish_grad, dim3(sblocks), dim3(64), 0, st, static_cast<const int*>(dx.p),
				static_cast<const float*>(dm.p), prm->m, static_cast<const float*>(dw.p), static_cast<const int64_t*>(ds.p), ns,
				static_cast<const double*>(dpart.p), ewald, static_cast<const int4*>(dh.p), static_cast<const double*>(dcs.p), nh,
				static_cast<double*>(dout.p));
		DCHK(hipGetLastError());
		DCHK(hipMemcpyAsync(out, dout.p, size_t(ns) * 32, hipMemcpyDeviceToHost, st));
		DCHK(hipStreamSynchronize(st));
	}
done:
#undef DCHK
	if (st) (void) hipStreamDestroy(st);
	return rc;
}

extern "C" const char* tg_direct_last_error(void) { return g_direct_err.c_str(); }
