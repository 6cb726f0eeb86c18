// Per-pair quantities of FFS order parameters on gfx950, in FP64.
//
// The reference evaluates its order parameters (src/Utilities/
// OrderParameters.cpp) on the host: a "bond" parameter counts its listed
// pairs whose hydrogen-bonding energy is below HB_CUTOFF (-0.1,
// src/Observables/OrderParameterValues.cpp:55-66), a "mindistance"
// parameter takes the smallest base-base (or centre-centre) distance of
// its listed pairs, the plain difference for pairs of one strand and the
// nearest image otherwise (OrderParameters.cpp:73-98).  Its CUDA FFS
// backend precomputes the same per-pair quantities on the GPU
// (hb_op_precalc, near_hb_op_precalc, dist_op_precalc,
// src/CUDA/Interactions/CUDA_DNA.cuh:909-1069), one thread per listed pair;
// so does this kernel, from the batch's FP64 state.  The host folds the
// per-pair values into parameters.
#include "../../include/oxh.h"
#include "oxh_device.h"
#include "oxh_internal.h"
#include "oxh_pair.h"

namespace oxh {

namespace {

// hydrogen-bonding energy of the pair (p, q) (DNAInteraction::
// _hydrogen_bonding, src/Interactions/DNAInteraction.cpp:779-902: zero for
// bonded neighbours), and how many of its seven factors (the Morse well
// below zero, the six angular modulations above zero) are active, the
// count the CUDA FFS backend's "nearly bonded" criterion uses
// (CUDA_DNA.cuh:1019-1030); nfac = -1 when the pair cannot bond at all
// (not complementary, or the base-base distance out of range)
__device__ __forceinline__ double hb_pair(const oxh_sys &S, const dp::Frame &fp, const dp::Frame &fq, const dv3 &rbase, int &nfac) {
	nfac = -1;
	const double rh2 = rbase.x * rbase.x + rbase.y * rbase.y + rbase.z * rbase.z;
	const int pbt = fp.btype, qbt = fq.btype;
	if(!(pbt + qbt == 3 && (double) HYDR_RCLOW * HYDR_RCLOW < rh2 && rh2 < (double) HYDR_RCHIGH * HYDR_RCHIGH)) return 0.0;
	const double hb_multi = (abs(qbt) >= 300 && abs(pbt) >= 300) ? S.hb_multi_d : 1.0;
	const double rmod = sqrt(rh2);
	const dv3 dir = {rbase.x / rmod, rbase.y / rmod, rbase.z / rmod};
	const dv3 &a1 = fp.a1, &a3 = fp.a3, &b1 = fq.a1, &b3 = fq.a3;
	const double cost1 = -dot(a1, b1), cost2 = -dot(b1, dir), cost3 = dot(a1, dir);
	const double cost4 = dot(a3, b3), cost7 = -dot(b3, dir), cost8 = dot(a3, dir);
	const double vf1 = dp::f1(S, rmod, 0, dp::type_of(qbt), dp::type_of(pbt));
	double f4[6], d;
	dp::cf4(cost1, S_HYDR_T1, f4[0], d);
	dp::cf4(cost2, S_HYDR_T2, f4[1], d);
	dp::cf4(cost3, S_HYDR_T2, f4[2], d);
	dp::cf4(cost4, S_HYDR_T4, f4[3], d);
	dp::cf4(cost7, S_HYDR_T7, f4[4], d);
	dp::cf4(cost8, S_HYDR_T7, f4[5], d);
	nfac = vf1 < 0.0 ? 1 : 0;
	for(int k = 0; k < 6; k++) nfac += f4[k] > 0.0 ? 1 : 0;
	return hb_multi * vf1 * f4[0] * f4[1] * f4[2] * f4[3] * f4[4] * f4[5];
}

// one listed pair per thread: (p, q, same strand) in the system's upload
// order, mapped to the batch's slots through slot_of
__global__ void k_pair_quantities(int n, int kind, int s, const int4 *__restrict__ pairs, const double4 *__restrict__ pos,
		const double4 *__restrict__ q64, const int2 *__restrict__ pinfo, const int2 *__restrict__ bonds, const int *__restrict__ slot_of,
		const oxh_sys *__restrict__ systems, double *__restrict__ out) {
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if(k >= n) return;
	const oxh_sys &S = systems[s];
	const int4 pr = pairs[k];
	const int p = slot_of[S.first + pr.x], q = slot_of[S.first + pr.y];
	const double4 P = pos[p], Q = pos[q];
	const bool plain = kind >= OXH_PAIR_BASE_DISTANCE && pr.z != 0;
	const dv3 r = plain ? dv3{Q.x - P.x, Q.y - P.y, Q.z - P.z} : dp::min_image_d(P, Q, S);
	Sites64 sp, sq;
	const dp::Frame fp = dp::make_frame_d(q64[p], pinfo[p].x, sp);
	const dp::Frame fq = dp::make_frame_d(q64[q], pinfo[q].x, sq);
	if(kind == OXH_PAIR_CENTRE_DISTANCE) {
		out[k] = sqrt(r.x * r.x + r.y * r.y + r.z * r.z);
		return;
	}
	const double pb = (double) POS_BASE;
	const dv3 rbase = {(r.x + pb * sq.a1.x) - pb * sp.a1.x, (r.y + pb * sq.a1.y) - pb * sp.a1.y, (r.z + pb * sq.a1.z) - pb * sp.a1.z};
	if(kind == OXH_PAIR_BASE_DISTANCE) {
		out[k] = sqrt(rbase.x * rbase.x + rbase.y * rbase.y + rbase.z * rbase.z);
		return;
	}
	const int2 bd = bonds[p];
	int nfac = -1;
	const double e = (bd.x == q || bd.y == q) ? 0.0 : hb_pair(S, fp, fq, rbase, nfac);
	if(kind == OXH_PAIR_HB_ENERGY) out[k] = e;
	else out[k] = nfac >= 6 ? 1.0 : 0.0;   // OXH_PAIR_NEAR_HB
}

}  // namespace

// ------------------------------------------ what the host reads, per system
// State and forces leave the card as the caller's arrays, upload order and
// axes for quaternions, into page-locked memory (small systems) or a buffer
// that a DMA moves; sums leave as sums.  What bounds these is the bus and the
// wait, so few transfers and no pageable memory: with five copies for a
// state, 14 for the terms and the stress, and the host rearranging or adding,
// 256 states of 48 nt took 20 ms, now 5; energies, terms, stress, bonds and
// forces of a 24,576-nt gas 850 us, now 281; the state of 196,608 nt 8 ms
// less.

namespace {

// out: pos, a1, a3, vel, L of the system's n particles, (n, 3) each
__global__ void __launch_bounds__(256) k_export_state(int n, const double4 *__restrict__ pos, const double4 *__restrict__ q64,
		const double4 *__restrict__ vel, const double4 *__restrict__ Lm, const int *__restrict__ orig, double *__restrict__ out) {
#pragma clang fp contract(off)   // the axes of the host's own conversion
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if(k >= n) return;
	const double4 p = pos[k], q = q64[k], v = vel[k], l = Lm[k];
	const size_t o = 3 * (size_t) orig[k], w = 3 * (size_t) n;
	const double sqx = q.x * q.x, sqy = q.y * q.y, sqz = q.z * q.z, sqw = q.w * q.w;
	const double xy = q.x * q.y, xz = q.x * q.z, xw = q.x * q.w, yz = q.y * q.z, yw = q.y * q.w, zw = q.z * q.w;
	auto put = [&](int row, double x, double y, double z) {
		double *t = out + row * w + o;
		t[0] = x;
		t[1] = y;
		t[2] = z;
	};
	put(0, p.x, p.y, p.z);
	put(1, sqx - sqy - sqz + sqw, 2. * (xy + zw), 2. * (xz - yw));
	put(2, 2. * (xz + yw), 2. * (yz - xw), -sqx - sqy + sqz + sqw);
	put(3, v.x, v.y, v.z);
	put(4, l.x, l.y, l.z);
}

// out: F (n, 3), T (n, 3), E (n)
template<class FT>
__global__ void __launch_bounds__(256) k_export_forces(int n, const FT *__restrict__ F, const FT *__restrict__ T, const int *__restrict__ orig,
		double *__restrict__ out) {
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if(k >= n) return;
	const FT f = F[k], t = T[k];
	const size_t i = orig[k], w = 3 * (size_t) n;
	out[3 * i] = f.x;
	out[3 * i + 1] = f.y;
	out[3 * i + 2] = f.z;
	out[w + 3 * i] = t.x;
	out[w + 3 * i + 1] = t.y;
	out[w + 3 * i + 2] = t.z;
	out[2 * w + i] = f.w;
}

// Sum over a workgroup of 1024 threads, in a fixed order
template<class T>
__device__ __forceinline__ T sum_1024(T v, T *sh) {
	sh[threadIdx.x] = v;
	__syncthreads();
	for(int off = 512; off > 0; off >>= 1) {
		if((int) threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
		__syncthreads();
	}
	return sh[0];
}

// out[c] = FP64 sum of row c (rows of width stride), workgroup c; with vel,
// out[rows + c] = sums of v_a v_b, (a, b) = xx, yy, zz, xy, xz, yz.  Four sums
// a thread: the loads of one workgroup are what bounds it.
__global__ void __launch_bounds__(1024) k_sums(int n, int rows, const double *__restrict__ x, size_t stride, const double4 *__restrict__ vel,
		double *__restrict__ out) {
	__shared__ double sh[1024];
	const int c = blockIdx.x, t = threadIdx.x, m = c - rows;
	double acc[4] = {0., 0., 0., 0.};
	auto term = [&](int i) -> double {
		if(m < 0) return x[c * stride + i];
		const double4 v = vel[i];
		const double a = m == 0 || m == 3 || m == 4 ? v.x : (m == 1 || m == 5 ? v.y : v.z);
		const double b = m == 0 ? v.x : (m == 1 || m == 3 ? v.y : v.z);
		return a * b;
	};
	for(int i = t; i < n; i += 4096)
#pragma unroll
		for(int u = 0; u < 4; u++)
			if(i + 1024 * u < n) acc[u] += term(i + 1024 * u);
	const double sum = sum_1024((acc[0] + acc[1]) + (acc[2] + acc[3]), sh);
	if(t == 0) out[c] = sum;
}

// out[s] = sum of count over system s's particles, workgroup s
__global__ void __launch_bounds__(1024) k_count(const oxh_sys *__restrict__ systems, const int *__restrict__ count, long long *__restrict__ out) {
	__shared__ long long sh[1024];
	const int s = blockIdx.x, first = systems[s].first, n = systems[s].n;
	long long acc = 0;
	for(int i = threadIdx.x; i < n; i += 1024) acc += count[first + i];
	acc = sum_1024(acc, sh);
	if(threadIdx.x == 0) out[s] = acc;
}

}  // namespace

void launch_export_state(const Batch &b, int first, int n, double *out) {
	k_export_state<<<(n + 255) / 256, 256, 0, b.stream>>>(n, b.pos + first, b.q64 + first, b.vel + first, b.Lm + first, b.orig + first, out);
}

void launch_export_forces(const Batch &b, int first, int n, double *out) {
	if(b.fp64) k_export_forces<<<(n + 255) / 256, 256, 0, b.stream>>>(n, b.F64 + first, b.T64 + first, b.orig + first, out);
	else k_export_forces<<<(n + 255) / 256, 256, 0, b.stream>>>(n, b.F + first, b.T + first, b.orig + first, out);
}

void launch_sums(const Batch &b, int n, int rows, const double *x, const double4 *vel, double *out) {
	k_sums<<<rows + (vel ? 6 : 0), 1024, 0, b.stream>>>(n, rows, x, (size_t) b.N, vel, out);
}

void launch_count(const Batch &b, long long *out) { k_count<<<b.nsys, 1024, 0, b.stream>>>(b.d_sys, b.hbcount, out); }

void launch_pair_quantities(hipStream_t st, const Batch &b, int sys, int kind, int n, const int4 *d_pairs, double *d_out) {
	if(n <= 0) return;
	if(b.model) {
		launch_rna_pair_quantities(st, b, sys, kind, n, d_pairs, d_out);
		return;
	}
	k_pair_quantities<<<(n + 255) / 256, 256, 0, st>>>(n, kind, sys, d_pairs, b.pos, b.q64, b.pinfo, b.bonds, b.slot_of, b.d_sys, d_out);
}

}  // namespace oxh
