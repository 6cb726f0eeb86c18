// One MD step per launch on gfx950, for batches whose steps are short.
//
// A step of the one-kernel-per-phase path is up to five launches (binning,
// ranks, lists, forces, integration), and a launch costs 4 to 5 us inside a
// graph even when it finds nothing to do, which is half of a step of a
// system of a few thousand nucleotides.  Nothing in a step needs the whole
// grid between forces and integration, or between lists and forces: a
// nucleotide's row, forces and integration are its own workgroup's work, and
// only read what the previous launch left.  So k_step does, for the
// nucleotides of its workgroup,
//   1. the list rows, when the system's skin check asked for them,
//   2. the forces (far pairs inline),
//   3. the second half of step k and the first half of step k + 1, into the
//      other set of state buffers (the neighbours still read this one),
//   4. the skin check and the binning for step k + 1.
// Flags and cell counters go round in three sets (read at k, written for
// k + 1, cleared for k + 2), cell slots and wrapped centres in two.
// Binning takes every step where the old path binned only before a rebuild:
// an atomic per nucleotide next to ~20 us of forces.  Cells hold their
// particles in arrival order; a row is put in the lists' order (cell, then
// index) by ranking its entries, so rows and forces are those of the other
// path.  Rows above STEP_ROW entries have a launch of their own before the
// step's, for the systems that have met one.
// Measured, per MD step, one kernel per phase -> this: 24,576-nt gas with
// Bussi 36.5 -> 33.2 us, 777 nt without cells 16.5 -> 13.0 us, a pool of eight
// jobs of 259 to 1,332 nt 43.6 -> 37.9 us.
// Not for dense batches (their lists are built cell by cell), far pairs in a
// kernel of their own, the half-list form, all-FP64, oxRNA or external
// forces, which keep the one-kernel-per-phase path.
#include <algorithm>
#include <type_traits>

#include "oxh_device.h"
#include "oxh_internal.h"
#include "oxh_list.h"
#include "oxh_pair.h"
#include "oxh_step.h"

namespace oxh {

namespace {

// keys of one row while it is built: (stencil cell << 24) | particle, close
// pairs from the front, far pairs from the back
constexpr int GROUP = BUILD_LANES;

// what decides whether j enters the row of particle i of a system with
// cells, as in build_row; the backbone sites are those of this state, which
// the row records (blist)
struct Candidates {
	const oxh_sys &S;
	const StepArgs &a;
	int i;
	double4 p;
	int2 bd;
	bool back;
	float4 p32, bi;
	__device__ __forceinline__ Candidates(int i_, const oxh_sys &S_, const StepArgs &a_) : S(S_), a(a_), i(i_) {
		p = a.pos[i];
		bd = a.bonds[i];
		back = S.far_back != 0;
		p32 = a.pos32[i];
		bi = back ? a.bpos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
	}
	__device__ __forceinline__ void test(int j, bool &close, bool &far) const {
		close = far = false;
		if(j < 0 || j == i || j == bd.x || j == bd.y) return;
		const float db2 = back ? back_dist2(bi, a.bpos[j], S) : 0.f;
		if(back && !(db2 < S.rgate2f)) return;
		classify_pair(S, p, p32, a.pos32[j], a.pos, j, true, close, far);
		if(far && back && !(db2 < S.rbf2)) far = false;
	}
};

// Row of particle i of a system with cells whose particles lie in the cells'
// arrival order (the 32 lanes of a group call it): the candidates, tests and
// row order of build_row.
__device__ __forceinline__ void build_row_binned(int i, int l, int s, const StepArgs &a, unsigned int *keys) {
	constexpr int K = GROUP;
	const oxh_sys &S = a.systems[s];
	const Candidates cand(i, S, a);
	const int g0 = (threadIdx.x & 63) & ~(K - 1);
	const uint64_t gmask = ((1ull << K) - 1ull) << g0;
	const uint64_t below = ((1ull << (threadIdx.x & 63)) - 1ull) & gmask;
	int *row = a.nbr + (size_t) i * a.max_neigh;
	const Stencil n = stencil_of(cand.p, cand.p32, S);
	int nc = 0, nf = 0;
	bool full = false;
	walk_stencil(
			n, l, S,
			[&](int c) {
				const int held = a.count[c];
				full |= held > a.cell_cap;
				return min(held, a.cell_cap);
			},
			[&](bool have, int c, int slot, int kc) {
				const int j = have ? a.raw[(size_t) c * a.cell_cap + slot] : -1;
				bool close, far;
				cand.test(j, close, far);
				const uint64_t bc = __ballot(close) & gmask, bf = __ballot(far) & gmask;
				const unsigned int key = ((unsigned int) kc << 24) | (unsigned int) j;
				if(close) {
					const int q = nc + __popcll(bc & below);
					if(q + nf < STEP_ROW) keys[q] = key;
				}
				if(far) {
					const int q = nf + __popcll(bf & below);
					if(nc + q < STEP_ROW) keys[STEP_ROW - 1 - q] = key;
				}
				nc += __popcll(bc);
				nf += __popcll(bf);
			});
	full = (__ballot(full) & gmask) != 0;
	if(nc + nf > min(a.max_neigh, STEP_ROW) || full) {
		if(l == 0) {
			atomicOr(&a.state[s].error,
					(full ? ERR_CELLS : 0) | (nc + nf > a.max_neigh ? ERR_LIST : 0) | (nc + nf > STEP_ROW ? ERR_ROW : 0));
			a.nnbr[i] = make_int2(0, 0);
			a.rlist[i] = cand.p;
			if(cand.back) a.blist[i] = cand.bi;
		}
		return;
	}
	// the keys' ranks are the entries' places
	__threadfence_block();
	for(int e = l; e < nc; e += K) {
		const unsigned int key = keys[e];
		int rank = 0;
		for(int m = 0; m < nc; m++) rank += keys[m] < key;
		row[rank] = (int) (key & 0xFFFFFFu);
	}
	const unsigned int *fk = keys + STEP_ROW - nf;
	for(int e = l; e < nf; e += K) {
		const unsigned int key = fk[e];
		int rank = 0;
		for(int m = 0; m < nf; m++) rank += fk[m] < key;
		row[a.max_neigh - 1 - rank] = (int) (key & 0xFFFFFFu);
	}
	if(l != 0) return;
	a.nnbr[i] = make_int2(nc, nf);
	a.rlist[i] = cand.p;
	if(cand.back) a.blist[i] = cand.bi;
}

// Rows of RB particles of a system without cells (row[r] < 0: none), the
// candidates, tests and row order of build_row.  A row by itself is a chain
// of a load, an FP64 distance and two ballots for every 32 candidates; RB
// rows over one set of loads, the next one under way, share its latency:
// a pool of eight jobs of 259 to 1,332 nt, 320 steps, 12.7 -> 12.0 ms.
template<int RB>
__device__ __forceinline__ void build_rows_all(const int (&row)[RB], int l, int s, const StepArgs &a) {
	constexpr int K = GROUP;
	const oxh_sys &S = a.systems[s];
	const int g0 = (threadIdx.x & 63) & ~(K - 1);
	const uint64_t gmask = ((1ull << K) - 1ull) << g0;
	const uint64_t below = ((1ull << (threadIdx.x & 63)) - 1ull) & gmask;
	double4 p[RB];
	int2 bd[RB];
	int nc[RB], nf[RB];
#pragma unroll
	for(int r = 0; r < RB; r++) {
		p[r] = a.pos[row[r] >= 0 ? row[r] : S.first];
		bd[r] = a.bonds[row[r] >= 0 ? row[r] : S.first];
		nc[r] = nf[r] = 0;
	}
	const int end = S.first + S.n;
	double4 next = a.pos[min(S.first + l, end - 1)];
	for(int j0 = S.first; j0 < end; j0 += K) {
		const int j = j0 + l;
		const double4 q = next;
		next = a.pos[min(j + K, end - 1)];
#pragma unroll
		for(int r = 0; r < RB; r++) {
			const bool test = row[r] >= 0 && j < end && j != row[r] && j != bd[r].x && j != bd[r].y;
			const double r2 = sqr_dist(p[r], q, S);
			const bool in = test && r2 < S.rv2, close = in && r2 < S.rclose2, far = in && !close;
			const uint64_t bc = __ballot(close) & gmask, bf = __ballot(far) & gmask;
			int *out = a.nbr + (size_t) row[r] * a.max_neigh;
			if(close) {
				const int k = nc[r] + __popcll(bc & below);
				if(k + nf[r] < a.max_neigh) out[k] = j;
			}
			if(far) {
				const int k = nf[r] + __popcll(bf & below);
				if(nc[r] + k < a.max_neigh) out[a.max_neigh - 1 - k] = j;
			}
			nc[r] += __popcll(bc);
			nf[r] += __popcll(bf);
		}
	}
	if(l != 0) return;
#pragma unroll
	for(int r = 0; r < RB; r++) {
		if(row[r] < 0) continue;
		const bool over = nc[r] + nf[r] > a.max_neigh;
		if(over) atomicOr(&a.state[s].error, ERR_LIST);
		a.nnbr[row[r]] = over ? make_int2(0, 0) : make_int2(nc[r], nf[r]);
		a.rlist[row[r]] = p[r];
	}
}

// Rows of a system that has rows longer than the keys held, before the step's
// own launch: cell after cell, an entry's place is the number of its cell's
// entries before it, so a row of any length comes out in the same order.  In
// k_step itself this code cost every other batch 0.9 % (24,576-nt gas), on
// scalar registers; so the step's kernel is the same for all systems of a
// pool, whatever their rows, and only this launch comes on top.
__global__ void __launch_bounds__(256) k_step_long_rows(StepArgs a) {
	constexpr int K = GROUP;
	if(!a.need[a.nsys]) return;
	const int t = blockIdx.x * blockDim.x + threadIdx.x, i = t / K, l = t % K;
	if(i >= a.N) return;
	const int s = a.pinfo[i].y;
	const oxh_sys &S = a.systems[s];
	if(!S.long_rows || !a.need[s] || padding(i, S)) return;
	const Candidates cand(i, S, a);
	const int g0 = (threadIdx.x & 63) & ~(K - 1);
	const uint64_t gmask = ((1ull << K) - 1ull) << g0;
	int *row = a.nbr + (size_t) i * a.max_neigh;
	const Stencil n = stencil_of(cand.p, cand.p32, S);
	int nc = 0, nf = 0;
	bool full = false;
	for(int oz = -n.R; oz <= n.R; oz++)
		for(int oy = -n.R; oy <= n.R; oy++)
			for(int ox = -n.R; ox <= n.R; ox++) {
				bool in_range;
				const int c = stencil_cell(n, oz, oy, ox, S, in_range);
				const int all = in_range ? a.count[c] : 0, held = min(all, a.cell_cap);
				full |= all > a.cell_cap;
				const int *in = a.raw + (size_t) c * a.cell_cap;
				int cc = 0, cf = 0;
				for(int m0 = 0; m0 < held; m0 += K) {
					const int j = m0 + l < held ? in[m0 + l] : -1;
					bool close = false, far = false;
					int rc = 0, rf = 0;
					for(int o0 = 0; o0 < held; o0 += K) {
						const int jo = o0 + l < held ? in[o0 + l] : -1;
						bool oc, of;
						cand.test(jo, oc, of);
						if(o0 == m0) {
							close = oc;
							far = of;
						}
						uint64_t bc = __ballot(oc) >> g0, bf = __ballot(of) >> g0;
#pragma unroll 1
						for(int t = 0; t < K; t++, bc >>= 1, bf >>= 1) {
							const bool before = __shfl(jo, t, K) < j;
							rc += before && (bc & 1);
							rf += before && (bf & 1);
						}
					}
					if(close && nc + rc < a.max_neigh) row[nc + rc] = j;
					if(far && nf + rf < a.max_neigh) row[a.max_neigh - 1 - nf - rf] = j;
					cc += __popcll(__ballot(close) & gmask);
					cf += __popcll(__ballot(far) & gmask);
				}
				nc += cc;
				nf += cf;
			}
	if(l != 0) return;
	const bool over = nc + nf > a.max_neigh || full;
	if(over) atomicOr(&a.state[s].error, (full ? ERR_CELLS : 0) | (nc + nf > a.max_neigh ? ERR_LIST : 0));
	a.nnbr[i] = over ? make_int2(0, 0) : make_int2(nc, nf);
	a.rlist[i] = cand.p;
	if(cand.back) a.blist[i] = cand.bi;
}

// particle i of step k: into its cell (slot in arrival order) and its
// wrapped FP32 centre, for a list build in this step
__device__ __forceinline__ void bin_particle(int i, const oxh_sys &S, const double4 &p, int *__restrict__ count, int *__restrict__ raw, int cap,
		float4 *__restrict__ pos32) {
	if(!S.use_cells) return;
	const int cx = cell_coord(p.x, S.inv_box[0], S.nc[0]);
	const int cy = cell_coord(p.y, S.inv_box[1], S.nc[1]);
	const int cz = cell_coord(p.z, S.inv_box[2], S.nc[2]);
	const int c = S.cell_first + (cz * S.nc[1] + cy) * S.nc[0] + cx;
	pos32[i] = make_float4((float) (p.x - S.box[0] * floor(p.x * S.inv_box[0])), (float) (p.y - S.box[1] * floor(p.y * S.inv_box[1])),
			(float) (p.z - S.box[2] * floor(p.z * S.inv_box[2])), 0.f);
	const int slot = atomicAdd(&count[c], 1);
	if(slot < cap) raw[(size_t) c * cap + slot] = i;
}

// first half of step k of particle i from the in buffers into the out ones,
// its skin check and binning; a particle whose system takes no part in step
// k is carried over
__device__ __forceinline__ void step_first(int i, int s, const oxh_sys &S, const StepArgs &a, int k, int *need, int *count, int *raw, float4 *pos32) {
	if(a.limit && k >= a.limit[s]) {
		if(a.pos_o != a.pos) {
			a.pos_o[i] = a.pos[i];
			a.q64_o[i] = a.q64[i];
			a.q32_o[i] = a.q32[i];
			a.bpos_o[i] = a.bpos[i];
		}
		return;
	}
	double4 r;
	if(first_step_particle(i, S, a.pos, a.vel, a.Lm, a.q64, a.q32_o, a.bpos_o, nullptr, a.F, a.T, a.rlist, a.bonds, a.pstep, a.blist, a.pos_o,
			a.q64_o, r)) {
		need[s] = 1;
		need[a.nsys] = 1;
	}
	bin_particle(i, S, r, count, raw, a.cell_cap, pos32);
}

// chunk start: every flag and counter set to zero
__global__ void k_step_begin(int nneed, int *__restrict__ need, int ncount, int *__restrict__ count) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i < nneed) need[i] = 0;
	if(i < ncount) count[i] = 0;
}

__global__ void __launch_bounds__(256) k_step_first(StepArgs a, int k) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= a.N) return;
	const int s = a.pinfo[i].y;
	const oxh_sys &S = a.systems[s];
	if(padding(i, S)) return;
	step_first(i, s, S, a, k, a.need, a.count, a.raw, a.pos32);
}

// LDS of a workgroup: the rows' keys (16 KB), then the packed form's list
template<bool PACK>
union StepShared {
	unsigned int keys[PACK_BS / GROUP][STEP_ROW];
	PackShared pack;
};
template<>
union StepShared<false> {
	unsigned int keys[PACK_BS / GROUP][STEP_ROW];
};

template<int K, bool PACK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_step(StepArgs a, int k, int go_on) {
	__shared__ StepShared<PACK> sh;
	const unsigned nblk = ((unsigned) a.N * K + blockDim.x - 1) / blockDim.x;
	const int blk = a.xcd ? xcd_block(nblk) : (int) blockIdx.x;
	if(blk < 0) return;   // whole padding workgroup
	const int tid = threadIdx.x, nper = blockDim.x / K, i0 = blk * nper;
	for(int c = blk * blockDim.x + tid; c < max(a.ncell, a.nsys + 1); c += nblk * blockDim.x) {
		if(c < a.ncell) a.count_clear[c] = 0;
		if(c <= a.nsys) a.need_clear[c] = 0;
	}
	// 1. list rows of this workgroup's particles
	if(a.need[a.nsys]) {
		// a group's rows are neighbours in the list's order, RB at a time
		constexpr int RB = K >= 32 ? 1 : (K == 16 ? 2 : 4);
		const int grp = tid / GROUP, l = tid % GROUP, ngrp = blockDim.x / GROUP, per = nper / ngrp;
		for(int r0 = grp * per; r0 < (grp + 1) * per; r0 += RB) {
			int row[RB], sr[RB];
			bool one = true;   // system without cells, the same for all
#pragma unroll
			for(int r = 0; r < RB; r++) {
				const int i = i0 + r0 + r;
				row[r] = i < a.N && a.need[a.pinfo[i].y] && !padding(i, a.systems[a.pinfo[i].y]) ? i : -1;
				sr[r] = row[r] >= 0 ? a.pinfo[i].y : -1;
				if(row[r] < 0) continue;
				if(l == 0 && i == a.systems[sr[r]].first) a.state[sr[r]].n_rebuilds += 1;
				if(a.systems[sr[r]].use_cells) one = false;
			}
			int s = -1;
#pragma unroll
			for(int r = 0; r < RB; r++) {
				if(sr[r] < 0) continue;
				if(s >= 0 && sr[r] != s) one = false;
				s = sr[r];
			}
			if(s < 0) continue;
			if(one) {
				build_rows_all<RB>(row, l, s, a);
				continue;
			}
#pragma unroll 1
			for(int r = 0; r < RB; r++) {
				const int i = i0 + r0 + r;
				if(i >= a.N) continue;
				const int si = a.pinfo[i].y;
				const oxh_sys &S = a.systems[si];
				if(!a.need[si] || padding(i, S)) continue;
				if(S.use_cells) {
					if(!S.long_rows) build_row_binned(i, l, si, a, sh.keys[grp]);
				}
				else {
					const int alone[1] = {i};
					build_rows_all<1>(alone, l, si, a);
				}
			}
		}
		__syncthreads();
	}
	// 2. forces
	const int i = i0 + tid / K, l = tid % K;
	const int ic = i < a.N ? i : a.N - 1;
	const int s = a.pinfo[ic].y;
	const bool act = i < a.N && !idle(i, a.systems[s], s, k, a.limit);
	if constexpr(PACK)
		particle_forces<false, true, true>(K, ic, l, a.N, a.pos, a.q64, a.q32, a.bpos, a.bonds, a.pinfo, a.nbr, a.nnbr, a.max_neigh, a.systems,
				a.state, a.F, a.T, nullptr, nullptr, nullptr, act, &sh.pack, i0, k, a.limit);
	else if(act)
		particle_forces<false, true>(K, i, l, a.N, a.pos, a.q64, a.q32, a.bpos, a.bonds, a.pinfo, a.nbr, a.nnbr, a.max_neigh, a.systems, a.state,
				a.F, a.T, nullptr, nullptr, nullptr);
	if(!go_on) return;
	// 3. and 4. integration over the step's boundary, one particle per thread
	__syncthreads();
	const int ip = i0 + tid;
	if(tid >= nper || ip >= a.N) return;
	const int sp = a.pinfo[ip].y;
	const oxh_sys &Sp = a.systems[sp];
	if(padding(ip, Sp)) return;
	if(!(a.limit && k >= a.limit[sp])) second_step_particle(ip, Sp, a.vel, a.Lm, a.F, a.T, a.orig, a.pstep);
	step_first(ip, sp, Sp, a, k + 1, a.need_next, a.count_next, a.raw_next, a.pos32_next);
}

template<int K>
void launch_k(hipStream_t st, const StepArgs &a, bool pack, int block, int k, int go_on) {
	if(pack) block = PACK_BS;
	const unsigned nblk = (unsigned) (((size_t) a.N * K + block - 1) / block);
	const dim3 grid(a.xcd ? xcd_grid(nblk) : nblk);
	if(pack) k_step<K, true><<<grid, block, 0, st>>>(a, k, go_on);
	else k_step<K, false><<<grid, block, 0, st>>>(a, k, go_on);
}

}  // namespace

bool fused_lanes(int lanes) { return lanes == 2 || lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32; }

void launch_step_begin(hipStream_t st, int nneed, int *need, int ncount, int *count) {
	const int n = std::max(nneed, ncount);
	k_step_begin<<<(n + 255) / 256, 256, 0, st>>>(nneed, need, ncount, count);
}

void launch_step_first(hipStream_t st, const StepArgs &a, int k) { k_step_first<<<(a.N + 255) / 256, 256, 0, st>>>(a, k); }

void launch_step_long_rows(hipStream_t st, const StepArgs &a) {
	const size_t threads = (size_t) a.N * GROUP;
	k_step_long_rows<<<(unsigned) ((threads + 255) / 256), 256, 0, st>>>(a);
}

void launch_step(hipStream_t st, const StepArgs &a, int lanes, bool pack, int block, int k, bool go_on) {
	switch(lanes) {
	case 2: launch_k<2>(st, a, pack, block, k, go_on); break;
	case 4: launch_k<4>(st, a, pack, block, k, go_on); break;
	case 16: launch_k<16>(st, a, pack, block, k, go_on); break;
	case 32: launch_k<32>(st, a, pack, block, k, go_on); break;
	default: launch_k<8>(st, a, pack, block, k, go_on); break;
	}
}

}  // namespace oxh
