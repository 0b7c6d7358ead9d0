// pp_device.hpp -- device helpers shared by the gfx950 kernels of
// libpp_hip.so (pp_kernels.hip: rebuild, colour passes, energy; pp_learn.hip:
// the learned proposal): team operations, counters, trial draws and the
// reference-order pair tests on a trial.
#pragma once
#pragma clang fp contract(off)

#include "pp_internal.h"

namespace ppd {

// ------------------------------------------------------------------------
// helpers

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous run of logical blocks so that neighbouring cells share an L2.
// nb must be a multiple of 8.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
	int per = nb >> 3;
	return (b & 7) * per + (b >> 3);
}

// Buffer b (0 or 1) of the double-buffered slot arrays.  A team-uniform b
// that is not wavefront-uniform (a selector read from a cell record) would
// index the kernel argument with a vector load; later loads through the
// pointer then wait on every load issued before them.  Selecting between the
// two scalar base pointers keeps them in registers.
template <class P>
__device__ __forceinline__ P *pick_buf(P *const (&buf)[2], int b) {
	const unsigned long long p0 = (unsigned long long) buf[0], p1 = (unsigned long long) buf[1];
	const unsigned lo = b ? (unsigned) p1 : (unsigned) p0, hi = b ? (unsigned) (p1 >> 32) : (unsigned) (p0 >> 32);
	return (P *) (((unsigned long long) hi << 32) | lo);
}

// The 12 components of slot j.  They lie together because the passes gather
// whole particles from a few cells' slot ranges: six 16-byte loads from one
// or two cache lines per particle, where an array per component took twelve
// loads from a dozen lines per run of slots.  Measured against that layout:
// 256 uneven replicas 4.51 -> 4.15 ms per step, the N=65536 learned sweep 514
// -> 496 us, N=32768 with one trial per member 2.6 % faster.
template <class D>
__device__ __forceinline__ D *part(D *f, int j) { return f + (size_t) NCOMP * j; }

// DPP controls (gfx9 encoding)
constexpr int DPP_QUAD_1032 = 0xB1;      // quad_perm [1,0,3,2]
constexpr int DPP_QUAD_2301 = 0x4E;      // quad_perm [2,3,0,1]
constexpr int DPP_ROW_MIRROR = 0x140;    // lane i <- 15 - i within a 16-lane row
constexpr int DPP_HALF_MIRROR = 0x141;   // lane i <- 7 - i within 8 lanes

// Sum over a team of T = 8, 16, 32 or 64 lanes, in every lane of the team,
// with VALU cross-lane moves only (a __shfl_xor is a ds_bpermute, an LDS
// round trip per step): DPP butterflies within a 16-lane row, then gfx950's
// row-pair and half-wave swaps.  Each step stays inside the team, so lanes of
// the other teams of the wavefront may be inactive.
template <int T>
__device__ __forceinline__ int team_sum(int v) {
	static_assert(T == 8 || T == 16 || T == 32 || T == 64, "team of 8 to 64 lanes");
	v += __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_1032, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_2301, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_HALF_MIRROR, 0xf, 0xf, false);
	if constexpr(T >= 16) v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_MIRROR, 0xf, 0xf, false);
	if constexpr(T >= 32) {
		// rows 2j and 2j+1 trade places between two copies: copy sum = row-pair sum
		const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
		v = (int) (p[0] + p[1]);
	}
	if constexpr(T >= 64) {
		const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
		v = (int) (p[0] + p[1]);
	}
	return v;
}

// Inclusive prefix sum over a whole wavefront (every lane active):
// Hillis-Steele steps within each 16-lane row (row_shr 1, 2, 4, 8, the
// lanes shifted in from outside the row reading 0), then row 0's total into
// row 1 and row 2's into row 3 (row_bcast:15), then the first half's total
// into rows 2 and 3 (row_bcast:31).
constexpr int DPP_ROW_SHR = 0x110;     // + k: lane i <- i - k within a row
constexpr int DPP_ROW_BCAST15 = 0x142;
constexpr int DPP_ROW_BCAST31 = 0x143;

__device__ __forceinline__ int wave_incl_scan(int v) {
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR + 1, 0xf, 0xf, true);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR + 2, 0xf, 0xf, true);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR + 4, 0xf, 0xf, true);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR + 8, 0xf, 0xf, true);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST15, 0xa, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST31, 0xc, 0xf, false);
	return v;
}

__device__ __forceinline__ int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// The slots of the 26 cells around cell (ix, iy, iz) of an n0 x n1 x n2 grid
// (st: the replica's cell starts), in the order of the directions m = 9 (dx +
// 1) + 3 (dy + 1) + dz + 1: row j < 9 holds the cells of directions 3j, 3j + 1
// and 3j + 2, whose slots are one range, or two where the row wraps around the
// box or (j = 4) leaves out the cell itself.  The row's candidates are
// [a1, b1), then [a2, b2).
__device__ __forceinline__ void row_ranges(const int *st, int ix, int iy, int iz, int n0, int n1, int n2, int j, int &a1,
                                           int &b1, int &a2, int &b2) {
	const int cx = wrapi(ix + j / 3 - 1, n0), cy = wrapi(iy + j % 3 - 1, n1);
	const int *row = st + (size_t) (cx * n1 + cy) * n2;
	const int zl = wrapi(iz - 1, n2), zh = wrapi(iz + 1, n2);
	// ends of the first range and starts of the second, as cells of the row
	int e1 = iz + 2, s2 = zh, e2 = zh;
	if(j == 4) e1 = zl + 1, e2 = zh + 1;
	else if(iz == 0) e1 = zl + 1, s2 = 0, e2 = 2;
	else if(iz == n2 - 1) e1 = n2, e2 = zh + 1;
	a1 = row[zl];
	b1 = row[e1];
	a2 = row[s2];
	b2 = row[e2];
}

// Slot of candidate i of those rows, counted through (a record holds the
// first REC_SLOTS; few cells have more).
__device__ inline int walk_slot(const int *st, int ix, int iy, int iz, int n0, int n1, int n2, int i) {
#pragma unroll 1  // (rare: nine copies at every use only displace the code that runs)
	for(int j = 0; j < 9; j++) {
		int a1, b1, a2, b2;
		row_ranges(st, ix, iy, iz, n0, n1, n2, j, a1, b1, a2, b2);
		if(i < b1 - a1) return a1 + i;
		i -= b1 - a1;
		if(i < b2 - a2) return a2 + i;
		i -= b2 - a2;
	}
	return 0;
}

// Slot of static neighbour i of a record (rec: the record or a copy).
__device__ __forceinline__ int rec_slot(const DevState &d, const int *rec, int i) {
	if(i < REC_SLOTS) return rec[REC_HEAD + i];
	const Rep &rp = d.reps[rec[REC_REP]];
	return walk_slot(d.start + rp.cell_off, rec[REC_IX], rec[REC_IY], rec[REC_IZ], rp.lg.n[0], rp.lg.n[1], rp.lg.n[2], i);
}

// The record of cell cloc = (ix, iy, iz) of a grid of n0 x n1 x n2 cells (st:
// its cells' first slots), by 16 lanes of a DPP row: lane j < 9 takes row j of
// the neighbourhood (row_ranges), a prefix sum over the lanes places its
// slots, lane 9 writes the header.  A pass finds all its data from this one
// record: its slot list needs no search, and lanes of one team write to one or
// two cache lines (a thread per record wrote 256 bytes at a time, from 52
// loads of its own).
__device__ __forceinline__ void write_record(int *rec, int tag, const int *st, int cloc, int ix, int iy, int iz, int n0,
                                             int n1, int n2, int r, int sel, int lane) {
	int a1 = 0, b1 = 0, a2 = 0, b2 = 0;
	if(lane < 9) row_ranges(st, ix, iy, iz, n0, n1, n2, lane, a1, b1, a2, b2);
	else if(lane == 9) {
		a1 = st[cloc];
		b1 = st[cloc + 1];
	}
	const int l1 = b1 - a1, len = lane < 9 ? l1 + b2 - a2 : 0;
	int inc = len;
	inc += __builtin_amdgcn_update_dpp(0, inc, DPP_ROW_SHR + 1, 0xf, 0xf, true);
	inc += __builtin_amdgcn_update_dpp(0, inc, DPP_ROW_SHR + 2, 0xf, 0xf, true);
	inc += __builtin_amdgcn_update_dpp(0, inc, DPP_ROW_SHR + 4, 0xf, 0xf, true);
	inc += __builtin_amdgcn_update_dpp(0, inc, DPP_ROW_SHR + 8, 0xf, 0xf, true);
	// candidates before the cell itself, for the header's lane
	const int m0 = __shfl(inc - len + l1, (int) (threadIdx.x & 63 & ~15) + 4);
	for(int e = 0, at = REC_HEAD + inc - len; e < len && at < REC_W; e++, at++) rec[at] = e < l1 ? a1 + e : a2 + e - l1;
	if(lane == 9) {
		rec[REC_TAG] = tag;
		rec[REC_M] = inc;
		rec[REC_S0] = a1;
		rec[REC_CNT] = l1;
		rec[REC_CELL] = cloc;
		rec[REC_REP] = r;
		rec[REC_SEL] = sel;
		rec[REC_M0] = m0;
		rec[REC_IX] = ix;
		rec[REC_IY] = iy;
		rec[REC_IZ] = iz;
	}
}

// A value the compiler knows nothing about: what is computed from it stays
// where it is written, not in registers across a loop that rarely needs it.
__device__ __forceinline__ int opaque(int v) {
	asm volatile("" : "+v"(v)::"memory");
	return v;
}

__device__ __forceinline__ int opaque_uniform(int v) {
	asm volatile("" : "+s"(v)::"memory");
	return v;
}

// The lanes of the wavefront where p holds (__ballot takes an int, which
// costs a select and a compare when p is a combined condition).
__device__ __forceinline__ unsigned long long ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// Whether p holds in some lane of the team.
template <int T>
__device__ __forceinline__ bool team_any(bool p) {
	const unsigned long long m = ballot(p);
	const int off = (threadIdx.x & 63) & ~(T - 1);
	if constexpr(T == 64) return m != 0ull;
	else if constexpr(T == 32) return (off ? (unsigned) (m >> 32) : (unsigned) m) != 0u;
	else return ((unsigned) (m >> off) & ((1u << T) - 1u)) != 0u;
}

// When a team is a whole wavefront (T = 64) every team-uniform value is
// wave-uniform: readfirstlane moves it to scalar registers.
template <int T>
__device__ __forceinline__ int uni(int v) {
	if constexpr(T == 64) return __builtin_amdgcn_readfirstlane(v);
	else return v;
}

// Lanes of one team live in one wavefront: order their LDS traffic.
__device__ __forceinline__ void team_sync() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ unsigned long long *ctr_at(unsigned long long *ctr, int r, int row, int slot) {
	return ctr + ((long long) (r * NCTR + row) * NSLOT + slot);
}

// Uniform axis on the unit sphere by Marsaglia's rejection method (the
// method of random_vector_on_sphere, utils.c:115-131), fed by Philox blocks
// (two candidate pairs per block) until a pair falls inside the unit disc.
// Each pair is accepted with probability pi/4; after AXIS_BLOCKS blocks
// (chance 0.215^128) the axis is +z or -z by a random bit, which keeps the
// axis law symmetric under a -> -a and so the proposal symmetric.
constexpr uint32_t AXIS_BLOCKS = 64;

__device__ __forceinline__ u32x4 axis_block(uint64_t seed, int r, uint64_t sweep, uint32_t cell, uint32_t col, uint32_t t,
                                            uint32_t blk) {
	return rng(seed, r, sweep, cell | (blk << 24), TAG_AXIS, col, t);
}

// v: block 0 of the draw (callers form it among their other draws, so that
// the Philox rounds of all of them overlap); have_next: block 1 is `next`.
__device__ __forceinline__ void sphere_axis_from(u32x4 v, bool have_next, u32x4 next, uint64_t seed, int r, uint64_t sweep,
                                                 uint32_t cell, uint32_t col, uint32_t t, double a[3]) {
	for(uint32_t blk = 0;;) {
		// the block's first accepted pair
		const double p1 = 1. - 2. * u01(v.x), p2 = 1. - 2. * u01(v.y), s1 = 1. - 2. * u01(v.z), s2 = 1. - 2. * u01(v.w);
		const double p = p1 * p1 + p2 * p2, s = s1 * s1 + s2 * s2;
		const bool one = p < 1.;
		const double q = one ? p : s, u1 = one ? p1 : s1, u2 = one ? p2 : s2;
		if(q < 1.) {
			const double f = 2. * __builtin_sqrt(1. - q);
			a[0] = u1 * f;
			a[1] = u2 * f;
			a[2] = 1. - 2. * q;
			return;
		}
		if(++blk == AXIS_BLOCKS) break;
		if(have_next && blk == 1) v = next;
		else v = axis_block(seed, r, sweep, cell, col, t, blk);
	}
	v = rng(seed, r, sweep, cell, TAG_AXIS_FALLBACK, col, t);
	a[0] = 0.;
	a[1] = 0.;
	a[2] = (v.x & 1u) ? 1. : -1.;
}

__device__ __forceinline__ void sphere_axis(uint64_t seed, int r, uint64_t sweep, uint32_t cell, uint32_t col,
                                            uint32_t t, double a[3]) {
	sphere_axis_from(axis_block(seed, r, sweep, cell, col, t, 0), false, u32x4{}, seed, r, sweep, cell, col, t, a);
}

template <int c>
__device__ __forceinline__ uint32_t quad_word(uint32_t v) {
	return (uint32_t) __builtin_amdgcn_update_dpp(0, (int) v, c * 0x55, 0xf, 0xf, true);
}
template <int c>
__device__ __forceinline__ u32x4 quad_block(u32x4 v) {
	return u32x4{quad_word<c>(v.x), quad_word<c>(v.y), quad_word<c>(v.z), quad_word<c>(v.w)};
}

// Trial t of cell cloc (colour col) in sweep `sweep`: member rank among
// cnt, displacement uniform in +-disp_max/2 per axis (MC.c:317-319), rotation
// by an angle uniform in [0, theta_max) about an axis uniform on the sphere
// (MC.c:321-325, utils.c:186-202).  Returns the 32 bits of the acceptance
// draw u = w 2^-32 (MC.c:332).
// by_quads (uniform): the four lanes of a quad make the same trial together,
// each drawing one of its blocks (the axis' second among them).  A lane alone
// draws three, one after the other where few wavefronts share the SIMD.
__device__ __forceinline__ uint32_t make_trial(const DevState &d, const Rep &rp, int r, uint64_t sweep, int cloc, int col,
                                               int t, int cnt, bool by_quads, double out[TRIAL_W]) {
	u32x4 ra, rb, rc, rd{};
	if(by_quads) {
		const uint32_t q = threadIdx.x & 3u;
		const u32x4 v = rng(d.seed, r, sweep, (uint32_t) cloc | (q == 3u ? 1u << 24 : 0u),
		                    q == 0u ? (uint32_t) TAG_TRIAL_A : (q == 1u ? (uint32_t) TAG_TRIAL_B : (uint32_t) TAG_AXIS),
		                    (uint32_t) col, (uint32_t) t);
		ra = quad_block<0>(v);
		rb = quad_block<1>(v);
		rc = quad_block<2>(v);
		rd = quad_block<3>(v);
	}
	else {
		ra = rng(d.seed, r, sweep, (uint32_t) cloc, TAG_TRIAL_A, (uint32_t) col, (uint32_t) t);
		rb = rng(d.seed, r, sweep, (uint32_t) cloc, TAG_TRIAL_B, (uint32_t) col, (uint32_t) t);
		rc = axis_block(d.seed, r, sweep, (uint32_t) cloc, (uint32_t) col, (uint32_t) t, 0);
	}
	double axis[3], st, ct, R[9];
	sincos(u01(rb.x) * rp.theta_max, &st, &ct);
	sphere_axis_from(rc, by_quads, rd, d.seed, r, sweep, (uint32_t) cloc, (uint32_t) col, (uint32_t) t, axis);
	out[0] = (double) __umulhi(ra.x, (uint32_t) cnt);
	out[1] = (u01(ra.y) - 0.5) * rp.disp_max;
	out[2] = (u01(ra.z) - 0.5) * rp.disp_max;
	out[3] = (u01(ra.w) - 0.5) * rp.disp_max;
	rotation_matrix(axis, st, ct, R);
#pragma unroll
	for(int c = 0; c < 9; c++) out[4 + c] = R[c];
	return rb.w;
}

// Trial geometry shared by the helpers of one team.
struct Trial {
	double px, py, pz, nx, ny, nz;
	double Lx, Ly, Lz, iLx, iLy, iLz, rc2, cosmax;
	double c2;  // cosmax^2 for the filter's check (a trial's own tests are exact)
};

// Minimum-image separation of q from the trial's new position, and its
// square (MC.c:232-240)
__device__ __forceinline__ double sep_new(const Trial &t, double qx, double qy, double qz, double &wx, double &wy,
                                          double &wz) {
	wx = kf_min_image(qx - t.nx, t.Lx, t.iLx);
	wy = kf_min_image(qy - t.ny, t.Ly, t.iLy);
	wz = kf_min_image(qz - t.nz, t.Lz, t.iLz);
	return wx * wx + wy * wy + wz * wz;
}

__device__ __forceinline__ bool overlaps_new(const Trial &t, double qx, double qy, double qz) {
	double dx, dy, dz;
	return sep_new(t, qx, qy, qz, dx, dy, dz) < 1.;
}

// Bonds of neighbour q with the old and the new position (one load of q for
// both: the particle stays in its cell, so the neighbourhood is the same),
// with the reference's arithmetic (MC.c:242-262).  q's orientation comes from
// load_o only when one of the two passes the p-side test.
template <class LoadO>
__device__ __forceinline__ void bonds_old_new_exact(const Trial &t, const double *Po, const double *Pn, double qx,
                                                    double qy, double qz, LoadO load_o, int &bo, int &bn) {
	double ox = kf_min_image(qx - t.px, t.Lx, t.iLx);
	double oy = kf_min_image(qy - t.py, t.Ly, t.iLy);
	double oz = kf_min_image(qz - t.pz, t.Lz, t.iLz);
	double o2 = ox * ox + oy * oy + oz * oz;
	double wx = kf_min_image(qx - t.nx, t.Lx, t.iLx);
	double wy = kf_min_image(qy - t.ny, t.Ly, t.iLy);
	double wz = kf_min_image(qz - t.nz, t.Lz, t.iLz);
	double w2 = wx * wx + wy * wy + wz * wz;
	bool po = false, pn = false;
	if(o2 < t.rc2) {
		kf_unit(ox, oy, oz, o2);
		po = kf_any_p(ox, oy, oz, Po, t.cosmax);
	}
	if(w2 < t.rc2) {
		kf_unit(wx, wy, wz, w2);
		pn = kf_any_p(wx, wy, wz, Pn, t.cosmax);
	}
	if(po || pn) {
		double Oq[9];
		load_o(Oq);
		bool ho, hn;
		kf_any_q2(ox, oy, oz, po, wx, wy, wz, pn, Oq, t.cosmax, ho, hn);
		bo += ho;
		bn += hn;
	}
}

// The bond decision of a pair closer than the bond range (MC_would_interact's
// angular part, MC.c:248-262), seen from p with separation (dx, dy, dz) towards
// q, its square d2 and p's patches P.  Seen from q the decision is the same
// (every step is the exact negation of p's).  q's orientation is read only
// when p's patches pass.
//
// The filter's answer, for c2 = cosmax^2: KF_YES, KF_NO, or KF_UNSURE inside
// its band.
template <class LoadO>
__device__ __forceinline__ unsigned pair_filter(double dx, double dy, double dz, double d2, const double *P, double c2,
                                                LoadO load_q) {
	const KfBand bd = kf_band(c2, d2);
	const unsigned fp = kf_fast_p(dx, dy, dz, P, bd);
	unsigned yes = 0u, unsure = fp >> 1;
	if(fp & 1u) {
		double Oq[9];
		load_q(Oq);
		const unsigned fq = kf_fast_q1(dx, dy, dz, kf_band_q(bd), Oq);
		unsure |= fq >> 1;
		yes = fq & 1u;
	}
	return unsure ? (unsigned) KF_UNSURE : yes;
}

// The reference's arithmetic.
template <class LoadO>
__device__ __forceinline__ bool pair_exact(double dx, double dy, double dz, double d2, const double *P, double cosmax,
                                           LoadO load_q) {
	kf_unit(dx, dy, dz, d2);
	if(!kf_any_p(dx, dy, dz, P, cosmax)) return false;
	double Oq[9];
	load_q(Oq);
	return kf_any_q(dx, dy, dz, Oq, cosmax);
}

// The filter, and the reference's arithmetic where it is unsure or not in use
// (c2 < 0).
template <class LoadO>
__device__ __forceinline__ bool pair_bonded(double dx, double dy, double dz, double d2, const double *P, double c2,
                                            double cosmax, LoadO load_q) {
	const unsigned f = c2 < 0. ? (unsigned) KF_UNSURE : pair_filter(dx, dy, dz, d2, P, c2, load_q);
	if(f == KF_UNSURE) return pair_exact(dx, dy, dz, d2, P, cosmax, load_q);
	return f == KF_YES;
}

// Bonds of neighbour q with a trial's new position by either half of
// pair_bonded, as the check of the filter at its thresholds asks for them:
// the filter's (a pair inside its band sets `band`) for the separation (wx, wy,
// wz) = sep_new(q) and its square w2, and the reference's.
template <class LoadO>
__device__ __forceinline__ void bonds_new_sep(const Trial &t, const double *Pn, double wx, double wy, double wz,
                                              double w2, LoadO load_o, int &bn, bool &band) {
	const unsigned f = w2 < t.rc2 ? pair_filter(wx, wy, wz, w2, Pn, t.c2, load_o) : (unsigned) KF_NO;
	bn += f == KF_YES;
	band |= f == KF_UNSURE;
}

template <class LoadO>
__device__ __forceinline__ void bonds_new_exact(const Trial &t, const double *Pn, double qx, double qy, double qz,
                                                LoadO load_o, int &bn) {
	double wx, wy, wz;
	const double w2 = sep_new(t, qx, qy, qz, wx, wy, wz);
	if(w2 < t.rc2) bn += pair_exact(wx, wy, wz, w2, Pn, t.cosmax, load_o);
}

}  // namespace ppd
