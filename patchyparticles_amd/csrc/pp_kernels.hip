// pp_kernels.hip -- gfx950 kernels of the Kern-Frenkel rototranslation hot path.
//
// Data layout in HBM (per context, all replicas concatenated):
//   f[2][slots][12]   double  x, y, z, O00..O22 of slot j (two buffers)
//   pid[2][slots]     int     particle index of slot j
//   start[C+1]        int     first slot of each cell, over the concatenated
//                             cell regions of all replicas (one region per
//                             replica, sized for its largest grid)
// Slots are grouped by cell at every rebuild (order inside a cell is
// whatever the atomics gave); the colour pass ranks a cell's members by
// particle index before it draws from them, so the trajectory depends only
// on the state and the seed, never on thread timing.
//
// Sweep = rebuild on a randomly shifted grid + 8 colour passes in random
// order.  In a pass every cell of one colour (i,j,k parities) is active; its
// neighbourhood holds no other active cell, so one team of T lanes per active
// cell can move that cell's particles while all others stay put.  A trial that
// leaves the cell is rejected, which keeps cell populations fixed during the
// pass: the team makes exactly as many sequential trials as the cell holds,
// so a sweep is exactly N attempts, as a reference sweep (MC.c:19-29).
#pragma clang fp contract(off)

#include "pp_device.hpp"

namespace ppd {

// ------------------------------------------------------------------------
// fills

// Workgroups of 256 threads for n values, which they take in turn: a launch
// has fewer than 2^32 threads (10^8 particles have 10^10 record words).
constexpr long long FILL_BLOCKS = 1 << 20;
static dim3 fill_grid(long long n) { return dim3((unsigned) std::min((n + 255) / 256, FILL_BLOCKS)); }
__device__ __forceinline__ long long fill_first() { return (long long) blockIdx.x * 256 + threadIdx.x; }
__device__ __forceinline__ long long fill_step() { return (long long) gridDim.x * 256; }

__global__ __launch_bounds__(256) void k_fill_i32(int *p, int v, long long n) {
	for(long long i = fill_first(); i < n; i += fill_step()) p[i] = v;
}

__global__ __launch_bounds__(256) void k_fill_u64(unsigned long long *p, unsigned long long v, long long n) {
	for(long long i = fill_first(); i < n; i += fill_step()) p[i] = v;
}

void launch_fill_i32(int *p, int v, long long n, hipStream_t s) {
	if(n > 0) hipLaunchKernelGGL(k_fill_i32, fill_grid(n), dim3(256), 0, s, p, v, n);
}

void launch_fill_u64(unsigned long long *p, unsigned long long v, long long n, hipStream_t s) {
	if(n > 0) hipLaunchKernelGGL(k_fill_u64, fill_grid(n), dim3(256), 0, s, p, v, n);
}

// Mark every cell record as no sweep's (tag 0).
__global__ __launch_bounds__(256) void k_clear_tags(int *rec, long long n) {
	for(long long i = fill_first(); i < n; i += fill_step()) rec[i * REC_W + REC_TAG] = 0;
}

void launch_clear_tags(const DevState &d, hipStream_t s) {
	const long long n = 8LL * std::max(d.total_act, 1);
	hipLaunchKernelGGL(k_clear_tags, fill_grid(n), dim3(256), 0, s, d.rec, n);
}

// Zero the energy-kernel rows (C_EBONDS, C_OVL) of every replica.
__global__ void k_zero_energy_rows(unsigned long long *ctr, int R) {
	int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= R * 2 * NSLOT) return;
	int r = i / (2 * NSLOT), k = i % (2 * NSLOT);
	int row = k < NSLOT ? C_EBONDS : C_OVL;
	*ctr_at(ctr, r, row, k % NSLOT) = 0ull;
}

// ------------------------------------------------------------------------
// rebuild: count -> scan (flips the buffer selector) -> scatter
//
// mode REB_KEEP   regroup on the current grid and shift
//      REB_SHIFT  new random grid shift for this sweep (uniform in one cell
//                 side per axis), recorded by the first slot of each replica
//      REB_TRIAL  NPT trial: the replicas with a trial in flight are counted
//                 on their trial grid with the trial scaling of one axis
//                 (MC.c:475-478); the others on their grid, unscaled, so that
//                 every replica's cells still start at its own first slot

__device__ __forceinline__ void sweep_shift(const DevState &d, int r, const Grid &G, uint64_t sweep, double sh[3]) {
	u32x4 v = rng(d.seed, r, sweep, 0, TAG_SHIFT, 0, 0);
	sh[0] = u01(v.x) * (G.box[0] / (double) G.n[0]);
	sh[1] = u01(v.y) * (G.box[1] / (double) G.n[1]);
	sh[2] = u01(v.z) * (G.box[2] / (double) G.n[2]);
}

// Replica whose cell region holds global cell c.
__device__ __forceinline__ int replica_of_cell(const DevState &d, int c) {
	int lo = 0, hi = d.R;
	while(hi - lo > 1) {
		const int mid = (lo + hi) >> 1;
		if(d.reps[mid].cell_off <= c) lo = mid;
		else hi = mid;
	}
	return lo;
}

// A trial that regroups the replica's particles into the spare buffer (a
// box trial whose grid the current lists cannot serve).
__device__ __forceinline__ bool trial_rebuilds(const Rep &rp) { return rp.trial_active && !rp.trial_fast; }

__device__ __forceinline__ void set_pass_geo(Rep &rp, const Grid &G, const double sh[3]) {
	PassGeo &p = rp.pg;
	double smax = 0., gap = G.box[0];
	for(int k = 0; k < 3; k++) {
		p.box[k] = G.box[k];
		p.inv_box[k] = G.inv_box[k];
		p.shift[k] = sh[k];
		p.side[k] = G.box[k] / (double) G.n[k];
		p.inv_side[k] = (float) ((double) G.n[k] / G.box[k]);
		smax = fmax(smax, p.side[k]);
		gap = fmin(gap, G.box[k] - p.side[k]);
	}
	p.filter = f32_filter(rp.cosmax, rp.rc2, smax);
	p.margin = 1e-5f;
	// A step of the box less a cell comes round the box into its own cell,
	// where the filter has the particle a box length away from its neighbours
	// (shorter ones that leave the cell are rejected by the in-cell test,
	// whatever their length); an infinite angle makes no rotation.  Everything
	// is exact then.
	if(!(0.5 * rp.disp_max < 0.999 * gap) || !(rp.theta_max < 1e300)) p.filter.eps_d2 = p.filter.eps_t = p.margin = F32_ALL;
	for(int k = 0; k < 3; k++) p.n[k] = G.n[k];
}

// The start of a sweep (REB_SHIFT) in a replica's table: the grid shift, the
// colour order and the passes' constants.
__device__ __forceinline__ void begin_sweep(const DevState &d, Rep &rp, int r, uint64_t sweep, const double sh[3]) {
	for(int k = 0; k < 3; k++) rp.g.shift[k] = sh[k];
	// random colour order of this sweep's 8 passes
	u32x4 v = rng(d.seed, r, sweep, 0, TAG_COLOUR, 0, 0);
	const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
	rp.col_perm = colour_perm_from(w4);
	set_pass_geo(rp, rp.g, sh);
}

// The lists a rebuild of the current state (not a trial) makes are by
// membership in the grid of shift sh.
__device__ __forceinline__ void begin_lists(Rep &rp, int mode, const double sh[3]) {
	rp.lg = rp.g;
	for(int k = 0; k < 3; k++) rp.lg.shift[k] = sh[k];
	rp.lists_ok = 1;
	rp.rec_ok = mode == REB_SHIFT;  // only that rebuild writes the cell records
}

// Empty what is collected anew in a sweep.
__device__ __forceinline__ void reset_sweep_lists(const DevState &d, int mode) {
	d.scan_ticket[0] = 0;
	if(mode == REB_SHIFT && d.pl_n) {
		// the sweep's list of close pairs, built after its passes
		d.pl_n[0] = 0;
		d.pl_n[1] = 0;
	}
}

// The place of a slot in cell c, counted in `count`.  The slots a
// grand-canonical replica does not use all go to one cell (parked): a
// wavefront's together (one by one, 900 of them took 8 us of a 12 us kernel).
__device__ __forceinline__ int take_place(int *count, int c, bool parked) {
	int at = 0;
	for(unsigned long long left = ballot(parked); left != 0ull;) {
		const int cl = __builtin_amdgcn_readlane(c, (int) __builtin_ctzll(left));
		const unsigned long long mates = ballot(parked && c == cl);
		if(parked && c == cl) {
			const int before = __popcll(mates & ((1ull << (threadIdx.x & 63)) - 1ull));
			int base = 0;
			if(before == 0) base = atomicAdd(&count[c], __popcll(mates));
			at = __builtin_amdgcn_readlane(base, (int) __builtin_ctzll(mates)) + before;
		}
		left &= ~mates;
	}
	if(!parked) at = atomicAdd(&count[c], 1);
	return at;
}

// ONE: a context of one replica, whose table then loads to scalar registers.
template <bool ONE>
__global__ void k_count(DevState d, int mode, uint64_t sweep, long long trace_pos) {
	int j = blockIdx.x * blockDim.x + threadIdx.x;
	// reset the scan's look-back state for the scan that follows
	for(int t = j; t < d.ntiles; t += gridDim.x * blockDim.x) d.scan_status[t] = 0ull;
	for(int t = j; t < d.R * 8; t += gridDim.x * blockDim.x) d.ccount[t] = 0;
	if(j == 0) reset_sweep_lists(d, mode);
	if(mode == REB_TRIAL)
		// replicas without a trial rebuild keep their lists as they are:
		// their cells' counts are the current populations, so the scan
		// reproduces their starts
		for(int c = j; c < d.C_total; c += gridDim.x * blockDim.x)
			if(!trial_rebuilds(d.reps[replica_of_cell(d, c)])) d.count[c] = d.start[c + 1] - d.start[c];
	if(j >= d.Ntot) return;
	const int r = ONE ? 0 : d.prep[j];
	Rep &rp = d.reps[r];
	const bool tr = (mode == REB_TRIAL) && trial_rebuilds(rp);
	if(mode == REB_TRIAL && !tr) return;
	const Grid &G = tr ? rp.tg : rp.g;
	double sh[3] = {G.shift[0], G.shift[1], G.shift[2]};
	if(mode == REB_SHIFT) {
		sweep_shift(d, r, G, sweep, sh);
		if(j == rp.p_off) {
			// energy trace: bonded pairs as they stand after the previous sweep
			if(d.trace && trace_pos >= 0 && trace_pos < d.trace_cap) {
				unsigned long long db = 0;
				for(int k = 0; k < NSLOT; k++) db += *ctr_at(d.ctr, r, C_DBONDS, k);
				d.trace[(long long) r * d.trace_cap + trace_pos] = rp.bonds_base + (long long) db;
			}
			begin_sweep(d, rp, r, sweep, sh);
		}
	}
	if(!tr && j == rp.p_off) begin_lists(rp, mode, sh);
	// a free or removed slot of a grand-canonical replica goes to the
	// replica's parking cell
	int c = rp.cell_off + rp.cell_cap;
	if(j - rp.p_off < rp.np_hw && pick_buf(d.pid, rp.sel)[j] >= 0) {
		const double *F = pick_buf(d.f, rp.sel);
		double p[3] = {part(F, j)[0], part(F, j)[1], part(F, j)[2]};
		if(tr)
			for(int k = 0; k < 3; k++) p[k] *= rp.trial_s[k];
		int ix = cell_coord(p[0], sh[0], G.inv_box[0], G.n[0]);
		int iy = cell_coord(p[1], sh[1], G.inv_box[1], G.n[1]);
		int iz = cell_coord(p[2], sh[2], G.inv_box[2], G.n[2]);
		c = rp.cell_off + (ix * G.n[1] + iy) * G.n[2] + iz;
	}
	d.cellid[j] = c;
	d.slot[j] = take_place(d.count, c, c == rp.cell_off + rp.cell_cap);
}

// A lane's PER consecutive cells of a tile: whole vectors where all PER
// are in the grid (base is a multiple of PER, the arrays 16-byte aligned).
template <int PER>
__device__ __forceinline__ void load_cells(const int *p, int base, int n, int v[PER]) {
	static_assert(PER == 2 || PER % 4 == 0, "2 or a multiple of 4 cells per lane");
	if(base + PER <= n) {
		if constexpr(PER == 2) {
			const int2 q = *(const int2 *) (p + base);
			v[0] = q.x;
			v[1] = q.y;
		}
		else
#pragma unroll
			for(int e = 0; e < PER; e += 4) {
				const int4 q = *(const int4 *) (p + base + e);
				v[e] = q.x;
				v[e + 1] = q.y;
				v[e + 2] = q.z;
				v[e + 3] = q.w;
			}
	}
	else
#pragma unroll
		for(int e = 0; e < PER; e++) v[e] = base + e < n ? p[base + e] : 0;
}

template <int PER>
__device__ __forceinline__ void store_cells(int *p, int base, int n, const int v[PER]) {
	if(base + PER <= n) {
		if constexpr(PER == 2) *(int2 *) (p + base) = make_int2(v[0], v[1]);
		else
#pragma unroll
			for(int e = 0; e < PER; e += 4) *(int4 *) (p + base + e) = make_int4(v[e], v[e + 1], v[e + 2], v[e + 3]);
	}
	else
#pragma unroll
		for(int e = 0; e < PER; e++)
			if(base + e < n) p[base + e] = v[e];
}

// Count and scan of one small replica in one workgroup, the cells' counts in
// LDS (d.count stays clear).  k_count and k_scan are mostly round trips to
// memory (the ticket, the counts, the look-back, the lists' atomics); here
// each round of 1024 particles costs about 2 us, so it ends at three.  Both
// kernels against this one: N=300 (512 cells) 9.1 -> 4.9 us, N=1000 (5832
// cells) 9.9 -> 7.3, N=2700 9.3 -> 8.8, N=4000 9.7 -> 11.6.
constexpr int CS_CELLS = 8192;     // cells, the parking cell included
constexpr int CS_PARTICLES = 3072;
constexpr int CS_THREADS = 1024, CS_PER = CS_CELLS / CS_THREADS;

__global__ __launch_bounds__(CS_THREADS) void k_count_scan(DevState d, int mode, uint64_t sweep, long long trace_pos) {
	__shared__ __attribute__((aligned(16))) int cnt[CS_CELLS];
	__shared__ int wsum[CS_THREADS / 64];
	const int t = threadIdx.x, lane = t & 63, w = t >> 6;
	Rep &rp = d.reps[0];
#pragma unroll
	for(int e = 0; e < CS_PER; e += 4) *(int4 *) (cnt + t * CS_PER + e) = make_int4(0, 0, 0, 0);
	const int n0 = rp.g.n[0], n1 = rp.g.n[1], n2 = rp.g.n[2], sel = rp.sel, parking = rp.cell_cap;
	double sh[3] = {rp.g.shift[0], rp.g.shift[1], rp.g.shift[2]};
	if(mode == REB_SHIFT) sweep_shift(d, 0, rp.g, sweep, sh);
	const double i0 = rp.g.inv_box[0], i1 = rp.g.inv_box[1], i2 = rp.g.inv_box[2];
	__syncthreads();
	for(int j = t; j < d.Ntot; j += CS_THREADS) {
		int c = parking;
		if(j < rp.np_hw && pick_buf(d.pid, sel)[j] >= 0) {
			const double *p = part((const double *) pick_buf(d.f, sel), j);
			c = (cell_coord(p[0], sh[0], i0, n0) * n1 + cell_coord(p[1], sh[1], i1, n1)) * n2 + cell_coord(p[2], sh[2], i2, n2);
		}
		d.cellid[j] = c;
		d.slot[j] = take_place(cnt, c, c == parking);
	}
	__syncthreads();
	// first slots
	int v[CS_PER], tot = 0;
#pragma unroll
	for(int e = 0; e < CS_PER; e++) {
		v[e] = cnt[t * CS_PER + e];
		tot += v[e];
	}
	const int inc = wave_incl_scan(tot);
	if(lane == 63) wsum[w] = inc;
	__syncthreads();
	int run = inc - tot;
	for(int k = 0; k < w; k++) run += wsum[k];
	int first[CS_PER];
#pragma unroll
	for(int e = 0; e < CS_PER; e++) {
		first[e] = run;
		run += v[e];
	}
	if(t * CS_PER < d.C_total) store_cells<CS_PER>(d.start, t * CS_PER, d.C_total, first);
	// the table's entries for this rebuild (every thread has read the old
	// ones), by wavefronts that make no list
	if(t == CS_THREADS - 64) {
		reset_sweep_lists(d, mode);
		if(mode == REB_SHIFT) begin_sweep(d, rp, 0, sweep, sh);
		begin_lists(rp, mode, sh);
		rp.sel = sel ^ 1;
		d.start[d.C_total] = d.Ntot;
	}
	if(w == 8 && mode == REB_SHIFT && d.trace && trace_pos >= 0 && trace_pos < d.trace_cap) {
		// energy trace: bonded pairs as they stand after the previous sweep
		static_assert(NSLOT == 64, "a lane per slot");
		unsigned long long db = *ctr_at(d.ctr, 0, C_DBONDS, lane);
		for(int o = 32; o > 0; o >>= 1) db += __shfl_xor(db, o);
		if(lane == 0) d.trace[trace_pos] = rp.bonds_base + (long long) db;
	}
	if(mode != REB_SHIFT || w >= 8) return;
	// the passes' lists: wavefront w takes the cells of colour w in order
	const int h1 = n1 / 2, h2 = n2 / 2, cells = n0 / 2 * h1 * h2;
	const int sa = 64 / (h1 * h2), sb = 64 % (h1 * h2) / h2, sc = 64 % h2;  // 64 cells on, per axis
	int a = lane / (h1 * h2), b = lane / h2 % h1, c = lane % h2, n = 0;
	int *list = d.clist + w * rp.act_cap;
	for(int k = lane; __any(k < cells); k += 64) {
		const int cloc = ((2 * a + (w >> 2)) * n1 + 2 * b + ((w >> 1) & 1)) * n2 + 2 * c + (w & 1);
		const bool on = k < cells && cnt[cloc] > 0;
		const unsigned long long m = ballot(on);
		if(on) list[n + __popcll(m & ((1ull << lane) - 1ull))] = cloc;
		n += __popcll(m);
		c += sc;
		b += sb;
		a += sa;
		if(c >= h2) {
			c -= h2;
			b++;
		}
		if(b >= h1) {
			b -= h1;
			a++;
		}
	}
	if(lane == 0) d.ccount[w] = n;
}

// (replica, colour) keys of the non-empty-cell lists counted per scan workgroup
constexpr int SCAN_KEYS = 512;

// Exclusive scan of the cell counts in one pass (decoupled look-back):
// workgroups take tiles in dispatch order from a ticket, publish their tile
// sum, then read their predecessors' published values, 64 at a time, back to
// the nearest one that carries an inclusive prefix.  A workgroup only ever waits for tiles with a
// smaller ticket, which are already running.  start[c] = first slot of cell
// c; count is cleared for the next rebuild; a flipping scan also switches
// every replica to the buffer the scatter fills.
// Sum of the cell counts of each scan tile.
template <int PER>
__global__ __launch_bounds__(256) void k_tile_sums(DevState d) {
	__shared__ int part[4];
	const int t = threadIdx.x, base = blockIdx.x * (256 * PER) + t * PER;
	int v[PER];
	load_cells<PER>(d.count, base, d.C_total, v);
	int tot = 0;
#pragma unroll
	for(int e = 0; e < PER; e++) tot += v[e];
	tot = team_sum<64>(tot);
	if((t & 63) == 0) part[t >> 6] = tot;
	__syncthreads();
	if(t == 0) d.tile_sum[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Exclusive prefix of the tile sums, in place (one workgroup).
__global__ __launch_bounds__(1024) void k_tile_scan(DevState d) {
	__shared__ int part[1024];
	const int t = threadIdx.x, n = d.ntiles;
	const int per = (n + 1023) / 1024, lo = t * per, hi = min(n, lo + per);
	int s = 0;
	for(int i = lo; i < hi; i++) s += d.tile_sum[i];
	part[t] = s;
	__syncthreads();
	for(int o = 1; o < 1024; o <<= 1) {
		const int v = t >= o ? part[t - o] : 0;
		__syncthreads();
		part[t] += v;
		__syncthreads();
	}
	int run = part[t] - s;
	for(int i = lo; i < hi; i++) {
		const int v = d.tile_sum[i];
		d.tile_sum[i] = run;
		run += v;
	}
}

// pre = 1: the tiles' exclusive prefixes are in d.tile_sum (k_tile_sums,
// k_tile_scan); pre = 0: a decoupled look-back finds them.
// PER cells per lane: tiles of 256 * PER cells.
// ONE: a context of one replica (its table in scalar registers).
template <int PER, bool ONE>
__global__ __launch_bounds__(256) void k_scan(DevState d, int flip, int lists, int pre) {
	__shared__ int wsum[4];
	__shared__ int sh_tile, sh_excl, sh_r0;
	__shared__ int lcnt[SCAN_KEYS], lbase[SCAN_KEYS];
	const int t = threadIdx.x;
	if(t == 0) sh_tile = atomicAdd(d.scan_ticket, 1);
	for(int k = t; k < SCAN_KEYS; k += 256) lcnt[k] = 0;
	__syncthreads();
	const int tile = sh_tile;
	const int base = tile * (256 * PER) + t * PER;
	if(t == 0 && lists && !ONE) {
		// replica of the tile's first cell
		int lo = 0, hi = d.R;
		while(hi - lo > 1) {
			int mid = (lo + hi) >> 1;
			if(d.reps[mid].cell_off <= tile * (256 * PER)) lo = mid;
			else hi = mid;
		}
		sh_r0 = lo;
	}
	int v[PER];
	load_cells<PER>(d.count, base, d.C_total, v);
	int tot = 0;
#pragma unroll
	for(int e = 0; e < PER; e++) tot += v[e];
	int lane = t & 63, wid = t >> 6;
	const int inc = wave_incl_scan(tot);
	if(lane == 63) wsum[wid] = inc;
	__syncthreads();
	if(pre) {
		if(t == 0) sh_excl = d.tile_sum[tile];
	}
	else if(wid == 0) {
		// wavefront 0 publishes the tile's sum and looks back over up to 64
		// predecessors at once: the nearest one with an inclusive prefix ends
		// the walk; one that has published nothing yet is polled again.  A
		// status word carries its flag and its value together, so relaxed
		// agent-scope atomics suffice (a release would write the XCD's L2
		// back on every publication).
		const int agg = wsum[0] + wsum[1] + wsum[2] + wsum[3];
		int excl = 0;
		if(lane == 0)
			__hip_atomic_store(&d.scan_status[tile], ((tile == 0 ? 2ull : 1ull) << 32) | (unsigned) agg,
			                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		int p = tile - 1, spins = 0;
		while(p >= 0) {
			const int q = p - lane;
			unsigned long long st = 2ull << 32;  // before tile 0: an inclusive prefix of 0
			if(q >= 0) st = __hip_atomic_load(&d.scan_status[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			const unsigned flag = (unsigned) (st >> 32);
			const unsigned long long m2 = __ballot(flag == 2u);
			const int l2 = m2 ? __ffsll((long long) m2) - 1 : 64;
			const unsigned long long upto = l2 >= 63 ? ~0ull : ((2ull << l2) - 1ull);
			if(__ballot(flag == 0u) & upto) {
				if(++spins > SCAN_SPIN_MAX) {
					if(lane == 0) atomicOr(d.err, (int) ERR_SCAN);
					break;
				}
				__builtin_amdgcn_s_sleep(1);
				continue;
			}
			int val = lane <= l2 ? (int) (st & 0xffffffffull) : 0;
			excl += team_sum<64>(val);
			if(l2 < 64) break;
			p -= 64;
		}
		if(lane == 0) {
			if(tile > 0)
				__hip_atomic_store(&d.scan_status[tile], (2ull << 32) | (unsigned) (excl + agg), __ATOMIC_RELAXED,
				                   __HIP_MEMORY_SCOPE_AGENT);
			sh_excl = excl;
		}
	}
	__syncthreads();
	int woff = 0;
	for(int w = 0; w < wid; w++) woff += wsum[w];
	// the cells' first slots; their counts cleared for the next rebuild
	{
		int first[PER], zero[PER];
		int run = sh_excl + woff + inc - tot;
#pragma unroll
		for(int e = 0; e < PER; e++) {
			first[e] = run;
			zero[e] = 0;
			run += v[e];
		}
		store_cells<PER>(d.start, base, d.C_total, first);
		store_cells<PER>(d.count, base, d.C_total, zero);
	}
	int lkey[PER], lpos[PER];
#pragma unroll
	for(int e = 0; e < PER; e++) {
		int c = base + e;
		lkey[e] = -1;
		lpos[e] = 0;
		if(c < d.C_total) {
			if(lists && v[e] > 0) {
				// the next passes visit only non-empty cells: list them by
				// colour, first counted per workgroup in LDS
				int lo = ONE ? 0 : sh_r0, hi = d.R;
				if constexpr(!ONE)
					while(hi - lo > 1) {
						int mid = (lo + hi) >> 1;
						if(d.reps[mid].cell_off <= c) lo = mid;
						else hi = mid;
					}
				const Rep &rp = d.reps[ONE ? 0 : lo];
				const int cloc = c - rp.cell_off;
				const int n1 = rp.g.n[1], n2 = rp.g.n[2];
				const int ix = cloc / (n1 * n2), iy = (cloc / n2) % n1, iz = cloc % n2;
				const int col = ((ix & 1) << 2) | ((iy & 1) << 1) | (iz & 1);
				const int key = ONE ? col : (lo - sh_r0) * 8 + col;
				if(cloc >= rp.g.n[0] * n1 * n2) {
					// the parking cell: free slots, no particles to move
				}
				else if(key < SCAN_KEYS) {
					lkey[e] = key;
					lpos[e] = atomicAdd(&lcnt[key], 1);
				}
				else {
					// a tile spanning more than SCAN_KEYS / 8 replicas: direct
					const int k = atomicAdd(&d.ccount[lo * 8 + col], 1);
					d.clist[rp.cell_off + col * rp.act_cap + k] = cloc;
				}
			}
		}
	}
	if(lists) {
		__syncthreads();
		for(int k = t; k < (ONE ? 8 : SCAN_KEYS); k += 256) {
			const int n = lcnt[k];
			if(n > 0) lbase[k] = atomicAdd(&d.ccount[((ONE ? 0 : sh_r0) + k / 8) * 8 + k % 8], n);
		}
		__syncthreads();
#pragma unroll
		for(int e = 0; e < PER; e++)
			if(lkey[e] >= 0) {
				const int r = ONE ? 0 : sh_r0 + lkey[e] / 8;
				const Rep &rp = d.reps[r];
				const int cloc = base + e - rp.cell_off;
				d.clist[rp.cell_off + (lkey[e] & 7) * rp.act_cap + lbase[lkey[e]] + lpos[e]] = cloc;
			}
	}
	if(tile == 0) {
		if(t == 0) d.start[d.C_total] = d.Ntot;
		if(flip)
			for(int r = t; r < d.R; r += 256) d.reps[r].sel ^= 1;
	}
}

// The layout of the passes' lists, after the scan has counted them:
// pfx[k][r] = first entry of replica r in the list of pass k, by wavefront k
// (the kernel boundary makes every workgroup's counts visible).  Also resets
// the ticket queue of the dependency-driven sweep and the lists of deferred
// cells.  A thread per pass adding 256 replicas one by one took 80 us; a
// wavefront's scan takes 5.
__device__ __forceinline__ void pass_prefix(const DevState &d, int k, int lane) {
	if(lane == 0) {
		if(k == 0 && d.ddq) *d.ddq = 0;
		if(d.ovf_n) d.ovf_n[k] = 0;
	}
	int *pf = d.pfx + k * (d.R + 1);
	if(lane == 0) pf[0] = 0;
	int base = 0;
	for(int r0 = 0; r0 < d.R; r0 += 64) {
		const int r = r0 + lane;
		int n = 0;
		if(r < d.R) n = d.ccount[r * 8 + (int) ((d.reps[r].col_perm >> (4 * k)) & 0xFu)];
		const int inc = wave_incl_scan(n);
		if(r < d.R) pf[r + 1] = base + inc;
		base += __builtin_amdgcn_readlane(inc, 63);
	}
}

__global__ __launch_bounds__(512) void k_pass_prefix(DevState d) { pass_prefix(d, threadIdx.x >> 6, threadIdx.x & 63); }

// The record of entry gi of pass k's list, by the 16 lanes of a team.
template <bool ONE>
__device__ __forceinline__ void build_record(const DevState &d, int k, int gi, int lane) {
	int r = 0;
	if constexpr(!ONE) {
		// the replica whose entries of pass k hold gi: the last r with
		// pfx[r] <= gi, the team's lanes probing 16 places at once
		const int *pf = d.pfx + k * (d.R + 1);
		for(int n = d.R; n > 1;) {
			const int step = (n + 15) / 16, at = r + lane * step;
			const bool le = lane * step < n && pf[at] <= gi;
			const int off = threadIdx.x & 63 & ~15;
			const unsigned m = (unsigned) (ballot(le) >> off) & 0xffffu;  // lane 0 always, then a run
			const int last = 31 - __clz((int) m);
			r += last * step;
			n = min(step, n - last * step);
		}
	}
	const Rep &rp = d.reps[r];
	const int kk = ONE ? gi : gi - d.pfx[k * (d.R + 1) + r];
	const int col = (int) ((rp.col_perm >> (4 * k)) & 0xFu);
	const int cloc = d.clist[rp.cell_off + col * rp.act_cap + kk];
	const int n0 = rp.g.n[0], n1 = rp.g.n[1], n2 = rp.g.n[2];
	const int ix = cloc / (n1 * n2), iy = (cloc / n2) % n1, iz = cloc % n2;
	write_record(d.rec + ((size_t) k * d.total_act + gi) * REC_W, (int) d.rec_tag, d.start + rp.cell_off, cloc, ix, iy, iz,
	             n0, n1, n2, r, rp.sel, lane);
}

// Workgroups of the scatter that build records (grid-stride over the listed
// cells): enough to fill the chip.
constexpr int REC_BLOCKS = 2048;
constexpr int PART_BLOCK = 256 / (NCOMP / 2);  // particles moved by one workgroup

// Move every particle to its cell's slot range.  After a flipping scan the
// source is the previous buffer (sel ^ 1); a trial writes into sel ^ 1.  Six
// lanes per particle, 16 bytes each: whole cache lines on both sides.
// With a new grid shift, workgroups past the particles' write the cell
// records of the sweep's passes.
// ONE: one replica, whose lists start at entry 0 of every pass; the first
// workgroup also writes the pass prefixes (k_pass_prefix's work), which the
// records then do not need.
template <bool ONE>
__global__ __launch_bounds__(256) void k_scatter(DevState d, int mode, int part_blocks) {
	if constexpr(ONE)
		if(mode == REB_SHIFT && blockIdx.x == 0)
			for(int k = threadIdx.x >> 6; k < 8; k += 4) pass_prefix(d, k, threadIdx.x & 63);
	if((int) blockIdx.x >= part_blocks) {
		const int team = (blockIdx.x - part_blocks) * 16 + threadIdx.x / 16, teams = (gridDim.x - part_blocks) * 16;
		int len[8], total = 0;
#pragma unroll
		for(int k = 0; k < 8; k++) {
			len[k] = ONE ? d.ccount[(d.reps[0].col_perm >> (4 * k)) & 0xFu] : d.pfx[k * (d.R + 1) + d.R];
			total += len[k];
		}
		for(int i = team; i < total; i += teams) {
			int k = 0, gi = i;
			while(gi >= len[k]) gi -= len[k++];
			build_record<ONE>(d, k, gi, threadIdx.x & 15);
		}
		return;
	}
	constexpr int PER = NCOMP / 2;  // lanes per particle
	const int e = threadIdx.x % PER;
	const int j = blockIdx.x * PART_BLOCK + threadIdx.x / PER;
	if((int) threadIdx.x >= PART_BLOCK * PER || j >= d.Ntot) return;
	const int r = ONE ? 0 : d.prep[j];
	Rep &rp = d.reps[r];
	const bool tr = (mode == REB_TRIAL) && trial_rebuilds(rp);
	if(mode == REB_TRIAL && !tr) return;
	const int sb = tr ? rp.sel : (rp.sel ^ 1);
	const int dst = d.start[d.cellid[j]] + d.slot[j];
	double2 v = ((const double2 *) part((const double *) pick_buf(d.f, sb), j))[e];
	if(tr) {
		// (components 0, 1 and 2 are the position)
		if(e == 0) v.x *= rp.trial_s[0], v.y *= rp.trial_s[1];
		if(e == 1) v.x *= rp.trial_s[2];
	}
	((double2 *) part(pick_buf(d.f, sb ^ 1), dst))[e] = v;
	if(e == 0) {
		pick_buf(d.pid, sb ^ 1)[dst] = pick_buf(d.pid, sb)[j];
		// the buffer this rebuild switches to holds the live particles first
		if(mode != REB_TRIAL && j == rp.p_off) rp.np_hw = rp.np;
	}
}

static void launch_scatter(const DevState &d, int mode, hipStream_t s) {
	const unsigned pb = (unsigned) std::max(1, (d.Ntot + PART_BLOCK - 1) / PART_BLOCK);
	unsigned gs = pb;
	if(mode == REB_SHIFT) gs += (unsigned) std::min<long long>(REC_BLOCKS, (8LL * d.total_act + 15) / 16);
	if(d.R == 1) hipLaunchKernelGGL(k_scatter<true>, dim3(gs), dim3(256), 0, s, d, mode, (int) pb);
	else hipLaunchKernelGGL(k_scatter<false>, dim3(gs), dim3(256), 0, s, d, mode, (int) pb);
}

void launch_rebuild(const DevState &d, int mode, uint64_t sweep, long long trace_pos, hipStream_t s) {
	const int B = 256;
	unsigned gp = (unsigned) ((d.Ntot + B - 1) / B);
	if(gp == 0) gp = 1;
	const int flip = mode != REB_TRIAL;
	if(flip && d.R == 1 && d.Ntot <= CS_PARTICLES && d.C_total <= CS_CELLS) {
		hipLaunchKernelGGL(k_count_scan, dim3(1), dim3(CS_THREADS), 0, s, d, mode, sweep, trace_pos);
		launch_scatter(d, mode, s);
		return;
	}
	if(d.R == 1) hipLaunchKernelGGL(k_count<true>, dim3(gp), dim3(B), 0, s, d, mode, sweep, trace_pos);
	else hipLaunchKernelGGL(k_count<false>, dim3(gp), dim3(B), 0, s, d, mode, sweep, trace_pos);
	const int lists = mode == REB_SHIFT ? 1 : 0;
	if(d.scan_tile == SCAN_TILE_SMALL) {
		// at most SCAN_SMALL_MAX_TILES tiles: one pass with a look-back
		if(d.R == 1) hipLaunchKernelGGL((k_scan<SCAN_TILE_SMALL / 256, true>), dim3(d.ntiles), dim3(256), 0, s, d, flip, lists, 0);
		else hipLaunchKernelGGL((k_scan<SCAN_TILE_SMALL / 256, false>), dim3(d.ntiles), dim3(256), 0, s, d, flip, lists, 0);
	}
	else {
		// large tiles are taken only beyond SCAN_SMALL_MAX_TILES small ones,
		// so they always come in more tiles than a look-back serves well:
		// tile sums, one scan of the sums, then the tiles
		static_assert(SCAN_SMALL_MAX_TILES * SCAN_TILE_SMALL / SCAN_TILE_LARGE > SCAN_LOOKBACK_MAX_TILES,
		              "grids of large tiles always exceed the look-back's tile limit");
		hipLaunchKernelGGL(k_tile_sums<SCAN_TILE_LARGE / 256>, dim3(d.ntiles), dim3(256), 0, s, d);
		hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, s, d);
		hipLaunchKernelGGL((k_scan<SCAN_TILE_LARGE / 256, false>), dim3(d.ntiles), dim3(256), 0, s, d, flip, lists, 1);
	}
	if(mode == REB_SHIFT && d.R != 1) hipLaunchKernelGGL(k_pass_prefix, dim3(1), dim3(512), 0, s, d);
	launch_scatter(d, mode, s);
}

// ------------------------------------------------------------------------
// the callers' arrays into slots, at creation

// Slot j of every replica: particle i of its replica (j = p_off + i) in both
// index tables and the first buffer, or a free slot (index -1).  r and O hold
// the replicas' particles back to back (replica k's from src_off[k]); 12 lanes
// per slot.
__global__ __launch_bounds__(256) void k_place(DevState d, int *prep, const int *src_off, const double *r, const double *O) {
	const long long n = (long long) d.Ntot * NCOMP;
	for(long long t = fill_first(); t < n; t += fill_step()) {
		const int j = (int) (t / NCOMP), e = (int) (t % NCOMP);
		int lo = 0, hi = d.R;
		while(hi - lo > 1) {
			const int mid = (lo + hi) >> 1;
			if(d.reps[mid].p_off <= j) lo = mid;
			else hi = mid;
		}
		const Rep &rp = d.reps[lo];
		const int i = j - rp.p_off;
		const bool there = i < rp.np;
		const size_t src = (size_t) src_off[lo] + (there ? i : 0);
		double v = 0.;
		if(there) v = e < 3 ? r[3 * src + e] : O[9 * src + e - 3];
		part(d.f[0], j)[e] = v;
		if(e == 0) {
			d.pid[0][j] = d.pid[1][j] = there ? i : -1;
			prep[j] = lo;
		}
	}
}

void launch_place(const DevState &d, int *prep, const int *src_off, const double *r, const double *O, hipStream_t s) {
	const long long t = (long long) d.Ntot * NCOMP;
	if(t > 0) hipLaunchKernelGGL(k_place, fill_grid(t), dim3(256), 0, s, d, prep, src_off, r, O);
}

// ------------------------------------------------------------------------
// particles in index order, for a download

// The slot (from the replica's first) of each particle index, in d.slot
// (scratch of a rebuild); the header of the output.  Replicas of fixed size.
__global__ __launch_bounds__(256) void k_index_slots(DevState d, int rep, double *out) {
	const Rep &rp = d.reps[rep];
	const int j = blockIdx.x * 256 + threadIdx.x;
	if(j == 0) {
		for(int k = 0; k < 3; k++) out[UNPACK_BOX + k] = rp.g.box[k];
		out[UNPACK_BAD] = 0.;
	}
	if(j >= rp.np) return;
	const int i = pick_buf(d.pid, rp.sel)[rp.p_off + j];
	if(i >= 0 && i < rp.np) d.slot[rp.p_off + i] = j;
}

// out: the header, r[np][3], O[np][9].  12 lanes take one particle's
// contiguous 96 bytes, so that the gather reads whole lines; an index that no
// slot holds, or that two hold, leaves UNPACK_BAD != 0.  The host used to sort
// the indices and place every value itself: 2.4 ms for N=32768, 0.5 ms
// with the copies now.
__global__ __launch_bounds__(256) void k_unpack(DevState d, int rep, double *out) {
	const Rep &rp = d.reps[rep];
	const unsigned n = (unsigned) rp.np;
	double *r = out + UNPACK_HEAD, *O = r + 3 * (size_t) n;
	for(long long t = fill_first(); t < (long long) n * NCOMP; t += fill_step()) {
		const unsigned i = (unsigned) (t / NCOMP), e = (unsigned) (t % NCOMP);
		const unsigned j = (unsigned) d.slot[rp.p_off + i];
		if(j >= n || pick_buf(d.pid, rp.sel)[rp.p_off + j] != (int) i) {
			out[UNPACK_BAD] = 1. + (double) i;
			continue;
		}
		const double v = part((const double *) pick_buf(d.f, rp.sel), rp.p_off + (int) j)[e];
		if(e < 3) r[3 * (size_t) i + e] = v;
		else O[9 * (size_t) i + e - 3] = v;
	}
}

void launch_unpack(const DevState &d, int rep, int np, double *out, hipStream_t s) {
	const long long t = (long long) np * NCOMP;
	hipLaunchKernelGGL(k_index_slots, dim3((unsigned) std::max(1, (np + 255) / 256)), dim3(256), 0, s, d, rep, out);
	if(np > 0) hipLaunchKernelGGL(k_unpack, fill_grid(t), dim3(256), 0, s, d, rep, out);
}

// ------------------------------------------------------------------------
// the colour pass

struct PassArgs {
	DevState d;
	uint64_t sweep;
	int pass;
	unsigned mark;  // dependency-driven sweeps: the value a finished cell publishes in done[]
};

// Per-team LDS for cells of up to CAP members (offsets in 8-byte words):
//   SH  the members' single-precision records: position relative to the
//       cell's centre, O, the count of bonds with static neighbours, the
//       bits of the bonds with the other members
//   FT  the trials in single precision: displacement, the largest energy
//       rise their draw accepts, R, the moving member's rank
//   OWN the members' exact state, ranked by particle index: x, y, z, O, and
//       the position relative to the cell's centre
//   TR  the trials' exact displacement and R
//   PID particle indices
//   NB  (neighbourhoods beyond the record's list) the rows' slot ranges
//   GEO the cell's centre, for the far neighbours
constexpr int OWN_W = 15;  // x, y, z, O[9], rel[3]
constexpr int TR_W = 12;   // dx, dy, dz, R[9]
constexpr int SH_W = 14;   // floats: rel[3], O[9], static bonds, member bond bits
constexpr int FT_W = 14;   // floats: dx, dy, dz, the rise it accepts, R[9], rank
constexpr int NB_W = 40;   // ints: first slots [0, 18) and exclusive prefix [20, 39) of the rows' ranges
constexpr int GEO_W = 3;   // the cell's centre
template <int CAP>
struct TeamLds {
	static constexpr int TRIALS = CAP > MAX_TRIALS_PER_CELL ? CAP : MAX_TRIALS_PER_CELL;
	static constexpr int SH = 0;
	static constexpr int FT = SH + CAP * SH_W / 2;
	static constexpr int OWN = FT + TRIALS * FT_W / 2;
	static constexpr int TR = OWN + CAP * OWN_W;
	static constexpr int GEO = TR + TRIALS * TR_W;
	static constexpr int PID = GEO + GEO_W;
	static constexpr int NB = PID + (CAP + 1) / 2;
	// (the small-cell pass defers the neighbourhoods that need NB)
	static constexpr int SIZE = NB + (CAP < CELL_CAP ? 0 : NB_W / 2);
	static_assert(SH_W % 2 == 0 && FT_W % 2 == 0, "whole words");
};
// The small-cell pass (16-lane teams): cells of up to SMALL_CAP members whose
// neighbours fit the record's list, in 3.9 KB of LDS per team where a general
// team takes 8.2, so that the registers and not the LDS limit the wavefronts
// of a CU; other cells are deferred to the general pass.
constexpr int SMALL_CAP = 8;
template <int CAP = CELL_CAP>
constexpr int team_lds() {
	return TeamLds<CAP>::SIZE;
}
static_assert(16 * team_lds<>() * sizeof(double) <= 160 * 1024, "16 general teams per CU");
static_assert(40 * team_lds<SMALL_CAP>() * sizeof(double) <= 160 * 1024, "40 small-cell teams per CU");
static_assert(MAX_TEAMS * team_lds<>() * sizeof(double) <= MAX_LDS_BYTES, "a workgroup's teams");

constexpr int MOST_EXP = 1 << 16;  // a trial whose draw accepts every tabulated rise
constexpr float F32_FAR = 1e15f;   // the position of an empty slot, in no band of any trial's
static_assert(3.f * (3.f * F32_POS_LIM) * (3.f * F32_POS_LIM) < F32_ALL &&
                  F32_ALL < (F32_FAR - 2.f * F32_POS_LIM) * (F32_FAR - 2.f * F32_POS_LIM),
              "the infinite band holds every particle and no empty slot");

// One lane's share of an accepted move, values v = 0..14 of the moving
// member's record: v < 3 the position, v < 12 O' = O R in the reference's
// order (utils.c:172-184), else the position relative to the cell's centre.
// own: three words of the member's record from `o`, tr: of the trial from
// `r` with stride 3.
struct MoveShare {
	int o, r, word;  // word: the value's place in the single-precision record
	bool dot;
};
__device__ __forceinline__ MoveShare move_share(int v) {
	MoveShare m;
	m.dot = v >= 3 && v < 12;
	m.o = m.dot ? 3 + 3 * ((v - 3) / 3) : (v < 15 ? v : 0);
	m.r = m.dot ? 3 + (v - 3) % 3 : (v < 3 ? v : (v >= 12 && v < 15 ? v - 12 : 0));
	m.word = v < 3 ? (v == 0 ? 12 : 13) : (v < 12 ? v : v - 12);
	return m;
}

// A read of another cell's particle data during a pass.  In the
// dependency-driven sweep (DD: the passes of a sweep in one launch, each cell
// starting once its neighbours of earlier passes are done) it is an
// agent-scope load, served where the writes of every XCD meet, so that no
// XCD's L2 can return a copy older than the neighbour's finished pass.
template <bool DD>
__device__ __forceinline__ double nbld(const double *p) {
	if constexpr(DD) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	else return *p;
}

// Wait (DD) until every non-empty neighbour cell that an earlier pass of this
// sweep works on has published `mark` in done[]: lane nb < 26 of the team
// watches the neighbour in direction m = nb < 13 ? nb : nb + 1 (offsets m / 9 -
// 1, (m / 3) % 3 - 1, m % 3 - 1).  Neighbours of later passes wait for this
// cell in turn, so none of them writes before this cell's reads.  The wait is
// bounded: past DD_SPIN_MAX polls the team reports ERR_DEPWAIT and goes on, so
// the launch always drains.
template <int T>
__device__ __forceinline__ void wait_neighbours(const DevState &d, const Rep &rp, int pass, int ix, int iy, int iz,
                                                unsigned mark, int lane) {
	bool need = false;
	const unsigned *w = nullptr;
	if(lane < 26) {
		const int n0 = rp.pg.n[0], n1 = rp.pg.n[1], n2 = rp.pg.n[2];
		const int m = lane < 13 ? lane : lane + 1;
		const int cx = wrapi(ix + m / 9 - 1, n0), cy = wrapi(iy + (m / 3) % 3 - 1, n1), cz = wrapi(iz + m % 3 - 1, n2);
		const int ncol = ((cx & 1) << 2) | ((cy & 1) << 1) | (cz & 1);
		int np = 0;
		while(np < 7 && (int) ((rp.col_perm >> (4 * np)) & 0xFu) != ncol) np++;
		const int c = rp.cell_off + (cx * n1 + cy) * n2 + cz;
		need = np < pass && d.start[c + 1] > d.start[c];
		w = d.done + c;
	}
	int spins = 0;
	while(team_any<T>(need)) {
		if(need) need = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != mark;
		if(++spins > DD_SPIN_MAX) {
			if(lane == 0) atomicOr(d.err, (int) ERR_DEPWAIT);
			break;
		}
		if(team_any<T>(need)) __builtin_amdgcn_s_sleep(1);
	}
	// no load of the neighbours' data moves above the wait
	__atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// One cell of a colour pass: entry gi of the pass's list of non-empty cells
// (all replicas), worked on by the T lanes of one team with its LDS block
// `blk`.  The cell's members make sequential trials.  Each lane keeps up to
// CPL of the cell's static neighbours (the 26 surrounding cells, fixed during
// the pass) in registers; a denser neighbourhood is handled T at a time from
// HBM.
//
// The static neighbours do not move during the pass: a member's bonds with
// them, and with the other members, are counted at the first trial that gets
// as far as its bonds, and kept as members move; later trials test only the
// new position.  The bond decision is symmetric to the bit.
//
// A trial is one dependent chain, and most wavefronts share their SIMD with
// at most one other, so its length sets the pass's time.  Hence the
// single-precision filter (F32Filter: about 150 VALU instructions per trial
// instead of 280 in FP64, half the registers, no LDS exchange of the new
// patches: the separation is rotated into each particle's body frame
// instead), the trial read one ahead, and the exact new state formed one
// value per lane on acceptance.  Measured, steps of 16 trials per cell: one
// system of N=32768 at rho 0.5 285 -> 207 us, 8 x 4096 427 -> 212 us (its 28
// candidates per cell also fit the second register slot now, where the FP64
// form read 1 in 4 cells' last neighbours from HBM at every trial), 256
// uneven replicas 4.15 -> 2.75 ms.
//
// DD: the pass is one of several in flight (k_pass_dd).  The cell's own
// loads and its trials come first; the team then waits for its neighbours of
// earlier passes, reads their data with agent-scope loads, and finally
// writes its members back with agent-scope stores, waits for them to
// complete, and publishes `mark` for its own cell.
//
// CAP < CELL_CAP (the small-cell pass): a cell of more than CAP members, or
// with more neighbours than its record lists, is not worked on here but
// listed for the general pass that follows.
template <int T, int CPL, bool ONE, bool DD, int CAP = CELL_CAP>
__device__ __forceinline__ void pass_cell(const DevState &d, uint64_t sweep, int pass, int gi, int lane, double *blk,
                                          unsigned mark) {
	using L = TeamLds<CAP>;
	static_assert(T == 16 || T == 32 || T == 64, "teams of 16, 32 or 64 lanes");
	float *shadow = (float *) (blk + L::SH);
	float *ftrial = (float *) (blk + L::FT);
	double *own = blk + L::OWN;
	double *trials = blk + L::TR;
	double *geo = blk + L::GEO;
	int *own_pid = (int *) (blk + L::PID);
	int *nb_tab = (int *) (blk + L::NB);

	// 1. the cell's record: its header, and this lane's neighbour; a record of
	// another sweep lies past the end of the pass's list.
	// One replica (ONE): few wavefronts, which wait for memory during 60 % of a
	// pass when cells make one trial per member.  Everything is then read at
	// once and pinned here: the compiler would move all but the tag behind the
	// check, one more round trip (N=32768: 11.6 -> 11.3 us; N=65536 at rho 0.3
	// with 16 lanes 12.8 -> 12.0).  A batch's many wavefronts hide that round
	// trip, and pay for the second slots' line and the idle lanes' loads (16 x
	// 131072 at rho 0.05: 830 -> 869 us).
	const int *rec = d.rec + ((size_t) pass * d.total_act + gi) * REC_W;
	int4 h0 = ((const int4 *) rec)[0], h1 = ((const int4 *) rec)[1], h2 = ((const int4 *) rec)[2];
	int e0, e1 = 0;
	if constexpr(ONE) {
		e0 = rec[REC_HEAD + min(lane, REC_SLOTS - 1)];
		if constexpr(CPL > 1) e1 = rec[REC_HEAD + min(T + lane, REC_SLOTS - 1)];
		// (not volatile: the scalar loads below stay scalar; the second
		// statement brings the lines of the replica's constants into the
		// scalar cache)
		const Rep &rq = d.reps[0];
		asm("" : "+v"(h0.x) : "v"(h0.y), "v"(h0.z), "v"(h0.w), "v"(h1.x), "v"(h1.y), "v"(h1.z), "v"(h2.x), "v"(h2.y), "v"(h2.z), "v"(e0), "v"(e1));
		asm("" : "+v"(h0.x) : "s"(rq.T), "s"(rq.pg.box[0]), "s"(rq.pg.shift[2]), "s"(rq.pg.inv_side[0]), "s"(rq.pg.thr[0]),
		             "s"(rq.pg.thr[ACC_TAB - 2]));
	}
	else e0 = lane < REC_SLOTS ? rec[REC_HEAD + lane] : -1;
	if(uni<T>(h0.x) != (int) d.rec_tag) return;
	const int M = uni<T>(h0.y);
	const int s0 = uni<T>(h0.z);
	const int cnt = uni<T>(h0.w);
	const int cloc = uni<T>(h1.x);
	const int r = ONE ? 0 : uni<T>(h1.y);
	const int sel = uni<T>(h1.z);
	const int ix = uni<T>(h2.x), iy = uni<T>(h2.y), iz = uni<T>(h2.z);
	if constexpr(CAP < CELL_CAP)
		if(cnt > d.small_cap || M > REC_SLOTS) {
			// (entries < total_act: each cell is listed at most once a pass)
			if(lane == 0) d.ovf[atomicAdd(d.ovf_n + pass, 1)] = gi;
			return;
		}
	// (a team of T < CELL_CAP lanes holds one member per lane)
	if(cnt > CELL_CAP || cnt > T) {
		if(lane == 0) {
			atomicOr(d.err, (int) ERR_CELL_CAP);
			// (DD) the neighbours of later passes do not wait for it
			if constexpr(DD)
				__hip_atomic_store(d.done + d.reps[r].cell_off + cloc, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		return;
	}
	const Rep &rp = d.reps[r];
	double *F = pick_buf(d.f, sel);
	int *PID = pick_buf(d.pid, sel);

	// 2. every load of the cell at once: the members, the static neighbours
	// and the replica's geometry.  Register slot u (u < CPL) of lane l holds
	// one neighbour: the last cnt lanes' first slot the cell's members (read
	// from the shadow records at every trial), the slots before them and the
	// second ones the static neighbours (l, and T - cnt + l); the rest (dense
	// neighbourhoods only) are read again at every trial.  A lane thus tests
	// one neighbour per trial whether the cell holds one member or several.
	const int nstat = T - cnt;        // first slots of static neighbours
	const int mi = lane - nstat;      // this lane's member
	const bool is_mem = mi >= 0;
	const int nreg = min(M, min(T * CPL - cnt, REC_SLOTS));
	int cq[CPL];
	cq[0] = is_mem || lane >= nreg ? -1 : e0;
	// (ONE finds the second slots' entries among the lanes, when it needs them)
	if constexpr(CPL > 1) cq[1] = !ONE && nstat + lane < nreg ? rec[REC_HEAD + nstat + lane] : -1;
	// the lane's member or first static neighbour, in one set of registers
	// (second slots follow once that one is converted).  ONE: lanes without one
	// read the first member, since a load under a condition would be waited for
	// at its end, before the trials are drawn.
	double pv[NCOMP];
	auto load_part = [&](int j) {
#pragma unroll
		for(int c = 0; c < NCOMP; c++) pv[c] = nbld<DD>(part(F, j) + c);
	};
	int my_pid = 0;
	if(ONE || is_mem) my_pid = PID[s0 + max(mi, 0)];
	if(ONE || is_mem || (!DD && cq[0] >= 0)) load_part(is_mem ? s0 + mi : (!DD && cq[0] >= 0 ? cq[0] : s0));
	// trials of the cell in this pass: one per member (a sweep is then N
	// attempts), or a fixed number per non-empty cell
	const int ntrial = d.trials_per_cell > 0 ? d.trials_per_cell : cnt;
	const PassGeo &pg = rp.pg;
	const int col = ((ix & 1) << 2) | ((iy & 1) << 1) | (iz & 1);
	// the cell's centre
	const double ce0 = pg.shift[0] + ((double) ix + 0.5) * pg.side[0], ce1 = pg.shift[1] + ((double) iy + 0.5) * pg.side[1],
	             ce2 = pg.shift[2] + ((double) iz + 0.5) * pg.side[2];

	// 3. the cell's trials, one lane each (Philox: no memory traffic), and
	// the particle indices into LDS.  A trial keeps the largest rise in bonds
	// lost that its draw accepts: u < exp(-j/T) (MC.c:332) falls with j, and
	// for the 32-bit draw w it reads w <= thr[j - 1] exactly, so a trial
	// decides by comparing two integers.
	// One replica: where every cell of the wavefront makes few trials, four lanes
	// take each, whose blocks otherwise follow one another (k_pass at N=1000:
	// 6.84 -> 6.57 us; a batch gains nothing, its wavefronts overlap).
	const bool by_quads = ONE && ballot(ntrial * 4 > T) == 0ull;
	const int mt = by_quads ? lane >> 2 : lane;
	if(mt < ntrial) {
		double tv[TRIAL_W];
		const uint32_t draw = make_trial(d, rp, r, sweep, cloc, col, mt, cnt, by_quads, tv);
		int most = 0;
#pragma unroll
		for(int j = 0; j < ACC_TAB - 1; j++) most += (int) ((j < pg.n_thr) & (draw <= pg.thr[j]));
		const int k = (int) tv[0];
		double *w = trials + mt * TR_W;
		float *f = ftrial + mt * FT_W;
#pragma unroll
		for(int e = 0; e < TR_W; e++) w[e] = tv[1 + e];
		f[0] = f32_pos(tv[1]);
		f[1] = f32_pos(tv[2]);
		f[2] = f32_pos(tv[3]);
		f[3] = __int_as_float(most < ACC_TAB - 1 ? most : MOST_EXP);
#pragma unroll
		for(int e = 0; e < 9; e++) f[4 + e] = (float) tv[4 + e];
		f[13] = __int_as_float(k);
	}
	static_assert(MAX_TRIALS_PER_CELL <= 16 && CELL_CAP <= 32, "one lane per trial");
	const int koff = (threadIdx.x & 63) & ~(T - 1);
	// the team's lanes of a wavefront mask
	auto team_bits = [&](unsigned long long m) {
		if constexpr(T == 64) return m;
		else if constexpr(T == 32) return koff ? (unsigned) (m >> 32) : (unsigned) m;
		else return (unsigned) (m >> koff) & ((1u << T) - 1u);
	};
	auto team_has = [&](unsigned long long m) { return team_bits(m) != 0; };
	auto count_bits = [](auto m) {
		if constexpr(sizeof(m) == 8) return (int) __popcll(m);
		else return (int) __popc(m);
	};
	if(is_mem) own_pid[mi] = my_pid;
	if(lane == 0) {
		geo[0] = ce0;
		geo[1] = ce1;
		geo[2] = ce2;
	}
	team_sync();
	// 4. members into LDS ranked by particle index; a lane's slots become
	// single precision, relative to the cell's centre
	bool wild = false;  // beyond the filter's error bounds
	auto rel3 = [&](const double *p, double *q) {
		q[0] = kf_min_image(p[0] - ce0, pg.box[0], pg.inv_box[0]);
		q[1] = kf_min_image(p[1] - ce1, pg.box[1], pg.inv_box[1]);
		q[2] = kf_min_image(p[2] - ce2, pg.box[2], pg.inv_box[2]);
		// (a sum, which a NaN passes through)
		wild |= !(__builtin_fabs(p[0]) + __builtin_fabs(p[1]) + __builtin_fabs(p[2]) < F32_MAX_POS);
	};
	auto check_o = [&](const float *o) {
		wild |= !f32_orientation_ok(o);
	};
	float qx[CPL], qy[CPL], qz[CPL], qo[CPL][9];
	// pv in single precision, into slot u
	auto convert = [&](int u, double *rel) {
		rel3(pv, rel);
		qx[u] = f32_pos(rel[0]);
		qy[u] = f32_pos(rel[1]);
		qz[u] = f32_pos(rel[2]);
#pragma unroll
		for(int c = 0; c < 9; c++) qo[u][c] = (float) pv[3 + c];
		check_o(qo[u]);
	};
	auto empty_slot = [&](int u) {
		qx[u] = qy[u] = qz[u] = F32_FAR;
#pragma unroll
		for(int c = 0; c < 9; c++) qo[u][c] = 0.f;
	};
	empty_slot(0);
	if(is_mem || (!DD && cq[0] >= 0)) {
		double rel[3];
		convert(0, rel);
		if(is_mem) {
			int rank = 0;
			for(int m = 0; m < cnt; m++) rank += own_pid[m] < my_pid;
			double *w = own + rank * OWN_W;
			float *s = shadow + rank * SH_W;
#pragma unroll
			for(int c = 0; c < NCOMP; c++) w[c] = pv[c];
#pragma unroll
			for(int c = 0; c < 3; c++) w[12 + c] = rel[c];
			s[0] = qx[0];
			s[1] = qy[0];
			s[2] = qz[0];
#pragma unroll
			for(int c = 0; c < 9; c++) s[3 + c] = qo[0][c];
			s[12] = __int_as_float(-1);  // bonds not counted yet
		}
	}
	if constexpr(DD) {
		// the neighbours' data once their earlier passes are done
		wait_neighbours<T>(d, rp, pass, ix, iy, iz, mark, lane);
		if(cq[0] >= 0) {
			double rel[3];
			load_part(cq[0]);
			convert(0, rel);
		}
	}
	// whether any team of the wavefront uses the second slot of its lanes, or
	// has neighbours beyond the register slots (scalar branches)
	const bool wave_2 = CPL > 1 && ballot(nreg > nstat) != 0ull;
	const bool wave_far = ballot(M > nreg) != 0ull;
	if constexpr(CPL > 1)
		if(wave_2) {
			if constexpr(ONE) {
				// (entry nstat + lane of the record's list)
				const int from = koff + ((nstat + lane) & (T - 1));
				const int x0 = __shfl(e0, from), x1 = __shfl(e1, from);
				cq[1] = nstat + lane < nreg ? (nstat + lane < T ? x0 : x1) : -1;
			}
			empty_slot(1);
			if(cq[1] >= 0) {
				double rel[3];
				load_part(cq[1]);
				convert(1, rel);
			}
		}
	F32Filter fl = pg.filter;
	float margin = pg.margin;
	// (the in-cell test too: from about 10^10 on, the roundings of cell_coord
	// itself pass its margin)
	if(team_any<T>(wild)) fl.eps_d2 = fl.eps_t = margin = F32_ALL;
	const float is0 = pg.inv_side[0], is1 = pg.inv_side[1], is2 = pg.inv_side[2];
	if(CAP == CELL_CAP && wave_far && M > REC_SLOTS) {
		// the rows' ranges, for the neighbours past the record's list
		if(lane < 9) {
			int a1, b1, a2, b2;
			row_ranges(d.start + rp.cell_off, ix, iy, iz, pg.n[0], pg.n[1], pg.n[2], lane, a1, b1, a2, b2);
			nb_tab[2 * lane] = a1;
			nb_tab[2 * lane + 1] = a2;
			nb_tab[20 + 2 * lane] = b1 - a1;
			nb_tab[20 + 2 * lane + 1] = b2 - a2;
		}
		team_sync();
		if(lane == 0) {
			int acc = 0;
			for(int e = 0; e < 18; e++) {
				const int n = nb_tab[20 + e];
				nb_tab[20 + e] = acc;
				acc += n;
			}
			nb_tab[38] = acc;
		}
	}
	team_sync();

	auto hide = [](int v) { if constexpr(T == 64) return opaque_uniform(v); else return opaque(v); };
	auto hide_rep = [&]() { if constexpr(ONE) return opaque_uniform(0); else return hide(r); };
	// The exact arithmetic of one pair: member k moved by trial t (t < 0: as
	// it stands) and static slot q, or member m >= 0.  OVERLAP (of a moved
	// member: where pairs overlap as they stand, which only a refused upload
	// leaves behind, their bond counts as any other), BOND or 0.
	enum : unsigned { OVERLAP = 1, BOND = 2, UNSURE = 4 };
	auto exact_pair = [&](int k, int t, int q, int m) -> unsigned {
		k = opaque(k);
		q = opaque(q);
		m = opaque(m);
		const double *p = own + k * OWN_W, *pm = own + max(m, 0) * OWN_W, *dt = trials + t * TR_W;
		const Rep &hp = d.reps[hide_rep()];
		double w[3];
		// (the member's value is read in either case and kept, so that no
		// pointer is chosen between LDS and HBM)
		auto other = [&](int c) {
			double v = pm[c];
			asm volatile("" : "+v"(v));
			if(m < 0) v = nbld<DD>(part(F, q) + c);
			return v;
		};
#pragma unroll
		for(int c = 0; c < 3; c++)
			w[c] = kf_min_image(other(c) - (t >= 0 ? p[c] + dt[c] : p[c]), hp.pg.box[c], hp.pg.inv_box[c]);
		const double w2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2], cosmax = hp.cosmax;
		if(w2 < (t >= 0 ? 1. : 0.)) return OVERLAP;
		if(!(w2 < hp.rc2)) return 0u;
		kf_unit(w[0], w[1], w[2], w2);
		// (one row, then one patch at a time: this path sets the kernel's
		// register count otherwise)
		double O[9];
		if(t >= 0) {
			double R[9];
#pragma unroll
			for(int c = 0; c < 9; c++) R[c] = dt[3 + c];
#pragma unroll
			for(int i = 0; i < 3; i++) {
				const double a0 = p[3 + 3 * i], a1 = p[4 + 3 * i], a2 = p[5 + 3 * i];
#pragma unroll
				for(int j = 0; j < 3; j++) O[3 * i + j] = a0 * R[j] + a1 * R[3 + j] + a2 * R[6 + j];
				__builtin_amdgcn_sched_barrier(0);
			}
		}
		else
#pragma unroll
			for(int c = 0; c < 9; c++) O[c] = p[3 + c];
		bool hit = false;
#pragma unroll
		for(int i = 0; i < 4; i++) {
			double v[3];
#pragma unroll
			for(int e = 0; e < 3; e++)
				v[e] = O[3 * e] * kf_base(i, 0) + O[3 * e + 1] * kf_base(i, 1) + O[3 * e + 2] * kf_base(i, 2);
			hit |= kf_dot(w[0], w[1], w[2], v[0], v[1], v[2]) > cosmax;
			__builtin_amdgcn_sched_barrier(0);
		}
		if(!hit) return 0u;
#pragma unroll
		for(int c = 0; c < 9; c++) O[c] = other(3 + c);
		return kf_any_q(w[0], w[1], w[2], O, cosmax) ? BOND : 0u;
	};
	// slot of static neighbour i (0 <= i < M)
	auto nb_slot = [&](int i) {
		if(i < REC_SLOTS) return rec[REC_HEAD + i];
		int lo = 0, hi = 18;
		while(hi - lo > 1) {
			const int mid = (lo + hi) >> 1;
			if(nb_tab[20 + mid] <= i) lo = mid;
			else hi = mid;
		}
		return nb_tab[lo] + (i - nb_tab[20 + lo]);
	};
	const MoveShare ms = move_share(lane);
	int c_acc = 0, d_bonds = 0;
	int next_k = __float_as_int(ftrial[13]);

	// 5. the trials
	for(int t = 0; t < ntrial; t++) {
		// the moving member's record (its rank was read one trial ahead), the
		// trial, another member's record for a member lane, and the lane's
		// share of the exact move
		const int k = next_k;
		const float *s = shadow + k * SH_W, *f = ftrial + t * FT_W;
		float sv[14], tv[13];
#pragma unroll
		for(int c = 0; c < 14; c++) sv[c] = s[c];
#pragma unroll
		for(int e = 0; e < 13; e++) tv[e] = f[e];
		if(is_mem) {
			if(mi == k) qx[0] = F32_FAR;
			else {
				const float *so = shadow + mi * SH_W;
				qx[0] = so[0];
				qy[0] = so[1];
				qz[0] = so[2];
#pragma unroll
				for(int c = 0; c < 9; c++) qo[0][c] = so[3 + c];
			}
		}
		const double *dt = trials + t * TR_W;
		const double *me = own + k * OWN_W + ms.o, *tm = dt + ms.r;
		const double o0 = me[0], o1 = me[1], o2 = me[2];
		const double r0 = tm[0], r1 = tm[3], r2 = tm[6];
		next_k = __float_as_int(f[FT_W + 13]);  // (past the last trial: not used)
		const float nx = sv[0] + tv[0], ny = sv[1] + tv[1], nz = sv[2] + tv[2];

		// a trial that leaves the cell, or overlaps a neighbour, is rejected;
		// what single precision cannot tell stays for the exact arithmetic
		const float x = __builtin_fmaxf(__builtin_fabsf(nx) * is0, __builtin_fmaxf(__builtin_fabsf(ny) * is1,
		                                                                         __builtin_fabsf(nz) * is2));
		// (conditions are kept as lane masks in scalar registers)
		const unsigned long long m_close = ballot(!(__builtin_fabsf(x - 0.5f) > margin));
		unsigned long long m_rej = ballot(x > 0.5f) & ~m_close, m_unsure = m_close;
		// slots in use by the wavefront's teams (a scalar branch)
		auto each_slot = [&](auto &&f) {
			f(0);
			if constexpr(CPL > 1)
				if(wave_2) f(1);
		};
		float dx[CPL], dy[CPL], dz[CPL], d2[CPL];
		unsigned long long m_near[CPL] = {}, m_onear[CPL] = {}, m_bond[CPL] = {}, m_obond[CPL] = {};
		each_slot([&](int u) {
			dx[u] = qx[u] - nx;
			dy[u] = qy[u] - ny;
			dz[u] = qz[u] - nz;
			d2[u] = norm2(dx[u], dy[u], dz[u]);
			m_near[u] = ballot(f32_near(d2[u], fl));
			m_rej |= ballot(d2[u] < 1.f) & ~m_near[u];
		});
		if(team_has(m_rej)) continue;

		// bonds at the new position: O'^T d = R^T (O^T d)
		each_slot([&](int u) {
			const unsigned long long m_in = ballot(d2[u] < fl.rc2);
			if(m_in != 0ull) {
				float a0, a1, a2, e0, e1, e2;
				bool yes, unsure;
				mul_t(sv + 3, dx[u], dy[u], dz[u], a0, a1, a2);
				mul_t(tv + 4, a0, a1, a2, e0, e1, e2);
				f32_bond(e0, e1, e2, dx[u], dy[u], dz[u], d2[u], qo[u], fl, yes, unsure);
				m_bond[u] = ballot(yes) & m_in & ~m_near[u];
				m_near[u] |= ballot(unsure) & m_in;
			}
			m_unsure |= m_near[u];
		});
		// the bonds at the present position, when not yet counted
		int s_old = __float_as_int(sv[12]);
		unsigned mb_old = __float_as_uint(sv[13]);
		const bool first = s_old < 0;
		const bool wave_first = ballot(first) != 0ull;
		if(wave_first)
			each_slot([&](int u) {
				const float ex = qx[u] - sv[0], ey = qy[u] - sv[1], ez = qz[u] - sv[2];
				const float e2 = norm2(ex, ey, ez);
				const unsigned long long m_in = ballot(e2 < fl.rc2);
				m_onear[u] = ballot(f32_near(e2, fl));
				if(m_in != 0ull) {
					float a0, a1, a2;
					bool yes, unsure;
					mul_t(sv + 3, ex, ey, ez, a0, a1, a2);
					f32_bond(a0, a1, a2, ex, ey, ez, e2, qo[u], fl, yes, unsure);
					m_obond[u] = ballot(yes) & m_in & ~m_onear[u];
					m_onear[u] |= ballot(unsure) & m_in;
				}
				m_unsure |= m_onear[u];
			});
		bool late = false;  // a rejection found by the exact arithmetic
		if(__builtin_expect(m_unsure != 0ull, 0)) {
			if(__builtin_amdgcn_inverse_ballot_w64(m_close)) {
				const Grid &G = d.reps[hide_rep()].g;
				const int at[3] = {ix, iy, iz};
#pragma unroll 1
				for(int a = 0; a < 3; a++)
					late |= cell_coord(own[k * OWN_W + a] + dt[a], G.shift[a], G.inv_box[a], G.n[a]) != at[a];
			}
#pragma unroll 1
			for(int v = 0; v < 2; v++)
#pragma unroll
				for(int u = 0; u < CPL; u++) {
					unsigned e = 0;
					if(__builtin_amdgcn_inverse_ballot_w64(v ? m_near[u] : m_onear[u]))
						e = exact_pair(k, v ? t : -1, cq[u], u == 0 && is_mem ? mi : -1);
					const unsigned long long m = ballot(e == BOND);
					if(v) m_bond[u] |= m;
					else m_obond[u] |= m;
					late |= v && e == OVERLAP;
				}
			late = team_any<T>(late);
		}
		// the counts: all bonds, and the members' as bits
		auto member_bits = [&](auto bits) { return (unsigned) (bits >> nstat); };
		int n_new = 0;
		unsigned mb = 0;
		each_slot([&](int u) {
			const auto bits = team_bits(m_bond[u]);
			n_new += count_bits(bits);
			if(u == 0) mb = member_bits(bits);
		});
		if(wave_first) {
			int n = 0;
			unsigned mo = 0;
			each_slot([&](int u) {
				const auto bits = team_bits(m_obond[u]);
				n += count_bits(bits);
				if(u == 0) mo = member_bits(bits);
			});
			mb_old = first ? mo : mb_old;
			s_old = first ? n - (int) __popc(mo) : s_old;
		}
		if(wave_far) {
			// the static neighbours beyond the register slots, from HBM
			int n = 0;  // bonds at the new position, and << 16 at the present one
			bool ov = false;
			for(int i = lane + nreg; i < M; i += T) {
				const int q = opaque(nb_slot(i));
				const Rep &hp = d.reps[hide_rep()];
				float rel[3], Oq[9];
				wild = false;
#pragma unroll
				for(int c = 0; c < 3; c++) {
					const double p = nbld<DD>(part(F, q) + c);
					rel[c] = (float) kf_min_image(p - geo[c], hp.pg.box[c], hp.pg.inv_box[c]);
					wild |= !(__builtin_fabs(p) < F32_MAX_POS);
				}
				const float fx = rel[0], fy = rel[1], fz = rel[2];
				const float reach = fl.rc2 + fl.eps_d2;
				const float gn2 = norm2(fx - nx, fy - ny, fz - nz), go2 = norm2(fx - sv[0], fy - sv[1], fz - sv[2]);
				if(!wild && !(gn2 < reach) && !(first && go2 < reach)) continue;
#pragma unroll
				for(int c = 0; c < 9; c++) Oq[c] = (float) nbld<DD>(part(F, q) + 3 + c);
				check_o(Oq);
#pragma unroll 1
				for(int v = first ? 0 : 1; v < 2; v++) {
					const float gx = fx - (v ? nx : sv[0]), gy = fy - (v ? ny : sv[1]), gz = fz - (v ? nz : sv[2]);
					const float g2 = v ? gn2 : go2;
					unsigned bf = v && g2 < 1.f ? (unsigned) OVERLAP : 0u;
					if(wild || f32_near(g2, fl)) bf = UNSURE;
					else if(bf == 0u && g2 < fl.rc2) {
						float a0, a1, a2, e0, e1, e2;
						mul_t(sv + 3, gx, gy, gz, a0, a1, a2);
						mul_t(tv + 4, a0, a1, a2, e0, e1, e2);
						bool is, maybe;
						f32_bond(v ? e0 : a0, v ? e1 : a1, v ? e2 : a2, gx, gy, gz, g2, Oq, fl, is, maybe);
						bf = maybe ? (unsigned) UNSURE : (is ? (unsigned) BOND : 0u);
					}
					if(bf == UNSURE) bf = exact_pair(k, v ? t : -1, q, -1);
					ov |= v && bf == OVERLAP;
					n += bf == BOND ? (v ? 1 : 1 << 16) : 0;
				}
			}
			late |= team_any<T>(ov);
			n = team_sum<T>(n);
			n_new += n & 0xffff;
			if(first) s_old += n >> 16;
		}
		const int db = n_new - (s_old + (int) __popc(mb_old));
		// MC.c:332: accept if dE <= 0 or a uniform draw u < exp(-dE/T), with
		// dE = -db an integer: the trial holds the largest rise it accepts
		// (MOST_EXP: at least ACC_TAB - 1, beyond which the factor is formed)
		bool acc = -db <= __float_as_int(tv[3]) && !late;
		if(acc && -db >= ACC_TAB) {
			const u32x4 rb = rng(d.seed, r, sweep, (uint32_t) hide(cloc), TAG_TRIAL_B, (uint32_t) col, (uint32_t) t);
			acc = u01(rb.w) < exp((double) db / d.reps[hide_rep()].T);
		}
		if(acc) {
			c_acc++;
			d_bonds += db;
			// the new state, one value per lane, exact and single precision;
			// lanes 0 to 2 write the new static count and member bits
			const double rv = ms.dot ? o0 * r0 + o1 * r1 + o2 * r2 : o0 + r0;
			const float rf = f32_pos(rv);
			if(lane < 15) {
				own[k * OWN_W + lane] = rv;
				shadow[k * SH_W + ms.word] =
				    lane == 0 ? __int_as_float(n_new - (int) __popc(mb)) : (lane <= 2 ? __uint_as_float(mb) : rf);
			}
			// the other members' bits for member k
			if(is_mem && mi != k) {
				unsigned *w = (unsigned *) (shadow + mi * SH_W + 13);
				*w = (*w & ~(1u << k)) | (((mb >> mi) & 1u) << k);
			}
		}
		else if(first && lane < 2)
			shadow[k * SH_W + 12 + lane] = lane == 0 ? __int_as_float(s_old) : __uint_as_float(mb_old);
		team_sync();
	}
	// 6. write the members back, ranked (the ranking permutes the cell's slots)
	if(c_acc > 0 || cnt > 1) {
		const int at = hide(s0);
		for(int e = lane; e < cnt * NCOMP; e += T) {
			int m = e / NCOMP, c = e - m * NCOMP;
			if constexpr(DD)
				__hip_atomic_store(part(F, at + m) + c, own[m * OWN_W + c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			else part(F, at + m)[c] = own[m * OWN_W + c];
		}
		if(is_mem) {
			int rank = 0;
			for(int m = 0; m < cnt; m++) rank += own_pid[m] < my_pid;
			PID[at + rank] = my_pid;
		}
	}
	if constexpr(DD) {
		// the members' stores have completed (the wavefront's memory
		// counter is zero) before the cell is published as done
		__atomic_signal_fence(__ATOMIC_SEQ_CST);
		__builtin_amdgcn_s_waitcnt(0);
		__atomic_signal_fence(__ATOMIC_SEQ_CST);
		if(lane == 0) __hip_atomic_store(d.done + rp.cell_off + cloc, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	if(lane == 0) {
		const int slot = gi & (NSLOT - 1);
		atomicAdd(ctr_at(d.ctr, r, C_TRY_ROTO, slot), (unsigned long long) ntrial);
		if(c_acc) {
			atomicAdd(ctr_at(d.ctr, r, C_ACC_ROTO, slot), (unsigned long long) c_acc);
			atomicAdd(ctr_at(d.ctr, r, C_DBONDS, slot), (unsigned long long) (long long) d_bonds);
		}
	}
}

// One colour pass per launch, one list entry per team.  The grid is sized
// for the largest list; teams past the end of the list find a record of
// another sweep and leave (reading the list's length first cost a dependent
// load in every workgroup).  Workgroups reach the 8 XCDs round-robin, and the
// list is in cell order, so each XCD takes runs of XCD_RUN workgroups:
// neighbouring cells, whose shared neighbours its L2 then serves.
constexpr int XCD_RUN = 16;

template <int T, int CPL, bool ONE, int CAP = CELL_CAP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pass(PassArgs a) {
	extern __shared__ double lds[];
	const int lane = threadIdx.x & (T - 1);
	const int team = threadIdx.x / T;
	const int i = blockIdx.x >> 3;
	const int blk = (i / XCD_RUN * 8 + (int) (blockIdx.x & 7)) * XCD_RUN + i % XCD_RUN;
	const int gi = uni<T>(blk * (int) (blockDim.x / T) + team);
	if(gi >= a.d.total_act) return;
	pass_cell<T, CPL, ONE, false, CAP>(a.d, a.sweep, a.pass, gi, lane, lds + team * team_lds<CAP>(), 0u);
}

// The cells the small-cell pass deferred (more than SMALL_CAP members), by
// the general 32-lane form: teams take the listed entries in turn.
template <bool ONE>
__global__ __launch_bounds__(128) void k_pass_ovf(PassArgs a) {
	extern __shared__ double lds[];
	constexpr int T = 32;
	const int lane = threadIdx.x & (T - 1);
	const int team = threadIdx.x / T;
	const int tpb = blockDim.x / T;
	const int n = a.d.ovf_n[a.pass];
	for(int e = blockIdx.x * tpb + team; e < n; e += gridDim.x * tpb)
		pass_cell<T, 2, ONE, false>(a.d, a.sweep, a.pass, a.d.ovf[e], lane, lds + team * team_lds<>(), 0u);
}

// The 8 colour passes of a sweep in one launch, driven by dependencies
// instead of kernel boundaries.  The sweep's work is one queue of tickets:
// the list of pass 0, then pass 1, ..., each padded to whole wavefronts so
// that the teams of one wavefront always work on one pass.  Each wavefront
// takes the next tickets when it starts; each team then runs its cell as the
// per-pass kernel does, after waiting for its neighbours of earlier passes
// (wait_neighbours), and publishes its own cell.  A cell's neighbours of
// earlier passes hold earlier tickets, taken by wavefronts that started
// before it and are running or done, so the work always progresses whatever
// is resident; the waits are bounded besides.  The grid covers the largest
// possible lists; wavefronts whose tickets lie past the sweep's end leave at
// once.  Results equal the per-pass launches' bit for bit: each cell sees its
// neighbourhood as the earlier passes left it, and its trials do not depend
// on timing.
template <int T, bool ONE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pass_dd(PassArgs a) {
	extern __shared__ double lds[];
	const DevState &d = a.d;
	constexpr int TPW = 64 / T;  // teams per wavefront
	const int lane = threadIdx.x & (T - 1);
	const int team = threadIdx.x / T;
	int t0 = 0;
	if((threadIdx.x & 63) == 0) t0 = atomicAdd(d.ddq, TPW);
	const int t = __builtin_amdgcn_readfirstlane(t0) + (threadIdx.x & 63) / T;
	int p = 0, base = 0, n = 0;
	for(; p < 8; p++) {
		n = d.pfx[p * (d.R + 1) + d.R];
		const int padded = (n + TPW - 1) / TPW * TPW;
		if(t < base + padded) break;
		base += padded;
	}
	if(p == 8 || t - base >= n) return;
	pass_cell<T, T < 64 ? 2 : 1, ONE, true>(d, a.sweep, p, t - base, lane, lds + team * team_lds<>(), a.mark);
}

// Grid-wide barrier of a cooperative launch (every workgroup resident).
// Arrivals count up in bar[0]; the last one resets it and advances the
// generation bar[1], which the others wait for.  The agent-scope fences
// publish each workgroup's writes before its arrival and make the others'
// visible after the wait.  The wait is bounded: past BAR_SPIN_MAX polls the
// workgroup reports ERR_BARRIER and goes on, so the grid always drains.
__device__ __forceinline__ void grid_barrier(unsigned *bar, int *err) {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
	__syncthreads();
	if(threadIdx.x == 0) {
		const unsigned gen = __hip_atomic_load(&bar[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		const unsigned arrived = __hip_atomic_fetch_add(&bar[0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
		if(arrived == gridDim.x - 1) {
			__hip_atomic_store(&bar[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			__hip_atomic_store(&bar[1], gen + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
		}
		else {
			int spins = 0;
			while(__hip_atomic_load(&bar[1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) == gen) {
				if(++spins > BAR_SPIN_MAX) {
					atomicOr(err, (int) ERR_BARRIER);
					break;
				}
				__builtin_amdgcn_s_sleep(2);
			}
		}
	}
	__syncthreads();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// The 8 colour passes of a sweep in one cooperative launch, separated by
// grid barriers.  Team g takes list entries g, g + teams, ... of each pass.
template <int T>
__global__ __launch_bounds__(256) void k_sweep_passes(PassArgs a) {
	extern __shared__ double lds[];
	const DevState &d = a.d;
	const int lane = threadIdx.x & (T - 1);
	const int team = threadIdx.x / T;
	const int tpb = blockDim.x / T;
	const int nteams = gridDim.x * tpb;
	const int g0 = uni<T>(blockIdx.x * tpb + team);
	double *own = lds + team * team_lds<>();
	for(int k = 0; k < 8; k++) {
		const int total = uni<T>(d.pfx[k * (d.R + 1) + d.R]);
		for(int gi = g0; gi < total; gi += nteams) pass_cell<T, T < 64 ? 2 : 1, false, false>(d, a.sweep, k, gi, lane, own, 0u);
		if(k < 7) grid_barrier(d.bar, d.err);
	}
}

template <int T, bool ONE>
static void pass_dd_T(const DevState &d, uint64_t sweep, unsigned mark, int block, hipStream_t s) {
	const int tpb = block / T;
	// every pass's largest list, one team per entry (wavefronts past the
	// sweep's tickets leave at once)
	const unsigned nb = (unsigned) std::max(1, 8 * ((d.total_act + tpb - 1) / tpb));
	PassArgs a{d, sweep, 0, mark};
	hipLaunchKernelGGL((k_pass_dd<T, ONE>), dim3(nb), dim3(block), pass_lds_bytes(T, block), s, a);
}

void launch_passes_dd(const DevState &d, uint64_t sweep, unsigned mark, int T, int block, hipStream_t s) {
	if(T == 32) {
		if(d.R == 1) pass_dd_T<32, true>(d, sweep, mark, block, s);
		else pass_dd_T<32, false>(d, sweep, mark, block, s);
	}
	else {
		if(d.R == 1) pass_dd_T<64, true>(d, sweep, mark, block, s);
		else pass_dd_T<64, false>(d, sweep, mark, block, s);
	}
}

template <int T, int CPL, bool ONE, int CAP = CELL_CAP>
static void pass_T(const DevState &d, uint64_t sweep, int pass, int block, hipStream_t s) {
	const int tpb = block / T;
	int nb = (d.total_act + tpb - 1) / tpb;
	nb = (nb + 8 * XCD_RUN - 1) / (8 * XCD_RUN) * (8 * XCD_RUN);  // whole runs on each XCD
	size_t lds = (size_t) tpb * team_lds<CAP>() * sizeof(double);
	PassArgs a{d, sweep, pass, 0u};
	hipLaunchKernelGGL((k_pass<T, CPL, ONE, CAP>), dim3(nb), dim3(block), lds, s, a);
	if constexpr(CAP < CELL_CAP) {
		// the deferred cells (usually none: the workgroups leave at once)
		constexpr int OB = 128;
		hipLaunchKernelGGL((k_pass_ovf<ONE>), dim3(256), dim3(OB), pass_lds_bytes(32, OB), s, a);
	}
}

int small_cell_cap() { return SMALL_CAP; }

size_t pass_lds_bytes(int T, int block) { return (size_t) (block / T) * team_lds<>() * sizeof(double); }

// The form is chosen per context: 16, 32 or 64 lanes per cell, and one
// replica (its constants then load to scalar registers for every team) or
// several.
template <int T>
static void pass_TK(const DevState &d, uint64_t sweep, int pass, int block, hipStream_t s) {
	if constexpr(T == 16) {
		// at most one particle per cell on average: cells that the small-cell
		// pass defers are rare
		if(d.Ntot <= d.C_total) {
			if(d.R == 1) pass_T<16, 2, true, SMALL_CAP>(d, sweep, pass, block, s);
			else pass_T<16, 2, false, SMALL_CAP>(d, sweep, pass, block, s);
			return;
		}
	}
	constexpr int CPL = T < 64 ? 2 : 1;  // register neighbours per lane
	if(d.R == 1) pass_T<T, CPL, true>(d, sweep, pass, block, s);
	else pass_T<T, CPL, false>(d, sweep, pass, block, s);
}

void launch_pass(const DevState &d, uint64_t sweep, int pass, int T, int block, hipStream_t s) {
	if(T == 16) pass_TK<16>(d, sweep, pass, block, s);
	else if(T == 32) pass_TK<32>(d, sweep, pass, block, s);
	else pass_TK<64>(d, sweep, pass, block, s);
}

static const void *sweep_kernel(int T) {
	return T == 32 ? (const void *) k_sweep_passes<32> : (const void *) k_sweep_passes<64>;
}

// co-resident workgroups of the cooperative launch
int sweep_blocks_max(int T, int block, int cus) {
	int per_cu = 0;
	if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, sweep_kernel(T), block, pass_lds_bytes(T, block)) != hipSuccess)
		return 0;
	return per_cu * cus;
}

hipError_t launch_sweep_passes(const DevState &d, uint64_t sweep, int T, int block, int blocks, hipStream_t s) {
	PassArgs a{d, sweep, 0, 0u};
	void *args[] = {&a};
	return hipLaunchCooperativeKernel(sweep_kernel(T), dim3(blocks), dim3(block), args, (unsigned) pass_lds_bytes(T, block), s);
}

// ------------------------------------------------------------------------
// energy: one team per slot, MC_energy semantics (MC.c:272-309): bonds of
// the particle with every neighbour, 0 and an overlap flag on any overlap.

template <int T>
struct NbLayout {
	static constexpr int S = (T >= 54) ? 2 : 1;
	static constexpr int STEP = T / S;
	static constexpr int PER = (27 + STEP - 1) / STEP;
};

// trial = 1: the energy of the replicas' box trials.  A trial that rebuilt
// its lists reads the spare buffer on the trial grid; a fast trial reads the
// current buffer through the current lists (membership by the list grid,
// computed from the unscaled positions exactly as the lists were built) and
// scales every position as the trial does before it measures separations.
// Once one team of a trial has met an overlap the trial is rejected
// whatever the bonds are: the replica's later teams stop at once.
// Workgroups reach the XCDs round-robin: each XCD takes a contiguous range of
// slots (neighbouring cells share its L2).
template <int T>
__global__ __launch_bounds__(256) void k_energy(DevState d, int trial, int per_particle) {
	using NB = NbLayout<T>;
	const int lane = threadIdx.x & (T - 1);
	const int team = threadIdx.x / T;
	const int j = xcd_remap(blockIdx.x, gridDim.x) * (blockDim.x / T) + team;
	if(j >= d.Ntot) return;
	const int r = d.prep[j];
	const Rep &rp = d.reps[r];
	if(j - rp.p_off >= rp.np) return;  // a free slot (the live particles come first after a rebuild)
	const bool tr = trial && rp.trial_active;
	if(trial && !tr) return;
	if(tr && (rp.trial_rec || rp.trial_pl)) return;  // k_energy_rec / k_energy_pairs take this trial
	if(tr && __hip_atomic_load(&d.vflag[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
	const bool fast = tr && rp.trial_fast;
	const Grid &G = tr ? (fast ? rp.lg : rp.tg) : rp.g;  // the grid of the lists' membership
	const Grid &B = tr ? rp.tg : rp.g;                    // the box of the separations
	const double s0 = fast ? rp.trial_s[0] : 1., s1 = fast ? rp.trial_s[1] : 1., s2 = fast ? rp.trial_s[2] : 1.;
	const int b = (tr && !fast) ? (rp.sel ^ 1) : rp.sel;
	const double *F = pick_buf(d.f, b);
	const double ux = part(F, j)[0], uy = part(F, j)[1], uz = part(F, j)[2];
	double O[9];
#pragma unroll
	for(int c = 0; c < 9; c++) O[c] = part(F, j)[3 + c];
	double P[4][3];
	kf_patches(O, P);
	const int n0 = G.n[0], n1 = G.n[1], n2 = G.n[2];
	const int ix = cell_coord(ux, G.shift[0], G.inv_box[0], n0);
	const int iy = cell_coord(uy, G.shift[1], G.inv_box[1], n1);
	const int iz = cell_coord(uz, G.shift[2], G.inv_box[2], n2);
	// (x * 1 is x: unscaled replicas are unchanged)
	const double px = ux * s0, py = uy * s1, pz = uz * s2;
	const double Lx = B.box[0], Ly = B.box[1], Lz = B.box[2];
	const double iLx = B.inv_box[0], iLy = B.inv_box[1], iLz = B.inv_box[2];
	const double c2 = rp.cosmax >= KF_FILTER_MIN_COS ? rp.cosmax * rp.cosmax : -1.;
	int nbond = 0;
	bool ov = false;
#pragma unroll
	for(int u = 0; u < NB::PER; u++) {
		int nb = lane / NB::S + u * NB::STEP;
		if(nb >= 27) continue;
		int cx = wrapi(ix + nb / 9 - 1, n0), cy = wrapi(iy + (nb / 3) % 3 - 1, n1), cz = wrapi(iz + nb % 3 - 1, n2);
		int cc = rp.cell_off + (cx * n1 + cy) * n2 + cz;
		int s = d.start[cc], e = d.start[cc + 1];
		for(int q = s + lane % NB::S; q < e; q += NB::S) {
			if(q == j) continue;
			double dx = kf_min_image(part(F, q)[0] * s0 - px, Lx, iLx);
			double dy = kf_min_image(part(F, q)[1] * s1 - py, Ly, iLy);
			double dz = kf_min_image(part(F, q)[2] * s2 - pz, Lz, iLz);
			double d2 = dx * dx + dy * dy + dz * dz;
			if(d2 < 1.) ov = true;
			else if(d2 < rp.rc2)
				nbond += (int) pair_bonded(dx, dy, dz, d2, &P[0][0], c2, rp.cosmax, [&](double *Oq) {
#pragma unroll
					for(int c = 0; c < 9; c++) Oq[c] = part(F, q)[3 + c];
				});
		}
	}
	nbond = team_sum<T>(nbond);
	const bool any = team_any<T>(ov);
	if(lane == 0) {
		if(tr && any) __hip_atomic_store(&d.vflag[r], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		int res = any ? 0 : nbond;
		if(per_particle) {
			int i = rp.p_off + pick_buf(d.pid, b)[j];
			d.out_bonds[i] = res;
			d.out_ovl[i] = any ? 1 : 0;
		}
		int slot = j & (NSLOT - 1);
		if(res) atomicAdd(ctr_at(d.ctr, r, C_EBONDS, slot), (unsigned long long) res);
		if(any) atomicAdd(ctr_at(d.ctr, r, C_OVL, slot), 1ull);
	}
}

// Bonded partners of every particle (the pairs output_print_bonds lists,
// output.c:213-268, with MC_interact's test): slot j's partners' particle
// indices at partners[(p_off + pid) * max_per + k], k < max_per, and their
// number at count[p_off + pid] (which may exceed max_per).  One thread per
// slot; an output path, not a hot one.
__global__ void k_bond_list(DevState d, int max_per, int *count, int *partners) {
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if(j >= d.Ntot) return;
	const int r = d.prep[j];
	const Rep &rp = d.reps[r];
	if(j - rp.p_off >= rp.np) return;
	const Grid &G = rp.g;
	const double *F = pick_buf(d.f, rp.sel);
	const int *PID = pick_buf(d.pid, rp.sel);
	const double px = part(F, j)[0], py = part(F, j)[1], pz = part(F, j)[2];
	double O[9];
	for(int c = 0; c < 9; c++) O[c] = part(F, j)[3 + c];
	double P[4][3];
	kf_patches(O, P);
	const int n0 = G.n[0], n1 = G.n[1], n2 = G.n[2];
	const int ix = cell_coord(px, G.shift[0], G.inv_box[0], n0);
	const int iy = cell_coord(py, G.shift[1], G.inv_box[1], n1);
	const int iz = cell_coord(pz, G.shift[2], G.inv_box[2], n2);
	const size_t me = (size_t) rp.p_off + PID[j];
	int nb = 0;
	for(int c = 0; c < 27; c++) {
		const int cx = wrapi(ix + c / 9 - 1, n0), cy = wrapi(iy + (c / 3) % 3 - 1, n1), cz = wrapi(iz + c % 3 - 1, n2);
		const int cc = rp.cell_off + (cx * n1 + cy) * n2 + cz;
		for(int q = d.start[cc]; q < d.start[cc + 1]; q++) {
			if(q == j) continue;
			double dx = kf_min_image(part(F, q)[0] - px, G.box[0], G.inv_box[0]);
			double dy = kf_min_image(part(F, q)[1] - py, G.box[1], G.inv_box[1]);
			double dz = kf_min_image(part(F, q)[2] - pz, G.box[2], G.inv_box[2]);
			const double d2 = dx * dx + dy * dy + dz * dz;
			if(d2 < 1. || !(d2 < rp.rc2)) continue;
			kf_unit(dx, dy, dz, d2);
			if(!kf_any_p(dx, dy, dz, &P[0][0], rp.cosmax)) continue;
			double Oq[9];
			for(int e = 0; e < 9; e++) Oq[e] = part(F, q)[3 + e];
			if(!kf_any_q(dx, dy, dz, Oq, rp.cosmax)) continue;
			if(nb < max_per) partners[me * max_per + nb] = PID[q];
			nb++;
		}
	}
	count[me] = nb;
}

void launch_bond_list(const DevState &d, int max_per, int *count, int *partners, hipStream_t s) {
	if(d.Ntot > 0)
		hipLaunchKernelGGL(k_bond_list, dim3((d.Ntot + 255) / 256), dim3(256), 0, s, d, max_per, count, partners);
}

void launch_energy_rows_zero(const DevState &d, hipStream_t s) {
	hipLaunchKernelGGL(k_zero_energy_rows, dim3((d.R * 2 * NSLOT + 255) / 256), dim3(256), 0, s, d.ctr, d.R);
}

// Lanes per particle: 32 where the 27 cells hold many candidates, 8 in dilute
// systems (fewer than 8 candidates on average over the cell capacity), where
// most of a 32-lane team would idle.  The result does not depend on it.
void launch_energy(const DevState &d, int trial, int per_particle, hipStream_t s) {
	launch_energy_rows_zero(d, s);
	if(d.Ntot <= 0) return;
	const int block = 256;
	const double cand = 27. * (double) d.Ntot / (double) (d.C_total > 0 ? d.C_total : 1);
	// a multiple of 8 workgroups: one contiguous range of slots per XCD
	auto grid = [&](int per) { return dim3((unsigned) ((((long long) d.Ntot + per - 1) / per + 7) & ~7LL)); };
	if(cand < 8.) hipLaunchKernelGGL(k_energy<8>, grid(block / 8), dim3(block), 0, s, d, trial, per_particle);
	else hipLaunchKernelGGL(k_energy<32>, grid(block / 32), dim3(block), 0, s, d, trial, per_particle);
}

// The pair of work item e of a record: the cell's member j with candidate k
// of the 13 directions m > 13, or two members; false for the half of the
// member pairs that is skipped.
__device__ __forceinline__ bool rec_pair(const DevState &d, const int *rec, int s0, int cnt, int m0, int m2, int e, int &j,
                                         int &q) {
	if(e < cnt * m2) {
		j = s0 + e / m2;
		q = rec_slot(d, rec, e % m2 + m0);
		return true;
	}
	const int a = (e - cnt * m2) / cnt, b2 = (e - cnt * m2) % cnt;
	j = s0 + a;
	q = s0 + b2;
	return a < b2;
}

// The energy of box trials on the current lists, from the sweep's cell
// records instead of per particle: listed cell i (of the 8 passes' lists one
// after another) pairs its members with each other once and with the
// members of its neighbours in the 13 directions m > 13 of the record (m =
// 9 (dx + 1) + 3 (dy + 1) + dz + 1), so every pair of particles in adjacent
// cells is seen exactly once.  The separation is formed from the cell's
// member as k_energy forms it from either particle (scaled positions, the
// trial box) and pair_bonded decides the bond, so a bonded pair adds 2 to
// the bond rows (the per-particle sum counts it twice) and an overlapping
// pair adds 1 to the overlap row: k_vol_decide reads the same totals.  Per
// listed cell this reads its record once, where k_energy reads 27 cell ranges
// per particle; on dilute systems most of them are empty.
// TT lanes per listed cell: 8 on dense systems; 1 on dilute ones, where a
// listed cell holds about one particle and one candidate, so that the lanes
// stream through the records instead of idling in teams.
template <int TT>
__global__ __launch_bounds__(256) void k_energy_rec(DevState d) {
	const int lane = threadIdx.x & (TT - 1);
	const int teams = gridDim.x * (blockDim.x / TT);
	int lens[8];
	int total = 0;
#pragma unroll
	for(int p = 0; p < 8; p++) {
		lens[p] = d.pfx[p * (d.R + 1) + d.R];
		total += lens[p];
	}
	for(int i0 = xcd_remap(blockIdx.x, gridDim.x) * (blockDim.x / TT) + threadIdx.x / TT; i0 < total; i0 += teams) {
		int p = 0, gi = i0;
		while(gi >= lens[p]) gi -= lens[p++];
		const int *rec = d.rec + ((size_t) p * d.total_act + gi) * REC_W;
		const int r = rec[REC_REP];
		const Rep &rp = d.reps[r];
		if(!rp.trial_active || !rp.trial_rec) continue;
		// (the early exit may read a stale flag: it only saves work)
		if(__hip_atomic_load(&d.vflag[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) continue;
		const int s0 = rec[REC_S0], cnt = rec[REC_CNT];
		const int m0 = rec[REC_M0], m2 = rec[REC_M] - m0;  // candidates in the 13 directions
		const double *F = pick_buf(d.f, rec[REC_SEL]);
		const double t0 = rp.trial_s[0], t1 = rp.trial_s[1], t2 = rp.trial_s[2];
		const double Lx = rp.tg.box[0], Ly = rp.tg.box[1], Lz = rp.tg.box[2];
		const double iLx = rp.tg.inv_box[0], iLy = rp.tg.inv_box[1], iLz = rp.tg.inv_box[2];
		const double c2 = rp.cosmax >= KF_FILTER_MIN_COS ? rp.cosmax * rp.cosmax : -1.;
		int nbond = 0, novl = 0;
		const int work = cnt * m2 + cnt * cnt;
		for(int e = lane; e < work; e += TT) {
			int j, q;
			if(!rec_pair(d, rec, s0, cnt, m0, m2, e, j, q)) continue;
			const double px = part(F, j)[0] * t0, py = part(F, j)[1] * t1, pz = part(F, j)[2] * t2;
			const double dx = kf_min_image(part(F, q)[0] * t0 - px, Lx, iLx);
			const double dy = kf_min_image(part(F, q)[1] * t1 - py, Ly, iLy);
			const double dz = kf_min_image(part(F, q)[2] * t2 - pz, Lz, iLz);
			const double d2 = dx * dx + dy * dy + dz * dz;
			if(d2 < 1.) novl++;
			else if(d2 < rp.rc2) {
				double O[9], P[4][3];
#pragma unroll
				for(int c = 0; c < 9; c++) O[c] = part(F, j)[3 + c];
				kf_patches(O, P);
				nbond += (int) pair_bonded(dx, dy, dz, d2, &P[0][0], c2, rp.cosmax, [&](double *Oq) {
#pragma unroll
					for(int c = 0; c < 9; c++) Oq[c] = part(F, q)[3 + c];
				});
			}
		}
		if constexpr(TT > 1) {
			nbond = team_sum<TT>(nbond);
			novl = team_sum<TT>(novl);
		}
		if(lane == 0) {
			const int slot = i0 & (NSLOT - 1);
			if(novl) {
				__hip_atomic_store(&d.vflag[r], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				atomicAdd(ctr_at(d.ctr, r, C_OVL, slot), (unsigned long long) novl);
			}
			else if(nbond)
				atomicAdd(ctr_at(d.ctr, r, C_EBONDS, slot), 2ull * (unsigned long long) nbond);
		}
	}
}

void launch_energy_rec(const DevState &d, int cus, hipStream_t s) {
	// a grid-stride loop over the listed cells: 8 workgroups per CU (a
	// multiple of 8: one contiguous range of cells per XCD); one lane per
	// cell when the 27 cells around a particle hold fewer than 8 candidates
	const int blocks = std::max(8, cus * 8) & ~7;
	const double cand = 27. * (double) d.Ntot / (double) (d.C_total > 0 ? d.C_total : 1);
	if(cand < 8.) hipLaunchKernelGGL(k_energy_rec<1>, dim3((unsigned) blocks), dim3(256), 0, s, d);
	else hipLaunchKernelGGL(k_energy_rec<8>, dim3((unsigned) blocks), dim3(256), 0, s, d);
}

// ------------------------------------------------------------------------
// Close pairs of the box trials.  At the start of a sweep's box trials the
// records give every pair of particles in adjacent cells once, as
// k_energy_rec enumerates them; of each replica that makes box trials, the
// pairs closer than PAIR_LIST_FACTOR bond ranges (minimum image in the
// current box) are listed.  A trial scales every separation by the axis
// factors accepted since the list was built (pl_scale) times its own.  While
// the smallest of those products s keeps s x PAIR_LIST_FACTOR above 1 (with a
// margin for the roundings of the list's test), an unlisted pair of adjacent
// cells stays beyond the bond range, and a fast trial already holds every
// pair within the bond range in adjacent cells: the trial's energy is the sum
// over the listed pairs, pair by pair as k_energy_rec takes it.

// Which replicas list their pairs this sweep (box trials on current lists
// whose records were written by this sweep's rebuild), and an empty list.
__device__ __forceinline__ bool lists_pairs(const Rep &rp) {
	return (rp.ensemble == 5 || rp.lx_move) && rp.rec_ok && rp.lists_ok;
}

// The replicas' pair state at the start of the sweep's box trials, by the
// building kernel's first workgroup (the rebuild has emptied the list).
__device__ __forceinline__ void pairs_reset(const DevState &d) {
	if(blockIdx.x != 0) return;
	for(int r = threadIdx.x; r < d.R; r += blockDim.x) {
		Rep &rp = d.reps[r];
		rp.pl_ok = lists_pairs(rp) ? 1 : 0;
		rp.pl_scale[0] = rp.pl_scale[1] = rp.pl_scale[2] = 1.;
	}
}

// Few cells: 16 lanes per listed cell share its pairs, and remember those they
// found close (a bit per step) while the workgroup reserves its places with
// one atomic.  A lane per cell walks a cell's pairs one after the other, two
// dependent loads each, twice: 28 us for N=1331 at rho 0.3, this 5.7.
__global__ __launch_bounds__(256) void k_pairs_build_team(DevState d) {
	constexpr int T = 16;
	__shared__ int wsum[4], base;
	pairs_reset(d);
	const int tl = threadIdx.x & (T - 1), lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	int lens[8];
	int total = 0;
#pragma unroll
	for(int p = 0; p < 8; p++) {
		lens[p] = d.pfx[p * (d.R + 1) + d.R];
		total += lens[p];
	}
	for(int g0 = blockIdx.x * (256 / T); g0 < total; g0 += gridDim.x * (256 / T)) {
		const int i0 = g0 + threadIdx.x / T;
		const int *rec = d.rec;
		int s0 = 0, cnt = 0, m0 = 0, m2 = 0, work = 0;
		const double *F = d.f[0];
		double L[3] = {1., 1., 1.}, iL[3] = {1., 1., 1.}, rl2 = 0.;
		if(i0 < total) {
			int p = 0, gi = i0;
			while(gi >= lens[p]) gi -= lens[p++];
			rec = d.rec + ((size_t) p * d.total_act + gi) * REC_W;
			const Rep &rp = d.reps[rec[REC_REP]];
			s0 = rec[REC_S0];
			cnt = rec[REC_CNT];
			m0 = rec[REC_M0];
			m2 = rec[REC_M] - m0;
			F = pick_buf(d.f, rec[REC_SEL]);
			for(int a = 0; a < 3; a++) {
				L[a] = rp.g.box[a];
				iL[a] = rp.g.inv_box[a];
			}
			rl2 = rp.rc2 * (PAIR_LIST_FACTOR * PAIR_LIST_FACTOR);
			if(lists_pairs(rp)) work = cnt * m2 + cnt * cnt;
		}
		// pair e, if it is one and close (bits: the first 32 steps' results)
		auto close = [&](int e, int &j, int &q) {
			if(!rec_pair(d, rec, s0, cnt, m0, m2, e, j, q)) return false;
			const double dx = kf_min_image(part(F, q)[0] - part(F, j)[0], L[0], iL[0]);
			const double dy = kf_min_image(part(F, q)[1] - part(F, j)[1], L[1], iL[1]);
			const double dz = kf_min_image(part(F, q)[2] - part(F, j)[2], L[2], iL[2]);
			return dx * dx + dy * dy + dz * dz < rl2;
		};
		int n = 0, j, q;
		unsigned bits = 0;
		for(int e = tl, k = 0; e < work; e += T, k++)
			if(close(e, j, q)) {
				n++;
				if(k < 32) bits |= 1u << k;
			}
		const int incl = wave_incl_scan(n);
		if(lane == 63) wsum[wave] = incl;
		__syncthreads();
		const int tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
		if(threadIdx.x == 0) base = tot > 0 ? atomicAdd(d.pl_n, tot) : 0;
		__syncthreads();
		int pos = base + incl - n;
		for(int w = 0; w < wave; w++) pos += wsum[w];
		if(base + tot > d.pl_cap) {
			if(threadIdx.x == 0) d.pl_n[1] = 1;
		}
		else
			for(int e = tl, k = 0; e < work; e += T, k++) {
				if(k < 32 ? !((bits >> k) & 1u) : !close(e, j, q)) continue;
				rec_pair(d, rec, s0, cnt, m0, m2, e, j, q);
				d.pl[pos++] = make_int2(j, q);
			}
		__syncthreads();  // (wsum and base are written again)
	}
}

// One lane per listed cell, the wavefront's lanes in step: each counts its
// close pairs, one atomic per wavefront reserves their places (in no fixed
// order: the trial energies are integer sums), then each writes them.  A
// list that would pass pl_cap is marked as overflowed; the trials then take
// their energy from the records.
__global__ __launch_bounds__(256) void k_pairs_build(DevState d) {
	pairs_reset(d);
	const int lane = threadIdx.x & 63;
	const int wave = (xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + (int) threadIdx.x) >> 6;
	const int waves = gridDim.x * (blockDim.x >> 6);
	int lens[8];
	int total = 0;
#pragma unroll
	for(int p = 0; p < 8; p++) {
		lens[p] = d.pfx[p * (d.R + 1) + d.R];
		total += lens[p];
	}
	for(int w0 = wave * 64; w0 < total; w0 += waves * 64) {
		const int i0 = w0 + lane;
		const int *rec = d.rec;
		bool on = false;
		int s0 = 0, cnt = 0, m0 = 0, m2 = 0;
		const double *F = d.f[0];
		double L[3] = {1., 1., 1.}, iL[3] = {1., 1., 1.}, rl2 = 0.;
		if(i0 < total) {
			int p = 0, gi = i0;
			while(gi >= lens[p]) gi -= lens[p++];
			rec = d.rec + ((size_t) p * d.total_act + gi) * REC_W;
			const Rep &rp = d.reps[rec[REC_REP]];
			on = lists_pairs(rp);
			if(on) {
				s0 = rec[REC_S0];
				cnt = rec[REC_CNT];
				m0 = rec[REC_M0];
				m2 = rec[REC_M] - m0;
				F = pick_buf(d.f, rec[REC_SEL]);
				for(int a = 0; a < 3; a++) {
					L[a] = rp.g.box[a];
					iL[a] = rp.g.inv_box[a];
				}
				rl2 = rp.rc2 * (PAIR_LIST_FACTOR * PAIR_LIST_FACTOR);
			}
		}
		auto close = [&](int j, int q) {
			const double dx = kf_min_image(part(F, q)[0] - part(F, j)[0], L[0], iL[0]);
			const double dy = kf_min_image(part(F, q)[1] - part(F, j)[1], L[1], iL[1]);
			const double dz = kf_min_image(part(F, q)[2] - part(F, j)[2], L[2], iL[2]);
			return dx * dx + dy * dy + dz * dz < rl2;
		};
		const int work = on ? cnt * m2 + cnt * cnt : 0;
		int n = 0;
		for(int e = 0; e < work; e++) {
			int j, q;
			if(rec_pair(d, rec, s0, cnt, m0, m2, e, j, q) && close(j, q)) n++;
		}
		const int incl = wave_incl_scan(n);
		const int tot = __builtin_amdgcn_readlane(incl, 63);
		int base = 0;
		if(tot > 0) {
			if(lane == 0) base = atomicAdd(d.pl_n, tot);
			base = __builtin_amdgcn_readfirstlane(base);
		}
		if(base + tot > d.pl_cap) {
			if(lane == 0) d.pl_n[1] = 1;
			continue;
		}
		int pos = base + incl - n;
		for(int e = 0; e < work; e++) {
			int j, q;
			if(rec_pair(d, rec, s0, cnt, m0, m2, e, j, q) && close(j, q)) d.pl[pos++] = make_int2(j, q);
		}
	}
}

void launch_pairs_build(const DevState &d, int cus, hipStream_t s) {
	// 16 lanes per cell while a lane per cell (at most one cell per particle)
	// would leave the chip idle, and where cells have many pairs; big dilute
	// systems, about one pair per cell, take a lane.  16 lanes / one lane, us:
	// N=60000 at rho 0.3 46 / 361, 120000 at 0.05 75 / 86, 400000 at 0.3 295 /
	// 691, at 0.1 291 / 224, 10^6 at 0.15 725 / 593, 2.1 10^6 at 0.05 1316 / 437.
	if(d.Ntot < cus * 512 || 27. * d.Ntot >= 6. * d.C_total) {
		const int blocks = std::max(1, std::min((d.Ntot + 15) / 16, cus * 8));
		hipLaunchKernelGGL(k_pairs_build_team, dim3((unsigned) blocks), dim3(256), 0, s, d);
		return;
	}
	const int blocks = std::max(8, cus * 8) & ~7;
	hipLaunchKernelGGL(k_pairs_build, dim3((unsigned) blocks), dim3(256), 0, s, d);
}

// Run-ahead box attempts (ahead: enqueued without the host reading each
// attempt's paths): an attempt proceeds on the close-pair list alone, which
// serves every fast trial in the common case; if some replica's trial needs
// more, the sequence stops there: the kernels of this and the later attempts
// leave at once, the proposal stays in place and its paths stay in vslow[0]
// for the host to take over from.  The attempt's own kernels read that from
// vslow[0]; its last one (k_vol_apply) marks the stop in vslow[1] before a
// later proposal could add to it.
__device__ __forceinline__ bool attempt_stopped(const DevState &d, int ahead) {
	return d.vslow[1] >= 0 || (ahead && (d.vslow[0] & ~(int) NEED_PAIRS));
}

// The trial energies from the close-pair list: one lane per pair, the
// separation and the bond decision as k_energy_rec forms them; a bonded pair
// adds 2 to the bond rows, an overlapping pair 1 to the overlap row.
__global__ __launch_bounds__(256) void k_energy_pairs(DevState d, int ahead) {
	if(attempt_stopped(d, ahead)) return;
	const int n = min(d.pl_n[0], d.pl_cap);
	const int stride = gridDim.x * blockDim.x;
	for(int k = xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; k < n; k += stride) {
		const int2 pq = d.pl[k];
		const int j = pq.x, q = pq.y;
		if((unsigned) j >= (unsigned) d.Ntot || (unsigned) q >= (unsigned) d.Ntot) continue;
		const int r = d.prep[j];
		const Rep &rp = d.reps[r];
		if(!rp.trial_active || !rp.trial_pl) continue;
		// (the early exit may read a stale flag: it only saves work)
		if(__hip_atomic_load(&d.vflag[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) continue;
		const double *F = pick_buf(d.f, rp.sel);
		const double t0 = rp.trial_s[0], t1 = rp.trial_s[1], t2 = rp.trial_s[2];
		const double px = part(F, j)[0] * t0, py = part(F, j)[1] * t1, pz = part(F, j)[2] * t2;
		const double dx = kf_min_image(part(F, q)[0] * t0 - px, rp.tg.box[0], rp.tg.inv_box[0]);
		const double dy = kf_min_image(part(F, q)[1] * t1 - py, rp.tg.box[1], rp.tg.inv_box[1]);
		const double dz = kf_min_image(part(F, q)[2] * t2 - pz, rp.tg.box[2], rp.tg.inv_box[2]);
		const double d2 = dx * dx + dy * dy + dz * dz;
		const int slot = k & (NSLOT - 1);
		if(d2 < 1.) {
			__hip_atomic_store(&d.vflag[r], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			atomicAdd(ctr_at(d.ctr, r, C_OVL, slot), 1ull);
		}
		else if(d2 < rp.rc2) {
			const double c2 = rp.cosmax >= KF_FILTER_MIN_COS ? rp.cosmax * rp.cosmax : -1.;
			double O[9], P[4][3];
#pragma unroll
			for(int c = 0; c < 9; c++) O[c] = part(F, j)[3 + c];
			kf_patches(O, P);
			if(pair_bonded(dx, dy, dz, d2, &P[0][0], c2, rp.cosmax, [&](double *Oq) {
#pragma unroll
				   for(int c = 0; c < 9; c++) Oq[c] = part(F, q)[3 + c];
			   }))
				atomicAdd(ctr_at(d.ctr, r, C_EBONDS, slot), 2ull);
		}
	}
}

void launch_energy_pairs(const DevState &d, int cus, int ahead, hipStream_t s) {
	const int blocks = std::max(8, cus * 8) & ~7;
	hipLaunchKernelGGL(k_energy_pairs, dim3((unsigned) blocks), dim3(256), 0, s, d, ahead);
}

// ------------------------------------------------------------------------
// Checkerboard invariant (a debug check; the reference is serial).  The
// particles of one colour's cells move concurrently, so no particle may lie
// within the bond range of a particle in another cell of the same colour.
// Counts the particles of replica `rep` that do, on the grid G (cells by
// cell_coord, colours by the cells' parities, separations by minimum image
// in G's box): brute force over the replica's live slots, every colour at
// once since each particle belongs to one.  One thread per slot.
__global__ void k_colour_conflicts(DevState d, int rep, int n0, int n1, int n2, unsigned long long *out) {
	const Rep &rp = d.reps[rep];
	// the grid of the current cell lists, or n0 x n1 x n2 cells over the box
	Grid G = rp.lg;
	if(n0 > 0) {
		set_grid_box(G, rp.g.box);
		G.n[0] = n0;
		G.n[1] = n1;
		G.n[2] = n2;
		G.shift[0] = G.shift[1] = G.shift[2] = 0.;
	}
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= rp.np_hw) return;
	const int j = rp.p_off + i;
	const int *PID = pick_buf(d.pid, rp.sel);
	if(PID[j] < 0) return;
	const double *F = pick_buf(d.f, rp.sel);
	const double x = part(F, j)[0], y = part(F, j)[1], z = part(F, j)[2];
	auto cell = [&](double a, double b, double c, int &cx, int &cy, int &cz) {
		cx = cell_coord(a, G.shift[0], G.inv_box[0], G.n[0]);
		cy = cell_coord(b, G.shift[1], G.inv_box[1], G.n[1]);
		cz = cell_coord(c, G.shift[2], G.inv_box[2], G.n[2]);
	};
	int ix, iy, iz;
	cell(x, y, z, ix, iy, iz);
	const int col = ((ix & 1) << 2) | ((iy & 1) << 1) | (iz & 1);
	bool hit = false;
	for(int k = 0; k < rp.np_hw && !hit; k++) {
		const int q = rp.p_off + k;
		if(q == j || PID[q] < 0) continue;
		const double qx = part(F, q)[0], qy = part(F, q)[1], qz = part(F, q)[2];
		int cx, cy, cz;
		cell(qx, qy, qz, cx, cy, cz);
		if((((cx & 1) << 2) | ((cy & 1) << 1) | (cz & 1)) != col || (cx == ix && cy == iy && cz == iz)) continue;
		const double dx = kf_min_image(qx - x, G.box[0], G.inv_box[0]);
		const double dy = kf_min_image(qy - y, G.box[1], G.inv_box[1]);
		const double dz = kf_min_image(qz - z, G.box[2], G.inv_box[2]);
		hit = dx * dx + dy * dy + dz * dz < rp.rc2;
	}
	if(hit) atomicAdd(out, 1ull);
}

// nside == nullptr: the grid of the replica's current cell lists; else
// nside cells per axis over its box, no shift.  `slots`: the replica's slot
// capacity (the grid covers it; threads past its live slots leave).
void launch_colour_conflicts(const DevState &d, int rep, int slots, const int *nside, unsigned long long *out,
                             hipStream_t s) {
	const int n = std::max(slots, 1);
	hipLaunchKernelGGL(k_colour_conflicts, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, d, rep,
	                   nside ? nside[0] : 0, nside ? nside[1] : 0, nside ? nside[2] : 0, out);
}

// ------------------------------------------------------------------------
// NPT volume move (MC.c:450-513): log-volume step along one random axis

// Whether the trial of a replica can be evaluated on its current lists: the
// lists' cells, rescaled with the trial, stay at least side_min wide on
// every axis, so every pair within the bond range still lies in adjacent
// cells (the margin in side_min covers the roundings of the membership).
// Otherwise (or when asked for every trial) the trial regroups the particles
// on its own grid into the spare buffer; the host launches that rebuild only
// when some replica needs it.
__device__ __forceinline__ void choose_trial_path(const DevState &d, Rep &rp, const double tb[3]) {
	bool fast = d.npt_trial_form != 2 && rp.lists_ok;
	for(int a = 0; a < 3; a++) fast = fast && tb[a] / (double) rp.lg.n[a] >= rp.side_min;
	rp.trial_fast = fast ? 1 : 0;
	// a fast trial takes its energy from the cell records while they describe
	// the lists (the sweep's shifting rebuild wrote them)
	rp.trial_rec = (fast && rp.rec_ok && (d.npt_trial_form == 0 || d.npt_trial_form == 3)) ? 1 : 0;
	// the close-pair list while the cumulative scaling keeps unlisted pairs
	// beyond the bond range (1e-9: the roundings of the list's test)
	double smin = 1e300;
	for(int a = 0; a < 3; a++) smin = fmin(smin, rp.pl_scale[a] * rp.trial_s[a]);
	rp.trial_pl = (rp.trial_rec && d.npt_trial_form == 0 && rp.pl_ok && d.pl_n && d.pl_n[1] == 0 &&
	               smin * PAIR_LIST_FACTOR >= 1. + 1e-9) ? 1 : 0;
	if(rp.trial_pl) rp.trial_rec = 0;
	atomicOr(d.vslow, fast ? (rp.trial_pl ? (int) NEED_PAIRS : (rp.trial_rec ? (int) NEED_RECORDS : (int) NEED_PARTICLES))
	                       : (int) (NEED_REBUILD | NEED_PARTICLES));
}

// One wavefront per replica; its lanes also clear the replica's energy rows for
// the trial energies.
__global__ __launch_bounds__(64) void k_vol_propose(DevState d, uint64_t sweep, int k) {
	const int r = blockIdx.x;
	if(d.vslow[1] >= 0) return;
	*ctr_at(d.ctr, r, C_EBONDS, threadIdx.x) = 0ull;
	*ctr_at(d.ctr, r, C_OVL, threadIdx.x) = 0ull;
	if(threadIdx.x != 0) return;
	Rep &rp = d.reps[r];
	rp.trial_active = 0;
	rp.trial_fast = 0;
	rp.trial_rec = 0;
	rp.trial_pl = 0;
	rp.vol_apply = 0;
	d.vflag[r] = 0;
	if(rp.ensemble != 5 && !rp.lx_move) return;
	u32x4 v = rng(d.seed, r, sweep, (uint32_t) k, TAG_VOLUME, 0, 0);  // attempt k of the sweep
	if(rp.ensemble != 5) {
		// box-shape move at constant volume (MC_change_Lx, MC.c:515-531):
		// Lx += U(-1/2, 1/2) Lx_change_max, Ly = Lz = sqrt(V / Lx), rejected
		// early outside [Lyz_min, Lyz_max] (or, here, without a valid grid)
		const double Lx = rp.g.box[0] + (u01(v.x) - 0.5) * rp.lx_change_max;
		const double Lyz = Lx > 0. ? sqrt(rp.V / Lx) : -1.;
		double tb[3] = {Lx, Lyz, Lyz};
		int tn[3];
		if(!(Lyz >= rp.lyz_min && Lyz <= rp.lyz_max) ||
		   !make_grid(tb, rp.side_min, rp.min_n, rp.even, rp.cap_n, tn)) {
			atomicAdd(ctr_at(d.ctr, r, C_TRY_VOL, 0), 1ull);
			return;
		}
		for(int a = 0; a < 3; a++) rp.trial_s[a] = tb[a] / rp.g.box[a];
		set_grid_box(rp.tg, tb);
		for(int a = 0; a < 3; a++) {
			rp.tg.n[a] = tn[a];
			rp.tg.shift[a] = rp.g.shift[a] * rp.trial_s[a];
		}
		rp.trial_kind = 1;
		rp.trial_active = 1;
		choose_trial_path(d, rp, tb);
		return;
	}
	const int dir = (int) (u01(v.x) * 3.);
	const double V0 = rp.g.box[0] * rp.g.box[1] * rp.g.box[2];
	const double lnV1 = log(V0) + (u01(v.y) - 0.5) * rp.rfm;
	const double V1 = exp(lnV1);
	double side = V1;
	for(int k = 0; k < 3; k++)
		if(k != dir) side /= rp.g.box[k];
	double tb[3] = {rp.g.box[0], rp.g.box[1], rp.g.box[2]};
	const double f = side / tb[dir];
	tb[dir] = side;
	int tn[3];
	const bool ok = make_grid(tb, rp.side_min, rp.min_n, rp.even, rp.cap_n, tn);
	if(!ok) {
		// the trial box cannot hold a checkerboard grid: the move is rejected
		atomicAdd(ctr_at(d.ctr, r, C_TRY_VOL, 0), 1ull);
		return;
	}
	set_grid_box(rp.tg, tb);
	for(int k = 0; k < 3; k++) {
		rp.tg.n[k] = tn[k];
		rp.tg.shift[k] = rp.g.shift[k];
	}
	rp.trial_dir = dir;
	rp.trial_f = f;
	for(int a = 0; a < 3; a++) rp.trial_s[a] = a == dir ? f : 1.;
	rp.trial_V = V1;
	rp.trial_V0 = V0;
	rp.trial_kind = 0;
	rp.trial_active = 1;
	choose_trial_path(d, rp, tb);
}

// The trial-energy paths the box attempt in flight needs (TrialNeed bits in
// vslow, gathered by k_vol_propose), written straight into the host's pinned
// word with the attempt's sequence number above them: the host waits for
// exactly this attempt's value without a copy or a stream synchronisation.
__global__ void k_vol_publish(DevState d, int *host_word, unsigned seq) {
	if(threadIdx.x == 0) {
		const int need = __hip_atomic_load(d.vslow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__hip_atomic_store(host_word, (int) ((seq << 4) | (unsigned) need), __ATOMIC_RELAXED,
		                   __HIP_MEMORY_SCOPE_SYSTEM);
	}
}

void launch_vol_publish(const DevState &d, int *host_word, unsigned seq, hipStream_t s) {
	hipLaunchKernelGGL(k_vol_publish, dim3(1), dim3(64), 0, s, d, host_word, seq);
}

void launch_vol_propose(const DevState &d, uint64_t sweep, int k, hipStream_t s) {
	static_assert(NSLOT == 64, "a lane per slot");
	hipLaunchKernelGGL(k_vol_propose, dim3(d.R), dim3(64), 0, s, d, sweep, k);
}

// One wavefront per replica, a lane per counter slot.
__global__ __launch_bounds__(64) void k_vol_decide(DevState d, uint64_t sweep, int k, int ahead) {
	const int r = blockIdx.x;
	Rep &rp = d.reps[r];
	unsigned long long eb = *ctr_at(d.ctr, r, C_EBONDS, threadIdx.x), ov = *ctr_at(d.ctr, r, C_OVL, threadIdx.x),
	                   db = *ctr_at(d.ctr, r, C_DBONDS, threadIdx.x);
	if(attempt_stopped(d, ahead) || !rp.trial_active) return;
	for(int o = 32; o > 0; o >>= 1) {
		eb += __shfl_xor(eb, o);
		ov += __shfl_xor(ov, o);
		db += __shfl_xor(db, o);
	}
	if(threadIdx.x != 0) return;
	const long long B1 = (long long) eb / 2;
	const long long B0 = rp.bonds_base + (long long) db;
	const double dE = (double) (B0 - B1);  // E' - E with E = -bonds
	// volume: MC.c:497-499; box shape: exp(-dE/T) at constant volume (the
	// Jacobian of the rescaling is 1), or, on request, the reference's
	// exp(+dE/T) (MC.c:562), which does not keep the Boltzmann distribution
	const double arg = rp.trial_kind == 1
	                       ? (rp.lx_ref_rule ? dE / rp.T : -dE / rp.T)
	                       : -(rp.P * (rp.trial_V - rp.trial_V0) + dE) / rp.T + (double) (rp.np + 1) * log(rp.trial_f);
	u32x4 v = rng(d.seed, r, sweep, (uint32_t) k, TAG_VOLUME, 0, 0);  // attempt k of the sweep
	atomicAdd(ctr_at(d.ctr, r, C_TRY_VOL, 0), 1ull);
	if(ov == 0 && u01(v.z) < exp(arg)) {
		if(rp.trial_fast) {
			// the positions are rescaled in place (k_vol_apply); the lists keep
			// their members, their grid is rescaled with the positions
			rp.vol_apply = 1;
			for(int a = 0; a < 3; a++) rp.pl_scale[a] *= rp.trial_s[a];
			set_grid_box(rp.lg, rp.tg.box);
			for(int a = 0; a < 3; a++) rp.lg.shift[a] *= rp.trial_s[a];
		}
		else {
			// the spare buffer holds the trial, grouped on the trial grid
			// (the cell records describe the old lists)
			rp.sel ^= 1;
			rp.lg = rp.tg;
			rp.lists_ok = 1;
			rp.rec_ok = 0;
			rp.pl_ok = 0;
			rp.np_hw = rp.np;
		}
		rp.g = rp.tg;
		if(rp.trial_kind == 0) rp.V = rp.trial_V;
		rp.bonds_base = B1 - (long long) db;
		atomicAdd(ctr_at(d.ctr, r, C_ACC_VOL, 0), 1ull);
	}
	else if(!rp.trial_fast)
		rp.lists_ok = 0;  // the lists now group the spare buffer, not the current one
	rp.trial_active = 0;
}

void launch_vol_decide(const DevState &d, uint64_t sweep, int k, int ahead, hipStream_t s) {
	hipLaunchKernelGGL(k_vol_decide, dim3(d.R), dim3(64), 0, s, d, sweep, k, ahead);
}

// The accepted fast trials: every position component times its trial scale,
// as the trial rebuild writes it (x * 1 is x).  Clears the trial paths for
// the next attempt, or marks where a run-ahead sequence stopped; either way
// the other workgroups find the same answer before and after.
// host_word (the last attempt of a run-ahead sequence): where it stopped
// (attempt + 1, 0 if it ran through) with the host's sequence number goes into
// that pinned word, and the stop is cleared for the attempts that follow (the
// paths in vslow[0] still hold this kernel's other workgroups back).
__global__ void k_vol_apply(DevState d, int k, int ahead, int *host_word, unsigned seq) {
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	const bool stopped = attempt_stopped(d, ahead);
	if(j == 0) {
		int stop = 0;
		if(stopped) {
			const int at = d.vslow[1] < 0 ? k : d.vslow[1];
			stop = at + 1;
			d.vslow[1] = host_word ? -1 : at;
		}
		else *d.vslow = 0;
		if(host_word)
			__hip_atomic_store(host_word, (int) ((seq << 8) | (unsigned) stop), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
	}
	if(stopped || j >= d.Ntot) return;
	const Rep &rp = d.reps[d.prep[j]];
	if(!rp.vol_apply) return;
	double *F = pick_buf(d.f, rp.sel);
	for(int c = 0; c < 3; c++) part(F, j)[c] *= rp.trial_s[c];
}

void launch_vol_apply(const DevState &d, int k, int ahead, int *host_word, unsigned seq, hipStream_t s) {
	hipLaunchKernelGGL(k_vol_apply, dim3((unsigned) std::max(1, (d.Ntot + 255) / 256)), dim3(256), 0, s, d, k, ahead, host_word,
	                   seq);
}

// ------------------------------------------------------------------------
// Grand-canonical insertions and removals (MC_add_remove, MC.c:342-448),
// made cell-local for the checkerboard: once per sweep, after the colour
// passes, every cell of one colour (drawn per replica and sweep; empty
// cells too) tries one insertion or one removal, each with probability 1/2.
//   insertion: a position uniform in the cell and an orientation uniform on
//     SO(3) (random_orientation, utils.c:133-169), accepted with
//     min(1, z v_c / (n_c + 1) exp(-dE/T)), dE = -(bonds of the new particle)
//   removal: a member uniform among the cell's n_c, accepted with
//     min(1, n_c / (z v_c) exp(-dE/T)), dE = +(the member's bonds)
// (MC.c:367 and MC.c:391 with the cell's volume and population in place of
// the box's).  Cells of one colour are a cell side apart, so their moves do
// not interact: each pair of moves satisfies detailed balance for
// z^N / N! exp(-E/T) on its own.  A cell's insertion takes a slot reserved
// for that cell (np + its index among the colour's cells), so the outcome
// does not depend on thread timing; a replica with fewer free slots than
// cells of one colour skips the phase and reports ERR_GC_FULL.

// Begin a GC phase: particle indices of each grand-canonical replica become
// 0 .. np - 1 in slot order.  After the sweep's passes every cell holds its
// members in order of particle index, so slot order is the same for every
// launch shape; this keeps the indices dense for the phase's insertions,
// which take indices from np on.
__global__ void k_gc_begin(DevState d, uint64_t sweep) {
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if(j >= d.Ntot) return;
	const int r = d.prep[j];
	Rep &rp = d.reps[r];
	if(!rp.gc) return;
	const int loc = j - rp.p_off;
	if(loc < rp.np) pick_buf(d.pid, rp.sel)[j] = loc;
	if(loc == 0) {
		const u32x4 v = rng(d.seed, r, sweep, 0, TAG_GC, 0, 0);
		rp.gc_colour = (int) (v.x & 7u);
		const int ncol = (rp.g.n[0] / 2) * (rp.g.n[1] / 2) * (rp.g.n[2] / 2);
		if(rp.np + ncol > rp.cap_np) {
			atomicOr(d.err, (int) ERR_GC_FULL);
			rp.gc_base = -1;
		}
		else {
			rp.gc_base = rp.np;
			rp.np_hw = rp.np + ncol;
			rp.lists_ok = 0;  // the phase adds and removes particles the lists do not show
			rp.rec_ok = 0;
		}
	}
}

// Orientation uniform on SO(3) as random_orientation builds it (utils.c:
// 133-169): three uniform unit vectors x, y, z, Gram-Schmidt in that order,
// rows (z, x, y), or (x, z, y) when that has determinant -1.
__device__ inline void gc_orientation(uint64_t seed, int r, uint64_t sweep, uint32_t cell, uint32_t col, double O[9]) {
	double v[9];
	for(int k = 0; k < 3; k++) sphere_axis(seed, r, sweep, cell, col, 0x8000u + (uint32_t) k, v + 3 * k);
	gram_schmidt_rows(v);
	const double *x = v, *y = v + 3, *z = v + 6;
	const double det = z[0] * (x[1] * y[2] - x[2] * y[1]) - z[1] * (x[0] * y[2] - x[2] * y[0]) +
	                   z[2] * (x[0] * y[1] - x[1] * y[0]);
	const double *r0 = det < 0. ? x : z, *r1 = det < 0. ? z : x;
	for(int k = 0; k < 3; k++) {
		O[k] = r0[k];
		O[3 + k] = r1[k];
		O[6 + k] = y[k];
	}
}

// Bonds of a particle at p with patches P against every particle of the 27
// cells around cell (ix, iy, iz) but slot `skip` (MC_energy, MC.c:272-309):
// T lanes, the cells shared out; every lane returns the team's count and
// whether any overlap was met.
template <int T>
__device__ inline int gc_bonds(const DevState &d, const Rep &rp, const double *F, int ix, int iy, int iz,
                               const double p[3], const double P[4][3], int skip, int lane, bool &any) {
	const Grid &G = rp.g;
	const int n0 = G.n[0], n1 = G.n[1], n2 = G.n[2];
	int nb_ = 0;
	bool ov = false;
	for(int nb = lane; nb < 27; nb += T) {
		const int cx = wrapi(ix + nb / 9 - 1, n0), cy = wrapi(iy + (nb / 3) % 3 - 1, n1), cz = wrapi(iz + nb % 3 - 1, n2);
		const int cc = rp.cell_off + (cx * n1 + cy) * n2 + cz;
		for(int q = d.start[cc]; q < d.start[cc + 1]; q++) {
			if(q == skip) continue;
			double dx = kf_min_image(part(F, q)[0] - p[0], G.box[0], G.inv_box[0]);
			double dy = kf_min_image(part(F, q)[1] - p[1], G.box[1], G.inv_box[1]);
			double dz = kf_min_image(part(F, q)[2] - p[2], G.box[2], G.inv_box[2]);
			const double d2 = dx * dx + dy * dy + dz * dz;
			if(d2 < 1.) ov = true;
			else if(d2 < rp.rc2) {
				kf_unit(dx, dy, dz, d2);
				if(kf_any_p(dx, dy, dz, &P[0][0], rp.cosmax)) {
					double Oq[9];
					for(int c = 0; c < 9; c++) Oq[c] = part(F, q)[3 + c];
					nb_ += kf_any_q(dx, dy, dz, Oq, rp.cosmax);
				}
			}
		}
	}
	any = team_any<T>(ov);
	return team_sum<T>(nb_);
}

// One team of 32 lanes per cell of the phase's colour, over every replica's
// cells (entry gi of the replicas' per-colour capacities).
__global__ __launch_bounds__(256) void k_gc_pass(DevState d, uint64_t sweep) {
	constexpr int T = 32;
	const int lane = threadIdx.x & (T - 1);
	const int gi = blockIdx.x * (blockDim.x / T) + threadIdx.x / T;
	if(gi >= d.total_act) return;
	int lo = 0, hi = d.R;
	while(hi - lo > 1) {
		const int mid = (lo + hi) >> 1;
		if(d.act_off[mid] <= gi) lo = mid;
		else hi = mid;
	}
	const int r = lo;
	const Rep &rp = d.reps[r];
	if(!rp.gc || rp.gc_base < 0) return;
	const int n0 = rp.g.n[0], n1 = rp.g.n[1], n2 = rp.g.n[2];
	const int h0 = n0 / 2, h1 = n1 / 2, h2 = n2 / 2;
	const int k = gi - d.act_off[r];
	if(k >= h0 * h1 * h2) return;
	const int col = rp.gc_colour;
	const int ix = 2 * (k / (h1 * h2)) + ((col >> 2) & 1), iy = 2 * ((k / h2) % h1) + ((col >> 1) & 1),
	          iz = 2 * (k % h2) + (col & 1);
	const int cloc = (ix * n1 + iy) * n2 + iz;
	const int c = rp.cell_off + cloc;
	const int s0 = d.start[c], cnt = d.start[c + 1] - s0;
	double *F = pick_buf(d.f, rp.sel);
	int *PID = pick_buf(d.pid, rp.sel);
	const u32x4 u = rng(d.seed, r, sweep, (uint32_t) cloc, TAG_GC, (uint32_t) col, 1);
	const u32x4 w = rng(d.seed, r, sweep, (uint32_t) cloc, TAG_GC, (uint32_t) col, 2);
	const double vc = (rp.g.box[0] / n0) * (rp.g.box[1] / n1) * (rp.g.box[2] / n2);
	const int cslot = gi & (NSLOT - 1);
	if(u01(u.x) < 0.5) {
		// insertion at a uniform point of the cell: the point where the
		// cell's own coordinate arithmetic puts it (a draw that rounds into a
		// neighbouring cell is rejected)
		double p[3];
		const double fr[3] = {u01(u.y), u01(u.z), u01(u.w)};
		const int ii[3] = {ix, iy, iz}, nn[3] = {n0, n1, n2};
		bool inside = true;
		for(int a = 0; a < 3; a++) {
			p[a] = rp.g.shift[a] + ((double) ii[a] + fr[a]) / (double) nn[a] * rp.g.box[a];
			inside = inside && cell_coord(p[a], rp.g.shift[a], rp.g.inv_box[a], nn[a]) == ii[a];
		}
		double O[9], P[4][3];
		gc_orientation(d.seed, r, sweep, (uint32_t) cloc, (uint32_t) col, O);
		kf_patches(O, P);
		bool ov = false;
		const int b = inside ? gc_bonds<T>(d, rp, F, ix, iy, iz, p, P, -1, lane, ov) : 0;
		if(lane != 0) return;
		atomicAdd(ctr_at(d.ctr, r, C_TRY_ADD, cslot), 1ull);
		// MC.c:367: exp(-dE/T) z V / (N + 1), dE = -b
		const double acc = exp((double) b / rp.T) * rp.activity * vc / (double) (cnt + 1);
		if(!inside || ov || !(u01(w.x) < acc)) return;
		const int slot = rp.p_off + rp.gc_base + k;
		for(int a = 0; a < 3; a++) part(F, slot)[a] = p[a];
		for(int a = 0; a < 9; a++) part(F, slot)[3 + a] = O[a];
		PID[slot] = rp.gc_base + k;
		atomicAdd(&d.reps[r].np, 1);
		atomicAdd(ctr_at(d.ctr, r, C_ACC_ADD, cslot), 1ull);
		if(b) atomicAdd(ctr_at(d.ctr, r, C_DBONDS, cslot), (unsigned long long) (long long) b);
	}
	else {
		if(cnt == 0) {
			if(lane == 0) atomicAdd(ctr_at(d.ctr, r, C_TRY_REM, cslot), 1ull);
			return;
		}
		// members sit in order of particle index: rank m is slot s0 + m
		const int q = s0 + (int) __umulhi(u.y, (uint32_t) cnt);
		const double p[3] = {part(F, q)[0], part(F, q)[1], part(F, q)[2]};
		double O[9], P[4][3];
		for(int a = 0; a < 9; a++) O[a] = part(F, q)[3 + a];
		kf_patches(O, P);
		bool ov = false;
		const int b = gc_bonds<T>(d, rp, F, ix, iy, iz, p, P, q, lane, ov);
		if(lane != 0) return;
		atomicAdd(ctr_at(d.ctr, r, C_TRY_REM, cslot), 1ull);
		// MC.c:391: exp(-dE/T) N / (V z), dE = +b
		const double acc = exp(-(double) b / rp.T) * (double) cnt / (vc * rp.activity);
		if(!(u01(w.x) < acc)) return;
		PID[q] = -1;
		atomicSub(&d.reps[r].np, 1);
		atomicAdd(ctr_at(d.ctr, r, C_ACC_REM, cslot), 1ull);
		if(b) atomicAdd(ctr_at(d.ctr, r, C_DBONDS, cslot), (unsigned long long) (long long) -b);
	}
}

void launch_gc_phase(const DevState &d, uint64_t sweep, hipStream_t s) {
	if(d.Ntot <= 0 || d.total_act <= 0) return;
	hipLaunchKernelGGL(k_gc_begin, dim3((d.Ntot + 255) / 256), dim3(256), 0, s, d, sweep);
	hipLaunchKernelGGL(k_gc_pass, dim3((d.total_act + 7) / 8), dim3(256), 0, s, d, sweep);
}

// ------------------------------------------------------------------------
// Gram-Schmidt of every orientation (MC_check_energy, MC.c:775)

__global__ void k_gram_schmidt(DevState d) {
	int j = blockIdx.x * blockDim.x + threadIdx.x;
	if(j >= d.Ntot) return;
	const Rep &rp = d.reps[d.prep[j]];
	if(j - rp.p_off >= rp.np) return;
	double *F = pick_buf(d.f, rp.sel);
	double O[9];
#pragma unroll
	for(int c = 0; c < 9; c++) O[c] = part(F, j)[3 + c];
	gram_schmidt_rows(O);
#pragma unroll
	for(int c = 0; c < 9; c++) part(F, j)[3 + c] = O[c];
}

void launch_gram_schmidt(const DevState &d, hipStream_t s) {
	hipLaunchKernelGGL(k_gram_schmidt, dim3((d.Ntot + 255) / 256), dim3(256), 0, s, d);
}

}  // namespace ppd
