// pp_learn.hip -- the learned proposal of the rototranslation sweep (gfx950).
//
// A move of particle p becomes: descriptor of p's neighbourhood -> MLP (BF16
// weights, FP32 accumulation on MFMA) -> a Gaussian displacement in p's body
// frame and a 4-component von Mises-Fisher mixture over the rotation axis (the
// angle is uniform in [0, theta_max), as the reference's) -> the proposed
// state -> the descriptor there -> the MLP again for the reverse density ->
// Metropolis-Hastings with the true Kern-Frenkel energy change and the
// forward/reverse proposal densities:
//   accept with min(1, exp(-dE/T) q(x'->x) / q(x->x')),
// so the stationary distribution is the reference's.  The rotation density
// factor of the angle is the same both ways (reverse = angle theta about -a in
// the body frame of O'), so only the axis densities enter.
//
// The same network is trained here: denoising samples from the sampler's
// states, analytic gradient of -log q, backward passes on MFMA, Adam.
#pragma clang fp contract(off)

#include "pp_device.hpp"

namespace ppd {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr float LOG_2PI = 1.8378770664093453f;

// ------------------------------------------------------------------------
// proposal density: decode the network output, log q, gradient of -log q

struct Prop {
	float mu[3], ls[3];
	float dir[NN_MIX][3], nrm[NN_MIX], lk[NN_MIX], lw[NN_MIX];
	bool ls_in[3], lk_in[NN_MIX];
};

__device__ inline void prop_decode(const float *y, Prop &p) {
	for(int k = 0; k < 3; k++) {
		p.mu[k] = y[k];
		const float v = y[3 + k];
		p.ls_in[k] = v > NN_LS_MIN && v < NN_LS_MAX;
		p.ls[k] = fminf(fmaxf(v, NN_LS_MIN), NN_LS_MAX);
	}
	float mx = -3.0e38f;
	for(int c = 0; c < NN_MIX; c++) mx = fmaxf(mx, y[6 + 5 * c + 4]);
	float se = 0.f;
	for(int c = 0; c < NN_MIX; c++) se += expf(y[6 + 5 * c + 4] - mx);
	const float lse = mx + logf(se);
	for(int c = 0; c < NN_MIX; c++) {
		const float *u = y + 6 + 5 * c;
		const float n = sqrtf(u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + 1e-12f);
		for(int j = 0; j < 3; j++) p.dir[c][j] = u[j] / n;
		p.nrm[c] = n;
		const float v = u[3];
		p.lk_in[c] = v > NN_LK_MIN && v < NN_LK_MAX;
		p.lk[c] = fminf(fmaxf(v, NN_LK_MIN), NN_LK_MAX);
		p.lw[c] = u[4] - lse;
	}
}

// log density of the vMF distribution on S^2 at cosine c to the mean:
// kappa / (4 pi sinh kappa) exp(kappa c)
__device__ inline float log_vmf(float lk, float c) {
	const float k = expf(lk);
	return lk - LOG_2PI - k - logf(-expm1f(-2.f * k)) + k * c;
}

// The same by the lanes of a cell's team: lane tl decodes mixture component
// tl % NN_MIX and the four meet within their quad, in the order of the
// components, so that every lane has the values of the serial form.
static_assert(NN_MIX == 4, "a quad of lanes");
struct PropLane {
	float mu[3], ls[3];
	float dir[3], k, lk, lw;  // of the lane's component (k = exp(lk))
};

template <int c>
__device__ __forceinline__ float quad_get(float v) {
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), c * 0x55, 0xf, 0xf, true));
}

// (every lane of the quad active)
__device__ __forceinline__ float quad_log_sum_exp(float l) {
	const float mx = fmaxf(fmaxf(fmaxf(fmaxf(-3.0e38f, quad_get<0>(l)), quad_get<1>(l)), quad_get<2>(l)), quad_get<3>(l));
	const float e = expf(l - mx);
	return mx + logf(quad_get<0>(e) + quad_get<1>(e) + quad_get<2>(e) + quad_get<3>(e));
}

__device__ __forceinline__ void prop_decode_lane(const float *y, int tl, PropLane &p) {
#pragma unroll
	for(int k = 0; k < 3; k++) {
		p.mu[k] = y[k];
		p.ls[k] = fminf(fmaxf(y[3 + k], NN_LS_MIN), NN_LS_MAX);
	}
	const float *u = y + 6 + 5 * (tl & (NN_MIX - 1));
	const float n = sqrtf(u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + 1e-12f);
#pragma unroll
	for(int j = 0; j < 3; j++) p.dir[j] = u[j] / n;
	p.lk = fminf(fmaxf(u[3], NN_LK_MIN), NN_LK_MAX);
	p.k = expf(p.lk);
	p.lw = u[4] - quad_log_sum_exp(u[4]);
}

__device__ __forceinline__ float prop_logq_lane(const PropLane &p, const float d[3], const float a[3]) {
	float lg = 0.f;
#pragma unroll
	for(int k = 0; k < 3; k++) {
		const float z = (d[k] - p.mu[k]) * expf(-p.ls[k]);
		lg += -0.5f * z * z - p.ls[k] - 0.5f * LOG_2PI;
	}
	const float l = p.lw + log_vmf(p.lk, p.dir[0] * a[0] + p.dir[1] * a[1] + p.dir[2] * a[2]);
	const float mx = fmaxf(fmaxf(fmaxf(fmaxf(-3.0e38f, quad_get<0>(l)), quad_get<1>(l)), quad_get<2>(l)), quad_get<3>(l));
	const float e = expf(l - mx);
	return lg + mx + logf(quad_get<0>(e) + quad_get<1>(e) + quad_get<2>(e) + quad_get<3>(e));
}

// -log q and its gradient with respect to the raw outputs y (g[NN_OUT_PAD])
__device__ inline float prop_loss_grad(const float *y, const float d[3], const float a[3], float *g) {
	Prop p;
	prop_decode(y, p);
	float loss = 0.f;
	for(int k = 0; k < 3; k++) {
		const float s2inv = expf(-2.f * p.ls[k]);
		const float diff = d[k] - p.mu[k];
		const float z2 = diff * diff * s2inv;
		loss += 0.5f * z2 + p.ls[k] + 0.5f * LOG_2PI;
		g[k] = -diff * s2inv;
		g[3 + k] = p.ls_in[k] ? 1.f - z2 : 0.f;
	}
	float l[NN_MIX], cs[NN_MIX], mx = -3.0e38f;
	for(int c = 0; c < NN_MIX; c++) {
		cs[c] = p.dir[c][0] * a[0] + p.dir[c][1] * a[1] + p.dir[c][2] * a[2];
		l[c] = p.lw[c] + log_vmf(p.lk[c], cs[c]);
		mx = fmaxf(mx, l[c]);
	}
	float se = 0.f;
	for(int c = 0; c < NN_MIX; c++) se += expf(l[c] - mx);
	const float lse = mx + logf(se);
	loss -= lse;
	for(int c = 0; c < NN_MIX; c++) {
		const float r = expf(l[c] - lse);  // responsibility
		const float w = expf(p.lw[c]);     // mixture weight
		const float k = expf(p.lk[c]);
		const float kcoth = k * (1.f + expf(-2.f * k)) / (-expm1f(-2.f * k));
		float *gc = g + 6 + 5 * c;
		for(int j = 0; j < 3; j++) gc[j] = -r * k * (a[j] - cs[c] * p.dir[c][j]) / p.nrm[c];
		gc[3] = p.lk_in[c] ? -r * (1.f + k * cs[c] - kcoth) : 0.f;
		gc[4] = w - r;
	}
	for(int e = NN_OUT; e < NN_OUT_PAD; e++) g[e] = 0.f;
	return loss;
}

// ------------------------------------------------------------------------
// descriptor

// Quaternion (x, y, z, w), w >= 0, of the rotation matrix M (rows), from its
// largest component.  The four cases choose operands: one square root and
// three divisions, where lanes of different cases ran them four times.
__device__ inline void quat_of(const double M[9], float q[4]) {
	const double tr = M[0] + M[4] + M[8];
	const bool cw = tr > 0.;
	const bool cx = !cw && M[0] > M[4] && M[0] > M[8];
	const bool cy = !cw && !cx && M[4] > M[8];
	const double d0 = cx ? M[0] : (cy ? M[4] : M[8]);  // its diagonal element, then the others
	const double d1 = cx ? M[4] : M[0];
	const double d2 = cx || cy ? M[8] : M[4];
	const double S = sqrt(cw ? tr + 1. : 1. + d0 - d1 - d2) * 2.;
	const double big = 0.25 * S;
	const double a0 = M[7] - M[5], a1 = M[2] - M[6], a2 = M[3] - M[1];
	const double s01 = M[1] + M[3], s02 = M[2] + M[6], s12 = M[5] + M[7];
	const double e0 = (cw || cx ? a0 : (cy ? s01 : s02)) / S;
	const double e1 = (cw || cy ? a1 : (cx ? s01 : s12)) / S;
	const double e2 = (cw ? a2 : (cx ? s02 : (cy ? s12 : a2))) / S;
	const bool cz = !cw && !cx && !cy;
	const double x = cx ? big : e0, y = cy ? big : e1, z = cz ? big : e2;
	const double w = cw ? big : (cx ? e0 : (cy ? e1 : e2));
	const double sg = w < 0. ? -1. : 1.;
	q[0] = (float) (sg * x);
	q[1] = (float) (sg * y);
	q[2] = (float) (sg * z);
	q[3] = (float) (sg * w);
}

// Descriptor of a particle at (p, O) among n candidate neighbours (pos(i, q)
// and ori(i, Oq) give candidate i): the NN_NB nearest within NN_RCUT (minimum
// image; squared distances compared in single precision, ties by candidate
// order), nearest first, each as its separation in the body frame of O and
// the quaternion of Oq O^T; zero-padded to NN_IN_PAD.  One wavefront per
// particle, in two phases with a workgroup barrier between them:
//   desc_collect: zero the row; the in-range candidates, in candidate order,
//                 into the wave's LDS list (at most DESC_CAND are kept);
//   desc_fill:    each listed candidate's rank by counting; the NN_NB first
//                 write their features.
constexpr int DESC_CAND = 128;

struct DescLds {
	float f[DESC_CAND];  // squared distance of an in-range candidate
	int i[DESC_CAND];    // its candidate index
};

template <int T>
__device__ __forceinline__ void zero_row(__bf16 *row, int tl) {
	for(int e = tl; e < NN_IN_PAD / 8; e += T) *(bf16x8 *) (row + 8 * e) = bf16x8{};
}

// T: lanes per particle (64: a wavefront, 16: a quarter of one); tl = lane % T.
template <int T, class Pos>
__device__ int desc_collect(const double p[3], int n, Pos pos, const double L[3], const double iL[3], DescLds &S,
                            __bf16 *row, int tl) {
	zero_row<T>(row, tl);
	const double rc2 = NN_RCUT * NN_RCUT;
	const int off = (threadIdx.x & 63) & ~(T - 1);
	const unsigned long long tm = T == 64 ? ~0ull : ((1ull << T) - 1ull);
	int nv = 0;
	for(int base = 0; base < n; base += T) {
		const int i = base + tl;
		bool ok = false;
		float f = 0.f;
		if(i < n) {
			double q[3];
			pos(i, q);
			const double dx = kf_min_image(q[0] - p[0], L[0], iL[0]);
			const double dy = kf_min_image(q[1] - p[1], L[1], iL[1]);
			const double dz = kf_min_image(q[2] - p[2], L[2], iL[2]);
			const double r2 = dx * dx + dy * dy + dz * dz;
			ok = r2 < rc2;
			f = (float) r2;
		}
		const unsigned long long m = (__ballot(ok) >> off) & tm;
		const int at = nv + __popcll(m & ((1ull << tl) - 1ull));
		if(ok && at < DESC_CAND) {
			S.f[at] = f;
			S.i[at] = i;
		}
		nv += __popcll(m);
	}
	return nv < DESC_CAND ? nv : DESC_CAND;
}

template <int T, class Pos, class Ori>
__device__ void desc_fill(const double p[3], const double O[9], int nv, Pos pos, Ori ori, const double L[3],
                          const double iL[3], const DescLds &S, __bf16 *row, int tl) {
	for(int e = tl; e < nv; e += T) {
		const float f = S.f[e];
		const int i = S.i[e];
		int rank = 0;
		for(int k = 0; k < nv; k++) {
			const float g = S.f[k];
			rank += (g < f) || (g == f && S.i[k] < i);
		}
		if(rank >= NN_NB) continue;
		double q[3], Oq[9];
		pos(i, q);
		ori(i, Oq);
		double d[3];
		for(int k = 0; k < 3; k++) d[k] = kf_min_image(q[k] - p[k], L[k], iL[k]);
		float v[NN_FEAT];
		for(int k = 0; k < 3; k++) v[k] = (float) (O[3 * k] * d[0] + O[3 * k + 1] * d[1] + O[3 * k + 2] * d[2]);
		double M[9];
		for(int a = 0; a < 3; a++)
			for(int b = 0; b < 3; b++) M[3 * a + b] = Oq[3 * a] * O[3 * b] + Oq[3 * a + 1] * O[3 * b + 1] + Oq[3 * a + 2] * O[3 * b + 2];
		quat_of(M, v + 3);
		for(int k = 0; k < NN_FEAT; k++) row[rank * NN_FEAT + k] = (__bf16) v[k];
	}
}

// ------------------------------------------------------------------------
// the MLP on MFMA (v_mfma_f32_16x16x32_bf16: lane l holds A[l%16][(l/16)*8+i],
// B[(l/16)*8+i][l%16], i < 8, and C[(l/16)*4+j][l%16], j < 4)

__host__ __device__ inline size_t frag_at(int l, int kb, int nt, int lane) {
	return (size_t) nn_woff(l) + ((size_t) (kb * (nn_n(l) / 16) + nt) * 64 + lane) * 8;
}
// fragments of W^T (K' = nn_n(l) rows, N' = nn_k(l) columns)
__host__ __device__ inline size_t fragT_at(int l, int kb, int nt, int lane) {
	return (size_t) nn_woff(l) + ((size_t) (kb * (nn_k(l) / 16) + nt) * 64 + lane) * 8;
}

constexpr int ACT_LD = NN_H + 8;  // LDS row stride of the activations (bf16)

// One row of network inputs as the host gives it, or as the samplers write it
// (NN_IN_PAD BF16 values): 8 consecutive inputs from column c (a multiple of 8).
__device__ __forceinline__ bf16x8 load_inputs(const __bf16 *x, size_t row, int c) {
	return *(const bf16x8 *) (x + row * NN_IN_PAD + c);
}
__device__ __forceinline__ bf16x8 load_inputs(const float *x, size_t row, int c) {
	// (rows of 84 floats: 16-byte aligned, and column 80 has four left)
	static_assert(NN_IN % 4 == 0 && NN_IN_PAD - NN_IN == 12, "whole vectors of four");
	const f32x4 *p = (const f32x4 *) (x + row * NN_IN + c);
	f32x4 lo = {}, hi = {};
	if(c < NN_IN) lo = p[0];
	if(c + 4 < NN_IN) hi = p[1];
	bf16x8 v;
#pragma unroll
	for(int e = 0; e < 4; e++) {
		v[e] = (__bf16) lo[e];
		v[4 + e] = (__bf16) hi[e];
	}
	return v;
}

// One wave per 16 rows: every layer of the MLP, activations in LDS.
// y: [rows][NN_OUT_PAD].
__global__ __launch_bounds__(64) void k_net_fwd(NetDev net, const float *x, int rows, float *y) {
	__shared__ __attribute__((aligned(16))) __bf16 act[2][16 * ACT_LD];
	const int lane = threadIdx.x;
	const int row0 = blockIdx.x * 16;
	if(row0 >= rows) return;
	const int r = lane & 15, g = lane >> 4;
	bf16x8 a0[NN_IN_PAD / 32];
	for(int kb = 0; kb < NN_IN_PAD / 32; kb++) {
		bf16x8 v = {};
		if(row0 + r < rows) v = load_inputs(x, (size_t) (row0 + r), kb * 32 + g * 8);
		a0[kb] = v;
	}
	int cur = 0;
	for(int l = 0; l < NN_LAYERS; l++) {
		const int nkb = nn_k(l) / 32, nnt = nn_n(l) / 16;
		for(int nt = 0; nt < nnt; nt++) {
			f32x4 acc = {0.f, 0.f, 0.f, 0.f};
			for(int kb = 0; kb < nkb; kb++) {
				const bf16x8 a = l == 0 ? a0[kb] : *(const bf16x8 *) (&act[cur][r * ACT_LD + kb * 32 + g * 8]);
				const bf16x8 b = *(const bf16x8 *) (net.frag + frag_at(l, kb, nt, lane));
				acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
			}
			const int col = nt * 16 + r;
			const float bias = net.b[nn_boff(l) + col];
			for(int j = 0; j < 4; j++) {
				const int row = g * 4 + j;
				const float v = acc[j] + bias;
				if(l < NN_LAYERS - 1) act[cur ^ 1][row * ACT_LD + col] = (__bf16) fmaxf(v, 0.f);
				else if(row0 + row < rows)
					y[(size_t) (row0 + row) * NN_OUT_PAD + col] = v;
			}
		}
		__syncthreads();
		cur ^= 1;
	}
}

// ------------------------------------------------------------------------
// gradients of the mean loss
//
// k_net_grad takes rows through the whole network and back and leaves each
// layer's inputs and output gradients for k_net_wgrad, transposed: blocks of
// 32 rows, in a block the 32 values of one column together.  An operand
// fragment of dW = A^T dZ (8 rows of one column per lane) is then one 16-byte
// load and a wavefront's fragment 1 KB in one piece; from row-major arrays it
// took eight 2-byte loads, and the gradients of a batch of 4096 49 us.

// value (row, col) of layer l's inputs / output gradients, m_pad rows in all
__host__ __device__ constexpr int nn_koff(int l) { return l == 0 ? 0 : nn_koff(l - 1) + nn_k(l - 1); }
__device__ __forceinline__ __bf16 *at_ptr(__bf16 *at, int m_pad, int l, int row, int col) {
	return at + (size_t) nn_koff(l) * m_pad + ((size_t) (row >> 5) * nn_k(l) + col) * 32 + (row & 31);
}
__device__ __forceinline__ __bf16 *zt_ptr(__bf16 *zt, int m_pad, int l, int row, int col) {
	return zt + (size_t) nn_boff(l) * m_pad + ((size_t) (row >> 5) * nn_n(l) + col) * 32 + (row & 31);
}

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;

constexpr int NG_ROWS = 16;             // rows of a tile
constexpr int NG_WAVES = NN_H / 16;     // one 16-column tile of a hidden layer per wavefront
constexpr int NG_BLOCKS = 256;          // a workgroup per CU, which takes every NG_BLOCKS-th tile

// -log q of each row, and the gradient of its mean over m rows with respect
// to every layer's output before the activation (BF16, as the MFMA operands
// of the weight gradients); rows in [m, m_pad) have none.  X: float (rows of
// the caller) or __bf16 (samples on the device, padded to m_pad rows).
//
// Bound by the chain of seven layers, not by the matrix cores (a batch of 4096
// is 1.2 GFLOP): each of the 8 wavefronts computes 16 columns of every layer
// with its weights (24 operand fragments, forward and transposed) held in
// registers from the start, so a layer costs its LDS exchange and at most
// four dependent MFMAs.  One kernel instead of three: the activations stay in
// LDS and registers, and ReLU's mask is the wavefront's own columns.
// Forward, loss and backward of 4096 rows: 58 -> 11.3 us (15 on a caller's floats).
template <class X>
__global__ __launch_bounds__(64 * NG_WAVES) void k_net_grad(NetDev net, const X *x, const float *target, int m, int m_pad,
                                                            __bf16 *at, __bf16 *zt, float *loss) {
	__shared__ __attribute__((aligned(16))) __bf16 xs[NG_ROWS * ACT_LD], act[2][NG_ROWS * ACT_LD];
	__shared__ __attribute__((aligned(16))) __bf16 dys[NG_ROWS * (NN_OUT_PAD + 8)];
	__shared__ float ys[NG_ROWS * NN_OUT_PAD];
	constexpr int DY_LD = NN_OUT_PAD + 8;
	const int t = threadIdx.x, lane = t & 63, w = t >> 6, r = lane & 15, g = lane >> 4;
	const int col = w * 16 + r;  // the lane's column of a hidden layer
	// the weights of this wavefront's columns
	bf16x8 f0[3], f1[4], f2[4], f3[4], b3, b2[4], b1[4];
	float bias[4];
#pragma unroll
	for(int kb = 0; kb < 3; kb++) f0[kb] = *(const bf16x8 *) (net.frag + frag_at(0, kb, w, lane));
#pragma unroll
	for(int kb = 0; kb < 4; kb++) {
		f1[kb] = *(const bf16x8 *) (net.frag + frag_at(1, kb, w, lane));
		f2[kb] = *(const bf16x8 *) (net.frag + frag_at(2, kb, w, lane));
		f3[kb] = *(const bf16x8 *) (net.frag + frag_at(3, kb, w & 1, lane));
		b2[kb] = *(const bf16x8 *) (net.fragT + fragT_at(2, kb, w, lane));
		b1[kb] = *(const bf16x8 *) (net.fragT + fragT_at(1, kb, w, lane));
	}
	b3 = *(const bf16x8 *) (net.fragT + fragT_at(3, 0, w, lane));
#pragma unroll
	for(int l = 0; l < 4; l++) bias[l] = net.b[nn_boff(l) + (l < 3 ? col : (w & 1) * 16 + r)];

	for(int row0 = blockIdx.x * NG_ROWS; row0 < m_pad; row0 += gridDim.x * NG_ROWS) {
		// the rows, and their transpose
		constexpr int XV = NN_IN_PAD / 8;
		if(t < NG_ROWS * XV) {
			const int row = t / XV, c = (t % XV) * 8;
			bf16x8 v = {};
			if(row0 + row < m) v = load_inputs(x, (size_t) (row0 + row), c);
			*(bf16x8 *) (xs + row * ACT_LD + c) = v;
		}
		__syncthreads();
		if(t < 2 * NN_IN_PAD) {
			const int c = t % NN_IN_PAD, h = t / NN_IN_PAD * 8;
			bf16x8 v;
#pragma unroll
			for(int e = 0; e < 8; e++) v[e] = xs[(h + e) * ACT_LD + c];
			*(bf16x8 *) at_ptr(at, m_pad, 0, row0 + h, c) = v;
		}
		// forward; the lane's values of hidden layer l + 1 in hv[l]
		bf16x4 hv[3];
		auto forward = [&](const __bf16 *A, const bf16x8 *f, int nkb, float b, f32x4 &out) {
			f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
			for(int kb = 0; kb < nkb; kb++) {
				const bf16x8 a = *(const bf16x8 *) (A + r * ACT_LD + kb * 32 + g * 8);
				acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, f[kb], acc, 0, 0, 0);
			}
#pragma unroll
			for(int j = 0; j < 4; j++) out[j] = acc[j] + b;
		};
		auto hidden = [&](const f32x4 &v, int l, __bf16 *to) {
#pragma unroll
			for(int j = 0; j < 4; j++) {
				hv[l][j] = (__bf16) fmaxf(v[j], 0.f);
				to[(g * 4 + j) * ACT_LD + col] = hv[l][j];
			}
			*(bf16x4 *) at_ptr(at, m_pad, l + 1, row0 + g * 4, col) = hv[l];
			__syncthreads();
		};
		f32x4 v;
		forward(xs, f0, 3, bias[0], v);
		hidden(v, 0, act[0]);
		forward(act[0], f1, 4, bias[1], v);
		hidden(v, 1, act[1]);
		forward(act[1], f2, 4, bias[2], v);
		hidden(v, 2, act[0]);
		if(w < NN_OUT_PAD / 16) {
			forward(act[0], f3, 4, bias[3], v);
#pragma unroll
			for(int j = 0; j < 4; j++) ys[(g * 4 + j) * NN_OUT_PAD + col] = v[j];
		}
		__syncthreads();
		// the loss and its gradient with respect to the outputs, a row per lane
		if(t < NG_ROWS) {
			const int i = row0 + t;
			float gr[NN_OUT_PAD], l = 0.f;
			if(i < m) {
				const float *tg = target + (size_t) i * 6;
				l = prop_loss_grad(ys + t * NN_OUT_PAD, tg, tg + 3, gr);
#pragma unroll
				for(int e = 0; e < NN_OUT_PAD; e++) gr[e] *= 1.f / (float) m;
			}
			else
#pragma unroll
				for(int e = 0; e < NN_OUT_PAD; e++) gr[e] = 0.f;
#pragma unroll
			for(int e = 0; e < NN_OUT_PAD; e++) dys[t * DY_LD + e] = (__bf16) gr[e];
			loss[i] = l;
		}
		__syncthreads();
		if(t < 2 * NN_OUT_PAD) {
			const int c = t % NN_OUT_PAD, h = t / NN_OUT_PAD * 8;
			bf16x8 o;
#pragma unroll
			for(int e = 0; e < 8; e++) o[e] = dys[(h + e) * DY_LD + c];
			*(bf16x8 *) zt_ptr(zt, m_pad, 3, row0 + h, c) = o;
		}
		// backward: dH3 = (dY W4^T) * [H3 > 0], then dH2, dH1
		auto masked = [&](const f32x4 &acc, int l, __bf16 *to) {
			bf16x4 z;
#pragma unroll
			for(int j = 0; j < 4; j++) {
				z[j] = (__bf16) (acc[j] * ((float) hv[l][j] > 0.f ? 1.f : 0.f));
				if(to) to[(g * 4 + j) * ACT_LD + col] = z[j];
			}
			*(bf16x4 *) zt_ptr(zt, m_pad, l, row0 + g * 4, col) = z;
			__syncthreads();
		};
		{
			const bf16x8 a = *(const bf16x8 *) (dys + r * DY_LD + g * 8);
			const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
			v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b3, zero, 0, 0, 0);
		}
		masked(v, 2, act[1]);
		forward(act[1], b2, 4, 0.f, v);
		masked(v, 1, act[0]);
		forward(act[0], b1, 4, 0.f, v);
		masked(v, 0, nullptr);
	}
}

// Weight and bias gradients: dW_l = A_l^T dZ_l and the column sums of dZ_l.
// A wavefront takes a 32 x 32 tile of one layer over one slice of the rows
// (two fragments of either operand for four MFMAs) and leaves partial sums:
// part[slice][NN_W + NN_B].  The 48 tiles alone would leave the chip idle, so
// the rows are cut into slices of at least NW_ROWS (a chain of 8 blocks), at
// most NW_SLICES of them, whose sums the next kernel adds in a fixed order.
// The bias sums are one MFMA with a matrix of ones, stored by the tiles of
// the first rows.  Batch of 4096: 49 + 11 us (a tile over all rows; the biases in
// a kernel of their own) -> 5.9 us.
constexpr int NW_ROWS = 256, NW_SLICES = 32;
constexpr int nw_tiles(int l) { return l < 0 ? 0 : nw_tiles(l - 1) + (nn_k(l) / 32) * (nn_n(l) / 32); }
constexpr int NW_TILES = nw_tiles(NN_LAYERS - 1);
constexpr int NW_WAVES = 4;
static_assert(NW_TILES % NW_WAVES == 0, "whole workgroups");
constexpr int NN_G = NN_W + NN_B;

int net_grad_slices(int m_pad) { return std::max(1, std::min(m_pad / NW_ROWS, NW_SLICES)); }

__global__ __launch_bounds__(64 * NW_WAVES) void k_net_wgrad(const __bf16 *at, const __bf16 *zt, int m_pad, float *part) {
	int t = blockIdx.x * NW_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = 0;
	while(t >= (nn_k(l) / 32) * (nn_n(l) / 32)) {
		t -= (nn_k(l) / 32) * (nn_n(l) / 32);
		l++;
	}
	const int K = nn_k(l), N = nn_n(l);
	const int k0 = t / (N / 32) * 32, n0 = t % (N / 32) * 32;
	const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
	const __bf16 *A = at + (size_t) nn_koff(l) * m_pad + (k0 + r) * 32 + g * 8;
	const __bf16 *Z = zt + (size_t) nn_boff(l) * m_pad + (n0 + r) * 32 + g * 8;
	const int blocks = m_pad / 32, S = gridDim.y, s = blockIdx.y;
	const int lo = (int) ((long long) blocks * s / S), hi = (int) ((long long) blocks * (s + 1) / S);
	f32x4 acc[2][2] = {}, sum[2] = {};
	bf16x8 ones;
#pragma unroll
	for(int e = 0; e < 8; e++) ones[e] = (__bf16) 1.f;
	for(int b = lo; b < hi; b++) {
		const __bf16 *pa = A + (size_t) b * K * 32, *pz = Z + (size_t) b * N * 32;
		const bf16x8 a0 = *(const bf16x8 *) pa, a1 = *(const bf16x8 *) (pa + 512);
		const bf16x8 z0 = *(const bf16x8 *) pz, z1 = *(const bf16x8 *) (pz + 512);
		acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, z0, acc[0][0], 0, 0, 0);
		acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, z1, acc[0][1], 0, 0, 0);
		acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, z0, acc[1][0], 0, 0, 0);
		acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, z1, acc[1][1], 0, 0, 0);
		sum[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, z0, sum[0], 0, 0, 0);
		sum[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, z1, sum[1], 0, 0, 0);
	}
	float *gw = part + (size_t) s * NN_G + nn_woff(l), *gb = part + (size_t) s * NN_G + NN_W + nn_boff(l);
#pragma unroll
	for(int i = 0; i < 2; i++)
#pragma unroll
		for(int c = 0; c < 2; c++)
#pragma unroll
			for(int j = 0; j < 4; j++) gw[(size_t) (k0 + i * 16 + g * 4 + j) * N + n0 + c * 16 + r] = acc[i][c][j];
	// (every row of the product with ones holds the column sums)
	if(k0 == 0 && g == 0) {
		gb[n0 + r] = sum[0][0];
		gb[n0 + 16 + r] = sum[1][0];
	}
}

// gradient e of the slices' partial sums (e < NN_W: a weight, else a bias)
__device__ __forceinline__ float slice_sum(const float *part, int slices, int e) {
	float g = 0.f;
	for(int s = 0; s < slices; s++) g += part[(size_t) s * NN_G + e];
	return g;
}

__global__ void k_net_reduce(const float *part, int slices, float *out) {
	const int e = blockIdx.x * blockDim.x + threadIdx.x;
	if(e < NN_G) out[e] = slice_sum(part, slices, e);
}

// BF16 operand fragments of W (forward) and W^T (backward): those of weight e.
__device__ __forceinline__ void pack_weight(const NetDev &net, int e, float w) {
	int l = 0;
	while(l + 1 < NN_LAYERS && e >= nn_woff(l + 1)) l++;
	const int loc = e - nn_woff(l), N = nn_n(l);
	const int k = loc / N, n = loc % N;
	const __bf16 v = (__bf16) w;
	net.frag[frag_at(l, k / 32, n / 16, ((k % 32) / 8) * 16 + n % 16) + k % 8] = v;
	net.fragT[fragT_at(l, n / 32, k / 16, ((n % 32) / 8) * 16 + k % 16) + n % 8] = v;
}

__global__ void k_net_pack(NetDev net) {
	const int e = blockIdx.x * blockDim.x + threadIdx.x;
	if(e < NN_W) pack_weight(net, e, net.w[e]);
}

// Adam (Kingma & Ba) on every weight and bias, from the gradients' partial
// sums; step t >= 1.  Leaves the operand fragments of the new weights.
__global__ void k_net_adam(NetDev net, const float *part, int slices, int t, float lr) {
	const int e = blockIdx.x * blockDim.x + threadIdx.x;
	if(e >= NN_G) return;
	const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
	const bool isw = e < NN_W;
	const int i = isw ? e : e - NN_W;
	float *w = isw ? net.w : net.b, *m = isw ? net.mw : net.mb, *v = isw ? net.vw : net.vb;
	const float g = slice_sum(part, slices, e);
	m[i] = b1 * m[i] + (1.f - b1) * g;
	v[i] = b2 * v[i] + (1.f - b2) * g * g;
	const float mh = m[i] / (1.f - powf(b1, (float) t)), vh = v[i] / (1.f - powf(b2, (float) t));
	const float nw = w[i] - lr * mh / (sqrtf(vh) + eps);
	w[i] = nw;
	if(isw) pack_weight(net, e, nw);
}

void launch_net_forward(const NetDev &net, const float *x, int m, float *y, hipStream_t s) {
	const int blocks = (m + 15) / 16;
	if(blocks > 0) hipLaunchKernelGGL(k_net_fwd, dim3(blocks), dim3(64), 0, s, net, x, m, y);
}

void launch_net_pack(const NetDev &net, hipStream_t s) {
	hipLaunchKernelGGL(k_net_pack, dim3((NN_W + 255) / 256), dim3(256), 0, s, net);
}

template <class X>
static void net_grad(const NetDev &net, const X *x, const float *target, int m, const NetScratch &q, hipStream_t s) {
	const int m_pad = (m + 31) & ~31;
	hipLaunchKernelGGL(k_net_grad<X>, dim3(std::min(m_pad / NG_ROWS, NG_BLOCKS)), dim3(64 * NG_WAVES), 0, s, net, x, target,
	                   m, m_pad, q.at, q.zt, q.loss);
	hipLaunchKernelGGL(k_net_wgrad, dim3(NW_TILES / NW_WAVES, net_grad_slices(m_pad)), dim3(64 * NW_WAVES), 0, s,
	                   (const __bf16 *) q.at, (const __bf16 *) q.zt, m_pad, q.part);
}

void launch_net_loss_grad(const NetDev &net, const float *x, const float *target, int m, const NetScratch &q, float *out,
                          hipStream_t s) {
	net_grad(net, x, target, m, q, s);
	hipLaunchKernelGGL(k_net_reduce, dim3((NN_G + 255) / 256), dim3(256), 0, s, (const float *) q.part,
	                   net_grad_slices((m + 31) & ~31), out);
}

void launch_net_train(const NetDev &net, const __bf16 *x, const float *target, int m, const NetScratch &q, hipStream_t s) {
	net_grad(net, x, target, m, q, s);
}

void launch_net_adam(const NetDev &net, int m, const NetScratch &q, int step, float lr, hipStream_t s) {
	hipLaunchKernelGGL(k_net_adam, dim3((NN_G + 255) / 256), dim3(256), 0, s, net, (const float *) q.part,
	                   net_grad_slices((m + 31) & ~31), step, lr);
}

// ------------------------------------------------------------------------
// random draws of a learned move

__device__ inline void gauss2(uint32_t u1, uint32_t u2, double &z0, double &z1) {
	const double a = (u1 + 0.5) * 2.3283064365386962890625e-10;  // (0, 1)
	const double b = u01(u2);
	const double rr = sqrt(-2. * log(a));
	double sn, cs;
	sincos(6.283185307179586 * b, &sn, &cs);
	z0 = rr * cs;
	z1 = rr * sn;
}

// Single-precision draws of a learned move.  The move applied is the one the
// density is evaluated at (body-frame displacement and axis as floats), so
// the precision of the transforms only shapes the proposal, not the
// acceptance rule.

// Wood 1994's cosine to the mean of a vMF sample (inverse CDF), and the sample
// from it and the azimuth's sine and cosine.
__device__ inline void vmf_sample(const float mu[3], float kappa, float u1, float sn, float cs, float out[3]) {
	float w;
	if(kappa < 1e-4f) w = 2.f * u1 - 1.f;
	else w = 1.f + logf(expf(-2.f * kappa) + u1 * (-expm1f(-2.f * kappa))) / kappa;
	w = fminf(1.f, fmaxf(-1.f, w));
	// an orthonormal pair perpendicular to mu
	float e1[3];
	if(fabsf(mu[0]) < 0.9f) e1[0] = 0.f, e1[1] = -mu[2], e1[2] = mu[1];
	else e1[0] = mu[2], e1[1] = 0.f, e1[2] = -mu[0];
	const float n1 = sqrtf(e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2]);
	for(int k = 0; k < 3; k++) e1[k] /= n1;
	const float e2[3] = {mu[1] * e1[2] - mu[2] * e1[1], mu[2] * e1[0] - mu[0] * e1[2], mu[0] * e1[1] - mu[1] * e1[0]};
	const float sw = sqrtf(fmaxf(0.f, 1.f - w * w));
	for(int k = 0; k < 3; k++) out[k] = w * mu[k] + sw * (cs * e1[k] + sn * e2[k]);
	const float no = sqrtf(out[0] * out[0] + out[1] * out[1] + out[2] * out[2]);
	for(int k = 0; k < 3; k++) out[k] /= no;
}

__device__ inline float u01f(uint32_t u) { return (float) (u >> 8) * 5.9604644775390625e-8f; }  // [0, 1)

// ------------------------------------------------------------------------
// the learned colour pass: one move per non-empty cell of the pass's list

struct CellView {
	const int *rec;
	int M, s0, cnt, cloc, r, sel;
};

__device__ inline CellView cell_view(const DevState &d, int pass, int gi) {
	CellView v;
	v.rec = d.rec + ((size_t) pass * d.total_act + gi) * REC_W;
	v.M = v.rec[REC_M];
	v.s0 = v.rec[REC_S0];
	v.cnt = v.rec[REC_CNT];
	v.cloc = v.rec[REC_CELL];
	v.r = v.rec[REC_REP];
	v.sel = v.rec[REC_SEL];
	return v;
}

// Candidates of one wave's cell, staged in LDS: their slots and positions
// (the first CAND_MAX; the rest are read from the record and global memory).
constexpr int CAND_MAX = 64;
struct CandLds {
	double x[CAND_MAX], y[CAND_MAX], z[CAND_MAX];
	int slot[CAND_MAX];
	int rec[REC_W];  // the cell's record
};

// candidate neighbours of the moving slot j: the cell's static neighbours and
// the other members of the cell
struct Cands {
	const DevState &d;
	const double *F;
	CellView v;
	int j;
	const CandLds *L = nullptr;  // staged slots / positions (filled by stage())
	__device__ int count() const { return v.M + v.cnt - 1; }
	__device__ int slot_of(int i) const {
		if(i < v.M) return rec_slot(d, L ? L->rec : v.rec, i);
		const int o = v.s0 + (i - v.M);
		return o < j ? o : o + 1;
	}
	__device__ int slot(int i) const { return (L && i < CAND_MAX) ? L->slot[i] : slot_of(i); }
	__device__ void pos(int i, double q[3]) const {
		if(L && i < CAND_MAX) {
			q[0] = L->x[i];
			q[1] = L->y[i];
			q[2] = L->z[i];
			return;
		}
		const int s = slot_of(i);
		for(int k = 0; k < 3; k++) q[k] = part(F, s)[k];
	}
	// lane-strided: candidate i is staged by lane i % T of the team, the
	// lane that reads it first (desc_collect, the energy loop)
	template <int T>
	__device__ void stage(CandLds &W, int tl) const {
		for(int i = tl; i < count() && i < CAND_MAX; i += T) {
			const int s = slot_of(i);
			W.slot[i] = s;
			W.x[i] = part(F, s)[0];
			W.y[i] = part(F, s)[1];
			W.z[i] = part(F, s)[2];
		}
	}
	__device__ void ori(int i, double O[9]) const {
		const int s = slot(i);
		for(int k = 0; k < 9; k++) O[k] = part(F, s)[3 + k];
	}
};

constexpr int PROP_W = 16;         // one drawn proposal: p'[3], O'[9], log q forward, axis[3]
constexpr int LP_ROWS = 16;        // rows of the MFMA tile = cells of one workgroup
constexpr int LP_TEAM = 16;        // lanes per cell: four cells per wavefront
constexpr int LP_WAVES = LP_ROWS * LP_TEAM / 64;

// LDS of one learned-pass workgroup
struct LpLds {
	__bf16 x[LP_ROWS * ACT_LD];       // descriptors
	__bf16 act[2][LP_ROWS * ACT_LD];  // hidden activations
	float y[LP_ROWS * NN_OUT_PAD];    // network outputs
	DescLds desc[LP_ROWS];
	double prop[LP_ROWS][PROP_W];     // the drawn proposal of each cell
	double cur[LP_ROWS][NCOMP];       // the moving particle
	CandLds cand[LP_ROWS];
};

// The operand fragments and biases of a wavefront's columns of one layer:
// 16-column tiles w and w + LP_WAVES, as far as the layer has them.
constexpr int LP_TILES = NN_H / 16 / LP_WAVES;
struct LayerOps {
	bf16x8 f[LP_TILES][NN_H / 32];
	float bias[LP_TILES];
};
template <int l>
__device__ __forceinline__ void load_ops(const NetDev &net, int wave, int lane, LayerOps &o) {
#pragma unroll
	for(int u = 0; u < LP_TILES; u++) {
		const int nt = wave + u * LP_WAVES;
		if(nt >= nn_n(l) / 16) return;
#pragma unroll
		for(int kb = 0; kb < nn_k(l) / 32; kb++) o.f[u][kb] = *(const bf16x8 *) (net.frag + frag_at(l, kb, nt, lane));
		o.bias[u] = net.b[nn_boff(l) + nt * 16 + (lane & 15)];
	}
}

// Layer l on the workgroup's 16 rows, A -> S.act / S.y, and a barrier.
template <int l>
__device__ __forceinline__ void lp_layer(LpLds &S, int wave, int lane, const LayerOps &o) {
	const int r = lane & 15, g = lane >> 4;
	const __bf16 *A = l == 0 ? S.x : S.act[l & 1];
	bf16x8 a[nn_k(l) / 32];
#pragma unroll
	for(int kb = 0; kb < nn_k(l) / 32; kb++) a[kb] = *(const bf16x8 *) (A + r * ACT_LD + kb * 32 + g * 8);
#pragma unroll
	for(int u = 0; u < LP_TILES; u++) {
		const int nt = wave + u * LP_WAVES, col = nt * 16 + r;
		if(nt >= nn_n(l) / 16) break;
		f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for(int kb = 0; kb < nn_k(l) / 32; kb++)
			acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kb], o.f[u][kb], acc, 0, 0, 0);
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const int row = g * 4 + j;
			const float v = acc[j] + o.bias[u];
			if constexpr(l < NN_LAYERS - 1) S.act[(l & 1) ^ 1][row * ACT_LD + col] = (__bf16) fmaxf(v, 0.f);
			else S.y[row * NN_OUT_PAD + col] = v;
		}
	}
	__syncthreads();
}

// The network on the workgroup's 16 rows, S.x -> S.y, after a barrier.  The
// weights come from L2 two layers ahead, so that a layer waits for LDS and
// MFMAs only.
__device__ __forceinline__ void lp_forward(const NetDev &net, LpLds &S, int wave, int lane) {
	static_assert(LP_TILES * LP_WAVES * 16 == NN_H && NN_LAYERS == 4, "whole column tiles per wavefront");
	LayerOps o0, o1, o2, o3;
	load_ops<0>(net, wave, lane, o0);
	load_ops<1>(net, wave, lane, o1);
	__syncthreads();
	load_ops<2>(net, wave, lane, o2);
	lp_layer<0>(S, wave, lane, o0);
	load_ops<3>(net, wave, lane, o3);
	lp_layer<1>(S, wave, lane, o1);
	lp_layer<2>(S, wave, lane, o2);
	lp_layer<3>(S, wave, lane, o3);
}

// The whole learned pass in one kernel: a workgroup takes 16 cells of the
// pass's list (the rows of one MFMA tile), 16 lanes per cell:
//   A  pick the moving member (uniform by rank of particle index, as the plain
//      pass), descriptor of the current state;      network forward (MFMA)
//   B  draw the proposal from the outputs; a move that leaves the cell is
//      rejected; descriptor of the proposed state;  network forward (MFMA)
//   C  reverse density, Kern-Frenkel energy change over the cell's
//      candidates (the reference's pair test), Metropolis-Hastings.
// Bound by instruction issue: a wavefront runs some 8000 instructions, most
// of them FP64 or the densities' transcendentals, whatever the share of its
// lanes that have a candidate.  With 32 lanes per cell (about 10 candidates
// within reach) and 95 KB of LDS, N=65536 at rho 0.3 was 409 workgroups on
// 256 CUs in two rounds, 55 us.  16 lanes and 67 KB halve the instructions
// and let every workgroup run at once; the mixture's components are one per
// lane; code that rarely runs (slots past a record's list) is no longer
// unrolled into every use, since the kernel exceeds the instruction cache.
// The Gaussian pairs and the axis' azimuth are likewise one draw per lane, and
// the weights come two layers ahead.  24.8 us.  (32 lanes in 128 registers, two
// workgroups per CU: 60 us, spills.)
__global__ __launch_bounds__(64 * LP_WAVES, 2) void k_learn_pass(DevState d, NetDev net, uint64_t sweep, int pass) {
	__shared__ __attribute__((aligned(16))) LpLds S;
	constexpr int T = LP_TEAM;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int tl = lane & (T - 1), cell = threadIdx.x / T;
	const int g0 = blockIdx.x * LP_ROWS;
	const int gi = g0 + cell;
	// a record of another sweep lies past the end of the pass's list (no read
	// of its length first); the whole workgroup leaves before any barrier
	const int *recs = d.rec + (size_t) pass * d.total_act * REC_W;
	const bool any = recs[(size_t) g0 * REC_W + REC_TAG] == (int) d.rec_tag;
	bool live = gi < d.total_act && recs[(size_t) min(gi, d.total_act - 1) * REC_W + REC_TAG] == (int) d.rec_tag;
	if(!any) return;
	CellView v{};
	const double *F = nullptr;
	int j = 0, nv = 0;
	__bf16 *row = S.x + cell * ACT_LD;
	DescLds &D = S.desc[cell];
	CandLds &CL = S.cand[cell];
	double *cur = S.cur[cell];
	double L[3], iL[3];
	if(live) {
		v = cell_view(d, pass, gi);
		// a cell of more members than the passes work on is not moved and is
		// reported; its threads stay for the barriers below
		if(v.cnt > CELL_CAP) {
			if(tl == 0) atomicOr(d.err, (int) ERR_CELL_CAP);
			live = false;
		}
		else
			for(int e = tl; e < REC_W / 4; e += T) ((int4 *) CL.rec)[e] = ((const int4 *) v.rec)[e];
	}
	__syncthreads();

	// ---- A
	if(live) {
		const Rep &rp = d.reps[v.r];
		for(int k = 0; k < 3; k++) {
			L[k] = rp.g.box[k];
			iL[k] = rp.g.inv_box[k];
		}
		F = pick_buf(d.f, v.sel);
		const int *PID = pick_buf(d.pid, v.sel);
		const u32x4 ra = rng(d.seed, v.r, sweep, (uint32_t) v.cloc, TAG_LEARN_A, (uint32_t) pass, 0);
		const int target = (int) __umulhi(ra.x, (uint32_t) v.cnt);
		const int me = tl < v.cnt ? PID[v.s0 + tl] : 0;
		for(int m0 = 0; m0 < v.cnt; m0 += T) {
			// (few cells hold more members than the team has lanes)
			const int id = m0 == 0 ? me : (m0 + tl < v.cnt ? PID[v.s0 + m0 + tl] : 0);
			int rk = 0;
			for(int b = 0; b < v.cnt; b++) rk += (b < T ? __shfl(me, (lane & ~(T - 1)) + b) : PID[v.s0 + b]) < id;
			const bool hit = m0 + tl < v.cnt && rk == target;
			const unsigned long long hm = (__ballot(hit) >> (lane & ~(T - 1))) & ((1ull << T) - 1ull);
			if(hm) j = v.s0 + m0 + (int) __builtin_ctzll(hm);
		}
		if(tl < NCOMP) cur[tl] = part(F, j)[tl];
		const Cands c{d, F, v, j, &CL};
		c.stage<T>(CL, tl);
		team_sync();
		double p[3];
		for(int k = 0; k < 3; k++) p[k] = cur[k];
		nv = desc_collect<T>(p, c.count(), [&](int i, double q[3]) { c.pos(i, q); }, L, iL, D, row, tl);
	}
	else
		zero_row<T>(row, tl);
	__syncthreads();
	if(live) {
		const Cands c{d, F, v, j, &CL};
		double p[3], O[9];
		for(int k = 0; k < 3; k++) p[k] = cur[k];
		for(int k = 0; k < 9; k++) O[k] = cur[3 + k];
		desc_fill<T>(
			p, O, nv, [&](int i, double q[3]) { c.pos(i, q); }, [&](int i, double Oq[9]) { c.ori(i, Oq); }, L, iL, D, row,
			tl);
	}
	lp_forward(net, S, wave, lane);

	// ---- B
	bool inside = false;
	if(live) {
		const Rep &rp = d.reps[v.r];
		PropLane pr;
		prop_decode_lane(S.y + cell * NN_OUT_PAD, tl, pr);
		const u32x4 ra = rng(d.seed, v.r, sweep, (uint32_t) v.cloc, TAG_LEARN_A, (uint32_t) pass, 1);
		const u32x4 rb = rng(d.seed, v.r, sweep, (uint32_t) v.cloc, TAG_LEARN_B, (uint32_t) pass, 0);
		// the Gaussian pairs (Box-Muller) by lanes 0 and 1 of each quad, the
		// azimuth of the axis by lane 2: one logarithm and one sine and cosine
		const int ql = tl & 3;
		const uint32_t ub = ql == 0 ? ra.y : (ql == 1 ? ra.w : rb.z);
		float sn, cs;
		sincosf(6.2831853f * u01f(ub), &sn, &cs);
		const float rr = sqrtf(-2.f * logf(((float) ((ql == 0 ? ra.x : ra.z) >> 8) + 0.5f) * 5.9604644775390625e-8f));
		const float z[3] = {quad_get<0>(rr * cs), quad_get<0>(rr * sn), quad_get<1>(rr * cs)};
		float dbody[3];
		for(int k = 0; k < 3; k++) dbody[k] = pr.mu[k] + expf(pr.ls[k]) * z[k];
		// mixture component by its weight, then the axis
		const float uc = u01f(rb.x), wc = expf(pr.lw);
		const float c0 = quad_get<0>(wc), c1 = c0 + quad_get<1>(wc), c2 = c1 + quad_get<2>(wc);
		const int comp = uc < c0 ? 0 : (uc < c1 ? 1 : (uc < c2 ? 2 : 3)), from = (lane & ~(NN_MIX - 1)) + comp;
		float dir[3];
		for(int k = 0; k < 3; k++) dir[k] = __shfl(pr.dir[k], from);
		const float kap = __shfl(pr.k, from);
		float axf[3];
		vmf_sample(dir, kap, u01f(rb.y), quad_get<2>(sn), quad_get<2>(cs), axf);
		const double ang = u01(rb.w) * d.learn.theta_max;
		double p[3], O[9];
		for(int k = 0; k < 3; k++) p[k] = cur[k];
		for(int k = 0; k < 9; k++) O[k] = cur[3 + k];
		// body -> lab: O^T d; O' = O R(a, angle) (utils.c:186-209)
		double np[3];
		for(int k = 0; k < 3; k++) np[k] = p[k] + (O[k] * dbody[0] + O[3 + k] * dbody[1] + O[6 + k] * dbody[2]);
		const double axd[3] = {axf[0], axf[1], axf[2]};
		double st, ct, R[9], On[9];
		sincos(ang, &st, &ct);
		rotation_matrix(axd, st, ct, R);
		mat_mul3(O, R, On);
		double *out = S.prop[cell];
		const float logq = prop_logq_lane(pr, dbody, axf);
		if(tl == 0) {
			for(int k = 0; k < 3; k++) out[k] = np[k];
			for(int k = 0; k < 9; k++) out[3 + k] = On[k];
			out[12] = logq;
			for(int k = 0; k < 3; k++) out[13 + k] = axd[k];
		}
		const int n0 = rp.g.n[0], n1 = rp.g.n[1], n2 = rp.g.n[2];
		const int ix = v.cloc / (n1 * n2), iy = (v.cloc / n2) % n1, iz = v.cloc % n2;
		inside = cell_coord(np[0], rp.g.shift[0], rp.g.inv_box[0], n0) == ix &&
		         cell_coord(np[1], rp.g.shift[1], rp.g.inv_box[1], n1) == iy &&
		         cell_coord(np[2], rp.g.shift[2], rp.g.inv_box[2], n2) == iz;
		if(inside) {
			const Cands c{d, F, v, j, &CL};
			nv = desc_collect<T>(np, c.count(), [&](int i, double q[3]) { c.pos(i, q); }, L, iL, D, row, tl);
		}
	}
	__syncthreads();
	if(live && inside) {
		const Cands c{d, F, v, j, &CL};
		const double *pp = S.prop[cell];
		double np[3], On[9];
		for(int k = 0; k < 3; k++) np[k] = pp[k];
		for(int k = 0; k < 9; k++) On[k] = pp[3 + k];
		desc_fill<T>(
			np, On, nv, [&](int i, double q[3]) { c.pos(i, q); }, [&](int i, double Oq[9]) { c.ori(i, Oq); }, L, iL, D, row,
			tl);
	}
	lp_forward(net, S, wave, lane);

	// ---- C (no barrier below: teams leave independently)
	if(!live) return;
	const int cslot = gi & (NSLOT - 1);
	if(tl == 0) {
		atomicAdd(ctr_at(d.ctr, v.r, C_TRY_ROTO, cslot), 1ull);
		atomicAdd(ctr_at(d.ctr, v.r, C_TRY_LEARN, cslot), 1ull);
	}
	if(!inside) return;
	const Rep &rp = d.reps[v.r];
	double *Fw = pick_buf(d.f, v.sel);
	const double *pp = S.prop[cell];
	double p[3], O[9], np[3], On[9];
	for(int k = 0; k < 3; k++) p[k] = cur[k];
	for(int k = 0; k < 9; k++) O[k] = cur[3 + k];
	for(int k = 0; k < 3; k++) np[k] = pp[k];
	for(int k = 0; k < 9; k++) On[k] = pp[3 + k];
	// reverse: displacement p - p' in the body frame of O', axis -a
	float rbody[3];
	for(int k = 0; k < 3; k++)
		rbody[k] = (float) (On[3 * k] * (p[0] - np[0]) + On[3 * k + 1] * (p[1] - np[1]) + On[3 * k + 2] * (p[2] - np[2]));
	const float rax[3] = {(float) -pp[13], (float) -pp[14], (float) -pp[15]};
	PropLane pr;
	prop_decode_lane(S.y + cell * NN_OUT_PAD, tl, pr);
	const double log_ratio = (double) prop_logq_lane(pr, rbody, rax) - pp[12];
	// energy change over the static neighbours and the other members, one
	// candidate per lane of the team
	Trial t;
	t.px = p[0];
	t.py = p[1];
	t.pz = p[2];
	t.nx = np[0];
	t.ny = np[1];
	t.nz = np[2];
	t.Lx = L[0];
	t.Ly = L[1];
	t.Lz = L[2];
	t.iLx = iL[0];
	t.iLy = iL[1];
	t.iLz = iL[2];
	t.rc2 = rp.rc2;
	t.cosmax = rp.cosmax;
	double Po[4][3], Pn[4][3];
	kf_patches(O, Po);
	kf_patches(On, Pn);
	const Cands c{d, Fw, v, j, &CL};
	const int n = c.count();
	int bo = 0, bn = 0;
	bool ov = false;
	for(int base = 0; base < n; base += T) {
		const int i = base + tl;
		if(i < n && !ov) {
			double q[3];
			c.pos(i, q);
			if(overlaps_new(t, q[0], q[1], q[2])) ov = true;
			else bonds_old_new_exact(t, &Po[0][0], &Pn[0][0], q[0], q[1], q[2], [&](double *Oq) { c.ori(i, Oq); }, bo, bn);
		}
		if(team_any<T>(ov)) break;
	}
	if(team_any<T>(ov)) return;
	const int db = team_sum<T>(bn) - team_sum<T>(bo);
	if(tl != 0) return;
	const double dE = (double) (-db);
	const u32x4 rc = rng(d.seed, v.r, sweep, (uint32_t) v.cloc, TAG_LEARN_B, (uint32_t) pass, 1);
	const double la = -dE / rp.T + log_ratio;
	if(la >= 0. || u01(rc.x) < exp(la)) {
		for(int k = 0; k < 3; k++) part(Fw, j)[k] = np[k];
		for(int k = 0; k < 9; k++) part(Fw, j)[3 + k] = On[k];
		atomicAdd(ctr_at(d.ctr, v.r, C_ACC_ROTO, cslot), 1ull);
		atomicAdd(ctr_at(d.ctr, v.r, C_ACC_LEARN, cslot), 1ull);
		if(db) atomicAdd(ctr_at(d.ctr, v.r, C_DBONDS, cslot), (unsigned long long) (long long) db);
	}
}

void launch_learned_pass(const DevState &d, const NetDev &net, uint64_t sweep, int pass, hipStream_t s) {
	const unsigned g = (unsigned) ((d.total_act + LP_ROWS - 1) / LP_ROWS);
	if(g > 0) hipLaunchKernelGGL(k_learn_pass, dim3(g), dim3(64 * LP_WAVES), 0, s, d, net, sweep, pass);
}

// Descriptors of particles idx[t] of a plain configuration, every other
// particle a candidate (the C ABI's pp_net_descriptor); one wave per particle.
__global__ __launch_bounds__(64) void k_descriptor(int n, const double *r, const double *O, Grid g, int m,
                                                   const int *idx, __bf16 *x) {
	__shared__ DescLds D;
	const int t = blockIdx.x, lane = threadIdx.x;
	if(t >= m) return;
	const int i = idx[t];
	double p[3], Oi[9];
	for(int k = 0; k < 3; k++) p[k] = r[3 * (size_t) i + k];
	for(int k = 0; k < 9; k++) Oi[k] = O[9 * (size_t) i + k];
	auto other = [&](int c) { return c < i ? c : c + 1; };
	auto pos = [&](int c, double q[3]) {
		for(int k = 0; k < 3; k++) q[k] = r[3 * (size_t) other(c) + k];
	};
	auto ori = [&](int c, double Oq[9]) {
		for(int k = 0; k < 9; k++) Oq[k] = O[9 * (size_t) other(c) + k];
	};
	__bf16 *row = x + (size_t) t * NN_IN_PAD;
	const int nv = desc_collect<64>(p, n - 1, pos, g.box, g.inv_box, D, row, lane);
	__syncthreads();
	desc_fill<64>(p, Oi, nv, pos, ori, g.box, g.inv_box, D, row, lane);
}

void launch_descriptor(int n, const double *r, const double *O, const Grid &g, int m, const int *idx, __bf16 *x,
                       hipStream_t s) {
	if(m > 0) hipLaunchKernelGGL(k_descriptor, dim3(m), dim3(64), 0, s, n, r, O, g, m, idx, x);
}

// ------------------------------------------------------------------------
// training samples: a random particle of the current state, displaced and
// rotated at random (the "current" state of a move), its descriptor there,
// and as target the move back: displacement in the perturbed body frame and
// the rotation axis (-a; the angle is uniform in both directions).  16 lanes
// per sample, which find its neighbours as a pass does, from a record (here in
// LDS) and positions staged once: a search through 27 ranges for every read of
// a candidate, by a wavefront per sample, took 33 us for 4096 samples; with the
// record 18; four samples per wavefront 11.3.

constexpr int TS_LANES = 16;               // lanes per sample
constexpr int TS_BLOCK = 256 / TS_LANES;   // samples of a workgroup

__global__ __launch_bounds__(256) void k_train_samples(DevState d, uint64_t seed, uint64_t step, int m, int m_pad,
                                                       double pos_noise, double theta_max, __bf16 *x, float *target) {
	constexpr int T = TS_LANES;
	__shared__ DescLds Ds[TS_BLOCK];
	__shared__ __attribute__((aligned(16))) CandLds Cs[TS_BLOCK];
	const int lane = threadIdx.x & (T - 1), team = threadIdx.x / T;
	const int b = blockIdx.x * TS_BLOCK + team;
	__bf16 *row = x + (size_t) b * NN_IN_PAD;
	const bool live = b < m;
	int nv = 0;
	double pt[3], Ot[9];
	CellView v{};
	int j = 0;
	const double *F = nullptr;
	double L[3], iL[3];
	CandLds &CL = Cs[team];
	auto cands = [&]() { return Cands{d, F, v, j, &CL}; };
	if(b < m_pad && !live) {
		zero_row<T>(row, lane);
		if(lane < 6) target[(size_t) b * 6 + lane] = 0.f;
	}
	if(live) {
		const uint32_t k0 = (uint32_t) seed, k1 = (uint32_t) (seed >> 32);
		const u32x4 r0 = philox(u32x4{(uint32_t) b, 0xA5A50000u, (uint32_t) step, (uint32_t) (step >> 32)}, k0, k1);
		const u32x4 r1 = philox(u32x4{(uint32_t) b, 0xA5A50001u, (uint32_t) step, (uint32_t) (step >> 32)}, k0, k1);
		// a uniform slot of the whole context: a uniform particle of a replica
		// chosen with probability proportional to its size
		j = (int) __umulhi(r0.x, (uint32_t) d.Ntot);
		const Rep &rp = d.reps[d.prep[j]];
		F = pick_buf(d.f, rp.sel);
		for(int k = 0; k < 3; k++) {
			L[k] = rp.g.box[k];
			iL[k] = rp.g.inv_box[k];
		}
		double p[3], O[9];
		for(int k = 0; k < 3; k++) p[k] = part(F, j)[k];
		for(int k = 0; k < 9; k++) O[k] = part(F, j)[3 + k];
		// its cell on the current grid (particles never leave their cells
		// between rebuilds) and the cells around it, as a pass's record
		const int n0 = rp.g.n[0], n1 = rp.g.n[1], n2 = rp.g.n[2];
		const int ix = cell_coord(p[0], rp.g.shift[0], rp.g.inv_box[0], n0);
		const int iy = cell_coord(p[1], rp.g.shift[1], rp.g.inv_box[1], n1);
		const int iz = cell_coord(p[2], rp.g.shift[2], rp.g.inv_box[2], n2);
		v.rec = CL.rec;
		v.cloc = (ix * n1 + iy) * n2 + iz;
		v.r = d.prep[j];
		v.sel = rp.sel;
		write_record(CL.rec, 0, d.start + rp.cell_off, v.cloc, ix, iy, iz, n0, n1, n2, v.r, v.sel, lane);
		team_sync();
		v.M = CL.rec[REC_M];
		v.s0 = CL.rec[REC_S0];
		v.cnt = CL.rec[REC_CNT];
		cands().stage<T>(CL, lane);
		// the perturbed state: Gaussian displacement, rotation by an angle
		// uniform in [0, theta_max) about a uniform axis
		double z[6];
		gauss2(r0.y, r0.z, z[0], z[1]);
		gauss2(r0.w, r1.x, z[2], z[3]);
		gauss2(r1.y, r1.z, z[4], z[5]);
		for(int k = 0; k < 3; k++) pt[k] = p[k] + pos_noise * z[k];
		double ax[3] = {z[3], z[4], z[5]};
		const double an = sqrt(ax[0] * ax[0] + ax[1] * ax[1] + ax[2] * ax[2]);
		for(int k = 0; k < 3; k++) ax[k] /= an;
		const double ang = u01(r1.w) * theta_max;
		double sn, cs, R[9];
		sincos(ang, &sn, &cs);
		rotation_matrix(ax, sn, cs, R);
		mat_mul3(O, R, Ot);
		if(lane == 0) {
			float *t = target + (size_t) b * 6;
			for(int k = 0; k < 3; k++)
				t[k] = (float) (Ot[3 * k] * (p[0] - pt[0]) + Ot[3 * k + 1] * (p[1] - pt[1]) + Ot[3 * k + 2] * (p[2] - pt[2]));
			for(int k = 0; k < 3; k++) t[3 + k] = (float) -ax[k];
		}
		const Cands c = cands();
		nv = desc_collect<T>(pt, c.count(), [&](int i, double q[3]) { c.pos(i, q); }, L, iL, Ds[team], row, lane);
	}
	__syncthreads();
	if(live) {
		const Cands c = cands();
		desc_fill<T>(
			pt, Ot, nv, [&](int i, double q[3]) { c.pos(i, q); }, [&](int i, double Oq[9]) { c.ori(i, Oq); }, L, iL, Ds[team],
			row, lane);
	}
}

void launch_train_samples(const DevState &d, uint64_t seed, uint64_t step, int m, double pos_noise, double theta_max,
                          __bf16 *x, float *target, hipStream_t s) {
	const int m_pad = (m + 31) & ~31;
	hipLaunchKernelGGL(k_train_samples, dim3((m_pad + TS_BLOCK - 1) / TS_BLOCK), dim3(256), 0, s, d, seed, step, m, m_pad,
	                   pos_noise, theta_max, x, target);
}

}  // namespace ppd
