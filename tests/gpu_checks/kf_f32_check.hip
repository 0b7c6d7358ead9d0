// kf_f32_check SIDE RANGE COSMAX -- the colour pass's single-precision pair
// test against the reference arithmetic, on pairs at its thresholds.
//
// For a cell of side SIDE (in bond ranges 1 + delta = RANGE) the host draws a
// member, a trial (displacement, rotation) that stays in the cell and a
// neighbour whose distance from the trial position lies within 1e-9 to 1e-3
// of contact or of the bond range, or whose patches lie as close to cosmax,
// or anywhere in reach; every position far outside the box as unwrapped ones
// are.  The device forms each pair as pass_cell does (positions relative to
// the cell's centre, O'^T d = R^T (O^T d)) and compares what the filter
// decides with the exact form (MC.c:232-262).  Prints one line
//   pairs P decided D unsure U mismatches M
// and exits 0 when M == 0.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "pp_device.hpp"

using namespace ppd;

struct Pair {
	double p[3], dr[3], R[9], Op[9], q[3], Oq[9], centre[3];
};

__global__ void k_check(const Pair *pairs, int n, double L, double side, double rc2, double cosmax, int *out) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= n) return;
	const Pair &t = pairs[i];
	const double iL = 1. / L;
	// the filter, as pass_cell forms its operands
	const F32Filter fl = f32_filter(cosmax, rc2, side);
	float d[3], O[9], R[9], Q[9];
	for(int c = 0; c < 3; c++) {
		const float nx = (float) kf_min_image(t.p[c] - t.centre[c], L, iL) + (float) t.dr[c];
		d[c] = (float) kf_min_image(t.q[c] - t.centre[c], L, iL) - nx;
	}
	for(int e = 0; e < 9; e++) {
		O[e] = (float) t.Op[e];
		R[e] = (float) t.R[e];
		Q[e] = (float) t.Oq[e];
	}
	const float d2 = norm2(d[0], d[1], d[2]);
	int got = 2;  // 0 no bond, 1 bond, 3 overlap, 2 undecided
	if(!f32_near(d2, fl)) {
		if(d2 < 1.f) got = 3;
		else if(!(d2 < fl.rc2)) got = 0;
		else {
			float a0, a1, a2, e0, e1, e2;
			mul_t(O, d[0], d[1], d[2], a0, a1, a2);
			mul_t(R, a0, a1, a2, e0, e1, e2);
			bool yes, unsure;
			f32_bond(e0, e1, e2, d[0], d[1], d[2], d2, Q, fl, yes, unsure);
			got = unsure ? 2 : (yes ? 1 : 0);
		}
	}
	// the reference arithmetic
	double w[3], On[9], P[4][3];
	for(int c = 0; c < 3; c++) w[c] = kf_min_image(t.q[c] - (t.p[c] + t.dr[c]), L, iL);
	const double w2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
	mat_mul3(t.Op, t.R, On);
	kf_patches(On, P);
	int want = 0;
	if(w2 < 1.) want = 3;
	else if(w2 < rc2) {
		kf_unit(w[0], w[1], w[2], w2);
		want = kf_any_p(w[0], w[1], w[2], &P[0][0], cosmax) && kf_any_q(w[0], w[1], w[2], t.Oq, cosmax) ? 1 : 0;
	}
	out[i] = got == 2 ? 2 : (got == want ? 0 : 1);
}

using Gen = std::mt19937_64;

static double uni(Gen &g) { return std::uniform_real_distribution<double>(0., 1.)(g); }

static void direction(Gen &g, double v[3]) {
	std::normal_distribution<double> N(0., 1.);
	double s = 0.;
	for(int c = 0; c < 3; c++) v[c] = N(g), s += v[c] * v[c];
	for(int c = 0; c < 3; c++) v[c] /= std::sqrt(s);
}

static void axis_angle(const double a[3], double th, double R[9]) {
	const double c = std::cos(th), s = std::sin(th);
	const double K[9] = {0, -a[2], a[1], a[2], 0, -a[0], -a[1], a[0], 0};
	for(int i = 0; i < 3; i++)
		for(int j = 0; j < 3; j++) R[3 * i + j] = (i == j ? c : 0.) + (1. - c) * a[i] * a[j] + s * K[3 * i + j];
}

static void mul(const double A[9], const double B[9], double C[9]) {
	for(int i = 0; i < 3; i++)
		for(int j = 0; j < 3; j++) C[3 * i + j] = A[3 * i] * B[j] + A[3 * i + 1] * B[3 + j] + A[3 * i + 2] * B[6 + j];
}

// A rotation that takes a random base patch to a direction at angle
// acos(cs) from `axis`, with a random spin.
static void aim(Gen &g, const double axis[3], double cs, double O[9]) {
	double w[3], dir[3];
	direction(g, w);
	const double dt = w[0] * axis[0] + w[1] * axis[1] + w[2] * axis[2];
	double s = 0.;
	for(int c = 0; c < 3; c++) w[c] -= dt * axis[c], s += w[c] * w[c];
	const double sn = std::sqrt(std::max(0., 1. - cs * cs));
	for(int c = 0; c < 3; c++) dir[c] = cs * axis[c] + sn * w[c] / std::sqrt(s);
	const int a = (int) (uni(g) * 4) & 3;
	double b[3], k[3], A[9], B[9];
	for(int c = 0; c < 3; c++) b[c] = kf_base(a, c);
	// half turn about the bisector of b and dir, then a spin about dir
	s = 0.;
	for(int c = 0; c < 3; c++) k[c] = b[c] + dir[c], s += k[c] * k[c];
	for(int c = 0; c < 3; c++) k[c] /= std::sqrt(s);
	axis_angle(k, M_PI, A);
	axis_angle(dir, 2. * M_PI * uni(g), B);
	mul(B, A, O);
}

int main(int argc, char **argv) {
	if(argc != 4) return 2;
	const double range = atof(argv[2]), side = atof(argv[1]) * range, cosmax = atof(argv[3]);
	const double L = 6. * side, rc2 = range * range;
	const int n = 1 << 19;
	Gen g(4321);
	auto near = [&]() { return (uni(g) < 0.5 ? -1. : 1.) * std::pow(10., -9. + 6. * uni(g)); };
	std::vector<Pair> pairs(n);
	for(int i = 0; i < n; i++) {
		Pair &t = pairs[i];
		double ax[3], u[3], mu[3], pn[3], On[9], Rt[9];
		for(int c = 0; c < 3; c++) {
			t.centre[c] = L * uni(g);
			const double off = L * std::floor(2001. * uni(g) - 1000.);  // unwrapped
			pn[c] = t.centre[c] + off + side * (uni(g) - 0.5);
			double at = t.centre[c] + off + side * (uni(g) - 0.5);      // the start, in the cell too
			if(i % 2) at = pn[c] - 0.05 * (uni(g) - 0.5);               // or a small step away
			t.p[c] = at;
			t.dr[c] = pn[c] - at;
			pn[c] = t.p[c] + t.dr[c];
		}
		direction(g, u);
		for(int c = 0; c < 3; c++) mu[c] = -u[c];
		// i mod 6: contact, bond range, p's patch, q's patch, both, in reach
		const int mode = i % 6;
		const double r = mode == 0 ? 1. + near() : (mode == 1 ? range * (1. + near()) : 1. + (range - 1.) * uni(g));
		auto cs = [&](bool at) { return std::min(1., at ? cosmax + near() : cosmax + (1. - cosmax) * (1.2 * uni(g) - 0.1)); };
		aim(g, u, cs(mode == 2 || mode == 4), On);
		aim(g, mu, cs(mode == 3 || mode == 4), t.Oq);
		// On = Op R
		direction(g, ax);
		axis_angle(ax, 0.5 * uni(g), t.R);
		for(int a = 0; a < 3; a++)
			for(int b = 0; b < 3; b++) Rt[3 * a + b] = t.R[3 * b + a];
		mul(On, Rt, t.Op);
		for(int c = 0; c < 3; c++) t.q[c] = pn[c] + r * u[c] + L * std::floor(5. * uni(g) - 2.);
	}
	Pair *dp = nullptr;
	int *dout = nullptr;
	if(hipMalloc(&dp, sizeof(Pair) * n) != hipSuccess || hipMalloc(&dout, sizeof(int) * n) != hipSuccess) return 2;
	if(hipMemcpy(dp, pairs.data(), sizeof(Pair) * n, hipMemcpyHostToDevice) != hipSuccess) return 2;
	hipLaunchKernelGGL(k_check, dim3(n / 256), dim3(256), 0, 0, dp, n, L, side, rc2, cosmax, dout);
	std::vector<int> out(n);
	if(hipMemcpy(out.data(), dout, sizeof(int) * n, hipMemcpyDeviceToHost) != hipSuccess) return 2;
	long unsure = 0, bad = 0;
	for(int v : out) {
		unsure += v == 2;
		bad += v == 1;
	}
	printf("pairs %d decided %ld unsure %ld mismatches %ld\n", n, n - unsure, unsure, bad);
	(void) hipFree(dp);
	(void) hipFree(dout);
	return bad == 0 ? 0 : 1;
}
