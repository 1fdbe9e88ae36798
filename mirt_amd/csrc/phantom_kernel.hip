// phantom_kernel.hip -- analytic cone-beam line integrals of ellipsoids on
// gfx950: ellipsoid_proj (fbp/ellipsoid_proj.m:35-125) with the
// detector-to-parallel coordinate maps of fbp/ir_coord_cb_flat_to_par.m and
// fbp/ir_coord_cb_arc_to_par.m, in FP64 as the MATLAB computes it.
//
// One lane per detector sample (s fastest, so the [ns nt na] writes are
// coalesced) and ELL_VIEWS views.  An ellipsoid is the unit ball under the
// linear map M = diag(1/r) Rz(-xy_angle): with the ray's foot point P and
// direction D of unit length, p = M (P - centre) and e = M D, the chord is
//   2 sqrt(B^2 - A C) / A = 2 sqrt(A - |p x e|^2) / A,  A = |e|^2,
// the form of ellipsoid_proj.m:110-118 by Lagrange's identity (p may be any
// point of the ray, and nothing large cancels); 0 where the ray misses (the
// "real part" trick of ellipsoid_proj.m:123).  P and D are made once per
// (sample, view) from the sines and cosines of the detector angles, which are
// ratios of lengths, and of the view angle (from the host), so no
// trigonometric function runs per view; a ray and ellipsoid then take 23 FP64
// operations, and 12 more where a lane of the wave hits.  The ellipsoid table
// sits in LDS, a row read once for the lane's views.
// Bound: FP64 VALU issue.  512 x 384 x 360 rays, 20 ellipsoids: 1.5 ms (3.5 ms
// with the reference's expressions evaluated per ray, a sincos per view and
// IEEE square roots and quotients).
// With oversampling (ellipsoid_proj.m:44-58) each lane evaluates its sample's
// No x No sub-samples and averages them in downsample3's order (along s, then
// along t).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "fdkhip.h"

namespace fdk {

// an ellipsoid: p = (a11 x + a12 y - ox, a21 x + a22 y - oy, irz z - oz), and 2 val
struct EllRow {
	double a11, a12, a21, a22, irz, ox, oy, oz, val2;
};

enum { ELL_PAR = 0, ELL_FLAT = 1, ELL_ARC = 2 };
constexpr int ELL_MAX = 512;        // ellipsoids per launch (LDS table)
constexpr int ELL_VIEWS = 4;        // views per lane

struct EllArgs {
	const double *s, *t;             // [ns], [nt] detector sample positions
	const double *cb, *sb, *zs;      // [na] cos and sin of the source angle, source height
	const EllRow *ell;               // [nell]
	int ns, nt, na, nell, no;        // no: oversampling factor
	double ds, dt, dso, dod;         // sample spacing (oversampling), distances
	int kind;
	double *proj;                    // [na][nt][ns]
};

// Parallel-beam coordinates (uu, vv) of a detector sample at beta = 0 and the
// sines and cosines of its azimuth and polar angle
__device__ __forceinline__ void par_coords(const EllArgs &a, double ss, double tt,
	double &uu, double &vv, double &saz, double &caz, double &spol, double &cpol)
{
	if (a.kind == ELL_PAR) {
		uu = ss;
		vv = tt;
		saz = spol = 0.0;
		caz = cpol = 1.0;
		return;
	}
	const double Ds = a.dso, Dc = a.dso + a.dod;
	if (a.kind == ELL_FLAT) {        // ir_coord_cb_flat_to_par.m
		const double r2 = Dc * Dc + ss * ss;
		const double r = sqrt(r2), R = sqrt(r2 + tt * tt);
		saz = ss / r;                // azim = atan(ss / Dc), polar = -atan(tt / r)
		caz = Dc / r;
		spol = -tt / R;
		cpol = r / R;
		uu = Ds * ss / r;
		vv = Ds * tt / R * Dc / r;
		return;
	}
	// arc (dfs = 0), ir_coord_cb_arc_to_par.m: focal radius Dc, source at (0, dso, 0);
	// azim = atan(tan(ss / Rf)), polar = -asin(tt / |(Rf, tt)|)
	const double Rf = Dc;
	double sg, cg;
	sincos(ss / Rf, &sg, &cg);
	const double en = sqrt(Rf * Rf + tt * tt);
	saz = cg < 0.0 ? -sg : sg;
	caz = fabs(cg);
	spol = -tt / en;
	cpol = fabs(Rf) / en;
	uu = saz * Ds;
	vv = (-caz * Ds) * spol;
}

// val2 sqrt(d) / A for d > 0: d / (A sqrt(d)) with the reciprocal square root
// of z = d A^2 taken by the instruction (about 2^-26) and one cubic step
// (within 2 ulp); the library's root and quotient where z leaves the middle
// of the range
__device__ __forceinline__ double chord(double d, double A, double val2)
{
	const double z = d * A * A;
	if (!(z > 1e-280 && z < 1e280))
		return val2 * sqrt(d) / A;
	double y = __builtin_amdgcn_rsq(z);
	const double e = fma(-z * y, y, 1.0);
	y = fma(y * e, fma(e, 0.375, 0.5), y);
	return val2 * (d * y);
}

// four waves per SIMD: 1.52 ms at the size above; three without spills of the
// per-view set-up 1.67 ms; 2 and 8 views per lane 1.58 and 1.70 ms
__global__ void __launch_bounds__(256, 4)
ellipsoid_proj_kernel(const EllArgs a)
{
	extern __shared__ EllRow E[];   // [nell]
	for (int k = threadIdx.x; k < a.nell; k += blockDim.x)
		E[k] = a.ell[k];
	__syncthreads();
	const long nst = (long) a.ns * a.nt;
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	const long vb = (long) blockIdx.z * gridDim.y + blockIdx.y;   // block of views
	if (i >= nst || vb * ELL_VIEWS >= a.na)
		return;
	const int is = (int) (i % a.ns), it = (int) (i / a.ns);
	const int v0 = (int) vb * ELL_VIEWS;
	const int nv = min(ELL_VIEWS, a.na - v0);
	double sum[ELL_VIEWS];
#pragma unroll
	for (int v = 0; v < ELL_VIEWS; ++v)
		sum[v] = 0.0;
	const int no = a.no;
	for (int jt = 0; jt < no; ++jt) {
		double row[ELL_VIEWS];       // this t sub-row, summed over the s sub-samples
#pragma unroll
		for (int v = 0; v < ELL_VIEWS; ++v)
			row[v] = 0.0;
		// sub-sample offsets of ellipsoid_proj.m:50-51: [-(No-1):2:(No-1)]/(2 No) * d
		const double tt = (no > 1) ? ((double) (2 * jt - (no - 1)) / (2.0 * no)) * a.dt + a.t[it]
			: a.t[it];
		for (int js = 0; js < no; ++js) {
			const double ss = (no > 1)
				? ((double) (2 * js - (no - 1)) / (2.0 * no)) * a.ds + a.s[is] : a.s[is];
			double uu, vv, saz, caz, spol, cpol;
			par_coords(a, ss, tt, uu, vv, saz, caz, spol, cpol);
			// per view: foot point (px, py, pz) and direction (dx, dy, spol)
			double px[ELL_VIEWS], py[ELL_VIEWS], pz[ELL_VIEWS], dx[ELL_VIEWS], dy[ELL_VIEWS];
			double ray[ELL_VIEWS];
#pragma unroll
			for (int v = 0; v < ELL_VIEWS; ++v) {
				const int vi = min(v0 + v, a.na - 1);
				const double cb = a.cb[vi], sb = a.sb[vi];
				const double c = fma(cb, caz, -(sb * saz)), s = fma(sb, caz, cb * saz);
				const double vs = vv * spol;
				px[v] = fma(uu, c, vs * s);
				py[v] = fma(uu, s, -(vs * c));
				pz[v] = fma(vv, cpol, a.zs[vi]);
				dx[v] = -s * cpol;
				dy[v] = c * cpol;
				ray[v] = 0.0;
			}
			for (int k = 0; k < a.nell; ++k) {
				const EllRow e = E[k];
				const double e3 = spol * e.irz;
#pragma unroll
				for (int v = 0; v < ELL_VIEWS; ++v) {
					const double p1 = fma(px[v], e.a11, fma(py[v], e.a12, -e.ox));
					const double p2 = fma(px[v], e.a21, fma(py[v], e.a22, -e.oy));
					const double p3 = fma(pz[v], e.irz, -e.oz);
					const double e1 = fma(dx[v], e.a11, dy[v] * e.a12);
					const double e2 = fma(dx[v], e.a21, dy[v] * e.a22);
					const double A = fma(e1, e1, fma(e2, e2, e3 * e3));
					const double w1 = fma(p2, e3, -(p3 * e2));
					const double w2 = fma(p3, e1, -(p1 * e3));
					const double w3 = fma(p1, e2, -(p2 * e1));
					const double d = A - fma(w1, w1, fma(w2, w2, w3 * w3));
					if (d > 0.0)
						ray[v] += chord(d, A, e.val2);
				}
			}
#pragma unroll
			for (int v = 0; v < ELL_VIEWS; ++v)
				row[v] += ray[v];
		}
#pragma unroll
		for (int v = 0; v < ELL_VIEWS; ++v)
			sum[v] += (no > 1) ? row[v] / no : row[v];
	}
#pragma unroll
	for (int v = 0; v < ELL_VIEWS; ++v)
		if (v < nv)
			a.proj[(long) (v0 + v) * nst + i] = (no > 1) ? sum[v] / no : sum[v];
}

} // namespace fdk

using namespace fdk;

int fdkhip_fail_msg(int code, const char *msg);   // fdk_api.hip

#define ELL_TRY(expr)                                                             \
	do {                                                                          \
		hipError_t e_ = (expr);                                                   \
		if (e_ != hipSuccess) {                                                   \
			rc = fdkhip_fail_msg(FDKHIP_EHIP, hipGetErrorString(e_));             \
			goto done;                                                            \
		}                                                                         \
	} while (0)

extern "C" int fdkhip_ellipsoid_proj(const double *s, int32_t ns, const double *t, int32_t nt,
	const double *beta, const double *source_zs, int32_t na, double dso, double dod,
	double dfs, const double *params, int32_t nell, int32_t oversample, double *proj_dev,
	void *stream)
{
	if (ns < 0 || nt < 0 || na < 0 || nell < 0)
		return fdkhip_fail_msg(FDKHIP_EARG, "negative size");
	if (nell > ELL_MAX)
		return fdkhip_fail_msg(FDKHIP_EUNSUPPORTED, "at most 512 ellipsoids per call");
	if (oversample < 1)
		return fdkhip_fail_msg(FDKHIP_EARG, "oversample must be >= 1");
	if ((long) ns * nt * na == 0)
		return FDKHIP_OK;
	if (!s || !t || !beta || !proj_dev || (nell > 0 && !params))
		return fdkhip_fail_msg(FDKHIP_EARG, "NULL argument");
	int kind;
	if (isinf(dso))
		kind = ELL_PAR;
	else if (isinf(dfs))
		kind = ELL_FLAT;
	else if (dfs == 0)
		kind = ELL_ARC;
	else
		return fdkhip_fail_msg(FDKHIP_EUNSUPPORTED, "not done");   // ellipsoid_proj.m:81
	if (oversample > 1 && ((ns > 1 && !(s[1] != s[0])) || (nt > 1 && !(t[1] != t[0]))))
		return fdkhip_fail_msg(FDKHIP_EARG, "uniform spacing required for oversampling");
	if (oversample > 1) {   // ellipsoid_proj.m:44-48
		const double ds = ns > 1 ? s[1] - s[0] : 0, dt = nt > 1 ? t[1] - t[0] : 0;
		for (int i = 1; i < ns; ++i)
			if (fabs((s[i] - s[i - 1]) / ds - 1) > 1e-6)
				return fdkhip_fail_msg(FDKHIP_EARG, "uniform spacing required for oversampling");
		for (int i = 1; i < nt; ++i)
			if (fabs((t[i] - t[i - 1]) / dt - 1) > 1e-6)
				return fdkhip_fail_msg(FDKHIP_EARG, "uniform spacing required for oversampling");
	}
	std::vector<EllRow> rows((size_t) nell);
	for (int k = 0; k < nell; ++k) {
		const double *p = params + 9 * (size_t) k;
		if (p[7] != 0)
			return fdkhip_fail_msg(FDKHIP_EUNSUPPORTED, "z rotation not done");   // :94
		const double xang = p[6] * (M_PI / 180);
		const double c = cos(xang), sn = sin(xang);
		rows[k] = EllRow{c / p[3], sn / p[3], -sn / p[4], c / p[4], 1 / p[5],
			(p[0] * c + p[1] * sn) / p[3], (p[1] * c - p[0] * sn) / p[4], p[2] / p[5],
			2 * p[8]};
	}
	hipStream_t st = (hipStream_t) stream;
	int rc = FDKHIP_OK;
	// one table for the kernel: s, t, cos and sin of beta, source heights, rows
	const size_t nd = (size_t) ns + nt + 3 * (size_t) na, nrow = rows.size();
	std::vector<double> tab(nd + nrow * (sizeof(EllRow) / sizeof(double)));
	std::copy(s, s + ns, tab.begin());
	std::copy(t, t + nt, tab.begin() + ns);
	for (int ia = 0; ia < na; ++ia) {
		tab[(size_t) ns + nt + ia] = cos(beta[ia]);
		tab[(size_t) ns + nt + na + ia] = sin(beta[ia]);
		tab[(size_t) ns + nt + 2 * (size_t) na + ia] = source_zs ? source_zs[ia] : 0.0;
	}
	if (nrow > 0)
		memcpy(tab.data() + nd, rows.data(), nrow * sizeof(EllRow));
	double *d_tab = nullptr;
	{
		ELL_TRY(hipMalloc(&d_tab, sizeof(double) * tab.size()));
		ELL_TRY(hipMemcpyAsync(d_tab, tab.data(), sizeof(double) * tab.size(),
			hipMemcpyHostToDevice, st));
		EllArgs a;
		a.s = d_tab;
		a.t = d_tab + ns;
		a.cb = a.t + nt;
		a.sb = a.cb + na;
		a.zs = a.sb + na;
		a.ell = (const EllRow *) (a.zs + na);
		a.ns = ns;
		a.nt = nt;
		a.na = na;
		a.nell = nell;
		a.no = oversample;
		a.ds = ns > 1 ? s[1] - s[0] : 0;
		a.dt = nt > 1 ? t[1] - t[0] : 0;
		a.dso = dso;
		a.dod = dod;
		a.kind = kind;
		a.proj = proj_dev;
		const long nst = (long) ns * nt;
		// samples along x, blocks of views along y and z: a grid has less than 2^32
		// threads along a dimension and at most 65535 workgroups along y and z
		const long vblocks = ((long) na + ELL_VIEWS - 1) / ELL_VIEWS;
		const unsigned gy = (unsigned) std::min(vblocks, 65535L);
		const dim3 grid((unsigned) ((nst + 255) / 256), gy, (unsigned) ((vblocks + gy - 1) / gy));
		hipLaunchKernelGGL(ellipsoid_proj_kernel, grid, dim3(256), nrow * sizeof(EllRow), st, a);
		ELL_TRY(hipGetLastError());
		// the host table above is released at return: wait for the copy
		ELL_TRY(hipStreamSynchronize(st));
	}
done:
	(void) hipFree(d_tab);
	return rc;
}
