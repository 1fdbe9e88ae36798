// mat_kernel.hip -- cbct_back_mat (fbp/cbct_back.m:142-270) on gfx950.
//
// The reference's MATLAB backprojector, the use_mex = 0 route of cbct_back:
// double precision throughout, every voxel of the mask against every view
// 1:ia_skip:na, with its own edge rules (cbct_back.m:221-233):
//   * s: a sample position bs outside [1, ns] (1-based) reads the extra zero
//     column ns+1, so it adds nothing (no one-bin fall-off as in the mex);
//   * t: bt is clamped to [1, nt] (replication of the edge rows) and bt = nt
//     reads rows nt-1 and nt with weight 1 on the last;
// and its own weights (cbct_back.m:244-249): mag^2 for flat and parallel
// detectors, dsd^2 / (r_loop^2 + y_betas^2) for the arc, r_loop = x_beta -
// offset_source.  Helical source positions (source_zs, one per view) enter
// tprime = mag * (zc - source_zs) as in cbct_back.m:219.
//
// Every product, quotient and sum is one IEEE double operation in the order
// the MATLAB expression evaluates it (the library is built with
// -ffp-contract=off, so nothing is fused), views are added to each voxel in
// view order starting from 0, as img2 = img2 + p0 does.  The per-view cos and
// sin come from the host's libm.
//
// The helical version (mex/src/fdk-helix/cbct_back_helix.m:185-350) adds,
// when MatArgs::zrange is set: per-slice view ranges (slice iz uses views
// ia_min:ia_skip:ia_max around the view whose source height is nearest, the
// host computes them), the cone-parallel geometry of rebinned views
// (cone_par: mag = dsd / (sqrt(dso^2 - x_beta^2) - (dso - y_betas)),
// sprime = x_beta, a source height offset asin(-x_beta / dso) *
// source_dz_per_rad, no distance weight) and a per-slice scale.
//
// Launch: a workgroup takes an 8 x 8 tile of image columns and up to MAT_NW
// chunks of MAT_ZC slices, one wave per chunk; lane = column, the lane's
// MAT_ZC accumulators stay in registers over all views.  Views go in stages
// of as many views as the workgroup has waves, through two LDS buffers: wave
// w computes the column geometry (x_beta, mag, bs, the weights, the arc's
// atan2) of stage view w for the tile's 64 columns, and every wave adds all
// of the stage's views to its own slices, so that geometry is computed once
// per (column, view), not once per 16 slices.  The 1-D grid is remapped so
// that neighbouring tiles, whose detector footprints overlap, run on the same
// XCD and share its L2.
//
// Bound: FP64 VALU issue, so the two quotients per update (tprime / dt, and
// the arc weight / (r_loop^2 + y_betas^2)) are taken by const_div below, four
// FP64 operations with the bits of the division instead of the about twelve
// of the compiler's sequence: dt is the same for the whole launch, the
// weight's divisor for a column's view, so their reciprocals are made once.
// 256 x 256 x 128 from 492 arc views of 888 x 64: 5.5 ms (14.7 ms with the
// compiler's divisions, 64-bit gather addresses and the geometry computed by
// every wave for itself).  512 x 512 x 256 from 984 such views: 79.5 ms (193.8),
// 38 VALU instructions per update, 25 of them FP64 sums, products and FMAs, 82 %
// of the CUs' VALU issue, HBM at 0.8 TB/s.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fdk_kernels.h"

namespace fdk {

namespace {

__device__ __forceinline__ int mat_xcd_block(int bid, int nblocks)
{
	const int xcd = bid & 7, local = bid >> 3;
	const int per = nblocks >> 3, rem = nblocks & 7;
	return xcd * per + min(xcd, rem) + local;
}

__device__ __forceinline__ double mat_sample(const float *p, long i)
{
	return (double) p[i];
}

__device__ __forceinline__ double mat_sample(const double *p, long i)
{
	return p[i];
}

// a / b, correctly rounded, from rh = RN(1 / b) and rl = (1 / b - rh) to one
// rounding: q = RN(a rh + RN(a rl)) is within one ulp of a / b, so the
// remainder a - q b is exact in one FMA and RN(q + r rh) is the correctly
// rounded quotient (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", IBM J. Res. Dev. 34(1), 1990, theorem 8.2).
// Needs |b| within [1e-60, 1e60] and no over- or underflow on the way: a NaN
// comes of an overflow, and |a| is 0 or at least DIV_MIN, where the quotient is
// above 2^-1000 and the remainder above 2^-910.  The kernel does workgroups
// again that see another dividend of the weight (tprime, the other dividend,
// may be smaller: bt = tprime / dt + wt is then wt).
__device__ __forceinline__ double const_div(double a, double b, double rh, double rl)
{
	const double q = fma(a, rh, a * rl);
	return fma(fma(-q, b, a), rh, q);
}

constexpr double DIV_MIN = 1e-240;   // above 2^-800

__device__ __forceinline__ bool mat_moderate(double x)
{
	return fabs(x) > 1e-60 && fabs(x) < 1e60;   // false for NaN
}

// two horizontally neighbouring samples in one load (4- or 8-byte aligned)
template <typename TP>
struct __attribute__((packed, aligned(sizeof(TP)))) MatPair {
	TP x, y;
};

// Column geometry of one view over the tile, per lane in LDS: fields of 64
// doubles, then the left sample column, then (helical) two words of flags: bit
// z of them says that slice z of the workgroup takes the view
// the distance weight: none (cone-parallel views), a factor (flat, parallel) or
// the arc's quotient
enum { MW_NONE = 0, MW_MUL, MW_DIV };

enum { MF_MAG = 0, MF_WR, MF_W, MF_RH, MF_RL, MF_ZOFF, MF_COUNT };
constexpr int MAT_VIEW_BYTES = MF_COUNT * 64 * 8 + 64 * 4 + 2 * 8;
static_assert(MAT_NW * MAT_ZC <= 128, "two words of slice flags");

// HELIX: the helical backprojector's per-slice view ranges and scales and
// cone-parallel geometry (compiled out of the axial route).  WGT: the distance
// weight (a branch per slice would keep the slices' gathers apart).  IDX: the
// type of byte offsets into a view (32 bits where a view is smaller than
// 4 GiB: the gathers then take a scalar base and one register of offset).
// FAST: quotients by const_div and both samples of a row in one load -- for
// the last column, whose right neighbour is the zero column ns+1, the pair to
// its left with the weights moved one sample over.  A FAST workgroup that
// meets a geometry or (FP64 views; FP32 samples are too large) a dividend
// outside const_div's range, or ends with a NaN sum (an
// infinite sample gives NaN in const_div and in a zero weight's product, where
// the reference may have an infinity or a number), sets its entry of a.redo;
// the other form, the reference's arithmetic to the letter, is launched after
// it over the same workgroups and does the marked ones again (all of them
// where the host does not launch FAST).
template <typename TP, bool HELIX, int WGT, typename IDX, bool FAST>
__global__ void __launch_bounds__(64 * MAT_NW, FAST ? 4 : 2) mat_kernel(const MatArgs a)
{
	extern __shared__ char mat_lds[];
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int nw = blockDim.x >> 6;                   // waves = chunks of this workgroup
	if (!FAST && a.redo && !a.redo[blockIdx.x])
		return;
	const int tx = (a.nx + 7) >> 3, ty = (a.ny + 7) >> 3;
	const int ngrp = (a.nzc + nw - 1) / nw;
	const int b = mat_xcd_block(blockIdx.x, tx * ty * ngrp);
	const int bxy = b % (tx * ty), bg = b / (tx * ty);
	// lanes past the image take its last column or row along and write nothing
	const int ixr = (bxy % tx) * 8 + (lane & 7), iyr = (bxy / tx) * 8 + (lane >> 3);
	const bool inimg = ixr < a.nx && iyr < a.ny;
	const int ix = min(ixr, a.nx - 1), iy = min(iyr, a.ny - 1);
	const long nxy = (long) a.nx * a.ny;
	const long col = ix + (long) iy * a.nx;
	const int z0 = (bg * nw + wave) * MAT_ZC;
	const int nk = max(min(MAT_ZC, a.nz - z0), 0);    // 0: a wave past the last chunk
	const bool live = !a.mask || a.mask[col];

	// cbct_back.m:160-165: xc = ([0:nx-1] - wx) * dx, likewise yc and zc
	const double xc = ((double) ix - a.wx) * a.dx;
	const double yc = ((double) iy - a.wy) * a.dy;
	// the slices' zc behind the stage buffers: a broadcast read per update, where
	// 16 more doubles per lane would not fit beside the accumulators
	const int stage_bytes = nw * MAT_VIEW_BYTES;
	double *zc = (double *) (mat_lds + 2 * stage_bytes) + wave * MAT_ZC;
	if (lane < MAT_ZC)
		zc[lane] = ((double) (z0 + lane) - a.wz) * a.dz;
	double acc[MAT_ZC];
#pragma unroll
	for (int k = 0; k < MAT_ZC; ++k)
		acc[k] = 0.0;
	const double ns1 = (double) a.ns + 1.0, ntd = (double) a.nt, nt1 = ntd - 1.0;
	const double dsd2 = a.dsd * a.dsd;
	// the views each slice takes (helical: its own range, cbct_back_helix.m:224-236);
	// the workgroup walks the union over all its slices
	int vlo = 0, vhi = a.nv - 1;
	if (HELIX) {
		vlo = a.nv;
		vhi = -1;
		for (int z = bg * nw * MAT_ZC; z < min((bg + 1) * nw * MAT_ZC, a.nz); ++z) {
			const int2 r = a.zrange[z];
			vlo = min(vlo, r.x <= r.y ? r.x : vlo);
			vhi = max(vhi, r.x <= r.y ? r.y : vhi);
		}
		vlo = max(vlo, 0);
		vhi = min(vhi, a.nv - 1);
	}

	bool bad = false;   // FAST: to be done again

	// setup of view v into a stage slot: the lane's column geometry
	auto setup = [&](char *slot, int v) {
		double *f = (double *) slot + lane;
		const double4 vw = a.views[v];              // {cos beta, sin beta, source_zs}
		// cbct_back.m:204-205
		const double x_beta = xc * vw.x + yc * vw.y;
		const double y_betas = a.dso - (-xc * vw.y + yc * vw.x);
		// cbct_back.m:208-220, cbct_back_helix.m:245-265
		double mag, sprime, r_loop = 0.0, zoff = 0.0;
		if (HELIX && a.cone_par) {
			mag = a.dsd / (sqrt(a.dso * a.dso - x_beta * x_beta) - (a.dso - y_betas));
			sprime = x_beta;
			zoff = asin(-x_beta / a.dso) * a.dz_per_rad;
		} else if (a.kind == KIND_PAR) {
			mag = 1.0;
			sprime = mag * x_beta;
		} else {
			mag = a.dsd / y_betas;
			if (a.kind == KIND_ARC) {
				r_loop = x_beta - a.offset_source;
				sprime = a.dsd * atan2(r_loop, y_betas);
			} else {
				sprime = mag * x_beta;
			}
		}
		// cbct_back.m:222-233 for s: out-of-range positions read column ns+1 (zero)
		double bs = sprime / a.ds + a.ws;
		if (!(bs >= 1.0 && bs <= (double) a.ns))
			bs = ns1;
		double is = floor(bs);
		if (is == ns1)
			is = (double) a.ns;
		// cbct_back.m:244-249 weights
		const double w = a.kind == KIND_ARC ? r_loop * r_loop + y_betas * y_betas : mag * mag;
		const double rh = 1.0 / w;
		f[MF_MAG * 64] = mag;
		f[MF_WR * 64] = bs - is;
		f[MF_W * 64] = w;
		f[MF_RH * 64] = rh;
		f[MF_RL * 64] = fma(-w, rh, 1.0) * rh;
		if (HELIX)
			f[MF_ZOFF * 64] = zoff;
		int *fi = (int *) (slot + MF_COUNT * 64 * 8);
		fi[lane] = (int) is - 1;                     // 0-based left column
		if (HELIX) {
#pragma unroll
			for (int h = 0; h < 2; ++h) {
				const int z = bg * nw * MAT_ZC + h * 64 + lane;
				const int2 r = a.zrange[min(z, a.nz - 1)];
				const unsigned long long m = __ballot(z < a.nz && v >= r.x && v <= r.y
					&& (v - r.x) % a.vstep == 0);
				if (lane == 0)
					((unsigned long long *) (fi + 64))[h] = m;
			}
		}
		bad = bad || !(mat_moderate(mag) && (WGT != MW_DIV || mat_moderate(w)) && fabs(zoff) < 1e60);
	};

	// adds a stage view to the wave's slices
	auto add_view = [&](const char *slot, int v) {
		const double *f = (const double *) slot + lane;
		double mag = f[MF_MAG * 64];
		const double wr = f[MF_WR * 64], w = f[MF_W * 64];
		const double rh = FAST && WGT == MW_DIV ? f[MF_RH * 64] : 0.0;
		const double rl = FAST && WGT == MW_DIV ? f[MF_RL * 64] : 0.0;
		const int is0 = ((const int *) (slot + MF_COUNT * 64 * 8))[lane];
		const double wl = 1.0 - wr;
		const bool right_zero = is0 + 1 >= a.ns;      // column ns+1 is the zero column
		const double zs = a.views[v].z;
		const double zsv = HELIX && a.cone_par ? zs + f[MF_ZOFF * 64] : zs;
		const char *pv = (const char *) a.proj + (long) v * a.view_stride * (long) sizeof(TP);
		const double wL = FAST && right_zero ? 0.0 : wl, wR = FAST && right_zero ? wl : wr;
		const IDX isl = (IDX) (right_zero && FAST ? is0 - 1 : is0);
		unsigned use = ~0u;                           // slices of this wave
		if (HELIX) {
			use = __builtin_amdgcn_readfirstlane(((const int *) (slot + MF_COUNT * 64 * 8))
				[64 + wave * MAT_ZC / 32]) >> (wave * MAT_ZC % 32);
			if (!(use & ((1u << MAT_ZC) - 1)))
				return;
		}
		// FLIGHT slices at a time: their positions and gathers, then their sums (as
		// many as the registers hold)
		constexpr int FLIGHT = HELIX || !FAST || sizeof(TP) == 8 ? 2 : 4;
#pragma unroll
		for (int k0 = 0; k0 < MAT_ZC; k0 += FLIGHT) {
			if (HELIX && !(use >> k0 & ((1u << FLIGHT) - 1)))
				continue;
			double wus[FLIGHT];
			MatPair<TP> u0[FLIGHT], u1[FLIGHT];
			// the group's positions wait for the sums of the group before (register
			// budget: the compiler would otherwise start many groups at once)
			asm volatile("" : "+v"(mag), "+v"(acc[k0 ? k0 - 1 : 0]));
#pragma unroll
			for (int g = 0; g < FLIGHT; ++g) {
				// cbct_back.m:219-233 for t: clamp to [1, nt], bt = nt uses rows nt-1, nt
				const double tprime = mag * (zc[k0 + g] - zsv);
				double bt = (FAST ? const_div(tprime, a.dt, a.rdt_h, a.rdt_l) : tprime / a.dt)
					+ a.wt;
				bt = fmax(bt, 1.0);                  // NaN -> 1, as MATLAB's max
				bt = fmin(bt, ntd);
				const double it = fmin(floor(bt), nt1);   // nt -> nt - 1
				wus[g] = bt - it;
				const int row = (int) it - 1;
				const IDX e = sizeof(IDX) == 4 ? (IDX) __umul24(row, a.ns) : (IDX) row * (IDX) a.ns;
				const char *p = pv + (e + isl) * (IDX) sizeof(TP);
				const char *q = p + (size_t) a.ns * sizeof(TP);
				if (FAST) {
					u0[g] = *(const MatPair<TP> *) p;
					u1[g] = *(const MatPair<TP> *) q;
				} else {
					u0[g].x = *(const TP *) p;
					u1[g].x = *(const TP *) q;
					u0[g].y = right_zero ? (TP) 0 : ((const TP *) p)[1];
					u1[g].y = right_zero ? (TP) 0 : ((const TP *) q)[1];
				}
			}
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int g = 0; g < FLIGHT; ++g) {
				const int k = k0 + g;
				if (HELIX && !(use >> k & 1))
					continue;
				// cbct_back.m:236-241
				const double wu = wus[g], wd = 1.0 - wu;
				const double p1 = wL * (double) u0[g].x + wR * (double) u0[g].y;
				const double p2 = wL * (double) u1[g].x + wR * (double) u1[g].y;
				double p0 = wd * p1 + wu * p2;
				if (WGT == MW_DIV) {
					const double d = p0 * dsd2;
					if (FAST && sizeof(TP) == 8)
						bad = bad || (fabs(d) < DIV_MIN && d != 0.0);
					p0 = FAST ? const_div(d, w, rh, rl) : d / w;
				} else if (WGT == MW_MUL)
					p0 = p0 * w;
				acc[k] = acc[k] + p0;                // cbct_back.m:251
			}
		}
	};

	// the column mask is the same for every wave: all of them leave together
	if (__any(live && inimg) && vlo <= vhi) {
		if (vlo + wave <= vhi)
			setup(mat_lds + wave * MAT_VIEW_BYTES, vlo + wave);
		__syncthreads();
		int buf = 0;
		for (int v0 = vlo; v0 <= vhi; v0 += nw, buf ^= 1) {
			if (v0 + nw + wave <= vhi)
				setup(mat_lds + (buf ^ 1) * stage_bytes + wave * MAT_VIEW_BYTES, v0 + nw + wave);
			const int n = min(nw, vhi - v0 + 1);
			for (int i = 0; i < n && nk > 0; ++i)
				add_view(mat_lds + buf * stage_bytes + i * MAT_VIEW_BYTES, v0 + i);
			__syncthreads();
		}
	}
	if (FAST) {
#pragma unroll
		for (int k = 0; k < MAT_ZC; ++k)
			bad = bad || acc[k] != acc[k];
		const int any = __syncthreads_or(bad);
		if (threadIdx.x == 0)
			a.redo[blockIdx.x] = any;
	}
	if (!inimg)
		return;
	double *out = a.image + col + (long) z0 * nxy;
	// cbct_back.m:264-266: (scale) * img, one double product per voxel
	// (cbct_back_helix.m:341-345: the slice's own scale); embed(img2, mask):
	// columns outside the mask are 0 (cbct_back.m:182-183, 261)
#pragma unroll
	for (int k = 0; k < MAT_ZC; ++k)
		if (k < nk)
			out[(long) k * nxy] = live ? ((HELIX && a.zscale) ? a.zscale[z0 + k] : a.scale) * acc[k]
				: 0.0;
}

} // namespace

// waves of a workgroup: one per chunk of slices, as many as the volume has, at
// most MAT_NW
static int mat_waves(const MatArgs &a)
{
	return a.nzc < MAT_NW ? a.nzc : MAT_NW;
}

long mat_blocks(const MatArgs &a)
{
	const int nw = mat_waves(a);
	return nw < 1 ? 0 : (long) ((a.nx + 7) / 8) * ((a.ny + 7) / 8) * ((a.nzc + nw - 1) / nw);
}

template <typename TP, bool HELIX, int WGT, typename IDX>
static hipError_t launch_mat_i(MatArgs a, int nw, unsigned blocks, hipStream_t s)
{
	const size_t lds = nw * (2 * MAT_VIEW_BYTES + MAT_ZC * 8);
	if (a.redo)
		hipLaunchKernelGGL((mat_kernel<TP, HELIX, WGT, IDX, true>), dim3(blocks), dim3(64 * nw),
			lds, s, a);
	hipLaunchKernelGGL((mat_kernel<TP, HELIX, WGT, IDX, false>), dim3(blocks), dim3(64 * nw),
		lds, s, a);
	return hipGetLastError();
}

template <typename TP, bool HELIX, int WGT>
static hipError_t launch_mat_t(const MatArgs &a, hipStream_t s)
{
	const long blocks = mat_blocks(a);
	if (blocks > 0x7fffffffL)
		return hipErrorInvalidValue;
	// 32-bit byte offsets, of 24-bit factors, while a view (and the row past its
	// last) stays below 4 GiB
	const bool small = ((size_t) a.nt + 1) * a.ns * sizeof(TP) < ((size_t) 1 << 32)
		&& a.ns < (1 << 24) && a.nt < (1 << 24);
	return small ? launch_mat_i<TP, HELIX, WGT, uint32_t>(a, mat_waves(a), (unsigned) blocks, s)
		: launch_mat_i<TP, HELIX, WGT, uint64_t>(a, mat_waves(a), (unsigned) blocks, s);
}

template <typename TP>
static hipError_t launch_mat_p(const MatArgs &a, hipStream_t s)
{
	const bool div = a.kind == KIND_ARC;
	if (!a.zrange)
		return div ? launch_mat_t<TP, false, MW_DIV>(a, s) : launch_mat_t<TP, false, MW_MUL>(a, s);
	if (a.cone_par)
		return launch_mat_t<TP, true, MW_NONE>(a, s);
	return div ? launch_mat_t<TP, true, MW_DIV>(a, s) : launch_mat_t<TP, true, MW_MUL>(a, s);
}

hipError_t launch_mat(const MatArgs &a, bool proj_fp64, hipStream_t s)
{
	if (a.nx <= 0 || a.ny <= 0 || a.nzc <= 0)
		return hipSuccess;
	return proj_fp64 ? launch_mat_p<double>(a, s) : launch_mat_p<float>(a, s);
}

} // namespace fdk
