// 2D fan-beam projector kernels for gfx950 (wave64).
//
// Forward projectors are line driven: one lane per detector bin, a loop over
// the image lines (rows for X views, columns for Y views) that integrates a
// contiguous image line over the ray's footprint by direct overlap sums.
// There are no prefix sums (no FP32 cancellation) and no texture hardware.
// Backprojectors are pixel driven gathers: one lane per pixel, a loop over
// views, a register accumulator and a single store; no atomics.
//
// Reference counterparts: DDFPFanKernelX/Y (DistanceDriven.cu:64-196),
// DDBPFanKernelX/Y (:500-614), PreweightBPKernelX/Y (:441-477),
// SiddonFanProjectionKernel / SiddonFanBackprojectionKernel (Siddon.cu:240-382),
// bpFanKernel3D (PixelDriven.cu:11-75).

#include "rn_fan_device.h"
#include "rn_tune.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace rn {

namespace {

using namespace fan;

// ---------------------------------------------------------------------------
// forward projectors (line driven)
// ---------------------------------------------------------------------------

// XCD > 0: 1-D grid whose workgroups are renumbered per XCD (as in
// k_siddon_fan_fp); S slices per lane share the ray's lines and shares.
template <int BLK, int XCD, int S>
__global__ __launch_bounds__(BLK) void k_dd_fan_fp(FanK g, const float* __restrict__ RX,
                                                   const float* __restrict__ RY, float* __restrict__ prj,
                                                   int view0, int nviews, int ns)
{
    int tile, vi, sg;
    if (XCD > 0) {
        const int per = gridDim.x / XCD;
        const int l = (blockIdx.x % XCD) * per + blockIdx.x / XCD;
        const int tiles = (g.nu + BLK - 1) / BLK;
        tile = l % tiles;
        vi = (l / tiles) % nviews;
        sg = l / (tiles * nviews);
    } else {
        tile = blockIdx.x;
        vi = blockIdx.y;
        sg = blockIdx.z;
    }
    const int iu = tile * BLK + threadIdx.x;
    const bool active = iu < g.nu;
    const long plane = (long)g.nx * g.ny;
    const int s0 = sg * S;
    const int nsl = min(S, ns - s0);
    float acc[S];
    dd_fp_ray_slices<float, S>(g, RX + s0 * plane, RY + s0 * plane, plane, nsl, view0 + vi,
                               active ? iu : g.nu - 1, active, acc);
    if (!active) return;
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        if (q >= nsl) break;
        prj[((long)(s0 + q) * nviews + vi) * g.nu + iu] = acc[q];
    }
}

// DD FP of G interleaved groups of 4 slices per lane (padded quad averaged
// planes), H parts of a wave per ray; writes the plain sinograms of the real
// slices [s][nviews][nu].
template <int BLK, int XCD, int G, int H>
__global__ __launch_bounds__(BLK) void k_dd_fan_fp_q(FanK g, const float4* __restrict__ QX,
                                                     const float4* __restrict__ QY, float* __restrict__ prj,
                                                     int view0, int nviews, int ns)
{
    int tile, vi, sg;
    if (XCD > 0) {
        const int per = gridDim.x / XCD;
        const int l = (blockIdx.x % XCD) * per + blockIdx.x / XCD;
        const int tiles = (g.nu + BLK / H - 1) / (BLK / H);
        tile = l % tiles;
        vi = (l / tiles) % nviews;
        sg = l / (tiles * nviews);
    } else {
        tile = blockIdx.x;
        vi = blockIdx.y;
        sg = blockIdx.z;
    }
    const int iu = tile * (BLK / H) + (int)(threadIdx.x >> 6) * (64 / H) + (int)(threadIdx.x & (64 / H - 1));
    const bool active = iu < g.nu;
    const int nquads = (ns + 3) / 4;
    const int q0 = sg * G;
    const int nq = min(G, nquads - q0);
    float4 acc[G];
    dd_fp_ray_quads<G, H>(g, QX + (long)q0 * g.ny * qpitch(g.nx), QY + (long)q0 * g.nx * qpitch(g.ny), nq,
                          view0 + vi, active ? iu : g.nu - 1, active, acc);
    if (!active || (threadIdx.x & 63) >= 64 / H) return;
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        if (k >= nq) break;
        const float v[4] = {acc[k].x, acc[k].y, acc[k].z, acc[k].w};
        #pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int sl = 4 * (q0 + k) + c;
            if (sl < ns) prj[((long)sl * nviews + vi) * g.nu + iu] = v[c];
        }
    }
}

// With meas != nullptr the epilogue writes the weighted residual
// wgt * (Ax - meas) of the OS-SQS data step (ossqs.cu:101-122) instead of Ax.
// Each lane projects its ray through S consecutive slices (the ray's lines,
// cells and weights are shared; the grid's slice index counts groups of S).
template <class T, int BLK, int XCD, int S>
__global__ __launch_bounds__(BLK) void k_siddon_fan_fp(FanK g, const T* __restrict__ Pyx,
                                                       const T* __restrict__ Pxy, T* __restrict__ prj,
                                                       int view0, int nviews, int ns,
                                                       const float* __restrict__ meas, const float* __restrict__ wgt,
                                                       int meas_nviews)
{
    // XCD > 0: 1-D grid of tiles * nviews * slice groups workgroups (a multiple
    // of XCD).  The hardware deals workgroups round-robin to the XCDs, so
    // workgroup h runs on XCD h % XCD; h is renumbered so that each XCD walks a
    // contiguous, slice-major range of (slice group, view, bin tile) and its L2
    // holds the images of only the slices it is working on.
    int tile, vi, sg;
    if (XCD > 0) {
        const int per = gridDim.x / XCD;
        const int l = (blockIdx.x % XCD) * per + blockIdx.x / XCD;
        const int tiles = (g.nu + BLK - 1) / BLK;
        tile = l % tiles;
        vi = (l / tiles) % nviews;
        sg = l / (tiles * nviews);
    } else {
        tile = blockIdx.x;
        vi = blockIdx.y;
        sg = blockIdx.z;
    }
    const int iu = tile * BLK + threadIdx.x;
    const bool active = iu < g.nu;
    const int view = view0 + vi;
    const long plane = (long)g.nx * g.ny;
    const int s0 = sg * S;
    const int nsl = min(S, ns - s0);
    T acc[S];
    siddon_fp_ray_slices<T, S>(g, Pyx + s0 * plane, Pxy + s0 * plane, plane, nsl, view, active ? iu : g.nu - 1,
                               active, acc);
    if (!active) return;
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        if (q >= nsl) break;
        const int s = s0 + q;
        T v = acc[q];
        if (meas != nullptr) {
            const long mi = ((long)s * meas_nviews + view) * g.nu + iu;
            v = (T)wgt[mi] * (v - (T)meas[mi]);
        }
        prj[((long)s * nviews + vi) * g.nu + iu] = v;
    }
}

// ---------------------------------------------------------------------------
// backprojectors (pixel driven gathers)
// ---------------------------------------------------------------------------

// One lane per pixel of S consecutive slices (the grid's z index counts
// groups of S): the bin ranges and weights are shared by the slices.  The views are
// summed in kBpSegs fixed segments whose sums are added in order, as the waves of the
// tile kernels and of the ragged batches do, with the same bits.
template <class T, int BX, int BY, int NB, int S>
__global__ __launch_bounds__(BX * BY) void k_siddon_fan_bp(FanK g, const T* __restrict__ prj,
                                                       T* __restrict__ img, int view0, int nviews, int ns,
                                                       int accumulate)
{
    const int iy = blockIdx.x * BX + threadIdx.x;
    const int ix = blockIdx.y * BY + threadIdx.y;
    const int s0 = blockIdx.z * S;
    const int nsl = min(S, ns - s0);
    if (ix >= g.nx || iy >= g.ny) return;
    const long sstride = (long)nviews * g.nu;
    T acc[S], tot[S];
    #pragma unroll
    for (int q = 0; q < S; ++q) tot[q] = vzero<T>();
    #pragma unroll 1
    for (int seg = 0; seg < kBpSegs; ++seg) {
        const int v0 = (int)((long)nviews * seg / kBpSegs), v1 = (int)((long)nviews * (seg + 1) / kBpSegs);
        siddon_bp_pixel_slices<T, NB, S>(g, prj + s0 * sstride + (long)v0 * g.nu, sstride, nsl, view0 + v0, v1 - v0,
                                         ix, iy, acc);
        #pragma unroll
        for (int q = 0; q < S; ++q) vadd(tot[q], acc[q]);
    }
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        if (q >= nsl) break;
        T* o = img + (long)(s0 + q) * g.nx * g.ny + (long)ix * g.ny + iy;
        *o = accumulate ? *o + tot[q] : tot[q];
    }
}

// Quad-layout Siddon FP + residual: each lane carries G groups of 4 slices
// (one float4 load per cell and group); the grid's slice index counts groups
// of G quads.  res = w * (Ax - meas) per component, or with PLAIN the plain
// sinograms prj = Ax of the real slices [s][nviews][nu].
template <int BLK, int XCD, int G, int H, bool PLAIN>
__global__ __launch_bounds__(BLK) void k_siddon_fan_fp_q(FanK g, const float4* __restrict__ Qyx,
                                                         const float4* __restrict__ Qxy, float4* __restrict__ res,
                                                         float* __restrict__ prj, int view0, int nviews, int ns,
                                                         const float4* __restrict__ meas,
                                                         const float4* __restrict__ wgt, int meas_nviews,
                                                         int res_vstride, int res_voff)
{
    int tile, vi, sg;
    if (XCD > 0) {
        const int per = gridDim.x / XCD;
        const int l = (blockIdx.x % XCD) * per + blockIdx.x / XCD;
        const int tiles = (g.nu + BLK / H - 1) / (BLK / H);
        tile = l % tiles;
        vi = (l / tiles) % nviews;
        sg = l / (tiles * nviews);
        if (sg * G >= (ns + 3) / 4) return;   // the grid is rounded up to whole rounds of XCDs
    } else {
        tile = blockIdx.x;
        vi = blockIdx.y;
        sg = blockIdx.z;
    }
    // H > 1: each wave carries 64 / H rays H times (one part of the lines each)
    const int iu = tile * (BLK / H) + (int)(threadIdx.x >> 6) * (64 / H) + (int)(threadIdx.x & (64 / H - 1));
    const bool active = iu < g.nu;
    const int view = view0 + vi;
    const int nquads = (ns + 3) / 4;
    const int q0 = sg * G;
    const int nq = min(G, nquads - q0);
    float4 acc[G];
    siddon_fp_ray_quads<G, H>(g, Qyx + (long)q0 * g.ny * qpitch(g.nx), Qxy + (long)q0 * g.nx * qpitch(g.ny), nq, view,
                           active ? iu : g.nu - 1, active, acc);
    if (!active || (threadIdx.x & 63) >= 64 / H) return;
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        if (k >= nq) break;
        if constexpr (PLAIN) {
            const float v[4] = {acc[k].x, acc[k].y, acc[k].z, acc[k].w};
            #pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int sl = 4 * (q0 + k) + c;
                if (sl < ns) prj[((long)sl * nviews + vi) * g.nu + iu] = v[c];
            }
            continue;
        }
        const long mi = ((long)(q0 + k) * meas_nviews + view) * g.nu + iu;
        const float4 m = meas[mi], w = wgt[mi];
        res[((long)(q0 + k) * res_vstride + res_voff + vi) * g.nu + iu] =
            make_float4(w.x * (acc[k].x - m.x), w.y * (acc[k].y - m.y), w.z * (acc[k].z - m.z),
                        w.w * (acc[k].w - m.w));
    }
}

// Quad-layout Siddon BP: one lane per pixel of G groups of 4 slices (one
// float4 load per bin and group); writes the plain images of the real slices.
// SEG: the views in nseg segments, as many as the tile kernels' waves, whose sums are
// added in order, with the same bits; else all views in one sum.
template <int BX, int BY, int NB, int G, bool SEG>
__global__ __launch_bounds__(BX * BY) void k_siddon_fan_bp_q(FanK g, const float4* __restrict__ prj,
                                                         float* __restrict__ img, int view0, int nviews, int ns,
                                                         int nseg)
{
    const int iy = blockIdx.x * BX + threadIdx.x;
    const int ix = blockIdx.y * BY + threadIdx.y;
    const int nquads = (ns + 3) / 4;
    const int q0 = blockIdx.z * G;
    const int nq = min(G, nquads - q0);
    if (ix >= g.nx || iy >= g.ny) return;
    const long sstride = (long)nviews * g.nu;
    const float4* P = prj + q0 * sstride;
    float4 acc[G];
    if constexpr (SEG) {
        float4 sum[G];
        #pragma unroll 1
        for (int seg = 0; seg < nseg; ++seg) {
            const int v0 = (int)((long)nviews * seg / nseg), v1 = (int)((long)nviews * (seg + 1) / nseg);
            siddon_bp_pixel_slices<float4, NB, G>(g, P + (long)v0 * g.nu, sstride, nq, view0 + v0, v1 - v0, ix, iy, sum);
            #pragma unroll
            for (int k = 0; k < G; ++k) {
                if (seg == 0) acc[k] = sum[k];
                else vadd(acc[k], sum[k]);
            }
        }
    } else {
        siddon_bp_pixel_slices<float4, NB, G>(g, P, sstride, nq, view0, nviews, ix, iy, acc);
    }
    const long plane = (long)g.nx * g.ny, pix = (long)ix * g.ny + iy;
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        if (k >= nq) break;
        const int s = 4 * (q0 + k);
        const float v[4] = {acc[k].x, acc[k].y, acc[k].z, acc[k].w};
        #pragma unroll
        for (int c = 0; c < 4; ++c)
            if (s + c < ns) img[(long)(s + c) * plane + pix] = v[c];
    }
}

// A lane's G groups of 4 slices of pixel (ix, iy): stored to the plain images
// img, or with UPD the OS-SQS update applied to them instead (sqs_update_core per
// slice, the arithmetic of k_sqs_update_q): the current image and its 4-neighbours
// are read as float4 groups from the interleaved copy u.Qold, the normaliser from
// u.D4, and the new image goes to u.Xn and, as float4 per group, to the other
// interleaved copies u.Qxy, u.Qyx (the launch reads none of the buffers it writes).
template <int G, bool UPD>
__device__ __forceinline__ void store_or_update(const FanK& g, const float4 (&acc)[G], float* __restrict__ img,
                                                const SqsUpd& u, int ix, int iy, int q0, int nq, int ns)
{
    const long plane = (long)g.nx * g.ny, pix = (long)ix * g.ny + iy;
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        if (k >= nq) break;
        const int s = 4 * (q0 + k);
        float v[4] = {acc[k].x, acc[k].y, acc[k].z, acc[k].w};
        if constexpr (UPD) {
            const int pxy = qpitch(g.ny), pyx = qpitch(g.nx);
            const float4* qo = u.Qold + (long)(q0 + k) * g.nx * pxy;
            const long c0 = (long)ix * pxy + kQPadL + iy;
            const float4 xc = qo[c0];
            // neighbours for the TV terms (padded lines: iy - 1 and iy + 1 stay inside
            // the line; the border cases below use the pixel value itself, as the
            // plain update)
            float4 xl = xc, xr = xc, yl = xc, yr = xc;
            if (u.beta2 != 0.0f) {
                if (ix > 0) xl = qo[c0 - pxy];
                if (ix < g.nx - 1) xr = qo[c0 + pxy];
                yl = qo[c0 - 1];
                yr = qo[c0 + 1];
            }
            const float4 d4 = u.D4[(long)(q0 + k) * plane + pix];
            const float xs[4] = {xc.x, xc.y, xc.z, xc.w}, xls[4] = {xl.x, xl.y, xl.z, xl.w};
            const float xrs[4] = {xr.x, xr.y, xr.z, xr.w}, yls[4] = {yl.x, yl.y, yl.z, yl.w};
            const float yrs[4] = {yr.x, yr.y, yr.z, yr.w}, ds[4] = {d4.x, d4.y, d4.z, d4.w};
            #pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float x = xs[c];
                const float dx0 = ix == 0 ? x : x - xls[c], dx1 = ix == g.nx - 1 ? x : x - xrs[c];
                const float dy0 = iy == 0 ? x : x - yls[c], dy1 = iy == g.ny - 1 ? x : x - yrs[c];
                float xn = 0.0f;
                if (s + c < ns) {
                    xn = sqs_update_core(x, dx0, dx1, dy0, dy1, v[c], ds[c], u.step, u.beta2, u.eps, u.lb, u.ub,
                                         u.crop);
                    u.Xn[(long)(s + c) * plane + pix] = xn;
                }
                v[c] = xn;
            }
            const float4 f = make_float4(v[0], v[1], v[2], v[3]);
            u.Qxy[(long)(q0 + k) * g.nx * pxy + (long)ix * pxy + kQPadL + iy] = f;
            u.Qyx[(long)(q0 + k) * g.ny * pyx + (long)iy * pyx + kQPadL + ix] = f;
        } else {
            #pragma unroll
            for (int c = 0; c < 4; ++c)
                if (s + c < ns) img[(long)(s + c) * plane + pix] = v[c];
        }
    }
}

// The Siddon BP of an 8 x 8-pixel tile of G interleaved slice groups, for geometries
// with FanK::tile.  The views are split evenly over the workgroup's nw waves; the
// waves' sums are added in LDS in wave order.  Per view the tile's bins of the G
// groups and of the view's ray table, CAP at a time, are loaded once per wave with
// coalesced dwordx4 loads, issued one step (a view, or a further CAP bins of it) ahead
// into registers, written to the wave's own LDS rows and gathered from there by every
// pixel: a fraction of the per-pixel gathers' vector-memory traffic.  One gather
// code for every step (no branch around the accumulators, which would cost copies
// of them): the step before the first takes no bin of the cleared rows.  A wave
// touches only its own rows and the LDS instructions of one wave execute in order, so
// the steps need no barrier; the fences keep the compiler from moving LDS accesses
// across the handovers.  The group rows are addressed as 32-bit byte offsets from the
// groups' base (the launcher checks that G groups fit).
//
// UPD: the epilogue applies the OS-SQS update instead of storing the gradient
// (store_or_update).
//
// Bound: LDS reads (nine per bin with 8 groups, 8 clocks each and shared by four
// SIMDs) and VALU (about 200 instructions, 64 to 96 of them FMAs).  ms, before (bin
// ranges per pixel through an atan, window as the lanes' minimum and maximum) ->
// now: 32 slices of 512^2, 96 views 0.168 -> 0.146; 16 slices, 1152 views 1.50 ->
// 1.27; 32 slices of 250^2, 360 views 0.40 -> 0.15; 6 slices of 256^2 0.28 -> 0.094.
extern __shared__ float4 dyn4[];

template <int G, int CAP, bool UPD>
__global__ __launch_bounds__(512, 4) void k_siddon_fan_bp_tile(FanK g, const float4* __restrict__ prj,
                                                               float* __restrict__ img, int view0, int nviews, int ns,
                                                               SqsUpd u)
{
    static_assert(CAP <= 64, "one load for the ray table row");
    // LDS rows 0 .. G - 1: the groups; row G: the ray table
    constexpr int CS = stage_pitch(CAP), kLds = (G + 1) * CS, kLoads = (G * CAP + 63) / 64;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y), nw = blockDim.y;
    const int tx = blockIdx.y * 8, ty = blockIdx.x * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7);
    float4* st = dyn4 + wv * kLds;
    for (int i = lane; i < kLds; i += 64) st[i] = vzero<float4>();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const bool inside = ix < g.nx && iy < g.ny;   // lanes outside stage but gather nothing
    const int q0 = blockIdx.z * G, nq = min(G, (ns + 3) / 4 - q0);
    const long sstride = (long)nviews * g.nu;
    const float4* P = prj + q0 * sstride;
    const float4* const sray = g.sray + (long)view0 * g.nu;
    const float yr = (float)iy - 0.5f * g.ny, xr = (float)ix - 0.5f * g.nx;
    float4 acc[G];
    #pragma unroll
    for (int q = 0; q < G; ++q) acc[q] = vzero<float4>();
    // staging load j of this lane: element i = 64 j + lane of the group rows, that is
    // group i / CAP, bin i % CAP of the window; the ray table row is one
    // more load by the first CAP lanes
    int bj[kLoads], slot[kLoads];   // slot: the zero entries of the rows before
    unsigned roff[kLoads];
    #pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int i = j * 64 + lane;
        bj[j] = i % CAP;
        slot[j] = G == 1 ? 0 : i / CAP;
        roff[j] = (unsigned)(min(i / CAP, nq - 1) * sstride) * 16u;
    }
    TileRange tr;
    tr.init(g, lane);
    float4 rg[kLoads], rr;
    int t0 = 0, t1 = -1;   // the step's bins (relative to its first one)
    bool xv = true;
    const int v0 = (int)((long)nviews * wv / nw), v1 = (int)((long)nviews * (wv + 1) / nw);
    int vi = v0 - 1, base = 0, span = -1, off = 0;
    for (bool more = true;;) {
        const int a0 = max(t0, 0), a1 = min(t1, CAP - 1);
        const float lr = xv ? yr : xr, cell = xv ? xr + 0.5f * g.nx : yr + 0.5f * g.ny;
        if (off + CAP <= span) {
            off += CAP;
            t0 -= CAP;
            t1 -= CAP;
        } else {
            off = 0;
            do {
                more = ++vi < v1;
                if (!more) break;
                if (((vi - v0) & 63) == 0) tr.batch(g, view0 + vi, lane, tx, ty, 0.0f);
                span = __builtin_amdgcn_readlane(tr.span, (vi - v0) & 63);
            } while (span < 0);
            if (more) {
                const int w = (vi - v0) & 63;
                base = __builtin_amdgcn_readlane(tr.base, w);
                tr.range(w, span, t0, t1);
                if (!inside) t1 = -1;
                xv = g.vcls[view0 + vi] == 0;
            }
        }
        if (more) {
            #pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP)
                    rg[j] = ld_at(P, roff[j] + (unsigned)(vi * g.nu + min(base + off + bj[j], g.nu - 1)) * 16u);
            if (lane < CAP) rr = ld_at(sray, (unsigned)(vi * g.nu + min(base + off + lane, g.nu - 1)) * 16u);
        }
        siddon_gather_staged<G, CAP>(st, a0, a1, lr, cell, acc);
        if (!more) break;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        #pragma unroll
        for (int j = 0; j < kLoads; ++j)
            if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP) st[j * 64 + lane + slot[j]] = rg[j];
        if (lane < CAP) st[G * CS + lane] = rr;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if (add_waves<G>(acc, dyn4 + nw * kLds, lane, wv, nw) && inside)
        store_or_update<G, UPD>(g, acc, img, u, ix, iy, q0, nq, ns);
}

// The same for one group of slices, whose bins cost less to gather from memory than
// to stage (nothing shares a window's loads): 96 views of 512^2 66 us, staged 79;
// 30 views of 256^2 12 and 14.
template <int NB, bool UPD>
__global__ __launch_bounds__(512) void k_siddon_fan_bp_tile1(FanK g, const float4* __restrict__ prj,
                                                             float* __restrict__ img, int view0, int nviews, int ns,
                                                             SqsUpd u)
{
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y), nw = blockDim.y;
    const int tx = blockIdx.y * 8, ty = blockIdx.x * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7), q0 = blockIdx.z;
    float4 acc[1] = {vzero<float4>()};
    siddon_bp_tile1<NB>(g, prj + (long)q0 * nviews * g.nu, view0, (int)((long)nviews * wv / nw),
                        (int)((long)nviews * (wv + 1) / nw), tx, ty, lane, acc);
    if (add_waves<1>(acc, dyn4, lane, wv, nw) && ix < g.nx && iy < g.ny)
        store_or_update<1, UPD>(g, acc, img, u, ix, iy, q0, 1, ns);
}

// Exact DD adjoint (dd_adj_tile): a workgroup takes an 8 x 8-pixel tile of G
// groups of 4 slices with kBpSegs waves that walk one view segment each; their
// sums are added in LDS in segment order.
//
// Bound: VALU and LDS reads (per wave and view about 60 instructions for the bin
// range and the staging, 20 per candidate bin and 4 per bin and group).  ms, per-slice
// gathers from memory -> bin ranges per pixel through an atan -> now: 32 slices of
// 256^2, 360 views, 512 bins 1.69 -> 0.41 -> 0.28; of 512^2, 1152 views 16.2 -> 3.1 ->
// 2.4; one slice of 256^2 0.65 -> 0.122 -> 0.109.
template <int G, int CAP, bool WIDE>
__global__ __launch_bounds__(64 * kBpSegs, 4) void k_dd_fan_adj(FanK g, const float4* __restrict__ wprj,
                                                                   float* __restrict__ img, int ns)
{
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int ty = blockIdx.x * 8, tx = blockIdx.y * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7);
    const int q0 = blockIdx.z * G, nq = min(G, (ns + 3) / 4 - q0);
    const long sstride = (long)g.nview * g.nu;
    float4 tot[G];
    dd_adj_tile<G, CAP, 3, WIDE>(g, wprj + q0 * sstride, sstride, nq, g.nview, wv, tx, ty, lane,
                                 dyn4 + wv * DdAdjStage<G, CAP>::kFloat4, tot);
    if (add_waves<G>(tot, dyn4 + kBpSegs * DdAdjStage<G, CAP>::kFloat4, lane, wv, kBpSegs) && ix < g.nx &&
        iy < g.ny)
        store_or_update<G, false>(g, tot, img, SqsUpd{}, ix, iy, q0, nq, ns);
}

// PreweightBPKernelX/Y: length factor for the iterative (non-FBP) DD BP.
__global__ void k_dd_preweight(FanK g, const float* __restrict__ prj, float* __restrict__ wprj)
{
    const int iu = blockIdx.x * blockDim.x + threadIdx.x;
    const int view = blockIdx.y;
    const int s = blockIdx.z;
    if (iu >= g.nu) return;
    const float ct = g.vcos[view], st = g.vsin[view];
    float f;
    if (g.vcls[view] == 0) f = g.dy / fabsf(ct * g.bcos[iu] + st * g.bsin[iu]);   // cos(t - a)
    else f = g.dx / fabsf(st * g.bcos[iu] - ct * g.bsin[iu]);                      // sin(t - a)
    const long i = ((long)s * g.nview + view) * g.nu + iu;
    wprj[i] = prj[i] * f;
}

// Reference-parity DD BP (DDBPFanKernelX/Y) of geometries without FanK::tile_dd: pixel
// edges projected through
// atan, average of the (pre-weighted) detector row over the footprint.  One
// lane per pixel of S consecutive slices (grid z counts groups of S): the
// footprint and the FBP weight are computed once for the S slices (their
// quotients through 1-ulp reciprocals).
// The pixel's S slices (value type T: float, or float4 for 4 interleaved
// slices) over every view: rows[q] are the wave-uniform bases of the S
// pre-weighted [view][nu] sinograms.
template <class T, int S>
__device__ __forceinline__ void dd_bp_pixel(const FanK& g, const T* const (&rows)[S], int ix, int iy, int fbp,
                                            T (&acc)[S])
{
    const float x = (ix - 0.5f * (g.nx - 1)) * g.dx, y = (iy - 0.5f * (g.ny - 1)) * g.dy;
    const float inv_da = 1.0f / g.da;
    const float boff = 0.5f * g.nu - g.off_a;
    #pragma unroll
    for (int q = 0; q < S; ++q) acc[q] = vzero<T>();
    for (int view = 0; view < g.nview; ++view) {
        const float ct = g.vcos[view], st = g.vsin[view];
        const float rx = x * ct + y * st, ry = -x * st + y * ct;
        float ex, ey;   // edge offset (rotated frame) of +-half a pixel
        if (g.vcls[view] == 0) { ex = 0.5f * g.dx * ct; ey = -0.5f * g.dx * st; }
        else                   { ex = 0.5f * g.dy * st; ey = 0.5f * g.dy * ct; }
        const float b1 = boff - atanf((rx - ex) * __builtin_amdgcn_rcpf(ry - ey + g.dso)) * inv_da;
        const float b2 = boff - atanf((rx + ex) * __builtin_amdgcn_rcpf(ry + ey + g.dso)) * inv_da;
        float fw = 1.0f;
        if (fbp) {
            const float d = g.dso + ry;
            fw = g.dso * g.dso * __builtin_amdgcn_rcpf(fmaf(rx, rx, d * d));
        }
        seg_acc_rows<T, S>(rows, (unsigned)(view * g.nu) * (unsigned)sizeof(T), g.nu, fminf(b1, b2),
                           fmaxf(b1, b2), fw, acc);
    }
}

template <int BX, int BY, int S>
__global__ __launch_bounds__(BX * BY) void k_dd_fan_bp(FanK g, const float* __restrict__ wprj,
                                                   float* __restrict__ img, int ns, int fbp)
{
    const int iy = blockIdx.x * BX + threadIdx.x;
    const int ix = blockIdx.y * BY + threadIdx.y;
    const int s0 = blockIdx.z * S;
    const int nsl = min(S, ns - s0);
    if (ix >= g.nx || iy >= g.ny) return;
    const long sstride = (long)g.nview * g.nu;
    const float* rows[S];   // wave-uniform slice bases
    #pragma unroll
    for (int q = 0; q < S; ++q) rows[q] = wprj + (long)(s0 + min(q, nsl - 1)) * sstride;
    float acc[S];
    dd_bp_pixel<float, S>(g, rows, ix, iy, fbp, acc);
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        if (q >= nsl) break;
        img[(long)(s0 + q) * g.nx * g.ny + (long)ix * g.ny + iy] = acc[q];
    }
}

// The same on 4-slice interleaved sinograms [q][view][nu] (float4): G groups
// per lane; writes the plain images of the real slices.
template <int BX, int BY, int G>
__global__ __launch_bounds__(BX * BY) void k_dd_fan_bp_q(FanK g, const float4* __restrict__ wprj,
                                                     float* __restrict__ img, int ns, int fbp)
{
    const int iy = blockIdx.x * BX + threadIdx.x;
    const int ix = blockIdx.y * BY + threadIdx.y;
    const int nquads = (ns + 3) / 4;
    const int q0 = blockIdx.z * G;
    const int nq = min(G, nquads - q0);
    if (ix >= g.nx || iy >= g.ny) return;
    const long sstride = (long)g.nview * g.nu;
    const float4* rows[G];
    #pragma unroll
    for (int k = 0; k < G; ++k) rows[k] = wprj + (long)(q0 + min(k, nq - 1)) * sstride;
    float4 acc[G];
    dd_bp_pixel<float4, G>(g, rows, ix, iy, fbp, acc);
    store_or_update<G, false>(g, acc, img, SqsUpd{}, ix, iy, q0, nq, ns);
}

// The footprint of the lane's pixel in one view of a TileProj batch (l: the view's
// lane): [lo, hi] relative to the tile's first bin, between the projections of the
// pixel's edges along x (X views) or y, and the view's weight over the footprint's
// width, kr / (r / r0)^2 / (hi - lo) with fbp, else 1 / (hi - lo).  FanK::tile_dd keeps
// the width above 1e-3 bins.
__device__ __forceinline__ void dd_bp_footprint(const FanK& g, const TileProj& tp, int l, int cls, float inv_da, int fbp,
                                                float& lo, float& hi, float& k)
{
    const float P = lane_f(tp.P, l), Q = lane_f(tp.Q, l), u0 = lane_f(tp.u0, l);
    const float en = cls == 0 ? P * (0.5f * g.dx) : Q * (0.5f * g.dy);
    const float ed = cls == 0 ? -Q * (0.5f * g.dx) : P * (0.5f * g.dy);
    const float num = fmaf(P, tp.px, Q * tp.py), den = fmaf(P, tp.py, fmaf(-Q, tp.px, 1.0f));
    auto bin = [&](float nn, float dd) {
        const float z = nn * __builtin_amdgcn_rcpf(dd), s = z * z;   // atan z to 5e-9 at |z| = 0.15
        return fmaf(z * inv_da, -fmaf(s, fmaf(s, fmaf(s, -1.0f / 7.0f, 0.2f), -1.0f / 3.0f), 1.0f), u0);
    };
    const float b1 = bin(num - en, den - ed), b2 = bin(num + en, den + ed);
    lo = fminf(b1, b2);
    hi = fmaxf(b1, b2);
    const float w = hi - lo;
    k = fbp ? lane_f(tp.kr, l) * __builtin_amdgcn_rcpf(fmaf(num, num, den * den) * w) : __builtin_amdgcn_rcpf(w);
}

// The DD BP of an 8 x 8-pixel tile of G interleaved slice groups, for geometries
// with FanK::tile_dd.  The views are split evenly over the workgroup's nw waves; the
// waves' sums are added in LDS in wave order.  Per view the tile's bins of the G
// groups' pre-weighted rows, CAP at a time, are loaded once per wave with coalesced
// dwordx4 loads, issued one step (a view, or a further CAP bins of it) ahead into
// registers, written to the wave's own LDS rows and averaged from there by every
// pixel.  One gather code for every step (no branch around the accumulators, which
// would cost copies of them): the step before the first adds zeros times the
// cleared rows.  A wave touches only its own rows and the LDS instructions of one
// wave execute in order, so the steps need no barrier; the fences keep the compiler
// from moving LDS accesses across the handovers.  The group rows are addressed as
// 32-bit byte offsets from the groups' base (the launcher checks that G groups fit).
//
// Bound: LDS reads (three bins of 8 groups per pixel and view are 192 clocks of a
// wave's 757) and VALU (195 instructions).  32 slices of 512^2, 1152 views, 736 bins,
// FBP: 2.27 -> 1.70 ms; before, every pixel's two edges went through atanf and the
// window was the lanes' minimum and maximum (386 instructions), and batches that fill
// no 8 groups or tiles that fill no chip read the bins per pixel from memory
// (256^2, 360 views, 1 and 32 slices: 0.20 -> 0.07, 0.39 -> 0.17 ms).
template <int G, int CAP>
__global__ __launch_bounds__(512, 4) void k_dd_fan_bp_tile(FanK g, const float4* __restrict__ wprj,
                                                           float* __restrict__ img, int ns, int fbp)
{
    constexpr int kLds = G * stage_pitch(CAP), kLoads = (G * CAP + 63) / 64;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y), nw = blockDim.y;
    const int tx = blockIdx.y * 8, ty = blockIdx.x * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7);
    float4* st = dyn4 + wv * kLds;
    for (int i = lane; i < kLds; i += 64) st[i] = vzero<float4>();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const bool inside = ix < g.nx && iy < g.ny;   // lanes outside stage but gather nothing
    const int q0 = blockIdx.z * G, nq = min(G, (ns + 3) / 4 - q0);
    const long sstride = (long)g.nview * g.nu;
    const float4* P = wprj + q0 * sstride;
    float4 acc[G];
    #pragma unroll
    for (int q = 0; q < G; ++q) acc[q] = vzero<float4>();
    // staging load j of this lane: element i = 64 j + lane, row i / CAP, bin
    // i % CAP (LDS slot i)
    int bj[kLoads], slot[kLoads];   // slot: the zero entries of the rows before
    unsigned roff[kLoads];
    #pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int i = j * 64 + lane;
        bj[j] = i % CAP;
        slot[j] = G == 1 ? 0 : i / CAP;
        roff[j] = (unsigned)(min(i / CAP, nq - 1) * sstride) * 16u;
    }
    const float inv_da = 1.0f / g.da;
    TileProj tp;
    tp.init(g, lane);
    float4 rg[kLoads];
    float lo = 0.0f, hi = -1.0f, k = 0.0f;   // the step's interval (relative to its first bin) and scale
    const int v0 = (int)((long)g.nview * wv / nw), v1 = (int)((long)g.nview * (wv + 1) / nw);
    int view = v0 - 1, base = 0, span = -1, off = 0;
    for (bool more = true;;) {
        const float l = lo, h = hi, kk = k;
        if (off + CAP <= span) {
            off += CAP;
            lo -= (float)CAP;
            hi -= (float)CAP;
        } else {
            off = 0;
            do {
                more = ++view < v1;
                if (!more) break;
                if (((view - v0) & 63) == 0) tp.batch(g, view, lane, tx, ty, 0.5 * g.nu - (double)g.off_a);
                span = __builtin_amdgcn_readlane(tp.span, (view - v0) & 63);
            } while (span < 0);
            if (more) {
                const int w = (view - v0) & 63;
                base = __builtin_amdgcn_readlane(tp.base, w);
                dd_bp_footprint(g, tp, w, g.vcls[view], inv_da, fbp, lo, hi, k);
                hi = inside ? fminf(hi, (float)(g.nu - base)) : -1.0f;
            }
        }
        if (more) {
            #pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP)
                    rg[j] = ld_at(P, roff[j] + (unsigned)(view * g.nu + min(base + off + bj[j], g.nu - 1)) * 16u);
        }
        seg_rel_staged<G, CAP>(st, l, h, (float)CAP, kk, acc);
        if (!more) break;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        #pragma unroll
        for (int j = 0; j < kLoads; ++j)
            if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP) st[j * 64 + lane + slot[j]] = rg[j];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if (add_waves<G>(acc, dyn4 + nw * kLds, lane, wv, nw) && inside)
        store_or_update<G, false>(g, acc, img, SqsUpd{}, ix, iy, q0, nq, ns);
}

// bpFanKernel3D with isFBP = true (the only mode the reference launches).
// Pixel-driven FBP backprojection (PixelDriven.cu:11-75): one pixel of S
// slices per lane; the view's detector coordinate (an atan), the linear
// interpolation weights and the FBP weight dso^2 / (rx^2 + (dso + ry)^2) are
// computed once and applied to the S slices, each with the arithmetic of a
// one-slice call (a tail group reads its last slice again and discards it).
template <int BX, int BY, int S>
__global__ __launch_bounds__(BX * BY) void k_pixel_fan_bp(FanK g, const float* __restrict__ prj,
                                                      float* __restrict__ img, int ns)
{
    const int iy = blockIdx.x * BX + threadIdx.x;
    const int ix = blockIdx.y * BY + threadIdx.y;
    const int s0 = blockIdx.z * S;
    if (ix >= g.nx || iy >= g.ny) return;
    const int nsl = min(S, ns - s0);
    const float x = (ix - 0.5f * (g.nx - 1)) * g.dx, y = (iy - 0.5f * (g.ny - 1)) * g.dy;
    const float inv_da = 1.0f / g.da;
    const long sstride = (long)g.nview * g.nu;
    float acc[S];
    #pragma unroll
    for (int q = 0; q < S; ++q) acc[q] = 0.0f;
    for (int view = 0; view < g.nview; ++view) {
        const float ct = g.vcos[view], st = g.vsin[view];
        const float rx = x * ct + y * st, ry = -x * st + y * ct;
        const float d = ry + g.dso;
        const float pu = g.cu - g.off_a - atanf(rx * __builtin_amdgcn_rcpf(d)) * inv_da;
        const float f0 = floorf(pu);
        const int i0 = (int)f0;
        const float f = pu - f0;
        const float w = g.dso * g.dso * __builtin_amdgcn_rcpf(fmaf(rx, rx, d * d));
        const bool in0 = i0 >= 0 && i0 < g.nu, in1 = i0 + 1 >= 0 && i0 + 1 < g.nu;
        const float* p = prj + ((long)s0 * g.nview + view) * g.nu;
        #pragma unroll
        for (int q = 0; q < S; ++q) {
            const float* pq = p + (long)min(q, nsl - 1) * sstride;
            const float v0 = in0 ? pq[i0] : 0.0f;
            const float v1 = in1 ? pq[i0 + 1] : 0.0f;
            acc[q] += ((1.0f - f) * v0 + f * v1) * w;
        }
    }
    #pragma unroll
    for (int q = 0; q < S; ++q)
        if (q < nsl) img[(long)(s0 + q) * g.nx * g.ny + (long)ix * g.ny + iy] = acc[q];
}

// ---------------------------------------------------------------------------
// layout helpers
// ---------------------------------------------------------------------------

// q_same[q][i][j] = (in[4q][i][j], .., in[4q+3][i][j]) (zero past nslices) and,
// if q_tr, q_tr[q][j][i] = the same value; 32 x 32 tiles through LDS.  Output
// lines have pitch p_same / p_tr and start off cells into the line.
// len (optional): the transposed values times len[j][i].z.
__global__ __launch_bounds__(256) void k_pack_quads(const float* __restrict__ in, float4* __restrict__ q_same,
                                                    float4* __restrict__ q_tr, int n1, int n2, int ns, int p_same,
                                                    int p_tr, int off, const float4* __restrict__ len)
{
    __shared__ float4 tile[32][33];
    const int j0 = blockIdx.x * 32, i0 = blockIdx.y * 32, q = blockIdx.z;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const long plane = (long)n1 * n2;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, j = j0 + tx;
        if (i < n1 && j < n2) {
            float v[4];
            #pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int s = 4 * q + c;
                v[c] = s < ns ? in[(long)s * plane + (long)i * n2 + j] : 0.0f;
            }
            const float4 f = make_float4(v[0], v[1], v[2], v[3]);
            tile[r][tx] = f;
            if (q_same != nullptr) q_same[(long)q * n1 * p_same + (long)i * p_same + off + j] = f;
        }
    }
    if (q_tr == nullptr) return;
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int j = j0 + r, i = i0 + tx;
        if (i < n1 && j < n2) {
            float4 f = tile[tx][r];
            if (len != nullptr) f = vscale(f, len[(long)j * n1 + i].z);
            q_tr[(long)q * n2 * p_tr + (long)j * p_tr + off + i] = f;
        }
    }
}

// Both padded quad orientations of 32 x 32-cell tiles of the images (AVG: of their
// averaged planes, the previous row for q_same and the previous column for q_tr,
// zero before the first), pad cells written as zeros by the border tiles.
//
// Bound: HBM (one read of the images, two padded quad copies written).  32 slices
// of 256^2, AVG: 7.7 us (6 TB/s) against 30 us for five launches (fill, two averages, two packs).
template <bool AVG>
__global__ __launch_bounds__(256) void k_pack_planes(const float* __restrict__ in, float4* __restrict__ q_same,
                                                     float4* __restrict__ q_tr, int n1, int n2, int ns)
{
    __shared__ float4 tile[33][33];   // [1 + row][1 + column], index 0: the previous row / column
    const int j0 = blockIdx.x * 32, i0 = blockIdx.y * 32, q = blockIdx.z;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int p_same = qpitch(n2), p_tr = qpitch(n1);
    const long plane = (long)n1 * n2;
    auto cell = [&](int i, int j) {
        float v[4];
        #pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int s = 4 * q + c;
            v[c] = s < ns && i >= 0 && j >= 0 && i < n1 && j < n2 ? in[(long)s * plane + (long)i * n2 + j] : 0.0f;
        }
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    auto mean = [](float4 a, float4 b) {
        return make_float4(0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z), 0.5f * (a.w + b.w));
    };
    #pragma unroll
    for (int r = 0; r < 32; r += 8) tile[1 + ty + r][1 + tx] = cell(i0 + ty + r, j0 + tx);
    if (AVG && ty == 0) tile[0][1 + tx] = cell(i0 - 1, j0 + tx);
    if (AVG && ty == 1) tile[1 + tx][0] = cell(i0 + tx, j0 - 1);
    __syncthreads();
    float4* os = q_same + (long)q * n1 * p_same + kQPadL;
    float4* ot = q_tr + (long)q * n2 * p_tr + kQPadL;
    #pragma unroll
    for (int r = ty; r < 32; r += 8) {
        int i = i0 + r, j = j0 + tx;
        if (i < n1 && j < n2)
            os[(long)i * p_same + j] = AVG ? mean(tile[r][1 + tx], tile[1 + r][1 + tx]) : tile[1 + r][1 + tx];
        i = i0 + tx;
        j = j0 + r;
        if (i < n1 && j < n2)
            ot[(long)j * p_tr + i] = AVG ? mean(tile[1 + tx][r], tile[1 + tx][1 + r]) : tile[1 + tx][1 + r];
    }
    // pads: row tx of the tile, pad cell ty
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (blockIdx.x == 0 && i0 + tx < n1 && ty < kQPadL) os[(long)(i0 + tx) * p_same - kQPadL + ty] = z;
    if (blockIdx.x == gridDim.x - 1 && i0 + tx < n1 && ty < kQPadR) os[(long)(i0 + tx) * p_same + n2 + ty] = z;
    if (blockIdx.y == 0 && j0 + tx < n2 && ty < kQPadL) ot[(long)(j0 + tx) * p_tr - kQPadL + ty] = z;
    if (blockIdx.y == gridDim.y - 1 && j0 + tx < n2 && ty < kQPadR) ot[(long)(j0 + tx) * p_tr + n1 + ty] = z;
}

__global__ __launch_bounds__(256) void k_permute_rows(const float* __restrict__ in, float* __restrict__ out,
                                                      const int* __restrict__ perm, int rows, int cols)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, b = blockIdx.z;
    if (c >= cols) return;
    out[((long)b * rows + j) * cols + c] = in[((long)b * rows + perm[j]) * cols + c];
}

__global__ __launch_bounds__(256) void k_transpose(const float* __restrict__ in, float* __restrict__ out,
                                                   int rows, int cols)
{
    __shared__ float tile[32][33];
    const long base = (long)blockIdx.z * rows * cols;
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + threadIdx.x;
        if (r < rows && c < cols) tile[k][threadIdx.x] = in[base + (long)r * cols + c];
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int c = c0 + k, r = r0 + threadIdx.x;
        if (r < rows && c < cols) out[base + (long)c * rows + r] = tile[threadIdx.x][k];
    }
}

// ry[s][i][j] = (in[i-1][j] + in[i][j]) / 2 and rx[s][j][i] = (in[i][j-1] + in[i][j]) / 2 of
// n0 x n1 images (zero before the first row and column), 32 x 32 tiles through LDS.
// Bound: launches at one slice (128^2: 4.0 us, and 8.6 us in three: two averages, one
// through memory to a transpose), else HBM.
__global__ __launch_bounds__(256) void k_avg_planes(const float* __restrict__ in, float* __restrict__ ry,
                                                    float* __restrict__ rx, int n0, int n1)
{
    __shared__ float tile[33][34];   // [1 + row][1 + column], index 0: the previous row / column
    const int j0 = blockIdx.x * 32, i0 = blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const long base = (long)blockIdx.z * n0 * n1;
    auto cell = [&](int i, int j) {
        return i >= 0 && j >= 0 && i < n0 && j < n1 ? in[base + (long)i * n1 + j] : 0.0f;
    };
    #pragma unroll
    for (int r = 0; r < 32; r += 8) tile[1 + ty + r][1 + tx] = cell(i0 + ty + r, j0 + tx);
    if (ty == 0) tile[0][1 + tx] = cell(i0 - 1, j0 + tx);
    if (ty == 1) tile[1 + tx][0] = cell(i0 + tx, j0 - 1);
    __syncthreads();
    #pragma unroll
    for (int r = ty; r < 32; r += 8) {
        if (i0 + r < n0 && j0 + tx < n1)
            ry[base + (long)(i0 + r) * n1 + j0 + tx] = 0.5f * (tile[r][1 + tx] + tile[1 + r][1 + tx]);
        if (i0 + tx < n0 && j0 + r < n1)
            rx[base + (long)(j0 + r) * n0 + i0 + tx] = 0.5f * (tile[1 + tx][r] + tile[1 + tx][1 + r]);
    }
}

__global__ void k_mix_gather(const float* __restrict__ src, float* __restrict__ dst, const float* __restrict__ M,
                             int n, int np, int nc, int nout)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int sd = blockIdx.y;  // (b*nout + o)*nc + c
    if (i >= n) return;
    const int c = sd % nc, bo = sd / nc, o = bo % nout, b = bo / nout;
    float v = 0.0f;
    const float* sp = src + (((long)b * n + i) * np) * nc + c;
    for (int p = 0; p < np; ++p) {
        const float m = M[o * np + p];
        if (m != 0.0f) v = fmaf(m, sp[(long)p * nc], v);
    }
    dst[(long)sd * n + i] = v;
}

__global__ void k_mix_scatter(const float* __restrict__ src, float* __restrict__ dst, const float* __restrict__ M,
                              int n, int np, int nc, int nout, int accumulate)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int dd = blockIdx.y;  // (b*nout + o)*nc + c
    if (i >= n) return;
    const int c = dd % nc, bo = dd / nc, o = bo % nout, b = bo / nout;
    float v = 0.0f;
    for (int p = 0; p < np; ++p) {
        const float m = M[o * np + p];
        if (m != 0.0f) v = fmaf(m, src[((long)(b * np + p) * nc + c) * n + i], v);
    }
    float* d = dst + (((long)b * n + i) * nout + o) * nc + c;
    *d = accumulate ? *d + v : v;
}

__global__ void k_fill(float* __restrict__ p, float v, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_axpy(float* __restrict__ y, const float* __restrict__ x, float a, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = fmaf(a, x[i], y[i]);
}

} // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

namespace {

// Line of the ray of detector angle a in view t, in image coordinates (FP64):
// X views (xv) X(Y) = A + B (Y - ny/2), Y views Y(X) = A + B (X - nx/2); L the
// path length per image line.
__device__ __forceinline__ void ray_line(bool xv, double nx, double ny, double dx, double dy, double dso, double a,
                                         double t, double& A, double& B, double& L)
{
    double sn, c;
    sincos(a - t, &sn, &c);
    const double sa = sin(a);
    if (xv) {
        A = 0.5 * nx + (dso / dx) * sa / c;
        B = (dy / dx) * sn / c;
        L = dy / fabs(c);
    } else {
        A = 0.5 * ny - (dso / dy) * sa / sn;
        B = (dx / dy) * c / sn;
        L = dx / fabs(sn);
    }
}

// FanK::sray and FanK::dray: the bin-centre ray (A, B, L) and the two edge rays
// of every (view, bin), FP64 rounded to float; bin k lies between the edges k
// and k + 1, edge e at angle (-(e - cu) - off_a) da + da / 2.  One lane per (view,
// bin): 0.03 ms for 1152 x 736 (0.1 s for the same loops on the host).
__global__ __launch_bounds__(256) void k_fan_rays(int nx, int ny, float dx, float dy, float dso, float da, float off_a,
                                                  int nu, const int* __restrict__ vcls, const float* __restrict__ deg,
                                                  float4* __restrict__ sray, float4* __restrict__ dray,
                                                  int* __restrict__ dwide)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (k == 0 && v == 0) *dwide = 1;
    if (k >= nu) return;
    const bool xv = vcls[v] == 0;
    const double t = (double)deg[v], cu = (nu - 1) / 2.0, off = (double)off_a, dd = (double)da;
    double A, B, L;
    auto line = [&](double a) { ray_line(xv, nx, ny, (double)dx, (double)dy, (double)dso, a, t, A, B, L); };
    line((-(k - cu) - off) * dd);
    sray[(size_t)v * nu + k] = make_float4((float)A, (float)B, (float)L, 0.0f);
    line((-(k - cu) - off) * dd + dd / 2.0);
    const float A0 = (float)A, B0 = (float)B;
    line((-((k + 1) - cu) - off) * dd + dd / 2.0);
    dray[(size_t)v * nu + k] = make_float4(A0, B0, (float)A, (float)B);
}

// Per view, vwide: 1 if every ray's line interval has a positive FP32 width on
// every image line, i.e. |B| exceeds the rounding of the end points
// A + B (j - n/2) (a few ulp of their largest magnitude) by a wide margin.
// dwide (1 before the launch): 0 if some DD footprint's width, affine in the
// line, changes sign or does not exceed the rounding of its end points by such a
// margin, or the product of two widths could leave the float range.
__global__ __launch_bounds__(256) void k_fan_ray_flags(int nx, int ny, int nu, const int* __restrict__ vcls,
                                                       const float4* __restrict__ sray,
                                                       const float4* __restrict__ dray, int* __restrict__ vwide,
                                                       int* __restrict__ dwide)
{
    const int v = blockIdx.x;
    const double h = 0.5 * (vcls[v] == 0 ? ny : nx);
    int ok = 1, okd = 1;
    for (int k = threadIdx.x; k < nu; k += blockDim.x) {
        const float4 r = sray[(size_t)v * nu + k];
        const double emax = fabs((double)r.x) + fabs((double)r.y) * (h + 1.0) + 1.0;
        if (!(fabs((double)r.y) > 1e-6 * emax)) ok = 0;
        const float4 d = dray[(size_t)v * nu + k];
        const double dA = (double)d.z - d.x, dB = (double)d.w - d.y;
        const double w0 = dA - dB * h, w1 = dA + dB * h;
        const double dmax = fmax(fabs((double)d.x), fabs((double)d.z)) +
                            fmax(fabs((double)d.y), fabs((double)d.w)) * h + 1.0;
        if (!(w0 * w1 > 0 && fmin(fabs(w0), fabs(w1)) > 1e-6 * dmax && dmax < 1e15)) okd = 0;
    }
    ok = __syncthreads_and(ok);
    okd = __syncthreads_and(okd);
    if (threadIdx.x != 0) return;
    vwide[v] = ok;
    if (!okd) *dwide = 0;
}

} // namespace

void FanTables::build(const FanGeo& g, const float* deg_host, hipStream_t st)
{
    RN_REQUIRE(g.nx > 0 && g.ny > 0 && g.nz > 0 && g.nu > 0 && g.nview > 0 && g.nv > 0, "fan dimensions must be positive");
    RN_REQUIRE(g.dx > 0 && g.dy > 0 && g.dz > 0 && g.da != 0 && g.dv > 0 && g.dso > 0, "fan spacings must be positive");
    RN_REQUIRE(deg_host != nullptr, "angle array is null");
    geo = g;
    deg.assign(deg_host, deg_host + g.nview);
    cls.resize(g.nview);
    const int nu = g.nu, nview = g.nview;
    // layout: vcos[nview] vsin[nview] vcls[nview] deg[nview] bsin[nu] bcos[nu]
    const size_t nf = 4 * (size_t)nview + 2 * (size_t)nu;
    host_.assign(nf, 0.0f);
    float* vcos = host_.data();
    float* vsin = vcos + nview;
    int* vcls = reinterpret_cast<int*>(vsin + nview);
    float* bsin = vsin + 3 * nview;
    float* bcos = bsin + nu;
    for (int v = 0; v < nview; v++) {
        const float d = deg_host[v];
        vcos[v] = (float)std::cos((double)d);
        vsin[v] = (float)std::sin((double)d);
        // the float32 host decision of DistanceDriven.cu:302 (glibc cosf/sinf)
        cls[v] = std::fabs(cosf(d)) > std::fabs(sinf(d)) ? 0 : 1;
        vcls[v] = cls[v];
    }
    std::copy(deg.begin(), deg.end(), vsin + 2 * nview);
    const double da = (double)g.da, cu = (nu - 1) / 2.0, off = (double)g.off_a;
    for (int k = 0; k < nu; k++) {
        const double a = (-(k - cu) - off) * da;
        bsin[k] = (float)std::sin(a);
        bcos[k] = (float)std::cos(a);
    }
    buf_.alloc(nf * sizeof(float));
    RN_HIP_CHECK(hipMemcpyAsync(buf_.get(), host_.data(), nf * sizeof(float), hipMemcpyHostToDevice, st));
    float* d = buf_.as<float>();
    k.nx = g.nx; k.ny = g.ny; k.nu = nu; k.nview = nview;
    k.dx = g.dx; k.dy = g.dy; k.da = g.da; k.off_a = g.off_a; k.dso = g.dso; k.dsd = g.dsd;
    k.cu = 0.5f * (nu - 1);
    k.vcos = d; k.vsin = d + nview; k.vcls = reinterpret_cast<const int*>(d + 2 * nview);
    k.bsin = d + 4 * nview; k.bcos = k.bsin + nu;
    // the ray tables and their flags, computed in FP64 on the device
    const size_t rays = (size_t)nview * nu;
    ray_.alloc(rays * sizeof(float4) + (nview + 1) * sizeof(int));
    dray_.alloc(rays * sizeof(float4));
    float4* sray = ray_.as<float4>();
    float4* dray = dray_.as<float4>();
    int* vwide = reinterpret_cast<int*>(sray + rays);
    hipLaunchKernelGGL(k_fan_rays, dim3(cdiv(nu, 256), nview), dim3(256), 0, st, g.nx, g.ny, g.dx, g.dy, g.dso, g.da,
                       g.off_a, nu, k.vcls, d + 3 * nview, sray, dray, vwide + nview);
    check_launch("fan_rays");
    hipLaunchKernelGGL(k_fan_ray_flags, dim3(nview), dim3(256), 0, st, g.nx, g.ny, nu, k.vcls, sray, dray, vwide,
                       vwide + nview);
    check_launch("fan_ray_flags");
    RN_HIP_CHECK(hipMemcpyAsync(&k.dwide, vwide + nview, sizeof(int), hipMemcpyDeviceToHost, st));
    RN_HIP_CHECK(hipStreamSynchronize(st));
    k.sray = sray;
    k.dray = dray;
    k.vwide = vwide;
    // pixel centres lie within R of the centre: |rx| / (dso - |ry|) <= R / (dso - R) < 1 if R < 0.45 dso
    const double R = 0.5 * std::sqrt((double)g.nx * g.dx * g.nx * g.dx + (double)g.ny * g.dy * g.ny * g.dy);
    k.unit_angle = R < 0.45 * (double)g.dso ? 1 : 0;
    // the tiles' points (an incomplete tile reaches over the image) lie within Rt of the
    // centre: half a tile over their distance from the source at most 1/4; and for DD
    // at most kTileMax, and the footprint of a pixel, cos(45 deg of view + the fan's angle) of it across
    // the ray, over 1e-3 bins
    const double hx = 4.0 * g.dx, hy = 4.0 * g.dy, ht = std::sqrt(hx * hx + hy * hy), Rt = R + 2.0 * ht;
    const double dso = (double)g.dso;
    k.tile = Rt < 0.9 * dso && ht <= 0.25 * (dso - Rt) ? 1 : 0;
    k.tile_dd = k.tile && ht <= fan::kTileMax * (dso - Rt) &&
                        std::cos(0.7854 + std::asin(Rt / dso)) * std::min(g.dx, g.dy) >=
                              1e-3 * std::fabs((double)g.da) * (dso + Rt) ? 1 : 0;
}

bool FanTables::matches(const FanGeo& g, const float* deg_host) const
{
    if (buf_.get() == nullptr) return false;
    if (std::memcmp(&g, &geo, sizeof(FanGeo)) != 0) return false;
    return std::memcmp(deg.data(), deg_host, sizeof(float) * g.nview) == 0;
}

// ---- launch shapes: candidates for the autotuner.  The shapes it may choose for a size give
// the same bits, the interleaved DD forward projection's (lines split over lanes) aside ----

namespace {

// MI355X: 8 XCDs, each with its own L2
constexpr int kXcds = 8;

template <int BLK, int XCD, int S>
void go_dd_fp(const FanK& g, const float* RX, const float* RY, float* prj, int ns, int view0, int nviews,
              hipStream_t st)
{
    const int ngroups = cdiv(ns, S);
    const long nblk = (long)cdiv(g.nu, BLK) * nviews * ngroups;
    if (XCD > 0 && nblk % XCD == 0 && nblk <= 0x7fffffffL) {
        hipLaunchKernelGGL((k_dd_fan_fp<BLK, XCD, S>), dim3((unsigned)nblk), dim3(BLK), 0, st, g, RX, RY, prj, view0,
                           nviews, ns);
    } else {
        hipLaunchKernelGGL((k_dd_fan_fp<BLK, 0, S>), dim3(cdiv(g.nu, BLK), nviews, ngroups), dim3(BLK), 0, st, g, RX,
                           RY, prj, view0, nviews, ns);
    }
}

template <int BLK, int XCD, int G, int H = 1>
void go_dd_fp_q(const FanK& g, const float4* QX, const float4* QY, float* prj, int ns, int view0, int nviews,
                hipStream_t st)
{
    const int ngroups = cdiv(cdiv(ns, 4), G);
    const long nblk = (long)cdiv(g.nu, BLK / H) * nviews * ngroups;
    if (XCD > 0 && nblk % XCD == 0 && nblk <= 0x7fffffffL) {
        hipLaunchKernelGGL((k_dd_fan_fp_q<BLK, XCD, G, H>), dim3((unsigned)nblk), dim3(BLK), 0, st, g, QX, QY, prj,
                           view0, nviews, ns);
    } else {
        hipLaunchKernelGGL((k_dd_fan_fp_q<BLK, 0, G, H>), dim3(cdiv(g.nu, BLK / H), nviews, ngroups), dim3(BLK), 0, st,
                           g, QX, QY, prj, view0, nviews, ns);
    }
}

template <int BLK, int XCD, int S>
void go_siddon_fp(const FanK& g, const float* Pyx, const float* Pxy, float* prj, int ns, int view0, int nviews,
                  const float* meas, const float* w, hipStream_t st)
{
    const int ngroups = cdiv(ns, S);
    const long nblk = (long)cdiv(g.nu, BLK) * nviews * ngroups;
    if (XCD > 0 && nblk % XCD == 0 && nblk <= 0x7fffffffL) {
        hipLaunchKernelGGL((k_siddon_fan_fp<float, BLK, XCD, S>), dim3((unsigned)nblk), dim3(BLK), 0, st, g, Pyx,
                           Pxy, prj, view0, nviews, ns, meas, w, g.nview);
    } else {
        hipLaunchKernelGGL((k_siddon_fan_fp<float, BLK, 0, S>), dim3(cdiv(g.nu, BLK), nviews, ngroups), dim3(BLK), 0,
                           st, g, Pyx, Pxy, prj, view0, nviews, ns, meas, w, g.nview);
    }
}

template <int BX, int BY, int NB, int S>
void go_siddon_bp(const FanK& g, const float* prj, float* img, int ns, int view0, int nviews, int acc,
                  hipStream_t st)
{
    hipLaunchKernelGGL((k_siddon_fan_bp<float, BX, BY, NB, S>), dim3(cdiv(g.ny, BX), cdiv(g.nx, BY), cdiv(ns, S)),
                       dim3(BX, BY), 0, st, g, prj, img, view0, nviews, ns, acc);
}

template <int G, int CAP>
void go_dd_adj(const FanK& g, const float4* wprj, float* img, int ns, hipStream_t st)
{
    const dim3 grd(cdiv(g.ny, 8), cdiv(g.nx, 8), cdiv(cdiv(ns, 4), G));
    const dim3 blk(64, kBpSegs);
    const size_t lds = ((size_t)kBpSegs * DdAdjStage<G, CAP>::kFloat4 + G * 64) * sizeof(float4);
    if (g.dwide) hipLaunchKernelGGL((k_dd_fan_adj<G, CAP, true>), grd, blk, lds, st, g, wprj, img, ns);
    else hipLaunchKernelGGL((k_dd_fan_adj<G, CAP, false>), grd, blk, lds, st, g, wprj, img, ns);
}

template <int BX, int BY, int S>
void go_dd_bp(const FanK& g, const float* wprj, float* img, int ns, int fbp, hipStream_t st)
{
    hipLaunchKernelGGL((k_dd_fan_bp<BX, BY, S>), dim3(cdiv(g.ny, BX), cdiv(g.nx, BY), cdiv(ns, S)), dim3(BX, BY), 0,
                       st, g, wprj, img, ns, fbp);
}

using DdFpFn = void (*)(const FanK&, const float*, const float*, float*, int, int, int, hipStream_t);
using SidFpFn = void (*)(const FanK&, const float*, const float*, float*, int, int, int, const float*, const float*,
                         hipStream_t);
using GatherFn = void (*)(const FanK&, const float*, float*, int, int, int, int, hipStream_t);
using DdBpFn = void (*)(const FanK&, const float*, float*, int, int, hipStream_t);

// 1-D blocks along the detector; 2-D pixel tiles (x lanes along y, the contiguous image axis)
const DdFpFn kDdFp[] = {go_dd_fp<128, kXcds, 1>, go_dd_fp<64, kXcds, 1>, go_dd_fp<256, kXcds, 1>,
                        go_dd_fp<128, 0, 1>,     go_dd_fp<64, 0, 1>,     go_dd_fp<128, kXcds, 2>,
                        go_dd_fp<64, kXcds, 2>,  go_dd_fp<128, 0, 2>};
constexpr int kNDdFp = sizeof(kDdFp) / sizeof(kDdFp[0]);
using DdFpQFn = void (*)(const FanK&, const float4*, const float4*, float*, int, int, int, hipStream_t);
const DdFpQFn kDdFpQ[] = {go_dd_fp_q<64, kXcds, 1, 2>,  go_dd_fp_q<128, kXcds, 1, 2>, go_dd_fp_q<256, kXcds, 1, 2>,
                          go_dd_fp_q<64, kXcds, 1, 4>,  go_dd_fp_q<128, kXcds, 1>,    go_dd_fp_q<64, kXcds, 1>,
                          go_dd_fp_q<256, kXcds, 1>,    go_dd_fp_q<128, 0, 1>,        go_dd_fp_q<64, 0, 1>,
                          go_dd_fp_q<128, kXcds, 2>,    go_dd_fp_q<64, kXcds, 2, 2>,  go_dd_fp_q<128, 0, 2>};
constexpr int kNDdFpQ = sizeof(kDdFpQ) / sizeof(kDdFpQ[0]);
// S: slices per lane (1 = one slice per lane; larger S shares the geometry work)
const SidFpFn kSidFp[] = {go_siddon_fp<128, 0, 1>,     go_siddon_fp<64, 0, 1>,     go_siddon_fp<256, 0, 1>,
                          go_siddon_fp<128, kXcds, 1>, go_siddon_fp<64, kXcds, 1>, go_siddon_fp<256, kXcds, 1>,
                          go_siddon_fp<128, 0, 2>,     go_siddon_fp<128, kXcds, 2>, go_siddon_fp<64, 0, 4>,
                          go_siddon_fp<128, 0, 4>,     go_siddon_fp<64, kXcds, 4>, go_siddon_fp<128, kXcds, 4>,
                          go_siddon_fp<256, kXcds, 4>, go_siddon_fp<128, kXcds, 8>};
const GatherFn kSidBp[] = {go_siddon_bp<16, 16, 3, 1>, go_siddon_bp<8, 8, 3, 1>,  go_siddon_bp<16, 16, 2, 1>,
                           go_siddon_bp<8, 8, 2, 1>,   go_siddon_bp<16, 16, 4, 1>, go_siddon_bp<8, 8, 4, 1>,
                           go_siddon_bp<8, 8, 2, 2>,   go_siddon_bp<8, 8, 2, 4>,   go_siddon_bp<16, 16, 2, 4>,
                           go_siddon_bp<8, 8, 3, 4>,   go_siddon_bp<8, 8, 2, 8>,   go_siddon_bp<16, 16, 2, 8>,
                           go_siddon_bp<8, 8, 3, 8>,   go_siddon_bp<8, 8, 2, 16>,  go_siddon_bp<16, 16, 2, 16>};
constexpr int kNSidFp = sizeof(kSidFp) / sizeof(kSidFp[0]);
constexpr int kNSidBp = sizeof(kSidBp) / sizeof(kSidBp[0]);
using DdAdjFn = void (*)(const FanK&, const float4*, float*, int, hipStream_t);
// groups of 4 slices per lane 1, 2, 4, 8; windows of 32 and 24 bins
const DdAdjFn kDdAdj[] = {go_dd_adj<1, 32>, go_dd_adj<1, 24>, go_dd_adj<2, 32>, go_dd_adj<2, 24>,
                          go_dd_adj<4, 32>, go_dd_adj<4, 24>, go_dd_adj<8, 32>, go_dd_adj<8, 24>};
const DdBpFn kDdBp[] = {go_dd_bp<16, 16, 1>, go_dd_bp<8, 32, 1>, go_dd_bp<32, 8, 1>, go_dd_bp<8, 8, 1>,
                       go_dd_bp<8, 8, 4>,   go_dd_bp<16, 16, 4>, go_dd_bp<8, 8, 8>, go_dd_bp<16, 16, 8>,
                       go_dd_bp<8, 8, 16>};
constexpr int kNDdBp = sizeof(kDdBp) / sizeof(kDdBp[0]);

template <int BX, int BY, int G>
void go_dd_bp_q(const FanK& g, const float4* wprj, float* img, int ns, int fbp, hipStream_t st)
{
    hipLaunchKernelGGL((k_dd_fan_bp_q<BX, BY, G>), dim3(cdiv(g.ny, BX), cdiv(g.nx, BY), cdiv(cdiv(ns, 4), G)),
                       dim3(BX, BY), 0, st, g, wprj, img, ns, fbp);
}
using DdBpQFn = void (*)(const FanK&, const float4*, float*, int, int, hipStream_t);
const DdBpQFn kDdBpQ[] = {go_dd_bp_q<8, 8, 4>,   go_dd_bp_q<16, 16, 2>, go_dd_bp_q<8, 8, 2>,
                          go_dd_bp_q<16, 16, 1>, go_dd_bp_q<8, 8, 1>};
constexpr int kNDdBpQ = sizeof(kDdBpQ) / sizeof(kDdBpQ[0]);

// nw: waves per tile, each with an even share of the views
template <int G, int CAP>
void go_dd_bp_tile(const FanK& g, const float4* wprj, float* img, int ns, int fbp, int nw, hipStream_t st)
{
    const dim3 grd(cdiv(g.ny, 8), cdiv(g.nx, 8), cdiv(cdiv(ns, 4), G));
    const size_t lds = ((size_t)nw * G * stage_pitch(CAP) + (nw > 1 ? G * 64 : 0)) * sizeof(float4);
    hipLaunchKernelGGL((k_dd_fan_bp_tile<G, CAP>), grd, dim3(64, nw), lds, st, g, wprj, img, ns, fbp);
}
using DdBpTileFn = void (*)(const FanK&, const float4*, float*, int, int, int, hipStream_t);
// groups of 4 slices per lane 1, 2, 4, 8; windows of 32 and 24 bins
const DdBpTileFn kDdBpTile[] = {go_dd_bp_tile<1, 32>, go_dd_bp_tile<1, 24>, go_dd_bp_tile<2, 32>, go_dd_bp_tile<2, 24>,
                             go_dd_bp_tile<4, 32>, go_dd_bp_tile<4, 24>, go_dd_bp_tile<8, 32>, go_dd_bp_tile<8, 24>};

// Candidates of a kernel with G = 1, 2, 4, 8 groups per lane, two each, in the order
// of preference for this batch: the fewest groups per lane that hold it first, then
// fewer; more groups than that last.  Groups are addressed with 32-bit byte offsets:
// G of them have to fit.
struct GroupOrder {
    int idx[8] = {}, n = 0;
    long tiles;   // tiles times batches of groups of the preferred shape
    GroupOrder(const FanK& g, int nslices)
    {
        const int nquads = cdiv(nslices, 4);
        auto add = [&](int lg) {
            if (lg > 0 && ((long)g.nview * g.nu * 16L << lg) >= 0x7fffffffL) return;
            idx[n++] = 2 * lg;
            idx[n++] = 2 * lg + 1;
        };
        const int best = nquads > 4 ? 3 : nquads > 2 ? 2 : nquads - 1;
        tiles = (long)cdiv(g.nx, 8) * cdiv(g.ny, 8) * cdiv(nquads, 1 << best);
        for (int lg = best; lg >= 0; lg--) add(lg);
        for (int lg = best + 1; lg < 4; lg++) add(lg);
    }
};

// The Siddon and DD gather kernels address one slice's image plane, ray table
// and sinogram rows with 32-bit byte offsets.
void require_offsets32(const FanK& g, int nviews, size_t elem)
{
    const long lim = 0x7fffffffL;
    RN_REQUIRE((long)g.nx * g.ny * (long)elem < lim && (long)g.nview * g.nu * 16L < lim &&
                   (long)nviews * g.nu * (long)elem < lim,
               "image plane, ray table or sinogram of one slice exceeds 2 GiB");
}

template <int BLK, int XCD, int G, int H, bool PLAIN>
void run_siddon_fp_q(const FanK& g, const float4* Qyx, const float4* Qxy, float4* res, float* prj, int ns, int view0,
                     int nviews, const float4* meas, const float4* w, int res_vstride, int res_voff, hipStream_t st)
{
    const int ngroups = cdiv(cdiv(ns, 4), G);
    const long nblk = (long)cdiv(g.nu, BLK / H) * nviews * ngroups;
    if (XCD > 0 && nblk + XCD <= 0x7fffffffL) {
        const long n = cdiv(nblk, XCD > 0 ? XCD : 1) * (long)XCD;
        hipLaunchKernelGGL((k_siddon_fan_fp_q<BLK, XCD, G, H, PLAIN>), dim3((unsigned)n), dim3(BLK), 0, st, g, Qyx, Qxy,
                           res, prj, view0, nviews, ns, meas, w, g.nview, res_vstride, res_voff);
    } else {
        hipLaunchKernelGGL((k_siddon_fan_fp_q<BLK, 0, G, H, PLAIN>), dim3(cdiv(g.nu, BLK / H), nviews, ngroups),
                           dim3(BLK), 0, st, g, Qyx, Qxy, res, prj, view0, nviews, ns, meas, w, g.nview, res_vstride,
                           res_voff);
    }
}

// weighted residuals of nquads groups
template <int BLK, int XCD, int G, int H = 1>
void go_siddon_fp_q(const FanK& g, const float4* Qyx, const float4* Qxy, float4* res, int nquads, int view0,
                    int nviews, const float4* meas, const float4* w, int res_vstride, int res_voff, hipStream_t st)
{
    run_siddon_fp_q<BLK, XCD, G, H, false>(g, Qyx, Qxy, res, nullptr, 4 * nquads, view0, nviews, meas, w, res_vstride,
                                           res_voff, st);
}

// plain sinograms of ns slices
template <int BLK, int XCD, int G, int H = 1>
void go_siddon_fp_qp(const FanK& g, const float4* Qyx, const float4* Qxy, float* prj, int ns, int view0, int nviews,
                     hipStream_t st)
{
    run_siddon_fp_q<BLK, XCD, G, H, true>(g, Qyx, Qxy, nullptr, prj, ns, view0, nviews, nullptr, nullptr, 0, 0, st);
}

// nseg: view segments of every pixel's sum
template <int BX, int BY, int NB, int G>
void go_siddon_bp_q(const FanK& g, const float4* prj, float* img, int ns, int view0, int nviews, int nseg,
                    hipStream_t st)
{
    const auto k = nseg > 1 ? k_siddon_fan_bp_q<BX, BY, NB, G, true> : k_siddon_fan_bp_q<BX, BY, NB, G, false>;
    hipLaunchKernelGGL(k, dim3(cdiv(g.ny, BX), cdiv(g.nx, BY), cdiv(cdiv(ns, 4), G)), dim3(BX, BY), 0, st, g, prj, img,
                       view0, nviews, ns, nseg);
}

using SidFpQFn = void (*)(const FanK&, const float4*, const float4*, float4*, int, int, int, const float4*,
                          const float4*, int, int, hipStream_t);
using SidBpQFn = void (*)(const FanK&, const float4*, float*, int, int, int, int, hipStream_t);
// G: groups of 4 slices per lane; H: parts of the line range per ray (the
// split shortens the waves of a launch that would leave a partial second
// round on the chip); candidates in order of preference (the tuner keeps the
// first within 3 % of the fastest)
const SidFpQFn kSidFpQ[] = {go_siddon_fp_q<64, kXcds, 1, 2>,  go_siddon_fp_q<128, kXcds, 1, 2>,
                            go_siddon_fp_q<256, kXcds, 1, 2>, go_siddon_fp_q<64, kXcds, 1, 4>,
                            go_siddon_fp_q<128, kXcds, 1>,    go_siddon_fp_q<64, kXcds, 1>,
                            go_siddon_fp_q<256, kXcds, 1>,    go_siddon_fp_q<128, 0, 1>,
                            go_siddon_fp_q<64, 0, 1>,         go_siddon_fp_q<128, kXcds, 2>,
                            go_siddon_fp_q<128, 0, 2>};
using SidFpQPFn = void (*)(const FanK&, const float4*, const float4*, float*, int, int, int, hipStream_t);
const SidFpQPFn kSidFpQP[] = {go_siddon_fp_qp<64, kXcds, 1, 2>,  go_siddon_fp_qp<128, kXcds, 1, 2>,
                              go_siddon_fp_qp<256, kXcds, 1, 2>, go_siddon_fp_qp<64, kXcds, 1, 4>,
                              go_siddon_fp_qp<128, kXcds, 1, 4>, go_siddon_fp_qp<128, kXcds, 1>,
                              go_siddon_fp_qp<64, kXcds, 1>,     go_siddon_fp_qp<256, kXcds, 1>,
                              go_siddon_fp_qp<128, 0, 1>,        go_siddon_fp_qp<64, 0, 1>,
                              go_siddon_fp_qp<128, kXcds, 2>,    go_siddon_fp_qp<64, kXcds, 2, 2>,
                              go_siddon_fp_qp<128, kXcds, 2, 2>, go_siddon_fp_qp<128, 0, 2>};
constexpr int kNSidFpQP = sizeof(kSidFpQP) / sizeof(kSidFpQP[0]);
// the shapes with a ray's lines split over 2 and over 4 lanes (bit i: candidate i)
constexpr uint32_t kSidFpQ2 = 0x7, kSidFpQ4 = 0x8, kSidFpQP2 = 0x1807, kSidFpQP4 = 0x18;
// The split is the sizes', not the tuner's: it decides the last bits.  4 lanes per ray,
// or 2 where the lines are long and the rays fill the chip without.  ms with 2 and with
// 4: one slice of 64^2, 15 views 0.012, 0.005; 256^2 x 16, 360 views 0.147, 0.143; 383^2
// x 6, 520 views 0.144, 0.139; 512^2, 96 views, one slice 0.060, 0.035, 5 slices 0.070,
// 0.071, 32 slices 0.228, 0.262; 462 x 512 x 5, 232 views of 328 0.093, 0.101.
bool split4(const FanK& g, int nslices, int nviews)
{
    return std::max(g.nx, g.ny) < 480 || (long)cdiv(nslices, 4) * nviews * g.nu < 100000;
}
// per-pixel gathers, for every geometry
const SidBpQFn kSidBpQ[] = {go_siddon_bp_q<16, 16, 2, 8>, go_siddon_bp_q<8, 8, 2, 8>, go_siddon_bp_q<16, 16, 2, 4>,
                            go_siddon_bp_q<8, 8, 2, 4>,   go_siddon_bp_q<8, 8, 2, 2>, go_siddon_bp_q<16, 16, 2, 2>,
                            go_siddon_bp_q<8, 8, 2, 1>,   go_siddon_bp_q<16, 16, 2, 1>, go_siddon_bp_q<8, 8, 3, 4>,
                            go_siddon_bp_q<8, 8, 3, 2>};
constexpr int kNSidFpQ = sizeof(kSidFpQ) / sizeof(kSidFpQ[0]);
constexpr int kNSidBpQ = sizeof(kSidBpQ) / sizeof(kSidBpQ[0]);

using SidBpTileFn = void (*)(const FanK&, const float4*, float*, int, int, int, const SqsUpd*, int, hipStream_t);
// u != nullptr: the OS-SQS update in the epilogue instead of img
// nw: waves per tile, each with an even share of the views.  CAP = 0: the gathers of one
// group from memory.
template <int G, int CAP, int NB = 2>
void go_siddon_bp_tile(const FanK& g, const float4* prj, float* img, int ns, int view0, int nviews, const SqsUpd* u,
                       int nw, hipStream_t st)
{
    const dim3 grd(cdiv(g.ny, 8), cdiv(g.nx, 8), cdiv(cdiv(ns, 4), G));
    const size_t lds = ((CAP == 0 ? 0 : (size_t)nw * (G + 1) * stage_pitch(CAP)) + (nw > 1 ? G * 64 : 0)) * sizeof(float4);
    const SqsUpd upd = u != nullptr ? *u : SqsUpd{};
    void (*k)(FanK, const float4*, float*, int, int, int, SqsUpd);
    if constexpr (CAP == 0) k = u != nullptr ? k_siddon_fan_bp_tile1<NB, true> : k_siddon_fan_bp_tile1<NB, false>;
    else k = u != nullptr ? k_siddon_fan_bp_tile<G, CAP, true> : k_siddon_fan_bp_tile<G, CAP, false>;
    hipLaunchKernelGGL(k, grd, dim3(64, nw), lds, st, g, prj, img, view0, nviews, ns, upd);
}
constexpr int kNSidBpTile = 7;
const SidBpTileFn kSidBpTile[kNSidBpTile] = {
    go_siddon_bp_tile<1, 0>,  go_siddon_bp_tile<2, 32>, go_siddon_bp_tile<2, 24>, go_siddon_bp_tile<4, 24>,
    go_siddon_bp_tile<4, 32>, go_siddon_bp_tile<8, 24>, go_siddon_bp_tile<8, 32>};
// fewer than 4 slices of a projector call: the gathers of one group, and for pins the
// staged shapes, from which one group has nothing to gain (250^2, 360 views: 0.055 ms;
// staged 0.071, with 2 to 8 groups per lane 0.079 to 0.13)
const SidBpTileFn kSidBpFew[] = {
    go_siddon_bp_tile<1, 0>,     go_siddon_bp_tile<1, 0, 3>, go_siddon_bp_tile<1, 0, 1>, go_siddon_bp_tile<1, 0, 4>,
    go_siddon_bp_tile<1, 32>,    go_siddon_bp_tile<1, 24>,   go_siddon_bp_tile<1, 48>,   go_siddon_bp_tile<2, 32>,
    go_siddon_bp_tile<2, 24>,    go_siddon_bp_tile<4, 32>,   go_siddon_bp_tile<4, 24>,   go_siddon_bp_tile<8, 32>,
    go_siddon_bp_tile<8, 24>};
constexpr int kNSidBpFew = sizeof(kSidBpFew) / sizeof(kSidBpFew[0]);
constexpr uint32_t kSidBpFewPick = 0xf;

// Candidate i of the interleaved BP for this launch: the tile shapes (FanK::tile), the
// fewest groups per lane that hold the batch first, then fewer, then more, where G
// groups' rows fit 32-bit offsets; then the gathers, at kNSidBpTile + their index.
struct SidBpOrder {
    int idx[kNSidBpTile + kNSidBpQ] = {}, n = 0;
    int layout;   // TuneKey::layout: the list depends on FanK::tile, which the sizes do not tell
    int nw = 1;   // view segments of every candidate's sums (a wave each by tiles)
    SidBpOrder(const FanK& g, int nslices, int nviews)
    {
        layout = g.tile ? 1 : 2;
        const int nquads = cdiv(nslices, 4);
        const int best = nquads > 4 ? 3 : nquads > 2 ? 2 : nquads - 1;
        // Waves per tile of the preferred shape: up to 8 while they do not fill the chip
        // (4096 of 4 and more groups, 4 a SIMD by their registers; more of the shorter
        // ones of 1 and 2 groups) or leave over 30 % of the last round idle, and each
        // keeps 8 views, over which its batch of tile projections pays.  Every shape takes
        // that many: the split decides the last bits.  us with 1, 2, 4, 8: one slice of
        // 256^2, 30 views 23, 15, 12, 12, 360 views 279, 184, 133, 87; 5 slices of 512^2 (2
        // groups), 1152 views 1117, 1088, 941, 966; 32 slices of 250^2 (8 groups), 360
        // views 438, 251, 200, 255; of 383^2 (2304 tiles), 520 views 561, 513, 428, 399; of
        // 512^2, 96 views 153, 177, 170, 202.  One where 4 and more groups meet bins wider
        // than 1.6 pixels on half a chip of tiles: the gathers with one sum are the faster
        // shape then (16 slices of 464 x 512, bins of 2.1 pixels: 248, tiles by 4 waves 324).
        const long tiles = (long)cdiv(g.nx, 8) * cdiv(g.ny, 8) * cdiv(nquads, 1 << best);
        const long full = best <= 1 ? 16384 : 4096;
        auto more = [&](long w) { return w < full || (w < 4 * full && 10 * w < 7 * full * ((w + full - 1) / full)); };
        const bool wide = best >= 2 && tiles >= 2048 && fabsf(g.da) * g.dso > 1.6f * std::max(g.dx, g.dy);
        while (g.tile && !wide && nw < 8 && more(tiles * nw) && nviews >= 8 * nw) nw *= 2;
        auto add = [&](int lg) {
            if (!g.tile || (long)(1 << lg) * nviews * g.nu * 16L >= 0x7fffffffL) return;
            for (int i = lg == 0 ? 0 : 2 * lg - 1; i <= 2 * lg; i++) idx[n++] = i;
        };
        for (int lg = best; lg >= 0; lg--) add(lg);
        for (int lg = best + 1; lg < 4; lg++) add(lg);
        for (int i = 0; i < kNSidBpQ; i++) idx[n++] = kNSidBpTile + i;
    }
};

void go_siddon_bp_any(int c, const FanK& g, const float4* prj, float* img, int ns, int view0, int nviews, int nw,
                      hipStream_t st)
{
    if (c < kNSidBpTile) kSidBpTile[c](g, prj, img, ns, view0, nviews, nullptr, nw, st);
    else kSidBpQ[c - kNSidBpTile](g, prj, img, ns, view0, nviews, nw, st);
}

} // namespace

void launch_dd_fan_fp(const FanK& g, const float* RX, const float* RY, float* prj_vu,
                      int nslices, int view0, int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    const int c = tune_choose({TK_DD_FP, g.nx, g.ny, g.nu, nviews, nslices}, kNDdFp,
                              [&](int i) { kDdFp[i](g, RX, RY, prj_vu, nslices, view0, nviews, st); }, st, true);
    kDdFp[c](g, RX, RY, prj_vu, nslices, view0, nviews, st);
    check_launch("dd_fan_fp");
}

void launch_dd_fan_fp_q(const FanK& g, const float4* QX, const float4* QY, float* prj_vu, int nslices, int view0,
                        int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    RN_REQUIRE(qplanes_fit32(g.nx, g.ny), "padded image plane of one slice group exceeds 2 GiB");
    const int c = tune_choose({TK_DD_FP_Q, g.nx, g.ny, g.nu, nviews, nslices}, kNDdFpQ,
                              [&](int i) { kDdFpQ[i](g, QX, QY, prj_vu, nslices, view0, nviews, st); }, st, true);
    kDdFpQ[c](g, QX, QY, prj_vu, nslices, view0, nviews, st);
    check_launch("dd_fan_fp_q");
}

void launch_siddon_fan_fp(const FanK& g, const float* Pyx, const float* Pxy, float* prj_vu,
                          int nslices, int view0, int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    const int c = tune_choose({TK_SIDDON_FP, g.nx, g.ny, g.nu, nviews, nslices}, kNSidFp, [&](int i) {
        kSidFp[i](g, Pyx, Pxy, prj_vu, nslices, view0, nviews, nullptr, nullptr, st);
    }, st, true);
    kSidFp[c](g, Pyx, Pxy, prj_vu, nslices, view0, nviews, nullptr, nullptr, st);
    check_launch("siddon_fan_fp");
}

void launch_siddon_fan_fp_residual(const FanK& g, const float* Pyx, const float* Pxy, float* res_vu,
                                   int nslices, int view0, int nviews, const float* meas_vu, const float* w_vu,
                                   hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    const int c = tune_choose({TK_SIDDON_FP, g.nx, g.ny, g.nu, nviews, nslices}, kNSidFp, [&](int i) {
        kSidFp[i](g, Pyx, Pxy, res_vu, nslices, view0, nviews, meas_vu, w_vu, st);
    }, st, true);
    kSidFp[c](g, Pyx, Pxy, res_vu, nslices, view0, nviews, meas_vu, w_vu, st);
    check_launch("siddon_fan_fp_residual");
}

void launch_siddon_fan_fp_residual_q(const FanK& g, const float4* Qyx, const float4* Qxy, float4* res_q,
                                     int nslices, int view0, int nviews, const float4* meas_q, const float4* w_q,
                                     int res_vstride, int res_voff, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    RN_REQUIRE(res_voff >= 0 && res_voff + nviews <= res_vstride, "residual view range out of its rows");
    require_offsets32(g, res_vstride, sizeof(float4));
    RN_REQUIRE(qplanes_fit32(g.nx, g.ny), "padded image plane of one slice group exceeds 2 GiB");
    const int nq = cdiv(nslices, 4);
    const int c = tune_choose({TK_SIDDON_FP_Q, g.nx, g.ny, g.nu, nviews, nslices}, kNSidFpQ, [&](int i) {
        kSidFpQ[i](g, Qyx, Qxy, res_q, nq, view0, nviews, meas_q, w_q, res_vstride, res_voff, st);
    }, st, true, split4(g, nslices, nviews) ? kSidFpQ4 : kSidFpQ2);
    kSidFpQ[c](g, Qyx, Qxy, res_q, nq, view0, nviews, meas_q, w_q, res_vstride, res_voff, st);
    check_launch("siddon_fan_fp_residual_q");
}

void launch_siddon_fan_fp_q(const FanK& g, const float4* Qyx, const float4* Qxy, float* prj_vu, int nslices,
                            int view0, int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    RN_REQUIRE(qplanes_fit32(g.nx, g.ny), "padded image plane of one slice group exceeds 2 GiB");
    const int c = tune_choose({TK_SIDDON_FP, g.nx, g.ny, g.nu, nviews, nslices, 1}, kNSidFpQP,
                              [&](int i) { kSidFpQP[i](g, Qyx, Qxy, prj_vu, nslices, view0, nviews, st); }, st, true,
                              split4(g, nslices, nviews) ? kSidFpQP4 : kSidFpQP2);
    kSidFpQP[c](g, Qyx, Qxy, prj_vu, nslices, view0, nviews, st);
    check_launch("siddon_fan_fp_q");
}

void launch_siddon_fan_bp_q(const FanK& g, const float4* prj_q, float* img_xy, int nslices, int view0,
                            int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float4));
    const SidBpOrder order(g, nslices, nviews);
    const TuneKey key{TK_SIDDON_BP, g.nx, g.ny, g.nu, nviews, nslices, order.layout};
    const int c = order.idx[tune_choose(key, order.n, [&](int i) {
        go_siddon_bp_any(order.idx[i], g, prj_q, img_xy, nslices, view0, nviews, order.nw, st);
    }, st, true)];
    go_siddon_bp_any(c, g, prj_q, img_xy, nslices, view0, nviews, order.nw, st);
    check_launch("siddon_fan_bp_q");
}

void launch_siddon_fan_bp_few(const FanK& g, const float4* prj_q, float* img_xy, int nslices, int view0, int nviews,
                              hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    const int c = tune_choose({TK_SIDDON_BP, g.nx, g.ny, g.nu, nviews, nslices, 1}, kNSidBpFew, [&](int i) {
        kSidBpFew[i](g, prj_q, img_xy, nslices, view0, nviews, nullptr, kBpSegs, st);
    }, st, true, kSidBpFewPick);
    kSidBpFew[c](g, prj_q, img_xy, nslices, view0, nviews, nullptr, kBpSegs, st);
    check_launch("siddon_fan_bp_few");
}

bool launch_siddon_fan_bp_q_update(const FanK& g, const float4* prj_q, float* img_xy, int nslices, int view0,
                                   int nviews, const SqsUpd& u, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return false;
    require_offsets32(g, nviews, sizeof(float4));
    const SidBpOrder order(g, nslices, nviews);
    // the launch shape is tuned on the plain backprojection (img_xy as its output)
    const TuneKey key{TK_SIDDON_BP_Q, g.nx, g.ny, g.nu, nviews, nslices, order.layout};
    const int c = order.idx[tune_choose(key, order.n, [&](int i) {
        go_siddon_bp_any(order.idx[i], g, prj_q, img_xy, nslices, view0, nviews, order.nw, st);
    }, st, true)];
    const bool fused = c < kNSidBpTile;
    if (fused) kSidBpTile[c](g, prj_q, nullptr, nslices, view0, nviews, &u, order.nw, st);
    else go_siddon_bp_any(c, g, prj_q, img_xy, nslices, view0, nviews, order.nw, st);
    check_launch("siddon_fan_bp_q_update");
    return fused;
}

void launch_siddon_fan_fp_f64(const FanK& g, const double* Pyx, const double* Pxy, double* prj_vu,
                              int nslices, int view0, int nviews, hipStream_t st)
{
    if (nslices <= 0 || nviews <= 0) return;
    require_offsets32(g, nviews, sizeof(double));
    dim3 blk(128), grd(cdiv(g.nu, 128), nviews, nslices);
    hipLaunchKernelGGL((k_siddon_fan_fp<double, 128, 0, 1>), grd, blk, 0, st, g, Pyx, Pxy, prj_vu, view0, nviews,
                       nslices, (const float*)nullptr, (const float*)nullptr, 0);
    check_launch("siddon_fan_fp_f64");
}

void launch_siddon_fan_bp_f64(const FanK& g, const double* prj_vu, double* img_xy, int nslices,
                              int view0, int nviews, hipStream_t st)
{
    if (nslices <= 0) return;
    require_offsets32(g, nviews, sizeof(double));
    dim3 blk(16, 16), grd(cdiv(g.ny, 16), cdiv(g.nx, 16), nslices);
    hipLaunchKernelGGL((k_siddon_fan_bp<double, 16, 16, 4, 1>), grd, blk, 0, st, g, prj_vu, img_xy, view0, nviews,
                       nslices, 0);
    check_launch("siddon_fan_bp_f64");
}

void launch_siddon_fan_bp(const FanK& g, const float* prj_vu, float* img_xy, int nslices,
                          int view0, int nviews, bool accumulate, hipStream_t st)
{
    if (nslices <= 0) return;
    require_offsets32(g, nviews, sizeof(float));
    const int c = tune_choose({TK_SIDDON_BP, g.nx, g.ny, g.nu, nviews, nslices}, kNSidBp, [&](int i) {
        kSidBp[i](g, prj_vu, img_xy, nslices, view0, nviews, 0, st);
    }, st, !accumulate);
    kSidBp[c](g, prj_vu, img_xy, nslices, view0, nviews, accumulate ? 1 : 0, st);
    check_launch("siddon_fan_bp");
}

void launch_dd_fan_adj(const FanK& g, const float4* wprj_q, float* img_xy, int nslices, hipStream_t st)
{
    if (nslices <= 0) return;
    RN_REQUIRE((long)g.nx * g.ny * 4L < 0x7fffffffL && (long)g.nview * g.nu * 16L < 0x7fffffffL,
               "image plane, ray table or sinogram of one slice exceeds 2 GiB");
    const GroupOrder order(g, nslices);
    const int c = tune_choose({TK_DD_ADJ, g.nx, g.ny, g.nu, g.nview, nslices}, order.n,
                              [&](int i) { kDdAdj[order.idx[i]](g, wprj_q, img_xy, nslices, st); }, st, true);
    kDdAdj[order.idx[c]](g, wprj_q, img_xy, nslices, st);
    check_launch("dd_fan_adj");
}

void launch_dd_preweight(const FanK& g, const float* prj_vu, float* wprj_vu, int nslices, hipStream_t st)
{
    if (nslices <= 0) return;
    dim3 blk(256), grd(cdiv(g.nu, 256), g.nview, nslices);
    hipLaunchKernelGGL(k_dd_preweight, grd, blk, 0, st, g, prj_vu, wprj_vu);
    check_launch("dd_preweight");
}

void launch_dd_fan_bp(const FanK& g, const float* wprj_vu, float* img_xy, int nslices, bool fbp, hipStream_t st)
{
    if (nslices <= 0) return;
    require_offsets32(g, g.nview, sizeof(float));
    const int c = tune_choose({fbp ? TK_DD_FBP : TK_DD_BP, g.nx, g.ny, g.nu, g.nview, nslices}, kNDdBp,
                              [&](int i) { kDdBp[i](g, wprj_vu, img_xy, nslices, fbp ? 1 : 0, st); }, st, true);
    kDdBp[c](g, wprj_vu, img_xy, nslices, fbp ? 1 : 0, st);
    check_launch("dd_fan_bp");
}

void launch_dd_fan_bp_tile(const FanK& g, const float4* wprj_q, float* img_xy, int nslices, bool fbp, hipStream_t st)
{
    if (nslices <= 0) return;
    require_offsets32(g, g.nview, nslices < 4 ? sizeof(float) : sizeof(float4));
    const GroupOrder order(g, nslices);
    // Eight waves per tile while one of the preferred shape would leave the 1024 SIMDs
    // fewer than 8 waves each (one slice of 512^2, 4096 waves: 0.73 ms by two, 0.65 by
    // eight).  Every shape takes that many: the split decides the last bits.
    const int nw = order.tiles < 8192 ? 8 : 1;
    // the kernel id of the layout the slices' count had without tiles
    const int id = nslices < 4 ? (fbp ? TK_DD_FBP : TK_DD_BP) : (fbp ? TK_DD_FBP_Q : TK_DD_BP_Q);
    const int c = tune_choose({id, g.nx, g.ny, g.nu, g.nview, nslices, 1}, order.n,
                              [&](int i) { kDdBpTile[order.idx[i]](g, wprj_q, img_xy, nslices, fbp ? 1 : 0, nw, st); }, st,
                              true);
    kDdBpTile[order.idx[c]](g, wprj_q, img_xy, nslices, fbp ? 1 : 0, nw, st);
    check_launch("dd_fan_bp_tile");
}

void launch_dd_fan_bp_q(const FanK& g, const float4* wprj_q, float* img_xy, int nslices, bool fbp, hipStream_t st)
{
    if (nslices <= 0) return;
    require_offsets32(g, g.nview, sizeof(float4));
    const int c = tune_choose({fbp ? TK_DD_FBP_Q : TK_DD_BP_Q, g.nx, g.ny, g.nu, g.nview, nslices}, kNDdBpQ,
                              [&](int i) { kDdBpQ[i](g, wprj_q, img_xy, nslices, fbp ? 1 : 0, st); }, st, true);
    kDdBpQ[c](g, wprj_q, img_xy, nslices, fbp ? 1 : 0, st);
    check_launch("dd_fan_bp_q");
}

template <int BX, int BY, int S>
void go_pixel_bp(const FanK& g, const float* prj_vu, float* img_xy, int nslices, hipStream_t st)
{
    hipLaunchKernelGGL((k_pixel_fan_bp<BX, BY, S>), dim3(cdiv(g.ny, BX), cdiv(g.nx, BY), cdiv(nslices, S)),
                       dim3(BX, BY), 0, st, g, prj_vu, img_xy, nslices);
}

using PixBpFn = void (*)(const FanK&, const float*, float*, int, hipStream_t);
const PixBpFn kPixBp[] = {go_pixel_bp<16, 16, 1>, go_pixel_bp<8, 8, 1>,   go_pixel_bp<16, 16, 2>,
                          go_pixel_bp<16, 16, 4>, go_pixel_bp<8, 8, 4>,   go_pixel_bp<16, 16, 8>,
                          go_pixel_bp<8, 32, 8>,  go_pixel_bp<16, 16, 16>};
constexpr int kNPixBp = sizeof(kPixBp) / sizeof(kPixBp[0]);

void launch_pixel_fan_bp(const FanK& g, const float* prj_vu, float* img_xy, int nslices, hipStream_t st)
{
    if (nslices <= 0) return;
    RN_REQUIRE(cdiv(g.nx, 8) <= 65535 && cdiv(nslices, 1) <= 65535, "pixel_fan_bp: grid too large");
    const int c = tune_choose({TK_PIXEL_BP, g.nx, g.ny, g.nu, g.nview, nslices}, kNPixBp,
                              [&](int i) { kPixBp[i](g, prj_vu, img_xy, nslices, st); }, st, true);
    kPixBp[c](g, prj_vu, img_xy, nslices, st);
    check_launch("pixel_fan_bp");
}

void launch_pack_quads(const float* in, float4* q_same, float4* q_tr, int n1, int n2, int nslices, bool padded,
                       hipStream_t st)
{
    if (nslices <= 0 || n1 <= 0 || n2 <= 0) return;
    dim3 grd(cdiv(n2, 32), cdiv(n1, 32), cdiv(nslices, 4));
    hipLaunchKernelGGL(k_pack_quads, grd, dim3(256), 0, st, in, q_same, q_tr, n1, n2, nslices,
                       padded ? qpitch(n2) : n2, padded ? qpitch(n1) : n1, padded ? kQPadL : 0,
                       (const float4*)nullptr);
    check_launch("pack_quads");
}

void launch_pack_quads_len(const FanK& g, const float* in, float4* q, int nslices, hipStream_t st)
{
    if (nslices <= 0) return;
    dim3 grd(cdiv(g.nview, 32), cdiv(g.nu, 32), cdiv(nslices, 4));
    hipLaunchKernelGGL(k_pack_quads, grd, dim3(256), 0, st, in, (float4*)nullptr, q, g.nu, g.nview, nslices, g.nview,
                       g.nu, 0, g.sray);
    check_launch("pack_quads_len");
}

void launch_pack_planes(const float* in, float4* q_same, float4* q_tr, int n1, int n2, int nslices, bool avg,
                        hipStream_t st)
{
    if (nslices <= 0 || n1 <= 0 || n2 <= 0) return;
    dim3 grd(cdiv(n2, 32), cdiv(n1, 32), cdiv(nslices, 4));
    hipLaunchKernelGGL(avg ? k_pack_planes<true> : k_pack_planes<false>, grd, dim3(256), 0, st, in, q_same, q_tr, n1,
                       n2, nslices);
    check_launch("pack_planes");
}

void launch_permute_rows(const float* in, float* out, const int* perm, int rows, int cols, int batch,
                         hipStream_t st)
{
    if (rows <= 0 || cols <= 0 || batch <= 0) return;
    hipLaunchKernelGGL(k_permute_rows, dim3(cdiv(cols, 256), rows, batch), dim3(256), 0, st, in, out, perm, rows,
                       cols);
    check_launch("permute_rows");
}

void launch_transpose(const float* in, float* out, int rows, int cols, int batch, hipStream_t st)
{
    if (batch <= 0 || rows <= 0 || cols <= 0) return;
    dim3 blk(32, 8), grd(cdiv(cols, 32), cdiv(rows, 32), batch);
    hipLaunchKernelGGL(k_transpose, grd, blk, 0, st, in, out, rows, cols);
    check_launch("transpose");
}

void launch_avg_planes(const float* in, float* ry, float* rx, int n0, int n1, int batch, hipStream_t st)
{
    if (batch <= 0) return;
    const dim3 grd(cdiv(n1, 32), cdiv(n0, 32), batch);
    hipLaunchKernelGGL(k_avg_planes, grd, dim3(256), 0, st, in, ry, rx, n0, n1);
    check_launch("avg_planes");
}

void launch_mix_gather(const float* src, float* dst, const float* M, int nB, int n, int np, int nc, int nout,
                       hipStream_t st)
{
    dim3 blk(256), grd(cdiv(n, 256), nB * nout * nc);
    hipLaunchKernelGGL(k_mix_gather, grd, blk, 0, st, src, dst, M, n, np, nc, nout);
    check_launch("mix_gather");
}

void launch_mix_scatter(const float* src, float* dst, const float* M, int nB, int n, int np, int nc, int nout,
                        bool accumulate, hipStream_t st)
{
    dim3 blk(256), grd(cdiv(n, 256), nB * nout * nc);
    hipLaunchKernelGGL(k_mix_scatter, grd, blk, 0, st, src, dst, M, n, np, nc, nout, accumulate ? 1 : 0);
    check_launch("mix_scatter");
}

void launch_fill(float* p, float v, size_t n, hipStream_t st)
{
    if (n == 0) return;
    hipLaunchKernelGGL(k_fill, dim3(cdiv((long)n, 256)), dim3(256), 0, st, p, v, n);
    check_launch("fill");
}

void launch_axpy(float* y, const float* x, float a, size_t n, hipStream_t st)
{
    if (n == 0) return;
    hipLaunchKernelGGL(k_axpy, dim3(cdiv((long)n, 256)), dim3(256), 0, st, y, x, a, n);
    check_launch("axpy");
}

} // namespace rn
