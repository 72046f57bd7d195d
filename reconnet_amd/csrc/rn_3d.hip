// 3D projectors for gfx950: arbitrary-geometry Siddon (parallel / cone),
// DD tomosynthesis, the cone OS-SQS data step and the helical BP.
//
// Reference counterparts: Siddon.cu:11-351 (tracing), SiddonParallel.cu:11-105,
// SiddonCone.cu:11-68, DistanceDriven3D.cu:139-227 / 409-559, ossqs.cu:163-333,
// Recon3D/HelicalBP.cu:10-83.
//
// Siddon tracing keeps the reference's voxel walk, but each crossing
// parameter is computed directly from the boundary index, (b - s) / d, instead
// of by repeated FP32 addition, so rounding does not accumulate along a ray.
// The arbitrary-geometry BP is the exact transpose of that walk; with detector
// axes and sources free per view there is no cheap footprint inversion, so it
// scatters with hardware float atomics (global_atomic_add_f32).  The DD
// tomosynthesis pair integrates footprints by direct 2D overlap sums in FP32
// instead of the reference's FP64 integral images.

#include "rn_3d.h"
#include "rn_fan.h"
#include "rn_tune.h"

#include <cmath>
#include <vector>

namespace rn {

namespace {

struct Grid3K {
    int nx, ny, nz;
    float dx, dy, dz, cx, cy, cz;
};

struct F3 { float x, y, z; };

__device__ __forceinline__ F3 ld3(const float* p, int i) { return F3{p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }

// MoveSourceDstNearGrid (SiddonParallel.cu:35-55, cudaMath.h:25-60)
__device__ void move_near_grid(F3& s, F3& t, const Grid3K& g)
{
    const float ex = g.nx * g.dx, ey = g.ny * g.dy, ez = g.nz * g.dz;
    const float r = sqrtf(ex * ex + ey * ey + ez * ez);
    float dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
    const float len = sqrtf(dx * dx + dy * dy + dz * dz);
    if (len >= 1e-6f) { dx /= len; dy /= len; dz /= len; }
    const float t0 = (g.cx - s.x) * dx + (g.cy - s.y) * dy + (g.cz - s.z) * dz;
    const float t1 = (t.x - g.cx) * dx + (t.y - g.cy) * dy + (t.z - g.cz) * dz;
    if (t0 > r) { s.x += (t0 - r) * dx; s.y += (t0 - r) * dy; s.z += (t0 - r) * dz; }
    if (t1 > r) { t.x -= (t1 - r) * dx; t.y -= (t1 - r) * dy; t.z -= (t1 - r) * dz; }
}

__device__ __forceinline__ void arb_ray(const ArbGeo& a, const Grid3K& g, bool parallel, const float* C,
                                        const float* U, const float* V, const float* S, int view, int iu, int iv,
                                        F3& src, F3& dst)
{
    const float u = (iu - a.off_u - (a.nu - 1) / 2.0f) * a.du;
    const float v = (iv - a.off_v - (a.nv - 1) / 2.0f) * a.dv;
    const F3 c = ld3(C, view), du = ld3(U, view), dv = ld3(V, view), sd = ld3(S, view);
    dst = F3{c.x + du.x * u + dv.x * v, c.y + du.y * u + dv.y * v, c.z + du.z * u + dv.z * v};
    if (parallel) {
        // GetSrcDstForParallel (SiddonParallel.cu:11-32)
        const float m1 = sqrtf((g.cx - c.x) * (g.cx - c.x) + (g.cy - c.y) * (g.cy - c.y) + (g.cz - c.z) * (g.cz - c.z));
        const float ex = g.nx * g.dx, ey = g.ny * g.dy, ez = g.nz * g.dz;
        const float m2 = sqrtf(ex * ex + ey * ey + ez * ez) / 2;
        const float m = fmaxf(m1, m2) * 1.1f;
        src = F3{c.x + sd.x * m + du.x * u + dv.x * v, c.y + sd.y * m + du.y * u + dv.y * v,
                 c.z + sd.z * m + du.z * u + dv.z * v};
    } else {
        src = sd;
    }
    move_near_grid(src, dst, g);
}

// Siddon walk (Siddon.cu:90-238).  f(voxel, length), voxel the linear index
// x*ny*nz + y*nz + z, or with OFF32 that index times 4 nC as a 32-bit byte
// offset, kept by adding the axis stride at each step (a slice's volume below
// 4 GiB: checked on the host).
template <bool OFF32, class F>
__device__ void siddon_walk(F3 src, F3 dst, const Grid3K& g, int nC, F f)
{
    const float eps = 1e-6f;
    const float dist = sqrtf((src.x - dst.x) * (src.x - dst.x) + (src.y - dst.y) * (src.y - dst.y) +
                             (src.z - dst.z) * (src.z - dst.z));
    const float sx = (src.x - g.cx) / g.dx + g.nx / 2.0f, sy = (src.y - g.cy) / g.dy + g.ny / 2.0f,
                sz = (src.z - g.cz) / g.dz + g.nz / 2.0f;
    const float tx = (dst.x - g.cx) / g.dx + g.nx / 2.0f, ty = (dst.y - g.cy) / g.dy + g.ny / 2.0f,
                tz = (dst.z - g.cz) / g.dz + g.nz / 2.0f;
    const float ddx = tx - sx, ddy = ty - sy, ddz = tz - sz;
    float a0x = 1, a1x = 0, a0y = 1, a1y = 0, a0z = 1, a1z = 0;
    if (fabsf(ddx) > eps) { a0x = -sx / ddx; a1x = (g.nx - sx) / ddx; } else if (sx < 0 || sx > g.nx) return;
    if (fabsf(ddy) > eps) { a0y = -sy / ddy; a1y = (g.ny - sy) / ddy; } else if (sy < 0 || sy > g.ny) return;
    if (fabsf(ddz) > eps) { a0z = -sz / ddz; a1z = (g.nz - sz) / ddz; } else if (sz < 0 || sz > g.nz) return;
    const float amin = fmaxf(0.f, fmaxf(fminf(a0x, a1x), fmaxf(fminf(a0y, a1y), fminf(a0z, a1z))));
    const float amax = fminf(1.f, fminf(fmaxf(a0x, a1x), fminf(fmaxf(a0y, a1y), fmaxf(a0z, a1z))));
    if (amax <= amin) return;
    int gx = (int)(sx + amin * ddx), gy = (int)(sy + amin * ddy), gz = (int)(sz + amin * ddz);
    if (fabsf(ddx) > eps) gx = min(max(gx, 0), g.nx - 1);
    if (fabsf(ddy) > eps) gy = min(max(gy, 0), g.ny - 1);
    if (fabsf(ddz) > eps) gz = min(max(gz, 0), g.nz - 1);
    if (gx < 0 || gx >= g.nx || gy < 0 || gy >= g.ny || gz < 0 || gz >= g.nz) return;
    const int px = ddx > 0, py = ddy > 0, pz = ddz > 0;
    // next boundary index per axis (OutboundFirstVoxel) and its crossing parameter
    float bx = (ddx > eps) ? gx + 1 : gx, by = (ddy > eps) ? gy + 1 : gy, bz = (ddz > eps) ? gz + 1 : gz;
    const bool mx = fabsf(ddx) > eps, my = fabsf(ddy) > eps, mz = fabsf(ddz) > eps;
    const float ix = mx ? dist / ddx : 0.f, iy = my ? dist / ddy : 0.f, iz = mz ? dist / ddz : 0.f;
    const float stx = px ? 1.f : -1.f, sty = py ? 1.f : -1.f, stz = pz ? 1.f : -1.f;
    float ax = mx ? (bx - sx) * ix : 2.f * dist;
    float ay = my ? (by - sy) * iy : 2.f * dist;
    float az = mz ? (bz - sz) * iz : 2.f * dist;
    // with no motion along an axis the reference keeps alpha = 2*dist + k*0
    float prev = amin * dist;
    const int maxit = g.nx + g.ny + g.nz + 4;
    // byte offset of the current voxel and the signed steps along each axis
    // (unsigned arithmetic: a step out of the grid ends the walk unused)
    const unsigned oz = 4u * (unsigned)nC, oy = oz * (unsigned)g.nz, ox = oy * (unsigned)g.ny;
    unsigned off = OFF32 ? ((unsigned)gx * (unsigned)g.ny + (unsigned)gy) * oy + (unsigned)gz * oz : 0u;
    const unsigned dox = px ? ox : 0u - ox, doy = py ? oy : 0u - oy, doz = pz ? oz : 0u - oz;
    for (int it = 0; it < maxit; ++it) {
        const int cx = gx, cy = gy, cz = gz;
        const unsigned coff = off;
        float now;
        bool done = false;
        if (ax < ay && ax < az) {
            now = ax;
            bx += stx; ax = mx ? (bx - sx) * ix : ax;
            gx += px ? 1 : -1; done = (gx >= g.nx || gx < 0);
            off += dox;
        } else if (ay < az) {
            now = ay;
            by += sty; ay = my ? (by - sy) * iy : ay;
            gy += py ? 1 : -1; done = (gy >= g.ny || gy < 0);
            off += doy;
        } else {
            now = az;
            bz += stz; az = mz ? (bz - sz) * iz : az;
            gz += pz ? 1 : -1; done = (gz >= g.nz || gz < 0);
            off += doz;
        }
        if (OFF32) f((long)coff, now - prev);
        else f(((long)cx * g.ny + cy) * g.nz + cz, now - prev);
        prev = now;
        if (done) break;
    }
}

// One ray per lane; a wave holds 64 adjacent detector rows of one column, so
// its rays share their in-plane path when the rows run along z and read
// adjacent z voxels (z is the innermost image index), and its outputs are
// adjacent; 4 columns per workgroup.
template <bool OFF32>
__global__ __launch_bounds__(256) void k_siddon_arb_fp(ArbGeo a, Grid3K g, int parallel, const float* __restrict__ img,
                                                       float* __restrict__ prj, const float* C, const float* U,
                                                       const float* V, const float* S, int nC)
{
    const int iv = blockIdx.x * 64 + (int)(threadIdx.x & 63);
    const int iu = blockIdx.y * 4 + (int)(threadIdx.x >> 6);
    const int view = blockIdx.z % a.nview, bc = blockIdx.z / a.nview;
    const int c = bc % nC, b = bc / nC;
    if (iu >= a.nu || iv >= a.nv) return;
    F3 s, t;
    arb_ray(a, g, parallel != 0, C, U, V, S, view, iu, iv, s, t);
    const float* base = img + (long)b * g.nx * g.ny * g.nz * nC + c;
    float val = 0.f;
    if (OFF32) {
        const char* bb = reinterpret_cast<const char*>(base);
        siddon_walk<true>(s, t, g, nC, [&](long off, float len) {
            val += *reinterpret_cast<const float*>(bb + (unsigned)off) * len;
        });
    } else {
        siddon_walk<false>(s, t, g, nC, [&](long vox, float len) { val += base[vox * nC] * len; });
    }
    prj[((((long)b * a.nu + iu) * a.nview + view) * a.nv + iv) * nC + c] = val;
}

// Siddon backprojection as a gather, the transpose of k_siddon_arb_fp: a
// voxel collects, per view, the rays of the detector cells that lie in the
// projection of its 8 corners, each weighted by the ray's chord through the
// voxel.  The ray is the walk's: from its start point (the source; for
// parallel views the detector point moved back by m along invRayDir) through
// the grid and on past the detector point, and it is used only if it enters
// the grid before the detector point (the walk's amin < amax with amax =
// min(1, exit)); moving the start point to the grid (MoveSourceDstNearGrid)
// keeps it outside the grid, so it changes no chord.  One wave holds a
// column of 64 voxels along z with (x, y) wave-uniform; no atomics, every
// voxel written once.

// [enter, exit] of the ray o + t d in the box [lo, hi] (empty: enter > exit);
// an axis with d = 0 keeps the interval if lo <= o < hi (the walk's voxel
// index of a stationary coordinate)
__device__ __forceinline__ void slab(const F3& o, const F3& d, const F3& lo, const F3& hi, float& t0, float& t1)
{
    t0 = -INFINITY;
    t1 = INFINITY;
    const float oc[3] = {o.x, o.y, o.z}, dc[3] = {d.x, d.y, d.z};
    const float lc[3] = {lo.x, lo.y, lo.z}, hc[3] = {hi.x, hi.y, hi.z};
    #pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (dc[k] != 0.0f) {
            const float inv = __builtin_amdgcn_rcpf(dc[k]);
            const float a0 = (lc[k] - oc[k]) * inv, a1 = (hc[k] - oc[k]) * inv;
            t0 = fmaxf(t0, fminf(a0, a1));
            t1 = fminf(t1, fmaxf(a0, a1));
        } else if (!(oc[k] >= lc[k] && oc[k] < hc[k])) {
            t1 = -INFINITY;
        }
    }
}

// [s0, s1] on the ray p(s) = s d - r (a voxel-centred frame) inside the box
// |p| <= h, as slab() with the half-open faces: an axis with d = 0 keeps the
// interval if -h < r <= h.  r is small (the ray passes within a few voxels of
// the centre), so the parameters carry float precision relative to the chord
// instead of relative to the source distance.
__device__ __forceinline__ void slab_local(const F3& r, const F3& d, const F3& h, float& s0, float& s1)
{
    s0 = -INFINITY;
    s1 = INFINITY;
    const float rc[3] = {r.x, r.y, r.z}, dc[3] = {d.x, d.y, d.z}, hc[3] = {h.x, h.y, h.z};
    #pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (dc[k] != 0.0f) {
            const float inv = __builtin_amdgcn_rcpf(dc[k]);
            const float a0 = (rc[k] - hc[k]) * inv, a1 = (rc[k] + hc[k]) * inv;
            s0 = fmaxf(s0, fminf(a0, a1));
            s1 = fminf(s1, fmaxf(a0, a1));
        } else if (!(rc[k] > -hc[k] && rc[k] <= hc[k])) {
            s1 = -INFINITY;
        }
    }
}

// the wave's copy of a value every active lane holds alike (an SGPR operand)
__device__ __forceinline__ float wave_uniform(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ double wave_uniform(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Per view, in FP64: the detector normal N = U x V, the dual basis (Ud, Vd) of
// (U, V) and the projection constants: cone A = (C - S).N, su, sv = (S - C).Ud,
// (S - C).Vd; parallel sdn, sdu, sdv = invRayDir.(N, Ud, Vd) and the start
// distance m of GetSrcDstForParallel (SiddonParallel.cu:11-32).
__global__ void k_siddon_arb_views(ArbGeo a, Grid3K g, int parallel, const float* C, const float* U, const float* V,
                                   const float* S, float4* __restrict__ vt)
{
    const int view = blockIdx.x * blockDim.x + threadIdx.x;
    if (view >= a.nview) return;
    double c[3], u[3], v[3], sd[3];
    for (int k = 0; k < 3; ++k) {
        c[k] = C[3 * view + k]; u[k] = U[3 * view + k]; v[k] = V[3 * view + k]; sd[k] = S[3 * view + k];
    }
    const double n[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
    const double uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2], vv = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    const double uv = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
    const double idet = 1.0 / (uu * vv - uv * uv);
    double ud[3], vd[3];
    for (int k = 0; k < 3; ++k) { ud[k] = (vv * u[k] - uv * v[k]) * idet; vd[k] = (uu * v[k] - uv * u[k]) * idet; }
    auto dot = [](const double* p, const double* q) { return p[0] * q[0] + p[1] * q[1] + p[2] * q[2]; };
    double w, wu, wv, m = 0.0;
    if (!parallel) {
        const double cs[3] = {c[0] - sd[0], c[1] - sd[1], c[2] - sd[2]};
        w = dot(cs, n); wu = -dot(cs, ud); wv = -dot(cs, vd);
    } else {
        w = dot(sd, n); wu = dot(sd, ud); wv = dot(sd, vd);
        // the walk's start distance, in its float arithmetic
        const float fx = g.cx - C[3 * view], fy = g.cy - C[3 * view + 1], fz = g.cz - C[3 * view + 2];
        const float ex = g.nx * g.dx, ey = g.ny * g.dy, ez = g.nz * g.dz;
        m = fmaxf(sqrtf(fx * fx + fy * fy + fz * fz), sqrtf(ex * ex + ey * ey + ez * ez) / 2) * 1.1f;
    }
    vt[4 * view + 0] = make_float4((float)n[0], (float)n[1], (float)n[2], (float)w);
    vt[4 * view + 1] = make_float4((float)ud[0], (float)ud[1], (float)ud[2], (float)wu);
    vt[4 * view + 2] = make_float4((float)vd[0], (float)vd[1], (float)vd[2], (float)wv);
    vt[4 * view + 3] = make_float4((float)m, 0.0f, 0.0f, 0.0f);
}

// What one lane's voxels take from one cone view whose detector rows run
// along z and whose columns lie in a horizontal plane (V = (0, 0, v),
// U.z = 0).  N and Ud are then horizontal and Vd = (0, 0, 1/v): a voxel's
// detector columns depend on (x, y) only, so the column range and each
// column's in-plane ray direction and x/y slabs are the wave's (a wave holds
// one (x, y)); the rows scale with z and each adds its z slab.  A lane holds
// ZPL voxels stacked in z from vlz (bottom face) and vcz (centre of the
// lowest, FP64); every row is loaded once for all of them.
struct SidBpCol {
    F3 vlo, vhi;          // the wave's x/y faces (z unused)
    F3 glo, ghi, hw;      // grid box, voxel half widths
    double vcx, vcy;      // the wave's voxel centre (x, y), FP64
    float cu, cv, gdz;
};

template <int ZPL>
__device__ __forceinline__ void siddon_rows_z_view(const ArbGeo& a, const SidBpCol& w, int view, const F3& Cv,
                                                   const F3& Uv, const F3& Vv, const F3& Sv, const float4& t0v,
                                                   const float4& t1v, const float4& t2v, float vlz, double vcz,
                                                   const float* __restrict__ q, int nC, float (&acc)[ZPL])
{
    const F3 N{t0v.x, t0v.y, t0v.z}, Ud{t1v.x, t1v.y, t1v.z};
    const float A = t0v.w, su = t1v.w, sv = t2v.w, vdz = t2v.z;
    float umin = INFINITY, umax = -INFINITY, tmin = INFINITY, tmax = -INFINITY;
    bool ok = true;
    #pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float wxk = ((k & 1) ? w.vhi.x : w.vlo.x) - Sv.x, wyk = ((k & 2) ? w.vhi.y : w.vlo.y) - Sv.y;
        const float den = fmaf(wxk, N.x, wyk * N.y);
        ok = ok && (den * A > 0.f);
        const float t = A * __builtin_amdgcn_rcpf(den);
        const float u = fmaf(t, fmaf(wxk, Ud.x, wyk * Ud.y), su);
        umin = fminf(umin, u); umax = fmaxf(umax, u);
        tmin = fminf(tmin, t); tmax = fmaxf(tmax, t);
    }
    if (!ok) return;
    // rows: the corners' v over the lane's stack of voxels
    const float z0 = (vlz - Sv.z) * vdz, z1 = (vlz + ZPL * w.gdz - Sv.z) * vdz;
    const float vmin = fminf(fminf(tmin * z0, tmax * z0), fminf(tmin * z1, tmax * z1)) + sv;
    const float vmax = fmaxf(fmaxf(tmin * z0, tmax * z0), fmaxf(tmin * z1, tmax * z1)) + sv;
    const float fu0 = umin / a.du + w.cu, fu1 = umax / a.du + w.cu;
    const float fv0 = vmin / a.dv + w.cv, fv1 = vmax / a.dv + w.cv;
    const int iu0 = max((int)ceilf(fminf(fu0, fu1) - 1e-3f), 0), iu1 = min((int)floorf(fmaxf(fu0, fu1) + 1e-3f), a.nu - 1);
    const int iv0 = max((int)ceilf(fminf(fv0, fv1) - 1e-3f), 0), iv1 = min((int)floorf(fmaxf(fv0, fv1) + 1e-3f), a.nv - 1);
    const double wx = wave_uniform(w.vcx - Sv.x), wy = wave_uniform(w.vcy - Sv.y), wz = vcz - Sv.z;
    // rows in float: the lowest voxel's z offset from the source split in two
    // floats, the detector centre's height above the source rounded once
    const float wz_hi = (float)wz, wz_lo = (float)(wz - wz_hi), czs = (float)((double)Cv.z - Sv.z);
    for (int iu = iu0; iu <= iu1; ++iu) {
        const double uc = (double)(iu - w.cu) * a.du;
        const double dxd = wave_uniform(fma((double)Uv.x, uc, (double)Cv.x) - Sv.x);
        const double dyd = wave_uniform(fma((double)Uv.y, uc, (double)Cv.y) - Sv.y);
        const float dx = wave_uniform((float)dxd), dy = wave_uniform((float)dyd);
        const float dxy2 = wave_uniform(fmaf(dx, dx, dy * dy));
        // tp: the column's in-plane closest approach to the voxel (any nearby
        // value serves: r is exact for the tp used); the ray's points are
        // S + (tp + s) d, at s d - r from the voxel centre
        const float tp = wave_uniform((float)(wx * dxd + wy * dyd) * __builtin_amdgcn_rcpf(dxy2));
        const float rx = wave_uniform((float)fma(-(double)tp, dxd, wx));
        const float ry = wave_uniform((float)fma(-(double)tp, dyd, wy));
        float xy0 = -INFINITY, xy1 = INFINITY;
        if (dx != 0.f) {
            const float inv = __builtin_amdgcn_rcpf(dx);
            const float a0 = (rx - w.hw.x) * inv, a1 = (rx + w.hw.x) * inv;
            xy0 = fmaxf(xy0, fminf(a0, a1)); xy1 = fminf(xy1, fmaxf(a0, a1));
        } else if (!(rx > -w.hw.x && rx <= w.hw.x)) {
            xy1 = -INFINITY;
        }
        if (dy != 0.f) {
            const float inv = __builtin_amdgcn_rcpf(dy);
            const float a0 = (ry - w.hw.y) * inv, a1 = (ry + w.hw.y) * inv;
            xy0 = fmaxf(xy0, fminf(a0, a1)); xy1 = fminf(xy1, fmaxf(a0, a1));
        } else if (!(ry > -w.hw.y && ry <= w.hw.y)) {
            xy1 = -INFINITY;
        }
        xy0 = wave_uniform(fmaxf(xy0, -tp));          // t >= 0: from the source on
        xy1 = wave_uniform(xy1);
        if (!(xy1 > xy0)) continue;
        // a voxel can lie beyond the detector point only if the column's rays
        // are still inside the voxel column there
        const bool far = xy1 > 1.f - tp;
        const float* qc = q + ((long)iu * a.nview + view) * a.nv * nC;
        // the row's ray height is affine in the row index
        const float dzs = Vv.z * a.dv, dz_0 = fmaf(-w.cv, dzs, czs);
        for (int iv = iv0; iv <= iv1; ++iv) {
            const float dz = fmaf(dzs, (float)iv, dz_0), rz = fmaf(-tp, dz, wz_hi) + wz_lo;
            const float len = __builtin_amdgcn_sqrtf(fmaf(dz, dz, dxy2));      // hardware sqrt, 1 ulp
            const float val = qc[(long)iv * nC];
            // the lowest voxel's z slab; voxel k's is shifted by k dz_vox / dz
            float zl, zh, st;
            if (dz != 0.f) {
                const float inv = __builtin_amdgcn_rcpf(dz);
                const float a0 = (rz - w.hw.z) * inv, a1 = (rz + w.hw.z) * inv;
                zl = fminf(a0, a1); zh = fmaxf(a0, a1); st = w.gdz * inv;
            } else {
                // a ray at a voxel's height for all t: voxel k holds it if
                // -h < rz + k dz_vox <= h
                zl = -INFINITY; zh = INFINITY; st = 0.f;
            }
            #pragma unroll
            for (int k = 0; k < ZPL; ++k) {
                if (dz == 0.f) {
                    const float rzk = fmaf((float)k, w.gdz, rz);
                    if (!(rzk > -w.hw.z && rzk <= w.hw.z)) continue;
                }
                const float s0 = fmaxf(xy0, fmaf((float)k, st, zl)), s1 = fminf(xy1, fmaf((float)k, st, zh));
                if (!(s1 > s0)) continue;
                if (far && s0 >= 1.f - tp) {
                    // a voxel beyond the detector point: the ray counts only if
                    // it entered the grid before that point
                    float g0, g1;
                    slab(Sv, F3{dx, dy, dz}, w.glo, w.ghi, g0, g1);
                    if (!(fminf(g1, 1.f) > fmaxf(g0, 0.f))) continue;
                }
                acc[k] = fmaf((s1 - s0) * len, val, acc[k]);
            }
        }
    }
}

// ROWS_Z: the caller has found every view to be an upright cone view (the
// kernel then has no general-view path: its FP64 ray set-up would double
// the register count); ZPL voxels per lane stacked in z (ROWS_Z only).
template <bool ROWS_Z, int ZPL>
__global__ __launch_bounds__(256) void k_siddon_arb_bp(ArbGeo a, Grid3K g, int parallel, const float* __restrict__ prj,
                                                       float* __restrict__ img, const float* C, const float* U,
                                                       const float* V, const float* S, const float4* __restrict__ vt,
                                                       int nC)
{
    static_assert(ROWS_Z || ZPL == 1, "stacked voxels need upright cone views");
    const int iz = (blockIdx.x * 64 + (threadIdx.x & 63)) * ZPL;
    const int iy = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (int)(threadIdx.x >> 6));
    const int ix = blockIdx.z % g.nx, bc = blockIdx.z / g.nx;
    if (iz >= g.nz || iy >= g.ny) return;
    const int cc = bc % nC, b = bc / nC;
    const float* q = prj + (long)b * a.nu * a.nview * a.nv * nC + cc;
    // wave-uniform values are kept in scalar registers (wave_uniform)
    SidBpCol w;
    const float vlz = g.cz + (iz - g.nz / 2.0f) * g.dz;
    w.vlo = F3{wave_uniform(g.cx + (ix - g.nx / 2.0f) * g.dx), wave_uniform(g.cy + (iy - g.ny / 2.0f) * g.dy), vlz};
    w.vhi = F3{wave_uniform(w.vlo.x + g.dx), wave_uniform(w.vlo.y + g.dy), vlz + g.dz};
    w.glo = F3{wave_uniform(g.cx - g.nx / 2.0f * g.dx), wave_uniform(g.cy - g.ny / 2.0f * g.dy),
               wave_uniform(g.cz - g.nz / 2.0f * g.dz)};
    w.ghi = F3{wave_uniform(g.cx + g.nx / 2.0f * g.dx), wave_uniform(g.cy + g.ny / 2.0f * g.dy),
               wave_uniform(g.cz + g.nz / 2.0f * g.dz)};
    // the voxel centre in FP64 and its half widths: chords are measured from a
    // point of the ray next to the voxel, because parameters counted from
    // the source (~600 mm away) lose ~5e-5 mm to float rounding
    w.vcx = wave_uniform(g.cx + (ix + 0.5 - g.nx / 2.0) * g.dx);
    w.vcy = wave_uniform(g.cy + (iy + 0.5 - g.ny / 2.0) * g.dy);
    const double vcz = g.cz + (iz + 0.5 - g.nz / 2.0) * g.dz;
    w.hw = F3{wave_uniform(0.5f * g.dx), wave_uniform(0.5f * g.dy), wave_uniform(0.5f * g.dz)};
    w.cu = wave_uniform((a.nu - 1) / 2.0f + a.off_u);
    w.cv = wave_uniform((a.nv - 1) / 2.0f + a.off_v);
    w.gdz = wave_uniform(g.dz);
    auto dot = [](const F3& p, const F3& r) { return p.x * r.x + p.y * r.y + p.z * r.z; };
    float acc[ZPL];
    #pragma unroll
    for (int k = 0; k < ZPL; ++k) acc[k] = 0.f;
    for (int view = 0; view < a.nview; ++view) {
        const F3 Cv = ld3(C, view), Uv = ld3(U, view), Vv = ld3(V, view), Sv = ld3(S, view);
        const float4 t0v = vt[4 * view], t1v = vt[4 * view + 1], t2v = vt[4 * view + 2];
        if (ROWS_Z || (!parallel && Vv.x == 0.f && Vv.y == 0.f && Uv.z == 0.f)) {
            siddon_rows_z_view<ZPL>(a, w, view, Cv, Uv, Vv, Sv, t0v, t1v, t2v, vlz, vcz, q, nC, acc);
            continue;
        }
        if constexpr (!ROWS_Z) {
            // any other view: the voxel's eight corners on the detector (u, v in mm)
            const F3 N{t0v.x, t0v.y, t0v.z}, Ud{t1v.x, t1v.y, t1v.z}, Vd{t2v.x, t2v.y, t2v.z};
            const F3 vlo = w.vlo, vhi = w.vhi;
            float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
            bool ok = true;
            float m = 0.f;
            if (!parallel) {
                const float A = t0v.w, su = t1v.w, sv = t2v.w;
                #pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const F3 wk{((k & 1) ? vhi.x : vlo.x) - Sv.x, ((k & 2) ? vhi.y : vlo.y) - Sv.y,
                                ((k & 4) ? vhi.z : vlo.z) - Sv.z};
                    const float den = dot(wk, N);
                    ok = ok && (den * A > 0.f);
                    const float t = A * __builtin_amdgcn_rcpf(den);
                    const float u = fmaf(t, dot(wk, Ud), su), v = fmaf(t, dot(wk, Vd), sv);
                    umin = fminf(umin, u); umax = fmaxf(umax, u);
                    vmin = fminf(vmin, v); vmax = fmaxf(vmax, v);
                }
            } else {
                const float sdn = t0v.w, sdu = t1v.w, sdv = t2v.w;
                ok = sdn != 0.f;
                const float isdn = -__builtin_amdgcn_rcpf(sdn);
                #pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const F3 wk{((k & 1) ? vhi.x : vlo.x) - Cv.x, ((k & 2) ? vhi.y : vlo.y) - Cv.y,
                                ((k & 4) ? vhi.z : vlo.z) - Cv.z};
                    const float tau = dot(wk, N) * isdn;
                    const float u = fmaf(tau, sdu, dot(wk, Ud)), v = fmaf(tau, sdv, dot(wk, Vd));
                    umin = fminf(umin, u); umax = fmaxf(umax, u);
                    vmin = fminf(vmin, v); vmax = fmaxf(vmax, v);
                }
                m = vt[4 * view + 3].x;
            }
            if (!ok) continue;
            // cells whose centre ray meets the corners' bounding box
            const float fu0 = umin / a.du + w.cu, fu1 = umax / a.du + w.cu;
            const float fv0 = vmin / a.dv + w.cv, fv1 = vmax / a.dv + w.cv;
            const int iu0 = max((int)ceilf(fminf(fu0, fu1) - 1e-3f), 0);
            const int iu1 = min((int)floorf(fmaxf(fu0, fu1) + 1e-3f), a.nu - 1);
            const int iv0 = max((int)ceilf(fminf(fv0, fv1) - 1e-3f), 0);
            const int iv1 = min((int)floorf(fmaxf(fv0, fv1) + 1e-3f), a.nv - 1);
            for (int iu = iu0; iu <= iu1; ++iu) {
                const double uc = (double)(iu - w.cu) * a.du;
                const float* qc = q + ((long)iu * a.nview + view) * a.nv * nC;
                for (int iv = iv0; iv <= iv1; ++iv) {
                    const double vc = (double)(iv - w.cv) * a.dv;
                    const double dst[3] = {Cv.x + Uv.x * uc + Vv.x * vc, Cv.y + Uv.y * uc + Vv.y * vc,
                                           Cv.z + Uv.z * uc + Vv.z * vc};
                    const double o[3] = {parallel ? dst[0] + (double)Sv.x * m : (double)Sv.x,
                                         parallel ? dst[1] + (double)Sv.y * m : (double)Sv.y,
                                         parallel ? dst[2] + (double)Sv.z * m : (double)Sv.z};
                    const double dd[3] = {dst[0] - o[0], dst[1] - o[1], dst[2] - o[2]};
                    const double wv[3] = {w.vcx - o[0], w.vcy - o[1], vcz - o[2]};
                    const float tp = (float)((wv[0] * dd[0] + wv[1] * dd[1] + wv[2] * dd[2]) /
                                             (dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2]));
                    const F3 r{(float)fma(-(double)tp, dd[0], wv[0]), (float)fma(-(double)tp, dd[1], wv[1]),
                               (float)fma(-(double)tp, dd[2], wv[2])};
                    const F3 d{(float)dd[0], (float)dd[1], (float)dd[2]};
                    float s0, s1;
                    slab_local(r, d, w.hw, s0, s1);
                    s0 = fmaxf(s0, -tp);
                    if (!(s1 > s0)) continue;
                    if (s0 >= 1.f - tp) {
                        // a voxel beyond the detector point: the ray counts only
                        // if it entered the grid before that point
                        const F3 of{(float)o[0], (float)o[1], (float)o[2]};
                        float g0, g1;
                        slab(of, d, w.glo, w.ghi, g0, g1);
                        if (!(fminf(g1, 1.f) > fmaxf(g0, 0.f))) continue;
                    }
                    acc[0] = fmaf((s1 - s0) * __builtin_amdgcn_sqrtf(dot(d, d)), qc[(long)iv * nC], acc[0]);
                }
            }
        }
    }
    float* out = img + ((((long)b * g.nx + ix) * g.ny + iy) * g.nz + iz) * nC + cc;
    #pragma unroll
    for (int k = 0; k < ZPL; ++k)
        if (iz + k < g.nz) out[(long)k * nC] = acc[k];
}

// Row windows of the cone backprojections: len(row) q(row) of every (slice, view,
// detector column), len the length from the source to the cell centre, as floats
// with kConePad zero rows before and 4 after (pitch nv + kConePad + 4).
constexpr int kConePad = 8;

__global__ __launch_bounds__(256) void k_cone_rows(ArbGeo a, const float* __restrict__ prj, const float* Cp,
                                                      const float* Up, const float* Vp, const float* Sp, int nC,
                                                      long n, float* __restrict__ Q)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int nvp = a.nv + kConePad + 4;
    const long col = i / nvp;
    const int iv = (int)(i - col * nvp) - kConePad;
    float f = 0.0f;
    if (iv >= 0 && iv < a.nv) {
        const int iu = (int)(col % a.nu);
        const long rest = col / a.nu;
        const int view = (int)(rest % a.nview);
        const long bc = rest / a.nview;
        const int cc = (int)(bc % nC), b = (int)(bc / nC);
        const F3 c = ld3(Cp, view), U = ld3(Up, view), V = ld3(Vp, view), s = ld3(Sp, view);
        const float uc = ((float)iu - ((a.nu - 1) / 2.0f + a.off_u)) * a.du;
        const float lx = fmaf(uc, U.x, c.x) - s.x, ly = fmaf(uc, U.y, c.y) - s.y;
        const float lzs = V.z * a.dv, lz_0 = fmaf(-((a.nv - 1) / 2.0f + a.off_v), lzs, fmaf(uc, U.z, c.z) - s.z);
        const float lz = fmaf(lzs, (float)iv, lz_0);
        f = sqrtf(fmaf(lz, lz, fmaf(lx, lx, ly * ly))) *
            prj[((((long)b * a.nu + iu) * a.nview + view) * a.nv + iv) * nC + cc];
    }
    Q[i] = f;
}

// NR adjacent rows of a window at byte offset off (rows -kConePad .. nv + 3)
template <int NR>
__device__ __forceinline__ void cone_rows(const char* __restrict__ Q, unsigned off, float (&v)[NR])
{
    typedef float F4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef float F2 __attribute__((ext_vector_type(2), aligned(4)));
    if constexpr (NR == 4) {
        const F4 x = *reinterpret_cast<const F4*>(Q + off);
        v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
    } else {
        static_assert(NR == 2 || NR == 3, "2, 3 or 4 rows");
        const F2 x = *reinterpret_cast<const F2*>(Q + off);
        v[0] = x[0]; v[1] = x[1];
        if constexpr (NR == 3) v[2] = *reinterpret_cast<const float*>(Q + off + 8u);
    }
}

// maximum over the wave's 64 lanes of a non-negative value
__device__ __forceinline__ int wave_max_nn(int v)
{
    #pragma unroll
    for (int d = 1; d < 64; d <<= 1) v = max(v, __shfl_xor(v, d));
    return __builtin_amdgcn_readfirstlane(v);
}

// Siddon backprojection of upright cone views from column lists: the transpose of
// the walk as in siddon_rows_z_view, organised as k_dd_cone_adj_list.  A group of
// LZ lanes takes one (x, y); per batch of LZ views each lane works out one view's
// detector columns through (x, y) (FP64 ray set-up, the in-plane slab interval
// [xy0, xy1] around the closest approach tp, the rows' affine coordinates) and
// appends them to the group's list; then the group's lanes take LZ consecutive
// voxels of the z range the batch reaches and walk the list.  A voxel's rows on
// an entry are those whose ray meets it between the in-plane crossings: the row
// coordinate (z - Sz) / (t dzs) - dz0 / dzs of its two z faces at t = tp + xy0
// and tp + xy1.  Their chords, in t, are the overlap of the z slab's interval
// with [xy0, xy1], measured from tp like the in-plane interval; the ray's length
// is already in the row windows.  A chord beyond the detector point counts only
// if the ray entered the grid before that point (g0 of the entry, in plane, and
// the row's z entry).
//
// Bound: VALU issue (about 25 instructions per entry and 19 per row, 2 rows per
// entry where a voxel covers less than 2).  190 x 177 x 99 voxels, 240 views, 49
// x 323: 0.93 ms with 16 lanes per (x, y) (0.95 with 32, 1.25 with 8), and 22 us
// for the row windows; 7.4 ms with 64 lanes along z testing every view, column
// and row for 2 stacked voxels each (siddon_rows_z_view).
constexpr int kSidCols = 2;          // list entries per view and round
constexpr int kSidZB = 128;          // z voxels of a workgroup's columns

struct SidEntry {
    float xy0, xy1, tp, Sz;          // in-plane interval around tp; source height
    float ia, ib, c;                 // rows: (z - Sz) ia - c at tp + xy0, ib at tp + xy1
    unsigned off;                    // byte offset of the column's row 0
    float dzc, dzs, g0, pad;         // row iv's ray rises dzc + (iv - cv) dzs (0 exactly on a
                                     // centred detector's middle row); grid entry in plane
};

// Sum over the list's n entries for the voxel whose centre is zh + zl, half height h.
// NR = 2, 3, 4: every entry's voxel meets at most NR rows; NR = 0: `chunks` x 4 rows.
template <int NR, bool FAR>
__device__ __forceinline__ float sid_list_sum(const float4* list, int n, const char* __restrict__ Q, float zh, float zl,
                                              float h, float cv, float fnv, float glz, float ghz, int chunks)
{
    float sum = 0.0f;
    #pragma unroll 2
    for (int i = 0; i < n; ++i) {
        const float4 A = list[3 * i], B = list[3 * i + 1], C = list[3 * i + 2];
        // voxel centre above the source, as a float pair
        const float w = zh - A.w, bb = w - zh;
        const float wl = ((zh - (w - bb)) - (A.w + bb)) + zl;
        const float ub = w - h, ut = w + h;
        const float rmin = fminf(fminf(ub * B.x, ub * B.y), fminf(ut * B.x, ut * B.y)) - B.z;
        const float r0 = ceilf(rmin - 1e-3f);
        auto rows = [&](float rf, const float* v, int count) {
            #pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j >= count) break;
                float dz = fmaf(C.y, (rf - cv) + (float)j, C.x), rz = fmaf(-A.z, dz, w) + wl;
                // a level ray lies in the voxel with -h < rz <= h
                const bool level = fabsf(dz) < 1e-30f;
                dz = level ? 1e-30f : dz;
                rz = level ? fmaf(-1e-6f, h, rz) : rz;
                const float inv = __builtin_amdgcn_rcpf(dz);
                const float m = rz * inv, k = h * inv;
                const float q0 = __builtin_amdgcn_fmed3f(m - k, A.x, A.y), q1 = __builtin_amdgcn_fmed3f(m + k, A.x, A.y);
                float ch = fabsf(q1 - q0);
                if (FAR) {
                    const float gz = fminf((glz - A.w) * inv, (ghz - A.w) * inv);
                    if (fminf(q0, q1) >= 1.0f - A.z && !(fmaxf(C.z, gz) < 1.0f)) ch = 0.0f;
                }
                // a row that misses the voxel adds nothing, whatever its value
                sum = ch > 0.0f ? fmaf(ch, v[j], sum) : sum;
            }
        };
        const float lo = -(float)kConePad;
        if constexpr (NR > 0) {
            const float rf = __builtin_amdgcn_fmed3f(r0, lo, fnv);
            float v[NR];
            cone_rows<NR>(Q, __float_as_uint(B.w) + (unsigned)((int)rf * 4), v);
            rows(rf, v, NR);
        } else {
            for (int c = 0; c < chunks; ++c) {
                const float rf = __builtin_amdgcn_fmed3f(r0 + 4.0f * (float)c, lo, fnv);
                float v[4];
                cone_rows<4>(Q, __float_as_uint(B.w) + (unsigned)((int)rf * 4), v);
                rows(rf, v, 4);
            }
        }
    }
    return sum;
}

template <int LZ>
__global__ __launch_bounds__(256, 4) void k_siddon_cone_bp_list(ArbGeo a, Grid3K g, const float* __restrict__ Q,
                                                                float* __restrict__ img, const float* Cp,
                                                                const float* Up, const float* Vp, const float* Sp,
                                                                const float4* __restrict__ vt, int nC)
{
    constexpr int NG = 64 / LZ, kCap = LZ * kSidCols;
    static_assert(sizeof(SidEntry) == 48, "three float4 per entry");
    __shared__ float4 lists[4][NG * kCap * 3];
    __shared__ float accs[4][NG * kSidZB];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int grp = lane / LZ, lg = lane % LZ;
    const int iy0 = ((int)blockIdx.y * 4 + wv) * NG;
    if (iy0 >= g.ny) return;                       // whole waves (no workgroup barrier below)
    const int iy = iy0 + grp, ix = blockIdx.z % g.nx, bc = blockIdx.z / g.nx;
    const int z0 = (int)blockIdx.x * kSidZB, z1 = min(z0 + kSidZB, g.nz);
    float4* list = lists[wv] + grp * kCap * 3;
    float* acc = accs[wv] + grp * kSidZB;
    for (int z = lg; z < kSidZB; z += LZ) acc[z] = 0.0f;
    const int nvp = a.nv + kConePad + 4;
    const char* Qb = reinterpret_cast<const char*>(Q + (long)bc * a.nview * a.nu * nvp);
    const float vlx = g.cx + (ix - g.nx / 2.0f) * g.dx, vly = g.cy + (iy - g.ny / 2.0f) * g.dy;
    const double vcx = g.cx + (ix + 0.5 - g.nx / 2.0) * g.dx, vcy = g.cy + (iy + 0.5 - g.ny / 2.0) * g.dy;
    const float hx = 0.5f * g.dx, hy = 0.5f * g.dy, hz = 0.5f * g.dz;
    const float glx = g.cx - g.nx / 2.0f * g.dx, ghx = g.cx + g.nx / 2.0f * g.dx;
    const float gly = g.cy - g.ny / 2.0f * g.dy, ghy = g.cy + g.ny / 2.0f * g.dy;
    const float glz = g.cz - g.nz / 2.0f * g.dz, ghz = g.cz + g.nz / 2.0f * g.dz;
    const float cu = (a.nu - 1) / 2.0f + a.off_u, cv = (a.nv - 1) / 2.0f + a.off_v;
    const float fz0 = (float)z0, fz1 = (float)z1, fnv = (float)a.nv, idz = 1.0f / g.dz;
    const unsigned long long gmask = LZ == 64 ? ~0ull : ((1ull << (LZ & 63)) - 1ull);
    for (int vb = 0; vb < a.nview; vb += LZ) {
        const int view = min(vb + lg, a.nview - 1);
        const F3 Cv = ld3(Cp, view), Uv = ld3(Up, view), Vv = ld3(Vp, view), Sv = ld3(Sp, view);
        const float4 t0v = vt[4 * view], t1v = vt[4 * view + 1];
        // columns whose centre ray can meet the voxel column: its corners on the detector
        float umin = INFINITY, umax = -INFINITY;
        bool ok = vb + lg < a.nview && iy < g.ny;
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float wxk = vlx + ((k & 1) ? g.dx : 0.0f) - Sv.x, wyk = vly + ((k & 2) ? g.dy : 0.0f) - Sv.y;
            const float den = fmaf(wxk, t0v.x, wyk * t0v.y);
            ok = ok && (den * t0v.w > 0.f);
            const float u = fmaf(t0v.w * __builtin_amdgcn_rcpf(den), fmaf(wxk, t1v.x, wyk * t1v.y), t1v.w);
            umin = fminf(umin, u); umax = fmaxf(umax, u);
        }
        int u0 = 0, ncol = 0;
        if (ok) {
            const float fu0 = umin / a.du + cu, fu1 = umax / a.du + cu;
            u0 = max((int)ceilf(fminf(fu0, fu1) - 1e-3f), 0);
            ncol = max(min((int)floorf(fmaxf(fu0, fu1) + 1e-3f), a.nu - 1) - u0 + 1, 0);
        }
        const int maxcol = wave_max_nn(ncol);
        const float dzs = Vv.z * a.dv, dzc = (float)((double)Cv.z - Sv.z), dz0 = fmaf(-cv, dzs, dzc);
        const float idzs = 1.0f / dzs;
        for (int cb = 0; cb < maxcol; cb += kSidCols) {
            int cnt = 0;
            float zl = 3.0e38f, zh = -3.0e38f, wmax = 0.0f;
            bool far = false;
            #pragma unroll
            for (int c = 0; c < kSidCols; ++c) {
                bool on = cb + c < ncol;
                SidEntry e{};
                if (on) {
                    const int iu = u0 + cb + c;
                    const double uc = (double)(iu - cu) * a.du;
                    const double wx = vcx - Sv.x, wy = vcy - Sv.y;
                    const double dxd = fma((double)Uv.x, uc, (double)Cv.x) - Sv.x;
                    const double dyd = fma((double)Uv.y, uc, (double)Cv.y) - Sv.y;
                    const float dx = (float)dxd, dy = (float)dyd;
                    // tp: the column's in-plane closest approach to the voxel
                    const float tp = (float)(wx * dxd + wy * dyd) * __builtin_amdgcn_rcpf(fmaf(dx, dx, dy * dy));
                    const float rx = (float)fma(-(double)tp, dxd, wx), ry = (float)fma(-(double)tp, dyd, wy);
                    float xy0 = -tp, xy1 = INFINITY, g0 = -INFINITY;      // from the source on
                    if (dx != 0.f) {
                        const float inv = __builtin_amdgcn_rcpf(dx);
                        const float a0 = (rx - hx) * inv, a1 = (rx + hx) * inv;
                        xy0 = fmaxf(xy0, fminf(a0, a1)); xy1 = fminf(xy1, fmaxf(a0, a1));
                        g0 = fmaxf(g0, fminf((glx - Sv.x) * inv, (ghx - Sv.x) * inv));
                    } else if (!(rx > -hx && rx <= hx)) {
                        xy1 = -INFINITY;
                    }
                    if (dy != 0.f) {
                        const float inv = __builtin_amdgcn_rcpf(dy);
                        const float a0 = (ry - hy) * inv, a1 = (ry + hy) * inv;
                        xy0 = fmaxf(xy0, fminf(a0, a1)); xy1 = fminf(xy1, fmaxf(a0, a1));
                        g0 = fmaxf(g0, fminf((gly - Sv.y) * inv, (ghy - Sv.y) * inv));
                    } else if (!(ry > -hy && ry <= hy)) {
                        xy1 = -INFINITY;
                    }
                    const float ta = tp + xy0, tb = tp + xy1;
                    on = xy1 > xy0 && ta > 0.0f;       // (ta > 0: the source lies off the grid, checked on the host)
                    if (on) {
                        e.xy0 = xy0; e.xy1 = xy1; e.tp = tp; e.Sz = Sv.z;
                        e.ia = idzs / ta; e.ib = idzs / tb; e.c = dz0 * idzs;
                        e.off = (unsigned)(((long)view * a.nu + iu) * nvp + kConePad) * 4u;
                        e.dzc = dzc; e.dzs = dzs; e.g0 = g0;
                        far = far || xy1 > 1.0f - tp;
                        // the voxels the rows' rays reach and the rows of one voxel
                        const float d1 = fmaf(dzs, fnv - 1.0f, dz0);
                        const float p = fminf(fminf(ta * dz0, tb * dz0), fminf(ta * d1, tb * d1));
                        const float q = fmaxf(fmaxf(ta * dz0, tb * dz0), fmaxf(ta * d1, tb * d1));
                        zl = fminf(zl, fmaf(Sv.z - g.cz + p, idz, 0.5f * g.nz));
                        zh = fmaxf(zh, fmaf(Sv.z - g.cz + q, idz, 0.5f * g.nz));
                        const float ds = fabsf(g.dz * e.ia);
                        wmax = fmaxf(wmax, fmaf(fmaf(fmaxf(fabsf(dz0), fabsf(d1)), fabsf(idzs), ds + 1.0f),
                                                (tb - ta) / ta, ds));
                    }
                }
                const unsigned long long gm = (__ballot(on) >> (grp * LZ)) & gmask;
                if (on) {
                    float4* d = list + 3 * (cnt + __popcll(gm & ((1ull << lg) - 1ull)));
                    d[0] = make_float4(e.xy0, e.xy1, e.tp, e.Sz);
                    d[1] = make_float4(e.ia, e.ib, e.c, __uint_as_float(e.off));
                    d[2] = make_float4(e.dzc, e.dzs, e.g0, 0.0f);
                }
                cnt += __popcll(gm);
            }
            const int n = wave_max_nn(cnt);
            // entries past the group's count: an empty interval on row 0 of the first column
            for (int i = cnt + lg; i < n; i += LZ) {
                list[3 * i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                list[3 * i + 1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                list[3 * i + 2] = make_float4(1.0f, 0.0f, 0.0f, 0.0f);
            }
            #pragma unroll
            for (int d = 1; d < LZ; d <<= 1) {
                zl = fminf(zl, __shfl_xor(zl, d));
                zh = fmaxf(zh, __shfl_xor(zh, d));
            }
            #pragma unroll
            for (int d = 1; d < 64; d <<= 1) wmax = fmaxf(wmax, __shfl_xor(wmax, d));
            wmax = wave_uniform(wmax) + 4e-3f;         // rows' rounding and the margin of the first row
            const bool anyfar = __any(far);
            const int zs = (int)__builtin_amdgcn_fmed3f(zl - 1.0f, fz0, fz1);
            const int ze = (int)__builtin_amdgcn_fmed3f(zh + 2.0f, fz0, fz1);
            const int passes = wave_max_nn(max((ze - zs + LZ - 1) / LZ, 0));
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            for (int m = 0; m < passes; ++m) {
                const int z = zs + m * LZ + lg;
                const double zc = g.cz + (z + 0.5 - g.nz / 2.0) * g.dz;
                const float ch = (float)zc, cl = (float)(zc - ch);
                float v;
                if (anyfar) v = sid_list_sum<0, true>(list, n, Qb, ch, cl, hz, cv, fnv, glz, ghz, ((int)wmax + 4) / 4);
                else if (wmax < 2.0f) v = sid_list_sum<2, false>(list, n, Qb, ch, cl, hz, cv, fnv, glz, ghz, 0);
                else if (wmax < 3.0f) v = sid_list_sum<3, false>(list, n, Qb, ch, cl, hz, cv, fnv, glz, ghz, 0);
                else if (wmax < 4.0f) v = sid_list_sum<4, false>(list, n, Qb, ch, cl, hz, cv, fnv, glz, ghz, 0);
                else v = sid_list_sum<0, false>(list, n, Qb, ch, cl, hz, cv, fnv, glz, ghz, ((int)wmax + 4) / 4);
                if (z < ze) acc[z - z0] += v;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    if (iy >= g.ny) return;
    const int cc = bc % nC, b = bc / nC;
    float* out = img + ((((long)b * g.nx + ix) * g.ny + iy) * g.nz) * nC + cc;
    for (int z = z0 + lg; z < z1; z += LZ) out[(long)z * nC] = acc[z - z0];
}

// ---- DD tomosynthesis ----

// average over [x1,x2] x [y1,y2] of a [ny][nx] plane (zero outside)
__device__ __forceinline__ float box_avg(const float* __restrict__ P, int nx, int ny, float x1, float x2, float y1,
                                         float y2)
{
    const float area = (x2 - x1) * (y2 - y1);
    const float lx = fmaxf(x1, 0.f), hx = fminf(x2, (float)nx);
    const float ly = fmaxf(y1, 0.f), hy = fminf(y2, (float)ny);
    if (!(hx > lx) || !(hy > ly)) return 0.f;
    const int m0 = (int)lx, m1 = min((int)hx, nx - 1), n0 = (int)ly, n1 = min((int)hy, ny - 1);
    float s = 0.f;
    for (int n = n0; n <= n1; ++n) {
        const float oy = fminf(hy, (float)(n + 1)) - fmaxf(ly, (float)n);
        if (oy <= 0.f) continue;
        float r = 0.f;
        for (int m = m0; m <= m1; ++m) {
            const float ox = fminf(hx, (float)(m + 1)) - fmaxf(lx, (float)m);
            r = fmaf(P[(long)n * nx + m], fmaxf(ox, 0.f), r);
        }
        s = fmaf(r, oy, s);
    }
    return s / area;
}

// vol_zyx: [slice][nz][ny][nx]
__global__ __launch_bounds__(128) void k_dd_tomo_fp(ArbGeo a, Grid3K g, const float* __restrict__ vol_zyx,
                                                    float* __restrict__ prj, const float* C, const float* S, int nC)
{
    const int iu = blockIdx.x * blockDim.x + threadIdx.x;
    const int view = blockIdx.y;
    const int bc = blockIdx.z;
    const int c = bc % nC, biv = bc / nC, iv = biv % a.nv, b = biv / a.nv;
    if (iu >= a.nu) return;
    const F3 cc = ld3(C, view), s0 = ld3(S, view);
    const float u = (iu - a.off_u - (a.nu - 1) / 2.0f) * a.du;
    const float v = (iv - a.off_v - (a.nv - 1) / 2.0f) * a.dv;
    auto tix = [&](float px) { return (px - g.cx) / g.dx + g.nx / 2.0f; };
    auto tiy = [&](float py) { return (py - g.cy) / g.dy + g.ny / 2.0f; };
    const float zc = (cc.z - g.cz) / g.dz + g.nz / 2.0f;
    const float sx = tix(s0.x), sy = tiy(s0.y), sz = (s0.z - g.cz) / g.dz + g.nz / 2.0f;
    float x1 = tix(cc.x + u - a.du / 2), x2 = tix(cc.x + u + a.du / 2);
    float y1 = tiy(cc.y + v - a.dv / 2), y2 = tiy(cc.y + v + a.dv / 2);
    if (x1 > x2) { const float t = x1; x1 = x2; x2 = t; }
    if (y1 > y2) { const float t = y1; y1 = y2; y2 = t; }
    const float dzs = zc - sz;
    const float rx1 = (x1 - sx) / dzs, rx2 = (x2 - sx) / dzs, ry1 = (y1 - sy) / dzs, ry2 = (y2 - sy) / dzs;
    const long plane = (long)g.nx * g.ny;
    const float* vol = vol_zyx + (long)(b * nC + c) * plane * g.nz;
    float val = 0.f;
    for (int iz = 0; iz < g.nz; ++iz) {
        const float h = (float)iz - sz;
        val += box_avg(vol + iz * plane, g.nx, g.ny, fmaf(rx1, h, sx), fmaf(rx2, h, sx), fmaf(ry1, h, sy),
                       fmaf(ry2, h, sy));
    }
    const float ddx = s0.x - (cc.x + u), ddy = s0.y - (cc.y + v), ddz = s0.z - cc.z;
    val *= g.dz / fabsf(ddz) * sqrtf(ddz * ddz + ddy * ddy + ddx * ddx);
    prj[((((long)b * a.nu + iu) * a.nview + view) * a.nv + iv) * nC + c] = val;
}

// wprj: [slice][nview][nv][nu] pre-weighted; out img reference layout
__global__ void k_dd_tomo_preweight(ArbGeo a, const float* __restrict__ prj_ref, float* __restrict__ w,
                                    const float* C, const float* S, int nC)
{
    const int iu = blockIdx.x * blockDim.x + threadIdx.x;
    const int view = blockIdx.y;
    const int bc = blockIdx.z;   // (b*nv + iv)*nC + c
    const int c = bc % nC, biv = bc / nC, iv = biv % a.nv, b = biv / a.nv;
    if (iu >= a.nu) return;
    const F3 cc = ld3(C, view), s0 = ld3(S, view);
    const float u = (iu - a.off_u - (a.nu - 1) / 2.0f) * a.du;
    const float v = (iv - a.off_v - (a.nv - 1) / 2.0f) * a.dv;
    const float ddx = s0.x - (cc.x + u), ddy = s0.y - (cc.y + v), ddz = s0.z - cc.z;
    // PreweightBPCartKernelXY (DistanceDriven3D.cu:429-430)
    const float wgt = a.dz / fabsf(ddz) * sqrtf(ddz * ddz + ddy * ddy + ddx * ddx);
    const float pv = prj_ref[((((long)b * a.nu + iu) * a.nview + view) * a.nv + iv) * nC + c];
    w[((((long)b * nC + c) * a.nview + view) * a.nv + iv) * a.nu + iu] = pv * wgt;
}

__global__ __launch_bounds__(256) void k_dd_tomo_bp(ArbGeo a, Grid3K g, const float* __restrict__ w,
                                                    float* __restrict__ img, const float* C, const float* S, int nC)
{
    const int iy = blockIdx.x * 16 + threadIdx.x;
    const int ix = blockIdx.y * 16 + threadIdx.y;
    const int bz = blockIdx.z;   // (b*nC + c)*nz + iz
    const int iz = bz % g.nz, bc = bz / g.nz, c = bc % nC, b = bc / nC;
    if (ix >= g.nx || iy >= g.ny) return;
    const float x = (ix - (g.nx - 1) / 2.0f) * g.dx + g.cx;
    const float y = (iy - (g.ny - 1) / 2.0f) * g.dy + g.cy;
    const float z = (iz - (g.nz - 1) / 2.0f) * g.dz + g.cz;
    const float cu = (a.nu - 1) / 2.0f + a.off_u, cv = (a.nv - 1) / 2.0f + a.off_v;
    const float* wb = w + (long)(b * nC + c) * a.nview * a.nv * a.nu;
    float val = 0.f;
    for (int view = 0; view < a.nview; ++view) {
        const F3 cc = ld3(C, view), s0 = ld3(S, view);
        // ProjectConeToDetCart (DistanceDriven3D.cu:478-489); its output is a bin-centre
        // index used directly as an integral-image coordinate (DistanceDriven3D.cu:544-553)
        const float r = (cc.z - s0.z) / (z - s0.z);
        float u1 = (s0.x - cc.x + r * (x - g.dx / 2 - s0.x)) / a.du + cu;
        float u2 = (s0.x - cc.x + r * (x + g.dx / 2 - s0.x)) / a.du + cu;
        float v1 = (s0.y - cc.y + r * (y - g.dy / 2 - s0.y)) / a.dv + cv;
        float v2 = (s0.y - cc.y + r * (y + g.dy / 2 - s0.y)) / a.dv + cv;
        if (u1 > u2) { const float t = u1; u1 = u2; u2 = t; }
        if (v1 > v2) { const float t = v1; v1 = v2; v2 = t; }
        val += box_avg(wb + (long)view * a.nv * a.nu, a.nu, a.nv, u1, u2, v1, v2);
    }
    img[((((long)b * g.nx + ix) * g.ny + iy) * g.nz + iz) * nC + c] = val;
}

// ---- circular cone-beam DD with a per-view main axis ----
//
// X views (|C.x - S.x| >= |C.y - S.y|, decided on the host) integrate over the
// planes x = voxel-centre x; Y views over y planes.  On plane p the footprint
// of detector cell (iu, iv) is [e1(p), e2(p)] x [z1(p), z2(p)] in index
// coordinates of the in-plane axis and of z: the plane crossings of the rays
// through the cell's u edges (at the cell's v centre) and through its v edges
// (at its u centre).  Each crossing is affine in the plane index, so a ray is
// described by four (alpha, beta) pairs and its per-plane length L.  The
// forward value is sum_p (rectangle average of plane p) * L; the adjoint
// gathers, per voxel, exactly those weights (overlap area / rectangle area * L).

// Tables of the cone DD pair, built in double on the host with the plan.
// ConeView: per view the constants of the plane-crossing geometry, resolved
// for the view's main axis m (x or y; n the other in-plane axis, p the plane
// index along m and j the voxel index along n).
struct alignas(16) ConeView {
    int xv;             // 1: main axis x
    float mp0, dm;      // plane p's main-axis offset from the source: mp0 + p dm
    float qn0, dn;      // n edge j relative to the source: qn0 + j dn
    float A, Cc, Um, Un;// detector centre minus source (n, m) and detU (m, n)
    float o;            // n index of the point on the plane at the source's n
    float a0;           // z index of the source
    float pad;
};
// ConeColumn: per (view, detector column) the ray constants that do not
// depend on the plane: the n index of the column's two u-edge rays on plane
// mp is mp k_e + o; the z index of row 0's lower edge on plane mp is
// mp A1 + a0; a row spans mp / T3 in z index; W the column weight dm /
// |main-axis run to the detector|, signed with the rows' z direction.
// Columns that cannot be hit (an edge ray parallel to the planes) hold
// k0 = k1 = 0 (an empty footprint) and W = 0.
struct alignas(32) ConeColumn { float k0, k1, A1, T3, W, pad[3]; };

// A group of LV lanes takes LV detector rows of one column; 64 / LV columns share
// a wave.  Per batch of LV planes each lane works out one plane's in-plane
// footprint [e1, e2] (the rows run along z, so it is the same for every row) and
// appends {offsets of cell rows j and j + 1, their shares / area, plane} to the
// group's list in LDS, one entry per pair of cells; then every lane walks the
// list with its own z footprint, z1 = a0 + mp (A1 + row / T3), |mp / T3| high:
// one LDS broadcast, two loads of 2 adjacent cells (3 where the footprint is
// over one voxel high) and 17 VALU instructions per entry.  A batch whose
// footprints leave the volume along z, or are over two voxels high, sums
// cell by cell within clamped bounds instead.
//
// Bound: instruction issue and the texture addresser alike: 3.5 ms at 256^2 x
// 128, 720 views, 64 x 512 (5.9 ms with the in-plane footprint worked out by every
// lane on every plane and four 4-byte loads).
//
// vol, prj: reference layouts [b][nx][ny][nz][c], [b][nu][nview][nv][c].  xcd: the
// 1-D grid (a multiple of 8) is renumbered so that each XCD walks a contiguous
// range of (column, row block, view): adjacent columns, whose footprints share
// cells, meet in one L2.  OFF32: byte offsets within one slice's volume below
// 4 GiB; C1: one channel (adjacent cells load as a pair).
template <int LV, bool OFF32, bool C1>
__global__ __launch_bounds__(256) void k_dd_cone_fp(ArbGeo a, Grid3K g, const float* __restrict__ vol,
                                                    float* __restrict__ prj, const float* Cp, const float* Up,
                                                    const float* Vp, const float* Sp,
                                                    const ConeView* __restrict__ views,
                                                    const ConeColumn* __restrict__ cols, int nC, int ncg, int nrb,
                                                    int nblocks, int xcd)
{
    typedef float F2 __attribute__((ext_vector_type(2), aligned(4)));
    constexpr int NG = 64 / LV;
    __shared__ float4 ents[4][64];
    __shared__ float emps[4][64];
    int l = blockIdx.x;
    if (xcd > 0) {
        l = (l % xcd) * ((int)gridDim.x / xcd) + l / xcd;
        if (l >= nblocks) return;
    }
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int grp = lane / LV, lg = lane % LV;
    const int iu0 = ((l % ncg) * 4 + wv) * NG;
    if (iu0 >= a.nu) return;                       // whole waves (no workgroup barrier below)
    const int rb = (l / ncg) % nrb, bz = l / (ncg * nrb);
    const int view = bz % a.nview, bc = bz / a.nview;
    const int cc = bc % nC, b = bc / nC;
    const int iu = iu0 + grp, iv = rb * LV + lg;
    const bool live = iu < a.nu && iv < a.nv;
    const float fiv = (float)min(iv, a.nv - 1);
    const ConeView vw = views[view];
    const ConeColumn col = cols[(long)view * a.nu + min(iu, a.nu - 1)];
    const int nm = vw.xv ? g.nx : g.ny, nn = vw.xv ? g.ny : g.nx;
    const char* base = reinterpret_cast<const char*>(vol + (long)b * g.nx * g.ny * g.nz * nC + cc);
    const float iT3 = col.T3 != 0.0f ? 1.0f / col.T3 : 0.0f, aT3 = fabsf(iT3);
    // z edges of this lane's row: a0 + mp sl0 and a0 + mp sl1
    const float sl0 = fmaf(fiv, iT3, col.A1), sl1 = fmaf(fiv + 1.0f, iT3, col.A1);
    const float fnz = (float)g.nz;
    const unsigned long long gmask = LV == 64 ? ~0ull : ((1ull << (LV & 63)) - 1ull);
    float4* ent = ents[wv] + grp * LV;
    float* emp = emps[wv] + grp * LV;
    // cell k of the row of cells along z that an entry's word names (a byte
    // offset, or the row's number where byte offsets do not fit 32 bits)
    auto cell = [&](float word, int k) -> const char* {
        const unsigned o = __float_as_uint(word);
        if (OFF32) return base + (unsigned)(o + (C1 ? (unsigned)k * 4u : __umul24((unsigned)k, (unsigned)nC * 4u)));
        return base + ((size_t)o * g.nz + k) * nC * 4;
    };
    auto ld = [](const char* p) { return *reinterpret_cast<const float*>(p); };
    float acc = 0.0f;
    for (int pb = 0; pb < nm; pb += LV) {
        const int p = pb + lg;
        const float mp = fmaf((float)p, vw.dm, vw.mp0);
        const float ea = fmaf(mp, col.k0, vw.o), eb = fmaf(mp, col.k1, vw.o);
        const float e1 = fminf(ea, eb), e2 = fmaxf(ea, eb);
        const float le = fmaxf(e1, 0.0f), he = fminf(e2, (float)nn);
        const float area = (e2 - e1) * fabsf(mp) * aT3;
        int j0 = 0, pairs = 0;
        if (p < nm && he > le && area > 0.0f && col.W != 0.0f) {
            j0 = (int)le;
            pairs = (min((int)he, nn - 1) - j0) / 2 + 1;
        }
        const float ia = __builtin_amdgcn_rcpf(area);
        const int rounds = wave_max_nn(pairs);
        // the batch's z footprints over all of the wave's rows: affine in mp
        const float mpA = fmaf((float)pb, vw.dm, vw.mp0), mpB = fmaf((float)(min(pb + LV, nm) - 1), vw.dm, vw.mp0);
        const float za = fmaf(mpA, sl0, vw.a0), zb = fmaf(mpB, sl0, vw.a0), zc = fmaf(mpA, sl1, vw.a0),
                    zd = fmaf(mpB, sl1, vw.a0);
        const float zlo = fminf(fminf(za, zb), fminf(zc, zd)), zhi = fmaxf(fmaxf(za, zb), fmaxf(zc, zd));
        const float hmax = fmaxf(fabsf(mpA), fabsf(mpB)) * aT3;
        const bool in = mpA * mpB > 0.0f && zlo >= 0.01f;
        const bool two = __all(in && zhi <= fnz - 1.01f && hmax <= 1.0f);
        const bool three = __all(in && zhi <= fnz - 2.01f && hmax <= 2.0f);
        const float sl = mpA * iT3 > 0.0f ? sl0 : sl1;       // the lower edge's
        for (int r = 0; r < rounds; ++r) {
            const bool on = r < pairs;
            const int j = j0 + 2 * r;
            const float fj = (float)j;
            const float oa = fminf(he, fj + 1.0f) - fmaxf(le, fj), ob = fmaxf(fminf(he, fj + 2.0f) - fmaxf(le, fj + 1.0f), 0.0f);
            const unsigned long long gm = (__ballot(on) >> (grp * LV)) & gmask;
            const int cnt = __popcll(gm), n = (wave_max_nn(cnt) + 3) & ~3;
            if (on) {
                const int pos = __popcll(gm & ((1ull << lg) - 1ull));
                const int k = ob > 0.0f ? j + 1 : j;
                const unsigned r1 = (unsigned)(vw.xv ? p * g.ny + j : j * g.ny + p);
                const unsigned r2 = (unsigned)(vw.xv ? p * g.ny + k : k * g.ny + p);
                const unsigned m = OFF32 ? (unsigned)g.nz * (unsigned)nC * 4u : 1u;
                ent[pos] = make_float4(__uint_as_float(r1 * m), __uint_as_float(r2 * m), oa * ia, ob * ia);
                emp[pos] = mp;
            }
            // entries past the group's count: a cell of the volume, on a plane of the
            // batch; their values (a NaN or an infinity among them) are dropped
            for (int i = cnt + lg; i < n; i += LV) {
                ent[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                emp[i] = mpA;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            // fours of entries that every group has, then the rest
            auto walk = [&](auto add) {
                int least = __builtin_amdgcn_readlane(cnt, 0), i = 0;
                #pragma unroll
                for (int k = 1; k < NG; ++k) least = min(least, __builtin_amdgcn_readlane(cnt, k * LV));
                for (; i + 4 <= least; i += 4) {
                    #pragma unroll
                    for (int k = 0; k < 4; ++k) acc = add(i + k, acc);
                }
                for (; i < n; i += 4) {
                    #pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float v = add(i + k, acc);
                        acc = i + k < cnt ? v : acc;
                    }
                }
            };
            if (two) {
                walk([&](int i, float s) {
                    const float4 e = ent[i];
                    const float m = emp[i];
                    const float z1 = fmaf(m, sl, vw.a0), fl = floorf(z1), h = fabsf(m) * aT3;
                    const float w1 = fmaxf((z1 - fl) + h - 1.0f, 0.0f), w0 = h - w1;
                    const char *pa = cell(e.x, (int)fl), *pb2 = cell(e.y, (int)fl);
                    float a0, a1, b0, b1;
                    if (C1) {
                        const F2 x = *reinterpret_cast<const F2*>(pa), y = *reinterpret_cast<const F2*>(pb2);
                        a0 = x[0]; a1 = x[1]; b0 = y[0]; b1 = y[1];
                    } else {
                        a0 = ld(pa); a1 = ld(pa + 4 * nC); b0 = ld(pb2); b1 = ld(pb2 + 4 * nC);
                    }
                    return fmaf(e.w, fmaf(b1, w1, b0 * w0), fmaf(e.z, fmaf(a1, w1, a0 * w0), s));
                });
            } else if (three) {
                walk([&](int i, float s) {
                    const float4 e = ent[i];
                    const float m = emp[i];
                    const float z1 = fmaf(m, sl, vw.a0), fl = floorf(z1), h = fabsf(m) * aT3;
                    const float t = (z1 - fl) + h;
                    const float w1 = __builtin_amdgcn_fmed3f(t - 1.0f, 0.0f, 1.0f), w2 = fmaxf(t - 2.0f, 0.0f);
                    const float w0 = (h - w1) - w2;
                    const char *pa = cell(e.x, (int)fl), *pb2 = cell(e.y, (int)fl);
                    const float sa = fmaf(ld(pa + 8 * nC), w2, fmaf(ld(pa + 4 * nC), w1, ld(pa) * w0));
                    const float sb = fmaf(ld(pb2 + 8 * nC), w2, fmaf(ld(pb2 + 4 * nC), w1, ld(pb2) * w0));
                    return fmaf(e.w, sb, fmaf(e.z, sa, s));
                });
            } else {
                for (int i = 0; i < n; ++i) {
                    if (i >= cnt) continue;
                    const float4 e = ent[i];
                    const float m = emp[i];
                    const float y0 = fmaf(m, sl0, vw.a0), y1 = fmaf(m, sl1, vw.a0);
                    const float lz = fmaxf(fminf(y0, y1), 0.0f), hz = fminf(fmaxf(y0, y1), fnz);
                    if (!(hz > lz)) continue;
                    const int k1 = min((int)hz, g.nz - 1);
                    float sa = 0.0f, sb = 0.0f;
                    for (int k = (int)lz; k <= k1; ++k) {
                        const float oz = fmaxf(fminf(hz, (float)(k + 1)) - fmaxf(lz, (float)k), 0.0f);
                        sa = fmaf(ld(cell(e.x, k)), oz, sa);
                        sb = fmaf(ld(cell(e.y, k)), oz, sb);
                    }
                    acc = fmaf(e.z, sa, acc);
                    if (e.w != 0.0f) acc = fmaf(e.w, sb, acc);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    if (!live) return;
    // path length per plane: dm / |main-axis run| times the ray's length to the cell
    const F3 c = ld3(Cp, view), U = ld3(Up, view), V = ld3(Vp, view), s = ld3(Sp, view);
    const float uc = (iu - a.off_u - (a.nu - 1) / 2.0f) * a.du, vc = (iv - a.off_v - (a.nv - 1) / 2.0f) * a.dv;
    const float lx = fmaf(vc, V.x, fmaf(uc, U.x, c.x)) - s.x, ly = fmaf(vc, V.y, fmaf(uc, U.y, c.y)) - s.y,
                lz = fmaf(vc, V.z, fmaf(uc, U.z, c.z)) - s.z;
    prj[((((long)b * a.nu + iu) * a.nview + view) * a.nv + iv) * nC + cc] =
        acc * fabsf(col.W) * sqrtf(fmaf(lx, lx, fmaf(ly, ly, lz * lz)));
}

// Row sums of the adjoint's second form: per (slice, view, detector column) the
// nv + 1 FP64 sums G[r] = sum over rows below r of len(row) q(row), len the
// length of the ray through the cell centre (the adjoint's row weight).
// Row sums: one wave per (slice, view, column), in table order; lanes take
// 64 rows at a time, an FP64 inclusive scan across the wave, then a carry.
__global__ __launch_bounds__(256) void k_dd_cone_rowsum(ArbGeo a, const float* __restrict__ prj, const float* Cp,
                                                        const float* Up, const float* Vp, const float* Sp, int nC,
                                                        long ncols, double* __restrict__ T)
{
    const long col = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (col >= ncols) return;
    const int lane = (int)(threadIdx.x & 63);
    const int iu = (int)(col % a.nu);
    const long rest = col / a.nu;
    const int view = (int)(rest % a.nview);
    const long bc = rest / a.nview;
    const int cc = (int)(bc % nC), b = (int)(bc / nC);
    const F3 c = ld3(Cp, view), U = ld3(Up, view), V = ld3(Vp, view), s = ld3(Sp, view);
    const float cu = (a.nu - 1) / 2.0f + a.off_u, cv = (a.nv - 1) / 2.0f + a.off_v;
    const float uc = ((float)iu - cu) * a.du;
    const float lx = fmaf(uc, U.x, c.x) - s.x, ly = fmaf(uc, U.y, c.y) - s.y;
    const float lxy2 = fmaf(lx, lx, ly * ly);
    const float zc0 = fmaf(uc, U.z, c.z) - s.z;
    const float lzs = V.z * a.dv, lz_0 = fmaf(-cv, lzs, zc0);
    const float* qcol = prj + (((long)b * a.nu + iu) * a.nview + view) * a.nv * nC + cc;
    double* G = T + col * (a.nv + 1);
    if (lane == 0) G[0] = 0.0;
    double carry = 0.0;
    for (int r0 = 0; r0 < a.nv; r0 += 64) {
        const int iv = r0 + lane;
        double f = 0.0;
        if (iv < a.nv) {
            const float lz = fmaf(lzs, (float)iv, lz_0);
            f = (double)(sqrtf(fmaf(lz, lz, lxy2)) * qcol[(long)iv * nC]);
        }
        #pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const double y = __shfl_up(f, d);
            if (lane >= d) f += y;
        }
        if (iv < a.nv) G[iv + 1] = carry + f;
        carry += __shfl(f, 63);
    }
}

// Exact transpose of k_dd_cone_fp: a voxel gathers, per view, the cells whose
// footprint on its plane overlaps it, with the forward pass's weight
// overlap / area * L.  The in-plane part (which detector columns meet the
// column (x, y) of voxels, with what share) does not depend on z, and along a
// detector column the rows' z edges on the plane are affine in z: the row
// coordinate of z index zi is s(zi) = zi ibdv + c, so a voxel takes the rows it
// covers, [s, s + |ibdv|], with weights clamp(s + |ibdv| - j, 0, 1) etc.
//
// A group of LZ lanes takes one (x, y); 64 / LZ of them share a wave.  Per batch
// of LZ views each lane works out one view's columns and appends {share, c,
// ibdv, row offset} to the group's list in LDS; then the group's lanes take LZ
// consecutive voxels of the z range the batch reaches and walk the list: one
// LDS broadcast, one load of 3 or 4 adjacent rows and 16 VALU instructions
// per entry and lane.  The sums over the batch go to the group's z column in
// LDS.
//
// Bound: VALU issue and the texture addresser alike (16-byte loads): 3.0 ms at
// 256^2 x 128, 720 views, 64 x 512, and 0.11 ms for the row windows.  Why this
// split: a cone detector's rows reach a quarter to a third of the z range, so
// 64 lanes along z with every lane's 2 voxels tested per view and column left
// 28 % of the lanes busy, the (x, y) geometry was repeated by every lane, and
// FP64 row sums cost 3 16-byte loads per 2 voxels (13.1 ms).  16 lanes per
// (x, y) cover that reach best (3.2 ms with 8, 4.4 with 32, 5.1 with 64).
constexpr int kConeZB = 256;        // z voxels of a workgroup's columns
constexpr int kConeCols = 4;        // list entries per view and round
constexpr float kConeMaxDs = 7.0f;  // rows per voxel beyond which the row-sum tables are used

// Sum over the list's n entries (a multiple of 4) for the voxel at z index fz.
// NR = 3 or 4: every entry's |ibdv| <= NR - 1; NR = 0: any, in chunks of 4 rows.
template <int NR>
__device__ __forceinline__ float cone_list_sum(const float4* list, int n, const char* __restrict__ Q, float fz,
                                               float lo, float hi, int chunks)
{
    float sum = 0.0f;
    for (int i = 0; i < n; i += 4) {
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float4 e = list[i + k];
            const float s = fmaf(fz, e.z, e.y), r0 = floorf(s);
            const float f = s - r0, t = f + fabsf(e.z);
            const unsigned off = __float_as_uint(e.w);
            if constexpr (NR > 0) {
                const int r = (int)__builtin_amdgcn_fmed3f(r0, lo, hi);
                float v[NR];
                cone_rows<NR>(Q, off + (unsigned)(r * 4), v);
                float d = (fminf(t, 1.0f) - f) * v[0];
                #pragma unroll
                for (int j = 1; j < NR; ++j) d = fmaf(__builtin_amdgcn_fmed3f(t - (float)j, 0.0f, 1.0f), v[j], d);
                sum = fmaf(e.x, d, sum);
            } else {
                float d = 0.0f;
                for (int c = 0; c < chunks; ++c) {
                    const int r = (int)__builtin_amdgcn_fmed3f(r0 + 4.0f * (float)c, lo, hi);
                    float v[4];
                    cone_rows<4>(Q, off + (unsigned)(r * 4), v);
                    #pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float q = (float)(4 * c + j);
                        const float w = __builtin_amdgcn_fmed3f(t - q, 0.0f, 1.0f);
                        d = fmaf(c + j == 0 ? w - f : w, v[j], d);
                    }
                }
                sum = fmaf(e.x, d, sum);
            }
        }
    }
    return sum;
}

// The same without the rows of weight 0: a NaN or an infinity there is not the voxel's.
__device__ __forceinline__ float cone_list_sum_met(const float4* list, int n, const char* __restrict__ Q, float fz,
                                                   float lo, float hi)
{
    float sum = 0.0f;
    #pragma unroll 1
    for (int i = 0; i < n; ++i) {
        const float4 e = list[i];
        const float s = fmaf(fz, e.z, e.y), r0 = floorf(s), f = s - r0, t = f + fabsf(e.z);
        float d = 0.0f;
        #pragma unroll 1
        for (float j = 0.0f; j < t; j += 1.0f) {
            const int r = (int)__builtin_amdgcn_fmed3f(r0 + j, lo, hi);
            const unsigned off = __float_as_uint(e.w) + (unsigned)(r * 4);   // (r may be negative: added in 32 bits)
            const float w = fminf(t - j, 1.0f) - (j == 0.0f ? f : 0.0f);
            d = fmaf(w, *reinterpret_cast<const float*>(Q + off), d);
        }
        sum = e.x != 0.0f ? fmaf(e.x, d, sum) : sum;
    }
    return sum;
}

template <int LZ>
__global__ __launch_bounds__(256, 4) void k_dd_cone_adj_list(ArbGeo a, Grid3K g, const float* __restrict__ Q,
                                                             float* __restrict__ img,
                                                             const ConeView* __restrict__ views,
                                                             const ConeColumn* __restrict__ cols, int nC)
{
    constexpr int NG = 64 / LZ;
    __shared__ float4 lists[4][64 * kConeCols];
    __shared__ float accs[4][NG * kConeZB];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int grp = lane / LZ, lg = lane % LZ;
    const int iy0 = ((int)blockIdx.y * 4 + wv) * NG;
    if (iy0 >= g.ny) return;                       // whole waves (no workgroup barrier below)
    const int iy = iy0 + grp, ix = blockIdx.z % g.nx, bc = blockIdx.z / g.nx;
    const int z0 = (int)blockIdx.x * kConeZB, z1 = min(z0 + kConeZB, g.nz);
    float4* list = lists[wv] + grp * (LZ * kConeCols);
    float* acc = accs[wv] + grp * kConeZB;
    for (int z = lg; z < kConeZB; z += LZ) acc[z] = 0.0f;
    const int nvp = a.nv + kConePad + 4;
    const char* Qb = reinterpret_cast<const char*>(Q + (long)bc * a.nview * a.nu * nvp);
    const float cu = (a.nu - 1) / 2.0f + a.off_u, idu = 1.0f / a.du;
    const float margin = 0.05f;
    const float fnv = (float)a.nv, lo = -(float)kConePad, fz0 = (float)z0, fz1 = (float)z1;
    const unsigned long long gmask = LZ == 64 ? ~0ull : ((1ull << (LZ & 63)) - 1ull);
    for (int vb = 0; vb < a.nview; vb += LZ) {
        const int view = min(vb + lg, a.nview - 1);
        const ConeView vw = views[view];
        const int p = vw.xv ? ix : iy, j = vw.xv ? iy : ix;
        const float mp = fmaf((float)p, vw.dm, vw.mp0);
        const float imp = __builtin_amdgcn_rcpf(mp);
        // u of the rays through the column's two in-plane edges
        float ulo = 3.0e38f, uhi = -3.0e38f;
        #pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float qe = fmaf((float)(j + e), vw.dn, vw.qn0) * imp;
            const float u = fmaf(-qe, vw.Cc, vw.A) * __builtin_amdgcn_rcpf(fmaf(qe, vw.Um, -vw.Un));
            ulo = fminf(ulo, u);
            uhi = fmaxf(uhi, u);
        }
        const float flo = fmaxf(ulo * idu + cu - 0.5f - margin, -1.0f);
        const float fhi = fminf(uhi * idu + cu + 0.5f + margin, (float)a.nu);
        int u0 = 0, ncol = 0;
        if (fhi >= flo && vb + lg < a.nview && iy < g.ny) {       // false for NaN
            u0 = max((int)ceilf(flo), 0);
            ncol = max(min((int)floorf(fhi), a.nu - 1) - u0 + 1, 0);
        }
        const int maxcol = wave_max_nn(ncol);
        for (int cb = 0; cb < maxcol; cb += kConeCols) {
            int cnt = 0;
            float zl = 3.0e38f, zh = -3.0e38f, dmax = 0.0f;
            #pragma unroll
            for (int c = 0; c < kConeCols; ++c) {
                bool on = cb + c < ncol;
                float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (on) {
                    const long ci = (long)view * a.nu + (u0 + cb + c);
                    const ConeColumn col = cols[ci];
                    // in-plane footprint of the column on plane p (index coordinates)
                    const float ea = fmaf(mp, col.k0, vw.o), eb = fmaf(mp, col.k1, vw.o);
                    const float e1 = fminf(ea, eb), e2 = fmaxf(ea, eb);
                    const float oe = fminf(e2, (float)(j + 1)) - fmaxf(e1, (float)j);
                    // row coordinate of z index zi: (zi - zA) / bdv = zi ibdv + s0
                    const float zA = fmaf(mp, col.A1, vw.a0), ibdv = imp * col.T3;
                    on = oe > 0.0f && e2 > e1 && fabsf(ibdv) <= kConeMaxDs && ibdv != 0.0f;
                    // share of the column times dm / |dpc|
                    e.x = oe * __builtin_amdgcn_rcpf(e2 - e1) * fabsf(col.W);
                    e.y = fminf(ibdv, 0.0f) - zA * ibdv;
                    e.z = ibdv;
                    e.w = __uint_as_float((unsigned)(ci * nvp + kConePad) * 4u);
                    const float zB = fmaf(fnv, __builtin_amdgcn_rcpf(ibdv), zA);
                    if (on) {
                        zl = fminf(zl, fminf(zA, zB));
                        zh = fmaxf(zh, fmaxf(zA, zB));
                        dmax = fmaxf(dmax, fabsf(ibdv));
                    }
                }
                const unsigned long long gm = (__ballot(on) >> (grp * LZ)) & gmask;
                if (on) list[cnt + __popcll(gm & ((1ull << lg) - 1ull))] = e;
                cnt += __popcll(gm);
            }
            const int n = (wave_max_nn(cnt) + 3) & ~3;
            for (int i = cnt + lg; i < n; i += LZ) list[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            // the voxels the batch reaches, the same for the group's lanes
            #pragma unroll
            for (int d = 1; d < LZ; d <<= 1) {
                zl = fminf(zl, __shfl_xor(zl, d));
                zh = fmaxf(zh, __shfl_xor(zh, d));
            }
            #pragma unroll
            for (int d = 1; d < 64; d <<= 1) dmax = fmaxf(dmax, __shfl_xor(dmax, d));
            dmax = wave_uniform(dmax);
            const int zs = (int)__builtin_amdgcn_fmed3f(zl - 1.0f, fz0, fz1);
            const int ze = (int)__builtin_amdgcn_fmed3f(zh + 2.0f, fz0, fz1);
            const int passes = wave_max_nn(max((ze - zs + LZ - 1) / LZ, 0));
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            for (int m = 0; m < passes; ++m) {
                const int z = zs + m * LZ + lg;
                const float fz = (float)z;
                float v;
                if (dmax <= 2.0f) v = cone_list_sum<3>(list, n, Qb, fz, lo, fnv, 0);
                else if (dmax <= 3.0f) v = cone_list_sum<4>(list, n, Qb, fz, lo, fnv, 0);
                else v = cone_list_sum<0>(list, n, Qb, fz, lo, fnv, ((int)dmax + 5) / 4);
                if (__any(z < ze && !(fabsf(v) < INFINITY))) {
                    const float u = cone_list_sum_met(list, n, Qb, fz, lo, fnv);
                    v = fabsf(v) < INFINITY ? v : u;
                }
                if (z < ze) acc[z - z0] += v;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    if (iy >= g.ny) return;
    const int cc = bc % nC, b = bc / nC;
    float* out = img + ((((long)b * g.nx + ix) * g.ny + iy) * g.nz) * nC + cc;
    for (int z = z0 + lg; z < z1; z += LZ) out[(long)z * nC] = acc[z - z0];
}

// The same from running row sums, for rows much finer than a voxel (and the
// launch-shape tuner's other candidates): the rows' z footprints on a column's
// plane tile z without gaps (row r covers [zA + r bdv, zA + (r + 1) bdv],
// bdv = beta dv), so the sum over rows of the z overlap times len q is bdv
// times the difference of the row sums, interpolated linearly within a row,
// at the voxel's two z edges.  ZPL + 1 lookups of one 16-byte pair
// (G[r], G[r + 1]) give ZPL voxels; the per-view and per-column geometry
// comes from the ConeView / ConeColumn tables (wave-uniform loads).  Same
// weights as the forward pass (the transpose holds to rounding).  A NaN or
// infinity in a row reaches every voxel above that row on the column's
// plane, not only the voxels the row overlaps.
template <int ZPL>
__global__ __launch_bounds__(256) void k_dd_cone_adj_tab(ArbGeo a, Grid3K g, const double* __restrict__ T,
                                                         float* __restrict__ img, const ConeView* __restrict__ views,
                                                         const ConeColumn* __restrict__ cols, int nC)
{
    const int iz = (blockIdx.x * 64 + (threadIdx.x & 63)) * ZPL;
    const int iy = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (int)(threadIdx.x >> 6));
    const int ix = blockIdx.z % g.nx, bc = blockIdx.z / g.nx;
    if (iz >= g.nz || iy >= g.ny) return;
    const int cc = bc % nC, b = bc / nC;
    const float cu = (a.nu - 1) / 2.0f + a.off_u;
    const float margin = 0.05f;
    const float fz = (float)iz, fnv = (float)a.nv;
    const float idu = 1.0f / a.du;
    const double* Tb = T + (long)bc * a.nview * a.nu * (a.nv + 1);
    float acc[ZPL];
    #pragma unroll
    for (int k = 0; k < ZPL; ++k) acc[k] = 0.f;
    for (int view = 0; view < a.nview; ++view) {
        const ConeView vw = views[view];
        const double* Tv = Tb + (long)view * a.nu * (a.nv + 1);
        const int p = vw.xv ? ix : iy, j = vw.xv ? iy : ix;
        const float mp = fmaf((float)p, vw.dm, vw.mp0);
        const float imp = __builtin_amdgcn_rcpf(mp);
        // u of the rays through the voxel's two in-plane edges
        float ulo = 3.0e38f, uhi = -3.0e38f;
        #pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float qe = fmaf((float)(j + e), vw.dn, vw.qn0) * imp;
            const float u = fmaf(-qe, vw.Cc, vw.A) * __builtin_amdgcn_rcpf(fmaf(qe, vw.Um, -vw.Un));
            ulo = fminf(ulo, u);
            uhi = fmaxf(uhi, u);
        }
        const float flo = fmaxf(ulo * idu + cu - 0.5f - margin, -1.0f);
        const float fhi = fminf(uhi * idu + cu + 0.5f + margin, (float)a.nu);
        if (!(fhi >= flo)) continue;                // also rejects NaN
        const int u0 = max((int)ceilf(flo), 0), u1 = min((int)floorf(fhi), a.nu - 1);
        const float smp = mp > 0.f ? 1.f : -1.f;
        for (int iu = u0; iu <= u1; ++iu) {
            const ConeColumn col = cols[(long)view * a.nu + iu];
            // in-plane footprint of the column on plane p (index coordinates)
            const float ea = fmaf(mp, col.k0, vw.o), eb = fmaf(mp, col.k1, vw.o);
            const float e1 = fminf(ea, eb), e2 = fmaxf(ea, eb);
            const float oe = fminf(e2, (float)(j + 1)) - fmaxf(e1, (float)j);
            if (!(oe > 0.f) || !(e2 > e1)) continue;
            // row coordinate of z index zi: s = (zi - zA) / bdv = zi ibdv + s0
            const float ibdv = imp * col.T3;
            if (!(fabsf(ibdv) < 1e20f)) continue;
            const float s0 = -fmaf(mp, col.A1, vw.a0) * ibdv;
            const float sb = fmaf(fz, ibdv, s0), st = fmaf(fz + (float)ZPL, ibdv, s0);
            if (!(fmaxf(sb, st) > 0.f && fminf(sb, st) < fnv)) continue;
            // oe / (e2 - e1) / |bdv| * dm / |dpc| times bdv
            const float wcol = oe * __builtin_amdgcn_rcpf(e2 - e1) * col.W * smp;
            // one 16-byte load per edge: G[r] and G[r + 1] (the address
            // processing of these loads bounds the kernel, so lanes whose
            // voxels miss the rows load nothing)
            const double* Gc = Tv + (long)iu * (a.nv + 1);
            double hp = 0.0;
            #pragma unroll
            for (int k = 0; k <= ZPL; ++k) {
                const float sk = __builtin_amdgcn_fmed3f(fmaf(fz + (float)k, ibdv, s0), 0.f, fnv);
                const unsigned r = min((unsigned)sk, (unsigned)(a.nv - 1));
                const double* gp = Gc + r;
                const double g0 = gp[0], g1 = gp[1];
                const double h = fma((double)(sk - (float)r), g1 - g0, g0);
                if (k > 0) acc[k - 1] = fmaf(wcol, (float)(h - hp), acc[k - 1]);
                hp = h;
            }
        }
    }
    float* out = img + ((((long)b * g.nx + ix) * g.ny + iy) * g.nz + iz) * nC + cc;
    #pragma unroll
    for (int k = 0; k < ZPL; ++k)
        if (iz + k < g.nz) out[(long)k * nC] = acc[k];
}

// ---- cone OS-SQS helpers ----

__global__ void k_cone_residual(const float* __restrict__ fp, const float* __restrict__ prj, float* __restrict__ r,
                                int nB, int nu, int nview, int cur, int start, int nvc)
{
    // fp, r: [b][nu][cur][nv*nC]; prj: [b][nu][nview][nv*nC]
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long per = (long)nu * cur * nvc;
    if (i >= per * nB) return;
    const long b = i / per, rem = i % per;
    const long iu = rem / ((long)cur * nvc), rem2 = rem % ((long)cur * nvc);
    const long vi = rem2 / nvc, k = rem2 % nvc;
    r[i] = fp[i] - prj[((b * nu + iu) * nview + start + vi) * nvc + k];
}

__global__ void k_cone_update(float* __restrict__ x, const float* __restrict__ bp, const float* __restrict__ D,
                              const float* __restrict__ mask, float step, float lb, float ub, int crop, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = (x[i] - step * (bp[i] / (D[i] + 1e-6f))) * mask[i];
    if (crop) v = v < lb ? lb : (v > ub ? ub : v);
    x[i] = v;
}

// ---- helical ----
//
// Weighted helical backprojection of parallel-cone data
// (bpHelicalParallelConebeam, Recon3D/HelicalBP.cu:10-83).  For a voxel at
// height z the views of one pi-window, i = iStart(z) .. iStart(z) + nviewPerPI - 1,
// each combine their conjugates k = i + m nviewPerPI (|m| <= mPI) as
// sum_m w_k P_k / (sum_m w_k + 1e-6), with P_k the bilinear sample at
//   u = x sin t_k - y cos t_k,
//   v = (z - zs_k(u)) dsd / (sqrt(dso^2 - u^2) - (x cos t_k + y sin t_k)),
//   zs_k(u) = zrot (k / (2 nviewPerPI) - asin(u / dso) / (2 pi)),
// and w_k the row taper of q = |2 v / (dv nv)|.
//
// Everything about a view except v is independent of z: a lane owns a
// column of ZC voxels (x, y fixed) and walks the union of their pi-windows;
// for each view it evaluates u, the magnification dsd / (...), zs_k and the column
// interpolation once, and then each of its voxels whose window contains the view
// costs a few instructions for v, the taper and a bilinear fetch.  The conjugates of
// a view lie half turns apart (up to the float PI of t_k, a rotation by a multiple of
// PI - pi): u and x cos t + y sin t change sign, the square root and the arc sine
// are worked out once.  A conjugate that no voxel of the wave sees inside the taper
// (q >= 1; at pitch 1 one of the three) is left before its loads.  The projections
// are copied with two zero rows before and after each view's, so that a row outside
// the detector needs no test.  A wave takes an 8 x 8 block of columns (its fetches
// land in one detector neighbourhood).  The sums run in the order above (i
// ascending, m ascending), the window start in the reference's float arithmetic.
//
// Bound: VALU.  256^2 x 128 voxels, three turns of 720 views, 64 x 512 detector: 6.4 ms
// (6.6 a call), 9.2 a call with the square root, arc sine and row tests per conjugate and
// every conjugate fetched.
// ---------------------------------------------------------------------------
// prj_k: [slice][nview][kHelPad + nv + kHelPad][nu]
constexpr int kHelPad = 2;
// per view k: (sin t_k, cos t_k, zk = zrot k / (2 nviewPerPI) as a float pair
// hi, lo), t_k = theta0 + k PI / nviewPerPI, in FP64
__global__ void k_helical_views(HelicalGeo h, float4* __restrict__ vt)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= h.nview) return;
    const double PI = (double)3.141592657f;
    const double t = (double)h.theta0 + k * PI / h.nviewPerPI;
    const double zk = (double)h.zrot * k / (2.0 * h.nviewPerPI);
    const float zhi = (float)zk;
    vt[k] = make_float4((float)sin(t), (float)cos(t), zhi, (float)(zk - zhi));
}

// asin by its Maclaurin series, sum_k C(2k, k) / (4^k (2k + 1)) x^(2k + 1),
// through x^15 for |x| <= 0.35 (truncation below 3e-10), asinf beyond
__device__ __forceinline__ float asin_series(float x)
{
    if (!(fabsf(x) <= 0.35f)) return asinf(x);
    const float x2 = x * x;
    float p = 1.396484375e-02f;
    p = fmaf(p, x2, 1.735276442e-02f);
    p = fmaf(p, x2, 2.237215909e-02f);
    p = fmaf(p, x2, 3.038194444e-02f);
    p = fmaf(p, x2, 4.464285714e-02f);
    p = fmaf(p, x2, 7.500000000e-02f);
    p = fmaf(p, x2, 1.666666667e-01f);
    p = fmaf(p, x2, 1.000000000e+00f);
    return x * p;
}

// two adjacent floats at a 4-byte-aligned address (one 8-byte load)
typedef float PairF __attribute__((ext_vector_type(2), aligned(4)));

template <int ZC>
__global__ __launch_bounds__(256) void k_helical_bp(HelicalGeo h, const float* __restrict__ prj,
                                                    const float4* __restrict__ vt, float* __restrict__ img, int nC,
                                                    int nzc)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int iy = blockIdx.x * 16 + (wv & 1) * 8 + (lane & 7);
    const int ix = blockIdx.y * 16 + (wv >> 1) * 8 + (lane >> 3);
    const int zb = blockIdx.z % nzc, bc = blockIdx.z / nzc;
    const int c = bc % nC, b = bc / nC;
    if (ix >= h.nx || iy >= h.ny) return;
    const float PI = 3.141592657f;                      // the reference's PI (Projector.h)
    const float x = (ix - (h.nx - 1) / 2.0f) * h.dx, y = (iy - (h.ny - 1) / 2.0f) * h.dy;
    const int z0 = zb * ZC;
    float zc[ZC];
    int is[ZC];
    int iLo = 0x7fffffff, iHi = -0x7fffffff;
    #pragma unroll
    for (int j = 0; j < ZC; ++j) {
        // the reference's float arithmetic, multiply-adds as FMAs (nvcc's
        // default contraction): the start is often an integer in exact
        // arithmetic, so its truncation follows these roundings
        zc[j] = fmaf((float)(z0 + j), h.dz, h.volZ0);
        is[j] = (int)(fmaf(zc[j] / h.zrot * 2.0f, PI, -PI / 4.0f) * (float)h.nviewPerPI / PI);
        if (z0 + j < h.nz) {
            iLo = min(iLo, is[j]);
            iHi = max(iHi, is[j] + h.nviewPerPI);
        }
    }
    // only views with a conjugate inside the data can contribute
    iLo = max(iLo, -h.mPI * h.nviewPerPI);
    iHi = min(iHi, h.nview + h.mPI * h.nviewPerPI);
    const long vpitch = (long)(h.nv + 2 * kHelPad) * h.nu;
    const float* pb = prj + (long)(b * nC + c) * h.nview * vpitch;
    const float zr2pi = h.zrot / (2 * PI);
    const float qs = 2.0f / h.nv;
    // (row and column coordinates; rows counted from the first pad row)
    const float cu = (h.nu - 1.0f) / 2.0f + h.off_u, cv = (h.nv - 1.0f) / 2.0f + h.off_v + (float)kHelPad;
    const float idso = 1.0f / h.dso, idu = 1.0f / h.du, dsdv = h.dsd / h.dv;
    const float rmax = (float)(h.nv + kHelPad);   // rows rmax, rmax + 1 are pads
    const float dpi = (float)((double)PI - 3.14159265358979323846);
    // the taper's phase in revolutions: cos((q - Q) / (1 - Q) pi / 2) = cos(2 pi r),
    // r = (q - Q) / (4 (1 - Q)), by the hardware cosine (taper weights enter as
    // sum w P / sum w; its error is far below the parity bound)
    const float tq = 0.25f / (1.0f - h.Q), qlive = fmaxf(1.0f, h.Q);
    float acc[ZC];
    #pragma unroll
    for (int j = 0; j < ZC; ++j) acc[j] = 0.0f;
    for (int i = iLo; i < iHi; ++i) {
        float val[ZC], tw[ZC];
        #pragma unroll
        for (int j = 0; j < ZC; ++j) val[j] = tw[j] = 0.0f;
        // the first conjugate inside the data: u, x cos t + y sin t, the square root and
        // zr2pi asin(u / dso)
        float ub = 0.0f, pbv = 0.0f, rt = 0.0f, as = 0.0f;
        int mb = 0x7fffffff;
        for (int m = -h.mPI; m <= h.mPI; ++m) {
            const int k = i + m * h.nviewPerPI;
            if (k < 0 || k >= h.nview) continue;
            const float4 tv = vt[k];                          // k is wave-uniform: scalar loads
            if (mb == 0x7fffffff) {
                mb = m;
                ub = x * tv.x - y * tv.y;
                pbv = x * tv.y + y * tv.x;
                rt = __builtin_amdgcn_sqrtf(h.dso * h.dso - ub * ub);
                as = zr2pi * asin_series(ub * idso);
            }
            const float dt = (float)(m - mb) * dpi, sg = ((m - mb) & 1) ? -1.0f : 1.0f;
            const float u = sg * fmaf(pbv, dt, ub);
            const float mag = dsdv * __builtin_amdgcn_rcpf(rt - sg * fmaf(-ub, dt, pbv));
            // source height zk - zr2pi asin(u / dso) as tv.z + zsl (tv.z exact in
            // float, so that z - tv.z loses nothing to the source's turn height)
            const float zsl = fmaf(-sg, as, tv.w);
            // v / dv, and which voxels see it inside the taper or on its bound (beyond the
            // source's circle u > dso: not numbers, as the sum then)
            float s[ZC];
            float qmin, qmax;
            #pragma unroll
            for (int j = 0; j < ZC; ++j) {
                s[j] = ((zc[j] - tv.z) - zsl) * mag;
                const float q = fabsf(s[j]) * qs;
                qmin = j == 0 ? q : fminf(qmin, q);
                qmax = j == 0 ? q : fmaxf(qmax, q);
            }
            if (!__any(!(qmin > qlive))) continue;
            const bool anytaper = __any(qmax > h.Q);
            const float pu = fmaf(u, idu, cu);
            const float fu = floorf(pu);
            const int u0 = (int)fu;
            const float au = pu - fu;
            const float wu0 = (u0 >= 0 && u0 < h.nu) ? 1.0f - au : 0.0f;
            const float wu1 = (u0 + 1 >= 0 && u0 + 1 < h.nu) ? au : 0.0f;
            // the two columns as one 8-byte load of the pair (ua, ua + 1),
            // ua = u0 clamped to [0, nu - 2]; the weights follow the columns
            // (u0 and u0 + 1 inside the pair where they fall in it)
            const int ua = min(max(u0, 0), h.nu - 2);
            const float wlo = (u0 == ua ? wu0 : 0.0f) + (u0 + 1 == ua ? wu1 : 0.0f);
            const float whi = (u0 == ua + 1 ? wu0 : 0.0f) + (u0 + 1 == ua + 1 ? wu1 : 0.0f);
            // the view's rows from wave-uniform bases and one 32-bit lane offset; every
            // voxel's two rows are loaded before any is used
            const float* pk = pb + (long)k * vpitch;
            const float* pn = pk + h.nu;
            float av[ZC], w[ZC];
            PairF r0[ZC], r1[ZC];
            #pragma unroll
            for (int j = 0; j < ZC; ++j) {
                const float pv = s[j] + cv, fv = floorf(pv);
                av[j] = pv - fv;
                const unsigned off = __umul24((unsigned)__builtin_amdgcn_fmed3f(fv, 0.0f, rmax), h.nu) + (unsigned)ua;
                r0[j] = *reinterpret_cast<const PairF*>(pk + off);
                r1[j] = *reinterpret_cast<const PairF*>(pn + off);
            }
            #pragma unroll
            for (int j = 0; j < ZC; ++j) w[j] = 1.0f;
            if (anytaper) {
                #pragma unroll
                for (int j = 0; j < ZC; ++j) {
                    const float q = fabsf(s[j]) * qs, c = __builtin_amdgcn_cosf((q - h.Q) * tq);
                    w[j] = q <= h.Q ? 1.0f : (q < 1.0f ? c * c : 0.0f);   // (Q = 1: no taper, c is not a number)
                }
            }
            #pragma unroll
            for (int j = 0; j < ZC; ++j) {
                const float a = fmaf(whi, r0[j].y, wlo * r0[j].x), d = fmaf(whi, r1[j].y, wlo * r1[j].x);
                // (a voxel outside its window: its sums are not used)
                val[j] = fmaf(fmaf(av[j], d, (1.0f - av[j]) * a), w[j], val[j]);
                tw[j] += w[j];
            }
        }
        #pragma unroll
        for (int j = 0; j < ZC; ++j)
            if (i >= is[j] && i < is[j] + h.nviewPerPI)
                acc[j] = fmaf(val[j], __builtin_amdgcn_rcpf(tw[j] + 1e-6f), acc[j]);   // 1-ulp reciprocal
    }
    #pragma unroll
    for (int j = 0; j < ZC; ++j)
        if (z0 + j < h.nz) img[((((long)b * h.nx + ix) * h.ny + iy) * h.nz + z0 + j) * nC + c] = acc[j];
}

// in [(b, c)][nu][nview nv] -> out [(b, c)][nview][kHelPad + nv + kHelPad][nu], pad rows zero
__global__ __launch_bounds__(256) void k_helical_rows(const float* __restrict__ in, float* __restrict__ out, int nu,
                                                      int nview, int nv)
{
    __shared__ float tile[32][33];
    const long rows = (long)nview * nv, bc = blockIdx.z;
    const long r0 = (long)blockIdx.x * 32;
    const int u0 = blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5, nr = nv + 2 * kHelPad;
    for (int j = ty; j < 32; j += 8)
        if (u0 + j < nu && r0 + tx < rows) tile[j][tx] = in[(bc * nu + u0 + j) * rows + r0 + tx];
    __syncthreads();
    const int u = u0 + tx;
    for (int j = ty; j < 32; j += 8) {
        const long r = r0 + j;
        if (r >= rows || u >= nu) continue;
        const int view = (int)(r / nv), v = (int)(r % nv);
        float* o = out + ((bc * nview + view) * nr + kHelPad) * (long)nu + u;
        o[(long)v * nu] = tile[tx][j];
        if (v == 0)
            for (int p = 1; p <= kHelPad; ++p) o[-(long)p * nu] = 0.0f;
        if (v == nv - 1)
            for (int p = 0; p < kHelPad; ++p) o[(long)(nv + p) * nu] = 0.0f;
    }
}

Grid3K grid_of(const ArbGeo& g) { return Grid3K{g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.cx, g.cy, g.cz}; }

} // namespace

bool arb_rows_along_z(const float* detU, const float* detV, int nview)
{
    if (!detU || !detV) return false;
    for (int v = 0; v < nview; v++)
        if (detV[3 * v] != 0.f || detV[3 * v + 1] != 0.f || detU[3 * v + 2] != 0.f) return false;
    return true;
}

void arb_rows(ArbGeo& g, const float* C, const float* U, const float* V, const float* S)
{
    g.rows_per_voxel = g.z_reach = 0.0f;
    if (!C || !S || !arb_rows_along_z(U, V, g.nview)) return;
    double most = 0.0, reach = 0.0;
    for (int v = 0; v < g.nview; v++) {
        const double dzs = std::fabs((double)V[3 * v + 2] * g.dv);
        // t of the grid's in-plane corners on the view's rays (1 on the detector): affine in (x, y)
        const double nx = U[3 * v + 1], ny = -(double)U[3 * v];
        const double A = (C[3 * v] - (double)S[3 * v]) * nx + (C[3 * v + 1] - (double)S[3 * v + 1]) * ny;
        double t = HUGE_VAL;
        for (int k = 0; k < 4; k++) {
            const double x = g.cx + ((k & 1) ? 0.5 : -0.5) * g.nx * g.dx, y = g.cy + ((k & 2) ? 0.5 : -0.5) * g.ny * g.dy;
            t = std::min(t, ((x - S[3 * v]) * nx + (y - S[3 * v + 1]) * ny) / A);
        }
        // the nearest voxel's rows: its height at t, plus what its in-plane
        // extent shifts the steepest row
        const double run = std::fabs(A) / std::sqrt(nx * nx + ny * ny);      // source to detector line
        const double dt = std::hypot((double)g.dx, (double)g.dy) / run;
        const double cz = std::fabs((double)C[3 * v + 2] - S[3 * v + 2]);
        const double steep = cz / dzs + 0.5 * g.nv + std::fabs((double)g.off_v) + 1.0;
        const double w = g.dz / (t * dzs) + steep * dt / t;
        if (!(t > 0.02) || !(w <= 1e6)) return;
        most = std::max(most, w);
        reach += ((g.cx - (double)S[3 * v]) * nx + (g.cy - (double)S[3 * v + 1]) * ny) / A * dzs * g.nv / g.dz;
    }
    g.rows_per_voxel = (float)most;
    g.z_reach = (float)(reach / g.nview);
}

void siddon_arb_fp(const ArbGeo& g, bool parallel, int nB, int nC, const float* img, float* prj,
                   const float* detCenter, const float* detU, const float* detV, const float* srcOrDir,
                   DevBuf& work, hipStream_t st)
{
    (void)work;
    RN_REQUIRE(detCenter && detU && detV && srcOrDir, "null geometry array");
    RN_REQUIRE((long)g.nview * nB * nC <= 65535 && cdiv(g.nu, 4) <= 65535, "siddon_arb_fp: grid too large");
    dim3 blk(256), grd(cdiv(g.nv, 64), cdiv(g.nu, 4), g.nview * nB * nC);
    // 32-bit voxel offsets when one slice's volume stays below 4 GiB
    auto k = (long)g.nx * g.ny * g.nz * nC * 4 < (1L << 32) ? k_siddon_arb_fp<true> : k_siddon_arb_fp<false>;
    hipLaunchKernelGGL(k, grd, blk, 0, st, g, grid_of(g), parallel ? 1 : 0, img, prj, detCenter, detU, detV, srcOrDir,
                       nC);
    check_launch("siddon_arb_fp");
}

void siddon_arb_bp(const ArbGeo& g, bool parallel, int nB, int nC, const float* prj, float* img,
                   const float* detCenter, const float* detU, const float* detV, const float* srcOrDir,
                   DevBuf& work, hipStream_t st)
{
    RN_REQUIRE(detCenter && detU && detV && srcOrDir, "null geometry array");
    RN_REQUIRE((long)g.nx * nB * nC <= 65535 && cdiv(g.ny, 4) <= 65535, "siddon_arb_bp: grid too large");
    work.ensure((size_t)g.nview * 4 * sizeof(float4));
    float4* vt = work.as<float4>();
    hipLaunchKernelGGL(k_siddon_arb_views, dim3(cdiv(g.nview, 256)), dim3(256), 0, st, g, grid_of(g),
                       parallel ? 1 : 0, detCenter, detU, detV, srcOrDir, vt);
    check_launch("siddon_arb_views");
    if (parallel || !g.rows_z) {
        dim3 grd(cdiv(g.nz, 64), cdiv(g.ny, 4), g.nx * nB * nC);
        hipLaunchKernelGGL((k_siddon_arb_bp<false, 1>), grd, dim3(256), 0, st, g, grid_of(g), parallel ? 1 : 0, prj, img,
                           detCenter, detU, detV, srcOrDir, vt, nC);
        check_launch("siddon_arb_bp");
        return;
    }
    // upright cone views: column lists with one (x, y) per 8, 16 or 32 lanes where
    // a voxel meets few rows (and the windows of one slice fit 4 GiB), else 1, 2
    // or 4 voxels per lane testing every view
    const int nvp = g.nv + kConePad + 4;
    const long n = (long)nB * nC * g.nu * g.nview * nvp;
    const bool lists = g.rows_per_voxel > 0 && g.rows_per_voxel <= kConeMaxDs &&
                       (long)g.nu * g.nview * nvp * 4L < (1L << 32) && (n + 255) / 256 < 0x7fffffffL;
    if (lists) {
        const size_t vt_bytes = (size_t)g.nview * 4 * sizeof(float4);
        if (work.size() < vt_bytes + (size_t)n * sizeof(float)) {
            // (the view table above was written to the buffer that is replaced)
            work.ensure(vt_bytes + (size_t)n * sizeof(float));
            vt = work.as<float4>();
            hipLaunchKernelGGL(k_siddon_arb_views, dim3(cdiv(g.nview, 256)), dim3(256), 0, st, g, grid_of(g), 0,
                               detCenter, detU, detV, srcOrDir, vt);
            check_launch("siddon_arb_views");
        }
        float* Q = reinterpret_cast<float*>(static_cast<char*>(work.get()) + vt_bytes);
        hipLaunchKernelGGL(k_cone_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, prj, detCenter, detU,
                           detV, srcOrDir, nC, n, Q);
        check_launch("cone_rows");
    }
    auto launch = [&](int c) {
        if (lists) {
            const float* Q = reinterpret_cast<const float*>(vt + (size_t)g.nview * 4);
            auto go = [&](auto kern, int lz) {
                const dim3 grd(cdiv(g.nz, kSidZB), cdiv(g.ny, 4 * (64 / lz)), g.nx * nB * nC);
                hipLaunchKernelGGL(kern, grd, dim3(256), 0, st, g, grid_of(g), Q, img, detCenter, detU, detV, srcOrDir,
                                   vt, nC);
            };
            if (c == 0) go(k_siddon_cone_bp_list<16>, 16);
            else if (c == 1) go(k_siddon_cone_bp_list<8>, 8);
            else go(k_siddon_cone_bp_list<32>, 32);
        } else {
            const int zpl = 1 << c;
            dim3 grd(cdiv(g.nz, 64 * zpl), cdiv(g.ny, 4), g.nx * nB * nC);
            auto k = c == 0 ? k_siddon_arb_bp<true, 1> : c == 1 ? k_siddon_arb_bp<true, 2> : k_siddon_arb_bp<true, 4>;
            hipLaunchKernelGGL(k, grd, dim3(256), 0, st, g, grid_of(g), 0, prj, img, detCenter, detU, detV, srcOrDir,
                               vt, nC);
        }
        check_launch("siddon_cone_bp");
    };
    // Lanes per (x, y) of the lists: a batch of that many views makes a partial sum, so
    // the geometry decides and not the tuner.  32, or 16 where the rows reach up to 15
    // voxels (8 up to 6) or just over 32 (beyond the centre, where the detector covers
    // part of the volume) and the (x, y) fill the chip.  ms with 8, 16
    // and 32: 190 x 177 x 99, reach 27 1.25, 0.93, 0.95; 207 x 205 x 28, reach 7.7 0.65,
    // 0.56, 0.87; 151^2 x 20, reach 5.5 0.49, 0.65, 1.03; 202^2 x 113, reach 31 0.94, 0.79,
    // 0.84; 60^2 x 95, reach 26 0.16, 0.090, 0.065; 128^2 x 64 all reached 1.40, 1.20, 1.06.
    const long waves = (long)g.nx * g.ny * nB * nC / 4;         // by 16 lanes
    const float reach = std::min(g.z_reach, (float)g.nz);
    const float over = g.z_reach < (float)g.nz ? 26.0f : 32.0f;
    int lz = 32;
    if (waves >= 1100 && (reach <= 15.0f || (waves >= 4096 && reach > over && reach <= 36.0f))) lz = 16;
    if (waves >= 4096 && reach <= (g.nz <= 8 ? 8.0f : 6.0f)) lz = 8;
    const uint32_t pick = !lists ? 7u : lz == 16 ? 1u : lz == 8 ? 2u : 4u;
    const TuneKey key{TK_SIDDON_CONE_BP, g.nx * g.ny, g.nz, g.nu * g.nv, g.nview, nB * nC, lists ? lz : 0};
    launch(tune_choose(key, 3, launch, st, true, pick));
}

void dd_tomo_fp(const ArbGeo& g, int nB, int nC, const float* img, float* prj,
                const float* detCenter, const float* src, DevBuf& work, hipStream_t st)
{
    RN_REQUIRE(detCenter && src, "null geometry array");
    const size_t nvol = (size_t)g.nx * g.ny * g.nz;
    const int ns = nB * nC;
    work.ensure(2 * ns * nvol * sizeof(float));
    float* t1 = work.as<float>();
    float* t2 = t1 + ns * nvol;
    // [b][x][y][z][c] -> [(b,c)][x][y][z] -> [(b,c)][z][x][y] -> [(b,c)][z][y][x]
    const float* base = img;
    if (nC > 1) {
        launch_transpose(img, t2, (int)nvol, nC, nB, st);
        base = t2;
    }
    launch_transpose(base, t1, g.nx * g.ny, g.nz, ns, st);
    launch_transpose(t1, t2, g.nx, g.ny, ns * g.nz, st);
    dim3 blk(128), grd(cdiv(g.nu, 128), g.nview, nB * g.nv * nC);
    hipLaunchKernelGGL(k_dd_tomo_fp, grd, blk, 0, st, g, grid_of(g), t2, prj, detCenter, src, nC);
    check_launch("dd_tomo_fp");
}

void dd_tomo_bp(const ArbGeo& g, int nB, int nC, const float* prj, float* img,
                const float* detCenter, const float* src, DevBuf& work, hipStream_t st)
{
    RN_REQUIRE(detCenter && src, "null geometry array");
    const size_t nprj = (size_t)nB * nC * g.nu * g.nview * g.nv;
    work.ensure(nprj * sizeof(float));
    dim3 b1(256), g1(cdiv(g.nu, 256), g.nview, nB * g.nv * nC);
    hipLaunchKernelGGL(k_dd_tomo_preweight, g1, b1, 0, st, g, prj, work.as<float>(), detCenter, src, nC);
    check_launch("dd_tomo_preweight");
    dim3 blk(16, 16), grd(cdiv(g.ny, 16), cdiv(g.nx, 16), nB * nC * g.nz);
    hipLaunchKernelGGL(k_dd_tomo_bp, grd, blk, 0, st, g, grid_of(g), work.as<float>(), img, detCenter, src, nC);
    check_launch("dd_tomo_bp");
}

void ConePlan::setup(const ArbGeo& g, const float* C, const float* U, const float* V, const float* S, hipStream_t st)
{
    RN_REQUIRE(g.nx > 0 && g.ny > 0 && g.nz > 0 && g.nu > 0 && g.nview > 0 && g.nv > 0, "cone dimensions must be positive");
    RN_REQUIRE(g.dx > 0 && g.dy > 0 && g.dz > 0 && g.du > 0 && g.dv > 0, "cone spacings must be positive");
    RN_REQUIRE(C && U && V && S, "null geometry array");
    const int n = g.nview;
    std::vector<float> h((size_t)12 * n);
    std::vector<int> cls(n);
    for (int v = 0; v < n; v++) {
        const float* u = U + 3 * v;
        const float* w = V + 3 * v;
        const float un = std::sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        const float wn = std::sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
        RN_REQUIRE(un > 0 && wn > 0, "detector axes must be non-zero");
        RN_REQUIRE(std::fabs(w[0]) <= 1e-6f * wn && std::fabs(w[1]) <= 1e-6f * wn,
                   "the cone DD projector needs detector columns parallel to z (detV = (0, 0, v))");
        RN_REQUIRE(std::fabs(u[2]) <= 1e-6f * un, "the cone DD projector needs detector rows normal to z (detU.z = 0)");
        cls[v] = std::fabs(C[3 * v] - S[3 * v]) >= std::fabs(C[3 * v + 1] - S[3 * v + 1]) ? 0 : 1;
    }
    std::copy(C, C + 3 * n, h.begin());
    std::copy(U, U + 3 * n, h.begin() + 3 * n);
    std::copy(V, V + 3 * n, h.begin() + 6 * n);
    std::copy(S, S + 3 * n, h.begin() + 9 * n);
    vec_.alloc(h.size() * sizeof(float));
    RN_HIP_CHECK(hipMemcpyAsync(vec_.get(), h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, st));
    // view and column tables of the DD adjoint, in double
    ds_max_ = 0.0;
    std::vector<ConeView> vt(n);
    std::vector<ConeColumn> ct((size_t)n * g.nu);
    const double cu = (g.nu - 1) / 2.0 + g.off_u, cv = (g.nv - 1) / 2.0 + g.off_v;
    for (int v = 0; v < n; v++) {
        const int xv = cls[v] == 0;
        const double Cm = C[3 * v + (xv ? 0 : 1)], Cn = C[3 * v + (xv ? 1 : 0)], Cz = C[3 * v + 2];
        const double Sm = S[3 * v + (xv ? 0 : 1)], Sn = S[3 * v + (xv ? 1 : 0)], Sz = S[3 * v + 2];
        const double Um = U[3 * v + (xv ? 0 : 1)], Un = U[3 * v + (xv ? 1 : 0)], Uz = U[3 * v + 2];
        const double Vz = V[3 * v + 2];
        const int nm = xv ? g.nx : g.ny, nn = xv ? g.ny : g.nx;
        const double dm = xv ? g.dx : g.dy, dn = xv ? g.dy : g.dx;
        const double gm = xv ? g.cx : g.cy, gn = xv ? g.cy : g.cx;
        ConeView& w = vt[v];
        w.xv = xv;
        w.mp0 = (float)((0.5 - 0.5 * nm) * dm + gm - Sm);
        w.dm = (float)dm;
        w.qn0 = (float)(gn - 0.5 * nn * dn - Sn);
        w.dn = (float)dn;
        w.A = (float)(Cn - Sn);
        w.Cc = (float)(Cm - Sm);
        w.Um = (float)Um;
        w.Un = (float)Un;
        w.o = (float)((Sn - gn) / dn + 0.5 * nn);
        w.a0 = (float)((Sz - g.cz) / g.dz + 0.5 * g.nz);
        w.pad = 0.f;
        for (int iu = 0; iu < g.nu; iu++) {
            ConeColumn& k = ct[(size_t)v * g.nu + iu];
            k = ConeColumn{0.f, 0.f, 0.f, 0.f, 0.f, {0.f, 0.f, 0.f}};
            const double uc = (iu - cu) * g.du;
            const double e0m = (uc - 0.5 * g.du) * Um + Cm - Sm, e0n = (uc - 0.5 * g.du) * Un + Cn - Sn;
            const double e1m = (uc + 0.5 * g.du) * Um + Cm - Sm, e1n = (uc + 0.5 * g.du) * Un + Cn - Sn;
            const double dpc = uc * Um + Cm - Sm;
            if (!(std::fabs(e0m) > 1e-6) || !(std::fabs(e1m) > 1e-6) || !(std::fabs(dpc) > 1e-6)) continue;
            const double zr0 = uc * Uz + Cz - Sz - (cv + 0.5) * g.dv * Vz;   // row 0's lower edge, from the source
            k.k0 = (float)(e0n / e0m / dn);
            k.k1 = (float)(e1n / e1m / dn);
            k.A1 = (float)(zr0 / dpc / g.dz);
            k.T3 = (float)(dpc * g.dz / (Vz * g.dv));
            k.W = (float)(dm / std::fabs(dpc) * (Vz / dpc > 0 ? 1.0 : -1.0));
        }
        // rows per voxel on the plane nearest to the source (unbounded if it lies
        // between the planes); the main-axis run to the detector is affine in the column
        const double m0 = w.mp0, m1 = w.mp0 + (nm - 1) * dm;
        const double t3 = std::max(std::fabs(-cu * g.du * Um + Cm - Sm), std::fabs((g.nu - 1 - cu) * g.du * Um + Cm - Sm)) *
                          g.dz / std::fabs(Vz * g.dv);
        ds_max_ = std::max(ds_max_, m0 * m1 > 0 ? t3 / std::min(std::fabs(m0), std::fabs(m1)) : HUGE_VAL);
    }
    views_.alloc(vt.size() * sizeof(ConeView));
    cols_.alloc(ct.size() * sizeof(ConeColumn));
    RN_HIP_CHECK(hipMemcpyAsync(views_.get(), vt.data(), vt.size() * sizeof(ConeView), hipMemcpyHostToDevice, st));
    RN_HIP_CHECK(hipMemcpyAsync(cols_.get(), ct.data(), ct.size() * sizeof(ConeColumn), hipMemcpyHostToDevice, st));
    RN_HIP_CHECK(hipStreamSynchronize(st));
    geo = g;
    geo.rows_z = arb_rows_along_z(U, V, n) ? 1 : 0;
    arb_rows(geo, C, U, V, S);
}

void ConePlan::dd_fp(int nB, int nC, const float* img, float* prj, hipStream_t st) const
{
    const ArbGeo& g = geo;
    RN_REQUIRE(nB > 0 && nC > 0 && (long)g.nview * nB * nC <= 65535, "cone batch too large for one launch");
    const float* v = vec_.as<float>();
    // byte offsets in 32 bits, channel strides by 24-bit multiplies
    const bool off32 = (long)g.nx * g.ny * g.nz * nC * 4 < (1L << 32) && g.nz < (1 << 24) && nC < (1 << 22);
    RN_REQUIRE((long)g.nx * g.ny < 0x7fffffffL, "dd_cone_fp: volume too large in plane");
    // rows per group of lanes: the split with the fewest idle lanes, wide first
    int lv = 64;
    for (int w : {32, 16})
        if (cdiv(g.nv, w) * w < cdiv(g.nv, lv) * lv) lv = w;
    const int ncg = cdiv(g.nu, 4 * (64 / lv)), nrb = cdiv(g.nv, lv);
    const long nblocks = (long)ncg * nrb * g.nview * nB * nC;
    RN_REQUIRE(nblocks + 8 < 0x7fffffffL, "dd_cone_fp: grid too large");
    auto launch = [&](int c) {
        const int xcd = c == 0 ? 8 : 0;
        const unsigned n = (unsigned)(c == 0 ? (nblocks + 7) / 8 * 8 : nblocks);
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(n), dim3(256), 0, st, g, grid_of(g), img, prj, v, v + 3 * g.nview,
                               v + 6 * g.nview, v + 9 * g.nview, views_.as<ConeView>(), cols_.as<ConeColumn>(), nC, ncg,
                               nrb, (int)nblocks, xcd);
        };
        auto pick = [&](auto k64, auto k32, auto k16) { lv == 64 ? go(k64) : lv == 32 ? go(k32) : go(k16); };
        if (!off32) pick(k_dd_cone_fp<64, false, false>, k_dd_cone_fp<32, false, false>, k_dd_cone_fp<16, false, false>);
        else if (nC == 1) pick(k_dd_cone_fp<64, true, true>, k_dd_cone_fp<32, true, true>, k_dd_cone_fp<16, true, true>);
        else pick(k_dd_cone_fp<64, true, false>, k_dd_cone_fp<32, true, false>, k_dd_cone_fp<16, true, false>);
        check_launch("dd_cone_fp");
    };
    const int c = tune_choose({TK_DD_CONE_FP, g.nx * g.ny, g.nz, g.nu * g.nv, g.nview, nB * nC}, 2, launch, st, true);
    launch(c);
}

void ConePlan::dd_adj(int nB, int nC, const float* prj, float* img, DevBuf& work, hipStream_t st) const
{
    const ArbGeo& g = geo;
    RN_REQUIRE(nB > 0 && nC > 0 && (long)g.nx * nB * nC <= 65535, "cone batch too large for one launch");
    const float* v = vec_.as<float>();
    const long ncols = (long)nB * nC * g.nu * g.nview;
    RN_REQUIRE((ncols + 3) / 4 < 0x7fffffffL, "dd_cone_adj: too many detector columns");
    // candidates 0-2: one (x, y) per 16, 8 or 32 lanes walking lists of columns
    // over row windows (up to kConeMaxDs rows per voxel: beyond, a voxel's rows
    // are better taken from two row sums; the windows of one slice in 4 GiB);
    // 3-5: 1, 2 or 4 voxels per lane from the row-sum table
    const int nvp = g.nv + kConePad + 4;
    // (the kernel's FP32 value of ds_max_, 4e-7 off at most, stays below kConeMaxDs too: it
    // drops columns beyond, and two chunks of 4 rows hold a voxel's)
    const bool windows = ds_max_ <= kConeMaxDs * (1.0 - 1e-5) && (long)g.nu * g.nview * nvp * 4L < (1L << 32);
    const int first = windows ? 0 : 3;
    auto launch = [&](int i) {
        const int c = first + i;
        if (c < 3) {
            work.ensure((size_t)ncols * nvp * sizeof(float));
            float* Q = work.as<float>();
            const long n = ncols * nvp;
            RN_REQUIRE((n + 255) / 256 < 0x7fffffffL, "dd_cone_adj: too many detector rows");
            hipLaunchKernelGGL(k_cone_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, prj, v,
                               v + 3 * g.nview, v + 6 * g.nview, v + 9 * g.nview, nC, n, Q);
            check_launch("cone_rows");
            auto go = [&](auto kern, int lz) {
                const dim3 grd(cdiv(g.nz, kConeZB), cdiv(g.ny, 4 * (64 / lz)), g.nx * nB * nC);
                hipLaunchKernelGGL(kern, grd, dim3(256), 0, st, g, grid_of(g), Q, img,
                                   views_.as<ConeView>(), cols_.as<ConeColumn>(), nC);
            };
            if (c == 0) go(k_dd_cone_adj_list<16>, 16);
            else if (c == 1) go(k_dd_cone_adj_list<8>, 8);
            else go(k_dd_cone_adj_list<32>, 32);
        } else {
            const int zpl = 1 << (c - 3);
            const dim3 grd(cdiv(g.nz, 64 * zpl), cdiv(g.ny, 4), g.nx * nB * nC);
            work.ensure((size_t)ncols * (g.nv + 1) * sizeof(double));
            double* T = work.as<double>();
            hipLaunchKernelGGL(k_dd_cone_rowsum, dim3((unsigned)cdiv(ncols, 4)), dim3(256), 0, st, g, prj, v,
                               v + 3 * g.nview, v + 6 * g.nview, v + 9 * g.nview, nC, ncols, T);
            check_launch("dd_cone_rowsum");
            auto k = c == 3 ? k_dd_cone_adj_tab<1> : c == 4 ? k_dd_cone_adj_tab<2> : k_dd_cone_adj_tab<4>;
            hipLaunchKernelGGL(k, grd, dim3(256), 0, st, g, grid_of(g), T, img, views_.as<ConeView>(),
                               cols_.as<ConeColumn>(), nC);
        }
        check_launch("dd_cone_adj");
    };
    // (the list is the geometry's, not the sizes')
    const TuneKey key{TK_DD_CONE_ADJ, g.nx * g.ny, g.nz, g.nu * g.nv, g.nview, nB * nC, windows ? 0 : 1};
    launch(tune_choose(key, 6 - first, launch, st, true));
}

void ConePlan::siddon_fp(int nB, int nC, const float* img, float* prj, DevBuf& work, hipStream_t st) const
{
    const float* v = vec_.as<float>();
    siddon_arb_fp(geo, false, nB, nC, img, prj, v, v + 3 * geo.nview, v + 6 * geo.nview, v + 9 * geo.nview, work, st);
}

void ConePlan::siddon_bp(int nB, int nC, const float* prj, float* img, DevBuf& work, hipStream_t st) const
{
    const float* v = vec_.as<float>();
    siddon_arb_bp(geo, false, nB, nC, prj, img, v, v + 3 * geo.nview, v + 6 * geo.nview, v + 9 * geo.nview, work, st);
}

void os_sqs_cone(const ArbGeo& g, int nB, int nC, float* x, const float* prj, const float* norm, const float* mask,
                 const float* detCenter, const float* detU, const float* detV, const float* src,
                 float lb, float ub, int nviewPerSubset, int nSubsets, float lambda, DevBuf& work, hipStream_t st)
{
    const size_t nimg = (size_t)nB * g.nx * g.ny * g.nz * nC;
    const int nvc = g.nv * nC;
    const size_t nsub = (size_t)nB * g.nu * nviewPerSubset * nvc;
    DevBuf fp(nsub * sizeof(float)), r(nsub * sizeof(float)), bp(nimg * sizeof(float));
    int start = 0;
    for (int k = 0; k < nSubsets && start < g.nview; k++) {
        const int cur = std::min(nviewPerSubset, g.nview - start);
        ArbGeo gs = g;
        gs.nview = cur;
        siddon_arb_fp(gs, false, nB, nC, x, fp.as<float>(), detCenter + 3 * start, detU + 3 * start,
                      detV + 3 * start, src + 3 * start, work, st);
        const long n = (long)nB * g.nu * cur * nvc;
        hipLaunchKernelGGL(k_cone_residual, dim3(cdiv(n, 256)), dim3(256), 0, st, fp.as<float>(), prj, r.as<float>(),
                           nB, g.nu, g.nview, cur, start, nvc);
        check_launch("cone_residual");
        siddon_arb_bp(gs, false, nB, nC, r.as<float>(), bp.as<float>(), detCenter + 3 * start, detU + 3 * start,
                      detV + 3 * start, src + 3 * start, work, st);
        hipLaunchKernelGGL(k_cone_update, dim3(cdiv((long)nimg, 256)), dim3(256), 0, st, x, bp.as<float>(), norm, mask,
                           lambda * nSubsets, lb, ub, lb < ub ? 1 : 0, nimg);
        check_launch("cone_update");
        start += cur;
    }
    RN_HIP_CHECK(hipStreamSynchronize(st));
}

// one lane per (row, channel) of a parallel ray: the rows of one (u, view)
// are contiguous in both layouts
// views per thread: the column's geometry (FP64, so that the interpolation
// weights carry no index rounding of the 2^12-view magnitudes) is set up once
constexpr int kRebinViews = 8;

__global__ __launch_bounds__(256) void k_helical_rebin(RebinGeo r, const float* __restrict__ fan,
                                                       float* __restrict__ par, int nC)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;      // iv * nC + c
    const int k0 = blockIdx.y * kRebinViews;
    const int lb = blockIdx.z;                                  // b * nu_p + l
    const int nq = r.nv_p * nC;
    if (q >= nq) return;
    const int l = lb % r.nu_p, b = lb / r.nu_p;
    const int iv = q / nC, c = q - iv * nC;
    const int kend = min(k0 + kRebinViews, r.nview_p);
    float* out = par + ((long)lb * r.nview_p) * nq + q;
    const double u = ((double)l - 0.5 * (r.nu_p - 1) - (double)r.off_u_p) * (double)r.du_p;
    const double sg = u / (double)r.dso;
    if (!(fabs(sg) < 1.0)) {
        for (int k = k0; k < kend; ++k) out[(long)k * nq] = 0.0f;
        return;
    }
    const double cg = sqrt(fma(-sg, sg, 1.0));
    // column s = dsd tan(g) and row height w = v / cos(g) on the flat detector
    const double fc = (double)r.dsd * sg / (cg * (double)r.du_f) + (double)r.off_u_f + 0.5 * (r.nu_f - 1);
    const double v = ((double)iv - 0.5 * (r.nv_p - 1) - (double)r.off_v_p) * (double)r.dv_p;
    const double fr = v / (cg * (double)r.dv_f) + (double)r.off_v_f + 0.5 * (r.nv_f - 1);
    const double gm = asin(sg) * r.idbeta;
    const double c0 = floor(fc), r0 = floor(fr);
    const float wc = (float)(fc - c0), wr = (float)(fr - r0);
    const bool in_cr = c0 > -2.0 && c0 < (double)r.nu_f && r0 > -2.0 && r0 < (double)r.nv_f;
    const int ic = in_cr ? (int)c0 : 0, ir = in_cr ? (int)r0 : 0;
    const float* base = fan + (long)b * r.nu_f * r.nview_f * r.nv_f * nC + c;
    for (int k = k0; k < kend; ++k) {
        const double fm = fma((double)k, r.kscale, r.moff) - gm;
        const double m0 = floor(fm);
        const float wm = (float)(fm - m0);
        float val = 0.0f;
        // the 8 corner samples; beyond the raw data's index range a sample is 0
        if (in_cr && m0 > -2.0 && m0 < (double)r.nview_f) {
            const int im = (int)m0;
            #pragma unroll
            for (int dc = 0; dc < 2; ++dc) {
                const int cc = ic + dc;
                if (cc < 0 || cc >= r.nu_f) continue;
                #pragma unroll
                for (int dm = 0; dm < 2; ++dm) {
                    const int mm = im + dm;
                    if (mm < 0 || mm >= r.nview_f) continue;
                    const float* row = base + ((long)cc * r.nview_f + mm) * r.nv_f * nC;
                    const float w2 = (dc ? wc : 1.0f - wc) * (dm ? wm : 1.0f - wm);
                    #pragma unroll
                    for (int dr = 0; dr < 2; ++dr) {
                        const int rr = ir + dr;
                        if (rr < 0 || rr >= r.nv_f) continue;
                        val = fmaf(row[(long)rr * nC], w2 * (dr ? wr : 1.0f - wr), val);
                    }
                }
            }
        }
        out[(long)k * nq] = val;
    }
}

void helical_rebin(const RebinGeo& r, int nB, int nC, const float* fan, float* par, hipStream_t st)
{
    RN_REQUIRE(nB > 0 && nC > 0, "nBatches and nChannels must be positive");
    RN_REQUIRE(r.nu_f > 0 && r.nview_f > 0 && r.nv_f > 0 && r.nu_p > 0 && r.nview_p > 0 && r.nv_p > 0,
               "rebinning dimensions must be positive");
    RN_REQUIRE(r.dso > 0 && r.dsd > 0 && r.du_f != 0 && r.dv_f != 0 && r.idbeta != 0 && std::isfinite(r.idbeta),
               "rebinning distances and spacings must be non-zero");
    RN_REQUIRE((long)nB * r.nu_p < 0x7fffffffL && r.nview_p < 65536, "rebinning grid too large");
    const dim3 grd(cdiv((long)r.nv_p * nC, 256), cdiv(r.nview_p, kRebinViews), nB * r.nu_p);
    hipLaunchKernelGGL(k_helical_rebin, grd, dim3(256), 0, st, r, fan, par, nC);
    check_launch("helical_rebin");
}

void helical_bp(const HelicalGeo& h, int nB, int nC, const float* prj, float* img, DevBuf& work, hipStream_t st)
{
    RN_REQUIRE(h.nu >= 2, "the helical backprojection needs at least 2 detector columns");
    RN_REQUIRE(h.nu < (1 << 24) && h.nv < (1 << 24) && (long)h.nu * h.nv < (1L << 31),
               "helical backprojection: detector too large");
    const size_t per = (size_t)h.nu * h.nview * h.nv, padded = (size_t)h.nu * h.nview * (h.nv + 2 * kHelPad);
    const size_t vt_off = ((size_t)nB * nC * (padded + per) + 3) / 4 * 4;   // 16-byte aligned view table
    work.ensure((vt_off + 4 * (size_t)h.nview) * sizeof(float));
    float* t1 = work.as<float>();
    float* t2 = t1 + (size_t)nB * nC * padded;
    float4* vt = reinterpret_cast<float4*>(t1 + vt_off);
    hipLaunchKernelGGL(k_helical_views, dim3(cdiv(h.nview, 256)), dim3(256), 0, st, h, vt);
    check_launch("helical_views");
    // [b][u][view][v][c] -> [(b, c)][u][view*v] -> [(b, c)][view][v][u]
    const float* base = prj;
    if (nC > 1) {
        // [b][u*view*v][c] -> [b][c][u*view*v]
        launch_transpose(prj, t2, (int)per, nC, nB, st);
        base = t2;
    }
    hipLaunchKernelGGL(k_helical_rows, dim3(cdiv((long)h.nview * h.nv, 32), cdiv(h.nu, 32), nB * nC), dim3(256), 0, st,
                       base, t1, h.nu, h.nview, h.nv);
    check_launch("helical_rows");
    // candidates: columns of 4, 8 or 2 voxels per lane
    auto launch = [&](int cand) {
        auto go = [&](auto kern, int zc) {
            const int nzc = cdiv(h.nz, zc);
            RN_REQUIRE((long)nB * nC * nzc <= 65535, "helical_bp: batch too large for one launch");
            const dim3 grd(cdiv(h.ny, 16), cdiv(h.nx, 16), nB * nC * nzc);
            hipLaunchKernelGGL(kern, grd, dim3(256), 0, st, h, t1, vt, img, nC, nzc);
        };
        if (cand == 0) go(k_helical_bp<4>, 4);
        else if (cand == 1) go(k_helical_bp<8>, 8);
        else go(k_helical_bp<2>, 2);
        check_launch("helical_bp");
    };
    const int c = tune_choose({TK_HELICAL_BP, h.nx * h.ny, h.nz, h.nu * h.nv, h.nview, nB * nC}, 3, launch, st, true);
    launch(c);
}

} // namespace rn
