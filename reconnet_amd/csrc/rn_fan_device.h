// Device helpers shared by the fan-beam kernels (line parameters of a ray,
// exact footprint averages and their transposes).
#pragma once

#include "rn_fan.h"

namespace rn {
namespace fan {

// Element at byte offset `boff` (32-bit) from a wave-uniform base: written so
// that the load is addressed as scalar base + 32-bit lane offset, with one
// offset computation shared by loads from several bases.  Callers keep every
// byte offset below 2^31 (checked on the host).
template <class T>
__device__ __forceinline__ T ld_at(const T* __restrict__ base, unsigned boff)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + boff);
}

// Values a lane carries: one slice (float, or double for the FP64
// normaliser) or four interleaved slices (float4, each component with the
// arithmetic of the float case).
template <class T>
__device__ __forceinline__ T vzero() { return T(0); }
template <>
__device__ __forceinline__ float4 vzero<float4>() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }
__device__ __forceinline__ void vadd(float& a, float b) { a += b; }
__device__ __forceinline__ void vadd(double& a, double b) { a += b; }
__device__ __forceinline__ void vadd(float4& a, float4 b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
// a += v * w (w converted to the value type first)
__device__ __forceinline__ void vmadd(float& a, float v, float w) { a += v * w; }
__device__ __forceinline__ void vmadd(double& a, double v, float w) { a += v * (double)w; }
__device__ __forceinline__ void vmadd(float4& a, float4 v, float w)
{
    a.x += v.x * w; a.y += v.y * w; a.z += v.z * w; a.w += v.w * w;
}
__device__ __forceinline__ float vscale(float v, float f) { return v * f; }
__device__ __forceinline__ double vscale(double v, float f) { return v * (double)f; }
__device__ __forceinline__ float4 vscale(float4 v, float f) { return make_float4(v.x * f, v.y * f, v.z * f, v.w * f); }

// ---------------------------------------------------------------------------
// geometry helpers
// ---------------------------------------------------------------------------

// acc[q] += scale * the average of row q (`rboff` bytes after the
// wave-uniform base rows[q]) over one interval [lo, hi] of its n
// piecewise-constant cells (zero outside [0, n)): the cells, their overlaps and the
// combined weight overlap * scale / width are computed once for the S rows,
// and each row adds one FMA per cell (a point interval, width 0, adds its
// cell times scale).
template <class T, int S>
__device__ __forceinline__ void seg_acc_rows(const T* const (&rows)[S], unsigned rboff, int n, float lo, float hi,
                                             float scale, T (&acc)[S])
{
    const float w = hi - lo;
    const float l = fmaxf(lo, 0.0f), h = fminf(hi, (float)n);
    if (!(h > l)) {
        if (w > 0.0f || !(lo >= 0.0f && lo < (float)n)) return;
        const unsigned boff = rboff + (unsigned)(int)lo * (unsigned)sizeof(T);
        #pragma unroll
        for (int q = 0; q < S; ++q) vmadd(acc[q], ld_at(rows[q], boff), scale);
        return;
    }
    const float k = scale / w;
    const int m0 = (int)l;
    const int m1 = min((int)h, n - 1);
    for (int m = m0; m <= m1; ++m) {
        const float pl = fmaxf(l, (float)m), ph = fminf(h, (float)(m + 1));
        const unsigned boff = rboff + (unsigned)m * (unsigned)sizeof(T);
        #pragma unroll
        for (int q = 0; q < S; ++q) vmadd(acc[q], ld_at(rows[q], boff), (ph - pl) * k);
    }
}

// Rows of CAP staged bins in LDS are CAP + 1 entries apart; the last one stays zero, and
// a lane without a bin reads it with weight 0 (a bin of the window would carry a NaN or
// an infinity to pixels that do not meet it).
constexpr int stage_pitch(int cap) { return cap + 1; }

// acc[q] += k * the integral over [lo, hi] (h0: the end of the row) of row q of G
// staged rows, their first entry the interval's origin; two bins without branches,
// further ones in a loop.
template <int G, int CAP>
__device__ __forceinline__ void seg_rel_staged(const float4* st, float lo, float hi, float h0, float k,
                                               float4 (&acc)[G])
{
    const float l = fmaxf(lo, 0.0f), h = fminf(hi, h0);
    const bool on0 = h > l;
    float f = floorf(l);
    int t = on0 ? (int)f : CAP;
    const float c0 = on0 ? (fminf(h, f + 1.0f) - l) * k : 0.0f;
    #pragma unroll
    for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * stage_pitch(CAP) + t], c0);
    f += 1.0f;
    const bool on1 = on0 && h > f;
    const float c1 = on1 ? (fminf(h, f + 1.0f) - f) * k : 0.0f;
    t = on1 ? t + 1 : CAP;
    #pragma unroll
    for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * stage_pitch(CAP) + t], c1);
    f += 1.0f;
    if (!on1) return;
    while (h > f) {
        ++t;
        const float c = (fminf(h, f + 1.0f) - f) * k;
        #pragma unroll
        for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * stage_pitch(CAP) + t], c);
        f += 1.0f;
    }
}

// ---------------------------------------------------------------------------
// per-ray forward projections and per-pixel gathers
// ---------------------------------------------------------------------------

// Sum over the cells of a line of n cells (zero outside [0, n)) of value times
// overlap with [lo, hi] (no division: the caller scales by L / |B|).
template <class T>
__device__ __forceinline__ T seg_sum(const T* __restrict__ line, int n, float lo, float hi)
{
    const float l = fmaxf(lo, 0.0f), h = fminf(hi, (float)n);
    T s = vzero<T>();
    if (!(h > l)) return s;
    const int m0 = (int)l;
    const int m1 = min((int)h, n - 1);
    for (int m = m0; m <= m1; ++m) {
        const float pl = fmaxf(l, (float)m), ph = fminf(h, (float)(m + 1));
        vmadd(s, line[m], ph - pl);
    }
    return s;
}

// seg_sum for hi - lo < 2 (at most three cells), without branches: the three
// loads are independent and every weight max(0, min(h, m+1) - max(l, m)) is
// zero for cells outside [l, h] (indices are clamped into the line).
// Siddon FP (exact ray / pixel intersection lengths), one line per image row
// (X views) or column (Y views): the ray crosses line j over [j, j+1] of the
// line axis, i.e. over [lo, hi] = [A + B (j - n/2), A + B (j + 1 - n/2)] of the
// cell axis, with path length L per line; the length inside a cell is L times
// the cell's share of [lo, hi], overlap / (hi - lo) with hi - lo taken from the
// same rounded end points (so a line's shares add up to one).  When the end
// points round to the same value (a ray along the line axis) the cell holding
// lo gets the whole length.
template <class T>
__device__ __forceinline__ T siddon_line_sum(const T* __restrict__ line, int n, float lo, float hi)
{
    const float w = hi - lo;
    if (w > 0.0f) return vscale(seg_sum<T>(line, n, lo, hi), __builtin_amdgcn_rcpf(w));
    return (lo >= 0.0f && lo < (float)n) ? line[(int)lo] : vzero<T>();
}

// A line of at most three cells for hi - lo < 2: the cells m0 .. m0 + 2 (indices
// clamped into the line) and their shares max(0, min(h, m + 1) - max(l, m))
// / (hi - lo), which vanish outside [l, h]; a zero-width interval gives the
// cell holding lo the whole share.  The cells and shares depend on the
// geometry only, so one Line3 serves every slice of a batch.
struct Line3 {
    unsigned i0, i1, i2;
    float w0, w1, w2;
};

__device__ __forceinline__ Line3 line3(int n, float lo, float hi)
{
    const float fn = (float)n;
    const float w = hi - lo;
    const float l = fminf(fmaxf(lo, 0.0f), fn), h = fminf(hi, fn);
    const int m0 = (int)l;                 // l in [m0, m0 + 1) unless l == n (then every weight is 0)
    const float f0 = (float)m0;
    const bool pos = w > 0.0f;
    const float inv = __builtin_amdgcn_rcpf(pos ? w : 1.0f);
    Line3 c;
    const float o0 = fmaxf(fminf(h, f0 + 1.0f) - l, 0.0f);
    c.w0 = (pos ? o0 : ((lo >= 0.0f && lo < fn) ? 1.0f : 0.0f)) * inv;
    c.w1 = fmaxf(fminf(h, f0 + 2.0f) - (f0 + 1.0f), 0.0f) * inv;
    c.w2 = fmaxf(fminf(h, f0 + 3.0f) - (f0 + 2.0f), 0.0f) * inv;
    const unsigned last = (unsigned)(n - 1);
    c.i0 = min((unsigned)m0, last);
    c.i1 = min((unsigned)m0 + 1u, last);
    c.i2 = min((unsigned)m0 + 2u, last);
    return c;
}

// acc += v0 w0 + v1 w1 [+ v2 w2] per value component (fused multiply-adds)
__device__ __forceinline__ void lmadd(float& a, float v0, float v1, float v2, const Line3& c, bool three)
{
    a = fmaf(v0, c.w0, a);
    a = fmaf(v1, c.w1, a);
    if (three) a = fmaf(v2, c.w2, a);
}
__device__ __forceinline__ void lmadd(double& a, double v0, double v1, double v2, const Line3& c, bool three)
{
    a = fma(v0, (double)c.w0, a);
    a = fma(v1, (double)c.w1, a);
    if (three) a = fma(v2, (double)c.w2, a);
}
__device__ __forceinline__ void lmadd(float4& a, float4 v0, float4 v1, float4 v2, const Line3& c, bool three)
{
    lmadd(a.x, v0.x, v1.x, v2.x, c, three);
    lmadd(a.y, v0.y, v1.y, v2.y, c, three);
    lmadd(a.z, v0.z, v1.z, v2.z, c, three);
    lmadd(a.w, v0.w, v1.w, v2.w, c, three);
}

// acc += the line starting `lboff` bytes after a wave-uniform base, over the
// first NC cells (NC = 2 when the interval is known to be narrower than one
// cell: the third share is then exactly 0 and its term is dropped)
template <class T, int NC>
__device__ __forceinline__ void line_madd_at(T& acc, const T* __restrict__ base, unsigned lboff, const Line3& c)
{
    const T v0 = ld_at(base, lboff + c.i0 * (unsigned)sizeof(T));
    const T v1 = ld_at(base, lboff + c.i1 * (unsigned)sizeof(T));
    const T v2 = NC == 2 ? v1 : ld_at(base, lboff + c.i2 * (unsigned)sizeof(T));
    lmadd(acc, v0, v1, v2, c, NC == 3);
}

// The narrow-ray line loop of siddon_fp_ray_slices: lines wj0 .. wj1 of the S
// slice bases; line j ends where line j + 1 starts (base + j + 1 is exact, so
// the shared end point is the same FMA result for both lines)
template <class T, int S, int NC>
__device__ __forceinline__ void fp_narrow_lines(const T* const (&Pq)[S], int n, float4 r, float base, int wj0,
                                                int wj1, T (&acc)[S])
{
    float ea = fmaf(r.y, base + (float)wj0, r.x);
    constexpr int kUnroll = S > 4 ? 1 : (S > 2 ? 2 : 4);
    #pragma unroll kUnroll
    for (int j = wj0; j <= wj1; ++j) {
        const float eb = fmaf(r.y, base + (float)(j + 1), r.x);
        const Line3 c = line3(n, fminf(ea, eb), fmaxf(ea, eb));
        const unsigned lboff = (unsigned)(j * n) * (unsigned)sizeof(T);
        #pragma unroll
        for (int q = 0; q < S; ++q) line_madd_at<T, NC>(acc[q], Pq[q], lboff, c);
        ea = eb;
    }
}

// Minimum and maximum of v over the 64 lanes of a wave (every lane active):
// pair, quad, half-row and row exchanges by DPP, then the four rows' values
// read into scalar registers, so the result is wave-uniform.  The exchanges'
// "old" operand is the operation's identity, so that each one compiles to a
// single min / max with a DPP source.
__device__ __forceinline__ int wave_min(int v)
{
    constexpr int id = 0x7fffffff;
    v = min(v, __builtin_amdgcn_update_dpp(id, v, 0xB1, 0xf, 0xf, false));    // quad_perm [1, 0, 3, 2]
    v = min(v, __builtin_amdgcn_update_dpp(id, v, 0x4E, 0xf, 0xf, false));    // quad_perm [2, 3, 0, 1]
    v = min(v, __builtin_amdgcn_update_dpp(id, v, 0x141, 0xf, 0xf, false));   // row_half_mirror
    v = min(v, __builtin_amdgcn_update_dpp(id, v, 0x140, 0xf, 0xf, false));   // row_mirror
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
__device__ __forceinline__ int wave_max(int v)
{
    constexpr int id = (int)0x80000000;
    v = max(v, __builtin_amdgcn_update_dpp(id, v, 0xB1, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(id, v, 0x4E, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(id, v, 0x141, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(id, v, 0x140, 0xf, 0xf, false));
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// One ray (bin iu of `view`) through S slices of one geometry: slice q reads
// planes Pyx + q * plane / Pxy + q * plane (slices q >= nsl read slice nsl - 1;
// the caller discards their sums).  Every lane of the wavefront calls it
// (inactive lanes with active = false and any valid iu).  The lines are walked
// over the union of the lanes' line ranges, so the loop and the line
// addresses are wave-uniform; lanes outside their own range add exact zeros.
// The cells met and their weights are computed once per line and applied to
// every slice, each slice with the arithmetic of a single-slice call.
template <class T, int S>
__device__ __forceinline__ void siddon_fp_ray_slices(const FanK& g, const T* __restrict__ Pyx,
                                                     const T* __restrict__ Pxy, long plane, int nsl, int view,
                                                     int iu, bool active, T (&acc)[S])
{
    const float4 r = g.sray[(long)view * g.nu + iu];
    const bool xv = g.vcls[view] == 0;
    const T* __restrict__ P = xv ? Pyx : Pxy;
    const int nl = xv ? g.ny : g.nx;     // lines
    const int n = xv ? g.nx : g.ny;      // cells per line
    const float base = -0.5f * (float)nl;
    // lines whose interval can meet [0, n]: A + B (j - nl/2) in [-|B| - 1, n + 1]
    // (one line of margin on each side; the other lines add exact zeros)
    int j0 = 0, j1 = nl - 1;
    if (r.y != 0.0f) {
        const float ib = 1.0f / r.y;
        const float ta = (-fabsf(r.y) - 1.0f - r.x) * ib - base, tb = ((float)n + 1.0f - r.x) * ib - base;
        const float tlo = fminf(fmaxf(fminf(ta, tb) - 1.0f, 0.0f), (float)nl);
        const float thi = fminf(fmaxf(ta, tb) + 1.0f, (float)(nl - 1));
        j0 = (int)tlo;
        j1 = thi >= tlo ? (int)thi : -1;
    } else if (!(r.x >= 0.0f && r.x < (float)n)) {
        j1 = -1;
    }
    if (!active) { j0 = nl; j1 = -1; }
    const int wj0 = wave_min(j0);
    const int wj1 = wave_max(j1);
    const T* Pq[S];                      // wave-uniform slice bases
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        Pq[q] = P + (long)min(q, nsl - 1) * plane;
        acc[q] = vzero<T>();
    }
    // [lo, hi] (rounded) spans at most three cells on every lane (two when
    // |B| < 1: the rounding error of the end points is far below 1e-3)
    const bool narrow = __all(!active || fabsf(r.y) <= 1.999f);
    if (narrow) {
        if (__all(!active || fabsf(r.y) <= 0.999f)) fp_narrow_lines<T, S, 2>(Pq, n, r, base, wj0, wj1, acc);
        else fp_narrow_lines<T, S, 3>(Pq, n, r, base, wj0, wj1, acc);
    } else {
        for (int j = wj0; j <= wj1; ++j) {
            const float lr = base + (float)j;
            const float ea = fmaf(r.y, lr, r.x), eb = fmaf(r.y, lr + 1.0f, r.x);
            #pragma unroll
            for (int q = 0; q < S; ++q)
                vadd(acc[q], siddon_line_sum<T>(Pq[q] + (long)j * n, n, fminf(ea, eb), fmaxf(ea, eb)));
        }
    }
    #pragma unroll
    for (int q = 0; q < S; ++q) acc[q] = vscale(acc[q], r.z);
}

// The padded-line variant of the narrow line loop for G interleaved slice
// groups (float4 cells; padded line j of group k starts at Pq[k] + j * pitch
// with kQPadL zero cells, so cell m is at + j * pitch + kQPadL + m, and ends
// with kQPadR zero cells; every offset from Pq[k] is non-negative).
// The crossing interval [lo, hi] of a line spans the cells m0 = floor(lo) ..
// m0 + NC - 1; the cell index is only clamped into the padded line, so an
// interval outside the image reads pad zeros, and the shares are
// (min(hi, m0 + 1) - lo, ..) / (hi - lo) without clamping to [0, n].  A
// zero-width interval gives cell m0 the whole share.
template <int G, int NC, bool WIDE>
__device__ __forceinline__ void fp_quad_lines_padded(const float4* const (&Pq)[G], int n, int pitch, float4 r,
                                                     float base, int wj0, int wj1, float4 (&acc)[G])
{
    float ea = fmaf(r.y, base + (float)wj0, r.x);
    float fj = base + (float)(wj0 + 1);
    #pragma unroll 2
    for (int j = wj0; j <= wj1; ++j) {
        const float eb = fmaf(r.y, fj, r.x);
        fj += 1.0f;
        const float lo = fminf(ea, eb), hi = fmaxf(ea, eb);
        const float w = hi - lo;
        const float f0 = floorf(lo);
        // clamped into the padded line: a clamped index only reads pad cells
        // (kQPadL, kQPadR >= NC), whatever the shares
        const int m0 = (int)__builtin_amdgcn_fmed3f(f0, -(float)kQPadL, (float)(n + kQPadR - NC));
        const bool pos = WIDE || w > 0.0f;   // WIDE: every interval of the view has w > 0
        const float inv = __builtin_amdgcn_rcpf(pos ? w : 1.0f);
        const float o0 = fminf(hi, f0 + 1.0f) - lo;
        float w0, w1, w2 = 0.0f;
        if (NC == 2) {
            w0 = (pos ? o0 : 1.0f) * inv;
            w1 = (w - o0) * inv;
        } else {
            const float o1 = fmaxf(fminf(hi, f0 + 2.0f) - (f0 + 1.0f), 0.0f);
            w0 = (pos ? o0 : 1.0f) * inv;
            w1 = o1 * inv;
            w2 = (w - o0 - o1) * inv;
        }
        const unsigned boff = (unsigned)(j * pitch + kQPadL + m0) * 16u;   // m0 >= -kQPadL
        #pragma unroll
        for (int k = 0; k < G; ++k) {
            const float4 v0 = ld_at(Pq[k], boff), v1 = ld_at(Pq[k], boff + 16u);
            float4& a = acc[k];
            a.x = fmaf(v0.x, w0, a.x); a.y = fmaf(v0.y, w0, a.y); a.z = fmaf(v0.z, w0, a.z); a.w = fmaf(v0.w, w0, a.w);
            a.x = fmaf(v1.x, w1, a.x); a.y = fmaf(v1.y, w1, a.y); a.z = fmaf(v1.z, w1, a.z); a.w = fmaf(v1.w, w1, a.w);
            if (NC == 3) {
                const float4 v2 = ld_at(Pq[k], boff + 32u);
                a.x = fmaf(v2.x, w2, a.x); a.y = fmaf(v2.y, w2, a.y);
                a.z = fmaf(v2.z, w2, a.z); a.w = fmaf(v2.w, w2, a.w);
            }
        }
        ea = eb;
    }
}

// One ray through G interleaved slice groups of padded quad images (Qyx for
// X views, Qxy for Y views; groups qstride cells apart, groups k >= nq read
// group nq - 1): the line range, wave-uniform loop and final scaling of
// siddon_fp_ray_slices with the padded line loop above (rays with |B| >= 2,
// none in ordinary geometries, take the clamped general path).  H = 2 or 4:
// the H parts of 64 / H lanes of the wave carry the same rays and walk
// consecutive parts of the wave's line range; their sums are added across the
// parts (every lane then holds the ray's total).
template <int G, int H = 1>
__device__ __forceinline__ void siddon_fp_ray_quads(const FanK& g, const float4* __restrict__ Qyx,
                                                    const float4* __restrict__ Qxy, int nq, int view, int iu,
                                                    bool active, float4 (&acc)[G])
{
    const float4 r = g.sray[(long)view * g.nu + iu];
    const bool xv = g.vcls[view] == 0;
    const float4* __restrict__ P = xv ? Qyx : Qxy;
    const int nl = xv ? g.ny : g.nx;     // lines
    const int n = xv ? g.nx : g.ny;      // cells per line
    const int pitch = qpitch(n);
    const long qstride = (long)nl * pitch;
    const float base = -0.5f * (float)nl;
    int j0 = 0, j1 = nl - 1;
    if (r.y != 0.0f) {
        const float ib = 1.0f / r.y;
        const float ta = (-fabsf(r.y) - 1.0f - r.x) * ib - base, tb = ((float)n + 1.0f - r.x) * ib - base;
        const float tlo = fminf(fmaxf(fminf(ta, tb) - 1.0f, 0.0f), (float)nl);
        const float thi = fminf(fmaxf(ta, tb) + 1.0f, (float)(nl - 1));
        j0 = (int)tlo;
        j1 = thi >= tlo ? (int)thi : -1;
    } else if (!(r.x >= 0.0f && r.x < (float)n)) {
        j1 = -1;
    }
    if (!active) { j0 = nl; j1 = -1; }
    int wj0 = wave_min(j0);
    int wj1 = wave_max(j1);
    static_assert(H == 1 || H == 2 || H == 4, "parts of a wave");
    const int len = wj1 - wj0 + 1;
    if (H > 1 && len > 0) {
        const int part = (int)(threadIdx.x & 63) / (64 / H);
        const int a = wj0 + len * part / H, b = wj0 + len * (part + 1) / H - 1;
        wj0 = a;
        wj1 = b;
    }
    const float4* Pq[G];                 // wave-uniform group bases at the start of padded line 0
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        Pq[k] = P + (long)min(k, nq - 1) * qstride;
        acc[k] = vzero<float4>();
    }
    if (__all(!active || fabsf(r.y) <= 0.999f)) {
        if (g.vwide[view]) fp_quad_lines_padded<G, 2, true>(Pq, n, pitch, r, base, wj0, wj1, acc);
        else fp_quad_lines_padded<G, 2, false>(Pq, n, pitch, r, base, wj0, wj1, acc);
    } else if (__all(!active || fabsf(r.y) <= 1.999f)) {
        fp_quad_lines_padded<G, 3, false>(Pq, n, pitch, r, base, wj0, wj1, acc);
    } else {
        for (int j = wj0; j <= wj1; ++j) {
            const float lr = base + (float)j;
            const float ea = fmaf(r.y, lr, r.x), eb = fmaf(r.y, lr + 1.0f, r.x);
            #pragma unroll
            for (int k = 0; k < G; ++k)
                vadd(acc[k], siddon_line_sum<float4>(Pq[k] + (long)j * pitch + kQPadL, n, fminf(ea, eb),
                                                     fmaxf(ea, eb)));
        }
    }
    #pragma unroll
    for (int o = 32; o >= 64 / H; o >>= 1) {
        #pragma unroll
        for (int k = 0; k < G; ++k) {
            acc[k].x += __shfl_xor(acc[k].x, o);
            acc[k].y += __shfl_xor(acc[k].y, o);
            acc[k].z += __shfl_xor(acc[k].z, o);
            acc[k].w += __shfl_xor(acc[k].w, o);
        }
    }
    #pragma unroll
    for (int k = 0; k < G; ++k) acc[k] = vscale(acc[k], r.z);
}

// ---- distance-driven forward projection on the line machinery ----
//
// DDFPFanKernelX/Y (DistanceDriven.cu:64-196): on line l (image row iy for X
// views, column ix for Y views; line coordinate lr = l - nl/2) the footprint
// of bin iu lies between its two edge rays, [e0, e1] with e_k = A_k + B_k lr
// (the FP64 table g.dray), and the ray's value adds the average of the
// line's row-averaged plane over that footprint; the sum is scaled by the
// path length per line L = dy/|cos(a - t)| (X) or dx/|sin(a - t)| (Y), the
// Siddon table's L.  The footprint average is the share arithmetic of the
// Siddon line intervals (overlap / width, the width unclipped), so the same
// branch-free two- or three-cell line code serves both projectors.

// Lines whose footprint can meet [0, n]: the union over the two edges of the
// lines where the edge lies in [-2, n + 2] (one line of margin on each side;
// the other lines add exact zeros while the footprint is narrower than 2).
__device__ __forceinline__ void dd_edge_lines(float A, float B, int n, int nl, float base, int& j0, int& j1)
{
    j0 = 0;
    j1 = nl - 1;
    if (B != 0.0f) {
        const float ib = 1.0f / B;
        const float ta = (-2.0f - A) * ib - base, tb = ((float)n + 2.0f - A) * ib - base;
        const float tlo = fminf(fmaxf(fminf(ta, tb) - 1.0f, 0.0f), (float)nl);
        const float thi = fminf(fmaxf(ta, tb) + 1.0f, (float)(nl - 1));
        j0 = (int)tlo;
        j1 = thi >= tlo ? (int)thi : -1;
    } else if (!(A >= -2.0f && A <= (float)n + 2.0f)) {
        j0 = nl;
        j1 = -1;
    }
}

// Line range of bin ray d = (A0, B0, A1, B1) and the largest footprint width
// over it (0 if the range is empty).
__device__ __forceinline__ void dd_ray_lines(float4 d, int n, int nl, float base, int& j0, int& j1, float& wmax)
{
    int a0, a1, b0, b1;
    dd_edge_lines(d.x, d.y, n, nl, base, a0, a1);
    dd_edge_lines(d.z, d.w, n, nl, base, b0, b1);
    j0 = min(a0, b0);
    j1 = max(a1, b1);
    wmax = 0.0f;
    if (j1 >= j0) {
        const float dA = d.z - d.x, dB = d.w - d.y;
        wmax = fmaxf(fabsf(fmaf(dB, base + (float)j0, dA)), fabsf(fmaf(dB, base + (float)j1, dA)));
    }
}

// Plain planes: lines wj0 .. wj1 of S slices, footprints at most NC cells wide
template <class T, int S, int NC>
__device__ __forceinline__ void dd_narrow_lines(const T* const (&Pq)[S], int n, float4 d, float base, int wj0,
                                                int wj1, T (&acc)[S])
{
    constexpr int kUnroll = S > 4 ? 1 : (S > 2 ? 2 : 4);
    #pragma unroll kUnroll
    for (int j = wj0; j <= wj1; ++j) {
        const float lr = base + (float)j;
        const float ea = fmaf(d.y, lr, d.x), eb = fmaf(d.w, lr, d.z);
        const Line3 c = line3(n, fminf(ea, eb), fmaxf(ea, eb));
        const unsigned lboff = (unsigned)(j * n) * (unsigned)sizeof(T);
        #pragma unroll
        for (int q = 0; q < S; ++q) line_madd_at<T, NC>(acc[q], Pq[q], lboff, c);
    }
}

// One bin of one view through S consecutive slices of the row-averaged planes
// RX [s][ny][nx] (X views) and RY [s][nx][ny] (Y views); slices q >= nsl read
// slice nsl - 1.  Wave-uniform line loop as in siddon_fp_ray_slices.
template <class T, int S>
__device__ __forceinline__ void dd_fp_ray_slices(const FanK& g, const T* __restrict__ RX, const T* __restrict__ RY,
                                                 long plane, int nsl, int view, int iu, bool active, T (&acc)[S])
{
    const float4 d = g.dray[(long)view * g.nu + iu];
    const float L = g.sray[(long)view * g.nu + iu].z;
    const bool xv = g.vcls[view] == 0;
    const T* __restrict__ P = xv ? RX : RY;
    const int nl = xv ? g.ny : g.nx;
    const int n = xv ? g.nx : g.ny;
    const float base = -0.5f * (float)nl;
    int j0, j1;
    float wmax;
    dd_ray_lines(d, n, nl, base, j0, j1, wmax);
    if (!active) { j0 = nl; j1 = -1; wmax = 0.0f; }
    const int wj0 = wave_min(j0);
    const int wj1 = wave_max(j1);
    const T* Pq[S];
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        Pq[q] = P + (long)min(q, nsl - 1) * plane;
        acc[q] = vzero<T>();
    }
    if (__all(wmax <= 0.999f)) {
        dd_narrow_lines<T, S, 2>(Pq, n, d, base, wj0, wj1, acc);
    } else if (__all(wmax <= 1.999f)) {
        dd_narrow_lines<T, S, 3>(Pq, n, d, base, wj0, wj1, acc);
    } else {
        for (int j = wj0; j <= wj1; ++j) {
            const float lr = base + (float)j;
            const float ea = fmaf(d.y, lr, d.x), eb = fmaf(d.w, lr, d.z);
            #pragma unroll
            for (int q = 0; q < S; ++q)
                vadd(acc[q], vscale(seg_sum<T>(Pq[q] + (long)j * n, n, fminf(ea, eb), fmaxf(ea, eb)),
                                    1.0f / fabsf(eb - ea)));
        }
    }
    #pragma unroll
    for (int q = 0; q < S; ++q) acc[q] = vscale(acc[q], L);
}

// Padded quad planes (see fp_quad_lines_padded): G groups, footprints at most
// NC cells wide
template <int G, int NC>
__device__ __forceinline__ void dd_quad_lines_padded(const float4* const (&Pq)[G], int n, int pitch, float4 d,
                                                     float base, int wj0, int wj1, float4 (&acc)[G])
{
    #pragma unroll 2
    for (int j = wj0; j <= wj1; ++j) {
        const float lr = base + (float)j;
        const float ea = fmaf(d.y, lr, d.x), eb = fmaf(d.w, lr, d.z);
        const float lo = fminf(ea, eb), hi = fmaxf(ea, eb);
        const float w = hi - lo;
        const float f0 = floorf(lo);
        const int m0 = (int)__builtin_amdgcn_fmed3f(f0, -(float)kQPadL, (float)(n + kQPadR - NC));
        const bool pos = w > 0.0f;
        const float inv = __builtin_amdgcn_rcpf(pos ? w : 1.0f);
        const float o0 = fminf(hi, f0 + 1.0f) - lo;
        float w0, w1, w2 = 0.0f;
        if (NC == 2) {
            w0 = (pos ? o0 : 1.0f) * inv;
            w1 = (w - o0) * inv;
        } else {
            const float o1 = fmaxf(fminf(hi, f0 + 2.0f) - (f0 + 1.0f), 0.0f);
            w0 = (pos ? o0 : 1.0f) * inv;
            w1 = o1 * inv;
            w2 = (w - o0 - o1) * inv;
        }
        const unsigned boff = (unsigned)(j * pitch + kQPadL + m0) * 16u;
        #pragma unroll
        for (int k = 0; k < G; ++k) {
            const float4 v0 = ld_at(Pq[k], boff), v1 = ld_at(Pq[k], boff + 16u);
            float4& a = acc[k];
            a.x = fmaf(v0.x, w0, a.x); a.y = fmaf(v0.y, w0, a.y); a.z = fmaf(v0.z, w0, a.z); a.w = fmaf(v0.w, w0, a.w);
            a.x = fmaf(v1.x, w1, a.x); a.y = fmaf(v1.y, w1, a.y); a.z = fmaf(v1.z, w1, a.z); a.w = fmaf(v1.w, w1, a.w);
            if (NC == 3) {
                const float4 v2 = ld_at(Pq[k], boff + 32u);
                a.x = fmaf(v2.x, w2, a.x); a.y = fmaf(v2.y, w2, a.y);
                a.z = fmaf(v2.z, w2, a.z); a.w = fmaf(v2.w, w2, a.w);
            }
        }
    }
}

// One bin ray through G interleaved slice groups of the padded quad averaged
// planes QX [q][ny][qpitch(nx)] (X views) and QY [q][nx][qpitch(ny)] (Y views);
// H parts of 64 / H lanes split the wave's line range as in
// siddon_fp_ray_quads.
template <int G, int H = 1>
__device__ __forceinline__ void dd_fp_ray_quads(const FanK& g, const float4* __restrict__ QX,
                                                const float4* __restrict__ QY, int nq, int view, int iu, bool active,
                                                float4 (&acc)[G])
{
    const float4 d = g.dray[(long)view * g.nu + iu];
    const float L = g.sray[(long)view * g.nu + iu].z;
    const bool xv = g.vcls[view] == 0;
    const float4* __restrict__ P = xv ? QX : QY;
    const int nl = xv ? g.ny : g.nx;
    const int n = xv ? g.nx : g.ny;
    const int pitch = qpitch(n);
    const long qstride = (long)nl * pitch;
    const float base = -0.5f * (float)nl;
    int j0, j1;
    float wmax;
    dd_ray_lines(d, n, nl, base, j0, j1, wmax);
    if (!active) { j0 = nl; j1 = -1; wmax = 0.0f; }
    int wj0 = wave_min(j0);
    int wj1 = wave_max(j1);
    static_assert(H == 1 || H == 2 || H == 4, "parts of a wave");
    const int len = wj1 - wj0 + 1;
    if (H > 1 && len > 0) {
        const int part = (int)(threadIdx.x & 63) / (64 / H);
        const int a = wj0 + len * part / H, b = wj0 + len * (part + 1) / H - 1;
        wj0 = a;
        wj1 = b;
    }
    const float4* Pq[G];
    #pragma unroll
    for (int k = 0; k < G; ++k) {
        Pq[k] = P + (long)min(k, nq - 1) * qstride;
        acc[k] = vzero<float4>();
    }
    if (__all(wmax <= 0.999f)) {
        dd_quad_lines_padded<G, 2>(Pq, n, pitch, d, base, wj0, wj1, acc);
    } else if (__all(wmax <= 1.999f)) {
        dd_quad_lines_padded<G, 3>(Pq, n, pitch, d, base, wj0, wj1, acc);
    } else {
        for (int j = wj0; j <= wj1; ++j) {
            const float lr = base + (float)j;
            const float ea = fmaf(d.y, lr, d.x), eb = fmaf(d.w, lr, d.z);
            #pragma unroll
            for (int k = 0; k < G; ++k)
                vadd(acc[k], vscale(seg_sum<float4>(Pq[k] + (long)j * pitch + kQPadL, n, fminf(ea, eb),
                                                    fmaxf(ea, eb)), 1.0f / fabsf(eb - ea)));
        }
    }
    #pragma unroll
    for (int o = 32; o >= 64 / H; o >>= 1) {
        #pragma unroll
        for (int k = 0; k < G; ++k) {
            acc[k].x += __shfl_xor(acc[k].x, o);
            acc[k].y += __shfl_xor(acc[k].y, o);
            acc[k].z += __shfl_xor(acc[k].z, o);
            acc[k].w += __shfl_xor(acc[k].w, o);
        }
    }
    #pragma unroll
    for (int k = 0; k < G; ++k) acc[k] = vscale(acc[k], L);
}

// atan from an odd polynomial on [-1, 1] (coefficients fitted here by
// iteratively reweighted least squares on Chebyshev nodes; maximum error
// 2.5e-7 rad) and, unless UNIT (|z| <= 1 known), atan(z) = sign(z) pi/2 -
// atan(1/z) outside.  Used only to locate the bins a pixel can meet;
// RN_ATAN_FAST_ERR bounds its error with FP32 evaluation included.
#define RN_ATAN_FAST_ERR 1.0e-6f
template <bool UNIT>
__device__ __forceinline__ float atan_fast(float z)
{
    const float az = fabsf(z);
    const bool inv = !UNIT && az > 1.0f;
    const float t = inv ? __builtin_amdgcn_rcpf(az) : az;
    const float s = t * t;
    float p = 0.006811782025349205f;
    p = fmaf(p, s, -0.033604191884230736f);
    p = fmaf(p, s, 0.07962364933877517f);
    p = fmaf(p, s, -0.13233341755196557f);
    p = fmaf(p, s, 0.1980781590519013f);
    p = fmaf(p, s, -0.3331736818605284f);
    p = fmaf(p, s, 0.9999961116602261f);
    float r = p * t;
    if (inv) r = 1.5707963267948966f - r;
    return copysignf(r, z);
}

// The projection of an 8 x 8-pixel tile onto the detector: its centre's angle
// th0 and distance r0 from the source once per view, every other point d of the
// tile relative to it,
//     theta(d) = th0 + atan(z),  z = (P dx + Q dy) / (1 + P dy - Q dx),
// (P, Q) the tangential direction over r0: |z| is about half the tile over r0
// (at most 1/4 with FanK::tile, kTileMax with FanK::tile_dd).  A wave owns a tile and works out 64 views
// at a time, one per lane; a view's numbers then reach the wave as scalars
// (v_readlane).  Bin coordinates are relative to `base`, the first bin the tile can
// meet; base + span is the last (span < 0: the tile misses the detector).
constexpr float kTileMax = 0.15f;
// view segments (one wave each, or in turn) of backprojections whose bits do not depend
// on the launch shape
constexpr int kBpSegs = 8;

// 1/15!, 1/14!, 1/13!, ..., 1/1!, 1/0!: sin and cos from the highest term down, in
// memory so that the loop over them keeps no registers between batches
__constant__ const double kTrig[16] = {
    1.0 / 1307674368000.0, 1.0 / 87178291200.0, 1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0,
    1.0 / 3628800.0, 1.0 / 362880.0, 1.0 / 40320.0, 1.0 / 5040.0, 1.0 / 720.0, 1.0 / 120.0, 1.0 / 24.0,
    1.0 / 6.0, 1.0 / 2.0, 1.0, 1.0};

__device__ __forceinline__ float lane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The tile's points to FP32 accuracy relative to a centre angle in FP64: an angle
// to about 1e-9 rad (an absolute bin coordinate in FP32 has 1e-7).
struct TileProj {
    float P, Q;         // per mm
    float u0;           // bin coordinate of the centre minus base
    float kr;           // dso^2 / r0^2
    int base, span;
    float px, py;       // this lane's pixel from the tile centre, mm

    __device__ __forceinline__ void init(const FanK& g, int lane)
    {
        px = ((float)(lane >> 3) - 3.5f) * g.dx;
        py = ((float)(lane & 7) - 3.5f) * g.dy;
    }
    // Views view .. view + 63 (this lane's: view + lane, clamped) of the tile whose
    // first pixel is (tx, ty); ub: bin coordinate of angle 0.
    __device__ __forceinline__ void batch(const FanK& g, int view, int lane, int tx, int ty, double ub)
    {
        // (opaque, so that nothing of the tile is kept in registers between batches)
        asm volatile("" : "+s"(tx), "+s"(ty));
        const int v = min(view + lane, g.nview - 1);
        const double c = g.vcos[v], s = g.vsin[v];
        const double x = (tx + 3.5 - 0.5 * (g.nx - 1)) * (double)g.dx, y = (ty + 3.5 - 0.5 * (g.ny - 1)) * (double)g.dy;
        const double rx = x * c + y * s, d = y * c - x * s + (double)g.dso;
        const double r2 = rx * rx + d * d;
        const float ir2 = 1.0f / (float)r2;
        P = (float)(c * d + s * rx) * ir2;
        Q = (float)(s * d - c * rx) * ir2;
        kr = g.dso * g.dso * ir2;
        // th0: an FP32 estimate t, then the small angle left, (rx cos t - d sin t) / r0,
        // with sin t and cos t from their Taylor series (|t| < 1.2: terms past t^15
        // are below 1e-12)
        const double t = (double)atan_fast<false>((float)rx / (float)d), q = t * t;
        double sn = kTrig[0], cn = kTrig[1];
        #pragma unroll 1
        for (int i = 2; i < 16; i += 2) {
            sn = fma(sn, -q, kTrig[i]);
            cn = fma(cn, -q, kTrig[i + 1]);
        }
        sn *= t;
        const double th = t + (double)((float)(rx * cn - d * sn) * sqrtf(ir2));
        const double u = ub - th / (double)g.da;
        // the tile's corners lie within |P| 4 dx + |Q| 4 dy of z's numerator, the
        // denominator within that (with dx and dy exchanged) of 1; atan z <= z
        const float m = fabsf(P) * 4.0f * g.dx + fabsf(Q) * 4.0f * g.dy;
        const float n = fabsf(P) * 4.0f * g.dy + fabsf(Q) * 4.0f * g.dx;
        const double w = (double)(m / ((1.0f - n) * fabsf(g.da)) + 0.02f);
        const double lo = fmin(fmax(floor(u - w), 0.0), (double)g.nu);
        const double hi = fmax(fmin(floor(u + w), (double)(g.nu - 1)), -1.0);
        base = (int)lo;
        span = (int)hi - base;
        u0 = (float)(u - lo);
    }
};

// The bins whose centre rays can meet each of the tile's pixels (a superset; the
// others have weight 0): centre coordinate u0 - m (1 - n), m and n the numerator
// and denominator of z in bins, to the second order, and one half width per view
// that covers the pixel's box, the remainder's bound and FP32.
struct TileRange {
    float P, Q;         // bins per mm
    float u0, hw;
    int base, span;
    float px, py, da;   // this lane's pixel from the tile centre, mm

    __device__ __forceinline__ void init(const FanK& g, int lane)
    {
        px = ((float)(lane >> 3) - 3.5f) * g.dx;
        py = ((float)(lane & 7) - 3.5f) * g.dy;
        da = g.da;
    }
    // as TileProj::batch; pad: further bins on either side
    __device__ __forceinline__ void batch(const FanK& g, int view, int lane, int tx, int ty, float pad)
    {
        asm volatile("" : "+s"(tx), "+s"(ty));
        const int v = min(view + lane, g.nview - 1);
        const float c = g.vcos[v], s = g.vsin[v], ida = 1.0f / g.da;
        const float x = ((float)tx + 3.5f - 0.5f * (float)(g.nx - 1)) * g.dx;
        const float y = ((float)ty + 3.5f - 0.5f * (float)(g.ny - 1)) * g.dy;
        const float rx = x * c + y * s, d = y * c - x * s + g.dso;
        const float ir2 = 1.0f / fmaf(rx, rx, d * d);
        P = (c * d + s * rx) * ir2;
        Q = (s * d - c * rx) * ir2;
        const float u = g.cu - g.off_a - atan_fast<false>(rx / d) * ida;
        const float m = fabsf(P) * 4.0f * g.dx + fabsf(Q) * 4.0f * g.dy;
        const float n = fabsf(P) * 4.0f * g.dy + fabsf(Q) * 4.0f * g.dx;
        const float zm = m / (1.0f - n), a = fabsf(ida);
        // FP32: the angle to RN_ATAN_FAST_ERR and 1e-6 of its rounded operands, the bin
        // coordinate to 1e-6 of its size
        const float eps = 0.02f + pad + (RN_ATAN_FAST_ERR + 1e-6f) * a + 1e-6f * (float)g.nu;
        // the pixel's corners (an eighth of the tile) move numerator and denominator; the
        // centre's z is m (1 - n) to n^2 z and atan z is z to z^3
        hw = (0.125f * zm / (1.0f - n) + n * n * zm + zm * zm * zm) * a + eps;
        const float w = zm * a + eps;
        const float lo = fminf(fmaxf(floorf(u - w), 0.0f), (float)g.nu);
        const float hi = fmaxf(fminf(floorf(u + w), (float)(g.nu - 1)), -1.0f);
        base = (int)lo;
        span = (int)hi - base;
        u0 = u - lo;
        P *= ida;
        Q *= ida;
    }
    // this lane's first and last bin, relative to base, in the view of lane l
    __device__ __forceinline__ void range(int l, int span_l, int& t0, int& t1) const
    {
        const float p = lane_f(P, l), q = lane_f(Q, l), h = lane_f(hw, l);
        const float m = fmaf(p, px, q * py), n1 = fmaf(fmaf(p, py, -q * px), da, -1.0f);
        const float u = fmaf(m, n1, lane_f(u0, l));
        t0 = max((int)ceilf(u - h), 0);
        t1 = min((int)floorf(u + h), span_l);
    }
};

// First and last bin whose centre ray can meet pixel (ix, iy) of view `view`:
// the pixel lies in the disc of radius rpix around its centre, whose rays span
// the detector angles atan(rx / d0) +- asin(s), s = rpix / dist, and
// asin(s) <= s (1 + 2 s) for 0 <= s <= 1.  UNIT: |rx / d0| <= 1 for every pixel
// and view of the geometry (FanK::unit_angle).
template <bool UNIT>
__device__ __forceinline__ void bin_range(const FanK& g, float xc, float yc, float rpix, float inv_da, int view,
                                          float pad, int& k0, int& k1)
{
    const float ct = g.vcos[view], st = g.vsin[view];
    const float rx = xc * ct + yc * st, ry = -xc * st + yc * ct;
    const float d0 = ry + g.dso;
    const float uc = g.cu - g.off_a - atan_fast<UNIT>(rx * __builtin_amdgcn_rcpf(d0)) * inv_da;
    const float sr = fminf(rpix * __builtin_amdgcn_rsqf(fmaf(rx, rx, d0 * d0)), 1.0f);
    const float hw = sr * fmaf(2.0f, sr, 1.0f) * fabsf(inv_da) + 0.02f + pad + RN_ATAN_FAST_ERR * fabsf(inv_da);
    k0 = max((int)ceilf(uc - hw), 0);
    k1 = min((int)floorf(uc + hw), g.nu - 1);
}

// Length of ray r in cell `cell` of line lr (the weight siddon_fp_ray_slices gives
// it), computed without branches: overlap and width of the interval between the
// line's crossings ea and eb (both have the sign of eb - ea).
__device__ __forceinline__ float siddon_cell_weight(const float4 r, float lr, float cell)
{
    const float ea = fmaf(r.y, lr, r.x), eb = fmaf(r.y, lr + 1.0f, r.x), c1 = cell + 1.0f;
    const float ov = __builtin_amdgcn_fmed3f(eb, cell, c1) - __builtin_amdgcn_fmed3f(ea, cell, c1);
    const bool pos = ea != eb;
    const float pt = (ea >= cell && ea < c1) ? 1.0f : 0.0f;
    const float inv = __builtin_amdgcn_rcpf(pos ? eb - ea : 1.0f);
    return (pos ? ov * inv : pt) * r.z;
}

// the bins k0 .. k1 of one view for S slices (slice q's row `rboff` bytes
// after the wave-uniform base pq[q]; the view's ray table row `rowoff` bytes
// after g.sray): the first NB unrolled (each under its own lane mask, so an
// empty range k1 < k0 adds nothing), the rest in a loop; each weight is
// computed once and applied to every slice.
template <class T, int NB, int S>
__device__ __forceinline__ void siddon_gather_bins(const float4* __restrict__ sray, unsigned rowoff,
                                                   const T* const (&pq)[S], unsigned rboff, int nu, int k0, int k1,
                                                   float lr, float cell, T (&acc)[S])
{
    #pragma unroll
    for (int j = 0; j < NB; ++j) {
        // lanes past k1 take no part (their loads are masked off, so they
        // cost no vector-memory bandwidth); the others add weight x value
        if (k0 + j <= k1) {
            const unsigned kk = (unsigned)(k0 + j);
            const float wt = siddon_cell_weight(ld_at(sray, rowoff + kk * 16u), lr, cell);
            const unsigned boff = rboff + kk * (unsigned)sizeof(T);
            #pragma unroll
            for (int q = 0; q < S; ++q) vmadd(acc[q], ld_at(pq[q], boff), wt);
        }
    }
    for (int k = k0 + NB; k <= k1; ++k) {
        const float wt = siddon_cell_weight(ld_at(sray, rowoff + (unsigned)k * 16u), lr, cell);
        const unsigned boff = rboff + (unsigned)k * (unsigned)sizeof(T);
        #pragma unroll
        for (int q = 0; q < S; ++q) vmadd(acc[q], ld_at(pq[q], boff), wt);
    }
}

// siddon_gather_bins for G slice groups from a wave's staged window in LDS:
// row q of `st` holds group q's values and row G the view's ray table, CAP
// bins per row from the window's first bin (every slot holds written values:
// the caller clears the rows before its first window); t0 .. t1 are the pixel's bins
// relative to that first bin.  The first two bins are taken by every lane with
// no branch around the accumulators (a lane past t1 reads the zero entry), which keeps
// the kernel in registers.  The rest in a loop.
template <int G, int CAP>
__device__ __forceinline__ void siddon_gather_staged(const float4* st, int t0, int t1, float lr, float cell,
                                                     float4 (&acc)[G])
{
    const bool on0 = t0 <= t1, on1 = t0 < t1;
    const int i0 = on0 ? t0 : CAP, i1 = on1 ? t0 + 1 : CAP;
    constexpr int CS = stage_pitch(CAP);
    const float c0 = siddon_cell_weight(st[G * CS + i0], lr, cell);
    const float c1 = siddon_cell_weight(st[G * CS + i1], lr, cell);
    const float w0 = on0 ? c0 : 0.0f, w1 = on1 ? c1 : 0.0f;
    #pragma unroll
    for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * CS + i0], w0);
    #pragma unroll
    for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * CS + i1], w1);
    for (int t = t0 + 2; t <= t1; ++t) {
        const float w = siddon_cell_weight(st[G * CS + t], lr, cell);
        #pragma unroll
        for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * CS + t], w);
    }
}

// Exact transpose of siddon_fp_ray_slices: pixel (ix, iy) gathers, over views
// view0 .. view0+nviews-1 of prj ([nviews][nu] per slice, slices sstride
// elements apart; slices q >= nsl read slice nsl - 1 and are discarded by the
// caller), the rays that cross it, with their weights there.
// The bin range and the weights are computed once per view for all S slices.
// The first NB bins of a pixel's range are taken without branches, the rest
// in a loop (NB changes only the speed).
template <class T, int NB, bool UNIT, int S>
__device__ __forceinline__ void siddon_bp_views(const FanK& g, const T* __restrict__ prj, long sstride, int nsl,
                                                int view0, int nviews, int ix, int iy, T (&acc)[S])
{
    const float xc = (ix - 0.5f * (g.nx - 1)) * g.dx, yc = (iy - 0.5f * (g.ny - 1)) * g.dy;
    const float rpix = 0.5f * sqrtf(g.dx * g.dx + g.dy * g.dy);
    const float inv_da = 1.0f / g.da;
    const float yr = (float)iy - 0.5f * g.ny;
    const float xr = (float)ix - 0.5f * g.nx;
    const T* pq[S];                             // wave-uniform slice bases
    #pragma unroll
    for (int q = 0; q < S; ++q) {
        pq[q] = prj + (long)min(q, nsl - 1) * sstride;
        acc[q] = vzero<T>();
    }
    for (int vi = 0; vi < nviews; ++vi) {
        const int view = view0 + vi;
        int k0, k1;
        bin_range<UNIT>(g, xc, yc, rpix, inv_da, view, 0.0f, k0, k1);
        const bool xv = g.vcls[view] == 0;
        const float lr = xv ? yr : xr;          // this pixel's line
        const float cell = xv ? (float)ix : (float)iy;
        siddon_gather_bins<T, NB, S>(g.sray, (unsigned)(view * g.nu) * 16u, pq,
                                     (unsigned)(vi * g.nu) * (unsigned)sizeof(T), g.nu, k0, k1, lr, cell, acc);
    }
}

template <class T, int NB, int S>
__device__ __forceinline__ void siddon_bp_pixel_slices(const FanK& g, const T* __restrict__ prj, long sstride,
                                                       int nsl, int view0, int nviews, int ix, int iy,
                                                       T (&acc)[S])
{
    if (g.unit_angle) siddon_bp_views<T, NB, true, S>(g, prj, sstride, nsl, view0, nviews, ix, iy, acc);
    else siddon_bp_views<T, NB, false, S>(g, prj, sstride, nsl, view0, nviews, ix, iy, acc);
}

// Views v0 .. v1 - 1 (rows of prj [view][nu], view0 + v in the tables) of one group of
// slices for this lane's pixel of the tile whose first pixel is (tx, ty), gathered from
// memory; every lane of the wave calls it.
template <int NB>
__device__ __forceinline__ void siddon_bp_tile1(const FanK& g, const float4* __restrict__ prj, int view0, int v0,
                                                int v1, int tx, int ty, int lane, float4 (&acc)[1])
{
    const int ix = tx + (lane >> 3), iy = ty + (lane & 7);
    const bool inside = ix < g.nx && iy < g.ny;
    const float4* const P[1] = {prj};
    const float4* const sray = g.sray + (long)view0 * g.nu;
    const float yr = (float)iy - 0.5f * g.ny, xr = (float)ix - 0.5f * g.nx;
    TileRange tr;
    tr.init(g, lane);
    for (int vi = v0; vi < v1; ++vi) {
        const int w = (vi - v0) & 63;
        if (w == 0) tr.batch(g, view0 + vi, lane, tx, ty, 0.0f);
        const int span = __builtin_amdgcn_readlane(tr.span, w);
        if (span < 0) continue;
        int t0, t1;
        tr.range(w, span, t0, t1);
        if (!inside) t1 = -1;
        const bool xv = g.vcls[view0 + vi] == 0;
        const unsigned row = (unsigned)(vi * g.nu + __builtin_amdgcn_readlane(tr.base, w)) * 16u;
        siddon_gather_bins<float4, NB, 1>(sray, row, P, row, g.nu, t0, t1, xv ? yr : xr, xv ? (float)ix : (float)iy,
                                          acc);
    }
}

// Exact transpose of the DD FP (dd_fp_ray_slices; no reference counterpart:
// the reference DD BP is not the adjoint of its FP).  The pixel enters line
// iy (or ix), its lower edge, and line iy + 1 (or ix + 1), its upper edge,
// with weight 1/2 each (each line averages two rows); on each it takes, from
// every bin whose footprint meets its segment, the FP's share overlap / width
// from the same edge rays.  One pass over the candidate bins serves both
// lines: the bins whose centre lies within half a bin of the angles the
// pixel's box spans (TileRange, or without FanK::tile bin_range, plus half a bin; the
// others have zero overlap).
//
// A wave takes an 8 x 8-pixel tile of G groups of 4 interleaved slices
// (float4 sinograms [view][nu], already multiplied by the rays' length per
// line) and stages, per view, the tile's bin window in its own LDS rows: the
// groups' values and the window's bin edges, (A, B) of one edge ray per entry,
// each edge shared by the two bins it separates.  As in k_siddon_fan_bp_tile: CAP
// bins at a time, loaded one step (a view, or a further CAP bins of it) ahead into
// registers, no barrier (a wave touches only its rows), rows cleared at the start
// (lanes without a bin read a row's zero entry).
//
// The views are summed in kBpSegs fixed segments whose sums are then added
// in order, one wave each, so that a batch and its slices alone give the same bits.
template <int G, int CAP>
struct DdAdjStage {
    static constexpr int kVals = G * stage_pitch(CAP);     // float4: the groups' bins
    static constexpr int kEdges = (CAP + 3) / 2;           // float4: CAP + 1 edges of 8 bytes and one unused
    static constexpr int kFloat4 = kVals + kEdges;         // LDS of one wave
};

// Shares of the bins t0 .. t1 (relative to the staged window, t0 >= 0 where
// t1 >= t0; empty otherwise) of lines lr and lr + 1 in cell [cell, cell + 1],
// applied to the G groups.  up: 1/2 if the upper line exists, else 0.  WIDE:
// every footprint of the geometry has a positive FP32 width (FanK::dwide).
template <int G, int CAP, int NB, bool WIDE>
__device__ __forceinline__ void dd_adj_gather(const float4* st, int t0, int t1, float lr, float cell, float up,
                                              float4 (&acc)[G])
{
    const float2* edge = reinterpret_cast<const float2*>(st + DdAdjStage<G, CAP>::kVals);
    const float c1 = cell + 1.0f, lu = lr + 1.0f;
    const int ts = t1 >= t0 ? t0 : 0;
    float2 e = edge[ts];
    float a0 = fmaf(e.y, lr, e.x), a1 = fmaf(e.y, lu, e.x);
    float q0 = __builtin_amdgcn_fmed3f(a0, cell, c1), q1 = __builtin_amdgcn_fmed3f(a1, cell, c1);
    // 1/2 share on line lr + up x share on line lr + 1 (overlap and width have
    // one sign: the edges are monotone); WIDE: both quotients by one reciprocal
    auto weight = [&](float b0, float b1, float p0, float p1) {
        const float w0 = b0 - a0, w1 = b1 - a1, v0 = p0 - q0, v1 = p1 - q1;
        if (WIDE) return fmaf(0.5f * v0, w1, up * v1 * w0) * __builtin_amdgcn_rcpf(w0 * w1);
        const float l0 = fminf(a0, b0), l1 = fminf(a1, b1);
        const float s0 = w0 != 0.0f ? v0 * __builtin_amdgcn_rcpf(w0) : ((l0 >= cell && l0 < c1) ? 1.0f : 0.0f);
        const float s1 = w1 != 0.0f ? v1 * __builtin_amdgcn_rcpf(w1) : ((l1 >= cell && l1 < c1) ? 1.0f : 0.0f);
        return fmaf(up, s1, 0.5f * s0);
    };
    // bin at slot t, its upper edge at slot t + 1
    auto bin = [&](int t, bool on) {
        e = edge[t + 1];
        const float b0 = fmaf(e.y, lr, e.x), b1 = fmaf(e.y, lu, e.x);
        const float p0 = __builtin_amdgcn_fmed3f(b0, cell, c1), p1 = __builtin_amdgcn_fmed3f(b1, cell, c1);
        const float wt = weight(b0, b1, p0, p1);
        const float w = on ? wt : 0.0f;
        #pragma unroll
        for (int q = 0; q < G; ++q) vmadd(acc[q], st[q * stage_pitch(CAP) + t], w);
        a0 = b0; a1 = b1; q0 = p0; q1 = p1;
    };
    #pragma unroll
    for (int j = 0; j < NB; ++j) {
        const bool on = t0 + j <= t1;
        bin(on ? t0 + j : CAP, on);
    }
    for (int t = t0 + NB; t <= t1; ++t) bin(t, true);
}

// View segment seg of kBpSegs of the G groups at P (groups sstride cells apart,
// groups k >= nq read group nq - 1 and are discarded by the caller) for this lane's
// pixel of the tile whose first pixel is (tx, ty); lanes outside the image stage only.
// st: this wave's DdAdjStage LDS.  Byte offsets from P stay below 2^31 (checked on the
// host).
template <int G, int CAP, int NB, bool WIDE>
__device__ __forceinline__ void dd_adj_tile(const FanK& g, const float4* __restrict__ P, long sstride, int nq,
                                            int nviews, int seg, int tx, int ty, int lane, float4* st,
                                            float4 (&acc)[G])
{
    using S = DdAdjStage<G, CAP>;
    static_assert(CAP < 64, "one load for the edges");
    constexpr int kLoads = (G * CAP + 63) / 64;
    for (int i = lane; i < S::kFloat4; i += 64) st[i] = vzero<float4>();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int ix = tx + (lane >> 3), iy = ty + (lane & 7);
    const bool inside = ix < g.nx && iy < g.ny;
    const float yr = (float)iy - 0.5f * g.ny, xr = (float)ix - 0.5f * g.nx;
    int bj[kLoads], slot[kLoads];   // slot: the zero entries of the rows before
    unsigned roff[kLoads];
    #pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int i = j * 64 + lane;
        bj[j] = i % CAP;
        slot[j] = G == 1 ? 0 : i / CAP;
        roff[j] = (unsigned)(min(i / CAP, nq - 1) * sstride) * 16u;
    }
    float4 rg[kLoads];
    float2 re;
    #pragma unroll
    for (int q = 0; q < G; ++q) acc[q] = vzero<float4>();
    TileRange tr;
    tr.init(g, lane);
    const int v0 = (int)((long)nviews * seg / kBpSegs), v1 = (int)((long)nviews * (seg + 1) / kBpSegs);
    // the candidate bins of view row vi: the tile's window [base, base + span] and
    // this lane's bins t0 .. t1 in it (span < 0: none)
    int t0 = 0, t1 = -1, base = 0, span = -1;
    auto prepare = [&](int vi) {
        if (g.tile) {
            const int w = (vi - v0) & 63;
            if (w == 0) tr.batch(g, vi, lane, tx, ty, 0.5f);
            span = __builtin_amdgcn_readlane(tr.span, w);
            if (span < 0) return;
            base = __builtin_amdgcn_readlane(tr.base, w);
            tr.range(w, span, t0, t1);
            if (!inside) t1 = -1;
        } else {
            const float rpix = 0.5f * sqrtf(g.dx * g.dx + g.dy * g.dy), inv_da = 1.0f / g.da;
            int k0, k1;
            bin_range<false>(g, ((float)ix - 0.5f * (g.nx - 1)) * g.dx, ((float)iy - 0.5f * (g.ny - 1)) * g.dy, rpix,
                             inv_da, vi, 0.5f, k0, k1);
            if (!inside || k1 < k0) { k0 = g.nu; k1 = -1; }
            base = wave_min(k0);
            span = wave_max(k1) - base;
            t0 = k0 - base;
            t1 = k1 - base;
        }
    };
    int vi = v0 - 1, off = 0;
    bool xv = true;
    for (bool more = true;;) {
        const int a0 = max(t0, 0), a1 = min(t1, CAP - 1);
        // the step's view: the pixel's line and cell, 1/2 if the line above exists
        const float lr = xv ? yr : xr, hl = 0.5f * (xv ? g.ny : g.nx);
        const float cell = xv ? xr + 0.5f * g.nx : yr + 0.5f * g.ny, up = lr + 1.0f < hl ? 0.5f : 0.0f;
        if (off + CAP <= span) {
            off += CAP;
            t0 -= CAP;
            t1 -= CAP;
        } else {
            off = 0;
            do {
                more = ++vi < v1;
                if (!more) break;
                prepare(vi);
            } while (span < 0);
            if (more) xv = g.vcls[vi] == 0;
        }
        if (more) {
            // CAP bins and their CAP + 1 edges (edge e is the first edge of bin e, the last
            // one the second edge of the last bin)
            #pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP)
                    rg[j] = ld_at(P, roff[j] + (unsigned)(vi * g.nu + min(base + off + bj[j], g.nu - 1)) * 16u);
            if (lane < CAP + 1) {
                const int e = min(base + off + lane, g.nu);
                const float2* d2 = reinterpret_cast<const float2*>(g.dray);
                re = ld_at(d2, (unsigned)((vi) * g.nu + e) * 16u - (e < g.nu ? 0u : 8u));
            }
        }
        dd_adj_gather<G, CAP, NB, WIDE>(st, a0, a1, lr, cell, up, acc);
        if (!more) break;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        #pragma unroll
        for (int j = 0; j < kLoads; ++j)
            if (64 * (j + 1) <= G * CAP || j * 64 + lane < G * CAP) st[j * 64 + lane + slot[j]] = rg[j];
        if (lane < CAP + 1) reinterpret_cast<float2*>(st + S::kVals)[lane] = re;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

// Adds the G values per lane of a workgroup's nw waves in wave order through
// red [G][64]; true in the wave that holds the sums (every wave calls it).
template <int G>
__device__ __forceinline__ bool add_waves(float4 (&v)[G], float4* red, int lane, int wv, int nw)
{
    if (nw == 1) return true;
    for (int w = 0; w < nw; ++w) {
        if (w == wv) {
            #pragma unroll
            for (int k = 0; k < G; ++k) {
                if (w > 0) {
                    const float4 r = red[k * 64 + lane];
                    v[k] = make_float4(r.x + v[k].x, r.y + v[k].y, r.z + v[k].z, r.w + v[k].w);
                }
                red[k * 64 + lane] = v[k];
            }
        }
        __syncthreads();
    }
    return wv == nw - 1;
}

} // namespace fan
} // namespace rn

namespace rn {

// The OS-SQS(-TV) update of one pixel of one slice (ossqs.cu:124-135 with the
// TV terms of TotalVariation.cu:9-68): x - (step g + beta2 gTV) / (D + beta2 nTV + 1e-6),
// cropped to [lb, ub] when crop is set.  dx0, dx1, dy0, dy1 are the differences
// to the 4-neighbours (the pixel value itself at the image border); gTV =
// sum d / psi / 2 and nTV = sum 1 / psi with psi = sqrt(d^2 + eps), here with
// reciprocal square roots (about 1 ulp each), and the quotient as a product
// with a 1-ulp reciprocal.  g: the backprojected weighted residual, d: the
// normaliser.
__device__ __forceinline__ float sqs_update_core(float x, float dx0, float dx1, float dy0, float dy1, float g,
                                                 float d, float step, float beta2, float eps, float lb, float ub,
                                                 int crop)
{
    float num = step * g;
    float den = d;
    if (beta2 != 0.0f) {
        const float r0 = __builtin_amdgcn_rsqf(fmaf(dx0, dx0, eps)), r1 = __builtin_amdgcn_rsqf(fmaf(dx1, dx1, eps));
        const float r2 = __builtin_amdgcn_rsqf(fmaf(dy0, dy0, eps)), r3 = __builtin_amdgcn_rsqf(fmaf(dy1, dy1, eps));
        const float gt = 0.5f * (dx0 * r0 + dx1 * r1 + dy0 * r2 + dy1 * r3);
        const float nt = r0 + r1 + r2 + r3;
        num = fmaf(beta2, gt, num);
        den = fmaf(beta2, nt, den);
    }
    float xn = x - num * __builtin_amdgcn_rcpf(den + 1e-6f);     // 1-ulp reciprocal
    if (crop) xn = xn < lb ? lb : (xn > ub ? ub : xn);
    return xn;
}

// sqs_update_core for pixel (ix, iy) of one slice Xs [nx][ny], pix = ix * ny + iy
__device__ __forceinline__ float sqs_pixel_update(const float* __restrict__ Xs, long pix, int ix, int iy, int nx,
                                                  int ny, float g, float d, float step, float beta2, float eps,
                                                  float lb, float ub, int crop)
{
    const float x = Xs[pix];
    float dx0 = 0.0f, dx1 = 0.0f, dy0 = 0.0f, dy1 = 0.0f;
    if (beta2 != 0.0f) {
        dx0 = ix == 0 ? x : x - Xs[pix - ny];
        dx1 = ix == nx - 1 ? x : x - Xs[pix + ny];
        dy0 = iy == 0 ? x : x - Xs[pix - 1];
        dy1 = iy == ny - 1 ? x : x - Xs[pix + 1];
    }
    return sqs_update_core(x, dx0, dx1, dy0, dy1, g, d, step, beta2, eps, lb, ub, crop);
}

} // namespace rn
