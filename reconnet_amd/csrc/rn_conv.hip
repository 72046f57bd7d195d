// 3x3 "same" convolutions of the learned prior (no reference counterpart).
//
// Network: 1 -> 32 -> 32 -> 32 -> 32 -> 1 channels, 3x3 kernels, ReLU after
// the first four layers, residual output y = x + conv5(...).
// Activations are BF16, NHWC ([B][H][W][32], 64 bytes per pixel); every
// product accumulates in FP32.
//
// The 32 -> 32 layers (forward and data gradient) run on gfx950 BF16 matrix
// cores (v_mfma_f32_32x32x16_bf16, A = weights, B = pixels); their weight
// gradient is an MFMA GEMM over pixels whose operands are transposed by the LDS
// reads themselves.  The 1 -> 32 layer and its and the 32 -> 1 layer's weight
// gradients use FP32 (VALU, FP32 MFMA), the 32 -> 1 layer split weights on MFMA.

#include "rn_conv.h"
#include "rn_tune.h"

#include <algorithm>
#include <type_traits>

namespace rn {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// two floats -> two bf16 (round to nearest even, NaN stays NaN) packed low | high << 16,
// one hardware conversion (v_cvt_pk_bf16_f32) for the pair
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    const f32x2 f = {lo, hi};
    const bf16x2 h = __builtin_convertvector(f, bf16x2);
    uint32_t u;
    __builtin_memcpy(&u, &h, sizeof(u));
    return u;
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v)
{
    bf16x8 r;
    __builtin_memcpy(&r, &v, sizeof(r));
    return r;
}

// ---------------------------------------------------------------------------
// layer 1: x (fp32 [B][H][W]) -> relu(conv(x) + b) (bf16 NHWC), w [9][32]
//
// One wave per 62 pixels of an image row: lane l holds column x0 + l - 1 of
// the three input rows (one load per row, zero outside the image), the left
// and right neighbours come from the adjacent lanes, and lanes 1 .. 62
// compute their pixel's 32 channels (lanes 0 and 63 only supply neighbours).
// The wave's 62 x 64 output bytes are gathered in LDS and written with
// contiguous 16-byte stores, 1 KB per instruction.
// ---------------------------------------------------------------------------
constexpr int kConvInTile = 62;

__global__ __launch_bounds__(256) void k_conv_in(const float* __restrict__ x, const float* __restrict__ w,
                                                 const float* __restrict__ b, uint16_t* __restrict__ out,
                                                 int H, int W, int tiles, long nwaves)
{
    // weights and biases are read at wave-uniform addresses (scalar loads)
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave >= nwaves) return;                  // whole waves
    const int tile = (int)(wave % tiles);
    const long row = wave / tiles;               // image * H + yh
    const int yh = (int)(row % H);
    const long img = (row - yh) * W;             // first pixel of the image
    const int xc = tile * kConvInTile + lane - 1;
    const bool col = xc >= 0 && xc < W;
    float c[3];
    #pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
        const int yy = yh + dy - 1;
        c[dy] = (col && yy >= 0 && yy < H) ? x[img + (long)yy * W + xc] : 0.0f;
    }
    float v[9];                                  // tap t = 3 dy + dx
    #pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
        v[3 * dy] = __shfl_up(c[dy], 1);
        v[3 * dy + 1] = c[dy];
        v[3 * dy + 2] = __shfl_down(c[dy], 1);
    }
    __shared__ uint4 sb[4][kConvInTile * 4];   // per wave: 62 pixels x 4 x 16 bytes
    uint4* ws = sb[(threadIdx.x >> 6) & 3];
    if (lane >= 1 && lane <= kConvInTile) {
        uint32_t packed[16];
        #pragma unroll
        for (int ch = 0; ch < 32; ch += 2) {
            float z0 = b[ch], z1 = b[ch + 1];
            #pragma unroll
            for (int t = 0; t < 9; ++t) {
                z0 = fmaf(w[t * 32 + ch], v[t], z0);
                z1 = fmaf(w[t * 32 + ch + 1], v[t], z1);
            }
            packed[ch / 2] = pack_bf16(fmaxf(z0, 0.0f), fmaxf(z1, 0.0f));
        }
        #pragma unroll
        for (int q = 0; q < 4; ++q)
            ws[(lane - 1) * 4 + q] = make_uint4(packed[4 * q], packed[4 * q + 1], packed[4 * q + 2], packed[4 * q + 3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    uint16_t* o = out + (img + (long)yh * W + tile * kConvInTile) * 32;
    const int npix = min(kConvInTile, W - tile * kConvInTile);
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = q * 64 + lane;               // 16-byte unit: pixel e / 4, channels 8 (e % 4) ..
        if (e / 4 < npix) reinterpret_cast<uint4*>(o)[e] = ws[e];
    }
}

// ---------------------------------------------------------------------------
// 32 -> 32 layer on MFMA: v_mfma_f32_32x32x16_bf16, which on gfx950 moves
// twice the flops per cycle of the 16x16x32 form (measured 2.17 against 1.22
// PFLOP/s on MI355X).  wt: [9][32 co][32 ci] bf16 (tap t = 3*dy + dx).
// mode 0: out = relu?(acc + bias); mode 1: out = acc * (mask > 0)
//
// Operands for tap t and input-channel half kc (ci 16 kc .. 16 kc + 15):
// A[m = co][k] on lane l: co = l % 32, ci = 16 kc + 8 (l / 32) .. + 7 (one
// 16-byte load of wt); B[k][n] on lane l: pixel n = l % 32 of a 32-pixel tile,
// the same 8 channels; D on lane l, register i: co = 8 (i / 4) + 4 (l / 32) +
// i % 4 of pixel l % 32.  Every output accumulates taps 0 .. 8, each with
// kc = 0 then 1, in that order, in the layer-by-layer and the fused kernels
// alike, so they give the same bits.
//
// Activation rows in LDS: [channel group g][pixel] 16-byte entries (g = 8
// channels) with a pitch of 4 (mod 16) entries, so the 32 lanes of a fragment
// read (same g, consecutive pixels) and a staging write (4 pixels x 4 groups
// per 16 lanes) hit distinct banks.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 zero16()
{
    f32x16 z;
    #pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}

// the 18 weight fragments of a 32 -> 32 layer
__device__ __forceinline__ void load_w32(const uint16_t* __restrict__ wt, int lane, bf16x8 (&wa)[9][2])
{
    #pragma unroll
    for (int tp = 0; tp < 9; ++tp)
        #pragma unroll
        for (int kc = 0; kc < 2; ++kc)
            wa[tp][kc] = as_bf16x8(*reinterpret_cast<const uint4*>(
                wt + ((tp * 32 + (lane & 31)) * 32 + 16 * kc + 8 * (lane >> 5))));
}

// One input row of a 32-pixel tile: f[dx][kc] are its fragments at column
// offset dx - 1; it adds taps 6 .. 8 to A (output row above), 3 .. 5 to Bm
// (same row) and 0 .. 2 to Cm (row below).
__device__ __forceinline__ void mid32_row(const bf16x8 (&wa)[9][2], const bf16x8 (&f)[3][2], f32x16& A, f32x16& Bm,
                                          f32x16& Cm)
{
    #pragma unroll
    for (int dx = 0; dx < 3; ++dx)
        #pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            A = mfma32(wa[6 + dx][kc], f[dx][kc], A);
            Bm = mfma32(wa[3 + dx][kc], f[dx][kc], Bm);
            Cm = mfma32(wa[dx][kc], f[dx][kc], Cm);
        }
}

// fragments of the tile whose dx = 0 pixel is entry p of the row buffer
template <int NPP>
__device__ __forceinline__ void frags32(const uint4* __restrict__ rb, int p, int lane, bf16x8 (&f)[3][2])
{
    #pragma unroll
    for (int dx = 0; dx < 3; ++dx)
        #pragma unroll
        for (int kc = 0; kc < 2; ++kc) f[dx][kc] = as_bf16x8(rb[(2 * kc + (lane >> 5)) * NPP + p + dx]);
}

template <int NW>
struct ConvRowStage {
    static constexpr int NP = 32 * NW + 2;                        // pixels of a staged row (1-pixel halo)
    static constexpr int NPP = NP + (((4 - NP) % 16) + 16) % 16;  // pitch = 4 (mod 16)
    static constexpr int NCH = NP * 4;                            // 16-byte chunks of a row
    static constexpr int NT = 64 * NW;                            // threads
    static constexpr int K = (NCH + NT - 1) / NT;                 // chunks per thread
};

template <int NW>
__device__ __forceinline__ void stage_load(const uint16_t* __restrict__ in, long img, int yy, int H, int W, int x0,
                                           int t, uint4 (&v)[ConvRowStage<NW>::K])
{
    using S = ConvRowStage<NW>;
    const bool rowok = yy >= 0 && yy < H;
    #pragma unroll
    for (int k = 0; k < S::K; ++k) {
        const int e = t + k * S::NT;
        const int x = x0 - 1 + (e >> 2);
        v[k] = make_uint4(0, 0, 0, 0);
        if (rowok && e < S::NCH && x >= 0 && x < W)
            v[k] = *reinterpret_cast<const uint4*>(in + (img + (long)yy * W + x) * 32 + 8 * (e & 3));
    }
}

template <int NW>
__device__ __forceinline__ void stage_store(uint4* __restrict__ buf, int t, const uint4 (&v)[ConvRowStage<NW>::K])
{
    using S = ConvRowStage<NW>;
    #pragma unroll
    for (int k = 0; k < S::K; ++k) {
        const int e = t + k * S::NT;
        if (e < S::NCH) buf[(e & 3) * S::NPP + (e >> 2)] = v[k];
    }
}

// One completed output row of a wave's 32 pixels: relu?(acc + bias) (mode 0)
// or acc * (mask > 0) (mode 1) as bf16, gathered in the wave's LDS tile
// (80-byte pixel pitch: conflict-free 8-byte writes) and written as two
// contiguous 16-byte stores per lane.
template <int MODE>
__device__ __forceinline__ void store32(const f32x16& acc, const float (&bv)[16], const uint16_t* __restrict__ mask,
                                        uint16_t* __restrict__ out, long rowbase, int xw, int W, int lane, int relu,
                                        uint4* __restrict__ tile)
{
    const int n = lane & 31, h = lane >> 5;
    uint2* tw = reinterpret_cast<uint2*>(tile);
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
        float z[4];
        if (MODE == 0) {
            #pragma unroll
            for (int e = 0; e < 4; ++e) {
                z[e] = acc[4 * q + e] + bv[4 * q + e];
                if (relu) z[e] = fmaxf(z[e], 0.0f);
            }
        } else {
            uint2 m = make_uint2(0, 0);
            if (xw + n < W) m = *reinterpret_cast<const uint2*>(mask + (rowbase + xw + n) * 32 + 8 * q + 4 * h);
            const uint16_t mk[4] = {(uint16_t)(m.x & 0xffff), (uint16_t)(m.x >> 16), (uint16_t)(m.y & 0xffff),
                                    (uint16_t)(m.y >> 16)};
            #pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = bf2f(mk[e]) > 0.0f ? acc[4 * q + e] : 0.0f;
        }
        tw[n * 10 + 2 * q + h] = make_uint2(pack_bf16(z[0], z[1]), pack_bf16(z[2], z[3]));
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    #pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int e = lane + 64 * k;                 // 16-byte chunk: pixel e / 4, channels 8 (e % 4) ..
        const uint4 v = tile[(e >> 2) * 5 + (e & 3)];
        if (xw + (e >> 2) < W) *reinterpret_cast<uint4*>(out + (rowbase + xw) * 32 + (long)e * 8) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// A workgroup of NW waves takes 32 NW adjacent columns and walks down L output
// rows of one image.  Each input row (the columns and a 1-pixel halo) is
// loaded once per workgroup, two rows ahead of its use, into one of two LDS
// row buffers, and feeds the three output rows that use it through three
// rolling accumulators; the oldest is complete after its third row and is
// stored.  The 18 weight fragments stay in registers.
template <int L, int MODE, int NW>
__global__ __launch_bounds__(64 * NW) void k_conv_mid(const uint16_t* __restrict__ in, const uint16_t* __restrict__ wt,
                                                    const float* __restrict__ bias,
                                                    const uint16_t* __restrict__ mask, uint16_t* __restrict__ out,
                                                    int H, int W, int relu)
{
    using S = ConvRowStage<NW>;
    __shared__ uint4 rows[2][4 * S::NPP];
    __shared__ uint4 tiles[NW][32 * 5];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wv = t >> 6;
    const int x0 = blockIdx.x * 32 * NW;                 // first column of the workgroup
    const int xw = x0 + 32 * wv;                         // first column of this wave
    const int y0 = blockIdx.y * L;
    const long img = (long)blockIdx.z * H * W;
    bf16x8 wa[9][2];
    load_w32(wt, lane, wa);
    float bv[16];
    #pragma unroll
    for (int i = 0; i < 16; ++i) bv[i] = (MODE == 0) ? bias[8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)] : 0.0f;
    f32x16 a0 = zero16(), a1 = zero16(), a2 = zero16();
    // step ir uses input row y0 - 1 + ir from buffer ir & 1
    uint4 nx[S::K], nn[S::K];
    stage_load<NW>(in, img, y0 - 1, H, W, x0, t, nx);
    stage_store<NW>(rows[0], t, nx);
    stage_load<NW>(in, img, y0, H, W, x0, t, nx);
    const int p0 = 32 * wv + (lane & 31);                // entry of the pixel left of this lane's pixel
    auto step = [&](int ir, f32x16& A, f32x16& Bm, f32x16& Cm) {
        __syncthreads();                                 // buffer ir & 1 complete, buffer (ir + 1) & 1 free
        bf16x8 f[3][2];
        frags32<S::NPP>(rows[ir & 1], p0, lane, f);
        if (ir + 2 < L + 2) stage_load<NW>(in, img, y0 + ir + 1, H, W, x0, t, nn);
        Cm = zero16();
        mid32_row(wa, f, A, Bm, Cm);
        const int yo = y0 + ir - 2;                      // the row A completes
        if (ir >= 2 && yo < H) store32<MODE>(A, bv, mask, out, img + (long)yo * W, xw, W, lane, relu, tiles[wv]);
        if (ir + 1 < L + 2) stage_store<NW>(rows[(ir + 1) & 1], t, nx);
        #pragma unroll
        for (int k = 0; k < S::K; ++k) nx[k] = nn[k];
    };
    for (int ir = 0; ir < L + 2; ir += 3) {
        step(ir, a0, a1, a2);
        if (ir + 1 < L + 2) step(ir + 1, a1, a2, a0);
        if (ir + 2 < L + 2) step(ir + 2, a2, a0, a1);
    }
}

// ---------------------------------------------------------------------------
// layer 5: y = xres + b + sum_t sum_ci a4[p + off_t][ci] w5[t][ci]   (fp32 out)
//
// As a 1x1 convolution on MFMA followed by a 3x3 sum on the VALU.  The FP32
// weights are split into w5 = hi + lo (hi = bf16(w5), lo = bf16(w5 - hi),
// about 16 significant bits together) and held as the 18 rows m = 2 t + h of
// a 32-row A operand (rows 18 .. 31 zero), so one v_mfma_f32_32x32x16_bf16
// pair per 32 pixels gives U[p][2 t + h] = sum_ci a4[p][ci] w5_h[t][ci] for
// all 9 taps; then S_h = sum over t = 0 .. 8 in order of U[p + off_t][2 t + h]
// and y = xres + (b + (S_0 + S_1)).  The layer-by-layer and the fused kernels
// both compute exactly this.
// ---------------------------------------------------------------------------
// A fragments (kc = 0, 1) of the split layer-5 weights
__device__ __forceinline__ void load_w5(const float* __restrict__ w, int lane, bf16x8 (&wa)[2])
{
    const int m = lane & 31, t = m >> 1;
    #pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
        uint32_t u[4];
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v[2];
            #pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int ci = 16 * kc + 8 * (lane >> 5) + 2 * e + q;
                const float wf = m < 18 ? w[t * 32 + ci] : 0.0f;
                const float hi = (float)(__bf16)wf;
                v[q] = (m & 1) ? wf - hi : hi;
            }
            u[e] = pack_bf16(v[0], v[1]);
        }
        wa[kc] = as_bf16x8(make_uint4(u[0], u[1], u[2], u[3]));
    }
}

// the U values (rows m < 18) of D on this lane into a U row [pixel][18]
__device__ __forceinline__ void put_u(const f32x16& U, float* __restrict__ urow, int p, int lane)
{
    #pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (m < 18) urow[p * 18 + m] = U[i];
    }
}

// S_0 + S_1 of the pixel whose left neighbour is entry p of the U rows
// r0 (row above), r1, r2 (row below)
__device__ __forceinline__ float sum_u(const float* __restrict__ r0, const float* __restrict__ r1,
                                       const float* __restrict__ r2, int p)
{
    const float* rr[3] = {r0, r1, r2};
    float s0 = 0.0f, s1 = 0.0f;
    #pragma unroll
    for (int t = 0; t < 9; ++t) {
        const float* u = rr[t / 3] + (p + t % 3) * 18 + 2 * t;
        s0 += u[0];
        s1 += u[1];
    }
    return s0 + s1;
}

// One wave: U for the 32 columns xw - 1 .. xw + 30 of each input row, outputs
// for the 30 columns xw .. xw + 29 of each of L rows (3 U rows in LDS).
template <int L>
__global__ __launch_bounds__(256) void k_conv_out(const uint16_t* __restrict__ a, const float* __restrict__ w,
                                                  float b5, const float* __restrict__ xres, float* __restrict__ y,
                                                  int H, int W)
{
    __shared__ float ur[4][3][32 * 18];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int n = lane & 31, h = lane >> 5;
    const int xw = (blockIdx.x * 4 + wv) * 30;
    const int col = xw - 1 + n;                         // this lane's U column
    const int y0 = blockIdx.y * L;
    const long img = (long)blockIdx.z * H * W;
    bf16x8 wa[2];
    load_w5(w, lane, wa);
    for (int ir = 0; ir < L + 2; ++ir) {
        const int yy = y0 + ir - 1;                     // input row
        bf16x8 f[2];
        #pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (yy >= 0 && yy < H && col >= 0 && col < W)
                v = *reinterpret_cast<const uint4*>(a + (img + (long)yy * W + col) * 32 + 16 * kc + 8 * h);
            f[kc] = as_bf16x8(v);
        }
        f32x16 U = mfma32(wa[0], f[0], zero16());
        U = mfma32(wa[1], f[1], U);
        put_u(U, ur[wv][ir % 3], n, lane);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int yo = yy - 1;
        if (ir >= 2 && yo < H && lane < 30 && xw + lane < W) {
            const float sv = sum_u(ur[wv][(ir + 1) % 3], ur[wv][(ir + 2) % 3], ur[wv][ir % 3], lane);
            const long q = img + (long)yo * W + xw + lane;
            y[q] = (xres ? xres[q] : 0.0f) + (b5 + sv);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

// ---------------------------------------------------------------------------
// The whole forward network in one launch (inference; no activation is kept).
//
// A workgroup computes a strip of 16 T computed columns (T tiles of 16
// pixels) over L output rows of one image, walking down the rows.  Each of
// its 4 waves owns layers: wave 0 the x rows and the 32 -> 1 output layer
// (MFMA), wave k = 1, 2, 3 the 32 -> 32 layer k + 1 (MFMA, its 72 VGPRs of
// weight fragments resident); wave 0 also runs the 1 -> 32 layer, on FP32
// MFMA.  They run as a row pipeline: at step s wave 0 writes a1 row
// y0 - 4 + s and wave k writes row y0 - 4 - 2k + s of its layer, each consuming the row its
// producer wrote at step s - 1 from a double-buffered LDS row (bf16,
// [channel group][pixel], 16 bytes per entry; pitch = 4 (mod 16) entries
// keeps the fragment reads and the row writes free of bank conflicts); one
// barrier per step; the output layer completes y row y0 - 12 + s.  Every
// stored value comes from the same operations in the same order as the
// layer-by-layer kernels (k_conv_in, k_conv_mid, k_conv_out: rolling
// accumulators over the three input rows, zero rows and columns outside the
// image), so the result is the same bits.  The strip's two edge columns see
// zero neighbours; that error moves one column inwards per 3x3 layer, so of
// the 16 T computed columns the middle 16 T - 8 are output (strips overlap by
// 8 columns), and the first 12 steps fill the pipeline.
// ---------------------------------------------------------------------------
template <int T>
struct FusedCnn {
    static constexpr int NP = 16 * T + 2;                        // pixels of a row incl. the zero halo
    static constexpr int NPP = NP + (((4 - NP) % 16) + 16) % 16;  // entry pitch of a channel group
    static constexpr int WO = 16 * T - 8;                         // output columns of a strip
};

template <int T>
__global__ __launch_bounds__(256, 2) void k_cnn_fwd(const float* __restrict__ x, const float* __restrict__ w1,
                                                   const float* __restrict__ b1, const uint16_t* __restrict__ w2,
                                                   const float* __restrict__ b2, const uint16_t* __restrict__ w3,
                                                   const float* __restrict__ b3, const uint16_t* __restrict__ w4,
                                                   const float* __restrict__ b4, const float* __restrict__ w5, float b5,
                                                   float* __restrict__ y, int H, int W, int nstrips, long total,
                                                   long per)
{
    using F = FusedCnn<T>;
    static_assert(T % 2 == 0, "32-pixel tiles of the 32 -> 32 layers");
    constexpr int NPP = F::NPP, NP = F::NP;
    __shared__ uint4 act[4][2][4 * NPP];     // rows of a1 .. a4
    __shared__ float xr[4][NP];              // x ring: rows y - 1, y, y + 1 of the a1 row and the next
    __shared__ float ur[3][NP * 18];         // U rows of the output layer (wave 0)
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    // The workgroup's rows: [blockIdx.x per, + per) of the (image, strip, row)
    // sequence, walked as segments of consecutive rows of one strip (a new
    // segment refills the pipeline).  Every wave runs the same segments.
    long i0 = (long)blockIdx.x * per;
    const long i1 = i0 + per < total ? i0 + per : total;
    int c0 = 0, y0 = 0, L = 0;               // first computed column, first row, rows of the segment
    long img = 0;
    auto next_segment = [&]() {
        if (i0 >= i1) return false;
        const long si = i0 / H;              // image * nstrips + strip
        y0 = (int)(i0 - si * H);
        L = (int)(i1 - i0 < (long)(H - y0) ? i1 - i0 : (long)(H - y0));
        c0 = (int)(si % nstrips) * F::WO - 4;
        img = (si / nstrips) * (long)H * W;
        i0 += L;
        __syncthreads();                     // the previous segment's last reads are done
        for (int i = t; i < 4 * 2 * 4 * NPP; i += 256) (&act[0][0][0])[i] = make_uint4(0, 0, 0, 0);
        return true;
    };

    // The 1 -> 32 layer on wave 0's matrix core, whose SIMD the 32 -> 32 layers
    // leave idle: per 32-pixel tile five v_mfma_f32_32x32x2f32 add taps 2 i
    // and 2 i + 1 to an accumulator that starts at the bias (tap 9 has weight
    // 0).  This is k_conv_in's arithmetic (z = b; z = fma(w[t], v[t], z) for
    // t = 0..8): the FP32 MFMA adds its two products in order with one
    // rounding each, the same bits as the FMA chain.  A lane holds w1[tap
    // 2 i + l / 32][co = l % 32] and the x value of that tap at pixel l % 32;
    // D is laid out as the 32 -> 32 layers' (channel 8 (r / 4) + 4 (l / 32) +
    // r % 4 of pixel l % 32 in register r).  At step s the a1 row y0 - 4 + s
    // uses x rows y0 - 5 + s .. y0 - 3 + s, in ring slots s % 4 .. (s + 2) % 4;
    // x row y0 - 2 + s goes into slot (s + 3) % 4 for the next step.
    if (wv == 0) {
        // ---- x rows, the 1 -> 32 layer and 32 -> 1 (1x1 MFMA + 3x3 sum, as k_conv_out) ----
        float wa1[5], ba1[16];
        {
            const int co = lane & 31, hk = lane >> 5;
            #pragma unroll
            for (int i = 0; i < 5; ++i) wa1[i] = 2 * i + hk < 9 ? w1[(2 * i + hk) * 32 + co] : 0.0f;
            #pragma unroll
            for (int r = 0; r < 16; ++r) ba1[r] = b1[8 * (r >> 2) + 4 * hk + (r & 3)];
        }
        auto conv_in_row = [&](int s) {
            const int r1 = y0 - 4 + s;
            uint2* a1w = reinterpret_cast<uint2*>(act[0][s & 1]);
            const int n = lane & 31, hk = lane >> 5;
            #pragma unroll
            for (int j = 0; j < T / 2; ++j) {
                const int pp = 32 * j + n;
                f32x16 z;
                #pragma unroll
                for (int r = 0; r < 16; ++r) z[r] = ba1[r];
                #pragma unroll
                for (int i = 0; i < 5; ++i) {
                    const int tp = 2 * i + hk;           // tap 3 dy + dx
                    const float v = tp < 9 ? xr[(s + tp / 3) & 3][pp + tp % 3] : 0.0f;
                    z = __builtin_amdgcn_mfma_f32_32x32x2f32(wa1[i], v, z, 0, 0, 0);
                }
                const int c = c0 + pp;
                const bool ok = r1 >= 0 && r1 < H && c >= 0 && c < W;
                #pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint2 ov = make_uint2(0, 0);
                    if (ok) {
                        ov.x = pack_bf16(fmaxf(z[4 * q], 0.0f), fmaxf(z[4 * q + 1], 0.0f));
                        ov.y = pack_bf16(fmaxf(z[4 * q + 2], 0.0f), fmaxf(z[4 * q + 3], 0.0f));
                    }
                    a1w[(q * NPP + pp + 1) * 2 + hk] = ov;
                }
            }
        };
        bf16x8 wa5[2];
        load_w5(w5, lane, wa5);
        // x rows: lane l holds columns c0 - 1 + l + 64 k of a row (zero outside the
        // image); each row is loaded one step before it enters the LDS ring, and
        // the residual values of the y row (columns c0 + l + 64 k) one step before
        // they are added
        constexpr int KX = (NP + 63) / 64;
        constexpr int KY = (16 * T + 63) / 64;
        auto fetch_x = [&](int row, float (&v)[KX]) {
            const bool rok = row >= 0 && row < H;
            #pragma unroll
            for (int k = 0; k < KX; ++k) {
                const int i = lane + 64 * k;
                const int c = c0 - 1 + i;
                v[k] = (rok && i < NP && c >= 0 && c < W) ? x[img + (long)row * W + c] : 0.0f;
            }
        };
        auto put_x = [&](int slot, const float (&v)[KX]) {
            #pragma unroll
            for (int k = 0; k < KX; ++k)
                if (lane + 64 * k < NP) xr[slot][lane + 64 * k] = v[k];
        };
        auto fetch_res = [&](int row, float (&v)[KY]) {
            #pragma unroll
            for (int k = 0; k < KY; ++k) {
                const int c = c0 + lane + 64 * k;
                v[k] = (row >= 0 && row < H && c >= 0 && c < W) ? x[img + (long)row * W + c] : 0.0f;
            }
        };
        float xn[KX], xres[KY];
        while (next_segment()) {
        for (int i = lane; i < 3 * NP * 18; i += 64) (&ur[0][0])[i] = 0.0f;
        fetch_x(y0 - 5, xn);
        put_x(0, xn);
        fetch_x(y0 - 4, xn);
        put_x(1, xn);
        fetch_x(y0 - 3, xn);
        put_x(2, xn);
        fetch_x(y0 - 2, xn);
        fetch_res(y0 - 12, xres);
        __syncthreads();
        // one pipeline step (U row y0 - 13 + s + dy of the output layer in ring
        // slot (s + 1 + dy) % 3; PH = s % 3)
        auto step = [&](auto ph, int s) {
            constexpr int PH = decltype(ph)::value;
            put_x((s + 3) & 3, xn);                     // x row y0 - 2 + s, for step s + 1
            fetch_x(y0 - 1 + s, xn);                    // for the step after
            conv_in_row(s);
            // output layer: U row of the a4 row y0 - 11 + s written at step s - 1,
            // then the 3x3 sum of y row y0 - 12 + s
            const uint4* a4r = act[3][(s + 1) & 1];
            const int n = lane & 31, h = lane >> 5;
            #pragma unroll
            for (int j = 0; j < T / 2; ++j) {
                const bf16x8 f0 = as_bf16x8(a4r[h * NPP + 32 * j + n + 1]);
                const bf16x8 f1 = as_bf16x8(a4r[(2 + h) * NPP + 32 * j + n + 1]);
                f32x16 U = mfma32(wa5[0], f0, zero16());
                U = mfma32(wa5[1], f1, U);
                put_u(U, ur[PH], 32 * j + n + 1, lane);
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const int ry = y0 - 12 + s;
            #pragma unroll
            for (int k = 0; k < KY; ++k) {
                const int pp = lane + 64 * k;           // computed column c0 + pp
                if (s >= 12 && ry < H && pp >= 4 && pp < 4 + F::WO && c0 + pp < W) {
                    const float sv = sum_u(ur[(PH + 1) % 3], ur[(PH + 2) % 3], ur[PH], pp);
                    y[img + (long)ry * W + c0 + pp] = xres[k] + (b5 + sv);
                }
            }
            fetch_res(ry + 1, xres);                    // for the next step
            __syncthreads();
        };
        for (int s = 0; s < L + 12; s += 3) {
            step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < L + 12) step(std::integral_constant<int, 1>{}, s + 1);
            if (s + 2 < L + 12) step(std::integral_constant<int, 2>{}, s + 2);
        }
        }
    } else {
        // ---- the 32 -> 32 layer wv + 1: relu(conv(a_wv) + b), T / 2 tiles of 32 pixels ----
        constexpr int T2 = T / 2;
        bf16x8 wa[9][2];
        load_w32(wv == 1 ? w2 : (wv == 2 ? w3 : w4), lane, wa);
        const float* bias = wv == 1 ? b2 : (wv == 2 ? b3 : b4);
        float bv[16];
        #pragma unroll
        for (int i = 0; i < 16; ++i) bv[i] = bias[8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)];
        const int n = lane & 31, h = lane >> 5;
        f32x16 m0[T2], m1[T2], m2[T2];
        while (next_segment()) {
        #pragma unroll
        for (int j = 0; j < T2; ++j) m0[j] = m1[j] = m2[j] = zero16();
        __syncthreads();
        // one pipeline step (accumulator roles rotate as in wave 0's steps)
        auto step = [&](int s, f32x16 (&A)[T2], f32x16 (&Bm)[T2], f32x16 (&Cm)[T2]) {
            const uint4* in = act[wv - 1][(s + 1) & 1];   // written at step s - 1
            uint2* ow = reinterpret_cast<uint2*>(act[wv][s & 1]);
            const int ro = y0 - 4 - 2 * wv + s;            // the row this step completes
            const bool rok = ro >= 0 && ro < H;
            // every tile's MFMAs first, then the completed rows
            #pragma unroll
            for (int j = 0; j < T2; ++j) {
                bf16x8 f[3][2];
                frags32<NPP>(in, 32 * j + n, lane, f);
                Cm[j] = zero16();
                mid32_row(wa, f, A[j], Bm[j], Cm[j]);
            }
            #pragma unroll
            for (int j = 0; j < T2; ++j) {
                // this lane holds channels 8 q + 4 h .. + 3 of pixel n of the tile
                const int c = c0 + 32 * j + n;
                const bool ok = rok && c >= 0 && c < W;
                #pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float z[4];
                    #pragma unroll
                    for (int e = 0; e < 4; ++e) z[e] = fmaxf(A[j][4 * q + e] + bv[4 * q + e], 0.0f);
                    uint2 ov = make_uint2(0, 0);
                    if (ok) { ov.x = pack_bf16(z[0], z[1]); ov.y = pack_bf16(z[2], z[3]); }
                    ow[(q * NPP + 32 * j + n + 1) * 2 + h] = ov;
                }
            }
            __syncthreads();
        };
        for (int s = 0; s < L + 12; s += 3) {
            step(s, m0, m1, m2);
            if (s + 1 < L + 12) step(s + 1, m1, m2, m0);
            if (s + 2 < L + 12) step(s + 2, m2, m0, m1);
        }
        }
    }
}

// layer-5 data gradient: dz4[p][ci] = (a4[p][ci] > 0) * sum_t dy[p - off_t] w5[t][ci]
__global__ __launch_bounds__(256) void k_out_dgrad(const float* __restrict__ dy, const float* __restrict__ w,
                                                   const uint16_t* __restrict__ a4, uint16_t* __restrict__ dz,
                                                   int B, int H, int W)
{
    __shared__ float sw[288];
    for (int i = threadIdx.x; i < 288; i += blockDim.x) sw[i] = w[i];
    __syncthreads();
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long npx = (long)B * H * W;
    if (p >= npx) return;
    const int xw = (int)(p % W), yh = (int)((p / W) % H);
    const long base = p - (long)yh * W - xw;
    float g[9];
    #pragma unroll
    for (int t = 0; t < 9; ++t) {
        // output pixel q = p - off_t receives a4[p] through tap t
        const int yy = yh - (t / 3 - 1), xx = xw - (t % 3 - 1);
        g[t] = (yy >= 0 && yy < H && xx >= 0 && xx < W) ? dy[base + (long)yy * W + xx] : 0.0f;
    }
    const uint4* am = reinterpret_cast<const uint4*>(a4 + p * 32);
    uint4* o = reinterpret_cast<uint4*>(dz + p * 32);
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint4 m = am[q];
        const uint32_t mu[4] = {m.x, m.y, m.z, m.w};
        uint32_t r[4];
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            float z[2];
            #pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int c = 8 * q + 2 * e + h;
                float s = 0.0f;
                #pragma unroll
                for (int t = 0; t < 9; ++t) s = fmaf(sw[t * 32 + c], g[t], s);
                const uint16_t mk = h ? (uint16_t)(mu[e] >> 16) : (uint16_t)(mu[e] & 0xffff);
                z[h] = bf2f(mk) > 0.0f ? s : 0.0f;
            }
            r[e] = pack_bf16(z[0], z[1]);
        }
        o[q] = make_uint4(r[0], r[1], r[2], r[3]);
    }
}

// ---------------------------------------------------------------------------
// weight gradients of the narrow layers (reduction over pixels, FP32 MFMA):
// mode 0 (layer 1): part[t][c] = sum_p x[p + off_t] dz1[p][c], part[9][c] = sum_p dz1[p][c]
// mode 1 (layer 5): part[t][c] = sum_p dy[p] a4[p + off_t][c] = sum_q a4[q][c] dy[q - off_t],
//                   part[9][0] = sum_p dy[p]
//
// Both are products of the 32-channel tensor's columns with the image's 9
// shifts, K = pixels: v_mfma_f32_16x16x4f32 takes 4 adjacent pixels, A = 16
// channels (lane l: channel pair l % 16 of pixel l / 16, one 4-byte load whose
// halves feed an even-channel and an odd-channel tile, widened to FP32
// exactly), B = the shifts (lane l: shift l % 16 of that pixel; column 9 is 1
// and gives the channel sums, columns 10 .. 15 are 0).  Nothing is rounded
// below FP32 and no LDS is needed.  A wave takes 64 pixels of one image row at
// a time, 16 steps whose loads are independent.
//
// Bound: the 64 bytes per pixel of the tensor, read once: 89 us for 16 x 512^2
// (3.0 TB/s; 56 us at the 4.8 TB/s of a large copy, the two matrix tiles alone
// 27 us).  With 32 lanes of 2-byte loads and 10 FMAs per pixel: 1.60 ms.
// ---------------------------------------------------------------------------
typedef uint32_t U32a2 __attribute__((aligned(2)));   // a channel pair: 2-byte aligned like the tensor

constexpr int kNarrowPx = 64;          // pixels of a wave's chunk

__global__ __launch_bounds__(256) void k_wgrad_narrow(const float* __restrict__ img, const uint16_t* __restrict__ act,
                                                      float* __restrict__ part, int H, int W, int chunks_per_row,
                                                      int nchunk, int mode)
{
    __shared__ float red[4][320];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n = lane & 15, k = lane >> 4;
    // shift of column n (mode 1 reads the image at q - off_t)
    const int sg = mode == 0 ? 1 : -1;
    const int oy = n < 9 ? sg * (n / 3 - 1) : 0, ox = n < 9 ? sg * (n % 3 - 1) : 0;
    const uint32_t fixed = n == 9 ? 0x3f800000u : 0u;               // 1.0f
    f32x4 ev = f32x4{0, 0, 0, 0}, od = f32x4{0, 0, 0, 0};
    float sum = 0.0f;                  // lanes n = 4 (shift 0): the image's sum
    for (int ch = (int)blockIdx.x * 4 + wv; ch < nchunk; ch += (int)gridDim.x * 4) {
        const int row = ch / chunks_per_row;                        // image * H + y
        const int c0 = (ch - row * chunks_per_row) * kNarrowPx;
        const int y = row % H + oy;
        const bool rok = y >= 0 && y < H, tap = n < 9 && rok;
        const float* src = img + (long)(rok ? row + oy : row) * W;  // the shift's image row
        const uint16_t* a = act + (long)row * W * 32 + 2 * n;
        // loads without branches (columns clamped into the row, dropped by
        // selects), 8 steps in flight
        #pragma unroll
        for (int s0 = 0; s0 < kNarrowPx / 4; s0 += 8) {
            if (c0 + 4 * s0 >= W) break;
            uint32_t u[8];
            float v[8];
            #pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int px = c0 + 4 * (s0 + s) + k;
                u[s] = *reinterpret_cast<const U32a2*>(a + (long)min(px, W - 1) * 32);
                v[s] = src[min(max(px + ox, 0), W - 1)];
            }
            #pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int px = c0 + 4 * (s0 + s) + k;
                const bool in = px < W;
                // masks, not selects: a select would sink its load under a branch
                const uint32_t inside = in ? 0xffffffffu : 0u;
                const uint32_t mok = (in && tap && px + ox >= 0 && px + ox < W) ? 0xffffffffu : 0u;
                const uint32_t w = u[s] & inside;
                const float f = __uint_as_float((__float_as_uint(v[s]) & mok) | (fixed & inside));
                sum += f;
                ev = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w << 16), f, ev, 0, 0, 0);
                od = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w & 0xffff0000u), f, od, 0, 0, 0);
            }
        }
    }
    // D on lane l, register i: shift l % 16, channel pair 4 (l / 16) + i
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (n < 10) {
            red[wv][n * 32 + 2 * (4 * k + i)] = ev[i];
            red[wv][n * 32 + 2 * (4 * k + i) + 1] = od[i];
        }
    }
    // A NaN or an infinity in the tensor times the zero of a tap off the image is not that
    // tap's: such sums are made again without those products (one lane per channel and
    // pixel parity).
    bool bad = false;
    #pragma unroll
    for (int i = 0; i < 4; ++i) bad = bad || !(fabsf(ev[i]) < INFINITY) || !(fabsf(od[i]) < INFINITY);
    if (__any(bad && n < 9)) {
        const int c = lane & 31;
        float s[9];
        #pragma unroll
        for (int t = 0; t < 9; ++t) s[t] = 0.0f;
        for (int ch = (int)blockIdx.x * 4 + wv; ch < nchunk; ch += (int)gridDim.x * 4) {
            const int row = ch / chunks_per_row, c0 = (ch - row * chunks_per_row) * kNarrowPx, y = row % H;
            for (int x = c0 + (lane >> 5); x < min(c0 + kNarrowPx, W); x += 2) {
                const float d = bf2f(act[((long)row * W + x) * 32 + c]);
                #pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const int dy = sg * (t / 3 - 1), dx = sg * (t % 3 - 1);
                    if (y + dy >= 0 && y + dy < H && x + dx >= 0 && x + dx < W)
                        s[t] = fmaf(img[(long)(row + dy) * W + x + dx], d, s[t]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        #pragma unroll
        for (int t = 0; t < 9; ++t) {
            s[t] += __shfl_xor(s[t], 32);
            float& r = red[wv][t * 32 + c];
            if (lane < 32 && !(fabsf(r) < INFINITY)) r = s[t];
        }
    }
    if (mode != 0) {
        // the image's sum over the four pixel groups of the shift-0 lanes, in place of the channel sums
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (lane == 4) red[wv][288] = sum;
    }
    __syncthreads();
    const int no = mode == 0 ? 320 : 289;       // the gradient's entries
    for (int i = threadIdx.x; i < no; i += 256)
        part[(long)blockIdx.x * no + i] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
}

// bias gradient of a 32-channel NHWC tensor: part[wg][c] = sum_p dz[p][c]
__global__ __launch_bounds__(256) void k_bias_grad(const uint16_t* __restrict__ dz, float* __restrict__ part, long npx)
{
    __shared__ float red[8][32];
    const int c = threadIdx.x & 31, grp = threadIdx.x >> 5;
    float s = 0.0f;
    for (long p = (long)blockIdx.x * 8 + grp; p < npx; p += (long)gridDim.x * 8) s += bf2f(dz[p * 32 + c]);
    red[grp][c] = s;
    __syncthreads();
    if (threadIdx.x < 32) {
        float t = 0.0f;
        for (int gidx = 0; gidx < 8; ++gidx) t += red[gidx][threadIdx.x];
        part[(long)blockIdx.x * 32 + threadIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------
// 32 -> 32 weight gradient on MFMA, with the layer's bias gradient:
//   dW[t][co][ci] = sum_p dz[p][co] in[p + off_t][ci],  db[co] = sum_p dz[p][co]
// GEMM with M = co, N = ci, K = pixels (v_mfma_f32_32x32x16_bf16).  A wave
// walks L rows of a 32-column strip.  Per step it stages one input row (34
// pixels) and one dz row (32 pixels) as they lie in memory, 64 bytes per pixel,
// in its own LDS rows; both operands need 8 pixels of one channel per lane, and
// ds_read_b64_tr_b16 delivers exactly that from the staged rows (a group of 16
// lanes reads 4 pixels x 16 channels and gets it transposed), so a tap's column
// shift is only another first pixel and nothing is copied or transposed by
// VALU work.  The dz fragments of three rows stay in registers, so each staged
// row feeds all 9 taps.  The next row is loaded into registers while this one
// is used.  No barrier: a wave touches only its own rows.
//
// Bound: one pass over both tensors: 125 us for 16 x 512^2 (4.3 TB/s; 112 us at
// the 4.8 TB/s of a large copy, the matrix cores need 36 us).  With nine shifted transposed
// copies written to LDS 2 bytes at a time it took 0.51 ms, and the bias
// gradient another 0.22 ms in a kernel of its own.
// ---------------------------------------------------------------------------
constexpr int kWgIn = 34 * 32, kWgDz = 32 * 32;          // bf16 elements of a wave's staged rows
constexpr int kWgOut = 9 * 1024 + 32;                    // gradient entries of a partial

typedef short s16x4 __attribute__((ext_vector_type(4)));

// 16 pixels x 32 channels from LDS rows of 32 channels, transposed: this lane
// holds channel lane % 32 of pixels 8 (lane / 32) .. + 7.  `row` points at the
// lane's own read address within the first pixel's row (tr_lane).
__device__ __forceinline__ bf16x8 tr_frag(const uint16_t* row)
{
    typedef __attribute__((address_space(3))) s16x4 Lds;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds*)row);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds*)(row + 4 * 32));
    const short v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    bf16x8 r;
    __builtin_memcpy(&r, v, sizeof(r));
    return r;
}

// element offset of a lane's read: pixel 8 (lane / 32) + (lane % 16) / 4, channels 16 ((lane / 16) % 2) + 4 (lane % 4) ..
__device__ __forceinline__ int tr_lane(int lane)
{
    return (8 * (lane >> 5) + ((lane & 15) >> 2)) * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
}

__global__ __launch_bounds__(256, 2) void k_wgrad_mid(const uint16_t* __restrict__ in, const uint16_t* __restrict__ dz,
                                                      float* __restrict__ part, int H, int W, int L, int nxs, int nys,
                                                      int nitems)
{
    constexpr int kStage = 4 * (kWgIn + kWgDz) * (int)sizeof(uint16_t), kRed = kWgOut * (int)sizeof(float);
    __shared__ __align__(16) char smem[kStage > kRed ? kStage : kRed];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint16_t* inS = reinterpret_cast<uint16_t*>(smem) + wv * (kWgIn + kWgDz);   // [34 px][32 ci]
    uint16_t* dzS = inS + kWgIn;                                               // [32 px][32 co]
    const int tl = tr_lane(lane);
    f32x16 acc[9], accb = zero16();
    #pragma unroll
    for (int t = 0; t < 9; ++t) acc[t] = zero16();
    bf16x8 ones;
    #pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.0f;
    const int px = lane >> 2, c8 = 8 * (lane & 3);        // this lane's 16-byte chunk of 16 pixels
    for (int it = (int)blockIdx.x * 4 + wv; it < nitems; it += (int)gridDim.x * 4) {
        const int ys = it % nys, t = it / nys, xs = t % nxs;
        const int x0 = xs * 32, y0 = ys * L, y1 = min(y0 + L, H);
        const long img = (long)(t / nxs) * H * W;
        uint4 vi[3], vd[2];
        // input row r (zero outside the image) and dz row r + 1 (zero outside this item's rows)
        auto load = [&](int r) {
            const bool rok = r >= 0 && r < H, dok = r + 1 >= y0 && r + 1 < y1;
            #pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int x = x0 - 1 + px + 16 * k;
                vi[k] = make_uint4(0, 0, 0, 0);
                if (rok && x >= 0 && x < W && px + 16 * k < 34)
                    vi[k] = *reinterpret_cast<const uint4*>(in + (img + (long)r * W + x) * 32 + c8);
            }
            #pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int x = x0 + px + 16 * k;
                vd[k] = make_uint4(0, 0, 0, 0);
                if (dok && x < W) vd[k] = *reinterpret_cast<const uint4*>(dz + (img + (long)(r + 1) * W + x) * 32 + c8);
            }
        };
        bf16x8 d0[2], d1[2], d2[2];      // dz rows r - 1, r, r + 1: pixels 0 .. 15 and 16 .. 31
        #pragma unroll
        for (int kc = 0; kc < 2; ++kc) d0[kc] = d1[kc] = as_bf16x8(make_uint4(0, 0, 0, 0));
        load(y0 - 1);
        for (int r = y0 - 1; r <= y1; ++r) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            #pragma unroll
            for (int k = 0; k < 3; ++k)
                if (px + 16 * k < 34) *reinterpret_cast<uint4*>(inS + (px + 16 * k) * 32 + c8) = vi[k];
            #pragma unroll
            for (int k = 0; k < 2; ++k) *reinterpret_cast<uint4*>(dzS + (px + 16 * k) * 32 + c8) = vd[k];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (r < y1) load(r + 1);
            #pragma unroll
            for (int kc = 0; kc < 2; ++kc) {
                d2[kc] = tr_frag(dzS + 16 * kc * 32 + tl);
                accb = mfma32(d2[kc], ones, accb);
            }
            // (dz rows of this item only: a zero in the others' place would turn a NaN or an
            // infinity of the input row into a tap's that has no such product)
            bf16x8 f[3][2];
            #pragma unroll
            for (int dx = 0; dx < 3; ++dx)
                #pragma unroll
                for (int kc = 0; kc < 2; ++kc) f[dx][kc] = tr_frag(inS + (16 * kc + dx) * 32 + tl);
            auto taps = [&](f32x16* a, const bf16x8 (&d)[2]) {
                #pragma unroll
                for (int dx = 0; dx < 3; ++dx)
                    #pragma unroll
                    for (int kc = 0; kc < 2; ++kc) a[dx] = mfma32(d[kc], f[dx][kc], a[dx]);
            };
            if (r + 1 < y1) taps(acc, d2);                          // input row above the dz row
            if (r >= y0 && r < y1) taps(acc + 3, d1);
            if (r > y0) taps(acc + 6, d0);                          // below
            #pragma unroll
            for (int kc = 0; kc < 2; ++kc) {
                d0[kc] = d1[kc];
                d1[kc] = d2[kc];
            }
        }
    }
    // the four waves' sums in LDS, wave after wave (a fixed order), then one partial per workgroup;
    // D on this lane, register i: co = 8 (i / 4) + 4 (lane / 32) + i % 4, ci = lane % 32
    float* red = reinterpret_cast<float*>(smem);
    for (int w = 0; w < 4; ++w) {
        __syncthreads();
        if (w != wv) continue;
        #pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int co = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            #pragma unroll
            for (int t = 0; t < 9; ++t) {
                float& q = red[t * 1024 + co * 32 + (lane & 31)];
                q = w == 0 ? acc[t][i] : q + acc[t][i];
            }
            if ((lane & 31) == 0) {
                float& q = red[9 * 1024 + co];
                q = w == 0 ? accb[i] : q + accb[i];
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kWgOut; i += 256) part[(long)blockIdx.x * kWgOut + i] = red[i];
}

// out[i] = sum_r part[r][i]: a workgroup takes 32 adjacent columns (128-byte
// row segments) with its 1024 threads as 32 row groups of 8 loads in flight,
// whose sums are added in LDS in a fixed order: 512 rows of 9248 in 5.0 us (3.8
// TB/s), 1024 rows of 320 in 4.6.  One thread per column walking the rows left at
// most 36 workgroups, each waiting on one load at a time.
constexpr int kRedCols = 32, kRedGroups = 32;

// Columns n0 and up go to out2 (the bias behind a layer's weights; dropped if null).
__global__ __launch_bounds__(kRedCols * kRedGroups) void k_reduce_rows(const float* __restrict__ part,
                                                                       float* __restrict__ out, int nrows, int n,
                                                                       int n0, float* __restrict__ out2)
{
    __shared__ float red[kRedGroups][kRedCols];
    const int c = threadIdx.x % kRedCols, grp = threadIdx.x / kRedCols;
    const int i = blockIdx.x * kRedCols + c;
    float s = 0.0f;
    if (i < n) {
        #pragma unroll 8
        for (int r = grp; r < nrows; r += kRedGroups) s += part[(long)r * n + i];
    }
    red[grp][c] = s;
    __syncthreads();
    if (grp != 0 || i >= n) return;
    float t = 0.0f;
    #pragma unroll
    for (int g = 0; g < kRedGroups; ++g) t += red[g][c];
    if (i < n0) out[i] = t;
    else if (out2 != nullptr) out2[i - n0] = t;
}

void reduce_rows(const float* part, float* out, int nrows, int n, hipStream_t st, int n0 = -1, float* out2 = nullptr)
{
    hipLaunchKernelGGL(k_reduce_rows, dim3((unsigned)cdiv(n, kRedCols)), dim3(kRedCols * kRedGroups), 0, st, part,
                       out, nrows, n, n0 < 0 ? n : n0, out2);
    check_launch("reduce_rows");
}

constexpr int kNConvMid = 5;

int grid_for(long work, int per_block, int cap)
{
    long g = (work + per_block - 1) / per_block;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (int)g;
}

} // namespace

void conv_in(const float* x, const float* w, const float* b, uint16_t* out, int B, int H, int W, hipStream_t st)
{
    RN_REQUIRE(B > 0 && H > 0 && W > 0, "conv_in: bad batch or image size");
    const int tiles = cdiv(W, kConvInTile);
    const long nwaves = (long)B * H * tiles;
    RN_REQUIRE(nwaves / 4 < 0x7fffffffL, "conv_in: batch too large for one launch");
    hipLaunchKernelGGL(k_conv_in, dim3((unsigned)cdiv(nwaves * 64, 256)), dim3(256), 0, st, x, w, b, out, H, W, tiles,
                       nwaves);
    check_launch("conv_in");
}

void conv_mid(const uint16_t* in, const uint16_t* wt, const float* bias, const uint16_t* mask, uint16_t* out,
              int B, int H, int W, bool relu, hipStream_t st)
{
    RN_REQUIRE(mask != nullptr || bias != nullptr, "conv_mid needs a bias (forward) or a mask (data gradient)");
    RN_REQUIRE(B > 0 && H > 0 && W > 0 && B <= 65535, "conv_mid: bad batch or image size");
    const int rl = relu ? 1 : 0;
    // candidates: workgroups of 2, 4 or 8 waves of 32 columns, 16 or 32 rows
    auto launch = [&](int c) {
        auto go = [&](auto kern, int nw, int rows) {
            const dim3 grd((unsigned)cdiv(W, 32 * nw), (unsigned)cdiv(H, rows), (unsigned)B);
            hipLaunchKernelGGL(kern, grd, dim3(64 * nw), 0, st, in, wt, bias, mask, out, H, W, rl);
        };
        if (c == 0) mask ? go(k_conv_mid<16, 1, 4>, 4, 16) : go(k_conv_mid<16, 0, 4>, 4, 16);
        else if (c == 1) mask ? go(k_conv_mid<16, 1, 2>, 2, 16) : go(k_conv_mid<16, 0, 2>, 2, 16);
        else if (c == 2) mask ? go(k_conv_mid<32, 1, 4>, 4, 32) : go(k_conv_mid<32, 0, 4>, 4, 32);
        else if (c == 3) mask ? go(k_conv_mid<32, 1, 2>, 2, 32) : go(k_conv_mid<32, 0, 2>, 2, 32);
        else mask ? go(k_conv_mid<16, 1, 8>, 8, 16) : go(k_conv_mid<16, 0, 8>, 8, 16);
        check_launch("conv_mid");
    };
    const int c = tune_choose({TK_CONV_MID, B, H, W, mask ? 1 : 0, rl}, kNConvMid, launch, st, true);
    launch(c);
}

void conv_out(const uint16_t* a4, const float* w5, float b5, const float* xres, float* y, int B, int H, int W,
              hipStream_t st)
{
    RN_REQUIRE(B > 0 && H > 0 && W > 0 && B <= 65535, "conv_out: bad batch or image size");
    constexpr int kRows = 16;
    const dim3 grd((unsigned)cdiv(W, 4 * 30), (unsigned)cdiv(H, kRows), (unsigned)B);
    hipLaunchKernelGGL(k_conv_out<kRows>, grd, dim3(256), 0, st, a4, w5, b5, xres, y, H, W);
    check_launch("conv_out");
}

void cnn_forward(const float* x, const float* w1, const float* b1, const uint16_t* w2, const float* b2,
                 const uint16_t* w3, const float* b3, const uint16_t* w4, const float* b4, const float* w5, float b5,
                 float* y, int B, int H, int W, hipStream_t st)
{
    RN_REQUIRE(B > 0 && H > 0 && W > 0, "cnn_forward: bad batch or image size");
    int dev = 0, ncu = 0;
    RN_HIP_CHECK(hipGetDevice(&dev));
    RN_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    // candidates: strips of T = 4 or 6 tiles of 16 columns; the (image, strip,
    // row) sequence cut into equal shares for 2 workgroups per CU (one round),
    // or into shares of 128 or 64 rows
    auto launch = [&](int c) {
        auto go = [&](auto kern, int wo, long per_rows) {
            const int nstrips = cdiv(W, wo);
            const long total = (long)B * nstrips * H;
            const long per = per_rows > 0 ? per_rows : (total + 2L * ncu - 1) / (2L * ncu);
            const long nwg = (total + per - 1) / per;
            RN_REQUIRE(nwg <= 0x7fffffffL, "cnn_forward: grid too large");
            hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(256), 0, st, x, w1, b1, w2, b2, w3, b3, w4, b4, w5, b5,
                               y, H, W, nstrips, total, per);
        };
        if (c == 0) go(k_cnn_fwd<4>, FusedCnn<4>::WO, 0);
        else if (c == 1) go(k_cnn_fwd<6>, FusedCnn<6>::WO, 0);
        else if (c == 2) go(k_cnn_fwd<4>, FusedCnn<4>::WO, 128);
        else go(k_cnn_fwd<4>, FusedCnn<4>::WO, 64);
        check_launch("cnn_forward");
    };
    const int c = tune_choose({TK_CNN_FWD, B, H, W, 0, 0}, 4, launch, st, true);
    launch(c);
}

void conv_out_dgrad(const float* dy, const float* w5, const uint16_t* a4, uint16_t* dz4, int B, int H, int W,
                    hipStream_t st)
{
    const long npx = (long)B * H * W;
    hipLaunchKernelGGL(k_out_dgrad, dim3(cdiv(npx, 256)), dim3(256), 0, st, dy, w5, a4, dz4, B, H, W);
    check_launch("conv_out_dgrad");
}

void wgrad_narrow(const float* img, const uint16_t* act, float* grad, int B, int H, int W, int mode, DevBuf& work,
                  hipStream_t st)
{
    const int chunks_per_row = cdiv(W, kNarrowPx);
    RN_REQUIRE(B > 0 && H > 0 && W > 0 && (long)B * H * chunks_per_row + 4096 < 0x7fffffffL,
               "wgrad_narrow: bad batch or image size");
    const int nchunk = B * H * chunks_per_row;
    // 4 workgroups per CU (16 waves of 16 loads in flight each), whole rounds of chunks
    const int blocks = grid_for(nchunk, 4, 1024);
    work.ensure((size_t)blocks * 320 * sizeof(float));
    hipLaunchKernelGGL(k_wgrad_narrow, dim3(blocks), dim3(256), 0, st, img, act, work.as<float>(), H, W,
                       chunks_per_row, nchunk, mode);
    check_launch("wgrad_narrow");
    reduce_rows(work.as<float>(), grad, blocks, mode == 0 ? 320 : 289, st);
}

void bias_grad(const uint16_t* dz, float* grad, long npx, DevBuf& work, hipStream_t st)
{
    const int blocks = grid_for(npx, 8 * 64, 1024);
    work.ensure((size_t)blocks * 32 * sizeof(float));
    hipLaunchKernelGGL(k_bias_grad, dim3(blocks), dim3(256), 0, st, dz, work.as<float>(), npx);
    check_launch("bias_grad");
    reduce_rows(work.as<float>(), grad, blocks, 32, st);
}

void wgrad_mid(const uint16_t* in, const uint16_t* dz, float* grad, float* gbias, int B, int H, int W, DevBuf& work,
               hipStream_t st)
{
    const int nxs = cdiv(W, 32);
    RN_REQUIRE(B > 0 && H > 0 && W > 0 && (long)B * nxs * H < (1L << 30), "wgrad_mid: bad batch or image size");
    // rows per item: one round of 2048 waves (2 per SIMD) where the batch has
    // that many strips of at least 8 rows, at most 64 rows (the two halo rows
    // of an item are read twice)
    const int L = (int)std::min<long>(64, std::max<long>(8, ((long)B * nxs * H + 2047) / 2048));
    const int nys = cdiv(H, L);
    const int nitems = B * nxs * nys;
    const int blocks = grid_for(nitems, 4, 512);
    work.ensure((size_t)blocks * kWgOut * sizeof(float));
    hipLaunchKernelGGL(k_wgrad_mid, dim3(blocks), dim3(256), 0, st, in, dz, work.as<float>(), H, W, L, nxs, nys,
                       nitems);
    check_launch("wgrad_mid");
    reduce_rows(work.as<float>(), grad, blocks, kWgOut, st, 9216, gbias);
}

} // namespace rn
