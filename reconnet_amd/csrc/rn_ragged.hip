// Persistent projector launches over a batch of 2D fan slices of uneven size
// (no reference counterpart: the reference ABI takes one geometry per call).
//
// Each slice has its own geometry, angle set and trig tables.  One launch of a
// fixed grid serves the whole batch: every wave repeatedly takes the next work
// item from a global counter (a 64-bin strip of one view for the FP, an 8 x 8
// pixel tile for the BP), finds its descriptor and runs the same per-ray /
// per-pixel code as the single-geometry kernels, so the results are identical
// to independent per-slice launches.  Consecutive slices of one geometry and
// angle set share a descriptor, up to kRagS of them: a lane then carries the
// ray or pixel through all of them, its geometry work done once (each slice
// with the arithmetic of a one-slice call; the forward projection takes a
// group in chunks of kRagFp).  Descriptors are ordered by
// decreasing cost so the heaviest start first.  Every wave leaves the loop once
// the counter passes the item total.

#include "rn_ragged.h"

#include "rn_fan_device.h"

#include <algorithm>
#include <numeric>

namespace rn {

namespace {

using namespace fan;

constexpr int kRagS = 8;    // slices of one geometry per backprojection descriptor
constexpr int kRagFp = 4;   // per forward descriptor (a group's chunks): the ray
                            // loops carry fewer registers and the launch more items
constexpr int kRagSidBp = 4;   // per Siddon backprojection descriptor (the same)

struct RagSlice {
    FanK g;
    const float* pa;     // FP: RX (DD) or Pyx (Siddon); BP: prj [nview][nu]
    const float* pb;     // FP: RY (DD) or Pxy (Siddon)
    float* out;          // FP: prj [nu][nview]; BP: img [nx][ny]
    int item0, tiles, nitems, nsl;   // nsl consecutive slices, nx * ny (image) / nu * nview (sinogram) apart
};

__device__ __forceinline__ int find_slice(const RagSlice* __restrict__ sl, int nsl, int item)
{
    int s = 0;
    while (s + 1 < nsl && sl[s + 1].item0 <= item) ++s;
    return s;
}

__device__ __forceinline__ int next_item(int* counter, int lane)
{
    int it = 0;
    if (lane == 0) it = atomicAdd(counter, 1);
    return __shfl(it, 0);
}

__global__ __launch_bounds__(256) void k_ragged_fp(const RagSlice* __restrict__ sl, int nsl, int total,
                                                   int* __restrict__ counter, int siddon)
{
    const int lane = threadIdx.x & 63;
    for (;;) {
        const int item = next_item(counter, lane);
        if (item >= total) break;
        const RagSlice& d = sl[find_slice(sl, nsl, item)];
        const int local = item - d.item0;
        const int view = local / d.tiles, iu = (local % d.tiles) * 64 + lane;
        const bool active = iu < d.g.nu;
        const long plane = (long)d.g.nx * d.g.ny, sino = (long)d.g.nu * d.g.nview;
        // every lane takes part (wave-uniform line loops)
        float acc[kRagFp];
        if (siddon)
            siddon_fp_ray_slices<float, kRagFp>(d.g, d.pa, d.pb, plane, d.nsl, view, active ? iu : d.g.nu - 1, active,
                                                acc);
        else
            dd_fp_ray_slices<float, kRagFp>(d.g, d.pa, d.pb, plane, d.nsl, view, active ? iu : d.g.nu - 1, active,
                                            acc);
        if (active) {
            #pragma unroll
            for (int q = 0; q < kRagFp; ++q)
                if (q < d.nsl) d.out[q * sino + (long)iu * d.g.nview + view] = acc[q];
        }
    }
}

// The next item of a workgroup.  (Every wave has read `next` before the barriers of
// add_waves, which thread 0 passes before it writes the next one.)
__device__ __forceinline__ int next_tile(int* counter, int* next, int lane, int wv)
{
    if (lane == 0 && wv == 0) *next = atomicAdd(counter, 1);
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*next);
}

// Siddon BP: pa holds the descriptor's kRagSidBp slices as one interleaved group; a
// workgroup takes one tile, its kBpSegs waves one view segment each, with the arithmetic
// of k_siddon_fan_bp_tile1 (FanK::tile) or k_siddon_fan_bp, and adds the segments' sums
// in order.
__global__ __launch_bounds__(64 * kBpSegs) void k_ragged_siddon_bp(const RagSlice* __restrict__ sl, int nsl, int total,
                                                                   int* __restrict__ counter)
{
    static_assert(kRagSidBp == 4, "one group per descriptor");
    __shared__ float4 red[64];
    __shared__ int next;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    for (;;) {
        const int item = next_tile(counter, &next, lane, wv);
        if (item >= total) break;
        const RagSlice& d = sl[__builtin_amdgcn_readfirstlane(find_slice(sl, nsl, item))];
        const int local = item - d.item0;
        const int tx = (local / d.tiles) * 8, ty = (local % d.tiles) * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7);
        const bool inside = ix < d.g.nx && iy < d.g.ny;
        const int v0 = (int)((long)d.g.nview * wv / kBpSegs), v1 = (int)((long)d.g.nview * (wv + 1) / kBpSegs);
        const float4* P = reinterpret_cast<const float4*>(d.pa);
        float4 acc[1] = {vzero<float4>()};
        if (d.g.tile)
            siddon_bp_tile1<2>(d.g, P, 0, v0, v1, tx, ty, lane, acc);
        else if (inside)
            siddon_bp_pixel_slices<float4, 4, 1>(d.g, P + (long)v0 * d.g.nu, 0, 1, v0, v1 - v0, ix, iy, acc);
        if (add_waves<1>(acc, red, lane, wv, kBpSegs) && inside) {
            const long plane = (long)d.g.nx * d.g.ny;
            const float v[4] = {acc[0].x, acc[0].y, acc[0].z, acc[0].w};
            #pragma unroll
            for (int c = 0; c < 4; ++c)
                if (c < d.nsl) d.out[c * plane + (long)ix * d.g.ny + iy] = v[c];
        }
    }
}

// DD adjoint: pa holds the descriptor's kRagS slices as kRagS / 4 interleaved
// groups (multiplied by the rays' length per line); a workgroup takes one tile, its
// kBpSegs waves one view segment each (dd_adj_tile), and adds the segments' sums
// in order.  WIDE: FanK::dwide of the launch's descriptors.
//
// Bound: as k_dd_fan_adj.  6 slices of 256^2 with 360 views, 6 of 384^2 with 720 and 4
// of 512^2 with 1152: 1.84 ms, 2.4 with one wave per tile and all its views (the queue
// then ended in a tail of 1152-view items).  80 registers let three workgroups share a
// CU (81: two, 2.35 ms).
template <bool WIDE>
__global__ __launch_bounds__(64 * kBpSegs, WIDE ? 6 : 4) void k_ragged_dd_adj(const RagSlice* __restrict__ sl, int nsl,
                                                                      int total, int* __restrict__ counter)
{
    constexpr int G = kRagS / 4, CAP = 32;
    __shared__ float4 stage[kBpSegs * DdAdjStage<G, CAP>::kFloat4];
    __shared__ float4 red[G * 64];
    __shared__ int next;
    const int lane = threadIdx.x, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    float4* st = stage + wv * DdAdjStage<G, CAP>::kFloat4;
    for (;;) {
        const int item = next_tile(counter, &next, lane, wv);
        if (item >= total) break;
        const RagSlice& d = sl[__builtin_amdgcn_readfirstlane(find_slice(sl, nsl, item))];
        const int local = item - d.item0;
        const int tx = (local / d.tiles) * 8, ty = (local % d.tiles) * 8, ix = tx + (lane >> 3), iy = ty + (lane & 7);
        const long plane = (long)d.g.nx * d.g.ny, sino = (long)d.g.nu * d.g.nview;
        float4 tot[G];
        dd_adj_tile<G, CAP, 3, WIDE>(d.g, reinterpret_cast<const float4*>(d.pa), sino, (d.nsl + 3) / 4, d.g.nview, wv,
                                     tx, ty, lane, st, tot);
        if (add_waves<G>(tot, red, lane, wv, kBpSegs) && ix < d.g.nx && iy < d.g.ny) {
            #pragma unroll
            for (int k = 0; k < G; ++k) {
                const float v[4] = {tot[k].x, tot[k].y, tot[k].z, tot[k].w};
                #pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (4 * k + c < d.nsl) d.out[(4 * k + c) * plane + (long)ix * d.g.ny + iy] = v[c];
            }
        }
    }
}

__global__ void k_zero_int(int* p) { *p = 0; }

int persistent_blocks()
{
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) !=
        hipSuccess || ncu <= 0)
        ncu = 256;
    return 4 * ncu;
}

} // namespace

struct RaggedBatch::Impl {
    std::vector<FanTables> tables;
    std::vector<long> img_off, sino_off;
    std::vector<int> first, count;   // descriptor k: slices first[k] .. first[k] + count[k] - 1
    std::vector<int> order;          // descriptors by decreasing cost
    long img_total = 0, sino_total = 0;
    DevBuf desc, counter, wa, wb, wq;
    std::vector<RagSlice> host;
};

RaggedBatch::RaggedBatch() : p_(new Impl) {}
RaggedBatch::~RaggedBatch() { delete p_; }

void RaggedBatch::setup(const std::vector<FanGeo>& geos, const std::vector<const float*>& angles, hipStream_t st)
{
    RN_REQUIRE(!geos.empty() && geos.size() == angles.size(), "ragged batch needs one angle set per slice");
    const int n = (int)geos.size();
    p_->tables.resize(n);
    p_->img_off.resize(n);
    p_->sino_off.resize(n);
    long io = 0, so = 0;
    for (int s = 0; s < n; s++) {
        RN_REQUIRE(geos[s].nz == 1 && geos[s].nv == 1, "ragged batches hold 2D slices");
        // the per-slice gathers address a plane, a ray table and a sinogram with 32-bit byte offsets
        RN_REQUIRE((long)geos[s].nx * geos[s].ny * 4L < 0x7fffffffL &&
                       (long)geos[s].nu * geos[s].nview * 16L < 0x7fffffffL,
                   "a ragged slice's image, ray table or sinogram exceeds 2 GiB");
        p_->tables[s].build(geos[s], angles[s], st);
        p_->img_off[s] = io;
        p_->sino_off[s] = so;
        io += (long)geos[s].nx * geos[s].ny;
        so += (long)geos[s].nu * geos[s].nview;
    }
    p_->img_total = io;
    p_->sino_total = so;
    // runs of consecutive slices with one geometry and angle set, in chunks of kRagS
    // (one chunk's interleaved groups of 4 slices are addressed with 32-bit byte offsets)
    auto fits = [&](int s, int count) {
        return (long)((count + 3) / 4) * geos[s].nu * geos[s].nview * 16L < 0x7fffffffL;
    };
    auto same = [&](int a, int b) {
        const FanGeo& x = geos[a];
        const FanGeo& y = geos[b];
        return x.nx == y.nx && x.ny == y.ny && x.nz == y.nz && x.dx == y.dx && x.dy == y.dy && x.dz == y.dz &&
               x.nu == y.nu && x.nview == y.nview && x.nv == y.nv && x.da == y.da && x.dv == y.dv &&
               x.off_a == y.off_a && x.off_v == y.off_v && x.dsd == y.dsd && x.dso == y.dso &&
               std::equal(angles[a], angles[a] + x.nview, angles[b]);
    };
    p_->first.clear();
    p_->count.clear();
    for (int s = 0; s < n; s++) {
        if (!p_->count.empty() && p_->count.back() < kRagS && same(p_->first.back(), s) &&
            fits(s, p_->count.back() + 1)) {
            ++p_->count.back();
        } else {
            p_->first.push_back(s);
            p_->count.push_back(1);
        }
    }
    const int nd = (int)p_->first.size();
    p_->order.resize(nd);
    std::iota(p_->order.begin(), p_->order.end(), 0);
    std::stable_sort(p_->order.begin(), p_->order.end(), [&](int a, int b) {
        const FanGeo& ga = geos[p_->first[a]];
        const FanGeo& gb = geos[p_->first[b]];
        return (double)ga.nx * ga.ny * ga.nview > (double)gb.nx * gb.ny * gb.nview;
    });
    p_->desc.alloc(nd * ((kRagS + kRagFp - 1) / kRagFp) * sizeof(RagSlice));
    p_->counter.alloc(sizeof(int));
    p_->wa.alloc(io * sizeof(float));
    p_->wb.alloc(io * sizeof(float));
    // the interleaved sinograms: whole groups of 4 slices per descriptor
    long qo = 0;
    for (int k = 0; k < nd; k++) {
        const FanGeo& g = geos[p_->first[k]];
        qo += (long)((p_->count[k] + 3) / 4) * g.nu * g.nview;
    }
    p_->wq.alloc(qo * sizeof(float4));
}

int RaggedBatch::size() const { return (int)p_->tables.size(); }
long RaggedBatch::image_elems() const { return p_->img_total; }
long RaggedBatch::sino_elems() const { return p_->sino_total; }

void RaggedBatch::forward(bool siddon, const float* img, float* prj, hipStream_t st)
{
    const int nd = (int)p_->first.size();
    float* A = p_->wa.as<float>();
    float* Bb = p_->wb.as<float>();
    p_->host.clear();
    int item = 0;
    for (int k = 0; k < nd; k++) {
        const int s = p_->first[p_->order[k]], cnt = p_->count[p_->order[k]];
        const FanGeo& g = p_->tables[s].geo;
        const float* P = img + p_->img_off[s];
        float* a = A + p_->img_off[s];
        float* b = Bb + p_->img_off[s];
        const float* pa;
        const float* pb;
        if (siddon) {
            launch_transpose(P, a, g.nx, g.ny, cnt, st);    // rows contiguous
            pa = a;
            pb = P;
        } else {
            // RY[x][y] = (P[x-1][y] + P[x][y]) / 2 ;  RX = transpose((P[x][y-1] + P[x][y]) / 2)
            launch_avg_planes(P, b, a, g.nx, g.ny, cnt, st);
            pa = a;
            pb = b;
        }
        // the group's slices in chunks of kRagFp, consecutive in both layouts
        const long plane = (long)g.nx * g.ny, sino = (long)g.nu * g.nview;
        for (int c0 = 0; c0 < cnt; c0 += kRagFp) {
            RagSlice d{};
            d.g = p_->tables[s].k;
            d.nsl = std::min(kRagFp, cnt - c0);
            d.pa = pa + c0 * plane;
            d.pb = pb + c0 * plane;
            d.out = prj + p_->sino_off[s] + c0 * sino;
            d.tiles = cdiv(g.nu, 64);
            d.nitems = d.tiles * g.nview;
            d.item0 = item;
            item += d.nitems;
            p_->host.push_back(d);
        }
    }
    const int nfd = (int)p_->host.size();
    RN_HIP_CHECK(hipMemcpyAsync(p_->desc.get(), p_->host.data(), nfd * sizeof(RagSlice), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, st, p_->counter.as<int>());
    hipLaunchKernelGGL(k_ragged_fp, dim3(persistent_blocks()), dim3(256), 0, st, p_->desc.as<RagSlice>(), nfd, item,
                       p_->counter.as<int>(), siddon ? 1 : 0);
    check_launch("ragged_fp");
    RN_HIP_CHECK(hipStreamSynchronize(st));
}

void RaggedBatch::backward(bool siddon, const float* prj, float* img, hipStream_t st)
{
    const int nd = (int)p_->first.size();
    float4* Q = p_->wq.as<float4>();
    p_->host.clear();
    const int chunk = siddon ? kRagSidBp : kRagS;
    // the DD adjoint's descriptors by FanK::dwide, a launch for each kind: a slice's bits
    // depend on its own geometry only
    std::vector<int> order = p_->order;
    int nwide = nd;
    if (!siddon)
        nwide = (int)(std::stable_partition(order.begin(), order.end(), [&](int k) {
                    return p_->tables[p_->first[k]].k.dwide != 0;
                }) - order.begin());
    int items[2] = {0, 0}, split = 0;   // per launch; the second one's first descriptor
    for (int k = 0; k < nd; k++) {
        int& item = items[k < nwide ? 0 : 1];
        const int s = p_->first[order[k]], cnt = p_->count[order[k]];
        const FanGeo& g = p_->tables[s].geo;
        if (siddon) launch_pack_quads(prj + p_->sino_off[s], nullptr, Q, g.nu, g.nview, cnt, false, st);
        else launch_pack_quads_len(p_->tables[s].k, prj + p_->sino_off[s], Q, cnt, st);
        const long plane = (long)g.nx * g.ny, sino = (long)g.nu * g.nview;
        for (int c0 = 0; c0 < cnt; c0 += chunk) {
            RagSlice d{};
            d.g = p_->tables[s].k;
            d.nsl = std::min(chunk, cnt - c0);
            d.pa = reinterpret_cast<const float*>(Q + c0 / 4 * sino);
            d.pb = nullptr;
            d.out = img + p_->img_off[s] + c0 * plane;
            d.tiles = cdiv(g.ny, 8);
            d.nitems = d.tiles * cdiv(g.nx, 8);
            d.item0 = item;
            item += d.nitems;
            p_->host.push_back(d);
        }
        Q += (long)((cnt + 3) / 4) * sino;
        if (k < nwide) split = (int)p_->host.size();
    }
    const int nbd = (int)p_->host.size();
    RN_HIP_CHECK(hipMemcpyAsync(p_->desc.get(), p_->host.data(), nbd * sizeof(RagSlice), hipMemcpyHostToDevice, st));
    auto launch = [&](auto kern, int d0, int d1, int total) {
        if (d1 == d0) return;
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, st, p_->counter.as<int>());
        hipLaunchKernelGGL(kern, dim3(persistent_blocks()), dim3(64, kBpSegs), 0, st, p_->desc.as<RagSlice>() + d0,
                           d1 - d0, total, p_->counter.as<int>());
        check_launch("ragged_bp");
    };
    if (siddon) {
        launch(k_ragged_siddon_bp, 0, nbd, items[0]);
    } else {
        launch(k_ragged_dd_adj<true>, 0, split, items[0]);
        launch(k_ragged_dd_adj<false>, split, nbd, items[1]);
    }
    RN_HIP_CHECK(hipStreamSynchronize(st));
}

} // namespace rn
