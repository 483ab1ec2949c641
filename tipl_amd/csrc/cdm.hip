// cdm.hip -- the CDM nonlinear registration loop on gfx950.
//
// Restates, MI355X-first:
//   compose_displacement        numerical/dif.hpp:90-115, 260-285
//   cdm_get_gradient (r, d)     reg/cdm.hpp:46-152 with get_window_at_width<2>
//                               (numerical/window.hpp:92-110), linear_regression
//                               (numerical/statistics.hpp:694-713), gradient_at
//                               (numerical/numerical.hpp:102-109)
//   cdm_solve_poisson           reg/cdm.hpp:158-254
//   cdm_max_displacement_length reg/cdm.hpp:260-296
//   accumulate_displacement     numerical/dif.hpp:166-186, 311-329
//   cdm_smooth                  reg/cdm.hpp:302-367
//   upsample_with_padding       numerical/resampling.hpp:849-891
//   cdm / cdm_cuda              reg/cdm.hpp:373-532
//
// Fields are packed float3 per voxel (the reference's image<3,vector<3>>).
// Kernels are launched on a 3-D grid of 64 x 4 thread tiles (x = one wave),
// so no index division is needed.  The per-iteration control (cost history,
// cdm_improved, smoothing schedule) runs on the host from one float cost
// read back per iteration; everything else stays on the device.
#include "cdm_control.hpp"
#include "device.hpp"
#include "field.hpp"
#include "field_limits.hpp"
#include "host_wait.hpp"
#include "internal.hpp"
#include "march_plan.hpp"
#include "regression.hpp"
#include "step_gate.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

namespace tiplhip {
namespace {

// Where a gradient field (new_d and its Jacobi iterates) keeps component c of
// voxel p: element p * ps + c * cs.  The loops keep these fields planar (one
// array per component), so that kernels which take one component each read
// whole lines: twelve sweeps 269 -> 204 us at 182x218x182, 120 against 216 at
// 160x192x160.  Packed like the displacement fields where a caller's buffer
// is, and where byte offsets, those of a grown tile's planes and rows outside
// the volume included, would pass 2^31.
struct Lay {
    uint32_t ps, cs;
};
__host__ __device__ inline Lay packed_layout() { return Lay{3u, 1u}; }
inline bool planar_fits(const FieldGeo& g) { return marched_field_fits(g.n, g.wh, size_t(g.w)); }
inline Lay grad_layout(const FieldGeo& g) { return planar_fits(g) ? Lay{1u, g.n} : packed_layout(); }

__device__ inline float3 ld_lay(const float* f, uint32_t p, const Lay& l)
{
    const size_t i = size_t(p) * l.ps;
    return make_float3(f[i], f[i + l.cs], f[i + 2 * size_t(l.cs)]);
}
__device__ inline void st_lay(float* f, uint32_t p, const Lay& l, float3 v)
{
    const size_t i = size_t(p) * l.ps;
    f[i] = v.x;
    f[i + l.cs] = v.y;
    f[i + 2 * size_t(l.cs)] = v.z;
}

// ---------------------------------------------------------------------------
// compose_displacement: Js(x) = Is(x + d(x)); exact copy where d(x) == 0.
// ---------------------------------------------------------------------------
// Js at voxel p = (x, y, z) under the displacement dv.
__device__ __forceinline__ uint8_t composed(const uint8_t* __restrict__ Is, const FieldGeo& g, int x, int y,
                                            int z, uint32_t p, const float3& dv)
{
    if (dv.x == 0.0f && dv.y == 0.0f && dv.z == 0.0f) return Is[p];
    const __amdgpu_buffer_rsrc_t r = make_rsrc(Is, g.n);
    VolGeo vg{g.w, g.h, g.d, g.wh, g.wm1, g.hm1, g.dm1};
    return uint8_t(sample_u8(r, vg, float(x) + dv.x, float(y) + dv.y, float(z) + dv.z));
}

__device__ __forceinline__ void compose_body(const uint8_t* __restrict__ Is,
                                             const float* __restrict__ d, const FieldGeo& g,
                                             uint8_t* __restrict__ Js, const Block& blk)
{
    const Vox v = voxel_of(g, blk);
    if (v.ok) Js[v.p] = composed(Is, g, v.x, v.y, v.z, v.p, ld3(d, v.p));
}

__global__ __launch_bounds__(256) void compose_kernel(const uint8_t* __restrict__ Is,
                                                      const float* __restrict__ d, FieldGeo g,
                                                      uint8_t* __restrict__ Js)
{
    compose_body(Is, d, g, Js, logical_block());
}

// ---------------------------------------------------------------------------
// cdm_get_gradient 'd' (SSD): the gradient of Js scaled by Js - It.
// accumulate = 0 writes nd = 0 + g (a fresh field); accumulate = 1 adds a
// further modality: nd = nd + (0 + g).  Per-block FP64 partial sums of the cost
// map go to `partials`.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gradient_d_kernel(const uint8_t* __restrict__ Js,
                                                         const uint8_t* __restrict__ It, FieldGeo g,
                                                         int accumulate, float* __restrict__ nd, Lay lay,
                                                         double* __restrict__ partials)
{
    const Vox v = this_voxel(g);
    float cost = 0.0f;
    if (v.ok) {
        const int dif = int(Js[v.p]) - int(It[v.p]);
        const float s = float(dif);
        cost = float(dif * dif);
        // gradient_at: central differences, 0 on the first/last slab.
        const uint32_t w = uint32_t(g.w);
        const float gx = (v.x + 1 < g.w && v.x) ? float(int(Js[v.p + 1]) - int(Js[v.p - 1])) : 0.0f;
        const float gy = (v.y + 1 < g.h && v.y) ? float(int(Js[v.p + w]) - int(Js[v.p - w])) : 0.0f;
        const float gz = (v.z + 1 < g.d && v.z) ? float(int(Js[v.p + g.wh]) - int(Js[v.p - g.wh])) : 0.0f;
        const float3 gr = make_float3(0.0f + gx * s, 0.0f + gy * s, 0.0f + gz * s);
        if (accumulate) {
            float3 o = ld_lay(nd, v.p, lay);
            o.x = o.x + gr.x;
            o.y = o.y + gr.y;
            o.z = o.z + gr.z;
            st_lay(nd, v.p, lay, o);
        } else {
            st_lay(nd, v.p, lay, gr);
        }
    }
    // deterministic per-block partial sum of the cost map
    __shared__ double part[4];
    double c = wave_sum_f64(double(cost));
    const uint32_t tid = threadIdx.y * blockDim.x + threadIdx.x;
    if ((tid & 63u) == 0) part[tid >> 6] = c;
    __syncthreads();
    if (tid == 0) partials[logical_block().lin] = (part[0] + part[1]) + (part[2] + part[3]);
}

// ---------------------------------------------------------------------------
// cdm_get_gradient 'r': local linear regression of Js onto It over the
// border-clipped 5x5x5 window (exact integer sums, then FP64 as in
// linear_regression), the gradient scaled by r2*(a*Js+b-It) where a > 0, with
// the window sums done as box filters.  accumulate and partials as above.  A block
// owns 16 x TY x TZ outputs.  It stages the bytes of Js and It with a 2-voxel
// halo (zero outside the volume) in LDS, aligned dwords as they lie in
// memory, and forms the 5-tap sums along x, then y, then z, one pass over LDS
// each: four barriers a block and no chain over planes.  The x sums of five
// bytes are four-byte dot products (v_dot4_u32_u8); sum Js and sum It share a
// word (at most 125 * 255 < 2^16 each).  Zero padding leaves the five integer
// sums of the border-clipped window unchanged; the window size is the product
// of the clipped extents, as get_window_at_width counts it.
// Latency bounds the small levels, integer and FP64 issue the large ones.
// Against the z-marching 64 x 4 column it replaces (three barriers a plane,
// byte-wise sums): 15.0 -> 5.0 us at 32x32x32 and below, 15.3 -> 5.6 at
// 40x48x40, 22.1 -> 12.0 at 80x96x80, 81 -> 62 at 160x192x160, 107 -> 92 at
// 182x218x182.
// ---------------------------------------------------------------------------

// A quiet-NaN float pattern the cost reduction never writes, and how long
// the host spins for an iteration's cost before it synchronises the stream.
constexpr uint32_t kCostPending = 0x7FC0C057u;
constexpr int kCostSpinUs = 2000;

constexpr int kGX = 16;     // outputs per tile row
constexpr int kGWords = 6;  // dwords that hold a row's 20 bytes at any alignment

template <int TY, int TZ, int NT>
__device__ __forceinline__ void gradient_r_box_body(const uint8_t* __restrict__ Js,
                                                    const uint8_t* __restrict__ It,
                                                    const FieldGeo& g, int accumulate,
                                                    float* __restrict__ nd, const Lay& lay,
                                                    double* __restrict__ partials,
                                                    const Block& blk)
{
    constexpr int RY = TY + 4, RZ = TZ + 4, kRows = RY * RZ;
    constexpr int kYSums = TY * RZ * kGX, kOut = TY * TZ * kGX;
    static_assert(kYSums % NT == 0 && kOut % NT == 0, "whole passes");
    __shared__ uint32_t words[2][kRows][kGWords];  // Js, It: a row's bytes from its first dword
    __shared__ uint32_t shift[2][kRows];           // byte of x = x0 - 2 in that dword
    __shared__ uint4 sums[kRows * kGX];            // {j | i << 16, jj, ii, ji}: x sums, then y sums
    const int tid = int(threadIdx.x);
    const int x0 = blk.x * kGX, y0 = blk.y * TY, z0 = blk.z * TZ;

    // half a row per task: three aligned dwords, bytes outside the row cleared.
    // A dword is read only if one of its bytes lies in the row, so it never
    // leaves the (dword-granular) allocation.
    for (int t = tid; t < 4 * kRows; t += NT) {
        const int half = t & 1, im = (t >> 1) & 1, r = t >> 2;
        const int ry = r % RY;
        const int gy = y0 - 2 + ry, gz = z0 - 2 + r / RY;
        uint32_t v[3] = {0u, 0u, 0u};
        uint32_t sh = 0;
        if (gy >= 0 && gy < g.h && gz >= 0 && gz < g.d) {
            const uint8_t* src = im ? It : Js;
            const uint32_t mis = uint32_t(reinterpret_cast<uintptr_t>(src)) & 3u;
            const long long at = (long long)gz * g.wh + (long long)gy * g.w + (x0 - 2) + int(mis);
            sh = uint32_t(at) & 3u;
            const uint32_t* q = reinterpret_cast<const uint32_t*>(src - mis) + (at >> 2) + 3 * half;
            const int xb = x0 - 2 - int(sh) + 12 * half;  // x of the first dword's first byte
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int x = xb + 4 * k;
                if (x > -4 && x < g.w) {
                    uint32_t m = ~0u;
                    if (x < 0) m <<= uint32_t(-x) * 8u;
                    if (x + 4 > g.w) m &= ~0u >> (uint32_t(x + 4 - g.w) * 8u);
                    v[k] = q[k] & m;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) words[im][r][3 * half + k] = v[k];
        if (half == 0) shift[im][r] = sh;
    }
    __syncthreads();
    // x sums of every staged row
    for (int c = tid; c < kRows * kGX; c += NT) {
        const int x = c & (kGX - 1), r = c / kGX;
        auto window = [&](int im, uint32_t& lo, uint32_t& last) {
            const uint32_t b = uint32_t(x) + shift[im][r];
            const uint32_t w0 = words[im][r][b >> 2], w1 = words[im][r][(b >> 2) + 1];
            lo = __builtin_amdgcn_alignbyte(w1, w0, b & 3u);
            last = (w1 >> ((b & 3u) * 8u)) & 0xffu;
        };
        uint32_t a, a4, b, b4;
        window(0, a, a4);
        window(1, b, b4);
        const uint32_t j = __builtin_amdgcn_udot4(a, 0x01010101u, a4, false);
        const uint32_t i = __builtin_amdgcn_udot4(b, 0x01010101u, b4, false);
        sums[c] = make_uint4(j | (i << 16), __builtin_amdgcn_udot4(a, a, __umul24(a4, a4), false),
                             __builtin_amdgcn_udot4(b, b, __umul24(b4, b4), false),
                             __builtin_amdgcn_udot4(a, b, __umul24(a4, b4), false));
    }
    __syncthreads();
    auto add = [](uint4& s, const uint4& t) {
        s.x += t.x;
        s.y += t.y;
        s.z += t.z;
        s.w += t.w;
    };
    // y sums, back into the same memory once every x sum has been read
    {
        uint4 ys[kYSums / NT];
#pragma unroll
        for (int u = 0; u < kYSums / NT; ++u) {
            const int c = tid + u * NT;
            const int x = c & (kGX - 1), r = c / kGX;
            const int at = ((r / TY) * RY + r % TY) * kGX + x;
            uint4 s = sums[at];
#pragma unroll
            for (int k = 1; k < 5; ++k) add(s, sums[at + k * kGX]);
            ys[u] = s;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kYSums / NT; ++u) sums[tid + u * NT] = ys[u];
    }
    __syncthreads();
    // z sums and the regression
    double cost_sum = 0.0;
#pragma unroll
    for (int u = 0; u < kOut / NT; ++u) {
        const int c = tid + u * NT;
        const int tx = c & (kGX - 1), ty = (c / kGX) % TY, tz = c / (kGX * TY);
        Vox v;
        v.x = x0 + tx;
        v.y = y0 + ty;
        v.z = z0 + tz;
        if (v.x >= g.w || v.y >= g.h || v.z >= g.d) continue;
        v.p = uint32_t(v.z) * g.wh + uint32_t(v.y) * uint32_t(g.w) + uint32_t(v.x);
        uint4 s = sums[c];
#pragma unroll
        for (int k = 1; k < 5; ++k) add(s, sums[c + k * TY * kGX]);
        const int r = (tz + 2) * RY + ty + 2;
        auto byte_at = [&](int im, int row, int dx) {
            const uint32_t b = uint32_t(tx + 2 + dx) + shift[im][row];
            return (words[im][row][b >> 2] >> ((b & 3u) * 8u)) & 0xffu;
        };
        const int nx = min(v.x + 2, g.w - 1) - max(v.x - 2, 0) + 1;
        const int ny = min(v.y + 2, g.h - 1) - max(v.y - 2, 0) + 1;
        const int nz = min(v.z + 2, g.d - 1) - max(v.z - 2, 0) + 1;
        float cost = 0.0f;
        const float sc = regress<125>(byte_at(0, r, 0), byte_at(1, r, 0),
                                 Sums5{s.x & 0xffffu, s.x >> 16, s.y, s.z, s.w}, nx * ny * nz, cost);
        float3 gr = make_float3(0.0f, 0.0f, 0.0f);
        if (cost != 0.0f || sc != 0.0f) {
            // gradient_at: central differences, 0 on the first/last slab.
            const float gx = (v.x + 1 < g.w && v.x) ? float(int(byte_at(0, r, 1)) - int(byte_at(0, r, -1))) : 0.0f;
            const float gy = (v.y + 1 < g.h && v.y) ? float(int(byte_at(0, r + 1, 0)) - int(byte_at(0, r - 1, 0))) : 0.0f;
            const float gz = (v.z + 1 < g.d && v.z) ? float(int(byte_at(0, r + RY, 0)) - int(byte_at(0, r - RY, 0))) : 0.0f;
            gr.x = 0.0f + gx * sc;
            gr.y = 0.0f + gy * sc;
            gr.z = 0.0f + gz * sc;
        }
        if (accumulate) {
            float3 o = ld_lay(nd, v.p, lay);
            o.x = o.x + gr.x;
            o.y = o.y + gr.y;
            o.z = o.z + gr.z;
            st_lay(nd, v.p, lay, o);
        } else {
            st_lay(nd, v.p, lay, gr);
        }
        cost_sum += double(cost);
    }
    __shared__ double part[NT / 64];
    const double cw = wave_sum_f64(cost_sum);
    if ((tid & 63) == 0) part[tid >> 6] = cw;
    __syncthreads();
    if (tid == 0) {
        double t = part[0];
        for (int i = 1; i < NT / 64; ++i) t += part[i];
        partials[blk.lin] = t;
    }
}

// Tile of the launch: 16 x 4 x 4 outputs on 256 threads, or 16 x 8 x 8 on 512
// for volumes of at least kGLargeVoxels, where there are workgroups enough
// and the smaller halo counts (2.25 instead of 4 x sums per output): 12.0
// against 12.7 us at 80x96x80, 92 against 107 at 182x218x182.
constexpr size_t kGLargeVoxels = size_t(1) << 19;

template <bool LARGE>
struct GradTile {
    static constexpr int kSide = LARGE ? 8 : 4;
    static constexpr int kThreads = LARGE ? 512 : 256;
};

inline bool grad_large(const FieldGeo& g) { return g.n >= kGLargeVoxels; }

template <bool LARGE>
__global__ __launch_bounds__(GradTile<LARGE>::kThreads) void gradient_r_box_kernel(
    const uint8_t* __restrict__ Js, const uint8_t* __restrict__ It, FieldGeo g, int accumulate,
    float* __restrict__ nd, Lay lay, double* __restrict__ partials)
{
    using Tile = GradTile<LARGE>;
    gradient_r_box_body<Tile::kSide, Tile::kSide, Tile::kThreads>(Js, It, g, accumulate, nd, lay, partials,
                                                                  logical_block());
}

dim3 box_grid(const FieldGeo& g)
{
    const int side = grad_large(g) ? GradTile<true>::kSide : GradTile<false>::kSide;
    return dim3(uint32_t((g.w + kGX - 1) / kGX), uint32_t((g.h + side - 1) / side),
                uint32_t((g.d + side - 1) / side));
}

// Sums the block partials in a fixed order, the same for every workgroup size
// that calls it, and stores float(sum / n): each of 256 threads sums its
// strided share, then waves and their totals in order.
struct CostReduce {
    const double* partials = nullptr;
    uint32_t count = 0;
    double n = 0.0;
    float* out = nullptr;
    float* host_out = nullptr;
};
constexpr uint32_t kReduceThreads = 256;

__device__ __forceinline__ void cost_reduce_body(const CostReduce& r, double* part)
{
    double acc = 0.0;
    if (threadIdx.x < kReduceThreads)
        for (uint32_t i = threadIdx.x; i < r.count; i += kReduceThreads) acc += r.partials[i];
    acc = wave_sum_f64(acc);
    if ((threadIdx.x & 63u) == 0 && threadIdx.x < kReduceThreads) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (uint32_t w = 0; w < kReduceThreads / 64; ++w) s += part[w];
        r.out[0] = float(s / r.n);
        if (r.host_out) r.host_out[0] = float(s / r.n);
    }
}

__global__ __launch_bounds__(kReduceThreads) void cost_reduce_kernel(const CostReduce r)
{
    __shared__ double part[kReduceThreads / 64];
    cost_reduce_body(r, part);
}

// Max of the per-block maxima (non-negative floats), as float bits.
__device__ __forceinline__ void max_reduce_body(const float* __restrict__ parts, uint32_t count,
                                                unsigned int* __restrict__ out,
                                                unsigned int* __restrict__ host_out)
{
    float m = 0.0f;
    for (uint32_t i = threadIdx.x; i < count; i += blockDim.x) m = fmaxf(m, parts[i]);
    __shared__ float part[16];
    m = wave_max_f32(m);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = 0.0f;
        for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) r = fmaxf(r, part[w]);
        out[0] = __float_as_uint(r);
        if (host_out) host_out[0] = __float_as_uint(r);
    }
}

__global__ __launch_bounds__(1024) void max_reduce_kernel(const float* __restrict__ parts,
                                                          uint32_t count,
                                                          unsigned int* __restrict__ out,
                                                          unsigned int* __restrict__ host_out)
{
    max_reduce_body(parts, count, out, host_out);
}

// ---------------------------------------------------------------------------
// cdm_solve_poisson: one Jacobi sweep, 7-point stencil with neighbours taken
// by flat index and dropped at the array ends.  FIRST: the previous iterate
// is nd * (-1/6), formed on the fly.  MAXLEN: also the max of
// float(sqrt(double(|v|^2))) (cdm_max_displacement_length) as float bits.
// ---------------------------------------------------------------------------
constexpr float kInvD2 = -0.5f / 3.0f;

// Volumes of at most this many voxels take poisson4_kernel (21 us for twelve
// sweeps of 40x48x40), larger ones poisson_march_kernel (39 against 68 us at
// 80x96x80).
constexpr size_t kPoisson4Voxels = size_t(1) << 18;

// ---------------------------------------------------------------------------
// One Jacobi sweep, marching z.  A block owns a 64 x 8 column of voxels
// over kPZ planes; each thread keeps the previous iterate of its own column
// at z-1, z, z+1 in registers (the +-wh neighbours), takes x-1 / x+1 from
// the neighbouring lanes of its wave, y-1 / y+1 from the block's LDS copy of
// the plane, and loads the neighbours that fall outside the tile by flat
// index -- which is exactly the reference's flat-index neighbourhood, row and
// plane wrap included.  Every value is combined in the reference's order.
// ---------------------------------------------------------------------------
constexpr int kPTY = 8, kPZ = 16;

dim3 poisson_grid(const FieldGeo& g)
{
    return dim3(uint32_t((g.w + kTX - 1) / kTX), uint32_t((g.h + kPTY - 1) / kPTY),
                uint32_t((g.d + kPZ - 1) / kPZ));
}

template <bool FIRST, bool MAXLEN>
__global__ __launch_bounds__(kTX * kPTY) void poisson_zm_kernel(const float* __restrict__ nd,
                                                                const float* __restrict__ a,
                                                                FieldGeo g, float* __restrict__ b,
                                                                float* __restrict__ maxparts)
{
    __shared__ float3 plane[kPTY][kTX];
    const int tx = int(threadIdx.x), ty = int(threadIdx.y);
    const Block blk = logical_block();
    const int x = blk.x * kTX + tx, y = blk.y * kPTY + ty;
    const int z0 = blk.z * kPZ, z1 = min(z0 + kPZ, g.d);
    const bool ok = x < g.w && y < g.h;
    const uint32_t n = g.n, w = uint32_t(g.w), wh = g.wh;
    auto A = [&](uint32_t q) -> float3 {
        if (FIRST) {
            const float3 t = ld3(nd, q);
            return make_float3(t.x * kInvD2, t.y * kInvD2, t.z * kInvD2);
        }
        return ld3(a, q);
    };
    const float3 zero3 = make_float3(0.0f, 0.0f, 0.0f);
    uint32_t p = uint32_t(z0) * wh + uint32_t(y) * w + uint32_t(x);
    float3 am = (ok && z0 >= 1) ? A(p - wh) : zero3;
    float3 ac = ok ? A(p) : zero3;
    float len_max = 0.0f;
    for (int z = z0; z < z1; ++z) {
        const float3 ap = (ok && z + 1 < g.d) ? A(p + wh) : zero3;
        plane[ty][tx] = ac;
        // x neighbours from the adjacent lanes of this row's wave
        const float lx0 = __shfl_up(ac.x, 1, kTX), lx1 = __shfl_up(ac.y, 1, kTX),
                    lx2 = __shfl_up(ac.z, 1, kTX);
        const float rx0 = __shfl_down(ac.x, 1, kTX), rx1 = __shfl_down(ac.y, 1, kTX),
                    rx2 = __shfl_down(ac.z, 1, kTX);
        __syncthreads();
        if (ok) {
            float3 r = ld3(nd, p);
            auto sub = [&](float3 t) {
                r.x = r.x - t.x;
                r.y = r.y - t.y;
                r.z = r.z - t.z;
            };
            if (p >= 1u) sub(tx > 0 ? make_float3(lx0, lx1, lx2) : A(p - 1u));
            if (p < n - 1u) sub((tx < kTX - 1 && x + 1 < g.w) ? make_float3(rx0, rx1, rx2) : A(p + 1u));
            if (p >= w) sub(ty > 0 ? plane[ty - 1][tx] : A(p - w));
            if (p < n - w) sub((ty < kPTY - 1 && y + 1 < g.h) ? plane[ty + 1][tx] : A(p + w));
            if (p >= wh) sub(am);
            if (p < n - wh) sub(ap);
            r.x = r.x * kInvD2;
            r.y = r.y * kInvD2;
            r.z = r.z * kInvD2;
            st3(b, p, r);
            if (MAXLEN) {
                float s2 = r.x * r.x + r.y * r.y;
                s2 = s2 + r.z * r.z;
                len_max = fmaxf(len_max, float(sqrt(double(s2))));
            }
        }
        __syncthreads();  // the plane buffer is rewritten next step
        am = ac;
        ac = ap;
        p += wh;
    }
    if (MAXLEN) {
        __shared__ float part[kPTY];
        const int tid = ty * kTX + tx;
        const float m = wave_max_f32(len_max);
        if ((tid & 63) == 0) part[tid >> 6] = m;
        __syncthreads();
        if (tid == 0) {
            float r = part[0];
            for (int i = 1; i < kPTY; ++i) r = fmaxf(r, part[i]);
            maxparts[blk.lin] = r;
        }
    }
}

// ---------------------------------------------------------------------------
// Two Jacobi sweeps per launch (s_t -> s_t+1 -> s_t+2), marching z.
//
// Tiles are laid out in flat-index space: the voxel at offset (i, j) of a
// tile of plane m is flat index P0(m) + j*w + i, P0(m) the flat index of the
// tile's first voxel.  The reference's neighbours p-1, p+1, p-w, p+w are then
// offsets (i-1, j), (i+1, j), (i, j-1), (i, j+1) -- row and plane wrap
// included -- and p-+wh is the same offset in planes m-+1.  A neighbour
// outside [0, n) is dropped by the reference; here it holds +0.0, and
// r - (+0.0) == r for every float r, so the results are bit-identical.
//
// Per plane m the block holds s_t on its tile grown by 2 (S ring, 3 planes),
// computes s_t+1 on the tile grown by 1 (T ring, 3 planes), then s_t+2 of
// plane m-1 on the tile itself.  The loop is software-pipelined: while it
// works on plane m from LDS, each thread's global loads for plane m+2 of s_t
// and for the new_d values of plane m+1 are in flight in registers.  Thread
// (tx, ty) computes s_t+1 at its own voxel (tx, ty) and keeps that new_d
// value for its s_t+2 output one plane later; threads 0..147 also compute
// the 148 positions of the ring around the tile.  HBM traffic per two
// sweeps: new_d and s_t read once, s_t+2 written once (36 B per voxel
// instead of 72).  A workgroup covers zq planes; small volumes use a small
// zq so that they still get enough workgroups.
// ---------------------------------------------------------------------------
constexpr int kQX = 64, kQY = 8, kQZMax = 16;
constexpr int kS2X = kQX + 4, kS2Y = kQY + 4;  // tile grown by 2
constexpr int kS1X = kQX + 2, kS1Y = kQY + 2;  // tile grown by 1
constexpr int kRing = kS1X * kS1Y - kQX * kQY;  // 148 positions around the tile
constexpr int kS2N = kS2X * kS2Y;               // 816

// planes per workgroup: about 512 workgroups or more, 2..16 planes each
int poisson2_zq(const FieldGeo& g)
{
    const long long tiles = (long long)((g.w + kQX - 1) / kQX) * ((g.h + kQY - 1) / kQY);
    const long long want = std::max<long long>(1, (tiles * g.d + 511) / 512);
    return int(std::min<long long>(kQZMax, std::max<long long>(2, want)));
}

dim3 poisson2_grid(const FieldGeo& g, int zq)
{
    return dim3(uint32_t((g.w + kQX - 1) / kQX), uint32_t((g.h + kQY - 1) / kQY),
                uint32_t((g.d + zq - 1) / zq));
}

// offset (i, j) of ring position r (-1 <= i <= kQX, -1 <= j <= kQY, not inside)
__device__ inline void ring_offset(int r, int& i, int& j)
{
    if (r < kS1X) { i = r - 1; j = -1; }
    else if (r < 2 * kS1X) { i = r - kS1X - 1; j = kQY; }
    else if (r < 2 * kS1X + kQY) { i = -1; j = r - 2 * kS1X; }
    else { i = kQX; j = r - 2 * kS1X - kQY; }
}

template <bool FIRST, bool MAXLEN>
__device__ __forceinline__ void poisson2_body(const float* __restrict__ nd, const float* __restrict__ a,
                                              const FieldGeo& g, int zq, float* __restrict__ b,
                                              float* __restrict__ maxparts, const Block& blk)
{
    __shared__ float3 S[3][kS2Y][kS2X];
    __shared__ float3 T[3][kS1Y][kS1X];
    const int tx = int(threadIdx.x), ty = int(threadIdx.y), tid = ty * kQX + tx;
    const int x0 = blk.x * kQX, y0 = blk.y * kQY;
    const int z0 = blk.z * zq, z1 = min(z0 + zq, g.d);
    const long long n = g.n, w = g.w, wh = g.wh;
    const long long base = (long long)y0 * w + x0;
    const float3 zero = make_float3(0.0f, 0.0f, 0.0f);

    // this thread's S positions (two at most) and its ring position
    const int e0 = tid, e1 = tid + kQX * kQY;
    const long long so0 = (long long)(e0 / kS2X - 2) * w + (e0 % kS2X - 2);
    const long long so1 = (long long)(e1 / kS2X - 2) * w + (e1 % kS2X - 2);
    const bool has1 = e1 < kS2N;
    int ri = 0, rj = 0;
    const bool has_ring = tid < kRing;
    if (has_ring) ring_offset(tid, ri, rj);
    const long long ro = (long long)rj * w + ri;
    const long long io = (long long)ty * w + tx;  // this thread's own voxel

    auto load_s = [&](long long q) -> float3 {
        if (q < 0 || q >= n) return make_float3(0.0f, 0.0f, 0.0f);
        const float3 t = ld3(FIRST ? nd : a, uint32_t(q));
        if (FIRST) return make_float3(t.x * kInvD2, t.y * kInvD2, t.z * kInvD2);
        return t;
    };
    auto load_r = [&](long long q) -> float3 {
        if (q < 0 || q >= n) return make_float3(0.0f, 0.0f, 0.0f);
        return ld3(nd, uint32_t(q));
    };
    auto valid = [&](long long q) { return q >= 0 && q < n; };
    // one Jacobi update in the reference's order from the six neighbours
    auto update = [](float3 r, float3 xm, float3 xp, float3 ym, float3 yp, float3 zm, float3 zp) {
        r.x = r.x - xm.x; r.y = r.y - xm.y; r.z = r.z - xm.z;
        r.x = r.x - xp.x; r.y = r.y - xp.y; r.z = r.z - xp.z;
        r.x = r.x - ym.x; r.y = r.y - ym.y; r.z = r.z - ym.z;
        r.x = r.x - yp.x; r.y = r.y - yp.y; r.z = r.z - yp.z;
        r.x = r.x - zm.x; r.y = r.y - zm.y; r.z = r.z - zm.z;
        r.x = r.x - zp.x; r.y = r.y - zp.y; r.z = r.z - zp.z;
        return make_float3(r.x * kInvD2, r.y * kInvD2, r.z * kInvD2);
    };
    auto store_s = [&](int m, float3 v0, float3 v1) {
        float3(*dst)[kS2X] = S[(m + 3) % 3];
        dst[e0 / kS2X][e0 % kS2X] = v0;
        if (has1) dst[e1 / kS2X][e1 % kS2X] = v1;
    };

    // prologue: S planes z0-2, z0-1 in LDS; S plane z0 and new_d of plane z0-1 in registers
    {
        const long long p = (long long)(z0 - 2) * wh + base;
        store_s(z0 - 2, load_s(p + so0), has1 ? load_s(p + so1) : zero);
        const long long p1 = p + wh;
        store_s(z0 - 1, load_s(p1 + so0), has1 ? load_s(p1 + so1) : zero);
    }
    long long pz = (long long)z0 * wh + base;  // plane m+1 during iteration m
    float3 s0 = load_s(pz + so0), s1 = has1 ? load_s(pz + so1) : zero;
    const long long pm = pz - wh;              // plane z0-1
    float3 r_in = load_r(pm + io), r_ring = has_ring ? load_r(pm + ro) : zero;
    bool v_in = valid(pm + io), v_ring = has_ring && valid(pm + ro);
    float3 r_prev = zero;  // new_d at this thread's voxel of plane m-1
    float len_max = 0.0f;

    for (int m = z0 - 1; m <= z1; ++m) {
        // S(m+1) from registers into the ring slot of plane m-2, then the next prefetch
        store_s(m + 1, s0, s1);
        const float3 c_in = r_in, c_ring = r_ring;
        const bool cv_in = v_in, cv_ring = v_ring;
        pz += wh;  // plane m+2
        s0 = load_s(pz + so0);
        s1 = has1 ? load_s(pz + so1) : zero;
        const long long pn = pz - wh;  // plane m+1
        r_in = load_r(pn + io);
        r_ring = has_ring ? load_r(pn + ro) : zero;
        v_in = valid(pn + io);
        v_ring = has_ring && valid(pn + ro);
        __syncthreads();
        // s_t+1 of plane m: this thread's voxel and its ring position
        {
            float3(*sm)[kS2X] = S[(m + 2) % 3];
            float3(*sc)[kS2X] = S[(m + 3) % 3];
            float3(*sp)[kS2X] = S[(m + 4) % 3];
            float3(*dst)[kS1X] = T[(m + 3) % 3];
            {
                const int ci = tx + 2, cj = ty + 2;
                dst[ty + 1][tx + 1] = cv_in ? update(c_in, sc[cj][ci - 1], sc[cj][ci + 1], sc[cj - 1][ci],
                                                     sc[cj + 1][ci], sm[cj][ci], sp[cj][ci])
                                            : zero;
            }
            if (has_ring) {
                const int ci = ri + 2, cj = rj + 2;
                dst[rj + 1][ri + 1] = cv_ring ? update(c_ring, sc[cj][ci - 1], sc[cj][ci + 1],
                                                       sc[cj - 1][ci], sc[cj + 1][ci], sm[cj][ci],
                                                       sp[cj][ci])
                                              : zero;
            }
        }
        __syncthreads();
        // s_t+2 of plane m-1 at this thread's voxel
        const int z = m - 1;
        if (z >= z0 && z < z1 && x0 + tx < g.w && y0 + ty < g.h) {
            float3(*tm)[kS1X] = T[(z + 2) % 3];
            float3(*tc)[kS1X] = T[(z + 3) % 3];
            float3(*tp)[kS1X] = T[(z + 4) % 3];
            const int cj = ty + 1, ci = tx + 1;
            const float3 r = update(r_prev, tc[cj][ci - 1], tc[cj][ci + 1], tc[cj - 1][ci],
                                    tc[cj + 1][ci], tm[cj][ci], tp[cj][ci]);
            st3(b, uint32_t((long long)z * wh + base + io), r);
            if (MAXLEN) {
                float s2 = r.x * r.x + r.y * r.y;
                s2 = s2 + r.z * r.z;
                len_max = fmaxf(len_max, float(sqrt(double(s2))));
            }
        }
        r_prev = c_in;
    }
    if (MAXLEN) {
        __shared__ float part[kQY];
        const float mx = wave_max_f32(len_max);
        if ((tid & 63) == 0) part[tid >> 6] = mx;
        __syncthreads();
        if (tid == 0) {
            float r = part[0];
            for (int i = 1; i < kQY; ++i) r = fmaxf(r, part[i]);
            maxparts[blk.lin] = r;
        }
    }
}

template <bool FIRST, bool MAXLEN>
__global__ __launch_bounds__(kQX * kQY) void poisson2_kernel(const float* __restrict__ nd,
                                                             const float* __restrict__ a,
                                                             FieldGeo g, int zq,
                                                             float* __restrict__ b,
                                                             float* __restrict__ maxparts)
{
    poisson2_body<FIRST, MAXLEN>(nd, a, g, zq, b, maxparts, logical_block());
}

// ---------------------------------------------------------------------------
// Four Jacobi sweeps per launch for small volumes.  The three components of
// the field are independent in cdm_solve_poisson, so a workgroup takes one
// component of one 8 x 8 x 8 tile, grown by 4 on every side to 16 x 16 x 16.
// Thread (lx, ly) holds its 16-voxel z column of the iterate and of new_d in
// registers: the p-+wh neighbours are its own registers, p-+1 come from the
// neighbouring lanes of its 16-lane row (DPP), p-+w from an LDS copy of the
// planes.  A sweep spoils one layer of the grown tile, so after four the
// 8 x 8 x 8 core is exact.  Offsets are flat-index offsets as in
// poisson2_kernel (row and plane wrap included); positions outside [0, n)
// read 0 through the buffer's range check and are kept +0.0, which is the
// reference's dropped neighbour (x - (+0.0) is x, -0.0 included).
// What bounds it is latency -- one round of loads, four barriers -- where
// poisson2_kernel chains a barrier pair and a load per plane.  Twelve sweeps:
// 44 -> 17 us at 32x32x32 and below, 45 -> 21 at 40x48x40; at 80x96x80 the
// halo's work (eight times the core's) takes over: 68, poisson_march_kernel 39.
// ---------------------------------------------------------------------------
constexpr int kCT = 8, kCH = 4, kCL = kCT + 2 * kCH;  // tile, halo (= sweeps), grown tile
constexpr int kCThreads = kCL * kCL;
static_assert(kCL == 16, "a tile row is one DPP row");

inline bool poisson4_fits(const FieldGeo& g) { return g.n <= kPoisson4Voxels; }

uint32_t poisson4_blocks(const FieldGeo& g)
{
    return 3u * uint32_t((g.w + kCT - 1) / kCT) * uint32_t((g.h + kCT - 1) / kCT) *
           uint32_t((g.d + kCT - 1) / kCT);
}

template <bool FIRST>
__device__ __forceinline__ void poisson4_body(const float* __restrict__ nd, const float* __restrict__ a,
                                              const FieldGeo& g, const Lay& lay, float* __restrict__ b,
                                              uint32_t blk)
{
    __shared__ float plane[2][kCL][kCL + 2][kCL];  // rows -1 .. 16 of every plane
    const int tid = int(threadIdx.x), lx = tid & (kCL - 1), ly = tid / kCL;
    const uint32_t gx = uint32_t((g.w + kCT - 1) / kCT), gy = uint32_t((g.h + kCT - 1) / kCT);
    const uint32_t comp = blk % 3u, tile = blk / 3u;
    const int x0 = int(tile % gx) * kCT, y0 = int((tile / gx) % gy) * kCT, z0 = int(tile / (gx * gy)) * kCT;
    const int w = g.w, wh = int(g.wh), n = int(g.n);
    const int q0 = (z0 - kCH) * wh + (y0 - kCH) * w + (x0 - kCH);  // the grown tile's first voxel
    const int q = q0 + ly * w + lx;
    const uint32_t bytes = ((g.n - 1u) * lay.ps + 1u) * 4u;
    const __amdgpu_buffer_rsrc_t rn = make_rsrc(nd + size_t(comp) * lay.cs, bytes);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc((FIRST ? nd : a) + size_t(comp) * lay.cs, bytes);
    const int pitch = int(lay.ps) * 4;
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int k) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (q + k * wh) * pitch, 0, 0));
    };
    float r[kCL], v[kCL];
#pragma unroll
    for (int k = 0; k < kCL; ++k) r[k] = load(rn, k);
    // tiles that reach past either end of the array keep those positions +0.0
    const bool ends = q0 < 0 || q0 + (kCL - 1) * (1 + w + wh) >= n;
    uint32_t inside = 0;
#pragma unroll
    for (int k = 0; k < kCL; ++k) inside |= uint32_t(q + k * wh >= 0 && q + k * wh < n) << k;
    if constexpr (FIRST) {
#pragma unroll
        for (int k = 0; k < kCL; ++k) v[k] = r[k] * kInvD2;
        if (ends) {
            // (the factor is negative: 0 read there has become -0.0)
#pragma unroll
            for (int k = 0; k < kCL; ++k) v[k] = (inside >> k) & 1u ? v[k] : 0.0f;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kCL; ++k) v[k] = load(ra, k);
    }
#pragma unroll
    for (int s = 1; s <= kCH; ++s) {
        float(*pl)[kCL + 2][kCL] = plane[s & 1];
#pragma unroll
        for (int k = s; k < kCL - s; ++k) pl[k][ly + 1][lx] = v[k];
        __syncthreads();
        float below = v[s - 1];
#pragma unroll
        for (int k = s; k < kCL - s; ++k) {
            const float c = v[k];
            const float xm = dpp_prev(c), xp = dpp_next(c);
            float t = r[k] - xm;
            t = t - xp;
            t = t - pl[k][ly][lx];
            t = t - pl[k][ly + 2][lx];
            t = t - below;
            t = t - v[k + 1];
            t = t * kInvD2;
            below = c;
            v[k] = t;
        }
        if (ends) {
#pragma unroll
            for (int k = s; k < kCL - s; ++k) v[k] = (inside >> k) & 1u ? v[k] : 0.0f;
        }
    }
    if (lx < kCH || lx >= kCH + kCT || ly < kCH || ly >= kCH + kCT) return;
    if (x0 + lx - kCH >= w || y0 + ly - kCH >= g.h) return;
#pragma unroll
    for (int k = kCH; k < kCH + kCT; ++k)
        if (z0 + k - kCH < g.d) b[size_t(q + k * wh) * lay.ps + size_t(comp) * lay.cs] = v[k];
}

template <bool FIRST>
__global__ __launch_bounds__(kCThreads) void poisson4_kernel(const float* __restrict__ nd,
                                                             const float* __restrict__ a, FieldGeo g,
                                                             Lay lay, float* __restrict__ b,
                                                             const CostReduce cost)
{
    uint32_t blk = blockIdx.x, blocks = gridDim.x;
    if (FIRST && cost.partials) {
        // one more workgroup, the first, sums the gradient's cost
        if (blk == 0) {
            __shared__ double part[kReduceThreads / 64];
            cost_reduce_body(cost, part);
            return;
        }
        --blk;
        --blocks;
    }
    poisson4_body<FIRST>(nd, a, g, lay, b, xcd_remap(blk, blocks));
}

// ---------------------------------------------------------------------------
// K Jacobi sweeps per launch for large volumes, marching z.  As in
// poisson4_kernel a workgroup takes one component, in flat-index offsets.
// Its waves stack in y: lane l of wave v holds the kMR rows v * kMR .. of
// column l, 64 x (kMWaves * kMR) columns in all, K of them halo on each side.
// At step m plane m of the input arrives and stage t = 1 .. K computes plane
// m - t from stage t - 1's planes m - t - 1, m - t, m - t + 1.  All planes
// live in registers: p-+wh are the thread's own, p-+1 the neighbouring
// lanes' (DPP wave shift), p-+w the thread's other rows; only a wave's first
// and last row go through LDS, written in one step and read in the next, so
// a step has one barrier for its K sweeps.  Rings of planes are indexed by
// the unrolled step, so no value is moved.
// Issue (about 160 vector instructions a step for 16 updates a thread) and the
// chain within a step bound it, at the four waves a SIMD that its registers
// leave: at 182x218x182 waves issue 37 to 40% of their cycles, wait to issue 21%
// and for data 40%.  Twelve sweeps, against six poisson2_kernel launches: 350 -> 204 us
// at 182x218x182, 245 -> 120 at 160x192x160, 75 -> 39 at 80x96x80.
// ---------------------------------------------------------------------------
constexpr int kMWaves = 8, kMR = 4, kMThreads = 64 * kMWaves, kMRows = kMWaves * kMR;
constexpr int kMK = 4;                   // sweeps per launch
constexpr uint32_t kMarchBlocks = 512;   // workgroups resident at a time: two a CU
constexpr int kMUnroll = 6;  // ring of six planes of input and new_d, three of each later stage

struct March {
    uint32_t gx, gy, gz;  // tiles
    int zc;               // planes per workgroup
    uint32_t blocks;
};

template <int K>
March march_of(const FieldGeo& g)
{
    March m;
    m.gx = uint32_t((g.w + 63 - 2 * K) / (64 - 2 * K));
    m.gy = uint32_t((g.h + kMRows - 1 - 2 * K) / (kMRows - 2 * K));
    const uint32_t cols = 3u * m.gx * m.gy;
    const MarchPlan p = march_plan(cols, g.d, 2 * K + 2, 2, kMarchBlocks);
    m.gz = p.runs;
    m.zc = p.planes;
    m.blocks = cols * m.gz;
    return m;
}

template <int K, bool FIRST>
__global__ __launch_bounds__(kMThreads, 4) void poisson_march_kernel(const float* __restrict__ nd,
                                                                  const float* __restrict__ a,
                                                                  FieldGeo g, March mg, Lay lay,
                                                                  float* __restrict__ b,
                                                                  const CostReduce cost)
{
    __shared__ __align__(16) float edge[2][K][kMWaves][2][64];
    uint32_t blk = blockIdx.x;
    if (FIRST && cost.partials) {
        // one more workgroup, the first, sums the gradient's cost
        if (blk == 0) {
            cost_reduce_body(cost, reinterpret_cast<double*>(edge));
            return;
        }
        --blk;
    }
    const int lane = int(threadIdx.x) & 63;
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const uint32_t L = xcd_remap(blk, mg.blocks);
    const uint32_t comp = L % 3u, tile = L / 3u;
    const int x0 = int(tile % mg.gx) * (64 - 2 * K) - K;
    const int y0 = int((tile / mg.gx) % mg.gy) * (kMRows - 2 * K) - K;
    const int z0 = int(tile / (mg.gx * mg.gy)) * mg.zc, z1 = min(z0 + mg.zc, g.d);
    const int w = g.w, wh = int(g.wh), n = int(g.n);
    const uint32_t bytes = ((g.n - 1u) * lay.ps + 1u) * 4u;
    const __amdgpu_buffer_rsrc_t rn = make_rsrc(nd + size_t(comp) * lay.cs, bytes);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc((FIRST ? nd : a) + size_t(comp) * lay.cs, bytes);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(b + size_t(comp) * lay.cs, bytes);
    const int pitch = int(lay.ps) * 4, row = w * pitch, slab = wh * pitch;
    const int q0 = (y0 + wv * kMR) * w + x0 + lane;  // row 0 of this thread in plane 0
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int at, float (&dst)[kMR]) {
#pragma unroll
        for (int j = 0; j < kMR; ++j)
            dst[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at + j * row, 0, 0));
    };
    // the tile's first and last position in plane 0, and whether any of its
    // planes reaches past the array
    const int first_q = y0 * w + x0, last_q = (y0 + kMRows - 1) * w + x0 + 63;
    const bool ends = first_q + (z0 - K) * wh < 0 || last_q + (z1 - 1 + K) * wh >= n;
    float in[kMUnroll][kMR], r[kMUnroll][kMR], st[K][3][kMR];
#pragma unroll
    for (int t = 1; t < K; ++t)
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int j = 0; j < kMR; ++j) st[t][k][j] = 0.0f;
#pragma unroll
    for (int k = 0; k < kMUnroll; ++k)
#pragma unroll
        for (int j = 0; j < kMR; ++j) in[k][j] = r[k][j] = 0.0f;
    const int first = z0 - K, last = z1 - 1 + K;
    // plane m of the input is in[(m - first) % 6], of new_d r[(m - first) % 6]
    int qm = q0 + first * wh;             // this thread's row 0 in plane m
    int at = (q0 + (first + 2) * wh) * pitch;  // and its byte offset in plane m + 2
    load(ra, at - 2 * slab, in[0]);
    if (!FIRST) load(rn, at - 2 * slab, r[0]);
    load(ra, at - slab, in[1]);
    const bool xy_out = lane >= K && lane < 64 - K && x0 + lane < w;
    for (int base = first; base <= last; base += kMUnroll) {
#pragma unroll
        for (int u = 0; u < kMUnroll; ++u) {
            const int m = base + u;
            if (m > last) break;
            // two planes ahead
            load(ra, at, in[(u + 2) % kMUnroll]);
            if (!FIRST) load(rn, at - slab, r[(u + 1) % kMUnroll]);
            if (FIRST) {
#pragma unroll
                for (int j = 0; j < kMR; ++j) {
                    r[u][j] = in[u][j];
                    in[u][j] = in[u][j] * kInvD2;
                }
                if (ends && (first_q + m * wh < 0 || last_q + m * wh >= n)) {
                    // positions outside the array hold +0.0 (0 read there has
                    // become -0.0)
#pragma unroll
                    for (int j = 0; j < kMR; ++j)
                        in[u][j] = uint32_t(qm + j * w) < uint32_t(n) ? in[u][j] : 0.0f;
                }
            }
            __syncthreads();
            const int par = u & 1;
#pragma unroll
            for (int t = 1; t <= K; ++t) {
                // stage t, plane m - t; needed from plane z0 - (K - t) on
                if (m - t < z0 - (K - t)) continue;
                const int c1 = (u - t + 12) % kMUnroll;  // ring slot of plane m - t
                auto src = [&](int d) -> float(&)[kMR] {  // stage t - 1, plane m - t + d
                    if (t == 1) return in[(u - 1 + d + 12) % kMUnroll];
                    return st[t - 1][(u - t + d + 12) % 3];
                };
                float(&c)[kMR] = src(0);
                float(&zm)[kMR] = src(-1);
                float(&zp)[kMR] = src(1);
                const float up = edge[par ^ 1][t - 1][wv > 0 ? wv - 1 : 0][1][lane];
                const float dn = edge[par ^ 1][t - 1][wv < kMWaves - 1 ? wv + 1 : wv][0][lane];
                float o[kMR];
#pragma unroll
                for (int j = 0; j < kMR; ++j) {
                    float x = r[c1][j] - wave_prev(c[j]);
                    x = x - wave_next(c[j]);
                    x = x - (j > 0 ? c[j - 1] : up);
                    x = x - (j < kMR - 1 ? c[j + 1] : dn);
                    x = x - zm[j];
                    x = x - zp[j];
                    o[j] = x * kInvD2;
                }
                if (t < K) {
                    if (ends) {
                        const int q = qm - t * wh;
#pragma unroll
                        for (int j = 0; j < kMR; ++j)
                            o[j] = uint32_t(q + j * w) < uint32_t(n) ? o[j] : 0.0f;
                    }
#pragma unroll
                    for (int j = 0; j < kMR; ++j) st[t][(u - t + 12) % 3][j] = o[j];
                } else if (m - K >= z0) {
                    const int to = at - (K + 2) * slab;
#pragma unroll
                    for (int j = 0; j < kMR; ++j) {
                        const int rj = wv * kMR + j;
                        if (rj >= K && rj < kMRows - K && y0 + rj < g.h && xy_out)
                            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[j]), rb, to + j * row, 0, 0);
                    }
                }
            }
            // this step's new planes: first and last row of the wave
#pragma unroll
            for (int t = 0; t < K; ++t) {
                float(&v)[kMR] = t == 0 ? in[u] : st[t][(u - t + 12) % 3];
                edge[par][t][wv][0][lane] = v[0];
                edge[par][t][wv][1][lane] = v[kMR - 1];
            }
            at += slab;
            qm += wh;
            // (keeps the two running offsets in two registers: the compiler
            // otherwise carries one per unrolled use and spills)
            asm volatile("" : "+v"(at), "+v"(qm));
        }
    }
}

// ---------------------------------------------------------------------------
// Every sweep in one launch for the smallest volumes: a workgroup takes one
// component, a thread kWVoxels / 1024 voxels by flat index, and each sweep
// goes through an LDS copy of the whole component with wh zeros on either
// side (a dropped neighbour).  One barrier a sweep; against three launches of
// poisson4_kernel, twelve sweeps 15.6 -> 9.6 us at 16x16x16.
// ---------------------------------------------------------------------------
constexpr int kWVoxels = 4096, kWThreads = 1024, kWPer = kWVoxels / kWThreads;

inline bool poisson_whole_fits(const FieldGeo& g) { return g.n <= uint32_t(kWVoxels); }

__global__ __launch_bounds__(kWThreads) void poisson_whole_kernel(const float* __restrict__ nd, FieldGeo g,
                                                                  Lay lay, int sweeps,
                                                                  float* __restrict__ b,
                                                                  const CostReduce cost)
{
    __shared__ __align__(16) float v[2][3 * kWVoxels];  // wh <= n zeros, n values, wh zeros
    uint32_t comp = blockIdx.x;
    if (cost.partials) {
        // one more workgroup, the first, sums the gradient's cost
        if (comp == 0) {
            cost_reduce_body(cost, reinterpret_cast<double*>(v));
            return;
        }
        --comp;
    }
    const int tid = int(threadIdx.x), n = int(g.n), w = g.w, wh = int(g.wh);
    for (int i = tid; i < wh; i += kWThreads) {
        v[0][i] = v[1][i] = 0.0f;
        v[0][wh + n + i] = v[1][wh + n + i] = 0.0f;
    }
    float r[kWPer], c[kWPer];
#pragma unroll
    for (int k = 0; k < kWPer; ++k) {
        const int p = tid + k * kWThreads;
        r[k] = p < n ? nd[size_t(p) * lay.ps + size_t(comp) * lay.cs] : 0.0f;
        c[k] = r[k] * kInvD2;
    }
    for (int s = 0; s < sweeps; ++s) {
        float* f = v[s & 1] + wh;
#pragma unroll
        for (int k = 0; k < kWPer; ++k) {
            const int p = tid + k * kWThreads;
            if (p < n) f[p] = c[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kWPer; ++k) {
            const int p = min(tid + k * kWThreads, n - 1);
            float t = r[k] - f[p - 1];
            t = t - f[p + 1];
            t = t - f[p - w];
            t = t - f[p + w];
            t = t - f[p - wh];
            t = t - f[p + wh];
            c[k] = t * kInvD2;
        }
    }
#pragma unroll
    for (int k = 0; k < kWPer; ++k) {
        const int p = tid + k * kWThreads;
        if (p < n) b[size_t(p) * lay.ps + size_t(comp) * lay.cs] = c[k];
    }
}

// cdm_max_displacement_length of a whole field: per-block maxima.
constexpr uint32_t kMaxLenBlocks = 1024;

__global__ __launch_bounds__(256) void max_length_kernel(const float* __restrict__ d, uint32_t n,
                                                         Lay lay, float* __restrict__ maxparts)
{
    float m = 0.0f;
    for (uint32_t p = blockIdx.x * 256u + threadIdx.x; p < n; p += gridDim.x * 256u) {
        const float3 r = ld_lay(d, p, lay);
        float s2 = r.x * r.x + r.y * r.y;
        s2 = s2 + r.z * r.z;
        m = fmaxf(m, float(sqrt(double(s2))));
    }
    m = wave_max_f32(m);
    __shared__ float part[4];
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) maxparts[blockIdx.x] = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}

// ---------------------------------------------------------------------------
// new_d *= k, then accumulate_displacement(cur, new_d) into out (which may be
// new_d itself where that is packed): new(x) = m(x + new(x)) - x with
// m(y) = cur(y) + y by trilinear interpolation; cur(x) where new(x) == 0 or the
// sample is outside.
// ---------------------------------------------------------------------------
// The accumulated displacement at voxel p = (x, y, z).
__device__ inline float3 accumulated(const float* __restrict__ cur, const float* __restrict__ nd,
                                     const Lay& lay, float k, const FieldGeo& g, uint32_t p, int x, int y,
                                     int z)
{
    float3 d = ld_lay(nd, p, lay);
    d.x = d.x * k;
    d.y = d.y * k;
    d.z = d.z * k;
    if (d.x != 0.0f || d.y != 0.0f || d.z != 0.0f) {
        Tri t;
        if (locate(g, d.x + float(x), d.y + float(y), d.z + float(z), t)) {
            const int ix = t.ix, iy = t.iy, iz = t.iz;
            float3 acc = make_float3(0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const float3 m = ld3(cur, corner(g, t.i0, c));
                const float mx = m.x + float(ix + (c & 1));
                const float my = m.y + float(iy + ((c >> 1) & 1));
                const float mz = m.z + float(iz + ((c >> 2) & 1));
                if (c == 0) {
                    acc.x = mx * t.w[0];
                    acc.y = my * t.w[0];
                    acc.z = mz * t.w[0];
                } else {
                    acc.x = acc.x + mx * t.w[c];
                    acc.y = acc.y + my * t.w[c];
                    acc.z = acc.z + mz * t.w[c];
                }
            }
            return make_float3(acc.x - float(x), acc.y - float(y), acc.z - float(z));
        }
    }
    return ld3(cur, p);
}

__global__ __launch_bounds__(256) void accumulate_kernel(const float* __restrict__ cur, const float* nd,
                                                         Lay lay, float k, FieldGeo g, float* out,
                                                         Lay out_lay)
{
    const Vox v = this_voxel(g);
    if (!v.ok) return;
    st_lay(out, v.p, out_lay, accumulated(cur, nd, lay, k, g, v.p, v.x, v.y, v.z));
}

// One packed float3 voxel through a raw buffer resource: a load past the
// end returns 0 and never faults.
__device__ inline float3 ld3_rsrc(__amdgpu_buffer_rsrc_t r, uint32_t p)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, int(p * 12u), 0, 0);
    return make_float3(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]));
}

// ---------------------------------------------------------------------------
// accumulate_displacement, cdm_smooth and the next iteration's
// compose_displacement in one pass: out = smooth(acc), acc = the accumulated
// field of accumulate_kernel, and Js(x) = Is(x + out(x)) where Js is given.
// A block owns TX x TY x TZ outputs, evaluates acc on them and on the six
// faces around them, keeps it in LDS, and smooths behind one barrier.  Offsets
// are flat-index offsets: a cell past the end of its row or plane is the next
// row's or plane's first voxel, as smooth's neighbours p-+1, p-+w, p-+wh are.
// Byte offsets into the field have 32 bits (field_fits_32).  A position outside
// [0, n) holds +0.0, which adds nothing to the neighbour sum (that sum starts
// at +0.0 and is never -0.0), as the reference drops it.  HBM traffic per
// voxel: new_d read, cur gathered, out written (36 B), Is gathered and Js
// written (2 B).  out must not alias cur or nd.  With keep, cur is also
// copied into keep (the best field taking the running one before the step, as
// the reference's loop does), keep aliasing neither.
// The eight 12-byte corner gathers bind the address unit (a quad of lanes a
// cycle or two), so large volumes stage cur on the tile grown by 2 in LDS and
// gather there; a sample that leaves it (a displacement of a voxel or more, a
// wrapped neighbour) is evaluated again from memory.  Then it is issue and the
// latency of three phases at four waves a SIMD (issuing 33%, waiting to issue 22%
// and for data 45% of the wave cycles, address unit 53% busy at 182x218x182).
// Against the z-marching kernel without compose and compose_kernel after it:
// 12.4 -> 5.1 us at 32x32x32, 24 -> 20 at 80x96x80, 177 -> 152 at
// 182x218x182 (164 unstaged).
// ---------------------------------------------------------------------------
template <int TX, int TY, int TZ, int NT, bool STAGED>
__device__ __forceinline__ void accumulate_smooth_body(
    const float* __restrict__ cur, const float* __restrict__ nd, const Lay& lay, float k, float w_6,
    float w_1, const FieldGeo& g, float* __restrict__ out, float* __restrict__ keep,
    const uint8_t* __restrict__ Is, uint8_t* __restrict__ Js, const Block& blk)
{
    constexpr int kCore = TX * TY * TZ;
    constexpr int kFx = TY * TZ, kFy = TX * TZ, kFz = TX * TY;  // one face along each axis
    constexpr int kCells = kCore + 2 * (kFx + kFy + kFz);
    constexpr int kSX = TX + 4, kSY = TY + 4, kSZ = TZ + 4, kSN = kSX * kSY * kSZ;
    constexpr int kWaves = NT / 64, kBatch = 10;
    static_assert(kCore % NT == 0 && kCells % NT == 0, "whole passes");
    static_assert(!STAGED || ((kSY * kSZ) % (kWaves * kBatch) == 0 && 3 * kSX <= 64),
                  "whole passes over the rows, each a wave wide at most");
    // cur on the grown tile, one array per component; then acc on the cells
    constexpr int kAccN = (TX + 2) * (TY + 2) * (TZ + 2);
    static_assert(kAccN <= kSN, "acc fits the staged field");
    __shared__ float field[3 * (STAGED ? kSN : kAccN)];
    float3(*A)[TY + 2][TX + 2] = reinterpret_cast<float3(*)[TY + 2][TX + 2]>(field);
    static_assert((NT & (NT - 1)) == 0, "the mask below");
    const int tid = int(threadIdx.x) & (NT - 1);  // (its range decides most of cell())
    const int x0 = blk.x * TX, y0 = blk.y * TY, z0 = blk.z * TZ;
    const __amdgpu_buffer_rsrc_t rcur = make_rsrc(cur, g.n * 12u);
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);

    // the running field on the outputs grown by 2, a row a wave at a time:
    // lane e takes dword e of the row's 3 (TX + 4)
    if constexpr (STAGED) {
        const int e = lane, cx = e / 3, gx = x0 - 2 + cx;
        const uint32_t col = (e < 3 * kSX) & (uint32_t(gx) < uint32_t(g.w)) ? 0u : ~0u;
        float* dst = &field[0] + (e % 3) * kSN + cx;
        for (int r0 = wv; r0 < kSY * kSZ; r0 += kWaves * kBatch) {
            float v[kBatch];
#pragma unroll
            for (int q = 0; q < kBatch; ++q) {
                const int r = r0 + q * kWaves;
                const int gy = y0 - 2 + r % kSY, gz = z0 - 2 + r / kSY;
                const uint32_t at = (uint32_t(gz) * g.wh + uint32_t(gy) * uint32_t(g.w) + uint32_t(x0 - 2)) * 12u;
                // rows and columns outside the volume read past the buffer: 0
                const uint32_t row = (uint32_t(gy) < uint32_t(g.h)) & (uint32_t(gz) < uint32_t(g.d)) ? 0u : ~0u;
                v[q] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(rcur, int((at + uint32_t(e) * 4u) | row | col), 0, 0));
            }
            if (e < 3 * kSX) {
#pragma unroll
                for (int q = 0; q < kBatch; ++q) dst[(r0 + q * kWaves) * kSX] = v[q];
            }
        }
    }
    auto cell = [&](int c, int& i, int& j, int& l) {
        if (c < kCore) {
            i = c % TX;
            j = (c / TX) % TY;
            l = c / (TX * TY);
            return;
        }
        c -= kCore;
        if (c < 2 * kFz) {
            l = c < kFz ? -1 : TZ;
            c = c < kFz ? c : c - kFz;
            i = c % TX;
            j = c / TX;
            return;
        }
        c -= 2 * kFz;
        if (c < 2 * kFy) {
            j = c < kFy ? -1 : TY;
            c = c < kFy ? c : c - kFy;
            i = c % TX;
            l = c / TX;
            return;
        }
        c -= 2 * kFy;
        i = c < kFx ? -1 : TX;
        c = c < kFx ? c : c - kFx;
        j = c % TY;
        l = c / TY;
    };
    // cell c's voxel (x, y, z), its index p, and whether it is one
    auto locate_cell = [&](int c, int& x, int& y, int& z, uint32_t& p) {
        int i, j, l;
        cell(c, i, j, l);
        x = x0 + i;
        y = y0 + j;
        z = z0 + l;
        // no output needs a cell more than one past the volume
        bool ok = x <= g.w && y <= g.h && z <= g.d;
        y = x < 0 ? y - 1 : x >= g.w ? y + 1 : y;
        x = x < 0 ? x + g.w : x >= g.w ? x - g.w : x;
        z = y < 0 ? z - 1 : y >= g.h ? z + 1 : z;
        y = y < 0 ? y + g.h : y >= g.h ? y - g.h : y;
        // (the last test: a cell one past both its row and a one-row plane)
        p = uint32_t(z) * g.wh + uint32_t(y) * uint32_t(g.w) + uint32_t(x);
        ok = ok && z >= 0 && z < g.d && p < g.n;
        p = ok ? p : 0u;
        return ok;
    };
    // every new_d value first: one latency for all evaluations of a thread
    constexpr int kEvals = kCells / NT;
    float3 d[kEvals];
#pragma unroll
    for (int u = 0; u < kEvals; ++u) {
        int x, y, z;
        uint32_t p;
        locate_cell(tid + u * NT, x, y, z, p);
        d[u] = ld_lay(nd, p, lay);
    }
    if constexpr (STAGED) __syncthreads();
    // accumulate_kernel's value, operation for operation: the eight corners
    // from the staged tile where it holds them (a displacement below a voxel
    // never leaves it), else from memory
    float3 acc[kEvals];
#pragma unroll
    for (int u = 0; u < kEvals; ++u) {
        int x, y, z;
        uint32_t p;
        const bool ok = locate_cell(tid + u * NT, x, y, z, p);
        const float dx = d[u].x * k, dy = d[u].y * k, dz = d[u].z * k;
        const bool moved = dx != 0.0f || dy != 0.0f || dz != 0.0f;
        const float sx = dx + float(x), sy = dy + float(y), sz = dz + float(z);
        const bool in = (fminf(fminf(sx, sy), sz) >= 0.0f) & (sx < g.wm1) & (sy < g.hm1) & (sz < g.dm1);
        const bool use = moved && in;
        const int ix = use ? int(cvt_u32_sat(sx)) : x, iy = use ? int(cvt_u32_sat(sy)) : y,
                  iz = use ? int(cvt_u32_sat(sz)) : z;
        const float p0 = sx - float(ix), p1 = sy - float(iy), p2 = sz - float(iz);
        const float n0 = 1.0f - p0, n1 = 1.0f - p1, n2 = 1.0f - p2;
        const float n0n1 = n0 * n1, p0n1 = p0 * n1, n0p1 = n0 * p1, p0p1 = p0 * p1;
        const float w[8] = {n0n1 * n2, p0n1 * n2, n0p1 * n2, p0p1 * n2,
                            n0n1 * p2, p0n1 * p2, n0p1 * p2, p0p1 * p2};
        const float gx[2] = {float(ix), float(ix + 1)}, gy[2] = {float(iy), float(iy + 1)},
                    gz[2] = {float(iz), float(iz + 1)};
        auto blend = [&](auto corner_at) {
            float3 t = make_float3(0.0f, 0.0f, 0.0f), m0 = t;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const float3 m = corner_at(c);
                const float mx = m.x + gx[c & 1];
                const float my = m.y + gy[(c >> 1) & 1];
                const float mz = m.z + gz[(c >> 2) & 1];
                if (c == 0) {
                    m0 = m;
                    t.x = mx * w[0];
                    t.y = my * w[0];
                    t.z = mz * w[0];
                } else {
                    t.x = t.x + mx * w[c];
                    t.y = t.y + my * w[c];
                    t.z = t.z + mz * w[c];
                }
            }
            t = make_float3(t.x - float(x), t.y - float(y), t.z - float(z));
            return make_float3(!ok ? 0.0f : use ? t.x : m0.x, !ok ? 0.0f : use ? t.y : m0.y,
                               !ok ? 0.0f : use ? t.z : m0.z);
        };
        const uint32_t i0 = ok ? uint32_t(iz) * g.wh + uint32_t(iy) * uint32_t(g.w) + uint32_t(ix) : 0u;
        auto from_memory = [&](int c) { return ld3_rsrc(rcur, corner(g, i0, c)); };
        if constexpr (!STAGED) {
            acc[u] = blend(from_memory);
            continue;
        }
        const int tx = ix - (x0 - 2), ty = iy - (y0 - 2), tz = iz - (z0 - 2);
        const bool staged = (uint32_t(tx) < uint32_t(kSX - 1)) & (uint32_t(ty) < uint32_t(kSY - 1)) &
                            (uint32_t(tz) < uint32_t(kSZ - 1));
        const float* q = &field[staged ? (tz * kSY + ty) * kSX + tx : 0];
        acc[u] = blend([&](int c) {
            const int o = (c & 1) + ((c & 2) ? kSX : 0) + ((c & 4) ? kSX * kSY : 0);
            return make_float3(q[o], q[o + kSN], q[o + 2 * kSN]);
        });
        if (__ballot(!staged)) {
            if (!staged) acc[u] = blend(from_memory);
        }
        // one evaluation's corners in registers at a time
        asm volatile("" ::: "memory");
    }
    if constexpr (STAGED) __syncthreads();  // the staged field has been read
#pragma unroll
    for (int u = 0; u < kEvals; ++u) {
        int i, j, l;
        cell(tid + u * NT, i, j, l);
        A[l + 1][j + 1][i + 1] = acc[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kCore / NT; ++u) {
        int i, j, l;
        cell(tid + u * NT, i, j, l);
        const int x = x0 + i, y = y0 + j, z = z0 + l;
        if (x >= g.w || y >= g.h || z >= g.d) continue;
        const float3 t[6] = {A[l + 1][j + 1][i + 2], A[l + 1][j + 1][i], A[l + 1][j + 2][i + 1],
                             A[l + 1][j][i + 1],     A[l + 2][j + 1][i + 1], A[l][j + 1][i + 1]};
        float3 v = make_float3(0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int e = 0; e < 6; ++e) {
            v.x = v.x + t[e].x;
            v.y = v.y + t[e].y;
            v.z = v.z + t[e].z;
        }
        const float3 c = A[l + 1][j + 1][i + 1];
        const uint32_t p = uint32_t(z) * g.wh + uint32_t(y) * uint32_t(g.w) + uint32_t(x);
        const float3 o = make_float3(c.x * w_1 + v.x * w_6, c.y * w_1 + v.y * w_6, c.z * w_1 + v.z * w_6);
        st3(out, p, o);
        if (keep) st3(keep, p, ld3(cur, p));
        if (Js) Js[p] = composed(Is, g, x, y, z, p, o);
    }
}

// Outputs per block of accumulate_smooth_kernel: large volumes take the tile
// with fewer faces (1.5 evaluations per output, not 2) and its staged field,
// small ones the tile with more workgroups, whose gathers are a shorter chain
// than staging first (5.1 against 8.0 us at 32x32x32).
template <bool LARGE>
struct AccTile {
    static constexpr int kX = LARGE ? 16 : 8, kY = LARGE ? 16 : 8, kZ = LARGE ? 8 : 4;
    static constexpr int kThreads = LARGE ? 512 : 256;
};
constexpr size_t kALargeVoxels = size_t(1) << 18;
inline bool acc_large(const FieldGeo& g) { return g.n >= kALargeVoxels; }

template <class Tile>
dim3 acc_grid_t(const FieldGeo& g)
{
    return dim3(uint32_t((g.w + Tile::kX - 1) / Tile::kX), uint32_t((g.h + Tile::kY - 1) / Tile::kY),
                uint32_t((g.d + Tile::kZ - 1) / Tile::kZ));
}
dim3 acc_grid(const FieldGeo& g)
{
    return acc_large(g) ? acc_grid_t<AccTile<true>>(g) : acc_grid_t<AccTile<false>>(g);
}

template <bool LARGE>
__global__ __launch_bounds__(AccTile<LARGE>::kThreads, 4) void accumulate_smooth_kernel(
    const float* __restrict__ cur, const float* __restrict__ nd, Lay lay, float k, float w_6, float w_1,
    FieldGeo g, float* __restrict__ out, const uint8_t* __restrict__ Is, uint8_t* __restrict__ Js,
    float* __restrict__ keep)
{
    using T = AccTile<LARGE>;
    accumulate_smooth_body<T::kX, T::kY, T::kZ, T::kThreads, LARGE>(cur, nd, lay, k, w_6, w_1, g, out, keep, Is,
                                                             Js, logical_block());
}

// ---------------------------------------------------------------------------
// Multi-field launches.  One launch runs one step of the CDM iteration for
// up to kMaxSegs fields -- the concurrent registrations of a server, each
// with its own shape and buffers.  The launch's workgroups are the fields'
// grids one after another (field s from begin[s]); each workgroup finds its
// field and its logical block within the field's grid, and runs the same
// body as the single-field kernel, so every field's results, its block
// partials included, are those of a launch of its own.  The table travels
// as a kernel argument (no upload).
// ---------------------------------------------------------------------------
constexpr int kMaxSegs = 8;

struct CdmStep {
    uint32_t nseg = 0, total = 0;
    uint32_t begin[kMaxSegs];
    uint32_t gx[kMaxSegs], gy[kMaxSegs];
    int zq[kMaxSegs];
    FieldGeo g[kMaxSegs];
    const uint8_t* Is[kMaxSegs];
    const uint8_t* It[kMaxSegs];
    uint8_t* Js[kMaxSegs];
    const float* cur[kMaxSegs];
    float* nd[kMaxSegs];
    const float* src[kMaxSegs];  // Jacobi: the sweeps' input
    float* dst[kMaxSegs];        // Jacobi: output; accumulate+smooth: the new field
    float* keep[kMaxSegs];       // accumulate+smooth: receives cur when set
    double* partials[kMaxSegs];
    float* maxparts[kMaxSegs];
    float* cost[kMaxSegs];
    float* host_cost[kMaxSegs];
    unsigned* maxlen[kMaxSegs];
    unsigned* host_maxlen[kMaxSegs];
    uint32_t count[kMaxSegs];    // reductions: partials of the field
    double n[kMaxSegs];
    float k[kMaxSegs], w_6[kMaxSegs], w_1[kMaxSegs];
};
static_assert(sizeof(CdmStep) <= 4096, "CdmStep travels as a kernel argument (4 KB at most)");

// This workgroup's field s and logical block within the field's grid
// (hardware order remapped so that each XCD takes a contiguous range).
__device__ inline Block seg_block(const CdmStep& st, int& s)
{
    const uint32_t L = xcd_remap(blockIdx.x, st.total);
    int k = 0;
#pragma unroll
    for (int i = 1; i < kMaxSegs; ++i)
        if (uint32_t(i) < st.nseg && st.begin[i] <= L) k = i;
    s = k;
    const uint32_t local = L - st.begin[k];
    const uint32_t gx = st.gx[k], gy = st.gy[k];
    Block b;
    b.x = int(local % gx);
    b.y = int((local / gx) % gy);
    b.z = int(local / (gx * gy));
    b.lin = local;
    return b;
}

__global__ __launch_bounds__(256) void compose_seg_kernel(const CdmStep st)
{
    int s;
    const Block b = seg_block(st, s);
    compose_body(st.Is[s], st.cur[s], st.g[s], st.Js[s], b);
}

template <bool LARGE>
__global__ __launch_bounds__(GradTile<LARGE>::kThreads) void gradient_seg_kernel(const CdmStep st)
{
    using Tile = GradTile<LARGE>;
    int s;
    const Block b = seg_block(st, s);
    gradient_r_box_body<Tile::kSide, Tile::kSide, Tile::kThreads>(st.Js[s], st.It[s], st.g[s], 0, st.nd[s],
                                                                  packed_layout(), st.partials[s], b);
}

// one workgroup per field
__global__ __launch_bounds__(kReduceThreads) void cost_reduce_seg_kernel(const CdmStep st)
{
    __shared__ double part[kReduceThreads / 64];
    const int s = int(blockIdx.x);
    cost_reduce_body(CostReduce{st.partials[s], st.count[s], st.n[s], st.cost[s], st.host_cost[s]}, part);
}

template <bool FIRST, bool MAXLEN>
__global__ __launch_bounds__(kQX * kQY) void poisson2_seg_kernel(const CdmStep st)
{
    int s;
    const Block b = seg_block(st, s);
    poisson2_body<FIRST, MAXLEN>(st.nd[s], st.src[s], st.g[s], st.zq[s], st.dst[s], st.maxparts[s], b);
}

// one workgroup per field; fields without a max_len slot are skipped
__global__ __launch_bounds__(1024) void max_reduce_seg_kernel(const CdmStep st)
{
    const int s = int(blockIdx.x);
    if (!st.maxlen[s]) return;
    max_reduce_body(st.maxparts[s], st.count[s], st.maxlen[s], st.host_maxlen[s]);
}

template <bool LARGE>
__global__ __launch_bounds__(AccTile<LARGE>::kThreads, 4) void accumulate_smooth_seg_kernel(const CdmStep st)
{
    using T = AccTile<LARGE>;
    int s;
    const Block b = seg_block(st, s);
    accumulate_smooth_body<T::kX, T::kY, T::kZ, T::kThreads, LARGE>(st.cur[s], st.nd[s], packed_layout(), st.k[s],
                                                             st.w_6[s], st.w_1[s], st.g[s], st.dst[s],
                                                             st.keep[s], st.Is[s], st.Js[s], b);
}

// cdm_smooth: dd = d*(1-s) + (s/6)*(neighbours +1, -1, +w, -w, +wh, -wh by
// flat index, dropped at the array ends).
__global__ __launch_bounds__(256) void smooth_kernel(const float* __restrict__ d,
                                                     float* __restrict__ dd, float w_6, float w_1,
                                                     FieldGeo g)
{
    const Vox v = this_voxel(g);
    if (!v.ok) return;
    const uint32_t p = v.p, n = g.n, w = uint32_t(g.w), wh = g.wh;
    float3 s = make_float3(0.0f, 0.0f, 0.0f);
    auto add = [&](uint32_t q) {
        const float3 t = ld3(d, q);
        s.x = s.x + t.x;
        s.y = s.y + t.y;
        s.z = s.z + t.z;
    };
    if (p + 1u < n) add(p + 1u);
    if (p >= 1u) add(p - 1u);
    if (p + w < n) add(p + w);
    if (p >= w) add(p - w);
    if (p + wh < n) add(p + wh);
    if (p >= wh) add(p - wh);
    const float3 c = ld3(d, p);
    st3(dd, p, make_float3(c.x * w_1 + s.x * w_6, c.y * w_1 + s.y * w_6, c.z * w_1 + s.z * w_6));
}

// best_d *= 2 then upsample_with_padding<linear>: out(p) = in2(p * 0.5),
// 0 outside.
__global__ __launch_bounds__(256) void upsample_kernel(const float* __restrict__ in, FieldGeo gi,
                                                       FieldGeo go, float* __restrict__ out)
{
    const Vox v = this_voxel(go);
    if (!v.ok) return;
    float x = float(v.x), y = float(v.y), z = float(v.z);
    x = x * 0.5f;
    y = y * 0.5f;
    z = z * 0.5f;
    Tri t;
    float3 acc = make_float3(0.0f, 0.0f, 0.0f);
    if (locate(gi, x, y, z, t)) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            float3 m = ld3(in, corner(gi, t.i0, c));
            m.x = m.x * 2.0f;
            m.y = m.y * 2.0f;
            m.z = m.z * 2.0f;
            if (c == 0) {
                acc.x = m.x * t.w[0];
                acc.y = m.y * t.w[0];
                acc.z = m.z * t.w[0];
            } else {
                acc.x = acc.x + m.x * t.w[c];
                acc.y = acc.y + m.y * t.w[c];
                acc.z = acc.z + m.z * t.w[c];
            }
        }
    }
    st3(out, v.p, acc);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

// Scratch memory of one CDM call, stream-ordered on the context's stream.

void zero(tiplhip_ctx* ctx, void* p, size_t bytes)
{
    TIPLHIP_CHECK(hipMemsetAsync(p, 0, bytes, ctx->stream));
}

void copy_d2d(tiplhip_ctx* ctx, void* dst, const void* src, size_t bytes)
{
    TIPLHIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
}

// Partials of the largest launch that writes one per block (the 'd' gradient
// and the Jacobi kernels take tile_grid or fewer blocks, the 'r' gradient
// box_grid).
uint32_t block_count(const FieldGeo& g)
{
    const dim3 t = tile_grid(g), b = box_grid(g);
    return std::max(t.x * t.y * t.z, b.x * b.y * b.z);
}

void launch_compose(hipStream_t stream, const uint8_t* Is, const float* d, const FieldGeo& g,
                    uint8_t* Js)
{
    hipLaunchKernelGGL(compose_kernel, tile_grid(g), dim3(kTX, kTY), 0, stream, Is, d, g, Js);
    TIPLHIP_CHECK(hipGetLastError());
}

// Queues the sum of a gradient's cost partials.
void launch_cost_reduce(hipStream_t stream, const CostReduce& r)
{
    hipLaunchKernelGGL(cost_reduce_kernel, dim3(1), dim3(kReduceThreads), 0, stream, r);
    TIPLHIP_CHECK(hipGetLastError());
}

// Queues the gradient; the sum of its cost partials is left to the caller.
CostReduce launch_gradient(hipStream_t stream, const uint8_t* Js, const uint8_t* It, const FieldGeo& g,
                     char type, int accumulate, float* nd, Lay lay, double* partials, float* cost_out,
                     float* host_cost = nullptr)
{
    uint32_t parts;
    if (type == 'd') {
        hipLaunchKernelGGL(gradient_d_kernel, tile_grid(g), dim3(kTX, kTY), 0, stream, Js, It, g,
                           accumulate, nd, lay, partials);
        const dim3 tg = tile_grid(g);
        parts = tg.x * tg.y * tg.z;
    } else {
        const dim3 bg = box_grid(g);
        if (grad_large(g))
            hipLaunchKernelGGL(gradient_r_box_kernel<true>, bg, dim3(GradTile<true>::kThreads), 0,
                               stream, Js, It, g, accumulate, nd, lay, partials);
        else
            hipLaunchKernelGGL(gradient_r_box_kernel<false>, bg, dim3(GradTile<false>::kThreads), 0,
                               stream, Js, It, g, accumulate, nd, lay, partials);
        parts = bg.x * bg.y * bg.z;
    }
    TIPLHIP_CHECK(hipGetLastError());
    return CostReduce{partials, parts, double(g.n), cost_out, host_cost};
}

// `sweeps` Jacobi sweeps: all in one launch for the smallest volumes
// (poisson_whole_kernel), four per launch else (poisson4_kernel for small
// volumes, poisson_march_kernel for large ones); of a packed field also the
// remainder, and all of a volume whose byte offsets pass 2^31, by two
// (poisson2_kernel) and one (the z-marching sweep).  Returns the buffer holding
// the result.  With maxlen, per-block maxima of the displacement length (from
// the last launch, or a pass of their own after a four-sweep one) are reduced by
// max_reduce_kernel.
float* launch_poisson(hipStream_t stream, const float* nd, float* a, float* b, const FieldGeo& g, Lay lay,
                      int sweeps, unsigned int* maxlen, float* maxparts,
                      const CostReduce& cost = CostReduce{}, unsigned int* host_maxlen = nullptr)
{
    // a gradient's cost partials, when given, are summed by one more workgroup
    // of the first launch
    const uint32_t extra = cost.partials ? 1u : 0u;
    float* src = a;
    float* dst = b;
    uint32_t last_blocks = 0;
    int done = 0;
    while (done < sweeps) {
        const bool first = done == 0;
        if (poisson_whole_fits(g)) {
            hipLaunchKernelGGL(poisson_whole_kernel, dim3(3u + extra), dim3(kWThreads), 0, stream, nd,
                               g, lay, sweeps, dst, cost);
            TIPLHIP_CHECK(hipGetLastError());
            done = sweeps;
            if (maxlen) {
                last_blocks = std::min(kMaxLenBlocks, block_count(g));
                hipLaunchKernelGGL(max_length_kernel, dim3(last_blocks), dim3(256), 0, stream, dst,
                                   g.n, lay, maxparts);
                TIPLHIP_CHECK(hipGetLastError());
            }
            std::swap(src, dst);
            continue;
        }
        if (sweeps - done >= kCH && poisson4_fits(g)) {
            const dim3 block(kCThreads);
            const uint32_t blocks = poisson4_blocks(g);
            if (first)
                hipLaunchKernelGGL(poisson4_kernel<true>, dim3(blocks + extra), block, 0, stream, nd,
                                   src, g, lay, dst, cost);
            else
                hipLaunchKernelGGL(poisson4_kernel<false>, dim3(blocks), block, 0, stream, nd, src, g,
                                   lay, dst, CostReduce{});
            TIPLHIP_CHECK(hipGetLastError());
            done += kCH;
            if (done == sweeps && maxlen) {
                last_blocks = std::min(kMaxLenBlocks, block_count(g));
                hipLaunchKernelGGL(max_length_kernel, dim3(last_blocks), dim3(256), 0, stream, dst,
                                   g.n, lay, maxparts);
                TIPLHIP_CHECK(hipGetLastError());
            }
            std::swap(src, dst);
            continue;
        }
        if (sweeps - done >= kMK && planar_fits(g)) {
            const March mg = march_of<kMK>(g);
            const dim3 block(kMThreads);
            if (first)
                hipLaunchKernelGGL((poisson_march_kernel<kMK, true>), dim3(mg.blocks + extra), block, 0,
                                   stream, nd, src, g, mg, lay, dst, cost);
            else
                hipLaunchKernelGGL((poisson_march_kernel<kMK, false>), dim3(mg.blocks), block, 0,
                                   stream, nd, src, g, mg, lay, dst, CostReduce{});
            TIPLHIP_CHECK(hipGetLastError());
            done += kMK;
            if (done == sweeps && maxlen) {
                last_blocks = std::min(kMaxLenBlocks, block_count(g));
                hipLaunchKernelGGL(max_length_kernel, dim3(last_blocks), dim3(256), 0, stream, dst,
                                   g.n, lay, maxparts);
                TIPLHIP_CHECK(hipGetLastError());
            }
            std::swap(src, dst);
            continue;
        }
        if (first && extra) launch_cost_reduce(stream, cost);
        TIPLHIP_REQUIRE(lay.ps == 3u, "one- and two-sweep launches take packed fields");
        const bool pair = sweeps - done >= 2;
        const bool last = done + (pair ? 2 : 1) == sweeps && maxlen;
        if (pair) {
            const int zq = poisson2_zq(g);
            const dim3 grid = poisson2_grid(g, zq), block(kQX, kQY);
            if (first && last)
                hipLaunchKernelGGL((poisson2_kernel<true, true>), grid, block, 0, stream, nd, src,
                                   g, zq, dst, maxparts);
            else if (first)
                hipLaunchKernelGGL((poisson2_kernel<true, false>), grid, block, 0, stream, nd,
                                   src, g, zq, dst, maxparts);
            else if (last)
                hipLaunchKernelGGL((poisson2_kernel<false, true>), grid, block, 0, stream, nd,
                                   src, g, zq, dst, maxparts);
            else
                hipLaunchKernelGGL((poisson2_kernel<false, false>), grid, block, 0, stream, nd,
                                   src, g, zq, dst, maxparts);
            last_blocks = grid.x * grid.y * grid.z;
            done += 2;
        } else {
            const dim3 grid = poisson_grid(g), block(kTX, kPTY);
            if (first && last)
                hipLaunchKernelGGL((poisson_zm_kernel<true, true>), grid, block, 0, stream, nd,
                                   src, g, dst, maxparts);
            else if (first)
                hipLaunchKernelGGL((poisson_zm_kernel<true, false>), grid, block, 0, stream, nd,
                                   src, g, dst, maxparts);
            else if (last)
                hipLaunchKernelGGL((poisson_zm_kernel<false, true>), grid, block, 0, stream, nd,
                                   src, g, dst, maxparts);
            else
                hipLaunchKernelGGL((poisson_zm_kernel<false, false>), grid, block, 0, stream, nd,
                                   src, g, dst, maxparts);
            last_blocks = grid.x * grid.y * grid.z;
            done += 1;
        }
        TIPLHIP_CHECK(hipGetLastError());
        std::swap(src, dst);
    }
    if (maxlen) {
        hipLaunchKernelGGL(max_reduce_kernel, dim3(1), dim3(1024), 0, stream, maxparts,
                           last_blocks, maxlen, host_maxlen);
        TIPLHIP_CHECK(hipGetLastError());
    }
    return src;
}

void launch_accumulate(hipStream_t stream, const float* cur, const float* nd, Lay lay, float k,
                       const FieldGeo& g, float* out, Lay out_lay)
{
    hipLaunchKernelGGL(accumulate_kernel, tile_grid(g), dim3(kTX, kTY), 0, stream, cur, nd, lay, k, g,
                       out, out_lay);
    TIPLHIP_CHECK(hipGetLastError());
}

// cdm_smooth's weight of a neighbour.
inline float smooth_w6(float smoothing) { return smoothing / float(2.0f * 3.0f); }

void launch_smooth(hipStream_t stream, const float* d, float* dd, float smoothing, const FieldGeo& g)
{
    const float w_6 = smooth_w6(smoothing), w_1 = 1.0f - smoothing;
    hipLaunchKernelGGL(smooth_kernel, tile_grid(g), dim3(kTX, kTY), 0, stream, d, dd, w_6, w_1, g);
    TIPLHIP_CHECK(hipGetLastError());
}

// accumulate then cdm_smooth with `smoothing` (non-zero) into out, and where
// the one-pass kernel runs compose_displacement of Is by out into Js, if Js is
// set; returns whether it did.  That kernel addresses the packed field in 32
// bits: a field of 2^32 bytes and more takes the two kernels it replaces, whose
// addresses are 64 bits wide, and nd (packed there) is overwritten.
bool launch_accumulate_smooth(hipStream_t stream, const float* cur, float* nd, Lay lay, float k,
                              float smoothing, const FieldGeo& g, float* out, const uint8_t* Is, uint8_t* Js,
                              float* keep = nullptr)
{
    if (!field_fits_32(g.n)) {
        launch_accumulate(stream, cur, nd, lay, k, g, nd, lay);
        launch_smooth(stream, nd, out, smoothing, g);
        return false;
    }
    const float w_6 = smooth_w6(smoothing), w_1 = 1.0f - smoothing;
    if (acc_large(g))
        hipLaunchKernelGGL(accumulate_smooth_kernel<true>, acc_grid(g), dim3(AccTile<true>::kThreads), 0,
                           stream, cur, nd, lay, k, w_6, w_1, g, out, Is, Js, keep);
    else
        hipLaunchKernelGGL(accumulate_smooth_kernel<false>, acc_grid(g), dim3(AccTile<false>::kThreads), 0,
                           stream, cur, nd, lay, k, w_6, w_1, g, out, Is, Js, keep);
    TIPLHIP_CHECK(hipGetLastError());
    return Js != nullptr;
}

void launch_upsample(hipStream_t stream, const float* in, const FieldGeo& gi, const FieldGeo& go,
                     float* out)
{
    hipLaunchKernelGGL(upsample_kernel, tile_grid(go), dim3(kTX, kTY), 0, stream, in, gi, go, out);
    TIPLHIP_CHECK(hipGetLastError());
}

struct CdmRun {
    tiplhip_ctx* ctx;
    tiplhip_cdm_param param;
    int nmod;
    const volatile uint8_t* terminated;
    int iterations = 0;
    bool no_early_exit = false;  // timing mode: run max_iterations exactly
    bool stopped = false;        // terminated by the caller
};

bool is_terminated(const CdmRun& r) { return r.terminated && *r.terminated; }

// ---------------------------------------------------------------------------
// Batched CDM iterations (the serving loop).  A registration whose context
// is attached to a CdmBatcher hands the device work of each iteration of its
// cdm() level loop to the batcher as one step; the batcher launches the
// steps of up to kMaxSegs registrations together, one *_seg launch per
// kernel, on its own stream.  Each registration keeps its own host control
// (cost history, cdm_improved, smoothing schedule) and each field's results
// are those of launches of its own, so a batched cdm() equals a plain one
// bit for bit.
// ---------------------------------------------------------------------------

// One registration's level loop as the batcher sees it.  The owner sets
// the step fields before CdmBatcher::run; the launch reads them under the
// gate's lock.
struct CdmJob : GateSlot {
    FieldGeo g{};
    dim3 tile, box, p2, acc;  // grids: compose, gradient, Jacobi, accumulate+smooth
    int zq_p2 = 0;
    const uint8_t* It = nullptr;
    const uint8_t* Is = nullptr;
    uint8_t* Js = nullptr;
    float* nd = nullptr;
    float* best = nullptr;
    float* cur = nullptr;     // the running field the iteration body reads
    float* pa = nullptr;      // Jacobi buffers: the solved new_d ends in pa
    float* pb = nullptr;
    double* partials = nullptr;
    float* maxparts = nullptr;
    float* d_cost = nullptr;
    unsigned* d_maxlen = nullptr;
    float* h_cost = nullptr;  // coherent host slots (device addresses)
    unsigned* h_maxlen = nullptr;
    hipEvent_t ready = nullptr;  // on the owner's stream: the level's inputs are written
    hipEvent_t done = nullptr;   // on the batch stream: the job's last step
    bool waited = false;         // the lane's stream has waited for `ready`
    int lane = 0;                // the batcher lane the job joined
    // the step: accumulate+smooth from s_src into s_out (s_keep <- s_src when
    // set) or plain copies, then the iteration body on cur
    bool smooth = false;
    const float* s_src = nullptr;
    float* s_nd = nullptr;
    float* s_out = nullptr;
    float* s_keep = nullptr;
    float k = 0.0f, smoothing = 0.0f;
    bool copy_best = false;   // without smoothing: best <- cur, then
    bool restore = false;     // cur <- best
    bool need_theta = false;  // the last Jacobi launch forms max_len
};

// Fills the workgroup ranges of a multi-field launch from one grid per field.
void set_grids(CdmStep& st, CdmJob* const* J, int n, dim3 CdmJob::*grid)
{
    uint32_t total = 0;
    for (int s = 0; s < n; ++s) {
        const dim3 d = J[s]->*grid;
        st.begin[s] = total;
        st.gx[s] = d.x;
        st.gy[s] = d.y;
        const uint64_t t = uint64_t(total) + uint64_t(d.x) * d.y * d.z;
        TIPLHIP_REQUIRE(t < (uint64_t(1) << 31), "batched CDM launch too large");
        total = uint32_t(t);
    }
    st.total = total;
}

// The step of a job that is alone in its batch (its copies are queued): the
// launches cdm_level makes, on packed fields.  Three to five of them instead of
// nine, whose sweeps take half the time (17 against 44 us at 32x32x32); most
// batches have one field unless the slots outnumber the lanes several times.
void launch_cdm_step_alone(hipStream_t stream, CdmJob& j)
{
    const Lay lay = packed_layout();
    if (j.smooth)
        launch_accumulate_smooth(stream, j.s_src, j.s_nd, lay, j.k, j.smoothing, j.g, j.s_out, j.Is, j.Js,
                                 j.s_keep);
    else
        launch_compose(stream, j.Is, j.cur, j.g, j.Js);
    const CostReduce reduce =
        launch_gradient(stream, j.Js, j.It, j.g, 'r', 0, j.nd, lay, j.partials, j.d_cost, j.h_cost);
    const float* solved = launch_poisson(stream, j.nd, j.pa, j.pb, j.g, lay, 12,
                                         j.need_theta ? j.d_maxlen : nullptr, j.maxparts, reduce, j.h_maxlen);
    if (solved != j.pa) std::swap(j.pa, j.pb);  // (the next step reads pa)
}

// Queues one step of every job in J (at most kMaxSegs) on `stream`, in the
// order of the reference's loop body: the previous iteration's update of the
// running field (reg/cdm.hpp:447-469), then compose_displacement, the
// gradient and cost, and cdm_solve_poisson's 12 sweeps (reg/cdm.hpp:420-462),
// exactly as cdm_level queues them for one field.
void launch_cdm_steps(hipStream_t stream, CdmJob* const* J, int n)
{
    TIPLHIP_REQUIRE(n >= 1 && n <= kMaxSegs, "1 to 8 fields per batched CDM step");
    for (int s = 0; s < n; ++s) {
        CdmJob& j = *J[s];
        if (!j.waited) {
            TIPLHIP_CHECK(hipStreamWaitEvent(stream, j.ready, 0));
            j.waited = true;
        }
        if (j.smooth) continue;
        const size_t fb = sizeof(float) * 3 * j.g.n;
        if (j.copy_best)
            TIPLHIP_CHECK(hipMemcpyAsync(j.best, j.cur, fb, hipMemcpyDeviceToDevice, stream));
        if (j.restore)
            TIPLHIP_CHECK(hipMemcpyAsync(j.cur, j.best, fb, hipMemcpyDeviceToDevice, stream));
    }
    if (n == 1) {
        launch_cdm_step_alone(stream, *J[0]);
        return;
    }
    // the field update of the jobs that have one, compose_displacement
    // included; one launch per tile shape among them
    for (const bool large : {false, true}) {
        CdmStep st;
        CdmJob* sm[kMaxSegs];
        int m = 0;
        for (int s = 0; s < n; ++s)
            if (J[s]->smooth && acc_large(J[s]->g) == large) sm[m++] = J[s];
        if (!m) continue;
        st.nseg = uint32_t(m);
        set_grids(st, sm, m, &CdmJob::acc);
        for (int s = 0; s < m; ++s) {
            const CdmJob& j = *sm[s];
            st.g[s] = j.g;
            st.cur[s] = j.s_src;
            st.nd[s] = j.s_nd;
            st.dst[s] = j.s_out;
            st.keep[s] = j.s_keep;
            st.Is[s] = j.Is;
            st.Js[s] = j.Js;
            st.k[s] = j.k;
            st.w_6[s] = smooth_w6(j.smoothing);
            st.w_1[s] = 1.0f - j.smoothing;
        }
        if (large)
            hipLaunchKernelGGL(accumulate_smooth_seg_kernel<true>, dim3(st.total),
                               dim3(AccTile<true>::kThreads), 0, stream, st);
        else
            hipLaunchKernelGGL(accumulate_smooth_seg_kernel<false>, dim3(st.total),
                               dim3(AccTile<false>::kThreads), 0, stream, st);
        TIPLHIP_CHECK(hipGetLastError());
    }
    // compose_displacement of the jobs whose field was not just updated
    {
        CdmStep st;
        CdmJob* cj[kMaxSegs];
        int m = 0;
        for (int s = 0; s < n; ++s)
            if (!J[s]->smooth) cj[m++] = J[s];
        if (m) {
            st.nseg = uint32_t(m);
            set_grids(st, cj, m, &CdmJob::tile);
            for (int s = 0; s < m; ++s) {
                st.g[s] = cj[s]->g;
                st.Is[s] = cj[s]->Is;
                st.Js[s] = cj[s]->Js;
                st.cur[s] = cj[s]->cur;
            }
            hipLaunchKernelGGL(compose_seg_kernel, dim3(st.total), dim3(kTX, kTY), 0, stream, st);
            TIPLHIP_CHECK(hipGetLastError());
        }
    }
    CdmStep st;
    st.nseg = uint32_t(n);
    bool theta = false;
    for (int s = 0; s < n; ++s) {
        const CdmJob& j = *J[s];
        st.g[s] = j.g;
        st.Is[s] = j.Is;
        st.It[s] = j.It;
        st.Js[s] = j.Js;
        st.cur[s] = j.cur;
        st.nd[s] = j.nd;
        st.partials[s] = j.partials;
        st.maxparts[s] = j.maxparts;
        st.cost[s] = j.d_cost;
        st.host_cost[s] = j.h_cost;
        st.maxlen[s] = j.need_theta ? j.d_maxlen : nullptr;
        st.host_maxlen[s] = j.h_maxlen;
        st.n[s] = double(j.g.n);
        theta = theta || j.need_theta;
    }
    // one gradient launch per tile shape among the fields
    for (const bool large : {false, true}) {
        CdmStep gs;
        CdmJob* gj[kMaxSegs];
        int m = 0;
        for (int s = 0; s < n; ++s)
            if (grad_large(J[s]->g) == large) gj[m++] = J[s];
        if (!m) continue;
        gs.nseg = uint32_t(m);
        set_grids(gs, gj, m, &CdmJob::box);
        for (int s = 0; s < m; ++s) {
            gs.g[s] = gj[s]->g;
            gs.It[s] = gj[s]->It;
            gs.Js[s] = gj[s]->Js;
            gs.nd[s] = gj[s]->nd;
            gs.partials[s] = gj[s]->partials;
        }
        if (large)
            hipLaunchKernelGGL(gradient_seg_kernel<true>, dim3(gs.total), dim3(GradTile<true>::kThreads), 0,
                               stream, gs);
        else
            hipLaunchKernelGGL(gradient_seg_kernel<false>, dim3(gs.total), dim3(GradTile<false>::kThreads),
                               0, stream, gs);
        TIPLHIP_CHECK(hipGetLastError());
    }
    for (int s = 0; s < n; ++s) st.count[s] = J[s]->box.x * J[s]->box.y * J[s]->box.z;
    hipLaunchKernelGGL(cost_reduce_seg_kernel, dim3(st.nseg), dim3(kReduceThreads), 0, stream, st);
    TIPLHIP_CHECK(hipGetLastError());
    set_grids(st, J, n, &CdmJob::p2);
    for (int s = 0; s < n; ++s) {
        st.zq[s] = J[s]->zq_p2;
        st.count[s] = J[s]->p2.x * J[s]->p2.y * J[s]->p2.z;
    }
    // 12 sweeps, two per launch: launch i reads pa (i even) or pb and writes
    // the other, so the solution ends in pa
    for (int i = 0; i < 6; ++i) {
        for (int s = 0; s < n; ++s) {
            st.src[s] = (i & 1) ? J[s]->pb : J[s]->pa;
            st.dst[s] = (i & 1) ? J[s]->pa : J[s]->pb;
        }
        const dim3 grid(st.total), block(kQX, kQY);
        if (i == 0)
            hipLaunchKernelGGL((poisson2_seg_kernel<true, false>), grid, block, 0, stream, st);
        else if (i == 5 && theta)
            hipLaunchKernelGGL((poisson2_seg_kernel<false, true>), grid, block, 0, stream, st);
        else
            hipLaunchKernelGGL((poisson2_seg_kernel<false, false>), grid, block, 0, stream, st);
        TIPLHIP_CHECK(hipGetLastError());
    }
    if (theta) {
        hipLaunchKernelGGL(max_reduce_seg_kernel, dim3(st.nseg), dim3(1024), 0, stream, st);
        TIPLHIP_CHECK(hipGetLastError());
    }
}

}  // namespace

// The batch executor of one device: `lanes` streams, each with a StepGate
// (at most kMaxSegs fields a batch, kGatherUs); a job keeps the lane it
// joined (the one with the fewest members), whose stream orders its steps.
// Levels above max_voxels run unbatched on their owner's stream: a batch is
// held to the pace of its largest field, and only a field of its own stream has
// the planar gradient field of the marched sweeps, which larger levels take.
// Measured on 32 uneven affine+CDM pairs (pairs/s, medians of six runs, which
// spread by 3 to 5), unbatched, then up to 2^18 voxels on 2, 3 and 4 lanes:
// 4 slots 71.0, 70.4, 70.6, 71.9; 8 slots 85.8, 84.8, 85.0, 84.2; 16 slots
// 89.7, 90.3, 91.1, 89.5; 32 slots 85.6, 84.2, 85.2, 85.5; 6 slots with both
// directions 53.4, 53.7, 55.2, 54.3.  Lines at 4096 and 70000 voxels on 16 slots
// and 4 lanes: 91.3, 88.4 (2^18: 91.2).  While a batch of one field took the
// batch's launches too, 4 lanes gave 64.4 on 4 slots, 78.0 on 8 and 87.6 on 16.
class CdmBatcher {
public:
    static constexpr int kGatherUs = 300;
    static constexpr int kDefaultLanes = 3;
    static constexpr size_t kDefaultMaxVoxels = size_t(1) << 18;

    CdmBatcher(int device, int lanes, size_t max_voxels) : device_(device), max_voxels_(max_voxels)
    {
        TIPLHIP_REQUIRE(lanes >= 1 && lanes <= 16, "1 to 16 CDM batch lanes");
        DeviceGuard dg(device);
        lanes_.resize(size_t(lanes));
        for (Lane& l : lanes_) {
            const hipError_t e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
            if (e != hipSuccess) {
                destroy_streams();  // the destructor does not run for a throwing constructor
                TIPLHIP_CHECK(e);
            }
            hipStream_t st = l.stream;
            l.gate.reset(new StepGate<CdmJob>(kMaxSegs, std::chrono::microseconds(kGatherUs),
                                              [this, st](CdmJob* const* J, int n) {
                                                  DeviceGuard g(device_);
                                                  launch_cdm_steps(st, J, n);
                                              }));
        }
    }
    ~CdmBatcher() { destroy_streams(); }
    CdmBatcher(const CdmBatcher&) = delete;
    CdmBatcher& operator=(const CdmBatcher&) = delete;

    int device() const { return device_; }
    size_t max_voxels() const { return max_voxels_; }
    hipStream_t stream(int lane) const { return lanes_[size_t(lane)].stream; }
    // Makes j a member of the least occupied lane; returns the lane.
    int join(CdmJob& j)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            size_t best = 0;
            for (size_t i = 1; i < lanes_.size(); ++i)
                if (lanes_[i].members < lanes_[best].members) best = i;
            ++lanes_[best].members;
            j.lane = int(best);
        }
        lanes_[size_t(j.lane)].gate->join();
        return j.lane;
    }
    // After the job's last step: the owner's stream waits for the lane's
    // stream, so the owner's later work and frees follow every step.
    void leave(CdmJob& j, hipStream_t owner)
    {
        Lane& l = lanes_[size_t(j.lane)];
        l.gate->leave([&] {
            TIPLHIP_CHECK(hipEventRecord(j.done, l.stream));
            TIPLHIP_CHECK(hipStreamWaitEvent(owner, j.done, 0));
        });
        std::lock_guard<std::mutex> lk(mu_);
        --l.members;
    }
    // Queues j's step; returns once it is launched (rethrows its launch error).
    // A failed launch fails every job of its batch: their steps may be partly
    // queued.
    void run(CdmJob& j) { lanes_[size_t(j.lane)].gate->run(j); }
    int64_t launches() const
    {
        int64_t n = 0;
        for (const Lane& l : lanes_) n += l.gate->batches();
        return n;
    }
    int64_t fields() const
    {
        int64_t n = 0;
        for (const Lane& l : lanes_) n += l.gate->steps();
        return n;
    }

private:
    struct Lane {
        hipStream_t stream = nullptr;
        std::unique_ptr<StepGate<CdmJob>> gate;
        int members = 0;
    };
    void destroy_streams()
    {
        int prev = -1;
        (void)hipGetDevice(&prev);
        (void)hipSetDevice(device_);
        for (Lane& l : lanes_) {
            if (!l.stream) continue;
            (void)hipStreamSynchronize(l.stream);
            (void)hipStreamDestroy(l.stream);
            l.stream = nullptr;
        }
        if (prev >= 0) (void)hipSetDevice(prev);
    }
    int device_;
    size_t max_voxels_;
    std::mutex mu_;
    std::vector<Lane> lanes_;
};

void cdm_batcher_counts(const CdmBatcher& b, int64_t* steps, int64_t* fields)
{
    *steps = b.launches();
    *fields = b.fields();
}

bool cdm_batching_enabled()
{
    const char* e = std::getenv("TIPLHIP_SERVER_CDM_BATCH");
    return !(e && e[0] == '0');
}

// TIPLHIP_CDM_LANES and TIPLHIP_CDM_BATCH_VOXELS, read when a device's
// batcher is created, override the lane count and the largest batched level.
std::shared_ptr<CdmBatcher> shared_cdm_batcher(int device)
{
    static std::mutex mu;
    static std::map<int, std::weak_ptr<CdmBatcher>> live;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<CdmBatcher> b = live[device].lock();
    if (!b) {
        int lanes = CdmBatcher::kDefaultLanes;
        size_t max_voxels = CdmBatcher::kDefaultMaxVoxels;
        if (const char* e = std::getenv("TIPLHIP_CDM_LANES")) lanes = std::atoi(e);
        if (const char* e = std::getenv("TIPLHIP_CDM_BATCH_VOXELS")) max_voxels = size_t(std::atoll(e));
        b = std::make_shared<CdmBatcher>(device, lanes, max_voxels);
        live[device] = b;
    }
    return b;
}

namespace {

// A job's membership of the batcher for one level: events created, `ready`
// recorded on the owner's stream and the job counted active; leave() (or
// the destructor) ends it.
struct CdmMembership {
    CdmBatcher& b;
    CdmJob& j;
    hipStream_t owner;
    bool joined = false;
    CdmMembership(CdmBatcher& batcher, CdmJob& job, hipStream_t s) : b(batcher), j(job), owner(s)
    {
        TIPLHIP_CHECK(hipEventCreateWithFlags(&j.ready, hipEventDisableTiming));
        TIPLHIP_CHECK(hipEventCreateWithFlags(&j.done, hipEventDisableTiming));
        TIPLHIP_CHECK(hipEventRecord(j.ready, owner));
        b.join(j);
        joined = true;
    }
    void leave()
    {
        if (!joined) return;
        joined = false;
        b.leave(j, owner);
    }
    ~CdmMembership()
    {
        try {
            leave();
        } catch (...) {
            // the lane is drained before the owner's buffers are freed
            (void)hipStreamSynchronize(b.stream(j.lane));
        }
        if (j.ready) (void)hipEventDestroy(j.ready);
        if (j.done) (void)hipEventDestroy(j.done);
    }
};

// cdm_level's iteration loop for one modality with the 'r' gradient, its
// device work run as batched steps.  The host control is cdm_level's, line
// for line; a decision's copies and the field update are queued with the
// next iteration's body (fused into accumulate+smooth where there is one).
bool cdm_iterate_batched(CdmRun& run, const uint8_t* It, const uint8_t* Is, const FieldGeo& g,
                         float* best_d)
{
    tiplhip_ctx* ctx = run.ctx;
    CdmBatcher& batch = *ctx->cdm_batch;
    TIPLHIP_REQUIRE(batch.device() == ctx->device, "CDM batcher of another device");
    const size_t fb = sizeof(float) * 3 * g.n;
    DevMem f0(ctx, fb), f1(ctx, fb), f2(ctx, fb), nd(ctx, fb), Js(ctx, g.n);
    const uint32_t nblocks = block_count(g);
    DevMem partials(ctx, sizeof(double) * nblocks), maxparts(ctx, sizeof(float) * nblocks);
    DevMem scal(ctx, sizeof(float) * 16 + sizeof(unsigned int));
    ctx->h_cdm.reserve(sizeof(float) * 16);
    uint32_t* slots = ctx->h_cdm.as<uint32_t>();

    CdmJob job;
    job.g = g;
    job.tile = tile_grid(g);
    job.box = box_grid(g);
    job.zq_p2 = poisson2_zq(g);
    job.p2 = poisson2_grid(g, job.zq_p2);
    job.acc = acc_grid(g);
    job.It = It;
    job.Is = Is;
    job.Js = Js.as<uint8_t>();
    job.nd = nd.as<float>();
    job.best = best_d;
    job.cur = f0.as<float>();
    job.pa = f1.as<float>();
    job.pb = f2.as<float>();
    job.partials = partials.as<double>();
    job.maxparts = maxparts.as<float>();
    job.d_cost = scal.as<float>();
    job.d_maxlen = reinterpret_cast<unsigned int*>(scal.as<float>() + 16);
    job.h_cost = static_cast<float*>(ctx->h_cdm.dev);
    job.h_maxlen = static_cast<unsigned int*>(ctx->h_cdm.dev) + 1;
    copy_d2d(ctx, job.cur, best_d, fb);

    CdmMembership member(batch, job, ctx->stream);
    // kernels of this job may be queued on either stream when a step throws
    const hipStream_t lane = batch.stream(job.lane);
    auto drain = [ctx, lane] {
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipStreamSynchronize(lane);
    };
    DrainOnUnwind<decltype(drain)> unwind(drain);
    auto sync_batch = [lane] { TIPLHIP_CHECK(hipStreamSynchronize(lane)); };

    float theta = 0.0f;
    std::vector<float> cost;
    float best_cost = 3.402823466e+38f;
    float cur_smoothing = 0.8f;
    // the last decision, carried out with the next step
    bool copy_best = false, restore = false, update = false;
    bool failed = false;
    float k = 0.0f;
    for (int index = 0; index < run.param.max_iterations; ++index) {
        if (is_terminated(run)) {
            run.stopped = true;
            break;
        }
        ++run.iterations;
        job.smooth = update && cur_smoothing != 0.0f;
        job.copy_best = job.restore = false;
        if (job.smooth) {
            // accumulate+smooth of the running field (best when it was
            // reset to it; best <- cur fused in) into the spare buffer,
            // which becomes the running field
            job.s_src = (restore && !copy_best) ? job.best : job.cur;
            job.s_keep = copy_best ? job.best : nullptr;
            job.s_nd = job.pa;
            job.s_out = job.pb;
            job.k = k;
            job.smoothing = cur_smoothing;
            float* spare = job.pb;
            job.pb = job.pa;
            job.pa = job.cur;
            job.cur = spare;
        } else {
            job.copy_best = copy_best;
            job.restore = restore;
        }
        copy_best = restore = update = false;
        job.need_theta = theta == 0.0f;
        slots[0] = kCostPending;
        slots[1] = kCostPending;
        batch.run(job);
        wait_for_slots(static_cast<const volatile uint32_t*>(slots), 1, kCostPending,
                       std::chrono::microseconds(kCostSpinUs), sync_batch);
        float sum_cost = 0.0f;
        std::memcpy(&sum_cost, &slots[0], sizeof(float));
        // zero cost: cdm() fails (its step's later kernels still run, and
        // may store into the slots: the exit below waits for them)
        if (sum_cost == 0.0f) {
            failed = true;
            break;
        }
        cost.push_back(sum_cost);
        if (cost.back() < best_cost) {
            best_cost = cost.back();
            if (index) copy_best = true;
        }
        if (!cdm_improved(cost)) {
            if (cur_smoothing <= run.param.smoothing) break;
            restore = true;
            cur_smoothing *= 0.5f;
            cost.clear();
        }
        if (job.need_theta) {
            wait_for_slots(static_cast<const volatile uint32_t*>(slots + 1), 1, kCostPending,
                           std::chrono::microseconds(kCostSpinUs), sync_batch);
            std::memcpy(&theta, &slots[1], sizeof(theta));
        }
        if (theta == 0.0f) break;
        k = run.param.speed / theta;
        update = true;
    }
    member.leave();
    // a decision not yet carried out: only its best <- cur matters now
    if (copy_best && !failed) copy_d2d(ctx, best_d, job.cur, fb);
    // every step has finished (and stored into the slots) before the
    // context's next call resets them
    TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    return !failed;
}

// One cdm() call at shape dim.  best_d is a zeroed device field of vox(dim).
bool cdm_level(CdmRun& run, const std::vector<const uint8_t*>& It,
               const std::vector<const uint8_t*>& Is, const int* dim, float* best_d,
               float resolution)
{
    tiplhip_ctx* ctx = run.ctx;
    const FieldGeo g = field_geo(dim);
    const size_t n = g.n, fb = sizeof(float) * 3 * n;
    if (!run.no_early_exit && std::min({dim[0], dim[1], dim[2]}) > run.param.min_dimension) {
        const int rd[3] = {(dim[0] + 1) / 2, (dim[1] + 1) / 2, (dim[2] + 1) / 2};
        const size_t rn = vox(rd);
        DevMem rbuf(ctx, 2 * size_t(run.nmod) * rn);
        std::vector<const uint8_t*> rIt, rIs;
        for (int i = 0; i < run.nmod; ++i) {
            uint8_t* t = rbuf.as<uint8_t>() + size_t(2 * i) * rn;
            uint8_t* s = rbuf.as<uint8_t>() + size_t(2 * i + 1) * rn;
            launch_downsample_u8(ctx, It[size_t(i)], dim, t);
            launch_downsample_u8(ctx, Is[size_t(i)], dim, s);
            rIt.push_back(t);
            rIs.push_back(s);
        }
        DevMem rbest(ctx, sizeof(float) * 3 * rn);
        zero(ctx, rbest.p, sizeof(float) * 3 * rn);
        if (!cdm_level(run, rIt, rIs, rd, rbest.as<float>(), resolution / 2.0f)) return false;
        launch_upsample(ctx->stream, rbest.as<float>(), field_geo(rd), g, best_d);
        if (resolution > 1.0f) return true;
    }
    if (run.stopped) return true;
    if (run.ctx->cdm_batch && run.nmod == 1 && run.param.gradient_type[0] != 'd' &&
        !run.no_early_exit && n <= run.ctx->cdm_batch->max_voxels() && field_fits_32(n))
        return cdm_iterate_batched(run, It[0], Is[0], g, best_d);

    // four fields rotate: the running field, the best field so far -- which may
    // be the running one: then `spare_field` holds the fourth -- and the two
    // Jacobi buffers.  accumulate+smooth writes the new running field into the
    // Jacobi buffer that does not hold the solved new_d.
    DevMem f0(ctx, fb), f1(ctx, fb), f2(ctx, fb), nd(ctx, fb), Js(ctx, n);
    float* cur = best_d;
    float* best = best_d;
    float* pa = f0.as<float>();
    float* pb = f1.as<float>();
    float* spare_field = f2.as<float>();
    const uint32_t nblocks = block_count(g);
    DevMem partials(ctx, sizeof(double) * nblocks), maxparts(ctx, sizeof(float) * nblocks);
    DevMem scal(ctx, sizeof(float) * 16 + sizeof(unsigned int));
    const Lay lay = grad_layout(g);
    float* d_cost = scal.as<float>();
    unsigned int* d_maxlen = reinterpret_cast<unsigned int*>(scal.as<float>() + 16);
    // the cost reductions store into ctx->h_cdm: if a step throws while one
    // is queued, drain the stream before the slots (and the buffers above)
    // can be reused
    auto drain = [ctx] { (void)hipStreamSynchronize(ctx->stream); };
    DrainOnUnwind<decltype(drain)> unwind(drain);

    float theta = 0.0f;
    std::vector<float> cost;
    float best_cost = 3.402823466e+38f;
    float cur_smoothing = 0.8f;
    bool composed = false;  // Js holds compose_displacement of cur
    std::vector<float> mod_cost(size_t(run.nmod));
    TIPLHIP_REQUIRE(run.nmod >= 1 && run.nmod <= 16, "1 to 16 modalities");
    ctx->h_cdm.reserve(sizeof(float) * 16);
    for (int index = 0; index < run.param.max_iterations; ++index) {
        if (is_terminated(run)) {
            run.stopped = true;
            break;
        }
        ++run.iterations;
        // Each modality's cost is also written into coherent host memory,
        // whose slots start as a NaN pattern the reduction never writes; the
        // host spins on them (a stream synchronisation after kCostSpinUs).
        // The Jacobi sweeps do not depend on the host's decision (the
        // reference solves the same new_d whatever cdm_improved says), so
        // they are queued before the host waits and run during the round trip.
        uint32_t* slots = ctx->h_cdm.as<uint32_t>();
        std::fill(slots, slots + run.nmod, kCostPending);
        float* h_cost = static_cast<float*>(ctx->h_cdm.dev);
        CostReduce reduce;
        for (int i = 0; i < run.nmod; ++i) {
            // (of a single modality the field update has composed Js)
            if (!composed) launch_compose(ctx->stream, Is[size_t(i)], cur, g, Js.as<uint8_t>());
            const char type = run.param.gradient_type[std::min(i, 7)] == 'd' ? 'd' : 'r';
            reduce = launch_gradient(ctx->stream, Js.as<uint8_t>(), It[size_t(i)], g, type, i > 0 ? 1 : 0,
                                     nd.as<float>(), lay, partials.as<double>(), d_cost + i, h_cost + i);
            // the last modality's sum rides on the first Poisson launch
            if (i + 1 < run.nmod) launch_cost_reduce(ctx->stream, reduce);
        }
        composed = false;
        const bool need_theta = theta == 0.0f;
        float* solved = launch_poisson(ctx->stream, nd.as<float>(), pa, pb, g, lay, 12,
                                       need_theta ? d_maxlen : nullptr, maxparts.as<float>(), reduce);
        wait_for_slots(static_cast<const volatile uint32_t*>(slots), size_t(run.nmod), kCostPending,
                       std::chrono::microseconds(kCostSpinUs),
                       [ctx] { TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream)); });
        for (int i = 0; i < run.nmod; ++i) std::memcpy(&mod_cost[size_t(i)], &slots[i], sizeof(float));
        float sum_cost = 0.0f;
        for (int i = 0; i < run.nmod; ++i) {
            sum_cost += mod_cost[size_t(i)];
            if (sum_cost == 0.0f && !run.no_early_exit) return false;
        }
        cost.push_back(sum_cost / float(run.nmod));
        if (cost.back() < best_cost) {
            best_cost = cost.back();
            if (best != cur) {
                spare_field = best;
                best = cur;
            }
        }
        if (!cdm_improved(cost) && !run.no_early_exit) {
            if (cur_smoothing <= run.param.smoothing) break;
            if (best != cur) {
                spare_field = cur;
                cur = best;
            }
            cur_smoothing *= 0.5f;
            cost.clear();
        }
        if (need_theta) {
            unsigned int bits = 0;
            read_back(ctx, d_maxlen, &bits, sizeof(bits));
            std::memcpy(&theta, &bits, sizeof(theta));
        }
        if (theta == 0.0f) break;
        const float k = run.param.speed / theta;
        // cdm_smooth with weight 0 leaves the running field as it was (the
        // accumulated field is then unused), as in the reference
        if (cur_smoothing != 0.0f) {
            float* spare = solved == pa ? pb : pa;
            composed = launch_accumulate_smooth(ctx->stream, cur, solved, lay, k, cur_smoothing, g, spare, Is[0],
                                                run.nmod == 1 ? Js.as<uint8_t>() : nullptr);
            pa = cur == best ? spare_field : cur;
            pb = solved;
            cur = spare;
        }
    }
    // timing mode reports the running field after the fixed iteration count
    const float* result = run.no_early_exit ? cur : best;
    if (result != best_d) copy_d2d(ctx, best_d, result, fb);
    TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    return true;
}

// The fixed schedule (an extension; see tiplhip_cdm_param): `levels`
// pyramid levels, all run, coarsest first, each for exactly
// param.level_iterations iterations of the loop body with no cost-driven
// control; the running field is kept and, with field_bandwidth > 0, smoothed
// by filter::gaussian each iteration in place of cdm_smooth.  `field` is a
// device field of vox(dim), overwritten.
void cdm_fixed(CdmRun& run, const std::vector<const uint8_t*>& It,
               const std::vector<const uint8_t*>& Is, const int* dim, float* field, int levels)
{
    tiplhip_ctx* ctx = run.ctx;
    const FieldGeo g = field_geo(dim);
    const size_t n = g.n, fb = sizeof(float) * 3 * n;
    if (levels > 1) {
        const int rd[3] = {(dim[0] + 1) / 2, (dim[1] + 1) / 2, (dim[2] + 1) / 2};
        const size_t rn = vox(rd);
        DevMem rbuf(ctx, 2 * size_t(run.nmod) * rn), rfield(ctx, sizeof(float) * 3 * rn);
        std::vector<const uint8_t*> rIt, rIs;
        for (int i = 0; i < run.nmod; ++i) {
            uint8_t* t = rbuf.as<uint8_t>() + size_t(2 * i) * rn;
            uint8_t* s = rbuf.as<uint8_t>() + size_t(2 * i + 1) * rn;
            launch_downsample_u8(ctx, It[size_t(i)], dim, t);
            launch_downsample_u8(ctx, Is[size_t(i)], dim, s);
            rIt.push_back(t);
            rIs.push_back(s);
        }
        cdm_fixed(run, rIt, rIs, rd, rfield.as<float>(), levels - 1);
        zero(ctx, field, fb);  // far-edge slabs of the upsampled field stay 0
        launch_upsample(ctx->stream, rfield.as<float>(), field_geo(rd), g, field);
    } else {
        zero(ctx, field, fb);
    }
    if (run.stopped) return;
    DevMem nd(ctx, fb), pa(ctx, fb), pb(ctx, fb), Js(ctx, n);
    const uint32_t nblocks = block_count(g);
    DevMem partials(ctx, sizeof(double) * nblocks), maxparts(ctx, sizeof(float) * nblocks);
    DevMem scal(ctx, sizeof(float) * 16 + sizeof(unsigned int));
    const Lay lay = grad_layout(g);
    float* d_cost = scal.as<float>();
    unsigned int* d_maxlen = reinterpret_cast<unsigned int*>(scal.as<float>() + 16);
    float theta = 0.0f;
    for (int index = 0; index < run.param.level_iterations; ++index) {
        if (is_terminated(run)) {
            run.stopped = true;
            return;
        }
        ++run.iterations;
        for (int i = 0; i < run.nmod; ++i) {
            launch_compose(ctx->stream, Is[size_t(i)], field, g, Js.as<uint8_t>());
            const char type = run.param.gradient_type[std::min(i, 7)] == 'd' ? 'd' : 'r';
            // (the fixed schedule does not look at the cost)
            launch_gradient(ctx->stream, Js.as<uint8_t>(), It[size_t(i)], g, type, i > 0 ? 1 : 0,
                            nd.as<float>(), lay, partials.as<double>(), d_cost + i);
        }
        const bool need_theta = theta == 0.0f;
        float* solved = launch_poisson(ctx->stream, nd.as<float>(), pa.as<float>(), pb.as<float>(), g, lay, 12,
                                       need_theta ? d_maxlen : nullptr, maxparts.as<float>());
        if (need_theta) {
            unsigned int bits = 0;
            read_back(ctx, d_maxlen, &bits, sizeof(bits));
            std::memcpy(&theta, &bits, sizeof(theta));
        }
        if (theta == 0.0f) break;
        float* spare = solved == pa.as<float>() ? pb.as<float>() : pa.as<float>();
        // (the gaussian reads a planar field where it marches four rounds a launch)
        const bool planar = gaussian_takes_planar(dim, unsigned(run.param.field_bandwidth));
        launch_accumulate(ctx->stream, field, solved, lay, run.param.speed / theta, g, spare,
                          planar ? Lay{1u, g.n} : packed_layout());
        if (run.param.field_bandwidth > 0) {
            launch_gaussian_to(ctx, spare, field, solved, dim, 3, unsigned(run.param.field_bandwidth), planar);
        } else if (run.param.smoothing != 0.0f) {
            // cdm_smooth with weight 0 leaves the field untouched, as in the reference
            launch_smooth(ctx->stream, spare, field, run.param.smoothing, g);
        }
    }
    TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
}

std::vector<const uint8_t*> volume_ptrs(tiplhip_ctx* ctx, const tiplhip_volume* const* v, int n,
                                        const int* dim)
{
    std::vector<const uint8_t*> out;
    for (int i = 0; i < n; ++i) {
        TIPLHIP_REQUIRE(v[i] != nullptr, "null volume");
        TIPLHIP_REQUIRE(v[i]->ctx && v[i]->ctx->device == ctx->device, "volume lives on another device");
        TIPLHIP_REQUIRE(std::equal(dim, dim + 3, v[i]->dim), "all CDM volumes must share one shape");
        out.push_back(v[i]->d);
    }
    return out;
}

}  // namespace

int cdm_device(tiplhip_ctx* ctx, const tiplhip_volume* const* It, const tiplhip_volume* const* Is,
               int n, const tiplhip_cdm_param* param, float* d_field,
               const volatile uint8_t* terminated, int* iterations)
{
    TIPLHIP_REQUIRE(n >= 1 && n <= 8, "between 1 and 8 modality pairs");
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    DeviceGuard dg(ctx->device);
    const int* dim = It[0] ? It[0]->dim : nullptr;
    TIPLHIP_REQUIRE(dim != nullptr, "null volume");
    auto vt = volume_ptrs(ctx, It, n, dim);
    auto vs = volume_ptrs(ctx, Is, n, dim);
    CdmRun run{ctx, {}, n, terminated};
    if (param)
        run.param = *param;
    else
        tiplhip_cdm_param_default(&run.param);
    TIPLHIP_REQUIRE(run.param.max_iterations >= 0, "negative iteration cap");
    TIPLHIP_REQUIRE(run.param.levels >= 0 && run.param.levels <= 16, "levels must be in [0, 16]");
    TIPLHIP_REQUIRE(run.param.field_bandwidth >= 0 &&
                        run.param.field_bandwidth <= int(kMaxGaussianBandwidth),
                    "field_bandwidth must be in [0, 16]");
    zero(ctx, d_field, sizeof(float) * 3 * vox(dim));
    bool ok = true;
    if (run.param.levels > 0) {
        TIPLHIP_REQUIRE(run.param.level_iterations >= 0, "negative iteration count");
        cdm_fixed(run, vt, vs, dim, d_field, run.param.levels);
    } else {
        ok = cdm_level(run, vt, vs, dim, d_field, run.param.resolution);
    }
    if (iterations) *iterations = run.iterations;
    if (!ok) return TIPLHIP_ERR_FAILED;
    return run.stopped ? TIPLHIP_ERR_TERMINATED : TIPLHIP_OK;
}

}  // namespace tiplhip

using namespace tiplhip;

extern "C" {

void tiplhip_cdm_param_default(tiplhip_cdm_param* p)
{
    if (!p) return;
    p->resolution = 2.0f;
    p->speed = 0.3f;
    p->smoothing = 0.05f;
    p->min_dimension = 16;
    p->max_iterations = 200;
    for (char& c : p->gradient_type) c = 'r';
    p->levels = 0;
    p->level_iterations = 0;
    p->field_bandwidth = 0;
}

int tiplhip_cdm(tiplhip_ctx* ctx, const tiplhip_volume* const* It, const tiplhip_volume* const* Is,
                int n, const tiplhip_cdm_param* param, float* field, const volatile uint8_t* terminated,
                int* iterations)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && It && Is && field, "null argument");
        TIPLHIP_REQUIRE(n >= 1 && It[0], "null volume");
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const size_t fb = sizeof(float) * 3 * vox(It[0]->dim);
        DevMem best(ctx, fb);
        const int rc = cdm_device(ctx, It, Is, n, param, best.as<float>(), terminated, iterations);
        if (rc == TIPLHIP_ERR_FAILED) throw Error(TIPLHIP_ERR_FAILED, "cdm returned false (zero cost)");
        copy_to_host(ctx, field, best.p, fb);
        // As in the reference, a terminated run still returns its best field.
        if (rc == TIPLHIP_ERR_TERMINATED) throw Error(TIPLHIP_ERR_TERMINATED, "terminated by the caller");
    });
}

int tiplhip_cdm_level_iterations(tiplhip_ctx* ctx, const tiplhip_volume* It,
                                 const tiplhip_volume* Is, const tiplhip_cdm_param* param,
                                 int iterations, float* field)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && It && Is, "null argument");
        TIPLHIP_REQUIRE(iterations >= 0, "negative iteration count");
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const int* dim = It->dim;
        auto vt = volume_ptrs(ctx, &It, 1, dim);
        auto vs = volume_ptrs(ctx, &Is, 1, dim);
        CdmRun run{ctx, {}, 1, nullptr};
        if (param)
            run.param = *param;
        else
            tiplhip_cdm_param_default(&run.param);
        run.param.max_iterations = iterations;
        run.no_early_exit = true;
        const size_t fb = sizeof(float) * 3 * vox(dim);
        DevMem best(ctx, fb);
        zero(ctx, best.p, fb);
        (void)cdm_level(run, vt, vs, dim, best.as<float>(), 1.0f);
        if (field) copy_to_host(ctx, field, best.p, fb);
    });
}

// ---- single steps on host buffers ----------------------------------------

int tiplhip_compose_displacement(tiplhip_ctx* ctx, const uint8_t* Is, const int dim[3],
                                 const float* d, uint8_t* Js)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && Is && d && Js, "null argument");
        check_dim(dim);
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo g = field_geo(dim);
        DevMem dI(ctx, g.n), dD(ctx, sizeof(float) * 3 * g.n), dJ(ctx, g.n);
        TIPLHIP_CHECK(hipMemcpyAsync(dI.p, Is, g.n, hipMemcpyHostToDevice, ctx->stream));
        TIPLHIP_CHECK(hipMemcpyAsync(dD.p, d, sizeof(float) * 3 * g.n, hipMemcpyHostToDevice, ctx->stream));
        launch_compose(ctx->stream, dI.as<uint8_t>(), dD.as<float>(), g, dJ.as<uint8_t>());
        TIPLHIP_CHECK(hipMemcpyAsync(Js, dJ.p, g.n, hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    });
}

int tiplhip_cdm_gradient(tiplhip_ctx* ctx, const uint8_t* Js, const uint8_t* It, const int dim[3],
                         char type, float* new_d, float* cost)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && Js && It && new_d, "null argument");
        TIPLHIP_REQUIRE(type == 'r' || type == 'd', "gradient type must be 'r' or 'd'");
        check_dim(dim);
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo g = field_geo(dim);
        DevMem dJ(ctx, g.n), dI(ctx, g.n), dN(ctx, sizeof(float) * 3 * g.n);
        DevMem part(ctx, sizeof(double) * block_count(g)), dc(ctx, sizeof(float));
        TIPLHIP_CHECK(hipMemcpyAsync(dJ.p, Js, g.n, hipMemcpyHostToDevice, ctx->stream));
        TIPLHIP_CHECK(hipMemcpyAsync(dI.p, It, g.n, hipMemcpyHostToDevice, ctx->stream));
        launch_cost_reduce(ctx->stream, launch_gradient(ctx->stream, dJ.as<uint8_t>(), dI.as<uint8_t>(), g, type, 0,
                                                dN.as<float>(), packed_layout(), part.as<double>(),
                                                dc.as<float>()));
        TIPLHIP_CHECK(hipMemcpyAsync(new_d, dN.p, sizeof(float) * 3 * g.n, hipMemcpyDeviceToHost, ctx->stream));
        float c = 0.0f;
        TIPLHIP_CHECK(hipMemcpyAsync(&c, dc.p, sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
        if (cost) *cost = c;
    });
}

int tiplhip_cdm_poisson(tiplhip_ctx* ctx, float* new_d, const int dim[3], int sweeps,
                        float* max_length)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && new_d, "null argument");
        TIPLHIP_REQUIRE(sweeps >= 1 && sweeps <= 1000, "sweeps must be in [1, 1000]");
        check_dim(dim);
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo g = field_geo(dim);
        const size_t fb = sizeof(float) * 3 * g.n;
        DevMem dN(ctx, fb), a(ctx, fb), b(ctx, fb), ml(ctx, sizeof(unsigned int)), mp(ctx, sizeof(float) * block_count(g));
        TIPLHIP_CHECK(hipMemcpyAsync(dN.p, new_d, fb, hipMemcpyHostToDevice, ctx->stream));
        float* out = launch_poisson(ctx->stream, dN.as<float>(), a.as<float>(), b.as<float>(), g, packed_layout(), sweeps,
                                    ml.as<unsigned int>(), mp.as<float>());
        TIPLHIP_CHECK(hipMemcpyAsync(new_d, out, fb, hipMemcpyDeviceToHost, ctx->stream));
        unsigned int bits = 0;
        TIPLHIP_CHECK(hipMemcpyAsync(&bits, ml.p, sizeof(bits), hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
        if (max_length) std::memcpy(max_length, &bits, sizeof(float));
    });
}

int tiplhip_accumulate_displacement(tiplhip_ctx* ctx, const float* cur, float* new_d,
                                    const int dim[3], float scale)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && cur && new_d, "null argument");
        check_dim(dim);
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo g = field_geo(dim);
        const size_t fb = sizeof(float) * 3 * g.n;
        DevMem dC(ctx, fb), dN(ctx, fb);
        TIPLHIP_CHECK(hipMemcpyAsync(dC.p, cur, fb, hipMemcpyHostToDevice, ctx->stream));
        TIPLHIP_CHECK(hipMemcpyAsync(dN.p, new_d, fb, hipMemcpyHostToDevice, ctx->stream));
        launch_accumulate(ctx->stream, dC.as<float>(), dN.as<float>(), packed_layout(), scale, g, dN.as<float>(),
                          packed_layout());
        TIPLHIP_CHECK(hipMemcpyAsync(new_d, dN.p, fb, hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    });
}

int tiplhip_cdm_smooth(tiplhip_ctx* ctx, const float* d, float* dd, const int dim[3], float smoothing)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && d && dd, "null argument");
        check_dim(dim);
        if (smoothing == 0.0f) return;  // cdm_smooth leaves dd untouched
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo g = field_geo(dim);
        const size_t fb = sizeof(float) * 3 * g.n;
        DevMem dD(ctx, fb), dO(ctx, fb);
        TIPLHIP_CHECK(hipMemcpyAsync(dD.p, d, fb, hipMemcpyHostToDevice, ctx->stream));
        launch_smooth(ctx->stream, dD.as<float>(), dO.as<float>(), smoothing, g);
        TIPLHIP_CHECK(hipMemcpyAsync(dd, dO.p, fb, hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    });
}

int tiplhip_upsample_field(tiplhip_ctx* ctx, const float* in, const int in_dim[3], float* out,
                           const int out_dim[3])
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && in && out, "null argument");
        check_dim(in_dim);
        check_dim(out_dim);
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const FieldGeo gi = field_geo(in_dim), go = field_geo(out_dim);
        DevMem dI(ctx, sizeof(float) * 3 * gi.n), dO(ctx, sizeof(float) * 3 * go.n);
        TIPLHIP_CHECK(hipMemcpyAsync(dI.p, in, sizeof(float) * 3 * gi.n, hipMemcpyHostToDevice, ctx->stream));
        launch_upsample(ctx->stream, dI.as<float>(), gi, go, dO.as<float>());
        TIPLHIP_CHECK(hipMemcpyAsync(out, dO.p, sizeof(float) * 3 * go.n, hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    });
}

}  // extern "C"
