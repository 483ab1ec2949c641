// filter.hip -- the binomial Gaussian filter of filter/gaussian.hpp:18-105 on gfx950.
//
// gaussian(I, bandwidth) applies `bandwidth` rounds of the separable [1 2 1]
// stencil, x then y then z, with replicate edges, and scales the result by
// 2^(-2*bandwidth*3) (bandwidth b has variance b/2 per axis).  Each pass of
// the reference writes a float array, so every intermediate value is rounded
// to float; one launch here runs one whole round (three passes), or four
// (gaussian_march_kernel), and keeps those roundings.  In the single round the
// x pass of a tile (with a one-voxel halo) is written to LDS, the y pass of it
// stays in registers, and the z pass combines three consecutive y-pass planes
// while the block marches along z.  HBM traffic per launch is one read (plus
// halo) and one write of the image instead of the reference's three of each a
// round.
//
// Works on float images of CH interleaved channels: CH = 1 for a scalar
// volume, CH = 3 for a vector<3,float> displacement field.
#include "device.hpp"
#include "internal.hpp"
#include "march_plan.hpp"

#include <algorithm>
#include <cmath>

namespace tiplhip {
namespace {

constexpr int kGX = 64;        // output columns per block (one wave)
constexpr int kGY = 8;         // output rows per block (2 per thread row)
constexpr int kGRows = kGY / 4;
constexpr int kGThreads = 256;

struct GaussGeo {
    int w, h, d;
    uint32_t wh;
};

// One round over a 64 x 8 column of `zq` output planes.  Each thread owns
// fixed slots of the haloed plane tile A (AR x AC floats): their in-plane
// source offsets (with the replicate clamp) are computed once, and the next
// plane's values are loaded into registers while the current plane is
// filtered, so the global-load latency overlaps the LDS passes.
template <int CH>
__global__ __launch_bounds__(kGThreads) void gaussian_round_kernel(const float* __restrict__ a,
                                                                   float* __restrict__ b, GaussGeo g,
                                                                   float scale, int zq)
{
    constexpr int AR = kGY + 2, AC = (kGX + 2) * CH, XC = kGX * CH;
    constexpr int NA = AR * AC;
    constexpr int NL = (NA + kGThreads - 1) / kGThreads;
    __shared__ float A[NA];
    __shared__ float X[AR][XC];
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * kGX + tx;
    // each XCD takes a contiguous range of blocks (x fastest), so the halo
    // rows and planes adjacent blocks share are read through one L2
    const uint32_t gx = gridDim.x, gy = gridDim.y;
    const uint32_t L = xcd_remap((blockIdx.z * gy + blockIdx.y) * gx + blockIdx.x, gx * gy * gridDim.z);
    const int x0 = int(L % gx) * kGX, y0 = int((L / gx) % gy) * kGY, z0 = int(L / (gx * gy)) * zq;
    const int zend = min(z0 + zq, g.d);
    const uint32_t plane = g.wh * uint32_t(CH);

    // slot k holds A[tid + 256 k]: row r = e / AC, column (x0-1+col) and
    // channel comp; a clamped neighbour is the centre itself (the
    // reference's replicate edge)
    uint32_t off[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        const int e = min(tid + kGThreads * k, NA - 1);
        const int r = e / AC, cc = e - r * AC;
        const int col = cc / CH, comp = cc - col * CH;
        const int gy = min(max(y0 - 1 + r, 0), g.h - 1);
        const int gx = min(max(x0 - 1 + col, 0), g.w - 1);
        off[k] = (uint32_t(gy) * uint32_t(g.w) + uint32_t(gx)) * uint32_t(CH) + uint32_t(comp);
    }
    float v[NL];
    {
        const uint32_t pz = uint32_t(min(max(z0 - 1, 0), g.d - 1));
#pragma unroll
        for (int k = 0; k < NL; ++k) v[k] = a[size_t(pz) * plane + off[k]];
    }

    float Yp[kGRows][CH], Yc[kGRows][CH];
#pragma unroll
    for (int j = 0; j < kGRows; ++j)
#pragma unroll
        for (int c = 0; c < CH; ++c) Yp[j][c] = Yc[j][c] = 0.0f;

    for (int zz = z0 - 1; zz <= zend; ++zz) {
#pragma unroll
        for (int k = 0; k < NL; ++k)
            if (tid + kGThreads * k < NA) A[tid + kGThreads * k] = v[k];
        if (zz < zend) {
            const uint32_t pz = uint32_t(min(zz + 1, g.d - 1));
#pragma unroll
            for (int k = 0; k < NL; ++k) v[k] = a[size_t(pz) * plane + off[k]];
        }
        __syncthreads();
        // x pass: (left + (c + c)) + right
        for (int e = tid; e < AR * kGX; e += kGThreads) {
            const int r = e / kGX, col = e - r * kGX;
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                float center = A[r * AC + (col + 1) * CH + c];
                center += center;
                X[r][col * CH + c] = (A[r * AC + col * CH + c] + center) + A[r * AC + (col + 2) * CH + c];
            }
        }
        __syncthreads();
        // y pass of this thread's rows of plane zz
        float Yn[kGRows][CH];
#pragma unroll
        for (int j = 0; j < kGRows; ++j) {
            const int r = ty + 4 * j;
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                float center = X[r + 1][tx * CH + c];
                center += center;
                Yn[j][c] = (X[r][tx * CH + c] + center) + X[r + 2][tx * CH + c];
            }
        }
        // z pass of plane zz-1 from the y passes of planes zz-2, zz-1, zz
        if (zz > z0) {
            const int x = x0 + tx;
            const uint32_t oz = uint32_t(zz - 1);
#pragma unroll
            for (int j = 0; j < kGRows; ++j) {
                const int y = y0 + ty + 4 * j;
                if (x < g.w && y < g.h) {
                    const size_t o = size_t(oz * g.wh + uint32_t(y) * uint32_t(g.w) + uint32_t(x)) * CH;
#pragma unroll
                    for (int c = 0; c < CH; ++c) {
                        float center = Yc[j][c];
                        center += center;
                        b[o + c] = ((Yp[j][c] + center) + Yn[j][c]) * scale;
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kGRows; ++j)
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                Yp[j][c] = Yc[j][c];
                Yc[j][c] = Yn[j][c];
            }
    }
}

// ---------------------------------------------------------------------------
// Four rounds per launch, marching z.  The channels are independent, so a
// workgroup takes one channel of a 64 x 32 column: lane l of wave v holds rows
// 4 v .. 4 v + 3 of column l in registers, and every intermediate value is the
// same float.  When plane m of the input arrives, round t takes plane
// m - 2 (t - 1) from round t - 1 (both neighbouring columns are lane shifts),
// finishes the y pass of the plane before it (a wave's first and last row
// meet the neighbouring waves' through LDS, written a step earlier) and hands
// on plane m - 2 t: one barrier a step for all rounds.  A round spoils one
// layer at an inner border of the column, so four columns and rows on each
// side are halo; columns and rows at the image's own border are placed at the
// column's, where the replicate edge is the value itself.
// Issue and the chain of rounds within a step bound it, as they do
// poisson_march_kernel.  Eight rounds of a field, planar in: 213 -> 119 us at
// 160x192x160, 73 -> 46 at 80x96x80, 60 -> 25 at 40x48x40.  (Plain shifts in
// columns without a border, and the z selects only in planes that need them,
// measured the same.)
// ---------------------------------------------------------------------------
constexpr int kMK = 4, kMWaves = 8, kMR = 4, kMRows = kMWaves * kMR;
constexpr uint32_t kMBlocks = 512;  // workgroups resident at a time: two a CU

struct GaussMarch {
    uint32_t gx, gy, gz;  // tiles
    int zc;               // planes per workgroup
    uint32_t blocks;
};

GaussMarch gauss_march(const GaussGeo& g, int channels)
{
    auto tiles = [](int n, int side) {
        return n <= side ? 1u : uint32_t((n - 2 * kMK + side - 2 * kMK - 1) / (side - 2 * kMK));
    };
    GaussMarch m;
    m.gx = tiles(g.w, 64);
    m.gy = tiles(g.h, kMRows);
    const uint32_t cols = uint32_t(channels) * m.gx * m.gy;
    const MarchPlan p = march_plan(cols, g.d, 3 * kMK + 2, 1, kMBlocks);
    m.gz = p.runs;
    m.zc = p.planes;
    m.blocks = cols * m.gz;
    return m;
}

// A field's layout: channel c of voxel p is element p * ps + c * cs.
struct GaussLay {
    uint32_t ps, cs;
};

__global__ __launch_bounds__(64 * kMWaves, 4) void gaussian_march_kernel(const float* __restrict__ a,
                                                                         GaussLay la,
                                                                         float* __restrict__ b,
                                                                         GaussLay lb, GaussGeo g,
                                                                         GaussMarch mg, uint32_t channels,
                                                                         float scale)
{
    __shared__ float edge[2][kMK][kMWaves][2][64];  // x passes: a wave's first and last row
    const int lane = int(threadIdx.x) & 63;
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const uint32_t L = xcd_remap(blockIdx.x, mg.blocks);
    const uint32_t chan = L % channels, tile = L / channels;
    const int w = g.w, h = g.h, wh = int(g.wh);
    const int x0 = min(int(tile % mg.gx) * (64 - 2 * kMK), max(w - 64, 0));
    const int y0 = min(int((tile / mg.gx) % mg.gy) * (kMRows - 2 * kMK), max(h - kMRows, 0));
    const int z0 = int(tile / (mg.gx * mg.gy)) * mg.zc, z1 = min(z0 + mg.zc, g.d);
    const uint32_t n = g.wh * uint32_t(g.d);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a + size_t(chan) * la.cs, ((n - 1u) * la.ps + 1u) * 4u);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(b + size_t(chan) * lb.cs, ((n - 1u) * lb.ps + 1u) * 4u);
    const int q0 = (y0 + wv * kMR) * w + x0 + lane;  // row 0 of this thread in plane 0
    // the image's last column and row, where they lie inside this column
    const bool narrow = w < 64, last_x = x0 + lane == w - 1;
    const int last_y = h - 1 - (y0 + wv * kMR);
    const bool top = y0 + wv * kMR == 0, bottom = last_y >= 0 && last_y < kMR;
    const bool out_x = (lane >= kMK || x0 == 0) && (lane < 64 - kMK || x0 + 64 >= w) && x0 + lane < w;
    const int row_a = w * int(la.ps) * 4, slab_a = wh * int(la.ps) * 4;
    const int row_b = w * int(lb.ps) * 4, slab_b = wh * int(lb.ps) * 4;
    const int first = z0 - kMK, last = z1 - 1 + 2 * kMK;
    int at = (q0 + (first + 2) * wh) * int(la.ps) * 4;  // this thread's row 0 in plane m + 2
    int to = (q0 + (first - 2 * kMK) * wh) * int(lb.ps) * 4;
    float in[3][kMR], X[kMK][kMR], Y[kMK][3][kMR];
    auto load = [&](int off, float (&dst)[kMR]) {
#pragma unroll
        for (int j = 0; j < kMR; ++j)
            dst[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ra, off + j * row_a, 0, 0));
    };
#pragma unroll
    for (int t = 0; t < kMK; ++t)
#pragma unroll
        for (int j = 0; j < kMR; ++j) X[t][j] = Y[t][0][j] = Y[t][1][j] = Y[t][2][j] = 0.0f;
    load(at - 2 * slab_a, in[0]);
    load(at - slab_a, in[1]);
    for (int base = first; base <= last; base += 6) {
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            const int m = base + u;
            if (m > last) break;
            load(at, in[(u + 2) % 3]);
            __syncthreads();
            const int par = u & 1;
            float v[kMR];  // the plane handed from round to round
#pragma unroll
            for (int j = 0; j < kMR; ++j) v[j] = in[u % 3][j];
#pragma unroll
            for (int t = 1; t <= kMK; ++t) {
                const int p = m - 2 * (t - 1);  // the plane round t takes in this step
                if (p < z0 - (kMK - t) - 1) break;
                // y pass of plane p - 1 from its x pass
                float(&x)[kMR] = X[t - 1];
                float(&yp)[kMR] = Y[t - 1][(u + 1) % 3];  // plane p - 3
                float(&yc)[kMR] = Y[t - 1][(u + 2) % 3];  // plane p - 2
                float(&yn)[kMR] = Y[t - 1][u % 3];        // plane p - 1
                float up = edge[par ^ 1][t - 1][wv > 0 ? wv - 1 : 0][1][lane];
                const float dn = edge[par ^ 1][t - 1][wv < kMWaves - 1 ? wv + 1 : wv][0][lane];
                if (top) up = x[0];
#pragma unroll
                for (int j = 0; j < kMR; ++j) {
                    const float c = x[j] + x[j];
                    yn[j] = ((j > 0 ? x[j - 1] : up) + c) + (j < kMR - 1 ? x[j + 1] : dn);
                }
                if (bottom) {
#pragma unroll
                    for (int j = 0; j < kMR; ++j)
                        if (j == last_y) yn[j] = ((j > 0 ? x[j - 1] : up) + (x[j] + x[j])) + x[j];
                }
                // x pass of plane p
#pragma unroll
                for (int j = 0; j < kMR; ++j) {
                    const float c = v[j];
                    float right = wave_next_or(c);
                    if (narrow) right = last_x ? c : right;
                    x[j] = (wave_prev_or(c) + (c + c)) + right;
                }
                edge[par][t - 1][wv][0][lane] = x[0];
                edge[par][t - 1][wv][1][lane] = x[kMR - 1];
                // z pass: plane p - 2
                const bool lowest = p - 2 == 0, highest = p - 2 == g.d - 1;
#pragma unroll
                for (int j = 0; j < kMR; ++j) {
                    const float c = yc[j] + yc[j];
                    v[j] = ((lowest ? yc[j] : yp[j]) + c) + (highest ? yc[j] : yn[j]);
                }
                if (t == kMK && p - 2 >= z0) {
#pragma unroll
                    for (int j = 0; j < kMR; ++j) {
                        const int r = wv * kMR + j;
                        const bool out_y = (r >= kMK || y0 == 0) && (r < kMRows - kMK || y0 + kMRows >= h) &&
                                           y0 + r < h;
                        if (out_y && out_x)
                            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[j] * scale), rb,
                                                                  to + j * row_b, 0, 0);
                    }
                }
            }
            at += slab_a;
            to += slab_b;
            // (keeps the running offsets in two registers, as in poisson_march_kernel)
            asm volatile("" : "+v"(at), "+v"(to));
        }
    }
}

GaussGeo gauss_geo(const int* dim)
{
    return GaussGeo{dim[0], dim[1], dim[2], uint32_t(dim[0]) * uint32_t(dim[1])};
}

// Whether the marched kernel's byte offsets, rows and planes past the volume
// included, stay below 2^31.
bool march_fits(const GaussGeo& g)
{
    return (size_t(g.wh) * (size_t(g.d) + 16) + 64 * size_t(g.w)) * 12 < (size_t(1) << 31);
}

void launch_march(tiplhip_ctx* ctx, const float* in, GaussLay li, float* out, GaussLay lo,
                  const GaussGeo& g, int channels, float scale)
{
    const GaussMarch m = gauss_march(g, channels);
    hipLaunchKernelGGL(gaussian_march_kernel, dim3(m.blocks), dim3(64 * kMWaves), 0, ctx->stream, in, li,
                       out, lo, g, m, uint32_t(channels), scale);
    TIPLHIP_CHECK(hipGetLastError());
}

// Planes per block: about 1024 blocks over the volume (each block reads two
// halo planes beyond its zq), at least 4 and at most 16 planes.
int gauss_zq(const GaussGeo& g)
{
    const long tiles = long((g.w + kGX - 1) / kGX) * long((g.h + kGY - 1) / kGY);
    const long zq = long(g.d) * tiles / 1024;
    return int(std::min(16L, std::max(4L, zq)));
}

void launch_round(tiplhip_ctx* ctx, const float* in, float* out, const GaussGeo& g, int channels,
                  float scale)
{
    const int zq = gauss_zq(g);
    const dim3 grid(uint32_t((g.w + kGX - 1) / kGX), uint32_t((g.h + kGY - 1) / kGY),
                    uint32_t((g.d + zq - 1) / zq));
    const dim3 block(kGX, 4);
    if (channels == 1)
        hipLaunchKernelGGL(gaussian_round_kernel<1>, grid, block, 0, ctx->stream, in, out, g, scale, zq);
    else
        hipLaunchKernelGGL(gaussian_round_kernel<3>, grid, block, 0, ctx->stream, in, out, g, scale, zq);
    TIPLHIP_CHECK(hipGetLastError());
}

void check_gaussian(const int* dim, int channels, unsigned bandwidth)
{
    TIPLHIP_REQUIRE(channels == 1 || channels == 3, "gaussian: channels must be 1 or 3");
    TIPLHIP_REQUIRE(bandwidth <= kMaxGaussianBandwidth, "gaussian: bandwidth above 16");
    TIPLHIP_REQUIRE(vox(dim) * size_t(channels) < (size_t(1) << 32),
                    "gaussian: image exceeds 2^32 floats");
}

}  // namespace

bool gaussian_takes_planar(const int* dim, unsigned bandwidth)
{
    return bandwidth >= unsigned(kMK) && march_fits(gauss_geo(dim));
}

void launch_gaussian_to(tiplhip_ctx* ctx, const float* src, float* dst, float* tmp,
                        const int* dim, int channels, unsigned bandwidth, bool planar)
{
    check_gaussian(dim, channels, bandwidth);
    const size_t bytes = sizeof(float) * size_t(channels) * vox(dim);
    if (bytes == 0) return;
    if (bandwidth == 0) {
        TIPLHIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
        return;
    }
    const GaussGeo g = gauss_geo(dim);
    // the scale is a power of two with a normal float value for bandwidth <= 16,
    // so scaling in float equals the reference's float(double(v) * scale)
    const float last_scale = std::ldexp(1.0f, -int(6 * bandwidth));
    const GaussLay packed{uint32_t(channels), 1u}, split{1u, uint32_t(vox(dim))};
    TIPLHIP_REQUIRE(!planar || gaussian_takes_planar(dim, bandwidth), "planar gaussian input not supported");
    // four rounds a launch, then single ones.  The launches alternate between
    // tmp and dst so that the last lands in dst and src is only read; the
    // marched ones leave their result planar unless a packed reader follows.
    const unsigned marched = march_fits(g) ? bandwidth / unsigned(kMK) : 0u;
    const unsigned launches = marched + (bandwidth - marched * unsigned(kMK));
    const float* in = src;
    GaussLay li = planar ? split : packed;
    for (unsigned k = 0; k < launches; ++k) {
        float* out = ((launches - 1 - k) % 2 == 0) ? dst : tmp;
        const float scale = k + 1 == launches ? last_scale : 1.0f;
        if (k < marched) {
            const GaussLay lo = k + 1 < marched ? split : packed;
            launch_march(ctx, in, li, out, lo, g, channels, scale);
            li = lo;
        } else {
            launch_round(ctx, in, out, g, channels, scale);
        }
        in = out;
    }
}

float* launch_gaussian(tiplhip_ctx* ctx, float* a, float* tmp, const int* dim, int channels,
                       unsigned bandwidth)
{
    check_gaussian(dim, channels, bandwidth);
    if (bandwidth == 0 || vox(dim) == 0) return a;
    // one launch: out of place; more: tmp and a in turn, the last into a
    const unsigned marched = march_fits(gauss_geo(dim)) ? bandwidth / unsigned(kMK) : 0u;
    const unsigned launches = marched + (bandwidth - marched * unsigned(kMK));
    float* dst = launches % 2 == 0 ? a : tmp;
    launch_gaussian_to(ctx, a, dst, dst == a ? tmp : a, dim, channels, bandwidth, false);
    return dst;
}

}  // namespace tiplhip

using namespace tiplhip;

extern "C" {

int tiplhip_gaussian(tiplhip_ctx* ctx, float* data, const int dim[3], int channels,
                     unsigned bandwidth)
{
    return guarded([&] {
        TIPLHIP_REQUIRE(ctx && data && dim, "null argument");
        TIPLHIP_REQUIRE(dim[0] > 0 && dim[1] > 0 && dim[2] > 0, "dims must be positive");
        TIPLHIP_REQUIRE(channels == 1 || channels == 3, "gaussian: channels must be 1 or 3");
        TIPLHIP_REQUIRE(bandwidth <= kMaxGaussianBandwidth, "gaussian: bandwidth above 16");
        if (bandwidth == 0) return;  // the reference returns the image unchanged
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        DeviceGuard dg(ctx->device);
        const size_t bytes = sizeof(float) * size_t(channels) * vox(dim);
        DeviceBuffer a, t;
        a.reserve(bytes);
        t.reserve(bytes);
        TIPLHIP_CHECK(hipMemcpyAsync(a.p, data, bytes, hipMemcpyHostToDevice, ctx->stream));
        float* r = launch_gaussian(ctx, a.as<float>(), t.as<float>(), dim, channels, bandwidth);
        TIPLHIP_CHECK(hipMemcpyAsync(data, r, bytes, hipMemcpyDeviceToHost, ctx->stream));
        TIPLHIP_CHECK(hipStreamSynchronize(ctx->stream));
    });
}

}  // extern "C"
