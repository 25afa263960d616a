// Layout changes at a program's edges (planar NCHW <-> channels-last), and
// transfers between page-locked host tensors and the arena as kernels on the
// program's own stream.
//
// Between device tensors relayout_kernel is bound by HBM: 39 MB read and
// written in 15 us, 5.2 TB/s (23.5 us through 32 x 32 scalar tiles).  A
// 64 x 64 tile (pixels x channels) goes through LDS with a row pitch of 65
// floats: a wave's 16-byte planar accesses are four 256-byte runs, its
// channels-last ones four runs of 64 channels, and the LDS accesses of both
// phases fall on distinct banks.  The next tile's loads are issued before the
// current tile is stored, so a workgroup keeps 16 KB of loads in flight.
//
// On host memory the PCIe link bounds them.  Writes of 256-byte runs reach
// 52 GB/s, so a result goes to the host from the layout change itself.
// Reads of such runs do not (36 to 40 GB/s, 34 with odd image sizes, where
// the accesses are 4 bytes wide), contiguous 16-byte reads do: 1.7 MB in
// 35 us against 51, so an input comes in through copy_floats_kernel and the
// layout change after it (5 us) reads HBM.  32 to 128 workgroups saturate the
// link (56 GB/s); more read slower (2048: 39 GB/s at 6 MB), so these grids
// are capped and walk their tiles.  Against a DMA copy no step waits for a
// copy engine, 10 to 45 us from a copy's end to the next kernel's start.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <string>

#include "../kernels.hpp"

namespace pdefa {
namespace k {
namespace {

constexpr int kTile = 64;
constexpr int kPitch = kTile + 1;
constexpr int kLanes = 256;
constexpr int kPer = kTile * kTile / kLanes;  // floats of a tile per lane
constexpr int kRelayoutBlocks = 2048;         // grid cap between device tensors (8 workgroups a CU)

struct TileGeom {
    int32_t tiles_p, tiles_c;
    int64_t tiles;
};

struct TilePos {
    int32_t n, c0, p0;
};

__device__ __forceinline__ TilePos tile_pos(const TileGeom& g, int64_t t) {
    TilePos q;
    q.p0 = static_cast<int32_t>(t % g.tiles_p) * kTile;
    t /= g.tiles_p;
    q.c0 = static_cast<int32_t>(t % g.tiles_c) * kTile;
    q.n = static_cast<int32_t>(t / g.tiles_c);
    return q;
}

// One side of a tile in a lane's registers: `rows` strided lines of `cols`
// contiguous floats (V: 16-byte runs, 16 lanes a line; else one line a wave).
// f(k, row, col) visits the lane's k-th group of 4 (V) or 1 floats.
template <bool V, typename F>
__device__ __forceinline__ void visit(int rows, int cols, F&& f) {
    const int tid = threadIdx.x;
    if constexpr (V) {
#pragma unroll
        for (int k = 0; k < kPer / 4; ++k) {
            const int r = tid / 16 + 16 * k, c = 4 * (tid % 16);
            f(k, r, c, r < rows && c < cols);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int r = tid / 64 + 4 * k, c = tid % 64;
            f(k, r, c, r < rows && c < cols);
        }
    }
}

template <bool V>
__device__ __forceinline__ void load_side(float (&v)[kPer], const float* p, int64_t stride, int rows, int cols) {
    visit<V>(rows, cols, [&](int k, int r, int c, bool ok) {
        if constexpr (V) {
            float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (ok) x = *reinterpret_cast<const float4*>(p + r * stride + c);
            v[4 * k] = x.x;
            v[4 * k + 1] = x.y;
            v[4 * k + 2] = x.z;
            v[4 * k + 3] = x.w;
        } else {
            v[k] = ok ? p[r * stride + c] : 0.0f;
        }
    });
}

template <bool V>
__device__ __forceinline__ void store_side(const float (&v)[kPer], float* p, int64_t stride, int rows, int cols) {
    visit<V>(rows, cols, [&](int k, int r, int c, bool ok) {
        if (!ok) return;
        if constexpr (V)
            *reinterpret_cast<float4*>(p + r * stride + c) =
                make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
        else
            p[r * stride + c] = v[k];
    });
}

// lds[row][col] <- v, and v <- lds transposed
template <bool V>
__device__ __forceinline__ void to_lds(const float (&v)[kPer], float* lds) {
    visit<V>(kTile, kTile, [&](int k, int r, int c, bool) {
#pragma unroll
        for (int j = 0; j < (V ? 4 : 1); ++j) lds[r * kPitch + c + j] = v[(V ? 4 * k : k) + j];
    });
}
template <bool V>
__device__ __forceinline__ void from_lds_t(float (&v)[kPer], const float* lds) {
    visit<V>(kTile, kTile, [&](int k, int r, int c, bool) {
#pragma unroll
        for (int j = 0; j < (V ? 4 : 1); ++j) v[(V ? 4 * k : k) + j] = lds[(c + j) * kPitch + r];
    });
}

// IN: planar source -> channels-last destination; else the other way.  VS,
// VD: 16-byte accesses on the source and destination side.  The mirror is a
// second copy of a planar destination, with its strides (nullptr: none).
template <bool IN, bool VS, bool VD>
__global__ __launch_bounds__(kLanes) void relayout_kernel(RelayoutArgs a, TileGeom g) {
    __shared__ float lds[kTile * kPitch];
    float v[kPer], w[kPer];
    auto load = [&](int64_t t) {
        const TilePos q = tile_pos(g, t);
        const int np = min(kTile, a.P - q.p0), nc = min(kTile, a.C - q.c0);
        if constexpr (IN)
            load_side<VS>(v, a.src + q.n * a.planar_n + q.c0 * a.planar_c + q.p0, a.planar_c, nc, np);
        else
            load_side<VS>(v, a.src + q.n * a.rows_n + q.p0 * a.rows_p + q.c0, a.rows_p, np, nc);
    };
    int64_t t = blockIdx.x;
    load(t);  // the grid has at most g.tiles workgroups
    while (t < g.tiles) {
        const TilePos q = tile_pos(g, t);
        const int np = min(kTile, a.P - q.p0), nc = min(kTile, a.C - q.c0);
        to_lds<VS>(v, lds);
        __syncthreads();
        t += gridDim.x;
        if (t < g.tiles) load(t);
        from_lds_t<VD>(w, lds);
        if constexpr (IN) {
            store_side<VD>(w, a.dst + q.n * a.rows_n + q.p0 * a.rows_p + q.c0, a.rows_p, np, nc);
        } else {
            const int64_t planar = q.n * a.planar_n + q.c0 * a.planar_c + q.p0;
            store_side<VD>(w, a.dst + planar, a.planar_c, nc, np);
            if (a.mirror) store_side<VD>(w, a.mirror + planar, a.planar_c, nc, np);
        }
        __syncthreads();
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <bool IN>
void launch_relayout(const RelayoutArgs& a, hipStream_t s) {
    if (!a.src || !a.dst) throw std::runtime_error("relayout: null pointer");
    if (IN && a.mirror) throw std::runtime_error("relayout: a mirror of a channels-last destination");
    if (a.N < 0 || a.C < 1 || a.P < 1 || a.planar_c < 0 || a.rows_p < 0 || a.planar_n < 0 || a.rows_n < 0)
        throw std::runtime_error("relayout: shape");
    if (a.N == 0) return;
    TileGeom g;
    g.tiles_p = (a.P + kTile - 1) / kTile;
    g.tiles_c = (a.C + kTile - 1) / kTile;
    g.tiles = static_cast<int64_t>(a.N) * g.tiles_p * g.tiles_c;
    const float* planar = IN ? a.src : a.dst;
    const float* rows = IN ? a.dst : a.src;
    const bool vp = a.P % 4 == 0 && a.planar_c % 4 == 0 && a.planar_n % 4 == 0 && aligned16(planar) &&
                    aligned16(a.mirror);
    const bool vr = a.C % 4 == 0 && a.rows_p % 4 == 0 && a.rows_n % 4 == 0 && aligned16(rows);
    const bool vs = IN ? vp : vr, vd = IN ? vr : vp;
    const dim3 grid(static_cast<unsigned>(std::min<int64_t>(g.tiles, a.host ? kTransferBlocks : kRelayoutBlocks)));
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kLanes), 0, s, a, g); };
    if (vs && vd) go(relayout_kernel<IN, true, true>);
    else if (vs) go(relayout_kernel<IN, true, false>);
    else if (vd) go(relayout_kernel<IN, false, true>);
    else go(relayout_kernel<IN, false, false>);
}

// One run a blockIdx.y: its float4s, four loads in flight a lane, and the
// floats after them.
struct CopyRuns {
    CopyRun r[2];
};
__global__ __launch_bounds__(kLanes) void copy_floats_kernel(CopyRuns runs) {
    const CopyRun r = runs.r[blockIdx.y];
    const int64_t n4 = r.n / 4;
    const int64_t tid = blockIdx.x * static_cast<int64_t>(kLanes) + threadIdx.x;
    const int64_t step = static_cast<int64_t>(gridDim.x) * kLanes;
    const float4* s = reinterpret_cast<const float4*>(r.src);
    float4* d = reinterpret_cast<float4*>(r.dst);
    for (int64_t i = tid; i < n4; i += 4 * step) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = s[min(i + u * step, n4 - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * step < n4) d[i + u * step] = v[u];
    }
    if (tid < r.n - 4 * n4) r.dst[4 * n4 + tid] = r.src[4 * n4 + tid];
}

}  // namespace

void launch_planar_to_rows(const RelayoutArgs& a, hipStream_t s) { launch_relayout<true>(a, s); }
void launch_rows_to_planar(const RelayoutArgs& a, hipStream_t s) { launch_relayout<false>(a, s); }

void launch_copy_floats(std::initializer_list<CopyRun> runs, hipStream_t s) {
    CopyRuns c;
    unsigned count = 0;
    int64_t most = 0;
    for (const CopyRun& r : runs) {
        if (r.n <= 0) continue;
        if (count == 2 || !r.dst || !r.src || !aligned16(r.dst) || !aligned16(r.src))
            throw std::runtime_error("copy: runs");
        c.r[count++] = r;
        most = std::max(most, r.n);
    }
    if (count == 0) return;
    const int64_t per = 16 * kLanes;  // floats of a workgroup's loads in flight
    const int64_t blocks = std::min<int64_t>((most + per - 1) / per, kTransferBlocks / count);
    hipLaunchKernelGGL(copy_floats_kernel, dim3(static_cast<unsigned>(blocks), count), dim3(kLanes), 0, s, c);
}

}  // namespace k
}  // namespace pdefa
