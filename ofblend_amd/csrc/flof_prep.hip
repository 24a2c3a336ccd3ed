// flof_prep.hip -- input preprocessing of the FlOF pipeline and the .uni
// grid file format.
//
// Reference: source/plugin/optflow4d.cpp -- repeatFrame4d :1254-1266,
// knExtrap4dLsSimple / knSetRemaining4d / extrap4dLsSimple :1323-1406;
// source/fileio.cpp -- UniHeader :38-44, getUniFileSize :572-599,
// writeGridUni / readGridUni (MNT2) :608-731, writeGrid4dUni /
// readGrid4dUni (M4T2) :834-999.

#include <zlib.h>

#include <algorithm>
#include <cstring>
#include <ctime>
#include <string>
#include <vector>

#include "flof_internal.h"

namespace flof {

// ---------------------------------------------------------------------------
// repeatFrame4d: every (bnd-interior) column takes its quadrilinear sample at
// time srct, written to slices [t_lo, t_hi].  A thread reads its column
// before writing it; other columns enter the sample with weight 0 only.
__global__ void k_repeat_frame(float *__restrict__ phi, Dims4 D, float srct, int t_lo,
                               int t_hi, int bnd)
{
    const int nx = D.X - 2 * bnd, ny = D.Y - 2 * bnd, nz = D.Z - 2 * bnd;
    if (nx <= 0 || ny <= 0 || nz <= 0) return;
    const int64_t n = (int64_t)nx * ny * nz;
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int i = bnd + (int)(c % nx);
        const int j = bnd + (int)((c / nx) % ny);
        const int k = bnd + (int)(c / ((int64_t)nx * ny));
        const float v = interp4<float>(phi, D, (float)i + 0.5f, (float)j + 0.5f,
                                       (float)k + 0.5f, srct + 0.5f);
        const int64_t c3 = (int64_t)i + (int64_t)D.X * j + D.sz * k;
        for (int t = t_lo; t <= t_hi; ++t) phi[c3 + D.st * t] = v;
    }
}

// ---------------------------------------------------------------------------
// extrap4dLsSimple.  The layers that the reference grows one after another are
// the cells' city-block distances to the marked cells, clipped to the interior:
// a shortest path to the nearest marked cell has only nearer, so unmarked,
// cells on it.  The distances are made by one pass per axis (a byte per cell
// wherever 254 is out of reach), which leaves a pass per layer for the values
// only, layer d from layer d - 1: 1 instead of 4 bytes per cell to look at.
// 40^3 x 60, 40 layers: 7.6 -> 3.8 us per layer, 310 -> 180 us in all.  Few
// layers, few cells or long lines grow layer by layer (extrap_grow).
//
// Distances above any layer, and the outer cells': never a layer's number.
template <class U> constexpr U EX_FAR = (U)~(U)0;
template <class U> __device__ __forceinline__ U ex_step(U a, uint32_t by)
{
    const uint32_t far = EX_FAR<U>;
    return (U)(far - a < by ? far : a + by);
}

// marks and distances along x: a wavefront per row, 64 cells at a time, the
// nearest marked cell to both sides from the ballot of the marks
template <class U>
__global__ void k_extrap_mark_x(const float *__restrict__ phi, U *__restrict__ dist, Dims4 D,
                                int inside, int64_t padded)
{
    const int lane = threadIdx.x & 63;
    const int64_t rows = (int64_t)D.Y * D.Z * D.T;
    const int64_t w0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
    const int64_t nw = ((int64_t)gridDim.x * blockDim.x) >> 6;
    if (w0 == 0)  // the last layer-kernel load
        for (int64_t c = D.st * D.T + lane; c < padded; c += 64) dist[c] = EX_FAR<U>;
    for (int64_t r = w0; r < rows; r += nw) {
        const int j = (int)(r % D.Y), k = (int)(r / D.Y % D.Z), t = (int)(r / D.Y / D.Z);
        const bool in = j >= 1 && k >= 1 && t >= 1 && j < D.Y - 1 && k < D.Z - 1 && t < D.T - 1;
        const int64_t c0 = r * D.X;
        auto marks = [&](int x0) {
            const int x = x0 + lane;
            const float v = in && x >= 1 && x < D.X - 1 ? phi[c0 + x] : 0.f;
            return (unsigned long long)__ballot(!inside ? v < 0.f : v > 0.f);
        };
        U carry = EX_FAR<U>;  // of the cell before the chunk, to its left
        for (int x0 = 0; x0 < D.X; x0 += 64) {
            const unsigned long long m = marks(x0);
            const unsigned long long lo = m & (~0ull >> (63 - lane)), hi = m >> lane;
            U d = ex_step(carry, 1 + lane);
            if (lo) d = (U)(lane - (63 - __clzll(lo)));
            carry = (U)__shfl((int)d, 63);
            if (hi) d = min(d, (U)(__ffsll((long long)hi) - 1));
            const int x = x0 + lane;
            if (x < D.X) dist[c0 + x] = in && x >= 1 && x < D.X - 1 ? d : EX_FAR<U>;
        }
        carry = EX_FAR<U>;  // of the cell behind the chunk, to its right
        for (int x0 = (D.X - 1) & ~63; x0 > 0; x0 -= 64) {
            const unsigned long long m = marks(x0);
            carry = m ? (U)(__ffsll((long long)m) - 1) : ex_step(carry, 64);
            const int x = x0 - 64 + lane;
            if (in && x >= 1) dist[c0 + x] = min(dist[c0 + x], ex_step(carry, 64 - lane));
        }
    }
}

// distances along y, z or t: a thread per interior line, down and up again, 16
// loads under way.  LAST: cells beyond `reach` take `set`.
template <class U, bool LAST>
__global__ void k_extrap_line(U *__restrict__ dist, float *__restrict__ phi, int nx, int64_t sx,
                              int n1, int64_t s1, int n2, int64_t s2, int len, int64_t stride,
                              uint32_t reach, float set)
{
    constexpr int B = 16;
    const int64_t lines = (int64_t)(nx - 2) * (n1 - 2) * (n2 - 2);
    for (int64_t l = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; l < lines;
         l += (int64_t)gridDim.x * blockDim.x) {
        const int64_t a = l / (nx - 2);
        const int64_t c0 = (1 + l % (nx - 2)) * sx + (1 + a % (n1 - 2)) * s1 +
                           (1 + a / (n1 - 2)) * s2 + stride;
        const int n = len - 2;
        U d = EX_FAR<U>;
        for (int b = 0; b < n; b += B) {
            U v[B];
#pragma unroll
            for (int i = 0; i < B; ++i) v[i] = dist[c0 + min(b + i, n - 1) * stride];
#pragma unroll
            for (int i = 0; i < B; ++i)
                if (b + i < n) {
                    d = min(v[i], ex_step(d, 1));
                    dist[c0 + (b + i) * stride] = d;
                }
        }
        d = EX_FAR<U>;
        for (int b = n - 1; b >= 0; b -= B) {
            U v[B];
#pragma unroll
            for (int i = 0; i < B; ++i) v[i] = dist[c0 + max(b - i, 0) * stride];
#pragma unroll
            for (int i = 0; i < B; ++i)
                if (b - i >= 0) {
                    d = min(v[i], ex_step(d, 1));
                    dist[c0 + (b - i) * stride] = d;
                    if (LAST && d > reach) phi[c0 + (b - i) * stride] = set;
                }
        }
    }
}

// The cells of layer d: mean of the neighbours in layer d - 1 (x-, x+, y-, y+,
// z-, z+, t-, t+ order) plus `direction`.  A launch of a few microseconds whose
// length is three dependent memory accesses: a thread looks at 16 bytes of
// distances, the block lists its cells of the layer, and the list's
// neighbours are all read at once (a launch that does nothing takes about 3
// of its 3.8 us).  (The neighbours' values are read whether
// they are used or not; another cell of the layer among them may be written
// meanwhile, its value is not used.)
template <class U>
__global__ void __launch_bounds__(256)
k_extrap_layer(float *__restrict__ phi, const U *__restrict__ dist, Dims4 D, int64_t groups,
               uint32_t d, float direction)
{
    constexpr int C = 16 / sizeof(U);
    __shared__ unsigned short list[256 * C];
    __shared__ int count;
    const int64_t off[8] = {-1, 1, -(int64_t)D.X, (int64_t)D.X, -D.sz, D.sz, -D.st, D.st};
    for (int64_t g0 = blockIdx.x * (int64_t)256; g0 < groups; g0 += (int64_t)gridDim.x * 256) {
        if (threadIdx.x == 0) count = 0;
        union {
            uint4 w;
            U u[C];
        } v;
        v.w = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (g0 + threadIdx.x < groups) v.w = ((const uint4 *)dist)[g0 + threadIdx.x];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < C; ++i)
            if (v.u[i] == d) list[atomicAdd(&count, 1)] = (unsigned short)(threadIdx.x * C + i);
        __syncthreads();
        for (int e = threadIdx.x; e < count; e += 256) {
            const int64_t c = g0 * C + list[e];
            U du[8];
            float f[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                du[q] = dist[c + off[q]];
                f[q] = phi[c + off[q]];
            }
            int nbs = 0;
            float avg = 0.f;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (du[q] == d - 1) {
                    avg = avg + f[q];
                    nbs++;
                }
            phi[c] = avg / (float)nbs + direction;
        }
        __syncthreads();
    }
}

// The same layers grown one after another: a byte per cell (wherever 253 is out
// of reach) holds its layer, "free" (interior, not reached yet) or "outer", and a
// pass turns the free cells next to layer d - 1 into layer d.  Two dependent
// accesses per pass: a cell's own byte, then its neighbours' bytes and values
// together.  (Neighbours may become layer d meanwhile: neither their old nor
// their new byte is d - 1.)
template <class U> constexpr U EG_FREE = (U)~(U)0;
template <class U> constexpr U EG_OUTER = EG_FREE<U> - 1;

template <class U>
__global__ void __launch_bounds__(256)
k_extrap_grow_mark(const float *__restrict__ phi, U *__restrict__ layer, Dims4 D, Coord4 C,
                   int inside)
{
    const int64_t n = D.st * D.T;
    for (int64_t c = blockIdx.x * (int64_t)256 + threadIdx.x; c < n;
         c += (int64_t)gridDim.x * 256) {
        int i, j, k, t;
        decompose((uint32_t)c, C, i, j, k, t);
        U u = EG_OUTER<U>;
        if (i >= 1 && j >= 1 && k >= 1 && t >= 1 && i < D.X - 1 && j < D.Y - 1 && k < D.Z - 1 &&
            t < D.T - 1) {
            const float v = phi[c];
            u = (!inside ? v < 0.f : v > 0.f) ? (U)0 : EG_FREE<U>;
        }
        layer[c] = u;
    }
}

// cells [c0, c1) hold the interior; last: free cells that stay free take `set`
template <class U>
__global__ void __launch_bounds__(256)
k_extrap_grow(float *__restrict__ phi, U *layer, Dims4 D, int64_t c0, int64_t c1, uint32_t d,
              float direction, int last, float set)
{
    const int64_t off[8] = {-1, 1, -(int64_t)D.X, (int64_t)D.X, -D.sz, D.sz, -D.st, D.st};
    for (int64_t c = c0 + blockIdx.x * (int64_t)256 + threadIdx.x; c < c1;
         c += (int64_t)gridDim.x * 256) {
        if (layer[c] != EG_FREE<U>) continue;
        U b[8];
        float f[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            b[q] = layer[c + off[q]];
            f[q] = phi[c + off[q]];
        }
        int nbs = 0;
        float avg = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (b[q] == d - 1) {
                avg = avg + f[q];
                nbs++;
            }
        if (nbs > 0) {
            layer[c] = (U)d;
            if (d >= 2) phi[c] = avg / (float)nbs + direction;  // (the first keeps its values)
        } else if (last) {
            phi[c] = set;
        }
    }
}

template <class U>
static void extrap_grow(flof_ctx *ctx, float *phi, const Dims4 &D, int distance, int layers,
                        bool inside)
{
    const int64_t n = D.st * D.T;
    if (D.X < 3 || D.Y < 3 || D.Z < 3 || D.T < 3) return;  // no interior cell
    Tmp tmp(ctx, (size_t)n * sizeof(U));
    U *layer = tmp.as<U>();
    const float direction = inside ? -1.f : 1.f;
    const float set = direction * (float)(distance + 2);
    hipLaunchKernelGGL(k_extrap_grow_mark<U>, dim3(grid_blocks(ctx, n)), dim3(256), 0,
                       ctx->stream, (const float *)phi, layer, D, make_coord4(D), inside ? 1 : 0);
    const int64_t c0 = D.st, c1 = n - D.st;  // (every neighbour of these is in the grid or outer)
    const int last = std::max(1, layers);
    for (int d = 1; d <= last; ++d)
        hipLaunchKernelGGL(k_extrap_grow<U>, dim3(grid_blocks(ctx, c1 - c0)), dim3(256), 0,
                           ctx->stream, phi, layer, D, c0, c1, (uint32_t)d, direction,
                           d == last ? 1 : 0, set);
}

template <class U>
static void extrap_layers(flof_ctx *ctx, float *phi, const Dims4 &D, int distance, int farthest,
                          bool inside)
{
    const int64_t n = D.st * D.T;
    const int64_t groups = (n * (int64_t)sizeof(U) + 15) / 16;
    const int64_t padded = groups * 16 / (int64_t)sizeof(U);
    Tmp tmp(ctx, (size_t)groups * 16);
    U *dist = tmp.as<U>();
    const float direction = inside ? -1.f : 1.f;
    const float set = direction * (float)(distance + 2);
    const int layers = std::min(distance, farthest);
    const uint32_t reach = (uint32_t)std::max(1, layers);
    const int64_t rows = (int64_t)D.Y * D.Z * D.T;
    hipLaunchKernelGGL(k_extrap_mark_x<U>, dim3(grid_blocks(ctx, rows * 64)), dim3(256), 0,
                       ctx->stream, (const float *)phi, dist, D, inside ? 1 : 0, padded);
    const int nx = D.X, ny = D.Y, nz = D.Z, nt = D.T;
    if (nx < 3 || ny < 3 || nz < 3 || nt < 3) return;
    auto blocks = [&](int a, int b, int c) {
        return dim3(grid_blocks(ctx, (int64_t)(a - 2) * (b - 2) * (c - 2)));
    };
    hipLaunchKernelGGL((k_extrap_line<U, false>), blocks(nx, nz, nt), dim3(256), 0, ctx->stream,
                       dist, phi, nx, (int64_t)1, nz, D.sz, nt, D.st, ny, (int64_t)nx, reach, set);
    hipLaunchKernelGGL((k_extrap_line<U, false>), blocks(nx, ny, nt), dim3(256), 0, ctx->stream,
                       dist, phi, nx, (int64_t)1, ny, (int64_t)nx, nt, D.st, nz, D.sz, reach, set);
    hipLaunchKernelGGL((k_extrap_line<U, true>), blocks(nx, ny, nz), dim3(256), 0, ctx->stream,
                       dist, phi, nx, (int64_t)1, ny, (int64_t)nx, nz, D.sz, nt, D.st, reach, set);
    for (int d = 2; d <= layers; ++d)
        hipLaunchKernelGGL(k_extrap_layer<U>, dim3(grid_blocks(ctx, groups)), dim3(256), 0,
                           ctx->stream, phi, (const U *)dist, D, groups, (uint32_t)d, direction);
}

// ---------------------------------------------------------------------------
// .uni format (fileio.cpp:38-44): "MNT2"/"M4T2" + header; M4T2 adds int dimT,
// then the slices; gzip level 1 on write.
struct UniHeader {
    int dimX, dimY, dimZ;
    int gridType, elementType, bytesPerElement;
    char info[256];
    unsigned long long timestamp;
};
static_assert(sizeof(UniHeader) == 288, "UniHeader layout");

struct Gz {
    gzFile f = nullptr;
    ~Gz()
    {
        if (f) gzclose(f);
    }
};

static void gz_read_all(gzFile f, void *dst, size_t bytes, const std::string &name)
{
    char *p = (char *)dst;
    while (bytes > 0) {
        const unsigned chunk = (unsigned)std::min<size_t>(bytes, 1u << 30);
        const int got = gzread(f, p, chunk);
        if (got <= 0) throw Error{FLOF_ERR_ARG, "can't read file " + name + ": truncated"};
        p += got;
        bytes -= (size_t)got;
    }
}
static void gz_write_all(gzFile f, const void *src, size_t bytes, const std::string &name)
{
    const char *p = (const char *)src;
    while (bytes > 0) {
        const unsigned chunk = (unsigned)std::min<size_t>(bytes, 1u << 30);
        const int put = gzwrite(f, p, chunk);
        if (put <= 0) throw Error{FLOF_ERR_ARG, "can't write file " + name};
        p += put;
        bytes -= (size_t)put;
    }
}

// grid type and element type codes written by the reference for 4D grids
// (Grid4dBase::Grid4dType, fileio.cpp:848-857)
static void uni_types(int elem, int &gridType, int &elementType, int &bpe)
{
    switch (elem) {
    case FLOF_INT: gridType = 2; elementType = 0; bpe = 4; break;
    case FLOF_VEC4: gridType = 8; elementType = 2; bpe = 16; break;
    default: gridType = 1; elementType = 1; bpe = 4; break;
    }
}

void uni_write4d(const std::string &name, const void *host, int X, int Y, int Z, int T,
                 int elem)
{
    UniHeader h;
    std::memset(&h, 0, sizeof(h));
    h.dimX = X;
    h.dimY = Y;
    h.dimZ = Z;
    uni_types(elem, h.gridType, h.elementType, h.bytesPerElement);
    std::snprintf(h.info, sizeof(h.info), "%s", "ofblend_amd flof (gfx950)");
    h.timestamp = (unsigned long long)std::time(nullptr);
    Gz gz;
    gz.f = gzopen(name.c_str(), "wb1");
    FLOF_REQUIRE(gz.f, FLOF_ERR_ARG, "can't open file " + name);
    gz_write_all(gz.f, "M4T2", 4, name);
    gz_write_all(gz.f, &h, sizeof(h), name);
    gz_write_all(gz.f, &T, sizeof(int), name);
    const size_t slice = (size_t)X * Y * Z * h.bytesPerElement;
    for (int t = 0; t < T; ++t) gz_write_all(gz.f, (const char *)host + slice * t, slice, name);
    const int rc = gzclose(gz.f);
    gz.f = nullptr;
    FLOF_REQUIRE(rc == Z_OK, FLOF_ERR_ARG, "error closing " + name);
}

// reads the header: returns "MNT2" or "M4T2" files' sizes (T = 1 for 3D)
static void uni_header(gzFile f, const std::string &name, UniHeader &h, int &T, bool &is4d)
{
    char id[5] = {0, 0, 0, 0, 0};
    gz_read_all(f, id, 4, name);
    if (!std::strcmp(id, "M4T2")) is4d = true;
    else if (!std::strcmp(id, "MNT2")) is4d = false;
    else throw Error{FLOF_ERR_ARG, "Unknown header in " + name};
    gz_read_all(f, &h, sizeof(h), name);
    T = 1;
    if (is4d) gz_read_all(f, &T, sizeof(int), name);
}

void uni_size(const std::string &name, int dims[4])
{
    Gz gz;
    gz.f = gzopen(name.c_str(), "rb");
    FLOF_REQUIRE(gz.f, FLOF_ERR_ARG, "can't open file " + name);
    UniHeader h;
    int T;
    bool is4d;
    uni_header(gz.f, name, h, T, is4d);
    dims[0] = h.dimX;
    dims[1] = h.dimY;
    dims[2] = h.dimZ;
    dims[3] = T;
}

// unifyGridType (fileio.cpp:470-479): Real <> levelset, Vec3 <> MAC bits
static int unify(int t)
{
    if (t & 1) t |= 16;
    if (t & 16) t |= 1;
    if (t & 4) t |= 8;
    if (t & 8) t |= 4;
    return t;
}

void uni_read(const std::string &name, void *host, int X, int Y, int Z, int T, int elem)
{
    Gz gz;
    gz.f = gzopen(name.c_str(), "rb");
    FLOF_REQUIRE(gz.f, FLOF_ERR_ARG, "can't open file " + name);
    UniHeader h;
    int fT;
    bool is4d;
    uni_header(gz.f, name, h, fT, is4d);
    int gt, et, bpe;
    uni_types(elem, gt, et, bpe);
    FLOF_REQUIRE(h.dimX == X && h.dimY == Y && h.dimZ == Z && fT == T, FLOF_ERR_DIM,
                 "grid dim doesn't match in " + name);
    FLOF_REQUIRE(h.bytesPerElement == bpe, FLOF_ERR_TYPE,
                 "grid element size doesn't match in " + name);
    FLOF_REQUIRE(unify(h.gridType) == unify(gt), FLOF_ERR_TYPE,
                 "grid type doesn't match in " + name);
    gz_read_all(gz.f, host, (size_t)X * Y * Z * T * bpe, name);
}

}  // namespace flof

using namespace flof;

#define API_TRY try {
#define API_CATCH(ctx)                                                        \
    }                                                                         \
    catch (const flof::Error &e)                                              \
    {                                                                         \
        flof::set_error(ctx, e);                                              \
        return e.code;                                                        \
    }                                                                         \
    catch (const std::exception &e)                                           \
    {                                                                         \
        flof::set_error(ctx, flof::Error{FLOF_ERR_ARG, e.what()});            \
        return FLOF_ERR_ARG;                                                  \
    }                                                                         \
    return FLOF_OK;

extern "C" {

int flof_repeat_frame4d(flof_grid4d *phi, float srct, float range, int bnd)
{
    flof_ctx *ctx = phi ? phi->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(phi && phi->elem == FLOF_REAL && phi->dtype == FLOF_F32, FLOF_ERR_TYPE,
                 "repeatFrame4d: REAL FP32 grid");
    const int t_lo = int(srct - range + 0.5f), t_hi = int(srct);
    if (t_hi < t_lo) return FLOF_OK;
    FLOF_REQUIRE(t_lo >= 0 && t_hi < phi->T && bnd >= 0, FLOF_ERR_RANGE,
                 "repeatFrame4d: slices outside the grid");
    FLOF_REQUIRE(phi->X >= 2 && phi->Y >= 2 && phi->Z >= 2 && phi->T >= 2, FLOF_ERR_DIM,
                 "repeatFrame4d: grid too small");
    Dims4 D = dims_of(phi);
    const int64_t n = (int64_t)std::max(0, D.X - 2 * bnd) * std::max(0, D.Y - 2 * bnd) *
                      std::max(0, D.Z - 2 * bnd);
    hipLaunchKernelGGL(k_repeat_frame, dim3(grid_blocks(ctx, n)), dim3(256), 0, ctx->stream,
                       (float *)phi->data, D, srct, t_lo, t_hi, bnd);
    check_launch("k_repeat_frame");
    API_CATCH(ctx)
}

int flof_extrap4d_ls_simple(flof_grid4d *phi, int distance, int inside)
{
    flof_ctx *ctx = phi ? phi->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(phi && phi->elem == FLOF_REAL && phi->dtype == FLOF_F32, FLOF_ERR_TYPE,
                 "extrap4dLsSimple: REAL FP32 grid");
    Dims4 D = dims_of(phi);
    // no interior cell is farther from another
    const int64_t farthest = (int64_t)D.X + D.Y + D.Z + D.T - 12;
    const int far = (int)std::max<int64_t>(0, std::min<int64_t>(farthest, 0x7fffffff));
    const int layers = std::min(distance, far);
    // The distances cost their serial passes along y, z and t (0.16 us per cell
    // of a line), and save about 1 us per layer beyond the fifth and million
    // interior cells.  Calls of 1, 4, 16, 40 layers, grown / by distances, us:
    // 16^4 17, 25, 67, 124 / 27, 44, 82, 138; 64^3 x 4 18, 30, 77, 166 / 42, 57,
    // 119, 236; 40^3 x 60 32, 73, 259, 423 / 70, 99, 216, 314; 64^4 69, 202, 797,
    // 1884 / 140, 222, 671, 1398.
    const int64_t interior = (int64_t)std::max(0, D.X - 2) * std::max(0, D.Y - 2) *
                             std::max(0, D.Z - 2) * std::max(0, D.T - 2);
    const bool grow = (double)(layers - 5) * (double)interior <=
                      160000. * ((double)D.Y + D.Z + D.T);
    float *p = (float *)phi->data;
    if (grow && layers < 254)
        extrap_grow<uint8_t>(ctx, p, D, distance, layers, inside != 0);
    else if (grow)
        extrap_grow<uint32_t>(ctx, p, D, distance, layers, inside != 0);
    else if (layers < 255)
        extrap_layers<uint8_t>(ctx, p, D, distance, far, inside != 0);
    else
        extrap_layers<uint32_t>(ctx, p, D, distance, far, inside != 0);
    check_launch("k_extrap_*");
    API_CATCH(ctx)
}

int flof_shift_forw_grid4d(flof_grid4d *phi, int overrideGoodRegion)
{
    flof_ctx *ctx = phi ? phi->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(phi && phi->elem == FLOF_REAL, FLOF_ERR_TYPE, "shiftForwGrid4d: REAL grid");
    FLOF_REQUIRE(overrideGoodRegion >= 0 && overrideGoodRegion <= phi->T, FLOF_ERR_RANGE,
                 "shiftForwGrid4d: good region outside the grid");
    // optflow4d.cpp:1598-1616: slices [0, good) take slices [shift, shift+good)
    const int shift = phi->T - overrideGoodRegion;
    const size_t sl = (size_t)phi->X * phi->Y * phi->Z * 4;
    for (int s = 0; s < overrideGoodRegion; s += std::max(1, shift)) {
        int len = shift;
        if (s + shift >= overrideGoodRegion) len = overrideGoodRegion - s;
        if (len <= 0 || shift <= 0) break;
        FLOF_HIP(hipMemcpyAsync((char *)phi->data + sl * s, (char *)phi->data + sl * (s + shift),
                                sl * len, hipMemcpyDeviceToDevice, ctx->stream));
    }
    API_CATCH(ctx)
}

int flof_uni_file_size(const char *name, int dims[4])
{
    try {
        FLOF_REQUIRE(name && dims, FLOF_ERR_ARG, "getUniFileSize: null argument");
        uni_size(name, dims);
    } catch (const flof::Error &e) {
        return e.code;
    }
    return FLOF_OK;
}

int flof_uni_write4d(const char *name, const void *host, int X, int Y, int Z, int T, int elem)
{
    try {
        FLOF_REQUIRE(name && host && X > 0 && Y > 0 && Z > 0 && T > 0, FLOF_ERR_ARG,
                     "writeGrid4dUni: bad argument");
        uni_write4d(name, host, X, Y, Z, T, elem);
    } catch (const flof::Error &e) {
        return e.code;
    }
    return FLOF_OK;
}

int flof_uni_read(const char *name, void *host, int X, int Y, int Z, int T, int elem)
{
    try {
        FLOF_REQUIRE(name && host, FLOF_ERR_ARG, "readGridUni: bad argument");
        uni_read(name, host, X, Y, Z, T, elem);
    } catch (const flof::Error &e) {
        return e.code;
    }
    return FLOF_OK;
}

// the reference formats file names with snprintf(pattern, index): accept
// exactly one integer conversion (%d / %i with optional flags and width)
static std::string format_index(const char *pattern, int idx)
{
    int conv = 0;
    for (const char *c = pattern; *c; ++c) {
        if (*c != '%') continue;
        if (c[1] == '%') {
            ++c;
            continue;
        }
        const char *e = c + 1;
        while (*e && std::strchr("0123456789-+ #", *e)) ++e;
        FLOF_REQUIRE(*e == 'd' || *e == 'i', FLOF_ERR_ARG,
                     std::string("file pattern needs one integer conversion: ") + pattern);
        ++conv;
        c = e;
    }
    FLOF_REQUIRE(conv == 1, FLOF_ERR_ARG,
                 std::string("file pattern needs one integer conversion: ") + pattern);
    char buf[4096];
    std::snprintf(buf, sizeof(buf), pattern, idx);
    return buf;
}

int flof_load_place_grid4d_uni(const char *fname, flof_grid4d *phi, const float offset[4],
                               const float scale[4], int fileIdxStart, int fileIdxEnd,
                               int debugSkipLoad, float spread, const float overrideSize[4],
                               float overrideTimeOff, int overrideGoodRegion,
                               float loadTimeScale, int rescaleSdfValues, float sdfIsoOff,
                               float repeatStartFrame)
{
    flof_ctx *ctx = phi ? phi->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(fname && phi && offset && scale, FLOF_ERR_ARG,
                 "loadPlaceGrid4d: null argument");
    // the size comes from the file of index fileIdxStart as passed
    int dims[4];
    uni_size(format_index(fname, fileIdxStart), dims);
    FLOF_REQUIRE(dims[0] >= 1 && dims[1] >= 1 && dims[2] >= 1, FLOF_ERR_DIM,
                 std::string("Invalid src size from ") + fname);
    const size_t fsz = (size_t)dims[0] * dims[1] * dims[2];
    std::vector<float> host(fsz);
    Tmp dev(ctx, fsz * 4);
    place_frames(
        phi, dims[0], dims[1], dims[2], nullptr,
        [&](int f) -> const float * {
            // kernels of the previous frame may still read the buffer
            FLOF_HIP(hipStreamSynchronize(ctx->stream));
            uni_read(format_index(fname, f), host.data(), dims[0], dims[1], dims[2], 1,
                     FLOF_REAL);
            FLOF_HIP(hipMemcpyAsync(dev.p, host.data(), fsz * 4, hipMemcpyHostToDevice,
                                    ctx->stream));
            FLOF_HIP(hipStreamSynchronize(ctx->stream));
            return dev.as<float>();
        },
        offset, scale, fileIdxStart, fileIdxEnd, debugSkipLoad, spread, overrideSize,
        overrideTimeOff, overrideGoodRegion, loadTimeScale, rescaleSdfValues, sdfIsoOff,
        repeatStartFrame);
    API_CATCH(ctx)
}

int flof_warp_state_open(flof_ctx *ctx, const char *fname, int useDefoVols, int doAligned,
                         float partialLoadFac, flof_warp_state **out)
{
    API_TRY
    FLOF_REQUIRE(ctx && fname && out, FLOF_ERR_ARG, "loadAdvectTimeSlice_OptInit: null argument");
    *out = nullptr;
    flof_warp_state *s = new flof_warp_state();
    s->ctx = ctx;
    s->use_vols = useDefoVols != 0;
    s->aligned = doAligned != 0;
    s->partial = partialLoadFac;
    const int rc = flof_warp_state_add(s, fname);
    if (rc != FLOF_OK) {
        delete s;
        return rc;
    }
    *out = s;
    API_CATCH(ctx)
}

int flof_warp_state_add(flof_warp_state *s, const char *fname)
{
    flof_ctx *ctx = s ? s->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(s && fname, FLOF_ERR_ARG, "loadAdvectTimeSlice_OptAdd: null argument");
    // without deformation volumes the reference ignores the call
    if (!s->defos.empty() && !s->use_vols) return FLOF_OK;
    FLOF_REQUIRE((int)s->defos.size() < 9, FLOF_ERR_RANGE, "Too many defovolumes loaded!");
    int d[4];
    uni_size(fname, d);
    FLOF_REQUIRE(d[0] >= 2 && d[1] >= 2 && d[2] >= 2 && d[3] >= 1, FLOF_ERR_DIM,
                 std::string("Invalid src size from ") + fname);
    flof_grid4d *g = nullptr;
    int rc = flof_grid4d_create(ctx, d[0], d[1], d[2], d[3], FLOF_VEC4, FLOF_F32, &g);
    if (rc != FLOF_OK) return rc;
    rc = flof_grid4d_load(g, fname);
    if (rc != FLOF_OK) {
        flof_grid4d_destroy(g);
        return rc;
    }
    s->defos.push_back(g);
    API_CATCH(ctx)
}

int flof_warp_state_run(flof_warp_state *s, float *dst, int dx, int dy, int dz,
                        flof_grid4d *phi, float time, float blendAlpha, float loadTimeScale,
                        const float defoOffset[4], const float defoScale[4],
                        const float defoFactor[4], const float overrideSize[4],
                        float overrideTimeOff, int zeroVel, float thirdAlpha, int bordSkip,
                        float fourthAlpha, float defoAniFac)
{
    if (!s || s->defos.empty()) return FLOF_ERR_ARG;
    if (!s->use_vols)
        return flof_advect_time_slice_opt(s->defos[0], dst, dx, dy, dz, phi, time, blendAlpha,
                                          loadTimeScale, defoOffset, defoScale, defoFactor,
                                          overrideSize, overrideTimeOff, zeroVel, bordSkip,
                                          defoAniFac);
    return flof_advect_time_slice_vols(s->defos.data(), (int)s->defos.size(), dst, dx, dy, dz,
                                       phi, time, blendAlpha, loadTimeScale, defoOffset,
                                       defoScale, defoFactor, overrideSize, overrideTimeOff,
                                       zeroVel, bordSkip, defoAniFac, s->aligned ? 1 : 0,
                                       s->partial, thirdAlpha, fourthAlpha);
}

int flof_warp_state_close(flof_warp_state *s)
{
    if (!s) return FLOF_ERR_ARG;
    for (flof_grid4d *g : s->defos) flof_grid4d_destroy(g);
    delete s;
    return FLOF_OK;
}

int flof_load_vel_rescaled(flof_grid4d *vel, const char *fname, const int defoSize[4],
                           const float defoOffset[4], const float defoScale[4],
                           const float defoFactor[4])
{
    flof_ctx *ctx = vel ? vel->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(vel && fname && defoOffset && defoScale && defoFactor, FLOF_ERR_ARG,
                 "loadVelRescaled: null argument");
    FLOF_REQUIRE(vel->elem == FLOF_VEC4, FLOF_ERR_TYPE, "loadVelRescaled: vel must be VEC4");
    int d[4];
    if (defoSize) {
        for (int i = 0; i < 4; ++i) d[i] = defoSize[i];
    } else {
        uni_size(fname, d);
    }
    // the deformation grid of the defo solver's size; load() rejects a file
    // of another size, as readGrid4dUni does
    flof_grid4d *ipol = nullptr;
    int rc = flof_grid4d_create(ctx, d[0], d[1], d[2], d[3], FLOF_VEC4, FLOF_F32, &ipol);
    if (rc != FLOF_OK) return rc;
    const float whole[4] = {-1.f, -1.f, -1.f, -1.f};
    rc = flof_grid4d_load(ipol, fname);
    if (rc == FLOF_OK) rc = flof_interpolate_grid4d(vel, ipol, defoOffset, defoScale, whole);
    if (rc == FLOF_OK) rc = flof_grid4d_mult_const(vel, defoFactor);
    flof_grid4d_destroy(ipol);  // waits for the stream before freeing
    return rc;
    API_CATCH(ctx)
}

int flof_grid4d_save(flof_grid4d *g, const char *name)
{
    flof_ctx *ctx = g ? g->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(g && name && g->dtype == FLOF_F32, FLOF_ERR_ARG, "Grid4d::save: bad argument");
    std::vector<char> host(g->bytes);
    FLOF_HIP(hipMemcpyAsync(host.data(), g->data, g->bytes, hipMemcpyDeviceToHost,
                            ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    uni_write4d(name, host.data(), g->X, g->Y, g->Z, g->T, g->elem);
    API_CATCH(ctx)
}

int flof_grid4d_load(flof_grid4d *g, const char *name)
{
    flof_ctx *ctx = g ? g->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(g && name && g->dtype == FLOF_F32, FLOF_ERR_ARG, "Grid4d::load: bad argument");
    std::vector<char> host(g->bytes);
    uni_read(name, host.data(), g->X, g->Y, g->Z, g->T, g->elem);
    FLOF_HIP(hipMemcpyAsync(g->data, host.data(), g->bytes, hipMemcpyHostToDevice,
                            ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

}  // extern "C"
