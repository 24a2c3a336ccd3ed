// flof_warmnet.hip -- the learned warm start of the multiscale solve (no
// reference counterpart; the reference always starts every level's CG from
// zero, source/plugin/optflow4d.cpp:284-303).
//
// A small space-time convolutional network maps the two SDFs of a solve,
// restricted to a coarse pyramid level, to a 4D flow; the flow is prolonged
// to the finest level and handed to the solve as its warm start (the solve
// keeps it only where its residual is not larger than the zero start's).
//
// Network (C = 16 channels, activations channels-last [cell][16]):
//   h0 = lift(i0/4, i1/4)                       pointwise 2 -> 16 (not stored)
//   4 blocks:  s = Ws * h + bs                  3x3x3 space conv 16 -> 16
//              a = relu(s)
//              h = h + (Wt * a + bt)            3-tap time conv 16 -> 16
//   block b spaces its taps 2^b cells apart (dilation 1, 2, 4, 8), so the
//   network sees 31 cells in x, y, z and t: as far as the flows reach
//   flow = head(h)                              pointwise 16 -> 4
// The convolutions run on the matrix cores with BF16 weights and BF16-rounded
// inputs, FP32 accumulation (tap after tap, two per instruction).  A value that only feeds convolutions (a, and
// the copies of h, dh and ds that they read) is stored in BF16, rounded once
// as the convolutions would round it; the residual chain h and its gradient
// stay FP32.  A wavefront computes out^T (16 channels x 16 cells) for two
// taps per instruction (16x16x32):
//   A (16 x 32) = weights   lane l: out channel l%16, k = 8*(l/16) .. +7
//   B (32 x 16) = inputs    lane l: cell l%16,        k = 8*(l/16) .. +7
//   D (16 x 16) = out^T     lane l: cell l%16, out channels 4*(l/16) .. +3
// with k = 16*(tap - 2*pair) + input channel.  The order of a sum's taps and
// their pairing decide its roundings, and through them which BF16 neighbour the
// next layer reads: they are part of the network's definition here, so that a
// flow does not change with the kernel that computes it.  The backward data
// pass is the same kernel with mirrored taps and transposed weights; the weight
// gradients have the cells as the reduction dimension.  Training is Adam on
// FP32 master weights.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "flof_internal.h"

namespace flof {

namespace wn {

constexpr int C = 16;       // channels
constexpr int NB = 4;       // residual blocks
constexpr int NS = 27;      // space taps
constexpr int NTT = 3;      // time taps
constexpr int PAIRS_S = 14;  // ceil(27 / 2)
constexpr int PAIRS_T = 2;   // ceil(3 / 2)

// parameter layout (FP32, flat)
constexpr int OFF_WL = 0;                   // [2][16]
constexpr int OFF_BL = OFF_WL + 2 * C;      // [16]
constexpr int OFF_BLK = OFF_BL + C;         // blocks
constexpr int BLK_WS = 0;                   // [27][16][16]  (tap, in, out)
constexpr int BLK_BS = BLK_WS + NS * C * C; // [16]
constexpr int BLK_WT = BLK_BS + C;          // [3][16][16]
constexpr int BLK_BT = BLK_WT + NTT * C * C;// [16]
constexpr int BLK_SIZE = BLK_BT + C;        // 7712
constexpr int OFF_WH = OFF_BLK + NB * BLK_SIZE;  // [16][4]
constexpr int OFF_BH = OFF_WH + C * 4;      // [4]
constexpr int NPARAM = OFF_BH + 4;          // 30964

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned short to_bf16(float f)
{
    return __builtin_bit_cast(unsigned short, (__bf16)f);
}

__device__ __forceinline__ bf16x8 pack8(const float4 &a, const float4 &b)
{
    u16x8 u;
    u[0] = to_bf16(a.x);
    u[1] = to_bf16(a.y);
    u[2] = to_bf16(a.z);
    u[3] = to_bf16(a.w);
    u[4] = to_bf16(b.x);
    u[5] = to_bf16(b.y);
    u[6] = to_bf16(b.z);
    u[7] = to_bf16(b.w);
    return __builtin_bit_cast(bf16x8, u);
}
__device__ __forceinline__ u16x4 pack4(const f32x4 &v)
{
    u16x4 u;
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = to_bf16(v[r]);
    return u;
}

struct Geo {
    int X, Y, Z, T;
    int n;    // cells (< 2^31, checked by the host)
    int dil;  // tap spacing of the convolutions
};

// Where a convolution's input comes from: a BF16 tensor [cell][16], or (block
// 0) the lift of the two level sets, formed where it is needed: 8 bytes per
// cell instead of 32 (BF16) or 64 (FP32 residual).
struct In {
    const unsigned short *b;
    const float *i0, *i1, *P;
};
// channel o of the lift
__device__ __forceinline__ float lift(const float *__restrict__ P, int o, float x0, float x1)
{
    return P[OFF_WL + o] * x0 + P[OFF_WL + C + o] * x1 + P[OFF_BL + o];
}

// ---------------------------------------------------------------------------
// The 3x3x3 space convolution.  Taps are d cells apart, so cells with equal
// (y mod d, z mod d) form planes of their own; a workgroup owns TY = 8 such
// rows of up to 64 x cells of one t step (`XW` wide, d columns of halo on each
// side, zero outside the grid) and marches through the planes of its z class,
// keeping three haloed planes in LDS as BF16 (the two 8-channel halves apart,
// so that the 16 lanes of an operand read 256 contiguous bytes).  Every input
// value is loaded about 1.25 times from memory and read 23 times from LDS;
// the form that gathered the taps from memory read 27 x 64 bytes per cell
// through the vector caches and rounded each value 27 times.
// A wavefront computes rows of a block of 16 x cells, with the weights in
// registers.  An operand is a row's 16 cells under the two taps of a pair.  The
// taps are taken in order, so most pairs' operands serve one output row; in
// each z plane one pair recurs two rows further on (the first two x taps of the
// rows y - 1 and y + 1, in the middle plane the last two) and is kept in
// registers in between: 94 LDS reads and 112 MFMA for eight rows.
// 64^4: 442 us (167 at the rate of memory); one read per MFMA 449, and taps
// paired over (z, x), whose operands serve three output rows each, 409, but
// that order of the sums gives another flow.  What is left is instruction issue,
// and the two barriers per plane with two workgroups per CU to cover them.
struct SpaceGeo {
    int X, Y, Z, T, d;
    int nxt, XW;      // x tiles and their width
    int nry, nrz;     // y and z classes that hold rows: min(d, Y), min(d, Z)
    int nyt, nzs;     // y tiles per y class, z segments per z class
    int zlen;         // planes per z segment
    int pitch;        // XW + 2 d
    int total;        // work items: fewer than the cells
    int first;        // the launch's first item
};
constexpr int SP_W = 64, SP_DMAX = 8;
template <int TY> struct SpLds {
    static constexpr int ROWS = TY + 2;
    static constexpr int HALF = ROWS * (SP_W + 2 * SP_DMAX) + 8;  // 16-byte slots of a half
    static constexpr int LOADS = (2 * ROWS * (SP_W + 2 * SP_DMAX) + 255) / 256;
};

struct SpItem {
    int x0, y0, ry, z0, z1, rz, t;  // first sub row y0 (rows ry + d yy), planes z0 .. z1 - 1
};
template <int TY>
__device__ __forceinline__ bool sp_item(const SpaceGeo &S, int L, SpItem &w)
{
    int r = L;
    const int yt = r % S.nyt;
    r /= S.nyt;
    w.ry = r % S.nry;
    r /= S.nry;
    const int zs = r % S.nzs;
    r /= S.nzs;
    w.rz = r % S.nrz;
    r /= S.nrz;
    const int xt = r % S.nxt;
    w.t = r / S.nxt;
    w.x0 = xt * S.XW;
    w.y0 = yt * TY;
    w.z0 = zs * S.zlen;
    const int zc = (S.Z - w.rz + S.d - 1) / S.d;  // planes of the class
    w.z1 = min(w.z0 + S.zlen, zc);
    return w.ry + S.d * w.y0 < S.Y && w.rz < S.Z && w.z0 < w.z1;
}

enum { SP_FWD = 0, SP_BWD = 1 };
// SP_FWD: out_b = bf16(relu(conv + bias)) (a positive value never rounds to
// zero, so its sign serves as the mask of the backward pass).
// SP_BWD: out_f = res + conv, out_b = bf16(out_f), and the workgroup's column
// sums of out_f (the gradient of the previous block's time bias).
// NR rows of NB blocks of 16 x cells per wavefront: of four blocks one each, of
// three two rows of each, of two four rows of one, of one two rows.
template <bool LIFT, int MODE, int NR, int NB>
__global__ void __launch_bounds__(256, 2)
k_space(const unsigned short *__restrict__ inb, const float *__restrict__ i0,
        const float *__restrict__ i1, const float *__restrict__ P,
        const bf16x8 *__restrict__ wf, const float *__restrict__ bias,
        const float *__restrict__ res, float *__restrict__ out_f,
        unsigned short *__restrict__ out_b, float *__restrict__ colsum, SpaceGeo S)
{
    constexpr int TY = 8;
    typedef SpLds<TY> L_;
    __shared__ bf16x8 lds[3][2][L_::HALF];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = lane >> 4, sub = grp >> 1, half = grp & 1;
    const int per = (int)gridDim.x / FLOF_NXCD;  // the grid is a multiple of 8
    const int L = S.first + ((int)blockIdx.x % FLOF_NXCD) * per + (int)blockIdx.x / FLOF_NXCD;
    f32x4 cs = {0.f, 0.f, 0.f, 0.f};
    SpItem w;
    if (L < S.total && sp_item<TY>(S, L, w)) {  // uniform over the workgroup
        const int d = S.d, pitch = S.pitch, X = S.X;
        const int64_t plane = (int64_t)X * S.Y;
        const int64_t tb = plane * S.Z * w.t;
        bf16x8 wr[PAIRS_S];
#pragma unroll
        for (int p = 0; p < PAIRS_S; ++p) wr[p] = wf[p * 64 + lane];
        // staged elements of this thread: 16-byte half sh of halo cells e; the
        // two halves of a cell by neighbouring lanes, or (the lift, whose
        // weights are then scalars of one half) by wavefronts
        const int sh = LIFT ? __builtin_amdgcn_readfirstlane(wave >> 1) : tid & 1;
        const int e0 = LIFT ? tid & 127 : tid >> 1;
        int off[L_::LOADS];
#pragma unroll
        for (int m = 0; m < L_::LOADS; ++m) {
            const int e = e0 + 128 * m;
            const int row = e / pitch, x = w.x0 - d + (e - row * pitch);
            const int y = w.ry + d * (w.y0 - 1 + row);
            off[m] = row < L_::ROWS && x >= 0 && x < X && y >= 0 && y < S.Y ? x + X * y : -1;
        }
        const int nst = L_::ROWS * pitch;
        bf16x8 st[L_::LOADS];
        bool st_ok = false;
        // loads are unconditional (cell 0 of the t step where the element lies
        // outside the grid, replaced by zero when it is written to LDS)
        auto fetch = [&](int zz) {
            const int z = w.rz + d * zz;
            const bool zok = zz >= 0 && z < S.Z;
            const int64_t zb = tb + (zok ? plane * z : 0);
            if (LIFT) {
                float x0[L_::LOADS], x1[L_::LOADS];
#pragma unroll
                for (int m = 0; m < L_::LOADS; ++m) {
                    const int o = max(off[m], 0);
                    x0[m] = i0[zb + o] * 0.25f;
                    x1[m] = i1[zb + o] * 0.25f;
                }
#pragma unroll
                for (int m = 0; m < L_::LOADS; ++m) {
                    float v[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = lift(P, 8 * sh + q, x0[m], x1[m]);
                    st[m] = pack8(make_float4(v[0], v[1], v[2], v[3]),
                                  make_float4(v[4], v[5], v[6], v[7]));
                }
            } else {
#pragma unroll
                for (int m = 0; m < L_::LOADS; ++m)
                    st[m] = __builtin_bit_cast(
                        bf16x8,
                        *(const u32x4 *)(inb + (zb + max(off[m], 0)) * C + 8 * sh));
            }
            st_ok = zok;
        };
        auto stash = [&](int zz) {
            bf16x8 *s = lds[(zz + 3) % 3][sh];
#pragma unroll
            for (int m = 0; m < L_::LOADS; ++m) {
                const int e = e0 + 128 * m;
                if (e < nst) s[e] = st_ok && off[m] >= 0 ? st[m] : bf16x8{};
            }
        };
        // the rows of this wavefront: LDS slot of the lane's cell one row before
        // the first, and the cells' offsets in a grid plane (-1: not an output)
        constexpr int GROUPS = TY / NR;  // of rows per x block
        const int xt = (NB > 1 ? 0 : wave / GROUPS * 16) + (lane & 15), r0 = wave % GROUPS * NR;
        const int base = r0 * pitch + xt + d + half * L_::HALF;
        int cell[NB][NR];
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int x = xt + 16 * k, y = w.ry + d * (w.y0 + r0 + j);
                cell[k][j] = x < S.XW && w.x0 + x < X && y < S.Y ? w.x0 + x + X * y : -1;
            }
        fetch(w.z0 - 1);
        stash(w.z0 - 1);
        fetch(w.z0);
        stash(w.z0);
        fetch(w.z0 + 1);
        const bf16x8 *flat = &lds[0][0][0];
        for (int zz = w.z0; zz < w.z1; ++zz) {
            __syncthreads();  // every wave is done with plane zz - 2's slot
            stash(zz + 1);
            __syncthreads();
            if (zz + 1 < w.z1) fetch(zz + 2);
            f32x4 acc[NB][NR];
#pragma unroll
            for (int k = 0; k < NB; ++k)
#pragma unroll
                for (int j = 0; j < NR; ++j) acc[k][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int s0 = ((zz + 2) % 3) * 2 * L_::HALF, s1 = (zz % 3) * 2 * L_::HALF,
                      s2 = ((zz + 1) % 3) * 2 * L_::HALF;
            bf16x8 keep[NB][NR + 2];  // operands of the pair that recurs, by row
#pragma unroll
            for (int p = 0; p < PAIRS_S; ++p) {
                auto tap = [&](int m) {
                    return (m / 9 == 0 ? s0 : m / 9 == 1 ? s1 : s2) + m / 3 % 3 * pitch +
                           (m % 3 - 1) * d;
                };
                const int o = base + (sub && 2 * p + 1 < NS ? tap(2 * p + 1) : tap(2 * p));
                const bool first = p == 0 || p == 5 || p == 9;    // taps 0 1, 10 11, 18 19
                const bool again = p == 3 || p == 8 || p == 12;   // taps 6 7, 16 17, 24 25
                if (first)
#pragma unroll
                    for (int row = 0; row < NR + 2; ++row)
#pragma unroll
                        for (int k = 0; k < NB; ++k) keep[k][row] = flat[o + row * pitch + 16 * k];
#pragma unroll
                for (int j = 0; j < NR; ++j)
#pragma unroll
                    for (int k = 0; k < NB; ++k) {
                        bf16x8 b = first   ? keep[k][j]
                                   : again ? keep[k][j + 2]
                                           : flat[o + j * pitch + 16 * k];
                        if (2 * p + 1 >= NS && sub) b = bf16x8{};  // the pair's missing tap
                        acc[k][j] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[p], b, acc[k][j], 0, 0, 0);
                    }
            }
            const int64_t zb = tb + plane * (w.rz + d * zz);
#pragma unroll
            for (int j = 0; j < NB * NR; ++j) {
                const int cl = cell[j / NR][j % NR];
                if (cl < 0) continue;
                const int64_t o = (zb + cl) * C + 4 * grp;
                f32x4 v = acc[j / NR][j % NR];
                if (MODE == SP_FWD) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] += bias[4 * grp + r];
                    u16x4 u;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        u[r] = to_bf16(fmaxf(v[r], 0.f));
                        if (v[r] > 0.f && u[r] == 0) u[r] = 1;
                    }
                    *(u16x4 *)(out_b + o) = u;
                } else {
                    const f32x4 rs = *(const f32x4 *)(res + o);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v[r] += rs[r];
                        cs[r] += v[r];
                    }
                    *(f32x4 *)(out_f + o) = v;
                    *(u16x4 *)(out_b + o) = pack4(v);
                }
            }
        }
    }
    if (MODE == SP_BWD) {
        __shared__ float sh[4][C];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            for (int m = 8; m >= 1; m >>= 1) cs[r] += __shfl_xor(cs[r], m, 64);
        if ((lane & 15) == 0)
            for (int r = 0; r < 4; ++r) sh[wave][4 * grp + r] = cs[r];
        __syncthreads();
        if (tid < C)
            colsum[((int64_t)S.first + blockIdx.x) * C + tid] =
                sh[0][tid] + sh[1][tid] + sh[2][tid] + sh[3][tid];
    }
}

// The forward space convolution of grids whose tiles would stay nearly empty:
// with few rows or planes per class of equal (y mod d, z mod d) a tile of k_space
// holds little else than halo (8 x 8 x 8 x 400, d = 8: 8 outputs of 128).  A
// wavefront takes 16 cells in a row and gathers their taps from memory, two per
// MFMA in the same order, all loads under way together.
template <bool LIFT>
__global__ void __launch_bounds__(256)
k_space_gather(const unsigned short *__restrict__ inb, const float *__restrict__ i0,
               const float *__restrict__ i1, const float *__restrict__ P,
               const bf16x8 *__restrict__ wf, const float *__restrict__ bias,
               unsigned short *__restrict__ out_b, Geo g, Coord4 D4)
{
    const int lane = threadIdx.x & 63;
    const int grp = lane >> 4, sub = grp >> 1, half = grp & 1;
    bf16x8 wr[PAIRS_S];
#pragma unroll
    for (int p = 0; p < PAIRS_S; ++p) wr[p] = wf[p * 64 + lane];
    const int waves = gridDim.x * 4;
    const int ntiles = (g.n + 15) >> 4;
    const int plane = g.X * g.Y;
    for (int tile = blockIdx.x * 4 + (threadIdx.x >> 6); tile < ntiles; tile += waves) {
        const int c = tile * 16 + (lane & 15);
        const bool live = c < g.n;
        int x, y, z, t;
        decompose((uint32_t)(live ? c : 0), D4, x, y, z, t);
        bool ok[PAIRS_S];
        int nc[PAIRS_S];
#pragma unroll
        for (int p = 0; p < PAIRS_S; ++p) {
            const int m0 = 2 * p, m1 = 2 * p + 1 < NS ? 2 * p + 1 : 2 * p;
            const int dx = g.dil * (sub ? m1 % 3 - 1 : m0 % 3 - 1);
            const int dy = g.dil * (sub ? m1 / 3 % 3 - 1 : m0 / 3 % 3 - 1);
            const int dz = g.dil * (sub ? m1 / 9 - 1 : m0 / 9 - 1);
            ok[p] = live && !(2 * p + 1 >= NS && sub) && x + dx >= 0 && x + dx < g.X &&
                    y + dy >= 0 && y + dy < g.Y && z + dz >= 0 && z + dz < g.Z;
            nc[p] = ok[p] ? c + dx + g.X * dy + plane * dz : 0;
        }
        bf16x8 b[PAIRS_S];
        if (LIFT) {
            float x0[PAIRS_S], x1[PAIRS_S];
#pragma unroll
            for (int p = 0; p < PAIRS_S; ++p) {
                x0[p] = i0[nc[p]] * 0.25f;
                x1[p] = i1[nc[p]] * 0.25f;
            }
#pragma unroll
            for (int p = 0; p < PAIRS_S; ++p) {
                float v[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = lift(P, 8 * half + q, x0[p], x1[p]);
                b[p] = pack8(make_float4(v[0], v[1], v[2], v[3]),
                             make_float4(v[4], v[5], v[6], v[7]));
            }
        } else {
#pragma unroll
            for (int p = 0; p < PAIRS_S; ++p)
                b[p] = __builtin_bit_cast(
                    bf16x8, *(const u32x4 *)(inb + (int64_t)nc[p] * C + 8 * half));
        }
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < PAIRS_S; ++p)
            v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[p], ok[p] ? b[p] : bf16x8{}, v, 0, 0,
                                                        0);
        if (!live) continue;
        u16x4 u;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] += bias[4 * grp + r];
            u[r] = to_bf16(fmaxf(v[r], 0.f));
            if (v[r] > 0.f && u[r] == 0) u[r] = 1;
        }
        *(u16x4 *)(out_b + (int64_t)c * C + 4 * grp) = u;
    }
}

// ---------------------------------------------------------------------------
// The 3-tap time convolution.  A wavefront owns 64 consecutive cells of the 3D
// grid (four tiles of 16) and marches through the t steps of one class mod d,
// the BF16 inputs at t - d, t, t + d in registers and the next one requested a
// step ahead, so every input is read once.  An MFMA takes the taps t - d (lanes
// 0..31) and t (lanes 32..63), a second one t + d alone.  A load brings the two
// 16-byte halves of 32 cells; a swap of the wavefront's halves turns it into
// the operands of two tiles with the cells in both halves, from which each tap
// takes its own.  Residual and stores have the layout of the result, 8 or 16
// bytes per lane of one contiguous stretch.  Bound by memory: forward 32 + 64
// bytes read and 64 + 32 written per cell.  64^4: 0.56 ms, 5.7 TB/s, the head's
// step 0.40 (1.03 ms before, reading each input three times in FP32).
// TM_FWD: v = res + (conv + bias); out_f (optional) = v, out_b (optional) =
// bf16(v); flow (optional) = the head of v: every lane gathers its cell's 16
// channels from the four lanes that hold them and sums one of the outputs,
// channel after channel.
// TM_BWD: v = conv where the mask tensor is positive, else 0; out_b = bf16(v),
// and the workgroup's column sums of v (the space bias gradient).
enum { TM_FWD = 0, TM_BWD = 1 };
struct TimeGeo {
    int64_t n3;
    int T, d;
    int nr;          // t classes that hold steps: min(d, T)
    int nch;         // stretches of 64 cells
    int klen, nseg;  // steps of a class per segment, segments
    int total;       // workgroups of 4 stretches: ceil(nch / 4) * nr * nseg
};
template <bool LIFT, int MODE, bool HEAD>
__global__ void __launch_bounds__(256)
k_time(const unsigned short *__restrict__ in, const bf16x8 *__restrict__ wf,
       const float *__restrict__ bias, const float *__restrict__ res, In lin,
       const unsigned short *__restrict__ mask, float *__restrict__ out_f,
       unsigned short *__restrict__ out_b, const float *__restrict__ P,
       float4 *__restrict__ flow, float *__restrict__ colsum, TimeGeo G)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = lane >> 4;
    const int nwg = (G.nch + 3) / 4;
    int r_ = blockIdx.x;
    const int ch = (r_ % nwg) * 4 + wave;
    r_ /= nwg;
    const int rt = r_ % G.nr, seg = r_ / G.nr;
    f32x4 cs = {0.f, 0.f, 0.f, 0.f};
    const int kc = (G.T - rt + G.d - 1) / G.d;  // steps of the class
    const int k0 = seg * G.klen, k1 = min(k0 + G.klen, kc);
    if (ch < G.nch && rt < G.T && k0 < k1) {
        const bf16x8 w0 = wf[lane], w1 = wf[64 + lane];
        f32x4 bs = {0.f, 0.f, 0.f, 0.f};
        if (MODE == TM_FWD)
#pragma unroll
            for (int r = 0; r < 4; ++r) bs[r] = bias[4 * grp + r];
        float wh[C], bh = 0.f;
        if (HEAD) {
#pragma unroll
            for (int i = 0; i < C; ++i) wh[i] = P[OFF_WH + i * 4 + grp];
            bh = P[OFF_BH + grp];
        }
        float l0[4], l1[4], lb[4];
        if (LIFT) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                l0[r] = P[OFF_WL + 4 * grp + r];
                l1[r] = P[OFF_WL + C + 4 * grp + r];
                lb[r] = P[OFF_BL + 4 * grp + r];
            }
        }
        int64_t c3[4];
        bool ok[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c3[j] = (int64_t)ch * 64 + 16 * j + (lane & 15);
            ok[j] = c3[j] < G.n3;
            if (!ok[j]) c3[j] = 0;
        }
        // the 16-byte half (lane >> 4) & 1 of cells 32 q + 16 (lane >> 5) + lane % 16
        const bool upper = lane >= 32;
        int64_t cl[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            cl[q] = (int64_t)ch * 64 + 32 * q + (upper ? 16 : 0) + (lane & 15);
            if (cl[q] >= G.n3) cl[q] = 0;
        }
        auto load = [&](u32x4 (&a)[2], int k) {
            const int t = rt + G.d * k;
            const bool in_t = k >= 0 && t < G.T;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                a[q] = u32x4{0, 0, 0, 0};
                if (in_t) a[q] = *(const u32x4 *)(in + (cl[q] + G.n3 * t) * C + 8 * (grp & 1));
            }
        };
        // the four tiles of a step, each in both halves of the wavefront
        auto spread = [&](const u32x4 (&a)[2], u32x4 (&b)[4]) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto v = __builtin_amdgcn_permlane32_swap(a[q][r], a[q][r], false, false);
                    b[2 * q][r] = v[0];
                    b[2 * q + 1][r] = v[1];
                }
        };
        u32x4 raw[2], am[4], ac[4], ap[4];
        load(raw, k0 - 1);
        spread(raw, am);
        load(raw, k0);
        spread(raw, ac);
        load(raw, k0 + 1);
        for (int k = k0; k < k1; ++k) {
            const int t = rt + G.d * k;
            spread(raw, ap);
            if (k + 1 < k1) load(raw, k + 2);
            f32x4 rs[4];
            s16x4 mk[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t c = c3[j] + G.n3 * t;
                if (MODE == TM_BWD) {
                    mk[j] = *(const s16x4 *)(mask + c * C + 4 * grp);
                } else if (LIFT) {
                    const float x0 = lin.i0[c] * 0.25f, x1 = lin.i1[c] * 0.25f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) rs[j][r] = l0[r] * x0 + l1[r] * x1 + lb[r];
                } else {
                    rs[j] = *(const f32x4 *)(res + c * C + 4 * grp);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f32x4 v = {0.f, 0.f, 0.f, 0.f};
                u32x4 b0, b1;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    b0[r] = upper ? ac[j][r] : am[j][r];
                    b1[r] = upper ? 0u : ap[j][r];
                }
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, __builtin_bit_cast(bf16x8, b0), v,
                                                            0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, __builtin_bit_cast(bf16x8, b1), v,
                                                            0, 0, 0);
                const int64_t c = c3[j] + G.n3 * t;
                if (MODE == TM_FWD) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = (v[r] + bs[r]) + rs[j][r];
                    if (ok[j]) {
                        if (out_f) *(f32x4 *)(out_f + c * C + 4 * grp) = v;
                        if (out_b) *(u16x4 *)(out_b + c * C + 4 * grp) = pack4(v);
                    }
                    if (HEAD) {
                        // hv[4 g + r]: channel r of lane group g
                        float hv[C];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const unsigned u = __float_as_uint(v[r]);
                            const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
#pragma unroll
                            for (int g = 0; g < 2; ++g) {
                                const auto e = __builtin_amdgcn_permlane16_swap(h[g], h[g], false,
                                                                                false);
                                hv[8 * g + r] = __uint_as_float(e[0]);
                                hv[8 * g + 4 + r] = __uint_as_float(e[1]);
                            }
                        }
                        float f = bh;
#pragma unroll
                        for (int i = 0; i < C; ++i) f += wh[i] * hv[i];
                        if (ok[j]) ((float *)flow)[4 * c + grp] = f;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (!(mk[j][r] > 0)) v[r] = 0.f;  // bf16 sign and zero as int16
                        if (ok[j]) cs[r] += v[r];
                    }
                    if (ok[j]) *(u16x4 *)(out_b + c * C + 4 * grp) = pack4(v);
                }
                am[j] = ac[j];
                ac[j] = ap[j];
            }
        }
    }
    if (MODE == TM_BWD) {
        __shared__ float sh[4][C];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            for (int m = 8; m >= 1; m >>= 1) cs[r] += __shfl_xor(cs[r], m, 64);
        if ((lane & 15) == 0)
            for (int r = 0; r < 4; ++r) sh[wave][4 * grp + r] = cs[r];
        __syncthreads();
        if (tid < C)
            colsum[(int64_t)blockIdx.x * C + tid] =
                sh[0][tid] + sh[1][tid] + sh[2][tid] + sh[3][tid];
    }
}

// A fragments of a conv (16x16x32, two taps) from W[tap][in][out] (FP32).
// transpose: the backward data pass, whose "out" channel is W's input channel
// and whose taps are mirrored.
__global__ void k_pack_frag(const float *__restrict__ W, bf16x8 *__restrict__ wf, int ntaps,
                            int npairs, int transpose)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= npairs * 64) return;
    const int p = idx >> 6, lane = idx & 63;
    const int o = lane & 15, grp = lane >> 4;
    const int m = 2 * p + (grp >> 1);
    float v[8];
    for (int q = 0; q < 8; ++q) {
        const int ii = 8 * (grp & 1) + q;
        float w = 0.f;
        if (m < ntaps)
            w = transpose ? W[((ntaps - 1 - m) * C + o) * C + ii] : W[(m * C + ii) * C + o];
        v[q] = w;
    }
    wf[idx] = pack8(make_float4(v[0], v[1], v[2], v[3]), make_float4(v[4], v[5], v[6], v[7]));
}

// ---------------------------------------------------------------------------
// Weight gradients, dW[tap][i][o] = sum_c in[c + off(tap)][i] dout[c][o] with
// the cells as the reduction dimension of MFMA 16x16x16: an operand is 4
// consecutive x cells of one channel, so the tiles are staged channel by
// channel in LDS.
// Space: tiles, classes and march of k_space with TY = 4 rows; the 27
// accumulators of a wavefront (108 registers) live through all of its work
// items, and the lanes' quads of x cells give three taps at once where their
// ranges overlap (d = 1: 12 bytes, d = 2: 16 bytes instead of 24).  At
// 50x46x44x40: 0.19-0.24 ms per convolution, where gathering every operand
// value from memory in three launches of 9 taps took 2.95 ms.
template <int TY> struct WgLds {
    static constexpr int ROWS = TY + 2;
    static constexpr int PITCH = SP_W + 2 * SP_DMAX + 4;
    // bytes of one channel; odd multiples of 32 spread the 16 channels over the banks
    static constexpr int CH = (3 * ROWS * PITCH * 2 + 31) / 64 * 64 + 32;
    static constexpr int DCH = (TY * SP_W * 2) / 64 * 64 + 32;
};
template <bool LIFT, int D>
__global__ void __launch_bounds__(256)
k_wgrad_space(const unsigned short *__restrict__ inb, const float *__restrict__ i0,
              const float *__restrict__ i1, const float *__restrict__ P,
              const unsigned short *__restrict__ dout, float *__restrict__ part, SpaceGeo S)
{
    constexpr int TY = 4;
    typedef WgLds<TY> L_;
    constexpr int LOADS = (2 * L_::ROWS * (SP_W + 2 * SP_DMAX) + 255) / 256;
    constexpr int DLOADS = (2 * TY * SP_W + 255) / 256;
    static_assert(3 * L_::ROWS * L_::PITCH * 2 <= L_::CH && TY * SP_W * 2 <= L_::DCH, "");
    __shared__ __attribute__((aligned(16))) char li[C * L_::CH];
    __shared__ __attribute__((aligned(16))) char ld[C * L_::DCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = lane >> 4, ch = lane & 15;
    const int d = D > 0 ? D : S.d, X = S.X;
    // a multiple of 4 columns: the quads' reads stay 8-byte aligned
    const int pitch = (S.XW + 3) / 4 * 4 + max(4, 2 * d);
    const int64_t plane = (int64_t)X * S.Y;
    f32x4 acc[NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int qx = (S.XW + 3) / 4;  // quads per row
    const int nq = TY * qx;
    for (int L = blockIdx.x; L < S.total; L += gridDim.x) {
        SpItem w;
        if (!sp_item<TY>(S, L, w)) continue;  // uniform over the workgroup
        const int64_t tb = plane * S.Z * w.t;
        const int sh = LIFT ? __builtin_amdgcn_readfirstlane(wave >> 1) : tid & 1;
        const int e0 = LIFT ? tid & 127 : tid >> 1;
        int off[LOADS], dof[DLOADS];
#pragma unroll
        for (int m = 0; m < LOADS; ++m) {
            const int e = e0 + 128 * m;
            const int row = e / pitch, x = w.x0 - d + (e - row * pitch);
            const int y = w.ry + d * (w.y0 - 1 + row);
            off[m] = row < L_::ROWS && x >= 0 && x < X && y >= 0 && y < S.Y ? x + X * y : -1;
        }
#pragma unroll
        for (int m = 0; m < DLOADS; ++m) {
            const int e = (tid + 256 * m) >> 1;
            const int row = e / (4 * qx), x = e - row * (4 * qx);
            const int y = w.ry + d * (w.y0 + row);
            dof[m] = row < TY && x < S.XW && w.x0 + x < X && y < S.Y ? w.x0 + x + X * y : -1;
        }
        const int nst = L_::ROWS * pitch, ndst = 2 * TY * 4 * qx;
        u16x8 st[LOADS], sd[DLOADS];
        bool st_ok = false;
        auto fetch = [&](int zz) {
            const int z = w.rz + d * zz;
            st_ok = zz >= 0 && z < S.Z;
            const int64_t zb = tb + (st_ok ? plane * z : 0);
#pragma unroll
            for (int m = 0; m < LOADS; ++m) {
                const int64_t c = zb + max(off[m], 0);
                if (LIFT) {
                    const float x0 = i0[c] * 0.25f, x1 = i1[c] * 0.25f;
#pragma unroll
                    for (int q = 0; q < 8; ++q) st[m][q] = to_bf16(lift(P, 8 * sh + q, x0, x1));
                } else {
                    st[m] = *(const u16x8 *)(inb + c * C + 8 * sh);
                }
            }
        };
        auto fetch_d = [&](int zz) {
            const int64_t zb = tb + plane * (w.rz + d * zz);
#pragma unroll
            for (int m = 0; m < DLOADS; ++m)
                sd[m] = *(const u16x8 *)(dout + (zb + max(dof[m], 0)) * C + 8 * (tid & 1));
        };
        auto stash = [&](int zz) {
            const int so = ((zz + 3) % 3) * L_::ROWS * pitch;
#pragma unroll
            for (int m = 0; m < LOADS; ++m) {
                const int e = e0 + 128 * m;
                if (!(st_ok && off[m] >= 0)) st[m] = u16x8{};
                if (e < nst) {
                    char *p = li + 8 * sh * L_::CH + (so + e) * 2;
#pragma unroll
                    for (int q = 0; q < 8; ++q) *(unsigned short *)(p + q * L_::CH) = st[m][q];
                }
            }
        };
        auto stash_d = [&]() {
#pragma unroll
            for (int m = 0; m < DLOADS; ++m) {
                const int e = tid + 256 * m;
                if (dof[m] < 0) sd[m] = u16x8{};
                if (e < ndst) {
                    char *p = ld + 8 * (tid & 1) * L_::DCH + (e >> 1) * 2;
#pragma unroll
                    for (int q = 0; q < 8; ++q) *(unsigned short *)(p + q * L_::DCH) = sd[m][q];
                }
            }
        };
        __syncthreads();  // the previous item's last step has been read
        fetch(w.z0 - 1);
        stash(w.z0 - 1);
        fetch(w.z0);
        stash(w.z0);
        fetch(w.z0 + 1);
        fetch_d(w.z0);
        for (int zz = w.z0; zz < w.z1; ++zz) {
            if (zz > w.z0) __syncthreads();  // every wave is done with the last step
            stash(zz + 1);
            stash_d();
            __syncthreads();
            if (zz + 1 < w.z1) {
                fetch(zz + 2);
                fetch_d(zz + 1);
            }
            for (int q0 = wave * 4; q0 < nq; q0 += 16) {
                const int q = q0 + grp;
                const bool ok = q < nq;
                const int row = ok ? q / qx : 0, x = ok ? 4 * (q - row * qx) : 0;
                s16x4 b = *(const s16x4 *)(ld + ch * L_::DCH + (row * 4 * qx + x) * 2);
                if (!ok) b = s16x4{0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 9; ++r) {
                    const int slot = (zz + r / 3 + 2) % 3;
                    const char *p = li + ch * L_::CH +
                                    ((slot * L_::ROWS + row + r % 3) * pitch + x) * 2;
                    s16x4 a0, a1, a2;
                    if (D == 1) {
                        const uint2 u = *(const uint2 *)p;
                        const unsigned v = *(const unsigned *)(p + 8);
                        a0 = __builtin_bit_cast(s16x4, u);
                        a1 = __builtin_bit_cast(
                            s16x4, make_uint2(__builtin_amdgcn_alignbit(u.y, u.x, 16),
                                              __builtin_amdgcn_alignbit(v, u.y, 16)));
                        a2 = __builtin_bit_cast(s16x4, make_uint2(u.y, v));
                    } else if (D == 2) {
                        const uint2 u = *(const uint2 *)p, v = *(const uint2 *)(p + 8);
                        a0 = __builtin_bit_cast(s16x4, u);
                        a1 = __builtin_bit_cast(s16x4, make_uint2(u.y, v.x));
                        a2 = __builtin_bit_cast(s16x4, v);
                    } else {
                        a0 = *(const s16x4 *)p;
                        a1 = *(const s16x4 *)(p + 2 * d);
                        a2 = *(const s16x4 *)(p + 4 * d);
                    }
                    acc[3 * r] =
                        __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0, b, acc[3 * r], 0, 0, 0);
                    acc[3 * r + 1] =
                        __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, b, acc[3 * r + 1], 0, 0, 0);
                    acc[3 * r + 2] =
                        __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a2, b, acc[3 * r + 2], 0, 0, 0);
                }
            }
        }
    }
    // D[i][o]: lane holds i = 4 grp + r, o = lane % 16
    float *dst = part + ((int64_t)blockIdx.x * 4 + wave) * NS * C * C;
#pragma unroll
    for (int m = 0; m < NS; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(m * C + 4 * grp + r) * C + ch] = acc[m][r];
}

// Time: a wavefront takes the stretches and t classes of k_time in turn; a
// step's input (t + d) and dout (t) go channel by channel through its own
// LDS rows (read back by the same wavefront), the inputs at t - d and t stay
// in registers.
constexpr int WT_ROW = 64 * 2 + 16;  // bytes of one channel's 64 cells
__global__ void __launch_bounds__(256)
k_wgrad_time(const unsigned short *__restrict__ in, const unsigned short *__restrict__ dout,
             float *__restrict__ part, TimeGeo G)
{
    __shared__ __attribute__((aligned(16))) char lds[4][2][C * WT_ROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = lane >> 4, ch = lane & 15;
    f32x4 acc[NTT];
#pragma unroll
    for (int m = 0; m < NTT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int items = G.nch * G.nr * G.nseg;
    for (int it = blockIdx.x * 4 + wave; it < items; it += gridDim.x * 4) {
        int r_ = it;
        const int chn = r_ % G.nch;
        r_ /= G.nch;
        const int rt = r_ % G.nr, seg = r_ / G.nr;
        const int kc = (G.T - rt + G.d - 1) / G.d;
        const int k0 = seg * G.klen, k1 = min(k0 + G.klen, kc);
        if (rt >= G.T || k0 >= k1) continue;
        // cells of this lane's two 16-byte halves: lane >> 1 and 32 + (lane >> 1)
        const int64_t cb = (int64_t)chn * 64;
        auto load = [&](const unsigned short *src, u16x8 (&v)[2], int k) {
            const int t = rt + G.d * k;
            const bool in_t = k >= 0 && t < G.T;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t c = cb + 32 * j + (lane >> 1);
                v[j] = u16x8{};
                if (in_t && c < G.n3)
                    v[j] = *(const u16x8 *)(src + (c + G.n3 * t) * C + 8 * (lane & 1));
            }
        };
        // through the wavefront's own rows (its lanes run in step; the waits
        // on LDS order the writes and the reads)
        auto turn = [&](const u16x8 (&v)[2], s16x4 (&o)[4], int slot) {
            char *p = lds[wave][slot];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    *(unsigned short *)(p + (8 * (lane & 1) + q) * WT_ROW +
                                        (32 * j + (lane >> 1)) * 2) = v[j][q];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = *(const s16x4 *)(p + ch * WT_ROW + (16 * j + 4 * grp) * 2);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        u16x8 raw[2], rawd[2];
        s16x4 am[4], ac[4], ap[4], b[4];
        load(in, raw, k0 - 1);
        turn(raw, am, 0);
        load(in, raw, k0);
        turn(raw, ac, 0);
        load(in, raw, k0 + 1);
        load(dout, rawd, k0);
        for (int k = k0; k < k1; ++k) {
            turn(raw, ap, 0);
            turn(rawd, b, 1);
            if (k + 1 < k1) {
                load(in, raw, k + 2);
                load(dout, rawd, k + 1);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(am[j], b[j], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ac[j], b[j], acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ap[j], b[j], acc[2], 0, 0, 0);
                am[j] = ac[j];
                ac[j] = ap[j];
            }
        }
    }
    float *dst = part + ((int64_t)blockIdx.x * 4 + wave) * NTT * C * C;
#pragma unroll
    for (int m = 0; m < NTT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(m * C + 4 * grp + r) * C + ch] = acc[m][r];
}

// rows x cols partial sums -> one row (FP64 sum over rows): a workgroup takes
// 16 columns with 16 row lanes each, so that few columns of many rows do not
// run as one serial chain (one thread per column took 355 us per call on
// average in a training step, this takes 12)
__global__ void __launch_bounds__(256)
k_sum_rows(const float *__restrict__ part, int rows, int cols, float *__restrict__ dst)
{
    __shared__ double sh[16][17];
    const int cl = threadIdx.x & 15, rl = threadIdx.x >> 4;
    const int col = blockIdx.x * 16 + cl;
    double s = 0.;
    if (col < cols) {
#pragma unroll 8
        for (int r = rl; r < rows; r += 16) s += (double)part[(int64_t)r * cols + col];
    }
    sh[rl][cl] = s;
    __syncthreads();
    if (rl == 0 && col < cols) {
        double t = 0.;
        for (int q = 0; q < 16; ++q) t += sh[q][cl];
        dst[col] = (float)t;
    }
}

// loss = mean((flow - tgt)^2) over 4n values: dy = 2 (flow - tgt) / (4n);
// per-block partial sums of the squared error (FP64)
__global__ void __launch_bounds__(256)
k_loss(const float4 *__restrict__ flow, const float4 *__restrict__ tgt,
       float4 *__restrict__ dy, int n, double *__restrict__ part)
{
    const float sc = 2.f / (4.f * (float)n);
    double s = 0.;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        const float4 f = flow[c], t = tgt[c];
        const float4 e = make_float4(f.x - t.x, f.y - t.y, f.z - t.z, f.w - t.w);
        s += (double)e.x * e.x + (double)e.y * e.y + (double)e.z * e.z + (double)e.w * e.w;
        dy[c] = make_float4(sc * e.x, sc * e.y, sc * e.z, sc * e.w);
    }
    __shared__ double sh[256];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// sums of the workgroup's v[0 .. N-1], one row of N partials (lane sums by
// shuffles, then the four wavefronts through LDS)
template <int N> __device__ __forceinline__ void block_cols(float (&v)[N], float *dst)
{
    __shared__ float sh[4][N];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        for (int m = 32; m >= 1; m >>= 1) v[q] += __shfl_xor(v[q], m, 64);
        if (lane == 0) sh[wave][q] = v[q];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < N; q += blockDim.x)
        dst[q] = sh[0][q] + sh[1][q] + sh[2][q] + sh[3][q];
}

// head backward: dh[c][i] = sum_d Wh[i][d] dy[c][d], FP32 and BF16; per-block
// partials of dWh[i][d] = sum_c h[c][i] dy[c][d] (64), dbh[d] = sum_c dy[c][d]
// (4) and sum_c dh[c][i] (16, the last block's time bias)
constexpr int HEAD_COLS = C * 4 + 4 + C;
__global__ void __launch_bounds__(256)
k_head_bwd(const float *__restrict__ h, const float4 *__restrict__ dy,
           const float *__restrict__ P, float *__restrict__ dh,
           unsigned short *__restrict__ dhb, int n, float *__restrict__ part)
{
    float g[HEAD_COLS];
#pragma unroll
    for (int q = 0; q < HEAD_COLS; ++q) g[q] = 0.f;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        const float4 e = dy[c];
        const float ev[4] = {e.x, e.y, e.z, e.w};
        const f32x4 *hc = (const f32x4 *)(h + (int64_t)c * C);
        f32x4 *dc = (f32x4 *)(dh + (int64_t)c * C);
        u16x4 *db = (u16x4 *)(dhb + (int64_t)c * C);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 hv = hc[q];
            f32x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 4 * q + r;
                float a = 0.f;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    a += P[OFF_WH + i * 4 + d] * ev[d];
                    g[i * 4 + d] += hv[r] * ev[d];
                }
                o[r] = a;
                g[C * 4 + 4 + i] += a;
            }
            dc[q] = o;
            db[q] = pack4(o);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) g[C * 4 + d] += ev[d];
    }
    block_cols<HEAD_COLS>(g, part + (int64_t)blockIdx.x * HEAD_COLS);
}

// lift backward: per-block partials of dWl[k][o] = sum_c x_k[c] dh0[c][o]
// (32) and dbl[o] = sum_c dh0[c][o] (16)
__global__ void __launch_bounds__(256)
k_lift_bwd(const float *__restrict__ i0, const float *__restrict__ i1,
           const float *__restrict__ dh, int n, float *__restrict__ part)
{
    float g[3 * C];
#pragma unroll
    for (int q = 0; q < 3 * C; ++q) g[q] = 0.f;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        const float x0 = i0[c] * 0.25f, x1 = i1[c] * 0.25f;
        const f32x4 *d = (const f32x4 *)(dh + (int64_t)c * C);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 v = d[q];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 4 * q + r;
                g[o] += x0 * v[r];
                g[C + o] += x1 * v[r];
                g[2 * C + o] += v[r];
            }
        }
    }
    block_cols<3 * C>(g, part + (int64_t)blockIdx.x * 3 * C);
}

__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

}  // namespace wn
}  // namespace flof

using namespace flof;
using namespace flof::wn;

struct flof_warmnet {
    flof_ctx *ctx = nullptr;
    float *P = nullptr;      // FP32 master parameters
    float *G = nullptr;      // gradients
    float *M = nullptr, *V = nullptr;  // Adam moments
    bf16x8 *frag = nullptr;  // packed A fragments, forward and backward
    int step = 0;
    bool frag_ok = false;
};

namespace {

// 16-byte fragment slots per block: space fwd, space bwd, time fwd, time bwd
constexpr int FRAG_S = PAIRS_S * 64, FRAG_T = PAIRS_T * 64;
constexpr int FRAG_BLK = 2 * FRAG_S + 2 * FRAG_T;

void pack_all(flof_warmnet *net)
{
    flof_ctx *ctx = net->ctx;
    for (int b = 0; b < NB; ++b) {
        const float *blk = net->P + OFF_BLK + b * BLK_SIZE;
        bf16x8 *f = net->frag + (size_t)b * FRAG_BLK;
        hipLaunchKernelGGL(k_pack_frag, dim3((FRAG_S + 255) / 256), dim3(256), 0, ctx->stream,
                           blk + BLK_WS, f, NS, PAIRS_S, 0);
        hipLaunchKernelGGL(k_pack_frag, dim3((FRAG_S + 255) / 256), dim3(256), 0, ctx->stream,
                           blk + BLK_WS, f + FRAG_S, NS, PAIRS_S, 1);
        hipLaunchKernelGGL(k_pack_frag, dim3(1), dim3(256), 0, ctx->stream, blk + BLK_WT,
                           f + 2 * FRAG_S, NTT, PAIRS_T, 0);
        hipLaunchKernelGGL(k_pack_frag, dim3(1), dim3(256), 0, ctx->stream, blk + BLK_WT,
                           f + 2 * FRAG_S + FRAG_T, NTT, PAIRS_T, 1);
    }
    check_launch("k_pack_frag");
    net->frag_ok = true;
}

Geo geo_of(const flof_grid4d *g)
{
    FLOF_REQUIRE(g->n() < (1ll << 31) / C, FLOF_ERR_DIM, "warm-start net: grid too large");
    return Geo{g->X, g->Y, g->Z, g->T, (int)g->n(), 1};
}

// tiles of a space conv with ty rows per workgroup; z segments of at least 4
// planes, as many as give the chip about `want` workgroups
SpaceGeo space_geo(const Geo &g, int ty, int want)
{
    SpaceGeo S;
    S.X = g.X;
    S.Y = g.Y;
    S.Z = g.Z;
    S.T = g.T;
    S.d = g.dil;
    S.nxt = (g.X + SP_W - 1) / SP_W;
    S.XW = (g.X + S.nxt - 1) / S.nxt;
    S.nry = std::min(g.dil, g.Y);
    S.nrz = std::min(g.dil, g.Z);
    S.nyt = ((g.Y + g.dil - 1) / g.dil + ty - 1) / ty;
    const int zc = (g.Z + g.dil - 1) / g.dil;
    const int64_t cols = (int64_t)g.T * S.nxt * S.nyt * S.nry * S.nrz;
    const int most = std::max(1, zc / 4);
    S.nzs = (int)std::max<int64_t>(1, std::min<int64_t>(most, (want + cols - 1) / cols));
    S.zlen = (zc + S.nzs - 1) / S.nzs;
    S.nzs = (zc + S.zlen - 1) / S.zlen;
    S.pitch = S.XW + 2 * g.dil;
    // nyt nry <= Y and nzs nrz <= Z
    S.total = (int)(cols * S.nzs);
    S.first = 0;
    return S;
}
int space_blocks(const SpaceGeo &S)
{
    return (S.total + FLOF_NXCD - 1) / FLOF_NXCD * FLOF_NXCD;
}
// stretches and t classes of a time conv; segments of at least 4 steps, as
// many as give the chip about 8192 wavefronts
TimeGeo time_geo(const Geo &g)
{
    TimeGeo G;
    G.n3 = (int64_t)g.X * g.Y * g.Z;
    G.T = g.T;
    G.d = g.dil;
    G.nr = std::min(g.dil, g.T);
    G.nch = (int)((G.n3 + 63) / 64);
    const int kc = (g.T + g.dil - 1) / g.dil;
    const int64_t cols = (int64_t)G.nch * G.nr;
    G.nseg = (int)std::max<int64_t>(
        1, std::min<int64_t>(std::max(1, kc / 4), (8192 + cols - 1) / cols));
    G.klen = (kc + G.nseg - 1) / G.nseg;
    G.nseg = (kc + G.klen - 1) / G.klen;
    G.total = (G.nch + 3) / 4 * G.nr * G.nseg;
    return G;
}

size_t bf_bytes(const Geo &g) { return (size_t)g.n * C * 2; }
size_t f_bytes(const Geo &g) { return (size_t)g.n * C * 4; }
unsigned short *u16p(const Tmp &t) { return t.as<unsigned short>(); }

template <bool LIFT, int MODE>
void launch_space(flof_ctx *ctx, const In &in, const bf16x8 *wf, const float *bias,
                  const float *res, float *out_f, unsigned short *out_b, float *colsum,
                  const SpaceGeo &S)
{
    // the workgroup's eight rows of x blocks over its four wavefronts
    auto k = S.XW <= 16   ? k_space<LIFT, MODE, 2, 1>
             : S.XW <= 32 ? k_space<LIFT, MODE, 4, 1>
             : S.XW <= 48 ? k_space<LIFT, MODE, 2, 3>
                          : k_space<LIFT, MODE, 8, 1>;
    // A launch takes fewer than 2^32 threads, more would run as what is left
    // of the count modulo 2^32: 2^23 workgroups each (thin grids with a long t).
    constexpr int MOST = 1 << 23;
    SpaceGeo part = S;
    for (int at = 0; at < S.total; at += MOST) {
        part.first = at;
        part.total = std::min(S.total, at + MOST);
        const int nb = (part.total - at + FLOF_NXCD - 1) / FLOF_NXCD * FLOF_NXCD;
        hipLaunchKernelGGL(k, dim3(nb), dim3(256), 0, ctx->stream, in.b, in.i0, in.i1, in.P, wf,
                           bias, res, out_f, out_b, colsum, part);
    }
    check_launch("k_space");
}

// a = relu(space conv of hb (block 0: of the lift) + bias), BF16
void space_fwd(flof_ctx *ctx, const In &in, bool first, const bf16x8 *wf, const float *bias,
               unsigned short *out, const Geo &g)
{
    const SpaceGeo S = space_geo(g, 8, 2048);
    // A plane of a tile stands for 128 outputs per x block of 16.  Counting the
    // two planes of halo, tiles that are to fill fewer than 32 of them each take
    // longer than the gathering form.  The network's flow, tiles only / by this
    // rule, us: 8 x 8 x 8 x 400 411 / 142, 3 x 3 x 3 x 3000 662 / 95, 16^3 x 64
    // 169 / 133, 33 x 17 x 9 x 40 178 / 140, 24^4 175 / 164; full tiles are 2.5
    // times as fast as gathers (32^4 299 / 465 if all were gathered).
    const int64_t planes = (int64_t)S.total * (S.zlen + 2) * ((S.XW + 15) / 16);
    if (32 * planes > (int64_t)g.n) {
        const int64_t tiles = ((int64_t)g.n + 15) / 16;
        const Coord4 D4{make_fastdiv((uint32_t)g.X), make_fastdiv((uint32_t)g.Y),
                        make_fastdiv((uint32_t)g.Z)};
        hipLaunchKernelGGL(first ? k_space_gather<true> : k_space_gather<false>,
                           dim3(grid_blocks(ctx, tiles * 64, 256, 4)), dim3(256), 0, ctx->stream,
                           in.b, in.i0, in.i1, in.P, wf, bias, out, g, D4);
        check_launch("k_space_gather");
        return;
    }
    if (first)
        launch_space<true, SP_FWD>(ctx, in, wf, bias, nullptr, nullptr, out, nullptr, S);
    else
        launch_space<false, SP_FWD>(ctx, in, wf, bias, nullptr, nullptr, out, nullptr, S);
}

// h' = res + (time conv of a + bias): FP32 and / or BF16, or its head
void time_fwd(flof_ctx *ctx, const unsigned short *a, const bf16x8 *wf, const float *bias,
              const float *res, const In &lin, float *hf, unsigned short *hb, const float *P,
              float4 *flow, const Geo &g)
{
    const TimeGeo G = time_geo(g);
    // (the lift feeds block 0, the head follows block 3)
    auto k = flow  ? k_time<false, TM_FWD, true>
             : res ? k_time<false, TM_FWD, false>
                   : k_time<true, TM_FWD, false>;
    hipLaunchKernelGGL(k, dim3(G.total), dim3(256), 0, ctx->stream, a, wf, bias,
                       res, lin, nullptr, hf, hb, P, flow, nullptr, G);
    check_launch("k_time");
}

// what a backward pass needs of a forward one: the BF16 conv inputs and the
// last block's FP32 output
struct Acts {
    Tmp hb[NB], ab[NB], h;
};

// the network's flow; with A its activations are kept
void forward(flof_ctx *ctx, flof_warmnet *net, const float *i0, const float *i1, const Geo &g0,
             Acts *A, float4 *flow)
{
    if (!net->frag_ok) pack_all(net);
    Tmp hf[2], hbt[2], abt;
    if (!A) abt = Tmp(ctx, bf_bytes(g0));
    const In lin{nullptr, i0, i1, net->P};
    for (int b = 0; b < NB; ++b) {
        const bool last = b == NB - 1;
        const float *blk = net->P + OFF_BLK + b * BLK_SIZE;
        const bf16x8 *f = net->frag + (size_t)b * FRAG_BLK;
        Geo g = g0;
        g.dil = 1 << b;
        In in = lin;
        if (b) in.b = u16p(A ? A->hb[b] : hbt[b & 1]);
        if (A) A->ab[b] = Tmp(ctx, bf_bytes(g));
        unsigned short *a = u16p(A ? A->ab[b] : abt);
        space_fwd(ctx, in, b == 0, f, blk + BLK_BS, a, g);
        Tmp &hn = last && A ? A->h : hf[(b + 1) & 1];
        if (!hn.p && (!last || A)) hn = Tmp(ctx, f_bytes(g));
        Tmp *hbn = last ? nullptr : A ? &A->hb[b + 1] : &hbt[(b + 1) & 1];
        if (hbn && !hbn->p) *hbn = Tmp(ctx, bf_bytes(g));
        time_fwd(ctx, a, f + 2 * FRAG_S, blk + BLK_BT, b ? hf[b & 1].as<float>() : nullptr, lin,
                 last && !A ? nullptr : hn.as<float>(), hbn ? u16p(*hbn) : nullptr, net->P,
                 last ? flow : nullptr, g);
    }
}

}  // namespace

void flof::warmnet_infer(flof_ctx *ctx, flof_warmnet *net, const float *i0, const float *i1,
                         const Dims4 &D, float4 *flow)
{
    FLOF_REQUIRE(net && net->ctx == ctx, FLOF_ERR_ARG,
                 "warm-start net: the network belongs to another context");
    const int64_t n = D.st * D.T;
    FLOF_REQUIRE(n >= 1 && n < (1ll << 30), FLOF_ERR_DIM,
                 "warm-start net: 1 to 2^30 cells");
    const Geo g0{D.X, D.Y, D.Z, D.T, (int)n, 1};
    forward(ctx, net, i0, i1, g0, nullptr, flow);
}


namespace {

// sum of `rows` rows of partials into dst, in FP64
void sum_rows(flof_ctx *ctx, const float *part, int rows, int cols, float *dst)
{
    hipLaunchKernelGGL(k_sum_rows, dim3((cols + 15) / 16), dim3(256), 0, ctx->stream, part, rows,
                       cols, dst);
    check_launch("k_sum_rows");
}

// two workgroups of the weight-gradient kernels per CU, as LDS admits
int wgrad_blocks(flof_ctx *ctx, int items)
{
    return std::max(1, std::min(items, ctx->num_cu * 2));
}

void wgrad_space(flof_ctx *ctx, const In &in, bool first, const unsigned short *dout,
                 const Geo &g, float *dW)
{
    const SpaceGeo S = space_geo(g, 4, 2048);
    const int nbk = wgrad_blocks(ctx, S.total);
    Tmp part(ctx, (size_t)nbk * 4 * NS * C * C * 4);
    auto k = first ? k_wgrad_space<true, 1>
                   : g.dil == 1 ? k_wgrad_space<false, 1>
                                : g.dil == 2 ? k_wgrad_space<false, 2> : k_wgrad_space<false, 0>;
    hipLaunchKernelGGL(k, dim3(nbk), dim3(256), 0, ctx->stream, in.b, in.i0, in.i1, in.P, dout,
                       part.as<float>(), S);
    check_launch("k_wgrad_space");
    sum_rows(ctx, part.as<float>(), nbk * 4, NS * C * C, dW);
}

void wgrad_time(flof_ctx *ctx, const unsigned short *in, const unsigned short *dout, const Geo &g,
                float *dW)
{
    const TimeGeo G = time_geo(g);
    const int nbk = wgrad_blocks(ctx, (G.nch * G.nr * G.nseg + 3) / 4);
    Tmp part(ctx, (size_t)nbk * 4 * NTT * C * C * 4);
    hipLaunchKernelGGL(k_wgrad_time, dim3(nbk), dim3(256), 0, ctx->stream, in, dout,
                       part.as<float>(), G);
    check_launch("k_wgrad_time");
    sum_rows(ctx, part.as<float>(), nbk * 4, NTT * C * C, dW);
}

// forward + loss + backward; gradients into net->G, returns the loss
double loss_grad(flof_warmnet *net, const float *i0, const float *i1, const float4 *tgt,
                 const Geo &g0)
{
    flof_ctx *ctx = net->ctx;
    const int n = g0.n;
    Acts A;
    Tmp flow(ctx, (size_t)n * 16), dy(ctx, (size_t)n * 16);
    forward(ctx, net, i0, i1, g0, &A, flow.as<float4>());
    const int lb = grid_blocks(ctx, n, 256, 4);
    Tmp lp(ctx, (size_t)lb * 8);
    hipLaunchKernelGGL(k_loss, dim3(lb), dim3(256), 0, ctx->stream,
                       (const float4 *)flow.as<float4>(), tgt, dy.as<float4>(), n,
                       lp.as<double>());
    check_launch("k_loss");
    Tmp dh(ctx, f_bytes(g0)), dh2(ctx, f_bytes(g0)), dhb(ctx, bf_bytes(g0)),
        dhb2(ctx, bf_bytes(g0)), dsb(ctx, bf_bytes(g0));
    const int hb = grid_blocks(ctx, n, 256, 4);
    Tmp hp(ctx, (size_t)hb * HEAD_COLS * 4), hs(ctx, HEAD_COLS * 4);
    hipLaunchKernelGGL(k_head_bwd, dim3(hb), dim3(256), 0, ctx->stream,
                       (const float *)A.h.as<float>(), (const float4 *)dy.as<float4>(),
                       (const float *)net->P, dh.as<float>(), u16p(dhb), n, hp.as<float>());
    check_launch("k_head_bwd");
    sum_rows(ctx, hp.as<float>(), hb, HEAD_COLS, hs.as<float>());
    FLOF_HIP(hipMemcpyAsync(net->G + OFF_WH, hs.p, (C * 4 + 4) * 4, hipMemcpyDeviceToDevice,
                            ctx->stream));
    FLOF_HIP(hipMemcpyAsync(net->G + OFF_BLK + (NB - 1) * BLK_SIZE + BLK_BT,
                            hs.as<float>() + C * 4 + 4, C * 4, hipMemcpyDeviceToDevice,
                            ctx->stream));
    const In lin{nullptr, i0, i1, net->P};
    for (int b = NB - 1; b >= 0; --b) {
        Geo g = g0;
        g.dil = 1 << b;
        float *gb = net->G + OFF_BLK + b * BLK_SIZE;
        const bf16x8 *f = net->frag + (size_t)b * FRAG_BLK;
        // h_{b+1} = h_b + Wt * a + bt
        wgrad_time(ctx, u16p(A.ab[b]), u16p(dhb), g, gb + BLK_WT);
        // ds = (Wt^T * dh) where a > 0; its sum is the space bias' gradient
        {
            const TimeGeo G = time_geo(g);
            Tmp cp(ctx, (size_t)G.total * C * 4);
            hipLaunchKernelGGL((k_time<false, TM_BWD, false>), dim3(G.total), dim3(256), 0, ctx->stream,
                               u16p(dhb), f + 2 * FRAG_S + FRAG_T, nullptr,
                               nullptr, lin, u16p(A.ab[b]), nullptr, u16p(dsb), nullptr, nullptr,
                               cp.as<float>(), G);
            check_launch("k_time (backward)");
            sum_rows(ctx, cp.as<float>(), G.total, C, gb + BLK_BS);
        }
        In in = lin;
        in.b = b ? u16p(A.hb[b]) : nullptr;
        wgrad_space(ctx, in, b == 0, u16p(dsb), g, gb + BLK_WS);
        // dh_b = dh_{b+1} + Ws^T * ds; its sum is block b - 1's time bias' gradient
        {
            const SpaceGeo S = space_geo(g, 8, 2048);
            const int nbk = space_blocks(S);
            Tmp cp(ctx, (size_t)nbk * C * 4);
            In ds = lin;
            ds.b = u16p(dsb);
            launch_space<false, SP_BWD>(ctx, ds, f + FRAG_S, nullptr, dh.as<float>(),
                                        dh2.as<float>(), u16p(dhb2), cp.as<float>(), S);
            if (b) sum_rows(ctx, cp.as<float>(), nbk, C, gb - BLK_SIZE + BLK_BT);
        }
        std::swap(dh, dh2);
        std::swap(dhb, dhb2);
    }
    const int fb = grid_blocks(ctx, n, 256, 4);
    Tmp fp(ctx, (size_t)fb * 3 * C * 4);
    hipLaunchKernelGGL(k_lift_bwd, dim3(fb), dim3(256), 0, ctx->stream, i0, i1,
                       (const float *)dh.as<float>(), n, fp.as<float>());
    check_launch("k_lift_bwd");
    sum_rows(ctx, fp.as<float>(), fb, 3 * C, net->G + OFF_WL);
    std::vector<double> h(lb);
    FLOF_HIP(hipMemcpyAsync(h.data(), lp.p, (size_t)lb * 8, hipMemcpyDeviceToHost,
                            ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    double s = 0.;
    for (double v : h) s += v;
    return s / (4.0 * (double)n);
}

void need_pair(const flof_grid4d *i0, const flof_grid4d *i1, const flof_grid4d *v,
               const char *what)
{
    FLOF_REQUIRE(i0 && i1 && v, FLOF_ERR_ARG, std::string(what) + ": null grid");
    FLOF_REQUIRE(i0->elem == FLOF_REAL && i1->elem == FLOF_REAL && v->elem == FLOF_VEC4 &&
                     i0->dtype == FLOF_F32 && i1->dtype == FLOF_F32 && v->dtype == FLOF_F32,
                 FLOF_ERR_TYPE, std::string(what) + ": REAL inputs and a VEC4 flow (FP32)");
    for (const flof_grid4d *q : {i1, v})
        FLOF_REQUIRE(q->X == i0->X && q->Y == i0->Y && q->Z == i0->Z && q->T == i0->T,
                     FLOF_ERR_DIM, std::string(what) + ": grid sizes differ");
}

}  // namespace

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

int flof_warmnet_num_params(void) { return NPARAM; }

int flof_warmnet_create(flof_ctx *ctx, uint64_t seed, flof_warmnet **out)
{
    API_TRY
    FLOF_REQUIRE(ctx && out, FLOF_ERR_ARG, "warmnet_create: null argument");
    *out = nullptr;
    flof_warmnet *net = new flof_warmnet();
    net->ctx = ctx;
    try {
        const size_t pb = (size_t)NPARAM * 4;
        FLOF_HIP(hipMalloc((void **)&net->P, pb));
        FLOF_HIP(hipMalloc((void **)&net->G, pb));
        FLOF_HIP(hipMalloc((void **)&net->M, pb));
        FLOF_HIP(hipMalloc((void **)&net->V, pb));
        FLOF_HIP(hipMalloc((void **)&net->frag, (size_t)NB * FRAG_BLK * sizeof(bf16x8)));
        FLOF_HIP(hipMemsetAsync(net->G, 0, pb, ctx->stream));
        FLOF_HIP(hipMemsetAsync(net->M, 0, pb, ctx->stream));
        FLOF_HIP(hipMemsetAsync(net->V, 0, pb, ctx->stream));
        // He-style initial weights from a seeded splitmix64 stream; the
        // residual branches and the head start small
        std::vector<float> w(NPARAM, 0.f);
        uint64_t s = seed;
        auto uni = [&]() {
            s += 0x9E3779B97F4A7C15ull;
            uint64_t z = s;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            return (double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
        };
        for (int q = 0; q < 2 * C; ++q) w[OFF_WL + q] = (float)(uni() * 1.0);
        for (int b = 0; b < NB; ++b) {
            float *blk = w.data() + OFF_BLK + b * BLK_SIZE;
            const double as = std::sqrt(3.0 / (NS * C)), at = 0.1 * std::sqrt(3.0 / (NTT * C));
            for (int q = 0; q < NS * C * C; ++q) blk[BLK_WS + q] = (float)(uni() * as);
            for (int q = 0; q < NTT * C * C; ++q) blk[BLK_WT + q] = (float)(uni() * at);
        }
        for (int q = 0; q < C * 4; ++q) w[OFF_WH + q] = (float)(uni() * 0.05);
        FLOF_HIP(hipMemcpyAsync(net->P, w.data(), pb, hipMemcpyHostToDevice, ctx->stream));
        FLOF_HIP(hipStreamSynchronize(ctx->stream));
    } catch (...) {
        flof_warmnet_destroy(net);
        throw;
    }
    *out = net;
    API_CATCH(ctx)
}

int flof_warmnet_destroy(flof_warmnet *net)
{
    if (!net) return FLOF_ERR_ARG;
    if (net->ctx) (void)hipStreamSynchronize(net->ctx->stream);
    for (void *p : {(void *)net->P, (void *)net->G, (void *)net->M, (void *)net->V,
                    (void *)net->frag})
        if (p) (void)hipFree(p);
    delete net;
    return FLOF_OK;
}

int flof_warmnet_get_params(flof_warmnet *net, float *host, int n)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net && host && n == NPARAM, FLOF_ERR_ARG, "warmnet_get_params: bad argument");
    FLOF_HIP(hipMemcpyAsync(host, net->P, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

int flof_warmnet_set_params(flof_warmnet *net, const float *host, int n)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net && host && n == NPARAM, FLOF_ERR_ARG, "warmnet_set_params: bad argument");
    FLOF_HIP(hipMemcpyAsync(net->P, host, (size_t)n * 4, hipMemcpyHostToDevice, ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    net->frag_ok = false;
    API_CATCH(ctx)
}

int flof_warmnet_get_grads(flof_warmnet *net, float *host, int n)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net && host && n == NPARAM, FLOF_ERR_ARG, "warmnet_get_grads: bad argument");
    FLOF_HIP(hipMemcpyAsync(host, net->G, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

int flof_warmnet_forward(flof_warmnet *net, flof_grid4d *i0, flof_grid4d *i1,
                         flof_grid4d *flow)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net, FLOF_ERR_ARG, "warmnet_forward: null net");
    need_pair(i0, i1, flow, "warmnet_forward");
    const Geo g = geo_of(i0);
    forward(ctx, net, (const float *)i0->data, (const float *)i1->data, g, nullptr,
            (float4 *)flow->data);
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

int flof_warmnet_loss_grad(flof_warmnet *net, flof_grid4d *i0, flof_grid4d *i1,
                           flof_grid4d *target, double *loss)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net, FLOF_ERR_ARG, "warmnet_loss_grad: null net");
    need_pair(i0, i1, target, "warmnet_loss_grad");
    const double l = loss_grad(net, (const float *)i0->data, (const float *)i1->data,
                               (const float4 *)target->data, geo_of(i0));
    if (loss) *loss = l;
    API_CATCH(ctx)
}

int flof_warmnet_adam(flof_warmnet *net, float lr, float beta1, float beta2, float eps)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net && lr > 0.f && beta1 >= 0.f && beta1 < 1.f && beta2 >= 0.f && beta2 < 1.f,
                 FLOF_ERR_ARG, "warmnet_adam: bad argument");
    net->step += 1;
    const float c1 = (float)(1.0 - std::pow((double)beta1, net->step));
    const float c2 = (float)(1.0 - std::pow((double)beta2, net->step));
    hipLaunchKernelGGL(k_adam, dim3((NPARAM + 255) / 256), dim3(256), 0, ctx->stream, net->P,
                       (const float *)net->G, net->M, net->V, NPARAM, lr, beta1, beta2, eps,
                       c1, c2);
    check_launch("k_adam");
    net->frag_ok = false;
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

int flof_warmnet_warm_start(flof_warmnet *net, flof_grid4d *i0, flof_grid4d *i1, int netX,
                            flof_grid4d *warm)
{
    flof_ctx *ctx = net ? net->ctx : nullptr;
    API_TRY
    FLOF_REQUIRE(net && netX >= 2, FLOF_ERR_ARG, "warmnet_warm_start: bad argument");
    need_pair(i0, i1, warm, "warmnet_warm_start");
    // the pyramid of the multiscale solve down to X <= netX
    std::vector<Dims4> dims{dims_of(i0)};
    while (dims.back().X > netX) {
        const Dims4 &D = dims.back();
        Dims4 Ds{D.X / 2, D.Y / 2, D.Z / 2, D.T / 2, 0, 0};
        Ds.sz = (int64_t)Ds.X * Ds.Y;
        Ds.st = Ds.sz * Ds.Z;
        FLOF_REQUIRE(Ds.X >= 2 && Ds.Y >= 2 && Ds.Z >= 2 && Ds.T >= 2, FLOF_ERR_DIM,
                     "warmnet_warm_start: pyramid level too small");
        dims.push_back(Ds);
    }
    const size_t L = dims.size();
    std::vector<Tmp> a(L), b(L), v(L);
    const float *ca = (const float *)i0->data, *cb = (const float *)i1->data;
    for (size_t l = 1; l < L; ++l) {
        const int64_t n = dims[l].st * dims[l].T;
        a[l] = Tmp(ctx, (size_t)n * 4);
        b[l] = Tmp(ctx, (size_t)n * 4);
        launch_pyramid(ctx, a[l].p, dims[l], ca, dims[l - 1], false, 1.f);
        launch_pyramid(ctx, b[l].p, dims[l], cb, dims[l - 1], false, 1.f);
        ca = a[l].as<float>();
        cb = b[l].as<float>();
    }
    const Dims4 &Dn = dims[L - 1];
    FLOF_REQUIRE(Dn.st * Dn.T < (1ll << 31) / C, FLOF_ERR_DIM, "warmnet: grid too large");
    const Geo g{Dn.X, Dn.Y, Dn.Z, Dn.T, (int)(Dn.st * Dn.T), 1};
    float4 *out = L == 1 ? (float4 *)warm->data : nullptr;
    if (L > 1) {
        v[L - 1] = Tmp(ctx, (size_t)g.n * 16);
        out = v[L - 1].as<float4>();
    }
    forward(ctx, net, ca, cb, g, nullptr, out);
    for (size_t l = L - 1; l >= 1; --l) {
        void *dst = l == 1 ? warm->data : nullptr;
        if (l > 1) {
            v[l - 1] = Tmp(ctx, (size_t)dims[l - 1].st * dims[l - 1].T * 16);
            dst = v[l - 1].p;
        }
        launch_pyramid(ctx, dst, dims[l - 1], v[l].p, dims[l], true, 2.f);
    }
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    API_CATCH(ctx)
}

}  // extern "C"
