// flof_resident.hip -- the PCG of small and middle pyramid levels as one
// resident launch (optflow4d.cpp:274-329, the same operations in the same
// order as the launch-per-kernel form in flof_solve.hip).
//
// Up to about 1.3 million interior cells the vectors of a level fit the chip's
// registers and LDS.  A workgroup of 512 threads per CU owns a box of cells,
// full rows in x, and keeps x, r and q (then z) of its cells in registers and
// p, with the faces of the neighbouring boxes, in LDS.  The launch-per-kernel
// form runs five dependent launches per iteration, each of which moves the
// vectors through memory.  Per iteration (cap 440 less cap 40, one level):
// 16^4 16.8 -> 7.9 us, 24^4 29.4 -> 13.5, 32^4 50.7 -> 18.8, 32^3 x 48 65.4 ->
// 26.3.  At 16^4 the two meetings are most of it; at 32^4 the arithmetic of 7
// cells per thread, about 1.3 us each, and the faces, 3 us.
//
// Per iteration the workgroups meet twice, for p.q and for z.r and max r.
// A meeting is an all-gather: every workgroup stores its partial sums as 64-bit
// words of 56 bits of payload and the meeting's number modulo 256 (each word
// is its own proof of arrival, whatever order they arrive in; a slot is never
// more than one meeting old), and reads those of all others until each carries
// that number; all then reduce the same values in the same order, so no second
// exchange distributes the result.  One costs 1.25 us and about 8.5 ns per
// workgroup; slots of 32 bytes are read faster than separate arrays.  The
// stores and loads have agent scope: they go past the L2 caches of the eight
// XCDs to the memory they share, and no fence (an L2 write-back and
// invalidation; it takes 16 us more per iteration at 32^4) is needed.  The
// faces travel the same way: before the second meeting every workgroup stores
// z of its outer cells, waits until the stores have been acknowledged, and only
// then stores its partial sums; after the meeting it reads z next to its box
// and forms the neighbours' new p = z + beta p from the copy of their old p it
// holds, the same operation on the same operands as theirs.
//
// No kernel here may spill: the vectors fill the registers, and a spill of the
// outer loop's values right after a divergent loop was seen to be emitted
// before the execution mask is restored, so that r of some lanes was lost
// (wrong sums from the second iteration on).  Hence fresh(), the loads
// without conditions and the vectors declared inside the loop; a kernel that
// was given scratch memory all the same is not launched.
//
// The launch is cooperative, so all workgroups are resident together, and the
// runtime runs such launches of several streams one after another: worker
// streams gain by it too (16 solves of 16^4 on one, 2, 4 and 16 streams 51, 43,
// 43, 44 ms and launched 123, 66, 48, 162; of 24^4 128, 118, 117, 118 and 308,
// 178, 144, 322).  A
// workgroup that still waits after two seconds (flof_ctx_set_resident_wait)
// gives up and says so in a word that all poll, so every wavefront ends
// whatever happens; the caller then sets the level up again and uses the other
// form.

#include <algorithm>
#include <cstring>

#include "flof_cg.h"

namespace flof {

namespace {

constexpr int RT = 512;           // threads per workgroup
constexpr int R_CPT = 11;         // cells per thread at most
constexpr int R_CELLS = 9800;     // LDS slots of p: own rows, y and z faces, padding
constexpr int R_ROWS = 400;       // own rows
constexpr int R_HROWS = 400;      // face rows in LDS
constexpr int R_SLAB = 1024;      // cells of a box's t slice: its faces in t stay in registers
constexpr int R_SLOT = 32;        // bytes of a workgroup's slot (three 64-bit words)

// sc1, the agent-scope cache policy of gfx950: past the L2 of the XCD
typedef unsigned u32v4 __attribute__((ext_vector_type(4)));
typedef unsigned u32v2 __attribute__((ext_vector_type(2)));
constexpr int AUX_SC1 = 16;

struct ResItem {
    ResLevel L;
    int py, pz, pt;
    int first, nwg;               // workgroups of this level
    FastDiv fnx;                  // X - 2
    char *slots;                  // [2][nwg][R_SLOT]
};

// a face cell: 16 bytes, one access, so that neighbouring lanes write whole lines
__device__ __forceinline__ void st_agent4(__amdgpu_buffer_rsrc_t b, int c, const float4 &v)
{
    const u32v4 u = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z),
                     __float_as_uint(v.w)};
    __builtin_amdgcn_raw_buffer_store_b128(u, b, (int)((unsigned)c << 4), 0, AUX_SC1);
}
// A cell past every exchange buffer (they hold fewer than 2^28 - 1): its load
// touches no memory and gives 0.  Loads under a condition would leave the
// compiler with values that it carries, and spills, through the iterations.
constexpr int NO_CELL = (1 << 28) - 1;
__device__ __forceinline__ float4 ld_agent4(__amdgpu_buffer_rsrc_t b, int c)
{
    const u32v4 u =
        __builtin_amdgcn_raw_buffer_load_b128(b, (int)((unsigned)c << 4), 0, AUX_SC1);
    return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z),
                       __uint_as_float(u.w));
}

// every earlier store of this wavefront has been acknowledged
__device__ __forceinline__ void stores_done()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    asm volatile("" ::: "memory");
}

// Keeps the compiler from carrying the addresses it derives from v (four 64-bit
// ones per cell) through the iterations in registers that the vectors need.
__device__ __forceinline__ void fresh(int &v) { asm volatile("" : "+v"(v)); }
// element c of an array whose byte offsets fit 32 bits (uniform base): global
// accesses with a 32-bit offset, where the pointers out of ResItem would be
// generic ones with a 64-bit address in registers each
typedef float f32v4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) char *GlobalBytes;
__device__ __forceinline__ float4 at(const float4 *a, int c)
{
    const f32v4 v = *(__attribute__((address_space(1))) f32v4 *)((GlobalBytes)a +
                                                                 ((unsigned)c << 4));
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void put(float4 *a, int c, const float4 &v)
{
    *(__attribute__((address_space(1))) f32v4 *)((GlobalBytes)a + ((unsigned)c << 4)) =
        f32v4{v.x, v.y, v.z, v.w};
}

struct Part {
    DD s;
    float m;
};
// v merged with the lanes that a DPP control pairs it with (rows not in
// `rows` keep v): register moves, where a shuffle goes through LDS and takes
// several times as long; six dependent steps per sum are on the critical path
// of every meeting
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ void dpp_merge(Part &v)
{
    auto mov = [](unsigned u) {
        return (unsigned)__builtin_amdgcn_update_dpp((int)u, (int)u, CTRL, ROWS, 0xf, false);
    };
    auto movd = [&](double x) {
        const unsigned long long u = (unsigned long long)__double_as_longlong(x);
        return __longlong_as_double((long long)((unsigned long long)mov((unsigned)u) |
                                                (unsigned long long)mov((unsigned)(u >> 32))
                                                    << 32));
    };
    const DD o{movd(v.s.hi), movd(v.s.lo)};
    v.m = fmaxf(v.m, __uint_as_float(mov(__float_as_uint(v.m))));
    if (ROWS == 0xf) {
        dd_merge(v.s, o);
    } else {
        DD t = v.s;
        dd_merge(t, o);
        if ((ROWS >> ((threadIdx.x & 63) >> 4)) & 1) v.s = t;
    }
}
// over 8 neighbouring lanes (each gets the result)
__device__ __forceinline__ void part8(Part &v)
{
    dpp_merge<0xB1>(v);   // quad_perm 1 0 3 2
    dpp_merge<0x4E>(v);   // quad_perm 2 3 0 1
    dpp_merge<0x141>(v);  // row_half_mirror
}
// over the wavefront: lane 63 gets the result
__device__ __forceinline__ Part wave_part(DD s, float m)
{
    Part v{s, m};
    part8(v);
    dpp_merge<0x140>(v);       // row_mirror
    dpp_merge<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    dpp_merge<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

// where a box ends: n cells in `parts` runs whose lengths differ by at most one
__host__ __device__ inline int part_at(int n, int parts, int i)
{
    return (int)((long long)n * i / parts);
}

// XG: x stays in memory (the thread's own cells) instead of registers
template <int CPT, bool XG>
__global__ void __launch_bounds__(RT)
k_cg_resident(const ResItem *__restrict__ items, int nitems, unsigned *abort_word,
              unsigned long long wait_ticks)
{
    __shared__ float4 lp[R_CELLS];
    __shared__ short4 nbr[R_ROWS];   // LDS distance to the rows y-1, y+1, z-1, z+1
    __shared__ int hrow[R_HROWS];    // first cell of a face row, -1: outer layer (p = 0)
    __shared__ double sh_hi[RT / 64], sh_lo[RT / 64];
    __shared__ float sh_m[RT / 64];
    __shared__ double g_hi[4], g_lo[4];
    __shared__ float g_m[4];
    __shared__ int g_fail;
    constexpr int HTM = CPT < 4 ? CPT : 4;  // cells per thread in the first two t slices

    int it_ = 0;
    while (it_ + 1 < nitems && (int)blockIdx.x >= items[it_ + 1].first) ++it_;
    const ResItem &I = items[it_];
    const Dims4 D = I.L.D;
    const int rank = (int)blockIdx.x - I.first, nwg = I.nwg;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int X = D.X, sz = (int)D.sz, stt = (int)D.st;
    const int nx = X - 2;
    const int iy = rank % I.py, iz = (rank / I.py) % I.pz, itb = rank / (I.py * I.pz);
    const int y0 = 1 + part_at(D.Y - 2, I.py, iy), y1 = 1 + part_at(D.Y - 2, I.py, iy + 1);
    const int z0 = 1 + part_at(D.Z - 2, I.pz, iz), z1 = 1 + part_at(D.Z - 2, I.pz, iz + 1);
    const int t0 = 1 + part_at(D.T - 2, I.pt, itb), t1 = 1 + part_at(D.T - 2, I.pt, itb + 1);
    const int by = y1 - y0, bz = z1 - z0, bt = t1 - t0;
    const int S = nx * by * bz, N = S * bt;
    const FastDiv fnx = I.fnx;
    const int px = nx + 1;                 // a zero column between rows
    const int rows = by * bz * bt;
    const int fy = bt * bz, fz = bt * by;  // rows of a y and of a z face
    const int hrows = 2 * (fy + fz);
    const int SP = by * bz * px;           // LDS distance of a t step
    const float4 *__restrict__ G = I.L.g;
    const float4 *__restrict__ PR = I.L.prec;
    float4 *const xg = I.L.x;
    const float offd = I.L.offd, diag = I.L.diag;
    const int use_offd = I.L.use_offd;
    // exchange of z, cells as in the grid (fewer than 2^28, checked by the host)
    const __amdgpu_buffer_rsrc_t ex = __builtin_amdgcn_make_buffer_rsrc(
        I.L.z, 0, (int)(unsigned)((uint64_t)D.st * D.T * 16), 0x00020000);
    CgState *st = I.L.st;
    const __amdgpu_buffer_rsrc_t slots = __builtin_amdgcn_make_buffer_rsrc(
        I.slots, 0, 2 * nwg * R_SLOT, 0x00020000);
    const int slotA = 0, slotB = nwg * R_SLOT;

    // --- tables, p and the faces -------------------------------------------
    for (int e = tid; e < R_CELLS; e += RT) lp[e] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int r = tid; r < rows; r += RT) {
        const int y = r % by, z = (r / by) % bz, t = r / (by * bz);
        const int ym = y > 0 ? r - 1 : rows + t * bz + z;
        const int yp = y < by - 1 ? r + 1 : rows + fy + t * bz + z;
        const int zm = z > 0 ? r - by : rows + 2 * fy + t * by + y;
        const int zp = z < bz - 1 ? r + by : rows + 2 * fy + fz + t * by + y;
        nbr[r] = make_short4((short)((ym - r) * px), (short)((yp - r) * px),
                             (short)((zm - r) * px), (short)((zp - r) * px));
    }
    for (int h = tid; h < hrows; h += RT) {
        int y, z, t;
        if (h < 2 * fy) {
            const int q = h % fy;
            z = z0 + q % bz;
            t = t0 + q / bz;
            y = h < fy ? y0 - 1 : y1;
        } else {
            const int q = (h - 2 * fy) % fz;
            y = y0 + q % by;
            t = t0 + q / by;
            z = h < 2 * fy + fz ? z0 - 1 : z1;
        }
        const bool outer = y < 1 || y >= D.Y - 1 || z < 1 || z >= D.Z - 1;
        hrow[h] = outer ? -1 : 1 + X * y + sz * z + stt * t;
    }
    if (tid == 0) g_fail = 0;
    __syncthreads();
    // the thread's cells e = tid + 512 m: x fastest, then y, z and t, with the
    // last t slice taken second, so that a thread's cells next to a face in t
    // are its first ones
    int gc[CPT];       // cell in the grid
    int la[CPT];       // LDS slot, own row << 16, face flag << 30
    float4 x[XG ? 1 : CPT], r[CPT];
    float4 th[HTM];    // p of the neighbour beyond the face in t
    bool th_in[HTM];   // it is an interior cell
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
        const int e = tid + RT * m;
        const bool live = e < N;
        const int ee = live ? e : 0;
        const int xx = ee % nx, q1 = ee / nx;
        const int y = q1 % by, q2 = q1 / by;
        const int z = q2 % bz, tq = q2 / bz;
        const int t = tq == 0 ? 0 : tq == 1 ? bt - 1 : tq - 1;
        const int row = (t * bz + z) * by + y;
        const bool face = y == 0 || y == by - 1 || z == 0 || z == bz - 1 || t == 0 || t == bt - 1;
        la[m] = (1 + row * px + xx) | row << 16 | (face ? 1 << 30 : 0);
        gc[m] = 1 + xx + X * (y0 + y) + sz * (z0 + z) + stt * (t0 + t);
        r[m] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!XG) x[XG ? 0 : m] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (live) {
            if (!XG) x[XG ? 0 : m] = at(xg, gc[m]);
            r[m] = at(I.L.r, gc[m]);
            lp[la[m] & 0xffff] = at(I.L.p, gc[m]);
        }
        if (m < HTM) {
            th[m < HTM ? m : 0] = make_float4(0.f, 0.f, 0.f, 0.f);
            const bool first = e < S, last = e >= S && e < 2 * S;
            const bool in = live && ((first && t0 > 1) || (last && t1 < D.T - 1));
            th_in[m < HTM ? m : 0] = in;
            if (in) th[m < HTM ? m : 0] = at(I.L.p, gc[m] + (first ? -stt : stt));
        }
    }
    const int nh = hrows * nx;
    for (int h = tid; h < nh; h += RT) {
        const int hr = h / nx, xx = h - hr * nx;
        const int g0 = hrow[hr];
        if (g0 >= 0) lp[1 + (rows + hr) * px + xx] = at(I.L.p, g0 + xx);
    }
    double sigma = st->sigma;
    const double acc_thr = st->acc, resIni = st->resIni;
    const int maxIter = st->maxIter;
    int iters = st->iters;
    double resRel = 0.;
    int status = 1, zero = 0;
    unsigned epoch = 0;
    __syncthreads();

    // partial sums of the workgroup -> slot (tagged) -> sums of all; false:
    // given up.  Every thread returns the same value.
    auto publish = [&](int slot0, const Part &v) {
        int lane = tid & 63, wv = wave;
        fresh(lane);
        fresh(wv);
        if (lane == 63) {
            sh_hi[wv] = v.s.hi;
            sh_lo[wv] = v.s.lo;
            sh_m[wv] = v.m;
        }
        __syncthreads();
        if (wave == 0) {
            static_assert(RT / 64 == 8, "part8 sums the workgroup's wavefronts");
            Part w{DD{sh_hi[lane & 7], sh_lo[lane & 7]}, sh_m[lane & 7]};
            part8(w);
            if (nwg == 1) {
                if (lane == 0) {
                    g_hi[0] = w.s.hi;
                    g_lo[0] = w.s.lo;
                    g_m[0] = w.m;
                }
            } else if (lane < 3) {
                // 56 bits of hi, lo and m (160 in all) and the tag per word
                const unsigned long long hi = (unsigned long long)__double_as_longlong(w.s.hi);
                const unsigned long long lo = (unsigned long long)__double_as_longlong(w.s.lo);
                const unsigned long long m = __float_as_uint(w.m);
                const unsigned long long u = lane == 0   ? hi << 8
                                             : lane == 1 ? lo << 8
                                                         : m << 24 | (hi >> 56) << 16 |
                                                               (lo >> 56) << 8;
                const u32v2 v2 = {(unsigned)u | (epoch & 0xff), (unsigned)(u >> 32)};
                __builtin_amdgcn_raw_buffer_store_b64(v2, slots,
                                                      slot0 + rank * R_SLOT + lane * 8, 0,
                                                      AUX_SC1);
            }
        }
    };
    auto gather = [&](int slot0, Part &out) -> bool {
        if (nwg > 1 && wave < 4 && wave * 64 < nwg) {
            DD s{0., 0.};
            float m = -INFINITY;
            bool fail = wait_ticks == 0;
            if (tid < nwg && !fail) {
                int p = slot0 + tid * R_SLOT;
                fresh(p);
                const unsigned tag = epoch & 0xff;
                const unsigned long long begin = wall_clock64();
                unsigned spins = 0;
                for (;;) {
                    asm volatile("" ::: "memory");  // read anew each time
                    const u32v4 a = __builtin_amdgcn_raw_buffer_load_b128(slots, p, 0, AUX_SC1);
                    const u32v2 b =
                        __builtin_amdgcn_raw_buffer_load_b64(slots, p + 16, 0, AUX_SC1);
                    if ((a.x & 0xff) == tag && (a.z & 0xff) == tag && (b.x & 0xff) == tag) {
                        const unsigned long long h = (unsigned long long)a.y << 32 | a.x;
                        const unsigned long long l = (unsigned long long)a.w << 32 | a.z;
                        const unsigned long long t = (unsigned long long)b.y << 32 | b.x;
                        s.hi = __longlong_as_double(
                            (long long)(h >> 8 | (t >> 16 & 0xff) << 56));
                        s.lo = __longlong_as_double((long long)(l >> 8 | (t >> 8 & 0xff) << 56));
                        m = __uint_as_float((unsigned)(t >> 24));
                        break;
                    }
                    if ((++spins & 63) == 0) {
                        // waited long enough, or another one gave up
                        if (__hip_atomic_load(abort_word, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT) != 0 ||
                            wall_clock64() - begin > wait_ticks) {
                            fail = true;
                            break;
                        }
                    }
                }
            }
            if (fail) {
                __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                g_fail = 1;
            }
            const Part v = wave_part(s, m);
            int wv = wave;
            fresh(wv);
            if (lane == 63) {
                g_hi[wv] = v.s.hi;
                g_lo[wv] = v.s.lo;
                g_m[wv] = v.m;
            }
        }
        __syncthreads();
        out.s = DD{g_hi[0], g_lo[0]};
        out.m = g_m[0];
        for (int w = 1; w * 64 < nwg; ++w) {
            dd_merge(out.s, DD{g_hi[w], g_lo[w]});
            out.m = fmaxf(out.m, g_m[w]);
        }
        return g_fail == 0;
    };

    for (;;) {
        ++epoch;
        int tv = tid;
        fresh(tv);
        float4 q[CPT];  // of this iteration only, so that the faces can have its registers
        // --- q = A p and p.q -------------------------------------------------
        // (one cell after another: the registers hold the vectors, not the
        // operands of many cells; only the gradients are loaded a cell ahead)
        DD acc{0., 0.};
        fresh(gc[0]);
        float4 gn = at(G, gc[0]);
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            const int e = tv + RT * m;
            if (RT * m >= N) break;
            const float4 gv = gn;
            fresh(la[m]);
            if (m + 1 < CPT) {
                fresh(gc[m + 1 < CPT ? m + 1 : 0]);
                gn = at(G, gc[m + 1 < CPT ? m + 1 : 0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (e >= N) continue;
            const int l = la[m] & 0xffff;
            const float4 pc = lp[l];
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (use_offd) {
                const short4 o = nbr[(la[m] >> 16) & 0x3fff];
                float4 tm, tp;
                if (m < HTM) {
                    const bool first = e < S, last = e >= S && e < 2 * S;
                    tm = lp[first ? l : l - SP];
                    tp = lp[last ? l : l + SP];
                    const float4 h = th[m < HTM ? m : 0];
                    if (first) tm = h;
                    if (last) tp = h;
                } else {
                    tm = lp[l - SP];
                    tp = lp[l + SP];
                }
                const float4 nb[8] = {tm,        lp[l + o.z], lp[l + o.x], lp[l - 1],
                                      lp[l + 1], lp[l + o.y], lp[l + o.w], tp};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    // (the most cells: half the neighbours in registers at a time)
                    if (CPT > 8 && k == 4) __builtin_amdgcn_sched_barrier(0);
                    v.x = v.x + offd * nb[k].x;
                    v.y = v.y + offd * nb[k].y;
                    v.z = v.z + offd * nb[k].z;
                    v.w = v.w + offd * nb[k].w;
                }
            }
            const float gg[4] = {gv.x, gv.y, gv.z, gv.w};
            const float pv[4] = {pc.x, pc.y, pc.z, pc.w};
            float o4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int d = 0; d < 4; ++d) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float b = gg[d] * gg[k];
                    if (d == k) b = b + diag;
                    o4[d] = o4[d] + b * pv[k];
                }
            }
            q[m] = make_float4(o4[0], o4[1], o4[2], o4[3]);
            dd_add4(acc, pc, q[m]);
            __builtin_amdgcn_sched_barrier(0);
        }
        publish(slotA, wave_part(acc, 0.f));
        Part tot;
        if (!gather(slotA, tot)) return;
        const double alpha = sigma / (tot.s.hi + tot.s.lo), nalpha = -alpha;
        fresh(tv);
        // --- r -= alpha q, z = r / diag (into q), z.r and max r ---------------
        DD sig{0., 0.};
        float mx = 0.f;  // the outer layer's r
        // (short steps: the preconditioner is loaded three cells ahead)
        float4 pn[3];
#pragma unroll
        for (int m = 0; m < 3 && m < CPT; ++m) {
            fresh(gc[m]);
            pn[m] = at(PR, gc[m]);
        }
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            if (RT * m >= N) break;
            const float4 pr = pn[m % 3];
            if (m + 3 < CPT) {
                fresh(gc[m + 3 < CPT ? m + 3 : 0]);
                pn[m % 3] = at(PR, gc[m + 3 < CPT ? m + 3 : 0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (tv + RT * m >= N) continue;
            float4 rc = r[m];
            rc.x = (float)((double)rc.x + nalpha * (double)q[m].x);
            rc.y = (float)((double)rc.y + nalpha * (double)q[m].y);
            rc.z = (float)((double)rc.z + nalpha * (double)q[m].z);
            rc.w = (float)((double)rc.w + nalpha * (double)q[m].w);
            r[m] = rc;
            const float4 z = f4mul(rc, pr);
            q[m] = z;
            mx = fmaxf(mx, fmaxf(fmaxf(rc.x, rc.y), fmaxf(rc.z, rc.w)));
            dd_add4(sig, z, rc);
            __builtin_amdgcn_sched_barrier(0);
        }
        // z of the outer cells, after the loop: a load that waits behind a
        // store waits for its acknowledgement from memory
        if (nwg > 1) {
#pragma unroll
            for (int m = 0; m < CPT; ++m)
                if (tv + RT * m < N && (la[m] >> 30) & 1) st_agent4(ex, gc[m], q[m]);
        }
        const Part pz_ = wave_part(sig, mx);
        stores_done();
        publish(slotB, pz_);
        fresh(tv);
        // x += alpha p while the others' sums arrive
        if (XG) {
            constexpr int XB = 4;
#pragma unroll
            for (int mb = 0; mb < CPT; mb += XB) {
                float4 xv[XB];
#pragma unroll
                for (int k = 0; k < XB; ++k) {
                    const int m = mb + k < CPT ? mb + k : 0;
                    fresh(gc[m]);
                    if (mb + k < CPT && tv + RT * m < N) xv[k] = at(xg, gc[m]);
                }
#pragma unroll
                for (int k = 0; k < XB; ++k) {
                    const int m = mb + k < CPT ? mb + k : 0;
                    fresh(la[m]);
                    if (mb + k < CPT && tv + RT * m < N)
                        put(xg, gc[m], x_plus(xv[k], alpha, lp[la[m] & 0xffff]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int m = 0; m < CPT; ++m) {
                fresh(la[m]);
                if (tv + RT * m < N)
                    x[XG ? 0 : m] = x_plus(x[XG ? 0 : m], alpha, lp[la[m] & 0xffff]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!gather(slotB, tot)) return;
        const double residual = (double)tot.m, sigmaNew = tot.s.hi + tot.s.lo;
        ++iters;
        resRel = (double)(float)(residual / resIni);
        if (residual <= acc_thr) {
            status = 0;
            break;
        }
        if (sigmaNew != sigmaNew || residual != residual) {
            status = 2;
            zero = 1;
            break;
        }
        const double beta = sigmaNew / sigma;
        sigma = sigmaNew;
        if (iters >= maxIter) break;
        // --- p = z + beta p, the faces' copies too ----------------------------
        auto next = [&](const float4 &z, const float4 &p) {
            return make_float4((float)((double)z.x + beta * (double)p.x),
                               (float)((double)z.y + beta * (double)p.y),
                               (float)((double)z.z + beta * (double)p.z),
                               (float)((double)z.w + beta * (double)p.w));
        };
        fresh(tv);
        // own cells first: the registers of z then take the faces under way
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
            fresh(la[m]);
            if (tv + RT * m < N) {
                const int l = la[m] & 0xffff;
                lp[l] = next(q[m], lp[l]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        fresh(tv);
        if (nwg > 1) {
            float4 zt[HTM];
#pragma unroll
            for (int m = 0; m < HTM; ++m) {
                fresh(gc[m]);
                zt[m] = ld_agent4(ex, th_in[m] ? gc[m] + (tv + RT * m < S ? -stt : stt) : NO_CELL);
            }
            // face cells under way per thread: all of them at once, each read
            // takes about 1 us
            constexpr int HB = CPT > 8 ? 9 : CPT > 4 ? 7 : 2 * CPT;
            for (int hb = tv; hb < nh; hb += HB * RT) {
                float4 zh[HB];
                int lh[HB];
#pragma unroll
                for (int k = 0; k < HB; ++k) {
                    const int h = hb + RT * k < nh ? hb + RT * k : 0;
                    const int hr = (int)fdiv((uint32_t)h, fnx), xx = h - hr * nx;
                    const int g0 = hrow[hr];
                    const bool in = hb + RT * k < nh && g0 >= 0;
                    lh[k] = in ? 1 + (rows + hr) * px + xx : -1;
                    zh[k] = ld_agent4(ex, in ? g0 + xx : NO_CELL);
                }
#pragma unroll
                for (int k = 0; k < HB; ++k)
                    if (lh[k] >= 0) lp[lh[k]] = next(zh[k], lp[lh[k]]);
            }
#pragma unroll
            for (int m = 0; m < HTM; ++m)
                if (th_in[m]) th[m] = next(zt[m], th[m]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < CPT; ++m)
        if (tid + RT * m < N) {
            if (!XG) put(xg, gc[m], x[XG ? 0 : m]);
            put(I.L.r, gc[m], r[m]);
        }
    if (rank == 0 && tid == 0) {
        st->sigma = sigma;
        st->iters = iters;
        st->resRel = resRel;
        st->status = status;
        st->zero = zero;
        st->done = 1;
    }
}

}  // namespace

// The estimate behind a plan: a wavefront's pass over 64 cells issues about
// 350 instructions, 0.6 us; a face cell costs its load and update; a meeting
// of several workgroups about 2.5 us, twice per iteration.
ResPlan resident_plan(const Dims4 &D, int budget, bool fewest)
{
    ResPlan best;
    const int nx = D.X - 2, ny = D.Y - 2, nz = D.Z - 2, nt = D.T - 2;
    if (nx < 1 || ny < 1 || nz < 1 || nt < 2 || D.st * D.T >= (1ll << 28) - 1) return best;
    const int px = nx + 1;
    for (int pt = 1; pt <= nt / 2 && pt <= budget; ++pt)
        for (int pz = 1; pz <= nz && pt * pz <= budget; ++pz)
            for (int py = 1; py <= ny && pt * pz * py <= budget; ++py) {
                // the largest box (part_at: lengths floor or ceil)
                const int by = (ny + py - 1) / py, bz = (nz + pz - 1) / pz,
                          bt = (nt + pt - 1) / pt;
                const int64_t slab = (int64_t)nx * by * bz, cells = slab * bt;
                const int64_t rows = (int64_t)by * bz * bt, hrows = 2ll * bt * (by + bz);
                if (cells > RT * R_CPT || slab > R_SLAB || rows > R_ROWS || hrows > R_HROWS ||
                    1 + (rows + hrows) * px > R_CELLS)
                    continue;
                const int nwg = py * pz * pt;
                const double faces = nwg > 1 ? (double)hrows * nx + 2. * slab : 0.;
                const double cost = 0.6 * (double)((cells + 255) / 256) + 0.15 * faces / 256. +
                                    (nwg > 1 ? 2.5 + 0.015 * nwg : 0.);
                const bool better = best.nwg == 0 ||
                                    (fewest ? nwg < best.nwg ||
                                                  (nwg == best.nwg && cost < best.cost)
                                            : cost < best.cost);
                if (better) {
                    best.py = py;
                    best.pz = pz;
                    best.pt = pt;
                    best.nwg = nwg;
                    best.cells = (int)cells;
                    best.cost = cost;
                }
            }
    return best;
}

bool resident_iterate(flof_ctx *ctx, const std::vector<ResLevel> &levels,
                      const std::vector<ResPlan> &plans)
{
    const int n = (int)levels.size();
    if (n == 0) return true;
    int total = 0, most = 0;
    for (const ResPlan &p : plans) {
        if (p.nwg < 1) return false;
        total += p.nwg;
        most = std::max(most, p.cells);
    }
    if (total > ctx->num_cu) return false;
    const size_t slot_bytes = (size_t)total * 2 * R_SLOT;
    Tmp slots(ctx, slot_bytes + 256), tab(ctx, (size_t)n * sizeof(ResItem));
    launch_fill(ctx, slots.p, slot_bytes + 256);
    unsigned *abort_word = (unsigned *)((char *)slots.p + slot_bytes);
    std::vector<ResItem> h(n);
    int first = 0;
    for (int j = 0; j < n; ++j) {
        ResItem &I = h[j];
        I.L = levels[j];
        I.py = plans[j].py;
        I.pz = plans[j].pz;
        I.pt = plans[j].pt;
        I.first = first;
        I.nwg = plans[j].nwg;
        I.fnx = make_fastdiv((uint32_t)(levels[j].D.X - 2));
        I.slots = slots.as<char>() + (size_t)first * 2 * R_SLOT;
        first += I.nwg;
    }
    FLOF_HIP(hipMemcpyAsync(tab.p, h.data(), (size_t)n * sizeof(ResItem), hipMemcpyHostToDevice,
                            ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));  // h lives on the stack
    const ResItem *dt = tab.as<ResItem>();
    int ni = n;
    // of the 100 MHz clock
    unsigned long long ticks = (unsigned long long)(std::min(ctx->resident_wait, 60.) * 1e8);
    void *args[] = {(void *)&dt, (void *)&ni, (void *)&abort_word, (void *)&ticks};
    const int cpt = (most + RT - 1) / RT;
    const void *k = cpt <= 1   ? (const void *)k_cg_resident<1, false>
                    : cpt <= 2 ? (const void *)k_cg_resident<2, false>
                    : cpt <= 4 ? (const void *)k_cg_resident<4, false>
                    : cpt <= 6 ? (const void *)k_cg_resident<6, false>
                    : cpt <= 8 ? (const void *)k_cg_resident<8, false>
                               : (const void *)k_cg_resident<R_CPT, true>;
    // no form that a compiler gave scratch memory (see the top of the file)
    hipFuncAttributes fa;
    if (hipFuncGetAttributes(&fa, k) != hipSuccess || fa.localSizeBytes != 0) {
        (void)hipGetLastError();
        return false;
    }
    const hipError_t e =
        hipLaunchCooperativeKernel(k, dim3(total), dim3(RT), args, 0, ctx->stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    unsigned gave_up = 0;
    FLOF_HIP(hipMemcpyAsync(&gave_up, abort_word, sizeof(unsigned), hipMemcpyDeviceToHost,
                            ctx->stream));
    FLOF_HIP(hipStreamSynchronize(ctx->stream));
    return gave_up == 0;
}

}  // namespace flof
