// pf_resident.hip -- colour sweeps of a whole solve in one launch, the grid resident on chip.
//
// A step of fixed-count SOR is 2 * iter_max half-sweeps of one grid.  As one launch per
// half-sweep each of them reads p, bb and porosity from memory again and pays a launch
// boundary (about 3 us).  The register files and LDS of 256 CUs hold 170 MB, so a grid of
// up to 4.2 M cells (FP64; 8.4 M in FP32) fits on the chip: each workgroup owns a tile and
// keeps it for the whole solve, p and bb in registers, p once more in LDS for the x and y
// neighbours.  Only the tile's surface moves between workgroups, once per half-sweep.
//
// Exchange.  A surface value travels as 8-byte words that carry 32 bits of the value and
// the half-sweep's 32-bit sequence number (two words a double, one a float), written and
// read past the L2 (device scope).  An aligned word is whole or not there, so a reader that
// sees the sequence number has the value: no fence, no flag, no cache write-back, and one
// trip through memory per half-sweep.  Each cell's message has two slots, by iteration
// parity.  A block writes a slot again two iterations later, when it has received
// messages that its neighbour sent after reading the slot.
//
// Waiting.  The blocks need each other and are at most one per CU, but the launch is an
// ordinary one: after a cooperative launch the process's other streams ran one after the
// other (16 rooms on three streams 150 -> 270 ms a step).  So nothing rests on their being
// resident together.  Every wait ends after a bounded number of polls; then, or as soon as
// another block has given up, a block leaves without a trace: results are written only after
// all blocks have counted themselves in at the end (commit).  The host looks at the count
// after the launch and runs the per-half-sweep kernels where it came to nothing.
//
// Arithmetic.  Per cell the operations and their order are those of sor_value (FP64) and
// sor32_value (FP32), on the same operands: a cell whose seven porosities are 1 takes the
// unit faces and the wave's divisor (sor_unit_value), any other cell its coefficients as
// sor_coefs (FP32: sor32_coefs) built them once per porosity field.
//
// Measured, us per half-sweep, one launch per half-sweep / resident: FP64 sphere 256x128x128
// 17.0 / 9.6, sphere 97x65x49 7.9 / 2.8, room 128^3 13.4 / 7.6; FP32 sphere 256x128x128
// 10.2 / 6.8, room 128^3 8.3 / 4.5.  What bounds it: an exchange takes about 1.6 us however little
// travels (a 64x64x64 grid on 256 blocks, 1.8 us); a tile of 16384 unit cells takes 5.0 us (FP64:
// 0.4 us of arithmetic per height pair); a tile around a body, whose waves read seven coefficients
// a cell, waits about 0.65 us a height pair for them, and its neighbours wait for it; in an FP64
// room, where nearly all waves read them, all tiles together read 6 to 9 TB/s.  Tiles of
// 32x32 columns: 64x16, which spread a body over twice the tiles, took 10.6 us on the sphere.
// Sends at the end of a wave's half-sweep instead of per height pair took 10.4, coefficients
// fetched a height pair ahead 11.6 (registers spill).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "pf_cells.h"
#include "pf_device.h"
#include "pf_kernels.h"

namespace pf {

namespace {

constexpr int RT = 32;              // widest tile in x and y
constexpr int RP = RT + 2;          // LDS pitch of a plane with its halo
constexpr int RPL = RP * RP;
constexpr int RMAXT = 1024;         // threads of a block, one per column of the tile

typedef unsigned long long u64;

constexpr int DEV = 16;   // device scope (sc1); the streaming hint (nt) made every exchange 0.5 us longer
// The compiler knows no other writer of the inbox: nothing may be merged with an earlier
// poll or moved out of the loop of polls.
__device__ __forceinline__ void memory_changes() { asm volatile("" ::: "memory"); }
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
using rsrc = __amdgpu_buffer_rsrc_t;

// A message at byte `off` of the inbox from scalar offset `base`.  One store instruction per
// message and consecutive lanes on consecutive messages: two 8-byte stores into one line
// wait for each other's trip to memory (2.9 us per height pair in FP64 that way).
template <typename T>
struct Msg;
template <>
struct Msg<double> {
    static constexpr int B = 16;
    static __device__ __forceinline__ void send(rsrc q, uint32_t off, int base, double v, uint32_t seq) {
        const u64 b = (u64)__double_as_longlong(v);
        const v4u m = {(unsigned)b, seq, (unsigned)(b >> 32), seq};
        __builtin_amdgcn_raw_buffer_store_b128(m, q, (int)off, base, DEV);
    }
    static __device__ __forceinline__ v4u get(rsrc q, uint32_t off, int base) {
        memory_changes();
        return __builtin_amdgcn_raw_buffer_load_b128(q, (int)off, base, DEV);
    }
    static __device__ __forceinline__ bool ok(const v4u &m, uint32_t seq) { return m.y == seq && m.w == seq; }
    static __device__ __forceinline__ double value(const v4u &m) {
        return __longlong_as_double((long long)(((u64)m.z << 32) | m.x));
    }
};
template <>
struct Msg<float> {
    static constexpr int B = 8;
    static __device__ __forceinline__ void send(rsrc q, uint32_t off, int base, float v, uint32_t seq) {
        const v2u m = {__float_as_uint(v), seq};
        __builtin_amdgcn_raw_buffer_store_b64(m, q, (int)off, base, DEV);
    }
    static __device__ __forceinline__ v2u get(rsrc q, uint32_t off, int base) {
        memory_changes();
        return __builtin_amdgcn_raw_buffer_load_b64(q, (int)off, base, DEV);
    }
    static __device__ __forceinline__ bool ok(const v2u &m, uint32_t seq) { return m.y == seq; }
    static __device__ __forceinline__ float value(const v2u &m) { return __uint_as_float(m.x); }
};

// Messages of one block and iteration parity: four sides of 2 * NS * RT cells (colour,
// height pair, position along the side), then bottom and top, one per column.
template <int NS>
constexpr int msg_items() { return 4 * 2 * NS * RT + 2 * RMAXT; }

// Block blockIdx runs on XCD blockIdx % 8.  The tiles of a row of tiles are turned by this
// much against the row's blocks, so that tiles that are neighbours in y and z, which read
// coefficients of the same body, are on different XCDs: a body's coefficients then share
// eight L2s (4 MB each) instead of the one or two that its x range falls on.  us a half-sweep
// without / with: FP64 boxes 256x128x128 13.1 / 10.2, sphere 10.3 / 9.6, room 128^3 8.2 / 7.6;
// FP32 8.1 / 7.1, 6.7 / 6.8, 4.8 / 4.5; where bx is no multiple of 8 the same.
__device__ __forceinline__ int tile_turn(const ResidentPlan &pl, int iy, int iz) {
    return (pl.bx % 8 == 0) ? 2 * iy + 4 * iz : iz;
}
__device__ __forceinline__ int block_of(const ResidentPlan &pl, int ix, int iy, int iz) {
    return (ix + (iy + iz) * 8 * pl.bx - tile_turn(pl, iy, iz)) % pl.bx + pl.bx * (iy + pl.by * iz);
}

struct Tile {
    int blk, ix, iy, iz;
    int x0, y0, z0;      // first cell (1-based)
    int hx, hy, hz;      // cells held
    int x, y;            // this thread's column
    bool act;
};
__device__ __forceinline__ Tile tile_of(const PfGeom &g, const ResidentPlan &pl) {
    Tile t;
    t.blk = (int)blockIdx.x;
    t.iy = (t.blk / pl.bx) % pl.by;
    t.iz = t.blk / (pl.bx * pl.by);
    t.ix = (t.blk + tile_turn(pl, t.iy, t.iz)) % pl.bx;
    t.x0 = t.ix * pl.tx + 1;
    t.y0 = t.iy * pl.ty + 1;
    t.z0 = t.iz * pl.tz + 1;
    t.hx = min(pl.tx, g.m - t.x0 + 1);
    t.hy = min(pl.ty, g.n - t.y0 + 1);
    t.hz = min(pl.tz, g.l - t.z0 + 1);
    // the columns of the west and east sides first, then the others row by row: consecutive
    // lanes then hold consecutive cells of a side, and its messages fill whole lines
    const int tid = (int)threadIdx.x, r = tid - 2 * t.hy;
    if (r < 0) {
        t.x = tid < t.hy ? 0 : t.hx - 1;
        t.y = tid < t.hy ? tid : tid - t.hy;
        t.act = true;
    } else {
        const int wx = max(t.hx - 2, 1);
        t.y = r / wx;
        t.x = 1 + r - t.y * wx;
        t.act = t.y < t.hy && t.hx > 2;
    }
    return t;
}

}  // namespace

// ------------------------------------------------------------------------------------
// Once per porosity field.  mask: per wave a bit for each colour and height pair
// (colour * NS + pair), set when all its cells there take the unit faces.  coef: for each
// clear bit, in order, seven rows of 64 lanes from the wave's place `first`: the cells'
// coefficients after the boundary rows' rules (ae, aw, an, as, at, ab) and ap (FP32: the
// reciprocal of ap that the sweep multiplies by).
// ------------------------------------------------------------------------------------
template <typename T, int NS, bool FAST, bool FILL>
__global__ __launch_bounds__(RMAXT) void k_resident_setup(PfGeom g, StepArgs a, ResidentPlan pl,
                                                          const T *__restrict__ PHI, const double *__restrict__ phi,
                                                          T *__restrict__ coef, uint32_t *__restrict__ mask,
                                                          const uint32_t *__restrict__ first) {
    const Tile t = tile_of(g, pl);
    const int tid = (int)threadIdx.x, wave = t.blk * ((int)blockDim.x >> 6) + (tid >> 6);
    const int i = t.x0 + t.x, j = t.y0 + t.y;
    uint32_t bits = 0;
    T *o = FILL ? coef + (int64_t)first[wave] * (7 * 64) + (tid & 63) : nullptr;
    const uint32_t m = FILL ? mask[wave] : 0u;
    for (int c = 0; c < 2; ++c)
        for (int s = 0; s < NS; ++s) {
            if (FILL && ((m >> (c * NS + s)) & 1u)) continue;
            const int z = 2 * s + ((i + j + t.z0 + c) & 1), k = t.z0 + z;
            bool unit = true;
            T cf[7] = {};
            if (t.act && z < t.hz) {
                const T fc = PHI[pf_soff(g, i, j, k)], fw = PHI[pf_soff(g, i - 1, j, k)],
                        fe = PHI[pf_soff(g, i + 1, j, k)], fs = PHI[pf_soff(g, i, j - 1, k)],
                        fn = PHI[pf_soff(g, i, j + 1, k)], fb = PHI[pf_soff(g, i, j, k - 1)],
                        ft = PHI[pf_soff(g, i, j, k + 1)];
                if (FILL) {
                    CoefT<T> q;
                    T ap;
                    if constexpr (std::is_same<T, double>::value) {
                        ap = sor_coefs<3, FAST>(g, a, i, j, k, fc, fw, fe, fs, fn, fb, ft, phi, q);
                    } else {
                        sor32_coefs<3>(g, a, i, j, k, fc, fw, fe, fs, fn, fb, ft, phi, (float)(a.dt / (a.dx * a.dx)),
                                       (float)(a.dt / (a.dy * a.dy)), (float)(a.dt / (a.dz * a.dz)), q, ap);
                        ap = __builtin_amdgcn_rcpf(ap);
                    }
                    cf[0] = q.ae; cf[1] = q.aw; cf[2] = q.an; cf[3] = q.as; cf[4] = q.at; cf[5] = q.ab; cf[6] = ap;
                }
                const T one = T(1);
                unit = fc == one && fw == one && fe == one && fs == one && fn == one && fb == one && ft == one &&
                       !(a.bc == PF_BC_AIR && is_edge_row(g, a, i, j, k));
            }
            if (FILL) {
                for (int q = 0; q < 7; ++q) o[q * 64] = cf[q];
                o += 7 * 64;
            } else if (__all(unit)) {
                bits |= 1u << (c * NS + s);
            }
        }
    if (!FILL && (tid & 63) == 0) mask[wave] = bits;
}

namespace {

template <typename T>
struct ResidentRun {
    PfGeom g;
    StepArgs a;
    ResidentPlan pl;
    int iters;
    uint32_t seq;      // half-sweep h carries seq + h
    T *X;              // p (FP64) or the correction (FP32), colour-split
    const T *R;        // right-hand side
    const T *coef;
    const uint32_t *mask, *first;
    u64 *inbox;
    u64 *slots;
    u64 *count, target;   // blocks that reached the end, over all launches: target with this one's
    unsigned polls;       // of a wait, at most
};

using lds_int = __attribute__((address_space(3))) volatile int *;
constexpr uint32_t NONE = 0xfffffff0u;   // no place: beyond every inbox

// What a thread keeps for the whole solve: the wave-uniform part and its column's.
template <typename T, int NS>
struct Work {
    // the grid, the tile and its neighbours (-1: none, the ghost cells keep their values)
    int gm, gn, gl, tid, nthr, nside, zc;
    Tile t;
    int bw, be, bs, bn, bb, bt;
    uint32_t seq, um;
    rsrc inbox;
    const T *coef;          // the wave's coefficients
    double unit_ap, omega, omega_c;
    DivK kap;
    T *L;
    lds_int dead;
    u64 *count;
    unsigned polls;
    // the column
    T b[2][NS];             // right-hand side by colour and height pair: cell (c, s) lies at z = 2s + q(c)
    T zlo, zhi;             // the cells below and above the column
    T ce, cw, cn, cz;       // unit faces after the x rows' rules: east, west, y, z
    T uap;                  // FP32: reciprocal of the unit ap
    double err;
    int q0, lc;             // height of the first cell of colour 0; the column's LDS offset
    int colb, colt;         // colours of the cells below and above
    uint32_t zo;            // its place among the bottom and top messages
    uint32_t ox, oy;        // where its side cells go, in bytes of the inbox
    uint32_t sp0, sp1;      // the side message this thread takes in, per colour: from, and
    int sd0, sd1;           // where to in LDS
};

// Byte offset of a side's messages in the inbox (32 bits: a plan is at most 256 blocks).
template <typename T, int NS>
__device__ __forceinline__ uint32_t box(int blk, int dir) {
    return (uint32_t)(blk * 2 * msg_items<NS>() + (dir < 4 ? dir * 2 * NS * RT : 8 * NS * RT + (dir - 4) * RMAXT)) *
           Msg<T>::B;
}

// Side message e of the 2 * NS * (hx + hy) that cells of colour cc send this tile: its byte
// in the inbox and its LDS place, or false where that cell does not exist.
template <typename T, int NS>
__device__ __forceinline__ bool side_item(const Work<T, NS> &w, int e, int cc, uint32_t &src, int &dst) {
    const Tile &t = w.t;
    const int ny = NS * t.hy, nx = NS * t.hx;
    int dir, pos, s;
    if (e < 2 * ny) {
        dir = e >= ny;
        const int f = e - dir * ny;
        s = f / t.hy;
        pos = f - s * t.hy;
    } else {
        const int f0 = e - 2 * ny;
        dir = 2 + (f0 >= nx);
        const int f = f0 - (dir - 2) * nx;
        s = f / t.hx;
        pos = f - s * t.hx;
    }
    const int b0 = w.bw, b1 = w.be, b2 = w.bs, b3 = w.bn;   // read before the choice: w stays in registers
    const int nb = dir == 0 ? b0 : dir == 1 ? b1 : dir == 2 ? b2 : b3;
    // the halo cell's own coordinates, and those of the cell it mirrors
    const int xh = dir == 0 ? 0 : dir == 1 ? t.hx + 1 : pos + 1;
    const int yh = dir < 2 ? pos + 1 : dir == 2 ? 0 : t.hy + 1;
    const int ci = t.x0 - 1 + xh;
    int cj = t.y0 - 1 + yh;
    const int gp = ci + cj + t.z0;
    if (cj == 0) cj = w.gn;
    else if (cj == w.gn + 1) cj = 1;
    const int z = 2 * s + ((ci + cj + t.z0 + cc) & 1);
    src = box<T, NS>(t.blk, dir) + (uint32_t)((cc * NS + s) * RT + pos) * Msg<T>::B;
    dst = ((((gp + z) & 1) * NS) + s) * RPL + yh * RP + xh;
    return nb >= 0 && z < t.hz;
}

constexpr u64 GONE = 1ull << 63;   // in the commit count: a block has given up

__device__ __forceinline__ u64 count_now(u64 *count) {
    return __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One more poll without success: true when the wait is over without its message.
__device__ __forceinline__ bool give_up(unsigned &spin, lds_int dead, u64 *count, unsigned polls) {
    ++spin;
    if (spin < polls && !*dead && ((spin & 255u) || !(count_now(count) & GONE))) return false;
    *dead = 1;
    return true;
}

// The end of a block (one thread): true when every block of the launch has come here, which
// brings the count to `target`, and none had given up before.  The two are decided by the
// one word, so all blocks get the same answer.
__device__ __forceinline__ bool commit(u64 *count, u64 target, bool dead, unsigned polls) {
    if (!dead) (void)__hip_atomic_fetch_add(count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    u64 v = count_now(count);
    for (unsigned spin = 0; !dead && spin < polls; ++spin) {
        if (v & GONE) return false;
        if (v >= target) return true;
        v = count_now(count);
    }
    while (!(v & GONE)) {
        if (v >= target) return true;
        if (__hip_atomic_compare_exchange_strong(count, &v, v | GONE, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return false;
    }
    return false;
}

// Half-sweep h, of colour C.
template <typename T, int NS, int C, bool ODDY>
__device__ __forceinline__ void half_sweep(Work<T, NS> &w, int h) {
    constexpr int O = 1 - C, B = Msg<T>::B, IT = msg_items<NS>();
    const Tile &t = w.t;
    // Values that every half-sweep derives addresses and lane masks from, hidden from the
    // compiler: hoisted out of the loop over half-sweeps, those of all height pairs together
    // do not fit the registers.
    int hz = t.hz, q0 = w.q0;
    uint32_t ox = w.ox, oy = w.oy, um = w.um;
    asm volatile("" : "+s"(hz), "+s"(um), "+v"(q0), "+v"(ox), "+v"(oy));
    if (h > 0) {
        // colour O, half-sweep h - 1, comes in
        const uint32_t seq = w.seq + (uint32_t)(h - 1);
        const int in = (((h - 1) >> 1) & 1) * IT * B;
        if (ODDY) __syncthreads();   // half-sweep h - 1 has read the halo cells that are written here
        const int inb = in + (int)box<T, NS>(t.blk, 4) + O * w.zc, inT = in + (int)box<T, NS>(t.blk, 5) + O * w.zc;
        const uint32_t sp = O ? w.sp1 : w.sp0;
        const int sd = O ? w.sd1 : w.sd0;
        bool w0 = w.bb >= 0 && t.act && w.colb == O, w1 = w.bt >= 0 && t.act && w.colt == O, w2 = sp != NONE;
        unsigned spin = 0;
        while (w0 || w1 || w2) {
            // every message still missing, in flight together; a lane that misses none of a
            // kind reads the first one's place and ignores it
            const auto m0 = Msg<T>::get(w.inbox, w0 ? w.zo : 0u, inb);
            const auto m1 = Msg<T>::get(w.inbox, w1 ? w.zo : 0u, inT);
            const auto m2 = Msg<T>::get(w.inbox, w2 ? sp : 0u, in);
            if (w0 && Msg<T>::ok(m0, seq)) { w.zlo = Msg<T>::value(m0); w0 = false; }
            if (w1 && Msg<T>::ok(m1, seq)) { w.zhi = Msg<T>::value(m1); w1 = false; }
            if (w2 && Msg<T>::ok(m2, seq)) { w.L[sd] = Msg<T>::value(m2); w2 = false; }
            if ((w0 || w1 || w2) && give_up(spin, w.dead, w.count, w.polls)) break;
        }
        for (int e = w.tid + w.nthr; e < w.nside; e += w.nthr) {
            uint32_t src;
            int dst;
            if (!side_item<T, NS>(w, e, O, src, dst)) continue;
            auto m = Msg<T>::get(w.inbox, src, in);
            while (!Msg<T>::ok(m, seq)) {
                if (give_up(spin, w.dead, w.count, w.polls)) break;
                m = Msg<T>::get(w.inbox, src, in);
            }
            w.L[dst] = Msg<T>::value(m);
        }
    }
    __syncthreads();
    if (!t.act) return;
    const uint32_t seq = w.seq + (uint32_t)h;
    const int to = ((h >> 1) & 1) * IT * B;
    const int tob = to + (int)box<T, NS>(w.bb, 5) + C * w.zc, tot = to + (int)box<T, NS>(w.bt, 4) + C * w.zc;
    const bool odd = C ? q0 == 0 : q0 == 1;   // this column's first cell of colour C lies at z = 1
    const T *X = w.L + O * NS * RPL + w.lc;
    T *Y = w.L + C * NS * RPL + w.lc;
    T below = w.zlo, mid = X[0];
    const float om32 = (float)w.omega;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (2 * s >= hz) break;
        // one height pair at a time: hoisted loads of all of them do not fit the registers
        __builtin_amdgcn_sched_barrier(0);
        const T pc = Y[s * RPL], rhs = w.b[C][s];
        const T pE = X[s * RPL + 1], pW = X[s * RPL - 1], pN = X[s * RPL + RP], pS = X[s * RPL - RP];
        const T above = s + 1 < NS ? X[(s + 1 < NS ? s + 1 : s) * RPL] : w.zhi;
        const T pB = odd ? mid : below;
        T pT = odd ? above : mid;
        below = mid;
        mid = above;
        const int z = 2 * s + (odd ? 1 : 0);
        if (2 * s + 2 >= hz) pT = (z + 1 == hz) ? w.zhi : pT;
        T pn;
        if ((um >> (C * NS + s)) & 1u) {
            if constexpr (std::is_same<T, double>::value) {
                const double num = (((((rhs - (w.ce * pE)) - (w.cw * pW)) - (w.cn * pN)) - (w.cn * pS)) -
                                    (w.cz * pT)) - (w.cz * pB);
                DivFast dv;
                double d = dv(num, w.kap);
                if (dv.slow) {
                    double ap = w.unit_ap;
                    asm("" : "+v"(ap));   // a vector register: the division's scaling takes no scalar here
                    d = num / ap;
                }
                pn = (d * w.omega) + (pc * w.omega_c);
            } else {
                float num = rhs - w.ce * pE - w.cw * pW - w.cn * pN - w.cn * pS;
                num = num - w.cz * pT - w.cz * pB;
                pn = num * w.uap * om32 + pc * (1.f - om32);
                asm volatile("" : "+v"(pn));   // kept apart from the other branch and its waits
            }
        } else {
            // the wave's sets of seven rows of 64, in the order of its clear bits
            const int BIT = C * NS + s;
            const int set = __builtin_popcount(~um & ((1u << BIT) - 1u));
            const auto co = gmem(w.coef + (int64_t)set * (7 * 64));
            T cf[7];
#pragma unroll
            for (int q = 0; q < 7; ++q) cf[q] = co[q * 64 + (uint32_t)(w.tid & 63)];
            if constexpr (std::is_same<T, double>::value) {
                const double num = (((((rhs - (cf[0] * pE)) - (cf[1] * pW)) - (cf[2] * pN)) - (cf[3] * pS)) -
                                    (cf[4] * pT)) - (cf[5] * pB);
                pn = ((num / cf[6]) * w.omega) + (pc * w.omega_c);
            } else {
                float num = rhs - cf[0] * pE - cf[1] * pW - cf[2] * pN - cf[3] * pS;
                num = num - cf[4] * pT - cf[5] * pB;
                pn = num * cf[6] * om32 + pc * (1.f - om32);
            }
        }
        if (z < hz) {
            Y[s * RPL] = pn;
            if (C == 1) w.err = max_keep_nan(w.err, fabs((double)pn - (double)pc));
            // out at once: the trip to memory overlaps the other height pairs
            const int side = to + (C * NS + s) * RT * B;
            if (ox != NONE) Msg<T>::send(w.inbox, ox, side, pn, seq);
            if (oy != NONE) Msg<T>::send(w.inbox, oy, side, pn, seq);
            if (s == 0 && w.bb >= 0 && z == 0) Msg<T>::send(w.inbox, w.zo, tob, pn, seq);
            if (2 * s + 2 >= hz && w.bt >= 0 && z == hz - 1) Msg<T>::send(w.inbox, w.zo, tot, pn, seq);
        }
    }
}

}  // namespace

template <typename T, int NS, bool ODDY>
__global__ __launch_bounds__(RMAXT) void k_sor_resident(ResidentRun<T> r) {
    extern __shared__ __align__(16) char lds_raw[];   // past `dead`, and still aligned for b64 access
    T *L = (T *)lds_raw;   // [coordinate parity][s][y + 1][x + 1]
    __shared__ int dead;
    Work<T, NS> w;
    w.t = tile_of(r.g, r.pl);
    const Tile &t = w.t;
    const int tid = (int)threadIdx.x, nthr = (int)blockDim.x;
    const int i = t.x0 + t.x, j = t.y0 + t.y;
    const bool periodic = r.a.bc == PF_BC_UNIFORM;
    const int bx = r.pl.bx, by = r.pl.by, bz = r.pl.bz;
    if (tid == 0) dead = 0;
    w.dead = (lds_int)&dead;
    w.count = r.count;
    w.polls = r.polls;
    w.L = L;
    w.gm = r.g.m;
    w.gn = r.g.n;
    w.gl = r.g.l;
    w.tid = tid;
    w.nthr = nthr;
    w.nside = 2 * NS * (t.hx + t.hy);
    w.seq = r.seq;
    w.inbox = __builtin_amdgcn_make_buffer_rsrc(r.inbox, 0, (int)((uint32_t)gridDim.x * 2 * msg_items<NS>() * Msg<T>::B),
                                                0x27000);
    w.unit_ap = r.a.unit_ap;
    w.omega = r.a.omega;
    w.omega_c = r.a.omega_c;
    const auto at = [&](int ix, int iy, int iz) __attribute__((always_inline)) {
        return block_of(r.pl, ix, iy, iz);
    };
    w.bw = t.ix > 0 ? at(t.ix - 1, t.iy, t.iz) : -1;
    w.be = t.ix < bx - 1 ? at(t.ix + 1, t.iy, t.iz) : -1;
    w.bs = (t.iy > 0 || periodic) ? at(t.ix, t.iy > 0 ? t.iy - 1 : by - 1, t.iz) : -1;
    w.bn = (t.iy < by - 1 || periodic) ? at(t.ix, t.iy < by - 1 ? t.iy + 1 : 0, t.iz) : -1;
    w.bb = (t.iz > 0 || periodic) ? at(t.ix, t.iy, t.iz > 0 ? t.iz - 1 : bz - 1) : -1;
    w.bt = (t.iz < bz - 1 || periodic) ? at(t.ix, t.iy, t.iz < bz - 1 ? t.iz + 1 : 0) : -1;

    // The tile and its halo into LDS, the column's right-hand side into registers.  Half-sweep 0
    // takes periodic ghosts as they are in memory (an uploaded pressure's are what the caller
    // gave), later ones the cells that they mirror.  Across an odd extent a ghost has its
    // reader's colour: those that colour 1 reads are first read in half-sweep 1, before any
    // message of that colour, so they come from their cells here.
    const bool oddz = periodic && (r.g.l & 1);
    {
        const int wx = t.hx + 2, wxy = wx * (t.hy + 2), nc = wxy * t.hz;
        for (int e = tid; e < nc; e += nthr) {
            const int z = e / wxy, yx = e - z * wxy, yy = yx / wx, xx = yx - yy * wx;
            const int ci = t.x0 - 1 + xx, cj = t.y0 - 1 + yy, ck = t.z0 + z, par = (ci + cj + ck) & 1;
            const int sj = (ODDY && par == 0) ? (cj == 0 ? r.g.n : cj == r.g.n + 1 ? 1 : cj) : cj;
            L[(par * NS + (z >> 1)) * RPL + yy * RP + xx] = r.X[pf_soff(r.g, ci, sj, ck)];
        }
    }
    w.q0 = (i + j + t.z0) & 1;   // colour 1: 1 - q0
    w.zlo = w.zhi = T(0);
    w.err = 0.;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int z = 2 * s + (c ? 1 - w.q0 : w.q0);
            w.b[c][s] = T(0);
            if (t.act && z < t.hz) w.b[c][s] = r.R[pf_soff(r.g, i, j, t.z0 + z)];
        }
    if (t.act) {
        const bool lo = oddz && t.z0 == 1 && ((i + j + 1) & 1);
        const bool hi = oddz && t.z0 + t.hz - 1 == r.g.l && ((i + j + r.g.l) & 1);
        w.zlo = r.X[pf_soff(r.g, i, j, lo ? r.g.l : t.z0 - 1)];
        w.zhi = r.X[pf_soff(r.g, i, j, hi ? 1 : t.z0 + t.hz)];
    }
    if constexpr (std::is_same<T, double>::value) {
        w.ce = w.cw = r.a.unit_ax;
        w.cn = r.a.unit_ay;
        w.cz = r.a.unit_az;
        w.uap = 0.;
    } else {
        const float cdx = (float)(r.a.dt / (r.a.dx * r.a.dx)), cdy = (float)(r.a.dt / (r.a.dy * r.a.dy)),
                    cdz = (float)(r.a.dt / (r.a.dz * r.a.dz));
        w.ce = w.cw = face32(1.f, 1.f, cdx);
        w.cn = face32(1.f, 1.f, cdy);
        w.cz = face32(1.f, 1.f, cdz);
        w.uap = __builtin_amdgcn_rcpf(-(w.ce + w.cw + w.cn + w.cn + w.cz + w.cz));
    }
    if (periodic) {   // the x rows' rules; an air room's edge cells are never unit cells
        if (i == 1) {
            w.ce = w.ce + w.cw;
            w.cw = T(0);
        }
        if (i == r.g.m) w.ce = w.cw = w.cn = w.cz = T(0);
    }
    w.kap = divk_make(r.a.unit_ap);
    {
        const int wave = __builtin_amdgcn_readfirstlane(t.blk * (nthr >> 6) + (tid >> 6));
        w.um = r.mask[wave];
        w.coef = r.coef + (int64_t)r.first[wave] * (7 * 64);
    }
    w.lc = (t.y + 1) * RP + t.x + 1;

    // where this column's side values go in the neighbours' inboxes (a tile is at least two
    // cells wide, so a column borders one tile at most in x and one in y)
    w.ox = w.oy = NONE;
    if (t.act) {
        const uint32_t ay = (uint32_t)(t.y * Msg<T>::B), ax = (uint32_t)(t.x * Msg<T>::B);
        if (t.x == 0 && w.bw >= 0) w.ox = box<T, NS>(w.bw, 1) + ay;
        if (t.x == t.hx - 1 && w.be >= 0) w.ox = box<T, NS>(w.be, 0) + ay;
        if (t.y == 0 && w.bs >= 0) w.oy = box<T, NS>(w.bs, 3) + ax;
        if (t.y == t.hy - 1 && w.bn >= 0) w.oy = box<T, NS>(w.bn, 2) + ax;
    }
    // the colour of the cells below and above (an odd periodic extent wraps a colour onto itself)
    w.colb = (i + j + ((t.z0 == 1 && w.bb >= 0) ? w.gl : t.z0 - 1)) & 1;
    w.colt = (i + j + ((t.z0 + t.hz - 1 == w.gl && w.bt >= 0) ? 1 : t.z0 + t.hz)) & 1;
    // where the sides are even columns 2q and 2q + 1 differ in colour, so each colour's bottom
    // and top messages are packed in its own half
    const bool odd_sides = ((t.hx | t.hy) & 1) != 0;
    w.zo = (uint32_t)(odd_sides ? tid : tid >> 1) * Msg<T>::B;
    w.zc = odd_sides ? 0 : RMAXT / 2 * Msg<T>::B;
    w.sp0 = w.sp1 = NONE;
    w.sd0 = w.sd1 = 0;
    if (tid < w.nside) {
        uint32_t src;
        int dst;
        if (side_item<T, NS>(w, tid, 0, src, dst)) { w.sp0 = src; w.sd0 = dst; }
        if (side_item<T, NS>(w, tid, 1, src, dst)) { w.sp1 = src; w.sd1 = dst; }
    }

    for (int h = 0; h < 2 * r.iters; h += 2) {
        half_sweep<T, NS, 0, ODDY>(w, h);
        half_sweep<T, NS, 1, ODDY>(w, h + 1);
    }

    __syncthreads();
    if (tid == 0) dead = commit(r.count, r.target, dead != 0, r.polls) ? 0 : 1;
    __syncthreads();
    if (dead) return;

    // the column and its periodic mirrors back to memory
    if (t.act) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int z = 2 * s + (c ? 1 - w.q0 : w.q0), k = t.z0 + z;
                if (z >= t.hz) continue;
                const T v = L[(c * NS + s) * RPL + w.lc];
                r.X[pf_soff(r.g, i, j, k)] = v;
                if (periodic) {
                    if (j == r.g.n) r.X[pf_soff(r.g, i, 0, k)] = v;
                    if (j == 1) r.X[pf_soff(r.g, i, r.g.n + 1, k)] = v;
                    if (k == r.g.l) r.X[pf_soff(r.g, i, j, 0)] = v;
                    if (k == 1) r.X[pf_soff(r.g, i, j, r.g.l + 1)] = v;
                }
            }
    }
    wave_max_to_slot(w.err, r.slots);
}

// ------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------
// Polls of a wait, at most: about 50 ms of them (a poll is a trip to memory, 0.8 us).  Blocks
// that wait for others to be placed wait for the end of kernels in their way, a few ms; longer
// than that is another process's resident launch that waits as well.  PF_RESIDENT_POLLS in the
// environment sets another number (tests: 1 makes launches give up).
static unsigned resident_polls() {
    const char *e = std::getenv("PF_RESIDENT_POLLS");
    const int v = (e && *e) ? std::atoi(e) : 0;
    return v > 0 ? (unsigned)v : 1u << 16;
}

static int ns_of(int tz) {
    const int h = (tz + 1) / 2;
    return h <= 1 ? 1 : h <= 2 ? 2 : h <= 4 ? 4 : h <= 8 ? 8 : 16;
}

// Estimated us of a half-sweep for the slowest tile, one around a body: all of its waves read
// coefficients.  A wave waits about 0.65 us a height pair for its seven loads, which other waves
// of the SIMD cover until the CU's loads themselves take longer (0.074 us a wave and pair in FP64,
// 0.034 in FP32); bottom and top messages cost by the tile's columns, more where they are not
// packed (odd sides), side messages by a thread's share of them.  Fitted to 340 timings of 53
// rooms, spheres and fields of boxes of 0.1 to 8 M cells with tilings of every shape; the
// error is 4 to 5 % (rms).
static double body_tile_us(const ResidentPlan &pl, int elem) {
    const double pairs = (pl.tz + 1) / 2, waves = pl.threads / 64, columns = pl.tx * pl.ty;
    const bool f64 = elem == 8, odd = ((pl.tx | pl.ty) & 1) != 0;
    const double wait = 0.65 * pairs, loads = (f64 ? 0.074 : 0.034) * pairs * waves;
    const double w2 = wait * wait, l2 = loads * loads;
    const double columns_us = f64 ? (odd ? 2.00e-3 : 1.66e-3) : (odd ? 0.93e-3 : 0.90e-3);
    return (f64 ? 0.63 : 0.67) + std::sqrt(std::sqrt(w2 * w2 + l2 * l2)) + columns_us * columns +
           (f64 ? 0.42 : 0.24) * 2 * (pl.tx + pl.ty) * pairs / pl.threads;
}
// The same for a tile of unit cells: arithmetic of the fullest SIMD, and the surface.
static double unit_tile_us(const ResidentPlan &pl) {
    const int surface = 2 * ((pl.bx > 1 ? pl.ty : 0) + pl.tx) * pl.tz + 2 * pl.tx * pl.ty;
    return (double)((pl.threads / 64 + 3) / 4) * ((pl.tz + 1) / 2) * 0.1 + surface * 0.0004;
}

// The tiling with the least body_tile_us, and of those within 3 % of it the one with the least
// unit_tile_us: the slowest tile sets the pace of all.  By unit_tile_us alone a mixed room of
// 105x113x87 got 15x17x22 tiles, eleven pairs in a row with nothing to cover their loads: 7.9 us a
// half-sweep, streamed 6.4, now (27x29x6) 3.6.  us before / now: FP64 boxes 57x100x141 7.3 / 4.1,
// sphere 139x117x46 7.3 / 3.8, room 160x128x96 8.3 / 7.3, sphere 256x128x128 unchanged; FP32 room
// 128^3 6.7 / 4.6, 192x160x128 12.6 / 7.3, boxes 93x87x121 8.0 / 3.3; the worst of 53 grids, FP64
// room 51x88x52, 2.53 / 2.59.
bool resident_plan(const PfGeom &g, int elem, int cus, ResidentPlan &pl) {
    pl = ResidentPlan{};
    if (g.dim != 3 || g.m < 2 || g.n < 2 || g.l < 2) return false;
    const int maxns = elem == 8 ? 8 : 16;
    const char *e = std::getenv("PF_RESIDENT");
    int fx = 0, fy = 0, fz = 0;
    if (e && *e && std::sscanf(e, "%d,%d,%d", &fx, &fy, &fz) != 3) return false;
    const bool forced = fx > 0 && fy > 0 && fz > 0;
    double least = 1e300, unit = 1e300;
    bool choosing = false;   // first pass: the least estimate; second: the choice
    auto consider = [&](int bx, int by, int bz) {
        const int tx = (g.m + bx - 1) / bx, ty = (g.n + by - 1) / by, tz = (g.l + bz - 1) / bz;
        if (tx > RT || ty > RT || tx * ty > RMAXT || (tz + 1) / 2 > maxns) return;
        bx = (g.m + tx - 1) / tx;
        by = (g.n + ty - 1) / ty;
        bz = (g.l + tz - 1) / tz;
        if (bx * by * bz > cus) return;
        if (g.m - (bx - 1) * tx < 2 || g.n - (by - 1) * ty < 2) return;   // every tile two cells wide
        const ResidentPlan q{bx, by, bz, tx, ty, tz, ns_of(tz), (tx * ty + 63) / 64 * 64};
        const double us = body_tile_us(q, elem);
        if (!choosing) {
            least = std::min(least, us);
        } else if (us <= 1.03 * least && unit_tile_us(q) < unit) {
            unit = unit_tile_us(q);
            pl = q;
        }
    };
    for (int pass = 0; pass < 2; ++pass) {
        choosing = pass == 1;
        if (forced) {
            consider(fx, fy, fz);
            continue;
        }
        for (int bx = (g.m + RT - 1) / RT; bx <= cus && bx <= g.m; ++bx)
            for (int by = (g.n + RT - 1) / RT; bx * by <= cus && by <= g.n; ++by)
                for (int bz = (g.l + 2 * maxns - 1) / (2 * maxns); bx * by * bz <= cus && bz <= g.l; ++bz)
                    consider(bx, by, bz);
    }
    return pl.bx > 0;
}

// The least iterations of a solve for which the one launch is faster.  It costs 30 to 80 us more
// than sweeps do (the grid in and out of the chip, the agreement at the end, the host's wait for
// it) and saves 4 to 15 us an iteration; us a step of 6 / 8 / 12 iterations, streamed and resident:
// FP64 sphere 48x40x40 77, 77 / 92, 83 / 122, 96; room 64^3 107, 105 / 125, 114 / 160, 130; room 128^3
// 317, 311 / 370, 339 / 477, 400; sphere 192x128x96 279, 290 / 321, 314 / 399, 363; FP32 sphere
// 192x128x96 280, 302 / 309, 319 / 366, 354; 256x192x160 845, 868 / 910, 916 / 1036, 1011.  2D:
// 256x128 51, 60 / 58, 64 / 76, 73; 768x384 78, 92 / 93, 102 / 124, 124; odd n, which the
// sweeps follow with refreshes of the ghost rows, 511x255 93, 80 / 116, 88 / 165, 102.  A tiling
// set in the environment is used for every solve of two or more.
int resident_min_iters(const PfGeom &g, int elem) {
    const char *e = std::getenv("PF_RESIDENT");
    if (e && *e) return 2;
    if (g.dim == 2) return (g.n & 1) ? 6 : 12;
    if ((int64_t)g.m * g.n * g.l <= (1 << 19)) return 6;
    return elem == 8 ? 8 : 12;
}

int resident_waves(const ResidentPlan &pl) { return pl.bx * pl.by * pl.bz * (pl.threads / 64); }
int64_t resident_sets(const ResidentPlan &pl, const std::vector<uint32_t> &mask, std::vector<uint32_t> &first) {
    const uint32_t all = pl.ns == 16 ? 0xffffffffu : (1u << (2 * pl.ns)) - 1u;
    uint32_t n = 0;
    first.resize(mask.size());
    for (size_t w = 0; w < mask.size(); ++w) {
        first[w] = n;
        n += (uint32_t)__builtin_popcount(~mask[w] & all);
    }
    return n;
}
int64_t resident_inbox_words(const ResidentPlan &pl, int elem) {
    return (int64_t)pl.bx * pl.by * pl.bz * 2 * (4 * 2 * pl.ns * RT + 2 * RMAXT) * (elem == 8 ? 2 : 1);
}
static size_t resident_lds(const ResidentPlan &pl, int elem) { return (size_t)2 * pl.ns * RPL * elem; }
// The kernel's 1,024-thread bound leaves a wave 128 registers, a quarter of a SIMD's: a CU holds
// sixteen waves, and blocks for as long as their LDS fits.
int resident_quarters(const ResidentPlan &pl, int elem) {
    const int by_waves = 16 / (pl.threads / 64), by_lds = (int)((size_t)(160 << 10) / (resident_lds(pl, elem) + 64));
    const int per_cu = std::min(by_waves, by_lds);
    return pl.bx * pl.by * pl.bz * (per_cu >= 4 ? 1 : per_cu >= 2 ? 2 : 4);
}

template <typename T, int NS, bool ODDY>
static hipError_t run_resident(hipStream_t st, ResidentRun<T> &r) {
    const size_t lds = resident_lds(r.pl, (int)sizeof(T));
    const void *f = (const void *)k_sor_resident<T, NS, ODDY>;
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    void *args[] = {&r};
    return hipLaunchKernel(f, dim3((unsigned)(r.pl.bx * r.pl.by * r.pl.bz)), dim3((unsigned)r.pl.threads), args, lds, st);
}
template <typename T, int NS>
static hipError_t run_resident(hipStream_t st, ResidentRun<T> &r) {
    const bool oddy = r.a.bc == PF_BC_UNIFORM && (r.g.n & 1);
    return oddy ? run_resident<T, NS, true>(st, r) : run_resident<T, NS, false>(st, r);
}

template <typename T>
hipError_t launch_resident(hipStream_t st, const PfGeom &g, const StepArgs &a, const ResidentPlan &pl, int iters,
                           uint32_t seq, T *X, const T *R, const T *coef, const uint32_t *mask, const uint32_t *first_set,
                           unsigned long long *inbox, unsigned long long *slots, unsigned long long *count,
                            unsigned long long target) {
    ResidentRun<T> r{g, a, pl, iters, seq, X, R, coef, mask, first_set, inbox, slots, count, target, resident_polls()};
    switch (pl.ns) {
        case 1: return run_resident<T, 1>(st, r);
        case 2: return run_resident<T, 2>(st, r);
        case 4: return run_resident<T, 4>(st, r);
        case 8: return run_resident<T, 8>(st, r);
        default: break;
    }
    if constexpr (sizeof(T) == 4) return run_resident<T, 16>(st, r);
    return hipErrorInvalidValue;
}
template hipError_t launch_resident<double>(hipStream_t, const PfGeom &, const StepArgs &, const ResidentPlan &, int,
                                            uint32_t, double *, const double *, const double *, const uint32_t *,
                                            const uint32_t *,
                                            unsigned long long *, unsigned long long *, unsigned long long *,
                                            unsigned long long);
template hipError_t launch_resident<float>(hipStream_t, const PfGeom &, const StepArgs &, const ResidentPlan &, int,
                                           uint32_t, float *, const float *, const float *, const uint32_t *,
                                           const uint32_t *,
                                           unsigned long long *, unsigned long long *, unsigned long long *,
                                            unsigned long long);

template <typename T, int NS>
static void run_resident_setup(hipStream_t st, const PfGeom &g, const StepArgs &a, const ResidentPlan &pl, const T *PHI,
                               const double *phi, T *coef, uint32_t *mask, const uint32_t *first, bool fast) {
    const dim3 gr((unsigned)(pl.bx * pl.by * pl.bz)), b((unsigned)pl.threads);
    if (!first)
        hipLaunchKernelGGL((k_resident_setup<T, NS, true, false>), gr, b, 0, st, g, a, pl, PHI, phi, coef, mask, first);
    else if (fast)
        hipLaunchKernelGGL((k_resident_setup<T, NS, true, true>), gr, b, 0, st, g, a, pl, PHI, phi, coef, mask, first);
    else
        hipLaunchKernelGGL((k_resident_setup<T, NS, false, true>), gr, b, 0, st, g, a, pl, PHI, phi, coef, mask, first);
}
template <typename T>
void launch_resident_setup(hipStream_t st, const PfGeom &g, const StepArgs &a, const ResidentPlan &pl, const T *PHI,
                           const double *phi, T *coef, uint32_t *mask, const uint32_t *first, bool fast) {
    if (pl.ns == 1) run_resident_setup<T, 1>(st, g, a, pl, PHI, phi, coef, mask, first, fast);
    else if (pl.ns == 2) run_resident_setup<T, 2>(st, g, a, pl, PHI, phi, coef, mask, first, fast);
    else if (pl.ns == 4) run_resident_setup<T, 4>(st, g, a, pl, PHI, phi, coef, mask, first, fast);
    else if (pl.ns == 8) run_resident_setup<T, 8>(st, g, a, pl, PHI, phi, coef, mask, first, fast);
    else if constexpr (sizeof(T) == 4) run_resident_setup<T, 16>(st, g, a, pl, PHI, phi, coef, mask, first, fast);
}
template void launch_resident_setup<double>(hipStream_t, const PfGeom &, const StepArgs &, const ResidentPlan &,
                                            const double *, const double *, double *, uint32_t *, const uint32_t *,
                                            bool);
template void launch_resident_setup<float>(hipStream_t, const PfGeom &, const StepArgs &, const ResidentPlan &,
                                           const float *, const double *, float *, uint32_t *, const uint32_t *, bool);

// ------------------------------------------------------------------------------------
// 2D: a block owns R rows over the whole width and holds them with 2K rows on each side.
// It runs K iterations on its own, every half-sweep updating one row fewer on each side (the
// rows whose neighbours are still exact), then takes the 2K rows on each side from their
// owners again: an exchange, which costs as much as several half-sweeps of so few cells, is
// paid once in K iterations.  A message has four slots, by exchange: where n is no multiple of
// R, the last block reads one block further than reads it, so a writer may be three exchanges
// ahead of that reader; such a grid takes three rounds at least, so that its rows are written
// back in place only after every block has loaded them.  The rows wrap in y.  A grid that one block holds needs no
// exchange.  p lives in LDS by colour, a cell's right-hand side and coefficients in its
// thread's registers, Q cells of each colour a thread.
//
// With n odd row 1 and row n hold the same colours and each takes the other's value of
// before the half-sweep (the reference refreshes the ghost rows between half-sweeps): there
// every thread reads before any writes.  The first half-sweep of a launch takes the ghost
// rows as they are in memory.
//
// Measured, us per iteration, before / resident: 48x24 (one block, q = 2) 3.05 (two iterations
// a launch) / 0.89; 256x128 4.67 / 2.57 with K,R = 2,1 (q = 3), 2.88 with 1,1 (q = 2), 2.50
// with 3,1 (q = 4), 2.72 with 2,2; 511x255, odd in y, 16.1 (a launch per half-sweep and per
// refresh of the ghost rows) / 4.2 with 2,1 (q = 5), 4.6 with 1,1.  A half-sweep is FP64 issue
// (about 55 instructions a cell) and the latency of one LDS read, update, write and barrier.
// ------------------------------------------------------------------------------------
namespace {

constexpr int R2T = 512;      // threads of a block; 256 registers each
constexpr int R2Q = 5;        // cells of one colour per thread, at most

template <typename T>
struct Resident2 {
    PfGeom g;
    StepArgs a;
    Resident2Plan pl;
    int iters;
    uint32_t seq;      // exchange t carries seq + t
    T *X;
    const T *R, *PHI;
    const double *phi;
    u64 *inbox;
    u64 *slots;
    u64 *count, target;   // blocks that reached the end, over all launches: target with this one's
    unsigned polls;       // of a wait, at most
};

// A cell's coefficients and what its division needs.
template <typename T>
struct Cell2;
template <>
struct Cell2<double> {
    double ae, aw, an, as, ap, s, r;
    template <bool FAST>
    __device__ __forceinline__ void set(const PfGeom &g, const StepArgs &a, int i, int j, const double *PHI,
                                        const double *phi) {
        Coef c;
        ap = sor_coefs<2, FAST>(g, a, i, j, 0, PHI[pf_soff(g, i, j, 0)], PHI[pf_soff(g, i - 1, j, 0)],
                                PHI[pf_soff(g, i + 1, j, 0)], PHI[pf_soff(g, i, j - 1, 0)], PHI[pf_soff(g, i, j + 1, 0)],
                                0., 0., phi, c);
        ae = c.ae;
        aw = c.aw;
        an = c.an;
        as = c.as;
        // the divisor as divk_make scales and inverts it, per lane
        bool f;
        s = __builtin_amdgcn_div_scale(1.0, ap, false, &f);
        const double r0 = __builtin_amdgcn_rcp(s);
        const double r1 = __builtin_fma(r0, __builtin_fma(-s, r0, 1.0), r0);
        r = __builtin_fma(r1, __builtin_fma(-s, r1, 1.0), r1);
    }
    __device__ __forceinline__ double update(const StepArgs &a, double b, double pc, double pW, double pE, double pS,
                                             double pN) const {
        const double num = (((b - (ae * pE)) - (aw * pW)) - (an * pN)) - (as * pS);
        DivFast dv;
        double d = dv(num, DivK{ap, s, r});
        if (dv.slow) d = num / ap;
        return (d * a.omega) + (pc * a.omega_c);
    }
};
template <>
struct Cell2<float> {
    float ae, aw, an, as, rap;
    template <bool FAST>
    __device__ __forceinline__ void set(const PfGeom &g, const StepArgs &a, int i, int j, const float *PHI,
                                        const double *phi) {
        CoefT<float> c;
        float ap;
        sor32_coefs<2>(g, a, i, j, 0, PHI[pf_soff(g, i, j, 0)], PHI[pf_soff(g, i - 1, j, 0)],
                       PHI[pf_soff(g, i + 1, j, 0)], PHI[pf_soff(g, i, j - 1, 0)], PHI[pf_soff(g, i, j + 1, 0)], 0.f,
                       0.f, phi, (float)(a.dt / (a.dx * a.dx)), (float)(a.dt / (a.dy * a.dy)),
                       (float)(a.dt / (a.dz * a.dz)), c, ap);
        ae = c.ae;
        aw = c.aw;
        an = c.an;
        as = c.as;
        rap = __builtin_amdgcn_rcpf(ap);
    }
    __device__ __forceinline__ float update(const StepArgs &a, float b, float pc, float pW, float pE, float pS,
                                            float pN) const {
        const float om = (float)a.omega;
        const float num = b - ae * pE - aw * pW - an * pN - as * pS;
        return num * rap * om + pc * (1.f - om);
    }
};

}  // namespace

template <typename T, int Q, bool FAST, bool ODD>
__global__ __launch_bounds__(R2T) void k_sor_resident2(Resident2<T> x) {
    extern __shared__ __align__(16) char lds_raw[];
    T *L = (T *)lds_raw;   // [colour][local row][slot]
    __shared__ int dead_flag;
    const lds_int dead = (lds_int)&dead_flag;
    const PfGeom &g = x.g;
    const StepArgs &a = x.a;
    constexpr int B = Msg<T>::B;
    const int H = g.H, n = g.n, K = x.pl.K, R = x.pl.R, NR = x.pl.rows, N = NR * H, halo = x.pl.whole ? 0 : 2 * K;
    const int tid = (int)threadIdx.x;
    const int v0 = (int)blockIdx.x * R + 1 - halo;   // the row held in local row 0 (before wrapping)
    const int own = min(R, n - ((int)blockIdx.x * R));
    auto jrow = [=](int r) __attribute__((always_inline)) {
        const int v = v0 + r;
        return v < 1 ? v + n : v > n ? v - n : v;
    };
    if (tid == 0) *dead = 0;

    // p of the held rows, ghost columns among it
    for (int e = tid; e < 2 * N; e += R2T) {
        const int c = e >= N, f = e - c * N, r = f / H, h = f - r * H;
        L[e] = x.X[(int64_t)c * g.HS + pf_hoff(g, h, jrow(r), 0)];
    }
    // this thread's cells: place in a colour of L, distance from the held rows' edge (-1: no
    // cell), row wraps, right-hand side and coefficients
    int at[Q], depth[2][Q], south[2][Q], north[2][Q];
    bool own_row[Q], odd_row[Q];
    T b[2][Q];
    Cell2<T> k[2][Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int f = tid + q * R2T, r = f / H, h = f - r * H;
        at[q] = f;
        own_row[q] = r >= halo && r < halo + own;
        odd_row[q] = jrow(min(r, NR - 1)) & 1;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            depth[c][q] = -1;
            b[c][q] = T(0);
            south[c][q] = north[c][q] = 0;
            k[c][q] = Cell2<T>{};
            if (f >= N) continue;
            const int j = jrow(r), i = 2 * h + ((c + j) & 1);
            if (i < 1 || i > g.m) continue;
            depth[c][q] = x.pl.whole ? 2 * K : min(r, NR - 1 - r);
            b[c][q] = x.R[pf_soff(g, i, j, 0)];
            k[c][q].template set<FAST>(g, a, i, j, x.PHI, x.phi);
            // a neighbouring row's cell has the other colour, or this one across the wrap of an odd n
            const int rs = r > 0 ? r - 1 : NR - 1, rn = r < NR - 1 ? r + 1 : 0;
            south[c][q] = ((i + jrow(rs)) & 1) * N + rs * H + h;
            north[c][q] = ((i + jrow(rn)) & 1) * N + rn * H + h;
        }
    }
    const rsrc inbox = __builtin_amdgcn_make_buffer_rsrc(x.inbox, 0, (int)((uint32_t)(8 * n) * (uint32_t)H * B), 0x27000);
    double err = 0.;
    __syncthreads();

    const int rounds = (x.iters + K - 1) / K;
    for (int t = 0; t < rounds; ++t) {
        if (t > 0) {
            // exchange t - 1: the rows on each side, four messages in flight per thread
            const uint32_t seq = x.seq + (uint32_t)(t - 1);
            const int par = ((t - 1) & 3) * 2 * n * H * B, items = 2 * halo * H * 2;
            unsigned spin = 0;
            for (int e0 = 0; e0 < items; e0 += 4 * R2T) {
                uint32_t src[4];
                int dst[4];
                bool want[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int e = e0 + tid + u * R2T, lr = e / (2 * H), w = e - lr * (2 * H), c = w >= H, h = w - c * H;
                    const int r = lr < halo ? lr : lr + NR - 2 * halo;
                    const int j = jrow(r), i = 2 * h + ((c + j) & 1);
                    want[u] = e < items && i >= 1 && i <= g.m;
                    src[u] = want[u] ? (uint32_t)(((j - 1) * 2 + c) * H + h) * B : 0u;
                    dst[u] = c * N + r * H + h;
                }
                while (want[0] || want[1] || want[2] || want[3]) {
                    decltype(Msg<T>::get(inbox, 0u, 0)) m[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) m[u] = Msg<T>::get(inbox, src[u], par);
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (want[u] && Msg<T>::ok(m[u], seq)) {
                            L[dst[u]] = Msg<T>::value(m[u]);
                            want[u] = false;
                        }
                    if ((want[0] || want[1] || want[2] || want[3]) && give_up(spin, dead, x.count, x.polls)) break;
                }
            }
            __syncthreads();
        }
        const int its = min(K, x.iters - t * K);
        for (int it = 0; it < its; ++it) {
            auto half = [&](auto HT) __attribute__((always_inline)) {
                constexpr int half_no = decltype(HT)::value;
                auto with = [&](auto CT) __attribute__((always_inline)) {
                    constexpr int C = decltype(CT)::value;
                    const int lost = 2 * it + half_no + 1;   // rows of each side no longer exact
                    const bool ghosts = half_no == 0 && t == 0 && it == 0;
                    T pn[Q];
                    bool on[Q];
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        on[q] = depth[C][q] >= lost;
                        if (!on[q]) continue;
                        const int f = at[q], sh = odd_row[q] ? 1 - C : C;
                        const T *O = L + (1 - C) * N + f;
                        T pS = L[south[C][q]], pN = L[north[C][q]];
                        if (ghosts) {
                            const int r = f / H, j = jrow(r), i = 2 * (f - r * H) + sh;
                            if (j == 1) pS = x.X[pf_soff(g, i, 0, 0)];
                            if (j == n) pN = x.X[pf_soff(g, i, n + 1, 0)];
                        }
                        const T pc = L[C * N + f];
                        pn[q] = k[C][q].update(a, b[C][q], pc, O[sh - 1], O[sh], pS, pN);
                        if (own_row[q]) err = max_keep_nan(err, fabs((double)pn[q] - (double)pc));
                    }
                    if (ODD) __syncthreads();
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        if (on[q]) L[C * N + at[q]] = pn[q];
                    __syncthreads();
                };
                if (half_no == 0) with(std::integral_constant<int, 1>{});   // (i + j) odd first
                else with(std::integral_constant<int, 0>{});
            };
            half(std::integral_constant<int, 0>{});
            half(std::integral_constant<int, 1>{});
        }
        if (t + 1 < rounds && !x.pl.whole) {
            const uint32_t seq = x.seq + (uint32_t)t;
            const int par = (t & 3) * 2 * n * H * B;
            for (int e = tid; e < 2 * own * H; e += R2T) {
                const int lr = e / (2 * H), w = e - lr * (2 * H), c = w >= H, h = w - c * H, j = v0 + halo + lr;
                Msg<T>::send(inbox, (uint32_t)(((j - 1) * 2 + c) * H + h) * B, par, L[c * N + (halo + lr) * H + h], seq);
            }
        }
    }

    if (!x.pl.whole) {
        __syncthreads();
        if (tid == 0) *dead = commit(x.count, x.target, *dead != 0, x.polls) ? 0 : 1;
        __syncthreads();
        if (*dead) return;
    }

    // the owned rows and their periodic mirrors back to memory
    for (int e = tid; e < 2 * own * H; e += R2T) {
        const int lr = e / (2 * H), w = e - lr * (2 * H), c = w >= H, h = w - c * H, j = v0 + halo + lr;
        const int i = 2 * h + ((c + j) & 1);
        if (i < 1 || i > g.m) continue;
        const T v = L[c * N + (halo + lr) * H + h];
        x.X[pf_soff(g, i, j, 0)] = v;
        if (j == n) x.X[pf_soff(g, i, 0, 0)] = v;
        if (j == 1) x.X[pf_soff(g, i, n + 1, 0)] = v;
    }
    wave_max_to_slot(err, x.slots);
}

bool resident2_plan(const PfGeom &g, int bc, int iters, Resident2Plan &pl) {
    pl = Resident2Plan{};
    if (g.dim != 2 || bc != PF_BC_UNIFORM || g.n < 3 || iters < 2) return false;
    const char *e = std::getenv("PF_RESIDENT");
    int fk = 0, fr = 0;
    if (e && *e && std::sscanf(e, "%d,%d", &fk, &fr) != 2) return false;
    const int64_t H = g.H;
    if (8 * H * g.n * 16 >= ((int64_t)1 << 31)) return false;   // byte offsets into the inbox are 32-bit
    double best = 1e300;
    auto consider = [&](int K, int R, bool whole) {
        const int64_t rows = whole ? g.n : R + 4 * K, q = (rows * H + R2T - 1) / R2T;
        const int64_t blocks = whole ? 1 : (g.n + R - 1) / R;
        if (q > R2Q || blocks > RESIDENT_CUS || (!whole && rows > g.n)) return;
        if (!whole && (iters + K - 1) / K < (g.n % R ? 3 : 2)) return;
        // us of a half-sweep and of an exchange, from the figures above
        const double half = 0.22 + 0.19 * (double)q;
        const double cost = whole ? 2 * half : 2 * half + (1.6 + 0.0002 * (double)(8 * K * H)) / K;
        if (cost < best) {
            best = cost;
            pl = Resident2Plan{whole ? iters : K, whole ? g.n : R, (int)rows, (int)q, (int)blocks, whole ? 1 : 0};
        }
    };
    if (fk > 0 && fr > 0) {
        consider(std::min(fk, iters / 2), fr, fr >= g.n);
    } else {
        consider(1, g.n, true);
        const int r0 = (g.n + RESIDENT_CUS - 1) / RESIDENT_CUS;
        for (int R = r0; R < r0 + 8; ++R)
            for (int K = 1; K <= std::min(8, iters / 2); ++K) consider(K, R, false);
    }
    return pl.blocks > 0;
}
int64_t resident2_inbox_words(const PfGeom &g, int elem) { return (int64_t)8 * g.n * g.H * (elem == 8 ? 2 : 1); }

template <typename T, int Q, bool FAST>
static hipError_t run_resident2(hipStream_t st, Resident2<T> &r) {
    const size_t lds = (size_t)2 * r.pl.rows * r.g.H * sizeof(T);
    const void *f = (r.g.n & 1) ? (const void *)k_sor_resident2<T, Q, FAST, true> : (const void *)k_sor_resident2<T, Q, FAST, false>;
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    void *args[] = {&r};
    return hipLaunchKernel(f, dim3((unsigned)r.pl.blocks), dim3(R2T), args, lds, st);
}

template <typename T>
hipError_t launch_resident2(hipStream_t st, const PfGeom &g, const StepArgs &a, const Resident2Plan &pl, int iters,
                            uint32_t seq, T *X, const T *R, const T *PHI, const double *phi, bool fast,
                            unsigned long long *inbox, unsigned long long *slots, unsigned long long *count,
                            unsigned long long target) {
    Resident2<T> r{g, a, pl, iters, seq, X, R, PHI, phi, inbox, slots, count, target, resident_polls()};
#define PF_R2(QQ)                                                                      \
    case QQ:                                                                           \
        return fast ? run_resident2<T, QQ, true>(st, r) : run_resident2<T, QQ, false>(st, r);
    switch (pl.q) {
        PF_R2(1)
        PF_R2(2)
        PF_R2(3)
        PF_R2(4)
        PF_R2(5)
        default: return hipErrorInvalidValue;
    }
#undef PF_R2
}
template hipError_t launch_resident2<double>(hipStream_t, const PfGeom &, const StepArgs &, const Resident2Plan &, int,
                                             uint32_t, double *, const double *, const double *, const double *, bool,
                                             unsigned long long *, unsigned long long *, unsigned long long *,
                                            unsigned long long);
template hipError_t launch_resident2<float>(hipStream_t, const PfGeom &, const StepArgs &, const Resident2Plan &, int,
                                            uint32_t, float *, const float *, const float *, const double *, bool,
                                            unsigned long long *, unsigned long long *, unsigned long long *,
                                            unsigned long long);

}  // namespace pf
