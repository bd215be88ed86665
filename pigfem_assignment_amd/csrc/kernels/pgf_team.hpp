// Jacobi-PCG in one cooperative launch: teams of blocks that stay resident
// and iterate together.
//
// What bounds it: a PCG iteration is two sums over the whole system (p.q, then
// r.z and r.r) around one pass over K.  As separate kernels that is five
// launches of 2.4-6 us each, which is the whole iteration for systems whose K
// fits the caches.  Here a team of blocks (all of the launch for one system)
// iterates by itself:
//
//  * a sum over the team costs one exchange through memory: every block
//    publishes its partial sums in its own slot, one wavefront of every block
//    reads all slots until none is empty and adds them in slot order, so every
//    block has the same total and takes the same decisions.  No
//    read-modify-write: a single arrival counter costs ~60 ns per block on one
//    line (15 us at 256 blocks); this exchange takes 1.6 us with 79 blocks, 2.1
//    to 2.7 with 240.
//  * "empty" is a NaN pattern no sum is published as.  Slots rotate over three
//    buffers: a block empties its slot of the buffer after next right after it
//    has read a sum, when every block has left the sum that last used it.
//  * the search direction is formed where it is used: each row publishes
//    (z, p_old) as one 16-byte pair, and whoever needs that column computes
//    p = z + beta p_old, so p needs no exchange of its own and an iteration
//    has two.
//  * a block keeps p of every column its rows touch in LDS (its window: its
//    own rows, then the other blocks' columns, its halo) and finds it by a
//    16-bit window index, so a product's gathers are LDS reads and the halo is
//    read from memory once per iteration.
//  * the pairs are the only data blocks read from each other.  They are
//    written through to memory and read past the caches of the reading die
//    (device-scope cache policy on the accesses themselves): a release and an
//    acquire fence of the agent instead, which write back and drop the die's
//    whole L2, take 4.5 us with 32 blocks per die, and K leaves the L2.
//  * K entries and window indices of a block stay in registers where they all
//    fit (KEEP steps a lane); otherwise they are streamed, the loads one
//    or two steps ahead of the products.
//  * the steps of a block's lane groups are laid out on the host: rows longer
//    than a step take consecutive steps of one lane group, so no lane waits in
//    a loop over a neighbour's long row, and every block has about as many.
//
// Every wait ends: a block leaves that has waited for one sum longer than
// WAIT_TICKS, and raises the abort flag, by which the host reports a device
// error.  No block looks at the flag: the others of its team, which are at the
// same sum or the next, run into the limit by themselves.  The launch is
// cooperative, so all blocks are resident.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

#include "../host/pgf_team.hpp"

namespace pgft {

constexpr int TT = TEAM_THREADS;                  // 512: 256 registers a lane for K entries
constexpr int MAX_TEAM = 256;                     // blocks per team (one pass of loads for one or two values)
constexpr unsigned long long EMPTY = ~0ull;       // slot not yet published
constexpr unsigned long long WAIT_TICKS = 2000000000ull;  // 20 s of the 100 MHz wall clock
constexpr size_t LDS_MAX = 158 * 1024;            // dynamic LDS a block may take (160 KiB less the static part)
constexpr int MAX_WINDOW = 65536;                 // 16-bit window indices

// per (system, right-hand side) state between launches and result
enum { T_RZ = 0, T_BETA, T_RR, T_RR0, T_TOL, T_IT, T_DONE, T_N = 8 };

// Where a block's vectors live.  WIN_ALL: window p, and r, q, 1/diag of its
// rows in LDS.  WIN_PQ: window p and q in LDS, r and 1/diag in memory.
enum Tier { WIN_ALL = 0, WIN_PQ = 1 };

template <typename TA>
struct TeamArgs {
    int n_teams, team_blocks;
    const int32_t* team_sys;  // [n_teams + 1] range of each team in sys_list
    const int32_t* sys_list;  // systems in the order their team solves them
    int* team_pos;            // [n_teams][2] next entry of the list, 1 if that system is under way
    const int32_t* row_ptr;   // [n_sys][team_blocks + 1] first row of each block
    const int64_t* step_ptr;  // [n_sys * team_blocks + 1]
    const StepRec* steps;
    const uint16_t* wcol;     // window index of each entry (first row of every group)
    const int64_t* halo_ptr;  // [n_sys * team_blocks + 1]
    const int32_t* halo;      // columns of each block's halo
    const int32_t* diag;      // entry of each row's diagonal, -1 without one
    const TA* A;
    int64_t ld;               // stride of the right-hand sides in b, x, r and zp
    const double* b;          // [NR][ld]
    const double* Ax;         // K x0 for a nonzero start (x then holds x0), or null
    double *x, *r, *dinv;     // [NR][ld] ([n] for dinv)
    double2* zp;              // [NR][ld] published (z, p): a wavefront stores whole lines
    int64_t zp_bytes;
    double* state;            // [n_sys][NR][T_N], systems in the order of their shares
    unsigned long long* slots;  // [n_teams][COPIES][team_slots]
    int* abort;
    double tol2;              // squared relative tolerance
    int maxit, launch_its;    // iterations per system, and per team in this launch
    int single;               // stopping rules of the single solve (see below)
};

template <int NR>
constexpr int slot_values() { return NR == 1 ? 3 : 2 * NR; }

// Every slot is published in COPIES places, one for the readers of each die,
// and has 64 bytes of its own: 256 wavefronts polling the same few lines wait
// on each other, and so do blocks that write one line.  One sum with 160 to
// 256 blocks: 2.8-3.3 us in one copy of packed slots (1.8 where the lines
// happened to lie well), 2.0-2.6 so; 2 to 32 copies and 128-byte slots are
// within 5 % of this.
constexpr int COPIES = 8, SLOT = 8;
static_assert(slot_values<4>() <= SLOT, "a slot holds every sum");
__host__ __device__ constexpr int64_t team_slots(int nb) {  // one copy: three buffers, on pages of its own
    return ((int64_t)3 * nb * SLOT + 511) / 512 * 512;
}

// ---- device-scope accesses of the pairs: SC1 on a buffer access (bit 4)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int SC1 = 16;
__device__ inline double2 pair_load(__amdgpu_buffer_rsrc_t rs, uint32_t i) {
    union { u32x4 u; double2 d; } v;
    v.u = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(i * 16u), 0, SC1);
    return v.d;
}
__device__ inline void pair_store(__amdgpu_buffer_rsrc_t rs, uint32_t i, double2 d) {
    union { u32x4 u; double2 d; } v;
    v.d = d;
    __builtin_amdgcn_raw_buffer_store_b128(v.u, rs, (int)(i * 16u), 0, SC1);
}

__device__ inline unsigned long long slot_load(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void slot_store(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- sums over lanes without LDS.  By data-parallel primitives: lanes ^1,
// ^2, 7 - i, 15 - i of a row of 16 (every lane gets the sum), ^4, ^8; by
// exchange of rows and halves: 16 and 32 apart.
template <int CTRL>
__device__ inline double dpp(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int G>
__device__ inline double lane_sum(double v) {
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    if (G >= 8) v += dpp<0x141>(v);
    if (G >= 16) v += dpp<0x140>(v);
    return v;
}
__device__ inline double xor4(double v) { return dpp<0x1B>(dpp<0x141>(v)); }
__device__ inline double xor8(double v) { return dpp<0x128>(v); }
// even rows (halves) get the sum of a, odd ones that of b, over the two
template <int APART>
__device__ inline double swap_add(double a, double b) {
    const unsigned long long ua = __double_as_longlong(a), ub = __double_as_longlong(b);
    auto swap = [](unsigned x, unsigned y) {
        if constexpr (APART == 16) return __builtin_amdgcn_permlane16_swap(x, y, false, false);
        else return __builtin_amdgcn_permlane32_swap(x, y, false, false);
    };
    const auto lo = swap((unsigned)ua, (unsigned)ub), hi = swap((unsigned)(ua >> 32), (unsigned)(ub >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}
constexpr int padded(int nv) { return nv <= 2 ? nv : nv <= 4 ? 4 : 8; }
// sums of v[0..NV) over the wavefront: every lane gets that of value
// lane / (64 / padded(NV)).  Each exchange halves the values a lane carries:
// 10 additions for 6 values, not 36, and no step through LDS (333 x 333 quads
// 9.3 -> 8.3 us per iteration, 64^3 x 6 tets 96 -> 94.7, with the loads below).
template <int NV>
__device__ inline double wave_sums(const double (&v)[NV]) {
    constexpr int VP = padded(NV);
    double w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = k < NV ? v[k] : 0.0;
    if (VP == 8)
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = swap_add<32>(w[k], w[k + 4]);
    else if (VP == 4)
#pragma unroll
        for (int k = 0; k < 2; ++k) w[k] = swap_add<32>(w[k], w[k + 2]);
    else
        w[0] = swap_add<32>(w[0], w[VP - 1]);
    if (VP == 8)
#pragma unroll
        for (int k = 0; k < 2; ++k) w[k] = swap_add<16>(w[k], w[k + 2]);
    else
        w[0] = swap_add<16>(w[0], w[VP == 4 ? 1 : 0]);
    if (VP == 8) {
        const bool odd = threadIdx.x & 8;
        w[0] = (odd ? w[1] : w[0]) + xor8(odd ? w[0] : w[1]);
    } else {
        w[0] += xor8(w[0]);
    }
    return lane_sum<8>(w[0]);
}

// a value all lanes agree on, in scalar registers
__device__ inline double uniform(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)u), hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// One block's end of the team's sums.
template <int NR>
struct TeamSum {
    static constexpr int TW = TT / 64;
    static_assert(TW == 8 && COPIES == 8 && SLOT == 8, "eight lanes add the wavefronts, publish and empty a value");
    unsigned long long* slots;  // this team's [COPIES][3][nb][SLOT]
    int nb, me, copy;
    unsigned phase;
    double (*red)[SLOT];        // [TW][SLOT] LDS
    double* tot;                // [SLOT] LDS
    int* bad;                   // LDS: the team gave up
    int* abort;

    // Sums v[0..NV) over the team; returns false if a wait ran out.  publish:
    // other blocks read pairs this block stored before.  Wavefronts other than
    // the first run `meanwhile`.
    template <int NV, typename F>
    __device__ bool operator()(double (&v)[NV], bool publish, F&& meanwhile) {
        constexpr int L = 64 / padded(NV);  // lanes a value has
        int lane = threadIdx.x & 63;
        // (kept out of the compiler's sight, which otherwise computes every
        // address below before the iteration and spills K entries for it)
        asm volatile("" : "+v"(lane));
        const int w = threadIdx.x >> 6, k = lane / L, j = lane % L;
        const double mine = wave_sums<NV>(v);
        if (j == 0 && k < NV) red[w][k] = mine;
        // every wavefront's pairs have left it before the publication
        if (publish) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (w == 0) {
            // of the block, in the first eight lanes of each value
            const double s = lane_sum<8>(j < TW && k < NV ? red[j][k] : 0.0);
            if (nb > 1) exchange<NV>(s, lane);
            else if (j == 0 && k < NV) tot[k] = s;
        } else {
            meanwhile();
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = uniform(tot[i]);
        return __builtin_amdgcn_readfirstlane(*bad) == 0;
    }

    // One store publishes every value in every copy, and the lanes of a load
    // read whole slots: with a load per value and 64 slots each, the sum of six
    // values over 42 blocks took 4.1 us and that of three 2.9 (six systems of 3
    // right-hand sides 11.2 -> 8.6 us per iteration, 32 larger ones 75.6 -> 63.6).
    template <int NV>
    __device__ void exchange(double s, int lane) {
        constexpr int VP = padded(NV), L = 64 / VP;
        constexpr int LOADS = std::min(MAX_TEAM / L, NR == 1 ? 8 : 16);  // at a time
        const int64_t per = team_slots(nb), at = (int64_t)(phase % 3) * nb * SLOT;
        const unsigned long long* buf = slots + copy * per + at;
        // the emptied slot of the next buffer is in memory before this
        // publication, after which another block may look for it
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane % L < COPIES && lane / L < NV) {
            unsigned long long u = __double_as_longlong(s);
            if (u == EMPTY) u = 0x7ff8000000000000ull;
            slot_store(&slots[lane % L * per + at + (int64_t)me * SLOT + lane / L], u);
        }
        // value lane % VP of blocks lane / VP, + L, ...
        const int k = lane % VP;
        const uint32_t mine = lane / VP * SLOT + k;
        double sum = 0.0;
        const unsigned long long t0 = wall_clock64();
        for (int m0 = 0; m0 < nb; m0 += LOADS * L) {
            unsigned long long got[LOADS];
            for (unsigned round = 0;; ++round) {
                bool all = true;
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    got[i] = 0ull;
                    const int m = m0 + i * L;  // (of the wavefront)
                    if (m < nb && m + lane / VP < nb && k < NV) got[i] = slot_load(buf + m * SLOT + mine);
                }
#pragma unroll
                for (int i = 0; i < LOADS; ++i) all = all && got[i] != EMPTY;
                if (__all(all)) break;
                if ((round & 255u) == 255u && wall_clock64() - t0 > WAIT_TICKS) {
                    if (lane == 0) {
                        *bad = 1;
                        __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    break;
                }
            }
#pragma unroll
            for (int i = 0; i < LOADS; ++i) sum += __longlong_as_double((long long)got[i]);
        }
        // nothing after this is read before the slots were
        asm volatile("" ::: "memory");
        if (VP == 1) sum += dpp<0xB1>(sum);
        if (VP <= 2) sum += dpp<0x4E>(sum);
        if (VP <= 4) sum += xor4(sum);
        sum += xor8(sum);
        sum = swap_add<16>(sum, sum);
        sum = swap_add<32>(sum, sum);
        if (lane < NV) tot[lane] = sum;
        // all values of this block's next slot but one, in all copies
        slot_store(&slots[lane / SLOT * per + ((int64_t)((phase + 2) % 3) * nb + me) * SLOT + lane % SLOT], EMPTY);
        ++phase;
    }
};

// One step of a lane group: U columns per lane (window indices in pairs), their
// entries in the group's rows.  The sums over the lanes are most of a product's
// instructions and cost lanes times steps, so a 2D group has 4 lanes with 5
// columns each, not 8 with 3 (333 x 333 quads: products 2.1 -> 1.2 us, 10.4 ->
// 9.2 us per iteration).  In 3D 16 lanes with 3 columns stay: 8 with 6 take 111
// us on 64^3 x 6 tets against 97 (coarser steps to stream and to balance).
template <typename TA, int DIM>
struct Step {
    static constexpr int U = team_cols(DIM);
    uint32_t c[(U + 1) / 2];
    TA v[DIM][U];
    __device__ int col(int u) const { return (int)(u & 1 ? c[u / 2] >> 16 : c[u / 2] & 0xffffu); }
};

template <typename TA, int NR, int DIM, int TIER, int KEEP>
__global__ __launch_bounds__(TT) void k_team_pcg(TeamArgs<TA> a) {
    constexpr int G = team_lanes(DIM), GP = TT / G, U = team_cols(DIM);
    constexpr bool ALL = TIER == WIN_ALL;
    constexpr int RB = ALL ? 1 : 4;  // rows per trip: operands in memory want several on the way
    constexpr int W = slot_values<NR>();
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ double s_red[TT / 64][SLOT], s_tot[SLOT];
    __shared__ int s_bad;
    const int t = threadIdx.x, sub = t % G;
    int team = blockIdx.x % a.n_teams, me = blockIdx.x / a.n_teams;
    // blocks go round-robin to the dies (XCDs): neighbouring shares of one
    // system on one die, so the entries they both read sit in one L2
    if (a.n_teams == 1 && a.team_blocks % 8 == 0) me = (blockIdx.x % 8) * (a.team_blocks / 8) + blockIdx.x / 8;
    TeamSum<NR> sum{a.slots + team * COPIES * team_slots(a.team_blocks), a.team_blocks, me,
                    (int)(blockIdx.x % COPIES), 0u, s_red, s_tot, &s_bad, a.abort};
    if (t == 0) s_bad = 0;
    __syncthreads();
    const __amdgpu_buffer_rsrc_t zrs =
        __builtin_amdgcn_make_buffer_rsrc(a.zp, (short)0, (int)(uint32_t)a.zp_bytes, 0x00027000);
    int pos = a.team_pos[2 * team], left = a.launch_its;
    bool resume = a.team_pos[2 * team + 1] != 0;
    const int end = a.team_sys[team + 1];
    while (pos < end && left > 0) {
        const int sys = a.sys_list[pos];
        const size_t share = (size_t)sys * a.team_blocks + me;
        const int32_t* rp = a.row_ptr + (size_t)sys * (a.team_blocks + 1) + me;
        const int row0 = rp[0], nrow = rp[1] - row0;
        const StepRec* steps = a.steps + a.step_ptr[share] * GP + t / G;  // this lane group's, GP apart
        const int ns = (int)(a.step_ptr[share + 1] - a.step_ptr[share]);
        const int64_t h0 = a.halo_ptr[share];
        const int nh = (int)(a.halo_ptr[share + 1] - h0);
        const int nw = nrow + nh;
        // LDS: p of the window by right-hand side [NR][nw], then q (z from the
        // update on) and r [NR][nrow], 1/diag [nrow]; the halo's columns [nh]
        // where K is in registers
        double* Lp = (double*)s_dyn;
        double* Lq = Lp + (size_t)nw * NR;
        double* Lr = Lq + (size_t)nrow * NR;
        double* Ld = Lr + (size_t)nrow * NR;
        uint32_t* Lh = (uint32_t*)(Ld + nrow);
        if (KEEP > 0) {
            for (int i = t; i < nh; i += TT) Lh[i] = (uint32_t)a.halo[h0 + i];
            __syncthreads();
        }
        double* xg = a.x + row0;
        double* rg = a.r + row0;
        const double2* zg = a.zp + row0;
        const double* dg = a.dinv + row0;
        double* st = a.state + (size_t)sys * NR * T_N;
        double rz[NR], beta[NR], rr[NR], rr0[NR], tol[NR];
        bool act[NR];
        int it[NR];
        auto store_pair = [&](int i, int c, double z, double p) {
            pair_store(zrs, (uint32_t)(c * a.ld + row0 + i), double2{z, p});
        };
        // (unconditional loads at clamped places, zeroed afterwards: a load
        // under a condition is a branch the next one waits behind)
        auto load_step = [&](const StepRec& r, Step<TA, DIM>& s) {
            const int k = (r.what >> 8) & 3, len = r.what & 255;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = sub + u * G;
                const int e = r.begin + min(j, max(len - 1, 0));
                const uint32_t w = a.wcol[e];
                if (u & 1) s.c[u / 2] |= (len > 0 ? w : 0u) << 16;
                else s.c[u / 2] = len > 0 ? w : 0u;
#pragma unroll
                for (int h = 0; h < DIM; ++h) s.v[h][u] = a.A[e + (h < k ? h : 0) * r.stride];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < DIM; ++h) s.v[h][u] = sub + u * G < len && h < k ? s.v[h][u] : (TA)0;
        };
        // row in the share << 4, first and last step, rows of the group
        auto info_of = [](const StepRec& r) {
            return r.row << 4 | (r.what & STEP_CONT ? 8 : 0) | (r.what & STEP_LAST ? 4 : 0) | ((r.what >> 8) & 3);
        };
        if (resume) {
            for (int i = t; i < nrow; i += TT) {
                if (ALL) Ld[i] = dg[i];
                for (int c = 0; c < NR; ++c) {
                    if (ALL) Lr[c * nrow + i] = rg[c * a.ld + i];
                    Lp[c * nw + i] = zg[c * a.ld + i].y;
                    Lq[c * nrow + i] = zg[c * a.ld + i].x;
                }
            }
            for (int c = 0; c < NR; ++c) {
                rz[c] = uniform(st[c * T_N + T_RZ]);
                beta[c] = uniform(st[c * T_N + T_BETA]);
                rr[c] = uniform(st[c * T_N + T_RR]);
                rr0[c] = uniform(st[c * T_N + T_RR0]);
                tol[c] = uniform(st[c * T_N + T_TOL]);
                it[c] = __builtin_amdgcn_readfirstlane((int)st[c * T_N + T_IT]);
                act[c] = uniform(st[c * T_N + T_DONE]) == 0.0;
            }
        } else {
            double v[W];
            for (int k = 0; k < W; ++k) v[k] = 0.0;
            for (int i = t; i < nrow; i += TT) {
                const int32_t dgi = a.diag[row0 + i];
                const double d = dgi >= 0 ? (double)a.A[dgi] : 0.0;
                const double di = d != 0.0 ? 1.0 / d : (a.single ? 1.0 : 0.0);
                a.dinv[row0 + i] = di;
                if (ALL) Ld[i] = di;
                for (int c = 0; c < NR; ++c) {
                    const int64_t e = c * a.ld + row0 + i;
                    const double bi = a.b[e], ri = a.Ax ? bi - a.Ax[e] : bi;
                    const double zi = di * ri;
                    if (!a.Ax) a.x[e] = 0.0;
                    if (ALL) Lr[c * nrow + i] = ri;
                    else a.r[e] = ri;
                    Lp[c * nw + i] = 0.0;
                    Lq[c * nrow + i] = zi;
                    store_pair(i, c, zi, 0.0);
                    v[c] += ri * zi;
                    v[NR + c] += ri * ri;
                    if (NR == 1) v[W - 1] += bi * bi;
                }
            }
            if (!sum(v, true, [] {})) return;
            for (int c = 0; c < NR; ++c) {
                rz[c] = v[c];
                rr[c] = v[NR + c];
                // the single solve is relative to ||b||, also from a nonzero start
                rr0[c] = NR == 1 && a.single ? v[W - 1] : rr[c];
                tol[c] = uniform(a.tol2 * rr0[c]);
                beta[c] = 0.0;
                it[c] = 0;
                act[c] = a.single ? (rr[c] > tol[c] && a.maxit > 0) : rr[c] != 0.0;
            }
        }
        bool any = false;
        for (int c = 0; c < NR; ++c) any = any || act[c];
        // K entries that stay in registers: every step (KEEP), or the first
        // AHEAD
        constexpr int AHEAD = DIM == 3 ? 2 : 1;  // steps on the way while streaming
        constexpr int NK = KEEP > 0 ? KEEP : AHEAD;
        Step<TA, DIM> keep[NK];
        int info[NK];
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            StepRec r = {0, 0, 0, 0};
            if (s < ns) r = steps[s * GP];
            info[s] = info_of(r);
            load_step(r, keep[s]);
        }
        StepRec rec1 = {0, 0, 0, 0};
        if (KEEP == 0 && ns > AHEAD) rec1 = steps[AHEAD * GP];
        while (any && left > 0) {
            // ---- p of the window
            // (every loop over rows or columns issues the loads of several
            // trips before it uses the first)
            constexpr int HB = NR == 1 ? 8 : 8 / NR;
            for (int i0 = t; i0 < nh; i0 += HB * TT) {
                uint32_t col[HB];
                double2 e[HB][NR];
#pragma unroll
                for (int k = 0; k < HB; ++k) {
                    const int i = min(i0 + k * TT, nh - 1);
                    col[k] = KEEP > 0 ? Lh[i] : (uint32_t)a.halo[h0 + i];
                }
#pragma unroll
                for (int k = 0; k < HB; ++k)
#pragma unroll
                    for (int c = 0; c < NR; ++c) e[k][c] = pair_load(zrs, (uint32_t)(c * a.ld) + col[k]);
#pragma unroll
                for (int k = 0; k < HB; ++k)
                    if (i0 + k * TT < nh)
#pragma unroll
                        for (int c = 0; c < NR; ++c)
                            Lp[c * nw + nrow + i0 + k * TT] = e[k][c].x + beta[c] * e[k][c].y;
            }
            for (int i = t; i < nrow; i += TT)
#pragma unroll
                for (int c = 0; c < NR; ++c) Lp[c * nw + i] = Lq[c * nrow + i] + beta[c] * Lp[c * nw + i];
            __syncthreads();
            // ---- q = K p, p.q: G lanes per group of rows with one column list
            double pq[NR];
            for (int c = 0; c < NR; ++c) pq[c] = 0.0;
            auto add = [&](const Step<TA, DIM>& s, double (&acc)[DIM][NR]) {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int c = 0; c < NR; ++c) {
                        const double p = Lp[c * nw + s.col(u)];
#pragma unroll
                        for (int h = 0; h < DIM; ++h) acc[h][c] += (double)s.v[h][u] * p;
                    }
            };
            double acc[DIM][NR];
            auto step = [&](const Step<TA, DIM>& s, int what) {
                if (!(what & 8))
#pragma unroll
                    for (int h = 0; h < DIM; ++h)
#pragma unroll
                        for (int c = 0; c < NR; ++c) acc[h][c] = 0.0;
                add(s, acc);
                if (!(what & 4)) return;  // uniform over the lane group
                const int k = what & 3, i = (what >> 4) + sub;
#pragma unroll
                for (int c = 0; c < NR; ++c) {
#pragma unroll
                    for (int h = 0; h < DIM; ++h) acc[h][c] = lane_sum<G>(acc[h][c]);
                    if (sub < k) {
                        double qi = acc[0][c];
                        if (sub == 1) qi = acc[1][c];
                        if (DIM == 3 && sub == 2) qi = acc[DIM - 1][c];
                        Lq[c * nrow + i] = qi;
                        pq[c] += Lp[c * nw + i] * qi;
                    }
                }
            };
            if (KEEP > 0) {
#pragma unroll
                for (int s = 0; s < NK; ++s)
                    if (s < ns) {
                        // FP32 entries stay FP32 in their registers: without
                        // this the compiler widens them once before the loop
                        if (sizeof(TA) == 4)
#pragma unroll
                            for (int h = 0; h < DIM; ++h)
#pragma unroll
                                for (int u = 0; u < U; ++u) asm volatile("" : "+v"(keep[s].v[h][u]));
                        step(keep[s], info[s]);
                    }
            } else {
                // one step's entries in use, AHEAD steps' on the way
                Step<TA, DIM> cur[AHEAD + 1];
                int ci[AHEAD + 1];
#pragma unroll
                for (int k = 0; k < AHEAD; ++k) {
                    cur[k] = keep[k];
                    ci[k] = info[k];
                }
                StepRec rn = rec1;
                for (int s = 0; s < ns; ++s) {
                    if (s + AHEAD < ns) {
                        ci[AHEAD] = info_of(rn);
                        load_step(rn, cur[AHEAD]);
                        if (s + AHEAD + 1 < ns) rn = steps[(size_t)(s + AHEAD + 1) * GP];
                    }
                    step(cur[0], ci[0]);
#pragma unroll
                    for (int k = 0; k < AHEAD; ++k) {
                        cur[k] = cur[k + 1];
                        ci[k] = ci[k + 1];
                    }
                }
            }
            if (!sum(pq, false, [] {})) return;
            double alpha[NR];
            for (int c = 0; c < NR; ++c) {
                alpha[c] = uniform(pq[c] != 0.0 && !(a.single && !isfinite(pq[c])) ? rz[c] / pq[c] : 0.0);
                if (!act[c]) alpha[c] = 0.0;
            }
            // ---- r -= alpha q, z = r / diag, the pair (z, p); r.z and r.r
            double v[2 * NR];
            for (int k = 0; k < 2 * NR; ++k) v[k] = 0.0;
            for (int i0 = t; i0 < nrow; i0 += RB * TT) {
                double di[RB], ri[RB][NR], qi[RB][NR], pi[RB][NR];
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    const int i = min(i0 + k * TT, nrow - 1);
                    di[k] = ALL ? Ld[i] : dg[i];
#pragma unroll
                    for (int c = 0; c < NR; ++c) {
                        ri[k][c] = ALL ? Lr[c * nrow + i] : rg[c * a.ld + i];
                        qi[k][c] = Lq[c * nrow + i];
                        pi[k][c] = Lp[c * nw + i];
                    }
                }
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    const int i = i0 + k * TT;
                    if (i >= nrow) continue;
#pragma unroll
                    for (int c = 0; c < NR; ++c) {
                        if (NR > 1 && !act[c]) {  // q back to z, which p is
                            Lq[c * nrow + i] = pi[k][c];
                            continue;
                        }
                        const double rn = ri[k][c] - alpha[c] * qi[k][c];
                        const double zi = di[k] * rn;
                        if (ALL) Lr[c * nrow + i] = rn;
                        else rg[c * a.ld + i] = rn;
                        store_pair(i, c, zi, pi[k][c]);
                        Lq[c * nrow + i] = zi;
                        v[c] += rn * zi;
                        v[NR + c] += rn * rn;
                    }
                }
            }
            // x += alpha p by the wavefronts that do not wait
            auto upx = [&] {
                constexpr int XT = TT - 64, XB = 4;
                for (int i0 = t - 64; i0 < nrow; i0 += XB * XT) {
                    double xo[XB][NR];
#pragma unroll
                    for (int k = 0; k < XB; ++k)
#pragma unroll
                        for (int c = 0; c < NR; ++c) xo[k][c] = xg[c * a.ld + min(i0 + k * XT, nrow - 1)];
#pragma unroll
                    for (int k = 0; k < XB; ++k) {
                        const int i = i0 + k * XT;
                        if (i >= nrow) continue;
#pragma unroll
                        for (int c = 0; c < NR; ++c)
                            if (act[c])
                                xg[c * a.ld + i] =
                                    xo[k][c] + alpha[c] * Lp[c * nw + i];
                    }
                }
            };
            if (!sum(v, true, upx)) return;
            any = false;
            for (int c = 0; c < NR; ++c) {
                if (!act[c]) continue;
                beta[c] = uniform(rz[c] != 0.0 ? v[c] / rz[c] : 0.0);
                rz[c] = v[c];
                rr[c] = v[NR + c];
                ++it[c];
                if (!(rr[c] > tol[c]) || it[c] >= a.maxit || (a.single && !isfinite(rr[c]))) {
                    act[c] = false;
                    // while other right-hand sides run, its p is the last z, of the
                    // rows and of the halo alike
                    if (NR > 1) beta[c] = 0.0;
                }
                any = any || act[c];
            }
            --left;
        }
        if (ALL && (any || a.single))  // to be resumed
            for (int i = t; i < nrow; i += TT)
                for (int c = 0; c < NR; ++c) rg[c * a.ld + i] = Lr[c * nrow + i];
        if (me == 0 && t == 0)
            for (int c = 0; c < NR; ++c) {
                st[c * T_N + T_RZ] = rz[c];
                st[c * T_N + T_BETA] = beta[c];
                st[c * T_N + T_RR] = rr[c];
                st[c * T_N + T_RR0] = rr0[c];
                st[c * T_N + T_TOL] = tol[c];
                st[c * T_N + T_IT] = it[c];
                st[c * T_N + T_DONE] = act[c] ? 0.0 : 1.0;
            }
        resume = any;
        if (any) break;
        ++pos;
        __syncthreads();  // the LDS arrays change hands
    }
    if (me == 0 && t == 0) {
        a.team_pos[2 * team] = pos;
        a.team_pos[2 * team + 1] = resume ? 1 : 0;
    }
}

// Window indices of every group's columns (entries of its first row): own
// rows first, then the place in the block's sorted halo.
static __global__ __launch_bounds__(256) void k_team_cols(int n_shares, int team_blocks, const int32_t* __restrict__ part,
                                                   const GroupRec* __restrict__ grp, const int32_t* __restrict__ col,
                                                   const int64_t* __restrict__ halo_ptr,
                                                   const int32_t* __restrict__ halo, uint16_t* __restrict__ wcol) {
    const int share = blockIdx.x;
    if (share >= n_shares) return;
    const int32_t* pt = part + (size_t)(share / team_blocks) * (team_blocks + 1) + share % team_blocks;
    const int g0 = pt[0], g1 = pt[1];
    const int row0 = grp[g0].row, nrow = grp[g1].row - row0;
    const int32_t* h = halo + halo_ptr[share];
    const int nh = (int)(halo_ptr[share + 1] - halo_ptr[share]);
    for (int g = g0 + (int)threadIdx.x / 8; g < g1; g += 32) {
        const GroupRec gr = grp[g];
        for (int j = threadIdx.x % 8; j < gr.len_k >> 2; j += 8) {
            const int c = col[gr.begin + j];
            int w = c - row0;
            if (w < 0 || w >= nrow) {
                int lo = 0, hi = nh;  // first halo entry >= c
                while (lo < hi) {
                    const int m = (lo + hi) >> 1;
                    if (h[m] < c) lo = m + 1;
                    else hi = m;
                }
                w = nrow + lo;
            }
            wcol[gr.begin + j] = (uint16_t)w;
        }
    }
}

// Passes a lane can keep in its registers.
template <typename TA, int NR, int DIM>
constexpr int max_keep() {
    return sizeof(TA) == 8 ? (DIM == 3 ? (NR < 3 ? 7 : 5) : (NR == 1 ? 6 : NR == 2 ? 5 : 4)) : (DIM == 3 ? 12 : 10);
}

// Teams laid out for some systems of a context: the host plan and its device
// arrays (freed with it).
struct Team {
    TeamPlan plan;
    int n_teams = 0;
    bool fits = false;               // there is a kernel for the plan
    std::vector<int32_t> sys;        // the systems, in the order of the plan's shares
    int32_t *row_ptr = nullptr, *list = nullptr, *halo = nullptr;
    int64_t *halo_ptr = nullptr, *step_ptr = nullptr;
    StepRec* steps = nullptr;
    uint16_t* wcol = nullptr;        // by matrix entry; a batch's teams share one array
    bool own_wcol = false;
    int* pos = nullptr;              // [n_teams][2], then the abort flag
    unsigned long long* slots = nullptr;
    char* block = nullptr;           // holds the other arrays
    Team() = default;
    Team(Team&& o) noexcept { *this = std::move(o); }
    Team& operator=(Team&& o) noexcept {
        std::swap(plan, o.plan);
        std::swap(n_teams, o.n_teams);
        std::swap(fits, o.fits);
        std::swap(sys, o.sys);
        std::swap(row_ptr, o.row_ptr);
        std::swap(list, o.list);
        std::swap(halo, o.halo);
        std::swap(halo_ptr, o.halo_ptr);
        std::swap(step_ptr, o.step_ptr);
        std::swap(steps, o.steps);
        std::swap(wcol, o.wcol);
        std::swap(own_wcol, o.own_wcol);
        std::swap(pos, o.pos);
        std::swap(slots, o.slots);
        std::swap(block, o.block);
        return *this;
    }
    ~Team() {
        void* p[] = {block, own_wcol ? wcol : nullptr, pos, slots};
        for (void* q : p)
            if (q) (void)hipFree(q);
    }
    int64_t n_slots() const { return (int64_t)n_teams * COPIES * team_slots(plan.blocks); }

    // Device arrays of a made plan: what the host laid out in one block and one
    // copy (seven of each: a new context's first solve of 100 x 100 quads 10.4 ms,
    // 6.7 so).  lists[t]: places in `sys` that team t solves, in its order.
    // wcol_in: the array to fill, or null for one of nnz entries of its own.
    hipError_t upload(const std::vector<std::vector<int32_t>>& lists, const GroupRec* d_grp, const int32_t* d_col,
                      int64_t nnz, uint16_t* wcol_in, hipStream_t stream) {
        n_teams = (int)lists.size();
        std::vector<int32_t> l{0};
        for (const auto& t : lists) l.push_back(l.back() + (int32_t)t.size());
        for (const auto& t : lists) l.insert(l.end(), t.begin(), t.end());
        std::vector<char> host;
        auto put = [&](const auto& v) {  // returns its place
            const size_t at = host.size(), n = sizeof(v[0]) * v.size();
            host.resize(at + (n + 255) / 256 * 256);
            std::copy_n((const char*)v.data(), n, host.data() + at);
            return at;
        };
        const size_t at_row = put(plan.row_ptr), at_list = put(l), at_halo = put(plan.halo), at_hptr = put(plan.halo_ptr),
                     at_sptr = put(plan.step_ptr), at_steps = put(plan.steps), at_part = put(plan.part);
        hipError_t e = hipSuccess;
        auto alloc = [&](auto*& d, size_t n) {
            if (e == hipSuccess) e = hipMalloc((void**)&d, sizeof(*d) * std::max<size_t>(n, 1));
            if (e != hipSuccess) d = nullptr;
        };
        alloc(block, host.size());
        alloc(pos, 2 * (size_t)n_teams + 1);
        alloc(slots, (size_t)n_slots());
        own_wcol = wcol_in == nullptr;
        wcol = wcol_in;
        if (own_wcol) alloc(wcol, (size_t)nnz);
        if (e != hipSuccess) return e;
        row_ptr = (int32_t*)(block + at_row);
        list = (int32_t*)(block + at_list);
        halo = (int32_t*)(block + at_halo);
        halo_ptr = (int64_t*)(block + at_hptr);
        step_ptr = (int64_t*)(block + at_sptr);
        steps = (StepRec*)(block + at_steps);
        e = hipMemcpyAsync(block, host.data(), host.size(), hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) {
            const int n_shares = (int)sys.size() * plan.blocks;
            hipLaunchKernelGGL(k_team_cols, dim3((unsigned)n_shares), dim3(256), 0, stream, n_shares, plan.blocks,
                               (const int32_t*)(block + at_part), d_grp, d_col, halo_ptr, halo, wcol);
            e = hipGetLastError();
        }
        const hipError_t done = hipStreamSynchronize(stream);  // (the host's copy goes)
        // the host keeps the sizes only
        plan.part = {}; plan.row_ptr = {}; plan.step_ptr = {}; plan.steps = {}; plan.halo_ptr = {}; plan.halo = {};
        return e == hipSuccess ? done : e;
    }

    template <typename TA>
    void args(TeamArgs<TA>& a) const {
        a.n_teams = n_teams;
        a.team_blocks = plan.blocks;
        a.team_sys = list;
        a.sys_list = list + n_teams + 1;
        a.team_pos = pos;
        a.row_ptr = row_ptr;
        a.step_ptr = step_ptr;
        a.steps = steps;
        a.wcol = wcol;
        a.halo_ptr = halo_ptr;
        a.halo = halo;
        a.slots = slots;
        a.abort = pos + 2 * n_teams;
    }
};

struct TeamShape {
    const void* kernel = nullptr;  // null: no kernel holds the plan's largest share
    unsigned lds = 0;
};

// The kernel for the plan's largest share: everything in LDS and K in registers
// where it fits, then K streamed, then r and 1/diag in memory.  us per
// iteration of a single solve, against five launches:
//   K in registers: 100 x 100 quads 5.3 (21.3), 333 x 333 8.3 (34.3),
//     40^3 x 6 tets with FP32 values 11.7 (40.7);
//   streamed: 460 x 460 quads 20.2 (49.4), 50^3 x 6 tets 34.6 (70.0);
//   r and 1/diag in memory: 64^3 x 6 tets 94.5 (159), 700 x 700 quads 43.6 (93.6).
// The halo's columns in LDS, beside K in registers, are 3 to 5 % of an iteration
// (100 x 100 quads 5.51 -> 5.32, 333 x 333 8.66 -> 8.26, 20^3 x 6 tets 7.22 ->
// 6.94); fetched ahead into registers they cost spills (8 columns a lane: 6.1,
// 9.1, 8.2).
// A window beyond the LDS was tried with gathers through the L2 and fences:
// 1000 x 1000 quads 212 (196), 80^3 x 6 tets 297 (279): those keep the launches.
template <typename TA, int NR, int DIM>
TeamShape team_shape(const TeamPlan& p) {
    const size_t win = sizeof(double) * NR * (size_t)p.max_window, row = sizeof(double) * (size_t)p.max_rows;
    const size_t all = win + row * (2 * NR + 1), pq = win + row * NR, halo = sizeof(uint32_t) * (size_t)p.max_window;
    constexpr int K = max_keep<TA, NR, DIM>();
    TeamShape s;
    if (p.max_window > MAX_WINDOW || pq > LDS_MAX) return s;
    if (all > LDS_MAX) s = {reinterpret_cast<const void*>(&k_team_pcg<TA, NR, DIM, WIN_PQ, 0>), (unsigned)pq};
    else if (p.max_passes > K || all + halo > LDS_MAX) s = {reinterpret_cast<const void*>(&k_team_pcg<TA, NR, DIM, WIN_ALL, 0>), (unsigned)all};
    else s = {reinterpret_cast<const void*>(&k_team_pcg<TA, NR, DIM, WIN_ALL, K>), (unsigned)(all + halo)};
    return s;
}

}  // namespace pgft
