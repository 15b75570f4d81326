// mdn_team.h -- persistent minimizer: whole minimizations in one kernel launch, each system by a
// team of 1 to 32 workgroups that share an XCD. Used for small single networks and for batches. The
// launch is an ordinary one; mdn_team_plan.h says which teams may be in flight together, and a team
// whose workgroups are not resident in time gives up before it has done anything that matters (the
// host then minimizes from the start again, without a team).
//
// A slot of the multi-kernel minimizer is four dependent launches (k_cg_pos, k_cg_ls, k_cg_gather,
// k_cg_fin), 6 to 7 us of launch and drain around a few us of work on a small network. Here the
// same four phases run inside one kernel, separated by team barriers: 0.85 us for up to 16
// workgroups of one XCD, 1.0 us for 32 (measured; a barrier over all XCDs costs 3.6 us, because
// every L2 has to be written back and invalidated). The finalize phase needs no barrier after it:
// every workgroup reduces the partials and takes the scalar decisions itself, on its own copy of
// the state, in the same order.
//
// The phases are spread over the team by wavefronts, each taking the 64 consecutive interactions,
// beads or coordinates that one wavefront of the slot kernels' blocks takes. The sums are taken in
// an order that does not depend on the number of workgroups:
//   SUM_SLOTS (single networks): the multi-kernel minimizer's order (wavefronts of a block, then
//     the columns as k_cg_fin's 1024 threads take them), so the result is that minimizer's bit for
//     bit (networks below GB_LARGE_BEADS beads with the same bead_energy);
//   SUM_STRIDED (batches): thread v of SUM_NT = 512 adds items v, v + 512, ... of each kind, then
//     the wavefronts' sums in order, as one workgroup of 512 threads that minimizes the system
//     alone does. Every item's energy goes through memory, and 8 wavefronts per value add them up,
//     the force sums in a phase of their own after the gather (one more barrier per slot).
//
// Memory between workgroups of one XCD goes through its L2: stores write through the L1, and every
// wavefront waits for its own stores before the barrier. A reader's L1 may hold an older copy:
// values read once (the slots, the bonded sums, the partials, the forces of the coordinate pass)
// are loaded past the L1 (agent-scope loads), and the barrier before the interactions, whose
// coordinates are read many times, ends with an agent-scope acquire, which invalidates the L1 (its
// cost grows with the workgroups of the XCD: 0.85 us at 4, 1.6 us at 16, 2.7 us at 32; the
// workgroup-scope invalidate, buffer_inv sc0, leaves the L1 as it is). Whether a team really
// shares an XCD is read from the hardware (XCC_ID) at the start; a team that does not takes
// agent-scope release and acquire fences at every barrier (correct, slower).
//
// Citations are relative to medyan-5.4.0/ in the reference tree.
#pragma once

#include "mdn_kernels.h"
#include "mdn_team_plan.h"

namespace mdn {

struct BatchItem {
    DevSys s;         // the system's tables
    CgBufs B;         // its CG vectors (B.x[0] holds the start coordinates)
    CgState* st;      // in: the start state, out: the final one
    double* report;   // out: [0..8] FP64 energy report at the start, [9..17] at the result, [18..26] scratch
    double* wpart;    // wavefront partials (team_wpart_doubles)
};

// Barrier counter and the mask of the XCDs its members run on, a cache line each; zero at launch.
struct TeamCtl {
    unsigned count, pad0[31];
    unsigned xmask, failed, pad1[30];   // failed: a workgroup gave up waiting
};

// workgroup size: 8 wavefronts at up to 256 VGPRs (12 wavefronts of 168 spill 48 to 72 of them and
// were no faster: 550 beads 1.70 against 1.65 ms per 80 iterations)
constexpr int TEAM_NT = 512;
constexpr int SUM_NT = 512;        // the threads whose order SUM_STRIDED keeps
enum { SUM_SLOTS = 0, SUM_STRIDED = 1 };
constexpr int TEAM_GB = 64;        // beads per gather column (k_cg_gather below GB_LARGE_BEADS beads)
// A barrier gives up after this many polls of its counter (97 ns each) and raises TeamCtl::failed, at
// which the others give up too: the kernel then ends instead of waiting for a workgroup that never
// arrives, and the host minimizes without a team. Polls, not time: a queue that is taken off the
// device and put back has not waited meanwhile. The first barrier waits until all workgroups are
// resident, for as long as other kernels hold the CUs: 25 ms, after which the slots, whose
// workgroups fit beside those kernels, are the better way. Beyond it every workgroup is resident
// and arrives after microseconds, or up to tens of milliseconds with deferred Simpson energies.
constexpr int TEAM_START_POLLS = 1 << 18, TEAM_POLLS = 1 << 24;

// Wavefront partials of one slot parity: energies [3][4 columns], bead kernel [2][4 nbb], gather [3][ngb]
MDN_HD inline long team_wpart_half(const DevSys& s) {
    const long ncol = s.blk[NFF] + s.nbb, ngb = (s.n_beads + TEAM_GB - 1) / TEAM_GB;
    return 12 * ncol + 8L * s.nbb + 3 * ngb;
}
// The items of SUM_STRIDED: the interactions (linkers, motors, excluded volume, boundary), then the
// beads with the filament terms they start
MDN_HD inline long team_items(const DevSys& s) {
    return (long)s.n[FF_LINKER] + s.n[FF_MOTOR] + s.n[FF_EXVOL] + s.n[FF_BOUNDARY] + s.n_beads;
}
constexpr int SUM_W = SUM_NT / 64;   // wavefront sums per value
MDN_HD inline long team_wpart_doubles(const DevSys& s, int sum) {
    return sum == SUM_STRIDED ? 3 * team_items(s) + 8 * SUM_W : 2 * team_wpart_half(s);
}

struct TeamShared {
    CgState S;
    double fold[8 * (FIN / 8)];
    double res[8];
    double red[FIN / 64];
    int bad, ndef, ok, k;
};

// This workgroup's place: wavefront gw of nw over the team.
struct Team {
    TeamCtl* c;
    unsigned target;
    int size, member, gw, nw;
    int polls;   // a barrier's limit
    bool local;
};

__device__ inline unsigned xcc_id() {
    unsigned v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
    return v & 31u;
}

// A value that another workgroup of the team wrote, loaded from the L2.
__device__ inline double team_load(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float team_load(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline bool team_failed(TeamCtl* c) {
    return __hip_atomic_load(&c->failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// All of the team's stores before it are visible after it, to team_load and, with INV, to every
// load. False (in every thread) when it gave up.
template <bool INV>
__device__ inline bool team_barrier(Team& t, TeamShared& sh) {
    if (t.size == 1) {   // one workgroup, one L1
        __syncthreads();
        return true;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's stores are in the L2
    __syncthreads();
    t.target += t.size;
    if (threadIdx.x == 0) {
        if (!t.local) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_fetch_add(&t.c->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int ok = 1;
        // (the difference: the counter may pass 2^32)
        for (int k = 0; t.polls < 0 ||
                        (int)(__hip_atomic_load(&t.c->count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - t.target) < 0; k++)
            if (k >= t.polls || ((k & 63) == 63 && team_failed(t.c))) {
                ok = 0;
                __hip_atomic_store(&t.c->failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        sh.ok = ok;
        if (INV || !t.local) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    return sh.ok != 0;
}

// k_cg_pos: wavefront v of its blocks takes the coordinates 768 (v / 4) + 64 (v % 4) + lane + 256 k.
template <int SUM>
__device__ inline void team_pos(const DevSys& s, const CgBufs& B, const CgState& S, const Team& t, double* wpos) {
    const int lane = threadIdx.x & 63, nv = 4 * s.nbb;
    const long ne = 3L * s.n_beads;
    const double* __restrict__ xc = B.x[S.parity];
    const double* __restrict__ dc = B.d[S.dpar];
    const double* __restrict__ fcur = B.f[S.fpar];
    double* __restrict__ xn = B.x[S.parity ^ 1];
    double* __restrict__ dn = B.d[S.dpar ^ 1];
    const bool move = S.phase == PH_MOVE;
    const bool first = S.ls_active == 0, pend = first && S.dir_pending;
    const double lam0 = S.ls_lambda, beta = S.dir_beta, lam = S.lambda;
    for (int v = t.gw; v < nv; v += t.nw) {
        const long e0 = 768L * (v >> 2) + 64 * (v & 3) + lane;
        double a[3], b[3], c[3], r[2] = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 3; k++) {   // every load before the first use
            const long e = e0 + 256 * k < ne ? e0 + 256 * k : ne - 1;
            a[k] = xc[e];
            b[k] = dc[e];
            c[k] = move ? 0.0 : team_load(fcur + e);
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const long e = e0 + 256 * k;
            if (e >= ne) continue;
            if (move) {
                xn[e] = a[k] + lam * b[k];
                continue;
            }
            const double de = pend ? c[k] + beta * b[k] : b[k];
            xn[e] = a[k] + lam0 * de;
            if (!first) B.xh[e] = a[k] + (lam0 * 0.5) * de;
            if (first) {
                r[0] += de * c[k];
                r[1] = rmax(r[1], fabs(de));
                if (pend) dn[e] = de;
            }
        }
        if (SUM == SUM_SLOTS && first && !move) {
            r[0] = wave_sum(r[0]);
            r[1] = wave_max(r[1]);
            if (lane == 0) {
                wpos[v] = r[0];
                wpos[nv + v] = r[1];
            }
        }
    }
}

// k_cg_ls: wavefront i of its blocks, the interaction blocks then the bead blocks.
// With SUM_STRIDED wen holds the items' energies, three values of team_items each.
template <typename R, int SUM>
__device__ inline void team_ls(const DevSys& s, const CgBufs& B, const CgState& S, const Team& t, double* wen) {
    const int lane = threadIdx.x & 63;
    const bool move = S.phase == PH_MOVE;
    const bool first = S.ls_active == 0;
    const bool need_e0 = !move && first && !S.ecur_valid, need_half = !move && !first;
    const int par = S.parity, T = s.blk[NFF];
    const bool be = s.bead_energy != 0;
    const int nint = be ? s.blk_nb : T, nevf = 4 * ev_force_blocks<R, true>(s), total = nevf + 4 * (nint + s.nbb);
    const long nc = SUM == SUM_STRIDED ? team_items(s) : 4L * (T + s.nbb);   // entries per value
    const double* __restrict__ xn = B.x[par ^ 1];
    const Pos p1{xn, nullptr, nullptr, 0.0, 0.0, 0};
    const Pos p2{B.xh, nullptr, nullptr, 0.0, 0.0, 0};
    const Pos p0{B.x[par], nullptr, nullptr, 0.0, 0.0, 0};
    R* const slots = static_cast<R*>(B.slots);
    for (int iv = t.gw; iv < total; iv += t.nw) {
        const int iw = __builtin_amdgcn_readfirstlane(iv);
        if (iw < nevf) {   // an excluded-volume force block
            const int q = 64 * iw + lane;
            if (q < s.n[FF_EXVOL]) {
                int fbad = 0;
                (void)term_ef<R>(s, FF_EXVOL, q, p1, slots, -1, &fbad);
                if (fbad) atomicAdd(B.bad_count, 1);
            }
            continue;
        }
        const int i = iw - nevf;
        const int blk = i >> 2;
        double v[3] = {0.0, 0.0, 0.0};
        long col = i, item = -1;
        bool energies = !move;
        if (blk >= nint) {   // a bead block: the bonded sums, and with bead_energy their energies
            const int b = 64 * (i - 4 * nint) + lane;
            col = 4L * T + (i - 4 * nint);
            energies = energies && be;
            if (b < s.n_beads) {
                item = nc - s.n_beads + b;
                const D3 acc = energies ? bonded_at_bead<R, true>(s, xn, b, s.pmask[b], D3{0.0, 0.0, 0.0}, &v[0])
                                        : bonded_at_bead<R>(s, xn, b, s.pmask[b], D3{0.0, 0.0, 0.0});
                s.bsum[3L * b] = acc.x;
                s.bsum[3L * b + 1] = acc.y;
                s.bsum[3L * b + 2] = acc.z;
                if (energies && need_half) v[1] = bead_bonded_energy<R>(s, B.xh, b);
                if (energies && need_e0) v[2] = bead_bonded_energy<R>(s, B.x[par], b);
            }
        } else {
            const int ff = ff_of_block(s, blk);
            const int q = (blk - s.fblk[ff]) * BLOCK + 64 * (i & 3) + lane;
            // energies only: the bead blocks or the blocks above hold the forces
            const bool only_e = ff == FF_STRETCH || ff == FF_BEND || (nevf > 0 && ff == FF_EXVOL);
            if (q < s.n[ff]) {
                item = q + (ff > FF_LINKER ? s.n[FF_LINKER] : 0) + (ff > FF_MOTOR ? s.n[FF_MOTOR] : 0) +
                       (ff > FF_EXVOL ? s.n[FF_EXVOL] : 0);
                int fbad = 0;
                if (move) {
                    if (!only_e) (void)term_ef<R>(s, ff, q, p1, slots, -1, &fbad);
                } else {
                    v[0] = term_ef<R>(s, ff, q, p1, only_e ? nullptr : slots, 0, &fbad);
                }
                if (fbad) atomicAdd(B.bad_count, 1);
                if (need_half) v[1] = term_ef<R>(s, ff, q, p2, (R*)nullptr, 1, &fbad);
                if (need_e0) v[2] = term_ef<R>(s, ff, q, p0, (R*)nullptr, 2, &fbad);
            }
        }
        if (!energies) continue;
        if constexpr (SUM == SUM_STRIDED) {
            if (item >= 0) {
                wen[item] = v[0];
                if (need_half) wen[nc + item] = v[1];
                if (need_e0) wen[2 * nc + item] = v[2];
            }
            continue;
        }
        v[0] = wave_sum(v[0]);
        if (lane == 0) wen[col] = v[0];
        if (need_half) {
            v[1] = wave_sum(v[1]);
            if (lane == 0) wen[nc + col] = v[1];
        }
        if (need_e0) {
            v[2] = wave_sum(v[2]);
            if (lane == 0) wen[2 * nc + col] = v[2];
        }
    }
}

// Bead b's force: its bonded sum, then its slots in ascending order, four slots' loads in flight.
template <typename R>
__device__ inline D3 team_bead_force(const DevSys& s, const R* __restrict__ slots, int b) {
    const int q0 = s.bstart[b], q1 = s.bstart[b + 1];
    D3 acc{team_load(s.bsum + 3L * b), team_load(s.bsum + 3L * b + 1), team_load(s.bsum + 3L * b + 2)};
    for (int q = q0; q < q1; q += 4) {
        R u[12];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const R* w = slots + 3L * min(q + j, q1 - 1);
            u[3 * j] = team_load(w);
            u[3 * j + 1] = team_load(w + 1);
            u[3 * j + 2] = team_load(w + 2);
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (q + j < q1) {
                acc.x += (double)u[3 * j];
                acc.y += (double)u[3 * j + 1];
                acc.z += (double)u[3 * j + 2];
            }
    }
    return acc;
}

// k_cg_gather: a wavefront per TEAM_GB = 64 beads.
template <typename R, int SUM>
__device__ inline void team_gather(const DevSys& s, const CgBufs& B, const CgState& S, const Team& t, double* wg,
                                   int ngb) {
    const int lane = threadIdx.x & 63;
    const bool cand = S.num_iter + 1 > S.force_call_limit / 2;
    double* __restrict__ fnext = B.f[S.fpar ^ 1];
    const double* __restrict__ fprev = B.f[S.fpar];
    const double* __restrict__ xn = B.x[S.parity ^ 1];
    double* __restrict__ xm = B.xmin[S.bkpar ^ 1];
    const R* slots = static_cast<const R*>(B.slots);
    for (int g = t.gw; g < ngb; g += t.nw) {
        const int b = TEAM_GB * g + lane;
        double v[3] = {0.0, 0.0, 0.0};
        if (b < s.n_beads) {
            const double p[3] = {fprev[3L * b], fprev[3L * b + 1], fprev[3L * b + 2]};
            const D3 acc = team_bead_force<R>(s, slots, b);
            const double fv[3] = {acc.x, acc.y, acc.z};
#pragma unroll
            for (int q = 0; q < 3; q++) {
                fnext[3L * b + q] = fv[q];
                v[0] += fv[q] * fv[q];
                v[1] += fv[q] * p[q];
                v[2] = rmax(v[2], fabs(fv[q]));
                if (cand) xm[3L * b + q] = xn[3L * b + q];
            }
        }
        if (SUM == SUM_STRIDED) continue;
        v[0] = wave_sum(v[0]);
        v[1] = wave_sum(v[1]);
        v[2] = wave_max(v[2]);
        if (lane == 0)
            for (int q = 0; q < 3; q++) wg[(long)q * ngb + g] = v[q];
    }
}

// SUM_STRIDED's sums: wavefront w of the SUM_NT threads for every value, into ws[value][wavefront]:
// E(lambda), E(lambda / 2), E(x), d.F, max|d|, F.F, F.F_prev, max|F|. The loads of SUM_IN items per
// thread are in flight at once (one at a time, an 11,900-bead network's sums took 13 us of a 31 us
// slot; four 8 us).
constexpr int SUM_IN = 12;

// Entries v, v + SUM_NT, ... of each run of a list, one run after the other.
template <int N>
__device__ inline double strided_sum(const double* e, const int (&cnt)[N], int v) {
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int n = cnt[k];
        for (int q = v; q < n; q += SUM_IN * SUM_NT) {
            double u[SUM_IN];
#pragma unroll
            for (int j = 0; j < SUM_IN; j++) u[j] = team_load(e + min(q + j * SUM_NT, n - 1));
#pragma unroll
            for (int j = 0; j < SUM_IN; j++)
                if (q + j * SUM_NT < n) a += u[j];
        }
        e += n;
    }
    return a;
}

// The energies and d.F, max|d|, while the forces are gathered: the last wavefronts of the team,
// which have the fewest beads to gather, take one wavefront of one kind each.
__device__ inline void team_sums_ls(const DevSys& s, const CgBufs& B, const CgState& S, const Team& t,
                                    const double* wen, double* ws) {
    if (S.phase != PH_LS) return;
    const int lane = threadIdx.x & 63, nb = s.n_beads;
    const bool first = S.ls_active == 0;
    const bool want[4] = {true, !first, first && S.ecur_valid == 0, first};
    const long nc = team_items(s);
    for (int task = t.nw - 1 - t.gw; task < 4 * SUM_W; task += t.nw) {
        const int kind = task / SUM_W, w = task % SUM_W, v = 64 * w + lane;
        if (!want[kind]) continue;
        if (kind < 3) {
            const int cnt[5] = {s.n[FF_LINKER], s.n[FF_MOTOR], s.n[FF_EXVOL], s.n[FF_BOUNDARY], nb};
            const double a = wave_sum(strided_sum(wen + kind * nc, cnt, v));
            if (lane == 0) ws[kind * SUM_W + w] = a;
            continue;
        }
        // the direction this launch used: the materialized one when it was pending
        const double* d = S.dir_pending ? B.d[S.dpar ^ 1] : B.d[S.dpar];
        const double* f = B.f[S.fpar];
        const int n = 3 * nb;
        double a = 0.0, m = 0.0;
        for (int q = v; q < n; q += SUM_IN * SUM_NT) {
            double u[SUM_IN], g[SUM_IN];
#pragma unroll
            for (int j = 0; j < SUM_IN; j++) {
                u[j] = team_load(d + min(q + j * SUM_NT, n - 1));
                g[j] = team_load(f + min(q + j * SUM_NT, n - 1));
            }
#pragma unroll
            for (int j = 0; j < SUM_IN; j++)
                if (q + j * SUM_NT < n) {
                    a += u[j] * g[j];
                    m = rmax(m, fabs(u[j]));
                }
        }
        a = wave_sum(a);
        m = wave_max(m);
        if (lane == 0) {
            ws[3 * SUM_W + w] = a;
            ws[4 * SUM_W + w] = m;
        }
    }
}

// The force sums, once every force is gathered.
__device__ inline void team_sums_f(const DevSys& s, const CgBufs& B, const CgState& S, const Team& t, double* ws) {
    constexpr int NI = SUM_IN / 2;   // beads in flight per thread
    const int lane = threadIdx.x & 63, nb = s.n_beads;
    const double* f = B.f[S.fpar ^ 1];
    const double* p = B.f[S.fpar];
    for (int w = t.gw; w < SUM_W; w += t.nw) {
        double a = 0.0, c = 0.0, m = 0.0;
        for (int b = 64 * w + lane; b < nb; b += NI * SUM_NT) {
            double u[3 * NI], g[3 * NI];
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const long i = 3L * min(b + j * SUM_NT, nb - 1) + q;
                    u[3 * j + q] = team_load(f + i);
                    g[3 * j + q] = team_load(p + i);
                }
#pragma unroll
            for (int j = 0; j < NI; j++)
                if (b + j * SUM_NT < nb)
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        a += u[3 * j + q] * u[3 * j + q];
                        c += u[3 * j + q] * g[3 * j + q];
                        m = rmax(m, fabs(u[3 * j + q]));
                    }
        }
        a = wave_sum(a);
        c = wave_sum(c);
        m = wave_max(m);
        if (lane == 0) {
            ws[5 * SUM_W + w] = a;
            ws[6 * SUM_W + w] = c;
            ws[7 * SUM_W + w] = m;
        }
    }
}

// A block's partial from its four wavefronts' (block_reduce_n's order).
__device__ inline double team_col_sum(const double* w) {
    return ((team_load(w) + team_load(w + 1)) + team_load(w + 2)) + team_load(w + 3);
}
__device__ inline double team_col_max(const double* w) {
    return rmax(rmax(rmax(team_load(w), team_load(w + 1)), team_load(w + 2)), team_load(w + 3));
}

// k_cg_fin, by every workgroup of the team on its own copy of the state: the columns are summed
// as that kernel's FIN threads sum them (thread v takes columns v, v + FIN, ...), its groups of 8
// lanes and its final wavefront reduction included.
template <int NT>
__device__ inline void team_columns(const DevSys& s, TeamShared& sh, const double* wen, const double* wpos,
                                    const double* wg, int ngb) {
    constexpr int NW = NT / 64;
    static_assert(NW >= 8, "one wavefront per reduced value");
    const CgState& S = sh.S;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int T = s.blk[NFF];
    const bool be = s.bead_energy != 0;
    const int ne0 = be ? s.blk_nb : T, ne = ne0 + (be ? s.nbb : 0);
    const long nc = 4L * (T + s.nbb), np = 4L * s.nbb;
    const bool ls = S.phase == PH_LS;
    const bool want_half = ls && S.ls_active != 0, want_x = ls && S.ls_active == 0 && S.ecur_valid == 0;
    const bool want_pos = ls && S.ls_active == 0;
    // every value's first column is loaded before any of them is used (one round trip), clamped
    // to a column that exists; the columns beyond FIN follow one value at a time
    const int nmax = max(max(ne, s.nbb), ngb);
    for (int vw = w; vw < FIN / 64; vw += NW) {
        const int v = 64 * vw + lane;
        // E(lambda), E(lambda / 2), E(x), d.F, max|d|, F.F, F.F_prev, max|F|
        double a[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (64 * vw < nmax) {
            auto ecol = [&](int c) { return 4L * (c < ne0 ? c : T + (c - ne0)); };
            const double* e = wen + ecol(max(0, min(v, ne - 1)));   // (a network may have no interactions)
            const double* p = wpos + 4L * min(v, s.nbb - 1);
            const double* g = wg + min(v, ngb - 1);
            double x[12], y[3];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[j] = team_load(e + j);
                x[4 + j] = team_load(p + j);
                x[8 + j] = team_load(p + np + j);
            }
#pragma unroll
            for (int j = 0; j < 3; j++) y[j] = team_load(g + (long)j * ngb);
            if (ls && v < ne) a[0] = ((x[0] + x[1]) + x[2]) + x[3];
            if (want_pos && v < s.nbb) {
                a[3] = ((x[4] + x[5]) + x[6]) + x[7];
                a[4] = rmax(0.0, rmax(rmax(rmax(x[8], x[9]), x[10]), x[11]));
            }
            if (v < ngb) {
                a[5] = y[0];
                a[6] = y[1];
                a[7] = rmax(0.0, y[2]);
            }
            if (ls)
                for (int c = v + FIN; c < ne; c += FIN) a[0] += team_col_sum(wen + ecol(c));
            if (want_half)
                for (int c = v; c < ne; c += FIN) a[1] += team_col_sum(wen + nc + ecol(c));
            if (want_x)
                for (int c = v; c < ne; c += FIN) a[2] += team_col_sum(wen + 2 * nc + ecol(c));
            if (want_pos)
                for (int c = v + FIN; c < s.nbb; c += FIN) {
                    a[3] += team_col_sum(wpos + 4L * c);
                    a[4] = rmax(a[4], team_col_max(wpos + np + 4L * c));
                }
            for (int c = v + FIN; c < ngb; c += FIN) {
                a[5] += team_load(wg + c);
                a[6] += team_load(wg + ngb + c);
                a[7] = rmax(a[7], team_load(wg + 2L * ngb + c));
            }
#pragma unroll
            for (int q = 0; q < 8; q++) a[q] = (q == 4 || q == 7) ? wave_fold8<1>(a[q]) : wave_fold8<0>(a[q]);
        }
        if ((lane & 7) == 7)
#pragma unroll
            for (int q = 0; q < 8; q++) sh.fold[q * (FIN / 8) + vw * 8 + (lane >> 3)] = a[q];
    }
    __syncthreads();
    if (w < 8) {
        const bool mx = w == 4 || w == 7;
        const double u0 = sh.fold[w * (FIN / 8) + lane], u1 = sh.fold[w * (FIN / 8) + lane + 64];
        static_assert(FIN / 8 == 128, "two values per lane");
        double r = mx ? rmax(u0, u1) : u0 + u1;
        r = mx ? wave_max(r) : wave_sum(r);
        if (lane == 0) sh.res[w] = r;
    }
}

// The reduced values into sh.res (SUM_SLOTS: team_columns; SUM_STRIDED: the wavefronts' sums in
// order), then the decisions of k_cg_fin, by every workgroup of the team on its own copy of the
// state.
template <int NT, int SUM>
__device__ inline bool team_fin(const DevSys& s, const CgBufs& B, TeamShared& sh, Team& t, const double* wen,
                                const double* wpos, const double* wg, int ngb) {
    CgState& S = sh.S;
    if (threadIdx.x == 0) {
        sh.ndef = __hip_atomic_load(s.defer_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh.bad = __hip_atomic_load(B.bad_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int phase0 = S.phase;
    const bool ls = phase0 == PH_LS;
    if constexpr (SUM == SUM_SLOTS) {
        team_columns<NT>(s, sh, wen, wpos, wg, ngb);
    } else if (threadIdx.x >= 64 && threadIdx.x < 72) {   // wen: the wavefront sums
        const int q = threadIdx.x - 64;
        const bool mx = q == 4 || q == 7;
        double u[SUM_W];
#pragma unroll
        for (int j = 0; j < SUM_W; j++) u[j] = team_load(wen + q * SUM_W + j);
        double r = u[0];
#pragma unroll
        for (int j = 1; j < SUM_W; j++) r = mx ? rmax(r, u[j]) : r + u[j];
        sh.res[q] = r;
    }
    __syncthreads();
    const int ndef = sh.ndef, bad0 = sh.bad;
    double dsum[3] = {0.0, 0.0, 0.0};
    int dbad[3] = {0, 0, 0};
    const bool reset = bad0 != 0 || ndef > 0;   // the same in every workgroup
    if (ls && ndef > 0) {
        // the deferred Simpson energies: one workgroup evaluates them, all read its results
        if (t.member == 0) run_defers_eval<NT, SUM == SUM_SLOTS ? FIN : SUM_NT>(s, ndef, sh.red);
        if (!team_barrier<true>(t, sh)) return false;
        if (threadIdx.x == 0) defer_sums(s, min(ndef, DEFER_CAP), dsum, dbad, 3);
    }
    if (reset) {
        if (!team_barrier<false>(t, sh)) return false;   // every workgroup has read both counts and the list
        if (t.member == 0 && threadIdx.x == 0) {
            __hip_atomic_store(s.defer_n, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(B.bad_count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (threadIdx.x == 0) {
        CgState Sr = S;   // the scalar control on a register copy
        int bad = bad0;
        const double acc[8] = {sh.res[0] + dsum[0], sh.res[1] + dsum[1], (double)dbad[0], (double)dbad[1],
                               sh.res[2] + dsum[2], (double)dbad[2], sh.res[3], Sr.max_dist / sh.res[4]};
        const double g[3] = {sh.res[5], sh.res[6], sh.res[7]};
        bool gather = phase0 == PH_MOVE;
        if (ls) {
            if (ndef > DEFER_CAP) {
                Sr.status = 9;
                Sr.done = 1;
            } else {
                ls_control(Sr, acc, bad);
                gather = !Sr.done && Sr.phase == PH_GATHER;
            }
        } else {
            Sr.n_move_launch += 1;
        }
        if (gather) gather_control(Sr, g, bad);
        S = Sr;
    }
    __syncthreads();
    return true;
}

// CG slots of one system until its state is done.
template <typename R, int NT, int SUM>
__device__ inline void team_run(const DevSys& s, const CgBufs& B, CgState* st, double* wpart, Team& t,
                                TeamShared& sh) {
    state_load(&sh.S, st);
    const int ngb = (s.n_beads + TEAM_GB - 1) / TEAM_GB;
    const long half = team_wpart_half(s), nc = 4L * (s.blk[NFF] + s.nbb), np = 4L * s.nbb;
    const long max_slots = slots_per_force_call(sh.S) * ((long)sh.S.force_call_limit + 16) + 128;
    for (long k = 0; k < max_slots && !sh.S.done; k++) {
        // SUM_SLOTS: the partials alternate between two halves, since a workgroup ahead of the
        // others writes the next slot's while they still read this one's (with SUM_STRIDED a
        // barrier lies between)
        double* wen = SUM == SUM_SLOTS ? wpart + (k & 1) * half : wpart;
        double* wpos = wen + 3 * nc;
        double* wg = wpos + 2 * np;
        double* ws = wpart + 3 * team_items(s);
        team_pos<SUM>(s, B, sh.S, t, wpos);
        if (!team_barrier<true>(t, sh)) break;
        team_ls<R, SUM>(s, B, sh.S, t, wen);
        if (!team_barrier<false>(t, sh)) break;
        if constexpr (SUM == SUM_STRIDED) team_sums_ls(s, B, sh.S, t, wen, ws);
        team_gather<R, SUM>(s, B, sh.S, t, wg, ngb);
        if (!team_barrier<false>(t, sh)) break;
        if constexpr (SUM == SUM_STRIDED) {
            team_sums_f(s, B, sh.S, t, ws);
            if (!team_barrier<false>(t, sh)) break;
        }
        if (!team_fin<NT, SUM>(s, B, sh, t, SUM == SUM_SLOTS ? wen : ws, wpos, wg, ngb)) break;
    }
    __syncthreads();
    if (threadIdx.x == 0 && !sh.S.done) {   // never reached by a correct state machine
        sh.S.status = 3;                    // MDN_ERR_STATE: did not terminate
        sh.S.done = 1;
    }
    if (t.member == 0) state_store(st, &sh.S);
    __syncthreads();   // the shared state is reused by the next system
}

// polls: the first barrier's limit. size 0: the team gave up, nothing is written.
__device__ inline Team team_start(TeamCtl* c, int size, int member, TeamShared& sh, int nwaves, int polls) {
    Team t;
    t.polls = polls;
    t.c = c;
    t.target = 0;
    t.size = size;
    t.member = member;
    t.nw = size * nwaves;
    t.gw = (threadIdx.x >> 6) * size + member;   // consecutive wavefronts on different workgroups
    t.local = false;
    if (size > 1) {
        if (threadIdx.x == 0)
            __hip_atomic_fetch_or(&c->xmask, 1u << xcc_id(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!team_barrier<false>(t, sh)) t.size = 0;
        t.polls = TEAM_POLLS;
        if (threadIdx.x == 0)
            sh.k = __popc(__hip_atomic_load(&c->xmask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        __syncthreads();
        t.local = sh.k == 1;
        __syncthreads();
    }
    return t;
}

// One system. Grid: stride * (size - 1) + 1 workgroups; workgroup stride * m is member m, the
// others end at once (workgroups go round-robin over the XCDs, so a stride of 8 keeps the team on one).
template <typename R, int NT>
__global__ void __launch_bounds__(NT) k_cg_team_one(DevSys s, CgBufs B, CgState* st, TeamCtl* ctl, double* wpart,
                                                    int size, int stride, int polls) {
    __shared__ TeamShared sh;
    if (blockIdx.x % stride) return;
    Team t = team_start(ctl, size, blockIdx.x / stride, sh, NT / 64, polls);
    if (t.size == 0) return;
    team_run<R, NT, SUM_SLOTS>(s, B, st, wpart, t, sh);
}

// A batch: every workgroup takes its place in its team; a team with a system of its own minimizes
// it, a single workgroup without one pulls systems order[k], k = 0, 1, ... until the queue passes n.
template <typename R, int NT>
__global__ void __launch_bounds__(NT) k_cg_team(const BatchItem* __restrict__ items, const TeamSlot* __restrict__ slot,
                                                const TeamInfo* __restrict__ team, TeamCtl* ctl,
                                                const int* __restrict__ order, int n, int* queue, int polls) {
    __shared__ TeamShared sh;
    const TeamSlot me = slot[blockIdx.x];
    if (me.team < 0) return;
    const TeamInfo ti = team[me.team];
    Team t = team_start(ctl + me.team, ti.size, me.member, sh, NT / 64, polls);
    if (t.size == 0) return;
    for (;;) {
        int i = ti.sys;
        if (i < 0) {
            __syncthreads();
            if (threadIdx.x == 0) sh.k = atomicAdd(queue, 1);
            __syncthreads();
            if (sh.k >= n) return;
            i = order[sh.k];
        }
        const BatchItem& it = items[i];
        team_run<R, NT, SUM_STRIDED>(it.s, it.B, it.st, it.wpart, t, sh);
        if (ti.sys >= 0) return;
    }
}

// =======================================================================================
// A batch's start and end: the set-up of mdn_minimize (CGMethod.hpp:876-896) and its final report,
// for every system in one launch each (blockIdx.y = the system; blocks past a system's own end at
// once)
// =======================================================================================
struct BatchParams {
    int method, try_recover, force_call_limit, energy_call_limit, report_on_call_limit;
    int line_search;      // MDN_LS_*
    double max_dist, lambda_max, grad_tol, energy_rel_tol;
};

__device__ inline bool batch_ok(const CgState* st) { return st->status == 0 && st->error_flags == 0; }

// The energy report's block partials: which = 0 at the start (x[0]), 1 at the result (systems
// that ended without an error).
template <typename R>
__global__ void __launch_bounds__(BLOCK) k_batch_energy(const BatchItem* __restrict__ items, int which) {
    __shared__ double lds[BLOCK / 64];
    const BatchItem& it = items[blockIdx.y];
    if ((int)blockIdx.x >= it.s.blk[NFF]) return;
    if (which == 1 && !batch_ok(it.st)) return;
    energy_block<R>(it.s, which == 1 ? it.B.x[it.st->parity] : it.B.x[0], it.B.partial, lds);
}
__global__ void __launch_bounds__(BLOCK) k_batch_energy_fin(const BatchItem* __restrict__ items, int which, int off) {
    __shared__ double lds[NFF * (BLOCK / 64)];
    const BatchItem& it = items[blockIdx.x];
    if (which == 1 && !batch_ok(it.st)) return;
    energy_fin(it.s, it.B.partial, it.report + off, lds);
}

// searchDir.assign(numDof, 0) and the count of pairs that need the force fallback
__global__ void __launch_bounds__(BLOCK) k_batch_zero(const BatchItem* __restrict__ items) {
    const BatchItem& it = items[blockIdx.y];
    const long n = 3L * it.s.n_beads;
    for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long)gridDim.x * BLOCK) it.B.d[0][i] = 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *it.B.bad_count = 0;
}

// the slots and bonded sums at the start (k_forces_terms with bead blocks)
template <typename R>
__global__ void __launch_bounds__(BLOCK, sizeof(R) == 4 ? 4 : 1) k_batch_terms(const BatchItem* __restrict__ items) {
    const BatchItem& it = items[blockIdx.y];
    if ((int)blockIdx.x >= it.s.blk_nb + it.s.nbb) return;
    terms_block<R>(it.s, it.B.x[0], static_cast<R*>(it.B.slots), it.B.bad_count, nullptr, it.s.blk_nb, 3, nullptr);
}

// the forces at the start into f[0]
template <typename R>
__global__ void __launch_bounds__(BLOCK) k_batch_gather(const BatchItem* __restrict__ items) {
    const BatchItem& it = items[blockIdx.y];
    const int b = blockIdx.x * BLOCK + threadIdx.x;
    if (b >= it.s.n_beads) return;
    const D3 a = team_bead_force<R>(it.s, static_cast<const R*>(it.B.slots), b);
    it.B.f[0][3L * b] = a.x;
    it.B.f[0][3L * b + 1] = a.y;
    it.B.f[0][3L * b + 2] = a.z;
}

// the start state (resetCGParams applied by the first line search), with F.F and max|F| summed as
// SUM_STRIDED sums them; e_off: the report that holds the start energy in the working precision
__global__ void __launch_bounds__(SUM_NT) k_batch_init(const BatchItem* __restrict__ items, BatchParams P, int e_off) {
    __shared__ double lds[2 * SUM_W];
    const BatchItem& it = items[blockIdx.x];
    double v[2] = {0.0, 0.0};
    for (int b = threadIdx.x; b < it.s.n_beads; b += SUM_NT)
        for (int q = 0; q < 3; q++) {
            const double f = it.B.f[0][3L * b + q];
            v[0] += f * f;
            v[1] = rmax(v[1], fabs(f));
        }
    const int op[2] = {0, 1};
    block_reduce_n<2, SUM_NT>(v, op, lds);
    if (threadIdx.x != 0) return;
    CgState S = CgState{};
    S.method = P.method;
    S.ls_algo = P.line_search;
    S.try_recover = P.try_recover;
    S.force_call_limit = max(P.force_call_limit, 3 * it.s.n_beads);
    S.energy_call_limit = P.energy_call_limit;
    S.max_dist = P.max_dist;
    S.lambda_max = P.lambda_max;
    S.grad_tol = P.grad_tol;
    S.energy_rel_tol = P.energy_rel_tol;
    S.num_energy_call = 1;
    S.num_force_call = 1;
    S.grad_inf_norm = v[1];
    S.energy_rel_change = INFINITY;
    S.prev_energy = it.report[e_off + 6];
    S.minimum_e = INFINITY;
    S.fdotf = v[0];
    S.dir_pending = 1;
    S.dir_beta = 0.0;
    S.dir_reset = 1;
    S.phase = PH_LS;
    S.ls_lambda = rmin(S.lambda_max, S.max_dist / S.grad_inf_norm);
    if (*it.B.bad_count) {
        // an excluded-volume pair needs the numerical force fallback, which a batch does not run
        // (reported as MDN_ERR_UNSUPPORTED, like a pause for it later in the run)
        S.status = ST_NEED_FORCEN;
        S.done = 1;
        *it.B.bad_count = 0;
    } else if (!isfinite(v[1]) || !isfinite(v[0])) {
        S.status = 4;   // MDN_ERR_NONFINITE: maxF not finite (CGMethod.hpp:202-212)
        S.done = 1;
    } else {
        S.done = (converged_s(S) || call_limit_s(S)) ? 1 : 0;
    }
    *it.st = S;
}

// copybackupcoordinates on a call limit (CGMethod.hpp:1579-1590); reserved[0] tells the host
__global__ void __launch_bounds__(BLOCK) k_batch_restore(const BatchItem* __restrict__ items, int report_on_call_limit) {
    const BatchItem& it = items[blockIdx.y];
    CgState* st = it.st;
    const bool on = batch_ok(st) && report_on_call_limit && call_limit(st) && st->have_min_e;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->reserved[0] = on ? 1 : 0;
    if (!on) return;
    double* x = it.B.x[st->parity];
    const double* xb = it.B.xmin[st->bkpar];
    const long n = 3L * it.s.n_beads;
    for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long)gridDim.x * BLOCK) x[i] = xb[i];
}

// The final CG state and the energy report (27 values) of every system of a batch, gathered into
// contiguous buffers for one read-back: states[i], reports[27 i ...]. Grid-stride over
// (system, word).
__global__ void __launch_bounds__(256) k_batch_collect(const BatchItem* __restrict__ items, int n,
                                                       CgState* __restrict__ states, double* __restrict__ reports) {
    constexpr int NW = sizeof(CgState) / sizeof(int);
    static_assert(sizeof(CgState) % sizeof(int) == 0, "CgState in whole words");
    const long total = (long)n * (NW + 27);
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (long)gridDim.x * blockDim.x) {
        const int i = (int)(k / (NW + 27)), w = (int)(k % (NW + 27));
        if (w < NW) reinterpret_cast<int*>(states + i)[w] = reinterpret_cast<const int*>(items[i].st)[w];
        else reports[27L * i + (w - NW)] = items[i].report[w - NW];
    }
}

// One launch for the start copies of a whole batch (each system's device coordinates into its
// x[0], and into a backup where a team that gives up would leave them overwritten): copy i moves
// c[i].n doubles from c[i].src to c[i].dst. Grid (blocks per copy, copies), both strided.
struct BatchCopy {
    const double* src;
    double* dst;
    long n;
};
__global__ void __launch_bounds__(256) k_batch_copy(const BatchCopy* __restrict__ c, int n) {
    for (int i = blockIdx.y; i < n; i += gridDim.y) {
        const BatchCopy e = c[i];
        for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < e.n; k += (long)gridDim.x * blockDim.x)
            e.dst[k] = e.src[k];
    }
}

__global__ void k_fill_int(int* p, int v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

}  // namespace mdn
