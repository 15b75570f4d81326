// mdn_mech.hip -- host side of the gfx950 mechanical-equilibration library: context, system
// upload (vectorize), neighbor-list rebuild, energy / force entry points and the
// device-driven conjugate-gradient minimizer, behind the C ABI of include/mdn_mech.h.
//
// Citations are relative to medyan-5.4.0/ in the reference tree.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <sys/mman.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/mdn_mech.h"
#include "mdn_kernels.h"
#include "mdn_team.h"

using namespace mdn;

// Scratch of the force evaluation without allocation (mdn_forces_noalloc): the slot vectors,
// the per-bead bonded sums, the excluded-volume pairs that need the numerical fallback and that
// fallback's partial sums. Every device the library runs on holds its own copy for the life of
// the process. The name is a host-side stand-in, not a device address: host code uses the
// address hipGetSymbolAddress returns for the current device (scratch_dev below), never the name.
constexpr size_t MDN_SCRATCH_BYTES = (size_t)MDN_NOALLOC_SCRATCH_MIB << 20;
static __device__ __align__(256) unsigned char scratch[MDN_SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_dev[MAX_DEVICES] = {};   // device address of `scratch`, per device

// Looks the array's address up on `device` (current) once; every later call returns it.
hipError_t scratch_lookup(int device) {
    if (device < 0 || device >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_dev[device]) return hipSuccess;
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess) g_scratch_dev[device] = static_cast<unsigned char*>(p);
    return e;
}

// stored slots per interaction (filament stretching / bending forces are computed by the gather)
constexpr int SLOTS_PER_TERM[NFF] = {0, 0, 4, 4, 4, 1};

template <typename T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    hipError_t ensure(size_t want) {
        if (want <= n && p) return hipSuccess;
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
        size_t m = std::max<size_t>(want, 1);
        hipError_t e = hipMalloc(&p, m * sizeof(T));
        if (e == hipSuccess) n = m;
        return e;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
};

// The CG state and, from TEAM_CTL_OFF on, the persistent minimizer's barrier: uploaded together.
constexpr size_t TEAM_CTL_OFF = 1024, CG_BYTES = TEAM_CTL_OFF + sizeof(TeamCtl);
static_assert(sizeof(CgState) <= TEAM_CTL_OFF, "the barrier follows the state");
TeamCtl* team_ctl(CgState* cg) { return reinterpret_cast<TeamCtl*>(reinterpret_cast<char*>(cg) + TEAM_CTL_OFF); }

struct HipErr {
    hipError_t e;
    const char* what;
};

}  // namespace

constexpr int STAGE_SLOTS = 16;   // chunks of a host copy in flight

struct mdn_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    bool uploaded = false, nl_built = false;

    // system (host copies used by vectorize)
    int n_beads = 0, n_cyl = 0, n_fil = 0;
    std::vector<int> cyl_b1, cyl_b2, cyl_fil, cyl_pos, cyl_type;
    std::vector<char> cyl_minus;
    std::vector<double> cyl_kexvol, cyl_eql;
    std::vector<mdn_boundary_element> elems;
    double bnd_cutoff = 0, rmax = 0, rmin = 0, grid[3] = {0, 0, 0};

    // device tables
    DBuf<int> str_b, bend_b, lnk_b, mot_b, ev_b, bnd_b, bnd_e, lnk_ord, mot_ord;
    std::vector<int> xl_ord[2];   // linkers, motors: device table position -> crosslink index
    DBuf<double> dof_next, dof_new;   // mdn_dof_serialize: the gathered coordinates, new beads
    DBuf<int> dof_src;
    int dof_next_n = -1;              // beads in dof_next (-1: none pending)
    DBuf<double> str_k, str_eql, bend_k, bend_eqt, lnk_k, lnk_eql, lnk_p1, lnk_p2, lnk_sf;
    DBuf<double> mot_k, mot_eql, mot_p1, mot_p2, mot_sf, ev_ks, bnd_krep, bnd_slen;
    DBuf<int> inc_s_start, inc_s, inc_cnt, inc_list, bstart, sorted_id, pos;
    DBuf<unsigned char> pmask;
    DBuf<int> bnbr, bterm;   // filament neighbours and term indices per bead (bonded_at_bead)
    DBuf<double> bsum;       // per-bead bonded sums, 3 * n_beads
    int bonded_gather_mode = -1;   // -1: the defaults below, else both of them
    int bg_eval = 1;                // force evaluations use the bonded sums (bead blocks)
    // parameter gradients / tangents: per cylinder the bending term it is the second cylinder of
    // (-1: none), per bending term its cylinder (host), per-pair excluded-volume energies, a vector
    DBuf<int> d_cyl_bend;
    std::vector<int> bend_cyl;
    DBuf<double> ev_U, grad_out, tan_v;
    DBuf<double> hb_v, hb_slots, hb_piece, hb_out;   // mdn_hvp_batch: per-product tangents, slots, pieces, results
    DBuf<double> piece;   // NBOND * 3 * n_beads values (FP64; the mixed path uses the first half as float)
    // cylinder tables for the NL
    DBuf<int> d_cyl_b1, d_cyl_b2, d_cyl_fil, d_cyl_pos, d_cyl_type;
    DBuf<char> d_cyl_minus;
    DBuf<int> d_fil_ends;      // [2 * n_fil]: first and last cylinder of each filament
    DBuf<double> load_out;     // boundary load forces [2][n_fil][stride]
    DBuf<double> d_cyl_kexvol, d_cyl_eql, d_krep_e, d_slen_e;
    // NL workspace
    DBuf<double> mid;
    DBuf<int> bin, bin_count, bin_start, place, nl_found, nl_list, nl_count, nl_off, pairs, bnd_cnt, bnd_off;
    // the binding-site search's own list (mdn_binding_pairs) and its per-pair counts
    DBuf<double> b_mid, mmid, b_mmid;
    DBuf<NlRec> members, b_members;
    DBuf<int> b_bin, b_bin_count, b_bin_start, b_place, b_count, b_off, b_pairs, b_scount, b_soff;
    DBuf<int> mbin, b_mbin;
    DBuf<float> b_site, b_free;
    DBuf<uint32_t> b_out;
    DBuf<unsigned char> cub_tmp;
    long n_pairs = 0;
    int n_bint = 0;
    std::vector<int> bnd_nneighbors;

    // state vectors
    DBuf<double> x[2], f, f2, xh, d[2], xmin[2], scratch_f, ext;   // f, f2: the CG force pair
    DBuf<double> slots;   // 3 values per slot; the mixed path uses the first half as float
    DBuf<double> partial;
    DBuf<int> bad_count, bad_list;
    DBuf<unsigned> ticket;
    DBuf<double> eout;
    DBuf<double> vstat;   // k_vec_stats partials (2 * VSTAT_BLOCKS)
    DBuf<CgState> cg;
    DBuf<double> fallback_partial;
    DBuf<EnDefer> defer;
    DBuf<int> defer_n;
    DBuf<int> fallback_ok;
    CgState* h_cg = nullptr;   // pinned
    double* h_eout = nullptr;  // pinned
    int* h_int = nullptr;      // pinned
    hipEvent_t stage_ev[STAGE_SLOTS] = {};   // copy_parts

    DevSys sys{};
    int cur = 0;   // which x buffer holds the current coordinates

    DBuf<double> team_part;   // wavefront partials of the persistent minimizer
    int team_size = -1;       // workgroups of the persistent minimizer: -1 by size, 0 never (MDN_CG_TEAM)
    int team_stride = 8, team_polls = TEAM_START_POLLS;   // MDN_TEAM_STRIDE, MDN_TEAM_POLLS
    int n_cu = 0;             // the device's
    int last_team[2] = {0, 0};   // mdn_last_team
    // batched minimizer (the lead context of a batch owns these)
    DBuf<TeamSlot> batch_slot;
    DBuf<TeamInfo> batch_team;
    DBuf<TeamCtl> batch_ctl;
    DBuf<BatchItem> batch_items;
    DBuf<CgState> batch_states;   // the batch's final states and reports, gathered for one read-back
    DBuf<double> batch_reports;
    DBuf<int> batch_order, batch_queue;
    DBuf<BatchCopy> batch_copy;   // start copies, backups

    bool use_graph = true;   // replay the CG slots as a captured hipGraph (MDN_CG_GRAPH=0: launch them directly)
    hipGraphExec_t graph_exec[2] = {nullptr, nullptr};   // per precision (MDN_PREC_*)
    hipGraph_t graph[2] = {nullptr, nullptr};
    long sys_gen = 0, graph_gen[2] = {-1, -1};
    long min_gen[2] = {-1, -1};   // the system generation of the last minimization, per precision
    CgState last_cg{};
};

namespace {

int fail(mdn_ctx* c, int code, const char* fmt, ...) {
    if (c) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        c->err = buf;
    }
    return code;
}

#define HIPCHK(call)                                                                            \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            return fail(ctx, MDN_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),  \
                        __FILE__, __LINE__);                                                    \
    } while (0)

#define HIPCHK_CTX(c, call)                                                                     \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            return fail((c), MDN_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),  \
                        __FILE__, __LINE__);                                                    \
    } while (0)

// Device-to-host read ordered after everything queued on the context's stream (a blocking
// hipMemcpy runs on the null stream, which does not wait for the non-blocking context stream).
hipError_t d2h(mdn_ctx* ctx, void* dst, const void* src, size_t bytes) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(ctx->stream);
}

// ---- host copies through pinned memory ------------------------------------------------------
// Copies go through a pinned ring where that is the faster way: a kernel moves the pieces between
// device and ring (k_copy_pieces), the CPU between ring and caller, chunk by chunk side by side, and
// pages of a result that the caller has not touched yet are mapped in one call per chunk ahead of the
// copy. The runtime's copy of more than 16 KB is a copy engine's: fast when the same stream used that
// engine last, 17 to 35 us more when a program goes through more than some 8 contexts, and a wait for
// the kernels queued before it. The ring's costs are the same always. Runtime and ring, us:
//     result, idle stream         13 KB 23, 14;  94 KB 13, 17;  256 KB 20, 23;  1 MB 62, 78;
//                                 2 MB 122, 129;  3 MB 182, 135;  8 MB 485, 385
//       one of 32 contexts        91 KB 51, 19
//       into fresh pages          24 KB 14, 18;  96 KB 29, 26;  256 KB 63, 49;  768 KB 170, 121;
//                                 1 MB 280, 180;  8 MB 2240, 1490
//     result behind kernels       7 KB 52, 42;  18 KB 57, 51;  76 KB 64, 58;  211 KB 78, 72;  with more
//       (mdn_hvp, whole call)     than one chunk it depends: 374 KB 100, 119;  456 KB 108, 127
//     input                       16 KB 13, 14;  64 KB 11, 15;  256 KB 16, 21;  1 MB 55, 78;  8 MB 250, 280
//       of mdn_forces             91 KB 53, 58;  one of 32 contexts 87, 59
//       of mdn_minimize           91 KB 832, 839;  96 contexts in turn 566, 533
//       four 144 KB parameters    61, 111
// So results of one chunk take the ring, larger ones beyond STAGE_LARGE and from STAGE_FRESH on into
// fresh pages. The runtime queues inputs, while each one through the ring is a wait: only a
// minimization's coordinates take it, for which that is little. A batch's many tables and coordinates
// take the ring together in both directions.
// Rings belong to the process, at most STAGE_RINGS per device: a call holds one while it copies
// and gives it back; a call that finds none free takes the runtime's copy. They are freed with
// the device's last context.
constexpr size_t STAGE_BYTES = 4u << 20, STAGE_MIN = 2048, STAGE_IN_MIN = 32u << 10, STAGE_ONE = 256u << 10;
constexpr size_t STAGE_FRESH = 768u << 10, STAGE_LARGE = 2u << 20;
constexpr int STAGE_RINGS = 4;
struct StagePool {
    std::mutex mu;
    std::vector<char*> free;
    int made = 0, users = 0;
};
StagePool g_stage[64];   // per device
TeamRoom g_team_room[64];   // likewise
TeamRoom* team_room_of(int device) { return device >= 0 && device < 64 ? &g_team_room[device] : nullptr; }
StagePool* stage_pool(int device) { return device >= 0 && device < 64 ? &g_stage[device] : nullptr; }

// the current device's ring for this call, or null
char* stage_acquire(int device) {
    StagePool* P = stage_pool(device);
    if (!P) return nullptr;
    {
        std::lock_guard<std::mutex> lk(P->mu);
        if (!P->free.empty()) {
            char* r = P->free.back();
            P->free.pop_back();
            return r;
        }
        if (P->made >= STAGE_RINGS) return nullptr;
        P->made++;
    }
    char* r = nullptr;
    if (hipHostMalloc(&r, STAGE_BYTES) == hipSuccess) return r;
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lk(P->mu);
    P->made--;
    return nullptr;
}
void stage_release(int device, char* r) {   // nothing queued reads or writes it
    StagePool* P = stage_pool(device);
    std::lock_guard<std::mutex> lk(P->mu);
    P->free.push_back(r);
}
void stage_join(int device) {
    if (StagePool* P = stage_pool(device)) {
        std::lock_guard<std::mutex> lk(P->mu);
        P->users++;
    }
}
void stage_leave(int device) {   // with the device current
    StagePool* P = stage_pool(device);
    if (!P) return;
    std::vector<char*> drop;
    {
        std::lock_guard<std::mutex> lk(P->mu);
        if (--P->users > 0) return;
        drop.swap(P->free);
        P->made -= (int)drop.size();
    }
    for (char* r : drop) (void)hipHostFree(r);
}

// ordinary pageable memory (anything else, pinned or on a device, is the runtime's to copy)
bool pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}
// The whole pages of [p, p + bytes), if there are enough of them for a call of their own.
constexpr uintptr_t HOST_PAGE = 4096;
bool whole_pages(const void* p, size_t bytes, uintptr_t* a, uintptr_t* b) {
    *a = (reinterpret_cast<uintptr_t>(p) + HOST_PAGE - 1) & ~(HOST_PAGE - 1);
    *b = (reinterpret_cast<uintptr_t>(p) + bytes) & ~(HOST_PAGE - 1);
    return *b >= *a + 16 * HOST_PAGE;
}
// Whether the first of them is not mapped yet.
bool fresh_pages(const void* p, size_t bytes) {
    uintptr_t a, b;
    unsigned char there = 0;
    return whole_pages(p, bytes, &a, &b) && mincore(reinterpret_cast<void*>(a), HOST_PAGE, &there) == 0 && !(there & 1);
}
// Maps them if the first is not mapped yet; their contents stay.
void map_pages(void* p, size_t bytes) {
    constexpr int POPULATE_WRITE = 23;   // MADV_POPULATE_WRITE (Linux 5.14; an older kernel refuses it)
    uintptr_t a, b;
    if (fresh_pages(p, bytes) && whole_pages(p, bytes, &a, &b))
        (void)madvise(reinterpret_cast<void*>(a), b - a, POPULATE_WRITE);
}

struct HostCopy { char* host; char* dev; size_t bytes; };

// The parts through a ring on the stream; complete on return. The events are the context's own: they
// end with its stream.
hipError_t copy_parts(mdn_ctx* ctx, const HostCopy* parts, int np, bool to_host) {
    size_t total = 0;
    for (int i = 0; i < np; i++) total += parts[i].bytes;
    // the ring's kernels and events belong to the calling thread's current device: on another one than
    // the context's (entry points that only read leave it as it is) the runtime copies
    int current = -1;
    hipError_t e = hipGetDevice(&current);
    char* r = total && e == hipSuccess && current == ctx->device ? stage_acquire(ctx->device) : nullptr;
    e = hipSuccess;
    if (!r) {
        for (int i = 0; i < np && e == hipSuccess; i++)
            e = to_host ? hipMemcpyAsync(parts[i].host, parts[i].dev, parts[i].bytes, hipMemcpyDeviceToHost, ctx->stream)
                        : hipMemcpyAsync(parts[i].dev, parts[i].host, parts[i].bytes, hipMemcpyHostToDevice, ctx->stream);
        return e == hipSuccess ? hipStreamSynchronize(ctx->stream) : e;
    }
    const size_t chunk = total <= STAGE_LARGE ? STAGE_ONE : 1u << 20;
    const int slots = (int)(STAGE_BYTES / chunk);
    struct Slot { HostCopy piece[COPY_PIECES]; size_t at[COPY_PIECES]; int n; } S[STAGE_SLOTS];
    int part = 0, put = 0, got = 0;   // slots filled and emptied
    size_t from = 0;
    auto fill = [&](int k) {   // the next chunk's pieces into slot k
        Slot& sl = S[k];
        sl.n = 0;
        for (size_t used = 0; part < np && sl.n < COPY_PIECES && used < chunk;) {
            const HostCopy& c = parts[part];
            const size_t len = std::min(c.bytes - from, chunk - used);
            if (len) {
                sl.piece[sl.n] = HostCopy{c.host + from, c.dev + from, len};
                sl.at[sl.n++] = k * chunk + used;
            }
            used += (len + 15) & ~(size_t)15;
            from += len;
            if (from == c.bytes) { part++; from = 0; }
        }
        CopyPieces cp;
        size_t most = 0;
        for (int q = 0; q < sl.n; q++) {
            char* pin = r + sl.at[q];
            if (!to_host) memcpy(pin, sl.piece[q].host, sl.piece[q].bytes);
            cp.src[q] = to_host ? sl.piece[q].dev : pin;
            cp.dst[q] = to_host ? pin : sl.piece[q].dev;
            cp.bytes[q] = (unsigned)sl.piece[q].bytes;
            most = std::max(most, sl.piece[q].bytes);
        }
        if (sl.n == 0) return;
        if (!ctx->stage_ev[k] && (e = hipEventCreateWithFlags(&ctx->stage_ev[k], hipEventDisableTiming)) != hipSuccess) return;
        hipLaunchKernelGGL(k_copy_pieces, dim3((unsigned)std::min<size_t>(32, (most + 16 * BLOCK - 1) / (16 * BLOCK)), sl.n),
                           dim3(BLOCK), 0, ctx->stream, cp);
        if ((e = hipGetLastError()) == hipSuccess) e = hipEventRecord(ctx->stage_ev[k], ctx->stream);
    };
    while (e == hipSuccess && (part < np || got < put)) {
        if (part < np && put - got < slots) {
            fill(put++ % slots);
            continue;
        }
        const int k = got++ % slots;
        if (S[k].n == 0) continue;
        if ((e = hipEventSynchronize(ctx->stage_ev[k])) != hipSuccess || !to_host) continue;
        for (int q = 0; q < S[k].n; q++) {
            map_pages(S[k].piece[q].host, S[k].piece[q].bytes);
            memcpy(S[k].piece[q].host, r + S[k].at[q], S[k].piece[q].bytes);
        }
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(ctx->stream);
    stage_release(ctx->device, r);
    return e;
}

// Host data onto the device: queued, or (ring) complete on return.
hipError_t copy_in(mdn_ctx* ctx, void* dev, const void* host, size_t bytes, bool ring = false) {
    if (!ring || bytes < STAGE_IN_MIN || bytes > STAGE_ONE || !pageable(host))
        return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream);
    const HostCopy c{const_cast<char*>(static_cast<const char*>(host)), static_cast<char*>(dev), bytes};
    return copy_parts(ctx, &c, 1, false);
}
// Device data to the host after everything queued on the stream; complete on return.
hipError_t copy_out(mdn_ctx* ctx, void* host, const void* dev, size_t bytes) {
    const bool ring = bytes <= STAGE_ONE ? bytes >= STAGE_MIN
                                         : bytes > STAGE_LARGE || (bytes >= STAGE_FRESH && fresh_pages(host, bytes));
    if (!ring || !pageable(host)) return d2h(ctx, host, dev, bytes);
    const HostCopy c{static_cast<char*>(host), const_cast<char*>(static_cast<const char*>(dev)), bytes};
    return copy_parts(ctx, &c, 1, true);
}

bool call_limit_host(const CgState& S) {
    return (S.energy_call_limit != 0 && S.num_energy_call > S.energy_call_limit) ||
           (S.force_call_limit != 0 && S.num_force_call > S.force_call_limit);
}

template <typename T>
hipError_t upload(mdn_ctx* ctx, DBuf<T>& b, const std::vector<T>& v) {
    hipError_t e = b.ensure(v.size());
    if (e != hipSuccess) return e;
    if (!v.empty()) e = copy_in(ctx, b.p, v.data(), v.size() * sizeof(T));
    return e;
}

int ceil_div(long a, long b) { return (int)((a + b - 1) / b); }
const int VSTAT_BLOCKS = 1024;   // grid of k_vec_stats

// Block and slot layout of the term / bead grids for the current interaction counts.
void layout(mdn_ctx* ctx) {
    DevSys& s = ctx->sys;
    s.n_beads = ctx->n_beads;
    // the longest-running blocks are dispatched first (excluded volume, crosslinks, boundary,
    // then the bonded terms): on grids larger than the chip holds at once, the cheap bonded
    // blocks then fill in around them instead of delaying them to the kernel's tail
    static const int order[NFF] = {FF_EXVOL, FF_LINKER, FF_MOTOR, FF_BOUNDARY, FF_BEND, FF_STRETCH};
    s.blk[0] = 0;
    for (int k = 0; k < NFF; k++) {
        s.dff[k] = order[k];
        s.fblk[order[k]] = s.blk[k];
        s.blk[k + 1] = s.blk[k] + ceil_div(s.n[order[k]], BLOCK);
    }
    s.slot0[0] = 0;
    for (int ff = 0; ff < NFF; ff++) s.slot0[ff + 1] = s.slot0[ff] + (long)SLOTS_PER_TERM[ff] * s.n[ff];
    s.blk[NFF + 1] = s.blk[NFF] + ceil_div(ctx->n_beads, BLOCK);
    s.nbb = std::max(1, ceil_div(ctx->n_beads, BLOCK));
    s.lsp = s.blk[NFF] + 2 * s.nbb;
    s.blk_nb = s.blk[4];   // excluded volume, linkers, motors, boundary
    // Force evaluations use the bonded sums (bead blocks in the terms kernel's grid recompute the
    // filament terms' forces per bead, which saves writing and re-reading five piece vectors per
    // bead); the minimizer chooses per precision (cg_bonded_sums). The same values either way; a
    // context can fix every choice (bonded_gather_mode).
    s.bonded_gather = 0;   // set per precision on the minimizer's copy (cg_sys)
    ctx->bg_eval = ctx->bonded_gather_mode >= 0 ? ctx->bonded_gather_mode : 1;
}

int bead_blocks(mdn_ctx* ctx) { return std::max(1, ceil_div(ctx->n_beads, BLOCK)); }
int gather_size(mdn_ctx* ctx) { return ctx->n_beads >= GB_LARGE_BEADS ? 128 : 64; }
int gather_blocks(mdn_ctx* ctx) { return std::max(1, ceil_div(ctx->n_beads, gather_size(ctx))); }
// the gather kernels at the context's beads-per-block
template <typename R>
void launch_gather_plain(mdn_ctx* ctx, const DevSys& s, int bmask, const R* slots, long lo, long hi, const double* base,
                         double* out, bool bg, const int* bad = nullptr) {
    int* host = ctx->h_int;
    const dim3 g(gather_blocks(ctx)), b(BLOCK);
    const bool l = gather_size(ctx) == 128;
    if (bg && l)
        hipLaunchKernelGGL((k_gather_plain<R, 128, true>), g, b, 0, ctx->stream, s, bmask, slots, lo, hi, base, out, bad,
                           host);
    else if (bg)
        hipLaunchKernelGGL((k_gather_plain<R, 64, true>), g, b, 0, ctx->stream, s, bmask, slots, lo, hi, base, out, bad,
                           host);
    else if (l)
        hipLaunchKernelGGL((k_gather_plain<R, 128, false>), g, b, 0, ctx->stream, s, bmask, slots, lo, hi, base, out, bad,
                           host);
    else
        hipLaunchKernelGGL((k_gather_plain<R, 64, false>), g, b, 0, ctx->stream, s, bmask, slots, lo, hi, base, out, bad,
                           host);
}
// The terms kernel's grid: every interaction block (pieces: the filament terms write their
// pieces), or the other force fields' blocks followed by the bead blocks of the bonded sums.
int force_blocks(const DevSys& s, bool pieces) { return pieces ? s.blk[NFF] : s.blk_nb + ceil_div(s.n_beads, BLOCK); }
int bead_block0(const DevSys& s, bool pieces) { return pieces ? -1 : s.blk_nb; }
template <typename R>
void launch_cg_gather(mdn_ctx* ctx, const DevSys& s, const CgState* st, const CgBufs& B) {
    const dim3 g(gather_blocks(ctx)), b(BLOCK);
    const bool l = gather_size(ctx) == 128, bg = s.bonded_gather != 0;
    if (bg && l) hipLaunchKernelGGL((k_cg_gather<R, 128, true>), g, b, 0, ctx->stream, s, st, B);
    else if (bg) hipLaunchKernelGGL((k_cg_gather<R, 64, true>), g, b, 0, ctx->stream, s, st, B);
    else if (l) hipLaunchKernelGGL((k_cg_gather<R, 128, false>), g, b, 0, ctx->stream, s, st, B);
    else hipLaunchKernelGGL((k_cg_gather<R, 64, false>), g, b, 0, ctx->stream, s, st, B);
}

void refresh_ptrs(mdn_ctx* ctx) {
    DevSys& s = ctx->sys;
    s.str_b = ctx->str_b.p; s.str_k = ctx->str_k.p; s.str_eql = ctx->str_eql.p;
    s.bend_b = ctx->bend_b.p; s.bend_k = ctx->bend_k.p; s.bend_eqt = ctx->bend_eqt.p;
    s.lnk_b = ctx->lnk_b.p; s.lnk_k = ctx->lnk_k.p; s.lnk_eql = ctx->lnk_eql.p; s.lnk_p1 = ctx->lnk_p1.p;
    s.lnk_p2 = ctx->lnk_p2.p; s.lnk_sf = ctx->lnk_sf.p;
    s.lnk_ord = ctx->lnk_ord.p; s.mot_ord = ctx->mot_ord.p;
    s.mot_b = ctx->mot_b.p; s.mot_k = ctx->mot_k.p; s.mot_eql = ctx->mot_eql.p; s.mot_p1 = ctx->mot_p1.p;
    s.mot_p2 = ctx->mot_p2.p; s.mot_sf = ctx->mot_sf.p;
    s.ev_b = ctx->ev_b.p; s.ev_ks = ctx->ev_ks.p;
    s.bnd_b = ctx->bnd_b.p; s.bnd_e = ctx->bnd_e.p; s.bnd_krep = ctx->bnd_krep.p; s.bnd_slen = ctx->bnd_slen.p;
    s.piece = (void*)ctx->piece.p; s.pmask = ctx->pmask.p;
    s.bnbr = ctx->bnbr.p; s.bterm = ctx->bterm.p; s.bsum = ctx->bsum.p;
    s.pos = ctx->pos.p; s.bstart = ctx->bstart.p; s.sorted_id = ctx->sorted_id.p;
    s.defer = ctx->defer.p; s.defer_n = ctx->defer_n.p;
    s.n_elem = (int)ctx->elems.size();
    for (int e = 0; e < s.n_elem; e++) {
        s.elem[e].kind = ctx->elems[e].kind;
        for (int q = 0; q < 4; q++) s.elem[e].p[q] = ctx->elems[e].p[q];
    }
}

// Size the per-evaluation buffers (slots, partials) for the current layout.
int ensure_eval_buffers(mdn_ctx* ctx) {
    const DevSys& s = ctx->sys;
    // padded by one gather chunk: the gather's chunk loads are unconditional
    HIPCHK(ctx->slots.ensure(3 * (size_t)std::max(1L, s.slot0[NFF]) + GCHUNK_PAD));
    // line-search partials (interaction blocks, then the line search's and the bead kernel's bead
    // blocks; this also covers the evaluation partials), then the CG gather's
    const long nls = (long)s.lsp;
    HIPCHK(ctx->partial.ensure((size_t)(nls + gather_blocks(ctx) + 1) * PSTRIDE));
    // the persistent minimizer's partials, for a network minimized alone or in a batch
    if (ctx->n_beads < GB_LARGE_BEADS)
        HIPCHK(ctx->team_part.ensure((size_t)std::max(team_wpart_doubles(s, SUM_SLOTS), team_wpart_doubles(s, SUM_STRIDED))));
    HIPCHK(ctx->pos.ensure((size_t)std::max(1L, s.slot0[NFF])));
    HIPCHK(ctx->sorted_id.ensure((size_t)std::max(1L, s.slot0[NFF])));
    HIPCHK(ctx->bad_list.ensure((size_t)std::max(1, s.n[FF_EXVOL])));
    return MDN_OK;
}

// The tile edge of the list kernel: the largest of 8, 4, 2 bins that still gives 1024 tiles (a
// workgroup each), so that small grids keep the chip busy, and whose halo holds on average at most
// half of what is staged in LDS: a halo beyond that is read from global memory, where a build took
// three times as long (420,000 beads, T = 4 and 8 at twice the bin width: 420 and 1,250 us).
void nl_tiles(NLDev& n) {
    const double per_bin = n.n_cyl / ((double)n.nb[0] * n.nb[1] * n.nb[2]);
    for (int T = 8, lt = 3; T >= 2; T /= 2, lt--) {
        n.T = T;
        n.lt = lt;
        long tiles = 1;
        for (int q = 0; q < 3; q++) {
            n.nt[q] = (n.nb[q] + T - 1) / T;
            tiles *= n.nt[q];
        }
        if (tiles >= 1024 && per_bin * (T + 2) * (T + 2) * (T + 2) <= NL_CAP / 2) break;
    }
}

// The bins of a list with n's range: 1.125 ranges wide (HybridNeighborListImpl.cpp:180).
void nl_grid(mdn_ctx* ctx, NLDev& n) {
    n.side = 1.125 * std::sqrt(n.rmaxsq);
    for (int q = 0; q < 3; q++) {
        n.grid[q] = ctx->grid[q];
        n.nb[q] = std::max(1, (int)std::ceil(ctx->grid[q] / n.side));
    }
    nl_tiles(n);
}

NLDev nl_view(mdn_ctx* ctx) {
    NLDev n{};
    n.n_cyl = ctx->n_cyl;
    n.cyl_b1 = ctx->d_cyl_b1.p; n.cyl_b2 = ctx->d_cyl_b2.p; n.cyl_fil = ctx->d_cyl_fil.p;
    n.cyl_pos = ctx->d_cyl_pos.p; n.cyl_type = ctx->d_cyl_type.p;
    n.cyl_kexvol = ctx->d_cyl_kexvol.p; n.cyl_eql = ctx->d_cyl_eql.p; n.cyl_minus = ctx->d_cyl_minus.p;
    // setneighborsearchparameters(..., float rMax, float rMin): squares formed in float
    // (HybridNeighborListImpl.h:74-80)
    float rmaxf = (float)ctx->rmax, rminf = (float)ctx->rmin;
    float rmaxsq = rmaxf * rmaxf, rminsq = rminf * rminf;
    n.rmaxsq = rmaxsq;
    n.rminsq = rminsq;
    n.ta = n.tb = -1;
    nl_grid(ctx, n);
    return n;
}

int exclusive_scan(mdn_ctx* ctx, const int* in, int* out, long n) {
    size_t bytes = 0;
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, ctx->stream));
    HIPCHK(ctx->cub_tmp.ensure(bytes));
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(ctx->cub_tmp.p, bytes, in, out, (int)n, ctx->stream));
    return MDN_OK;
}

int need_system(mdn_ctx* ctx, bool need_nl) {
    if (!ctx) return MDN_ERR_ARG;
    if (!ctx->uploaded) return fail(ctx, MDN_ERR_STATE, "no system uploaded (mdn_system_upload)");
    if (need_nl && !ctx->nl_built) return fail(ctx, MDN_ERR_STATE, "neighbor lists not built (mdn_nl_build)");
    return MDN_OK;
}

int set_coords_dev(mdn_ctx* ctx, const double* coord) {
    if (coord)
        HIPCHK(copy_in(ctx, ctx->x[ctx->cur].p, coord, sizeof(double) * 3 * ctx->n_beads));
    return MDN_OK;
}

// The term kernel at device coordinates x into slots (in the arithmetic type R); the pairs whose
// closed-form forces are non-finite are counted and listed. pieces: the filament terms' pieces for
// a gather that reads them; else the bonded sums of the pieces selected by bmask on top of base
// (null: zero) for a gather that starts from them.
template <typename R>
void launch_terms(mdn_ctx* ctx, const DevSys& s, const double* x, R* slots, bool pieces, int bmask, const double* base,
                  int* bad_count, int* bad_list) {
    if (force_blocks(s, pieces) > 0)
        hipLaunchKernelGGL(k_forces_terms<R>, dim3(force_blocks(s, pieces)), dim3(BLOCK), 0, ctx->stream, s, x, slots,
                           bad_count, bad_list, bead_block0(s, pieces), bmask, base);
}

constexpr int FORCEN_BLOCKS = 240;

// forceN (FP64 in both paths) for the nbad listed pairs, into their slots: retried once with beads
// 1 and 2 moved out of plane (CylinderExclVolRepulsion.cpp:1198-1204). Each pair writes only its
// own slots, so the order does not matter.
template <typename R>
int settle_pairs(mdn_ctx* ctx, const DevSys& s, const double* x, R* slots, const int* bad_list, int nbad,
                 double* partial, int* ok_dev) {
    for (int i = 0; i < nbad; i++) {
        HIPCHK(d2h(ctx, ctx->h_int + 1, bad_list + i, sizeof(int)));
        const int t = ctx->h_int[1];
        int ok = 0;
        for (int mv = 0; mv < 2 && !ok; mv++) {
            hipLaunchKernelGGL(k_exvol_forceN_rows, dim3(FORCEN_BLOCKS), dim3(BLOCK), 0, ctx->stream, s, x, t, mv,
                               partial);
            hipLaunchKernelGGL(k_exvol_forceN_finish<R>, dim3(1), dim3(64), 0, ctx->stream, s, x, t, mv,
                               FORCEN_BLOCKS, (const double*)partial, slots, ok_dev);
            HIPCHK(hipGetLastError());
            HIPCHK(d2h(ctx, ctx->h_int + 2, ok_dev, sizeof(int)));
            ok = ctx->h_int[2];
        }
        if (!ok)
            return fail(ctx, MDN_ERR_NONFINITE,
                        "excluded-volume pair %d: force non-finite after the numerical fallback", t);
    }
    return MDN_OK;
}
int settle_pairs(mdn_ctx* ctx, const double* x, int prec, int nbad) {
    HIPCHK(ctx->fallback_partial.ensure(6 * FORCEN_BLOCKS));
    HIPCHK(ctx->fallback_ok.ensure(1));
    const DevSys& s = ctx->sys;
    return prec == MDN_PREC_MIXED
               ? settle_pairs<float>(ctx, s, x, (float*)ctx->slots.p, ctx->bad_list.p, nbad, ctx->fallback_partial.p,
                                     ctx->fallback_ok.p)
               : settle_pairs<double>(ctx, s, x, ctx->slots.p, ctx->bad_list.p, nbad, ctx->fallback_partial.p,
                                      ctx->fallback_ok.p);
}

// Term forces at x with the fallback settled, into ctx->slots (synchronous).
int eval_slots(mdn_ctx* ctx, const double* x, int prec, bool pieces) {
    HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
    if (prec == MDN_PREC_MIXED)
        launch_terms<float>(ctx, ctx->sys, x, (float*)ctx->slots.p, pieces, 3, nullptr, ctx->bad_count.p, ctx->bad_list.p);
    else
        launch_terms<double>(ctx, ctx->sys, x, ctx->slots.p, pieces, 3, nullptr, ctx->bad_count.p, ctx->bad_list.p);
    HIPCHK(hipGetLastError());
    HIPCHK(d2h(ctx, ctx->h_int, ctx->bad_count.p, sizeof(int)));
    return ctx->h_int[0] ? settle_pairs(ctx, x, prec, ctx->h_int[0]) : MDN_OK;
}

// One force evaluation at device coordinates x into out: base + the bonded pieces selected by
// bmask (bit 0 stretching, bit 1 bending) + the slots with id in [lo, hi). start() queues the terms
// and the gather, before the host knows whether a pair needs the numerical fallback (rare: the
// gather then writes nothing); after the caller's wait finish() settles those pairs and queues
// the gather again. So an evaluation costs one wait.
struct ForceEval {
    mdn_ctx* ctx;
    const double* x;
    int prec, bmask;
    long lo, hi;
    const double* base;
    double* out;

    void gather(const int* bad) {
        const bool bg = ctx->bg_eval != 0;
        if (prec == MDN_PREC_MIXED)
            launch_gather_plain<float>(ctx, ctx->sys, bmask, (const float*)ctx->slots.p, lo, hi, base, out, bg, bad);
        else
            launch_gather_plain<double>(ctx, ctx->sys, bmask, (const double*)ctx->slots.p, lo, hi, base, out, bg, bad);
    }
    int start() {
        const bool pieces = ctx->bg_eval == 0;
        HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
        if (prec == MDN_PREC_MIXED)
            launch_terms<float>(ctx, ctx->sys, x, (float*)ctx->slots.p, pieces, bmask, base, ctx->bad_count.p,
                                ctx->bad_list.p);
        else
            launch_terms<double>(ctx, ctx->sys, x, ctx->slots.p, pieces, bmask, base, ctx->bad_count.p, ctx->bad_list.p);
        gather(ctx->bad_count.p);
        HIPCHK(hipGetLastError());
        return MDN_OK;
    }
    // after a synchronization of the stream: *redone when the forces were gathered again (queued)
    int finish(bool* redone) {
        *redone = ctx->h_int[0] != 0;
        if (!*redone) return MDN_OK;
        const int st = settle_pairs(ctx, x, prec, ctx->h_int[0]);
        if (st) return st;
        gather(nullptr);
        HIPCHK(hipGetLastError());
        return MDN_OK;
    }
};

// Per-FF energies at device coordinates x into out[0..8] (pinned host memory), queued.
void launch_energy(mdn_ctx* ctx, const double* x, int prec, double* out) {
    const DevSys& s = ctx->sys;
    int grid = std::max(1, s.blk[NFF]);
    if (prec == MDN_PREC_MIXED)
        hipLaunchKernelGGL(k_energy_report<float>, dim3(grid), dim3(BLOCK), 0, ctx->stream, s, x, ctx->partial.p);
    else
        hipLaunchKernelGGL(k_energy_report<double>, dim3(grid), dim3(BLOCK), 0, ctx->stream, s, x, ctx->partial.p);
    hipLaunchKernelGGL(k_energy_report_fin, dim3(1), dim3(BLOCK), 0, ctx->stream, s, (const double*)ctx->partial.p, out);
}
int check_energy(mdn_ctx* ctx, const double* e) {
    if (e[8] != 0.0)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%.0f excluded-volume pairs need the Simpson energy (capacity %d)", e[8],
                    DEFER_CAP);
    return MDN_OK;
}

// Per-FF energies at device coordinates x into ctx->h_eout[0..8] (synchronous).
int energy_report(mdn_ctx* ctx, const double* x, int prec) {
    launch_energy(ctx, x, prec, ctx->h_eout);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return check_energy(ctx, ctx->h_eout);
}

void fill_report(const double* e, mdn_energy_report* out) {
    for (int ff = 0; ff < NFF; ff++) out->ff[ff] = e[ff];
    out->total = e[6];
}

}  // namespace

// =========================================================================================
// C ABI
// =========================================================================================
extern "C" {

int mdn_abi_version(void) { return MDN_ABI_VERSION; }

const char* mdn_last_error(const mdn_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int mdn_ctx_create(int device, mdn_ctx** out) {
    if (!out) return MDN_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return MDN_ERR_HIP;
    if (device < 0 || device >= n) return MDN_ERR_ARG;
    mdn_ctx* ctx = new mdn_ctx();
    ctx->device = device;
    // MDN_BONDED_GATHER=0 / 1 at context creation fixes whether the filament terms' forces go
    // through per-bead bonded sums (1) or the piece arrays (0), for force evaluations and the
    // minimizer alike; unset: the measured defaults (layout, cg_bonded_sums)
    if (const char* env = getenv("MDN_BONDED_GATHER")) ctx->bonded_gather_mode = atoi(env) != 0 ? 1 : 0;
    // MDN_CG_GRAPH=0 at context creation: the minimizer launches each batch of slots directly
    // instead of replaying a captured graph (the same kernels and decisions; for tools that do
    // not follow graph launches)
    if (const char* env = getenv("MDN_CG_GRAPH")) ctx->use_graph = atoi(env) != 0;
    // MDN_CG_TEAM at context creation: 0 = always the four-kernel slots, n = a team of n
    // workgroups of one XCD for every network; unset: by the network's size (team_workgroups)
    // (the result does not depend on it)
    if (const char* env = getenv("MDN_CG_TEAM")) ctx->team_size = std::max(0, std::min(TEAM_MAX, atoi(env)));
    // for tests, at context creation: MDN_TEAM_POLLS = a team's wait for its workgroups at the start,
    // in polls (0: whoever is not the last gives up, -1: everyone does); MDN_TEAM_STRIDE = the distance of a single network's team
    // members in the grid (8: one XCD; 1: spread over all of them). The result depends on neither.
    if (const char* env = getenv("MDN_TEAM_POLLS")) ctx->team_polls = std::max(-1, std::min(TEAM_START_POLLS, atoi(env)));
    if (const char* env = getenv("MDN_TEAM_STRIDE")) ctx->team_stride = std::max(1, std::min(8, atoi(env)));
    if (hipSetDevice(device) != hipSuccess ||
        hipDeviceGetAttribute(&ctx->n_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return MDN_ERR_HIP;
    }
    if (scratch_lookup(device) != hipSuccess) {   // the no-allocation entry point's array
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return MDN_ERR_HIP;
    }
    if (hipHostMalloc(&ctx->h_cg, CG_BYTES) != hipSuccess ||
        hipHostMalloc(&ctx->h_eout, sizeof(double) * 32) != hipSuccess ||
        hipHostMalloc(&ctx->h_int, sizeof(int) * 16) != hipSuccess) {
        delete ctx;
        return MDN_ERR_HIP;
    }
    if (ctx->ticket.ensure(8) != hipSuccess || ctx->eout.ensure(32) != hipSuccess ||
        ctx->vstat.ensure(2 * VSTAT_BLOCKS) != hipSuccess ||
        ctx->bad_count.ensure(1) != hipSuccess || ctx->cg.ensure(CG_BYTES / sizeof(CgState) + 1) != hipSuccess ||
        ctx->defer.ensure(DEFER_CAP) != hipSuccess ||
        ctx->defer_n.ensure(1) != hipSuccess) {
        delete ctx;
        return MDN_ERR_HIP;
    }
    (void)hipMemset(ctx->ticket.p, 0, sizeof(unsigned) * 8);
    (void)hipMemset(ctx->defer_n.p, 0, sizeof(int));
    stage_join(device);
    if (char* r = stage_acquire(device)) stage_release(device, r);   // made before the first call needs it
    *out = ctx;
    return MDN_OK;
}

int mdn_ctx_destroy(mdn_ctx* ctx) {
    if (!ctx) return MDN_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    for (int q = 0; q < 2; q++) {
        if (ctx->graph_exec[q]) (void)hipGraphExecDestroy(ctx->graph_exec[q]);
        if (ctx->graph[q]) (void)hipGraphDestroy(ctx->graph[q]);
    }
    DBuf<int>* ib[] = {&ctx->str_b, &ctx->bend_b, &ctx->lnk_b, &ctx->mot_b, &ctx->lnk_ord, &ctx->mot_ord, &ctx->ev_b,
                       &ctx->bnd_b, &ctx->bnd_e,
                       &ctx->inc_s_start, &ctx->inc_s, &ctx->inc_cnt, &ctx->inc_list,
                       &ctx->d_cyl_b1, &ctx->d_cyl_b2, &ctx->d_cyl_fil, &ctx->d_cyl_pos,
                       &ctx->d_cyl_type, &ctx->bin, &ctx->bin_count, &ctx->bin_start, &ctx->place,
                       &ctx->nl_found, &ctx->nl_list, &ctx->nl_count, &ctx->nl_off, &ctx->pairs, &ctx->bnd_cnt, &ctx->bnd_off,
                       &ctx->bad_count, &ctx->bad_list, &ctx->fallback_ok, &ctx->bstart,
                       &ctx->sorted_id, &ctx->pos, &ctx->dof_src, &ctx->b_bin, &ctx->b_bin_count,
                       &ctx->b_bin_start, &ctx->b_place, &ctx->b_count, &ctx->b_off,
                       &ctx->b_pairs, &ctx->b_scount, &ctx->b_soff};
    ctx->members.release();
    ctx->b_members.release();
    ctx->b_mid.release();
    ctx->mmid.release();
    ctx->b_mmid.release();
    ctx->mbin.release();
    ctx->b_mbin.release();
    ctx->b_site.release();
    ctx->b_free.release();
    ctx->b_out.release();
    for (auto* b : ib) b->release();
    DBuf<double>* db[] = {&ctx->str_k, &ctx->str_eql, &ctx->bend_k, &ctx->bend_eqt, &ctx->lnk_k, &ctx->lnk_eql,
                          &ctx->lnk_p1, &ctx->lnk_p2, &ctx->lnk_sf, &ctx->mot_k, &ctx->mot_eql, &ctx->mot_p1,
                          &ctx->mot_p2, &ctx->mot_sf, &ctx->ev_ks, &ctx->bnd_krep, &ctx->bnd_slen,
                          &ctx->d_cyl_kexvol, &ctx->d_cyl_eql, &ctx->d_krep_e, &ctx->d_slen_e, &ctx->mid,
                          &ctx->x[0], &ctx->x[1], &ctx->f, &ctx->f2, &ctx->xh, &ctx->d[0], &ctx->d[1],
                          &ctx->xmin[0], &ctx->xmin[1], &ctx->scratch_f, &ctx->ext, &ctx->partial, &ctx->eout,
                          &ctx->vstat, &ctx->fallback_partial, &ctx->dof_next, &ctx->dof_new};
    for (auto* b : db) b->release();
    ctx->d_cyl_minus.release();
    ctx->d_fil_ends.release();
    ctx->load_out.release();
    ctx->pmask.release();
    ctx->bnbr.release();
    ctx->bterm.release();
    ctx->bsum.release();
    ctx->d_cyl_bend.release();
    ctx->ev_U.release();
    ctx->grad_out.release();
    ctx->tan_v.release();
    ctx->hb_v.release();
    ctx->hb_slots.release();
    ctx->hb_piece.release();
    ctx->hb_out.release();
    ctx->piece.release();
    ctx->cub_tmp.release();
    ctx->slots.release();
    ctx->ticket.release();
    ctx->defer.release();
    ctx->defer_n.release();
    ctx->team_part.release();
    ctx->batch_slot.release();
    ctx->batch_team.release();
    ctx->batch_ctl.release();
    ctx->batch_items.release();
    ctx->batch_states.release();
    ctx->batch_reports.release();
    ctx->batch_order.release();
    ctx->batch_queue.release();
    ctx->batch_copy.release();
    ctx->cg.release();
    if (ctx->h_cg) (void)hipHostFree(ctx->h_cg);
    if (ctx->h_eout) (void)hipHostFree(ctx->h_eout);
    if (ctx->h_int) (void)hipHostFree(ctx->h_int);
    for (hipEvent_t e : ctx->stage_ev)
        if (e) (void)hipEventDestroy(e);
    stage_leave(ctx->device);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return MDN_OK;
}

int relayout(mdn_ctx* ctx);

// LinkerStretching / MotorGhostStretching::vectorize (LinkerStretching.cpp:30-57,
// MotorGhostStretching.cpp:30-57): the crosslink tables (beads of both cylinders, k, rest length,
// binding positions) and the static slot incidence, per bead the crosslink slots in ascending
// slot order. The counts are set and the block / slot layout recomputed; the merged bead-sorted
// layout is then stale until relayout (or the next neighbor-list build). Indices are validated
// by the callers.
int set_crosslinks(mdn_ctx* ctx, const mdn_crosslink* linkers, int n_linkers, const mdn_crosslink* motors,
                   int n_motors) {
    DevSys& s = ctx->sys;
    std::vector<int> xb[2];
    std::vector<double> xk[2], xe[2], xp1[2], xp2[2];
    for (int w = 0; w < 2; w++) {
        const int n = w ? n_motors : n_linkers;
        const mdn_crosslink* xl = w ? motors : linkers;
        xb[w].resize(4 * (size_t)n);
        xk[w].resize(n); xe[w].resize(n); xp1[w].resize(n); xp2[w].resize(n);
        for (int j = 0; j < n; j++) {
            const int c1 = xl[j].cyl1, c2 = xl[j].cyl2;
            xb[w][4 * j] = ctx->cyl_b1[c1]; xb[w][4 * j + 1] = ctx->cyl_b2[c1];
            xb[w][4 * j + 2] = ctx->cyl_b1[c2]; xb[w][4 * j + 3] = ctx->cyl_b2[c2];
            xk[w][j] = xl[j].kstr; xe[w][j] = xl[j].eql; xp1[w][j] = xl[j].pos1; xp2[w][j] = xl[j].pos2;
        }
    }
    s.n[FF_LINKER] = n_linkers;
    s.n[FF_MOTOR] = n_motors;
    layout(ctx);
    if (s.slot0[NFF] > 0x7fffffffL) return fail(ctx, MDN_ERR_UNSUPPORTED, "too many interactions");
    // static incidence CSR: per bead, slots of linkers / motors ascending
    std::vector<int> cnt(ctx->n_beads + 1, 0);
    auto each_static = [&](auto&& fn) {
        for (int w = 0; w < 2; w++)
            for (size_t t = 0; t < xk[w].size(); t++)
                for (int q = 0; q < 4; q++) fn(xb[w][4 * t + q], s.slot0[2 + w] + 4L * t + q);
    };
    each_static([&](int b, long) { cnt[b + 1]++; });
    for (int b = 0; b < ctx->n_beads; b++) cnt[b + 1] += cnt[b];
    std::vector<int> inc(std::max(1, cnt[ctx->n_beads]));
    {
        std::vector<int> cur(cnt.begin(), cnt.end() - 1);
        each_static([&](int b, long sl) { inc[cur[b]++] = (int)sl; });   // visited in slot order
    }
    HIPCHK(upload(ctx, ctx->inc_s_start, cnt)); HIPCHK(upload(ctx, ctx->inc_s, inc));
    // The device tables in the threads' order: by the first bead of the first cylinder (stable:
    // ties keep the interaction order); ord[i] is the crosslink's own index (its slots).
    // MDN_XL_ORDER=0 keeps the interaction order (the forces are the same).
    const char* env = getenv("MDN_XL_ORDER");
    const bool sorted = !(env && env[0] == '0');
    std::vector<int> sb[2];
    std::vector<double> sk[2], se[2], sp1[2], sp2[2];
    for (int w = 0; w < 2; w++) {
        std::vector<int>& ord = ctx->xl_ord[w];
        const size_t n = xk[w].size();
        ord.resize(n);
        for (size_t j = 0; j < n; j++) ord[j] = (int)j;
        const std::vector<int>& b = xb[w];
        if (sorted)
            std::stable_sort(ord.begin(), ord.end(), [&b](int i, int j) { return b[4 * (size_t)i] < b[4 * (size_t)j]; });
        sb[w].resize(4 * n); sk[w].resize(n); se[w].resize(n); sp1[w].resize(n); sp2[w].resize(n);
        for (size_t i = 0; i < n; i++) {
            const int t = ord[i];
            for (int q = 0; q < 4; q++) sb[w][4 * i + q] = b[4 * (size_t)t + q];
            sk[w][i] = xk[w][t]; se[w][i] = xe[w][t]; sp1[w][i] = xp1[w][t]; sp2[w][i] = xp2[w][t];
        }
    }
    for (int w = 0; w < 2; w++) {
        std::vector<int> ordu(ctx->xl_ord[w]);
        if (ordu.empty()) ordu.push_back(0);
        HIPCHK(upload(ctx, w ? ctx->mot_ord : ctx->lnk_ord, ordu));
        HIPCHK(upload(ctx, w ? ctx->mot_b : ctx->lnk_b, sb[w]));
        HIPCHK(upload(ctx, w ? ctx->mot_k : ctx->lnk_k, sk[w]));
        HIPCHK(upload(ctx, w ? ctx->mot_eql : ctx->lnk_eql, se[w]));
        HIPCHK(upload(ctx, w ? ctx->mot_p1 : ctx->lnk_p1, sp1[w]));
        HIPCHK(upload(ctx, w ? ctx->mot_p2 : ctx->lnk_p2, sp2[w]));
        HIPCHK((w ? ctx->mot_sf : ctx->lnk_sf).ensure(std::max<size_t>(1, xk[w].size())));
        HIPCHK(hipStreamSynchronize(ctx->stream));   // the host vectors above end with this scope
    }
    return MDN_OK;
}

int mdn_system_upload(mdn_ctx* ctx, const mdn_system_desc* d, const double* coord) {
    if (!ctx || !d) return fail(ctx, MDN_ERR_ARG, "null argument");
    HIPCHK(hipSetDevice(ctx->device));
    if (d->n_beads <= 0 || d->n_filaments < 0) return fail(ctx, MDN_ERR_ARG, "bad bead / filament counts");
    if (!coord && ctx->dof_next_n != d->n_beads)
        return fail(ctx, MDN_ERR_ARG, "no coordinates: coord is NULL and mdn_dof_serialize gathered %d beads, not %d",
                    ctx->dof_next_n, d->n_beads);
    if (d->n_boundary > MAXELEM) return fail(ctx, MDN_ERR_UNSUPPORTED, "at most %d boundary elements", MAXELEM);
    ctx->uploaded = ctx->nl_built = false;
    int st = MDN_OK;
    ctx->n_beads = d->n_beads;
    ctx->n_fil = d->n_filaments;
    int n_cyl = 0;
    for (int f = 0; f < d->n_filaments; f++) {
        int nb = d->fil_bead_offset[f + 1] - d->fil_bead_offset[f];
        if (nb < 2) return fail(ctx, MDN_ERR_ARG, "filament %d has %d beads (needs >= 2)", f, nb);
        n_cyl += nb - 1;
    }
    ctx->n_cyl = n_cyl;
    ctx->cyl_b1.assign(n_cyl, 0); ctx->cyl_b2.assign(n_cyl, 0); ctx->cyl_fil.assign(n_cyl, 0);
    ctx->cyl_pos.assign(n_cyl, 0); ctx->cyl_type.assign(n_cyl, 0); ctx->cyl_minus.assign(n_cyl, 0);
    ctx->cyl_kexvol.assign(n_cyl, 0); ctx->cyl_eql.assign(n_cyl, 0);
    // FilamentStretching::vectorize (FilamentStretching.cpp:26-45)
    std::vector<int> str_b(2 * (size_t)n_cyl);
    std::vector<double> str_k(n_cyl), str_eql(n_cyl);
    int c = 0;
    for (int f = 0; f < d->n_filaments; f++) {
        int off = d->fil_bead_offset[f], nb = d->fil_bead_offset[f + 1] - off;
        for (int k = 0; k < nb - 1; k++, c++) {
            int b1 = d->fil_beads[off + k], b2 = d->fil_beads[off + k + 1];
            if (b1 < 0 || b1 >= d->n_beads || b2 < 0 || b2 >= d->n_beads)
                return fail(ctx, MDN_ERR_ARG, "filament %d bead index out of range", f);
            ctx->cyl_b1[c] = b1; ctx->cyl_b2[c] = b2; ctx->cyl_fil[c] = f; ctx->cyl_pos[c] = k;
            ctx->cyl_type[c] = d->fil_type ? d->fil_type[f] : 0;
            ctx->cyl_minus[c] = (k == 0);
            ctx->cyl_kexvol[c] = d->cyl_kexvol[c];
            ctx->cyl_eql[c] = d->cyl_eql[c];
            str_b[2 * c] = b1; str_b[2 * c + 1] = b2;
            str_k[c] = d->cyl_kstr[c]; str_eql[c] = d->cyl_eql[c];
        }
    }
    // FilamentBending::vectorize (FilamentBending.cpp:29-60)
    int n_bend = n_cyl - d->n_filaments;
    std::vector<int> bend_b(3 * (size_t)std::max(0, n_bend));
    std::vector<double> bend_k(std::max(0, n_bend)), bend_eqt(std::max(0, n_bend));
    std::vector<int> cyl_bend(std::max(1, n_cyl), -1);
    ctx->bend_cyl.assign(std::max(0, n_bend), 0);
    {
        int i = 0;
        c = 0;
        for (int f = 0; f < d->n_filaments; f++) {
            int nb = d->fil_bead_offset[f + 1] - d->fil_bead_offset[f];
            for (int k = 1; k < nb - 1; k++, i++) {
                int cp = c + k - 1, cc = c + k;
                bend_b[3 * i] = ctx->cyl_b1[cp];
                bend_b[3 * i + 1] = ctx->cyl_b1[cc];
                bend_b[3 * i + 2] = ctx->cyl_b2[cc];
                bend_k[i] = d->cyl_kbend[cc];
                bend_eqt[i] = d->cyl_eqtheta[cc];
                ctx->bend_cyl[i] = cc;
                cyl_bend[cc] = i;
            }
            c += nb - 1;
        }
    }
    for (int w = 0; w < 2; w++) {
        const int n = w ? d->n_motors : d->n_linkers;
        const mdn_crosslink* xl = w ? d->motors : d->linkers;
        if (n < 0 || (n > 0 && !xl)) return fail(ctx, MDN_ERR_ARG, "bad %s table", w ? "motor" : "linker");
        for (int j = 0; j < n; j++)
            if (xl[j].cyl1 < 0 || xl[j].cyl1 >= n_cyl || xl[j].cyl2 < 0 || xl[j].cyl2 >= n_cyl)
                return fail(ctx, MDN_ERR_ARG, "%s %d: cylinder index out of range", w ? "motor" : "linker", j);
    }
    ctx->elems.assign(d->boundary, d->boundary + d->n_boundary);
    for (auto& e : ctx->elems)
        if (e.kind != MDN_BND_PLANE && e.kind != MDN_BND_SPHERE)
            return fail(ctx, MDN_ERR_ARG, "unknown boundary element kind %d", e.kind);
    ctx->bnd_cutoff = d->boundary_cutoff;
    ctx->rmax = d->exvol_rmax;
    ctx->rmin = d->exvol_rmin;
    for (int q = 0; q < 3; q++) ctx->grid[q] = d->grid_size[q];
    if (!(ctx->rmax > 0)) return fail(ctx, MDN_ERR_ARG, "exvol_rmax must be > 0");

    DevSys& s = ctx->sys;
    s = DevSys{};
    s.n[FF_STRETCH] = n_cyl;
    s.n[FF_BEND] = n_bend;
    s.n[FF_LINKER] = 0;
    s.n[FF_MOTOR] = 0;
    s.n[FF_EXVOL] = 0;
    s.n[FF_BOUNDARY] = 0;
    layout(ctx);

    // per bead, which bonded pieces it has, in the reference's per-bead order: stretching term
    // with the bead as bead 2, as bead 1; bending term as bead 3, 2, 1
    std::vector<unsigned char> pmask(ctx->n_beads, 0);
    {
        auto put = [&](int b, int k) {
            unsigned char& m = pmask[b];
            if (m & (1u << k)) return false;   // a bead listed twice in the filament tables
            m |= (unsigned char)(1u << k);
            return true;
        };
        bool ok = true;
        for (int t = 0; t < n_cyl; t++) ok = put(str_b[2 * t + 1], 0) && put(str_b[2 * t], 1) && ok;
        for (int t = 0; t < n_bend; t++)
            ok = put(bend_b[3 * t + 2], 2) && put(bend_b[3 * t + 1], 3) && put(bend_b[3 * t], 4) && ok;
        if (!ok) return fail(ctx, MDN_ERR_ARG, "a bead appears more than once in the filament bead lists");
    }
    // per bead, its neighbours along the filament and the indices of the stretching term it
    // starts and the bending term it is the middle bead of (cylinders and bending terms are
    // numbered filament after filament, as above)
    const int nbd = ctx->n_beads;
    std::vector<int> bnbr(4 * (size_t)nbd), bterm(2 * (size_t)nbd, 0);
    for (int b = 0; b < nbd; b++)
        for (int q = 0; q < 4; q++) bnbr[(size_t)q * nbd + b] = b;
    for (int f = 0; f < d->n_filaments; f++) {
        const int off = d->fil_bead_offset[f], nf = d->fil_bead_offset[f + 1] - off;
        for (int j = 0; j < nf; j++) {
            const int b = d->fil_beads[off + j];
            const int step[4] = {-2, -1, 1, 2};
            for (int q = 0; q < 4; q++)
                if (j + step[q] >= 0 && j + step[q] < nf) bnbr[(size_t)q * nbd + b] = d->fil_beads[off + j + step[q]];
            bterm[b] = off - f + j;
            bterm[(size_t)nbd + b] = off - 2 * f + j - 1;
        }
    }
    for (int t = 0; t < n_cyl; t++)   // the numbering the recomputation relies on
        if (bterm[str_b[2 * t]] != t || bnbr[2 * (size_t)nbd + str_b[2 * t]] != str_b[2 * t + 1])
            return fail(ctx, MDN_ERR_STATE, "stretching term %d: inconsistent filament tables", t);
    for (int t = 0; t < n_bend; t++)
        if (bterm[(size_t)nbd + bend_b[3 * t + 1]] != t || bnbr[(size_t)nbd + bend_b[3 * t + 1]] != bend_b[3 * t] ||
            bnbr[2 * (size_t)nbd + bend_b[3 * t + 1]] != bend_b[3 * t + 2])
            return fail(ctx, MDN_ERR_STATE, "bending term %d: inconsistent filament tables", t);
    HIPCHK(upload(ctx, ctx->bnbr, bnbr));
    HIPCHK(upload(ctx, ctx->bterm, bterm));
    {   // the bead blocks' neighbours from the indices alone when beads run filament by filament
        const int total = d->n_filaments > 0 ? d->fil_bead_offset[d->n_filaments] : 0;
        bool contig = true;
        for (int k = 0; k < total && contig; k++) contig = d->fil_beads[k] == k;
        const char* env = getenv("MDN_BEAD_TABLES");   // 1: always read the neighbour tables
        ctx->sys.bcontig = contig && !(env && env[0] == '1') ? 1 : 0;
    }
    HIPCHK(ctx->bsum.ensure(3 * (size_t)nbd));
    HIPCHK(upload(ctx, ctx->str_b, str_b)); HIPCHK(upload(ctx, ctx->str_k, str_k)); HIPCHK(upload(ctx, ctx->str_eql, str_eql));
    HIPCHK(upload(ctx, ctx->bend_b, bend_b)); HIPCHK(upload(ctx, ctx->bend_k, bend_k)); HIPCHK(upload(ctx, ctx->bend_eqt, bend_eqt));
    if ((st = set_crosslinks(ctx, d->linkers, d->n_linkers, d->motors, d->n_motors))) return st;
    HIPCHK(upload(ctx, ctx->pmask, pmask));
    HIPCHK(upload(ctx, ctx->d_cyl_bend, cyl_bend));
    HIPCHK(ctx->piece.ensure(NBOND * 3 * (size_t)ctx->n_beads));
    // cylinder tables for the neighbor lists
    HIPCHK(upload(ctx, ctx->d_cyl_b1, ctx->cyl_b1)); HIPCHK(upload(ctx, ctx->d_cyl_b2, ctx->cyl_b2));
    HIPCHK(upload(ctx, ctx->d_cyl_fil, ctx->cyl_fil)); HIPCHK(upload(ctx, ctx->d_cyl_pos, ctx->cyl_pos));
    HIPCHK(upload(ctx, ctx->d_cyl_type, ctx->cyl_type)); HIPCHK(upload(ctx, ctx->d_cyl_minus, ctx->cyl_minus));
    HIPCHK(upload(ctx, ctx->d_cyl_kexvol, ctx->cyl_kexvol)); HIPCHK(upload(ctx, ctx->d_cyl_eql, ctx->cyl_eql));
    {
        std::vector<int> ends(2 * (size_t)std::max(1, ctx->n_fil), 0);
        for (int f = 0, c0 = 0; f < ctx->n_fil; f++) {
            const int nb = d->fil_bead_offset[f + 1] - d->fil_bead_offset[f];
            ends[2 * f] = c0;               // minus-end cylinder
            ends[2 * f + 1] = c0 + nb - 2;  // plus-end cylinder
            c0 += nb - 1;
        }
        HIPCHK(upload(ctx, ctx->d_fil_ends, ends));
    }
    {
        std::vector<double> ke(ctx->elems.size()), se(ctx->elems.size());
        for (size_t e = 0; e < ctx->elems.size(); e++) { ke[e] = ctx->elems[e].krep; se[e] = ctx->elems[e].slen; }
        HIPCHK(upload(ctx, ctx->d_krep_e, ke)); HIPCHK(upload(ctx, ctx->d_slen_e, se));
    }
    // state vectors
    size_t nv = 3 * (size_t)ctx->n_beads;
    for (auto* b : {&ctx->x[0], &ctx->x[1], &ctx->f, &ctx->f2, &ctx->xh, &ctx->d[0], &ctx->d[1],
                    &ctx->xmin[0], &ctx->xmin[1], &ctx->scratch_f, &ctx->ext})
        HIPCHK(b->ensure(nv));
    ctx->cur = 0;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->x[0].p, coord, sizeof(double) * nv));
    } else {
        HIPCHK(hipMemcpyAsync(ctx->x[0].p, ctx->dof_next.p, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
    }
    ctx->dof_next_n = -1;
    refresh_ptrs(ctx);
    if ((st = ensure_eval_buffers(ctx))) return st;
    refresh_ptrs(ctx);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    ctx->uploaded = true;
    return MDN_OK;
}

// serializeDof (DofSerializer.hpp:64-92) from the device coordinates: bead i of the next system is
// current bead src[i], or (src[i] < 0) the next new bead of new_coord.
int mdn_dof_serialize(mdn_ctx* ctx, int32_t n_beads, const int32_t* src, const double* new_coord) {
    int st = need_system(ctx, false);
    if (st) return st;
    if (n_beads <= 0 || !src) return fail(ctx, MDN_ERR_ARG, "n_beads must be positive and src given");
    const int n_old = ctx->n_beads;
    std::vector<char> used(n_old, 0);
    int n_new = 0;
    for (int i = 0; i < n_beads; i++) {
        const int s = src[i];
        if (s < 0) { n_new++; continue; }
        if (s >= n_old) return fail(ctx, MDN_ERR_ARG, "src[%d] = %d: the current system has %d beads", i, s, n_old);
        if (used[s]) return fail(ctx, MDN_ERR_ARG, "src[%d] = %d: current bead named twice", i, s);
        used[s] = 1;
    }
    if (n_new > 0 && !new_coord) return fail(ctx, MDN_ERR_ARG, "%d new beads and no new_coord", n_new);
    HIPCHK(hipSetDevice(ctx->device));
    // the gather map: >= 0 a current bead, -1 - k the k-th new bead
    std::vector<int> g(n_beads);
    for (int i = 0, k = 0; i < n_beads; i++) g[i] = src[i] >= 0 ? src[i] : -1 - k++;
    HIPCHK(upload(ctx, ctx->dof_src, g));
    HIPCHK(ctx->dof_new.ensure(3 * (size_t)std::max(1, n_new)));
    if (n_new > 0)
        HIPCHK(hipMemcpyAsync(ctx->dof_new.p, new_coord, sizeof(double) * 3 * n_new, hipMemcpyHostToDevice,
                              ctx->stream));
    HIPCHK(ctx->dof_next.ensure(3 * (size_t)n_beads));
    const long ne = 3L * n_beads;
    hipLaunchKernelGGL(k_dof_gather, dim3(ceil_div(ne, BLOCK)), dim3(BLOCK), 0, ctx->stream, n_beads,
                       (const int*)ctx->dof_src.p, (const double*)ctx->x[ctx->cur].p, (const double*)ctx->dof_new.p,
                       ctx->dof_next.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));   // g ends with this scope
    ctx->dof_next_n = n_beads;
    return MDN_OK;
}

int mdn_crosslinks_update(mdn_ctx* ctx, const mdn_crosslink* linkers, int32_t n_linkers,
                          const mdn_crosslink* motors, int32_t n_motors) {
    int st = need_system(ctx, false);
    if (st) return st;
    HIPCHK(hipSetDevice(ctx->device));
    for (int w = 0; w < 2; w++) {   // validate everything before any state changes
        const int n = w ? n_motors : n_linkers;
        const mdn_crosslink* xl = w ? motors : linkers;
        if (n < 0 || (n > 0 && !xl)) return fail(ctx, MDN_ERR_ARG, "bad %s table", w ? "motor" : "linker");
        for (int j = 0; j < n; j++)
            if (xl[j].cyl1 < 0 || xl[j].cyl1 >= ctx->n_cyl || xl[j].cyl2 < 0 || xl[j].cyl2 >= ctx->n_cyl)
                return fail(ctx, MDN_ERR_ARG, "%s %d: cylinder index out of range", w ? "motor" : "linker", j);
    }
    if ((st = set_crosslinks(ctx, linkers, n_linkers, motors, n_motors))) return st;
    refresh_ptrs(ctx);
    if (ctx->nl_built) {
        if ((st = relayout(ctx))) return st;
    } else {
        ctx->sys_gen++;
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

int mdn_system_counts(mdn_ctx* ctx, int64_t* out) {
    if (!ctx || !out) return MDN_ERR_ARG;
    out[0] = ctx->n_beads;
    out[1] = ctx->n_cyl;
    for (int ff = 0; ff < NFF; ff++) out[2 + ff] = ctx->sys.n[ff];
    return MDN_OK;
}

int mdn_set_coords(mdn_ctx* ctx, const double* coord) {
    int st = need_system(ctx, false);
    if (st) return st;
    if (!coord) return fail(ctx, MDN_ERR_ARG, "null coord");
    st = set_coords_dev(ctx, coord);
    if (st) return st;
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

int mdn_displace(mdn_ctx* ctx, const double* delta, int32_t n_var) {
    int st = need_system(ctx, false);
    if (st) return st;
    if (!delta || n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    HIPCHK(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_axpy_inplace, dim3(std::max(1, ceil_div(n_var, BLOCK))), dim3(BLOCK), 0, ctx->stream,
                       ctx->x[ctx->cur].p, delta, (long)n_var);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

int mdn_perturb(mdn_ctx* ctx, uint64_t seed, uint64_t stream, double sigma) {
    int st = need_system(ctx, false);
    if (st) return st;
    if (!(sigma >= 0.0)) return fail(ctx, MDN_ERR_ARG, "sigma must be >= 0");
    HIPCHK(hipSetDevice(ctx->device));
    const long n = 3L * ctx->n_beads;
    hipLaunchKernelGGL(k_perturb, dim3(std::max(1, ceil_div(n, BLOCK))), dim3(BLOCK), 0, ctx->stream,
                       ctx->x[ctx->cur].p, n, (unsigned long long)seed, (unsigned long long)stream, sigma);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

int mdn_get_coords(mdn_ctx* ctx, double* coord) {
    int st = need_system(ctx, false);
    if (st) return st;
    HIPCHK(copy_out(ctx, coord, ctx->x[ctx->cur].p, sizeof(double) * 3 * ctx->n_beads));
    return MDN_OK;
}

// The block / slot layout for the current interaction counts and the bead-sorted slot layout: the
// static crosslink incidence, then the excluded-volume and boundary slots from the tables of the
// last neighbor-list build.
int relayout(mdn_ctx* ctx) {
    int st = MDN_OK;
    const long np = ctx->sys.n[FF_EXVOL];
    const int nbi = ctx->sys.n[FF_BOUNDARY];
    layout(ctx);
    if ((st = ensure_eval_buffers(ctx))) return st;
    refresh_ptrs(ctx);
    HIPCHK(ctx->inc_cnt.ensure(ctx->n_beads + 1));
    HIPCHK(ctx->bstart.ensure(ctx->n_beads + 1));
    const long ndyn = 4L * np + nbi, total = ctx->sys.slot0[NFF];
    HIPCHK(ctx->inc_list.ensure((size_t)std::max(1L, total)));
    refresh_ptrs(ctx);
    const int dyn_blocks = ceil_div(ndyn, BLOCK), bb = bead_blocks(ctx);
    hipLaunchKernelGGL(k_inc_static, dim3(ceil_div(ctx->n_beads + 1, BLOCK)), dim3(BLOCK), 0, ctx->stream, ctx->n_beads,
                       (const int*)ctx->inc_s_start.p, ctx->inc_cnt.p);
    if (ndyn > 0)
        hipLaunchKernelGGL(k_inc_count, dim3(dyn_blocks), dim3(BLOCK), 0, ctx->stream, ctx->sys, ctx->inc_cnt.p);
    if ((st = exclusive_scan(ctx, ctx->inc_cnt.p, ctx->bstart.p, ctx->n_beads + 1))) return st;
    hipLaunchKernelGGL(k_inc_fill, dim3(dyn_blocks + bb), dim3(BLOCK), 0, ctx->stream, ctx->sys, dyn_blocks,
                       (const int*)ctx->inc_s_start.p, (const int*)ctx->inc_s.p, (const int*)ctx->bstart.p,
                       ctx->inc_cnt.p, ctx->inc_list.p, ctx->sorted_id.p, ctx->pos.p);
    if (ndyn > 0)
        hipLaunchKernelGGL(k_inc_place, dim3(ceil_div(total, BLOCK)), dim3(BLOCK), 0, ctx->stream, ctx->sys, total,
                           (const int*)ctx->inc_s_start.p, (const int*)ctx->bstart.p, (const int*)ctx->inc_list.p,
                           ctx->sorted_id.p, ctx->pos.p);
    HIPCHK(hipGetLastError());
    refresh_ptrs(ctx);
    ctx->sys_gen++;
    return MDN_OK;
}

// The buffers of one hybrid neighbor list build (midpoints, bins, members, per-cylinder counts
// and offsets, the pair array).
struct NlBufs {
    DBuf<double>& mid;
    DBuf<int>& bin; DBuf<int>& bin_count; DBuf<int>& bin_start; DBuf<int>& place; DBuf<NlRec>& members;
    DBuf<int>& count; DBuf<int>& off; DBuf<int>& pairs;
    DBuf<int>& mbin; DBuf<double>& mmid;   // each member's bin and midpoint, in bin order
};

// HybridCylinderCylinderNL::reset for one list: midpoints, counting sort into bins, the
// 27-bin stencil (count, scan, emit in order). Queued; the pairs are counted in B.off[n_cyl], the
// flags of k_nl_report follow the bins' counts.
static long nl_tile_count(const NLDev& n) { return (long)n.nt[0] * n.nt[1] * n.nt[2]; }
static long nl_flags(const NLDev& n) { return nl_tile_count(n) * n.T * n.T * n.T + 1; }   // in bin_count
static int count_pairs(mdn_ctx* ctx, const NLDev& n, const double* x, NlBufs& B) {
    int st = MDN_OK;
    const long nbins = nl_flags(n) - 1;   // tile by tile, the last tiles padded
    if (nbins > (1L << 30)) return fail(ctx, MDN_ERR_UNSUPPORTED, "neighbor-list grid too large (%ld bins)", nbins);
    const int nc = n.n_cyl;
    const size_t n1 = std::max(1, nc);
    HIPCHK(B.mid.ensure(3 * n1));
    HIPCHK(B.bin.ensure(n1));
    HIPCHK(B.bin_count.ensure(nbins + 3));
    HIPCHK(B.bin_start.ensure(nbins + 1));
    HIPCHK(B.place.ensure(n1));
    HIPCHK(B.members.ensure(n1));
    HIPCHK(B.mbin.ensure(n1));
    HIPCHK(B.mmid.ensure(3 * n1));
    HIPCHK(B.count.ensure(nc + 1));
    HIPCHK(B.off.ensure(nc + 1));
    HIPCHK(ctx->nl_found.ensure(NL_HITS * n1));
    HIPCHK(hipMemsetAsync(B.bin_count.p, 0, sizeof(int) * (nbins + 3), ctx->stream));
    int* flags = B.bin_count.p + nl_flags(n);
    hipLaunchKernelGGL(k_nl_bin, dim3(ceil_div(nc + 1, BLOCK)), dim3(BLOCK), 0, ctx->stream, n, x, B.mid.p, B.bin.p,
                       B.place.p, B.bin_count.p, flags, B.count.p);
    HIPCHK(hipGetLastError());
    if ((st = exclusive_scan(ctx, B.bin_count.p, B.bin_start.p, nbins + 1))) return st;
    hipLaunchKernelGGL(k_nl_fill, dim3(ceil_div(n1, BLOCK)), dim3(BLOCK), 0, ctx->stream, n, B.bin.p, B.bin_start.p,
                       (const int*)B.place.p, (const double*)B.mid.p, B.members.p, B.mbin.p, B.mmid.p);
    hipLaunchKernelGGL(k_nl_tile<0>, dim3(nl_tile_count(n)), dim3(BLOCK), 0, ctx->stream, n, (const int*)B.bin_start.p,
                       (const NlRec*)B.members.p, (const int*)B.mbin.p, (const double*)B.mmid.p, B.count.p, flags + 1,
                       ctx->nl_found.p, (const int*)nullptr, (int*)nullptr, (int*)nullptr);
    HIPCHK(hipGetLastError());
    return exclusive_scan(ctx, B.count.p, B.off.p, nc + 1);
}
// After count_pairs: one wait for the counts (with the boundary interactions before each of ne + 1
// element bounds, from their offsets, if given), then the pairs, ordered by cylinder then
// neighbour (queued). *np = the pairs.
static int emit_pairs(mdn_ctx* ctx, const NLDev& n, NlBufs& B, int ne, const int* bnd_off, long* np, const char* what) {
    const int nc = n.n_cyl;
    int* flags = B.bin_count.p + nl_flags(n);
    hipLaunchKernelGGL(k_nl_report, dim3(1), dim3(64), 0, ctx->stream, nc, (const int*)B.off.p, (const int*)flags, ne,
                       bnd_off, ctx->h_int);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (ctx->h_int[1] != 0) {
        return fail(ctx, MDN_ERR_NL_BOUNDS, "%d cylinder midpoints outside the neighbor-list grid [0, %g)x[0, %g)x[0, %g)",
                    ctx->h_int[1], ctx->grid[0], ctx->grid[1], ctx->grid[2]);
    }
    *np = ctx->h_int[0];
    if (*np > 0x7fffffffL / 4) return fail(ctx, MDN_ERR_UNSUPPORTED, "too many %s pairs (%ld)", what, *np);
    HIPCHK(B.pairs.ensure(2 * (size_t)std::max(1L, *np)));
    if (ctx->h_int[2] == 0)
        hipLaunchKernelGGL(k_nl_emit, dim3(std::max(1, ceil_div(nc, BLOCK))), dim3(BLOCK), 0, ctx->stream, nc,
                           (const int*)B.off.p, (const int*)ctx->nl_found.p, (int2*)B.pairs.p);
    else {
        HIPCHK(ctx->nl_list.ensure((size_t)*np));
        hipLaunchKernelGGL(k_nl_tile<1>, dim3(nl_tile_count(n)), dim3(BLOCK), 0, ctx->stream, n,
                           (const int*)B.bin_start.p, (const NlRec*)B.members.p, (const int*)B.mbin.p,
                           (const double*)B.mmid.p, B.count.p, flags + 1, ctx->nl_found.p, (const int*)B.off.p,
                           ctx->nl_list.p, B.pairs.p);
        hipLaunchKernelGGL(k_nl_place, dim3(ceil_div(*np, BLOCK)), dim3(BLOCK), 0, ctx->stream, *np, (const int*)B.off.p,
                           (const int*)ctx->nl_list.p, B.pairs.p);
    }
    HIPCHK(hipGetLastError());
    return MDN_OK;
}

int mdn_nl_build(mdn_ctx* ctx, const double* coord, int64_t* n_pairs_out) {
    int st = need_system(ctx, false);
    if (st) return st;
    HIPCHK(hipSetDevice(ctx->device));
    // The rebuild reallocates the pair, excluded-volume and boundary tables that the system
    // record and the captured minimizer graphs point at; until the new layout is complete
    // (relayout), nothing may use them: a failure on the way leaves the lists unbuilt.
    ctx->nl_built = false;
    if ((st = set_coords_dev(ctx, coord))) return st;
    const double* x = ctx->x[ctx->cur].p;
    NLDev n = nl_view(ctx);
    const int nc = ctx->n_cyl;
    long np = 0;
    NlBufs B{ctx->mid, ctx->bin, ctx->bin_count, ctx->bin_start, ctx->place, ctx->members,
             ctx->nl_count, ctx->nl_off, ctx->pairs, ctx->mbin, ctx->mmid};
    if ((st = count_pairs(ctx, n, x, B))) return st;
    // boundary NL (BoundaryCylinderRepulsion::vectorize): counted before the one wait for both
    const int ne = (int)ctx->elems.size();
    const long nbc = (long)ne * nc;
    ctx->sys.n_elem = ne;
    HIPCHK(ctx->bnd_cnt.ensure(nbc + 1));
    HIPCHK(ctx->bnd_off.ensure(nbc + 1));
    hipLaunchKernelGGL(k_bnd_count, dim3(ceil_div(nbc + 1, BLOCK)), dim3(BLOCK), 0, ctx->stream, n, ctx->sys,
                       ctx->bnd_cutoff, ctx->mid.p, ctx->bnd_cnt.p);
    if ((st = exclusive_scan(ctx, ctx->bnd_cnt.p, ctx->bnd_off.p, nbc + 1))) return st;
    if ((st = emit_pairs(ctx, n, B, ne, ctx->bnd_off.p, &np, "excluded-volume"))) return st;
    // per-element counts (nneighbors) come from the offsets at element boundaries
    const int* eoff = ctx->h_int + 3;
    const int nbi = eoff[ne];
    ctx->bnd_nneighbors.assign(ne, 0);
    for (int e = 0; e < ne; e++) ctx->bnd_nneighbors[e] = eoff[e + 1] - eoff[e];
    // CylinderExclVolume::vectorize
    HIPCHK(ctx->ev_b.ensure(4 * (size_t)std::max(1L, np)));
    HIPCHK(ctx->ev_ks.ensure((size_t)std::max(1L, np)));
    if (np > 0)
        hipLaunchKernelGGL(k_ev_vectorize, dim3(ceil_div(np, BLOCK)), dim3(BLOCK), 0, ctx->stream, n, np,
                           ctx->pairs.p, ctx->ev_b.p, ctx->ev_ks.p);
    ctx->n_pairs = np;
    HIPCHK(ctx->bnd_b.ensure(std::max(1, nbi)));
    HIPCHK(ctx->bnd_e.ensure(std::max(1, nbi)));
    HIPCHK(ctx->bnd_krep.ensure(std::max(1, nbi)));
    HIPCHK(ctx->bnd_slen.ensure(std::max(1, nbi)));
    if (nbc > 0)
        hipLaunchKernelGGL(k_bnd_emit, dim3(ceil_div(nbc, BLOCK)), dim3(BLOCK), 0, ctx->stream, n, ctx->sys,
                           ctx->bnd_cnt.p, ctx->bnd_off.p, ctx->d_krep_e.p, ctx->d_slen_e.p, ctx->bnd_b.p,
                           ctx->bnd_e.p, ctx->bnd_krep.p, ctx->bnd_slen.p);
    ctx->n_bint = nbi;
    // new layout
    ctx->sys.n[FF_EXVOL] = (int)np;
    ctx->sys.n[FF_BOUNDARY] = nbi;
    if ((st = relayout(ctx))) return st;
    HIPCHK(hipStreamSynchronize(ctx->stream));
    ctx->nl_built = true;
    if (n_pairs_out) *n_pairs_out = np;
    return MDN_OK;
}

int mdn_boundary_load_forces(mdn_ctx* ctx, const double* coord, int32_t n_types, const double* monomer_size,
                             const int32_t* num_monomers, int32_t stride, double* load_plus, double* load_minus) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!monomer_size || !num_monomers || !load_plus || !load_minus) return fail(ctx, MDN_ERR_ARG, "null argument");
    if (n_types < 1 || n_types > MAX_FIL_TYPES)
        return fail(ctx, MDN_ERR_ARG, "n_types must be in [1, %d]", MAX_FIL_TYPES);
    LoadParams P;
    memset(&P, 0, sizeof(P));
    P.n_types = n_types;
    P.stride = stride;
    for (int t = 0; t < n_types; t++) {
        if (num_monomers[t] < 0 || num_monomers[t] > stride)
            return fail(ctx, MDN_ERR_ARG, "num_monomers[%d] = %d outside [0, stride = %d]", t, num_monomers[t], stride);
        P.mon_size[t] = monomer_size[t];
        P.num_mon[t] = num_monomers[t];
    }
    for (int c = 0; c < ctx->n_cyl; c++)
        if (ctx->cyl_type[c] < 0 || ctx->cyl_type[c] >= n_types)
            return fail(ctx, MDN_ERR_ARG, "filament %d has type %d, not below n_types = %d", ctx->cyl_fil[c],
                        ctx->cyl_type[c], n_types);
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * 3 * ctx->n_beads));
        x = ctx->ext.p;
    }
    const long n_out = 2L * ctx->n_fil * stride;
    if (n_out > 0) {
        HIPCHK(ctx->load_out.ensure(n_out));
        hipLaunchKernelGGL(k_load_forces, dim3(ceil_div(n_out, BLOCK)), dim3(BLOCK), 0, ctx->stream, nl_view(ctx),
                           ctx->sys, x, (const int*)ctx->d_fil_ends.p, (const int*)ctx->bnd_cnt.p,
                           (const double*)ctx->d_krep_e.p, (const double*)ctx->d_slen_e.p, ctx->n_fil, P,
                           ctx->load_out.p);
        HIPCHK(hipGetLastError());
        const size_t half = sizeof(double) * (size_t)ctx->n_fil * stride;
        HIPCHK(hipMemcpyAsync(load_plus, ctx->load_out.p, half, hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(hipMemcpyAsync(load_minus, ctx->load_out.p + (size_t)ctx->n_fil * stride, half, hipMemcpyDeviceToHost,
                              ctx->stream));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

// HybridBindingSearchManager::updateAllPossibleBindingsstencilHYBD (HybridBindingSearchManager.cpp:
// 759-966): the binder's hybrid list (addtoHNeighborList, :1024-1039: range cyl_size + rmax,
// lower bound max(rmin - cyl_size, 0), in float), then the site pairs of every listed pair,
// counted, scanned and emitted in list order.
int mdn_binding_pairs(mdn_ctx* ctx, const mdn_binding_params* p, const double* coord, uint32_t* out,
                      int64_t capacity, int64_t* n_out) {
    int st = need_system(ctx, false);
    if (st) return st;
    if (!p || !n_out) return fail(ctx, MDN_ERR_ARG, "null argument");
    if (p->n_sites <= 0 || !p->site_pos) return fail(ctx, MDN_ERR_ARG, "n_sites must be positive, site_pos given");
    if (p->shift_bits <= 0 || p->shift_bits > 16 || p->n_sites > (1 << p->shift_bits))
        return fail(ctx, MDN_ERR_ARG, "shift_bits %d cannot hold %d sites", p->shift_bits, p->n_sites);
    if (((long)ctx->n_cyl << p->shift_bits) > 0xffffffffL)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%d cylinders << %d bits exceed 32 bits", ctx->n_cyl, p->shift_bits);
    if (!(p->rmax > 0) || p->rmin < 0 || p->site_step < 0) return fail(ctx, MDN_ERR_ARG, "bad range or site step");
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * 3 * ctx->n_beads));
        x = ctx->ext.p;
    }
    // the list's range in float, as addtoHNeighborList and setneighborsearchparameters form it
    const float rmaxsq_b = p->rmax * p->rmax, rminsq_b = p->rmin * p->rmin;
    const float rmax_l = p->cyl_size + std::sqrt(rmaxsq_b);
    const float rmin_l = std::max(std::sqrt(rminsq_b) - p->cyl_size, 0.0f);
    NLDev n = nl_view(ctx);
    n.rmaxsq = rmax_l * rmax_l;
    n.rminsq = rmin_l * rmin_l;
    nl_grid(ctx, n);
    n.ta = std::min(p->ftype1, p->ftype2);
    n.tb = std::max(p->ftype1, p->ftype2);
    HIPCHK(ctx->b_site.ensure(p->n_sites));
    HIPCHK(hipMemcpyAsync(ctx->b_site.p, p->site_pos, sizeof(float) * p->n_sites, hipMemcpyHostToDevice, ctx->stream));
    if (p->site_free) {
        const size_t nf = (size_t)ctx->n_cyl * p->n_sites;
        HIPCHK(ctx->b_free.ensure(std::max<size_t>(1, nf)));
        HIPCHK(copy_in(ctx, ctx->b_free.p, p->site_free, sizeof(float) * nf));
    }
    long np = 0;
    NlBufs B{ctx->b_mid, ctx->b_bin, ctx->b_bin_count, ctx->b_bin_start, ctx->b_place, ctx->b_members,
             ctx->b_count, ctx->b_off, ctx->b_pairs, ctx->b_mbin, ctx->b_mmid};
    if ((st = count_pairs(ctx, n, x, B))) return st;
    if ((st = emit_pairs(ctx, n, B, 0, nullptr, &np, "binding-list"))) return st;
    BindDev b{};
    b.n_sites = p->n_sites;
    b.shift = p->shift_bits;
    b.step = p->site_step;
    b.ftype1 = std::min(p->ftype1, p->ftype2);   // the reference's _filamentIDvec pair, ascending
    b.ftype2 = std::max(p->ftype1, p->ftype2);
    b.rminsq = rminsq_b;
    b.rmaxsq = rmaxsq_b;
    b.p2_first = p->p2_first;
    b.p2_last = p->p2_last;
    b.site = ctx->b_site.p;
    b.free = p->site_free ? ctx->b_free.p : nullptr;
    HIPCHK(ctx->b_scount.ensure(np + 1));
    HIPCHK(ctx->b_soff.ensure(np + 1));
    const int G = ceil_div(np + 1, BLOCK);
    hipLaunchKernelGGL(k_bind_sites<0>, dim3(G), dim3(BLOCK), 0, ctx->stream, n, b, x, np, (const int*)ctx->b_pairs.p,
                       ctx->b_scount.p, (const int*)nullptr, (uint32_t*)nullptr);
    HIPCHK(hipGetLastError());
    if ((st = exclusive_scan(ctx, ctx->b_scount.p, ctx->b_soff.p, np + 1))) return st;
    HIPCHK(d2h(ctx, ctx->h_int, ctx->b_soff.p + np, sizeof(int)));
    const long total = ctx->h_int[0];
    *n_out = total;
    if (!out) return MDN_OK;
    if (capacity < total)
        return fail(ctx, MDN_ERR_CAPACITY, "%ld binding pairs, capacity %ld", total, (long)capacity);
    if (total == 0) return MDN_OK;
    HIPCHK(ctx->b_out.ensure(2 * (size_t)total));
    hipLaunchKernelGGL(k_bind_sites<1>, dim3(G), dim3(BLOCK), 0, ctx->stream, n, b, x, np, (const int*)ctx->b_pairs.p,
                       ctx->b_scount.p, (const int*)ctx->b_soff.p, ctx->b_out.p);
    HIPCHK(hipGetLastError());
    HIPCHK(copy_out(ctx, out, ctx->b_out.p, sizeof(uint32_t) * 2 * total));
    return MDN_OK;
}

int mdn_nl_pairs(mdn_ctx* ctx, int32_t* out, int64_t cap, int64_t* n_pairs) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (n_pairs) *n_pairs = ctx->n_pairs;
    if (cap < ctx->n_pairs) return fail(ctx, MDN_ERR_CAPACITY, "need room for %ld pairs", ctx->n_pairs);
    if (ctx->n_pairs > 0)
        HIPCHK(copy_out(ctx, out, ctx->pairs.p, sizeof(int) * 2 * ctx->n_pairs));
    return MDN_OK;
}

int mdn_boundary_list(mdn_ctx* ctx, int32_t* out_beads, int64_t cap, int32_t* out_nneighbors,
                      int64_t* n_interactions) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (n_interactions) *n_interactions = ctx->n_bint;
    if (cap < ctx->n_bint) return fail(ctx, MDN_ERR_CAPACITY, "need room for %d interactions", ctx->n_bint);
    if (ctx->n_bint > 0 && out_beads)
        HIPCHK(copy_out(ctx, out_beads, ctx->bnd_b.p, sizeof(int) * ctx->n_bint));
    if (out_nneighbors)
        for (size_t e = 0; e < ctx->bnd_nneighbors.size(); e++) out_nneighbors[e] = ctx->bnd_nneighbors[e];
    return MDN_OK;
}

static int energy_impl(mdn_ctx* ctx, const double* coord, mdn_energy_report* out, int prec) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!out) return fail(ctx, MDN_ERR_ARG, "null report");
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * 3 * ctx->n_beads));
        x = ctx->ext.p;
    }
    if ((st = energy_report(ctx, x, prec))) return st;
    fill_report(ctx->h_eout, out);
    return MDN_OK;
}

int mdn_energy(mdn_ctx* ctx, const double* coord, mdn_energy_report* out) {
    return energy_impl(ctx, coord, out, MDN_PREC_FP64);
}

int mdn_energy_mixed(mdn_ctx* ctx, const double* coord, mdn_energy_report* out) {
    return energy_impl(ctx, coord, out, MDN_PREC_MIXED);
}

static int forces_impl(mdn_ctx* ctx, int ff, const double* coord, double* force, int32_t n_var, int prec) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!force || n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * n_var));
        x = ctx->ext.p;
    }
    long lo = 0, hi = ctx->sys.slot0[NFF];
    const double* base = nullptr;
    if (ff >= 0) {
        lo = ctx->sys.slot0[ff];
        hi = ctx->sys.slot0[ff + 1];
        HIPCHK(copy_in(ctx, ctx->scratch_f.p, force, sizeof(double) * n_var));
        base = ctx->scratch_f.p;
    }
    const int bmask = ff < 0 ? 3 : ff == FF_STRETCH ? 1 : ff == FF_BEND ? 2 : 0;
    ForceEval ev{ctx, x, prec, bmask, lo, hi, base, ctx->f.p};
    if ((st = ev.start())) return st;
    HIPCHK(hipStreamSynchronize(ctx->stream));
    bool redone;
    if ((st = ev.finish(&redone))) return st;
    HIPCHK(copy_out(ctx, force, ctx->f.p, sizeof(double) * n_var));
    return MDN_OK;
}

int mdn_forces(mdn_ctx* ctx, const double* coord, double* force, int32_t n_var) {
    return forces_impl(ctx, -1, coord, force, n_var, MDN_PREC_FP64);
}

int mdn_ff_forces(mdn_ctx* ctx, int32_t ff, const double* coord, double* force, int32_t n_var) {
    if (ff < 0 || ff >= NFF) return fail(ctx, MDN_ERR_ARG, "force field index %d", ff);
    return forces_impl(ctx, ff, coord, force, n_var, MDN_PREC_FP64);
}

int mdn_crosslink_stretch_forces(mdn_ctx* ctx, double* linker_out, double* motor_out) {
    int st = need_system(ctx, true);
    if (st) return st;
    // the tensions are stored in the device tables' order: back to the crosslinks' own order
    for (int w = 0; w < 2; w++) {
        double* out = w ? motor_out : linker_out;
        const int n = ctx->sys.n[w ? FF_MOTOR : FF_LINKER];
        if (!out || n == 0) continue;
        std::vector<double> tmp(n);
        HIPCHK(d2h(ctx, tmp.data(), (w ? ctx->mot_sf : ctx->lnk_sf).p, sizeof(double) * n));
        const std::vector<int>& ord = ctx->xl_ord[w];
        for (int i = 0; i < n; i++) out[ord[i]] = tmp[i];
    }
    return MDN_OK;
}

// dE/dtheta at device coordinates x into ctx->grad_out: the per-pair excluded-volume energies,
// then one thread per cylinder. check: settle the pairs whose closed-form energy is deferred (a
// host sync on a device count, then the Simpson energy of each listed pair); without it the
// caller has established that no pair at x is deferred.
static int param_grad_launch(mdn_ctx* ctx, const double* x, int prec, bool check) {
    const DevSys& s = ctx->sys;
    const int np = s.n[FF_EXVOL];
    if (np > 0) {
        HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
        hipLaunchKernelGGL(k_ev_pair_energy, dim3(ceil_div(np, BLOCK)), dim3(BLOCK), 0, ctx->stream, s, x, ctx->ev_U.p,
                           ctx->bad_count.p, ctx->bad_list.p);
        HIPCHK(hipGetLastError());
    }
    if (np > 0 && check) {
        HIPCHK(hipMemcpyAsync(ctx->h_int, ctx->bad_count.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(hipStreamSynchronize(ctx->stream));
        const int nbad = ctx->h_int[0];
        if (nbad > 0) {
            std::vector<int> redo(nbad);
            HIPCHK(d2h(ctx, redo.data(), ctx->bad_list.p, sizeof(int) * nbad));
            std::sort(redo.begin(), redo.end());
            for (int t : redo)
                hipLaunchKernelGGL(k_ev_pair_energyN, dim3(1), dim3(BLOCK), 0, ctx->stream, s, x, t, ctx->ev_U.p);
            HIPCHK(hipGetLastError());
            std::vector<double> U(nbad);
            for (int i = 0; i < nbad; i++)
                HIPCHK(hipMemcpyAsync(&U[i], ctx->ev_U.p + redo[i], sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
            HIPCHK(hipStreamSynchronize(ctx->stream));
            for (int i = 0; i < nbad; i++)
                if (U[i] <= -1.0)
                    return fail(ctx, MDN_ERR_NONFINITE,
                                "excluded-volume pair %d: energy non-finite after the Simpson fallback", redo[i]);
        }
    }
    if (ctx->n_cyl > 0) {
        if (prec == MDN_PREC_MIXED)
            hipLaunchKernelGGL(k_param_grad<float>, dim3(ceil_div(ctx->n_cyl * PG_LANES, BLOCK)), dim3(BLOCK), 0, ctx->stream, s,
                               ctx->n_cyl, (const int*)ctx->d_cyl_b1.p, (const int*)ctx->d_cyl_bend.p, x,
                               (const double*)ctx->ev_U.p, ctx->grad_out.p);
        else
            hipLaunchKernelGGL(k_param_grad<double>, dim3(ceil_div(ctx->n_cyl * PG_LANES, BLOCK)), dim3(BLOCK), 0, ctx->stream, s,
                               ctx->n_cyl, (const int*)ctx->d_cyl_b1.p, (const int*)ctx->d_cyl_bend.p, x,
                               (const double*)ctx->ev_U.p, ctx->grad_out.p);
    }
    HIPCHK(hipGetLastError());
    return MDN_OK;
}

static int param_grad_impl(mdn_ctx* ctx, const double* coord, double* out, int64_t n_out, int prec) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!out || n_out != 3L * ctx->n_cyl) return fail(ctx, MDN_ERR_ARG, "n_out must be 3*n_cylinders = %d", 3 * ctx->n_cyl);
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * 3 * ctx->n_beads));
        x = ctx->ext.p;
    }
    HIPCHK(ctx->ev_U.ensure(std::max(1, ctx->sys.n[FF_EXVOL])));
    HIPCHK(ctx->grad_out.ensure(3 * (size_t)std::max(1, ctx->n_cyl)));
    if ((st = param_grad_launch(ctx, x, prec, true))) return st;
    HIPCHK(copy_out(ctx, out, ctx->grad_out.p, sizeof(double) * 3 * ctx->n_cyl));
    return MDN_OK;
}

int mdn_param_grad(mdn_ctx* ctx, const double* coord, double* out, int64_t n_out) {
    return param_grad_impl(ctx, coord, out, n_out, MDN_PREC_FP64);
}

int mdn_param_grad_mixed(mdn_ctx* ctx, const double* coord, double* out, int64_t n_out) {
    return param_grad_impl(ctx, coord, out, n_out, MDN_PREC_MIXED);
}

// The tangent terms of nv products at device coordinates x: product k's tangent at v + k n_var,
// its slots at slots + k slot_stride, its pieces at piece + k piece_stride. Excluded-volume pairs
// without a tangent are counted in bad_count (zeroed by the caller).
static void launch_tangents(mdn_ctx* ctx, const double* x, int prec, const double* v, int nv, double* slots,
                            long slot_stride, double* piece, long piece_stride) {
    const DevSys& s = ctx->sys;
    if (s.blk[NFF] == 0 || nv == 0) return;
    const long n_var = 3L * ctx->n_beads;
    const dim3 g(s.blk[NFF], nv);
    if (prec == MDN_PREC_MIXED)
        hipLaunchKernelGGL(k_tangent_terms<DualF>, g, dim3(BLOCK), 0, ctx->stream, s, x, v, n_var, slots, slot_stride,
                           piece, piece_stride, ctx->bad_count.p);
    else
        hipLaunchKernelGGL(k_tangent_terms<DualD>, g, dim3(BLOCK), 0, ctx->stream, s, x, v, n_var, slots, slot_stride,
                           piece, piece_stride, ctx->bad_count.p);
}

// -(dF/dx) v of nv products into out + k n_var from their slots and pieces (one launch); the
// count of pairs without a tangent into ctx->h_int[0].
static void gather_tangents(mdn_ctx* ctx, int nv, const double* slots, long slot_stride, double* piece,
                            long piece_stride, double* out) {
    const DevSys& s = ctx->sys;
    const dim3 g(gather_blocks(ctx), nv), b(BLOCK);
    const long n_var = 3L * ctx->n_beads;
    if (gather_size(ctx) == 128)
        hipLaunchKernelGGL(k_gather_tangents<128>, g, b, 0, ctx->stream, s, slots, slot_stride, piece, piece_stride, out,
                           n_var, (const int*)ctx->bad_count.p, ctx->h_int);
    else
        hipLaunchKernelGGL(k_gather_tangents<64>, g, b, 0, ctx->stream, s, slots, slot_stride, piece, piece_stride, out,
                           n_var, (const int*)ctx->bad_count.p, ctx->h_int);
}

// H v into ctx->scratch_f for the device tangent ctx->tan_v at device coordinates x (the tangent
// pieces of every interaction, then the FP64 gather); excluded-volume pairs without a tangent are
// counted in bad_count.
static int hvp_launch(mdn_ctx* ctx, const double* x, int prec) {
    HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
    launch_tangents(ctx, x, prec, ctx->tan_v.p, 1, ctx->slots.p, 0L, ctx->piece.p, 0L);
    HIPCHK(hipGetLastError());
    gather_tangents(ctx, 1, ctx->slots.p, 0L, ctx->piece.p, 0L, ctx->scratch_f.p);
    HIPCHK(hipGetLastError());
    return MDN_OK;
}

static int hvp_impl(mdn_ctx* ctx, const double* coord, const double* v, double* out, int32_t n_var, int prec) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!v || !out || n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * n_var));
        x = ctx->ext.p;
    }
    HIPCHK(ctx->tan_v.ensure(n_var));
    HIPCHK(copy_in(ctx, ctx->tan_v.p, v, sizeof(double) * n_var));
    if ((st = hvp_launch(ctx, x, prec))) return st;
    HIPCHK(copy_out(ctx, out, ctx->scratch_f.p, sizeof(double) * n_var));
    if (ctx->h_int[0] != 0)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%d excluded-volume pairs need the numerical force fallback (no tangent)",
                    ctx->h_int[0]);
    return MDN_OK;
}

int mdn_hvp(mdn_ctx* ctx, const double* coord, const double* v, double* out, int32_t n_var) {
    return hvp_impl(ctx, coord, v, out, n_var, MDN_PREC_FP64);
}

int mdn_hvp_mixed(mdn_ctx* ctx, const double* coord, const double* v, double* out, int32_t n_var) {
    return hvp_impl(ctx, coord, v, out, n_var, MDN_PREC_MIXED);
}

int mdn_hvp_batch(mdn_ctx* ctx, int32_t precision, const double* coord, const double* V, double* out, int32_t n_var,
                  int32_t n_vec) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (precision != MDN_PREC_FP64 && precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", precision);
    if (!V || !out || n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    if (n_vec < 1) return fail(ctx, MDN_ERR_ARG, "n_vec must be positive");
    HIPCHK(hipSetDevice(ctx->device));
    const DevSys& s = ctx->sys;
    const double* x = ctx->x[ctx->cur].p;
    if (coord) {
        HIPCHK(copy_in(ctx, ctx->ext.p, coord, sizeof(double) * n_var));
        x = ctx->ext.p;
    }
    // per product: its tangent, its slots (with the gather's padding), its pieces, its result
    const int chunk = std::min<int>(n_vec, MDN_HVP_BATCH_CHUNK);
    const long slot_stride = 3 * std::max(1L, s.slot0[NFF]) + GCHUNK_PAD;
    const long piece_stride = (long)NBOND * 3 * ctx->n_beads;
    HIPCHK(ctx->hb_v.ensure((size_t)chunk * n_var));
    HIPCHK(ctx->hb_slots.ensure((size_t)chunk * slot_stride));
    HIPCHK(ctx->hb_piece.ensure((size_t)chunk * piece_stride));
    HIPCHK(ctx->hb_out.ensure((size_t)chunk * n_var));
    HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
    for (int k0 = 0; k0 < n_vec; k0 += chunk) {
        const int nv = std::min(chunk, n_vec - k0);
        HIPCHK(copy_in(ctx, ctx->hb_v.p, V + (size_t)k0 * n_var, sizeof(double) * nv * n_var));
        launch_tangents(ctx, x, precision, ctx->hb_v.p, nv, ctx->hb_slots.p, slot_stride, ctx->hb_piece.p, piece_stride);
        HIPCHK(hipGetLastError());
        gather_tangents(ctx, nv, ctx->hb_slots.p, slot_stride, ctx->hb_piece.p, piece_stride, ctx->hb_out.p);
        HIPCHK(hipGetLastError());
        HIPCHK(copy_out(ctx, out + (size_t)k0 * n_var, ctx->hb_out.p, sizeof(double) * nv * n_var));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (ctx->h_int[0] != 0)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%d excluded-volume pairs need the numerical force fallback (no tangent)",
                    ctx->h_int[0]);
    return MDN_OK;
}

int mdn_set_params(mdn_ctx* ctx, const double* kstr, const double* eql, const double* kbend) {
    int st = need_system(ctx, false);
    if (st) return st;
    HIPCHK(hipSetDevice(ctx->device));
    const int nc = ctx->n_cyl;
    if (kstr) HIPCHK(copy_in(ctx, ctx->str_k.p, kstr, sizeof(double) * nc));
    if (eql) {
        for (int c = 0; c < nc; c++) ctx->cyl_eql[c] = eql[c];
        HIPCHK(upload(ctx, ctx->str_eql, ctx->cyl_eql));
        HIPCHK(upload(ctx, ctx->d_cyl_eql, ctx->cyl_eql));
        if (ctx->nl_built && ctx->n_pairs > 0)   // kRepScaled = krep L0_i L0_j
            hipLaunchKernelGGL(k_ev_vectorize, dim3(ceil_div(ctx->n_pairs, BLOCK)), dim3(BLOCK), 0, ctx->stream,
                               nl_view(ctx), ctx->n_pairs, (const int*)ctx->pairs.p, ctx->ev_b.p, ctx->ev_ks.p);
    }
    if (kbend) {
        std::vector<double> bk(ctx->bend_cyl.size());
        for (size_t i = 0; i < bk.size(); i++) bk[i] = kbend[ctx->bend_cyl[i]];
        HIPCHK(upload(ctx, ctx->bend_k, bk));
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

int mdn_forces_mixed(mdn_ctx* ctx, const double* coord, double* force, int32_t n_var) {
    return forces_impl(ctx, -1, coord, force, n_var, MDN_PREC_MIXED);
}

}  // extern "C"

// ----------------------------------------------------------------------------------------
// Force evaluation without allocation
// ----------------------------------------------------------------------------------------
namespace {

// Byte offsets of the evaluation's buffers in `scratch` (each 256-byte aligned): the fallback
// count and flag, the fallback partials (6 per block of the 240-block Simpson rule), the list of
// pairs that need it, the bonded sums (3 doubles per bead) and last the slot vectors (3 values of
// R per slot, padded by one gather chunk, which the gather reads unconditionally).
struct ScratchLayout {
    size_t bad_count, ok, partial, bad_list, bsum, slots, total;
};
size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }
ScratchLayout scratch_layout(const DevSys& s, int n_beads, size_t rsize) {
    ScratchLayout L;
    L.bad_count = 0;
    L.ok = 256;
    L.partial = 512;
    L.bad_list = up256(L.partial + sizeof(double) * 6 * FORCEN_BLOCKS);
    L.bsum = up256(L.bad_list + sizeof(int) * (size_t)std::max(1, s.n[FF_EXVOL]));
    L.slots = up256(L.bsum + sizeof(double) * 3 * (size_t)std::max(1, n_beads));
    L.total = L.slots + rsize * (3 * (size_t)std::max(1L, s.slot0[NFF]) + GCHUNK_PAD);
    return L;
}

template <typename R>
int forces_noalloc_t(mdn_ctx* ctx, unsigned char* scr, const double* x, double* out) {
    DevSys s = ctx->sys;   // the same tables, with the bonded sums in the scratch
    const ScratchLayout L = scratch_layout(s, ctx->n_beads, sizeof(R));
    int* bad_count = reinterpret_cast<int*>(scr + L.bad_count);
    int* ok = reinterpret_cast<int*>(scr + L.ok);
    double* partial = reinterpret_cast<double*>(scr + L.partial);
    int* bad_list = reinterpret_cast<int*>(scr + L.bad_list);
    s.bsum = reinterpret_cast<double*>(scr + L.bsum);
    R* slots = reinterpret_cast<R*>(scr + L.slots);
    // the terms, then the gather before the host knows whether a pair needs the numerical fallback
    // and writes nothing if one does. Two launches and one wait bound the call: with a launch that
    // cleared the count and a wait for it between the two it took 35 us at 550 beads, 38 at 42,000
    // and 62 at 420,000; now 21, 24 and 48. The count is zero between calls.
    launch_terms<R>(ctx, s, x, slots, false, 3, nullptr, bad_count, bad_list);
    launch_gather_plain<R>(ctx, s, 3, (const R*)slots, 0L, s.slot0[NFF], (const double*)nullptr, out, true, bad_count);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (ctx->h_int[0] == 0) return MDN_OK;
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(1), 0, ctx->stream, bad_count, 0);
    const int st = settle_pairs<R>(ctx, s, x, slots, bad_list, ctx->h_int[0], partial, ok);
    if (st) return st;
    launch_gather_plain<R>(ctx, s, 3, (const R*)slots, 0L, s.slot0[NFF], (const double*)nullptr, out, true);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDN_OK;
}

}  // namespace

extern "C" {

int mdn_forces_noalloc(mdn_ctx* ctx, int32_t precision, const double* coord_dev, double* force_dev, int32_t n_var) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!coord_dev || !force_dev) return fail(ctx, MDN_ERR_ARG, "null coordinate or force buffer");
    if (n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    if (precision != MDN_PREC_FP64 && precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", precision);
    const ScratchLayout L =
        scratch_layout(ctx->sys, ctx->n_beads, precision == MDN_PREC_MIXED ? sizeof(float) : sizeof(double));
    if (L.total > MDN_SCRATCH_BYTES)
        return fail(ctx, MDN_ERR_CAPACITY,
                    "the evaluation needs %zu bytes of scratch; mdn_forces_noalloc has %zu (%d MiB): use mdn_forces",
                    L.total, MDN_SCRATCH_BYTES, MDN_NOALLOC_SCRATCH_MIB);
    HIPCHK(hipSetDevice(ctx->device));
    unsigned char* scr = ctx->device < MAX_DEVICES ? g_scratch_dev[ctx->device] : nullptr;
    if (!scr) return fail(ctx, MDN_ERR_STATE, "no scratch address for device %d", ctx->device);
    return precision == MDN_PREC_MIXED ? forces_noalloc_t<float>(ctx, scr, coord_dev, force_dev)
                                       : forces_noalloc_t<double>(ctx, scr, coord_dev, force_dev);
}

// ----------------------------------------------------------------------------------------
// CGMethod::minimize on the device
// ----------------------------------------------------------------------------------------
// Line-search partial blocks: the interaction blocks (k_cg_ls), then the bead blocks (k_cg_pos).
static int ls_blocks(mdn_ctx* ctx) { return ctx->sys.lsp; }

static CgBufs cg_bufs(mdn_ctx* ctx) {
    CgBufs B;
    B.done_host = ctx->h_int + 4;
    B.x[0] = ctx->x[0].p; B.x[1] = ctx->x[1].p;
    B.d[0] = ctx->d[0].p; B.d[1] = ctx->d[1].p;
    B.xmin[0] = ctx->xmin[0].p; B.xmin[1] = ctx->xmin[1].p;
    B.f[0] = ctx->f.p; B.f[1] = ctx->f2.p; B.xh = ctx->xh.p;
    B.slots = (void*)ctx->slots.p; B.partial = ctx->partial.p; B.bad_count = ctx->bad_count.p;
    B.gpartial = ctx->partial.p + (long)PSTRIDE * ls_blocks(ctx);   // after the line-search partials
    return B;
}

// The minimizer's kernels use the bonded sums (bonded_gather); below CG_BEAD_ENERGY_BEADS beads
// the line search keeps the filament terms' own blocks for their energies, from there on the bead
// blocks take the energies too and those blocks leave the grid (bead_energy). Measured per CG
// iteration (same process, piece arrays -> this choice): 42,000 beads FP64 32.2 -> 31.2-32.3 us,
// mixed 30.5 -> 29.6 us (bead-block energies there: 32.9 and 30.8 us); 420,000 beads FP64 75.3 ->
// 68.4 us, mixed 65.5 -> 63.0 us (own energy blocks there: 73.1 and 67.9 us).
static const int CG_BEAD_ENERGY_BEADS = 100000;
static bool cg_bonded_sums(const mdn_ctx* ctx, int prec) {
    (void)prec;
    return ctx->bonded_gather_mode >= 0 ? ctx->bonded_gather_mode != 0 : true;
}
// the system record the minimizer's kernels of precision prec take
static DevSys cg_sys(const mdn_ctx* ctx, int prec) {
    DevSys s = ctx->sys;
    s.bonded_gather = cg_bonded_sums(ctx, prec) ? 1 : 0;
    s.bead_energy = ctx->n_beads >= CG_BEAD_ENERGY_BEADS ? 1 : 0;
    return s;
}

extern "C++" {
// FP64 excluded-volume force blocks of their own pay while the chip is not full without them (80
// iterations without the rebuild, one thread per pair -> two: 14,700 beads in a cube 2.22 -> 2.07 ms,
// 42,000 2.53 -> 2.48, 84,000 3.04 -> 3.02, 126,000 3.31 -> 3.42; in a sphere 42,000 2.26 -> 2.08,
// 84,000 2.47 -> 2.42, 126,000 2.62 -> 2.69, 420,000 4.84 -> 4.93). Denser networks fill it with fewer
// beads (40 iterations): 42,000 beads with 153,000 pairs 2.76 -> 2.73, 228,000 2.54 -> 2.56, 507,000
// 5.61 -> 5.73; 94,500 with 186,000 2.75 -> 2.77, 366,000 4.05 -> 4.12; 21,000 with 127,000 3.10 -> 3.07,
// 287,000 5.16 -> 5.13.
static const long EV_SPLIT_BEADS = 100000, EV_SPLIT_WORK = 140000;
static bool ev_split(const DevSys& s) {
    return s.n_beads < EV_SPLIT_BEADS && s.n_beads + s.n[FF_EXVOL] / 2L < EV_SPLIT_WORK;
}
template <typename R>
static void launch_slot(mdn_ctx* ctx, const DevSys& s, const CgBufs& B) {
    const int gbk = gather_blocks(ctx);
    hipLaunchKernelGGL(k_cg_pos, dim3(bead_blocks(ctx)), dim3(BLOCK), 0, ctx->stream, s, (const CgState*)ctx->cg.p, B);
    // the excluded-volume force blocks, all interaction blocks, then (bonded_gather) the bead blocks;
    // with bead_energy the filament terms' blocks are left out
    const int lsg = s.bonded_gather ? (s.bead_energy ? s.blk_nb : s.blk[NFF]) + s.nbb : s.blk[NFF];
    bool split = false;
    if constexpr (sizeof(R) == 8) split = ev_split(s);
    if constexpr (sizeof(R) == 8)
        if (split)
            hipLaunchKernelGGL((k_cg_ls<R, true>), dim3(std::max(1, ev_force_blocks<R, true>(s) + lsg)), dim3(BLOCK), 0,
                               ctx->stream, s, (const CgState*)ctx->cg.p, B);
    if (!split)
        hipLaunchKernelGGL((k_cg_ls<R, false>), dim3(std::max(1, lsg)), dim3(BLOCK), 0, ctx->stream, s,
                           (const CgState*)ctx->cg.p, B);
    launch_cg_gather<R>(ctx, s, (const CgState*)ctx->cg.p, B);
    hipLaunchKernelGGL(k_cg_fin, dim3(1), dim3(FIN), 0, ctx->stream, s, ctx->cg.p, B, gbk);
}
}  // extern "C++"

// A batch of minimizer slots captured once per system layout and replayed as a hipGraph; the
// kernels take every decision from the device state, so replays need no host work.
static const int CG_BATCH = 16, LAUNCH_BATCH = 4;

static int cg_graph(mdn_ctx* ctx, int prec) {
    if (ctx->graph_exec[prec] && ctx->graph_gen[prec] == ctx->sys_gen) return MDN_OK;
    if (ctx->graph_exec[prec]) (void)hipGraphExecDestroy(ctx->graph_exec[prec]);
    if (ctx->graph[prec]) (void)hipGraphDestroy(ctx->graph[prec]);
    ctx->graph_exec[prec] = nullptr;
    ctx->graph[prec] = nullptr;
    CgBufs B = cg_bufs(ctx);
    const DevSys s = cg_sys(ctx, prec);
    HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    for (int i = 0; i < CG_BATCH; i++) {
        if (prec == MDN_PREC_MIXED) launch_slot<float>(ctx, s, B);
        else launch_slot<double>(ctx, s, B);
    }
    HIPCHK(hipStreamEndCapture(ctx->stream, &ctx->graph[prec]));
    HIPCHK(hipGraphInstantiate(&ctx->graph_exec[prec], ctx->graph[prec], nullptr, nullptr, 0));
    ctx->graph_gen[prec] = ctx->sys_gen;
    return MDN_OK;
}

// The work of a network in the persistent minimizer, in beads: in a batch an excluded-volume pair
// costs what about eight beads do.
static long team_cost(const DevSys& s) {
    return s.n_beads + s.n[FF_LINKER] + s.n[FF_MOTOR] + 8L * s.n[FF_EXVOL] + s.n[FF_BOUNDARY];
}
static long team_one_work(const DevSys& s) {
    return s.n_beads + s.n[FF_LINKER] + s.n[FF_MOTOR] + 2L * s.n[FF_EXVOL] + s.n[FF_BOUNDARY];
}
// Workgroups of the persistent minimizer for a single network; 0: the four-kernel slots.
static int team_workgroups(const mdn_ctx* ctx) {
    if (!cg_bonded_sums(ctx, 0) || ctx->n_beads >= GB_LARGE_BEADS) return 0;
    const int room = team_room(ctx->n_cu);
    return ctx->team_size >= 0 ? std::min(ctx->team_size, room) : team_size_one(team_one_work(ctx->sys), room);
}

// The persistent minimizer on one system from its device state until that is done. The barrier's
// words at team_ctl(cg) are zero. A team of more than one has its share of the device's TeamRoom.
static int launch_team(mdn_ctx* ctx, int prec, int size) {
    const DevSys s = cg_sys(ctx, prec);
    const CgBufs B = cg_bufs(ctx);
    const int stride = size > 1 ? ctx->team_stride : 1;
    const dim3 g(stride * (size - 1) + 1), b(TEAM_NT);
    TeamCtl* ctl = team_ctl(ctx->cg.p);
    if (prec == MDN_PREC_MIXED)
        hipLaunchKernelGGL((k_cg_team_one<float, TEAM_NT>), g, b, 0, ctx->stream, s, B, ctx->cg.p, ctl, ctx->team_part.p, size,
                           stride, ctx->team_polls);
    else
        hipLaunchKernelGGL((k_cg_team_one<double, TEAM_NT>), g, b, 0, ctx->stream, s, B, ctx->cg.p, ctl, ctx->team_part.p, size,
                           stride, ctx->team_polls);
    HIPCHK(hipGetLastError());
    return MDN_OK;
}

// The two events that mark the last batches of slots.
struct SlotEvents {
    hipEvent_t e[2] = {nullptr, nullptr};
    hipError_t create() {
        const hipError_t r = hipEventCreateWithFlags(&e[0], hipEventDisableTiming);
        return r != hipSuccess ? r : hipEventCreateWithFlags(&e[1], hipEventDisableTiming);
    }
    ~SlotEvents() {
        for (hipEvent_t v : e)
            if (v) (void)hipEventDestroy(v);
    }
};

// One minimization. With teams, by a team where that is the faster form; *gave_up: its workgroups
// waited for each other too long, and the start is as it was (coord has not been written; without it
// the device coordinates are put back).
static int minimize_run(mdn_ctx* ctx, const mdn_cg_params* p, double* coord, double* force_out, mdn_min_result* res,
                        bool teams, bool* gave_up) {
    int st;
    const int prec = p->precision;
    memset(res, 0, sizeof(*res));
    ctx->last_team[0] = 0;
    ctx->last_team[1] = teams ? 0 : 1;
    const int nv = 3 * ctx->n_beads;
    // startMinimization + initial energy / forces (CGMethod.hpp:876-896); the start is in x[0]
    if (coord)
        HIPCHK(copy_in(ctx, ctx->x[0].p, coord, sizeof(double) * nv, true));
    else if (ctx->cur != 0)   // the context's device coordinates
        HIPCHK(hipMemcpyAsync(ctx->x[0].p, ctx->x[ctx->cur].p, sizeof(double) * nv, hipMemcpyDeviceToDevice,
                              ctx->stream));
    ctx->cur = 0;
    // the reported energies are FP64 in both precisions; the minimizer's own energies and forces
    // are evaluated in the requested precision
    // (the reports, the forces and F.F and maxF, a fixed-order reduction, in one wait)
    double *rep = ctx->h_eout, *rep_mixed = ctx->h_eout + 10, *stats = ctx->h_eout + 24;
    launch_energy(ctx, ctx->x[0].p, MDN_PREC_FP64, rep);
    if (prec == MDN_PREC_MIXED) launch_energy(ctx, ctx->x[0].p, prec, rep_mixed);
    ForceEval fe{ctx, ctx->x[0].p, prec, 3, 0, ctx->sys.slot0[NFF], nullptr, ctx->f.p};
    if ((st = fe.start())) return st;
    const int nsb = std::min(VSTAT_BLOCKS, std::max(1, ceil_div(nv, BLOCK)));
    bool redo = true;
    for (int pass = 0; pass < 2 && redo; pass++) {   // again when a pair took the numerical fallback
        hipLaunchKernelGGL(k_vec_stats, dim3(nsb), dim3(BLOCK), 0, ctx->stream, (const double*)ctx->f.p, (long)nv,
                           ctx->vstat.p);
        hipLaunchKernelGGL(k_vec_stats_fin, dim3(1), dim3(BLOCK), 0, ctx->stream, (const double*)ctx->vstat.p, nsb, stats);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(ctx->stream));
        if (pass) break;
        if ((st = check_energy(ctx, rep))) return st;
        fill_report(rep, &res->energies_before);
        if (prec == MDN_PREC_MIXED && (st = check_energy(ctx, rep_mixed))) return st;
        if ((st = fe.finish(&redo))) return st;
    }
    const double e_start = prec == MDN_PREC_MIXED ? rep_mixed[6] : rep[6];
    const double ff = stats[0], mx = stats[1];
    CgState& S = *ctx->h_cg;
    memset((void*)ctx->h_cg, 0, CG_BYTES);
    S.method = p->method;
    S.ls_algo = p->line_search;
    S.try_recover = p->try_recover;
    S.force_call_limit = std::max(p->force_call_limit, 3 * ctx->n_beads);
    S.energy_call_limit = p->energy_call_limit;
    S.max_dist = p->max_dist;
    S.lambda_max = p->lambda_max;
    S.grad_tol = p->grad_tol;
    S.energy_rel_tol = p->energy_rel_tol;
    S.num_energy_call = 1;
    S.num_force_call = 1;
    S.grad_inf_norm = mx;
    S.energy_rel_change = INFINITY;
    S.prev_energy = e_start;
    S.minimum_e = INFINITY;
    S.fdotf = ff;
    // resetCGParams before the loop (d = F + 0 d, lastFDotF = F.F, F_prev = F), applied by the
    // first line-search launch
    S.dir_pending = 1;
    S.dir_beta = 0.0;
    S.dir_reset = 1;
    S.phase = PH_LS;
    S.ls_lambda = rmin(S.lambda_max, S.max_dist / S.grad_inf_norm);
    res->force_call_limit = S.force_call_limit;
    res->energy_call_limit = S.energy_call_limit;
    res->grad_tol = S.grad_tol;
    res->energy_rel_tol = S.energy_rel_tol;
    if (!std::isfinite(mx) || !std::isfinite(ff)) return fail(ctx, MDN_ERR_NONFINITE, "maxF is not finite at the start");
    const bool limit0 = (S.force_call_limit != 0 && S.num_force_call > S.force_call_limit);
    S.done = (S.grad_inf_norm < S.grad_tol || S.energy_rel_change < S.energy_rel_tol || limit0) ? 1 : 0;
    HIPCHK(hipMemsetAsync(ctx->d[0].p, 0, sizeof(double) * nv, ctx->stream));   // searchDir.assign(numDof, 0)
    HIPCHK(hipMemcpyAsync(ctx->cg.p, &S, CG_BYTES, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
    // a team of several needs its share of the device's room for teams (none left: the slots)
    TeamHold hold(team_room_of(ctx->device));
    int team = teams ? team_workgroups(ctx) : 0;
    if (team > 1 && !S.done && !hold.take(team, team_room(ctx->n_cu))) team = 0;
    if (!S.done) ctx->last_team[0] = team;
    if (team > 1 && !S.done && !coord)   // the start, should the team give up
        HIPCHK(hipMemcpyAsync(ctx->ext.p, ctx->x[0].p, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
    // The slots are captured into a graph once they minimize a layout a second time: a graph made
    // for one minimization (a layout that the next neighbor-list rebuild replaces) costs more to
    // instantiate than its replays save over launching the same kernels directly.
    const bool graph = !team && ctx->use_graph && (ctx->graph_gen[prec] == ctx->sys_gen || ctx->min_gen[prec] == ctx->sys_gen);
    if (!team) ctx->min_gen[prec] = ctx->sys_gen;
    if (graph && (st = cg_graph(ctx, prec))) return st;
    const DevSys slot_sys = cg_sys(ctx, prec);
    const CgBufs slot_bufs = cg_bufs(ctx);

    // Batches of slots are launched back to back; the host looks at the done flag, which the last
    // slot writes to pinned memory, after batch i while batch i + 1 runs, so the device never idles
    // waiting for the host. The slots left of the two batches return at once (9 us each): a batch
    // is a graph's CG_BATCH slots or, launched directly, LAUNCH_BATCH, 16 launches that the host
    // issues in half the time they run (80 iterations of 42,000 beads with batches of 16 and a
    // copy of the flag after each: 2960 us, so 2890; of 420,000: 7140 and 6995).
    const int per = graph ? CG_BATCH : LAUNCH_BATCH;
    const long max_batches = ((slots_per_force_call(S) * ((long)S.force_call_limit + 16)) / CG_BATCH + 8) * (CG_BATCH / per);
    long launched = 0;
    SlotEvents ev;
    if (!team) HIPCHK(ev.create());
    int n_forcen = 0;
    for (;;) {
        bool done = S.done != 0;
        volatile int* h_done = slot_bufs.done_host;
        *h_done = 0;
        int k = 0;
        long here = 0;
        if (team && !done) {
            if (n_forcen) HIPCHK(hipMemsetAsync(team_ctl(ctx->cg.p), 0, sizeof(TeamCtl), ctx->stream));
            if ((st = launch_team(ctx, prec, team))) return st;
            if (force_out) map_pages(force_out, sizeof(double) * nv);   // while the device works
            done = true;
        }
        while (!done && launched < max_batches) {
            if (graph) {
                HIPCHK(hipGraphLaunch(ctx->graph_exec[prec], ctx->stream));
            } else {
                for (int i = 0; i < per; i++) {
                    if (prec == MDN_PREC_MIXED) launch_slot<float>(ctx, slot_sys, slot_bufs);
                    else launch_slot<double>(ctx, slot_sys, slot_bufs);
                }
                HIPCHK(hipGetLastError());
            }
            launched++;
            here++;
            HIPCHK(hipEventRecord(ev.e[k], ctx->stream));
            if (here > 1) {
                if (launched == 2 && force_out) map_pages(force_out, sizeof(double) * nv);   // while the device works
                HIPCHK(hipEventSynchronize(ev.e[k ^ 1]));
                if (*h_done) done = true;
            }
            k ^= 1;
        }
        HIPCHK(d2h(ctx, ctx->h_cg, ctx->cg.p, CG_BYTES));
        if (team_ctl(ctx->h_cg)->failed) {
            HIPCHK(hipMemsetAsync(ctx->defer_n.p, 0, sizeof(int), ctx->stream));   // (bad_count: cleared by the evaluation)
            if (!coord)
                HIPCHK(hipMemcpyAsync(ctx->x[0].p, ctx->ext.p, sizeof(double) * nv, hipMemcpyDeviceToDevice, ctx->stream));
            *gave_up = true;
            return MDN_OK;
        }
        if (!(S.done && S.status == ST_NEED_FORCEN)) break;
        // The step's forces need the numerical excluded-volume fallback (forceN,
        // CylinderExclVolRepulsion.cpp:984-1254): recompute them at the new coordinates with it
        // (same positions, so every other slot is bit-identical), then run this step's gather
        // again and resume.
        n_forcen++;
        const DevSys cs = cg_sys(ctx, prec);
        if ((st = eval_slots(ctx, ctx->x[S.parity ^ 1].p, prec, !cs.bonded_gather))) return st;
        HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
        S.status = 0;
        S.done = 0;
        S.reserved[1] = n_forcen;
        HIPCHK(hipMemcpyAsync(ctx->cg.p, &S, sizeof(CgState), hipMemcpyHostToDevice, ctx->stream));
        const CgBufs B = cg_bufs(ctx);
        const int gbk = gather_blocks(ctx);
        if (prec == MDN_PREC_MIXED) launch_cg_gather<float>(ctx, cs, (const CgState*)ctx->cg.p, B);
        else launch_cg_gather<double>(ctx, cs, (const CgState*)ctx->cg.p, B);
        hipLaunchKernelGGL(k_cg_fin, dim3(1), dim3(FIN), 0, ctx->stream, cs, ctx->cg.p, B, gbk);
        HIPCHK(hipGetLastError());
        // the state after this step's finalize (and the host state's upload above) is complete
        // before the pinned copy is overwritten
        HIPCHK(d2h(ctx, &S, ctx->cg.p, sizeof(CgState)));
    }
    hold.give();
    ctx->last_cg = S;
    if (!S.done) return fail(ctx, MDN_ERR_STATE, "minimizer did not terminate within %ld batches", launched);
    ctx->cur = S.parity;
    res->error_flags = S.error_flags;
    res->num_energy_call = S.num_energy_call;
    res->num_force_call = S.num_force_call;
    res->num_iter = S.num_iter;
    res->num_safe_mode = S.num_safe_mode;
    res->num_recovery = S.num_recovery;
    res->grad_inf_norm = S.grad_inf_norm;
    res->energy_rel_change = S.energy_rel_change;
    if (S.status == 9)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "more excluded-volume pairs need the Simpson energy than the "
                    "minimizer's capacity (%d per line-search launch)", DEFER_CAP);
    if (S.status != 0) return fail(ctx, S.status, "minimization stopped with status %d", S.status);
    const bool limit = (S.energy_call_limit != 0 && S.num_energy_call > S.energy_call_limit) ||
                       (S.force_call_limit != 0 && S.num_force_call > S.force_call_limit);
    res->call_limit_exceeded = limit;
    res->converged_grad = S.grad_inf_norm < S.grad_tol;
    res->converged_energy = S.energy_rel_change < S.energy_rel_tol;
    double* xres = ctx->x[ctx->cur].p;
    if (S.error_flags == 0) {
        if (p->report_on_call_limit && limit && S.have_min_e) {   // copybackupcoordinates
            HIPCHK(hipMemcpyAsync(xres, ctx->xmin[S.bkpar].p, sizeof(double) * nv, hipMemcpyDeviceToDevice,
                                  ctx->stream));
            res->restored_min_energy = 1;
        }
        if ((st = energy_report(ctx, xres, MDN_PREC_FP64))) return st;
        fill_report(ctx->h_eout, &res->energies_after);
        res->num_energy_call += 1;
    }
    if (coord) HIPCHK(copy_out(ctx, coord, xres, sizeof(double) * nv));
    if (force_out) HIPCHK(copy_out(ctx, force_out, (S.fpar ? ctx->f2 : ctx->f).p, sizeof(double) * nv));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (S.error_flags & MDN_MIN_ERR_LINESEARCH) return fail(ctx, MDN_ERR_LINESEARCH, "line search failed (recovery disabled)");
    return MDN_OK;
}

int mdn_minimize(mdn_ctx* ctx, const mdn_cg_params* p, double* coord, double* force_out, mdn_min_result* res) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (!p || !res) return fail(ctx, MDN_ERR_ARG, "null argument");
    if (p->precision != MDN_PREC_FP64 && p->precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", p->precision);
    if (p->method < 0 || p->method > 2) return fail(ctx, MDN_ERR_ARG, "unknown descent method %d", p->method);
    if (p->line_search != MDN_LS_BACKTRACKING && p->line_search != MDN_LS_QUADRATIC)
        return fail(ctx, MDN_ERR_ARG, "unknown line search %d", p->line_search);
    HIPCHK(hipSetDevice(ctx->device));
    bool gave_up = false;
    st = minimize_run(ctx, p, coord, force_out, res, true, &gave_up);
    return gave_up ? minimize_run(ctx, p, coord, force_out, res, false, &gave_up) : st;
}

}  // extern "C"

// ----------------------------------------------------------------------------------------
// Batched minimizer: many independent systems, one persistent kernel
// ----------------------------------------------------------------------------------------
static void fill_result(const CgState& S, const double* rep_before, const double* rep_after, bool have_after,
                        mdn_min_result* res) {
    memset(res, 0, sizeof(*res));
    fill_report(rep_before, &res->energies_before);
    if (have_after) fill_report(rep_after, &res->energies_after);
    res->error_flags = S.error_flags;
    res->num_energy_call = S.num_energy_call + (have_after ? 1 : 0);
    res->num_force_call = S.num_force_call;
    res->force_call_limit = S.force_call_limit;
    res->energy_call_limit = S.energy_call_limit;
    res->num_iter = S.num_iter;
    res->num_safe_mode = S.num_safe_mode;
    res->num_recovery = S.num_recovery;
    res->grad_inf_norm = S.grad_inf_norm;
    res->grad_tol = S.grad_tol;
    res->energy_rel_change = S.energy_rel_change;
    res->energy_rel_tol = S.energy_rel_tol;
    res->call_limit_exceeded = call_limit_host(S);
    res->converged_grad = S.grad_inf_norm < S.grad_tol;
    res->converged_energy = S.energy_rel_change < S.energy_rel_tol;
    res->restored_min_energy = S.reserved[0];
}

// One system's coordinates or forces: among the parts that go through the ring together, or, from
// pinned or device memory (which the ring's copies by the CPU must not touch), queued by the runtime.
static hipError_t batch_copy(mdn_ctx* L, std::vector<HostCopy>& parts, double* host, double* dev, size_t bytes, bool to_host) {
    if (!pageable(host))
        return to_host ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, L->stream)
                       : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, L->stream);
    parts.push_back(HostCopy{(char*)host, (char*)dev, bytes});
    return hipSuccess;
}

// The persistent kernel of a planned batch.
static int launch_batch(mdn_ctx* L, const TeamPlan& P, int prec) {
    const dim3 g(P.slot.size()), b(TEAM_NT);
    auto launch = [&](auto k) {
        hipLaunchKernelGGL(k, g, b, 0, L->stream, (const BatchItem*)L->batch_items.p, (const TeamSlot*)L->batch_slot.p,
                           (const TeamInfo*)L->batch_team.p, L->batch_ctl.p, (const int*)L->batch_order.p, (int)P.order.size(),
                           L->batch_queue.p, L->team_polls);
        return hipGetLastError();
    };
    if (prec == MDN_PREC_MIXED) HIPCHK_CTX(L, launch(k_cg_team<float, TEAM_NT>));
    else HIPCHK_CTX(L, launch(k_cg_team<double, TEAM_NT>));
    return MDN_OK;
}

extern "C" {

// One batch on the lead context L's stream and buffers. code[i]: system i's status. With teams, large
// systems by teams; again: the systems whose team gave up waiting for its workgroups, each at its
// start (their results are not set).
static int batched_run(mdn_ctx* L, mdn_ctx* const* ctxs, int n, const mdn_cg_params* p, double* const* coords,
                       double* const* forces_out, mdn_min_result* results, int* code, bool teams, std::vector<int>* again) {
    // every context's own work is complete before the lead stream reads its buffers
    for (int i = 0; i < n; i++)
        if (ctxs[i] != L) HIPCHK_CTX(L, hipStreamSynchronize(ctxs[i]->stream));
    std::vector<BatchItem> items(n);
    std::vector<long> cost(n);
    // the systems that start from their device coordinates: x[cur] -> x[0], and where a team takes
    // them into ext, all in one launch
    std::vector<BatchCopy> copies;
    std::vector<const double*> start(n, nullptr);
    std::vector<HostCopy> in;   // what goes onto the device: the given coordinates, then the tables
    long max_nv = 1;
    int max_blk = 1, max_nbb = 1, max_terms = 1;
    for (int i = 0; i < n; i++) {
        mdn_ctx* c = ctxs[i];
        const long nv = 3L * c->n_beads;
        max_nv = std::max(max_nv, nv);
        if (coords[i])
            HIPCHK_CTX(L, batch_copy(L, in, coords[i], c->x[0].p, sizeof(double) * nv, false));
        else   // the context's device coordinates
            start[i] = c->x[c->cur].p;
        if (start[i] && c->cur != 0) copies.push_back(BatchCopy{start[i], c->x[0].p, nv});
        c->cur = 0;
        BatchItem& it = items[i];
        it.s = c->sys;
        it.s.bonded_gather = 1;
        it.s.bead_energy = 1;   // the filament terms' energies with their forces, by the bead blocks
        it.B = cg_bufs(c);
        it.st = c->cg.p;
        it.report = c->eout.p;
        HIPCHK_CTX(L, c->team_part.ensure((size_t)team_wpart_doubles(it.s, SUM_STRIDED)));   // large systems
        it.wpart = c->team_part.p;
        cost[i] = team_cost(it.s);
        max_blk = std::max(max_blk, it.s.blk[NFF]);
        max_nbb = std::max(max_nbb, it.s.nbb);
        max_terms = std::max(max_terms, it.s.blk_nb + it.s.nbb);
    }
    BatchParams P{};
    P.method = p->method;
    P.line_search = p->line_search;
    P.try_recover = p->try_recover;
    P.force_call_limit = p->force_call_limit;
    P.energy_call_limit = p->energy_call_limit;
    P.report_on_call_limit = p->report_on_call_limit;
    P.max_dist = p->max_dist;
    P.lambda_max = p->lambda_max;
    P.grad_tol = p->grad_tol;
    P.energy_rel_tol = p->energy_rel_tol;
    // one workgroup per CU (8 wavefronts at 179 to 250 VGPRs fill it); MDN_BATCH_MAX_WORKGROUPS caps
    // them, so that every workgroup pulls several systems (what a batch larger than the chip does)
    int groups = std::max(1, L->n_cu);
    if (const char* env = getenv("MDN_BATCH_MAX_WORKGROUPS"))
        if (atoi(env) > 0) groups = std::min(groups, atoi(env));
    // a batch's teams may fill every XCD: they need the whole room for teams (taken: single workgroups)
    TeamHold hold(team_room_of(L->device));
    TeamPlan plan = plan_teams(cost, groups, teams ? TEAM_MAX : 1);
    const int room = team_room(L->n_cu);
    if (plan.teamed > 0 && !hold.take(room, room, TEAM_ROOM_WAIT)) plan = plan_teams(cost, groups, 1);
    for (const TeamInfo& t : plan.team)
        if (t.size > 1 && start[t.sys])
            copies.push_back(BatchCopy{start[t.sys], ctxs[t.sys]->ext.p, 3L * ctxs[t.sys]->n_beads});
    const size_t nq = std::max<size_t>(1, plan.order.size());
    HIPCHK_CTX(L, L->batch_items.ensure(n));
    HIPCHK_CTX(L, L->batch_order.ensure(nq));
    HIPCHK_CTX(L, L->batch_queue.ensure(1));
    HIPCHK_CTX(L, L->batch_copy.ensure(std::max<size_t>(1, copies.size())));
    HIPCHK_CTX(L, L->batch_slot.ensure(plan.slot.size()));
    HIPCHK_CTX(L, L->batch_team.ensure(plan.team.size()));
    HIPCHK_CTX(L, L->batch_ctl.ensure(plan.team.size()));
    auto table = [&](void* dev, const void* host, size_t bytes) {
        if (bytes) in.push_back(HostCopy{(char*)host, (char*)dev, bytes});
    };
    table(L->batch_items.p, items.data(), sizeof(BatchItem) * n);
    table(L->batch_copy.p, copies.data(), sizeof(BatchCopy) * copies.size());
    table(L->batch_slot.p, plan.slot.data(), sizeof(TeamSlot) * plan.slot.size());
    table(L->batch_team.p, plan.team.data(), sizeof(TeamInfo) * plan.team.size());
    table(L->batch_order.p, plan.order.data(), sizeof(int) * plan.order.size());
    HIPCHK_CTX(L, copy_parts(L, in.data(), (int)in.size(), false));
    HIPCHK_CTX(L, hipMemsetAsync(L->batch_ctl.p, 0, sizeof(TeamCtl) * plan.team.size(), L->stream));
    HIPCHK_CTX(L, hipMemsetAsync(L->batch_queue.p, 0, sizeof(int), L->stream));
    const BatchItem* di = L->batch_items.p;
    int st;
    if (!copies.empty()) {
        const dim3 cgrid((unsigned)std::min(64L, std::max(1L, (long)ceil_div(max_nv, 256L))),
                         (unsigned)std::min<size_t>(copies.size(), 4096));
        hipLaunchKernelGGL(k_batch_copy, cgrid, dim3(256), 0, L->stream, (const BatchCopy*)L->batch_copy.p, (int)copies.size());
    }
    // a grid's second dimension holds at most 65535 systems: the launches below go in parts
    for (int i0 = 0; i0 < n; i0 += 32768) {
        const unsigned m = (unsigned)std::min(n - i0, 32768);
        const bool mixed = p->precision == MDN_PREC_MIXED;
        const dim3 vg((unsigned)std::min(64, max_nbb), m), b(BLOCK);
        const BatchItem* d = di + i0;
        hipLaunchKernelGGL(k_batch_zero, vg, b, 0, L->stream, d);
        hipLaunchKernelGGL(k_batch_energy<double>, dim3(max_blk, m), b, 0, L->stream, d, 0);
        hipLaunchKernelGGL(k_batch_energy_fin, dim3(m), b, 0, L->stream, d, 0, 0);
        if (mixed) {   // the minimizer's own start energy
            hipLaunchKernelGGL(k_batch_energy<float>, dim3(max_blk, m), b, 0, L->stream, d, 0);
            hipLaunchKernelGGL(k_batch_energy_fin, dim3(m), b, 0, L->stream, d, 0, 18);
            hipLaunchKernelGGL(k_batch_terms<float>, dim3(max_terms, m), b, 0, L->stream, d);
            hipLaunchKernelGGL(k_batch_gather<float>, dim3(max_nbb, m), b, 0, L->stream, d);
        } else {
            hipLaunchKernelGGL(k_batch_terms<double>, dim3(max_terms, m), b, 0, L->stream, d);
            hipLaunchKernelGGL(k_batch_gather<double>, dim3(max_nbb, m), b, 0, L->stream, d);
        }
        hipLaunchKernelGGL(k_batch_init, dim3(m), dim3(SUM_NT), 0, L->stream, d, P, mixed ? 18 : 0);
        HIPCHK_CTX(L, hipGetLastError());
    }
    if ((st = launch_batch(L, plan, p->precision))) return st;
    for (int i0 = 0; i0 < n; i0 += 32768) {
        const unsigned m = (unsigned)std::min(n - i0, 32768);
        const BatchItem* d = di + i0;
        hipLaunchKernelGGL(k_batch_restore, dim3((unsigned)std::min(64, max_nbb), m), dim3(BLOCK), 0, L->stream, d,
                           P.report_on_call_limit);
        hipLaunchKernelGGL(k_batch_energy<double>, dim3(max_blk, m), dim3(BLOCK), 0, L->stream, d, 1);
        hipLaunchKernelGGL(k_batch_energy_fin, dim3(m), dim3(BLOCK), 0, L->stream, d, 1, 9);
    }
    HIPCHK_CTX(L, hipGetLastError());
    // results: every system's state and report gathered on the device and read back at once, then
    // the coordinates (and forces) of every system queued with one synchronization
    HIPCHK_CTX(L, L->batch_states.ensure((size_t)n));
    HIPCHK_CTX(L, L->batch_reports.ensure(27 * (size_t)n));
    hipLaunchKernelGGL(k_batch_collect, dim3(std::min(1024, std::max(1, ceil_div(60L * n, 256)))), dim3(256), 0,
                       L->stream, (const BatchItem*)L->batch_items.p, n, L->batch_states.p, L->batch_reports.p);
    HIPCHK_CTX(L, hipGetLastError());
    std::vector<CgState> states(n);
    std::vector<double> reports(27 * (size_t)n);
    std::vector<TeamCtl> ctl(plan.team.size());
    const HostCopy head[3] = {{(char*)states.data(), (char*)L->batch_states.p, sizeof(CgState) * n},
                              {(char*)ctl.data(), (char*)L->batch_ctl.p, sizeof(TeamCtl) * ctl.size()},
                              {(char*)reports.data(), (char*)L->batch_reports.p, sizeof(double) * 27 * n}};
    HIPCHK_CTX(L, copy_parts(L, head, 3, true));
    hold.give();
    std::vector<char> failed(n, 0);
    for (size_t t = 0; t < plan.team.size(); t++) {
        const int i = plan.team[t].sys;
        if (!ctl[t].failed || i < 0) continue;   // (a workgroup that pulls systems waits for nobody)
        failed[i] = 1;
        again->push_back(i);
        HIPCHK_CTX(L, hipMemsetAsync(ctxs[i]->defer_n.p, 0, sizeof(int), L->stream));
        if (start[i])
            HIPCHK_CTX(L, hipMemcpyAsync(ctxs[i]->x[0].p, ctxs[i]->ext.p, sizeof(double) * 3 * ctxs[i]->n_beads,
                                         hipMemcpyDeviceToDevice, L->stream));
    }
    std::sort(again->begin(), again->end());
    if (teams) {
        L->last_team[0] = plan.teamed;
        L->last_team[1] = (int)again->size();
    }
    std::vector<HostCopy> out;
    for (int i = 0; i < n; i++) {
        if (failed[i]) continue;
        mdn_ctx* c = ctxs[i];
        const CgState& S = states[i];
        const size_t bytes = sizeof(double) * 3 * c->n_beads;
        if (coords[i]) HIPCHK_CTX(L, batch_copy(L, out, coords[i], c->x[S.parity].p, bytes, true));
        if (forces_out && forces_out[i])
            HIPCHK_CTX(L, batch_copy(L, out, forces_out[i], (S.fpar ? c->f2 : c->f).p, bytes, true));
    }
    HIPCHK_CTX(L, copy_parts(L, out.data(), (int)out.size(), true));
    HIPCHK_CTX(L, hipStreamSynchronize(L->stream));
    for (int i = 0; i < n; i++) {
        if (failed[i]) continue;
        mdn_ctx* c = ctxs[i];
        const CgState& S = states[i];
        const double* rep = reports.data() + 27L * i;
        c->last_cg = S;
        c->cur = S.parity;
        const bool ok = S.status == 0 && S.error_flags == 0;
        fill_result(S, rep, rep + 9, ok, &results[i]);
        if (S.status != 0) {
            code[i] = (S.status == ST_NEED_FORCEN || S.status == 9) ? MDN_ERR_UNSUPPORTED : S.status;
            fail(c, code[i], S.status == ST_NEED_FORCEN ? "an excluded-volume pair needed the numerical force fallback, "
                                                       "which the batched minimizer does not run"
                          : S.status == 9 ? "more excluded-volume pairs need the Simpson energy than the capacity"
                                          : "minimization stopped with status %d", S.status);
        } else if (ok && rep[9 + 8] != 0.0) {
            code[i] = MDN_ERR_UNSUPPORTED;
            fail(c, code[i], "excluded-volume pairs beyond the Simpson-energy capacity");
        } else if (S.error_flags & MDN_MIN_ERR_LINESEARCH) {
            code[i] = MDN_ERR_LINESEARCH;
            fail(c, code[i], "line search failed (recovery disabled)");
        }
    }
    return MDN_OK;
}

int mdn_minimize_batched(mdn_ctx* const* ctxs, int32_t n, const mdn_cg_params* p, double* const* coords,
                         double* const* forces_out, mdn_min_result* results) {
    if (!ctxs || n <= 0 || !ctxs[0]) return MDN_ERR_ARG;
    mdn_ctx* L = ctxs[0];
    if (!p || !coords || !results) return fail(L, MDN_ERR_ARG, "null argument");
    if (p->precision != MDN_PREC_FP64 && p->precision != MDN_PREC_MIXED)
        return fail(L, MDN_ERR_ARG, "unknown precision %d", p->precision);
    if (p->method < 0 || p->method > 2) return fail(L, MDN_ERR_ARG, "unknown descent method %d", p->method);
    if (p->line_search != MDN_LS_BACKTRACKING && p->line_search != MDN_LS_QUADRATIC)
        return fail(L, MDN_ERR_ARG, "unknown line search %d", p->line_search);
    for (int i = 0; i < n; i++) {
        mdn_ctx* c = ctxs[i];
        if (!c) return fail(L, MDN_ERR_ARG, "system %d: null context", i);
        if (c->device != L->device) return fail(L, MDN_ERR_ARG, "system %d is on another device", i);
        for (int j = 0; j < i; j++)
            if (ctxs[j] == c) return fail(L, MDN_ERR_ARG, "system %d repeats context %d", i, j);
        int st = need_system(c, true);
        if (st) return fail(L, st, "system %d: %s", i, c->err.c_str());
    }
    HIPCHK_CTX(L, hipSetDevice(L->device));
    std::vector<int> code(n, MDN_OK), again;
    int st = batched_run(L, ctxs, n, p, coords, forces_out, results, code.data(), true, &again);
    if (st) return st;
    if (!again.empty()) {   // by single workgroups, which wait for nobody
        const int m = (int)again.size();
        std::vector<mdn_ctx*> sub(m);
        std::vector<double*> x(m), f(m);
        std::vector<mdn_min_result> res(m);
        std::vector<int> sub_code(m, MDN_OK), none;
        for (int j = 0; j < m; j++) {
            sub[j] = ctxs[again[j]];
            x[j] = coords[again[j]];
            f[j] = forces_out ? forces_out[again[j]] : nullptr;
        }
        if ((st = batched_run(L, sub.data(), m, p, x.data(), f.data(), res.data(), sub_code.data(), false, &none))) return st;
        for (int j = 0; j < m; j++) {
            results[again[j]] = res[j];
            code[again[j]] = sub_code[j];
        }
    }
    for (int i = 0; i < n; i++)   // the first failing system's status
        if (code[i] != MDN_OK) {
            if (ctxs[i] != L) fail(L, code[i], "system %d: %s", i, ctxs[i]->err.c_str());
            return code[i];
        }
    return MDN_OK;
}

// [workgroup size, largest-first order (1), tuned in that call (0)]: fixed, and no times.
int mdn_last_batch_schedule(mdn_ctx* ctx, int32_t* out3, double* tune_ms) {
    if (!ctx || !out3) return MDN_ERR_ARG;
    out3[0] = TEAM_NT;
    out3[1] = 1;
    out3[2] = 0;
    if (tune_ms)
        for (int c = 0; c < MDN_BATCH_CANDIDATES; c++) tune_ms[c] = 0.0;
    return MDN_OK;
}

int mdn_last_team(mdn_ctx* ctx, int32_t* out2) {
    if (!ctx || !out2) return MDN_ERR_ARG;
    out2[0] = ctx->last_team[0];
    out2[1] = ctx->last_team[1];
    return MDN_OK;
}

// Launch statistics of the last minimization: [line-search launches that did work, steps resumed
// after the host-run forceN fallback, force gathers, CG iterations].
int mdn_last_min_stats(mdn_ctx* ctx, int64_t* out) {
    if (!ctx || !out) return MDN_ERR_ARG;
    out[0] = ctx->last_cg.n_ls_launch;
    out[1] = ctx->last_cg.reserved[1];   // steps resumed after the host-run forceN fallback
    out[2] = ctx->last_cg.n_gather_launch;
    out[3] = ctx->last_cg.num_iter;
    return MDN_OK;
}

// ----------------------------------------------------------------------------------------
// Benchmark helpers: device-resident coordinates, HIP events on the context stream
// ----------------------------------------------------------------------------------------
extern "C++" {
template <typename R>
static int bench_forces_t(mdn_ctx* ctx, int32_t iters, double* ms_per_eval, double* kernel_ms) {
    const DevSys& s = ctx->sys;
    const double* x = ctx->x[ctx->cur].p;
    R* slots = reinterpret_cast<R*>(ctx->slots.p);
    const bool pieces = !ctx->bg_eval;
    const int nb = std::max(1, force_blocks(s, pieces));
    int st;
    // warm-up (and fallback check) once
    if ((st = eval_slots(ctx, x, sizeof(R) == 4 ? MDN_PREC_MIXED : MDN_PREC_FP64, pieces))) return st;
    hipEvent_t e0, e1, k0, k1;
    HIPCHK(hipEventCreate(&e0)); HIPCHK(hipEventCreate(&e1)); HIPCHK(hipEventCreate(&k0)); HIPCHK(hipEventCreate(&k1));
    // whole evaluation: terms + gather
    HIPCHK(hipEventRecord(e0, ctx->stream));
    for (int i = 0; i < iters; i++) {
        hipLaunchKernelGGL(k_forces_terms<R>, dim3(nb), dim3(BLOCK), 0, ctx->stream, s, x, slots,
                           ctx->bad_count.p, ctx->bad_list.p, bead_block0(s, pieces), 3, (const double*)nullptr);
        launch_gather_plain<R>(ctx, s, 3, (const R*)slots, 0L, s.slot0[NFF], (const double*)nullptr, ctx->f.p, !pieces);
    }
    HIPCHK(hipEventRecord(e1, ctx->stream));
    // dominant kernel alone
    HIPCHK(hipEventRecord(k0, ctx->stream));
    for (int i = 0; i < iters; i++)
        hipLaunchKernelGGL(k_forces_terms<R>, dim3(nb), dim3(BLOCK), 0, ctx->stream, s, x, slots,
                           ctx->bad_count.p, ctx->bad_list.p, bead_block0(s, pieces), 3, (const double*)nullptr);
    HIPCHK(hipEventRecord(k1, ctx->stream));
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventSynchronize(k1));
    float a = 0, b = 0;
    HIPCHK(hipEventElapsedTime(&a, e0, e1));
    HIPCHK(hipEventElapsedTime(&b, k0, k1));
    if (ms_per_eval) *ms_per_eval = a / iters;
    if (kernel_ms) *kernel_ms = b / iters;
    (void)hipEventDestroy(e0); (void)hipEventDestroy(e1); (void)hipEventDestroy(k0); (void)hipEventDestroy(k1);
    return MDN_OK;
}
}  // extern "C++"

int mdn_bench_forces(mdn_ctx* ctx, int32_t precision, int32_t iters, double* ms_per_eval, double* kernel_ms) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (precision != MDN_PREC_FP64 && precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", precision);
    if (iters <= 0) return fail(ctx, MDN_ERR_ARG, "iters must be positive");
    HIPCHK(hipSetDevice(ctx->device));
    return precision == MDN_PREC_MIXED ? bench_forces_t<float>(ctx, iters, ms_per_eval, kernel_ms)
                                       : bench_forces_t<double>(ctx, iters, ms_per_eval, kernel_ms);
}

// n_vec products (tangents at hb_v) as mdn_hvp_batch launches them, into hb_out.
static int hvp_batch_launch(mdn_ctx* ctx, const double* x, int prec, int n_vec, long slot_stride, long piece_stride) {
    HIPCHK(hipMemsetAsync(ctx->bad_count.p, 0, sizeof(int), ctx->stream));
    launch_tangents(ctx, x, prec, ctx->hb_v.p, n_vec, ctx->hb_slots.p, slot_stride, ctx->hb_piece.p, piece_stride);
    HIPCHK(hipGetLastError());
    gather_tangents(ctx, n_vec, ctx->hb_slots.p, slot_stride, ctx->hb_piece.p, piece_stride, ctx->hb_out.p);
    HIPCHK(hipGetLastError());
    return MDN_OK;
}

int mdn_bench_adjoint(mdn_ctx* ctx, int32_t precision, int32_t iters, const double* v, int32_t n_var, int32_t n_vec,
                      double* ms_per_hvp, double* ms_per_param_grad) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (precision != MDN_PREC_FP64 && precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", precision);
    if (iters <= 0) return fail(ctx, MDN_ERR_ARG, "iters must be positive");
    if (!v || n_var != 3 * ctx->n_beads) return fail(ctx, MDN_ERR_ARG, "n_var must be 3*n_beads = %d", 3 * ctx->n_beads);
    if (n_vec < 1 || n_vec > MDN_HVP_BATCH_CHUNK)
        return fail(ctx, MDN_ERR_ARG, "n_vec must be in [1, %d]", MDN_HVP_BATCH_CHUNK);
    HIPCHK(hipSetDevice(ctx->device));
    const DevSys& s = ctx->sys;
    const double* x = ctx->x[ctx->cur].p;
    const long slot_stride = 3 * std::max(1L, s.slot0[NFF]) + GCHUNK_PAD;
    const long piece_stride = (long)NBOND * 3 * ctx->n_beads;
    if (n_vec == 1) {
        HIPCHK(ctx->tan_v.ensure(n_var));
        HIPCHK(copy_in(ctx, ctx->tan_v.p, v, sizeof(double) * n_var));
    } else {
        HIPCHK(ctx->hb_v.ensure((size_t)n_vec * n_var));
        HIPCHK(ctx->hb_slots.ensure((size_t)n_vec * slot_stride));
        HIPCHK(ctx->hb_piece.ensure((size_t)n_vec * piece_stride));
        HIPCHK(ctx->hb_out.ensure((size_t)n_vec * n_var));
        HIPCHK(hipMemcpyAsync(ctx->hb_v.p, v, sizeof(double) * n_vec * n_var, hipMemcpyHostToDevice, ctx->stream));
    }
    auto hvps = [&]() {
        return n_vec == 1 ? hvp_launch(ctx, x, precision)
                          : hvp_batch_launch(ctx, x, precision, n_vec, slot_stride, piece_stride);
    };
    HIPCHK(ctx->ev_U.ensure(std::max(1, s.n[FF_EXVOL])));
    HIPCHK(ctx->grad_out.ensure(3 * (size_t)std::max(1, ctx->n_cyl)));
    // once with the checks: every pair has a tangent and a closed-form energy at x, so the timed
    // launches below do exactly the work of mdn_hvp (mdn_hvp_batch) and mdn_param_grad on the device
    if ((st = hvps())) return st;
    HIPCHK(hipMemcpyAsync(ctx->h_int, ctx->bad_count.p, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (ctx->h_int[0] != 0)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%d excluded-volume pairs need the numerical force fallback (no tangent)",
                    ctx->h_int[0]);
    if ((st = param_grad_launch(ctx, x, precision, true))) return st;
    HIPCHK(hipStreamSynchronize(ctx->stream));
    if (s.n[FF_EXVOL] > 0 && ctx->h_int[0] != 0)
        return fail(ctx, MDN_ERR_UNSUPPORTED, "%d excluded-volume pairs need the Simpson energy", ctx->h_int[0]);
    hipEvent_t e0, e1, e2;
    HIPCHK(hipEventCreate(&e0)); HIPCHK(hipEventCreate(&e1)); HIPCHK(hipEventCreate(&e2));
    HIPCHK(hipEventRecord(e0, ctx->stream));
    for (int i = 0; i < iters && !st; i++) st = hvps();
    HIPCHK(hipEventRecord(e1, ctx->stream));
    for (int i = 0; i < iters && !st; i++) st = param_grad_launch(ctx, x, precision, false);
    HIPCHK(hipEventRecord(e2, ctx->stream));
    HIPCHK(hipEventSynchronize(e2));
    float a = 0, b = 0;
    HIPCHK(hipEventElapsedTime(&a, e0, e1));
    HIPCHK(hipEventElapsedTime(&b, e1, e2));
    (void)hipEventDestroy(e0); (void)hipEventDestroy(e1); (void)hipEventDestroy(e2);
    if (st) return st;
    if (ms_per_hvp) *ms_per_hvp = a / iters / n_vec;
    if (ms_per_param_grad) *ms_per_param_grad = b / iters;
    return MDN_OK;
}

int mdn_bench_energy(mdn_ctx* ctx, int32_t precision, int32_t iters, double* ms_per_eval) {
    int st = need_system(ctx, true);
    if (st) return st;
    if (precision != MDN_PREC_FP64 && precision != MDN_PREC_MIXED)
        return fail(ctx, MDN_ERR_ARG, "unknown precision %d", precision);
    if (iters <= 0) return fail(ctx, MDN_ERR_ARG, "iters must be positive");
    HIPCHK(hipSetDevice(ctx->device));
    const double* x = ctx->x[ctx->cur].p;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0)); HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, ctx->stream));
    for (int i = 0; i < iters; i++) launch_energy(ctx, x, precision, ctx->h_eout);
    HIPCHK(hipEventRecord(e1, ctx->stream));
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventSynchronize(e1));
    float a = 0;
    HIPCHK(hipEventElapsedTime(&a, e0, e1));
    if (ms_per_eval) *ms_per_eval = a / iters;
    (void)hipEventDestroy(e0); (void)hipEventDestroy(e1);
    return MDN_OK;
}

}  // extern "C"
