// mc.hip -- photon-packet transport on CDNA4: one packet per lane.
//
// Replaces the photon loop of mcpolar.f90:151-170 (sourcephCO2,
// sourceph.f90:7-49; tauint1 / wall_dist / update_pos / find,
// inttau2.f90:7-239; HG scattering in place of stokes, stokes.f90:6-153).
//
// Design:
//  * Each lane owns one packet at a time.  A wave starts on its own first
//    packets; the rest are handed out from a queue head in device memory, a
//    chunk per wave at a time, so waves that draw short histories take more
//    packets and the grid drains together.  The random stream of a packet
//    depends only on its index, never on the lane or the order in which
//    packets are taken.
//  * Random numbers: Philox4x32-10, key = seed, counter = (packet id, event,
//    stream).  One 4-word block per event: launch (radius, azimuth, specular
//    test, first tau), interaction (albedo test, HG cos, HG azimuth, next
//    tau), Fresnel test at a z face.  The FP64 oracle draws identically.
//  * Two phases.  A walk step moves every lane that needs no random numbers
//    across one voxel face (or finds that its next interaction lies inside
//    the current voxel, or that it reached a z face of the grid where a
//    Fresnel test is due).  Such a lane then waits with its event pending.
//    The random phase (one Philox block plus the launch, interaction or
//    Fresnel event for every pending lane) runs once at least `rng_batch`
//    lanes of the wave wait, or every lane with a packet does: the costly
//    part then runs with most lanes active instead of for one or two.
//  * Voxel walk (Amanatides-Woo DDA): per packet segment an origin o (cm,
//    grid coordinates), the distance t travelled from it, and the distances
//    Tx, Ty, Tz from o to the next face crossed on each axis.  A crossing
//    takes the smallest T, adds one voxel's span on that axis to it, and
//    steps the cell and the linear voxel index.  Scattering or a reflection
//    starts a new segment.  Voxels with mu_t = 0 (ablated) are crossed in
//    free flight.  Where mu_t follows from the material (the table model), a
//    crossing loads the material's byte and takes mu_t from the table in LDS,
//    and an event loads nothing: 8 MB instead of 40 MB of grid at 200^3, of
//    which each XCD's 4 MB L2 holds the part under the beam.
//  * What bounds it: on fresh tissue, whose deposits the LDS box takes, issue
//    and latency of the loop (1e8 packets on the 200^3 skin, 3.4 device adds a
//    packet: 59.5 ms, 57.0 with the device adds left out); past a crater or in
//    a wide beam, the device adds (the same skin after 3 cycles, 52.9 a packet:
//    271 ms at 2.0e10 adds/s, 162 without them); a short run, the chain of events of
//    its longest packets.  The pass as straight code with selects, the
//    absorbed packets' tally merged into the pass, LDS counts of rare ends,
//    the byte loads, and no draws from a drained queue took 1e8 packets on the
//    fresh skin from 82 to 59.5 ms, on the crater with 31 device adds a packet from
//    187 to 160, with 54 from 306.6 to 304.8 (another card 10 % less), 1e6 at
//    100^3 from 6.5 to 4.6 (one 1024-lane block a CU).
//  * Tally: path length is summed in a register while the packet stays in a
//    voxel and written with one FP64 atomic add per voxel visit (at exit or
//    absorption).  The absorbed fraction per voxel is mu_a * L.  Voxels with
//    mu_t = 0 absorb nothing and are crossed without a tally.  The global
//    atomic rate (~2.4e10/s on MI355X whatever the address spread) bounds
//    a kernel that sends every visit to the device tally.  Each
//    block therefore sums the visits to a cube of voxels on the beam axis in
//    LDS (mc_box_kernel), placed in z where the last run's path was largest
//    (box_plane_kernel, box_window_kernel), and adds the cube to the tally
//    once at exit.  By default the box holds fixed-point sums in 16-bit
//    integers, two voxels per 32-bit word (units of 2^-13 of dx + dy + dz):
//    four times the voxels of an FP64 box in the same LDS, integer LDS adds
//    cost less than FP64 ones, and an integer sum does not depend on the
//    order of the adds.  Each add that wraps a 16-bit slot hands 2^16 units
//    to the device tally (box_carry), so no sum is lost.
//  * Transcendentals use the hardware approximations (v_log, v_sin/v_cos
//    in revolutions, v_sqrt, v_rcp/v_rsq; ~1 ulp): they only shape sampled
//    distances and directions, whose distributions the parity tests check.
#include "tam_internal.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float neg_ln(float u) { return -0.69314718f * __builtin_amdgcn_logf(u); }
// sin and cos of 2*pi*t for t in [0, 1): the hardware takes revolutions
__device__ __forceinline__ void sincos_rev(float t, float* s, float* c)
{
    *s = __builtin_amdgcn_sinf(t);
    *c = __builtin_amdgcn_cosf(t);
}

__device__ __forceinline__ float fresnel(float ni, float nt, float ci)
{
    const float si = fsqrt(fmaxf(0.f, 1.f - ci * ci));
    const float st = ni * rcp(nt) * si;
    if (st >= 1.f) return 1.f;
    const float ct = fsqrt(1.f - st * st);
    const float rs = (ni * ci - nt * ct) * rcp(ni * ci + nt * ct);
    const float rp = (ni * ct - nt * ci) * rcp(ni * ct + nt * ci);
    return 0.5f * (rs * rs + rp * rp);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// the wave's lowest active lane holds v; every lane gets it
__device__ __forceinline__ uint64_t bcast_first(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// distance from o (inside [lo, lo + d]) to the face crossed first along u
__device__ __forceinline__ float face_dist(float o, float lo, float d, float u, float iu)
{
    return u > 0.f ? (lo + d - o) * iu : (u < 0.f ? (lo - o) * iu : 3.0e38f);
}

constexpr uint32_t kMaxEvents = 1u << 24;   // walk steps + random events of one packet
constexpr int kBoxUnitBits = 13;            // fixed-point box unit: 2^-13 of dx + dy + dz

constexpr long kLdsOwn = 1024;              // LDS per block kept for the kernel's own use (counts, material table)
constexpr long kCountLds = sizeof(unsigned long long) * TAM_CNT_N;     // a block's counts, static
constexpr int kTabMax = 64;                 // materials in the LDS of a kernel without the box
// Entries per wave in a batched block's own LDS: what kLdsOwn holds beside the
// counts.  Tissues of more entries take mu_t from the array as before (eight of
// four materials and air, 4 blocks a CU: 44.5 ms; with one material 43.8).
constexpr int kBatchTab = 4;
constexpr long kBatchLds = 4 * (kCountLds + kBatchTab * (long)sizeof(MatEntry));   // a batched block's static LDS
static_assert(kCountLds <= kLdsOwn && kBatchLds <= kLdsOwn, "the boxes leave kLdsOwn bytes of a block's LDS");

// The LDS tally box of a launch: voxels [o, o + n).
struct BoxGeom {
    int o[3], n[3];
};

// A fixed-point box add whose carry test is still to run: the slot (-1:
// none), its word's value before the add, the add, and the tally voxel.
struct BoxAdd {
    int i;
    uint32_t old, q, v;
};

// Path length into the tally: voxels inside the block's LDS box are summed
// there (BT = uint16_t: 16-bit fixed point, two slots per 32-bit word, slot
// bi in half bi & 1; BT = double: FP64), the rest go to the FP64 device tally
// directly.  Returns 1 for a deposit into the box.  A fixed-point add leaves
// its carry test in pa (box_carry), so that the LDS return is awaited after
// the lane's other work; a deposit of 2^16 units or more (a path over 8
// (dx + dy + dz) in one visit) goes to the tally directly.
template <bool BOX, class BT>
__device__ __forceinline__ uint32_t tally_add(const McArgs& a, BT* box, const BoxGeom& g, uint32_t v, int ci,
                                              int cj, int ck, float l, BoxAdd& pa)
{
    if (BOX) {
        const unsigned bx = (unsigned)(ci - g.o[0]), by = (unsigned)(cj - g.o[1]), bz = (unsigned)(ck - g.o[2]);
        if (bx < (unsigned)g.n[0] && by < (unsigned)g.n[1] && bz < (unsigned)g.n[2]) {
            const unsigned bi = bx + (unsigned)g.n[0] * (by + (unsigned)g.n[1] * bz);
            if constexpr (std::is_same<BT, uint16_t>::value) {
                const float qf = rintf(l * a.box_scale);
                if (qf < 65536.f) {
                    pa.i = (int)bi;
                    pa.q = (uint32_t)qf;
                    pa.v = v;
                    pa.old = __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(box) + (bi >> 1),
                                                    pa.q << ((bi & 1u) * 16u), __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
                    return 1u;
                }
            } else {
                __hip_atomic_fetch_add(&box[bi], (BT)l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                return 1u;
            }
        }
    }
    unsafeAtomicAdd(&a.tally[v], (double)l);
    return 0u;
}

// The carry test of a 16-bit box add.  A word holds the slots of two voxels
// that are x-neighbours: the even slot in the low half, the next voxel in the
// high half.  An add to the low half that wraps it carries 1 into the high
// half: the low voxel's 2^16 units go to the tally, and 1 unit comes off the
// high voxel there.  An add (to either half) that takes the word past 2^32
// wraps the high half: the high voxel's 2^16 units go to the tally.  The
// returned old value shows each wrap to exactly the add that made it, so the
// slots plus these carries always equal the sums of the adds.
template <class BT>
__device__ __forceinline__ void box_carry(const McArgs& a, BT* box, BoxAdd& pa)
{
    if constexpr (std::is_same<BT, uint16_t>::value) {
        if (pa.i >= 0) {
            const uint32_t sh = ((uint32_t)pa.i & 1u) * 16u;
            const uint32_t vlo = sh ? pa.v - 1u : pa.v, vhi = vlo + 1u;
            if (sh == 0u && (pa.old & 0xffffu) + pa.q >= 0x10000u) {
                unsafeAtomicAdd(&a.tally[vlo], 65536.0 * a.box_quantum);
                unsafeAtomicAdd(&a.tally[vhi], -a.box_quantum);
            }
            if ((uint64_t)pa.old + ((uint64_t)pa.q << sh) >= 0x100000000ull)
                unsafeAtomicAdd(&a.tally[vhi], 65536.0 * a.box_quantum);
        }
        pa.i = -1;
    }
}

// A box slot's sum in path length
__device__ __forceinline__ double box_path(uint16_t s, const McArgs& a) { return (double)s * a.box_quantum; }
__device__ __forceinline__ double box_path(double s, const McArgs&) { return s; }

// A packet's state in its lane.  The first two take walk passes, the next
// three wait for the random phase.
enum : int { ST_WALK = 0, ST_DEAD = 1, ST_LAUNCH = 2, ST_INTERACT = 3, ST_FRESNEL = 4, ST_IDLE = 5 };

// Product and difference that keep their own rounding: a walk must take the
// same steps in every kernel, so what the compiler may contract is not left
// to the code around it.
__device__ __forceinline__ float mul_r(float x, float y)
{
#pragma clang fp contract(off)
    return x * y;
}
__device__ __forceinline__ float sub_r(float x, float y)
{
#pragma clang fp contract(off)
    return x - y;
}

// Packets that a wave draws at once while `left` are in the queue: half of its
// share of them (per: 0.5 / waves), 64 to 256.  The draws are returning adds to one
// address, 12 ns each one after the other, so they are few while much is left: 1e7
// packets of a pure absorber, which end after one event, took 1.95 ms in draws of 64,
// 0.89 of 256, 0.65 so.  A wave's last draw is a packet a lane, so that the waves
// end together (quarter shares: 0.85 ms; up to 1024 at once: 0.38, but 1e7 long
// histories at 100^3 31.2 ms against 30.5).
__host__ __device__ __forceinline__ uint32_t draw_size(uint64_t left, float per)
{
    const float c = (float)left * per;
    return c >= 256.f ? 256u : c >= 64.f ? (uint32_t)c & ~63u : 64u;
}

// The transport of one instance by the calling wave's lanes, until its
// packet queue is drained; the fate counters go to sums (TAM_CNT_N words of
// LDS).
// nw > 0: the launch's nw waves all start on this queue, wave `wid` with its
// own first share of the packets; the queue head counts what is drawn after
// those.
// TAB: mu_t is a function of the material (McArgs.mut_by_mat) and tab is the
// material table in LDS: a crossing then loads one byte per lane, which keeps
// a 200^3 grid's transport in the XCDs' L2, and an event loads nothing.
// Otherwise tab is the table in device memory and a crossing loads mu_t.
template <bool BOX, class BT, bool TAB>
__device__ __forceinline__ void transport(const McArgs& a, BT* box, const BoxGeom& g, const MatEntry* tab,
                                          unsigned long long* sums, uint32_t wid, uint32_t nw)
{
    unsigned long long* head = a.counters + TAM_CNT_N;     // queue head, packets drawn
    const uint32_t nxy = (uint32_t)a.nx * (uint32_t)a.ny;
    const float idx_ = rcp(a.dx), idy_ = rcp(a.dy);
    const float ztop = a.dz * (float)a.nz;
    const uint32_t batch = (uint32_t)a.rng_batch;
    const uint64_t npk = a.dyn_npk ? (uint64_t)*a.dyn_npk : a.npk;
    const uint32_t stream = a.dyn_stream ? *a.dyn_stream : a.stream;
    auto count = [&](int i) { atomicAdd(&sums[i], 1ull); };     // escapes and other rare ends

    uint32_t c_cross = 0, c_inter = 0, c_tally = 0, c_box = 0, c_abs = 0, c_spec = 0;
    BoxAdd pa{-1, 0u, 0u, 0u};

    // wave-uniform queue state: packets [pool, pool_end) are this wave's.
    // The first share, at most a packet per lane, needs no draw, and with
    // fewer packets than lanes it spreads them over all waves.
    const uint64_t share = nw ? (npk >= (uint64_t)nw * 64u ? 64u : (npk + nw - 1) / nw) : 0u;
    const uint64_t queue0 = share * nw;                    // first packet the head hands out
    bool dry = queue0 >= npk;                              // nothing left to draw
    const float per = nw ? 0.5f / (float)nw : 0.f;
    uint32_t chunk = nw ? draw_size(dry ? 0u : npk - queue0, per) : 256u;      // packets drawn at once
    uint64_t pool = share * wid, pool_end = pool + share;
    if (pool_end > npk) pool_end = npk > pool ? npk : pool;

    int st = ST_IDLE;
    uint64_t pid = 0;
    uint32_t ev = 0, nev = 0;                  // Philox event counter; steps of this packet
    int ci = 0, cj = 0, ck = 0;
    uint32_t v = 0;                            // linear voxel index of (ci, cj, ck)
    float mu = 0.f;                            // mu_t of voxel v
    int mat = 0;                               // material of v (TAB; otherwise loaded when an event is pending)
    float ox = 0.f, oy = 0.f, oz = 0.f;        // segment origin, cm
    float t = 0.f;                             // distance travelled from the origin
    float Tx = 0.f, Ty = 0.f, Tz = 0.f;        // distance from the origin to the next face per axis
    float ux = 0.f, uy = 0.f, uz = -1.f;
    float sx = 0.f, sy = 0.f, sz = 0.f;        // path across one voxel per axis (unused where u == 0)
    float tau = 0.f, lacc = 0.f;               // optical depth left; path in this voxel
    float nin = 1.f, nout = 1.f;               // indices at a pending Fresnel test

    for (;;) {
        // ---- lanes without a packet take the next ones from the queue
        const uint64_t wm = ballot(st == ST_IDLE);
        if (wm) {
            const uint32_t cnt = (uint32_t)__popcll(wm);
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(wm >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)wm, 0u));
            const uint64_t avail = pool_end - pool;
            uint64_t mine = pool + rank;
            if (avail < cnt) {
                uint64_t nb = npk;
                const uint32_t got = chunk;
                if (!dry) {
                    if (rank == 0 && st == ST_IDLE) nb = queue0 + atomicAdd(head, (unsigned long long)got);
                    // the lowest lane wanting a packet is not always the lowest
                    // active lane: pass the chunk base through the wave
                    nb = __shfl(nb, (int)(__ffsll((long long)wm) - 1), 64);
                    nb = bcast_first(nb);
                    // a wave's last lanes end one by one: each would draw again,
                    // and the returning adds of all waves to the head queue up
                    dry = nb + got >= npk;
                    if (nw && !dry) chunk = draw_size(npk - nb - got, per);
                }
                if (rank >= avail) mine = nb + (rank - avail);
                pool = nb + (cnt - avail);
                pool_end = nb + got;
                if (pool_end > npk) pool_end = npk > nb ? npk : nb;
                if (pool > pool_end) pool = pool_end;
            } else {
                pool += cnt;
            }
            if (st == ST_IDLE) {
                if (mine >= npk) break;            // queue drained: this lane is done
                st = ST_LAUNCH;
                pid = a.p0 + mine;
                ev = 0;
                nev = 0;
            }
        }

        const uint64_t am = ballot(true);
        // `batch` of 64 lanes, in proportion where fewer are left: the wave of
        // a draining queue does not wait for all of its last lanes
        const uint32_t need = max(1u, ((uint32_t)__popcll(am) * batch + 32u) >> 6);
        const uint64_t pm = ballot(st >= ST_LAUNCH);
        if ((uint32_t)__popcll(pm) >= need || pm == am) {
            // ================= random phase: lanes with a pending event ====
            if (st >= ST_LAUNCH) {
                const uint4 r = philox4x32_10(make_uint4((uint32_t)pid, (uint32_t)(pid >> 32), ev, stream),
                                              a.key0, a.key1);
                ++ev;
                const int kind = st;
                st = ST_WALK;
                if (kind == ST_LAUNCH) {
                    // sourcephCO2 with a beam profile (sourceph.f90:7-49)
                    const float u0 = u01(r.x), u1 = u01(r.y), u2 = u01(r.z), u3 = u01(r.w);
                    const float rad = (a.beam == TAM_BEAM_TOPHAT) ? a.radius * fsqrt(u0)
                                                                   : a.radius * fsqrt(0.5f * neg_ln(u0));
                    float sn, cs;
                    sincos_rev(u1, &sn, &cs);
                    const float x = a.cx + rad * cs, y = a.cy + rad * sn;
                    ci = (int)floorf(x * idx_);
                    cj = (int)floorf(y * idy_);
                    ck = a.nz - 1;
                    const bool inside = x >= 0.f && y >= 0.f && ci >= 0 && ci < a.nx && cj >= 0 && cj < a.ny;
                    // Every launch lane sets the whole walk state: a packet
                    // that misses the grid or is reflected ends here, and its
                    // state is never read (voxel 0 stands in for its loads).
                    // One straight path keeps the state in its registers.
                    v = inside ? (uint32_t)ci + (uint32_t)a.nx * (uint32_t)cj + nxy * (uint32_t)ck : 0u;
                    mat = a.mat[v];
                    if (!TAB) mu = a.mut[v];
                    const bool spec = inside && u2 < tab[mat].rsp_top;
                    c_spec += spec ? 1u : 0u;
                    if (!inside) count(TAM_CNT_MISSED);
                    if (!inside || spec) st = ST_IDLE;
                    const float xl = (float)ci * a.dx, yl = (float)cj * a.dy;
                    ox = fminf(fmaxf(x, xl), xl + a.dx);
                    oy = fminf(fmaxf(y, yl), yl + a.dy);
                    oz = ztop;
                    ux = 0.f; uy = 0.f; uz = -1.f;
                    sx = 0.f; sy = 0.f; sz = a.dz;
                    t = 0.f;
                    Tx = 3.0e38f; Ty = 3.0e38f; Tz = a.dz;
                    tau = neg_ln(u3);
                    lacc = 0.f;
                }
                if (kind == ST_INTERACT) {
                    const MatEntry me = tab[mat];
                    if (TAB) mu = me.mut;
                    // interaction inside voxel v, tau / mu beyond the current point
                    const float s = tau * rcp(mu);
                    lacc += s;
                    const float tt = t + s;
                    const float xl = (float)ci * a.dx, yl = (float)cj * a.dy, zl = (float)ck * a.dz;
                    ox = fminf(fmaxf(ox + tt * ux, xl), xl + a.dx);
                    oy = fminf(fmaxf(oy + tt * uy, yl), yl + a.dy);
                    oz = fminf(fmaxf(oz + tt * uz, zl), zl + a.dz);
                    ++c_inter;
                    if (!(u01(r.x) < me.albedo)) {
                        // absorbed: the next walk pass leaves its path in the
                        // tally and ends the packet
                        ++c_abs;
                        st = ST_DEAD;
                    } else {
                        // Henyey-Greenstein deflection, MCML direction-cosine update
                        float ct;
                        if (me.inv2g == 0.f) {
                            ct = 2.f * u01(r.y) - 1.f;
                        } else {
                            const float q = me.omg2 * rcp(1.f - me.g + 2.f * me.g * u01(r.y));
                            ct = (me.opg2 - q * q) * me.inv2g;
                        }
                        ct = fminf(fmaxf(ct, -1.f), 1.f);
                        const float st_ = fsqrt(1.f - ct * ct);
                        float sp, cp;
                        sincos_rev(u01(r.z), &sp, &cp);
                        float nx_, ny_, nz_;
                        if (fabsf(uz) > 0.99999f) {
                            nx_ = st_ * cp;
                            ny_ = st_ * sp;
                            nz_ = uz >= 0.f ? ct : -ct;
                        } else {
                            const float w2 = 1.f - uz * uz;
                            const float rt = __builtin_amdgcn_rsqf(w2);    // 1/sqrt(1-uz^2)
                            nx_ = st_ * (ux * uz * cp - uy * sp) * rt + ux * ct;
                            ny_ = st_ * (uy * uz * cp + ux * sp) * rt + uy * ct;
                            nz_ = -st_ * cp * (w2 * rt) + uz * ct;
                        }
                        const float inv = __builtin_amdgcn_rsqf(nx_ * nx_ + ny_ * ny_ + nz_ * nz_);
                        ux = nx_ * inv; uy = ny_ * inv; uz = nz_ * inv;
                        const float iux = rcp(ux), iuy = rcp(uy), iuz = rcp(uz);
                        sx = mul_r(a.dx, fabsf(iux));
                        sy = mul_r(a.dy, fabsf(iuy));
                        sz = mul_r(a.dz, fabsf(iuz));
                        t = 0.f;
                        Tx = face_dist(ox, xl, a.dx, ux, iux);
                        Ty = face_dist(oy, yl, a.dy, uy, iuy);
                        Tz = face_dist(oz, zl, a.dz, uz, iuz);
                        tau = neg_ln(u01(r.w));
                    }
                }
                if (kind == ST_FRESNEL) {
                    // Fresnel test at a z face of the grid (the crossing is tallied)
                    const bool top = uz > 0.f;
                    if (u01(r.x) < fresnel(nin, nout, fabsf(uz))) {
                        // reflect: new segment from the point on the face
                        const float xl = (float)ci * a.dx, yl = (float)cj * a.dy, zl = (float)ck * a.dz;
                        ox = fminf(fmaxf(ox + t * ux, xl), xl + a.dx);
                        oy = fminf(fmaxf(oy + t * uy, yl), yl + a.dy);
                        oz = top ? zl + a.dz : zl;
                        Tx -= t;
                        Ty -= t;
                        t = 0.f;
                        uz = -uz;
                        Tz = sz;
                    } else {
                        count(TAM_CNT_ESC0 + (top ? TAM_FACE_ZHI : TAM_FACE_ZLO));
                        st = ST_IDLE;
                    }
                }
            }
        }
        // ================= walk phase: face crossings, one per lane and
        // pass, until `need` lanes wait for a random event or a packet (or
        // every lane does).  Staying in this loop keeps the walk state in
        // place between crossings.  A pass is nearly straight code: the three
        // axes' steps are selects, and only tallies and grid faces branch.
        {
            uint64_t sm = ballot(st >= ST_LAUNCH);
            while ((uint32_t)__popcll(sm) < need && sm != am) {
                if (st < ST_LAUNCH) {
                    if (TAB) mu = tab[mat].mut;
                    const bool by = Ty < Tx;
                    const float txy = by ? Ty : Tx;
                    const bool bz = Tz < txy;
                    const float tn = bz ? Tz : txy;
                    const bool live = st == ST_WALK;
                    const float s = live ? fmaxf(tn - t, 0.f) : 0.f;
                    const float ms = mul_r(mu, s);
                    if (nev >= kMaxEvents && live) {
                        // a packet that neither escapes nor is absorbed within
                        // kMaxEvents steps (e.g. total internal reflection in a
                        // non-absorbing slab) is abandoned, so every lane's loop ends
                        count(TAM_CNT_KILLED);
                        st = ST_IDLE;
                    } else if (ms < tau || !live) {
                        // crossing (or a dead packet's last tally)
                        ++nev;
                        lacc += s;
                        // mu_t = 0 (ablated): nothing is absorbed, and an add costs
                        if (mu > 0.f) {
                            c_box += tally_add<BOX, BT>(a, box, g, v, ci, cj, ck, lacc, pa);
                            ++c_tally;
                        }
                        lacc = 0.f;
                        if (!live) {
                            st = ST_IDLE;
                        } else {
                            tau = sub_r(tau, ms);
                            t = tn;
                            ++c_cross;
                            const bool ay = by && !bz, ax = !by && !bz;
                            const int kx = ux > 0.f ? 1 : -1, ky = uy > 0.f ? 1 : -1, kz = uz > 0.f ? 1 : -1;
                            const bool zface = bz && (unsigned)(ck + kz) >= (unsigned)a.nz;
                            const bool az = bz && !zface;
                            Tx += ax ? sx : 0.f;
                            Ty += ay ? sy : 0.f;
                            Tz += az ? sz : 0.f;
                            ci += ax ? kx : 0;
                            cj += ay ? ky : 0;
                            ck += az ? kz : 0;
                            v += (uint32_t)(ax ? kx : (ay ? (ky > 0 ? a.nx : -a.nx) : (az ? (kz > 0 ? (int)nxy : -(int)nxy) : 0)));
                            if (zface || (unsigned)ci >= (unsigned)a.nx || (unsigned)cj >= (unsigned)a.ny) {
                                int face = ax ? (kx > 0 ? TAM_FACE_XHI : TAM_FACE_XLO)
                                              : (ky > 0 ? TAM_FACE_YHI : TAM_FACE_YLO);
                                st = ST_IDLE;
                                if (zface) {
                                    // z face of the grid: Fresnel test where the index changes
                                    nout = kz > 0 ? a.n_zhi : a.n_zlo;
                                    nin = tab[TAB ? mat : (int)a.mat[v]].n;
                                    if (nout > 0.f && nout != nin) st = ST_FRESNEL;
                                    face = kz > 0 ? TAM_FACE_ZHI : TAM_FACE_ZLO;
                                }
                                if (st == ST_IDLE) count(TAM_CNT_ESC0 + face);
                            } else if (TAB) {
                                mat = a.mat[v];
                            } else {
                                mu = a.mut[v];
                            }
                        }
                        box_carry<BT>(a, box, pa);
                    } else {
                        ++nev;
                        st = ST_INTERACT;
                        if (!TAB) mat = a.mat[v];
                    }
                }
                sm = ballot(st >= ST_LAUNCH);
            }
        }
    }

    // ---- the wave's work counters ------------------------------------------
    // (lanes leave the loop one by one as the queue drains; the reduction
    // runs once every lane of the wave has left)
    const uint32_t vals[6] = {c_abs, c_spec, c_cross, c_inter, c_tally, c_box};
    const int slot[6] = {TAM_CNT_ABSORBED, TAM_CNT_SPECULAR, TAM_CNT_CROSS, TAM_CNT_INTER, TAM_CNT_TALLY, TAM_CNT_BOX};
    const bool leader = (threadIdx.x & 63) == 0;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const uint32_t w = wave_sum(vals[i]);
        if (leader && w) atomicAdd(&sums[slot[i]], (unsigned long long)w);
    }
}

// A block's counts (LDS) reach the device counters as one add each:
// thousands of waves adding to the same few addresses would take as long as a
// short run.
__device__ __forceinline__ void add_counts(const McArgs& a, const unsigned long long* sums, int i)
{
    if (i < TAM_CNT_N && sums[i]) atomicAdd(&a.counters[i], sums[i]);
}

// the material table's first `ntab` entries into LDS, by the block's threads
__device__ __forceinline__ void stage_table(const McArgs& a, MatEntry* tab, int ntab, int i, int n)
{
    const float* src = reinterpret_cast<const float*>(a.mtab);
    float* dst = reinterpret_cast<float*>(tab);
    for (int q = i; q < ntab * (int)(sizeof(MatEntry) / 4); q += n) dst[q] = src[q];
}

// a.ntab > 0: the launch's dynamic LDS holds that many table entries
template <bool TAB>
__global__ __launch_bounds__(256) void mc_kernel(McArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char mc_lds[];
    __shared__ unsigned long long sums[TAM_CNT_N];
    MatEntry* tab = reinterpret_cast<MatEntry*>(mc_lds);
    if (threadIdx.x < TAM_CNT_N) sums[threadIdx.x] = 0ull;
    if (TAB) stage_table(a, tab, a.ntab, threadIdx.x, 256);
    __syncthreads();
    transport<false, double, TAB>(a, nullptr, BoxGeom{}, TAB ? tab : a.mtab, sums,
                                  blockIdx.x * 4u + (threadIdx.x >> 6), gridDim.x * 4u);
    __syncthreads();
    add_counts(a, sums, threadIdx.x);
}

// The same with the block-private LDS tally box: cleared first, added to the
// device tally (one atomic per touched voxel) once every wave of the block
// has drained the queue.  NT = 256, or 1024: one block of 16 waves per CU
// holds one box of the CU's whole LDS instead of four quarter-size copies.
// BT = uint16_t (16-bit fixed point, the default box) or double.
// The material table (TAB) follows the box in the dynamic LDS.
template <int NT, class BT, bool TAB>
__global__ __launch_bounds__(NT) void mc_box_kernel(McArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char box_lds[];
    BT* box = reinterpret_cast<BT*>(box_lds);
    // geometry: chosen by box_window_kernel (inside the grid, at most the
    // LDS this launch was given), or the launch's default
    BoxGeom g;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        g.o[q] = a.box_geom ? __builtin_amdgcn_readfirstlane(a.box_geom[q]) : a.box_o[q];
        g.n[q] = a.box_geom ? __builtin_amdgcn_readfirstlane(a.box_geom[3 + q]) : a.box_n[q];
    }
    const int nbox = g.n[0] * g.n[1] * g.n[2];
    for (int i = threadIdx.x; i < nbox; i += NT) box[i] = (BT)0;
    __shared__ unsigned long long sums[TAM_CNT_N];
    MatEntry* tab = reinterpret_cast<MatEntry*>(box_lds + a.tab_off);
    if (threadIdx.x < TAM_CNT_N) sums[threadIdx.x] = 0ull;
    if (TAB) stage_table(a, tab, a.ntab, threadIdx.x, NT);
    __syncthreads();
    transport<true, BT, TAB>(a, box, g, TAB ? tab : a.mtab, sums, blockIdx.x * (NT / 64) + (threadIdx.x >> 6),
                             gridDim.x * (NT / 64));
    __syncthreads();
    add_counts(a, sums, threadIdx.x);
    // Each block starts its adds at another place of the box: blocks end
    // together, and all of them walking the box from its start meet on the
    // same few memory channels.
    const uint32_t nxy = (uint32_t)a.nx * (uint32_t)a.ny;
    const int start = (int)((uint64_t)blockIdx.x * (uint32_t)nbox / gridDim.x) & ~63;
    for (int q = threadIdx.x; q < nbox; q += NT) {
        const int i = q + start < nbox ? q + start : q + start - nbox;
        const double s = box_path(box[i], a);
        if (s != 0.0) {
            const int bx = i % g.n[0], by = (i / g.n[0]) % g.n[1], bz = i / (g.n[0] * g.n[1]);
            const uint32_t v = (uint32_t)(g.o[0] + bx) + (uint32_t)a.nx * (uint32_t)(g.o[1] + by) +
                               nxy * (uint32_t)(g.o[2] + bz);
            unsafeAtomicAdd(&a.tally[v], s);
        }
    }
}

// Placement of the LDS tally box in z.  box_plane_kernel: one block per z
// plane sums the last run's tally (path length, in proportion to the voxel
// visits, i.e. the deposits a box would take) over the box's footprint,
// skipping voxels removed since (mu_t = 0: ablated after that run);
// box_window_kernel: one block sums every window of d consecutive planes
// (plane sums staged in LDS, one window per lane) and keeps the largest,
// ties to the higher window; with no path at all the box sits at the top.
struct BoxPlace {
    int sd, d, ox, oy;                             // footprint sd x sd at (ox, oy), d planes
};

__global__ __launch_bounds__(256) void box_plane_kernel(const double* __restrict__ src, const float* __restrict__ mut,
                                                        int nx, int ny, BoxPlace bp, double* __restrict__ psum)
{
    __shared__ double red[4];
    const int k = blockIdx.x;
    double t = 0.0;
    for (int q = threadIdx.x; q < bp.sd * bp.sd; q += 256) {
        const int i = bp.ox + q % bp.sd, j = bp.oy + q / bp.sd;
        const long v = (long)i + (long)nx * (j + (long)ny * k);
        if (mut[v] > 0.f) t += src[v];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) psum[k] = red[0] + red[1] + red[2] + red[3];
}

constexpr int BOX_MAX_NZ = 4096;                  // tam_create's largest grid edge

__global__ __launch_bounds__(256) void box_window_kernel(const double* __restrict__ psum, int nz, BoxPlace bp,
                                                         int* __restrict__ out)
{
    __shared__ double sp[BOX_MAX_NZ];
    __shared__ double wb[4];
    __shared__ int wo[4];
    for (int k = threadIdx.x; k < nz; k += 256) sp[k] = psum[k];
    __syncthreads();
    double best = -1.0;                            // sums are >= 0: any window beats it
    int bo = -1;
    for (int o = threadIdx.x; o <= nz - bp.d; o += 256) {   // window [o, o + d)
        double w = 0.0;
        for (int k = 0; k < bp.d; ++k) w += sp[o + k];
        if (w > best || (w == best && o > bo)) {
            best = w;
            bo = o;
        }
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const double ow = __shfl_xor(best, s, 64);
        const int oo = __shfl_xor(bo, s, 64);
        if (ow > best || (ow == best && oo > bo)) {
            best = ow;
            bo = oo;
        }
    }
    if ((threadIdx.x & 63) == 0) {
        wb[threadIdx.x >> 6] = best;
        wo[threadIdx.x >> 6] = bo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q)
            if (wb[q] > best || (wb[q] == best && wo[q] > bo)) {
                best = wb[q];
                bo = wo[q];
            }
        out[0] = bp.ox;
        out[1] = bp.oy;
        out[2] = best > 0.0 ? bo : nz - bp.d;
        out[3] = bp.sd;
        out[4] = bp.sd;
        out[5] = bp.d;
    }
}

// The cube of at most wbox voxels that a batched wave sums in LDS: inside the grid
// (sd <= nx, ny; d <= nz); none on a grid one voxel wide
struct BatchCube {
    int sd, d;
};
__host__ __device__ inline BatchCube batch_cube(int nx, int ny, int nz, int wbox)
{
    int sd = (int)cbrtf((float)wbox);
    while ((long)(sd + 1) * (sd + 1) * (sd + 1) <= wbox) ++sd;
    while (sd > 1 && (long)sd * sd * sd > wbox) --sd;
    sd = sd < nx ? sd : nx;
    sd = sd < ny ? sd : ny;
    // the two voxels of a word share a row; a grid one voxel wide has no such
    // pair (a carry would go past its column, and past its tally at the top)
    sd &= ~1;
    if (sd < 2) return BatchCube{0, 0};
    const int d = wbox / (sd * sd);
    return BatchCube{sd, d < nz ? d : nz};
}

// Many instances in one launch: a wave takes packets from one instance's
// queue until it drains, then moves on to the next instance (starting at its
// own index, so the waves spread over the instances); each instance keeps its
// own queue, tally and counters, and the instance's arguments stay uniform
// over the wave.  With wbox > 0 each wave owns an LDS slice of 16-bit
// fixed-point voxels (slots: the largest cube of the instances): for every instance it works on (with the box enabled,
// of either kind) it sums its
// visits to a cube under the top face on that instance's beam axis there,
// and adds the cube to the instance's tally when it moves on.  The waves of
// a block work on different instances, so the slices are per wave and only
// wave-level ordering is needed.
__global__ __launch_bounds__(256) void mc_batch_kernel(const McArgs* __restrict__ tab, int n, int wbox, int slots)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_slices[];
    // slots is a multiple of 8, so every slice starts on a 16-byte boundary
    uint16_t* box = reinterpret_cast<uint16_t*>(lds_slices) + (size_t)(threadIdx.x >> 6) * (size_t)slots;
    // per wave: counts of the current instance and its material table
    __shared__ unsigned long long wsums[4][TAM_CNT_N];
    __shared__ __attribute__((aligned(16))) MatEntry wtab[4][kBatchTab];
    static_assert(sizeof(wsums) + sizeof(wtab) == kBatchLds, "static LDS of a batched block");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    unsigned long long* sums = wsums[threadIdx.x >> 6];
    MatEntry* mtl = wtab[threadIdx.x >> 6];
    for (int k = 0; k < n; ++k) {
        const int i = (wave + k) % n;
        const McArgs a = tab[i];
        // an instance that the other waves have drained costs no box either
        if (a.npk == 0 || __hip_atomic_load(a.counters + TAM_CNT_N, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >=
                              a.npk)
            continue;
        BoxGeom g{};
        if (wbox > 0 && a.box_enable) {
            const BatchCube q = batch_cube(a.nx, a.ny, a.nz, wbox);
            const int sd = q.sd, d = q.d;
            g.n[0] = g.n[1] = sd;
            g.n[2] = d;
            g.o[0] = max(0, min((int)lroundf(a.cx / a.dx) - sd / 2, a.nx - sd));
            g.o[1] = max(0, min((int)lroundf(a.cy / a.dy) - sd / 2, a.ny - sd));
            g.o[2] = a.nz - d;
        }
        const int nb = g.n[0] * g.n[1] * g.n[2];
        const bool small = nb < 8;                         // no box worth its clearing
        const bool tabbed = a.mut_by_mat && a.nmat <= kBatchTab;
        if (lane < TAM_CNT_N) sums[lane] = 0ull;
        if (tabbed) stage_table(a, mtl, a.nmat, lane, 64);
        if (!small)
            for (int q = lane; q < nb; q += 64) box[q] = 0;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");   // the zeros land before any add
        __builtin_amdgcn_wave_barrier();
        if (small) transport<false, double, false>(a, nullptr, g, a.mtab, sums, 0u, 0u);
        else if (tabbed) transport<true, uint16_t, true>(a, box, g, mtl, sums, 0u, 0u);
        else transport<true, uint16_t, false>(a, box, g, a.mtab, sums, 0u, 0u);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");   // every lane's adds land before the flush
        __builtin_amdgcn_wave_barrier();
        add_counts(a, sums, lane);
        if (small) continue;
        const uint32_t nxy = (uint32_t)a.nx * (uint32_t)a.ny;
        for (int q = lane; q < nb; q += 64) {
            const double s = box_path(box[q], a);
            if (s != 0.0) {
                const int bx = q % g.n[0], by = (q / g.n[0]) % g.n[1], bz = q / (g.n[0] * g.n[1]);
                const uint32_t v = (uint32_t)(g.o[0] + bx) + (uint32_t)a.nx * (uint32_t)(g.o[1] + by) +
                                   nxy * (uint32_t)(g.o[2] + bz);
                unsafeAtomicAdd(&a.tally[v], s);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");   // the flush reads finish before the next zeros
        __builtin_amdgcn_wave_barrier();
    }
}

// Atomic-rate probe: each lane adds 1.0 to `per_lane` xorshift-chosen slots.
__global__ __launch_bounds__(256) void atomic_rate_kernel(double* t, uint32_t slots, uint32_t per_lane)
{
    uint32_t x = (blockIdx.x * 256u + threadIdx.x) * 2654435761u + 0x9E3779B9u;
    for (uint32_t i = 0; i < per_lane; ++i) {
        x ^= x << 13;
        x ^= x >> 17;
        x ^= x << 5;
        unsafeAtomicAdd(&t[x % slots], 1.0);
    }
}

}  // namespace

hipError_t launch_atomic_rate(double* t, long slots, long count, hipStream_t s)
{
    // 2048 blocks of 256 lanes; per_lane adds each
    const long lanes = 2048L * 256L;
    long per = count / lanes;
    if (per < 1) per = 1;
    if (slots < 1 || slots > 0xffffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(atomic_rate_kernel, dim3(2048), dim3(256), 0, s, t, (uint32_t)slots, (uint32_t)per);
    return hipGetLastError();
}

// The current device's CUs, and LDS per CU and per block (160 KiB each on MI355X)
McDevice mc_device()
{
    int dev = 0;
    McDevice d{0, 0, 0};
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&d.ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess || d.ncu <= 0) d.ncu = 256;
    if (hipDeviceGetAttribute(&d.lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess ||
        d.lds_cu <= 0)
        d.lds_cu = 64 * 1024;
    if (hipDeviceGetAttribute(&d.lds_blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        d.lds_blk <= 0)
        d.lds_blk = 64 * 1024;
    return d;
}

// 16-bit slots that a batched wave's cube may have: a quarter of its block's share
// of the CU's LDS, less 1 KiB for the kernel's own use, a multiple of 8
int mc_batch_slots(const McDevice& dev, int bpc)
{
    const long per_block = std::min((long)dev.lds_blk - kLdsOwn, (long)dev.lds_cu / bpc - kLdsOwn);
    return per_block > 0 ? (int)(per_block / 4 / 2) & ~7 : 0;
}

// The slots of a launch's largest cube, a multiple of 8: what the launch asks for,
// so that the counts and tables of a block (960 bytes) come in beside it.  LDS is
// given out in steps of 1280 bytes; with all of a third of a CU's LDS but 1 KiB asked for,
// 2 blocks a CU were resident instead of 3 (eight tissues of four materials
// 46.3 ms at 3 a CU, 42.2 so; of one 41.5, 40.9).
int mc_batch_cube(const McArgs* tab, int n, int wbox)
{
    long most = 0;
    for (int i = 0; i < n; ++i)
        if (wbox > 0 && tab[i].npk > 0 && tab[i].box_enable) {
            const BatchCube q = batch_cube(tab[i].nx, tab[i].ny, tab[i].nz, wbox);
            most = std::max(most, (long)q.sd * q.sd * q.d);
        }
    return (int)((most + 7) & ~7L);
}

extern "C" int tam_internal_batch_slots(const int32_t* edges, int n, int ncu, int lds_cu, int lds_blk, int bpc,
                                        int32_t* cube)
{
    std::vector<McArgs> tab((size_t)n);
    const int wbox = mc_batch_slots(McDevice{ncu, lds_cu, lds_blk}, bpc);
    for (int i = 0; i < n; ++i) {
        McArgs& a = tab[(size_t)i];
        a = McArgs{};
        a.npk = 1;
        a.box_enable = 1;
        a.nx = edges[3 * i]; a.ny = edges[3 * i + 1]; a.nz = edges[3 * i + 2];
        const BatchCube q = wbox > 0 ? batch_cube(a.nx, a.ny, a.nz, wbox) : BatchCube{0, 0};
        cube[2 * i] = q.sd;
        cube[2 * i + 1] = q.d;
    }
    return mc_batch_cube(tab.data(), n, wbox);
}

hipError_t launch_mc_batch(const McArgs* tab, const McArgs* dtab, int n, long total_npk, int blocks_per_cu,
                           hipStream_t s)
{
    if (n <= 0 || total_npk <= 0) return hipSuccess;
    const McDevice dev = mc_device();
    const int bpc = blocks_per_cu > 0 ? blocks_per_cu : 8;
    long blocks = (long)dev.ncu * bpc;
    const long need = (total_npk + 255) / 256;
    if (need < blocks) blocks = need;
    const int wbox = mc_batch_slots(dev, bpc), slots = mc_batch_cube(tab, n, wbox);
    const size_t lds = sizeof(uint16_t) * 4 * (size_t)slots;
    hipLaunchKernelGGL(mc_batch_kernel, dim3((unsigned)blocks), dim3(256), lds, s, dtab, n, wbox, slots);
    return hipGetLastError();
}

void mc_box_units(McArgs& a)
{
    a.box_scale = (float)std::ldexp(1.0 / ((double)a.dx + a.dy + a.dz), kBoxUnitBits);
    a.box_quantum = 1.0 / (double)a.box_scale;
}

// the most dynamic LDS that a box launch may ask for
long mc_lds_limit(long lds_blk) { return lds_blk - kCountLds; }

hipError_t mc_prepare(int dev)
{
    int lds_blk = 0;
    hipError_t e = hipDeviceGetAttribute(&lds_blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess || lds_blk <= 64 * 1024) return e;
    // allow the kernels all of a block's LDS but their static part (outside any
    // graph capture): a material table may take what the box leaves of it
    const int box_lds = (int)mc_lds_limit(lds_blk);
    const void* box_kernels[] = {
        (const void*)mc_box_kernel<256, uint16_t, false>, (const void*)mc_box_kernel<1024, uint16_t, false>,
        (const void*)mc_box_kernel<256, double, false>,   (const void*)mc_box_kernel<1024, double, false>,
        (const void*)mc_box_kernel<256, uint16_t, true>,  (const void*)mc_box_kernel<1024, uint16_t, true>,
        (const void*)mc_box_kernel<256, double, true>,    (const void*)mc_box_kernel<1024, double, true>};
    for (const void* k : box_kernels) {
        e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, box_lds);
        if (e != hipSuccess) return e;
    }
    return hipFuncSetAttribute((const void*)mc_batch_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               lds_blk - (int)kBatchLds);
}

// The launch of a transport run: box or not, how many blocks, and where the
// material table lies.
McPlan mc_plan(const McArgs& a, const McDevice& dev)
{
    McPlan p{};
    // blocks_per_cu 256-lane blocks per CU (autotuned): the most waves of a run
    const int shape = a.blocks_per_cu > 0 ? a.blocks_per_cu : 8;
    // A launch with fewer packets than a quarter of the shape's lanes (the reference's
    // own run: 125 000 packets per cycle of a few deposits each) goes without
    // the box: clearing and flushing the box would cost more than it saves.
    const bool few = (double)a.npk < 64.0 * (double)dev.ncu * shape;
    if (a.box_enable && !few) {
        // a multiple of 4 runs as bpc / 4 blocks of 1024 lanes: the same waves
        // per CU, one box per 16 waves
        const bool wide = shape % 4 == 0;
        p.lanes = wide ? 1024 : 256;
        p.per_cu = wide ? shape / 4 : shape;
        // A block's box costs a clearing and a device add per touched voxel,
        // and waves that share a SIMD slow each other's longest packets: 16
        // waves a CU (all of a smaller shape's), further ones where each has
        // 1024 packets (8 blocks of 256 lanes a CU at 100^3: 3e6 packets 12.7
        // ms on 256 blocks of 1024 lanes, 13.9 on 512; 1e7 39.3 on both).  In
        // waves, so that 256-lane blocks fill a CU too: 1e6 packets at 100^3,
        // shapes 2, 3, 6: 5.0, 5.6, 6.3 ms; with one block a CU of whatever size
        // 6.7, 6.8, 6.7.
        const int64_t all = (int64_t)dev.ncu * p.per_cu, wave_blocks = p.lanes / 64;
        const int64_t justified = (int64_t)(a.npk / (uint64_t)(wave_blocks * 1024));
        const int64_t least = (int64_t)dev.ncu * (16 / wave_blocks);
        p.blocks = a.full_grid ? all : std::min(all, std::max(least, justified));
        // LDS tally box: the shape's blocks of a CU share its LDS (160 KiB on
        // MI355X, also the most one block may take; a run of fewer blocks keeps
        // the shape's box, since the deposits that are rounded to its units are
        // part of the result), 1 KiB per block kept for the kernel's own use: with 16-bit sums 42^2 x 46 voxels at 1 block per CU
        // (1 or 4 blocks_per_cu), 34^2 x 34 at 2 (2 or 8), 28^2 x 34 at 3; with
        // FP64 27^3, 21^3, 18^2 x 20.  The cube sits on the beam axis (its x edge
        // even with 16-bit sums, so the two voxels of a word share a row).  Its z range is where
        // the last run's path was largest, or the top face (where most of the
        // path of a surface beam lies) before any run.  On the c1 skin cycles a
        // cube caught more deposits past the first cycle than flatter (d ~ s/2,
        // s/8) or taller (d ~ 2s) boxes of the same volume, and than a per-launch
        // choice among depths of 2-32 planes made from the last run's path.
        // The box holds 16-bit fixed-point sums (box_enable 1: four times the
        // voxels of FP64) or FP64 ones (box_enable 2).  Fixed-point unit: 2^-13 of
        // dx + dy + dz, so a deposit is rounded by at most ~1e-4 of a voxel-sized
        // path, and a slot wraps (one carry) every ~40 typical deposits.
        const bool fx = a.box_enable == 1;
        const long esz = fx ? 2 : 8;
        const long vox = std::min((long)dev.lds_blk - kLdsOwn, (long)dev.lds_cu / p.per_cu - kLdsOwn) / esz;
        p.sd = std::min((int)std::cbrt((double)vox), std::min(a.nx, a.ny));
        if (fx && p.sd > 1) p.sd &= ~1;
        p.d = p.sd > 0 ? (int)std::min<long>(a.nz, vox / ((long)p.sd * p.sd)) : 0;
        p.box = p.sd >= 4 && p.d >= 1;
        if (p.box) {
            const int64_t lds = (int64_t)esz * p.sd * p.sd * p.d;
            // the material table goes behind the box where that keeps the resident
            // blocks: LDS is given out in steps of lds_cu / 128
            p.tab_off = (int)((lds + 15) & ~(int64_t)15);
            const int64_t tab_lds = p.tab_off + (int64_t)sizeof(MatEntry) * a.nmat;
            const int64_t step = dev.lds_cu / 128;
            const bool tab = a.mut_by_mat && tab_lds + kCountLds <= lds + kLdsOwn &&
                             (tab_lds + kCountLds + step - 1) / step * step * p.per_cu <= dev.lds_cu;
            p.ntab = tab ? a.nmat : 0;
            p.lds = tab ? tab_lds : lds;
            return p;
        }
    }
    // A short run takes as long as its longest packet's chain of events,
    // and a wave's pass costs the same for 4 lanes as for 64: up to 8
    // waves a CU (2 per SIMD) share fewer than 64 packets each, down to
    // 4; past that every wave starts with a full set of lanes.  20 000
    // packets at 64^3: 1.35 ms, against 2.7 ms on full waves alone
    // (1.6 at 4 waves a CU, 1.35 at 16); 125 000 packets of a pure
    // absorber: 40 us, against 68 (44 at 16 waves a CU).  Past 16 waves a CU
    // each has 1024 packets, as with the box: 400 000 packets at shape 8 on a
    // 37x51x45 and a 100^3 cube and on the 200^3 skin 3.4, 4.8 and 2.8 ms,
    // against 4.1, 5.4 and 2.9 on a wave per 64 packets; of the pure absorber,
    // whose packets are then drawn, 0.15 against 0.11.
    p = McPlan{};
    p.lanes = 256;
    p.per_cu = shape;
    auto up = [](uint64_t n, uint64_t d) { return (int64_t)(n / d + (n % d != 0)); };
    const int64_t all = (int64_t)dev.ncu * shape;
    const int64_t waves = std::max({std::min(up(a.npk, 4), (int64_t)8 * dev.ncu),
                                    std::min(up(a.npk, 64), (int64_t)16 * dev.ncu), up(a.npk, 1024)});
    p.blocks = a.full_grid ? all : std::min(all, up((uint64_t)waves, 4));
    p.ntab = a.mut_by_mat && a.nmat <= kTabMax ? a.nmat : 0;
    p.lds = (int64_t)sizeof(MatEntry) * p.ntab;
    return p;
}

extern "C" void tam_internal_mc_plan(const int64_t* in, int64_t* out)
{
    McArgs a{};
    a.npk = (uint64_t)in[0];
    a.nx = (int)in[1]; a.ny = (int)in[2]; a.nz = (int)in[3];
    a.blocks_per_cu = (int)in[4]; a.box_enable = (int)in[5];
    a.nmat = (int)in[6]; a.mut_by_mat = (int)in[7]; a.full_grid = (int)in[8];
    const McPlan p = mc_plan(a, McDevice{(int)in[9], (int)in[10], (int)in[11]});
    const int64_t r[] = {p.box, p.lanes, p.per_cu, p.blocks, p.sd, p.d, p.ntab, p.tab_off, p.lds, mc_lds_limit(in[11])};
    std::copy(std::begin(r), std::end(r), out);
}

extern "C" int64_t tam_internal_mc_draws(int64_t npk, int64_t waves, int64_t* last)
{
    int64_t at = waves * std::min<int64_t>(64, (npk + waves - 1) / waves), n = 0;
    *last = 0;
    for (; at < npk; ++n) at += *last = draw_size((uint64_t)(npk - at), 0.5f / (float)waves);
    return n;
}

hipError_t launch_mc(const McArgs& a, hipStream_t s)
{
    const long nvox = (long)a.nx * a.ny * a.nz;
    // the run's counters, and the tally unless the run adds to it
    auto clear = [&] { return launch_clear(a.tally, a.clear_tally ? nvox : 0, a.counters, TAM_CNT_SLOTS, s); };
    if (a.npk == 0) return clear();
    const McPlan p = mc_plan(a, mc_device());
    McArgs b = a;
    mc_box_units(b);
    b.box_n[0] = b.box_n[1] = b.box_n[2] = 0;
    b.box_geom = nullptr;
    b.ntab = p.ntab;
    b.tab_off = p.tab_off;
    const dim3 grid((unsigned)p.blocks), block((unsigned)p.lanes);
    const size_t lds = (size_t)p.lds;
    if (p.box) {
        BoxPlace bp{};
        bp.sd = p.sd;
        bp.d = p.d;
        bp.ox = std::max(0, std::min((int)std::lround(a.cx / a.dx) - bp.sd / 2, a.nx - bp.sd));
        bp.oy = std::max(0, std::min((int)std::lround(a.cy / a.dy) - bp.sd / 2, a.ny - bp.sd));
        b.box_o[0] = bp.ox;
        b.box_o[1] = bp.oy;
        b.box_o[2] = a.nz - bp.d;
        b.box_n[0] = b.box_n[1] = bp.sd;
        b.box_n[2] = bp.d;
        if (a.box_psum && a.box_geom) {
            hipLaunchKernelGGL(box_plane_kernel, dim3((unsigned)a.nz), dim3(256), 0, s, a.tally, a.mut, a.nx, a.ny,
                               bp, a.box_psum);
            hipLaunchKernelGGL(box_window_kernel, dim3(1), dim3(256), 0, s, a.box_psum, a.nz, bp, a.box_geom);
            b.box_geom = a.box_geom;
        }
        const hipError_t ef = clear();
        if (ef != hipSuccess) return ef;
#define TAM_BOX(NT_, BT_)                                                                       \
    do {                                                                                        \
        if (p.ntab) hipLaunchKernelGGL((mc_box_kernel<NT_, BT_, true>), grid, block, lds, s, b); \
        else hipLaunchKernelGGL((mc_box_kernel<NT_, BT_, false>), grid, block, lds, s, b);       \
    } while (0)
        const bool wide = p.lanes == 1024;
        if (a.box_enable == 1) {
            if (wide) TAM_BOX(1024, uint16_t);
            else TAM_BOX(256, uint16_t);
        } else {
            if (wide) TAM_BOX(1024, double);
            else TAM_BOX(256, double);
        }
#undef TAM_BOX
    } else {
        const hipError_t ef = clear();
        if (ef != hipSuccess) return ef;
        if (p.ntab) hipLaunchKernelGGL((mc_kernel<true>), grid, block, lds, s, b);
        else hipLaunchKernelGGL((mc_kernel<false>), grid, block, lds, s, b);
    }
    return hipGetLastError();
}
