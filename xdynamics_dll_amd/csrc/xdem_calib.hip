// xdem_calib.hip -- FP64 forward runs of one scene with checkpoints, and their discrete
// adjoint with respect to the contact material (friction, restitution, modulus scale).
//
// Forward step (the reference's operations, xdem_calib.hpp):
//   k_cal_position  position and Euler-parameter update, cell hash (impl:54-72, 135-190)
//   cell sort       the stable sort of the launcher layer, on the run's stream
//   k_cal_contacts  sphere-sphere contacts over the 27 cells in the reference's order, then
//                   the walls in id order, rolling resistance and the velocity update; velocity
//                   and rate go to the other buffer of a pair (neighbours read the old ones);
//                   optionally records the step's contacts (the tape) for the reverse sweep.
// Reverse step (the same code on Dual<N>, each kernel's vector-Jacobian product from its local
// Jacobian):
//   k_cal_rev_tail      rolling resistance + velocity update of each sphere
//   k_cal_rev_contacts  every recorded contact of each sphere: cotangents of both spheres'
//                       positions, velocities and angular velocities (atomics for the
//                       neighbour), of the history entry it read, and of theta
//   k_cal_rev_head      angular velocity from (e, e_dot), then the position update
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "xdem_calib.h"
#include "xdem_calib.hpp"
#include "xdem_capi.h"
#include "xdem_contact.hpp"
#include "xdem_sort.hpp"

using namespace xdem;
using namespace xdem::calib;

namespace {

constexpr uint32_t kPlaneTag = 0x80000000u;
constexpr int kTape = XDEM_CALIB_TAPE;
constexpr int kCapMax = XDEM_CALIB_MAX_CAPACITY;
constexpr int kPlSlots = XDEM_MAX_P2PL_COUNT;
constexpr int kThreads = 128;

// One state of the run: what a step reads and writes, plus the step's recorded extras.
struct StateView {
    double *pos, *vel, *acc, *ep, *ev, *ea, *tmax, *rres;
    uint32_t *pp_count, *pp_id;
    double* pp_tsd;
    uint32_t *pl_count, *pl_id;
    double* pl_tsd;
};

struct CalArgs {
    uint32_t n, cap, nplane, ncell;
    double dt, h, gx, gy, gz;
    double wo[3], cs;
    uint32_t gsize[3];
    Law law;
    int flat_inertia;
    Material mat_pp;
    const Material* mat_pl;
    const xdem_plane_info* planes;
    const double* plane_dbi;
    double mu, rest, s;              // theta
    const double* mass;
    const double* inertia;
    StateView st;                    // current state (contact kernel: positions already updated)
    double* vel_out;
    double* ev_out;
    uint32_t *hash, *index;
    const uint32_t *sorted, *cstart, *cend;
    uint32_t* err;
};

// ------------------------------------------------------------------------- small helpers
__host__ __device__ inline V3<double> ld3d(const double* p) { return {p[0], p[1], p[2]}; }
__host__ __device__ inline V4<double> ld4d(const double* p) { return {p[0], p[1], p[2], p[3]}; }

__device__ inline void st4d(double* p, V4<double> v) { p[0] = v.x; p[1] = v.y; p[2] = v.z; p[3] = v.w; }

__device__ inline void grid_of(const CalArgs& A, V3<double> x, int g[3])
{
    g[0] = (int)floor((x.x - A.wo[0]) / A.cs);
    g[1] = (int)floor((x.y - A.wo[1]) / A.cs);
    g[2] = (int)floor((x.z - A.wo[2]) / A.cs);
}

__device__ inline uint32_t hash_of(const CalArgs& A, int gx, int gy, int gz)
{
    const uint32_t x = (uint32_t)gx & (A.gsize[0] - 1);
    const uint32_t y = (uint32_t)gy & (A.gsize[1] - 1);
    const uint32_t z = (uint32_t)gz & (A.gsize[2] - 1);
    return (z * A.gsize[1]) * A.gsize[0] + y * A.gsize[0] + x;
}

template <int N> __host__ __device__ inline V3<Dual<N>> seed3(V3<double> v, int k0)
{
    return {Dual<N>::input(v.x, k0), Dual<N>::input(v.y, k0 + 1), Dual<N>::input(v.z, k0 + 2)};
}
template <int N> __host__ __device__ inline V4<Dual<N>> seed4(V4<double> v, int k0)
{
    return {Dual<N>::input(v.x, k0), Dual<N>::input(v.y, k0 + 1), Dual<N>::input(v.z, k0 + 2),
            Dual<N>::input(v.w, k0 + 3)};
}

// cotangent accumulation: out[k] += bar * d/dk of the dual y
template <int N> __host__ __device__ inline void vjp_add(double (&out)[N], const Dual<N>& y, double bar)
{
    if (bar == 0.0) return;
    for (int k = 0; k < N; k++) out[k] += bar * y.d[k];
}
template <int N> __host__ __device__ inline void vjp_add3(double (&out)[N], const V3<Dual<N>>& y, V3<double> bar)
{
    vjp_add(out, y.x, bar.x);
    vjp_add(out, y.y, bar.y);
    vjp_add(out, y.z, bar.z);
}

// ----------------------------------------------------------------------------- forward
// The recorded step k: the state the contact kernel read (positions and Euler parameters after
// the position update; velocities, rates and accelerations as before the step), the Euler
// parameters before the position update, the history before the step, the tape and the contact
// sums F, M, T, R.
struct StepRec {
    double *pos1, *ep0, *ep1, *vel, *ev, *ea, *pp_tsd, *pl_tsd, *sums;
    uint32_t* tape_code;
    uint16_t* tape_slot;
    uint8_t* tape_n;
};

__device__ inline void copy_flat(double* to, const double* from, size_t len)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < len; t += stride) to[t] = from[t];
}

// The first n threads each move a sphere. With a record, all threads copy what the contact kernel
// changes later (15 copies between the kernels of a recorded step otherwise) and the owners add
// the positions and Euler parameters.
template <bool RECORD> __global__ __launch_bounds__(kThreads) void k_cal_position(CalArgs A, StepRec r)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const StateView& s = A.st;
    if (RECORD) {
        const size_t N = A.n;
        copy_flat(r.vel, s.vel, 3 * N);
        copy_flat(r.ev, s.ev, 4 * N);
        copy_flat(r.ea, s.ea, 4 * N);
        copy_flat(r.pp_tsd, s.pp_tsd, 2 * A.cap * N);
        copy_flat(r.pl_tsd, s.pl_tsd, 2 * kPlSlots * N);
    }
    if (i >= A.n) return;
    const size_t i4 = 4 * (size_t)i;
    const V4<double> p4 = ld4d(s.pos + i4);
    V3<double> p = {p4.x, p4.y, p4.z};
    V4<double> e = ld4d(s.ep + i4);
    if (RECORD) st4d(r.ep0 + i4, e);
    position_update<double>(A.dt, A.h, p, e, ld3d(s.vel + 3 * (size_t)i), ld4d(s.ev + i4), ld3d(s.acc + 3 * (size_t)i),
                            ld4d(s.ea + i4));
    const V4<double> p1 = {p.x, p.y, p.z, p4.w};
    st4d(s.pos + i4, p1);
    st4d(s.ep + i4, e);
    if (RECORD) {
        st4d(r.pos1 + i4, p1);
        st4d(r.ep1 + i4, e);
    }
    int g[3];
    grid_of(A, p, g);
    A.hash[i] = hash_of(A, g[0], g[1], g[2]);
    A.index[i] = i;
}

__device__ inline void tape_put(const StepRec& r, uint32_t i, uint32_t at, uint32_t code, int slot_in, int slot_out,
                                uint32_t& err)
{
    if (at >= (uint32_t)kTape) {
        err |= XDEM_ERR_P2P_OVERFLOW;
        return;
    }
    r.tape_code[(size_t)i * kTape + at] = code;
    r.tape_slot[(size_t)i * kTape + at] = (uint16_t)((slot_in + 1) | ((slot_out + 1) << 8));
}

// One overlapping pair (pair_side's operations) on its own, for sphere_pair_add: returns whether
// it sets the tangential force. Set: out = Fn + Ft, its moment, the rolling resistance, Ft. Not
// set: out = Fn, the lever arm, the rolling resistance.
__device__ inline bool pair_eval(const Law& L, const PairK<double>& c, double rfric, V3<double> xi, double ir,
                                 V3<double> xj, double jr, V3<double> vi, V3<double> vj, V3<double> wi, V3<double> wj,
                                 double& sd0, double& sd1, double out[10])
{
    const V3<double> rp = xj - xi;
    const double dist = length(rp);
    const double cdist = (ir + jr) - dist;
    const V3<double> unit = rp / dist;
    const V3<double> cpt = xi + ir * unit;
    const V3<double> dcpr = cpt - xi;
    const V3<double> dcpr_j = cpt - xj;
    const V3<double> rv = (vj + cross(wj, dcpr_j)) - (vi + cross(wi, dcpr));
    V3<double> Fn, Ft = {0.0, 0.0, 0.0};
    const bool set = calib::force_law(L.model, L.gpu_law, L.dt, c, cdist, sd0, sd1, rv, unit, Ft, Fn);
    const V3<double> f = set ? Fn + Ft : Fn;
    const V3<double> m = set ? cross(dcpr, f) : dcpr;
    const double Rij = jr ? ir * jr / (ir + jr) : ir;
    out[0] = f.x; out[1] = f.y; out[2] = f.z;
    out[3] = m.x; out[4] = m.y; out[5] = m.z;
    out[6] = Rij * rfric * length(Fn);
    out[7] = Ft.x; out[8] = Ft.y; out[9] = Ft.z;
    return set;
}

// The rest of sphere i's step after its sphere contacts (sums F, M = T and Rp, n_seen of them):
// the walls in id order (impl:950-1080, one launch per wall), rolling resistance (impl:2420-2454),
// the velocity update.
template <bool RECORD>
__device__ inline void own_tail(const CalArgs& A, const StepRec& r, uint32_t i, V3<double> Fp, V3<double> Mp, double Rp,
                                uint32_t n_seen, const Theta<double>& th, uint32_t& err)
{
    const StateView& s = A.st;
    const V4<double> ip = ld4d(s.pos + 4 * (size_t)i);
    const V3<double> xi = {ip.x, ip.y, ip.z};
    const double ir = ip.w, im = A.mass[i];
    const V3<double> vi = ld3d(s.vel + 3 * (size_t)i);
    const V4<double> ei = ld4d(s.ep + 4 * (size_t)i), di = ld4d(s.ev + 4 * (size_t)i);
    const V3<double> wi = ang_vel(ei, di);
    if (n_seen > A.cap) err |= XDEM_ERR_P2P_OVERFLOW;
    s.pp_count[i] = min(n_seen, A.cap);
    uint32_t nt = min(n_seen, (uint32_t)kTape);
    V3<double> F = V3<double>{0.0, 0.0, 0.0} + Fp;
    V3<double> M = V3<double>{0.0, 0.0, 0.0} + Mp;
    V3<double> Tm = ld3d(s.tmax + 3 * (size_t)i) + Mp;
    double R = s.rres[i] + Rp;

    // ---- walls
    for (uint32_t w = 0; w < A.nplane; w++) {
        const xdem_plane_info& pl = A.planes[w];
        const size_t lb = (size_t)i * kPlSlots;
        uint32_t l_id[kPlSlots];
        double l_sd[2 * kPlSlots];
        for (int q = 0; q < kPlSlots; q++) {
            l_id[q] = s.pl_id[lb + q];
            l_sd[2 * q] = s.pl_tsd[2 * (lb + q)];
            l_sd[2 * q + 1] = s.pl_tsd[2 * (lb + q) + 1];
        }
        const uint32_t kid = pl.id;
        uint32_t nn = kid ? s.pl_count[i] : 0u;
        if (nn > (uint32_t)kPlSlots) nn = kPlSlots;
        Sums<double> ps = zero_sums<double>();
        const V3<double> dp = xi - V3<double>{pl.xw.x, pl.xw.y, pl.xw.z};
        const V3<double> wp = {dot(dp, V3<double>{pl.u1.x, pl.u1.y, pl.u1.z}), dot(dp, V3<double>{pl.u2.x, pl.u2.y, pl.u2.z}),
                               dot(dp, V3<double>{pl.uw.x, pl.uw.y, pl.uw.z})};
        V3<double> u0 = {0.0, 0.0, 0.0};
        const double cd = plane_detect<double>(pl, xi, wp, u0, ir);
        if (cd > 0) {
            double sd0 = 0.0, sd1 = 0.0;
            int slot_in = -1;
            for (int q = 0; q < kPlSlots; q++)
                if (l_id[q] == kid) {
                    sd0 = l_sd[2 * q];
                    sd1 = l_sd[2 * q + 1];
                    slot_in = q;
                    break;
                }
            const PairK<double> c = pair_k<double>(A.law.model, A.mat_pl[w], th, ir, 0.0, im, 0.0);
            plane_side<double>(A.law, c, A.mat_pl[w].rfric, pl, A.plane_dbi + 15 * (size_t)w, xi, ir, vi, wi, sd0, sd1,
                               ps);
            int slot_out = -1;
            if (nn < (uint32_t)kPlSlots) {
                s.pl_tsd[2 * (lb + nn)] = sd0;
                s.pl_tsd[2 * (lb + nn) + 1] = sd1;
                s.pl_id[lb + nn] = kid;
                slot_out = (int)nn;
                nn++;
            } else {
                err |= XDEM_ERR_PLANE_OVERFLOW;
            }
            if (RECORD) {
                tape_put(r, i, nt, kPlaneTag | w, slot_in, slot_out, err);
                nt = min(nt + 1u, (uint32_t)kTape);
            }
        }
        s.pl_count[i] = nn;
        F = F + ps.F;
        M = M + ps.M;
        Tm = Tm + ps.T;
        R = R + ps.R;
    }
    if (RECORD) {
        r.tape_n[i] = (uint8_t)nt;
        const double o[10] = {F.x, F.y, F.z, M.x, M.y, M.z, Tm.x, Tm.y, Tm.z, R};
        for (int q = 0; q < 10; q++) r.sums[10 * (size_t)i + q] = o[q];
    }

    // ---- rolling resistance, then the velocity update
    if (R != 0.0) {
        const double J = A.flat_inertia ? A.inertia[i] : A.inertia[3 * (size_t)i];
        rolling<double>(A.dt, J, wi, Tm, R, M);
        Tm = {0.0, 0.0, 0.0};
        R = 0.0;
    }
    s.tmax[3 * (size_t)i] = Tm.x;
    s.tmax[3 * (size_t)i + 1] = Tm.y;
    s.tmax[3 * (size_t)i + 2] = Tm.z;
    s.rres[i] = R;
    V3<double> v = vi, acc = ld3d(s.acc + 3 * (size_t)i);
    V4<double> ev = di, ea = ld4d(s.ea + 4 * (size_t)i);
    velocity_update<double>(A.dt, V3<double>{A.gx, A.gy, A.gz}, im, ld3d(A.inertia + 3 * (size_t)i), ei, F, M, v, acc,
                            ev, ea);
    A.vel_out[3 * (size_t)i] = v.x;
    A.vel_out[3 * (size_t)i + 1] = v.y;
    A.vel_out[3 * (size_t)i + 2] = v.z;
    A.ev_out[4 * (size_t)i] = ev.x;
    A.ev_out[4 * (size_t)i + 1] = ev.y;
    A.ev_out[4 * (size_t)i + 2] = ev.z;
    A.ev_out[4 * (size_t)i + 3] = ev.w;
    s.acc[3 * (size_t)i] = acc.x;
    s.acc[3 * (size_t)i + 1] = acc.y;
    s.acc[3 * (size_t)i + 2] = acc.z;
    s.ea[4 * (size_t)i] = ea.x;
    s.ea[4 * (size_t)i + 1] = ea.y;
    s.ea[4 * (size_t)i + 2] = ea.z;
    s.ea[4 * (size_t)i + 3] = ea.w;
    if (!(isfinite(acc.x) && isfinite(acc.y) && isfinite(acc.z))) err |= XDEM_ERR_NONFINITE;
}

constexpr uint32_t kWaveMax = 16;   // spheres of a wave of k_cal_contacts
constexpr uint32_t kWaves = 2;      // waves of its blocks

// Spheres to a wave: as few as put all on two waves per SIMD (of 1,024) in one round, an even
// number from 2 to kWaveMax.
inline uint32_t wave_spheres(uint32_t n) { return std::min(kWaveMax, std::max(2u, (n + 2047u) / 2048u + 1u) & ~1u); }

// What the lanes of a wave hand each other.
struct WaveStage {
    double own[11][kWaveMax];            // position and radius, velocity, angular velocity, mass
    double h[kWaveMax][2 * kCapMax];     // the history before the step
    uint32_t id[kWaveMax][kCapMax];
    uint32_t old_count[kWaveMax];
    uint32_t queue_k[128], queue_s[128]; // overlapping pairs: neighbour, owner | rank << 8
    double v[10][64];                    // evaluated pairs
    unsigned long long pairs[kWaveMax];  // per owner: its pairs among the 64
};

// The overlapping spheres of a half wave's sphere, 32 candidates at a time in the reference's
// order: the 27 cells, x fastest, each by position in the sorted list. Lane c < 27 holds cell c.
struct Neighbours {
    uint32_t start, count, incl, total;

    __device__ __forceinline__ void open(const CalArgs& A, bool valid, V3<double> x)
    {
        const uint32_t c = threadIdx.x & 31u;
        start = 0u;
        count = 0u;
        if (valid && c < 27u) {
            int g[3];
            grid_of(A, x, g);
            const uint32_t h = hash_of(A, g[0] + (int)(c % 3u) - 1, g[1] + (int)(c / 3u % 3u) - 1, g[2] + (int)(c / 9u) - 1);
            start = A.cstart[h];
            const uint32_t end = A.cend[h];
            if (start != 0xffffffffu && end > start) count = end - start;
        }
        incl = count;
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) {
            const uint32_t t = __shfl_up(incl, off, 32);
            if ((int)c >= off) incl += t;
        }
        total = __shfl(incl, 31, 32);
    }
    // position in the sorted list of candidate x < total
    __device__ __forceinline__ uint32_t entry(uint32_t x) const
    {
        uint32_t L = 0;   // the cells that end at or before x
#pragma unroll
        for (uint32_t w = 16; w; w >>= 1) {
            const uint32_t e = __shfl(incl, (int)(L + w - 1u), 32);
            if (e <= x) L += w;
        }
        const uint32_t first = __shfl(incl - count, (int)L, 32);
        return __shfl(start, (int)L, 32) + (x - first);
    }
};

// Sphere-sphere contacts (impl:613-733): a wave takes G spheres, one per owner lane, and walks the
// cells of two at a time, a candidate a lane. Overlapping pairs go to a queue, which is evaluated
// 64 at a time; the owners add their pairs' results in visiting order. Then the owners take the
// walls, rolling resistance and the velocity update. Bound by dependent loads (cell, sorted
// index, position, the pair's state) and by the chain of square roots and divisions of a pair:
// 5,000 spheres 53 -> 19 us against a thread per sphere with its slots in scratch.
template <bool RECORD>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void k_cal_contacts(CalArgs A, StepRec r, uint32_t G)
{
    __shared__ WaveStage stage[kWaves];
    const uint32_t lane = threadIdx.x & 63u, half = lane >> 5, c = lane & 31u;
    WaveStage& st = stage[threadIdx.x >> 6];
    const uint32_t base = (blockIdx.x * kWaves + (threadIdx.x >> 6)) * G;
    if (base >= A.n) return;
    const uint32_t n_own = min(G, A.n - base);
    const StateView& s = A.st;
    const Theta<double> th = {A.mu, A.rest, A.s};
    const uint32_t cap = A.cap;
    uint32_t err = 0;
    if (lane < n_own) {
        const size_t i = base + lane;
        const V4<double> p = ld4d(s.pos + 4 * i);
        const V3<double> v = ld3d(s.vel + 3 * i);
        const V3<double> w = ang_vel(ld4d(s.ep + 4 * i), ld4d(s.ev + 4 * i));
        st.own[0][lane] = p.x; st.own[1][lane] = p.y; st.own[2][lane] = p.z; st.own[3][lane] = p.w;
        st.own[4][lane] = v.x; st.own[5][lane] = v.y; st.own[6][lane] = v.z;
        st.own[7][lane] = w.x; st.own[8][lane] = w.y; st.own[9][lane] = w.z;
        st.own[10][lane] = A.mass[i];
        st.old_count[lane] = min(s.pp_count[i], cap);
    }
    for (uint32_t q = lane; q < n_own * cap; q += 64u) {
        const size_t at = (size_t)base * cap + q;
        st.id[q / cap][q % cap] = s.pp_id[at];
        st.h[q / cap][2u * (q % cap)] = s.pp_tsd[2 * at];
        st.h[q / cap][2u * (q % cap) + 1u] = s.pp_tsd[2 * at + 1];
    }
    wave_lds_sync();

    // ---- sphere-sphere
    const MatK<double> mk = mat_k<double>(A.mat_pp, th);
    V3<double> F = {0.0, 0.0, 0.0}, M = {0.0, 0.0, 0.0}, Ft = {0.0, 0.0, 0.0};
    double R = 0.0;
    uint32_t queued = 0, n_seen = 0;
    for (uint32_t o0 = 0; o0 < n_own; o0 += 2u) {
        const uint32_t o = o0 + half;
        const bool valid = o < n_own;
        const uint32_t os = valid ? o : 0u;
        const V3<double> xi = {st.own[0][os], st.own[1][os], st.own[2][os]};
        const double ir = st.own[3][os];
        Neighbours near;
        near.open(A, valid, xi);
        const uint32_t longest = max(__shfl(near.total, 0, 64), __shfl(near.total, 32, 64));
        uint32_t rank0 = 0;   // the half's sphere: its overlapping candidates so far
        for (uint32_t r0 = 0;; r0 += 32u) {
            if (r0 < longest) {
                const uint32_t x = r0 + c, at = near.entry(x);
                const uint32_t k = x < near.total ? A.sorted[at] : A.n;
                bool hit = false;
                if (k != base + o && k < A.n) {
                    const V4<double> jp = ld4d(s.pos + 4 * (size_t)k);
                    hit = (ir + jp.w) - length(V3<double>{jp.x, jp.y, jp.z} - xi) > 0;
                }
                const unsigned long long all = __ballot(hit);
                const uint32_t mine = (uint32_t)(all >> (32u * half));
                if (hit) {
                    const uint32_t q = queued + (uint32_t)__popcll(all & ((1ull << lane) - 1ull));
                    st.queue_k[q] = k;
                    st.queue_s[q] = o | (rank0 + (uint32_t)__popc(mine & ((1u << c) - 1u))) << 8;
                }
                rank0 += (uint32_t)__popc(mine);
                queued += (uint32_t)__popcll(all);
            }
            const bool walked = r0 + 32u >= longest, last = walked && o0 + 2u >= n_own;
            while (queued >= 64u || (last && queued)) {
                const uint32_t m = min(queued, 64u);
                if (lane < kWaveMax) st.pairs[lane] = 0ull;
                wave_lds_sync();
                bool set = false;
                if (lane < m) {
                    const uint32_t k = st.queue_k[lane], qs = st.queue_s[lane], L = qs & 255u, rank = qs >> 8;
                    const V3<double> pi = {st.own[0][L], st.own[1][L], st.own[2][L]};
                    const double pr = st.own[3][L];
                    double sd0 = 0.0, sd1 = 0.0;
                    int slot_in = -1;
                    const uint32_t oc = st.old_count[L];
                    for (uint32_t q = 0; q < oc; q++)
                        if (st.id[L][q] == k) { slot_in = (int)q; break; }
                    if (slot_in >= 0) { sd0 = st.h[L][2 * slot_in]; sd1 = st.h[L][2 * slot_in + 1]; }
                    const V4<double> jp = ld4d(s.pos + 4 * (size_t)k);
                    const V3<double> wj = ang_vel(ld4d(s.ep + 4 * (size_t)k), ld4d(s.ev + 4 * (size_t)k));
                    const PairK<double> pk = pair_k<double>(A.law.model, A.mat_pp, mk, th, pr, jp.w, st.own[10][L], A.mass[k]);
                    double v[10];
                    set = pair_eval(A.law, pk, A.mat_pp.rfric, pi, pr, V3<double>{jp.x, jp.y, jp.z}, jp.w,
                                    V3<double>{st.own[4][L], st.own[5][L], st.own[6][L]}, ld3d(s.vel + 3 * (size_t)k),
                                    V3<double>{st.own[7][L], st.own[8][L], st.own[9][L]}, wj, sd0, sd1, v);
                    if (rank < cap) {
                        const size_t q = (size_t)(base + L) * cap + rank;
                        s.pp_id[q] = k;
                        s.pp_tsd[2 * q] = sd0;
                        s.pp_tsd[2 * q + 1] = sd1;
                    }
                    if (RECORD) tape_put(r, base + L, rank, k, slot_in, rank < cap ? (int)rank : -1, err);
#pragma unroll
                    for (int q = 0; q < 10; q++) st.v[q][lane] = v[q];
                    atomicOr(&st.pairs[L], 1ull << lane);
                }
                const unsigned long long sets = __ballot(set);
                wave_lds_sync();
                if (lane < n_own) {
                    // in visiting order; Ft: the last tangential force set, for a pair without one
                    // of its own
                    for (unsigned long long b = st.pairs[lane]; b; b &= b - 1ull) {
                        const uint32_t q = (uint32_t)__ffsll((long long)b) - 1u;
                        n_seen++;
                        double v[7];
#pragma unroll
                        for (int z = 0; z < 7; z++) v[z] = st.v[z][q];
                        const bool own_ft = (sets >> q) & 1ull;
                        PairSums acc = {F, M, R};
                        sphere_pair_add<double>(v, own_ft, Ft, acc);
                        F = acc.F; M = acc.M; R = acc.R;
                        if (A.law.stale_ft && own_ft) Ft = {st.v[7][q], st.v[8][q], st.v[9][q]};
                    }
                }
                // the rest of the queue moves to its front
                const uint32_t left = queued - m;
                uint32_t k = 0, qs = 0;
                if (lane < left) { k = st.queue_k[64u + lane]; qs = st.queue_s[64u + lane]; }
                wave_lds_sync();
                if (lane < left) { st.queue_k[lane] = k; st.queue_s[lane] = qs; }
                queued = left;
                wave_lds_sync();
            }
            if (walked) break;
        }
    }
    if (lane < n_own) own_tail<RECORD>(A, r, base + lane, F, M, R, n_seen, th, err);
    if (err) atomicOr(A.err, err);
}

// ----------------------------------------------------------------------------- reverse

// Cotangents of a state (the reverse sweep's lambda): positions 3 per sphere.
struct Lam {
    double *pos, *vel, *acc, *ep, *ev, *ea, *pp_tsd, *pl_tsd;
};

struct RevArgs {
    CalArgs A;          // sizes, law, materials, theta, mass, inertia
    StepRec r;
    Lam la;             // after the step (read)
    Lam lb;             // before the step (written)
    double* le1;        // [4n] cotangent of e' from the tail and the angular velocity
    double* lom;        // [3n] cotangent of the angular velocity w(e', e_dot)
    double* lpos1;      // [3n] cotangent of the updated positions from the contacts
    double* bar;        // [10n] cotangents of F (3), contact moment (3), Tm (3), Tr (1)
    double* gtheta;     // [3]
};

// A reverse kernel gives each lane one input direction of a sphere's Jacobian: Dual<1> values
// whose derivative is taken with respect to input `dir` (every lane of the sphere repeats the
// values). A thread per sphere on Dual<15> and Dual<23> kept hundreds of registers' worth of
// derivatives in scratch memory on a few waves: for 5,000 spheres k_cal_rev_tail 292 -> 11.7 us,
// k_cal_rev_contacts 91 -> 12.4 us.
typedef Dual<1> D1;

__device__ inline D1 in1(double x, int k, int dir)
{
    D1 r(x);
    r.d[0] = k == dir ? 1.0 : 0.0;
    return r;
}
__device__ inline V3<D1> in3(V3<double> v, int k0, int dir) { return {in1(v.x, k0, dir), in1(v.y, k0 + 1, dir), in1(v.z, k0 + 2, dir)}; }
__device__ inline V4<D1> in4(V4<double> v, int k0, int dir)
{
    return {in1(v.x, k0, dir), in1(v.y, k0 + 1, dir), in1(v.z, k0 + 2, dir), in1(v.w, k0 + 3, dir)};
}

// Rolling resistance and the velocity update of sphere i. The translational part and the
// rate update are linear and taken by hand; the Euler parameter accelerations (rolling
// resistance, A(e)^T M, calculate_uceom) are differentiated with respect to e' (0-3), e_dot
// (4-7), the contact moment (8-10), Tm (11-13) and Tr (14), one direction a lane, 16 lanes a
// sphere. The contact sums are the recorded ones.
constexpr uint32_t kTailLanes = 16;

__global__ __launch_bounds__(256) void k_cal_rev_tail(RevArgs R)
{
    const CalArgs& A = R.A;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = t / kTailLanes;
    const int dir = (int)(t % kTailLanes);
    if (i >= A.n) return;
    const StepRec& r = R.r;
    const Lam &la = R.la, &lb = R.lb;
    const double* sum = r.sums + 10 * (size_t)i;
    const double hdt = 0.5 * A.dt, inv_m = 1.0 / A.mass[i];
    // v' = (v + hdt acc) + hdt a, acc' = a = (F + m g) / m; ev' = (ev + hdt ea) + hdt mea, ea' = mea
    const V4<double> lev = ld4d(la.ev + 4 * (size_t)i), lea = ld4d(la.ea + 4 * (size_t)i);
    const V4<D1> e1 = in4(ld4d(r.ep1 + 4 * (size_t)i), 0, dir);
    const V4<D1> ev = in4(ld4d(r.ev + 4 * (size_t)i), 4, dir);
    V3<D1> M = in3(ld3d(sum + 3), 8, dir);
    const V3<D1> Tm = in3(ld3d(sum + 6), 11, dir);
    const D1 Tr = in1(sum[9], 14, dir);
    if (Tr.v != 0.0) {
        const double J = A.flat_inertia ? A.inertia[i] : A.inertia[3 * (size_t)i];
        rolling<D1>(A.dt, J, ang_vel(e1, ev), Tm, Tr, M);
    }
    const V4<D1> mea = uceom<D1>(ld3d(A.inertia + 3 * (size_t)i), e1, ev, to_local(M, e1));
    double g[1] = {0.0};
    vjp_add(g, mea.x, hdt * lev.x + lea.x);
    vjp_add(g, mea.y, hdt * lev.y + lea.y);
    vjp_add(g, mea.z, hdt * lev.z + lea.z);
    vjp_add(g, mea.w, hdt * lev.w + lea.w);
    const size_t i3 = 3 * (size_t)i, i4 = 4 * (size_t)i, ib = 10 * (size_t)i;
    if (dir < 4) {
        R.le1[i4 + dir] = g[0];
    } else if (dir < 8) {
        const double l = la.ev[i4 + dir - 4];
        lb.ev[i4 + dir - 4] = l + g[0];
        lb.ea[i4 + dir - 4] = hdt * l;
    } else if (dir < 11) {
        const int q = dir - 8;
        const double l = la.vel[i3 + q];
        lb.vel[i3 + q] = l;
        lb.acc[i3 + q] = hdt * l;
        R.bar[ib + q] = inv_m * (hdt * l + la.acc[i3 + q]);
        R.bar[ib + 3 + q] = g[0];
    } else if (dir < 14) {
        const int q = dir - 11;
        R.bar[ib + 6 + q] = g[0];
        R.lom[i3 + q] = 0.0;
        R.lpos1[i3 + q] = 0.0;
    } else if (dir == 14) {
        R.bar[ib + 9] = g[0];
    }
}

// The contacts of a sphere, in the forward's order, 32 lanes a sphere. A sphere-sphere contact
// is differentiated with respect to x_i (directions 0-2), x_j (3-5), v_i (6-8), v_j (9-11), w_i
// (12-14), w_j (15-17), the history entry read (18-19) and theta (20-22); a wall contact with
// respect to the same without the j ones; the previous pair's tangential force enters as a
// constant. Lane e also keeps the cotangent of history value e of the sphere's pair slots (at
// most 32) and, below 6, of its wall slots: slots that the step did not write pass theirs on.
constexpr int kPairN = 23;
constexpr uint32_t kContactLanes = 32;
static_assert(2 * XDEM_CALIB_MAX_CAPACITY <= kContactLanes, "a lane for every history value");

__global__ __launch_bounds__(256) void k_cal_rev_contacts(RevArgs R)
{
    const CalArgs& A = R.A;
    const StepRec& r = R.r;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = t / kContactLanes;
    const int dir = (int)(t % kContactLanes);
    double gth = 0.0;   // lanes 20-22: cotangent of theta
    if (i < A.n) {
        const V4<double> ip = ld4d(r.pos1 + 4 * (size_t)i);
        const V3<double> xi = {ip.x, ip.y, ip.z};
        const double ir = ip.w, im = A.mass[i];
        const V3<double> vi = ld3d(r.vel + 3 * (size_t)i);
        const V3<double> wi = ang_vel(ld4d(r.ep1 + 4 * (size_t)i), ld4d(r.ev + 4 * (size_t)i));
        const double* bar = R.bar + 10 * (size_t)i;
        const V3<double> bF = {bar[0], bar[1], bar[2]}, bM = {bar[3], bar[4], bar[5]}, bT = {bar[6], bar[7], bar[8]};
        const double bR = bar[9];
        const uint32_t nt = r.tape_n[i];
        const size_t sb = (size_t)i * A.cap, lb = (size_t)i * kPlSlots;
        const Theta<D1> th = {in1(A.mu, 20, dir), in1(A.rest, 21, dir), in1(A.s, 22, dir)};
        V3<double> Ft = {0.0, 0.0, 0.0};   // the previous pair's tangential force (values)
        double own = 0.0;                  // cotangent of x_i, v_i or w_i (lanes 0-2, 6-8, 12-14)
        double pp = 0.0, pl = 0.0;         // of this lane's history values before the step
        uint32_t written_pp = 0u, written_pl = 0u;   // slots this step wrote (bit masks)
        for (uint32_t m = 0; m < nt; m++) {
            const uint32_t code = r.tape_code[(size_t)i * kTape + m];
            const uint16_t sl = r.tape_slot[(size_t)i * kTape + m];
            const int slot_in = (int)(sl & 0xffu) - 1, slot_out = (int)(sl >> 8) - 1;
            const bool wall = (code & kPlaneTag) != 0u;
            const double* tsd = wall ? r.pl_tsd + 2 * lb : r.pp_tsd + 2 * sb;
            const double* lam = wall ? R.la.pl_tsd + 2 * lb : R.la.pp_tsd + 2 * sb;
            D1 s0 = in1(slot_in >= 0 ? tsd[2 * slot_in] : 0.0, 18, dir);
            D1 s1 = in1(slot_in >= 0 ? tsd[2 * slot_in + 1] : 0.0, 19, dir);
            // cotangents of this contact's new history entry
            const double bs0 = slot_out >= 0 ? lam[2 * slot_out] : 0.0;
            const double bs1 = slot_out >= 0 ? lam[2 * slot_out + 1] : 0.0;
            Sums<D1> acc = zero_sums<D1>();
            uint32_t k = i;
            if (!wall) {
                if (slot_out >= 0) written_pp |= 1u << slot_out;
                k = code;
                const V4<double> jp = ld4d(r.pos1 + 4 * (size_t)k);
                const V3<double> vj = ld3d(r.vel + 3 * (size_t)k);
                const V3<double> wj = ang_vel(ld4d(r.ep1 + 4 * (size_t)k), ld4d(r.ev + 4 * (size_t)k));
                const PairK<D1> c = pair_k<D1>(A.law.model, A.mat_pp, th, ir, jp.w, im, A.mass[k]);
                V3<D1> FtD = {D1(Ft.x), D1(Ft.y), D1(Ft.z)};
                pair_side<D1>(A.law, c, A.mat_pp.rfric, in3(xi, 0, dir), ir, in3(V3<double>{jp.x, jp.y, jp.z}, 3, dir), jp.w,
                              in3(vi, 6, dir), in3(vj, 9, dir), in3(wi, 12, dir), in3(wj, 15, dir), s0, s1, FtD, acc);
                Ft = {FtD.x.v, FtD.y.v, FtD.z.v};
            } else {
                if (slot_out >= 0) written_pl |= 1u << slot_out;
                const uint32_t w = code & ~kPlaneTag;
                const PairK<D1> c = pair_k<D1>(A.law.model, A.mat_pl[w], th, ir, 0.0, im, 0.0);
                plane_side<D1>(A.law, c, A.mat_pl[w].rfric, A.planes[w], A.plane_dbi + 15 * (size_t)w, in3(xi, 0, dir), ir,
                               in3(vi, 6, dir), in3(wi, 12, dir), s0, s1, acc);
            }
            double g[1] = {0.0};
            vjp_add3(g, acc.F, bF);
            vjp_add3(g, acc.M, bM);
            vjp_add3(g, acc.T, bT);
            vjp_add(g, acc.R, bR);
            vjp_add(g, s0, bs0);
            vjp_add(g, s1, bs1);
            // x_i, v_i, w_i stay in the lane, x_j, v_j, w_j go to the neighbour
            if (dir < 18) {
                const int kind = dir / 6, q = dir % 3;
                if (dir % 6 < 3) own += g[0];
                else if (!wall && g[0] != 0.0)
                    atomicAdd((kind == 0 ? R.lpos1 : (kind == 1 ? R.lb.vel : R.lom)) + 3 * (size_t)k + q, g[0]);
            } else if (dir >= 20 && dir < kPairN) {
                gth += g[0];
            }
            const double g18 = __shfl(g[0], 18, kContactLanes), g19 = __shfl(g[0], 19, kContactLanes);
            if (slot_in == dir / 2) {
                if (wall) pl += dir & 1 ? g19 : g18;
                else pp += dir & 1 ? g19 : g18;
            }
        }
        if (dir < 18 && dir % 6 < 3 && own != 0.0) {
            const int kind = dir / 6;
            atomicAdd((kind == 0 ? R.lpos1 : (kind == 1 ? R.lb.vel : R.lom)) + 3 * (size_t)i + dir % 3, own);
        }
        // slots this step did not write keep their values: their cotangents pass through
        if (dir < (int)(2u * A.cap))
            R.lb.pp_tsd[2 * sb + dir] = written_pp & (1u << (dir / 2)) ? pp : pp + R.la.pp_tsd[2 * sb + dir];
        if (dir < 2 * kPlSlots)
            R.lb.pl_tsd[2 * lb + dir] = written_pl & (1u << (dir / 2)) ? pl : pl + R.la.pl_tsd[2 * lb + dir];
    }
    // theta: the block's spheres, then one atomic per component
    __shared__ double part[256 / kContactLanes][3];
    if (dir >= 20 && dir < kPairN) part[threadIdx.x / kContactLanes][dir - 20] = gth;
    __syncthreads();
    if (threadIdx.x < 3u) {
        double v = 0.0;
        for (uint32_t q = 0; q < 256u / kContactLanes; q++) v += part[q][threadIdx.x];
        if (v != 0.0) atomicAdd(R.gtheta + threadIdx.x, v);
    }
}

// The angular velocity w(e', e_dot) and the position update of sphere i: the cotangents of
// the state before the step.
constexpr int kHeadN = 12;   // e (0-3), e_dot (4-7), e_ddot (8-11)

__global__ __launch_bounds__(64) void k_cal_rev_head(RevArgs R)
{
    const CalArgs& A = R.A;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n) return;
    const StepRec& r = R.r;
    const Lam &la = R.la, &lb = R.lb;
    // w = 2 G(e') e_dot: its cotangent adds to e' and e_dot
    double le1[4], lev[4];
    for (int q = 0; q < 4; q++) {
        le1[q] = R.le1[4 * (size_t)i + q] + la.ep[4 * (size_t)i + q];
        lev[q] = lb.ev[4 * (size_t)i + q];
    }
    {
        typedef Dual<8> D;
        const V3<D> w = ang_vel(seed4<8>(ld4d(r.ep1 + 4 * (size_t)i), 0), seed4<8>(ld4d(r.ev + 4 * (size_t)i), 4));
        double g[8];
        for (int q = 0; q < 8; q++) g[q] = 0.0;
        vjp_add3(g, w, ld3d(R.lom + 3 * (size_t)i));
        for (int q = 0; q < 4; q++) {
            le1[q] += g[q];
            lev[q] += g[4 + q];
        }
    }
    // position: p' = p + dt v + h a
    const V3<double> lp = ld3d(la.pos + 3 * (size_t)i) + ld3d(R.lpos1 + 3 * (size_t)i);
    for (int q = 0; q < 3; q++) {
        const double l = q == 0 ? lp.x : (q == 1 ? lp.y : lp.z);
        lb.pos[3 * (size_t)i + q] = l;
        lb.vel[3 * (size_t)i + q] += A.dt * l;
        lb.acc[3 * (size_t)i + q] += A.h * l;
    }
    // Euler parameters: e' = normalise(e + dt e_dot + h e_ddot)
    typedef Dual<kHeadN> D;
    V3<D> pd = {D(0.0), D(0.0), D(0.0)};
    V4<D> e = seed4<kHeadN>(ld4d(r.ep0 + 4 * (size_t)i), 0);
    position_update<D>(A.dt, A.h, pd, e, V3<D>{D(0.0), D(0.0), D(0.0)}, seed4<kHeadN>(ld4d(r.ev + 4 * (size_t)i), 4),
                       V3<D>{D(0.0), D(0.0), D(0.0)}, seed4<kHeadN>(ld4d(r.ea + 4 * (size_t)i), 8));
    double g[kHeadN];
    for (int q = 0; q < kHeadN; q++) g[q] = 0.0;
    vjp_add(g, e.x, le1[0]);
    vjp_add(g, e.y, le1[1]);
    vjp_add(g, e.z, le1[2]);
    vjp_add(g, e.w, le1[3]);
    for (int q = 0; q < 4; q++) {
        lb.ep[4 * (size_t)i + q] = g[q];
        lb.ev[4 * (size_t)i + q] = lev[q] + g[4 + q];
        lb.ea[4 * (size_t)i + q] += g[8 + q];
    }
}

__global__ void k_fill_zero(double* p, size_t n)
{
    for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x) p[k] = 0.0;
}

}  // namespace

// ============================================================================ host side
struct xdem_calib {
    xdem_calib_config cfg;
    hipStream_t stream = nullptr;
    uint32_t n = 0, cap = 12, nplane = 0, ncell = 0, every = 100, max_steps = 0, nseg = 0;
    double dt = 0.0, h = 0.0, g[3] = {0, 0, 0}, wo[3] = {0, 0, 0}, cs = 0.0;
    uint32_t gsize[3] = {128, 128, 128};
    Law law;
    Material mat_pp;
    std::vector<double> h_pos, h_vel, h_acc;   // initial state
    std::vector<void*> allocs;
    // device
    double *mass = nullptr, *inertia = nullptr;
    Material* d_mat_pl = nullptr;
    xdem_plane_info* d_planes = nullptr;
    double* d_plane_dbi = nullptr;
    StateView st;                               // current state (vel/ev: buffer 0 or 1)
    double *vel_buf[2] = {nullptr, nullptr}, *ev_buf[2] = {nullptr, nullptr};
    int sv = 0;
    uint32_t *hash = nullptr, *index = nullptr, *sorted = nullptr, *cstart = nullptr, *cend = nullptr;
    uint32_t* sort_buf[4] = {nullptr, nullptr, nullptr, nullptr};   // of the cell sort, with its scratch
    void* sort_scratch = nullptr;
    uint32_t* err = nullptr;
    // checkpoints: nseg states (doubles and slot arrays, packed)
    char* ckpt = nullptr;
    size_t state_bytes = 0;
    // segment records: every step's StepRec arrays and tape, packed per step
    char* recs = nullptr;
    size_t rec_bytes = 0;
    // reverse sweep
    double* lam[2] = {nullptr, nullptr};        // two Lam sets, packed
    size_t lam_doubles = 0;
    double *le1 = nullptr, *lom = nullptr, *lpos1 = nullptr, *bar = nullptr, *gtheta = nullptr;
    double theta[3] = {0, 0, 0};
    unsigned first_step = 0, last_steps = 0;   // the steps of the last forward run at theta
    bool have_forward = false;

    template <class P> hipError_t alloc(P** p, size_t bytes)
    {
        void* q = nullptr;
        hipError_t e = hipMalloc(&q, bytes ? bytes : 16);
        if (e != hipSuccess) return e;
        allocs.push_back(q);
        *p = static_cast<P*>(q);
        return hipSuccess;
    }

    // packed layout of a state: pos 4n, vel 3n, acc 3n, ep 4n, ev 4n, ea 4n, tmax 3n, rres n,
    // pp_tsd 2 cap n, pl_tsd 6n (doubles), then pp_count n, pp_id cap n, pl_count n, pl_id 3n
    size_t state_doubles() const { return (size_t)n * (4 + 3 + 3 + 4 + 4 + 4 + 3 + 1 + 2 * cap + 2 * kPlSlots); }
    size_t state_u32() const { return (size_t)n * (1 + cap + 1 + kPlSlots); }

    CalArgs args() const
    {
        CalArgs A;
        std::memset(&A, 0, sizeof(A));
        A.n = n; A.cap = cap; A.nplane = nplane; A.ncell = ncell;
        A.dt = dt; A.h = h; A.gx = g[0]; A.gy = g[1]; A.gz = g[2];
        for (int k = 0; k < 3; k++) { A.wo[k] = wo[k]; A.gsize[k] = gsize[k]; }
        A.cs = cs;
        A.law = law;
        A.flat_inertia = cfg.quirks.flat_inertia;
        A.mat_pp = mat_pp;
        A.mat_pl = d_mat_pl;
        A.planes = d_planes;
        A.plane_dbi = d_plane_dbi;
        A.mu = theta[0]; A.rest = theta[1]; A.s = theta[2];
        A.mass = mass;
        A.inertia = inertia;
        A.st = st;
        A.st.vel = vel_buf[sv];
        A.st.ev = ev_buf[sv];
        A.vel_out = vel_buf[sv ^ 1];
        A.ev_out = ev_buf[sv ^ 1];
        A.hash = hash; A.index = index; A.sorted = sorted; A.cstart = cstart; A.cend = cend;
        A.err = err;
        return A;
    }

    // copy the current state to/from a packed buffer
    hipError_t pack(char* dst) const
    {
        double* d = reinterpret_cast<double*>(dst);
        uint32_t* u = reinterpret_cast<uint32_t*>(d + state_doubles());
        const size_t N = n;
        const double* src[10] = {st.pos, vel_buf[sv], st.acc, st.ep, ev_buf[sv], st.ea, st.tmax, st.rres, st.pp_tsd, st.pl_tsd};
        const size_t len[10] = {4 * N, 3 * N, 3 * N, 4 * N, 4 * N, 4 * N, 3 * N, N, 2 * cap * N, 2 * kPlSlots * N};
        size_t o = 0;
        hipError_t e = hipSuccess;
        for (int k = 0; k < 10 && e == hipSuccess; k++) {
            e = hipMemcpyAsync(d + o, src[k], sizeof(double) * len[k], hipMemcpyDeviceToDevice, stream);
            o += len[k];
        }
        const uint32_t* us[4] = {st.pp_count, st.pp_id, st.pl_count, st.pl_id};
        const size_t ul[4] = {N, cap * N, N, kPlSlots * N};
        o = 0;
        for (int k = 0; k < 4 && e == hipSuccess; k++) {
            e = hipMemcpyAsync(u + o, us[k], sizeof(uint32_t) * ul[k], hipMemcpyDeviceToDevice, stream);
            o += ul[k];
        }
        return e;
    }
    hipError_t unpack(const char* srcb)
    {
        const double* d = reinterpret_cast<const double*>(srcb);
        const uint32_t* u = reinterpret_cast<const uint32_t*>(d + state_doubles());
        sv = 0;
        const size_t N = n;
        double* dst[10] = {st.pos, vel_buf[0], st.acc, st.ep, ev_buf[0], st.ea, st.tmax, st.rres, st.pp_tsd, st.pl_tsd};
        const size_t len[10] = {4 * N, 3 * N, 3 * N, 4 * N, 4 * N, 4 * N, 3 * N, N, 2 * cap * N, 2 * kPlSlots * N};
        size_t o = 0;
        hipError_t e = hipSuccess;
        for (int k = 0; k < 10 && e == hipSuccess; k++) {
            e = hipMemcpyAsync(dst[k], d + o, sizeof(double) * len[k], hipMemcpyDeviceToDevice, stream);
            o += len[k];
        }
        uint32_t* ud[4] = {st.pp_count, st.pp_id, st.pl_count, st.pl_id};
        const size_t ul[4] = {N, cap * N, N, kPlSlots * N};
        o = 0;
        for (int k = 0; k < 4 && e == hipSuccess; k++) {
            e = hipMemcpyAsync(ud[k], u + o, sizeof(uint32_t) * ul[k], hipMemcpyDeviceToDevice, stream);
            o += ul[k];
        }
        return e;
    }

    // record layout of one step: pos1 4n, ep0 4n, ep1 4n, vel 3n, ev 4n, ea 4n, pp_tsd 2 cap n,
    // pl_tsd 6n, sums 10n (doubles); tape_code kTape n (u32); tape_slot kTape n (u16); tape_n n (u8)
    size_t rec_size() const
    {
        size_t b = sizeof(double) * n * (4 + 4 + 4 + 3 + 4 + 4 + 2 * (size_t)cap + 2 * kPlSlots + 10);
        b += (sizeof(uint32_t) + sizeof(uint16_t)) * (size_t)n * kTape + (size_t)n;
        return (b + 255) & ~(size_t)255;
    }
    StepRec rec_view(size_t k) const
    {
        double* d = reinterpret_cast<double*>(recs + k * rec_bytes);
        const size_t N = n;
        StepRec r;
        r.pos1 = d; d += 4 * N;
        r.ep0 = d; d += 4 * N;
        r.ep1 = d; d += 4 * N;
        r.vel = d; d += 3 * N;
        r.ev = d; d += 4 * N;
        r.ea = d; d += 4 * N;
        r.pp_tsd = d; d += 2 * cap * N;
        r.pl_tsd = d; d += 2 * kPlSlots * N;
        r.sums = d; d += 10 * N;
        r.tape_code = reinterpret_cast<uint32_t*>(d);
        r.tape_slot = reinterpret_cast<uint16_t*>(r.tape_code + kTape * N);
        r.tape_n = reinterpret_cast<uint8_t*>(r.tape_slot + kTape * N);
        return r;
    }

    Lam lam_view(int k) const
    {
        double* p = lam[k];
        const size_t N = n;
        Lam L;
        L.pos = p; p += 3 * N;
        L.vel = p; p += 3 * N;
        L.acc = p; p += 3 * N;
        L.ep = p; p += 4 * N;
        L.ev = p; p += 4 * N;
        L.ea = p; p += 4 * N;
        L.pp_tsd = p; p += 2 * cap * N;
        L.pl_tsd = p; p += 2 * kPlSlots * N;
        return L;
    }

    // one forward step; rec (optional) receives the step's record
    hipError_t step(const StepRec* rec)
    {
        hipError_t e;
        const CalArgs A = args();
        const StepRec r = rec ? *rec : StepRec{};
        const uint32_t blocks = (n + kThreads - 1) / kThreads, G = wave_spheres(n);
        // the copies of a record keep 1,024 blocks busy
        if (rec) hipLaunchKernelGGL(k_cal_position<true>, dim3(std::max(blocks, 1024u)), dim3(kThreads), 0, stream, A, r);
        else hipLaunchKernelGGL(k_cal_position<false>, dim3(blocks), dim3(kThreads), 0, stream, A, r);
        if ((e = hipGetLastError())) return e;
        if ((e = cell_sort(hash, index, sorted, cstart, cend, n, ncell, sort_buf, sort_scratch, stream))) return e;
        const dim3 cg((n + kWaves * G - 1) / (kWaves * G)), cb(64 * kWaves);
        if (rec) hipLaunchKernelGGL(k_cal_contacts<true>, cg, cb, 0, stream, A, r, G);
        else hipLaunchKernelGGL(k_cal_contacts<false>, cg, cb, 0, stream, A, r, G);
        if ((e = hipGetLastError())) return e;
        sv ^= 1;
        return hipSuccess;
    }

    hipError_t reset()
    {
        hipError_t e;
        const size_t N = n;
        sv = 0;
        if ((e = hipMemcpyAsync(st.pos, h_pos.data(), sizeof(double) * 4 * N, hipMemcpyHostToDevice, stream))) return e;
        if ((e = hipMemcpyAsync(vel_buf[0], h_vel.data(), sizeof(double) * 3 * N, hipMemcpyHostToDevice, stream))) return e;
        if ((e = hipMemcpyAsync(st.acc, h_acc.data(), sizeof(double) * 3 * N, hipMemcpyHostToDevice, stream))) return e;
        std::vector<double> ep(4 * N, 0.0);
        for (size_t i = 0; i < N; i++) ep[4 * i] = 1.0;
        if ((e = hipMemcpyAsync(st.ep, ep.data(), sizeof(double) * 4 * N, hipMemcpyHostToDevice, stream))) return e;
        if ((e = hipStreamSynchronize(stream))) return e;   // ep is a local
        if ((e = hipMemsetAsync(ev_buf[0], 0, sizeof(double) * 4 * N, stream))) return e;
        if ((e = hipMemsetAsync(st.ea, 0, sizeof(double) * 4 * N, stream))) return e;
        if ((e = hipMemsetAsync(st.tmax, 0, sizeof(double) * 3 * N, stream))) return e;
        if ((e = hipMemsetAsync(st.rres, 0, sizeof(double) * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pp_count, 0, sizeof(uint32_t) * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pp_id, 0, sizeof(uint32_t) * cap * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pp_tsd, 0, sizeof(double) * 2 * cap * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pl_count, 0, sizeof(uint32_t) * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pl_id, 0, sizeof(uint32_t) * kPlSlots * N, stream))) return e;
        if ((e = hipMemsetAsync(st.pl_tsd, 0, sizeof(double) * 2 * kPlSlots * N, stream))) return e;
        return hipSuccess;
    }
};

#define CAL_CHECK(x)                                 \
    do {                                             \
        hipError_t e_ = (x);                         \
        if (e_ != hipSuccess) return XDEM_E_HIP;     \
    } while (0)

extern "C" {

int xdem_calib_create(const xdem_scene* s, const xdem_calib_config* cfg_in, xdem_calib** out)
{
    if (!s || !out || s->np == 0 || !s->pos || !s->mass || !s->inertia) return XDEM_E_INVALID;
    if (s->nplane && (!s->planes || !s->plane_dbi || !s->plane_cp)) return XDEM_E_INVALID;
    if (!(s->dt > 0.0) || !(s->cell_size > 0.0)) return XDEM_E_INVALID;
    if (s->contact_model != 0 && s->contact_model != 1) return XDEM_E_INVALID;
    xdem_calib_config cfg = {};
    if (cfg_in) cfg = *cfg_in;
    if (cfg.quirks.velocity_not_updated) return XDEM_E_UNSUPPORTED;
    if (s->cp_pp.coh != 0.0) return XDEM_E_UNSUPPORTED;
    for (unsigned k = 0; k < s->nplane; k++)
        if (s->plane_cp[k].coh != 0.0 || s->planes[k].id != k) return XDEM_E_UNSUPPORTED;
    const unsigned cap = cfg.capacity ? cfg.capacity : 12u;
    if (cap > (unsigned)kCapMax || s->nplane > 8u) return XDEM_E_INVALID;
    xdem_calib* c = new (std::nothrow) xdem_calib();
    if (!c) return XDEM_E_INVALID;
    c->cfg = cfg;
    c->n = s->np;
    c->cap = cap;
    c->nplane = s->nplane;
    c->every = cfg.checkpoint_every ? cfg.checkpoint_every : 100u;
    c->max_steps = cfg.max_steps ? cfg.max_steps : c->every;
    c->nseg = (c->max_steps + c->every - 1) / c->every;
    c->dt = s->dt;
    c->h = 0.5 * s->dt * s->dt;
    for (int k = 0; k < 3; k++) { c->g[k] = s->gravity[k]; c->wo[k] = s->world_origin[k]; }
    c->cs = s->cell_size;
    // The buckets of the cells: at least four to a sphere, so that clearing and sorting cost what
    // the spheres need (128^3 of them: 5.5 us to clear, three digits to sort). Contacts and their
    // order are those of 128 a side while spheres a side or more apart cannot overlap, that is
    // while no sphere is larger than a cell.
    double rmax = 0.0;
    for (size_t i = 0; i < s->np; i++) rmax = std::max(rmax, s->pos[4 * i + 3]);
    uint32_t side = 128;
    if (2.0 * rmax <= s->cell_size)
        for (side = 16; side < 128 && (uint64_t)side * side * side < 4 * (uint64_t)s->np;) side *= 2;
    for (uint32_t& q : c->gsize) q = side;
    c->ncell = c->gsize[0] * c->gsize[1] * c->gsize[2];
    c->law.model = s->contact_model;
    c->law.gpu_law = cfg.quirks.gpu_force_law != 0;
    c->law.stale_ft = cfg.quirks.stale_ft != 0;
    c->law.dt = s->dt;
    const xdem_contact_property& p = s->cp_pp;
    c->mat_pp = {p.Ei, p.Ej, p.pri, p.prj, p.rfric, p.sratio};
    const size_t N = s->np;
    c->h_pos.assign(s->pos, s->pos + 4 * N);
    c->h_vel.assign(3 * N, 0.0);
    if (s->vel) c->h_vel.assign(s->vel, s->vel + 3 * N);
    c->h_acc.assign(3 * N, 0.0);
    for (size_t i = 0; i < N; i++) c->h_acc[3 * i + 1] = s->gravity[1];   // acc = (0, g.y, 0) at the start
    auto fail = [&](int rc) {
        xdem_calib_destroy(c);
        return rc;
    };
    if (hipSetDevice(cfg.device) != hipSuccess) return fail(XDEM_E_HIP);
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) return fail(XDEM_E_HIP);
#define ALLOC(p, bytes) if (c->alloc(&(p), (bytes)) != hipSuccess) return fail(XDEM_E_HIP)
    ALLOC(c->mass, sizeof(double) * N);
    ALLOC(c->inertia, sizeof(double) * 3 * N);
    ALLOC(c->d_mat_pl, sizeof(Material) * std::max(1u, s->nplane));
    ALLOC(c->d_planes, sizeof(xdem_plane_info) * std::max(1u, s->nplane));
    ALLOC(c->d_plane_dbi, sizeof(double) * 15 * std::max(1u, s->nplane));
    ALLOC(c->st.pos, sizeof(double) * 4 * N);
    ALLOC(c->vel_buf[0], sizeof(double) * 3 * N);
    ALLOC(c->vel_buf[1], sizeof(double) * 3 * N);
    ALLOC(c->st.acc, sizeof(double) * 3 * N);
    ALLOC(c->st.ep, sizeof(double) * 4 * N);
    ALLOC(c->ev_buf[0], sizeof(double) * 4 * N);
    ALLOC(c->ev_buf[1], sizeof(double) * 4 * N);
    ALLOC(c->st.ea, sizeof(double) * 4 * N);
    ALLOC(c->st.tmax, sizeof(double) * 3 * N);
    ALLOC(c->st.rres, sizeof(double) * N);
    ALLOC(c->st.pp_count, sizeof(uint32_t) * N);
    ALLOC(c->st.pp_id, sizeof(uint32_t) * cap * N);
    ALLOC(c->st.pp_tsd, sizeof(double) * 2 * cap * N);
    ALLOC(c->st.pl_count, sizeof(uint32_t) * N);
    ALLOC(c->st.pl_id, sizeof(uint32_t) * kPlSlots * N);
    ALLOC(c->st.pl_tsd, sizeof(double) * 2 * kPlSlots * N);
    ALLOC(c->hash, sizeof(uint32_t) * N);
    ALLOC(c->index, sizeof(uint32_t) * N);
    ALLOC(c->sorted, sizeof(uint32_t) * N);
    ALLOC(c->cstart, sizeof(uint32_t) * c->ncell);
    ALLOC(c->cend, sizeof(uint32_t) * c->ncell);
    for (uint32_t*& q : c->sort_buf) ALLOC(q, sizeof(uint32_t) * N);
    ALLOC(c->sort_scratch, cell_sort_scratch_bytes(c->n));
    ALLOC(c->err, sizeof(uint32_t));
    c->state_bytes = (sizeof(double) * c->state_doubles() + sizeof(uint32_t) * c->state_u32() + 255) & ~(size_t)255;
    ALLOC(c->ckpt, c->state_bytes * c->nseg);
    c->rec_bytes = c->rec_size();
    ALLOC(c->recs, c->rec_bytes * c->every);
    c->lam_doubles = N * (3 + 3 + 3 + 4 + 4 + 4 + 2 * (size_t)cap + 2 * kPlSlots);
    ALLOC(c->lam[0], sizeof(double) * c->lam_doubles);
    ALLOC(c->lam[1], sizeof(double) * c->lam_doubles);
    ALLOC(c->le1, sizeof(double) * 4 * N);
    ALLOC(c->lom, sizeof(double) * 3 * N);
    ALLOC(c->lpos1, sizeof(double) * 3 * N);
    ALLOC(c->bar, sizeof(double) * 10 * N);
    ALLOC(c->gtheta, sizeof(double) * 3);
#undef ALLOC
    std::vector<Material> mpl(std::max(1u, s->nplane));
    for (unsigned k = 0; k < s->nplane; k++) {
        const xdem_contact_property& q = s->plane_cp[k];
        mpl[k] = {q.Ei, q.Ej, q.pri, q.prj, q.rfric, q.sratio};
    }
    hipStream_t st = c->stream;
    if (hipMemcpyAsync(c->mass, s->mass, sizeof(double) * N, hipMemcpyHostToDevice, st) ||
        hipMemcpyAsync(c->inertia, s->inertia, sizeof(double) * 3 * N, hipMemcpyHostToDevice, st) ||
        hipMemcpyAsync(c->d_mat_pl, mpl.data(), sizeof(Material) * mpl.size(), hipMemcpyHostToDevice, st) ||
        (s->nplane && hipMemcpyAsync(c->d_planes, s->planes, sizeof(xdem_plane_info) * s->nplane, hipMemcpyHostToDevice, st)) ||
        (s->nplane && hipMemcpyAsync(c->d_plane_dbi, s->plane_dbi, sizeof(double) * 15 * s->nplane, hipMemcpyHostToDevice, st)) ||
        hipMemsetAsync(c->err, 0, sizeof(uint32_t), st) || hipStreamSynchronize(st))
        return fail(XDEM_E_HIP);
    *out = c;
    return XDEM_OK;
}

int xdem_calib_destroy(xdem_calib* c)
{
    if (!c) return XDEM_E_INVALID;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (void* p : c->allocs) (void)hipFree(p);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return XDEM_OK;
}

int xdem_calib_forward(xdem_calib* c, const double theta[3], unsigned int nsteps, double* pos_out)
{
    if (!c || !theta) return XDEM_E_INVALID;
    if (nsteps > c->max_steps) return XDEM_E_INVALID;
    if (!(theta[0] >= 0.0) || !(theta[1] > 0.0) || !std::isfinite(theta[2])) return XDEM_E_INVALID;
    CAL_CHECK(hipSetDevice(c->cfg.device));
    for (int k = 0; k < 3; k++) c->theta[k] = theta[k];
    CAL_CHECK(c->reset());
    for (unsigned k = 0; k < nsteps; k++) {
        if (k % c->every == 0) CAL_CHECK(c->pack(c->ckpt + (k / c->every) * c->state_bytes));
        CAL_CHECK(c->step(nullptr));
    }
    CAL_CHECK(hipStreamSynchronize(c->stream));
    c->first_step = 0;
    c->last_steps = nsteps;
    c->have_forward = true;
    if (pos_out)
        CAL_CHECK(hipMemcpy(pos_out, c->st.pos, sizeof(double) * 4 * (size_t)c->n, hipMemcpyDeviceToHost));
    return XDEM_OK;
}

int xdem_calib_forward_from(xdem_calib* c, const double theta[3], unsigned int start, unsigned int nsteps,
                            double* pos_out)
{
    if (!c || !theta) return XDEM_E_INVALID;
    if (!c->have_forward) return XDEM_E_NOT_READY;
    // the run restarts from a stored state of the last run: at a checkpoint it passed
    if (start % c->every != 0 || start > c->last_steps || start >= nsteps || nsteps > c->max_steps) return XDEM_E_INVALID;
    if (!(theta[0] >= 0.0) || !(theta[1] > 0.0) || !std::isfinite(theta[2])) return XDEM_E_INVALID;
    CAL_CHECK(hipSetDevice(c->cfg.device));
    if (start == c->last_steps) {
        // the end state of the last run is not a stored one unless a checkpoint was written there
        CAL_CHECK(c->pack(c->ckpt + (start / c->every) * c->state_bytes));
    }
    CAL_CHECK(c->unpack(c->ckpt + (start / c->every) * c->state_bytes));
    for (int k = 0; k < 3; k++) c->theta[k] = theta[k];
    for (unsigned k = start; k < nsteps; k++) {
        if (k % c->every == 0 && k != start) CAL_CHECK(c->pack(c->ckpt + (k / c->every) * c->state_bytes));
        CAL_CHECK(c->step(nullptr));
    }
    CAL_CHECK(hipStreamSynchronize(c->stream));
    c->first_step = start;
    c->last_steps = nsteps;
    if (pos_out)
        CAL_CHECK(hipMemcpy(pos_out, c->st.pos, sizeof(double) * 4 * (size_t)c->n, hipMemcpyDeviceToHost));
    return XDEM_OK;
}

int xdem_calib_state(xdem_calib* c, double* pos, double* vel, double* ep, double* ev)
{
    if (!c) return XDEM_E_INVALID;
    CAL_CHECK(hipSetDevice(c->cfg.device));
    CAL_CHECK(hipStreamSynchronize(c->stream));
    const size_t N = c->n;
    if (pos) CAL_CHECK(hipMemcpy(pos, c->st.pos, sizeof(double) * 4 * N, hipMemcpyDeviceToHost));
    if (vel) CAL_CHECK(hipMemcpy(vel, c->vel_buf[c->sv], sizeof(double) * 3 * N, hipMemcpyDeviceToHost));
    if (ep) CAL_CHECK(hipMemcpy(ep, c->st.ep, sizeof(double) * 4 * N, hipMemcpyDeviceToHost));
    if (ev) CAL_CHECK(hipMemcpy(ev, c->ev_buf[c->sv], sizeof(double) * 4 * N, hipMemcpyDeviceToHost));
    return XDEM_OK;
}

int xdem_calib_backward(xdem_calib* c, const double* dL_dpos, double grad[3])
{
    if (!c || !dL_dpos || !grad) return XDEM_E_INVALID;
    if (!c->have_forward) return XDEM_E_NOT_READY;
    CAL_CHECK(hipSetDevice(c->cfg.device));
    hipStream_t st = c->stream;
    const size_t N = c->n;
    const dim3 zg(256), zb(256);
    hipLaunchKernelGGL(k_fill_zero, zg, zb, 0, st, c->lam[0], c->lam_doubles);
    hipLaunchKernelGGL(k_fill_zero, zg, zb, 0, st, c->gtheta, (size_t)3);
    CAL_CHECK(hipGetLastError());
    int la = 0;
    CAL_CHECK(hipMemcpyAsync(c->lam_view(la).pos, dL_dpos, sizeof(double) * 3 * N, hipMemcpyHostToDevice, st));
    const unsigned nsteps = c->last_steps;
    const dim3 grid((c->n + 63) / 64), block(64);
    const dim3 tail_grid((unsigned)(((size_t)c->n * kTailLanes + 255) / 256));
    const dim3 contact_grid((unsigned)(((size_t)c->n * kContactLanes + 255) / 256));
    const int seg0 = (int)(c->first_step / c->every);
    for (int seg = (int)((nsteps + c->every - 1) / c->every) - 1; seg >= seg0; seg--) {
        const unsigned k0 = (unsigned)seg * c->every, k1 = std::min(nsteps, k0 + c->every);
        // recompute the segment from its checkpoint, recording every step
        CAL_CHECK(c->unpack(c->ckpt + (size_t)seg * c->state_bytes));
        for (unsigned k = k0; k < k1; k++) {
            const StepRec r = c->rec_view(k - k0);
            CAL_CHECK(c->step(&r));
        }
        // and sweep it backwards
        for (int k = (int)k1 - 1; k >= (int)k0; k--) {
            RevArgs R;
            std::memset(&R, 0, sizeof(R));
            R.A = c->args();
            R.r = c->rec_view((size_t)(k - (int)k0));
            R.la = c->lam_view(la);
            R.lb = c->lam_view(la ^ 1);
            R.le1 = c->le1; R.lom = c->lom; R.lpos1 = c->lpos1; R.bar = c->bar; R.gtheta = c->gtheta;
            hipLaunchKernelGGL(k_cal_rev_tail, tail_grid, dim3(256), 0, st, R);
            hipLaunchKernelGGL(k_cal_rev_contacts, contact_grid, dim3(256), 0, st, R);
            hipLaunchKernelGGL(k_cal_rev_head, grid, block, 0, st, R);
            CAL_CHECK(hipGetLastError());
            la ^= 1;
        }
    }
    CAL_CHECK(hipMemcpyAsync(grad, c->gtheta, sizeof(double) * 3, hipMemcpyDeviceToHost, st));
    CAL_CHECK(hipStreamSynchronize(st));
    return XDEM_OK;
}

int xdem_calib_error_word(xdem_calib* c, unsigned int* out, int clear)
{
    if (!c || !out) return XDEM_E_INVALID;
    CAL_CHECK(hipSetDevice(c->cfg.device));
    CAL_CHECK(hipStreamSynchronize(c->stream));
    CAL_CHECK(hipMemcpy(out, c->err, sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (clear) CAL_CHECK(hipMemset(c->err, 0, sizeof(uint32_t)));
    return XDEM_OK;
}

int xdem_calib_pair_eval(const xdem_contact_property* cp, int contact_model, const xdem_quirks* q, double dt,
                         double ir, double jr, double im, double jm, const double in[23], double out[12], double* jac)
{
    if (!cp || !q || !in || !out) return XDEM_E_INVALID;
    Law L;
    L.model = contact_model;
    L.gpu_law = q->gpu_force_law != 0;
    L.stale_ft = q->stale_ft != 0;
    L.dt = dt;
    const Material m = {cp->Ei, cp->Ej, cp->pri, cp->prj, cp->rfric, cp->sratio};
    for (int k = 0; k < 12; k++) out[k] = 0.0;
    if (jac)
        for (int k = 0; k < 12 * kPairN; k++) jac[k] = 0.0;
    typedef Dual<kPairN> D;
    const Theta<D> th = {D::input(in[20], 20), D::input(in[21], 21), D::input(in[22], 22)};
    const PairK<D> c = pair_k<D>(contact_model, m, th, ir, jr, im, jm);
    auto v3 = [&](int k) { return V3<double>{in[k], in[k + 1], in[k + 2]}; };
    D s0 = D::input(in[18], 18), s1 = D::input(in[19], 19);
    V3<D> Ft = {D(0.0), D(0.0), D(0.0)};
    Sums<D> acc = zero_sums<D>();
    const bool hit = pair_side<D>(L, c, cp->rfric, seed3<kPairN>(v3(0), 0), ir, seed3<kPairN>(v3(3), 3), jr,
                                  seed3<kPairN>(v3(6), 6), seed3<kPairN>(v3(9), 9), seed3<kPairN>(v3(12), 12),
                                  seed3<kPairN>(v3(15), 15), s0, s1, Ft, acc);
    if (!hit) return 0;
    const D* o[12] = {&acc.F.x, &acc.F.y, &acc.F.z, &acc.M.x, &acc.M.y, &acc.M.z, &acc.T.x, &acc.T.y, &acc.T.z, &acc.R, &s0, &s1};
    for (int r = 0; r < 12; r++) {
        out[r] = o[r]->v;
        if (jac)
            for (int k = 0; k < kPairN; k++) jac[r * kPairN + k] = o[r]->d[k];
    }
    return 1;
}

}  // extern "C"
