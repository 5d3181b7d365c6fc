// Small :dipole replicas stepped inside one launch per call ("resident"):
// the spins stay in registers and LDS for all steps, and workgroups exchange
// the sites on their borders through words that carry their own validity.
//
// Reference semantics: step!(::System{0}, ::Langevin) and
// step!(::System{0}, ::ImplicitMidpoint), src/Integrators.jl:313-332, 379-413;
// fast_isapprox, :361-371.
//
// A replica's sites are cut into parts of at most 64 (one wavefront; a
// replica of up to kResOneWg sites is one part of up to eight wavefronts).
// Part p keeps its own sites and the neighbours it reads from other parts
// (its halo) in LDS, two buffers in turn, and every bond slot of a site as
// a 16-bit index into them.  A round is one exchange: every lane publishes
// its site, the workgroup's other wavefronts poll the halo sites, one
// workgroup barrier, next stage.  Langevin takes two rounds per step (the
// predictor's S' and the corrector's S); the midpoint one per fixed-point
// iteration plus one per step.
//
// A published dipole is split into 8-byte words, each 4 data bytes and the
// 4-byte round number, stored and loaded with relaxed agent-scope atomics:
// the flag-with-the-data words that collective libraries publish as their
// low-latency (LL) protocol, hence the prefix ll_.
// A reader polls until every word carries its round: the data needs no
// fence, no flag and no cache write-back, and one store-to-load latency
// across the XCDs is all a round costs, against a release, an arrival
// counter, a generation and an acquire for a grid barrier.  Two slots
// alternate: a part
// publishes round n + 2 only after it has read every reader's round n + 1,
// which that reader published after reading round n (bonds are symmetric,
// which the plan checks), so no word is overwritten while it is awaited.
//
// What bounds it: the exchange and the FP64 chain of one site, about 2 us a
// round.  Cubic 16^3 FP64 (64 parts): Langevin 11.2 -> 4.3 us per step
// (two launches before), midpoint 93 -> 48 us per step of 14 iterations (a
// grid barrier per iteration before: 6.6 -> 3.4 us).  378 sites in one
// workgroup: 8.9 -> 3.9 us per step (spins through global memory before).
// Parts of 64 sites, one wavefront on a compute unit to itself, keep the
// chain as short as it gets; three more wavefronts poll the halo (about 96
// sites of a cubic part), so its words arrive side by side.
#include <algorithm>
#include <map>

#include "snh_gather.h"

namespace snh {

namespace {

__device__ __forceinline__ void ll_store(unsigned long long* p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned long long ll_load(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A real as tagged words: two for FP64, one for FP32.
template <typename T>
constexpr int kWords = sizeof(T) == 8 ? 2 : 1;

__device__ __forceinline__ void ll_put(unsigned long long* p, size_t stride, double v, unsigned tag)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v), t = (unsigned long long)tag << 32;
    ll_store(p, (b & 0xffffffffull) | t);
    ll_store(p + stride, (b >> 32) | t);
}

__device__ __forceinline__ void ll_put(unsigned long long* p, size_t, float v, unsigned tag)
{
    ll_store(p, (unsigned long long)__float_as_uint(v) | (unsigned long long)tag << 32);
}

__device__ __forceinline__ double ll_value(const unsigned long long* w, double)
{
    return __longlong_as_double((long long)((w[0] & 0xffffffffull) | (w[1] << 32)));
}

__device__ __forceinline__ float ll_value(const unsigned long long* w, float)
{
    return __uint_as_float((unsigned)w[0]);
}

// What a workgroup knows of its part, its lane's site and its LDS.
template <typename T>
struct Part {
    ResWg w;
    int t, nt;       // thread, threads of the workgroup
    bool own;        // this thread holds a site
    SiteCoord sc;    // its site
    T* buf;          // [2][3][nsite]
    const unsigned short* nbr;  // [nslot][nlane]
    int nsite;
    bool lost;       // a wait timed out: no further waits
};

template <typename T>
__device__ __forceinline__ V3<T> lds_get(const T* b, int nsite, int k)
{
    return {b[k], b[nsite + k], b[2 * nsite + k]};
}

template <typename T>
__device__ __forceinline__ void lds_put(T* b, int nsite, int k, V3<T> v)
{
    b[k] = v.x;
    b[nsite + k] = v.y;
    b[2 * nsite + k] = v.z;
}

// Site of lane entry e (cell * na + sublattice, -1: idle) of replica r.
template <typename T>
__device__ __forceinline__ SiteCoord res_site(const Couplings<T>& C, int r, int e)
{
    SiteCoord sc;
    sc.blk = 0;
    sc.r = r;
    sc.R = C.reps[r];
    sc.valid = e >= 0;
    const int v = e >= 0 ? e : 0;
    sc.c = v / C.na;
    sc.i = v - sc.c * C.na;
    const int q = fdiv(sc.c, sc.R.L1, sc.R.inv1);
    sc.c1 = sc.c - q * sc.R.L1;
    sc.c3 = fdiv(q, sc.R.L2, sc.R.inv2);
    sc.c2 = q - sc.c3 * sc.R.L2;
    sc.g = sc.R.off + (uint32_t)((sc.c1 + C.G.w1) + sc.R.P1 * ((sc.c2 + C.G.w2) + sc.R.P2 * (sc.c3 + C.G.w3))) +
           sc.R.pcell * (uint32_t)sc.i;
    sc.edge = (sc.c1 < C.G.w1) | (sc.c1 >= sc.R.L1 - C.G.w1) | (sc.c2 < C.G.w2) | (sc.c2 >= sc.R.L2 - C.G.w2) |
              (sc.c3 < C.G.w3) | (sc.c3 >= sc.R.L3 - C.G.w3);
    return sc;
}

// Loads the part's tables; kUni: one sublattice (its couplings then stay in
// scalar registers).
template <typename T, bool kUni>
__device__ __forceinline__ Part<T> res_part(const Couplings<T>& C, const ResArgs& A)
{
    extern __shared__ double res_lds[];
    Part<T> P;
    P.w = A.wg[blockIdx.x];
    P.t = (int)threadIdx.x;
    P.nt = (int)blockDim.x;
    P.nsite = P.w.nlane + P.w.nhalo;
    P.buf = reinterpret_cast<T*>(res_lds);
    unsigned short* nbr = reinterpret_cast<unsigned short*>(P.buf + 6 * P.nsite);
    const int n = A.nslot * P.w.nlane;
    for (int k = P.t; k < n; k += P.nt) nbr[k] = A.nbr[P.w.nbr0 + k];
    P.nbr = nbr;
    P.sc = res_site(C, P.w.r, P.t < P.w.nlane ? A.lane[P.w.lane0 + P.t] : -1);
    if (kUni) P.sc.i = 0;
    P.own = P.sc.valid;
    P.lost = false;
    return P;
}

// dE/dS at the thread's site from the LDS copy b: the terms and their order
// are those of local_field.  An isotropic bond is one fused multiply-add per
// component in the launched Heun stages and a product and a sum in the
// launched midpoint sweeps (whose general form the compiler cannot fuse);
// kFused follows suit, so that Langevin states agree bitwise, and midpoint
// ones in FP64.
template <typename T, int CH, bool kIso, bool kFused>
__device__ __forceinline__ V3<T> res_field(const Couplings<T>& C, const Part<T>& P, const T* b, V3<T> s)
{
    const int i = P.sc.i;
    V3<T> g = {C.zee[3 * i], C.zee[3 * i + 1], C.zee[3 * i + 2]};
    const int b0 = C.bstart[i], n = C.bstart[i + 1] - b0;
    for (int c0 = 0; c0 < n; c0 += CH) {
        V3<T> sj[CH];
#pragma unroll
        for (int k = 0; k < CH; k++) sj[k] = lds_get(b, P.nsite, P.nbr[(c0 + k) * P.w.nlane + P.t]);
#pragma unroll
        for (int k = 0; k < CH; k++) {
            const int q = b0 + c0 + k;
            if (kIso && kFused) {
                const T J0 = C.bJ0[q];
                g.x += J0 * sj[k].x;
                g.y += J0 * sj[k].y;
                g.z += J0 * sj[k].z;
            } else if (kIso) {
#pragma clang fp contract(off)
                const T J0 = C.bJ0[q];
                g.x += J0 * sj[k].x;
                g.y += J0 * sj[k].y;
                g.z += J0 * sj[k].z;
            } else {
                add_bond_field(C, q, s, sj[k], g);
            }
        }
    }
    add_onsite_field(C, i, s, g);
    return g;
}

// The thread's site of round `tag` for the parts that read it.
template <typename T>
__device__ __forceinline__ void res_publish(const ResArgs& A, const Part<T>& P, unsigned tag, V3<T> v)
{
    unsigned long long* p = A.ex + (size_t)(tag & 1) * 3 * kWords<T> * A.nex + P.w.ex0 + P.t;
    ll_put(p, A.nex, v.x, tag);
    ll_put(p + kWords<T> * (size_t)A.nex, A.nex, v.y, tag);
    ll_put(p + 2 * kWords<T> * (size_t)A.nex, A.nex, v.z, tag);
}

// Ends a wait that lasted too long: every thread of the launch stops waiting,
// the launch runs to its end on whatever it holds, and the host, which kept
// the state of the call's start, makes the call again stage by stage.
template <typename T>
__device__ __forceinline__ bool res_give_up(const ResArgs& A, Part<T>& P, unsigned n)
{
    if (n > A.spin || ((n & 255u) == 0 && __hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))) {
        __hip_atomic_store(A.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        P.lost = true;
    }
    return P.lost;
}

// The halo of round `tag` into the LDS copy b.  The wavefronts without sites
// of their own come first in the assignment.
template <typename T>
__device__ __forceinline__ void res_halo(const ResArgs& A, Part<T>& P, unsigned tag, T* b)
{
    constexpr int W = 3 * kWords<T>;
    const unsigned long long* base = A.ex + (size_t)(tag & 1) * W * A.nex + P.w.exr;
    const int first = P.t >= P.w.nlane ? P.t - P.w.nlane : P.t + P.nt - P.w.nlane;
    for (int h = first; h < P.w.nhalo; h += P.nt) {
        const unsigned long long* p = base + A.halo[P.w.halo0 + h];
        unsigned long long w[W];
        unsigned n = 0;
        bool ok;
        do {
            ok = true;
#pragma unroll
            for (int k = 0; k < W; k++) w[k] = ll_load(p + (size_t)k * A.nex);
#pragma unroll
            for (int k = 0; k < W; k++) ok &= (unsigned)(w[k] >> 32) == tag;
        } while (!ok && !P.lost && !res_give_up(A, P, ++n));
        lds_put(b, P.nsite, P.w.nlane + h,
                V3<T>{ll_value(w, T(0)), ll_value(w + kWords<T>, T(0)), ll_value(w + 2 * kWords<T>, T(0))});
    }
}

// The state and its halo from the planes X into the LDS copy b.
template <typename T>
__device__ __forceinline__ void res_load(const Couplings<T>& C, const ResArgs& A, const Part<T>& P, const T* X, T* b)
{
    for (int h = P.t; h < P.w.nhalo; h += P.nt) {
        const SiteCoord q = res_site(C, P.w.r, A.lane[P.w.laner + A.halo[P.w.halo0 + h]]);
        lds_put(b, P.nsite, P.w.nlane + h, planes(X, C.total)(q.g));
    }
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// The thread's site of the call's start, in the order of the host's states.
template <typename T>
__device__ __forceinline__ void res_keep(const Part<T>& P, T* __restrict__ keep, V3<T> s)
{
    T* p = keep + 3 * (size_t)(P.sc.c + P.sc.R.ncell * P.sc.i);
    p[0] = s.x;
    p[1] = s.y;
    p[2] = s.z;
}

template <typename T, int CH, bool kIso, bool kUni, int NT>
__global__ __launch_bounds__(NT) void k_res_langevin(Couplings<T> C, ResArgs A, T* X, T* __restrict__ keep,
                                                     NoiseArgs<T> nz, T dt, T lambda, int nsteps)
{
    Part<T> P = res_part<T, kUni>(C, A);
    T* const b0 = P.buf;                 // S
    T* const b1 = P.buf + 3 * P.nsite;   // S'
    const uint32_t site = (uint32_t)(P.sc.c + P.sc.R.ncell * P.sc.i);
    const T kap = C.kappa[P.sc.i];
    const bool noisy = lambda != (T)0;
    const unsigned long long step0 = nz.step;
    V3<T> s = {0, 0, 0}, xi = {0, 0, 0};
    if (P.own) {
        s = planes(X, C.total)(P.sc.g);
        if (keep) res_keep(P, keep, s);
        lds_put(b0, P.nsite, P.t, s);
        if (noisy) xi = dipole_noise(nz, P.sc.r, site, P.sc.g);
    }
    res_load(C, A, P, X, b0);
    __syncthreads();
    unsigned tag = 0;
    for (int n = 0; n < nsteps; n++) {
        const bool last = n == nsteps - 1;
        V3<T> sp = {0, 0, 0}, h = {0, 0, 0};
        ++tag;
        if (P.own) {
            const V3<T> g = res_field<T, CH, kIso, true>(C, P, b0, s);
            heun_predict(s, g, xi, noisy, kap, dt, lambda, sp, h);
            if (P.w.nhalo) res_publish(A, P, tag, sp);
            lds_put(b1, P.nsite, P.t, sp);
            // the next step's noise while the neighbours' S' is under way
            if (noisy && !last) {
                nz.step = step0 + (unsigned long long)(n + 1);
                xi = dipole_noise(nz, P.sc.r, site, P.sc.g);
            }
        }
        res_halo(A, P, tag, b1);
        __syncthreads();
        ++tag;
        if (P.own) {
            const V3<T> d = rhs_det(sp, res_field<T, CH, kIso, true>(C, P, b1, sp), dt, lambda);
            s = normalize_dipole(V3<T>{h.x + d.x / 2, h.y + d.y / 2, h.z + d.z / 2}, kap);
            if (P.w.nhalo && !last) res_publish(A, P, tag, s);
            lds_put(b0, P.nsite, P.t, s);
        }
        if (last) break;
        res_halo(A, P, tag, b0);
        __syncthreads();
    }
    if (P.own) store3_images(X, C.total, P.sc, C.G, s);
}

// The residual of residual round `tag` (counted apart from the halo rounds:
// a part that publishes residual m + 2 has read everybody's m + 1, published
// after they read m): every wavefront with sites publishes its sum, the last
// wavefront of each workgroup collects them in one order, so all parts of a
// replica see the same total.
template <typename T>
__device__ __forceinline__ void res_residual(const ResArgs& A, Part<T>& P, unsigned tag, double* tot)
{
    if (P.t < P.nt - 64) return;
    const int lane = P.t & 63;
    const unsigned long long* base = A.res + (size_t)(tag & 1) * 2 * A.nres + P.w.resr;
    double v = 0;
    for (int k = lane; k < P.w.nresr; k += 64) {
        unsigned long long w[2];
        unsigned n = 0;
        bool ok;
        do {
            w[0] = ll_load(base + k);
            w[1] = ll_load(base + A.nres + k);
            ok = (unsigned)(w[0] >> 32) == tag && (unsigned)(w[1] >> 32) == tag;
        } while (!ok && !P.lost && !res_give_up(A, P, ++n));
        v += ll_value(w, 0.0);
    }
    v = wave_sum(v);
    if (lane == 0) *tot = v;
}

template <typename T, int CH, bool kIso, bool kUni, int NT>
__global__ __launch_bounds__(NT) void k_res_midpoint(Couplings<T> C, ResArgs A, T* X, T* __restrict__ keep, T dt,
                                                     T lambda, const double* __restrict__ atol2, int max_iters, int nsteps,
                                                     int* __restrict__ iters_out, int* __restrict__ fail_step,
                                                     T* Sdd)
{
    __shared__ double red[2][kResOneWg / 64];  // one part: the wavefronts' sums; several: [p][0] the total
    Part<T> P = res_part<T, kUni>(C, A);
    const T kap = C.kappa[P.sc.i];
    const double a2 = atol2[P.w.r];
    const bool parts = P.w.nresr != 0;  // several workgroups share the replica
    const int nwave = P.w.nlane / 64;
    V3<T> s = {0, 0, 0}, prev = {0, 0, 0};
    if (P.own) {
        s = planes(X, C.total)(P.sc.g);
        if (keep) res_keep(P, keep, s);
    }
    unsigned tag = 0, rtag = 0;
    int p = 0, it = 0, failed = -1;
    __syncthreads();  // the bond table
    for (int n = 0; n < nsteps; n++) {
        // the first guess S' = S: Shat = kappa n((S + S)/2) = kappa n(S)
        V3<T> h = {0, 0, 0};
        prev = s;
        T* b = P.buf + 3 * p * P.nsite;
        ++tag;
        if (P.own) {
            h = normalize_dipole(s, kap);
            if (P.w.nhalo) res_publish(A, P, tag, h);
            lds_put(b, P.nsite, P.t, h);
        }
        res_halo(A, P, tag, b);
        __syncthreads();
        it = 0;
        bool conv = false;
        while (!conv && it < max_iters) {
            ++it;
            ++tag;
            ++rtag;
            const T* cur = P.buf + 3 * p * P.nsite;
            p ^= 1;
            b = P.buf + 3 * p * P.nsite;
            double d2 = 0;
            if (P.own) {
                const V3<T> d = rhs_det(h, res_field<T, CH, kIso, false>(C, P, cur, h), dt, lambda);
                const V3<T> o = {s.x + d.x, s.y + d.y, s.z + d.z};
                h = normalize_dipole(V3<T>{(s.x + o.x) / 2, (s.y + o.y) / 2, (s.z + o.z) / 2}, kap);
                if (P.w.nhalo) res_publish(A, P, tag, h);
                lds_put(b, P.nsite, P.t, h);
                const double ex = (double)prev.x - (double)o.x, ey = (double)prev.y - (double)o.y,
                             ez = (double)prev.z - (double)o.z;
                d2 = ex * ex + ey * ey + ez * ez;
                prev = o;
            }
            if (P.t < P.w.nlane) {
                d2 = wave_sum(d2);
                if ((P.t & 63) == 0) {
                    if (parts)
                        ll_put(A.res + (size_t)(rtag & 1) * 2 * A.nres + P.w.res0 + (P.t >> 6), A.nres, d2, rtag);
                    else
                        red[p][P.t >> 6] = d2;
                }
            }
            res_halo(A, P, tag, b);
            if (parts) res_residual(A, P, rtag, &red[p][0]);
            __syncthreads();
            double tot = red[p][0];
            if (!parts)
                for (int k = 1; k < nwave; k++) tot += red[p][k];
            conv = tot <= a2 && !isnan(tot);  // uniform over the replica's parts
        }
        if (!conv) {
            failed = n;
            break;
        }
        if (P.own) s = normalize_dipole(prev, kap);
        p ^= 1;  // the last iteration's copy may still be read
    }
    if (P.own) {
        store3_images(X, C.total, P.sc, C.G, s);
        if (Sdd) store3(Sdd, C.total, P.sc.g, prev);
    }
    if (P.w.first && P.t == 0) {
        iters_out[P.w.r] = it;
        if (failed >= 0) fail_step[P.w.r] = failed;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Plan

bool plan_resident(int na, const std::vector<std::array<int, 3>>& dims, const std::vector<int>& bstart,
                   const std::vector<std::array<int, 4>>& slots, size_t elem, size_t lds_max, ResPlan& out)
{
    out = ResPlan{};
    out.uni = na == 1;
    for (int i = 0; i < na; i++) out.nslot = std::max(out.nslot, bstart[i + 1] - bstart[i]);
    struct ClassPlan {
        int nwg = 0, nres = 0, lane0 = 0;
        std::vector<ResWg> wg;
    };
    std::map<std::array<int, 3>, ClassPlan> cls;
    for (size_t r = 0; r < dims.size(); r++) {
        const auto& L = dims[r];
        const long long ncell = (long long)L[0] * L[1] * L[2], ns = ncell * na;
        if (ns > kResMaxSites) return false;
        auto found = cls.find(L);
        if (found == cls.end()) {
            ClassPlan K;
            // lanes: one part, or parts of at most 64 sites from boxes of cells
            std::vector<std::vector<int>> part;  // entries cell * na + sublattice
            if (ns <= kResOneWg) {
                part.emplace_back();
                for (long long c = 0; c < ncell; c++)
                    for (int i = 0; i < na; i++) part[0].push_back((int)(c * na + i));
            } else {
                // the box with the fewest parts, then the smallest surface
                const int most = std::max(1, 64 / na);
                int box[3] = {1, 1, 1};
                double best = 1e300;
                for (int a = 1; a <= std::min(L[0], most); a++)
                    for (int b = 1; a * b <= most && b <= L[1]; b++)
                        for (int c = 1; a * b * c <= most && c <= L[2]; c++) {
                            const double n = (double)((L[0] + a - 1) / a) * ((L[1] + b - 1) / b) * ((L[2] + c - 1) / c);
                            const double cost = n * (1e3 + a * b + b * c + c * a);
                            if (cost < best) {
                                best = cost;
                                box[0] = a, box[1] = b, box[2] = c;
                            }
                        }
                for (int z = 0; z < L[2]; z += box[2])
                    for (int y = 0; y < L[1]; y += box[1])
                        for (int x = 0; x < L[0]; x += box[0]) {
                            std::vector<int> v;
                            for (int c3 = z; c3 < std::min(z + box[2], L[2]); c3++)
                                for (int c2 = y; c2 < std::min(y + box[1], L[1]); c2++)
                                    for (int c1 = x; c1 < std::min(x + box[0], L[0]); c1++)
                                        for (int i = 0; i < na; i++)
                                            v.push_back((c1 + L[0] * (c2 + L[1] * c3)) * na + i);
                            for (size_t k = 0; k < v.size(); k += 64)
                                part.emplace_back(v.begin() + k, v.begin() + std::min(v.size(), k + 64));
                        }
            }
            K.nwg = (int)part.size();
            // exchange position (within the replica) of every site
            std::vector<int> at(ns), who(ns);
            int ex = 0;
            K.lane0 = (int)out.lane.size();
            for (size_t p = 0; p < part.size(); p++) {
                ResWg w{};
                w.nlane = ((int)part[p].size() + 63) / 64 * 64;
                w.lane0 = K.lane0 + ex;
                w.ex0 = ex;
                w.res0 = K.nres;
                w.first = p == 0;
                K.nres += w.nlane / 64;
                for (size_t k = 0; k < part[p].size(); k++) {
                    at[part[p][k]] = ex + (int)k;
                    who[part[p][k]] = (int)p;
                    out.lane.push_back(part[p][k]);
                }
                out.lane.resize(out.lane.size() + w.nlane - part[p].size(), -1);
                ex += w.nlane;
                K.wg.push_back(w);
            }
            std::vector<std::array<int, 3>> fwd(slots.size());  // bond offsets wrapped to 0..L-1
            for (size_t q = 0; q < slots.size(); q++)
                for (int a = 0; a < 3; a++) fwd[q][a] = (slots[q][a] % L[a] + L[a]) % L[a];
            std::vector<int> near;  // bonded sites of the part's entries, slot after slot
            // the exchange needs every bond to have its reverse
            for (int i = 0; i < na && part.size() > 1; i++)
                for (int q = bstart[i]; q < bstart[i + 1]; q++) {
                    const int j = slots[q][3];
                    bool back = false;
                    for (int k = bstart[j]; k < bstart[j + 1] && !back; k++) {
                        back = slots[k][3] == i;
                        for (int a = 0; a < 3; a++) back = back && (slots[q][a] + slots[k][a]) % L[a] == 0;
                    }
                    if (!back) return false;
                }
            std::vector<int> halo, order(ex, -1);  // exchange position -> order in the halo
            for (size_t p = 0; p < part.size(); p++) {
                ResWg& w = K.wg[p];
                halo.clear();
                near.clear();
                for (int e : part[p]) {
                    const int i = e % na, c = e / na, c12 = c / L[0], x1 = c % L[0], x2 = c12 % L[1], x3 = c12 / L[1];
                    for (int q = bstart[i]; q < bstart[i + 1]; q++) {
                        int y1 = x1 + fwd[q][0], y2 = x2 + fwd[q][1], y3 = x3 + fwd[q][2];
                        y1 -= y1 >= L[0] ? L[0] : 0, y2 -= y2 >= L[1] ? L[1] : 0, y3 -= y3 >= L[2] ? L[2] : 0;
                        const int f = (y1 + L[0] * (y2 + L[1] * y3)) * na + slots[q][3];
                        near.push_back(f);
                        if (who[f] == (int)p || order[at[f]] >= 0) continue;
                        order[at[f]] = 0;
                        halo.push_back(at[f]);
                    }
                }
                std::sort(halo.begin(), halo.end());  // neighbouring lanes read neighbouring words
                w.halo0 = (int)out.halo.size();
                w.nhalo = (int)halo.size();
                for (int h = 0; h < w.nhalo; h++) order[halo[h]] = h;
                out.halo.insert(out.halo.end(), halo.begin(), halo.end());
                w.nbr0 = (int)out.nbr.size();
                if (w.nlane + w.nhalo > 65535) return false;
                out.nbr.resize(out.nbr.size() + (size_t)out.nslot * w.nlane, 0);
                const int* nf = near.data();
                for (size_t k = 0; k < part[p].size(); k++) {
                    const int i = part[p][k] % na;
                    for (int q = bstart[i]; q < bstart[i + 1]; q++) {
                        const int f = *nf++;
                        out.nbr[w.nbr0 + (size_t)(q - bstart[i]) * w.nlane + k] =
                            (unsigned short)(who[f] == (int)p ? at[f] - w.ex0 : w.nlane + order[at[f]]);
                    }
                }
                for (int x : halo) order[x] = -1;
                const size_t lds = ((size_t)6 * elem * (w.nlane + w.nhalo) + 2 * (size_t)out.nslot * w.nlane + 15) / 16 * 16;
                if (lds > lds_max) return false;
                out.lds = std::max(out.lds, lds);
                out.threads = std::max(out.threads, part.size() > 1 ? kResThreads : w.nlane);
            }
            found = cls.emplace(L, std::move(K)).first;
        }
        const ClassPlan& K = found->second;
        const int exr = out.nex, resr = out.nres;
        for (ResWg w : K.wg) {
            w.r = (int)r;
            w.laner = K.lane0;
            w.exr = exr;
            w.ex0 += exr;
            w.resr = resr;
            w.res0 += resr;
            w.nresr = K.nwg > 1 ? K.nres : 0;
            out.wg.push_back(w);
            out.nex += w.nlane;
        }
        out.nres += K.nres;
        out.shared |= K.nwg > 1;
    }
    return true;
}

// ---------------------------------------------------------------------------
// Launchers

namespace {

// Clears the words of a launch's rounds (no round is number 0) and its
// iteration and failure reports.
__global__ void k_res_clear(unsigned long long* __restrict__ w, size_t n, int* __restrict__ iters,
                            int* __restrict__ fail, int R)
{
    const size_t k0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    for (size_t k = k0; k < n; k += step) w[k] = 0;
    for (size_t k = k0; k < (size_t)R; k += step) {
        iters[k] = 0;
        fail[k] = -1;
    }
}

template <typename T, bool kLangevin, int CH, bool kIso, bool kUni>
hipError_t launch_res(const ResPlan& P, void** args, hipStream_t st)
{
    const void* fn;
    if (kLangevin)
        fn = P.threads <= kResThreads ? reinterpret_cast<const void*>(&k_res_langevin<T, CH, kIso, kUni, kResThreads>)
                                      : reinterpret_cast<const void*>(&k_res_langevin<T, CH, kIso, kUni, kResOneWg>);
    else
        fn = P.threads <= kResThreads ? reinterpret_cast<const void*>(&k_res_midpoint<T, CH, kIso, kUni, kResThreads>)
                                      : reinterpret_cast<const void*>(&k_res_midpoint<T, CH, kIso, kUni, kResOneWg>);
    allow_dynamic_lds(fn, P.lds);
    // parts that wait for each other must all be resident
    if (P.shared)
        return hipLaunchCooperativeKernel(fn, dim3((unsigned)P.wg.size()), dim3(P.threads), args, (unsigned)P.lds, st);
    return hipLaunchKernel(fn, dim3((unsigned)P.wg.size()), dim3(P.threads), args, P.lds, st);
}

template <typename T, bool kLangevin>
hipError_t launch_res_forms(const Couplings<T>& C, const ResPlan& P, void** args, hipStream_t st)
{
#define SNH_RES(CH)                                                                                    \
    (C.iso ? (P.uni ? launch_res<T, kLangevin, CH, true, true>(P, args, st)                            \
                    : launch_res<T, kLangevin, CH, true, false>(P, args, st))                          \
           : (P.uni ? launch_res<T, kLangevin, CH, false, true>(P, args, st)                           \
                    : launch_res<T, kLangevin, CH, false, false>(P, args, st)))
    return C.chunk == 9 ? SNH_RES(9) : SNH_RES(6);  // every bond list is a multiple of chunk (6, 9 or 18)
#undef SNH_RES
}

}  // namespace

size_t res_words(const ResPlan& P, size_t elem)
{
    return P.shared ? 2 * ((elem == 8 ? 6 : 3) * (size_t)P.nex + 2 * (size_t)P.nres) : 0;
}

void launch_res_clear(unsigned long long* words, size_t n, int* iters, int* fail, int R, hipStream_t st)
{
    const size_t k = std::max<size_t>(n, (size_t)R);
    hipLaunchKernelGGL(k_res_clear, dim3((unsigned)std::min<size_t>((k + 255) / 256, 256)), dim3(256), 0, st, words, n,
                       iters, fail, R);
}

template <typename T>
hipError_t launch_res_langevin(const Couplings<T>& C, const ResPlan& P, const ResArgs& A, T* X, T* keep,
                               const NoiseArgs<T>& nz, T dt, T lambda, int nsteps, hipStream_t st)
{
    Couplings<T> c = C;
    ResArgs a = A;
    NoiseArgs<T> z = nz;
    void* args[] = {&c, &a, &X, &keep, &z, &dt, &lambda, &nsteps};
    return launch_res_forms<T, true>(C, P, args, st);
}

template <typename T>
hipError_t launch_res_midpoint(const Couplings<T>& C, const ResPlan& P, const ResArgs& A, T* X, T* keep, T dt, T lambda,
                               const double* atol2, int max_iters, int nsteps, int* iters_out, int* fail_step,
                               T* Sdd, hipStream_t st)
{
    Couplings<T> c = C;
    ResArgs a = A;
    void* args[] = {&c, &a, &X, &keep, &dt, &lambda, &atol2, &max_iters, &nsteps, &iters_out, &fail_step, &Sdd};
    return launch_res_forms<T, false>(C, P, args, st);
}

#define SNH_INST(T)                                                                                             \
    template hipError_t launch_res_langevin<T>(const Couplings<T>&, const ResPlan&, const ResArgs&, T*, T*,     \
                                               const NoiseArgs<T>&, T, T, int, hipStream_t);                    \
    template hipError_t launch_res_midpoint<T>(const Couplings<T>&, const ResPlan&, const ResArgs&, T*, T*, T,  \
                                               T, const double*, int, int, int*, int*, T*, hipStream_t);
SNH_INST(float)
SNH_INST(double)

}  // namespace snh
