// Readout and upload of states: the planes of the device against the host's
// [site][component] doubles.
//
// Reference semantics: sys.dipoles, sys.coherents (src/System/Types.jl:
// 133-134), expected_spin (src/Operators/Spin.jl:72-87), sc.data
// (src/SampledCorrelations/SampledCorrelations.jl:3).
//
// The reordering runs here, a chunk at a time, so that a transfer is a
// packed copy through pinned memory, and the host's only pass over a chunk
// (widening to doubles) overlaps the next one's copy.  It bounds a transfer
// at the rate of that pass: 4.2 million FP32 dipoles read into their eight
// systems 28 -> 6.8 ms (a host loop over padded planes from a pageable copy
// before).  A packed word per
// thread keeps the stores coalesced; the three planes' reads of one site run
// are shared through the cache.
#include "snh_state.h"

namespace snh {

namespace {

constexpr int kStateThreads = 256;

// Site s of the host order.
__device__ __forceinline__ SiteCoord state_site(const StateMap& M, long long s)
{
    int lo = 0, hi = M.R;  // rsite[lo] <= s < rsite[hi]
    while (hi - lo > 1) {
        const int m = (lo + hi) >> 1;
        if (s >= M.rsite[m]) lo = m; else hi = m;
    }
    SiteCoord sc;
    sc.blk = 0;
    sc.r = lo;
    sc.R = M.reps[lo];
    const uint32_t k = (uint32_t)(s - M.rsite[lo]);
    sc.i = (int)(k / (uint32_t)sc.R.ncell);
    sc.c = (int)(k - (uint32_t)sc.i * (uint32_t)sc.R.ncell);
    const int q = fdiv(sc.c, sc.R.L1, sc.R.inv1);
    sc.c1 = sc.c - q * sc.R.L1;
    sc.c3 = fdiv(q, sc.R.L2, sc.R.inv2);
    sc.c2 = q - sc.c3 * sc.R.L2;
    sc.g = sc.R.off + (uint32_t)((sc.c1 + M.G.w1) + sc.R.P1 * ((sc.c2 + M.G.w2) + sc.R.P2 * (sc.c3 + M.G.w3))) +
           sc.R.pcell * (uint32_t)sc.i;
    sc.edge = (sc.c1 < M.G.w1) | (sc.c1 >= sc.R.L1 - M.G.w1) | (sc.c2 < M.G.w2) | (sc.c2 >= sc.R.L2 - M.G.w2) |
              (sc.c3 < M.G.w3) | (sc.c3 >= sc.R.L3 - M.G.w3);
    sc.valid = true;
    return sc;
}

template <typename T>
__global__ __launch_bounds__(kStateThreads) void k_state_pack(StateMap M, const T* __restrict__ P, int np,
                                                              long long e0, long long n, T* __restrict__ out)
{
    const long long k = (long long)blockIdx.x * kStateThreads + threadIdx.x;
    if (k >= n) return;
    const long long s = (e0 + k) / np;
    const int p = (int)(e0 + k - s * np);
    out[k] = ldg(P + (size_t)p * M.total, state_site(M, s).g);
}

template <typename T>
__global__ __launch_bounds__(kStateThreads) void k_state_unpack(StateMap M, const T* __restrict__ in, int np,
                                                                long long s0, long long n, T* __restrict__ P)
{
    const long long k = (long long)blockIdx.x * kStateThreads + threadIdx.x;
    if (k >= n) return;
    const SiteCoord sc = state_site(M, s0 + k);
    for (int p = 0; p < np; p++) {
        const T v = in[k * np + p];
        T* const plane = P + (size_t)p * M.total;
        stg(plane, sc.g, v);
        for_each_ghost(sc, M.G, [&](uint32_t g) { stg(plane, g, v); });
    }
}

// expected_spin: (2 Re c, 2 Im c, sum m_k |Z_k|^2), c = sum conj(Z_k) off_k Z_{k+1}
template <typename T>
__global__ __launch_bounds__(kStateThreads) void k_state_spin(StateMap M, const T* __restrict__ Z, int N,
                                                              long long s0, long long n, double* __restrict__ out)
{
    const long long k = (long long)blockIdx.x * kStateThreads + threadIdx.x;
    if (k >= n) return;
    const uint32_t g = state_site(M, s0 + k).g;
    double cr = 0, ci = 0, nz = 0, ar = 0, ai = 0;  // a: component a - 1
    const double s = (N - 1) / 2.0;
    for (int a = 0; a < N; a++) {
        const double zr = ldg(Z + (size_t)(2 * a) * M.total, g), zi = ldg(Z + (size_t)(2 * a + 1) * M.total, g);
        if (a > 0) {
            const double off = sqrt(2 * (s + 1) * a - (double)a * (a + 1)) / 2;
            cr += off * (ar * zr + ai * zi);
            ci += off * (ar * zi - ai * zr);
        }
        nz += (s - a) * (zr * zr + zi * zi);
        ar = zr;
        ai = zi;
    }
    out[3 * k] = 2 * cr;
    out[3 * k + 1] = 2 * ci;
    out[3 * k + 2] = nz;
}

__global__ __launch_bounds__(kStateThreads) void k_corr_pack(const double2* __restrict__ data, int nc, int na, int nt,
                                                             long long ncell, long long d0, long long n,
                                                             double2* __restrict__ out)
{
    const long long k = (long long)blockIdx.x * kStateThreads + threadIdx.x;
    if (k >= n) return;
    long long d = d0 + k;
    const int c = (int)(d % nc);
    d /= nc;
    const int i = (int)(d % na);
    d /= na;
    const int j = (int)(d % na);
    d /= na;
    const long long q = d % ncell, w = d / ncell;
    out[k] = data[((((long long)c * na + i) * nt + w) * na + j) * ncell + q];
}

dim3 blocks_of(long long n) { return dim3((unsigned)((n + kStateThreads - 1) / kStateThreads)); }

}  // namespace

template <typename T>
void launch_state_pack(const StateMap& M, const T* P, int np, long long e0, long long n, T* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_state_pack<T>, blocks_of(n), dim3(kStateThreads), 0, st, M, P, np, e0, n, out);
}

template <typename T>
void launch_state_unpack(const StateMap& M, const T* in, int np, long long s0, long long n, T* P, hipStream_t st)
{
    hipLaunchKernelGGL(k_state_unpack<T>, blocks_of(n), dim3(kStateThreads), 0, st, M, in, np, s0, n, P);
}

template <typename T>
void launch_state_spin(const StateMap& M, const T* Z, int N, long long s0, long long n, double* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_state_spin<T>, blocks_of(n), dim3(kStateThreads), 0, st, M, Z, N, s0, n, out);
}

void launch_corr_pack(const void* data, int nc, int na, int nt, long long ncell, long long d0, long long n, void* out,
                      hipStream_t st)
{
    hipLaunchKernelGGL(k_corr_pack, blocks_of(n), dim3(kStateThreads), 0, st, static_cast<const double2*>(data), nc,
                       na, nt, ncell, d0, n, static_cast<double2*>(out));
}

#define SNH_INST(T)                                                                                              \
    template void launch_state_pack<T>(const StateMap&, const T*, int, long long, long long, T*, hipStream_t);   \
    template void launch_state_unpack<T>(const StateMap&, const T*, int, long long, long long, T*, hipStream_t); \
    template void launch_state_spin<T>(const StateMap&, const T*, int, long long, long long, double*, hipStream_t);
SNH_INST(float)
SNH_INST(double)

}  // namespace snh
