// :dipole-mode kernels: local field by bond-stencil gather, fused stochastic
// Heun stages, spherical-midpoint sweeps, FP64 energy.
//
// Reference semantics (Sunny.jl 0.9.2):
//   set_energy_grad_dipoles!  src/System/Interactions.jl:516-592
//   rhs_dipole!               src/Integrators.jl:266-275
//   fill_noise!               src/Integrators.jl:288-298
//   step!(::System{0}, ::Langevin)          src/Integrators.jl:313-332
//   step!(::System{0}, ::ImplicitMidpoint)  src/Integrators.jl:379-413
//   energy / energy_aux       src/System/Interactions.jl:401-508
//
// The reference scatters each non-culled bond into both ends (J*Sj to i,
// J'*Si to j).  Here every directed bond (i -> j, J) and its reverse
// (j -> i, J') is in the table and each site gathers over its own bonds: no
// write conflicts, one coalesced load per neighbour plane.
//
// Heun in two kernels with two gathers per step.  The corrector's update
//   S + (dS1 + dS2)/2,  dS2 = -S' x xi  -  S' x (dt g' - dt lambda S' x g')
// is linear in the noise term, so the predictor, which knows S' and xi,
// stores H = S + dS1/2 - (S' x xi)/2 and the corrector only gathers S'.
#include "snh_gather.h"

namespace snh {

// ---------------------------------------------------------------------------
// Kernels

// Heun predictor at one site: dS1 = rhs(S, xi, dE(S)); S' = kappa*normalize(S + dS1);
// H = S + dS1/2 - (S' x xi)/2.
template <typename T, int CH, bool kIso>
__device__ __forceinline__ void dipole_predict_site(const Couplings<T>& C, const SiteCoord& sc,
                                                    const T* __restrict__ S, T* __restrict__ Sp, T* __restrict__ H,
                                                    const T* __restrict__ phi, const NoiseArgs<T>& nz, T dt,
                                                    T lambda)
{
    const Planes<T> Sv = planes(S, C.total);
    const SpinSrc<T, false> src{Sv, Sv};
    const V3<T> s = Sv(sc.g);
    const V3<T> g = local_field<T, CH, false, kIso>(C, sc, src, s, phi);
    const bool noisy = lambda != (T)0;
    const V3<T> xi = noisy ? dipole_noise(nz, sc.r, (uint32_t)(sc.c + sc.R.ncell * sc.i), sc.g) : V3<T>{0, 0, 0};
    V3<T> sp, h;
    heun_predict(s, g, xi, noisy, C.kappa[sc.i], dt, lambda, sp, h);
    store3_images(Sp, C.total, sc, C.G, sp);
    store3(H, C.total, sc.g, h);
}

template <typename T, int CH, bool kIso>
__global__ __launch_bounds__(kBlock) void k_dipole_predict(Couplings<T> C, const T* __restrict__ S,
                                                           T* __restrict__ Sp, T* __restrict__ H,
                                                           const T* __restrict__ phi, NoiseArgs<T> nz, T dt,
                                                           T lambda)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    if (sc.valid) dipole_predict_site<T, CH, kIso>(C, sc, S, Sp, H, phi, nz, dt, lambda);
}

// Heun corrector at one site: S <- kappa*normalize(H + rhs_det(S', dE(S'))/2).
template <typename T, int CH, bool kIso>
__device__ __forceinline__ void dipole_correct_site(const Couplings<T>& C, const SiteCoord& sc,
                                                    const T* __restrict__ Sp, const T* __restrict__ H,
                                                    T* __restrict__ Sout, const T* __restrict__ phi, T dt, T lambda)
{
    const Planes<T> Pv = planes(Sp, C.total);
    const SpinSrc<T, false> src{Pv, Pv};
    const V3<T> sp = Pv(sc.g);
    const V3<T> d = rhs_det(sp, local_field<T, CH, false, kIso>(C, sc, src, sp, phi), dt, lambda);
    const V3<T> h = planes(H, C.total)(sc.g);
    store3_images(Sout, C.total, sc, C.G,
                  normalize_dipole(V3<T>{h.x + d.x / 2, h.y + d.y / 2, h.z + d.z / 2}, C.kappa[sc.i]));
}

template <typename T, int CH, bool kIso>
__global__ __launch_bounds__(kBlock) void k_dipole_correct(Couplings<T> C, const T* __restrict__ Sp,
                                                           const T* __restrict__ H, T* __restrict__ Sout,
                                                           const T* __restrict__ phi, T dt, T lambda)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    if (sc.valid) dipole_correct_site<T, CH, kIso>(C, sc, Sp, H, Sout, phi, dt, lambda);
}

// Materialised midpoint Shat (when a global term, Ewald, needs it).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dipole_mid_hat(Couplings<T> C, const T* __restrict__ S,
                                                           const T* __restrict__ S1, T* __restrict__ Shat,
                                                           const int* __restrict__ conv_iter)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    if (!sc.valid || conv_iter[sc.r] != 0) return;
    const SpinSrc<T, true> src{planes(S, C.total), planes(S1, C.total)};
    store3_images(Shat, C.total, sc, C.G, src.get(sc.g, C.kappa[sc.i]));
}

// One fixed-point sweep at one site with Shat given (gathered with its
// images): S2 = S + rhs(Shat) at the site, the next iteration's Shat =
// kappa*normalize((S + S2)/2) with images when hat_out is non-null (S2 then
// has no images); returns |S1 - S2|^2 in FP64.
template <typename T, int CH>
__device__ __forceinline__ double dipole_mid_sweep_site(const Couplings<T>& C, const SiteCoord& sc, const T* S,
                                                        const T* S1, T* S2, const T* Shat, const T* phi, T dt,
                                                        T lambda, T* hat_out)
{
    const Planes<T> Hv = planes(Shat, C.total);
    const SpinSrc<T, false> src{Hv, Hv};
    const V3<T> h = Hv(sc.g);
    const V3<T> g = local_field<T, CH>(C, sc, src, h, phi);
    const V3<T> d = rhs_det(h, g, dt, lambda);
    const V3<T> s = planes(S, C.total)(sc.g);
    const V3<T> o = {s.x + d.x, s.y + d.y, s.z + d.z};
    if (hat_out) {
        store3(S2, C.total, sc.g, o);
        store3_images(hat_out, C.total, sc, C.G,
                      normalize_dipole(V3<T>{(s.x + o.x) / 2, (s.y + o.y) / 2, (s.z + o.z) / 2}, ldc(C.kappa, sc.i)));
    } else {
        store3_images(S2, C.total, sc, C.G, o);
    }
    const V3<T> p = planes(S1, C.total)(sc.g);
    const double ex = (double)p.x - (double)o.x, ey = (double)p.y - (double)o.y, ez = (double)p.z - (double)o.z;
    return ex * ex + ey * ey + ez * ez;
}

// One fixed-point sweep of the spherical midpoint method:
//   Shat = kappa*normalize((S + S1)/2);  S2 = S + rhs(Shat, 0, dE(Shat)),
// plus the FP64 residual sum |S1 - S2|^2 per block (fast_isapprox).
// hat_out non-null (with kHatGiven): the next iteration's Shat =
// kappa*normalize((S + S2)/2) is written with its ghost images, and S2 is
// only read at its own site afterwards (no images).
template <typename T, int CH, bool kHatGiven>
__global__ __launch_bounds__(kBlock) void k_dipole_mid_iter(Couplings<T> C, const T* __restrict__ S,
                                                            const T* __restrict__ S1, T* __restrict__ S2,
                                                            const T* __restrict__ Shat, const T* __restrict__ phi,
                                                            T dt, T lambda, double* __restrict__ partial,
                                                            const int* __restrict__ conv_iter,
                                                            T* __restrict__ hat_out)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    if (conv_iter[sc.r] != 0) return;  // block-uniform: the whole block belongs to replica r
    double d2 = 0;
    if (sc.valid && kHatGiven) {
        d2 = dipole_mid_sweep_site<T, CH>(C, sc, S, S1, S2, Shat, phi, dt, lambda, hat_out);
    } else if (sc.valid) {
        const SpinSrc<T, true> src{planes(S, C.total), planes(S1, C.total)};
        const V3<T> h = src.get(sc.g, C.kappa[sc.i]);
        const V3<T> g = local_field<T, CH>(C, sc, src, h, phi);
        const V3<T> d = rhs_det(h, g, dt, lambda);
        const V3<T> s = planes(S, C.total)(sc.g);
        const V3<T> o = {s.x + d.x, s.y + d.y, s.z + d.z};
        store3_images(S2, C.total, sc, C.G, o);
        const V3<T> p = planes(S1, C.total)(sc.g);
        const double ex = (double)p.x - (double)o.x, ey = (double)p.y - (double)o.y, ez = (double)p.z - (double)o.z;
        d2 = ex * ex + ey * ey + ez * ez;
    }
    const double t = block_sum(d2);
    if (threadIdx.x == 0) partial[sc.blk] = t;
}

// S = kappa*normalize(S'') for replicas that converged at iteration `iter`;
// S'' of iteration m lives in Sa when m is odd, Sb when m is even.  With
// hat_next non-null the first Shat of the next step, kappa*normalize((S +
// S)/2) as k_dipole_mid_hat forms it, is written too (with images).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dipole_mid_finalize(Couplings<T> C, T* __restrict__ S,
                                                                const T* __restrict__ Sa, const T* __restrict__ Sb,
                                                                const int* __restrict__ conv_iter, int iter,
                                                                T* __restrict__ hat_next)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    const int c = sc.valid ? conv_iter[sc.r] : 0;  // iter 0: every converged replica
    if (c == 0 || (iter != 0 && c != iter)) return;
    const T* src = (c & 1) ? Sa : Sb;
    const T kap = C.kappa[sc.i];
    const V3<T> s = normalize_dipole(planes(src, C.total)(sc.g), kap);
    store3_images(S, C.total, sc, C.G, s);
    if (hat_next)
        store3_images(hat_next, C.total, sc, C.G,
                      normalize_dipole(V3<T>{(s.x + s.x) / 2, (s.y + s.y) / 2, (s.z + s.z) / 2}, kap));
}

// The same for the tiled sweep's implicit iterates: S'' of iteration m is
// 2 mu_m Shat_{m+1} - S, with Shat_{m+1} in Ho (m odd) or He (m even) and
// mu_m in Mo or Me (every converged replica).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dipole_mid_finalize_mu(Couplings<T> C, T* __restrict__ S, const T* Ho,
                                                                   const T* He, const T* __restrict__ Mo,
                                                                   const T* __restrict__ Me,
                                                                   const int* __restrict__ conv_iter, T* hat_next)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    const int c = sc.valid ? conv_iter[sc.r] : 0;
    if (c == 0) return;
    const V3<T> h = planes((c & 1) ? Ho : He, C.total)(sc.g);
    const T t = 2 * ldg((c & 1) ? Mo : Me, sc.g);
    const V3<T> s0 = planes(S, C.total)(sc.g);
    const T kap = C.kappa[sc.i];
    const V3<T> s = normalize_dipole(V3<T>{t * h.x - s0.x, t * h.y - s0.y, t * h.z - s0.z}, kap);
    store3_images(S, C.total, sc, C.G, s);
    if (hat_next)  // may be the buffer h came from: each site reads its own entry first
        store3_images(hat_next, C.total, sc, C.G,
                      normalize_dipole(V3<T>{(s.x + s.x) / 2, (s.y + s.y) / 2, (s.z + s.z) / 2}, kap));
}

template <typename T, int CH>
__global__ __launch_bounds__(kBlock) void k_dipole_grad(Couplings<T> C, const T* __restrict__ S,
                                                        const T* __restrict__ phi, T* __restrict__ dE)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    if (!sc.valid) return;
    const Planes<T> Sv = planes(S, C.total);
    const SpinSrc<T, false> src{Sv, Sv};
    store3(dE, C.total, sc.g, local_field<T, CH>(C, sc, src, Sv(sc.g), phi));
}

// energy_aux over non-culled bonds, Zeeman, anisotropy, Ewald (1/2 mu.phi).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dipole_energy(Couplings<T> C, const T* __restrict__ S,
                                                          const T* __restrict__ phi, double* __restrict__ partial)
{
    const SiteCoord sc = site_coord(C.blocks, C.reps, C.G);
    double e = 0;
    if (sc.valid) {
        const int i = sc.i;
        const Planes<T> Sv = planes(S, C.total);
        const V3<T> s = Sv(sc.g);
        const T* gm = C.gmat + 9 * i;
        const T* B = C.field + 3 * i;
        for (int a = 0; a < 3; a++)
            e += (double)B[a] * ((double)gm[3 * a] * s.x + (double)gm[3 * a + 1] * s.y + (double)gm[3 * a + 2] * s.z);
        T ea, gx = 0, gy = 0, gz = 0;
        stevens_grad<T>(s.x, s.y, s.z, C.stev + 28 * i, C.kmax[i], gx, gy, gz, &ea);
        e += (double)ea;
        const int* __restrict__ dl = C.bdelta + sc.R.dcls * C.nb;
        for (int b = C.bstart[i]; b < C.bstart[i + 1]; b++) {
            const int fl = C.bflag[b];
            if (fl & kBondCulled) continue;
            const V3<T> sj = Sv(sc.g + (uint32_t)dl[b]);
            const T* J = C.bJ + 9 * b;
            double v = (double)C.bscalar[b];
            v += (double)s.x * ((double)J[0] * sj.x + (double)J[1] * sj.y + (double)J[2] * sj.z);
            v += (double)s.y * ((double)J[3] * sj.x + (double)J[4] * sj.y + (double)J[5] * sj.z);
            v += (double)s.z * ((double)J[6] * sj.x + (double)J[7] * sj.y + (double)J[8] * sj.z);
            if (fl & kBondBiquad) {
                T Qi[5], Qj[5];
                quadrupole(s, Qi);
                quadrupole(sj, Qj);
                const T* Bq = C.bQ + 25 * b;
                for (int p = 0; p < 5; p++)
                    for (int q = 0; q < 5; q++) v += (double)Qi[p] * (double)Bq[5 * p + q] * (double)Qj[q];
            }
            e += v;
        }
        if (phi) {  // 1/2 mu.phi with mu = -g S
            const V3<T> p = planes(phi, C.total)(sc.g);
            const double mx = -((double)gm[0] * s.x + (double)gm[1] * s.y + (double)gm[2] * s.z);
            const double my = -((double)gm[3] * s.x + (double)gm[4] * s.y + (double)gm[5] * s.z);
            const double mz = -((double)gm[6] * s.x + (double)gm[7] * s.y + (double)gm[8] * s.z);
            e += 0.5 * (mx * p.x + my * p.y + mz * p.z);
        }
    }
    const double t = block_sum(e);
    if (threadIdx.x == 0) partial[sc.blk] = t;
}

// One block per replica: out[r] = sum of partial[rblk[r] .. rblk[r+1]).
__global__ __launch_bounds__(kBlock) void k_reduce_partials(const double* __restrict__ partial,
                                                            const int* __restrict__ rblk, double* __restrict__ out)
{
    const int r = blockIdx.x;
    double v = 0;
    for (int k = rblk[r] + threadIdx.x; k < rblk[r + 1]; k += kBlock) v += partial[k];
    const double t = block_sum(v);
    if (threadIdx.x == 0) out[r] = t;
}

// fast_isapprox (Integrators.jl:361-371) per replica: converged when the sum is
// <= atol^2 and not NaN.  Records the iteration of convergence.
__global__ __launch_bounds__(kBlock) void k_midpoint_check(const double* __restrict__ partial,
                                                           const int* __restrict__ rblk,
                                                           const double* __restrict__ atol2,
                                                           int* __restrict__ conv_iter, int iter)
{
    const int r = blockIdx.x;
    if (conv_iter[r] != 0) return;  // uniform over the block
    double v = 0;
    for (int k = rblk[r] + threadIdx.x; k < rblk[r + 1]; k += kBlock) v += partial[k];
    const double t = block_sum(v);
    if (threadIdx.x == 0 && t <= atol2[r] && !isnan(t)) conv_iter[r] = iter;
}

// Plain streaming copy (float4 lanes) used to calibrate traffic counters.
__global__ __launch_bounds__(256) void k_copy_planes(const float4* __restrict__ src, float4* __restrict__ dst, size_t n)
{
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
        dst[k] = src[k];
}

void launch_copy_planes(const void* src, void* dst, size_t bytes, hipStream_t st)
{
    const size_t n = bytes / sizeof(float4);
    hipLaunchKernelGGL(k_copy_planes, dim3(4096), dim3(256), 0, st, reinterpret_cast<const float4*>(src),
                       reinterpret_cast<float4*>(dst), n);
}

__global__ void k_fill_int(int* __restrict__ p, int n, int v)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}

// After step s of a budgeted group: fail_step[r] = s for replicas that have
// not converged within the budget (the first such step), max_iter[r] = the
// largest iteration count of the group so far, last_it[r] = this step's
// count; conv_iter[r] is cleared for the next step.
__global__ void k_mid_budget(int* __restrict__ conv_iter, int* __restrict__ fail_step, int* __restrict__ max_iter,
                             int* __restrict__ last_it, int R, int s)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= R) return;
    const int c = conv_iter[r];
    if (c == 0 && fail_step[r] < 0) fail_step[r] = s;
    if (s == 0 || c > max_iter[r]) max_iter[r] = c;
    last_it[r] = c;
    conv_iter[r] = 0;
}

__global__ void k_step_set(unsigned long long* __restrict__ p, unsigned long long v)
{
    if (threadIdx.x == 0) p[0] = v;
}

__global__ void k_step_advance(unsigned long long* __restrict__ p)
{
    if (threadIdx.x == 0) p[0] += 1;
}

// ---------------------------------------------------------------------------
// Launchers

template <typename T>
void launch_dipole_predict(const Couplings<T>& C, int nblocks, const T* S, T* Sp, T* H, const T* phi,
                           const NoiseArgs<T>& nz, T dt, T lambda, hipStream_t st)
{
#define SNH_PRED(CH, ISO)                                                                                      \
    hipLaunchKernelGGL((k_dipole_predict<T, CH, ISO>), dim3(nblocks), dim3(kBlock), 0, st, C, S, Sp, H, phi, nz, dt, \
                       lambda)
    if (C.chunk == 18) {
        if (C.iso) SNH_PRED(18, true); else SNH_PRED(18, false);
    } else if (C.chunk == 9) {
        if (C.iso) SNH_PRED(9, true); else SNH_PRED(9, false);
    } else {
        if (C.iso) SNH_PRED(6, true); else SNH_PRED(6, false);
    }
#undef SNH_PRED
}

template <typename T>
void launch_dipole_correct(const Couplings<T>& C, int nblocks, const T* Sp, const T* H, T* Sout, const T* phi, T dt,
                           T lambda, hipStream_t st)
{
#define SNH_CORR(CH, ISO)                                                                                      \
    hipLaunchKernelGGL((k_dipole_correct<T, CH, ISO>), dim3(nblocks), dim3(kBlock), 0, st, C, Sp, H, Sout, phi, dt, \
                       lambda)
    if (C.chunk == 18) {
        if (C.iso) SNH_CORR(18, true); else SNH_CORR(18, false);
    } else if (C.chunk == 9) {
        if (C.iso) SNH_CORR(9, true); else SNH_CORR(9, false);
    } else {
        if (C.iso) SNH_CORR(6, true); else SNH_CORR(6, false);
    }
#undef SNH_CORR
}

template <typename T>
void launch_dipole_midpoint_hat(const Couplings<T>& C, int nblocks, const T* S, const T* S1, T* Shat,
                                const int* conv_iter, hipStream_t st)
{
    hipLaunchKernelGGL(k_dipole_mid_hat<T>, dim3(nblocks), dim3(kBlock), 0, st, C, S, S1, Shat, conv_iter);
}

template <typename T>
void launch_dipole_midpoint_iter(const Couplings<T>& C, int nblocks, const T* S, const T* S1, T* S2,
                                 const T* Shat, const T* phi, T dt, T lambda, double* partial, const int* conv_iter,
                                 T* hat_out, hipStream_t st)
{
    if (Shat)
        hipLaunchKernelGGL((k_dipole_mid_iter<T, 6, true>), dim3(nblocks), dim3(kBlock), 0, st, C, S, S1, S2, Shat,
                           phi, dt, lambda, partial, conv_iter, hat_out);
    else
        hipLaunchKernelGGL((k_dipole_mid_iter<T, 6, false>), dim3(nblocks), dim3(kBlock), 0, st, C, S, S1, S2, Shat,
                           phi, dt, lambda, partial, conv_iter, (T*)nullptr);
}

template <typename T>
void launch_dipole_midpoint_finalize(const Couplings<T>& C, int nblocks, T* S, const T* Sa, const T* Sb,
                                     const int* conv_iter, int iter, T* hat_next, hipStream_t st)
{
    hipLaunchKernelGGL(k_dipole_mid_finalize<T>, dim3(nblocks), dim3(kBlock), 0, st, C, S, Sa, Sb, conv_iter, iter,
                       hat_next);
}

template <typename T>
void launch_dipole_midpoint_finalize_mu(const Couplings<T>& C, int nblocks, T* S, const T* Ho, const T* He,
                                        const T* Mo, const T* Me, const int* conv_iter, T* hat_next, hipStream_t st)
{
    hipLaunchKernelGGL(k_dipole_mid_finalize_mu<T>, dim3(nblocks), dim3(kBlock), 0, st, C, S, Ho, He, Mo, Me,
                       conv_iter, hat_next);
}

template <typename T>
void launch_dipole_grad(const Couplings<T>& C, int nblocks, const T* S, const T* phi, T* dE, hipStream_t st)
{
    hipLaunchKernelGGL((k_dipole_grad<T, 6>), dim3(nblocks), dim3(kBlock), 0, st, C, S, phi, dE);
}

template <typename T>
void launch_dipole_energy(const Couplings<T>& C, int nblocks, const T* S, const T* phi, double* partial,
                          hipStream_t st)
{
    hipLaunchKernelGGL(k_dipole_energy<T>, dim3(nblocks), dim3(kBlock), 0, st, C, S, phi, partial);
}

void launch_reduce_partials(const double* partial, const int* rblk, int R, double* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_reduce_partials, dim3(R), dim3(kBlock), 0, st, partial, rblk, out);
}

void launch_midpoint_check(const double* partial, const int* rblk, int R, const double* atol2, int* conv_iter,
                           int iter, hipStream_t st)
{
    hipLaunchKernelGGL(k_midpoint_check, dim3(R), dim3(kBlock), 0, st, partial, rblk, atol2, conv_iter, iter);
}

void launch_fill_int(int* p, int n, int v, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_int, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
}

void launch_mid_budget(int* conv_iter, int* fail_step, int* max_iter, int* last_it, int R, int s, hipStream_t st)
{
    hipLaunchKernelGGL(k_mid_budget, dim3((R + 255) / 256), dim3(256), 0, st, conv_iter, fail_step, max_iter,
                       last_it, R, s);
}

void launch_step_set(unsigned long long* p, unsigned long long v, hipStream_t st)
{
    hipLaunchKernelGGL(k_step_set, dim3(1), dim3(64), 0, st, p, v);
}

void launch_step_advance(unsigned long long* p, hipStream_t st)
{
    hipLaunchKernelGGL(k_step_advance, dim3(1), dim3(64), 0, st, p);
}

#define SNH_INST(T)                                                                                              \
    template void launch_dipole_predict<T>(const Couplings<T>&, int, const T*, T*, T*, const T*,                \
                                           const NoiseArgs<T>&, T, T, hipStream_t);                             \
    template void launch_dipole_correct<T>(const Couplings<T>&, int, const T*, const T*, T*, const T*, T, T,     \
                                           hipStream_t);                                                         \
    template void launch_dipole_midpoint_hat<T>(const Couplings<T>&, int, const T*, const T*, T*, const int*,    \
                                                hipStream_t);                                                    \
    template void launch_dipole_midpoint_iter<T>(const Couplings<T>&, int, const T*, const T*, T*, const T*,     \
                                                 const T*, T, T, double*, const int*, T*, hipStream_t);                     \
    template void launch_dipole_midpoint_finalize_mu<T>(const Couplings<T>&, int, T*, const T*, const T*,        \
                                                        const T*, const T*, const int*, T*, hipStream_t);       \
    template void launch_dipole_midpoint_finalize<T>(const Couplings<T>&, int, T*, const T*, const T*,           \
                                                     const int*, int, T*, hipStream_t);                              \
    template void launch_dipole_grad<T>(const Couplings<T>&, int, const T*, const T*, T*, hipStream_t);          \
    template void launch_dipole_energy<T>(const Couplings<T>&, int, const T*, const T*, double*, hipStream_t);

SNH_INST(float)
SNH_INST(double)

}  // namespace snh
