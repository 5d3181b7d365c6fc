// State readout and upload between the device's planes and the host's
// site-major arrays (snh_state.hip).
#pragma once
#include "snh_internal.h"

namespace snh {

// Interior sites in host order (replica after replica, cell + ncell * sublattice)
// and where each lives in the planes.
struct StateMap {
    const ReplicaInfo* reps;
    const long long* rsite;  // [R+1] first host site of every replica
    int R;
    uint32_t total;
    Ghost G;
};

// Values e0 .. e0 + n - 1 of the host array [site][np], packed to out.
template <typename T>
void launch_state_pack(const StateMap& M, const T* P, int np, long long e0, long long n, T* out, hipStream_t st);
// Sites s0 .. s0 + n - 1 from in ([site][np]) into the planes and their ghost images.
template <typename T>
void launch_state_unpack(const StateMap& M, const T* in, int np, long long s0, long long n, T* P, hipStream_t st);
// Expected spins of the kets of sites s0 .. s0 + n - 1, computed in FP64: out [site][3].
template <typename T>
void launch_state_spin(const StateMap& M, const T* Z, int N, long long s0, long long n, double* out, hipStream_t st);
// Values d0 .. d0 + n - 1 (complex) of the correlations in the caller's order
// [w][q][j][i][c] (c fastest) from data [c][i][w][j][q].
void launch_corr_pack(const void* data, int nc, int na, int nt, long long ncell, long long d0, long long n, void* out,
                      hipStream_t st);

}  // namespace snh
