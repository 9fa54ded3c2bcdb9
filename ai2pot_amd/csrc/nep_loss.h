// What the kernels of the NEP training loss share (nep_loss.hip: any shape; nep_loss_wave.hip: the common shapes).
#pragma once
#include "a2p_common.h"
#include "loss_kernels.h"

namespace a2p {
namespace nepdev {

template <typename T>
struct NepLossArgs {
    int K, n_r, n_a, l_max, H, ntypes, D;
    const T *coeffs, *w0, *b0, *w1, *q_scaler;
    T rr, ra;
    int B, P, U;
    const int *binum, *bilist, *bnumneigh, *bfirstneigh;
    const T* brcs;
    const int* btypes;
    const T *cE, *dFs, *dVs;
    T* gpart;          // [B, P, nrow] gradient row of every atom
    int nrow;
    int E;             // table entries per neighbour (generic kernel)
    int* status;
    losskern::LossRmse<T> errors;      // (rmse null: not wanted, or a launch of its own)
};

__device__ __forceinline__ int l_of_lm(int m) { return m < 3 ? 1 : m < 8 ? 2 : m < 15 ? 3 : 4; }

}  // namespace nepdev

// A wavefront per atom: whether the shape is covered (and the LDS it takes), the length of an atom's gradient row, and the
// two launches (per-atom rows, sums over the atoms of every structure and species).
template <typename T>
bool nep_loss_wave_supported(const nepdev::NepLossArgs<T>& a, size_t* lds_bytes);
template <typename T>
int nep_loss_wave_row(const nepdev::NepLossArgs<T>& a);
template <typename T>
int nep_loss_wave_run(const nepdev::NepLossArgs<T>& a, size_t lds_bytes, T* dcoeffs, T* dw0, T* db0, T* dw1, T* dbias,
                      hipStream_t stream);

}  // namespace a2p
