// rbc_update.hpp -- the group update at the end of a step (rbc_update.hip): its arguments and
// launcher, for one run or for the members of a batch (blockIdx.z).
#pragma once

#include <hip/hip_runtime.h>

#include "rbc_device.hpp"
#include "rbc_internal.hpp"

namespace rbc {

template <typename T>
struct UpdateArgs {
    DevGeom g;
    int nchunk;
    int L0;
    int L1;
    int stride;
    T Pr;
    T dt;
    T a_cur;
    T a_prev;
    int use_prev;
    const int* cgrp;
    const int* cbeg;
    const int* gmem;
    const T* gmat;
    const T* k2a;
    cpx<T>* Xt;
    cpx<T>* Xf;
    cpx<T>* Xg;
    const cpx<T>* Nt;
    const cpx<T>* Nf;
    const cpx<T>* Ng;
    cpx<T>* Rt;
    cpx<T>* Rf;
    cpx<T>* Rg;
    cpx<T>* XF;
    cpx<T>* XG;
    const cpx<T>* NF;
    const cpx<T>* NG;
    cpx<T>* RF;
    cpx<T>* RG;
    int* health;
};

template <typename T>
UpdateArgs<T> update_args(const DevGeom& g, const Buffers& b, int L0, int L1, int stride, double Pr, double dt,
                          StepCoef sc, void* const X[3], void* const N[3], void* const R[3], void* XF, void* XG,
                          const void* NF, const void* NG, void* RF, void* RG);
// batch: member arguments on the device (mode UPD_STEP), a: any member's (launch shape)
template <typename T>
void launch_update(const UpdateArgs<T>& a, int mode, const UpdateArgs<T>* batch, int nchunk_max, int B,
                   hipStream_t s);

}  // namespace rbc
