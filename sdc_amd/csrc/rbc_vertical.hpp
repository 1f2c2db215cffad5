// rbc_vertical.hpp -- the matrix-core vertical transforms (rbc_vertical.hip): their arguments and
// launchers, for one run or for the members of a batch (blockIdx.z).
#pragma once

#include <hip/hip_runtime.h>

#include "rbc_device.hpp"
#include "rbc_internal.hpp"

namespace rbc {

template <typename T>
struct EvalArgs {
    DevGeom g;
    int TS, NP;      // waves the level tiles and the three parts are split over
    int nwork, per;  // waves with work; logical blocks per XCD
    const cpx<T>*Xt, *Xf, *Xg, *XF, *XG;
    const T *tab, *evtab, *kx, *ky;
    cpx<T>* lev;
};
template <typename T>
struct ProjectArgs {
    DevGeom g;
    int nks, per;  // k-steps of four half-levels; logical blocks per XCD
    const cpx<T>*D, *fgw;
    const T *tab, *prtab, *kx, *ky;
    T Pr;
    cpx<T>*Nt, *Nf, *Ng, *NF, *NG;
};

template <typename T>
EvalArgs<T> eval_args(const DevGeom& g, const Buffers& b, void* const X[3], const void* XF,
                                   const void* XG);
template <typename T>
ProjectArgs<T> project_args(const DevGeom& g, const Buffers& b, double Pr, void* const Nout[3],
                                         void* NFo, void* NGo);
template <typename T>
void launch_eval(const EvalArgs<T>& a, const EvalArgs<T>* batch, int B, hipStream_t s);
template <typename T>
void launch_project(const ProjectArgs<T>& a, const ProjectArgs<T>* batch, int B, hipStream_t s);

}  // namespace rbc
