// rbc_update.hip -- the end of a time step: inverse B, AB2 combination and implicit Euler of theta,
// f and g per |k|^2 group, the mean flow F and G, the symmetry of the kx = 0 column and the health
// check, in one launch; and the same operators by themselves (inverse_B_matrix.cu,
// linear_implicit_operator.cu).
#include "rbc_update.hpp"

namespace rbc {

// a copy by components: whole 16-byte copies between address spaces keep the members of a chunk in
// scratch memory instead of registers
template <typename T>
__device__ __forceinline__ cpx<T> by_parts(const cpx<T>& v) {
    return mk(v.x, v.y);
}

// F, G: inverse B = 2 Pr (imag 0), implicit factor 1/(1 + dt Pr (m pi)^2) (imag 0); lane m.
template <typename T, int MODE>
__device__ __forceinline__ void update_FG(int m, int L, T Pr, T dt, T a_cur, T a_prev, int use_prev, cpx<T>* XF,
                                          cpx<T>* XG, const cpx<T>* NF, const cpx<T>* NG, cpx<T>* RF, cpx<T>* RG,
                                          int& bad) {
    if (m >= L) return;
    const T mpi = T(m + 1) * T(M_PI);
    const T fac = T(1) / (T(1) + dt * Pr * mpi * mpi);
    auto one = [&](cpx<T>* X, const cpx<T>* N, cpx<T>* R) {
        if constexpr (MODE == UPD_INVB) {
            R[m] = mk(T(2) * Pr * N[m].x, T(0));
        } else if constexpr (MODE == UPD_IMPLICIT) {
            X[m] = mk(fac * X[m].x, T(0));
        } else {
            const cpx<T> r = mk(T(2) * Pr * N[m].x, T(0));
            cpx<T> x = X[m] + cscale(r, a_cur);
            if (use_prev) x = x + cscale(R[m], a_prev);
            R[m] = r;
            const T v = fac * x.x;
            bad |= !isfinite(v);
            X[m] = mk(v, T(0));
        }
    };
    one(XF, NF, RF);
    one(XG, NG, RG);
}

// implicit factor of g: 1 / (1 + dt Pr (k^2 + (m pi)^2)), the inner sum rounded before the product
// whatever the surrounding code lets the compiler contract
template <typename T>
__device__ __forceinline__ T g_factor(T k2, T mpi, T dtPr) {
    T q;
    {
#pragma clang fp contract(off)
        const T m2 = mpi * mpi;
        q = k2 + m2;
    }
    return T(1) / (T(1) + dtPr * q);
}

// One |k|^2 group shares the class matrices C^-1 (n_c x n_c, n_c = 2 L_c) and B^-1_f (L_c x L_c) of
// its two parity classes (modes m = c, c + 2, ...).  A wave takes a chunk of a group's members with
// the matrices in registers: lane (class c, row r) keeps row r of C^-1 (n_c <= NC values) and of
// B^-1_f (L_c <= NC / 2 values).  W = 32 lanes per class serve L <= 32 (one wave holds both
// classes), W = 64 serve L <= 64 (a wave per class and chunk).  Per member
//   MODE UPD_STEP:     R = B^-1 N;  X += a_cur R;  X += a_prev R_prev;  X = C^-1 X;  R_prev = R
//   MODE UPD_INVB:     R = B^-1 N              (inverse_B_matrix::calculate_inverse)
//   MODE UPD_IMPLICIT: X = C^-1 X              (linear_implicit_operator::calculate_operator)
// with the diagonal factors of g (inverse_B_matrix.cu:276-300, linear_implicit_operator.cu:419-458).
// Bound by memory: 15 state passes and the factor records, and, on grids of less than a few thousand
// chunks, by the chain matrices -> members -> two matrix-vector sums.  All loads of a chunk's matrices
// and of three members are in flight at once; everything after them is registers and LDS broadcasts.
// us a step, against one block of 64 lanes per group with the matrices read per member from memory
// (W = 64) and a kernel whose FP64 members lived in scratch memory (W = 32): 1024 x 128 x 40 FP32
// 217 -> 120, 128^2 x 48 FP64 396 -> 33, 256^2 x 24 FP64 45 -> 36, 128^2 x 16 FP32 9.8 -> 8.2; 512^2
// x 32 FP32 72 + 6 (the end of the step apart) -> 75.  Allocations held to one more wave per SIMD
// (launch bounds) cost 1 to 2 us at each of these sizes.
//
// A step ends with make_real on the kx = 0 column (util.cu): row r (0 < r < N/2) becomes
// conj(row N - r) and (0, 0) real.  The wave of row N - r writes both, the wave of row r keeps its
// result to itself, so the column needs no pass of its own; the wave of (0, 0) also takes F, G and
// the health check (by themselves a launch of 3 to 6 us a step).  A non-finite
// coefficient anywhere in the state reaches every mode within one nonlinear evaluation (each
// Fourier mode of a product sums every grid point), so theta(0,0), F and G show it by the end of
// the step that consumed it.  health[1] counts the steps; health[0] keeps 1 + the count of the
// first step that ended non-finite.
template <typename T, int NC, int W, int MODE>
__device__ __forceinline__ void update_body(
    DevGeom g, int nchunk, int L0, int L1, int stride, T Pr, T dt, T a_cur, T a_prev, int use_prev,
    const int* __restrict__ cgrp, const int* __restrict__ cbeg, const int* __restrict__ gmem,
    const T* __restrict__ gmat, const T* __restrict__ k2a, cpx<T>* __restrict__ Xt, cpx<T>* __restrict__ Xf,
    cpx<T>* __restrict__ Xg, const cpx<T>* __restrict__ Nt, const cpx<T>* __restrict__ Nf,
    const cpx<T>* __restrict__ Ng, cpx<T>* __restrict__ Rt, cpx<T>* __restrict__ Rf, cpx<T>* __restrict__ Rg,
    cpx<T>* __restrict__ XF, cpx<T>* __restrict__ XG, const cpx<T>* __restrict__ NF, const cpx<T>* __restrict__ NG,
    cpx<T>* __restrict__ RF, cpx<T>* __restrict__ RG, int* __restrict__ health) {
    constexpr int NCLS = 64 / W;  // classes a wave holds
    __shared__ cpx<T> shm[4][NCLS][2][W];  // [wave][class][0: N_f, 1: rhs][j]
    // the wave index as a wave-uniform value: chunk, group and member indices then live in
    // scalar registers and come from scalar loads, which the vector loads do not wait for
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = blockIdx.x * 4 + wave, ch = NCLS == 2 ? unit : unit >> 1;
    if (ch >= nchunk) return;  // whole wave leaves; no block-wide barrier below
    const int grp = cgrp[ch], b0 = cbeg[ch], b1 = cbeg[ch + 1];
    const int L = g.L, NYc = g.NYc, n0 = 2 * L0;
    // p = 0 is the first member of its chunk (members ascend).  With a wave per class, class 0's
    // wave does both classes of that chunk, so that one lane knows all that the health check reads.
    const bool mean = gmem[b0] == 0;
    int bad = 0;
    int ucls = NCLS == 2 ? 0 : unit & 1;
    if (NCLS == 1 && mean && ucls == 1) return;
#pragma unroll 1
    for (;;) {
        const int cls = NCLS == 2 ? lane >> 5 : ucls, r = lane & (W - 1);
        const int Lc = cls ? L1 : L0, nc = 2 * Lc;
        const T* rec = gmat + (size_t)grp * stride;
        const T* Cinv = rec + (cls ? (size_t)n0 * n0 : 0);
        const T* Binv = rec + (size_t)n0 * n0 + (size_t)(2 * L1) * (2 * L1) + (cls ? (size_t)L0 * L0 : 0);
        // Every load below is issued by every lane (lanes outside the class read element 0 of a
        // valid array and discard it), and the matrix-vector sums run over the full NC / NC / 2
        // terms with zero matrix entries and zero LDS slots beyond the class size: no branch depends
        // on the class sizes, so the compiler can keep the next member's loads in flight across the
        // current member's arithmetic.  The extra terms add exact zeros.
        T crow[NC], brow[NC / 2];
        {
            const T* csrc = nc > 0 ? Cinv : rec;
            const T* bsrc = Lc > 0 ? Binv : rec;
            if constexpr (MODE != UPD_INVB) {
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    const bool in = j < nc && r < nc;
                    const T v = csrc[in ? (size_t)j * nc + r : 0];
                    crow[j] = in ? v : T(0);
                }
            }
            if constexpr (MODE != UPD_IMPLICIT) {
#pragma unroll
                for (int j = 0; j < NC / 2; ++j) {
                    const bool in = j < Lc && r < Lc;
                    const T v = bsrc[in ? (size_t)j * Lc + r : 0];
                    brow[j] = in ? v : T(0);
                }
            }
        }
        const int ci = NCLS == 2 ? cls : 0;
        cpx<T>* snf = shm[wave][ci][0];
        cpx<T>* srhs = shm[wave][ci][1];
        snf[r] = srhs[r] = mk<T>(0, 0);  // slots beyond the class stay 0
        const bool tf = r < Lc;
        const int m = tf ? cls + 2 * r : 0;  // theta/f mode of this lane (element 0 outside the class)
        // g mode of this lane: one wave holds all of them (W = 32), or its class's (W = 64)
        const bool gl = NCLS == 2 ? lane < L : tf;
        const int mg = NCLS == 2 ? (gl ? lane : 0) : m;
        // one member's loads (issued together)
        struct Member {
            cpx<T> nf, xt, xf, nt, rt, rf, ng, xg, rg;
            T k2;
            int p;
        };
        auto fetch = [&](int mi, Member& d) __attribute__((always_inline)) {
            const int p = gmem[mi];
            const size_t base = (size_t)p * L;
            d.p = p;
            d.k2 = k2a[p];
            if constexpr (MODE != UPD_IMPLICIT) {
                d.nf = by_parts(Nf[base + m]);
                d.nt = by_parts(Nt[base + m]);
                d.ng = by_parts(Ng[base + mg]);
            }
            if constexpr (MODE != UPD_INVB) {
                d.xt = by_parts(Xt[base + m]);
                d.xf = by_parts(Xf[base + m]);
                d.xg = by_parts(Xg[base + mg]);
            }
            if constexpr (MODE == UPD_STEP) {  // read also without history (then unused)
                d.rt = by_parts(Rt[base + m]);
                d.rf = by_parts(Rf[base + m]);
                d.rg = by_parts(Rg[base + mg]);
            }
        };
        auto update = [&](const Member& d) __attribute__((always_inline)) {
            const int p = d.p;
            const size_t base = (size_t)p * L;
            const T k2 = d.k2;
            cpx<T> x1, x2, acc = mk<T>(0, 0), xg = mk<T>(0, 0);
            if constexpr (MODE == UPD_IMPLICIT) {
                x1 = by_parts(d.xt);
                x2 = by_parts(d.xf);
            } else {
                if (tf) snf[r] = by_parts(d.nf);
                wave_sync();
                if (tf) {
                    cpx<T> rf = mk<T>(0, 0);
#pragma unroll
                    for (int j = 0; j < NC / 2; ++j) rf = rf + cscale(snf[j], brow[j]);
                    const cpx<T> rt = cscale(d.nt, T(2));
                    if constexpr (MODE == UPD_STEP) {
                        x1 = d.xt + cscale(rt, a_cur);
                        x2 = d.xf + cscale(rf, a_cur);
                        if (use_prev) {
                            x1 = x1 + cscale(d.rt, a_prev);
                            x2 = x2 + cscale(d.rf, a_prev);
                        }
                    }
                    Rt[base + m] = rt;
                    Rf[base + m] = rf;
                }
            }
            if constexpr (MODE != UPD_INVB) {
                if (tf) {
                    srhs[r] = by_parts(x1);
                    srhs[Lc + r] = by_parts(x2);
                }
                wave_sync();
                if (r < nc) {
#pragma unroll
                    for (int j = 0; j < NC; ++j) acc = acc + cscale(srhs[j], crow[j]);
                }
            }
            // g: diagonal factors, one vertical mode per lane
            if (gl) {
                const T mpi = T(mg + 1) * T(M_PI);
                auto nz = [&](cpx<T> v) { return mk(k2 != T(0) ? v.x : T(0), k2 != T(0) ? v.y : T(0)); };
                if constexpr (MODE == UPD_INVB) {
                    Rg[base + mg] = nz(cscale(d.ng, T(-2) * Pr / k2));
                } else if constexpr (MODE == UPD_IMPLICIT) {
                    xg = nz(cscale(d.xg, g_factor<T>(k2, mpi, dt * Pr)));
                } else {
                    const cpx<T> rg = nz(cscale(d.ng, T(-2) * Pr / k2));
                    cpx<T> x3 = d.xg + cscale(rg, a_cur);
                    if (use_prev) x3 = x3 + cscale(d.rg, a_prev);
                    Rg[base + mg] = rg;
                    xg = nz(cscale(x3, g_factor<T>(k2, mpi, dt * Pr)));
                }
            }
            if constexpr (MODE != UPD_INVB) {
                cpx<T>* X = r < Lc ? Xt : Xf;
                const int mm = cls + 2 * (r < Lc ? r : r - Lc);
                if (MODE != UPD_STEP || p >= NYc) {
                    if (r < nc) X[base + mm] = acc;
                    if (gl) Xg[base + mg] = xg;
                } else if (p == 0) {
                    if (r < nc) X[mm] = mk(acc.x, T(0));
                    if (gl) Xg[mg] = mk(xg.x, T(0));
                    bad |= tf && !isfinite(acc.x);
                } else if (2 * p > NYc) {  // rows [N - a, N - 1] of the column, compact [a + 1, 2 a]
                    const size_t mir = (size_t)(NYc - p) * L;
                    if (r < nc) {
                        X[base + mm] = acc;
                        X[mir + mm] = conjg(acc);
                    }
                    if (gl) {
                        Xg[base + mg] = xg;
                        Xg[mir + mg] = conjg(xg);
                    }
                }
            }
            wave_sync();
        };
        // The (at most four) members of a chunk two ahead: member i + 2's loads are in flight while
        // member i is computed.  Three register sets taken in turn, so that no set is copied (a copy
        // would wait for its loads); loads return in issue order, so a member waits for its own only.
        static_assert(kUpdateChunk == 4, "written out for four members");
        const int cnt = b1 - b0;
        Member d0, d1, d2;
        fetch(b0, d0);
        if (cnt > 1) fetch(b0 + 1, d1);
        if (cnt > 2) fetch(b0 + 2, d2);
        update(d0);
        if (cnt > 1) {
            if (cnt > 3) fetch(b0 + 3, d0);
            update(d1);
            if (cnt > 2) update(d2);
            if (cnt > 3) update(d0);
        }
        if (NCLS == 2 || !mean || ucls == 1) break;
        ucls = 1;
    }
    if (mean) {
        update_FG<T, MODE>(lane, L, Pr, dt, a_cur, a_prev, use_prev, XF, XG, NF, NG, RF, RG, bad);
        if constexpr (MODE == UPD_STEP) {
            const bool any = __any(bad);
            if (lane == 0) {
                const int n = health[1];
                if (any && health[0] == 0) health[0] = n + 1;
                health[1] = n + 1;
            }
        }
    }
}

template <typename T, int NC, int W, int MODE>
__global__ void __launch_bounds__(256) k_update(DevGeom g, int nchunk, int L0, int L1, int stride, T Pr, T dt, T a_cur,
                                     T a_prev, int use_prev, const int* __restrict__ cgrp,
                                     const int* __restrict__ cbeg, const int* __restrict__ gmem,
                                     const T* __restrict__ gmat, const T* __restrict__ k2a, cpx<T>* __restrict__ Xt,
                                     cpx<T>* __restrict__ Xf, cpx<T>* __restrict__ Xg,
                                     const cpx<T>* __restrict__ Nt, const cpx<T>* __restrict__ Nf,
                                     const cpx<T>* __restrict__ Ng, cpx<T>* __restrict__ Rt,
                                     cpx<T>* __restrict__ Rf, cpx<T>* __restrict__ Rg, cpx<T>* __restrict__ XF,
                                     cpx<T>* __restrict__ XG, const cpx<T>* __restrict__ NF,
                                     const cpx<T>* __restrict__ NG, cpx<T>* __restrict__ RF,
                                     cpx<T>* __restrict__ RG, int* __restrict__ health) {
    update_body<T, NC, W, MODE>(g, nchunk, L0, L1, stride, Pr, dt, a_cur, a_prev, use_prev, cgrp, cbeg, gmem,
                                  gmat, k2a, Xt, Xf, Xg, Nt, Nf, Ng, Rt, Rf, Rg, XF, XG, NF, NG, RF, RG, health);
}
// member blockIdx.z of a batch
template <typename T, int NC, int W>
__global__ void __launch_bounds__(256) k_update_batch(const UpdateArgs<T>* __restrict__ tab) {
    const UpdateArgs<T>& a = tab[blockIdx.z];
    update_body<T, NC, W, UPD_STEP>(a.g, a.nchunk, a.L0, a.L1, a.stride, a.Pr, a.dt, a.a_cur, a.a_prev,
                                  a.use_prev, a.cgrp, a.cbeg, a.gmem, a.gmat, a.k2a, a.Xt, a.Xf, a.Xg, a.Nt,
                                  a.Nf, a.Ng, a.Rt, a.Rf, a.Rg, a.XF, a.XG, a.NF, a.NG, a.RF, a.RG, a.health);
}

template <typename T>
UpdateArgs<T> update_args(const DevGeom& g, const Buffers& b, int L0, int L1, int stride, double Pr, double dt,
                          StepCoef sc, void* const X[3], void* const N[3], void* const R[3], void* XF, void* XG,
                          const void* NF, const void* NG, void* RF, void* RG) {
    using C = cpx<T>;
    return {g, b.nchunk, L0, L1, stride, (T)Pr, (T)dt, (T)sc.a_cur, (T)sc.a_prev, sc.use_prev, b.cgrp, b.cbeg, b.gmem,
            (const T*)b.gmat, (const T*)b.k2, (C*)X[0], (C*)X[1], (C*)X[2], (const C*)N[0], (const C*)N[1],
            (const C*)N[2], (C*)R[0], (C*)R[1], (C*)R[2], (C*)XF, (C*)XG, (const C*)NF, (const C*)NG, (C*)RF, (C*)RG,
            b.health};
}

template <typename T, int NC, int W, int MODE>
static void launch_one(const UpdateArgs<T>& a, dim3 gr, hipStream_t s) {
    hipLaunchKernelGGL((k_update<T, NC, W, MODE>), gr, dim3(256), 0, s, a.g, a.nchunk, a.L0, a.L1, a.stride, a.Pr, a.dt, a.a_cur, a.a_prev,
                                  a.use_prev, a.cgrp, a.cbeg, a.gmem, a.gmat, a.k2a, a.Xt, a.Xf, a.Xg, a.Nt,
                                  a.Nf, a.Ng, a.Rt, a.Rf, a.Rg, a.XF, a.XG, a.NF, a.NG, a.RF, a.RG, a.health);
}

template <typename T>
void launch_update(const UpdateArgs<T>& a, int mode, const UpdateArgs<T>* batch, int nchunk_max, int B,
                   hipStream_t s) {
    // W = 32: a wave per chunk; W = 64: two.  NC is the row length that the registers hold, the
    // next of 16, 32, 48 and 64 over n_0 = 2 ceil(L / 2).
    const int units = (a.g.L <= 32 ? 1 : 2) * (batch ? nchunk_max : a.nchunk);
    const dim3 gr((units + 3) / 4, 1, batch ? B : 1);
    if constexpr (sizeof(T) == 4) {
        if (batch) {  // FP32 storage and L <= 32 only
            if (a.g.L <= 16) hipLaunchKernelGGL((k_update_batch<T, 16, 32>), gr, dim3(256), 0, s, batch);
            else hipLaunchKernelGGL((k_update_batch<T, 32, 32>), gr, dim3(256), 0, s, batch);
            return;
        }
    }
#define RBC_UPD_M(NCV, WV)                                                           \
    if (mode == UPD_STEP) launch_one<T, NCV, WV, UPD_STEP>(a, gr, s);                \
    else if (mode == UPD_INVB) launch_one<T, NCV, WV, UPD_INVB>(a, gr, s);           \
    else launch_one<T, NCV, WV, UPD_IMPLICIT>(a, gr, s)
    if (a.g.L <= 16) {
        RBC_UPD_M(16, 32);
    } else if (a.g.L <= 32) {
        RBC_UPD_M(32, 32);
    } else if (a.g.L <= 48) {
        RBC_UPD_M(48, 64);
    } else {
        RBC_UPD_M(64, 64);
    }
#undef RBC_UPD_M
}

#define RBC_INST(T)                                                                                                  \
    template UpdateArgs<T> update_args<T>(const DevGeom&, const Buffers&, int, int, int, double, double, StepCoef,   \
                                          void* const[3], void* const[3], void* const[3], void*, void*, const void*, \
                                          const void*, void*, void*);                                                \
    template void launch_update<T>(const UpdateArgs<T>&, int, const UpdateArgs<T>*, int, int, hipStream_t);
RBC_INST(float)
RBC_INST(double)
#undef RBC_INST

}  // namespace rbc
