// rbc_vertical.hip -- vertical transforms on the matrix cores.
//
// FP64, and FP32 with more than 32 vertical modes, fold the parity of the vertical basis in: the
// Gauss-Legendre levels are symmetric about the mid-plane and every basis function is even or odd
// there: C_m, C''_m and S_m are even for 0-based even m and odd for odd m, C'_m and S'_m the other way
// round.  So only the lower half of the levels is summed: a level q and its mirror nq - 1 - q share
// the two class sums (even m, odd m), which add for one and subtract for the other, and the
// projection folds the two levels into their sum and difference first.  Half the products and half
// the basis tables of the plain sums.
//
// FP32 up to 32 modes is bound by memory with the plain sums too, and keeps them: term by term in
// the order of m and of the levels (*_plain).
//
// Products: v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32 (wave64): A (16 x 4) lane l holds row l % 16,
// k = l / 16; B (4 x 16) lane l holds column l % 16, k = l / 16; D (16 x 16) register r of lane l holds
// column l % 16, row 4 (l / 16) + r (FP32) or 4 r + l / 16 (FP64); each entry is the chain of four
// FMAs in k order.  The FP32 tables store their rows permuted (parity_row) so that in both types
// register r of lane group h = l / 16 stands for row 4 r + h: the four lane groups of a mode then
// write consecutive vertical modes.  A column is a horizontal mode; its real and imaginary part run
// as two products with the same A operand, so a lane loads and stores whole complex values.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "rbc_ctx.hpp"
#include "rbc_device.hpp"
#include "rbc_vertical.hpp"

namespace rbc {

namespace {

template <typename T>
struct Mat16;
template <>
struct Mat16<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ v4 run(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mat16<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ v4 run(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};

// class pair (even m, odd m) of one table entry
template <typename T>
struct alignas(2 * sizeof(T)) pair2 {
    T c[2];
};

// two consecutive complex values; PAIRED: wide loads (the address is a multiple of 16 bytes)
template <typename T, bool PAIRED>
__device__ __forceinline__ void load_two(const cpx<T>* p, cpx<T>& a, cpx<T>& b, bool second) {
    if constexpr (PAIRED) {
        struct alignas(16) two {
            cpx<T> v[2];
        };
        const two t = *reinterpret_cast<const two*>(p);
        a = t.v[0];
        b = t.v[1];
    } else {
        a = p[0];
        b = second ? p[1] : mk(T(0), T(0));
    }
}

// ---------------------------------------------------------------------------------------
// Evaluation (mode -> level).  A wave takes 16 modes and, for each of three parts in turn, the level
// tiles (16 half-levels, 32 levels) ts, ts + TS, ...:
//   part 0: u, v from f (C') and g (S)   part 1: w from f (C)   part 2: the gradient of theta (S, S')
// The part's mode values stay in registers over its tiles: NS k-steps of 4 per parity class
// (L <= 8 NS).  No LDS.  Grids with few modes split the tiles (TS) and the parts (NP = 3) over waves.
// The mean flow at k = 0 (u += sum S_m F_m, v += sum S_m G_m, where f and g do not contribute) is
// written by a block of its own, one level per thread, instead of the wave of mode 0.
//
// Bound: HBM, 3 L values read and 6 nq written per mode.  us, before (VALU sums) -> now: 256^2 x 24 FP64
// 87 -> 26, 32^2 x 8 FP64 24 -> 4.1, 1024 x 128 x 40 FP32 152 -> 54.
// ---------------------------------------------------------------------------------------
template <typename T, int NS, bool PAIRED>
__device__ __forceinline__ void eval_parity_body(const EvalArgs<T>& A) {
    using M = Mat16<T>;
    using v4 = typename M::v4;
    const DevGeom& g = A.g;
    const int TS = A.TS, NP = A.NP;
    const pair2<T>* __restrict__ tab = reinterpret_cast<const pair2<T>*>(A.tab);
    const cpx<T>*__restrict__ Xt = A.Xt, *__restrict__ Xf = A.Xf, *__restrict__ Xg = A.Xg;
    cpx<T>* __restrict__ lev = A.lev;
    const int L = g.L, P = g.P, PS = g.PS, nq = g.nq, nh = (nq + 1) / 2, nt = (nh + 15) / 16;
    const size_t fs = (size_t)nq * PS;
    if (blockIdx.x == gridDim.x - 1) {  // the mean flow at mode 0
        for (int e = threadIdx.x; e < 2 * nq; e += 256) {
            const int l = e >> 1;
            const cpx<T>* F = (e & 1) ? A.XG : A.XF;
            const T* tb = A.evtab + (size_t)l * 4 * L + 2 * L;
            cpx<T> s = mk(T(0), T(0));
#pragma unroll 8
            for (int m = 0; m < L; ++m) s = s + cscale(F[m], tb[m]);
            lev[(e & 1) * fs + (size_t)l * PS] = s;
        }
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = xcd_logical_block(blockIdx.x, A.per) * 4 + wave;
    if (w >= A.nwork) return;
    const int part0 = NP == 1 ? 0 : w % NP, part1 = NP == 1 ? 3 : part0 + 1;
    const int ts = (w / NP) % TS, p0 = (w / NP / TS) * 16;
    const int col = lane & 15, h = lane >> 4;
    const int p = p0 + col;
    const bool pvalid = p < P;
    const int pc = pvalid ? p : P - 1;
    const T kx = A.kx[pc], ky = A.ky[pc];
    const size_t row = (size_t)pc * L;
    auto load = [&](const cpx<T>* X, cpx<T> (&b)[2][NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int m = 8 * s + 2 * h;
            b[0][s] = b[1][s] = mk(T(0), T(0));
            if (m < L) load_two<T, PAIRED>(X + row + m, b[0][s], b[1][s], m + 1 < L);
        }
    };
    // class sums of one table over the tile: d[class][re, im]
    auto sums = [&](int table, int t, const cpx<T> (&b)[2][NS], v4 (&d)[2][2]) {
        const pair2<T>* tb = tab + ((size_t)(table * nt + t) * NS) * 64 + lane;
        d[0][0] = d[0][1] = d[1][0] = d[1][1] = v4{};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const pair2<T> a = tb[s * 64];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                d[c][0] = M::run(a.c[c], b[c][s].x, d[c][0]);
                d[c][1] = M::run(a.c[c], b[c][s].y, d[c][1]);
            }
        }
    };
    // level q = 16 t + 4 h + r gets even + odd, its mirror even - odd (even, odd in z)
    auto store = [&](int field, int t, int r, cpx<T> even, cpx<T> odd) {
        const int q = 16 * t + 4 * r + h;
        if (!pvalid || q >= nh) return;
        cpx<T>* o = lev + field * fs + p;
        o[(size_t)q * PS] = even + odd;
        if (2 * q + 1 != nq) o[(size_t)(nq - 1 - q) * PS] = even - odd;
    };
    auto val = [](const v4 (&d)[2], int r) { return mk(d[0][r], d[1][r]); };  // (re, im) of row r
    if (part0 == 0) {
        cpx<T> bf[2][NS], bg[2][NS];
        load(Xf, bf);
        load(Xg, bg);
        for (int t = ts; t < nt; t += TS) {
            v4 F[2][2], G[2][2];
            sums(0, t, bf, F);  // C': odd in z for class 0
            sums(2, t, bg, G);  // S: even in z for class 0
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const cpx<T> f0 = val(F[0], r), f1 = val(F[1], r), g0 = val(G[0], r), g1 = val(G[1], r);
                const cpx<T> ue = imul(f1, kx) + imul(g0, ky), uo = imul(f0, kx) + imul(g1, ky);
                const cpx<T> ve = imul(f1, ky) - imul(g0, kx), vo = imul(f0, ky) - imul(g1, kx);
                if (p != 0) {
                    store(0, t, r, ue, uo);
                    store(1, t, r, ve, vo);
                }
            }
        }
        if (part1 > 1) {
            const T k2 = kx * kx + ky * ky;
            for (int t = ts; t < nt; t += TS) {
                v4 F[2][2];
                sums(1, t, bf, F);
#pragma unroll
                for (int r = 0; r < 4; ++r) store(2, t, r, cscale(val(F[0], r), k2), cscale(val(F[1], r), k2));
            }
        }
    } else if (part0 == 1) {
        cpx<T> bf[2][NS];
        load(Xf, bf);
        const T k2 = kx * kx + ky * ky;
        for (int t = ts; t < nt; t += TS) {
            v4 F[2][2];
            sums(1, t, bf, F);
#pragma unroll
            for (int r = 0; r < 4; ++r) store(2, t, r, cscale(val(F[0], r), k2), cscale(val(F[1], r), k2));
        }
    }
    if (part1 == 3) {
        cpx<T> bt[2][NS];
        load(Xt, bt);
        for (int t = ts; t < nt; t += TS) {
            v4 S[2][2], Z[2][2];
            sums(2, t, bt, S);
            sums(3, t, bt, Z);  // S': odd in z for class 0
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const cpx<T> e = val(S[0], r), o = val(S[1], r);
                store(3, t, r, imul(e, kx), imul(o, kx));
                store(4, t, r, imul(e, ky), imul(o, ky));
                store(5, t, r, val(Z[1], r), val(Z[0], r));
            }
        }
    }
}

template <typename T, int NS, bool PAIRED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : (NS >= 8 ? 3 : 4))))
k_eval_parity(EvalArgs<T> a) {
    eval_parity_body<T, NS, PAIRED>(a);
}
// member blockIdx.z of a batch
template <typename T, int NS, bool PAIRED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : (NS >= 8 ? 3 : 4))))
k_eval_parity_batch(const EvalArgs<T>* __restrict__ tab) {
    eval_parity_body<T, NS, PAIRED>(tab[blockIdx.z]);
}

// ---------------------------------------------------------------------------------------
// Projection (level -> mode).  A wave takes 16 modes and 16 vertical modes of each parity class (L <= 32:
// all of them; else blockIdx.y picks the half), and sums over a range of half-levels: per k-step of 4 it
// loads the five level combinations at the levels and at their mirrors, forms sums and
// differences, and multiplies by the table rows of both classes; k^2 goes onto the operand of the
// C table, so that f has one accumulator.  The next k-step's operands load while the current one
// multiplies.  KS waves of a block split the levels and add their sums through LDS in a fixed order.
//
// Bound: HBM, 5 nq values read and 3 L written per mode.  us, before (VALU sums) -> now: 256^2 x 24
// FP64 162 -> 28, 32^2 x 8 FP64 38 -> 6.2, 1024 x 128 x 40 FP32 337 -> 59; the 16-byte stores of consecutive modes
// were 8 us of the last.
// ---------------------------------------------------------------------------------------
template <typename T, int KS>
__device__ __forceinline__ void project_parity_body(const ProjectArgs<T>& A) {
    using M = Mat16<T>;
    using v4 = typename M::v4;
    const DevGeom& g = A.g;
    const int nks = A.nks;
    const T Pr = A.Pr;
    const pair2<T>* __restrict__ ptab = reinterpret_cast<const pair2<T>*>(A.tab);
    const cpx<T>* __restrict__ D = A.D;
    __shared__ v4 part[KS > 1 ? KS / 2 : 1][KS > 1 ? 12 : 1][64];
    const int L = g.L, P = g.P, PS = g.PS, nq = g.nq, nh = (nq + 1) / 2;
    const int lb = xcd_logical_block(blockIdx.x, A.per), mt = blockIdx.y;
    if (blockIdx.x == gridDim.x - 1) {  // the mean flow, in a block of its own
        if (mt == 0) mean_flow_projection<T>(g, A.fgw, A.prtab, Pr, A.NF, A.NG);
        return;
    }
    if (lb * 16 >= P) return;
    const int lane = threadIdx.x & 63, wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, h = lane >> 4;
    const int p = lb * 16 + col;
    const bool pvalid = p < P;
    const int pc = pvalid ? p : P - 1;
    const T kx = A.kx[pc], ky = A.ky[pc], k2 = kx * kx + ky * ky;
    const size_t fs = (size_t)nq * PS;
    const int spw = (nks + KS - 1) / KS, sbeg = wk * spw, send = min(nks, sbeg + spw);
    struct Operands {
        cpx<T> a[5], b[5];
        pair2<T> t[5];
    };
    auto fetch = [&](int s, Operands& o) {
        const int q = min(4 * s + h, nh - 1);  // past the last level: table entries 0
        const cpx<T>* lo = D + (size_t)q * PS + pc;
        const cpx<T>* hi = D + (size_t)(nq - 1 - q) * PS + pc;
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            o.a[t] = lo[t * fs];
            o.b[t] = hi[t * fs];
        }
        const pair2<T>* tb = ptab + ((size_t)(mt * nks + s) * 5) * 64 + lane;
#pragma unroll
        for (int t = 0; t < 5; ++t) o.t[t] = tb[t * 64];
    };
    v4 F[2][2] = {}, G[2][2] = {}, H[2][2] = {};
    auto step = [&](const Operands& o) {
        cpx<T> sum[5], dif[5];
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            sum[t] = o.a[t] + o.b[t];
            dif[t] = o.a[t] - o.b[t];
        }
        const cpx<T> s1k = cscale(sum[1], k2), d1k = cscale(dif[1], k2);
        auto mul = [&](v4 (&acc)[2], T a, cpx<T> b) {
            acc[0] = M::run(a, b.x, acc[0]);
            acc[1] = M::run(a, b.y, acc[1]);
        };
        // tables: 0 wC', 1 wC'', 2 wC, 3 wS, 4 wS'; class 0 of C', S' is odd in z, of the others even
        mul(F[0], o.t[0].c[0], dif[0]);
        mul(F[1], o.t[0].c[1], sum[0]);
        mul(G[0], o.t[3].c[0], sum[2]);
        mul(G[1], o.t[3].c[1], dif[2]);
        mul(H[0], o.t[3].c[0], sum[4]);
        mul(H[1], o.t[3].c[1], dif[4]);
        mul(F[0], o.t[1].c[0], sum[1]);
        mul(F[1], o.t[1].c[1], dif[1]);
        mul(G[0], o.t[4].c[0], dif[3]);
        mul(G[1], o.t[4].c[1], sum[3]);
        mul(F[0], o.t[2].c[0], s1k);
        mul(F[1], o.t[2].c[1], d1k);
    };
    {
        Operands o0, o1;
        int s = sbeg;
        if (s < send) fetch(s, o0);
        for (; s + 2 <= send; s += 2) {
            fetch(s + 1, o1);
            __builtin_amdgcn_sched_barrier(0);
            step(o0);
            __builtin_amdgcn_sched_barrier(0);
            fetch(min(s + 2, send - 1), o0);  // the last one is not used
            __builtin_amdgcn_sched_barrier(0);
            step(o1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (s < send) step(o0);
    }
    if constexpr (KS > 1) {
        v4* acc[12];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[i] = &F[i >> 1][i & 1];
            acc[4 + i] = &G[i >> 1][i & 1];
            acc[8 + i] = &H[i >> 1][i & 1];
        }
#pragma unroll
        for (int half = KS / 2; half > 0; half >>= 1) {
            if (wk >= half && wk < 2 * half) {
#pragma unroll
                for (int i = 0; i < 12; ++i) part[wk - half][i][lane] = *acc[i];
            }
            __syncthreads();
            if (wk < half) {
#pragma unroll
                for (int i = 0; i < 12; ++i) *acc[i] += part[wk][i][lane];
            }
            if (half > 1) __syncthreads();
        }
        if (wk > 0) return;
    }
    if (!pvalid) return;
    // lane: mode p, vertical modes 32 mt + 8 r + 2 h + class: register r of the four lane groups covers 8
    // consecutive modes, and the two classes of a lane are one 16-byte (FP32, even L) or two stores
    const T ft = T(-1), fp = T(-1) / Pr;
    const int m0 = 32 * mt + 2 * h;
    const size_t at = (size_t)p * L + m0;
    struct alignas(16) two {
        cpx<T> v[2];
    };
    auto write = [&](cpx<T>* out, const v4 (&d)[2][2], T f) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const cpx<T> a = mk(f * d[0][0][r], f * d[0][1][r]), b = mk(f * d[1][0][r], f * d[1][1][r]);
            if (L % 2 == 0) {
                if (m0 + 8 * r < L) *reinterpret_cast<two*>(out + at + 8 * r) = two{{a, b}};
            } else {
                if (m0 + 8 * r < L) out[at + 8 * r] = a;
                if (m0 + 8 * r + 1 < L) out[at + 8 * r + 1] = b;
            }
        }
    };
    write(A.Nt, H, ft);
    write(A.Nf, F, fp);
    write(A.Ng, G, fp);
}

template <typename T, int KS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : (KS == 1 ? 4 : 3))))
k_project_parity(ProjectArgs<T> a) {
    project_parity_body<T, KS>(a);
}
// member blockIdx.z of a batch
template <typename T, int KS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : (KS == 1 ? 4 : 3))))
k_project_parity_batch(const ProjectArgs<T>* __restrict__ tab) {
    project_parity_body<T, KS>(tab[blockIdx.z]);
}

// ---------------------------------------------------------------------------------------
// FP32, L <= 32, plain sums.  Evaluation: as eval_parity_body, over all level tiles (16 levels), NS
// k-steps of 4 modes (L <= 4 NS); a k-step's entries of the four tables are one 16-byte load.  A wave with all
// three parts runs their five sums side by side.
// Bound: HBM, 3 L values read and 6 nq written per mode.  us, before (32 x 32 tiles staged through LDS)
// -> now: 512^2 x 32 93 -> 78 (4.0 TB/s), 256^2 x 24 21.8 -> 20.9, 128^2 x 16 13.7 -> 9.5 (HIP events).  The five
// sums side by side at four waves per SIMD, a few registers spilled, beat three waves without spills (86) and
// the theta sums in a pass of their own (92).
// ---------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename V>
__device__ __forceinline__ V* at_byte(V* base, unsigned off) {  // uniform base, 32-bit offset per lane
    return reinterpret_cast<V*>((char*)base + off);
}
template <typename V>
__device__ __forceinline__ const V* at_byte(const V* base, unsigned off) {
    return reinterpret_cast<const V*>((const char*)base + off);
}

template <int NS>
__device__ __forceinline__ void eval_plain_body(const EvalArgs<float>& A) {
#pragma clang fp contract(off)
    using M = Mat16<float>;
    const DevGeom& g = A.g;
    const int L = g.L, P = g.P, PS = g.PS, nq = g.nq, nt = (nq + 15) / 16, TS = A.TS;
    const size_t fs = (size_t)nq * PS;
    cpx<float>* __restrict__ lev = A.lev;
    if (blockIdx.x == gridDim.x - 1) {  // the mean flow at mode 0
        for (int e = threadIdx.x; e < 2 * nq; e += 256) {
            const int l = e >> 1;
            const cpx<float>* F = (e & 1) ? A.XG : A.XF;
            const float* tb = A.evtab + (size_t)l * 4 * L + 2 * L;
            cpx<float> s = mk(0.f, 0.f);
#pragma unroll 8
            for (int m = 0; m < L; ++m) s = mk(__builtin_fmaf(F[m].x, tb[m], s.x), __builtin_fmaf(F[m].y, tb[m], s.y));
            lev[(e & 1) * fs + (size_t)l * PS] = s;
        }
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = xcd_logical_block(blockIdx.x, A.per) * 4 + wave;
    if (w >= A.nwork) return;
    const int part = A.NP == 1 ? -1 : w % A.NP;  // -1: all three
    const int ts = (w / A.NP) % TS, p0 = (w / A.NP / TS) * 16;
    const int col = lane & 15, h = lane >> 4;
    const int p = p0 + col;
    const bool pvalid = p < P;
    const int pc = pvalid ? p : P - 1;
    const float kx = A.kx[pc], ky = A.ky[pc], k2 = __builtin_fmaf(kx, kx, ky * ky);
    const size_t row = (size_t)pc * L;
    auto load = [&](const cpx<float>* __restrict__ X, cpx<float> (&b)[NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s) b[s] = 4 * s + h < L ? X[row + 4 * s + h] : mk(0.f, 0.f);
    };
    auto entry = [&](int t, int s) {  // a lane's C', C, S, S' of a k-step
        return *at_byte(reinterpret_cast<const f32x4*>(A.tab) + ((size_t)t * NS + s) * 64, 16u * lane);
    };
    auto mul = [&](f32x4 (&d)[2], float a, cpx<float> b) {
        d[0] = M::run(a, b.x, d[0]);
        d[1] = M::run(a, b.y, d[1]);
    };
    // byte offsets inside one level field stay below 2^31 (vertical_plain)
    auto store = [&](int field, int t, int r, cpx<float> v) {
        const int l = 16 * t + 4 * r + h;
        if (pvalid && l < nq) *at_byte(lev + field * fs, 8u * ((unsigned)l * PS + p)) = v;
    };
    auto velocity = [&](int t, const f32x4 (&F)[2], const f32x4 (&G)[2]) {
        if (p == 0) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // i kx F + i ky G, i ky F - i kx G
            store(0, t, r, mk(-__builtin_fmaf(kx, F[1][r], ky * G[1][r]), __builtin_fmaf(kx, F[0][r], ky * G[0][r])));
            store(1, t, r,
                  mk(-__builtin_fmaf(ky, F[1][r], -(kx * G[1][r])), __builtin_fmaf(ky, F[0][r], -(kx * G[0][r]))));
        }
    };
    auto vertical = [&](int t, const f32x4 (&F)[2]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) store(2, t, r, mk(k2 * F[0][r], k2 * F[1][r]));
    };
    auto gradient = [&](int t, const f32x4 (&S)[2], const f32x4 (&Z)[2]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            store(3, t, r, mk(-(kx * S[1][r]), kx * S[0][r]));
            store(4, t, r, mk(-(ky * S[1][r]), ky * S[0][r]));
            store(5, t, r, mk(Z[0][r], Z[1][r]));
        }
    };
    if (part < 0) {
        cpx<float> bf[NS], bg[NS], bt[NS];
        load(A.Xf, bf);
        load(A.Xg, bg);
        load(A.Xt, bt);
        for (int t = ts; t < nt; t += TS) {
            f32x4 F[2] = {}, C[2] = {}, G[2] = {}, S[2] = {}, Z[2] = {};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const f32x4 a = entry(t, s);
                mul(F, a[0], bf[s]);
                mul(C, a[1], bf[s]);
                mul(G, a[2], bg[s]);
                mul(S, a[2], bt[s]);
                mul(Z, a[3], bt[s]);
            }
            velocity(t, F, G);
            vertical(t, C);
            gradient(t, S, Z);
        }
        return;
    }
    if (part == 0) {
        cpx<float> bf[NS], bg[NS];
        load(A.Xf, bf);
        load(A.Xg, bg);
        for (int t = ts; t < nt; t += TS) {
            f32x4 F[2] = {}, G[2] = {};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const f32x4 a = entry(t, s);
                mul(F, a[0], bf[s]);
                mul(G, a[2], bg[s]);
            }
            velocity(t, F, G);
        }
    } else if (part == 1) {
        cpx<float> bf[NS];
        load(A.Xf, bf);
        for (int t = ts; t < nt; t += TS) {
            f32x4 C[2] = {};
#pragma unroll
            for (int s = 0; s < NS; ++s) mul(C, entry(t, s)[1], bf[s]);
            vertical(t, C);
        }
    }
    if (part == 2) {
        cpx<float> bt[NS];
        load(A.Xt, bt);
        for (int t = ts; t < nt; t += TS) {
            f32x4 S[2] = {}, Z[2] = {};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const f32x4 a = entry(t, s);
                mul(S, a[2], bt[s]);
                mul(Z, a[3], bt[s]);
            }
            gradient(t, S, Z);
        }
    }
}

template <int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_eval_plain(EvalArgs<float> a) {
    eval_plain_body<NS>(a);
}
template <int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
k_eval_plain_batch(const EvalArgs<float>* __restrict__ tab) {  // member blockIdx.z
    eval_plain_body<NS>(tab[blockIdx.z]);
}

// Projection: a wave takes 16 modes and all vertical modes, m = 2 (row) + half in two tiles.  The sums run
// over pairs of levels: f: C' D0 at both, then C'' D1 at both (the four k of one instruction; and C D1 in
// a sum of its own, times k^2 at the end), g: S D2 at both, then S' D3, theta: S D4.  Lane groups h = 0, 1
// so load D0 and D2 at the pair, 2, 3 load D1 and D3.  The C D1 and S D4 sums take two pairs at a time.
// KS waves split the pairs into contiguous ranges and their sums are added in order.
// Bound: HBM, 5 nq values read and 3 L written per mode.  us, before -> now: 512^2 x 32 77 -> 78, 256^2 x 24 27.7
// -> 21.1, 128^2 x 16 14.1 -> 9.0 (HIP events).  The operands two steps ahead at two waves per SIMD: one step ahead at
// three waves 87.
template <int KS>
__device__ __forceinline__ void project_plain_body(const ProjectArgs<float>& A) {
#pragma clang fp contract(off)
    using M = Mat16<float>;
    const DevGeom& g = A.g;
    __shared__ f32x4 part[KS > 1 ? KS - 1 : 1][KS > 1 ? 16 : 1][64];
    const int L = g.L, P = g.P, PS = g.PS, nq = g.nq, npair = (nq + 1) / 2;
    if (blockIdx.x == gridDim.x - 1) {  // the mean flow, in a block of its own
        mean_flow_projection<float>(g, A.fgw, A.prtab, A.Pr, A.NF, A.NG);
        return;
    }
    const int lb = xcd_logical_block(blockIdx.x, A.per);
    if (lb * 16 >= P) return;
    const int lane = threadIdx.x & 63, wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, h = lane >> 4;
    const int p = lb * 16 + col;
    const bool pvalid = p < P;
    const int pc = pvalid ? p : P - 1;
    const float kx = A.kx[pc], ky = A.ky[pc], k2 = __builtin_fmaf(kx, kx, ky * ky);
    const size_t fs = (size_t)nq * PS;
    const int ppw = (npair + KS - 1) / KS, sbeg = wk * ppw, send = min(npair, sbeg + ppw);
    // Operands by a uniform base and a 32-bit byte offset per lane (one level combination stays below 2^31
    // bytes and nq >= 8: vertical_plain), unclamped: past the last level the tables hold zeros and the
    // reads, at most 3 levels past the fifth combination, fall into the sixth field of the level buffer,
    // which the evaluation writes.
    // tables: per pair, (f half 0, f half 1, g half 0, g half 1), then per pair as the first of two, (C half 0, 1, S
    // half 0, 1)
    const cpx<float>* __restrict__ D = A.D;
    const f32x4* __restrict__ tab = reinterpret_cast<const f32x4*>(A.tab);
    const unsigned lrow = 8u * PS;  // bytes of a level
    const unsigned of = 8u * pc + (h & 1) * lrow + (h >> 1) * (unsigned)nq * lrow, oc = 8u * pc + h * lrow;
    struct Operands {
        cpx<float> f[2], g[2], c, t;
        f32x4 ap[2], aq;
    };
    auto fetch = [&](int s, Operands& o) {  // pairs s and s + 1
        const unsigned at = 2u * s * lrow;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            o.f[u] = *at_byte(D, of + at + 2 * u * lrow);            // D0 or D1
            o.g[u] = *at_byte(D + 2 * fs, of + at + 2 * u * lrow);   // D2 or D3
            o.ap[u] = *at_byte(tab + (size_t)min(s + u, npair - 1) * 64, 16u * lane);
        }
        o.c = *at_byte(D + fs, oc + at);
        o.t = *at_byte(D + 4 * fs, oc + at);
        o.aq = *at_byte(tab + (size_t)(npair + s) * 64, 16u * lane);
        if (s + 1 >= send && h >= 2) o.c = o.t = mk(0.f, 0.f);  // the second pair is another range's
    };
    f32x4 F[2][2] = {}, C[2][2] = {}, G[2][2] = {}, H[2][2] = {};  // [half][re, im]
    auto step = [&](int s, const Operands& o) {
        auto mul = [&](f32x4 (&d)[2], float a, cpx<float> b) {
            d[0] = M::run(a, b.x, d[0]);
            d[1] = M::run(a, b.y, d[1]);
        };
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (u == 0 || s + 1 < send) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    mul(F[c], o.ap[u][c], o.f[u]);
                    mul(G[c], o.ap[u][2 + c], o.g[u]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            mul(C[c], o.aq[c], o.c);
            mul(H[c], o.aq[2 + c], o.t);
        }
    };
    if (sbeg < send) {
        // two steps of two pairs ahead: three operand sets in turn over a loop unrolled three times, so that
        // none is copied (a copy would wait for its loads)
        Operands o[3];
        const int last = npair - 1;
        fetch(sbeg, o[0]);
        fetch(min(sbeg + 2, last), o[1]);
        int s = sbeg;
        for (; s + 4 < send; s += 6) {  // at least three more steps, the last possibly of one pair
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                __builtin_amdgcn_sched_barrier(0);
                fetch(min(s + 2 * u + 4, last), o[(u + 2) % 3]);
                __builtin_amdgcn_sched_barrier(0);
                step(s + 2 * u, o[u]);
            }
        }
        if (s < send) step(s, o[0]);
        if (s + 2 < send) step(s + 2, o[1]);
    }
    if constexpr (KS > 1) {
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                part[wk - 1][i][lane] = F[i >> 1][i & 1];
                part[wk - 1][4 + i][lane] = C[i >> 1][i & 1];
                part[wk - 1][8 + i][lane] = G[i >> 1][i & 1];
                part[wk - 1][12 + i][lane] = H[i >> 1][i & 1];
            }
        }
        __syncthreads();
        if (wk > 0) return;
#pragma unroll 1
        for (int k = 0; k < KS - 1; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                F[i >> 1][i & 1] += part[k][i][lane];
                C[i >> 1][i & 1] += part[k][4 + i][lane];
                G[i >> 1][i & 1] += part[k][8 + i][lane];
                H[i >> 1][i & 1] += part[k][12 + i][lane];
            }
    }
    if (!pvalid) return;
    const float ft = -1.f, fp = -1.f / A.Pr;
    const size_t at = (size_t)p * L + 2 * h;
    struct alignas(16) two {
        cpx<float> v[2];
    };
    auto put = [&](cpx<float>* out, int r, cpx<float> a, cpx<float> b) {  // m = 8 r + 2 h, + 1
        if (L % 2 == 0) {
            if (8 * r + 2 * h < L) *reinterpret_cast<two*>(out + at + 8 * r) = two{{a, b}};
        } else {
            if (8 * r + 2 * h < L) out[at + 8 * r] = a;
            if (8 * r + 2 * h + 1 < L) out[at + 8 * r + 1] = b;
        }
    };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        cpx<float> f[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
            f[c] = mk(fp * __builtin_fmaf(k2, C[c][0][r], F[c][0][r]), fp * __builtin_fmaf(k2, C[c][1][r], F[c][1][r]));
        put(A.Nt, r, mk(ft * H[0][0][r], ft * H[0][1][r]), mk(ft * H[1][0][r], ft * H[1][1][r]));
        put(A.Nf, r, f[0], f[1]);
        put(A.Ng, r, mk(fp * G[0][0][r], fp * G[0][1][r]), mk(fp * G[1][0][r], fp * G[1][1][r]));
    }
}

template <int KS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2)))
k_project_plain(ProjectArgs<float> a) {
    project_plain_body<KS>(a);
}
template <int KS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2)))
k_project_plain_batch(const ProjectArgs<float>* __restrict__ tab) {  // member blockIdx.z
    project_plain_body<KS>(tab[blockIdx.z]);
}

// number of k-steps of 4 per parity class, rounded up to the sizes the evaluation is built for
int parity_steps(int L) {
    const int s = (L + 7) / 8;
    return s == 7 ? 8 : s;
}

// the row of the sums (level or class index) that operand row rho holds: D register r of lane group
// h then stands for row 4 r + h
int parity_row(int rho, bool f64) { return f64 ? rho : 4 * (rho & 3) + (rho >> 2); }

}  // namespace

bool vertical_plain(int L, int nq, int PS, bool f64) {
    return !f64 && L <= 32 && nq >= 8 && (double)nq * PS * 8.0 < 2147483648.0;
}

// the plain forms' tables: ev [tile][k-step][64][4]; pr, per pair of levels [64][4], twice
// (project_plain_body)
static void plain_tables(int L, int nq, const std::vector<double>& ev, const std::vector<double>& pr,
                         std::vector<double>& evP, std::vector<double>& prP) {
    const int nt = (nq + 15) / 16, ns = (L + 3) / 4, np = (nq + 1) / 2;
    evP.assign((size_t)nt * ns * 64 * 4, 0.0);
    for (int tile = 0; tile < nt; ++tile)
        for (int s = 0; s < ns; ++s)
            for (int ln = 0; ln < 64; ++ln)
                for (int t = 0; t < 4; ++t) {  // C', C, S, S'
                    const int l = 16 * tile + parity_row(ln & 15, false), m = 4 * s + (ln >> 4);
                    if (l < nq && m < L) evP[(((size_t)tile * ns + s) * 64 + ln) * 4 + t] = ev[((size_t)l * 4 + t) * L + m];
                }
    prP.assign((size_t)2 * np * 64 * 4, 0.0);
    auto at = [&](int t, int l, int m) { return l < nq && m < L ? pr[((size_t)l * 5 + t) * L + m] : 0.0; };
    for (int s = 0; s < np; ++s)
        for (int ln = 0; ln < 64; ++ln)
            for (int c = 0; c < 2; ++c) {
                const int h = ln >> 4, m = 2 * parity_row(ln & 15, false) + c, l = 2 * s + (h & 1);
                double* a = &prP[((size_t)s * 64 + ln) * 4];
                double* b = &prP[((size_t)(np + s) * 64 + ln) * 4];
                a[c] = at(h < 2 ? 0 : 1, l, m);      // wC', wC''
                a[2 + c] = at(h < 2 ? 3 : 4, l, m);  // wS, wS'
                b[c] = at(2, 2 * s + h, m);          // wC
                b[2 + c] = at(3, 2 * s + h, m);      // wS
            }
}

void vertical_tables(int L, int nq, int PS, bool f64, const std::vector<double>& ev, const std::vector<double>& pr,
                   std::vector<double>& evP, std::vector<double>& prP) {
    if (vertical_plain(L, nq, PS, f64)) return plain_tables(L, nq, ev, pr, evP, prP);
    const int nh = (nq + 1) / 2, nt = (nh + 15) / 16, ns = parity_steps(L), nks = (nh + 3) / 4, mtn = (L + 31) / 32;
    evP.assign((size_t)4 * nt * ns * 64 * 2, 0.0);
    for (int t = 0; t < 4; ++t)
        for (int tile = 0; tile < nt; ++tile)
            for (int s = 0; s < ns; ++s)
                for (int ln = 0; ln < 64; ++ln)
                    for (int c = 0; c < 2; ++c) {
                        const int q = 16 * tile + parity_row(ln & 15, f64), m = 2 * (4 * s + (ln >> 4)) + c;
                        if (q < nh && m < L)
                            evP[((((size_t)t * nt + tile) * ns + s) * 64 + ln) * 2 + c] = ev[((size_t)q * 4 + t) * L + m];
                    }
    prP.assign((size_t)mtn * nks * 5 * 64 * 2, 0.0);
    for (int mt = 0; mt < mtn; ++mt)
        for (int s = 0; s < nks; ++s)
            for (int t = 0; t < 5; ++t)
                for (int ln = 0; ln < 64; ++ln)
                    for (int c = 0; c < 2; ++c) {
                        const int q = 4 * s + (ln >> 4), m = 2 * (16 * mt + parity_row(ln & 15, f64)) + c;
                        // an odd number of levels: the middle one is its own mirror
                        const double half = 2 * q + 1 == nq ? 0.5 : 1.0;
                        if (q < nh && m < L)
                            prP[((((size_t)mt * nks + s) * 5 + t) * 64 + ln) * 2 + c] =
                                half * pr[((size_t)q * 5 + t) * L + m];
                    }
}

template <typename T>
EvalArgs<T> eval_args(const DevGeom& g, const Buffers& b, void* const X[3], const void* XF,
                                   const void* XG) {
    const bool plain = vertical_plain(g.L, g.nq, g.PS, sizeof(T) == 8);
    const int nt = ((plain ? g.nq : (g.nq + 1) / 2) + 15) / 16, mg = (g.P + 15) / 16;
    EvalArgs<T> a;
    a.g = g;
    // one wave per 16 modes while those fill the chip, else the parts and then the tiles split too
    a.NP = mg >= 2048 ? 1 : 3;
    a.TS = 1;
    while (a.TS < nt && mg * a.NP * a.TS < 2048) ++a.TS;
    a.nwork = mg * a.NP * a.TS;
    a.per = ((a.nwork + 3) / 4 + 7) / 8;
    a.Xt = (const cpx<T>*)X[0];
    a.Xf = (const cpx<T>*)X[1];
    a.Xg = (const cpx<T>*)X[2];
    a.XF = (const cpx<T>*)XF;
    a.XG = (const cpx<T>*)XG;
    a.tab = (const T*)b.evP;
    a.evtab = (const T*)b.evtab;
    a.kx = (const T*)b.kx;
    a.ky = (const T*)b.ky;
    a.lev = (cpx<T>*)b.lev;
    return a;
}

template <typename T>
ProjectArgs<T> project_args(const DevGeom& g, const Buffers& b, double Pr, void* const Nout[3],
                                         void* NFo, void* NGo) {
    const int nh = (g.nq + 1) / 2, mg = (g.P + 15) / 16;
    ProjectArgs<T> a;
    a.g = g;
    a.nks = (nh + 3) / 4;
    a.per = (mg + 7) / 8;
    a.D = (const cpx<T>*)b.lev;
    a.fgw = (const cpx<T>*)b.fgw;
    a.tab = (const T*)b.prP;
    a.prtab = (const T*)b.prtab;
    a.kx = (const T*)b.kx;
    a.ky = (const T*)b.ky;
    a.Pr = (T)Pr;
    a.Nt = (cpx<T>*)Nout[0];
    a.Nf = (cpx<T>*)Nout[1];
    a.Ng = (cpx<T>*)Nout[2];
    a.NF = (cpx<T>*)NFo;
    a.NG = (cpx<T>*)NGo;
    return a;
}

// batch: nullptr for one run (arguments a), else B members' arguments on the device, of a's launch shape
template <typename T>
void launch_eval(const EvalArgs<T>& a, const EvalArgs<T>* batch, int B, hipStream_t s) {
    const dim3 grid(8 * a.per + 1, 1, B);
#define RBC_EVP(NSV, PV)                                                                                  \
    if (batch) hipLaunchKernelGGL((k_eval_parity_batch<T, NSV, PV>), grid, dim3(256), 0, s, batch);       \
    else hipLaunchKernelGGL((k_eval_parity<T, NSV, PV>), grid, dim3(256), 0, s, a)
#define RBC_EVP2(NSV)          \
    if (a.g.L % 2 == 0) {      \
        RBC_EVP(NSV, true);    \
    } else {                   \
        RBC_EVP(NSV, false);   \
    }
    if constexpr (sizeof(T) == 4) {
        if (vertical_plain(a.g.L, a.g.nq, a.g.PS, false)) {
#define RBC_EVPL(NSV)                                                                                     \
    case NSV:                                                                                             \
        if (batch) hipLaunchKernelGGL(k_eval_plain_batch<NSV>, grid, dim3(256), 0, s, batch);             \
        else hipLaunchKernelGGL(k_eval_plain<NSV>, grid, dim3(256), 0, s, a);                             \
        break;
            switch ((a.g.L + 3) / 4) {
                RBC_EVPL(1) RBC_EVPL(2) RBC_EVPL(3) RBC_EVPL(4) RBC_EVPL(5) RBC_EVPL(6) RBC_EVPL(7) RBC_EVPL(8)
            }
#undef RBC_EVPL
            return;
        }
    }
    switch (parity_steps(a.g.L)) {
        case 1: RBC_EVP2(1); break;
        case 2: RBC_EVP2(2); break;
        case 3: RBC_EVP2(3); break;
        case 4: RBC_EVP2(4); break;
        case 5: RBC_EVP2(5); break;
        case 6: RBC_EVP2(6); break;
        default: RBC_EVP2(8); break;
    }
#undef RBC_EVP2
#undef RBC_EVP
}

template <typename T>
void launch_project(const ProjectArgs<T>& a, const ProjectArgs<T>* batch, int B, hipStream_t s) {
    const dim3 grid(8 * a.per + 1, (a.g.L + 31) / 32, B);
    if constexpr (sizeof(T) == 4) {
        if (vertical_plain(a.g.L, a.g.nq, a.g.PS, false)) {
            // one wave per 16 modes while those fill the chip, else four
#define RBC_PPL(KSV)                                                                                      \
    if (batch) hipLaunchKernelGGL(k_project_plain_batch<KSV>, grid, dim3(64 * KSV), 0, s, batch);         \
    else hipLaunchKernelGGL(k_project_plain<KSV>, grid, dim3(64 * KSV), 0, s, a)
            if ((a.g.P + 63) / 64 >= 512) {
                RBC_PPL(1);
            } else {
                RBC_PPL(4);
            }
#undef RBC_PPL
            return;
        }
    }
#define RBC_PRP(KSV)                                                                                       \
    if (batch) hipLaunchKernelGGL((k_project_parity_batch<T, KSV>), grid, dim3(64 * KSV), 0, s, batch);    \
    else hipLaunchKernelGGL((k_project_parity<T, KSV>), grid, dim3(64 * KSV), 0, s, a)
    // one wave per 16 modes while those fill the chip, else the levels split (us, KS = 1 / 2 / 4): 1024 x 128 x 40
    // FP32 74.4 / 76.2 / 79.0, 256^2 x 24 FP64 32.2 / 29.9 / 34.1, 64^2 x 8 FP64 9.5 / 8.6 / 8.6
    const int work = (a.g.P + 15) / 16 * (int)grid.y;
    if (work >= 2048) {
        RBC_PRP(1);
    } else if (work >= 512) {
        RBC_PRP(2);
    } else {
        RBC_PRP(4);
    }
#undef RBC_PRP
}

#define RBC_INST(T)                                                                                                   \
    template EvalArgs<T> eval_args<T>(const DevGeom&, const Buffers&, void* const[3], const void*,       \
                                                   const void*);                                                      \
    template ProjectArgs<T> project_args<T>(const DevGeom&, const Buffers&, double, void* const[3],      \
                                                         void*, void*);                                               \
    template void launch_eval<T>(const EvalArgs<T>&, const EvalArgs<T>*, int, hipStream_t);        \
    template void launch_project<T>(const ProjectArgs<T>&, const ProjectArgs<T>*, int, hipStream_t);
RBC_INST(float)
RBC_INST(double)
#undef RBC_INST

}  // namespace rbc
