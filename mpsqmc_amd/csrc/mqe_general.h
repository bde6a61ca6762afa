// mqe_general.h -- the general walker kernel (any couplings, bonds, field and
// precision): one 256-thread workgroup owns one walker for a whole step, with
// the operands in global memory.  The algorithm is described in mqe_engine.hip.
#ifndef MQE_GENERAL_H
#define MQE_GENERAL_H

#include "mqe_kernels.h"

namespace mqe {

struct UniDims {  // bond dimensions in LDS, read as uniform values
    const int *p;
    __device__ __forceinline__ int operator[](int k) const { return uni(p[k]); }
};

// ---------------------------------------------------------------------------
// per-walker context
// ---------------------------------------------------------------------------
// CH: the products are chained in registers (chain2, chain2_16); the host selects
// this instance only when every trial and walker bond is at most 64.
template <typename T, bool CH>
struct Ctx {
    const Sys *S;
    const T *trial;
    T *phi, *Lenv, *Renv;
    const long *woff, *eoff, *moff;
    UniDims tv, wv;      // LDS copies of bond dims
    ScratchLayout sl;
    T *ts;               // T scratch
    double *ds;          // double scratch
    double *red;         // LDS reduction scratch (>= MQE_NT + 16*MQE_WAVES)
    long qlds_doubles;   // dynamic LDS: the workspace of the LQ (0: none)
    int tile;            // output tile shape of the FP32 matrix-core products (TILE_*)

    const float *trialT; // FP32: the trial with every T_k[s] transposed (t_{k+1} x t_k), or nullptr

    __device__ T *site(int k) const { return phi + uni(woff[k]); }
    __device__ const T *tsite(int k) const { return trial + uni(S->toff[k]); }
    // site k of the trial as the second operand of a product T_k[s] F: FP32 takes
    // the transposed copy (four values along the inner index per load), FP64 the
    // plain one (its inner index is strided over the lanes)
    static constexpr bool TRT = sizeof(T) == sizeof(float);
    __device__ const T *tsiteR(int k) const {
        if constexpr (TRT) return trialT + uni(S->toff[k]);
        else return tsite(k);
    }

    __device__ T *Lk(int k) const { return Lenv + uni(eoff[k]); }
    __device__ T *Rk(int k) const { return Renv + uni(eoff[k]); }
    __device__ T *Mk(int k) const { return Renv + uni(moff[k]); }  // right norm environment (w_k x w_k)
};

// Chained-product issue functions (CH instance only): they start their items at
// wave wave0, return the wave for the next independent call and leave the
// workgroup barrier to the caller.
//
// G(s', s) = T_i[s']^T L_i phi_i[s] (t_{i+1} x w_{i+1}) into out + s' ssp + s ss
// (ld ldo).  One intermediate L_i phi_i[s] feeds both s' when the walker bond
// spans two 32-column strips (four items either way).
template <typename T, bool CH>
__device__ __forceinline__ int issue_G(const Ctx<T, CH> &C, int i, const T *Lenv_i, T *out, int ldo, long ssp, long ss,
                                       int wave0) {
    if constexpr (CH) {
        const int ti = C.tv[i], tn = C.tv[i + 1], wi = C.wv[i], wn = C.wv[i + 1];
        const T *Ti = C.tsite(i), *ph = C.site(i);
        auto unit = [&](int u) {
            const int sp = u >> 1, s = u & 1;
            ChainOps<T> o;
            o.A = Lenv_i;
            o.B[0] = o.B[1] = ph + (size_t)s * wi * wn;
            o.C[0] = o.C[1] = Ti + (size_t)sp * ti * tn;
            o.D[0] = o.D[1] = out + (size_t)sp * ssp + (size_t)s * ss;
            return o;
        };
        auto both = [&](int s) {
            ChainOps<T> o;
            o.A = Lenv_i;
            o.B[0] = o.B[1] = ph + (size_t)s * wi * wn;
            o.C[0] = Ti;
            o.C[1] = Ti + (size_t)ti * tn;
            o.D[0] = out + (size_t)s * ss;
            o.D[1] = out + (size_t)ssp + (size_t)s * ss;
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wn > 32) return chain2<false, true, 1, 2>(wave0, 2, ti, wn, wi, tn, ti, wi, ti, ldo, false, both);
            if (wn == 32) return chain2<false, true, 1, 1>(wave0, 4, ti, wn, wi, tn, ti, wi, ti, ldo, false, unit);
        } else {
            if (wn > 16) return chain2_16<false, true, 1, 2, T>(wave0, 2, ti, wn, wi, tn, ti, wi, ti, ldo, false, both);
        }
        return chain2_16<false, true, 1, 1, T>(wave0, 4, ti, wn, wi, tn, ti, wi, ti, ldo, false, unit);
    }
    return wave0;
}

// V(t', t) = T_j[t'] R_{j+1} phi_j[t]^T (t_j x w_j) into the V scratch (see compute_V).
template <typename T, bool CH>
__device__ __forceinline__ int issue_V(const Ctx<T, CH> &C, int j, int wave0) {
    if constexpr (CH) {
        constexpr bool TRT = Ctx<T, CH>::TRT;
        const int tj = C.tv[j], tn = C.tv[j + 1], wj = C.wv[j], wn = C.wv[j + 1], ldc = TRT ? tn : tj;
        const T *R = C.Rk(j + 1), *ph = C.site(j), *TTj = C.tsiteR(j);
        T *V = C.ts + C.sl.V;
        auto unit = [&](int u) {
            const int tp = u >> 1, t = u & 1;
            ChainOps<T> o;
            o.A = R;
            o.B[0] = o.B[1] = ph + (size_t)t * wj * wn;
            o.C[0] = o.C[1] = TTj + (size_t)tp * tj * tn;
            o.D[0] = o.D[1] = V + (size_t)tp * tj * 2 * wj + (size_t)t * tj * wj;
            return o;
        };
        auto both = [&](int t) {
            ChainOps<T> o;
            o.A = R;
            o.B[0] = o.B[1] = ph + (size_t)t * wj * wn;
            o.C[0] = TTj;
            o.C[1] = TTj + (size_t)tj * tn;
            o.D[0] = V + (size_t)t * tj * wj;
            o.D[1] = V + (size_t)tj * 2 * wj + (size_t)t * tj * wj;
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wj > 32) return chain2<true, TRT, 1, 2>(wave0, 2, tn, wj, wn, tj, tn, wj, ldc, tj, false, both);
            if (wj == 32) return chain2<true, TRT, 1, 1>(wave0, 4, tn, wj, wn, tj, tn, wj, ldc, tj, false, unit);
        } else {
            if (wj > 16) return chain2_16<true, TRT, 1, 2, T>(wave0, 2, tn, wj, wn, tj, tn, wj, ldc, tj, false, both);
        }
        return chain2_16<true, TRT, 1, 1, T>(wave0, 4, tn, wj, wn, tj, tn, wj, ldc, tj, false, unit);
    }
    return wave0;
}

// Y = L_i phi_i (t_i x 2 w_{i+1});  G = T_i^T Y (2 t_{i+1} x 2 w_{i+1}), block
// (s', s) = T_i[s']^T L_i phi_i[s] at G + s' t + s w (2t), ld 2t.
template <typename T, bool CH>
__device__ __forceinline__ void compute_G(const Ctx<T, CH> &C, int i, const T *Lenv_i) {
    const int ti = C.tv[i], tn = C.tv[i + 1], wi = C.wv[i], wn = C.wv[i + 1];
    T *Y = C.ts + C.sl.Y, *G = C.ts + C.sl.G;
    if constexpr (CH) {
        issue_G(C, i, Lenv_i, G, 2 * tn, tn, (long)wn * 2 * tn, 0);
        __syncthreads();
        return;
    }
    gemm<false, false, T>(ti, 2 * wn, wi, Lenv_i, ti, C.site(i), wi, Y, ti, false, C.tile);
    __syncthreads();
    gemm<true, false, T>(2 * tn, 2 * wn, ti, C.tsite(i), ti, Y, ti, G, 2 * tn, false, C.tile);
    __syncthreads();
}

// The four blocks G(s', s) of bond i+1 as contiguous channels ch = 2 s' + s
// (t_{i+1} x w_{i+1}, ld t_{i+1}) at A.  CH: no barrier at the end (the
// caller's), the return value is the wave for the next independent call.
template <typename T, bool CH>
__device__ __forceinline__ int compute_G_channels(const Ctx<T, CH> &C, int i, T *A, int wave0 = 0) {
    const int tn = C.tv[i + 1], wn = C.wv[i + 1];
    if constexpr (CH) return issue_G(C, i, C.Lk(i), A, tn, 2L * tn * wn, (long)tn * wn, wave0);
    compute_G(C, i, C.Lk(i));
    const T *G = C.ts + C.sl.G;
    for (int e = threadIdx.x; e < 4 * tn * wn; e += MQE_NT) {
        const int ch = e / (tn * wn), r = e % (tn * wn), a = r % tn, b = r / tn;
        const int sp = ch >> 1, s = ch & 1;
        A[e] = G[(size_t)sp * tn + (size_t)s * wn * 2 * tn + a + (size_t)2 * tn * b];
    }
    __syncthreads();
    return wave0;
}

// W[t] = R_{j+1} phi_j[t]^T (t_{j+1} x w_j);  V[t'] = T_j[t'] W (t_j x 2 w_j);
// block (t', t) at V + t' (t_j 2 w_j) + t (t_j w_j), ld t_j.
template <typename T, bool CH>
__device__ __forceinline__ void compute_V(const Ctx<T, CH> &C, int j) {
    if constexpr (CH) {
        issue_V(C, j, 0);
        __syncthreads();
        return;
    }
    const int tj = C.tv[j], tn = C.tv[j + 1], wj = C.wv[j], wn = C.wv[j + 1];
    T *W = C.ts + C.sl.W, *V = C.ts + C.sl.V;
    const T *R = C.Rk(j + 1), *ph = C.site(j);
    gemm_batch<false, true, T>(2, tn, wj, wn, R, tn, 0, ph, wj, (long)wj * wn, W, tn, (long)tn * wj, false, C.tile);
    __syncthreads();
    const T *Tj = C.tsite(j);
    gemm_batch<false, false, T>(2, tj, 2 * wj, tn, Tj, tj, (long)tj * tn, W, tn, 0, V, tj, (long)tj * 2 * wj, false,
                                C.tile);
    __syncthreads();
}

// Carry four channels (t_k x w_k, ld t_k, contiguous at src) through site k
// into dst (t_{k+1} x w_{k+1}): dst_ch = sum_s T_k[s]^T src_ch phi_k[s].
template <typename T, bool CH>
__device__ __forceinline__ void carry_channels(const Ctx<T, CH> &C, int k, const T *src, T *dst) {
    constexpr int nch = 4;
    const int tk = C.tv[k], tn = C.tv[k + 1], wk = C.wv[k], wn = C.wv[k + 1];
    const T *Tk = C.tsite(k);
    if constexpr (CH) {
        const T *ph = C.site(k);
        auto unit = [&](int ch) {
            ChainOps<T> o;
            o.A = src + (size_t)ch * tk * wk;
            o.B[0] = ph;
            o.B[1] = ph + (size_t)wk * wn;
            o.C[0] = Tk;
            o.C[1] = Tk + (size_t)tk * tn;
            o.D[0] = o.D[1] = dst + (size_t)ch * tn * wn;
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wn >= 32) {
                chain2<false, true, 2, 1>(0, nch, tk, wn, wk, tn, tk, wk, tk, tn, false, unit);
                __syncthreads();
                return;
            }
        }
        chain2_16<false, true, 2, 1, T>(0, nch, tk, wn, wk, tn, tk, wk, tk, tn, false, unit);
        __syncthreads();
        return;
    }
    T *Y = C.ts + C.sl.Y4;  // Y_ch = src_ch phi_k (tk x 2 wn), the four channels one after the other
    const long sy = (long)tk * 2 * wn;
    gemm_batch<false, false, T>(nch, tk, 2 * wn, wk, src, tk, (long)tk * wk, C.site(k), wk, 0, Y, tk, sy, false,
                                C.tile);
    __syncthreads();
    // dst_ch = T_k[0]^T Y_ch[0] + T_k[1]^T Y_ch[1], one accumulation chain per output tile
    gemm2<true, false, T>(tn, wn, tk, Tk, Tk + (size_t)tk * tn, tk, Y, Y + (size_t)tk * wn, tk, dst, tn, C.tile, nch, 0,
                          sy, (long)tn * wn);
    __syncthreads();
}

// Carry nch channels of a right part (t_{k+1} x w_{k+1}, ld t_{k+1}, contiguous at
// src) through site k into dst (t_k x w_k): dst_ch = sum_s T_k[s] src_ch phi_k[s]^T.
template <typename T, bool CH>
__device__ __forceinline__ void carry_left(const Ctx<T, CH> &C, int k, const T *src, T *dst, int nch) {
    const int tk = C.tv[k], tn = C.tv[k + 1], wk = C.wv[k], wn = C.wv[k + 1];
    const T *ph = C.site(k);
    if constexpr (CH) {
        constexpr bool TRT = Ctx<T, CH>::TRT;
        const int ldc = TRT ? tn : tk;
        const T *TTk = C.tsiteR(k);
        auto unit = [&](int ch) {
            ChainOps<T> o;
            o.A = src + (size_t)ch * tn * wn;
            o.B[0] = ph;
            o.B[1] = ph + (size_t)wk * wn;
            o.C[0] = TTk;
            o.C[1] = TTk + (size_t)tk * tn;
            o.D[0] = o.D[1] = dst + (size_t)ch * tk * wk;
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wk >= 32) {
                chain2<true, TRT, 2, 1>(0, nch, tn, wk, wn, tk, tn, wk, ldc, tk, false, unit);
                __syncthreads();
                return;
            }
        }
        chain2_16<true, TRT, 2, 1, T>(0, nch, tn, wk, wn, tk, tn, wk, ldc, tk, false, unit);
        __syncthreads();
        return;
    }
    T *Y = C.ts + C.sl.Y4;  // Y_ch[s] = src_ch phi_k[s]^T, the two blocks of a channel one after the other
    const long sy = (long)tn * 2 * wk;
#pragma nounroll
    for (int s = 0; s < 2; ++s)
        gemm_batch<false, true, T>(nch, tn, wk, wn, src, tn, (long)tn * wn, ph + (size_t)s * wk * wn, wk, 0,
                                   Y + (size_t)s * tn * wk, tn, sy, false, C.tile);
    __syncthreads();
    const T *Tk = C.tsite(k);
    gemm2<false, false, T>(tk, wk, tn, Tk, Tk + (size_t)tk * tn, tk, Y, Y + (size_t)tn * wk, tn, dst, tk, C.tile, nch,
                           0, sy, (long)tk * wk);
    __syncthreads();
}

// Two-site mixed tensor M[(s'+2t')*4 + (s+2t)] = <G(s',s), V(t',t)> at a bond
// with trial dim tb and walker dim wb.  g[ch], ch = 2 s' + s, with leading dim gld.
template <typename T, bool CH>
// Rout (or nullptr): also writes the right environment V(0,0) + V(1,1) there.
__device__ __forceinline__ void pair_tensor(const Ctx<T, CH> &C, int tb, int wb, const T *const g[4], int gld, double *M,
                                            T *Rout = nullptr) {
    const T *V = C.ts + C.sl.V;
    double acc[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.0;
    const int nel = tb * wb;
    // two elements of a thread per pass, the loads of both before the store to
    // Rout (which the compiler cannot separate from them); the second index is
    // clamped into the block, its element skipped below (same order of sums)
    for (int e0 = threadIdx.x; e0 < nel; e0 += 2 * MQE_NT) {
        T gt[2][4], vt[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = min(e0 + u * MQE_NT, nel - 1);
            const int a = e % tb, b = e / tb;
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                const int tp = ch >> 1, t = ch & 1;
                gt[u][ch] = g[ch][a + (size_t)gld * b];
                vt[u][ch] = V[(size_t)tp * tb * 2 * wb + (size_t)t * tb * wb + a + (size_t)tb * b];
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = e0 + u * MQE_NT;
            if (e < nel) {
                if (Rout) Rout[e] = vt[u][0] + vt[u][3];
#pragma unroll
                for (int sp = 0; sp < 2; ++sp)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int tp = 0; tp < 2; ++tp)
#pragma unroll
                            for (int t = 0; t < 2; ++t)
                                acc[(sp + 2 * tp) * 4 + (s + 2 * t)] +=
                                    (double)gt[u][2 * sp + s] * (double)vt[u][2 * tp + t];
            }
        }
    }
    block_sum_n<16>(acc, C.red);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < 16; ++q) M[q] = acc[q];
    }
    __syncthreads();
}

// Bond energies <trial|S_i . S_j|phi> of a site j with partners further left take the
// three operator channels of site j (R[0] = S^z, R[1] = S^-, R[2] = S^+ applied at site
// j; t x w, ld t, contiguous), carried left to the partner's bond i + 1, and the blocks
// G(s', s) of site i there:
// S_i . S_j = S^z S^z + (S^+ S^- + S^- S^+) / 2, with S^z = diag(-1/2, 1/2),
// S^+ = |1><0|, S^- = |0><1| in the basis ordered by m (OpSz.cpp, OpSx.cpp,
// OpISy.cpp).

// The channels at site j's own bond from its blocks V(t', t); Rout (or nullptr): also
// writes R_j = V(0,0) + V(1,1) there.  Ends with a barrier.
template <typename T, bool CH>
__device__ __forceinline__ void operator_channels(const Ctx<T, CH> &C, int tb, int wb, T *R, T *Rout) {
    const T *V = C.ts + C.sl.V;
    const int n = tb * wb;
    const T *V00 = V, *V01 = V + n, *V10 = V + 2 * (size_t)n, *V11 = V + 3 * (size_t)n;  // V(t', t) at t' 2 n + t n
    // two elements of a thread per pass, loads before the stores (as in
    // pair_tensor; the clamped second index is skipped below)
    for (int e0 = threadIdx.x; e0 < n; e0 += 2 * MQE_NT) {
        T v00[2], v11[2], v01[2], v10[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = min(e0 + u * MQE_NT, n - 1);
            v00[u] = V00[e];
            v11[u] = V11[e];
            v01[u] = V01[e];
            v10[u] = V10[e];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = e0 + u * MQE_NT;
            if (e < n) {
                R[e] = (T)0.5 * (v11[u] - v00[u]);
                R[n + e] = v01[u];
                R[2 * (size_t)n + e] = v10[u];
                if (Rout) Rout[e] = v00[u] + v11[u];
            }
        }
    }
    __syncthreads();
}

// This thread's part of the bond energy of (i, j): the channels R at bond i + 1 with
// the blocks G(s', s) of site i in the G scratch (block at s' t + s 2 t w, ld 2 t).
template <typename T, bool CH>
__device__ __forceinline__ double pair_energy_part(const Ctx<T, CH> &C, int tb, int wb, const T *R) {
    const T *G = C.ts + C.sl.G;
    const int n = tb * wb;
    const size_t os = (size_t)wb * 2 * tb;
    double acc = 0.0;
    for (int e = threadIdx.x; e < n; e += MQE_NT) {
        const int a = e % tb, b = e / tb;
        const size_t o = a + (size_t)2 * tb * b;
        const T g00 = G[o], g01 = G[o + os], g10 = G[o + tb], g11 = G[o + tb + os];
        const T rz = R[e], rm = R[n + e], rp = R[2 * (size_t)n + e];
        acc += 0.5 * (((double)g11 - (double)g00) * (double)rz + (double)g10 * (double)rm + (double)g01 * (double)rp);
    }
    return acc;
}

// The four blocks G(s', s) of site `first` carried to the left of site `bond`
// (contiguous channels at A, B is the other buffer); first < 0: none.
template <typename T>
struct Carried {
    int first, bond;
    T *A, *B;
};

// Mixed tensor for the pair (i, j) from L_i, sites i..j and R_{j+1}.  `more`: the
// next coupling has the same first site and will take the channels on from bond
// j (in a torus or a frustrated lattice a site has several partners to its right:
// 85 instead of 248 carries in the 4x4 torus with diagonals; with the same for
// the energy and uniform addresses a step of 48 walkers at D = 20 in FP64 went
// from 7.6 to 3.25 ms).
template <typename T, bool CH>
__device__ __forceinline__ void pair_for_coupling(const Ctx<T, CH> &C, int i, int j, bool more, Carried<T> &cr,
                                                  double *M) {
    const int tn = C.tv[i + 1], wn = C.wv[i + 1];
    const T *g[4];
    int gld;
    if (j == i + 1 && !more) {
        T *G = C.ts + C.sl.G;
        if constexpr (CH) {  // G and V in one barrier interval
            issue_V(C, j, issue_G(C, i, C.Lk(i), G, 2 * tn, tn, (long)wn * 2 * tn, 0));
            __syncthreads();
        } else {
            compute_G(C, i, C.Lk(i));
            compute_V(C, j);
        }
        for (int ch = 0; ch < 4; ++ch) {
            const int sp = ch >> 1, s = ch & 1;
            g[ch] = G + (size_t)sp * tn + (size_t)s * wn * 2 * tn;
        }
        gld = 2 * tn;
    } else {
        // the four blocks as contiguous channels (ch = 2 s' + s), carried to bond j
        int wq = 0;
        if (cr.first != i || cr.bond > j) {
            wq = compute_G_channels(C, i, cr.A);
            cr.first = i;
            cr.bond = i + 1;
        }
        if constexpr (CH) {  // G channels and V in one barrier interval
            issue_V(C, j, wq);
            __syncthreads();
        }
        for (; cr.bond < j; ++cr.bond) {
            carry_channels(C, cr.bond, cr.A, cr.B);
            T *t = cr.A; cr.A = cr.B; cr.B = t;
        }
        const int tb = C.tv[j], wb = C.wv[j];
        for (int ch = 0; ch < 4; ++ch) g[ch] = cr.A + (size_t)ch * tb * wb;
        gld = tb;
        if constexpr (!CH) compute_V(C, j);
    }
    pair_tensor(C, C.tv[j], C.wv[j], g, gld, M);
}

// L_{k+1} = sum_s T_k[s]^T L_k phi_k[s]
template <typename T, bool CH>
__device__ __forceinline__ int issue_L(const Ctx<T, CH> &C, int k, int wave0) {
    if constexpr (CH) {
        const int tk = C.tv[k], tn = C.tv[k + 1], wk = C.wv[k], wn = C.wv[k + 1];
        const T *ph = C.site(k), *Tk = C.tsite(k);
        auto unit = [&](int) {
            ChainOps<T> o;
            o.A = C.Lk(k);
            o.B[0] = ph;
            o.B[1] = ph + (size_t)wk * wn;
            o.C[0] = Tk;
            o.C[1] = Tk + (size_t)tk * tn;
            o.D[0] = o.D[1] = C.Lk(k + 1);
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wn >= 32) return chain2<false, true, 2, 1>(wave0, 1, tk, wn, wk, tn, tk, wk, tk, tn, true, unit);
        }
        return chain2_16<false, true, 2, 1, T>(wave0, 1, tk, wn, wk, tn, tk, wk, tk, tn, true, unit);
    }
    return wave0;
}

template <typename T, bool CH>
__device__ __forceinline__ void advance_L(const Ctx<T, CH> &C, int k) {
    if constexpr (CH) {
        issue_L(C, k, 0);
        __syncthreads();
        return;
    }
    const int tk = C.tv[k], tn = C.tv[k + 1], wk = C.wv[k], wn = C.wv[k + 1];
    T *Y = C.ts + C.sl.Y;
    gemm<false, false, T>(tk, 2 * wn, wk, C.Lk(k), tk, C.site(k), wk, Y, tk, false, C.tile);
    __syncthreads();
    const T *Tk = C.tsite(k);
    T *Ln = C.Lk(k + 1);
    gemm2<true, false, T>(tn, wn, tk, Tk, Tk + (size_t)tk * tn, tk, Y, Y + (size_t)tk * wn, tk, Ln, tn, C.tile);
    __syncthreads();
}

// R_k = sum_t T_k[t] R_{k+1} phi_k[t]^T (the diagonal blocks of V at bond k)
template <typename T, bool CH>
__device__ __forceinline__ int issue_R(const Ctx<T, CH> &C, int k, int wave0) {
    if constexpr (CH) {
        const int tk = C.tv[k], tn = C.tv[k + 1], wk = C.wv[k], wn = C.wv[k + 1];
        constexpr bool TRT = Ctx<T, CH>::TRT;
        const int ldc = TRT ? tn : tk;
        const T *ph = C.site(k), *TTk = C.tsiteR(k);
        auto unit = [&](int) {
            ChainOps<T> o;
            o.A = C.Rk(k + 1);
            o.B[0] = ph;
            o.B[1] = ph + (size_t)wk * wn;
            o.C[0] = TTk;
            o.C[1] = TTk + (size_t)tk * tn;
            o.D[0] = o.D[1] = C.Rk(k);
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wk >= 32) return chain2<true, TRT, 2, 1>(wave0, 1, tn, wk, wn, tk, tn, wk, ldc, tk, true, unit);
        }
        return chain2_16<true, TRT, 2, 1, T>(wave0, 1, tn, wk, wn, tk, tn, wk, ldc, tk, true, unit);
    }
    return wave0;
}

template <typename T, bool CH>
__device__ __forceinline__ void rebuild_R(const Ctx<T, CH> &C, int k) {
    if constexpr (CH) {
        issue_R(C, k, 0);
        __syncthreads();
        return;
    }
    compute_V(C, k);
    const int tk = C.tv[k], wk = C.wv[k];
    const T *V = C.ts + C.sl.V;
    T *Rk = C.Rk(k);
    for (int e = threadIdx.x; e < tk * wk; e += MQE_NT) Rk[e] = V[e] + V[(size_t)tk * 2 * wk + (size_t)tk * wk + e];
    __syncthreads();
}

// Right norm environment M_k = sum_s phi_k[s] M_{k+1} phi_k[s]^T (w_k x w_k):
// the norm of the walker's part right of bond k in the current gauge.
// (CH issue function: M_{k+1} is symmetric, M_k = sum_s phi_k[s] (M_{k+1} phi_k[s]^T))
template <typename T, bool CH>
__device__ __forceinline__ int issue_M(const Ctx<T, CH> &C, int k, int wave0) {
    if constexpr (CH) {
        const int wk = C.wv[k], wn = C.wv[k + 1];
        const T *ph = C.site(k), *Mn = C.Mk(k + 1);
        T *Mk = C.Mk(k);
        auto unit = [&](int) {
            ChainOps<T> o;
            o.A = Mn;
            o.B[0] = o.C[0] = ph;
            o.B[1] = o.C[1] = ph + (size_t)wk * wn;
            o.D[0] = o.D[1] = Mk;
            return o;
        };
        if constexpr (sizeof(T) == sizeof(float)) {
            if (wk >= 32) return chain2<true, false, 2, 1>(wave0, 1, wn, wk, wn, wk, wn, wk, wk, wk, false, unit);
        }
        return chain2_16<true, false, 2, 1, T>(wave0, 1, wn, wk, wn, wk, wn, wk, wk, wk, false, unit);
    }
    return wave0;
}

template <typename T, bool CH>
__device__ __forceinline__ void advance_M(const Ctx<T, CH> &C, int k) {
    const int wk = C.wv[k], wn = C.wv[k + 1];
    T *X = C.ts + C.sl.Y;
    const T *ph = C.site(k), *Mn = C.Mk(k + 1);
    T *Mk = C.Mk(k);
    if constexpr (CH) {
        issue_M(C, k, 0);
        __syncthreads();
        return;
    }
    gemm_batch<false, false, T>(2, wk, wn, wn, ph, wk, (long)wk * wn, Mn, wn, 0, X, wk, (long)wk * wn, false, C.tile);
    __syncthreads();
    gemm2<false, true, T>(wk, wk, wn, X, X + (size_t)wk * wn, wk, ph, ph + (size_t)wk * wn, wk, Mk, wk, C.tile);
    __syncthreads();
}

// Squared norm with the left norm environment N (bond k) and the right norm
// environment M_{k+1}: sum_s tr(phi_k[s]^T N phi_k[s] M_{k+1}).
template <typename T, bool CH>
__device__ __forceinline__ double norm2_at_M(const Ctx<T, CH> &C, int k, const T *N) {
    const int wk = C.wv[k], wn = C.wv[k + 1];
    T *Z = C.ts + C.sl.Y, *Z2 = C.ts + C.sl.TMP;
    const T *ph = C.site(k), *Mn = C.Mk(k + 1);
    gemm<false, false, T>(wk, 2 * wn, wk, N, wk, ph, wk, Z, wk, false, C.tile);
    __syncthreads();
    gemm_batch<false, false, T>(2, wk, wn, wn, Z, wk, (long)wk * wn, Mn, wn, 0, Z2, wk, (long)wk * wn, false, C.tile);
    __syncthreads();
    double acc = 0.0;
    for (int e = threadIdx.x; e < wk * 2 * wn; e += MQE_NT) acc += (double)ph[e] * (double)Z2[e];
    return block_sum(acc, C.red);
}

template <typename T, bool CH>
__device__ __forceinline__ void scale_site(const Ctx<T, CH> &C, int k, double f) {
    T *ph = C.site(k);
    const int n = C.wv[k] * C.wv[k + 1] * 2;
    for (int e = threadIdx.x; e < n; e += MQE_NT) ph[e] = (T)((double)ph[e] * f);
    __syncthreads();
}

// (x[e], x[e + n]) <- (c00 x[e] + c01 x[e + n], c10 x[e] + c11 x[e + n]) for
// e < n: a 2 x 2 operator on the physical index of a site stored as two blocks
// of n.  Four elements of a thread are in flight at a time, their loads issued
// before their stores (one element at a time, every load waited for the store
// before it: the compiler cannot tell that they do not overlap).
template <typename T>
__device__ __forceinline__ void mix_pair(T *x, int n, T c00, T c01, T c10, T c11) {
    for (int e0 = threadIdx.x; e0 < n; e0 += 4 * MQE_NT) {
        T a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = e0 + q * MQE_NT;
            a[q] = e < n ? x[e] : T(0);
            b[q] = e < n ? x[e + n] : T(0);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = e0 + q * MQE_NT;
            if (e < n) {
                x[e] = c00 * a[q] + c01 * b[q];
                x[e + n] = c10 * a[q] + c11 * b[q];
            }
        }
    }
}

// phi_k[s] <- sum_s0 O[s + 2 s0] phi_k[s0]
template <typename T, bool CH>
__device__ __forceinline__ void apply_op(const Ctx<T, CH> &C, int k, const double *O) {
    const T o00 = (T)O[0], o10 = (T)O[1], o01 = (T)O[2], o11 = (T)O[3];
    mix_pair(C.site(k), C.wv[k] * C.wv[k + 1], o00, o01, o10, o11);
    __syncthreads();
}

// FP64 LQ of a site ph (wk x 2 wn): ph <- Q (right-orthonormal), LM <- Lmat (wk x wk).
// The factorisation is a serial chain of column steps; it runs with every
// column in registers where the site fits (at most 128 x 64, reflectors in LDS),
// by panels of 32 columns in registers up to 256 x 128, and over columns in LDS
// and memory above.  One step of 200 walkers of a 15-site
// ring in a field at D = 20 (two sweeps of LQ): 2121 us with the columns in LDS,
// 1634 us in registers; 128 walkers of 16 sites at D = 16 in FP64, where one or
// two walkers a step take this sweep and the others wait: 1230 and 1042 us.
// A function of its own, not inlined: its register columns in the kernel's body
// made the products of the other walkers spill (a step of the 6x6 snake at D = 128
// without canonical walkers 115 ms, 134 ms with the panels inlined).
// AQ, RQ, TAU: the walker's scratch; nq: doubles of dynamic LDS.
template <typename T, bool CH>
__device__ __noinline__ void lq_factor(T *ph_, T *LM_, double *AQ_, double *RQ_, double *TAU_, int wk_, int wn_,
                                       int Dw, int nq) {
    extern __shared__ double qlds_dyn[];
    constexpr bool PANELS = !CH;  // (chained: every bond is at most 64)
    const int wk = uni(wk_), wn = uni(wn_);
    T *ph = (T *)uni((long)ph_), *LM = (T *)uni((long)LM_);
    double *AQ = (double *)uni((long)AQ_);
    nq = uni(nq);
    const int m = 2 * wn, n = wk;
    auto load = [&](int r, int c) { return (double)ph[c + (size_t)wk * r]; };
    auto put_r = [&](int r, int c, double x) {  // Lmat = R^T
        LM[c + (size_t)n * r] = (T)x;
        if (r != c) LM[r + (size_t)n * c] = T(0);
    };
    auto put_q = [&](int r, int c, double x) { ph[c + (size_t)wk * r] = (T)x; };
    const bool fits = nq > 0 && n <= m;
    if (fits && m <= QR_REGS_M && n <= QR_REGS_N && nq >= (m <= 64 && n <= 32 ? 65 : 129) * n) {
        qr_in_regs<sizeof(T) == 8>(m, n, qlds_dyn + n, qlds_dyn, true, load, put_r, put_q);
    } else if (PANELS && fits && m <= QR_PANELS_M && n <= QR_PANELS_N && nq >= QR_PANELS_M * QR_PANEL + n) {
        qr_panels<sizeof(T) == 8>(m, n, qlds_dyn + n, qlds_dyn, AQ, load, put_r, put_q);
    } else {
        double *R = (double *)uni((long)RQ_);
        double *tau = nq > 0 ? qlds_dyn : (double *)uni((long)TAU_);
        const int D = uni(Dw), nl = nq > 0 ? min(n, (nq - D) / m) : 0;
        const QRCols col{AQ, nq > 0 ? qlds_dyn + D : nullptr, m, n - nl};
        for (int e = threadIdx.x; e < m * n; e += MQE_NT) {
            const int r = e % m, c = e / m;
            col(c)[r] = (double)ph[c + (size_t)wk * r];
        }
        __syncthreads();
        householder_qr(col, n, R, tau);
        for (int e = threadIdx.x; e < m * n; e += MQE_NT) {
            const int r = e % m, c = e / m;
            ph[c + (size_t)wk * r] = (T)col(c)[r];
        }
        for (int e = threadIdx.x; e < n * n; e += MQE_NT) {
            const int a = e % n, b = e / n;
            LM[e] = (T)R[b + (size_t)n * a];
        }
    }
    __syncthreads();
}

// LQ of site k: phi_k <- Q, phi_{k-1} <- phi_{k-1} Lmat, then
// R_k = sum_t T_k[t] R_{k+1} Q[t]^T.  Leaves V (all four blocks) computed for bond k.
template <typename T, bool CH>
__device__ __forceinline__ void lq_site(const Ctx<T, CH> &C, int k) {
    const int wk = C.wv[k], wn = C.wv[k + 1], wp = C.wv[k - 1];
    T *LM = C.ts + C.sl.LM;
    lq_factor<T, CH>(C.site(k), LM, C.ds + C.sl.AQ, C.ds + C.sl.RQ, C.ds + C.sl.TAU, wk, wn, C.S->Dw,
                     (int)C.qlds_doubles);
    // push Lmat into the left neighbour
    T *pl = C.site(k - 1), *tmp = C.ts + C.sl.TMP;
    gemm_batch<false, false, T>(2, wp, wk, wk, pl, wp, (long)wp * wk, LM, wk, 0, tmp, wp, (long)wp * wk, false, C.tile);
    __syncthreads();
    for (int e = threadIdx.x; e < 2 * wp * wk; e += MQE_NT) pl[e] = tmp[e];
    __syncthreads();
    // right environment of bond k
    compute_V(C, k);
    const int tk = C.tv[k];
    const T *V = C.ts + C.sl.V;
    T *Rk = C.Rk(k);
    for (int e = threadIdx.x; e < tk * wk; e += MQE_NT) Rk[e] = V[e] + V[(size_t)tk * 2 * wk + (size_t)tk * wk + e];
    __syncthreads();
}

// <trial|phi> and sum_s sz[s] <trial|S^z_0|phi> at site 0 (L_0 = 1, right part via R_1).
template <typename T, bool CH>
__device__ __forceinline__ void site0_overlap(const Ctx<T, CH> &C, double *ov, double *szv) {
    const int t1 = C.tv[1], w1 = C.wv[1];
    const T *T0 = C.tsite(0), *p0 = C.site(0), *R1 = C.Rk(1);
    double a[2] = {0.0, 0.0};
    for (int e = threadIdx.x; e < t1 * w1; e += MQE_NT) {
        const int al = e % t1, be = e / t1;
        const double r = (double)R1[al + (size_t)t1 * be];
        for (int s = 0; s < 2; ++s) a[s] += (double)T0[al + (size_t)t1 * s] * (double)p0[be + (size_t)w1 * s] * r;
    }
    block_sum_n<2>(a, C.red);
    *ov = a[0] + a[1];
    *szv = C.S->Sz[0] * a[0] + C.S->Sz[1] * a[1];
}

// Right-canonicalise the whole walker with R environments, normalise at site 0.
// Returns the (sign-fixed) overlap of the normalised state.
template <typename T, bool CH>
__device__ __forceinline__ double right_canonicalize(const Ctx<T, CH> &C) {
    const int L = C.S->L;
    set_one(C.Rk(L));
    for (int k = L - 1; k >= 1; --k) lq_site(C, k);
    double ov, szv;
    site0_overlap(C, &ov, &szv);
    double nrm2 = 0.0;
    {
        const T *p0 = C.site(0);
        double s = 0.0;
        for (int e = threadIdx.x; e < 2 * C.wv[1]; e += MQE_NT) s += (double)p0[e] * (double)p0[e];
        nrm2 = block_sum(s, C.red);
    }
    const double nrm = sqrt(nrm2);
    double O = ov / nrm;
    double f = 1.0 / nrm;
    if (O < 0.0) { O = -O; f = -f; }
    scale_site(C, 0, f);
    return O;
}

// Energy sweep from the right end (L_k valid for all k), see file header.
// Returns e_tot = <trial|H|phi> of the state as it was on entry and writes the
// overlap of the normalised state to *O_out, <trial|phi> before normalisation to *Ou.
template <typename T, bool CH>
__device__ __forceinline__ double energy_sweep(const Ctx<T, CH> &C, double *O_out, double *Ou, bool canon) {
    const Sys &S = *C.S;
    const int L = S.L;
    __shared__ double M[16];
    set_one(C.Rk(L));
    set_one(C.Mk(L));
    double etot = 0.0;
    for (int k = L - 1; k >= 1; --k) {
        bool nn_ready = false;   // G of the coupling (k-1, k) already formed
        bool r_pending = false;  // R_k still to be written (by the next pair tensor)
        if (canon) {
            lq_site(C, k);  // V of bond k now holds T_k R_{k+1} Q_k^T blocks
        } else {
            // light sweep: no re-orthonormalisation; site k is rescaled to the
            // Frobenius norm sqrt(w_k) of a right-canonical site when it is more
            // than a factor 4 away from it, and the factor moved into site k-1
            // (the state is unchanged).  This keeps every
            // tensor, and the environments built from them, at the magnitudes of
            // the canonical form: a unit-norm target would shrink R_k by about
            // sqrt(w) per site and underflow FP32 on long chains at large D.
            // Then R_k and the right norm environment M_k.
            {
                const int wk = C.wv[k], wn = C.wv[k + 1];
                const T *ph = C.site(k);
                double s2 = 0.0;
                for (int e = threadIdx.x; e < 2 * wk * wn; e += MQE_NT) s2 += (double)ph[e] * (double)ph[e];
                const double f = sqrt(block_sum(s2, C.red) / (double)wk);
                // only a site that has drifted by more than a factor 4 is rescaled:
                // that bounds every magnitude just as well and skips the two
                // passes over the tensors at most sites of most steps
                if (f > 0.0 && isfinite(f) && (f > 4.0 || f < 0.25)) {
                    scale_site(C, k, 1.0 / f);
                    scale_site(C, k - 1, f);
                }
            }
            if constexpr (CH) {
                // V, M_k and the nearest-neighbour G of bond k (the last coupling
                // ending at k, if it is (k-1, k)) in one barrier interval
                const int wq = issue_M(C, k, issue_V(C, k, 0));
                const int ql = uni(S.cs_ptr[k + 1]) - 1;
                if (ql >= uni(S.cs_ptr[k]) && uni(S.first[S.cs_idx[ql]]) == k - 1) {
                    const int tn = C.tv[k], wn = C.wv[k];
                    issue_G(C, k - 1, C.Lk(k - 1), C.ts + C.sl.G, 2 * tn, tn, (long)wn * 2 * tn, wq);
                    nn_ready = true;
                }
                __syncthreads();
            } else {
                compute_V(C, k);
            }
            if (uni(S.cs_ptr[k + 1]) > uni(S.cs_ptr[k])) {
                r_pending = true;  // R_k from the first pair tensor of the site
            } else {
                const int tk = C.tv[k], wk = C.wv[k];
                const T *V = C.ts + C.sl.V;
                T *Rk = C.Rk(k);
                for (int e = threadIdx.x; e < tk * wk; e += MQE_NT)
                    Rk[e] = V[e] + V[(size_t)tk * 2 * wk + (size_t)tk * wk + e];
            }
            if constexpr (!CH) advance_M(C, k);
        }
        const int q0 = uni(S.cs_ptr[k]), nall = uni(S.cs_ptr[k + 1]) - q0;
        const bool nn = nall > 0 && uni(S.first[S.cs_idx[q0 + nall - 1]]) == k - 1;
        const int nq = nn ? nall - 1 : nall;
        if (nn) {
            const int c = uni(S.cs_idx[q0 + nq]), i = k - 1;
            const int tn = C.tv[i + 1], wn = C.wv[i + 1];
            const T *g[4];
            if (!nn_ready) compute_G(C, i, C.Lk(i));
            const T *G = C.ts + C.sl.G;
            for (int ch = 0; ch < 4; ++ch) {
                const int sp = ch >> 1, s = ch & 1;
                g[ch] = G + (size_t)sp * tn + (size_t)s * wn * 2 * tn;
            }
            pair_tensor(C, C.tv[k], C.wv[k], g, 2 * tn, M, r_pending ? C.Rk(k) : nullptr);
            r_pending = false;
            double e = 0.0;
            for (int q2 = 0; q2 < 16; ++q2) e += S.SS[q2] * M[q2];
            etot += S.Jc[c] * e;
        }
        if (nq > 0) {
            // long range: the three operator channels of site k start at its bond and
            // go left once for all its partners, from the nearest to the farthest; each
            // coupling meets the blocks G of its own first site and is summed, times J,
            // in FP64 (adding J S_i of the partners up in one set of FP32 channels
            // instead rounds every coupling to the largest of them; a step of the 6x6
            // snake at D = 128, 256 walkers: 130 ms that way, 120 ms this way, of a
            // 15-site ring at D = 20, 200 walkers: 1317 and 1327 us)
            T *A = C.ts + C.sl.GcA, *B = C.ts + C.sl.GcB;
            double ep = 0.0;
            int bond = k;
            for (int q = q0 + nq - 1; q >= q0; --q) {
                const int c = uni(S.cs_idx[q]), i = uni(S.first[c]);
                const int tn = C.tv[i + 1], wn = C.wv[i + 1];
                // (i <= k - 2 and the partners differ: at least one carry, whose
                // barrier covers G)
                if constexpr (CH) issue_G(C, i, C.Lk(i), C.ts + C.sl.G, 2 * tn, tn, (long)wn * 2 * tn, 0);
                else compute_G(C, i, C.Lk(i));
                if (bond == k) operator_channels(C, C.tv[k], C.wv[k], A, r_pending ? C.Rk(k) : nullptr);
                for (; bond > i + 1; --bond) {
                    carry_left(C, bond - 1, A, B, 3);
                    T *t = A; A = B; B = t;
                }
                ep += S.Jc[c] * pair_energy_part(C, tn, wn, A);
                if (q > q0) __syncthreads();  // G is formed anew
            }
            etot += block_sum(ep, C.red);
        }
        if (S.h != 0.0) {
            // <trial|S^z_k|phi> = sum_t sz[t] <L'_k, V(t,t)>, L'_k the current-gauge left env
            compute_G(C, k - 1, C.Lk(k - 1));
            const int tk = C.tv[k], wk = C.wv[k];
            const T *G = C.ts + C.sl.G, *V = C.ts + C.sl.V;
            double a[2] = {0.0, 0.0};
            for (int e = threadIdx.x; e < tk * wk; e += MQE_NT) {
                const int al = e % tk, be = e / tk;
                const double lp = (double)G[al + (size_t)2 * tk * be] +
                                  (double)G[tk + (size_t)wk * 2 * tk + al + (size_t)2 * tk * be];
                a[0] += lp * (double)V[al + (size_t)tk * be];
                a[1] += lp * (double)V[(size_t)tk * 2 * wk + (size_t)tk * wk + al + (size_t)tk * be];
            }
            block_sum_n<2>(a, C.red);
            etot -= S.h * (S.Sz[0] * a[0] + S.Sz[1] * a[1]);
        }
    }
    double ov, szv;
    site0_overlap(C, &ov, &szv);
    if (S.h != 0.0) etot -= S.h * szv;
    double nrm2;
    if (canon) {
        const T *p0 = C.site(0);
        double s = 0.0;
        for (int e = threadIdx.x; e < 2 * C.wv[1]; e += MQE_NT) s += (double)p0[e] * (double)p0[e];
        nrm2 = block_sum(s, C.red);
    } else {
        nrm2 = norm2_at_M(C, 0, C.Lk(0));  // L_0 = 1 is also the left norm environment of site 0
    }
    const double nrm = sqrt(nrm2);
    double O = ov / nrm, f = 1.0 / nrm;
    if (O < 0.0) { O = -O; f = -f; }
    scale_site(C, 0, f);
    *O_out = O;
    *Ou = ov;
    return etot;
}

template <typename T, bool CH>
__device__ __forceinline__ void apply_field_everywhere(const Ctx<T, CH> &C) {
    const double O[4] = {C.S->ssp[0], 0.0, 0.0, C.S->ssp[1]};
    for (int k = 0; k < C.S->L; ++k) apply_op(C, k, O);
}

// combos, PDF over the grid, CDF sample and the sampled operators of one
// coupling (MPSQMC2.cpp:540-588, MPSstate.cpp:589-631) for at most 256 grid
// points: every wave computes the same result (lane q < 16 forms combo q, lane
// l owns grid points 4l .. 4l+3; wave-wide sums and scan), so no workgroup
// barrier is needed.  M: the 16 mixed matrix elements (LDS).
__device__ __forceinline__ void wave_sample(const double *M, const double *tS, const double *tU, const double *tVT,
                                            const double *grid, int Ng, double O, double u, double &pdfnorm,
                                            int &gs, double &fstar, double (&Ux)[4], double (&Vx)[4]) {
    const int lane = threadIdx.x & 63;
    double cq = 0.0;
    if (lane < 16) {
        // combos[a + 4b] = sqrt(s_a s_b) <trial| U_a (x) V_b |phi>
        const int a = lane & 3, bb = lane >> 2;
        double sacc = 0.0;
        for (int sp = 0; sp < 2; ++sp)
            for (int ss = 0; ss < 2; ++ss) {
                const double ua = tU[sp + 2 * (ss + 2 * a)];
                for (int tp = 0; tp < 2; ++tp)
                    for (int t = 0; t < 2; ++t) sacc += ua * tVT[bb + 4 * (tp + 2 * t)] * M[(sp + 2 * tp) * 4 + (ss + 2 * t)];
            }
        cq = sqrt(tS[a] * tS[bb]) * sacc;
    }
    double cb[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) cb[q] = readlane_d(cq, q);
    auto quad = [&](const double *x) {  // sum_{l,r} comb[l + 4r] x_l x_r
        double f = 0.0;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            double t = 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r) t += cb[l + 4 * r] * x[r];
            f += x[l] * t;
        }
        return f;
    };
    const double pref = 4.0 / (O * Ng);
    double pv[4], loc = 0.0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int g = 4 * lane + t;
        double v = 0.0;
        if (g < Ng) {
            const double f = quad(grid + 4 * g);
            v = (f > 0.0 ? f : 0.0) * pref;
        }
        pv[t] = v;
        loc += v;
    }
    pdfnorm = wave_sum(loc);
    const double inv = 1.0 / pdfnorm;
    double ln = 0.0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        pv[t] *= inv;
        ln += pv[t];
    }
    // count of the grid points g < Ng - 1 whose cumulative probability is <= u
    double run = wave_exclusive_scan(ln), cnt = 0.0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        run += pv[t];
        if (4 * lane + t < Ng - 1 && run <= u) cnt += 1.0;
    }
    gs = (int)wave_sum(cnt);
    const double *xs = grid + 4 * gs;
    fstar = quad(xs);
#pragma unroll
    for (int q = 0; q < 4; ++q) Ux[q] = Vx[q] = 0.0;
    for (int k = 0; k < 4; ++k) {
        const double pf = sqrt(tS[k] * 4.0) * xs[k];  // sqrt(4 S_k) x_k (MPSstate.cpp:591,616)
        for (int up = 0; up < 2; ++up)
            for (int dn = 0; dn < 2; ++dn) {
                Ux[up + 2 * dn] += pf * tU[up + 2 * (dn + 2 * k)];
                Vx[up + 2 * dn] += pf * tVT[k + 4 * (up + 2 * dn)];
            }
    }
}

template <typename T, bool CH>
__global__ __launch_bounds__(MQE_NT, 2) void walker_kernel(Sys S, Pool P, const T *trial, int flags) {
    const int n = *P.n;
    if ((int)blockIdx.x >= n) return;
    if (*P.status & 4) return;  // the population overflowed: keep the state as it was
    const int b = uni(P.list ? P.list[blockIdx.x] : (int)blockIdx.x);  // population position
    const int slot = uni(P.order[b]);
    const Ctl ctl = *P.ctl;
    const int L = S.L;

    __shared__ int tv[MQE_MAXL + 1], wv[MQE_MAXL + 1];
    __shared__ double red[MQE_NT + 16 * MQE_WAVES];
    __shared__ double M[16], comb[16];

    __shared__ int sh_tile;
    for (int k = threadIdx.x; k <= L; k += MQE_NT) {
        tv[k] = S.tvd[k];
        wv[k] = P.wvd[(size_t)slot * (L + 1) + k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int mb = 1;
        for (int k = 0; k <= L; ++k) mb = max(mb, wv[k]);
        sh_tile = S.tiles[bond_bucket(mb)];
    }
    __syncthreads();

    Ctx<T, CH> C;
    C.tile = uni(sh_tile);
    C.S = &S;
    C.trial = trial;
    C.trialT = S.trialT;
    C.phi = (T *)P.phi + (size_t)slot * P.wflat;
    C.Lenv = (T *)P.Lenv + (size_t)slot * P.eflat;
    C.Renv = (T *)P.Renv + (size_t)slot * P.eflat;
    C.woff = P.woff;
    C.eoff = P.eoff;
    C.moff = P.moff;
    C.tv = UniDims{tv};
    C.wv = UniDims{wv};
    C.sl = scratch_layout(S.Dt, S.Dw, S.Ng);
    char *base = P.scratch + (size_t)b * P.scratch_bytes;
    C.ts = (T *)base;
    long tb = (C.sl.t_total * (long)sizeof(T) + 255) & ~255L;
    C.ds = (double *)(base + tb);
    C.red = red;
    C.qlds_doubles = P.qlds;

    double w = P.w[slot];
    double O = P.O[slot];

    set_one(C.Lk(0));

    const bool prep = flags & F_PREP;
    int p = 0;  // left environments L_k are valid for k <= p
    if (!prep) {
    // ---------------- propagation (MPSQMC2.cpp:532-600) ----------------
    if (S.h != 0.0) {
        apply_field_everywhere(C);
        O = right_canonicalize(C);
    }
    // The walker is not normalised between couplings: the sampled operator of
    // the right site is scaled so that the overlap stays O (see the file
    // header), and the energy sweep takes the norm.  rv: right environments R_k are
    // valid for k >= rv.
    int rv = 1;
    Carried<T> cr{-1, 0, C.ts + C.sl.GcA, C.ts + C.sl.GcB};
    for (int c = 0; c < S.nC; ++c) {
        const int i = uni(S.first[c]), j = uni(S.second[c]), inext = uni(S.nextfirst[c]);
        const bool more = inext == i;
        // the left environments up to L_i and the right ones down to R_{j+1}: two
        // independent chains (CH: one step of each per barrier interval)
        if constexpr (CH) {
            while (p < i || rv > j + 1) {
                int wq = 0;
                if (p < i) wq = issue_L(C, p++, wq);
                if (rv > j + 1) issue_R(C, --rv, wq);
                __syncthreads();
            }
        } else {
            while (p < i) {
                advance_L(C, p);
                ++p;
            }
            while (rv > j + 1) rebuild_R(C, --rv);
        }
        pair_for_coupling(C, i, j, more, cr, M);
        const double *tS = S.tS + 4 * c, *tU = S.tU + 16 * c, *tVT = S.tVT + 16 * c;
        const double u = P.u ? P.u[(size_t)b * S.nC + c] : philox_uniform(P.seed, (uint32_t)b, (uint32_t)c, (uint32_t)ctl.step, 0u);
        double pdfnorm, fstar, Ux[4], Vx[4];
        int gs;
        if (S.Ng <= 256) {
            wave_sample(M, tS, tU, tVT, S.grid, S.Ng, O, u, pdfnorm, gs, fstar, Ux, Vx);
        } else {
            // larger grids: the workgroup forms the PDF and scans it (MPSQMC2.cpp:540-588)
            if (threadIdx.x < 16) {
                const int a = threadIdx.x & 3, bb = threadIdx.x >> 2;
                double sacc = 0.0;
                for (int sp = 0; sp < 2; ++sp)
                    for (int ss = 0; ss < 2; ++ss) {
                        const double ua = tU[sp + 2 * (ss + 2 * a)];
                        for (int tp = 0; tp < 2; ++tp)
                            for (int t = 0; t < 2; ++t)
                                sacc += ua * tVT[bb + 4 * (tp + 2 * t)] * M[(sp + 2 * tp) * 4 + (ss + 2 * t)];
                    }
                comb[threadIdx.x] = sqrt(tS[a] * tS[bb]) * sacc;
            }
            __syncthreads();
            double *pdf = C.ds + C.sl.PDF, *cum = C.ds + C.sl.CUM;
            const int Ng = S.Ng;
            const double pref = 4.0 / (O * Ng);
            double part = 0.0;
            for (int g = threadIdx.x; g < Ng; g += MQE_NT) {
                const double *x = S.grid + 4 * g;
                double f = 0.0;
                for (int l = 0; l < 4; ++l)
                    for (int r = 0; r < 4; ++r) f += comb[l + 4 * r] * x[l] * x[r];
                const double v = (f > 0.0 ? f : 0.0) * pref;
                pdf[g] = v;
                part += v;
            }
            pdfnorm = block_sum(part, red);
            const double inv = 1.0 / pdfnorm;
            for (int g = threadIdx.x; g < Ng; g += MQE_NT) pdf[g] *= inv;
            __syncthreads();
            block_inclusive_scan(Ng, pdf, cum, red);
            double cnt = 0.0;
            for (int g = threadIdx.x; g < Ng - 1; g += MQE_NT) cnt += (cum[g] <= u) ? 1.0 : 0.0;
            gs = (int)block_sum(cnt, red);
            const double *x = S.grid + 4 * gs;
            fstar = 0.0;
            for (int l = 0; l < 4; ++l)
                for (int r = 0; r < 4; ++r) fstar += comb[l + 4 * r] * x[l] * x[r];
            for (int q = 0; q < 4; ++q) Ux[q] = Vx[q] = 0.0;
            for (int k = 0; k < 4; ++k) {
                const double pf = sqrt(tS[k] * 4.0) * x[k];  // MPSstate.cpp:591,616
                for (int up = 0; up < 2; ++up)
                    for (int dn = 0; dn < 2; ++dn) {
                        Ux[up + 2 * dn] += pf * tU[up + 2 * (dn + 2 * k)];
                        Vx[up + 2 * dn] += pf * tVT[k + 4 * (up + 2 * dn)];
                    }
            }
        }
        w *= pdfnorm;
        if (threadIdx.x == 0) {
            if (P.idx) P.idx[(size_t)b * S.nC + c] = gs;
            if (!(pdfnorm > 0.0) || !isfinite(pdfnorm)) atomicOr(P.status, 1);
        }
        // the sampled operators on sites i and j (MPSstate.cpp:575-633), the right
        // one scaled by O / <trial|B(x) phi> = O / (4 f*) so that the overlap stays O;
        // for nearest neighbours whose next coupling starts right of i, the left
        // boundary moves to j: L_{i+1} = sum_{s,s0} Ux[s,s0] G(s, s0).  One pass.
        const double alpha = O / (4.0 * fstar);
        const bool nn_move = j == i + 1 && inext > i;
        {
            T *pi = C.site(i), *pj = C.site(j);
            const int bi = C.wv[i] * C.wv[i + 1], bj = C.wv[j] * C.wv[j + 1];
            const T u00 = (T)Ux[0], u10 = (T)Ux[1], u01 = (T)Ux[2], u11 = (T)Ux[3];
            const T v00 = (T)(alpha * Vx[0]), v10 = (T)(alpha * Vx[1]), v01 = (T)(alpha * Vx[2]),
                    v11 = (T)(alpha * Vx[3]);
            mix_pair(pi, bi, u00, u01, u10, u11);
            mix_pair(pj, bj, v00, v01, v10, v11);
            if (more) {  // the carried channels with the new site i
                const int nb = C.tv[j] * C.wv[j];
                mix_pair(cr.A, nb, u00, u01, u10, u11);
                mix_pair(cr.A + 2 * (size_t)nb, nb, u00, u01, u10, u11);
            } else {
                cr.first = -1;
            }
            if (nn_move) {
                const int tn = C.tv[i + 1], wn = C.wv[i + 1];
                const T *G = C.ts + C.sl.G;
                T *Ln = C.Lk(i + 1);
                for (int e = threadIdx.x; e < tn * wn; e += MQE_NT) {
                    const int a = e % tn, bq = e / tn;
                    const size_t o = a + (size_t)2 * tn * bq;
                    const T g00 = G[o], g01 = G[o + (size_t)wn * 2 * tn], g10 = G[o + tn],
                            g11 = G[o + tn + (size_t)wn * 2 * tn];
                    Ln[a + (size_t)tn * bq] = u00 * g00 + u01 * g01 + u10 * g10 + u11 * g11;
                }
            }
            __syncthreads();
        }
        p = nn_move ? i + 1 : i;  // else site i changed: L_{i+1} is rebuilt when needed
        rv = max(rv, j + 1);  // site j changed
    }
    if (S.h != 0.0) {
        apply_field_everywhere(C);
        p = 0;
    }
    }
    while (p < L - 1) {
        advance_L(C, p);
        ++p;
    }
    // ---------------- local energy (Walker.cpp:72-77) ----------------
    // (one energy sweep for both kinds of call: a second inlined copy would only
    // double the kernel's code)
    double On, Ou;
    const bool canon = prep || canon_walker(ctl, slot, P.since[slot]);
    const double e = energy_sweep(C, &On, &Ou, canon);
    if (threadIdx.x == 0) {
        P.since[slot] = canon ? 0 : P.since[slot] + 1;
        P.O[slot] = On;
        if (prep) {
            P.EL[slot] = e / O;  // stored overlap, MPSQMC2.cpp:447 / Walker.cpp:72-77
        } else {
            P.w[slot] = w;
            P.EL[slot] = e / Ou;
            if (!isfinite(w)) atomicOr(P.status, 2);
        }
    }
}
}  // namespace mqe

#endif
