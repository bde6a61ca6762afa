// mqe_svd.h -- FP64 factorisations of one matrix per workgroup for the device
// recompression of walkers (MPSstate::CompressState, MPSstate.cpp:379-404; the
// two-site SVD of TwoSiteObject.cpp:119-184): the triangular factor of a
// Householder QR and a one-sided Jacobi SVD (Hestenes).
//
// Jacobi: the columns of X are rotated pairwise until they are mutually
// orthogonal, X_in W = X_out with W orthogonal, so column j of X_out is the left
// singular vector U_j times s_j.  Only U and s are needed (the caller forms the
// other factor as U^T theta), so W is not kept.  All column pairs of one round
// of a round-robin tournament are disjoint and rotate in parallel (a group of
// lanes per pair), one workgroup barrier per round; a sweep is one tournament,
// and sweeps repeat until one rotates nothing.
//
// What bounds it: the chain of one round (LDS read, three dot products, the
// rotation's square roots and divisions, LDS write, barrier), a few hundred
// cycles that nothing overlaps.  Hence few columns (the caller reduces the
// two-site matrix to its rank first), columns in LDS, the two columns of a pair
// in registers between the dot products and the rotation, and sums by lane
// exchange inside 16-lane rows.
#ifndef MQE_SVD_H
#define MQE_SVD_H

#include "mqe_device.h"

namespace mqe {

// Rotation of columns x, y (rows long) by a group of TPP lanes (lane gl); NE > 0:
// rows <= TPP NE, the elements stay in registers; NE = 0: any length.
// Returns whether the pair was rotated.
template <int TPP, int NE>
__device__ __forceinline__ bool jacobi_pair(double *x, double *y, int rows, int gl, double tol2) {
    constexpr int N = NE > 0 ? NE : 1;
    double u[N], v[N], a = 0.0, b = 0.0, g = 0.0;
    if constexpr (NE > 0) {
#pragma unroll
        for (int t = 0; t < N; ++t) {
            const int i = gl + TPP * t;
            u[t] = i < rows ? x[i] : 0.0;
            v[t] = i < rows ? y[i] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < N; ++t) {
            a += u[t] * u[t];
            b += v[t] * v[t];
            g += u[t] * v[t];
        }
    } else {
        for (int i = gl; i < rows; i += TPP) {
            const double p = x[i], q = y[i];
            a += p * p;
            b += q * q;
            g += p * q;
        }
    }
    a = lanes_sum<TPP>(a);
    b = lanes_sum<TPP>(b);
    g = lanes_sum<TPP>(g);
    if (g == 0.0 || g * g <= tol2 * (a * b)) return false;
    // The angle needs no more than the hardware's approximate reciprocal and
    // root (about 1e-7): what is left of g is removed by the next sweep.  Only
    // c^2 + s^2 = 1 has to hold to rounding: c = (1 + t^2)^(-1/2) takes a third
    // order correction.
    const double zeta = 0.5 * (b - a) * __builtin_amdgcn_rcp(g), z2 = 1.0 + zeta * zeta;
    const double root = z2 < 1e300 ? z2 * __builtin_amdgcn_rsq(z2) : fabs(zeta);
    const double t = copysign(__builtin_amdgcn_rcp(fabs(zeta) + root), zeta);
    const double q2 = 1.0 + t * t, c0 = __builtin_amdgcn_rsq(q2), er = 1.0 - q2 * c0 * c0;
    const double c = c0 + c0 * er * (0.5 + 0.375 * er), s = c * t;
    if constexpr (NE > 0) {
#pragma unroll
        for (int t2 = 0; t2 < N; ++t2) {
            const int i = gl + TPP * t2;
            if (i < rows) {
                x[i] = c * u[t2] - s * v[t2];
                y[i] = s * u[t2] + c * v[t2];
            }
        }
    } else {
        for (int i = gl; i < rows; i += TPP) {
            const double p = x[i], q = y[i];
            x[i] = c * p - s * q;
            y[i] = s * p + c * q;
        }
    }
    return true;
}

template <int TPP, int NE>
__device__ __forceinline__ void jacobi_sweeps(double *X, int rows, int cols, int ld, int *sh_flag) {
    const int tid = threadIdx.x, gl = tid & (TPP - 1), grp = tid / TPP;
    constexpr int groups = MQE_NT / TPP;
    const int np = (cols + 1) / 2;  // pairs per round
    const int pm = 2 * np - 1;      // players (cols rounded up to even; one dummy if odd) minus the fixed one
    // orthogonality tolerance: the rounding floor of a dot product grows like sqrt(rows)
    const double tol = 1e-15 * fmax(1.0, sqrt((double)rows) * 0.25), tol2 = tol * tol;
    for (int sweep = 0; sweep < 60; ++sweep) {
        if (tid == 0) *sh_flag = 0;
        __syncthreads();
        bool rotated = false;
        for (int r = 0; r < pm; ++r) {
            for (int pr = grp; pr < np; pr += groups) {
                // circle method: player 0 stays, the others move on by one seat a round
                const int pb = pm - pr;
                int p = pr == 0 ? 0 : pr - 1 + r, q = pb - 1 + r;
                if (p >= pm) p -= pm;
                if (q >= pm) q -= pm;
                p += pr == 0 ? 0 : 1;
                q += 1;
                if (p >= cols || q >= cols) continue;  // paired with the dummy
                rotated |= jacobi_pair<TPP, NE>(X + (size_t)ld * min(p, q), X + (size_t)ld * max(p, q), rows, gl, tol2);
            }
            __syncthreads();
        }
        if (rotated && gl == 0) atomicOr(sh_flag, 1);
        __syncthreads();
        const int any = *sh_flag;
        __syncthreads();  // every thread has read the flag before it is reset
        if (!any) break;
    }
}

// X: rows x cols (ld >= rows) -> U diag(sig), sig: cols.  Whole workgroup; ends with a barrier.
__device__ inline void jacobi_left_vectors(double *X, int rows, int cols, int ld, double *sig, int *sh_flag) {
    // lanes per pair and elements per lane by the column length: two columns of
    // up to 16 elements a lane fit the registers
    if (rows <= 64) jacobi_sweeps<16, 4>(X, rows, cols, ld, sh_flag);
    else if (rows <= 128) jacobi_sweeps<8, 16>(X, rows, cols, ld, sh_flag);
    else jacobi_sweeps<16, 0>(X, rows, cols, ld, sh_flag);
    const int gl = threadIdx.x & 15;
    for (int j = threadIdx.x >> 4; j < cols; j += MQE_NT / 16) {
        const double *x = X + (size_t)ld * j;
        double s2 = 0.0;
        for (int i = gl; i < rows; i += 16) s2 += x[i] * x[i];
        s2 = lanes_sum<16>(s2);
        if (gl == 0) sig[j] = sqrt(s2);
    }
    __syncthreads();
}

// Upper triangle of the R factor of A (rows x cols, rows >= cols, ld) in place;
// below the diagonal the reflectors remain.  tau: cols doubles.  16 lanes per
// column, a lane owns the rows congruent to it; the group of column j + 1 forms
// its reflector as soon as it has applied reflector j, so a column step costs
// one barrier.  Whole workgroup; ends with a barrier.
__device__ inline void householder_r(double *A, int rows, int cols, int ld, double *tau) {
    const int gl = threadIdx.x & 15, grp = threadIdx.x >> 4;
    constexpr int groups = MQE_NT / 16;
    // reflector of column j: v_j = 1 implied, v_i (i > j) stored, R(j, j) on the diagonal
    auto reflect = [&](int j) {
        double *x = A + (size_t)ld * j;
        double ss = 0.0, alpha = 0.0;
        for (int i = gl + (j & ~15); i < rows; i += 16) {
            const double xi = x[i];
            if (i > j) ss += xi * xi;
            if (i == j) alpha = xi;
        }
        ss = lanes_sum<16>(ss);
        alpha = lanes_sum<16>(alpha);
        double tj = 0.0;
        if (ss != 0.0) {
            const double bt = -copysign(sqrt(alpha * alpha + ss), alpha), sc = 1.0 / (alpha - bt);
            tj = (bt - alpha) / bt;
            for (int i = gl + (j & ~15); i < rows; i += 16) {
                if (i > j) x[i] *= sc;
                if (i == j) x[i] = bt;
            }
        }
        if (gl == 0) tau[j] = tj;
    };
    if (grp == 0) reflect(0);
    __syncthreads();
    for (int j = 0; j < cols; ++j) {
        const double tj = tau[j];
        const double *v = A + (size_t)ld * j;
        // a group's first column is the one next to j, if it owns that
        for (int c = j + 1 + ((grp - (j + 1)) & (groups - 1)); c < cols; c += groups) {
            double *x = A + (size_t)ld * c;
            if (tj != 0.0) {
                double s = 0.0;
                for (int i = gl + (j & ~15); i < rows; i += 16)
                    if (i >= j) s += (i == j ? 1.0 : v[i]) * x[i];
                s = tj * lanes_sum<16>(s);
                for (int i = gl + (j & ~15); i < rows; i += 16)
                    if (i >= j) x[i] -= s * (i == j ? 1.0 : v[i]);
            }
            if (c == j + 1) reflect(c);
        }
        __syncthreads();
    }
}

// A lower bound of the smallest singular value of the upper triangular R (n x n,
// ld n): 1 / |R^-1|_F, with R^-1 formed in W (n x n).  0 if R is singular.  red:
// block_sum scratch.  Whole workgroup.
__device__ inline double least_singular_bound(const double *R, int n, double *W, double *red) {
    for (int e = threadIdx.x; e < n * n; e += MQE_NT) W[e] = e % n == e / n ? 1.0 : 0.0;
    __syncthreads();
    // back substitution for all columns at once: row k of R^-1, then its part of the rows above
    for (int k = n - 1; k >= 0; --k) {
        const double d = 1.0 / R[k + (size_t)n * k];
        for (int j = k + (int)(threadIdx.x >> 4); j < n; j += MQE_NT / 16) {
            const double x = W[k + (size_t)n * j] * d;
            for (int i = threadIdx.x & 15; i < k; i += 16) W[i + (size_t)n * j] -= R[i + (size_t)n * k] * x;
        }
        __syncthreads();
    }
    double s = 0.0;
    for (int e = threadIdx.x; e < n * n; e += MQE_NT) {
        const double x = W[e] / R[e % n + (size_t)n * (e % n)];
        s += x * x;
    }
    s = block_sum(s, red);
    return s > 0.0 && isfinite(s) ? 1.0 / sqrt(s) : 0.0;
}

// rank[j]: position of column j when the values are sorted in decreasing order
// (ties by index); ord[rank[j]] = j.  Whole workgroup.
__device__ inline void sort_descending(const double *sig, int n, int *ord) {
    for (int j = threadIdx.x; j < n; j += MQE_NT) {
        const double s = sig[j];
        int rk = 0;
        for (int i = 0; i < n; ++i) rk += (sig[i] > s || (sig[i] == s && i < j)) ? 1 : 0;
        ord[rk] = j;
    }
    __syncthreads();
}

}  // namespace mqe

#endif
