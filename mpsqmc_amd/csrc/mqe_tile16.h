// mqe_tile16.h -- FP32 MFMA walker kernel for nearest-neighbour chains with all
// trial and walker bond dimensions <= 16: one wave owns a walker for a whole step.
//
// Storage and algorithm are those of mqe_tile32.h (32 x 32 zero-padded blocks in
// global memory, of which only the leading 16 x 16 parts are touched here), so
// the two kernels can take turns on one population.
//
// Every matrix is a 16 x 16 tile in four registers of each lane in the
// accumulator layout of v_mfma_f32_16x16x4f32: lane (j, g), j = lane % 16,
// g = lane / 16, holds rows 4g .. 4g + 3 of column j.  With the inner index taken
// in the order k = 4g + e (MFMA e), that layout of X is the A operand of X^T and
// that of Y the B operand of Y, so X^T Y is four MFMAs without any data movement
// (mm below).  The environments and pair blocks of a coupling therefore stay in
// registers; one 16 x 16 transposition through LDS per coupling (L or R) is left.
//
// What bounds it: the serial chain of a coupling within one walker (three
// dependent matrix products, the 16 dot products' lane sums, the FP64 sampling).
// The 32 x 32 kernel with its four waves spends eight times the matrix work on
// such bonds (D <= 16 in 32 x 32 tiles) and two to four workgroup barriers per
// coupling; one step with population control of 64 walkers of 10 sites at D = 8
// takes 119 us (32 x 32: 260), of 1000 walkers of 50 sites 690 us (2003).
#ifndef MQE_TILE16_H
#define MQE_TILE16_H

#include "mqe_kernels.h"

namespace mqe {
namespace t16 {

typedef float v4 __attribute__((ext_vector_type(4)));

constexpr int GB = 1024;   // floats per global block
constexpr int GLD = 32;    // its leading dimension
constexpr int LD = 20;     // LDS leading dimension (16-byte aligned columns)
constexpr int TB = 16 * LD;

struct Lane {
    int j, g;  // column, row group
};

// the tile of X in the accumulator layout
__device__ __forceinline__ v4 ld_n(Lane l, const float *X, int ld) { return *(const v4 *)(X + ld * l.j + 4 * l.g); }
// the tile of X^T
__device__ __forceinline__ v4 ld_t(Lane l, const float *X, int ld) {
    v4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = X[l.j + ld * (4 * l.g + e)];
    return x;
}
__device__ __forceinline__ void st_n(Lane l, v4 x, float *X, int ld) { *(v4 *)(X + ld * l.j + 4 * l.g) = x; }

// acc + X^T Y
__device__ __forceinline__ v4 mm(v4 x, v4 y, v4 acc = v4{0.f, 0.f, 0.f, 0.f}) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ float dot4(v4 a, v4 b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3]; }

__device__ __forceinline__ v4 unit_tile(Lane l) { return v4{l.j == 0 && l.g == 0 ? 1.f : 0.f, 0.f, 0.f, 0.f}; }

// sixteen wave-wide sums by a reduce-scatter: lane l receives the sum of s[l / 4]
__device__ __forceinline__ double reduce16(const double (&s)[16]) {
    const int lane = threadIdx.x & 63;
    double a[8], b[4], c[2];
#pragma unroll
    for (int q = 0; q < 8; ++q) a[q] = halves_sum(s[q], s[q + 8]);
#pragma unroll
    for (int q = 0; q < 4; ++q) b[q] = rows_sum(a[q], a[q + 4]);
    const bool hi8 = lane & 8, hi4 = lane & 4;
#pragma unroll
    for (int q = 0; q < 2; ++q) c[q] = (hi8 ? b[q + 2] : b[q]) + dpp_d<0x140>(hi8 ? b[q] : b[q + 2]);  // row_mirror
    double d = (hi4 ? c[1] : c[0]) + dpp_d<0x141>(hi4 ? c[0] : c[1]);                              // row_half_mirror
    d += dpp_d<0xB1>(d);  // quad_perm [1,0,3,2]
    d += dpp_d<0x4E>(d);  // quad_perm [2,3,0,1]
    return d;
}

struct W16 {
    const Sys *S;
    const float *TN, *TT;  // trial blocks, plain and transposed
    float *phi, *Lg, *Rg;
    __device__ const float *tn(int k, int s) const { return TN + (size_t)(2 * k + s) * GB; }
    __device__ const float *tt(int k, int s) const { return TT + (size_t)(2 * k + s) * GB; }
    __device__ float *ph(int k, int s) const { return phi + (size_t)(2 * k + s) * GB; }
    __device__ float *L(int k) const { return Lg + (size_t)k * GB; }
    __device__ float *R(int k) const { return Rg + (size_t)k * GB; }
};

__global__ __launch_bounds__(64, 2) void walker16_kernel(Sys S, Pool P, const float *TN, const float *TT, int flags) {
    const int n = *P.n;
    if ((int)blockIdx.x >= n) return;
    if (*P.status & 4) return;  // the population overflowed: keep the state as it was
    const int b = P.list ? P.list[blockIdx.x] : (int)blockIdx.x;  // population position
    const int slot = P.order[b];
    const Ctl ctl = *P.ctl;
    const int Lc = S.L, lane = threadIdx.x;
    const Lane ln{lane & 15, lane >> 4};
    __shared__ __attribute__((aligned(16))) float xpose[TB], cen[2 * TB], LM[TB];
    __shared__ double QV[32 * 16], qtau[16];
    W16 C;
    C.S = &S;
    C.TN = TN;
    C.TT = TT;
    C.phi = (float *)P.phi + (size_t)slot * P.wflat;
    C.Lg = (float *)P.Lenv + (size_t)slot * P.eflat;
    C.Rg = (float *)P.Renv + (size_t)slot * P.eflat;
    double *bond = P.bondE ? P.bondE + (size_t)slot * (S.nC + 1) : nullptr;
    double wt = P.w[slot];
    const double O = P.O[slot];
    const bool prep = flags & F_PREP;
    // X -> X^T (one wave: the barriers only order the LDS accesses)
    auto transpose = [&](v4 x) {
        st_n(ln, x, xpose, LD);
        __syncthreads();
        const v4 y = ld_t(ln, xpose, LD);
        __syncthreads();
        return y;
    };
    v4 cN[2];  // the center tensor phi_k[s]

    if (prep) {
        // left environments of the loaded state
        v4 LT = unit_tile(ln);
        for (int k = 0; k < Lc - 1; ++k) {
            v4 l{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 2; ++s)
                l = mm(ld_n(ln, C.tn(k, s), GLD), mm(LT, ld_n(ln, C.ph(k, s), GLD)), l);
            st_n(ln, l, C.L(k + 1), GLD);
            LT = transpose(l);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) cN[s] = ld_n(ln, C.ph(Lc - 1, s), GLD);
    } else {
        // ---------------- propagation (MPSQMC2.cpp:532-600), h = 0 ----------------
        // normalisation as in the 32 x 32 kernel: the overlap stays O throughout
        const int Ng = S.Ng;
        double gx[4][4];  // this lane's grid points 4 lane .. 4 lane + 3
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) gx[t][q] = 4 * lane + t < Ng ? S.grid[4 * (4 * lane + t) + q] : 0.0;
        // Trotter tables by lane: combo (a, bb) of lane % 16 = a + 4 bb takes ua, vb and
        // sab; lanes 0-3 form the left operator's entries and lanes 4-7 the right one's from tab
        struct Tab {
            double ua[4], vb[4], sab, tab[4];
        };
        auto table = [&](int c, Tab &T) {
            const double *tS = S.tS + 4 * c, *tU = S.tU + 16 * c, *tVT = S.tVT + 16 * c;
            const int a = lane & 3, bb = (lane >> 2) & 3;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                T.ua[q] = tU[q + 4 * a];    // U_a(s', s), q = s' + 2s
                T.vb[q] = tVT[bb + 4 * q];  // VT_bb(t', t), q = t' + 2t
                T.tab[q] = 2.0 * sqrt(tS[q]) * ((lane & 4) ? tVT[q + 4 * a] : tU[a + 4 * q]);
            }
            T.sab = sqrt(tS[a]) * sqrt(tS[bb]);
        };
        // operands of a coupling: phi_j, phi_j^T, R_{j+1}^T and the trial's sites
        struct Ops {
            v4 n[2], t[2], RT, ti[2], tj[2];
        };
        auto fetch = [&](int c, Ops &o) {
            const int j = c + 1;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                o.n[s] = ld_n(ln, C.ph(j, s), GLD);
                o.t[s] = ld_t(ln, C.ph(j, s), GLD);
                o.ti[s] = ld_n(ln, C.tn(c, s), GLD);
                o.tj[s] = ld_n(ln, C.tt(j, s), GLD);
            }
            o.RT = j + 1 < Lc ? ld_t(ln, C.R(j + 1), GLD) : unit_tile(ln);
        };
        v4 LT = unit_tile(ln);
#pragma unroll
        for (int s = 0; s < 2; ++s) cN[s] = ld_n(ln, C.ph(0, s), GLD);
        Ops op;
        Tab tb;
        fetch(0, op);
        table(0, tb);
        double ublk = 0.0;  // uniforms of 64 couplings, one per lane
        for (int c = 0; c < S.nC; ++c) {
            if ((c & 63) == 0 && c + lane < S.nC)
                ublk = P.u ? P.u[(size_t)b * S.nC + c + lane]
                           : philox_uniform(P.seed, (uint32_t)b, (uint32_t)(c + lane), (uint32_t)ctl.step, 0u);
            Ops nx;
            Tab tn;
            const int cn = min(c + 1, S.nC - 1);
            fetch(cn, nx);
            table(cn, tn);
            // Y[s] = L_i phi_i[s], W[t] = R_{j+1} phi_j[t]^T; G(s',s) = T_i[s']^T Y[s], V(t',t) = T_j[t'] W[t]
            v4 Y[2], W[2], G[4], V[4];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                Y[s] = mm(LT, cN[s]);
                W[s] = mm(op.RT, op.t[s]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                G[q] = mm(op.ti[q >> 1], Y[q & 1]);  // q = 2s' + s
                V[q] = mm(op.tj[q >> 1], W[q & 1]);  // q = 2t' + t
            }
            // M[(s' + 2t') 4 + (s + 2t)] = <G(s',s), V(t',t)>: FP32 over a lane's four elements, FP64 across lanes
            double sm[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int sp = (q >> 2) & 1, tp = q >> 3, s = q & 1, t = (q >> 1) & 1;
                sm[q] = (double)dot4(G[2 * sp + s], V[2 * tp + t]);
            }
            const double red = reduce16(sm);
            double m[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) m[q] = readlane_d(red, 4 * q);
            // combos, PDF, CDF sample (MPSQMC2.cpp:540-588)
            double cq = 0.0;
#pragma unroll
            for (int x = 0; x < 4; ++x) {  // x = s' + 2s
                double mv = 0.0;
#pragma unroll
                for (int y = 0; y < 4; ++y)  // y = t' + 2t
                    mv += tb.vb[y] * m[((x & 1) + 2 * (y & 1)) * 4 + ((x >> 1) + 2 * (y >> 1))];
                cq += tb.ua[x] * mv;
            }
            cq *= tb.sab;
            double cb[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) cb[q] = readlane_d(cq, q);
            if (P.plab_on && lane < 16) {  // labels combos/O: the walker's record and the training rows
                const float lv = (float)(cq / O);
                P.plab[((size_t)slot * S.nC + c) * 16 + lane] = lv;
                if (P.lab) {
                    const long base = *P.nsamp, row = base + (long)b * S.nC + c;
                    if (base + (long)n * S.nC <= P.maxsamp) P.lab[row * 16 + lane] = lv;
                }
            }
            // f(x) = sum_{l,r} comb[l + 4r] x_l x_r through the symmetric part
            double hs[10];
            {
                int k = 0;
#pragma unroll
                for (int l = 0; l < 4; ++l)
#pragma unroll
                    for (int r = l; r < 4; ++r) hs[k++] = r == l ? cb[5 * l] : cb[l + 4 * r] + cb[r + 4 * l];
            }
            auto quad = [&](const double (&x)[4]) {
                double f = 0.0;
                int k = 0;
#pragma unroll
                for (int l = 0; l < 4; ++l) {
                    double t = 0.0;
#pragma unroll
                    for (int r = l; r < 4; ++r) t += hs[k++] * x[r];
                    f += x[l] * t;
                }
                return f;
            };
            const double pref = 4.0 / (O * Ng);
            double pv[4], fv[4], loc = 0.0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                fv[t] = quad(gx[t]);
                pv[t] = 4 * lane + t < Ng ? (fv[t] > 0.0 ? fv[t] : 0.0) * pref : 0.0;
                loc += pv[t];
            }
            // cum_g <= u is tested as cum_g * norm <= u * norm on one scan of the unnormalised PDF
            const double incl = wave_inclusive_scan(loc), pdfnorm = readlane_d(incl, 63);
            const double ut = readlane_d(ublk, c & 63) * pdfnorm;
            double run = dpp_d<0x138>(incl);  // exclusive prefix (wave_shr:1)
            int gs = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                run += pv[t];
                gs += __popcll(__ballot(4 * lane + t < Ng - 1 && run <= ut));
            }
            gs = __builtin_amdgcn_readfirstlane(gs);
            wt *= pdfnorm;
            if (lane == 0) {
                if (P.idx) P.idx[(size_t)b * S.nC + c] = gs;
                if (!(pdfnorm > 0.0) || !isfinite(pdfnorm)) atomicOr(P.status, 1);
            }
            // the grid point and f there from the lane that owns it
            const int gl = gs >> 2, gt = gs & 3;
            auto pick = [&](double a0, double a1, double a2, double a3) {
                const double x = gt & 1 ? a1 : a0, y = gt & 1 ? a3 : a2;
                return readlane_d(gt & 2 ? y : x, gl);
            };
            double xs[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) xs[q] = pick(gx[0][q], gx[1][q], gx[2][q], gx[3][q]);
            const double fstar = pick(fv[0], fv[1], fv[2], fv[3]);  // <trial|B(x*) phi> / 4
            // sampled operators: sqrt(4 S_k) x_k U_k, VT_k (MPSstate.cpp:591,616), the right one
            // scaled by O / <trial|B(x) phi> so that the overlap stays O
            double ov = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) ov += tb.tab[q] * xs[q];
            if (lane & 4) ov *= O / (4.0 * fstar);
            const float of = (float)ov;
            float u[4], v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                u[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(of), q));
                v[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(of), 4 + q));
            }
            // L_{i+1} = sum_{s',s} Ux(s',s) G(s',s), phi'_i = Ux phi_i, phi'_j = Vx phi_j (the next left site)
            v4 l, p0, p1, q0, q1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                l[e] = u[0] * G[0][e] + u[2] * G[1][e] + u[1] * G[2][e] + u[3] * G[3][e];
                p0[e] = u[0] * cN[0][e] + u[2] * cN[1][e];
                p1[e] = u[1] * cN[0][e] + u[3] * cN[1][e];
                q0[e] = v[0] * op.n[0][e] + v[2] * op.n[1][e];
                q1[e] = v[1] * op.n[0][e] + v[3] * op.n[1][e];
            }
            st_n(ln, l, C.L(c + 1), GLD);
            st_n(ln, p0, C.ph(c, 0), GLD);
            st_n(ln, p1, C.ph(c, 1), GLD);
            cN[0] = q0;
            cN[1] = q1;
            LT = transpose(l);
            op = nx;
            tb = tn;
        }
    }
    __syncthreads();  // the environments and tensors stored above are read by other lanes below

    // ---------------- local energy (Walker.cpp:72-77), right to left ----------------
    // canonical: FP64 LQ of every site; else R_k and the right norm environment M_k
    // only (as in the 32 x 32 kernel)
    const bool canon = prep || canon_walker(ctl, slot, P.since[slot]);
    double etot = 0.0;
    v4 RT = unit_tile(ln), Rn = RT, Mk = RT, cT[2];
    const v4 zero{0.f, 0.f, 0.f, 0.f};
    if (!canon) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            st_n(ln, cN[s], C.ph(Lc - 1, s), GLD);
            cT[s] = transpose(cN[s]);
        }
    }
    struct Ops {
        v4 n[2], t[2], LT, ti[2], tk[2];
    };
    auto fetch = [&](int k, Ops &o) {  // site k - 1, its left environment, the trial's sites k - 1 and k
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            o.n[s] = ld_n(ln, C.ph(k - 1, s), GLD);
            o.t[s] = ld_t(ln, C.ph(k - 1, s), GLD);
            o.ti[s] = ld_n(ln, C.tn(k - 1, s), GLD);
            o.tk[s] = ld_n(ln, C.tt(k, s), GLD);
        }
        o.LT = k > 1 ? ld_t(ln, C.L(k - 1), GLD) : unit_tile(ln);
    };
    const int *wvd = P.wvd + (size_t)slot * (Lc + 1);
    Ops op;
    fetch(Lc - 1, op);
    for (int k = Lc - 1; k >= 1; --k) {
        Ops nx;
        fetch(max(k - 1, 1), nx);
        if (canon) {
            const int wk = wvd[k], wn = wvd[k + 1];
#pragma unroll
            for (int s = 0; s < 2; ++s) st_n(ln, cN[s], cen + s * TB, LD);
            st_n(ln, zero, LM, LD);
            __syncthreads();
            // A = phi^T, row r = column + w_{k+1} s: four lanes a column, eight rows a lane
            auto el = [&](int r, int c) -> float & {
                const int s = r >= wn ? 1 : 0;
                return cen[s * TB + c + LD * (r - s * wn)];
            };
            qr_regs<4, 8>(
                2 * wn, wk, QV, qtau, true, [&](int r, int c) { return (double)el(r, c); },
                [&](int r, int c, double x) { LM[c + LD * r] = (float)x; },
                [&](int r, int c, double x) { el(r, c) = (float)x; });
            __syncthreads();
            const v4 lm = ld_n(ln, LM, LD);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                cN[s] = ld_n(ln, cen + s * TB, LD);
                cT[s] = ld_t(ln, cen + s * TB, LD);
                st_n(ln, cN[s], C.ph(k, s), GLD);
                op.n[s] = mm(op.t[s], lm);  // phi_{k-1} Lmat
            }
            __syncthreads();
        }
        v4 W[2], Y[2], G[4], V[4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            W[s] = mm(RT, cT[s]);
            Y[s] = mm(op.LT, op.n[s]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            V[q] = mm(op.tk[q >> 1], W[q & 1]);
            G[q] = mm(op.ti[q >> 1], Y[q & 1]);
        }
        if (!canon) {
            v4 Z[2], mn = zero;  // M_k = sum_t phi_k[t] (M_{k+1} phi_k[t]^T), M symmetric
#pragma unroll
            for (int s = 0; s < 2; ++s) Z[s] = mm(Mk, cT[s]);
#pragma unroll
            for (int s = 0; s < 2; ++s) mn = mm(cT[s], Z[s], mn);
            Mk = mn;
        }
        Rn = V[0] + V[3];
        st_n(ln, Rn, C.R(k), GLD);
        RT = transpose(Rn);
        double e = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int sp = (q >> 2) & 1, tp = q >> 3, s = q & 1, t = (q >> 1) & 1;
            e += S.SS[q] * (double)dot4(G[2 * sp + s], V[2 * tp + t]);
        }
        e = S.Jc[k - 1] * wave_sum(e);
        etot += e;
        if (bond && lane == 0) bond[k - 1] = e;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            cN[s] = op.n[s];
            cT[s] = op.t[s];
        }
        op = nx;
    }
    // <trial|phi> and the squared norm at site 0 (row 0 of phi_0 and T_0; rows al of R_1, M_1)
    double a = 0.0, n2 = 0.0;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double p = (double)__shfl(cN[s][0], ln.j);
        const float t0 = C.tn(0, s)[GLD * ln.j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int al = 4 * ln.g + e;
            a += (double)__shfl(t0, al) * p * (double)Rn[e];
            if (!canon) n2 += (double)__shfl(cN[s][0], al) * (double)Mk[e] * p;
            else if (al == 0) n2 += p * p;
        }
    }
    const double ovl = wave_sum(a), nrm = sqrt(wave_sum(n2));
    double On = ovl / nrm, f = 1.0 / nrm;
    if (On < 0.0) { On = -On; f = -f; }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        v4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (float)((double)cN[s][e] * f);
        st_n(ln, x, C.ph(0, s), GLD);
    }
    if (lane == 0) {
        if (bond) bond[S.nC] = ovl;
        P.since[slot] = canon ? 0 : P.since[slot] + 1;
        P.O[slot] = On;
        if (prep) {
            P.EL[slot] = etot / O;
        } else {
            P.w[slot] = wt;
            P.EL[slot] = etot / ovl;
            if (!isfinite(wt)) atomicOr(P.status, 2);
        }
    }
}

}  // namespace t16
}  // namespace mqe

#endif
