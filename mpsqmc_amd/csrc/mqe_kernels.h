// mqe_kernels.h -- what the walker kernels and the host engine share: the control
// block, the system, the population, the scratch layout, and the launch
// functions of the kernels that live in translation units of their own.
#ifndef MQE_KERNELS_H
#define MQE_KERNELS_H

#include "mqe_device.h"

#define MQE_MAXL 256
#define MQE_MAXG 4096

namespace mqe {

enum : int { F_PREP = 1, F_PROP = 2 };

// Step control block in device memory.  The launches of a step read their
// step-dependent values from here instead of taking them as arguments, so the
// same launches can be captured once in a graph and replayed (the launch-list
// kernel sets the block in an eager step and advances it in a captured one).
struct Ctl {
    int step;         // device-RNG step word of the propagation; the energy's step number
    int pstep;        // device-RNG step word of population control
    long pc;          // propagations before this one (phase of the re-orthonormalisation)
    int canon_every;  // walker slot s re-orthonormalises when (s + pc) % canon_every == canon_every - 1
    int trace_cap;    // rows of the device trace
};

// Re-orthonormalisation is staggered over the walker slots: each propagation
// re-orthonormalises the slots of one phase, so every step costs the same and a
// walker that keeps its slot does it every canon_every steps.  A walker also
// carries the number of propagations since its last re-orthonormalisation
// (`since`, copied with it), and one that reaches canon_every - 1 does it
// regardless of its slot's phase: copies moved to new slots, and copies of
// copies, never go longer without it than a walker that stays put.
__host__ __device__ inline bool canon_walker(const Ctl &c, int slot, int since) {
    return c.canon_every <= 1 || since >= c.canon_every - 1 ||
           (int)((slot + c.pc) % c.canon_every) == c.canon_every - 1;
}

// Read-only description of the system (device pointers).
struct Sys {
    int L, nC, Ng, gdim, Dt, Dw;
    const int *tvd;    // L+1 trial bond dims
    const long *toff;  // L site offsets into the trial
    const int *first, *second, *nextfirst;
    const double *Jc;                // nC
    const double *tS, *tU, *tVT;     // per coupling: 4, 16, 16
    const double *grid;              // Ng * gdim
    const int *cs_ptr, *cs_idx;      // couplings grouped by their second site (CSR, L+1)
    double SS[16];                   // S.S two-site tensor, index (s'+2t')*4 + (s+2t)
    double Sz[2];
    double h;
    double ssp[2];                   // exp(h dtau m / 2)
    int tiles[8];                    // FP32 product tile shape by walker bond bucket (max bond 1-16, 17-32, ...)
    const float *trialT;             // FP32 general path: T_k[s]^T (t_{k+1} x t_k) at toff[k] + s t_k t_{k+1}
};

// bond bucket of a walker: its largest bond in steps of 16 (0: <= 16, ..., 7: > 112)
__host__ __device__ inline int bond_bucket(int maxbond) { return min(7, max(0, (maxbond - 1) / 16)); }

// The walker population (device pointers).
struct Pool {
    void *phi, *Renv, *Lenv;
    int *wvd;
    double *w, *O, *eh, *EL;
    const int *order;
    const int *n;
    int *idx;
    const double *u;       // host-supplied uniforms (n*nC, walker-major) or nullptr
    long wflat, eflat;
    const long *woff, *eoff;
    const long *moff;      // general path: right norm environments M_k at Renv + moff[k] (w_k x w_k)
    unsigned long long seed;
    const Ctl *ctl;        // step control block
    const int *list;       // population positions in launch order (nullptr: block b = position b)
    int *since;            // per slot: propagations since the last re-orthonormalisation
    int *status;
    char *scratch;
    long scratch_bytes;
    int padded;            // 1: tile32 storage (32x32 zero-padded blocks per site and physical index)
    // learned proposal (tile path)
    double *bondE;         // per slot: nC bond energies <trial|h_c|phi> and <trial|phi> (or nullptr)
    int nbe;               // entries of bondE per slot (nC + 1)
    int qlds;              // general path: doubles of dynamic LDS for the LQ workspace (0: none)
    const float *pred;     // predicted labels, row b*nC + c, 16 each (or nullptr)
    double mix;            // weight of the uniform part of the learned proposal
    float *lab;            // label rows of the sample buffer (or nullptr)
    float *plab;           // per slot and coupling: the labels of the last recorded propagation (16 each)
    int plab_on;           // the walker kernel records them in this launch
    const long *nsamp;     // rows already in the sample buffer
    long maxsamp;          // its capacity in rows
};

// Scratch layout of one workgroup (sizes in elements).
struct ScratchLayout {
    long Y, Y4, G, GcA, GcB, W, V, TMP, LM, t_total;  // T region
    long AQ, RQ, TAU, PDF, CUM, d_total;              // double region
};

__host__ __device__ inline ScratchLayout scratch_layout(int Dt, int Dw, int Ng) {
    ScratchLayout s;
    const long Dm = Dt > Dw ? Dt : Dw;
    long o = 0;
    s.Y = o; o += Dm * 2 * Dm;
    s.Y4 = o; o += 8L * Dt * Dw;  // the four carried channels times site k
    s.G = o; o += 4L * Dt * Dw;
    s.GcA = o; o += 4L * Dt * Dw;
    s.GcB = o; o += 4L * Dt * Dw;
    s.W = o; o += 2L * Dt * Dw;
    s.V = o; o += 4L * Dt * Dw;
    s.TMP = o; o += 2L * Dw * Dw;
    s.LM = o; o += (long)Dw * Dw;
    s.t_total = o;
    o = 0;
    const long panels = Dw <= QR_PANELS_N ? panel_doubles((int)Dw) : 0;  // the LQ's reflectors
    s.AQ = o; o += 2L * Dw * Dw > panels ? 2L * Dw * Dw : panels;
    s.RQ = o; o += (long)Dw * Dw;
    s.TAU = o; o += Dw;
    s.PDF = o; o += Ng;
    s.CUM = o; o += Ng;
    s.d_total = o;
    return s;
}

template <typename T>
__host__ __device__ inline long scratch_bytes_for(int Dt, int Dw, int Ng) {
    ScratchLayout s = scratch_layout(Dt, Dw, Ng);
    long tb = s.t_total * (long)sizeof(T);
    tb = (tb + 255) & ~255L;
    return tb + s.d_total * (long)sizeof(double) + 256;
}
// Launch functions of the walker kernels (one translation unit each, compiled
// concurrently).  lds_attr: raise the kernel's dynamic LDS limit to `lds` bytes.
struct WalkerLaunch {
    int grid;
    size_t lds;
    hipStream_t stream;
};
void launch_walker_f32(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *trial, int flags);
void launch_walker_f32_chained(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *trial, int flags);
void launch_walker_f64(const WalkerLaunch &l, const Sys &S, const Pool &P, const double *trial, int flags);
void launch_walker_f64_chained(const WalkerLaunch &l, const Sys &S, const Pool &P, const double *trial, int flags);
hipError_t lds_attr_f32(size_t lds);
hipError_t lds_attr_f32_chained(size_t lds);
hipError_t lds_attr_f64(size_t lds);
hipError_t lds_attr_f64_chained(size_t lds);

namespace t32 {
constexpr int MAXG_T32 = 256;  // grid points: four per lane of one wave
// TN / TT: the trial in padded blocks, plain and transposed; learn: the learned proposal
void launch_walker32(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *TN, const float *TT, int flags,
                     bool learn);
hipError_t lds_attr32();
}  // namespace t32

namespace t16 {
// the same storage and trial blocks; bonds up to MAXD, no learned proposal
constexpr int MAXD = 16;
void launch_walker16(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *TN, const float *TT, int flags);
}  // namespace t16

}  // namespace mqe

#endif
