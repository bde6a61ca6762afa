// mqe_device.h -- workgroup-cooperative device primitives of the walker engine.
//
// One 256-thread workgroup (four wave64s) owns one walker.  All matrices are
// column-major with explicit leading dimensions and are addressed through
// generic pointers, so the same routines run on global (L2-resident) scratch
// and on LDS.
#ifndef MQE_DEVICE_H
#define MQE_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define MQE_NT 256
#define MQE_WAVES (MQE_NT / 64)

namespace mqe {

// Wave-uniform values.  Bond dimensions, site numbers and the tensors' addresses
// are the same in every lane of a workgroup, but the compiler cannot know it of
// values that come from LDS or memory: held in vector registers they made every
// loop bound a lane mask, every address 64-bit vector arithmetic and every buffer
// resource a loop over the lanes' values.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long uni(long x) {
    const unsigned lo = (unsigned)uni((int)(unsigned)x), hi = (unsigned)uni((int)(unsigned)((unsigned long)x >> 32));
    return (long)(((unsigned long)hi << 32) | lo);
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
// Data-parallel-primitive (DPP) lane exchange of a double within rows of 16
// lanes; CTRL is the DPP control word (quad_perm 0x00-0xFF, row_mirror 0x140,
// row_half_mirror 0x141).  All lanes of the row must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const int lo2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xF, 0xF, true);
    const int hi2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi2, lo2);
}

__device__ __forceinline__ double readlane_d_(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// sum over aligned groups of G = 4, 8 or 16 lanes; every lane receives it
template <int G>
__device__ __forceinline__ double lanes_sum(double v) {
    v += dpp_d<0xB1>(v);                            // quad_perm [1,0,3,2]
    v += dpp_d<0x4E>(v);                            // quad_perm [2,3,0,1]
    if constexpr (G >= 8) v += dpp_d<0x141>(v);   // row_half_mirror
    if constexpr (G >= 16) v += dpp_d<0x140>(v);  // row_mirror
    return v;
}

// (x, y) -> x + y of the partner half: for lanes 0-31 x(l) + x(l + 32), for
// lanes 32-63 y(l - 32) + y(l), with one v_permlane32_swap per dword
__device__ __forceinline__ double halves_sum(double x, double y) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(x), (unsigned)__double2loint(y),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y),
                                                     false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// (x, y) -> for 16-lane rows 0 and 2 x(l) + x(l + 16), for rows 1 and 3
// y(l - 16) + y(l), with one v_permlane16_swap per dword (it returns rows
// (x0, y0, x2, y2) and (x1, y1, x3, y3); checked on gfx950)
__device__ __forceinline__ double rows_sum(double x, double y) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(x), (unsigned)__double2loint(y),
                                                     false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y),
                                                     false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// DPP move of a double with a row mask; lanes of disabled rows receive 0
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_dm(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    const int lo2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xF, false);
    const int hi2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xF, false);
    return __hiloint2double(hi2, lo2);
}

// inclusive prefix sum over the 64 lanes with DPP only: row_shr 1, 2, 4, 8
// inside each 16-lane row, then row_bcast:15 (rows 1, 3) and row_bcast:31
// (rows 2, 3) carry the row totals (lane semantics checked on gfx950)
__device__ __forceinline__ double wave_inclusive_scan(double v) {
    v += dpp_d<0x111>(v);
    v += dpp_d<0x112>(v);
    v += dpp_d<0x114>(v);
    v += dpp_d<0x118>(v);
    v += dpp_dm<0x142, 0xA>(v);
    v += dpp_dm<0x143, 0xC>(v);
    return v;
}

// sum over the wave64; every lane receives the total (lane 63 of the scan)
__device__ __forceinline__ double wave_sum(double v) {
    return readlane_d_(wave_inclusive_scan(v), 63);
}

// value of v in lane l (l wave-uniform)
__device__ __forceinline__ double readlane_d(double v, int l) { return readlane_d_(v, l); }

// exclusive prefix sum over the lanes of the wave64 (lane 0 receives 0):
// the inclusive scan shifted by one lane (DPP wave_shr:1)
__device__ __forceinline__ double wave_exclusive_scan(double v) {
    return dpp_d<0x138>(wave_inclusive_scan(v));
}

// Sum over the workgroup; every thread receives the total.  sh: >= MQE_WAVES doubles.
__device__ __forceinline__ double block_sum(double v, double *sh) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < MQE_WAVES; ++w) t += sh[w];
    return t;
}

// K simultaneous sums; sh: >= K*MQE_WAVES doubles.
template <int K>
__device__ __forceinline__ void block_sum_n(double (&v)[K], double *sh) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) sh[wid * K + k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < MQE_WAVES; ++w) t += sh[w * K + k];
        v[k] = t;
    }
}

// Inclusive prefix sum of x[0..n) into y[0..n) (double), whole workgroup.
// sh: >= MQE_NT + MQE_WAVES doubles.
__device__ __forceinline__ void block_inclusive_scan(int n, const double *x, double *y, double *sh) {
    const int tid = threadIdx.x;
    const int per = (n + MQE_NT - 1) / MQE_NT;
    const int b0 = tid * per, b1 = min(n, b0 + per);
    double loc = 0.0;
    for (int i = b0; i < b1; ++i) loc += x[i];
    // wave inclusive scan of the per-thread totals
    const int lane = tid & 63, wid = tid >> 6;
    double s = loc;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        double o = __shfl_up(s, off, 64);
        if (lane >= off) s += o;
    }
    __syncthreads();
    if (lane == 63) sh[MQE_NT + wid] = s;
    __syncthreads();
    double base = 0.0;
    for (int w = 0; w < wid; ++w) base += sh[MQE_NT + w];
    double run = base + s - loc;  // exclusive prefix of this thread's chunk
    for (int i = b0; i < b1; ++i) { run += x[i]; y[i] = run; }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// FP32 GEMM on the matrix cores, whole workgroup.  The output is cut into
// tiles, one wave per tile at a time, each a chain of MFMAs over the k slices.
// A lane's operand values of a slice are one run along k, loaded straight into
// the MFMA operand registers without predication: rows and columns beyond the
// matrix are clamped to its last row / column (they only feed output elements
// that are not stored), and the loads run two slices (of this tile or the first of
// the wave's next tile) ahead of the MFMAs.  Two forms: gemm_mfma below for single
// products in LDS or memory, gemm_tiles_buf for the walkers' products.
// ---------------------------------------------------------------------------

// 16-byte loads along k need 16-byte aligned bases, leading dimension and batch stride
__device__ __forceinline__ bool aligned16(const float *X0, const float *X1, int ld, long s) {
    return ((((uintptr_t)X0) | ((uintptr_t)X1) | ((uintptr_t)ld * 4u) | ((uintptr_t)s * 4u)) & 15u) == 0;
}

// TS x TS output tiles (TS = 32: v_mfma_f32_32x32x2f32, TS = 16:
// v_mfma_f32_16x16x4f32), NW adjacent tiles along n per wave sharing the A
// run (NW = 2 only with TS = 32).  16-deep slices; within the slice at k0,
// MFMA u takes kk = k0 + KL (l / TS) + u in lane l (KL = 8 for TS = 32, 4 for
// TS = 16), which holds A(l % TS, kk) and B(kk, l % TS).  Accumulator slot q
// of lane l is element (8(q/4) + 4(l/32) + q%4, l % 32) of a 32 x 32 tile,
// (4(l/16) + q, l % 16) of a 16 x 16 tile.
template <int TS>
struct TileGeom {
    static constexpr int KL = TS == 32 ? 8 : 4;  // k values per lane and slice
    static constexpr int NACC = TS == 32 ? 16 : 4;
};

template <int TS, int NW>
__device__ __forceinline__ void tile_store(float *C0, int ldc, long sC, int tb, int m, int n, int tm, int tn, int r,
                                           int h, bool acc,
                                           const float (&c)[NW][TileGeom<TS>::NACC]) {
    constexpr int NACC = TileGeom<TS>::NACC;
    const int bt = tb / (tm * tn), t = tb - bt * (tm * tn);
    const int r0 = (t % tm) * TS;
    float *C = C0 + (size_t)bt * sC;
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        const int bc = (t / tm) * TS * NW + TS * q + r;
        if (bc < n) {
#pragma unroll
            for (int e = 0; e < NACC; ++e) {
                const int rr = TS == 32 ? r0 + 8 * (e >> 2) + 4 * h + (e & 3) : r0 + 4 * h + e;
                if (rr < m) {
                    float v = c[q][e];
                    if (acc) v += C[rr + (size_t)ldc * bc];
                    C[rr + (size_t)ldc * bc] = v;
                }
            }
        }
    }
}

template <int TS>
__device__ __forceinline__ void mfma_step(float a, float b, float (&c)[TileGeom<TS>::NACC]) {
    typedef float vacc __attribute__((ext_vector_type(TileGeom<TS>::NACC)));
    vacc x;
#pragma unroll
    for (int e = 0; e < TileGeom<TS>::NACC; ++e) x[e] = c[e];
    if constexpr (TS == 32)
        x = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, x, 0, 0, 0);
    else
        x = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, x, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < TileGeom<TS>::NACC; ++e) c[e] = x[e];
}

// Buffer resources over one walker's or the trial's arrays: the 64-bit base in
// scalar registers and 32-bit byte offsets per lane.  An offset at or beyond
// BUF_RANGE reads 0 and drops a store (the hardware range check).
constexpr int BUF_RANGE = 0x7ffffff0;
constexpr int BUF_OOB = 0x7ffffff8;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, BUF_RANGE, 0x00020000);
}
// (the b32 / b128 builtins move raw 32-bit words: bit casts, not conversions)
template <typename T = float>
__device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t r, int voff) {
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, voff, 0, 0));
}
__device__ __forceinline__ void buf_st(float v, __amdgpu_buffer_rsrc_t r, int voff, int imm) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, voff, imm, 0);
}
__device__ __forceinline__ void buf_st(double v, __amdgpu_buffer_rsrc_t r, int voff, int imm) {
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, voff, imm, 0);
}
__device__ __forceinline__ void buf_ld4(__amdgpu_buffer_rsrc_t r, int voff, float *v) {
    const float4 x = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
    v[0] = x.x;
    v[1] = x.y;
    v[2] = x.z;
    v[3] = x.w;
}

// Run of NV operand values of a slice through a buffer resource: voff the lane's
// byte offset, soff the slice's, step the bytes per k (stored across k), left the
// values of the lane's run inside the matrix (TAIL: the others read 0).
template <bool KC, bool VEC, bool TAIL, int NV>
__device__ __forceinline__ void load_run_buf(__amdgpu_buffer_rsrc_t r, int voff, int soff, int step, int left,
                                             float (&v)[NV]) {
    if constexpr (KC && VEC) {
#pragma unroll
        for (int j = 0; j < NV / 4; ++j) {
            const float4 x = __builtin_bit_cast(
                float4, __builtin_amdgcn_raw_buffer_load_b128(r, !TAIL || 4 * j < left ? voff + 16 * j : BUF_OOB, soff, 0));
            v[4 * j] = x.x;
            v[4 * j + 1] = x.y;
            v[4 * j + 2] = x.z;
            v[4 * j + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int o = KC ? voff + 4 * u : voff;
            v[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, !TAIL || u < left ? o : BUF_OOB,
                                                                                 KC ? soff : soff + step * u, 0));
        }
    }
}

// C(m x n) = sum_{s < nseg} op(A_s) op(B_s) (nseg = 1 or 2 terms of one shape and
// leading dimensions), for nb products at once (A_s + b sA and so on; their tiles are
// shared among the four waves), operands in global memory, uniform shapes (bonds above
// 64).  acc: C += instead of C =.  A cursor in scalar registers steps through the
// (tile, term, slice) items, each load is one instruction (scalar slice offset, the
// lane's offset of the tile) issued two items ahead of its MFMAs, and a last partial
// slice reads zeros past k.  One wave per SIMD has to
// issue everything between its MFMAs itself: with the operand addresses formed
// from the item's number per load (divisions, 64-bit vector arithmetic) a step of
// 256 walkers of the 6x6 snake at D = 128 took 151 ms, with the cursor 141 ms in
// 32 x 32 and 130 ms in 32 x 64 tiles (with the energies' carries as they are now 135
// and 120 ms).
// VEC: operands stored along k are 16-byte aligned and k is a multiple of 4.
template <bool TA, bool TB, int TS, int NW, bool VEC>
__device__ __forceinline__ void gemm_tiles_buf(int m, int n, int k, const float *A0, const float *A1, int lda,
                                             const float *B0, const float *B1, int ldb, float *C0, int ldc, bool acc,
                                             int nseg, int nb, long sA, long sB, long sC) {
    constexpr int KL = TileGeom<TS>::KL, NACC = TileGeom<TS>::NACC;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane % TS, h = lane / TS;
    const int tm = (m + TS - 1) / TS, tn = (n + TS * NW - 1) / (TS * NW), ntile = nb * tm * tn;
    if (w >= ntile) return;
    const int ntw = (ntile - w + MQE_WAVES - 1) / MQE_WAVES;  // tiles of this wave
    const int nsk = (k + 15) >> 4, nsl = nseg * nsk, nit = ntw * nsl;
    const int stA = TA ? 4 : 4 * lda, stB = TB ? 4 * ldb : 4;  // bytes per k
    // cursor: tile j, term seg, slice sl
    int j = 0, seg = 0, sl = 0, va = 0, vb[NW], bt = 0;
    __amdgpu_buffer_rsrc_t ra, rb;
    auto base = [&]() {
        ra = buf_rsrc((seg ? A1 : A0) + (size_t)bt * sA);
        rb = buf_rsrc((seg ? B1 : B0) + (size_t)bt * sB);
    };
    auto tile = [&]() {
        const int tb = w + MQE_WAVES * j;
        bt = tb / (tm * tn);
        const int t = tb - bt * (tm * tn), tq = t / tm;
        const int ar = min((t - tq * tm) * TS + r, m - 1);
        va = TA ? 4 * (lda * ar + KL * h) : 4 * (ar + lda * KL * h);
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            const int bc = min(tq * TS * NW + TS * q + r, n - 1);
            vb[q] = TB ? 4 * (bc + ldb * KL * h) : 4 * (ldb * bc + KL * h);
        }
        base();
    };
    tile();
    auto load = [&](float (&a)[KL], float (&b)[NW][KL]) {
        const int oa = stA * 16 * sl, ob = stB * 16 * sl;
        if (16 * sl + 16 <= k) {
            load_run_buf<TA, VEC, false, KL>(ra, va, oa, stA, 0, a);
#pragma unroll
            for (int q = 0; q < NW; ++q) load_run_buf<!TB, VEC, false, KL>(rb, vb[q], ob, stB, 0, b[q]);
        } else {
            const int left = k - 16 * sl - KL * h;
            load_run_buf<TA, VEC, true, KL>(ra, va, oa, stA, left, a);
#pragma unroll
            for (int q = 0; q < NW; ++q) load_run_buf<!TB, VEC, true, KL>(rb, vb[q], ob, stB, left, b[q]);
        }
        // next item (the last one repeats: its loads are not used)
        if (++sl == nsk) {
            if (seg + 1 < nseg) {
                ++seg;
                sl = 0;
                base();
            } else if (j + 1 < ntw) {
                ++j;
                seg = sl = 0;
                tile();
            } else {
                sl = nsk - 1;
            }
        }
    };
    float a0[KL], b0[NW][KL], a1[KL], b1[NW][KL], a2[KL], b2[NW][KL], c[NW][NACC];
#pragma unroll
    for (int q = 0; q < NW; ++q)
#pragma unroll
        for (int e = 0; e < NACC; ++e) c[q][e] = 0.f;
    int done = 0, tdone = w;  // slices of the tile being summed, its number
    auto step = [&](const float (&a)[KL], const float (&b)[NW][KL]) {
#pragma unroll
        for (int u = 0; u < KL; ++u)
#pragma unroll
            for (int q = 0; q < NW; ++q) mfma_step<TS>(a[u], b[q][u], c[q]);
        if (++done == nsl) {  // the tile is complete
            tile_store<TS, NW>(C0, ldc, sC, tdone, m, n, tm, tn, r, h, acc, c);
            done = 0;
            tdone += MQE_WAVES;
#pragma unroll
            for (int q = 0; q < NW; ++q)
#pragma unroll
                for (int e = 0; e < NACC; ++e) c[q][e] = 0.f;
        }
    };
    load(a0, b0);
    load(a1, b1);
#pragma nounroll
    for (int i = 0; i < nit; i += 3) {
        load(a2, b2);
        __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the MFMAs
        step(a0, b0);
        if (i + 1 >= nit) break;
        load(a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        step(a1, b1);
        if (i + 2 >= nit) break;
        load(a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        step(a2, b2);
    }
}

// C = op(A) op(B), operands in LDS or memory (the proposal network's layers), in
// 32 x 32 tiles.  k a multiple of 16 and 16-byte aligned operands along k: one
// pipelined chain over the (tile, slice) items of a wave, the operands of the item two
// ahead loaded unconditionally (past the end the last item reloads itself) with a fixed
// instruction sequence, so the wait for an item's operands covers only its own loads.
// Else: per tile and slice, zeros at k and beyond, no pipelining.
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_mfma(int m, int n, int k, const float *A, int lda, const float *B, int ldb,
                                          float *C, int ldc) {
    constexpr int TS = 32, KL = TileGeom<TS>::KL, NACC = TileGeom<TS>::NACC;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane % TS, h = lane / TS;
    const int tm = (m + TS - 1) / TS, tn = (n + TS - 1) / TS, ntile = tm * tn;
    if (w >= ntile) return;
    // a lane's row of op(A) and column of op(B) in tile t, clamped into the matrices
    auto row = [&](int t) {
        const int ar = min((t % tm) * TS + r, m - 1);
        return TA ? A + (size_t)lda * ar : A + ar;
    };
    auto col = [&](int t) {
        const int bc = min((t / tm) * TS + r, n - 1);
        return TB ? B + bc : B + (size_t)ldb * bc;
    };
    float c[1][NACC];
#pragma unroll
    for (int e = 0; e < NACC; ++e) c[0][e] = 0.f;
    if (k >= 16 && (k & 15) == 0 && (!TA || aligned16(A, A, lda, 0)) && (TB || aligned16(B, B, ldb, 0))) {
        // KC: stored along k
        auto run = [&](auto KC, const float *p, int ld, int kb, float (&v)[KL]) {
            if constexpr (decltype(KC)::value) {
                const float4 *q = (const float4 *)(p + kb);
#pragma unroll
                for (int j = 0; j < KL / 4; ++j) {
                    const float4 x = q[j];
                    v[4 * j] = x.x;
                    v[4 * j + 1] = x.y;
                    v[4 * j + 2] = x.z;
                    v[4 * j + 3] = x.w;
                }
            } else {
#pragma unroll
                for (int u = 0; u < KL; ++u) v[u] = p[(size_t)ld * (kb + u)];
            }
        };
        const int ntw = (ntile - w + MQE_WAVES - 1) / MQE_WAVES;  // tiles of this wave
        const int nsl = k >> 4, nit = ntw * nsl;
        auto load = [&](int i, float (&a)[KL], float (&b)[KL]) {
            const int j = i / nsl, kb = 16 * (i - j * nsl) + KL * h, t = w + MQE_WAVES * j;
            run(std::integral_constant<bool, TA>(), row(t), lda, kb, a);
            run(std::integral_constant<bool, !TB>(), col(t), ldb, kb, b);
        };
        // three operand sets in rotation (the loop is unrolled by three, so no
        // register copies wait on loads in flight)
        float a0[KL], b0[KL], a1[KL], b1[KL], a2[KL], b2[KL];
        auto step = [&](int i, const float (&a)[KL], const float (&b)[KL]) {
#pragma unroll
            for (int u = 0; u < KL; ++u) mfma_step<TS>(a[u], b[u], c[0]);
            if ((i + 1) % nsl == 0) {  // the tile is complete
                tile_store<TS, 1>(C, ldc, 0, w + MQE_WAVES * (i / nsl), m, n, tm, tn, r, h, false, c);
#pragma unroll
                for (int e = 0; e < NACC; ++e) c[0][e] = 0.f;
            }
        };
        load(0, a0, b0);
        load(min(1, nit - 1), a1, b1);
        for (int i = 0; i < nit; i += 3) {
            load(min(i + 2, nit - 1), a2, b2);
            __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the MFMAs
            step(i, a0, b0);
            if (i + 1 >= nit) break;
            load(min(i + 3, nit - 1), a0, b0);
            __builtin_amdgcn_sched_barrier(0);
            step(i + 1, a1, b1);
            if (i + 2 >= nit) break;
            load(min(i + 4, nit - 1), a1, b1);
            __builtin_amdgcn_sched_barrier(0);
            step(i + 2, a2, b2);
        }
        return;
    }
    for (int t = w; t < ntile; t += MQE_WAVES) {
        const float *pa = row(t), *pb = col(t);
#pragma unroll
        for (int e = 0; e < NACC; ++e) c[0][e] = 0.f;
        for (int k0 = 0; k0 < k; k0 += 16) {
            float a[KL], b[KL];
#pragma unroll
            for (int u = 0; u < KL; ++u) {
                const int kk = k0 + KL * h + u;
                a[u] = kk < k ? (TA ? pa[kk] : pa[(size_t)lda * kk]) : 0.f;
                b[u] = kk < k ? (TB ? pb[(size_t)ldb * kk] : pb[kk]) : 0.f;
            }
#pragma unroll
            for (int u = 0; u < KL; ++u) mfma_step<TS>(a[u], b[u], c[0]);
        }
        tile_store<TS, 1>(C, ldc, 0, t, m, n, tm, tn, r, h, false, c);
    }
}

// Output tile shapes of the FP32 matrix-core products (chosen per walker bond
// bucket by the engine's tile table).
enum : int { TILE_16 = 16, TILE_32 = 32, TILE_WIDE = 64 };

// The matrix-core product with the output tile shape `tile` (uniform shapes and
// addresses, operands in global memory).
template <bool TA, bool TB, int TS, int NW>
__device__ __forceinline__ void gemm_shape(int m, int n, int k, const float *A0, const float *A1, int lda,
                                           const float *B0, const float *B1, int ldb, float *C, int ldc, bool acc,
                                           int nseg, int nb, long sA, long sB, long sC) {
    const bool vec = (k & 3) == 0 && (!TA || aligned16(A0, nseg > 1 ? A1 : A0, lda, sA)) &&
                     (TB || aligned16(B0, nseg > 1 ? B1 : B0, ldb, sB));
    if (vec)
        gemm_tiles_buf<TA, TB, TS, NW, true>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, acc, nseg, nb, sA, sB, sC);
    else
        gemm_tiles_buf<TA, TB, TS, NW, false>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, acc, nseg, nb, sA, sB, sC);
}
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_f32(int m, int n, int k, const float *A0, const float *A1, int lda,
                                         const float *B0, const float *B1, int ldb, float *C, int ldc, bool acc,
                                         int nseg, int nb, long sA, long sB, long sC, int tile) {
    if (tile == TILE_16)
        gemm_shape<TA, TB, 16, 1>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, acc, nseg, nb, sA, sB, sC);
    else if (tile == TILE_WIDE && n > 32)
        gemm_shape<TA, TB, 32, 2>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, acc, nseg, nb, sA, sB, sC);
    else
        gemm_shape<TA, TB, 32, 1>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, acc, nseg, nb, sA, sB, sC);
}

// Vector-unit product (FP64, and FP32 products too small for the matrix cores).
template <bool TA, bool TB, typename T>
__device__ __forceinline__ void gemm_valu(int m, int n, int k, const T *A0, const T *A1, int lda, const T *B0,
                                          const T *B1, int ldb, T *C, int ldc, bool acc, int nseg, int nb, long sA,
                                          long sB, long sC) {
    const int mn = m * n;
    for (int e = threadIdx.x; e < nb * mn; e += MQE_NT) {
        const int bt = e / mn, x = e - bt * mn;
        const int r = x % m, c = x / m;
        T *Cb = C + (size_t)bt * sC;
        T s = acc ? Cb[r + (size_t)ldc * c] : T(0);
        for (int sg = 0; sg < nseg; ++sg) {
            const T *Ab = (sg ? A1 : A0) + (size_t)bt * sA, *Bb = (sg ? B1 : B0) + (size_t)bt * sB;
            const T *ap = TA ? (Ab + (size_t)lda * r) : (Ab + r);
            const T *bp = TB ? (Bb + c) : (Bb + (size_t)ldb * c);
            for (int q = 0; q < k; ++q) {
                const T av = TA ? ap[q] : ap[(size_t)lda * q];
                const T bv = TB ? bp[(size_t)ldb * q] : bp[q];
                s += av * bv;
            }
        }
        Cb[r + (size_t)ldc * c] = s;
    }
}

// ---------------------------------------------------------------------------
// nb products of one shape, C_b (+)= op(A_b) op(B_b) with A_b = A + b sA (and so
// on), as one workgroup call: the output tiles of all of them are shared among
// the four waves (small products keep every wave busy) and one barrier after
// the call covers the batch.
// ---------------------------------------------------------------------------
template <bool TA, bool TB, typename T>
__device__ __forceinline__ void gemm_batch(int nb, int m, int n, int k, const T *A, int lda, long sA, const T *B,
                                           int ldb, long sB, T *C, int ldc, long sC, bool acc, int tile = TILE_32) {
    if constexpr (sizeof(T) == sizeof(float)) {
        if (m >= 8 && n >= 8 && k >= 4) {
            gemm_f32<TA, TB>(m, n, k, (const float *)A, (const float *)A, lda, (const float *)B, (const float *)B, ldb,
                             (float *)C, ldc, acc, 1, nb, sA, sB, sC, tile);
            return;
        }
    }
    gemm_valu<TA, TB, T>(m, n, k, A, A, lda, B, B, ldb, C, ldc, acc, 1, nb, sA, sB, sC);
}

// Two-term product C = op(A0) op(B0) + op(A1) op(B1) (the sums over a physical
// index): one accumulation chain per output tile.
template <bool TA, bool TB, typename T>
__device__ __forceinline__ void gemm2(int m, int n, int k, const T *A0, const T *A1, int lda, const T *B0,
                                      const T *B1, int ldb, T *C, int ldc, int tile = TILE_32, int nb = 1, long sA = 0,
                                      long sB = 0, long sC = 0) {
    if constexpr (sizeof(T) == sizeof(float)) {
        if (m >= 8 && n >= 8 && k >= 4) {
            gemm_f32<TA, TB>(m, n, k, (const float *)A0, (const float *)A1, lda, (const float *)B0, (const float *)B1,
                             ldb, (float *)C, ldc, false, 2, nb, sA, sB, sC, tile);
            return;
        }
    }
    gemm_valu<TA, TB, T>(m, n, k, A0, A1, lda, B0, B1, ldb, C, ldc, false, 2, nb, sA, sB, sC);
}

template <typename T>
__device__ __forceinline__ void set_one(T *p) {
    if (threadIdx.x == 0) p[0] = (T)1;
    __syncthreads();
}

// ---------------------------------------------------------------------------
// GEMM: C(m x n) (+)= op(A) op(B).  op(A) is m x k: A(r,q) = TA ? A[q + lda*r] : A[r + lda*q].
// FP32 products of useful size run on the matrix cores with the output tile
// shape `tile`, the rest (and all of FP64) on the vector units.
// ---------------------------------------------------------------------------
template <bool TA, bool TB, typename T>
__device__ __forceinline__ void gemm(int m, int n, int k, const T *A, int lda, const T *B, int ldb, T *C, int ldc,
                                     bool acc, int tile = TILE_32) {
    gemm_batch<TA, TB, T>(1, m, n, k, A, lda, 0, B, ldb, 0, C, ldc, 0, acc, tile);
}

// ---------------------------------------------------------------------------
// Two chained FP32 matrix-core products with the intermediate in registers:
//   F_f = A op(B_f)                      (m1 x n1, inner dimension k1)
//   ND = 1:  D_0 = sum_f op(C_f) F_f     (f < NF, NF = 1, 2)
//   ND = 2:  D_d = op(C_d) F_0           (d < 2, NF = 1: two outputs of one F)
// (D_d: mD x n1; inner dimension m1 <= 64, mD <= 64) for nu independent units
// (operands of unit u from get(u)), whole workgroup, no barrier inside.  A
// wave takes (unit, 32-column strip) items: for each f it forms the strip of
// F_f in two 32 x 32 accumulator tiles (rows >= m1 zeroed) and feeds the
// accumulator slots straight into the second chain as its B operand,
// accumulating the (at most two) row tiles of each D strip in registers.  The
// second chain takes its inner index in the order the accumulators hold it:
// MFMA q of F row tile t uses rows 32t + 8(q/4) + 4h + q%4 (h = lane half),
// exactly accumulator slot q of lane (column, h), so no lane exchange is
// needed; op(C) is loaded in the same order.
// Items go to waves round-robin starting at wave0; the return value is the
// wave that takes the next item, so independent calls share the waves
// between two barriers.
// TB: B_f stored n1 x k1 (op(B) = B^T).  TC: C stored m1 x mD (op(C) = C^T,
// contiguous along the inner index), else mD x m1.  All matrices column-major.
// ---------------------------------------------------------------------------
template <typename T>
struct ChainOps {
    const T *A;      // m1 x k1, leading dimension lda
    const T *B[2];   // B_f
    const T *C[2];   // C_f (ND = 1) or C_d (ND = 2)
    T *D[2];         // D_d, mD x n1, leading dimension ldd
};

typedef float v16f_c __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16f_c mfma32(float a, float b, v16f_c c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// qsplit: the two row tiles of D are separate items (the F strips formed for
// each), for calls with too few items to keep the four waves busy.
template <bool TB, bool TC, int NF, int ND, class Get>
__device__ __forceinline__ int chain2(int wave0, int nu, int m1, int n1, int k1, int mD, int lda, int ldb, int ldc,
                                      int ldd, bool qsplit, Get get) {
    static_assert(ND == 1 || NF == 1, "two outputs take one intermediate");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool two = m1 > 32;     // second row tile of F
    const bool twoD = mD > 32;    // second row tile of D
    const int nq = qsplit && twoD ? 2 : 1;
    const int nstrip = (n1 + 31) >> 5, nitems = nu * nstrip * nq;
    const int sa = 4 * lda, sb = TB ? 4 * ldb : 4;  // bytes per k step of A and op(B)
    const int kf = k1 & ~15;      // whole 16-deep slices
#pragma nounroll
    for (int it = (w - wave0 + 2 * MQE_WAVES) % MQE_WAVES; it < nitems; it += MQE_WAVES) {
        const int qi = it % nq, rest = it / nq;
        const int u = rest / nstrip, c0 = (rest - u * nstrip) * 32;
        const bool do0 = nq == 1 || qi == 0, do1 = twoD && (nq == 1 || qi == 1);  // D row tiles of this item
        const ChainOps<float> op = get(u);
        // the lane coordinates as opaque values inside the loops: the per-element
        // offsets below are then formed next to their loads instead of being
        // hoisted out of the loops and held in registers throughout
        int r = lane & 31, h = lane >> 5;
        v16f_c D0, D1;  // the (at most two) row tiles of the D strip being formed
#pragma nounroll
        for (int f = 0; f < NF; ++f) {
            asm volatile("" : "+v"(r), "+v"(h));
            const int col = min(c0 + r, n1 - 1);
            const int vA0 = 4 * min(r, m1 - 1), vA1 = 4 * min(32 + r, m1 - 1);
            const int vB = TB ? 4 * col : 4 * ldb * col;
            const int row0 = min(r, mD - 1), row1 = min(32 + r, mD - 1);
            // ---- first chain: the F_f strip; lane (r, h) takes k = k0 + 8h + q of the
            // slice at k0; in the last, partial slice k >= k1 reads 0 ----
            v16f_c F0, F1;
#pragma unroll
            for (int e = 0; e < 16; ++e) F0[e] = F1[e] = 0.f;
            const auto rA = buf_rsrc(op.A), rB = buf_rsrc(f == 0 ? op.B[0] : op.B[1]);
            auto slice = [&](int k0, bool tail) {
                float a0[8], a1[8], bv[8];
                const int kl = k0 + 8 * h;
                // tail: k >= k1 reads 0 (offset beyond the range)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const bool ok = !tail || kl + q < k1;
                    a0[q] = buf_ld(rA, ok ? vA0 + sa * (kl + q) : BUF_OOB);
                    bv[q] = buf_ld(rB, ok ? vB + sb * (kl + q) : BUF_OOB);
                }
                if (two) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) a1[q] = buf_ld(rA, !tail || kl + q < k1 ? vA1 + sa * (kl + q) : BUF_OOB);
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) F0 = mfma32(a0[q], bv[q], F0);
                if (two) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) F1 = mfma32(a1[q], bv[q], F1);
                }
            };
#pragma nounroll
            for (int k0 = 0; k0 < kf; k0 += 16) slice(k0, false);
            if (kf < k1) slice(kf, true);
            if (m1 & 31) {  // rows of F beyond m1 (clamped A rows) must not contribute
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = 8 * (e >> 2) + 4 * h + (e & 3);
                    if (row >= m1) F0[e] = 0.f;
                    if (32 + row >= m1) F1[e] = 0.f;
                }
            }
            // ---- second chain: D_d (+)= op(C) F_f, row tile by row tile; a D strip
            // is stored once its last term is in ----
#pragma nounroll
            for (int d = 0; d < ND; ++d) {
                asm volatile("" : "+v"(r), "+v"(h));
                if (ND == 2 || f == 0) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) D0[e] = D1[e] = 0.f;
                }
                const float *Cp = (ND == 1 ? f : d) == 0 ? op.C[0] : op.C[1];
                const auto rC = buf_rsrc(Cp);
                const bool vecC = TC && (m1 & 3) == 0 && (ldc & 3) == 0 && aligned16(Cp, Cp, 0, 0);
                auto chunk = [&](int row, int t, float (&cv)[16]) {
                    if (TC && vecC) {
                        // a run at or beyond m1 meets zero rows of F: any values of C do
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            buf_ld4(rC, 4 * (ldc * row + min(32 * t + 8 * g + 4 * h, m1 - 4)), cv + 4 * g);
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int k = min(32 * t + 8 * (e >> 2) + 4 * h + (e & 3), m1 - 1);
                            cv[e] = buf_ld(rC, TC ? 4 * (ldc * row + k) : 4 * (row + ldc * k));
                        }
                    }
                };
                auto rowtile = [&](int row, v16f_c &Dq) {
                    float c0v[16], c1v[16];
                    chunk(row, 0, c0v);
                    if (two) chunk(row, 1, c1v);
#pragma unroll
                    for (int q = 0; q < 16; ++q) Dq = mfma32(c0v[q], F0[q], Dq);
                    if (two) {
#pragma unroll
                        for (int q = 0; q < 16; ++q) Dq = mfma32(c1v[q], F1[q], Dq);
                    }
                };
                if (do0) rowtile(row0, D0);
                if (do1) rowtile(row1, D1);
                if (f == NF - 1) {
                    // rows 8(e/4) + 4h + e%4 (+32) of column c0 + r; outside D the store is dropped
                    const int vd = c0 + r < n1 ? 4 * (ldd * (c0 + r) + 4 * h) : BUF_OOB;
                    const auto rD = buf_rsrc(d == 0 ? op.D[0] : op.D[1]);
                    if (do0) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int rr = 8 * (e >> 2) + 4 * h + (e & 3), imm = 4 * (8 * (e >> 2) + (e & 3));
                            buf_st(D0[e], rD, rr < mD ? vd : BUF_OOB, imm);
                        }
                    }
                    if (do1) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int rr = 32 + 8 * (e >> 2) + 4 * h + (e & 3), imm = 4 * (32 + 8 * (e >> 2) + (e & 3));
                            buf_st(D1[e], rD, rr < mD ? vd : BUF_OOB, imm);
                        }
                    }
                }
            }
        }
    }
    return (wave0 + nitems) % MQE_WAVES;
}

// The same chained products with 16-column strips (v_mfma_f32_16x16x4f32):
// F row tiles and D row tiles of 16 rows (at most four each), lane (c, g)
// (c = lane % 16, g = lane / 16) takes k = k0 + 4g + q of a 16-deep slice, and
// accumulator slot e of lane (c, g) holds row 4g + e of its tile, so MFMA e of
// F tile t in the second chain takes rows 16t + 4g + e.  For walker bonds below
// 32 (no half-empty strips, twice the items); wider bonds keep 32-column strips
// (a bond of 48 in three 16-column strips re-reads A and C three times and
// measured 20 % slower than two 32-column strips).
// qsplit: the D row tiles 0-1 and 2-3 are separate items.
// SEP (NF = 2): the two terms of D are summed by themselves and then added
// (shorter sums, a smaller rounding error, sixteen more registers).
// FP64 (v_mfma_f64_16x16x4f64) takes all bonds up to 64 this way.  Its
// accumulator slot e of lane (c, g) holds row g + 4e, so MFMA e of F tile t in
// the second chain takes rows 16t + g + 4e.  The general products' vector-unit
// loops read both operands of every multiplication from memory and pass the
// intermediate through it; 48 walkers of the 4x4 torus at D = 20 took 18.4 ms a
// step with them and take 7.6 ms with the chains; 128 walkers of a 16-site chain at
// D = 16: 1042 and 739 us.
template <typename T>
struct Chain16;
template <>
struct Chain16<float> {
    typedef float V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mfma(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int e) { return 4 * g + e; }
    static constexpr int ROW_G = 4, ROW_E = 1;  // row = ROW_G g + ROW_E e
};
template <>
struct Chain16<double> {
    typedef double V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mfma(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int e) { return g + 4 * e; }
    static constexpr int ROW_G = 1, ROW_E = 4;
};

template <bool TB, bool TC, int NF, int ND, typename T, bool SEP = false, class Get>
__device__ __forceinline__ int chain2_16(int wave0, int nu, int m1, int n1, int k1, int mD, int lda, int ldb, int ldc,
                                         int ldd, bool qsplit, Get get) {
    typedef Chain16<T> CT;
    typedef typename CT::V4 V4;
    constexpr int SZ = sizeof(T);
    static_assert(ND == 1 || NF == 1, "two outputs take one intermediate");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int MT = (m1 + 15) >> 4, QT = (mD + 15) >> 4;  // F and D row tiles (<= 4)
    const int nq = qsplit && QT > 2 ? 2 : 1;
    const int nstrip = (n1 + 15) >> 4, nitems = nu * nstrip * nq;
    const int sa = SZ * lda, sb = TB ? SZ * ldb : SZ;  // bytes per k step of A and op(B)
    const int kf = k1 & ~15;
#pragma nounroll
    for (int it = (w - wave0 + 2 * MQE_WAVES) % MQE_WAVES; it < nitems; it += MQE_WAVES) {
        const int qi = it % nq, rest = it / nq;
        const int u = rest / nstrip, c0 = (rest - u * nstrip) * 16;
        const int q0 = nq == 1 ? 0 : 2 * qi, q1 = nq == 1 ? QT : min(QT, 2 * qi + 2);  // D row tiles of this item
        const ChainOps<T> op = get(u);
        int c = lane & 15, g = lane >> 4;
        V4 D[4], D0[SEP ? 4 : 1];
#pragma nounroll
        for (int f = 0; f < NF; ++f) {
            asm volatile("" : "+v"(c), "+v"(g));
            const int col = min(c0 + c, n1 - 1);
            const int vB = TB ? SZ * col : SZ * ldb * col;
            // ---- first chain: the F_f strip (16 columns), up to four 16-row tiles ----
            V4 F[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) F[t] = V4{0, 0, 0, 0};
            const auto rA = buf_rsrc(op.A), rB = buf_rsrc(f == 0 ? op.B[0] : op.B[1]);
            // the last, partial slice takes k = kf + 4q + g, so that a step wholly past k1 is left out
            auto slice = [&](int k0, bool tail) {
                T a[4][4], bv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = tail ? k0 + 4 * q + g : k0 + 4 * g + q;
                    const bool ok = !tail || k < k1;
                    bv[q] = buf_ld<T>(rB, ok ? vB + sb * k : BUF_OOB);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        a[t][q] = t < MT ? buf_ld<T>(rA, ok ? SZ * min(16 * t + c, m1 - 1) + sa * k : BUF_OOB) : T(0);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (tail && k0 + 4 * q >= k1) break;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (t < MT) F[t] = CT::mfma(a[t][q], bv[q], F[t]);
                }
            };
#pragma nounroll
            for (int k0 = 0; k0 < kf; k0 += 16) slice(k0, false);
            if (kf < k1) slice(kf, true);
            if (m1 & 15) {  // rows of F beyond m1 (clamped A rows) must not contribute
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (16 * t + CT::row(g, e) >= m1) F[t][e] = T(0);
            }
            // ---- second chain: D_d (+)= op(C) F_f, 16-row tile by tile ----
#pragma nounroll
            for (int d = 0; d < ND; ++d) {
                asm volatile("" : "+v"(c), "+v"(g));
                const T *Cp = (ND == 1 ? f : d) == 0 ? op.C[0] : op.C[1];
                const auto rC = buf_rsrc(Cp);
                const bool vecC = TC && SZ == 4 && (m1 & 3) == 0 && (ldc & 3) == 0 && (((uintptr_t)Cp) & 15u) == 0;
                if (SEP && f == 1) {
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd) D0[SEP ? qd : 0] = D[qd];
                }
                if (SEP || ND == 2 || f == 0) {
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd) D[qd] = V4{0, 0, 0, 0};
                }
#pragma unroll
                for (int qd = 0; qd < 4; ++qd) {
                    if (qd < q0 || qd >= q1) continue;
                    const int row = min(16 * qd + c, mD - 1);
                    T cv[4][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        if (t >= MT) continue;
                        if (TC && SZ == 4 && vecC) {
                            // a run at or beyond m1 meets zero rows of F: any values of C do
                            buf_ld4(rC, 4 * (ldc * row + min(16 * t + 4 * g, m1 - 4)), (float *)cv[t]);
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int k = min(16 * t + CT::row(g, e), m1 - 1);
                                cv[t][e] = buf_ld<T>(rC, TC ? SZ * (ldc * row + k) : SZ * (row + ldc * k));
                            }
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        if (t >= MT) continue;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (CT::ROW_G == 1 && 16 * t + 4 * e >= m1) break;  // rows 4e .. 4e + 3 of F are zero
                            D[qd] = CT::mfma(cv[t][e], F[t][e], D[qd]);
                        }
                    }
                }
                if (SEP && f == 1) {
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd) D[qd] += D0[SEP ? qd : 0];
                }
                if (f == NF - 1) {
                    // row 16 qd + row(g, e) of column c0 + c; outside D the store is dropped
                    const int vd = c0 + c < n1 ? SZ * (ldd * (c0 + c) + CT::ROW_G * g) : BUF_OOB;
                    const auto rD = buf_rsrc(d == 0 ? op.D[0] : op.D[1]);
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd) {
                        if (qd < q0 || qd >= q1) continue;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            buf_st(D[qd][e], rD, 16 * qd + CT::row(g, e) < mD ? vd : BUF_OOB, SZ * (16 * qd + CT::ROW_E * e));
                    }
                }
            }
        }
    }
    return (wave0 + nitems) % MQE_WAVES;
}

// ---------------------------------------------------------------------------
// Householder QR (LAPACK geqrf/orgqr conventions), FP64, whole workgroup.
// A: m x n (m >= n), column c at Ac(c) (columns c < c_split at A + m c, the
// others at B + m (c - c_split): the caller may keep the trailing columns,
// which receive most of the updates, in LDS).  On exit the columns hold Q and
// R (n x n, ld n) the upper triangle.  tau: n.
// Column c belongs to wave c % 4 for the whole factorisation: the owner of
// column j forms reflector j from its (already updated) column, one
// workgroup barrier publishes it, and every wave applies it to its own
// columns, four columns at a time, with the 64 lanes running down the rows
// (coalesced) and wave reductions for the dot products.  Q is accumulated
// backwards the same way (one barrier per reflector).
// ---------------------------------------------------------------------------
struct QRCols {
    double *A, *B;
    int m, c_split;
    __device__ double *operator()(int c) const { return c < c_split ? A + (size_t)m * c : B + (size_t)m * (c - c_split); }
};

__device__ __forceinline__ void reflect_own_columns(const QRCols &col, int n, int j, double tj, int w, int lane) {
    const int m = col.m;
    const double *vj = col(j);
    int c = j + 1 + ((w - (j + 1)) & (MQE_WAVES - 1));  // first column > j owned by this wave
    for (; c < n; c += 4 * MQE_WAVES) {
        double *cp[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) cp[q] = col(c + MQE_WAVES * q < n ? c + MQE_WAVES * q : c);
        double s[4] = {0.0, 0.0, 0.0, 0.0};
        for (int i = j + lane; i < m; i += 64) {
            const double v = i == j ? 1.0 : vj[i];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c + MQE_WAVES * q < n) s[q] += v * cp[q][i];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = tj * wave_sum(s[q]);
        for (int i = j + lane; i < m; i += 64) {
            const double v = i == j ? 1.0 : vj[i];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c + MQE_WAVES * q < n) cp[q][i] -= s[q] * v;
        }
    }
}

__device__ __forceinline__ void householder_qr(const QRCols &col, int n, double *R, double *tau) {
    const int m = col.m;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int j = 0; j < n; ++j) {
        if (w == (j & (MQE_WAVES - 1))) {
            double *aj = col(j);
            double ss = 0.0;
            for (int i = j + 1 + lane; i < m; i += 64) {
                const double a = aj[i];
                ss += a * a;
            }
            ss = wave_sum(ss);
            const double alpha = aj[j];
            double tj = 0.0, beta = alpha, scale = 0.0;
            if (ss != 0.0) {
                beta = -copysign(sqrt(alpha * alpha + ss), alpha);
                tj = (beta - alpha) / beta;
                scale = 1.0 / (alpha - beta);
            }
            if (tj != 0.0) {
                for (int i = j + 1 + lane; i < m; i += 64) aj[i] *= scale;
                if (lane == 0) aj[j] = beta;
            }
            if (lane == 0) tau[j] = tj;
        }
        __syncthreads();
        const double tj = tau[j];
        if (tj != 0.0) reflect_own_columns(col, n, j, tj, w, lane);
    }
    __syncthreads();
    for (int e = tid; e < n * n; e += MQE_NT) {
        const int r = e % n, c = e / n;
        R[e] = (r <= c) ? col(c)[r] : 0.0;
    }
    __syncthreads();
    for (int j = n - 1; j >= 0; --j) {
        const double tj = tau[j];
        if (tj != 0.0) reflect_own_columns(col, n, j, tj, w, lane);
        __syncthreads();  // every wave has read reflector j
        if (w == (j & (MQE_WAVES - 1))) {
            double *aj = col(j);
            for (int i = lane; i < m; i += 64) aj[i] = (i < j) ? 0.0 : (i == j ? 1.0 - tj : -tj * aj[i]);
        }
    }
    __syncthreads();
}

// 1 / sqrt(x) and 1 / x of a positive normal x to within rounding: the hardware's
// approximations (about 1e-7) with one third-order correction
__device__ __forceinline__ double rsqrt_d(double x) {
    const double r = __builtin_amdgcn_rsq(x), e = fma(-x * r, r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
__device__ __forceinline__ double recip_d(double x) {
    const double r = __builtin_amdgcn_rcp(x), e = fma(-x, r, 1.0);
    return fma(r * e, 1.0 + e, r);
}

// Binary exponent of a column held by G lanes (the sum of its magnitudes; 0 for a
// column of zeros or one that is not finite).
template <int G, int NE>
__device__ __forceinline__ int column_exponent(const double (&a)[NE]) {
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < NE; ++t) s += fabs(a[t]);
    return __builtin_amdgcn_frexp_exp(lanes_sum<G>(s));
}
template <int NE>
__device__ __forceinline__ void scale_column(double (&a)[NE], int e) {
#pragma unroll
    for (int t = 0; t < NE; ++t) a[t] = __builtin_amdgcn_ldexp(a[t], e);
}

// ---------------------------------------------------------------------------
// The same factorisation with every column in registers: LPC lanes own a column
// (lane ln its rows ln + LPC t, t < NE), so m <= LPC NE and n <= threads / LPC.
// Column j goes to LDS (V, ld LPC NE, n columns) as soon as reflector j - 1 is
// applied to it, unscaled, and every group forms the reflector from it while it
// applies it: v = (a_jj + sign(a_jj) |a|, a_j+1.., a_m), tau = 1 / (|a| (|a| +
// |a_jj|)), so the norm, root and reciprocal need no exchange of their own and a
// column costs one barrier.  tau: n doubles in LDS.
// load(r, c): element of A (called once per element, before the first barrier);
// put_r(r, c, x): R(r, c) for r <= c, after the last barrier (V may be
// overwritten there if want_q is false); want_q: put_q(r, c, x) gets Q, after a
// barrier past the last read of V.  Ends without a barrier.
// SCALE: every column is brought to unit magnitude by a power of two first and its
// column of R back afterwards (exact; the column of Q is the same).  The unscaled v
// and n2 hold squares, so without it a column below 1e-145 was left as it is: needed
// for FP64 elements, which can be that small, not for the squares of FP32 ones.
// What is left out then is below 1e-145 of its column.
// What bounds it: the chain of one column (LDS read, dot products, group sums,
// root and reciprocal, update, LDS write, barrier), which nothing overlaps within
// a walker.  So rows past m are zeros instead of bounds checks, groups that are
// done run along with a zero factor, and there is no division on the chain: with
// the owner of a column forming its reflector first, and a branch per element,
// one sweep over the 31 inner sites of a D = 32 chain added 1258 us to a step,
// now 681 us.
// ---------------------------------------------------------------------------
template <int LPC, int NE, bool SCALE = false, class Load, class PutR, class PutQ>
__device__ __forceinline__ void qr_regs(int m, int n, double *V, double *tau, bool want_q, Load load, PutR put_r,
                                        PutQ put_q) {
    constexpr int LDV = LPC * NE;
    const int g = threadIdx.x / LPC, ln = threadIdx.x % LPC;
    const int glast = __builtin_amdgcn_readfirstlane((int)(threadIdx.x | 63) / LPC);  // the wave's last column
    double a[NE], x[NE];
#pragma unroll
    for (int t = 0; t < NE; ++t) {
        const int r = ln + LPC * t;
        a[t] = r < m && g < n ? load(r, g) : 0.0;
        x[t] = 0.0;
    }
    const int ex = SCALE ? column_exponent<LPC>(a) : 0;
    if (SCALE) scale_column(a, -ex);
    __syncthreads();  // V may overlay what load() reads
    double *vg = V + LDV * g + ln;
    if (g == 0) {
#pragma unroll
        for (int t = 0; t < NE; ++t) vg[LPC * t] = a[t];
    }
    __syncthreads();
    for (int j = 0; j < n; ++j) {
        if (g == j - 1) {  // v_{j-1} in its final form, for Q
#pragma unroll
            for (int t = 0; t < NE; ++t) vg[LPC * t] = x[t];
        }
        if (glast >= j) {
            // the raw column j; the rows above j hold R already
            const double *vj = V + LDV * j;
            const double alpha = vj[j];
            double ss = 0.0, s = 0.0, aj = 0.0;
#pragma unroll
            for (int t = 0; t < NE; ++t) x[t] = vj[ln + LPC * t];
#pragma unroll
            for (int t = 0; t < NE; ++t) {
                const int r = ln + LPC * t;
                x[t] = r > j ? x[t] : 0.0;
                aj += r == j ? a[t] : 0.0;
                ss += x[t] * x[t];
                s += x[t] * a[t];
            }
            ss = lanes_sum<LPC>(ss);
            s = lanes_sum<LPC>(s);
            aj = lanes_sum<LPC>(aj);
            const double n2 = fma(alpha, alpha, ss), nrm = n2 * rsqrt_d(n2), d = nrm + fabs(alpha);
            const bool on = ss > 0.0 && n2 > 1e-290;  // (the products of anything smaller are lost to underflow)
            const double vjj = on ? copysign(d, alpha) : 1.0, tj = on ? recip_d(nrm * d) : 0.0;
            const double f = g >= j ? tj * fma(vjj, aj, s) : 0.0;
#pragma unroll
            for (int t = 0; t < NE; ++t) {
                x[t] = ln + LPC * t == j ? vjj : x[t];
                a[t] = fma(-f, x[t], a[t]);
            }
            if (g == j) tau[j] = tj;
            if (g == j + 1 && g < n) {
#pragma unroll
                for (int t = 0; t < NE; ++t) vg[LPC * t] = a[t];
            }
        }
        __syncthreads();
    }
    if (g < n) {
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            const int r = ln + LPC * t;
            if (r <= g) put_r(r, g, SCALE ? __builtin_amdgcn_ldexp(a[t], ex) : a[t]);
        }
    }
    if (!want_q) return;
    if (g == n - 1) {
#pragma unroll
        for (int t = 0; t < NE; ++t) vg[LPC * t] = x[t];
    }
    __syncthreads();
    // Q column c = H_0 H_1 ... H_c e_c; the groups of a wave take the same
    // reflector at the same time, so its LDS reads are broadcasts, and the next
    // reflector is read while the current one is applied
#pragma unroll
    for (int t = 0; t < NE; ++t) a[t] = ln + LPC * t == g ? 1.0 : 0.0;
    const int k0 = min(n - 1, glast);
    double tk = tau[k0];
#pragma unroll
    for (int t = 0; t < NE; ++t) x[t] = V[LDV * k0 + ln + LPC * t];
    for (int k = k0; k >= 0; --k) {
        const int kn = max(k - 1, 0);
        double y[NE], s = 0.0;
        const double tn = tau[kn];
#pragma unroll
        for (int t = 0; t < NE; ++t) y[t] = V[LDV * kn + ln + LPC * t];
#pragma unroll
        for (int t = 0; t < NE; ++t) s += x[t] * a[t];
        s = k <= g ? tk * lanes_sum<LPC>(s) : 0.0;
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            a[t] = fma(-s, x[t], a[t]);
            x[t] = y[t];
        }
        tk = tn;
    }
    __syncthreads();
    if (g < n) {
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            const int r = ln + LPC * t;
            if (r < m) put_q(r, g, a[t]);
        }
    }
}

// qr_regs with the split by size: 8 lanes a column up to 64 x 32, 4 lanes up to
// 128 x 64.  qr_doubles: LDS of V and tau for any matrix of at most 2 D x D.
constexpr int QR_REGS_M = 128, QR_REGS_N = 64;
__host__ __device__ constexpr long qr_doubles(int D) { return (D <= 32 ? 64L : 128L) * D + D; }
template <bool SCALE, class Load, class PutR, class PutQ>
__device__ __forceinline__ void qr_in_regs(int m, int n, double *V, double *tau, bool want_q, Load load, PutR put_r,
                                           PutQ put_q) {
    if (m <= 64 && n <= 32) qr_regs<8, 8, SCALE>(m, n, V, tau, want_q, load, put_r, put_q);
    else qr_regs<4, 32, SCALE>(m, n, V, tau, want_q, load, put_r, put_q);
}

// ---------------------------------------------------------------------------
// The factorisation of larger matrices (m <= 256, n <= 128) by panels of 32
// columns: 8 lanes own a column of the panel in registers (32 rows a lane), the
// panel's reflectors lie in LDS (V, 256 x 32) and, for later, in memory (W, one
// 256 x 32 block per panel; panel_doubles).  A panel first takes the reflectors
// of the panels before it, read back one panel at a time and applied without
// barriers, then factorises itself as in qr_regs; the panels of Q take all
// reflectors the same way backwards.  Arguments as for qr_regs, tau: n doubles.
// What bounds it: FP64 arithmetic of one reflector on 32 columns, about 300
// cycles, times the 320 + 320 reflector passes of a 256 x 128 matrix.  With the
// columns in LDS and memory one factorisation of that size took 3.7 ms, now 0.7 ms.
// (A step of the 6x6 snake at D = 128, 256 walkers: 211 -> 151 ms.)
// ---------------------------------------------------------------------------
constexpr int QR_PANEL = 32, QR_PANELS_M = 256, QR_PANELS_N = 128;
__host__ __device__ constexpr long panel_doubles(int n) {
    return (long)QR_PANELS_M * QR_PANEL * ((n + QR_PANEL - 1) / QR_PANEL);
}
template <bool SCALE, class Load, class PutR, class PutQ>
__device__ __forceinline__ void qr_panels(int m, int n, double *V, double *tau, double *W, Load load, PutR put_r,
                                          PutQ put_q) {
    constexpr int LPC = 8, NE = 32, LDV = QR_PANELS_M, PC = QR_PANEL, BLOCK = LDV * PC;
    const int g = threadIdx.x / LPC, ln = threadIdx.x % LPC;
    const int glast = __builtin_amdgcn_readfirstlane((int)(threadIdx.x | 63) / LPC);
    const int np = (n + PC - 1) / PC;
    double a[NE], x[NE];
    double *vg = V + LDV * g + ln;
    auto fetch = [&](int q) {
        __syncthreads();  // every wave is done with the panel in LDS
        const double *src = W + (size_t)q * BLOCK;
#pragma unroll 8
        for (int e = threadIdx.x; e < BLOCK; e += MQE_NT) V[e] = src[e];
        __syncthreads();
    };
    // reflectors k0, k0 + dir, .. (kc of them) of the panel in LDS, its first column q0, to a; own: only k <= g
    auto apply = [&](int q0, int kc, int k0, int dir, bool own) {
        auto read = [&](int k, double (&v)[NE]) {
#pragma unroll
            for (int t = 0; t < NE; ++t) v[t] = V[LDV * k + ln + LPC * t];
        };
        auto step = [&](int k, const double (&v)[NE]) {
            double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int t = 0; t < NE; ++t) s[t & 3] += v[t] * a[t];
            const double d = lanes_sum<LPC>((s[0] + s[1]) + (s[2] + s[3]));
            const double f = !own || k <= g ? tau[q0 + k] * d : 0.0;
#pragma unroll
            for (int t = 0; t < NE; ++t) a[t] = fma(-f, v[t], a[t]);
        };
        double y[NE];
        read(k0, x);
#pragma nounroll
        for (int i = 0; i < kc; i += 2) {
            const int k = k0 + dir * i, k1 = k + dir, k2 = k1 + dir;
            if (i + 1 < kc) read(k1, y);
            step(k, x);
            if (i + 2 < kc) read(k2, x);
            if (i + 1 < kc) step(k1, y);
        }
    };
    for (int c = 0; c < np; ++c) {
        const int base = PC * c, nc = min(PC, n - base);
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            const int r = ln + LPC * t;
            a[t] = r < m && g < nc ? load(r, base + g) : 0.0;
        }
        const int ex = SCALE ? column_exponent<LPC>(a) : 0;
        if (SCALE) scale_column(a, -ex);
        for (int q = 0; q < c; ++q) {
            if (q != c - 1 || c > 1) fetch(q);  // panel 0 is still in LDS when panel 1 needs it
            apply(PC * q, PC, 0, 1, false);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NE; ++t) x[t] = 0.0;
        if (g == 0) {
#pragma unroll
            for (int t = 0; t < NE; ++t) vg[LPC * t] = a[t];
        }
        __syncthreads();
        for (int jj = 0; jj < nc; ++jj) {
            const int j = base + jj;
            if (g == jj - 1) {
#pragma unroll
                for (int t = 0; t < NE; ++t) vg[LPC * t] = x[t];
            }
            if (glast >= jj) {
                const double *vj = V + LDV * jj;
                const double alpha = vj[j];
                double ss[2] = {0.0, 0.0}, s[2] = {0.0, 0.0}, aj = 0.0;
#pragma unroll
                for (int t = 0; t < NE; ++t) x[t] = vj[ln + LPC * t];
#pragma unroll
                for (int t = 0; t < NE; ++t) {
                    const int r = ln + LPC * t;
                    x[t] = r > j ? x[t] : 0.0;
                    aj = r == j ? a[t] : aj;
                    ss[t & 1] += x[t] * x[t];
                    s[t & 1] += x[t] * a[t];
                }
                const double sx = lanes_sum<LPC>(ss[0] + ss[1]), sa = lanes_sum<LPC>(s[0] + s[1]);
                aj = lanes_sum<LPC>(aj);
                const double n2 = fma(alpha, alpha, sx), nrm = n2 * rsqrt_d(n2), d = nrm + fabs(alpha);
                const bool on = sx > 0.0 && n2 > 1e-290;
                const double vjj = on ? copysign(d, alpha) : 1.0, tj = on ? recip_d(nrm * d) : 0.0;
                const double f = g >= jj ? tj * fma(vjj, aj, sa) : 0.0;
#pragma unroll
                for (int t = 0; t < NE; ++t) {
                    x[t] = ln + LPC * t == j ? vjj : x[t];
                    a[t] = fma(-f, x[t], a[t]);
                }
                if (g == jj) tau[j] = tj;
                if (g == jj + 1 && g < nc) {
#pragma unroll
                    for (int t = 0; t < NE; ++t) vg[LPC * t] = a[t];
                }
            }
            __syncthreads();
        }
        if (g == nc - 1) {
#pragma unroll
            for (int t = 0; t < NE; ++t) vg[LPC * t] = x[t];
        }
        if (g < nc) {
#pragma unroll
            for (int t = 0; t < NE; ++t) {
                const int r = ln + LPC * t;
                if (r <= base + g) put_r(r, base + g, SCALE ? __builtin_amdgcn_ldexp(a[t], ex) : a[t]);
            }
        }
        __syncthreads();
        if (c < np - 1 || np > 1) {
            double *dst = W + (size_t)c * BLOCK;
#pragma unroll 8
            for (int e = threadIdx.x; e < LDV * nc; e += MQE_NT) dst[e] = V[e];
        }
    }
    // Q by panels: column base + g starts as a unit vector
    for (int p = np - 1; p >= 0; --p) {
        const int base = PC * p;
#pragma unroll
        for (int t = 0; t < NE; ++t) a[t] = ln + LPC * t == base + g ? 1.0 : 0.0;
        for (int q = p; q >= 0; --q) {
            if (q != np - 1) fetch(q);  // the last panel's reflectors are in LDS
            const int kc = min(PC, n - PC * q);
            apply(PC * q, kc, kc - 1, -1, q == p);
        }
        if (base + g < n) {
#pragma unroll
            for (int t = 0; t < NE; ++t) {
                const int r = ln + LPC * t;
                if (r < m) put_q(r, base + g, a[t]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) counter-based RNG.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t philox_u32(uint64_t key, uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3) {
    uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c0;
}

__device__ __forceinline__ double philox_uniform(uint64_t key, uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3) {
    return (double)philox_u32(key, c0, c1, c2, c3) * (1.0 / 4294967296.0);
}

}  // namespace mqe

#endif
