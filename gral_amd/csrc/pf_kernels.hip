// HIP kernels of the prognostic microscale flow solver (gfx950).
//
// One SIMPLE iteration (PrognosticFlowfield.cs:584-1178) is a sequence of
//   stencil passes   - sub-domain BCs, divergence, velocity correction, averages:
//                      one thread per (column, level), k contiguous -> coalesced;
//   Gauss-Seidel passes - pressure TDMA, U/V/W momentum, TKE/eps:
//                      the reference updates columns in place in lexicographic
//                      sweep order (a outer, b inner).  A column depends on the
//                      new values of (a-1,b) and (a,b-1) only, so all columns of
//                      one anti-diagonal a+b=t are independent.  A pass is one
//                      launch of strips: workgroups of consecutive rows that
//                      advance as a wavefront, the Thomas recurrences, serial in
//                      k, of a strip's columns on one wave (lane = row).  Very
//                      tall columns take one launch per anti-diagonal instead,
//                      one wave per column (lanes over k for the coefficients,
//                      one lane for the recurrences).
// This replays the reference's deterministic (single-thread) order exactly.
#include <cmath>
#include <mutex>
#include <type_traits>
#include "pf_device.h"
#include "pf_strip.h"

#define WAVE 64

// ------------------------------------------------------------------------
// diagonal -> column mapping
// ------------------------------------------------------------------------
// Sweep indices a in [oa, ob] (outer), b in [ia, ib] (inner); diagonal t
// holds the columns with (a-oa)+(b-ia) == t, enumerated by a.
__device__ __forceinline__ bool diag_col(int t, int oa, int ob, int ia, int ib, int idx, int &a, int &b) {
    int nb = ib - ia;
    int amin = max(oa, oa + t - nb);
    int amax = min(ob, oa + t);
    a = amin + idx;
    if (a > amax) return false;
    b = ia + (t - (a - oa));
    return true;
}

// ------------------------------------------------------------------------
// utility
// ------------------------------------------------------------------------
// Workgroups are dealt to the 8 XCDs (each with its own L2) round robin by
// their position in the grid.  For kernels whose neighbouring blocks read each
// other's columns, xcd_block() renumbers the blocks of a launch whose x extent is
// a multiple of 8 so that every XCD takes one contiguous range of logical
// blocks; it is a bijection on [0, n) and returns -1 for the padding blocks.
#define NXCD 8
__device__ __forceinline__ int xcd_block(int n) {
    int b = blockIdx.x, x = b % NXCD, idx = b / NXCD;
    int per = n / NXCD, rem = n % NXCD;
    int cnt = per + (x < rem ? 1 : 0);
    if (idx >= cnt) return -1;
    return x * per + min(x, rem) + idx;
}
// column metadata from the per-column table (see gral_pf_prepare)
struct Meta {
    int KK, VI, KSTART, KKmi, KKmj;
    bool adv, vegp;
};
__device__ __forceinline__ Meta unpack_meta(int4 m) {
    Meta r;
    r.KK = m.x; r.VI = m.y; r.KSTART = m.z & 0xffff; r.adv = (m.z >> 16) & 1; r.vegp = (m.z >> 17) & 1;
    r.KKmi = m.w & 0xffff; r.KKmj = (m.w >> 16) & 0xffff;
    return r;
}

// The cell kernels (divergence, velocity correction, averages) walk the
// interior columns of one sweep row i (j = 2..NJJ-1 are contiguous in memory,
// nkp levels each) as one flat run of floats: a block per row, each thread
// four consecutive levels of one column per step (16-byte accesses; nkp is a
// multiple of 4), so every load of a wave is contiguous and a block keeps
// many independent loads in flight.  Blocks take rows in XCD order.  With
// blocks of 1024 threads (16 waves; about 8 steps per thread on a 400-column
// row) the cell and boundary kernels of the 8-situation city batch take
// 2.01 ms per iteration, against 2.06 with 512, 2.10 with 256, 2.19 with 128.
#ifndef CELL_THREADS
#define CELL_THREADS 1024
#endif

__global__ void k_fill_u32(unsigned *p, size_t n, unsigned v) {
    size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < n) p[g] = v;
}
// Clears the strip synchronisation blocks of the iteration's sweeps; for the
// per-diagonal sweeps (diag) also the pressure row scratch of every situation
// (PIMP/QIMP rows are fresh arrays at the start of each pressure pass; the
// strips keep them in LDS).
__global__ void k_zero_rows(const Dom *__restrict__ ds, int diag) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];
    size_t n = (size_t)d.nj2 * d.nkp;
    size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (diag && g < n) {
        d.prow_q[g] = 0.0f;
        d.prow_p[g] = 0.0f;
    }
    if (d.sync && g < (size_t)5 * d.sync_stride) d.sync[SYNC_BLOCK0 + g] = 0;
    if (d.sync && g == 0) d.sync[1] += 1;                     // the hand-off tags of this iteration's sweeps
}

// ------------------------------------------------------------------------
// Sub-domain boundary conditions, PrognosticFlowfield.cs:595-714
// ------------------------------------------------------------------------
// E/W: each row j is independent; within a row the reference scans i upwards
// and later i read what earlier i wrote, so one thread per (j,k) scans i.  One
// block per row: the row's ADVDOM and VerticalIndex are staged in LDS first,
// and one wave lists the row's edge cells (ADVDOM = 1 next to a cell outside
// the sub-domains, or at the first / last interior index) in increasing order,
// so the scan visits only the cells where the reference's loop does anything,
// in the reference's order.
// LDS per block: [n] VI, [n] edge list, its length, then [n] ADVDOM bytes.
__host__ __device__ inline size_t bc_lds_bytes(int n) { return (size_t)(2 * n + 1) * sizeof(int) + n; }
// the indices x in [3, last] with adv[x] = 1 and at least one of adv[x-1] < 1,
// adv[x+1] < 1, x = 3, x = last, ascending, into edges[]; returns their count
// (to every thread of the block)
__device__ __forceinline__ int bc_edges(const uint8_t *adv, int last, int *edges, int *count) {
    if (threadIdx.x < WAVE) {
        const int lane = threadIdx.x;
        int cnt = 0;
        for (int base = 3; base <= last; base += WAVE) {
            const int x = base + lane;
            const bool e = x <= last && adv[x] == 1 && (adv[x - 1] < 1 || x == 3 || adv[x + 1] < 1 || x == last);
            const unsigned long long m = __ballot(e);
            if (e) edges[cnt + __popcll(m & ((1ull << lane) - 1))] = x;
            cnt += __popcll(m);
        }
        if (lane == 0) *count = cnt;
    }
    __syncthreads();
    return *count;
}
__global__ void k_bc_ew(const Dom *__restrict__ ds) {
    extern __shared__ int bc_row[];
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    if ((int)blockIdx.y >= d.njj - 1) return;

    int j = blockIdx.y + 2;                   // 2..NJJ
    const int n = d.nii + 2;
    int *svi = bc_row, *sedge = bc_row + n;
    uint8_t *sadv = reinterpret_cast<uint8_t *>(bc_row + 2 * n + 1);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const size_t c = c2(d, i, j);
        svi[i] = d.vi[c];
        sadv[i] = d.adv[c];
    }
    __syncthreads();
    const int nedge = bc_edges(sadv, d.nii - 1, sedge, bc_row + 2 * n);
    for (int k = threadIdx.x + 1; k <= d.kadvmax; k += blockDim.x)
    for (int q = 0; q < nedge; ++q) {
        const int i = sedge[q];
        if (k > svi[i]) continue;
        bool iM = (sadv[i - 1] < 1) || (i == 3);
        bool iP = (sadv[i + 1] < 1) || (i == d.nii - 1);
        if (iM) {
            float u = d.uk[c3(d, i - 2, j) + k];
            if (u >= 0) d.uk[c3(d, i - 1, j) + k] = u;
            d.vk[c3(d, i - 2, j) + k] = d.vk[c3(d, i - 1, j) + k];
            d.wk[c3(d, i - 2, j) + k] = d.wk[c3(d, i - 1, j) + k];
        }
        if (iP) {
            float u = d.uk[c3(d, i + 2, j) + k];
            if (u <= 0) d.uk[c3(d, i + 1, j) + k] = u;
            d.vk[c3(d, i + 1, j) + k] = d.vk[c3(d, i, j) + k];
            d.wk[c3(d, i + 1, j) + k] = d.wk[c3(d, i, j) + k];
        }
    }
}

// N/S: as E/W with the roles of i and j exchanged (the edge list over j)
__global__ void k_bc_ns(const Dom *__restrict__ ds) {
    extern __shared__ int bc_row[];
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    if ((int)blockIdx.y >= d.nii - 1) return;

    int i = blockIdx.y + 2;                   // 2..NII
    const int n = d.njj + 2;
    int *svi = bc_row, *sedge = bc_row + n;
    uint8_t *sadv = reinterpret_cast<uint8_t *>(bc_row + 2 * n + 1);
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const size_t c = c2(d, i, j);
        svi[j] = d.vi[c];
        sadv[j] = d.adv[c];
    }
    __syncthreads();
    const int nedge = bc_edges(sadv, d.njj - 1, sedge, bc_row + 2 * n);
    for (int k = threadIdx.x + 1; k <= d.kadvmax; k += blockDim.x)
    for (int q = 0; q < nedge; ++q) {
        const int j = sedge[q];
        if (k > svi[j]) continue;
        bool jM = (sadv[j - 1] < 1) || (j == 3);
        bool jP = (sadv[j + 1] < 1) || (j == d.njj - 1);
        if (jM) {
            float v = d.vk[c3(d, i, j - 2) + k];
            if (v >= 0) d.vk[c3(d, i, j - 1) + k] = v;
            d.uk[c3(d, i, j - 2) + k] = d.uk[c3(d, i, j - 1) + k];
            d.wk[c3(d, i, j - 2) + k] = d.wk[c3(d, i, j - 1) + k];
        }
        if (jP) {
            float v = d.vk[c3(d, i, j + 2) + k];
            if (v <= 0) d.vk[c3(d, i, j + 1) + k] = v;
            d.uk[c3(d, i, j + 1) + k] = d.uk[c3(d, i, j) + k];
            d.wk[c3(d, i, j + 1) + k] = d.wk[c3(d, i, j) + k];
        }
    }
    // top of the sub-domains, VI -> VI+1 (PrognosticFlowfield.cs:698-714): the
    // N/S pass of this row has written all it writes of the row's columns, and
    // no other row writes them
    if (i > d.nii - 1) return;
    __syncthreads();
    for (int j = 2 + threadIdx.x; j <= d.njj - 1; j += blockDim.x) {
        if (sadv[j] != 1) continue;
        const int k = svi[j];
        const size_t o = c3(d, i, j);
        d.wk[o + k + 1] = d.wk[o + k];
        d.uk[o + k + 1] = d.uk[o + k];
        d.vk[o + k + 1] = d.vk[o + k];
    }
}

// ------------------------------------------------------------------------
// Mass divergence, PrognosticFlowfield.cs:723-758, over the active cells
// (ADVDOM = 1, KKART < k <= VI); DPM = 0 there.  The array keeps DIV / DTIME,
// the only form the pressure sweep reads (its source term, :853), divided here
// in the bandwidth-bound pass rather than on the sweep's serial path (the same
// correctly rounded division, so the same bits).
// ------------------------------------------------------------------------
__global__ __launch_bounds__(CELL_THREADS) void k_divergence(const Dom *__restrict__ ds) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    const int blk = xcd_block(d.nii - 2);
    if (blk < 0) return;
    const int i = 2 + blk, nkp = d.nkp, n4 = ((d.njj - 2) * nkp) >> 2;
    const size_t row = c3(d, i, 2), ip = (size_t)d.nj2 * nkp;
    for (int q = threadIdx.x; q < n4; q += CELL_THREADS) {
        const int e = q << 2, jo = e / nkp, k0 = e - jo * nkp;
        const Meta m = unpack_meta(ldg4i(d.meta + c2(d, i, 2 + jo)));
        if (!m.adv || k0 + 3 <= m.KK || k0 > m.VI) continue;
        const size_t o = row + e;
        const float4 u = ldg4(d.uk + o), ue = ldg4(d.uk + o + ip), v = ldg4(d.vk + o), vn = ldg4(d.vk + o + nkp);
        const float4 w = ldg4(d.wk + o);
        const float uu[4] = {u.x, u.y, u.z, u.w}, uue[4] = {ue.x, ue.y, ue.z, ue.w};
        const float vv[4] = {v.x, v.y, v.z, v.w}, vvn[4] = {vn.x, vn.y, vn.z, vn.w};
        const float ww[5] = {w.x, w.y, w.z, w.w, d.wk[o + 4]};
        float r[4];
        bool on[4];
#pragma unroll
        for (int u4 = 0; u4 < 4; ++u4) {
            const int k = k0 + u4;
            on[u4] = m.KK < k && k <= m.VI;
            r[u4] = 0.0f;
            if (on[u4]) {
                const float dz = d.dzk[k];
                const float t1 = (uu[u4] - uue[u4]) * d.dyk * dz;
                const float t2 = (vv[u4] - vvn[u4]) * d.dxk * dz;
                r[u4] = (k > m.KK + 1) ? t1 + t2 + (ww[u4] - ww[u4 + 1]) * d.area : t1 + t2 - ww[u4 + 1] * d.area;
                r[u4] = r[u4] / d.dtime;
            }
        }
        if (on[0] && on[1] && on[2] && on[3]) {
            stg4(d.div + o, r[0], r[1], r[2], r[3]);
            stg4(d.dpm + o, 0.0f, 0.0f, 0.0f, 0.0f);
        } else {
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4)
                if (on[u4]) { d.div[o + u4] = r[u4]; d.dpm[o + u4] = 0.0f; }
        }
    }
}

// ------------------------------------------------------------------------
// Pressure-correction GS-TDMA, PrognosticFlowfield.cs:770-901.
// Sweep: a = j1 in [2,NJJ-1] (outer), b = i1 in [2,NII-1] (inner).
// PIMP/QIMP live per sweep row in global scratch, zeroed at the start of the
// pass, so the top coupling PIMP[VI+1] sees what the last earlier column of
// the same row left there, as in the reference.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(WAVE) void k_pressure(const Dom *__restrict__ ds, int t, int IS, int JS, int slot) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice

    extern __shared__ float sm[];
    int a, b;
    if (!diag_col(t, 2, d.njj - 1, 2, d.nii - 1, blockIdx.x, a, b)) return;
    int j = (JS == -1) ? d.njj - a + 1 : a;
    int i = (IS == -1) ? d.nii - b + 1 : b;
    size_t c = c2(d, i, j);
    if (d.adv[c] != 1) return;
    const int nkp = d.nkp, tid = threadIdx.x;
    float *sDIM = sm, *sP = sDIM + nkp, *sQ = sP + nkp, *sN = sQ + nkp, *sO = sN + nkp;
    int KK = d.kk[c], VI = d.vi[c];
    size_t o = c3(d, i, j), oim = c3(d, i - 1, j), oip = c3(d, i + 1, j), ojm = c3(d, i, j - 1), ojp = c3(d, i, j + 1);
    float DXK = d.dxk, DYK = d.dyk;
    for (int k = KK + 1 + tid; k <= VI; k += WAVE) {
        float dz = d.dzk[k];
        float DIM = d.div[o + k] + (d.dpm[oim + k] + d.dpm[oip + k]) / DXK * DYK * dz +
                    (d.dpm[ojm + k] - d.dpm[ojp + k]) / DYK * DXK * dz;
        sDIM[k] = DIM;
    }
    for (int k = KK + tid; k <= VI; k += WAVE) sO[k] = d.dpm[o + k];
    size_t row = (size_t)j * nkp;
    __syncthreads();
    if (tid == 0) {
        float Pn = d.prow_p[row + VI + 1], Qn = d.prow_q[row + VI + 1];
        for (int k = VI; k > KK; --k) {
            float ATP = d.atp[k];
            float TERMP = 1 / (d.app[k] - ATP * Pn);
            float P = d.abp[k] * TERMP;
            float Q = (ATP * Qn + sDIM[k]) * TERMP;
            sP[k] = P; sQ[k] = Q;
            Pn = P; Qn = Q;
        }
        float dprev = sO[KK];
        for (int k = KK + 1; k <= VI; ++k) {
            float temp = sP[k] * dprev + sQ[k];
            sN[k] = temp;
            dprev = temp;
        }
    }
    __syncthreads();
    float rmax = 0.0f;
    for (int k = KK + 1 + tid; k <= VI; k += WAVE) {
        float temp = sN[k];
        double q = (double)conv_to_int((double)temp * d.frund) / d.frund;
        float r = (float)fabs((double)sO[k] - q);
        rmax = r > rmax ? r : rmax;
        d.dpm[o + k] = temp;
        d.dpmnew[o + k] = d.dpmnew[o + k] + d.relaxp * temp;
        d.prow_p[row + k] = sP[k];
        d.prow_q[row + k] = sQ[k];
    }
    for (int off = WAVE / 2; off > 0; off >>= 1) {
        float other = __shfl_xor(rmax, off);
        rmax = other > rmax ? other : rmax;
    }
    const int rs = slot - d.iter_off;                 // this situation's residual slot
    if (tid == 0 && rmax > 0.0f && slot >= 0 && rs >= 0 && rs < d.resid_cap) atomicMax((unsigned *)&d.resid[rs], __float_as_uint(rmax));
}

// ------------------------------------------------------------------------
// Velocity correction with FP64 quantisation, PrognosticFlowfield.cs:904-949,
// over the columns with ADVDOM = 1 at (i,j), (i-1,j) or (i,j-1), levels 1..VI.
// ------------------------------------------------------------------------
__device__ __forceinline__ bool corr_column(const DomG &d, int i, int j, bool adv) {
    return adv || d.adv[c2(d, i - 1, j)] == 1 || d.adv[c2(d, i, j - 1)] == 1;
}
__global__ __launch_bounds__(CELL_THREADS) void k_correction(const Dom *__restrict__ ds) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    const int blk = xcd_block(d.nii - 2);
    if (blk < 0) return;
    const int i = 2 + blk, nkp = d.nkp, n4 = ((d.njj - 2) * nkp) >> 2;
    const size_t row = c3(d, i, 2), ip = (size_t)d.nj2 * nkp;
    const bool q = !d.noquant;
    for (int t = threadIdx.x; t < n4; t += CELL_THREADS) {
        const int e = t << 2, jo = e / nkp, k0 = e - jo * nkp, j = 2 + jo;
        const Meta m = unpack_meta(ldg4i(d.meta + c2(d, i, j)));
        if (k0 > m.VI || !corr_column(d, i, j, m.adv)) continue;
        const size_t o = row + e;
        const float4 p = ldg4(d.dpm + o), pw = ldg4(d.dpm + o - ip), ps = ldg4(d.dpm + o - nkp);
        const float4 u = ldg4(d.uk + o), v = ldg4(d.vk + o), w = ldg4(d.wk + o);
        const float pp[5] = {d.dpm[o - 1], p.x, p.y, p.z, p.w};              // pp[u4 + 1]: level k0 + u4
        const float ppw[4] = {pw.x, pw.y, pw.z, pw.w}, pps[4] = {ps.x, ps.y, ps.z, ps.w};
        float uu[4] = {u.x, u.y, u.z, u.w}, vv[4] = {v.x, v.y, v.z, v.w}, ww[4] = {w.x, w.y, w.z, w.w};
        bool onu[4], onv[4], on[4];
#pragma unroll
        for (int u4 = 0; u4 < 4; ++u4) {
            const int k = k0 + u4;
            on[u4] = k >= 1 && k <= m.VI;
            onu[u4] = on[u4] && i > 2 && m.KKmi < k;              // KKART(i,j) < k and KKART(i-1,j) < k
            onv[u4] = on[u4] && j > 2 && m.KKmj < k;
            const float dpmk = pp[u4 + 1];
            if (onu[u4]) {
                const float x = uu[u4] + (ppw[u4] - dpmk) / d.dxk * d.dtime;
                uu[u4] = q ? quantise(x, d.frund) : x;
            }
            if (onv[u4]) {
                const float x = vv[u4] + (pps[u4] - dpmk) / d.dyk * d.dtime;
                vv[u4] = q ? quantise(x, d.frund) : x;
            }
            if (on[u4]) {
                if (m.KK + 1 < k) {
                    const float x = ww[u4] + (pp[u4] - dpmk) / (d.dzk[k] + d.dzk[k - 1]) * 2.0f * d.dtime;
                    ww[u4] = q ? quantise(x, d.frund) : x;
                } else {
                    ww[u4] = 0.0f;
                }
            }
        }
        if (onu[0] && onu[1] && onu[2] && onu[3]) stg4(d.uk + o, uu[0], uu[1], uu[2], uu[3]);
        else
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) if (onu[u4]) d.uk[o + u4] = uu[u4];
        if (onv[0] && onv[1] && onv[2] && onv[3]) stg4(d.vk + o, vv[0], vv[1], vv[2], vv[3]);
        else
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) if (onv[u4]) d.vk[o + u4] = vv[u4];
        if (on[0] && on[1] && on[2] && on[3]) stg4(d.wk + o, ww[0], ww[1], ww[2], ww[3]);
        else
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) if (on[u4]) d.wk[o + u4] = ww[u4];
    }
}

// ------------------------------------------------------------------------
// Cell-centred averages, PrognosticFlowfield.cs:958-1014 (+ UKS row copies),
// over the correction's columns, levels KSTART..VI.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(CELL_THREADS) void k_averages(const Dom *__restrict__ ds) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    const int blk = xcd_block(d.nii - 2);
    if (blk < 0) return;
    const int i = 2 + blk, nkp = d.nkp, n4 = ((d.njj - 2) * nkp) >> 2;
    const size_t row = c3(d, i, 2), ip = (size_t)d.nj2 * nkp;
    const bool copy_n = d.adv[c2(d, i, d.njj)] == 1;
    for (int t = threadIdx.x; t < n4; t += CELL_THREADS) {
        const int e = t << 2, jo = e / nkp, k0 = e - jo * nkp, j = 2 + jo;
        const Meta m = unpack_meta(ldg4i(d.meta + c2(d, i, j)));
        if (k0 + 3 < m.KSTART || k0 > m.VI || !corr_column(d, i, j, m.adv)) continue;
        const size_t o = row + e;
        const float4 u = ldg4(d.uk + o), ue = ldg4(d.uk + o + ip), v = ldg4(d.vk + o), vn = ldg4(d.vk + o + nkp);
        const float4 w = ldg4(d.wk + o);
        const float uu[4] = {u.x, u.y, u.z, u.w}, uue[4] = {ue.x, ue.y, ue.z, ue.w};
        const float vv[4] = {v.x, v.y, v.z, v.w}, vvn[4] = {vn.x, vn.y, vn.z, vn.w};
        const float ww[5] = {w.x, w.y, w.z, w.w, d.wk[o + 4]};
        float ru[4], rv[4], rw[4];
        bool on[4], onuv[4], onw[4];
#pragma unroll
        for (int u4 = 0; u4 < 4; ++u4) {
            const int k = k0 + u4;
            on[u4] = k >= m.KSTART && k <= m.VI;
            onuv[u4] = on[u4] && m.KK < k;
            onw[u4] = on[u4] && m.KK + 1 < k;
            ru[u4] = 0.5f * (uu[u4] + uue[u4]);
            rv[u4] = 0.5f * (vv[u4] + vvn[u4]);
            rw[u4] = 0.5f * (ww[u4] + ww[u4 + 1]);
        }
        if (onuv[0] && onuv[1] && onuv[2] && onuv[3]) {
            stg4(d.uks + o, ru[0], ru[1], ru[2], ru[3]);
            stg4(d.vks + o, rv[0], rv[1], rv[2], rv[3]);
        } else {
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4)
                if (onuv[u4]) { d.uks[o + u4] = ru[u4]; d.vks[o + u4] = rv[u4]; }
        }
        if (onw[0] && onw[1] && onw[2] && onw[3]) stg4(d.wks + o, rw[0], rw[1], rw[2], rw[3]);
        else
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) if (onw[u4]) d.wks[o + u4] = rw[u4];
        // UKS[i][1] = UKS[i][2] and UKS[i][NJJ] = UKS[i][NJJ-1] (if ADVDOM there) over
        // KSTART..VI: the new value where it was just written, else the old one
        const bool cs = (j == 2), cn = (j == d.njj - 1) && copy_n;
        if (cs || cn) {
            const size_t oc = cs ? c3(d, i, 1) : c3(d, i, d.njj);
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4)
                if (on[u4]) d.uks[oc + k0 + u4] = onuv[u4] ? ru[u4] : d.uks[o + u4];
        }
    }
}

// VKS[1][j] = VKS[2][j], VKS[NII][j] = VKS[NII-1][j] (PrognosticFlowfield.cs:1019-1039)
__global__ void k_avg_edges(const Dom *__restrict__ ds) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    if ((int)blockIdx.x >= d.njj - 2) return;

    int j = blockIdx.x + 2;                  // 2..NJJ-1
    bool w = d.adv[c2(d, 1, j)] == 1, e = d.adv[c2(d, d.nii - 1, j)] == 1;
    size_t o1 = c3(d, 1, j), o2 = c3(d, 2, j), on = c3(d, d.nii, j), on1 = c3(d, d.nii - 1, j);
    for (int k = threadIdx.x; k < d.nkp; k += blockDim.x) {
        if (w) d.vks[o1 + k] = d.vks[o2 + k];
        if (e) d.vks[on + k] = d.vks[on1 + k];
    }
}

// ------------------------------------------------------------------------
// Mixing-length momentum (turbulence model 1): U/V/W-prognostic-microscale_1.cs
// ------------------------------------------------------------------------
// The reference evaluates a column in vector blocks of W lanes starting at
// KSTART, KSTART+W, ..., the last block moved down to KEND-W.  Every lane
// quantity is lane-local except the gate of the eddy-viscosity cross terms,
// which tests the block start (k_block > KKART+1); block_base() returns the
// start of the block whose lane k enters the recurrence.
// W = 8: Vector<float> solvers (U/V/W-prognostic-microscale_1.cs, AVX2 width);
// W = 16: the 512-bit solvers (U/V/W-prognostic-microscale_1_Vec512.cs), which
// also fuse some multiply-adds (see v512 below).  The host accepts only 8 or 16.
__device__ __forceinline__ int block_base(int k, int KSTART, int KEND, int W) {
    const int sh = (W == 16) ? 4 : 3;
    int base = KSTART + (((k - KSTART) >> sh) << sh);
    if (base > KEND - W) base = KEND - W;
    return base;
}

struct ColInfo {
    int i, j, KK, KSTART, VI, W;
    bool as, an, aw, ae, vegp;
    float cutk, cov, ht, ho, z0s;
    __device__ __forceinline__ bool v512() const { return W == 16; }
};

__device__ __forceinline__ ColInfo col_info(const DomG &d, int i, int j) {
    ColInfo q;
    size_t c = c2(d, i, j);
    q.i = i; q.j = j; q.KK = d.kk[c]; q.VI = d.vi[c];
    q.cutk = d.cutk[c]; q.cov = d.cov[c]; q.ht = d.ht[c]; q.ho = d.ho[c]; q.z0s = d.z0s[c];
    q.KSTART = (q.cutk == 0) ? q.KK + 1 : 1;
    q.vegp = d.vegp != nullptr && d.vegp[c] != 0;
    q.as = (d.adv[c2(d, i, j - 1)] < 1) || (j == 2);
    q.an = (d.adv[c2(d, i, j + 1)] < 1) || (j == d.njj - 1);
    q.aw = (d.adv[c2(d, i - 1, j)] < 1) || (i == 2);
    q.ae = (d.adv[c2(d, i + 1, j)] < 1) || (i == d.nii - 1);
    q.W = d.simd;
    return q;
}

// mixing-length eddy viscosity (U-prognostic-microscale_1.cs:216-268), lane-local;
// the 512-bit solvers fuse the half-cell offset into the ground height
// (U-prognostic-microscale_1_Vec512.cs:218)
__device__ __forceinline__ float ml_visc(const DomG &d, const ColInfo &q, int k, const gf32 *UK, const gf32 *VK) {
    if (!(k > q.KK + 1)) return 0.0f;
    float dz = d.dzk[k];
    float zs = q.v512() ? d.hok[k] - fmaf(dz, 0.5f, d.hok[q.KK]) : d.hok[k] - d.hok[q.KK] - dz * 0.5f;
    float mixL = vminf(0.071f * zs, 100.0f);
    if (q.cov > 0) mixL *= (1.0f - 0.99f * q.cov);
    float in = (UK[k + 1] - UK[k - 1]) / (2.0f * dz);
    float dudz = in * in;
    in = (VK[k + 1] - VK[k - 1]) / (2.0f * dz);
    float dvdz = in * in;
    return vminf(mixL * mixL * sqrtf(0.5f * (dudz + dvdz)), 15.0f);
}

// power-law weight D*max(0,(1-0.1P)^5) in float (Vector path)
__device__ __forceinline__ float plaw_f(float D, float P) {
    float in = 1.0f - 0.1f * P;
    return D * vmaxf(0.0f, in * in * in * in * in);
}

// power-law coefficient plus its upwind flux Fp = max(+-F, 0):
// D*max(0, x^5) + Fp (U-prognostic-microscale_1.cs:345-367), or, in the 512-bit
// solvers, FMA(D, max(0, x*((x*x)*(x*x))), Fp) (U-prognostic-microscale_1_Vec512.cs:355-377)
__device__ __forceinline__ float plaw_coef(bool v512, float D, float P, float Fp) {
    if (!v512) return plaw_f(D, P) + Fp;
    float in = 1.0f - 0.1f * P;
    return fmaf(D, vmaxf(0.0f, in * ((in * in) * (in * in))), Fp);
}

struct Coef { float A, B, C, D; };

// Diffusion, advection and power-law coefficients shared by the three
// mixing-length solvers.  F* are the face fluxes of the component.
__device__ __forceinline__ void ml_coeffs(const DomG &d, const ColInfo &q, int k, float VIS, float FE, float FW,
                                          float FS, float FN, float FT, float FB, float &AW1, float &AS1,
                                          float &AE1, float &AN1, float &BIM, float &CIM, float &AIM) {
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float mv = vmaxf(VIS, d.vishmin);
    float DE = mv * dykdzk / d.dxk, DW = DE;
    float DS = mv * dxkdzk / d.dyk, DN = DS;
    float DT = mv * d.area / dz;
    float DB = (k > q.KK + 1) ? DT : 0.0f;
    if (q.as) DS = 0; if (q.an) DN = 0; if (q.aw) DW = 0; if (q.ae) DE = 0;
    DE = vmaxf(DE, 0.0001f); DB = vmaxf(DB, 0.0001f); DW = vmaxf(DW, 0.0001f);
    DS = vmaxf(DS, 0.0001f); DN = vmaxf(DN, 0.0001f); DT = vmaxf(DT, 0.0001f);
    float PE = fabsf(FE / DE), PB = fabsf(FB / DB), PW = fabsf(FW / DW);
    float PS = fabsf(FS / DS), PN = fabsf(FN / DN), PT = fabsf(FT / DT);
    const bool v = q.v512();
    BIM = plaw_coef(v, DT, PT, vmaxf(-FT, 0.0f));
    CIM = plaw_coef(v, DB, PB, vmaxf(FB, 0.0f));
    AE1 = plaw_coef(v, DE, PE, vmaxf(-FE, 0.0f));
    AW1 = plaw_coef(v, DW, PW, vmaxf(FW, 0.0f));
    AS1 = plaw_coef(v, DS, PS, vmaxf(FS, 0.0f));
    AN1 = plaw_coef(v, DN, PN, vmaxf(-FN, 0.0f));
    AIM = BIM + CIM + AW1 + AS1 + AE1 + AN1 + d.ap0[k];
}

// wall function at k = KKART+1 for U and V (U-prognostic-microscale_1.cs:419-450)
__device__ __forceinline__ float ml_wall_uv(const DomG &d, const ColInfo &q, int k, float vel, const gf32 *UKS,
                                            const gf32 *UKS_W, const gf32 *VKS, const gf32 *VKS_W) {
    float in = 0.5f * (UKS_W[k] + UKS[k]);
    float in2 = 0.5f * (VKS_W[k] + VKS[k]);
    float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.1f);
    float us;
    if (q.cutk < 1) {
        us = q.ht * wh;
        if (q.z0s >= d.dzk[k] * 0.1f) {
            int ind = k + 1;
            float a = 0.5f * (UKS_W[ind] + UKS[ind]);
            float b = 0.5f * (VKS_W[ind] + VKS[ind]);
            us = q.ht * sqrtf(a * a + b * b);
        }
    } else {
        us = q.ho * wh;
    }
    return vel / wh * (us * us) * d.area;
}

// Pieces of the mixing-length source term D of one cell.  Everything here is
// fixed during a sweep (it reads only arrays the sweep does not write, plus the
// cell's own column, which is updated only when its own turn comes), except
// the four neighbour values of the swept component, which enter as
//   D = AW1*X_W + AS1*X_S + AE1*X_E + AN1*X_N + e + f + g  [- w]  [+ cross]
// summed left to right exactly as the reference does.  The 512-bit solvers
// form the neighbour part as FMA(AW1,X_W,AS1*X_S) + FMA(AE1,X_E,AN1*X_N)
// (not V without vegetation), and U without vegetation folds g into
// f = FMA(DDPX, DYKDZK, g) (U-prognostic-microscale_1_Vec512.cs:404-421).
struct MlPieces {
    float AW1, AS1, AE1, AN1, A, B, C;
    float e, f, g, w;          // g: Coriolis(+vegetation) term of U/V; vegetation drag (subtracted) of W
    float c0, X1, X2, X3, X4;  // cross terms: c0 = VIS/DXK, X* the neighbour-free gradients (W: X1 = whole term)
};

__device__ __forceinline__ bool ml_cross_on(const ColInfo &q, int k) {
    return block_base(k, q.KSTART, q.VI + 1, q.W) > q.KK + 1;
}

// face fluxes of the component's control volume at level k (U-prognostic-
// microscale_1.cs:313-330, V-...:317-331, W-...:286-300), in the reference's order
template <int COMP>
__device__ __forceinline__ void ml_fluxes(const DomG &d, const ColInfo &q, int k, float &FE, float &FW, float &FS,
                                          float &FN, float &FT, float &FB) {
    const int i = q.i, j = q.j;
    const float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    if (COMP == 0) {
        const gf32 *UKS_W = d.uks + c3(d, i - 1, j);
        const gf32 *VKS_W = d.vks + c3(d, i - 1, j), *VKS_WS = d.vks + c3(d, i - 1, j - 1);
        const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *VKS_WN = d.vks + c3(d, i - 1, j + 1);
        const gf32 *VKS_N = d.vks + c3(d, i, j + 1), *WKS_W = d.wks + c3(d, i - 1, j);
        FE = UKS[k] * dykdzk;
        FW = UKS_W[k] * dykdzk;
        FS = 0.25f * (VKS_W[k] + VKS[k] + VKS_WS[k] + VKS_S[k]) * dxkdzk;
        FN = 0.25f * (VKS_W[k] + VKS[k] + VKS_WN[k] + VKS_N[k]) * dxkdzk;
        FT = 0.25f * (WKS_W[k] + WKS[k] + WKS_W[k + 1] + WKS[k + 1]) * d.area;
        FB = (k > q.KK + 1) ? 0.25f * (WKS_W[k] + WKS[k] + WKS_W[k - 1] + WKS[k - 1]) * d.area : 0.0f;
    } else if (COMP == 1) {
        const gf32 *UKS_W = d.uks + c3(d, i - 1, j), *UKS_E = d.uks + c3(d, i + 1, j);
        const gf32 *UKS_S = d.uks + c3(d, i, j - 1), *UKS_ES = d.uks + c3(d, i + 1, j - 1);
        const gf32 *UKS_WS = d.uks + c3(d, i - 1, j - 1);
        const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *WKS_S = d.wks + c3(d, i, j - 1);
        FE = 0.25f * (UKS[k] + UKS_E[k] + UKS_S[k] + UKS_ES[k]) * dykdzk;
        FW = 0.25f * (UKS[k] + UKS_W[k] + UKS_S[k] + UKS_WS[k]) * dykdzk;
        FS = VKS_S[k] * dxkdzk;
        FN = VKS[k] * dxkdzk;
        FT = 0.25f * (WKS_S[k] + WKS[k] + WKS_S[k + 1] + WKS[k + 1]) * d.area;
        FB = (k > q.KK + 1) ? 0.25f * (WKS_S[k] + WKS[k] + WKS_S[k - 1] + WKS[k - 1]) * d.area : 0.0f;
    } else {
        const gf32 *UKS_W = d.uks + c3(d, i - 1, j), *UKS_E = d.uks + c3(d, i + 1, j);
        const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *VKS_N = d.vks + c3(d, i, j + 1);
        FE = 0.25f * (UKS[k] + UKS_E[k] + UKS[k - 1] + UKS_E[k - 1]) * dykdzk;
        FW = 0.25f * (UKS[k] + UKS_W[k] + UKS[k - 1] + UKS_W[k - 1]) * dykdzk;
        FS = 0.25f * (VKS[k] + VKS_S[k] + VKS[k - 1] + VKS_S[k - 1]) * dxkdzk;
        FN = 0.25f * (VKS[k] + VKS_N[k] + VKS[k - 1] + VKS_N[k - 1]) * dxkdzk;
        FT = WKS[k] * d.area;
        FB = (k > q.KK + 1) ? WKS[k - 1] * d.area : 0.0f;
    }
}

__device__ MlPieces u1_pieces(const DomG &d, const ColInfo &q, int k) {
    int i = q.i, j = q.j;
    const gf32 *UK = d.uk + c3(d, i, j), *VK = d.vk + c3(d, i, j);
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    const gf32 *UKS_W = d.uks + c3(d, i - 1, j);
    const gf32 *VKS_W = d.vks + c3(d, i - 1, j), *VKS_WS = d.vks + c3(d, i - 1, j - 1);
    const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *VKS_WN = d.vks + c3(d, i - 1, j + 1);
    const gf32 *VKS_N = d.vks + c3(d, i, j + 1), *VKS_EN = d.vks + c3(d, i + 1, j + 1);
    const gf32 *VKS_ES = d.vks + c3(d, i + 1, j - 1);
    const gf32 *WKS_W = d.wks + c3(d, i - 1, j), *WK_E = d.wk + c3(d, i + 1, j);
    const gf32 *DPMNEW = d.dpmnew + c3(d, i, j), *DPMNEW_W = d.dpmnew + c3(d, i - 1, j);
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float VIS = ml_visc(d, q, k, UK, VK);
    float FE, FW, FS, FN, FT, FB;
    ml_fluxes<0>(d, q, k, FE, FW, FS, FN, FT, FB);
    MlPieces o;
    ml_coeffs(d, q, k, VIS, FE, FW, FS, FN, FT, FB, o.AW1, o.AS1, o.AE1, o.AN1, o.B, o.C, o.A);
    float ap0 = d.ap0[k];
    float u = UK[k];
    o.e = ap0 * 0.5f * (UKS_W[k] + UKS[k]);
    o.f = (DPMNEW_W[k] - DPMNEW[k]) * dykdzk;
    if (q.vegp) {
        float in2 = 0.5f * (VKS_W[k] + VKS[k]);
        float in = 0.5f * (UKS_W[k] + UKS[k]);
        float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.01f);
        float veg = d.veg[c3(d, i, j) + k - 1];
        o.g = (d.cor * (d.ug - u) - veg * u * wh) * d.area * dz;
    } else {
        o.g = d.cor * (d.ug - u) * d.area * dz;
        if (q.v512()) o.f = fmaf(DPMNEW_W[k] - DPMNEW[k], dykdzk, o.g);
    }
    o.w = (k == q.KK + 1) ? ml_wall_uv(d, q, k, u, UKS, UKS_W, VKS, VKS_W) : 0.0f;
    o.c0 = VIS / d.dxk;
    o.X1 = (0.5f * (VKS_EN[k] + VKS_N[k]) - 0.5f * (VKS_N[k] + VKS_WN[k])) * dxkdzk;        // DVDXN
    o.X2 = (0.5f * (VKS_ES[k] + VKS_S[k]) - 0.5f * (VKS_S[k] + VKS_WS[k])) * dxkdzk;        // DVDXS
    o.X3 = (0.5f * (WK_E[k] + WKS[k]) - 0.5f * (WKS[k] + WKS_W[k])) * d.area;                // DWDXT
    o.X4 = (0.5f * (WK_E[k - 1] + WKS[k - 1]) - 0.5f * (WKS[k - 1] + WKS_W[k - 1])) * d.area; // DWDXB
    return o;
}

__device__ MlPieces v1_pieces(const DomG &d, const ColInfo &q, int k) {
    int i = q.i, j = q.j;
    const gf32 *UK = d.uk + c3(d, i, j), *VK = d.vk + c3(d, i, j);
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    const gf32 *UKS_W = d.uks + c3(d, i - 1, j), *UKS_E = d.uks + c3(d, i + 1, j);
    const gf32 *UKS_S = d.uks + c3(d, i, j - 1), *UKS_ES = d.uks + c3(d, i + 1, j - 1);
    const gf32 *UKS_WS = d.uks + c3(d, i - 1, j - 1), *UKS_EN = d.uks + c3(d, i + 1, j + 1);
    const gf32 *UKS_WN = d.uks + c3(d, i - 1, j + 1);
    const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *VKS_W = d.vks + c3(d, i - 1, j);
    const gf32 *WKS_S = d.wks + c3(d, i, j - 1), *WK_N = d.wk + c3(d, i, j + 1);
    const gf32 *DPMNEW = d.dpmnew + c3(d, i, j), *DPMNEW_S = d.dpmnew + c3(d, i, j - 1);
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float VIS = ml_visc(d, q, k, UK, VK);
    float FE, FW, FS, FN, FT, FB;
    ml_fluxes<1>(d, q, k, FE, FW, FS, FN, FT, FB);
    MlPieces o;
    ml_coeffs(d, q, k, VIS, FE, FW, FS, FN, FT, FB, o.AW1, o.AS1, o.AE1, o.AN1, o.B, o.C, o.A);
    float ap0 = d.ap0[k];
    float v = VK[k];
    o.e = ap0 * 0.5f * (VKS_S[k] + VKS[k]);
    o.f = (DPMNEW_S[k] - DPMNEW[k]) * dxkdzk;
    if (q.vegp) {
        float in2 = 0.5f * (VKS_W[k] + VKS[k]);
        float in = 0.5f * (UKS_W[k] + UKS[k]);
        float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.01f);
        float veg = d.veg[c3(d, i, j) + k - 1];
        o.g = (d.cor * (d.vg - v) - veg * v * wh) * d.area * dz;
    } else {
        o.g = d.cor * (d.vg - v) * d.area * dz;
    }
    o.w = (k == q.KK + 1) ? ml_wall_uv(d, q, k, v, UKS, UKS_W, VKS, VKS_W) : 0.0f;
    o.c0 = VIS / d.dxk;
    o.X1 = (0.5f * (UKS_EN[k] + UKS_E[k]) - 0.5f * (UKS_E[k] + UKS_ES[k])) * dxkdzk;        // DUDYE
    o.X2 = (0.5f * (UKS_WN[k] + UKS_W[k]) - 0.5f * (UKS_W[k] + UKS_WS[k])) * dxkdzk;        // DUDYW
    o.X3 = (0.5f * (WK_N[k] + WKS[k]) - 0.5f * (WKS[k] + WKS_S[k])) * d.area;                // DWDYT
    // the reference takes WKS of the southern column at k, not k-1, here
    o.X4 = (0.5f * (WK_N[k - 1] + WKS[k - 1]) - 0.5f * (WKS[k - 1] + WKS_S[k])) * d.area;    // DWDYB
    return o;
}

__device__ MlPieces w1_pieces(const DomG &d, const ColInfo &q, int k) {
    int i = q.i, j = q.j;
    const gf32 *UK = d.uk + c3(d, i, j), *VK = d.vk + c3(d, i, j), *WK = d.wk + c3(d, i, j);
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    const gf32 *UKS_W = d.uks + c3(d, i - 1, j), *UKS_E = d.uks + c3(d, i + 1, j);
    const gf32 *VKS_S = d.vks + c3(d, i, j - 1), *VKS_N = d.vks + c3(d, i, j + 1);
    const gf32 *DPMNEW = d.dpmnew + c3(d, i, j);
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float VIS = ml_visc(d, q, k, UK, VK);
    float FE, FW, FS, FN, FT, FB;
    ml_fluxes<2>(d, q, k, FE, FW, FS, FN, FT, FB);
    MlPieces o;
    ml_coeffs(d, q, k, VIS, FE, FW, FS, FN, FT, FB, o.AW1, o.AS1, o.AE1, o.AN1, o.B, o.C, o.A);
    float ap0 = d.ap0[k];
    float w = WK[k];
    o.e = ap0 * 0.5f * (WKS[k - 1] + WKS[k]);
    o.f = (DPMNEW[k - 1] - DPMNEW[k]) * d.area;
    if (q.vegp) {
        float in2 = 0.5f * (VKS_S[k] + VKS[k]);
        float in = 0.5f * (UKS_W[k] + UKS[k]);
        float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.01f);
        float veg = d.veg[c3(d, i, j) + k - 1];
        o.g = veg * w * wh * d.area * dz;
    } else {
        o.g = 0.0f;
    }
    o.w = 0.0f;
    float DUDZE = (0.5f * (UKS[k + 1] + UKS[k]) - 0.5f * (UKS[k] + UKS[k - 1])) * dykdzk;
    float DUDZW = (0.5f * (UKS_W[k + 1] + UKS_W[k]) - 0.5f * (UKS_W[k] + UKS_W[k - 1])) * dykdzk;
    float DVDZN = (0.5f * (VKS[k + 1] + VKS[k]) - 0.5f * (VKS[k] + VKS[k - 1])) * dxkdzk;
    float DVDZS = (0.5f * (VKS_S[k + 1] + VKS_S[k]) - 0.5f * (VKS_S[k] + VKS_S[k - 1])) * dxkdzk;
    float DWDZT = (WK[k + 1] - w) * d.area;
    float DWDZB = (w - WK[k - 1]) * d.area;
    o.c0 = 0.0f;
    o.X1 = VIS / dz * (DUDZE - DUDZW + DVDZN - DVDZS + DWDZT - DWDZB);
    o.X2 = o.X3 = o.X4 = 0.0f;
    return o;
}

// D of one cell from its pieces and the four neighbour values (and the cell's
// own old value x), in the reference's order of operations.
template <int COMP>
__device__ __forceinline__ float ml_source(const DomG &d, const ColInfo &q, int k, float dz, const MlPieces &o, float xw,
                                           float xs, float xe, float xn, float x) {
    float D;
    if (q.v512() && (COMP != 1 || q.vegp))
        D = fmaf(o.AW1, xw, o.AS1 * xs) + fmaf(o.AE1, xe, o.AN1 * xn);
    else
        D = o.AW1 * xw + o.AS1 * xs + o.AE1 * xe + o.AN1 * xn;
    D = D + o.e + o.f;
    if (COMP != 2) {
        if (COMP != 0 || !q.v512() || q.vegp) D = D + o.g;
        if (k == q.KK + 1) D -= o.w;
        if (ml_cross_on(q, k)) {
            if (COMP == 0) {
                float dykdzk = d.dyk * dz;
                float DUDXE = (xe - x) * dykdzk;
                float DUDXW = (x - xw) * dykdzk;
                D += o.c0 * (DUDXE - DUDXW + o.X1 - o.X2 + o.X3 - o.X4);
            } else {
                float dxkdzk = d.dxk * dz;
                float DVDYN = (xn - x) * dxkdzk;
                float DVDYS = (x - xs) * dxkdzk;
                D += o.c0 * (o.X1 - o.X2 + DVDYN - DVDYS + o.X3 - o.X4);
            }
        }
    } else {
        if (q.vegp) D = D - o.g;
        if (ml_cross_on(q, k)) D += o.X1;
    }
    return D;
}

template <int COMP>
__device__ __forceinline__ MlPieces ml_pieces(const DomG &d, const ColInfo &q, int k) {
    if (COMP == 0) return u1_pieces(d, q, k);
    if (COMP == 1) return v1_pieces(d, q, k);
    return w1_pieces(d, q, k);
}

// neighbour values X_W, X_S, X_E, X_N of the swept component at level k
template <int COMP>
__device__ __forceinline__ void ml_neighbours(const DomG &d, int i, int j, int k, float &xw, float &xs, float &xe,
                                              float &xn, float &x) {
    const gf32 *X = COMP == 0 ? d.uk : COMP == 1 ? d.vk : d.wk;
    xw = X[c3(d, i - 1, j) + k];
    xe = X[c3(d, i + 1, j) + k];
    xs = X[c3(d, i, j - 1) + k];
    xn = X[c3(d, i, j + 1) + k];
    x = X[c3(d, i, j) + k];
}

template <int COMP>
__device__ Coef ml_cell(const DomG &d, const ColInfo &q, int k) {
    MlPieces o = ml_pieces<COMP>(d, q, k);
    float xw, xs, xe, xn, x;
    ml_neighbours<COMP>(d, q.i, q.j, k, xw, xs, xe, xn, x);
    return Coef{o.A, o.B, o.C, ml_source<COMP>(d, q, k, d.dzk[k], o, xw, xs, xe, xn, x)};
}
__device__ Coef u1_cell(const DomG &d, const ColInfo &q, int k) { return ml_cell<0>(d, q, k); }
__device__ Coef v1_cell(const DomG &d, const ColInfo &q, int k) { return ml_cell<1>(d, q, k); }
__device__ Coef w1_cell(const DomG &d, const ColInfo &q, int k) { return ml_cell<2>(d, q, k); }

// ------------------------------------------------------------------------
// k-eps (model 2) and no-diffusion (model 0) momentum, _2.cs / _0.cs
// ------------------------------------------------------------------------
__device__ __forceinline__ float plaw_d(float D, float P) {   // D*FloatMax(0,(float)Pow5(1-0.1*P))
    double x = 1.0 - 0.1 * (double)P;
    return D * vmaxf(0.0f, (float)(x * x * x * x * x));
}

// wall function of the scalar U/V solvers (U-prognostic-microscale_2.cs:188-212)
__device__ __forceinline__ float ke_wall_uv(const DomG &d, const ColInfo &q, int k, float vel, const gf32 *UKSim,
                                            const gf32 *UKS, const gf32 *VKSim, const gf32 *VKS) {
    double a = 0.5 * (double)(UKSim[k] + UKS[k]);
    double b = 0.5 * (double)(VKSim[k] + VKS[k]);
    float wh = vmaxf((float)sqrt(a * a + b * b), 0.01f);
    float us;
    if (q.cutk < 1) {
        us = q.ht * wh;
        if ((double)q.z0s >= (double)d.dzk[k] * 0.1) {
            double a1 = 0.5 * (double)(UKSim[k + 1] + UKS[k + 1]);
            double b1 = 0.5 * (double)(VKSim[k + 1] + VKS[k + 1]);
            us = q.ht * (float)sqrt(a1 * a1 + b1 * b1);
        }
    } else {
        us = q.ho * wh;
    }
    return vel / wh * (us * us) * d.area;
}

// Everything of one k-eps (DIFF) or no-diffusion cell of U/V but the four
// neighbour values of the swept component (U-prognostic-microscale_2.cs:100-260,
// V-prognostic-microscale_2.cs, _0.cs): the coefficients, e = the old-velocity
// sum of the transient term (its double product with AP0 is formed with the
// neighbour part), f = the pressure term, g = the Coriolis term, w = the wall
// term at KKART+1, c0 = VIS/DXK and X1..X4 the neighbour-free gradients of the
// cross-diffusion term above KKART+1.
template <bool IS_V, bool DIFF>
__device__ MlPieces ke_uv_pieces(const DomG &d, const ColInfo &q, int k) {
    int i = q.i, j = q.j;
    const gf32 *X = (IS_V ? d.vk : d.uk) + c3(d, i, j);
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    const gf32 *UKSim = d.uks + c3(d, i - 1, j), *VKSim = d.vks + c3(d, i - 1, j);
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float VIS = 0, DE = 0, DW = 0, DS = 0, DN = 0, DT = 0, DB = 0;
    if (DIFF) {
        float zs = d.hok[k] - d.hok[q.KK] - dz * 0.5f;
        VIS = sqrtf(d.turb[c3(d, i, j) + k]) * zs * 0.09f;
        DE = vmaxf(VIS, d.vishmin) * dykdzk / d.dxk; DW = DE;
        DS = vmaxf(VIS, d.vishmin) * dxkdzk / d.dyk; DN = DS;
        DT = vmaxf(VIS, d.vishmin) * d.area / dz;
        if (k > q.KK + 1) DB = DT;
        if (q.as) DS = 0; if (q.an) DN = 0; if (q.aw) DW = 0; if (q.ae) DE = 0;
    }
    float FE, FW, FS, FN, FT, FB = 0;
    if (!IS_V) {
        const gf32 *VKSimjm = d.vks + c3(d, i - 1, j - 1), *VKSjm = d.vks + c3(d, i, j - 1);
        const gf32 *VKSimjp = d.vks + c3(d, i - 1, j + 1), *VKSjp = d.vks + c3(d, i, j + 1);
        const gf32 *WKSim = d.wks + c3(d, i - 1, j);
        FE = UKS[k] * dykdzk;
        FW = UKSim[k] * dykdzk;
        FS = 0.25f * (VKSim[k] + VKS[k] + VKSimjm[k] + VKSjm[k]) * dxkdzk;
        FN = 0.25f * (VKSim[k] + VKS[k] + VKSimjp[k] + VKSjp[k]) * dxkdzk;
        FT = 0.25f * (WKSim[k] + WKS[k] + WKSim[k + 1] + WKS[k + 1]) * d.area;
        if (k > q.KK + 1) FB = 0.25f * (WKSim[k] + WKS[k] + WKSim[k - 1] + WKS[k - 1]) * d.area;
    } else {
        const gf32 *UKSip = d.uks + c3(d, i + 1, j), *UKSjm = d.uks + c3(d, i, j - 1);
        const gf32 *UKSipjm = d.uks + c3(d, i + 1, j - 1), *UKSimjm = d.uks + c3(d, i - 1, j - 1);
        const gf32 *VKSjm = d.vks + c3(d, i, j - 1), *WKSjm = d.wks + c3(d, i, j - 1);
        FE = 0.25f * (UKS[k] + UKSip[k] + UKSjm[k] + UKSipjm[k]) * dykdzk;
        FW = 0.25f * (UKS[k] + UKSim[k] + UKSjm[k] + UKSimjm[k]) * dykdzk;
        FS = VKSjm[k] * dxkdzk;
        FN = VKS[k] * dxkdzk;
        FT = 0.25f * (WKSjm[k] + WKS[k] + WKSjm[k + 1] + WKS[k + 1]) * d.area;
        if (k > q.KK + 1) FB = 0.25f * (WKSjm[k] + WKS[k] + WKSjm[k - 1] + WKS[k - 1]) * d.area;
    }
    MlPieces o;
    float BIM, CIM, AE1, AW1, AS1, AN1;
    if (DIFF) {
        DE = vmaxf(DE, 0.0001f); DB = vmaxf(DB, 0.0001f); DW = vmaxf(DW, 0.0001f);
        DS = vmaxf(DS, 0.0001f); DN = vmaxf(DN, 0.0001f); DT = vmaxf(DT, 0.0001f);
        float PE = fabsf(FE / DE), PB = fabsf(FB / DB), PW = fabsf(FW / DW);
        float PS = fabsf(FS / DS), PN = fabsf(FN / DN), PT = fabsf(FT / DT);
        BIM = plaw_d(DT, PT) + vmaxf(-FT, 0.0f);
        CIM = plaw_d(DB, PB) + vmaxf(FB, 0.0f);
        AE1 = plaw_d(DE, PE) + vmaxf(-FE, 0.0f);
        AW1 = plaw_d(DW, PW) + vmaxf(FW, 0.0f);
        AS1 = plaw_d(DS, PS) + vmaxf(FS, 0.0f);
        AN1 = plaw_d(DN, PN) + vmaxf(-FN, 0.0f);
    } else {
        BIM = vmaxf(-FT, 0.0f); CIM = vmaxf(FB, 0.0f); AE1 = vmaxf(-FE, 0.0f);
        AW1 = vmaxf(FW, 0.0f); AS1 = vmaxf(FS, 0.0f); AN1 = vmaxf(-FN, 0.0f);
    }
    float ap0 = d.ap0[k];
    o.A = BIM + CIM + AW1 + AS1 + AE1 + AN1 + ap0;
    o.B = BIM; o.C = CIM; o.AW1 = AW1; o.AS1 = AS1; o.AE1 = AE1; o.AN1 = AN1;
    const gf32 *DPMNEW = d.dpmnew + c3(d, i, j);
    const gf32 *DPMNEWm = d.dpmnew + (IS_V ? c3(d, i, j - 1) : c3(d, i - 1, j));
    float ddp = DPMNEWm[k] - DPMNEW[k];
    float x = X[k];
    o.e = IS_V ? (d.vks[c3(d, i, j - 1) + k] + VKS[k]) : (UKSim[k] + UKS[k]);
    o.f = ddp * (IS_V ? dxkdzk : dykdzk);
    o.g = d.cor * ((IS_V ? d.vg : d.ug) - x) * d.area * dz;
    o.w = (k == q.KK + 1) ? ke_wall_uv(d, q, k, x, UKSim, UKS, VKSim, VKS) : 0.0f;
    o.c0 = o.X1 = o.X2 = o.X3 = o.X4 = 0.0f;
    if (DIFF && k > q.KK + 1) {
        o.c0 = VIS / d.dxk;
        if (!IS_V) {
            const gf32 *VKSipjp = d.vks + c3(d, i + 1, j + 1), *VKSjp = d.vks + c3(d, i, j + 1);
            const gf32 *VKSimjp = d.vks + c3(d, i - 1, j + 1), *VKSipjm = d.vks + c3(d, i + 1, j - 1);
            const gf32 *VKSjm = d.vks + c3(d, i, j - 1), *VKSimjm = d.vks + c3(d, i - 1, j - 1);
            const gf32 *WKip = d.wk + c3(d, i + 1, j), *WKSim = d.wks + c3(d, i - 1, j);
            o.X1 = (0.5f * (VKSipjp[k] + VKSjp[k]) - 0.5f * (VKSjp[k] + VKSimjp[k])) * dxkdzk;          // DVDXN
            o.X2 = (0.5f * (VKSipjm[k] + VKSjm[k]) - 0.5f * (VKSjm[k] + VKSimjm[k])) * dxkdzk;          // DVDXS
            o.X3 = (0.5f * (WKip[k] + WKS[k]) - 0.5f * (WKS[k] + WKSim[k])) * d.area;                   // DWDXT
            o.X4 = (0.5f * (WKip[k - 1] + WKS[k - 1]) - 0.5f * (WKS[k - 1] + WKSim[k - 1])) * d.area;   // DWDXB
        } else {
            const gf32 *UKSipjp = d.uks + c3(d, i + 1, j + 1), *UKSip = d.uks + c3(d, i + 1, j);
            const gf32 *UKSipjm = d.uks + c3(d, i + 1, j - 1), *UKSimjp = d.uks + c3(d, i - 1, j + 1);
            const gf32 *UKSimjm = d.uks + c3(d, i - 1, j - 1);
            const gf32 *WKjp = d.wk + c3(d, i, j + 1), *WKSjm = d.wks + c3(d, i, j - 1);
            o.X1 = (0.5f * (UKSipjp[k] + UKSip[k]) - 0.5f * (UKSip[k] + UKSipjm[k])) * dxkdzk;          // DUDYE
            o.X2 = (0.5f * (UKSimjp[k] + UKSim[k]) - 0.5f * (UKSim[k] + UKSimjm[k])) * dxkdzk;          // DUDYW
            o.X3 = (0.5f * (WKjp[k] + WKS[k]) - 0.5f * (WKS[k] + WKSjm[k])) * d.area;                   // DWDYT
            o.X4 = (0.5f * (WKjp[k - 1] + WKS[k - 1]) - 0.5f * (WKS[k - 1] + WKSjm[k - 1])) * d.area;   // DWDYB
        }
    }
    return o;
}

// W of the k-eps / no-diffusion solvers (W-prognostic-microscale_2.cs, _0.cs):
// e = the old-velocity sum of the transient term, f = the pressure term, X1 =
// the whole cross-diffusion term above KKART+1 (it reads no neighbour of W).
template <bool DIFF>
__device__ MlPieces ke_w_pieces(const DomG &d, const ColInfo &q, int k) {
    int i = q.i, j = q.j;
    const gf32 *WK = d.wk + c3(d, i, j);
    const gf32 *UKS = d.uks + c3(d, i, j), *VKS = d.vks + c3(d, i, j), *WKS = d.wks + c3(d, i, j);
    const gf32 *UKSim = d.uks + c3(d, i - 1, j), *UKSip = d.uks + c3(d, i + 1, j);
    const gf32 *VKSjm = d.vks + c3(d, i, j - 1), *VKSjp = d.vks + c3(d, i, j + 1);
    const gf32 *DPMNEW = d.dpmnew + c3(d, i, j);
    float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    float uks = UKS[k], uks_m = UKS[k - 1], vks = VKS[k], vks_m = VKS[k - 1];
    float VIS = 0, DE = 0, DW = 0, DS = 0, DN = 0, DT = 0, DB = 0;
    if (DIFF) {
        float zs = d.hok[k] - d.hok[q.KK] - dz * 0.5f;
        VIS = sqrtf(d.turb[c3(d, i, j) + k]) * zs * 0.09f;
        DE = vmaxf(VIS, d.vishmin) * dykdzk / d.dxk; DW = DE;
        DS = vmaxf(VIS, d.vishmin) * dxkdzk / d.dyk; DN = DS;
        DT = vmaxf(VIS, d.vishmin) * d.area / dz;
        if (k > q.KK + 1) DB = DT;
        if (q.as) DS = 0; if (q.an) DN = 0; if (q.aw) DW = 0; if (q.ae) DE = 0;
    }
    float FE = 0.25f * (uks + UKSip[k] + uks_m + UKSip[k - 1]) * dykdzk;
    float FW = 0.25f * (uks + UKSim[k] + uks_m + UKSim[k - 1]) * dykdzk;
    float FS = 0.25f * (vks + VKSjm[k] + vks_m + VKSjm[k - 1]) * dxkdzk;
    float FN = 0.25f * (vks + VKSjp[k] + vks_m + VKSjp[k - 1]) * dxkdzk;
    float FT = WKS[k] * d.area;
    float FB = (k > q.KK + 1) ? WKS[k - 1] * d.area : 0.0f;
    float BIM, CIM, AE1, AW1, AS1, AN1;
    if (DIFF) {
        DE = vmaxf(DE, 0.0001f); DB = vmaxf(DB, 0.0001f); DW = vmaxf(DW, 0.0001f);
        DS = vmaxf(DS, 0.0001f); DN = vmaxf(DN, 0.0001f); DT = vmaxf(DT, 0.0001f);
        float PE = fabsf(FE / DE), PB = fabsf(FB / DB), PW = fabsf(FW / DW);
        float PS = fabsf(FS / DS), PN = fabsf(FN / DN), PT = fabsf(FT / DT);
        BIM = plaw_d(DT, PT) + vmaxf(-FT, 0.0f);
        CIM = plaw_d(DB, PB) + vmaxf(FB, 0.0f);
        AE1 = plaw_d(DE, PE) + vmaxf(-FE, 0.0f);
        AW1 = plaw_d(DW, PW) + vmaxf(FW, 0.0f);
        AS1 = plaw_d(DS, PS) + vmaxf(FS, 0.0f);
        AN1 = plaw_d(DN, PN) + vmaxf(-FN, 0.0f);
    } else {
        BIM = vmaxf(-FT, 0.0f); CIM = vmaxf(FB, 0.0f); AE1 = vmaxf(-FE, 0.0f);
        AW1 = vmaxf(FW, 0.0f); AS1 = vmaxf(FS, 0.0f); AN1 = vmaxf(-FN, 0.0f);
    }
    MlPieces o;
    float ap0 = d.ap0[k];
    o.A = BIM + CIM + AW1 + AS1 + AE1 + AN1 + ap0;
    o.B = BIM; o.C = CIM; o.AW1 = AW1; o.AS1 = AS1; o.AE1 = AE1; o.AN1 = AN1;
    o.e = WKS[k - 1] + WKS[k];
    o.f = (DPMNEW[k - 1] - DPMNEW[k]) * d.area;
    o.g = o.w = o.c0 = o.X1 = o.X2 = o.X3 = o.X4 = 0.0f;
    if (DIFF && k > q.KK + 1) {
        float DUDZE = (0.5f * (UKS[k + 1] + uks) - 0.5f * (uks + uks_m)) * dykdzk;
        float DUDZW = (0.5f * (UKSim[k + 1] + UKSim[k]) - 0.5f * (UKSim[k] + UKSim[k - 1])) * dykdzk;
        float DVDZN = (0.5f * (VKS[k + 1] + vks) - 0.5f * (vks + vks_m)) * dxkdzk;
        float DVDZS = (0.5f * (VKSjm[k + 1] + VKSjm[k]) - 0.5f * (VKSjm[k] + VKSjm[k - 1])) * dxkdzk;
        float DWDZT = (WK[k + 1] - WK[k]) * d.area;
        float DWDZB = (WK[k] - WK[k - 1]) * d.area;
        o.X1 = VIS / dz * (DUDZE - DUDZW + DVDZN - DVDZS + DWDZT - DWDZB);
    }
    return o;
}

// D of a k-eps / no-diffusion cell from its pieces, the four neighbour values
// and the cell's own old value x: the neighbour sum in float, then the
// transient, pressure and Coriolis terms added in double in the reference's
// order, rounded to float; the wall term (U, V at KKART+1) and the
// cross-diffusion term follow in float.
template <int COMP, bool DIFF>
__device__ __forceinline__ float ke_source(const DomG &d, const ColInfo &q, int k, float dz, float ap0, const MlPieces &o,
                                           float xw, float xs, float xe, float xn, float x) {
    float partial = o.AW1 * xw + o.AS1 * xs + o.AE1 * xe + o.AN1 * xn;
    double t5 = (double)ap0 * 0.5 * (double)o.e;
    if (COMP == 2) {
        float D = (float)((double)partial + t5 + (double)o.f);
        if (DIFF && k > q.KK + 1) D += o.X1;
        return D;
    }
    float D = (float)((double)partial + t5 + (double)o.f + (double)o.g);
    if (k == q.KK + 1) D -= o.w;
    if (DIFF && k > q.KK + 1) {
        if (COMP == 0) {
            float dykdzk = d.dyk * dz;
            float DUDXE = (xe - x) * dykdzk;
            float DUDXW = (x - xw) * dykdzk;
            D += o.c0 * (DUDXE - DUDXW + o.X1 - o.X2 + o.X3 - o.X4);
        } else {
            float dxkdzk = d.dxk * dz;
            float DVDYN = (xn - x) * dxkdzk;
            float DVDYS = (x - xs) * dxkdzk;
            D += o.c0 * (o.X1 - o.X2 + DVDYN - DVDYS + o.X3 - o.X4);
        }
    }
    return D;
}

template <int COMP, bool DIFF>
__device__ Coef ke_cell(const DomG &d, const ColInfo &q, int k) {
    MlPieces o = (COMP == 2) ? ke_w_pieces<DIFF>(d, q, k) : ke_uv_pieces<COMP == 1, DIFF>(d, q, k);
    float xw, xs, xe, xn, x;
    ml_neighbours<COMP>(d, q.i, q.j, k, xw, xs, xe, xn, x);
    return Coef{o.A, o.B, o.C, ke_source<COMP, DIFF>(d, q, k, d.dzk[k], d.ap0[k], o, xw, xs, xe, xn, x)};
}

// ------------------------------------------------------------------------
// Momentum column kernel: one wavefront per column of diagonal t.
//   COMP 0:U 1:V 2:W;  KIND 0: mixing length (Vector<float> path, TERMP form)
//   1: k-eps, 2: no diffusion (scalar path, division form)
// ------------------------------------------------------------------------
template <int COMP, int KIND>
__global__ __launch_bounds__(WAVE) void k_momentum(const Dom *__restrict__ ds, int t, int IS, int JS) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice

    extern __shared__ float sm[];
    const int nkp = d.nkp, tid = threadIdx.x;
    // sweep ranges (outer i1, inner j1): U i1 from 3; V j1 from 3
    const int oa = (COMP == 0) ? 3 : 2, ia = (COMP == 1) ? 3 : 2;
    int a, b;
    if (!diag_col(t, oa, d.nii - 1, ia, d.njj - 1, blockIdx.x, a, b)) return;
    int i = (IS == -1) ? d.nii - a + 1 : a;
    int j = (JS == -1) ? d.njj - b + 1 : b;
    if (d.adv[c2(d, i, j)] != 1) return;
    ColInfo q = col_info(d, i, j);
    float *sA = sm, *sB = sA + nkp, *sC = sB + nkp, *sD = sC + nkp, *sX = sD + nkp;
    gf32 *X = (COMP == 0 ? d.uk : COMP == 1 ? d.vk : d.wk) + c3(d, i, j);
    for (int k = q.KSTART + tid; k <= q.VI; k += WAVE) {
        Coef cf;
        if (KIND == 0) cf = (COMP == 0) ? u1_cell(d, q, k) : (COMP == 1) ? v1_cell(d, q, k) : w1_cell(d, q, k);
        else cf = ke_cell<COMP, KIND == 1>(d, q, k);
        sA[k] = cf.A; sB[k] = cf.B; sC[k] = cf.C; sD[k] = cf.D;
    }
    for (int k = q.KSTART + tid; k <= q.VI + 1; k += WAVE) sX[k] = X[k];
    __syncthreads();
    if (tid == 0) {
        const int KKP1 = q.KK + 1;
        float Pp = 0, Qp = 0;
        for (int k = q.KSTART; k <= q.VI; ++k) {
            float A = sA[k], B = sB[k], Cc = sC[k], Dd = sD[k], P, Q;
            if (KIND == 0) {
                if (k > KKP1) { float T = 1 / (A - Cc * Pp); P = B * T; Q = (Dd + Cc * Qp) * T; }
                else { float T = 1 / A; P = B * T; Q = Dd * T; }
            } else {
                if (k > KKP1) { P = B / (A - Cc * Pp); Q = (Dd + Cc * Qp) / (A - Cc * Pp); }
                else { P = B / A; Q = Dd / A; }
            }
            sA[k] = P; sB[k] = Q;
            Pp = P; Qp = Q;
        }
        // relaxed back-substitution; U/V skip levels inside the building or its
        // upstream neighbour, W updates every level (W-prognostic-microscale_1.cs:445-448)
        int KKm = q.KK;
        if (COMP == 0) KKm = max(q.KK, d.kk[c2(d, i - 1, j)]);
        if (COMP == 1) KKm = max(q.KK, d.kk[c2(d, i, j - 1)]);
        float up = sX[q.VI + 1];
        for (int k = q.VI; k >= q.KSTART; --k) {
            float x = sX[k];
            if (COMP == 2 || KKm < k) {
                x = x + d.relax * (sA[k] * up + sB[k] - x);
                sX[k] = x;
            }
            up = x;
        }
    }
    __syncthreads();
    for (int k = q.KSTART + tid; k <= q.VI; k += WAVE) X[k] = sX[k];
}

// ------------------------------------------------------------------------
// TKE / dissipation (k-eps), TKE-prognostic-microscale.cs:25-352
// ------------------------------------------------------------------------
// Per-column pointers and neighbour data of the TKE sweep, and the per-level
// coefficients (TKE-prognostic-microscale.cs:100-337) that the sweep's
// in-place neighbours (TURB, TDISS of the four neighbour columns) do not touch.
struct TkeCol {
    size_t o, c;
    const gf32 *TURB, *TDISS, *UK, *VK, *WK;
    const gf32 *UKip, *UKjp, *UKipjp, *UKjm, *UKipjm, *VKjp, *VKip, *VKipjp, *VKim, *VKimjp, *WKip, *WKim, *WKjp, *WKjm;
    int kkip, kkim, kkjp, kkjm;
    bool cip, cim, cjp, cjm;
};
__device__ __forceinline__ TkeCol tke_col_ptrs(const DomG &d, int i, int j) {
    TkeCol t;
    t.c = c2(d, i, j);
    t.o = c3(d, i, j);
    t.TURB = d.turb + t.o; t.TDISS = d.tdiss + t.o;
    t.UK = d.uk + t.o; t.VK = d.vk + t.o; t.WK = d.wk + t.o;
    t.UKip = d.uk + c3(d, i + 1, j); t.UKjp = d.uk + c3(d, i, j + 1); t.UKipjp = d.uk + c3(d, i + 1, j + 1);
    t.UKjm = d.uk + c3(d, i, j - 1); t.UKipjm = d.uk + c3(d, i + 1, j - 1);
    t.VKjp = d.vk + c3(d, i, j + 1); t.VKip = d.vk + c3(d, i + 1, j); t.VKipjp = d.vk + c3(d, i + 1, j + 1);
    t.VKim = d.vk + c3(d, i - 1, j); t.VKimjp = d.vk + c3(d, i - 1, j + 1);
    t.WKip = d.wk + c3(d, i + 1, j); t.WKim = d.wk + c3(d, i - 1, j);
    t.WKjp = d.wk + c3(d, i, j + 1); t.WKjm = d.wk + c3(d, i, j - 1);
    return t;
}
__device__ __forceinline__ TkeCol tke_col(const DomG &d, int i, int j) {
    TkeCol t = tke_col_ptrs(d, i, j);
    t.kkip = d.kk[c2(d, i + 1, j)]; t.kkim = d.kk[c2(d, i - 1, j)];
    t.kkjp = d.kk[c2(d, i, j + 1)]; t.kkjm = d.kk[c2(d, i, j - 1)];
    t.cip = d.cutk[c2(d, i + 1, j)] > 0; t.cim = d.cutk[c2(d, i - 1, j)] > 0;
    t.cjp = d.cutk[c2(d, i, j + 1)] > 0; t.cjm = d.cutk[c2(d, i, j - 1)] > 0;
    return t;
}

struct TkeCell {
    float A, B1, C1, B2, C2, AW1, AS1, AE1, AN1;
    float w1, PRO, PBO, w2, EPS;      // ap0*TURB, production, buoyancy, ap0*TDISS, eps source
    int wf;                           // wall function replaces the back-substitution
    float wt, we;
};

__device__ __forceinline__ TkeCell tke_cell(const DomG &d, const ColInfo &q, const TkeCol &t, int k) {
    const float DXK = d.dxk, DYK = d.dyk, AREA = d.area, DXK_Rez = 1 / DXK, DYK_Rez = 1 / DYK;
    const float Ceps = 1, Ceps1 = 1.44f, Ceps2 = 1.92f;
    const int KK = q.KK;
    const gf32 *TURB = t.TURB, *TDISS = t.TDISS, *UK = t.UK, *VK = t.VK, *WK = t.WK;
    const gf32 *UKip = t.UKip, *UKjp = t.UKjp, *UKipjp = t.UKipjp, *UKjm = t.UKjm, *UKipjm = t.UKipjm;
    const gf32 *VKjp = t.VKjp, *VKip = t.VKip, *VKipjp = t.VKipjp, *VKim = t.VKim, *VKimjp = t.VKimjp;
    const gf32 *WKip = t.WKip, *WKim = t.WKim, *WKjp = t.WKjp, *WKjm = t.WKjm;
    TkeCell r;
    float dz = d.dzk[k];
    float dxkdzk = DXK * dz, dykdzk = DYK * dz, DZK_Rez = 1 / dz;
    float zs = d.hok[k] - d.hok[KK] - dz * 0.5f;
    float VIS = sqrtf(TURB[k]) * zs * 0.09f;
    VIS = mminf(VIS, 15.0f);
    float DE = mmaxf(VIS, d.vishmin) * dykdzk * DXK_Rez, DW = DE;
    float DS = mmaxf(VIS, d.vishmin) * dxkdzk * DYK_Rez, DN = DS;
    float DT = mmaxf(VIS, d.vishmin) * AREA * DZK_Rez, DB = 0;
    float DTEPS = mmaxf(VIS / Ceps, d.visvmin) * AREA * DZK_Rez, DBEPS = 0;
    if (k > KK + 1) { DB = DT; DBEPS = DTEPS; }
    if (q.as) DS = 0; if (q.an) DN = 0; if (q.aw) DW = 0; if (q.ae) DE = 0;
    float FE = UKip[k] * dykdzk, FW = UK[k] * dykdzk, FS = VK[k] * dxkdzk, FN = VKjp[k] * dxkdzk;
    float FT = WK[k + 1] * AREA, FB = 0;
    if (k > KK + 1) FB = WK[k] * AREA;
    DE = mmaxf(DE, 0.0001f); DB = mmaxf(DB, 0.0001f); DW = mmaxf(DW, 0.0001f);
    DS = mmaxf(DS, 0.0001f); DN = mmaxf(DN, 0.0001f); DT = mmaxf(DT, 0.0001f);
    DBEPS = mmaxf(DBEPS, 0.0001f); DTEPS = mmaxf(DTEPS, 0.0001f);
    float PE = fabsf(FE / DE), PB = fabsf(FB / DB), PW = fabsf(FW / DW);
    float PS = fabsf(FS / DS), PN = fabsf(FN / DN), PT = fabsf(FT / DT);
    float PBEPS = fabsf(FN / DBEPS);   // the reference uses FN here
    float PTEPS = fabsf(FT / DTEPS);
    float x;
    x = 1 - 0.1f * PT; float BIM = DT * mmaxf(0, x * x * x * x * x) + mmaxf(-FT, 0);
    x = 1 - 0.1f * PB; float CIM = DB * mmaxf(0, x * x * x * x * x) + mmaxf(FB, 0);
    x = 1 - 0.1f * PE; float AE1 = DE * mmaxf(0, x * x * x * x * x) + mmaxf(-FE, 0);
    x = 1 - 0.1f * PW; float AW1 = DW * mmaxf(0, x * x * x * x * x) + mmaxf(FW, 0);
    x = 1 - 0.1f * PS; float AS1 = DS * mmaxf(0, x * x * x * x * x) + mmaxf(FS, 0);
    x = 1 - 0.1f * PN; float AN1 = DN * mmaxf(0, x * x * x * x * x) + mmaxf(-FN, 0);
    // the reference weights the eps system with DT/DB, not DTEPS/DBEPS
    x = 1 - 0.1f * PTEPS; float BIMEPS = DT * mmaxf(0, x * x * x * x * x) + mmaxf(-FT, 0);
    x = 1 - 0.1f * PBEPS; float CIMEPS = DB * mmaxf(0, x * x * x * x * x) + mmaxf(FB, 0);
    float ap0 = d.ap0[k];
    float AIM = BIM + CIM + AW1 + AS1 + AE1 + AN1 + ap0;
    float UX1 = UKip[k], UX2 = UK[k];
    float VX1 = 0.5f * (VKip[k] + VKipjp[k]), VX2 = 0.5f * (VKim[k] + VKimjp[k]);
    float WX1 = 0.5f * (WKip[k] + WKip[k + 1]), WX2 = 0.5f * (WKim[k] + WKim[k + 1]);
    float UY1 = 0.5f * (UKjp[k] + UKipjp[k]), UY2 = 0.5f * (UKjm[k] + UKipjm[k]);
    float VY1 = VKjp[k], VY2 = VK[k];
    float WY1 = 0.5f * (WKjp[k] + WKjp[k + 1]), WY2 = 0.5f * (WKjm[k] + WKjm[k + 1]);
    float DUDX = (UX1 - UX2) * DXK_Rez;
    float DVDX = (VX1 - VX2) * DXK_Rez * 0.5f;
    float DWDX = (WX1 - WX2) * DXK_Rez * 0.5f;
    float DUDY = (UY1 - UY2) * DYK_Rez * 0.5f;
    float DVDY = (VY1 - VY2) * DYK_Rez;
    float DWDY = (WY1 - WY2) * DYK_Rez * 0.5f;
    float DUDZ = UK[k + 1] * DZK_Rez * 0.5f;
    float DVDZ = VK[k + 1] * DZK_Rez * 0.5f;
    float DWDZ = WK[k + 1] * DZK_Rez * 0.5f;
    if (k > KK + 1) {
        DUDZ = (UK[k + 1] - UK[k - 1]) * DZK_Rez * 0.5f;
        DVDZ = (VK[k + 1] - VK[k - 1]) * DZK_Rez * 0.5f;
        DWDZ = (WK[k + 1] - WK[k - 1]) * DZK_Rez * 0.5f;
    }
    float s1 = DUDY + DVDX, s2 = DUDZ + DWDX, s3 = DVDZ + DWDY;
    float PROTURB = VIS * AREA * dz *
                    (2.0f * (DUDX * DUDX) + 2.0f * (DVDY * DVDY) + 2.0f * (DWDZ * DWDZ) + s1 * s1 + s2 * s2 + s3 * s3 - TDISS[k]);
    float PROBOU = (float)((double)(-d.potdtdz) * 9.81 / 283.0 * (double)VIS * 1.35 * (double)AREA * (double)dz);
    r.A = AIM; r.B1 = BIM; r.C1 = CIM; r.B2 = BIMEPS; r.C2 = CIMEPS;
    r.AW1 = AW1; r.AS1 = AS1; r.AE1 = AE1; r.AN1 = AN1;
    r.w1 = ap0 * TURB[k]; r.PRO = PROTURB; r.PBO = PROBOU;
    r.w2 = ap0 * TDISS[k];
    r.EPS = TDISS[k] / TURB[k] * (Ceps1 * PROTURB - Ceps2 * TDISS[k]);
    // wall functions of the back-substitution (they read only UK/VK/WK)
    int wf = 0; float wt = 0, we = 0;
    if (KK < k) {
        float us;
        if ((k == KK + 1) && (q.cutk == 0)) {
            wf = 1;
            const size_t cc = t.c;
            if (d.tke_br[cc]) {
                double s = sqrt((0.5 * (double)(UK[k + 1] + UKip[k + 1])) * (0.5 * (double)(UK[k + 1] + UKip[k + 1])) +
                                (0.5 * (double)(VK[k + 1] + VKjp[k + 1])) * (0.5 * (double)(VK[k + 1] + VKjp[k + 1])));
                us = (float)(d.tke_a[cc] * s);
            } else {
                double s = sqrt((0.5 * (double)(UK[k + 1] + UKip[k])) * (0.5 * (double)(UK[k + 1] + UKip[k])) +
                                (0.5 * (double)(VK[k] + VKjp[k])) * (0.5 * (double)(VK[k] + VKjp[k])));
                us = (float)(d.tke_a[cc] * s);
            }
            wt = (float)(3.33 * (double)(us * us));
            we = (float)((double)(us * us * us) / d.tke_den[cc]);
        } else if ((k == KK + 1) && (q.cutk > 0)) {
            wf = 1;
            double a1 = 0.5 * (double)(UK[k] + UKip[k]), b1 = 0.5 * (double)(VK[k] + VKjp[k]);
            us = q.ho * (float)sqrt(a1 * a1 + b1 * b1);
            wt = (float)(3.33 * (double)(us * us));
            we = (float)((double)(us * us * us) / ((double)dz * 0.5 * 0.4));
        } else if (((k == t.kkip + 1) && t.cip) || ((k == t.kkim + 1) && t.cim)) {
            wf = 1;
            double a1 = 0.5 * (double)(WK[k] + WK[k + 1]), b1 = 0.5 * (double)(VK[k] + VKjp[k]);
            us = (float)((double)d.ufx * sqrt(a1 * a1 + b1 * b1));
            wt = (float)(3.33 * (double)(us * us));
            we = (float)((double)(us * us * us) / ((double)d.bz0 * 0.4));
        } else if (((k == t.kkjp + 1) && t.cjp) || ((k == t.kkjm + 1) && t.cjm)) {
            wf = 1;
            double a1 = 0.5 * (double)(WK[k] + WK[k + 1]), b1 = 0.5 * (double)(UK[k] + UKip[k]);
            us = (float)((double)d.ufx * sqrt(a1 * a1 + b1 * b1));
            wt = (float)(3.33 * (double)(us * us));
            we = (float)((double)(us * us * us) / ((double)d.bz0 * 0.4));
        }
    }
    r.wf = wf; r.wt = wt; r.we = we;
    return r;
}

__global__ __launch_bounds__(WAVE) void k_tke(const Dom *__restrict__ ds, int t, int IS, int JS) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice

    extern __shared__ float sm[];
    const int nkp = d.nkp, tid = threadIdx.x;
    int a, b;
    if (!diag_col(t, 2, d.nii - 1, 2, d.njj - 1, blockIdx.x, a, b)) return;
    int i = (IS == -1) ? d.nii - a + 1 : a;
    int j = (JS == -1) ? d.njj - b + 1 : b;
    size_t c = c2(d, i, j);
    if (d.adv[c] != 1) return;
    ColInfo q = col_info(d, i, j);
    float *sA = sm, *sB1 = sA + nkp, *sC1 = sB1 + nkp, *sD1 = sC1 + nkp, *sB2 = sD1 + nkp, *sC2 = sB2 + nkp,
          *sD2 = sC2 + nkp, *sT = sD2 + nkp, *sE = sT + nkp, *sWT = sE + nkp, *sWE = sWT + nkp;
    int *sWF = (int *)(sWE + nkp);
    const TkeCol tc = tke_col(d, i, j);
    size_t o = tc.o;
    const gf32 *TURB = tc.TURB, *TDISS = tc.TDISS;
    const gf32 *TURBim = d.turb + c3(d, i - 1, j), *TURBip = d.turb + c3(d, i + 1, j);
    const gf32 *TURBjm = d.turb + c3(d, i, j - 1), *TURBjp = d.turb + c3(d, i, j + 1);
    const gf32 *TDISSim = d.tdiss + c3(d, i - 1, j), *TDISSip = d.tdiss + c3(d, i + 1, j);
    const gf32 *TDISSjm = d.tdiss + c3(d, i, j - 1), *TDISSjp = d.tdiss + c3(d, i, j + 1);
    int KK = q.KK;
    for (int k = q.KSTART + tid; k <= q.VI; k += WAVE) {
        const TkeCell e = tke_cell(d, q, tc, k);
        float DIMTURB = e.AW1 * TURBim[k] + e.AS1 * TURBjm[k] + e.AE1 * TURBip[k] + e.AN1 * TURBjp[k] + e.w1 + e.PRO + e.PBO;
        float DIMTDISS = e.AW1 * TDISSim[k] + e.AS1 * TDISSjm[k] + e.AE1 * TDISSip[k] + e.AN1 * TDISSjp[k] + e.w2 + e.EPS;
        sA[k] = e.A; sB1[k] = e.B1; sC1[k] = e.C1; sD1[k] = DIMTURB; sB2[k] = e.B2; sC2[k] = e.C2; sD2[k] = DIMTDISS;
        sWF[k] = e.wf; sWT[k] = e.wt; sWE[k] = e.we;
    }
    for (int k = q.KSTART + tid; k <= q.VI + 1; k += WAVE) { sT[k] = TURB[k]; sE[k] = TDISS[k]; }
    __syncthreads();
    if (tid == 0) {
        float P1 = 0, Q1 = 0, P2 = 0, Q2 = 0;
        for (int k = q.KSTART; k <= q.VI; ++k) {
            float A = sA[k];
            float p1, q1, p2, q2;
            if (k > KK + 1) {
                p1 = sB1[k] / (A - sC1[k] * P1);
                q1 = (sD1[k] + sC1[k] * Q1) / (A - sC1[k] * P1);
                p2 = sB2[k] / (A - sC2[k] * P2);
                q2 = (sD2[k] + sC2[k] * Q2) / (A - sC2[k] * P2);
            } else {
                p1 = sB1[k] / A; q1 = sD1[k] / A; p2 = sB2[k] / A; q2 = sD2[k] / A;
            }
            sB1[k] = p1; sD1[k] = q1; sB2[k] = p2; sD2[k] = q2;
            P1 = p1; Q1 = q1; P2 = p2; Q2 = q2;
        }
        float tup = sT[q.VI + 1], eup = sE[q.VI + 1];
        for (int k = q.VI; k >= q.KSTART; --k) {
            float tv = sT[k], ev = sE[k];
            if (KK < k) {
                if (sWF[k]) { tv = sWT[k]; ev = sWE[k]; }
                else { tv = sB1[k] * tup + sD1[k]; ev = sB2[k] * eup + sD2[k]; }
                tv = (float)mmaxd((double)tv, 0.001);
                ev = (float)mmaxd((double)ev, 0.0000001);
                sT[k] = tv; sE[k] = ev;
            }
            tup = tv; eup = ev;
        }
    }
    __syncthreads();
    gf32 *TW = d.turb + o, *EW = d.tdiss + o;
    for (int k = q.KSTART + tid; k <= q.VI; k += WAVE) { TW[k] = sT[k]; EW[k] = sE[k]; }
}

// ------------------------------------------------------------------------
// Strip wavefront path (mixing-length model and pressure)
// ------------------------------------------------------------------------
// A workgroup owns consecutive sweep rows (b) with one wave per row, a chain
// wave and a control wave.  Row wave r owns row b0 + r and at local step s handles column
// a = oa + s - r, so every local step is one anti-diagonal of the strip.  Each
// step is two phases separated by workgroup barriers: (1) every active row wave
// finishes its column's source terms (lanes over k) with the two neighbours the
// step before updated, read from LDS, (2) the chain wave runs the serial Thomas
// recurrences of all the strip's columns (lane = row) while the row waves store
// the column before, work up the next one and load the one after.
#define STRIP_WAVES 16            // waves of a strip at most: 14 rows, the chain and the control wave

// coefficient records written by k_ml_coef and read by the strip sweeps; per
// cell, two records, each written whole, in one pass:
//   planes: U, V {AW, AS, AE, AN | f, g, e, c0 | X1, X2, X3, X4} (REC_UV floats),
//           W    {AW, AS, AE, AN | f, g, e, X1}                   (REC_W floats),
//   written by the first pass of k_ml_coef;
//   rec3 = {C, T, P}, written after the P/TERMP recurrence.
// The U/V wall term exists only at KKART+1 and is kept per column (wcol).
#define REC_UV 12
#define REC_W 8
template <int COMP> __device__ __forceinline__ constexpr int rec_floats() { return COMP == 2 ? REC_W : REC_UV; }

__device__ __forceinline__ void sweep_to_ij(const DomG &d, int comp_is_pressure, int a, int b, int IS, int JS, int &i, int &j) {
    if (comp_is_pressure) {   // a = j1, b = i1
        j = (JS == -1) ? d.njj - a + 1 : a;
        i = (IS == -1) ? d.nii - b + 1 : b;
    } else {                  // a = i1, b = j1
        i = (IS == -1) ? d.nii - a + 1 : a;
        j = (JS == -1) ? d.njj - b + 1 : b;
    }
}

// workgroup barrier that orders LDS only; global loads stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// odd LDS row stride: lanes of one wave that walk different columns at the
// same relative level hit different banks
__device__ __forceinline__ int lds_stride(int nkp) { return nkp | 1; }

#define COEF_COLS 16
#define SCOL 16           // words of column data per column in k_ml_coef
// All neighbour-independent work of one mixing-length sweep for every column
// at once.  A block of 4 waves takes COEF_COLS consecutive columns of the
// sweep; their active levels are laid out one after another and dealt to the
// block's 256 lanes (a lane per level, whatever the column heights), which
// compute the coefficients.  One wave then runs the P/TERMP recurrence of all
// COEF_COLS columns at once (lane = column), and the lanes write the last part
// of each cell's record.  Each record is written once, as float4 / float3 stores.
// WFIX: the solver width when every situation of the launch has it (the
// width-dependent arithmetic then folds at compile time), 0 to read it per
// situation.  KIND 0: mixing length (rec3 = {C, TERMP, P}); KIND 1: k-eps and
// KIND 2: no diffusion, whose solvers divide by the TDMA denominator instead
// of multiplying by its reciprocal (rec3 = {C, denominator, P}).
template <int COMP, int WFIX, int KIND = 0>
__global__ __launch_bounds__(4 * WAVE) void k_ml_coef(const Dom *__restrict__ ds, int IS, int JS) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    gf32 *planes = d.planes;

    extern __shared__ float sm[];
    const int nkp = d.nkp, nkl = lds_stride(nkp);
    const int lane = threadIdx.x % WAVE;
    const int oa = (COMP == 0) ? 3 : 2, ia = (COMP == 1) ? 3 : 2;
    const int na = d.nii - 1 - oa + 1, nb = d.njj - 1 - ia + 1;
    // per column c: A, B, C over k at sm + c*3*nkl, and the column's data
    // (read once per column here, not once per level)
    int *scol = (int *)(sm + 3 * COEF_COLS * nkl);         // [COEF_COLS][SCOL]
    int *stot = scol + SCOL * COEF_COLS;
    const int blk = xcd_block((na * nb + COEF_COLS - 1) / COEF_COLS);
    if (blk < 0) return;                                      // uniform over the block
    const int col0 = blk * COEF_COLS;
    if (threadIdx.x < WAVE) {
        int c = lane, n = 0;
        if (c < COEF_COLS) {
            int col = col0 + c;
            int i = 0, j = 0;
            Meta m;
            m.adv = false;
            if (col < na * nb) {
                sweep_to_ij(d, 0, oa + col / nb, ia + col % nb, IS, JS, i, j);
                m = unpack_meta(ldg4i(d.meta + c2(d, i, j)));
            }
            if (m.adv) {
                // U and V: the levels inside a building are neither updated nor
                // read by the recurrence above them
                if (COMP != 2) m.KSTART = m.KK + 1;
                n = m.VI - m.KSTART + 1;
                const ColInfo q = col_info(d, i, j);
                int *sc = scol + c * SCOL;
                sc[7] = (q.as ? 1 : 0) | (q.an ? 2 : 0) | (q.aw ? 4 : 0) | (q.ae ? 8 : 0) | (q.vegp ? 16 : 0);
                sc[8] = __float_as_int(q.cutk); sc[9] = __float_as_int(q.cov); sc[10] = __float_as_int(q.ht);
                sc[11] = __float_as_int(q.ho); sc[12] = __float_as_int(q.z0s);
            }
            scol[c * SCOL + 0] = m.KSTART; scol[c * SCOL + 1] = m.KK; scol[c * SCOL + 2] = m.VI;
            scol[c * SCOL + 3] = i; scol[c * SCOL + 4] = j; scol[c * SCOL + 6] = m.adv ? 1 : 0;
        }
        // inclusive prefix sum of the level counts over the lanes
        int incl = n;
        for (int off = 1; off < WAVE; off <<= 1) {
            int v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (c < COEF_COLS) scol[c * SCOL + 5] = incl - n;
        if (lane == WAVE - 1) stot[0] = incl;
    }
    lds_barrier();
    const int total = stot[0];
    // the column holding item t is the last c with first[c] <= t: first[] does
    // not decrease, and every later column starts beyond t
    auto column_of = [&](int t) {
        int lo = 0;
        for (int step = COEF_COLS / 2; step > 0; step >>= 1)
            if (scol[(lo + step) * SCOL + 5] <= t) lo += step;
        return lo;
    };
    for (int t = threadIdx.x; t < total; t += 4 * WAVE) {
        const int c = column_of(t);
        const int *sc = scol + c * SCOL;
        const int k = sc[0] + (t - sc[5]);
        ColInfo q;
        q.KSTART = sc[0]; q.KK = sc[1]; q.VI = sc[2]; q.i = sc[3]; q.j = sc[4];
        const int fl = sc[7];
        q.as = fl & 1; q.an = (fl >> 1) & 1; q.aw = (fl >> 2) & 1; q.ae = (fl >> 3) & 1; q.vegp = (fl >> 4) & 1;
        q.cutk = __int_as_float(sc[8]); q.cov = __int_as_float(sc[9]); q.ht = __int_as_float(sc[10]);
        q.ho = __int_as_float(sc[11]); q.z0s = __int_as_float(sc[12]);
        q.W = WFIX ? WFIX : d.simd;
        MlPieces p;
        if constexpr (KIND != 0)
            p = (COMP == 2) ? ke_w_pieces<KIND == 1>(d, q, k) : ke_uv_pieces<COMP == 1, KIND == 1>(d, q, k);
        else p = ml_pieces<COMP>(d, q, k);
        float *sA = sm + (size_t)c * 3 * nkl;
        sA[k] = p.A; sA[nkl + k] = p.B; sA[2 * nkl + k] = p.C;
        gf32 *P = planes + (c3(d, q.i, q.j) + k) * rec_floats<COMP>();
        stg4(P, p.AW1, p.AS1, p.AE1, p.AN1);
        if (COMP == 2) {
            stg4(P + 4, p.f, p.g, p.e, p.X1);
        } else {
            stg4(P + 4, p.f, p.g, p.e, p.c0);
            stg4(P + 8, p.X1, p.X2, p.X3, p.X4);
            if (k == q.KK + 1) d.wcol[c2(d, q.i, q.j)] = p.w;
        }
    }
    lds_barrier();
    if (threadIdx.x < COEF_COLS && scol[threadIdx.x * SCOL + 6]) {
        const int c = threadIdx.x;
        float *__restrict__ A = sm + (size_t)c * 3 * nkl;
        float *__restrict__ Bq = A + nkl;
        float *__restrict__ Cq = Bq + nkl;
        const int KSTART = scol[c * SCOL + 0], KKP1 = scol[c * SCOL + 1] + 1, VI = scol[c * SCOL + 2];
        float Pp = 0;
        for (int k = KSTART; k <= VI; ++k) {
            float T, P;
            if (KIND != 0) {
                T = (k > KKP1) ? A[k] - Cq[k] * Pp : A[k];
                P = Bq[k] / T;
            } else {
                T = (k > KKP1) ? 1 / (A[k] - Cq[k] * Pp) : 1 / A[k];
                P = Bq[k] * T;
            }
            A[k] = T;          // T replaces A, P replaces B
            Bq[k] = P;
            Pp = P;
        }
    }
    lds_barrier();
    for (int t = threadIdx.x; t < total; t += 4 * WAVE) {
        const int c = column_of(t);
        const int k = scol[c * SCOL + 0] + (t - scol[c * SCOL + 5]);
        const float *sA = sm + (size_t)c * 3 * nkl;
        gf32 *P = d.rec3 + (c3(d, scol[c * SCOL + 3], scol[c * SCOL + 4]) + k) * 3;
        stg3(P, sA[2 * nkl + k], sA[k], sA[nkl + k]);                   // C, T (or the denominator), P
    }
}


// ------------------------------------------------------------------------
// Strip-pipelined sweeps.  Strip B reads the last row of strip B-1 (its new
// values, and for the pressure sweep the QIMP row scratch) and nothing else
// from other strips, so it only has to stay a strip's rows behind strip B-1: one
// launch holds the whole sweep, whose serial path is about (a range) + rows *
// (number of strips) local steps.
//
// Strips are numbered by a ticket per sweep kind (sync[SYNC_BLOCK0 + kind *
// sync_stride], cleared at the start of every iteration) in the order their
// workgroups start, so the strip a workgroup waits for is held by a workgroup
// that is already running, whatever the dispatch order.  Every wait is bounded
// (STRIP_TIMEOUT_TICKS of the constant 100 MHz clock): on timeout the strip sets
// the situation's sticky error flag (sync[0]) and goes on without waiting, so the
// kernel always ends; the host reports the error.
// ------------------------------------------------------------------------
#define STRIP_TIMEOUT_TICKS 200000000ull

__device__ __forceinline__ void store_agent(gi32 *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------------
// Strip rows in LDS.  A row's operands are stored by level relative to the
// column's first free level, t = k - KKART - 1: the recurrences of all rows then
// start at t = 0 on a 16-byte boundary whatever the columns' ground heights, and
// walk chunks of CHK levels with ds_read_b128 / ds_write_b128 (a lone wave
// issues an instruction every 4.5 cycles and a dependent one every 8.4, so with
// 4-byte LDS accesses the recurrences were bound by their own instruction
// stream: 46 and 55 cycles per level forward and back, 31 and 46 with 16-byte
// accesses, against 25 and 42 for their 3 and 5 dependent operations).  An array
// holds strip_low() levels below t = 0 (W inside buildings; the lowest chunk
// is where lanes that are done store) and one spare chunk above the tallest
// column (read ahead, or written by lanes past their own end).  The row stride
// is 4 modulo 64 words: the 16-byte accesses of the chain wave's lanes fall into
// different banks.
// ------------------------------------------------------------------------
#define CHK 8
__host__ __device__ inline int strip_low(int nlow) { return ((nlow + CHK - 1) & ~(CHK - 1)) + CHK; }
__host__ __device__ inline int strip_len(int nlow, int nact) { return strip_low(nlow) + ((nact + CHK - 1) & ~(CHK - 1)) + CHK; }
__host__ __device__ inline int strip_stride(int arrays, int len) { return arrays * len + ((4 - arrays * len) & 63); }

struct Chunk { float v[CHK]; };
__device__ __forceinline__ Chunk ld_chunk(const float *p) {
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    return Chunk{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}
__device__ __forceinline__ void st_chunk(float *p, const Chunk &c) {
    *(float4 *)p = make_float4(c.v[0], c.v[1], c.v[2], c.v[3]);
    *(float4 *)(p + 4) = make_float4(c.v[4], c.v[5], c.v[6], c.v[7]);
}
// largest value over the 16 lanes of each row of the wave (lanes 0-15, 16-31,
// ...): rotations within the row instead of LDS permutes
__device__ __forceinline__ int row_max(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x122, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x121, 0xf, 0xf, false));
    return v;
}

// The chunk loops are straight-line blocks of CHK_BLOCK chunks: within a block
// the compiler waits for exactly the reads a chunk needs, while a loop's back
// edge makes it wait for every LDS access in flight.  Each chunk issues the
// next chunk's reads before its own operations, in one group: an LDS access
// between two dependent operations costs more than its issue.  Measured on one
// wave, 40 levels, in cycles per level: forward 29.6, back 39.7, pressure up
// 24.6; with two chunks per loop round 34.7, 49.8, 29.3; with the reads between
// the operations 37.6, 44.7, 25.4.
#define CHK_BLOCK 8

// The first operands of a recurrence that the step's assembly does not change are
// read before the barrier that ends it, while the chain wave waits there anyway
// (city of 400 x 400, 20 iterations: 137.3 -> 133.5 ms).
// chunk_of: the chunk of t = n - 1; without a column (n = 0) the one below t = 0
__device__ __forceinline__ int chunk_of(int n) { return (n - 1) & ~(CHK - 1); }

// forward: Q[t] = (D[t] + C[t]*Q[t-1]) * T[t] for nch chunks from t = 0, where
// Q[0] = D[0]*T[0]; Q replaces D
template <bool DIV>
__device__ __forceinline__ void strip_fwd(float *DQ, const float *C, const float *T, int nch, const Chunk &c0, const Chunk &t0) {
    float q = 0.0f;
    Chunk d[2], c[2] = {c0}, t[2] = {t0};
    d[0] = ld_chunk(DQ);
    c[0].v[0] = -0.0f;                                        // -0*0 added to D[0] leaves it as it is
    for (int b = 0; b < nch; b += CHK_BLOCK) {
#pragma unroll
        for (int h = 0; h < CHK_BLOCK; ++h) {
            if (b + h >= nch) return;
            const int k = h & 1, n = k ^ 1;
            d[n] = ld_chunk(DQ + (h + 1) * CHK); c[n] = ld_chunk(C + (h + 1) * CHK); t[n] = ld_chunk(T + (h + 1) * CHK);
            __builtin_amdgcn_sched_barrier(0);                // the next chunk's reads stay ahead of this chunk
#pragma unroll
            for (int u = 0; u < CHK; ++u) {
                const float s = d[k].v[u] + c[k].v[u] * q;
                q = DIV ? s / t[k].v[u] : s * t[k].v[u];
                d[k].v[u] = q;
            }
            st_chunk(DQ + h * CHK, d[k]);
        }
        DQ += CHK_BLOCK * CHK; C += CHK_BLOCK * CHK; T += CHK_BLOCK * CHK;
    }
}

// relaxed back-substitution from t = n-1 down, nch chunks starting with the one
// that holds t = n-1: X[t] += relax*(P[t]*X[t+1] + Q[t] - X[t]).  part: some lane's
// column ends inside its first chunk.  Lanes that are done go on in the chunk
// at low (the arrays' start).
__device__ __forceinline__ void strip_back(const float *P, const float *Q, float *X, float relax, int n, int nch, bool part,
                                           int low, const Chunk &p0, const Chunk &x0, float up) {
    int o = chunk_of(n);
    const int top = n - o;
    Chunk p[2] = {p0}, q[2], x[2] = {x0};
    q[0] = ld_chunk(Q + o);
    for (int b = 0; b < nch; b += CHK_BLOCK) {
#pragma unroll
        for (int h = 0; h < CHK_BLOCK; ++h) {
            if (b + h >= nch) return;
            const int k = h & 1, m = k ^ 1, on = max(o - CHK, -low);
            p[m] = ld_chunk(P + on); q[m] = ld_chunk(Q + on); x[m] = ld_chunk(X + on);
            __builtin_amdgcn_sched_barrier(0);
            if (h == 0 && part && b == 0) {
#pragma unroll
                for (int u = CHK - 1; u >= 0; --u) {
                    const float r = x[k].v[u] + relax * (p[k].v[u] * up + q[k].v[u] - x[k].v[u]);
                    up = (u >= top) ? up : r;
                    x[k].v[u] = r;
                }
            } else {
#pragma unroll
                for (int u = CHK - 1; u >= 0; --u) {
                    up = x[k].v[u] + relax * (p[k].v[u] * up + q[k].v[u] - x[k].v[u]);
                    x[k].v[u] = up;
                }
            }
            st_chunk(X + o, x[k]);
            o = on;
        }
    }
}

// Hand-off between strips: the last row's new values go to the next strip as
// 8-byte {value, tag} words, each one store, so the reader needs no progress
// counter: a word whose tag is this sweep's holds this sweep's value.  The tag
// counts the situation's iterations (sync[1], advanced by k_zero_rows) and
// names the sweep, so no word of an earlier sweep matches.  Against a progress
// counter the writer need not wait for its stores and the reader not for a poll
// before its loads.  The words also keep the next strip from overwriting old
// values this one still reads: a momentum sweep hands on every level the last row's
// column reads, updated or not (hand_sent(), hand_needed()); the pressure and TKE
// sweeps and the line strips update all the levels they read.
typedef unsigned long long __attribute__((address_space(1))) gu64;
__device__ __forceinline__ unsigned hand_tag(const DomG &d, int kind) { return 8u * (unsigned)d.sync[1] + (unsigned)kind; }
__device__ __forceinline__ void hand_put(gu64 *p, float v, unsigned tag) {
    __hip_atomic_store(p, ((unsigned long long)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long hand_get(const gu64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// bounded wait of a whole wave for the words of the lanes that need one
struct HandWait {
    gi32 *error;
    unsigned long long deadline;
    bool dead;
    __device__ __forceinline__ void wait(const gu64 *p, bool need, unsigned tag, unsigned long long &w) {
        for (int spins = 0; __any(need && (unsigned)(w >> 32) != tag) && !dead; ++spins) {
            if (wall_clock64() > deadline || spins > (1 << 22)) {
                store_agent(error, 1);
                dead = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            if (need) w = hand_get(p);
        }
    }
};

// LDS positions as byte offsets from the workgroup's dynamic LDS, and columns of
// a field as a uniform byte address plus a 32-bit lane offset: with the offset
// opaque to the compiler at every use the access takes the scalar-base form,
// otherwise it widens the offset once and adds 64-bit addresses per access.
__device__ __forceinline__ float &lds_at(float *sm, int byte_off) { return *(float *)((char *)sm + byte_off); }
typedef const char __attribute__((address_space(1))) gc8;
__device__ __forceinline__ const gf32 *lane_at(const gf32 *base, unsigned byte_off) {
    asm volatile("" : "+v"(byte_off));
    return (const gf32 *)((gc8 *)base + byte_off);
}

template <int COMP>
__device__ __forceinline__ StripCol strip_col(int4 m) { return strip_col<COMP>(m.x, m.y, m.z, m.w); }

// Raw operands of one column, as loaded one step before they are worked up:
// records, own and old neighbour values, the -IS / -JS neighbours' values as
// memory holds them (used where this sweep does not update them) and, for row 0
// of a strip, the hand-off words of the previous strip's last row.
struct MlRaw {
    float4 v0, v2, v3;
    float3 v1;
    float x, xa, xb, ni, nj;
    unsigned long long hw;
};
// What a column's assembly needs beside the two new neighbour values
struct MlIn {
    float ai, aj, pa, pb;      // coefficients of the new neighbours, products of the old ones
    float ao, xo;              // coefficient and value of the old i neighbour (512-bit solvers fuse their product)
    float e, f, g, w, x, dd, eo, y1, y2, y3, y4, c0, t;
    double t5, fd, gd;
    float ni, nj;
    int li, lj;                // LDS positions of the new neighbours' values
    bool si, sj, cross;        // they hold this level; the cross terms apply
};

// One strip of a momentum sweep.  R row waves own a sweep row each, the chain
// wave runs the recurrences of all rows (lane = row), the control wave prepares
// the chain wave's column data and hands the last row's results to the next
// strip.  A local step s has two phases between barriers:
//   1. every row reads the two new neighbour values of its column (a = oa+s-r)
//      from LDS and finishes the source term D; everything else in D was worked
//      up before;
//   2. the chain wave runs the forward recurrence and the back-substitution,
//      while the rows work up the column of step s+1 (loaded a whole step
//      before: coefficients to LDS, products of the old neighbours and the
//      cross terms' fixed parts to registers), issue the loads of step s+2 and
//      store the column of step s-1.
// Bound by the recurrences (40 levels: about 31 + 46 cycles per level) plus phase
// 1.  M: 64-level groups a column of this sweep can span.  WFIX: the solver
// width when every situation of the launch has it, else 0.
// KIND 0: mixing length; KIND 1: k-eps, KIND 2: no diffusion (sources by
// ke_source's arithmetic, the TDMA divides by the denominators k_ml_coef stored).
template <int COMP, int WFIX, int KIND, int M>
__global__ __launch_bounds__(STRIP_WAVES * WAVE) void k_ml_strip(const Dom *__restrict__ ds, int IS, int JS) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    extern __shared__ __align__(16) float sm[];
    // the fields the steps use, read once: a scalar load inside a step would
    // wait for its latency and, sharing its counter, for the LDS accesses
    const int nkp = d.nkp, nii = d.nii, njj = d.njj, nj2 = d.nj2, hcols = nii;
    const int low = strip_low((COMP == 2) ? d.nlow : 0), len = strip_len((COMP == 2) ? d.nlow : 0, d.nact);
    const int rs = strip_stride(9, len);
    const int oa = (COMP == 0) ? 3 : 2, ia = (COMP == 1) ? 3 : 2, ob = nii - 1, ib = njj - 1, na = ob - oa + 1;
    const int R = blockDim.x / WAVE - 2;                      // rows of a strip (strip_rows())
    const int nstrip = (ib - ia + R) / R, nsteps = na + R - 1;
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    gi32 *sync = d.sync + SYNC_BLOCK0 + (size_t)(1 + COMP) * d.sync_stride;
    // per row: D (replaced by Q), then per step parity C, T, P and X (the old
    // column, replaced by the new one)
    float *sdzk = sm + (size_t)R * rs, *sap0 = sdzk + nkp;         // [nkp] each
    int4 *sinfo = (int4 *)(sap0 + nkp);                       // [2][16] per row by step parity, for the chain wave
    int *sctl = (int *)(sinfo + 32);
    if (threadIdx.x == 0) sctl[0] = __hip_atomic_fetch_add(&sync[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = threadIdx.x; k < nkp; k += blockDim.x) { sdzk[k] = d.dzk[k]; sap0[k] = d.ap0[k]; }
    __syncthreads();
    const int B = __builtin_amdgcn_readfirstlane(sctl[0]);
    if (B >= nstrip) return;                                  // uniform over the workgroup
    const unsigned tag = hand_tag(d, 1 + COMP);
    gu64 *hand = (gu64 *)d.hand;                              // [strip][nii][nkp] words
    const int4 *meta = (const int4 *)d.meta;
    // The chain and the control wave run loops of their own with the same
    // barriers per step as the row waves (s_barrier counts waves, wherever they
    // are in the code), so none of the row waves' registers is live in the
    // recurrences.  They issue ahead of the row waves on their SIMDs (wave
    // priority): the recurrences are the step's serial path.
    if (r == R) {
        __builtin_amdgcn_s_setprio(3);
        const float relax = d.relax;
        float *L = sm + (size_t)(lane < R ? lane : 0) * rs + low;
        lds_barrier();                                        // the control wave's data of step 0
        for (int s = 0; s < nsteps; ++s) {
            // lane's levels (0: no column), the longest chains in chunks
            const int4 si = sinfo[(s & 1) * 16 + (lane & 15)];
            const int n = lane < R ? si.x : 0;
            const int fmax = __builtin_amdgcn_readfirstlane(si.y), bmax = __builtin_amdgcn_readfirstlane(si.z);
            const bool part = __builtin_amdgcn_readfirstlane(si.w) != 0;
            float *Lp = L + (1 + 4 * (s & 1)) * len;
            const int o = chunk_of(n);
            const Chunk c0 = ld_chunk(Lp), t0 = ld_chunk(Lp + len), p0 = ld_chunk(Lp + 2 * len + o), x0 = ld_chunk(Lp + 3 * len + o);
            const float up = Lp[3 * len + n];
            lds_barrier();                                    // the rows' sources are assembled
            if (n > 0) {
                strip_fwd<KIND != 0>(L, Lp, Lp + len, fmax, c0, t0);
                strip_back(Lp + 2 * len, L, Lp + 3 * len, relax, n, bmax, part, low, p0, x0, up);
            }
            lds_barrier();                                    // the recurrences are done
        }
        return;
    }
    if (r == R + 1) {
        __builtin_amdgcn_s_setprio(2);
        // lane r's column at step s is a = oa + s - r of row b; its metadata is
        // requested a step ahead
        const int b = ia + B * R + lane;
        const bool lane_ok = lane < R && b <= ib;
        int cidx = ((IS == -1) ? nii - oa + 1 : oa) * nj2 + ((JS == -1) ? njj - b + 1 : b) - lane * IS * nj2;
        auto meta_at = [&](int s) {
            const int l = s - lane;
            int4 m = make_int4(0, -1, 0, 0);
            if (lane_ok && l >= 0 && l < na) m = ldg4i((const DomG::P<const int4>)meta + cidx);
            cidx += IS * nj2;
            return m;
        };
        int4 mq = meta_at(0);
        StripCol c{0, -1, 0, 0, 0};                           // the column of step s
        auto info = [&](int s) {                              // ... of step s, into LDS
            const StripCol cn = strip_col<COMP>(mq);
            mq = meta_at(s + 1);
            const int n = cn.VI < 0 ? 0 : cn.VI - cn.KK;
            const int nb = n > 0 ? ((n - 1) >> 3) - ((cn.kend - cn.KK - 1) >> 3) + 1 : 0;
            const int part = __any((n & (CHK - 1)) != 0);
            const int fm = row_max((n + CHK - 1) >> 3), bm = row_max(nb);
            if (lane < 16) sinfo[(s & 1) * 16 + lane] = make_int4(n, fm, bm, part);
            return cn;
        };
        const bool send = B + 1 < nstrip;
        gu64 *h = hand + ((size_t)B * hcols - (R - 1)) * nkp; // the last row's column at step s: + s*nkp
        c = info(0);
        lds_barrier();
        for (int s = 0; s < nsteps; ++s) {
            lds_barrier();
            const StripCol cn = info(s + 1);
            lds_barrier();                                    // the recurrences are done
            const StripLevels hl = hand_sent<COMP>(c);
            const int hi = __builtin_amdgcn_readlane(hl.hi, R - 1);
            if (send && hi >= 0) {
                // the last row's results, the only column another strip reads, go
                // out while the rows assemble the next step; below the first updated
                // level only the tag counts
                const int lo = __builtin_amdgcn_readlane(hl.lo, R - 1), kkl = __builtin_amdgcn_readlane(c.KK, R - 1);
                const float *xn = sm + (size_t)(R - 1) * rs + (4 + 4 * (s & 1)) * len + low - (kkl + 1);
                for (int k = lo + lane; k <= hi; k += WAVE) hand_put(h + (size_t)s * nkp + k, xn[k], tag);
            }
            c = cn;
        }
        return;
    }
    const int b = ia + B * R + r;
    const bool row_ok = b <= ib, from_prev = r == 0 && B > 0;
    const bool ip = IS == 1, jp = JS == 1, v512 = KIND == 0 && (WFIX ? WFIX : d.simd) == 16;
    const int wlev = v512 ? 16 : 8;                           // levels of a vector block
    HandWait hwait{d.sync, wall_clock64() + STRIP_TIMEOUT_TICKS, false};
    // neighbour levels the sweep updates: the same row's previous column always
    // lies in the sweep, the previous row's only if there is one
    const bool has_j = r > 0 || B > 0;
    const float ddf = (COMP == 0) ? d.dyk : d.dxk;
    const int rowb = 4 * r * rs;                              // the row's LDS, in bytes
    const gf32 *X = (COMP == 0 ? d.uk : COMP == 1 ? d.vk : d.wk), *planes = d.planes, *rec3 = d.rec3, *wcol = d.wcol;
    // the row's column at l = s - r: column index cidx, one sweep step apart dcol
    const int dcol = IS * nj2;
    int l2 = -r;                                              // l of the step whose metadata is requested
    int cidx2 = ((IS == -1) ? nii - oa + 1 : oa) * nj2 + ((JS == -1) ? njj - b + 1 : b) - r * dcol;
    int4 m2, m2j;                                             // requested a step before their use
    auto request = [&]() {                                    // metadata of the next column and its -JS neighbour
        m2 = m2j = make_int4(0, -1, 0, 0);
        if (row_ok && l2 >= 0 && l2 < na) {
            m2 = ldc4i(meta + cidx2);
            if (has_j) m2j = ldc4i(meta + (cidx2 - JS));
        }
        ++l2;
        cidx2 += dcol;
    };
    // byte offsets of a lane in the columns it loads, from the lowest of them
    const unsigned fi = 4u * (unsigned)nj2 * (unsigned)nkp, fj = 4u * (unsigned)nkp, base = fi + fj;
    const unsigned off_c = base + 4u * lane, off_a = ip ? off_c + fi : off_c - fi, off_b = jp ? off_c + fj : off_c - fj;
    const unsigned off_i = ip ? off_c - fi : off_c + fi, off_j = jp ? off_c - fj : off_c + fj;
    const unsigned off_p = (unsigned)(4 * rec_floats<COMP>()) * lane, off_r = 12u * lane, off_h = 8u * lane;
    const StripCol none{0, -1, 0, 0, 0};
    StripCol c0 = none, c1 = none, c1j = none, c2m = none;    // columns of step s, s+1 (and its -JS neighbour), s-1
    unsigned o0 = 0, o1 = 0, op = 0;                          // their first cells
    MlRaw raw[M];
    MlIn in[M];
    float wraw = 0.0f;
    // requests the operands of the row's next column; p: the one before it
    auto issue = [&](const StripCol &p, const StripCol &cn, const StripCol &cnj) {
        c1 = cn;
        c1j = cnj;
        const int ci = cidx2 - 2 * dcol, l = l2 - 2;          // request() is one column ahead
        if (c1.VI < 0) return;
        o1 = (unsigned)ci * (unsigned)nkp;
        const int kb = (COMP == 2) ? c1.ks : c1.KK + 1;       // first level with a source
        const size_t o = (size_t)o1 + kb;
        const gf32 *Pc = planes + o * rec_floats<COMP>(), *R3 = rec3 + o * 3;
        const gf32 *Xl = X + o - (base >> 2);
        const gf32 *H = (const gf32 *)(hand + ((size_t)(B - 1) * hcols + l) * nkp + kb);
        const bool old_i = p.kend > kb || p.VI < c1.VI, old_j = c1j.kend > kb || c1j.VI < c1.VI;
        const int top = c1.VI + 1 - kb;
        if (COMP != 2) wraw = wcol[ci];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (lane + WAVE * m <= top) {
                MlRaw &q = raw[m];
                const gf32 *P = lane_at(Pc + m * WAVE * rec_floats<COMP>(), off_p);
                q.v0 = ldg4(P); q.v2 = ldg4(P + 4);
                if (COMP != 2) q.v3 = ldg4(P + 8);
                q.v1 = ldg3(lane_at(R3 + m * WAVE * 3, off_r));
                const gf32 *Xm = Xl + m * WAVE;
                q.x = *lane_at(Xm, off_c);
                q.xa = *lane_at(Xm, off_a);
                q.xb = *lane_at(Xm, off_b);
                if (old_i) q.ni = *lane_at(Xm, off_i);
                if (old_j) q.nj = *lane_at(Xm, off_j);
                if (from_prev) q.hw = hand_get((const gu64 *)lane_at(H + m * WAVE * 2, off_h));
            }
        }
    };
    // works up the operands of step s: recurrence operands to LDS, the rest to in[]
    auto work_up = [&](int s, const StripCol &p) {
        const StripCol &c = c1;
        if (c.VI < 0) return;
        const int kb = (COMP == 2) ? c.ks : c.KK + 1;
        // LDS of level k: at(k) + 4*lane, X of this and the other parity
        const int sc = rowb + 4 * ((1 + 4 * (s & 1)) * len + low + kb - (c.KK + 1)), l4 = 4 * len;
        const int sx = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + kb - (p.KK + 1));
        const int sj = rowb - 4 * rs + 4 * ((8 - 4 * (s & 1)) * len + low + kb - (c1j.KK + 1));
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int t4 = 4 * (lane + WAVE * m), k = kb + lane + WAVE * m;
            MlRaw &q = raw[m];
            MlIn &a = in[m];
            if (k <= c.VI + 1) lds_at(sm, sc + 3 * l4 + t4) = q.x;
            if (k <= c.VI) {
                lds_at(sm, sc + t4) = q.v1.x;
                lds_at(sm, sc + l4 + t4) = q.v1.y;
                lds_at(sm, sc + 2 * l4 + t4) = q.v1.z;
                const float aw = q.v0.x, as = q.v0.y, ae = q.v0.z, an = q.v0.w;
                a.ai = ip ? aw : ae; a.aj = jp ? as : an;
                a.ao = ip ? ae : aw; a.xo = q.xa;
                a.pa = a.ao * q.xa; a.pb = (jp ? an : as) * q.xb;
                a.e = q.v2.z; a.f = q.v2.x; a.g = q.v2.y;
                a.x = q.x; a.t = q.v1.y;
                bool cross = KIND != 2 && k > c.KK + 1;
                if (KIND == 0) cross = min(c.ks + ((k - c.ks) & -wlev), c.VI + 1 - wlev) > c.KK + 1;   // block_base()
                a.cross = cross;
                if (COMP == 2) {
                    a.y1 = cross ? q.v2.w : -0.0f;            // -0: adding it changes nothing
                } else {
                    a.c0 = q.v2.w;
                    a.w = (lane + WAVE * m == 0) ? wraw : 0.0f;
                    a.dd = ddf * sdzk[k];
                    a.y1 = q.v3.x; a.y2 = q.v3.y; a.y3 = q.v3.z; a.y4 = q.v3.w;
                    const bool fwd = (COMP == 0) ? ip : jp;   // the new value is the lower neighbour's
                    const float xold = (COMP == 0) ? q.xa : q.xb;
                    a.eo = (fwd ? xold - q.x : q.x - xold) * a.dd;
                    if (COMP == 1) {
                        a.y1 = a.y1 - a.y2;
                        if (fwd) a.y1 = a.y1 + a.eo;
                    }
                    if (COMP == 0 && v512 && !c.veg) a.g = -0.0f;
                }
                if (KIND != 0) {
                    a.t5 = (double)sap0[k] * 0.5 * (double)a.e;
                    a.fd = (double)a.f; a.gd = (double)a.g;
                }
                a.ni = q.ni; a.nj = q.nj;
                a.si = k >= p.kend && k <= p.VI;
                a.sj = k >= c1j.kend && k <= c1j.VI;
                // a safe position where the neighbour does not hold the level
                a.li = a.si ? sx + t4 : 0;
                a.lj = a.sj ? sj + t4 : 0;
            }
        }
        if (from_prev) {
            const gu64 *h = hand + ((size_t)(B - 1) * hcols + (s - r)) * nkp;
            const StripLevels hl = hand_needed<COMP>(c, c1j);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = kb + lane + WAVE * m;
                const bool need = k >= hl.lo && k <= hl.hi;
                hwait.wait(h + k, need, tag, raw[m].hw);
                if (need && k >= c1j.kend) in[m].nj = __uint_as_float((unsigned)raw[m].hw);
                in[m].sj = false;                             // the value is in nj
                in[m].lj = 0;
            }
        }
    };
    StripCol c2, c2j;                                         // column of step s+2
    auto located = [&]() {
        c2 = strip_col<COMP>(m2);
        c2j = strip_col<COMP>(m2j);
        request();
    };
    request();
    located();
    issue(none, c2, c2j);
    located();
    work_up(0, none);
    c0 = c1; o0 = o1;
    issue(c0, c2, c2j);
    lds_barrier();                                            // the control wave's data of step 0
    for (int s = 0; s < nsteps; ++s) {
        // phase 1: the new neighbours enter the source terms of step s
        if (c0.VI >= 0) {
            const int kb = (COMP == 2) ? c0.ks : c0.KK + 1;
            const int sd = rowb + 4 * (low + kb - (c0.KK + 1));
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = kb + lane + WAVE * m;
                if (k <= c0.VI) {
                    const MlIn &a = in[m];
                    float vi = lds_at(sm, a.li), vj = lds_at(sm, a.lj);
                    vi = a.si ? vi : a.ni;
                    vj = a.sj ? vj : a.nj;
                    const float mi = a.ai * vi, mj = a.aj * vj;
                    float D;
                    if (v512 && (COMP != 1 || c0.veg)) {
                        // FMA(AW, X_W, AS*X_S) + FMA(AE, X_E, AN*X_N)
                        const float ts = jp ? mj : a.pb, tn = jp ? a.pb : mj;
                        const float xw = ip ? vi : a.xo, xe = ip ? a.xo : vi, aw = ip ? a.ai : a.ao, ae = ip ? a.ao : a.ai;
                        D = fmaf(aw, xw, ts) + fmaf(ae, xe, tn);
                    } else {                                  // AW*X_W + AS*X_S + AE*X_E + AN*X_N; selects, no branches
                        D = (ip ? mi : a.pa) + (jp ? mj : a.pb) + (ip ? a.pa : mi) + (jp ? a.pb : mj);
                    }
                    if (KIND != 0) {
                        if (COMP == 2) D = (float)((double)D + a.t5 + a.fd);
                        else D = (float)((double)D + a.t5 + a.fd + a.gd);
                    } else {
                        D = D + a.e + a.f;
                        D = (COMP == 2) ? D - a.g : D + a.g;
                    }
                    if (COMP != 2) {
                        D -= a.w;
                        if (KIND != 2) {
                            float z;
                            if (COMP == 0) {
                                const float en = (ip ? a.x - vi : vi - a.x) * a.dd;
                                z = (ip ? a.eo - en : en - a.eo) + a.y1 - a.y2 + a.y3 - a.y4;
                            } else {
                                const float en = (jp ? a.x - vj : vj - a.x) * a.dd;
                                z = (jp ? a.y1 - en : a.y1 + en - a.eo) + a.y3 - a.y4;
                            }
                            D += a.cross ? a.c0 * z : -0.0f;
                        }
                    } else if (KIND != 2) {
                        D += a.y1;
                    }
                    // below KKART+1 (W inside buildings) Q is D over the diagonal;
                    // the chain forms the one at KKART+1 itself
                    if (COMP == 2 && k <= c0.KK) D = (KIND != 0) ? D / a.t : D * a.t;
                    lds_at(sm, sd + 4 * (lane + WAVE * m)) = D;
                }
            }
        }
        lds_barrier();
        // phase 2, beside the recurrences
        float xst[M];
        const StripCol done = c2m;                            // the column of step s-1, before its buffer is reused
        const unsigned od = op;
        if (done.VI >= 0) {
            const int sn = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + done.kend - (done.KK + 1) + lane);
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (done.kend + lane + WAVE * m <= done.VI) xst[m] = lds_at(sm, sn + 4 * WAVE * m);
        }
        located();                                            // ahead of the work: the barrier waits for scalar loads
        if (s + 1 < nsteps) work_up(s + 1, c0);
        c2m = c0; op = o0;
        c0 = c1; o0 = o1;
        if (s + 1 < nsteps) issue(c0, c2, c2j);
        else c0 = none;
        if (done.VI >= 0) {
            gf32 *Xp = (gf32 *)X + (size_t)od + done.kend;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (done.kend + lane + WAVE * m <= done.VI) *(gf32 *)lane_at(Xp + WAVE * m, off_c - base) = xst[m];
        }
        lds_barrier();                                        // the recurrence outputs are ready
    }
    if (c2m.VI >= 0) {
        const float *xn = sm + (size_t)r * rs + (4 + 4 * ((nsteps - 1) & 1)) * len + low - (c2m.KK + 1);
        gf32 *Xp = (gf32 *)X + (size_t)op;
        for (int k = c2m.kend + lane; k <= c2m.VI; k += WAVE) Xp[(unsigned)k] = xn[k];
    }
}

// Pressure sweep on strips (a = j1 outer, b = i1 inner), laid out as
// k_ml_strip.  The QIMP row scratch of a sweep row, which every column of the
// row starts its elimination from and leaves its values in, travels with the
// wavefront through LDS (ring slot (a - oa) mod RING; the rows of a step
// hold consecutive sweep rows): the control wave puts the row the previous strip
// handed over into row 0's slot, each row merges its column's Q, and the control
// wave hands the row on after the last row's merge.
// Chains per column: Q[t] = (A[t]*Q[t+1] + D[t])*T[t] from the top (A = ATP; 3
// dependent operations a level), then N[t] = P[t]*N[t-1] + Q[t] from the bottom (2).
#define RING 16
__device__ __forceinline__ void strip_pdown(float *DQ, const float *A, const float *T, float qtop, int n, int nch, bool part,
                                            int low, const Chunk &a0, const Chunk &t0) {
    int o = chunk_of(n);
    const int top = n - o;
    float qn = qtop;
    Chunk d[2], a[2] = {a0}, t[2] = {t0};
    d[0] = ld_chunk(DQ + o);
    for (int b = 0; b < nch; b += CHK_BLOCK) {
#pragma unroll
        for (int h = 0; h < CHK_BLOCK; ++h) {
            if (b + h >= nch) return;
            const int k = h & 1, m = k ^ 1, on = max(o - CHK, -low);
            d[m] = ld_chunk(DQ + on); a[m] = ld_chunk(A + on); t[m] = ld_chunk(T + on);
            __builtin_amdgcn_sched_barrier(0);
            if (h == 0 && part && b == 0) {
#pragma unroll
                for (int u = CHK - 1; u >= 0; --u) {
                    const float q = (a[k].v[u] * qn + d[k].v[u]) * t[k].v[u];
                    qn = (u >= top) ? qn : q;
                    d[k].v[u] = q;
                }
            } else {
#pragma unroll
                for (int u = CHK - 1; u >= 0; --u) {
                    qn = (a[k].v[u] * qn + d[k].v[u]) * t[k].v[u];
                    d[k].v[u] = qn;
                }
            }
            st_chunk(DQ + o, d[k]);
            o = on;
        }
    }
}
__device__ __forceinline__ void strip_pup(const float *P, const float *Q, float *N, float bottom, int nch, const Chunk &p0) {
    float x = bottom;
    Chunk p[2] = {p0}, q[2];
    q[0] = ld_chunk(Q);
    for (int b = 0; b < nch; b += CHK_BLOCK) {
#pragma unroll
        for (int h = 0; h < CHK_BLOCK; ++h) {
            if (b + h >= nch) return;
            const int k = h & 1, m = k ^ 1;
            p[m] = ld_chunk(P + (h + 1) * CHK); q[m] = ld_chunk(Q + (h + 1) * CHK);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < CHK; ++u) {
                x = p[k].v[u] * x + q[k].v[u];
                q[k].v[u] = x;
            }
            st_chunk(N + h * CHK, q[k]);
        }
        P += CHK_BLOCK * CHK; Q += CHK_BLOCK * CHK; N += CHK_BLOCK * CHK;
    }
}

// raw operands of one column, loaded a step before they are worked up
struct PrRaw {
    float div, t, p, pa, pb;       // DIV / DTIME, TERMP, PIMP, old DPM in the +IS (i) and +JS (j) directions
    float ni, nj;                  // -IS / -JS neighbours as memory holds them
    unsigned long long hw;
};
struct PrIn {
    float div, pa, pb, dz, ni, nj;
    int li, lj;
    bool si, sj;
};

template <int M>
__global__ __launch_bounds__(STRIP_WAVES * WAVE) void k_pressure_strip(const Dom *__restrict__ ds, int IS, int JS, int slot) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];
    extern __shared__ __align__(16) float sm[];
    const int nkp = d.nkp, nii = d.nii, njj = d.njj, nj2 = d.nj2, hcols = njj;
    const int low = strip_low(0), len = strip_len(0, d.nact), rs = strip_stride(9, len);
    const int oa = 2, ia = 2, ob = njj - 1, ib = nii - 1, na = ob - oa + 1;
    const int R = blockDim.x / WAVE - 2;                      // rows of a strip (strip_rows())
    const int nstrip = (ib - ia + R) / R, nsteps = na + R - 1;
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    gi32 *sync = d.sync + SYNC_BLOCK0;
    // per row: D (replaced by Q), then per step parity A, T, P and the new DPM
    float *ring = sm + (size_t)R * rs;                        // [RING][nkp] QIMP row scratch
    float *sdzk = ring + RING * nkp, *satp = sdzk + nkp;      // [nkp] each
    int4 *sinfo = (int4 *)(satp + nkp);                       // [2][16] per row by step parity, for the chain wave
    int *sctl = (int *)(sinfo + 32);
    if (threadIdx.x == 0) sctl[0] = __hip_atomic_fetch_add(&sync[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = threadIdx.x; k < nkp; k += blockDim.x) { sdzk[k] = d.dzk[k]; satp[k] = d.atp[k]; }
    __syncthreads();
    const int B = __builtin_amdgcn_readfirstlane(sctl[0]);
    if (B >= nstrip) return;                                  // uniform over the workgroup
    const unsigned tag = hand_tag(d, 0);
    gu64 *hand = (gu64 *)d.hand, *handq = hand + d.hand_words;        // new DPM, row scratch: [strip][njj][nkp]
    const int4 *meta = (const int4 *)d.meta;
    HandWait hwait{d.sync, wall_clock64() + STRIP_TIMEOUT_TICKS, false};
    const bool send = B + 1 < nstrip;
    if (r == R) {                                             // chain wave, as in k_ml_strip
        __builtin_amdgcn_s_setprio(3);
        float *L = sm + (size_t)(lane < R ? lane : 0) * rs + low;
        // The last row's new values, which the next strip waits for, go out while
        // the rows assemble the next step: this wave waits for no load, so the
        // stores cost it their issue only.
        const float *xl = sm + (size_t)(R - 1) * rs + 4 * len + low;
        gu64 *h = hand + ((size_t)B * hcols - R) * nkp;       // + s*nkp: the last row's column of step s - 1
        int n = 0, top = 0;
        auto send_last = [&](int s) {
            const int nl = __builtin_amdgcn_readlane(n, R - 1), kl = __builtin_amdgcn_readlane(top, R - 1) - nl;
            if (send)
                for (int t = lane; t < nl; t += WAVE) hand_put(h + (size_t)s * nkp + kl + t, xl[4 * ((s - 1) & 1) * len + t], tag);
        };
        lds_barrier();                                        // the control wave's data of step 0
        for (int s = 0; s < nsteps; ++s) {
            // levels (0: no column), chunks | partial chunk << 16, VI + 1, DPM below the column
            const int4 si = sinfo[(s & 1) * 16 + (lane & 15)];
            send_last(s);
            n = lane < R ? si.x : 0;
            top = si.z;
            const int fm = __builtin_amdgcn_readfirstlane(si.y);
            const float *rq = ring + (size_t)((s - lane) & (RING - 1)) * nkp + top;
            float *Lp = L + (1 + 4 * (s & 1)) * len;
            const int o = chunk_of(n);
            const Chunk a0 = ld_chunk(Lp + o), t0 = ld_chunk(Lp + len + o), p0 = ld_chunk(Lp + 2 * len);
            lds_barrier();                                    // the rows' sources are assembled
            if (n > 0) {
                strip_pdown(L, Lp, Lp + len, *rq, n, fm & 0xffff, (fm >> 16) != 0, low, a0, t0);
                strip_pup(Lp + 2 * len, L, Lp + 3 * len, __int_as_float(si.w), fm & 0xffff, p0);
            }
            lds_barrier();                                    // the recurrences are done
        }
        send_last(nsteps);
        lds_barrier();                                        // the last columns are merged into the ring
        return;
    }
    if (r == R + 1) {                                         // control wave
        __builtin_amdgcn_s_setprio(2);
        const int b = ia + B * R + lane;
        const bool lane_ok = lane < R && b <= ib;
        int cidx = ((IS == -1) ? nii - b + 1 : b) * nj2 + ((JS == -1) ? njj - oa + 1 : oa) - lane * JS;
        // lane r's column: its metadata is requested two steps ahead, the DPM below
        // it one step ahead
        auto meta_at = [&](int s) {
            const int l = s - lane;
            int4 m = make_int4(0, -1, 0, 0);
            if (lane_ok && l >= 0 && l < na) m = ldg4i((const DomG::P<const int4>)meta + cidx);
            cidx += JS;
            return m;
        };
        int4 mq = meta_at(0), mb = make_int4(0, -1, 0, 0);
        float bot = 0.0f;
        auto advance = [&](int s) {                           // metadata of step s arrives, its DPM is requested
            const int c = cidx - JS;
            mb = mq;
            mq = meta_at(s + 1);
            bot = 0.0f;
            if (mb.z & 0x10000) bot = d.dpm[(size_t)c * nkp + mb.x];
        };
        auto info = [&](int s) {
            const int n = (mb.z & 0x10000) ? mb.y - mb.x : 0;
            const int part = __any((n & (CHK - 1)) != 0) ? 0x10000 : 0;
            const int fm = row_max((n + CHK - 1) >> 3);
            if (lane < 16) sinfo[(s & 1) * 16 + lane] = make_int4(n, fm | part, n > 0 ? mb.y + 1 : 0, __float_as_int(bot));
        };
        // row 0's row scratch, as the previous strip hands it over: the words of a
        // step are requested a step ahead, two groups of 64 levels at once
        unsigned long long qw[2] = {0, 0}, qn[2];
        auto qrequest = [&](int s) {
#pragma unroll
            for (int m = 0; m < 2; ++m)
                if (B > 0 && s < na && lane + WAVE * m < nkp)
                    qw[m] = hand_get(handq + ((size_t)(B - 1) * hcols + s) * nkp + lane + WAVE * m);
        };
        auto qstore = [&](int s) {
            if (s >= na) return;
            float *rq = ring + (size_t)(s & (RING - 1)) * nkp;
            const gu64 *hq = handq + ((size_t)(B - 1) * hcols + s) * nkp;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int k = lane + WAVE * m;
                if (B > 0) hwait.wait(hq + k, k < nkp, tag, qn[m]);
                if (k < nkp) rq[k] = B > 0 ? __uint_as_float((unsigned)qn[m]) : 0.0f;
            }
            for (int k = lane + 2 * WAVE; k - lane < nkp; k += WAVE) {
                unsigned long long w = 0;
                if (B > 0) hwait.wait(hq + k, k < nkp, tag, w);
                if (k < nkp) rq[k] = __uint_as_float((unsigned)w);
            }
        };
        advance(0);
        qrequest(0);
        info(0);
        qn[0] = qw[0]; qn[1] = qw[1];
        qstore(0);
        advance(1);
        qrequest(1);
        gu64 *h = handq + ((size_t)B * hcols - R) * nkp;      // + s*nkp: the last row's row scratch of step s - 1
        auto send_ring = [&](int s) {
            const int l = s - R;
            if (send && l >= 0 && l < na) {
                const float *rq = ring + (size_t)(l & (RING - 1)) * nkp;
                for (int k = lane; k < nkp; k += WAVE) hand_put(h + (size_t)s * nkp + k, rq[k], tag);
            }
        };
        lds_barrier();
        for (int s = 0; s < nsteps; ++s) {
            // the loads of the step before arrive and the next are issued ahead of
            // this step's stores: a wait for a load covers the stores before it
            info(s + 1);
            qn[0] = qw[0]; qn[1] = qw[1];
            advance(s + 2);
            qrequest(s + 2);
            lds_barrier();
            qstore(s + 1);
            send_ring(s);
            lds_barrier();
        }
        lds_barrier();
        send_ring(nsteps);
        return;
    }
    const int b = ia + B * R + r;
    const bool row_ok = b <= ib, from_prev = r == 0 && B > 0, has_i = r > 0 || B > 0, jp = JS == 1;
    const float DXK = d.dxk, DYK = d.dyk, relaxp = d.relaxp;
    // a division by a power of two is a multiplication by its reciprocal, bit for bit
    const float rx = 1.0f / DXK, ry = 1.0f / DYK;
    const bool p2 = (((__float_as_uint(DXK) | __float_as_uint(DYK)) & 0x7fffffu) == 0) && fabsf(log2f(DXK)) < 100.0f &&
                    fabsf(log2f(DYK)) < 100.0f;
    const int rowb = 4 * r * rs;
    const gf32 *DPM = d.dpm, *DIV = d.div, *PT = d.ptab[IS == 1 ? 0 : 1], *TT = d.ttab[IS == 1 ? 0 : 1];
    gf32 *DPMNEW = d.dpmnew;
    int l2 = -r;
    int cidx2 = ((IS == -1) ? nii - b + 1 : b) * nj2 + ((JS == -1) ? njj - oa + 1 : oa) - r * JS;
    int4 m2, m2i;
    auto request = [&]() {                                    // metadata of the next column and its -IS neighbour
        m2 = m2i = make_int4(0, -1, 0, 0);
        if (row_ok && l2 >= 0 && l2 < na) {
            m2 = ldc4i(meta + cidx2);
            if (has_i) m2i = ldc4i(meta + (cidx2 - IS * nj2));
        }
        ++l2;
        cidx2 += JS;
    };
    const unsigned fi = 4u * (unsigned)nj2 * (unsigned)nkp, fj = 4u * (unsigned)nkp, base = fi + fj;
    const unsigned off_l = 4u * lane, off_c = base + off_l, off_a = IS == 1 ? off_c + fi : off_c - fi;
    const unsigned off_b = jp ? off_c + fj : off_c - fj, off_i = IS == 1 ? off_c - fi : off_c + fi;
    const unsigned off_j = jp ? off_c - fj : off_c + fj, off_h = 8u * lane;
    const StripCol none{0, -1, 0, 0, 0};
    StripCol c0 = none, c1 = none, c1i = none, c2m = none, c2, c2i;   // steps s, s+1 (and its -IS neighbour), s-1, s+2
    unsigned o0 = 0, o1 = 0, op = 0;
    PrRaw raw[M];
    PrIn in[M];
    float dn[M] = {}, pmax = 0.0f, pmin = 0.0f;
    auto located = [&]() {
        c2 = strip_col<0>(m2);                                // kend unused
        c2i = strip_col<0>(m2i);
        request();
    };
    auto issue = [&](const StripCol &p, const StripCol &cn, const StripCol &cni) {
        c1 = cn;
        c1i = cni;
        const int ci = cidx2 - 2 * JS, l = l2 - 2;
        if (c1.VI < 0) return;
        o1 = (unsigned)ci * (unsigned)nkp;
        const size_t o = (size_t)o1 + c1.KK + 1;
        const gf32 *Xl = DPM + o - (base >> 2);
        const gf32 *H = (const gf32 *)(hand + ((size_t)(B - 1) * hcols + l) * nkp + c1.KK + 1);
        const bool old_j = p.KK > c1.KK || p.VI < c1.VI, old_i = c1i.KK > c1.KK || c1i.VI < c1.VI;
        const int n = c1.VI - c1.KK;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (lane + WAVE * m < n) {
                PrRaw &q = raw[m];
                q.div = *lane_at(DIV + o + m * WAVE, off_l);
                q.t = *lane_at(TT + o + m * WAVE, off_l);
                q.p = *lane_at(PT + o + m * WAVE, off_l);
                const gf32 *Xm = Xl + m * WAVE;
                q.pa = *lane_at(Xm, off_a);
                q.pb = *lane_at(Xm, off_b);
                if (old_i) q.ni = *lane_at(Xm, off_i);
                if (old_j) q.nj = *lane_at(Xm, off_j);
                if (from_prev) q.hw = hand_get((const gu64 *)lane_at(H + m * WAVE * 2, off_h));
            }
        }
    };
    auto work_up = [&](int s, const StripCol &p) {
        const StripCol &c = c1;
        if (c.VI < 0) return;
        const int sc = rowb + 4 * ((1 + 4 * (s & 1)) * len + low), l4 = 4 * len;
        const int sj = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + c.KK - p.KK);
        const int si = rowb - 4 * rs + 4 * ((8 - 4 * (s & 1)) * len + low + c.KK - c1i.KK);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int t4 = 4 * (lane + WAVE * m), k = c.KK + 1 + lane + WAVE * m;
            PrRaw &q = raw[m];
            PrIn &a = in[m];
            if (k <= c.VI) {
                lds_at(sm, sc + t4) = satp[k];
                lds_at(sm, sc + l4 + t4) = q.t;
                lds_at(sm, sc + 2 * l4 + t4) = q.p;
                a.dz = sdzk[k];
                a.div = q.div; a.pa = q.pa; a.pb = q.pb; a.ni = q.ni; a.nj = q.nj;
                a.sj = k > p.KK && k <= p.VI;
                a.si = k > c1i.KK && k <= c1i.VI;
                a.lj = a.sj ? sj + t4 : 0;
                a.li = a.si ? si + t4 : 0;
            }
        }
        if (from_prev) {
            const gu64 *h = hand + ((size_t)(B - 1) * hcols + (s - r)) * nkp;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = c.KK + 1 + lane + WAVE * m;
                const bool need = k <= c.VI && k > c1i.KK && k <= c1i.VI;
                hwait.wait(h + k, need, tag, raw[m].hw);
                if (need) in[m].ni = __uint_as_float((unsigned)raw[m].hw);
                in[m].si = false;                             // the value is in ni
                in[m].li = 0;
            }
        }
    };
    // merges the Q of the column of step s into its ring slot
    auto merge = [&](int s, const StripCol &c) {
        if (c.VI < 0) return;
        float *rq = ring + (size_t)((s - r) & (RING - 1)) * nkp + c.KK + 1;
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (lane + WAVE * m < c.VI - c.KK) rq[lane + WAVE * m] = lds_at(sm, rowb + 4 * (low + lane + WAVE * m));
    };
    request();
    located();
    issue(none, c2, c2i);
    located();
    work_up(0, none);
    c0 = c1; o0 = o1;
    issue(c0, c2, c2i);
    lds_barrier();                                            // the control wave's data of step 0
    for (int s = 0; s < nsteps; ++s) {
        // phase 1: the previous column's Q to the ring, the sources of step s over it
        merge(s - 1, c2m);
        if (c0.VI >= 0) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (lane + WAVE * m < c0.VI - c0.KK) {
                    const PrIn &a = in[m];
                    float vi = lds_at(sm, a.li), vj = lds_at(sm, a.lj);
                    vi = a.si ? vi : a.ni;
                    vj = a.sj ? vj : a.nj;
                    const float sx = vi + a.pa, sy = (jp ? vj : a.pb) - (jp ? a.pb : vj);
                    float qx, qy;
                    if (p2) { qx = sx * rx; qy = sy * ry; }
                    else { qx = sx / DXK; qy = sy / DYK; }
                    lds_at(sm, rowb + 4 * (low + lane + WAVE * m)) = a.div + qx * DYK * a.dz + qy * DXK * a.dz;
                }
            }
        }
        lds_barrier();
        // phase 2, beside the recurrences
        float xst[M], dnst[M];
        const StripCol done = c2m;                            // the column of step s-1, before its buffer is reused
        const unsigned od = op;
        if (done.VI >= 0) {
            const int sn = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + lane);
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < done.VI - done.KK) {
                    xst[m] = lds_at(sm, sn + 4 * WAVE * m);
                    dnst[m] = dn[m];
                }
        }
        located();
        if (s + 1 < nsteps) work_up(s + 1, c0);
        c2m = c0; op = o0;
        c0 = c1; o0 = o1;
        if (s + 1 < nsteps) issue(c0, c2, c2i);
        else c0 = none;
        if (c2m.VI >= 0) {                                    // DPMNEW of the column of step s, for its store
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < c2m.VI - c2m.KK) dn[m] = *lane_at(DPMNEW + (size_t)op + c2m.KK + 1 + m * WAVE, off_l);
        }
        if (done.VI >= 0) {
            const size_t o = (size_t)od + done.KK + 1;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < done.VI - done.KK) {
                    pmax = xst[m] > pmax ? xst[m] : pmax;
                    pmin = xst[m] < pmin ? xst[m] : pmin;
                    *(gf32 *)lane_at(DPM + o + m * WAVE, off_l) = xst[m];
                    *(gf32 *)lane_at(DPMNEW + o + m * WAVE, off_l) = dnst[m] + relaxp * xst[m];
                }
        }
        lds_barrier();                                        // the recurrence outputs are ready
    }
    merge(nsteps - 1, c2m);
    lds_barrier();
    if (c2m.VI >= 0) {
        const size_t o = (size_t)op + c2m.KK + 1;
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (lane + WAVE * m < c2m.VI - c2m.KK) {
                const float x = sm[(size_t)r * rs + (4 + 4 * ((nsteps - 1) & 1)) * len + low + lane + WAVE * m];
                pmax = x > pmax ? x : pmax;
                pmin = x < pmin ? x : pmin;
                ((gf32 *)DPM)[o + lane + WAVE * m] = x;
                DPMNEW[o + lane + WAVE * m] = dn[m] + relaxp * x;
            }
    }
    // residual: the largest |old DPM - quantised new DPM|.  The divergence pass has
    // zeroed the old DPM of every cell, and the quantisation is monotonic, so it
    // is taken from the extreme new values, once per lane instead of per cell.
    const float ra = (float)fabs((double)conv_to_int((double)pmax * d.frund) / d.frund);
    const float rb = (float)fabs((double)conv_to_int((double)pmin * d.frund) / d.frund);
    float rmax = ra > rb ? ra : rb;
    for (int off = WAVE / 2; off > 0; off >>= 1) {
        float other = __shfl_xor(rmax, off);
        rmax = other > rmax ? other : rmax;
    }
    const int rsl = slot - d.iter_off;                // this situation's residual slot
    if (lane == 0 && rmax > 0.0f && slot >= 0 && rsl >= 0 && rsl < d.resid_cap) atomicMax((unsigned *)&d.resid[rsl], __float_as_uint(rmax));
}

static inline int lds_limit(const void *kern, size_t bytes);
// ------------------------------------------------------------------------
// Strips for sweeps whose column system is two first-order recurrences (the
// diagnostic pressure sweep, the transposed momentum sweep): the strip and
// hand-off scheme of k_ml_strip, with the LDS arrays of a row indexed by the level
// itself and 0 outside a column's levels, so that a neighbour's value needs no
// offset and the recurrences of all rows run over the same chunks.  R row waves
// own a sweep row each, wave R runs the recurrences (lane = row) and hands the
// last row's results on; the steps and phases are those of k_ml_strip, without
// a control wave: a row leaves its column's levels in LDS a step ahead.  Bound by
// the recurrences.  OP supplies the operands and the recurrences (DgOp, MomOp,
// PrAdjOp); M: 64-level groups of a column.  OP::SCRATCH: each step has a row of
// values by level that its columns, one after another along the rows, take (and
// clear) at their own levels and add to at the level above them; it starts at 0.
// ------------------------------------------------------------------------
struct LineSweep {
    int ni, nj;                  // rows, steps of the sweep
    int c0, di, dj;              // column index of (0, 0), its change per row and per step
    int nk;                      // levels of a stored column
    int *sync;                   // [0] error flag, [1] tag base, [ticket] 0 before the launch
    int ticket, kind;            // kind: names the sweep in the tag
    unsigned long long *hand;    // [strips][nj][nk]
    unsigned long long *handq;   // [strips][nj][nk], the row scratch of the OPs that have one
};
struct LineCol { int lo, hi, x; };                             // its levels (lo > hi: none) and the OP's own datum
typedef int __attribute__((address_space(4))) ci32;
__host__ __device__ inline int line_len(int nk) { return (nk + 2 * CHK - 1) / CHK * CHK; }      // one spare chunk
template <class OP>
__host__ __device__ inline int line_arrays() { return 3 + 2 * OP::NBUF + OP::SCRATCH; }
template <class OP>
static size_t line_lds(int nk, int rows) {
    const int len = line_len(nk);
    return sizeof(float) * ((size_t)rows * strip_stride(line_arrays<OP>(), len) + (size_t)(OP::NTAB + OP::SCRATCH * RING) * len) + 32 * sizeof(int4) + 16;
}
template <class OP, int M>
__global__ __launch_bounds__(STRIP_WAVES * WAVE) void k_line_strip(OP op, LineSweep w) {
    extern __shared__ __align__(16) float sm[];
    const int nk = w.nk, len = line_len(nk), rs = strip_stride(line_arrays<OP>(), len);
    const int R = blockDim.x / WAVE - 1;
    const int nstrip = (w.ni + R - 1) / R, nsteps = w.nj + R - 1;
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    gi32 *sync = (gi32 *)w.sync;
    // per row: D (or what the recurrences make of it), the results of even and odd
    // steps, the operands of even and odd steps, the scratch values taken
    float *tab = sm + (size_t)R * rs;                         // [NTAB][len] operands that depend on the level alone
    float *ring = tab + OP::NTAB * len;                       // [RING][len] row scratch of a step (slot: step mod RING)
    int4 *sinfo = (int4 *)(ring + OP::SCRATCH * RING * len);             // [2][16] levels of the rows' columns by step parity
    int *sctl = (int *)(sinfo + 32);
    const LineCol none{1 << 20, -1, 0};
    if (threadIdx.x == 0) sctl[0] = __hip_atomic_fetch_add(&sync[w.ticket], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < 32) sinfo[threadIdx.x] = make_int4(none.lo, none.hi, 0, 0);
    for (int k = threadIdx.x; k < OP::NTAB * len; k += blockDim.x) tab[k] = (k % len < nk) ? op.table(k / len, k % len) : 0.0f;
    __syncthreads();
    const int B = __builtin_amdgcn_readfirstlane(sctl[0]);
    if (B >= nstrip) return;                                  // uniform over the workgroup
    const unsigned tag = 8u * (unsigned)sync[1] + (unsigned)w.kind;
    gu64 *hand = (gu64 *)w.hand, *handq = (gu64 *)w.handq;
    if (r == R) {                                             // chain wave
        __builtin_amdgcn_s_setprio(3);
        float *L = sm + (size_t)(lane < R ? lane : 0) * rs;
        const float *xl = sm + (size_t)(R - 1) * rs + len;
        gu64 *h = hand + ((size_t)B * w.nj - R) * nk;         // + s*nk: the last row's column of step s - 1
        gu64 *hq = handq + ((size_t)B * w.nj - R) * nk;
        const bool send = B + 1 < nstrip;
        int lo = none.lo, hi = none.hi;
        auto send_last = [&](int s) {
            if (!send || s < R) return;                       // l = s - R is a step of the last row
            const int a = __builtin_amdgcn_readlane(lo, R - 1), b = __builtin_amdgcn_readlane(hi, R - 1);
            float v[M];
#pragma unroll
            for (int m = 0; m < M; ++m) v[m] = xl[((s - 1) & 1) * len + min(lane + WAVE * m, len - 1)];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = lane + WAVE * m;
                if (k < nk) hand_put(h + (size_t)s * nk + k, (k >= a && k <= b) ? v[m] : 0.0f, tag);
                if (OP::SCRATCH && k < nk) hand_put(hq + (size_t)s * nk + k, ring[((s - R) & (RING - 1)) * len + k], tag);
            }
        };
        lds_barrier();                                        // the rows' operands and levels of step 0
        for (int s = 0; s < nsteps; ++s) {
            const int4 si = sinfo[(s & 1) * 16 + (lane & 15)];
            send_last(s);
            lo = lane < R ? si.x : none.lo;
            hi = lane < R ? si.y : none.hi;
            const bool on = lo <= hi;
            // chunks of the lowest bottom, the highest bottom and the highest top
            const int NC = len / CHK;
            const int clo = NC - __builtin_amdgcn_readfirstlane(row_max(on ? NC - lo / CHK : 0));
            const int chi = __builtin_amdgcn_readfirstlane(row_max(on ? lo / CHK : 0));
            const int ct = __builtin_amdgcn_readfirstlane(row_max(on ? (hi + OP::SCRATCH) / CHK : 0));
            lds_barrier();                                    // the rows' sources are assembled
            if (on) {
                op.chain(L, L + (1 + (s & 1)) * len, L + (3 + (s & 1) * OP::NBUF) * len, tab, len, lo, clo, chi, ct);
                if (OP::SCRATCH) ring[((s - lane) & (RING - 1)) * len + hi + 1] += L[hi + 1];
            }
            lds_barrier();                                    // the recurrences are done
        }
        send_last(nsteps);
        return;
    }
    const int b = B * R + r;
    const bool row_ok = b < w.ni, from_prev = r == 0 && B > 0;
    HandWait hwait{sync, wall_clock64() + STRIP_TIMEOUT_TICKS, false};
    const int rowb = 4 * r * rs, c00 = w.c0 + b * w.di;
    LineCol q2 = none, c2 = none, c1 = none, c0 = none, cm = none;    // requested, steps s+2, s+1, s, s-1
    int l2 = -r - 1;                                          // step (of this row) q2 belongs to
    typename OP::Raw raw[M];
    typename OP::In in[M] = {};
    unsigned long long hw[M], hs[M];
    int kb[M];                                                // byte offsets of the lane's levels in an array
#pragma unroll
    for (int m = 0; m < M; ++m) kb[m] = 4 * min(lane + WAVE * m, len - 1);
    float vin[M] = {};                                        // row 0: the new values of the previous strip's last row
    auto located = [&]() {                                    // q2 arrives, the next is requested
        c2 = q2;
        ++l2;
        q2 = none;
        if (row_ok && l2 >= 0 && l2 < w.nj) q2 = op.levels(c00 + l2 * w.dj);
    };
    auto issue = [&]() {                                      // loads of the column at c2, l = l2 - 1
        c1 = c2;
        const int l = l2 - 1, c = c00 + l * w.dj;
        if (OP::SCRATCH && from_prev && l >= 0 && l < w.nj)
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < nk) hs[m] = hand_get(handq + ((size_t)(B - 1) * w.nj + l) * nk + lane + WAVE * m);
        if (c1.lo > c1.hi) return;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int k = lane + WAVE * m;
            if (k >= c1.lo && k <= c1.hi) op.load(raw[m], c, w.di, w.dj, k);
            if (from_prev && k < nk) hw[m] = hand_get(hand + ((size_t)(B - 1) * w.nj + l) * nk + k);
        }
    };
    auto work_up = [&](int s) {                               // c1 is the column of step s
        if (lane == 0) sinfo[(s & 1) * 16 + r] = make_int4(c1.lo, c1.hi, 0, 0);
        if (OP::SCRATCH && r == 0 && s < w.nj)                // the scratch of step s as the rows before this strip left it
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = lane + WAVE * m;
                if (B > 0) hwait.wait(handq + ((size_t)(B - 1) * w.nj + s) * nk + k, k < nk, tag, hs[m]);
                if (k < len) ring[(s & (RING - 1)) * len + k] = (B > 0 && k < nk) ? __uint_as_float((unsigned)hs[m]) : 0.0f;
            }
        if (c1.lo > c1.hi) return;
        const int ob = rowb + 4 * (3 + (s & 1) * OP::NBUF) * len;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int k = lane + WAVE * m;
            const bool on = k >= c1.lo && k <= c1.hi;
            if (k < len) op.stage(raw[m], in[m], on, k, &lds_at(sm, ob + 4 * k), len, tab);
        }
        if (from_prev) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = lane + WAVE * m;
                hwait.wait(hand + ((size_t)(B - 1) * w.nj + (s - r)) * nk + k, k < nk, tag, hw[m]);
                vin[m] = k < nk ? __uint_as_float((unsigned)hw[m]) : 0.0f;
            }
        }
    };
    located();                                                // requests step 0's column
    located();
    issue();
    located();
    work_up(0);
    c0 = c1;
    issue();
    lds_barrier();
    for (int s = 0; s < nsteps; ++s) {
        const int xn = rowb + 4 * (2 - (s & 1)) * len;        // new values of step s - 1: own, row r - 1's at xn - 4*rs
        if (c0.lo <= c0.hi) {                                 // phase 1
            LineCol ci = none;
            const int xi = xn - (r > 0 ? 4 * rs : 0);
            if (r > 0) {
                const int4 si = sinfo[((s + 1) & 1) * 16 + r - 1];
                ci.lo = si.x;
                ci.hi = si.y;
            }
            float vi[M], vj[M];                               // all reads ahead of the operations, without branches
#pragma unroll
            for (int m = 0; m < M; ++m) {
                vi[m] = lds_at(sm, xi + kb[m]);
                vj[m] = lds_at(sm, xn + kb[m]);
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = lane + WAVE * m;
                const float a = (k >= ci.lo && k <= ci.hi) ? vi[m] : vin[m], b = (k >= cm.lo && k <= cm.hi) ? vj[m] : 0.0f;
                const float d = op.source(in[m], k, c0, a, b);
                const bool on = k >= c0.lo && k <= c0.hi;
                if (k < len) lds_at(sm, rowb + 4 * k) = on ? d : 0.0f;
                if (OP::SCRATCH && k < len) {
                    float *q = ring + ((s - r) & (RING - 1)) * len + k;
                    lds_at(sm, rowb + 4 * ((3 + 2 * OP::NBUF) * len + k)) = on ? *q : 0.0f;
                    if (on) *q = 0.0f;
                }
            }
        }
        lds_barrier();
        // phase 2, beside the recurrences
        float xst[M];
        const LineCol done = cm;
        const int cd = c00 + (s - 1 - r) * w.dj;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int k = lane + WAVE * m;
            if (k >= done.lo && k <= done.hi) xst[m] = lds_at(sm, xn + 4 * k);
        }
        located();
        if (s + 1 < nsteps) work_up(s + 1);
        cm = c0;
        c0 = s + 1 < nsteps ? c1 : none;
        if (s + 1 < nsteps) issue();
        if (done.lo <= done.hi)
#pragma unroll
            for (int m = 0; m < M; ++m) op.store(cd, lane + WAVE * m, done, xst[m]);
        lds_barrier();
    }
    if (cm.lo <= cm.hi) {
        const int cd = c00 + (nsteps - 1 - r) * w.dj, xn = rowb + 4 * (1 + ((nsteps - 1) & 1)) * len;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int k = lane + WAVE * m;
            op.store(cd, k, cm, k < len ? lds_at(sm, xn + 4 * k) : 0.0f);
        }
    }
}
// rows of a strip: as strip_rows() for one situation
static inline int line_rows(int ni) { return ni > 40 ? 10 : STRIP_ROWS_MIN; }
template <class OP, int M>
static int launch_line(const OP &op, const LineSweep &w, hipStream_t s) {
    const int rows = line_rows(w.ni);
    const size_t shm = line_lds<OP>(w.nk, rows);
    if (lds_limit((const void *)k_line_strip<OP, M>, shm)) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL((k_line_strip<OP, M>), dim3((w.ni + rows - 1) / rows), dim3((rows + 1) * WAVE), shm, s, op, w);
    return 0;
}

static inline int ndiag(int oa, int ob, int ia, int ib) { return (ob - oa) + (ib - ia) + 1; }
static inline int diag_len(int t, int oa, int ob, int ia, int ib) {
    int nb = ib - ia;
    int amin = oa + t - nb > oa ? oa + t - nb : oa;
    int amax = ob < oa + t ? ob : oa + t;
    return amax - amin + 1;
}

// ------------------------------------------------------------------------
// Diagnostic post-pass: DiagnosticFlowfield.Calculate (DiagnosticFlowfield.cs:
// 24-436) and the final vertical-velocity mass adjustment of MicroscaleFlat
// (MicroscaleFlat.cs:388-462) or MicroscaleTerrain (MicroscaleTerrain.cs:
// 862-933).  It works on full-height columns (levels 0..NKK+1), in its own
// arrays; one situation per launch, passed by value.
// ------------------------------------------------------------------------
__device__ __forceinline__ size_t dg3(const DiagArgs &g, int i, int j) { return ((size_t)i * g.nj2 + j) * (size_t)g.nkh; }

// DPM = 0 for i in [1,NII], j in [1,NJJ], k in [1,NKK+1] (DiagnosticFlowfield.cs:40-49);
// the columns the sweep visits from k = 0, where the sweep writes 0
__global__ void k_dg_zero(DiagArgs g) {
    int c = blockIdx.x, i = 1 + c / g.njj, j = 1 + c % g.njj;
    if (i > g.nii) return;
    size_t o = dg3(g, i, j);
    const bool inner = i > 1 && i < g.nii && j > 1 && j < g.njj;
    for (int k = (inner ? 0 : 1) + threadIdx.x; k <= g.nkk + 1; k += blockDim.x) g.dpm[o + k] = 0.0f;
}

// mass divergence of every interior column (:53-80); block = one column
__global__ void k_dg_divergence(DiagArgs g) {
    int nj = g.njj - 2, i = 2 + blockIdx.x / nj, j = 2 + blockIdx.x % nj;
    int KK = g.kk[(size_t)i * g.nj2 + j];
    size_t o = dg3(g, i, j), oip = dg3(g, i + 1, j), ojp = dg3(g, i, j + 1);
    const float DXK = g.dxk, DYK = g.dyk;
    for (int k = KK + 1 + threadIdx.x; k <= g.nkk - 1; k += blockDim.x) {
        float dz = g.dzk[k];
        float t = (g.uk[o + k] - g.uk[oip + k]) * DYK * dz + (g.vk[o + k] - g.vk[ojp + k]) * DXK * dz;
        g.div[o + k] = (k > KK + 1) ? t + (g.wk[o + k] - g.wk[o + k + 1]) * DXK * DYK : t - g.wk[o + k + 1] * DXK * DYK;
    }
}

// pressure correction of the diagnostic pass (:84-341).  Every column is solved
// from NKK-1 down to KKART+1 and PIMP[NKK] is never written, so TERMP and PIMP at
// level k are the same in every column whose bottom lies below k; at the bottom
// level only ABP (and so PIMP) differs, and there PIMP multiplies DPM[KKART] = 0.
// The host runs that recurrence once (term, p_in); the recurrences left to a
// column are QIMP[k] = (ATP[k] QIMP[k+1] + DIM[k]) TERMP[k] from QIMP[NKK] = 0
// down and DPM[k] = PIMP[k] DPM[k-1] + QIMP[k] from DPM[KKART] = 0 up.  Columns
// outside the sweep hold DPM = 0.  Bound by the 5 dependent operations a level (56
// cycles with their LDS accesses): 5.5 ms a sweep of 397 x 397 columns of 221
// levels, 11.1 ms with one launch per anti-diagonal (4 to 12 rows a strip: within 3%).
struct DgOp {
    enum { NTAB = 4, NBUF = 0, SCRATCH = 0 };                              // tables: ATP, TERMP, PIMP, DZK
    DiagArgs g;
    float rx, ry;                                             // 1 / DXK, 1 / DYK
    int p2, jp;                                               // both powers of two (their reciprocals are exact); JS == 1
    struct Raw { float div, pa, pb; };                        // old DPM in the sweep's directions i and j
    struct In { float div, pa, pb, dz; };
    __device__ __forceinline__ float table(int a, int k) const {
        return a == 0 ? g.atp[k] : a == 1 ? g.term[k] : a == 2 ? g.p_in[k] : g.dzk[k];
    }
    __device__ __forceinline__ LineCol levels(int c) const { return LineCol{((const ci32 *)g.kk)[c] + 1, g.nkk - 1, 0}; }
    __device__ __forceinline__ void load(Raw &q, int c, int di, int dj, int k) const {
        const gf32 *X = (const gf32 *)g.dpm;
        q.div = ((const gf32 *)g.div)[(size_t)c * g.nkh + k];
        q.pa = X[(size_t)(c + di) * g.nkh + k];
        q.pb = X[(size_t)(c + dj) * g.nkh + k];
    }
    __device__ __forceinline__ void stage(const Raw &q, In &a, bool on, int k, float *, int len, const float *tab) const {
        if (!on) return;
        a.div = q.div / g.dtime;
        a.pa = q.pa;
        a.pb = q.pb;
        a.dz = tab[3 * len + k];
    }
    __device__ __forceinline__ float source(const In &a, int, const LineCol &, float vi, float vj) const {
        const float sx = vi + a.pa, sy = (jp ? vj : a.pb) - (jp ? a.pb : vj);
        const float qx = p2 ? sx * rx : sx / g.dxk, qy = p2 ? sy * ry : sy / g.dyk;
        return a.div + qx * g.dyk * a.dz + qy * g.dxk * a.dz;
    }
    __device__ __forceinline__ void chain(float *L, float *N, float *, const float *tab, int len, int lo, int clo, int chi,
                                          int ct) const {
        const float *A = tab, *T = tab + len;
        const int top = g.nkk - 1;
        {
            float q = 0.0f;
            Chunk d[2], a[2], t[2];
            int o = ct * CHK;
            d[0] = ld_chunk(L + o); a[0] = ld_chunk(A + o); t[0] = ld_chunk(T + o);
#pragma unroll
            for (int u = 0; u < CHK; ++u) {                   // Q stays 0 above the top
                d[0].v[u] = o + u > top ? 0.0f : d[0].v[u];
                a[0].v[u] = o + u > top ? 0.0f : a[0].v[u];
            }
            for (int c = ct; c >= clo;) {
#pragma unroll
                for (int h = 0; h < CHK_BLOCK; ++h) {
                    if (c < clo) break;
                    const int k = h & 1, m = k ^ 1, on = max(o - CHK, 0);
                    d[m] = ld_chunk(L + on); a[m] = ld_chunk(A + on); t[m] = ld_chunk(T + on);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = CHK - 1; u >= 0; --u) {
                        q = (a[k].v[u] * q + d[k].v[u]) * t[k].v[u];
                        d[k].v[u] = q;
                    }
                    st_chunk(L + o, d[k]);
                    o = on;
                    --c;
                }
            }
        }
        // up to the chunk of the highest bottom a lane starts when its level comes
        const float *P = tab + 2 * len + clo * CHK, *Q = L + clo * CHK;
        N += clo * CHK;
        float x = 0.0f;
        int c = clo;
        for (; c <= chi; ++c) {
            Chunk p = ld_chunk(P), w = ld_chunk(Q);
#pragma unroll
            for (int u = 0; u < CHK; ++u) {
                x = (c * CHK + u >= lo) ? p.v[u] * x + w.v[u] : 0.0f;
                w.v[u] = x;
            }
            st_chunk(N, w);
            P += CHK; Q += CHK; N += CHK;
        }
        if (c <= ct) strip_pup(P, Q, N, x, ct - c + 1, ld_chunk(P));
    }
    __device__ __forceinline__ void store(int c, int k, const LineCol &q, float x) const {
        if (k >= q.lo && k <= q.hi) ((gf32 *)g.dpm)[(size_t)c * g.nkh + k] = x;
    }
};

// The same sweep with one launch per anti-diagonal and one wave per column, for
// columns of more levels than k_line_strip holds: the lanes build DIM and stage the
// tables in LDS, and lane 0 runs the two recurrences over LDS.
#define DG_UNROLL 8
__global__ __launch_bounds__(WAVE) void k_dg_pressure(DiagArgs g, int t, int IS, int JS) {
    extern __shared__ float sm[];
    int a, b;
    if (!diag_col(t, 2, g.njj - 1, 2, g.nii - 1, blockIdx.x, a, b)) return;
    int j = (JS == -1) ? g.njj - a + 1 : a;
    int i = (IS == -1) ? g.nii - b + 1 : b;
    const int KK = g.kk[(size_t)i * g.nj2 + j];
    const int nkh = g.nkh, top = g.nkk - 1;
    // LDS: DIM, ATP, TERMP, P (then the new DPM) and Q, nkh levels each
    float *sDIM = sm, *sA = sDIM + nkh, *sT = sA + nkh, *sP = sT + nkh, *sQ = sP + nkh;
    size_t o = dg3(g, i, j), oim = dg3(g, i - 1, j), oip = dg3(g, i + 1, j), ojm = dg3(g, i, j - 1), ojp = dg3(g, i, j + 1);
    const float DXK = g.dxk, DYK = g.dyk;
    for (int k = KK + 1 + threadIdx.x; k <= top; k += WAVE) {
        float dz = g.dzk[k];
        sDIM[k] = g.div[o + k] / g.dtime + (g.dpm[oim + k] + g.dpm[oip + k]) / DXK * DYK * dz +
                  (g.dpm[ojm + k] - g.dpm[ojp + k]) / DYK * DXK * dz;
        sA[k] = g.atp[k];
        sT[k] = g.term[k];
        sP[k] = (k > KK + 1) ? g.p_in[k] : g.p_bot[k];
    }
    __syncthreads();
    if (threadIdx.x == 0 && top > KK) {
        // QIMP[k] = (ATP[k] QIMP[k+1] + DIM[k]) TERMP[k], k = top .. KK+1, in blocks
        // of DG_UNROLL levels whose operands are read before the block's chain
        float Qn = 0.0f;
        int k = top;
        for (; k - DG_UNROLL + 1 > KK; k -= DG_UNROLL) {
            float ca[DG_UNROLL], cd[DG_UNROLL], ct[DG_UNROLL];
#pragma unroll
            for (int u = 0; u < DG_UNROLL; ++u) { ca[u] = sA[k - u]; cd[u] = sDIM[k - u]; ct[u] = sT[k - u]; }
#pragma unroll
            for (int u = 0; u < DG_UNROLL; ++u) {
                Qn = (ca[u] * Qn + cd[u]) * ct[u];
                sQ[k - u] = Qn;
            }
        }
        for (; k > KK; --k) {
            Qn = (sA[k] * Qn + sDIM[k]) * sT[k];
            sQ[k] = Qn;
        }
        // DPM[k] = PIMP[k] DPM[k-1] + QIMP[k], k = KK+1 .. top; written over P
        float dprev = 0.0f;
        k = KK + 1;
        for (; k + DG_UNROLL - 1 <= top; k += DG_UNROLL) {
            float cp[DG_UNROLL], cq[DG_UNROLL];
#pragma unroll
            for (int u = 0; u < DG_UNROLL; ++u) { cp[u] = sP[k + u]; cq[u] = sQ[k + u]; }
#pragma unroll
            for (int u = 0; u < DG_UNROLL; ++u) {
                dprev = cp[u] * dprev + cq[u];
                sP[k + u] = dprev;
            }
        }
        for (; k <= top; ++k) {
            dprev = sP[k] * dprev + sQ[k];
            sP[k] = dprev;
        }
    }
    __syncthreads();
    // DPM[0] = 0 and DPM[k] = 0 up to KKART (the reference writes them each sweep)
    for (int k = threadIdx.x; k <= top; k += WAVE) g.dpm[o + k] = (k > KK) ? sP[k] : 0.0f;
}

// velocity correction without quantisation (:345-410); thread per (column, level)
__global__ void k_dg_correction(DiagArgs g) {
    int nj = g.njj - 2, i = 2 + blockIdx.x / nj, j = 2 + blockIdx.x % nj;
    size_t c = (size_t)i * g.nj2 + j;
    int KK = g.kk[c], KKim = g.kk[c - g.nj2], KKjm = g.kk[c - 1];
    size_t o = dg3(g, i, j), oim = dg3(g, i - 1, j), ojm = dg3(g, i, j - 1);
    const float DXK = g.dxk, DYK = g.dyk, DT = g.dtime;
    for (int k = 1 + threadIdx.x; k < g.nkk; k += blockDim.x) {
        float d0 = g.dpm[o + k];
        float DDPX = g.dpm[oim + k] - d0;
        float DDPY = g.dpm[ojm + k] - d0;
        float DDPZ = (k > KK + 1) ? g.dpm[o + k - 1] - d0 : 0.0f;
        g.uk[o + k] = (KK < k && KKim < k) ? g.uk[o + k] + DDPX / DXK * DT : 0.0f;
        g.vk[o + k] = (KK < k && KKjm < k) ? g.vk[o + k] + DDPY / DYK * DT : 0.0f;
        g.wk[o + k] = (KK + 1 < k) ? g.wk[o + k] + DDPZ * 2 / (g.dzk[k] + g.dzk[k - 1]) * DT : 0.0f;
    }
}

// vertical velocity from the mass balance of each cell, serial in k; thread per column
__global__ void k_dg_wmass(DiagArgs g) {
    int nj = g.njj - 2, ncol = (g.nii - 2) * nj;
    int cidx = blockIdx.x * blockDim.x + threadIdx.x;
    if (cidx >= ncol) return;
    int i = 2 + cidx / nj, j = 2 + cidx % nj;
    size_t c = (size_t)i * g.nj2 + j;
    if (!g.terrain && !(g.level <= 1 || g.adv[c] == 0)) return;
    const float DXK = g.dxk, DYK = g.dyk, DSN = g.terrain ? g.dyk : g.dxk;
    int KK = g.kk[c], KKim = g.kk[c - g.nj2], KKip = g.kk[c + g.nj2], KKjm = g.kk[c - 1], KKjp = g.kk[c + 1];
    size_t o = dg3(g, i, j), oip = dg3(g, i + 1, j), ojp = dg3(g, i, j + 1);
    for (int k = KK + 1; k < g.nkk; ++k) {
        float dz = g.dzk[k];
        float fwo1 = (k <= KKim) ? 0.0f : dz * DYK * g.uk[o + k];
        float fwo2 = (k <= KKip) ? 0.0f : dz * DYK * g.uk[oip + k];
        float fsn1 = (k <= KKjm) ? 0.0f : dz * DSN * g.vk[o + k];
        float fsn2 = (k <= KKjp) ? 0.0f : dz * DSN * g.vk[ojp + k];
        float fbt1 = ((k <= KK + 1) || (k == 1)) ? 0.0f : DXK * DYK * g.wk[o + k];
        g.wk[o + k + 1] = (fwo1 - fwo2 + fsn1 - fsn2 + fbt1) / (DXK * DYK);
    }
}

static bool pow2(float x) { int e; return x > 0.0f && std::frexp(x, &e) == 0.5f && e > -100 && e < 100; }
// 8-byte words of the diagnostic sweep's hand-off buffer; 0: its columns have more
// levels than the strips hold
extern "C" size_t pf_diag_hand(int nii, int njj, int nkh) {
    if (nkh > 4 * WAVE || nii < 3 || njj < 3) return 0;
    const int rows = line_rows(nii - 2);
    return (size_t)((nii - 2 + rows - 1) / rows) * (njj - 2) * nkh;
}
extern "C" int pf_launch_diagnostic(const DiagArgs *ga, int iterations, hipStream_t s) {
    const DiagArgs &g = *ga;
    int ncol = (g.nii - 2) * (g.njj - 2);
    const bool strips = g.hand != nullptr;                    // pf_diag_hand() words, cleared, and DG_SYNC cleared ints
    hipLaunchKernelGGL(k_dg_zero, dim3(g.nii * g.njj), dim3(64), 0, s, g);
    for (int it = 1; it <= iterations; ++it) {
        hipLaunchKernelGGL(k_dg_divergence, dim3(ncol), dim3(64), 0, s, g);
        int IS = 1, JS = 1;
        switch (it % 4) {
            case 0: IS = 1; JS = 1; break;
            case 1: IS = 1; JS = -1; break;
            case 2: IS = -1; JS = -1; break;
            default: IS = -1; JS = 1; break;
        }
        int oa = 2, ob = g.njj - 1, ia = 2, ib = g.nii - 1;
        size_t shm = sizeof(float) * 5 * (size_t)g.nkh;
        if (strips) {
            const int i0 = IS == -1 ? ib : ia, j0 = JS == -1 ? ob : oa;
            const DgOp op{g, 1.0f / g.dxk, 1.0f / g.dyk, pow2(g.dxk) && pow2(g.dyk), JS == 1};
            const LineSweep w{ib - ia + 1, ob - oa + 1, i0 * g.nj2 + j0, IS * g.nj2, JS, g.nkh, g.sync, 1 + it, it, g.hand, nullptr};
            const int e = g.nkh <= 2 * WAVE ? launch_line<DgOp, 2>(op, w, s) : launch_line<DgOp, 4>(op, w, s);
            if (e) return e;
        } else
            for (int t = 0; t < ndiag(oa, ob, ia, ib); ++t)
                hipLaunchKernelGGL(k_dg_pressure, dim3(diag_len(t, oa, ob, ia, ib)), dim3(WAVE), shm, s, g, t, IS, JS);
        hipLaunchKernelGGL(k_dg_correction, dim3(ncol), dim3(64), 0, s, g);
    }
    hipLaunchKernelGGL(k_dg_wmass, dim3((ncol + 63) / 64), dim3(64), 0, s, g);
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// host-side launchers
// ------------------------------------------------------------------------
// ------------------------------------------------------------------------
// Strip-pipelined TKE sweep (TKE-prognostic-microscale.cs:25-352).
// k_tke_coef writes, for every active cell above KKART, what the sweep's
// in-place neighbours do not touch: the neighbour coefficients AW..AN, the
// remaining source terms, the halves of the two Thomas recurrences that need
// no source (P and its denominator, per level), and the wall function.  The
// strip kernel then only assembles the neighbour terms, runs the two Q
// recurrences and the back-substitution, and writes back.  Record per cell
// (TKE_REC floats, written whole by the first pass): {AW, AS, AE, AN |
// ap0*TURB, PROTURB, PROBOU, ap0*TDISS | EPS source, C1, C2, wall flag | wall
// TURB, wall TDISS, 0, 0}; after the records (at TKE_REC*n3 floats), per cell
// {den1, P1, den2, P2}, written whole by the last pass.
// ------------------------------------------------------------------------
#define TKE_REC 16
__device__ __forceinline__ size_t tke_rec4(const DomG &d) { return (size_t)TKE_REC * (d.nii + 2) * d.nj2 * d.nkp; }
#define TKE_SCOL 16       // ints of column data per column in k_tke_coef

// A block of 4 waves takes COEF_COLS consecutive columns (j fastest); their
// levels KKART+1..VI are laid out one after another and dealt to the 256
// lanes, which compute the cells (tke_cell) and write the first three float4
// of each record and the wall values.  One wave then runs the two P
// recurrences of all COEF_COLS columns at once (lane = column), and the lanes
// write the fourth float4.
__global__ __launch_bounds__(4 * WAVE) void k_tke_coef(const Dom *__restrict__ ds) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    extern __shared__ float sm[];
    const int nkp = d.nkp, nkl = lds_stride(nkp);
    const int lane = threadIdx.x % WAVE;
    const int na = d.nii - 2, nb = d.njj - 2;
    // per column c: A, B1, C1, B2, C2 over k at sm + c*5*nkl, and the column's data
    int *scol = (int *)(sm + 5 * COEF_COLS * nkl);        // [COEF_COLS][TKE_SCOL]
    int *stot = scol + TKE_SCOL * COEF_COLS;
    const int blk = xcd_block((na * nb + COEF_COLS - 1) / COEF_COLS);
    if (blk < 0) return;                                      // uniform over the block
    const int col0 = blk * COEF_COLS;
    if (threadIdx.x < WAVE) {
        int c = lane, n = 0;
        if (c < COEF_COLS) {
            int *sc = scol + c * TKE_SCOL;
            const int col = col0 + c;
            int act = 0;
            if (col < na * nb) {
                const int i = 2 + col / nb, j = 2 + col % nb;
                if (d.adv[c2(d, i, j)] == 1) {
                    const ColInfo q = col_info(d, i, j);
                    const TkeCol t = tke_col(d, i, j);
                    act = 1;
                    n = q.VI - q.KK;
                    sc[0] = q.KK; sc[1] = q.VI; sc[2] = i; sc[3] = j;
                    sc[6] = (q.as ? 1 : 0) | (q.an ? 2 : 0) | (q.aw ? 4 : 0) | (q.ae ? 8 : 0) | (t.cip ? 16 : 0) |
                            (t.cim ? 32 : 0) | (t.cjp ? 64 : 0) | (t.cjm ? 128 : 0);
                    sc[7] = t.kkip; sc[8] = t.kkim; sc[9] = t.kkjp; sc[10] = t.kkjm;
                    sc[11] = __float_as_int(q.cutk); sc[12] = __float_as_int(q.ho);
                }
            }
            sc[5] = act;
        }
        // inclusive prefix sum of the level counts over the lanes
        int incl = n;
        for (int off = 1; off < WAVE; off <<= 1) {
            int v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (c < COEF_COLS) scol[c * TKE_SCOL + 4] = incl - n;
        if (lane == WAVE - 1) stot[0] = incl;
    }
    lds_barrier();
    const int total = stot[0];
    auto column_of = [&](int t) {
        int lo = 0;
        for (int step = COEF_COLS / 2; step > 0; step >>= 1)
            if (scol[(lo + step) * TKE_SCOL + 4] <= t) lo += step;
        return lo;
    };
    for (int t = threadIdx.x; t < total; t += 4 * WAVE) {
        const int c = column_of(t);
        const int *sc = scol + c * TKE_SCOL;
        const int k = sc[0] + 1 + (t - sc[4]);
        ColInfo q;
        q.KK = sc[0]; q.VI = sc[1]; q.i = sc[2]; q.j = sc[3]; q.KSTART = q.KK + 1; q.W = d.simd;
        const int fl = sc[6];
        q.as = fl & 1; q.an = (fl >> 1) & 1; q.aw = (fl >> 2) & 1; q.ae = (fl >> 3) & 1; q.vegp = false;
        q.cutk = __int_as_float(sc[11]); q.ho = __int_as_float(sc[12]); q.cov = q.ht = q.z0s = 0.0f;
        TkeCol tc = tke_col_ptrs(d, q.i, q.j);
        tc.cip = (fl >> 4) & 1; tc.cim = (fl >> 5) & 1; tc.cjp = (fl >> 6) & 1; tc.cjm = (fl >> 7) & 1;
        tc.kkip = sc[7]; tc.kkim = sc[8]; tc.kkjp = sc[9]; tc.kkjm = sc[10];
        const TkeCell e = tke_cell(d, q, tc, k);
        gf32 *r = d.planes + (tc.o + k) * TKE_REC;
        stg4(r, e.AW1, e.AS1, e.AE1, e.AN1);
        stg4(r + 4, e.w1, e.PRO, e.PBO, e.w2);
        stg4(r + 8, e.EPS, e.C1, e.C2, e.wf ? 1.0f : 0.0f);
        stg4(r + 12, e.wt, e.we, 0.0f, 0.0f);
        float *sA = sm + (size_t)c * 5 * nkl;
        sA[k] = e.A; sA[nkl + k] = e.B1; sA[2 * nkl + k] = e.C1; sA[3 * nkl + k] = e.B2; sA[4 * nkl + k] = e.C2;
    }
    lds_barrier();
    if (threadIdx.x < COEF_COLS && scol[threadIdx.x * TKE_SCOL + 5]) {
        // P = B/(A - C*P_prev) above KKART+1, B/A at KKART+1 (the recurrence
        // restarts there; the levels below it do not reach the ones above);
        // den1, P1, den2, P2 replace A, B1, C1, B2
        const int c = threadIdx.x;
        float *__restrict__ A = sm + (size_t)c * 5 * nkl;
        float *__restrict__ B1 = A + nkl, *__restrict__ C1 = B1 + nkl, *__restrict__ B2 = C1 + nkl;
        float *__restrict__ C2 = B2 + nkl;
        const int lo = scol[c * TKE_SCOL + 0] + 1, VI = scol[c * TKE_SCOL + 1];
        float P1 = 0, P2 = 0;
        for (int k = lo; k <= VI; ++k) {
            const float a = A[k];
            float den1 = a, den2 = a;
            if (k > lo) { den1 = a - C1[k] * P1; den2 = a - C2[k] * P2; }
            P1 = B1[k] / den1;
            P2 = B2[k] / den2;
            A[k] = den1; B1[k] = P1; C1[k] = den2; B2[k] = P2;
        }
    }
    lds_barrier();
    for (int t = threadIdx.x; t < total; t += 4 * WAVE) {
        const int c = column_of(t);
        const int *sc = scol + c * TKE_SCOL;
        const int k = sc[0] + 1 + (t - sc[4]);
        const float *sA = sm + (size_t)c * 5 * nkl;
        stg4(d.planes + tke_rec4(d) + (c3(d, sc[2], sc[3]) + k) * 4, sA[k], sA[nkl + k], sA[2 * nkl + k], sA[3 * nkl + k]);
    }
}

// Relaxation-free back-substitution of the TKE sweep from t = n-1 down, chunks
// as in strip_back: X[t] = max(P[t]*X[t+1] + Q[t], floor), or the wall value V[t]
// (already floored) where there is one (V != -1; wall values are not negative),
// X[n] = top; X replaces V.  The reference floors with the double-precision
// Math.Max(x, floor_): floor is floor_ rounded to float, which lies above floor_
// for both of its values, so x is replaced exactly where x < floor, and a NaN
// stays.
#define TKE_NO_WALL (-1.0f)
__device__ __forceinline__ void strip_tke_back(const float *P, const float *Q, float *V, float top, float floor, int n, int nch,
                                               bool part, int low, const Chunk &p0, const Chunk &v0) {
    int o = chunk_of(n);
    const int tl = n - o;
    float up = top;
    Chunk p[2] = {p0}, q[2], v[2] = {v0};
    q[0] = ld_chunk(Q + o);
    for (int b = 0; b < nch; b += CHK_BLOCK) {
#pragma unroll
        for (int h = 0; h < CHK_BLOCK; ++h) {
            if (b + h >= nch) return;
            const int k = h & 1, m = k ^ 1, on = max(o - CHK, -low);
            p[m] = ld_chunk(P + on); q[m] = ld_chunk(Q + on); v[m] = ld_chunk(V + on);
            __builtin_amdgcn_sched_barrier(0);
            const bool sel = h == 0 && part && b == 0;
#pragma unroll
            for (int u = CHK - 1; u >= 0; --u) {
                float x = p[k].v[u] * up + q[k].v[u];
                x = x < floor ? floor : x;
                x = v[k].v[u] != TKE_NO_WALL ? v[k].v[u] : x;
                if (h == 0) up = (sel && u >= tl) ? up : x;
                else up = x;
                v[k].v[u] = x;
            }
            st_chunk(V + o, v[k]);
            o = on;
        }
    }
}

// raw operands of one column of the TKE sweep, loaded a step before they are worked up
struct TkeRaw {
    float4 c0, c1, c2;              // record words 0..11
    float4 c3;                      // den1, P1, den2, P2
    float2 c4;                      // wall TURB, wall TDISS
    float ta, ea, tb, eb;           // old TURB/TDISS in the +IS (a) and +JS (b) directions
    float nit, nie, njt, nje;       // -IS / -JS neighbours as memory holds them
    unsigned long long ht, he;      // row 0: the previous strip's last row
};
struct TkeIn {
    float ai, aj, at, bt, ae, be;   // coefficients of the new neighbours, products of the old ones
    float w1, pro, pbo, w2, eps;
    float nit, nie, njt, nje;
    int li, lj;
    bool si, sj;
};

// Strip sweep of TURB and TDISS, laid out as k_ml_strip (row, chain and control
// waves, two phases a step).  The chain wave runs both recurrences of every row
// at once: lane r TURB of row r, lane 16 + r TDISS of row r.
#define TKE_ARRAYS 18
template <int M>
__global__ __launch_bounds__(STRIP_WAVES * WAVE) void k_tke_strip(const Dom *__restrict__ ds, int IS, int JS) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];                   // situation of this launch slice
    extern __shared__ __align__(16) float sm[];
    const int nkp = d.nkp, nii = d.nii, njj = d.njj, nj2 = d.nj2, hcols = nii;
    const int low = strip_low(0), len = strip_len(0, d.nact), rs = strip_stride(TKE_ARRAYS, len), fs = 9 * len;
    const int oa = 2, ia = 2, ob = nii - 1, ib = njj - 1, na = ob - oa + 1;
    const int R = blockDim.x / WAVE - 2;
    const int nstrip = (ib - ia + R) / R, nsteps = na + R - 1;
    const int r = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    gi32 *sync = d.sync + SYNC_BLOCK0 + (size_t)4 * d.sync_stride;
    // per row, for TURB and (fs further) TDISS: D (replaced by Q), then per step
    // parity C, the denominator, P and the wall value (replaced by the new value)
    int4 *sinfo = (int4 *)(sm + (size_t)R * rs);              // [2][32] per chain lane by step parity
    int *sctl = (int *)(sinfo + 64);
    if (threadIdx.x == 0) sctl[0] = __hip_atomic_fetch_add(&sync[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int B = __builtin_amdgcn_readfirstlane(sctl[0]);
    if (B >= nstrip) return;                                  // uniform over the workgroup
    const unsigned tag = hand_tag(d, 4);
    gu64 *handt = (gu64 *)d.hand, *hande = handt + d.hand_words;      // TURB, TDISS: [strip][nii][nkp]
    const int4 *meta = (const int4 *)d.meta;
    const bool send = B + 1 < nstrip;
    if (r == R) {                                             // chain wave
        __builtin_amdgcn_s_setprio(3);
        const int f = (lane >> 4) & 1, cl = (lane & 15) < R ? lane & 15 : 0;
        float *L = sm + (size_t)cl * rs + f * fs + low;
        const float floor = f ? 0.0000001f : 0.001f;
        // the last row's new values go out while the rows assemble the next step
        const float *xl = sm + (size_t)(R - 1) * rs + 4 * len + low;
        const size_t hb = ((size_t)B * hcols - R) * nkp;      // + s*nkp: the last row's column of step s - 1
        int n = 0, vi = 0;
        auto send_last = [&](int s) {
            const int nl = __builtin_amdgcn_readlane(n, R - 1), kl = __builtin_amdgcn_readlane(vi, R - 1) - nl + 1;
            if (send)
                for (int t = lane; t < nl; t += WAVE) {
                    const float *x = xl + 4 * ((s - 1) & 1) * len + t;
                    hand_put(handt + hb + (size_t)s * nkp + kl + t, x[0], tag);
                    hand_put(hande + hb + (size_t)s * nkp + kl + t, x[fs], tag);
                }
        };
        lds_barrier();                                        // the control wave's data of step 0
        for (int s = 0; s < nsteps; ++s) {
            // levels (0: no column), chunks | partial chunk << 16, VI, value above the column
            const int4 si = sinfo[(s & 1) * 32 + (lane & 31)];
            send_last(s);
            n = (lane < 32 && (lane & 15) < R) ? si.x : 0;
            vi = si.z;
            const int fm = __builtin_amdgcn_readfirstlane(si.y);
            float *Lp = L + (1 + 4 * (s & 1)) * len;
            const int o = chunk_of(n);
            const Chunk c0 = ld_chunk(Lp), t0 = ld_chunk(Lp + len), p0 = ld_chunk(Lp + 2 * len + o), v0 = ld_chunk(Lp + 3 * len + o);
            lds_barrier();                                    // the rows' sources are assembled
            if (n > 0) {
                strip_fwd<true>(L, Lp, Lp + len, fm & 0xffff, c0, t0);
                strip_tke_back(Lp + 2 * len, L, Lp + 3 * len, __int_as_float(si.w), floor, n, fm & 0xffff, (fm >> 16) != 0, low, p0, v0);
            }
            lds_barrier();                                    // the recurrences are done
        }
        send_last(nsteps);
        return;
    }
    if (r == R + 1) {                                         // control wave
        __builtin_amdgcn_s_setprio(2);
        const int row = lane & 15, b = ia + B * R + row;
        const bool lane_ok = lane < 32 && row < R && b <= ib;
        const gf32 *F = lane < 16 ? d.turb : d.tdiss;
        int cidx = ((IS == -1) ? nii - oa + 1 : oa) * nj2 + ((JS == -1) ? njj - b + 1 : b) - row * IS * nj2;
        // a column's metadata is requested two steps ahead, the value above it one
        auto meta_at = [&](int s) {
            const int l = s - row;
            int4 m = make_int4(0, -1, 0, 0);
            if (lane_ok && l >= 0 && l < na) m = ldg4i((const DomG::P<const int4>)meta + cidx);
            cidx += IS * nj2;
            return m;
        };
        int4 mq = meta_at(0), mb = make_int4(0, -1, 0, 0);
        float top = 0.0f;
        auto advance = [&](int s) {                           // metadata of step s arrives, its top value is requested
            const int c = cidx - IS * nj2;
            mb = mq;
            mq = meta_at(s + 1);
            top = 0.0f;
            if (mb.z & 0x10000) top = F[(size_t)c * nkp + mb.y + 1];
        };
        auto info = [&](int s) {
            const int n = (mb.z & 0x10000) ? mb.y - mb.x : 0;
            const int part = __any((n & (CHK - 1)) != 0) ? 0x10000 : 0;
            const int fm = row_max((n + CHK - 1) >> 3);
            if (lane < 32) sinfo[(s & 1) * 32 + lane] = make_int4(n, fm | part, mb.y, __float_as_int(top));
        };
        advance(0);
        info(0);
        advance(1);
        lds_barrier();
        for (int s = 0; s < nsteps; ++s) {
            info(s + 1);
            advance(s + 2);
            lds_barrier();
            lds_barrier();
        }
        return;
    }
    const int b = ia + B * R + r;
    const bool row_ok = b <= ib, from_prev = r == 0 && B > 0, has_j = r > 0 || B > 0, ip = IS == 1, jp = JS == 1;
    HandWait hwait{d.sync, wall_clock64() + STRIP_TIMEOUT_TICKS, false};
    const int rowb = 4 * r * rs, dcol = IS * nj2;
    gf32 *TW = d.turb, *EW = d.tdiss;
    const gf32 *planes = d.planes, *rec4 = d.planes + tke_rec4(d);
    int l2 = -r;
    int cidx2 = ((IS == -1) ? nii - oa + 1 : oa) * nj2 + ((JS == -1) ? njj - b + 1 : b) - r * dcol;
    int4 m2, m2j;
    auto request = [&]() {                                    // metadata of the next column and its -JS neighbour
        m2 = m2j = make_int4(0, -1, 0, 0);
        if (row_ok && l2 >= 0 && l2 < na) {
            m2 = ldc4i(meta + cidx2);
            if (has_j) m2j = ldc4i(meta + (cidx2 - JS));
        }
        ++l2;
        cidx2 += dcol;
    };
    const unsigned fi = 4u * (unsigned)nj2 * (unsigned)nkp, fj = 4u * (unsigned)nkp, base = fi + fj;
    const unsigned off_l = 4u * lane, off_c = base + off_l, off_a = ip ? off_c + fi : off_c - fi, off_b = jp ? off_c + fj : off_c - fj;
    const unsigned off_i = ip ? off_c - fi : off_c + fi, off_j = jp ? off_c - fj : off_c + fj;
    const unsigned off_p = 4u * TKE_REC * lane, off_q = 16u * lane, off_h = 8u * lane;
    const StripCol none{0, -1, 0, 0, 0};
    StripCol c0 = none, c1 = none, c1j = none, c2m = none, c2, c2j;   // steps s, s+1 (and its -JS neighbour), s-1, s+2
    unsigned o0 = 0, o1 = 0, op = 0;
    TkeRaw raw[M];
    TkeIn in[M];
    auto located = [&]() {
        c2 = strip_col<2>(m2);                                // kend unused
        c2j = strip_col<2>(m2j);
        request();
    };
    auto issue = [&](const StripCol &p, const StripCol &cn, const StripCol &cnj) {
        c1 = cn;
        c1j = cnj;
        const int ci = cidx2 - 2 * dcol, l = l2 - 2;
        if (c1.VI < 0) return;
        o1 = (unsigned)ci * (unsigned)nkp;
        const size_t o = (size_t)o1 + c1.KK + 1;
        const gf32 *Tl = TW + o - (base >> 2), *El = EW + o - (base >> 2);
        const size_t ho = ((size_t)(B - 1) * hcols + l) * nkp + c1.KK + 1;
        const gf32 *Ht = (const gf32 *)(handt + ho), *He = (const gf32 *)(hande + ho);
        const bool old_i = p.KK > c1.KK || p.VI < c1.VI, old_j = c1j.KK > c1.KK || c1j.VI < c1.VI;
        const int n = c1.VI - c1.KK;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (lane + WAVE * m < n) {
                TkeRaw &q = raw[m];
                const gf32 *P = lane_at(planes + (o + m * WAVE) * TKE_REC, off_p);
                q.c0 = ldg4(P); q.c1 = ldg4(P + 4); q.c2 = ldg4(P + 8); q.c4 = ldg2(P + 12);
                q.c3 = ldg4(lane_at(rec4 + (o + m * WAVE) * 4, off_q));
                const gf32 *Tm = Tl + m * WAVE, *Em = El + m * WAVE;
                q.ta = *lane_at(Tm, off_a); q.ea = *lane_at(Em, off_a);
                q.tb = *lane_at(Tm, off_b); q.eb = *lane_at(Em, off_b);
                if (old_i) { q.nit = *lane_at(Tm, off_i); q.nie = *lane_at(Em, off_i); }
                if (old_j) { q.njt = *lane_at(Tm, off_j); q.nje = *lane_at(Em, off_j); }
                if (from_prev) {
                    q.ht = hand_get((const gu64 *)lane_at(Ht + m * WAVE * 2, off_h));
                    q.he = hand_get((const gu64 *)lane_at(He + m * WAVE * 2, off_h));
                }
            }
        }
    };
    auto work_up = [&](int s, const StripCol &p) {
        const StripCol &c = c1;
        if (c.VI < 0) return;
        const int sc = rowb + 4 * ((1 + 4 * (s & 1)) * len + low), l4 = 4 * len, f4 = 4 * fs;
        const int si = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + c.KK - p.KK);
        const int sj = rowb - 4 * rs + 4 * ((8 - 4 * (s & 1)) * len + low + c.KK - c1j.KK);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int t4 = 4 * (lane + WAVE * m), k = c.KK + 1 + lane + WAVE * m;
            TkeRaw &q = raw[m];
            TkeIn &a = in[m];
            if (k <= c.VI) {
                const bool wall = q.c2.w != 0.0f;
                const float wt = q.c4.x < 0.001f ? 0.001f : q.c4.x, we = q.c4.y < 0.0000001f ? 0.0000001f : q.c4.y;
                lds_at(sm, sc + t4) = q.c2.y;
                lds_at(sm, sc + l4 + t4) = q.c3.x;
                lds_at(sm, sc + 2 * l4 + t4) = q.c3.y;
                lds_at(sm, sc + 3 * l4 + t4) = wall ? wt : TKE_NO_WALL;
                lds_at(sm, sc + f4 + t4) = q.c2.z;
                lds_at(sm, sc + f4 + l4 + t4) = q.c3.z;
                lds_at(sm, sc + f4 + 2 * l4 + t4) = q.c3.w;
                lds_at(sm, sc + f4 + 3 * l4 + t4) = wall ? we : TKE_NO_WALL;
                const float aw = q.c0.x, as = q.c0.y, ae = q.c0.z, an = q.c0.w;
                const float oi = ip ? ae : aw, oj = jp ? an : as;
                a.ai = ip ? aw : ae; a.aj = jp ? as : an;
                a.at = oi * q.ta; a.ae = oi * q.ea; a.bt = oj * q.tb; a.be = oj * q.eb;
                a.w1 = q.c1.x; a.pro = q.c1.y; a.pbo = q.c1.z; a.w2 = q.c1.w; a.eps = q.c2.x;
                a.nit = q.nit; a.nie = q.nie; a.njt = q.njt; a.nje = q.nje;
                a.si = k > p.KK && k <= p.VI;
                a.sj = k > c1j.KK && k <= c1j.VI;
                a.li = a.si ? si + t4 : 0;
                a.lj = a.sj ? sj + t4 : 0;
            }
        }
        if (from_prev) {
            const size_t ho = ((size_t)(B - 1) * hcols + (s - r)) * nkp;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = c.KK + 1 + lane + WAVE * m;
                const bool need = k <= c.VI && k > c1j.KK && k <= c1j.VI;
                hwait.wait(handt + ho + k, need, tag, raw[m].ht);
                hwait.wait(hande + ho + k, need, tag, raw[m].he);
                if (need) {
                    in[m].njt = __uint_as_float((unsigned)raw[m].ht);
                    in[m].nje = __uint_as_float((unsigned)raw[m].he);
                }
                in[m].sj = false;                             // the values are in njt, nje
                in[m].lj = 0;
            }
        }
    };
    request();
    located();
    issue(none, c2, c2j);
    located();
    work_up(0, none);
    c0 = c1; o0 = o1;
    issue(c0, c2, c2j);
    lds_barrier();                                            // the control wave's data of step 0
    for (int s = 0; s < nsteps; ++s) {
        // phase 1: the new neighbours enter the sources of step s
        if (c0.VI >= 0) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (lane + WAVE * m < c0.VI - c0.KK) {
                    const TkeIn &a = in[m];
                    float ti = lds_at(sm, a.li), ei = lds_at(sm, a.li + 4 * fs), tj = lds_at(sm, a.lj), ej = lds_at(sm, a.lj + 4 * fs);
                    ti = a.si ? ti : a.nit; ei = a.si ? ei : a.nie;
                    tj = a.sj ? tj : a.njt; ej = a.sj ? ej : a.nje;
                    const float mti = a.ai * ti, mtj = a.aj * tj, mei = a.ai * ei, mej = a.aj * ej;
                    const float D1 = (ip ? mti : a.at) + (jp ? mtj : a.bt) + (ip ? a.at : mti) + (jp ? a.bt : mtj) + a.w1 + a.pro + a.pbo;
                    const float D2 = (ip ? mei : a.ae) + (jp ? mej : a.be) + (ip ? a.ae : mei) + (jp ? a.be : mej) + a.w2 + a.eps;
                    const int q = rowb + 4 * (low + lane + WAVE * m);
                    lds_at(sm, q) = D1;
                    lds_at(sm, q + 4 * fs) = D2;
                }
            }
        }
        lds_barrier();
        // phase 2, beside the recurrences
        float xt[M], xe[M];
        const StripCol done = c2m;                            // the column of step s-1, before its buffer is reused
        const unsigned od = op;
        if (done.VI >= 0) {
            const int sn = rowb + 4 * ((8 - 4 * (s & 1)) * len + low + lane);
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < done.VI - done.KK) { xt[m] = lds_at(sm, sn + 4 * WAVE * m); xe[m] = lds_at(sm, sn + 4 * fs + 4 * WAVE * m); }
        }
        located();
        if (s + 1 < nsteps) work_up(s + 1, c0);
        c2m = c0; op = o0;
        c0 = c1; o0 = o1;
        if (s + 1 < nsteps) issue(c0, c2, c2j);
        else c0 = none;
        if (done.VI >= 0) {
            const size_t o = (size_t)od + done.KK + 1;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + WAVE * m < done.VI - done.KK) {
                    *(gf32 *)lane_at(TW + o + m * WAVE, off_l) = xt[m];
                    *(gf32 *)lane_at(EW + o + m * WAVE, off_l) = xe[m];
                }
        }
        lds_barrier();                                        // the recurrence outputs are ready
    }
    if (c2m.VI >= 0) {
        const size_t o = (size_t)op + c2m.KK + 1;
        const float *x = sm + (size_t)r * rs + (4 + 4 * ((nsteps - 1) & 1)) * len + low;
        for (int t = lane; t < c2m.VI - c2m.KK; t += WAVE) { TW[o + t] = x[t]; EW[o + t] = x[fs + t]; }
    }
}

// raises a kernel's dynamic LDS limit to bytes (above the default 64 KB; the
// device's is 160 KB) the first time a launch needs it; 1 on failure
static inline int lds_limit(const void *kern, size_t bytes) {
    static std::mutex mu;
    static const void *keys[64];                 // more than there are strip and coefficient kernels
    static size_t set[64];
    static int n = 0;
    if (bytes <= 65536) return 0;
    std::lock_guard<std::mutex> g(mu);
    int q = 0;
    while (q < n && keys[q] != kern) ++q;
    if (q < n && bytes <= set[q]) return 0;
    if (q == n && n == 64) return 1;
    if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return 1;
    keys[q] = kern;
    set[q] = bytes;
    if (q == n) ++n;
    return 0;
}
typedef void (*PressureKernel)(const Dom *, int, int, int);
static PressureKernel pressure_strip(const Dom *hd, int nsit) {
    int n = 0;
    for (int q = 0; q < nsit; ++q) n = max(n, hd[q].nact);
    return n <= WAVE ? k_pressure_strip<1> : k_pressure_strip<2>;
}
static size_t pressure_strip_lds(const Dom *hd, int nsit, int rows) {
    size_t m = 0;
    for (int q = 0; q < nsit; ++q)
        m = max(m, sizeof(float) * ((size_t)rows * strip_stride(9, strip_len(0, hd[q].nact)) + (RING + 2) * hd[q].nkp) +
                       32 * sizeof(int4) + 16);
    return m;
}
// LDS of the momentum strips of a launch (w: the W sweep, whose columns go down
// into the buildings) and the 64-level groups its tallest column spans
static inline size_t ml_strip_lds(const Dom *hd, int nsit, bool w, int rows) {
    size_t m = 0;
    for (int q = 0; q < nsit; ++q) {
        const int len = strip_len(w ? hd[q].nlow : 0, hd[q].nact);
        m = max(m, sizeof(float) * ((size_t)rows * strip_stride(9, len) + 2 * hd[q].nkp) + 32 * sizeof(int4) + 16);
    }
    return m;
}
static size_t ml_strip_lds_w(const Dom *hd, int nsit, int rows) { return ml_strip_lds(hd, nsit, true, rows); }
static size_t tke_strip_lds(const Dom *hd, int nsit, int rows) {
    size_t m = 0;
    for (int q = 0; q < nsit; ++q)
        m = max(m, sizeof(float) * (size_t)rows * strip_stride(TKE_ARRAYS, strip_len(0, hd[q].nact)) + 64 * sizeof(int4) + 16);
    return m;
}
typedef void (*StripKernel)(const Dom *, int, int);
static StripKernel tke_strip(const Dom *hd, int nsit) {
    int n = 0;
    for (int q = 0; q < nsit; ++q) n = max(n, hd[q].nact);
    return n <= WAVE ? k_tke_strip<1> : k_tke_strip<2>;
}
// Rows of a strip.  A strip is a workgroup of rows + 2 waves; fewer rows mean
// less work per step and CU, more strips and (a sweep's path is its column
// range plus rows per strip) about the same number of steps.  Ten rows while
// all strips of the launch find a CU of their own, not counting those of stream
// groups that run beside it (400 x 400 city, one situation: pressure, U and V
// sweeps 1.33, 1.41 and 1.38 ms against 1.42, 1.48 and 1.48 with 14), else 14
// (eight situations: 1.62, 2.04 and 1.71 ms against 1.80, 2.16 and 1.91 with ten).
// Short sweeps, whose path is mostly the fill of their first strips, take seven
// (25 rows: 60 against 65 us).  swap: the pressure sweep, whose rows run along i;
// lds: the kernel's LDS at a row count (tall columns take fewer rows).
#define LDS_BYTES (160 * 1024)
static int strip_rows(const Dom *hd, int nsit, bool swap, size_t (*lds)(const Dom *, int, int)) {
    long n = 0, longest = 0;
    for (int q = 0; q < nsit; ++q) {
        const int nb = (swap ? hd[q].nii : hd[q].njj) - 2;
        n += (nb + 9) / 10;
        longest = max(longest, (long)nb);
    }
    int rows = n > 256 ? 14 : longest > 40 ? 10 : STRIP_ROWS_MIN;
    while (rows > STRIP_ROWS_MIN && lds(hd, nsit, rows) > LDS_BYTES) rows = rows > 10 ? 10 : STRIP_ROWS_MIN;
    return rows;
}
template <int COMP, int WFIX, int KIND>
static StripKernel ml_strip(const Dom *hd, int nsit) {
    int n = 0;
    for (int q = 0; q < nsit; ++q) n = max(n, (COMP == 2 ? hd[q].nlow : 0) + hd[q].nact + 1);
    // buildings add to the W sweep's columns; with 4 groups (from 193 levels) it spills 76 to 156
    // bytes a lane at the 128 registers that 16 waves leave, the 16-wide one with 3 groups 20
    if constexpr (COMP == 2)
        if (n > 2 * WAVE) return n <= 3 * WAVE ? k_ml_strip<COMP, WFIX, KIND, 3> : k_ml_strip<COMP, WFIX, KIND, 4>;
    return n <= WAVE ? k_ml_strip<COMP, WFIX, KIND, 1> : k_ml_strip<COMP, WFIX, KIND, 2>;
}
template <int COMP>
static int ml_strip_limit(int model, const Dom *hd, int nsit) {
    bool w8 = true;
    for (int q = 0; q < nsit; ++q) w8 = w8 && hd[q].simd == 8;
    const StripKernel k = model == 2 ? ml_strip<COMP, 0, 1>(hd, nsit) : model == 0 ? ml_strip<COMP, 0, 2>(hd, nsit) :
                          w8 ? ml_strip<COMP, 8, 0>(hd, nsit) : ml_strip<COMP, 0, 0>(hd, nsit);
    return lds_limit((const void *)k, ml_strip_lds(hd, nsit, COMP == 2, strip_rows(hd, nsit, false, ml_strip_lds_w)));
}
// longest diagonal t over the situations; the pressure sweep runs a over j
// (outer) and b over i, the momentum sweeps a over i and b over j
static inline int diag_len_max(const Dom *hd, int nsit, int t, int oa, int ia, bool pressure) {
    int m = 0;
    for (int q = 0; q < nsit; ++q) {
        int ob = pressure ? hd[q].njj - 1 : hd[q].nii - 1, ib = pressure ? hd[q].nii - 1 : hd[q].njj - 1;
        if (t < ndiag(oa, ob, ia, ib)) m = max(m, diag_len(t, oa, ob, ia, ib));
    }
    return m;
}

// Optional per-launch timing: events recorded on the solver's stream right
// before and after every launch, tagged with the kernel family.
struct Probe {
    hipEvent_t *ev;      // 2*cap events
    int *fam;            // cap family tags
    int cap, n;
};
enum { FAM_STENCIL = 0, FAM_PRESSURE = 1, FAM_U = 2, FAM_V = 3, FAM_W = 4, FAM_TKE = 5, FAM_COEF = 6 };

struct Launcher {
    hipStream_t s;
    Probe *pr;
    long long n = 0;
    template <class F>
    void go(int fam, F &&f) {
        bool rec = pr && pr->n < pr->cap;
        if (rec) { (void)hipEventRecord(pr->ev[2 * pr->n], s); }
        f();
        if (rec) { (void)hipEventRecord(pr->ev[2 * pr->n + 1], s); pr->fam[pr->n] = fam; pr->n++; }
        ++n;
    }
};

// One momentum sweep on strips (the coefficient pre-pass, then the strips) over
// a in [oa, nii-1], b in [ia, njj-1]; go(family, launch), family -1: the sweep's own.
template <class Go>
static void launch_ml_strip(const Dom *hd, int nsit, const Dom *dd, StripKernel coef, StripKernel strip, int oa, int ia,
                            int is, int js, int rows, hipStream_t s, Go &&go) {
    int nblk = 0, nst = 0, nkp = 0;
    for (int q = 0; q < nsit; ++q) {
        int ob = hd[q].nii - 1, ib = hd[q].njj - 1;
        int na = ob - oa + 1, nb = ib - ia + 1;
        nblk = max(nblk, ((na * nb + COEF_COLS - 1) / COEF_COLS + NXCD - 1) / NXCD * NXCD);
        nst = max(nst, (ib - ia + rows) / rows);
        nkp = max(nkp, hd[q].nkp);
    }
    const unsigned Z = (unsigned)nsit;
    const size_t shm_c = sizeof(float) * 3 * (nkp | 1) * COEF_COLS + sizeof(int) * (SCOL * COEF_COLS + 4);
    go(FAM_COEF, [&] { hipLaunchKernelGGL(coef, dim3(nblk, 1, Z), dim3(4 * WAVE), shm_c, s, dd, is, js); });
    const size_t shm_t = ml_strip_lds(hd, nsit, oa == 2 && ia == 2, rows);
    go(-1, [&] { hipLaunchKernelGGL(strip, dim3(nst, 1, Z), dim3((rows + 2) * WAVE), shm_t, s, dd, is, js); });
}

// Launches one SIMPLE iteration of nsit situations that advance in lock step
// (same iteration number, hence the same sweep directions).  hd: host copies
// of the situations' Dom, dd: the same array in device memory.  Grid slice z
// of every launch is situation z; grid x/y are sized for the largest
// situation and each kernel skips what lies outside its own grid.  All
// situations share the turbulence model and the sweep kind.
static int launch_iteration(const Dom *hd, int nsit, const Dom *dd, int iter, int slot, hipStream_t s,
                            long long *launches, Probe *probe, bool proj);
extern "C" int pf_launch_iteration(const Dom *hd, int nsit, const Dom *dd, int iter, int slot, hipStream_t s,
                                   long long *launches, Probe *probe) {
    return launch_iteration(hd, nsit, dd, iter, slot, s, launches, probe, false);
}
// The pressure-correction part of iteration iter only (divergence, pressure
// sweep, velocity correction): the forward of the adjoint.  No residual slot.
extern "C" int pf_launch_projection(const Dom *hd, const Dom *dd, int iter, hipStream_t s, long long *launches) {
    return launch_iteration(hd, 1, dd, iter, -1, s, launches, nullptr, true);
}
static int launch_iteration(const Dom *hd, int nsit, const Dom *dd, int iter, int slot, hipStream_t s,
                            long long *launches, Probe *probe, bool proj) {
    if (nsit < 1) return 0;
    Launcher L{s, probe};
    const Dom &d0 = hd[0];
    int nii = 0, njj = 0, nk = 0, nkp = 0, nj2 = 0;
    for (int q = 0; q < nsit; ++q) {
        nii = max(nii, hd[q].nii); njj = max(njj, hd[q].njj); nk = max(nk, hd[q].kadvmax);
        nkp = max(nkp, hd[q].nkp); nj2 = max(nj2, hd[q].nj2);
    }
    const unsigned Z = (unsigned)nsit;
    const int rows_p = strip_rows(hd, nsit, true, pressure_strip_lds);
    const int rows = strip_rows(hd, nsit, false, ml_strip_lds_w), rows_t = strip_rows(hd, nsit, false, tke_strip_lds);
    int kb = (nk + 63) / 64;
    int IS = 1, JS = 1;
    switch (iter % 4) {
        case 0: IS = -1; JS = 1; break;
        case 1: IS = -1; JS = -1; break;
        case 2: IS = 1; JS = -1; break;
        default: break;
    }
    // every strip kernel this iteration launches gets its dynamic-LDS limit
    // before the first launch, so a refusal leaves the fields untouched
    if (d0.tiled == 2) {
        int bad = lds_limit((const void *)pressure_strip(hd, nsit), pressure_strip_lds(hd, nsit, rows_p));
        bad |= ml_strip_limit<0>(d0.model, hd, nsit) | ml_strip_limit<1>(d0.model, hd, nsit) | ml_strip_limit<2>(d0.model, hd, nsit);
        if (d0.model == 2) {
            bad |= lds_limit((const void *)k_tke_coef,
                             sizeof(float) * 5 * (nkp | 1) * COEF_COLS + sizeof(int) * (TKE_SCOL * COEF_COLS + 4));
            bad |= lds_limit((const void *)tke_strip(hd, nsit), tke_strip_lds(hd, nsit, rows_t));
        }
        if (bad) return (int)hipErrorInvalidValue;
    }
    int ncols = (nii - 2) * (njj - 2);
    const size_t bc_shm = bc_lds_bytes(max(nii, njj) + 2);
    const unsigned bc_threads = (unsigned)min(64 * kb, 1024);
    if (!proj) {
        L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_bc_ew, dim3(1, njj - 1, Z), dim3(bc_threads), bc_shm, s, dd); });
        L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_bc_ns, dim3(1, nii - 1, Z), dim3(bc_threads), bc_shm, s, dd); });
    }
    const int nrow8 = (nii - 2 + NXCD - 1) / NXCD * NXCD;                 // x extent of the cell kernels (rows)
    L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_divergence, dim3(nrow8, 1, Z), dim3(CELL_THREADS), 0, s, dd); });
    size_t nrow = d0.tiled ? 0 : (size_t)nj2 * nkp;
    for (int q = 0; q < nsit; ++q) nrow = max(nrow, (size_t)5 * hd[q].sync_stride);
    L.go(FAM_STENCIL, [&] {
        hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)((nrow + 255) / 256), 1, Z), dim3(256), 0, s, dd, d0.tiled ? 0 : 1);
    });
    if (d0.tiled == 2) {
        int nst = 0;
        for (int q = 0; q < nsit; ++q) nst = max(nst, (hd[q].nii - 3 + rows_p) / rows_p);
        const size_t shm = pressure_strip_lds(hd, nsit, rows_p);
        L.go(FAM_PRESSURE, [&] {
            hipLaunchKernelGGL(pressure_strip(hd, nsit), dim3(nst, 1, Z), dim3((rows_p + 2) * WAVE), shm, s, dd, IS, JS, slot);
        });
    } else {
        int oa = 2, ob = njj - 1, ia = 2, ib = nii - 1;
        size_t shm = sizeof(float) * 5 * nkp;
        for (int t = 0; t < ndiag(oa, ob, ia, ib); ++t) {
            int len = diag_len_max(hd, nsit, t, 2, 2, true);
            if (len > 0)
                L.go(FAM_PRESSURE, [&] {
                    hipLaunchKernelGGL(k_pressure, dim3(len, 1, Z), dim3(WAVE), shm, s, dd, t, IS, JS, slot);
                });
        }
    }
    L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_correction, dim3(nrow8, 1, Z), dim3(CELL_THREADS), 0, s, dd); });
    if (proj) {
        if (launches) *launches += L.n;
        return (int)hipGetLastError();
    }
    L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_averages, dim3(nrow8, 1, Z), dim3(CELL_THREADS), 0, s, dd); });
    L.go(FAM_STENCIL, [&] { hipLaunchKernelGGL(k_avg_edges, dim3(njj - 2, 1, Z), dim3(64), 0, s, dd); });
    size_t shm = sizeof(float) * 5 * nkp;
    // per-diagonal sweeps: sweep ranges a in [oa, nii-1] (outer), b in [ia, njj-1]
    auto sweep = [&](int fam, auto kern, int oa, int ia, int is, int js) {
        int nd = ndiag(oa, nii - 1, ia, njj - 1);
        for (int t = 0; t < nd; ++t) {
            int len = diag_len_max(hd, nsit, t, oa, ia, false);
            if (len > 0)
                L.go(fam, [&] { hipLaunchKernelGGL(kern, dim3(len, 1, Z), dim3(WAVE), shm, s, dd, t, is, js); });
        }
    };
    auto strip_sweep = [&](int fam, StripKernel coef, StripKernel strip, int oa, int ia, int is, int js) {
        launch_ml_strip(hd, nsit, dd, coef, strip, oa, ia, is, js, rows, s,
                        [&](int f, auto &&go) { L.go(f < 0 ? fam : f, go); });
    };
    bool all_w8 = true;
    for (int q = 0; q < nsit; ++q) all_w8 = all_w8 && hd[q].simd == 8;
    if (d0.model == 1 && d0.tiled == 2 && all_w8) {
        strip_sweep(FAM_U, k_ml_coef<0, 8>, ml_strip<0, 8, 0>(hd, nsit), 3, 2, IS, JS);
        strip_sweep(FAM_V, k_ml_coef<1, 8>, ml_strip<1, 8, 0>(hd, nsit), 2, 3, -IS, -JS);
        strip_sweep(FAM_W, k_ml_coef<2, 8>, ml_strip<2, 8, 0>(hd, nsit), 2, 2, IS, JS);
    } else if (d0.model == 1 && d0.tiled == 2) {
        strip_sweep(FAM_U, k_ml_coef<0, 0>, ml_strip<0, 0, 0>(hd, nsit), 3, 2, IS, JS);
        strip_sweep(FAM_V, k_ml_coef<1, 0>, ml_strip<1, 0, 0>(hd, nsit), 2, 3, -IS, -JS);
        strip_sweep(FAM_W, k_ml_coef<2, 0>, ml_strip<2, 0, 0>(hd, nsit), 2, 2, IS, JS);
    } else if (d0.model == 1) {
        sweep(FAM_U, k_momentum<0, 0>, 3, 2, IS, JS);
        sweep(FAM_V, k_momentum<1, 0>, 2, 3, -IS, -JS);
        sweep(FAM_W, k_momentum<2, 0>, 2, 2, IS, JS);
    } else if (d0.model == 2) {
        if (d0.tiled == 2) {
            // the k-eps V solver sweeps in the same directions as U and W
            strip_sweep(FAM_U, k_ml_coef<0, 0, 1>, ml_strip<0, 0, 1>(hd, nsit), 3, 2, IS, JS);
            strip_sweep(FAM_V, k_ml_coef<1, 0, 1>, ml_strip<1, 0, 1>(hd, nsit), 2, 3, IS, JS);
            strip_sweep(FAM_W, k_ml_coef<2, 0, 1>, ml_strip<2, 0, 1>(hd, nsit), 2, 2, IS, JS);
        } else {
            sweep(FAM_U, k_momentum<0, 1>, 3, 2, IS, JS);
            sweep(FAM_V, k_momentum<1, 1>, 2, 3, IS, JS);
            sweep(FAM_W, k_momentum<2, 1>, 2, 2, IS, JS);
        }
        if (d0.tiled == 2) {
            // strip-pipelined TKE: the neighbour-independent pre-pass, then the strips
            int nblk_t = 0;
            for (int q = 0; q < nsit; ++q)
                nblk_t = max(nblk_t, (((hd[q].nii - 2) * (hd[q].njj - 2) + COEF_COLS - 1) / COEF_COLS + NXCD - 1) / NXCD * NXCD);
            const size_t shm_c = sizeof(float) * 5 * (nkp | 1) * COEF_COLS + sizeof(int) * (TKE_SCOL * COEF_COLS + 4);
            if (lds_limit((const void *)k_tke_coef, shm_c)) return (int)hipErrorInvalidValue;
            L.go(FAM_COEF, [&] { hipLaunchKernelGGL(k_tke_coef, dim3(nblk_t, 1, Z), dim3(4 * WAVE), shm_c, s, dd); });
            int nst = 0;
            for (int q = 0; q < nsit; ++q) nst = max(nst, (hd[q].njj - 3 + rows_t) / rows_t);
            const size_t shm_k = tke_strip_lds(hd, nsit, rows_t);
            L.go(FAM_TKE, [&] {
                hipLaunchKernelGGL(tke_strip(hd, nsit), dim3(nst, 1, Z), dim3((rows_t + 2) * WAVE), shm_k, s, dd, IS, JS);
            });
        } else {
            size_t shm_t = sizeof(float) * 12 * nkp;
            int nd = ndiag(2, nii - 1, 2, njj - 1);
            for (int t = 0; t < nd; ++t) {
                int len = diag_len_max(hd, nsit, t, 2, 2, false);
                if (len > 0)
                    L.go(FAM_TKE, [&] { hipLaunchKernelGGL(k_tke, dim3(len, 1, Z), dim3(WAVE), shm_t, s, dd, t, IS, JS); });
            }
        }
    } else if (d0.tiled == 2) {
        strip_sweep(FAM_U, k_ml_coef<0, 0, 2>, ml_strip<0, 0, 2>(hd, nsit), 3, 2, IS, JS);
        strip_sweep(FAM_V, k_ml_coef<1, 0, 2>, ml_strip<1, 0, 2>(hd, nsit), 2, 3, IS, JS);
        strip_sweep(FAM_W, k_ml_coef<2, 0, 2>, ml_strip<2, 0, 2>(hd, nsit), 2, 2, IS, JS);
    } else {
        sweep(FAM_U, k_momentum<0, 2>, 3, 2, IS, JS);
        sweep(FAM_V, k_momentum<1, 2>, 2, 3, IS, JS);
        sweep(FAM_W, k_momentum<2, 2>, 2, 2, IS, JS);
    }
    if (launches) *launches += L.n;
    return (int)hipGetLastError();
}

extern "C" int pf_fill_u32(unsigned *p, size_t n, unsigned v, hipStream_t s) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// Flow-field file payloads, GFFWrite.cs: int16 of value*100 (FP32 product)
// kind 0 (:167-225): column records (u, v, w per level), clamp then truncate;
// kind 1 (:256-360): level-major rows u(j), v(j), w(j), clamp then truncate;
// kind 2 (:388-510): KKART, then per column u, v, w from max(KKART,1) up,
//                    MathF.Round (half to even) then clamp;
// kind 3 (:79-133, *.tke): TURB, clamp then Convert.ToInt16 (half to even).
// u and v of file level k are UK/VK[k-1], w is WK[k].  A NaN packs to 0.
// ------------------------------------------------------------------------
__device__ __forceinline__ float gff_at(const GffArgs &g, int f, size_t col, int k) {
    return k < g.nlo ? g.lo[f][col * (size_t)g.nkp + k] : g.up[f][col * (size_t)g.nup + (k - g.nlo)];
}
__device__ __forceinline__ int16_t gff_trunc(float v) {
    if (v != v) return 0;                                     // NaN
    if (v > 32767.0f) v = 32767.0f;
    else if (v < -32768.0f) v = -32768.0f;
    return (int16_t)(int)v;                                   // truncation toward zero
}
__device__ __forceinline__ int16_t gff_round(float v) {
    if (v != v) return 0;
    v = rintf(v);                                             // half to even
    if (v > 32767.0f) v = 32767.0f;
    else if (v < -32768.0f) v = -32768.0f;
    return (int16_t)(int)v;
}

// kinds 0 and 3: one block per column (a, b), threads over levels
__global__ void k_gff_column(GffArgs g) {
    const int nb = (g.kind == 3) ? g.njj : g.njj + 1;
    const int a = blockIdx.x / nb, b = blockIdx.x % nb;
    const size_t col = (size_t)(a + 1) * g.nj2 + (b + 1);
    if (g.kind == 3) {
        int16_t *o = g.out + ((size_t)a * g.njj + b) * g.nkk;
        for (int k = 1 + threadIdx.x; k <= g.nkk; k += blockDim.x) o[k - 1] = gff_round(gff_at(g, 3, col, k) * 100.0f);
        return;
    }
    int16_t *o = g.out + ((size_t)a * (g.njj + 1) + b) * (size_t)(g.nkk + 1) * 3;
    for (int kq = threadIdx.x; kq <= g.nkk; kq += blockDim.x) {
        o[3 * kq] = gff_trunc(gff_at(g, 0, col, kq) * 100.0f);
        o[3 * kq + 1] = gff_trunc(gff_at(g, 1, col, kq) * 100.0f);
        o[3 * kq + 2] = gff_trunc(gff_at(g, 2, col, kq + 1) * 100.0f);
    }
}

// kind 1: block (a, 64 columns b), levels in tiles of 32: the column reads
// (contiguous in k) are transposed through LDS into the rows of the file
// (contiguous in b)
#define GFF_BJ 64
#define GFF_KT 32
__global__ void __launch_bounds__(256) k_gff_rows(GffArgs g) {
    __shared__ int16_t tile[3][GFF_KT][GFF_BJ + 2];
    const int a = blockIdx.x, b0 = blockIdx.y * GFF_BJ;
    const int n = g.njj + 1, nb = min(GFF_BJ, n - b0), nk = g.nkk + 1;
    for (int k0 = 0; k0 < nk; k0 += GFF_KT) {
        const int kt = min(GFF_KT, nk - k0);
        for (int t = threadIdx.x; t < GFF_BJ * GFF_KT; t += blockDim.x) {
            const int cb = t / GFF_KT, kk = t % GFF_KT;
            if (cb < nb && kk < kt) {
                const size_t col = (size_t)(a + 1) * g.nj2 + (b0 + cb + 1);
                const int kq = k0 + kk;
                tile[0][kk][cb] = gff_trunc(gff_at(g, 0, col, kq) * 100.0f);
                tile[1][kk][cb] = gff_trunc(gff_at(g, 1, col, kq) * 100.0f);
                tile[2][kk][cb] = gff_trunc(gff_at(g, 2, col, kq + 1) * 100.0f);
            }
        }
        __syncthreads();
        for (int t = threadIdx.x; t < GFF_KT * 3 * GFF_BJ; t += blockDim.x) {
            const int cb = t % GFF_BJ, cp = (t / GFF_BJ) % 3, kk = t / (3 * GFF_BJ);
            if (cb < nb && kk < kt) {
                const size_t row = ((size_t)(k0 + kk) * (g.nii + 1) + a) * 3 + cp;
                g.out[row * n + b0 + cb] = tile[cp][kk][cb];
            }
        }
        __syncthreads();
    }
}

// kind 2: block per column (a, b) of the record part; block 0 also writes KKART
__global__ void k_gff_terrain(GffArgs g) {
    const int a = blockIdx.x / (g.njj + 1), b = blockIdx.x % (g.njj + 1);
    if (blockIdx.x == 0)
        for (size_t t = threadIdx.x; t < (size_t)g.nii * g.njj; t += blockDim.x) {
            const int ia = (int)(t / g.njj), jb = (int)(t % g.njj);
            g.out[t] = g.kk[(size_t)(ia + 1) * g.nj2 + (jb + 1)];
        }
    const size_t col = (size_t)(a + 1) * g.nj2 + (b + 1);
    const int k0 = max((int)g.kk[col], 1);
    const int n = g.nkk + 2 - k0;
    int16_t *o = g.out + (size_t)g.nii * g.njj + g.off[blockIdx.x];
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        o[t] = gff_round(gff_at(g, 0, col, k0 - 1 + t) * 100.0f);
        o[n + t] = gff_round(gff_at(g, 1, col, k0 - 1 + t) * 100.0f);
        o[2 * n + t] = gff_round(gff_at(g, 2, col, k0 + t) * 100.0f);
    }
}

// ------------------------------------------------------------------------
// The particle model's wind at a particle (Zeitschleife.IntWindCalculate,
// Intwind.cs:31-170): the level from HOKART (terrain: BinarySearch of the
// height above AHMIN, Intwind.cs:174-210; flat terrain with buildings: the
// first level whose top is at or above the particle), u and v linear in x and
// y across the cell faces (in double: the particle coordinate is a double),
// w linear in z between the level's bottom and top faces.
// ------------------------------------------------------------------------
__device__ __forceinline__ float wind_field(const WindArgs &a, int f, int i, int j, int k) {
    const size_t c = (size_t)i * a.nj2 + j;
    return k < a.nlo ? a.lo[f][c * a.nkp + k] : a.up[f][c * a.nup + (k - a.nlo)];
}

__global__ __launch_bounds__(256) void k_wind_at_particles(WindArgs a) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    const int i = a.ci[p], j = a.cj[p];
    const float z = a.z[p];
    float f1 = 0.0f;
    int k;
    if (a.topo) {
        f1 = z - a.ahmin;
        int low = 1, high = a.nkk;
        const int q = high >> 3;
        if (a.hok[q] >= f1) high = q;
        else low = q;
        while (low <= high) {
            const int mid = (low + high) >> 1;
            if (a.hok[mid] >= f1) high = mid - 1;
            else low = mid + 1;
        }
        k = min(low, a.nkk);
    } else {
        k = 1;
        while (k <= a.nkk && !(z <= a.hok[k])) ++k;
        k = min(k, a.nkk);
    }
    const float DXK = a.dxk, DYK = a.dyk;
    const float u1 = wind_field(a, 0, i, j, k), u2 = wind_field(a, 0, i + 1, j, k);
    const float ox = (float)a.ikoo + (float)(i - 1) * DXK;
    a.ux[p] = (float)((double)u1 + (double)((u2 - u1) / DXK) * (a.x[p] - (double)ox));
    const float v1 = wind_field(a, 1, i, j, k), v2 = wind_field(a, 1, i, j + 1, k);
    const float oy = (float)a.jkoo + (float)(j - 1) * DYK;
    a.uy[p] = (float)((double)v1 + (double)((v2 - v1) / DYK) * (a.y[p] - (double)oy));
    const float w1 = wind_field(a, 2, i, j, k), w2 = wind_field(a, 2, i, j, k + 1);
    const float dz = a.topo ? f1 - a.hok[k - 1] : (z + a.ahint[p]) - a.hok[k - 1];
    a.uz[p] = w1 + ((w2 - w1) / a.dzk[k]) * dz;
    a.ck[p] = k;
}

extern "C" int pf_launch_wind(const WindArgs *wa, hipStream_t s) {
    if (wa->n <= 0) return 0;
    hipLaunchKernelGGL(k_wind_at_particles, dim3((unsigned)((wa->n + 255) / 256)), dim3(256), 0, s, *wa);
    return (int)hipGetLastError();
}

extern "C" int pf_launch_gff(const GffArgs *ga, hipStream_t s) {
    const GffArgs g = *ga;
    if (g.kind == 0)
        hipLaunchKernelGGL(k_gff_column, dim3((unsigned)((g.nii + 1) * (g.njj + 1))), dim3(256), 0, s, g);
    else if (g.kind == 3)
        hipLaunchKernelGGL(k_gff_column, dim3((unsigned)(g.nii * g.njj)), dim3(256), 0, s, g);
    else if (g.kind == 1)
        hipLaunchKernelGGL(k_gff_rows, dim3((unsigned)(g.nii + 1), (unsigned)((g.njj + GFF_BJ) / GFF_BJ)), dim3(256), 0, s, g);
    else
        hipLaunchKernelGGL(k_gff_terrain, dim3((unsigned)((g.nii + 1) * (g.njj + 1))), dim3(256), 0, s, g);
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// FP64 mass imbalance of the current velocity field: over the active cells
// (ADVDOM = 1, 2 <= i <= NII-1, 2 <= j <= NJJ-1, KKART < k <= VerticalIndex)
// the sum of |DIV|, with DIV evaluated in FP32 exactly as the divergence pass
// forms it (PrognosticFlowfield.cs:723-758, the bottom flux dropped at
// KKART+1), and the sum of the absolute fluxes through the cell faces the
// same expression uses.  Each FP32 term is widened to double before it is
// accumulated.  Stage 1: a fixed range of columns per block, one column per
// wave with the lanes over k (coalesced), wavefront butterfly reductions in
// double, one partial pair per block.  Stage 2: one block per situation sums
// the partials.  The partition and the reduction trees are fixed, so the
// result is the same bits on every run.
// ------------------------------------------------------------------------
#define MASS_THREADS 256
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    return v;
}
__device__ __forceinline__ void block_sum2_f64(double &a, double &b) {
    __shared__ double red[MASS_THREADS / WAVE][2];
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    a = wave_sum_f64(a);
    b = wave_sum_f64(b);
    if (lane == 0) { red[w][0] = a; red[w][1] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = 0; b = 0;
        for (int q = 0; q < MASS_THREADS / WAVE; ++q) { a += red[q][0]; b += red[q][1]; }
    }
}
__global__ __launch_bounds__(MASS_THREADS) void k_mass_partial(const Dom *__restrict__ ds, double *__restrict__ partial) {
    const DomG &d = reinterpret_cast<const DomG *>(ds)[blockIdx.z];
    const int nj = d.njj - 2, ncols = (d.nii - 2) * nj;
    const int per = (ncols + (int)gridDim.x - 1) / (int)gridDim.x;
    const int c0 = (int)blockIdx.x * per, c1 = min(ncols, c0 + per);
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    double sd = 0, sf = 0;
    for (int col = c0 + w; col < c1; col += MASS_THREADS / WAVE) {
        const int i = 2 + col / nj, j = 2 + col % nj;
        const size_t c = c2(d, i, j);
        if (d.adv[c] != 1) continue;
        const int KK = d.kk[c], VI = d.vi[c];
        const size_t o = c3(d, i, j), oip = c3(d, i + 1, j), ojp = c3(d, i, j + 1);
        for (int k = KK + 1 + lane; k <= VI; k += WAVE) {
            const float dz = d.dzk[k];
            const float u0 = d.uk[o + k], u1 = d.uk[oip + k], v0 = d.vk[o + k], v1 = d.vk[ojp + k];
            const float w0 = d.wk[o + k], w1 = d.wk[o + k + 1];
            const float t1 = (u0 - u1) * d.dyk * dz;
            const float t2 = (v0 - v1) * d.dxk * dz;
            const float dv = (k > KK + 1) ? t1 + t2 + (w0 - w1) * d.area : t1 + t2 - w1 * d.area;
            sd += (double)fabsf(dv);
            double f = (double)fabsf(u0 * d.dyk * dz) + (double)fabsf(u1 * d.dyk * dz) +
                       (double)fabsf(v0 * d.dxk * dz) + (double)fabsf(v1 * d.dxk * dz) + (double)fabsf(w1 * d.area);
            if (k > KK + 1) f += (double)fabsf(w0 * d.area);
            sf += f;
        }
    }
    block_sum2_f64(sd, sf);
    if (threadIdx.x == 0) {
        double *p = partial + 2 * ((size_t)blockIdx.z * gridDim.x + blockIdx.x);
        p[0] = sd;
        p[1] = sf;
    }
}
__global__ __launch_bounds__(MASS_THREADS) void k_mass_final(const double *__restrict__ partial, int nblk,
                                                             double *__restrict__ out) {
    const double *p = partial + 2 * (size_t)blockIdx.x * nblk;
    double sd = 0, sf = 0;
    for (int b = threadIdx.x; b < nblk; b += MASS_THREADS) { sd += p[2 * b]; sf += p[2 * b + 1]; }
    block_sum2_f64(sd, sf);
    if (threadIdx.x == 0) { out[2 * blockIdx.x] = sd; out[2 * blockIdx.x + 1] = sf; }
}
// partial: [nsit][nblk][2] doubles of scratch; out: [nsit][2] (sum |DIV|, sum |face flux|)
extern "C" int pf_launch_mass(const Dom *dd, int nsit, int nblk, double *partial, double *out, hipStream_t s) {
    if (nsit < 1 || nblk < 1) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mass_partial, dim3((unsigned)nblk, 1, (unsigned)nsit), dim3(MASS_THREADS), 0, s, dd, partial);
    hipLaunchKernelGGL(k_mass_final, dim3((unsigned)nsit), dim3(MASS_THREADS), 0, s, partial, nblk, out);
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// Adjoint of one mixing-length momentum sweep (U/V/W-prognostic-microscale_1.cs:
// coefficients :194-470, Thomas forward :473-504, relaxed back-substitution
// :514-524) with respect to the swept component X, with everything else the
// sweep reads held fixed (UKS, VKS, WKS, DPMNEW, the other components).  X
// enters a column's equations through the eddy viscosity (own column, levels
// k-1 and k+1: the conductances, hence every power-law coefficient, and the
// cross-term factor), the Coriolis/vegetation and wall terms (own level), the
// cross terms (own level and the two neighbours along the component), the four
// neighbour couplings (new values of the two columns visited before it, old
// values of the two after it) and the relaxation.  Of a column's transpose only the
// recurrence through Q and the couplings to the two columns visited before it
// reach other columns, so three kernels do the transpose: k_adj_mom_pre computes
// every column's Thomas coefficients and couplings from the checkpointed fields
// (all columns at once), a strip sweep in reverse order carries the adjoint from
// column to column, and k_adj_mom runs the rest of each column's transpose (all
// columns at once) back through the coefficient assembly.  The adjoint handed to
// another column has one writer and is gathered by its receiver, so the result
// is deterministic.
// ------------------------------------------------------------------------

// d VIS / d X[k+1] of ml_visc (d VIS / d X[k-1] is its negative) for the
// component whose vertical shear enters VIS (U: UK, V: VK; W's VIS holds no WK)
template <int COMP>
__device__ __forceinline__ float ml_visc_dx(const DomG &d, const ColInfo &q, int k, const gf32 *UK, const gf32 *VK) {
    if (COMP == 2 || !(k > q.KK + 1)) return 0.0f;
    const float dz = d.dzk[k];
    const float zs = q.v512() ? d.hok[k] - fmaf(dz, 0.5f, d.hok[q.KK]) : d.hok[k] - d.hok[q.KK] - dz * 0.5f;
    float mixL = vminf(0.071f * zs, 100.0f);
    if (q.cov > 0) mixL *= (1.0f - 0.99f * q.cov);
    const float iu = (UK[k + 1] - UK[k - 1]) / (2.0f * dz), iv = (VK[k + 1] - VK[k - 1]) / (2.0f * dz);
    const float r = sqrtf(0.5f * (iu * iu + iv * iv));
    if (!(mixL * mixL * r < 15.0f) || !(r > 0.0f)) return 0.0f;      // at the cap of 15, or no shear
    return mixL * mixL * 0.5f * ((COMP == 0) ? iu : iv) / r / (2.0f * dz);
}

// d A / d D of a power-law coefficient A = D max(0, (1 - 0.1 P)^5) + F+ with
// P = |F / D| and F fixed
__device__ __forceinline__ float plaw_dd(float P) {
    const float x = 1.0f - 0.1f * P;
    if (!(x > 0.0f)) return 0.0f;
    const float x4 = (x * x) * (x * x);
    return x4 * x + 0.5f * x4 * P;
}

// d A / d VIS of the six coefficients of ml_coeffs (AE1, AW1, AS1, AN1, BIM, CIM)
__device__ __forceinline__ void ml_coeffs_dvis(const DomG &d, const ColInfo &q, int k, float VIS, float FE, float FW,
                                               float FS, float FN, float FT, float FB, float *g) {
    const float dz = d.dzk[k], dxkdzk = d.dxk * dz, dykdzk = d.dyk * dz;
    const float mv = vmaxf(VIS, d.vishmin), dmv = VIS > d.vishmin ? 1.0f : 0.0f;
    auto face = [&](bool off, float geo, float F) {           // conductance mv*geo, floored at 1e-4
        if (off) return 0.0f;
        const float Dr = mv * geo;
        if (!(Dr > 0.0001f)) return 0.0f;
        return dmv * geo * plaw_dd(fabsf(F / Dr));
    };
    const float gE = dykdzk / d.dxk, gS = dxkdzk / d.dyk, gT = d.area / dz;
    g[0] = face(q.ae, gE, FE);
    g[1] = face(q.aw, gE, FW);
    g[2] = face(q.as, gS, FS);
    g[3] = face(q.an, gS, FN);
    g[4] = face(false, gT, FT);
    g[5] = face(!(k > q.KK + 1), gT, FB);
}

// What the transposed sweep needs of each column besides the adjoints handed to
// it, for every cell of the situation (0 where the sweep does not go): the Thomas
// coefficients T, P, C (0 where the recurrence starts) and Q, and the couplings
// through which its DIM adjoint reaches the columns visited before it (ca, cb:
// along i and j; cc: VIS/DXK of the cross terms along the component's own
// direction, else 0); per column {KSTART, first level the sweep updates, VI}
// (VI = -1: none).  Blocks of MA_COLS columns: the lanes work the cells, then
// lane c runs column c's recurrence.
#define MA_COLS 8
template <int COMP>
__global__ __launch_bounds__(4 * WAVE) void k_adj_mom_pre(const Dom *__restrict__ ds, MomAdj m, int IS, int JS) {
    const DomG &d = *reinterpret_cast<const DomG *>(ds);
    extern __shared__ float sm[];
    const int nkp = d.nkp, nkl = nkp | 1, ncol = (d.nii + 2) * d.nj2, col0 = blockIdx.x * MA_COLS;
    float *sA = sm, *sB = sA + MA_COLS * nkl, *sC = sB + MA_COLS * nkl, *sD = sC + MA_COLS * nkl, *sT = sD + MA_COLS * nkl;
    int *scol = (int *)(sT + MA_COLS * nkl);                  // [MA_COLS][4]
    const int oa = (COMP == 0) ? 3 : 2, ia = (COMP == 1) ? 3 : 2;
    const gf32 *XA = (const gf32 *)m.xa, *XB = (COMP == 0) ? d.uk : (COMP == 1) ? d.vk : d.wk;
    if (threadIdx.x < MA_COLS) {
        const int c = col0 + threadIdx.x, i = c / d.nj2, j = c % d.nj2;
        int *sc = scol + 4 * threadIdx.x;
        sc[0] = 1; sc[1] = 0; sc[2] = -1; sc[3] = 0;
        if (c < ncol) {
            const int a = (IS == -1) ? d.nii - i + 1 : i, b = (JS == -1) ? d.njj - j + 1 : j;
            if (a >= oa && a <= d.nii - 1 && b >= ia && b <= d.njj - 1 && d.adv[c] == 1) {
                const ColInfo q = col_info(d, i, j);
                int KKm = 0;
                if (COMP == 0) KKm = max(q.KK, d.kk[c2(d, i - 1, j)]);
                if (COMP == 1) KKm = max(q.KK, d.kk[c2(d, i, j - 1)]);
                sc[0] = q.KSTART;
                sc[1] = max(q.KSTART, KKm + 1);
                if (COMP == 2) sc[1] = q.KSTART;
                sc[2] = q.VI;
                sc[3] = q.KK;
            }
            m.col[c] = make_int4(sc[0], sc[1], sc[2], 0);
        }
    }
    __syncthreads();
    const int cl = threadIdx.x / (4 * WAVE / MA_COLS), lv = threadIdx.x % (4 * WAVE / MA_COLS), c = col0 + cl;
    const int ks = scol[4 * cl], vi = scol[4 * cl + 2], KK = scol[4 * cl + 3];
    if (c < ncol) {
        const int i = c / d.nj2, j = c % d.nj2;
        const size_t o = (size_t)c * nkp;
        ColInfo q{};
        if (vi >= ks) q = col_info(d, i, j);
        for (int k = lv; k < nkp; k += 4 * WAVE / MA_COLS) {
            float ca = 0.0f, cb = 0.0f, cc = 0.0f;
            if (k >= ks && k <= vi) {
                const MlPieces pc = ml_pieces<COMP>(d, q, k);
                const size_t di = (size_t)d.nj2 * nkp;
                const float xpa = XA[o - IS * (ptrdiff_t)di + k], xna = XB[o + IS * (ptrdiff_t)di + k];
                const float xpb = XA[o - JS * (ptrdiff_t)nkp + k], xnb = XB[o + JS * (ptrdiff_t)nkp + k], x = XB[o + k];
                const float xw = (IS == 1) ? xpa : xna, xe = (IS == 1) ? xna : xpa;
                const float xs = (JS == 1) ? xpb : xnb, xn = (JS == 1) ? xnb : xpb;
                const int p = cl * nkl + k;
                sA[p] = pc.A; sB[p] = pc.B; sC[p] = pc.C;
                sD[p] = ml_source<COMP>(d, q, k, d.dzk[k], pc, xw, xs, xe, xn, x);
                ca = (IS == 1) ? pc.AW1 : pc.AE1;
                cb = (JS == 1) ? pc.AS1 : pc.AN1;
                if (COMP != 2 && ml_cross_on(q, k)) cc = pc.c0;
            }
            m.ca[o + k] = ca; m.cb[o + k] = cb; m.cc[o + k] = cc;
        }
    }
    __syncthreads();
    if (threadIdx.x < MA_COLS) {
        const int *sc = scol + 4 * threadIdx.x;
        float Pp = 0.0f, Qp = 0.0f;
        for (int k = sc[0]; k <= sc[2]; ++k) {                // as the sweep ran it
            const int p = threadIdx.x * nkl + k;
            float T;
            if (k > sc[3] + 1) { T = 1 / (sA[p] - sC[p] * Pp); Pp = sB[p] * T; Qp = (sD[p] + sC[p] * Qp) * T; }
            else { T = 1 / sA[p]; Pp = sB[p] * T; Qp = sD[p] * T; }
            sT[p] = T; sB[p] = Pp; sD[p] = Qp;
        }
    }
    __syncthreads();
    if (c < ncol)
        for (int k = lv; k < nkp; k += 4 * WAVE / MA_COLS) {
            const size_t g = (size_t)c * nkp + k;
            const int p = cl * nkl + k;
            const bool on = k >= ks && k <= vi;
            m.T[g] = on ? sT[p] : 0.0f;
            m.P[g] = on ? sB[p] : 0.0f;
            m.Q[g] = on ? sD[p] : 0.0f;
            m.C[g] = on && k > KK + 1 ? sC[p] : 0.0f;
            m.db[g] = 0.0f;
        }
}

// the adjoint column c hands to the a- (along i) and b-predecessor at level k
template <int COMP>
__device__ __forceinline__ float adj_mom_pa(float db, float ca, float cc, float dk) {
    return (COMP == 0 && cc != 0.0f) ? db * ca + db * cc * dk : db * ca;
}
template <int COMP>
__device__ __forceinline__ float adj_mom_pb(float db, float cb, float cc, float dk) {
    return (COMP == 1 && cc != 0.0f) ? db * cb + db * cc * dk : db * cb;
}

// The transposed sweep itself, on strips, in the reverse order of the sweep: the
// adjoint of a column's X after is gin and what its two successors hand it, and
// of the column's transposed recurrences only the one through Q reaches another
// column: g[k] = sG[k] + ub, Q_bar[k] = g relax, ub = Q_bar[k] P[k] up from the
// first updated level, then Qt = Q_bar[k] + Qc, D_bar[k] = Qt T[k],
// Qc = Qt C[k] T[k] down.  Bound by these.  The transpose of one component on 254 x
// 254 columns of up to 47 levels: pre-pass 0.18, strips 1.21, the rest 0.49 ms;
// with the whole column's transpose in one launch per anti-diagonal 19.5 ms.
template <int COMP>
struct MomOp {
    enum { NTAB = 1, NBUF = 3, SCRATCH = 0 };                              // table: DYK DZK (U) or DXK DZK (V); operands: P, C, T
    MomAdj m;
    const float *dzk;
    float h, relax;                                           // DYK (U), DXK (V)
    int nkp;
    struct Raw { float g, P, C, T, ca, cb, cc; };
    struct In { float g, ca, cb, cc, dk; };
    __device__ __forceinline__ float table(int, int k) const { return h * dzk[k]; }
    __device__ __forceinline__ LineCol levels(int c) const {
        const int4 v = ldc4i((const DomG::P<const int4>)m.col + c);
        return LineCol{v.x, v.z, v.y};
    }
    __device__ __forceinline__ void load(Raw &q, int c, int di, int dj, int k) const {
        const size_t o = (size_t)c * nkp + k, oi = (size_t)(c - di) * nkp + k, oj = (size_t)(c - dj) * nkp + k;
        q.g = ((const gf32 *)m.gin)[o];
        q.P = ((const gf32 *)m.P)[o];
        q.C = ((const gf32 *)m.C)[o];
        q.T = ((const gf32 *)m.T)[o];
        q.ca = ((const gf32 *)m.ca)[oi];
        q.cb = ((const gf32 *)m.cb)[oj];
        if (COMP != 2) q.cc = ((const gf32 *)m.cc)[COMP == 0 ? oi : oj];
    }
    __device__ __forceinline__ void stage(const Raw &q, In &a, bool on, int k, float *buf, int len, const float *tab) const {
        buf[0] = on ? q.P : 0.0f;
        buf[len] = on ? q.C : 0.0f;
        buf[2 * len] = on ? q.T : 0.0f;
        a.g = q.g; a.ca = q.ca; a.cb = q.cb; a.cc = q.cc;
        a.dk = tab[k];
    }
    __device__ __forceinline__ float source(const In &a, int k, const LineCol &q, float vi, float vj) const {
        const float g = a.g + adj_mom_pa<COMP>(vi, a.ca, a.cc, a.dk) + adj_mom_pb<COMP>(vj, a.cb, a.cc, a.dk);
        return k >= q.x ? g : 0.0f;                           // below, the sweep left X as it was
    }
    __device__ __forceinline__ void chain(float *L, float *N, float *buf, const float *, int len, int, int clo, int,
                                          int ct) const {
        const float *P = buf + clo * CHK, *C = buf + len, *T = buf + 2 * len;
        float *D = L + clo * CHK;
        {
            float ub = 0.0f;
            Chunk d[2], p[2];
            d[0] = ld_chunk(D); p[0] = ld_chunk(P);
            for (int c = clo; c <= ct;) {
#pragma unroll
                for (int h8 = 0; h8 < CHK_BLOCK; ++h8) {
                    if (c > ct) break;
                    const int k = h8 & 1, n = k ^ 1;
                    d[n] = ld_chunk(D + CHK); p[n] = ld_chunk(P + CHK);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = 0; u < CHK; ++u) {
                        const float qb = (d[k].v[u] + ub) * relax;
                        ub = qb * p[k].v[u];
                        d[k].v[u] = qb;
                    }
                    st_chunk(D, d[k]);
                    D += CHK; P += CHK;
                    ++c;
                }
            }
        }
        float qc = 0.0f;
        Chunk b[2], e[2], t[2];
        int o = ct * CHK;
        b[0] = ld_chunk(L + o); e[0] = ld_chunk(C + o); t[0] = ld_chunk(T + o);
        for (int c = ct; c >= clo;) {
#pragma unroll
            for (int h8 = 0; h8 < CHK_BLOCK; ++h8) {
                if (c < clo) break;
                const int k = h8 & 1, n = k ^ 1, on = max(o - CHK, 0);
                b[n] = ld_chunk(L + on); e[n] = ld_chunk(C + on); t[n] = ld_chunk(T + on);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = CHK - 1; u >= 0; --u) {
                    const float qt = b[k].v[u] + qc;
                    b[k].v[u] = qt * t[k].v[u];
                    qc = qt * e[k].v[u] * t[k].v[u];
                }
                st_chunk(N + o, b[k]);
                o = on;
                --c;
            }
        }
    }
    __device__ __forceinline__ void store(int c, int k, const LineCol &q, float x) const {
        if (k >= q.lo && k <= q.hi) ((gf32 *)m.db)[(size_t)c * nkp + k] = x;
    }
};

// The rest of a column's transpose, which no other column waits for: both
// transposed recurrences with the handed adjoints known, and the assembly
// transposed.  One wave per column.  DIAG: the whole of it, for the columns of
// anti-diagonal t, launched from the last one to the first, where the pre-pass's
// column data or the hand-off words find no memory (254 x 254 columns 19.5 ms a
// component, 1.9 in the three kernels).
#define MA_SLOTS 18
template <int COMP, bool DIAG>
__global__ __launch_bounds__(WAVE) void k_adj_mom(const Dom *__restrict__ ds, MomAdj m, int t, int IS, int JS) {
    const DomG &d = *reinterpret_cast<const DomG *>(ds);       // its swept field is X before the sweep
    extern __shared__ float sm[];
    int i = blockIdx.x / d.nj2, j = blockIdx.x % d.nj2;
    if (DIAG) {
        int a, b;
        if (!diag_col(t, (COMP == 0) ? 3 : 2, d.nii - 1, (COMP == 1) ? 3 : 2, d.njj - 1, blockIdx.x, a, b)) return;
        sweep_to_ij(d, 0, a, b, IS, JS, i, j);
        if (d.adv[c2(d, i, j)] != 1) return;
    } else if (m.col[blockIdx.x].z < 0) return;
    const ColInfo q = col_info(d, i, j);
    const int nkp = d.nkp, lane = threadIdx.x;
    const int KK = q.KK, KKP1 = KK + 1, KSTART = q.KSTART, VI = q.VI;
    int KKm = KK;
    if (COMP == 0) KKm = max(KK, d.kk[c2(d, i - 1, j)]);
    if (COMP == 1) KKm = max(KK, d.kk[c2(d, i, j - 1)]);
    const gf32 *XB = (COMP == 0) ? d.uk : (COMP == 1) ? d.vk : d.wk;
    const gf32 *XA = (const gf32 *)m.xa;
    const size_t o = c3(d, i, j), opa = c3(d, i - IS, j), ona = c3(d, i + IS, j), opb = c3(d, i, j - JS),
                 onb = c3(d, i, j + JS);
    float *sA = sm, *sB = sA + nkp, *sC = sB + nkp, *sD = sC + nkp, *sT = sD + nkp, *sP = sT + nkp, *sQ = sP + nkp;
    float *sG = sQ + nkp, *sXa = sG + nkp, *sAb = sXa + nkp, *sBb = sAb + nkp, *sCb = sBb + nkp, *sDb = sCb + nkp;
    // sR: own X before from the relaxation; sUp / sDn / sMid: from the assembly, for own X before at k+1 /
    // k-1 / k (sUp first holds the adjoint of P between the two transposed recurrences); sQb: adjoint of Q
    float *sR = sDb + nkp, *sUp = sR + nkp, *sDn = sUp + nkp, *sMid = sDn + nkp, *sQb = sMid + nkp;
    const float dyk = d.dyk, dxk = d.dxk;
    // 1. the column's equations from the checkpointed fields, and dL/dX after
    for (int k = KSTART + lane; k <= VI; k += WAVE) {
        const MlPieces pc = ml_pieces<COMP>(d, q, k);
        const float xpa = XA[opa + k], xna = XB[ona + k], xpb = XA[opb + k], xnb = XB[onb + k], x = XB[o + k];
        const float xw = (IS == 1) ? xpa : xna, xe = (IS == 1) ? xna : xpa;
        const float xs = (JS == 1) ? xpb : xnb, xn = (JS == 1) ? xnb : xpb;
        sA[k] = pc.A; sB[k] = pc.B; sC[k] = pc.C;
        sD[k] = ml_source<COMP>(d, q, k, d.dzk[k], pc, xw, xs, xe, xn, x);
        if (DIAG) {
            sG[k] = m.gin[o + k] + m.gpa[ona + k] + m.gpb[onb + k];
        } else {
            const float dk = (COMP == 0 ? dyk : dxk) * d.dzk[k];
            sG[k] = m.gin[o + k] + adj_mom_pa<COMP>(m.db[ona + k], m.ca[ona + k], m.cc[ona + k], dk) +
                    adj_mom_pb<COMP>(m.db[onb + k], m.cb[onb + k], m.cc[onb + k], dk);
            sT[k] = m.T[o + k]; sP[k] = m.P[o + k]; sQ[k] = m.Q[o + k];
        }
    }
    for (int k = KSTART + lane; k <= VI + 1; k += WAVE) sXa[k] = XA[o + k];
    __syncthreads();
    if (lane == 0) {
        if (DIAG) {                                           // Thomas forward, as the sweep ran it
            float Pp = 0.0f, Qp = 0.0f;
            for (int k = KSTART; k <= VI; ++k) {
                float T;
                if (k > KKP1) { T = 1 / (sA[k] - sC[k] * Pp); Pp = sB[k] * T; Qp = (sD[k] + sC[k] * Qp) * T; }
                else { T = 1 / sA[k]; Pp = sB[k] * T; Qp = sD[k] * T; }
                sT[k] = T; sP[k] = Pp; sQ[k] = Qp;
            }
        }
        // relaxed back-substitution X_k += relax (P_k X_{k+1} + Q_k - X_k) from VI down, transposed
        const float rl = d.relax;
        float ub = 0.0f;
        for (int k = KSTART; k <= VI; ++k) {
            const float g = sG[k] + ub;
            if (COMP == 2 || KKm < k) {
                sR[k] = g * (1.0f - rl);
                sQb[k] = g * rl;
                sUp[k] = g * rl * sXa[k + 1];
                ub = g * rl * sP[k];
            } else {
                sR[k] = g;
                sQb[k] = 0.0f;
                sUp[k] = 0.0f;
                ub = 0.0f;
            }
        }
        sR[VI + 1] = ub;                                  // X[VI+1] is the top value the first level read
        // Thomas forward transposed (VI down to KSTART)
        float Pc = 0.0f, Qc = 0.0f;
        for (int k = VI; k >= KSTART; --k) {
            const float Qt = sQb[k] + Qc, Pt = sUp[k] + Pc;
            const float B = sB[k], C = sC[k], D = sD[k], T = sT[k];
            float Ab, Bb, Cb, Db;
            if (k > KKP1) {
                const float Pm = sP[k - 1], Qm = sQ[k - 1];
                Db = Qt * T;
                const float Tb = Qt * (D + C * Qm) + Pt * B;
                Bb = Pt * T;
                Cb = Qt * Qm * T;
                Qc = Qt * C * T;
                const float denb = -Tb * T * T;
                Ab = denb;
                Cb += -denb * Pm;
                Pc = -denb * C;
            } else {
                Db = Qt * T;
                Bb = Pt * T;
                Ab = -(Qt * D + Pt * B) * T * T;
                Cb = 0.0f;
                Pc = 0.0f;
                Qc = 0.0f;
            }
            sAb[k] = Ab; sBb[k] = Bb; sCb[k] = Cb; sDb[k] = Db;
        }
    }
    __syncthreads();
    // 3. the assembly transposed, lanes over levels
    for (int k = KSTART + lane; k <= VI; k += WAVE) {
        const MlPieces pc = ml_pieces<COMP>(d, q, k);
        const float xpa = XA[opa + k], xna = XB[ona + k], xpb = XA[opb + k], xnb = XB[onb + k], x = XB[o + k];
        const float xw = (IS == 1) ? xpa : xna, xe = (IS == 1) ? xna : xpa;
        const float xs = (JS == 1) ? xpb : xnb, xn = (JS == 1) ? xnb : xpb;
        const float Ab = sAb[k], Bb = sBb[k], Cb = sCb[k], Db = sDb[k];
        const float dz = d.dzk[k];
        // AIM = BIM + CIM + AW1 + AS1 + AE1 + AN1 + AP0, D = AW1 X_W + AS1 X_S + AE1 X_E + AN1 X_N + ...
        const float awb = Ab + Db * xw, asb = Ab + Db * xs, aeb = Ab + Db * xe, anb = Ab + Db * xn;
        const float bimb = Bb + Ab, cimb = Cb + Ab;
        float xwb = Db * pc.AW1, xsb = Db * pc.AS1, xeb = Db * pc.AE1, xnb_ = Db * pc.AN1, xb = 0.0f;
        float visb = 0.0f, up = 0.0f, dn = 0.0f;
        const bool cross = ml_cross_on(q, k);
        if (COMP != 2) {
            const gf32 *UKS = d.uks + o, *VKS = d.vks + o;
            const gf32 *UKS_W = d.uks + c3(d, i - 1, j), *VKS_W = d.vks + c3(d, i - 1, j);
            float gfac = -d.cor;                              // g = (Cor (UG - x) [- VEG x wh]) AREA DZ
            if (q.vegp) {
                const float in2 = 0.5f * (VKS_W[k] + VKS[k]), in = 0.5f * (UKS_W[k] + UKS[k]);
                const float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.01f);
                gfac = -d.cor - d.veg[o + k - 1] * wh;
            }
            xb += Db * gfac * d.area * dz;
            if (k == KKP1) xb -= Db * ml_wall_uv(d, q, k, 1.0f, UKS, UKS_W, VKS, VKS_W);   // w = x / wh us^2 AREA
            if (cross) {
                if (COMP == 0) {
                    const float dk = dyk * dz;
                    const float S = (xe - x) * dk - (x - xw) * dk + pc.X1 - pc.X2 + pc.X3 - pc.X4;
                    const float Sb = Db * pc.c0;
                    xeb += Sb * dk; xwb += Sb * dk; xb -= 2.0f * Sb * dk;
                    visb += Db * S / dxk;                    // c0 = VIS / DXK
                } else {
                    const float dk = dxk * dz;
                    const float S = pc.X1 - pc.X2 + (xn - x) * dk - (x - xs) * dk + pc.X3 - pc.X4;
                    const float Sb = Db * pc.c0;
                    xnb_ += Sb * dk; xsb += Sb * dk; xb -= 2.0f * Sb * dk;
                    visb += Db * S / dxk;
                }
            }
            float FE, FW, FS, FN, FT, FB, g6[6];
            ml_fluxes<COMP>(d, q, k, FE, FW, FS, FN, FT, FB);
            const gf32 *UK = d.uk + o, *VK = d.vk + o;
            const float VIS = ml_visc(d, q, k, UK, VK);
            ml_coeffs_dvis(d, q, k, VIS, FE, FW, FS, FN, FT, FB, g6);
            visb += aeb * g6[0] + awb * g6[1] + asb * g6[2] + anb * g6[3] + bimb * g6[4] + cimb * g6[5];
            const float dvx = ml_visc_dx<COMP>(d, q, k, UK, VK);
            up = visb * dvx;
            dn = -visb * dvx;
        } else {
            if (q.vegp) {                                     // D -= VEG x wh AREA DZ
                const gf32 *UKS = d.uks + o, *VKS = d.vks + o, *UKS_W = d.uks + c3(d, i - 1, j);
                const gf32 *VKS_S = d.vks + c3(d, i, j - 1);
                const float in2 = 0.5f * (VKS_S[k] + VKS[k]), in = 0.5f * (UKS_W[k] + UKS[k]);
                const float wh = vmaxf(sqrtf(in * in + in2 * in2), 0.01f);
                xb -= Db * d.veg[o + k - 1] * wh * d.area * dz;
            }
            if (cross) {                                      // X1 = VIS/DZ (... + (X_{k+1} - x) AREA - (x - X_{k-1}) AREA)
                const float VIS = ml_visc(d, q, k, d.uk + o, d.vk + o);
                const float c = Db * (VIS / dz) * d.area;
                up = c; dn = c; xb -= 2.0f * c;
            }
        }
        sUp[k] = up; sDn[k] = dn; sMid[k] = xb;
        if (DIAG) {                                           // the adjoints of the predecessors' new values
            m.gpa[o + k] = (IS == 1) ? xwb : xeb;
            m.gpb[o + k] = (JS == 1) ? xsb : xnb_;
        }
        // the adjoints of the successors' old values
        m.gna[o + k] = (IS == 1) ? xeb : xwb;
        m.gnb[o + k] = (JS == 1) ? xnb_ : xsb;
    }
    __syncthreads();
    // 4. own X before, levels KSTART-1 .. VI+1, summed in a fixed order
    for (int k = KSTART - 1 + lane; k <= VI + 1; k += WAVE) {
        float v = 0.0f;
        if (k >= KSTART && k <= VI) v = sR[k] + sMid[k];
        if (k == VI + 1) v = sR[VI + 1];
        if (k - 1 >= KSTART && k - 1 <= VI) v += sUp[k - 1];
        if (k + 1 >= KSTART && k + 1 <= VI) v += sDn[k + 1];
        m.gout[o + k] = v;
    }
}

// dL/dX before of every cell: its own column's part, the adjoints its
// predecessors handed to its old value, and, where the sweep left X as it was
// (columns it does not visit, levels outside KSTART..VI), dL/dX after with the
// adjoints its successors handed to its new value.  Thread per cell and level.
template <int COMP, bool DIAG>
__global__ void k_adj_mom_combine(const Dom *__restrict__ ds, MomAdj m, int IS, int JS) {
    const DomG &d = *reinterpret_cast<const DomG *>(ds);
    const size_t n3 = (size_t)(d.nii + 2) * d.nj2 * d.nkp;
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n3) return;
    const int k = (int)(g % d.nkp);
    const size_t c = g / d.nkp;
    const int i = (int)(c / d.nj2), j = (int)(c % d.nj2);
    const int oa = (COMP == 0) ? 3 : 2, ia = (COMP == 1) ? 3 : 2;
    auto inside = [&](int ii, int jj) { return ii >= 0 && ii <= d.nii + 1 && jj >= 0 && jj <= d.njj + 1; };
    float v = m.gout[g];
    if (inside(i - IS, j)) v += m.gna[c3(d, i - IS, j) + k];
    if (inside(i, j - JS)) v += m.gnb[c3(d, i, j - JS) + k];
    bool done = false;
    if (i >= 1 && i <= d.nii && j >= 1 && j <= d.njj && d.adv[c] == 1) {
        const int a = (IS == -1) ? d.nii - i + 1 : i, b = (JS == -1) ? d.njj - j + 1 : j;
        if (a >= oa && a <= d.nii - 1 && b >= ia && b <= d.njj - 1) {
            const int KK = d.kk[c];
            const int KSTART = (d.cutk[c] == 0) ? KK + 1 : 1;
            done = k >= KSTART && k <= d.vi[c];
        }
    }
    if (!done) {
        v += m.gin[g];
        const float dk = (COMP == 0 ? d.dyk : d.dxk) * d.dzk[k];
        const size_t na = c3(d, i + IS, j) + k, nb = c3(d, i, j + JS) + k;
        if (inside(i + IS, j)) v += DIAG ? m.gpa[na] : adj_mom_pa<COMP>(m.db[na], m.ca[na], m.cc[na], dk);
        if (inside(i, j + JS)) v += DIAG ? m.gpb[nb] : adj_mom_pb<COMP>(m.db[nb], m.cb[nb], m.cc[nb], dk);
    }
    m.gres[g] = v;
}

__global__ void k_mom_fill(float *p, size_t n) {
    size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < n) p[g] = 0.0f;
}

// One sweep of momentum component comp (0 U, 1 V, 2 W) of the mixing-length
// model in the directions (IS, JS) the iteration gives it: the strips where the
// situation has them, else one launch per anti-diagonal (the same result bit for
// bit; 254 x 254 columns: 0.9 to 1.1 ms on strips with the pre-pass, 9.1 ms with the
// launches per anti-diagonal).
extern "C" int pf_launch_momentum_sweep(const Dom *hd, const Dom *dd, int comp, int IS, int JS, hipStream_t s) {
    const Dom &h = *hd;
    if (h.model != 1 || comp < 0 || comp > 2) return (int)hipErrorInvalidValue;
    const int oa = (comp == 0) ? 3 : 2, ia = (comp == 1) ? 3 : 2, ob = h.nii - 1, ib = h.njj - 1;
    if (ob < oa || ib < ia) return 0;
    if (h.tiled == 2) {
        const int rows = strip_rows(hd, 1, false, ml_strip_lds_w);
        if (comp == 0 ? ml_strip_limit<0>(1, hd, 1) : comp == 1 ? ml_strip_limit<1>(1, hd, 1) : ml_strip_limit<2>(1, hd, 1))
            return (int)hipErrorInvalidValue;
        const bool w8 = h.simd == 8;
        const StripKernel strip = comp == 0 ? (w8 ? ml_strip<0, 8, 0>(hd, 1) : ml_strip<0, 0, 0>(hd, 1)) :
                                  comp == 1 ? (w8 ? ml_strip<1, 8, 0>(hd, 1) : ml_strip<1, 0, 0>(hd, 1)) :
                                              (w8 ? ml_strip<2, 8, 0>(hd, 1) : ml_strip<2, 0, 0>(hd, 1));
        const StripKernel coef = comp == 0 ? (w8 ? k_ml_coef<0, 8> : k_ml_coef<0, 0>) :
                                 comp == 1 ? (w8 ? k_ml_coef<1, 8> : k_ml_coef<1, 0>) : (w8 ? k_ml_coef<2, 8> : k_ml_coef<2, 0>);
        hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)((5 * h.sync_stride + 255) / 256)), dim3(256), 0, s, dd, 0);
        launch_ml_strip(hd, 1, dd, coef, strip, oa, ia, IS, JS, rows, s, [](int, auto &&f) { f(); });
        return (int)hipGetLastError();
    }
    const size_t shm = sizeof(float) * 5 * h.nkp;
    for (int t = 0; t < ndiag(oa, ob, ia, ib); ++t) {
        const unsigned len = (unsigned)diag_len(t, oa, ob, ia, ib);
        if (comp == 0) hipLaunchKernelGGL((k_momentum<0, 0>), dim3(len), dim3(WAVE), shm, s, dd, t, IS, JS);
        else if (comp == 1) hipLaunchKernelGGL((k_momentum<1, 0>), dim3(len), dim3(WAVE), shm, s, dd, t, IS, JS);
        else hipLaunchKernelGGL((k_momentum<2, 0>), dim3(len), dim3(WAVE), shm, s, dd, t, IS, JS);
    }
    return (int)hipGetLastError();
}

// The transpose of that sweep: dd is the situation's descriptor with the swept
// field pointing at X before the sweep.
extern "C" int pf_launch_momentum_vjp(const Dom *hd, const Dom *dd, const MomAdj *ma, int comp, int IS, int JS,
                                      hipStream_t s) {
    const Dom &h = *hd;
    if (h.model != 1 || comp < 0 || comp > 2) return (int)hipErrorInvalidValue;
    const MomAdj m = *ma;
    const size_t n3 = (size_t)(h.nii + 2) * h.nj2 * h.nkp;
    const unsigned fb = (unsigned)((n3 + 255) / 256);
    const bool diag = m.hand == nullptr;                      // no column data and words: per anti-diagonal
    float *z[5] = {m.gout, m.gna, m.gnb, m.gpa, m.gpb};
    for (int q = 0; q < (diag ? 5 : 3); ++q) hipLaunchKernelGGL(k_mom_fill, dim3(fb), dim3(256), 0, s, z[q], n3);
    const int oa = (comp == 0) ? 3 : 2, ia = (comp == 1) ? 3 : 2, ob = h.nii - 1, ib = h.njj - 1, ni = h.nii - oa, nj = h.njj - ia;
    const int ncol = (h.nii + 2) * h.nj2;
    const size_t shm_p = (sizeof(float) * 5 * (h.nkp | 1) + sizeof(int) * 4) * MA_COLS, shm = sizeof(float) * MA_SLOTS * h.nkp;
    int e = 0;
    auto run = [&](auto tag) {
        constexpr int C = decltype(tag)::value;
        if (diag) {
            for (int t = ndiag(oa, ob, ia, ib) - 1; t >= 0; --t)
                hipLaunchKernelGGL((k_adj_mom<C, true>), dim3((unsigned)diag_len(t, oa, ob, ia, ib)), dim3(WAVE), shm, s, dd, m, t, IS, JS);
            hipLaunchKernelGGL((k_adj_mom_combine<C, true>), dim3(fb), dim3(256), 0, s, dd, m, IS, JS);
            return;
        }
        hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)((5 * h.sync_stride + 255) / 256)), dim3(256), 0, s, dd, 0);
        hipLaunchKernelGGL(k_adj_mom_pre<C>, dim3((ncol + MA_COLS - 1) / MA_COLS), dim3(4 * WAVE), shm_p, s, dd, m, IS, JS);
        if (ni > 0 && nj > 0) {
            // the sweep's order reversed: from its last row and column back
            const int i0 = IS == 1 ? h.nii - 1 : 2, j0 = JS == 1 ? h.njj - 1 : 2;
            const MomOp<C> op{m, h.dzk, C == 0 ? h.dyk : h.dxk, h.relax, h.nkp};
            const LineSweep w{ni, nj, i0 * h.nj2 + j0, -IS * h.nj2, -JS, h.nkp, h.sync, SYNC_BLOCK0, 6, m.hand, nullptr};
            e = h.nkp <= WAVE ? launch_line<MomOp<C>, 1>(op, w, s) : launch_line<MomOp<C>, 2>(op, w, s);
            if (e) return;
            hipLaunchKernelGGL((k_adj_mom<C, false>), dim3(ncol), dim3(WAVE), shm, s, dd, m, 0, IS, JS);
        }
        hipLaunchKernelGGL((k_adj_mom_combine<C, false>), dim3(fb), dim3(256), 0, s, dd, m, IS, JS);
    };
    if (comp == 0) run(std::integral_constant<int, 0>()); else if (comp == 1) run(std::integral_constant<int, 1>());
    else run(std::integral_constant<int, 2>());
    if (e) return e;
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// The transposed pressure sweep (S^T of pf_adjoint.hip) on strips, in the reverse
// order of the sweep.  x_bar[k] = pb[k] + what the two successors hand down, then
// the transposed substitution x_bar[k-1] += P[k] x_bar[k] top-down with Q_bar[k] =
// (Q_bar handed by later columns) + x_bar[k], and the transposed elimination
// bottom-up: DIM_bar[k] = TERMP[k] (Q_bar[k] + carry), carry = ATP[k] TERMP[k] (..).
// The carry above the column's top goes to the last earlier column of the same
// sweep row that holds level VI+1: the row scratch.  Bound by the recurrences (3500
// of a step's 5500 cycles, 66 levels of the rows' columns together): 1.37 ms a
// sweep of 254 x 254 columns, 2.5 ms with one launch per anti-diagonal.
// ------------------------------------------------------------------------
struct PrAdjOp {
    enum { NTAB = 3, NBUF = 3, SCRATCH = 1 };                 // tables: DYK DZK/DXK, DXK DZK/DYK, ATP; operands: P, TERMP, ATP*TERMP
    AdjArgs a;
    const float *dzk, *atp;
    float dxk, dyk, dtime, sgn;                               // sgn: the sign with which the columns along j enter DIM
    int nkp;
    struct Raw { float x, p, t; };
    struct In { float x, ui, uj; };
    __device__ __forceinline__ float table(int q, int k) const {
        return q == 0 ? dyk * dzk[k] / dxk : q == 1 ? dxk * dzk[k] / dyk : atp[k];
    }
    __device__ __forceinline__ LineCol levels(int c) const {
        const int4 v = ldc4i((const DomG::P<const int4>)a.col + c);
        return LineCol{v.x, v.y, 0};
    }
    __device__ __forceinline__ void load(Raw &q, int c, int, int, int k) const {
        const size_t o = (size_t)c * nkp + k;
        q.x = ((const gf32 *)a.pb)[o];
        q.p = ((const gf32 *)a.ptab)[o];
        q.t = ((const gf32 *)a.ttab)[o];
    }
    __device__ __forceinline__ void stage(const Raw &q, In &i, bool on, int k, float *buf, int len, const float *tab) const {
        buf[0] = on ? q.p : 0.0f;
        buf[len] = on ? q.t : 0.0f;
        buf[2 * len] = on ? tab[2 * len + k] * q.t : 0.0f;
        i.x = q.x;
        i.ui = tab[k];
        i.uj = tab[len + k];
    }
    __device__ __forceinline__ float source(const In &i, int, const LineCol &, float vi, float vj) const {
        return i.x + vi * i.ui + sgn * vj * i.uj;
    }
    __device__ __forceinline__ void chain(float *L, float *N, float *buf, const float *, int len, int, int clo, int,
                                          int ct) const {
        const float *E = L + (3 + 2 * NBUF) * len, *P = buf, *T = buf + len + clo * CHK, *A = buf + 2 * len + clo * CHK;
        {
            float t = 0.0f;                                   // P[k+1] x_bar[k+1]
            Chunk d[2], e[2], p[2];
            int o = ct * CHK;
            d[0] = ld_chunk(L + o); e[0] = ld_chunk(E + o); p[0] = ld_chunk(P + o);
            for (int c = ct; c >= clo;) {
#pragma unroll
                for (int h8 = 0; h8 < CHK_BLOCK; ++h8) {
                    if (c < clo) break;
                    const int k = h8 & 1, n = k ^ 1, on = max(o - CHK, 0);
                    d[n] = ld_chunk(L + on); e[n] = ld_chunk(E + on); p[n] = ld_chunk(P + on);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = CHK - 1; u >= 0; --u) {
                        const float x = d[k].v[u] + t;
                        t = p[k].v[u] * x;
                        e[k].v[u] += x;
                    }
                    st_chunk(L + o, e[k]);
                    o = on;
                    --c;
                }
            }
        }
        float carry = 0.0f;
        float *Q = L + clo * CHK;
        N += clo * CHK;
        Chunk q[2], t[2], b[2];
        q[0] = ld_chunk(Q); t[0] = ld_chunk(T); b[0] = ld_chunk(A);
        for (int c = clo; c <= ct;) {
#pragma unroll
            for (int h8 = 0; h8 < CHK_BLOCK; ++h8) {
                if (c > ct) break;
                const int k = h8 & 1, n = k ^ 1;
                q[n] = ld_chunk(Q + CHK); t[n] = ld_chunk(T + CHK); b[n] = ld_chunk(A + CHK);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < CHK; ++u) {
                    const float qt = q[k].v[u] + carry;
                    carry = b[k].v[u] * qt;
                    t[k].v[u] *= qt;
                    q[k].v[u] = qt;
                }
                st_chunk(N, t[k]);
                st_chunk(Q, q[k]);                            // at VI+1: the carry
                Q += CHK; T += CHK; A += CHK; N += CHK;
                ++c;
            }
        }
    }
    __device__ __forceinline__ void store(int c, int k, const LineCol &q, float x) const {
        if (k >= q.lo && k <= q.hi) ((gf32 *)a.db)[(size_t)c * nkp + k] = x / dtime;      // DIM = DIV / DTIME + ...
    }
};
// launches it; hipErrorInvalidValue where the columns have more levels than the strips hold
extern "C" int pf_launch_adjoint_sweep(const Dom *hd, const Dom *dd, const AdjArgs *args, int IS, int JS, hipStream_t s) {
    const Dom &h = *hd;
    if (h.nkp > 4 * WAVE) return (int)hipErrorInvalidValue;
    const int ni = h.nii - 2, nj = h.njj - 2;
    if (ni < 1 || nj < 1) return 0;
    hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)((5 * h.sync_stride + 255) / 256)), dim3(256), 0, s, dd, 0);
    const int i0 = IS == 1 ? h.nii - 1 : 2, j0 = JS == 1 ? h.njj - 1 : 2;
    const PrAdjOp op{*args, h.dzk, h.atp, h.dxk, h.dyk, h.dtime, JS == 1 ? 1.0f : -1.0f, h.nkp};
    const LineSweep w{ni, nj, i0 * h.nj2 + j0, -IS * h.nj2, -JS, h.nkp, h.sync, SYNC_BLOCK0, 7, args->hand, args->handq};
    return h.nkp <= WAVE ? launch_line<PrAdjOp, 1>(op, w, s) : h.nkp <= 2 * WAVE ? launch_line<PrAdjOp, 2>(op, w, s) :
                                                                                  launch_line<PrAdjOp, 4>(op, w, s);
}
