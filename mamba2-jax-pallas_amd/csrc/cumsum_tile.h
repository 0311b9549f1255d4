// The workgroup's part of chunk_cumsum (chunk_cumsum.hip), shared with the
// preparation kernel of the one-pass layer (ssd_walk.hip).
#pragma once

#include "m2_common.h"

namespace m2cum {

constexpr int HB = 16;                 // heads per workgroup: one wavefront each
constexpr int CUM_THREADS = HB * 64;

struct CumsumArgs {
    const void* dt;
    const float* A;
    const float* bias;
    const int32_t* seq;       // [b, L] or NULL (weights / decay only)
    float* dA;
    float* dto;
    float* wts;               // [b, H, nc, Q] or NULL
    float* scl;               // [b, H, nc] or NULL
    int L, H, Q, nc, softplus, nhb, nblocks;
    float lo, hi;
};

// PPL: positions per lane (Q <= 64 PPL); CPW: chunks per workgroup (1, or 2
// where one chunk per workgroup would need more than one round of the CUs:
// all loads of both chunks go out before the first wait, so the two load
// round trips overlap instead of following each other)
template <typename TD, int PPL, int CPW>
M2_DEV void cumsum_block(const CumsumArgs& a, int work, float (&tile)[CPW][64 * PPL][HB + 1]) {
    const int ncw = (a.nc + CPW - 1) / CPW;
    const int hb = work % a.nhb, cw = (work / a.nhb) % ncw, bi = work / (a.nhb * ncw);
    const int Q = a.Q, L = a.L, H = a.H;
    const int lane = threadIdx.x & 63, w = wave_id();
    const int h = hb * HB + w;
    // every global load of the workgroup is issued before the first wait:
    // the head's A / bias and the chunks' seq ids, then the dt tiles
    const float Ah = a.A[min(h, H - 1)];
    const float bias = a.bias ? a.bias[min(h, H - 1)] : 0.f;
    int sq[CPW][PPL];
    int se[CPW], sprev[CPW];
    const int hh = threadIdx.x % HB, r0 = threadIdx.x / HB;
    TD raw[CPW][PPL];
#pragma unroll
    for (int k = 0; k < CPW; ++k) {
        // a workgroup's second chunk past the last one repeats the last (its
        // loads stay in bounds; it stores nothing)
        const int c = min(cw * CPW + k, a.nc - 1);
        const int qhi = min(Q, L - c * Q);          // valid positions of the chunk
        const int64_t tok0 = (int64_t)bi * L + (int64_t)c * Q;
        se[k] = 0; sprev[k] = 0;
        if (a.seq) {
#pragma unroll
            for (int j = 0; j < PPL; ++j) sq[k][j] = a.seq[tok0 + min(lane + 64 * j, qhi - 1)];
            se[k] = a.seq[tok0 + qhi - 1];
            if (c > 0) sprev[k] = a.seq[tok0 - 1];
        }
        // ---- coalesced tile load: thread t -> head t % 16, rows t / 16 + 64 i;
        // addresses clamped into the valid rows / heads (masked below)
        const TD* dtp = reinterpret_cast<const TD*>(a.dt) + tok0 * H + min(hb * HB + hh, H - 1);
#pragma unroll
        for (int i = 0; i < PPL; ++i) raw[k][i] = dtp[(int64_t)min(r0 + 64 * i, qhi - 1) * H];
    }
#pragma unroll
    for (int k = 0; k < CPW; ++k)
#pragma unroll
        for (int i = 0; i < PPL; ++i)
            if (r0 + 64 * i < Q) tile[k][r0 + 64 * i][hh] = to_f32(raw[k][i]);
    __syncthreads();
    if (h >= H) return;                             // no barrier follows
#pragma unroll
    for (int k = 0; k < CPW; ++k) {
    const int c = cw * CPW + k;
    if (c >= a.nc) break;
    const int qhi = min(Q, L - c * Q);

    float v[PPL], dA[PPL];
    float carry = 0.f;
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const int q = lane + 64 * j;
        float d = q < Q ? tile[k][q][w] : 0.f;
        if (a.bias) d += bias;
        if (a.softplus) d = softplus_f(d);
        d = fminf(fmaxf(d, a.lo), a.hi);
        v[j] = q < qhi ? d : 0.f;
        dA[j] = wave_scan(v[j] * Ah) + carry;
        carry = lane63(dA[j]);
    }
    const float total = carry;                      // == dA[Q - 1] exactly
    float* const rowp = a.dA + (((int64_t)bi * H + h) * a.nc + c) * Q;
    const int64_t off = rowp - a.dA;
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const int q = lane + 64 * j;
        if (q >= Q) continue;
        a.dA[off + q] = dA[j];
        a.dto[off + q] = v[j];
        if (a.wts) {
            float wv = expf(fminf(total - dA[j], 0.f)) * v[j];
            if (a.seq && (q >= qhi || se[k] < 0 || sq[k][j] != se[k])) wv = 0.f;
            a.wts[off + q] = wv;
        }
    }
    if (a.scl && lane == 0) {
        const bool keep = !a.seq || se[k] == sprev[k];
        a.scl[((int64_t)bi * H + h) * a.nc + c] = keep ? expf(total) : 0.f;
    }
    }
}

}  // namespace m2cum
