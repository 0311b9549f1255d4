// Skinny GEMM for the decode step's projections: y[M, N] = x[M, K] W^T (+ bias),
// M <= 64 (the decode batch), bf16 operands, float32 accumulation.
//
// A decode step reads every projection weight once per token, so these
// products are HBM-bound on the weights (M * K * N MACs for 2 * K * N bytes).
// The weights are K-contiguous ([N, K], the layout torch.nn.functional.linear
// takes).  Up to 16 rows run k_skinny_stream (below) unless K is short;
// k_skinny_gemm takes the rest: each lane loads 8 consecutive k of one output column as one
// 16-byte access, which is exactly a 16x16x32 bf16 MFMA's B-operand fragment.
// One workgroup per 16 output columns (fewer where that leaves CUs idle); its
// 4, 8 or 16 wavefronts (enough for ~2048 over the chip) split K and meet in
// LDS, so every weight byte is read once; x (a few KB) comes from the cache.
// MT = ceil(M / 16) row tiles share each weight fragment.
//
// k_skinny_gemm_norm is the same product for a decode step's first rows
// (M <= 16, M * K <= 32768) whose x is the output of an RMSNorm (optionally SiLU-gated, over
// groups): every workgroup normalises the rows itself into LDS (bf16; a few
// KB read from L2) while its first weight fragments load, so the norm costs no
// launch and no HBM round trip of its output; the epilogue can add the
// (output-dtype rounded) result into a float32 residual stream instead of, or
// besides, storing it -- each output column belongs to one workgroup, so the
// add needs no synchronisation.
#include "conv_ops.h"
#include "norm_ops.h"

namespace {

constexpr int UNROLL = 4;          // k steps of 32 per load batch (two batches in flight)

struct GemmArgs {
    const bf16* x;
    const bf16* w;
    const void* bias;
    void* y;
    int64_t ldx, ldw, ldy;
    int M, N, K;
    int bias_bf16, y_bf16;
    int cw;                 // output columns per workgroup (<= 16)
};

// rows 16 t + 4 (lane >> 4) + i of column n (+ bias): D layout of a 16x16 MFMA
M2_DEV void store_tile(const GemmArgs& a, const f32x4& v, int n, int t) {
    float bv = 0.f;
    if (a.bias)
        bv = a.bias_bf16 ? (float)reinterpret_cast<const bf16*>(a.bias)[n]
                         : reinterpret_cast<const float*>(a.bias)[n];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 16 * t + 4 * ((threadIdx.x & 63) >> 4) + i;
        if (m < a.M) {
            const float r = v[i] + bv;
            if (a.y_bf16) reinterpret_cast<bf16*>(a.y)[(int64_t)m * a.ldy + n] = (bf16)r;
            else reinterpret_cast<float*>(a.y)[(int64_t)m * a.ldy + n] = r;
        }
    }
}

// MT 16-row tiles of x, NW wavefronts splitting K
template <int MT, int NW>
__global__ void __launch_bounds__(NW * 64) k_skinny_gemm(GemmArgs a) {
    __shared__ f32x4 red[NW - 1][MT][64];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int n0 = blockIdx.x * a.cw;
    const int col = lane & 15, kq = (lane >> 4) * 8;   // fragment column / k offset
    const bool colok = col < a.cw;                     // lanes past cw load and store nothing
    const int nb = min(n0 + col, a.N - 1);             // clamped: tail columns are masked on store
    const bf16* wr = a.w + (int64_t)nb * a.ldw;
    // this wavefront's k range, in steps of 32
    const int nsteps = (a.K + 31) / 32;
    const int per = (nsteps + NW - 1) / NW;
    const int s0 = w * per, s1 = min(nsteps, s0 + per);

    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = zero4();
    const bf16x8 zf = {};
    // two load batches (named arrays: register indices must be constants)
    bf16x8 ba[UNROLL], aa[UNROLL][MT], bb[UNROLL], ab[UNROLL][MT];
    auto load = [&](bf16x8 (&bf)[UNROLL], bf16x8 (&af)[UNROLL][MT], int s) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int k = (s + u) * 32 + kq;
            const bool ok = s + u < s1 && k < a.K;
            bf[u] = ok && colok ? *reinterpret_cast<const bf16x8*>(wr + k) : zf;
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int m = 16 * t + col;
                af[u][t] = ok && m < a.M ? *reinterpret_cast<const bf16x8*>(a.x + (int64_t)m * a.ldx + k)
                                         : zf;
            }
        }
    };
    auto mma = [&](const bf16x8 (&bf)[UNROLL], const bf16x8 (&af)[UNROLL][MT]) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[u][t], bf[u], acc[t], 0, 0, 0);
    };
    // the next batch's loads are issued before the current batch's MFMAs
    load(ba, aa, s0);
    for (int s = s0; s < s1; s += 2 * UNROLL) {
        if (s + UNROLL < s1) load(bb, ab, s + UNROLL);
        mma(ba, aa);
        if (s + UNROLL >= s1) break;
        if (s + 2 * UNROLL < s1) load(ba, aa, s + 2 * UNROLL);
        mma(bb, ab);
    }
    // K-split partial sums meet in wavefront 0
    if (w > 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t) red[w - 1][t][lane] = acc[t];
    }
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < NW - 1; ++j) {
            const f32x4 o = red[j][t][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][i] += o[i];
        }
    const int n = n0 + col;
    if (!colok || n >= a.N) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) store_tile(a, acc[t], n, t);
}

// ---------------------------------------------------------------------------
// k_skinny_stream: the same product at up to 16 rows, for a weight stream as
// deep as LDS allows.  A workgroup takes cw columns (CT tiles of 16) and splits K
// over its NW wavefronts; each wavefront keeps the x fragments of its K range in
// registers (2 PU k steps; every column tile reuses them) and streams its part
// of the weights through a ring of D 2 KB units of its own by direct global ->
// LDS loads: 16 columns (or, first, the rows of x) x 64 k, whole 128-byte lines.
// No wavefront waits for
// another before the final sum, and no load result passes through registers, so
// up to D NW 2 KB = 128 KB per CU stay in flight; k_skinny_gemm holds 8 KB per
// wavefront in 64-byte pieces and reads x again for every 16 columns.  Measured
// alone at 16 rows, weights past the cache: 2560 x 10576 22.6 -> 12.2 us (4.4
// TB/s), 5120 x 2560 12.7 -> 8.5, 2560 x 50288 83 -> 53 (4.9 TB/s), 1536 x 6448
// 10.1 -> 6.5, 768 x 3352 4.45 -> 4.1 (of which ~3.5 any kernel takes).
// ---------------------------------------------------------------------------
template <int N> M2_DEV void wait_units(int later) {   // at most `later` <= N units in flight
    if constexpr (N == 0) wait_vmem<0>();
    else if (later >= N) wait_vmem<2 * N>();
    else wait_units<N - 1>(later);
}

template <int CT, int PU, int NW, int D>
__global__ void __launch_bounds__(NW * 64) k_skinny_stream(GemmArgs a) {
    constexpr int NU = (1 + CT) * PU;                  // units of a wavefront: x, then the weights
    __shared__ __align__(16) char ring[NW][D * 2048];
    static_assert(CT * 1024 <= D * 2048, "the partial sums reuse the ring");
    const int lane = threadIdx.x & 63, w = wave_id();
    const int n0 = blockIdx.x * a.cw;
    const int nc = min(a.cw, a.N - n0);                // this workgroup's columns
    const int k0 = w * PU * 64;                        // this wavefront's K range
    const int col = lane & 15, kg = lane >> 4;
    // lane l of load i of a unit brings 16-byte chunk l % 8 (swizzled by the row)
    // of the tile's row 8 i + l / 8; rows past the last column (the last row of x)
    // repeat it, so that every unit is two loads
    const int row = lane >> 3, ch = (lane & 7) ^ row;
    uint32_t vo[1 + CT][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        vo[0][i] = 2 * (uint32_t)(min(8 * i + row, a.M - 1) * a.ldx);
#pragma unroll
        for (int c = 0; c < CT; ++c)
            vo[1 + c][i] = 2 * (uint32_t)(min(16 * c + 8 * i + row, nc - 1) * a.ldw);
    }
    const uint32_t ring_lds = lds_addr(&ring[w][0]);
    const bf16* w0 = a.w + (int64_t)n0 * a.ldw;
    auto issue = [&](int q) {                          // unit q: x or column tile q / PU - 1, 64 k from k
        const int c = q / PU, k = k0 + 64 * (q % PU);
        const bf16* base = c == 0 ? a.x : w0;
        const uint32_t dst = ring_lds + (q % D) * 2048;
        // (chunks past the end of K repeat the last one; masked below)
        const bool whole = k + 64 <= a.K;
        const bf16* src = whole ? base + k : base;
        const uint32_t o = whole ? 16 * ch : 2 * min(k + 8 * ch, a.K - 8);
        dma16s(src, vo[c][0] + o, dst);
        dma16s(src, vo[c][1] + o, dst + 1024);
    };
#pragma unroll
    for (int q = 0; q < (D < NU ? D : NU); ++q) issue(q);
    f32x4 acc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] = zero4();
    const int fo = (col & 7) * 128 + (col >> 3) * 1024;
    const bf16x8 zf = {};
    bf16x8 xf[2 * PU];
#pragma unroll
    for (int q = 0; q < NU; ++q) {
        wait_units<D - 1>(NU - 1 - q);
        const char* u = &ring[w][(q % D) * 2048] + fo;
        bf16x8 bf[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
            bf[ks] = *reinterpret_cast<const bf16x8*>(u + (((4 * ks + kg) ^ (col & 7)) * 16));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (q + D < NU) issue(q + D);                  // the slot just read
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int s = 2 * (q % PU) + ks;
            if (k0 + 32 * s + 8 * kg >= a.K) bf[ks] = zf;        // past the end of K
            if (q < PU) xf[s] = bf[ks];
            else acc[q / PU - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[s], bf[ks], acc[q / PU - 1], 0, 0, 0);
        }
    }
    // the K-split partial sums of tile c meet in wavefront c
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4*>(&ring[w][c * 1024 + 16 * lane]) = acc[c];
    __syncthreads();
    if (w >= CT) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(&ring[0][w * 1024 + 16 * lane]);
#pragma unroll
    for (int j = 1; j < NW; ++j) {
        const f32x4 o = *reinterpret_cast<const f32x4*>(&ring[j][w * 1024 + 16 * lane]);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += o[i];
    }
    if (16 * w + col < nc) store_tile(a, v, n0 + 16 * w + col, 0);
}

constexpr int NORM_MAXM = 16;       // rows of the normalising GEMM (one row tile)
constexpr int NORM_MAXG = 8;        // norm groups per row
constexpr int NORM_MAXX = 32768;    // normalised elements (M x K) held in LDS
constexpr int KEEP = 4;             // chunks a thread keeps through the norm
constexpr int PRE = 2;              // rows whose epilogue operands load with the prologue

struct NormGemmArgs {
    m2conv::UpdArgs cv;     // conv update of columns [conv_lo, conv_lo + cv.D) (CONV)
    int64_t conv_lo;
    m2norm::NormArgs n;     // the rows to normalise (out unused: they go to LDS)
    const bf16* w;
    const void* bias;
    void* y;
    float* res;
    int64_t ldw, ldy, r_rs;
    int M, N, K;
    int bias_bf16, y_bf16;
    int cw;                 // output columns per workgroup (<= 16)
};

template <int NW, bool CONV>
__global__ void __launch_bounds__(NW * 64) k_skinny_gemm_norm(NormGemmArgs a) {
    extern __shared__ __align__(16) bf16 xs[];          // [M][K] normalised rows
    __shared__ f32x4 red[NW - 1][64];
    __shared__ float part[NW][NORM_MAXM * NORM_MAXG];    // per-wavefront sums of squares
    const int lane = threadIdx.x & 63, w = wave_id();
    const int n0 = blockIdx.x * a.cw;
    const int col = lane & 15, kq = (lane >> 4) * 8;
    const bool colok = col < a.cw;                     // lanes past cw load and store nothing
    const int nb = min(n0 + col, a.N - 1);
    const bf16* wr = a.w + (int64_t)nb * a.ldw;
    const int K = a.K, M = a.M;
    const int nsteps = (K + 31) / 32;
    const int per = (nsteps + NW - 1) / NW;
    const int s0 = w * per, s1 = min(nsteps, s0 + per);
    const bf16x8 zf = {};
    bf16x8 ba[UNROLL], bb[UNROLL];
    // the weights are read once per decode step: non-temporal loads leave the
    // cache to the rows and the states (LM decode at batch 1, A/B on one box:
    // 130m 0.506 -> 0.465 ms, 2.7b 2.550 -> 2.517 ms per token; the same in
    // k_skinny_gemm took the 2.7b step at batch 16 from 5.15 to 5.33 ms)
    auto loadw = [&](bf16x8 (&bf)[UNROLL], int s) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int k = (s + u) * 32 + kq;
            bf[u] = s + u < s1 && k < K && colok
                        ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(wr + k)) : zf;
        }
    };
    // the first two weight batches are in flight while the rows are normalised
    // (LM decode at batch 1, A/B on one box: 130m 0.467 -> 0.448 ms per token,
    // 2.7b 2.522 -> 2.533; with only the first batch early the 130m step keeps
    // most of its prologue wait)
    loadw(ba, s0);
    loadw(bb, s0 + UNROLL);

    // what wavefront 0's epilogue reads -- bias, the residual, the conv channel's
    // state row, weights and bias -- is loaded here too, for the first PRE rows:
    // asked for at the end, each would be a memory round trip of the whole kernel
    const int n = n0 + col;
    const bool mine = w == 0 && colok && n < a.N;
    const bool cvn = CONV && n >= a.conv_lo && n < a.conv_lo + a.cv.D;
    const int64_t cc = n - a.conv_lo;                  // conv channel of this column
    float bv = 0.f, pres[PRE] = {}, cw[4] = {}, cb = 0.f;
    float4 pst[PRE];
    if (mine) {
        if (a.bias)
            bv = a.bias_bf16 ? (float)reinterpret_cast<const bf16*>(a.bias)[n]
                             : reinterpret_cast<const float*>(a.bias)[n];
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int m = 4 * (lane >> 4) + i;
            if (m >= M) continue;
            if (cvn) pst[i] = *reinterpret_cast<const float4*>(
                reinterpret_cast<const float*>(a.cv.nstate) + ((int64_t)m * a.cv.D + cc) * 4);
            else if (a.res) pres[i] = a.res[(int64_t)m * a.r_rs + n];
        }
        if (cvn && lane < 16 * ((M + 3) / 4)) m2conv::conv_weights<4>(a.cv, cc, cw, cb);
    }

    // ---- the rows' RMSNorm (as k_rms_norm: same operand / output rounding)
    const m2norm::NormArgs& na = a.n;
    const int G = (int)na.ngroups, gs = (int)na.gs, n4 = gs / 4, NT = NW * 64;
    auto rows = [&](int m, int g, const char*& xr, const char*& zr) {
        xr = reinterpret_cast<const char*>(na.x) + ((int64_t)m * na.x_rs + (int64_t)g * gs) * (na.x_bf16 ? 2 : 4);
        zr = na.z ? reinterpret_cast<const char*>(na.z) + ((int64_t)m * na.z_rs + (int64_t)g * gs) * (na.z_bf16 ? 2 : 4)
                  : nullptr;
    };
    // 1 / rms of (row, group) mg from the wavefronts' sums of squares
    auto inv_rms = [&](int mg) {
        float tot = 0.f;
#pragma unroll
        for (int j = 0; j < NW; ++j) tot += part[j][mg];
        float ms = tot / (float)gs;
        if (na.r_x) ms = m2norm::rbf(ms);
        float den = ms + na.eps;
        if (na.r_x) den = m2norm::rbf(den);
        float rms = sqrtf(den);
        if (na.r_x) rms = m2norm::rbf(rms);
        return 1.f / rms;
    };
    auto wave_sum = [&](float v) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        return v;
    };
    const int MG = M * G, cpr = (n4 + NT - 1) / NT;    // (row, group)s, chunks per thread of each
    if (MG * cpr <= KEEP) {
        // every chunk of the rows and its weights loaded once, at once, and kept
        // in registers from the sum of squares to the scaling (the epilogue's
        // operands come in beside them): slot i holds chunk i % cpr of (row, group)
        // i / cpr.  With the early epilogue operands, decode of 130m at batch 1:
        // 494 -> 474 us per token (73 launches, bit-identical)
        float v[KEEP][4], sz[KEEP][4], wt[KEEP][4];
        int off[KEEP];
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const int mg = i / cpr, c = (i - mg * cpr) * NT + (int)threadIdx.x;
            off[i] = -1;
            if (mg < MG && c < n4) {
                const int m = mg / G, g = mg - m * G;
                const char *xr, *zr;
                rows(m, g, xr, zr);
                off[i] = m * K + g * gs + 4 * c;
                m2norm::ldc<4>(na.w, (int64_t)g * gs + 4 * c, na.w_bf16, na.vec, wt[i]);
                m2norm::operand<4>(na, xr, zr, nullptr, 4 * c, v[i], sz[i]);
            }
        }
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            if (off[i] >= 0) {
#pragma unroll
                for (int k = 0; k < 4; ++k) ss += na.r_x ? m2norm::rbf(v[i][k] * v[i][k]) : v[i][k] * v[i][k];
            }
            const int mg = i / cpr;
            if (mg < MG && i == mg * cpr + cpr - 1) {  // the (row, group)'s last slot
                ss = wave_sum(ss);
                if (lane == 0) part[w][mg] = ss;
                ss = 0.f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (off[i] >= 0) m2norm::output<4>(na, xs, off[i], inv_rms(i / cpr), v[i], sz[i], wt[i]);
    } else {
        for (int m = 0; m < M; ++m)
            for (int g = 0; g < G; ++g) {
                const char *xr, *zr;
                rows(m, g, xr, zr);
                float ss = 0.f;
                for (int c = threadIdx.x; c < n4; c += NT) {
                    float v[4], sz[4];
                    m2norm::operand<4>(na, xr, zr, nullptr, 4 * c, v, sz);
#pragma unroll
                    for (int k = 0; k < 4; ++k) ss += na.r_x ? m2norm::rbf(v[k] * v[k]) : v[k] * v[k];
                }
                ss = wave_sum(ss);
                if (lane == 0) part[w][m * G + g] = ss;
            }
        __syncthreads();
        for (int m = 0; m < M; ++m)
            for (int g = 0; g < G; ++g) {
                const float inv = inv_rms(m * G + g);
                const char *xr, *zr;
                rows(m, g, xr, zr);
                for (int c = threadIdx.x; c < n4; c += NT) {
                    float v[4], sz[4], wt[4];
                    m2norm::ldc<4>(na.w, (int64_t)g * gs + 4 * c, na.w_bf16, na.vec, wt);
                    m2norm::operand<4>(na, xr, zr, nullptr, 4 * c, v, sz);
                    m2norm::output<4>(na, xs + m * K + g * gs, 4 * c, inv, v, sz, wt);
                }
            }
    }
    __syncthreads();

    // ---- y = x' W^T: A fragments from LDS (rows >= M are zero)
    f32x4 acc = zero4();
    auto mma = [&](const bf16x8 (&bf)[UNROLL], int s) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int k = (s + u) * 32 + kq;
            const bf16x8 af = s + u < s1 && k < K && col < M
                                  ? *reinterpret_cast<const bf16x8*>(xs + col * K + k) : zf;
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf[u], acc, 0, 0, 0);
        }
    };
    for (int s = s0; s < s1; s += 2 * UNROLL) {
        if (s > s0 && s + UNROLL < s1) loadw(bb, s + UNROLL);
        mma(ba, s);
        if (s + UNROLL >= s1) break;
        if (s + 2 * UNROLL < s1) loadw(ba, s + 2 * UNROLL);
        mma(bb, s + UNROLL);
    }
    if (w > 0) red[w - 1][lane] = acc;
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int j = 0; j < NW - 1; ++j) {
        const f32x4 o = red[j][lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += o[i];
    }
    if (!mine) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 4 * (lane >> 4) + i;
        if (m < M) {
            float v = acc[i] + bv;
            if (a.y_bf16) v = (float)(bf16)v;        // the output dtype, also for the residual add
            if (cvn) {
                // the decode conv update of this column's channel (width 4, f32
                // state in place): each (row, channel) belongs to this lane only
                float* st = reinterpret_cast<float*>(a.cv.nstate) + ((int64_t)m * a.cv.D + cc) * 4;
                const float4 o = i < PRE ? pst[i < PRE ? i : 0] : *reinterpret_cast<const float4*>(st);
                const float sv[4] = {o.y, o.z, o.w, v};
                *reinterpret_cast<float4*>(st) = make_float4(sv[0], sv[1], sv[2], sv[3]);
                m2conv::conv_store(a.cv, m, cc, m2conv::conv_channel<4>(a.cv, sv, cw, cb));
                continue;
            }
            if (a.y) {
                if (a.y_bf16) reinterpret_cast<bf16*>(a.y)[(int64_t)m * a.ldy + n] = (bf16)v;
                else reinterpret_cast<float*>(a.y)[(int64_t)m * a.ldy + n] = v;
            }
            if (a.res) {
                float* r = a.res + (int64_t)m * a.r_rs + n;
                *r = (i < PRE ? pres[i < PRE ? i : 0] : *r) + v;
            }
        }
    }
}

template <int MT>
void launch_mt(const GemmArgs& k, int64_t ngroups, hipStream_t s) {
    // enough wavefronts to keep the weight stream in flight: >= ~2048 over the
    // chip, each with at least two load batches of k steps
    const int nsteps = (k.K + 31) / 32;
    const dim3 grid((unsigned)ngroups);
    // (16 wavefronts of 1024 threads only for one row tile: more row tiles
    // need more than the 128 registers such a workgroup leaves a lane)
    if (ngroups * 4 >= 2048 || nsteps < 8 * 2 * UNROLL) {
        hipLaunchKernelGGL((k_skinny_gemm<MT, 4>), grid, dim3(4 * 64), 0, s, k);
    } else if constexpr (MT == 1) {
        if (ngroups * 8 >= 2048 || nsteps < 16 * 2 * UNROLL)
            hipLaunchKernelGGL((k_skinny_gemm<1, 8>), grid, dim3(8 * 64), 0, s, k);
        else
            hipLaunchKernelGGL((k_skinny_gemm<1, 16>), grid, dim3(16 * 64), 0, s, k);
    } else {
        hipLaunchKernelGGL((k_skinny_gemm<MT, 8>), grid, dim3(8 * 64), 0, s, k);
    }
}

// Where k_skinny_stream is the faster of the two at up to 16 rows, over 13 K from 64
// to 8192, 10 N from 256 to 50288 and 1 to 16 rows (us k_skinny_gemm /
// k_skinny_stream, weights past the cache).  By N and K alone, so that a row's result
// does not depend on how many rows come with it.
bool stream_faster(const GemmArgs& k, int64_t cus) {
    // two or three column tiles per workgroup, one round of them: from 384 on (4
    // rows: 384 x 6448 4.0 / 3.8, 512 x 10576 5.1 / 4.4; 64 x 6448 2.9 / 3.1)
    if (k.N > 16 * cus && k.N <= 48 * cus) return k.K >= 384;
    // one tile, or several rounds: short K ranges pay neither for 16 wavefronts (4
    // rows: 512 x 2048 3.3 / 3.5, 768 x 3352 3.9 / 3.8) nor for every round's start
    // (64 x 50288 5.4 / 11.3, 512 x 50288 12.8 / 17.0).  From 768 on it depends on
    // the rows, as k_skinny_gemm reads x again for every 16 columns: 768 x 50288 19.3 /
    // 21.9 at 4, 25.9 / 22.4 at 16; so does K 2048, whose rows 4 KB apart meet on the
    // same memory channels: 2048 x 8192 9.4 / 10.0 and 12.0 / 10.3
    return k.K >= 768;
}

// k_skinny_stream for up to 16 rows and K up to 8192 (8 units of x fragments in
// each of 16 wavefronts): false where it does not apply.  8 wavefronts with
// twice the ring each where several column tiles follow each other and a K range
// is at most 6 units; 16 for a single tile, whose loads all go out at once.
// Units of a K range by the wavefronts: 1 to 6 with 8; with 16 4 to 8 (K behind 8
// wavefronts' 48 units), or 1 to 8 for a single tile.
template <int CT, int NW, int D, int PU = (NW == 16 && CT > 1) ? 4 : 1>
bool launch_stream_pu(const GemmArgs& k, int pu, const dim3& grid, hipStream_t s) {
    if constexpr (PU <= (NW == 16 ? 8 : 6)) {
        if (pu != PU) return launch_stream_pu<CT, NW, D, PU + 1>(k, pu, grid, s);
        hipLaunchKernelGGL((k_skinny_stream<CT, PU, NW, D>), grid, dim3(NW * 64), 0, s, k);
        return true;
    }
    return false;
}

bool launch_stream(GemmArgs k, hipStream_t s) {
    const int64_t cus = m2::cu_count();
    if (k.M > 16 || k.K > 8192 || k.ldx >= (1 << 24) || k.ldw >= (1 << 24)) return false;   // 32-bit offsets
    if (!stream_faster(k, cus)) return false;
    // columns per workgroup: as even over whole rounds of the CUs as up to three
    // tiles allow, at least 4
    const int64_t r = (k.N + 48 * cus - 1) / (48 * cus);
    const int64_t cw = (k.N + r * cus - 1) / (r * cus);
    k.cw = (int)(cw < 4 ? 4 : cw);
    const dim3 grid((unsigned)((k.N + k.cw - 1) / k.cw));
    const int ct = (k.cw + 15) / 16, units = (k.K + 63) / 64;
    const int nw = units > 8 * 6 || ct == 1 ? 16 : 8;
    const int pu = (units + nw - 1) / nw;
    if (nw == 16) {
        if (ct == 1) return launch_stream_pu<1, 16, 4>(k, pu, grid, s);
        if (ct == 2) return launch_stream_pu<2, 16, 4>(k, pu, grid, s);
        return launch_stream_pu<3, 16, 4>(k, pu, grid, s);
    }
    if (ct == 2) return launch_stream_pu<2, 8, 8>(k, pu, grid, s);
    return launch_stream_pu<3, 8, 8>(k, pu, grid, s);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Output columns per workgroup: 16 (a full MFMA tile) when that gives at
// least one workgroup per CU, else as few as spread the columns over every CU
// (at least 4): the weight stream then comes in through all the CUs instead
// of a few, e.g. the 2.7b out-projection (N 2560: 160 workgroups of 16
// columns) as 256 workgroups of 10.  MFMA lanes past cw carry zeros.
int cols_per_wg(int64_t N) {
    const int64_t cus = m2::cu_count();
    if ((N + 15) / 16 >= cus) return 16;
    const int64_t cw = (N + cus - 1) / cus;
    return (int)(cw < 4 ? 4 : cw > 16 ? 16 : cw);
}

}  // namespace

namespace m2 {

int launch_skinny_gemm(const m2_skinny_gemm_args& a, hipStream_t s) {
    const char* who = "skinny_gemm";
    M2_REQUIRE(a.x && a.w && a.y, M2_ERR_INVALID, "%s: x, w and y are required", who);
    M2_REQUIRE(a.M >= 1 && a.M <= 64 && a.N >= 1 && a.K >= 8, M2_ERR_INVALID,
               "%s: need 1 <= M <= 64, N >= 1, K >= 8 (got %lld, %lld, %lld)", who,
               (long long)a.M, (long long)a.N, (long long)a.K);
    M2_REQUIRE(a.K % 8 == 0 && a.ldx % 8 == 0 && a.ldw % 8 == 0 && a.ldx >= a.K && a.ldw >= a.K &&
                   a.ldy >= a.N && aligned16(a.x) && aligned16(a.w),
               M2_ERR_UNSUPPORTED,
               "%s: K and the x / w row strides must be multiples of 8 elements on 16-byte "
               "aligned bases", who);
    M2_REQUIRE(a.x_dtype == M2_BF16 && a.w_dtype == M2_BF16, M2_ERR_UNSUPPORTED,
               "%s: x and w must be bf16", who);
    M2_REQUIRE(a.y_dtype == M2_BF16 || a.y_dtype == M2_F32, M2_ERR_UNSUPPORTED, "%s: y dtype %d",
               who, a.y_dtype);
    M2_REQUIRE(!a.bias || a.bias_dtype == M2_BF16 || a.bias_dtype == M2_F32, M2_ERR_UNSUPPORTED,
               "%s: bias dtype %d", who, a.bias_dtype);
    M2_REQUIRE(a.N < (1ll << 35) && a.K < (1 << 30), M2_ERR_UNSUPPORTED, "%s: too large", who);
    GemmArgs k{};
    k.x = reinterpret_cast<const bf16*>(a.x);
    k.w = reinterpret_cast<const bf16*>(a.w);
    k.bias = a.bias; k.y = a.y;
    k.ldx = a.ldx; k.ldw = a.ldw; k.ldy = a.ldy;
    k.M = (int)a.M; k.N = (int)a.N; k.K = (int)a.K;
    k.bias_bf16 = a.bias_dtype == M2_BF16; k.y_bf16 = a.y_dtype == M2_BF16;
    if (launch_stream(k, s)) return check_launch(who);
    k.cw = cols_per_wg(a.N);
    const int64_t ng = (a.N + k.cw - 1) / k.cw;
    if (a.M <= 16) launch_mt<1>(k, ng, s);
    else if (a.M <= 32) launch_mt<2>(k, ng, s);
    else launch_mt<4>(k, ng, s);
    return check_launch(who);
}

int launch_skinny_gemm_norm(const m2_skinny_gemm_norm_args& a, hipStream_t s) {
    const char* who = "skinny_gemm_norm";
    M2_REQUIRE(a.x && a.norm_weight && a.w && (a.y || a.residual), M2_ERR_INVALID,
               "%s: x, norm_weight, w and y or residual are required", who);
    M2_REQUIRE(a.M >= 1 && a.M <= NORM_MAXM && a.N >= 1 && a.K >= 8 && a.M * a.K <= NORM_MAXX,
               M2_ERR_UNSUPPORTED, "%s: need 1 <= M <= %d, M * K <= %d (got %lld, %lld)", who,
               NORM_MAXM, NORM_MAXX, (long long)a.M, (long long)a.K);
    M2_REQUIRE(a.group_size > 0 && a.K % a.group_size == 0 && a.K / a.group_size <= NORM_MAXG,
               M2_ERR_UNSUPPORTED, "%s: K / group_size must be a whole number <= %d", who, NORM_MAXG);
    M2_REQUIRE(a.K % 8 == 0 && a.ldw % 8 == 0 && a.ldw >= a.K && aligned16(a.w) && a.w_dtype == M2_BF16,
               M2_ERR_UNSUPPORTED, "%s: w must be bf16 [N, K] with 16-byte aligned rows", who);
    M2_REQUIRE(!a.y || ((a.y_dtype == M2_BF16 || a.y_dtype == M2_F32) && a.ldy >= a.N),
               M2_ERR_UNSUPPORTED, "%s: y dtype %d", who, a.y_dtype);
    M2_REQUIRE(!a.bias || a.bias_dtype == M2_BF16 || a.bias_dtype == M2_F32, M2_ERR_UNSUPPORTED,
               "%s: bias dtype %d", who, a.bias_dtype);
    M2_REQUIRE(!a.residual || a.residual_row_stride >= a.N, M2_ERR_INVALID,
               "%s: residual row stride", who);
    M2_REQUIRE(a.N < (1ll << 31), M2_ERR_UNSUPPORTED, "%s: too large", who);
    // the norm as m2_rms_norm_gated sees it, storing bf16 (the LDS rows)
    m2_rms_norm_gated_args na{};
    na.x = a.x; na.z = a.z; na.weight = a.norm_weight;
    na.x_row_stride = a.x_row_stride; na.z_row_stride = a.z_row_stride; na.out_row_stride = a.K;
    na.rows = a.M; na.hidden = a.K; na.group_size = a.group_size; na.eps = a.eps;
    na.x_dtype = a.x_dtype; na.z_dtype = a.z_dtype; na.w_dtype = a.norm_weight_dtype;
    na.out_dtype = M2_BF16; na.norm_before_gate = a.norm_before_gate;
    NormGemmArgs k{};
    bool c4;
    if (int rc = prepare_norm(na, k.n, c4, true)) return rc;
    M2_REQUIRE(c4 && k.n.vec, M2_ERR_UNSUPPORTED,
               "%s: the rows need 4-element aligned groups, strides and bases", who);
    k.n.out = nullptr;
    k.w = reinterpret_cast<const bf16*>(a.w); k.bias = a.bias; k.y = a.y; k.res = a.residual;
    k.ldw = a.ldw; k.ldy = a.ldy; k.r_rs = a.residual_row_stride;
    k.M = (int)a.M; k.N = (int)a.N; k.K = (int)a.K;
    // y_dtype is the rounding of the result also when only the residual is written
    M2_REQUIRE(a.y_dtype == M2_BF16 || a.y_dtype == M2_F32, M2_ERR_UNSUPPORTED, "%s: y dtype %d",
               who, a.y_dtype);
    k.bias_bf16 = a.bias_dtype == M2_BF16; k.y_bf16 = a.y_dtype == M2_BF16;
    k.cw = cols_per_wg(a.N);
    const int64_t ng = (a.N + k.cw - 1) / k.cw;
    const int nsteps = (int)((a.K + 31) / 32);
    k.conv_lo = -1;
    if (a.with_conv) {
        const m2_causal_conv1d_update_args& c = a.conv;
        M2_REQUIRE(c.width == 4 && c.state_dtype == M2_F32 && c.new_state == c.conv_state &&
                       c.batch == a.M && a.conv_begin >= 0 && a.conv_begin + c.dim <= a.N &&
                       c.x_dtype == a.y_dtype && aligned16(c.conv_state),
                   M2_ERR_UNSUPPORTED, "%s: the conv update needs width 4, an f32 state updated in "
                   "place, batch M, x_dtype == y_dtype and columns inside N", who);
        if (int rc = prepare_conv_update(c, k.cv, true)) return rc;
        k.conv_lo = a.conv_begin;
    }
    const size_t shm = (size_t)a.M * a.K * 2;
    const dim3 grid((unsigned)ng);
    const bool cv = a.with_conv;
    // as the plain product: enough wavefronts to keep the weight stream in flight
    if (ng * 4 >= 2048 || nsteps < 8 * 2 * UNROLL) {
        if (cv) hipLaunchKernelGGL((k_skinny_gemm_norm<4, true>), grid, dim3(4 * 64), shm, s, k);
        else hipLaunchKernelGGL((k_skinny_gemm_norm<4, false>), grid, dim3(4 * 64), shm, s, k);
    } else if (ng * 8 >= 2048 || nsteps < 16 * 2 * UNROLL) {
        if (cv) hipLaunchKernelGGL((k_skinny_gemm_norm<8, true>), grid, dim3(8 * 64), shm, s, k);
        else hipLaunchKernelGGL((k_skinny_gemm_norm<8, false>), grid, dim3(8 * 64), shm, s, k);
    } else {
        if (cv) hipLaunchKernelGGL((k_skinny_gemm_norm<16, true>), grid, dim3(16 * 64), shm, s, k);
        else hipLaunchKernelGGL((k_skinny_gemm_norm<16, false>), grid, dim3(16 * 64), shm, s, k);
    }
    return check_launch(who);
}

}  // namespace m2
