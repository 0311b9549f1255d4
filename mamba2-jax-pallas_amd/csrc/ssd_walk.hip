// k_ssd_walk: chunk_state + state_passing + chunk_scan of the combined forward
// in one pass for bf16 inputs (head dim 64 or 32, dstate 64 / 128 / 256).
//
//   y[m, :] = exp(dA[m]) C[m, :] bf16(h_c)^T                       (carried state)
//           + sum_{k <= m} CB[m, k] exp(dA[m] - dA[k]) dt[k] x[k, :]  (intra chunk)
//           + D x[m, :],   then y *= silu(z[m, :]) when z is given
//   h_{c+1} = exp(dA[last]) h_c + sum_q w[q] x[q, :]^T B[q, :]
//
// One workgroup walks the chunks (of 64 positions) of one chain -- a (batch,
// head), all 64 head-dim rows, half of them, or a head of 32 -- with the running
// state in MFMA accumulators, so neither the chunk states nor the states entering
// each chunk pass through HBM: x, B, C and dt come in once and y goes out once.
// CB = bf16(C B^T), shared by the heads of a group, is built ahead by k_walk_prep
// in the register layout the walk reads.  Chains too few for the CUs are cut
// into segments (k_seg_states gives each segment's end state from a zero start;
// the walk of a segment combines those before it into its initial state).
//
// 16 wavefronts, one role each, four per SIMD: carry wavefronts 0-3 (row tile t
// of the chunk: C h^T), intra wavefronts 4-7 (row tile T: its T + 1 units of the
// intra-chunk product), state wavefronts 8-11, and data wavefronts 12-15, which
// bring x, B and the chunk's dA / dt / weights by direct global -> LDS loads into
// a ring of R slots and store the y tiles staged in LDS (the sum of the carry and
// the intra wavefronts' tiles).  The compute wavefronts' only vector loads are
// the C rows and CB units of the next chunk, held in a second register set while
// the current one is used; they store nothing, so the compiler can count those
// loads.  One barrier per chunk (A) where the bf16 state and the y tiles fit
// twice beside the ring; else a second one (B) ends every read of them before
// the new ones are written.  The data wavefronts issue between A and B: between
// B and A every other wavefront would wait for them.
//
// What bounds it: with all CUs busy a step (64 positions) at dstate 128 takes
// 1.0 us for half a head, of which the compute alone takes 0.9 and the loads and
// stores alone 1.0 (timing builds without the other); the rows of B and C and
// CB that each workgroup reads from L2 are 37 of its 42 KB.  The layer at 128
// heads, dstate 128, 4096 tokens takes 79 us (2.7 TB/s over its compulsory 223
// MB) against 107 for the state pass and the scan, at 256 heads, dstate 256, 182
// against 276, at 24 heads and 30011 tokens 135 against 364 in 10 segments.
// Chunks of 128 would halve the barriers, but their operands do not fit LDS
// twice at dstate 256.  One wavefront for carry and intra together: 93 against
// 82 us at the first shape; loads issued by two wavefronts: 100.
//
// Follows reference ops/ssd_naive.py:189-318 (chunk_scan), :77-182 (states).
#include <cfloat>
#include <type_traits>

#include "cumsum_tile.h"
#include "m2_internal.h"

namespace {

constexpr int Q = 64;                     // positions per chunk of the walk
constexpr int NWAVES = 16;
constexpr int ND = 4;                     // data wavefronts
constexpr int THREADS = NWAVES * 64;
constexpr float LOG2E = 1.4426950408889634f;
constexpr int LDS_BYTES = 160 * 1024;
// CB units of a chunk (10 of 16 x 16, 64 lanes x 4 bf16 each)
constexpr int CBU = 10 * 256;

typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;

M2_DEV f32x4 mma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
M2_DEV f32x4 mma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
M2_DEV float ex2(float v) { return __builtin_amdgcn_exp2f(v); }
// silu(v) in bf16 (z's dtype), from the hardware exp2 and reciprocal: their last
// bits are far below bf16's, and two role's wavefronts gate every element (the
// full-precision exp and division cost more than the rest of the chunk)
M2_DEV float gate(float v) {
    return (float)(bf16)(v * __builtin_amdgcn_rcpf(1.f + ex2(-v * LOG2E)));
}

// ---------------------------------------------------------------------------
// k_walk_prep: chunk_cumsum (for chunks of 64, with the state weights) and CB in
// one launch: both are a short load -> compute -> store round trip, so running
// them side by side costs little more than the longer one.  The first ncum
// blocks are chunk_cumsum's; block ncum + i builds the CB units of (batch,
// chunk, group) i: the chunk's B and C rows go through LDS, wavefront u < 10
// computes unit (t, kt), kt <= t: lane (ln, kg) holds CB[16 t + ln][16 kt +
// 4 kg + i], i < 4, bf16-rounded, 0 above the diagonal and past the last
// position.  Tile t starts at unit t (t + 1) / 2; its units lie in pairs
// ([lane][unit a, unit b]: one 16-byte load), a last odd one alone.
// ---------------------------------------------------------------------------
struct CbArgs {
    const bf16* B;
    const bf16* C;
    bf16* cb;
    int L, G, N, nc, ncum, nwork;
};

constexpr int PREP_CPW = 2;               // chunks per cumsum block

template <int NS>
M2_DEV void cb_block(const CbArgs& a, int work, char* sm) {
    constexpr int N = 32 * NS, ROW = 2 * N + 16;             // padded row: 8 rows on distinct banks
    constexpr int NL = 2 * Q * N / 8 / m2cum::CUM_THREADS;   // 16-byte loads per thread
    const int g = work % a.G, bc = work / a.G;
    const int c = bc % a.nc, bi = bc / a.nc;
    const int lane = threadIdx.x & 63, u = wave_id();
    const int ln = lane & 15, kg = lane >> 4;
    const int valid = min(Q, a.L - c * Q);
    const int64_t tok0 = (int64_t)bi * a.L + (int64_t)c * Q;
    bf16x8 v[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int e = threadIdx.x + i * m2cum::CUM_THREADS;  // rows 0-63: B, 64-127: C
        const int r = e / (N / 8), col = e % (N / 8);
        const bf16* src = r < Q ? a.B : a.C;
        v[i] = *reinterpret_cast<const bf16x8*>(src + ((tok0 + min(r & (Q - 1), valid - 1)) * a.G + g) * N + 8 * col);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int e = threadIdx.x + i * m2cum::CUM_THREADS;
        *reinterpret_cast<bf16x8*>(sm + e / (N / 8) * ROW + e % (N / 8) * 16) = v[i];
    }
    __syncthreads();
    if (u >= 10) return;                                     // no barrier follows
    const int t = u >= 6 ? 3 : u >= 3 ? 2 : u >= 1 ? 1 : 0;
    const int kt = u - t * (t + 1) / 2;
    const int m = 16 * t + ln;
    f32x4 acc = zero4();
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) {
        const bf16x8 bf = *reinterpret_cast<const bf16x8*>(sm + (16 * kt + ln) * ROW + 64 * ns + 16 * kg);
        const bf16x8 cf = *reinterpret_cast<const bf16x8*>(sm + (Q + m) * ROW + 64 * ns + 16 * kg);
        acc = mma32(bf, cf, acc);
    }
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = 16 * kt + 4 * kg + i;
        w[i] = (k > m || m >= valid) ? 0.f : acc[i];
    }
    const u32x2 p = {pk_bf16(w[0], w[1]), pk_bf16(w[2], w[3])};
    const bool paired = (kt ^ 1) <= t;
    bf16* o = a.cb + (int64_t)work * CBU + (t * (t + 1) / 2 + (kt & ~1)) * 256
            + (paired ? lane * 8 + (kt & 1) * 4 : lane * 4);
    *reinterpret_cast<u32x2*>(o) = p;
}

template <typename TD, int NS>
__global__ void __launch_bounds__(m2cum::CUM_THREADS) k_walk_prep(m2cum::CumsumArgs ca, CbArgs ba) {
    typedef float Tile[PREP_CPW][64][m2cum::HB + 1];
    constexpr int CBS = 2 * Q * (64 * NS + 16);
    __shared__ __align__(16) char sm[CBS > (int)sizeof(Tile) ? CBS : (int)sizeof(Tile)];
    if ((int)blockIdx.x < ba.ncum)
        m2cum::cumsum_block<TD, 1, PREP_CPW>(ca, xcd_remap(blockIdx.x, ba.ncum), *reinterpret_cast<Tile*>(sm));
    else
        cb_block<NS>(ba, xcd_remap(blockIdx.x - ba.ncum, ba.nwork), sm);
}

// ---------------------------------------------------------------------------
// the walk
// ---------------------------------------------------------------------------
struct WalkArgs {
    const bf16* x;
    const bf16* B;
    const bf16* C;
    const bf16* z;
    const bf16* cb;
    const float* dA;       // [b, H, nc, Q]
    const float* dt;
    const float* wts;
    const float* A;        // [H]
    const float* D;
    const float* init;
    float* out;
    float* fin;
    float* segst;          // [b, H, nseg - 1, P, N]: each segment's end state from a zero start
    float* segdec;         // [b, H, nseg - 1]: its decay, prod exp(dA[last])
    int L, H, G, P, nc, D_has_hdim, nwork;
    int cps, nseg;         // chunks per segment, segments of a chain
    int sub;               // the walk's chunks in one of the layer's (cps: a multiple, if nseg > 1)
};

// A > 0 (dA rises): the layer's state weights exp(min(dA[last] - dA, 0)) dt are
// clamped over its own chunks of `sub` of the walk's, while its output is not.
// The state wavefronts of such a head (RISING below) keep two states: the layer's, with
// those weights, and one without the clamp for the outputs inside a chunk.
M2_DEV bool rising(const WalkArgs& a, int h) { return a.sub > 1 && a.A[h] > 0.f; }
// dA over the layer's chunk that starts at the walk's chunk c (dl: the chain's dA[last])
M2_DEV float chunk_total(const float* dl, int c, int sub, int nc) {
    float t = 0.f;
    for (int i = c; i < min(c + sub, nc); ++i) t += dl[(int64_t)i * Q];
    return t;
}

template <int NS, int PT>
struct WCfg {
    static constexpr int N = 32 * NS, PW = 16 * PT;          // dstate, head-dim rows
    static constexpr int XROW = PW * 2, XCPR = XROW / 16;    // x row bytes, 16-byte chunks
    static constexpr int BROW = N * 2, BCPR = BROW / 16;
    static constexpr int XB = Q * XROW, BB = Q * BROW;
    static constexpr int AUXB = 3 * Q * 4;                   // dA, dt, weights
    static constexpr int SLOT = XB + BB + AUXB;
    static constexpr int HS = PW * N * 2;                    // bf16 state
    static constexpr int YT = Q * PW * 4, YS = 2 * YT;       // staged y tiles: carried, intra
    static constexpr int FT = 4 * 64 * 4;                    // decay factors per y wavefront
    // double-buffered state and y tiles (one barrier per chunk) where a ring of
    // two slots still fits beside them: at dstate 128 a whole head with two
    // barriers and three slots took 107 us (128 heads, 4096 tokens) against 98, at
    // dstate 256 halves (256 heads) 282 against 261
    static constexpr bool DB = 2 * SLOT + 2 * (HS + YS) + FT + 256 <= LDS_BYTES;
    static constexpr int NBUF = DB ? 2 : 1;
    static constexpr int FIXED = NBUF * (HS + YS) + FT + 256;
    static constexpr int R = 4 * SLOT + FIXED <= LDS_BYTES ? 4 : 3 * SLOT + FIXED <= LDS_BYTES ? 3 : 2;
    // direct loads per chunk: 1 KB each of x and B (split over the data
    // wavefronts), dA, dt and the weights (256 bytes each; wavefronts 0, 1, 2)
    static constexpr int XL = XB / 1024 / ND, BL = BB / 1024 / ND;
    static constexpr int LPC0 = XL + BL + 1, LPC1 = XL + BL;
    static constexpr int WAIT0 = (R - 2) * LPC0, WAIT1 = (R - 2) * LPC1;
    // state tiles: wavefront s takes row tile s (PT 4, all N columns) or row
    // tile s & 1 and columns (N / 2) (s >> 1) .. (PT 2)
    static constexpr int NH = PT == 4 ? 1 : 2, NT = N / 16 / NH;
    // a data wavefront's first B load starts at pattern 0
    static_assert(BL % (BCPR >= 8 ? (64 / BCPR >= 8 ? 1 : BCPR / 8) : 1) == 0, "B offset patterns");
    static_assert(XB % (1024 * ND) == 0 && BB % (1024 * ND) == 0, "even load split");
    static_assert(R * SLOT + FIXED <= LDS_BYTES, "LDS budget");
    static_assert(WAIT0 <= 63, "vmcnt range");
};

// 16-byte chunk swizzles.  x and B rows are read transposed: 8 consecutive
// rows at one chunk pair (an even mask keeps pairs together); state rows 16
// bytes per lane by 16 consecutive rows at one chunk.
template <int RB> M2_DEV int tswz(int r) {
    return RB == 64 ? ((r >> 2) & 1) << 1 : RB == 128 ? ((r >> 1) & 3) << 1 : (r & 7) << 1;
}
template <int CPR> M2_DEV int sswz(int r) { return CPR == 8 ? ((r >> 1) & 7) : (r & 15); }

template <bool NT> M2_DEV void store_out(const f32x4& v, float* p) {
    if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
    else *reinterpret_cast<f32x4*>(p) = v;
}

// One of the ND data wavefronts' loads of a chunk: a quarter of its x and B rows,
// and (wavefronts 0, 1, 2) its dA, dt or weights.  Lane l of load u brings
// 16-byte chunk 64 u + l of a tile (row, swizzled column).  The address of a
// full chunk's load is a scalar base plus a per-lane offset that repeats from
// load to load (the swizzle's period is 8 rows), so a load costs a few scalar
// instructions; the last, ragged chunk clamps its rows per lane.
template <int NS, int PT>
struct Loader {
    typedef WCfg<NS, PT> S;
    static constexpr int XROW = S::XROW, BROW = S::BROW, XB = S::XB, BB = S::BB;
    static constexpr int XR = 64 / S::XCPR, BR = 64 / S::BCPR;      // rows per load
    static constexpr int BP = BR >= 8 ? 1 : 8 / BR;                 // B offset patterns
    const bf16 *xs, *bs;
    const float* auxp;
    int64_t xst, bst;
    uint32_t ring_lds, xv, bv[BP];
    int L, li, lane;

    M2_DEV Loader(const WalkArgs& a, const char* ring, int bi, int h, int g, int p0, int li_, int lane_)
        : L(a.L), li(li_), lane(lane_) {
        // scalar from here on, so that a load's base needs no v_readfirstlane
        xs = (const bf16*)uniform_ptr(a.x + ((int64_t)bi * a.L * a.H + h) * a.P + p0);
        bs = (const bf16*)uniform_ptr(a.B + ((int64_t)bi * a.L * a.G + g) * S::N);
        xst = (int64_t)a.H * a.P;
        bst = (int64_t)a.G * S::N;
        auxp = (const float*)uniform_ptr((li == 0 ? a.dA : li == 1 ? a.dt : a.wts) + ((int64_t)bi * a.H + h) * a.nc * Q);
        ring_lds = lds_addr(ring);
        xv = 2 * (uint32_t)(lane / S::XCPR * xst + ((lane % S::XCPR) ^ tswz<XROW>(lane / S::XCPR)) * 8);
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int r = lane / S::BCPR;
            bv[q] = 2 * (uint32_t)(r * bst + ((lane % S::BCPR) ^ tswz<BROW>(BR * q + r)) * 8);
        }
    }
    M2_DEV void issue(int c, int k) const {
        const uint32_t sb = ring_lds + k * S::SLOT;
        if ((c + 1) * Q <= L) {
            const bf16* xc = xs + (c * Q + li * S::XL * XR) * xst;
#pragma unroll
            for (int uu = 0; uu < S::XL; ++uu)
                dma16s(xc + uu * XR * xst, xv, sb + 1024 * (li * S::XL + uu));
            const bf16* bc = bs + (c * Q + li * S::BL * BR) * bst;
#pragma unroll
            for (int uu = 0; uu < S::BL; ++uu)
                dma16s(bc + uu * BR * bst, bv[uu % BP], sb + XB + 1024 * (li * S::BL + uu));
        } else {
#pragma unroll 1
            for (int uu = 0; uu < S::XL; ++uu) {
                const int u = li * S::XL + uu, r = u * XR + lane / S::XCPR;
                const int64_t t = min(c * Q + r, L - 1);         // past the end: weight 0
                dma16(xs + t * xst + ((lane % S::XCPR) ^ tswz<XROW>(r)) * 8, sb + 1024 * u);
            }
#pragma unroll 1
            for (int uu = 0; uu < S::BL; ++uu) {
                const int u = li * S::BL + uu, r = u * BR + lane / S::BCPR;
                const int64_t t = min(c * Q + r, L - 1);
                dma16(bs + t * bst + ((lane % S::BCPR) ^ tswz<BROW>(r)) * 8, sb + XB + 1024 * u);
            }
        }
        if (li < 3) dma4s(auxp + c * Q, 4 * lane, sb + XB + BB + li * Q * 4);
    }
};

// The running state h^T of a state wavefront sw: tiles acc[j][i] = h[p][n], p =
// prow (of the chain's rows), n = n0 + 16 j + 4 kg + i.
template <int NS, int PT>
struct StateTiles {
    typedef WCfg<NS, PT> S;
    static constexpr int N = S::N, NT = S::NT, XROW = S::XROW, BROW = S::BROW, XB = S::XB, BB = S::BB;
    static constexpr int NB8 = NT < 8 ? NT : 8;
    f32x4 acc[NT];
    int n0, prow, kg, xo0, bo[NB8];

    M2_DEV StateTiles(int sw, int lane) {
        const int ln = lane & 15, pt = PT == 4 ? sw : (sw & 1);
        kg = lane >> 4;
        n0 = PT == 4 ? 0 : (sw >> 1) * (N / 2);
        prow = 16 * pt + ln;
        // MFMA operand offsets: K step ks covers rows 32 ks .. + 31, MFMA k index
        // j < 4 is row 32 ks + 4 kg + j, j >= 4 is 16 more; the row swizzles repeat
        // every 8 rows (and move chunk bits 1-3: tile j + 8 is tile j moved by 256 bytes)
        const int rA = 4 * kg + (ln >> 2);
        const int c4 = ln & 3, cb8 = 8 * (c4 & 1);
        xo0 = rA * XROW + (((2 * pt + (c4 >> 1)) ^ tswz<XROW>(rA)) * 16) + cb8;
#pragma unroll
        for (int j = 0; j < NB8; ++j)
            bo[j] = XB + rA * BROW + (((n0 / 8 + 2 * j + (c4 >> 1)) ^ tswz<BROW>(rA)) * 16) + cb8;
    }
    // offset of acc[0] in a [.., P, N] state whose row p0 is the chain's first
    M2_DEV int64_t off(int64_t bh, int P, int p0) const { return (bh * P + p0 + prow) * N + n0 + 4 * kg; }
    M2_DEV void zero() {
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = zero4();
    }
    // acc = acc f + src
    M2_DEV void combine(const float* src, float f) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const float4 v = *reinterpret_cast<const float4*>(src + 16 * j);
            acc[j][0] = acc[j][0] * f + v.x; acc[j][1] = acc[j][1] * f + v.y;
            acc[j][2] = acc[j][2] * f + v.z; acc[j][3] = acc[j][3] * f + v.w;
        }
    }
    M2_DEV void store(float* dst) const {
#pragma unroll
        for (int j = 0; j < NT; ++j)
            *reinterpret_cast<float4*>(dst + 16 * j) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
    }
    // the bf16 state into LDS rows [PW][N]
    M2_DEV void publish(char* hs) const {
#pragma unroll
        for (int j = 0; j < NT; ++j) publish(j, acc[j], hs);
    }
    M2_DEV void publish(int j, const f32x4& v, char* hs) const {
        const int n = n0 + 16 * j + 4 * kg;
        const u32x2 p = {pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3])};
        *reinterpret_cast<u32x2*>(hs + prow * (2 * N) + (((n >> 3) ^ sswz<S::BCPR>(prow)) * 16) + 2 * (n & 7)) = p;
    }
    // h <- exp(dA[last]) h + B^T (w x) over the chunk in `slot`; returns exp(dA[last])
    M2_DEV float step(const char* slot) {
        const float* aux = reinterpret_cast<const float*>(slot + XB + BB);
        const float* wt = aux + 2 * Q;
        const float dl = aux[Q - 1];
        float sc = 0.f;
        // the LDS operands of a batch (KSB K steps, JB tiles) are read first,
        // so that the reads' latencies overlap
        constexpr int KSB = NT <= 4 ? 2 : 1, JB = NT == 16 ? 4 : NT;
#pragma unroll
        for (int k0 = 0; k0 < 2; k0 += KSB) {
            float4 wa[KSB], wb[KSB];
            bf16x4 xa[KSB], xb[KSB];
            bf16x8 xh[KSB], xl[KSB];
#pragma unroll
            for (int q = 0; q < KSB; ++q) {
                const int ks = k0 + q;
                wa[q] = *reinterpret_cast<const float4*>(wt + 32 * ks + 4 * kg);
                wb[q] = *reinterpret_cast<const float4*>(wt + 32 * ks + 4 * kg + 16);
                xa[q] = ds_read_tr(slot + xo0 + (32 * ks) * XROW);
                xb[q] = ds_read_tr(slot + xo0 + (32 * ks + 16) * XROW);
            }
#pragma unroll
            for (int j0 = 0; j0 < NT; j0 += JB) {
                bf16x4 ba[KSB][JB], bb[KSB][JB];
#pragma unroll
                for (int q = 0; q < KSB; ++q)
#pragma unroll
                    for (int j = 0; j < JB; ++j) {
                        const int o = bo[(j0 + j) % NB8] + (j0 / 8) * 256 + 32 * (k0 + q) * BROW;
                        ba[q][j] = ds_read_tr(slot + o);
                        bb[q][j] = ds_read_tr(slot + o + 16 * BROW);
                    }
                __builtin_amdgcn_sched_barrier(0);
                if (k0 == 0) {
                    sc = ex2(dl * LOG2E);
#pragma unroll
                    for (int j = 0; j < JB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[j0 + j][r] *= sc;
                }
                if (j0 == 0) {
                    // w x split into packed bf16 hi / lo pairs (two MFMAs): near-fp32
#pragma unroll
                    for (int q = 0; q < KSB; ++q) {
                        const u32x2 pa = __builtin_bit_cast(u32x2, xa[q]), pb = __builtin_bit_cast(u32x2, xb[q]);
                        uint32_t hi[4], lo[4];
                        split2(bf16_lo(pa[0]) * wa[q].x, bf16_hi(pa[0]) * wa[q].y, hi[0], lo[0]);
                        split2(bf16_lo(pa[1]) * wa[q].z, bf16_hi(pa[1]) * wa[q].w, hi[1], lo[1]);
                        split2(bf16_lo(pb[0]) * wb[q].x, bf16_hi(pb[0]) * wb[q].y, hi[2], lo[2]);
                        split2(bf16_lo(pb[1]) * wb[q].z, bf16_hi(pb[1]) * wb[q].w, hi[3], lo[3]);
                        xh[q] = as_bf16x8(hi[0], hi[1], hi[2], hi[3]);
                        xl[q] = as_bf16x8(lo[0], lo[1], lo[2], lo[3]);
                    }
                }
#pragma unroll
                for (int q = 0; q < KSB; ++q)
#pragma unroll
                    for (int j = 0; j < JB; ++j) {
                        const bf16x8 bf = __builtin_shufflevector(ba[q][j], bb[q][j], 0, 1, 2, 3, 4, 5, 6, 7);
                        acc[j0 + j] = mma32(bf, xh[q], acc[j0 + j]);
                        acc[j0 + j] = mma32(bf, xl[q], acc[j0 + j]);
                    }
            }
        }
        return sc;
    }
    // The same for a rising chain, a tile at a time (a second state may be live):
    // out(j, h_j f + B^T (w x)), w = exp(expo(dA)) dt.
    template <typename E, typename O>
    M2_DEV void tiles(const f32x4 (&h)[NT], const char* slot, float f, E expo, O out) const {
        const float* aux = reinterpret_cast<const float*>(slot + XB + BB);
        bf16x8 xh[2], xl[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int q = 32 * ks + 16 * i;
                const float4 d = *reinterpret_cast<const float4*>(aux + q + 4 * kg);
                const float4 t = *reinterpret_cast<const float4*>(aux + Q + q + 4 * kg);
                const u32x2 p = __builtin_bit_cast(u32x2, ds_read_tr(slot + xo0 + q * XROW));
                split2(bf16_lo(p[0]) * (ex2(expo(d.x) * LOG2E) * t.x), bf16_hi(p[0]) * (ex2(expo(d.y) * LOG2E) * t.y),
                       hi[2 * i], lo[2 * i]);
                split2(bf16_lo(p[1]) * (ex2(expo(d.z) * LOG2E) * t.z), bf16_hi(p[1]) * (ex2(expo(d.w) * LOG2E) * t.w),
                       hi[2 * i + 1], lo[2 * i + 1]);
            }
            xh[ks] = as_bf16x8(hi[0], hi[1], hi[2], hi[3]);
            xl[ks] = as_bf16x8(lo[0], lo[1], lo[2], lo[3]);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            const int o = bo[j % NB8] + (j / 8) * 256;
            f32x4 v = h[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= f;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const bf16x4 ba = ds_read_tr(slot + o + 32 * ks * BROW);
                const bf16x4 bb = ds_read_tr(slot + o + (32 * ks + 16) * BROW);
                const bf16x8 bf = __builtin_shufflevector(ba, bb, 0, 1, 2, 3, 4, 5, 6, 7);
                v = mma32(bf, xh[ks], v);
                v = mma32(bf, xl[ks], v);
            }
            out(j, v);
        }
    }
    // the layer's state: total, the dA of the layer's chunk; before, that of its
    // earlier chunks of the walk.  The state takes all of the factor exp(total)
    // (returned) with the layer's chunk's first
    M2_DEV float step_clamped(const char* slot, float total, float before, bool first) {
        const float f = first ? ex2(total * LOG2E) : 1.f;
        tiles(acc, slot, f, [&](float d) { return fminf(total - (d + before), 0.f); },
              [&](int j, const f32x4& v) { acc[j] = v; });
        return f;
    }
    // the unclamped state behind h
    template <typename O> M2_DEV void step_free(const f32x4 (&h)[NT], const char* slot, O out) const {
        const float dl = reinterpret_cast<const float*>(slot + XB + BB)[Q - 1];
        tiles(h, slot, ex2(dl * LOG2E), [&](float d) { return dl - d; }, out);
    }
};

// ---- a carry wavefront (row tile t of the chunk): ysc = exp(dA[m]) C[m, :] h_c^T.
// C rows (and z) are loaded one chunk ahead.
template <int NS, int PT, bool HASZ>
struct CRegs {
    bf16x8 c[NS];
    bf16x4 z[HASZ ? PT : 1];
};
template <int NS, int PT, bool HASZ>
M2_DEV void carry_path(const WalkArgs& a, const char* ring, const char* hs, char* ys, int t,
                       int bi, int h, int g, int p0, int c0, int c1) {
    typedef WCfg<NS, PT> S;
    constexpr int N = S::N, BCPR = S::BCPR;
    const int lane = threadIdx.x & 63;
    const int ln = lane & 15, kg = lane >> 4;
    const int m = 16 * t + ln;                               // this lane's row of the chunk
    const int64_t b0 = (int64_t)bi * a.L, rs = (int64_t)a.G * N;
    const bf16* cbase = a.C + (b0 * a.G + g) * N + 8 * kg;
    typedef CRegs<NS, PT, HASZ> Y;
    auto load = [&](Y& r, int c) {
        const int row = min(c * Q + m, a.L - 1);
        const bf16* cp = cbase + row * rs;
#pragma unroll
        for (int ns = 0; ns < NS; ++ns) r.c[ns] = *reinterpret_cast<const bf16x8*>(cp + 32 * ns);
        if constexpr (HASZ) {
            const bf16* zp = a.z + ((b0 + row) * a.H + h) * a.P + p0 + 4 * kg;
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) r.z[pt] = *reinterpret_cast<const bf16x4*>(zp + 16 * pt);
        }
    };
    auto body = [&](Y& cur, Y& nxt, int c, int k) {
        lds_barrier();                                       // A
        load(nxt, min(c + 1, c1 - 1));
        const float* dAs = reinterpret_cast<const float*>(ring + k * S::SLOT + S::XB + S::BB);
        const float f = ex2(dAs[m] * LOG2E);
        const char* hc = hs + (S::DB ? (c & 1) * S::HS : 0);
        f32x4 cs[PT];
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) cs[pt] = zero4();
        // fragments in batches (their latencies overlap; 4 at dstate 256 for the registers)
        constexpr int NF = PT * NS, BR = NS == 8 ? 4 : NF < 8 ? NF : 8;
#pragma unroll
        for (int f0 = 0; f0 < NF; f0 += BR) {
            bf16x8 sf[BR];
#pragma unroll
            for (int q = 0; q < BR; ++q) {
                const int ns = (f0 + q) / PT, p = 16 * ((f0 + q) % PT) + ln;
                sf[q] = *reinterpret_cast<const bf16x8*>(hc + p * (2 * N) + (((4 * ns + kg) ^ sswz<BCPR>(p)) * 16));
            }
#pragma unroll
            for (int q = 0; q < BR; ++q)
                cs[(f0 + q) % PT] = mma32(sf[q], cur.c[(f0 + q) / PT], cs[(f0 + q) % PT]);
        }
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                cs[pt][i] *= f;
                if (HASZ) cs[pt][i] *= gate((float)cur.z[pt][i]);
            }
        if constexpr (!S::DB) lds_barrier();                 // B
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
            *reinterpret_cast<f32x4*>(ys + (S::DB ? (c & 1) * S::YS : 0) + m * (S::PW * 4) + 16 * ((4 * pt + kg) ^ (ln & (4 * PT - 1)))) = cs[pt];
    };
    Y r0, r1;
    load(r0, c0);
    int k = 0;
    for (int c = c0; c < c1; c += 2) {
        body(r0, r1, c, k);
        k = k + 1 == S::R ? 0 : k + 1;
        if (c + 1 < c1) {
            body(r1, r0, c + 1, k);
            k = k + 1 == S::R ? 0 : k + 1;
        }
    }
    lds_barrier();                                           // the last chunk's y staged
}

// ---- an intra-chunk wavefront (row tile T): ysw = sum_{k <= m} CB exp(dA[m] -
// dA[k]) dt[k] x[k, :] + D x[m, :].  Its CB units are loaded one chunk ahead.
template <int PT, int T, bool HASZ>
struct WRegs {
    u32x4 cb2[(T + 1) / 2 > 0 ? (T + 1) / 2 : 1];   // CB unit pairs
    u32x2 cb1;                                       // the last unit of an odd count
    bf16x4 z[HASZ ? PT : 1];
};
template <int NS, int PT, bool HASZ, int T>
M2_DEV void intra_path(const WalkArgs& a, const char* ring, char* ys, float* ft, const float* Ds,
                       int bi, int h, int g, int p0, int c0, int c1) {
    typedef WCfg<NS, PT> S;
    constexpr int XROW = S::XROW;
    constexpr int NU = T + 1, NPAIR = NU / 2;
    const int lane = threadIdx.x & 63;
    const int ln = lane & 15, kg = lane >> 4;
    const int m = 16 * T + ln;                               // this lane's row of the chunk
    const int64_t b0 = (int64_t)bi * a.L;
    const bf16* cbb = a.cb + ((int64_t)bi * a.nc * a.G + g) * CBU + (T * (T + 1) / 2) * 256;
    typedef WRegs<PT, T, HASZ> Y;
    auto load = [&](Y& r, int c) {
        const bf16* cu = cbb + (int64_t)c * a.G * CBU;
#pragma unroll
        for (int q = 0; q < NPAIR; ++q) r.cb2[q] = *reinterpret_cast<const u32x4*>(cu + q * 512 + lane * 8);
        if constexpr (NU % 2 == 1) r.cb1 = *reinterpret_cast<const u32x2*>(cu + NPAIR * 512 + lane * 4);
        if constexpr (HASZ) {
            const bf16* zp = a.z + ((b0 + min(c * Q + m, a.L - 1)) * a.H + h) * a.P + p0 + 4 * kg;
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) r.z[pt] = *reinterpret_cast<const bf16x4*>(zp + 16 * pt);
        }
    };
    // x^T fragment reads: lane (ln, kg) of a 16-lane group reads row
    // 16 kt + r0 of the group's 4 x 16 block at chunk ch; the row swizzle
    // repeats every 8 rows, so a k-tile moves the offset by 16 rows
    int xo[PT];
    {
        const int r0 = 4 * kg + (ln >> 2);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
            xo[pt] = r0 * XROW + (((2 * pt + ((ln & 3) >> 1)) ^ tswz<XROW>(r0)) * 16) + 8 * (ln & 1);
    }
    const bool fold_d = a.D && !a.D_has_hdim;
    const float dval = fold_d ? Ds[0] : 0.f;

    auto body = [&](Y& cur, Y& nxt, int c, int k) {
        lds_barrier();                                       // A
        load(nxt, min(c + 1, c1 - 1));
        const char* slot = ring + k * S::SLOT;
        const float* dAs = reinterpret_cast<const float*>(slot + S::XB + S::BB);
        const float* dts = dAs + Q;
        // the chunk's decay values and every x fragment are read first, so that
        // the reads' latencies overlap
        const float dAm = dAs[m], dAr = dAs[16 * T];
        const float dl = dAs[lane], tl = dts[lane];
        const float4 dk = *reinterpret_cast<const float4*>(dAs + 16 * T + 4 * kg);
        const float4 tk = *reinterpret_cast<const float4*>(dts + 16 * T + 4 * kg);
        bf16x4 xf[NU][PT];
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) xf[u][pt] = ds_read_tr(slot + u * 16 * XROW + xo[pt]);
        __builtin_amdgcn_sched_barrier(0);
        // Off-diagonal weights CB exp(dA[m] - dA[k]) dt[k] through the tile's first
        // row r, exp(dA[m] - dA[r]) (exp(dA[r] - dA[k]) dt[k]), the second factor one
        // exp per lane from a table: dA is monotonic (dt' >= 0), so neither factor
        // overflows or vanishes before the product does.
        if (T > 0 && lane < 16 * T) ft[lane] = ex2((dAr - dl) * LOG2E) * tl;
        float wv[NU][4];
        auto cbu = [&](int u, float (&v)[4]) {
            uint32_t lo, hi;
            if (u / 2 < NPAIR) { lo = cur.cb2[u / 2][2 * (u & 1)]; hi = cur.cb2[u / 2][2 * (u & 1) + 1]; }
            else { lo = cur.cb1[0]; hi = cur.cb1[1]; }
            v[0] = bf16_lo(lo); v[1] = bf16_hi(lo); v[2] = bf16_lo(hi); v[3] = bf16_hi(hi);
        };
        {   // the diagonal unit: direct weights for k <= m, 0 above (where the
            // exponent may overflow), + D on the diagonal
            const int k0 = 16 * T + 4 * kg;
            const float dkv[4] = {dk.x, dk.y, dk.z, dk.w}, tkv[4] = {tk.x, tk.y, tk.z, tk.w};
            float v[4];
            cbu(T, v);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float e = ex2((dAm - dkv[i]) * LOG2E);
                float r = k0 + i > m ? 0.f : v[i] * e * tkv[i];
                if (k0 + i == m) r += dval;
                wv[T][i] = r;
            }
        }
        if (T > 0) {
            const float e = ex2((dAm - dAr) * LOG2E);
#pragma unroll
            for (int u = 0; u < T; ++u) {
                const float4 f = *reinterpret_cast<const float4*>(ft + 16 * u + 4 * kg);
                float v[4];
                cbu(u, v);
                wv[u][0] = v[0] * f.x * e; wv[u][1] = v[1] * f.y * e;
                wv[u][2] = v[2] * f.z * e; wv[u][3] = v[3] * f.w * e;
            }
        }
        // y^T += x^T W^T, W split into bf16 hi + lo; a pair of units fills the
        // 8 k of a 16x16x32 MFMA
        f32x4 acc[PT];
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) acc[pt] = zero4();
        auto split4 = [&](const float (&v)[4], bf16x4& hi, bf16x4& lo) {
            uint32_t h01, l01, h23, l23;
            split2(v[0], v[1], h01, l01);
            split2(v[2], v[3], h23, l23);
            const u32x2 hv = {h01, h23}, lv = {l01, l23};
            hi = __builtin_bit_cast(bf16x4, hv);
            lo = __builtin_bit_cast(bf16x4, lv);
        };
#pragma unroll
        for (int q = 0; q < NPAIR; ++q) {
            bf16x4 ha, la, hb, lb;
            split4(wv[2 * q], ha, la);
            split4(wv[2 * q + 1], hb, lb);
            const bf16x8 wh = __builtin_shufflevector(ha, hb, 0, 1, 2, 3, 4, 5, 6, 7);
            const bf16x8 wl = __builtin_shufflevector(la, lb, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) {
                const bf16x8 x8 = __builtin_shufflevector(xf[2 * q][pt], xf[2 * q + 1][pt], 0, 1, 2, 3, 4, 5, 6, 7);
                acc[pt] = mma32(x8, wh, acc[pt]);
                acc[pt] = mma32(x8, wl, acc[pt]);
            }
        }
        if constexpr (NU % 2 == 1) {
            bf16x4 wh, wl;
            split4(wv[T], wh, wl);
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) {
                acc[pt] = mma16(xf[T][pt], wh, acc[pt]);
                acc[pt] = mma16(xf[T][pt], wl, acc[pt]);
            }
        }
        if (a.D && a.D_has_hdim) {
#pragma unroll
            for (int pt = 0; pt < PT; ++pt) {
                const int q0 = 16 * pt + 4 * kg;
                const bf16x4 xv = *reinterpret_cast<const bf16x4*>(
                    slot + m * XROW + (((q0 >> 3) ^ tswz<XROW>(m)) * 16) + 2 * (q0 & 7));
                const float4 d4 = *reinterpret_cast<const float4*>(Ds + q0);
                const float dv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[pt][i] += dv[i] * (float)xv[i];
            }
        }
        if constexpr (HASZ) {
#pragma unroll
            for (int pt = 0; pt < PT; ++pt)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[pt][i] *= gate((float)cur.z[pt][i]);
        }
        if constexpr (!S::DB) lds_barrier();                 // B
        // row m of the staged tiles, 16-byte chunk 4 pt + kg, XOR-swizzled by the row
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
            *reinterpret_cast<f32x4*>(ys + (S::DB ? (c & 1) * S::YS : 0) + m * (S::PW * 4) + 16 * ((4 * pt + kg) ^ (ln & (4 * PT - 1)))) = acc[pt];
    };

    Y r0, r1;
    load(r0, c0);
    int k = 0;
    for (int c = c0; c < c1; c += 2) {
        body(r0, r1, c, k);
        k = k + 1 == S::R ? 0 : k + 1;
        if (c + 1 < c1) {
            body(r1, r0, c + 1, k);
            k = k + 1 == S::R ? 0 : k + 1;
        }
    }
    lds_barrier();                                           // the last chunk's y staged
}

// ---- a state wavefront: h_{c+1} from chunk c, published in bf16 for the carry
// wavefronts.
template <int NS, int PT, bool RISING>
M2_DEV void state_path(const WalkArgs& a, const char* ring, char* hs, int sw, int bi, int h, int seg, int p0, int c0, int c1) {
    typedef WCfg<NS, PT> S;
    constexpr int R = S::R, SLOT = S::SLOT;
    int lane = threadIdx.x & 63;
    // keeps the rare path's address registers its own, not live beside the other's
    if constexpr (RISING) asm volatile("" : "+v"(lane));
    StateTiles<NS, PT> st(sw, lane);
    st.zero();
    const int64_t bh = (int64_t)bi * a.H + h;
    if (a.init) st.combine(a.init + st.off(bh, a.P, p0), 0.f);
    for (int i = 0; i < seg; ++i) {                          // the segments before this one
        const int64_t o = bh * (a.nseg - 1) + i;
        st.combine(a.segst + st.off(o, a.P, p0), a.segdec[o]);
    }
    st.publish(hs + (S::DB ? (c0 & 1) * S::HS : 0));
    int k = 0;
    if constexpr (!RISING) {
        for (int c = c0; c < c1; ++c) {
            lds_barrier();                                   // A
            st.step(ring + k * SLOT);
            if constexpr (!S::DB) lds_barrier();             // B
            st.publish(hs + (S::DB ? ((c + 1) & 1) * S::HS : 0));    // h_{c+1}
            k = k + 1 == R ? 0 : k + 1;
        }
    } else {
        // st: the layer's state (c0 starts a chunk of the layer); free: the unclamped
        // one, needed for more than the next chunk only where a chunk of the layer is
        // more than two of the walk's (head dim 32)
        constexpr bool KEEP = PT == 2;
        const float* dl = a.dA + bh * a.nc * Q + Q - 1;
        // before each publish: its addresses are formed anew, kept they would spill
        auto fresh = [&]() { asm volatile("" : "+v"(st.prow), "+v"(KEEP ? st.n0 : st.kg)); };
        f32x4 free[S::NT];
        float total = 0.f, before = 0.f;
        for (int c = c0; c < c1; ++c) {
            const bool first = c % a.sub == 0, last = (c + 1) % a.sub == 0;
            const char* slot = ring + k * SLOT;
            char* const hn = hs + (S::DB ? ((c + 1) & 1) * S::HS : 0);
            if (first) {
                total = chunk_total(dl, c, a.sub, a.nc);
                before = 0.f;
                if constexpr (KEEP) {
#pragma unroll
                    for (int j = 0; j < S::NT; ++j) free[j] = st.acc[j];
                }
            }
            lds_barrier();                                   // A
            if constexpr (!S::DB) lds_barrier();             // B: slots change hands at A only
            if (!last) {
                fresh();
                if constexpr (KEEP) st.step_free(free, slot, [&](int j, const f32x4& v) { free[j] = v; st.publish(j, v, hn); });
                else st.step_free(st.acc, slot, [&](int j, const f32x4& v) { st.publish(j, v, hn); });
            }
            st.step_clamped(slot, total, before, first);
            if (last) {
                fresh();
                st.publish(hn);
            }
            before += dl[(int64_t)c * Q];
            k = k + 1 == R ? 0 : k + 1;
        }
    }
    lds_barrier();
    if (a.fin && seg == a.nseg - 1) st.store(a.fin + st.off(bh, a.P, p0));
}

// (16 wavefronts leave a lane 128 registers: at dstate 256 with whole heads the
// state wavefronts spill 14, 56 bytes of scratch, no other instance any.  The data
// wavefronts must not: a scratch access would count in their waits.)
template <int NS, int PT, bool HASZ, bool NTO>
__global__ void __launch_bounds__(THREADS) k_ssd_walk(WalkArgs a) {
    typedef WCfg<NS, PT> S;
    constexpr int R = S::R, SLOT = S::SLOT, PW = S::PW;
    __shared__ __align__(16) char ring[R * SLOT];
    __shared__ __align__(16) char hs[S::NBUF * S::HS];
    __shared__ __align__(16) char ys[S::NBUF * S::YS];
    __shared__ __align__(16) float ftab[4][64];
    __shared__ __align__(16) float Ds[64];

    // work = ((batch nseg + segment) H + head) (P / PW) + row part: the parts of a head and the
    // heads of a group, which read the same x, B, C and CB, share an XCD
    const int work = xcd_remap(blockIdx.x, a.nwork);
    const int NPART = PT == 4 || a.P == PW ? 1 : 2;
    const int p0 = (work % NPART) * PW;
    const int bsh = work / NPART;
    const int h = bsh % a.H, seg = bsh / a.H % a.nseg, bi = bsh / a.H / a.nseg;
    const int g = h / (a.H / a.G);
    const int c0 = seg * a.cps, c1 = min(a.nc, c0 + a.cps);
    const int lane = threadIdx.x & 63, w = wave_id();
    if (a.D && threadIdx.x < PW) Ds[threadIdx.x] = a.D_has_hdim ? a.D[h * a.P + p0 + threadIdx.x] : a.D[h];
    __syncthreads();

    if (w < 4) {
        carry_path<NS, PT, HASZ>(a, ring, hs, ys, w, bi, h, g, p0, c0, c1);
        return;
    }
    if (w < 8) {
        char* const yw = ys + S::YT;
        switch (w) {
            case 4: intra_path<NS, PT, HASZ, 0>(a, ring, yw, ftab[0], Ds, bi, h, g, p0, c0, c1); break;
            case 5: intra_path<NS, PT, HASZ, 1>(a, ring, yw, ftab[1], Ds, bi, h, g, p0, c0, c1); break;
            case 6: intra_path<NS, PT, HASZ, 2>(a, ring, yw, ftab[2], Ds, bi, h, g, p0, c0, c1); break;
            default: intra_path<NS, PT, HASZ, 3>(a, ring, yw, ftab[3], Ds, bi, h, g, p0, c0, c1); break;
        }
        return;
    }

    if (w >= 12) {
        // ---- the data wavefronts: each brings a quarter of every chunk's loads
        // into its slot (chunk c -> slot (c - c0) % R) and stores a quarter of the
        // y tiles staged between a chunk's barrier B and the next A.
        const int li = w - 12;
        constexpr int CPR = 4 * PT, RPS = 64 / CPR;          // 16-byte chunks per row, rows per store
        float* ob = a.out + ((int64_t)bi * a.L * a.H + h) * a.P + p0;
        const int ch = lane % CPR, r0 = li * RPS + lane / CPR;   // rows r0 + ND RPS it
        constexpr int NIT = Q / RPS / ND, BT = NIT < 4 ? NIT : 4; // stores per chunk, per batch
        auto store = [&](int c) {
            const int valid = a.L - c * Q;
            float* oc = ob + (int64_t)(c * Q + r0) * a.H * a.P + 4 * ch;
            // the reads of a batch first, so that their latencies overlap
#pragma unroll
            for (int b = 0; b < NIT; b += BT) {
                f32x4 u[BT], v[BT];
#pragma unroll
                for (int q = 0; q < BT; ++q) {
                    const int m = r0 + ND * RPS * (b + q);
                    const int o = (S::DB ? (c & 1) * S::YS : 0) + m * (PW * 4) + 16 * (ch ^ (m & 15 & (CPR - 1)));
                    u[q] = *reinterpret_cast<const f32x4*>(ys + o);
                    v[q] = *reinterpret_cast<const f32x4*>(ys + S::YT + o);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < BT; ++q) {
                    const int m = r0 + ND * RPS * (b + q);
                    if (valid >= Q || m < valid)
                        store_out<NTO>(u[q] + v[q], oc + (int64_t)(ND * RPS * (b + q)) * a.H * a.P);
                }
            }
        };
        const Loader<NS, PT> ld(a, ring, bi, h, g, p0, li, lane);
#pragma unroll
        for (int i = 0; i < R - 1; ++i) ld.issue(min(c0 + i, c1 - 1), i);
        int k = R - 1;                                       // the slot of chunk c + R - 1
        for (int c = c0; c < c1; ++c) {
            // the loads of chunk c done: vmcnt counts down in issue order, and
            // behind them came the loads of R - 2 chunks and, from the R-th chunk
            // on, the NIT stores of R - 1 (all of them full chunks: the last one's
            // follow the loop).  Not waiting for the stores too is worth 3 % with a
            // ring of two (128 whole heads at dstate 128: 101 -> 98 us)
            if (c < c0 + R) wait_vmem<S::WAIT1>();
            else if (li < 3) wait_vmem<S::WAIT0 + (R - 1) * NIT>();
            else wait_vmem<S::WAIT1 + (R - 1) * NIT>();
            lds_barrier();                                   // A: chunk c's slot complete, chunk c - 1's free
            // between A and B, where the other wavefronts compute: between B and A
            // they would wait for it
            ld.issue(min(c + R - 1, c1 - 1), k);             // past the end: an unused slot
            if (c > c0) store(c - 1);
            if constexpr (!S::DB) lds_barrier();             // B
            k = k + 1 == R ? 0 : k + 1;
        }
        lds_barrier();
        store(c1 - 1);
        wait_vmem<0>();     // the tail chunks re-loaded into unused slots
        return;
    }

    // ---- the state wavefronts
    if (rising(a, h)) state_path<NS, PT, true>(a, ring, hs, w - 8, bi, h, seg, p0, c0, c1);
    else state_path<NS, PT, false>(a, ring, hs, w - 8, bi, h, seg, p0, c0, c1);
}

// ---------------------------------------------------------------------------
// k_seg_states: the end state of every segment but a chain's last, from a zero
// start, and its decay: the walk of segment s combines those of the segments
// before it into its initial state.  Where there are fewer chains than CUs, the
// segments of a chain run side by side at the price of reading x and B (and
// forming their state products) twice.  4 state and 4 data wavefronts, as in
// the walk; one barrier per chunk.
// ---------------------------------------------------------------------------
template <int NS, int PT>
__global__ void __launch_bounds__(512) k_seg_states(WalkArgs a) {
    typedef WCfg<NS, PT> S;
    constexpr int R = 3;
    __shared__ __align__(16) char ring[R * S::SLOT];
    const int work = xcd_remap(blockIdx.x, a.nwork);         // (b (nseg - 1) + segment) H + head
    const int h = work % a.H, seg = work / a.H % (a.nseg - 1), bi = work / a.H / (a.nseg - 1);
    const int c0 = seg * a.cps, c1 = c0 + a.cps;
    const int lane = threadIdx.x & 63, w = wave_id();
    if (w >= 4) {
        const int li = w - 4;
        const Loader<NS, PT> ld(a, ring, bi, h, h / (a.H / a.G), 0, li, lane);
#pragma unroll
        for (int i = 0; i < R - 1; ++i) ld.issue(min(c0 + i, c1 - 1), i);
        int k = R - 1;
        for (int c = c0; c < c1; ++c) {
            if (li < 3) wait_vmem<(R - 2) * S::LPC0>();
            else wait_vmem<(R - 2) * S::LPC1>();
            lds_barrier();                                   // chunk c's slot complete, chunk c - 1's free
            ld.issue(min(c + R - 1, c1 - 1), k);
            k = k + 1 == R ? 0 : k + 1;
        }
        wait_vmem<0>();
        return;
    }
    StateTiles<NS, PT> st(w, lane);
    st.zero();
    const int64_t bh = (int64_t)bi * a.H + h;
    float dec = 1.f;
    int k = 0;
    if (rising(a, h)) {
        const float* dl = a.dA + bh * a.nc * Q + Q - 1;
        float total = 0.f, before = 0.f;
        for (int c = c0; c < c1; ++c) {
            const bool first = c % a.sub == 0;
            if (first) { total = chunk_total(dl, c, a.sub, a.nc); before = 0.f; }
            lds_barrier();
            dec *= st.step_clamped(ring + k * S::SLOT, total, before, first);
            before += dl[(int64_t)c * Q];
            k = k + 1 == R ? 0 : k + 1;
        }
        // an overflowing factor must not turn a zero state into NaN
        dec = fminf(dec, FLT_MAX);
    } else {
        for (int c = c0; c < c1; ++c) {
            lds_barrier();
            dec *= st.step(ring + k * S::SLOT);
            k = k + 1 == R ? 0 : k + 1;
        }
    }
    const int64_t o = bh * (a.nseg - 1) + seg;
    st.store(a.segst + st.off(o, a.P, 0));
    if (threadIdx.x == 0) a.segdec[o] = dec;
}

}  // namespace

namespace m2 {

// How the walk splits a problem: row parts per head (0: the two-pass path) and
// chunks per segment of a chain.
struct WalkPlan {
    int parts;
    int64_t cps, nseg;
};

// Time of a plan in us, for choosing between plans.  A workgroup's step (one
// chunk) takes c0 + c1 w with w workgroups running side by side (one per CU):
// they share the memory system.  Measured at 4096 tokens, whole heads and
// halves: dstate 64 1.05 / 1.42 us at 128 / 256 workgroups (halves 0.73 /
// 0.89), dstate 128 1.43 / 2.0 (0.86 / 1.0), dstate 256 2.1 / 2.5 (1.6 / 2.0);
// the segment pass 0.5 / 0.8 at 200 / 450 at dstate 128 (two per CU fit).  With
// more than one round of workgroups a last partial round costs as much as a full
// one, and halves 1.35 times more than in step (320 heads at 4096 tokens: 257 us
// whole, 266 halves).  Each round adds its start (first loads in flight), a
// further segment its state's combination; the z gate a third of a step (128
// heads, 4096 tokens: 123 us against 79).
static double walk_cost(int64_t bh, int64_t nc, int64_t cps, int parts, bool half, int dstate, bool z, int64_t cus) {
    static const double step[3][2][2] = {{{0.68, 0.0029}, {0.57, 0.00125}},
                                         {{0.85, 0.0041}, {0.59, 0.0015}},
                                         {{1.70, 0.0032}, {1.20, 0.0031}}};
    static const double pre[3] = {0.7, 0.8, 3.0}, comb[3] = {0.2, 0.35, 1.5};
    const int n = dstate == 64 ? 0 : dstate == 128 ? 1 : 2;
    const int64_t nseg = (nc + cps - 1) / cps;
    const double scale = 256.0 / (double)cus;
    auto rounds = [&](int64_t wg, int64_t cap, double f, double c0, double c1, double late) {
        const int64_t r = (wg + cap - 1) / cap;
        const double st = f * (c0 + c1 * scale * (double)(r > 1 ? cap : wg));
        return r * (2.4 + cps * st * (r > 1 ? late : 1.0));
    };
    const double* c = step[n][half ? 1 : 0];
    double t = 8.0 + rounds(bh * nseg * parts, cus, z ? 1.3 : 1.0, c[0], c[1], half ? 1.35 : 1.05);
    if (nseg > 1)
        t += 4.0 + comb[n] * (double)(nseg - 1)
           + rounds(bh * (nseg - 1), n == 2 ? cus : 2 * cus, pre[n], 0.3, 0.0017, 1.0);
    return t;
}

// The two passes' time: 22 us for their three launches and chunk_cumsum, the
// state pass (states_cost) and the scan at 5.2 TB/s, 4.7 past half a GB (128 heads
// at 4096 tokens 55 us for 289 MB, 512 heads 230 us for 1.09 GB).  Over 110
// shapes (2 to 5120 chains, 38 to 30011 tokens, each dstate, some with z) the
// choice loses 1 % on average against the best of every plan and path; the
// widest gaps it decides: 2 heads x 20000 tokens 43 us against 162 for the two
// passes, 24 x 30011 135 against 364, 256 x 8192 at dstate 256 394 against 485,
// and 320 x 4096 at dstate 128 257 against 239.
static double two_pass_cost(const m2_ssd_combined_args& a) {
    const double x = 2.0 * a.batch * a.seqlen * a.nheads * 64, bc = 4.0 * a.batch * a.seqlen * a.ngroups * a.dstate;
    const double nc = (double)((a.seqlen + a.chunk_size - 1) / a.chunk_size);
    const double by = x * (a.z ? 4.0 : 3.0) + bc + 2.0 * a.batch * nc * a.nheads * 64 * a.dstate;
    return 22.0 + states_cost(a) + by / (by > 5e8 ? 4.7e6 : 5.2e6);
}

static WalkPlan walk_plan(const m2_ssd_combined_args& a) {
    const WalkPlan none{0, 0, 0};
    if (a.dtype != M2_BF16 || (a.headdim != 64 && a.headdim != 32) || a.seq_idx || a.varlen_states) return none;
    if (a.dstate != 64 && a.dstate != 128 && a.dstate != 256) return none;
    if (a.ngroups <= 0 || a.nheads % a.ngroups || a.chunk_size % Q) return none;
    if (a.headdim == 64 && a.chunk_size > 2 * Q) return none;       // state_path's rising chains
    // x and B come by 16-byte direct loads
    if (((uintptr_t)a.x | (uintptr_t)a.B) & 15) return none;
    if (dispatch_override(M2_KNOB_STATES_SPLIT)) return none;
    // dt' >= 0, so that dA is monotonic: the intra-chunk weights' two factors need
    // it, and it leaves the clamp of the state weights to the sign of A (rising())
    if (!(a.dt_max >= 0.f && (a.dt_softplus || a.dt_min >= 0.f))) return none;
    const int64_t nc = (a.seqlen + Q - 1) / Q, ncw = (a.seqlen + a.chunk_size - 1) / a.chunk_size;
    const int64_t bh = a.batch * a.nheads;
    // CB and the segment states lie in the workspace slot of the passed states
    auto fits = [&](int64_t cps) {
        const int64_t nseg = (nc + cps - 1) / cps;
        return 2 * a.batch * nc * a.ngroups * CBU + 512 + 4 * bh * (nseg - 1) * (a.headdim * a.dstate + 1)
               <= 2 * bh * ncw * a.headdim * a.dstate;
    };
    const bool p32 = a.headdim == 32;         // a whole head is what half of one of 64 is
    // chunks per segment: whole chunks of the layer (see rising())
    const int64_t sub = a.chunk_size / Q;
    auto seg_chunks = [&](int64_t seg) { return seg == 1 ? nc : (nc + seg * sub - 1) / (seg * sub) * sub; };
    const int force = dispatch_override(M2_KNOB_LAYER);
    if (force == 3 || !fits(nc)) return none;
    if (force) {
        const int64_t cps = seg_chunks(force >= 4 ? force / 2 : 1);
        if (!fits(cps)) return none;
        return {p32 ? 1 : force >= 4 ? 1 + (force & 1) : force, cps, (nc + cps - 1) / cps};
    }
    WalkPlan best = none;
    double tb = 0.0;
    for (int parts = 1; parts <= (p32 ? 1 : 2); ++parts)
        for (int64_t seg = 1; seg <= 32 && seg <= nc; ++seg) {
            const int64_t cps = seg_chunks(seg);
            // segments only where the chains leave CUs idle
            if (seg > 1 && (cps < 2 || !fits(cps) || bh * parts >= cu_count())) break;
            const double t = walk_cost(bh, nc, cps, parts, p32 || parts == 2, (int)a.dstate, a.z != nullptr, cu_count());
            if (!best.parts || t < tb) { best = {parts, cps, (nc + cps - 1) / cps}; tb = t; }
        }
    // head dim 32 has no two-pass form, the other path is the five staged kernels:
    // 4 x 6814 tokens of 10 heads 137 -> 45 us, 2 x 141 of 208 heads 61 -> 23, and no
    // slower at any of 25 shapes
    return p32 || tb < two_pass_cost(a) ? best : none;
}

int ssd_walk_plan(const m2_ssd_combined_args& a) {
    const WalkPlan p = walk_plan(a);
    return p.parts ? (int)(2 * p.nseg) + p.parts - 1 : 0;
}

int launch_ssd_walk_prep(const m2_ssd_combined_args& a, float* dA, float* dt, float* wts, void* cb,
                         hipStream_t s) {
    M2_REQUIRE(a.dt_dtype == M2_F32 || a.dt_dtype == M2_BF16, M2_ERR_UNSUPPORTED,
               "ssd_walk: dt dtype %d", a.dt_dtype);
    m2cum::CumsumArgs k{};
    k.dt = a.dt; k.A = a.A; k.bias = a.dt_bias;
    k.dA = dA; k.dto = dt; k.wts = wts;
    k.L = (int)a.seqlen; k.H = (int)a.nheads; k.Q = Q; k.nc = (int)((a.seqlen + Q - 1) / Q);
    k.softplus = a.dt_softplus; k.lo = a.dt_min; k.hi = a.dt_max;
    k.nhb = (int)((a.nheads + m2cum::HB - 1) / m2cum::HB);
    CbArgs c{};
    c.B = (const bf16*)a.B; c.C = (const bf16*)a.C; c.cb = (bf16*)cb;
    c.L = k.L; c.G = (int)a.ngroups; c.N = (int)a.dstate; c.nc = k.nc;
    const int64_t ncum = (int64_t)k.nhb * ((k.nc + PREP_CPW - 1) / PREP_CPW) * a.batch;
    const int64_t ncb = a.batch * k.nc * a.ngroups;
    M2_REQUIRE(ncum + ncb < (1ll << 31), M2_ERR_UNSUPPORTED, "ssd_walk: too many blocks");
    k.nblocks = c.ncum = (int)ncum; c.nwork = (int)ncb;
    const unsigned grid = (unsigned)(ncum + ncb);
#define M2_WALK_PREP(NSV)                                                                  \
    {                                                                                      \
        if (a.dt_dtype == M2_F32) k_walk_prep<float, NSV><<<grid, m2cum::CUM_THREADS, 0, s>>>(k, c); \
        else k_walk_prep<bf16, NSV><<<grid, m2cum::CUM_THREADS, 0, s>>>(k, c);             \
    }
    if (a.dstate == 64) M2_WALK_PREP(2)
    else if (a.dstate == 128) M2_WALK_PREP(4)
    else M2_WALK_PREP(8)
#undef M2_WALK_PREP
    return check_launch("ssd_walk (prep)");
}

int launch_ssd_walk(const m2_ssd_combined_args& a, const float* dA, const float* dt,
                    const float* wts, void* cb, hipStream_t s) {
    const WalkPlan p = walk_plan(a);
    M2_REQUIRE(p.parts > 0, M2_ERR_UNSUPPORTED, "ssd_walk: unsupported shape / dtype");
    WalkArgs k{};
    k.x = (const bf16*)a.x; k.B = (const bf16*)a.B; k.C = (const bf16*)a.C; k.z = (const bf16*)a.z;
    k.cb = (const bf16*)cb; k.dA = dA; k.dt = dt; k.wts = wts; k.A = a.A; k.D = a.D; k.init = a.initial_states;
    k.out = a.out; k.fin = a.final_states;
    k.L = (int)a.seqlen; k.H = (int)a.nheads; k.G = (int)a.ngroups;
    k.P = (int)a.headdim; k.nc = (int)((a.seqlen + Q - 1) / Q); k.D_has_hdim = a.D_has_hdim;
    k.cps = (int)p.cps; k.nseg = (int)p.nseg; k.sub = (int)(a.chunk_size / Q);
    const int64_t bh = a.batch * a.nheads, nwork = bh * p.nseg * p.parts;
    M2_REQUIRE(nwork < (1ll << 31), M2_ERR_UNSUPPORTED, "ssd_walk: too many workgroups");
    // behind CB, 256-byte aligned: the segment states, then their decays
    k.segst = (float*)((char*)cb + (2 * a.batch * k.nc * a.ngroups * CBU + 255) / 256 * 256);
    k.segdec = k.segst + bh * (p.nseg - 1) * a.headdim * a.dstate;
    if (p.nseg > 1) {
        k.nwork = (int)(bh * (p.nseg - 1));
        const unsigned g = (unsigned)k.nwork;
#define M2_SEG_L(NSV)                                                                      \
    {                                                                                      \
        if (k.P == 32) k_seg_states<NSV, 2><<<g, 512, 0, s>>>(k);                          \
        else k_seg_states<NSV, 4><<<g, 512, 0, s>>>(k);                                    \
    }
        if (a.dstate == 64) M2_SEG_L(2)
        else if (a.dstate == 128) M2_SEG_L(4)
        else M2_SEG_L(8)
#undef M2_SEG_L
    }
    k.nwork = (int)nwork;
    // outputs up to the 256 MB Infinity Cache are stored non-temporally (they
    // then do not evict the inputs still being read), as in k_scan_q128
    const bool nt = (double)a.batch * a.seqlen * a.nheads * a.headdim * 4 <= 256.0 * (1 << 20);
#define M2_WALK_L(NSV, PTV, ZV)                                                            \
    {                                                                                      \
        if (nt) k_ssd_walk<NSV, PTV, ZV, true><<<(unsigned)nwork, THREADS, 0, s>>>(k);     \
        else k_ssd_walk<NSV, PTV, ZV, false><<<(unsigned)nwork, THREADS, 0, s>>>(k);       \
    }
#define M2_WALK_P(NSV)                                                                     \
    {                                                                                      \
        if (p.parts == 1 && k.P == 64) { if (a.z) M2_WALK_L(NSV, 4, true) else M2_WALK_L(NSV, 4, false) } \
        else { if (a.z) M2_WALK_L(NSV, 2, true) else M2_WALK_L(NSV, 2, false) }            \
    }
    if (a.dstate == 64) M2_WALK_P(2)
    else if (a.dstate == 128) M2_WALK_P(4)
    else M2_WALK_P(8)
#undef M2_WALK_P
#undef M2_WALK_L
    return check_launch("ssd_walk");
}

}  // namespace m2
