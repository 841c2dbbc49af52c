// attention_split.hip — the attention core over long contexts (gqa_attention.rs:327-418 after the prologue), spread
// over the chip: scores by position tiles, the softmax per (head, row), the weighted V sum by slices of the head's
// dimensions. The single-launch core (ops.hip) gives one work-group a whole (head, row): 96 of 256 CUs for a four-row
// launch, each reading its K and V rows alone, bound by the loads one CU keeps in flight. A --spec 3 round's launches
// (four rows, then the MTP's one) with 24 query heads of 256 on 4 K/V heads, mean per launch: at 8,000 positions
// 440 us, here 18 (scores) + 19 (softmax) + 61 (weighted sum); at 1,000 116 us, here 10 + 6 + 12.4. A prompt chunk of
// 64 rows at 2,600 positions: 740 us, here 50 + 35 + 104.
//
// Same arithmetic in the same order: each score is one chain over d from 0 (products and sums rounded one by one),
// each softmax sum the reference's 8 interleaved chains, each output one chain over the positions. Only independent
// chains are spread; none is split.
//
// Products on the matrix cores: a K = 1 f32 matrix product with a zero addend returns each a * b rounded once, which
// is the chain's product; v_mfma_f32_4x4x1_16b gives the 64 x 4 products of a wave's 64 positions (or dimensions)
// with 4 query rows (or probability rows) in one issue, where the vector ALU needs 4, so the vector ALU only adds.
// (A product of -0 comes back as +0: added to a chain that starts at +0 and is never -0, it changes nothing.)
//
// The six query heads that share a K/V head, times the launch's rows, are M vectors over the same K and V rows:
// vector m = row * G + head in the group.
#include "ops.h"
#include "quant_dev.h"

#include <atomic>

namespace aq {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Products of 64 values (a: lane = value) with 4 (b: vector lane & 3) or 16 (vector lane & 15) others.
template <int MG>
__device__ __forceinline__ auto outer(float a, float b) {
    if constexpr (MG == 4) return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, f32x4{}, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, f32x16{}, 0, 0, 0);
}

// m / G for the vector indices (m * G < 2^32), inv = 0xFFFFFFFF / G + 1; G = 1 has inv = 0.
__device__ __forceinline__ int div_g(int m, uint32_t inv) { return inv ? (int)__umulhi((uint32_t)m, inv) : m; }

// ---------------------------------------------------------------------------------------------------- scores
// Work-group: 64 positions x up to WAVES * MG vectors of one K/V head. K rows and query rows pass through the LDS in
// pieces of D dimensions (the next piece's loads in flight in registers); A = K (lane = position), B = the query
// values. MG = 4 (decode and verify batches, 24 vectors at 4 rows): lane (b, j) holds the scores of positions
// 4b .. 4b + 3 for vector j, and D = 128 because few work-groups leave each piece's load latency exposed. MG = 16
// (prompt pieces): v_mfma_f32_16x16x1_4b, lane (g, j) holds positions 16b + 4g + r for vector j, one query read and one
// issue for 16 vectors.
constexpr int SC_P = 64, SC_UNITS = 8; // positions; float4s of a piece per thread
template <int MG>
struct ScShape {
    static constexpr int WAVES = MG == 4 ? 6 : 4, NT = WAVES * 64, PER = WAVES * MG; // threads, vectors
};
constexpr int sc_str(int d) { return d + 4; } // row stride in the LDS: b128 reads without bank conflicts
constexpr int sc_rows(int d, int nt) { return SC_UNITS * nt / (d / 4); } // rows the threads' units fill

template <int MG, int D>
__global__ void __launch_bounds__(ScShape<MG>::NT) attn_scores_kernel(AttnArgs a) {
    using S = ScShape<MG>;
    constexpr int D4 = D / 4, STR = sc_str(D), NT = S::NT;
    static_assert(sc_rows(D, NT) >= SC_P + S::PER, "a piece's units per thread");
    extern __shared__ __align__(16) float sm[]; // sc_rows rows: the 64 K rows, then the query rows (and unread ones)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int G = a.nh / a.nkv, M = G * a.t, kvh = blockIdx.y;
    const uint32_t ginv = 0xFFFFFFFFu / (uint32_t)G + 1u;
    const int m0 = (int)blockIdx.z * S::PER, mn = min(S::PER, M - m0); // this work-group's vectors
    const size_t p0 = (size_t)blockIdx.x * SC_P, total = a.base + a.t;
    if (p0 > a.base + (size_t)((m0 + mn - 1) / G)) return; // uniform: past every row's last position
    const int hd = a.hd;
    // each thread's float4s of a piece (D4 per row); rows past the last vector repeat it
    const float *src[SC_UNITS];
#pragma unroll
    for (int i = 0; i < SC_UNITS; i++) {
        const int u = tid + i * NT, r = u / D4;
        if (r < SC_P) {
            src[i] = a.kcache + min(p0 + (size_t)r, total - 1) * a.stride + (size_t)kvh * hd;
        } else {
            const int m = m0 + min(r - SC_P, mn - 1), row = div_g(m, ginv);
            src[i] = a.q + (size_t)(uint32_t)((row * a.nh + kvh * G + (m - row * G)) * hd);
        }
        src[i] += 4 * (u % D4);
    }
    // narrow launches are short of work-groups to hide a load's latency behind: two pieces in flight from the start
    constexpr bool TWO = MG == 4;
    f32x4 va[SC_UNITS], vb[SC_UNITS];
    auto load = [&](f32x4 (&v)[SC_UNITS], int d0) {
#pragma unroll
        for (int i = 0; i < SC_UNITS; i++) v[i] = *reinterpret_cast<const f32x4 *>(src[i] + d0);
    };
    float acc[MG];
#pragma unroll
    for (float &x : acc) x = 0.0f;
    const bool live = wave * MG < mn;
    const int ml = wave * MG + (lane & (MG - 1)); // this lane's vector
    // its query row in the LDS (clamped: past the end, computed and not written)
    const float *qr = sm + (SC_P + min(ml, mn - 1)) * STR, *kr = sm + lane * STR;
    auto piece = [&](f32x4 (&v)[SC_UNITS], int d0) { // hd % D == 0
        if (d0 > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < SC_UNITS; i++) {
            const int u = tid + i * NT;
            *reinterpret_cast<f32x4 *>(sm + (u / D4) * STR + 4 * (u % D4)) = v[i];
        }
        __syncthreads();
        if (d0 + (TWO ? 2 : 1) * D < hd) load(v, d0 + (TWO ? 2 : 1) * D);
        if (!live) return;
        // steps of 4 dimensions, NB steps' LDS reads in flight ahead of the steps that use them; a rolled loop, since
        // straight-line code over the whole piece runs once per launch and waits on the instruction cache
        constexpr int NB = MG == 4 ? 2 : 1, NS = D / 4 / NB;
        static_assert(NS % 2 == 0, "batches in pairs");
        float4 k4[2][NB], q4[2][NB];
        auto rd = [&](int b, int s) {
#pragma unroll
            for (int e = 0; e < NB; e++) {
                k4[b][e] = *reinterpret_cast<const float4 *>(kr + 4 * (s * NB + e));
                q4[b][e] = *reinterpret_cast<const float4 *>(qr + 4 * (s * NB + e));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto steps = [&](int b) {
#pragma unroll
            for (int e = 0; e < NB; e++) {
                const float4 k = k4[b][e], q = q4[b][e];
                const auto x0 = outer<MG>(k.x, q.x), x1 = outer<MG>(k.y, q.y);
                const auto x2 = outer<MG>(k.z, q.z), x3 = outer<MG>(k.w, q.w);
#pragma unroll
                for (int r = 0; r < MG; r++) acc[r] += x0[r];
#pragma unroll
                for (int r = 0; r < MG; r++) acc[r] += x1[r];
#pragma unroll
                for (int r = 0; r < MG; r++) acc[r] += x2[r];
#pragma unroll
                for (int r = 0; r < MG; r++) acc[r] += x3[r];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        rd(0, 0);
#pragma unroll 1
        for (int s = 0; s < NS; s += 2) {
            rd(1, s + 1);
            steps(0);
            if (s + 2 < NS) rd(0, s + 2);
            steps(1);
        }
    };
    load(va, 0);
    if constexpr (TWO) {
        if (D < hd) load(vb, D);
        for (int d0 = 0; d0 < hd; d0 += 2 * D) {
            piece(va, d0);
            if (d0 + D < hd) piece(vb, d0 + D);
        }
    } else {
        for (int d0 = 0; d0 < hd; d0 += D) piece(va, d0);
    }
    if (ml >= mn) return;
    const int m = m0 + ml, row = div_g(m, ginv);
    float *dst = a.gsc + (size_t)(row * a.nh + kvh * G + (m - row * G)) * a.gsc_stride + p0;
#pragma unroll
    for (int b = 0; b < MG / 4; b++)
        *reinterpret_cast<float4 *>(dst + (MG == 4 ? 4 * (lane >> 2) : 16 * b + 4 * (lane >> 4))) =
            make_float4(acc[4 * b] * a.scaling, acc[4 * b + 1] * a.scaling, acc[4 * b + 2] * a.scaling,
                        acc[4 * b + 3] * a.scaling);
}

// --------------------------------------------------------------------------------------------------- softmax
// softmax.rs:22-49 of one score row in place: max, exp, the sum as 8 interleaved chains (+ the sequential tail),
// divide. One work-group per (head, row); the row passes through the LDS in pieces of SM_N values (a multiple of 8,
// so a chain continues from piece to piece); a row of one piece stays there from the first load to the last store.
constexpr int SM_N = 8192;

__global__ void __launch_bounds__(512) attn_softmax_kernel(AttnArgs a) {
    __shared__ float xs[SM_N], red[16];
    const int h = blockIdx.x, i = blockIdx.y, tid = threadIdx.x;
    constexpr int NT = 512;
    const size_t len = a.base + i + 1;
    float *row = a.gsc + ((size_t)i * a.nh + h) * a.gsc_stride;
    const bool one = len <= (size_t)SM_N;
    float mx = -INFINITY;
    for (size_t t0 = 0; t0 < len; t0 += 8 * NT) { // 8 loads in flight per thread
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const size_t tt = t0 + u * NT + tid;
            v[u] = tt < len ? row[tt] : -INFINITY;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const size_t tt = t0 + u * NT + tid;
            if (one && tt < len) xs[tt] = v[u];
            mx = v[u] > mx ? v[u] : mx;
        }
    }
    for (int off = 32; off >= 1; off >>= 1) {
        const float o = __shfl_xor(mx, off);
        mx = o > mx ? o : mx;
    }
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = red[0];
    for (int w = 1; w < NT / 64; w++) mx = red[w] > mx ? red[w] : mx;
    const size_t n8 = len / 8 * 8;
    float part = 0.0f; // chain tid (tid < 8)
    for (size_t c0 = 0; c0 < len; c0 += SM_N) {
        const int n = (int)(len - c0 < (size_t)SM_N ? len - c0 : (size_t)SM_N);
        if (c0 > 0) __syncthreads(); // the chains have read the previous piece
        for (int e = tid; e < n; e += NT) {
            const float v = exp_f((one ? xs[e] : row[c0 + e]) - mx);
            xs[e] = v;
            if (!one) row[c0 + e] = v;
        }
        __syncthreads();
        if (tid < 8) part = seq_sum<false>(xs, tid, n / 8 * 8, 8, part);
    }
    __syncthreads();
    if (tid < 8) red[tid] = part;
    __syncthreads();
    if (tid == 0) {
        float s = reduce8_f(red);
        for (size_t e = n8; e < len; e++) s += xs[e % SM_N]; // the last piece is still in the LDS
        red[8] = s;
    }
    __syncthreads();
    const float ssum = red[8];
    for (size_t tt = tid; tt < len; tt += NT) row[tt] = (one ? xs[tt] : row[tt]) / ssum;
}

// ---------------------------------------------------------------------------------------------- weighted sum
// Work-group: DS dimensions of one K/V head x 4 waves of vectors. The V rows' slice and the vectors' probability rows
// stream through a ring of direct global-to-LDS copies, T positions a stage, RING - 1 stages ahead; every wave
// issues the same number of copies per stage, so its count of outstanding copies tells that a stage has landed.
//
// NARROW (decode and verify batches): 32 dimensions x 8 vectors, a wave 32 x 2, one chain per lane, so as many waves
// as there are chains of 64. A chain is len adds long whatever the split, so its wave's issue bounds it (two vector
// instructions, half an LDS read and the waits: 17 cycles per position); 32 dimensions rather than 64 halve the V bytes
// a CU takes in per position, which bound it before (35 cycles). Else (prompt pieces, more chains than the chip has
// lanes): 64 dimensions x 32 vectors, a wave 64 x 8, products on the matrix cores, lane (b, j) = dimensions 4b .. 4b + 3
// of vectors j and 4 + j.
template <bool NARROW>
struct VsShape {
    static constexpr int T = NARROW ? 256 : 64, DS = NARROW ? 32 : 64, MW = NARROW ? 2 : 8, RING = NARROW ? 3 : 5;
    static constexpr int PSTR = T + 4;                       // a vector's probabilities in a stage
    static constexpr int STAGE = T * DS + 4 * MW * PSTR;     // floats
    static constexpr int LPP = DS / 4, PPC = 64 / LPP;       // lanes per position, positions per copy
    static constexpr int NV = T / PPC / 4, NDMA = NV + MW;   // copies per wave and stage
    static_assert((RING - 2) * NDMA <= 63, "the outstanding-copy counter's range");
};

__device__ __forceinline__ void vs_dma16(uint32_t lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void vs_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <bool NARROW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) attn_wsum_kernel(AttnArgs a) {
    using S = VsShape<NARROW>;
    constexpr int DS = S::DS, MW = S::MW, RING = S::RING, T = S::T, NV = S::NV, LPP = S::LPP, PPC = S::PPC;
    extern __shared__ __align__(16) float sm[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.nh / a.nkv, M = G * a.t, hd = a.hd, nslice = hd / DS;
    // the slabs (K/V head, slice) vary fastest over the grid, so the work-groups that read one slab of V run on one
    // XCD (work-group i on XCD i mod 8) when the slab count is a multiple of 8
    const int slab = (int)blockIdx.x, kvh = slab / nslice, d0 = (slab % nslice) * DS;
    const int mg = (int)blockIdx.y * 4 * MW, mw = mg + wave * MW; // the work-group's and the wave's first vector
    const uint32_t glen = (uint32_t)a.base + (uint32_t)((min(mg + 4 * MW, M) - 1) / G) + 1; // its longest row
    const int nst = (int)((glen + T - 1) / T);
    const uint32_t lds0 = (uint32_t)(uintptr_t)sm;
    // a copy: PPC positions x DS dimensions of V (lane = position, float4), or T probabilities of a vector
    const float *vsrc = a.vcache + (size_t)kvh * hd + d0 + 4 * (lane % LPP);
    const uint32_t vrow = (uint32_t)(wave * NV * PPC + lane / LPP), stride = (uint32_t)a.stride;
    const float *vp = vsrc + (uint64_t)vrow * stride;
    const float *prow[MW]; // the wave's probability rows (clamped: past the end, computed and not written)
#pragma unroll
    for (int k = 0; k < MW; k++) {
        const int m = min(mw + k, M - 1);
        prow[k] = a.gsc + ((size_t)(m / G) * a.nh + (size_t)kvh * G + m % G) * a.gsc_stride;
    }
    uint32_t it0 = 0, ibuf = lds0; // the next stage to issue: its first position and its place
    const uint32_t lend = lds0 + RING * S::STAGE * 4, plast = (uint32_t)a.gsc_stride - 4;
    auto issue = [&]() {
        const uint32_t vb = ibuf + (uint32_t)(wave * NV * PPC * DS * 4);
        if (it0 + T <= glen) {
#pragma unroll
            for (int i = 0; i < NV; i++) vs_dma16(vb + (uint32_t)(i * PPC * DS * 4), vp + (uint64_t)(i * PPC) * stride);
        } else { // the last stage: positions past the end are clamped, read and not added
#pragma unroll
            for (int i = 0; i < NV; i++)
                vs_dma16(vb + (uint32_t)(i * PPC * DS * 4),
                         vsrc + (uint64_t)min(it0 + vrow + (uint32_t)(i * PPC), glen - 1) * stride);
        }
        if (lane < T / 4) {
            const uint32_t tp = min(it0 + 4u * (uint32_t)lane, plast);
#pragma unroll
            for (int k = 0; k < MW; k++)
                vs_dma16(ibuf + (uint32_t)((T * DS + (wave * MW + k) * S::PSTR) * 4), prow[k] + tp);
        }
        vp += (uint64_t)T * stride;
        it0 += T;
        ibuf = ibuf + S::STAGE * 4 == lend ? lds0 : ibuf + S::STAGE * 4;
    };
#pragma unroll 1
    for (int s = 0; s < RING - 1; s++)
        if (s < nst) issue();
    float acc[NARROW ? 1 : MW];
#pragma unroll
    for (float &x : acc) x = 0.0f;
    // the lane's vectors' row lengths (positions past a row's end are not added), and the positions every vector of
    // the wave takes (rows grow with the vector's index): whole stages up to there need no guard
    uint32_t mylen[NARROW ? 1 : 2];
    if constexpr (NARROW) {
        mylen[0] = (uint32_t)a.base + (uint32_t)(min(mw + (lane >> 5), M - 1) / G) + 1;
    } else {
#pragma unroll
        for (int k = 0; k < 2; k++) mylen[k] = (uint32_t)a.base + (uint32_t)(min(mw + 4 * k + (lane & 3), M - 1) / G) + 1;
    }
    const uint32_t full = (uint32_t)a.base + (uint32_t)(min(mw, M - 1) / G) + 1;
    const uint32_t wend = (uint32_t)a.base + (uint32_t)((min(mw + MW, M) - 1) / G) + 1; // the longest
    const int voff = NARROW ? lane & 31 : lane, poff = T * DS + (wave * MW + (NARROW ? lane >> 5 : lane & 3)) * S::PSTR;
    int rbuf = 0; // the stage being read, in floats
    for (int st = 0; st < nst; st++) {
        if (st + RING - 2 < nst) vs_wait_barrier<(RING - 2) * S::NDMA>();
        else vs_wait_barrier<0>();
        if (st + RING - 1 < nst) issue();
        const float *V = sm + rbuf + voff, *P = sm + rbuf + poff;
        rbuf = rbuf + S::STAGE == RING * S::STAGE ? 0 : rbuf + S::STAGE;
        const uint32_t t0 = (uint32_t)st * T;
        // batches of B positions: the next one's LDS reads are in flight while this one's chains run
        constexpr int B = 16;
        float v[2][B], p1[2], p8[2][NARROW ? 1 : 2][NARROW ? 1 : B];
        auto rd = [&](int b, int u0) {
#pragma unroll
            for (int u = 0; u < B; u++) v[b][u] = V[(u0 + u) * DS];
            if constexpr (NARROW) {
                p1[b] = P[u0 + (lane & 15)]; // each row of 16 lanes holds its vector's 16 probabilities
            } else {
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int u = 0; u < B; u += 4) {
                        const float4 p4 = *reinterpret_cast<const float4 *>(P + k * 4 * S::PSTR + u0 + u);
                        p8[b][k][u] = p4.x;
                        p8[b][k][u + 1] = p4.y;
                        p8[b][k][u + 2] = p4.z;
                        p8[b][k][u + 3] = p4.w;
                    }
            }
        };
        auto chains = [&](int b) {
            if constexpr (NARROW) {
                // the product reads the row's lane u (DPP row broadcast): one LDS read of 16 probabilities per batch
                float x[B];
#define AQ_VS(U) x[U] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(p1[b]), 0x150 + U, 0xF, 0xF, true)) * v[b][U];
                AQ_VS(0) AQ_VS(1) AQ_VS(2) AQ_VS(3) AQ_VS(4) AQ_VS(5) AQ_VS(6) AQ_VS(7)
                AQ_VS(8) AQ_VS(9) AQ_VS(10) AQ_VS(11) AQ_VS(12) AQ_VS(13) AQ_VS(14) AQ_VS(15)
#undef AQ_VS
#pragma unroll
                for (int u = 0; u < B; u++) acc[0] += x[u];
            } else {
#pragma unroll
                for (int u = 0; u < B; u += 4) {
                    f32x4 x[4], y[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        x[e] = outer<4>(v[b][u + e], p8[b][0][u + e]);
                        y[e] = outer<4>(v[b][u + e], p8[b][NARROW ? 0 : 1][u + e]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            acc[r] += x[e][r];
                            acc[4 + r] += y[e][r];
                        }
                }
            }
        };
        if (t0 + T <= full) {
            rd(0, 0);
#pragma unroll
            for (int g = 0; g < T / B; g++) {
                if (g + 1 < T / B) rd((g + 1) & 1, (g + 1) * B);
                __builtin_amdgcn_sched_barrier(0);
                chains(g & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else { // the wave's rows end inside the stage: whole batches, then the positions where their ends differ
            const int nf = full > t0 ? (int)(full - t0) / B : 0;
#pragma unroll 1
            for (int g = 0; g < nf; g++) {
                rd(0, g * B);
                chains(0);
            }
            const int ne = wend > t0 ? (int)min(wend - t0, (uint32_t)T) : 0;
#pragma unroll 1
            for (int u = nf * B; u < ne; u++) {
                if constexpr (NARROW) {
                    const float s = acc[0] + P[u] * V[u * DS];
                    acc[0] = t0 + (uint32_t)u < mylen[0] ? s : acc[0];
                } else {
                    const f32x4 x = outer<4>(V[u * DS], P[u]), y = outer<4>(V[u * DS], P[4 * S::PSTR + u]);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float s0 = acc[r] + x[r], s1 = acc[4 + r] + y[r];
                        acc[r] = t0 + (uint32_t)u < mylen[0] ? s0 : acc[r];
                        acc[4 + r] = t0 + (uint32_t)u < mylen[1] ? s1 : acc[4 + r];
                    }
                }
            }
        }
    }
    // times the sigmoid output gate
#pragma unroll
    for (int k = 0; k < (NARROW ? 1 : 2); k++) {
        const int m = mw + (NARROW ? lane >> 5 : 4 * k + (lane & 3));
        if (m >= M) continue;
        const size_t i = (size_t)(m / G), h = (size_t)kvh * G + m % G;
        const float *gate = a.qg + i * 2 * a.nh * hd + h * 2 * hd + hd;
        float *out = a.out + (i * a.nh + h) * hd;
        if constexpr (NARROW) {
            const int d = d0 + (lane & 31);
            out[d] = acc[0] * sigmoid_f(gate[d]);
        } else {
            const int d = d0 + 4 * (lane >> 2);
            const float4 g4 = *reinterpret_cast<const float4 *>(gate + d);
            *reinterpret_cast<float4 *>(out + d) =
                make_float4(acc[4 * k] * sigmoid_f(g4.x), acc[4 * k + 1] * sigmoid_f(g4.y),
                            acc[4 * k + 2] * sigmoid_f(g4.z), acc[4 * k + 3] * sigmoid_f(g4.w));
        }
    }
}

// Allow a kernel more than 64 KB of dynamic LDS, once per kernel and device.
int raise_lds(const void *kernel, size_t lds, std::atomic<uint64_t> &raised) {
    int dev = 0;
    AQ_HIP(hipGetDevice(&dev));
    const uint64_t bit = 1ull << (dev & 63);
    if (lds <= 64 * 1024 || (raised.load() & bit)) return 0;
    AQ_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    raised.fetch_or(bit);
    return 0;
}

template <bool NARROW>
int launch_wsum(const AttnArgs &a, int M, hipStream_t stream) {
    using S = VsShape<NARROW>;
    static std::atomic<uint64_t> raised{0};
    const dim3 grid((unsigned)(a.nkv * (a.hd / S::DS)), (unsigned)((M + 4 * S::MW - 1) / (4 * S::MW)));
    const size_t lds = (size_t)S::RING * S::STAGE * sizeof(float);
    const int rc = raise_lds(reinterpret_cast<const void *>(attn_wsum_kernel<NARROW>), lds, raised);
    if (rc) return rc;
    hipLaunchKernelGGL(attn_wsum_kernel<NARROW>, grid, dim3(256), lds, stream, a);
    return 0;
}

int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(AQ_EHIP, std::string(what) + " launch: " + hipGetErrorString(e));
}

} // namespace

// From ATTN_SPLIT_MIN positions: the four launches after the prologue cost nearly the same at any length near there, the
// single-launch core's time grows with it. 24 heads of 256 on 4 at 256 positions: 1 row 20.6 us (scores 8.5, softmax 3.9,
// weighted sum 5.4, quantiser 2.8), 4 rows 22, 8 rows 23.4 against 32.5 in one launch (24.5 at 192 positions, 47 at 448);
// 6 heads on 1 the same. In decode steps and verify batches (1, 2, 4 and 8 rows, five head shapes) the two cross between
// 115 and 165 positions, so 256 is past it for all of them. A chunk of 64 rows: 50 us against 103; 45 against 45 with 6
// heads on 1 K/V head. Of 16 rows: 43 against 42 at 256 positions, 51 against 62 at 448.
bool attn_split_fits(const AttnArgs &a) {
    const auto al16 = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    return a.gsc && a.base + a.t >= (size_t)ATTN_SPLIT_MIN && a.hd % 64 == 0 && a.stride % 4 == 0 && a.gsc_stride % 64 == 0 &&
           (a.base + a.t + 63) / 64 * 64 <= a.gsc_stride && al16(a.kcache) && al16(a.vcache) && al16(a.q) &&
           al16(a.qg) && al16(a.out) && al16(a.gsc) && a.nkv <= 65535 && a.t <= 4096 && a.base < (1u << 30);
}

int launch_attention_split(const AttnArgs &a, hipStream_t stream) {
    AQ_REQUIRE(attn_split_fits(a), "attention: shape not built for the split core");
    const int G = a.nh / a.nkv, M = G * a.t;
    const size_t total = a.base + a.t;
    int rc;
    {
        // four vectors per wave and six waves (the 24 vectors of a --spec 3 verify; waves without vectors load); a
        // prompt piece's many vectors take 16 per wave, four waves, so a K tile is read M / 64 times. Up to 48 vectors
        // (8 rows of 6 heads) the narrow form is always the faster (24 vectors: 10.3 against 16.9 us at 256 positions);
        // at 384 vectors 18.8 against 18.2 at 256 positions, 42 against 27 at 1,000. In between the wide form is taken
        // and loses up to 7 us on short contexts (96 vectors: 10.6 against 17.4 at 256 positions, 12.1 against 18.0 at
        // 1,000).
        const bool wide = M > 48;
        const int nt = wide ? ScShape<16>::NT : ScShape<4>::NT, per = wide ? ScShape<16>::PER : ScShape<4>::PER;
        const int d = !wide && a.hd % 128 == 0 ? 128 : 64;
        const dim3 grid((unsigned)((total + SC_P - 1) / SC_P), (unsigned)a.nkv, (unsigned)((M + per - 1) / per));
        const size_t lds = (size_t)sc_rows(d, nt) * sc_str(d) * sizeof(float);
        if (wide) hipLaunchKernelGGL((attn_scores_kernel<16, 64>), grid, dim3(nt), lds, stream, a);
        else if (d == 128) hipLaunchKernelGGL((attn_scores_kernel<4, 128>), grid, dim3(nt), lds, stream, a);
        else hipLaunchKernelGGL((attn_scores_kernel<4, 64>), grid, dim3(nt), lds, stream, a);
        if ((rc = launched("attention scores"))) return rc;
    }
    hipLaunchKernelGGL(attn_softmax_kernel, dim3((unsigned)a.nh, (unsigned)a.t), dim3(512), 0, stream, a);
    if ((rc = launched("attention softmax"))) return rc;
    // one chain per lane until the waves outnumber the SIMDs, then eight per lane: 49,152 chains (8 rows of 24 heads on 4)
    // 5.8 us against 16.3 at 256 positions, 12.5 against 43.7 at 1,000; 393,216 (64 rows) 28.3 against 18.8 and 61
    // against 47. Just past the line the one-chain form would still be the faster (98,304: 10.7 against 17 and 21
    // against 44).
    rc = (size_t)M * a.nkv * a.hd > 64 * 1024 ? launch_wsum<false>(a, M, stream) : launch_wsum<true>(a, M, stream);
    if (rc) return rc;
    if ((rc = launched("attention weighted sum"))) return rc;
    if (a.out_q8k) return launch_q8k_quantize(a.q8k, (size_t)a.t, a.out, (size_t)a.nh * a.hd, stream);
    return 0;
}

} // namespace aq
