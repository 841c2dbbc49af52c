// kq_q8f.hip — K-quant weights x Q8_0 activations: the reference's opt-in `--q8-fine` form (matvec.rs:127-160
// `set_q8_fine` / `act_kind`, dot.rs:69-160 `dot_q4_k_q8` / `dot_q5_k_q8` / `dot_q6_k_q8`).
//
// Arithmetic (per weight row and activation column, no FMA): for every 32-element sub-block s of super-block sb,
// against the activation's Q8_0 block xb = 8 sb + s, eight exact i32 lanes p32[i] = sum over elements 4i..4i+3 of
// code * x; Q6_K takes its -32 offset in integer from lane 0 (32 * sum x[0..16]) and lane 4 (32 * sum x[16..32]).
// Then acc[i] += f32(p32[i]) * (d32[xb] * (d * sc)) with sc the sub-block scale (Q6_K: the group scale of lanes 0..3
// or 4..7), in sub-block order; Q4_K / Q5_K also accm[s] += (m[s] * -dmin) * (d32[xb] * f32(sum x[xb])) in
// super-block order. The result is reduce8(acc) [+ reduce8(accm)], reduce8(v) = ((v0+v4)+(v2+v6)) + ((v1+v5)+(v3+v7)).
//
// Mapping, one short column (more, or a long one: the block kernel below). Thread (row, lane l) runs the chains acc[l]
// and accm[l] of its row, super-blocks in order. Its weight bytes are one 16-byte load of the tile plane per super-block
// (the lane's 4 codes of all 8 sub-blocks) plus the row's scales; its activation codes are the 4 bytes 4l..4l+3 of each
// Q8_0 block, read from the natural-order code plane (the same buffer the Q8_0 / Q4_0 kernels read). A 64-lane wave
// holds 8 rows x 8 lanes; the 8 lanes of a row are adjacent, so the Q6_K half-block sums (4 lanes) are two DPP adds and
// the final reduce8 is three exchanges within the row's 8 lanes, in the reference's pairing. 256 threads = 32 rows.
#include "aq_common.h"
#include "quant_dev.h"

namespace aq {
namespace {

constexpr int Q8F_ROWS = 32; // rows per 256-thread work-group

struct Q8fArgs {
    const uint8_t *qa, *qb, *sc, *dm;
    int rows, nb; // weight rows; super-blocks per row
    const int8_t *xq;  // ncols x n codes, natural order
    const float *xd;   // ncols x nb32 block scales (the f16 widened)
    const int32_t *xs; // ncols x nb32 code sums
    size_t n, nb32;
    int ncols;
    float *y;
    const float *resid;
};

__device__ __forceinline__ float f16lo(uint32_t w) {
    _Float16 f;
    const uint16_t h = (uint16_t)(w & 0xFFFF);
    __builtin_memcpy(&f, &h, 2);
    return (float)f;
}

__device__ __forceinline__ int sdot4(uint32_t a, uint32_t b) { return __builtin_amdgcn_sdot4((int)a, (int)b, 0, false); }

// quant.rs:45-51 get_scale_min_k4 over the 12 packed bytes (words w1..w3 of the row's 16-byte scale record).
__device__ __forceinline__ void scales_k4(uint32_t w1, uint32_t w2, uint32_t w3, int sc[8], int mn[8]) {
    const uint8_t q[12] = {(uint8_t)w1, (uint8_t)(w1 >> 8), (uint8_t)(w1 >> 16), (uint8_t)(w1 >> 24),
                           (uint8_t)w2, (uint8_t)(w2 >> 8), (uint8_t)(w2 >> 16), (uint8_t)(w2 >> 24),
                           (uint8_t)w3, (uint8_t)(w3 >> 8), (uint8_t)(w3 >> 16), (uint8_t)(w3 >> 24)};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        sc[s] = q[s] & 63;
        mn[s] = q[s + 4] & 63;
        sc[s + 4] = (q[s + 8] & 0xF) | ((q[s] >> 6) << 4);
        mn[s + 4] = (q[s + 8] >> 4) | ((q[s + 4] >> 6) << 4);
    }
}

// Exchange within the 8 adjacent lanes of a row: the value of lane (l ^ m).
__device__ __forceinline__ float xor_row(float v, int m) { return __shfl_xor(v, m, 64); }

// reduce8 of the values the 8 lanes of a row hold (lane l: v_l); every lane of the row gets the result.
__device__ __forceinline__ float row_reduce8(float v) {
    const float a = v + xor_row(v, 4); // lanes 0..3: v0+v4, v1+v5, v2+v6, v3+v7
    const float b = a + xor_row(a, 2); // lane 0: (v0+v4)+(v2+v6); lane 1: (v1+v5)+(v3+v7)
    return b + xor_row(b, 1);
}

template <int T>
__global__ void __launch_bounds__(256) kq_q8f_kernel(Q8fArgs a) {
    const int tid = threadIdx.x, l = tid & 7;
    const int row = blockIdx.x * Q8F_ROWS + (tid >> 3);
    const size_t r = (size_t)min(row, a.rows - 1); // the rows past the end read the last row and write nothing
    const size_t nb = (size_t)a.nb;
    float acc = 0.0f, accm = 0.0f;
    for (size_t sb = 0; sb < nb; sb++) {
        const uint4 q = *reinterpret_cast<const uint4 *>(a.qa + kq_qa_off(r, sb, nb, l));
        const uint4 s4 = *reinterpret_cast<const uint4 *>(a.sc + kq_sc_off(r, sb, nb));
        uint32_t code[8];   // the lane's 4 codes of sub-block s, one byte each
        float dsc[8];       // d * sc of the scale that multiplies this lane in sub-block s
        float mind = 0.0f;  // Q4_K / Q5_K: m[l] * -dmin, the min of sub-block l
        if constexpr (T == AQ_TYPE_Q6_K) {
            const uint2 h = *reinterpret_cast<const uint2 *>(a.qb + kq_qb6_off(r, sb, nb, l));
            const float d = f16lo(*reinterpret_cast<const uint16_t *>(a.dm + kq_dm_off(r, sb, nb)));
            const uint32_t qw[4] = {q.x, q.y, q.z, q.w}, hw[2] = {h.x, h.y}, sw[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int g = s >> 2, k = s & 3; // half, sub-block within the half (dot.rs:128-141)
                const uint32_t lo = (qw[g * 2 + (k & 1)] >> (4 * (k >> 1))) & 0x0F0F0F0Fu;
                const uint32_t hi = ((hw[g] >> (2 * k)) & 0x03030303u) << 4;
                code[s] = lo | hi;
                const int gi = 2 * s + (l >> 2); // group scale sc[g*8 + 2k] (lanes 0..3) or sc[g*8 + 2k + 1]
                const int scv = (int8_t)(sw[gi >> 2] >> (8 * (gi & 3)));
                dsc[s] = d * (float)scv;
            }
        } else {
            const float d = f16lo(s4.x), dmin = f16lo(s4.x >> 16);
            int sc[8], mn[8];
            scales_k4(s4.y, s4.z, s4.w, sc, mn);
            const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
            uint32_t h5 = 0;
            if constexpr (T == AQ_TYPE_Q5_K) h5 = *reinterpret_cast<const uint32_t *>(a.qb + kq_qb5_off(r, sb, nb, l));
#pragma unroll
            for (int s = 0; s < 8; s++) {
                uint32_t c = (qw[s >> 1] >> (4 * (s & 1))) & 0x0F0F0F0Fu;
                if constexpr (T == AQ_TYPE_Q5_K) c |= ((h5 >> s) & 0x01010101u) << 4;
                code[s] = c;
                dsc[s] = d * (float)sc[s];
            }
            int ml = mn[0];
#pragma unroll
            for (int s = 1; s < 8; s++) ml = l == s ? mn[s] : ml;
            mind = (float)ml * -dmin;
        }
        const uint32_t *xw = reinterpret_cast<const uint32_t *>(a.xq + sb * 256) + l;
        const float *xd = a.xd + sb * 8;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const uint32_t xv = xw[s * 8];
            int p = sdot4(code[s], xv);
            if constexpr (T == AQ_TYPE_Q6_K) {
                // 32 * (sum of the x codes of this lane's half-block), taken from lanes 0 and 4 only
                int hs = sdot4(xv, 0x01010101u);
                hs += dpp_mov<0xB1>(hs); // quad_perm [1,0,3,2]
                hs += dpp_mov<0x4E>(hs); // quad_perm [2,3,0,1]
                if ((l & 3) == 0) p -= 32 * hs;
            }
            const float f = xd[s] * dsc[s];
            acc += (float)p * f;
        }
        if constexpr (T != AQ_TYPE_Q6_K) accm += mind * (xd[l] * (float)a.xs[sb * 8 + l]);
    }
    float v = row_reduce8(acc);
    if constexpr (T != AQ_TYPE_Q6_K) v = v + row_reduce8(accm);
    if (l == 0 && row < a.rows) a.y[row] = a.resid ? a.resid[row] + v : v;
}

// Four columns. The matrix core's 4x4 block products fit the chains: block (row quad, lane l) of a wave's sixteen
// holds the four rows' codes 4l..4l+3 of a sub-block (one VGPR, exactly the weight tile's order) against four columns'
// (v_mfma_i32_4x4x4_16b_i8: every p32[l], exact), and the factors d32 * (d * sc) are outer products of four rows' scales
// and four columns' (v_mfma_f32_4x4x1_16b with a zero addend: the product, rounded once). A thread (row quad, l, column)
// is left with its four rows' conversion, product and add per sub-block, and unpacks one row's codes for all columns.
// Each lane decodes one scale and one min of the row's eight (Q6_K: two of sixteen); ds_swizzle hands them round.
// The columns' codes, scales and sums pass through the LDS, Q8M_CH super-blocks at a time, the next ones and the next
// weights in flight meanwhile. With a thread per chain and column, each wave's activation loads (8 rows reading the same
// 4 bytes) and 5 vector operations per sub-block and column took 57 us at 17408 x 5120 Q4_K, 4 columns, and 217 us at
// 5120 x 17408 Q6_K; here 22.5 and 43, bound by the waves' own instructions (2.1 waves per SIMD; 0.6 at 5120 rows).
// Four waves per work-group: two (21.6 and 53 us) and one (23.5 and 43) stage the columns more often or share a SIMD.
constexpr int Q8M_CH = 4;    // super-blocks per LDS stage
constexpr int Q8M_WAVES = 4; // waves per work-group, 8 rows each

typedef int q8i4 __attribute__((ext_vector_type(4)));
typedef float q8f4 __attribute__((ext_vector_type(4)));
typedef uint32_t q8u4 __attribute__((ext_vector_type(4)));
typedef uint32_t q8u2 __attribute__((ext_vector_type(2)));

template <int T>
__global__ void __launch_bounds__(Q8M_WAVES * 64) kq_q8f_block_kernel(Q8fArgs a) {
    constexpr int CH = Q8M_CH, TH = Q8M_WAVES * 64;
    constexpr bool K6 = T == AQ_TYPE_Q6_K;
    __shared__ __attribute__((aligned(16))) uint32_t lx[2][CH][2][32][4]; // codes: [s / 4][lane][s % 4]
    __shared__ __attribute__((aligned(16))) float ld[2][CH][2][4][4];     // d32: [s / 4][column][s % 4]
    // Q4_K / Q5_K: d32 * sum, [s * 4 + column]; Q6_K: -32 * (sum of 16 codes) where lane l = 0 or 4 takes it, else zero
    __shared__ __attribute__((aligned(16))) int lm[2][CH][K6 ? 256 : 32];
    const int tid = threadIdx.x, lane = tid & 63, l = (lane >> 2) & 7, j = lane & 3, l32 = lane & 31;
    const int row0 = (int)blockIdx.x * Q8M_WAVES * 8 + (tid >> 6) * 8 + (lane >> 5) * 4;
    const size_t r = (size_t)min(row0 + j, a.rows - 1); // rows past the end read the last row and write nothing
    const int c0 = (int)blockIdx.y * 4, nb = a.nb, nch = (nb + CH - 1) / CH;
    const size_t nbz = (size_t)nb;

    constexpr int NX = 4 * CH * 16 / TH, NDV = 4 * CH * 8;
    q8u4 xr[NX];
    float dr;
    int sr;
    auto load_x = [&](int ch) {
#pragma unroll
        for (int u = 0; u < NX; u++) {
            const int e = u * TH + tid, c = min(c0 + (e >> 6), a.ncols - 1), sb = min(ch * CH + ((e >> 4) & 3), nb - 1);
            xr[u] = *reinterpret_cast<const q8u4 *>(a.xq + (size_t)c * a.n + (size_t)sb * 256 + (e & 15) * 16);
        }
        const int e = min(tid, NDV - 1), c = min(c0 + (e >> 5), a.ncols - 1);
        const size_t at = (size_t)c * a.nb32 + (size_t)min(ch * CH + ((e >> 3) & 3), nb - 1) * 8 + (e & 7);
        dr = a.xd[at];
        if constexpr (!K6) sr = a.xs[at];
    };
    auto store_x = [&](int b) {
#pragma unroll
        for (int u = 0; u < NX; u++) {
            const int e = u * TH + tid, cj = e >> 6, sb = (e >> 4) & 3, s = (e >> 1) & 7, hf = e & 1;
#pragma unroll
            for (int w = 0; w < 4; w++) lx[b][sb][s >> 2][(hf * 4 + w) * 4 + cj][s & 3] = xr[u][w];
            if constexpr (K6) {
                int hs = 0;
#pragma unroll
                for (int w = 0; w < 4; w++) hs += sdot4(xr[u][w], 0x01010101u);
                lm[b][sb][((s >> 2) * 32 + hf * 16 + cj) * 4 + (s & 3)] = -32 * hs;
            }
        }
        if (tid < NDV) {
            const int cj = tid >> 5, sb = (tid >> 3) & 3, s = tid & 7;
            ld[b][sb][s >> 2][cj][s & 3] = dr;
            if constexpr (!K6) lm[b][sb][s * 4 + cj] = __float_as_int(dr * (float)sr);
        }
    };
    q8u4 qr[2][CH], cr[2][CH];
    q8u2 hr[2][CH];
    uint32_t dm[2][CH];
    auto load_w = [&](int b, int ch) {
#pragma unroll
        for (int u = 0; u < CH; u++) {
            const size_t sb = (size_t)min(ch * CH + u, nb - 1);
            qr[b][u] = __builtin_nontemporal_load(reinterpret_cast<const q8u4 *>(a.qa + kq_qa_off(r, sb, nbz, l)));
            cr[b][u] = __builtin_nontemporal_load(reinterpret_cast<const q8u4 *>(a.sc + kq_sc_off(r, sb, nbz)));
            if constexpr (T == AQ_TYPE_Q5_K)
                hr[b][u].x =
                    __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(a.qb + kq_qb5_off(r, sb, nbz, l)));
            if constexpr (K6) {
                hr[b][u] = __builtin_nontemporal_load(reinterpret_cast<const q8u2 *>(a.qb + kq_qb6_off(r, sb, nbz, l)));
                dm[b][u] = *reinterpret_cast<const uint16_t *>(a.dm + kq_dm_off(r, sb, nbz));
            }
        }
    };
    float acc[4] = {}, accm[4] = {};
    const uint32_t lo4 = l < 4 ? ~0u : 0u;
    auto compute = [&](int b, int ch) {
#pragma unroll
        for (int u = 0; u < CH; u++) {
            if (ch * CH + u >= nb) break;
            const q8u4 q = qr[b][u], c4 = cr[b][u];
            int code[8];
            float dsv[2], md = 0.0f; // this lane's scale (Q6_K: of sub-blocks l % 4 and l % 4 + 4), its min
            if constexpr (K6) {
                const float d = f16lo(dm[b][u]);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const int g = s >> 2, k = s & 3;
                    const uint32_t hi = k < 2 ? hr[b][u][g] << (4 - 2 * k) : hr[b][u][g] >> (2 * k - 4);
                    code[s] = (int)(((q[g * 2 + (k & 1)] >> (4 * (k >> 1))) & 0x0F0F0F0Fu) | (hi & 0x30303030u));
                }
                // groups 2 s + (l >= 4) of s = l % 4 and l % 4 + 4
                const int sh = ((2 * (l & 3) + (l >> 2)) & 3) * 8, odd = l & 2;
                dsv[0] = d * (float)(int8_t)((odd ? c4.y : c4.x) >> sh);
                dsv[1] = d * (float)(int8_t)((odd ? c4.w : c4.z) >> sh);
            } else {
                const float d = f16lo(c4.x), dmin = f16lo(c4.x >> 16);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    uint32_t c = (q[s >> 1] >> (4 * (s & 1))) & 0x0F0F0F0Fu;
                    if constexpr (T == AQ_TYPE_Q5_K)
                        c |= (s < 4 ? hr[b][u].x << (4 - s) : hr[b][u].x >> (s - 4)) & 0x10101010u;
                    code[s] = (int)c;
                }
                // quant.rs:45-51 get_scale_min_k4 of sub-block l
                const int sh = (l & 3) * 8;
                const uint32_t w1 = c4.y >> sh, w2 = c4.z >> sh, w3 = c4.w >> sh;
                const uint32_t sc = (w1 & 63 & lo4) | (((w3 & 15) | ((w1 >> 2) & 0x30)) & ~lo4);
                const uint32_t mn = (w2 & 63 & lo4) | ((((w3 >> 4) & 15) | ((w2 >> 2) & 0x30)) & ~lo4);
                dsv[0] = d * (float)(int)sc;
                md = (float)(int)mn * -dmin;
            }
            float ds[8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                // the lane of the same row that decoded sub-block s (Q6_K: its half's group of it)
                constexpr int AND = K6 ? 0x13 : 0x03;
                const int v = __float_as_int(dsv[K6 ? s >> 2 : 0]);
                int o = 0;
                switch (K6 ? s & 3 : s) {
                case 0: o = __builtin_amdgcn_ds_swizzle(v, AND | (0 << 7)); break;
                case 1: o = __builtin_amdgcn_ds_swizzle(v, AND | (1 << 7)); break;
                case 2: o = __builtin_amdgcn_ds_swizzle(v, AND | (2 << 7)); break;
                case 3: o = __builtin_amdgcn_ds_swizzle(v, AND | (3 << 7)); break;
                case 4: o = __builtin_amdgcn_ds_swizzle(v, AND | (4 << 7)); break;
                case 5: o = __builtin_amdgcn_ds_swizzle(v, AND | (5 << 7)); break;
                case 6: o = __builtin_amdgcn_ds_swizzle(v, AND | (6 << 7)); break;
                default: o = __builtin_amdgcn_ds_swizzle(v, AND | (7 << 7)); break;
                }
                ds[s] = __int_as_float(o);
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const q8u4 x4 = *reinterpret_cast<const q8u4 *>(lx[b][u][h][l32]);
                const q8f4 d4 = *reinterpret_cast<const q8f4 *>(ld[b][u][h][j]);
                q8i4 z4 = {};
                if constexpr (K6) z4 = *reinterpret_cast<const q8i4 *>(&lm[b][u][(h * 32 + l32) * 4]);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const q8i4 z = {z4[k], z4[k], z4[k], z4[k]};
                    const q8i4 p = __builtin_amdgcn_mfma_i32_4x4x4i8(code[h * 4 + k], (int)x4[k], z, 0, 0, 0);
                    const q8f4 f = __builtin_amdgcn_mfma_f32_4x4x1f32(ds[h * 4 + k], d4[k], q8f4{}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i] += (float)p[i] * f[i];
                }
            }
            if constexpr (!K6) {
                const float dx = __int_as_float(lm[b][u][l32]);
                const q8f4 f = __builtin_amdgcn_mfma_f32_4x4x1f32(md, dx, q8f4{}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) accm[i] += f[i];
            }
        }
    };
    if constexpr (K6)
        for (int i = tid; i < 2 * CH * 256; i += TH) (&lm[0][0][0])[i] = 0;
    load_x(0);
    load_w(0, 0);
    if constexpr (K6) __syncthreads();
    store_x(0);
    __syncthreads();
    for (int ch = 0; ch < nch; ch += 2) {
        load_x(min(ch + 1, nch - 1));
        load_w(1, min(ch + 1, nch - 1));
        compute(0, ch);
        store_x(1);
        __syncthreads();
        if (ch + 1 >= nch) break;
        load_x(min(ch + 2, nch - 1));
        load_w(0, min(ch + 2, nch - 1));
        compute(1, ch + 1);
        store_x(0);
        __syncthreads();
    }
    // reduce8 over the lanes of a row (4 threads apart), in the pairing of row_reduce8
    auto reduce = [&](float v) {
        v = v + xor_row(v, 16);
        v = v + xor_row(v, 8);
        return v + xor_row(v, 4);
    };
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v = reduce(acc[i]);
        if constexpr (!K6) v = v + reduce(accm[i]);
        const int c = c0 + j, row = row0 + i;
        if (l == 0 && c < a.ncols && row < a.rows) {
            const size_t o = (size_t)c * a.rows + row;
            a.y[o] = a.resid ? a.resid[o] + v : v;
        }
    }
}

template <int T>
int launch_t(const Q8fArgs &a, hipStream_t stream) {
    // One column of up to 24 super-blocks: a thread per chain, no stage to fill (17408 x 5120 Q4_K 21.8 against 24.2 us,
    // 1024 x 5120 Q5_K 12.0 against 13.6; at 24 super-blocks both 16.3; at 68, 5120 x 17408 Q4_K, 50.9 against 38.1).
    if (a.ncols == 1 && a.nb <= 24) {
        const dim3 grid((unsigned)((a.rows + Q8F_ROWS - 1) / Q8F_ROWS));
        hipLaunchKernelGGL(kq_q8f_kernel<T>, grid, dim3(256), 0, stream, a);
    } else { // columns in fours (eight per thread: 36 us against 34 at 17408 x 5120, 72 against 58 at 5120 x 17408)
        const dim3 grid((unsigned)((a.rows + Q8M_WAVES * 8 - 1) / (Q8M_WAVES * 8)), (unsigned)((a.ncols + 3) / 4));
        hipLaunchKernelGGL(kq_q8f_block_kernel<T>, grid, dim3(Q8M_WAVES * 64), 0, stream, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : fail(AQ_EHIP, "kq_q8f launch");
}

} // namespace

int launch_kq_q8f(const Weight &w, const Act &x, size_t ncols, float *y, const float *resid, hipStream_t stream) {
    AQ_REQUIRE(is_kquant(w.type), "kq_q8f: K-quant weights only");
    AQ_REQUIRE(w.cols == x.n && w.cols % 256 == 0, "kq_q8f: activation length must equal the weight's columns "
                                                    "(a multiple of 256, matvec.rs:73-77)");
    AQ_REQUIRE(ncols >= 1 && ncols <= x.ncols && ncols <= 16, "kq_q8f: ncols out of range");
    AQ_REQUIRE(w.rows >= 1 && w.rows <= (size_t)INT32_MAX, "kq_q8f: rows out of range");
    Q8fArgs a{};
    a.qa = w.qa;
    a.qb = w.qb;
    a.sc = w.sc;
    a.dm = w.dm;
    a.rows = (int)w.rows;
    a.nb = (int)w.nb;
    a.xq = x.q0;
    a.xd = x.d0;
    a.xs = x.s0;
    a.n = x.n;
    a.nb32 = x.nb32;
    a.ncols = (int)ncols;
    a.y = y;
    a.resid = resid;
    switch (w.type) {
    case AQ_TYPE_Q4_K: return launch_t<AQ_TYPE_Q4_K>(a, stream);
    case AQ_TYPE_Q5_K: return launch_t<AQ_TYPE_Q5_K>(a, stream);
    default: return launch_t<AQ_TYPE_Q6_K>(a, stream);
    }
}

} // namespace aq
