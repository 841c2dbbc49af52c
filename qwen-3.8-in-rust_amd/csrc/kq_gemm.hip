// kq_gemm.hip — weight x activation products over many columns (a prompt chunk's rows: model.rs:443-461 prefill,
// where every projection is a matmul over the chunk's tokens, matvec.rs:369-393). Each output equals the single-
// column dot bit for bit: the integer lane sums are exact and each output's f32 chains advance super-block by
// super-block (block by block for Q8_0 / Q4_0) in the reference's order.
//
// K-quants x Q8_K (kdot.rs:37-140, 176-333) on v_mfma_f32_16x16x32_f16. The reference's lane l of a super-block is
// the 32 elements 32s + 4l + b (s = sub-block, b = 0..3), and its sum is sum_s sc[s] * sum_b q * x. One matrix-core
// product over K = 32 covers exactly lane l: k-group g of the operands (lanes 16g .. 16g + 15) takes sub-blocks 2g and
// 2g + 1, four elements each. Q4_K / Q5_K: the weight operand is q * sc (codes <= 31, scales <= 63: at most 1953, exact
// in f16), the activation codes as f16 (the quantiser writes them so: Act::gh), every partial sum an integer below
// 2^23, exact in f32 - the product returns f32(sumi[l]), nothing to convert. Q6_K: the signed 8-bit group scale
// sc = 16 hi + lo goes into two f16 operands q * lo and q * hi (unsigned codes <= 63: exact), the reference's -32 offset
// enters the hi sum as -2 (bs[2l] sc[2l] + bs[2l + 1] sc[2l + 1]) (kdot.rs:125-129, the reference's lane split of it; a
// K = 4 product of the group sums, |.| <= 2032, exact in f16), and fma(16, hi sum, lo sum) rounds the exact integer
// once, as the reference's conversion does. The products that the f32 chains start from come from the matrix cores
// too: d = dx * d and -dx * dmin of a 16 x 64 tile are one K = 1 f32 outer product each (rounded once, no FMA), and
// the Q4_K / Q5_K min sums prod[i] one K = 4 product of the mins and the group sums.
//
// Q8_0 / Q4_0 x Q8_0 (dot.rs:29-66): one product over K = 32 is one block's exact i32 sum for the tile (Q4_0: of the
// codes less 8), then acc += (dw * dx) * f32(isum) per output.
//
// Work (K-quants): a work-group of eight waves owns two 16-row tiles x CT 16-column tiles; wave (rt, w) takes the lane
// slots w and w + 4 (and min lane w) of row tile rt, for all of K. The eight lane chains are independent until the final
// reduction, so nothing passes between the waves before that, and each weight code is unpacked once per work-group
// (with a wave per column tile, as the Q8_0 / Q4_0 kernel below has it, every code is unpacked four times: Q4_K 388
// vector instructions per 16 x 16 x 256 step, of which 112 are the f32 chains; here ~150 per 16 x 64 x 256 step and
// wave, 96 of them the chains). Two row tiles share the activation operands, which come through the LDS by direct copies
// several steps ahead: a wave's loads return in order, so operands loaded straight into registers wait for the weights'
// memory latency. Q4_K 17408 x 5120 at 64 columns: of 56 us the vector instructions are ~21 by count over the chip's
// SIMDs, the matrix cores' ~8 beside them; two waves per SIMD with a barrier every step, the copies (~350 MB of
// activation operands) and a last partial pass over the CUs leave the rest uncovered. Measured, 64 columns: Q4_K
// 17408 x 5120 94 -> 56 us, Q6_K 5120 x 17408 211 -> 87, Q5_K 5120 x 6144 45 -> 26, Q4_K 10240 x 5120 -> 35; 37 columns:
// Q6_K 5120 x 17408 208 -> 73 us.
#include "aq_common.h"

#include <atomic>

namespace aq {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4i mma(uint64_t a, uint64_t b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)a, (long)b, c, 0, 0, 0);
}
__device__ __forceinline__ uint64_t pack2(uint32_t lo, uint32_t hi) { return (uint64_t)lo | ((uint64_t)hi << 32); }
__device__ __forceinline__ float h2f(uint32_t bits16) {
    _Float16 f;
    const uint16_t h = (uint16_t)(bits16 & 0xFFFF);
    __builtin_memcpy(&f, &h, 2);
    return (float)f;
}
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct GemmArgs {
    const uint8_t *qa, *qb, *sc, *dm;
    int rows, nb, ncols;
    // Q8_K activations (lane-slot order) or Q8_0 (natural order)
    const int8_t *xq;
    const float *xd;
    size_t n;
    // the many-column Q8_K form (Act::gh, gm; gcap columns)
    const uint16_t *gh;
    const uint8_t *gm;
    uint32_t gcap;
    int nfull; // K-quants: work-groups over all column tiles; those past them take one each
    float *y;
    const float *resid;
};

// ---- LDS staging ----
// Operands reach the LDS by direct global-to-LDS copies (global_load_lds_*: each active lane's 16 or 4 bytes land at
// m0 + 16 * lane or m0 + 4 * lane), issued a ring's buffers less one ahead, so the
// loads' latency is covered without holding the data in registers. Every wave issues the same number of copies per
// step (a whole wave never skips one), so its count of outstanding vector-memory operations says which step has
// landed; a work-group barrier after the wait makes every wave's copies of that step visible and, at the same
// time, frees the buffer read one step earlier for the next copies.
constexpr int GEMM_CUS = 256;

__device__ __forceinline__ void dma16(uint32_t lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g) : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(g) : "memory", "m0");
}
// Wait until at most N of this wave's vector-memory operations are outstanding (and its LDS operations are done),
// then meet the work-group; one asm statement, so no memory access moves across it.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// ---- K-quants ----
__device__ __forceinline__ f16x2 bits2(uint32_t w) { return __builtin_bit_cast(f16x2, w); }
__device__ __forceinline__ f16x2 splat2(float v) { return f16x2{(_Float16)v, (_Float16)v}; }
// Two unsigned bytes of w (byte selectors of v_perm_b32 in the low and high half) as the f16 pair 1024 + byte.
template <uint32_t SEL>
__device__ __forceinline__ f16x2 magic2(uint32_t w) {
    return bits2(__builtin_amdgcn_perm(0x64646464u, w, SEL));
}
// (x & mask) | base in one instruction (one operand of the three may be scalar).
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t base) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(base));
    return r;
}
__device__ __forceinline__ f16x2 fma2(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ f16x8 cat(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// A wave's raw weights of one super-block: lane (li, g) holds row li's codes of lane slots w and w + 4 for sub-blocks 2g
// and 2g + 1, and row li's scale record.
template <int T>
struct KqRaw {
    uint32_t c[T == AQ_TYPE_Q4_K ? 2 : (T == AQ_TYPE_Q5_K ? 4 : 6)];
    u32x4 rec;
    uint32_t d6;
};
// Its matrix-core weight operands.
struct KqOps {
    f16x8 lo[2], hi[2]; // lane slots w, w + 4 (hi: Q6_K)
    f16x4 m[2];         // the mins, or the Q6_K group scales of lanes w and w + 4
    float d, dmin;
};

// One super-block step in the LDS. Per row tile its four 4-row weight tiles, each as in memory: qa (512 B), qb (Q5_K
// 128 B, Q6_K 256 B), the four 16-byte scale records (a stride of 16 or 48 banks: the operand reads meet no bank
// conflicts); Q6_K then the tiles' f16 d (8 B each). Activations: per lane slot and column tile the operand's 1 KB run;
// the column tiles' group sums and d as in memory (ACT_GM B each).
template <int T, int CT>
struct KqStage {
    static constexpr int QB = T == AQ_TYPE_Q4_K ? 0 : (T == AQ_TYPE_Q5_K ? 128 : 256);
    static constexpr int TB = 512 + QB + 64, WL = TB / 16;           // a 4-row tile: bytes, lanes of its one copy
    static constexpr int WB = 4 * TB + (T == AQ_TYPE_Q6_K ? 32 : 0); // a 16-row tile
    static constexpr int XB = 2 * WB, GM = XB + 8 * CT * 1024, BYTES = GM + 4 * ACT_GM;
    static constexpr int NDMA = CT + 2 + (T == AQ_TYPE_Q6_K ? 1 : 0); // copies per wave per step
    // stages: as many as the CU's 160 KB hold for one work-group per CU at three and four column tiles, two below
    static constexpr int LDS = CT >= 3 ? 163840 : 81920;
    static constexpr int RING = LDS / BYTES < 6 ? LDS / BYTES : 6;
    static_assert(RING >= 3, "stages");
};

// A wave's copies of successive steps: running source addresses (each lane's own), and the stage to fill.
template <int T, int CT>
struct KqCopier {
    using S = KqStage<T, CT>;
    const uint8_t *w, *dm, *m; // weights, Q6_K f16 d, group sums
    const uint16_t *x;
    uint32_t wstride, xstride, mstride; // bytes, f16, bytes per step
    uint32_t lds0, wo, mo, xo, dofs, buf;
    int lane;

    __device__ __forceinline__ KqCopier(const GemmArgs &a, uint32_t lds, int r0, int ct0, int wave, int lane_) {
        lane = lane_;
        const int rt = wave >> 2, w4 = wave & 3;
        const size_t t = kq_tile((size_t)min(r0 + 16 * rt + 4 * w4, a.rows - 1), 0, (size_t)a.nb);
        // wave w4 copies 4-row tile w4 of its row tile
        if (lane < 32) {
            w = a.qa + t * 512 + lane * 16;
            wstride = 512;
        } else if (lane < 32 + S::QB / 16) {
            w = a.qb + t * S::QB + (lane - 32) * 16;
            wstride = S::QB;
        } else {
            w = a.sc + t * 64 + (min(lane, S::WL - 1) - 32 - S::QB / 16) * 16;
            wstride = 64;
        }
        dm = a.dm + t * 8 + 4 * (lane & 1);
        // lane slot `wave` of every column tile; column tile `wave`'s group sums (repeated past the last tile)
        x = a.gh + act_gh(a.gcap, 0, wave, 16 * (size_t)ct0, 0) + 8 * lane;
        xstride = a.gcap * 256;
        const int ct = min(wave, CT - 1);
        m = a.gm + act_gm(a.gcap, 0, 16 * (size_t)(ct0 + ct)) + 16 * min(lane, ACT_GM / 16 - 1);
        mstride = a.gcap / 16 * ACT_GM;
        lds0 = buf = lds;
        wo = (uint32_t)(rt * S::WB + w4 * S::TB);
        dofs = (uint32_t)(rt * S::WB + 4 * S::TB + w4 * 8);
        xo = (uint32_t)(S::XB + wave * CT * 1024);
        mo = (uint32_t)(S::GM + ct * ACT_GM);
    }
    __device__ __forceinline__ void issue() {
        if (lane < S::WL) dma16(buf + wo, w);
        if constexpr (T == AQ_TYPE_Q6_K) {
            if (lane < 2) dma4(buf + dofs, dm);
            dm += 8;
        }
        // the column tiles' runs are contiguous on both sides: one LDS base, the instruction's offset moves both
        if constexpr (CT == 1)
            dma16(buf + xo, x);
        else if constexpr (CT == 2)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                         "global_load_lds_dwordx4 %1, off offset:1024" ::"s"(buf + xo), "v"(x) : "memory", "m0");
        else if constexpr (CT == 3)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                         "global_load_lds_dwordx4 %1, off offset:1024\n\tglobal_load_lds_dwordx4 %1, off offset:2048"
                         ::"s"(buf + xo), "v"(x) : "memory", "m0");
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                         "global_load_lds_dwordx4 %1, off offset:1024\n\tglobal_load_lds_dwordx4 %1, off offset:2048\n\t"
                         "global_load_lds_dwordx4 %1, off offset:3072" ::"s"(buf + xo), "v"(x) : "memory", "m0");
        if (lane < ACT_GM / 16) dma16(buf + mo, m);
        w += wstride;
        x += xstride;
        m += mstride;
        buf = buf + S::BYTES == lds0 + S::RING * S::BYTES ? lds0 : buf + S::BYTES;
    }
};

// CT: 16-column tiles of the work-group (1..4).
template <int T, int CT>
__device__ __forceinline__ void kq_gemm_body(const GemmArgs &a, uint8_t *gm_lds, const int r0, const int ct0) {
    using S = KqStage<T, CT>;
    constexpr bool Q6 = T == AQ_TYPE_Q6_K;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rt = wave >> 2, w = wave & 3;
    const int g = lane >> 4, li = lane & 15, k4 = li >> 2, r4 = li & 3;
    const int nb = a.nb, c0 = 16 * ct0;
    const uint32_t magic = 0x64006400u; // 2^10's exponent in both halves: or-ed with packed integers, 1024 + v

    auto unpack = [&](KqOps &p, const KqRaw<T> &k) {
        if constexpr (Q6) {
            // group scales of sub-blocks 2g, 2g + 1: byte 0 = 2g lanes 0-3, 1 = 2g lanes 4-7, 2 and 3 the same of 2g + 1
            const uint32_t sw = g == 0 ? k.rec[0] : g == 1 ? k.rec[1] : g == 2 ? k.rec[2] : k.rec[3];
            const uint32_t l4 = sw & 0x0F0F0F0Fu, h4 = ((sw ^ 0x80808080u) >> 4) & 0x0F0F0F0Fu;
            // pairs (lanes 0-3, lanes 4-7) of sub-blocks 2g and 2g + 1
            const f16x2 la = magic2<0x04010400u>(l4) + splat2(-1024.0f), lb = magic2<0x04030402u>(l4) + splat2(-1024.0f);
            const f16x2 ha = magic2<0x04010400u>(h4) + splat2(-1032.0f), hb4 = magic2<0x04030402u>(h4) + splat2(-1032.0f);
            const f16x2 cla = la * splat2(-1024.0f), clb = lb * splat2(-1024.0f);
            const f16x2 cha = ha * splat2(-1024.0f), chb = hb4 * splat2(-1024.0f);
            const int sh = 4 * (g & 1);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t wa = k.c[2 * h] >> sh, wb = k.c[2 * h + 1] >> sh, wh = k.c[4 + h] >> sh;
                const uint32_t wa8 = wa >> 8, wb8 = wb >> 8, wh8 = wh >> 8;
                const f16x2 p0 = bits2(and_or(wa, 0x000F000Fu, magic) | ((wh & 0x00030003u) << 4));
                const f16x2 p1 = bits2(and_or(wa8, 0x000F000Fu, magic) | ((wh8 & 0x00030003u) << 4));
                const f16x2 p2 = bits2(and_or(wb, 0x000F000Fu, magic) | ((wh & 0x000C000Cu) << 2));
                const f16x2 p3 = bits2(and_or(wb8, 0x000F000Fu, magic) | ((wh8 & 0x000C000Cu) << 2));
                const f16x2 fl = f16x2{la[h], la[h]}, gl = f16x2{cla[h], cla[h]}, fl2 = f16x2{lb[h], lb[h]}, gl2 = f16x2{clb[h], clb[h]};
                const f16x2 fh = f16x2{ha[h], ha[h]}, gh = f16x2{cha[h], cha[h]}, fh2 = f16x2{hb4[h], hb4[h]}, gh2 = f16x2{chb[h], chb[h]};
                p.lo[h] = cat(fma2(p0, fl, gl), fma2(p1, fl, gl), fma2(p2, fl2, gl2), fma2(p3, fl2, gl2));
                p.hi[h] = cat(fma2(p0, fh, gh), fma2(p1, fh, gh), fma2(p2, fh2, gh2), fma2(p3, fh2, gh2));
            }
            // -2 sc of groups 2w, 2w + 1 (lane w) and 2w + 8, 2w + 9 (lane w + 4): w uniform
            const uint32_t ow = (w & 1) ? 0x00030002u : 0x00010000u; // bytes of the word
            const uint32_t swo0 = w < 2 ? k.rec[0] : k.rec[1], swo1 = w < 2 ? k.rec[2] : k.rec[3];
            auto m2 = [&](uint32_t word) { // -2 * the two signed bytes, as f16
                const uint32_t u = word ^ 0x80808080u;
                const f16x2 v = bits2(__builtin_amdgcn_perm(0x64646464u, u, 0x04000400u + ow)) + splat2(-1152.0f);
                return v * splat2(-2.0f);
            };
            const f16x2 o0 = m2(swo0), o1 = m2(swo1);
            const _Float16 z = (_Float16)0.0f;
            p.m[0] = f16x4{o0[0], o0[1], z, z};
            p.m[1] = f16x4{z, z, o1[0], o1[1]};
            p.d = h2f(k.d6);
        } else {
            const uint32_t x = k.rec[0], y = k.rec[1], z = k.rec[2], u = k.rec[3];
            // 6-bit scales of sub-blocks 2g, 2g + 1 (quant.rs:45-51): bytes 2g, 2g + 1 of the low or high word
            const uint32_t sc_lo = y & 0x3F3F3F3Fu, sc_hi = (u & 0x0F0F0F0Fu) | ((y >> 2) & 0x30303030u);
            const uint32_t scw = (g < 2 ? sc_lo : sc_hi) >> (16 * (g & 1));
            // (s0, s1 / 16) and -1024 times it: (1024 + q) s0 - 1024 s0 and (1024 + 16 q) s1 / 16 - 64 s1, both exact
            const f16x2 s = (magic2<0x04010400u>(scw) + splat2(-1024.0f)) * f16x2{(_Float16)1.0f, (_Float16)0.0625f};
            const f16x2 cs = s * splat2(-1024.0f);
            const f16x2 s0 = f16x2{s[0], s[0]}, s1 = f16x2{s[1], s[1]}, q0 = f16x2{cs[0], cs[0]}, q1 = f16x2{cs[1], cs[1]};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t v = k.c[h], v8 = v >> 8;
                if constexpr (T == AQ_TYPE_Q4_K) {
                    p.lo[h] = cat(fma2(bits2(and_or(v, 0x000F000Fu, magic)), s0, q0),
                                  fma2(bits2(and_or(v8, 0x000F000Fu, magic)), s0, q0),
                                  fma2(bits2(and_or(v, 0x00F000F0u, magic)), s1, q1),
                                  fma2(bits2(and_or(v8, 0x00F000F0u, magic)), s1, q1));
                } else {
                    const uint32_t t = k.c[2 + h] >> (2 * g), t8 = t >> 8; // bits 0, 1 of each byte: sub-blocks 2g, 2g + 1
                    const f16x2 b0 = bits2(and_or(v, 0x000F000Fu, magic) | ((t & 0x00010001u) << 4));
                    const f16x2 b1 = bits2(and_or(v8, 0x000F000Fu, magic) | ((t8 & 0x00010001u) << 4));
                    const f16x2 b2 = bits2(and_or(v, 0x00F000F0u, magic) | ((t & 0x00020002u) << 7));
                    const f16x2 b3 = bits2(and_or(v8, 0x00F000F0u, magic) | ((t8 & 0x00020002u) << 7));
                    p.lo[h] = cat(fma2(b0, s0, q0), fma2(b1, s0, q0), fma2(b2, s1, q1), fma2(b3, s1, q1));
                }
            }
            // mins of sub-blocks 2w, 2w + 1 (w uniform): bytes 2w, 2w + 1 of the 8, each for both its 16-groups
            const uint32_t mw = and_or(u >> (w < 2 ? 0 : 4), w < 2 ? 0u : 0x0F0F0F0Fu,
                                       (z >> (w < 2 ? 0 : 2)) & (w < 2 ? 0x3F3F3F3Fu : 0x30303030u));
            const uint32_t odd = (w & 1) ? 0x00020002u : 0u;
            const f16x2 ma = bits2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04000400u + odd)) + splat2(-1024.0f);
            const f16x2 mb = bits2(__builtin_amdgcn_perm(0x64646464u, mw, 0x04010401u + odd)) + splat2(-1024.0f);
            p.m[0] = f16x4{ma[0], ma[1], mb[0], mb[1]};
            p.d = h2f(x);
            p.dmin = -h2f(x >> 16);
        }
    };

    float acc[2][CT][4], accm[CT][4];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[0][ct][j] = acc[1][ct][j] = accm[ct][j] = 0.0f;
    KqCopier<T, CT> copier(a, (uint32_t)(uintptr_t)gm_lds, r0, ct0, wave, lane);
#pragma unroll 1
    for (int s = 0; s < S::RING - 1; s++)
        if (s < nb) copier.issue();

    KqRaw<T> k;
    f16x8 xb[2][CT];
    float dx;
    u32x2 bs;
    auto read = [&](int stage) {
        const uint8_t *st = gm_lds + stage * S::BYTES, *W = st + rt * S::WB;
        // the step's operands: row li's codes of lane slots w, w + 4 and its record; dx and the group sums of column
        // 16 g + li (the outer products' four column tiles)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint8_t *cw = W + k4 * S::TB + h * 256 + (w * 4 + r4) * 16; // the row's qa run of lane slot w + 4h
            if constexpr (Q6) {
                const u32x2 x = *reinterpret_cast<const u32x2 *>(cw + 8 * (g >> 1));
                k.c[2 * h] = x[0];
                k.c[2 * h + 1] = x[1];
                k.c[4 + h] = *reinterpret_cast<const uint32_t *>(W + k4 * S::TB + 512 + (w * 4 + r4) * 16 + h * 8 + 4 * (g >> 1));
            } else {
                k.c[h] = *reinterpret_cast<const uint32_t *>(cw + 4 * g);
                if constexpr (T == AQ_TYPE_Q5_K)
                    k.c[2 + h] = *reinterpret_cast<const uint32_t *>(W + k4 * S::TB + 512 + (w * 4 + r4) * 8 + h * 4);
            }
        }
        k.rec = *reinterpret_cast<const u32x4 *>(W + k4 * S::TB + 512 + S::QB + r4 * 16);
        if constexpr (Q6) k.d6 = *reinterpret_cast<const uint16_t *>(W + 4 * S::TB + 2 * li);
        const uint8_t *gm = st + S::GM + g * ACT_GM; // (past the last column tile: whatever is there, not used)
        dx = *reinterpret_cast<const float *>(gm + 512 + 4 * li);
        if constexpr (Q6) { // groups 2w, 2w + 1 and 2w + 8, 2w + 9
            bs[0] = *reinterpret_cast<const uint32_t *>(gm + 32 * li + 4 * w);
            bs[1] = *reinterpret_cast<const uint32_t *>(gm + 32 * li + 4 * w + 16);
        } else { // groups 4w .. 4w + 3: sub-blocks 2w, 2w + 1
            bs = *reinterpret_cast<const u32x2 *>(gm + 32 * li + 8 * w);
        }
        // lane slots w and w + 4 are slots 2w and 2w + 1
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
                xb[h][ct] = *reinterpret_cast<const f16x8 *>(st + S::XB + (((2 * w + h) * CT + ct) * 64 + lane) * 16);
    };

    // A step's products go to the matrix cores from registers; while they run the next stage's copies are met and its
    // operands read from the LDS, whose latency and bandwidth then hide behind the step's f32 chains.
    if (S::RING - 1 <= nb) wait_vm_barrier<(S::RING - 2) * S::NDMA>();
    else wait_vm_barrier<0>();
    read(0);
    KqOps ops;
    unpack(ops, k);
    int rd = 1; // the next stage to read
    for (int sb = 0; sb < nb; sb++) {
        const f16x4 bsv = __builtin_bit_cast(f16x4, bs);
        f32x16 dd, dmn, pm, off[2];
        dd = __builtin_amdgcn_mfma_f32_16x16x1f32(ops.d, dx, f32x16{}, 0, 0, 0);
        if constexpr (Q6) {
            off[0] = __builtin_amdgcn_mfma_f32_16x16x4f16(ops.m[0], bsv, f32x16{}, 0, 0, 0);
            off[1] = __builtin_amdgcn_mfma_f32_16x16x4f16(ops.m[1], bsv, f32x16{}, 0, 0, 0);
        } else {
            dmn = __builtin_amdgcn_mfma_f32_16x16x1f32(ops.dmin, dx, f32x16{}, 0, 0, 0);
            pm = __builtin_amdgcn_mfma_f32_16x16x4f16(ops.m[0], bsv, f32x16{}, 0, 0, 0);
        }
        f32x4 sl[2][CT], sh4[Q6 ? 2 : 1][Q6 ? CT : 1];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                sl[h][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ops.lo[h], xb[h][ct], f32x4{}, 0, 0, 0);
                if constexpr (Q6) {
                    const f32x4 o = f32x4{off[h][4 * ct], off[h][4 * ct + 1], off[h][4 * ct + 2], off[h][4 * ct + 3]};
                    sh4[h][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ops.hi[h], xb[h][ct], o, 0, 0, 0);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        if (sb + 1 < nb) {
            // stage sb + 1 has landed, and every wave has read stage sb
            if (sb + S::RING - 1 < nb) wait_vm_barrier<(S::RING - 3) * S::NDMA>();
            else wait_vm_barrier<0>();
            if (sb + S::RING - 1 < nb) copier.issue();
            read(rd);
            rd = rd + 1 == S::RING ? 0 : rd + 1;
        }
        // the f32 chains (kdot.rs:37-140), in super-block order
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float d = dd[4 * ct + j];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    float v = sl[h][ct][j];
                    if constexpr (Q6) v = __builtin_fmaf(16.0f, sh4[h][ct][j], v); // the exact integer, rounded once
                    acc[h][ct][j] += d * v;
                }
                if constexpr (!Q6) accm[ct][j] += dmn[4 * ct + j] * pm[4 * ct + j];
            }

        unpack(ops, k);
    }

    // reduce8 / reduce4 over the waves' lanes: ((l0 + l4) + (l2 + l6)) + ((l1 + l5) + (l3 + l7)), (m0 + m2) + (m1 + m3).
    // The partials take the ring's place: every copy has landed and been read.
    __syncthreads();
    float *part = reinterpret_cast<float *>(gm_lds) + rt * 8 * CT * 256; // [wave][ct][j][lane], then the min lanes
    float *partm = part + 4 * CT * 256;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int e = ((w * CT + ct) * 4 + j) * 64 + lane;
            part[e] = acc[0][ct][j] + acc[1][ct][j];
            if constexpr (!Q6) partm[e] = accm[ct][j];
        }
    __syncthreads();
    if (w >= CT) return; // wave w finishes column tile w
    const int col = c0 + 16 * w + li;
    if (col >= a.ncols) return;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int orow = r0 + 16 * rt + 4 * g + j;
        if (orow >= a.rows) continue;
        const int e = (w * 4 + j) * 64 + lane, q = CT * 256;
        float v = (part[e] + part[2 * q + e]) + (part[q + e] + part[3 * q + e]);
        if constexpr (!Q6) v = v + ((partm[e] + partm[2 * q + e]) + (partm[q + e] + partm[3 * q + e]));
        const size_t o = (size_t)col * a.rows + orow;
        a.y[o] = a.resid ? a.resid[o] + v : v;
    }
}

template <int T, int CT>
constexpr size_t kq_lds() {
    constexpr size_t a = (size_t)KqStage<T, CT>::BYTES * KqStage<T, CT>::RING, b = (size_t)KqStage<T, 1>::BYTES * KqStage<T, 1>::RING;
    return a > b ? a : b;
}

template <int T, int CT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) kq_gemm_kernel(GemmArgs a) {
    extern __shared__ __align__(16) uint8_t gm_lds[];
    const int b = (int)blockIdx.x, k = b - a.nfull;
    if (CT == 1 || k < 0) kq_gemm_body<T, CT>(a, gm_lds, 32 * b, 0);
    else kq_gemm_body<T, 1>(a, gm_lds, 32 * (a.nfull + k / CT), k % CT);
}

// One step of a Q8_0 / Q4_0 work-group (32 rows x 64 columns, 8 waves of one 16 x 16 tile each) = 8 blocks (256
// elements). In the LDS a row's or column's codes of the step are one run (256 bytes; Q4_0 rows 128), its 16-byte chunk q
// at position q ^ the row's or column's number in the tile (Q4_0: of its pair), so that a copy's lanes read whole runs
// from memory and the tile's 16 lanes read 16 different bank groups. Then per wave a region of 20 units: the 8 f32 d of 8
// of its tile's columns, and the 8 f16 d of 4 of the work-group's rows.
template <int T>
struct Q8Stage {
    static constexpr int QC = T == AQ_TYPE_Q8_0 ? 16 : 8; // code chunks per row
    static constexpr int WB = 32 * QC * 16, XB = 64 * 256, DB = 320;
    static constexpr int BYTES = WB + XB + 8 * DB;
    static constexpr int RING = 3; // stages; two work-groups' rings fit a CU (six, one work-group each: no faster)
};

// Four copies per wave, or two where its column tile is past the columns.
template <int T>
__device__ __forceinline__ void q8_issue(const GemmArgs &a, uint32_t buf, size_t st, int r0, int c0, int wave, int lane,
                                         bool xlive) {
    using S = Q8Stage<T>;
    const size_t nb = (size_t)a.nb; // 32-blocks per row
    if (T == AQ_TYPE_Q8_0 || lane < 32) { // four rows' codes
        const int i = 4 * wave + lane / S::QC, p = lane % S::QC, q = p ^ (T == AQ_TYPE_Q8_0 ? i & 15 : (i >> 1) & 7);
        const size_t row = (size_t)min(r0 + i, a.rows - 1);
        dma16(uni(buf + (uint32_t)(wave * 64 * S::QC)), a.qa + (row * nb + st * 8) * (S::QC * 2) + (size_t)q * 16);
    }
#pragma unroll
    for (int u = 0; u < 2 && xlive; u++) { // eight columns' codes
        const int i = 8 * wave + 4 * u + (lane >> 4);
        const size_t col = (size_t)min(c0 + i, a.ncols - 1);
        dma16(uni(buf + (uint32_t)(S::WB + (2 * wave + u) * 1024)),
              a.xq + col * a.n + st * 256 + (size_t)(((lane & 15) ^ i) & 15) * 16);
    }
    if (lane < 20) {
        const size_t col = (size_t)min(c0 + 8 * wave + (lane >> 1), a.ncols - 1);
        const size_t row = (size_t)min(r0 + 4 * wave + (lane & 3), a.rows - 1);
        const uint8_t *xs = reinterpret_cast<const uint8_t *>(a.xd + col * nb + st * 8 + 4 * (lane & 1));
        dma16(uni(buf + (uint32_t)(S::WB + S::XB + wave * S::DB)), lane < 16 ? xs : a.dm + (row * nb + st * 8) * 2);
    }
}

// Q8_0 / Q4_0 weights x Q8_0 activations: one product over K = 32 per block (v_mfma_i32_16x16x32_i8), its factors
// d * d of four blocks at once as outer products (v_mfma_f32_16x16x1 with a zero addend: each rounded once), so a thread
// is left with its four outputs' conversion, product and add per block. Q4_0's codes less 8 (dot.rs:48-66) enter as the
// signed bytes 16 (code - 8) - one shift and one and-xor of the packed byte - and the weights' d divided by 16, both exact.
// As 16 rows and four waves per work-group, one work-group per CU, the columns passed through the LDS for every 16 rows
// (~7.5 TB/s of cache reads) and the factors were 12 of 28 vector operations per block. 64 columns: Q4_0 17408 x 5120
// 92 -> 51 us, 5120 x 17408 119 -> 67, 12288 x 5120 52 -> 33; Q8_0 5120 x 6144 37 -> 24. Bound by a wave's own latency per
// step (two waves per SIMD at 5120 rows: 0.75 us of it without any copies, the copies alone 0.4).
template <int T>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) q8_gemm_kernel(GemmArgs a) {
    using S = Q8Stage<T>;
    extern __shared__ __align__(16) uint8_t gm_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, li = lane & 15, ct = wave & 3, rt = wave >> 2;
    const int r0 = (int)blockIdx.x * 32;
    const int c0 = (int)blockIdx.y * 64;
    const bool live = c0 + 16 * ct < a.ncols;
    const bool xlive = c0 + 16 * (wave >> 1) < a.ncols; // the tile whose columns this wave copies
    const int nst = a.nb / 8; // steps
    const uint32_t lds0 = (uint32_t)(uintptr_t)gm_lds;
    const int wrow = 16 * rt + li, wx = T == AQ_TYPE_Q8_0 ? li : li >> 1;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < S::RING - 1; s++)
        if (s < nst) q8_issue<T>(a, lds0 + (uint32_t)(s * S::BYTES), (size_t)s, r0, c0, wave, lane, xlive);

    int slot = 0;
    for (int st = 0; st < nst; st++) {
        if (st + S::RING - 2 >= nst) wait_vm_barrier<0>();
        else if (xlive) wait_vm_barrier<(S::RING - 2) * 4>();
        else wait_vm_barrier<(S::RING - 2) * 2>();
        if (st + S::RING - 1 < nst)
            q8_issue<T>(a, lds0 + (uint32_t)((slot == 0 ? S::RING - 1 : slot - 1) * S::BYTES), (size_t)(st + S::RING - 1),
                        r0, c0, wave, lane, xlive);
        const uint8_t *W = gm_lds + slot * S::BYTES;
        slot = slot == S::RING - 1 ? 0 : slot + 1;
        if (!live) continue;
        const uint8_t *X = W + S::WB + ct * 4096 + li * 256, *D = W + S::WB + S::XB;
        const uint8_t *dw = D + (wrow >> 2) * S::DB + 256 + (li & 3) * 16 + g * 2;
        const uint8_t *dx = D + (2 * ct + (li >> 3)) * S::DB + (li & 7) * 32 + g * 4;
        W += wrow * (16 * S::QC) + 8 * (g & 1);
        X += 8 * (g & 1);
        // operands, then products, then the chains: left to itself the compiler ties each block's chain to its own reads
        uint64_t wv[8], xv[8];
        float dv[2], dxv[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            dv[h] = h2f(*reinterpret_cast<const uint16_t *>(dw + 8 * h));
            dxv[h] = *reinterpret_cast<const float *>(dx + 16 * h);
        }
#pragma unroll
        for (int b = 0; b < 8; b++) {
            if constexpr (T == AQ_TYPE_Q8_0) wv[b] = *reinterpret_cast<const uint64_t *>(W + ((2 * b + (g >> 1)) ^ wx) * 16);
            else wv[b] = *reinterpret_cast<const uint64_t *>(W + (b ^ wx) * 16);
            xv[b] = *reinterpret_cast<const uint64_t *>(X + ((2 * b + (g >> 1)) ^ li) * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 f[2];
        v4i c[8];
#pragma unroll
        for (int h = 0; h < 2; h++)
            f[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(T == AQ_TYPE_Q4_0 ? dv[h] * 0.0625f : dv[h], dxv[h], f32x16{}, 0, 0, 0);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            uint64_t wa = wv[b];
            if constexpr (T == AQ_TYPE_Q4_0) { // elements 8g .. 8g + 7: bytes 8 (g & 1) .., low nibbles for g < 2, else high
                const int sh = g < 2 ? 4 : 0;
                wa = pack2((((uint32_t)wa << sh) & 0xF0F0F0F0u) ^ 0x80808080u,
                           (((uint32_t)(wa >> 32) << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
            }
            c[b] = mma(wa, xv[b], v4i{0, 0, 0, 0});
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < 8; b++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] += f[b >> 2][4 * (b & 3) + j] * (float)c[b][j];
    }
    const int ocol = c0 + 16 * ct + li;
    if (live && ocol < a.ncols) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int row = r0 + 16 * rt + 4 * g + j;
            if (row >= a.rows) continue;
            const size_t o = (size_t)ocol * a.rows + row;
            a.y[o] = a.resid ? a.resid[o] + acc[j] : acc[j];
        }
    }
}

template <int T>
int launch_q8_gemm(const GemmArgs &ga, hipStream_t stream) {
    static std::atomic<uint64_t> raised{0}; // per device: the ring's dynamic LDS allowed
    int dev = 0;
    AQ_HIP(hipGetDevice(&dev));
    constexpr int lds = Q8Stage<T>::BYTES * Q8Stage<T>::RING;
    if (!(raised.load() & (1ull << (dev & 63)))) {
        AQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(q8_gemm_kernel<T>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        raised.fetch_or(1ull << (dev & 63));
    }
    const dim3 grid((unsigned)((ga.rows + 31) / 32), (unsigned)((ga.ncols + 63) / 64));
    hipLaunchKernelGGL(q8_gemm_kernel<T>, grid, dim3(512), lds, stream, ga);
    return hipGetLastError() == hipSuccess ? 0 : fail(AQ_EHIP, "q8_gemm launch");
}

template <int T, int CT>
int launch_kq_ct(GemmArgs ga, hipStream_t stream) {
    static std::atomic<uint64_t> raised{0}; // per device: the ring's dynamic LDS allowed
    int dev = 0;
    AQ_HIP(hipGetDevice(&dev));
    const size_t lds = kq_lds<T, CT>();
    if (!(raised.load() & (1ull << (dev & 63)))) {
        AQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kq_gemm_kernel<T, CT>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        raised.fetch_or(1ull << (dev & 63));
    }
    // A last pass over the CUs whose column tiles fit one pass runs one column tile per work-group (a step of one tile
    // costs 0.55 of a step of four): the 544 work-groups of 17408 rows are 2.1 passes of 256.
    const int n = (ga.rows + 31) / 32, over = n % GEMM_CUS;
    ga.nfull = CT > 2 && n > GEMM_CUS && over * CT <= GEMM_CUS ? n - over : n;
    const unsigned grid = (unsigned)(ga.nfull + (n - ga.nfull) * CT);
    hipLaunchKernelGGL((kq_gemm_kernel<T, CT>), dim3(grid), dim3(512), lds, stream, ga);
    return hipGetLastError() == hipSuccess ? 0 : fail(AQ_EHIP, "kq_gemm launch");
}

template <int T>
int launch_kq_gemm(const GemmArgs &ga, hipStream_t stream) {
    switch ((ga.ncols + 15) / 16) {
    case 1: return launch_kq_ct<T, 1>(ga, stream);
    case 2: return launch_kq_ct<T, 2>(ga, stream);
    case 3: return launch_kq_ct<T, 3>(ga, stream);
    default: return launch_kq_ct<T, 4>(ga, stream);
    }
}

} // namespace

int launch_gemm(const Weight &w, const Act &x, size_t ncols, float *y, const float *resid, hipStream_t stream) {
    AQ_REQUIRE(ncols >= 1 && ncols <= x.ncols, "gemm: ncols out of range");
    AQ_REQUIRE(w.cols == x.n, "gemm: activation length != weight columns");
    AQ_REQUIRE(w.rows >= 1 && w.rows <= (size_t)INT32_MAX && ncols <= (size_t)INT32_MAX, "gemm: shape");
    GemmArgs ga{};
    ga.qa = w.qa;
    ga.qb = w.qb;
    ga.sc = w.sc;
    ga.dm = w.dm;
    ga.rows = (int)w.rows;
    ga.nb = (int)w.nb;
    ga.ncols = (int)ncols;
    ga.n = x.n;
    ga.y = y;
    ga.resid = resid;
    if (is_kquant(w.type)) {
        AQ_REQUIRE(w.cols % 256 == 0, "gemm: K-quant columns must be a multiple of 256");
        AQ_REQUIRE(x.gh && x.gm && x.gcap >= ncols && x.gcol == 0, "gemm: the activation has no many-column form");
        AQ_REQUIRE(ncols <= 64, "gemm: at most 64 columns");
        ga.gh = x.gh;
        ga.gm = x.gm;
        ga.gcap = (uint32_t)x.gcap;
        switch (w.type) {
        case AQ_TYPE_Q4_K: return launch_kq_gemm<AQ_TYPE_Q4_K>(ga, stream);
        case AQ_TYPE_Q5_K: return launch_kq_gemm<AQ_TYPE_Q5_K>(ga, stream);
        default: return launch_kq_gemm<AQ_TYPE_Q6_K>(ga, stream);
        }
    }
    AQ_REQUIRE(w.type == AQ_TYPE_Q8_0 || w.type == AQ_TYPE_Q4_0, "gemm: weight type");
    AQ_REQUIRE(w.cols % 256 == 0, "gemm: Q8_0 / Q4_0 columns must be a multiple of 256");
    ga.xq = x.q0;
    ga.xd = x.d0;
    if (w.type == AQ_TYPE_Q8_0) return launch_q8_gemm<AQ_TYPE_Q8_0>(ga, stream);
    return launch_q8_gemm<AQ_TYPE_Q4_0>(ga, stream);
}

} // namespace aq
