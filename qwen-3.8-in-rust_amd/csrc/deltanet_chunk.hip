// deltanet_chunk.hip — the Gated-DeltaNet mixer's core over a prompt chunk's rows (gated_deltanet.rs:197-255, which steps
// the recurrence token by token; arithmetic as dn_core_body in ops.hip, gated_deltanet.rs:261-375), in three launches:
//   inputs      every row and channel at once: conv + SiLU, l2norm of q and k, the decays and betas, the new conv window;
//   recurrence  the rows in order, state columns spread over the chip;
//   output      every row and head at once: the gated RMSNorm and its Q8_0 form.
// In one launch per chunk a head's rows, norms and outputs shared one work-group: 48 of 256 CUs, two waves per SIMD, the
// ordered sums over the keys handed between waves through the LDS and work-group barriers, 138 us per 64 rows at
// 48 heads x 128 x 128; here 6 + 55 + 6. The recurrence is bound by its own adds (0.85 us per row).
//
// The recurrence keeps each ordered sum inside a wave: lane (c, j) holds the DK / 8 keys j * DK / 8 .. of state column c,
// a sum runs through the lanes of a column in key order, the running value moved one lane up after each lane's terms
// (DPP row shift). Every lane adds at every step (only the lane whose turn it is holds the true sum), 128 adds per sum;
// what the split saves is the element-wise work: 16 keys per lane instead of 32, and no barrier.
#include "ops.h"
#include "quant_dev.h"

namespace aq {
namespace {

// The chunk's scratch: per row [q normalised and scaled | k normalised | v], then the decays and betas [t][nv].
struct DnPre {
    float *qkv, *decay, *beta;
    int kd, vd, cd;
};
__host__ __device__ inline DnPre dn_pre(const DnArgs &a) {
    DnPre p;
    p.kd = a.nk * a.dk;
    p.vd = a.nv * a.dv;
    p.cd = 2 * p.kd + p.vd;
    p.qkv = a.pre;
    p.decay = a.pre + (size_t)a.t * p.cd;
    p.beta = p.decay + (size_t)a.t * a.nv;
    return p;
}

// conv.rs:11-36 of channel ch at row i over the inputs of rows i - 3 .. i (before row 0: the window), then SiLU.
__device__ __forceinline__ float conv_silu(const DnArgs &a, int cd, int ch, int i) {
    float acc = 0.0f;
    const float4 w = *reinterpret_cast<const float4 *>(a.conv_w + (size_t)ch * 4);
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int r = i - 3 + e;
        x[e] = r < 0 ? a.conv_src[(size_t)ch * 3 + r + 3] : a.mixed[(size_t)r * cd + ch];
    }
    acc += w.x * x[0];
    acc += w.y * x[1];
    acc += w.z * x[2];
    acc += w.w * x[3];
    return silu_f(acc);
}

// Work-group (x, row): x < nk the q and k channels of K head x; then 256 v channels each; the last one the gates.
// The last row's work-groups also write their channels' new conv window (the last three input rows).
__global__ void __launch_bounds__(256) dn_inputs_kernel(DnArgs a) {
    __shared__ float sq[512], inv[2];
    const DnPre p = dn_pre(a);
    const int tid = threadIdx.x, i = blockIdx.y, x = blockIdx.x, nvb = (p.vd + 255) / 256, dk = a.dk;
    auto window = [&](int ch) {
        if (i == a.t - 1 && a.conv_dst)
            for (int e = 0; e < 3; e++) a.conv_dst[(size_t)ch * 3 + e] = a.mixed[(size_t)(a.t - 3 + e) * p.cd + ch];
    };
    if (x < a.nk) {
        float v[2];
        for (int k = 0; k < 2; k++) { // 2 dk <= 512 channels
            const int c = tid + k * 256;
            if (c >= 2 * dk) break;
            const int ch = (c < dk ? 0 : p.kd - dk) + x * dk + c;
            v[k] = conv_silu(a, p.cd, ch, i);
            sq[c] = v[k] * v[k];
            window(ch);
        }
        __syncthreads();
        // deltanet.rs:19-29 l2norm: one ordered sum for q, one for k, each in eight lanes of wave 0 (lane m of a sum
        // holds terms m T .. m T + T - 1, the running sum moved one lane up after each lane's terms)
        if (tid < 64) {
            const int s = (tid >> 3) & 1, m = tid & 7, T = dk / 8;
            float ss = 0.0f;
            const float *src = sq + s * dk + m * T;
            if (dk == 128) {
                float r[16];
#pragma unroll
                for (int u = 0; u < 16; u++) r[u] = src[u];
#pragma unroll
                for (int st = 0; st < 8; st++) {
                    if (st > 0)
                        ss = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x111, 0xF, 0xF, false));
#pragma unroll
                    for (int u = 0; u < 16; u++) ss += r[u];
                }
            } else {
                for (int st = 0; st < 8; st++) {
                    if (st > 0)
                        ss = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x111, 0xF, 0xF, false));
                    for (int u = 0; u < T; u++) ss += src[u];
                }
            }
            if (tid < 16 && m == 7) inv[s] = 1.0f / sqrtf(ss + 1e-6f);
        }
        __syncthreads();
        for (int k = 0; k < 2; k++) {
            const int c = tid + k * 256;
            if (c >= 2 * dk) break;
            const bool isq = c < dk;
            const int ch = (isq ? 0 : p.kd - dk) + x * dk + c;
            p.qkv[(size_t)i * p.cd + ch] = isq ? (v[k] * inv[0]) * a.qscale : v[k] * inv[1];
        }
    } else if (x < a.nk + nvb) {
        const int c = (x - a.nk) * 256 + tid;
        if (c >= p.vd) return;
        const int ch = 2 * p.kd + c;
        p.qkv[(size_t)i * p.cd + ch] = conv_silu(a, p.cd, ch, i);
        window(ch);
    } else {
        for (int h = tid; h < a.nv; h += 256) {
            const size_t e = (size_t)i * a.nv + h;
            p.decay[e] = exp_f(a.ssm_a[h] * softplus_f(a.a[e] + a.dt_bias[h])); // deltanet.rs:32-35 gate_g
            p.beta[e] = sigmoid_f(a.b[e]);
        }
    }
}

// Sum over a column's eight lanes in key order: acc from the lane below, then this lane's terms; lane 7 ends with it.
template <int KH>
__device__ __forceinline__ float lane_chain(const float (&x)[KH]) {
    float acc = 0.0f;
#pragma unroll
    for (int m = 0; m < 8; m++) {
        if (m > 0) acc = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc), 0x111, 0xF, 0xF, false));
#pragma unroll
        for (int k = 0; k < KH; k++) acc += x[k];
    }
    return acc;
}
// Lane 7 of each group of eight, to all eight.
__device__ __forceinline__ float from_lane7(float v) {
    // rows of 16: lanes 0-7 take lane 7's value, lanes 8-15 lane 15's
    const int lo = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x157, 0xF, 0x3, true); // row_newbcast:7
    const int r = __builtin_amdgcn_update_dpp(lo, __float_as_int(v), 0x15F, 0xF, 0xC, false); // row_newbcast:15
    return __int_as_float(r);
}

// Work-group (head, 32 columns): wave w columns 8 w .. 8 w + 7, lane = column * 8 + key part. deltanet.rs:43-86 per row:
// S *= decay; kv = sum_k S k; delta = (v - kv) beta; S += k delta; o = sum_k S q. The next row's inputs are loaded while
// this one's sums run.
template <int DK>
__global__ void __launch_bounds__(256) dn_recurrence_kernel(DnArgs a) {
    constexpr int KH = DK / 8;
    static_assert(KH % 4 == 0, "whole float4s of a row per lane");
    const DnPre p = dn_pre(a);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dv = a.dv;
    const int ncb = (dv + 31) / 32, h = (int)blockIdx.x / ncb, c0 = ((int)blockIdx.x % ncb) * 32 + wave * 8;
    if (c0 >= dv) return; // whole waves: dv is a multiple of 8
    const int c = c0 + (lane >> 3), j = lane & 7, kh = h % a.nk;
    float *srec = a.rec + ((size_t)h * DK + j * KH) * dv + c;
    float s[KH], k[2][KH], q[2][KH], v[2], de[2], be[2];
#pragma unroll
    for (int u = 0; u < KH; u++) s[u] = srec[(size_t)u * dv];
    auto load = [&](int b, int i) {
        const float *row = p.qkv + (size_t)i * p.cd;
        const float *qs = row + kh * DK + j * KH, *ks = row + p.kd + kh * DK + j * KH;
#pragma unroll
        for (int u = 0; u < KH; u += 4) {
            const float4 q4 = *reinterpret_cast<const float4 *>(qs + u), k4 = *reinterpret_cast<const float4 *>(ks + u);
            q[b][u] = q4.x;
            q[b][u + 1] = q4.y;
            q[b][u + 2] = q4.z;
            q[b][u + 3] = q4.w;
            k[b][u] = k4.x;
            k[b][u + 1] = k4.y;
            k[b][u + 2] = k4.z;
            k[b][u + 3] = k4.w;
        }
        v[b] = row[2 * p.kd + h * dv + c];
        de[b] = p.decay[(size_t)i * a.nv + h];
        be[b] = p.beta[(size_t)i * a.nv + h];
    };
    auto step = [&](int b, int i) {
        float x[KH];
#pragma unroll
        for (int u = 0; u < KH; u++) {
            s[u] *= de[b];
            x[u] = s[u] * k[b][u];
        }
        const float kv = lane_chain<KH>(x);
        const float delta = from_lane7((v[b] - kv) * be[b]); // lane 7 holds the sum, and its own v and beta
#pragma unroll
        for (int u = 0; u < KH; u++) {
            s[u] += k[b][u] * delta;
            x[u] = s[u] * q[b][u];
        }
        const float o = lane_chain<KH>(x);
        if (j == 7) a.out[(size_t)i * p.vd + h * dv + c] = o;
    };
    load(0, 0);
    int i = 0;
    for (; i + 1 < a.t; i += 2) {
        load(1, i + 1);
        step(0, i);
        load(0, i + 2 < a.t ? i + 2 : a.t - 1);
        step(1, i + 1);
    }
    if (i < a.t) step(0, i);
#pragma unroll
    for (int u = 0; u < KH; u++) srec[(size_t)u * dv] = s[u];
}

// The isolated recurrence of a verify batch: inputs as given (4-byte aligned), the state written as it stands after row
// a.keep - 1 (keep 0: not at all), the work split as above: one launch over 192 work-groups at 48 heads x 128 x 128, where
// the heads' own work-groups ran every row and then the kept ones again: 10.4 us for 4 rows instead of 17. (One kernel
// for both kept the chunk's loads from overlapping its sums: 70 us per 64 rows instead of 55.)
typedef float dn_f4u __attribute__((ext_vector_type(4), aligned(4)));

template <int DK>
__global__ void __launch_bounds__(256) dn_raw_kernel(DnArgs a) {
    constexpr int KH = DK / 8;
    const DnPre p = dn_pre(a);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dv = a.dv;
    const int ncb = (dv + 31) / 32, h = (int)blockIdx.x / ncb, c0 = ((int)blockIdx.x % ncb) * 32 + wave * 8;
    if (c0 >= dv) return; // whole waves: dv is a multiple of 8
    const int c = c0 + (lane >> 3), j = lane & 7, kh = h % a.nk;
    float *srec = a.rec + ((size_t)h * DK + j * KH) * dv + c;
    float s[KH], k[2][KH], q[2][KH], v[2], de[2], be[2];
#pragma unroll
    for (int u = 0; u < KH; u++) s[u] = srec[(size_t)u * dv];
    auto load = [&](int b, int i) {
        const size_t at = (size_t)kh * DK + j * KH, e = (size_t)i * a.nv + h;
        const float *qs = a.rq + (size_t)i * p.kd + at;
        const float *ks = a.rk + (size_t)i * p.kd + at;
        if constexpr (KH % 4 == 0) {
#pragma unroll
            for (int u = 0; u < KH; u += 4) {
                const dn_f4u q4 = *reinterpret_cast<const dn_f4u *>(qs + u);
                const dn_f4u k4 = *reinterpret_cast<const dn_f4u *>(ks + u);
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    q[b][u + w] = q4[w];
                    k[b][u + w] = k4[w];
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < KH; u++) {
                q[b][u] = qs[u];
                k[b][u] = ks[u];
            }
        }
        v[b] = a.rv[(size_t)i * p.vd + h * dv + c];
        de[b] = exp_f(a.rg[e]);
        be[b] = a.rbeta[e];
    };
    auto store = [&]() {
#pragma unroll
        for (int u = 0; u < KH; u++) srec[(size_t)u * dv] = s[u];
    };
    auto step = [&](int b, int i) {
        float x[KH];
#pragma unroll
        for (int u = 0; u < KH; u++) {
            s[u] *= de[b];
            x[u] = s[u] * k[b][u];
        }
        const float kv = lane_chain<KH>(x);
        const float delta = from_lane7((v[b] - kv) * be[b]); // lane 7 holds the sum, and its own v and beta
#pragma unroll
        for (int u = 0; u < KH; u++) {
            s[u] += k[b][u] * delta;
            x[u] = s[u] * q[b][u];
        }
        const float o = lane_chain<KH>(x);
        if (j == 7) a.out[(size_t)i * p.vd + h * dv + c] = o;
        if (i + 1 == a.keep) store();
    };
    load(0, 0);
    int i = 0;
    for (; i + 1 < a.t; i += 2) {
        load(1, i + 1);
        step(0, i);
        load(0, i + 2 < a.t ? i + 2 : a.t - 1);
        step(1, i + 1);
    }
    if (i < a.t) step(0, i);
}

// A model's key head sizes (a prompt chunk), and the smaller ones that the isolated recurrence takes as well.
template <bool RAW>
bool launch_recurrence(const DnArgs &a, hipStream_t stream) {
    const dim3 grid((unsigned)(a.nv * ((a.dv + 31) / 32)));
    if constexpr (RAW) {
        switch (a.dk) {
        case 8: hipLaunchKernelGGL(dn_raw_kernel<8>, grid, dim3(256), 0, stream, a); return true;
        case 16: hipLaunchKernelGGL(dn_raw_kernel<16>, grid, dim3(256), 0, stream, a); return true;
        case 32: hipLaunchKernelGGL(dn_raw_kernel<32>, grid, dim3(256), 0, stream, a); return true;
        case 64: hipLaunchKernelGGL(dn_raw_kernel<64>, grid, dim3(256), 0, stream, a); return true;
        case 128: hipLaunchKernelGGL(dn_raw_kernel<128>, grid, dim3(256), 0, stream, a); return true;
        }
    } else {
        switch (a.dk) {
        case 64: hipLaunchKernelGGL(dn_recurrence_kernel<64>, grid, dim3(256), 0, stream, a); return true;
        case 128: hipLaunchKernelGGL(dn_recurrence_kernel<128>, grid, dim3(256), 0, stream, a); return true;
        }
    }
    return false;
}

// Work-group (head, row): y = (w * (o * inv_rms(o))) * silu(z) (rmsnorm.rs:37-46) in place over the recurrence's output,
// and its Q8_0 form.
__global__ void __launch_bounds__(256) dn_output_kernel(DnArgs a) {
    __shared__ float so[256], ro;
    const int p = blockIdx.x, i = blockIdx.y, tid = threadIdx.x, dv = a.dv, vd = a.nv * dv;
    const size_t e = (size_t)i * vd + (size_t)p * dv + tid;
    const bool live = tid < dv;
    float zv = 0.0f, w = 0.0f;
    if (live) {
        so[tid] = a.out[e];
        zv = a.z[e];
        w = a.ssm_norm[tid];
    }
    __syncthreads();
    if (tid < 64) { // eight interleaved sums, then reduce8 (the launch's head sizes are multiples of 8)
        const int m = tid & 7;
        float r8 = tid < 8 ? seq_sum<true>(so, m, dv / 8 * 8, 8, 0.0f) : 0.0f;
        r8 = r8 + __int_as_float(dpp_mov<0x104>(__float_as_int(r8))); // row_shl:4
        r8 = r8 + __int_as_float(dpp_mov<0x102>(__float_as_int(r8))); // row_shl:2
        r8 = r8 + __int_as_float(dpp_mov<0x101>(__float_as_int(r8))); // row_shl:1
        if (tid == 0) ro = 1.0f / sqrtf(r8 / (float)dv + a.eps);
    }
    __syncthreads();
    if (!live) return;
    const float v = (w * (so[tid] * ro)) * silu_f(zv);
    a.out[e] = v;
    if (a.out_q80) q8_0_block_half(a.q80, i, (size_t)p * (dv / 32) + (tid >> 5), v, tid & 63); // dv % 32 == 0
}

int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(AQ_EHIP, std::string(what) + " launch: " + hipGetErrorString(e));
}

} // namespace

size_t dn_chunk_floats(const DnArgs &a) {
    return (size_t)a.t * (2 * (size_t)a.nk * a.dk + (size_t)a.nv * a.dv + 2 * (size_t)a.nv);
}

int launch_dn_chunk(const DnArgs &a, hipStream_t stream) {
    AQ_REQUIRE(a.out && a.z && a.ssm_norm && a.pre && a.write_state && a.t >= 3 && a.t <= 4096,
               "deltanet: more than 8 rows are a prompt chunk (output, state written)");
    AQ_REQUIRE(a.dv % 8 == 0 && a.dv <= 256 && 2 * a.dk <= 512 && ((uintptr_t)a.pre & 15) == 0 &&
                   ((uintptr_t)a.conv_w & 15) == 0,
               "deltanet: chunk shape");
    const int vd = a.nv * a.dv;
    hipLaunchKernelGGL(dn_inputs_kernel, dim3((unsigned)(a.nk + (vd + 255) / 256 + 1), (unsigned)a.t), dim3(256), 0, stream, a);
    int rc = launched("deltanet inputs");
    if (rc) return rc;
    if (!launch_recurrence<false>(a, stream))
        return fail(AQ_EUNSUP, "deltanet: head dims (k, v) not built: " + std::to_string(a.dk) + ", " + std::to_string(a.dv));
    if ((rc = launched("deltanet recurrence"))) return rc;
    hipLaunchKernelGGL(dn_output_kernel, dim3((unsigned)a.nv, (unsigned)a.t), dim3(256), 0, stream, a);
    return launched("deltanet output");
}

int launch_dn_raw(const DnArgs &a, hipStream_t stream) {
    AQ_REQUIRE(a.t >= 1 && a.nk >= 1 && a.nv >= 1 && a.nv % a.nk == 0, "deltanet: head counts");
    AQ_REQUIRE(a.dv >= 1 && a.dv <= 256, "deltanet: head_dim_v must be 1..256");
    AQ_REQUIRE(a.rec, "deltanet: no state");
    AQ_REQUIRE(a.rq && a.rk && a.rv && a.rg && a.rbeta && a.out && a.keep <= a.t, "deltanet: raw inputs");
    const bool built = a.dk == a.dv ? a.dk <= 128 : (a.dk == 128 && a.dv == 256) || (a.dk == 64 && a.dv == 128);
    if (!built || !launch_recurrence<true>(a, stream))
        return fail(AQ_EUNSUP, "deltanet: head dims (k, v) not built: " + std::to_string(a.dk) + ", " + std::to_string(a.dv));
    return launched("deltanet recurrence");
}

} // namespace aq
