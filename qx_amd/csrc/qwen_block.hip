// Qwen3-30B-A3B attention half with group-32 Q4 projections
// (PreparedQwenLayer::encode_with_expert_cache, crates/qx-runtime-v2/src/lib.rs:
// 904-973; kernels qx_qwen_rms_norm / qx_qwen_residual_rms_norm,
// kernels/qwen_attention.metal:4-58, and the Q4 stage qx_q4_gemv,
// kernels/q4_expert.metal:31-58), f16 activations between stages:
//
//   kernel 1  rms_norm(hidden) -> f16 -> Q4 q (4096 rows), k, v (512 rows each)
//             over 2048 columns -> f16 q/k/v in the workspace
//   then      the Qwen front end (per-head q/k RMSNorm + RoPE, K/V append)
//             and split-K decode attention: on equal 16-bit caches one
//             launch (decode_mfma_front_kernel, decode_attention.hip), else
//             rope_append.hip's kernel, then the decode
//   kernel 3  Q4 o projection (2048 rows over 4096 columns) -> f16
//   kernel 4  hidden_after = f16(hidden + o); moe_input = f16(rms_norm(hidden_after))
//
// A Q4 row is summed group by group (32 columns a lane), then across the wave;
// the reference's Qwen stage folds each row sequentially in one thread, so the
// two agree to rounding, which f16 outputs mostly absorb.  The norms reduce
// per wave, then across waves, and use the consensus rsqrt of the Metal
// kernels.
#include "common.h"
#include "consensus_math.h"
#include "internal.h"
#include "q4_common.h"

namespace qxh {

namespace {

constexpr int kQwenHidden = 2048;
constexpr int kQwenQRows = 4096;
constexpr int kQwenKvRows = 512;
constexpr float kQwenEps = 1e-6f;

// Sum of x^2 over a 2048-wide vector held as x[t + 256 k] (k < 8) by the
// 256 threads of the workgroup; every thread gets the total.  Ends with a
// barrier.
__device__ __forceinline__ float square_sum_256(const float (&x)[8], float* wave_sums) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += x[k] * x[k];
    s = group_sum<64>(s);
    if ((threadIdx.x & 63) == 0) wave_sums[threadIdx.x >> 6] = s;
    __syncthreads();
    return (wave_sums[0] + wave_sums[1]) + (wave_sums[2] + wave_sums[3]);
}

__device__ __forceinline__ float qwen_inverse_rms(float total) {
    return consensus_rsqrt(total / (float)kQwenHidden + kQwenEps);
}

// ---- Q4 rows, a group per lane ------------------------------------------------
// A wave takes whole rows: lane l holds group l (and l + 64 of the 128-group o
// rows) of each, one 16-byte load a row, and the same group's 32 input values
// for all of them, in registers.  The inputs are f16 values, kept as 16 pairs,
// and every product is a v_fma_mix_f32: f16 factors, fp32 accumulation.
// Nibbles s and s + 4 of a code word (values 8 w + s and 8 w + s + 4 of the
// group) become a pair of f16 codes with one mask and one packed subtraction
// (0x6400 | n is 1024 + n), so the inputs are paired the same way.
//
// 10.6 MB of codes a layer: both kernels are bound by their dispatch and one
// round trip to HBM (4.5 and 4.0 to 4.5 us traced; the codes alone take 0.9 and 0.7).
// Measured, 48 layers at 32768 positions, us a token: a row's codes dealt
// back to the reference's 32 lanes through LDS (two LDS reads and eight VALU
// instructions a value) 1565; a group per lane, each wave normalising the
// whole hidden state from its own 64-byte slices 1343; the norm shared by the
// workgroup, whose 16-byte loads are coalesced, 1284.
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
// Inputs in LDS: a group's 32 values in 40 halves, so that the 16-byte reads
// of 64 lanes, a group each, fall on all banks.
constexpr int kGroupPad = 40;

// Eight consecutive f16 values as the pairs (s, s + 4).
__device__ __forceinline__ u32x4 pair_up(const u32x4& raw) {
    return u32x4{__builtin_amdgcn_perm(raw[2], raw[0], 0x05040100u), __builtin_amdgcn_perm(raw[2], raw[0], 0x07060302u),
                 __builtin_amdgcn_perm(raw[3], raw[1], 0x05040100u), __builtin_amdgcn_perm(raw[3], raw[1], 0x07060302u)};
}

__device__ __forceinline__ void read_pairs(const uint16_t* s_x, int group, h2 (&x)[16]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(s_x + group * kGroupPad + 8 * w);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint32_t word = v[s];  // a bit cast of the element itself reads element 0
            x[4 * w + s] = __builtin_bit_cast(h2, word);
        }
    }
}

// sum over a group of (code - 7) * x
__device__ __forceinline__ float group_dot(const u32x4& codes, const h2 (&x)[16]) {
    float acc[2] = {0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const h2 c = __builtin_bit_cast(h2, ((codes[w] >> (4 * s)) & 0x000f000fu) | 0x64006400u) -
                         h2{(_Float16)1031.0f, (_Float16)1031.0f};
            const h2 v = x[4 * w + s];
            acc[0] = __builtin_fmaf((float)c[0], (float)v[0], acc[0]);
            acc[1] = __builtin_fmaf((float)c[1], (float)v[1], acc[1]);
        }
    return acc[0] + acc[1];
}

// grid 256 workgroups x 5 waves of 4 rows: 20 of the 5120 stacked [q; k; v]
// rows a CU (no wave straddles two matrices).
constexpr int kQkvWaves = 5, kQkvRows = 4;
static_assert((kQwenQRows + 2 * kQwenKvRows) % (kQkvWaves * kQkvRows) == 0 && kQwenQRows % kQkvRows == 0 &&
                  kQwenKvRows % kQkvRows == 0,
              "whole workgroups, waves inside one matrix");

__global__ __launch_bounds__(64 * kQkvWaves) void qwen_norm_qkv_kernel(QwenBlockArgs a) {
    const int lane = threadIdx.x & 63;
    const int grow = (int)(blockIdx.x * kQkvWaves + (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kQkvRows;
    Q4View m;
    int row;
    uint16_t* out;
    if (grow < kQwenQRows) {
        m = a.wq;
        row = grow;
        out = a.query;
    } else if (grow < kQwenQRows + kQwenKvRows) {
        m = a.wk;
        row = grow - kQwenQRows;
        out = a.key;
    } else {
        m = a.wv;
        row = grow - kQwenQRows - kQwenKvRows;
        out = a.value;
    }
    constexpr int kGroups = kQwenHidden / 32;  // 64
    static_assert(kGroups == 64, "a group per lane");
    // Threads 0-255 normalise eight values each; the pairs go to the lanes
    // that hold their groups through LDS.  Loads complete in order: the hidden
    // state and norm weights (L2) first, then the Q4 rows from HBM, so the norm
    // runs while the rows are in flight.
    __shared__ __attribute__((aligned(16))) uint16_t s_x[kGroups * kGroupPad];
    __shared__ float wave_sums[4];
    const int t = threadIdx.x & 255;
    const bool norms = threadIdx.x < 256;
    const u32x4 hraw = load16_any(a.hidden + 8 * t);
    u32x4 wraw[2], codes[kQkvRows];
    uint16_t scale[kQkvRows];
#pragma unroll
    for (int i = 0; i < 2; ++i) wraw[i] = load16_any(a.input_norm + 8 * t + 4 * i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < kQkvRows; ++r) {
        codes[r] = load16<false>(m.packed + (size_t)(row + r) * (kQwenHidden / 2) + lane * 16);
        scale[r] = m.scales[(row + r) * kGroups + lane];
    }
    __builtin_amdgcn_sched_barrier(0);
    float x[8];
    Unpack<F16>::run(hraw, x);
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(x[i], x[i], ss);
    ss = group_sum<64>(ss);
    if (norms && lane == 0) wave_sums[threadIdx.x >> 6] = ss;
    __syncthreads();
    if (norms) {
        const float inv = qwen_inverse_rms((wave_sums[0] + wave_sums[1]) + (wave_sums[2] + wave_sums[3]));
        u32x4 y;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            h2 v;
#pragma unroll
            for (int e = 0; e < 2; ++e) v[e] = (_Float16)(x[s + 4 * e] * inv * __uint_as_float(wraw[e][s]));
            y[s] = __builtin_bit_cast(uint32_t, v);
        }
        *reinterpret_cast<u32x4*>(s_x + (t >> 2) * kGroupPad + 8 * (t & 3)) = y;
    }
    __syncthreads();
    h2 pairs[16];
    read_pairs(s_x, lane, pairs);
    float sum[kQkvRows];
#pragma unroll
    for (int r = 0; r < kQkvRows; ++r)
        sum[r] = group_sum<64>(group_dot(codes[r], pairs) * f16_bits_to_float(scale[r]));
    if (lane < kQkvRows) {
        float v = sum[0];
#pragma unroll
        for (int r = 1; r < kQkvRows; ++r)
            if (lane == r) v = sum[r];
        out[row + lane] = f16_bits(v);
    }
}

// grid 256 workgroups x 4 waves, two o rows per wave over the 4096 attention
// values: groups l and l + 64 of each.
constexpr int kOutRows = 2;

__global__ __launch_bounds__(256) void qwen_out_kernel(QwenBlockArgs a) {
    const int lane = threadIdx.x & 63;
    const int row = (int)(blockIdx.x * 4 + (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kOutRows;
    constexpr int kGroups = kQwenQRows / 32;  // 128
    __shared__ __attribute__((aligned(16))) uint16_t s_x[kGroups * kGroupPad];
    u32x4 codes[kOutRows][2], raw[2];
    uint16_t scale[kOutRows][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) raw[j] = load16<false>(a.attention + 8 * (threadIdx.x + 256 * j));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < kOutRows; ++r)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            codes[r][j] = load16<false>(a.wo.packed + (size_t)(row + r) * (kQwenQRows / 2) + (lane + 64 * j) * 16);
            scale[r][j] = a.wo.scales[(row + r) * kGroups + lane + 64 * j];
        }
    __builtin_amdgcn_sched_barrier(0);  // every request out before the first use
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c = threadIdx.x + 256 * j;
        *reinterpret_cast<u32x4*>(s_x + (c >> 2) * kGroupPad + 8 * (c & 3)) = pair_up(raw[j]);
    }
    __syncthreads();
    h2 x[2][16];
    read_pairs(s_x, lane, x[0]);
    read_pairs(s_x, lane + 64, x[1]);
    float sum[kOutRows];
#pragma unroll
    for (int r = 0; r < kOutRows; ++r)
        sum[r] = group_sum<64>(__builtin_fmaf(group_dot(codes[r][0], x[0]), f16_bits_to_float(scale[r][0]),
                                              group_dot(codes[r][1], x[1]) * f16_bits_to_float(scale[r][1])));
    if (lane < kOutRows) a.projection[row + lane] = f16_bits(lane == 0 ? sum[0] : sum[1]);
}

// One workgroup: hidden_after = f16(hidden + projection) (qx_qwen_residual_rms_norm,
// kernels/qwen_attention.metal:31-58), then moe_input = f16(hidden_after *
// inverse * norm) over the f16 values.
__global__ __launch_bounds__(256) void qwen_residual_norm_kernel(QwenBlockArgs a) {
    __shared__ float wave_sums[4];
    const int t = threadIdx.x;
    // every load before the first store: the stores may alias the inputs as
    // far as the compiler knows, so interleaving them would serialise the
    // eight loads of each array into eight round trips
    uint16_t hb[8], pb[8];
    float x[8], w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int i = t + 256 * k;
        hb[k] = a.hidden[i];
        pb[k] = a.projection[i];
        w[k] = a.post_norm[i];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        x[k] = round_f16(f16_bits_to_float(hb[k]) + f16_bits_to_float(pb[k]));
        a.hidden_after[t + 256 * k] = f16_bits(x[k]);
    }
    const float inv = qwen_inverse_rms(square_sum_256(x, wave_sums));
#pragma unroll
    for (int k = 0; k < 8; ++k) a.moe_input[t + 256 * k] = f16_bits(x[k] * inv * w[k]);
}

}  // namespace

hipError_t launch_qwen_norm_qkv(const QwenBlockArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(qwen_norm_qkv_kernel, dim3((kQwenQRows + 2 * kQwenKvRows) / (kQkvWaves * kQkvRows)),
                       dim3(64 * kQkvWaves), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_qwen_out(const QwenBlockArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(qwen_out_kernel, dim3(kQwenHidden / (4 * kOutRows)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_qwen_residual_norm(const QwenBlockArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(qwen_residual_norm_kernel, dim3(1), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace qxh
