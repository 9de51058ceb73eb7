// Causal prefill attention: the routing of every prefill call, and the exact
// pass over prefill_rows (prefill_rows.h) behind the pipelined kernel.
#include "prefill_rows.h"

namespace qxh {

// The exact pass after the pipelined kernel (bf16 caches), a few workgroups
// walking the query blocks.  Usually no V value is outside the f16 range:
// every workgroup then exits after one scan of the tile flags that the V^T
// pre-pass wrote for this call's tiles, so the launch costs little more than
// its dispatch.  Otherwise each flagged block runs on the exact path.
template <int D, int HW, int QW>
__global__ __launch_bounds__(512, 1) void prefill_exact_pass_kernel(PrefillArgs a, uint32_t blocks) {
    __shared__ __attribute__((aligned(16))) char lds[prefill_rows_lds_bytes<D>()];
    const uint32_t tiles = (a.start + a.tokens + 63) / 64;
    bool any = false;
    for (uint32_t i = threadIdx.x; i < a.kv_heads * tiles; i += blockDim.x)
        any |= a.tile_flags[(size_t)(i / tiles) * a.tile_flag_stride + i % tiles] != 0;
    if (!__syncthreads_or(any)) return;
    for (uint32_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        prefill_rows<D, HW, QW>(a, lds, b);
        __syncthreads();  // the next block overwrites the LDS tiles
    }
}

// workgroups of the exact pass after the pipelined kernel: one per CU at most
constexpr uint32_t kExactPassWgs = 256;

// Causal rows on the split-K decode kernels, for short prompts on any cache
// (and longer ones on Qwen-shape fp32 caches): the cached prefix is streamed,
// split over the CUs like a decode, once for every row or, on equal 16-bit
// caches, once for the rows that share a workgroup (decode_mfma_rows_kernel).
// That grows with rows x context but has no fixed cost beyond a decode's, while
// the pipelined MFMA prefill (equal 16-bit K/V) first rewrites the layer's whole
// V prefix into the f16 V^T scratch (bf16 and Qwen-shape caches; Granite f16
// caches skip that pass).
// Rows run on the decode kernels up to 8 of them, or, below 64, while rows x
// context stays under the crossover measured against the kernel the call would
// take otherwise (rows / tiled, us, 9-63 rows over 64-30000 cached positions,
// each case timed both ways):
// - Qwen (960000 up to 32 rows, 500000 beyond): 30000 + 16 38.9 / 66.1, 16000
//   + 32 41.2 / 50.1, 24000 + 32 54.4 / 59.6, 30000 + 24 54.0 / 66.2, 30000 +
//   32 64.4 / 66.3, 8000 + 48 38.2 / 44.0, 12000 + 48 47.4 / 48.2, 8000 + 63
//   44.8 / 44.2, 16000 + 63 70.4 / 51.2;
// - Granite f16 (500000, and at least 64 cached positions) and bf16 (500000):
//   the rows win over the whole range, f16 250 + 9 3.9 / 8.7, 2000 + 48 9.9 /
//   14.6, 3900 + 63 12.6 / 19.5, bf16 3900 + 63 13.2 / 22.3;
// - the Granite split-product kernel (36000; fp32 keys with tiered values
//   48500): Fp32KFp16V 500 + 63 16.9 / 19.4, 1000 + 32 18.2 / 19.0, 1500 + 24
//   19.0 / 16.7; fp32 K/V 1000 + 32 19.9 / 20.9, 1500 + 24 20.5 / 18.1, 3000 +
//   12 21.8 / 19.8; Fp16KFp32V 500 + 63 18.9 / 19.9, 4000 + 9 25.4 / 21.4;
//   tiered 4000 + 9 20.7 / 24.2, 4000 + 12 20.4 / 24.4, 1500 + 32 19.9 / 18.4;
// - the other Granite plans (tiered values with 16-bit keys): 40000;
// - Qwen with tiered values (150000), whose decode rows keep splits toward
//   2048 workgroups.
constexpr uint32_t kDecodeRowsAlways = 8;
static bool rows_on_decode(const ShapeDims& s, int key_dtype, int value_dtype, uint32_t start, uint32_t tokens) {
    if (tokens <= kDecodeRowsAlways) return true;
    if (tokens >= 64) return false;
    const uint64_t length = (uint64_t)start + tokens;
    if (s.group >= 8)
        return tokens * length <= (value_dtype == I8T ? 150000u : tokens <= 32 ? 960000u : 500000u);
    if (prefill_f32_supported(s, key_dtype, value_dtype))
        return tokens * length <= (value_dtype == I8T ? 48500u : 36000u);
    if (key_dtype == F16 && value_dtype == F16) return start >= 64 && tokens * length <= 500000u;
    if (key_dtype == BF16 && value_dtype == BF16) return tokens * length <= 500000u;
    return tokens * length <= 40000u;
}

static bool prefill_on_decode(const ShapeDims& s, int key_dtype, int value_dtype, uint32_t start, uint32_t tokens) {
    return key_dtype == F32 || key_dtype != value_dtype || !prefill_pipe_supported(s) ||
           rows_on_decode(s, key_dtype, value_dtype, start, tokens);
}

// Equal 16-bit caches take a query of another dtype on causal rows alone (the
// pipelined kernel reads the cache's own), up to this many of them: a limit of
// the call, so it does not follow rows_on_decode's crossover, which lies above
// it everywhere.
static bool takes_other_query(const ShapeDims& s, int key_dtype, uint32_t start, uint32_t tokens) {
    if (tokens <= kDecodeRowsAlways) return true;
    const uint64_t length = (uint64_t)start + tokens;
    if (tokens >= 64) return false;
    if (s.group >= 8) return (tokens - 6) * length <= 126000u;
    return key_dtype == F16 ? start >= 64 && tokens * length <= 70000u : tokens * length <= 90000u;
}

// fp32 and mixed K/V caches at the Granite shape beyond a few rows take the
// split-product kernel (prefill_f32.hip); Qwen-shape fp32 caches and
// tiered values stay on causal decode rows.
static bool prefill_on_f32(const ShapeDims& s, int key_dtype, int value_dtype, uint32_t start, uint32_t tokens) {
    return prefill_f32_supported(s, key_dtype, value_dtype) && !rows_on_decode(s, key_dtype, value_dtype, start, tokens);
}

// Tiered values with 16-bit keys take the pipelined MFMA prefill when the
// rows would (its V^T pre-pass reading the tiers); the others stay on the
// decode kernels.
static bool tiered_on_pipe(const ShapeDims& s, int key_dtype, int value_dtype, uint32_t start, uint32_t tokens) {
    return value_dtype == I8T && key_dtype != F32 && prefill_pipe_supported(s) &&
           !rows_on_decode(s, key_dtype, value_dtype, start, tokens);
}

// Covers every start position: below 64 rows a call may take either path.
uint64_t prefill_workspace_bytes(const ShapeDims& s, int key_dtype, int value_dtype, uint32_t capacity,
                                 uint32_t tokens) {
    const bool pipe_dtypes = key_dtype != F32 && (key_dtype == value_dtype || value_dtype == I8T) &&
                             prefill_pipe_supported(s);
    const uint64_t rows = decode_causal_workspace_bound(s, key_dtype, value_dtype, capacity, tokens);
    if (prefill_f32_supported(s, key_dtype, value_dtype) && tokens > kDecodeRowsAlways) {
        const uint64_t f32 = prefill_f32_workspace_bytes(s, capacity, tokens);
        return rows > f32 ? rows : f32;
    }
    if (!pipe_dtypes || tokens <= kDecodeRowsAlways) return rows;
    const uint64_t pipe = prefill_pipe_workspace_bytes(s, value_dtype, capacity, tokens);
    return tokens < 64 && rows > pipe ? rows : pipe;
}

hipError_t launch_prefill_attention(const ShapeDims& s, const KvLayer& kv, uint32_t start_position, uint32_t tokens,
                                    const void* query, int query_dtype, void* out, int out_dtype, void* workspace,
                                    hipStream_t st, int* dispatches) {
    *dispatches = 0;
    if (tiered_on_pipe(s, kv.key_dtype, kv.value_dtype, start_position, tokens)) {
        if (kv.key_dtype != query_dtype) return hipErrorNotSupported;
        return launch_prefill_pipe(s, kv, start_position, tokens, query, query_dtype, out, out_dtype, workspace, st,
                                   dispatches);
    }
    if (prefill_on_f32(s, kv.key_dtype, kv.value_dtype, start_position, tokens))
        return launch_prefill_f32(s, kv, start_position, tokens, query, query_dtype, out, out_dtype, workspace, st,
                                  dispatches);
    if (prefill_on_decode(s, kv.key_dtype, kv.value_dtype, start_position, tokens)) {
        if (kv.key_dtype != F32 && kv.key_dtype == kv.value_dtype && kv.key_dtype != query_dtype &&
            prefill_pipe_supported(s) && !takes_other_query(s, kv.key_dtype, start_position, tokens))
            return hipErrorNotSupported;
        const DecodePlan p = plan_decode_causal(s, kv.key_dtype, kv.value_dtype, start_position, tokens);
        return launch_decode_causal_rows(s, kv, p, start_position, tokens, query, query_dtype, out, out_dtype, workspace,
                                         st, dispatches);
    }
    if (kv.key_dtype != query_dtype) return hipErrorNotSupported;
    hipError_t e = launch_prefill_pipe(s, kv, start_position, tokens, query, query_dtype, out, out_dtype, workspace, st,
                                       dispatches);
    if (e != hipSuccess || query_dtype != BF16) return e;
    // bf16: the exact pass, for the rows the pipelined kernel left behind
    PrefillArgs a{};
    a.query = query;
    a.keys = kv.keys;
    a.values = kv.values;
    a.out = out;
    a.head_stride = kv.head_stride;
    a.start = start_position;
    a.tokens = tokens;
    a.q_heads = s.q_heads;
    a.group = s.group;
    a.out_dtype = out_dtype;
    a.scale_log2 = s.scale * kLog2e;
    a.kv_heads = s.kv_heads;
    a.tile_flags = reinterpret_cast<const uint32_t*>(workspace);
    a.tile_flag_stride = prefill_pipe_vt_tiles(kv.capacity);
    if (s.head_dim == 64 && s.group == 2) {
        a.qblocks = (tokens + 127) / 128;
        a.xcd_map = (8 % s.kv_heads == 0) && ((uint64_t)a.qblocks * s.kv_heads) % 8 == 0;
        const uint32_t blocks = a.qblocks * s.kv_heads;
        hipLaunchKernelGGL((prefill_exact_pass_kernel<64, 2, 4>), dim3(blocks < kExactPassWgs ? blocks : kExactPassWgs),
                           dim3(512), 0, st, a, blocks);
    } else if (s.head_dim == 128 && s.group == 8) {
        a.qblocks = (tokens + 31) / 32;
        a.xcd_map = (8 % s.kv_heads == 0) && ((uint64_t)a.qblocks * s.kv_heads) % 8 == 0;
        const uint32_t blocks = a.qblocks * s.kv_heads;
        hipLaunchKernelGGL((prefill_exact_pass_kernel<128, 8, 1>), dim3(blocks < kExactPassWgs ? blocks : kExactPassWgs),
                           dim3(512), 0, st, a, blocks);
    } else {
        return hipErrorNotSupported;
    }
    *dispatches += 1;
    return hipGetLastError();
}

}  // namespace qxh
