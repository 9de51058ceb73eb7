// Causal prefill on fp32 and mixed K/V caches at the Granite shape (16 q /
// 8 kv heads, d 64): the reference's KV plans Fp32KFp16V (its default) and
// Fp16KFp32V, fp32 K/V, their bf16 twins, and fp32 keys with tiered values.
// fp32 accuracy rules out rounding an operand to 16 bits, and the fp32 matrix
// cores run at a sixteenth of the 16-bit rate, so every fp32 operand is split
// into 16-bit pieces that hold all of its 24 significand bits, and each
// product is the sum of the piece products that matter:
//
//   x = x0 + x1 + x2      bf16: x0 is x rounded to nearest, x1 and x2 what is
//                         left rounded to nearest; f16 values are two pieces and
//                         bf16 values one, exactly.  bf16 has fp32's exponents,
//                         so a small probability keeps its bits as well (as f16
//                         pieces, below 2^-15 of the largest, it lost them: 4e-4
//                         of the result where a large value has a weight of
//                         2^-24)
//   x . y = sum of xi . yj with i + j <= 2, accumulated in fp32, the small
//                         products first.  |x1| <= 2^-8 and |x2| <= 2^-17 of x's
//                         leading bit, so x1 y2 + x2 y1, which is left out, is at
//                         most 2^-24 of the product, what an fp32 product is
//                         rounded by (2^-22 where x0 was cut off instead)
//
// A tile's products are summed by themselves before they join the running sums,
// so against 64 bits the result is closer than the fp32 matrix cores' was: 0.29
// to 0.69 of its error over six K/V plans, prompts of 30 to 3063 positions and
// scores spread by 0.1 to 4.
//
// Bound: a tile of Fp32KFp16V is 176 MFMAs a wave (2816 cycles of matrix core;
// 8192 on the fp32 cores) beside the softmax and the splits on the VALU.  At 2048
// tokens the matrix core is busy 31% of the kernel's cycles and the other vector
// instructions, at 4 cycles each, 34%; the rest is waits, with two waves a SIMD
// that meet at the tile's barriers.  1900 tokens take 70 us a layer, 97 on the
// fp32 cores.
//
// Transposed FlashAttention-2 on 16x16x32 MFMAs (operand layout: mfma.h):
//
//   S^T[pos][q]  = K[pos][:] . Q^T[:][q]       A = K pieces (LDS), B = Q^T pieces (registers)
//   O^T[d][q]   += V^T[d][pos] . P^T[pos][q]    A = V pieces (LDS, transposed reads), B = P^T pieces
//
// The S^T blocks leave in lane (g, i) exactly the positions that the
// transposed V reads (vt_operand_rows32) give it, so P^T needs no exchange.
//
// A workgroup of 4 waves owns a query block of 64 tokens x the 2 heads of a
// kv head (128 columns; wave w: tokens 16w .. 16w + 15, both heads), the
// column layout of the pipelined Granite kernel, so its split-KV partials go
// through the same prefill_combine_kernel.  K and V tiles of 64 positions are
// read with 16-byte loads, split once per workgroup and written to LDS as one
// 8 KB plane per piece, 16-byte chunks XOR-swizzled by row & 7 (conflict-free
// for both kinds of operand read); the next tile's loads are in flight while
// the current one is computed.  The online softmax keeps per-column (m, l) in
// every lane, m a score as the product left it; a score's distance from it is
// scaled by softmax scale x log2(e) in fp32 and exponentiated with v_exp_f32.
//
// A piece of an infinity, or a product that overflows where the whole one
// does not, would turn into a NaN, and the last piece of a value near fp32's
// least would lose bits below bf16's least, so a workgroup that meets a
// magnitude of 2^60 or more (a non-finite f16 value, say), a NaN, or an fp32
// value below 2^-80 that is not zero takes that tile's two products on the fp32
// matrix cores, straight from the cache, and keeps what a column does not
// attend out of its sums.  Keys and queries need no such least: what a piece
// loses there is below 2^-60 of a score's unit.  Nor do probabilities: a piece
// loses less than 2^-126 of the largest one, and v_exp_f32 itself ends there.
// 1900 tokens with such a value in every tile take 155 to 167 us a layer, with
// one in all no more than without.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "internal.h"
#include "mfma.h"
#include "prefill_split.h"

namespace qxh {

namespace {

constexpr int kD = 64;
constexpr float kNoScore = -3.4028234e38f;   // the running maximum before any score
constexpr int kTierBlockF32 = 32;           // elements per INT8 scale block of a tiered value cache
constexpr int kPlaneBytes = kPrefillTile * kD * 2;
constexpr float kSplitLimit = 0x1p60f;      // magnitudes the split products take
constexpr float kSplitLeast = 0x1p-80f;     // and the least of a value that is not zero

__device__ __forceinline__ f32x4 mma4(float a, float b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The next bf16 piece of the pair (a, b), packed (a in the low half), rounded
// to nearest; what it leaves of them stays in a and b.
__device__ __forceinline__ uint32_t round_bf16(float& a, float& b) {
    const uint32_t w = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
    a -= __uint_as_float(w << 16);
    b -= __uint_as_float(w & 0xffff0000u);
    return w;
}

// 8 values as NP packed bf16 pieces (the values are used up).
template <int NP> __device__ __forceinline__ void split8(float (&f)[8], u32x4 (&p)[NP]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NP; ++n) p[n][i] = round_bf16(f[2 * i], f[2 * i + 1]);
}

// NaN if one of them is (v_maximum3_f32, two values an instruction).
__device__ __forceinline__ float max_abs8(const float (&f)[8], float m) {
#pragma unroll
    for (int i = 0; i < 8; ++i) m = __builtin_elementwise_maximum(m, __builtin_fabsf(f[i]));
    return m;
}

// The least magnitude that is not zero (and m), as 2 |x| - 1 in its bits: zero
// wraps around to the largest.
__device__ __forceinline__ uint32_t min_bits8(const float (&f)[8], uint32_t m) {
#pragma unroll
    for (int i = 0; i < 8; ++i) m = min(m, (__float_as_uint(f[i]) << 1) - 1u);
    return m;
}

__device__ __forceinline__ bool finite(float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; }

// Byte offset of 16-byte chunk `col` of tile row `row` in a plane.
__device__ __forceinline__ int plane_chunk(int row, int col) { return row * (kD * 2) + ((col ^ (row & 7)) << 4); }

// 16 consecutive elements of a row, widened (the fp32 path's operands).
template <int DT> __device__ __forceinline__ void load_row16(const void* base, size_t idx, float (&f)[16]) {
    const char* p = reinterpret_cast<const char*>(base) + idx * (DT == F32 ? 4 : 2);
    constexpr int E = DT == F32 ? 4 : 8;  // elements a load
#pragma unroll
    for (int i = 0; i < 16 / E; ++i) {
        float x[E];
        Unpack<DT>::run(load16<false>(p + 16 * i), x);
#pragma unroll
        for (int e = 0; e < E; ++e) f[E * i + e] = x[e];
    }
}

// A 64 x 64 tile of one dtype: thread t moves chunks of 8 elements, chunk k at
// row t / 8 + 32 k, elements 8 (t % 8) .. + 7, and writes PIECES planes.
template <int DT, bool VALUES> struct SplitIo {
    static constexpr int EB = DT == F32 ? 4 : 2;
    static constexpr int PIECES = DT == F32 ? 3 : DT == F16 ? 2 : 1;
    static constexpr int WORDS = DT == F32 ? 2 : 1;  // 16-byte loads a chunk
    struct Raw {
        u32x4 w[2][WORDS];
    };
    // rows at or past kv_len read the last row instead (their positions are masked)
    __device__ __forceinline__ static void load(Raw& raw, const char* base, uint32_t tile, uint32_t kv_len, int tid) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t row = min(tile * kPrefillTile + (uint32_t)(tid >> 3) + 32 * k, kv_len - 1);
            const char* p = base + ((size_t)row * kD + 8 * (tid & 7)) * EB;
#pragma unroll
            for (int i = 0; i < WORDS; ++i) raw.w[k][i] = load16<false>(p + 16 * i);
        }
    }
    // returns whether a magnitude is outside of the split's range or NaN
    __device__ __forceinline__ static bool store(const Raw& raw, char* lds, int tid) {
        constexpr bool kLeast = VALUES && DT == F32;
        float m = 0.0f;
        uint32_t least = ~0u;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            char* dst = lds + plane_chunk((tid >> 3) + 32 * k, tid & 7);
            float f[8];
            if constexpr (DT == F32) {
                float lo[4], hi[4];
                Unpack<F32>::run(raw.w[k][0], lo);
                Unpack<F32>::run(raw.w[k][WORDS - 1], hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f[i] = lo[i];
                    f[4 + i] = hi[i];
                }
            } else {
                Unpack<DT>::run(raw.w[k][0], f);
            }
            m = max_abs8(f, m);
            if constexpr (kLeast) least = min_bits8(f, least);
            if constexpr (PIECES == 1) {
                *reinterpret_cast<u32x4*>(dst) = raw.w[k][0];
            } else {
                u32x4 p[PIECES];
                split8<PIECES>(f, p);
#pragma unroll
                for (int i = 0; i < PIECES; ++i) *reinterpret_cast<u32x4*>(dst + i * kPlaneBytes) = p[i];
            }
        }
        return !(m < (DT == F16 ? 65536.0f : kSplitLimit)) ||
               (kLeast && least < (__builtin_bit_cast(uint32_t, kSplitLeast) << 1) - 1u);
    }
    __device__ __forceinline__ static float at(const PrefillPipeArgs&, const char* base, uint32_t, uint32_t row,
                                               int dim) {
        return load_f32<DT>(base, (size_t)row * kD + dim);
    }
};

// The V tile of a tiered value cache: thread t widens elements 16 (t % 4)
// .. + 15 of row t / 4 (half of one 32-element block).  A row below the
// boundary is 16 INT8 codes times the block's f16 scale (exact in fp32), a
// row at or above it 16 f16 values from its window slot.
struct TieredSplitIo {
    static constexpr int EB = 1;  // bytes per element of `values` (the INT8 codes)
    static constexpr int PIECES = 3;
    struct Raw {
        u32x4 w[2];
    };
    __device__ __forceinline__ static uint32_t row_of(uint32_t tile, uint32_t kv_len, int tid) {
        return min(tile * kPrefillTile + (uint32_t)(tid >> 2), kv_len - 1);
    }
    __device__ __forceinline__ static void load(Raw& raw, const PrefillPipeArgs& a, uint32_t kvh, uint32_t tile,
                                                uint32_t kv_len, int tid) {
        const uint32_t row = row_of(tile, kv_len, tid);
        const int col = 16 * (tid & 3);
        if (row < a.tier) {
            const size_t e = (size_t)kvh * a.head_stride + (size_t)row * kD + col;
            raw.w[0] = load16<false>(reinterpret_cast<const int8_t*>(a.values) + e);
            raw.w[1] = u32x4{(uint32_t)a.value_scales[e / kTierBlockF32], 0u, 0u, 0u};
        } else {
            const uint16_t* w =
                a.value_ring + (size_t)kvh * a.ring_head_stride + (size_t)(row & a.window_mask) * kD + col;
            raw.w[0] = load16<false>(w);
            raw.w[1] = load16<false>(w + 8);
        }
    }
    __device__ __forceinline__ static bool store(const Raw& raw, char* lds, const PrefillPipeArgs& a, uint32_t tile,
                                                 uint32_t kv_len, int tid) {
        float f[2][8];
        if (row_of(tile, kv_len, tid) < a.tier) {
            const float sc = (float)__builtin_bit_cast(half_t, (uint16_t)raw.w[1][0]);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int32_t code = (int32_t)(raw.w[0][i >> 2] << (24 - 8 * (i & 3))) >> 24;
                f[i >> 3][i & 7] = (float)code * sc;
            }
        } else {
            Unpack<F16>::run(raw.w[0], f[0]);
            Unpack<F16>::run(raw.w[1], f[1]);
        }
        float m = 0.0f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            m = max_abs8(f[k], m);
            u32x4 p[3];
            split8<3>(f[k], p);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                *reinterpret_cast<u32x4*>(lds + i * kPlaneBytes + plane_chunk(tid >> 2, 2 * (tid & 3) + k)) = p[i];
        }
        return !(m < kSplitLimit);
    }
    __device__ __forceinline__ static float at(const PrefillPipeArgs& a, const char*, uint32_t kvh, uint32_t row,
                                               int dim) {
        if (row < a.tier) {
            const size_t e = (size_t)kvh * a.head_stride + (size_t)row * kD + dim;
            return (float)reinterpret_cast<const int8_t*>(a.values)[e] *
                   (float)__builtin_bit_cast(half_t, a.value_scales[e / kTierBlockF32]);
        }
        return (float)__builtin_bit_cast(
            half_t, a.value_ring[(size_t)kvh * a.ring_head_stride + (size_t)(row & a.window_mask) * kD + dim]);
    }
};

__device__ __forceinline__ f32x4 mma_bf(const u32x4& a, const u32x4& b, const f32x4& c) {
    return MfmaT<BF16>::mma(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c);
}

}  // namespace

// grid (qblocks x kv_heads, chunks of the longest block), block 256.
template <int KDT, int VDT>
__global__ __launch_bounds__(256, 2) void prefill_f32_kernel(PrefillPipeArgs a) {
    using KIo = SplitIo<KDT, false>;
    using VIo = std::conditional_t<VDT == I8T, TieredSplitIo, SplitIo<VDT == I8T ? F16 : VDT, true>>;
    constexpr int NK = KIo::PIECES, NV = VIo::PIECES;
    constexpr int kStageBytes = (NK + NV) * kPlaneBytes;
    // two stages where two workgroups of them still share a CU's 160 KB
    constexpr int STAGES = kStageBytes < 40 * 1024 ? 2 : 1;
    __shared__ __attribute__((aligned(16))) char lds[STAGES][kStageBytes];
    __shared__ __attribute__((aligned(16))) uint32_t wide[2][4];  // [tile parity][wave]: the tile exceeds the split

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lg = lane >> 4, li = lane & 15;

    // block -> (kv head, query block), longest rows first; each XCD serves
    // one kv head when the grid allows, so the head's K/V stays in its L2
    const uint32_t nqb = a.qblocks;
    uint32_t kvh, qidx;
    if (a.xcd_map) {
        const uint32_t lin = blockIdx.x, xcd = lin & 7, slot = lin >> 3;
        const uint32_t per = 8 / a.kv_heads;
        kvh = xcd / per;
        qidx = slot * per + (xcd % per);
    } else {
        kvh = blockIdx.x / nqb;
        qidx = blockIdx.x % nqb;
    }
    const uint32_t qblock = nqb - 1 - qidx;
    const uint32_t T = a.tokens;
    const uint32_t wg_t0 = qblock * kPrefillTile;
    const uint32_t kv_len = a.start + min(T, wg_t0 + kPrefillTile);
    const uint32_t n = (kv_len + kPrefillTile - 1) / kPrefillTile;
    const uint32_t ch_tiles = a.chunk_tiles ? a.chunk_tiles : n;
    const uint32_t nchunks = (n + ch_tiles - 1) / ch_tiles;
    const uint32_t chunk = blockIdx.y;
    if (chunk >= nchunks) return;  // uniform, before any barrier
    const uint32_t t0 = chunk * ch_tiles, t1 = min(n, t0 + ch_tiles);
    const uint32_t m = t1 - t0;

    // this wave's columns: tokens w_t0 + li of heads 2 kvh + nt
    const uint32_t w_t0 = wg_t0 + 16 * wave;
    const bool wave_live = w_t0 < T;
    const uint32_t w_last = min(T - 1, w_t0 + 15);
    const uint32_t wave_n = wave_live ? (a.start + w_last) / kPrefillTile + 1 : 0;
    const uint32_t wave_m = wave_n > t0 ? min(wave_n, t1) - t0 : 0;  // its tiles in the chunk
    const uint32_t tok = w_t0 + li;
    const uint32_t qpos = a.start + tok;  // position of column li's query
    const float c = a.scale_log2;

    const char* kbase = reinterpret_cast<const char*>(a.keys) + (size_t)kvh * a.head_stride * KIo::EB;
    const char* vbase = reinterpret_cast<const char*>(a.values) + (size_t)kvh * a.head_stride * VIo::EB;

    typename KIo::Raw kraw;
    typename VIo::Raw vraw;
    auto load_tile = [&](uint32_t tile) __attribute__((always_inline)) {
        KIo::load(kraw, kbase, tile, kv_len, tid);
        if constexpr (VDT == I8T) VIo::load(vraw, a, kvh, tile, kv_len, tid);
        else VIo::load(vraw, vbase, tile, kv_len, tid);
    };
    bool qwide = false;
    auto store_tile = [&](uint32_t tile, uint32_t r) __attribute__((always_inline)) {
        char* dst = lds[r % STAGES];
        bool w = KIo::store(kraw, dst, tid);
        if constexpr (VDT == I8T) w |= VIo::store(vraw, dst + NK * kPlaneBytes, a, tile, kv_len, tid);
        else w |= VIo::store(vraw, dst + NK * kPlaneBytes, tid);
        const uint32_t any = __any(w | qwide) ? 1u : 0u;
        if (lane == 0) wide[r & 1][wave] = any;
    };

    // The query goes out before the chunk's first tile: loads complete in
    // order, so its pieces are formed while the tile is in flight.
    // Q^T pieces: lane (g, i) holds dims 32h + 8g .. + 7 of column i
    u32x4 q[2][2][3];  // [head][h][piece]
    {
        const size_t qrow = ((size_t)min(tok, T - 1) * a.q_heads + (size_t)kvh * 2) * kD + 8 * lg;
        u32x4 raw[4][2];
        if (a.query_dtype == F32) {
            const float* p = reinterpret_cast<const float*>(a.query) + qrow;
#pragma unroll
            for (int x = 0; x < 8; ++x) raw[x >> 1][x & 1] = load16<false>(p + 32 * (x >> 1) + 4 * (x & 1));
        } else {
            const uint16_t* p = reinterpret_cast<const uint16_t*>(a.query) + qrow;
#pragma unroll
            for (int x = 0; x < 4; ++x) raw[x][0] = raw[x][1] = load16<false>(p + 32 * x);
        }
        load_tile(t0);
        __builtin_amdgcn_sched_barrier(0);
        float mq = 0.0f;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            float f[8];
            if (a.query_dtype == F32) {
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(raw[x][e >> 2][e & 3]);
            } else if (a.query_dtype == F16) {
                Unpack<F16>::run(raw[x][0], f);
            } else {
                Unpack<BF16>::run(raw[x][0], f);
            }
            mq = max_abs8(f, mq);
            split8<3>(f, q[x >> 1][x & 1]);
        }
        qwide = !(mq < kSplitLimit);
    }
    store_tile(t0, 0);
    __syncthreads();

    f32x4 oacc[4][2];  // [output block db][head nt]: lane (g, i) holds dims 16db + 4g + j of column i
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) oacc[db][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The running maximum is a score as the product left it: the exponent of
    // its own probability is then exactly zero at any magnitude (scaled first,
    // the rounding of a large score would be left in the exponent).
    float smrun[2] = {kNoScore, kNoScore}, lsum[2] = {0.f, 0.f};

    // operand addresses inside a stage: K rows 16 pb + i, chunk 4 h + g; V
    // rows 32 h + 4 g + i / 4 (+ 16), dims 16 db + 4 (i % 4)
    const int k_off = plane_chunk(li, lg);
    const int v_row = 4 * lg + (li >> 2);

    auto compute = [&](const char* st, uint32_t kt, bool split) __attribute__((always_inline)) {
        int l = lane;  // the lane number as the fp32 path sees it
        if (!split) asm volatile("" : "+v"(l));  // nothing of it is computed (and held in registers) outside it
        // S^T = K . Q^T, four 16-position blocks
        f32x4 sacc[4][2];
        if (split) {
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
                u32x4 k[2][NK];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < NK; ++i)
                        k[h][i] = *reinterpret_cast<const u32x4*>(st + i * kPlaneBytes + pb * 16 * kD * 2 +
                                                                  (k_off ^ (h * 64)));
#pragma unroll
                for (int sum = 2; sum >= 0; --sum)  // the small products first
#pragma unroll
                    for (int i = 0; i < NK; ++i)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
#pragma unroll
                            for (int nt = 0; nt < 2; ++nt)
                                if (i <= sum) acc[nt] = mma_bf(k[h][i], q[nt][h][sum - i], acc[nt]);
                sacc[pb][0] = acc[0];
                sacc[pb][1] = acc[1];
            }
        } else {
            // contraction slot s of lane group g is dim 16 g + s in both operands
            const size_t qr = ((size_t)min(w_t0 + (l & 15), T - 1) * a.q_heads + (size_t)kvh * 2) * kD + 16 * (l >> 4);
            float qf[2][16];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                if (a.query_dtype == F32) load_row16<F32>(a.query, qr + nt * kD, qf[nt]);
                else if (a.query_dtype == F16) load_row16<F16>(a.query, qr + nt * kD, qf[nt]);
                else load_row16<BF16>(a.query, qr + nt * kD, qf[nt]);
            }
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                const uint32_t row = min(kt * kPrefillTile + 16 * pb + (uint32_t)(l & 15), kv_len - 1);
                float k[16];
                load_row16<KDT>(kbase, (size_t)row * kD + 16 * (l >> 4), k);
                f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                for (int s = 0; s < 16; ++s)
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt) acc[nt] = mma4(k[s], qf[nt][s], acc[nt]);
                sacc[pb][0] = acc[0];
                sacc[pb][1] = acc[1];
                __builtin_amdgcn_sched_barrier(0);  // few registers before many loads in flight
            }
        }
        // causal mask, online softmax per column
        if ((kt + 1) * kPrefillTile > a.start + w_t0 + 1) {  // some position of the tile is past the first row's
#pragma unroll
            for (int pb = 0; pb < 4; ++pb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t pos = kt * kPrefillTile + 16 * pb + 4 * lg + j;
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt) sacc[pb][nt][j] = pos <= qpos ? sacc[pb][nt][j] : -INFINITY;
                }
        }
        float alpha[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            float smax = -INFINITY;
#pragma unroll
            for (int pb = 0; pb < 4; ++pb)
#pragma unroll
                for (int j = 0; j < 4; ++j) smax = fmaxf(smax, sacc[pb][nt][j]);
            smax = max_xor32(max_xor16(smax));
            const float mnew = fmaxf(smrun[nt], smax);
            alpha[nt] = fast_exp2((smrun[nt] - mnew) * c);
            smrun[nt] = mnew;
            float ps = 0.0f;
#pragma unroll
            for (int pb = 0; pb < 4; ++pb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float p = fast_exp2((sacc[pb][nt][j] - mnew) * c);
                    sacc[pb][nt][j] = p;
                    ps += p;
                }
            lsum[nt] = __builtin_fmaf(lsum[nt], alpha[nt], ps);
        }
        // O^T += V^T . P^T
        if (!split) {
            // A masked position has weight zero, and zero times an infinity is
            // NaN: past the positions that every column of the wave attends,
            // the matrix product takes finite values only, and the others go
            // one by one to the columns that attend them.
            const uint32_t common = a.start + w_t0 + 1;
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) oacc[db][nt] *= alpha[nt];
            uint32_t apart = 0;  // bit 4 pb + j: this lane's value at that position is one of them
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                const uint32_t pos = kt * kPrefillTile + 16 * pb + 4 * (uint32_t)(l >> 4);
                float v[4][4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int db = 0; db < 4; ++db)
                        v[j][db] = VIo::at(a, vbase, kvh, min(pos + j, kv_len - 1), 16 * db + (l & 15));
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int db = 0; db < 4; ++db) {
                        if (pos + j >= common && !finite(v[j][db])) {
                            v[j][db] = 0.0f;
                            apart |= 1u << (4 * pb + j);
                        }
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt) oacc[db][nt] = mma4(v[j][db], sacc[pb][nt][j], oacc[db][nt]);
                    }
                __builtin_amdgcn_sched_barrier(0);  // few registers before many loads in flight
            }
            const uint32_t end = min((kt + 1) * kPrefillTile, a.start + w_last + 1);
#pragma unroll 1
            for (uint32_t pos = max(common, kt * kPrefillTile); pos < end; ++pos) {
                const uint32_t bit = (pos >> 2 & 12) | (pos & 3);
                const int group = pos >> 2 & 3;  // of lanes that holds the position
                if (!__any((l >> 4) == group && (apart >> bit & 1))) continue;
                float p[2] = {0.0f, 0.0f};
#pragma unroll
                for (int b = 0; b < 16; ++b)
                    if (bit == (uint32_t)b) {
                        p[0] = sacc[b >> 2][0][b & 3];
                        p[1] = sacc[b >> 2][1][b & 3];
                    }
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) p[nt] = __shfl(p[nt], 16 * group + (l & 15));
                if (pos > qpos) continue;
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float v = VIo::at(a, vbase, kvh, pos, 16 * db + 4 * (l >> 4) + j);
                        if (finite(v)) continue;
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt)
                            oacc[db][nt][j] = __builtin_fmaf(p[nt], v, oacc[db][nt][j]);
                    }
            }
            return;
        }
        const char* vt = st + NK * kPlaneBytes;
        auto v_operand = [&](int h, int piece, int db) __attribute__((always_inline)) {
            // rows r and r + 16 share row & 7, so one chunk address serves both
            const char* p = vt + piece * kPlaneBytes + h * 32 * kD * 2 + plane_chunk(v_row, 2 * db + ((li & 3) >> 1)) +
                            8 * (li & 1);
            const i16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p));
            const i16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p + 16 * kD * 2));
            return __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        // the tile's products are summed by themselves and added to O once: the
        // running sums of a long chain are rounded once a tile
        u32x4 p[2][2][3];  // [h][head][piece]
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                float f[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = sacc[2 * h + (e >> 2)][nt][e & 3];
                split8<3>(f, p[h][nt]);
            }
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            u32x4 v[2][NV];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < NV; ++i) v[h][i] = __builtin_bit_cast(u32x4, v_operand(h, i, db));
#pragma unroll
            for (int sum = 2; sum >= 0; --sum)
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt)
                            if (i <= sum) acc[nt] = mma_bf(v[h][i], p[h][nt][sum - i], acc[nt]);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    oacc[db][nt][j] = __builtin_fmaf(oacc[db][nt][j], alpha[nt], acc[nt][j]);
        }
    };

    for (uint32_t r = 0; r < m; ++r) {
        const bool more = r + 1 < m;
        if (more) load_tile(t0 + r + 1);  // in flight during this tile's math
        if (r < wave_m) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(wide[r & 1]);
            const bool split = __builtin_amdgcn_readfirstlane(w[0] | w[1] | w[2] | w[3]) == 0;
            compute(lds[r % STAGES], t0 + r, split);
        }
        if constexpr (STAGES == 1) __syncthreads();
        // two stages: the other one was last read in round r - 1, before its barrier
        if (more) store_tile(t0 + r + 1, r + 1);
        __syncthreads();
    }

    if (!wave_live) return;
    // the four 16-lane groups hold disjoint positions of each column
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) lsum[nt] = sum_xor32(sum_xor16(lsum[nt]));
    if (nchunks > 1) {
        const size_t slot = (((size_t)kvh * nqb + qblock) * a.max_chunks + chunk) * 128;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const size_t colx = slot + wave * 32 + nt * 16 + li;
            if (lg == 0) {
                a.part_ml[2 * colx] = smrun[nt] * c;
                a.part_ml[2 * colx + 1] = lsum[nt];
            }
#pragma unroll
            for (int db = 0; db < 4; ++db)
                *reinterpret_cast<f32x4*>(a.part_o + colx * kD + 16 * db + 4 * lg) = oacc[db][nt];
        }
        return;
    }
    if (tok >= T) return;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const float inv = 1.0f / lsum[nt];
        const size_t obase = ((size_t)tok * a.q_heads + (size_t)kvh * 2 + nt) * kD + 4 * lg;
#pragma unroll
        for (int db = 0; db < 4; ++db) store4_any(a.out, obase + 16 * db, oacc[db][nt] * inv, a.out_dtype);
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Split KV.  The longest block's chain of tiles sets the time until the chip is
// full, and each chunk costs a workgroup's start and a merge, so a block's KV
// range is cut
// - into enough chunks for kF32TargetWgs workgroups (two per CU), each at
//   least kF32MinTiles tiles, or one where a block has kF32FewTiles at most, and
// - into chunks of about kF32ChunkTiles tiles while that makes at most
//   kF32MostWgs workgroups: with more blocks than CUs the longest block's
//   chain would set the time.
// Measured, Fp32KFp16V, us per layer of 8 (merge included), start + T: at least
// 8 tiles a chunk / this rule 0 + 256 20.3 / 14.5, 0 + 700 43.8 / 25.4, 900 +
// 100 35.9 / 19.6, 2000 + 500 58.3 / 45.8; two tiles at least throughout / this
// rule 63 + 66 15.8 / 13.2, 100 + 64 17.1 / 13.3, 0 + 192 16.8 / 13.9; toward
// 512 workgroups only / this rule 64 + 2999 138.0 / 126.7; toward 2048 with 2
// tiles / this rule 2000 + 500 53.7 / 45.8, 1000 + 1000 65.3 / 58.1, 0 + 1900
// 67.1 / 69.9.
constexpr uint32_t kF32TargetWgs = 512;
constexpr uint32_t kF32MinTiles = 2;
constexpr uint32_t kF32FewTiles = 4;
constexpr uint32_t kF32ChunkTiles = 8;
constexpr uint32_t kF32MostWgs = 2048;
constexpr uint32_t kF32MaxChunks = 32;
constexpr uint32_t kF32Columns = 128;

bool prefill_f32_supported(const ShapeDims& s, int key_dtype, int value_dtype) {
    if (s.head_dim != kD || s.group != 2) return false;
    // tiered values with fp32 keys: the reference's proposed plan (16-bit
    // keys with tiered values take the pipelined kernel)
    if (value_dtype == I8T) return key_dtype == F32;
    return key_dtype == F32 || value_dtype == F32;
}

static uint32_t f32_blocks(const ShapeDims& s, uint32_t tokens) {
    return (tokens + kPrefillTile - 1) / kPrefillTile * s.kv_heads;
}

// chunks of a block of `tiles` tiles
static uint32_t f32_chunks(const ShapeDims& s, uint32_t tokens, uint32_t tiles) {
    const uint32_t wgs = f32_blocks(s, tokens);
    const uint32_t fill = std::min((kF32TargetWgs + wgs - 1) / wgs, tiles <= kF32FewTiles ? tiles : tiles / kF32MinTiles);
    const uint32_t cut = std::min(kF32MostWgs / wgs, tiles / kF32ChunkTiles);
    return std::max(1u, std::min(kF32MaxChunks, std::max(fill, cut)));
}

// Partial slots of a block in a cache of `capacity` positions: chunks for
// kF32MostWgs workgroups, of a tile at least, which is no less than f32_chunks
// takes at any start.  Over short caches it makes the size grow with the prompt,
// so that a workspace asked for a program's longest prompt serves the others.
static uint32_t f32_max_chunks(const ShapeDims& s, uint32_t tokens, uint32_t capacity) {
    const uint32_t wgs = f32_blocks(s, tokens), tiles = (capacity + kPrefillTile - 1) / kPrefillTile;
    return std::max(1u, std::min({kF32MaxChunks, (kF32MostWgs + wgs - 1) / wgs, tiles}));
}

static uint32_t f32_chunk_tiles(const ShapeDims& s, uint32_t start, uint32_t tokens) {
    const uint32_t n_max = (start + tokens + kPrefillTile - 1) / kPrefillTile;
    const uint32_t chunks = f32_chunks(s, tokens, n_max);
    return chunks <= 1 ? 0 : (n_max + chunks - 1) / chunks;
}

uint64_t prefill_f32_workspace_bytes(const ShapeDims& s, uint32_t capacity, uint32_t tokens) {
    const uint32_t mc = f32_max_chunks(s, tokens, capacity);
    if (mc <= 1) return 0;
    const uint64_t slots = (uint64_t)f32_blocks(s, tokens) * mc * kF32Columns;
    return slots * (2 + kD) * sizeof(float);
}

hipError_t launch_prefill_f32(const ShapeDims& s, const KvLayer& kv, uint32_t start, uint32_t tokens, const void* query,
                              int query_dtype, void* out, int out_dtype, void* workspace, hipStream_t st,
                              int* dispatches) {
    *dispatches = 0;
    if (!prefill_f32_supported(s, kv.key_dtype, kv.value_dtype)) return hipErrorNotSupported;
    PrefillPipeArgs a{};
    a.query = query;
    a.query_dtype = query_dtype;
    a.keys = kv.keys;
    a.values = kv.values;
    a.value_scales = reinterpret_cast<const uint16_t*>(kv.value_scales);
    a.value_ring = reinterpret_cast<const uint16_t*>(kv.value_ring);
    a.ring_head_stride = kv.ring_head_stride;
    a.window_mask = kv.window ? kv.window - 1 : 0;
    a.tier = kv.tier;
    a.out = out;
    a.head_stride = kv.head_stride;
    a.start = start;
    a.tokens = tokens;
    a.q_heads = s.q_heads;
    a.group = s.group;
    a.out_dtype = out_dtype;
    a.scale_log2 = s.scale * kLog2e;
    a.kv_heads = s.kv_heads;
    a.qblocks = (tokens + kPrefillTile - 1) / kPrefillTile;
    a.xcd_map = (8 % s.kv_heads == 0) && ((uint64_t)a.qblocks * s.kv_heads) % 8 == 0;
    a.chunk_tiles = f32_chunk_tiles(s, start, tokens);
    a.max_chunks = f32_max_chunks(s, tokens, kv.capacity);
    const uint64_t slots = (uint64_t)a.qblocks * s.kv_heads * a.max_chunks * kF32Columns;
    a.part_ml = reinterpret_cast<float*>(workspace);
    a.part_o = a.part_ml + 2 * slots;
    const uint32_t tiles = (start + tokens + kPrefillTile - 1) / kPrefillTile;
    const uint32_t chunks = a.chunk_tiles ? (tiles + a.chunk_tiles - 1) / a.chunk_tiles : 1;
    const dim3 grid(a.qblocks * s.kv_heads, chunks);
    const int kd = kv.key_dtype, vd = kv.value_dtype;
    if (kd == F32 && vd == F32) hipLaunchKernelGGL((prefill_f32_kernel<F32, F32>), grid, dim3(256), 0, st, a);
    else if (kd == F32 && vd == F16) hipLaunchKernelGGL((prefill_f32_kernel<F32, F16>), grid, dim3(256), 0, st, a);
    else if (kd == F32 && vd == BF16) hipLaunchKernelGGL((prefill_f32_kernel<F32, BF16>), grid, dim3(256), 0, st, a);
    else if (kd == F32 && vd == I8T) hipLaunchKernelGGL((prefill_f32_kernel<F32, I8T>), grid, dim3(256), 0, st, a);
    else if (kd == F16 && vd == F32) hipLaunchKernelGGL((prefill_f32_kernel<F16, F32>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((prefill_f32_kernel<BF16, F32>), grid, dim3(256), 0, st, a);
    *dispatches = 1;
    if (chunks > 1) {
        hipLaunchKernelGGL((prefill_combine_kernel<64, 2, 4>), dim3(a.qblocks * s.kv_heads, kF32Columns / 16),
                           dim3(256), 0, st, a);
        *dispatches = 2;
    }
    return hipGetLastError();
}

}  // namespace qxh
