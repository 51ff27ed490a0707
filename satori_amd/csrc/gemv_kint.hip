// Q8_K activation quantizer and the integer K-format products (Q4_K x Q8_K, Q6_K x Q8_K) for gfx950.
//
// Both reproduce the reference bit for bit:
//  - the quantizer is Q8KCodec.QuantizeBlock (src/Satori.Core/Q8KCodec.cs:44-76): first-largest |x| with
//    a strict comparison, -127/max and 1/inverse as correctly rounded divisions, the product and the
//    12582912 add rounded separately (the library is compiled with -ffp-contract=off and the operations
//    are spelled with explicit round-to-nearest intrinsics);
//  - the products are exact int32 sums (v_dot4_i32_i8), and the per-block FP32 expression and the
//    block-order accumulation of each row are those of QuantizedKAvx2Kernel.ExecuteQuantizedTiled
//    (src/Satori.Core/QuantizedKAvx2Kernel.cs:47-99), so each output equals the reference's float.
#include <type_traits>

#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"
#include "ops_device.hpp"
#include "q8k_device.hpp"

namespace satori {
namespace {

// ------------------------------------------------------------------------------------------------
// Q8_K quantizer (one wave per block; the per-block arithmetic is in q8k_device.hpp).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void q8k_quantize_kernel(const float* __restrict__ x, int columns,
                                                          uint8_t* __restrict__ out) {
    const int block = blockIdx.x;
    const int position = blockIdx.y;
    const int blocks = columns / 256;
    const int lane = threadIdx.x;
    const float* src = x + static_cast<int64_t>(position) * columns + block * 256;
    uint8_t* dst = out + (static_cast<int64_t>(position) * blocks + block) * kQ8KBlockBytes;
    float v[4];
    q8k_load_values(src, lane, v);
    const Q8KLane q = q8k_quantize_values(v, lane);
    if (q.zero) {
        uint32_t* d32 = reinterpret_cast<uint32_t*>(dst);
        for (int i = lane; i < kQ8KBlockBytes / 4; i += 64) d32[i] = 0u;
        return;
    }
    reinterpret_cast<uint32_t*>(dst + 4)[lane] = q.packed;
    if ((lane & 3) == 0) reinterpret_cast<int16_t*>(dst + 260)[lane >> 2] = static_cast<int16_t>(q.group_sum);
    if (lane == 0) reinterpret_cast<float*>(dst)[0] = q.scale;
}

// ------------------------------------------------------------------------------------------------
// Integer product. A workgroup owns s.rows_per_wg rows (4 to 64) of one member at one position. It quantizes the
// position's FP32 activation row to Q8_K itself (one wave per block, bit-exact as above; every workgroup
// computes the same bytes) straight into LDS as separate arrays (codes, group sums, scales), so no separate
// quantization launch precedes the product and code reads are 16-byte aligned.
// Work items are (row, block) pairs, 4 lanes of 64 weights each; the G lanes' int32 partials are summed
// exactly, the pair's leader forms the block's FP32 term and stores it in LDS, and finally one thread per row
// adds its terms in block order. A row wider than the LDS holds (more than kint_max_blocks() blocks) is
// staged and summed in chunks of blocks, in block order, so the sum is the same sequential one.
// ------------------------------------------------------------------------------------------------
constexpr int kThreads = 256;
constexpr int kTileRows = 64;
// The staged Q8_K codes of block b start at dword kCodeStride * b: 64 code dwords plus 4 of padding, so the
// 16 (row, block) pairs of a wave, which read 16 consecutive blocks at the same offset, hit 16 different
// groups of LDS banks instead of the same four.
constexpr int kCodeStride = 68;
constexpr int kActDwords = kCodeStride + 1 + 8;  // codes, scale, group sums per block
// Activation loads a thread issues before the weight loads: passes of 16 Q8_K blocks (48 blocks preloaded)
// and elements of the RmsNorm sum of squares (2,048 columns).
constexpr int kQ8KPasses = 3;  // 48 blocks
constexpr int kNormPreload = 8;
// An RmsNorm input row of at most this many columns keeps its summed values (residual + addend) in LDS
// between the sum of squares and the quantization, instead of reading both operands again.
constexpr int kNormStageColumns = 8192;


__device__ __forceinline__ int sdot4(uint32_t a, uint32_t b, int c) {
    return __builtin_amdgcn_sdot4(static_cast<int>(a), static_cast<int>(b), c, false);
}

// Two int16 products and a sum, exact.
__device__ __forceinline__ int sdot2(uint32_t a, uint32_t b, int c) {
    typedef short s16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(s16x2, a), __builtin_bit_cast(s16x2, b), c, false);
}

struct ActTile {
    uint32_t* codes;   // [blocks][64] dwords
    int16_t* sums;     // [blocks][16]
    float* scales;     // [blocks]
};

// Q4_K pair, lane c of 4 = group g: qs[32g, 32g + 32), low nibbles are weights 64g + i of sub-block 2g,
// high nibbles weights 64g + 32 + i of sub-block 2g + 1 (Q4KCodec.DotProduct / MinProduct, Q4KCodec.cs:117-153).
struct Q4KRaw {
    u32x4 head;  // d, dmin, scales[12]
    u32x4 qs0, qs1;
};

__device__ __forceinline__ void q4k_load(const uint8_t* block, int c, Q4KRaw& r) {
    r.head = load16_a4(block);
    r.qs0 = load16_a4(block + 16 + 32 * c);
    r.qs1 = load16_a4(block + 32 + 32 * c);
}

__device__ __forceinline__ void q4k_dot(const Q4KRaw& r, const ActTile& act, int b, int g, int& dot, int& min_part) {
    int s0, m0, s1, m1;
    q4k_scale_min(2 * g, r.head, s0, m0);
    q4k_scale_min(2 * g + 1, r.head, s1, m1);
    const uint32_t* codes = act.codes + kCodeStride * b + 16 * g;
    const u32x4 lo0 = *reinterpret_cast<const u32x4*>(codes), lo1 = *reinterpret_cast<const u32x4*>(codes + 4);
    const u32x4 hi0 = *reinterpret_cast<const u32x4*>(codes + 8), hi1 = *reinterpret_cast<const u32x4*>(codes + 12);
    int lo = 0, hi = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        lo = sdot4(r.qs0[w] & 0x0F0F0F0Fu, lo0[w], lo);
        lo = sdot4(r.qs1[w] & 0x0F0F0F0Fu, lo1[w], lo);
        hi = sdot4((r.qs0[w] >> 4) & 0x0F0F0F0Fu, hi0[w], hi);
        hi = sdot4((r.qs1[w] >> 4) & 0x0F0F0F0Fu, hi1[w], hi);
    }
    dot = s0 * lo + s1 * hi;
    const int16_t* sums = act.sums + 16 * b;
    min_part = m0 * (sums[4 * g] + sums[4 * g + 1]) + m1 * (sums[4 * g + 2] + sums[4 * g + 3]);
}

// Q6_K pair, lane c of 4: half h = c / 2, slice t = c % 2, i.e. weights 128h + 32k + 16t + i
// (Q6KCodec.DotProduct, Q6KCodec.cs:114-146, with the -32 centring applied through the group sums:
// sum sc * (q - 32) * code = sum sc * q * code - 32 * sum sc * bsum, both exact), read from the regrouped
// device layout (Q6KLayout).
using Q6KRaw = Q6KQuarter;

__device__ __forceinline__ int q6k_dot(const Q6KRaw& r, const ActTile& act, int b, int c) {
    const int h = c >> 1, t = c & 1;
    int dotk[4] = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t a = r.qla[w], bq = r.qlb[w], hb = r.qh[w];
        const uint32_t q[4] = {
            (a & 0x0F0F0F0Fu) | ((hb << 4) & 0x30303030u),
            (bq & 0x0F0F0F0Fu) | ((hb << 2) & 0x30303030u),
            ((a >> 4) & 0x0F0F0F0Fu) | (hb & 0x30303030u),
            ((bq >> 4) & 0x0F0F0F0Fu) | ((hb >> 2) & 0x30303030u),
        };
#pragma unroll
        for (int k = 0; k < 4; ++k)
            dotk[k] = sdot4(q[k], act.codes[kCodeStride * b + 32 * h + 8 * k + 4 * t + w], dotk[k]);
    }
    const int16_t* sums = act.sums + 16 * b;
    int total = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int sc = static_cast<int8_t>(r.sc >> (8 * k));  // scale 8h + 2k + t
        total += sc * (dotk[k] - 32 * sums[8 * h + 2 * k + t]);
    }
    return total;
}

// LDS: staged activations, the row terms, then (input transforms) 256 doubles for the RmsNorm reduction at an
// 8-byte aligned dword offset. Sized for the largest tile so one bound serves every launch.
__host__ __device__ inline int kint_red_offset(int blocks, int tile_rows) {
    return ((kActDwords + tile_rows) * blocks + 1) & ~1;
}

static_assert(kThreads == kOpsThreads, "the RmsNorm reduction is the operators' 256-thread tree");

// The members of a launch of up to kKintInlineMembers matrices travel in the kernel arguments, so the first
// weight loads depend on no global-memory read; larger groups read a device array of descriptors.
struct KintMembers {
    MatDesc m[kKintInlineMembers];
};

// PAIRED: a two-member launch (gate, up) whose workgroups own the same s.rows_per_wg rows of both members
// (2 * rows_per_wg <= 64 row sums, all in the first wave), carrying SwiGlu and its Q8_K bytes on (see
// OutputSwiGluQ8K).
template <int FORMAT, int XF, bool INLINE, bool PAIRED>
__global__ __launch_bounds__(kThreads) void gemv_kint_kernel(KintMembers inline_members,
                                                              const MatDesc* __restrict__ group, LaunchShape s,
                                                              InputTransform xf, OutputSwiGluQ8K out) {
    static_assert(!PAIRED || INLINE, "paired launches pass their two members in the kernel arguments");
    constexpr int G = 4;  // lanes per (row, block) pair
    constexpr int kBlockBytes = FORMAT == kQ4_K ? 144 : 210;
    constexpr int kPairsPerStep = kThreads / G;
    using Raw = typename std::conditional<FORMAT == kQ4_K, Q4KRaw, Q6KRaw>::type;
    // Inline members come from the kernel arguments through the scalar cache; a larger group's descriptor is
    // one global load.
    const MatDesc m = INLINE ? inline_members.m[PAIRED ? 0 : blockIdx.y] : group[blockIdx.y];
    const int tile_rows = s.rows_per_wg;
    const int row_begin = blockIdx.x * tile_rows;
    if (row_begin >= m.rows) return;
    const int rows = min(tile_rows, m.rows - row_begin);
    // Rows of the workgroup's terms: its rows of m, then (paired) the same rows of the second member.
    const int vrows = PAIRED ? 2 * rows : rows;
    const int vtile = PAIRED ? 2 * tile_rows : tile_rows;
    const int position = blockIdx.z;
    const int nb = s.blocks;
    // Blocks staged at a time: the whole row when it fits the LDS, else chunks of K blocks walked in block
    // order (each chunk's terms are added to the row sums before the next chunk is staged).
    const int K = s.chunk_blocks;

    extern __shared__ uint32_t smem[];
    ActTile act;
    act.codes = smem;                                                          // kCodeStride * K dwords
    act.scales = reinterpret_cast<float*>(smem + kCodeStride * K);             // K
    act.sums = reinterpret_cast<int16_t*>(smem + (kCodeStride + 1) * K);       // 16 * K int16 = 8 * K dwords
    float* terms = reinterpret_cast<float*>(smem + kActDwords * K);            // tile_rows * K

    // Work items are (row, block) pairs of the chunk in row-major order; the G lanes of a pair share its
    // index, so the DPP group sums stay inside the pair. The next pair's payload is loaded before the
    // current one is reduced.
    const int lane = threadIdx.x & 63;
    const int c = lane % G;
    const uint8_t* w1 = PAIRED ? inline_members.m[1].w : m.w;  // the second member's payload (paired)
    // Pair p of the chunk starting at block b0 with kb blocks: row p / kb of the tile (paired: rows past
    // `rows` are the second member's), block b0 + p % kb.
    auto load_pair = [&](int b0, int kb, int p, Raw& r) {
        int row = p / kb;
        const int b = b0 + p % kb;
        const uint8_t* w = m.w;
        if (PAIRED && row >= rows) {
            row -= rows;
            w = w1;
        }
        if constexpr (FORMAT == kQ4_K) {
            q4k_load(w + static_cast<int64_t>(row_begin + row) * s.row_bytes + b * kBlockBytes, c, r);
        } else {
            // Q6_K: block b of tile row `row` is block (row_begin + row) * nb + b of the matrix.
            q6k_load_quarter(w, static_cast<int64_t>(m.rows) * nb, static_cast<int64_t>(row_begin + row) * nb + b,
                             c, r);
        }
    };
    // This slot's pairs are p0, p0 + kPairsPerStep, ...; kDepth of them are loaded before the activations
    // are staged, and each processed pair's registers are refilled with the pair kDepth further on, so kDepth
    // loads stay in flight.
    constexpr int kDepth = 3;
    const int p0 = threadIdx.x / G;
    int kb = min(K, nb);
    int mine = p0 < vrows * kb ? (vrows * kb - 1 - p0) / kPairsPerStep + 1 : 0;
    const float* xrow = m.x + static_cast<int64_t>(position) * s.columns;
    auto quad = [](const float* p, int i) {
        const u32x4 raw = load16_a4(reinterpret_cast<const uint8_t*>(p + i));
        return f32x4{__uint_as_float(raw[0]), __uint_as_float(raw[1]), __uint_as_float(raw[2]),
                     __uint_as_float(raw[3])};
    };

    // The activation side is loaded first, then the weights: the waits for the activations then do not
    // cover the weight loads issued after them. Every thread issues the same loads (addresses past the end
    // are clamped and their values unused), so the load counts the waits are computed from are static.
    // Launches of up to kKintInlineMembers members (the decode step's latency-bound groups) do this; larger
    // groups stream from HBM and keep the registers for occupancy (the preloads take the plain-input Q4_K
    // kernel from 127 to 138 VGPRs, three waves per SIMD instead of four: 8960 x 1536 grouped measured
    // 5.53 against 5.86 TB/s).
    constexpr bool kPreload = INLINE;
    const int tid = threadIdx.x;
    const int j16 = tid & 15, bl0 = tid >> 4;
    f32x4 xpre[4];                 // plain input: this thread's 16 values of the first pass
    // Q8_K input: lane j16 of a 16-lane row copies block bl's code dwords [4 j16, 4 j16 + 4), and lane 0 its
    // scale, lanes 1 and 2 its group sums; the first kQ8KPasses passes are loaded here.
    u32x4 qcodes[kQ8KPasses], qaux[kQ8KPasses];
    auto q8k_load = [&](const uint8_t* row, int bl, u32x4& codes, u32x4& aux) {
        const uint8_t* block = row + static_cast<int64_t>(bl) * kQ8KBlockBytes;
        codes = load16_a4(block + 4 + 16 * j16);
        aux = load16_a4(block + (j16 == 0 ? 0 : 260 + 16 * (min(j16, 2) - 1)));
    };
    float npre_a[kNormPreload], npre_b[kNormPreload];  // RmsNorm input: the first terms of the sum of squares
    f32x4 wpre[4];                                      // RmsNorm input: the norm weights of the first pass
    if constexpr (XF == kInputPlain && kPreload) {
        const int i0 = 256 * min(bl0, kb - 1) + 16 * j16;
#pragma unroll
        for (int q = 0; q < 4; ++q) xpre[q] = quad(xrow, i0 + 4 * q);
    } else if constexpr (XF == kInputQ8K && kPreload) {
#pragma unroll
        for (int k = 0; k < kQ8KPasses; ++k)
            q8k_load(reinterpret_cast<const uint8_t*>(xf.a), min(bl0 + 16 * k, kb - 1), qcodes[k], qaux[k]);
    } else if constexpr (XF == kInputAddRmsNorm) {
#pragma unroll
        for (int k = 0; k < kNormPreload; ++k) {
            const int i = min(tid + kThreads * k, s.columns - 1);
            npre_a[k] = xf.a[i];
            npre_b[k] = xf.b ? xf.b[i] : 0.0f;
        }
        const int i0 = 256 * min(bl0, kb - 1) + 16 * j16;
#pragma unroll
        for (int q = 0; q < 4; ++q) wpre[q] = quad(xf.w, i0 + 4 * q);
    }
    Raw buf[kDepth];
#pragma unroll
    for (int i = 0; i < kDepth; ++i) load_pair(0, kb, min(p0 + i * kPairsPerStep, vrows * kb - 1), buf[i]);

    // Q8_K of the position's activations: one 16-lane row per block, sixteen blocks per pass. With an input
    // transform the activations are computed here from the operator's operands, in the operator's own
    // arithmetic (the RmsNorm sum of squares over the same 256-thread partition and tree, over the whole row).
    double scale = 0.0;
    // Summed RmsNorm input (residual + addend) kept in LDS after the reduction's 256 doubles.
    float* rstage = reinterpret_cast<float*>(smem + kint_red_offset(K, vtile) + 2 * kThreads);
    const bool rstaged = XF == kInputAddRmsNorm && s.columns <= kNormStageColumns;
    if constexpr (XF == kInputAddRmsNorm) {
        double* red = reinterpret_cast<double*>(smem + kint_red_offset(K, vtile));
        const bool writer = xf.residual_out && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0;
        double part = 0;
        auto term = [&](int i, float a, float b) {
            const float r = xf.b ? __fadd_rn(a, b) : a;
            if (writer) xf.residual_out[i] = r;
            if (rstaged) rstage[i] = r;  // visible to every thread after the reduction's barriers
            const double v = r;
            part = part + v * v;
        };
#pragma unroll
        for (int k = 0; k < kNormPreload; ++k)
            if (tid + kThreads * k < s.columns) term(tid + kThreads * k, npre_a[k], npre_b[k]);
        for (int i = tid + kThreads * kNormPreload; i < s.columns; i += kThreads)
            term(i, xf.a[i], xf.b ? xf.b[i] : 0.0f);
        scale = rms_scale(block_sum_256(part, red), s.columns, xf.epsilon);
    }
    // Block order from +0, as the reference accumulator (QuantizedKAvx2Kernel.cs:63, 90-94). A skipped
    // block stores +0, and adding +0 to a sum that starts at +0 never changes it.
    float acc = 0.0f;
    for (int b0 = 0;;) {
        if constexpr (XF == kInputQ8K) {
            // The producer's Q8_K row (Q8KCodec layout, 292 bytes per block: scale, 256 codes, 16 int16 group
            // sums) copied into the LDS arrays, one 16-lane row per block.
            const uint8_t* row = reinterpret_cast<const uint8_t*>(xf.a) + static_cast<int64_t>(b0) * kQ8KBlockBytes;
            auto put = [&](int bl, const u32x4& codes, const u32x4& aux) {
                *reinterpret_cast<u32x4*>(act.codes + kCodeStride * bl + 4 * j16) = codes;
                if (j16 == 0) {
                    act.scales[bl] = __uint_as_float(aux[0]);
                } else if (j16 <= 2) {
                    uint32_t* sums = reinterpret_cast<uint32_t*>(act.sums) + 8 * bl + 4 * (j16 - 1);
#pragma unroll
                    for (int e = 0; e < 4; ++e) sums[e] = aux[e];
                }
            };
            int bl = bl0;
            if (kPreload && b0 == 0) {
#pragma unroll
                for (int k = 0; k < kQ8KPasses; ++k)
                    if (bl0 + 16 * k < kb) put(bl0 + 16 * k, qcodes[k], qaux[k]);
                bl += 16 * kQ8KPasses;
            }
            for (; bl < kb; bl += kThreads / 16) {
                u32x4 codes, aux;
                q8k_load(row, bl, codes, aux);
                put(bl, codes, aux);
            }
        } else {
            auto stage = [&](int bl, const f32x4 (&x4)[4]) {
                float v[16];
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[4 * q + e] = x4[q][e];
                const Q8KRow16 qr = q8k_quantize_row16(v, lane);
                *reinterpret_cast<u32x4*>(act.codes + kCodeStride * bl + 4 * j16) =
                    u32x4{qr.packed[0], qr.packed[1], qr.packed[2], qr.packed[3]};
                act.sums[16 * bl + j16] = static_cast<int16_t>(qr.group_sum);
                if (j16 == 0) act.scales[bl] = qr.scale;
            };
            int bl = bl0;
            if constexpr (XF == kInputPlain && kPreload) {
                if (b0 == 0) {
                    if (bl < kb) stage(bl, xpre);
                    bl += kThreads / 16;
                }
            }
            for (; bl < kb; bl += kThreads / 16) {
                const int i0 = 256 * (b0 + bl) + 16 * j16;
                f32x4 x4[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (XF == kInputPlain) {
                        x4[q] = quad(xrow, i0 + 4 * q);
                    } else if constexpr (XF == kInputAddRmsNorm) {
                        const bool first = b0 == 0 && bl == bl0;  // the pass whose weights were preloaded
                        const f32x4 w4 = first ? wpre[q] : quad(xf.w, i0 + 4 * q);
                        f32x4 r4;
                        if (rstaged) {
                            r4 = *reinterpret_cast<const f32x4*>(rstage + i0 + 4 * q);
                        } else {
                            const f32x4 a4 = quad(xf.a, i0 + 4 * q);
                            f32x4 b4 = {0.0f, 0.0f, 0.0f, 0.0f};
                            if (xf.b) b4 = quad(xf.b, i0 + 4 * q);
#pragma unroll
                            for (int e = 0; e < 4; ++e) r4[e] = xf.b ? __fadd_rn(a4[e], b4[e]) : a4[e];
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) x4[q][e] = rms_value(r4[e], scale, w4[e]);
                    } else {
                        const f32x4 g4 = quad(xf.a, i0 + 4 * q), u4 = quad(xf.b, i0 + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) x4[q][e] = swiglu_value(g4[e], u4[e]);
                    }
                }
                stage(bl, x4);
            }
        }
        __syncthreads();  // activations of the chunk staged
        // The FP32 term of pair p (valid on the pair's last lane).
        auto term_of = [&](const Raw& cur, int p) {
            const int bl = p % kb;  // block of the chunk (its staged activations)
            float term = 0.0f;
            if constexpr (FORMAT == kQ4_K) {
                int dot, min_part;
                q4k_dot(cur, act, bl, c, dot, min_part);
                dot = group_sum_last_int<G>(dot);
                min_part = group_sum_last_int<G>(min_part);
                const float a = act.scales[bl];
                if (a != 0.0f) {  // zero activation block: skipped (QuantizedKAvx2Kernel.cs:86)
                    const float dA = __fmul_rn(half_bits_to_float(cur.head[0] & 0xFFFFu), a);
                    const float dminA = __fmul_rn(half_bits_to_float(cur.head[0] >> 16), a);
                    term = __fsub_rn(__fmul_rn(dA, static_cast<float>(dot)),
                                     __fmul_rn(dminA, static_cast<float>(min_part)));
                }
            } else {
                int dot = q6k_dot(cur, act, bl, c);
                dot = group_sum_last_int<G>(dot);
                const float a = act.scales[bl];
                if (a != 0.0f) term = __fmul_rn(__fmul_rn(a, q6k_d(cur)), static_cast<float>(dot));
            }
            return term;
        };
        // The slot's pairs in order; each processed pair's registers are refilled with the pair kDepth further
        // on. (Computing a round's kDepth pairs unconditionally, to interleave their chains, measured slower on
        // the decode step's small launches: the slots there hold fewer than kDepth pairs.)
        for (int base = 0; base < mine; base += kDepth) {
#pragma unroll
            for (int i = 0; i < kDepth; ++i) {
                const int k = base + i;
                if (k < mine) {
                    const float t = term_of(buf[i], p0 + k * kPairsPerStep);
                    if (c == G - 1) terms[p0 + k * kPairsPerStep] = t;
                    if (k + kDepth < mine) load_pair(b0, kb, p0 + (k + kDepth) * kPairsPerStep, buf[i]);
                }
            }
        }
        __syncthreads();  // the chunk's terms are in LDS
        if (threadIdx.x < vrows) {
            const float* t = terms + threadIdx.x * kb;
            for (int b = 0; b < kb; ++b) acc = __fadd_rn(acc, t[b]);
        }
        b0 += K;
        if (b0 >= nb) break;
        // Next chunk: its first pairs' payload is requested before the LDS is released.
        kb = min(K, nb - b0);
        mine = p0 < vrows * kb ? (vrows * kb - 1 - p0) / kPairsPerStep + 1 : 0;
#pragma unroll
        for (int i = 0; i < kDepth; ++i) load_pair(b0, kb, min(p0 + i * kPairsPerStep, vrows * kb - 1), buf[i]);
        __syncthreads();  // every thread is done with this chunk's activations and terms
    }
    if constexpr (!PAIRED) {
        if (threadIdx.x < rows) store_f32(m.y + static_cast<int64_t>(position) * m.rows + row_begin + threadIdx.x, acc);
    } else if (threadIdx.x < 64) {
        // The first wave holds every row sum: lane t < rows the first member's row row_begin + t, lane rows + t
        // the second member's.
        const int t = threadIdx.x;
        if (t < vrows) store_f32((t < rows ? m.y : inline_members.m[1].y) + row_begin + (t < rows ? t : t - rows), acc);
        const float up = __shfl(acc, (t + rows) & 63, 64);
        const float activated = swiglu_value(acc, up);
        if (!out.q8k) {  // SwiGlu only
            if (t < rows) store_f32(out.activated + row_begin + t, activated);
            return;
        }
        // SwiGlu of the workgroup's rows, stored as agent-scope atomics so the workgroup that quantizes the run
        // reads them coherently from any XCD, then waited for (every store of this wave acknowledged) before
        // this workgroup is counted in: a count the quantizer sees implies the values it reads are there.
        if (t < rows)
            __hip_atomic_store(out.activated + row_begin + t, activated, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t seen = 0;
        if (t == 0)
            seen = __hip_atomic_fetch_add(out.counters + (row_begin >> 8), 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        seen = static_cast<uint32_t>(__shfl(static_cast<int>(seen), 0, 64));
        const uint32_t arrivals = 256u / static_cast<uint32_t>(tile_rows);  // a power of two
        if (((seen + 1u) & (arrivals - 1u)) == 0u) {
            // The last of the run's workgroups: Q8_K of its 256 SwiGlu values (Q8KCodec.QuantizeBlock).
            const int run = row_begin >> 8;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = __hip_atomic_load(out.activated + 256 * run + 4 * t + i, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            const Q8KLane q = q8k_quantize_values(v, t);
            uint8_t* dst = out.q8k + static_cast<int64_t>(run) * kQ8KBlockBytes;
            if (q.zero) {
                uint32_t* d32 = reinterpret_cast<uint32_t*>(dst);
                for (int i = t; i < kQ8KBlockBytes / 4; i += 64) d32[i] = 0u;
            } else {
                reinterpret_cast<uint32_t*>(dst + 4)[t] = q.packed;
                if ((t & 3) == 0) reinterpret_cast<int16_t*>(dst + 260)[t >> 2] = static_cast<int16_t>(q.group_sum);
                if (t == 0) reinterpret_cast<float*>(dst)[0] = q.scale;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The same product over a few positions (multi_pays: from 2, mostly to 15). A workgroup owns a tile of rows of one member at up to
// kMultiPositions positions: it quantizes those positions' rows, then unpacks every (row, block) pair's weights
// once for all of them. What bounds the product at these sizes is the vector ALU (unpacking, the quantization every
// workgroup repeats) and one latency chain, not HBM; a launch slice per position repeated all of it per position.
// One workgroup of 512 threads per CU keeps the repeated quantization to one per CU. Each output is formed exactly
// as gemv_kint_kernel forms it.
// ------------------------------------------------------------------------------------------------
constexpr int kMultiThreads = 512;
constexpr int kMultiPositions = 8;
constexpr int kMultiLdsBytes = 144 * 1024;
constexpr int kMultiMembers = 32;  // of one launch

// The tiles of members of different sizes, numbered over the members: one workgroup each, so that consecutive workgroups,
// which are dealt to the XCDs in turn, all have rows. (In a grid as wide as the largest member, with the smaller ones'
// workgroups without rows in between, the others were dealt unevenly, and one that found no free CU in its XCD ran in a
// second round: members of 8399, 64 and 5917 rows x 4096 Q6_K over 3 positions 26.1 us, numbered 16.0, two of 7190 15.5.)
// Members of one size keep the grid, whose y is the member: finding it in the arguments takes 0.3 to 0.5 us more.
struct MultiTiles {
    int first[kMultiMembers];  // of each member; past the last member INT32_MAX
};

// A position's activations of a chunk of K blocks, in dwords: the codes, then the group sums, then the scales, and the
// next position's behind them at a whole 16 bytes. Codes and sums are read and written 8 and 16 bytes at a time, and an
// LDS access that wide has to lie on a multiple of its width. (Sums behind the scales and positions 77 K dwords apart
// were off it for every K that is not a multiple of 4.)
constexpr int multi_sums(int K) { return kCodeStride * K; }
constexpr int multi_scales(int K) { return multi_sums(K) + 8 * K; }
constexpr int multi_position(int K) { return (multi_scales(K) + K + 3) & ~3; }
constexpr bool multi_aligned() {
    for (int K = 1; K <= kMultiLdsBytes / (kActDwords * 4); ++K)
        if (multi_sums(K) % 4 || multi_position(K) % 4) return false;
    return kCodeStride % 4 == 0;
}
static_assert(multi_aligned(), "16-byte LDS accesses of the staged activations");

template <int FORMAT, bool INLINE, bool NUMBERED>
__global__ __launch_bounds__(kMultiThreads) void gemv_kint_multi_kernel(KintMembers inline_members,
                                                                         const MatDesc* __restrict__ group,
                                                                         LaunchShape s, int per, MultiTiles tiles) {
    constexpr int G = 4;  // lanes per (row, block) pair
    constexpr int kSlots = kMultiThreads / G, kRows16 = kMultiThreads / 16;
    constexpr int kDepth = 2;  // pairs whose payload is in flight
    using Raw = typename std::conditional<FORMAT == kQ4_K, Q4KRaw, Q6KRaw>::type;
    int member = blockIdx.y, tile = blockIdx.x;
    if constexpr (NUMBERED) {
        int begin = 0;
#pragma unroll
        for (int i = 1; i < (INLINE ? kKintInlineMembers : kMultiMembers); ++i)
            if (tile >= tiles.first[i]) {
                member = i;
                begin = tiles.first[i];
            }
        tile -= begin;
    }
    const MatDesc m = INLINE ? inline_members.m[member] : group[member];
    const int row_begin = tile * s.rows_per_wg;
    const int rows = min(s.rows_per_wg, m.rows - row_begin);
    const int first = blockIdx.z * per, np = min(per, s.positions - first);
    const int nb = s.blocks, K = s.chunk_blocks;
    const int tid = threadIdx.x, lane = tid & 63, c = lane % G, j16 = tid & 15;

    // Per position: codes, group sums and scales of K blocks; then the terms, [position][row][block].
    extern __shared__ uint32_t smem[];
    auto act_of = [&](int pp) {
        uint32_t* base = smem + pp * multi_position(K);
        return ActTile{base, reinterpret_cast<int16_t*>(base + multi_sums(K)),
                       reinterpret_cast<float*>(base + multi_scales(K))};
    };
    float* terms = reinterpret_cast<float*>(smem + np * multi_position(K));

    auto load_pair = [&](int b0, int kb, int p, Raw& r) {
        const int row = row_begin + p / kb, b = b0 + p % kb;
        if constexpr (FORMAT == kQ4_K)
            q4k_load(m.w + static_cast<int64_t>(row) * s.row_bytes + b * 144, c, r);
        else
            q6k_load_quarter(m.w, static_cast<int64_t>(m.rows) * nb, static_cast<int64_t>(row) * nb + b, c, r);
    };
    auto load_x = [&](int b0, int kb, int item, f32x4 (&x4)[4]) {  // 16 values of (position, block) `item`
        const int pp = item / kb, b = b0 + item % kb;
        const float* src = m.x + static_cast<int64_t>(first + pp) * s.columns + 256 * b + 16 * j16;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x4 raw = load16_a4(reinterpret_cast<const uint8_t*>(src + 4 * q));
            x4[q] = f32x4{__uint_as_float(raw[0]), __uint_as_float(raw[1]), __uint_as_float(raw[2]),
                          __uint_as_float(raw[3])};
        }
    };

    float acc[2] = {0.0f, 0.0f};  // sums t = tid, tid + threads of rows * np: row t % rows of position t / rows, in block order
    const int p0 = tid / G;
    for (int b0 = 0; b0 < nb; b0 += K) {
        const int kb = min(K, nb - b0), pairs = rows * kb, items = np * kb;
        // The first activations, then the first pairs' weights; a 16-lane row per (position, block), 32 at a time.
        // (Two or four blocks side by side per row measured 5-40% slower: the quantization is bound by its instructions.)
        int item = tid >> 4;
        f32x4 x4[4];
        load_x(b0, kb, min(item, items - 1), x4);
        Raw buf[kDepth];
#pragma unroll
        for (int i = 0; i < kDepth; ++i) load_pair(b0, kb, min(p0 + i * kSlots, pairs - 1), buf[i]);
        for (; item < items; item += kRows16) {
            float v[16];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * q + e] = x4[q][e];
            if (item + kRows16 < items) load_x(b0, kb, item + kRows16, x4);
            const Q8KRow16 qr = q8k_quantize_row16(v, lane);
            const ActTile act = act_of(item / kb);
            const int bl = item % kb;
            *reinterpret_cast<u32x4*>(act.codes + kCodeStride * bl + 4 * j16) =
                u32x4{qr.packed[0], qr.packed[1], qr.packed[2], qr.packed[3]};
            act.sums[16 * bl + j16] = static_cast<int16_t>(qr.group_sum);
            if (j16 == 0) act.scales[bl] = qr.scale;
        }
        __syncthreads();  // activations of the chunk staged
        for (int base = p0; base < pairs; base += kDepth * kSlots) {
#pragma unroll
            for (int i = 0; i < kDepth; ++i) {
                const int p = base + i * kSlots;
                if (p < pairs) {
                    const int bl = p % kb;
                    if constexpr (FORMAT == kQ4_K) {
                        const Raw& r = buf[i];
                        int s0, m0, s1, m1;
                        q4k_scale_min(2 * c, r.head, s0, m0);
                        q4k_scale_min(2 * c + 1, r.head, s1, m1);
                        const uint32_t mm0 = m0 * 0x10001u, mm1 = m1 * 0x10001u;
                        uint32_t lo[8], hi[8];
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            lo[w] = r.qs0[w] & 0x0F0F0F0Fu;
                            lo[4 + w] = r.qs1[w] & 0x0F0F0F0Fu;
                            hi[w] = (r.qs0[w] >> 4) & 0x0F0F0F0Fu;
                            hi[4 + w] = (r.qs1[w] >> 4) & 0x0F0F0F0Fu;
                        }
                        const float d = half_bits_to_float(r.head[0] & 0xFFFFu), dmin = half_bits_to_float(r.head[0] >> 16);
                        for (int pp = 0; pp < np; ++pp) {
                            const ActTile act = act_of(pp);
                            const uint32_t* codes = act.codes + kCodeStride * bl + 16 * c;
                            int dl = 0, dh = 0;
#pragma unroll
                            for (int q = 0; q < 2; ++q) {
                                const u32x4 l = *reinterpret_cast<const u32x4*>(codes + 4 * q);
                                const u32x4 h = *reinterpret_cast<const u32x4*>(codes + 8 + 4 * q);
#pragma unroll
                                for (int w = 0; w < 4; ++w) {
                                    dl = sdot4(lo[4 * q + w], l[w], dl);
                                    dh = sdot4(hi[4 * q + w], h[w], dh);
                                }
                            }
                            const uint2 sums = *reinterpret_cast<const uint2*>(act.sums + 16 * bl + 4 * c);
                            const int dot = group_sum_last_int<G>(__mul24(s0, dl) + __mul24(s1, dh));
                            const int mins = group_sum_last_int<G>(sdot2(sums.x, mm0, sdot2(sums.y, mm1, 0)));
                            const float a = act.scales[bl];
                            float term = 0.0f;  // zero activation block: skipped (QuantizedKAvx2Kernel.cs:86)
                            if (a != 0.0f)
                                term = __fsub_rn(__fmul_rn(__fmul_rn(d, a), static_cast<float>(dot)),
                                                 __fmul_rn(__fmul_rn(dmin, a), static_cast<float>(mins)));
                            if (c == G - 1) terms[pp * pairs + p] = term;
                        }
                    } else {
                        const Raw& r = buf[i];
                        const int h = c >> 1, t = c & 1;
                        uint32_t q[4][4];
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            const uint32_t a = r.qla[w], bq = r.qlb[w], hb = r.qh[w];
                            q[0][w] = (a & 0x0F0F0F0Fu) | ((hb << 4) & 0x30303030u);
                            q[1][w] = (bq & 0x0F0F0F0Fu) | ((hb << 2) & 0x30303030u);
                            q[2][w] = ((a >> 4) & 0x0F0F0F0Fu) | (hb & 0x30303030u);
                            q[3][w] = ((bq >> 4) & 0x0F0F0F0Fu) | ((hb >> 2) & 0x30303030u);
                        }
                        const float d = q6k_d(r);
                        for (int pp = 0; pp < np; ++pp) {
                            const ActTile act = act_of(pp);
                            const uint32_t* codes = act.codes + kCodeStride * bl + 32 * h + 4 * t;
                            const u32x4 sums = *reinterpret_cast<const u32x4*>(act.sums + 16 * bl + 8 * h);  // pair k: t = 0, 1
                            int total = 0;
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                const u32x4 x = *reinterpret_cast<const u32x4*>(codes + 8 * k);
                                int dot = 0;
#pragma unroll
                                for (int w = 0; w < 4; ++w) dot = sdot4(q[k][w], x[w], dot);
                                total += __mul24(static_cast<int8_t>(r.sc >> (8 * k)),
                                                 dot - 32 * static_cast<int16_t>(sums[k] >> (16 * t)));
                            }
                            const int dot = group_sum_last_int<G>(total);
                            const float a = act.scales[bl];
                            const float term = a != 0.0f ? __fmul_rn(__fmul_rn(a, d), static_cast<float>(dot)) : 0.0f;
                            if (c == G - 1) terms[pp * pairs + p] = term;
                        }
                    }
                    if (p + kDepth * kSlots < pairs) load_pair(b0, kb, p + kDepth * kSlots, buf[i]);
                }
            }
        }
        __syncthreads();  // the chunk's terms are in LDS
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int t = tid + k * kMultiThreads;
            if (t < rows * np)
                for (int b = 0; b < kb; ++b) acc[k] = __fadd_rn(acc[k], terms[(t / rows) * pairs + (t % rows) * kb + b]);
        }
        if (b0 + K < nb) __syncthreads();  // every thread is done with this chunk's activations and terms
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int t = tid + k * kMultiThreads;
        if (t < rows * np) store_f32(m.y + static_cast<int64_t>(first + t / rows) * m.rows + row_begin + t % rows, acc[k]);
    }
}

}  // namespace

hipError_t launch_q8k_quantize(const float* x, int columns, int positions, uint8_t* out, hipStream_t stream) {
    if (columns <= 0 || positions <= 0) return hipSuccess;
    dim3 grid(columns / 256, positions);
    q8k_quantize_kernel<<<grid, 64, 0, stream>>>(x, columns, out);
    return hipGetLastError();
}

size_t kint_lds_bytes(int blocks, int rms_columns) {
    const size_t staged = rms_columns <= kNormStageColumns ? static_cast<size_t>(rms_columns) * sizeof(float) : 0;
    return static_cast<size_t>(kint_red_offset(blocks, kTileRows)) * sizeof(uint32_t) + kThreads * sizeof(double) +
           staged;
}

int kint_max_blocks() {
    return static_cast<int>((64 * 1024 - kThreads * sizeof(double) - 4) / ((kActDwords + kTileRows) * sizeof(uint32_t)));
}

namespace {

template <int XF, bool PAIRED = false>
hipError_t launch_kint(const MatDesc* members, const MatDesc* device_members, int count, LaunchShape s,
                       const InputTransform& xf, hipStream_t stream, const OutputSwiGluQ8K& out = {}) {
    if (count <= 0 || s.rows_max <= 0 || s.positions <= 0) return hipSuccess;
    if (count > kKintInlineMembers && !device_members) return hipErrorInvalidValue;
    if (PAIRED && (count != 2 || s.positions != 1 || s.rows_max % 256 != 0 || members[0].rows != s.rows_max ||
                   members[1].rows != s.rows_max))
        return hipErrorInvalidValue;
    // Rows per workgroup: 64, halved (down to 4) while the grid has fewer than 1024 workgroups and either a
    // thread slot would hold more than three (row, block) pairs (the pairs it prefetches before quantizing)
    // or the grid has fewer than 192 workgroups. Measured on the decode step's groups: q/k/v and o take 8-16
    // rows, gate/up 32, down (35 blocks) 4; large grouped launches keep 64. Then halved while a workgroup
    // would stream more than 256 KB of payload, so long rows leave no long tail of workgroups at the end of
    // a launch (1536 x 8960 grouped: Q6_K 5.43 -> 5.76 TB/s, Q4_K 5.70 -> 5.86 TB/s at 32 rows; 16 rows
    // measured slower).
    const int64_t launched = static_cast<int64_t>(count) * s.positions;
    auto groups_for = [&](int t) { return launched * ((s.rows_max + t - 1) / t); };
    int tile = kTileRows;
    while (tile > 4 && groups_for(tile) < 1024 && (tile * s.blocks > 192 || groups_for(tile) < 192)) tile /= 2;
    while (tile > 4 && static_cast<int64_t>(tile) * s.row_bytes > 256 * 1024) tile /= 2;
    // Paired: each workgroup owns `tile` rows of both members, so half the rows of the unpaired tile keep the
    // work per workgroup and the workgroup count (at most 32 rows, so the 2 * tile row sums fit one wave).
    if (PAIRED) tile = max(4, min(32, tile / 2));
    s.rows_per_wg = tile;
    // Rows wider than the LDS holds are staged kint_max_blocks() blocks at a time.
    s.chunk_blocks = s.blocks < kint_max_blocks() ? s.blocks : kint_max_blocks();
    dim3 grid((s.rows_max + tile - 1) / tile, PAIRED ? 1 : count, s.positions);
    const size_t lds = kint_lds_bytes(s.chunk_blocks, XF == kInputAddRmsNorm ? s.columns : 0);
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    KintMembers inline_members{};
    const MatDesc* group = nullptr;
    if (count <= kKintInlineMembers)
        for (int i = 0; i < count; ++i) inline_members.m[i] = members[i];
    else
        group = device_members;
    if constexpr (PAIRED) {
        if (s.format == kQ4_K)
            gemv_kint_kernel<kQ4_K, XF, true, true><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
        else if (s.format == kQ6_K)
            gemv_kint_kernel<kQ6_K, XF, true, true><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    if (s.format == kQ4_K && group)
        gemv_kint_kernel<kQ4_K, XF, false, false><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
    else if (s.format == kQ4_K)
        gemv_kint_kernel<kQ4_K, XF, true, false><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
    else if (s.format == kQ6_K && group)
        gemv_kint_kernel<kQ6_K, XF, false, false><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
    else if (s.format == kQ6_K)
        gemv_kint_kernel<kQ6_K, XF, true, false><<<grid, kThreads, lds, stream>>>(inline_members, group, s, xf, out);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace

namespace {

constexpr int kMultiRows = 128;  // two sums per thread at kMultiPositions

int multi_slices(int positions) { return (positions + kMultiPositions - 1) / kMultiPositions; }

// Whether the positions share a workgroup: where a launch slice per position would be bound by its throughput (about
// 18 M weights x positions), and by more than what quantizing a slice's positions in every workgroup takes. Measured over
// the same calls as kmfma_pays (us, a slice per position against this): 4096 x 4096 Q4_K 7.2 and 5.2 at 2 positions, 22.0
// and 14.6 at 15; 14380 x 1280 Q6_K 31.5 and 12.0 at 12; 8000 x 768 Q4_K 5.8 and 5.1 at 6; 3088 x 10752 Q6_K 56 and 27 at
// 12; but 742 x 4608 Q4_K 6.0 and 8.0 at 8, 721 x 2816 5.8 and 7.1 at 15, 512 x 1024 4.4 and 5.0 at 8. Q6_K, whose
// slices take longer a product, from 0.8 of that (835 x 9728 at 4 11.1 and 8.9).
bool multi_pays(int format, int64_t rows, int blocks, int positions) {
    const int slices = multi_slices(positions), per = (positions + slices - 1) / slices;
    const int64_t line = 18000000 + 150000 * static_cast<int64_t>(per) * blocks;
    return rows * blocks * 256 * positions >= (format == kQ6_K ? line * 4 / 5 : line);
}

// In slices of at most kMultiPositions positions, with one workgroup per CU over all slices; at most kMultiMembers
// members a launch.
hipError_t launch_kint_multi(const MatDesc* members, const MatDesc* device_members, int count, LaunchShape s,
                             hipStream_t stream) {
    for (; count > kMultiMembers; count -= kMultiMembers, members += kMultiMembers, device_members += kMultiMembers) {
        const hipError_t e = launch_kint_multi(members, device_members, kMultiMembers, s, stream);
        if (e != hipSuccess) return e;
    }
    const int slices = multi_slices(s.positions);
    const int per = (s.positions + slices - 1) / slices;
    int64_t rows = 0;
    for (int i = 0; i < count; ++i) rows += members[i].rows;
    int64_t tile = std::max<int64_t>(4, (rows * slices + kCus - 1) / kCus);
    // No more than one workgroup per CU where the rounding of each slice's and member's last tile made a few more: they
    // run in a second round (297 x 2816 Q6_K over 48 positions, 258 workgroups: 16.0 us; 40 positions 9.5).
    auto workgroups = [&](int64_t t) {
        int64_t n = 0;
        for (int i = 0; i < count; ++i) n += (members[i].rows + t - 1) / t;
        return n * slices;
    };
    while (tile < kMultiRows && workgroups(tile) > kCus) ++tile;
    s.rows_per_wg = static_cast<int>(std::min<int64_t>(tile, kMultiRows));
    // (Up to three dwords a position round its activations up to 16 bytes.)
    const int per_block = per * (kActDwords + s.rows_per_wg) * static_cast<int>(sizeof(uint32_t));
    const int most = (kMultiLdsBytes - per * 3 * static_cast<int>(sizeof(uint32_t))) / per_block;
    s.chunk_blocks = std::min(s.blocks, most);
    const bool in_arguments = count <= kKintInlineMembers;
    KintMembers inline_members{};
    MultiTiles tiles;
    std::fill(tiles.first, tiles.first + kMultiMembers, INT32_MAX);
    const auto tiles_of = [&](int rows_of) { return (rows_of + s.rows_per_wg - 1) / s.rows_per_wg; };
    int64_t total = 0;
    bool even = true;
    for (int i = 0; i < count; ++i) {
        if (in_arguments) inline_members.m[i] = members[i];
        tiles.first[i] = static_cast<int>(std::min<int64_t>(total, INT32_MAX));
        total += tiles_of(members[i].rows);
        even = even && tiles_of(members[i].rows) == tiles_of(s.rows_max);
    }
    if (total > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid = even ? dim3(tiles_of(s.rows_max), count, slices) : dim3(static_cast<unsigned>(total), 1, slices);
    const size_t lds = sizeof(uint32_t) * static_cast<size_t>(per) *
                       (multi_position(s.chunk_blocks) + s.rows_per_wg * s.chunk_blocks);
    auto go = [&](auto kernel) {
        kernel<<<grid, kMultiThreads, lds, stream>>>(inline_members, device_members, s, per, tiles);
        return hipGetLastError();
    };
    auto pick = [&](auto format) {
        constexpr int F = decltype(format)::value;
        if (even) return in_arguments ? go(gemv_kint_multi_kernel<F, true, false>) : go(gemv_kint_multi_kernel<F, false, false>);
        return in_arguments ? go(gemv_kint_multi_kernel<F, true, true>) : go(gemv_kint_multi_kernel<F, false, true>);
    };
    if (s.format == kQ4_K) return pick(std::integral_constant<int, kQ4_K>{});
    if (s.format == kQ6_K) return pick(std::integral_constant<int, kQ6_K>{});
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemv_kint(const MatDesc* members, const MatDesc* device_members, int count, LaunchShape s,
                            hipStream_t stream) {
    if (count > 0 && s.rows_max > 0 && s.positions > 1) {
        if (count > kKintInlineMembers && !device_members) return hipErrorInvalidValue;
        int64_t rows = 0;
        for (int i = 0; i < count; ++i) rows += members[i].rows;
        if (multi_pays(s.format, rows, s.blocks, s.positions)) return launch_kint_multi(members, device_members, count, s, stream);
    }
    return launch_kint<kInputPlain>(members, device_members, count, s, InputTransform{}, stream);
}

hipError_t launch_gemv_kint_transformed(const MatDesc* members, const MatDesc* device_members, int count,
                                        LaunchShape s, const InputTransform& xf, hipStream_t stream) {
    if (s.positions != 1 || !xf.a) return hipErrorInvalidValue;
    switch (xf.kind) {
        case kInputPlain: return launch_kint<kInputPlain>(members, device_members, count, s, xf, stream);
        case kInputAddRmsNorm:
            if (!xf.w) return hipErrorInvalidValue;
            return launch_kint<kInputAddRmsNorm>(members, device_members, count, s, xf, stream);
        case kInputSwiGlu:
            if (!xf.b) return hipErrorInvalidValue;
            return launch_kint<kInputSwiGlu>(members, device_members, count, s, xf, stream);
        case kInputQ8K: return launch_kint<kInputQ8K>(members, device_members, count, s, xf, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gemv_kint_swiglu(const MatDesc* members, LaunchShape s, const InputTransform& xf,
                                   const OutputSwiGluQ8K& out, hipStream_t stream) {
    if (s.positions != 1 || !out.activated || (out.q8k && !out.counters)) return hipErrorInvalidValue;
    switch (xf.kind) {
        case kInputPlain: return launch_kint<kInputPlain, true>(members, nullptr, 2, s, xf, stream, out);
        case kInputAddRmsNorm:
            if (!xf.a || !xf.w) return hipErrorInvalidValue;
            return launch_kint<kInputAddRmsNorm, true>(members, nullptr, 2, s, xf, stream, out);
        case kInputQ8K:
            if (!xf.a) return hipErrorInvalidValue;
            return launch_kint<kInputQ8K, true>(members, nullptr, 2, s, xf, stream, out);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace satori
