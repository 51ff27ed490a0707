// Several-position FP32-activation product for Q8_0 and Q4_0 on the matrix cores (gfx950 bf16 MFMA): the
// batched form of QuantizedMatVec.ExecuteBatch for the legacy formats (ExecuteBatchFloat / ExecuteBatchRows,
// src/Satori.Core/QuantizedMatVec.cs:221-347), with the arithmetic of the scalar reference per block
// (QuantizedMatVec.ExecuteScalar, QuantizedMatVec.cs:45-78: sum = q . x over the block's 32 weights, then
// total += Scale * sum), so the weights are read once per position tile instead of once per position.
//
// Exact operands. A block's codes q are small integers (Q8_0: -128..127; Q4_0: -8..7, used as 16 q), exact in
// bf16. Each activation x is split into three bf16 parts x = hi + lo + lolo, each the next 8 significant bits
// cut by truncation (x - hi and (x - hi) - lo are exact in FP32, and the last part has at most 8 significant
// bits). bf16 has FP32's exponent range, but a part below 2^-126 would be a bf16 subnormal: its bits below
// 2^-133 do not fit and the matrix cores may flush it. So every x is first lifted by 2^24: every bit of a
// lifted FP32 number, subnormals included, weighs at least 2^-125, and the split is exact for every finite x.
// Every q * part product is exact in FP32 (at most 16 significant bits), and the block sum sum_k q_k x_k is
// three bf16 MFMA chains accumulating in FP32. Only the FP32 additions round, in an order of their own, and the
// final scaling by 2^-24 rounds once where the result is subnormal: within 1e-5 * sum |w x| + n * 2^-149 of
// the reference, like every FP32 path here. A lifted sum stays below 2^118 while |x| < 2^40 (2^26 blocks of the
// largest code and scale); a position holding a larger, infinite or NaN activation is flagged while it is
// split, and its tile is computed once more from activations as they are (finish_flagged), whose sums overflow and
// propagate where the reference's do.
//
// Launches. fbatch_kernel: a workgroup of eight waves walks (row group, position unit) tiles of 64 RH rows x 32 TP
// positions, WAYS = 8 / RH blocks a round: each wave owns 64 rows x 32 TP positions of one of the round's blocks, and
// the ways' sums are added at the end of the tile. The tiles' rounds are dealt to one workgroup per CU in equal
// contiguous ranges (the chip is full and ends together whatever the shape: 4096 x 4096 over 256 positions has 64
// tiles, over 12 positions 32); a tile cut between workgroups goes through partial sums in the scratch, added by
// fbatch_fixup_kernel. Up to 64 positions, and in smaller products, the activations are split by the workgroups that
// use them (FUSED, 128 rows and four ways); in larger ones (fbatch_plan) once by fbatch_pack_kernel into memory,
// since every row group would split them again, and then take 256 rows and two ways: twice the rows halve the parts'
// bytes a workgroup reads, which then bound it (128 rows: 1.3 GB through L2 in 94 us at 11008 x 4096 Q4_0 over 256
// positions; 256 rows 0.83 GB). Short rows under many outputs take whole tiles instead (fbatch_tiles_kernel).
// Measured, whole call in a queue of calls (us, before: one 32 x 32 tile per wave and block, its workgroups one
// per 128 rows and position tile): 256 positions 11008 x 4096 Q4_0 152 -> 83, 4096 x 4096 Q8_0 64 -> 41, 256 x 8192
// Q8_0 116 -> 16; 64 positions 4096 x 4096 Q8_0 62 -> 18; 12 positions (the single-position kernel) 29 -> 14.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace satori {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTile = 32;                              // rows and positions of one matrix-core tile
constexpr int kThreads = 256;                          // of the pack and fix-up kernels
constexpr int kPartBytes = 1024;                       // one part of one K step of one (block, tile)
constexpr int kBlockTileBytes = 3 * 2 * kPartBytes;    // 3 parts x 2 K steps of 16 columns
constexpr float kLift = 0x1p24f;
constexpr int kLiftExponent = 24;
constexpr uint32_t kFlagBits = 0x5F80u;                // a lifted part of 2^64: |x| from 2^40 on (infinite, NaN) is flagged
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Parts of the packed form: for 32-column block b and 32-position tile t, 6 KB at (b * tiles + t) * 6144:
// part s (0: hi, 1: lo, 2: lolo), K step st at (2s + st) * 1024, lane l = 32h + p holding the 8 bf16 of position
// 32t + p at columns 32b + slot_column(st, h) .. + 7. Positions past the last are zero. The scratch holds, beside the
// partial sums and their flags, one word per (block, tile, K step): the tile's flagged positions in that slot's columns.
//
// The columns of a block are dealt to the K steps so that a lane's codes are contiguous: Q8_0 lane half h
// holds bytes 16h .. 16h + 15 of the record, Q4_0 bytes 8h .. 8h + 7 (low nibbles in step 0, high in step 1).
template <int FORMAT>
__device__ __forceinline__ int slot_column(int st, int h) {
    return FORMAT == kQ8_0 ? 16 * h + 8 * st : 16 * st + 8 * h;
}

// Eight activations lifted and split into their bf16 parts, packed in pairs; true when one must be flagged.
__device__ __forceinline__ bool split8(const float (&v)[8], u32x4 (&part)[3]) {
    u16x2 largest = {0, 0};
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        uint32_t p[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float x = __fmul_rn(v[e + i], kLift);
            p[0][i] = __float_as_uint(x);
            const float r = __fsub_rn(x, __uint_as_float(p[0][i] & 0xFFFF0000u));  // exact
            p[1][i] = __float_as_uint(r);
            p[2][i] = __float_as_uint(__fsub_rn(r, __uint_as_float(p[1][i] & 0xFFFF0000u)));  // at most 8 bits
        }
#pragma unroll
        for (int s = 0; s < 3; ++s) part[s][e >> 1] = __builtin_amdgcn_perm(p[s][1], p[s][0], 0x07060302u);
        largest = __builtin_elementwise_max(largest, __builtin_bit_cast(u16x2, part[0][e >> 1] & 0x7FFF7FFFu));
    }
    return max(largest[0], largest[1]) >= kFlagBits;
}

__device__ __forceinline__ void load8(const float* src, float (&v)[8]) {
    const u32x4 a = load16_a4(reinterpret_cast<const uint8_t*>(src));
    const u32x4 b = load16_a4(reinterpret_cast<const uint8_t*>(src + 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = __uint_as_float(a[e]);
        v[4 + e] = __uint_as_float(b[e]);
    }
}

// One wave per (block, position tile, K step), lane by lane the 8 activations of its operand slot, split.
template <int FORMAT>
__global__ __launch_bounds__(kThreads) void fbatch_pack_kernel(const float* __restrict__ x, int columns, int positions,
                                                               int tiles, uint8_t* __restrict__ parts,
                                                               uint32_t* __restrict__ flags) {
    const int64_t item = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int blocks = columns / 32;
    if (item >= static_cast<int64_t>(blocks) * tiles * 128) return;  // whole waves
    const int lane = static_cast<int>(item & 63), st = static_cast<int>((item >> 6) & 1);
    const int64_t bt = item >> 7;  // b * tiles + t
    const int b = static_cast<int>(bt / tiles), t = static_cast<int>(bt - static_cast<int64_t>(b) * tiles);
    const int p = t * kTile + (lane & 31);
    float v[8];
    load8(x + static_cast<int64_t>(min(p, positions - 1)) * columns + 32 * b + slot_column<FORMAT>(st, lane >> 5), v);
    if (p >= positions)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
    u32x4 part[3];
    const uint64_t flagged = __ballot(split8(v, part));
    uint8_t* dst = parts + bt * kBlockTileBytes + st * kPartBytes + 16 * lane;
#pragma unroll
    for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x4*>(dst + 2 * s * kPartBytes) = part[s];
    if (lane == 0) flags[2 * bt + st] = static_cast<uint32_t>(flagged) | static_cast<uint32_t>(flagged >> 32);
}

// Two small integers as a pair of bf16 (exact: at most 8 significant bits): the high halves of their FP32
// patterns, byte i low, joined by one byte permute.
__device__ __forceinline__ uint32_t pack_bytes(uint32_t w, int i) {
    return __builtin_amdgcn_perm(__float_as_uint(sbyte_to_float(w, i + 1)), __float_as_uint(sbyte_to_float(w, i)),
                                 0x07060302u);
}

// Pair k % 4 of the lane's second operand (8 codes of its row) for K step k / 4 of a block: Q8_0 from its 16
// signed bytes, Q4_0 from its 8 nibble bytes (each nibble q - 8 in two's complement) as the bytes 16 (q - 8).
template <int FORMAT>
__device__ __forceinline__ uint32_t code_pair(const uint32_t (&raw)[4], int k) {
    if constexpr (FORMAT == kQ8_0) return pack_bytes(raw[k >> 1], 2 * (k & 1));
    const uint32_t w = raw[k >> 1 & 1];
    return pack_bytes((k < 4 ? w << 4 : w) & 0xF0F0F0F0u, 2 * (k & 1));
}

__device__ __forceinline__ f32x16 mfma_bf16(const bf16x8& a, const bf16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

struct FbatchArgs {
    const uint8_t* w;       // device layout (code records, then FP16 scales)
    const float* x;         // [positions][columns]
    const uint8_t* parts;   // packed form: split activations
    const uint32_t* flags;  // packed form: flagged positions per (block, tile, K step)
    float* partial;         // two slots per workgroup: the cut tiles at the ends of its range
    uint32_t* slot_flags;   // fused form: flagged positions found by a piece (TP words a slot)
    uint32_t* tile_flags;   // fused form: flagged positions of a tile that was not cut (TP words a tile)
    float* y;               // [positions][rows]
    int rows, blocks, positions, tiles;
    int units;              // position units: ceil(tiles / TP)
    int rounds;             // rounds per tile: ceil(blocks / ways)
    int total;              // tiles x rounds (fbatch_tiles_kernel: tiles)
    int workgroups;         // ranges: the first total % workgroups hold total / workgroups + 1 rounds, the others one less
    int share, longer;      // total / workgroups, total % workgroups
};

// Floats of one partial slot: [row half][row tile][position tile][output / 4][lane][output % 4].
constexpr int slot_floats(int TP, int RH) { return 2 * RH * TP * 1024; }

// First round of range i of the launch, and the range that holds round r.
__device__ __forceinline__ int range_start(const FbatchArgs& a, int i) { return a.share * i + min(i, a.longer); }
__device__ __forceinline__ int range_of(const FbatchArgs& a, int r) {
    const int in_longer = a.longer * (a.share + 1);
    return r < in_longer ? r / (a.share + 1) : a.longer + (r - in_longer) / a.share;
}

// Eight activations of a flagged position, in parts. Elements of 2^-80 and more are taken as they are (Q4_0: divided by 16,
// the other factor of its codes 16 q): their parts are above 2^-126, and every sum of products overflows where the plain
// one does. An infinite or NaN element is its first part alone. Smaller ones (SMALL) are lifted into parts of their own.
constexpr float kSmallLine = 0x1p-80f;
template <int FORMAT, bool SMALL>
__device__ __forceinline__ void split8_unlifted(const float (&v)[8], u32x4 (&part)[3]) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        uint32_t p[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float x = __fmul_rn(v[e + i], SMALL ? kLift : FORMAT == kQ4_0 ? 0.0625f : 1.0f);
            const float magnitude = __builtin_fabsf(v[e + i]);
            if ((magnitude < kSmallLine) != SMALL) x = 0.0f;
            p[0][i] = magnitude != magnitude ? 0x7FC00000u : __float_as_uint(x);
            float r = __fsub_rn(x, __uint_as_float(__float_as_uint(x) & 0xFFFF0000u));
            if (!(magnitude < INFINITY)) r = 0.0f;
            p[1][i] = __float_as_uint(r);
            p[2][i] = __float_as_uint(__fsub_rn(r, __uint_as_float(p[1][i] & 0xFFFF0000u)));
        }
#pragma unroll
        for (int s = 0; s < 3; ++s) part[s][e >> 1] = __builtin_amdgcn_perm(p[s][1], p[s][0], 0x07060302u);
    }
}

// Whether one of the wave's elements is below 2^-80 (zeros too).
__device__ __forceinline__ bool any_small(const u32x4 (&v)[4]) {
    float least = INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) least = __builtin_fminf(least, __builtin_fabsf(__uint_as_float(v[j][e])));
    return __ballot(least < kSmallLine) != 0;
}

// Outputs of the flagged positions of one 32-row x 32-position tile, by 4 G waves, each the block sums
// (QuantizedMatVec.cs:45-78) of every 4 G-th block over the whole tile on the matrix cores, added to those of the waves
// before it. A wave reads its block's activations in whole lines, a block ahead, and passes them through its own LDS
// (32 rows of kFlaggedStride floats) into operand order: read in operand order, a line took four requests that the L1
// did not hold together, and that bound it (11008 x 4096 Q4_0 over 256 positions, every one flagged, 315 us against
// 250). Measured (us, a batch without flagged positions, with one, with all; in brackets before, when each flagged
// position was summed in FP32 after another): 11008 x 4096 Q4_0 over 256 96, 176, 250 (144, 2,597); 4096 x 4096 Q8_0 over
// 256 45, 101, 106 (80, 1,164), over 12 15, 35, 34 (27, 159).
constexpr int kFlaggedStride = 36;  // padded off the banks
template <int FORMAT, int G>
__device__ void finish_flagged(const FbatchArgs& a, int row0, int p0, uint32_t mask, float* lds) {
    constexpr int kRecord = FORMAT == kQ8_0 ? 32 : 16, kWaves = 4 * G;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5, row = row0 + (lane & 31);
    const uint32_t first = static_cast<uint32_t>(min(row, a.rows - 1)) * a.blocks;  // (a payload has at most 2^31 - 1 bytes)
    const uint32_t record = first * kRecord + (FORMAT == kQ8_0 ? 16 : 8) * h;
    const uint8_t* scales = a.w + static_cast<int64_t>(a.rows) * a.blocks * kRecord;
    const float* x[4];  // piece lane % 8 of positions 8 j + lane / 8
#pragma unroll
    for (int j = 0; j < 4; ++j)
        x[j] = a.x + static_cast<int64_t>(min(p0 + 8 * j + (lane >> 3), a.positions - 1)) * a.blocks * 32 + 4 * (lane & 7);
    float* mine = lds + wave * (32 * kFlaggedStride);
    struct Block {
        u32x4 x[4];
        uint32_t raw[4];
        uint32_t scale;
    };
    auto load = [&](int b, Block& o) {
        b = min(b, a.blocks - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.x[j] = load16_a4(reinterpret_cast<const uint8_t*>(x[j] + 32 * b));
        if constexpr (FORMAT == kQ8_0) {
            const u32x4 v = load16_a4(a.w + (record + static_cast<uint32_t>(b) * kRecord));
#pragma unroll
            for (int e = 0; e < 4; ++e) o.raw[e] = v[e];
        } else {
            const uint64_t v = load8_a8(a.w + (record + static_cast<uint32_t>(b) * kRecord));
            o.raw[0] = static_cast<uint32_t>(v);
            o.raw[1] = static_cast<uint32_t>(v >> 32);
        }
        o.scale = load2_a2(scales + (first + b) * 2u);
    };
    auto wave_sync = [] {  // LDS written by lanes of this wave, read by others of it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    float acc[16] = {};
    Block now;
    load(wave, now);
    for (int b = wave; b < a.blocks; b += kWaves) {
        const bool small_too = any_small(now.x);
        wave_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<u32x4*>(mine + (8 * j + (lane >> 3)) * kFlaggedStride + 4 * (lane & 7)) = now.x[j];
        wave_sync();
        float v[2][8];
        u32x4 codes[2];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const f32x4 q = *reinterpret_cast<const f32x4*>(mine + (lane & 31) * kFlaggedStride +
                                                                slot_column<FORMAT>(st, h) + e);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[st][e + i] = q[i];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) codes[st][k] = code_pair<FORMAT>(now.raw, 4 * st + k);
        }
        const float scale = half_bits_to_float(now.scale);
        load(b + kWaves, now);
        // The sums of the block's smaller or larger elements, scaled and added up.
        auto add = [&](auto small) {
            f32x16 d = {};
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                u32x4 part[3];
                split8_unlifted<FORMAT, decltype(small)::value>(v[st], part);
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    d = mfma_bf16(__builtin_bit_cast(bf16x8, part[s]), __builtin_bit_cast(bf16x8, codes[st]), d);
                __builtin_amdgcn_sched_barrier(0);  // (one step's parts at a time: 128 registers, none spilled)
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float sum =
                    decltype(small)::value ? __builtin_amdgcn_ldexpf(d[i], -kLiftExponent - (FORMAT == kQ4_0 ? 4 : 0)) : d[i];
                acc[i] = __fadd_rn(acc[i], __fmul_rn(scale, sum));
            }
        };
        add(std::false_type{});
        if (small_too) add(std::true_type{});
    }
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) {
        if (wave == w) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (w > 0) acc[i] = __fadd_rn(lds[64 * i + lane], acc[i]);
                if (w + 1 < kWaves) lds[64 * i + lane] = acc[i];
            }
        }
        __syncthreads();
    }
    if (wave != kWaves - 1 || row >= a.rows) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int at = 8 * (i >> 2) + 4 * h + (i & 3), p = p0 + at;
        if (p < a.positions && (mask >> at & 1u)) store_f32(a.y + static_cast<int64_t>(p) * a.rows + row, acc[i]);
    }
}

// What bounds it: the matrix cores at many positions (6 MFMAs of 32 cycles per 32 x 32 tile and block), then the
// staged activations' way from L2 (a 128-row tile reads 6 KB of parts per 32 positions and block); at few
// positions the weights from HBM. A wave's 64-row x 64-position tile reuses each LDS read of the parts for two row
// tiles and each converted code for two position tiles, so that neither the LDS (3.5 KB a tile and block) nor
// the vector ALU (16 FMAs and 12-15 conversions) is ahead of the matrix cores.
// Ranges are dealt so that consecutive ones, which share rows of weights, run on one XCD (workgroup ids go
// round-robin over the eight).
template <int FORMAT, int TP, bool FUSED, int RH, int WAYS>
__global__ __launch_bounds__(64 * RH * WAYS, 2) void fbatch_kernel(FbatchArgs a) {
    constexpr int kThreads = 64 * RH * WAYS, kGroupRows = 64 * RH;
    static_assert(FUSED ? 2 * TP % RH == 0 : WAYS == 2, "staging passes");
    constexpr int kAhead = FUSED && TP == 1 ? 2 : 1;  // rounds in registers on their way into the LDS
    constexpr int kRecord = FORMAT == kQ8_0 ? 32 : 16;
    constexpr int kPieces = FORMAT == kQ8_0 ? 2 : 1;                 // 16-byte pieces of a record
    constexpr int kPlane = kGroupRows * 16 + 16;                     // one piece of every row, padded off its banks
    constexpr int kUnitBytes = TP * kBlockTileBytes;
    constexpr int kXBytes = WAYS * kUnitBytes;
    constexpr int kRoundBytes = kXBytes + WAYS * kPieces * kPlane;
    constexpr int kSlots = 2 * TP / RH;                              // fused form: operand slots per thread
    constexpr int kScaleRounds = 8 / WAYS;                           // rounds whose scales are staged together
    constexpr int kXLoads = kXBytes / 16 / kThreads;                 // packed form: pieces per thread
    __shared__ __align__(16) uint8_t lds[2 * kRoundBytes];
    __shared__ __align__(16) uint8_t lds_scales[2 * kGroupRows * 16];
    __shared__ uint32_t lds_flags[TP];

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int rh = (tid >> 6) % RH, way = (tid >> 6) / RH;
    const int per_xcd = a.workgroups >> 3;
    const int range = (a.workgroups & 7) == 0 ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
    const int end = range_start(a, range + 1);
    const int blocks = a.blocks;
    const uint8_t* scales = a.w + static_cast<int64_t>(a.rows) * blocks * kRecord;

    for (int at = range_start(a, range); at < end;) {
        const int tile = at / a.rounds, r0 = at - tile * a.rounds, r1 = min(a.rounds, r0 + (end - at));
        const int group = tile / a.units, t0 = (tile - group * a.units) * TP;  // row group, first position tile
        const int row0 = group * kGroupRows;

        // ---- staging: this thread's pieces of a round (WAYS blocks from WAYS r on; a block past the last reads the last
        // again, and is not computed). Addresses are a uniform base per round and a fixed 32-bit offset (a
        // payload is at most 2^31 - 1 bytes). ----
        u32x4 wregs[kAhead][kPieces];
        uint32_t woff[kPieces];
        constexpr int kRowPieces = WAYS * kPieces;  // of one row in a round: consecutive bytes
        const int wblk = tid % kRowPieces / kPieces;
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
            woff[j] = static_cast<uint32_t>(min(row0 + (tid + kThreads * j) / kRowPieces, a.rows - 1)) * blocks * kRecord +
                      16 * (tid % kRowPieces);
        const int wdst = kXBytes + tid % kRowPieces * kPlane + tid / kRowPieces * 16;
        u32x4 xregs[kAhead][FUSED ? 2 * kSlots : kXLoads];
        bool flagged[TP] = {};
        const uint8_t* xsrc[TP];
        if constexpr (FUSED) {  // slots (position tile, block, K step (tid / 64) % 2, lane), the threads' passes in that order
#pragma unroll
            for (int j = 0; j < TP; ++j)
                xsrc[j] = reinterpret_cast<const uint8_t*>(
                    a.x + static_cast<int64_t>(min((t0 + j) * kTile + (lane & 31), a.positions - 1)) * blocks * 32 +
                    slot_column<FORMAT>((tid >> 6) & 1, h));
        }
        auto slot_tile = [](int j) { return j * kThreads / 128 / WAYS; };
        auto slot_block = [&](int j) { return (tid >> 7) + j * kThreads / 128 % WAYS; };
        auto load_round = [&](int r, u32x4 (&wreg)[kPieces], u32x4 (&xreg)[FUSED ? 2 * kSlots : kXLoads]) {
            const int last = blocks - 1 - WAYS * r;  // the round's last block
            const uint8_t* wbase = a.w + static_cast<int64_t>(WAYS * r) * kRecord;
            const uint32_t back = static_cast<uint32_t>(wblk - min(wblk, last)) * kRecord;
#pragma unroll
            for (int j = 0; j < kPieces; ++j) wreg[j] = *(const SATORI_GLOBAL u32x4*)(wbase + (woff[j] - back));
            if constexpr (FUSED) {
#pragma unroll
                for (int j = 0; j < kSlots; ++j) {
                    const int64_t b = WAYS * r + min(slot_block(j), last);
                    xreg[2 * j] = load16_a4(xsrc[slot_tile(j)] + b * 128);
                    xreg[2 * j + 1] = load16_a4(xsrc[slot_tile(j)] + b * 128 + 16);
                }
            } else {
                // The unit's position tiles of a block are adjacent: piece c of the round is byte 16 (c % pieces) of
                // block c / pieces.
                constexpr int kPiecesX = kUnitBytes / 16;
                const uint32_t stride = static_cast<uint32_t>(a.units) * kUnitBytes, second = last > 0 ? stride : 0u;
                const uint8_t* base = a.parts + static_cast<int64_t>(WAYS * r) * stride + (t0 / TP) * kUnitBytes;
#pragma unroll
                for (int j = 0; j < kXLoads; ++j) {
                    const int c = tid + kThreads * j;
                    xreg[j] = *(const SATORI_GLOBAL u32x4*)(base + (c < kPiecesX ? 16u * c : 16u * (c - kPiecesX) + second));
                }
            }
        };
        auto store_round = [&](uint8_t* buf, const u32x4 (&wreg)[kPieces], const u32x4 (&xreg)[FUSED ? 2 * kSlots : kXLoads]) {
#pragma unroll
            for (int j = 0; j < kPieces; ++j)
                *reinterpret_cast<u32x4*>(buf + wdst + j * (kThreads / kRowPieces) * 16) = wreg[j];
            if constexpr (FUSED) {
#pragma unroll
                for (int j = 0; j < kSlots; ++j) {
                    const int t = slot_tile(j);
                    float v[8];  // (positions past the last are the last one again: computed, never stored)
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(xreg[2 * j + (e >> 2)][e & 3]);
                    u32x4 part[3];
                    flagged[t] |= split8(v, part);
                    uint8_t* dst = buf + (slot_block(j) * TP + t) * kBlockTileBytes + ((tid >> 6) & 1) * kPartBytes + 16 * lane;
#pragma unroll
                    for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x4*>(dst + 2 * s * kPartBytes) = part[s];
                }
            } else {
#pragma unroll
                for (int j = 0; j < kXLoads; ++j) *reinterpret_cast<u32x4*>(buf + 16 * (tid + kThreads * j)) = xreg[j];
            }
        };
        // The rows' scales of eight blocks (kScaleRounds rounds) at a time, 16 bytes a row (2-byte aligned; up to 14 bytes
        // past the last row's end, inside the payload's slack): one line read per row and eight blocks, where two bytes a
        // lane and round took half of the kernel's L2 requests.
        u32x4 sreg;
        const uint8_t* ssrc = scales + static_cast<uint32_t>(min(row0 + tid % kGroupRows, a.rows - 1)) * blocks * 2u;
        auto load_scales = [&](int g) { sreg = *(const SATORI_GLOBAL u32x4_a2*)(ssrc + 16 * min(g, (blocks - 1) >> 3)); };
        auto store_scales = [&](int g) {
            if (tid < kGroupRows) *reinterpret_cast<u32x4*>(lds_scales + ((g & 1) * kGroupRows + tid) * 16) = sreg;
        };

        // ---- rounds: computed from one LDS buffer while the next round is stored into the other and the one after
        // it is on its way into registers ----
        float acc[2][TP][16];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[rt][tp][i] = 0.0f;
        load_scales(r0 / kScaleRounds);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (r0 + u < r1) load_round(r0 + u, wregs[u], xregs[u]);
        store_scales(r0 / kScaleRounds);
        store_round(lds, wregs[0], xregs[0]);
        load_scales(r0 / kScaleRounds + 1);
        if (r0 + kAhead < r1) load_round(r0 + kAhead, wregs[0], xregs[0]);
        for (int base = r0; base < r1; base += kAhead)
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {  // round r + 1 waits in register set (u + 1) % kAhead
            const int r = base + u;
            if (r >= r1) break;
            uint8_t* cur = lds + ((r - r0) & 1) * kRoundBytes;
            uint8_t* other = lds + ((r - r0 + 1) & 1) * kRoundBytes;
            __syncthreads();  // round r staged; the other buffer is no longer read
            // This way's operands of its block, requested before the staging so that they arrive behind it.
            const bool live = WAYS * r + way < blocks;  // (a way without a block only takes part in the staging)
            const uint8_t* xcur = cur + way * kUnitBytes + 16 * lane;
            float scale[2];
            uint32_t raw[2][4];
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const int row = 64 * rh + 32 * rt + (lane & 31);
                scale[rt] = half_bits_to_float(*reinterpret_cast<const uint16_t*>(
                    lds_scales + ((r / kScaleRounds & 1) * kGroupRows + row) * 16 + 2 * (r % kScaleRounds * WAYS + way)));
                if (FORMAT == kQ4_0) scale[rt] *= 0.0625f;  // (codes 16 q)
                if constexpr (FORMAT == kQ8_0) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(cur + kXBytes + (2 * way + h) * kPlane + 16 * row);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[rt][e] = v[e];
                } else {
                    const uint2 v = *reinterpret_cast<const uint2*>(cur + kXBytes + way * kPlane + 16 * row + 8 * h);
                    raw[rt][0] = v.x;
                    raw[rt][1] = v.y;
                }
            }
            bf16x8 xa[6];
#pragma unroll
            for (int s = 0; s < 6; ++s) xa[s] = *reinterpret_cast<const bf16x8*>(xcur + s * kPartBytes);
            if (r + 1 < r1) {
                if ((r + 1) % kScaleRounds == 0) {
                    store_scales((r + 1) / kScaleRounds);
                    load_scales((r + 1) / kScaleRounds + 1);
                }
                store_round(other, wregs[(u + 1) % kAhead], xregs[(u + 1) % kAhead]);
            }
            if (r + 1 + kAhead < r1) load_round(r + 1 + kAhead, wregs[(u + 1) % kAhead], xregs[(u + 1) % kAhead]);
            if (!live) continue;  // (its barrier is the next round's: every wave takes the same number)
            __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
            // One product chain per (row tile, position tile). Each step issues one MFMA and, in its shadow, part of
            // the vector work beside it: the second row tile's conversions under the first chain, then the
            // previous tile's FMAs; each position tile's parts are read while the last chain on the one before
            // runs. (Left to the compiler, the conversions and FMAs ran between the chains: MFMA and vector
            // time added up: the loop without its staging took 58 us at 11008 x 4096 Q4_0 over 256 positions, 44 at the
            // rate a loop of MFMAs with as many vector instructions beside them reaches.)
            u32x4 wop[2][2];
#pragma unroll
            for (int k = 0; k < 8; ++k) wop[0][k >> 2][k & 3] = code_pair<FORMAT>(raw[0], k);
            f32x16 prev;
#pragma unroll
            for (int k = 0; k < 2 * TP; ++k) {
                const int rt = k & 1, tp = k >> 1;
                f32x16 d = {};
#pragma unroll
                for (int s = 0; s < 6; ++s) {
                    d = mfma_bf16(xa[s], __builtin_bit_cast(bf16x8, wop[rt][s & 1]), d);
                    if (k == 0) {
                        if (s < 4) {
                            wop[1][s >> 1][2 * s & 3] = code_pair<FORMAT>(raw[1], 2 * s);
                            wop[1][s >> 1][2 * s + 1 & 3] = code_pair<FORMAT>(raw[1], 2 * s + 1);
                        }
                    } else {
#pragma unroll
                        for (int i = s < 1 ? 0 : 3 * s - 2 - (s == 1); i < (s < 1 ? 0 : 3 * s + 1); ++i)
                            acc[rt ^ 1][(k - 1) >> 1][i] = __builtin_fmaf(scale[rt ^ 1], prev[i], acc[rt ^ 1][(k - 1) >> 1][i]);
                    }
                    if (rt == 1 && tp + 1 < TP)
                        xa[s] = *reinterpret_cast<const bf16x8*>(xcur + (tp + 1) * kBlockTileBytes + s * kPartBytes);
                    __builtin_amdgcn_sched_barrier(0);
                }
                prev = d;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[1][TP - 1][i] = __builtin_fmaf(scale[1], prev[i], acc[1][TP - 1][i]);
        }

        // ---- the tile's sums: the ways' are added pairwise, then stored, or left as a partial.
        // Four outputs (positions p .. p + 3 of a lane's row) are adjacent in the LDS and in a partial. ----
        if (FUSED && tid < TP) lds_flags[tid] = 0u;
        __syncthreads();
        f32x4* sums = reinterpret_cast<f32x4*>(lds);
        auto quad_at = [&](int rt, int tp, int q) { return (((rh * 2 + rt) * TP + tp) * 4 + q) * 64 + lane; };
        if (way > 0)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        sums[(way - 1) * (slot_floats(TP, RH) / 4) + quad_at(rt, tp, q)] =
                            f32x4{acc[rt][tp][4 * q], acc[rt][tp][4 * q + 1], acc[rt][tp][4 * q + 2], acc[rt][tp][4 * q + 3]};
        if constexpr (FUSED) {
#pragma unroll
            for (int j = 0; j < TP; ++j) {
                const uint64_t f = __ballot(flagged[j]);
                const uint32_t word = static_cast<uint32_t>(f) | static_cast<uint32_t>(f >> 32);
                if (lane == 0 && word) atomicOr(&lds_flags[j], word);
            }
        }
        __syncthreads();
        if (way == 0) {
            const bool whole = r0 == 0 && r1 == a.rounds;
            const int slot = 2 * range + (r0 == 0 ? 1 : 0);  // the range's first segment, or its last
            f32x4* out = reinterpret_cast<f32x4*>(a.partial + static_cast<int64_t>(slot) * slot_floats(TP, RH));
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const int row = row0 + 64 * rh + 32 * rt + (lane & 31);
#pragma unroll
                for (int tp = 0; tp < TP; ++tp)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        f32x4 o[WAYS];
                        o[0] = f32x4{acc[rt][tp][4 * q], acc[rt][tp][4 * q + 1], acc[rt][tp][4 * q + 2], acc[rt][tp][4 * q + 3]};
#pragma unroll
                        for (int w = 1; w < WAYS; ++w) o[w] = sums[(w - 1) * (slot_floats(TP, RH) / 4) + quad_at(rt, tp, q)];
#pragma unroll
                        for (int n = WAYS / 2; n > 0; n /= 2)
#pragma unroll
                            for (int w = 0; w < n; ++w)
#pragma unroll
                                for (int e = 0; e < 4; ++e) o[w][e] = __fadd_rn(o[w][e], o[w + n][e]);
                        const f32x4 v = o[0];
                        if (!whole) {
                            out[quad_at(rt, tp, q)] = v;
                            continue;
                        }
                        const int p = (t0 + tp) * kTile + 8 * q + 4 * h;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (row < a.rows && p + e < a.positions)
                                store_f32(a.y + static_cast<int64_t>(p + e) * a.rows + row,
                                          __builtin_amdgcn_ldexpf(v[e], -kLiftExponent));
                    }
            }
            if (FUSED && tid < TP) (whole ? a.tile_flags + tile * TP : a.slot_flags + slot * TP)[tid] = lds_flags[tid];
        }
        __syncthreads();  // the sums and flags are read
        at += r1 - r0;
    }
}

// Short rows under many outputs: a workgroup is one tile of 128 rows x 32 positions, W blocks a round, with as many of them
// on a CU as fit, so that one's loads and stores pass behind another's products. (What bounds fbatch_kernel there is its
// chain: a tile has one to nine rounds, and one workgroup a CU waits for each tile's first loads, 2.4 us a round in all.
// A product of three tiles a workgroup, 13771 x 288 Q8_0 over 224 positions, took it 25.7 us, 16.4 with tiles four times as
// large, 14.0 here.) Wave
// (way, row tile) multiplies block W k + way of round k for 32 rows; the split activations of a round go through the LDS,
// double-buffered, the weights straight into registers, both requested two rounds ahead. The ways' sums are added in order.
template <int FORMAT, int W>
__global__ __launch_bounds__(256 * W) void fbatch_tiles_kernel(FbatchArgs a) {
    constexpr int kRecord = FORMAT == kQ8_0 ? 32 : 16;
    constexpr int kThreads = 256 * W, kRoundBytes = W * kBlockTileBytes, kPieces = kRoundBytes / 16;
    constexpr int kLoads = (kPieces + kThreads - 1) / kThreads, kSumBytes = (W - 1) * 4 * 64 * 16 * 4;
    __shared__ __align__(16) uint8_t lds[2 * kRoundBytes > kSumBytes ? 2 * kRoundBytes : kSumBytes];
    const int per_xcd = gridDim.x >> 3;
    const int u = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (u >= a.total) return;  // whole workgroup
    const int group = u / a.tiles, t = u - group * a.tiles;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, rt = (tid >> 6) & 3, way = tid >> 8;
    const int row = group * 128 + 32 * rt + (lane & 31), blocks = a.blocks, rounds = a.rounds;
    const uint32_t first = static_cast<uint32_t>(min(row, a.rows - 1)) * blocks;  // (a payload has at most 2^31 - 1 bytes)
    const uint32_t record = first * kRecord + (FORMAT == kQ8_0 ? 16 : 8) * h;
    const uint8_t* scales = a.w + static_cast<int64_t>(a.rows) * blocks * kRecord;
    const uint8_t* parts = a.parts + static_cast<int64_t>(t) * kBlockTileBytes;
    const int64_t stride = static_cast<int64_t>(a.tiles) * kBlockTileBytes;

    struct Weights {
        uint32_t raw[4];
        uint32_t scale;
    };
    auto load_weights = [&](int r, Weights& o) {  // (a block past the last reads the last, and is not computed)
        const uint32_t b = min(W * r + way, blocks - 1);
        if constexpr (FORMAT == kQ8_0) {
            const u32x4 v = load16_a4(a.w + (record + b * kRecord));
#pragma unroll
            for (int e = 0; e < 4; ++e) o.raw[e] = v[e];
        } else {
            const uint64_t v = load8_a8(a.w + (record + b * kRecord));
            o.raw[0] = static_cast<uint32_t>(v);
            o.raw[1] = static_cast<uint32_t>(v >> 32);
        }
        o.scale = load2_a2(scales + (first + b) * 2u);
    };
    u32x4 staged[kLoads];
    auto load_parts = [&](int r) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int c = min(tid + kThreads * j, kPieces - 1), b = min(W * r + c / 384, blocks - 1);
            staged[j] = *(const SATORI_GLOBAL u32x4*)(parts + b * stride + 16 * (c % 384));
        }
    };
    auto store_parts = [&](int r) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j)
            if (tid + kThreads * j < kPieces)
                *reinterpret_cast<u32x4*>(lds + (r & 1) * kRoundBytes + 16 * (tid + kThreads * j)) = staged[j];
    };

    float acc[16] = {};
    Weights w[2];
    load_parts(0);
    load_weights(0, w[0]);
    load_weights(1, w[1]);
    store_parts(0);
    load_parts(1);
    __syncthreads();  // round 0 staged
    for (int r0 = 0; r0 < rounds; r0 += 2)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int r = r0 + n;
            if (r >= rounds) break;
            const uint8_t* mine = lds + n * kRoundBytes + way * kBlockTileBytes + 16 * lane;
            if (W * r + way < blocks) {
                float scale = half_bits_to_float(w[n].scale);
                if (FORMAT == kQ4_0) scale *= 0.0625f;  // (codes 16 q)
                f32x16 d = {};
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    u32x4 codes;
#pragma unroll
                    for (int k = 0; k < 4; ++k) codes[k] = code_pair<FORMAT>(w[n].raw, 4 * st + k);
#pragma unroll
                    for (int s = 0; s < 3; ++s)
                        d = mfma_bf16(*reinterpret_cast<const bf16x8*>(mine + (2 * s + st) * kPartBytes),
                                      __builtin_bit_cast(bf16x8, codes), d);
                }
                load_weights(r + 2, w[n]);
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(scale, d[i], acc[i]);
            }
            if (r + 1 < rounds) {
                store_parts(r + 1);
                load_parts(r + 2);
            }
            __syncthreads();  // round r + 1 staged, round r's buffer read
        }
    if constexpr (W > 1) {
        f32x4* sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (way > 0)
                sums[(((way - 1) * 4 + rt) * 4 + q) * 64 + lane] = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        __syncthreads();
        if (way > 0) return;
#pragma unroll
        for (int n = 1; n < W; ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 v = sums[(((n - 1) * 4 + rt) * 4 + q) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[4 * q + e] = __fadd_rn(acc[4 * q + e], v[e]);
            }
    }
    if (row >= a.rows) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int p = t * kTile + 8 * (i >> 2) + 4 * h + (i & 3);
        if (p < a.positions) store_f32(a.y + static_cast<int64_t>(p) * a.rows + row, __builtin_amdgcn_ldexpf(acc[i], -kLiftExponent));
    }
}

// The flagged positions of fbatch_tiles_kernel's product, over what it stored there: every workgroup looks at all flags and,
// where there are any, computes its share of the 32 x 32 tiles that hold some.
template <int FORMAT>
__global__ __launch_bounds__(kThreads) void fbatch_flagged_kernel(FbatchArgs a) {
    __shared__ uint32_t flagged[8];  // (256 positions at most)
    __shared__ __align__(16) float lds[4 * 32 * kFlaggedStride];
    if (threadIdx.x < 8) flagged[threadIdx.x] = 0u;
    __syncthreads();
    bool any = false;
    for (int i = threadIdx.x; i < 2 * a.blocks * a.tiles; i += kThreads) {
        const uint32_t word = a.flags[i];
        if (word) atomicOr(&flagged[(i >> 1) % a.tiles], word);
        any |= word != 0u;
    }
    if (!__syncthreads_or(any)) return;
    const int row_tiles = (a.rows + kTile - 1) / kTile;
    for (int u = blockIdx.x; u < row_tiles * a.tiles; u += gridDim.x) {
        const int t = u % a.tiles;
        if (flagged[t]) finish_flagged<FORMAT, 1>(a, u / a.tiles * kTile, t * kTile, flagged[t], lds);
    }
}

// One workgroup per 32 x 32 tile of every (row group, position unit) tile: adds the pieces of a cut tile and computes
// the flagged positions of any tile. Thread (g, wave q, lane) adds pieces g, g + G, ... of outputs 4q .. 4q + 3 of its
// lane, four chains at a time, then the chains and the G sums in a fixed order: with many pieces (a few rows of many
// columns) a single chain of their loads took longer than the product (256 x 14336 Q8_0 over 8 positions: 21.9 us
// against 13.3) and rounded more. The flags are requested beside the pieces: finish_flagged's registers leave four
// workgroups a CU, whose round trips count (requested after the pieces' sums: 11008 x 4096 Q4_0 over 256 positions 86.2
// us against 83.4, 4096 x 4096 Q8_0 over 12 13.5 against 13.2).
template <int FORMAT, int TP, bool FUSED, int RH, int G>
__global__ __launch_bounds__(kThreads * G, 4) void fbatch_fixup_kernel(FbatchArgs a) {
    constexpr int kGroupRows = 64 * RH, kSubs = 2 * RH * TP, kWaves = 4 * G;
    __shared__ uint32_t lds_flags[kWaves];
    __shared__ __align__(16) float lds[kWaves * 32 * kFlaggedStride];
    f32x4* lds_sums = reinterpret_cast<f32x4*>(lds);  // (G - 1 sums a thread, read before finish_flagged)
    static_assert((G - 1) * kThreads * sizeof(f32x4) <= sizeof(lds) && kTile * kTile * sizeof(float) <= sizeof(lds));
    const int tile = blockIdx.x / kSubs, sub = blockIdx.x - tile * kSubs;  // sub = (2 rh + rt) * TP + tp
    const int first = range_of(a, tile * a.rounds), last = range_of(a, (tile + 1) * a.rounds - 1);
    const int tid = threadIdx.x % kThreads, g = threadIdx.x / kThreads, q = tid >> 6, lane = tid & 63, h = lane >> 5;
    const int group = tile / a.units, tp = sub % TP, t = (tile - group * a.units) * TP + tp;
    const int row0 = group * kGroupRows + 32 * (sub / TP);
    const int row = row0 + (lane & 31);
    const bool cut = first != last;
    // The piece that starts the tile is its range's last segment, the others their range's first.
    auto slot_of = [&](int i) { return 2 * i + (i == first ? 1 : 0); };
    uint32_t word = 0u;
    if constexpr (FUSED) {
        if (!cut)
            word = a.tile_flags[tile * TP + tp];
        else
            for (int i = first + threadIdx.x; i <= last; i += kThreads * G) word |= a.slot_flags[slot_of(i) * TP + tp];
    } else {
        for (int i = threadIdx.x; i < 2 * a.blocks; i += kThreads * G)
            word |= a.flags[2 * (static_cast<int64_t>(i >> 1) * a.tiles + t) + (i & 1)];
    }
    f32x4 sum[4] = {};  // one chain per piece in flight
    if (cut)
        for (int i0 = first + g; i0 <= last; i0 += 4 * G) {  // four pieces' loads in flight
            f32x4 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = *(const SATORI_GLOBAL f32x4*)(a.partial + static_cast<int64_t>(slot_of(min(i0 + j * G, last))) * slot_floats(TP, RH) +
                                                     ((sub * 4 + q) * 64 + lane) * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i0 + j * G <= last)
#pragma unroll
                    for (int k = 0; k < 4; ++k) sum[j][k] = __fadd_rn(sum[j][k], v[j][k]);
        }
    f32x4 acc;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = __fadd_rn(__fadd_rn(sum[0][k], sum[1][k]), __fadd_rn(sum[2][k], sum[3][k]));
    if (G > 1 && g > 0) lds_sums[(g - 1) * kThreads + tid] = acc;
    if (__ballot(word != 0u))
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) word |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(word), o, 64));
    if (lane == 0) lds_flags[threadIdx.x >> 6] = word;
    __syncthreads();
    uint32_t flagged = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) flagged |= lds_flags[w];
    if (cut && g == 0) {
#pragma unroll
        for (int j = 0; j < G - 1; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = __fadd_rn(acc[k], lds_sums[j * kThreads + tid][k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = 8 * q + 4 * h + k, p = t * kTile + i;
            if (row < a.rows && p < a.positions && !((flagged >> i) & 1u))
                store_f32(a.y + static_cast<int64_t>(p) * a.rows + row, __builtin_amdgcn_ldexpf(acc[k], -kLiftExponent));
        }
    }
    if (flagged) {  // whole workgroup
        __syncthreads();  // the sums are read
        finish_flagged<FORMAT, G>(a, row0, t * kTile, flagged, lds);
    }
}

// How a launch is cut, for the device's CU count.
struct FbatchPlan {
    int TP, RH, ways;
    bool fused, whole;  // whole: fbatch_tiles_kernel
    int tiles, units, rounds, total, workgroups;
    size_t parts;                                                           // bytes of the split activations
    size_t slot_flags_offset, tile_flags_offset, flags_offset, scratch;     // (the partial sums first)
};

// Short rows under many outputs go to fbatch_tiles_kernel: it needs a workgroup for half of the CUs at least, and past 36
// blocks an even deal and more rows a workgroup are worth more. Measured over 60 shapes at 14 counts of 33 to 256 positions
// (us, fbatch_kernel against this): 13771 x 288 at 224 29.7 and 16.3, 9132 x 160 at 256 21.5 and 13.2, 7429 x 1120 at 128
// Q4_0 24.7 and 20.9, 3798 x 576 at 256 20.7 and 15.0, but 7227 x 1760 at 64 23.2 and 24.8, 1772 x 8000 at 64 22 and 90,
// 372 x 192 at 110 8.2 and 9.6.
bool whole_tiles(int rows, int blocks, int tiles) {
    return tiles > 1 && blocks <= 36 && static_cast<int64_t>((rows + 127) / 128) * tiles >= 128;
}

FbatchPlan fbatch_plan(int rows, int columns, int positions, int cus) {
    FbatchPlan p{};
    const int blocks = columns / 32;
    p.tiles = (positions + kTile - 1) / kTile;
    // Activations converted by each workgroup for itself (fused) while that costs less than the pack launch and its
    // bytes: measured (us, fused against packed) 256 x 14336 Q8_0 at 90 positions 17.8 against 24.2, 4096 x 1024 at 132
    // 19.6 against 22.5, 4096 x 4096 at 132 36.0 against 37.2, 11008 x 1024 at 256 40.7 against 36.4. One position tile a
    // unit (the weights read and converted once per tile, but twice the units to spread) for small products, and longer
    // where two a unit would leave half a unit empty: 512 x 512 at 256 9.1 against 10.7, 608 x 9024 at 64 15.9 against
    // 19.5, 2572 x 576 at 256 16.2 against 19.4, 4096 x 4096 at 64 19.2 against 18.9, 4580 x 1120 at 256 28.2 against 25.9,
    // 9880 x 1984 at 82 29.1 against 31.8.
    const int64_t products = static_cast<int64_t>(rows) * columns * positions;
    p.TP = products < 400000000 || (p.tiles % 2 == 1 && products < 1800000000) || p.tiles == 1 ? 1 : 2;
    p.fused = p.tiles <= 2 || products < 2300000000;
    p.RH = p.fused ? 2 : 4;
    p.ways = 8 / p.RH;
    if (whole_tiles(rows, blocks, p.tiles)) {
        const int64_t n = static_cast<int64_t>((rows + 127) / 128) * p.tiles;
        p.whole = true;
        p.fused = false;
        p.TP = 1;
        p.RH = 2;
        // As many ways as keep every workgroup on the chip at once (two of 16 waves a CU, four of eight or eight of four).
        p.ways = n <= 2 * cus ? 4 : n <= 4 * cus ? 2 : 1;
        p.units = p.tiles;
        p.rounds = (blocks + p.ways - 1) / p.ways;
        p.total = static_cast<int>(n);
        p.parts = static_cast<size_t>(blocks) * p.tiles * kBlockTileBytes;
        p.workgroups = static_cast<int>(std::min<int64_t>(cus, 4 * n));  // of fbatch_flagged_kernel
        p.scratch = static_cast<size_t>(blocks) * p.tiles * 8;           // (flags_offset 0)
        return p;
    }
    p.units = (p.tiles + p.TP - 1) / p.TP;
    p.tiles = p.units * p.TP;  // whole units: the packed form's last tile may be all zero
    p.rounds = (blocks + p.ways - 1) / p.ways;
    // (Below 2^31 for every payload of at most 2^31 - 1 bytes: a round of a tile is 64 columns of 128 rows or more.)
    p.total = (rows + 64 * p.RH - 1) / (64 * p.RH) * p.units * p.rounds;
    int n = std::min(p.total, cus);  // one workgroup of eight waves per CU
    if (n >= 8) n -= n % 8;
    p.workgroups = n;
    p.parts = p.fused ? 0 : static_cast<size_t>(blocks) * p.tiles * kBlockTileBytes;
    p.slot_flags_offset = static_cast<size_t>(p.workgroups) * 2 * slot_floats(p.TP, p.RH) * sizeof(float);
    p.tile_flags_offset = p.slot_flags_offset + static_cast<size_t>(p.workgroups) * 2 * p.TP * 4;
    p.flags_offset = p.tile_flags_offset + static_cast<size_t>(p.total / p.rounds) * p.TP * 4;
    p.scratch = p.flags_offset + (p.fused ? 0 : static_cast<size_t>(blocks) * p.tiles * 8);
    return p;
}

int device_cus() {
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0)
        return 256;
    return cus;
}

template <int FORMAT, int TP, bool FUSED, int RH, int WAYS>
hipError_t launch_product(const FbatchArgs& a, hipStream_t stream) {
    fbatch_kernel<FORMAT, TP, FUSED, RH, WAYS><<<static_cast<unsigned>(a.workgroups), 64 * RH * WAYS, 0, stream>>>(a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const unsigned grid = static_cast<unsigned>(a.total / a.rounds) * 2 * RH * TP;
    if (a.rounds > 4 * a.share)  // more than about five pieces a tile
        fbatch_fixup_kernel<FORMAT, TP, FUSED, RH, 4><<<grid, 4 * kThreads, 0, stream>>>(a);
    else
        fbatch_fixup_kernel<FORMAT, TP, FUSED, RH, 1><<<grid, kThreads, 0, stream>>>(a);
    return hipGetLastError();
}

template <int FORMAT>
hipError_t launch_format(FbatchArgs a, const FbatchPlan& p, uint8_t* parts, uint32_t* flags, hipStream_t stream) {
    if (p.fused) return p.TP == 1 ? launch_product<FORMAT, 1, true, 2, 4>(a, stream) : launch_product<FORMAT, 2, true, 2, 4>(a, stream);
    const int64_t items = static_cast<int64_t>(a.blocks) * p.tiles * 128;
    if ((items + kThreads - 1) / kThreads > INT32_MAX) return hipErrorInvalidValue;
    fbatch_pack_kernel<FORMAT><<<static_cast<unsigned>((items + kThreads - 1) / kThreads), kThreads, 0, stream>>>(
        a.x, a.blocks * 32, a.positions, p.tiles, parts, flags);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    a.parts = parts;
    a.flags = flags;
    if (!p.whole) return launch_product<FORMAT, 2, false, 4, 2>(a, stream);
    const unsigned grid = (static_cast<unsigned>(a.total) + 7) / 8 * 8;
    if (p.ways == 4)
        fbatch_tiles_kernel<FORMAT, 4><<<grid, 1024, 0, stream>>>(a);
    else if (p.ways == 2)
        fbatch_tiles_kernel<FORMAT, 2><<<grid, 512, 0, stream>>>(a);
    else
        fbatch_tiles_kernel<FORMAT, 1><<<grid, 256, 0, stream>>>(a);
    const hipError_t launched = hipGetLastError();
    if (launched != hipSuccess) return launched;
    fbatch_flagged_kernel<FORMAT><<<static_cast<unsigned>(a.workgroups), kThreads, 0, stream>>>(a);
    return hipGetLastError();
}

}  // namespace

// From 32 positions on always; below, where the weights the single-position kernel would read again outweigh the second
// launch and, a row, its share of the partial sums; Q4_0, whose weights are half as many bytes, from 1.1 of that. Measured
// against that kernel over 90 shapes at 11 counts of 4 to 31 positions (us, FP32 activations, this against that kernel):
// Q8_0 4096 x 4096 14.2 and 10.4 at 4, 14.0 and 26.1 at 12; 8175 x 2176 16.0 and 12.6 at 6, 16.3 and 18.2 at 12; 10460 x
// 736 13.2 and 9.8 at 12; 4096 x 1024 10.4 and 9.1 at 20; Q4_0 11008 x 4096 22.5 and 21.5 at 4, 22.6 and 36.6 at 8; 1135 x
// 3808 11.6 and 8.5 at 8, 11.7 and 12.3 at 16. At 11 of those 1,980 calls the rule takes this product where the other
// kernel is more than 3% faster.
bool fbatch_pays(int format, int rows, int columns, int positions) {
    if (positions >= kTile) return true;
    const int64_t line = 60000000 + 4000 * static_cast<int64_t>(rows);
    return positions >= 4 &&
           static_cast<int64_t>(rows) * columns * (positions - 1) >= (format == kQ4_0 ? line + line / 10 : line);
}

// What a matrix holds for its batches: the split activations of any count of as many position tiles, and 256 bytes a tile
// so that it grows with the tiles in every form (a matrix's first call at a count of tiles leaves a buffer, without
// which that count may not be captured).
size_t fbatch_held_bytes(int rows, int columns, int positions) {
    const int tiles = (positions + kTile - 1) / kTile;
    return fbatch_plan(rows, columns, tiles * kTile, device_cus()).parts + static_cast<size_t>(tiles) * 256;
}

size_t fbatch_scratch_bytes(int rows, int columns, int positions) {
    // The largest of this and every smaller position count, so that a buffer made for one call serves the smaller
    // ones: the first and the last count of each number of tiles (between them the form changes at most from one of
    // the two to the other).
    const int cus = device_cus();
    size_t bytes = 0;
    for (int first = 1; first <= positions; first += kTile)
        for (int n : {first, std::min(positions, first + kTile - 1)})
            bytes = std::max(bytes, fbatch_plan(rows, columns, n, cus).scratch);
    return bytes;
}

hipError_t launch_gemv_fbatch(const uint8_t* w, int format, const float* x, uint8_t* parts, uint8_t* scratch, float* y,
                              int rows, int columns, int positions, hipStream_t stream) {
    if (rows <= 0 || positions <= 0 || columns <= 0) return hipSuccess;
    if ((format != kQ8_0 && format != kQ4_0) || columns % 32 != 0) return hipErrorInvalidValue;
    const FbatchPlan p = fbatch_plan(rows, columns, positions, device_cus());
    FbatchArgs a{};
    a.w = w;
    a.x = x;
    a.y = y;
    if (!p.fused && !parts) return hipErrorInvalidValue;
    a.partial = reinterpret_cast<float*>(scratch);
    a.slot_flags = reinterpret_cast<uint32_t*>(scratch + p.slot_flags_offset);
    a.tile_flags = reinterpret_cast<uint32_t*>(scratch + p.tile_flags_offset);
    uint32_t* flags = reinterpret_cast<uint32_t*>(scratch + p.flags_offset);
    a.rows = rows;
    a.blocks = columns / 32;
    a.positions = positions;
    a.tiles = p.tiles;
    a.units = p.units;
    a.rounds = p.rounds;
    a.total = p.total;
    a.workgroups = p.workgroups;
    a.share = p.total / p.workgroups;
    a.longer = p.total % p.workgroups;
    return format == kQ8_0 ? launch_format<kQ8_0>(a, p, parts, flags, stream)
                           : launch_format<kQ4_0>(a, p, parts, flags, stream);
}

}  // namespace satori
