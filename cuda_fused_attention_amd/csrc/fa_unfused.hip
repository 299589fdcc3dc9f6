// v0: the unfused attention baseline on gfx950 — three kernels with the fp32
// score matrix materialised in HBM, following the reference's algorithm
// (kernels/v0_unfused.cu:19-155): S = scale * Q.K^T with fp32 sums (masked
// entries -FLT_MAX), a stable row softmax in place, O = bf16(P.V) summed over
// every key. Any head_dim.
//
// What is MI355X-specific:
//   * both products run on the matrix cores, P V with P split into three bf16
//     parts, and S is written in 16-byte pieces of whole rows;
//   * softmax keeps a whole row in registers (up to 32768 columns), so S is
//     read once and written once — 16 B of HBM traffic per score in total
//     (write S, read S, write P, read P) against the reference's 5 passes.
// Algorithmic bytes per launch: 16*B*H*N^2 + 8*B*H*N*D (HBM roofline).

#include <atomic>
#include <cfloat>
#include <cstdint>

#include "fa_common.hpp"
#include "../../include/fa_mi355x.h"

namespace {

using fa::bf16x8;
using fa::f32x16;
using fa::f32x4;

// A buffer offset past the end of every buffer: a copy from there writes zeros.
constexpr uint32_t kNowhere = 0x80000000u;
// Largest head_dim whose tiles (up to 128 rows) keep 32-bit byte offsets below
// kNowhere; wider ones take the element-wise loads.
constexpr int kMaxCopyDim = 1 << 22;

// Four floats at any address a float may have: rows of an odd length put them
// at multiples of 4 bytes only.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// Keeps LDS accesses of one wave in program order for the compiler (the LDS
// serves one wave's accesses in order, so its lanes need no barrier to see
// each other's writes).
__device__ __forceinline__ void wave_lds_fence()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

constexpr int kTile = 64;      // edge of the smallest tile of scores (grid limits)
constexpr int kThreads = 256;  // four waves

// One MFMA operand of a Q, K or V row: bf16 columns [col, col + 8) of a row that
// exists, zero past the last column (cols % 8 == 0 and a 16-byte aligned base
// for kVec: the piece is then one 16-byte load, wholly inside or outside).
template <bool kVec>
__device__ __forceinline__ bf16x8 load_operand(const uint16_t* __restrict__ row, int col, int cols)
{
    if (kVec) return col < cols ? *reinterpret_cast<const bf16x8*>(row + col) : bf16x8{};
    bf16x8 r = {};
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (col + e < cols) r[e] = __builtin_bit_cast(__bf16, row[col + e]);
    return r;
}

// S[bh][q][k] = scale * sum_d Q[q][d] K[k][d]; causal k > q -> -FLT_MAX.
// Grid: (tiles, B*H), all tiles or, causal, those of the lower triangle: the
// others are not written, since the causal softmax and P V read no score of a
// key past the query (skipping them inside the whole grid left one XCD with 24
// live tiles of 17 on average at seq_len 2048). 256 threads: four waves in a 2 x 2
// arrangement, each with kBlocks x kBlocks blocks of 32 x 32 scores, so one
// workgroup writes a tile of 64 * kBlocks rows and columns.
//
// A product of two bf16 values is exact in fp32, so the matrix cores
// (v_mfma_f32_32x32x16_bf16, fp32 sums) compute what fp32 FMAs did. Those were
// bound by the vector unit: 110 us at (2,8,2048,64), 196 at head_dim 128. Now
// the write of S bounds the kernel: 60 us (4.5 TB/s) and 70 us. Q and K are
// copied to LDS without registers: staged through registers they cost 5 us more,
// and operand loads straight from global memory, which touch 32 rows per
// instruction, 13 us at head_dim 64 and 28 at 128.
template <bool kVec, int kBlocks>
__global__ __launch_bounds__(kThreads) void v0_scores_kernel(const uint16_t* __restrict__ q,
                                                              const uint16_t* __restrict__ k,
                                                              float* __restrict__ s, int n, int d,
                                                              int tiles_k, float scale, int causal)
{
    constexpr int kEdge = 64 * kBlocks;  // the workgroup's tile
    constexpr int kCols = 64;            // columns of Q and K staged at a time
    constexpr int kPieces = kCols / 8;   // 16-byte pieces of a staged row
    constexpr int kRowScores = 32 * kBlocks;  // scores of a row that one wave holds
    constexpr int kPitch = kRowScores + 4;    // floats of a row in the transposing buffer
    constexpr int kStageBytes = 2 * kEdge * kCols * 2;
    constexpr int kOutBytes = 4 * 32 * kPitch * 4;
    __shared__ __attribute__((aligned(16))) unsigned char lds[kStageBytes > kOutBytes ? kStageBytes : kOutBytes];
    uint16_t* const qs = reinterpret_cast<uint16_t*>(lds);
    uint16_t* const ks = qs + kEdge * kCols;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int i = lane & 31;
    const int h = lane >> 5;
    int tile_q = static_cast<int>(blockIdx.x) / tiles_k;
    int tile_k = static_cast<int>(blockIdx.x) % tiles_k;
    if (causal)
    {
        // Tile x of the lower triangle in row order: row r starts at r(r+1)/2.
        const unsigned x = blockIdx.x;
        unsigned r = static_cast<unsigned>((__builtin_sqrtf(8.0f * static_cast<float>(x) + 1.0f) - 1.0f) * 0.5f);
        while (r * (r + 1) / 2 > x) --r;
        while ((r + 1) * (r + 2) / 2 <= x) ++r;
        tile_q = __builtin_amdgcn_readfirstlane(static_cast<int>(r));
        tile_k = __builtin_amdgcn_readfirstlane(static_cast<int>(x - r * (r + 1) / 2));
    }
    const int tile_q0 = tile_q * kEdge;
    const int tile_k0 = tile_k * kEdge;
    const int wave_q = (wave >> 1) * 32 * kBlocks;  // the wave's first row in the tile
    const int wave_k = (wave & 1) * 32 * kBlocks;   // and column
    const int q0 = tile_q0 + wave_q;
    const int k0 = tile_k0 + wave_k;
    const size_t bh = blockIdx.y;
    const uint16_t* q_slab = q + bh * n * d;
    const uint16_t* k_slab = k + bh * n * d;
    float* const s_wave = s + bh * n * n + static_cast<size_t>(q0) * n + k0;

    f32x16 acc[kBlocks][kBlocks];
#pragma unroll
    for (int x = 0; x < kBlocks; ++x)
#pragma unroll
        for (int y = 0; y < kBlocks; ++y) acc[x][y] = f32x16{};

    // Piece c of staged row r lies at piece c ^ (r/2 % 8): the 16 rows that
    // one phase of an operand read touches then cover all banks.
    auto piece = [](int row, int c) { return row * kCols + ((c ^ ((row >> 1) & 7)) << 3); };
    const size_t row_bytes = static_cast<size_t>(d) * 2;
    auto tile_rsrc = [&](const uint16_t* slab, int row0) {
        return fa::make_rsrc(fa::scalar_ptr(slab + static_cast<size_t>(row0) * d), 0,
                             static_cast<uint32_t>(min(kEdge, n - row0) * row_bytes));
    };
    const fa::i32x4 q_rsrc = tile_rsrc(q_slab, tile_q0);
    const fa::i32x4 k_rsrc = tile_rsrc(k_slab, tile_k0);
    for (int c0 = 0; c0 < d; c0 += kCols)
    {
        if (c0) __syncthreads();  // the last columns have been read
#pragma unroll
        for (int u = 0; u < kEdge * kPieces / kThreads; ++u)
        {
            const int x = u * kThreads + threadIdx.x;
            const int row = x / kPieces;
            if constexpr (kVec)
            {
                // The 64 pieces of a wave go to consecutive places; rows past
                // the sequence end and columns past the last read as zero.
                const int col = c0 + 8 * (x % kPieces ^ ((row >> 1) & 7));
                const uint32_t from = col < d ? static_cast<uint32_t>(row * row_bytes + 2 * col) : kNowhere;
                const uint32_t to = (u * kThreads + wave * 64) * 16;
                fa::dma16(q_rsrc, from, fa::lds_addr(qs) + to);
                fa::dma16(k_rsrc, from, fa::lds_addr(ks) + to);
            }
            else
            {
                // Rows past the sequence end stage the last row: their scores
                // are not stored.
                const int c = x % kPieces;
                const bf16x8 a = load_operand<kVec>(q_slab + static_cast<size_t>(min(tile_q0 + row, n - 1)) * d, c0 + 8 * c, d);
                const bf16x8 b = load_operand<kVec>(k_slab + static_cast<size_t>(min(tile_k0 + row, n - 1)) * d, c0 + 8 * c, d);
                *reinterpret_cast<bf16x8*>(qs + piece(row, c)) = a;
                *reinterpret_cast<bf16x8*>(ks + piece(row, c)) = b;
            }
        }
        if constexpr (kVec) fa::wait_vm_lgkm0<0>();
        __syncthreads();
#pragma unroll
        for (int step = 0; step < kCols / 16; ++step)
            if (c0 + 16 * step < d)
            {
                bf16x8 a[kBlocks], b[kBlocks];
#pragma unroll
                for (int x = 0; x < kBlocks; ++x)
                {
                    a[x] = *reinterpret_cast<const bf16x8*>(qs + piece(wave_q + 32 * x + i, 2 * step + h));
                    b[x] = *reinterpret_cast<const bf16x8*>(ks + piece(wave_k + 32 * x + i, 2 * step + h));
                }
#pragma unroll
                for (int x = 0; x < kBlocks; ++x)
#pragma unroll
                    for (int y = 0; y < kBlocks; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[y], a[x], acc[x][y], 0, 0, 0);
            }
    }
    __syncthreads();  // every operand has been read: the buffer is free
    if (q0 >= n || k0 >= n) return;

    // Accumulator r of block (x, y): query 32x + i, key 32y + 8(r/4) + 4h + r%4.
    // A block of 32 rows at a time goes through the wave's own part of LDS
    // and out in 16-byte pieces of whole rows. Straight from the registers a
    // store writes 4 bytes per lane: 7 us more at (2,8,2048,64).
    float* const buf = reinterpret_cast<float*>(lds) + wave * 32 * kPitch;
    const bool inside = q0 + kRowScores <= n && k0 + kRowScores <= n;
    const bool masked = causal && k0 + kRowScores - 1 > q0;
#pragma unroll
    for (int x = 0; x < kBlocks; ++x)
    {
#pragma unroll
        for (int y = 0; y < kBlocks; ++y)
#pragma unroll
            for (int g = 0; g < 4; ++g)
            {
                const int col = 32 * y + 8 * g + 4 * h;
                f32x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    out[e] = masked && k0 + col + e > q0 + 32 * x + i ? -FLT_MAX : acc[x][y][4 * g + e] * scale;
                *reinterpret_cast<f32x4*>(buf + i * kPitch + col) = out;
            }
        wave_lds_fence();
        constexpr int kLanes = kRowScores / 4;  // lanes per row
#pragma unroll
        for (int u = 0; u < 32 * kLanes / 64; ++u)
        {
            const int row = u * (64 / kLanes) + lane / kLanes;
            const int col = lane % kLanes * 4;
            const f32x4 out = *reinterpret_cast<const f32x4*>(buf + row * kPitch + col);
            float* const dst = s_wave + static_cast<size_t>(32 * x + row) * n + col;
            if (inside) *reinterpret_cast<f32x4u*>(dst) = out;
            else if (q0 + 32 * x + row < n)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k0 + col + e < n) dst[e] = out[e];
        }
        wave_lds_fence();
    }
}

// Maximum or sum over the kWaves waves that share a row (kWaves == 1: no LDS,
// no barrier; otherwise the whole workgroup, which is one row).
template <int kWaves>
__device__ __forceinline__ float row_max(float x, float* scratch)
{
    x = fa::wave_max(x);
    if constexpr (kWaves > 1)
    {
        if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = x;
        __syncthreads();
        x = scratch[0];
        for (int w = 1; w < kWaves; ++w) x = fmaxf(x, scratch[w]);
        __syncthreads();
    }
    return x;
}

template <int kWaves>
__device__ __forceinline__ float row_sum(float x, float* scratch)
{
    x = fa::wave_sum(x);
    if constexpr (kWaves > 1)
    {
        if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = x;
        __syncthreads();
        x = scratch[0];
        for (int w = 1; w < kWaves; ++w) x += scratch[w];
        __syncthreads();
    }
    return x;
}

__device__ __forceinline__ float softmax_exp(float x, float row_max)
{
    return __builtin_amdgcn_exp2f((x - row_max) * fa::kLog2e);
}

// A row in the registers of kWaves waves (1, then four rows per workgroup, or
// all 4), kVecs float4 per lane: read once, written once, at any address and
// length up to 256 * kWaves * kVecs. The floats before the first 16-byte
// boundary and after the last are taken one each by lanes 0.. and 4... Same
// stages as kernels/v0_unfused.cu:51-94: max, exp(x - max) and sum, multiply
// by 1/sum (sum <= 0 -> 1). Bound by HBM: 6.3-7.2 TB/s read and written from
// 256 columns on. Rows of a length or address off 16 bytes, and of more than
// 8192 columns, took three passes before (14532 x 1211: 41 us, now 23).
//
// kCausal: row r is query r % cols of its slab, and the scores of later keys
// are taken as -FLT_MAX without being read (the whole row of weights is
// written).
template <int kWaves, int kVecs, bool kCausal>
__global__ __launch_bounds__(kThreads) void v0_softmax_rows_reg_kernel(float* __restrict__ s, int rows, int cols)
{
    __shared__ float scratch[kThreads / 64];
    constexpr int kLanes = 64 * kWaves;  // lanes per row
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = static_cast<int>(blockIdx.x) * (kThreads / kLanes) + wave / kWaves;
    if (row >= rows) return;  // one wave per row: no barrier follows
    const int t = threadIdx.x % kLanes;
    const int live = kCausal ? row % cols + 1 : cols;  // scores of the row that are read
    float* const first = s + static_cast<size_t>(row) * cols;
    const int head = min(cols, static_cast<int>(-reinterpret_cast<uintptr_t>(first) >> 2) & 3);
    const int nvec = (cols - head) >> 2;
    const int tail = cols - head - 4 * nvec;
    float4* const body = reinterpret_cast<float4*>(first + head);
    // The single float of lanes 0 .. head - 1 and 4 .. 3 + tail.
    const bool single = t < head || (t >= 4 && t < 4 + tail);
    const int one = t < head ? t : head + 4 * nvec + t - 4;

    float4 v[kVecs];
    float x = single && (!kCausal || one < live) ? first[one] : -FLT_MAX;
    float local_max = x;
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
    {
        const int idx = t + i * kLanes;
        if constexpr (kCausal)
        {
            const int key = head + 4 * idx;
            v[i] = make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX);
            if (idx < nvec && key < live)
            {
                const float4 y = body[idx];
                v[i].x = y.x;
                if (key + 1 < live) v[i].y = y.y;
                if (key + 2 < live) v[i].z = y.z;
                if (key + 3 < live) v[i].w = y.w;
            }
        }
        else if (idx < nvec) v[i] = body[idx];
    }
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
        if (t + i * kLanes < nvec) local_max = fmaxf(local_max, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
    const float max = row_max<kWaves>(local_max, scratch);

    float local_sum = 0.0f;
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
        if (t + i * kLanes < nvec)
        {
            v[i].x = softmax_exp(v[i].x, max);
            v[i].y = softmax_exp(v[i].y, max);
            v[i].z = softmax_exp(v[i].z, max);
            v[i].w = softmax_exp(v[i].w, max);
            local_sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
        }
    if (single)
    {
        x = softmax_exp(x, max);
        local_sum += x;
    }
    const float total = row_sum<kWaves>(local_sum, scratch);
    const float inverse = 1.0f / (total > 0.0f ? total : 1.0f);

#pragma unroll
    for (int i = 0; i < kVecs; ++i)
    {
        const int idx = t + i * kLanes;
        if (idx < nvec) body[idx] = make_float4(v[i].x * inverse, v[i].y * inverse, v[i].z * inverse, v[i].w * inverse);
    }
    if (single) first[one] = x * inverse;
}

// Longer rows: the reference's three passes over the row in HBM.
__global__ __launch_bounds__(kThreads) void v0_softmax_rows_loop_kernel(float* __restrict__ s, int cols, int causal)
{
    constexpr int kWaves = kThreads / 64;
    __shared__ float scratch[kWaves];
    float* row = s + static_cast<size_t>(blockIdx.x) * cols;
    const int live = causal ? static_cast<int>(blockIdx.x % static_cast<unsigned>(cols)) + 1 : cols;
    float local_max = -FLT_MAX;
    for (int c = threadIdx.x; c < live; c += kThreads) local_max = fmaxf(local_max, row[c]);
    const float max = row_max<kWaves>(local_max, scratch);
    float local_sum = 0.0f;
    for (int c = threadIdx.x; c < cols; c += kThreads)
    {
        const float e = softmax_exp(c < live ? row[c] : -FLT_MAX, max);
        row[c] = e;
        local_sum += e;
    }
    const float total = row_sum<kWaves>(local_sum, scratch);
    const float inverse = 1.0f / (total > 0.0f ? total : 1.0f);
    for (int c = threadIdx.x; c < cols; c += kThreads) row[c] *= inverse;
}

// A float as three bf16 values whose sum it is exactly (8 bits of the
// significand each, by truncation; what lies below the smallest subnormal is
// dropped), for two floats at a time: the words' low halves come from a.
struct Split3
{
    uint32_t hi, mid, lo;
};

__device__ __forceinline__ Split3 split3(float a, float b)
{
    auto top = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
    auto pack = [](float x, float y) { return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u); };
    const float a1 = a - top(a), b1 = b - top(b);
    const float a2 = a1 - top(a1), b2 = b1 - top(b1);
    return {pack(a, b), pack(a1, b1), pack(a2, b2)};
}

// The values of an operand of V that are finite, and the others; zero elsewhere.
struct FiniteSplit
{
    bf16x8 finite, other;
};

__device__ __forceinline__ FiniteSplit split_finite(bf16x8 v)
{
    const u32x4 bits = __builtin_bit_cast(u32x4, v);
    u32x4 finite, other;
#pragma unroll
    for (int e = 0; e < 4; ++e)
    {
        const uint32_t lo = (bits[e] & 0x7f80u) == 0x7f80u ? 0xffffu : 0u;
        const uint32_t hi = (bits[e] & 0x7f800000u) == 0x7f800000u ? 0xffff0000u : 0u;
        other[e] = bits[e] & (lo | hi);
        finite[e] = bits[e] & ~(lo | hi);
    }
    return {__builtin_bit_cast(bf16x8, finite), __builtin_bit_cast(bf16x8, other)};
}

// O[bh][q][c] = bf16_rne(sum_k P[q][k] V[k][c]) for 32 queries and 32 * kDims
// columns per workgroup (grid: (blocks of 32 queries, in eights, * tiles of
// columns, B*H)). Four waves: wave w takes the 32-key tiles w, w + 4, .., so a
// workgroup reads whole rows of P, and the waves' sums are added in order at the
// end. Nothing is shared between the waves before that, so the walk has no barrier.
//
// Each fp32 weight is split into three bf16 values (split3), and their products
// with V, which fp32 holds exactly, are summed in fp32 by the matrix cores
// (v_mfma_f32_16x16x32_bf16): the precision of fp32 FMAs at a third of the bf16
// rate. Only beside an infinity in V do the parts differ from the weight: one
// that is zero gives NaN where the weight itself gives an infinity. A wave whose
// sums hold a NaN walks its tiles again with the parts times V's finite values
// and, for the others, the weight's being zero or not: finite inputs pay under
// 1 % for the test, (2,8,2048,64) with a column of infinities 287 us for 205.
// As in the fused kernel the product is taken transposed, O^T = V^T P^T:
// lane l holds query l % 16, and V^T comes from the row-major tile in LDS
// through ds_read_b64_tr_b16. The keys of a P operand are chosen so that the
// four lanes of a row load 64 bytes of it in one instruction (lane group g: keys
// 4g .. and 16 + 4g ..); 32 x 32 blocks, whose two lanes of a row load 32 bytes,
// were 3 % slower at (2,8,2048,64), 10 % at (1,4,4096,256). A tile of V goes to
// LDS by copies without registers, and the next tile's P and V are fetched a
// tile ahead.
//
// fp32 FMAs from LDS tiles were bound by the vector unit and its LDS reads (227
// us at (2,8,2048,64)). Now memory bounds it: 73 us for 268 MB of P, beside which
// the weights that the softmax left in the last-level cache are written back (the
// three kernels together move 1.07 GB in 204 us, the card's copy rate). 32
// queries per workgroup and keys split over the waves give four times the
// workgroups of 128 queries, for the same reads of P (V is read once per
// workgroup, from the L2).
//
// kCausal: the weights of keys past a query are one value per row, the row's
// last weight: 0, except in a row whose scores are all -infinity (there the
// softmax spreads the weight over the masked keys). Tiles wholly above the
// diagonal take it from a register instead of reading P. Their products stay,
// so that a NaN or infinity in V reaches every row, as it does in a product
// with the whole matrix; where the value is 0 in all rows, one part does.
template <int kDims, bool kVec, bool kCausal>
__global__ __launch_bounds__(kThreads) void v0_pv_kernel(const float* __restrict__ p,
                                                          const uint16_t* __restrict__ v,
                                                          uint16_t* __restrict__ o, int n, int d,
                                                          int tiles_d, int vec_o)
{
    constexpr int kWaves = kThreads / 64;
    constexpr int kPitch = 32 * kDims;              // bf16 elements of a staged row
    constexpr int kPieces = 4 * kDims;              // its 16-byte pieces
    constexpr int kLoads = 32 * kPieces / 64;       // pieces per lane and tile
    constexpr int kTileElems = 32 * kPitch;
    constexpr int kMergeFloats = kWaves * 16 * 64;  // one 32-column block of each wave
    constexpr int kTileBytes = kWaves * 2 * kTileElems * 2;  // two tiles per wave
    // One phase of a transposing read touches a pair of pieces (16 columns) of
    // eight consecutive rows: pair x of row r lies at pair x ^ turn(r), which
    // puts the eight in distinct banks.
    auto turn = [](int row) { return kDims == 4 ? row & 7 : kDims == 2 ? (row >> 1) & 3 : (row >> 2) & 1; };
    __shared__ __attribute__((aligned(16))) unsigned char
        lds[kTileBytes > 2 * kMergeFloats * 4 ? kTileBytes : 2 * kMergeFloats * 4];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int i = lane & 15;
    const int g = lane >> 4;
    const int n_tiles = (n + 31) / 32;
    // Workgroups go to the 8 XCDs in turn: the column tiles of a query block take
    // numbers 8 apart, so that they share an XCD and its L2 serves P to all but
    // the first.
    const int round = static_cast<int>(blockIdx.x) / (8 * tiles_d);
    const int place = static_cast<int>(blockIdx.x) % (8 * tiles_d);
    const int q_block = round * 8 + place % 8;
    if (q_block >= n_tiles) return;
    const int q0 = (kCausal ? n_tiles - 1 - q_block : q_block) * 32;  // causal: most work first
    const int c0 = place / 8 * 32 * kDims;
    const size_t bh = blockIdx.y;
    // The row of P of lane `of` in block y.
    auto p_row_of = [&](int of, int y) {
        return p + bh * n * n + static_cast<size_t>(min(q0 + 16 * y + (of & 15), n - 1)) * n + 4 * (of >> 4);
    };
    const float* const p_row[2] = {p_row_of(lane, 0), p_row_of(lane, 1)};
    const uint16_t* const v_slab = v + bh * n * d;
    uint16_t* const tiles = reinterpret_cast<uint16_t*>(lds) + wave * 2 * kTileElems;
    const int live_tiles = kCausal ? min(n_tiles, q0 / 32 + 1) : n_tiles;  // tiles of P that are read
    float masked[2] = {0.0f, 0.0f};
    if (kCausal && live_tiles < n_tiles)
#pragma unroll
        for (int y = 0; y < 2; ++y) masked[y] = p_row[y][n - 1 - 4 * g];
    const bool masked_zero = kCausal && !__any(!(masked[0] == 0.0f && masked[1] == 0.0f));

    f32x4 acc[2 * kDims][2];  // 16 columns x 16 queries each

    // Weights of keys 32t + 16j + 4g .. + 3 (j = 0, 1) of the lane's query of
    // block y; zero past the last key.
    auto load_p = [&](const float* row, int t, int y, f32x4 (&w)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            const int key = 32 * t + 16 * j + 4 * g;
            const float* const src = row + 32 * t + 16 * j;
            if (kCausal && t >= live_tiles)
#pragma unroll
                for (int e = 0; e < 4; ++e) w[j][e] = key + e < n ? masked[y] : 0.0f;
            else if (32 * t + 32 <= n) w[j] = *reinterpret_cast<const f32x4u*>(src);
            else
#pragma unroll
                for (int e = 0; e < 4; ++e) w[j][e] = key + e < n ? src[e] : 0.0f;
        }
    };
    // The tile's rows of V into buffer `to`, 16 bytes per lane and copy; zero past
    // the last key and column. Element-wise loads (a row that is no whole number
    // of pieces, or an address off 16 bytes) go through registers.
    uint32_t from[kLoads];
    if constexpr (kVec)
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
        {
            const int row = (u * 64 + lane) / kPieces;
            const int col = c0 + ((u * 64 + lane) % kPieces ^ (2 * turn(row))) * 8;
            from[u] = col < d ? static_cast<uint32_t>((row * d + col) * 2) : kNowhere;
        }
    auto load_v = [&](int t, uint16_t* to) {
        if constexpr (kVec)
        {
            const fa::i32x4 rsrc = fa::make_rsrc(fa::scalar_ptr(v_slab + static_cast<size_t>(32 * t) * d), 0,
                                                 static_cast<uint32_t>(min(32, n - 32 * t) * d * 2));
#pragma unroll
            for (int u = 0; u < kLoads; ++u) fa::dma16(rsrc, from[u], fa::lds_addr(to) + u * 1024);
        }
        else
#pragma unroll
            for (int u = 0; u < kLoads; ++u)
            {
                const int row = (u * 64 + lane) / kPieces;
                const int c = (u * 64 + lane) % kPieces;
                const bf16x8 x = 32 * t + row < n
                                     ? load_operand<kVec>(v_slab + static_cast<size_t>(32 * t + row) * d, c0 + 8 * c, d)
                                     : bf16x8{};
                *reinterpret_cast<bf16x8*>(to + row * kPitch + (c ^ (2 * turn(row))) * 8) = x;
            }
    };
    // Source lanes of the transposing reads: the 16 lanes of group g read keys
    // 4g .. 4g + 3 (and 16 + 4g ..), each lane four of 16 columns.
    const int tr_row = 4 * g + (i >> 2);
    auto v_operand = [&](const uint16_t* tile, int x) {
        const uint16_t* const lo_at = tile + tr_row * kPitch + 16 * (x ^ turn(tr_row)) + 4 * (i & 3);
        const uint16_t* const hi_at = tile + (16 + tr_row) * kPitch + 16 * (x ^ turn(16 + tr_row)) + 4 * (i & 3);
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(lo_at));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(hi_at));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    // The parts of a lane's weights as B operands: element e is key
    // 16(e/4) + 4g + e%4.
    auto split_weights = [](const f32x4 (&w)[2], bf16x8 (&part)[3]) {
        u32x4 bits[3];
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            const f32x4 z = w[e / 2];
            const Split3 s3 = e % 2 ? split3(z[2], z[3]) : split3(z[0], z[1]);
            bits[0][e] = s3.hi;
            bits[1][e] = s3.mid;
            bits[2][e] = s3.lo;
        }
#pragma unroll
        for (int z = 0; z < 3; ++z) part[z] = __builtin_bit_cast(bf16x8, bits[z]);
    };
    auto clear = [&]() {
#pragma unroll
        for (int x = 0; x < 2 * kDims; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = f32x4{};
    };
    clear();
    f32x4 w_next[2][2];
    if (wave < n_tiles)
    {
        load_v(wave, tiles);
#pragma unroll
        for (int y = 0; y < 2; ++y) load_p(p_row[y], wave, y, w_next[y]);
    }
    int buffer = 0;
    for (int t = wave; t < n_tiles; t += kWaves)
    {
        f32x4 w[2][2];
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int j = 0; j < 2; ++j) w[y][j] = w_next[y][j];
        // The tile has landed; the other buffer was read in the last step.
        fa::wait_vm_lgkm0<0>();
        wave_lds_fence();
        const uint16_t* const tile = tiles + buffer * kTileElems;
        buffer ^= 1;
        if (t + kWaves < n_tiles)
        {
            load_v(t + kWaves, tiles + buffer * kTileElems);
#pragma unroll
            for (int y = 0; y < 2; ++y) load_p(p_row[y], t + kWaves, y, w_next[y]);
        }
        if (kCausal && masked_zero && t >= live_tiles)
        {
#pragma unroll
            for (int x = 0; x < 2 * kDims; ++x)
            {
                const bf16x8 va = v_operand(tile, x);
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, bf16x8{}, acc[x][y], 0, 0, 0);
            }
            wave_lds_fence();
            continue;
        }
        bf16x8 part[2][3];
#pragma unroll
        for (int y = 0; y < 2; ++y) split_weights(w[y], part[y]);
#pragma unroll
        for (int x = 0; x < 2 * kDims; ++x)
        {
            const bf16x8 va = v_operand(tile, x);
#pragma unroll
            for (int z = 2; z >= 0; --z)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, part[y][z], acc[x][y], 0, 0, 0);
        }
        wave_lds_fence();
    }
    f32x4 all = f32x4{};  // NaN if any sum is
#pragma unroll
    for (int x = 0; x < 2 * kDims; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) all += acc[x][y];
    const float one = (all[0] + all[1]) + (all[2] + all[3]);
    if (__any(one != one))
    {
        // The lane number anew, so that the first walk keeps no row address for
        // this one (two more registers cost a workgroup per CU).
        int lane_again = threadIdx.x & 63;
        asm volatile("" : "+v"(lane_again));
        clear();
        for (int t = wave; t < n_tiles; t += kWaves)
        {
            load_v(t, tiles);
            fa::wait_vm_lgkm0<0>();
            wave_lds_fence();
#pragma unroll
            for (int y = 0; y < 2; ++y)
            {
                f32x4 w[2];
                load_p(p_row_of(lane_again, y), t, y, w);
                // One operand at a time: no more registers than the walk above.
                bf16x8 part[3];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    part[0][e] = __builtin_bit_cast(__bf16, static_cast<uint16_t>(w[e / 4][e % 4] != 0.0f ? 0x3f80 : 0));
#pragma unroll
                for (int x = 0; x < 2 * kDims; ++x)
                {
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(split_finite(v_operand(tiles, x)).other, part[0],
                                                                        acc[x][y], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                split_weights(w, part);
#pragma unroll
                for (int x = 0; x < 2 * kDims; ++x)
                {
                    const bf16x8 va = split_finite(v_operand(tiles, x)).finite;
#pragma unroll
                    for (int z = 2; z >= 0; --z)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, part[z], acc[x][y], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // Every operand has been read before the next tile lands.
            fa::wait_vm_lgkm0<0>();
            wave_lds_fence();
        }
    }

    // 32 columns of the sums at a time: each wave writes its own, wave x % 4
    // adds them in wave order and stores. acc[x][y][e]: column 16x + 4g + e.
    __syncthreads();  // every tile has been read
#pragma unroll
    for (int x = 0; x < kDims; ++x)
    {
        float* const area = reinterpret_cast<float*>(lds) + (x & 1) * kMergeFloats;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *reinterpret_cast<f32x4*>(area + ((wave * 4 + u) * 64 + lane) * 4) = acc[2 * x + u / 2][u % 2];
        __syncthreads();
        if (wave != x % kWaves) continue;
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            f32x4 sum = *reinterpret_cast<const f32x4*>(area + (u * 64 + lane) * 4);
#pragma unroll
            for (int y = 1; y < kWaves; ++y) sum += *reinterpret_cast<const f32x4*>(area + ((y * 4 + u) * 64 + lane) * 4);
            const int row = q0 + 16 * (u % 2) + i;
            const int col = c0 + 32 * x + 16 * (u / 2) + 4 * g;
            if (row >= n) continue;
            uint16_t* const dst = o + bh * n * d + static_cast<size_t>(row) * d + col;
            if (vec_o && col < d)
                *reinterpret_cast<uint2*>(dst) =
                    make_uint2(fa::pack_bf16x2(sum[0], sum[1]), fa::pack_bf16x2(sum[2], sum[3]));
            else if (!vec_o)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < d) dst[e] = fa::float_to_bf16_bits(sum[e]);
        }
    }
}

// Tiles of 128 x 128 scores where the launch has two for every CU (five for every
// four beyond head_dim 128, where they save more reads of Q and K), else of 64 x 64:
// four times the workgroups, each with a quarter of the work. (All three kernels
// with large tiles over those with small ones, 400 launches: up to head_dim 128 at
// 256 to 320, 384 to 448 and 512 to 640 large tiles 1.06, 1.03 and 1.01 times the
// time, beyond 128 1.03, 0.99 and 0.99; 0.98 from 768 on.)
hipError_t launch_scores(bool vec, const uint16_t* q, const uint16_t* k, float* s, int bh, int n, int d, float scale,
                         int causal, hipStream_t stream)
{
    const long long wide = (n + 127) / 128;
    const long long launched = bh * (causal ? wide * (wide + 1) / 2 : wide * wide);
    const bool two = 4 * launched >= (d > 128 ? 5LL : 8LL) * fa::device_compute_units();
    const int tiles = two ? static_cast<int>(wide) : (n + 63) / 64;
    const dim3 grid(static_cast<unsigned>(causal ? tiles * (tiles + 1LL) / 2 : 1LL * tiles * tiles),
                    static_cast<unsigned>(bh));
    const auto kernel = vec ? (two ? v0_scores_kernel<true, 2> : v0_scores_kernel<true, 1>)
                            : (two ? v0_scores_kernel<false, 2> : v0_scores_kernel<false, 1>);
    return fa::launch_kernel(kernel, grid, dim3(kThreads), stream, q, k, s, n, d, tiles, scale, causal);
}

inline bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// Columns per workgroup: all of them up to 128 (P is then read once), else
// equal tiles of at most 128.
template <bool kCausal>
hipError_t launch_pv(const float* p, const uint16_t* v, uint16_t* o, int bh, int n, int d, hipStream_t stream)
{
    const bool vec = (d % 8 == 0) && d <= kMaxCopyDim && aligned16(v);
    const int vec_o = (d % 4 == 0) && (reinterpret_cast<uintptr_t>(o) & 7u) == 0;
    const int blocks_d = (d + 31) / 32;
    const int tiles_d = (blocks_d + 3) / 4;
    const int dims = (blocks_d + tiles_d - 1) / tiles_d;
    const dim3 grid(static_cast<unsigned>(((n + 31) / 32 + 7) / 8 * 8 * tiles_d), static_cast<unsigned>(bh));
    auto launch = [&](auto kernel) {
        return fa::launch_kernel(kernel, grid, dim3(kThreads), stream, p, v, o, n, d, tiles_d, vec_o);
    };
    switch (dims)
    {
        case 1: return launch(vec ? v0_pv_kernel<1, true, kCausal> : v0_pv_kernel<1, false, kCausal>);
        case 2: return launch(vec ? v0_pv_kernel<2, true, kCausal> : v0_pv_kernel<2, false, kCausal>);
        case 3: return launch(vec ? v0_pv_kernel<3, true, kCausal> : v0_pv_kernel<3, false, kCausal>);
        default: return launch(vec ? v0_pv_kernel<4, true, kCausal> : v0_pv_kernel<4, false, kCausal>);
    }
}

constexpr int kMaxGridY = 65535;

// One wave per row up to 1024 columns (no barrier, four rows per workgroup:
// 16384 x 256 took 14.5 us with a workgroup per row, 6 to 7 so), then four (2048
// columns: 74 us against 78 for 32768 rows).
template <bool kCausal>
hipError_t launch_softmax(float* s, int rows, int cols, hipStream_t stream)
{
    const dim3 block(kThreads);
    const unsigned row_count = static_cast<unsigned>(rows);
    auto wave = [&](auto kernel) { return fa::launch_kernel(kernel, dim3((row_count + 3) / 4), block, stream, s, rows, cols); };
    auto four = [&](auto kernel) { return fa::launch_kernel(kernel, dim3(row_count), block, stream, s, rows, cols); };
    if (cols <= 256) return wave(v0_softmax_rows_reg_kernel<1, 1, kCausal>);
    if (cols <= 512) return wave(v0_softmax_rows_reg_kernel<1, 2, kCausal>);
    if (cols <= 1024) return wave(v0_softmax_rows_reg_kernel<1, 4, kCausal>);
    if (cols <= 2048) return four(v0_softmax_rows_reg_kernel<4, 2, kCausal>);
    if (cols <= 4096) return four(v0_softmax_rows_reg_kernel<4, 4, kCausal>);
    if (cols <= 8192) return four(v0_softmax_rows_reg_kernel<4, 8, kCausal>);
    if (cols <= 16384) return four(v0_softmax_rows_reg_kernel<4, 16, kCausal>);
    if (cols <= 32768) return four(v0_softmax_rows_reg_kernel<4, 32, kCausal>);
    return fa::launch_kernel(v0_softmax_rows_loop_kernel, dim3(row_count), block, stream, s, cols, kCausal ? 1 : 0);
}

// Shape and pointer checks shared by the v0 entry points (the workspace is
// checked by the caller): hipSuccess, -1 for an empty shape (nothing to
// launch) or hipErrorInvalidValue.
int validate_unfused(const void* q, const void* k, const void* v, void* o, int batch, int heads, int seq_len,
                     int head_dim)
{
    if (batch < 0 || heads < 0 || seq_len < 0 || head_dim <= 0) return hipErrorInvalidValue;
    const long long bh = static_cast<long long>(batch) * heads;
    if (bh == 0 || seq_len == 0) return -1;  // empty: nothing to launch
    if (!q || !k || !v || !o) return hipErrorInvalidValue;
    if (bh > kMaxGridY) return hipErrorInvalidValue;
    const long long tiles = (static_cast<long long>(seq_len) + kTile - 1) / kTile;
    if (tiles * tiles > 0x7fffffffLL) return hipErrorInvalidValue;
    if (bh * seq_len > 0x7fffffffLL) return hipErrorInvalidValue;  // softmax grid
    return hipSuccess;
}

int launch_unfused_impl(const void* q, const void* k, const void* v, void* o, float* workspace, int batch,
                        int heads, int seq_len, int head_dim, int causal, hipEvent_t const* events,
                        hipStream_t stream)
{
    const int status = validate_unfused(q, k, v, o, batch, heads, seq_len, head_dim);
    if (status == -1) return hipSuccess;
    if (status != hipSuccess) return status;
    if (!workspace) return hipErrorInvalidValue;

    const int bh = batch * heads;
    const int n = seq_len;
    const int d = head_dim;
    const float scale = fa_default_scale(d);
    const uint16_t* qb = static_cast<const uint16_t*>(q);
    const uint16_t* kb = static_cast<const uint16_t*>(k);
    const uint16_t* vb = static_cast<const uint16_t*>(v);
    uint16_t* ob = static_cast<uint16_t*>(o);

    if (events)
    {
        const hipError_t e = hipEventRecord(events[0], stream);
        if (e != hipSuccess) return e;
    }
    const bool vec_qk = (d % 8 == 0) && d <= kMaxCopyDim && aligned16(q) && aligned16(k);
    hipError_t e = launch_scores(vec_qk, qb, kb, workspace, bh, n, d, scale, causal, stream);
    if (e != hipSuccess) return e;
    if (events && (e = hipEventRecord(events[1], stream)) != hipSuccess) return e;

    // The softmax sees the workspace as one [B*H*N, N] matrix.
    e = causal ? launch_softmax<true>(workspace, bh * n, n, stream) : launch_softmax<false>(workspace, bh * n, n, stream);
    if (e != hipSuccess) return e;
    if (events && (e = hipEventRecord(events[2], stream)) != hipSuccess) return e;

    e = causal ? launch_pv<true>(workspace, vb, ob, bh, n, d, stream) : launch_pv<false>(workspace, vb, ob, bh, n, d, stream);
    if (e != hipSuccess) return e;
    if (events && (e = hipEventRecord(events[3], stream)) != hipSuccess) return e;
    return hipSuccess;
}

// The allocation-free v0 entry point's score workspace: a file-scope device
// array, one copy per GPU, held for the life of the process. In host code
// its name is only a stand-in for the symbol; the device address is looked
// up once per device (noalloc_scratch) and only that address is used.
constexpr size_t kNoAllocScratchBytes = size_t{64} << 20;
__device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;

// Device address of `scratch` on the current device (hipGetSymbolAddress,
// once per device, cached), or null with the HIP status in *status.
float* noalloc_scratch(int* status)
{
    static std::atomic<uintptr_t> cache[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices)
    {
        *status = e != hipSuccess ? e : hipErrorInvalidDevice;
        return nullptr;
    }
    uintptr_t addr = cache[dev].load(std::memory_order_acquire);
    if (addr == 0)
    {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
        {
            *status = e != hipSuccess ? e : hipErrorInvalidSymbol;
            return nullptr;
        }
        addr = reinterpret_cast<uintptr_t>(ptr);
        cache[dev].store(addr, std::memory_order_release);
    }
    *status = hipSuccess;
    return reinterpret_cast<float*>(addr);
}

int launch_unfused_noalloc(const void* q, const void* k, const void* v, void* o, int batch, int heads, int seq_len,
                           int head_dim, int causal, hipStream_t stream)
{
    // The same checks as the workspace entry, minus the workspace pointer.
    int status = validate_unfused(q, k, v, o, batch, heads, seq_len, head_dim);
    if (status == -1) return hipSuccess;
    if (status != hipSuccess) return status;
    const size_t need = fa_unfused_workspace_bytes(batch, heads, seq_len, head_dim);
    if (need > kNoAllocScratchBytes) return hipErrorInvalidValue;
    float* ws = noalloc_scratch(&status);
    if (!ws) return status;
    // The softmax reads no score that the scores kernel has not written and
    // writes every weight, so the array needs no clearing between calls.
    return launch_unfused_impl(q, k, v, o, ws, batch, heads, seq_len, head_dim, causal, nullptr, stream);
}

}  // namespace

extern "C" {

size_t fa_unfused_noalloc_max_workspace_bytes(void) { return kNoAllocScratchBytes; }

int fa_launch_attention_unfused_noalloc(const void* q, const void* k, const void* v, void* o, int batch, int heads,
                                        int seq_len, int head_dim, int causal, void* stream)
{
    return fa::record_status(launch_unfused_noalloc(q, k, v, o, batch, heads, seq_len, head_dim, causal,
                                                    static_cast<hipStream_t>(stream)));
}

float fa_default_scale(int head_dim) { return 1.0f / sqrtf(static_cast<float>(head_dim)); }

double fa_attention_flops(int batch, int heads, int seq_len, int head_dim, int causal)
{
    const double n = static_cast<double>(seq_len);
    const double pairs = causal ? n * (n + 1.0) / 2.0 : n * n;
    return 4.0 * pairs * static_cast<double>(head_dim) * static_cast<double>(batch) * static_cast<double>(heads);
}

size_t fa_unfused_workspace_bytes(int batch, int heads, int seq_len, int /*head_dim*/)
{
    if (batch <= 0 || heads <= 0 || seq_len <= 0) return 0;
    return static_cast<size_t>(batch) * heads * seq_len * static_cast<size_t>(seq_len) * sizeof(float);
}

int fa_launch_softmax_rows_inplace(float* s, int rows, int cols, void* stream)
{
    if (rows < 0 || cols < 0) return fa::record_status(hipErrorInvalidValue);
    if (rows == 0 || cols == 0) return hipSuccess;
    if (!s) return fa::record_status(hipErrorInvalidValue);
    return fa::record_status(launch_softmax<false>(s, rows, cols, static_cast<hipStream_t>(stream)));
}

int fa_launch_attention_unfused(const void* q, const void* k, const void* v, void* o, float* workspace,
                                int batch, int heads, int seq_len, int head_dim, int causal, void* stream)
{
    return fa::record_status(launch_unfused_impl(q, k, v, o, workspace, batch, heads, seq_len, head_dim, causal,
                                                 nullptr, static_cast<hipStream_t>(stream)));
}

int fa_launch_attention_unfused_profile(const void* q, const void* k, const void* v, void* o, float* workspace,
                                        int batch, int heads, int seq_len, int head_dim, int causal,
                                        void* const* events, void* stream)
{
    return fa::record_status(launch_unfused_impl(q, k, v, o, workspace, batch, heads, seq_len, head_dim, causal,
                                                 reinterpret_cast<hipEvent_t const*>(events),
                                                 static_cast<hipStream_t>(stream)));
}

}  // extern "C"
