// Product of a MACKO fp16 matrix with several vectors on the matrix cores (gfx950, wave64).
//
//   Y[n, r] = sum_c M[r, c] X[n, c]        X [batch, ldx], Y [batch, ldy], row-major fp16
//
// A workgroup of 16 waves owns a block of up to 16 * RT rows and up to 128 vectors and walks the
// columns in chunks.  Per chunk every wave
//   1. requests the pieces of X it will multiply (16 bytes per lane, straight into registers in the
//      operand layout of v_mfma_f32_16x16x32_f16),
//   2. writes its RT rows' part of the chunk into LDS as plain dense fp16: zeroes first, then one
//      2-byte store per stored entry at the entry's column (the prefix sum of nibbles of the
//      single-vector kernels, one row per wave at a time),
//   3. requests the entries of the chunk after this one,
//   4. meets the others at a barrier and multiplies: A from LDS, B from the registers of step 1.
// The dense chunk is double-buffered, so one barrier per chunk is enough and waves that still
// scatter run beside waves that already multiply.  The 16 waves share a chunk's products by groups
// of 16 * NTW vectors and, within a group, by columns; their partial sums meet in LDS at the end, in
// a fixed order.
//
// Every stored entry costs one LDS store however many vectors there are, and a vector costs one read
// of X per row block; the gather kernels read LDS once per entry for a few vectors and stream the
// matrix again for the next few.  Measured on 11008 x 4096 at density 0.5, 128 vectors: 341 us through the
// gather kernels in groups of eight (17 TFLOP/s), 27.4 here (211 TFLOP/s of stored entries, twice that
// on the matrix cores).  What bounds it now: no unit alone.  Of the 54500 cycles a wave of that launch lives
// the vector units are busy 25000 (decoding), LDS 28300 (12400 of them bank conflicts) and the matrix cores
// 12300, by the counters; waves wait for 40 % of their cycles, for one another and for X out of L2.
//
// A zero of the dense chunk times an Inf or NaN of X is a NaN that the sparse product does not have
// (it never reads columns without an entry).  Such a product can only make a sum non-finite, so every
// sum that is not finite is computed again from its row's entries alone.
#include <atomic>

#include "macko_packed.h"
#include "macko_spmv_detail.h"

namespace macko {
namespace {

using namespace spmv_detail;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kTileWaves = 16;
constexpr int kTileThreads = kTileWaves * kWave;
constexpr int kRowUnit = 4;      // row blocks start at multiples of 4 rows (8-byte stores of Y)
constexpr int kTilePad = 8;      // spare columns behind every row of the dense chunk, 16 bytes
constexpr int kTileFront = 16;   // the same in front of the first row
// Elements of X (batch * cols) from which on it is brought into operand order first.  Packing is a
// launch of its own, about 3 us back to back (4.9 in a kernel trace, which counts the dispatch); read as it is, a wave's load touches 16 cache lines instead of 8
// whole ones and L2 delivers about 14 instead of 48 bytes a cycle to a compute unit, by the launches' times (4096 x 4096 at density
// 0.5: 16 vectors 9.7 us as they are and 10.8 packed, 24 vectors 12.0 and 11.4, 128 vectors 26 and 18).
// Vectors that are not 16-byte aligned cost a second line per lane: packed from 4 vectors on (777 x 3333,
// 4 vectors: 8.8 us as they are, 7.5 packed).
constexpr long long kPackFrom = 100000;
constexpr long long kPackUnalignedFrom = 12000;

// One of the matrices of a launch.  Several with the same columns and vectors stand below each other; their rows
// are numbered on, and where there is more than one, every one but the last ends on a whole unit of four rows.
struct TileSource {
    const u32 *values;
    const u32 *deltas;
    const int *row_ptr;
    uint16_t *y;
    int first;   // its first row; behind the last matrix: no row
    u32 padded;
    u32 ldy;
};
constexpr int kMaxSources = MACKO_PACKED_MATRICES;

// What a launch of one matrix and one of several have in common, and the launch's arguments: with one matrix a wave
// fetches no more of them than it needs (4096 x 4096, 8 vectors: 0.15 us a launch).
struct TileCommon {
    const uint16_t *x;
    int rows, cols, batch;   // rows of all matrices
    u32 ldx;
    int chunk;            // columns per chunk, a multiple of 64
    int n_chunks;
    u32 units_q, units_rem;  // 4-row units per row block (even_split)
    int vector_blocks;
    int group_shift;      // log2 of the number of vector groups of a workgroup (1, 2, 4)
    int vector_store;     // 8-byte stores of Y are aligned
    const u32x4 *packed;  // X in operand order (pack_vectors_kernel), null: read X itself
    int packed_tiles;     // vector tiles in it
    int packed_steps;     // 64-column steps in it
    const uint16_t *residual;  // added to Y before it is rounded (laid out like Y, may be Y), or null
};
template <int SOURCES>
struct TileArgs : TileCommon {
    TileSource source[SOURCES];
};

__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// v clamped to [lo, hi], signed; lo differs from lane to lane or sits in a vector register anyway, hi
// is wave-uniform (one instruction; the compiler makes three of a minimum and a maximum)
__device__ __forceinline__ u32 clamp_between(u32 v, int lo, int hi)
{
    u32 r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(lo), "s"(hi));
    return r;
}

// sum of row [e0, e1)'s entries times one vector (x(c): its element c as bits), by one wave; columns
// clamped to the vector
template <typename X>
__device__ __forceinline__ float exact_row_times_vector(const u32 *values, const u32 *deltas, u32 e0, u32 e1, X x, int cols)
{
    const int lane = threadIdx.x & (kWave - 1);
    const uint16_t *vals = reinterpret_cast<const uint16_t *>(values);
    const unsigned char *nibs = reinterpret_cast<const unsigned char *>(deltas);
    float acc = 0.f;
    int column = -1;
    for (u32 j0 = e0; j0 < e1; j0 += kWave) {
        const u32 j = j0 + lane;
        int step = 0;
        float v = 0.f;
        if (j < e1) {
            step = ((nibs[j >> 1] >> (4 * (j & 1))) & 15) + 1;
            v = half_bits_to_float(vals[j]);
        }
        const int incl = wave_scan_inclusive(step);
        int c = column + incl;
        c = c < 0 ? 0 : (c >= cols ? cols - 1 : c);
        if (j < e1) acc = __builtin_fmaf(v, half_bits_to_float(x(c)), acc);
        column += __builtin_amdgcn_readlane(incl, kWave - 1);
    }
    return wave_sum(acc);
}

// X in operand order (macko_packed.h).  A wave packs one block.
__global__ void __launch_bounds__(256) pack_vectors_kernel(const uint16_t *__restrict__ x, u32x4 *__restrict__ packed,
                                                           int cols, int batch, u32 ldx, int tiles, int blocks)
{
    const int block = blockIdx.x * 4 + uniform(threadIdx.x >> 6);
    if (block >= blocks) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int k64 = block / tiles, tile = block - k64 * tiles;
    const int piece = k64 * 8 + (lane & 7), k = piece * 8;
    const int last_piece = cols - 8;
    u32x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int n = tile * 16 + h * 8 + (lane >> 3);
        const u32 row = (u32)(n < batch ? n : batch - 1) * ldx;
        __builtin_memcpy(&v[h], x + row + (u32)(k < last_piece ? k : last_piece), 16);
        if (n >= batch) v[h] = u32x4{0u, 0u, 0u, 0u};
    }
    if (k64 * 64 + 64 > cols) {
        const int by = k > last_piece ? k - last_piece : 0;
        v[0] = shift_down(v[0], by);
        v[1] = shift_down(v[1], by);
    }
    u32x4 *dst = packed + packed_piece(piece, tile * 16 + (lane >> 3), tiles);
    dst[0] = v[0];
    dst[8] = v[1];
}

// SEVERAL: more than one matrix, which a wave looks up for each of its rows.
template <int RT, int NTW, int SC, bool PACKED, bool SEVERAL>
__global__ void __launch_bounds__(kTileThreads) spmv_tile_kernel(const TileArgs<SEVERAL ? kMaxSources : 1> a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    typedef __attribute__((address_space(3))) u32x4 *lds_w32x4;
    typedef __attribute__((address_space(3))) uint16_t *lds_w16;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = uniform(tid >> 6);
    const int sub = lane & 15, quarter = lane >> 4;

    // Workgroups go round-robin to the 8 XCDs: XCD k takes the k-th contiguous eighth, vector blocks
    // of one row block next to each other, so that they share the matrix behind one L2.
    u32 id = blockIdx.x;
    if ((gridDim.x & 7) == 0) id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const u32 row_block = id / (u32)a.vector_blocks;
    const int vector0 = (int)(id - row_block * (u32)a.vector_blocks) * ((NTW * 16) << a.group_shift);
    const int row0 = (int)even_split(row_block, a.units_q, a.units_rem) * kRowUnit;
    const int row_end_unclamped = (int)even_split(row_block + 1, a.units_q, a.units_rem) * kRowUnit;
    const int row1 = row_end_unclamped < a.rows ? row_end_unclamped : a.rows;
    const int group = wave & ((1 << a.group_shift) - 1);
    const int part = wave >> a.group_shift;
    const int parts = kTileWaves >> a.group_shift;

    auto source_of = [&](int row) __attribute__((always_inline)) {
        int m = 0;
        if constexpr (SEVERAL)
            for (int k = 1; k < kMaxSources; ++k) m += row >= a.source[k].first ? 1 : 0;
        return m;
    };
    __amdgpu_buffer_rsrc_t rs_values[SEVERAL ? RT : 1], rs_deltas[SEVERAL ? RT : 1];
    auto describe = [&](int slot, const TileSource &m) __attribute__((always_inline)) {
        rs_values[slot] = __builtin_amdgcn_make_buffer_rsrc((void *)m.values, 0, (int)(m.padded * 2), 0x00020000);
        rs_deltas[slot] = __builtin_amdgcn_make_buffer_rsrc((void *)m.deltas, 0, (int)(m.padded / 2), 0x00020000);
    };
    if constexpr (!SEVERAL) describe(0, a.source[0]);

    // ---- my rows: row j of mine is row (wave + 16 j) of the block.  pos: next entry (a multiple of 8),
    //      end: behind the row's last entry, col: column of the entry in front of pos ------------------
    int pos[RT], end[RT], col[RT];
    u32x4 tile_v[RT];
    u32 tile_d[RT];
    auto request = [&](auto slot) __attribute__((always_inline)) {
        constexpr int J = decltype(slot)::value;
        const bool any = pos[J] < end[J];
        const u32 vo = any ? (u32)pos[J] * 2 + (u32)lane * 16 : kNoTileValues;
        const u32 dof = any ? ((u32)pos[J] >> 1) + (u32)lane * 4 : kNoTileDeltas;
        tile_v[J] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_values[SEVERAL ? J : 0], (int)vo, 0, 0));
        tile_d[J] = __builtin_amdgcn_raw_buffer_load_b32(rs_deltas[SEVERAL ? J : 0], (int)dof, 0, 0);
    };
    int begin[RT];  // the row's first entry: what stands in front of it in its group of 8 is the row before's
    static_for<RT>([&](auto slot) {
        constexpr int J = decltype(slot)::value;
        const int row = row0 + wave + 16 * J;
        const TileSource &m = a.source[source_of(row)];
        if constexpr (SEVERAL) describe(J, m);
        u32 e0 = 0, e1 = 0;
        if (row < row1) {
            const int *row_ptr = m.row_ptr + (SEVERAL ? row - m.first : row);
            e0 = (u32)uniform(row_ptr[0]);
            e1 = (u32)uniform(row_ptr[1]);
            e0 = e0 < m.padded ? e0 : m.padded;
            e1 = e1 < m.padded ? e1 : m.padded;
        }
        if (e1 < e0) e1 = e0;
        begin[J] = (int)e0;
        pos[J] = (int)(e0 & ~7u);
        end[J] = e1 == e0 ? pos[J] : (int)e1;
        col[J] = -1 - (int)(e0 & 7u);
        request(slot);
    });

    float4v acc[RT][NTW];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NTW; ++t) acc[r][t] = float4v{0.f, 0.f, 0.f, 0.f};

    const u32 stride = (u32)a.chunk * 2 + kTilePad * 2;   // bytes per row of the dense chunk
    const u32 buffer_bytes = stride * (16 * RT);
    const u32 lds0 = (u32)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds + kTileFront;

    // byte offset of vector n's first column in X, per vector tile of mine
    u32 x_off[NTW];
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
        int n = vector0 + (group * NTW + t) * 16 + sub;
        n = n < a.batch ? n : a.batch - 1;
        x_off[t] = (u32)n * a.ldx * 2;
    }
    const int last_piece = a.cols - 8;  // where the last whole piece of 8 columns starts

    // ---- X: 64 columns per step, in operand order: packed, two kilobyte loads per vector tile and
    //      step; else lane (sub, quarter) takes columns 16 quarter .. + 15 of vector sub ---------------
    u32x4 b[SC][NTW][2];
    auto request_vectors = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SC; ++i) {
            const int k64 = c * a.chunk + (part + parts * i) * 64;
            if constexpr (PACKED) {
                int step = k64 >> 6;
                step = step < a.packed_steps ? step : a.packed_steps - 1;
#pragma unroll
                for (int t = 0; t < NTW; ++t) {
                    int tile = (vector0 >> 4) + group * NTW + t;
                    tile = tile < a.packed_tiles ? tile : a.packed_tiles - 1;
                    const u32x4 *block = a.packed + (size_t)(u32)(step * a.packed_tiles + tile) * kBlockPieces;
                    b[i][t][0] = block[lane];
                    b[i][t][1] = block[lane + 64];
                }
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    int k = k64 + quarter * 16 + s * 8;
                    k = k < last_piece ? k : last_piece;
#pragma unroll
                    for (int t = 0; t < NTW; ++t)
                        __builtin_memcpy(&b[i][t][s], reinterpret_cast<const unsigned char *>(a.x) + (x_off[t] + (u32)k * 2), 16);
                }
            }
        }
    };

    // ---- my rows' part of a chunk, dense, into LDS; then the entries of the chunk behind it are requested
    auto scatter = [&](int c) __attribute__((always_inline)) {
        const int c0 = c * a.chunk;
        const u32 buffer = lds0 + (c & 1 ? buffer_bytes : 0u);
        static_for<RT>([&](auto slot) {
            constexpr int J = decltype(slot)::value;
            const u32 row_addr = buffer + (u32)(wave + 16 * J) * stride;
            for (u32 o = (u32)lane * 16; o < (u32)a.chunk * 2; o += kWave * 16)
                *(lds_w32x4)(uintptr_t)(row_addr + o) = u32x4{0u, 0u, 0u, 0u};
            // entries whose column lies outside the chunk go to the spare columns around the row
            const int lo = (int)row_addr - kTilePad * 2, hi = (int)row_addr + a.chunk * 2;
            auto pass = [&]() __attribute__((always_inline)) -> bool {  // true: the chunk goes on behind this tile
                u32x4 v = tile_v[J];
                u32 d = tile_d[J];
                if (pos[J] < begin[J] && lane == 0) d &= ~0u << (4 * (begin[J] - pos[J]));
                if (pos[J] + kTile > end[J]) {  // behind the row's end: zeros at columns nothing else takes
                    const int left = end[J] - pos[J] - lane * kChunk;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const u32 keep = left >= 2 * w + 2 ? ~0u : (left == 2 * w + 1 ? 0xffffu : 0u);
                        v[w] &= keep;
                    }
                }
                const u32 step = __builtin_amdgcn_udot8(d, 0x22222222u, 16u, false);
                const u32 incl = (u32)wave_scan_inclusive((int)step);
                const u32 origin = row_addr + 2u * (u32)(col[J] - c0);
                const u32 base = origin + 2u + (incl - step);
                if ((int)base < hi) {  // lanes wholly behind the chunk write nothing
                    u32 at[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) at[k] = __builtin_amdgcn_udot8(d, twos_upto(k), base, false);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 8; ++k) at[k] = clamp_between(at[k], lo, hi);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const u32 w = v[k >> 1];
                        *(lds_w16)(uintptr_t)(at[k] + 2u * k) = (uint16_t)((k & 1) ? w >> 16 : w);
                    }
                }
                // lanes whose last entry lies behind the chunk stay for the next one
                const unsigned long long stay = __ballot((int)(origin + incl) >= hi);
                if (stay == 0) {
                    pos[J] += kTile;
                    col[J] += __builtin_amdgcn_readlane((int)incl, kWave - 1) >> 1;
                    return pos[J] < end[J];
                }
                const int f = __builtin_ctzll(stay);
                pos[J] += f * kChunk;
                col[J] += __builtin_amdgcn_readlane((int)(incl - step), f) >> 1;
                return false;
            };
            if (pos[J] < end[J]) {
                bool more = pass();
                while (__builtin_expect(more, 0)) {
                    request(slot);
                    more = pass();
                }
            }
        });
        static_for<RT>([&](auto slot) { request(slot); });
    };

    auto multiply = [&](int c) __attribute__((always_inline)) {
        const int c0 = c * a.chunk;
        const u32 buffer = lds0 + (c & 1 ? buffer_bytes : 0u);
#pragma unroll
        for (int i = 0; i < SC; ++i) {
            const int step = part + parts * i;
            const int k64 = c0 + step * 64;
            if (step * 64 < a.chunk && k64 < a.cols) {
                if (!PACKED && k64 + 64 > a.cols) {  // columns beyond the vectors: zeros
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int k = k64 + quarter * 16 + s * 8;
                        const int by = k > last_piece ? k - last_piece : 0;
#pragma unroll
                        for (int t = 0; t < NTW; ++t) b[i][t][s] = shift_down(b[i][t][s], by);
                    }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const u32 at = buffer + (u32)sub * stride + (u32)(step * 64 + quarter * 16 + s * 8) * 2;
                    u32x4 av[RT];
#pragma unroll
                    for (int r = 0; r < RT; ++r) av[r] = *(lds_w32x4)(uintptr_t)(at + (u32)(16 * r) * stride);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int t = 0; t < NTW; ++t)
                            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, av[r]),
                                                                               __builtin_bit_cast(half8, b[i][t][s]),
                                                                               acc[r][t], 0, 0, 0);
                }
            }
        }
    };

    // Between two barriers every wave multiplies chunk c and scatters chunk c + 1; half of the waves of
    // every SIMD do it in one order and half in the other, so that matrix cores, vector units and LDS
    // work side by side.
    scatter(0);
    const int last = a.n_chunks - 1;
    if ((wave >> 2) & 1) {
        request_vectors(0);
        lds_barrier();
        for (int c = 0; c < last; ++c) {
            multiply(c);
            __builtin_amdgcn_sched_barrier(0);
            request_vectors(c + 1);
            __builtin_amdgcn_sched_barrier(0);
            scatter(c + 1);
            lds_barrier();
        }
    } else {
        lds_barrier();
        for (int c = 0; c < last; ++c) {
            request_vectors(c);
            __builtin_amdgcn_sched_barrier(0);
            scatter(c + 1);
            multiply(c);
            lds_barrier();
        }
        request_vectors(last);
    }
    multiply(last);
    lds_barrier();

    // ---- the partial sums of a vector tile meet in LDS: [row tile][vector tile][part], 1 KB each ---------
    const int groups = 1 << a.group_shift;
    const u32 red = lds0 - kTileFront;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
            const u32 slot = (u32)((r * groups + group) * NTW + t) * (u32)parts + (u32)part;
            *(lds_w32x4)(uintptr_t)(red + slot * 1024 + (u32)lane * 16) = __builtin_bit_cast(u32x4, acc[r][t]);
        }
    lds_barrier();
    const int n_tiles = RT * groups * NTW;
    for (int tile = wave; tile < n_tiles; tile += kTileWaves) {
        float4v sum = float4v{0.f, 0.f, 0.f, 0.f};
        for (int p = 0; p < parts; ++p)
            sum += __builtin_bit_cast(float4v, *(lds_w32x4)(uintptr_t)(red + (u32)(tile * parts + p) * 1024 + (u32)lane * 16));
        const int r = tile / (groups * NTW);
        const int n = vector0 + (tile - r * groups * NTW) * 16 + sub;
        const int row = row0 + r * 16 + quarter * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float one = sum[i];
            const u32 bits = __builtin_bit_cast(u32, one);
            unsigned long long bad = __ballot(n < a.batch && row + i < row1 && (bits & 0x7f800000u) == 0x7f800000u);
            while (__builtin_expect(bad != 0, 0)) {
                const int L = __builtin_ctzll(bad);
                bad &= bad - 1;
                const int bad_row = __builtin_amdgcn_readlane(row, L) + i;
                const int bad_n = __builtin_amdgcn_readlane(n, L);
                const TileSource &m = a.source[source_of(bad_row)];
                const int *row_ptr = m.row_ptr + (SEVERAL ? bad_row - m.first : bad_row);
                u32 e0 = (u32)uniform(row_ptr[0]), e1 = (u32)uniform(row_ptr[1]);
                e0 = e0 < m.padded ? e0 : m.padded;
                e1 = e1 < m.padded ? e1 : m.padded;
                const float exact = exact_row_times_vector(
                    m.values, m.deltas, e0, e1,
                    [&](int c) {
                        if constexpr (PACKED)
                            return reinterpret_cast<const uint16_t *>(a.packed + packed_piece(c >> 3, bad_n, a.packed_tiles))[c & 7];
                        else
                            return a.x[(size_t)bad_n * a.ldx + (size_t)c];
                    },
                    a.cols);
                sum[i] = lane == L ? exact : sum[i];
            }
        }
        if (n < a.batch) {
            uint16_t *y = a.source[0].y;
            u32 ldy = a.source[0].ldy;
            int at = row;
            if constexpr (SEVERAL) {  // my four rows are of one matrix
#pragma unroll
                for (int k = 1; k < kMaxSources; ++k)
                    if (row >= a.source[k].first) {
                        y = a.source[k].y;
                        ldy = a.source[k].ldy;
                        at = row - a.source[k].first;
                    }
            }
            uint16_t *dst = y + (size_t)n * ldy + at;
            if (!SEVERAL && a.residual != nullptr) {
                const uint16_t *add = a.residual + (size_t)n * ldy + row;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row + i < row1) sum[i] += half_bits_to_float(add[i]);
            }
            if (a.vector_store && row + 4 <= row1) {
                const u32 lo = (u32)float_to_half_bits(sum[0]) | ((u32)float_to_half_bits(sum[1]) << 16);
                const u32 hi = (u32)float_to_half_bits(sum[2]) | ((u32)float_to_half_bits(sum[3]) << 16);
                *reinterpret_cast<u32x2 *>(dst) = u32x2{lo, hi};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row + i < row1) dst[i] = float_to_half_bits(sum[i]);
            }
        }
    }
}

template <int RT, int NTW, int SC, bool PACKED, bool SEVERAL>
int launch_tile(const TileArgs<kMaxSources> &all, unsigned grid, size_t lds_bytes, hipStream_t stream)
{
    TileArgs<SEVERAL ? kMaxSources : 1> a;
    static_cast<TileCommon &>(a) = all;
    for (int k = 0; k < (SEVERAL ? kMaxSources : 1); ++k) a.source[k] = all.source[k];
    auto kernel = spmv_tile_kernel<RT, NTW, SC, PACKED, SEVERAL>;
    if (lds_bytes > 64 * 1024) {
        // one-time opt-in to more than 64 KiB of dynamic LDS, per device and kernel
        static std::atomic<bool> done[64];
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        if (dev < 0 || dev >= 64 || !done[dev].load(std::memory_order_acquire)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            if (dev >= 0 && dev < 64) done[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kTileThreads), lds_bytes, stream, a);
    return (int)hipGetLastError();
}

TileArgs<kMaxSources> no_matrices()
{
    TileArgs<kMaxSources> a{};
    for (TileSource &m : a.source) m.first = 0x7fffffff;
    return a;
}

size_t tile_lds_bytes(const TileShape &s)
{
    const size_t dense = kTileFront + 2 * (size_t)(16 * s.row_tiles) * ((size_t)s.chunk * 2 + kTilePad * 2);
    const size_t sums = (size_t)s.row_tiles * s.wave_tiles * kTileWaves * 1024;
    return dense > sums ? dense : sums;
}

int launch_tile_shape(TileArgs<kMaxSources> a, const TileShape &s, int max_lds, hipStream_t stream)
{
    const int groups = 1 << s.group_shift, parts = kTileWaves / groups;
    const size_t lds = tile_lds_bytes(s);
    const long long units = (a.rows + kRowUnit - 1) / kRowUnit;
    if (lds > (size_t)max_lds || s.chunk % 64 != 0 || s.chunk <= 0 || s.chunk > 64 * parts * s.steps || s.row_blocks < 1 ||
        (units + s.row_blocks - 1) / s.row_blocks > 4 * s.row_tiles)
        return MACKO_E_INVALID_ARGUMENT;
    a.chunk = s.chunk;
    a.n_chunks = (a.cols + s.chunk - 1) / s.chunk;
    a.units_q = (u32)(units / s.row_blocks);
    a.units_rem = (u32)(units % s.row_blocks);
    a.group_shift = s.group_shift;
    const int vectors = 16 * s.wave_tiles * groups;
    a.vector_blocks = (a.batch + vectors - 1) / vectors;
    const bool several = a.source[1].first < a.rows;
    a.vector_store = 1;
    for (const TileSource &m : a.source)
        if (m.first < a.rows && (m.ldy % 4 != 0 || (reinterpret_cast<uintptr_t>(m.y) & 7) != 0)) a.vector_store = 0;
    const long long grid = s.row_blocks * a.vector_blocks;
    if (grid >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
    a.packed_tiles = packed_tiles(a.batch);
    a.packed_steps = packed_steps(a.cols);
#define MACKO_TILE(RT_, NTW_, SC_)                                                                                 \
    if (s.row_tiles == RT_ && s.wave_tiles == NTW_ && s.steps == SC_) {                                            \
        if (several) return launch_tile<RT_, NTW_, SC_, true, true>(a, (unsigned)grid, lds, stream);               \
        if (a.packed != nullptr) return launch_tile<RT_, NTW_, SC_, true, false>(a, (unsigned)grid, lds, stream);  \
        return launch_tile<RT_, NTW_, SC_, false, false>(a, (unsigned)grid, lds, stream);                          \
    }
    MACKO_TILE(1, 1, 1) MACKO_TILE(2, 1, 1) MACKO_TILE(3, 1, 1)
    MACKO_TILE(1, 1, 2) MACKO_TILE(2, 1, 2) MACKO_TILE(3, 1, 2)
    MACKO_TILE(1, 2, 1) MACKO_TILE(2, 2, 1) MACKO_TILE(3, 2, 1)
    MACKO_TILE(1, 2, 2) MACKO_TILE(2, 2, 2) MACKO_TILE(3, 2, 2)
#undef MACKO_TILE
    return MACKO_E_INVALID_ARGUMENT;
}


// Estimated cycles of a launch: what one workgroup's chunk asks of the vector units (about 60
// instructions per row and 512 entries), of the path from L2 (X: 48 bytes a cycle from operand order,
// 14 from X itself with 16 vectors, and with one vector half the time: fewer cache lines a load), of LDS
// and of the matrix cores overlaps to about 0.6 of the sum, behind a start and an end of about 9000 cycles.
double tile_cost(const TileShape &s, long long units, int cols, double density, int batch, bool packed, int compute_units)
{
    const int groups = 1 << s.group_shift;
    const int vectors = 16 * s.wave_tiles * groups;
    const long long workgroups = s.row_blocks * ((batch + vectors - 1) / vectors);
    const double rounds = (double)((workgroups + compute_units - 1) / compute_units);
    const double rows = 4.0 * (double)((units + s.row_blocks - 1) / s.row_blocks);
    const double passes = density * s.chunk / 504.0 > 1.0 ? density * s.chunk / 504.0 : 1.0;
    const double chunk = s.chunk;
    const double valu = rows * passes * 60.0;
    const double x = vectors * chunk * 2.0 * (packed ? 1.0 / 48.0 : (0.5 + (batch < 16 ? batch / 32.0 : 0.5)) / 14.0);
    const double lds = rows * passes * 53.0 + rows * chunk / 64.0 + groups * 16.0 * s.row_tiles * chunk / 64.0;
    const double mfma = s.row_tiles * (vectors / 16) * chunk / 8.0;
    const int n_chunks = (cols + s.chunk - 1) / s.chunk;
    return rounds * (9000.0 + 0.6 * n_chunks * (valu + x + lds + mfma));
}

// The shape of a launch.  Small batches: one vector tile per workgroup and all 16 waves on different
// columns.  From 5 vector tiles on blocks of 64 and of 128 vectors are both looked at: blocks of 128
// decode a row once instead of twice, blocks of 64 read half as much of X per workgroup, which wins
// where there are few rows per compute unit (4096 x 4096, density 0.5, 128 vectors: 18.3 us against
// 20.4; 11008 x 4096: 39.4 against 28.4).
bool choose_tile_shape(TileShape *best, int rows, int cols, long long padded, int batch, bool packed, const DeviceInfo &info,
                       double *cycles = nullptr)
{
    const long long units = ((long long)rows + kRowUnit - 1) / kRowUnit;
    const double density = (double)padded / ((double)rows * (double)cols);
    const int tiles = (batch + 15) / 16;
    double least = 0.0;
    bool found = false;
    for (int shift = tiles <= 1 ? 0 : (tiles <= 4 ? 1 : 2); shift >= (tiles > 4 ? 1 : (tiles <= 1 ? 0 : 1)); --shift) {
        TileShape s;
        s.group_shift = shift;
        s.wave_tiles = tiles > 2 ? 2 : 1;
        const int vectors = (16 * s.wave_tiles) << shift;
        const int blocks = (batch + vectors - 1) / vectors;
        const int parts = kTileWaves >> shift;
        // as many workgroups as compute units, or a whole number of times that, in blocks of at most 48 rows
        const long long fewest = (units * blocks + 12ll * info.compute_units - 1) / (12ll * info.compute_units);
        for (long long k = fewest; k < fewest + 3; ++k) {
            s.row_blocks = info.compute_units * k / blocks;
            if (s.row_blocks * 12 < units) s.row_blocks = (units + 11) / 12;
            if (s.row_blocks > units) s.row_blocks = units;
            const long long per_block = (units + s.row_blocks - 1) / s.row_blocks;
            s.row_tiles = (int)((per_block + 3) / 4);
            // columns per chunk: what LDS holds twice, what a wave's registers hold of X, and no more
            // entries per row than one tile has (with a margin for the spread between rows)
            int chunk = 64 * parts * 2;
            const int by_lds = ((info.max_lds_bytes - kTileFront) / (2 * 16 * s.row_tiles) - 2 * kTilePad) / 2;
            const int by_density = density > 0.1 ? (int)(470.0 / density) : 4096;
            chunk = chunk < by_lds ? chunk : by_lds;
            chunk = chunk < by_density ? chunk : by_density;
            chunk = chunk < 64 ? 64 : chunk / 64 * 64;
            const int n_chunks = (cols + chunk - 1) / chunk;
            s.chunk = ((cols + n_chunks - 1) / n_chunks + 63) / 64 * 64;
            s.steps = s.chunk > 64 * parts ? 2 : 1;
            if (tile_lds_bytes(s) > (size_t)info.max_lds_bytes) break;
            const double cost = tile_cost(s, units, cols, density, batch, packed, info.compute_units);
            if (!found || cost < least) {
                found = true;
                least = cost;
                *best = s;
            }
            if (s.row_tiles == 1) break;  // smaller blocks only read X more often
        }
    }
    if (cycles != nullptr) *cycles = least;
    return found;
}

}  // namespace

// Whether this kernel can do a product of several vectors (which it should do: batched_on_tiles, macko_spmv.hip).
bool spmv_tile_takes(int rows, int cols, long long padded, int batch, long long ldx)
{
    if (rows == 0 || padded == 0 || cols < 64) return false;
    // offsets into X and into its operand-order copy are 32-bit
    return (long long)batch * ldx * 2 < (1ll << 32) && (long long)packed_bytes(cols, batch) < (1ll << 32);
}

// The time by the cost above, at 2.4 GHz, and the packing launch.  Right to about 10 % on either side where it
// decides about the route (28672 x 4096, 8 vectors, density 0.05: 40.7 us, estimated 40; 5120 x 13824, 8, 0.1: 24.4, 21).
int spmv_tile_estimate(int rows, int cols, long long padded, int batch, bool packed, const DeviceInfo &info, TileShape *shape, double *us)
{
    double cycles = 0.0;
    if (!choose_tile_shape(shape, rows, cols, padded, batch, packed, info, &cycles)) return MACKO_E_INVALID_ARGUMENT;
    *us = cycles * (1.06 / 2400.0) + (packed ? 2.9 : 0.0);
    return 0;
}

size_t spmv_tile_workspace(int cols, int batch, const void *x, long long ldx)
{
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) & 15) == 0) && (ldx & 7) == 0;
    if ((long long)batch * cols < (aligned || batch < 4 ? kPackFrom : kPackUnalignedFrom)) return 0;
    return packed_bytes(cols, batch);
}

int spmv_tile_launch(const SpmvArgs &args, int batch, const TileShape &shape, void *workspace, const DeviceInfo &info, hipStream_t stream)
{
    TileArgs<kMaxSources> a = no_matrices();
    a.source[0] = TileSource{args.values, args.deltas, args.row_ptr, args.y, 0, (u32)args.padded, (u32)args.ldy};
    a.x = args.x;
    a.rows = args.rows;
    a.cols = args.cols;
    a.batch = batch;
    a.ldx = (u32)args.ldx;
    if (workspace != nullptr) {
        const int e = spmv_tile_pack(args.x, args.cols, batch, args.ldx, workspace, stream);
        if (e != 0) return e;
        a.packed = (const u32x4 *)workspace;
    }
    return launch_tile_shape(a, shape, info.max_lds_bytes, stream);
}

int spmv_tile_pack(const uint16_t *x, int cols, int batch, long long ldx, void *packed, hipStream_t stream)
{
    const int tiles = packed_tiles(batch), blocks = tiles * packed_steps(cols);
    hipLaunchKernelGGL(pack_vectors_kernel, dim3((blocks + 3) / 4), dim3(256), 0, stream, x, (u32x4 *)packed, cols, batch, (u32)ldx,
                       tiles, blocks);
    return (int)hipGetLastError();
}

}  // namespace macko

namespace macko {
namespace {

int packed_product(const macko_packed_matrix *matrices, int n, const void *packed, const void *residual, int cols, int batch, void *stream)
{
    if (matrices == nullptr || n < 1 || n > kMaxSources || cols < 64 || batch < 1 || (n > 1 && residual != nullptr)) return MACKO_E_INVALID_ARGUMENT;
    TileArgs<kMaxSources> a = no_matrices();
    long long rows = 0, padded = 0;
    int used = 0;
    for (int k = 0; k < n; ++k) {
        const macko_packed_matrix &m = matrices[k];
        if (m.rows < 0 || m.padded_entries < 0 || m.padded_entries % kChunk != 0 || m.padded_entries >= (1ll << 31) - 8192 ||
            m.ldy < m.rows || m.ldy >= (1ll << 31))
            return MACKO_E_INVALID_ARGUMENT;
        if (m.rows == 0) continue;
        if (m.row_ptr == nullptr || m.y == nullptr || packed == nullptr ||
            (m.padded_entries > 0 && (m.values == nullptr || m.deltas == nullptr)) || packed_bytes(cols, batch) >= (1ull << 32))
            return MACKO_E_INVALID_ARGUMENT;
        if ((reinterpret_cast<uintptr_t>(m.values) & 15) || (reinterpret_cast<uintptr_t>(m.deltas) & 3) ||
            (reinterpret_cast<uintptr_t>(m.row_ptr) & 3) || (reinterpret_cast<uintptr_t>(packed) & 15) ||
            (reinterpret_cast<uintptr_t>(residual) & 1) || (reinterpret_cast<uintptr_t>(m.y) & 1))
            return MACKO_E_INVALID_ARGUMENT;
        if (rows % kRowUnit != 0) return MACKO_E_INVALID_ARGUMENT;  // the matrix in front does not end on a whole unit
        a.source[used++] = TileSource{(const u32 *)m.values, (const u32 *)m.deltas, m.row_ptr, (uint16_t *)m.y, (int)rows,
                                      (u32)m.padded_entries, (u32)m.ldy};
        rows += m.rows;
        padded += m.padded_entries;
        if (used > 1 && rows >= (1ll << 31) - kRowUnit) return MACKO_E_INVALID_ARGUMENT;
    }
    if (rows == 0) return 0;
    DeviceInfo info;
    const int rc = device_info(&info);
    if (rc != 0) return rc;
    a.rows = (int)rows;
    a.cols = cols;
    a.batch = batch;
    a.packed = (const u32x4 *)packed;
    a.residual = (const uint16_t *)residual;
    TileShape shape;
    if (!choose_tile_shape(&shape, a.rows, cols, padded, batch, true, info)) return MACKO_E_INVALID_ARGUMENT;
    return launch_tile_shape(a, shape, info.max_lds_bytes, as_stream(stream));
}

}  // namespace
}  // namespace macko

// Products of vectors that are in operand order already: several matrices share one packing, and
// what produces the vectors writes them that way (macko_prefill.hip).  No upstream counterpart.
extern "C" int macko_packed_bytes(int32_t cols, int32_t batch, int64_t *bytes)
{
    using namespace macko;
    if (bytes == nullptr || cols < 64 || batch < 1 || packed_bytes(cols, batch) >= (1ull << 32)) return MACKO_E_INVALID_ARGUMENT;
    *bytes = (int64_t)packed_bytes(cols, batch);
    return 0;
}

extern "C" int macko_pack_f16(const void *x, int32_t cols, int32_t batch, int64_t ldx, void *packed, void *stream)
{
    using namespace macko;
    if (x == nullptr || packed == nullptr || cols < 64 || batch < 1 || ldx < cols || (reinterpret_cast<uintptr_t>(x) & 1) ||
        (reinterpret_cast<uintptr_t>(packed) & 15) || packed_bytes(cols, batch) >= (1ull << 32) ||
        (long long)batch * ldx * 2 >= (1ll << 32))
        return MACKO_E_INVALID_ARGUMENT;
    return spmv_tile_pack((const uint16_t *)x, cols, batch, ldx, packed, as_stream(stream));
}

extern "C" int macko_spmv_f16_packed(const void *values, const void *deltas, const int32_t *row_ptr, const void *packed,
                                     const void *residual, void *y, int32_t rows, int32_t cols, int64_t padded_entries,
                                     int32_t batch, int64_t ldy, void *stream)
{
    using namespace macko;
    const macko_packed_matrix one = {values, deltas, row_ptr, y, rows, padded_entries, ldy};
    return packed_product(&one, 1, packed, residual, cols, batch, stream);
}

extern "C" int macko_spmv_f16_packed_several(const macko_packed_matrix *matrices, int32_t n_matrices, const void *packed,
                                             int32_t cols, int32_t batch, void *stream)
{
    return macko::packed_product(matrices, n_matrices, packed, nullptr, cols, batch, stream);
}
