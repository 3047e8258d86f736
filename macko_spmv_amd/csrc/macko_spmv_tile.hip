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
// on the matrix cores; spmv_pipe_kernel below takes such products now, 23.6 with packing, 27.9 here).  What bounds it: no unit alone.  Of the 54500 cycles a wave of that launch lives
// the vector units are busy 25000 (decoding), LDS 28300 (12400 of them bank conflicts) and the matrix cores
// 12300, by the counters; waves wait for 40 % of their cycles, for one another and for X out of L2.
//
// A zero of the dense chunk times an Inf or NaN of X is a NaN that the sparse product does not have
// (it never reads columns without an entry).  Such a product can only make a sum non-finite, so every
// sum that is not finite is computed again from its row's entries alone.
#include <atomic>
#include <cmath>

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

// One of the matrices of a launch.
struct TileSource {
    uint16_t *y;
    u32 ldy;
    u32 padded;
    const u32 *values;
    const u32 *deltas;
    const int *row_ptr;
};
constexpr int kMaxSources = MACKO_PACKED_MATRICES;

// Several with the same columns and vectors stand below each other; their rows are numbered on, and every one but the
// last ends on a whole unit of four rows.  first: a matrix's first row; behind the last matrix: no row.
// unit_rows: what row blocks are whole multiples of, kRowUnit or 2 * kRowUnit.  Then the launch has two matrices of as many rows, gate
// and up, whose units of four rows alternate, and the results are not the products but silu(gate) * up, in operand order at source[0].y:
// the two rows of an element are 16 lanes apart where a launch's sums come together.  11008 x 4096 each at 0.5, 128 vectors: 54.3 us and
// 5.0 for the gate's own launch, now 55.4 (kernel trace; 2 us a layer by the clock, 6 where launches are what a layer takes).
template <int SOURCES>
struct TileSources {
    TileSource source[SOURCES];
    int first[SOURCES];
    int unit_rows;
};
template <>
struct TileSources<1> {
    TileSource source[1];
};

// What a launch of one matrix and one of several have in common.  A launch's arguments are its matrices, then these; with
// one matrix a wave fetches no more of them than it needs (4096 x 4096, 8 vectors: 0.15 us a launch).  They end, and the grid's
// size behind them stands, within 128 bytes, and what the loop needs is fetched at once, in front of row_ptr: 8.53 us,
// 8.57 with a third line of 64 bytes to wait for and x fetched behind row_ptr.
struct TileCommon {
    const uint16_t *x;
    int rows, cols, batch;   // rows of all matrices
    u32 ldx;
    int chunk;            // columns per chunk, a multiple of 64
    int n_chunks;
    u32 units_q, units_rem;  // 4-row units per row block (even_split)
    int vector_blocks;
    union {
        int group_shift;  // spmv_tile_kernel: log2 of the number of vector groups of a workgroup (1, 2, 4)
        int block_chunks; // spmv_pipe_kernel: chunks whose products are one sum
    };
    int vector_store;     // 8-byte stores of Y are aligned
    const u32x4 *packed;  // X in operand order (pack_vectors_kernel), null: read X itself
    int packed_tiles;     // vector tiles in it
    int packed_steps;     // 64-column steps in it
    const uint16_t *residual;  // added to Y before it is rounded (laid out like Y, may be Y), or null
};
template <int SOURCES>
struct TileArgs : TileSources<SOURCES>, TileCommon {
};
static_assert(sizeof(TileArgs<1>) == 120, "one matrix: two lines of 64 bytes with the grid's size");

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

// Whether the launch's matrices are gate and up (TileSources), and the rows of which its row blocks are multiples.
template <int SOURCES>
__device__ __forceinline__ int unit_rows_of(const TileArgs<SOURCES> &a)
{
    if constexpr (SOURCES > 1) return a.unit_rows;
    return kRowUnit;
}
template <int SOURCES>
__device__ __forceinline__ bool gated(const TileArgs<SOURCES> &a) { return SOURCES > 1 && unit_rows_of(a) != kRowUnit; }

// The matrix a row of the launch belongs to, and its row_ptr from that row on.
template <bool SEVERAL, int SOURCES>
__device__ __forceinline__ int source_of(const TileArgs<SOURCES> &a, int row)
{
    if (gated(a)) return (row >> 2) & 1;
    int m = 0;
    if constexpr (SEVERAL)
        for (int k = 1; k < SOURCES; ++k) m += row >= a.first[k] ? 1 : 0;
    return m;
}

template <int SOURCES>
__device__ __forceinline__ const int *row_ptr_at(const TileArgs<SOURCES> &a, int matrix, int row)
{
    if constexpr (SOURCES > 1) row = gated(a) ? (row >> 3 << 2) + (row & 3) : row - a.first[matrix];
    return a.source[matrix].row_ptr + row;
}

// The end of a launch: the partial sums of every tile of 16 rows and 16 vectors lie in LDS at `red`
// ([row tile][vector tile][part], 1 KB each), are added in a fixed order and stored.
template <bool PACKED, bool SEVERAL, int SOURCES>
__device__ __forceinline__ void finish_tiles(const TileArgs<SOURCES> &a, u32 red, int n_tiles, int vector_tiles, int parts, int vector0,
                                             int row0, int row1)
{
    typedef __attribute__((address_space(3))) u32x4 *lds_w32x4;
    const int lane = threadIdx.x & (kWave - 1), wave = uniform(threadIdx.x >> 6), sub = lane & 15, quarter = lane >> 4;
    for (int tile = wave; tile < n_tiles; tile += kTileWaves) {
        float4v sum = float4v{0.f, 0.f, 0.f, 0.f};
        u32 at = red + (u32)(tile * parts) * 1024 + (u32)lane * 16;
        // Up to eight parts are read together, and added one after the other as before: a read behind each addition was what a
        // launch of few vectors ended with (4096 x 4096, 8 vectors at 0.5: 8.76 us, four together 8.48, eight 8.43; 5 at 0.2
        // 6.05, 5.72, 5.65; 777 x 3333, 8 at 0.25 7.44, 7.13, 7.07; 11008 x 4096, 8 at 0.5 16.16, 15.89, 15.82).
        auto add = [&](auto count) __attribute__((always_inline)) {
            constexpr int N = decltype(count)::value;
            float4v some[N];
#pragma unroll
            for (int p = 0; p < N; ++p) some[p] = __builtin_bit_cast(float4v, *(lds_w32x4)(uintptr_t)(at + 1024 * p));
#pragma unroll
            for (int p = 0; p < N; ++p) sum += some[p];
            at += 1024 * N;
        };
        int left = parts;  // 2, 4, 8 or 16
        for (; left >= 8; left -= 8) add(index_constant<8>{});
        if (left & 4) add(index_constant<4>{});
        if (left & 2) add(index_constant<2>{});
        const int r = tile / vector_tiles;
        const int n = vector0 + (tile - r * vector_tiles) * 16 + sub;
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
                const int matrix = source_of<SEVERAL>(a, bad_row);
                const TileSource &m = a.source[matrix];
                const int *row_ptr = row_ptr_at(a, matrix, bad_row);
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
        if constexpr (SEVERAL) {
            if (gated(a)) {  // lanes of an even quarter have four rows of the gate, those 16 further on the same rows of up
                const u32 lo = (u32)float_to_half_bits(sum[0]) | ((u32)float_to_half_bits(sum[1]) << 16);
                const u32 hi = (u32)float_to_half_bits(sum[2]) | ((u32)float_to_half_bits(sum[3]) << 16);
                const u32 up_lo = (u32)__shfl_xor((int)lo, 16), up_hi = (u32)__shfl_xor((int)hi, 16);
                auto both = [](u32 g, u32 u) __attribute__((always_inline)) {
                    const float first = silu_mul(half_bits_to_float((uint16_t)g), half_bits_to_float((uint16_t)u));
                    const float second = silu_mul(half_bits_to_float((uint16_t)(g >> 16)), half_bits_to_float((uint16_t)(u >> 16)));
                    return (u32)float_to_half_bits(first) | ((u32)float_to_half_bits(second) << 16);
                };
                if ((quarter & 1) == 0 && row < row1 && n < a.packed_tiles * 16) {
                    const int column = row >> 3 << 2;
                    u32x2 *piece = reinterpret_cast<u32x2 *>(reinterpret_cast<u32x4 *>(a.source[0].y) + packed_piece(column >> 3, n, a.packed_tiles));
                    piece[(column >> 2) & 1] = n < a.batch ? u32x2{both(lo, up_lo), both(hi, up_hi)} : u32x2{0u, 0u};
                }
                continue;
            }
        }
        if (n < a.batch) {
            uint16_t *y = a.source[0].y;
            u32 ldy = a.source[0].ldy;
            int at = row;
            if constexpr (SEVERAL) {  // my four rows are of one matrix
#pragma unroll
                for (int k = 1; k < kMaxSources; ++k)
                    if (row >= a.first[k]) {
                        y = a.source[k].y;
                        ldy = a.source[k].ldy;
                        at = row - a.first[k];
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
    if constexpr (SEVERAL) {
        if (gated(a) && row1 == a.rows) {  // the columns that fill up the last block of 64
            const int first = a.rows >> 4, pieces = packed_steps(a.rows >> 1) * 8 - first;
            for (int i = (int)threadIdx.x; i < pieces * vector_tiles * 16; i += kTileThreads) {
                const int n = vector0 + i % (vector_tiles * 16), p = first + i / (vector_tiles * 16);
                if (n < a.packed_tiles * 16)
                    reinterpret_cast<u32x4 *>(a.source[0].y)[packed_piece(p, n, a.packed_tiles)] = u32x4{0u, 0u, 0u, 0u};
            }
        }
    }
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
    const int row0 = (int)even_split(row_block, a.units_q, a.units_rem) * unit_rows_of(a);
    const int row_end_unclamped = (int)even_split(row_block + 1, a.units_q, a.units_rem) * unit_rows_of(a);
    const int row1 = row_end_unclamped < a.rows ? row_end_unclamped : a.rows;
    const int group = wave & ((1 << a.group_shift) - 1);
    const int part = wave >> a.group_shift;
    const int parts = kTileWaves >> a.group_shift;

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
        const int matrix = source_of<SEVERAL>(a, row);
        const TileSource &m = a.source[matrix];
        if constexpr (SEVERAL) describe(J, m);
        u32 e0 = 0, e1 = 0;
        if (row < row1) {
            const int *row_ptr = row_ptr_at(a, matrix, row);
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
    finish_tiles<PACKED, SEVERAL>(a, red, RT * groups * NTW, groups * NTW, parts, vector0, row0, row1);
}

// The same product with the waves in two roles: 12 of the 16 scatter (one unit of 4 rows each, 48 rows per
// workgroup), one on every SIMD multiplies (two groups of 16 * NTW vectors, the columns of a group in two parts), and a
// barrier per chunk hands a dense chunk over.  For enough rows to give every compute unit about 48 and more than 16
// vectors, where spmv_tile_kernel, whose waves do both, holds a chunk's X, the sums and the entries in the same 128
// registers and can afford neither long chunks nor more than one row per pass:
//   - a pass works four rows at once, 16 lanes each, E consecutive entries a lane (16 * E per row and chunk; the prefix
//     sum has four steps instead of six, and what a pass costs besides its entries is shared by four rows);
//   - no column is clamped: rows stand 16 * E columns apart in LDS, which is as far as the entries of a lane that reaches
//     beyond its chunk can go on either side;
//   - entries are requested into one of two register sets as soon as this chunk's stores are on their way.  The requests of all
//     waves queue behind those for X for 200 to 1100 cycles (stamps of a launch), which the stores, in front of them, need
//     not wait for; they are there well before the next chunk (128 vectors at 0.5: 21.85 us with the requests in front, 20.98);
//   - only the columns of a chunk are cleared, not what lies between rows, where only entries of other chunks go (three stores
//     a wave and chunk at 0.5 instead of six), in front of the first look at the entries.
// The multiplying waves run at a higher priority: a matrix instruction and a v_dot8 of another wave on the same SIMD
// exclude each other (measured: a v_dot8 takes 18 cycles beside a stream of matrix instructions, a plain addition 10).
// 11008 x 4096, vectors in operand order, three matrices in turn, spmv_tile_kernel and this one: 128 vectors at density 0.5
// 24.8 and 20.4 us, 0.3 24.7 and 18.6, 0.15 25.0 and 17.3, 0.05 24.6 and 15.9; 64 vectors at 0.2 18.0 and 14.7; 28672 x 1024, 64
// vectors, 0.1: 22.4 and 15.1; 12288 x 4096, 32 vectors at 0.5 18.0 and 16.1.  What bounds it: 2.2 us in front of the first product and
// 1.5 behind the last one (row_ptr, the first entries, the sums).  Between them a chunk of 384 columns takes 3100 cycles by the
// counters (128 vectors at 0.5), in which LDS is busy for 2100 (each of the 16 stores of a pass for 7: 32 lanes at random places meet in a bank three or four
// times), the path from L2 for 2000 (X: 1 MB per compute unit at 64 bytes a cycle), vector and matrix instructions, which exclude
// each other, for 2500.  While it took 21.9 us: 21.2 with the entries always in L2 and 18.6 with X in L1 as well.  Tried and not faster: 8 + 8 waves, both
// roles at one priority (22.7), a chunk's places worked out behind the stores of the one before, by all or by some of the waves (21.5 to
// 22.0), the next unit's A requested between products, lines touched some chunks ahead; chunks that end anywhere in the
// ring of units: the compiler then waits for all loads or spills.
constexpr int kPipeProducers = 12;
constexpr int kPipeRowTiles = 3;
constexpr int kPipeParts = 2;          // of the columns, per group of vectors
constexpr int kPipeGroups = 2;
constexpr int kPipeLanes = 16;         // lanes per row of a pass
// Units of 32 columns of X a wave has in flight; chunks are whole rounds of them.  A unit of X is asked for behind the entries of
// the next chunk, and loads return in order: with two units on the way the products wait for them (11008 x 4096, 128 vectors at 0.5:
// 20.98 us, with three 20.56; 33 to 64 vectors of 16 entries a lane and more than 4000 columns, 102 products of 6000 rows and more: 10 to 13 %
// slower with two).  Two where a lane has 8 entries: chunks of up to 640 columns in whole rounds of 128 are worth more
// (128 vectors at 0.15: 17.4 us, 18.7 with three; 33 to 64 vectors with four, in rounds of 256, 640 columns in two chunks 11 % slower, 128 columns 4 to 6 %,
// from 641 columns on the same within 2 %).  Up to 32 vectors two as well: with those (and two sets of sums) a wave needs 64 registers at
// most, so that two workgroups of short chunks share a compute unit (VGPR_LIMITS, _build.py).  1226 products of 17 to 32 vectors, three or
// four units and one workgroup, two and two: above 12288 rows 19 % slower in the mean up to 250 columns (28379 x 244, 21 vectors
// at 0.17 8.43 and 7.27 us), 3 to 4 % from 250 to 4000 columns.
constexpr int pipe_depth(int wave_tiles, int entries) { return wave_tiles > 1 && entries == 16 ? 3 : 2; }
constexpr int pipe_chunk_step(int wave_tiles, int entries) { return 32 * kPipeParts * pipe_depth(wave_tiles, entries); }
// Column parts of a result: two waves', of each of them two or three where there are registers for it (sets), and blocks of chunks,
// whose sums the scattering waves keep and add up: with several chunks at least as many as spmv_tile_kernel has for the same product
// (4 or 8; 12 with three sets in two blocks), so that a sum in fp32 is as exact.  Results of 10^5 that are not the exact one rounded to fp16, with
// the two waves' parts alone, by spmv_tile_kernel, and here (4096 columns): 11008 rows at 0.5, 128 vectors 190, 159, 158; 3 x 4096 rows
// 188, 128, 127; 11008 rows at 0.3, 64 vectors 183, 126, 123.  A block's end is a barrier and 48 KB through LDS: 11008 x 4096 at
// 0.5, 128 vectors 22.5 us without and 22.9 with two blocks when that was measured.  One chunk (up to 640 columns with 8 entries a
// lane, 512 with 16) has no blocks: up to ten matrix instructions a part (pipe_us says what that is worth).  One chunk in two blocks, the first
// one's sums through LDS behind the dense columns, was as exact as the other kernel and took 10 to 17 % longer.
constexpr int pipe_sets(int wave_tiles, int entries) { return wave_tiles > 2 ? 1 : wave_tiles == 2 && entries == 16 ? 3 : 2; }  // a divisor of the depth
constexpr int pipe_pad(int entries) { return entries * 16 + 8; }  // columns between rows; 16-byte aligned, rows on other banks

template <int NTW, int E, bool SEVERAL>
__global__ void __launch_bounds__(kTileThreads) spmv_pipe_kernel(const TileArgs<SEVERAL ? kMaxSources : 1> a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    typedef __attribute__((address_space(3))) u32x4 *lds_w32x4;
    typedef __attribute__((address_space(3))) uint16_t *lds_w16;
    constexpr int RT = kPipeRowTiles, L = kPipeLanes, W = E / 8;  // W: words of nibbles a lane has
    constexpr int DEPTH = pipe_depth(NTW, E);
    static_assert(E == 8 || E == 16, "entries per lane");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);

    u32 id = blockIdx.x;  // XCD k takes the k-th contiguous eighth, as above
    if ((gridDim.x & 7) == 0) id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const u32 row_block = id / (u32)a.vector_blocks;
    const int vector0 = (int)(id - row_block * (u32)a.vector_blocks) * (NTW * 16 * kPipeGroups);
    const int row0 = (int)even_split(row_block, a.units_q, a.units_rem) * unit_rows_of(a);
    const int row_end_unclamped = (int)even_split(row_block + 1, a.units_q, a.units_rem) * unit_rows_of(a);
    const int row1 = row_end_unclamped < a.rows ? row_end_unclamped : a.rows;

    const u32 stride = (u32)a.chunk * 2 + pipe_pad(E) * 2;   // bytes per row of the dense chunk
    const u32 buffer_bytes = stride * (16 * RT);
    const u32 red = (u32)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    const u32 lds0 = red + pipe_pad(E) * 2;
    const int last = a.n_chunks - 1;
    const int parts = last >= a.block_chunks ? 2 * kPipeParts : kPipeParts;   // of the sums that meet in LDS in the end
    // a block's sums lie where the first entries of a wave's rows may go in front of the next rows
    const bool overlap = kRowUnit * stride - pipe_pad(E) * 2 < 1024 * NTW;

    if (wave < kPipeProducers) {
        const int l = lane & (L - 1), h = lane / L;   // lane of a row, row of the unit
        const int unit_row = row0 + wave * kRowUnit, row = unit_row + h;
        const int matrix = source_of<SEVERAL>(a, unit_row);
        const TileSource &m = a.source[matrix];
        const __amdgpu_buffer_rsrc_t rs_values = __builtin_amdgcn_make_buffer_rsrc((void *)m.values, 0, (int)(m.padded * 2), 0x00020000);
        const __amdgpu_buffer_rsrc_t rs_deltas = __builtin_amdgcn_make_buffer_rsrc((void *)m.deltas, 0, (int)(m.padded / 2), 0x00020000);
        u32x4 tile_v[2][W];
        u32 tile_d[2][W];
        int pos = 0, end = 0;   // my next entry (the row's next entry + l * E), behind the row's last entry
        // 2 * (column behind the entry in front of the row's next) + where the row stands in the buffer
        u32 at_column;
        u32 front = ~0u;        // takes out the nibbles of the row before mine, in its first group of 8
        const u32 my_row = (u32)(wave * kRowUnit + h) * stride;
        {
            u32 e0 = 0, e1 = 0;
            if (row < row1) {
                const int *row_ptr = row_ptr_at(a, matrix, row);
                e0 = (u32)row_ptr[0];
                e1 = (u32)row_ptr[1];
            }
            e0 = e0 < m.padded ? e0 : m.padded;
            e1 = e1 < m.padded ? e1 : m.padded;
            pos = (int)(e0 & ~7u) + l * E;
            end = e1 > e0 ? (int)e1 : 0;
            at_column = my_row - 2u * (e0 & 7u);
            if (l == 0) front = ~0u << (4 * (e0 & 7u));
        }
        auto request = [&](auto set) __attribute__((always_inline)) {
            constexpr int S = decltype(set)::value;
            const bool any = pos < end;
            const u32 vo = any ? (u32)pos * 2 : kNoTileValues;
            const u32 dof = any ? (u32)pos >> 1 : kNoTileDeltas;
            if constexpr (W == 2) {  // checked word by word against the end of the array
                const u32x2 both = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_deltas, (int)dof, 0, 0));
                tile_d[S][0] = both.x;
                tile_d[S][W - 1] = both.y;
            } else {
                tile_d[S][0] = __builtin_amdgcn_raw_buffer_load_b32(rs_deltas, (int)dof, 0, 0);
            }
#pragma unroll
            for (int w = 0; w < W; ++w)  // the whole offset is the lane's: what a scalar one adds need not be part of the range check
                tile_v[S][w] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_values, (int)(vo + 16 * w), 0, 0));
        };
        float4v kept[NTW];   // the sums of the blocks behind: tile row, group and part by my number, as the multiplying waves hand them over
#pragma unroll
        for (int t = 0; t < NTW; ++t) kept[t] = float4v{0.f, 0.f, 0.f, 0.f};
        int block_left = a.block_chunks + 2;
        auto keep = [&](u32 from) __attribute__((always_inline)) {
            float4v sum[NTW];
            lds_barrier();
#pragma unroll
            for (int t = 0; t < NTW; ++t) sum[t] = __builtin_bit_cast(float4v, *(lds_w32x4)(uintptr_t)(from + 1024 * t));
            if (overlap) lds_barrier();
#pragma unroll
            for (int t = 0; t < NTW; ++t) kept[t] += sum[t];
            block_left = a.block_chunks;
        };
        u32 base = 0, buffer = 0, shift = 0;
        // Where my entries of set S go in this chunk, and which of the row's lanes belong to later ones: pos and
        // at_column move on.  True: a row has more entries in the chunk than a pass holds.
        auto place = [&](auto set) __attribute__((always_inline)) -> bool {
            constexpr int S = decltype(set)::value;
            tile_d[S][0] &= front;
            const int left = end - pos;
            if (__builtin_expect(__ballot(left > 0 && left < E) != 0, 0)) {  // entries behind the row's end: zeros, at columns nothing else takes
#pragma unroll
                for (int w = 0; w < 4 * W; ++w) {
                    const u32 keep = left >= 2 * w + 2 ? ~0u : (left == 2 * w + 1 ? 0xffffu : 0u);
                    tile_v[S][w >> 2][w & 3] &= keep;
                }
            }
            u32 step = 2u * E;
#pragma unroll
            for (int w = 0; w < W; ++w) step = __builtin_amdgcn_udot8(tile_d[S][w], 0x22222222u, step, false);
            u32 incl = step;  // sum over the lanes of the row up to mine
            incl += (u32)__builtin_amdgcn_update_dpp(0, (int)incl, 0x111, 0xF, 0xF, true);   // row_shr:1
            incl += (u32)__builtin_amdgcn_update_dpp(0, (int)incl, 0x112, 0xF, 0xF, true);
            incl += (u32)__builtin_amdgcn_update_dpp(0, (int)incl, 0x114, 0xF, 0xF, true);
            incl += (u32)__builtin_amdgcn_update_dpp(0, (int)incl, 0x118, 0xF, 0xF, true);
            const u32 origin = at_column + shift;
            const int hi = (int)(my_row + (buffer + (u32)a.chunk * 2));
            base = left > 0 ? origin + (incl - step) : 0x7ffffff0u;
            // the last lane whose last entry still belongs to this chunk: what it adds to the column and its number grow together
            int key = (int)(origin + incl) - 2 >= hi ? 0 : (int)(incl << 8 | (u32)(l + 1));
            auto larger = [&](int o) { key = o > key ? o : key; };
            larger(__builtin_amdgcn_update_dpp(0, key, 0xB1, 0xF, 0xF, true));    // quad_perm 1,0,3,2
            larger(__builtin_amdgcn_update_dpp(0, key, 0x4E, 0xF, 0xF, true));    // quad_perm 2,3,0,1
            larger(__builtin_amdgcn_update_dpp(0, key, 0x141, 0xF, 0xF, true));   // row_half_mirror
            larger(__builtin_amdgcn_update_dpp(0, key, 0x140, 0xF, 0xF, true));   // row_mirror
            const int done = key & 0xff;   // lanes
            pos += left > 0 ? done * E : 0;   // a lane behind the row's end stays there: the rest of the columns is no number of entries
            at_column += (u32)key >> 8;
            front = done ? ~0u : front;
            return __ballot(done == L && pos < end) != 0;
        };
        auto write = [&](auto set) __attribute__((always_inline)) {
            constexpr int S = decltype(set)::value;
            const int hi = (int)(my_row + (buffer + (u32)a.chunk * 2));
            if ((int)base < hi) {  // lanes wholly behind the chunk write nothing
                u32 at[E];
                u32 from = base;
#pragma unroll
                for (int w = 0; w < W; ++w) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) at[8 * w + k] = __builtin_amdgcn_udot8(tile_d[S][w], twos_upto(k), from, false);
                    from = at[8 * w + 7];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < E; ++k) {
                    const u32 w = tile_v[S][k >> 3][(k >> 1) & 3];
                    *(lds_w16)(uintptr_t)(at[k] + 2u * k) = (uint16_t)((k & 1) ? w >> 16 : w);
                }
            }
        };
        request(index_constant<0>{});
        const u32 my_rows = (u32)(wave * kRowUnit) * stride + (u32)lane * 16;
        auto scatter = [&](auto set, int c) __attribute__((always_inline)) {
            constexpr int S = decltype(set)::value;
            constexpr index_constant<1 - S> other{};
            buffer = lds0 + (S ? buffer_bytes : 0u);
            shift = buffer - (u32)(c * a.chunk) * 2;
            if (--block_left == 0) keep(buffer + my_rows);  // the chunk two before was the last one of a block, and its buffer holds the block's sums
            u32 z = buffer + my_row + (u32)l * 16;   // my row's columns, zero; what is between rows is never read
            for (int left = a.chunk; left > 0; left -= 8 * L, z += 16 * L) *(lds_w32x4)(uintptr_t)z = u32x4{0u, 0u, 0u, 0u};
            __builtin_amdgcn_sched_barrier(0);
            bool more = place(set);
            __builtin_amdgcn_sched_barrier(0);
            write(set);
            __builtin_amdgcn_sched_barrier(0);
            request(other);
            while (__builtin_expect(more, 0)) {
                more = place(other);
                write(other);
                request(other);
            }
            lds_barrier();
        };
        for (int c = 0;; c += 2) {
            scatter(index_constant<0>{}, c);
            if (c >= last) break;
            scatter(index_constant<1>{}, c + 1);
            if (c + 1 >= last) break;
        }
        if (--block_left == 0) keep(lds0 + (last & 1 ? 0u : buffer_bytes) + my_rows);
        lds_barrier();
        if (parts > kPipeParts)
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                const u32 slot = (u32)((wave >> 1) * NTW + t) * (u32)parts + (u32)(kPipeParts + (wave & 1));
                *(lds_w32x4)(uintptr_t)(red + slot * 1024 + (u32)lane * 16) = __builtin_bit_cast(u32x4, kept[t]);
            }
    } else {
        __builtin_amdgcn_s_setprio(1);
        const int sub = lane & 15, quarter = lane >> 4;
        const int group = wave & 1, part = (wave >> 1) & 1;
        constexpr int SETS = pipe_sets(NTW, E);
        float4v acc[SETS][RT][NTW];
        auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < SETS; ++s)
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int t = 0; t < NTW; ++t) acc[s][r][t] = float4v{0.f, 0.f, 0.f, 0.f};
        };
        auto summed = [&](int r, int t) __attribute__((always_inline)) {
            float4v sum = acc[0][r][t];
#pragma unroll
            for (int s = 1; s < SETS; ++s) sum += acc[s][r][t];
            return __builtin_bit_cast(u32x4, sum);
        };
        // A unit is 32 columns: half (u & 1) of the 64-column block u >> 1 of the operand order.  Mine are every
        // other one: the same half of every block.  Beyond the last block it is requested again, for columns
        // that hold zeros.
        u32x4 b[DEPTH][NTW];
        const __amdgpu_buffer_rsrc_t rs_x =
            __builtin_amdgcn_make_buffer_rsrc((void *)a.packed, 0, (int)((u32)(a.packed_tiles * a.packed_steps) * (kBlockPieces * 16)), 0x00020000);
        int x_of[NTW];
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
            int tile = (vector0 >> 4) + group * NTW + t;
            tile = tile < a.packed_tiles ? tile : a.packed_tiles - 1;
            x_of[t] = (tile * kBlockPieces + part * 64 + lane) * 16;
        }
        const u32 x_step = (u32)a.packed_tiles * (kBlockPieces * 16), x_last = (u32)(a.packed_steps - 1) * x_step;
        u32 x_at = 0;
        auto request = [&](auto slot) __attribute__((always_inline)) {
            constexpr int J = decltype(slot)::value;
#pragma unroll
            for (int t = 0; t < NTW; ++t)
                b[J][t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_x, x_of[t], (int)x_at, 0));
            x_at = x_at < x_last ? x_at + x_step : x_last;
            __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
        };
        static_for<DEPTH>([&](auto slot) { request(slot); });
        lds_barrier();
        const u32 mine = lds0 + (u32)sub * stride + (u32)quarter * 32 + (u32)part * 16;
        // (loops that end at their bottom: with one that may not run at all, the compiler keeps the sums and zeros side by side)
        for (int c = 0;;) {
            clear();
            const int behind = c + a.block_chunks <= last ? c + a.block_chunks : last + 1;
            do {
                u32 at = mine + (c & 1 ? buffer_bytes : 0u);
                const int rest = a.cols - c * a.chunk;
                int left = rest < a.chunk ? rest : a.chunk;
                do {
                    static_for<DEPTH>([&](auto slot) {
                        constexpr int J = decltype(slot)::value;
                        u32x4 av[RT];
#pragma unroll
                        for (int r = 0; r < RT; ++r) av[r] = *(lds_w32x4)(uintptr_t)(at + (u32)(16 * r) * stride);
                        at += 128;
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int r = 0; r < RT; ++r)
#pragma unroll
                            for (int t = 0; t < NTW; ++t)
                                acc[J % SETS][r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    __builtin_bit_cast(half8, av[r]), __builtin_bit_cast(half8, b[J][t]), acc[J % SETS][r][t], 0, 0, 0);
                        request(slot);
                    });
                } while ((left -= pipe_chunk_step(NTW, E)) > 0);
                lds_barrier();
            } while (++c < behind);
            if (c > last) break;
            // into the buffer that has just been read, each to the rows of the wave that keeps it
            const u32 to = lds0 + (c & 1 ? 0u : buffer_bytes) + (u32)(group * kPipeParts + part) * (kRowUnit * stride) + (u32)lane * 16;
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int t = 0; t < NTW; ++t) *(lds_w32x4)(uintptr_t)(to + (u32)(r * 4) * (kRowUnit * stride) + 1024 * t) = summed(r, t);
            lds_barrier();
            if (overlap) lds_barrier();
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                const u32 slot = (u32)((r * kPipeGroups + group) * NTW + t) * (u32)parts + (u32)part;
                *(lds_w32x4)(uintptr_t)(red + slot * 1024 + (u32)lane * 16) = summed(r, t);
            }
        __builtin_amdgcn_s_setprio(0);
    }
    lds_barrier();
    finish_tiles<true, SEVERAL>(a, red, RT * kPipeGroups * NTW, kPipeGroups * NTW, parts, vector0, row0, row1);
}

template <bool SEVERAL, auto KERNEL>
int launch_with(const TileArgs<kMaxSources> &all, unsigned grid, size_t lds_bytes, hipStream_t stream)
{
    TileArgs<SEVERAL ? kMaxSources : 1> a;
    static_cast<TileCommon &>(a) = all;
    if constexpr (SEVERAL)
        static_cast<TileSources<kMaxSources> &>(a) = all;
    else
        a.source[0] = all.source[0];
    if (lds_bytes > 64 * 1024) {
        // one-time opt-in to more than 64 KiB of dynamic LDS, per device and kernel
        static std::atomic<bool> done[64];
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        if (dev < 0 || dev >= 64 || !done[dev].load(std::memory_order_acquire)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            if (dev >= 0 && dev < 64) done[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL(KERNEL, dim3(grid), dim3(kTileThreads), lds_bytes, stream, a);
    return (int)hipGetLastError();
}

template <int RT, int NTW, int SC, bool PACKED, bool SEVERAL>
int launch_tile(const TileArgs<kMaxSources> &a, unsigned grid, size_t lds_bytes, hipStream_t stream)
{
    return launch_with<SEVERAL, spmv_tile_kernel<RT, NTW, SC, PACKED, SEVERAL>>(a, grid, lds_bytes, stream);
}

TileArgs<kMaxSources> no_matrices()
{
    TileArgs<kMaxSources> a{};
    for (int &row : a.first) row = 0x7fffffff;
    a.unit_rows = kRowUnit;
    return a;
}

// Chunks of a block.
int pipe_block_chunks(const TileShape &s, int n_chunks)
{
    const int have = kPipeParts * pipe_sets(s.wave_tiles, s.lane_entries), parts = kTileWaves >> s.group_shift, blocks = (parts + have - 1) / have;
    // what a wave keeps is handed over in its four rows
    if (kRowUnit * 2 * (s.chunk + pipe_pad(s.lane_entries)) < 1024 * s.wave_tiles) return n_chunks;
    return (n_chunks + blocks - 1) / blocks;
}

size_t pipe_lds_bytes(const TileShape &s)
{
    const size_t pad = 2 * (size_t)pipe_pad(s.lane_entries);
    const size_t dense = pad + 2 * (size_t)(16 * kPipeRowTiles) * (2 * (size_t)s.chunk + pad);
    const size_t sums = (size_t)kPipeRowTiles * s.wave_tiles * kPipeGroups * 2 * kPipeParts * 1024;
    return dense > sums ? dense : sums;
}

size_t tile_lds_bytes(const TileShape &s)
{
    const size_t dense = kTileFront + 2 * (size_t)(16 * s.row_tiles) * ((size_t)s.chunk * 2 + kTilePad * 2);
    const size_t sums = (size_t)s.row_tiles * s.wave_tiles * kTileWaves * 1024;
    return dense > sums ? dense : sums;
}

int launch_tile_shape(TileArgs<kMaxSources> a, const TileShape &s, int max_lds, hipStream_t stream)
{
    const bool pipe = s.lane_entries > 0;
    const int groups = pipe ? kPipeGroups : 1 << s.group_shift, parts = kTileWaves / groups;
    const size_t lds = pipe ? pipe_lds_bytes(s) : tile_lds_bytes(s);
    const long long units = (a.rows + a.unit_rows - 1) / a.unit_rows;
    if (lds > (size_t)max_lds || s.chunk <= 0 || s.row_blocks < 1 ||
        (pipe ? s.chunk % pipe_chunk_step(s.wave_tiles, s.lane_entries) != 0 || a.packed == nullptr : s.chunk % 64 != 0 || s.chunk > 64 * parts * s.steps) ||
        (units + s.row_blocks - 1) / s.row_blocks * a.unit_rows > 16 * (pipe ? kPipeRowTiles : s.row_tiles))
        return MACKO_E_INVALID_ARGUMENT;
    a.chunk = s.chunk;
    a.n_chunks = (a.cols + s.chunk - 1) / s.chunk;
    a.units_q = (u32)(units / s.row_blocks);
    a.units_rem = (u32)(units % s.row_blocks);
    if (pipe)
        a.block_chunks = pipe_block_chunks(s, a.n_chunks);
    else
        a.group_shift = s.group_shift;
    const int vectors = 16 * s.wave_tiles * groups;
    a.vector_blocks = (a.batch + vectors - 1) / vectors;
    const bool several = a.first[1] < a.rows;
    a.vector_store = 1;
    for (int k = 0; k < kMaxSources; ++k)
        if (a.first[k] < a.rows && (a.source[k].ldy % 4 != 0 || (reinterpret_cast<uintptr_t>(a.source[k].y) & 7) != 0)) a.vector_store = 0;
    const long long grid = s.row_blocks * a.vector_blocks;
    if (grid >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
    a.packed_tiles = packed_tiles(a.batch);
    a.packed_steps = packed_steps(a.cols);
#define MACKO_PIPE(NTW_, E_)                                                                                       \
    if (pipe && s.wave_tiles == NTW_ && s.lane_entries == E_) {                                                    \
        if (several) return launch_with<true, spmv_pipe_kernel<NTW_, E_, true>>(a, (unsigned)grid, lds, stream);   \
        return launch_with<false, spmv_pipe_kernel<NTW_, E_, false>>(a, (unsigned)grid, lds, stream);              \
    }
    MACKO_PIPE(1, 8) MACKO_PIPE(2, 8) MACKO_PIPE(4, 8) MACKO_PIPE(1, 16) MACKO_PIPE(2, 16) MACKO_PIPE(4, 16)
#undef MACKO_PIPE
#define MACKO_TILE(RT_, NTW_, SC_)                                                                                 \
    if (!pipe && s.row_tiles == RT_ && s.wave_tiles == NTW_ && s.steps == SC_) {                                   \
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
                       double *cycles, int most_shift = 2)
{
    const long long units = ((long long)rows + kRowUnit - 1) / kRowUnit;
    const double density = (double)padded / ((double)rows * (double)cols);
    const int tiles = (batch + 15) / 16;
    double least = 0.0;
    bool found = false;
    const int first_shift = tiles <= 1 ? 0 : (tiles <= 4 ? 1 : 2);
    for (int shift = first_shift < most_shift ? first_shift : most_shift; shift >= (tiles > 4 ? 1 : (tiles <= 1 ? 0 : 1)); --shift) {
        TileShape s{};
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
    *cycles = least;
    return found;
}

// Parts of a sum in a launch of spmv_pipe_kernel.
int pipe_parts(const TileShape &s, int cols)
{
    const int n_chunks = (cols + s.chunk - 1) / s.chunk, block = pipe_block_chunks(s, n_chunks);
    return kPipeParts * pipe_sets(s.wave_tiles, s.lane_entries) * ((n_chunks + block - 1) / block);
}

// The estimated time in us of a launch of spmv_pipe_kernel, for the choice between it and spmv_tile_kernel, whose estimate it
// is compared with: per round of workgroups, per block's end, per chunk and pass (of 16 entries a lane it costs more than one of
// 8) and per column and vector.  Fitted, to what decides rather than to the time itself (8 % off in the median), to 7000 products
// of packed vectors that both kernels can do: 64 to 28672 rows and columns, densities 0.04 to 0.95, 17 to 256 vectors.
// Where its sums have fewer parts than the other kernel's (one chunk; few chunks and more than 64 vectors) and a part is more than two
// matrix instructions, 4 to 30 % more of its results are not the exact one rounded to fp16.  That has to be worth something: the
// estimate is higher there (4963 x 570 at 0.18, 82 vectors, goes to the other kernel: 7.2 us, 5.9 here).  What it leaves here takes 23 % less
// time than there, and over 7000 products 1.5 % more results are not the rounded ones than by the other kernel alone, 1.9 % without it.
double pipe_us(const TileShape &s, int cols, int batch, const DeviceInfo &info, double passes)
{
    const int vectors = 16 * kPipeGroups * s.wave_tiles;
    const long long blocks = (batch + vectors - 1) / vectors;
    const double full = (double)((s.row_blocks * blocks + info.compute_units - 1) / info.compute_units);
    const int n_chunks = (cols + s.chunk - 1) / s.chunk;
    const double ends = (n_chunks - 1) / pipe_block_chunks(s, n_chunks);
    const int parts = pipe_parts(s, cols);
    if (parts < kTileWaves >> s.group_shift && cols > 64 * parts) {
        const double columns = n_chunks > 1 ? n_chunks * s.chunk : (cols + 127) / 128 * 128;
        return 0.93 + full * (3.25 + 0.35 * ends + n_chunks * (s.lane_entries == 8 ? 0.31 : 0.56) * passes + columns / 512.0 * (0.31 + 0.26 * s.wave_tiles));
    }
    const double round = s.wave_tiles == 4 ? 4.15 : s.wave_tiles == 2 ? 3.9 : 3.8;
    const double products = s.wave_tiles == 4 ? 1.28 : s.wave_tiles == 2 ? 0.75 : 0.6;   // 512 columns
    // two units of X on the way wait longer where X leaves L2 (4962 x 20544 at 0.1, 38 vectors 53.9 us, by the other kernel 39.7)
    const double columns = cols + (s.lane_entries == 8 && cols > 8192 ? 0.5 * (cols - 8192) : 0.0);
    return full * (round + 0.17 * ends + n_chunks * (s.lane_entries == 8 ? 0.22 : 0.38) * passes + columns / 512.0 * products);
}

// The shape of a launch of spmv_pipe_kernel and its estimated time.  group_shift: spmv_tile_kernel's, whose parts of a sum it has.
bool choose_pipe_shape(TileShape *shape, int rows, int cols, long long padded, int batch, int group_shift, const DeviceInfo &info, double *us)
{
    if (batch <= 16 || rows < 1 || padded < 1) return false;
    TileShape s{};
    s.group_shift = group_shift;
    s.wave_tiles = batch > 64 ? 4 : batch > 32 ? 2 : 1;
    const int vectors = 16 * kPipeGroups * s.wave_tiles;
    const long long blocks = (batch + vectors - 1) / vectors;
    const long long units = ((long long)rows + kRowUnit - 1) / kRowUnit, most = 4 * kPipeRowTiles;
    // as many workgroups as compute units, or a whole number of times that, in blocks of at most 48 rows
    const long long rounds = (units * blocks + most * info.compute_units - 1) / (most * info.compute_units);
    s.row_blocks = info.compute_units * rounds / blocks;
    if (s.row_blocks * most < units) s.row_blocks = (units + most - 1) / most;
    if (s.row_blocks > units) return false;
    const double density = (double)padded / ((double)rows * (double)cols);
    for (int e = 8; e <= 16; e += 8) {
        s.lane_entries = e;
        const int step = pipe_chunk_step(s.wave_tiles, e), whole = (cols + step - 1) / step * step;
        // columns per chunk: what LDS holds twice, and what a pass holds of a row's entries (with a margin for the spread
        // between rows, for the lane that is not done and for what stands in front of the first entry)
        const int pad = pipe_pad(e);
        int chunk = ((info.max_lds_bytes - 2 * pad) / (2 * 16 * kPipeRowTiles) - 2 * pad) / 2 / step * step;
        chunk = chunk < whole ? chunk : whole;
        const int held = (cols + 127) / 128 * 128;  // a chunk may end a round of units behind the last column, and a pass has no entries there
        auto fits = [&](int c) {
            const double mean = (c < held ? c : held) * density;
            return mean + 3.0 * std::sqrt(mean * (density < 1.0 ? 1.0 - density : 0.0)) + e + 8 <= kPipeLanes * e;
        };
        while (chunk > 0 && !fits(chunk)) chunk -= step;
        if (chunk < (e == 8 ? 512 : 384) && chunk < whole) continue;
        // 513 to 576 columns take two chunks, whose sums are two parts each, though one would hold them
        const int n_chunks = cols > 512 && cols <= chunk && e == 16 ? 2 : (cols + chunk - 1) / chunk;
        s.chunk = ((cols + n_chunks - 1) / n_chunks + step - 1) / step * step;
        if (pipe_lds_bytes(s) > (size_t)info.max_lds_bytes) continue;
        *us = pipe_us(s, cols, batch, info, 1.0);
        *shape = s;
        return true;
    }
    return false;
}

constexpr double kTileUsPerCycle = 1.06 / 2400.0;

// The kernel and the shape of a launch, and its estimated time in us (without packing; at 2.4 GHz).  Right to about 10 %
// where it decides about the route (28672 x 4096, 8 vectors, density 0.05: 40.7 us, estimated 40; 5120 x 13824, 8, 0.1:
// 24.4, 21).  several: of more than one matrix, which spmv_tile_kernel looks up row by row; its estimate is that for one
// (up to 64 vectors, 280 launches of two and three matrices of 512 to 4096 columns: what is taken is 0.1 % behind the better one, with the line
// for one matrix 1 %).  Fewer columns were not among them and have the line for one matrix.
bool choose_shape(TileShape *shape, int rows, int cols, long long padded, int batch, bool packed, const DeviceInfo &info, double *us,
                  int most_shift = 2, bool several = false)
{
    double cycles = 0.0, pipe_us = 0.0;
    if (!choose_tile_shape(shape, rows, cols, padded, batch, packed, info, &cycles, most_shift)) return false;
    *us = cycles * kTileUsPerCycle;
    TileShape pipe;
    if (packed && choose_pipe_shape(&pipe, rows, cols, padded, batch, shape->group_shift, info, &pipe_us) &&
        pipe_us < (several && cols >= 512 && pipe.wave_tiles <= 2 ? 1.03 : 0.97) * *us) {
        *shape = pipe;
        *us = pipe_us;
    }
    return true;
}

}  // namespace

// Whether this kernel can do a product of several vectors (which it should do: batched_on_tiles, macko_spmv.hip).
bool spmv_tile_takes(int rows, int cols, long long padded, int batch, long long ldx)
{
    if (rows == 0 || padded == 0 || cols < 64) return false;
    // offsets into X and into its operand-order copy are 32-bit
    return (long long)batch * ldx * 2 < (1ll << 32) && (long long)packed_bytes(cols, batch) < (1ll << 32);
}

int spmv_tile_estimate(int rows, int cols, long long padded, int batch, bool packed, const DeviceInfo &info, TileShape *shape, double *us)
{
    if (!choose_shape(shape, rows, cols, padded, batch, packed, info, us)) return MACKO_E_INVALID_ARGUMENT;
    *us += packed ? 2.9 : 0.0;
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
    a.source[0] = TileSource{args.y, (u32)args.ldy, (u32)args.padded, args.values, args.deltas, args.row_ptr};
    a.first[0] = 0;
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

// Whether several matrices of one launch are better launched one by one.  A launch has one shape, which suits the mean density, and
// XCDs have consecutive rows: with a much denser matrix among them, its rows take more passes a chunk and the XCDs that have
// it work on when the others are done.  What its rows take is what the launch takes; the estimate for that is up to 20 %
// low with the tile kernel, so launches apart are given 10 %.  4096 columns, us, one launch / one by one: 2 x 11008 rows
// at densities 0.9 and 0.1, 16 vectors 46.4 / 35.2, 128 51.1 / 46.2; 3 x 4096 at 0.9, 0.1 and 0.1, 16 vectors 24.9 / 22.8, but
// 128 23.5 / 41.7; at 0.5 each, 16 vectors 17.3 / 25.4, 128 22.9 / 43.5, which is not asked: up to a tenth above the mean a
// matrix's rows fit the launch's passes.
bool better_apart(const TileArgs<kMaxSources> &a, int used, const TileShape &shape, const DeviceInfo &info)
{
    double entries = 0.0, densest = 0.0;
    for (int k = 0; k < used; ++k) {
        const int rows = (k + 1 < used ? a.first[k + 1] : a.rows) - a.first[k];
        const double density = (double)a.source[k].padded / ((double)rows * (double)a.cols);
        entries += a.source[k].padded;
        densest = density > densest ? density : densest;
    }
    if (densest * (double)a.rows * (double)a.cols <= 1.1 * entries) return false;
    double apart = 0.0, together = 0.0;
    for (int k = 0; k < used; ++k) {
        const int rows = (k + 1 < used ? a.first[k + 1] : a.rows) - a.first[k];
        TileShape own;
        double us = 0.0;
        if (!choose_shape(&own, rows, a.cols, a.source[k].padded, a.batch, true, info, &us)) return false;
        apart += us;
    }
    if (shape.lane_entries > 0) {
        const double held = kPipeLanes * shape.lane_entries;
        together = pipe_us(shape, a.cols, a.batch, info, std::ceil((densest * shape.chunk + shape.lane_entries + 8) / held));
    } else {
        const long long units = ((long long)a.rows + kRowUnit - 1) / kRowUnit;
        const double whole = std::ceil(densest * shape.chunk / 504.0) * 504.0 / shape.chunk;   // passes
        together = tile_cost(shape, units, a.cols, whole, a.batch, true, info.compute_units) * kTileUsPerCycle;
    }
    return together > 0.9 * apart;
}

// `together`: only say whether the matrices are better launched together.  `gated_out`: of gate and up (checked by
// the callers), silu(gate) * up in operand order.
int packed_product(const macko_packed_matrix *matrices, int n, const void *packed, const void *residual, int cols, int batch, void *stream,
                   void *gated_out = nullptr, int32_t *together = nullptr)
{
    if (matrices == nullptr || n < 1 || n > kMaxSources || cols < 64 || batch < 1 || (n > 1 && residual != nullptr)) return MACKO_E_INVALID_ARGUMENT;
    const bool products = gated_out == nullptr && together == nullptr;
    TileArgs<kMaxSources> a = no_matrices();
    long long rows = 0, padded = 0;
    int used = 0;
    for (int k = 0; k < n; ++k) {
        const macko_packed_matrix &m = matrices[k];
        if (m.rows < 0 || m.padded_entries < 0 || m.padded_entries % kChunk != 0 || m.padded_entries >= (1ll << 31) - 8192 ||
            (products && (m.ldy < m.rows || m.ldy >= (1ll << 31))))
            return MACKO_E_INVALID_ARGUMENT;
        if (m.rows == 0) continue;
        if (m.row_ptr == nullptr || (products && m.y == nullptr) || packed == nullptr ||
            (m.padded_entries > 0 && (m.values == nullptr || m.deltas == nullptr)) || packed_bytes(cols, batch) >= (1ull << 32))
            return MACKO_E_INVALID_ARGUMENT;
        if ((reinterpret_cast<uintptr_t>(m.values) & 15) || (reinterpret_cast<uintptr_t>(m.deltas) & 3) ||
            (reinterpret_cast<uintptr_t>(m.row_ptr) & 3) || (reinterpret_cast<uintptr_t>(packed) & 15) ||
            (reinterpret_cast<uintptr_t>(residual) & 1) || (products && (reinterpret_cast<uintptr_t>(m.y) & 1)))
            return MACKO_E_INVALID_ARGUMENT;
        if (rows % kRowUnit != 0) return MACKO_E_INVALID_ARGUMENT;  // the matrix in front does not end on a whole unit
        a.first[used] = (int)rows;
        a.source[used++] = TileSource{(uint16_t *)m.y, (u32)m.ldy, (u32)m.padded_entries, (const u32 *)m.values, (const u32 *)m.deltas, m.row_ptr};
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
    double us = 0.0;
    int most_shift = 2;
    if (used > 1) {  // a launch has no fewer parts of a sum than the smallest of its matrices has on its own
        int least = 0;
        auto rows_of = [&](int k) { return (k + 1 < used ? a.first[k + 1] : a.rows) - a.first[k]; };
        for (int k = 1; k < used; ++k) least = rows_of(k) < rows_of(least) ? k : least;
        if (choose_tile_shape(&shape, rows_of(least), cols, a.source[least].padded, batch, true, info, &us)) most_shift = shape.group_shift;
    }
    if (!choose_shape(&shape, a.rows, cols, padded, batch, true, info, &us, most_shift, used > 1)) return MACKO_E_INVALID_ARGUMENT;
    const bool apart = used > 1 && gated_out == nullptr && better_apart(a, used, shape, info);
    if (together != nullptr) {
        *together = apart ? 0 : 1;
        return 0;
    }
    if (gated_out != nullptr) {
        a.unit_rows = 2 * kRowUnit;
        for (int k = 0; k < used; ++k) {
            a.source[k].y = (uint16_t *)gated_out;
            a.source[k].ldy = 0;
        }
    }
    if (apart) {
        for (int k = 0; k < n; ++k) {
            const int e = packed_product(matrices + k, 1, packed, nullptr, cols, batch, stream);
            if (e != 0) return e;
        }
        return 0;
    }
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

extern "C" int macko_packed_together(const macko_packed_matrix *matrices, int32_t n_matrices, const void *packed, int32_t cols,
                                     int32_t batch, int32_t *together)
{
    if (together == nullptr) return MACKO_E_INVALID_ARGUMENT;
    *together = 1;
    return macko::packed_product(matrices, n_matrices, packed, nullptr, cols, batch, nullptr, nullptr, together);
}

extern "C" int macko_spmv_f16_packed_silu(const macko_packed_matrix *gate, const macko_packed_matrix *up, const void *packed, void *out,
                                          int32_t cols, int32_t batch, void *stream)
{
    using namespace macko;
    if (gate == nullptr || up == nullptr || gate->rows != up->rows || gate->rows < 64 || gate->rows % 8 != 0 || gate->rows >= (1 << 30) ||
        out == nullptr || (reinterpret_cast<uintptr_t>(out) & 15) || batch < 1 || packed_bytes(gate->rows, batch) >= (1ull << 32))
        return MACKO_E_INVALID_ARGUMENT;
    const macko_packed_matrix both[2] = {*gate, *up};
    return packed_product(both, 2, packed, nullptr, cols, batch, stream, out);
}
