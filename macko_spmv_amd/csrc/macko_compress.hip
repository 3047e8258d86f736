// MACKO compressors (fp16 and int8 values) and fp16 decompressor for gfx950 (wave64).
//
// The fp16 format is restated from src/macko_spmv/cuda/cpu_compressor.cuh:6-73 of the upstream
// package as a per-column rule that needs no sequential walk:
//   column x of a row stores an entry when its element is non-zero as a float (so -0.0 does
//   not count and NaN does), or when x - p is a positive multiple of 16, p being the column
//   of the previous non-zero (-1 before the first) -- a padding entry.  The nibble of a
//   non-zero is (x - p - 1) & 15, of a padding entry 15.  Entries after the row's last
//   non-zero are not stored.  A stored element keeps its bits (a padding entry keeps the sign
//   of its zero); a NaN is stored as 0x7fff, the result of CUDA's float->half conversion that
//   the upstream code routes every value through.
//
// The int8 format (compress_rows_int8_cpu, cpu_compressor.cuh:75-117) follows the same rule on
// int8 elements, except that the padding entries after a row's last non-zero ARE stored.
//
// Pass 1 (count_rows_kernel + scan_rows_kernel) produces row_ptr; pass 2 (fill_rows_kernel)
// writes values and nibbles.  One wave owns one row in both passes (a few long rows: eight waves a row, each a piece
// of whole tiles); lanes take 8 consecutive columns and learn the previous non-zero's column from a DPP running maximum.

#include "macko_packed.h"
#include "macko_spmv_detail.h"

namespace macko {
namespace {

constexpr int kRowsPerBlock = 4;              // waves per workgroup, one row each
constexpr int kBlock = kRowsPerBlock * kWave;
constexpr int kNoColumn = (int)0x80000000;
constexpr int kAhead = 4;                     // tiles of its row a wave keeps in flight

// The two element formats.  A chunk is the 8 consecutive elements a lane handles per tile; a half of it
// (4 elements, kHalfWords words) is what one look-up in the table of byte selectors packs together.
struct Fp16Format {
    typedef uint16_t Elem;
    typedef u32x4 Chunk;                          // 8 halves
    typedef Chunk __attribute__((aligned(2))) AnyChunk;  // where a row starts at any element
    static constexpr bool kKeepTrailing = false;  // padding entries behind the last non-zero are dropped
    static constexpr int kHalfWords = 2;
    static __device__ __forceinline__ Chunk shift(const Chunk &v, int by) { return shift_down(v, by); }  // by >= 0 elements
    static __device__ __forceinline__ u32 at(const Chunk &v, int i) { return (v[i >> 1] >> (16 * (i & 1))) & 0xffffu; }
    static __device__ __forceinline__ void put(Chunk &v, int i, u32 bits) { v[i >> 1] |= bits << (16 * (i & 1)); }
    // non-zero as a float: -0.0 is a zero, NaN is not
    static __device__ __forceinline__ bool nonzero(u32 bits) { return (bits & 0x7fffu) != 0; }
    // bit i set when element i is non-zero
    static __device__ __forceinline__ u32 nonzero_bits(const Chunk &v)
    {
        u32 m = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) m |= min1(v[w] & 0x7fff7fffu) << (2 * w);
        return (m | (m >> 15)) & 0xffu;
    }
    // what is stored: the element itself, a NaN as 0x7fff
    static __device__ __forceinline__ u32 stored(u32 bits) { return (bits & 0x7fffu) > 0x7c00u ? 0x7fffu : bits; }
    // a half is a NaN when its low 15 bits exceed 0x7c00
    static __device__ __forceinline__ bool any_nan(const Chunk &v)
    {
        const Halves a = __builtin_elementwise_max(magnitude(v[0]), magnitude(v[1]));
        const Halves b = __builtin_elementwise_max(magnitude(v[2]), magnitude(v[3]));
        const Halves top = __builtin_elementwise_max(__builtin_elementwise_max(a, b), Halves{0x7c00, 0x7c00});
        return __builtin_bit_cast(u32, top) != 0x7c007c00u;
    }
    // byte selectors that bring the elements of a half whose bits are set in m to its front, word `w` of it
    static __device__ __forceinline__ u32 selectors(u32 m, int w)
    {
        u32 sel = 0;
        int n = -2 * w;
        for (u32 i = 0; i < 4; ++i)
            if ((m >> i) & 1u) {
                if (n == 0 || n == 1) sel |= ((2 * i) | (2 * i + 1) << 8) << (16 * n);
                ++n;
            }
        return sel;
    }
    static __device__ __forceinline__ void pack(const Chunk &v, int half, const u32 *sel, u32 (&out)[4])
    {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const u32 both = __builtin_amdgcn_perm(v[2 * half + 1], v[2 * half], sel[w]);
            out[2 * w] = both;
            out[2 * w + 1] = both >> 16;
        }
    }

private:
    typedef unsigned short Halves __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ Halves magnitude(u32 w) { return __builtin_bit_cast(Halves, w & 0x7fff7fffu); }
    static __device__ __forceinline__ u32 min1(u32 w)
    {
        return __builtin_bit_cast(u32, __builtin_elementwise_min(__builtin_bit_cast(Halves, w), Halves{1, 1}));
    }
};
struct Int8Format {
    typedef unsigned char Elem;
    typedef u32x2 Chunk;                         // 8 bytes
    typedef Chunk __attribute__((aligned(1))) AnyChunk;
    static constexpr bool kKeepTrailing = true;  // cpu_compressor.cuh:75-117 has no withdrawal step
    static constexpr int kHalfWords = 1;
    static __device__ __forceinline__ Chunk shift(const Chunk &v, int by)
    {
        return by < 8 ? __builtin_bit_cast(Chunk, __builtin_bit_cast(unsigned long long, v) >> (8 * by)) : Chunk{};
    }
    static __device__ __forceinline__ u32 at(const Chunk &v, int i) { return (v[i >> 2] >> (8 * (i & 3))) & 0xffu; }
    static __device__ __forceinline__ void put(Chunk &v, int i, u32 bits) { v[i >> 2] |= bits << (8 * (i & 3)); }
    static __device__ __forceinline__ bool nonzero(u32 bits) { return bits != 0; }
    static __device__ __forceinline__ u32 nonzero_bits(const Chunk &v)
    {
        // bit 7 of a byte: whether it is non-zero
        auto high = [](u32 w) { return (w | ((w & 0x7f7f7f7fu) + 0x7f7f7f7fu)) & 0x80808080u; };
        const u32 m = (high(v[0]) >> 7) | (high(v[1]) >> 3);  // bits 0, 8, 16, 24 and 4, 12, 20, 28
        return (m | (m >> 7) | (m >> 14) | (m >> 21)) & 0xffu;
    }
    static __device__ __forceinline__ u32 stored(u32 bits) { return bits; }
    static __device__ __forceinline__ bool any_nan(const Chunk &) { return false; }
    static __device__ __forceinline__ u32 selectors(u32 m, int)
    {
        u32 sel = 0;
        int n = 0;
        for (u32 i = 0; i < 4; ++i)
            if ((m >> i) & 1u) sel |= i << (8 * n++);
        return sel;
    }
    static __device__ __forceinline__ void pack(const Chunk &v, int half, const u32 *sel, u32 (&out)[4])
    {
        const u32 all = __builtin_amdgcn_perm(0u, v[half], sel[0]);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = all >> (8 * i);
    }
};

// 8 consecutive elements of a row, whatever its alignment (a 16-byte load that starts at any element costs
// at most one cache line more per wave; element by element, as this was where rows are not 16-byte aligned,
// it took eight loads).  The row's last elements come from a load that ends with the row and are moved to
// their place when they are used (cut8), so that no lane has a path of its own.  STREAM: the dense matrix
// will not be read again soon (non-temporal hint).  Columns are unsigned: those of the last tile and of the tiles asked
// for ahead may lie beyond 2^31.
template <typename F, bool STREAM>
__device__ __forceinline__ typename F::Chunk load8(const typename F::Elem *__restrict__ row, u32 col, u32 cols)
{
    typename F::Chunk v = {};
    if (cols >= 8) {
        const typename F::AnyChunk *p = reinterpret_cast<const typename F::AnyChunk *>(row + (col < cols - 8 ? col : cols - 8));
        v = STREAM ? __builtin_nontemporal_load(p) : *p;
    } else {
#pragma unroll
        for (u32 i = 0; i < 8; ++i) F::put(v, (int)i, col + i < cols ? (u32)row[col + i] : 0u);
    }
    return v;
}

// what load8 gave for columns [col, col + 8) of the tile that starts at `first`: zero beyond `cols`
template <typename F>
__device__ __forceinline__ typename F::Chunk cut8(typename F::Chunk v, u32 first, u32 col, u32 cols)
{
    if (first + kTile > cols && cols >= 8) {  // wave-uniform
        const int by = (int)(col - (cols - 8));
        v = F::shift(v, by > 0 ? by : 0);
    }
    return v;
}

// Column of the last non-zero strictly before this lane's chunk, given the lane's own last
// non-zero column (kNoColumn if none) and the carry from earlier passes.  Also returns the
// last non-zero column of the whole pass through `pass_last`.
__device__ __forceinline__ int previous_nonzero(int own_last, int carry, int &pass_last)
{
    const int incl = wave_scan_max_inclusive(own_last);
    pass_last = __builtin_amdgcn_readlane(incl, kWave - 1);
    const int before = __builtin_amdgcn_update_dpp(kNoColumn, incl, 0x138, 0xF, 0xF, false);  // wave_shr:1
    return before > carry ? before : carry;
}

__device__ __forceinline__ int wave_sum_int(int x)
{
    return __builtin_amdgcn_readlane(wave_scan_inclusive(x), kWave - 1);
}

// Columns [begin, end) of a row, whole tiles but for the row's end: the first and the last non-zero (kNoColumn where
// there is none), and the entries up to the last one, taken as if a non-zero stood in front of `begin`.
struct Piece {
    int first, last, entries;
};

// The wave's piece of a row that PIECES waves share.
template <int PIECES>
__device__ __forceinline__ void piece_columns(int piece, int cols, int &begin, int &end)
{
    begin = 0;
    end = cols;
    if (PIECES > 1) {
        const u32 per = (((u32)cols + kTile - 1) / kTile + PIECES - 1) / PIECES * kTile;
        const u32 from = (u32)piece * per;   // both may lie beyond 2^31
        begin = from < (u32)cols ? (int)from : cols;
        end = from + per < (u32)cols ? (int)(from + per) : cols;
    }
}

template <typename F, bool STREAM>
__device__ __forceinline__ Piece count_piece(const typename F::Elem *__restrict__ src, int begin, int end, int cols, int lane)
{
    typedef typename F::Chunk Chunk;
    int carry = begin - 1;  // column of the last non-zero seen in earlier passes
    int mine = 0;
    int least = kNoColumn;  // -1 - the lane's first non-zero
    // kAhead tiles of the row are in flight at any time: a wave walks its columns alone, so what hides
    // the memory latency is the depth of its own queue
    Chunk ahead[kAhead];
#pragma unroll
    for (u32 k = 0; k < kAhead; ++k) {
        const u32 col = (u32)begin + k * kTile + (u32)lane * kChunk;
        ahead[k] = (u32)begin + k * kTile < (u32)end ? load8<F, STREAM>(src, col, cols) : Chunk{};
    }
    for (u32 c0 = begin; c0 < (u32)end; c0 += kAhead * kTile) {
#pragma unroll
        for (u32 k = 0; k < kAhead; ++k) {
            const u32 at = c0 + k * kTile + (u32)lane * kChunk;
            const int col = (int)at;   // of a lane that holds elements
            if (c0 + k * kTile >= (u32)end) break;  // wave-uniform
            const Chunk v = cut8<F>(ahead[k], c0 + k * kTile, at, cols);
            if (c0 + (k + kAhead) * kTile < (u32)end) ahead[k] = load8<F, STREAM>(src, at + kAhead * kTile, cols);
            const u32 nz = F::nonzero_bits(v);
            const int own_last = nz ? col + (31 - __builtin_clz(nz)) : kNoColumn;
            int pass_last;
            const int p = previous_nonzero(own_last, carry, pass_last);
            // every non-zero is an entry; padding entries can only stand in front of the first
            // non-zero of my 8 columns (the others follow their predecessor within 8 columns)
            if (nz) {
                const int first = col + __builtin_ctz(nz);
                mine += __builtin_popcount(nz) + ((first - p - 1) >> 4);
                if (least == kNoColumn) least = -1 - first;
            }
            carry = pass_last > carry ? pass_last : carry;
        }
    }
    const int most = __builtin_amdgcn_readlane(wave_scan_max_inclusive(least), kWave - 1);
    return {most == kNoColumn ? kNoColumn : -1 - most, carry >= begin ? carry : kNoColumn, wave_sum_int(mine)};
}

// Puts a piece behind the pieces before it: `entries` counts up to the last non-zero so far, `last`.
__device__ __forceinline__ void append_piece(const Piece &piece, int begin, int &entries, int &last)
{
    if (piece.first == kNoColumn) return;
    entries += piece.entries - ((piece.first - begin) >> 4) + ((piece.first - last - 1) >> 4);
    last = piece.last;
}

// PIECES waves work one row, PIECES = 1: kRowsPerBlock rows of a wave each.
template <int PIECES>
constexpr int kBlockOf = PIECES > 1 ? PIECES * kWave : kBlock;

template <typename F, bool STREAM, int PIECES>
__global__ void __launch_bounds__(kBlockOf<PIECES>) count_rows_kernel(const typename F::Elem *__restrict__ dense, int rows,
                                                                      int cols, int *__restrict__ counts)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int row = PIECES > 1 ? (int)blockIdx.x : (int)blockIdx.x * kRowsPerBlock + wave;
    if (row >= rows) return;
    int begin, end;
    piece_columns<PIECES>(wave, cols, begin, end);
    const Piece piece = count_piece<F, STREAM>(dense + (size_t)row * (size_t)cols, begin, end, cols, lane);
    int total = 0, last = -1;
    if (PIECES > 1) {
        __shared__ Piece pieces[PIECES];
        if (lane == 0) pieces[wave] = piece;
        __syncthreads();
        if (threadIdx.x != 0) return;
        for (int w = 0; w < PIECES; ++w) {
            piece_columns<PIECES>(w, cols, begin, end);
            append_piece(pieces[w], begin, total, last);
        }
    } else {
        append_piece(piece, 0, total, last);
    }
    if (F::kKeepTrailing) total += (cols - 1 - last) >> 4;  // padding entries at last+16, last+32, ... < cols
    if (lane == 0) counts[row] = total;
}

// row_ptr[0] = 0, row_ptr[r+1] = counts[0] + ... + counts[r].  `counts` aliases row_ptr + 1.
// One workgroup walks the rows in slices of kScanSlice, 8 consecutive rows a thread in two 16-byte accesses (4-byte
// aligned), the next slice on its way while one is summed; a slice's waves meet in LDS once.  Bound by latency.  With the
// slices through LDS, for coalesced accesses, and four barriers each, 11008 rows took 5.1 us and 49152 rows 12.7; now 4.2 and 9.5.
constexpr int kScanPer = 8;
constexpr int kScanSlice = 1024 * kScanPer;
__global__ void __launch_bounds__(1024) scan_rows_kernel(int *__restrict__ row_ptr, u32 rows, int *total_out, int *total_first)
{
    struct __attribute__((packed, aligned(4))) Rows {
        int at[kScanPer];
    };
    __shared__ int wave_totals[2][16];  // of this slice and of the one before
    const u32 tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid >> 6;
    int *counts = row_ptr + 1;
    Rows ahead;
    auto request = [&](u32 first) __attribute__((always_inline)) {
        if (first + kScanPer <= rows) {
            ahead = *reinterpret_cast<const Rows *>(counts + first);
        } else {
#pragma unroll
            for (int j = 0; j < kScanPer; ++j) ahead.at[j] = first + j < rows ? counts[first + j] : 0;
        }
    };
    request(tid * kScanPer);
    if (total_first != nullptr) {
        // The total first, for a host thread that waits for this word to change rather than for the stream: it allocates
        // the outputs and launches what fills them in about the time that the rest here takes (whole call with
        // this and the scan below: 11008 x 4096 60.6 -> 58.3 us, 28672 x 8192 218 -> 210, 49152 x 64 55.8 -> 48.2; up to 4096
        // rows the same within 1 us).  A total
        // that the count pass adds up by itself was known sooner still, but its atomic additions cost it more: 28672 x 8192 4 % slower.
        constexpr int kAtOnce = 3 * kScanPer;  // loads on the way
        int sum = 0;
        for (u32 s0 = 0; s0 < rows; s0 += kAtOnce * 1024) {
            int v[kAtOnce];
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j) {
                const u32 i = s0 + j * 1024 + tid;
                v[j] = i < rows ? counts[i] : 0;
            }
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j) sum += v[j];
        }
        const int of_wave = wave_sum_int(sum);
        if (lane == 0) wave_totals[1][wave] = of_wave;
        __syncthreads();
        if (wave == 0) {
            const int total = wave_sum_int(lane < 16 ? wave_totals[1][lane] : 0);
            if (lane == 0) __hip_atomic_store(total_first, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    int running = 0;  // sum of all earlier slices
    for (int s0 = 0, turn = 0; s0 < rows; s0 += kScanSlice, turn ^= 1) {
        const u32 first = s0 + tid * kScanPer;
        Rows mine;
        int sum = 0;
#pragma unroll
        for (int j = 0; j < kScanPer; ++j) mine.at[j] = sum += ahead.at[j];
        if (s0 + kScanSlice < rows) request(first + kScanSlice);
        const int incl = wave_scan_inclusive(sum);
        // read behind this barrier, and written again behind the next: every wave is through with it then
        if (lane == kWave - 1) wave_totals[turn][wave] = incl;
        __syncthreads();
        int base = running + incl - sum;
        int slice_total = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const int t = wave_totals[turn][w];
            base += w < wave ? t : 0;
            slice_total += t;
        }
        running += slice_total;
#pragma unroll
        for (int j = 0; j < kScanPer; ++j) mine.at[j] += base;
        if (first + kScanPer <= rows) {
            *reinterpret_cast<Rows *>(counts + first) = mine;
        } else {
#pragma unroll
            for (int j = 0; j < kScanPer; ++j)
                if (first + j < rows) counts[first + j] = mine.at[j];
        }
    }
    if (tid == 0) row_ptr[0] = 0;
    if (total_out != nullptr) {  // who sees this one finds row_ptr complete
        __syncthreads();
        if (tid == 0) __hip_atomic_store(total_out, running, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Orders this wave's LDS writes before its later LDS reads by other lanes.  The staging area is
// private to the wave and a wave's LDS operations are carried out in the order issued, so this is
// a matter of instruction order only: fences of wavefront scope, which wait for nothing (a wider
// scope would also wait for the row's loads in flight and the stores on their way out).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pass 2.  The wave stages the entries of its row in LDS at the offset they have inside their
// 8-entry group of the output, so that every complete group leaves as one 16-byte store of
// values and one 4-byte store of nibbles.
//
// Values: a lane packs each half of its 8 columns with byte permutes (selectors by the half's mask) and
// stores the 4 elements one by one, wanted or not, the last ones first.  What a half stores behind its own
// entries lands where a later half has an entry of a lower number, which is stored after it; a wave's LDS
// operations are carried out in the order issued.  So no element needs an address or a test of its own.
// A half without entries stores to a spare place (it would share its place with the half behind it).
// Nibbles: 256-entry table by the lane's entry mask, packed; one or two OR operations on words that are
// zero beforehand.
// What bounds it is memory: 11008 x 4096 fp16 at density 0.5 reads 90 MB and writes 56 in 33.2 us (4.4 TB/s).
// With a 4-byte LDS store per column behind a select, and the groups packed from those words again, it took
// 39.7, half of them vector instructions.  Waiting for a row's loads all at once, so that no tile's wait
// for its load is also one for the stores of the tile before, with 8 tiles in flight: 36.4.
//
// Groups cut by a row boundary are shared with the
// neighbouring row's wave: their values go out as 2-byte stores and their nibbles as bytes.  A
// byte holds two nibbles; where a row ends on an odd entry its last nibble shares a byte with the
// first nibble of the next non-empty row.  That byte is written by the earlier row's wave, which
// works the later row's first nibble out for itself from that row's first 16 columns (the column
// of its first non-zero, or 15 for a padding entry); the later row's wave leaves the byte alone.
// So every byte of `deltas` and every element of `values` has exactly one writer, and neither
// array needs to be cleared beforehand.
//
// PIECES > 1: the waves of a workgroup share a row, where a wave per row leaves most of the chip idle and walks its row
// tile after tile (300 x 49152: 110 us for both passes, 39 with eight waves).  What a piece needs of those before it,
// its first entry's place and the last non-zero, the waves find by counting their pieces (the read that follows comes from the
// cache) and exchanging three numbers through LDS.  Pieces meet in a group as rows do.
template <typename F, bool STREAM, int PIECES>
__global__ void __launch_bounds__(kBlockOf<PIECES>) fill_rows_kernel(const typename F::Elem *__restrict__ dense, int rows,
                                                                     int cols, const int *__restrict__ row_ptr,
                                                                     typename F::Elem *__restrict__ values,
                                                                     u32 *__restrict__ delta_words, int padded,
                                                                     const spmv_detail::PlanArgs cuts, int cut_blocks)
{
    // The first workgroups make the product's cuts, a thread each (macko_spmv_plan_build): beside the rows they cost
    // nothing, behind them a launch (11008 x 4096: 5 us).
    if ((int)blockIdx.x < cut_blocks) {
        const u32 k = blockIdx.x * kBlockOf<PIECES> + threadIdx.x;
        if (k <= cuts.n_waves) spmv_detail::write_cut(cuts, k);
        return;
    }
    typedef typename F::Elem Elem;
    typedef typename F::Chunk Chunk;
    // the carried part of a group, a tile's entries, and what the last half stores behind its own
    constexpr int kStage = 8 + kTile + 8;
    constexpr int kWaves = kBlockOf<PIECES> / kWave;
    constexpr int kNibbleWords = kTile / 8 + 2;
    __shared__ __attribute__((aligned(16))) Elem stage_all[kWaves][kStage + 4 * kWave];  // + 4 spare places per lane
    __shared__ u32 nibbles_all[kWaves][kNibbleWords];
    // gap_table[m]: the nibbles of a lane whose entries are the set bits of m, packed, lowest first: the
    // distance to the previous set bit less one, and 0 for the first, whose distance reaches back into
    // earlier lanes and is put in by the lane itself
    __shared__ u32 gap_table[256];
    __shared__ __attribute__((aligned(8))) u32 pack_table[16][F::kHalfWords];
    __shared__ Piece pieces[PIECES];
    static_assert(kBlockOf<PIECES> >= 256, "one table entry per thread");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int row = PIECES > 1 ? (int)blockIdx.x - cut_blocks : ((int)blockIdx.x - cut_blocks) * kRowsPerBlock + wave;
    const Elem *src = dense + (size_t)row * (size_t)cols;
    int begin, end;
    piece_columns<PIECES>(wave, cols, begin, end);
    if (PIECES > 1) {
        const Piece piece = count_piece<F, false>(src, begin, end, cols, lane);
        if (lane == 0) pieces[wave] = piece;
    }

    // kAhead tiles of the row in flight
    Chunk ahead[kAhead];
#pragma unroll
    for (u32 k = 0; k < kAhead; ++k) {
        const u32 col = (u32)begin + k * kTile + (u32)lane * kChunk;
        ahead[k] = row < rows && (u32)begin + k * kTile < (u32)end ? load8<F, STREAM>(src, col, cols) : Chunk{};
    }
    if (const u32 m = threadIdx.x; m < 256) {
        u32 word = 0;
        int previous = -1, n = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if ((m >> i) & 1u) {
                if (previous >= 0) word |= (u32)(i - previous - 1) << (4 * n);
                previous = i;
                ++n;
            }
        gap_table[m] = word;
        if (m < 16 * F::kHalfWords) pack_table[m / F::kHalfWords][m % F::kHalfWords] = F::selectors(m / F::kHalfWords, m % F::kHalfWords);
    }
    __syncthreads();
    if (row >= rows) return;
    const int e0 = row_ptr[row];
    const int e1 = row_ptr[row + 1];
    // the wave's entries, and the last non-zero in front of its columns
    int start = e0, stop = e1, carry = -1;
    int inner_nibble = 0;  // the first nibble of the next piece's entries, where there are some
    if (PIECES > 1) {
        int entries = 0, other_begin, other_end;
        for (int w = 0; w < wave; ++w) {
            piece_columns<PIECES>(w, cols, other_begin, other_end);
            append_piece(pieces[w], other_begin, entries, carry);
        }
        // up to column c a row holds its entries up to its last non-zero in front of c, and the padding entries behind it
        // (but none behind the row's last entry)
        start = e0 + entries + ((begin - 1 - carry) >> 4);
        start = start < e1 ? start : e1;
        int last = carry;
        append_piece(pieces[wave], begin, entries, last);
        if (end < cols) {
            stop = e0 + entries + ((end - 1 - last) >> 4);
            stop = stop < e1 ? stop : e1;
        }
        int next = kNoColumn;
        for (int w = PIECES - 1; w > wave; --w) next = pieces[w].first != kNoColumn ? pieces[w].first : next;
        const int pad = last + ((end - last + 15) >> 4 << 4);  // the first padding entry from `end` on, unless a non-zero comes before
        inner_nibble = next != kNoColumn && next < pad ? next - last - 1 & 15 : 15;
        start = uniform(start);
        stop = uniform(stop);
        carry = uniform(carry);
        inner_nibble = uniform(inner_nibble);
    }
    Elem *stage = stage_all[wave];
    u32 *nibbles = nibbles_all[wave];
    Chunk *value_groups = reinterpret_cast<Chunk *>(values);
    unsigned char *delta_bytes = reinterpret_cast<unsigned char *>(delta_words);

    if (row == rows - 1 && (PIECES == 1 || wave == 0)) {  // the unused tail of the last 8-entry group (an odd e1's byte has its owner)
        for (int i = e1 + lane; i < padded; i += kWave) values[i] = 0;
        for (int i = ((e1 + 1) >> 1) + lane; i < (padded >> 1); i += kWave) delta_bytes[i] = 0;
    }
    if (start == stop) return;

    // The first nibble behind my row, wanted if my last entry is the low half of a byte: asked for
    // now, on the guess that the next row is not empty, and looked at when my row is done.
    const bool shares_last_byte = (stop & 1) != 0;
    const bool probe_lane = lane < 16 && lane < cols;
    int next_end = e1;
    u32 next_probe = 0;
    if (shares_last_byte && stop == e1 && row + 1 < rows) {
        next_end = row_ptr[row + 2];
        if (probe_lane) next_probe = dense[(size_t)(row + 1) * (size_t)cols + lane];
    }
    auto first_nibble_behind = [&]() -> u32 {
        if (PIECES > 1 && stop != e1) return (u32)inner_nibble;
        int r2 = row + 1;
        if (r2 >= rows) return 0u;  // my row holds the last entry: the rest of the byte is padding
        if (next_end == e1) {       // empty rows behind mine: walk on to the next one that is not
            do {
                ++r2;
            } while (r2 < rows && row_ptr[r2 + 1] == e1);
            if (r2 >= rows) return 0u;
            next_probe = probe_lane ? (u32)dense[(size_t)r2 * (size_t)cols + lane] : 0u;
        }
        // a row with entries whose first 16 columns are zero starts with the padding entry of column 15
        const unsigned long long m = __ballot(probe_lane && F::nonzero(next_probe));
        return m ? (u32)__builtin_ctzll(m) : 15u;
    };

    // entry base + i is stage[i] and nibble i of `nibbles`; [lo, hi) is staged and not yet written out;
    // nibbles that are not staged are zero
    int base = start & ~7;
    int lo = start - base;
    int hi = lo;
    nibbles[lane] = 0;
    if (lane < kNibbleWords - kWave) nibbles[kWave + lane] = 0;
    wave_lds_fence();

    // writes out groups [0, n_groups) of the stage; group g holds entries [a, b) with
    // a = lo for group 0 and b = hi - 8g for a last, incomplete group (which ends the row)
    auto flush = [&](int n_groups, u32 nibble_behind) {
        for (int g = lane; g < n_groups; g += kWave) {
            const Chunk v = *reinterpret_cast<const Chunk *>(stage + 8 * g);
            const u32 word = nibbles[g];
            const int a = g == 0 ? lo : 0;
            const int b = hi - 8 * g < 8 ? hi - 8 * g : 8;
            const int out = (base >> 3) + g;
            if (a == 0 && b == 8) {
                if (STREAM) {
                    value_groups[out] = v;
                    delta_words[out] = word;
                } else {
                    __builtin_nontemporal_store(v, value_groups + out);
                    __builtin_nontemporal_store(word, delta_words + out);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (i >= a && i < b) values[8 * (size_t)out + i] = (Elem)F::at(v, i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool low_mine = 2 * j >= a && 2 * j < b;
                    const bool high_mine = 2 * j + 1 >= a && 2 * j + 1 < b;
                    // low nibble mine: my byte, whoever the high nibble belongs to
                    if (low_mine) {
                        const u32 both = (word >> (8 * j)) & 0xffu;
                        delta_bytes[4 * (size_t)out + j] = (unsigned char)(high_mine ? both : (both & 15u) | (nibble_behind << 4));
                    }
                }
            }
        }
    };

    bool row_done = false;
    for (u32 c0 = begin; c0 < (u32)end && !row_done; c0 += kAhead * kTile) {
#pragma unroll
        for (u32 k = 0; k < kAhead; ++k) {
            if (row_done || c0 + k * kTile >= (u32)end) break;  // wave-uniform
            const u32 at = c0 + k * kTile + (u32)lane * kChunk;
            const int col = (int)at;   // of a lane that holds elements
            Chunk v = cut8<F>(ahead[k], c0 + k * kTile, at, cols);
            if (c0 + (k + kAhead) * kTile < (u32)end) ahead[k] = load8<F, STREAM>(src, at + kAhead * kTile, cols);
            const u32 nz = F::nonzero_bits(v);
            const int own_last = nz ? col + (31 - __builtin_clz(nz)) : kNoColumn;
            int pass_last;
            const int p = previous_nonzero(own_last, carry, pass_last);
            carry = pass_last > carry ? pass_last : carry;
            // Non-zeros are entries.  A padding entry stands at p + 16, p + 32, ...: among my 8
            // columns at most one, and only in front of my first non-zero (behind it the previous
            // non-zero is less than 8 columns away).
            const u32 pad_at = (u32)p + (((at - (u32)p + 15) >> 4) << 4) - at;  // my column index of it
            const u32 first_nz = nz ? (u32)__builtin_ctz(nz) : 8;
            const bool has_pad = pad_at < first_nz && at + pad_at < (u32)cols;
            const u32 entry_bits = nz | (has_pad ? 1u << pad_at : 0u);
            // a padding entry is 16 columns or a multiple of that behind p: 15, too
            const u32 first = has_pad ? 15u : (at + first_nz - (u32)p - 1) & 15u;
            const int mine = __builtin_popcount(entry_bits);
            const int incl = wave_scan_inclusive(mine);
            const int produced = __builtin_amdgcn_readlane(incl, kWave - 1);
            // entries past the row's end are padding entries behind its last non-zero: not stored
            const int room = stop - (base + hi);
            const int n_new = produced < room ? produced : room;
            // Those dropped entries are whole lanes: behind the row's last non-zero a lane holds at
            // most its one padding entry, and the lane of the last non-zero has its padding entry
            // in front of it.  So a lane keeps all of its entries or none.
            const int slot = incl - mine;
            const u32 kept = slot < n_new ? entry_bits : 0u;
            if (__builtin_expect(__ballot(F::any_nan(v)) != 0ull, 0)) {  // NaNs are stored in one form
                Chunk vs = Chunk{};
#pragma unroll
                for (int i = 0; i < 8; ++i) F::put(vs, i, F::stored(F::at(v, i)));
                v = vs;
            }
            const int index = hi + slot;
            u32 packed[2][4];
            Elem *place[2];
            const u32 half_mask[2] = {kept & 15u, kept >> 4};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32 sel[F::kHalfWords];
#pragma unroll
                for (int w = 0; w < F::kHalfWords; ++w) sel[w] = pack_table[half_mask[h]][w];
                F::pack(v, h, sel, packed[h]);
                place[h] = stage + (half_mask[h] ? index + (h ? __builtin_popcount(half_mask[0]) : 0) : kStage + 4 * lane);
            }
#pragma unroll
            for (int j = 3; j >= 0; --j) {
                place[0][j] = (Elem)packed[0][j];
                place[1][j] = (Elem)packed[1][j];
                wave_lds_fence();
            }
            if (kept) {
                const u32 word = gap_table[kept] | first;
                const int shift = 4 * (index & 7);
                const u32 behind = (word >> 1) >> (31 - shift);
                __hip_atomic_fetch_or(nibbles + (index >> 3), word << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                if (behind) __hip_atomic_fetch_or(nibbles + (index >> 3) + 1, behind, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
            hi += n_new;
            wave_lds_fence();
            row_done = base + hi == stop;
            const int n_groups = row_done ? (hi + 7) >> 3 : hi >> 3;
            flush(n_groups, row_done && shares_last_byte ? first_nibble_behind() : 0u);
            if (row_done) break;
            if (n_groups > 0) {  // carry the incomplete group to the front of the stage
                const Chunk moved = *reinterpret_cast<const Chunk *>(stage + 8 * n_groups);
                const u32 moved_nibbles = nibbles[n_groups];
                wave_lds_fence();
                if (lane == 0) *reinterpret_cast<Chunk *>(stage) = moved;
                nibbles[lane] = lane == 0 ? moved_nibbles : 0u;
                if (lane < kNibbleWords - kWave) nibbles[kWave + lane] = 0;
                wave_lds_fence();
                base += 8 * n_groups;
                lo = 0;
                hi &= 7;
            }
        }
    }
}

// One wave per row, one entry per lane per pass.  `padded` bounds every read of values / deltas, so
// a row_ptr that points past the arrays cannot make the kernel read outside them.
__global__ void __launch_bounds__(kBlock) decode_rows_kernel(const uint16_t *__restrict__ values,
                                                             const unsigned char *__restrict__ deltas,
                                                             const int *__restrict__ row_ptr, int rows, int cols,
                                                             long long padded, uint16_t *__restrict__ dense)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int row = blockIdx.x * kRowsPerBlock + uniform(threadIdx.x >> 6);
    if (row >= rows) return;
    long long e0 = row_ptr[row];
    long long e1 = row_ptr[row + 1];
    e0 = e0 < 0 ? 0 : (e0 > padded ? padded : e0);
    e1 = e1 < e0 ? e0 : (e1 > padded ? padded : e1);
    uint16_t *dst = dense + (size_t)row * (size_t)cols;
    int column = -1;  // column of the last entry decoded so far
    for (long long j0 = e0; j0 < e1; j0 += kWave) {
        const long long j = j0 + lane;
        int step = 0;
        uint16_t val = 0;
        if (j < e1) {
            step = ((deltas[j >> 1] >> (4 * (j & 1))) & 15) + 1;
            val = values[j];
        }
        const int incl = wave_scan_inclusive(step);
        const int c = column + incl;
        if (j < e1 && c < cols) dst[c] = val;
        column += __builtin_amdgcn_readlane(incl, kWave - 1);
    }
}

// dst[0 .. n_vec) = 0, 16 bytes per thread and step (a fill kernel rather than a memset node, so
// the call can sit in a captured graph).
__global__ void __launch_bounds__(256) zero_fill_kernel(u32x4 *__restrict__ dst, size_t n_vec, uint16_t *__restrict__ tail,
                                                        int n_tail)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t first = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = first; i < n_vec; i += stride) dst[i] = u32x4{0u, 0u, 0u, 0u};
    if (first < (size_t)n_tail) tail[first] = 0;
}

}  // namespace
}  // namespace macko

namespace macko {
namespace {

// The fill pass reads the matrix again after the count pass: up to about half the last-level
// cache (256 MB) both leave it there (measured: 5 % faster at 90 MB), and the results are stored with
// the non-temporal hint, so that they do not take its place there (whole call, 11008 x 4096 at density 0.5:
// 73.4 -> 65.9 us, at 0.9 78.7 -> 75.3, 4096 x 11008 73.5 -> 63.7); beyond that the matrix is read
// with that hint (2 % faster at 470 MB and more) and the results are not stored with it (28672 x 8192 at 0.3: 243 us,
// with it 269).
template <typename Elem>
bool streams_past_cache(int32_t rows, int32_t cols)
{
    return (size_t)rows * (size_t)cols * sizeof(Elem) > ((size_t)128 << 20);
}

// Which matrices have a row worked by kPieces waves instead of one (both passes; fp16, from a graph, us, 1 / 8 waves):
// 64 x 2048 12.0 / 10.6, 64 x 8192 24.5 / 12.7, 64 x 49152 108 / 28, 300 x 49152 110 / 39, 500 x 8192 25.1 / 16.3;
// 800 x 4096 16.7 / 17.1, 800 x 8192 26.1 / 22.2; 1200 x 4096 19.0 / 19.1, 1200 x 8192 28.4 / 25.1, 1200 x 32768 86 / 60;
// 1800 x 12288 39.3 / 40.3, 1800 x 32768 89 / 83; 2600 x 8192 34.5 / 40.9; 5000 x 8192 50 / 66 (density 0.5; at 0.05 the
// same within 4 %; int8 512 x 2048 11.6 / 11.5, 500 x 49152 98 / 35, 1280 x 8192 25.4 / 23.0).  Four waves are up to 10 % faster than eight around 1000 x 4096 and up to 30 % slower at few rows,
// sixteen gain up to 10 % more below 200 rows of 32768 columns and lose up to 40 % elsewhere.
constexpr int kPieces = 8;
bool rows_in_pieces(int32_t rows, int32_t cols)
{
    return rows <= 512 ? cols >= 2048 : rows <= 1280 && cols >= 8192;
}

template <typename F>
int compress_count(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr, int32_t *total, bool first, void *stream)
{
    typedef typename F::Elem Elem;
    if (rows < 0 || cols < 0 || row_ptr == nullptr) return MACKO_E_INVALID_ARGUMENT;
    if ((long long)rows * (long long)cols >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
    if (rows > 0 && cols > 0 && dense == nullptr) return MACKO_E_INVALID_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(dense) & (sizeof(Elem) - 1)) || (reinterpret_cast<uintptr_t>(row_ptr) & 3) ||
        (reinterpret_cast<uintptr_t>(total) & 3))
        return MACKO_E_INVALID_ARGUMENT;  // before anything is launched
    hipStream_t s = as_stream(stream);
    if (rows > 0) {
        const bool stream_reads = streams_past_cache<Elem>(rows, cols);
        auto launch = [&](auto kernel, int blocks, int threads) {
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(threads), 0, s, (const Elem *)dense, rows, cols, row_ptr + 1);
        };
        if (rows_in_pieces(rows, cols))
            stream_reads ? launch(count_rows_kernel<F, true, kPieces>, rows, kBlockOf<kPieces>)
                         : launch(count_rows_kernel<F, false, kPieces>, rows, kBlockOf<kPieces>);
        else
            stream_reads ? launch(count_rows_kernel<F, true, 1>, (rows + kRowsPerBlock - 1) / kRowsPerBlock, kBlock)
                         : launch(count_rows_kernel<F, false, 1>, (rows + kRowsPerBlock - 1) / kRowsPerBlock, kBlock);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(scan_rows_kernel, dim3(1), dim3(1024), 0, s, row_ptr, (u32)rows, first ? nullptr : total, first ? total : nullptr);
    return (int)hipGetLastError();
}

template <typename F>
int compress_fill(const void *dense, int32_t rows, int32_t cols, const int32_t *row_ptr, void *values,
                  void *deltas, int64_t padded_entries, const spmv_detail::PlanArgs &cuts, void *stream)
{
    typedef typename F::Elem Elem;
    if (rows < 0 || cols < 0 || padded_entries < 0 || padded_entries % kChunk != 0)
        return MACKO_E_INVALID_ARGUMENT;
    if ((long long)rows * (long long)cols >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
    if (padded_entries == 0) return 0;
    if (dense == nullptr || row_ptr == nullptr || values == nullptr || deltas == nullptr)
        return MACKO_E_INVALID_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(dense) & (sizeof(Elem) - 1)) ||
        (reinterpret_cast<uintptr_t>(values) & (sizeof(typename F::Chunk) - 1)) ||
        (reinterpret_cast<uintptr_t>(deltas) & 3))
        return MACKO_E_INVALID_ARGUMENT;
    hipStream_t s = as_stream(stream);
    if (rows == 0) return MACKO_E_INVALID_ARGUMENT;  // entries without rows
    const bool stream_reads = streams_past_cache<Elem>(rows, cols);
    auto launch = [&](auto kernel, int blocks, int threads) {
        const int cut_blocks = cuts.n_waves > 0 ? (int)(cuts.n_waves + threads) / threads : 0;
        hipLaunchKernelGGL(kernel, dim3(blocks + cut_blocks), dim3(threads), 0, s, (const Elem *)dense, rows, cols, row_ptr,
                           (Elem *)values, (u32 *)deltas, (int)padded_entries, cuts, cut_blocks);
    };
    if (rows_in_pieces(rows, cols))
        stream_reads ? launch(fill_rows_kernel<F, true, kPieces>, rows, kBlockOf<kPieces>)
                     : launch(fill_rows_kernel<F, false, kPieces>, rows, kBlockOf<kPieces>);
    else
        stream_reads ? launch(fill_rows_kernel<F, true, 1>, (rows + kRowsPerBlock - 1) / kRowsPerBlock, kBlock)
                     : launch(fill_rows_kernel<F, false, 1>, (rows + kRowsPerBlock - 1) / kRowsPerBlock, kBlock);
    return (int)hipGetLastError();
}

}  // namespace
}  // namespace macko

extern "C" int macko_compress_f16_count(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                        void *stream)
{
    return macko::compress_count<macko::Fp16Format>(dense, rows, cols, row_ptr, nullptr, false, stream);
}

extern "C" int macko_compress_f16_fill(const void *dense, int32_t rows, int32_t cols, const int32_t *row_ptr,
                                       void *values, void *deltas, int64_t padded_entries, void *stream)
{
    return macko::compress_fill<macko::Fp16Format>(dense, rows, cols, row_ptr, values, deltas, padded_entries, {}, stream);
}

extern "C" int macko_compress_f16_fill_plan(const void *dense, int32_t rows, int32_t cols, const int32_t *row_ptr,
                                            void *values, void *deltas, int64_t padded_entries, int32_t *plan,
                                            int32_t plan_entries, void *stream)
{
    using namespace macko;
    spmv_detail::PlanArgs cuts;
    const int rc = spmv_plan_args(row_ptr, rows, cols, padded_entries, plan, plan_entries, &cuts);
    if (rc != 0) return rc;
    return compress_fill<Fp16Format>(dense, rows, cols, row_ptr, values, deltas, padded_entries, cuts, stream);
}

extern "C" int macko_compress_f16_count_total(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                              int32_t *total, void *stream)
{
    return macko::compress_count<macko::Fp16Format>(dense, rows, cols, row_ptr, total, false, stream);
}

extern "C" int macko_compress_i8_count_total(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                             int32_t *total, void *stream)
{
    return macko::compress_count<macko::Int8Format>(dense, rows, cols, row_ptr, total, false, stream);
}

extern "C" int macko_compress_f16_count_early(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                              int32_t *total, void *stream)
{
    return macko::compress_count<macko::Fp16Format>(dense, rows, cols, row_ptr, total, true, stream);
}

extern "C" int macko_compress_i8_count_early(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                             int32_t *total, void *stream)
{
    return macko::compress_count<macko::Int8Format>(dense, rows, cols, row_ptr, total, true, stream);
}

extern "C" int macko_compress_i8_count(const void *dense, int32_t rows, int32_t cols, int32_t *row_ptr,
                                       void *stream)
{
    return macko::compress_count<macko::Int8Format>(dense, rows, cols, row_ptr, nullptr, false, stream);
}

extern "C" int macko_compress_i8_fill(const void *dense, int32_t rows, int32_t cols, const int32_t *row_ptr,
                                      void *values, void *deltas, int64_t padded_entries, void *stream)
{
    return macko::compress_fill<macko::Int8Format>(dense, rows, cols, row_ptr, values, deltas, padded_entries, {}, stream);
}

extern "C" int macko_decompress_f16(const void *values, const void *deltas, const int32_t *row_ptr, int32_t rows,
                                    int32_t cols, int64_t padded_entries, void *dense, void *stream)
{
    using namespace macko;
    if (rows < 0 || cols < 0 || padded_entries < 0) return MACKO_E_INVALID_ARGUMENT;
    if ((long long)rows * (long long)cols >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
    if (rows == 0 || cols == 0) return 0;
    if (dense == nullptr || row_ptr == nullptr) return MACKO_E_INVALID_ARGUMENT;
    if (padded_entries > 0 && (values == nullptr || deltas == nullptr)) return MACKO_E_INVALID_ARGUMENT;
    if (reinterpret_cast<uintptr_t>(dense) & 1) return MACKO_E_INVALID_ARGUMENT;
    hipStream_t s = as_stream(stream);
    {   // zeros first: whole 16-byte pieces from the first aligned address on, the few elements around them singly
        const size_t n = (size_t)rows * (size_t)cols;
        uint16_t *d = (uint16_t *)dense;
        size_t head = ((16 - (reinterpret_cast<uintptr_t>(d) & 15)) & 15) / 2;
        if (head > n) head = n;
        const size_t n_vec = (n - head) / 8;
        const size_t rest = n - head - 8 * n_vec;
        if (head > 0)
            hipLaunchKernelGGL(zero_fill_kernel, dim3(1), dim3(256), 0, s, (u32x4 *)nullptr, (size_t)0, d, (int)head);
        size_t blocks = (n_vec + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        if (blocks < 1) blocks = 1;
        hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)blocks), dim3(256), 0, s, (u32x4 *)(d + head), n_vec,
                           d + head + 8 * n_vec, (int)rest);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(decode_rows_kernel, dim3((rows + kRowsPerBlock - 1) / kRowsPerBlock), dim3(kBlock), 0, s,
                       (const uint16_t *)values, (const unsigned char *)deltas, row_ptr, rows, cols,
                       (long long)padded_entries, (uint16_t *)dense);
    return (int)hipGetLastError();
}
