// What a Llama-architecture decoder does between the projections of a prompt (gfx950, wave64), for all
// its tokens at once: RMS norm, rotary embedding and cache append, causal attention, SiLU gate.  The
// results that a projection consumes are written in its operand order (macko_packed.h), so that no
// packing pass and no copy stands between the two.  The upstream harness runs stock Hugging Face modules
// for these parts (python_scripts/util_run_pruned_llm.py:136-160); there is no upstream kernel to mirror.
// Activations fp16, arithmetic fp32 (the two products of the attention on the matrix cores).  Through
// torch's elementwise operators these parts were 35 launches of about 5 us per layer (128 tokens, dim 4096);
// here they are five.

#include "macko_decode.h"
#include "macko_packed.h"

namespace macko {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
__device__ __forceinline__ float lo(u32 w) { return h2f((uint16_t)(w & 0xffffu)); }
__device__ __forceinline__ float hi(u32 w) { return h2f((uint16_t)(w >> 16)); }
__device__ __forceinline__ u32 pack2(float l, float h) { return (u32)f2h(l) | ((u32)f2h(h) << 16); }

// rmsnorm(x) * w in operand order (PACKED) or as rows.  One workgroup per token (and, packed, per token
// that only fills up the last block of 16).
// Bound by latency (128 x 4096: 1 MB in, 1 MB out, two round trips to memory and one reduction).
constexpr int kNormThreads = 512;
constexpr int kNormPieces = 4;  // pieces of a row a thread keeps in registers (up to 16384 columns)
template <bool PACKED>
__global__ void __launch_bounds__(kNormThreads) rmsnorm_rows_kernel(const u32x4 *__restrict__ x, const u32x4 *__restrict__ w,
                                                                    u32x4 *__restrict__ out, int cols, int batch, int tiles,
                                                                    float eps)
{
    __shared__ float scratch[kNormThreads / kWave];
    const int n = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int pieces = cols >> 3, padded = PACKED ? packed_steps(cols) * 8 : pieces;
    if (PACKED && n >= batch) {
        for (int p = tid; p < padded; p += kNormThreads) out[packed_piece(p, n, tiles)] = u32x4{0, 0, 0, 0};
        return;
    }
    const u32x4 *row = x + (size_t)n * pieces;
    u32x4 kept[kNormPieces];
    float ss = 0.f;
    auto add = [&](const u32x4 &v) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += lo(v[e]) * lo(v[e]) + hi(v[e]) * hi(v[e]);
    };
#pragma unroll
    for (int i = 0; i < kNormPieces; ++i) {
        const int p = tid + i * kNormThreads;
        kept[i] = p < pieces ? row[p] : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < kNormPieces; ++i) add(kept[i]);
    for (int p = tid + kNormPieces * kNormThreads; p < pieces; p += kNormThreads) add(row[p]);
    const float ws = wave_sum(ss);
    if (lane == 0) scratch[wave] = ws;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < kNormThreads / kWave; ++i) total += scratch[i];
    const float inv = rsqrtf(total / (float)cols + eps);
    auto put = [&](int p, const u32x4 &v) {
        u32x4 o = {0, 0, 0, 0};
        if (p < pieces) {
            const u32x4 g = w[p];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pack2(lo(v[e]) * inv * lo(g[e]), hi(v[e]) * inv * hi(g[e]));
        }
        out[PACKED ? packed_piece(p, n, tiles) : (size_t)n * pieces + (size_t)p] = o;
    };
#pragma unroll
    for (int i = 0; i < kNormPieces; ++i) {
        const int p = tid + i * kNormThreads;
        if (p < padded) put(p, kept[i]);
    }
    for (int p = tid + kNormPieces * kNormThreads; p < padded; p += kNormThreads) put(p, p < pieces ? row[p] : u32x4{0, 0, 0, 0});
}

// packed = silu(gate) * up.  A wave packs one block, as pack_vectors_kernel does.
__global__ void __launch_bounds__(256) pack_silu_mul_kernel(const u32x4 *__restrict__ gate, const u32x4 *__restrict__ up,
                                                            u32x4 *__restrict__ packed, int cols, int batch, int tiles, int blocks)
{
    const int block = blockIdx.x * 4 + uniform(threadIdx.x >> 6);
    if (block >= blocks) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int k64 = block / tiles, tile = block - k64 * tiles;
    const int p = k64 * 8 + (lane & 7), pieces = cols >> 3;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int n = tile * 16 + h * 8 + (lane >> 3);
        u32x4 o = {0, 0, 0, 0};
        if (n < batch && p < pieces) {
            const u32x4 g = gate[(size_t)n * pieces + p], u = up[(size_t)n * pieces + p];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pack2(silu_mul(lo(g[e]), lo(u[e])), silu_mul(hi(g[e]), hi(u[e])));
        }
        packed[packed_piece(p, n, tiles)] = o;
    }
}

// q and k rotated (element i with i + head_dim / 2, cos / sin fp16 [batch, head_dim], whose two halves are
// the same), q in place, k and v into the caches [heads, max_len, head_dim] at the tokens' positions.
// A thread has 8 elements of the first half of a head and the 8 that belong to them.
__global__ void __launch_bounds__(256) rope_append_rows_kernel(u32x4 *__restrict__ q, const u32x4 *__restrict__ k,
                                                               const u32x4 *__restrict__ v, const u32x4 *__restrict__ cos_rows,
                                                               const u32x4 *__restrict__ sin_rows,
                                                               const long long *__restrict__ positions, u32x4 *__restrict__ k_cache,
                                                               u32x4 *__restrict__ v_cache, int batch, int n_heads, int half_pieces,
                                                               int max_len)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int per_token = n_heads * half_pieces;
    if (i >= batch * per_token) return;
    const int n = i / per_token, rest = i - n * per_token, head = rest / half_pieces, p = rest - head * half_pieces;
    long long pos = positions[n];
    pos = pos < 0 ? 0 : (pos >= max_len ? max_len - 1 : pos);
    const size_t at = ((size_t)n * n_heads + head) * (2 * half_pieces) + p;
    const size_t slot = ((size_t)head * max_len + (size_t)pos) * (2 * half_pieces) + p;
    const u32x4 c = cos_rows[(size_t)n * 2 * half_pieces + p], s = sin_rows[(size_t)n * 2 * half_pieces + p];
    auto rotate = [&](const u32x4 &a, const u32x4 &b, u32x4 &first, u32x4 &second) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            first[e] = pack2(lo(a[e]) * lo(c[e]) - lo(b[e]) * lo(s[e]), hi(a[e]) * hi(c[e]) - hi(b[e]) * hi(s[e]));
            second[e] = pack2(lo(b[e]) * lo(c[e]) + lo(a[e]) * lo(s[e]), hi(b[e]) * hi(c[e]) + hi(a[e]) * hi(s[e]));
        }
    };
    const u32x4 q0 = q[at], q1 = q[at + half_pieces], k0 = k[at], k1 = k[at + half_pieces], v0 = v[at], v1 = v[at + half_pieces];
    u32x4 a, b;
    rotate(q0, q1, a, b);
    q[at] = a;
    q[at + half_pieces] = b;
    rotate(k0, k1, a, b);
    k_cache[slot] = a;
    k_cache[slot + half_pieces] = b;
    v_cache[slot] = v0;
    v_cache[slot + half_pieces] = v1;
}

// Attention of 16 tokens of one head over the cache positions up to each token's own.  The workgroup's four
// waves take 32 positions at a time in turn, each with its own running maxima and sums, and meet at the end.
// Both products run transposed, S^T = K Q^T and O^T = V^T P^T, because the result layout of the first is
// then the operand layout of the second: a lane holds keys 4 quarter + i of both 16-key tiles for one
// token, which are the eight k-slots (in an order V^T is simply read in) it has to provide.  V^T comes
// from a copy of the 32 rows in LDS.  The output goes out in operand order for the next projection.
constexpr int kAttnWaves = 4;
template <int HD>
__global__ void __launch_bounds__(kAttnWaves *kWave) prefill_attention_kernel(const u32x4 *__restrict__ q,
                                                                              const u32x4 *__restrict__ k_cache,
                                                                              const u32x4 *__restrict__ v_cache,
                                                                              const long long *__restrict__ positions,
                                                                              u32x2 *__restrict__ packed, int batch, int n_heads,
                                                                              int max_len, int tiles, float scale)
{
    constexpr int PIECES = HD / 8;       // 16-byte pieces of a row
    constexpr int KSTEPS = HD / 32;      // steps of the first product
    constexpr int DTILES = HD / 16;      // 16-dimension tiles of the second
    constexpr int VROW = HD + 8;         // halves per row of the copy of V
    __shared__ __attribute__((aligned(16))) uint16_t v_lds[kAttnWaves][32 * VROW];
    __shared__ __attribute__((aligned(16))) float4v o_lds[kAttnWaves][DTILES][kWave];
    __shared__ float m_lds[kAttnWaves][16], l_lds[kAttnWaves][16];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
    const int sub = lane & 15, quarter = lane >> 4;
    const int head = blockIdx.x % n_heads, tile = blockIdx.x / n_heads;
    const int n = tile * 16 + sub;
    const float none = -3.0e38f;

    int pos = -1;  // of my token; -1 where there is none
    if (n < batch) {
        const long long p = positions[n];
        pos = (int)(p < 0 ? 0 : (p >= max_len ? max_len - 1 : p));
    }
    int last = pos;
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) {
        const int other = __shfl_xor(last, off);
        last = other > last ? other : last;
    }
    const int keys = uniform(last) + 1;

    half8 qf[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
        const u32x4 piece = n < batch ? q[((size_t)n * n_heads + head) * PIECES + s * 4 + quarter] : u32x4{0, 0, 0, 0};
        qf[s] = __builtin_bit_cast(half8, piece);
    }
    const u32x4 *kh = k_cache + (size_t)head * max_len * PIECES;
    const u32x4 *vh = v_cache + (size_t)head * max_len * PIECES;
    uint16_t *mine = v_lds[wave];

    float m = none, l = 0.f;
    float4v o[DTILES];
#pragma unroll
    for (int d = 0; d < DTILES; ++d) o[d] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * 32; k0 < keys; k0 += kAttnWaves * 32) {
        u32x4 kf[2][KSTEPS], vv[PIECES / 2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int key = k0 + h * 16 + sub;
            key = key < keys ? key : keys - 1;
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) kf[h][s] = kh[(size_t)key * PIECES + s * 4 + quarter];
        }
#pragma unroll
        for (int u = 0; u < PIECES / 2; ++u) {  // rows behind the last key stay zero: their weights are, too
            const int i = u * kWave + lane, key = k0 + i / PIECES;
            vv[u] = key < keys ? vh[(size_t)key * PIECES + i % PIECES] : u32x4{0, 0, 0, 0};
        }
        float4v st[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            st[h] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s)
                st[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, kf[h][s]), qf[s], st[h], 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < PIECES / 2; ++u) {
            const int i = u * kWave + lane;
            *reinterpret_cast<u32x4 *>(mine + (i / PIECES) * VROW + (i % PIECES) * 8) = vv[u];
        }
        float top = m;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = k0 + h * 16 + quarter * 4 + i;
                const float s = key <= pos ? st[h][i] * scale : none;
                st[h][i] = s;
                top = fmaxf(top, s);
            }
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        const float keep = __expf(m - top);
        m = top;
        l *= keep;
        half8 pf;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = k0 + h * 16 + quarter * 4 + i;
                const float s = st[h][i];
                const float w = key <= pos ? __expf(s - top) : 0.f;
                l += w;
                pf[h * 4 + i] = (_Float16)w;
            }
        // the copy is private to the wave, whose LDS operations are carried out in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int d = 0; d < DTILES; ++d) {
            half8 vt;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int row = (j >> 2) * 16 + quarter * 4 + (j & 3);
                vt[j] = __builtin_bit_cast(_Float16, mine[row * VROW + d * 16 + sub]);
            }
            o[d] *= keep;
            o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vt, pf, o[d], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (quarter == 0) {
        m_lds[wave][sub] = m;
        l_lds[wave][sub] = l;
    }
#pragma unroll
    for (int d = 0; d < DTILES; ++d) o_lds[wave][d][lane] = o[d];
    __syncthreads();
    float weight[kAttnWaves], top = none, total = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) top = fmaxf(top, m_lds[w][sub]);
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
        weight[w] = __expf(m_lds[w][sub] - top);
        total += weight[w] * l_lds[w][sub];
    }
    // No weights at all (every score -inf) are 0 / 0, as in a softmax; vectors that do not exist are 0 * 0.  Chosen in
    // front of the product, which then is rounded to fp16 once, together with the conversion.
    const float inv = pos >= 0 ? 1.0f / total : 0.f;
    for (int d = wave; d < DTILES; d += kAttnWaves) {
        float4v sum = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) sum += weight[w] * o_lds[w][d][lane];
        sum = pos >= 0 ? sum : float4v{0.f, 0.f, 0.f, 0.f};
        sum *= inv;
        const int c = head * HD + d * 16 + quarter * 4;  // four columns of vector n
        packed[packed_piece(c >> 3, n, tiles) * 2 + ((c >> 2) & 1)] = u32x2{pack2(sum[0], sum[1]), pack2(sum[2], sum[3])};
    }
}

bool aligned16(const void *p) { return p != nullptr && (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool packable(int32_t cols, int32_t batch) { return cols >= 64 && (cols & 7) == 0 && batch >= 1 && packed_bytes(cols, batch) < (1ull << 32); }

}  // namespace
}  // namespace macko

extern "C" int macko_prefill_pack_rmsnorm_f16(const void *x, const void *weight, void *packed, int32_t cols, int32_t batch,
                                              float eps, void *stream)
{
    using namespace macko;
    if (!packable(cols, batch) || !aligned16(x) || !aligned16(weight) || !aligned16(packed)) return MACKO_E_INVALID_ARGUMENT;
    hipLaunchKernelGGL(rmsnorm_rows_kernel<true>, dim3(packed_tiles(batch) * 16), dim3(kNormThreads), 0, as_stream(stream), (const u32x4 *)x,
                       (const u32x4 *)weight, (u32x4 *)packed, cols, batch, packed_tiles(batch), eps);
    return (int)hipGetLastError();
}

extern "C" int macko_rmsnorm_rows_f16(const void *x, const void *weight, void *y, int32_t cols, int32_t batch, float eps, void *stream)
{
    using namespace macko;
    if (cols <= 0 || (cols & 7) || batch < 1 || !aligned16(x) || !aligned16(weight) || !aligned16(y)) return MACKO_E_INVALID_ARGUMENT;
    hipLaunchKernelGGL(rmsnorm_rows_kernel<false>, dim3(batch), dim3(kNormThreads), 0, as_stream(stream), (const u32x4 *)x,
                       (const u32x4 *)weight, (u32x4 *)y, cols, batch, 0, eps);
    return (int)hipGetLastError();
}

extern "C" int macko_prefill_pack_silu_mul_f16(const void *gate, const void *up, void *packed, int32_t cols, int32_t batch, void *stream)
{
    using namespace macko;
    if (!packable(cols, batch) || !aligned16(gate) || !aligned16(up) || !aligned16(packed)) return MACKO_E_INVALID_ARGUMENT;
    const int tiles = packed_tiles(batch), blocks = tiles * packed_steps(cols);
    hipLaunchKernelGGL(pack_silu_mul_kernel, dim3((blocks + 3) / 4), dim3(256), 0, as_stream(stream), (const u32x4 *)gate,
                       (const u32x4 *)up, (u32x4 *)packed, cols, batch, tiles, blocks);
    return (int)hipGetLastError();
}

extern "C" int macko_prefill_rope_append_f16(void *q, const void *k, const void *v, const void *cos_rows, const void *sin_rows,
                                             const int64_t *positions, void *k_cache, void *v_cache, int32_t batch, int32_t n_heads,
                                             int32_t head_dim, int32_t max_len, void *stream)
{
    using namespace macko;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(cos_rows) || !aligned16(sin_rows) || !positions ||
        !aligned16(k_cache) || !aligned16(v_cache))
        return MACKO_E_INVALID_ARGUMENT;
    if (batch <= 0 || n_heads <= 0 || head_dim <= 0 || (head_dim & 15) || max_len <= 0 ||
        (long long)batch * n_heads * head_dim >= (1ll << 31))
        return MACKO_E_INVALID_ARGUMENT;
    const int half_pieces = head_dim / 16, threads = batch * n_heads * half_pieces;
    hipLaunchKernelGGL(rope_append_rows_kernel, dim3((threads + 255) / 256), dim3(256), 0, as_stream(stream), (u32x4 *)q,
                       (const u32x4 *)k, (const u32x4 *)v, (const u32x4 *)cos_rows, (const u32x4 *)sin_rows,
                       (const long long *)positions, (u32x4 *)k_cache, (u32x4 *)v_cache, batch, n_heads, half_pieces, max_len);
    return (int)hipGetLastError();
}

extern "C" int macko_prefill_attention_f16(const void *q, const void *k_cache, const void *v_cache, const int64_t *positions,
                                           void *packed, int32_t batch, int32_t n_heads, int32_t head_dim, int32_t max_len,
                                           float scale, void *stream)
{
    using namespace macko;
    if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !positions || !aligned16(packed)) return MACKO_E_INVALID_ARGUMENT;
    if ((head_dim != 64 && head_dim != 128) || n_heads <= 0 || max_len <= 0 || (long long)n_heads * head_dim >= (1ll << 24) ||
        !packable(n_heads * head_dim, batch))
        return MACKO_E_INVALID_ARGUMENT;
    const int tiles = packed_tiles(batch);
    if ((long long)tiles * n_heads >= (1ll << 31)) return MACKO_E_INVALID_ARGUMENT;
#define MACKO_PREFILL(HD_)                                                                                                 \
    hipLaunchKernelGGL(prefill_attention_kernel<HD_>, dim3(tiles * n_heads), dim3(kAttnWaves *kWave), 0, as_stream(stream), \
                       (const u32x4 *)q, (const u32x4 *)k_cache, (const u32x4 *)v_cache, (const long long *)positions,      \
                       (u32x2 *)packed, batch, n_heads, max_len, tiles, scale)
    if (head_dim == 128)
        MACKO_PREFILL(128);
    else
        MACKO_PREFILL(64);
#undef MACKO_PREFILL
    return (int)hipGetLastError();
}
