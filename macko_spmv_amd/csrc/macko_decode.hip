// Glue kernels of the batch-1 decode harness (gfx950, wave64): everything a Llama-architecture
// decode step does between the projections, one launch each, so that the step is dominated by the
// matrix-vector products it is there to measure.  The upstream harness runs stock Hugging Face
// modules for these parts (python_scripts/util_run_pruned_llm.py:136-160); there is no upstream
// kernel to mirror.  All activations are fp16, all arithmetic fp32.  The current position is read
// from device memory so a captured HIP graph can be replayed for every token.

#include "macko_common.h"
#include "macko_decode.h"

namespace macko {
namespace {

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

// The rotation of a pair (x0, x1 = the element half a head further on), spelled out so that every kernel
// that rotates rounds alike.
__device__ __forceinline__ float rope_first(float x0, float x1, float c, float s) { return __builtin_fmaf(x0, c, -(x1 * s)); }
__device__ __forceinline__ float rope_second(float x0, float x1, float c, float s) { return __builtin_fmaf(x0, s, x1 * c); }

// Sum over the workgroup (blockDim.x a multiple of 64, at most 1024); every thread gets the total.
// `scratch` is 16 floats that no other reduction of the same kernel uses (so no barrier is needed
// in front of the write).
__device__ __forceinline__ float block_sum(float v, float *scratch)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6, n_waves = blockDim.x >> 6;
    const float w = wave_sum(v);
    if (lane == 0) scratch[wave] = w;
    __syncthreads();
    float total = 0.f;
    for (int i = 0; i < n_waves; ++i) total += scratch[i];
    return total;
}

__device__ __forceinline__ float block_max(float v, float *scratch)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6, n_waves = blockDim.x >> 6;
    float m = v;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) scratch[wave] = m;
    __syncthreads();
    float total = scratch[0];
    for (int i = 1; i < n_waves; ++i) total = fmaxf(total, scratch[i]);
    return total;
}

// y = x * rsqrt(mean(x^2) + eps) * w, one workgroup.
__global__ void __launch_bounds__(1024) rmsnorm_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
                                                       uint16_t *__restrict__ y, int n, float eps)
{
    __shared__ float scratch[16];
    float ss = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = h2f(x[i]);
        ss += v * v;
    }
    const float inv = rsqrtf(block_sum(ss, scratch) / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += blockDim.x) y[i] = f2h(h2f(x[i]) * inv * h2f(w[i]));
}

// Rotary embedding of q and k (rotate-half convention: element i pairs with i + head_dim/2), k and
// v appended to the caches at the current position.  One workgroup per head, head_dim/2 threads.
// q, k, v: [n_heads * head_dim]; cos, sin: [max_len, head_dim/2] fp32; caches [n_heads, max_len, head_dim].
__global__ void rope_append_kernel(const uint16_t *__restrict__ q, const uint16_t *__restrict__ k,
                                   const uint16_t *__restrict__ v, const float *__restrict__ cos_table,
                                   const float *__restrict__ sin_table, const long long *__restrict__ position,
                                   uint16_t *__restrict__ q_out, uint16_t *__restrict__ k_cache,
                                   uint16_t *__restrict__ v_cache, int head_dim, int max_len)
{
    const int head = blockIdx.x, i = threadIdx.x, half = head_dim >> 1;
    long long pos = position[0];
    pos = pos < 0 ? 0 : (pos >= max_len ? max_len - 1 : pos);
    const float c = cos_table[pos * half + i], s = sin_table[pos * half + i];
    const size_t in = (size_t)head * head_dim;
    const size_t slot = ((size_t)head * max_len + (size_t)pos) * head_dim;
    const float q0 = h2f(q[in + i]), q1 = h2f(q[in + i + half]);
    q_out[in + i] = f2h(rope_first(q0, q1, c, s));
    q_out[in + i + half] = f2h(rope_second(q0, q1, c, s));
    const float k0 = h2f(k[in + i]), k1 = h2f(k[in + i + half]);
    k_cache[slot + i] = f2h(rope_first(k0, k1, c, s));
    k_cache[slot + i + half] = f2h(rope_second(k0, k1, c, s));
    v_cache[slot + i] = v[in + i];
    v_cache[slot + i + half] = v[in + i + half];
}

// Single-query attention over positions 0..position of one head per workgroup (512 threads):
// scores, softmax, weighted sum of v.  head_dim <= 256 and a multiple of 8; max_len <= kMaxLen.
// With ROPE the kernel first does what rope_append_kernel does for its head (q, k, v are then the
// raw projections; the rotated q is rounded to fp16 as if it had been written out), so a decode
// step needs one launch for both.  The row it appends is used from LDS, not read back.
// The kernel is latency-bound (a head's cache is a few hundred KB), so what matters is how few
// dependent memory round trips there are: HD = head_dim as a compile-time constant lets a thread
// issue all loads of its k row at once (HD = 0: any head_dim, loops of runtime length), and the k
// row of a thread's first position and the v pieces of its first kVPre positions are requested
// before anything else is computed, together with q, k, v of the new token.
constexpr int kAttnThreads = 512;
constexpr int kMaxLen = 4096;
constexpr int kVPre = 8;
template <bool ROPE, int HD>
__global__ void __launch_bounds__(kAttnThreads) attention_kernel(const uint16_t *__restrict__ q,
                                                                  const uint16_t *__restrict__ k_new,
                                                                  const uint16_t *__restrict__ v_new,
                                                                  const float *__restrict__ cos_table,
                                                                  const float *__restrict__ sin_table,
                                                                  uint16_t *k_cache, uint16_t *v_cache,
                                                                  const long long *__restrict__ position,
                                                                  uint16_t *__restrict__ out, int head_dim_arg,
                                                                  int max_len, float scale)
{
    __shared__ float scores[kMaxLen];
    __shared__ __attribute__((aligned(16))) float qs[256];
    __shared__ __attribute__((aligned(16))) uint16_t ks[256];  // the appended row (ROPE only)
    __shared__ __attribute__((aligned(16))) uint16_t vs[256];
    __shared__ float partial[kAttnThreads * 8];  // groups x head_dim
    __shared__ float max_scratch[16], sum_scratch[16];
    const int head_dim = HD ? HD : head_dim_arg;
    const int head = blockIdx.x, tid = threadIdx.x;
    long long pos = position[0];
    pos = pos < 0 ? 0 : (pos >= max_len ? max_len - 1 : pos);
    const int len = (int)pos + 1;
    const int own = ROPE ? (int)pos : -1;  // the row this launch appends
    const uint16_t *kh = k_cache + (size_t)head * max_len * head_dim;
    const uint16_t *vh = v_cache + (size_t)head * max_len * head_dim;
    const int lanes_per_row = head_dim >> 3;
    const int groups = kAttnThreads / lanes_per_row;
    const int g = tid / lanes_per_row, j = tid - g * lanes_per_row;

    // ---- cache loads that depend on nothing computed here -------------------------------------------
    constexpr int NV = HD > 0 ? HD / 8 : 1;
    u32x4 kpre[NV];
    if (HD > 0) {
        const bool fetch = tid < len && tid != own;
        const u32x4 *row = reinterpret_cast<const u32x4 *>(kh + (size_t)tid * head_dim);
#pragma unroll
        for (int jj = 0; jj < NV; ++jj) kpre[jj] = fetch ? row[jj] : u32x4{0, 0, 0, 0};
    }
    u32x4 vpre[kVPre];
#pragma unroll
    for (int u = 0; u < kVPre; ++u) {
        const int pu = g + u * groups;
        const bool fetch = g < groups && pu < len && pu != own;
        vpre[u] = fetch ? reinterpret_cast<const u32x4 *>(vh + (size_t)pu * head_dim)[j] : u32x4{0, 0, 0, 0};
    }

    // ---- q (rotated with ROPE), and the new cache row -------------------------------------------------
    if (ROPE) {
        const int half = head_dim >> 1;
        if (tid < half) {
            const int i = tid;
            const float c = cos_table[pos * half + i], s = sin_table[pos * half + i];
            const size_t in = (size_t)head * head_dim;
            const size_t slot = ((size_t)head * max_len + (size_t)pos) * head_dim;
            const float q0 = h2f(q[in + i]), q1 = h2f(q[in + i + half]);
            qs[i] = h2f(f2h(rope_first(q0, q1, c, s))) * scale;
            qs[i + half] = h2f(f2h(rope_second(q0, q1, c, s))) * scale;
            const float k0 = h2f(k_new[in + i]), k1 = h2f(k_new[in + i + half]);
            const uint16_t r0 = f2h(rope_first(k0, k1, c, s)), r1 = f2h(rope_second(k0, k1, c, s));
            const uint16_t v0 = v_new[in + i], v1 = v_new[in + i + half];
            ks[i] = r0;
            ks[i + half] = r1;
            vs[i] = v0;
            vs[i + half] = v1;
            k_cache[slot + i] = r0;
            k_cache[slot + i + half] = r1;
            v_cache[slot + i] = v0;
            v_cache[slot + i + half] = v1;
        }
    } else if (tid < head_dim) {
        qs[tid] = h2f(q[(size_t)head * head_dim + tid]) * scale;
    }
    __syncthreads();

    // ---- scores -----------------------------------------------------------------------------------------
    auto dot8 = [&](const u32x4 kv, int jj, float acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc += h2f((uint16_t)(kv[e] & 0xffffu)) * qs[8 * jj + 2 * e];
            acc += h2f((uint16_t)(kv[e] >> 16)) * qs[8 * jj + 2 * e + 1];
        }
        return acc;
    };
    float local_max = -3.0e38f;
    for (int p = tid; p < len; p += kAttnThreads) {
        float acc = 0.f;
        if (p == own) {
            for (int jj = 0; jj < lanes_per_row; ++jj) acc = dot8(reinterpret_cast<const u32x4 *>(ks)[jj], jj, acc);
        } else if (HD > 0) {
            if (p != tid) {  // beyond the row requested up front
                const u32x4 *row = reinterpret_cast<const u32x4 *>(kh + (size_t)p * head_dim);
#pragma unroll
                for (int jj = 0; jj < NV; ++jj) kpre[jj] = row[jj];
            }
#pragma unroll
            for (int jj = 0; jj < NV; ++jj) acc = dot8(kpre[jj], jj, acc);
        } else {
            const u32x4 *row = reinterpret_cast<const u32x4 *>(kh + (size_t)p * head_dim);
            for (int jj = 0; jj < lanes_per_row; ++jj) acc = dot8(row[jj], jj, acc);
        }
        scores[p] = acc;
        local_max = fmaxf(local_max, acc);
    }
    const float m = block_max(local_max, max_scratch);
    float local_sum = 0.f;
    for (int p = tid; p < len; p += kAttnThreads) {
        const float e = __expf(scores[p] - m);
        scores[p] = e;
        local_sum += e;
    }
    const float inv = 1.0f / block_sum(local_sum, sum_scratch);  // also orders the scores[] writes

    // ---- weighted sum of v: a thread owns 8 consecutive dims (one 16-byte piece per position) of the
    //      positions p = g, g + groups, ...; the groups' partial sums meet in LDS --------------------------
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto add_row = [&](const u32x4 vv, float wgt) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[2 * e] += wgt * h2f((uint16_t)(vv[e] & 0xffffu));
            acc[2 * e + 1] += wgt * h2f((uint16_t)(vv[e] >> 16));
        }
    };
    if (g < groups) {
#pragma unroll
        for (int u = 0; u < kVPre; ++u) {
            const int pu = g + u * groups;
            if (pu < len) add_row(pu == own ? reinterpret_cast<const u32x4 *>(vs)[j] : vpre[u], scores[pu]);
        }
        for (int p = g + kVPre * groups; p < len; p += 4 * groups) {
            u32x4 vv[4];
            float wgt[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int pu = p + u * groups;
                const bool ok = pu < len;
                vv[u] = !ok ? u32x4{0, 0, 0, 0}
                            : (pu == own ? reinterpret_cast<const u32x4 *>(vs)[j]
                                         : reinterpret_cast<const u32x4 *>(vh + (size_t)pu * head_dim)[j]);
                wgt[u] = ok ? scores[pu] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) add_row(vv[u], wgt[u]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) partial[g * head_dim + 8 * j + e] = acc[e];
    }
    __syncthreads();
    if (tid < head_dim) {
        float total = 0.f;
        for (int gg = 0; gg < groups; ++gg) total += partial[gg * head_dim + tid];
        out[(size_t)head * head_dim + tid] = f2h(total * inv);
    }
}

template <bool ROPE>
void launch_attention(const void *q, const void *k, const void *v, const float *cos_table, const float *sin_table,
                      void *k_cache, void *v_cache, const int64_t *position, void *out, int n_heads, int head_dim,
                      int max_len, float scale, hipStream_t stream)
{
#define MACKO_ATTN(HD_)                                                                                         \
    hipLaunchKernelGGL((attention_kernel<ROPE, HD_>), dim3(n_heads), dim3(kAttnThreads), 0, stream,             \
                       (const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)v, cos_table, sin_table,      \
                       (uint16_t *)k_cache, (uint16_t *)v_cache, (const long long *)position, (uint16_t *)out,   \
                       head_dim, max_len, scale)
    if (head_dim == 128)
        MACKO_ATTN(128);
    else if (head_dim == 64)
        MACKO_ATTN(64);
    else
        MACKO_ATTN(0);
#undef MACKO_ATTN
}

// Rotary, cache append and single-query attention with a head's context in kParts pieces, one workgroup
// each, laid out for memory: a cache row is HD / 8 neighbouring lanes of 16 bytes, so that a wave's load
// is 1 KB of consecutive rows, and all of a piece's first rows are in flight before anything is computed.
// q (and the appended k row) are rotated by every lane for its own 8 dimensions, straight from memory, and
// each lane group keeps its own running maximum, sum and weighted sum of v: nothing waits for another wave
// until the groups meet in LDS.  The pieces are merged by the product that consumes them: merged here, the
// last of a head's workgroups would have to wait for the others' results to cross the chip.
// 32 heads, HD = 128, 385 positions (6.3 MB): 4.6 us against 11.7 with a workgroup of 512 threads per head
// and a thread per row (64 cache lines per load, a quarter of the compute units); 2000 positions 8.7
// against 33.  At short contexts an empty launch and two round trips to memory are left (4.1 us).
// Four pieces for every number of heads: never slower than the whole head (4 to 64 heads of 64 or 128, 1 to 4000
// positions: 4.1 to 21.9 us against 4.3 to 56.2), but not the best split for few heads and long contexts (8 heads
// of 128, 4000 positions: 9.4 us for 16 MB on 32 workgroups).
constexpr int kParts = MACKO_ATTENTION_PARTS;
constexpr int kPartThreads = 512;
constexpr int kPartLoads = 4;  // cache rows a lane group has in flight, of k and of v each

// Sum over the 8 or 16 neighbouring lanes that hold a row; every one of them gets it.
template <int LANES>
__device__ __forceinline__ float row_group_sum(float x)
{
    static_assert(LANES == 8 || LANES == 16, "lanes per row");
    x += dpp_f32<0xB1, 0xF, true>(x);   // quad_perm 1,0,3,2
    x += dpp_f32<0x4E, 0xF, true>(x);   // quad_perm 2,3,0,1
    x += dpp_f32<0x141, 0xF, true>(x);  // row_half_mirror: the other four of my eight
    if (LANES == 16) x += dpp_f32<0x140, 0xF, true>(x);  // row_mirror: the other eight of my sixteen
    return x;
}

template <int HD>
__global__ void __launch_bounds__(kPartThreads) attention_parts_kernel(const uint16_t *__restrict__ q,
                                                                       const uint16_t *__restrict__ k_new,
                                                                       const uint16_t *__restrict__ v_new,
                                                                       const float *__restrict__ cos_table,
                                                                       const float *__restrict__ sin_table, uint16_t *k_cache,
                                                                       uint16_t *v_cache, const long long *__restrict__ position,
                                                                       float *__restrict__ parts, int max_len, float scale)
{
    constexpr int LANES = HD / 8;                 // lanes per cache row
    constexpr int GROUPS = kPartThreads / LANES;  // rows per load of the workgroup
    constexpr int SHARES = kPartThreads / HD;     // threads that share an output dimension at the end
    static_assert(GROUPS <= kWave && GROUPS % SHARES == 0, "one group per lane below");
    __shared__ float o_lds[GROUPS][HD + 4];
    __shared__ float m_lds[kWave], l_lds[kWave], share_lds[SHARES][HD];
    const int head = blockIdx.x / kParts, part = blockIdx.x % kParts;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int group = tid / LANES, piece = tid % LANES;
    long long pos64 = position[0];
    pos64 = pos64 < 0 ? 0 : (pos64 >= max_len ? max_len - 1 : pos64);
    const int pos = uniform((int)pos64), len = pos + 1;
    const int per_part = (len + kParts - 1) / kParts;
    const int begin = part * per_part;
    const int end = begin + per_part < len ? begin + per_part : len;  // nothing to do if begin >= end
    // rows beyond the piece read as zero, without traffic
    const __amdgpu_buffer_rsrc_t ks = __builtin_amdgcn_make_buffer_rsrc(k_cache + (size_t)head * max_len * HD, 0, end * (HD * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t vs = __builtin_amdgcn_make_buffer_rsrc(v_cache + (size_t)head * max_len * HD, 0, end * (HD * 2), 0x00020000);

    // ---- what the new token brings: 8 dimensions per lane, and their partners half a head away ---------
    constexpr int HALF = LANES / 2;
    const u32x4 *qh = reinterpret_cast<const u32x4 *>(q + (size_t)head * HD);
    const u32x4 *kh = reinterpret_cast<const u32x4 *>(k_new + (size_t)head * HD);
    const u32x4 q_mine = qh[piece], q_other = qh[piece ^ HALF], k_mine = kh[piece], k_other = kh[piece ^ HALF];
    const u32x4 v_mine = reinterpret_cast<const u32x4 *>(v_new + (size_t)head * HD)[piece];
    const float4 *ct = reinterpret_cast<const float4 *>(cos_table + (size_t)pos * (HD / 2) + (piece % HALF) * 8);
    const float4 *st = reinterpret_cast<const float4 *>(sin_table + (size_t)pos * (HD / 2) + (piece % HALF) * 8);
    const float4 c4[2] = {ct[0], ct[1]}, s4[2] = {st[0], st[1]};

    u32x4 kv[kPartLoads], vv[kPartLoads];
    auto request = [&](int base) __attribute__((always_inline)) {
        const u32 first = (u32)base * (HD * 2) + (u32)tid * 16;
#pragma unroll
        for (int u = 0; u < kPartLoads; ++u)
            kv[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ks, (int)(first + u * (kPartThreads * 16)), 0, 0));
#pragma unroll
        for (int u = 0; u < kPartLoads; ++u)
            vv[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vs, (int)(first + u * (kPartThreads * 16)), 0, 0));
    };
    request(begin);

    auto at = [](const u32x4 &v, int e) { return h2f((uint16_t)((e & 1) ? v[e >> 1] >> 16 : v[e >> 1] & 0xffffu)); };
    // rope_first for the lanes of the first half of the head, rope_second for the others, in one form:
    // a * b + p * w with (a, b, p, w) = (x0, c, x1, -s) or (x0, s, x1, c)
    const bool first = piece < HALF;
    float rb[8], rw[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float4 cq = c4[e >> 2], sq = s4[e >> 2];
        const float c = (e & 3) == 0 ? cq.x : (e & 3) == 1 ? cq.y : (e & 3) == 2 ? cq.z : cq.w;
        const float s = (e & 3) == 0 ? sq.x : (e & 3) == 1 ? sq.y : (e & 3) == 2 ? sq.z : sq.w;
        rb[e] = first ? c : s;
        rw[e] = first ? -s : c;
    }
    auto rotated = [&](const u32x4 &mine, const u32x4 &other, int e) -> uint16_t {
        const float x0 = first ? at(mine, e) : at(other, e), x1 = first ? at(other, e) : at(mine, e);
        return f2h(__builtin_fmaf(x0, rb[e], x1 * rw[e]));
    };
    float qr[8];
    u32x4 k_row = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        qr[e] = h2f(rotated(q_mine, q_other, e)) * scale;
        k_row[e >> 1] |= (u32)rotated(k_mine, k_other, e) << (16 * (e & 1));
    }
    if (pos >= begin && pos < end && group == 0) {  // the piece that holds the new row appends it
        reinterpret_cast<u32x4 *>(k_cache + ((size_t)head * max_len + pos) * HD)[piece] = k_row;
        reinterpret_cast<u32x4 *>(v_cache + ((size_t)head * max_len + pos) * HD)[piece] = v_mine;
    }

    const float none = -3.0e38f;
    float m = none, l = 0.f;
    float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int base = begin; base < end; base += GROUPS * kPartLoads) {
        float score[kPartLoads];
        float top = m;
#pragma unroll
        for (int u = 0; u < kPartLoads; ++u) {
            const int p = base + u * GROUPS + group;
            const u32x4 row = p == pos ? k_row : kv[u];
            float acc = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = __builtin_fmaf(at(row, e), qr[e], acc);
            acc = row_group_sum<LANES>(acc);
            score[u] = p < end ? acc : none;
            top = fmaxf(top, score[u]);
        }
        const float keep = __expf(m - top);
        m = top;
        l *= keep;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] *= keep;
#pragma unroll
        for (int u = 0; u < kPartLoads; ++u) {
            const int p = base + u * GROUPS + group;
            const float w = p < end ? __expf(score[u] - top) : 0.f;
            const u32x4 row = p == pos ? v_mine : vv[u];
            l += w;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = __builtin_fmaf(w, at(row, e), o[e]);
        }
        if (base + GROUPS * kPartLoads < end) request(base + GROUPS * kPartLoads);
    }

    // ---- the groups' results: SHARES threads per dimension, then one -----------------------------------
    float4 *dst = reinterpret_cast<float4 *>(&o_lds[group][piece * 8]);
    dst[0] = float4{o[0], o[1], o[2], o[3]};
    dst[1] = float4{o[4], o[5], o[6], o[7]};
    if (piece == 0) {
        m_lds[group] = m;
        l_lds[group] = l;
    }
    __syncthreads();
    const float gm = lane < GROUPS ? m_lds[lane] : none;
    float top = gm;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    const float weight = lane < GROUPS ? __expf(gm - top) : 0.f;
    const float total = wave_sum(lane < GROUPS ? weight * l_lds[lane] : 0.f);
    const int d = tid % HD, share = uniform(tid / HD);
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < GROUPS / SHARES; ++i) {
        const int g = share * (GROUPS / SHARES) + i;
        const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), g));
        acc = __builtin_fmaf(w, o_lds[g][d], acc);
    }
    share_lds[share][d] = acc;
    __syncthreads();
    if (tid < HD) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < SHARES; ++i) sum += share_lds[i][tid];
        parts[(size_t)blockIdx.x * HD + tid] = sum;
    }
    if (tid == 0) {
        float *pair = parts + (size_t)gridDim.x * HD + (size_t)blockIdx.x * 2;
        pair[0] = top;
        pair[1] = total;
    }
}

// y = W rmsnorm(x) for a dense W (the output layer of a decode step), the norm applied by every workgroup to its own copy
// of x while its waves' first rows are on their way.  A wave owns consecutive rows and reads them whole, the next
// one requested before the present one is summed: the lanes hold the normed x (rounded to fp16, as the separate norm
// kernel writes it) for the pieces of 8 columns that they read, NP of them each.
// Bound by memory, which is read once (non-temporal): 32000 x 4096 (262 MB) 46.1 us (5.7 TB/s) against 53.7 for the BLAS's
// matrix-vector product behind the norm kernel, x 2048 23.3 against 29.7, x 1024 13.4 against 18.7, x 512 9.1 against 23.4.
constexpr int kHeadThreads = 512;
constexpr int kHeadPieces = 8;   // at most: 4096 columns (with 16, two rows and x do not fit in the registers)
template <int NP>
__global__ void __launch_bounds__(kHeadThreads) norm_matvec_kernel(const u32x4 *__restrict__ w, const u32x4 *__restrict__ x,
                                                                    const u32x4 *__restrict__ norm, uint16_t *__restrict__ y,
                                                                    int rows, int pieces, float eps, int rows_q, int rows_rem)
{
    const int lane = threadIdx.x & (kWave - 1), wave = uniform(threadIdx.x >> 6);
    const int k = blockIdx.x * (kHeadThreads / kWave) + wave;
    int row = k * rows_q + (k < rows_rem ? k : rows_rem);
    const int end = row + rows_q + (k < rows_rem ? 1 : 0);
    u32x4 a[2][NP];
    auto request = [&](auto set, int r) __attribute__((always_inline)) {
        constexpr int S = decltype(set)::value;
        const u32x4 *p = w + (size_t)(r < rows ? r : rows - 1) * (size_t)pieces;  // behind my last row: not used
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int at = lane + i * kWave;
            a[S][i] = at < pieces ? __builtin_nontemporal_load(p + at) : u32x4{0, 0, 0, 0};
        }
    };
    auto half_at = [](u32 v, int e) { return h2f((uint16_t)(e ? v >> 16 : v & 0xffffu)); };
    u32x4 xn[NP], g[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int at = lane + i * kWave;
        xn[i] = at < pieces ? x[at] : u32x4{0, 0, 0, 0};
        g[i] = at < pieces ? norm[at] : u32x4{0, 0, 0, 0};
    }
    if (row < end) request(index_constant<0>{}, row);
    // every wave sums the whole vector; the sum of its lanes' parts has one order
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = half_at(xn[i][e >> 1], e & 1);
            ss = __builtin_fmaf(v, v, ss);
        }
    const float inv = rsqrtf(wave_sum(ss) / (float)(pieces * 8) + eps);
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint16_t lo = f2h(half_at(xn[i][e], 0) * inv * half_at(g[i][e], 0));
            const uint16_t hi = f2h(half_at(xn[i][e], 1) * inv * half_at(g[i][e], 1));
            xn[i][e] = (u32)lo | ((u32)hi << 16);
        }
    auto finish = [&](auto set, int r) __attribute__((always_inline)) {
        constexpr int S = decltype(set)::value;
        float acc[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                acc[e & 1] = __builtin_fmaf(half_at(a[S][i][e >> 1], e & 1), half_at(xn[i][e >> 1], e & 1), acc[e & 1]);
        const float total = wave_sum(acc[0] + acc[1]);
        if (lane == 0) y[r] = f2h(total);
    };
    while (row < end) {
        if (row + 1 < end) request(index_constant<1>{}, row + 1);
        finish(index_constant<0>{}, row);
        if (++row >= end) break;
        if (row + 1 < end) request(index_constant<0>{}, row + 1);
        finish(index_constant<1>{}, row);
        ++row;
    }
}

// out[i] = silu(gate[i]) * up[i]
__global__ void silu_mul_kernel(const uint16_t *__restrict__ gate, const uint16_t *__restrict__ up,
                                uint16_t *__restrict__ out, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float gv = h2f(gate[i]);
        out[i] = f2h(gv / (1.0f + __expf(-gv)) * h2f(up[i]));
    }
}

}  // namespace
}  // namespace macko

extern "C" int macko_decode_rmsnorm_f16(const void *x, const void *weight, void *y, int32_t n, float eps, void *stream)
{
    using namespace macko;
    if (x == nullptr || weight == nullptr || y == nullptr || n <= 0) return MACKO_E_INVALID_ARGUMENT;
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(1), dim3(1024), 0, as_stream(stream), (const uint16_t *)x,
                       (const uint16_t *)weight, (uint16_t *)y, n, eps);
    return (int)hipGetLastError();
}

extern "C" int macko_decode_rope_append_f16(const void *q, const void *k, const void *v, const float *cos_table,
                                            const float *sin_table, const int64_t *position, void *q_out,
                                            void *k_cache, void *v_cache, int32_t n_heads, int32_t head_dim,
                                            int32_t max_len, void *stream)
{
    using namespace macko;
    if (!q || !k || !v || !cos_table || !sin_table || !position || !q_out || !k_cache || !v_cache)
        return MACKO_E_INVALID_ARGUMENT;
    if (n_heads <= 0 || head_dim <= 0 || (head_dim & 1) || head_dim > 2048 || max_len <= 0)
        return MACKO_E_INVALID_ARGUMENT;
    hipLaunchKernelGGL(rope_append_kernel, dim3(n_heads), dim3(head_dim / 2), 0, as_stream(stream),
                       (const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)v, cos_table, sin_table,
                       (const long long *)position, (uint16_t *)q_out, (uint16_t *)k_cache, (uint16_t *)v_cache,
                       head_dim, max_len);
    return (int)hipGetLastError();
}

extern "C" int macko_decode_attention_f16(const void *q, const void *k_cache, const void *v_cache,
                                          const int64_t *position, void *out, int32_t n_heads, int32_t head_dim,
                                          int32_t max_len, float scale, void *stream)
{
    using namespace macko;
    if (!q || !k_cache || !v_cache || !position || !out) return MACKO_E_INVALID_ARGUMENT;
    if (n_heads <= 0 || head_dim <= 0 || head_dim > 256 || (head_dim & 7) || max_len <= 0 || max_len > kMaxLen)
        return MACKO_E_INVALID_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(k_cache) & 15) || (reinterpret_cast<uintptr_t>(v_cache) & 15))
        return MACKO_E_INVALID_ARGUMENT;
    launch_attention<false>(q, nullptr, nullptr, nullptr, nullptr, const_cast<void *>(k_cache),
                            const_cast<void *>(v_cache), position, out, n_heads, head_dim, max_len, scale,
                            as_stream(stream));
    return (int)hipGetLastError();
}

extern "C" int macko_decode_rope_attention_f16(const void *q, const void *k, const void *v, const float *cos_table,
                                               const float *sin_table, const int64_t *position, void *k_cache,
                                               void *v_cache, void *out, int32_t n_heads, int32_t head_dim,
                                               int32_t max_len, float scale, void *stream)
{
    using namespace macko;
    if (!q || !k || !v || !cos_table || !sin_table || !position || !k_cache || !v_cache || !out)
        return MACKO_E_INVALID_ARGUMENT;
    if (n_heads <= 0 || head_dim <= 0 || head_dim > 256 || (head_dim & 7) || max_len <= 0 || max_len > kMaxLen)
        return MACKO_E_INVALID_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(k_cache) & 15) || (reinterpret_cast<uintptr_t>(v_cache) & 15))
        return MACKO_E_INVALID_ARGUMENT;
    launch_attention<true>(q, k, v, cos_table, sin_table, k_cache, v_cache, position, out, n_heads, head_dim,
                           max_len, scale, as_stream(stream));
    return (int)hipGetLastError();
}

extern "C" int macko_decode_rope_attention_parts_f16(const void *q, const void *k, const void *v, const float *cos_table,
                                                     const float *sin_table, const int64_t *position, void *k_cache,
                                                     void *v_cache, float *parts, int32_t n_heads, int32_t head_dim,
                                                     int32_t max_len, float scale, void *stream)
{
    using namespace macko;
    if (!q || !k || !v || !cos_table || !sin_table || !position || !k_cache || !v_cache || !parts)
        return MACKO_E_INVALID_ARGUMENT;
    if (n_heads <= 0 || (head_dim != 64 && head_dim != 128) || max_len <= 0 || max_len > kMaxLen) return MACKO_E_INVALID_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
         reinterpret_cast<uintptr_t>(cos_table) | reinterpret_cast<uintptr_t>(sin_table) | reinterpret_cast<uintptr_t>(k_cache) |
         reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(parts)) & 15)
        return MACKO_E_INVALID_ARGUMENT;
#define MACKO_PARTS(HD_)                                                                                             \
    hipLaunchKernelGGL(attention_parts_kernel<HD_>, dim3(n_heads * kParts), dim3(kPartThreads), 0, as_stream(stream), \
                       (const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)v, cos_table, sin_table,          \
                       (uint16_t *)k_cache, (uint16_t *)v_cache, (const long long *)position, parts, max_len, scale)
    if (head_dim == 128)
        MACKO_PARTS(128);
    else
        MACKO_PARTS(64);
#undef MACKO_PARTS
    return (int)hipGetLastError();
}

extern "C" int macko_decode_silu_mul_f16(const void *gate, const void *up, void *out, int32_t n, void *stream)
{
    using namespace macko;
    if (!gate || !up || !out || n <= 0) return MACKO_E_INVALID_ARGUMENT;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream),
                       (const uint16_t *)gate, (const uint16_t *)up, (uint16_t *)out, n);
    return (int)hipGetLastError();
}

extern "C" int macko_decode_norm_matvec_f16(const void *w, const void *x, const void *norm_weight, void *y, int32_t rows,
                                            int32_t cols, float eps, void *stream)
{
    using namespace macko;
    if (rows < 0 || cols <= 0 || (cols & 7) || cols > kHeadPieces * kWave * 8) return MACKO_E_INVALID_ARGUMENT;
    if (rows == 0) return 0;
    if (!w || !x || !norm_weight || !y || (reinterpret_cast<uintptr_t>(y) & 1) ||
        ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(norm_weight)) & 15))
        return MACKO_E_INVALID_ARGUMENT;
    DeviceInfo info;
    const int rc = device_info(&info);
    if (rc != 0) return rc;
    const int pieces = cols / 8, per_group = kHeadThreads / kWave;
    // two workgroups per compute unit, and no wave without a row
    int groups = (rows + per_group - 1) / per_group;
    if (groups > 2 * info.compute_units) groups = 2 * info.compute_units;
    const int waves = groups * per_group;
#define MACKO_HEAD(NP_)                                                                                                  \
    if (pieces <= NP_ * kWave) {                                                                                         \
        hipLaunchKernelGGL(norm_matvec_kernel<NP_>, dim3(groups), dim3(kHeadThreads), 0, as_stream(stream),              \
                           (const u32x4 *)w, (const u32x4 *)x, (const u32x4 *)norm_weight, (uint16_t *)y, rows, pieces,   \
                           eps, rows / waves, rows % waves);                                                             \
        return (int)hipGetLastError();                                                                                   \
    }
    MACKO_HEAD(1)
    MACKO_HEAD(2)
    MACKO_HEAD(4)
    MACKO_HEAD(8)
#undef MACKO_HEAD
    return MACKO_E_INVALID_ARGUMENT;
}
