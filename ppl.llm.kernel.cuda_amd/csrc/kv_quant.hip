// KV-cache quantise/append for gfx950: fp16 K/V -> symmetric int8 in groups of 8
// channels with one fp16 scale per group, scattered into the cache.
//
// Arithmetic restated from the reference kernel
// (src/ppl/kernel/llm/cuda/pmx/multi_head_cache_attention/kernel.cu:128-154):
//   absmax over the group in half; scale = half(float(absmax) / 127.0f);
//   scale = scale > eps ? scale : eps with eps = half(1e-5f) (a half subnormal);
//   q = (int8) round-half-even( half(x / scale) ).
// The half quotient is the correctly rounded binary32 quotient rounded once more to
// binary16, which equals the correctly rounded half quotient (24 >= 2*11 + 2); the
// binary32 quotient comes from one division per group (the reciprocal of the scale) and
// a residual correction per element, see quantise_group.  The integer rounding is an
// addition in half (1536 + h, ulp one) -- HIP's __half2short_rn truncates, so it is not used.
//
// Decomposition (this file's own): a flat grid over (new token, group of 8
// channels); one lane owns one group of K and the same group of V: two 128-bit
// loads, two 64-bit int8 stores, two 16-bit scale stores.  The sequence of a
// token is found by bisection over seqstarts, so no workgroup is launched per
// (position, sequence) pair that does not exist.
#include <cmath>
#include <cstring>

#include "device_common.h"
#include "launch_params.h"

namespace pmxhip {

namespace {

constexpr int kQuantThreads = 256;

struct Quantised {
    u32x2 q;
    half_t scale;
};

// float(h.x) * b + c and float(h.y) * b + c with the half operand read in place (one instruction, one rounding)
__device__ __forceinline__ float fma_half_lo(half2_t h, float b, float c)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float fma_half_hi(half2_t h, float b, float c)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(b), "v"(c));
    return r;
}
// float(h.x) - a * b and float(h.y) - a * b (the negation is a source modifier)
__device__ __forceinline__ float half_lo_minus_product(half2_t h, float a, float b)
{
    float r;
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(r) : "v"(a), "v"(b), "v"(h));
    return r;
}
__device__ __forceinline__ float half_hi_minus_product(half2_t h, float a, float b)
{
    float r;
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(a), "v"(b), "v"(h));
    return r;
}

__device__ __forceinline__ Quantised quantise_group(const u32x4 raw)
{
    half2_t x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = bitcast<half2_t>(raw[i]);
    // absmax in half, two channels at a time (sign bits cleared, packed maximum), then the two halves of the result
    half2_t m2 = bitcast<half2_t>(raw[0] & 0x7fff7fffu);
#pragma unroll
    for (int i = 1; i < 4; ++i) m2 = __builtin_elementwise_max(m2, bitcast<half2_t>(raw[i] & 0x7fff7fffu));
    const half_t amax = m2.x > m2.y ? m2.x : m2.y;
    const half_t eps = (half_t)1e-5f;
    // float(amax) / 127.0f, correctly rounded, without the division sequence: with r = fl(1 / 127), q0 = a * r,
    // e = fma(-q0, 127, a), q = fma(e, r, q0).  Equal to the correctly rounded quotient for every positive finite
    // half a (all 31 743 compared in exact arithmetic on the CPU).
    const float af = (float)amax;
    const float r127 = 1.0f / 127.0f;
    const float s0 = af * r127;
    half_t s = (half_t)__builtin_fmaf(__builtin_fmaf(-s0, 127.0f, af), r127, s0);
    s = s > eps ? s : eps;
    const float sf = (float)s;
    // One correctly rounded reciprocal per group, then a residual step per element:
    //   q0 = x * rcp, e = fma(-q0, sf, x), quotient = fma(e, rcp, q0).
    // Rounded to half this equals the correctly rounded quotient for every pair of a finite half x and a half
    // scale >= eps (all 2.0e9 pairs compared on the CPU; the one difference, -0 / s -> +0, yields the same int8 0).
    // The half channels enter the mixed-precision multiply-adds in place, two quotients are rounded to half by one
    // packed conversion, and the integer rounding is an addition: 1536 + h in half has an ulp of one, so the sum
    // is h rounded to the nearest integer with ties to even, and its low byte is that integer in two's
    // complement (|h| <= 127.4, the sum stays inside [1024, 2048)).
    const float rcp = 1.0f / sf;
    const half2_t magic = {(half_t)1536.0f, (half_t)1536.0f};
    uint32_t biased[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a0 = fma_half_lo(x[i], rcp, 0.0f), a1 = fma_half_hi(x[i], rcp, 0.0f);
        const float e0 = half_lo_minus_product(x[i], a0, sf), e1 = half_hi_minus_product(x[i], a1, sf);
        const float q0 = __builtin_fmaf(e0, rcp, a0), q1 = __builtin_fmaf(e1, rcp, a1);
        typedef float float2_t __attribute__((ext_vector_type(2)));
        const half2_t h = __builtin_convertvector(float2_t{q0, q1}, half2_t); // round to nearest even, both at once
        biased[i] = bitcast<uint32_t>(h + magic);
    }
    Quantised r;
    // bytes 0 and 2 of each word are the integers of its two channels
    r.q = u32x2{__builtin_amdgcn_perm(biased[1], biased[0], 0x06040200u), __builtin_amdgcn_perm(biased[3], biased[2], 0x06040200u)};
    r.scale = s;
    return r;
}

// largest b in [0, n) with starts[b] <= v   (starts non-decreasing, starts[0] <= v < starts[n]);
// being the largest, it is never an empty sequence
template <typename PTR>
__device__ __forceinline__ int sequence_of(PTR starts, int n, int64_t v)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (starts[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The same index found by the wave's lanes together: the number of sequences that end at or before v (every lane
// of the wave must be here, with the same v).  Each lane compares one entry per 64, all requested at once: one
// memory latency where the bisection has log2(n) of them in a row.
constexpr int kCountedSequences = 1024;
__device__ __forceinline__ int sequence_by_count(const int64_t* starts, int n, int64_t v, int lane)
{
    int count = 0;
    for (int i0 = 0; i0 < n; i0 += kWave) {
        const int i = i0 + lane;
        const bool ends_before = i < n && starts[i + 1] <= v;
        count += __builtin_popcountll(__builtin_amdgcn_ballot_w64(ends_before));
    }
    return count < n ? count : n - 1;
}

} // namespace

// stride_tokens: tokens between a thread's units, (workgroups * threads) / groups_per_token; the host sizes the launch
// so that this division is exact whenever a thread takes more than one unit, which keeps a thread on one
// (head, channel group) for all its units: the two integer divisions below then happen once, not once per unit.
// WAVE_TOKEN: a token row has a multiple of 64 groups, so the 64 lanes of a wave always work on one token: what
// follows from the token alone (its sequence, position, cache row and the row bases) is then found once per wave
// on the scalar unit, with scalar loads of the index arrays, and a lane adds only its offset inside the row.
template <bool PAGED, bool WAVE_TOKEN>
__global__ __launch_bounds__(kQuantThreads) void kv_quantize_kernel(const QuantLaunch a, const uint32_t stride_tokens)
{
    const uint32_t groups_per_head = (uint32_t)a.head_dim >> 3;
    const uint32_t groups_per_token = (uint32_t)a.num_kv_heads * groups_per_head;
    const const_i64_ptr seqstarts = as_constant(a.seqstarts);
    const const_i64_ptr start_pos = as_constant(a.start_pos);
    const const_i64_ptr cachestarts = as_constant(a.cachestarts);
    const int64_t first = seqstarts[0];
    const int64_t n_tokens = seqstarts[a.batch] - first;
    const uint32_t u0 = blockIdx.x * kQuantThreads + threadIdx.x; // the host keeps workgroups * threads below 2^31
    uint32_t tok0 = u0 / groups_per_token;
    const uint32_t gi = u0 - tok0 * groups_per_token;
    if (WAVE_TOKEN) tok0 = __builtin_amdgcn_readfirstlane(tok0);
    const uint32_t h = gi / groups_per_head;
    const uint32_t d0 = (gi - h * groups_per_head) << 3;
    const uint32_t in_idx = h * (uint32_t)a.head_dim + d0;                   // halves inside a K/V row
    const int64_t out_idx = a.layer_idx * a.cache_stride_l + (int64_t)h * a.cache_stride_h + d0;
    for (int64_t tok = tok0; tok < n_tokens; tok += stride_tokens) {
        const int64_t in_tok = first + tok;
        // the rows to quantise do not depend on the sequence: requested first, they travel during the index lookups
        const u32x4 kraw = *(const u32x4*)((const half_t*)a.current_key + in_tok * a.current_key_stride_s + in_idx);
        const u32x4 vraw = *(const u32x4*)((const half_t*)a.current_value + in_tok * a.current_value_stride_s + in_idx);
        // decode steps have one new token per sequence: token i then belongs to sequence i, which two independent
        // loads confirm; otherwise the sequence is found by bisection (a chain of dependent loads)
        // (the sequence's start_pos is requested together with them, so that the decode step's chain of dependent
        // loads is index arrays -> page table -> stores)
        int b;
        int64_t pos;
        const int64_t ti = tok < a.batch ? tok : 0;
        const int64_t s0 = seqstarts[ti], s1 = seqstarts[ti + 1], sp = start_pos[ti];
        if (tok < a.batch && s0 == in_tok && s1 > in_tok) {
            b = (int)tok;
            pos = sp;
        } else {
            b = sequence_of(seqstarts, (int)a.batch, in_tok);
            pos = start_pos[b] + (in_tok - seqstarts[b]);
        }
        const int64_t tb = PAGED ? (int64_t)b * a.cachestarts_stride_b : (int64_t)b;
        const int64_t row = PAGED ? cachestarts[tb + (pos >> 7)] + (pos & (kPage - 1)) : cachestarts[tb] + pos;

        const Quantised kq = quantise_group(kraw);
        const Quantised vq = quantise_group(vraw);

        const int64_t k_out = row * a.cache_stride_s + out_idx;
        const int64_t v_out = k_out + a.cache_stride_kv;
        // Non-temporal: a wave writes whole lines (16 lanes x 8 bytes per row of a head, 64 scales), nothing here
        // reads them again, and lines left dirty in the memory-side cache are written back during the kernel that
        // runs next: the decode launch behind a prefill step's append (28 MB of rows) then took 17 us longer.
        __builtin_nontemporal_store(kq.q, (u32x2*)(a.cache + k_out));
        __builtin_nontemporal_store(vq.q, (u32x2*)(a.cache + v_out));
        __builtin_nontemporal_store(kq.scale, &((half_t*)a.scale)[k_out >> 3]);
        __builtin_nontemporal_store(vq.scale, &((half_t*)a.scale)[v_out >> 3]);
    }
}

// Rotary position embedding of Q and K (interleaved pairs, reference:
// src/ppl/kernel/llm/cuda/pmx/rotary_position_embedding.cu:35-91, 268-343), optionally fused with the
// quantise/append above: a workgroup takes a few consecutive tokens; the cos/sin of a token's position are computed
// once per pair (not once per head) and shared through LDS; a lane then rotates one group of 8 channels
// of a query head, or rotates and quantises the same group of K and quantises that of V.
//
// Angle (one definition for device and CPU): inv = 1.0f / float(pow(theta', i / (rotary_dim / 2)));
// angle = inv * float(pos) (linear scaling: inv * (float(pos) / factor)); cos and sin are those of the
// binary32 angle, correctly rounded to binary32 (evaluated in binary64).  The reference evaluates the
// same formula with the approximate __powf / __sincosf intrinsics.
//
// LOOP: the launch has fewer workgroups than the step may have tokens (launch_rope) and they walk the tokens in turn; without it
// every token has its workgroup and the code of a turn stands alone.  DIVIDE: a unit's token and head by integer divisions,
// where the reciprocals are not exact.  Neither is decided in the kernel: at decode sizes what it waits for is
// its own instructions on their way from memory, and with both in one kernel a step of few heads took a fifth longer (8 / 8 heads of 64,
// 128 decode sequences, fused 5.2 us in a replayed graph, 4.3 apart; 32 / 8 of 128 5.5 and 5.0; the mixed step 39.1 and 38.6).
template <bool PAGED, bool LOOP, bool DIVIDE>
__global__ __launch_bounds__(kQuantThreads) void rope_append_kernel(const RopeLaunch a)
{
    // a workgroup takes as many consecutive tokens as its threads can compute coefficients for in one go
    __shared__ float s_cos[kQuantThreads], s_sin[kQuantThreads];
    __shared__ int64_t s_row[kQuantThreads / 4];
    const int pairs = a.head_dim >> 1, rd2 = a.rotary_dim >> 1;
    const int tokens_per_wg = a.tokens_per_wg; // at most kQuantThreads / pairs; pairs <= 128
    const int64_t first = a.seqstarts[0];
    const int64_t n_tokens = a.seqstarts[a.batch] - first;
    const bool append = a.cache != nullptr;
    for (int64_t tok0 = (int64_t)blockIdx.x * tokens_per_wg; tok0 < n_tokens; tok0 += (int64_t)gridDim.x * tokens_per_wg) {
    int thread = threadIdx.x;
    if constexpr (LOOP) asm volatile("" : "+v"(thread)); // (nothing that depends on it is held from turn to turn)

    // the rows of this workgroup's tokens, as units of 8 channels: the query heads' groups, and the key heads' (a key unit
    // also carries the same group of V when the step appends)
    const int gph = a.head_dim >> 3; // groups of 8 channels per head
    const int q_units = (int)a.num_heads * gph;
    const int k_units = (int)a.num_key_heads * gph;
    int n_here = tokens_per_wg;
    if (tok0 + n_here > n_tokens) n_here = (int)(n_tokens - tok0);
    const int q_work = n_here * q_units, k_work = n_here * k_units;
    const half_t* const value = (const half_t*)(append ? a.value : a.key); // (read for nothing where nothing is appended)
    const int64_t value_stride = append ? a.value_stride_s : a.key_stride_s;

    struct Unit {
        int tl, h, d0;
        int64_t in_tok, idx;
    };
    auto unit_of = [&](int w, int per_token, uint32_t magic) -> Unit {
        Unit r;
        r.tl = DIVIDE ? w / per_token : (int)__umulhi((uint32_t)w, magic);
        const int u = w - r.tl * per_token;
        r.h = DIVIDE ? u / gph : (int)__umulhi((uint32_t)u, a.gph_magic);
        r.d0 = (u - r.h * gph) << 3;
        r.in_tok = first + tok0 + r.tl;
        r.idx = (int64_t)u << 3;
        return r;
    };
    // Units beyond the work load the last unit's rows: every load of a batch is issued whatever the remainder, so that
    // the wait for a batch leaves the next one in flight.
    constexpr int kQueries = 3; // query units per thread and batch; key units one
    // The query units start at the wave behind the last key unit's: a token of few heads has its query and key units in different
    // waves (8 / 1 heads of 128, 128 decode sequences, fused: 4.7 us where they share one, 4.4 so).
    const int q_thread = (thread - ((k_work + kWave - 1) & ~(kWave - 1))) & (kQuantThreads - 1);
    auto load_queries = [&](int w0, u32x4 (&rows)[kQueries]) {
#pragma unroll
        for (int j = 0; j < kQueries; ++j) {
            const int w = w0 + q_thread + j * kQuantThreads;
            const Unit r = unit_of(w < q_work ? w : q_work - 1, q_units, a.q_magic);
            rows[j] = *(const u32x4*)((const half_t*)a.query + r.in_tok * a.query_stride_s + r.idx);
        }
    };
    auto load_key = [&](int w0, u32x4& k, u32x4& v) {
        const int w = w0 + (int)thread;
        const Unit r = unit_of(w < k_work ? w : k_work - 1, k_units, a.k_magic);
        k = *(const u32x4*)((const half_t*)a.key + r.in_tok * a.key_stride_s + r.idx);
        v = *(const u32x4*)(value + r.in_tok * value_stride + r.idx);
    };

    // The rows depend on nothing that follows (index arrays -> sequence -> cos/sin and cache row), so a thread's
    // first units are requested before all that and travel meanwhile; a decode step, with a token per workgroup
    // and a few units per thread, has no others.
    u32x4 q_row[kQueries], k_row = {0, 0, 0, 0}, v_row = {0, 0, 0, 0};
    if (k_units > 0) load_key(0, k_row, v_row);
    load_queries(0, q_row);

    {
        const int tl = thread / pairs, i = thread - tl * pairs;
        const int64_t tok = tok0 + tl;
        const bool active = tl < tokens_per_wg && tok < n_tokens;
        const int64_t in_tok = first + tok;
        // The token's sequence.  One new token per sequence (a decode step): token i belongs to sequence i, which two
        // independent loads confirm.  Otherwise the lanes of the wave count, for each token the wave covers, the
        // sequences that end before it (one latency); beyond kCountedSequences sequences every thread bisects (a
        // chain of dependent loads).
        int b = -1;
        int64_t pos = 0;
        const bool count_search = a.batch <= kCountedSequences;
        if (active && (n_tokens == a.batch || !count_search)) {
            const int64_t ti = tok < a.batch ? tok : 0;
            const int64_t s0 = a.seqstarts[ti], s1 = a.seqstarts[ti + 1], sp = a.start_pos[ti];
            if (tok < a.batch && s0 == in_tok && s1 > in_tok) {
                b = (int)tok;
                pos = sp;
            }
        }
        if (count_search) { // every lane of the wave is here
            const int wave0 = thread & ~(kWave - 1);
            const int tl_hi = (wave0 + kWave - 1) / pairs;
            for (int t = wave0 / pairs; t <= tl_hi; ++t) {
                const int64_t tk = tok0 + t;
                if (t >= tokens_per_wg || tk >= n_tokens) break;
                if (__builtin_amdgcn_ballot_w64(tl == t && b < 0) == 0) continue;
                const int bt = sequence_by_count(a.seqstarts, (int)a.batch, first + tk, thread & (kWave - 1));
                if (tl == t && b < 0) {
                    b = bt;
                    pos = a.start_pos[bt] + (first + tk - a.seqstarts[bt]);
                }
            }
        } else if (active && b < 0) {
            b = sequence_of(a.seqstarts, (int)a.batch, in_tok);
            pos = a.start_pos[b] + (in_tok - a.seqstarts[b]);
        }
        if (active) {
            float c = 1.f, s = 0.f;
            if (i < rd2) {
                float th = a.theta;
                if (a.scaling_type == 2) { // dynamic: rotary_position_embedding.cu:68-91
                    const int64_t pos_end = a.start_pos[b] + (a.seqstarts[b + 1] - a.seqstarts[b]);
                    if (pos_end > a.max_position_embeddings) {
                        const float base = ((a.scaling_factor * (float)pos_end) / (float)a.max_position_embeddings) - (a.scaling_factor - 1.f);
                        const float expn = (float)rd2 / (float)(rd2 - 1);
                        th = a.theta * (float)pow((double)base, (double)expn);
                    }
                }
                // theta^(i / rd2) is the same for every token unless the dynamic scaling applies: then it comes in the
                // launch arguments and the binary64 pow leaves the kernel
                const float inv = a.has_inv_freq ? a.inv_freq[i] : 1.0f / (float)pow((double)th, (double)((float)i / (float)rd2));
                const float p = a.scaling_type == 1 ? (float)pos / a.scaling_factor : (float)pos;
                const float angle = inv * p;
                double sd, cd;
                sincos((double)angle, &sd, &cd); // one argument reduction for both
                c = (float)cd;
                s = (float)sd;
            }
            s_cos[thread] = c;
            s_sin[thread] = s;
            if (i == 0 && append)
                s_row[tl] = token_row<PAGED>(a.cachestarts, PAGED ? (int64_t)b * a.cachestarts_stride_b : (int64_t)b, pos);
        }
    }
    __syncthreads();

    auto rotate = [&](const u32x4 raw, int d0, int tl) -> u32x4 {
        u32x4 out;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int i = (d0 >> 1) + w;
            const half2_t h = bitcast<half2_t>(raw[w]);
            if (i < rd2) {
                const float x = (float)h.x, y = (float)h.y, c = s_cos[tl * pairs + i], s = s_sin[tl * pairs + i];
                const half2_t r = {(half_t)(x * c - y * s), (half_t)(y * c + x * s)};
                out[w] = bitcast<uint32_t>(r);
            } else {
                out[w] = raw[w];
            }
        }
        return out;
    };

    auto finish_query = [&](int w, const u32x4 raw) {
        const Unit r = unit_of(w, q_units, a.q_magic);
        *(u32x4*)((half_t*)a.rotated_query + r.in_tok * a.rotated_query_stride_s + r.idx) = rotate(raw, r.d0, r.tl);
    };
    auto finish_key = [&](int w, u32x4 raw, const u32x4 vraw) {
        const Unit r = unit_of(w, k_units, a.k_magic);
        if (!a.bypass_key) raw = rotate(raw, r.d0, r.tl);
        if (a.rotated_key) *(u32x4*)((half_t*)a.rotated_key + r.in_tok * a.rotated_key_stride_s + r.idx) = raw;
        if (append) {
            const Quantised kq = quantise_group(raw);
            const Quantised vq = quantise_group(vraw);
            const int64_t k_out = s_row[r.tl] * a.cache_stride_s + a.layer_idx * a.cache_stride_l + (int64_t)r.h * a.cache_stride_h + r.d0;
            const int64_t v_out = k_out + a.cache_stride_kv;
            __builtin_nontemporal_store(kq.q, (u32x2*)(a.cache + k_out));
            __builtin_nontemporal_store(vq.q, (u32x2*)(a.cache + v_out));
            __builtin_nontemporal_store(kq.scale, &((half_t*)a.scale)[k_out >> 3]);
            __builtin_nontemporal_store(vq.scale, &((half_t*)a.scale)[v_out >> 3]);
        }
    };
    // The next units travel while these are rotated and stored: one after the other, each waiting for its own rows, a
    // workgroup of four tokens of 32 query / 8 kv heads of 128 spent seven memory latencies in a row.
    int w0 = 0;
    for (; w0 + kQuantThreads <= k_work; w0 += kQuantThreads) {
        u32x4 k_next, v_next;
        load_key(w0 + kQuantThreads, k_next, v_next);
        finish_key(w0 + (int)thread, k_row, v_row);
        k_row = k_next;
        v_row = v_next;
    }
    if (w0 + (int)thread < k_work) finish_key(w0 + (int)thread, k_row, v_row);
    for (w0 = 0; w0 + kQueries * kQuantThreads <= q_work; w0 += kQueries * kQuantThreads) {
        u32x4 next[kQueries];
        load_queries(w0 + kQueries * kQuantThreads, next);
#pragma unroll
        for (int j = 0; j < kQueries; ++j) finish_query(w0 + q_thread + j * kQuantThreads, q_row[j]);
#pragma unroll
        for (int j = 0; j < kQueries; ++j) q_row[j] = next[j];
    }
#pragma unroll
    for (int j = 0; j < kQueries; ++j) {
        const int w = w0 + q_thread + j * kQuantThreads;
        if (w < q_work) finish_query(w, q_row[j]);
    }
    if constexpr (!LOOP) return;
    __syncthreads(); // the next tokens' coefficients overwrite these
    }
}

static uint32_t bitcast_host(float v)
{
    uint32_t u;
    memcpy(&u, &v, sizeof(u));
    return u;
}

int launch_rope(const RopeLaunch& a_in, int compute_units, hipStream_t stream)
{
    if (a_in.max_tokens <= 0) return kLaunchOk;
    if (a_in.head_dim > 256 || a_in.head_dim < 8) return kLaunchNoKernel;
    RopeLaunch a = a_in;
    const int pairs = a.head_dim / 2, rd2 = a.rotary_dim / 2;
    a.has_inv_freq = 0;
    if (a.scaling_type != 2 && rd2 <= 128) {
        // a model has one such table: the thread's last one is kept (64 powers cost as much as the launch)
        static thread_local struct { float theta; int rd2; float table[128]; } last = {0.f, -1, {}};
        if (last.rd2 != rd2 || bitcast_host(last.theta) != bitcast_host(a.theta)) {
            for (int i = 0; i < rd2; ++i) last.table[i] = 1.0f / (float)pow((double)a.theta, (double)((float)i / (float)rd2));
            last.theta = a.theta;
            last.rd2 = rd2;
        }
        memcpy(a.inv_freq, last.table, sizeof(float) * rd2);
        a.has_inv_freq = 1;
    }
    // A workgroup computes the coefficients of its tokens once and shares them through LDS: as many tokens as its
    // threads have pairs for, but no more than leaves two workgroups per CU (a decode step has a token per sequence,
    // and a workgroup works through its tokens' rows one after the other)
    int tokens_per_wg = kQuantThreads / pairs;
    const int64_t spread = a.max_tokens / (2 * (int64_t)(compute_units > 0 ? compute_units : 256));
    if (tokens_per_wg > spread) tokens_per_wg = spread > 1 ? (int)spread : 1;
    a.tokens_per_wg = tokens_per_wg;
    // n / d = mulhi(n, floor(2^32 / d) + 1) for n d < 2^32 and d >= 2: exact for every unit of a workgroup, or divide
    const uint64_t gph = (uint64_t)(a.head_dim >> 3);
    bool exact = gph >= 2;
    auto magic = [&](uint64_t per_token) -> uint32_t {
        if (per_token == 0) return 0; // (no such unit)
        if (per_token >= (1u << 16) || (uint64_t)tokens_per_wg * per_token * per_token >= (1ull << 32)) exact = false;
        return (uint32_t)((1ull << 32) / per_token + 1);
    };
    a.q_magic = magic((uint64_t)a.num_heads * gph);
    a.k_magic = magic((uint64_t)a.num_key_heads * gph);
    a.gph_magic = magic(gph);
    // max_tokens is batch * max_seqlen, in a mixed step many times the rows there are: about as many workgroups as the chip holds
    // at once (67 vector registers: seven per CU) walk the tokens in turn.  Seven, eight or fourteen per CU measure the same
    // (mixed step 43.1 us over one set of rows).
    int64_t blocks = (a.max_tokens + tokens_per_wg - 1) / tokens_per_wg;
    const int64_t resident = 8 * (int64_t)(compute_units > 0 ? compute_units : 256);
    const bool loop = blocks > resident;
    if (loop) blocks = resident;
    const dim3 grid((unsigned)blocks);
#define PMX_ROPE(LOOP, DIVIDE) \
    do { \
        if (a.cache_mode == 1) hipLaunchKernelGGL((rope_append_kernel<true, LOOP, DIVIDE>), grid, dim3(kQuantThreads), 0, stream, a); \
        else hipLaunchKernelGGL((rope_append_kernel<false, LOOP, DIVIDE>), grid, dim3(kQuantThreads), 0, stream, a); \
    } while (0)
    if (!exact) PMX_ROPE(true, true);
    else if (loop) PMX_ROPE(true, false);
    else PMX_ROPE(false, false);
#undef PMX_ROPE
    return kLaunchOk;
}

int launch_kv_quantize(const QuantLaunch& a, int compute_units, hipStream_t stream)
{
    const int64_t groups_per_token = (int64_t)a.num_kv_heads * (a.head_dim >> 3);
    const int64_t max_units = a.max_tokens * groups_per_token;
    if (max_units <= 0) return kLaunchOk;
    int64_t blocks = (max_units + kQuantThreads - 1) / kQuantThreads;
    // grid-stride beyond this: eight workgroups per CU hold every wave slot at once, and a lane then takes two or
    // three units in turn (11 104 new tokens of 8 heads x 128 channels on 256 CUs: 23.4 us against 28 us with four
    // times as many workgroups and one unit per lane, 36 us with 32 times as many, most of them without a unit;
    // 25 us with half as many)
    const int64_t cap = (int64_t)(compute_units > 0 ? compute_units : 256) * 8;
    if (blocks > cap) {
        // a whole number of token rows per sweep of the grid, so that a thread keeps its (head, channel group):
        // the workgroup count is a multiple of groups_per_token / gcd(groups_per_token, threads per workgroup)
        int64_t g = groups_per_token, t = kQuantThreads;
        while (t != 0) {
            const int64_t r = g % t;
            g = t;
            t = r;
        }
        const int64_t unit = groups_per_token / g;
        blocks = cap / unit * unit;
        if (blocks == 0) blocks = unit;
    }
    if (blocks * kQuantThreads >= (int64_t)1 << 31) return kLaunchNoKernel;
    // exact when blocks was rounded above; otherwise no thread takes a second unit and the value only has to carry
    // a thread beyond the last token
    const uint32_t stride_tokens = (uint32_t)((blocks * kQuantThreads + groups_per_token - 1) / groups_per_token);
    const bool wave_token = groups_per_token % kWave == 0;
    const dim3 grid((unsigned)blocks), block(kQuantThreads);
    if (a.cache_mode == 1) {
        if (wave_token) hipLaunchKernelGGL((kv_quantize_kernel<true, true>), grid, block, 0, stream, a, stride_tokens);
        else hipLaunchKernelGGL((kv_quantize_kernel<true, false>), grid, block, 0, stream, a, stride_tokens);
    } else {
        if (wave_token) hipLaunchKernelGGL((kv_quantize_kernel<false, true>), grid, block, 0, stream, a, stride_tokens);
        else hipLaunchKernelGGL((kv_quantize_kernel<false, false>), grid, block, 0, stream, a, stride_tokens);
    }
    return kLaunchOk;
}

} // namespace pmxhip
