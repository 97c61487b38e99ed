// Decode attention over the int8 group-8 KV cache, variant for whole sequences of every shape, for five to sixteen query heads per
// kv head at head_dim 128 over long token ranges, for the shared pieces of a single sequence and for a few sequences at head_dim 64 (reference: src/ppl/kernel/llm/cuda/pmx/multi_head_cache_attention/kernel.cu:1090-1891,
// the GQCA kernel, which also puts the query heads of a kv head on tensor cores), and for short prefill chunks.
//
// With that many query heads the per-head arithmetic of the VALU kernels outweighs the cache stream.
// Here a wave owns one kv head and treats its query heads as the columns of two small matrix products per block of
// 32 tokens:
//   S^T = K Q^T   (32 tokens x C columns)
//   O^T = V^T P^T (head_dim channels x C columns)
// so the arithmetic per cache byte no longer grows with the number of query heads; what stays on the
// VALU is the dequantisation (once per byte) and a softmax over 32 x C logits per block.
//
// Two forms: C = 16 on v_mfma_f32_16x16x32_f16 (half the MFMA time, half the logits per lane) and C = 32 on
// v_mfma_f32_32x32x16_f16.  More columns than that (multi-query models: 48 or 71 query heads on one kv head) run as
// passes (blockIdx.z), each of which reads the cache again: the bytes of one kv head are few and stay in the L2.
//
// Exactness follows the prefill kernel: K^ = int8 * scale, V^ and p are kept as hi + lo pairs of halves
// (2 MFMAs per QK step, 3 per PV step), so no fp16 rounding of the dequantised cache enters the result.  Those pairs hold 22 bits
// where the quad and general kernels, which served some of these batches before, multiply p and V in float32, and the product of the two
// low parts, 2^-22 of a term, is left out.  Against float64 the error is no larger than theirs: the float32 pieces of one sequence of
// 512 tokens are off by 3.3e-7 (rms, of 8 / 8 heads of 64) to 4.8e-7 (32 / 8 of 128), on the quad kernel by 4.4e-7 (8 / 8 of 64), and the half
// outputs of twelve shapes of decode batches and seven of short chunks by their rounding to half alone (2.06e-4 to 2.10e-4, to four
// digits; 12 / 3 heads of 96, 20 chunks of 1-5 rows 2.064e-4, on the tile kernel, whose row sums run over p's high halves, 2.075e-4).
//
// The cache rows travel from memory into a wave-private LDS ring without registers (global_load_lds), two blocks
// ahead of the arithmetic, and across sequences: the blocks of a range are one stream to the requests, so the first
// rows of a sequence are on their way while the one before it is finished.  Both operands are read from the ring in
// the lanes that need them:
//   K: a lane holds one token's share of the channels, as 16-byte pieces;
//   V: the rows of O^T are numbered so that a lane's row of every product lies in ONE quantisation group -- row r is
//      group r (C = 16: product e has channel 8 r + e) -- and the k-order is the order in which the S^T accumulators
//      hold their tokens.  A lane then reads eight bytes of each of its eight tokens, and its operands of eight
//      products are byte e of those words times the token's scale of its own group: no transposition through LDS.
//      (The scales of a group's tokens come with the transposing LDS read: its column i is group i.)
// A ring slot is 10 KB at head_dim 128, two slots and eight waves are the 160 KB of a CU.
//
// What bounds it: over long ranges the arithmetic beside the cache stream (a wave's requests alone stream at 7.1 TB/s; two waves
// per SIMD have some 460 vector instructions and 40 products per block to issue), with short sequences the chain of look-ups,
// first rows and results of every wave.  Layer calls against the kernel of decode_attn_mfma.hip, which transposes V through LDS and requests
// a block ahead into registers: 64 q / 8 kv heads of 128, 32 sequences of 10923-32768 tokens 338 -> 320 us, four of 30000-32768 72.1 -> 68.7
// (over short ranges that one is the faster: decode_ring).  Whole sequences in one launch, against ranges and a combine launch: 32 / 8 heads,
// four of 85-256 14.7 -> 9.3; 8 / 1 heads of 256, 448 of 92-148 38.6 -> 19.1; 28 / 4 heads, 49 of 138-381 18.7 -> 15.2.
// The form of 32 columns holds 255-256 VGPRs at head_dim 128 and spills two to four (12-20 bytes of scratch a lane); no other form spills.
//
// Ranges, pieces and the workspace are those of decode_attn.hip: one workgroup (a wave per kv head: four, or two
// or one when the kv heads do not come in fours) per token range, cuts on multiples of 32 tokens, float32 pieces merged by decode_combine_kernel.
#include "decode_common.h"

namespace pmxhip {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

constexpr int kMfmaBlock = 32;   // tokens per wave iteration
constexpr float kPShift = 14.0f; // p is kept as 2^14 * exp2(logit - max): its half parts stay normal numbers

// 4 bytes per lane to LDS address `lds` + 4 * lane (load_to_lds16's narrow sibling: scale rows are 4-byte aligned only)
__device__ __forceinline__ void load_to_lds4(uint32_t lds, uint32_t offset, const void* base)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
// the wave's LDS reads are done: what they read may be overwritten by a request from memory
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A query fragment requested ahead of its use; await_query is the statement that makes it readable.
__device__ __forceinline__ void request_query(f16x8& dst, const half_t* p)
{
    asm volatile("global_load_dwordx4 %0, %1, off" : "+v"(dst) : "v"(p) : "memory");
}
// (every path's wait comes before the one statement that all fragments pass through: no copy of a fragment can be
// placed between its request and its wait)
template <int N, int KS>
__device__ __forceinline__ void await_query(f16x8 (&q)[KS], bool requests_behind)
{
    if (requests_behind) wait_vector_memory<N>();
    else wait_vector_memory<0>();
    if constexpr (KS == 8) asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]), "+v"(q[4]), "+v"(q[5]), "+v"(q[6]), "+v"(q[7])::"memory");
    else if constexpr (KS == 6) asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]), "+v"(q[4]), "+v"(q[5])::"memory");
    else if constexpr (KS == 4) asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3])::"memory");
    else if constexpr (KS == 3) asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2])::"memory");
    else asm volatile("" : "+v"(q[0]), "+v"(q[1])::"memory");
}

// The 16-byte chunk of a token's row that LDS position c holds: XORed with the token, so that both the K reads (eight
// consecutive tokens, one chunk) and the V reads (a row per 16 lanes) cover all banks.
template <int D>
__device__ __forceinline__ int ring_swizzle(int token)
{
    return D == 96 ? 0 : (D == 64 ? (token >> 1) & 3 : (token ^ (token >> 3)) & 7);
}

// halves (hi, lo) of two elements x * scale
__device__ __forceinline__ void dequantise(half2_t x, half2_t s, half2_t& hi, half2_t& lo)
{
    hi = x * s;
    lo = __builtin_elementwise_fma(x, s, -hi);
}
__device__ __forceinline__ f16x8 join(half2_t a, half2_t b, half2_t c, half2_t d)
{
    return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// the output of one column of an empty sequence, a quarter or half per lane of the column: the reference yields
// 0/(0+1e-6) = 0 (kernel.cu:516)
__device__ __forceinline__ void zero_column(const DecodeLaunch& a, int b, int head, int pos, int part, int parts)
{
    int64_t row = b;
    if (a.seqstarts != nullptr) {
        row = a.seqstarts[b] + pos;
        if (row >= a.seqstarts[b + 1]) return;
    }
    half_t* const out = (half_t*)a.output + row * a.output_stride_s + (int64_t)head * a.head_dim;
    for (int c = 4 * part; c < a.head_dim; c += 4 * parts) *(f16x4*)(out + c) = f16x4{0, 0, 0, 0};
}

// over the lanes of a column (lane ^ 32, and lane ^ 16 with four of them) through the vector unit's lane swaps: a
// data-share permute would have to wait for every LDS read already queued behind it
template <bool FOUR, typename F>
__device__ __forceinline__ float across_lanes(float v, F f)
{
    if constexpr (FOUR) {
        const u32x2 r = __builtin_amdgcn_permlane16_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
        v = f(bitcast<float>(r[0]), bitcast<float>(r[1]));
    }
    const u32x2 r = __builtin_amdgcn_permlane32_swap(bitcast<uint32_t>(v), bitcast<uint32_t>(v), false, false);
    return f(bitcast<float>(r[0]), bitcast<float>(r[1]));
}

constexpr int ring_slots(int D) { return D == 256 ? 1 : 2; }
constexpr int ring_slot_bytes(int D) { return 80 * D; } // K rows, V rows (32 D each), their scales (8 D each)

// One wave's work.  C: columns (16 or 32).  D: head_dim.
// Chunks (a.seqstarts given): the sequences have a few query tokens each instead of one (short prefill chunks, the
// candidate tokens of speculative decoding).  The columns of a kv head are then (query position, query head) pairs,
// column = position * (query heads per kv head) + head, a.num_kv_repeats counts those columns and a.num_heads the
// columns of all kv heads; a column attends the tokens below its own causal limit.  Everything else -- ranges, pieces,
// workspace -- is the decode step's, with columns in place of query heads.
// SEQ: the launch has a single range and workgroup x takes sequence x whole (nothing is left to merge).
// T: waves that share the tokens of every piece (short batches): each takes a run of its blocks, and their sums are merged
// through LDS before the piece is written.  NW waves with a kv head each, or T waves on one.
template <int C, int D, int NW, int T, bool SEQ>
__device__ __forceinline__ void decode_columns(const DecodeLaunch& a, char* const rings, const int wave, const int pass, const int G)
{
    static_assert(NW == 1 || T == 1, "kv heads or shares");
    static_assert(C == 16 || C == 32, "columns");
    static_assert(D == 64 || D == 96 || D == 128 || (D == 256 && C == 16), "head_dim");
    constexpr bool N16 = C == 16;
    constexpr int L = ring_slots(D);          // blocks requested ahead
    constexpr int SLOT = ring_slot_bytes(D);
    constexpr int GPT = D / 8;                // quantisation groups per token
    constexpr int CPR = D / 16;               // 16-byte chunks per row, and 4-byte pieces per row of scales
    constexpr int NI = D / 32;                // requests per block for the rows of K (or V), and as many for their scales
    constexpr int NK = 2 * NI;
    constexpr int KS = N16 ? D / 32 : D / 16; // k-steps of S^T
    constexpr int SETS = D == 256 ? 2 : 1;    // C = 16: sets of 16 groups
    constexpr int NE = N16 ? (D == 64 ? 4 : 8) : (D == 64 ? 2 : 4); // products per set: bytes of a lane's share of a group
    constexpr int TV = N16 ? 8 : 16;          // tokens whose V bytes a lane holds
    // whether a block's K bytes are read from the ring during the products of the block before it (where registers allow)
    constexpr bool K_AHEAD = L == 2 && (N16 || D == 64);

    char* const ring = rings + wave * (L * SLOT);
    const int lane = threadIdx.x & 63;
    const int col = N16 ? lane & 15 : lane & 31; // column of both products' results; row (token, channel) of their A operands
    const int kb = N16 ? lane >> 4 : lane >> 5;  // which block of eight along k
    const int l16 = lane & 15;
    const int gq = pass * C + col; // this lane's column among the kv head's G
    const int GR = a.seqstarts != nullptr ? (int)a.chunk_q_heads : G; // query heads per kv head
    const int cpos = a.seqstarts != nullptr ? gq / GR : 0;            // the column's query position within its sequence's chunk
    const int cg = gq - cpos * GR;                                    // ... and its query head within the kv head's group
    const int kvh = blockIdx.y * NW + (T > 1 ? 0 : wave);
    const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_address(ring));

    const const_i64_ptr kvstarts = as_constant(a.kvstarts);
    const const_i64_ptr cachestarts = as_constant(a.cachestarts);
    const bool paged = a.cache_mode == 1;
    int64_t kv_base = 0, r0, r1;
    if constexpr (SEQ) { // the workgroup's range is sequence blockIdx.x
        const int b = blockIdx.x;
        r0 = sequence_origin(kvstarts[b], b);
        r1 = r0 + (kvstarts[b + 1] - kvstarts[b]);
    } else {
        kv_base = kvstarts[0];
        const int64_t total = stream_length(kvstarts[a.decoding_batches] - kv_base, a.decoding_batches);
        const int64_t per = tokens_per_range(total, a.ranges, kMfmaBlock, a.min_tokens_per_range);
        r0 = (int64_t)blockIdx.x * per;
        if (r0 >= total) return;
        r1 = (r0 + per < total) ? r0 + per : total;
    }

    const int64_t head_off = a.layer_idx * a.cache_stride_l + (int64_t)kvh * a.cache_stride_h;
    const uint32_t stride_s32 = (uint32_t)a.cache_stride_s; // the host checks that a block's span fits 32 bits
    const char* const cache_k = (const char*)a.cache + head_off;
    const char* const cache_v = cache_k + a.cache_stride_kv;
    const char* const scale_k = (const char*)a.scale + (head_off >> 3) * 2;
    const char* const scale_v = scale_k + (a.cache_stride_kv >> 3) * 2;
    const float sm_scale = a.attn_scale * kLog2e;

    // ---- pieces of the range: the sequences it covers, in order ----
    struct Piece {
        int b, pa, pe, len;
        int64_t start; // kvstarts[b]
    };
    auto find_piece = [&](int b, Piece& p) -> bool { // the first non-empty piece of a sequence >= b
        for (; b < (SEQ ? (int)blockIdx.x + 1 : (int)a.decoding_batches); ++b) {
            const int64_t start = kvstarts[b];
            const int64_t first_token = start - kv_base;
            if (stream_length(first_token, b) >= r1) break;
            const int64_t len = kvstarts[b + 1] - start;
            int64_t pa, pe;
            piece_bounds(r0, r1, sequence_origin(first_token, b), len, kMfmaBlock, pa, pe);
            if (pe <= pa) continue;
            p.b = b;
            p.pa = (int)pa;
            p.pe = (int)pe;
            p.len = (int)len;
            p.start = start;
            return true;
        }
        return false;
    };

    // ---- requests: the blocks of all pieces in order, L of them ahead of the arithmetic ----
    uint32_t row_off[NI], scale_off[NI]; // this lane's chunk of a row, and its piece of a row of scales, per request
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int t = (64 * i + lane) / CPR, c = (64 * i + lane) % CPR;
        row_off[i] = (uint32_t)t * stride_s32 + 16 * (uint32_t)(c ^ ring_swizzle<D>(t));
        scale_off[i] = (uint32_t)t * (stride_s32 >> 2) + 4 * (uint32_t)c;
    }
    Piece ahead;       // the piece of the next block to request
    int ahead_pos = 0; // its first token
    int64_t ahead_entry = 0; // page table entry of that block, or the sequence's first row
    bool ahead_ok = false;
    auto look_up_row = [&]() { ahead_entry = cachestarts[paged ? (int64_t)ahead.b * a.cachestarts_stride_b + (ahead_pos >> 7) : (int64_t)ahead.b]; };
    auto advance = [&]() {
        ahead_pos += kMfmaBlock;
        if (ahead_pos >= ahead.pe) {
            ahead_ok = T == 1 && find_piece(ahead.b + 1, ahead); // (shared pieces: the ring is the place where they are merged)
            ahead_pos = ahead.pa;
        }
        if (ahead_ok) look_up_row();
    };
    auto request = [&](int slot, bool v) {
        // a block of 32 tokens starts on a multiple of 32 and so lies inside one 128-token page
        const int64_t boff = lane_value((ahead_entry + (paged ? ahead_pos & (kPage - 1) : ahead_pos)) * a.cache_stride_s, 0);
        const char* const rows = (v ? cache_v : cache_k) + boff;
        const char* const scales = (v ? scale_v : scale_k) + (boff >> 3) * 2;
        const uint32_t to = __builtin_amdgcn_readfirstlane(ring_lds + slot * SLOT + (v ? 32 * D : 0));
        const uint32_t to_scales = __builtin_amdgcn_readfirstlane(ring_lds + slot * SLOT + 64 * D + (v ? 8 * D : 0));
        const int last = ahead.pe - 1 - ahead_pos;
        if (last >= kMfmaBlock - 1) {
#pragma unroll
            for (int i = 0; i < NI; ++i) load_to_lds16<D % 128 == 0>(to + 1024 * i, row_off[i], rows); // (whole lines: non-temporal)
#pragma unroll
            for (int i = 0; i < NI; ++i) load_to_lds4(to_scales + 256 * i, scale_off[i], scales);
        } else { // a piece's last block: tokens beyond the piece re-read its last one (their logits are masked)
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int t = (64 * i + lane) / CPR, c = (64 * i + lane) % CPR;
                load_to_lds16<false>(to + 1024 * i, (uint32_t)(t < last ? t : last) * stride_s32 + 16 * (uint32_t)(c ^ ring_swizzle<D>(t)), rows);
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int t = (64 * i + lane) / CPR, c = (64 * i + lane) % CPR;
                load_to_lds4(to_scales + 256 * i, (uint32_t)(t < last ? t : last) * (stride_s32 >> 2) + 4 * (uint32_t)c, scales);
            }
        }
    };

    Piece cur;
    int first_sequence = blockIdx.x;
    if constexpr (!SEQ) first_sequence = find_sequence(kvstarts, a.kvstarts, (int)a.decoding_batches, r0, lane);
    if (!find_piece(first_sequence, cur)) {
        if (SEQ && gq < G) zero_column(a, (int)blockIdx.x, kvh * GR + cg, cpos, kb, N16 ? 4 : 2); // an empty sequence
        return;
    }

    // ---- query fragments (B operand of S^T): column gq, channels q_ch + ... of k-step s ----
    f16x8 qf[KS];
    int64_t q_row = 0; // row of the query and output tensors
    int qlen = 1;
    bool on = false;
    auto rows_of = [&](const Piece& p) { // the piece's query rows
        q_row = p.b;
        qlen = 1;
        if (a.seqstarts != nullptr) {
            q_row = as_constant(a.seqstarts)[p.b];
            qlen = (int)(as_constant(a.seqstarts)[p.b + 1] - q_row);
        }
        on = gq < G && cpos < qlen;
        if (qlen <= 0 && q_row > 0) --q_row; // a sequence without query rows: its columns read a row that exists
    };
    auto request_queries = [&]() {
        const half_t* qp = (const half_t*)a.query + (q_row + (on ? cpos : 0)) * a.query_stride_s + (int64_t)(kvh * GR + (on ? cg : 0)) * D;
        qp += N16 ? (D == 96 ? 8 : 16) * kb : D / 2 * kb;
#pragma unroll
        for (int s = 0; s < KS; ++s) request_query(qf[s], qp + (N16 ? (D == 96 ? 32 * s : 64 * (s >> 1) + 8 * (s & 1)) : 8 * s));
    };
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    bool next_requested = false; // the block after the current one is on its way
    bool requested = false;      // a K and a V block were requested behind the query fragments
    auto start = [&](const Piece& run) {
        ahead = run;
        ahead_pos = run.pa;
        ahead_ok = true;
        look_up_row(); // (its latency beside that of the query rows' look-up)
        rows_of(run);
        request_queries();
        if constexpr (T == 1) { // (a loop, because the code of a workgroup's start is fetched as it runs)
#pragma unroll 1
            for (int n = 0; n < 2 * L && ahead_ok; ++n) {
                request(n >> 1, n & 1);
                if (n & 1) advance();
                next_requested = n > 1;
            }
        } else {
            request(0, false);
            request(0, true);
            advance();
            if (L == 2 && ahead_ok) {
                request(1, false);
                request(1, true);
                advance();
                next_requested = true;
            }
        }
        requested = next_requested;
    };
    auto settle_queries = [&]() { // the fragments are there; columns without a query row are zero
        await_query<2 * NK>(qf, T > 1 || requested); // (T > 1: at least the first block's K and V were requested behind them)
        const uint32_t keep = on ? ~0u : 0u;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = bitcast<f16x8>(bitcast<u32x4>(qf[s]) & keep);
    };
    if (T == 1) start(cur);

    // ---- this lane's LDS reads: byte offsets inside a slot ----
    // K: token col (C = 16: and 16 + col)
    // V: tokens of the lane's k-block, in the order of its S^T results: C = 16: 16 (k / 4) + 4 kb + k % 4;
    //    C = 32: 16 (k / 8) + 8 (k / 4 % 2) + 4 kb + k % 4
    auto v_token = [&](int k) { return N16 ? 16 * (k >> 2) + 4 * kb + (k & 3) : 8 * (k >> 2) + 4 * kb + (k & 3); };
    // where the lane's bytes lie in a row: C = 16: the group's eight (head_dim 64: rows r and r + 8 share a group, four
    // bytes each); C = 32: rows r and r + 16 share a group, four bytes each (head_dim 64: four rows, two bytes each).
    // head_dim 96: the rows beyond group 11 repeat it and are dropped at the end.
    const int v_byte = N16 ? (D == 64 ? 8 * (col & 7) + 4 * (col >> 3) : 8 * (D == 96 && col > 11 ? 11 : col))
                           : (D == 64 ? 8 * (col & 7) + 2 * (col >> 3) : 8 * (D == 96 && (col & 15) > 11 ? 11 : col & 15) + 4 * (col >> 4));
    // (transposing read: within 16 lanes, lane i receives element i % 4 of lanes i / 4, 4 + i / 4, ...: four tokens of group i)
    const int vs_byte = 8 * (D == 64 ? l16 & 1 : (D == 96 && (l16 & 3) > 2 ? 2 : l16 & 3));

    // K of one block: eight key bytes per k-step and their scale, of token col (C = 16: and of 16 + col)
    constexpr int TT = N16 ? 2 : 1; // tiles of C tokens
    u32x2 kw[TT][KS];
    half_t ks[TT][KS];
    auto read_k = [&](const char* at) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
                const int tk = 16 * t + col;
                const char* const row = at + tk * D;
                const char* const sc = at + 64 * D + tk * (2 * GPT);
                const int sw = ring_swizzle<D>(tk);
                if constexpr (N16 && D == 96) {
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        kw[t][s] = *(const u32x2*)(row + 32 * s + 8 * kb);
                        ks[t][s] = *(const half_t*)(sc + 8 * s + 2 * kb);
                    }
                } else {
                    uint32_t sw32[KS / 2]; // C = 32: the lane's groups follow each other
                    if constexpr (!N16 && D == 128) *(u32x4*)sw32 = *(const u32x4*)(sc + 16 * kb);
                    if constexpr (!N16 && D == 64) *(u32x2*)sw32 = *(const u32x2*)(sc + 8 * kb);
#pragma unroll
                    for (int s = 0; s < KS; s += 2) {
                        const int chunk = N16 ? 2 * s + kb : KS / 2 * kb + (s >> 1);
                        const u32x4 w = *(const u32x4*)(row + 16 * (chunk ^ sw));
                        kw[t][s] = u32x2{w[0], w[1]};
                        kw[t][s + 1] = u32x2{w[2], w[3]};
                        const half2_t s2 = !N16 && D != 96 ? bitcast<half2_t>(sw32[s / 2]) : *(const half2_t*)(sc + 4 * chunk);
                        ks[t][s] = s2[0];
                        ks[t][s + 1] = s2[1];
                    }
                }
        }
    };

    // hands out this lane's results, four consecutive channels at a time
    auto for_channels = [&](auto&& use, const auto& o) {
        if constexpr (N16 && T == 1 && D != 64) {
            // A lane's results are 32 consecutive channels, 32 kb + ...; written as they are, the four lanes of a column would
            // touch four lines with every store.  The 4 x 4 pieces of four channels change places between those lanes instead
            // (64 q / 8 kv heads, 20 chunks of 2 query tokens over 1500-3000: 44.2 -> 41.4 us).
#pragma unroll
            for (int set = 0; set < SETS; ++set)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    u32x4 p[4]; // channels 32 kb + 16 half + 4 j + ...
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int x = 0; x < 4; ++x) p[j][x] = bitcast<uint32_t>(o[set * NE + 4 * (j & 1) + x][2 * half + (j >> 1)]);
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const u32x2 a02 = __builtin_amdgcn_permlane32_swap(p[0][x], p[2][x], false, false);
                        const u32x2 a13 = __builtin_amdgcn_permlane32_swap(p[1][x], p[3][x], false, false);
                        const u32x2 b01 = __builtin_amdgcn_permlane16_swap(a02[0], a13[0], false, false);
                        const u32x2 b23 = __builtin_amdgcn_permlane16_swap(a02[1], a13[1], false, false);
                        p[0][x] = b01[0];
                        p[1][x] = b01[1];
                        p[2][x] = b23[0];
                        p[3][x] = b23[1];
                    }
#pragma unroll
                    for (int k = 0; k < (D == 96 ? 3 : 4); ++k) { // head_dim 96: the rows beyond group 11 are lane 3's
                        const f32x4 v = bitcast<f32x4>(p[k]);
                        use(128 * set + 32 * k + 16 * half + 4 * kb, v[0], v[1], v[2], v[3]);
                    }
                }
        } else if constexpr (N16) { // product e of a set, result i <-> row 4 kb + i
#pragma unroll
            for (int set = 0; set < SETS; ++set)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 4 * kb + i;
                    if (D == 96 && r > 11) continue;
                    const int ch = D == 64 ? 8 * (r & 7) + 4 * (r >> 3) : 128 * set + 8 * r;
#pragma unroll
                    for (int e = 0; e < NE; e += 4) use(ch + e, o[set * NE + e][i], o[set * NE + e + 1][i], o[set * NE + e + 2][i], o[set * NE + e + 3][i]);
                }
        } else if constexpr (D == 64) { // result e <-> row 8 (e / 4) + 4 kb + e % 4
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int w = 0; w < 2; ++w) use(8 * (4 * kb + i) + 4 * w, o[0][8 * w + i], o[1][8 * w + i], o[0][8 * w + 4 + i], o[1][8 * w + 4 + i]);
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 8 * (e >> 2) + 4 * kb + (e & 3);
                if (D == 96 && (r & 15) > 11) continue;
                use(8 * (r & 15) + 4 * (r >> 4), o[0][e], o[1][e], o[2][e], o[3][e]);
            }
        }
    };

    bool k_read = false; // the next block's K bytes are in registers
    for (int slot = 0;;) { // pieces
        Piece run = cur; // this wave's blocks of the piece
        bool working = true;
        if (T > 1) {
            const int blocks = (cur.pe - cur.pa + kMfmaBlock - 1) / kMfmaBlock, each = (blocks + T - 1) / T;
            run.pa = cur.pa + wave * each * kMfmaBlock;
            if ((wave + 1) * each < blocks) run.pe = run.pa + each * kMfmaBlock;
            working = wave * each < blocks; // (wave-uniform)
            slot = 0;
            next_requested = false;
#pragma unroll
            for (int s = 0; s < KS; ++s) qf[s] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (working) {
                start(run);
                settle_queries();
            } else {
                rows_of(run);
            }
        } else {
            settle_queries();
        }
        const bool on_cur = on;
        const int64_t q_row_cur = q_row;
        // tokens this column attends: all of the sequence, or (causal chunk) those up to its own position
        const bool causal = a.seqstarts != nullptr && a.chunk_causal != 0;
        const int col_lim = causal ? cur.len - qlen + cpos + 1 : cur.len;
        const int first_cut = causal ? cur.len - qlen + 1 : cur.len; // the smallest limit of any column
        const half_t* mask_row = nullptr;
        if (a.attn_mask != nullptr) {
            const int h = kvh * G + (gq < G ? gq : 0);
            mask_row = (const half_t*)a.attn_mask + (int64_t)h * a.mask_stride_h + (int64_t)cur.b * a.mask_stride_s + cur.start;
        }

        typedef __attribute__((ext_vector_type(N16 ? 4 : 16))) float acc_t;
        acc_t o_acc[SETS * NE];
#pragma unroll
        for (int i = 0; i < SETS * NE; ++i)
#pragma unroll
            for (int e = 0; e < (N16 ? 4 : 16); ++e) o_acc[i][e] = 0.f;
        float m_run = kNegBig, l_run = 0.f;
        Piece next = cur;
        bool has_next = false;

        if (K_AHEAD && (T > 1 ? working : !k_read)) {
            if (next_requested) wait_vector_memory<NK + 2 * NK>();
            else wait_vector_memory<NK>();
            read_k(ring + slot * SLOT);
        }
        for (int pos = run.pa; working; pos += kMfmaBlock) {
            const bool last_block = pos + kMfmaBlock >= run.pe;
            const char* const at = ring + slot * SLOT;

            // ---- S^T = K Q^T ----
            if constexpr (!K_AHEAD) {
                if (L == 2 && next_requested) wait_vector_memory<NK + 2 * NK>();
                else wait_vector_memory<NK>();
                read_k(at);
            }
            acc_t s_acc[TT];
#pragma unroll
            for (int t = 0; t < TT; ++t) {
#pragma unroll
                for (int e = 0; e < (N16 ? 4 : 16); ++e) s_acc[t][e] = 0.f;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const half2_t sc = {ks[t][s], ks[t][s]};
                    const uint32_t f0 = kw[t][s][0] ^ kFlipSigns, f1 = kw[t][s][1] ^ kFlipSigns;
                    half2_t h0, h1, h2, h3, g0, g1, g2, g3;
                    dequantise(cvt_bytes01(f0), sc, h0, g0);
                    dequantise(cvt_bytes23(f0), sc, h1, g1);
                    dequantise(cvt_bytes01(f1), sc, h2, g2);
                    dequantise(cvt_bytes23(f1), sc, h3, g3);
                    const f16x8 ah = join(h0, h1, h2, h3), al = join(g0, g1, g2, g3);
                    if constexpr (N16) {
                        s_acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, qf[s], s_acc[t], 0, 0, 0);
                        s_acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, qf[s], s_acc[t], 0, 0, 0);
                    } else {
                        s_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, qf[s], s_acc[t], 0, 0, 0);
                        s_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, qf[s], s_acc[t], 0, 0, 0);
                    }
                }
            }
            if (T == 1 && last_block) {
                has_next = find_piece(cur.b + 1, next);
                if (has_next) {
                    rows_of(next);
                    request_queries();
                }
            }
            // (the query fragments of a following piece go first: they are needed before the rows requested here)
            requested = ahead_ok;
            if (requested) {
                wait_lds_reads();
                request(slot, false);
            }

            // ---- V bytes: on their way from LDS while the softmax runs (head_dim 256: a set of groups at a time, below) ----
            if (L == 2 && next_requested) {
                if (requested) wait_vector_memory<NK + 2 * NK>();
                else wait_vector_memory<2 * NK>();
            } else {
                if (requested) wait_vector_memory<NK>();
                else wait_vector_memory<0>();
            }
            constexpr int VW = NE > 4 ? 2 : 1; // words per token
            uint32_t vw[TV][VW];
            half2_t vs[TV / 2];
            auto read_v = [&](const int set) {
#pragma unroll
                for (int k = 0; k < TV; ++k) {
                    const int tk = v_token(k);
                    const int byte = 128 * set + v_byte;
                    const char* const p = at + 32 * D + tk * D + 16 * ((byte >> 4) ^ ring_swizzle<D>(tk)) + (byte & 15);
                    if constexpr (VW == 2) {
                        const u32x2 w = *(const u32x2*)p;
                        vw[k][0] = w[0];
                        vw[k][1] = w[1];
                    } else if constexpr (NE == 4) {
                        vw[k][0] = *(const uint32_t*)p;
                    } else {
                        vw[k][0] = *(const uint16_t*)p;
                    }
                }
#pragma unroll
                for (int k = 0; k < TV; k += 4) {
                    const int tk = v_token(k) + (l16 >> 2); // v_token(k) is a multiple of 4 plus k % 4 = 0
                    const char* const p = at + 72 * D + tk * (2 * GPT) + 32 * set + vs_byte;
                    const s16x4 s4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p);
                    vs[k / 2] = bitcast<half2_t>(__builtin_shufflevector(s4, s4, 0, 1));
                    vs[k / 2 + 1] = bitcast<half2_t>(__builtin_shufflevector(s4, s4, 2, 3));
                }
            };
            if (SETS == 1) read_v(0);

            // ---- online softmax per column; token of result e (of tile t): ----
            auto token_of = [&](int t, int e) { return pos + (N16 ? 16 * t + 4 * kb + e : 8 * (e >> 2) + 4 * kb + (e & 3)); };
            constexpr int NL = N16 ? 4 : 16;
            if (a.attn_mask != nullptr) {
#pragma unroll
                for (int t = 0; t < TT; ++t)
#pragma unroll
                    for (int e = 0; e < NL; ++e) {
                        const int tk = token_of(t, e);
                        s_acc[t][e] += (float)mask_row[tk < run.pe ? tk : run.pe - 1] * (kLog2e / sm_scale);
                    }
            }
            if (pos + kMfmaBlock > run.pe || pos + kMfmaBlock > first_cut) { // a piece's last block, or one that reaches a column's causal limit (wave-uniform)
                const int lim = col_lim < run.pe ? col_lim : run.pe;
#pragma unroll
                for (int t = 0; t < TT; ++t)
#pragma unroll
                    for (int e = 0; e < NL; ++e)
                        if (token_of(t, e) >= lim) s_acc[t][e] = -INFINITY;
            }
            // maximum of the raw dot products; the (positive) logit scale is applied to it afterwards
            float mx = kNegBig;
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int e = 0; e < NL; ++e) mx = fmaxf(mx, s_acc[t][e]);
            mx *= sm_scale;
            mx = across_lanes<N16>(mx, [](float x, float y) { return fmaxf(x, y); });
            const float m_new = fmaxf(m_run, mx);
            if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) { // wave-uniform and rare once a few blocks were seen
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int i = 0; i < SETS * NE; ++i)
#pragma unroll
                    for (int e = 0; e < NL; ++e) o_acc[i][e] *= alpha;
                m_run = m_new;
            }
            const float bias = kPShift - m_run;
            constexpr int PT = N16 ? 1 : 2; // k-steps of O^T
            f16x8 ph[PT], pl[PT];
            float lsum = 0.f;
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int e = 0; e < NL; e += 2) {
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[t][e], sm_scale, bias));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[t][e + 1], sm_scale, bias));
                    lsum += p0 + p1;
                    // both parts rounded to nearest: p within 2^-23 of itself (up to three times that, and always below it, when they are cut off)
                    const half2_t h = __builtin_convertvector(f32x2{p0, p1}, half2_t);
                    const half2_t l = __builtin_convertvector(f32x2{sub_half_lo(p0, h), sub_half_hi(p1, h)}, half2_t);
                    const int k = 4 * t + e; // C = 16: tile t's four results follow each other
                    ph[k >> 3][k & 7] = h.x;
                    ph[k >> 3][(k & 7) + 1] = h.y;
                    pl[k >> 3][k & 7] = l.x;
                    pl[k >> 3][(k & 7) + 1] = l.y;
                }
            l_run += lsum;

            // ---- O^T += V^T P^T ----
            auto request_v = [&]() {
                if (!requested) return;
                wait_lds_reads();
                request(slot, true);
                advance();
            };
            if (SETS == 1) request_v();
            if (K_AHEAD && next_requested) { // the next block's K, through LDS during the products
                if (requested) wait_vector_memory<NK + 2 * NK>();
                else wait_vector_memory<NK>();
                read_k(ring + (slot ^ 1) * SLOT);
                k_read = true;
            }
#pragma unroll
            for (int set = 0; set < SETS; ++set) {
                if (SETS > 1) {
                    read_v(set);
                    if (set + 1 == SETS) request_v();
                }
#pragma unroll
                for (int t = 0; t < PT; ++t)
#pragma unroll
                    for (int e = 0; e < NE; ++e) {
                        constexpr uint32_t kSel[4] = {0x0c040c00u, 0x0c050c01u, 0x0c060c02u, 0x0c070c03u}; // byte e & 3 of two words
                        half2_t h[4], l[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int k = 8 * t + 2 * i;
                            const half2_t x = pk_sub_1152(__builtin_amdgcn_perm(vw[k + 1][e >> 2], vw[k][e >> 2], kSel[e & 3]) ^ 0x64806480u);
                            dequantise(x, vs[k / 2], h[i], l[i]);
                        }
                        const f16x8 vh = join(h[0], h[1], h[2], h[3]), vl = join(l[0], l[1], l[2], l[3]);
                        acc_t& o = o_acc[set * NE + e];
                        if constexpr (N16) {
                            o = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph[t], o, 0, 0, 0);
                            o = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl[t], o, 0, 0, 0);
                            o = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[t], o, 0, 0, 0);
                        } else {
                            o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph[t], o, 0, 0, 0);
                            o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[t], o, 0, 0, 0);
                            o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[t], o, 0, 0, 0);
                        }
                    }
            }
            next_requested = L == 2 && requested;
            if (L == 2) slot ^= 1;
            if (last_block) break;
        }

        // ---- end of the piece ----
        const float l_tot = across_lanes<N16>(l_run, [](float x, float y) { return x + y; });
        const bool whole = cur.pa == 0 && cur.pe == cur.len;
        const int64_t piece = (int64_t)blockIdx.x + cur.b;
        const int h = kvh * G + gq; // the column among all columns: its slot in the pieces' workspace
        half_t* const op = (half_t*)a.output + (q_row_cur + cpos) * a.output_stride_s + (int64_t)(kvh * GR + cg) * D;
        float* const pp = a.partial_out + (piece * a.num_heads + h) * D;
        if constexpr (T == 1) {
            const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
            if (on_cur) {
                for_channels([&](int ch, float x0, float x1, float x2, float x3) {
                    if (whole) *(f16x4*)(op + ch) = f16x4{(half_t)(x0 * inv), (half_t)(x1 * inv), (half_t)(x2 * inv), (half_t)(x3 * inv)};
                    else *(f32x4*)(pp + ch) = f32x4{x0 * inv, x1 * inv, x2 * inv, x3 * inv};
                }, o_acc);
                if (!whole && kb == 0) {
                    a.partial_ml[(piece * a.num_heads + h) * 2 + 0] = m_run;
                    a.partial_ml[(piece * a.num_heads + h) * 2 + 1] = l_tot * 0x1p-14f; // p carries the factor 2^kPShift
                }
            }
        } else {
            // every wave's sums into its own ring (all its requests have been read), [column][channel], 16-byte pieces XORed
            // with the column so that the columns' stores spread over the banks; then (maximum, exp-sum) per column
            constexpr int ROW = D * 4, P4 = D / 4, SW = P4 % 32 == 0 ? 31 : (P4 % 16 == 0 ? 15 : 7);
            static_assert(C * ROW + C * 8 <= L * SLOT, "the sums fit the ring");
            wave_lds_handoff();
            for_channels([&](int ch, float x0, float x1, float x2, float x3) {
                *(f32x4*)(ring + col * ROW + 16 * ((ch >> 2) ^ (col & SW))) = f32x4{x0, x1, x2, x3};
            }, o_acc);
            if (kb == 0) *(float2*)(ring + C * ROW + 8 * col) = float2{m_run, l_tot};
            __syncthreads();
            // column c4 / P4, piece c4 % P4 of its row; the thread's own column only where the two agree
            for (int i = threadIdx.x; i < C * P4; i += T * kWave) {
                const int c = i / P4, q = i % P4;
                const int gc = pass * C + c, pc = a.seqstarts != nullptr ? gc / GR : 0;
                if (gc >= G || pc >= qlen) continue;
                float2 ml[T];
                float M = kNegBig, den = 0.f;
                f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    ml[t] = *(const float2*)(rings + t * (L * SLOT) + C * ROW + 8 * c);
                    M = fmaxf(M, ml[t].x);
                }
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const float w = __builtin_amdgcn_exp2f(ml[t].x - M);
                    den += ml[t].y * w;
                    v += *(const f32x4*)(rings + t * (L * SLOT) + c * ROW + 16 * (q ^ (c & SW))) * w;
                }
                v *= den > 0.f ? 1.f / den : 0.f;
                if (whole) {
                    half_t* const to = (half_t*)a.output + (q_row_cur + pc) * a.output_stride_s + (int64_t)(kvh * GR + gc - pc * GR) * D;
                    *(f16x4*)(to + 4 * q) = f16x4{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
                } else {
                    const int64_t slot_of = piece * a.num_heads + kvh * G + gc;
                    *(f32x4*)(a.partial_out + slot_of * D + 4 * q) = v;
                    if (q == 0) *(float2*)(a.partial_ml + slot_of * 2) = float2{M, den * 0x1p-14f}; // p carries the factor 2^kPShift
                }
            }
            has_next = find_piece(cur.b + 1, next);
            if (has_next) __syncthreads(); // the rings are requested into again
        }
        if (!has_next) break;
        cur = next;
    }
}


// The passes of a workgroup: blockIdx.z, or (chunks taken sequence by sequence) as many as the sequence's own rows need, so
// that no row depends on the caller's bound of them.
template <int C, int D, int NW, int T, bool SEQ>
__device__ __forceinline__ void decode_passes(const DecodeLaunch& a, char* const rings, const int wave)
{
    if constexpr (!SEQ) {
        decode_columns<C, D, NW, T, false>(a, rings, wave, blockIdx.z, (int)a.num_kv_repeats);
    } else {
        int columns = (int)a.num_kv_repeats;
        if (a.seqstarts != nullptr) {
            const const_i64_ptr seqstarts = as_constant(a.seqstarts);
            columns = (int)(seqstarts[blockIdx.x + 1] - seqstarts[blockIdx.x]) * a.chunk_q_heads;
        }
        for (int pass = blockIdx.z; pass * C < columns; pass += gridDim.z) {
            int pass_in = pass; // (nothing of a pass is computed ahead of the loop, where it would only hold registers)
            asm volatile("" : "+s"(pass_in));
            decode_columns<C, D, NW, T, true>(a, rings, wave, pass_in, columns);
            if (T > 1) __syncthreads(); // the rings are requested into again
        }
    }
}

} // namespace

template <int D, int NW, int T, bool SEQ>
__global__ __launch_bounds__(NW * T * kWave, 2) void decode_attention_mfma16_kernel(const DecodeLaunch a)
{
    __shared__ __attribute__((aligned(16))) char s_rings[NW * T * ring_slots(D) * ring_slot_bytes(D)];
    decode_passes<16, D, NW, T, SEQ>(a, s_rings, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

template <int D, int NW, int T>
__global__ __launch_bounds__(NW * T * kWave, 2) void decode_attention_mfma32_kernel(const DecodeLaunch a)
{
    __shared__ __attribute__((aligned(16))) char s_rings[NW * T * ring_slots(D) * ring_slot_bytes(D)];
    decode_passes<32, D, NW, T, true>(a, s_rings, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

template <int D, int NW, int T, bool SEQ>
static void launch_decode_columns_form(const DecodeLaunch& a, hipStream_t stream)
{
    const dim3 grid((unsigned)(SEQ ? a.decoding_batches : a.ranges), (unsigned)(a.num_kv_heads / NW), (unsigned)a.num_passes);
    const dim3 block(NW * T * kWave);
    if constexpr (SEQ && D != 256) {
        if (a.kernel == kDecodeKernelMfma32) {
            hipLaunchKernelGGL((decode_attention_mfma32_kernel<D, NW, T>), grid, block, 0, stream, a);
            return;
        }
    }
    hipLaunchKernelGGL((decode_attention_mfma16_kernel<D, NW, T, SEQ>), grid, block, 0, stream, a);
}

// (over ranges: head_dim 64 and 128, decode_select.cpp)
template <int D, int NW, int T>
static void launch_decode_columns_seq(const DecodeLaunch& a, hipStream_t stream)
{
    if (a.by_sequence) {
        launch_decode_columns_form<D, NW, T, true>(a, stream);
        return;
    }
    if constexpr (D == 64 || D == 128) launch_decode_columns_form<D, NW, T, false>(a, stream);
}

template <int D>
static void launch_decode_columns_d(const DecodeLaunch& a, hipStream_t stream)
{
    if (a.shared_pieces == 8) { // (whole sequences only)
        launch_decode_columns_form<D, 1, 8, true>(a, stream);
        return;
    }
    if (a.shared_pieces == 4) {
        launch_decode_columns_seq<D, 1, 4>(a, stream);
        return;
    }
    switch (a.kv_heads_per_group) { // a wave per kv head
    case 4: launch_decode_columns_seq<D, 4, 1>(a, stream); break;
    case 2: launch_decode_columns_seq<D, 2, 1>(a, stream); break;
    default: launch_decode_columns_seq<D, 1, 1>(a, stream); break;
    }
}

void launch_decode_columns(const DecodeLaunch& a, hipStream_t stream)
{
    switch (a.head_dim) {
    case 64: launch_decode_columns_d<64>(a, stream); break;
    case 96: launch_decode_columns_d<96>(a, stream); break;
    case 128: launch_decode_columns_d<128>(a, stream); break;
    default: launch_decode_columns_d<256>(a, stream); break;
    }
}

} // namespace pmxhip
