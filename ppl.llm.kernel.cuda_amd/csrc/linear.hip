// Output projection behind the attention: output(M, N) = input(M, K) * weight(N, K)^T + bias, fp16 in and out,
// fp32 accumulate -- the single-rank case of the reference's row_parallel_linear
// (src/ppl/kernel/llm/cuda/pmx/row_parallel_linear.cu:25-110: one cublasLt GEMM, then an all-reduce only when the
// communicator has more than one rank).
//
// Both operands are contiguous along K, the k dimension of the MFMA instructions for both of their inputs, so a fragment
// is 16 bytes of a row and nothing is ever transposed.  The kernels here move rows from memory straight into LDS
// (global_load_lds, 16 bytes per lane: no staging registers, so the depth of the pipeline costs LDS only) and differ in
// who shares what:
//   stream_linear_kernel  decode-sized M: a workgroup owns a small tile of the output over the whole of K, its four waves
//                         split K between them, each with a ring of its own and no barrier before the end
//   tile_linear_kernel    from a few hundred rows: a workgroup owns a large tile, its waves share every stage of a common ring
//   skinny_linear_kernel  rows that lie too far apart for the 32-bit row offsets of the other two, and a few long rows without workspace
// linear_choose() picks kernel, tile and number of k ranges from a cost per workgroup that was measured for each.
#include "device_common.h"
#include "launch_params.h"

#include <math.h>

namespace pmxhip {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kLinWaves = 8;
constexpr int kLinThreads = 64 * kLinWaves;
constexpr int kLinCols = 16;   // output columns per workgroup
constexpr int kLinRows = 128;  // input rows per workgroup
constexpr int kLinMB = kLinRows / 16;
constexpr int kLinKStep = 32;
constexpr int kWDepth = 4, kADepth = 2;

// XCD-aware numbering: workgroups are dealt to the eight XCDs in turn; XCD x takes a contiguous piece of the tiles, so
// that tiles which share rows of an operand share an L2 cache
__device__ __forceinline__ int xcd_tile(int total)
{
    const int q = total >> 3, r = total & 7, x = blockIdx.x & 7, p = blockIdx.x >> 3;
    return x * q + (x < r ? x : r) + p;
}

// acc + the four outputs that follow it, as halves with the bias added
__device__ __forceinline__ f16x4 finish4(const f32x4 v, const void* bias, int64_t n)
{
    f32x4 s = v;
    if (bias) {
        const f16x4 b = *(const f16x4*)((const half_t*)bias + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += (float)b[e];
    }
    f16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (half_t)s[e];
    return o;
}

} // namespace

// ---- any row stride: a workgroup owns 16 output columns and up to 128 rows, fragments straight from memory --------------
// Eight waves take the 32-wide k steps in turn (adjacent 64-byte pieces of a weight row), keep the weight requests four
// steps ahead and the input requests two, and add their partial tiles through LDS at the end, in a fixed order.
// It runs where the rows of an operand lie 2^23 halves or more apart, and on few long rows without workspace (linear_choose); with ordinary strides the input that every
// workgroup re-reads (M * K * 2 bytes) makes it 42 us on (128, 4096, 4096), where stream_linear_kernel takes 11.6.
__global__ __launch_bounds__(kLinThreads) void skinny_linear_kernel(const LinearLaunch a)
{
    __shared__ __attribute__((aligned(16))) float s_part[kLinWaves][kLinRows][kLinCols]; // 64 KB
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15;  // weight row (output column) / input row within a 16-row block
    const int kq = lane >> 4;   // which 8 of the 32 k of a step
    const int64_t n0 = (int64_t)blockIdx.x * kLinCols;
    const int64_t m0 = (int64_t)blockIdx.y * kLinRows;
    const int ksteps = (int)(a.k / kLinKStep);
    const int my_steps = (ksteps - wave + kLinWaves - 1) / kLinWaves; // steps wave, wave + 8, ...

    const half_t* wp = (const half_t*)a.weight + (n0 + r16) * a.weight_stride + 8 * kq;
    const half_t* ip[kLinMB];
#pragma unroll
    for (int mb = 0; mb < kLinMB; ++mb) {
        int64_t m = m0 + 16 * mb + r16;
        if (m > a.m - 1) m = a.m - 1; // rows beyond the batch re-read its last row; their results are not stored
        ip[mb] = (const half_t*)a.input + m * a.input_stride + 8 * kq;
    }

    f32x4 acc[kLinMB];
#pragma unroll
    for (int mb = 0; mb < kLinMB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};

    f16x8 wf[kWDepth];
    f16x8 af[kADepth][kLinMB];
    auto k_of = [&](int i) { return (int64_t)(i * kLinWaves + wave) * kLinKStep; };
    auto load_w = [&](int i, f16x8& dst) {
        const int ic = i < my_steps ? i : my_steps - 1; // past the end: a harmless repeat of the last step
        dst = __builtin_nontemporal_load((const f16x8*)(wp + k_of(ic))); // every weight byte is used once
    };
    auto load_a = [&](int i, f16x8* dst) {
        const int ic = i < my_steps ? i : my_steps - 1;
#pragma unroll
        for (int mb = 0; mb < kLinMB; ++mb) dst[mb] = *(const f16x8*)(ip[mb] + k_of(ic));
    };
    if (my_steps > 0) {
#pragma unroll
        for (int d = 0; d < kWDepth; ++d) load_w(d, wf[d]);
#pragma unroll
        for (int d = 0; d < kADepth; ++d) load_a(d, af[d]);
        // the rings are indexed with compile-time constants: the loop runs over groups of kWDepth steps
        for (int i0 = 0; i0 < my_steps; i0 += kWDepth) {
#pragma unroll
            for (int d = 0; d < kWDepth; ++d) {
                const int i = i0 + d;
                if (i < my_steps) {
                    const f16x8 w = wf[d];
                    f16x8 cur[kLinMB];
#pragma unroll
                    for (int mb = 0; mb < kLinMB; ++mb) cur[mb] = af[d % kADepth][mb];
                    load_w(i + kWDepth, wf[d]);
                    load_a(i + kADepth, af[d % kADepth]);
#pragma unroll
                    for (int mb = 0; mb < kLinMB; ++mb)
                        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, cur[mb], acc[mb], 0, 0, 0);
                }
            }
        }
    }

    // accumulator element e of block mb: row 16 mb + r16, column 4 kq + e
#pragma unroll
    for (int mb = 0; mb < kLinMB; ++mb) *(f32x4*)&s_part[wave][16 * mb + r16][4 * kq] = acc[mb];
    __syncthreads();
    // one thread per (row, four columns): the eight partial tiles are added in wave order
    {
        const int row = tid >> 2, c4 = (tid & 3) * 4;
        f32x4 sum = *(const f32x4*)&s_part[0][row][c4];
#pragma unroll
        for (int w = 1; w < kLinWaves; ++w) sum += *(const f32x4*)&s_part[w][row][c4];
        if (a.bias) {
            const f16x4 b = *(const f16x4*)((const half_t*)a.bias + n0 + c4);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += (float)b[e];
        }
        if (m0 + row < a.m) {
            f16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (half_t)sum[e];
            *(f16x4*)((half_t*)a.output + (m0 + row) * a.output_stride + n0 + c4) = o;
        }
    }
}

// ---- decode-sized M ------------------------------------------------------------------------------------------------
// What bounds it: a CU fills its LDS at about 100 GB/s (measured over tiles from 16 x 16 to 64 x 64: 4 us and then 10 us per
// megabyte of rows of either operand), the chip streams weights at 5.7 TB/s (8192 x 8192, one row: 23.5 us).  So the tile is
// the one nearest to square that still gives every CU a workgroup -- (TN + TM) * K * 2 bytes are what a CU has to pull --
// and K is not split over workgroups where that can be avoided: the float32 partial tiles of a split and the launch that
// adds them cost more than the wider tile saves ((128, 4096, 4096): 11.6 us with 32 x 64 tiles and one k range, 15.5 with
// 64 x 128 and four).
// Each of the four waves takes every fourth 64-k piece (128 bytes, one whole line, of every row), streams it through its
// own ring of NS stages and waits for nothing but its own requests.  LDS rows are 128 bytes without padding (the DMA
// writes lane i at 16 i); the 16-byte chunk c of row r lies in slot c ^ ((r >> 1) & 7), so that the fragment reads of
// sixteen rows cover all 64 banks.  The four partial tiles meet in LDS and are added in wave order.
// NT: the weights carry the non-temporal hint (one row tile, so every weight byte is used once).  It pays where the weights come
// from memory, and costs where they wait in the 256 MB memory-side cache.  One row, microseconds with the hint / without,
// calls that take 600 MB of matrices in turn (a model's layers) and calls on one matrix: 134 MB 25.2 / 28.9 and 23.5 / 22.0,
// 117 MB 22.1 / 25.3 and 20.8 / 19.3, 52 MB 14.0 / 14.5 and 14.1 / 10.6, 50 MB 12.2 / 12.9 and 11.2 / 10.3, 33 MB 7.7 / 7.7 and
// 5.5 / 5.2, with 32 rows 13.2 / 12.2 and 10.2 / 9.1: on from 64 MB.
// Against the form with fragments loaded into registers that this replaces: (1, 4096, 4096) 10.3 -> 7.0 us, (16, 4096,
// 4096) 10.9 -> 7.9, (128, 4096, 4096) 22.2 -> 11.6, (32, 8192, 8192) 36.7 -> 24.5, (32, 5120, 5120) 25.6 -> 11.0.
constexpr int kStreamWaves = 4;

template <int TN, int TM, int NS, bool NT>
__global__ __launch_bounds__(64 * kStreamWaves) void stream_linear_kernel(const LinearLaunch a, const int splits,
                                                                          float* __restrict__ partial)
{
    constexpr int W = kStreamWaves;
    constexpr bool BIG = TN >= 32 && TM >= 32;   // 32x32x16 products, else 16x16x32
    constexpr int FR = BIG ? 32 : 16;
    constexpr int FN = TN / FR, FM = TM / FR;
    constexpr int KS = BIG ? 4 : 2;              // k steps of a 64-k piece
    constexpr int AE = BIG ? 16 : 4;
    constexpr int LW = TN / 8, LX = TM / 8;      // requests of a stage (8 rows each)
    constexpr int STAGE = (TN + TM) * 128;
    constexpr int RS = TN + 4;                   // floats per row of a partial tile
    constexpr int RING = W * NS * STAGE, RED = W * TM * RS * 4;
    __shared__ __attribute__((aligned(128))) char smem[RING > RED ? RING : RED];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // row tiles innermost: the tiles that share weight rows run side by side on one XCD
    const int nt = (int)((a.n + TN - 1) / TN), mt = (int)((a.m + TM - 1) / TM);
    int t = xcd_tile(nt * mt * splits);
    const int64_t m0 = (int64_t)(t % mt) * TM;
    t /= mt;
    const int split = t / nt;
    const int64_t n0 = (int64_t)(t % nt) * TN;
    const int pieces_all = (int)(a.k >> 6);
    const int per = (pieces_all + splits - 1) / splits; // the host keeps every range non-empty
    const int pieces = pieces_all - split * per < per ? pieces_all - split * per : per;
    const int mine = (pieces - wave + W - 1) / W;       // pieces wave, wave + 4, ... of the range

    // request j of an operand: rows 8 j .. 8 j + 7, lane i takes slot i % 8 of row i / 8.  Rows beyond the operand re-read
    // its last row; their results are not stored.
    const char* const src_w = (const char*)a.weight + (n0 * a.weight_stride + (int64_t)split * per * 64) * 2;
    const char* const src_x = (const char*)a.input + (m0 * a.input_stride + (int64_t)split * per * 64) * 2;
    uint32_t vw[LW], vx[LX];
#pragma unroll
    for (int j = 0; j < LW; ++j) {
        const int r = 8 * j + (lane >> 3);
        const int64_t row = n0 + r < a.n ? r : a.n - 1 - n0;
        vw[j] = (uint32_t)(row * a.weight_stride * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int j = 0; j < LX; ++j) {
        const int r = 8 * j + (lane >> 3);
        const int64_t row = m0 + r < a.m ? r : a.m - 1 - m0;
        vx[j] = (uint32_t)(row * a.input_stride * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    const uint32_t ring = wave * NS * STAGE;
    const uint32_t lds0 = lds_address(smem) + ring;
    // stage s into the ring at `buf`; past the end: a harmless repeat of the last piece, so that the wait counts stay the same
    auto issue = [&](int s, uint32_t buf) {
        int p = wave + W * s;
        p = p < pieces ? p : pieces - 1;
        const int64_t k = (int64_t)p * 128;
#pragma unroll
        for (int j = 0; j < LW; ++j) load_to_lds16<NT>(lds0 + buf + j * 1024, vw[j], src_w + k);
#pragma unroll
        for (int j = 0; j < LX; ++j) load_to_lds16<false>(lds0 + buf + TN * 128 + j * 1024, vx[j], src_x + k);
    };

    const int rf = lane & (FR - 1), hq = lane / FR;
    typedef float acc_t __attribute__((ext_vector_type(AE)));
    acc_t acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int e = 0; e < AE; ++e) acc[i][j][e] = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) issue(s, s * STAGE);
    uint32_t cur = 0;
    for (int i = 0; i < mine; ++i) {
        wait_vector_memory<(NS - 1) * (LW + LX)>();
        f16x8 fw[KS][FN], fx[KS][FM];
        const char* const base = smem + ring + cur + rf * 128;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int slot = (ks * (BIG ? 2 : 4) + hq) ^ ((rf >> 1) & 7);
#pragma unroll
            for (int f = 0; f < FN; ++f) fw[ks][f] = *(const f16x8*)(base + f * FR * 128 + (slot << 4));
#pragma unroll
            for (int f = 0; f < FM; ++f) fx[ks][f] = *(const f16x8*)(base + TN * 128 + f * FR * 128 + (slot << 4));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the stage is in registers: its slot may be refilled
        issue(i + NS, cur);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int f = 0; f < FN; ++f)
#pragma unroll
                for (int g = 0; g < FM; ++g) {
                    if constexpr (BIG) acc[f][g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fw[ks][f], fx[ks][g], acc[f][g], 0, 0, 0);
                    else acc[f][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[ks][f], fx[ks][g], acc[f][g], 0, 0, 0);
                }
        __builtin_amdgcn_sched_barrier(0);
        cur = cur + STAGE == NS * STAGE ? 0 : cur + STAGE;
    }
    wait_and_meet<0>(); // the rings are idle: their space takes the partial tiles, [wave][row][column]
    float* const red = (float*)smem;
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int g = 0; g < FM; ++g)
#pragma unroll
            for (int r = 0; r < AE / 4; ++r) {
                const int m = g * FR + rf, n = f * FR + 8 * r + 4 * hq;
                *(f32x4*)&red[(wave * TM + m) * RS + n] =
                    f32x4{acc[f][g][4 * r], acc[f][g][4 * r + 1], acc[f][g][4 * r + 2], acc[f][g][4 * r + 3]};
            }
    __syncthreads();
    for (int i = threadIdx.x; i < TM * TN / 4; i += 64 * W) {
        const int m = i / (TN / 4), n = (i % (TN / 4)) * 4;
        if (m0 + m >= a.m || n0 + n >= a.n) continue;
        f32x4 sum = *(const f32x4*)&red[m * RS + n];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += *(const f32x4*)&red[(w * TM + m) * RS + n];
        if (splits > 1) *(f32x4*)(partial + ((int64_t)split * a.m + m0 + m) * a.n + n0 + n) = sum;
        else *(f16x4*)((half_t*)a.output + (m0 + m) * a.output_stride + n0 + n) = finish4(sum, a.bias, n0 + n);
    }
}

// ---- from a few hundred rows: a compute-bound GEMM -------------------------------------------------------------------------
// A workgroup of WN x WM waves owns TN output columns x TM rows and walks K in stages of 32 k; a stage (64 bytes of every
// row) is moved by all waves together, the ring holds NS of them.  Per stage a wave has two k steps, and their fragments
// are read one step ahead: the second step's while the first multiplies, and -- behind the stage's one barrier, which says
// that the next stage has landed and that this one may be refilled -- the next stage's first while the second multiplies,
// so neither the LDS reads nor the barrier stand between products.  Requests are NS - 1 stages ahead.
// LDS rows are 64 bytes: chunk c of row r lies in slot c ^ ((r >> 2) & 3) (sixteen rows cover all banks).
// With 256 x 256 tiles and eight waves a wave has 4 x 2 tiles of 32 x 32: 12 fragment reads per 16 products.
// (4000, 4096, 4096), 256 tiles for 256 CUs, 122 us = 1097 TFLOP/s, the same with 3, 4 or 5 stages, either wave shape and with
// or without raised wave priority; 8192 in all three 1170 (a large library product reaches 1150-1180 here).  (11104, 4096, 4096),
// 704 tiles in three rounds of 256: 355-370 us by box = 1010-1050 TFLOP/s; the weight-streaming kernel that took these sizes before:
// 1067.  Counters of that call: the matrix pipes are busy for 58 % of the shader cycles (63 % of those in which tiles run), at a
// clock that falls to 1.75 GHz under them; waves stand at a wait or barrier for 31 % of their time.
template <int TN, int TM, int WN, int WM, int NS>
__global__ __launch_bounds__(64 * WN * WM, 2) void tile_linear_kernel(const LinearLaunch a, const int splits, float* __restrict__ partial)
{
    constexpr int WAVES = WN * WM;
    constexpr int FN = TN / WN / 32, FM = TM / WM / 32;
    constexpr int STAGE = (TN + TM) * 64;
    constexpr int LI = (TN + TM) / 16 / WAVES; // requests per wave and stage, 16 rows each
    static_assert(LI * WAVES * 16 == TN + TM, "every wave makes the same number of requests");
    constexpr int EP = TN / WN + 8;            // halves per row of the epilogue's staging area
    constexpr int RING = NS * STAGE, EPB = WAVES * 32 * EP * 2;
    constexpr int kGroupM = 8;                 // row tiles that are walked together through the column tiles
    __shared__ __attribute__((aligned(128))) char smem[RING > EPB ? RING : EPB];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    const int wn = wave % WN, wm = wave / WN;

    const int nt = (int)((a.n + TN - 1) / TN), mt = (int)((a.m + TM - 1) / TM);
    int t = xcd_tile(nt * mt * splits);
    const int split = t / (nt * mt);
    t -= split * (nt * mt);
    const int grp = t / (kGroupM * nt);
    const int gm = mt - grp * kGroupM < kGroupM ? mt - grp * kGroupM : kGroupM;
    t -= grp * kGroupM * nt;
    const int64_t m0 = (int64_t)(grp * kGroupM + t % gm) * TM, n0 = (int64_t)(t / gm) * TN;
    const int steps_all = (int)(a.k >> 5);
    const int per = (steps_all + splits - 1) / splits; // the host keeps every range non-empty
    const int stages = steps_all - split * per < per ? steps_all - split * per : per;

    // request q: rows 16 q .. of the stage, weight rows first; lane i takes slot i % 4 of row i / 4.  Rows beyond an
    // operand re-read its last row; their results are not stored.
    const char* const src_w = (const char*)a.weight + (n0 * a.weight_stride + (int64_t)split * per * 32) * 2;
    const char* const src_x = (const char*)a.input + (m0 * a.input_stride + (int64_t)split * per * 32) * 2;
    uint32_t voff[LI];
#pragma unroll
    for (int j = 0; j < LI; ++j) {
        const int q = wave * LI + j;
        const bool is_w = q < TN / 16;
        int64_t r = (is_w ? q : q - TN / 16) * 16 + (lane >> 2);
        const int64_t last = is_w ? a.n - 1 - n0 : a.m - 1 - m0;
        if (r > last) r = last;
        voff[j] = (uint32_t)(r * (is_w ? a.weight_stride : a.input_stride) * 2) + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
    }
    const uint32_t lds0 = lds_address(smem);
    auto issue = [&](int s, uint32_t buf) {
        const int64_t k = (int64_t)(s < stages ? s : stages - 1) * 64; // past the end: a harmless repeat
#pragma unroll
        for (int j = 0; j < LI; ++j) {
            const int q = wave * LI + j;
            load_to_lds16<false>(lds0 + buf + q * 1024, voff[j], (q < TN / 16 ? src_w : src_x) + k);
        }
    };
    const uint32_t fo0 = l32 * 64 + ((h ^ ((l32 >> 2) & 3)) << 4);       // first k step of a stage
    const uint32_t fo1 = l32 * 64 + (((2 + h) ^ ((l32 >> 2) & 3)) << 4); // second
    const uint32_t wbase = wn * (TN / WN) * 64, xbase = TN * 64 + wm * (TM / WM) * 64;
    struct Fragments {
        f16x8 w[FN], x[FM];
    };
    auto read = [&](Fragments& f, uint32_t buf, uint32_t fo) {
#pragma unroll
        for (int i = 0; i < FN; ++i) f.w[i] = *(const f16x8*)(smem + buf + wbase + fo + i * 2048);
#pragma unroll
        for (int i = 0; i < FM; ++i) f.x[i] = *(const f16x8*)(smem + buf + xbase + fo + i * 2048);
    };
    f32x16 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    auto products = [&](const Fragments& f) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[i], f.x[j], acc[i][j], 0, 0, 0);
    };

    Fragments f0, f1;
#pragma unroll
    for (int s = 0; s < NS; ++s) issue(s, s * STAGE);
    wait_and_meet<(NS - 1) * LI>();
    read(f0, 0, fo0);
    uint32_t cur = 0;
    for (int i = 0; i < stages; ++i) {
        const uint32_t nxt = cur + STAGE == NS * STAGE ? 0 : cur + STAGE;
        read(f1, cur, fo1);
        __builtin_amdgcn_sched_barrier(0);
        products(f0);
        __builtin_amdgcn_sched_barrier(0);
        wait_and_meet<(NS - 2) * LI>(); // stage i + 1 has landed; every wave has stage i in registers
        issue(i + NS, cur);
        read(f0, nxt, fo0);
        __builtin_amdgcn_sched_barrier(0);
        products(f1);
        __builtin_amdgcn_sched_barrier(0);
        cur = nxt;
    }
    wait_and_meet<0>();

    // element 4 r + e of tile (i, j): row 32 j + l32, column 32 i + 8 r + 4 h + e of the wave's part
    const int64_t wn0 = n0 + wn * (TN / WN), wm0 = m0 + wm * (TM / WM);
    auto quad = [&](int i, int j, int r) {
        return f32x4{acc[i][j][4 * r], acc[i][j][4 * r + 1], acc[i][j][4 * r + 2], acc[i][j][4 * r + 3]};
    };
    if (splits > 1) {
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            const int64_t row = wm0 + 32 * j + l32;
            if (row >= a.m) continue;
            float* const p = partial + ((int64_t)split * a.m + row) * a.n + wn0 + 4 * h;
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (wn0 + 32 * i + 8 * r < a.n) *(f32x4*)(p + 32 * i + 8 * r) = quad(i, j, r);
        }
        return;
    }
    // Whole rows leave the workgroup: a lane holds 8-byte pieces of one row, so the wave turns 32 rows at a time round in its
    // own part of the idle ring and stores 16 bytes per lane (8 where output rows are aligned to 8 bytes only).
    half_t* const ep = (half_t*)smem + wave * 32 * EP;
    const bool wide_rows = ((uintptr_t)a.output & 15u) == 0 && (a.output_stride & 7) == 0;
    constexpr int CH = TN / WN / 8, RPI = 64 / CH; // 16-byte pieces per row, rows per store instruction
#pragma unroll
    for (int j = 0; j < FM; ++j) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = 32 * i + 8 * r + 4 * h;
                *(f16x4*)(ep + l32 * EP + c) = finish4(quad(i, j, r), wn0 + c < a.n ? a.bias : nullptr, wn0 + c);
            }
        wave_lds_handoff();
#pragma unroll
        for (int r0 = 0; r0 < 32; r0 += RPI) {
            const int row = r0 + lane / CH, piece = lane % CH;
            const u32x4 v = *(const u32x4*)(ep + row * EP + 8 * piece);
            const int64_t m = wm0 + 32 * j + row, n = wn0 + 8 * piece;
            if (m < a.m && n < a.n) {
                half_t* const dst = (half_t*)a.output + m * a.output_stride + n;
                if (wide_rows) {
                    *(u32x4*)dst = v;
                } else {
                    *(u32x2*)dst = u32x2{v[0], v[1]};
                    *(u32x2*)(dst + 4) = u32x2{v[2], v[3]};
                }
            }
        }
        wave_lds_handoff();
    }
}

// output = half(sum over the k ranges of the partial tiles, in range order, + bias); four columns per thread
__global__ __launch_bounds__(256) void linear_reduce_kernel(const LinearLaunch a, const int splits, const float* __restrict__ partial)
{
    const int64_t quads = a.n >> 2;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.m * quads) return;
    const int64_t row = i / quads, c4 = (i - row * quads) * 4;
    f32x4 sum = *(const f32x4*)(partial + row * a.n + c4);
    for (int s = 1; s < splits; ++s) sum += *(const f32x4*)(partial + ((int64_t)s * a.m + row) * a.n + c4);
    if (a.bias) {
        const f16x4 b = *(const f16x4*)((const half_t*)a.bias + c4);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += (float)b[e];
    }
    f16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (half_t)sum[e];
    *(f16x4*)((half_t*)a.output + row * a.output_stride + c4) = o;
}

// ---- which kernel, which tile, how many k ranges ------------------------------------------------------------------------
// A round of workgroups over the CUs takes a start (prologue and epilogue) plus its k length times a cost per k; a split adds
// the partial tiles' way through memory and a second launch (4 us + 8 bytes per element and range at 5.5 TB/s); no call
// beats its weights at 5.7 TB/s.  The constants are a fit to 1800 timings (nine tiles x 1, 2 and 4 ranges x M = 1 .. 6000 on
// seven weight shapes from 2048 x 2048 to 4096 x 14336, repeated calls on one matrix, which the memory-side cache held): the tile
// that the estimate picks takes 1.01 times what the best one takes in the mean, 1.15 at worst.
// More than one k range costs the caller a workspace.  Up to 32 MiB of partial tiles are taken for any gain in the estimate; more
// have to be worth it by 5 %, and they take at most 256 MiB, what the memory-side cache holds between the launch that writes
// them and the one that adds them.  (Without these bounds prompts asked for up to 700 MB, (3472, 14336, 14336) for 398 MB of
// them at an estimate of 1360.2 against 1360.6 us.)  Measured with the split against without, estimates less than 5 % apart:
// (2187, 4096, 14336) 143 MB 358 against 298 us, (343, 8192, 8192) 45 MB 79 against 68, (925, 5120, 5120) 38 MB 76 against 73; below 32 MiB it goes either way: (33, 8192, 8192) 24.8 against 28.5, (300, 4096, 14336) 58.4 against 63.5,
// (91, 8192, 8192) 36.5 against 27.7.
namespace {
constexpr float kLinearSplitGain = 0.05f;
constexpr int64_t kLinearSplitFreeBytes = (int64_t)32 << 20, kLinearSplitBytes = (int64_t)256 << 20;
struct LinearTile {
    LinearKernel kernel;
    int tn, tm;
    float start_us, ns_per_k; // of a round of workgroups
};
constexpr LinearTile kLinearTiles[] = {
    {kLinStream, 16, 16, 0.7f, 0.88f}, {kLinStream, 32, 32, 1.5f, 1.7f}, {kLinStream, 32, 64, 1.4f, 2.45f},
    {kLinStream, 64, 64, 2.4f, 3.3f},  {kLinTile, 64, 64, 0.f, 4.4f},    {kLinTile, 128, 64, 0.4f, 6.9f},
    {kLinTile, 128, 128, 1.1f, 9.3f},  {kLinTile, 256, 128, 1.8f, 16.5f}, {kLinTile, 256, 256, 5.7f, 23.2f},
};
constexpr int kLinearTileCount = (int)(sizeof(kLinearTiles) / sizeof(kLinearTiles[0]));
// rows of a tile are addressed as a 64-bit base plus a 32-bit byte offset: up to 256 rows of less than 2^23 halves
constexpr int64_t kLinearMaxStride = (int64_t)1 << 23;

struct LinearChoice {
    int tile = -1; // index into kLinearTiles
    int splits = 1;
    float us = 0.f;
};

LinearChoice linear_choose(int64_t m, int64_t n, int64_t k, int compute_units, int64_t workspace_bytes)
{
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    if (workspace_bytes > kLinearSplitBytes) workspace_bytes = kLinearSplitBytes;
    LinearChoice one, split; // the best of one k range or a small workspace; the best of the others
    const float stream_us = 2.f + (float)n * (float)k * 2.f / 5.7e6f;
    for (int i = 0; i < kLinearTileCount; ++i) {
        const LinearTile& c = kLinearTiles[i];
        const int64_t unit = c.kernel == kLinStream ? 64 : 32; // k of a pipeline stage
        if (k % unit != 0) continue;
        const int64_t tiles = ((n + c.tn - 1) / c.tn) * ((m + c.tm - 1) / c.tm);
        if (tiles > (1 << 20)) continue; // a launch has fewer than 2^32 threads
        for (int s = 1; s <= 4; s *= 2) {
            if (s > 1 && (workspace_bytes < s * m * n * (int64_t)sizeof(float) || k / unit < 8 * s)) break;
            const int64_t per = (k / unit + s - 1) / s;
            if ((s - 1) * per >= k / unit) break; // every range has at least one stage
            const int64_t rounds = (tiles * s + cus - 1) / cus;
            float us = (float)rounds * (c.start_us + (float)(per * unit) * c.ns_per_k * 1e-3f);
            if (s > 1) us += 4.f + (float)s * (float)m * (float)n * 8.f / 5.5e6f;
            us = fmaxf(us, stream_us) + 0.1f * fminf(us, stream_us); // what overlaps the stream still shows a little
            const bool large = s > 1 && s * m * n * (int64_t)sizeof(float) > kLinearSplitFreeBytes;
            LinearChoice& best = large ? split : one;
            if (best.tile < 0 || us < best.us) {
                best.tile = i;
                best.splits = s;
                best.us = us;
            }
        }
    }
    const LinearChoice best = split.tile >= 0 && split.us < one.us * (1.f - kLinearSplitGain) ? split : one;
    // Long rows of an odd number of 32 k have no tile of the streaming kernel; where a caller without workspace leaves a few of the large
    // tiles to walk them alone, the 16-column form has more workgroups: (1, 2064, 4128) 16.3 against 17.3 us, (8, 512, 8224) 25.9 against
    // 30.7, (16, 2560, 14368) 49.1 against 51.7.  With 32 rows, 3072 columns or 2080 k it is level or behind.
    if (best.splits == 1 && k % 64 != 0 && k >= 4096 && m <= 16 && n / kLinCols * 8 <= 5 * cus) return LinearChoice();
    return best;
}
} // namespace

LinearPlan linear_plan(int64_t m, int64_t n, int64_t k, int compute_units, int64_t workspace_bytes)
{
    LinearPlan plan;
    if (m <= 0 || n <= 0 || k <= 0) return plan;
    const LinearChoice c = linear_choose(m, n, k, compute_units, workspace_bytes);
    if (c.tile < 0) return plan;
    plan.kernel = kLinearTiles[c.tile].kernel;
    plan.tile_n = kLinearTiles[c.tile].tn;
    plan.tile_m = kLinearTiles[c.tile].tm;
    plan.splits = c.splits;
    if (c.splits > 1) plan.workspace_bytes = (int64_t)c.splits * m * n * (int64_t)sizeof(float);
    return plan;
}

int launch_linear(const LinearLaunch& a, int compute_units, void* workspace, int64_t workspace_bytes, hipStream_t stream)
{
    if (a.m <= 0 || a.n <= 0) return kLaunchOk;
    if (a.n % kLinCols != 0 || a.k % kLinKStep != 0 || a.k <= 0) return kLaunchNoKernel;
    // as many k ranges as the workspace holds partial tiles for; none: one k range
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15u)) workspace_bytes = 0;
    const LinearChoice plan = linear_choose(a.m, a.n, a.k, compute_units, workspace_bytes);
    if (plan.tile < 0 || a.weight_stride >= kLinearMaxStride || a.input_stride >= kLinearMaxStride) {
        const int64_t mblocks = (a.m + kLinRows - 1) / kLinRows;
        if (a.n / kLinCols > 0x7fffffff || mblocks > 65535) return kLaunchNoKernel;
        hipLaunchKernelGGL(skinny_linear_kernel, dim3((unsigned)(a.n / kLinCols), (unsigned)mblocks), dim3(kLinThreads), 0, stream, a);
        return kLaunchOk;
    }
    const LinearTile& c = kLinearTiles[plan.tile];
    const int splits = plan.splits;
    float* const part = (float*)workspace;
    const dim3 grid((unsigned)(((a.n + c.tn - 1) / c.tn) * ((a.m + c.tm - 1) / c.tm) * splits));
    // one row tile: every weight byte is used once; from 64 MB on the hint pays more than it costs (stream_linear_kernel)
    const bool nt = a.m <= c.tm && a.n * a.k >= ((int64_t)32 << 20);
#define PMX_STREAM(TN, TM, NS) \
    do { \
        if (nt) hipLaunchKernelGGL((stream_linear_kernel<TN, TM, NS, true>), grid, dim3(64 * kStreamWaves), 0, stream, a, splits, part); \
        else hipLaunchKernelGGL((stream_linear_kernel<TN, TM, NS, false>), grid, dim3(64 * kStreamWaves), 0, stream, a, splits, part); \
    } while (0)
#define PMX_TILE(TN, TM, WN, WM, NS) \
    hipLaunchKernelGGL((tile_linear_kernel<TN, TM, WN, WM, NS>), grid, dim3(64 * WN * WM), 0, stream, a, splits, part)
    switch (plan.tile) {
    case 0: PMX_STREAM(16, 16, 4); break;
    case 1: PMX_STREAM(32, 32, 3); break;
    case 2: PMX_STREAM(32, 64, 2); break;
    case 3: PMX_STREAM(64, 64, 2); break;
    case 4: PMX_TILE(64, 64, 2, 2, 8); break;
    case 5: PMX_TILE(128, 64, 2, 2, 6); break;
    case 6: PMX_TILE(128, 128, 4, 2, 4); break;
    case 7: PMX_TILE(256, 128, 4, 2, 4); break;
    default: PMX_TILE(256, 256, 2, 4, 4); break;
    }
#undef PMX_STREAM
#undef PMX_TILE
    if (splits > 1) {
        const int64_t threads = a.m * (a.n >> 2);
        hipLaunchKernelGGL(linear_reduce_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, a, splits,
                           (const float*)workspace);
    }
    return kLaunchOk;
}

} // namespace pmxhip
