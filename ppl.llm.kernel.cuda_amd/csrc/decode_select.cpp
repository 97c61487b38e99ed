// Which kernel runs the token ranges of a decode step, and the grouping of heads and tokens it implies.
// Host only.  The plan (pmxhip_decode_plan_make*) and the launch (pmxhip_decode_attention*) both come here, so
// the unit of the range cuts that the token-range kernel uses is by construction the one the combine kernel uses.
#include "launch_params.h"

namespace pmxhip {

namespace {

int largest_pow2_divisor_upto(int64_t n, int cap)
{
    int r = 1;
    while (r * 2 <= cap && n % (r * 2) == 0) r *= 2;
    return r;
}

// head_dim 64, 128 or 256: up to four query heads per kv head on one set of waves; head_dim 256, and head_dim 128
// with kv heads in eights: up to eight on two sets.  At head_dim 64 and 128 a wave holds two kv heads: an odd number of them leaves
// the last half-wave idle, which a single kv head does not pay for (half of every wave).
bool quad_serves(int64_t head_dim, int64_t g, int64_t num_kv_heads)
{
    if (head_dim == 256) return g <= 8;
    if ((head_dim != 128 && head_dim != 64) || num_kv_heads == 1) return false;
    return g <= 4 || (head_dim == 128 && g <= 8 && num_kv_heads % 8 == 0);
}

} // namespace

namespace {
const char* kernel_name(int32_t kernel, bool by_sequence)
{
    switch (kernel) {
        case kDecodeKernelGeneral: return "decode_attention_kernel";
        case kDecodeKernelQuad: return "decode_attention_quad_kernel";
        case kDecodeKernelMfma16: return "decode_attention_mfma16_kernel";
        case kDecodeKernelMfma32: return by_sequence ? "decode_attention_mfma32_kernel" : "decode_attention_mfma_kernel";
        default: return "";
    }
}
} // namespace
const char* decode_kernel_name(const DecodeLaunch& a) { return kernel_name(a.kernel, a.by_sequence != 0); }
const char* decode_kernel_name(int32_t kernel) { return kernel_name(kernel, false); }

bool decode_choose(int64_t head_dim, int64_t num_heads, int64_t num_kv_heads, int32_t requested, DecodeChoice* out)
{
    if (head_dim != 64 && head_dim != 96 && head_dim != 128 && head_dim != 256) return false;
    if (num_kv_heads <= 0 || num_heads <= 0 || num_heads % num_kv_heads != 0) return false;
    const int64_t g = num_heads / num_kv_heads;
    int32_t kernel = requested;
    if (kernel == kDecodeKernelAuto) {
        // Many query heads per kv head: their VALU arithmetic outweighs the cache stream, so they become MFMA
        // columns (five and more; three and four as well on a single kv head, which would use half of the quad
        // kernel's lanes): 16 or 32 columns at head_dim 128, 32 at head_dim 64, and beyond 32 query heads per kv head
        // (multi-query models) as many passes of 32 columns as they need.  Up to four: the quad kernel, whose row
        // loads stream whole lines (head_dim 256: up to eight, on two sets of waves).  Everything else (head_dim 96,
        // a single kv head with one or two query heads, head_dim 256 with more than eight per kv head) stays on
        // the general kernel.
        if (head_dim == 128 && (g >= 5 || (g >= 3 && num_kv_heads == 1)))
            kernel = g <= kDecodeMfma16Columns ? kDecodeKernelMfma16 : kDecodeKernelMfma32;
        else if (head_dim == 64 && (g >= 5 || (g >= 3 && num_kv_heads == 1)))
            kernel = kDecodeKernelMfma32;
        else if (quad_serves(head_dim, g, num_kv_heads) && (g <= 4 || head_dim == 256))
            kernel = kDecodeKernelQuad;
        else
            kernel = kDecodeKernelGeneral;
    }
    DecodeChoice c{};
    c.kernel = kernel;
    switch (kernel) {
        case kDecodeKernelGeneral: {
            const int lanes_per_slot = head_dim == 64 ? 4 : (head_dim == 256 ? 16 : 8);
            const int slots_per_wave = 64 / lanes_per_slot;
            c.kv_heads_per_group = largest_pow2_divisor_upto(num_kv_heads, slots_per_wave < 8 ? slots_per_wave : 8);
            int gt = 1;
            while (gt < g && gt < 8) gt *= 2;
            c.q_heads_per_pass = gt;
            c.num_passes = (int32_t)((g + gt - 1) / gt);
            c.wg_tokens = decode_wg_tokens((int)head_dim, c.kv_heads_per_group);
            c.wgs_per_cu = 2;
            c.wgs_per_cu_short = c.wgs_per_cu;
            break;
        }
        case kDecodeKernelQuad: {
            if (!quad_serves(head_dim, g, num_kv_heads)) return false;
            // a wave holds two kv heads of 128 channels or one of 256; four, two or one waves per set
            const int per_wave = head_dim == 256 ? 1 : 2;
            const int64_t pairs = (num_kv_heads + per_wave - 1) / per_wave;
            c.kv_heads_per_group = per_wave * (pairs % 4 == 0 ? 4 : (pairs % 2 == 0 ? 2 : 1));
            c.q_heads_per_pass = g <= 1 ? 1 : (g <= 2 ? 2 : (g <= 4 ? 4 : 8)); // rows of the 4x4x4 products in use
            c.num_passes = 1;
            c.wg_tokens = head_dim == 64 ? 2 * kDecodeQuadTokens : kDecodeQuadTokens; // head_dim 64: blocks of 32 tokens
            // A CU holds eight of this kernel's waves, two per SIMD.  A long stream is cut for four, one per SIMD: the
            // second wave adds nothing to what the chip streams (each wave keeps three blocks of rows in flight), and
            // half as many ranges are half as many pieces to write and to combine.  Short batches, whose ranges are a
            // few blocks, still spread over all eight (their waves mostly wait), and so do the form with two sets of
            // waves per workgroup (head_dim 256 with more than four query heads per kv head: 43 against 57 us on 8 / 1
            // heads) and the workgroups of two waves (four kv heads: two such workgroups per CU ran 22 % slower than
            // four, 216 against 177 us -- their waves do not end up one per SIMD).
            const int waves = c.kv_heads_per_group / per_wave; // per set
            c.wgs_per_cu_short = 8 / waves;
            if (head_dim == 256 && g > 4) c.wgs_per_cu_short = c.wgs_per_cu_short > 1 ? c.wgs_per_cu_short / 2 : 1; // twice the waves per workgroup
            const bool one_per_simd = !(head_dim == 256 && g > 4) && waves != 2;
            c.wgs_per_cu = one_per_simd ? c.wgs_per_cu_short / 2 : c.wgs_per_cu_short;
            break;
        }
        case kDecodeKernelMfma16:
        case kDecodeKernelMfma32: {
            const int cols = kernel == kDecodeKernelMfma16 ? kDecodeMfma16Columns : kDecodeMfmaColumns;
            // the 16-column form: head_dim 128, one pass; the 32-column form: head_dim 128 or 64, any number of passes
            if (kernel == kDecodeKernelMfma16 ? (head_dim != 128 || g > cols) : (head_dim != 128 && head_dim != 64)) return false;
            c.kv_heads_per_group = num_kv_heads % 4 == 0 ? 4 : (num_kv_heads % 2 == 0 ? 2 : 1); // a wave per kv head
            c.q_heads_per_pass = cols;
            c.num_passes = (int32_t)((g + cols - 1) / cols);
            c.wg_tokens = kDecodeMfmaTokens;
            c.wgs_per_cu = kDecodeMfmaWavesPerCu / c.kv_heads_per_group;
            c.wgs_per_cu_short = c.wgs_per_cu;
            break;
        }
        default: return false;
    }
    *out = c;
    return true;
}

namespace {

constexpr double kLaneOffsets = 2147483648.0; // what a 32-bit lane offset reaches
// Bytes that the 32-bit lane offsets of a kernel span: the tokens of one wave block times the row stride, the kv
// heads that share a wave's 64-bit base times the head stride, and a row.
double lane_offset_span(const DecodeChoice& c, int64_t head_dim, int64_t stride_s, int64_t stride_h)
{
    int64_t tokens = c.wg_tokens, heads_apart = 0;
    switch (c.kernel) {
        case kDecodeKernelGeneral:
            tokens = c.wg_tokens / 4;               // a wave's block; the four waves have bases of their own
            heads_apart = c.kv_heads_per_group - 1; // every wave spans the group's kv heads
            break;
        case kDecodeKernelQuad:
            heads_apart = head_dim == 256 ? 0 : 1;  // the wave's second kv head; the first is in the wave's base
            break;
        default: break;                             // a wave per kv head: the head is in the base
    }
    return (double)tokens * (double)stride_s + (double)heads_apart * (double)stride_h + (double)head_dim;
}

// Makes the choice fit a cache layout: the kernels address a row as a 64-bit base per wave plus a 32-bit offset per
// lane, and where the kv heads of a wave lie further apart than such an offset reaches (cache_stride_h of a layout
// that keeps the heads outermost) the general kernel takes fewer kv heads per workgroup and, unless the quad kernel
// was requested, a kernel with a wave per kv head takes its steps.  The number of ranges of a plan stays valid: it
// does not depend on the grouping.  False: no kernel serves the strides (a block of tokens alone spans 2 GiB, or a
// stride is negative).
bool fit_cache_strides(int64_t head_dim, int64_t num_heads, int64_t num_kv_heads, int32_t requested,
                              int64_t stride_s, int64_t stride_h, DecodeChoice* c)
{
    if (stride_s < 0 || stride_h < 0) return false;
    if (lane_offset_span(*c, head_dim, stride_s, stride_h) < kLaneOffsets) return true;
    if (c->kernel == kDecodeKernelGeneral) {
        // fewer kv heads per wave (more tokens instead) until the heads' distance fits; one kv head per workgroup
        // has no head term at all
        while (c->kv_heads_per_group > 1) {
            c->kv_heads_per_group /= 2;
            c->wg_tokens = decode_wg_tokens((int)head_dim, c->kv_heads_per_group);
            if (lane_offset_span(*c, head_dim, stride_s, stride_h) < kLaneOffsets) return true;
        }
        return false;
    }
    if (c->kernel == kDecodeKernelQuad && requested == kDecodeKernelAuto) {
        // two kv heads further apart than a lane offset reaches: a kernel with a wave per kv head takes the step
        DecodeChoice alt;
        const int64_t g = num_heads / num_kv_heads;
        const int32_t other = head_dim == 128 && g <= kDecodeMfma16Columns ? kDecodeKernelMfma16
                              : (head_dim == 128 || head_dim == 64 ? kDecodeKernelMfma32 : kDecodeKernelGeneral);
        if (!decode_choose(head_dim, num_heads, num_kv_heads, other, &alt)) return false;
        *c = alt;
        return fit_cache_strides(head_dim, num_heads, num_kv_heads, other, stride_s, stride_h, c);
    }
    return false;
}

} // namespace

bool decode_choose_columns(int64_t head_dim, int64_t columns, int64_t num_kv_heads, DecodeChoice* out)
{
    if ((head_dim != 64 && head_dim != 96 && head_dim != 128 && head_dim != 256) || columns <= 0 || num_kv_heads <= 0) return false;
    DecodeChoice c{};
    c.kernel = columns <= kDecodeMfma16Columns || head_dim == 256 ? kDecodeKernelMfma16 : kDecodeKernelMfma32;
    const int cols = c.kernel == kDecodeKernelMfma16 ? kDecodeMfma16Columns : kDecodeMfmaColumns;
    c.kv_heads_per_group = num_kv_heads % 4 == 0 ? 4 : (num_kv_heads % 2 == 0 ? 2 : 1); // a wave per kv head
    c.q_heads_per_pass = cols;
    c.num_passes = (int32_t)((columns + cols - 1) / cols);
    c.wg_tokens = kDecodeMfmaTokens;
    c.wgs_per_cu = kDecodeMfmaWavesPerCu / c.kv_heads_per_group;
    c.wgs_per_cu_short = c.wgs_per_cu;
    *out = c;
    return true;
}

namespace {

// (kv head, pass) workgroups of one sequence or range on the column kernels
int64_t column_groups(int64_t head_dim, int64_t columns, int64_t num_kv_heads)
{
    DecodeChoice c;
    return decode_choose_columns(head_dim, columns, num_kv_heads, &c) ? num_kv_heads * c.num_passes : 0;
}

// Workgroups of eight waves that a CU holds: their rings are all of its LDS, half of it at head_dim 64.
int64_t eight_wave_groups_per_cu(int64_t head_dim) { return head_dim == 64 ? 2 : 1; }

// Waves that share a sequence's tokens when every workgroup has a sequence (and kv head, and pass) of its own: eight while
// that leaves no workgroup waiting for a CU, four up to two rounds of workgroups, beyond that there are waves enough (a
// wave per kv head).  32 q / 8 kv heads of 128, lengths L/3 to L: 16 sequences of 512 tokens 11.1 / 11.6 us with eight / four
// waves, 64 of 256 14.9 / 11.6 and 19.3 with one, 64 of 1024 35.3 / 30.8 / 64.0.
int decode_share(int64_t workgroups, int64_t head_dim, int compute_units)
{
    if (compute_units <= 0) return 1;
    if (workgroups <= eight_wave_groups_per_cu(head_dim) * compute_units) return 8;
    return workgroups <= (head_dim == 256 ? 4 : 5) * (int64_t)compute_units ? 4 : 1;
}

// The quad kernel takes its shapes sequence by sequence where every one of its waves (two kv heads, eight to a CU) has a sequence to
// begin with: 32 q / 8 kv heads of 128, 512 sequences of 100-300 tokens 57 us, 61 on the column kernel, 68 cut into ranges.  With
// one query head per kv head, a quarter of the column kernel's work, from where that kernel has a wave per pair: 32 / 32 heads of
// 128, 100 sequences of 43-128 23.5 us, 31.4 on the column kernel, 26.8 over ranges.  With a mask, whose values the column kernel
// waits for together with its rows, from where that kernel's waves come in a second round: 32 / 8 heads, 300 sequences of 100-300
// 48.8 us, 56.9 on the column kernel; 16 / 4 heads, 512 of them 47.3 and 45.1.
bool quad_by_sequence(int64_t sequences, int64_t num_kv_heads, int64_t g, bool mask, int compute_units)
{
    if (g > 4 || compute_units <= 0) return false;
    const int64_t pairs = sequences * num_kv_heads;
    return pairs >= 16 * (int64_t)compute_units || (g == 1 && pairs > 5 * (int64_t)compute_units) || (mask && pairs > 8 * (int64_t)compute_units);
}

// One to four sequences cut into ranges run on the column kernels where those are the faster ones: 32 q / 8 kv heads of 128, one
// sequence of 1024 / 4096 / 16384 tokens 14.1 / 15.3 / 21.4 us on the quad kernel, 11.3 / 12.8 / 19.5 here; four of 1024 / 2048 /
// 4096 14.0 / 16.7 / 19.1 and 11.6 / 13.3 / 16.9.  Not with one query head per kv head at head_dim 128 (the quad kernel has a
// quarter of the arithmetic to do there: one of 4096 15.5 against 18.8) and not at head_dim 256.  From five on the quad kernel is
// the faster one (five of 333-1000 14.0 against 14.9, of 1333-4000 19.9 against 22.7; eight 16.0 / 15.1 and 24.1 / 25.1).
constexpr int64_t kFewSequences = 4;
bool few_sequences_on_columns(int64_t sequences, int64_t head_dim, int64_t g)
{
    return sequences <= kFewSequences && (head_dim == 64 || (head_dim == 128 && g >= 2));
}

// The quad kernel's form for whole sequences has one set of waves.
bool quad_takes_whole(const DecodeLaunch& a) { return a.num_kv_repeats <= 4 && decode_quad_launch_ok(a); }

// How long the sequences of a batch may be (its longest) to be taken whole instead of cut into ranges with a combine launch
// behind them, by the (sequence, kv head, pass) workgroups per CU: the crossing of the two times, measured over 30 head shapes x
// 1-512 sequences x 64-16384 tokens and short chunks of 1-32 columns, lengths L / 3 to L, ten layers in turn.  Where shapes of
// a row differ the shorter one stands, so that a batch next to the line is seldom slower than over ranges (of 1900 batches 3 by
// more than 8 %).  Few workgroups leave the chip idle and ranges fill it; from one per CU on the waves are there either
// way, and ranges even out the lengths.  Past eight per CU the waves come in a second round.  While workgroups are few, eight waves
// share a sequence and another 256 tokens are another block for each: the step's time rises there at once (32 / 32 heads of 96, one
// sequence: whole 0.93 of the time over ranges at 500 tokens, 1.18 at 600; 24 / 1 of 128, seven: 0.99 at 250, 1.20 at 320; 16 / 16 of
// 256, four: 0.95 and 1.12), so those lines lie on multiples of 256.
struct WholeUpTo {
    double masked;         // with a mask, times this where the column kernels run: they wait for its values, the quad kernel streams them
    int32_t tokens[15];    // workgroups per CU up to kWholeLoads[i], and beyond
};
constexpr double kWholeLoads[14] = {0.05, 0.1, 0.2, 0.4, 0.75, 1, 1.6, 2, 2.75, 3.5, 5, 8, 15.99, 32};
constexpr WholeUpTo kWholeColumns16 = {0.6, {440, 470, 500, 512, 825, 1150, 765, 765, 595, 590, 520, 500, 400, 500, 500}};
constexpr WholeUpTo kWholeColumns32 = {0.6, {256, 256, 256, 580, 1300, 1600, 1400, 1400, 1290, 1200, 1200, 900, 700, 600, 600}};
constexpr WholeUpTo kWholeColumns64 = {0.9, {600, 710, 740, 1030, 1500, 1030, 800, 560, 700, 550, 650, 720, 400, 550, 550}}; // head_dim 64
constexpr WholeUpTo kWholeQuad64 = {0.45, {850, 850, 850, 1600, 1600, 1000, 800, 600, 560, 560, 530, 380, 380, 900, 900}};
constexpr WholeUpTo kWholeQuad128One = {1.0, {480, 480, 510, 512, 512, 512, 350, 295, 175, 175, 140, 500, 220, 200, 200}}; // one query head per kv head
constexpr WholeUpTo kWholeQuad128 = {0.6, {500, 512, 512, 512, 970, 1000, 880, 680, 640, 340, 300, 300, 150, 400, 400}};
constexpr WholeUpTo kWholeQuad256One = {1.0, {256, 256, 256, 256, 420, 430, 250, 185, 90, 90, 0, 190, 190, 190, 190}};
constexpr WholeUpTo kWholeQuad256 = {0.55, {450, 450, 470, 512, 760, 780, 550, 500, 300, 260, 160, 160, 160, 200, 200}};
constexpr WholeUpTo kWholeQuad256Two = {1.0, {256, 512, 512, 1140, 1600, 1600, 1600, 1600, 1600, 1600, 1600, 1600, 1600, 1600, 1600}}; // two sets of waves
constexpr WholeUpTo kWholeGeneralOne = {0.75, {512, 512, 512, 512, 512, 512, 350, 285, 200, 170, 145, 145, 128, 100, 0}};
constexpr WholeUpTo kWholeGeneralFour = {1.0, {930, 930, 1100, 1600, 1600, 1600, 980, 980, 700, 600, 560, 500, 370, 530, 530}};
constexpr int32_t kAnyLength = INT32_MAX; // many query heads on the general kernel: several times the column kernels' time
constexpr WholeUpTo kWholeGeneral = {1.0, {870, 1400, 1400, kAnyLength, kAnyLength, kAnyLength, kAnyLength, kAnyLength, kAnyLength, kAnyLength,
                                           kAnyLength, kAnyLength, kAnyLength, kAnyLength, kAnyLength}};

const WholeUpTo& whole_row(const DecodeChoice& by_shape, int64_t head_dim, int64_t g, int64_t num_kv_heads)
{
    switch (by_shape.kernel) {
        case kDecodeKernelMfma16: return kWholeColumns16;
        case kDecodeKernelMfma32: return head_dim == 64 ? kWholeColumns64 : kWholeColumns32;
        case kDecodeKernelQuad:
            if (head_dim == 64) return kWholeQuad64;
            if (head_dim == 128) return g == 1 ? kWholeQuad128One : kWholeQuad128;
            return g == 1 ? kWholeQuad256One : (g <= 4 ? kWholeQuad256 : kWholeQuad256Two);
        default: return head_dim == 96 && num_kv_heads > 1 && g <= 4 ? (g == 1 ? kWholeGeneralOne : kWholeGeneralFour) : kWholeGeneral;
    }
}

// `columns`: query heads per kv head, or the (position, head) columns of a short chunk
int64_t whole_up_to(const DecodeChoice& by_shape, int64_t sequences, int64_t head_dim, int64_t columns, int64_t num_kv_heads, bool mask, int cus)
{
    const WholeUpTo& row = whole_row(by_shape, head_dim, columns, num_kv_heads);
    const double load = (double)(sequences * column_groups(head_dim, columns, num_kv_heads)) / cus;
    int i = 0;
    while (i < 14 && load > kWholeLoads[i]) ++i;
    int64_t tokens = row.tokens[i];
    // (at head_dim 64 a masked step over ranges is another kernel's, and slower as well)
    const bool quad = by_shape.kernel == kDecodeKernelQuad;
    const bool streams_mask = quad && (head_dim == 64 ? columns > 1 : quad_by_sequence(sequences, num_kv_heads, columns, true, cus));
    if (mask && tokens != kAnyLength && !streams_mask) tokens = (int64_t)(row.masked * (double)tokens);
    // the pieces of few columns cost less, those of many more (32 / 8 heads of 128, 100 chunks of one row: level at 476 tokens, of two
    // rows at 616, of four at 957)
    if (by_shape.kernel != kDecodeKernelQuad && by_shape.kernel != kDecodeKernelGeneral && load > 1) {
        if (columns < 5) tokens = tokens * 3 / 5;
        else if (columns >= 12 && columns <= kDecodeMfma16Columns) tokens = tokens * 5 / 4;
        else if (columns > kDecodeMfmaColumns && head_dim == 64) tokens *= 2; // (the range kernel's passes: 71 / 1 heads, 300 of 1600)
    }
    if (by_shape.kernel == kDecodeKernelMfma32 && head_dim == 64 && sequences <= kFewSequences && tokens > 590) tokens = 590;
    // a step of a few sequences has ranges of the column kernels' own
    if (by_shape.kernel == kDecodeKernelQuad && few_sequences_on_columns(sequences, head_dim, columns)) {
        const int64_t most = head_dim != 64 ? 480 : (sequences == 1 ? 512 : 700);
        if (tokens > most) tokens = most;
    }
    return tokens;
}

// What short chunks cost (us) sequence by sequence, against the tile kernel.  A wave's block of 32 tokens takes `alone` with a wave
// per SIMD and `shared` with two; a workgroup starts in 3.5.
constexpr double kSequenceMargin = 0.8;
double sequence_cost(int64_t sequences, int64_t max_kvlen, int64_t head_dim, int64_t columns, int64_t num_kv_heads, int cus)
{
    const int64_t wgs = sequences * column_groups(head_dim, columns, num_kv_heads);
    const double wide = columns > kDecodeMfma16Columns && head_dim != 256 ? 1.15 : 1.0;
    const double shared = wide * (head_dim == 64 ? 1.6 : head_dim == 96 ? 2.6 : head_dim == 128 ? 3.0 : 4.6);
    const double alone = wide * (head_dim == 64 ? 1.24 : head_dim == 96 ? 1.55 : head_dim == 128 ? 1.75 : 2.8);
    const int share = decode_share(wgs, head_dim, cus);
    const double blocks = (double)((max_kvlen + 32 * share - 1) / (32 * share));
    if (share == 8) return 4.4 + shared * blocks * (wgs > cus ? 2 : 1);
    if (share == 4 && wgs <= cus) return 4.4 + alone * blocks;
    if (share == 4 && wgs <= 2 * cus) return 4.6 + shared * blocks;
    const double rounds = share == 4 ? wgs / (2.0 * cus) : wgs / (8.0 * cus);
    if (rounds <= 1) return 4.5 + (wgs <= 4 * cus ? alone : shared) * blocks;
    return 1 + rounds * (3.5 + 0.8 * shared * blocks);
}

} // namespace

// The column and MFMA kernels take the maximum of the raw products and divide the mask by the scale: it has to be positive, and not so
// small that a mask divided by it passes the maximum they begin with.  The quad and general kernels scale first.
bool columns_scale(float attn_scale) { return attn_scale >= 1e-20f; }

// The kernel of a launch without a request, in place of the choice by shape.
static void choose_launch(const DecodeLaunch& a, int compute_units, DecodeChoice* c)
{
    const int64_t g = a.num_heads / a.num_kv_heads;
    // the column kernels' blocks are 32 tokens, the quad kernel's at head_dim 128 and 256 16: rows further apart stay where they fit
    DecodeChoice columns{};
    const bool fit = columns_scale(a.attn_scale) && decode_choose_columns(a.head_dim, g, a.num_kv_heads, &columns) &&
                     lane_offset_span(columns, a.head_dim, a.cache_stride_s, a.cache_stride_h) < kLaneOffsets;
    if (a.ranges == 1) {
        // A single range is for kernels that take every sequence whole (a kernel over ranges would walk the batch with one
        // workgroup), and the plan knows neither mask nor buffers.  What the quad kernel cannot take whole is the column kernels',
        // except one query head per kv head at head_dim 64 where those have a wave per pair: 8 / 8 heads, 512 sequences of 100-300
        // tokens with a mask 53.0 us on the column kernel, 37.9 on the general one, with rows of 8 bytes 46.9 and 36.2.
        if (c->kernel == kDecodeKernelQuad) {
            if (quad_takes_whole(a) && quad_by_sequence(a.decoding_batches, a.num_kv_heads, g, a.attn_mask != nullptr, compute_units)) return;
            if (a.head_dim == 64 && g == 1 && a.num_kv_heads % 8 == 0 && !quad_takes_whole(a) &&
                decode_share(a.decoding_batches * a.num_kv_heads, a.head_dim, compute_units) == 1 && compute_units > 0) {
                decode_choose(a.head_dim, a.num_heads, a.num_kv_heads, kDecodeKernelGeneral, c);
                return;
            }
        }
        if (fit) *c = columns;
        else if (c->kernel == kDecodeKernelQuad && !quad_takes_whole(a)) decode_choose(a.head_dim, a.num_heads, a.num_kv_heads, kDecodeKernelGeneral, c);
    } else if (fit && c->kernel == kDecodeKernelQuad && few_sequences_on_columns(a.decoding_batches, a.head_dim, g)) {
        *c = columns;
    }
}

int64_t decode_choose_ranges(const DecodeChoice& by_shape, int64_t sequences, int64_t max_kvlen, int64_t head_dim, int64_t num_heads,
                             int64_t num_kv_heads, int compute_units, bool automatic, bool mask)
{
    const int64_t g = num_heads / num_kv_heads;
    const int64_t max_tokens = sequences * (max_kvlen > 0 ? max_kvlen : 1);
    DecodeChoice c = by_shape;
    if (automatic && compute_units > 0) {
        if (max_kvlen <= whole_up_to(by_shape, sequences, head_dim, g, num_kv_heads, mask, compute_units)) return 1;
        if (c.kernel == kDecodeKernelQuad && few_sequences_on_columns(sequences, head_dim, g)) decode_choose_columns(head_dim, g, num_kv_heads, &c);
    }
    const bool columns = c.kernel == kDecodeKernelMfma16 || c.kernel == kDecodeKernelMfma32;
    const int min_tokens = decode_min_tokens_per_range(c.wg_tokens);
    const int64_t groups = ((num_kv_heads + c.kv_heads_per_group - 1) / c.kv_heads_per_group) * c.num_passes;
    const int64_t shared_groups = column_groups(head_dim, g, num_kv_heads);
    if (automatic && c.kernel == kDecodeKernelMfma16 && sequences == 1 && max_tokens * shared_groups <= kSharedStreamTokens) {
        // a single sequence: ranges of 128 tokens or more that four waves share, one workgroup per CU
        const int64_t most = compute_units / shared_groups;
        const int64_t useful = (max_tokens + 127) / 128;
        return useful < most ? useful : (most > 1 ? most : 2);
    }
    // as many ranges as the kernel wants workgroups per CU for a long stream (the quad kernel one wave per SIMD, the
    // others two; more, smaller workgroups where a wave serves one or two kv heads)
    const int64_t long_slots = (int64_t)compute_units * c.wgs_per_cu;
    const int64_t slots = (int64_t)compute_units * c.wgs_per_cu_short; // what the rules for short batches below count with
    int64_t ranges = (long_slots + groups - 1) / groups;
    // A short batch: ranges of about 128 tokens (twice the smallest) where those still fill half of the slots,
    // shorter ones -- down to the smallest -- only to get that far: a piece has a fixed cost, and an idle CU costs more.
    const int64_t comfortable = 2 * (int64_t)min_tokens;
    const int64_t useful = (max_tokens + comfortable - 1) / comfortable;
    if (ranges > useful) {
        ranges = useful;
        const int64_t half = slots / 2 / groups > 1 ? slots / 2 / groups : 1;
        if (ranges < half) {
            const int64_t finer = (max_tokens + min_tokens - 1) / min_tokens;
            ranges = half < finer ? half : finer;
            // The column kernels' smallest is a block: 64 q / 8 kv heads of 128, one sequence of 4096 tokens 15.1 us with ranges of 64
            // tokens and 13.8 with 32, four of 1024 15.5 and 12.8; 14 / 2 heads of 64, 16 of 1024 13.0 and 10.5.  With 32 columns at
            // head_dim 128 up to a wave per CU and pass: 48 / 1 heads, 16 sequences of 100-300 13.1 us with 69 ranges, 11.4 with
            // 138, but 30 of 233-700 17.1 with 321 and 18.9 with 512.
            if (automatic && columns) {
                const int64_t most = c.kernel == kDecodeKernelMfma32 && head_dim == 128 ? slots / 4 / groups : half;
                const int64_t finest = (max_tokens + kDecodeMfmaTokens - 1) / kDecodeMfmaTokens;
                const int64_t blocks = most < finest ? most : finest;
                if (blocks > ranges) ranges = blocks;
            }
        }
        // a step of a few sequences: below a workgroup per two CUs the ranges go down to the kernel's floor
        const int64_t sparse = compute_units / 2 / groups > 1 ? compute_units / 2 / groups : 1;
        if (ranges < sparse) {
            const int floor_tokens = decode_floor_tokens_per_range(c.wg_tokens);
            const int64_t finest = (max_tokens + floor_tokens - 1) / floor_tokens;
            ranges = sparse < finest ? sparse : finest;
        }
    }
    return ranges > 1 ? ranges : 1;
}

// The two kernels of 16 columns over ranges (decode_attn_mfma.hip has the other's figures): the ring's where a single sequence's
// pieces are shared by four waves, at head_dim 64, and where four waves of a workgroup walk 500 tokens and more per range (28 / 4
// heads: 100 sequences of 1333-4000, 520 per range, 68.5 -> 67.9 us, 300 of them 196 -> 188; 64 / 8 heads, 30 of them, 310 per range,
// 49.9 and 50.6).  One or two waves per workgroup gain nothing from it (10 / 2 heads, 100 sequences of 5333-16000 127 against 133 us), nor does a
// mask, whose values are awaited together with the rows (28 / 4 heads, 300 of 1333-4000 219 against 221).  Without a length: as long
// streams, but for a few sequences.
bool decode_ring(const DecodeLaunch& a, int64_t max_kvlen)
{
    if (a.kernel != kDecodeKernelMfma16 || a.by_sequence) return false;
    if (a.head_dim != 128 || a.shared_pieces > 1) return true;
    if (a.kv_heads_per_group != 4 || a.attn_mask != nullptr) return false;
    if (max_kvlen <= 0) return a.decoding_batches > kFewSequences;
    return 0.67 * (double)max_kvlen * (double)a.decoding_batches >= 500.0 * (double)a.ranges;
}

// How the kernel takes the launch: by_sequence, shared_pieces and ring.
static void choose_form(DecodeLaunch* a, int compute_units, int64_t max_kvlen)
{
    a->by_sequence = 0;
    a->shared_pieces = 1;
    const bool columns = a->kernel == kDecodeKernelMfma16 || a->kernel == kDecodeKernelMfma32;
    a->ring = 0;
    a->by_sequence = a->ranges == 1 && (a->kernel != kDecodeKernelQuad || quad_takes_whole(*a));
    if (!columns) return;
    const int64_t wgs = (a->by_sequence ? a->decoding_batches : a->ranges) * a->num_kv_heads * a->num_passes;
    if (a->by_sequence) a->shared_pieces = decode_share(wgs, a->head_dim, compute_units);
    else if (a->kernel == kDecodeKernelMfma16 && a->decoding_batches == 1 && wgs <= compute_units) a->shared_pieces = 4;
    a->ring = decode_ring(*a, max_kvlen);
}

bool decode_quad_launch_ok(const DecodeLaunch& a)
{
    if (a.output_stride_s % 8 != 0 || (reinterpret_cast<uintptr_t>(a.output) & 15u) != 0) return false;
    if (a.attn_mask != nullptr) {
        if (a.head_dim == 64) return false; // no mask form at head_dim 64
        if (a.num_kv_repeats > 4 || a.mask_stride_h < 0) return false;
        if (((double)a.num_heads * (double)a.mask_stride_h + 64.0) * 2.0 >= 4294967296.0) return false;
    }
    return true;
}

DecodeSelect decode_select(DecodeLaunch* a, int32_t requested, bool columns, int compute_units, int64_t max_kvlen, DecodeChoice* out)
{
    DecodeChoice c{};
    *out = c;
    if (columns ? !decode_choose_columns(a->head_dim, a->num_kv_repeats, a->num_kv_heads, &c)
                : !decode_choose(a->head_dim, a->num_heads, a->num_kv_heads, requested, &c))
        return DecodeSelect::kNoKernel;
    if (!columns && requested == kDecodeKernelAuto) choose_launch(*a, compute_units, &c);
    if ((c.kernel == kDecodeKernelMfma16 || c.kernel == kDecodeKernelMfma32) && !columns_scale(a->attn_scale)) {
        if (columns || requested != kDecodeKernelAuto) return DecodeSelect::kScale;
        decode_choose(a->head_dim, a->num_heads, a->num_kv_heads, kDecodeKernelGeneral, &c);
    }
    if (c.kernel == kDecodeKernelQuad && !decode_quad_launch_ok(*a)) {
        if (requested == kDecodeKernelQuad) return DecodeSelect::kQuadBuffers;
        // (with a mask at head_dim 64: 32 / 8 heads, 100 sequences of 233-700 51.0 us on the general kernel, 40 / 8 35.2 on this one)
        const bool columns64 = a->head_dim == 64 && a->attn_mask != nullptr && a->num_kv_repeats > 1 && columns_scale(a->attn_scale);
        decode_choose(a->head_dim, a->num_heads, a->num_kv_heads, columns64 ? kDecodeKernelMfma32 : kDecodeKernelGeneral, &c);
    }
    const bool fits = fit_cache_strides(a->head_dim, a->num_heads, a->num_kv_heads, requested, a->cache_stride_s, a->cache_stride_h, &c);
    *out = c;
    if (!fits) return DecodeSelect::kCacheStrides;
    a->kernel = c.kernel;
    a->kv_heads_per_group = c.kv_heads_per_group;
    a->q_heads_per_pass = c.q_heads_per_pass;
    a->num_passes = c.num_passes;
    a->wg_tokens = c.wg_tokens;
    a->min_tokens_per_range = decode_floor_tokens_per_range(c.wg_tokens);
    choose_form(a, compute_units, max_kvlen);
    return DecodeSelect::kSelected;
}

int decode_wg_tokens(int head_dim, int kv_heads_per_group)
{
    const int lps = head_dim == 64 ? 4 : (head_dim == 256 ? 16 : 8); // lanes per slot
    return kDecodeSlotTokens * (64 / lps / kv_heads_per_group) * kDecodeGeneralWaves;
}

// Short chunks (a few query tokens per sequence: speculative decoding's candidates, the tail of a chunked prefill)
// leave most of the tile kernel's 256 columns empty and are bound by its tile staging.  Where a kv head's (query
// position, query head) pairs fit the 32 columns of the decode step's MFMA kernel they run there instead, over token
// ranges with a combine kernel, which streams the cache at the decode rate.  That path has no mask, alibi or fp16-K/V
// form and serves head_dim 64 and 128.
bool prefill_chunk_shape(int64_t max_seqlen, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim)
{
    constexpr int64_t kPrefillChunkColumns = 32;
    if (head_dim != 64 && head_dim != 128) return false;
    if (num_kv_heads <= 0 || num_heads % num_kv_heads != 0 || max_seqlen <= 0) return false;
    return max_seqlen * (num_heads / num_kv_heads) <= kPrefillChunkColumns;
}

// Chunks of up to 32 columns go sequence by sequence where that is faster than ranges (whole_up_to) or, which is what serves head_dim 96
// and 256 and calls without a workspace, than the tile kernel, whose workgroups have 256 columns for them: 64 q / 8 kv heads of 128, 147
// chunks of 2-4 rows over up to 391 tokens 63 -> 52 us over ranges, 16 / 4 heads, 15 of 2 over 433 17.1 -> 14.0; against the tile kernel
// 16 / 16 heads of 256, 30 of 2-18 over 3208 429 -> 192 us, 8 / 1 heads of 256, 178 of 1-2 over 591 59 -> 24, 32 / 32 heads of 96, four
// of 2 over 6971 114 -> 97.
bool prefill_by_sequence(int64_t sequences, int64_t max_seqlen, int64_t max_kvlen, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                         bool ranges_served, int compute_units)
{
    constexpr int64_t kMostColumns = 32; // (a pass of the 32-column form, two of the 16-column form at head_dim 256)
    if (num_kv_heads <= 0 || num_heads % num_kv_heads != 0 || max_seqlen <= 0 || sequences <= 0 || max_kvlen <= 0 || compute_units <= 0) return false;
    const int64_t columns = max_seqlen * (num_heads / num_kv_heads);
    DecodeChoice c;
    if (columns > kMostColumns || !decode_choose_columns(head_dim, columns, num_kv_heads, &c)) return false;
    if (ranges_served) { // (the kernel over ranges: prefill_chunk_kernel)
        c.kernel = columns <= kDecodeMfma16Columns && head_dim == 128 ? kDecodeKernelMfma16 : kDecodeKernelMfma32;
        return max_kvlen <= whole_up_to(c, sequences, head_dim, columns, num_kv_heads, false, compute_units);
    }
    const double cost = sequence_cost(sequences, max_kvlen, head_dim, columns, num_kv_heads, compute_units);
    // the tile kernel: a workgroup per (sequence, kv head) and CU, 3.4 us for 64 kv tokens, or the tokens of few of them shared out
    const double tile = (head_dim == 256 ? 7.0 : head_dim == 64 ? 2.4 : 3.4) / 64 * (double)max_kvlen;
    const double rounds = (double)(sequences * num_kv_heads) / compute_units;
    const double alone = rounds < 1 ? 8 + tile : 4 + rounds * (4 + 0.75 * tile), shared = 30 + rounds * tile;
    return cost < kSequenceMargin * (rounds < 1 && shared < alone ? shared : alone);
}

} // namespace pmxhip
