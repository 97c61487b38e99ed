// Prints what the host decides for decode calls: one call per input line, one line of output each (test_decode_select.py).
// The device's compute units are an input, so the choice can be checked where there is no GPU.
#include "decode_select.cpp"

#include <cstdio>

using namespace pmxhip;

int main()
{
    long long sequences, max_kvlen, ranges, heads, kv_heads, head_dim, mask, output_offset, output_stride, stride_s, stride_h, requested, cus, sized;
    double scale;
    while (scanf("%lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lld %lf %lld %lld %lld", &sequences, &max_kvlen, &ranges, &heads, &kv_heads,
                 &head_dim, &mask, &output_offset, &output_stride, &stride_s, &stride_h, &scale, &requested, &cus, &sized) == 15) {
        DecodeChoice c;
        if (!decode_choose(head_dim, heads, kv_heads, (int32_t)requested, &c)) {
            printf("no-kernel\n");
            continue;
        }
        if (ranges == 0)
            ranges = decode_choose_ranges(c, sequences, max_kvlen, head_dim, heads, kv_heads, (int)cus, requested == kDecodeKernelAuto, mask == 2);
        DecodeLaunch a{};
        alignas(16) static char buffer[64];
        a.output = buffer + output_offset;
        a.attn_mask = mask ? buffer : nullptr;
        a.attn_scale = (float)scale;
        a.num_kv_repeats = heads / kv_heads;
        a.output_stride_s = output_stride;
        a.mask_stride_s = 4096;
        a.cache_stride_s = stride_s;
        a.cache_stride_h = stride_h;
        a.decoding_batches = sequences;
        a.num_heads = heads;
        a.num_kv_heads = kv_heads;
        a.head_dim = (int32_t)head_dim;
        a.ranges = (int32_t)ranges;
        const DecodeSelect rc = decode_select(&a, (int32_t)requested, false, (int)cus, sized ? max_kvlen : 0, &c);
        if (rc != DecodeSelect::kSelected) {
            printf("%s %lld\n", rc == DecodeSelect::kNoKernel ? "no-kernel" : rc == DecodeSelect::kQuadBuffers ? "quad-buffers" : rc == DecodeSelect::kScale ? "scale" : "strides", ranges);
            continue;
        }
        printf("%s %lld %d %d %d\n", decode_kernel_name(a), ranges, a.by_sequence, a.shared_pieces, a.ring);
    }
    return 0;
}
