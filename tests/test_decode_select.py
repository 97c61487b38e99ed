"""Which kernel a decode call runs and whether it takes its sequences whole, on the CPU: csrc/decode_select.cpp compiled with
g++ behind a small program that reads calls and prints the decision for a given number of compute units."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GENERAL, QUAD, MFMA16, MFMA32, MFMA = ("decode_attention_kernel", "decode_attention_quad_kernel", "decode_attention_mfma16_kernel",
                                       "decode_attention_mfma32_kernel", "decode_attention_mfma_kernel")


@pytest.fixture(scope="module")
def select(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("select") / "decode_select_check")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "ppl.llm.kernel.cuda_amd", "csrc"),
                    os.path.join(ROOT, "tests", "select", "decode_select_check.cpp"), "-o", exe], check=True, timeout=300)

    def call(sequences, heads, kv_heads, head_dim, max_kvlen, ranges=0, mask=False, output_offset=0, output_stride=None, stride_s=None,
             stride_h=None, scale=0.088, requested=0, cus=256, sized=False, ring=False):
        """(kernel, ranges, whole sequences) of one call, or ("refused", ranges, reason).  mask: "planned" = the plan knows of it;
        sized: the launch knows the longest sequence; ring: (waves that share a piece, the ring kernel) instead"""
        d = head_dim
        fields = (sequences, max_kvlen, ranges, heads, kv_heads, d, 2 if mask == "planned" else int(mask), output_offset,
                  heads * d if output_stride is None else output_stride, 2 * kv_heads * d if stride_s is None else stride_s,
                  d if stride_h is None else stride_h, scale, requested, cus, int(sized))
        out = subprocess.run([exe], input=" ".join(str(f) for f in fields) + "\n", capture_output=True, text=True, check=True, timeout=60).stdout.split()
        if len(out) < 5:
            return "refused", int(out[1]) if len(out) > 1 else 0, out[0]
        return (int(out[3]), out[4] == "1") if ring else (out[0], int(out[1]), out[2] == "1")
    return call


MANY_SHORT = [(512, 32, 8, 128, 300), (128, 32, 32, 128, 200), (512, 8, 8, 64, 300), (512, 16, 8, 256, 150), (600, 9, 9, 64, 100)]


@pytest.mark.parametrize("shape", MANY_SHORT)
def test_many_short_sequences_are_taken_whole_whatever_the_mask_and_the_buffers(select, shape):
    """The plan of one range knows neither mask nor output: a kernel over ranges would walk the batch with one workgroup."""
    assert select(*shape) == (QUAD, 1, True)
    hq, d = shape[1], shape[3]
    instead = GENERAL if shape[1:4] == (8, 8, 64) else MFMA16
    assert select(*shape, mask=True) == (instead if d == 64 else QUAD, 1, True)  # the quad kernel has no mask form at head_dim 64
    for form in (dict(output_offset=8), dict(output_stride=hq * d + 4), dict(mask=True, output_offset=8)):
        assert select(*shape, **form) == (instead, 1, True), form


@pytest.mark.parametrize("form", [dict(), dict(mask=True), dict(output_offset=8)])
def test_a_single_range_without_a_request_is_never_one_workgroup(select, form):
    for hq, hkv, d in [(8, 8, 64), (32, 8, 64), (14, 2, 64), (5, 1, 64), (32, 32, 96), (40, 1, 96), (32, 32, 128), (32, 8, 128), (64, 8, 128),
                       (28, 4, 128), (8, 1, 128), (5, 5, 128), (48, 1, 128), (16, 16, 256), (16, 8, 256), (8, 1, 256), (24, 1, 256)]:
        for n in (1, 4, 5, 60, 512, 3000):
            kernel, ranges, whole = select(n, hq, hkv, d, 200, ranges=1, **form)
            assert whole and ranges == 1, (n, hq, hkv, d, kernel)


# (sequences, query heads, kv heads, head_dim, longest): measured per decode call, whole sequences / ranges + combine
WHOLE = [(60, 8, 8, 64, 500), (100, 32, 8, 64, 300), (16, 14, 2, 64, 700), (32, 32, 8, 128, 256), (5, 32, 8, 128, 500), (60, 64, 8, 128, 500),
         (300, 8, 1, 128, 500), (512, 8, 1, 128, 500), (100, 40, 1, 96, 8000), (300, 24, 2, 256, 8000), (30, 24, 1, 256, 8000), (300, 32, 32, 128, 128),
         (512, 32, 8, 128, 300), (300, 8, 1, 256, 1600), (512, 16, 8, 256, 150), (1, 32, 32, 96, 500), (7, 16, 4, 128, 500), (7, 24, 1, 128, 250),
         (4, 16, 16, 256, 250), (16, 8, 1, 256, 510), (4, 32, 8, 64, 600)]
CUT = [(300, 8, 8, 64, 1600), (100, 8, 8, 64, 2400), (300, 32, 8, 64, 1000), (100, 40, 8, 64, 4000), (300, 14, 2, 64, 8000), (300, 48, 1, 128, 2400),
       (100, 32, 32, 96, 200), (300, 32, 32, 96, 128), (30, 8, 8, 96, 1000), (300, 16, 8, 128, 500), (160, 32, 32, 128, 300), (160, 16, 16, 256, 200),
       (5, 8, 1, 128, 700), (160, 28, 4, 128, 1000), (300, 64, 8, 128, 500), (1, 32, 32, 96, 600), (2, 32, 32, 96, 600), (7, 8, 8, 96, 600),
       (2, 32, 32, 128, 600), (7, 16, 4, 128, 600), (7, 64, 8, 128, 600), (7, 24, 1, 128, 320), (4, 16, 16, 256, 320), (7, 8, 8, 256, 320),
       (1, 8, 1, 256, 320), (7, 32, 32, 64, 1030), (1, 32, 8, 64, 600)]


def test_sequences_are_taken_whole_where_that_was_measured_faster(select):
    for shape in WHOLE:
        assert select(*shape)[1:] == (1, True), shape
    for shape in CUT:
        kernel, ranges, whole = select(*shape)
        assert ranges > 1 and not whole, shape
    # a mask that the quad kernel streams changes nothing, one that the column kernels wait for takes whole sequences half as far
    for shape in ((512, 32, 8, 128, 300), (600, 16, 8, 256, 150), (300, 32, 32, 128, 128)):
        assert select(*shape, mask="planned") == (QUAD, 1, True), shape
    assert select(60, 64, 8, 128, 800)[2] is False and select(60, 64, 8, 128, 700)[2] is True
    assert select(60, 64, 8, 128, 500, mask="planned")[2] is False and select(60, 64, 8, 128, 300, mask="planned")[2] is True
    # longer sequences are never taken whole where shorter ones are cut, and a plan that knows of a mask takes no more of them whole
    for n, hq, hkv, d, _ in WHOLE + CUT:
        whole = [select(n, hq, hkv, d, kv)[2] for kv in (64, 200, 700, 2000, 6000, 60000)]
        assert whole == sorted(whole, reverse=True), (n, hq, hkv, d, whole)
        masked = [select(n, hq, hkv, d, kv, mask="planned")[2] for kv in (64, 200, 700, 2000, 6000, 60000)]
        assert all(w or not m for w, m in zip(whole, masked)), (n, hq, hkv, d, whole, masked)


def test_sixteen_columns_over_ranges_run_on_the_ring_kernel_over_long_streams_of_four_waves(select):
    def ring(*shape, **kw):
        return select(*shape, ring=True, **kw)
    assert ring(32, 64, 8, 128, 32768, sized=True) == (1, True) and ring(300, 28, 4, 128, 4000, sized=True) == (1, True)
    assert ring(30, 64, 8, 128, 2400, sized=True) == (1, False) and ring(100, 28, 4, 128, 1600, sized=True) == (1, False)
    assert ring(32, 64, 8, 128, 32768, sized=True, mask=True) == (1, False)
    for shape in ((100, 8, 1, 128, 16000), (100, 10, 2, 128, 16000)):  # one or two waves per workgroup
        assert ring(*shape, sized=True) == (1, False) and ring(*shape) == (1, False)
    assert ring(32, 64, 8, 128, 32768) == (1, True) and ring(3, 64, 8, 128, 32768) == (1, False)  # no length given
    assert ring(1, 64, 8, 128, 8192) == (4, True) and ring(3, 8, 8, 64, 8192) == (1, True)
    assert ring(32, 64, 8, 128, 200) == (8, False)  # whole sequences
    assert select(30, 48, 1, 128, 700)[1] == 329 and select(16, 48, 1, 128, 1000)[1] == 256 and select(16, 48, 1, 128, 600)[1] == 256


def test_rows_too_far_apart_for_the_column_kernels_stay_where_they_fit(select):
    """32 rows of a column kernel's block have to lie within 2 GiB, 16 of the quad kernel's."""
    far = 100 << 20
    for n, kv in ((1, 300), (4, 300), (4, 8192), (64, 8192), (64, 200), (2000, 200)):  # whatever the number of sequences and ranges
        kernel, ranges, whole = select(n, 32, 8, 128, kv, stride_s=far)
        assert kernel == QUAD and whole == (ranges == 1), (n, kv)
        kernel, ranges, whole = select(n, 16, 8, 256, kv, stride_s=far, ranges=1)
        assert kernel == QUAD and whole, (n, kv)
        kernel, ranges, whole = select(n, 32, 8, 128, kv, stride_s=far, output_offset=8, ranges=1)
        assert kernel == GENERAL and whole, (n, kv)
        assert select(n, 12, 3, 96, kv, stride_s=30 << 20, ranges=1)[::2] == (MFMA16, True)
        assert select(n, 4, 4, 96, kv, stride_s=far, ranges=1) == select(n, 4, 4, 96, kv, stride_s=far, ranges=1, requested=1)
        # neither the kernel by shape nor another one takes them: refused, as for ever
        assert select(n, 64, 8, 128, kv, stride_s=far)[::2] == ("refused", "strides")
    assert select(4, 32, 8, 128, 8192, stride_s=60 << 20)[0] == MFMA16


def test_scales_that_are_not_positive_run_on_kernels_that_scale_first(select):
    for scale in (-0.3, 0.0, 1e-30, float("nan")):
        for n, hq, hkv, d, kv in [(2, 32, 8, 128, 300), (4, 32, 8, 128, 8192), (64, 32, 8, 128, 200), (2000, 8, 8, 64, 200), (64, 64, 8, 128, 8192),
                                  (64, 64, 8, 128, 200), (3, 14, 2, 64, 900), (64, 48, 1, 128, 200), (30, 12, 3, 96, 200), (8, 24, 2, 256, 300)]:
            for form in (dict(), dict(mask=True), dict(output_offset=8)):
                kernel, ranges, whole = select(n, hq, hkv, d, kv, scale=scale, **form)
                assert kernel in (QUAD, GENERAL) and whole == (ranges == 1), (scale, n, hq, hkv, d, kv, form)
        assert select(64, 64, 8, 128, 8192, scale=scale, requested=3)[::2] == ("refused", "scale")
    assert select(64, 64, 8, 128, 8192, scale=1e-6)[0] == MFMA16


def test_a_single_sequence_is_shared_by_four_waves_up_to_a_length_that_its_kv_heads_set(select):
    for shape, most in (((1, 32, 8, 128, 32768), 32), ((1, 28, 4, 128, 65536), 64), ((1, 8, 1, 128, 262144), 256), ((1, 8, 1, 128, 40000), 256)):
        assert select(*shape)[1] == most and select(*shape, ring=True) == (4, True), shape
    for shape in ((1, 32, 8, 128, 40000), (1, 28, 4, 128, 70000)):
        assert select(*shape)[1] > 256 // shape[2] and select(*shape, ring=True)[0] == 1, shape


def test_ranges_and_requests_keep_their_kernels(select):
    assert select(64, 32, 8, 128, 4096)[::2] == (QUAD, False)
    assert select(64, 32, 8, 128, 4096, mask=True)[::2] == (QUAD, False)
    assert select(64, 32, 8, 128, 4096, output_offset=8)[::2] == (GENERAL, False)
    assert select(64, 8, 8, 64, 4096, mask=True)[::2] == (GENERAL, False)
    assert select(64, 32, 8, 64, 4096, mask=True)[::2] == (MFMA, False)
    assert select(64, 64, 8, 128, 4096, mask=True)[::2] == (MFMA16, False)
    assert select(64, 48, 1, 128, 4096)[::2] == (MFMA, False)
    assert select(2, 32, 8, 128, 8192, mask=True)[::2] == (MFMA16, False)
    assert select(512, 32, 8, 128, 300, requested=2)[0] == QUAD
    assert select(512, 32, 8, 128, 300, requested=2, output_offset=8)[::2] == ("refused", "quad-buffers")
    assert select(512, 32, 8, 128, 300, requested=1)[0] == GENERAL
