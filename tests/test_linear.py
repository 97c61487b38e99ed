"""The output projection behind the attention (single-rank row_parallel_linear,
src/ppl/kernel/llm/cuda/pmx/row_parallel_linear.cu:25-110): output = input * weight^T + bias, half tensors, float32
accumulation.  CPU: the oracle against numpy in binary64, exact cases and invariants.  GPU: the HIP kernel against
the oracle through the C ABI.

Tolerance of the GPU result against the oracle: both accumulate in float32 and round once to half, in different
orders, so they differ by at most one half ulp of the result plus the float32 accumulation noise:
|got - ref| <= 2^-10 |ref| + 2e-6 * sum_k |a_k w_k|."""
import numpy as np
import pytest


def draw(rng, m, n, k, outliers=True):
    a = rng.standard_normal((m, k), dtype=np.float32)
    if outliers:
        a[:, rng.choice(k, size=max(1, k // 50), replace=False)] *= 10.0
    w = (rng.standard_normal((n, k), dtype=np.float32) / np.sqrt(k)).astype(np.float16)
    b = rng.standard_normal(n, dtype=np.float32).astype(np.float16)
    return a.astype(np.float16), w, b


def assert_close(got, a, w, b, what):
    ref = a.astype(np.float64) @ w.astype(np.float64).T + (0 if b is None else b.astype(np.float64))
    mag = np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)).T
    err = np.abs(got.astype(np.float64) - ref)
    tol = 2.0 ** -10 * np.abs(ref) + 2e-6 * mag + 1e-7
    assert (err <= tol).all(), "%s: %d of %d outside tolerance, worst %g over %g" % (
        what, int((err > tol).sum()), err.size, float((err - tol).max()), float(tol.flat[np.argmax(err - tol)]))


def test_oracle_matches_numpy_float64(oracle):
    rng = np.random.default_rng(11)
    for m, n, k in ((5, 16, 32), (33, 48, 96), (128, 64, 512)):
        a, w, b = draw(rng, m, n, k)
        assert_close(oracle.row_parallel_linear(a, w, b), a, w, b, "oracle %s" % ((m, n, k),))
        assert_close(oracle.row_parallel_linear(a, w, None), a, w, None, "oracle, no bias")


def test_oracle_exact_cases(oracle):
    rng = np.random.default_rng(12)
    # small integers: every product and sum is exact in float32 and in half
    a = rng.integers(-3, 4, (7, 64)).astype(np.float16)
    w = rng.integers(-2, 3, (32, 64)).astype(np.float16)
    b = rng.integers(-5, 6, 32).astype(np.float16)
    want = a.astype(np.int64) @ w.astype(np.int64).T + b.astype(np.int64)
    assert np.array_equal(oracle.row_parallel_linear(a, w, b).astype(np.int64), want)
    # identity weight copies the input; a zero input leaves the bias
    x = rng.standard_normal((9, 32)).astype(np.float16)
    eye = np.eye(32, dtype=np.float16)
    assert np.array_equal(oracle.row_parallel_linear(x, eye), x)
    assert np.array_equal(oracle.row_parallel_linear(np.zeros_like(x), eye, b), np.tile(b, (9, 1)))
    # a transposed operand or swapped indices would fail this one: weight rows select single input channels
    sel = np.zeros((16, 32), dtype=np.float16)
    cols = rng.choice(32, size=16, replace=False)
    sel[np.arange(16), cols] = 1
    assert np.array_equal(oracle.row_parallel_linear(x, sel), x[:, cols])
    # linear in the input (exactly, for power-of-two factors)
    a2, w2, _ = draw(rng, 6, 16, 64)
    assert np.array_equal(oracle.row_parallel_linear(a2 * np.float16(2), w2), oracle.row_parallel_linear(a2, w2) * np.float16(2))


def test_c_entry_point_rejects_bad_arguments_without_launching(pkg, hip_lib):
    f = hip_lib.pmxhip_row_parallel_linear
    assert f(None, 16, 16, None, 0, 32, 16, 32, 32, 16, 0, None, 16) == 0            # no rows: nothing to do
    assert f(None, 16, 16, None, 4, 32, 24, 32, 32, 24, 0, None, 16) == 2            # out_features % 16
    assert f(None, 16, 16, None, 4, 40, 16, 40, 40, 16, 0, None, 16) == 2            # in_features % 32
    assert f(None, None, 16, None, 4, 32, 16, 32, 32, 16, 0, None, 16) == 4          # null input
    assert f(None, 16, 16, None, 4, 32, 16, 16, 32, 16, 0, None, 16) == 4            # input stride shorter than a row
    assert f(None, 24, 16, None, 4, 32, 16, 32, 32, 16, 0, None, 16) == 2            # input not 16-byte aligned
    assert f(None, 16, 16, None, -1, 32, 16, 32, 32, 16, 0, None, 16) == 4


def test_k_ranges_are_worth_their_workspace(pkg, hip_lib):
    """Whatever the shape, a call asks for at most 256 MiB of partial tiles, and prompts whose tiles fill the chip for none: more
    than 32 MiB have to be estimated 5 % faster.  With less workspace the plan has fewer ranges, never more than fit."""
    plan = pkg.ops.row_parallel_linear_plan
    assert plan(3472, 14336, 14336, cus=256).workspace_size == 0  # 784 tiles of 256 x 256: 1360.2 against 1360.6 us
    assert plan(2187, 14336, 4096, cus=256).workspace_size == 0
    assert 0 < plan(33, 8192, 8192, cus=256).workspace_size <= 32 << 20
    splits = 0
    for k, n in [(2048, 2048), (4096, 4096), (8192, 8192), (14336, 4096), (4096, 14336), (14336, 14336), (28672, 8192), (8192, 28672),
                 (1024, 8192), (4128, 4112)]:
        for m in sorted({int(2 ** (e / 6)) for e in range(90)} | {5110, 4603}):
            p = plan(m, k, n, cus=256)
            assert p.workspace_size == (p.k_ranges * m * n * 4 if p.k_ranges > 1 else 0) and p.workspace_size <= 1 << 28, (m, k, n)
            assert p.k_ranges in (1, 2, 4) and k % (64 if p.kernel == pkg._lib.LINEAR_KERNEL_STREAM else 32) == 0
            assert plan(m, k, n, workspace_size=0, cus=256).k_ranges == 1
            if p.k_ranges > 1:
                splits += 1
                same = plan(m, k, n, workspace_size=p.workspace_size, cus=256)
                assert (same.kernel, same.tile_n, same.tile_m, same.k_ranges) == (p.kernel, p.tile_n, p.tile_m, p.k_ranges)
                less = plan(m, k, n, workspace_size=p.workspace_size - 1, cus=256)
                assert less.workspace_size < p.workspace_size
    assert splits > 50


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 16, 32), (7, 48, 96), (128, 4096, 4096), (64, 1024, 8192), (200, 256, 512),
                                   (128, 14336 // 8, 4096), (3, 4096, 32), (129, 32, 4064), (17, 64, 64), (128, 128, 3136),
                                   (300, 8192, 1024), (5, 64, 2240), (1, 64, 512), (16, 128, 1024), (17, 64, 1536), (33, 192, 2048),
                                   (65, 64, 512), (130, 192, 2048), (240, 4096, 4096),
                                   # many rows (a prefill chunk's)
                                   (384, 256, 512), (1000, 512, 1024), (2500, 1024, 2048), (640, 4096, 4096)])
def test_hip_linear_matches_oracle(pkg, oracle, shape, vendor_gemm=False):
    import torch
    m, n, k = shape
    rng = np.random.default_rng(100 + m + n)
    a, w, b = draw(rng, m, n, k)
    da, dw, db = (torch.from_numpy(x).cuda() for x in (a, w, b))
    ws_bytes = pkg.ops.row_parallel_linear_workspace_size(m, k, n, vendor_gemm=vendor_gemm)
    for bias, with_ws in ((db, True), (None, True), (db, False)):  # with the k-split's workspace and without
        out = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda") if with_ws and ws_bytes else None
        pkg.ops.row_parallel_linear(da, dw, bias, out, workspace=ws, vendor_gemm=vendor_gemm)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert_close(got, a, w, b if bias is not None else None, "hip %s" % (shape,))
        if m * n * k <= 1 << 26:  # the oracle's triple loop, where it finishes in seconds
            # against the oracle's own half result: one rounding to half on either side plus two float32
            # accumulations in different orders (where sums cancel, an ulp of the small result is far below that noise)
            ref = oracle.row_parallel_linear(a, w, b if bias is not None else None).astype(np.float64)
            mag = np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)).T
            assert (np.abs(got.astype(np.float64) - ref) <= 2.0 ** -10 * np.abs(ref) + 4e-6 * mag + 1e-7).all()
    if vendor_gemm:
        return
    # twice the same call: the partial tiles are added in a fixed order
    out2 = torch.empty_like(out)
    pkg.ops.row_parallel_linear(da, dw, db, out2)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), out2.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(384, 256, 512), (1000, 512, 1024), (2500, 1024, 2048), (200, 256, 512)])
def test_hip_linear_vendor_gemm_on_request(pkg, oracle, shape):
    """PMXHIP_LINEAR_VENDOR_GEMM: from 384 rows on the GEMM goes to hipBLASLt where that loads (below, and where it
    does not, the flag changes nothing); same tolerance against the oracle."""
    if not pkg.ops.vendor_gemm_available():
        pytest.skip("hipBLASLt cannot be loaded on this box")
    test_hip_linear_matches_oracle(pkg, oracle, shape, vendor_gemm=True)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [37, 700])
def test_hip_linear_strided_rows_and_attention_hand_off(pkg, oracle, m):
    """Rows with padding between them (the strides of the C ABI), and the attention output (B, Hq, D) used in place
    as the (B, Hq * D) input; a decode-sized and a prefill-sized row count."""
    import torch
    rng = np.random.default_rng(7)
    hq, d, n = 8, 64, 128
    k = hq * d
    a, w, b = draw(rng, m, n, k)
    buf_in = torch.zeros((m, k + 64), dtype=torch.float16, device="cuda")
    buf_in[:, :k] = torch.from_numpy(a).cuda()
    buf_out = torch.full((m, n + 32), float("nan"), dtype=torch.float16, device="cuda")
    pkg.ops.row_parallel_linear(buf_in[:, :k], torch.from_numpy(w).cuda(), torch.from_numpy(b).cuda(), buf_out[:, :n])
    torch.cuda.synchronize()
    assert_close(buf_out[:, :n].cpu().numpy(), a, w, b, "strided")
    assert torch.isnan(buf_out[:, n:]).all()
    attn = torch.from_numpy(a).cuda().view(m, hq, d)  # the decode output as the operator writes it
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    pkg.ops.row_parallel_linear(attn, torch.from_numpy(w).cuda(), None, out)
    torch.cuda.synchronize()
    assert_close(out.cpu().numpy(), a, w, None, "attention output in place")


# (M, N, K) and the kernel (1 = stream, 2 = tile), tile (columns, rows) and k ranges that serve it with a workspace on 256 CUs: one
# for every tile, with rows, columns and k that are no multiples of it; every tile that takes several k ranges, with a
# number of pipeline stages that the ranges do not divide; weights that carry the non-temporal hint
PLANS = [
    ((5, 8208, 4160), (1, 16, 16, 1)), ((33, 2064, 4160), (1, 32, 32, 1)), ((37, 4112, 4096), (1, 32, 64, 1)),
    ((129, 4112, 4160), (1, 64, 64, 1)),                                     # 65 k pieces for four waves
    ((129, 4112, 576), (2, 64, 64, 1)), ((333, 4112, 1056), (2, 128, 64, 1)), ((1000, 2576, 4128), (2, 128, 128, 1)),
    ((640, 4112, 14368), (2, 256, 256, 4)), ((2049, 4112, 1056), (2, 256, 256, 1)),
    ((16, 1024, 8256), (1, 16, 16, 4)), ((20, 4096, 14400), (1, 32, 32, 2)), ((40, 4096, 14400), (1, 64, 64, 4)),
    ((80, 4096, 14400), (1, 64, 64, 2)), ((129, 32, 4064), (2, 64, 64, 4)), ((70, 2064, 8224), (2, 128, 64, 4)),
    ((600, 2064, 8224), (2, 128, 128, 2)), ((200, 4112, 8224), (2, 256, 128, 4)),
    ((257, 4112, 14336), (2, 256, 128, 4)),
]


@pytest.mark.parametrize("shape,want", PLANS)
def test_plan_of_the_tile_edges(pkg, hip_lib, shape, want):
    """Changed constants would move these shapes to other kernels, and the test below with them."""
    m, n, k = shape
    p = pkg.ops.row_parallel_linear_plan(m, k, n, cus=256)
    assert (p.kernel, p.tile_n, p.tile_m, p.k_ranges) == want


@pytest.mark.parametrize("shape,kernel", [((1, 2064, 4128), 0), ((16, 2560, 14368), 0), ((17, 2560, 14368), 2), ((16, 2576, 14368), 2),
                                          ((8, 512, 4064), 2), ((8, 512, 8192), 1)])
def test_plan_without_workspace(pkg, hip_lib, shape, kernel):
    """Few long rows of an odd number of 32 k: the 16-column form, at the edges of its rule; with a workspace the k range is split."""
    m, n, k = shape
    assert pkg.ops.row_parallel_linear_plan(m, k, n, workspace_size=0, cus=256).kernel == kernel
    if kernel == 0:
        assert pkg.ops.row_parallel_linear_plan(m, k, n, cus=256).k_ranges > 1


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 2064, 4128), (16, 2560, 14368), (7, 16, 4128)])
def test_hip_linear_few_long_rows(pkg, oracle, shape):
    """... whose sums are the oracle's within the same tolerance, with the workspace and without."""
    test_hip_linear_matches_oracle(pkg, oracle, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,want", PLANS)
def test_hip_linear_tile_edges(pkg, oracle, shape, want):
    """float32 sums in another order than the oracle's and one rounding to half, as above; and the partial tiles of several k
    ranges are added in a fixed order: the same call twice gives the same bits."""
    import torch
    m, n, k = shape
    p = pkg.ops.row_parallel_linear_plan(m, k, n)
    assert (p.kernel, p.tile_n, p.tile_m, p.k_ranges) == want
    test_hip_linear_matches_oracle(pkg, oracle, shape)
    if p.k_ranges > 1:
        rng = np.random.default_rng(m)
        a, w, b = (torch.from_numpy(x).cuda() for x in draw(rng, m, n, k))
        outs = []
        for fill in (float("nan"), 1.0):
            ws = torch.full((p.workspace_size // 4,), fill, dtype=torch.float32, device="cuda")
            outs.append(torch.empty((m, n), dtype=torch.float16, device="cuda"))
            pkg.ops.row_parallel_linear(a, w, b, outs[-1], workspace=ws)
            torch.cuda.synchronize()
            assert not (ws == 1.0).all() and not torch.isnan(ws).all()  # the partial tiles went through it
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 700])
def test_hip_linear_rows_far_apart_and_output_rows_on_8_bytes(pkg, m):
    """Weight rows 2^23 halves apart (beyond the 32-bit row offsets of the tile kernels), and output rows that start on
    8-byte addresses only."""
    import torch
    rng = np.random.default_rng(m)
    n, k = 48, 64
    a, w, b = draw(rng, m, n, k)
    far = torch.zeros((n, 1 << 23), dtype=torch.float16, device="cuda")
    far[:, :k] = torch.from_numpy(w).cuda()
    for weight, bias in ((far[:, :k], b), (torch.from_numpy(w).cuda(), None)):
        out = torch.full((m, n + 4), float("nan"), dtype=torch.float16, device="cuda")
        pkg.ops.row_parallel_linear(torch.from_numpy(a).cuda(), weight, None if bias is None else torch.from_numpy(bias).cuda(), out[:, :n])
        torch.cuda.synchronize()
        assert_close(out[:, :n].cpu().numpy(), a, w, bias, "far rows" if bias is not None else "8-byte rows")
        assert torch.isnan(out[:, n:]).all()
