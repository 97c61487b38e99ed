"""Host-side checks that need no GPU: the C-ABI library loads and exports every
symbol the header declares, heuristic_prepare validates and derives what the
reference's does (utils.cu:68-131, 162-165, 210-214, 318-324), and the split plan
is sized consistently.  No kernel is launched."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "pmx_hip", "c_api.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"PMXHIP_API\s+[\w\s\*]+?\b(pmxhip_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol(pkg, hip_lib):
    names = declared_symbols()
    assert len(names) >= 17
    for n in names:
        assert hasattr(hip_lib, n), n
    assert sorted(pkg._lib.EXPORTED_SYMBOLS) == names
    assert b"gfx950" in hip_lib.pmxhip_version()


def test_python_structures_follow_the_header(pkg):
    """Every ctypes structure has the header's fields in the header's order and types (some are filled by position)."""
    L = pkg._lib
    text = open(os.path.join(ROOT, "include", "pmx_hip", "c_api.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    kinds = {"int64_t": L.c_i64, "int32_t": L.c_i32, "float": L.c_f32, "pmxhip_tensor_shape": L.TensorShape}
    classes = dict(kvstore_params=L.KvstoreParams, decode_params=L.DecodeParams, decode_plan=L.DecodePlan, prefill_params=L.PrefillParams,
                   tensor_shape=L.TensorShape, mhca_prepare_args=L.MhcaPrepareArgs, mhca_derived=L.MhcaDerived,
                   reorder_stride=L.ReorderStride, rope_params=L.RopeParams, linear_plan=L.LinearPlan)
    bodies = dict(re.findall(r"typedef struct pmxhip_(\w+) \{(.*?)\} pmxhip_\1;", text, flags=re.S))
    assert sorted(bodies) == sorted(classes)
    for name, cls in classes.items():
        want = []
        for decl in filter(None, (d.strip() for d in bodies[name].split(";"))):
            kind, rest = re.match(r"(?:const )?(\w+)\s*(.*)", decl, flags=re.S).groups()
            for field in rest.split(","):
                field = field.strip()
                array = re.match(r"(\w+)\[(\d+)\]$", field)
                if field.startswith("*"):
                    want.append((field.lstrip("* "), L.c_vp))
                elif array:
                    want.append((array.group(1), kinds[kind] * int(array.group(2))))
                else:
                    want.append((field, kinds[kind]))
        assert [tuple(f) for f in cls._fields_] == want, name


def base_args(**over):
    kw = dict(query_shape=(6, 32, 128), current_key_shape=(6, 8, 128), current_value_shape=(6, 8, 128),
              output_shape=(6, 32, 128), batch=6, decoding_batches=6, max_seqlen=1, max_kvlen=4096, layer_idx=0,
              num_layer=1, num_heads=32, num_kv_heads=8, head_dim=128, cache_mode=1, page_size=128,
              cache_stride_s=1024, cache_stride_l=2 * 1024 * 4096, cache_stride_h=128, cache_stride_kv=1024 * 4096,
              cachestarts_stride_b=32, compute_units_override=256)
    kw.update(over)
    return kw


def prepare(pkg, **over):
    op = pkg.ops.DynamicBatchingMultiHeadCacheAttention()
    return op, op.heuristic_prepare(**base_args(**over))


def test_prepare_derives_the_reference_values(pkg, hip_lib):
    op, rc = prepare(pkg)
    assert rc == pkg.ops.RC_SUCCESS
    c = op.cfg
    assert c.prefill_batches == 0
    assert (c.q_stride_s, c.k_stride_s, c.v_stride_s, c.o_stride_s) == (4096, 1024, 1024, 4096)
    assert c.num_kv_repeats == 4
    import numpy as np
    assert c.attn_scale == float(np.float32(1.0 / np.sqrt(np.float32(128))))
    assert c.decoding_algo == 3  # INFINITY_GQCA is what the reference would name for G = 4
    assert c.decoding_multi_block_counter_size == 0
    assert c.workspace_size == c.decoding_multi_block_partial_out_size + c.decoding_multi_block_partial_log_sum_exp_size
    # mask strides: 3-d and 2-d masks (utils.cu:117-126)
    op, rc = prepare(pkg, attn_mask=1 << 20, attn_mask_shape=(32, 6, 4104))
    assert rc == 0 and (op.cfg.mask_stride_h, op.cfg.mask_stride_s) == (6 * 4104, 4104)
    op, rc = prepare(pkg, attn_mask=1 << 20, attn_mask_shape=(6, 4104))
    assert rc == 0 and (op.cfg.mask_stride_h, op.cfg.mask_stride_s) == (0, 4104)
    op, rc = prepare(pkg, batch=9, decoding_batches=6)
    assert rc == 0 and op.cfg.prefill_batches == 3


@pytest.mark.parametrize("over,code", [
    (dict(query_shape=(6, 31, 128)), 2),          # leading dim on query heads
    (dict(output_shape=(6, 16, 128)), 2),
    (dict(current_key_shape=(6, 4, 128)), 2),
    (dict(current_value_shape=(6, 4, 128)), 2),
    (dict(page_size=64), 2),                      # paged mode needs 128-token pages
    (dict(num_heads=30, query_shape=(6, 30, 128), output_shape=(6, 30, 128)), 2),  # 30 % 8 != 0
    (dict(attn_mask=1 << 20, attn_mask_shape=(4104,)), 2),        # mask must be 2-d or 3-d
    (dict(attn_mask=1 << 20, attn_mask_shape=(6, 4100)), 2),      # last dim % 8
    (dict(specify_decoding_multi_block=3), 4),
    (dict(specify_decoding_multi_block=-1), 4),
    (dict(specify_decoding_tpb=128), 4),
    (dict(enable_sharemem_mhca=False, enable_infinity_mhca=False, enable_infinity_gqca=False), 1),  # no algorithm
    # prefill sequences at a head_dim the prefill stage does not have: refused before anything is enqueued
    (dict(batch=9, decoding_batches=6, max_seqlen=40, head_dim=80, query_shape=(90, 32, 80),
          current_key_shape=(90, 8, 80), current_value_shape=(90, 8, 80), output_shape=(90, 32, 80)), 2),
    (dict(batch=9, decoding_batches=6, max_seqlen=40, head_dim=32, query_shape=(90, 32, 32),
          current_key_shape=(90, 8, 32), current_value_shape=(90, 8, 32), output_shape=(90, 32, 32)), 2),
])
def test_prepare_error_branches(pkg, hip_lib, over, code):
    _, rc = prepare(pkg, **over)
    assert rc == code


def test_prepare_accepts_what_the_reference_accepts(pkg, hip_lib):
    for over in (dict(specify_decoding_tpb=256), dict(specify_decoding_tpb=512), dict(cache_mode=0, page_size=0),
                 dict(enable_infinity_gqca=False), dict(enable_sharemem_mhca=False),
                 dict(specify_decoding_multi_block=0), dict(specify_decoding_multi_block=2),
                 # decode-only batches take every head_dim of the decode kernels
                 dict(head_dim=256, query_shape=(6, 32, 256), current_key_shape=(6, 8, 256),
                      current_value_shape=(6, 8, 256), output_shape=(6, 32, 256)),
                 dict(head_dim=96, query_shape=(6, 32, 96), current_key_shape=(6, 8, 96),
                      current_value_shape=(6, 8, 96), output_shape=(6, 32, 96)),
                 # and batches with prefill sequences the four head dims of the reference's flash attention
                 dict(batch=9, decoding_batches=6, max_seqlen=40, head_dim=256, query_shape=(90, 32, 256),
                      current_key_shape=(90, 8, 256), current_value_shape=(90, 8, 256), output_shape=(90, 32, 256)),
                 dict(batch=9, decoding_batches=6, max_seqlen=40, head_dim=96, query_shape=(90, 32, 96),
                      current_key_shape=(90, 8, 96), current_value_shape=(90, 8, 96), output_shape=(90, 32, 96))):
        op, rc = prepare(pkg, **over)
        assert rc == 0, over
    op, _ = prepare(pkg, specify_decoding_multi_block=0)
    assert op.cfg.decoding_multi_block_size == 1 and op.cfg.workspace_size == 0
    op, _ = prepare(pkg, enable_infinity_gqca=False)
    assert op.cfg.decoding_algo == 1  # SHAREMEM_MHCA
    op, _ = prepare(pkg, enable_infinity_gqca=False, enable_sharemem_mhca=False)
    assert op.cfg.decoding_algo == 2  # INFINITY_MHCA


def test_forward_before_prepare_is_rejected(pkg, hip_lib):
    import ctypes
    h = hip_lib.pmxhip_mhca_create()
    try:
        assert hip_lib.pmxhip_mhca_set_workspace(h, None) == 4
        d = pkg._lib.MhcaDerived()
        assert hip_lib.pmxhip_mhca_get_derived(h, ctypes.byref(d)) == 4
    finally:
        hip_lib.pmxhip_mhca_destroy(h)


def test_decode_plan(pkg, hip_lib):
    plan = pkg.ops.decode_plan(128, 32, 8, 128, 8192, cus=256)
    assert plan.kv_heads_per_group == 8 and plan.q_heads_per_pass == 4 and plan.num_passes == 1
    assert plan.num_token_ranges == 256  # the quad kernel: a long stream is cut for one wave per SIMD
    pieces = plan.num_token_ranges + 128
    assert plan.partial_out_size == pieces * 32 * 128 * 4 and plan.partial_ml_size == pieces * 32 * 2 * 4
    plan = pkg.ops.decode_plan(64, 32, 32, 128, 4096, cus=256)  # MHA: 4 groups of 8 kv heads
    assert plan.kv_heads_per_group == 8 and plan.q_heads_per_pass == 1 and plan.num_token_ranges == 64
    plan = pkg.ops.decode_plan(32, 64, 8, 128, 32768, cus=256)  # G = 8: MFMA kernel, 4 kv heads per workgroup, 16 columns
    assert plan.q_heads_per_pass == 16 and plan.num_passes == 1 and plan.kv_heads_per_group == 4
    assert plan.num_token_ranges == 256
    plan = pkg.ops.decode_plan(64, 8, 1, 128, 8192, cus=256)  # one kv head: one wave per workgroup, eight workgroups per CU
    assert plan.q_heads_per_pass == 16 and plan.kv_heads_per_group == 1 and plan.num_token_ranges == 2048
    plan = pkg.ops.decode_plan(64, 16, 2, 128, 8192, cus=256)
    assert plan.q_heads_per_pass == 16 and plan.kv_heads_per_group == 2 and plan.num_token_ranges == 1024
    plan = pkg.ops.decode_plan(64, 16, 4, 128, 8192, cus=256)  # four kv heads: two waves per workgroup, four workgroups per CU
    assert plan.q_heads_per_pass == 4 and plan.kv_heads_per_group == 4 and plan.num_token_ranges == 1024
    plan = pkg.ops.decode_plan(4, 48, 3, 64, 512, cus=256)  # G = 16 at head_dim 64: 32 MFMA columns; 3 kv heads -> 1 per group
    assert plan.q_heads_per_pass == 32 and plan.num_passes == 1 and plan.kv_heads_per_group == 1
    plan = pkg.ops.decode_plan(4, 48, 3, 64, 512, cus=256, kernel=pkg._lib.DECODE_KERNEL_GENERAL)  # -> two passes of 8
    assert plan.q_heads_per_pass == 8 and plan.num_passes == 2 and plan.kv_heads_per_group == 1
    plan = pkg.ops.decode_plan(1, 8, 8, 64, 30, cus=256)    # tiny: one range, no workspace
    assert plan.num_token_ranges == 1 and plan.workspace_size == 0
    plan = pkg.ops.decode_plan(4, 8, 8, 64, 512, cus=256, ranges_hint=7)
    assert plan.num_token_ranges == 7
    with pytest.raises(pkg.ops.PmxError):
        pkg.ops.decode_plan(4, 8, 8, 80, 512, cus=256)  # head_dim 80
    with pytest.raises(pkg.ops.PmxError):
        pkg.ops.decode_plan(4, 9, 8, 64, 512, cus=256)


def test_decode_plan_names_its_kernel(pkg, hip_lib):
    """The plan reports the token-range kernel it was made for, and a requested kernel is honoured or refused."""
    L = pkg._lib
    auto = {(32, 8, 128): L.DECODE_KERNEL_QUAD, (32, 32, 128): L.DECODE_KERNEL_QUAD, (64, 8, 128): L.DECODE_KERNEL_MFMA16,
            (96, 4, 128): L.DECODE_KERNEL_MFMA32, (9, 3, 128): L.DECODE_KERNEL_QUAD, (6, 3, 128): L.DECODE_KERNEL_QUAD, (3, 1, 128): L.DECODE_KERNEL_MFMA16,
            (5, 5, 128): L.DECODE_KERNEL_QUAD, (2, 1, 128): L.DECODE_KERNEL_GENERAL, (3, 1, 64): L.DECODE_KERNEL_MFMA32,
            (8, 8, 64): L.DECODE_KERNEL_QUAD, (32, 8, 64): L.DECODE_KERNEL_QUAD, (40, 8, 64): L.DECODE_KERNEL_MFMA32,
            (9, 3, 64): L.DECODE_KERNEL_QUAD, (12, 4, 96): L.DECODE_KERNEL_GENERAL, (16, 16, 256): L.DECODE_KERNEL_QUAD,
            (40, 8, 256): L.DECODE_KERNEL_QUAD, (8, 1, 256): L.DECODE_KERNEL_QUAD, (72, 8, 256): L.DECODE_KERNEL_GENERAL, (66, 2, 128): L.DECODE_KERNEL_MFMA32, (48, 1, 128): L.DECODE_KERNEL_MFMA32,
            (71, 1, 64): L.DECODE_KERNEL_MFMA32, (2, 1, 64): L.DECODE_KERNEL_GENERAL}
    for (hq, hkv, d), want in auto.items():
        assert pkg.ops.decode_plan(16, hq, hkv, d, 4096, cus=256).kernel == want, (hq, hkv, d)
    # more than 32 query heads per kv head: passes of 32 columns (multi-query models)
    for (hq, hkv, d), passes in {(48, 1, 128): 2, (71, 1, 64): 3, (66, 2, 128): 2, (128, 4, 128): 1, (128, 8, 64): 1}.items():
        plan = pkg.ops.decode_plan(16, hq, hkv, d, 4096, cus=256)
        assert (plan.kernel, plan.q_heads_per_pass, plan.num_passes) == (L.DECODE_KERNEL_MFMA32, 32, passes), (hq, hkv, d)
    # requests: every kernel on the Llama-3-70B shape (8 query heads per kv head, kv heads in eights)
    for k, (kvhb, gt, ranges) in {L.DECODE_KERNEL_GENERAL: (8, 8, 512), L.DECODE_KERNEL_QUAD: (8, 8, 256),
                                  L.DECODE_KERNEL_MFMA16: (4, 16, 256), L.DECODE_KERNEL_MFMA32: (4, 32, 256)}.items():
        plan = pkg.ops.decode_plan(32, 64, 8, 128, 32768, cus=256, kernel=k)
        assert (plan.kernel, plan.kv_heads_per_group, plan.q_heads_per_pass, plan.num_token_ranges) == (k, kvhb, gt, ranges)
    for hq, hkv, d, k in [(40, 8, 64, L.DECODE_KERNEL_QUAD), (32, 8, 96, L.DECODE_KERNEL_QUAD), (32, 8, 64, L.DECODE_KERNEL_MFMA16),
                          (40, 2, 128, L.DECODE_KERNEL_MFMA16), (32, 8, 96, L.DECODE_KERNEL_MFMA32), (16, 4, 256, L.DECODE_KERNEL_MFMA32),
                          (10, 2, 128, L.DECODE_KERNEL_QUAD), (2, 1, 128, L.DECODE_KERNEL_QUAD), (32, 8, 128, 5), (32, 8, 128, -1)]:
        with pytest.raises(pkg.ops.PmxError):
            pkg.ops.decode_plan(16, hq, hkv, d, 4096, cus=256, kernel=k)


def test_decode_plan_takes_short_sequences_whole(pkg, hip_lib):
    """Batches of short sequences need no ranges (and so no workspace); long ones, and requested kernels, are cut as before."""
    L = pkg._lib
    for n, hq, hkv, d, kv in [(32, 32, 8, 128, 256), (4, 32, 8, 128, 256), (64, 14, 2, 64, 256), (448, 8, 1, 256, 148), (12, 32, 8, 64, 553)]:
        plan = pkg.ops.decode_plan(n, hq, hkv, d, kv, cus=256)
        assert plan.num_token_ranges == 1 and plan.workspace_size == 0, (n, hq, hkv, d, kv)
        assert pkg.ops.decode_plan(n, hq, hkv, d, kv, cus=256, ranges_hint=5).num_token_ranges == 5
    for n, hq, hkv, d, kv in [(64, 32, 8, 128, 4096), (1, 32, 8, 128, 4096), (16, 64, 8, 128, 8192), (8, 16, 8, 256, 8192)]:
        plan = pkg.ops.decode_plan(n, hq, hkv, d, kv, cus=256)
        assert plan.num_token_ranges > 1 and plan.workspace_size > 0, (n, hq, hkv, d, kv)
    assert pkg.ops.decode_plan(32, 32, 8, 128, 256, cus=256, kernel=L.DECODE_KERNEL_QUAD).num_token_ranges > 1
    # a single sequence: at most a workgroup per (range, kv head) on every compute unit
    plan = pkg.ops.decode_plan(1, 32, 8, 128, 32768, cus=256)
    assert plan.num_token_ranges == 32


def test_c_entry_points_reject_bad_arguments_without_launching(pkg, hip_lib):
    """Argument checks run before any device work, so they can be exercised on the host."""
    import ctypes
    L = pkg._lib
    p = L.KvstoreParams()
    p.head_dim = 12
    p.num_kv_heads = 1
    p.batch = 1
    p.max_seqlen = 1
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 2  # head_dim % 8 (kernel.cu:2040)
    p.head_dim = 64
    p.cache_mode = 2
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 2  # invalid cache_mode (kernel.cu:2050)
    p.cache_mode = 1
    p.page_size = 64
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 2
    p.page_size = 128
    p.cache_stride_s = 12
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 2  # strides % 8
    p.cache_stride_s = 64
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 4  # null pointers
    p.batch = 0
    assert hip_lib.pmxhip_kv_cache_quantize(ctypes.byref(p), None) == 0  # nothing to do
    assert hip_lib.pmxhip_kv_cache_quantize(None, None) == 4

    d = L.DecodeParams()
    assert hip_lib.pmxhip_decode_attention(ctypes.byref(d), None) == 0  # no decode sequences (kernel.cu:2084)
    d.decoding_batches = 2
    d.head_dim = 80
    assert hip_lib.pmxhip_decode_attention(ctypes.byref(d), None) == 2
    d.head_dim = 128
    d.num_heads, d.num_kv_heads, d.num_kv_repeats = 8, 3, 2
    assert hip_lib.pmxhip_decode_attention(ctypes.byref(d), None) == 2
    d.num_heads, d.num_kv_heads, d.num_kv_repeats = 8, 2, 4
    d.cache_mode = 3
    assert hip_lib.pmxhip_decode_attention(ctypes.byref(d), None) == 2
    d.cache_mode = 0
    assert hip_lib.pmxhip_decode_attention(ctypes.byref(d), None) == 4  # null pointers
    assert b"null" in hip_lib.pmxhip_last_error()

    f = L.PrefillParams()
    f.batch, f.decoding_batches = 2, 3
    assert hip_lib.pmxhip_prefill_attention(ctypes.byref(f), None) == 4
    f.batch, f.decoding_batches = 3, 3
    assert hip_lib.pmxhip_prefill_attention(ctypes.byref(f), None) == 0  # no prefill sequences (kernel.cu:2130)
    f.batch, f.max_seqlen, f.head_dim = 4, 8, 96
    assert hip_lib.pmxhip_prefill_attention(ctypes.byref(f), None) == 2


def test_prefill_parts_lie_behind_the_decode_pieces(pkg, hip_lib):
    """The operator's workspace: the decode stage's pieces, then -- where the query tiles are split over their kv tokens -- the
    parts, so that the two stages may run side by side."""
    rows, kvlen = 1200, 1900
    over = dict(batch=4, decoding_batches=3, max_seqlen=rows, max_kvlen=kvlen, query_shape=(rows + 3, 8, 128), num_heads=8,
                current_key_shape=(rows + 3, 8, 128), current_value_shape=(rows + 3, 8, 128), output_shape=(rows + 3, 8, 128))
    plan = pkg.ops.decode_plan(3, 8, 8, 128, kvlen, cus=256)
    split = pkg.ops.prefill_split_workspace_size(4, 3, rows, kvlen, rows, 8, 8, 128, cus=256)
    assert plan.workspace_size > 0 and split > 0
    op, rc = prepare(pkg, **over)
    assert rc == 0 and op.cfg.workspace_size == (plan.workspace_size + 255) // 256 * 256 + split
    op, rc = prepare(pkg, specify_decoding_multi_block=0, **over)
    assert rc == 0 and op.cfg.workspace_size == 0


def mixed_args(q_lens, max_kvlen, hq=32, hkv=8, d=128, decodes=3):
    rows = int(sum(q_lens)) + decodes
    return dict(batch=len(q_lens) + decodes, decoding_batches=decodes, max_seqlen=int(max(q_lens)), max_kvlen=max_kvlen, num_heads=hq,
                num_kv_heads=hkv, head_dim=d, query_shape=(rows, hq, d), current_key_shape=(rows, hkv, d),
                current_value_shape=(rows, hkv, d), output_shape=(rows, hq, d))


def test_short_prompts_beside_long_decode_sequences_are_not_split(pkg, hip_lib):
    """max_kvlen may be a decode sequence's: alone it asks for no workspace (and no second launch) for the prompts.  Their own
    length, where the caller gives it, does."""
    args = mixed_args([70], 4096)
    pieces = pkg.ops.decode_plan(3, 32, 8, 128, 4096, cus=256).workspace_size
    op, rc = prepare(pkg, **args)
    assert rc == 0 and op.cfg.workspace_size == pieces
    op, rc = prepare(pkg, prefill_max_kvlen=70, **args)
    assert rc == 0 and op.cfg.workspace_size == pieces
    op, rc = prepare(pkg, prefill_max_kvlen=3000, **args)
    assert rc == 0 and op.cfg.workspace_size > pieces + (1 << 20)


def test_unknown_history_is_split_only_where_the_kernels_agree(pkg, hip_lib):
    """The rule of split_stream in csrc/prefill_attn.hip, in numpy: whatever the prompts' history, a batch that the host splits
    beside decode sequences without knowing it is split by the kernels (else the second launch is for nothing)."""
    import numpy as np
    rng = np.random.default_rng(21)
    split = 0
    for _ in range(4000):
        hkv = int(rng.choice([1, 2, 4, 8, 16]))
        hq = hkv * int(rng.choice([1, 2, 4, 8]))
        d = int(rng.choice([64, 96, 128, 256]))
        cols = 128 if d == 256 else 256
        ppw, ranges = cols // (hq // hkv), 256 // hkv
        q = rng.integers(1, int(rng.choice([100, 1000, 4000])), size=int(rng.integers(1, 12)))
        prior = rng.integers(0, int(rng.choice([1, 300, 8000])) + 1, size=len(q))
        size = pkg.ops.prefill_split_workspace_size(len(q) + 1, 1, int(q.max()), 0, int(q.sum()), hq, hkv, d, cus=256)
        if size == 0:
            continue
        split += 1
        for causal in (True, False):
            step, base = (ppw, prior) if causal else (0, prior + q)
            tiles = -(-q // ppw)
            total = int((tiles * (64 + base) + step * (tiles * (tiles + 1) // 2)).sum())
            per = max(-(-total // ranges), 192)
            assert int((64 + base + step * tiles).max()) - per >= 512, (q, prior, hq, hkv, d, causal)
    assert split > 100


def test_calls_take_tensors_with_dimensions_of_one_behind_the_row(pkg, hip_lib, monkeypatch):
    """A query of (rows, heads, head_dim, 1) and a weight of (out, in, 1) are the same rows."""
    import torch
    monkeypatch.setattr(pkg.ops, "_ptr", lambda t: 16 if t is not None else None)
    monkeypatch.setattr(pkg.ops, "_stream", lambda stream=None: None)
    rows = torch.empty((0, 4, 64, 1), dtype=torch.float16)
    pkg.ops.rotary_position_embedding(rows, rows, rows, rows, rows, rows, theta=1e4, rotary_dim=64, batch=0, max_seqlen=0)
    p = pkg.ops._rope_params(rows, rows[:, :2], rows, rows, rows, rows, theta=1e4, rotary_dim=64, batch=0, max_seqlen=0)
    assert (p.num_heads, p.num_key_heads, p.head_dim, p.query_stride_s, p.rotated_key_stride_s) == (4, 2, 64, 256, 128)
    pkg.ops.row_parallel_linear(torch.empty((0, 64), dtype=torch.float16), torch.empty((32, 64, 1), dtype=torch.float16), None,
                                torch.empty((0, 32), dtype=torch.float16))


def test_current_stream_without_the_private_call(pkg, monkeypatch):
    """A torch without the private raw-stream call serves the public one."""
    import importlib.util
    import types
    import torch
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    spec = importlib.util.spec_from_file_location(pkg.__name__ + ".ops_again", pkg.ops.__file__)
    ops = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(ops)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=4711))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert ops._stream() == 4711
    assert ops._stream(types.SimpleNamespace(cuda_stream=12)) == 12


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU; asking for more ends with a message that says so, before any device work."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "ONE GPU" in r.stderr and r.stdout.strip() == ""
