"""The work a serving program gives this library, as cases that can be timed and compared.

A case is a dict of plain values.  Its `kind` is one of the library's public entry points:

  "step"    one layer call of the attention operator, DynamicBatchingMultiHeadCacheAttention.forward(): quantise/append
            of the step's new K/V rows, decode attention over the int8 cache, and the prefill attention of its prompts
  "rope"    RoPE of a step's query and key rows fused with the quantise/append, ops.rope_key_value_cache()
  "linear"  the output projection behind the attention, ops.row_parallel_linear()

Sequence lengths follow from the case alone (`lens` seeds them), values from the seed of prepare(): standard normal
half rows with 2 % of the channels of every kv head ten times as large, as the activations of a transformer have them.
"""
import math

import numpy as np
import torch

import __graft_entry__ as entry

pkg = entry.load_package()
ops, workloads, harness = pkg.ops, pkg.workloads, pkg.harness


def _step(name, hq, hkv, d, mode, lens, dec=0, kv=(1, 1), spread="uniform", pre=0, q=(1, 1), prior=(0, 0),
          cache_prefill=True, alibi=False, kind="step"):
    """`dec` decode sequences of kv[0]..kv[1] tokens, then `pre` prompts of q[0]..q[1] new tokens over
    prior[0]..prior[1] tokens that are in the cache already; mode 0 = contiguous cache, 1 = pages of 128 tokens."""
    case = dict(kind=kind, heads=hq, kv_heads=hkv, head_dim=d, mode=mode, lens=lens, decodes=dec, kv_min=kv[0], kv_max=kv[1],
                spread=spread, prompts=pre, q_min=q[0], q_max=q[1], prior_min=prior[0], prior_max=prior[1],
                cache_prefill=cache_prefill, alibi=alibi)
    if name:
        case["name"] = name
    return case


def _linear(name, m, k, n, bias):
    case = dict(kind="linear", rows=m, in_features=k, out_features=n, bias=bias)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # four short conversations of a small multi-head model: three launches and nothing to stream
        _step("decode_four_short", 8, 8, 64, 0, 1001, dec=4, kv=(128, 512)),
        # one user, one long conversation: latency of a step that has to be split over the whole chip
        _step("decode_one_sequence", 32, 8, 128, 1, 1, dec=1, kv=(4096, 4096)),
        # multi-head attention, contiguous cache, a batch of ordinary length
        _step("decode_mha", 32, 32, 128, 0, 1002, dec=64, kv=(512, 4096)),
        # grouped-query attention, paged cache: the serving batch that the bench line is quoted on
        _step("decode_gqa", 32, 8, 128, 1, 1003, dec=128, kv=(1024, 8192), spread="log"),
        # a larger model's heads over long contexts
        _step("decode_gqa8_long", 64, 8, 128, 1, 1004, dec=32, kv=(8192, 32768), spread="log"),
        # many short conversations: a large chat batch, where starting a sequence counts more than streaming it
        _step("decode_many_short", 32, 8, 128, 1, 7, dec=512, kv=(100, 300)),
        # continuous batching: decode sequences and chunked prompts over their history in one step
        _step("mixed_step", 32, 8, 128, 1, 1005, dec=240, kv=(512, 4096), pre=16, q=(256, 1024), prior=(0, 2048)),
        # speculative decoding: a few drafted tokens per sequence to verify over a long history
        _step("draft_tokens", 32, 8, 128, 1, 5, pre=64, q=(2, 8), prior=(1024, 3072)),
        # first prompts: nothing in the cache yet, attention over the step's own half K/V rows
        _step("first_prompts", 32, 8, 128, 1, 11, pre=12, q=(300, 3000), cache_prefill=False),
        # RoPE + append in front of the mixed step
        _step("rope_append_mixed", 32, 8, 128, 1, 1005, dec=240, kv=(512, 4096), pre=16, q=(256, 1024), prior=(0, 2048),
              kind="rope"),
        # output projection of a decode step and of the query rows of a step with prompts
        _linear("o_proj_decode", 128, 4096, 4096, False),
        _linear("o_proj_prompts", 11104, 4096, 4096, False),
    ]


# (query heads, kv heads, head_dim) of the batches that the tests and the benchmark of this repository run: multi-head,
# grouped-query, multi-query, and what a tensor-parallel rank holds of them
_HEADS = [(8, 8, 64), (32, 8, 64), (14, 2, 64), (32, 32, 96), (32, 32, 128), (32, 8, 128), (64, 8, 128), (28, 4, 128),
          (16, 4, 128), (8, 1, 128), (5, 5, 128), (48, 1, 128), (16, 16, 256), (16, 8, 256), (8, 1, 256)]
_WIDTHS = [(2048, 2048), (4096, 4096), (5120, 5120), (8192, 8192), (14336, 4096), (4096, 6144), (1024, 8192)]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["mixed"] * 2 + ["draft"] + ["first"] * 2 + ["rope"] * 2 + ["linear"] * 3)
    lens, mode = rng.randrange(1, 1 << 30), rng.choice([0, 1, 1])
    if kind == "linear":
        k, n = rng.choice(_WIDTHS)
        top = min(11000, int(1.8e11 / (k * n)))
        return _linear("", _log_int(rng, 1, top), k, n, rng.random() < 0.3)
    hq, hkv, d = rng.choice(_HEADS)
    per_token = hkv * (2 * d + d // 2)
    budget = 1.0e9 / per_token  # kv tokens of at most a gigabyte of cache

    def decodes(most):
        hi = _log_int(rng, 128, 32768)
        lo = max(64, int(hi * rng.uniform(0.2, 1.0)))
        return dict(dec=max(1, min(_log_int(rng, 1, 512), int(most / hi))), kv=(lo, hi), spread=rng.choice(["uniform", "log"]))

    def prompts(most_flops, rows):
        hi = _log_int(rng, 64, rows)
        lo = max(17, int(hi * rng.uniform(0.3, 1.0)))
        prior = rng.choice([0, 512, 2048, 4096])
        each = 4.0 * hq * d * hi * (prior + hi / 2)
        return dict(pre=max(1, min(_log_int(rng, 1, 32), int(most_flops / each), 16000 // hi)), q=(lo, hi), prior=(prior // 4, prior))

    if kind == "decode":
        return _step("", hq, hkv, d, mode, lens, **decodes(budget))
    if kind == "mixed":
        return _step("", hq, hkv, d, mode, lens, alibi=rng.random() < 0.15, **decodes(0.5 * budget), **prompts(1.5e11, 2048))
    if kind == "draft":
        top = max(2, 32 * hkv // hq)
        lo = rng.randint(1, 2)
        prior = _log_int(rng, 200, 8192)
        seqs = max(1, min(_log_int(rng, 1, 256), int(budget / (prior + top))))
        return _step("", hq, hkv, d, mode, lens, pre=seqs, q=(lo, rng.randint(lo, top)), prior=(prior // 2, prior))
    if kind == "first":
        p = prompts(1.5e11, 3000)
        p["prior"] = (0, 0)
        return _step("", hq, hkv, d, mode, lens, cache_prefill=False, alibi=rng.random() < 0.15, **p)
    p = prompts(1.0e12, 2048) if rng.random() < 0.5 else {}
    return _step("", hq, hkv, d, mode, lens, kind="rope", **decodes(0.25 * budget), **p)


def _lengths(case):
    """(kv lengths of the decode sequences, new tokens of the prompts, tokens the prompts have in the cache)."""
    rng = np.random.default_rng(case["lens"])

    def some(lo, hi, n, spread="uniform"):
        if spread == "log":
            return np.floor(np.exp(rng.uniform(np.log(lo), np.log(hi), n))).astype(np.int64)
        return rng.integers(lo, hi + 1, n)
    kv = some(case["kv_min"], case["kv_max"], case["decodes"], case["spread"])
    q = some(case["q_min"], case["q_max"], case["prompts"])
    prior = some(case["prior_min"], case["prior_max"], case["prompts"])
    return kv, q, prior


def _rows(bt, gen, n, heads):
    """Half rows [n, heads, head_dim] with the outlier channels of each kv head."""
    x = torch.randn((n, heads, bt.head_dim), device="cuda", generator=gen, dtype=torch.float32).to(torch.float16)
    gain = np.ones((bt.num_kv_heads, bt.head_dim), dtype=np.float16)
    for h in range(bt.num_kv_heads):
        gain[h, bt.outlier_channels[h]] = 10.0
    return x.mul_(torch.from_numpy(gain.repeat(heads // bt.num_kv_heads, axis=0)).cuda())


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["kind"] == "linear":
        m, k, n = case["rows"], case["in_features"], case["out_features"]
        x = torch.randn((m, k), device="cuda", generator=gen).to(torch.float16)
        w = (torch.randn((n, k), device="cuda", generator=gen) * k ** -0.5).to(torch.float16)
        bias = torch.randn((n,), device="cuda", generator=gen).to(torch.float16) if case["bias"] else None
        nbytes = ops.row_parallel_linear_workspace_size(m, k, n)
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
        return dict(kind="linear", x=x, w=w, bias=bias, ws=ws, out=torch.zeros((m, n), dtype=torch.float16, device="cuda"))

    kv, q_lens, prior = _lengths(case)
    # the pool is as large as any placement of the sequences needs (contiguous runs lie up to three tokens apart)
    pool = 8 + int(kv.sum() + q_lens.sum() + prior.sum()) + 4 * (len(kv) + len(q_lens))
    bt, _ = workloads.custom_batch(seed, case["heads"], case["kv_heads"], case["head_dim"], case["mode"], kv, q_lens, prior,
                                   outliers=True, pool_tokens_at_least=pool)
    dev = harness.DeviceBatch(bt)
    # what the cache holds before the step: quantised by the library from half rows, all sequences in one call
    n_old = int(bt.start_pos.sum())
    if n_old:
        starts = torch.from_numpy(np.concatenate([[0], np.cumsum(bt.start_pos)])).cuda()
        ops.key_value_cache(_rows(bt, gen, n_old, bt.num_kv_heads), _rows(bt, gen, n_old, bt.num_kv_heads), starts,
                            dev.cachestarts, torch.zeros_like(dev.start_pos), dev.cache, dev.scale, batch=bt.batch,
                            max_seqlen=int(bt.start_pos.max()), num_layer=1, layer_idx=0, num_kv_heads=bt.num_kv_heads,
                            head_dim=bt.head_dim, **dev.layout_kwargs())
    n_new = int(bt.q_lens.sum())
    dev.query = _rows(bt, gen, n_new, bt.num_heads)
    dev.new_key, dev.new_value = _rows(bt, gen, n_new, bt.num_kv_heads), _rows(bt, gen, n_new, bt.num_kv_heads)
    dev.output = torch.zeros_like(dev.query)
    if case["kind"] == "rope":
        return dict(kind="rope", dev=dev, rotated=torch.zeros_like(dev.query))
    more = {}
    if case["alibi"]:
        more["alibi_slopes"] = 2.0 ** (-8.0 * torch.arange(1, bt.num_heads + 1, device="cuda", dtype=torch.float32) / bt.num_heads)
    if not case["cache_prefill"]:
        more["enable_cache_prefill"] = False
    return dict(kind="step", dev=dev, op=dev.make_operator(**more))


def run(state):
    if state["kind"] == "linear":
        ops.row_parallel_linear(state["x"], state["w"], state["bias"], state["out"], workspace=state["ws"])
        return state["out"]
    dev = state["dev"]
    if state["kind"] == "rope":
        bt = dev.bt
        ops.rope_key_value_cache(dev.query, dev.new_key, dev.new_value, dev.start_pos, dev.seqstarts, dev.cachestarts,
                                 state["rotated"], None, dev.cache, dev.scale, num_layer=1, layer_idx=0, theta=10000.0,
                                 rotary_dim=bt.head_dim, batch=bt.batch, max_seqlen=bt.max_seqlen, **dev.layout_kwargs())
        return {"query": state["rotated"], "cache": dev.cache, "scale": dev.scale}
    rc = state["op"].forward()
    if rc != ops.RC_SUCCESS:
        raise ops.PmxError(rc, "forward")
    return {"output": dev.output, "cache": dev.cache, "scale": dev.scale}


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["rows"], case["in_features"], case["out_features"]
        return {"bytes": 2 * (m * k + n * k + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    kv, q, prior = _lengths(case)
    new = int(case["decodes"] + q.sum())
    per_token = hkv * (2 * d + d // 2)           # int8 K and V rows with a half scale for every 8 channels
    step_rows = new * (2 * hq * d * 2 + hkv * 2 * d * 2)  # query in, output out, new K and V in
    if case["kind"] == "rope":
        return {"bytes": new * per_token + step_rows, "flops": 0}
    # every cached row once (read, or written by this step's append) where it is attended over from the cache
    tokens = int(kv.sum() + (prior.sum() + q.sum() if case["cache_prefill"] else q.sum()))
    pairs = int(kv.sum() + (q * prior + q * (q + 1) // 2).sum())
    return {"bytes": tokens * per_token + step_rows, "flops": 4 * hq * d * pairs}


def tolerance(case):
    if case["kind"] == "rope":
        return "exact"  # rotation in binary64, quantiser in IEEE arithmetic
    # against the same call in binary64 (dequantised cache, softmax and sums) the listed cases show rel 1.9e-4 to 2.1e-4 and
    # max 4.5e-4 to 6.3e-4, of which the rounding of the output to half alone is 2.1e-4 and 4.9e-4: four times that.
    # The cache's bytes and scales, which a step returns as well, are whole values and the same to the bit.
    return {"rel": 8.5e-4, "max": 2.6e-3}
