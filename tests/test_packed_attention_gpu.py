"""Attention of several query tokens per sequence on the packed-row MFMA kernels (gfx950): over
the paged cache and, for head_dim 128, over contiguous keys, against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
# bf16 output: 2^-9 of the value for its rounding, doubled for the fp32 sums before it
REL = 4e-3


def rand(shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(torch.bfloat16).to(DEV)


def to_np(t):
    return t.double().cpu().numpy()


def run_attention(inputs, attrs, engine):
    import json

    import dli

    names = list(inputs)
    graph = dli.Graph.from_json(json.dumps({
        "format": "dli.graph.v1", "model_type": "attention", "inputs": names, "outputs": ["out"],
        "nodes": [{"name": "a", "op": "attention", "inputs": names, "outputs": ["out"],
                   "attrs": attrs}]}))
    return engine.run(graph, inputs)["out"]


def check(out, ref):
    out = to_np(out)
    assert np.isfinite(out).all()
    assert np.linalg.norm(out - ref) <= REL * np.linalg.norm(ref)
    assert np.abs(out - ref).max() <= 2 * REL * max(1.0, np.abs(ref).max())


def paged_case(hq, hkv, d, sq, past, causal, block_size=64, capacity=None, stale=0.0):
    """Engine with `past[b]` random tokens cached per sequence, and the call's result next to the
    oracle's inputs. stale: what unused cache slots hold."""
    import dli

    batch = len(past)
    engine = dli.Engine().load_plugin()
    engine.configure_kv_cache(block_size=block_size, max_seq_len=capacity or max(past) + sq)
    engine.reserve_kv_cache("L", "bfloat16", batch, hkv, d)
    entry = engine.kv_cache_entry("L")
    entry["key_pool"].fill_(stale)
    entry["value_pool"].fill_(stale)
    hist_k, hist_v = rand((batch, hkv, max(past), d), 1), rand((batch, hkv, max(past), d), 2)
    table = entry["block_table"].cpu().numpy()
    for b in range(batch):
        for j in range(past[b]):
            blk, slot = table[b, j // block_size], j % block_size
            entry["key_pool"][blk, :, slot] = hist_k[b, :, j]
            entry["value_pool"][blk, :, :, slot] = hist_v[b, :, j]
    q, k, v = (rand((batch, h, sq, d), 3 + i) for i, h in enumerate((hq, hkv, hkv)))
    pos = torch.tensor(past, dtype=torch.int32, device=DEV)
    return engine, {"q": q, "k": k, "v": v, "positions": pos}, hist_k, hist_v


def check_paged(engine, inputs, hist_k, hist_v, past, causal):
    out = run_attention(inputs, {"causal": causal, "kv_cache": "L"}, engine)
    q, k, v = inputs["q"], inputs["k"], inputs["v"]
    for b, n in enumerate(past):
        keys = np.concatenate([to_np(hist_k[b:b + 1, :, :n]), to_np(k[b:b + 1])], 2)
        vals = np.concatenate([to_np(hist_v[b:b + 1, :, :n]), to_np(v[b:b + 1])], 2)
        check(out[b:b + 1], ops.attention(to_np(q[b:b + 1]), keys, vals, causal=causal))


# rows per KV head (sq * group) on both sides of the 64- and 128-row tiles; contexts on both sides
# of a 64-key tile, few enough for one key split and long enough for many
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,sq,past,causal", [
    (14, 2, 2, [64], True), (28, 4, 9, [63, 1], True), (28, 4, 10, [130, 257], True),
    (4, 4, 64, [0, 65], True), (4, 4, 65, [5], True), (6, 1, 43, [127, 700], False),
    (3, 3, 129, [1000, 500], True)])
def test_paged_chunk(d, hq, hkv, sq, past, causal):
    check_paged(*paged_case(hq, hkv, d, sq, past, causal), past, causal)


def test_paged_chunk_large_blocks_and_spare_capacity():
    """Cache blocks of two tiles; a capacity far above the tokens held (empty key splits)."""
    check_paged(*paged_case(14, 2, 64, 5, [90, 30], True, block_size=128, capacity=4096), [90, 30],
                True)


# the lines of the split rule: few row tiles (unsplit up to 4 key tiles, 3 splits of 5, then the most
# that 64 tiles give), and 128 of them (1 and 2 splits)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("batch,hq,hkv,past,tiles", [
    (1, 4, 2, 50, 1), (1, 4, 2, 100, 2), (1, 4, 2, 180, 3), (1, 4, 2, 4000, 64),
    (1, 4, 2, 253, 4), (1, 4, 2, 254, 5),
    (4, 64, 32, 40, 11), (4, 64, 32, 700, 12)])
def test_paged_chunk_split_rule(d, batch, hq, hkv, past, tiles):
    case = paged_case(hq, hkv, d, 3, [past] * batch, True, capacity=64 * tiles)
    check_paged(*case, [past] * batch, True)


@pytest.mark.parametrize("d", [64, 128])
def test_paged_chunk_never_reads_hidden_values(d):
    """NaN in unused cache slots, and infinite or NaN values of the chunk's last token: rows that
    do not see them are unaffected."""
    past, sq = [70, 200], 20
    engine, inputs, hist_k, hist_v = paged_case(14, 2, d, sq, past, True, stale=float("nan"))
    check_paged(engine, inputs, hist_k, hist_v, past, True)
    clean = run_attention(inputs, {"causal": True, "kv_cache": "L"}, engine)
    inputs["v"][:, :, -1, ::2] = float("inf")
    inputs["v"][:, :, -1, 1::2] = float("nan")
    out = run_attention(inputs, {"causal": True, "kv_cache": "L"}, engine)
    err = (out[:, :, :-1].double() - clean[:, :, :-1].double()).norm()
    assert err <= REL * clean[:, :, :-1].double().norm()
    assert torch.isinf(out[:, :, -1, ::2]).all() and torch.isnan(out[:, :, -1, 1::2]).all()


@pytest.mark.parametrize("sq,sk,hq,hkv,causal", [(16, 16, 4, 4, True), (18, 100, 28, 4, True),
                                                 (77, 77, 7, 1, True), (40, 130, 6, 2, False),
                                                 (130, 65, 2, 2, True)])
def test_dense_head_dim_128(sq, sk, hq, hkv, causal):
    import dli

    q, k, v = rand((2, hq, sq, 128), 11), rand((2, hkv, sk, 128), 12), rand((2, hkv, sk, 128), 13)
    out = run_attention({"q": q, "k": k, "v": v}, {"causal": causal}, dli.Engine().load_plugin())
    if causal and sq > sk:  # queries before the first key: zeros
        assert (out[:, :, :sq - sk] == 0).all()
        out, q = out[:, :, sq - sk:], q[:, :, sq - sk:]
    check(out, ops.attention(to_np(q), to_np(k), to_np(v), causal=causal))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk,hq,hkv,causal", [(16, 16, 4, 4, True), (18, 100, 28, 4, True),
                                                 (77, 77, 7, 1, True), (40, 130, 6, 2, False),
                                                 (130, 65, 2, 2, True)])
def test_dense_f32(d, sq, sk, hq, hkv, causal):
    """fp32 throughout: the scores' and sums' roundings, about sqrt(d) and sqrt(keys) ulps."""
    import dli

    g = torch.Generator().manual_seed(21)
    q, k, v = (torch.randn(2, h, s, d, generator=g).to(DEV)
               for h, s in ((hq, sq), (hkv, sk), (hkv, sk)))
    out = run_attention({"q": q, "k": k, "v": v}, {"causal": causal}, dli.Engine().load_plugin())
    if causal and sq > sk:  # queries before the first key: zeros
        assert (out[:, :, :sq - sk] == 0).all()
        out, q = out[:, :, sq - sk:], q[:, :, sq - sk:]
    ref = ops.attention(to_np(q), to_np(k), to_np(v), causal=causal)
    assert np.linalg.norm(to_np(out) - ref) <= 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("d", [64, 128])
def test_dense_f32_never_reads_hidden_values(d):
    import dli

    g = torch.Generator().manual_seed(22)
    q, k, v = (torch.randn(1, h, 50, d, generator=g).to(DEV) for h in (4, 2, 2))
    engine = dli.Engine().load_plugin()
    clean = run_attention({"q": q, "k": k, "v": v}, {"causal": True}, engine)
    v[:, :, -1, ::2], v[:, :, -1, 1::2] = float("inf"), float("nan")
    out = run_attention({"q": q, "k": k, "v": v}, {"causal": True}, engine)
    err = (out[:, :, :-1] - clean[:, :, :-1]).norm()
    assert err <= 1e-6 * clean[:, :, :-1].norm()
    assert torch.isinf(out[:, :, -1, ::2]).all() and torch.isnan(out[:, :, -1, 1::2]).all()


@pytest.mark.parametrize("scale", [0.0, -0.1, 0.3])
@pytest.mark.parametrize("dtype,d,layout", [
    (torch.bfloat16, 128, "bhsd"), (torch.float32, 64, "bhsd"), (torch.float32, 128, "bhsd"),
    (torch.bfloat16, 64, "bhsd"), (torch.bfloat16, 64, "bshd")])
def test_dense_scale_of_any_sign(dtype, d, layout, scale):
    import dli

    g = torch.Generator().manual_seed(31)
    q, k, v = (torch.randn(2, h, s, d, generator=g).to(dtype).to(DEV)
               for h, s in ((6, 20), (2, 90), (2, 90)))
    out = run_attention({"q": q, "k": k, "v": v},
                        {"causal": True, "scale": scale, "output_layout": layout},
                        dli.Engine().load_plugin())
    out = out.transpose(1, 2) if layout == "bshd" else out
    check(out, ops.attention(to_np(q), to_np(k), to_np(v), causal=True, scale=scale))


@pytest.mark.parametrize("scale", [0.0, -0.1, 0.3])
@pytest.mark.parametrize("d", [64, 128])
def test_paged_chunk_scale_of_any_sign(d, scale):
    past = [70, 200]
    engine, inputs, hist_k, hist_v = paged_case(6, 2, d, 7, past, True)
    out = run_attention(inputs, {"causal": True, "kv_cache": "L", "scale": scale}, engine)
    q, k, v = inputs["q"], inputs["k"], inputs["v"]
    for b, n in enumerate(past):
        keys = np.concatenate([to_np(hist_k[b:b + 1, :, :n]), to_np(k[b:b + 1])], 2)
        vals = np.concatenate([to_np(hist_v[b:b + 1, :, :n]), to_np(v[b:b + 1])], 2)
        check(out[b:b + 1], ops.attention(to_np(q[b:b + 1]), keys, vals, causal=True, scale=scale))


def check_spoiled(run, clean, v, seen):
    """Infinities of both signs and a NaN at `seen` of the values: the heads that read them give them
    back, other dimensions keep their values."""
    v[seen + (slice(0, 1),)], v[seen + (slice(5, 6),)] = float("inf"), float("-inf")
    v[seen + (slice(9, 10),)] = float("nan")
    out = run()
    assert (out[..., 0] == float("inf")).all() and (out[..., 5] == float("-inf")).all()
    assert torch.isnan(out[..., 9]).all()
    rest = [d for d in range(out.shape[-1]) if d not in (0, 5, 9)]
    err = (out[..., rest].double() - clean[..., rest].double()).norm()
    assert err <= REL * clean[..., rest].double().norm()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,past", [(5, 200), (70, 130), (3, 4000)])
def test_paged_chunk_infinite_value_of_a_cached_key(d, sq, past):
    """A key that every row sees, in a tile without hidden keys (and in one key split of several)."""
    engine, inputs, _, _ = paged_case(14, 2, d, sq, [past], True)
    attrs = {"causal": True, "kv_cache": "L"}
    clean = run_attention(inputs, attrs, engine)
    entry = engine.kv_cache_entry("L")
    blk = int(entry["block_table"][0, 0])
    values = entry["value_pool"].transpose(2, 3)  # [block, head, slot, d]
    check_spoiled(lambda: run_attention(inputs, attrs, engine), clean, values,
                  (blk, slice(None), 3))


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float32, 64),
                                     (torch.float32, 128)])
def test_dense_infinite_value_of_a_seen_key(dtype, d):
    import dli

    g = torch.Generator().manual_seed(41)
    q, k, v = (torch.randn(2, h, s, d, generator=g).to(dtype).to(DEV)
               for h, s in ((6, 40), (2, 200), (2, 200)))
    engine = dli.Engine().load_plugin()
    run = lambda: run_attention({"q": q, "k": k, "v": v}, {"causal": True}, engine)
    check_spoiled(run, run(), v, (slice(None), slice(None), 3))


@pytest.mark.parametrize("d,paged", [(128, False), (64, True), (128, True)])
def test_probabilities_keep_fp32(d, paged):
    """Two keys of almost the same probability p with values 1 and -1: the output is their
    difference, about 2^-13 p, over the row sum. An fp32 probability is off by about 2 ulps, 2^-23 p,
    so the difference by 2^-9 of itself, like the rounding of the output; probabilities of 17 or 18
    bits are off by up to 2^-5 of it."""
    import dli

    batch, hkv, sq, sk, delta = 8, 4, 16, 200, 2.0 ** -13
    c = torch.linspace(0.05, 0.95, batch * hkv).view(batch, hkv).to(torch.bfloat16).to(DEV)
    q = torch.zeros(batch, 2 * hkv, sq, d, dtype=torch.bfloat16, device=DEV)
    q[..., :2] = 1
    k = torch.zeros(batch, hkv, sk, d, dtype=torch.bfloat16, device=DEV)
    k[..., 0] = -100  # probability 0
    k[:, :, 9, 0] = 0  # the row maximum
    k[:, :, 70, 0] = k[:, :, 71, 0] = -c
    k[:, :, 71, 1] = -delta
    v = torch.zeros_like(k)
    v[:, :, 70], v[:, :, 71] = 1, -1
    engine, attrs = dli.Engine().load_plugin(), {"scale": 1.0}
    if paged:
        past = sk - sq
        engine.configure_kv_cache(block_size=64, max_seq_len=sk)
        engine.reserve_kv_cache("L", "bfloat16", batch, hkv, d)
        entry = engine.kv_cache_entry("L")
        for j in range(past):
            blocks = entry["block_table"][:, j // 64].long()
            entry["key_pool"][blocks, :, j % 64] = k[:, :, j]
            entry["value_pool"][blocks, :, :, j % 64] = v[:, :, j]
        out = run_attention({"q": q, "k": k[:, :, past:].contiguous(),
                             "v": v[:, :, past:].contiguous(),
                             "positions": torch.full((batch,), past, device=DEV)},
                            {**attrs, "kv_cache": "L"}, engine)
    else:
        out = run_attention({"q": q, "k": k, "v": v}, attrs, engine)
    pa, pb = torch.exp(-c.double()), torch.exp(-c.double() - delta)
    ref = ((pa - pb) / (1 + pa + pb)).repeat_interleave(2, 1)[:, :, None, None]
    assert ((out.double() - ref).abs() <= 2.0 ** -7 * ref).all()


# the lines of the dense rules: fp32 query rows x keys of 49152 (row kernel) and above, 96 keys and more; bf16 with 256
# 64-row tiles and more (128-row tiles)
@pytest.mark.parametrize("dtype,d,batch,hq,hkv,sq,sk", [
    (torch.float32, 64, 2, 8, 2, 32, 96), (torch.float32, 64, 2, 8, 2, 33, 96),
    (torch.float32, 128, 1, 3, 1, 16, 96), (torch.float32, 128, 1, 3, 1, 16, 97),
    (torch.bfloat16, 128, 4, 64, 32, 64, 70), (torch.bfloat16, 128, 4, 64, 32, 65, 70)])
def test_dense_rule_lines(dtype, d, batch, hq, hkv, sq, sk):
    import dli

    g = torch.Generator().manual_seed(51)
    q, k, v = (torch.randn(batch, h, s, d, generator=g).to(dtype).to(DEV)
               for h, s in ((hq, sq), (hkv, sk), (hkv, sk)))
    out = run_attention({"q": q, "k": k, "v": v}, {"causal": True}, dli.Engine().load_plugin())
    group = hq // hkv
    mask = torch.ones(sq, sk, dtype=torch.bool, device=DEV).tril(sk - sq)
    for h in range(hq):
        score = torch.matmul(q[:, h].double(), k[:, h // group].double().transpose(1, 2).contiguous())
        p = torch.softmax((score / d ** 0.5).masked_fill(~mask, -np.inf), -1)
        ref = torch.matmul(p, v[:, h // group].double())
        err = (out[:, h].double() - ref).norm()
        assert err <= (1e-6 if dtype == torch.float32 else REL) * ref.norm()
