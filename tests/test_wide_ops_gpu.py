"""The 16-byte forms of the memory-bound operators next to their element forms: values, and which bytes
the KV append writes."""
import json

import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
ULP = {"float32": 2.0 ** -23, "bfloat16": 2.0 ** -7, "float16": 2.0 ** -10}


def run(op, inputs, attrs=None, outputs=("out",)):
    import dli

    graph = dli.Graph.from_json(json.dumps({
        "format": "dli.graph.v1", "model_type": op, "inputs": list(inputs),
        "outputs": list(outputs), "nodes": [{"name": "n", "op": op, "inputs": list(inputs),
                                             "outputs": list(outputs), "attrs": attrs or {}}]}))
    out = dli.Engine().load_plugin().run(graph, inputs)
    return [out[name] for name in outputs]


def rand(shape, dtype, seed, offset=0):
    """Contiguous random tensor, `offset` elements past a 16-byte boundary."""
    n = 1
    for s in shape:
        n *= s
    base = torch.randn(n + offset, generator=torch.Generator().manual_seed(seed))
    return base.to(DTYPES[dtype]).cuda()[offset:].view(shape)


# whole chunks, a broadcast operand of whole and of broken chunks, a rest, unaligned starts
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("shape,bshape,offset", [
    ((64, 896), (64, 896), 0), ((3, 5, 16), (16,), 0), ((6, 24), (12,), 0), ((5, 7), (7,), 0),
    ((1,), (1,), 0), ((16, 64), (16, 64), 1), ((5000, 1024), (5000, 1024), 0)])
def test_add_mul_silu_relu_exact(dtype, shape, bshape, offset):
    a, b = rand(shape, dtype, 1, offset), rand(bshape, dtype, 2)
    a.view(-1)[0] = float("inf")
    bb = b.reshape(-1).repeat(a.numel() // b.numel()).view(shape)
    t = DTYPES[dtype]
    assert torch.equal(run("add", {"a": a, "b": b})[0], (a.float() + bb.float()).to(t))
    assert torch.equal(run("mul", {"a": a, "b": b})[0], (a.float() * bb.float()).to(t))
    assert torch.equal(run("relu", {"x": a})[0], a.clamp_min(0))
    x, out = a.double(), run("silu", {"x": a})[0].double()
    ref = x / (1 + torch.exp(-x))
    keep = torch.isfinite(ref)
    # the output's rounding and the exponential's, relative to the argument
    bound = ULP[dtype] * ref.abs() + (4 + x.abs()) * 2.0 ** -22 * ref.abs() + 1e-7
    assert ((out - ref).abs()[keep] <= bound[keep]).all()


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("b,hq,hk,s,d,pairs,offset", [
    (2, 14, 2, 33, 64, 32, 0), (1, 3, 1, 5, 128, 64, 0), (2, 2, 2, 7, 24, 12, 0),
    (1, 2, 1, 6, 64, 20, 0), (1, 2, 1, 6, 6, 3, 0), (1, 4, 2, 9, 64, 32, 1)])
def test_rotary(dtype, b, hq, hk, s, d, pairs, offset):
    q, k = rand((b, hq, s, d), dtype, 3, offset), rand((b, hk, s, d), dtype, 4, offset)
    table = rand((2, s + 3, pairs), "float32", 5)
    pos = torch.arange(b, device="cuda") * 2 + 1  # the last sequence runs past the table
    out = run("rotary_embedding", {"q": q, "k": k, "cos": table[0], "sin": table[1], "p": pos}, {},
              ("oq", "ok"))
    for x, y in ((q, out[0]), (k, out[1])):
        ref = x.double().clone()
        for i in range(b):
            at = torch.arange(s, device="cuda") + pos[i]
            ok = at < s + 3
            c, n = (table[j].double()[at[ok]] for j in range(2))
            e, o = x[i, :, ok, 0:2 * pairs:2].double(), x[i, :, ok, 1:2 * pairs:2].double()
            ref[i, :, ok, 0:2 * pairs:2] = e * c - o * n
            ref[i, :, ok, 1:2 * pairs:2] = e * n + o * c
        err = (y.double() - ref).abs()
        assert (err <= ULP[dtype] * ref.abs() + 2.0 ** -21 * x.double().abs().max() * 4).all()


@pytest.mark.parametrize("d,block,cap", [(64, 64, 192), (128, 64, 128), (8, 16, 96), (72, 20, 100),
                                         (256, 64, 128)])
@pytest.mark.parametrize("s", [15, 16, 17, 40])
def test_kv_append_places_every_token(d, block, cap, s):
    """Positions on and off the 8-slot runs, before the cache and past its end."""
    import dli

    for positions in ([0, 8], [3, block - 1], [cap - 16, cap - 7], [-4, 24]):
        engine = dli.Engine().load_plugin()
        engine.configure_kv_cache(block_size=block, max_seq_len=cap)
        engine.reserve_kv_cache("L", "bfloat16", 2, 3, d)
        entry = engine.kv_cache_entry("L")
        for name in ("key_pool", "value_pool"):
            entry[name].fill_(7.0)
        expect = {n: entry[n].clone() for n in ("key_pool", "value_pool")}
        q, k, v = (rand((2, 3, s, d), "bfloat16", 6 + i) for i in range(3))
        table, slots = entry["block_table"].cpu(), entry["block_table"].shape[1] * block
        for b, p in enumerate(positions):
            for t in range(s):
                if 0 <= p + t < slots:
                    blk = int(table[b, (p + t) // block])
                    expect["key_pool"][blk, :, (p + t) % block] = k[b, :, t]
                    expect["value_pool"][blk, :, :, (p + t) % block] = v[b, :, t]
        graph = dli.Graph.from_json(json.dumps({
            "format": "dli.graph.v1", "model_type": "attention", "inputs": ["q", "k", "v", "p"],
            "outputs": ["out"], "nodes": [{"name": "a", "op": "attention",
                                           "inputs": ["q", "k", "v", "p"], "outputs": ["out"],
                                           "attrs": {"causal": True, "kv_cache": "L"}}]}))
        engine.run(graph, {"q": q, "k": k, "v": v, "p": torch.tensor(positions, device="cuda")})
        entry = engine.kv_cache_entry("L")
        for name in expect:
            assert torch.equal(entry[name], expect[name]), (name, positions)


# a row in one wave: 2, 4 and 8 chunks of 8 per lane, whole and with a rest
@pytest.mark.parametrize("rows,hidden", [(5, 1024), (5, 1032), (2, 1536), (9, 2048), (5, 2056),
                                         (3, 4088), (4, 4096), (70000, 1032)])
def test_rms_norm_rows(rows, hidden):
    x, w = rand((rows, hidden), "bfloat16", 9), rand((hidden,), "bfloat16", 10)
    out = run("rms_norm", {"x": x, "w": w}, {"eps": 1e-6})[0].double()
    xd = x.double()
    ref = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * w.double()
    # the output's rounding, half a step; the fp32 sum and root are far below
    assert ((out - ref).abs() <= 0.51 * ULP["bfloat16"] * ref.abs()).all()
