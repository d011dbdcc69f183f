"""bf16 and f16 linears over the edges of their routes (skinny kernels of 4 and 16 waves, tiled MFMA
GEMM with and without K parts, the general kernel) against float64."""
import json

import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16}
UNIT = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 2.0 ** -24}  # half an ulp, at most


def linear(x, w, bias, attrs):
    import dli

    inputs = {"x": x, "w": w, **({} if bias is None else {"b": bias})}
    graph = dli.Graph.from_json(json.dumps({
        "format": "dli.graph.v1", "model_type": "linear", "inputs": list(inputs),
        "outputs": ["out"], "nodes": [{"name": "l", "op": "linear", "inputs": list(inputs),
                                       "outputs": ["out"], "attrs": attrs}]}))
    return dli.Engine().load_plugin().run(graph, inputs)["out"]


def check(x, w, bias, out, out_dtype, relu=False):
    """Every element within the rounding of the output plus that of fp32 sums over K terms."""
    x64, w64 = x.double(), w.double()
    ref = x64 @ w64.t()
    terms = x64.abs() @ w64.abs().t()
    if bias is not None:
        ref, terms = ref + bias.double(), terms + bias.double().abs()
    if relu:
        ref = ref.clamp_min(0)
    tiny = 2.0 ** -24 if out_dtype == "float16" else 0.0  # the subnormal spacing of the output
    bound = UNIT[out_dtype] * ref.abs() + x.shape[1] * 2.0 ** -23 * terms + tiny
    assert ((out.double() - ref).abs() <= bound).all()


def inputs(dtype, m, n, k, seed=0):
    g = torch.Generator().manual_seed(seed)
    t = DTYPES[dtype]
    return (torch.randn(m, k, generator=g).to(t).cuda(),
            (torch.randn(n, k, generator=g) * 0.05).to(t).cuda(),
            torch.randn(n, generator=g).to(t).cuda())


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("m,n,k", [
    (1, 10, 4096), (16, 17, 64), (17, 896, 896), (33, 4096, 128), (64, 4096, 1024),
    (65, 33, 64),  # 16 waves, their row blocks, and the first row count past them
    (8, 4097, 128), (9, 8200, 256), (16, 4100, 3584),  # 4 waves and past their x limit
    (9, 100, 8192), (40, 896, 4864), (64, 70, 2304),  # decode-sized, K parts
    (3, 50, 72), (70, 200, 8), (129, 130, 136),  # K not a multiple of 64
    (77, 896, 4864), (300, 65, 1600), (300, 896, 4872),  # many rows, K parts, a short last part
    (1700, 1700, 96),  # 128 x 128 tiles
    (5, 7, 33)])  # the general kernel
def test_linear16_routes(dtype, m, n, k):
    x, w, b = inputs(dtype, m, n, k)
    check(x, w, b, linear(x, w, b, {}), dtype)
    check(x, w, None, linear(x, w, None, {"activation": "relu", "out_dtype": "float32"}),
          "float32", relu=True)
    check(x, w, b, linear(x, w, b, {"activation": "relu"}), dtype, relu=True)


@pytest.mark.parametrize("m", [4, 40, 100])
def test_f16_subnormals_count(m):
    """Subnormal float16 weights (below 2^-14) are not flushed by any route."""
    x, w, _ = inputs("float16", m, 96, 1024, 3)
    w = (w.float() * 2.0 ** -14).half()
    assert 0 < w.abs().max() < 2.0 ** -14
    check(x, w, None, linear(x, w, None, {"out_dtype": "float32"}), "float32")


@pytest.mark.parametrize("m", [4, 40, 200])
def test_f16_infinities_and_nan_stay_in_their_row(m):
    x, w, b = inputs("float16", m, 80, 2048, 4)
    clean = linear(x, w, b, {})
    x[1, 5], x[2, 7] = float("inf"), float("nan")
    out = linear(x, w, b, {})
    assert not torch.isfinite(out[1]).any() and torch.isnan(out[2]).all()
    keep = [i for i in range(m) if i not in (1, 2)]
    assert torch.equal(out[keep], clean[keep])


@pytest.mark.parametrize("m,n,k", [(77, 896, 4864), (300, 104, 2312), (70, 200, 136)])
def test_linear_residual_rows(m, n, k):
    """linear_residual of a prompt's rows, with K parts and without: the sum is rounded to bf16
    before the residual is added."""
    import dli

    x, w, b = inputs("bfloat16", m, n, k, 5)
    res = torch.randn(m, n, generator=torch.Generator().manual_seed(6)).bfloat16().cuda()
    names = ["x", "w", "r", "b"]
    graph = dli.Graph.from_json(json.dumps({
        "format": "dli.graph.v1", "model_type": "linear_residual", "inputs": names,
        "outputs": ["out"], "nodes": [{"name": "l", "op": "linear_residual", "inputs": names,
                                       "outputs": ["out"]}]}))
    out = dli.Engine().load_plugin().run(graph, {"x": x, "w": w, "r": res, "b": b})["out"].double()
    v = x.double() @ w.double().t() + b.double()
    terms = x.double().abs() @ w.double().abs().t() + b.double().abs()
    ref = res.double() + v
    # the linear output's rounding, the fp32 sums', then the result's
    bound = UNIT["bfloat16"] * (v.abs() + ref.abs()) * 1.01 + k * 2.0 ** -23 * terms
    assert ((out - ref).abs() <= bound).all()
