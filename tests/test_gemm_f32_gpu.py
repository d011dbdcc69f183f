"""fp32 linear, matmul and conv2d over the edges of their forms (few rows, K groups, K parts, unaligned
rows), against float64, and the operands that the three-term products hand to the fp32 instruction."""
import json

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def rand(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).cuda()


def run(op, inputs, attrs):
    import dli

    graph = dli.Graph.from_json(json.dumps({
        "format": "dli.graph.v1", "model_type": op, "inputs": list(inputs), "outputs": ["out"],
        "nodes": [{"name": "n", "op": op, "inputs": list(inputs), "outputs": ["out"],
                   "attrs": attrs}]}))
    return dli.Engine().load_plugin().run(graph, inputs)["out"]


def close(out, ref, terms, k):
    """Each product within 2^-24 of its value (what the split leaves out is below 2^-30), at most one
    rounding of the partial sums per product, and those of the parts, the bias and the output."""
    assert ((out.double() - ref).abs() <= (k + 4) * 2.0 ** -23 * terms).all()
    assert (out.double() - ref).norm() <= 1e-6 * terms.norm()


def check_linear(x, w, b, relu=False):
    out = run("linear", {"x": x, "w": w, "b": b}, {"activation": "relu"} if relu else {})
    ref = x.double() @ w.double().t() + b.double()
    terms = x.double().abs() @ w.double().abs().t() + b.double().abs()
    close(out, ref.clamp_min(0) if relu else ref, terms, x.shape[1])


@pytest.mark.parametrize("m,n,k", [
    (1, 64, 4), (16, 65, 32), (100, 65, 28),  # one slice: one group
    (16, 65, 36), (1, 64, 64), (16, 4096, 1024), (3, 10, 4096), (5, 896, 4864),  # 16-row tiles
    (17, 63, 36), (64, 4096, 1024), (64, 10, 4096), (40, 130, 4100),  # one row tile
    (65, 64, 64), (77, 128, 896), (256, 1024, 100), (200, 896, 2000),  # K groups, parts
    (1000, 1100, 260), (513, 2050, 32),  # one group
    (7, 9, 3), (70, 100, 33), (100, 70, 1001)])  # K % 4 != 0
def test_linear_f32_forms(m, n, k):
    x, w, b = rand((m, k), 1), rand((n, k), 2, 0.05), rand((n,), 3)
    check_linear(x, w, b)
    check_linear(x, w, b, relu=True)


def test_linear_f32_unaligned_rows():
    """A weight that does not start on 16 bytes takes the 4-byte loads."""
    base = rand((100 * 64 + 1,), 4, 0.1)
    w = base[1:].view(100, 64)
    assert w.data_ptr() % 16 != 0
    check_linear(rand((70, 64), 5), w, rand((100,), 6))


@pytest.mark.parametrize("m", [4, 40, 100, 300])
@pytest.mark.parametrize("scale", [2.0 ** 60, 2.0 ** -60])
def test_linear_f32_magnitudes(m, scale):
    x, w, b = rand((m, 256), 7) * scale, rand((80, 256), 8), rand((80,), 9) * scale
    check_linear(x, w, b)


@pytest.mark.parametrize("m,n,k", [(4, 70, 1), (4, 70, 4), (40, 70, 2), (100, 65, 4), (100, 65, 3),
                                   (300, 600, 12), (900, 1200, 4)])
@pytest.mark.parametrize("worst", [False, True])
def test_short_f32_products_keep_every_term(m, n, k, worst):
    """Products of one sign: h h' and the small terms are rounded once each and once more together, at
    most 2^-24 of the sum of the products apiece, the small terms' 2^-7 of that. Without m l' and
    l m' an operand of 1.0000 1111 1111 1111 1111 (`worst`) loses 2^-21 of every product."""
    x, w = (1 + torch.rand(s, generator=torch.Generator().manual_seed(i)).cuda()
            for i, s in ((24, (m, k)), (25, (n, k))))
    if worst:
        x[:], w[:] = (torch.tensor(0x3F80FFFF, dtype=torch.int32).view(torch.float32).item(),) * 2
    ref = x.double() @ w.double().t()
    bound = (2 + 2.0 ** -6) * 2.0 ** -24 * ref
    for out in (run("linear", {"x": x, "w": w}, {}),
                run("matmul", {"a": x, "b": w.t().contiguous()}, {}),
                run("conv2d", {"x": x.t().reshape(1, k, 1, m).contiguous(), "w": w.view(n, k, 1, 1)},
                    {}).view(n, m).t()):
        assert ((out.double() - ref).abs() <= bound).all()


# exponents of the operands; the last bits of a normal value below 2^-110 lie below the smallest bf16
# (2^-133), and below 2^-126 values are subnormal
@pytest.mark.parametrize("m", [4, 40, 100, 300])
@pytest.mark.parametrize("low,high", [(-108, 60), (-114, 60), (-120, 0), (-126, 60), (-132, 100),
                                      (-140, 100)])
def test_f32_products_of_tiny_operands(m, low, high):
    if low + high < -100:  # results of 2^-120: their own roundings are subnormal steps of 2^-149
        high += 60
    x, w = rand((m, 256), 18) * 2.0 ** low, rand((80, 256), 19) * 2.0 ** high
    tiny = x.double().abs().max()
    assert 0 < tiny < 2.0 ** (low + 4)
    check_linear(x, w, torch.zeros(80, device="cuda"))
    check_linear(w, x, torch.zeros(m, device="cuda"))
    check_linear(x[:, :251].contiguous(), w[:, :251].contiguous(), torch.zeros(80, device="cuda"))
    close(run("matmul", {"a": x, "b": w.t().contiguous()}, {}), x.double() @ w.double().t(),
          x.double().abs() @ w.double().abs().t(), 256)
    # one tiny value among ordinary ones, in a column of w that is 2^100
    x, w = rand((m, 64), 20), rand((80, 64), 21)
    x[:, 5], w[:, 5] = x[:, 5] * 2.0 ** low, 2.0 ** 100
    check_linear(x, w, torch.zeros(80, device="cuda"))


@pytest.mark.parametrize("n,c,kern", [(3, 16, 3), (2, 3, 7)])
def test_conv2d_f32_of_tiny_operands(n, c, kern):
    x, k = rand((n, c, 12, 12), 22) * 2.0 ** -125, rand((70, c, kern, kern), 23) * 2.0 ** 60
    out = run("conv2d", {"x": x, "w": k}, {"padding": [1, 1]})
    ref, terms = (F.conv2d(p.double().cpu(), q.double().cpu(), padding=1).cuda()
                  for p, q in ((x, k), (x.abs(), k.abs())))
    close(out, ref, terms, c * kern * kern)


@pytest.mark.parametrize("m", [4, 40, 100, 300])
def test_linear_f32_infinities_and_nan(m):
    """Infinite and NaN operands, and sums past the fp32 range, give what fp32 arithmetic gives; the
    other rows keep their values."""
    x, w, b = rand((m, 512), 10), rand((72, 512), 11).abs() + 0.5, rand((72,), 12)
    clean = run("linear", {"x": x, "w": w, "b": b}, {})
    x[0, 3] = float("inf")
    x[1, 500] = float("nan")
    x[2, :] = 3e38
    x[3, 8], x[3, 9] = float("inf"), float("-inf")
    out = run("linear", {"x": x, "w": w, "b": b}, {})
    assert (out[0] == float("inf")).all() and (out[2] == float("inf")).all()
    assert torch.isnan(out[1]).all() and torch.isnan(out[3]).all()
    err = (out[4:] - clean[4:]).abs()
    assert (err <= 512 * 2.0 ** -23 * (x[4:].abs() @ w.abs().t())).all()


def test_matmul_f32_forms():
    for m, n, k in ((5, 70, 64), (100, 65, 260), (600, 1100, 96), (33, 40, 7)):
        a, b = rand((m, k), 13), rand((k, n), 14, 0.1)
        close(run("matmul", {"a": a, "b": b}, {}), a.double() @ b.double(),
              a.double().abs() @ b.double().abs(), k)


@pytest.mark.parametrize("n,c,h,w,oc,kern,stride,pad", [
    (1, 64, 16, 16, 192, 3, 1, 1), (3, 192, 8, 8, 384, 3, 1, 1),  # K groups and parts
    (40, 64, 8, 8, 256, 3, 1, 1),  # parts of one group
    (64, 16, 16, 16, 192, 3, 1, 1),  # one group, one part
    (2, 5, 9, 7, 33, 3, 2, 1), (2, 7, 11, 11, 10, 5, 2, 2), (3, 12, 5, 5, 65, 1, 1, 0),
    (70, 4, 3, 3, 20, 3, 1, 0), (2, 4, 12, 12, 20, 7, 1, 3), (5, 8, 6, 6, 70, 5, 1, 2)])
def test_conv2d_f32_forms(n, c, h, w, oc, kern, stride, pad):
    x, k, b = rand((n, c, h, w), 15), rand((oc, c, kern, kern), 16, 0.1), rand((oc,), 17)
    attrs = {"stride": [stride, stride], "padding": [pad, pad], "activation": "relu"}
    out = run("conv2d", {"x": x, "w": k, "b": b}, attrs)
    ref, terms = (F.conv2d(p.double().cpu(), q.double().cpu(), r.double().cpu(), stride=stride,
                           padding=pad).cuda()
                  for p, q, r in ((x, k, b), (x.abs(), k.abs(), b.abs())))
    close(out, ref.clamp_min(0), terms, c * kern * kern)


def test_f32_rows_past_one_grid():
    """More than 64 x 65535 rows go in two launches; more than 128 x 65535 are refused."""
    m, n, k = 64 * 65535 + 70, 3, 4
    x, w, b = rand((m, k), 26), rand((n, k), 27), rand((n,), 28)
    check_linear(x, w, b, relu=True)
    close(run("matmul", {"a": x, "b": w.t().contiguous()}, {}), x.double() @ w.double().t(),
          x.double().abs() @ w.double().abs().t(), k)
    x = torch.zeros(128 * 65535 + 1, k, device="cuda")
    with pytest.raises(ValueError, match="m too large"):
        run("linear", {"x": x, "w": w}, {})
    with pytest.raises(ValueError, match="m too large"):
        run("matmul", {"a": x, "b": w.t().contiguous()}, {})


# 16 slices per group and part, every one whole: the walks start at different slices; one column less:
# all at the first
@pytest.mark.parametrize("m,n,k", [(3, 2047, 16384), (16, 2048, 16384), (3, 2047, 16380)])
def test_linear_f32_few_rows_over_a_long_k(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(29)
    x, w, b = (torch.randn(s, generator=g, device="cuda") for s in ((m, k), (n, k), (n,)))
    check_linear(x, w, b)
    x[1, k - 5] = float("inf")  # the tiles again with the fp32 instruction
    out = run("linear", {"x": x, "w": w, "b": b}, {})
    assert torch.equal(out[1], float("inf") * w[:, k - 5])
    rest = [0] + list(range(2, m))
    close(out[rest], x[rest].double() @ w.double().t() + b.double(),
          x[rest].double().abs() @ w.double().abs().t() + b.double().abs(), k)
