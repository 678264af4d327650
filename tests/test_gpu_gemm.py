"""The linear layers' matrix products (ops.gemm) and the layers on them (linear.linear): every order, tile shape, type and way of combining products, at the
edges of tiles and at the rows that the choice of products turns on.

Tolerances.  A product is one rounding of an fp32 sum of exact products.  That rounding is at most half a unit in the last of 8 (bf16) or 11 (fp16) bits,
2^-9 = 1.95e-3 or 2^-12 = 2.4e-4 of the value, and so is the relative L2 error against the fp64 product of the same inputs; the fp32 sums add some 1e-6.
"""
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu
REL = {torch.bfloat16: 2e-3, torch.float16: 2.6e-4}


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


def _matrix(g, rows, cols, dtype, ld=None):
    """rows x cols, in lines of ld elements whose rest is not a number."""
    m = torch.full((rows, ld or cols), float("nan"), device="cuda", dtype=dtype)
    m[:, :cols] = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
    return m[:, :cols]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [1, 2, 3, 4])
@pytest.mark.parametrize("order", ["xwt", "xw", "xtx"])
@pytest.mark.parametrize("rows, cols, depth, count, total", [
    (1, 8, 64, 1, False),            # smaller than any tile, one step
    (264, 520, 128, 3, False),       # a tile and a few rows and columns more; two steps
    (257, 136, 448, 2, True),        # products summed: steps of one after the other
    (2304, 256, 192, 1, False),      # a full group of rows of tiles and one more
])
def test_products(pkg, order, shape, dtype, rows, cols, depth, count, total):
    ops = pkg.ops
    g = torch.Generator(device="cuda").manual_seed(rows + depth)
    if order == "xtx":
        rows, depth = (rows + 7) // 8 * 8, depth + (5 if depth > 64 else 0)        # any depth; rows in eights
    ld = 1024                        # (operands whose lines run along the output need lines of at least 256)
    a_shape = (depth, rows) if order == "xtx" else (rows, depth)
    b_shape = (cols, depth) if order == "xwt" else (depth, cols)
    a = [_matrix(g, *a_shape, dtype, 2304 if a_shape[1] > ld else ld) for _ in range(count)]
    b = [_matrix(g, *b_shape, dtype, ld) for _ in range(count)]
    got = ops.gemm(order, a, b, total=total, shape=shape)
    left = [x.double().t() if order == "xtx" else x.double() for x in a]
    want = [x @ (y.double().t() if order == "xwt" else y.double()) for x, y in zip(left, b)]
    for y, w in zip([got] if total else got, [sum(want)] if total else want):
        assert torch.isfinite(y).all() and _rel(y, w) < REL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape, rows, cols", [(1, 4360, 4360), (2, 4360, 4360), (3, 4360, 4360), (4, 4360, 4360), (4, 264, 33032)])
@pytest.mark.parametrize("order", ["xwt", "xw", "xtx"])
def test_products_of_more_tiles_than_workgroups(pkg, order, shape, rows, cols, dtype):
    """Workgroups that walk several tiles: their loads, waits (which count the stores of the tile before) and accumulators over a tile's end.  256 workgroups, of 128 x 128 tiles
    512; 324, 630, 630, 1225 and 777 tiles.  Steps per tile: one (every step a tile's first), two and five, in one product, three products and sums of two and three."""
    ops = pkg.ops
    g = torch.Generator(device="cuda").manual_seed(shape)
    wide = {1: (256, 256), 2: (256, 128), 3: (128, 256), 4: (128, 128)}[shape]
    assert -(-rows // wide[0]) * -(-cols // wide[1]) > (512 if shape == 4 else 256)
    for depth, count, total in ((64, 1, False), (64, 3, True), (128, 2, True), (320, 1, False), (128, 3, False)):
        depth += 5 if order == "xtx" and depth > 64 else 0
        a_shape, b_shape = (depth, rows) if order == "xtx" else (rows, depth), (cols, depth) if order == "xwt" else (depth, cols)
        a, b = [_matrix(g, *a_shape, dtype) for _ in range(count)], [_matrix(g, *b_shape, dtype, b_shape[1] + -b_shape[1] % 8) for _ in range(count)]
        got = ops.gemm(order, a, b, total=total, shape=shape)
        want = [(x.double().t() if order == "xtx" else x.double()) @ (y.double().t() if order == "xwt" else y.double()) for x, y in zip(a, b)]
        for y, w in zip([got] if total else got, [sum(want)] if total else want):
            assert torch.isfinite(y).all() and _rel(y, w) < REL[dtype]
            # (a tile that is wrong as a whole would be a few thousandths of all: every block of rows and of columns by itself as well)
            d = (y.double() - w).pow(2)
            for dim in (0, 1):
                assert (d.sum(dim) <= (4 * REL[dtype]) ** 2 * w.pow(2).sum(dim)).all()


def test_refused_matrices(pkg):
    ops = pkg.ops
    m = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)
    for order, a, b in (("xwt", m(64, 72), m(64, 72)),              # contraction not in 64s
                        ("xwt", m(64, 64), m(12, 64)),              # columns not in eights
                        ("xtx", m(64, 12), m(64, 256))):            # rows not in eights
        with pytest.raises(AssertionError):
            ops.gemm(order, [a], [b])
        assert ops.gemm(order, [a], [b], if_preferred=True) is None
    with pytest.raises(NotImplementedError):                        # lines along the output shorter than the loads' offsets
        ops.gemm("xw", [m(64, 64)], [m(64, 128)])
    with pytest.raises(ValueError):
        ops.gemm("xwt", [m(64, 64)], [m(64, 128)])


def _layers(n, depth, cols, dtype):
    torch.manual_seed(3)
    return [nn.Linear(depth, cols, bias=False, device="cuda", dtype=dtype) for _ in range(n)]


# rows on both sides of where the products of a layer, and of its backward pass, become the package's own
@pytest.mark.parametrize("rows", [255, 264, 1024, 1560, 8200])
@pytest.mark.parametrize("n, depth, cols", [(1, 512, 1024), (3, 512, 512), (1, 1024, 4608)])
def test_layers_and_gradients(pkg, rows, n, depth, cols):
    from sys import modules
    linear = modules[pkg.__name__ + ".linear"].linear
    layers = _layers(n, depth, cols, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(2, rows // 2 if rows % 2 == 0 else rows, depth, device="cuda", generator=g).bfloat16()
    with torch.no_grad():
        values = linear(layers, x)
    x.requires_grad_(True)
    ys = linear(layers, x)
    dys = [torch.randn(y.shape, device="cuda", generator=g).bfloat16() for y in ys]
    grads = torch.autograd.grad(ys, [x] + [m.weight for m in layers], dys)
    xd, wd = x.detach().double().reshape(-1, depth), [m.weight.detach().double() for m in layers]
    dd = [d.double().reshape(-1, cols) for d in dys]
    for y, v, w in zip(ys, values, wd):
        assert torch.equal(y, v) and y.shape == (*x.shape[:-1], cols) and _rel(y.detach().reshape(-1, cols), xd @ w.t()) < 2e-3
    # (the library's three products are rounded one by one and their two additions again: no more than three roundings of the whole)
    assert _rel(grads[0].reshape(-1, depth), sum(d @ w for d, w in zip(dd, wd))) < 2e-3 * (1 if n == 1 else 3)
    for gw, d in zip(grads[1:], dd):
        assert _rel(gw, d.t() @ xd) < 2e-3


def test_layer_gradients_of_a_part_and_twice(pkg):
    """One output without a gradient, frozen weights, gradients that are differentiated again, and a gradient that is not dense."""
    from sys import modules
    linear = modules[pkg.__name__ + ".linear"].linear
    layers = _layers(3, 512, 512, torch.bfloat16)
    layers[1].weight.requires_grad_(False)
    x = torch.randn(1040, 512, device="cuda").bfloat16().requires_grad_(True)
    q, k, v = linear(layers, x)
    dx, dw = torch.autograd.grad(q.sum() + 2 * k.sum(), [x, layers[0].weight])
    ones = torch.ones(1040, 512, device="cuda", dtype=torch.float64)
    assert _rel(dx, ones @ layers[0].weight.detach().double() + 2 * ones @ layers[1].weight.detach().double()) < 3 * 2e-3
    assert _rel(dw, ones.t() @ x.detach().double()) < 2e-3
    (dx,) = torch.autograd.grad((linear(layers[:1], x)[0] ** 2).sum() / 512, x, create_graph=True)
    (ddx,) = torch.autograd.grad(dx.square().sum(), x)          # y = x w^T, dx = 2 y w / 512, ddx = 2 (2 / 512)^2 x (w^T w)^2
    h = layers[0].weight.detach().double()
    h = h.t() @ h * (2 / 512)
    # (four products in a row, each rounded)
    assert _rel(ddx, 2 * x.detach().double() @ h @ h) < 4 * 2e-3


def test_layer_gradients_of_dual_cotangents(pkg):
    """A graph recorded outside of any dual level, its gradients then dual: their tangents come through where the own products are preferred.  (Batched
    cotangents: on the CPU, test_host.py.)"""
    from sys import modules
    from torch.autograd import forward_ad as fwad
    linear = modules[pkg.__name__ + ".linear"].linear
    layers = _layers(3, 512, 512, torch.bfloat16)
    rn = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    x, dy, tdy = rn(1560, 512).requires_grad_(True), [rn(1560, 512) for _ in layers], [rn(1560, 512) for _ in layers]
    ys, wrt = linear(layers, x), [x] + [m.weight for m in layers]
    assert pkg.ops.gemm("xw", dy, [m.weight.detach() for m in layers], total=True, if_preferred=True) is not None
    plain = [torch.autograd.grad(ys, wrt, d, retain_graph=True) for d in (dy, tdy)]
    with fwad.dual_level():
        got = [fwad.unpack_dual(t) for t in torch.autograd.grad(ys, wrt, [fwad.make_dual(d, t) for d, t in zip(dy, tdy)])]
    for i, pair in enumerate(got):        # (the gradients are linear in the cotangent)
        for part, want in zip(pair, (plain[0][i], plain[1][i])):
            assert part is not None and _rel(part, want.double()) < 4 * 2e-3       # (up to three roundings on one side, one on the other)


@pytest.mark.parametrize("how", ["hook", "subclass", "bias", "autocast", "float", "strided", "jvp", "vmap", "flops", "function mode"])
def test_layers_with_a_meaning_of_their_own_go_through_the_module(pkg, how):
    from sys import modules
    lin = modules[pkg.__name__ + ".linear"]
    dtype = torch.float32 if how == "float" else torch.bfloat16
    (m,) = _layers(1, 512, 512, dtype)
    x = torch.randn(2048, 512, device="cuda").to(dtype)
    calls = []
    if how == "hook":
        m.register_forward_hook(lambda *a: calls.append(1))
    if how == "subclass":
        class Scaled(nn.Linear):
            def forward(self, x):
                return 2 * super().forward(x)
        m.__class__ = Scaled
    if how == "bias":
        m.bias = nn.Parameter(torch.ones(512, device="cuda", dtype=dtype))
    if how == "strided":
        x = torch.randn(2048, 1024, device="cuda").to(dtype)[:, ::2]
    with torch.no_grad():
        if how == "jvp":
            got = torch.func.jvp(lambda t: lin.linear([m], t)[0], (x,), (x,))
            want = torch.func.jvp(lambda t: m(t), (x,), (x,))
        elif how == "vmap":
            t = x.view(2, 1024, 512)
            got, want = (torch.func.vmap(lambda t: lin.linear([m], t)[0])(t),), (torch.func.vmap(m)(t),)
        elif how == "flops":
            from torch.utils.flop_counter import FlopCounterMode
            with FlopCounterMode(display=False) as counter:
                got, want = (lin.linear([m], x)[0],), (m(x),)
            assert counter.get_total_flops() == 2 * 2 * 2048 * 512 * 512
        elif how == "function mode":
            class Doubled(torch.overrides.TorchFunctionMode):
                def __torch_function__(self, fn, types, args=(), kwargs=None):
                    y = fn(*args, **(kwargs or {}))
                    return 2 * y if fn is torch.nn.functional.linear else y
            with Doubled():
                got, want = (lin.linear([m], x)[0],), (m(x),)
        else:
            with torch.autocast("cuda", dtype=torch.float16, enabled=how == "autocast"):
                got, want = (lin.linear([m], x)[0],), (m(x),)
    assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(got, want))
    assert how != "hook" or len(calls) == 2


@pytest.mark.parametrize("how", ["one frame", "one row", "slice"])
def test_layers_of_dense_inputs_with_strides_of_their_own(pkg, how):
    """Dense is what is_contiguous calls so: a dimension of one has any stride."""
    from sys import modules
    lin = modules[pkg.__name__ + ".linear"]
    (m,) = _layers(1, 512, 512, torch.bfloat16)
    x = torch.randn(1, 2048, 512, device="cuda").bfloat16()
    x = {"one frame": x.transpose(0, 1), "one row": x.view(2048, 1, 512).as_strided((2048, 1, 512), (512, 8, 1)), "slice": x[:, 8:1600]}[how]
    assert x.is_contiguous() and lin._own(x.shape[:-1].numel(), 512, 512, 1, False)[0]
    with torch.no_grad():
        got = lin.linear([m], x)[0]
    assert got.shape == x.shape and _rel(got, x.double() @ m.weight.double().t()) < 2e-3
    x = x.clone(memory_format=torch.preserve_format).requires_grad_(True)
    dx, dw = torch.autograd.grad(lin.linear_one(m, x), [x, m.weight], got)
    g, w = got.double().reshape(-1, 512), m.weight.detach().double()
    assert _rel(dx.reshape(-1, 512), g @ w) < 2e-3 and _rel(dw, g.t() @ x.detach().double().reshape(-1, 512)) < 2e-3


def test_products_replayed_from_a_graph(pkg):
    ops = pkg.ops
    a, b = torch.randn(1560, 512, device="cuda").bfloat16(), torch.randn(768, 512, device="cuda").bfloat16()
    want = ops.gemm("xwt", [a], [b])[0]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        (y,) = ops.gemm("xwt", [a], [b])
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        a.copy_(a.flip(0))
        want = ops.gemm("xwt", [a], [b])[0]
