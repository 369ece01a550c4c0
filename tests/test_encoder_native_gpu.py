"""The encoder's products and norms in pieces (ftc_linear.hip) through the C ABI, against float64;
the encoder's native forward against the composition of its modules."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


class Weight(ctypes.Structure):
    _fields_ = [("w", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("rows", ctypes.c_int64),
                ("cols", ctypes.c_int64), ("pieces", ctypes.c_void_p), ("scale", ctypes.c_void_p),
                ("bias_out", ctypes.c_void_p), ("norm", ctypes.c_void_p)]


def ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else None)


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def whole(pieces, scale):
    rows, cols = pieces.shape
    h = pieces.view(torch.float16).view(rows, cols // 32, 2, 32).double()
    return (h[:, :, 0] + h[:, :, 1]).reshape(rows, cols) * scale.double()[:, None]


PRODUCTS = [
    # tokens, columns, features: edges of the 128 x 256 tile, one to many k-steps, more tiles than
    # workgroups
    (1, 64, 4), (127, 96, 252), (128, 64, 256), (129, 512, 260), (1000, 160, 1536), (70000, 64, 288),
    (300, 1024, 512),
]


@pytest.mark.parametrize("shape", PRODUCTS, ids=lambda s: "t%d_k%d_f%d" % s)
def test_products_in_pieces(shape):
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    gen = torch.Generator(device="cuda").manual_seed(T + K + F)
    x, w, b, r = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,), (T, F)))
    # rows far apart in size, and values far apart within a row
    x *= torch.exp2(torch.randint(-60, 60, (T, 1), device="cuda", generator=gen).float())
    w *= torch.exp2(torch.randint(-20, 20, (F, 1), device="cuda", generator=gen).float())
    x[:, ::3] *= 2.0 ** -12
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    xp, xs, wp, ws, bo, wn = new(T, K), new(T), new(F, K), new(F), new(F), new(F)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), ctypes.c_int64(T), ctypes.c_int64(K), ptr(xp), ptr(xs), stream()) == 0
    for whole_rows, rows in ((whole(xp, xs), x), (whole(wp, ws), w)):
        # one unit in the last place of fp32, or 2^-39 of the row's largest
        assert ((whole_rows - rows.double()).abs() <= 2.0 ** -23 * rows.double().abs()
                + 2.0 ** -39 * rows.double().abs().amax(1, keepdim=True)).all()
    assert torch.equal(bo, b)
    assert ((wn.double() - w.double().abs().sum(1)).abs() <= 1e-5 * w.double().abs().sum(1)).all()

    def run(residual=None, out=None, pieces=None, scale=None):
        rc = lib.ftc_linear_split(ptr(xp), ptr(xs), ctypes.c_int64(T), ptr(wp), ptr(ws), ptr(bo), ptr(wn),
                                  ctypes.c_int64(F), ctypes.c_int64(K), ptr(residual), ptr(out), ptr(pieces),
                                  ptr(scale), stream())
        assert rc == 0, _native.last_error()
    exact = x.double() @ w.double().t()
    # pieces: 2^-23 per value and 2^-24 for lo lo; sums: 2^-24 per rounding of K / 32 + 3 partial sums
    bound = (x.double().abs() @ w.double().abs().t()) * (3 * 2.0 ** -23 + (K / 32 + 3) * 2.0 ** -24) \
        + 2.0 ** -23 * (b.double().abs() + exact.abs())
    out = new(T, F)
    run(out=out)
    assert ((out.double() - (exact + b.double())).abs() <= bound).all()
    run(residual=r, out=out)
    assert ((out.double() - (exact + b.double() + r.double())).abs() <= bound + 2.0 ** -23 * r.double().abs()).all()
    if F % 32 == 0:
        hp, hs = new(T, F), new(T)
        run(pieces=hp, scale=hs)
        # (the row's bound, max|x| max_f sum|w| + max|b|, is at most K + 1 times what the products reach)
        largest = 2 * (x.double().abs().amax(1, keepdim=True) * w.double().abs().sum(1).max() + b.double().abs().max())
        want = (exact + b.double()).clamp_min(0)
        assert ((whole(hp, hs) - want).abs() <= bound + 2.0 ** -22 * want + 2.0 ** -39 * largest).all()


@pytest.mark.parametrize("shape", [
    # the four tiles a product is cut into: more tiles than workgroups and fewer, rows and features that
    # end inside a tile, steps fewer and more than a tile's buffers
    (4990, 512, 1540), (9990, 160, 1536), (4100, 160, 288), (16500, 64, 288), (70001, 96, 260), (129, 96, 544),
    (33, 64, 64)], ids=lambda s: "t%d_k%d_f%d" % s)
def test_products_are_the_same_on_every_tile(shape):
    """A result is a sum in one order whatever tile it lies in: the last rows in a product of their
    own, on the smallest tile, come out bit for bit as in the whole one."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    few = min(T, 31)
    gen = torch.Generator(device="cuda").manual_seed(T)
    x, w, b, r = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,), (T, F)))
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    xp, xs, wp, ws, bo, wn = new(T, K), new(T), new(F, K), new(F), new(F), new(F)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), ctypes.c_int64(T), ctypes.c_int64(K), ptr(xp), ptr(xs), stream()) == 0

    def run(first, residual=None, relu=False):
        out, scale = new(T - first, F), new(T - first)
        rc = lib.ftc_linear_split(ptr(xp[first:]), ptr(xs[first:]), ctypes.c_int64(T - first), ptr(wp), ptr(ws),
                                  ptr(bo), ptr(wn), ctypes.c_int64(F), ctypes.c_int64(K),
                                  ptr(residual[first:]) if residual is not None else None, None if relu else ptr(out),
                                  ptr(out) if relu else None, ptr(scale) if relu else None, stream())
        assert rc == 0, _native.last_error()
        return out, scale
    for more in ({}, {"residual": r}) + (({"relu": True},) if F % 32 == 0 else ()):
        (all_rows, all_scales), (rows, scales) = run(0, **more), run(T - few, **more)
        if "relu" in more:
            assert torch.equal(all_scales[T - few:], scales) and (all_scales > 0).all()
            all_rows, rows = whole(all_rows, all_scales), whole(rows, scales)
        assert not all_rows.isnan().any() and torch.equal(all_rows[T - few:], rows)


@pytest.mark.parametrize("shape", [
    # on the largest tile over more than one round of workgroups, where a tile's rows go out under the next
    # one's products: the fewest steps that have room for that, rows and features that end inside a tile, and a
    # product large enough for its rows to be streamed
    (10237, 320, 1532), (20477, 512, 544), (22600, 512, 1536)], ids=lambda s: "t%d_k%d_f%d" % s)
def test_rows_that_leave_under_the_next_tile(shape):
    """Every row is bit for bit what products of a few thousand rows give (other tiles, rows at once)."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    gen = torch.Generator(device="cuda").manual_seed(T)
    x, w, b = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,)))
    # (one bias beside which some rows' features are too small for pieces under one bound, others' not)
    x *= torch.exp2(torch.randint(-6, 6, (T, 1), device="cuda", generator=gen).float())
    b[F // 2] = 2.0 ** 10
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    xp, xs, wp, ws, bo, wn = new(T, K), new(T), new(F, K), new(F), new(F), new(F)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), ctypes.c_int64(T), ctypes.c_int64(K), ptr(xp), ptr(xs), stream()) == 0

    def run(first, last, relu):
        out, scale = new(last - first, F), new(last - first)
        rc = lib.ftc_linear_split(ptr(xp[first:]), ptr(xs[first:]), ctypes.c_int64(last - first), ptr(wp), ptr(ws),
                                  ptr(bo), ptr(wn), ctypes.c_int64(F), ctypes.c_int64(K), None,
                                  None if relu else ptr(out), ptr(out) if relu else None,
                                  ptr(scale) if relu else None, stream())
        assert rc == 0, _native.last_error()
        return out, scale
    for relu in (False, True) if F % 32 == 0 else (False,):
        rows, scales = run(0, T, relu)
        for first in range(0, T, 2500):
            last = min(first + 2500, T)
            part, part_scales = run(first, last, relu)
            assert torch.equal(rows[first:last].view(torch.int32), part.view(torch.int32))
            if relu:
                assert torch.equal(scales[first:last], part_scales) and (part_scales > 0).all()
        if not relu:
            assert not rows.isnan().any()


def test_relu_keeps_nan_and_takes_any_bias_below_zero():
    """Features switched off by a bias of the type's lowest value or -inf leave the other features'
    precision alone; NaN in a weight or a bias comes out as NaN, as from torch's relu."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = 130, 64, 288
    gen = torch.Generator(device="cuda").manual_seed(8)
    x, w, b = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,)))
    b[3], b[200], b[7], w[260, 5] = float("-inf"), torch.finfo(torch.float32).min, float("nan"), float("nan")
    new = lambda *s: torch.zeros(s, device="cuda")
    xp, xs, wp, ws, bo, wn, hp, hs = new(T, K), new(T), new(F, K), new(F), new(F), new(F), new(T, F), new(T)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), ctypes.c_int64(T), ctypes.c_int64(K), ptr(xp), ptr(xs), stream()) == 0
    assert lib.ftc_linear_split(ptr(xp), ptr(xs), ctypes.c_int64(T), ptr(wp), ptr(ws), ptr(bo), ptr(wn),
                                ctypes.c_int64(F), ctypes.c_int64(K), None, None, ptr(hp), ptr(hs), stream()) == 0
    got, want = whole(hp, hs), torch.relu(x.double() @ w.double().t() + b.double())
    assert torch.equal(got.isnan(), want.isnan()) and want[:, [7, 260]].isnan().all()
    assert (got[:, [3, 200]] == 0).all()
    # K + 1 roundings of sums of absolute products below 200, pieces of the row's bound below 2^-38 of it
    assert (got - want).nan_to_num().abs().max() <= (K + 1) * 2.0 ** -24 * 200


@pytest.mark.parametrize("shape", [(130, 64, 288), (7, 96, 4160), (1, 64, 32)], ids=lambda s: "t%d_k%d_f%d" % s)
@pytest.mark.parametrize("large", ["weight", "bias", "zero_rows"])
def test_relu_features_of_very_different_size(large, shape):
    """A feature with large weights or a large bias leaves the other features of a row where it is
    switched off their precision (a row's pieces hold values down to 2^-17 of the row's largest)."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    gen = torch.Generator(device="cuda").manual_seed(F)
    x, w, b = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,)))
    if large == "weight":       # (off in the rows of odd number)
        w[F // 2] = 2.0 ** 24
        x[::2], x[1::2] = x[::2].abs(), -x[1::2].abs()
    elif large == "bias":       # (off: the row's own product is below minus the bias)
        w[F // 2], b[F // 2] = -2.0 ** 14, 2.0 ** 14
        x[1::2] = x[1::2].abs() + 1
    else:
        x[1::2] = 0
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    xp, xs, wp, ws, bo, wn, hp, hs = new(T, K), new(T), new(F, K), new(F), new(F), new(F), new(T, F), new(T)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), ctypes.c_int64(T), ctypes.c_int64(K), ptr(xp), ptr(xs), stream()) == 0
    assert lib.ftc_linear_split(ptr(xp), ptr(xs), ctypes.c_int64(T), ptr(wp), ptr(ws), ptr(bo), ptr(wn),
                                ctypes.c_int64(F), ctypes.c_int64(K), None, None, ptr(hp), ptr(hs), stream()) == 0
    got, want = whole(hp, hs), torch.relu(x.double() @ w.double().t() + b.double())
    assert (hs > 0).all()
    # as in test_products_in_pieces, and 2^-39 of the row's own largest
    bound = (x.double().abs() @ w.double().abs().t()) * (3 * 2.0 ** -23 + (K / 32 + 3) * 2.0 ** -24) \
        + 2.0 ** -22 * (b.double().abs() + want) + 2.0 ** -39 * want.amax(1, keepdim=True)
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("rows_cols", [(1, 32), (5, 96), (130, 512), (33, 1056), (3, 4096)], ids=lambda s: "r%d_c%d" % s)
def test_layer_norm_in_pieces(rows_cols):
    from fast_transformers_amd import _native
    R, C = rows_cols
    gen = torch.Generator(device="cuda").manual_seed(R + C)
    x, g, b = (torch.randn(*s, device="cuda", generator=gen) for s in ((R, C), (C,), (C,)))
    x = x * 3 + 5
    out, pieces, scale = (torch.full(s, float("nan"), device="cuda") for s in ((R, C), (R, C), (R,)))
    rc = _native.load().ftc_layer_norm_split(ptr(x), ptr(g), ptr(b), ctypes.c_float(1e-5), ctypes.c_int64(R),
                                             ctypes.c_int64(C), ptr(out), ptr(pieces), ptr(scale), stream())
    assert rc == 0, _native.last_error()
    want = torch.nn.functional.layer_norm(x.double(), (C,), g.double(), b.double(), 1e-5)
    plain = torch.nn.functional.layer_norm(x, (C,), g, b, 1e-5).double()
    assert (out.double() - want).abs().max() <= max(4 * (plain - want).abs().max(), 2e-6)
    assert (whole(pieces, scale) - out.double()).abs().max() <= 2.0 ** -23 * out.double().abs().max()


@pytest.mark.parametrize("sizes", [(2, 300, 2, 8, 64, 64, 1024), (3, 129, 3, 4, 32, 32, 512), (1, 7, 1, 4, 64, 32, 96)],
                         ids=lambda s: "n%d_l%d_x%d_h%d_e%d_m%d_f%d" % s)
@pytest.mark.parametrize("ragged", [False, True], ids=["full", "ragged"])
@pytest.mark.parametrize("final", [True, False], ids=["final_norm", "no_norm"])
def test_encoder_native_forward(sizes, ragged, final):
    from fast_transformers_amd import attention, masking
    N, L, layers, H, E, M, ff = sizes
    torch.manual_seed(L)
    with torch.device("cuda"):
        model = attention.build_causal_linear_encoder(layers, H, E, M, ff, final_normalization=final).eval()
    x = torch.rand(N, L, H * M, device="cuda")
    mask = masking.TriangularCausalMask(L, device="cuda")
    lengths = masking.LengthMask(torch.randint(1, L + 1, (N,), device="cuda"), max_len=L) if ragged else None
    calls = []
    from fast_transformers_amd.attention import encoder as module
    native = module.encoder_forward_hip
    module.encoder_forward_hip = lambda *a: (calls.append(1), native(*a))[1]
    try:
        with torch.no_grad():
            got = model(x, attn_mask=mask, length_mask=lengths)
            assert calls == [1]
            # a hook on any part asks for the modules themselves
            handle = model.layers[0].linear1.register_forward_hook(lambda *a: None)
            want = model(x, attn_mask=mask, length_mask=lengths)
            handle.remove()
        assert calls == [1]
        # something to differentiate: the modules
        out = model(x, attn_mask=mask, length_mask=lengths)
        assert calls == [1] and out.requires_grad
        with pytest.raises(RuntimeError):
            model(x, length_mask=lengths)          # not causal: refused as before
    finally:
        module.encoder_forward_hip = native
    # two fp32 evaluations: 1e-6 per layer of the largest value (norms keep rows near one)
    assert (got - want).abs().max() <= 4e-6 * layers * want.abs().max()


def small_encoder(monkeypatch):
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import encoder as module
    torch.manual_seed(3)
    with torch.device("cuda"):
        model = attention.build_causal_linear_encoder(2, 2, 32, 32, 64).eval().requires_grad_(False)
    calls, native = [], module.encoder_forward_hip
    monkeypatch.setattr(module, "encoder_forward_hip", lambda *a: (calls.append(1), native(*a))[1])
    return model, masking.TriangularCausalMask(40, device="cuda"), calls


@pytest.mark.parametrize("form", ["offset", "permuted", "strided"])
def test_encoder_takes_any_layout_of_its_input(monkeypatch, form):
    model, mask, calls = small_encoder(monkeypatch)
    rows = torch.rand(2, 40, 64, device="cuda")
    if form == "offset":  # dense, and four bytes off a boundary of sixteen
        x = torch.empty(2 * 40 * 64 + 1, device="cuda")[1:].view(2, 40, 64).copy_(rows)
    elif form == "permuted":
        x = rows.permute(2, 0, 1).contiguous().permute(1, 2, 0)
    else:
        x = torch.empty(2, 40, 65, device="cuda")[..., :64].copy_(rows)
    assert torch.equal(model(x, attn_mask=mask), model(rows, attn_mask=mask)) and len(calls) == 2


def test_encoder_keeps_its_modules_where_operations_are_observed(monkeypatch):
    from torch.utils.flop_counter import FlopCounterMode
    model, mask, calls = small_encoder(monkeypatch)
    x = torch.rand(2, 40, 64, device="cuda")
    with torch.device("cuda"):
        want = model(x, attn_mask=mask)
    assert calls == [1]
    with FlopCounterMode(display=False) as flops:
        got = [model(x, attn_mask=mask)]
    assert flops.get_total_flops() > 0
    with torch.autograd.forward_ad.dual_level():
        got.append(model(x, attn_mask=mask))
    inner = model.layers[1].linear2
    inner.forward = lambda y: type(inner).forward(inner, y)
    got.append(model(x, attn_mask=mask))
    assert calls == [1]
    # two fp32 evaluations, as above
    assert all((g - want).abs().max() <= 8e-6 * want.abs().max() for g in got)


@pytest.mark.parametrize("cls", ["Linear", "LayerNorm", "Dropout"])
def test_encoder_keeps_its_modules_where_a_class_has_another_forward(monkeypatch, cls):
    model, mask, calls = small_encoder(monkeypatch)
    x = torch.rand(2, 40, 64, device="cuda")
    cls, seen = getattr(torch.nn, cls), []
    plain = cls.forward
    monkeypatch.setattr(cls, "forward", lambda self, y: (seen.append(1), plain(self, y))[1])
    model(x, attn_mask=mask)
    assert seen and not calls


def test_encoder_takes_a_mask_that_only_says_it_is_causal(monkeypatch):
    from types import SimpleNamespace
    model, mask, calls = small_encoder(monkeypatch)
    x = torch.rand(2, 40, 64, device="cuda")
    got = model(x, attn_mask=SimpleNamespace(lower_triangular=True))
    want = model(x, attn_mask=mask)
    assert (got - want).abs().max() <= 8e-6 * want.abs().max()  # (two fp32 evaluations, as above)


def test_encoder_keeps_its_modules_beyond_the_native_sizes(monkeypatch):
    from fast_transformers_amd import attention, masking, _native
    model, _, calls = small_encoder(monkeypatch)
    N, L = 1 << 13, 1 << 13   # 2^26 rows, as a view of one (none of them is read)
    x = torch.rand(1, 1, 64, device="cuda").expand(N, L, 64)
    assert model._fused_forward(x, masking.TriangularCausalMask(L, device="cuda"), None) is None
    with torch.device("cuda"):
        wide = attention.build_causal_linear_encoder(1, 2, 32, 32, (1 << 20) + 32).eval().requires_grad_(False)
    assert wide(x[:1, :3], attn_mask=masking.TriangularCausalMask(3, device="cuda")).shape == (1, 3, 64) and not calls
    # the C entries refuse them before they launch anything
    room = torch.zeros(64, device="cuda")
    lib, some, big, n = _native.load(), ptr(room), ctypes.c_int64((1 << 20) + 32), ctypes.c_int64(64)
    assert lib.ftc_linear_split(some, some, n, some, some, some, some, big, n, None, some, None, None, stream()) == -2
    assert lib.ftc_linear_split(some, some, n, some, some, some, some, n, big, None, some, None, None, stream()) == -2
    assert lib.ftc_split_rows(some, ctypes.c_int64(1 << 26), n, some, some, stream()) == -2
    for rows, cols in ((64, big.value), (big.value, 64)):
        item = Weight(some.value, None, rows, cols, some.value, some.value, some.value, some.value)
        assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == -2


@pytest.mark.parametrize("final", [True, False], ids=["final_norm", "no_norm"])
@pytest.mark.parametrize("ff", [512, 1024, 2048])
def test_encoder_needs_no_more_memory_than_its_modules(ff, final):
    from fast_transformers_amd import attention, masking
    with torch.device("cuda"):
        model = attention.build_causal_linear_encoder(3, 8, 64, 64, ff, final_normalization=final).eval()
    model.requires_grad_(False)
    x, mask = torch.rand(10, 2048, 512, device="cuda"), masking.TriangularCausalMask(2048, device="cuda")

    def peak():
        model(x, attn_mask=mask)     # (workspaces and library handles stay)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        model(x, attn_mask=mask)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before
    native = peak()
    handle = model.layers[0].linear1.register_forward_hook(lambda *a: None)
    modules = peak()
    handle.remove()
    # (a layer's weights in pieces and the scales of the rows come on top)
    weights = 4 * 512 * (4 * 512 + 2 * ff + 16) + 2 * 4 * x.shape[0] * x.shape[1]
    assert native <= modules + 1.1 * weights


@pytest.mark.parametrize("count", [1, 47, 48])
def test_weights_of_many_matrices_are_cut_in_one_launch(count):
    """Each matrix comes out as in a launch of its own, whatever its number and whatever stands beside it."""
    from fast_transformers_amd import _native
    lib = _native.load()
    gen = torch.Generator(device="cuda").manual_seed(count)
    kept, items, alone = [], (Weight * count)(), (Weight * 1)()
    for i in range(count):
        F, K = 4 * (1 + i % 9), 32 * (1 + i % 5)
        w, b = torch.randn(F, K, device="cuda", generator=gen), torch.randn(F, device="cuda", generator=gen)
        outs = [[torch.full(s, float("nan"), device="cuda") for s in ((F, K), (F,), (F,), (F,))] for _ in range(2)]
        for item, (p, s, bo, n) in ((items[i], outs[0]), (alone[0], outs[1])):
            item.w, item.bias, item.rows, item.cols = w.data_ptr(), b.data_ptr() if i % 2 else None, F, K
            item.pieces, item.scale, item.bias_out, item.norm = (t.data_ptr() for t in (p, s, bo, n))
        assert lib.ftc_split_weights(alone, 1, stream()) == 0
        kept.append((w, b, outs))
    assert lib.ftc_split_weights(items, count, stream()) == 0, _native.last_error()
    for w, b, (together, single) in kept:
        for x, y in zip(together, single):
            assert torch.equal(x.view(torch.int32), y.view(torch.int32))
        assert (whole(*together[:2]) - w.double()).abs().max() <= 2.0 ** -22 * w.abs().max()
    assert lib.ftc_split_weights((Weight * 49)(), 49, stream()) == -1


@pytest.mark.parametrize("weights", ["both", "beta", "none"])
@pytest.mark.parametrize("shape", [
    # tokens, columns, features: each of the four tiles, rows and features that end inside one, more tiles than
    # workgroups, steps fewer and more than a tile's buffers
    (4990, 512, 1536), (9990, 160, 1536), (4100, 160, 288), (70001, 96, 256), (129, 96, 544), (33, 64, 64), (1, 64, 32)],
    ids=lambda s: "t%d_k%d_f%d" % s)
def test_a_norm_that_is_added_is_the_norm_that_was_stored(shape, weights):
    """Products that make a layer norm's rows again from (mean, r) add the same values, bit for bit, as from its rows,
    also where their own go over the rows before the norm."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    gen = torch.Generator(device="cuda").manual_seed(T + F)
    x, w, b, r = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,), (T, F)))
    r = r * 3 + 5 * torch.randn(T, 1, device="cuda", generator=gen)
    gamma = torch.randn(F, device="cuda", generator=gen) if weights == "both" else None
    beta = torch.randn(F, device="cuda", generator=gen) if weights != "none" else None
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    n = lambda i: ctypes.c_int64(i)
    xp, xs, wp, ws, bo, wn = new(T, K), new(T), new(F, K), new(F), new(F), new(F)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), n(T), n(K), ptr(xp), ptr(xs), stream()) == 0
    rows, pieces, scale, stats, pieces2, scale2 = new(T, F), new(T, F), new(T), new(T, 2), new(T, F), new(T)
    eps = ctypes.c_float(1e-5)
    assert lib.ftc_layer_norm_split(ptr(r), ptr(gamma), ptr(beta), eps, n(T), n(F), ptr(rows), ptr(pieces), ptr(scale), stream()) == 0
    assert lib.ftc_layer_norm_stats_split(ptr(r), ptr(gamma), ptr(beta), eps, n(T), n(F), ptr(stats), ptr(pieces2),
                                          ptr(scale2), stream()) == 0, _native.last_error()
    assert torch.equal(pieces.view(torch.int32), pieces2.view(torch.int32)) and torch.equal(scale, scale2)
    want, got = new(T, F), new(T, F)
    assert lib.ftc_linear_split(ptr(xp), ptr(xs), n(T), ptr(wp), ptr(ws), ptr(bo), ptr(wn), n(F), n(K), ptr(rows),
                                ptr(want), None, None, stream()) == 0
    for out in (got, r):
        assert lib.ftc_linear_split_normed(ptr(xp), ptr(xs), n(T), ptr(wp), ptr(ws), ptr(bo), n(F), n(K), ptr(r), ptr(stats),
                                           ptr(gamma), ptr(beta), ptr(out), stream()) == 0, _native.last_error()
        assert torch.equal(out, want)


@pytest.mark.parametrize("final", [True, False], ids=["final_norm", "no_norm"])
@pytest.mark.parametrize("sizes", [
    # d, heads, E, M, feed-forward: d beyond the heads' widths and the feed-forward width, by much and by a block;
    # beyond one of them; heads beyond d and the feed-forward width
    (512, 2, 32, 32, 128), (224, 2, 32, 32, 64), (512, 2, 64, 64, 1024), (256, 4, 64, 64, 64), (128, 8, 32, 64, 64)],
    ids=lambda s: "d%d_h%d_e%d_m%d_f%d" % s)
def test_encoder_whose_width_is_not_that_of_its_heads(sizes, final):
    """The model's width, the heads' and the feed-forward width are independent of each other: rows of any of them
    find room, and nothing beside them changes."""
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import encoder as module
    d, H, E, M, ff = sizes
    N, L, layers = 3, 130, 2
    torch.manual_seed(d + H)
    with torch.device("cuda"):
        model = attention.TransformerEncoder(
            [attention.TransformerEncoderLayer(
                attention.AttentionLayer(attention.CausalLinearAttention(E), d, H, d_keys=E, d_values=M), d, ff)
             for _ in range(layers)], torch.nn.LayerNorm(d) if final else None).eval().requires_grad_(False)
    x, mask = torch.rand(N, L, d, device="cuda"), masking.TriangularCausalMask(L, device="cuda")
    calls, native = [], module.encoder_forward_hip
    module.encoder_forward_hip = lambda *a: (calls.append(1), native(*a))[1]
    try:
        got = model(x, attn_mask=mask)
        assert calls == [1]
        handle = model.layers[0].linear1.register_forward_hook(lambda *a: None)
        want = model(x, attn_mask=mask)
        handle.remove()
    finally:
        module.encoder_forward_hip = native
    assert calls == [1]
    # two fp32 evaluations, as above
    assert (got - want).abs().max() <= 4e-6 * layers * want.abs().max()


@pytest.mark.parametrize("kind", ["plain", "residual", "norm", "relu"])
@pytest.mark.parametrize("shape", [
    # products of more than 176 MB, whose rows leave in whole lines past the caches: rows that are added on the two
    # largest tiles, features that end inside a line, too few steps for rows to leave under the next tile
    (26000, 512, 676), (45003, 512, 512), (60011, 256, 544), (31000, 1024, 352)], ids=lambda s: "t%d_k%d_f%d" % s)
def test_streamed_rows(shape, kind):
    """Rows that are streamed are bit for bit those of products too small for it, also over the rows that they add."""
    from fast_transformers_amd import _native
    lib = _native.load()
    T, K, F = shape
    relu, adds = kind == "relu", kind in ("residual", "norm")
    if relu:
        F = F // 32 * 32
    assert 4 * T * (K + (2 if adds else 1) * F) >= 176 << 20 or not adds
    gen = torch.Generator(device="cuda").manual_seed(T + F)
    x, w, b, r = (torch.randn(*s, device="cuda", generator=gen) for s in ((T, K), (F, K), (F,), (T, F)))
    gamma, beta = torch.randn(F, device="cuda", generator=gen), torch.randn(F, device="cuda", generator=gen)
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    n = lambda i: ctypes.c_int64(i)
    xp, xs, wp, ws, bo, wn = new(T, K), new(T), new(F, K), new(F), new(F), new(F)
    item = Weight(w.data_ptr(), b.data_ptr(), F, K, wp.data_ptr(), ws.data_ptr(), bo.data_ptr(), wn.data_ptr())
    assert lib.ftc_split_weights(ctypes.byref(item), 1, stream()) == 0, _native.last_error()
    assert lib.ftc_split_rows(ptr(x), n(T), n(K), ptr(xp), ptr(xs), stream()) == 0
    stats = torch.stack((r.mean(1), 1 / r.std(1)), 1).contiguous()   # (any two numbers a row will do)

    def run(first, last, out, scale):
        rows, at = n(last - first), slice(first, last)
        if kind == "norm":
            rc = lib.ftc_linear_split_normed(ptr(xp[at]), ptr(xs[at]), rows, ptr(wp), ptr(ws), ptr(bo), n(F), n(K),
                                             ptr(r[at]), ptr(stats[at]), ptr(gamma), ptr(beta), ptr(out), stream())
        else:
            rc = lib.ftc_linear_split(ptr(xp[at]), ptr(xs[at]), rows, ptr(wp), ptr(ws), ptr(bo), ptr(wn), n(F), n(K),
                                      ptr(r[at]) if adds else None, None if relu else ptr(out),
                                      ptr(out) if relu else None, ptr(scale) if relu else None, stream())
        assert rc == 0, _native.last_error()
    want, want_scale, got, got_scale = new(T, F), new(T), new(T, F), new(T)
    for first in range(0, T, 5000):
        last = min(first + 5000, T)
        run(first, last, want[first:last], want_scale[first:last])
    for out in (got, r) if adds else (got,):
        run(0, T, out, got_scale)
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
    if relu:
        assert torch.equal(got_scale, want_scale) and (got_scale > 0).all()
    else:
        assert not got.isnan().any()


def test_encoder_of_few_tokens_needs_little_more_memory_than_its_modules():
    """Up to eight layers have their weights in pieces at a time: at most 64 MB of them."""
    from fast_transformers_amd import attention, masking
    with torch.device("cuda"):
        model = attention.build_causal_linear_encoder(12, 8, 64, 64, 1024).eval().requires_grad_(False)
    x, mask = torch.rand(4, 338, 512, device="cuda"), masking.TriangularCausalMask(338, device="cuda")

    def peak():
        model(x, attn_mask=mask)     # (workspaces and library handles stay)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        model(x, attn_mask=mask)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before
    native = peak()
    handle = model.layers[0].linear1.register_forward_hook(lambda *a: None)
    modules = peak()
    handle.remove()
    assert native <= modules + (64 << 20) + 2 * 4 * x.shape[0] * x.shape[1]
