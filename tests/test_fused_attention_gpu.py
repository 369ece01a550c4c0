"""ftc_causal_linear_attention: feature map, key-length mask, causal product and normaliser in
one launch, called through the C ABI and checked against

(a) the outputs of the reference's own CausalLinearAttention
    (tests/golden/attention_causal_linear.npz, written by tests/golden/make_encoder_golden.py),
(b) the CPU restatement ``oracle.causal_linear_attention`` (float32 as the reference runs it,
    float64 as the anchor) on seeded inputs: every supported pair of head dimensions,
    chunk and segment boundaries, ragged / zero / over-long key lengths, (N, L, H, X) views,
(c) properties that hold at any size: rows are weighted means of the values seen so far
    (constant values come back unchanged), prefix property, independence of masked keys,
and, at module level, against the composition of separate operator calls that training uses.

Tolerance: 1e-4 relative to the largest magnitude of the chain (fp32 bar of the operator),
and an element-wise violation fraction (1e-5 + 1e-4 |want|) no worse than twice what the
float32 CPU restatement shows against float64, plus 6e-4.
"""
import ctypes
import math
import os

import numpy as np
import pytest
import torch

import oracle
from parity import scale_error, violation_fraction

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU")
    from fast_transformers_amd import _native
    return _native.load()


def fused(lib, q, k, v, lengths, eps, out=None):
    """q, k, v: (N, L, H, X) device tensors (any strides the ABI takes); straight C ABI call."""
    from fast_transformers_amd import _native
    N, L, H, E = q.shape
    M = v.shape[3]
    if out is None:
        out = torch.full((N, L, H, M), float("nan"), device=q.device, dtype=torch.float32)
    nbytes = lib.ftc_causal_linear_attention_workspace_bytes(N, H, L, E, M, _native.FTC_F32)
    assert nbytes >= 0, _native.last_error()
    ws = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=q.device)
    d = [_native.describe(t.permute(0, 2, 1, 3)) for t in (q, k, v, out)]
    rc = lib.ftc_causal_linear_attention(
        ctypes.byref(d[0]), ctypes.byref(d[1]), ctypes.byref(d[2]),
        ctypes.c_void_p(lengths.data_ptr()) if lengths is not None else None,
        ctypes.c_float(eps), ctypes.byref(d[3]), ctypes.c_void_p(ws.data_ptr()), nbytes,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.last_error()
    torch.cuda.synchronize()
    assert int(ws[8:12].view(torch.int32).item()) == 0, "a wavefront gave up waiting"
    return out


def inputs(N, L, H, E, M, seed, scale=1.5):
    gen = torch.Generator().manual_seed(seed)
    q = scale * torch.randn(N, L, H, E, generator=gen)
    k = scale * torch.randn(N, L, H, E, generator=gen)
    v = torch.randn(N, L, H, M, generator=gen)
    return q, k, v


def gate(got, q, k, v, lengths, eps):
    """got: (N, L, H, M) on the host."""
    want32 = oracle.causal_linear_attention(q, k, v, lengths, eps)
    want64 = oracle.causal_linear_attention(q.double(), k.double(), v.double(), lengths, eps)
    nhl = lambda t: t.permute(0, 2, 1, 3)
    assert torch.isfinite(got).all()
    assert scale_error(nhl(got), nhl(want32)) <= 1e-4
    assert scale_error(nhl(got), nhl(want64)) <= max(4 * scale_error(nhl(want32), nhl(want64)), 2e-6)
    v_ref = violation_fraction(want32, want64)
    assert violation_fraction(got, want64) <= 2 * v_ref + 6e-4
    assert violation_fraction(got, want32) <= 2 * v_ref + 6e-4


def test_against_the_reference_modules_outputs(lib):
    data = np.load(os.path.join(os.path.dirname(__file__), "golden", "attention_causal_linear.npz"))
    q, k, v, y = (torch.from_numpy(data["b_" + x]) for x in ("q", "k", "v", "y"))
    lengths = torch.from_numpy(data["b_lengths"])
    got = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), float(data["b_eps"])).cpu()
    assert (got - y).abs().max().item() <= 1e-4 * max(1.0, y.abs().max().item())
    assert violation_fraction(got, y) == 0.0


SHAPES = [
    # N, L, H, E, M, key lengths (None: all)
    (2, 1, 2, 64, 64, None),
    (2, 31, 3, 64, 64, [31, 7]),
    (1, 32, 2, 64, 32, [32]),
    (3, 33, 1, 32, 64, [33, 0, 32]),
    (2, 100, 4, 32, 32, [64, 100]),
    (2, 1000, 8, 64, 64, [1000, 517]),
    (1, 4096, 2, 64, 64, [3000]),          # several segments; the length cuts one of them
    (2, 4100, 3, 32, 64, [4100, 33]),      # whole segments beyond the length
    (1, 2500, 5, 64, 32, [9999]),          # longer than the sequence: every key counts
    (3, 777, 2, 32, 32, None),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_against_the_cpu_restatement(lib, shape):
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=100 + L)
    lengths = torch.tensor(lens) if lens is not None else None
    got = fused(lib, q.cuda(), k.cuda(), v.cuda(),
                lengths.cuda() if lengths is not None else None, 1e-6).cpu()
    gate(got, q, k, v, lengths, 1e-6)


def test_strided_views_and_eps(lib):
    """Rows taken out of wider storage (the fused projection layout of an attention layer)
    and a large eps."""
    N, L, H, E, M = 2, 300, 4, 64, 64
    q, k, v = inputs(N, L, H, E, M, seed=7)
    wide = torch.zeros(N, L, H, 3 * 64, device="cuda")
    wide[..., :64], wide[..., 64:128], wide[..., 128:] = q.cuda(), k.cuda(), v.cuda()
    out_wide = torch.full((N, L, H, 2 * M), float("nan"), device="cuda")
    lengths = torch.tensor([300, 123])
    fused(lib, wide[..., :64], wide[..., 64:128], wide[..., 128:], lengths.cuda(), 0.25,
          out=out_wide[..., M:])
    assert torch.isnan(out_wide[..., :M]).all()
    gate(out_wide[..., M:].cpu(), q, k, v, lengths, 0.25)


def test_constant_values_come_back_and_masked_keys_do_not_matter(lib):
    N, L, H, E, M = 2, 5000, 4, 64, 64
    q, k, _ = inputs(N, L, H, E, M, seed=8)
    v = torch.full((N, L, H, M), -3.25)
    lengths = torch.tensor([5000, 1234]).cuda()
    got = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths, 0.0)
    assert (got + 3.25).abs().max().item() < 1e-4
    # keys and values beyond the length are never seen
    k2, v2 = k.clone(), torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(9))
    v3 = v2.clone()
    k2[1, 1234:] = 50.0
    v3[1, 1234:] = 1e6
    a = fused(lib, q.cuda(), k.cuda(), v2.cuda(), lengths, 1e-6)
    b = fused(lib, q.cuda(), k2.cuda(), v3.cuda(), lengths, 1e-6)
    assert torch.equal(a, b)


def test_prefix_property_at_full_size(lib):
    """Config 4's operator shape: the first rows of a long call equal a short call's rows to
    rounding (the segmentation differs), and a repeated call is bit-identical."""
    N, L, H, E, M = 10, 4096, 8, 64, 64
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, M, seed=4))
    whole = fused(lib, q, k, v, None, 1e-6)
    again = fused(lib, q, k, v, None, 1e-6)
    assert torch.equal(whole, again)
    short = fused(lib, q[:, :1500].contiguous(), k[:, :1500].contiguous(),
                  v[:, :1500].contiguous(), None, 1e-6)
    assert scale_error(whole[:, :1500].permute(0, 2, 1, 3), short.permute(0, 2, 1, 3)) <= 2e-6
    # a bounded sample against the CPU restatement
    got = whole[:2].cpu()
    gate(got, q[:2].cpu(), k[:2].cpu(), v[:2].cpu(), None, 1e-6)


def test_sizes_without_a_fused_kernel_are_refused(lib):
    from fast_transformers_amd import _native
    assert lib.ftc_causal_linear_attention_workspace_bytes(1, 1, 64, 48, 64, _native.FTC_F32) == -2
    assert lib.ftc_causal_linear_attention_workspace_bytes(1, 1, 64, 64, 64, _native.FTC_BF16) == -2
    q = torch.zeros(1, 64, 1, 48, device="cuda")
    v = torch.zeros(1, 64, 1, 64, device="cuda")
    d = [_native.describe(t.permute(0, 2, 1, 3)) for t in (q, q, v, v.clone())]
    rc = lib.ftc_causal_linear_attention(ctypes.byref(d[0]), ctypes.byref(d[1]), ctypes.byref(d[2]),
                                         None, ctypes.c_float(1e-6), ctypes.byref(d[3]), None, 0,
                                         None)
    assert rc == -2 and "fused" in _native.last_error()


@pytest.fixture(params=["planned", "workgroup"])
def form(request, monkeypatch):
    """Which kernel takes the launch: as planned, or the workgroup form at any size."""
    from fast_transformers_amd import causal_product as cp
    if request.param == "workgroup":
        monkeypatch.setenv("FTC_WG", "1")
        cp.reload_tuning()
    yield request.param
    if request.param == "workgroup":
        monkeypatch.delenv("FTC_WG")
        cp.reload_tuning()


def taken_by(form, L):
    """Of these tests' shapes, the chain-parallel kernel has those of short chains."""
    return b"scan_tp_kernel<NORM>" if form == "planned" and L <= 320 else b"scan_wg_kernel<NORM>"


CHAIN_PARALLEL_SHAPES = [
    # N, L, H, E, M, key lengths: whole chains, cut chains, an exchange of segment sums (one and two
    # levels), ragged ends, keys that end before, inside and on a chunk, segments without any key;
    # one and two groups of 32 feature columns, half of the consumers without value columns
    (3, 97, 8, 64, 64, [97, 64, 1]), (5, 300, 8, 64, 64, [300, 0, 299, 33, 160]),
    (2, 1000, 16, 64, 64, [1000, 417]), (3, 520, 8, 64, 32, [520, 100, 40]),
    (3, 520, 8, 32, 64, [520, 100, 40]), (2, 2500, 8, 64, 64, [2500, 700]),
    (1, 9000, 16, 64, 64, [4000]),
]


@pytest.mark.parametrize("shape", CHAIN_PARALLEL_SHAPES, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_chain_parallel_form(lib, shape, form):
    """Chain counts, lengths and key lengths of every kind, against the CPU restatement in float64."""
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=70 + L)
    lengths = torch.tensor(lens)
    out = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
    assert lib.ftc_last_kernel() == taken_by(form, L)
    gate(out.cpu(), q, k, v, lengths, 1e-6)


# whole, cut and exchanged chains (the exchange's first pass walks the segments in which the keys end)
MASKED_SHAPES = [(3, 97, 8, 64, 64, [97, 64, 1]), (2, 1000, 16, 64, 64, [1000, 417]), (3, 520, 8, 32, 64, [520, 100, 40]),
                 (1, 9000, 16, 64, 64, [4010])]


@pytest.mark.parametrize("padding", [1e8, 1e30])
@pytest.mark.parametrize("shape", MASKED_SHAPES, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_masked_rows_do_not_set_a_scale(lib, shape, padding, form):
    """Keys and values at or beyond the length leave every row as it is, bit for bit."""
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=170 + L)
    lengths = torch.tensor(lens)
    want = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
    assert lib.ftc_last_kernel() == taken_by(form, L)
    for n, length in enumerate(lens):
        k[n, length:], v[n, length:] = 60.0, padding
    got = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
    assert torch.equal(got, want)
    gate(got.cpu(), q, k, v, lengths, 1e-6)


@pytest.mark.parametrize("small", ["q_rows", "k_early_rows", "v_columns", "v_early_rows"])
@pytest.mark.parametrize("shape", [(3, 300, 8, 64, 64), (2, 1000, 16, 64, 64), (3, 520, 8, 32, 64)],
                         ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s)
def test_small_rows_and_columns_beside_large_ones(lib, shape, small, form):
    """Every row and column of the result is within 2e-6 of float64 on its own scale (a few fp32
    roundings; the float32 restatement is not, where it adds 1 to an expm1 near -1): a row's weights are
    normalised, so rows of small phi(q) or phi(k) beside large ones are still of order one, and columns
    and earlier rows of small values keep their bits beside large ones."""
    N, L, H, E, M = shape
    q, k, v = inputs(N, L, H, E, M, seed=90 + L, scale=1.0)
    if small == "q_rows":
        q[:, 5::32] -= 14
    elif small == "k_early_rows":
        k[:, :16] -= 14
    elif small == "v_columns":
        v[..., ::2] *= 2.0 ** -20
    else:
        v[:, 48:] *= 2.0 ** 20
    got = fused(lib, q.cuda(), k.cuda(), v.cuda(), None, 1e-6).cpu().double()
    want = oracle.causal_linear_attention(q.double(), k.double(), v.double(), None, 1e-6)
    for dim in (1, 3):
        assert ((got - want).norm(dim=dim) / want.norm(dim=dim)).max().item() <= 2e-6


MANY_CHAINS = [
    # N, L, H, E, M, key lengths: chains walked whole, cut in two to five, and with an exchange of segment
    # sums (one and two levels); single positions, ragged ends, keys that end before, inside and on a
    # chunk, segments without any key; one and two groups of 32 feature columns
    (41, 1, 1, 64, 64, [1, 0] * 20 + [5]), (41, 33, 1, 64, 64, [33, 32, 1] * 13 + [0, 7]),
    (6, 97, 8, 64, 64, [97, 64, 1, 0, 33, 96]), (300, 40, 1, 64, 64, list(range(300))),
    (6, 1000, 8, 64, 64, [1000, 417, 0, 999, 512, 31]), (3, 2100, 8, 64, 64, [2100, 2049, 500]),
    (2, 8192, 12, 64, 64, [8192, 3001]), (6, 520, 8, 64, 32, [520, 100, 40, 0, 511, 256]),
    (6, 520, 8, 32, 64, [520, 100, 40, 0, 511, 256]),
]


@pytest.mark.parametrize("shape", MANY_CHAINS, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_many_chains(lib, shape):
    """The chain-parallel form on three bf16 pieces, against the CPU restatement in float64; keys and
    values at or beyond the length leave every row as it is, bit for bit."""
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=270 + L)
    lengths = torch.tensor(lens)
    out = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
    assert lib.ftc_last_kernel().startswith(b"scan_tp_kernel<NORM>")
    gate(out.cpu(), q, k, v, lengths, 1e-6)
    for n, length in enumerate(lens):
        k[n, length:], v[n, length:] = 60.0, 1e30
    assert torch.equal(fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6), out)


@pytest.mark.parametrize("shape", [(1, 512, 4, 64, 64), (5, 640, 4, 64, 64), (9, 900, 4, 64, 64), (10, 1300, 4, 64, 64),
                                   (9, 1600, 4, 64, 64), (2, 500, 4, 64, 32), (10, 1000, 4, 64, 32), (14, 1280, 4, 64, 32),
                                   (20, 1900, 4, 64, 32), (4, 300, 4, 32, 64), (6, 500, 4, 32, 64), (12, 890, 4, 32, 64),
                                   (16, 1400, 4, 32, 64)], ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s)
def test_fewest_chains_of_the_chain_parallel_form(lib, shape):
    """The shapes at the lines between the two forms, on this side of them."""
    N, L, H, E, M = shape
    q, k, v = inputs(N, L, H, E, M, seed=310 + L)
    out = fused(lib, q.cuda(), k.cuda(), v.cuda(), None, 1e-6)
    assert lib.ftc_last_kernel().startswith(b"scan_tp_kernel<NORM>")
    gate(out.cpu(), q, k, v, None, 1e-6)


@pytest.mark.parametrize("shape", [(20, 300, 3, 64, 64), (10, 1000, 6, 64, 64), (64, 900, 2, 64, 32), (25, 129, 2, 32, 64)],
                         ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s)
def test_segments_that_start_at_half_a_trip(lib, shape):
    """Cuts at 2 modulo 4 chunks: the first walk begins with half a trip through its register sets."""
    N, L, H, E, M = shape
    q, k, v = inputs(N, L, H, E, M, seed=290 + L)
    lengths = torch.arange(N) * L // N + 1
    out = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
    assert lib.ftc_last_kernel() == b"scan_tp_kernel<NORM>"
    gate(out.cpu(), q, k, v, lengths, 1e-6)


@pytest.mark.parametrize("small", ["q_rows", "k_early_rows", "v_columns", "v_early_rows"])
@pytest.mark.parametrize("shape", [(6, 300, 8, 64, 64), (3, 2100, 8, 64, 64), (6, 520, 8, 64, 32)],
                         ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s)
def test_many_chains_small_rows_and_columns_beside_large_ones(lib, shape, small):
    test_small_rows_and_columns_beside_large_ones(lib, shape, small, "planned")
    assert lib.ftc_last_kernel().startswith(b"scan_tp_kernel<NORM>")


def test_many_chains_in_the_workgroup_forms_workspace(lib):
    """A workspace that the exchange of the chain-parallel form does not fit in gets the workgroup form."""
    from fast_transformers_amd import _native
    N, L, H, E, M = 3, 2100, 8, 64, 64
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, M, seed=5))
    want = fused(lib, q, k, v, None, 1e-6)
    assert lib.ftc_last_kernel() == b"scan_tp_kernel<NORM> (exchange)"
    full = lib.ftc_causal_linear_attention_workspace_bytes(N, H, L, E, M, _native.FTC_F32)
    ws, out = torch.zeros(full, dtype=torch.uint8, device="cuda"), torch.empty_like(want)
    d = [_native.describe(t.permute(0, 2, 1, 3)) for t in (q, k, v, out)]

    def call(nbytes):
        return lib.ftc_causal_linear_attention(
            *(ctypes.byref(x) for x in d[:3]), None, ctypes.c_float(1e-6), ctypes.byref(d[3]),
            ctypes.c_void_p(ws.data_ptr()), nbytes, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    least = next(b for b in range(1 << 16, full, 1 << 12) if call(b) == 0)
    torch.cuda.synchronize()
    assert least < full and lib.ftc_last_kernel() == b"scan_wg_kernel<NORM>"
    assert ((out - want).norm() / want.norm()).item() <= 2e-6


def _count_backward_calls():
    """Context that counts the calls of the fused backward (autograd runs it on a thread of its
    own, where ftc_last_kernel() of this thread does not see it)."""
    import contextlib
    from fast_transformers_amd import causal_product as cpm

    @contextlib.contextmanager
    def counting():
        calls = []
        native = cpm.causal_linear_attention_backward_hip
        cpm.causal_linear_attention_backward_hip = lambda *a: (calls.append(1), native(*a))[1]
        try:
            yield calls
        finally:
            cpm.causal_linear_attention_backward_hip = native
    return counting()


def _composition(cla):
    """Context that makes the module compose its result from operator calls (what sizes and
    feature maps without a fused kernel get)."""
    import contextlib

    @contextlib.contextmanager
    def off():
        covers = cla.fused_attention_covers
        cla.fused_attention_covers = lambda *a: False
        try:
            yield
        finally:
            cla.fused_attention_covers = covers
    return off()


def test_module_takes_the_fused_path_and_agrees_with_the_composition(lib):
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import causal_linear_attention as cla
    N, L, H, E, M = 2, 700, 4, 64, 64
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, M, seed=11))
    lengths = masking.LengthMask(torch.tensor([700, 301]).cuda(), max_len=L)
    full = masking.LengthMask(torch.full((N,), L).cuda(), max_len=L)
    mask = masking.TriangularCausalMask(L, device="cuda")
    module = attention.CausalLinearAttention(E).cuda()
    calls = []
    native = cla.causal_linear_attention_hip
    cla.causal_linear_attention_hip = lambda *a: (calls.append(1), native(*a))[1]
    try:
        with torch.no_grad():
            y_fused = module(q, k, v, mask, full, lengths)
        assert calls == [1]
        with _composition(cla):
            y_composed = module(q.clone().requires_grad_(True), k, v, mask, full, lengths)
        assert calls == [1] and y_composed.requires_grad
    finally:
        cla.causal_linear_attention_hip = native
    assert scale_error(y_fused.permute(0, 2, 1, 3), y_composed.detach().permute(0, 2, 1, 3)) <= 1e-5
    gate(y_fused.cpu(), q.cpu(), k.cpu(), v.cpu(), torch.tensor([700, 301]), module.eps)


@pytest.mark.parametrize("E", [64, 128])
def test_a_replaced_size_check_composes(lib, E):
    """A module whose ``fused_attention_covers`` has been replaced (how the composition is measured beside
    the fused calls) asks the replacement, in training too."""
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import causal_linear_attention as cla
    N, L, H = 2, 70, 3
    q, k, v = (t.cuda().requires_grad_(True) for t in inputs(N, L, H, E, E, seed=13))
    full, mask = masking.LengthMask(torch.full((N,), L).cuda(), max_len=L), masking.TriangularCausalMask(L, device="cuda")
    module = attention.CausalLinearAttention(E)
    assert "CausalAttention" in module(q, k, v, mask, full, full).grad_fn.name()
    with _composition(cla):
        assert module(q, k, v, mask, full, full).grad_fn.name() == "MulBackward0"


@pytest.mark.parametrize("E", [64, 128])
def test_a_feature_map_with_other_methods_is_not_fused(lib, E):
    """A subclass, a method set on the object or a hook that changes elu(x) + 1: the composition, which
    calls it."""
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import causal_linear_attention as cla
    N, L, H = 2, 70, 3
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, E, seed=12))
    full, mask = masking.LengthMask(torch.full((N,), L).cuda(), max_len=L), masking.TriangularCausalMask(L, device="cuda")

    class Doubled(cla.ActivationFunctionFeatureMap):
        def forward_keys(self, x):
            return self(2 * x)
    subclass = attention.CausalLinearAttention(E, feature_map=Doubled.factory(cla._elu_plus_one))
    method, hook = attention.CausalLinearAttention(E), attention.CausalLinearAttention(E)
    method.feature_map.forward_keys = lambda x: cla._elu_plus_one(2 * x)
    hook.feature_map.register_forward_hook(lambda _, args, y: y + 1)
    plain = attention.CausalLinearAttention(E)
    with torch.no_grad():
        want = plain(q, 2 * k, v, mask, full, full)
        for module in (subclass, method):
            got = module(q, k, v, mask, full, full)
            assert scale_error(got.permute(0, 2, 1, 3), want.permute(0, 2, 1, 3)) <= 1e-5
        unhooked = plain(q, k, v, mask, full, full)
        assert ((hook(q, k, v, mask, full, full) - unhooked).norm() / unhooked.norm()).item() > 1e-2


def _dense_attention(q, k, v, lengths, eps):
    """The closed form of the reference's API test (tests/causal_product/test_causal_product.py:
    34-40) with the feature map and the key-length mask of the module, on (N, L, H, X) tensors
    of any float type: differentiable, so that autograd gives the gradients to compare with."""
    Q = torch.nn.functional.elu(q) + 1
    K = torch.nn.functional.elu(k) + 1
    L = q.shape[1]
    keep = (torch.arange(L, device=q.device)[None, :] < lengths[:, None]).to(q.dtype)
    K = K * keep[:, :, None, None]
    QK = torch.einsum("nlhe,nshe->nhls", Q, K)
    QK = QK * torch.tril(torch.ones(L, L, dtype=q.dtype, device=q.device))
    Z = 1 / (QK.sum(dim=-1) + eps)                       # (N, H, L)
    return torch.einsum("nhls,nshm->nlhm", QK, v) * Z.permute(0, 2, 1)[..., None]


BACKWARD_SHAPES = [
    # N, L, H, E, M, key lengths
    (2, 300, 3, 64, 64, [300, 117]), (1, 1000, 8, 64, 64, [1000]), (3, 257, 2, 32, 32, [257, 40, 200]),
    (2, 513, 2, 64, 32, [513, 400]), (2, 200, 4, 32, 64, [0, 200]), (1, 33, 1, 64, 64, [33]),
]


@pytest.mark.parametrize("shape", BACKWARD_SHAPES, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_backward_against_autograd_in_float64(lib, shape, form):
    """ftc_causal_linear_attention_backward (through the autograd Function the module uses)
    against autograd through the dense closed form in float64; the same closed form in
    float32 shows what that arithmetic alone costs."""
    from fast_transformers_amd.causal_product import CausalLinearAttentionFunction
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=31 + L)
    g = torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(32 + L))
    lengths = torch.tensor(lens)
    eps = 1e-6

    def grads(dtype, device):
        qq, kk, vv = (t.to(device=device, dtype=dtype).requires_grad_(True) for t in (q, k, v))
        out = _dense_attention(qq, kk, vv, lengths.to(device), eps)
        out.backward(g.to(device=device, dtype=dtype))
        return [out.detach().cpu()] + [t.grad.cpu() for t in (qq, kk, vv)]

    exact = grads(torch.float64, "cpu")
    plain = grads(torch.float32, "cuda")
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    nlh = lambda t: t.permute(0, 2, 1, 3)
    out = CausalLinearAttentionFunction.apply(nlh(qd), nlh(kd), nlh(vd), lengths.cuda(), eps)
    short = shape in (BACKWARD_SHAPES[0], BACKWARD_SHAPES[4])   # chains that the planner walks whole or cut
    assert lib.ftc_last_kernel() == taken_by(form, L if short else 1000)
    with _count_backward_calls() as calls:
        nlh(out).backward(g.cuda())
    assert calls == [1]
    torch.cuda.synchronize()
    got = [nlh(out).detach().cpu()] + [t.grad.cpu() for t in (qd, kd, vd)]
    for name, a, b, c in zip(("out", "grad_queries", "grad_keys", "grad_values"), got, plain, exact):
        assert torch.isfinite(a).all(), name
        nlhx = lambda t: t.permute(0, 2, 1, 3).double()
        e_hip, e_plain = scale_error(nlhx(a), nlhx(c)), scale_error(nlhx(b), nlhx(c))
        print("%-13s vs float64: hip %.3e  dense fp32 autograd %.3e" % (name, e_hip, e_plain), flush=True)
        assert e_hip <= max(4 * e_plain, 5e-6), name
    # keys at or beyond the key length have no gradient, as in the reference (their features
    # are multiplied by zero)
    for n_, len_ in enumerate(lens):
        assert (got[2][n_, len_:] == 0).all()


# 64 x 64 rows, whose three scans run straight from the inputs: single positions, one row short of a chunk and
# one past it, keys that end inside and before a chunk; chains walked whole and cut; segment sums exchanged
DIRECT_SHAPES = [
    (2, 1, 3, [1, 0]), (1, 31, 1, [31]), (2, 33, 2, [33, 5]), (3, 129, 8, [129, 0, 64]), (2, 700, 20, [700, 333]),
    (1, 900, 4, [900]), (1, 2500, 2, [2217]), (15, 97, 8, [97, 32, 0, 65, 96] * 3),
]


@pytest.mark.parametrize("small", [None, "v_late_rows", "g_late_rows"])
@pytest.mark.parametrize("shape", DIRECT_SHAPES, ids=lambda s: "n%d_l%d_h%d" % s[:3])
def test_gradients_straight_from_the_inputs(lib, shape, small):
    """Against autograd through the closed form in float64, eps = 1 (no gradient is a difference of nearly equal
    numbers then).  Rows of values or of the gradient that are tiny beside the others' leave the normaliser's
    share of a gradient far beyond the units of the scans' own products."""
    from fast_transformers_amd import causal_product as cp
    N, L, H, lens = shape
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = inputs(N, L, H, 64, 64, seed=81 + L)
    g = torch.randn(N, L, H, 64, generator=torch.Generator().manual_seed(82 + L))
    if small:
        (v if small[0] == "v" else g)[:, (2 * L) // 3:] *= 2.0 ** -40
    lengths = torch.tensor(lens)

    def grads(dtype):
        leaves = [t.to(dtype).requires_grad_(True) for t in (q, k, v)]
        _dense_attention(*leaves, lengths, 1.0).backward(g.to(dtype))
        return [t.grad for t in leaves]
    exact, plain = grads(torch.float64), grads(torch.float32)
    dev = [nlh(t.cuda()) for t in (q, k, v, g)]
    out, den = nlh(torch.empty(N, L, H, 64, device="cuda")), torch.empty(N, H, L, device="cuda")
    cp.causal_linear_attention_hip(*dev[:3], lengths.cuda(), 1.0, out, den)
    got = [nlh(torch.full((N, L, H, 64), float("nan"), device="cuda")) for _ in range(3)]
    cp.causal_linear_attention_backward_hip(*dev[:3], lengths.cuda(), out, den, dev[3], *got)
    assert lib.ftc_last_kernel() == b"attention backward: three scans"
    torch.cuda.synchronize()
    cp.check_workspaces()
    for name, a, b, c in zip("qkv", got, plain, exact):
        a, b, c = a.cpu().double(), nlh(b).double(), nlh(c)
        e_hip, e_plain = scale_error(a, c), scale_error(b, c)
        assert torch.isfinite(a).all() and e_hip <= max(4 * e_plain, 2e-6), (name, e_hip, e_plain)
    # each gradient by itself is the same
    for i in range(3):
        alone = [None] * 3
        alone[i] = torch.empty_like(got[i])
        cp.causal_linear_attention_backward_hip(*dev[:3], lengths.cuda(), out, den, dev[3], *alone)
        assert ((alone[i] - got[i]).norm() <= 2e-6 * got[i].norm()).item()
    # a gradient written over grad_out, which the scans would still read
    over = dev[3].clone(memory_format=torch.preserve_format)
    cp.causal_linear_attention_backward_hip(*dev[:3], lengths.cuda(), out, den, over, None, None, over)
    assert lib.ftc_last_kernel() != b"attention backward: three scans"
    assert ((over - got[2]).norm() <= 2e-6 * got[2].norm()).item()


@pytest.mark.parametrize("shape", [(15, 1000, 4), (1, 2500, 2), (2, 700, 20)], ids=lambda s: "n%d_l%d_h%d" % s)
@pytest.mark.parametrize("over", ["queries", "keys", "inside_a_buffer_of_queries"])
def test_gradient_of_values_written_over_an_input(lib, shape, over):
    """grad_values alone may lie over the queries or the keys: chains that are cut or whose segments exchange sums read
    rows of both in several workgroups, so the scan has to read copies.  Beside them in one buffer is not over them."""
    from fast_transformers_amd import causal_product as cp
    N, L, H = shape
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = (nlh(t.cuda()) for t in inputs(N, L, H, 64, 64, seed=51 + L))
    g = nlh(torch.randn(N, L, H, 64, generator=torch.Generator().manual_seed(52 + L)).cuda())
    out, den = nlh(torch.empty(N, L, H, 64, device="cuda")), torch.empty(N, H, L, device="cuda")
    cp.causal_linear_attention_hip(q, k, v, None, 1e-6, out, den)
    want = torch.empty_like(v)
    cp.causal_linear_attention_backward_hip(q, k, v, None, out, den, g, None, None, want)
    assert lib.ftc_last_kernel() == b"attention backward: three scans"
    if over == "inside_a_buffer_of_queries":
        wide = torch.empty(N, L, H, 128, device="cuda")
        wide[..., :64], q = nlh(q), nlh(wide[..., :64])
        got = nlh(wide[..., 64:])
    else:
        got = (q if over == "queries" else k).clone(memory_format=torch.preserve_format)
        q, k = (got, k) if over == "queries" else (q, got)
    cp.causal_linear_attention_backward_hip(q, k, v, None, out, den, g, None, None, got)
    torch.cuda.synchronize()
    beside = over == "inside_a_buffer_of_queries"
    assert (lib.ftc_last_kernel() == b"attention backward: three scans") == beside
    assert ((got - want).norm() <= 2e-6 * want.norm()).item()


@pytest.mark.parametrize("shape", DIRECT_SHAPES[3:7], ids=lambda s: "n%d_l%d_h%d" % s[:3])
def test_normaliser_sums_of_columns_of_very_different_size(lib, shape):
    """The normaliser's share of a gradient is a sum of fp32 rows: a column of features 2^-14 beside the others, met
    where the values are too small to take part, has the relative error of such a sum (2^-24 a term and 14 ln 2 2^-24
    for the exp2 of each feature, together 1e-6; in two fp16 pieces under the ceiling of all columns 1e-5 to 1e-4)."""
    from fast_transformers_amd import causal_product as cp
    N, L, H, lens = shape
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = inputs(N, L, H, 64, 64, seed=91 + L)
    g = torch.randn(N, L, H, 64, generator=torch.Generator().manual_seed(92 + L))
    late = L // 2
    v[:, late:] *= 2.0 ** -40
    for t, column in ((k, 5), (q, 9)):      # phi: zero before, 2^-14 and its neighbours from there on
        t[:, :late, :, column] = -200.0
        t[:, late:, :, column] = t[:, late:, :, column] / 4 - 9.7
    lengths = torch.full((N,), L)

    leaves = [t.double().requires_grad_(True) for t in (q, k, v)]
    _dense_attention(*leaves, lengths, 1.0).backward(g.double())
    exact = [t.grad for t in leaves]
    dev = [nlh(t.cuda()) for t in (q, k, v, g)]
    out, den = nlh(torch.empty(N, L, H, 64, device="cuda")), torch.empty(N, H, L, device="cuda")
    cp.causal_linear_attention_hip(*dev[:3], lengths.cuda(), 1.0, out, den)
    got = [nlh(torch.empty(N, L, H, 64, device="cuda")) for _ in range(3)]
    cp.causal_linear_attention_backward_hip(*dev[:3], lengths.cuda(), out, den, dev[3], *got)
    assert lib.ftc_last_kernel() == b"attention backward: three scans"
    for i, column in ((0, 5), (1, 9)):
        a, c = (x[:, late:, :, column].double() for x in (nlh(got[i]).cpu(), exact[i]))
        error = ((a - c).norm() / c.norm()).item()
        print("qk"[i], "column", column, "vs float64: %.3e" % error, flush=True)
        assert error <= 2e-6, (i, error)


@pytest.mark.parametrize("what", ["q_nan", "k_nan", "v_nan", "g_nan", "q_minus_inf", "k_minus_inf", "g_inf", "k_nan_beyond_the_length",
                                  "tiny_denominator"])
@pytest.mark.parametrize("shape", [(2, 300, 4), (1, 2500, 2)], ids=lambda s: "n%d_l%d_h%d" % s)
def test_non_finite_rows_reach_the_same_gradients_on_either_route(lib, shape, what):
    """The direct route and the launches around dense copies (taken where a gradient lies over grad_out): the same
    values are finite, and those agree."""
    from fast_transformers_amd import causal_product as cp
    N, L, H = shape
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = inputs(N, L, H, 64, 64, seed=61 + L)
    g = torch.randn(N, L, H, 64, generator=torch.Generator().manual_seed(62 + L))
    nan, inf = float("nan"), float("inf")
    if what == "q_nan":
        q[0, 40, 0, 3] = nan
    elif what == "k_nan":
        k[0, 200, 1, 5] = nan
    elif what == "v_nan":
        v[0, 150, 1, 7] = nan
    elif what == "g_nan":
        g[0, 77, 0, 9] = nan
    elif what == "q_minus_inf":
        q[0, 40, 0, 3] = -inf
    elif what == "k_minus_inf":
        k[0, 200, 1, 5] = -inf
    elif what == "g_inf":
        g[0, 77, 0, 9] = inf
    elif what == "k_nan_beyond_the_length":
        k[0, 290, 0] = nan
    elif what == "tiny_denominator":   # dd and g / den far beyond those of the other rows
        q[0, 60, 1] = -40.0
    q, k, v, g = (nlh(t.cuda()) for t in (q, k, v, g))
    lengths = torch.full((N,), 280).cuda()
    out, den = nlh(torch.empty(N, L, H, 64, device="cuda")), torch.empty(N, H, L, device="cuda")
    cp.causal_linear_attention_hip(q, k, v, lengths, 0.0, out, den)
    got = [nlh(torch.empty(N, L, H, 64, device="cuda")) for _ in range(3)]
    cp.causal_linear_attention_backward_hip(q, k, v, lengths, out, den, g, *got)
    assert lib.ftc_last_kernel() == b"attention backward: three scans"
    over = g.clone(memory_format=torch.preserve_format)
    want = [torch.empty_like(got[0]), torch.empty_like(got[1]), over]
    cp.causal_linear_attention_backward_hip(q, k, v, lengths, out, den, over, *want)
    assert lib.ftc_last_kernel() != b"attention backward: three scans"
    torch.cuda.synchronize()
    cp.check_workspaces()
    for name, a, b in zip("qkv", got, want):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), name
        a, b = (torch.where(torch.isfinite(b), x, torch.zeros_like(x)) for x in (a, b))
        for c in range(N * H):          # (each chain at its own scale)
            x, y = a[c // H, c % H], b[c // H, c % H]
            assert ((x - y).norm() <= 1e-5 * y.norm()).item(), (name, c)


@pytest.mark.parametrize("shape", [(2, 300, 4), (1, 2500, 2)], ids=lambda s: "n%d_l%d_h%d" % s)
def test_gradients_of_parts_of_one_buffer(lib, shape):
    """q, k and v as parts of one projection's rows, their gradients as parts of another's."""
    from fast_transformers_amd import causal_product as cp
    N, L, H = shape
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = (t.cuda() for t in inputs(N, L, H, 64, 64, seed=66 + L))
    g = nlh(torch.randn(N, L, H, 64, generator=torch.Generator().manual_seed(67 + L)).cuda())
    packed, grads = torch.stack([q, k, v], 2), torch.full((N, L, 3, H, 64), float("nan"), device="cuda")
    out, den = nlh(torch.empty(N, L, H, 64, device="cuda")), torch.empty(N, H, L, device="cuda")
    cp.causal_linear_attention_hip(nlh(q), nlh(k), nlh(v), None, 1e-6, out, den)
    want = [nlh(torch.empty_like(q)) for _ in range(3)]
    cp.causal_linear_attention_backward_hip(nlh(q), nlh(k), nlh(v), None, out, den, g, *want)
    got = [nlh(grads[:, :, i]) for i in range(3)]
    cp.causal_linear_attention_backward_hip(*(nlh(packed[:, :, i]) for i in range(3)), None, out, den, g, *got)
    assert lib.ftc_last_kernel() == b"attention backward: three scans"
    for a, b in zip(got, want):
        assert torch.equal(a, b)


WIDE_SHAPES = [
    # N, L, H, E, M, key lengths: single positions, ragged ends, keys that end before, inside and on a
    # chunk; cut chains, whole ones of a round and more of workgroups, exchanges of segment sums; one and
    # two blocks of state rows and of value columns
    (2, 1, 2, 128, 128, [1, 0]), (2, 33, 3, 128, 128, [33, 7]), (3, 129, 2, 128, 64, [129, 0, 64]),
    (1, 1100, 4, 128, 128, [900]), (70, 97, 2, 128, 128, [97, 32, 0, 65, 96] * 14), (2, 300, 3, 64, 128, [300, 117]),
    (2, 257, 2, 32, 128, [257, 40]), (2, 260, 2, 128, 32, [224, 260]), (1, 2500, 1, 128, 128, [2500]),
]


@pytest.mark.parametrize("shape", WIDE_SHAPES, ids=lambda s: "n%d_l%d_h%d_e%d_m%d" % s[:5])
def test_module_at_rows_of_128(lib, shape):
    """The module's fused calls at widths of 128, forward and backward, against the dense closed form in
    float64, with the bounds of the narrower widths (above); masked keys and values do not matter; a
    gradient that 16-byte loads do not reach is copied; rows that they do not reach are composed."""
    from fast_transformers_amd import attention, causal_product as cp
    from fast_transformers_amd.masking import LengthMask, TriangularCausalMask
    N, L, H, E, M, lens = shape
    assert not cp.fused_attention_covers(torch.empty(1, 1, 1, E, device="cuda"), torch.empty(1, 1, 1, M, device="cuda"))
    q, k, v = inputs(N, L, H, E, M, seed=41 + L)
    g = torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(42 + L))
    lengths, eps = torch.tensor(lens), 1e-6
    module, mask = attention.CausalLinearAttention(E), TriangularCausalMask(L, device="cuda")
    keys = LengthMask(lengths.cuda(), max_len=L)

    def grads(f, dtype, *t):
        t = [x.to(device="cuda", dtype=dtype).requires_grad_(True) for x in t]
        out = f(*t)
        return [out.detach()] + list(torch.autograd.grad(out, t, g.to(device="cuda", dtype=dtype)))
    dense = lambda a, b, c: _dense_attention(a, b, c, lengths.cuda(), eps)
    fused_module = lambda a, b, c: module(a, b, c, mask, keys, keys)
    exact, plain = grads(dense, torch.float64, q, k, v), grads(dense, torch.float32, q, k, v)
    got = grads(fused_module, torch.float32, q, k, v)
    torch.cuda.synchronize()
    for name, a, b, c in zip(("out", "grad_queries", "grad_keys", "grad_values"), got, plain, exact):
        assert torch.isfinite(a).all(), name
        nlhx = lambda t: t.permute(0, 2, 1, 3).double().cpu()
        e_hip, e_plain = scale_error(nlhx(a), nlhx(c)), scale_error(nlhx(b), nlhx(c))
        assert e_hip <= max(4 * e_plain, 5e-6), name
    masked_k, masked_v = k.cuda(), v.cuda()
    for n, length in enumerate(lens):
        assert (got[2][n, length:] == 0).all()
        masked_k[n, length:], masked_v[n, length:] = 60.0, 1e30
    with torch.no_grad():
        again = fused_module(q.cuda(), masked_k, masked_v)
    assert lib.ftc_last_kernel().startswith(b"scan_tp_kernel<NORM>") and torch.equal(again, got[0])
    # the same call with its gradient, and then with its queries, one value off the 16-byte boundary
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    t = [x.cuda().requires_grad_(True) for x in (q, k, v)]
    out = fused_module(*t)
    assert "CppNode" in out.grad_fn.name()
    for a, b in zip(torch.autograd.grad(out, t, off(g.cuda())), got[1:]):
        assert torch.equal(a, b)
    out = fused_module(off(q.cuda()).requires_grad_(True), *t[1:])
    assert "CppNode" not in out.grad_fn.name()
    assert scale_error(out.detach().permute(0, 2, 1, 3).cpu(), got[0].permute(0, 2, 1, 3).cpu()) <= 5e-6


def test_backward_finite_differences(lib):
    """Directional derivatives of sum(out * w) along random directions, by central differences
    of the float64 closed form, against the fused backward's gradients."""
    from fast_transformers_amd.causal_product import CausalLinearAttentionFunction
    N, L, H, E, M = 1, 150, 2, 64, 64
    q, k, v = inputs(N, L, H, E, M, seed=41)
    w = torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(42))
    lengths = torch.tensor([131])
    eps = 1e-6
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    nlh = lambda t: t.permute(0, 2, 1, 3)
    out = CausalLinearAttentionFunction.apply(nlh(qd), nlh(kd), nlh(vd), lengths.cuda(), eps)
    (nlh(out) * w.cuda()).sum().backward()
    f = lambda a, b, c: (_dense_attention(a.double(), b.double(), c.double(), lengths, eps) * w.double()).sum()
    gen = torch.Generator().manual_seed(43)
    for name, base, grad in (("queries", 0, qd.grad), ("keys", 1, kd.grad), ("values", 2, vd.grad)):
        for _ in range(3):
            args = [q, k, v]
            direction = torch.randn(args[base].shape, generator=gen)
            h = 1e-4
            plus, minus = list(args), list(args)
            plus[base] = args[base].double() + h * direction.double()
            minus[base] = args[base].double() - h * direction.double()
            fd = ((f(*plus) - f(*minus)) / (2 * h)).item()
            an = (grad.cpu().double() * direction.double()).sum().item()
            print("d/d%s: finite difference %.6e, backward %.6e" % (name, fd, an), flush=True)
            assert abs(fd - an) <= 1e-4 * max(1.0, abs(fd))


def test_module_trains_through_the_fused_backward(lib):
    """Under grad the module runs the fused forward and its backward, and the parameters'
    gradients agree with those of the composition of operator calls."""
    from fast_transformers_amd import attention, masking
    from fast_transformers_amd.attention import causal_linear_attention as cla
    N, L, H, E, M = 2, 400, 4, 64, 64
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, M, seed=51))
    lengths = masking.LengthMask(torch.tensor([400, 255]).cuda(), max_len=L)
    full = masking.LengthMask(torch.full((N,), L).cuda(), max_len=L)
    mask = masking.TriangularCausalMask(L, device="cuda")
    module = attention.CausalLinearAttention(E).cuda()
    w = torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(52)).cuda()

    def run():
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        y = module(*leaves, mask, full, lengths)
        (y * w).sum().backward()
        return y.detach(), [t.grad for t in leaves]

    with _count_backward_calls() as calls:
        y_fused, g_fused = run()
        assert calls == [1]
        with _composition(cla):
            y_comp, g_comp = run()
        assert calls == [1]
    nlh = lambda t: t.permute(0, 2, 1, 3)
    assert scale_error(nlh(y_fused), nlh(y_comp)) <= 1e-5
    for name, a, b in zip(("queries", "keys", "values"), g_fused, g_comp):
        err = scale_error(nlh(a), nlh(b))
        print("grad %s: fused against composition %.3e" % (name, err), flush=True)
        assert err <= 2e-5, name


def test_non_finite_inputs_propagate_as_in_the_composition(lib):
    """The feature map elu(x) + 1 keeps NaN (and maps -inf to 0, +inf to +inf), in the fused
    launch as in the composition of operator calls that training uses: the same rows come out
    non-finite either way."""
    from fast_transformers_amd import attention, masking
    N, L, H, E, M = 1, 300, 2, 64, 64
    q, k, v = (t.cuda() for t in inputs(N, L, H, E, M, seed=12))
    q[0, 40, 0, 3] = float("nan")     # one query row of head 0
    k[0, 200, 1, 5] = float("nan")    # a key of head 1: every row from 200 on
    q[0, 10, 1, 7] = float("-inf")    # phi(-inf) = 0: harmless
    full = masking.LengthMask(torch.full((N,), L).cuda(), max_len=L)
    mask = masking.TriangularCausalMask(L, device="cuda")
    module = attention.CausalLinearAttention(E).cuda()
    with torch.no_grad():
        y_fused = module(q, k, v, mask, full, full)
    y_composed = module(q.clone().requires_grad_(True), k, v, mask, full, full).detach()
    bad_fused, bad_composed = ~torch.isfinite(y_fused), ~torch.isfinite(y_composed)
    assert torch.equal(bad_fused.any(dim=-1), bad_composed.any(dim=-1))
    assert bad_fused[0, 40, 0].all() and bad_fused[0, 200:, 1].all()
    assert not bad_fused[0, :40, 0].any() and not bad_fused[0, :200, 1].any()
    ok = ~bad_fused
    assert (y_fused[ok] - y_composed[ok]).abs().max() <= 1e-4 * y_composed[ok].abs().max()


@pytest.mark.parametrize("E,M", [(64, 64), (64, 32), (32, 64), (128, 128)])
@pytest.mark.parametrize("what", ["large", "small"])
def test_denominators_at_the_ends_of_the_range(lib, E, M, what):
    """Denominators of 3 x 2^126, whose reciprocal is below 2^-126, and of 2^-127 (3 x 2^-122 beside an eps that
    leaves that much of it): rows are quotients all the same.  One feature counts, of three keys."""
    from fast_transformers_amd import _native
    N, L, H = 8, 500, 4
    v = torch.rand(N, L, H, M, generator=torch.Generator().manual_seed(41))    # (three of them stay below 4)
    q, k = torch.full((N, L, H, E), -200.0), torch.full((N, L, H, E), -200.0)   # phi is zero
    k[:, :3, :, 5] = q[..., 5] = 2.0 ** 63 if what == "large" else -61 * math.log(2.0)
    eps = 0.0 if what == "large" else -(3 * 2.0 ** -122 - 2.0 ** -127)
    q, k, v, lengths = q.cuda(), k.cuda(), v.cuda(), torch.full((N,), 3).cuda()
    out, den = torch.empty(N, L, H, M, device="cuda"), torch.empty(N, H, L, 1, device="cuda")
    nbytes = lib.ftc_causal_linear_attention_wide_workspace_bytes(N, H, L, E, M, _native.FTC_F32)
    assert nbytes >= 0, _native.last_error()
    ws = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    d = [_native.describe(t.permute(0, 2, 1, 3)) for t in (q, k, v, out)] + [_native.describe(den)]
    rc = lib.ftc_causal_linear_attention_wide_forward(
        *(ctypes.byref(x) for x in d[:3]), ctypes.c_void_p(lengths.data_ptr()), ctypes.c_float(eps), ctypes.byref(d[3]),
        ctypes.byref(d[4]), ctypes.c_void_p(ws.data_ptr()), nbytes, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.last_error()
    torch.cuda.synchronize()
    assert lib.ftc_last_kernel().startswith(b"scan_tp_kernel<NORM>")
    got, d = out.cpu()[:, 2:].double(), den.cpu().permute(0, 2, 1, 3)[:, 2:].double()
    products = 2.0 ** 126 if what == "large" else 2.0 ** -122
    assert bool(((d == 3 * products) if what == "large" else (d - 2.0 ** -127).abs() < 2.0 ** -129).all()), d.max().item()
    want = v.cpu()[:, :3].double().sum(1, keepdim=True) * products / d
    # (a reciprocal below 2^-126 is rounded to 2^-149, 2^-22 of it; an exponent of 61 ln 2 is rounded twice on its way
    # into an exp2, which has 2 x 61 ln 2 2^-24 of it for each of two features)
    error = ((got - want).abs() / want).max().item()
    assert error <= (2.0 ** -20 if what == "large" else 2e-5), error


def test_forward_and_backward_replay_in_a_graph(lib):
    """Both entry points only enqueue kernels (fill kernels instead of memsets, nothing
    allocated), so a forward + backward pair can be captured in a HIP graph.  Every replay,
    with direct launches on other data in between, reproduces the direct results bit for bit."""
    from fast_transformers_amd import causal_product as cp
    N, L, H, E, M = 2, 600, 4, 64, 64
    nlh = lambda t: t.permute(0, 2, 1, 3)
    q, k, v = (nlh(t.cuda()) for t in inputs(N, L, H, E, M, seed=71))
    q2, k2, v2 = (nlh(t.cuda()) for t in inputs(N, L, H, E, M, seed=72))
    g = nlh(torch.randn(N, L, H, M, generator=torch.Generator().manual_seed(73)).cuda())
    lengths = torch.tensor([600, 431]).cuda()
    out = nlh(torch.empty(N, L, H, M, device="cuda"))
    den = torch.empty(N, H, L, device="cuda")
    grads = [nlh(torch.empty(N, L, H, X, device="cuda")) for X in (E, E, M)]

    def pair():
        cp.causal_linear_attention_hip(q, k, v, lengths, 1e-6, out, den)
        cp.causal_linear_attention_backward_hip(q, k, v, lengths, out, den, g, *grads)

    pair()
    torch.cuda.synchronize()
    want = [t.clone() for t in [out] + grads]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the wrapper's workspace for this stream exists before capture
        pair()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        pair()
    other = nlh(torch.empty(N, L, H, M, device="cuda"))
    for replay in range(4):
        for t in [out, den] + grads:
            t.fill_(float("nan"))
        cp.causal_linear_attention_hip(q2, k2, v2, None, 1e-6, other)   # the program's own work
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, got, ref in zip(("out", "dq", "dk", "dv"), [out] + grads, want):
            assert torch.equal(got, ref), (replay, name)
    assert torch.isfinite(other).all()


# few chains in an exchange: the shortest and the first longer ones on either side of its lines, a last segment of one
# position, segments in which the keys end or that have none
FEW_CHAINS = [((1, 865, 3, 64, 64, [865]), True), ((2, 1024, 3, 64, 64, [1024, 1]), True), ((1, 1185, 8, 64, 64, [700]), True),
              ((1, 1000, 7, 64, 64, [1000]), False), ((3, 1590, 4, 64, 64, [1590, 33, 128]), True),
              ((1, 2049, 1, 64, 64, [2048]), True), ((1, 1590, 13, 64, 64, [1590]), False)]


@pytest.mark.parametrize("shape,exchanges", FEW_CHAINS, ids=lambda s: "n%d_l%d_h%d" % s[:3] if isinstance(s, tuple) else "")
def test_few_chains_exchange_their_segment_sums(lib, shape, exchanges):
    N, L, H, E, M, lens = shape
    q, k, v = inputs(N, L, H, E, M, seed=270 + L)
    lengths = torch.tensor(lens)
    for _ in range(2):   # (the control block is left as it was found)
        out = fused(lib, q.cuda(), k.cuda(), v.cuda(), lengths.cuda(), 1e-6)
        assert lib.ftc_last_kernel() == (b"scan_tp_kernel<NORM> (exchange)" if exchanges else b"scan_wg_kernel<NORM>")
        gate(out.cpu(), q, k, v, lengths, 1e-6)
