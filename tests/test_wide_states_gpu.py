"""States of 65 to 128 rows: chains of 32 chunks or more, walked whole, cut, or with an exchange;
widths that do not fill either block; rows whose scale changes along the chain; a state handed in and
out.  Gate: no further from float64 than four times the fp32 oracle, or 2e-6 of the chain's largest
(the gate of the narrower states) -- and, where rows or columns of very different size stand side by
side, the same for every row and every column on its own."""
import pytest
import torch

import oracle
from parity import scale_error

pytestmark = pytest.mark.gpu

#        N  H  L     E    M
SHAPES = [(1, 2, 1000, 68, 16),    # one quad in the second block, three consumers without columns
          (2, 3, 1024, 96, 64),    # the second block half full; whole chunks
          (1, 3, 1025, 100, 100),  # one row in the last chunk; a second block of columns
          (1, 2, 1061, 128, 128),
          (24, 6, 993, 72, 68),    # more chains than half the workgroups
          (2, 8, 2052, 72, 68)]    # exchange


@pytest.fixture(scope="module")
def cp():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU (torch.cuda.is_available() is False)")
    from fast_transformers_amd import causal_product
    return causal_product


def _gate(got, ref, exact):
    assert torch.isfinite(got).all()
    assert scale_error(got, exact) <= max(4 * scale_error(ref, exact), 2e-6)


def _check(cp, Q, K, V, G):
    q, k, v, g = (t.cuda() for t in (Q, K, V, G))
    outs = [torch.full_like(t, float("nan")) for t in (v, q, k, v)]
    cp.causal_dot_product_hip(q, k, v, outs[0])
    cp.causal_dot_backward_hip(q, k, v, g, *outs[1:])
    cp.check_workspaces()
    wide = [t.double() for t in (Q, K, V, G)]
    refs = [oracle.forward(Q, K, V)] + list(oracle.backward(Q, K, V, G))
    exact = [oracle.forward(*wide[:3])] + list(oracle.backward(*wide))
    for got, ref, ex in zip(outs, refs, exact):
        _gate(got.cpu(), ref, ex)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_wide_states(cp, shape):
    _check(cp, *oracle.make_inputs(*shape, seed=70 + shape[2]))


@pytest.mark.parametrize("how", ["rising", "zeros", "large"])
def test_scales_along_the_chain(cp, how):
    Q, K, V, G = oracle.make_inputs(1, 2, 1050, 128, 72, seed=7)
    if how == "rising":      # both ceilings rise, the second block's rows first
        up = torch.logspace(-6, 4, 1050)[:, None]
        K = K * up
        K[..., 64:] *= 8
        V = V * up.sqrt()
    elif how == "zeros":     # whole chunks of zeros, at the start and in the middle, in one block or both
        K[:, :, :70] = 0
        K[:, :, 300:400, 64:] = 0
        Q[:, :, 500:600, :64] = 0
        V[:, :, 640:705] = 0
    else:                    # a state far beyond 2^14 scaled units
        K = K.abs() + 1
        V = V.abs() + 1
    _check(cp, Q, K, V, G)


@pytest.mark.parametrize("L", [1000, 1056])
def test_state_in_and_out(cp, L):
    N, H, E, M = 2, 3, 104, 84
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=L)
    S = 50 * torch.randn(N, H, E, M, generator=torch.Generator().manual_seed(1))
    out, last = cp.causal_dot_product_with_state(Q.cuda(), K.cuda(), V.cuda(), S.cuda())
    Kd, Vd = K.double(), V.double()
    exact = oracle.forward(Q.double(), Kd, Vd) + Q.double() @ S.double()
    ref = oracle.forward(Q, K, V) + Q @ S
    _gate(out.cpu(), ref, exact)
    _gate(last.cpu(), S + K.transpose(-1, -2) @ V, S.double() + Kd.transpose(-1, -2) @ Vd)


def _each(got, exact, dim):
    """The largest 2-norm error of a row (dim 3) or column (dim 2) over its own 2-norm."""
    got, exact = got.double(), exact.double()
    return ((got - exact).norm(dim=dim) / exact.norm(dim=dim)).max().item()


@pytest.mark.parametrize("shape", [(1, 8, 1061, 128, 128), (4, 32, 1024, 100, 68)], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
@pytest.mark.parametrize("small", ["q_rows", "q_columns", "k_columns", "v_columns", "g_rows", "g_columns", "v_early_rows"])
def test_small_rows_and_columns_beside_large_ones(cp, small, shape):
    """Every row and column of a result is as close to float64, on its own scale, as the fp32
    oracle's: no operand's large values set the precision of its small ones."""
    Q, K, V, G = oracle.make_inputs(*shape, seed=11)
    if small == "v_early_rows":  # rows 48 and on set no scale for the rows before them
        V[:, :, 48:] *= 2.0 ** 20
    else:
        t = dict(q=Q, k=K, v=V, g=G)[small[0]]
        t[..., 5::32, :] *= 2.0 ** -20 if small.endswith("rows") else 1
        t[..., ::2] *= 2.0 ** -20 if small.endswith("columns") else 1
    q, k, v, g = (t.cuda() for t in (Q, K, V, G))
    outs = [torch.full_like(t, float("nan")) for t in (v, q, k, v)]
    cp.causal_dot_product_hip(q, k, v, outs[0])
    cp.causal_dot_backward_hip(q, k, v, g, *outs[1:])
    cp.check_workspaces()
    wide = [t.double() for t in (Q, K, V, G)]
    refs = [oracle.forward(Q, K, V)] + list(oracle.backward(Q, K, V, G))
    exact = [oracle.forward(*wide[:3])] + list(oracle.backward(*wide))
    for got, ref, ex in zip(outs, refs, exact):
        for dim in (2, 3):
            assert _each(got.cpu(), ex, dim) <= max(4 * _each(ref, ex, dim), 2e-6)


@pytest.mark.parametrize("shape", [(1, 1, 289, 128, 128), (1, 4, 416, 128, 128), (2, 4, 385, 128, 64), (2, 5, 705, 96, 96),
                                   (5, 4, 449, 128, 64)], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_short_chains_of_wide_states(shape, dtype):
    """Few short chains walked whole or cut where they were split with an exchange: a last chunk of one row, states
    handed in and out; no further from float64 than the oracle's own order."""
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    gen = torch.Generator().manual_seed(L)
    Q, K = (torch.nn.functional.elu(torch.randn(N, H, L, E, generator=gen)) + 1 for _ in range(2))
    V, S = torch.randn(N, H, L, M, generator=gen), 5 * torch.randn(N, H, E, M, generator=gen)
    q, k, v = (t.cuda().to(dtype) for t in (Q, K, V))
    Q, K, V = (t.float().cpu() for t in (q, k, v))
    out, state = cp.causal_dot_product_with_state(q, k, v, S.cuda())
    exact = oracle.forward(Q.double(), K.double(), V.double()) + Q.double() @ S.double()
    plain = oracle.forward(Q, K, V) + Q @ S
    assert scale_error(out.cpu(), exact) <= max(4 * scale_error(plain, exact), 2e-6)
    final = S.double() + K.double().transpose(2, 3).contiguous() @ V.double()
    assert scale_error(state.cpu(), final) <= 2e-6
    assert torch.equal(out, cp.causal_dot_product_with_state(q, k, v, S.cuda())[0])


@pytest.mark.parametrize("widths", [(128, 128), (128, 64)], ids=lambda s: "e%d_m%d" % s)
@pytest.mark.parametrize("L", [257, 270, 288, 385, 390, 400])
def test_states_of_a_short_bf16_prefill(widths, L):
    """The state that a few chains of 9 or 13 chunks hand out is a sum of sums of four chunks, not one running sum: no
    further from float64 than such sums, rounded after every 16 products as the matrix instructions add them, come out."""
    import fast_transformers_amd.causal_product as cp
    (E, M), C = widths, 6
    gen = torch.Generator().manual_seed(L)
    Q, K = ((torch.nn.functional.elu(torch.randn(1, C, L, E, generator=gen)) + 1).bfloat16() for _ in range(2))
    V = torch.randn(1, C, L, M, generator=gen).bfloat16()
    S = 20 * torch.randn(1, C, E, M, generator=gen)
    out, state = cp.causal_dot_product_with_state(Q.cuda(), K.cuda(), V.cuda(), S.cuda())
    K64, V64 = K.double(), V.double()
    final = S.double() + K64.transpose(2, 3).contiguous() @ V64
    total = S.clone()
    for first in range(0, L, 128):
        part = torch.zeros_like(total)
        for at in range(first, min(first + 128, L), 16):
            k, v = (t[:, :, at:min(at + 16, L)] for t in (K64, V64))
            part = (part.double() + k.transpose(2, 3).contiguous() @ v).float()
        total = total + part
    error = lambda t: ((t.double() - final).norm() / final.norm()).item()
    # (a running sum: 1.07 times; sums of the same products in another order within 1.02)
    assert error(state.cpu()) <= 1.05 * error(total)
    exact = oracle.forward(Q.double(), K64, V64) + Q.double() @ S.double()
    plain = oracle.forward(Q.float(), K.float(), V.float()) + Q.float() @ S
    assert scale_error(out.cpu(), exact) <= max(4 * scale_error(plain, exact), 2e-6)


@pytest.mark.parametrize("shape", [(1, 1, 289, 128, 128), (1, 4, 416, 128, 128), (2, 4, 385, 128, 64), (2, 5, 705, 96, 96),
                                   (5, 4, 449, 128, 64), (2, 5, 736, 128, 128)], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_short_chains_of_wide_states_without_a_state(shape):
    """The same fp32 chains in a plain forward, which walks them whole or cut (those that a state is handed in or out of
    stay with the kernels that split L): rows no further from float64 than the fp32 oracle's."""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=500 + L)
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(Q.cuda(), K.cuda(), V.cuda(), out)
    assert _native.load().ftc_last_kernel() == b"scan_tp_kernel"
    exact, plain = oracle.forward(*(t.double() for t in (Q, K, V))), oracle.forward(Q, K, V)
    norm = lambda t: ((t.double() - exact).norm() / exact.norm()).item()
    assert norm(out.cpu()) <= max(norm(plain), 1.5e-7)
    assert scale_error(out.cpu(), exact) <= max(4 * scale_error(plain, exact), 2e-6)
