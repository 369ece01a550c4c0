"""The scales of the chain-parallel kernel's fp16 path (states of up to 64 rows): every fp32
value is scaled by a power of two that follows the largest magnitude met so far in the walk
and is cut into two fp16 pieces; the state has a scale of its own.  These cases drive what the
seeded N(0,1) / elu+1 inputs of the other tests never reach: operands many orders of magnitude
away from one, ceilings that rise all along a chain, states beyond 2^14 scaled units, all-zero
chunks, and states handed in that dwarf (or are dwarfed by) the rows.

Everything is compared with the CPU oracle (the reference's own fp32 order) and anchored on
float64: per chain, or per row where rows differ in scale, the HIP result may be at most four
times as far from float64 as the checker is (or 2e-6 of the scale)."""
import pytest
import torch

import oracle
from parity import scale_error

pytestmark = pytest.mark.gpu

KERNELS = (b"scan_tph_kernel", b"scan_tph_kernel (exchange)")


@pytest.fixture(scope="module")
def cp():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU (torch.cuda.is_available() is False)")
    from fast_transformers_amd import causal_product
    from fast_transformers_amd import _native
    _native.load()
    return causal_product


def _last_kernel():
    from fast_transformers_amd import _native
    return _native.load().ftc_last_kernel()


def _run(cp, Q, K, V, G):
    N, H, L, E = Q.shape
    M = V.shape[3]
    q, k, v, g = (t.cuda() for t in (Q, K, V, G))
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(q, k, v, out)
    assert _last_kernel() in KERNELS, _last_kernel()
    grads = [torch.full((N, H, L, X), float("nan"), device="cuda") for X in (E, E, M)]
    cp.causal_dot_backward_hip(q, k, v, g, *grads)
    assert _last_kernel() in KERNELS, _last_kernel()
    torch.cuda.synchronize()
    return [out.cpu()] + [t.cpu() for t in grads]


def _references(Q, K, V, G):
    refs = [oracle.forward(Q, K, V)] + list(oracle.backward(Q, K, V, G))
    Qd, Kd, Vd, Gd = (t.double() for t in (Q, K, V, G))
    exact = [oracle.forward(Qd, Kd, Vd)] + list(oracle.backward(Qd, Kd, Vd, Gd))
    return refs, exact


def _row_error(got, want):
    """max over rows of max|got - want| / max|want| of that row (rows of all-zero want: the
    absolute error must be zero too)."""
    got, want = got.double(), want.double()
    num = (got - want).abs().amax(dim=-1)
    den = want.abs().amax(dim=-1)
    err = torch.where(den > 0, num / den.clamp_min(1e-300), num)
    return err.max().item()


def _gate(tag, got, ref, exact, metric=scale_error, floor=2e-6):
    assert torch.isfinite(got).all(), tag
    e_hip, e_cpu, e_both = metric(got, exact), metric(ref, exact), metric(got, ref)
    print("%-34s vs float64: hip %.3e cpu %.3e; hip vs cpu %.3e" % (tag, e_hip, e_cpu, e_both),
          flush=True)
    assert e_hip <= max(4 * e_cpu, floor), tag
    assert e_both <= 1e-4, tag


NAMES = ("product", "dQ", "dK", "dV")


@pytest.mark.parametrize("scales", [(1e-3, 1e-4, 1e-5, 1e-6), (3e4, 1e-7, 1e3, 1e-9),
                                    (1e-12, 1e-12, 1e10, 1e5), (1.0, 1.0, 1.0, 2.0 ** -60)],
                         ids=["small", "mixed", "tiny_qk", "tiny_grad"])
def test_operands_far_from_one(cp, scales):
    """Operands scaled by arbitrary factors: the scales of the pieces follow them, so the
    results are as accurate as for operands near one (fp16's range is never met)."""
    N, H, L, E, M = 6, 8, 700, 64, 64
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=71)
    Q, K, V, G = (t * s for t, s in zip((Q, K, V, G), scales))
    refs, exact = _references(Q, K, V, G)
    for name, got, ref, ex in zip(NAMES, _run(cp, Q, K, V, G), refs, exact):
        _gate("%s x%s" % (name, scales), got, ref, ex)


@pytest.mark.parametrize("reverse", [False, True], ids=["rising", "falling_rows_of_the_reverse_scans"])
def test_ceilings_that_rise_along_the_chain(cp, reverse):
    """Rows whose magnitude grows by 2^24 along the walk: every few chunks a ceiling rises, the
    state is rescaled, and early rows keep the accuracy of their own scale (error per row).
    Run forwards for the scans that walk up, flipped for those that walk down."""
    N, H, L, E, M = 6, 8, 1200, 64, 64
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=72)
    ramp = torch.exp2(torch.arange(L, dtype=torch.float32) / 50.0)[None, None, :, None]
    if reverse:
        ramp = torch.flip(ramp, dims=[2])
    Q, K, V, G = Q * ramp, K * ramp, V * ramp, G * ramp
    refs, exact = _references(Q, K, V, G)
    outs = _run(cp, Q, K, V, G)
    # the scans that walk in the direction of growth: product and dQ forwards, dK and dV flipped
    for name, got, ref, ex in zip(NAMES, outs, refs, exact):
        if (name in ("product", "dQ")) != reverse:
            _gate("%s rows" % name, got, ref, ex, metric=_row_error, floor=4e-6)
        else:
            _gate("%s chains" % name, got, ref, ex)


def test_rows_smaller_than_those_before_them(cp):
    """The rows of `a` are scaled by the ceiling of their own chunk, not of the walk so far:
    rows that fall by 2^-20 along the chain keep the accuracy of their own scale (error per
    row), as in the reference."""
    N, H, L, E, M = 6, 8, 800, 64, 64
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=73)
    ramp = torch.exp2(-20.0 * torch.arange(L, dtype=torch.float32) / L)[None, None, :, None]
    Q, G = Q * ramp, G * ramp
    refs, exact = _references(Q, K, V, G)
    outs = _run(cp, Q, K, V, G)
    for name, got, ref, ex in zip(NAMES, outs, refs, exact):
        if name in ("product", "dQ"):
            _gate("%s rows" % name, got, ref, ex, metric=_row_error, floor=4e-6)
        else:
            _gate("%s chains" % name, got, ref, ex)


@pytest.mark.parametrize("shape", [(8, 16, 8192, 64, 64), (1, 4, 40000, 64, 64), (2, 64, 4096, 32, 64)],
                         ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_states_beyond_the_range_of_a_piece(cp, shape):
    """All-positive U[0,1) operands on long chains: the state grows like the position, far
    beyond 2^14 scaled units, so its pieces need the extra scale 2^-s (whole chains and
    segments that exchange their sums)."""
    N, H, L, E, M = shape
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=74, positive_uniform=True)
    h = min(H, 3)   # (the CPU oracle takes a second per long chain)
    Qs, Ks, Vs, Gs = (t[:1, :h].contiguous() for t in (Q, K, V, G))
    refs, exact = _references(Qs, Ks, Vs, Gs)
    outs = _run(cp, Q, K, V, G)
    for name, got, ref, ex in zip(NAMES, outs, refs, exact):
        _gate("%s %s" % (name, shape), got[:1, :h], ref, ex)


def test_zero_chunks_and_zero_operands(cp):
    N, H, L, E, M = 6, 8, 640, 64, 64
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=75)
    for t in (Q, K, V, G):
        t[:, :, 64:200] = 0        # whole chunks of zeros in every operand
        t[:, :, 300:303] = 0
    K[1] = 0                        # a batch entry whose keys are all zero
    V[0, 3] = 0
    refs, exact = _references(Q, K, V, G)
    for name, got, ref, ex in zip(NAMES, _run(cp, Q, K, V, G), refs, exact):
        assert torch.isfinite(got).all(), name
        assert scale_error(got, ref) <= 1e-4, name
        assert (got[ref == 0] == 0).all(), name    # exact zeros stay exact zeros
    zero = torch.zeros(N, H, L, E)
    outs = _run(cp, zero, zero, zero[..., :M], zero[..., :M])
    assert all((t == 0).all() for t in outs)


@pytest.mark.parametrize("factor", [1e6, 1e-6, 1.0])
def test_state_handed_in_at_another_scale(cp, factor):
    """A caller's state far larger (or smaller) than what the rows add to it."""
    N, H, L, E, M = 8, 8, 500, 64, 64
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=76)
    S0 = torch.randn(N, H, E, M, generator=torch.Generator().manual_seed(77)) * factor
    want, want_state = oracle.forward_with_state(Q, K, V, S0)
    ex, ex_state = oracle.forward_with_state(Q.double(), K.double(), V.double(), S0.double())
    out, state = cp.causal_dot_product_with_state(Q.cuda(), K.cuda(), V.cuda(), S0.cuda())
    assert _last_kernel() in KERNELS
    _gate("product from a state x%g" % factor, out.cpu(), want, ex)
    _gate("final state x%g" % factor, state.cpu(), want_state, ex_state)


@pytest.mark.parametrize("shape", [(1, 16, 16384), (10, 8, 1000), (1, 3, 400)], ids=lambda s: "n%d_h%d_l%d" % s)
@pytest.mark.parametrize("zeros", ["keys_tail", "values_tail", "both_tail", "all_with_state", "then_small"])
def test_stretches_of_zeros_next_to_a_state(shape, zeros):
    """Masked keys or padded values: whole segments of zeros that receive a state from elsewhere
    (the segments before them, the caller), and small values after nothing but zeros.  Against
    float64 sums of the same inputs, at the scale gate of the other tests (2e-6 of the chain's
    largest; four times that for the state's longest sums)."""
    from fast_transformers_amd import causal_product as cp
    N, H, L = shape
    E = M = 64
    gen = torch.Generator().manual_seed(21)
    Q, K, V = (torch.rand(N, H, L, w, generator=gen) for w in (E, E, M))
    S = torch.rand(N, H, E, M, generator=gen) * 100 if zeros in ("all_with_state", "then_small") else None
    if zeros in ("keys_tail", "both_tail"):
        K[:, :, L * 3 // 4:] = 0
    if zeros in ("values_tail", "both_tail"):
        V[:, :, L * 3 // 4:] = 0
    if zeros == "all_with_state":
        K.zero_(), V.zero_()
    if zeros == "then_small":
        K[:, :, :L // 2] = 0
        K[:, :, L // 2:] *= 2.0 ** -70
    got, state = cp.causal_dot_product_with_state(Q.cuda(), K.cuda(), V.cuda(),
                                                  S.cuda() if S is not None else None)
    cp.check_workspaces()
    want, want_state = oracle.forward_with_state(Q.double(), K.double(), V.double(),
                                                 S.double() if S is not None else None)
    assert scale_error(got.cpu(), want) <= 8e-6
    assert scale_error(state.cpu(), want_state) <= 8e-6
