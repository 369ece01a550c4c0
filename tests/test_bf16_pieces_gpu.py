"""bf16 rows on the chain-parallel kernel that multiplies them as they are (scan_tp_bf16_kernel):
states of up to 128 rows, few and many chains, whole, cut and with an exchange of segment sums,
against float64 as tests/test_bf16_rows_gpu.py does."""
import ctypes

import pytest
import torch

import oracle
from parity import scale_error
from test_bf16_rows_gpu import _check_gradients, _inputs, _last_kernel

pytestmark = pytest.mark.gpu

OURS = (b"scan_tp_bf16_kernel", b"scan_tp_bf16_kernel (exchange)")


@pytest.fixture(scope="module")
def cp():
    from fast_transformers_amd import causal_product
    return causal_product


# N, H, L, E, M: one and many blocks of state rows and of columns, blocks that are filled to 4, 32 and 64
# rows; one position, the ends of chunks; whole chains, cut ones, one and two levels of exchange.  And the
# launches of the forward, dQ, dK and dV alone and all three (the last one): w: whole or cut chains, x: an
# exchange, s: the kernels that split L
SHAPES = {
    (1, 3, 1, 128, 128): "wwwww", (2, 4, 33, 128, 128): "wwwww", (4, 4, 600, 128, 128): "wwwww",
    (1, 4, 4096, 128, 128): "xxxxx", (1, 2, 9000, 128, 128): "xxxxx", (3, 8, 300, 96, 96): "wwwww",
    (3, 8, 257, 68, 100): "wwwww", (2, 8, 500, 128, 64): "wwwww", (3, 8, 500, 64, 128): "wwwww",
    (6, 8, 257, 36, 124): "wwwww", (2, 8, 97, 64, 64): "wwwww", (10, 8, 333, 64, 64): "wwwww",
    (1, 4, 5000, 64, 64): "xxxxx", (3, 8, 300, 32, 128): "wssww", (6, 8, 300, 128, 32): "wwwww",
    (2, 8, 200, 32, 32): "wwwww",
}
LAUNCH = dict(zip("wxs", OURS + (b"scan_mfma_kernel",)))


@pytest.mark.parametrize("shape", list(SHAPES), ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_forward_and_backward(cp, shape):
    N, H, L, E, M = shape
    Qb, Kb, Vb, G = _inputs(N, H, L, E, M, 60 + L)
    q, k, v = Qb.cuda(), Kb.cuda(), Vb.cuda()
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(q, k, v, out)
    used = [_last_kernel()]
    exact = oracle.forward(Qb.double(), Kb.double(), Vb.double())
    ref = oracle.forward(Qb.float(), Kb.float(), Vb.float())
    assert torch.isfinite(out).all()
    assert scale_error(out.cpu(), exact) <= max(2 * scale_error(ref, exact), 1e-6)
    grads = [torch.full((N, H, L, X), float("nan"), device="cuda", dtype=torch.bfloat16) for X in (E, E, M)]
    for i in range(3):   # one gradient at a time, then all: the launches differ
        alone = [None] * 3
        alone[i] = torch.full_like(grads[i], float("nan"))
        cp.causal_dot_backward_hip(q, k, v, G.cuda(), *alone)
        used.append(_last_kernel())
        grads[i] = alone[i]
    _check_gradients(str(shape), grads, Qb, Kb, Vb, G)
    together = [torch.full_like(g, float("nan")) for g in grads]
    cp.causal_dot_backward_hip(q, k, v, G.cuda(), *together)
    used.append(_last_kernel())
    _check_gradients(str(shape), together, Qb, Kb, Vb, G)
    assert used == [LAUNCH[x] for x in SHAPES[shape]]


@pytest.mark.parametrize("shape", [(2, 8, 700, 128, 128), (1, 3, 4500, 64, 64), (3, 8, 150, 96, 40)], ids=str)
def test_states_handed_in_and_out(cp, shape):
    """A piece of a sequence after another: rows and states against the whole in float64, the state
    within 2e-7 (fp32 sums of every eight chunks, added up)."""
    N, H, L, E, M = shape
    Qb, Kb, Vb, _ = _inputs(N, H, 2 * L, E, M, 70)
    q, k, v = Qb.cuda(), Kb.cuda(), Vb.cuda()
    first, state = cp.causal_dot_product_with_state(q[:, :, :L], k[:, :, :L], v[:, :, :L])
    second, last = cp.causal_dot_product_with_state(q[:, :, L:], k[:, :, L:], v[:, :, L:], state)
    assert _last_kernel() in OURS
    got = torch.cat([first, second], dim=2).cpu()
    exact = oracle.forward(Qb.double(), Kb.double(), Vb.double())
    assert scale_error(got, exact) <= 1e-6
    want = torch.einsum("nhle,nhlm->nhem", Kb.double(), Vb.double())
    assert ((last.cpu().double() - want).norm() / want.norm()).item() <= 2e-7


def test_rows_on_eight_byte_boundaries_and_interleaved_heads(cp):
    N, H, L, E, M = 2, 5, 130, 128, 100
    Qb, Kb, Vb, G = _inputs(N, H, L, E, M, 80)

    def placed(t):   # (N, L, H, X) storage, rows 8 bytes after a 16-byte boundary
        X = t.shape[3]
        buf = torch.zeros(N, L, H, X + 4, device="cuda", dtype=t.dtype)
        view = buf[..., 4:].permute(0, 2, 1, 3)
        view.copy_(t)
        return view
    q, k, v = placed(Qb), placed(Kb), placed(Vb)
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(q, k, v, out)
    assert _last_kernel() in OURS
    exact = oracle.forward(Qb.double(), Kb.double(), Vb.double())
    assert scale_error(out.cpu(), exact) <= 1e-6
    grads = [placed(torch.zeros_like(t)) for t in (Qb, Kb, Vb)]
    cp.causal_dot_backward_hip(q, k, v, G.cuda(), *grads)
    _check_gradients("eight bytes", grads, Qb, Kb, Vb, G)
    for g in grads:   # nothing beside the rows
        assert (g.permute(0, 2, 1, 3).as_strided((N, L, H, 4), (L * H * (g.shape[3] + 4), H * (g.shape[3] + 4),
                                                               g.shape[3] + 4, 1), 0) == 0).all()


def test_small_rows_and_columns_beside_large_ones(cp):
    """Every row and column of the product is within a few fp32 roundings on its own scale."""
    N, H, L, E, M = 2, 8, 500, 128, 128
    for small in ("q_rows", "k_columns", "v_columns"):
        Qb, Kb, Vb, _ = (t.double() for t in _inputs(N, H, L, E, M, 90))
        if small == "q_rows":
            Qb[:, :, 5::32] *= 2.0 ** -20
        elif small == "k_columns":
            Kb[..., ::2] *= 2.0 ** -20
            Qb[..., ::2] *= 2.0 ** 20
        else:
            Vb[..., ::2] *= 2.0 ** -20
        out = torch.empty(N, H, L, M, device="cuda")
        cp.causal_dot_product_hip(*(t.bfloat16().cuda() for t in (Qb, Kb, Vb)), out)
        assert _last_kernel() in OURS
        want = oracle.forward(Qb, Kb, Vb)
        got = out.cpu().double()
        for dim in (2, 3):
            assert ((got - want).norm(dim=dim) / want.norm(dim=dim)).max().item() <= 2e-6


def test_without_room_for_an_exchange(cp):
    """A workspace that the exchange does not fit in: the kernels that split L, not an error."""
    from fast_transformers_amd import _native
    lib = _native.load()
    N, H, L, E, M = 1, 4, 2154, 32, 32
    tensors = [t.cuda() for t in _inputs(N, H, L, E, M, 95)]
    want, got = ([torch.full_like(t, float("nan")) for t in tensors[:3]] for _ in range(2))
    cp.causal_dot_backward_hip(*tensors, *want)
    assert _last_kernel() == b"scan_tp_bf16_kernel (exchange)"
    full = lib.ftc_causal_dot_backward_workspace_bytes(N, H, L, E, M, _native.FTC_BF16)
    ws = torch.zeros(full, dtype=torch.uint8, device="cuda")
    d = [_native.describe(t) for t in tensors + got]
    call = lambda nbytes: lib.ftc_causal_dot_backward(
        *(ctypes.byref(x) for x in d), ctypes.c_void_p(ws.data_ptr()), nbytes,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    least = next(b for b in range(1 << 16, full + 1, 1 << 12) if call(b) == 0)
    torch.cuda.synchronize()
    assert least < full and _last_kernel() == b"scan_mfma_kernel"
    for a, b in zip(got, want):   # (either rounds an fp32 result to bf16)
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() <= 2e-3


@pytest.mark.parametrize("shape,kernel", [
    # long chains of 32 columns: cut, whole beyond the caches, an exchange of five and of ten segments
    ((1, 128, 2590, 32, 32), OURS[0]), ((1, 160, 5690, 32, 32), OURS[0]), ((8, 19, 4001, 64, 32), OURS[0]),
    ((3, 16, 5999, 64, 32), OURS[1]), ((2, 12, 11003, 64, 32), OURS[1])], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s
    if isinstance(s, tuple) else "")
def test_long_forward_scans_with_32_columns(cp, shape, kernel):
    N, H, L, E, M = shape
    Qb, Kb, Vb, _ = _inputs(N, H, L, E, M, 70 + L)
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(Qb.cuda(), Kb.cuda(), Vb.cuda(), out)
    assert _last_kernel() == kernel
    exact = oracle.forward(Qb.double(), Kb.double(), Vb.double())
    ref = oracle.forward(Qb.float(), Kb.float(), Vb.float())
    assert scale_error(out.cpu(), exact) <= max(2 * scale_error(ref, exact), 1e-6)
    norm = lambda t: ((t.double() - exact).norm() / exact.norm()).item()
    assert norm(out.cpu()) <= max(norm(ref), 1e-7)


@pytest.mark.parametrize("shape,kernel", [
    # whole chains of more than 128 chunks, in one round of workgroups and in three; an exchange on few chains
    ((4, 16, 4127, 32, 32), OURS[0]), ((2, 100, 5153, 32, 32), OURS[0]), ((1, 20, 11003, 32, 32), OURS[1]),
    ((5, 8, 6001, 32, 32), OURS[1])], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s if isinstance(s, tuple) else "")
def test_long_narrow_backward_scans(cp, shape, kernel):
    N, H, L, E, M = shape
    Qb, Kb, Vb, G = _inputs(N, H, L, E, M, 80 + L)
    grads = [torch.full((N, H, L, X), float("nan"), device="cuda", dtype=torch.bfloat16) for X in (E, E, M)]
    cp.causal_dot_backward_hip(Qb.cuda(), Kb.cuda(), Vb.cuda(), G.cuda(), *grads)
    assert _last_kernel() == kernel
    _check_gradients(str(shape), grads, Qb, Kb, Vb, G)
