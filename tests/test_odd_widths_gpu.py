"""fp32 rows of odd widths (and rows that are not 16-byte aligned) read and written where they lie
by the fp16-piece kernel, against the CPU oracle anchored on float64."""
import pytest
import torch

import oracle
from parity import scale_error

pytestmark = pytest.mark.gpu

SHAPES = [
    # N, H, L, E, M: quads that straddle the width by one, two and three words; one and two groups of
    # 32 state rows; two blocks of output columns; the smallest widths; whole, cut and exchanged chains;
    # both state shapes of a backward call in one launch (80 chains) and in two (99)
    (9, 11, 97, 25, 33), (10, 8, 130, 25, 33), (2, 4, 77, 41, 46), (3, 5, 65, 63, 63), (1, 3, 200, 8, 9),
    (2, 4, 300, 50, 70), (1, 5, 1500, 51, 27), (1, 3, 9000, 31, 62), (40, 4, 33, 30, 10),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_odd_widths_in_place(shape, monkeypatch):
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    monkeypatch.setenv("FTC_ODD", "1")  # (also where the copies would run on another kernel)
    cp.reload_tuning()
    try:
        _odd_widths_in_place(shape, cp, _native)
    finally:
        monkeypatch.delenv("FTC_ODD")
        cp.reload_tuning()


def _odd_widths_in_place(shape, cp, _native):
    N, H, L, E, M = shape
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=900 + L)
    nlh = lambda t: t.permute(0, 2, 1, 3).contiguous().cuda().permute(0, 2, 1, 3)  # NLHE storage
    q, k, v, g = (nlh(t) for t in (Q, K, V, G))
    # results inside larger buffers: nothing around a row may be touched
    def boxed(X):
        box = torch.full((N, L, H, X + 3), 7.0, device="cuda")
        return box, box[..., 1:X + 1].permute(0, 2, 1, 3)
    boxes, outs = zip(*(boxed(X) for X in (M, E, E, M)))
    cp.causal_dot_product_hip(q, k, v, outs[0])
    assert b"scan_tph_kernel" in _native.load().ftc_last_kernel()
    cp.causal_dot_backward_hip(q, k, v, g, *outs[1:])
    assert b"scan_tph_kernel" in _native.load().ftc_last_kernel()
    cp.check_workspaces()
    for box in boxes:
        assert (box[..., 0] == 7).all() and (box[..., -2:] == 7).all()
    want = (oracle.forward(Q, K, V),) + tuple(oracle.backward(Q, K, V, G))
    exact = (oracle.forward(Q.double(), K.double(), V.double()),) + \
        tuple(oracle.backward(Q.double(), K.double(), V.double(), G.double()))
    for got, ref, ex in zip(outs, want, exact):
        # no further from float64 than four times the fp32 oracle (or 2e-6 of the chain's largest)
        assert scale_error(got.cpu(), ex) <= max(4 * scale_error(ref, ex), 2e-6)


@pytest.mark.parametrize("shape,cuts", [((1, 2, 295, 31, 31), "0,2,4,8,10"), ((1, 2, 745, 25, 33), "0,10,18,22,24")],
                         ids=["32_rows", "64_rows"])
def test_three_pieces_cut_at_half_a_trip(shape, cuts):
    """Segments that start at 2 modulo 4 chunks, after a first walk of two positions and of more; one and two groups
    of 32 state rows."""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    line = _native.plan((N, H, L, E), (N, H, L, M))
    assert line.startswith("scan_tp_kernel: 1 scan") and "cuts at chunks %s," % cuts in line
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=41)
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    cp.causal_dot_product_hip(Q.cuda(), K.cuda(), V.cuda(), out)
    assert _native.load().ftc_last_kernel() == b"scan_tp_kernel"
    exact = oracle.forward(Q.double(), K.double(), V.double())
    assert scale_error(out.cpu(), exact) <= max(4 * scale_error(oracle.forward(Q, K, V), exact), 2e-6)


def test_odd_widths_with_no_room_for_an_exchange():
    """A long chain whose segments would exchange their sums, with a workspace that has room for
    the generic kernel only: served as before, and not refused."""
    import ctypes
    from fast_transformers_amd import _native
    N, H, L, E, M = 1, 3, 9000, 50, 50
    lib = _native.load()
    plan = _native.plan((N, H, L, E), (N, H, L, M))
    assert "scan_tph_kernel (exchange)" in plan
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=31)
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    q, k, v = (t.cuda() for t in (Q, K, V))
    d = [_native.describe(t) for t in (q, k, v, out)]
    room = int(plan.split("workspace ")[1].split()[0]) - 256
    ws = torch.zeros(room, dtype=torch.uint8, device="cuda")
    rc = lib.ftc_causal_dot_product(*(ctypes.byref(t) for t in d), ctypes.c_void_p(ws.data_ptr()),
                                    ctypes.c_size_t(room), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.last_error()
    assert lib.ftc_last_kernel() == b"generic_scan_kernel"
    exact = oracle.forward(Q.double(), K.double(), V.double())
    assert scale_error(out.cpu(), exact) <= max(4 * scale_error(oracle.forward(Q, K, V), exact), 2e-6)


def _each(got, exact, dim):
    """The largest 2-norm error of a row (dim 3) or column (dim 2) over its own 2-norm."""
    got, exact = got.double(), exact.double()
    return ((got - exact).norm(dim=dim) / exact.norm(dim=dim)).max().item()


def test_odd_widths_with_no_room_for_their_copies():
    """A workspace for the VALU kernel alone has that kernel run, although rows read where they lie
    would not need more."""
    import ctypes
    from fast_transformers_amd import _native
    N, H, L, E, M = 2, 8, 333, 50, 50
    lib = _native.load()
    assert "scan_tph_kernel" in _native.plan((N, H, L, E), (N, H, L, M))
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=32)
    Q[..., ::2] *= 2.0 ** -20
    V[..., ::2] *= 2.0 ** -20
    out = torch.full((N, H, L, M), float("nan"), device="cuda")
    q, k, v = (t.cuda() for t in (Q, K, V))
    d = [_native.describe(t) for t in (q, k, v, out)]
    room = 8 << 20
    assert room < lib.ftc_causal_dot_product_workspace_bytes(N, H, L, E, M, 0)
    ws = torch.zeros(room, dtype=torch.uint8, device="cuda")
    rc = lib.ftc_causal_dot_product(*(ctypes.byref(t) for t in d), ctypes.c_void_p(ws.data_ptr()),
                                    ctypes.c_size_t(room), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _native.last_error()
    assert lib.ftc_last_kernel() == b"generic_scan_kernel"
    exact, ref = oracle.forward(Q.double(), K.double(), V.double()), oracle.forward(Q, K, V)
    for dim in (2, 3):
        assert _each(out.cpu(), exact, dim) <= max(4 * _each(ref, exact, dim), 2e-6)


# calls whose aligned counterparts run on kernels that hold every fp32 value exactly: too few rows
# for copies; few chains of narrow rows; of a backward call, some scans only (the results named)
EXACT = [((1, 1, 100, 25, 33), "oqkv"), ((1, 1, 1356, 18, 18), "oqkv"), ((9, 11, 1531, 25, 33), "ov")]


@pytest.mark.parametrize("shape, results", EXACT, ids=lambda s: s if isinstance(s, str) else "n%d_h%d_l%d_e%d_m%d" % s)
@pytest.mark.parametrize("small", ["q_rows", "q_columns", "k_columns", "v_columns", "g_rows", "g_columns", "v_early_rows"])
def test_small_rows_and_columns_beside_large_ones(small, shape, results):
    """Every row and column is as close to float64, on its own scale, as the fp32 oracle's, where
    the widths' multiples of 32 are."""
    import fast_transformers_amd.causal_product as cp
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
    for name, got, ref, ex in zip("oqkv", outs, refs, exact):
        for dim in (2, 3):
            if name in results:
                assert _each(got.cpu(), ex, dim) <= max(4 * _each(ref, ex, dim), 2e-6)


THREE_PIECES = [
    # N, H, L, E, M: states of one and two groups of 32 rows and of one and two blocks of 64; quads that
    # straddle the width of a first and of a second block by one, two and three words; widths on either
    # side of a block; one to three blocks of output columns; whole, cut and exchanged chains; scans of a
    # backward call in one launch and in two
    (9, 11, 97, 25, 33), (3, 2, 200, 10, 9), (2, 4, 300, 63, 31), (1, 3, 2100, 18, 18), (2, 3, 333, 33, 70),
    (2, 4, 130, 65, 63), (3, 3, 220, 70, 70), (1, 5, 900, 95, 97), (1, 2, 2600, 99, 101), (2, 2, 260, 127, 127),
    (1, 4, 150, 110, 150), (5, 8, 33, 75, 11), (2, 4, 100, 35, 77), (1, 6, 90, 127, 63),
]


@pytest.mark.parametrize("shape", THREE_PIECES, ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_odd_widths_in_place_on_three_pieces(shape, monkeypatch):
    """As above on the kernel of three bf16 pieces, with rows that have NaN beside them and with a state
    handed in and out."""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    monkeypatch.setenv("FTC_ODD", "2")  # (also where another kernel would take them)
    cp.reload_tuning()
    try:
        Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=950 + L)

        def boxed(t, X, fill):
            box = torch.full((N, L, H, X + 3), fill, device="cuda")
            view = box[..., 1:X + 1].permute(0, 2, 1, 3)
            if t is not None:
                view.copy_(t)
            return box, view
        q, k, v, g = (boxed(t, t.shape[3], float("nan"))[1] for t in (Q, K, V, G))
        boxes, outs = zip(*(boxed(None, X, 7.0) for X in (M, E, E, M)))
        cp.causal_dot_product_hip(q, k, v, outs[0])
        assert b"scan_tp_kernel" in _native.load().ftc_last_kernel()
        cp.causal_dot_backward_hip(q, k, v, g, *outs[1:])
        if max(E, M) <= 128:
            assert b"scan_tp_kernel" in _native.load().ftc_last_kernel()
        s0 = torch.randn(N, H, E, M, generator=torch.Generator().manual_seed(L))
        out, s1 = cp.causal_dot_product_with_state(q, k, v, s0.cuda())
        cp.check_workspaces()
        for box in boxes:
            assert (box[..., 0] == 7).all() and (box[..., -2:] == 7).all()
        want = (oracle.forward(Q, K, V),) + tuple(oracle.backward(Q, K, V, G))
        d = [t.double() for t in (Q, K, V, G)]
        exact = (oracle.forward(*d[:3]),) + tuple(oracle.backward(*d))
        for got, ref, ex in zip(outs, want, exact):
            assert scale_error(got.cpu(), ex) <= max(4 * scale_error(ref, ex), 2e-6)
        with_state = exact[0] + d[0] @ s0.double()
        assert scale_error(out.cpu(), with_state) <= max(4 * scale_error(want[0], exact[0]), 2e-6)
        assert scale_error(s1.cpu(), s0.double() + d[1].transpose(2, 3) @ d[2]) <= max(4 * scale_error(want[0], exact[0]), 2e-6)
    finally:
        monkeypatch.delenv("FTC_ODD")
        cp.reload_tuning()


def test_many_long_chains_in_place():
    """More than two rounds of workgroups on chains of more than 128 chunks: as close to float64 as the
    fp32 oracle (copies were two to four times as far away)."""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = 9, 20, 4100, 9, 11
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=961)
    grads = [torch.full_like(t, float("nan")).cuda() for t in (Q, K, V)]
    cp.causal_dot_backward_hip(*(t.cuda() for t in (Q, K, V, G)), *grads)
    assert _native.load().ftc_last_kernel() == b"scan_tp_kernel"
    exact, ref = oracle.backward(*(t.double() for t in (Q, K, V, G))), oracle.backward(Q, K, V, G)
    for got, r, ex in zip(grads, ref, exact):
        assert ((got.cpu() - ex).norm() / ex.norm()).item() <= max(((r - ex).norm() / ex.norm()).item(), 5e-7)


TOGETHER = [
    # N, H, L, E, M (widths that need no copies): two state shapes side by side, whole, cut and exchanged
    # chains, one and two groups of 32 rows, a single chunk, ragged ends; 32 x 32; and two shapes of which
    # one has two blocks of rows, with one to three blocks of columns between the scans
    (2, 3, 70, 32, 64), (1, 1, 32, 64, 32), (5, 4, 300, 24, 48), (2, 4, 2050, 64, 32), (1, 2, 5000, 60, 20),
    (9, 9, 90, 20, 36), (4, 8, 200, 32, 32), (2, 2, 33, 20, 24), (1, 1, 3500, 32, 32),
    (2, 3, 70, 64, 128), (3, 4, 300, 128, 32), (1, 5, 33, 72, 100), (6, 5, 700, 100, 40), (1, 2, 450, 96, 128),
]


@pytest.mark.parametrize("shape", TOGETHER, ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_narrow_scans_share_a_launch(shape):
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    plan = _native.plan((N, H, L, E), (N, H, L, M), backward=True)
    assert plan.startswith("scan_tp_kernel") and ": 3 scans" in plan and plan.count("workgroups") == 1
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=970 + L)
    d = [t.double() for t in (Q, K, V, G)]
    q, k, v, g = (t.permute(0, 2, 1, 3).contiguous().cuda().permute(0, 2, 1, 3) for t in (Q, K, V, G))
    outs = [torch.empty_like(t) for t in (v, q, k, v)]
    cp.causal_dot_product_hip(q, k, v, outs[0])
    cp.causal_dot_backward_hip(q, k, v, g, *outs[1:])
    s0 = torch.randn(N, H, E, M, generator=torch.Generator().manual_seed(L))
    out, s1 = cp.causal_dot_product_with_state(q, k, v, s0.cuda())
    if E == M:   # (32 x 32: a single scan of these sizes is taken too)
        assert _native.load().ftc_last_kernel().startswith(b"scan_tp_kernel")
    cp.check_workspaces()
    want = (oracle.forward(Q, K, V),) + tuple(oracle.backward(Q, K, V, G))
    exact = (oracle.forward(*d[:3]),) + tuple(oracle.backward(*d))
    for got, ref, ex in zip(outs, want, exact):
        assert scale_error(got.cpu(), ex) <= max(4 * scale_error(ref, ex), 2e-6)
    bound = max(4 * scale_error(want[0], exact[0]), 2e-6)
    assert scale_error(out.cpu(), exact[0] + d[0] @ s0.double()) <= bound
    assert scale_error(s1.cpu(), s0.double() + d[1].transpose(2, 3) @ d[2]) <= bound
    # one gradient by itself is the same to rounding, whatever launch it is in
    alone = torch.empty_like(q)
    cp.causal_dot_backward_hip(q, k, v, g, None, alone, None)
    assert scale_error(alone.cpu(), exact[2]) <= max(4 * scale_error(want[2], exact[2]), 2e-6)


CLIPPED = [
    # N, H, L, E, M, backward: tiles that rows do not fill, of each state shape; widths one, two and three values into a
    # quad, on it, and the narrowest; ends of chains inside a chunk, chains of a chunk and some; one launch of
    # two scans, a call whose other scans run where their rows lie, operands that need no copy
    (9, 11, 1531, 25, 33, True), (16, 21, 413, 9, 34, True), (3, 20, 1000, 45, 31, True), (2, 3, 97, 27, 63, True),
    (1, 4, 5000, 33, 32, False), (1, 2, 800, 32, 127, False), (30, 20, 70, 64, 35, False), (1, 3, 2000, 31, 64, False),
    (30, 20, 70, 62, 64, True),
]


@pytest.mark.parametrize("shape", CLIPPED, ids=lambda s: "n%d_h%d_l%d_e%d_m%d_%s" % (s[:5] + ("bwd" if s[5] else "fwd",)))
def test_results_of_copies_go_where_they_belong(shape):
    """Scans on copies whose kernel splits L store odd rows themselves: the oracle's values, and nothing around them."""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M, backward = shape
    plan = _native.plan((N, H, L, E), (N, H, L, M), backward=backward)
    if shape[:2] != (2, 3):   # (rows too few for copies)
        assert "scan_dma_kernel" in plan and ", 0 results copied back" in plan, plan
    Q, K, V, G = oracle.make_inputs(N, H, L, E, M, seed=700 + L)

    def boxed(X):   # rows of odd strides, on 4-byte boundaries, among other values
        box = torch.full((N, H, L + 1, X + 3), 7.0, device="cuda")
        box[:, :, :L, 1:1 + X] = float("nan")
        return box, box[:, :, :L, 1:1 + X]

    q, k, v, g = (t.cuda() for t in (Q, K, V, G))
    if backward:
        boxes = [boxed(X) for X in (E, E, M)]
        for _ in range(2):
            cp.causal_dot_backward_hip(q, k, v, g, *(o for _, o in boxes))
        exact = oracle.backward(*(t.double() for t in (Q, K, V, G)))
        ref = oracle.backward(Q, K, V, G)
    else:
        boxes = [boxed(M)]
        for _ in range(2):
            cp.causal_dot_product_hip(q, k, v, boxes[0][1])
        exact, ref = [oracle.forward(*(t.double() for t in (Q, K, V)))], [oracle.forward(Q, K, V)]
    for (box, out), want, plain in zip(boxes, exact, ref):
        assert scale_error(out.cpu(), want) <= max(4 * scale_error(plain, want), 2e-6)
        box[:, :, :L, 1:-2] = 7.0
        assert (box == 7.0).all()


@pytest.mark.parametrize("offset", [0, 8, 64], ids=["same", "eight_rows_on", "two_chunks_on"])
@pytest.mark.parametrize("shape", [(30, 20, 70, 64, 35), (2, 5, 1500, 32, 41)], ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_an_odd_result_over_rows_that_are_read_in_place(shape, offset):
    """Scans on copies of v whose a and b stay where they are, and a result of odd rows that goes over those, from the
    same row on or from later ones: as if it had gone elsewhere.  (Beside them it goes where it belongs at once.)"""
    from fast_transformers_amd import _native
    import fast_transformers_amd.causal_product as cp
    N, H, L, E, M = shape
    plan = _native.plan((N, H, L, E), (N, H, L, M))
    assert "1 operand copied" in plan and ", 0 results copied back" in plan and "scan_dma_kernel" in plan, plan
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=720 + L)
    exact, ref = oracle.forward(*(t.double() for t in (Q, K, V))), oracle.forward(Q, K, V)
    k, v = K.cuda(), V.cuda()
    room = torch.zeros(N, H, L + 64, E + 64, device="cuda")
    for first in (E, 0) if M > E else (E, E - M):   # beside the rows of q, over them
        q, out = room[:, :, :L, :E], room[:, :, offset:offset + L, first:first + M]
        q.copy_(Q)
        cp.causal_dot_product_hip(q, k, v, out)
        assert scale_error(out.cpu(), exact) <= max(4 * scale_error(ref, exact), 2e-6)
    cp.check_workspaces()
