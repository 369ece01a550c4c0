"""Chains of a few positions with a state handed in and out (ftc_short.hip), against the CPU
oracle in float64."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    # N, H, L, E, M: one position; remainders of the 64 columns and of the row groups; widths that
    # do not allow 16-byte loads; the widest state; the largest number of positions
    (32, 8, 1, 64, 64), (1, 1, 1, 1, 1), (2, 3, 1, 25, 33), (3, 2, 1, 512, 130), (2, 2, 1, 40, 100),
    (4, 8, 2, 64, 64), (4, 8, 4, 64, 68), (2, 5, 5, 64, 64), (3, 7, 8, 64, 64), (2, 2, 8, 128, 128),
    (2, 2, 7, 65, 129),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("with_initial", [True, False], ids=["continued", "fresh"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_h%d_l%d_e%d_m%d" % s)
def test_short_scan_with_state(shape, with_initial, dtype):
    from fast_transformers_amd import _native
    from fast_transformers_amd.causal_product import causal_dot_product_with_state
    N, H, L, E, M = shape
    Q, K, V, _ = oracle.make_inputs(N, H, L, E, M, seed=11, dtype=dtype)
    S = torch.randn(N, H, E, M, generator=torch.Generator().manual_seed(5)) if with_initial else None
    # rows as the (N, L, H, X) storage of a model has them
    nlh = lambda t: t.permute(0, 2, 1, 3).contiguous().cuda().permute(0, 2, 1, 3)
    got = causal_dot_product_with_state(nlh(Q), nlh(K), nlh(V), S.cuda() if with_initial else None)
    if L == 1 or dtype == torch.float32:
        assert _native.load().ftc_last_kernel() == b"short_scan_kernel"
    want = oracle.forward_with_state(Q.double(), K.double(), V.double(),
                                     S.double() if with_initial else None)
    # fp32 sums of at most E + 8 terms of either sign: (E + 8) 2^-24 of the sum of magnitudes
    mag = oracle.forward_with_state(Q.double(), K.double(), V.double().abs(),
                                    S.double().abs() if with_initial else None)
    for g, w, m in zip(got, want, mag):
        assert ((g.double().cpu() - w).abs() <= (E + L) * 2.0 ** -24 * m + 1e-30).all()
