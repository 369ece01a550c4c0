"""Host-side planning of the launches (which kernel, how chains are cut, how much workspace),
read through ``ftc_causal_dot_plan``: nothing is launched, no GPU is needed.

The figures pinned here are the planner's rules as documented where the planner lives
(csrc/ftc_mfma.hip): one workgroup per chain segment on up to 256 CUs, chains of up to 64
chunks cut without an exchange at multiples of four chunks (two where fp32 rows are multiplied in
three bf16 pieces) with later segments shorter,
longer chains on few CUs with an exchange, everything the MFMA kernels do not cover on the
generic kernel."""
import re

import pytest

from fast_transformers_amd import _native


def lines(q, v, **kw):
    return [l for l in _native.plan(q, v, **kw).split("\n") if l]


def kernel(line):
    """The launch's kernel, with its form: "scan_tp_bf16_kernel (exchange)"."""
    return line.split(":")[0]


def field(line, pattern):
    m = re.search(pattern, line)
    assert m, (pattern, line)
    return m.group(1)


def test_headline_shape():
    fwd = lines((10, 8, 1000, 64), (10, 8, 1000, 64))
    assert len(fwd) == 1 and fwd[0].startswith("scan_tph_kernel:")
    assert "3 segments" in fwd[0] and "cuts at chunks 0,20,28,32" in fwd[0]
    assert "240 workgroups" in fwd[0] and "workspace 0 bytes" in fwd[0]
    bwd = lines((10, 8, 1000, 64), (10, 8, 1000, 64), backward=True)
    assert len(bwd) == 1 and bwd[0].startswith("scan_tph_kernel: 3 scans")
    assert "1 segment " in bwd[0] and "240 workgroups" in bwd[0]


def test_long_chains_exchange_their_segment_sums():
    fwd = lines((1, 16, 65536, 64), (1, 16, 65536, 64))
    assert fwd[0].startswith("scan_tph_kernel (exchange):")
    assert "16 segments of 4096 rows" in fwd[0] and "256 workgroups" in fwd[0]
    need = int(field(fwd[0], r"workspace (\d+) bytes"))
    lib = _native.load()
    assert 0 < need <= lib.ftc_causal_dot_product_workspace_bytes(1, 16, 65536, 64, 64, 0)
    # three scans of 16 chains: one round of workgroups would need segments of 412 chunks, so
    # just under two rounds of shorter ones
    bwd = lines((1, 16, 65536, 64), (1, 16, 65536, 64), backward=True)
    assert bwd[0].startswith("scan_tph_kernel (exchange): 3 scans")
    assert "10 segments of 6656 rows" in bwd[0] and "480 workgroups" in bwd[0]
    need = int(field(bwd[0], r"workspace (\d+) bytes"))
    assert 0 < need <= lib.ftc_causal_dot_backward_workspace_bytes(1, 16, 65536, 64, 64, 0)
    # more workgroups than CUs: three rounds for 32 chains of 2048 chunks
    bwd = lines((2, 16, 65536, 64), (2, 16, 65536, 64), backward=True)
    assert bwd[0].startswith("scan_tph_kernel (exchange): 3 scans")
    assert "8 segments of 8192 rows" in bwd[0] and "768 workgroups" in bwd[0]
    # chains of 257 to 1024 chunks on 112 workgroups or more are walked whole, in any number of
    # rounds; on fewer they exchange
    bwd = lines((4, 16, 16384, 64), (4, 16, 16384, 64), backward=True)
    assert bwd[0].startswith("scan_tph_kernel: 3 scans") and "1 segment of 16384 rows" in bwd[0]
    assert lines((4, 16, 16384, 64), (4, 16, 16384, 64))[0].startswith("scan_tph_kernel (exchange):")
    assert lines((3, 64, 16384, 64), (3, 64, 16384, 64), backward=True)[0].startswith("scan_tph_kernel: 3 scans")
    assert lines((3, 64, 16384, 64), (3, 64, 16384, 64))[0].startswith("scan_tph_kernel: 1 scan")
    assert lines((1, 36, 16384, 64), (1, 36, 16384, 64), backward=True)[0].startswith("scan_tph_kernel (exchange)")
    assert lines((4, 64, 40000, 64), (4, 64, 40000, 64), backward=True)[0].startswith("scan_dma_kernel")
    assert lines((8, 16, 8192, 64), (8, 16, 8192, 64), backward=True)[0].startswith("scan_tph_kernel:")
    # two segments of up to 64 chunks: chains cut in two without an exchange instead
    assert lines((1, 96, 4096, 64), (1, 96, 4096, 64))[0].startswith("scan_tph_kernel: 1 scan")
    assert "cuts at chunks 0,92,128" in lines((1, 32, 4096, 64), (1, 32, 4096, 64), backward=True)[0]
    assert lines((1, 96, 8192, 64), (1, 96, 8192, 64))[0].startswith("scan_tph_kernel (exchange):")
    # config 4's operator shape
    op = lines((10, 8, 4096, 64), (10, 8, 4096, 64))
    assert op[0].startswith("scan_tph_kernel (exchange):") and "3 segments of 1408 rows" in op[0]


def test_what_the_chain_parallel_kernel_leaves_to_the_others():
    # rows that lie too far apart for one 32-bit descriptor per chain
    far = (144 * 8192 * 65536, 8192 * 65536, 65536, 1)
    out = lines((1, 144, 8192, 64), (1, 144, 8192, 64), strides=(far, far, far))
    assert not out[0].startswith("scan_tp_kernel")
    # more chains than two rounds of workgroups
    many = lines((64, 16, 128, 64), (64, 16, 128, 64))
    assert many[0].startswith("scan_dma_kernel")
    # ... which chains of 16 chunks or more fill without losing to them
    assert lines((64, 16, 512, 64), (64, 16, 512, 64), backward=True)[0].startswith("scan_tph_kernel: 3 scans")
    assert lines((64, 16, 256, 64), (64, 16, 256, 64), backward=True)[0].startswith("scan_dma_kernel")
    assert lines((32, 16, 256, 64), (32, 16, 256, 64), backward=True)[0].startswith("scan_tph_kernel: 3 scans")
    # other state sizes and element types
    assert lines((10, 8, 1000, 32), (10, 8, 1000, 32))[0].startswith("scan_dma_kernel")
    # (32 rows or columns: the chain-parallel kernel on whole chains unless both are 32,
    # the kernels that split L where it would need an exchange)
    assert lines((10, 8, 1000, 32), (10, 8, 1000, 128))[0].startswith("scan_tph_kernel:")
    assert lines((4, 16, 16384, 32), (4, 16, 16384, 128))[0].startswith("scan_dma_kernel")
    # few chains too short for an exchange: cut or whole on the chain-parallel kernel all the same
    assert lines((1, 3, 500, 128), (1, 3, 500, 128))[0].startswith("scan_mfma_kernel")
    assert lines((1, 3, 500, 128), (1, 3, 500, 128), backward=True)[0].startswith("scan_tp_kernel: 3 scans")
    assert lines((1, 8, 640, 64), (1, 8, 640, 64))[0].startswith("scan_tph_kernel: 1 scan")
    # bf16 rows: the chain-parallel kernel that multiplies them as they are, on whole and cut chains and with
    # an exchange, but for single scans of few wide chains and the shapes with 32 rows or columns below
    def bf16(N, H, L, E, M, backward=False):
        return lines((N, H, L, E), (N, H, L, M), backward=backward, dtype=_native.FTC_BF16)
    tp, tpx = "scan_tp_bf16_kernel", "scan_tp_bf16_kernel (exchange)"
    for N, H, L in ((4, 8, 1000), (10, 8, 1000), (14, 8, 1000), (16, 8, 1000), (16, 16, 1000), (16, 8, 4096),
                    (24, 8, 4096)):
        assert kernel(bf16(N, H, L, 64, 64)[0]) == tp, (N, H, L)
    assert kernel(bf16(1, 8, 2048, 64, 64)[0]) == tpx
    assert bf16(1, 8, 2048, 64, 64, True)[0].startswith(tpx + ": 3 scans")
    whole = bf16(1, 64, 16384, 64, 64, True)[0]
    assert whole.startswith(tp + ": 3 scans") and "1 segment of 16384 rows" in whole
    assert bf16(10, 8, 1000, 64, 64, True)[0].startswith(tp + ": 3 scans")
    # narrow keys, wide values: with a workgroup for every CU the backward's scans (bf16 results) walk their
    # chains whole, however long; the forward, whose fp32 results would have to be exchanged, and half as
    # many chains are left to the kernels that split L
    wide_values = bf16(4, 32, 16384, 32, 128, True)
    assert [kernel(l) for l in wide_values] == [tp, tp] and all("1 segment of 16384 rows" in l for l in wide_values)
    assert "2 scans" in wide_values[0] and "state 128 x 32" in wide_values[0] and "state 32 x 128" in wide_values[1]
    assert kernel(bf16(4, 32, 16384, 32, 128)[0]) == "scan_mfma_kernel"
    assert {kernel(l) for l in bf16(2, 32, 16384, 32, 128, True)} == {"scan_mfma_kernel"}
    # other launches that those kernels are faster at: many short chains, single scans of 32 x 32 on few long
    # chains, of wide states on fewer than eight workgroups
    assert kernel(bf16(64, 16, 128, 64, 64)[0]) == kernel(bf16(16, 64, 128, 64, 64, True)[0]) == "scan_mfma_kernel"
    assert kernel(bf16(64, 16, 512, 64, 64)[0]) == kernel(bf16(16, 64, 512, 64, 64, True)[0]) == tp
    assert kernel(bf16(1, 16, 4096, 32, 32)[0]) == "scan_mfma_kernel"
    assert kernel(bf16(1, 16, 4096, 32, 32, True)[0]) == tpx and kernel(bf16(32, 8, 4096, 32, 32)[0]) == tp
    assert kernel(bf16(1, 1, 1000, 128, 128)[0]) == "scan_mfma_kernel" and kernel(bf16(1, 8, 1000, 128, 128)[0]) == tpx
    # widths that the kernels that split L would only take as padded copies
    assert kernel(bf16(6, 8, 257, 48, 40)[0]) == tp
    assert kernel(bf16(8, 8, 130, 20, 20)[0]) == tp
    # rows of 128 values
    assert kernel(bf16(10, 8, 1000, 128, 128, True)[0]) == tp
    # odd widths: zero-padded dense copies for the matrix-core kernels when there are enough
    # rows to pay for the extra launches; states of more than 128 rows stay generic
    # (queries and keys are copied, the values and the product stay where they are; in the
    # backward the two copies serve all three scans, and dQ and dK are copied back)
    odd = lines((8, 16, 4096, 25), (8, 16, 4096, 64))
    assert odd[0].startswith("pad_rows_kernel: 2 operands") and "0 results" in odd[0]
    assert odd[1].startswith("scan_tph_kernel") and "state 32 x 64" in odd[1]
    odd = lines((8, 16, 4096, 25), (8, 16, 4096, 64), backward=True)
    assert odd[0].startswith("pad_rows_kernel: 2 operands") and "2 results" in odd[0]
    assert odd[1].startswith("scan_tph_kernel: 2 scans") and "state 64 x 32" in odd[1]
    # ... and where every operand would be copied, the kernel that takes odd widths where they lie, on any
    # number of workgroups; not where one shape has no plan of its own and all of them need an exchange
    wide = lines((8, 16, 4096, 99), (8, 16, 4096, 101), backward=True)
    assert len(wide) == 1 and wide[0].startswith("scan_tp_kernel: 3 scans") and "768 workgroups" in wide[0]
    assert lines((9, 20, 4100, 9), (9, 20, 4100, 11), backward=True)[0].startswith("scan_tp_kernel: 3 scans")
    assert lines((1, 200, 9000, 75), (1, 200, 9000, 10), backward=True)[0].startswith("pad_rows_kernel: 4 operands")
    # ... nor many short chains of up to 32 rows or columns
    assert lines((1, 1896, 16, 18), (1, 1896, 16, 84), backward=True)[0].startswith("pad_rows_kernel: 4 operands")
    assert lines((1, 600, 16, 18), (1, 600, 16, 84), backward=True)[0].startswith("scan_tp_kernel: 2 scans")
    assert lines((1, 4000, 16, 70), (1, 4000, 16, 70), backward=True)[0].startswith("scan_tp_kernel: 3 scans")
    assert lines((2, 2, 40, 10), (2, 2, 40, 3))[0].startswith("generic_scan_kernel")
    # (bf16 rows of such a scan are converted into fp32 copies on the way)
    assert lines((1, 2, 8192, 300), (1, 2, 8192, 64), dtype=_native.FTC_BF16)[0] \
        .startswith("pad_rows_kernel: 3 operands")
    assert lines((1, 2, 100, 300), (1, 2, 100, 64), dtype=_native.FTC_BF16)[0] \
        .startswith("generic_scan_kernel")   # (too few rows for the copies)
    # states of 129 to 512 rows: up to four scans over a split of the rows, the later ones'
    # rows added to the first one's
    three = lines((1, 2, 8192, 300), (1, 2, 8192, 64))
    assert [l.split(":")[0].split(" ")[0] for l in three] == \
        ["scan_tp_kernel", "scan_tp_kernel", "add_rows_kernel", "scan_tph_kernel", "add_rows_kernel"]
    assert "state 128 x 64" in three[0] and "state 128 x 64" in three[1] and "state 44 x 64" in three[3]
    two = lines((1, 2, 8192, 200), (1, 2, 8192, 64))
    assert "state 128 x 64" in two[0] and "state 72 x 64" in two[1] and two[2].startswith("add_rows_kernel: 1 result")
    two = lines((4, 8, 1000, 200), (4, 8, 1000, 200), backward=True)
    assert two[0].startswith("scan_tp_kernel: 3 scans") and "state 128 x 200" in two[0]
    assert "state 72 x 200" in two[1] and two[2].startswith("add_rows_kernel: 3 results")
    odd = lines((2, 4, 700, 255), (2, 4, 700, 129))
    assert odd[0].startswith("pad_rows_kernel: 3 operands") and "state 128 x 160" in odd[1]
    odd = lines((2, 4, 700, 255), (2, 4, 700, 129), backward=True)
    assert odd[0].startswith("pad_rows_kernel: 4 operands") and "3 results" in odd[0]
    # nothing to do
    assert lines((0, 8, 100, 64), (0, 8, 100, 64)) == []


@pytest.mark.parametrize("L", [33, 129, 500, 1000, 1500, 2048])
@pytest.mark.parametrize("chains", [(2, 8), (5, 8), (10, 8), (30, 4)])
def test_cut_chains(chains, L):
    """Cuts at multiples of four chunks, the last one at the end, at most 256 workgroups, and
    the longest workgroup (a chunk walked for its state alone counted as 0.6 of a full one)
    no longer than with equal segments (of whole groups of four chunks)."""
    N, H = chains
    line = lines((N, H, L, 64), (N, H, L, 64))[0]
    if not line.startswith("scan_tph_kernel:"):
        return
    cuts = [int(x) for x in field(line, r"cuts at chunks ([\d,]*\d)").split(",")]
    nseg = int(field(line, r"(\d+) segments? of"))
    assert len(cuts) == nseg + 1 and cuts[0] == 0 and cuts[-1] == (L + 31) // 32
    assert all(c % 4 == 0 for c in cuts[:-1])
    lengths = [b - a for a, b in zip(cuts, cuts[1:])]
    assert all(x > 0 for x in lengths)
    longest = max(0.6 * a + (b - a) for a, b in zip(cuts, cuts[1:]))
    step = -(-(-(-cuts[-1] // nseg)) // 4) * 4   # equal segments of whole groups of four
    equal = [min(i * step, cuts[-1]) for i in range(nseg + 1)]
    assert longest <= max(0.6 * a + (b - a) for a, b in zip(equal, equal[1:])) + 1e-9
    assert N * H * nseg <= 256 and int(field(line, r"(\d+) workgroups")) == N * H * nseg


def test_wide_states_on_the_chain_parallel_kernel():
    """fp32 states of more than 32 and up to 128 rows and columns, widths multiples of 4: two
    blocks of rows per chunk, a workgroup per block of 64 output columns."""
    fwd = lines((8, 16, 4096, 128), (8, 16, 4096, 128))
    assert len(fwd) == 1 and fwd[0].startswith("scan_tp_kernel: 1 scan")
    assert "state 128 x 128" in fwd[0] and "256 workgroups" in fwd[0] and "workspace 0 bytes" in fwd[0]
    bwd = lines((8, 16, 4096, 128), (8, 16, 4096, 128), backward=True)
    assert len(bwd) == 1 and bwd[0].startswith("scan_tp_kernel: 3 scans") and "768 workgroups" in bwd[0]
    # widths that leave the last block partly empty need no copies
    odd = lines((8, 16, 4096, 100), (8, 16, 4096, 68), backward=True)
    assert [l.split(":")[0] for l in odd] == ["scan_tp_kernel", "scan_tp_kernel"]
    assert "2 scans" in odd[0] and "state 68 x 100" in odd[0] and "state 100 x 68" in odd[1]
    # one block of columns: as many workgroups as chains
    assert "256 workgroups" in lines((16, 16, 4000, 128), (16, 16, 4000, 64))[0]
    # long chains: segment sums are exchanged, also with more workgroups than CUs
    long = lines((4, 16, 16384, 128), (4, 16, 16384, 128), backward=True)
    assert long[0].startswith("scan_tp_kernel (exchange): 3 scans") and "2 segments of 8192 rows" in long[0]
    need = int(field(long[0], r"workspace (\d+) bytes"))
    assert need == 65536 + 2 * 4 * 768 * 128 * 16 * 4
    # more workgroups than CUs: segments chosen so that the rounds of 256 are full
    rounds = lines((1, 16, 20000, 128), (1, 16, 20000, 128), backward=True)
    assert "8 segments of 2560 rows" in rounds[0] and "768 workgroups" in rounds[0]
    # few chains: shapes that the kernels which split L also take go to those below half
    # the CUs, the others go to the chain-parallel kernel at any size
    assert lines((1, 8, 512, 128), (1, 8, 512, 128))[0].startswith("scan_mfma_kernel")
    assert lines((1, 8, 256, 128), (1, 8, 256, 128))[0].startswith("scan_tp_kernel: 1 scan")
    assert lines((1, 8, 512, 128), (1, 8, 512, 128), backward=True)[0].startswith("scan_tp_kernel: 3 scans")
    assert lines((1, 40, 16384, 128), (1, 40, 16384, 32))[0].startswith("scan_mfma_kernel")
    # ... unless four or more segments of every chain fit one round of workgroups: an exchange
    # from 24 chunks on, in segments of down to four chunks
    few = lines((1, 8, 2048, 128), (1, 8, 2048, 128))[0]
    assert few.startswith("scan_tp_kernel (exchange):") and "16 segments of 128 rows" in few
    few = lines((1, 16, 2048, 64), (1, 16, 2048, 64))[0]
    assert few.startswith("scan_tph_kernel (exchange):") and "16 segments of 128 rows" in few
    assert lines((1, 16, 1024, 64), (1, 16, 1024, 64), backward=True)[0].startswith("scan_tph_kernel: 3 scans")
    assert lines((1, 16, 2048, 64), (1, 16, 2048, 64), backward=True)[0].startswith("scan_tph_kernel (exchange)")
    assert lines((1, 1, 2048, 64), (1, 1, 2048, 64))[0].startswith("scan_dma_kernel")
    assert lines((1, 4, 500, 100), (1, 4, 500, 100))[0].startswith("scan_tp_kernel: 1 scan")
    assert lines((1, 4, 1000, 100), (1, 4, 1000, 100))[0].startswith("scan_tp_kernel (exchange): 1 scan")
    # thousands of chains of one or two chunks with a small state, 32-wide shapes on more
    # than two rounds of workgroups: the other routes
    assert lines((512, 16, 64, 20), (512, 16, 64, 20))[0].startswith("pad_rows_kernel")
    assert lines((512, 16, 64, 32), (512, 16, 64, 128))[0].startswith("scan_dma_kernel")
    assert lines((512, 16, 64, 100), (512, 16, 64, 100))[0].startswith("scan_tp_kernel")
    # 32-wide shapes on few workgroups: the kernels that split L unless the chains are short
    assert lines((1, 32, 4096, 32), (1, 32, 4096, 128))[0].startswith("scan_dma_kernel")
    assert lines((1, 32, 1024, 32), (1, 32, 1024, 128))[0].startswith("scan_tph_kernel:")
    assert lines((1, 64, 4096, 32), (1, 64, 4096, 128))[0].startswith("scan_tph_kernel:")
    cut = lines((1, 64, 8192, 32), (1, 64, 8192, 128))[0]
    assert cut.startswith("scan_tph_kernel:") and "2 segments" in cut
    assert lines((1, 128, 4096, 128), (1, 128, 4096, 32))[0].startswith("scan_mfma_kernel")
    assert lines((1, 256, 4096, 128), (1, 256, 4096, 32))[0].startswith("scan_tp_kernel:")
    assert lines((1, 64, 512, 128), (1, 64, 512, 32))[0].startswith("scan_tp_kernel:")
    assert lines((1, 128, 4096, 64), (1, 128, 4096, 32))[0].startswith("scan_tph_kernel:")
    assert lines((1, 64, 2048, 64), (1, 64, 2048, 32))[0].startswith("scan_dma_kernel")
    assert lines((1, 16, 2048, 32), (1, 16, 2048, 96))[0].startswith("scan_tph_kernel:")
    # ... and long ones where whole chains fill three quarters of the CUs
    assert lines((1, 128, 16384, 32), (1, 128, 16384, 128))[0].startswith("scan_tph_kernel: 1 scan")
    # bf16 rows have a kernel of their own, widths that are not multiples of 4 go another way
    assert kernel(lines((8, 16, 4096, 128), (8, 16, 4096, 128), dtype=_native.FTC_BF16)[0]) == "scan_tp_bf16_kernel"
    assert lines((8, 16, 4096, 98), (8, 16, 4096, 128))[0].startswith("pad_rows_kernel")


SWEEP = [(N, H, L, E, M) for (N, H) in [(1, 1), (1, 16), (2, 8), (10, 8), (64, 16)]
         for L in [1, 64, 1000, 4096, 20000] for (E, M) in [(64, 64), (32, 128), (96, 64), (25, 70), (128, 128), (100, 36), (200, 64), (255, 129), (511, 300)]]


@pytest.mark.parametrize("backward", [False, True])
def test_the_workspace_query_covers_every_launch(backward):
    lib = _native.load()
    query = lib.ftc_causal_dot_backward_workspace_bytes if backward \
        else lib.ftc_causal_dot_product_workspace_bytes
    for dtype in (_native.FTC_F32, _native.FTC_BF16):
        for N, H, L, E, M in SWEEP:
            granted = query(N, H, L, E, M, dtype)
            assert granted >= 0
            for line in lines((N, H, L, E), (N, H, L, M), dtype=dtype, backward=backward):
                need = int(field(line, r"workspace (\d+) bytes")) if "workspace" in line else 0
                assert need <= granted, (N, H, L, E, M, dtype, line, granted)


@pytest.mark.parametrize("dtype", [_native.FTC_F32, _native.FTC_BF16], ids=["f32", "bf16"])
def test_workspace_queries_cover_every_plan(dtype):
    """Whatever route the planner takes, no launch of the plan needs more workspace than the
    query of its entry point answers: widths on either side of every limit of the planner (32,
    64, 128 rows; multiples of 4 and of 32 and neither), also bf16 rows whose two state shapes
    call for copies of different element types."""
    lib = _native.load()
    widths = [10, 25, 32, 33, 48, 64, 65, 96, 100, 128, 129, 132, 200, 255, 256, 300]
    worst = 0.0
    for (N, H, L) in [(10, 8, 2048), (2, 3, 700), (1, 2, 8192), (40, 16, 64)]:
        for E in widths:
            for M in widths:
                for backward in (False, True):
                    text = lines((N, H, L, E), (N, H, L, M), backward=backward, dtype=dtype)
                    need = max([int(x) for l in text for x in re.findall(r"workspace (\d+) bytes", l)]
                               or [0])
                    query = (lib.ftc_causal_dot_backward_workspace_bytes if backward else
                             lib.ftc_causal_dot_product_workspace_bytes)(N, H, L, E, M, dtype)
                    assert need <= query, ((N, H, L, E, M), backward, need, query, text)
                    if query:
                        worst = max(worst, need / query)
    assert worst > 0.5   # (the queries are not wildly generous either)


def test_rows_of_more_than_512_values_are_cut_into_pieces():
    """fp32 rows wider than 512: column slices of v and out, row parts of a and b whose results
    are added; every piece is planned like a scan of its own and the queries cover the lot."""
    lib = _native.load()
    fwd = lines((1, 2, 300, 600), (1, 2, 300, 520))
    # two row parts of 300 for each of two column slices of 288 and 232
    assert sum("state 128 x 288" in l for l in fwd) == 4 and sum("state 44 x 232" in l for l in fwd) == 2
    assert sum(l.startswith("add_rows_kernel: rows 300 ..") for l in fwd) == 2
    for (N, H, L, E, M) in [(1, 2, 300, 600, 520), (2, 2, 100, 513, 33), (1, 1, 64, 1100, 40),
                            (1, 2, 256, 64, 1030), (3, 4, 2048, 700, 900)]:
        for backward in (False, True):
            text = lines((N, H, L, E), (N, H, L, M), backward=backward)
            need = max(int(x) for l in text for x in re.findall(r"workspace (\d+) bytes", l))
            query = (lib.ftc_causal_dot_backward_workspace_bytes if backward else
                     lib.ftc_causal_dot_product_workspace_bytes)(N, H, L, E, M, _native.FTC_F32)
            assert 0 < need <= query, ((N, H, L, E, M), backward, need, query)
    # bf16 rows of that width: refused, by the queries as by the calls
    assert lib.ftc_causal_dot_product_workspace_bytes(1, 2, 300, 600, 520, _native.FTC_BF16) < 0
    assert b"fp32" in lib.ftc_last_error()


def test_odd_widths_lie_in_place_only_where_their_copies_run_on_the_same_kernel():
    """The padded shape's own plan names the kernel that the copies would run on."""
    up = lambda w: (w + 31) // 32 * 32
    seen = set()
    for N, H, L, E, M in [(1, 1, 100, 25, 33), (1, 1, 1356, 18, 18), (9, 11, 1531, 25, 33), (8, 16, 4096, 50, 50),
                          (2, 8, 333, 50, 50), (1, 3, 9000, 31, 62), (3, 5, 65, 63, 63), (64, 32, 100, 10, 9),
                          (1, 16, 24853, 63, 63), (24, 8, 1, 19, 41), (5, 32, 1, 60, 61)]:
        odd = lines((N, H, L, E), (N, H, L, M))
        aligned = lines((N, H, L, up(E)), (N, H, L, up(M)))
        in_place = odd[0].startswith("scan_tph_kernel")
        assert in_place == (aligned[0].startswith("scan_tph_kernel") and N * H * L >= 512)
        seen.add(in_place)
    assert seen == {False, True}
    # a backward call may have both
    mixed = lines((9, 11, 1531, 25, 33)[:4], (9, 11, 1531, 33), backward=True)
    assert mixed[0].startswith("scan_tph_kernel: 2 scans") and mixed[1].startswith("pad_rows_kernel: 3 operands")
    assert mixed[2].startswith("scan_dma_kernel: 1 scan")


def cut_chunks(line):
    return [int(x) for x in field(line, r"cuts at chunks ([\d,]*\d)").split(",")]


def test_cuts_on_three_pieces(monkeypatch):
    """fp32 rows in three bf16 pieces may start a segment at every second chunk, of chains of up to 64 chunks; bf16
    rows start at every fourth."""
    assert cut_chunks(lines((1, 24, 500, 100), (1, 24, 500, 100))[0]) == [0, 2, 10, 14, 16]
    assert cut_chunks(lines((1, 2, 295, 31), (1, 2, 295, 31))[0]) == [0, 2, 4, 8, 10]     # 32 rows, one position first
    assert cut_chunks(lines((1, 2, 745, 25), (1, 2, 745, 33))[0]) == [0, 10, 18, 22, 24]  # 64 rows
    long = lines((1, 60, 4000, 100), (1, 60, 4000, 100))[0]
    assert long.startswith("scan_tp_kernel: 1 scan") and cut_chunks(long) == [0, 84, 125]
    bf16 = lines((1, 40, 1000, 64), (1, 40, 1000, 64), dtype=_native.FTC_BF16)[0]
    assert bf16.startswith("scan_tp_bf16_kernel: 1 scan") and cut_chunks(bf16) == [0, 16, 24, 28, 32]
    # the fused attention's launches have the cuts of a single scan on that kernel, from three segments on
    # (tests/test_fused_attention_gpu.py runs these; FTC_TPH=0 keeps two fp16 pieces out)
    monkeypatch.setenv("FTC_TPH", "0")
    _native.load().ftc_tuning_reload()
    try:
        for (N, L, H, E, M), cuts in [((20, 300, 3, 64, 64), [0, 2, 6, 8, 10]), ((10, 1000, 6, 64, 64), [0, 10, 22, 28, 32]),
                                      ((25, 129, 2, 32, 64), [0, 2, 4, 5])]:
            line = lines((N, H, L, E), (N, H, L, M))[0]
            assert line.startswith("scan_tp_kernel: 1 scan") and cut_chunks(line) == cuts
    finally:
        monkeypatch.delenv("FTC_TPH")
        _native.load().ftc_tuning_reload()



@pytest.mark.parametrize("chunks", list(range(24, 60)) + [101, 193])
@pytest.mark.parametrize("heads", [3, 8])
def test_segments_of_few_chains_have_four_chunks(chunks, heads):
    """An exchange on few chains has a segment for every four chunks, the last one what is left, wherever that
    is at most 192 workgroups; its workspace is what the query answers."""
    L = 32 * chunks - 5
    line = lines((1, heads, L, 64), (1, heads, L, 64))[0]
    assert line.startswith("scan_tph_kernel (exchange): 1 scan")
    segments, rows = (int(field(line, p)) for p in (r"(\d+) segments of", r"segments of (\d+) rows"))
    fours = -(-chunks // 4)
    if heads * fours <= 192:
        assert (segments, rows) == (fours, 128)
    assert (segments - 1) * rows < L <= segments * rows
    need = int(field(line, r"workspace (\d+) bytes"))
    assert 0 < need <= _native.load().ftc_causal_dot_product_workspace_bytes(1, heads, L, 64, 64, 0)


def test_short_chains_of_wide_states_on_few_workgroups():
    """A single scan of more than 64 state rows: up to 10 chunks on any number of workgroups, from eight on up to 13, from
    twenty on up to where an exchange begins; bf16 rows up to 13, from twelve workgroups on any number."""
    def fwd(chains, chunks, E=128, M=128, dtype=_native.FTC_F32):
        s = (1, chains, 32 * chunks - 3)
        return kernel(lines(s + (E,), s + (M,), dtype=dtype)[0])
    tp, split = "scan_tp_kernel", "scan_mfma_kernel"
    for chains, chunks, E, M, want in [(1, 10, 128, 128, tp), (1, 11, 128, 128, split), (3, 13, 128, 128, split),
                                       (4, 13, 128, 128, tp), (7, 13, 128, 64, split), (8, 13, 128, 64, tp),
                                       (8, 14, 128, 128, split), (9, 23, 128, 128, split), (10, 14, 128, 128, tp),
                                       (10, 23, 96, 96, tp), (20, 23, 128, 64, tp), (8, 9, 128, 32, split)]:
        assert fwd(chains, chunks, E, M) == want, (chains, chunks, E, M)
    tp = "scan_tp_bf16_kernel"
    for chains, chunks, M, want in [(1, 13, 128, tp), (1, 14, 128, split), (5, 14, 128, split), (6, 27, 128, tp),
                                    (11, 27, 64, split), (12, 14, 64, tp)]:
        assert fwd(chains, chunks, 128, M, _native.FTC_BF16) == want, (chains, chunks, M)


@pytest.mark.parametrize("chains,L,route", [
    (64, 4128, "whole"), (85, 16384, "whole"), (85, 32768, "whole"), (180, 8192, "whole"), (20, 11000, "exchange"),
    (40, 6000, "exchange"), (18, 16384, "exchange"), (86, 16384, None), (32, 11000, None), (112, 8192, None),
    (64, 32800, None)])
def test_long_narrow_backward_scans_of_bf16_rows(chains, L, route):
    """32 x 32: by how full the rounds of workgroups are, or few enough chains for an exchange of sums."""
    got = lines((1, chains, L, 32), (1, chains, L, 32), backward=True, dtype=_native.FTC_BF16)[0]
    want = {"whole": "scan_tp_bf16_kernel", "exchange": "scan_tp_bf16_kernel (exchange)", None: "scan_mfma_kernel"}
    assert kernel(got) == want[route]


@pytest.mark.parametrize("chains,L,D,splits", [
    (95, 1600, 32, True), (96, 1600, 32, False), (127, 2600, 32, True), (128, 2600, 32, False), (159, 8192, 32, True),
    (160, 8192, 32, False), (160, 8224, 32, True), (79, 3300, 64, True), (80, 3300, 64, False), (47, 6000, 64, True),
    (48, 6000, 64, False), (47, 8224, 64, True), (48, 8224, 64, False), (23, 11000, 64, True), (24, 11000, 64, False)])
def test_long_forward_scans_of_bf16_rows_with_32_columns(chains, L, D, splits):
    got = lines((1, chains, L, D), (1, chains, L, 32), dtype=_native.FTC_BF16)[0]
    assert (kernel(got) == "scan_mfma_kernel") == splits
    assert splits or kernel(got).startswith("scan_tp_bf16_kernel")


@pytest.mark.parametrize("E,M,chains,L,most", [
    # (each call's time with segments of four chunks was 1.02 to 1.07 of that with eight)
    (64, 128, 14, 1100, 192), (64, 128, 4, 4000, 192), (48, 48, 28, 1100, 192), (25, 33, 28, 1100, 192),
    (27, 63, 8, 4000, 192), (32, 32, 8, 3778, 192)])
def test_small_states_do_not_exchange_on_too_many_workgroups(E, M, chains, L, most):
    """Rounding a chain's segments up to one for every four chunks stops where that were more workgroups than gain
    from it, for every state of up to 64 rows."""
    chunks = -(-L // 32)
    assert chunks % 4 and chains * -(-chunks // 4) * -(-M // 64) > most
    line = lines((1, chains, L, E), (1, chains, L, M))[0]
    assert "(exchange)" in line and int(field(line, r"segments of (\d+) rows")) == 256, line


@pytest.mark.parametrize("chains,L,E,M", [(8, 989, 75, 10), (9, 1681, 120, 31), (3, 5154, 75, 10), (4, 4000, 99, 101),
                                          (32, 989, 120, 31)])
def test_two_odd_shapes_stay_in_one_launch(chains, L, E, M):
    """The length of an exchange's segments does not decide whether scans of two odd shapes share a launch (two took 1.1
    to 1.3 times as long, or left dQ and dK 1.5 times as far from float64)."""
    got = lines((1, chains, L, E), (1, chains, L, M), backward=True)
    assert len(got) == 1 and kernel(got[0]).startswith("scan_tp_kernel") and "3 scans" in got[0], got


@pytest.mark.parametrize("chains,L", [(120, 8192), (124, 7000), (180, 5154), (186, 4128)])
def test_narrow_backward_scans_of_bf16_rows_split_where_the_rounds_are_not_full(chains, L):
    """Rounds of workgroups seven tenths full, which whole chains of this length take 1.02 to 1.05 times as long over."""
    got = lines((1, chains, L, 32), (1, chains, L, 32), backward=True, dtype=_native.FTC_BF16)
    assert kernel(got[0]) == "scan_mfma_kernel"


@pytest.mark.parametrize("chains,L,D", [(160, 2500, 32), (176, 3200, 32), (192, 3778, 32), (136, 3778, 64), (80, 6000, 64),
                                        (96, 9000, 64), (136, 8224, 64), (200, 9000, 64)])
def test_forward_scans_of_bf16_rows_with_32_columns_that_split(chains, L, D):
    """Where the rows fit the caches and a round of workgroups is not full, or an exchange leaves its rounds a quarter
    empty: 1.06 to 1.24 times as long on the chain-parallel kernel."""
    got = lines((1, chains, L, D), (1, chains, L, 32), dtype=_native.FTC_BF16)
    assert kernel(got[0]) == "scan_mfma_kernel"


@pytest.mark.parametrize("chains,L", [(8, 3140), (10, 2490), (12, 2360), (12, 2650)])
def test_fused_attention_exchanges_in_segments_of_four_chunks(chains, L):
    """Up to a whole round of workgroups (the limit of plain scans made them eight: 1.02 to 1.04 times as long as before
    those chains exchanged at all).  Two states of 128 x 16 values for each of the four consumers of every segment."""
    fours = -(-L // 128)
    assert 192 < chains * fours <= 256
    need = _native.load().ftc_causal_linear_attention_workspace_bytes(1, chains, L, 64, 64, 0)
    assert need >= 2 * 4 * chains * fours * 128 * 16 * 4


@pytest.mark.parametrize("chains,L,E,M,backward,dtype", [
    (1, 416, 128, 64, True, _native.FTC_BF16), (3, 380, 96, 64, True, _native.FTC_BF16),
    (7, 760, 128, 96, True, _native.FTC_BF16), (6, 860, 128, 96, True, _native.FTC_BF16),
    (10, 736, 128, 96, False, _native.FTC_F32)])
def test_short_chains_of_wide_states_that_split(chains, L, E, M, backward, dtype):
    """1.03 to 1.06 times as long walked whole."""
    got = lines((1, chains, L, E), (1, chains, L, M), backward=backward, dtype=dtype)
    assert kernel(got[-1]) == "scan_mfma_kernel", got
