"""The prefill kernels of cq_qtile.hip and cq_qtile0.hip where they can go wrong, against the CPU oracle.

Bound: the sums of 32 (Q4_0, Q8_0) and 256 elements are exact integers on both sides; what differs is f32 rounding of 1.5 - 2.5 operations per block and the
order of a split, nblocks <= 448 of them: below sqrt(448) * 3 * 2^-24 = 3.8e-6 of the terms' norm.  That norm is ||x|| ||w|| / sqrt(k), what a dot product
of such vectors has on average: a single result may cancel to far less, and its error does not with it.
"""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from candle_amd import _lib
from tests.util import normal, rel_l2

pytestmark = pytest.mark.gpu
BOUND = 4e-6
FMT = {"q4_0": (2, oracle.Q4_0), "q8_0": (8, oracle.Q8_0), "q4k": (12, oracle.Q4K), "q5k": (13, oracle.Q5K), "q6k": (14, oracle.Q6K)}
# shapes that the joint product, or one of two, would split or give narrower tiles
REFUSED_PAIRS = {("q6k", 129, 14338, 256), ("q6k", 225, 14337, 1792), ("q4k", 300, 14336, 2560)} | {(f, 97, 7169, 1536) for f in FMT}
REFUSED_APART = {(f, 400, 5632, 2048) for f in FMT}
OUT = {0: torch.float32, 1: torch.float16, 30: torch.bfloat16}


def run(code, blocks, x, n, out=0, shift=0, room=None):
    """cq_qmatmul_forward of x [m, k] with the weights `shift` bytes past a 256-byte boundary, the result between two rows of canaries.
    room: bytes of workspace, less than cq_qmatmul_workspace_bytes asks for, with canaries behind them."""
    L = _lib.lib()
    m, k = x.shape
    raw = torch.zeros(len(blocks) + 512, dtype=torch.uint8, device="cuda")
    raw[shift:shift + len(blocks)] = torch.from_numpy(blocks).cuda()
    xd = torch.from_numpy(x).cuda()
    y = torch.full((m + 2, n), 77.0, dtype=OUT[out], device="cuda")
    full = L.cq_qmatmul_workspace_bytes(code, m, k, n)
    nb = full if room is None else room
    ws = torch.full((full + 256,), 173, dtype=torch.uint8, device="cuda")
    rc = L.cq_qmatmul_forward(code, raw.data_ptr() + shift, ctypes.c_void_p(xd.data_ptr()), 0, ctypes.c_void_p(y[1].data_ptr()), out, m, k, n,
                              ctypes.c_void_p(ws.data_ptr()), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check("cq_qmatmul_forward", rc)
    torch.cuda.synchronize()
    assert (ws[nb:] == 173).all()
    y = y.float().cpu().numpy()
    assert (y[0] == 77).all() and (y[-1] == 77).all()
    return y[1:-1]


def row_error(got, want, x, w, k):
    """Largest error of a row [m, n] relative to the norm that rows x against the weights w have on average."""
    size = np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(w.astype(np.float64)) / np.sqrt(k)
    return float((np.linalg.norm(got.astype(np.float64) - want, axis=1) / size).max())


def check(fmt, m, n, k, out=0, shift=0, room=None):
    print(f"case {fmt} m={m} n={n} k={k} out={out} shift={shift}", flush=True)
    code, odt = FMT[fmt]
    w = normal(7 + m, (n, k), 0.02)
    blocks = oracle.from_float(odt, w.reshape(-1))
    x = normal(9 + n, (m, k))
    got, want = run(code, blocks, x, n, out, shift, room), oracle.matmul(odt, x, blocks, n)
    eps = {0: 0.0, 1: 2.0 ** -11, 30: 2.0 ** -8}[out]                # one rounding to the output type
    excess = np.maximum(np.abs(got - want) - eps * np.abs(want) - (2.0 ** -25 if out == 1 else 0), 0)        # (f16 results below 2^-14 are multiples of 2^-24)
    assert row_error(excess, 0, x, w, k) <= BOUND


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("m,n,k", [(66, 256, 256), (65, 1, 512), (97, 257, 768), (128, 31, 2304), (129, 260, 1280), (70, 292, 14336), (300, 510, 512), (65, 2, 1536), (97, 257, 2048), (129, 260, 1792),
                                   (300, 512, 1536)])
def test_tile_edges(fmt, m, n, k):
    # one row past a 32-row tile, one column past a workgroup's 256, one super-block, odd numbers of them, k split over workgroups and not;
    # Q6_K of less than 1536 of k or with an odd number of blocks (n k / 256 odd) takes the general kernel
    check(fmt, m, n, k)


@pytest.mark.parametrize("fmt", ["q4k", "q5k", "q6k"])
@pytest.mark.parametrize("m,n,k", [(33, 129, 1536), (64, 127, 1792), (140, 9002, 1536), (17, 33030, 1536), (300, 9002, 1536), (600, 9002, 1536), (800, 9002, 1536)])
def test_workgroups_of_four_and_eight_waves(fmt, m, n, k):
    """The shapes that qtile_plan gives workgroups of four waves with tiles of 32, 32 and 64 rows, then of eight with 32, 64 (Q4_K: of four), 96 and 128.
    Against 64 bits on the same rounded activations."""
    from perf import cases
    name = {"q4k": "q4_k", "q5k": "q5_k", "q6k": "q6_k"}[fmt]
    b = cases.blocks(name, 3, "w", n, k)
    w, x = cases.values(name, b, n, k), normal(9 + n, (m, k))
    want = cases.product(name, torch.from_numpy(x).cuda(), w).cpu().numpy()
    got = run(FMT[fmt][0], b.reshape(-1).cpu().numpy(), x, n)
    assert row_error(got, want, x, w.cpu().numpy(), k) <= BOUND


@pytest.mark.parametrize("fmt", ["q4k", "q5k", "q6k"])
@pytest.mark.parametrize("m,n,k", [(97, 14338, 256), (128, 14338, 512), (129, 14338, 768), (225, 14338, 2304), (417, 7170, 2560), (385, 9002, 1536)])
def test_wide_tiles(fmt, m, n, k):
    """Tiles of 96 and 128 rows, the last one with one to four 32-row tiles of rows; one, two, three and more super-blocks (the rings hold two to four), odd numbers of
    them (Q6_K rows then begin on 2 bytes; below 1536 of k it takes the general kernel), columns that end inside a wave's 32.  Against 64 bits, bound as above."""
    from perf import cases
    name = {"q4k": "q4_k", "q5k": "q5_k", "q6k": "q6_k"}[fmt]
    print(f"case {fmt} m={m} n={n} k={k}", flush=True)
    b = cases.blocks(name, 4, "w", n, k)
    w, x = cases.values(name, b, n, k), normal(11 + n, (m, k))
    got = run(FMT[fmt][0], b.reshape(-1).cpu().numpy(), x, n)
    assert row_error(got, cases.product(name, torch.from_numpy(x).cuda(), w).cpu().numpy(), x, w.cpu().numpy(), k) <= BOUND


@pytest.mark.parametrize("fmt", ["q4k", "q5k", "q6k"])
@pytest.mark.parametrize("gap", [0, 16])
@pytest.mark.parametrize("m,n,k", [(97, 7169, 1536), (129, 14338, 256), (225, 14337, 1792), (300, 14336, 2560), (400, 5632, 2048)])
def test_silu_of_a_pair(fmt, gap, m, n, k):
    """cq_nn_qmatmul_swiglu_pair, the second weight right behind the first or not: bit for bit what the products and cq_nn_silu_mul give, canaries around it; rows and
    columns that end inside a tile and one whose last tiles have no rows.  Whatever the shape, it is taken whole or refused."""
    L = _lib.lib()
    print(f"case {fmt} gap={gap} m={m} n={n} k={k}", flush=True)
    from perf import cases
    code, name = FMT[fmt][0], {"q4k": "q4_k", "q5k": "q5_k", "q6k": "q6_k"}[fmt]
    w = cases.blocks(name, 6, "w", 2 * n, k).reshape(-1)
    nb = w.numel() // 2
    raw = torch.zeros(2 * nb + gap, dtype=torch.uint8, device="cuda")
    raw[:nb], raw[nb + gap:] = w[:nb], w[nb:]
    x = torch.from_numpy(normal(12 + n, (m, k))).cuda()
    st = torch.cuda.current_stream().cuda_stream
    wsb = L.cq_qmatmul_workspace_bytes(code, m, k, 2 * n)
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    y = torch.full((m + 2, n), 77.0, device="cuda")
    args = (code, raw.data_ptr(), raw.data_ptr() + nb + gap, x.data_ptr(), y[1].data_ptr(), m, k, n, ws.data_ptr())
    rc = L.cq_nn_qmatmul_swiglu_pair(*args, wsb, st)
    taken = rc == 0
    assert taken or rc == -6
    assert taken == ((fmt, m, n, k) not in REFUSED_PAIRS and (gap == 0 or (fmt, m, n, k) not in REFUSED_APART))
    assert L.cq_nn_qmatmul_swiglu_pair(*args, 256, st) == -5
    torch.cuda.synchronize()
    if not taken:
        assert (y == 77.0).all()
        return
    assert (y[0] == 77.0).all() and (y[m + 1] == 77.0).all()
    want = torch.empty((m, n), device="cuda")
    gate, up = torch.empty((m, n), device="cuda"), torch.empty((m, n), device="cuda")
    for at, to in ((0, gate), (nb + gap, up)):
        _lib.check("cq_qmatmul_forward", L.cq_qmatmul_forward(code, raw.data_ptr() + at, x.data_ptr(), 0, to.data_ptr(), 0, m, k, n, ws.data_ptr(), wsb, st))
    if gap == 0:                                           # (as one product of 2 n rows, which is not split where those of n may be)
        both = torch.empty((m, 2 * n), device="cuda")
        _lib.check("cq_qmatmul_forward", L.cq_qmatmul_forward(code, raw.data_ptr(), x.data_ptr(), 0, both.data_ptr(), 0, m, k, 2 * n, ws.data_ptr(), wsb, st))
        gate, up = both[:, :n].contiguous(), both[:, n:].contiguous()
    pad = (-n) % 4                                         # (cq_nn_silu_mul takes four elements at a time)
    gate, up = (torch.nn.functional.pad(t, (0, pad)).contiguous() for t in (gate, up))
    want = torch.empty_like(gate)
    _lib.check("cq_nn_silu_mul", L.cq_nn_silu_mul(gate.data_ptr(), up.data_ptr(), want.data_ptr(), m, n + pad, n + pad, n + pad, st))
    torch.cuda.synchronize()
    assert torch.equal(y[1:m + 1], want[:, :n])


@pytest.mark.parametrize("out", [0, 1])
@pytest.mark.parametrize("m,n,k", [(129, 5632, 2048), (150, 5633, 2304), (290, 3585, 4096), (300, 7681, 2048), (449, 4609, 2048)])
def test_tiles_of_160_rows(m, n, k, out):
    """Q4_0 in tiles of five parts of 32 rows, the last one with one to five of them; ragged columns, K split and not."""
    check("q4_0", m, n, k, out)


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("out", [1, 30])
@pytest.mark.parametrize("n,k", [(130, 512), (260, 4096)])
def test_half_results(fmt, out, n, k):
    check(fmt, 67, n, k, out)                              # written by the product itself, and by the sum over the splits


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("out", [0, 1, 30])
@pytest.mark.parametrize("m,n,k", [(33, 131, 512), (101, 70, 768), (70, 291, 2304)])
def test_rows_of_results_off_four_columns(fmt, out, m, n, k):
    check(fmt, m, n, k, out)                               # four columns at a time on any element, the last one to three alone


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("out", [0, 1, 30])
@pytest.mark.parametrize("m,n,k", [(17, 1, 4096), (70, 291, 9984), (33, 1026, 2304), (131, 515, 14336)])
def test_split_sums_of_any_number_of_columns(fmt, out, m, n, k):
    """Planes have rows of whole fours of columns, the result has not: nothing behind a row's last column is read or written."""
    L = _lib.lib()
    assert L.cq_qmatmul_workspace_bytes(FMT[fmt][0], m, k, n) > L.cq_act_scratch_bytes(FMT[fmt][0], k, m) + 4 * m * n
    check(fmt, m, n, k, out)


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("out", [0, 1])
@pytest.mark.parametrize("m,n,k,splits", [(67, 260, 1536, 1), (67, 260, 4096, 4)])
def test_least_workspace(fmt, out, m, n, k, splits):
    """The quantized rows, one plane of results and the general kernels' `splits` of them: enough for a call, with canaries right behind; less is refused."""
    L = _lib.lib()
    code = FMT[fmt][0]
    up = lambda b: (b + 255) // 256 * 256
    least = L.cq_act_scratch_bytes(code, k, m) + up(4 * m * n) + (up(4 * splits * m * n) if splits > 1 else 0)
    assert least < L.cq_qmatmul_workspace_bytes(code, m, k, n)
    p = ctypes.c_void_p(4096)                              # (refused before anything is read)
    assert L.cq_qmatmul_forward(code, p, p, 0, p, out, m, k, n, p, least - 1, None) == -5      # CQ_ERR_WORKSPACE
    check(fmt, m, n, k, out, room=least)


@pytest.mark.parametrize("fmt,shift", [("q4_0", 2), ("q4_0", 8), ("q8_0", 6), ("q8_0", 16), ("q6k", 2), ("q6k", 4), ("q4k", 16), ("q5k", 48)])
def test_weights_at_other_addresses(fmt, shift):
    check(fmt, 66, 96, 1792, shift=shift)                   # Q4_0 / Q8_0 off 16 bytes, Q6_K off 4: the general kernels


@pytest.mark.parametrize("fmt,bb", [("q4_0", 18), ("q8_0", 34)])
@pytest.mark.parametrize("d", [np.inf, -np.inf, np.nan, 65504.0, 6e-8])
def test_extreme_block_scales(fmt, bb, d):
    """The scale of one block infinite, NaN, the largest and the smallest: the same values, infinities and NaN as the oracle's sums."""
    code, odt = FMT[fmt]
    n, k, m = 96, 512, 70
    blocks = oracle.from_float(odt, normal(3, (n, k), 0.02).reshape(-1)).reshape(n, k // 32, bb)
    blocks[[0, 40, 95], [0, 7, 15], :2] = np.frombuffer(np.float16(d).tobytes(), dtype=np.uint8)
    x = normal(4, (m, k))
    x[5, :32] = 0.0                                        # a sum of zero times an infinite scale
    want = oracle.matmul(odt, x, blocks.reshape(-1), n)
    got = run(code, blocks.reshape(-1), x, n)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)])
    assert rel_l2(got[ok], want[ok]) <= BOUND


@pytest.mark.parametrize("fmt,bb,at", [("q4k", 144, 0), ("q4k", 144, 2), ("q5k", 176, 0), ("q5k", 176, 2), ("q6k", 210, 208)])
@pytest.mark.parametrize("d", [np.inf, -np.inf, np.nan, 65504.0, 6e-8])
def test_extreme_super_block_scales(fmt, bb, at, d):
    """d or dmin of a super-block: results that are not finite where the oracle's are not.  Its eight partial sums may make NaN of an infinity, never the reverse."""
    code, odt = FMT[fmt]
    n, k, m = 96, 1536, 70
    blocks = oracle.from_float(odt, normal(3, (n, k), 0.02).reshape(-1)).reshape(n, k // 256, bb)
    blocks[[0, 40, 95], [0, 3, 5], at:at + 2] = np.frombuffer(np.float16(d).tobytes(), dtype=np.uint8)
    x = normal(4, (m, k))
    x[5, :256] = 0.0                                       # sums of zero times an infinite scale
    want = oracle.matmul(odt, x, blocks.reshape(-1), n)
    got = run(code, blocks.reshape(-1), x, n)
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), ok)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and (not np.isnan(d) or np.isnan(got[~ok]).all())
    assert rel_l2(got[ok], want[ok]) <= BOUND


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0", "q6k", "q5k"])
@pytest.mark.parametrize("tokens", [70, 1200])
@pytest.mark.parametrize("E,n", [(5, 268), (4, 267), (3, 1028)])
def test_grouped_experts(fmt, tokens, E, n):
    """A few experts with tiles of 32 and of 128 rows, the last ones part full, columns past the last workgroup's; Q6_K: an odd number of blocks a row, and of
    rows too: every second expert begins 2 bytes past a dword; Q4_0: 32-row tiles of up to 1024 columns are the general kernel's."""
    import candle_amd as ca
    code, odt = FMT[fmt]
    k, topk = 1792, 2
    w = normal(21, (E, n, k), 0.02)
    blocks = oracle.from_float(odt, w.reshape(-1))
    qt = ca.QTensor.new(ca.QStorage.from_data(blocks, "cuda", ca.GgmlDType(odt)), (E, n, k))
    x = normal(22, (tokens, 1, k))
    ids = np.random.default_rng(5).integers(0, E, (tokens, topk)).astype(np.uint32)
    ids[: tokens // 2, 0] = 3
    got = qt.indexed_moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids.astype(np.int32)).cuda()).cpu().numpy()
    per = len(blocks) // E
    for e in range(E):
        t, s = np.nonzero(ids == e)
        want = oracle.matmul(odt, x[t, 0], blocks[e * per:(e + 1) * per], n)
        assert row_error(got[t, s], want, x[t, 0], w[e], k) <= BOUND


@pytest.mark.parametrize("fmt,m,n,k,splits", [("q8_0", 131, 8192, 2304, 2), ("q4_0", 777, 2048, 2048, 2), ("q8_0", 131, 11008, 4096, 2), ("q6k", 24, 256, 4096, 4), ("q6k", 65, 1024, 4096, 4),
                                              ("q6k", 300, 512, 2048, 2)])
def test_split_sums_round_no_more_than_the_general_kernels(fmt, m, n, k, splits):
    """Against 64 bits: however K is split, f32 sums may round no more than in the general kernels' `splits` chains, added one after the other.

    An f32 rounding has an rms of 0.425 * 2^-24 of its value (half an ulp, uniform, over mantissas of 1 to 2).  A chain of c terms rounds partial sums of 1 .. c
    terms, the sum of the chains those of all terms so far, and each term itself rounds once or twice before it is added (1.5 units); 5 % for the rest.
    """
    from perf import cases
    name = {"q4k": "q4_k", "q5k": "q5_k", "q6k": "q6_k"}.get(fmt, fmt)
    b = cases.blocks(name, 3, "w", n, k)
    x = normal(9 + n, (m, k))
    want = cases.product(name, torch.from_numpy(x).cuda(), cases.values(name, b, n, k)).cpu().numpy()
    got = run(FMT[fmt][0], b.reshape(-1).cpu().numpy(), x, n)
    terms, nsb = (8 if fmt in ("q4_0", "q8_0") else 1), k // 256
    ends = [nsb * z // splits * terms for z in range(splits + 1)]
    total = ends[-1]
    variance = sum((e - s) * (e - s + 1) / 2 for s, e in zip(ends, ends[1:])) + sum(ends[2:]) + 1.5 * total
    assert rel_l2(got, want) <= 1.05 * 0.425 * 2.0 ** -24 * np.sqrt(variance / total)


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("rows,n,k", [(9, 31, 1536), (17, 260, 4096), (33, 520, 512), (67, 257, 2304), (131, 260, 1280)])
def test_matmul_of_quantized_rows(fmt, rows, n, k):
    """cq_matmul, which has no planes to split k with, into rows of a larger stride: nothing between them is written."""
    L = _lib.lib()
    code, odt = FMT[fmt]
    w = normal(31, (n, k), 0.02)
    blocks = oracle.from_float(odt, w.reshape(-1))
    x = normal(32, (rows, k))
    wd, xd = torch.from_numpy(blocks).cuda(), torch.from_numpy(x).cuda()
    scratch = torch.empty(L.cq_act_scratch_bytes(code, k, rows), dtype=torch.uint8, device="cuda")
    y = torch.full((rows, n + 3), 77.0, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    _lib.check("cq_quantize_act", L.cq_quantize_act(code, xd.data_ptr(), 0, scratch.data_ptr(), k, rows, s))
    _lib.check("cq_matmul", L.cq_matmul(code, wd.data_ptr(), scratch.data_ptr(), y.data_ptr(), k, n, rows, n + 3, s))
    y = y.cpu().numpy()
    assert (y[:, n:] == 77).all()
    assert row_error(y[:, :n], oracle.matmul(odt, x, blocks, n), x, w, k) <= BOUND


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("n,k", [(8197, 256), (8197, 2304), (16385, 3072)])
def test_few_rows_keep_the_bits_of_many(fmt, n, k):
    """Unsplit, a result is one chain of blocks: rows in a tile of 32 (whichever operand comes first there, which the size of the weights decides for Q8_0) have the bits they
    have among 2000, in tiles of 128."""
    from perf import cases
    L = _lib.lib()
    code = FMT[fmt][0]
    w = cases.blocks(fmt, 8, "w", n, k).reshape(-1)
    x = torch.from_numpy(normal(33 + n, (2000, k))).cuda()
    s = torch.cuda.current_stream().cuda_stream

    def product(rows):
        scratch = torch.empty(L.cq_act_scratch_bytes(code, k, rows), dtype=torch.uint8, device="cuda")
        y = torch.full((rows + 1, n), 77.0, device="cuda")
        _lib.check("cq_quantize_act", L.cq_quantize_act(code, x.data_ptr(), 0, scratch.data_ptr(), k, rows, s))
        _lib.check("cq_matmul", L.cq_matmul(code, w.data_ptr(), scratch.data_ptr(), y.data_ptr(), k, n, rows, n, s))
        assert bool((y[rows] == 77).all())
        return y[:rows]

    many = product(2000)
    for rows in (9, 31, 32):
        print(f"case {fmt} rows={rows} n={n} k={k}", flush=True)
        assert torch.equal(product(rows), many[:rows])


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("E,n,pairs", [(16, 2052, 528), (16, 4100, 528), (16, 8196, 530), (40, 2052, 1200), (64, 2048, 1600), (33, 4097, 513)])
def test_grouped_tiles_of_32_rows_keep_bits(fmt, E, n, pairs):
    """Experts on either side of the limits between the two orders of operands (Q4_0): the bits of each expert's own product, which no other rows change."""
    import candle_amd as ca
    from perf import cases
    L = _lib.lib()
    code, k = FMT[fmt][0], 512
    print(f"case {fmt} E={E} n={n} pairs={pairs}", flush=True)
    b = cases.blocks(fmt, 9, "w", E * n, k).reshape(-1)
    qt = ca.QTensor.new(ca.QStorage.from_data(b.cpu().numpy(), "cuda", ca.GgmlDType(FMT[fmt][1])), (E, n, k))
    x = torch.from_numpy(normal(34, (pairs, 1, k))).cuda()
    ids = torch.arange(pairs, dtype=torch.int32, device="cuda").reshape(-1, 1) % E
    got = qt.indexed_moe_forward(x, ids)[:, 0]
    per, s = b.numel() // E, torch.cuda.current_stream().cuda_stream
    for e in (0, 1, E // 2, E - 1):
        rows = x[e::E, 0].contiguous()
        scratch = torch.empty(L.cq_act_scratch_bytes(code, k, len(rows)), dtype=torch.uint8, device="cuda")
        y = torch.empty((len(rows), n), device="cuda")
        _lib.check("cq_quantize_act", L.cq_quantize_act(code, rows.data_ptr(), 0, scratch.data_ptr(), k, len(rows), s))
        _lib.check("cq_matmul", L.cq_matmul(code, b.data_ptr() + e * per, scratch.data_ptr(), y.data_ptr(), k, n, len(rows), n, s))
        assert torch.equal(got[e::E], y), e


@pytest.mark.parametrize("fmt,bb", [("q4_0", 18), ("q8_0", 34)])
@pytest.mark.parametrize("d", [np.inf, np.nan, 65504.0])
def test_extreme_block_scales_of_few_rows(fmt, bb, d):
    """As test_extreme_block_scales, in one tile of 32 rows."""
    code, odt = FMT[fmt]
    n, k, m = 99, 512, 21
    blocks = oracle.from_float(odt, normal(3, (n, k), 0.02).reshape(-1)).reshape(n, k // 32, bb)
    blocks[[0, 40, 98], [0, 7, 15], :2] = np.frombuffer(np.float16(d).tobytes(), dtype=np.uint8)
    x = normal(4, (m, k))
    x[5, :32] = 0.0
    want = oracle.matmul(odt, x, blocks.reshape(-1), n)
    got = run(code, blocks.reshape(-1), x, n)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)])
    assert rel_l2(got[ok], want[ok]) <= BOUND


@pytest.mark.parametrize("out", [0, 1, 30])
@pytest.mark.parametrize("m,n,k", [(666, 11818, 1024), (523, 14363, 1024), (725, 10915, 1024), (577, 13370, 1024), (770, 10073, 1024), (963, 2872, 2304), (1156, 2316, 2304), (390, 1320, 10496),
                                   (261, 7728, 2816), (130, 5572, 2816)])
def test_every_last_tile_of_160_rows(m, n, k, out):
    """Q4_0 in tiles of five parts of 32 rows, the last one with one to five of them; ragged columns, K not split (the first five) and split.  Against 64 bits, bound as above, and one
    rounding to the type of the results."""
    from perf import cases
    print(f"case m={m} n={n} k={k} out={out}", flush=True)
    b = cases.blocks("q4_0", 4, "w", n, k)
    w, x = cases.values("q4_0", b, n, k), normal(11 + n, (m, k))
    want = cases.product("q4_0", torch.from_numpy(x).cuda(), w).cpu().numpy()
    excess = np.maximum(np.abs(run(2, b.reshape(-1).cpu().numpy(), x, n, out) - want) - {0: 0.0, 1: 2.0 ** -11, 30: 2.0 ** -8}[out] * np.abs(want) - (2.0 ** -25 if out == 1 else 0), 0)
    assert row_error(excess, 0, x, w.cpu().numpy(), k) <= BOUND


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("E,n,pairs", [(16, 8196, 448), (33, 2052, 513), (40, 4100, 600), (64, 2048, 1100)])
def test_more_grouped_tiles_of_32_rows_keep_bits(fmt, E, n, pairs):
    """Fewer pairs an expert: the activations first in the first three (Q4_0; 726, 297 and 680 expected workgroups)."""
    test_grouped_tiles_of_32_rows_keep_bits(fmt, E, n, pairs)


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0"])
def test_every_last_tile_keeps_the_bits(fmt):
    """Tiles of 32 to 128 rows (Q4_0: 160), the last one with each number of parts of 32 rows: one chain of blocks a result, so the bits of the rows among 2000; and those against 64 bits."""
    from perf import cases
    L = _lib.lib()
    code, n, k = FMT[fmt][0], 16384, 768
    w = cases.blocks(fmt, 8, "w", n, k).reshape(-1)
    x = torch.from_numpy(normal(36, (2000, k))).cuda()
    s = torch.cuda.current_stream().cuda_stream

    def product(rows):
        print(f"case {fmt} rows={rows}", flush=True)
        scratch = torch.empty(L.cq_act_scratch_bytes(code, k, rows), dtype=torch.uint8, device="cuda")
        y = torch.full((rows + 1, n), 77.0, device="cuda")
        _lib.check("cq_quantize_act", L.cq_quantize_act(code, x.data_ptr(), 0, scratch.data_ptr(), k, rows, s))
        _lib.check("cq_matmul", L.cq_matmul(code, w.data_ptr(), scratch.data_ptr(), y.data_ptr(), k, n, rows, n, s))
        assert bool((y[rows] == 77).all())
        return y[:rows]

    many = product(2000)
    values = cases.values(fmt, w.reshape(-1, cases.BLOCK_BYTES[fmt][1]), n, k)
    assert row_error(many.cpu().numpy(), cases.product(fmt, x, values).cpu().numpy(), x.cpu().numpy(), values.cpu().numpy(), k) <= BOUND
    for rows in (33, 64, 129, 160, 161, 193, 257, 288, 289, 321, 352, 385, 417, 449, 481, 512, 513, 545, 577, 609):
        assert torch.equal(product(rows), many[:rows]), rows
