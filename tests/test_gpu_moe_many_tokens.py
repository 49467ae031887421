"""Expert layers of thousands of tokens: the router's eight-by-eight form and the grouping kernel beyond the pairs that its threads keep."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from candle_amd import _lib
from tests.util import normal, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,experts,hidden", [(1027, 64, 516), (513, 128, 2048), (700, 100, 260), (8200, 8, 64), (1407, 64, 516), (1409, 64, 516), (1001, 100, 260), (12300, 8, 64), (511, 128, 2048)])
def test_router_logits(tokens, experts, hidden):
    """Against float64.  hidden products summed lane by lane (hidden / 64 in a row) and over 64 lanes: below 2^-24 * (hidden / 64 + 6) of the terms' sum."""
    print(f"case {tokens} {experts} {hidden}", flush=True)
    x, w = normal(1, (tokens, hidden)), normal(2, (experts, hidden))
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    ids = torch.empty((tokens, 2), dtype=torch.int32, device="cuda")
    tw = torch.empty((tokens, 2), device="cuda")
    logits = torch.full((tokens + 1, experts), 9.0, device="cuda")
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    _lib.check("cq_nn_moe_route", _lib.lib().cq_nn_moe_route(vp(xd), vp(wd), vp(ids), vp(tw), vp(logits), tokens, hidden, experts, 2, 1,
                                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    got = logits.cpu().numpy()
    x, w = x.astype(np.float64), w.astype(np.float64)
    assert (np.abs(got[:tokens] - x @ w.T) <= 2.0 ** -24 * (hidden / 64 + 6 + 1) * (np.abs(x) @ np.abs(w).T)).all()
    assert (got[tokens] == 9).all()


@pytest.mark.parametrize("tokens", [2049, 6144, 6150, 9000])            # two pairs a token: 12288 stay in registers
def test_grouping_many_pairs(tokens):
    import candle_amd as ca
    E, n, k = 7, 20, 256
    blocks = oracle.from_float(oracle.Q8_0, normal(5, (E, n, k), 0.02).reshape(-1))
    qt = ca.QTensor.new(ca.QStorage.from_data(blocks, "cuda", ca.GgmlDType(oracle.Q8_0)), (E, n, k))
    x = normal(6, (tokens, 1, k))
    ids = np.random.default_rng(tokens).integers(0, E + 1, (tokens, 2)).astype(np.int32)      # E: no such expert, a row of zeros
    got = qt.indexed_moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()).cpu().numpy()
    per = len(blocks) // E
    for e in range(E):
        t, s = np.nonzero(ids == e)
        assert rel_l2(got[t, s], oracle.matmul(oracle.Q8_0, x[t, 0], blocks[e * per:(e + 1) * per], n)) <= 2e-6
    assert (got[ids == E] == 0).all()


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("tokens", [140, 3072, 3073])                   # two pairs a token: up to 6144 are decoded pair by pair, more by loads asked for together
def test_grouping_at_the_change_of_form(tokens, weights):
    import candle_amd as ca
    E, n, k, top = 7, 20, 256, 2
    blocks = oracle.from_float(oracle.Q8_0, normal(5, (E, n, k), 0.02).reshape(-1))
    qt = ca.QTensor.new(ca.QStorage.from_data(blocks, "cuda", ca.GgmlDType(oracle.Q8_0)), (E, n, k))
    pairs = tokens * top
    rng = np.random.default_rng(pairs)
    experts, order = rng.integers(0, E, pairs).astype(np.int32), rng.permutation(pairs).astype(np.int32)
    x = normal(6, (pairs if weights else tokens, k))
    tw = rng.uniform(0.1, 1, pairs).astype(np.float32) if weights else None
    cuda = lambda a: torch.from_numpy(a).cuda()
    got = ca.moe_gemm_gguf(cuda(x), qt, cuda(tw) if weights else None, cuda(order), cuda(experts), top, True).cpu().numpy()
    assert rel_l2(got, oracle.moe_gemm_gguf(oracle.Q8_0, x, blocks, (E, n, k), order, experts, tw, top)) <= 2e-6
    ids = rng.integers(0, E + 1, (tokens, top)).astype(np.int32)        # E: no such expert, a row of zeros
    x = normal(7, (tokens, k))
    got = qt.indexed_moe_forward(cuda(x[:, None]), cuda(ids)).cpu().numpy()
    for e in range(E):
        t, s = np.nonzero(ids == e)
        assert rel_l2(got[t, s], oracle.matmul(oracle.Q8_0, x[t], blocks[e * len(blocks) // E:(e + 1) * len(blocks) // E], n)) <= 2e-6
    assert (got[ids == E] == 0).all()


@pytest.mark.parametrize("dtype", [oracle.Q8_0, oracle.Q6K])
@pytest.mark.parametrize("E,tokens,top,order", [(3, 2048, 3, "tokens"), (3, 2049, 3, "shuffled"), (1024, 700, 2, "tokens"), (1025, 700, 2, "tokens"), (1, 300, 2, "shuffled"),
                                                (70, 30, 65, "tokens"), (9, 1025, 6, "twice")])
def test_grouping_of_lists(dtype, E, tokens, top, order):
    """Lists of pairs at the edges of what a thread takes at a time (6144 pairs), of hundreds of experts and of a wave's 64 pairs, in token order
    (a row is quantized once for its pairs), shuffled, and with every entry of the first half listed again in place of one of the second: valid pairs get their
    product, and pairs that name no expert or no token write nothing."""
    import candle_amd as ca
    n, k = 12, 256
    blocks = oracle.from_float(dtype, normal(5, (E, n, k), 0.02).reshape(-1))
    qt = ca.QTensor.new(ca.QStorage.from_data(blocks, "cuda", ca.GgmlDType(dtype)), (E, n, k))
    pairs, rng = tokens * top, np.random.default_rng(tokens)
    experts, order_of = rng.integers(0, E, pairs).astype(np.int32), np.arange(pairs, dtype=np.int32)
    if order == "shuffled":
        order_of = rng.permutation(pairs).astype(np.int32)
    if order == "twice":
        half = pairs // 2
        order_of[half:2 * half], experts[half:2 * half] = order_of[:half], experts[:half]
    bad = rng.choice(pairs // 2, 9, replace=False)
    if order != "twice":
        experts[bad[:3]], experts[bad[3:5]] = -1, E
        order_of[bad[5:7]], order_of[bad[7:]] = -1, pairs
    x, L = normal(6, (tokens, k)), _lib.lib()
    cuda = lambda a: torch.from_numpy(a).cuda()
    xd, od, ed = cuda(x), cuda(order_of), cuda(experts)
    out = torch.full((pairs, n), 7.0, device="cuda")
    ws = torch.full((L.cq_moe_gemm_workspace_bytes(int(dtype), E, top, pairs, n, k, 0),), 255, dtype=torch.uint8, device="cuda")
    _lib.check("cq_moe_gemm_gguf", L.cq_moe_gemm_gguf(int(dtype), xd.data_ptr(), qt.device_ptr(), od.data_ptr(), ed.data_ptr(), None, out.data_ptr(), E, top, pairs, n, k, 1,
                                                      ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    got, want = out.cpu().numpy(), np.full((pairs, n), 7.0, np.float32)
    valid = (experts >= 0) & (experts < E) & (order_of >= 0) & (order_of < pairs)
    per = len(blocks) // E
    for e in range(E):
        rows = order_of[valid & (experts == e)]
        if len(rows):
            want[rows] = oracle.matmul(dtype, x[rows // top], blocks[e * per:(e + 1) * per], n)
    hit = np.zeros(pairs, bool)
    hit[order_of[valid]] = True
    assert rel_l2(got[hit], want[hit]) <= 2e-6 and (got[~hit] == 7.0).all() and (~hit).any()


@pytest.mark.parametrize("dtype", [oracle.Q8_0, oracle.Q6K])
@pytest.mark.parametrize("E,tokens,top", [(5, 128, 16), (5, 129, 16), (40, 160, 17), (40, 200, 20), (512, 700, 3), (513, 1365, 3), (513, 1366, 3), (1024, 600, 8), (1025, 800, 8)])
def test_grouping_of_lists_in_any_order(dtype, E, tokens, top):
    """A list in token order, sorted by expert and shuffled gives the same bits: on either side of the numbers of pairs and experts at which another kernel groups or
    quantizes them, with groups of pairs that hold parts of two tokens, and with experts that have no pair."""
    import candle_amd as ca
    n, k, pairs = 12, 512, tokens * top
    blocks = oracle.from_float(dtype, normal(5, (E, n, k), 0.02).reshape(-1))
    qt = ca.QTensor.new(ca.QStorage.from_data(blocks, "cuda", ca.GgmlDType(dtype)), (E, n, k))
    rng = np.random.default_rng(tokens)
    experts = rng.integers(0, E, pairs).astype(np.int32)
    experts[rng.choice(pairs, 5, replace=False)] = -1
    x, L = normal(6, (tokens, k)), _lib.lib()
    cuda = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    xd, got = cuda(x), []
    ws = torch.full((L.cq_moe_gemm_workspace_bytes(int(dtype), E, top, pairs, n, k, 0),), 255, dtype=torch.uint8, device="cuda")
    for order in (np.arange(pairs), np.argsort(experts, kind="stable"), rng.permutation(pairs)):
        ed, od, out = cuda(experts[order]), cuda(order.astype(np.int32)), torch.full((pairs, n), 7.0, device="cuda")
        _lib.check("cq_moe_gemm_gguf", L.cq_moe_gemm_gguf(int(dtype), xd.data_ptr(), qt.device_ptr(), od.data_ptr(), ed.data_ptr(), None, out.data_ptr(), E, top, pairs, n, k, 1,
                                                          ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        got.append(out.cpu().numpy())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    want, per = np.full((pairs, n), 7.0, np.float32), len(blocks) // E
    for e in range(E):
        p = np.flatnonzero(experts == e)
        if len(p):
            want[p] = oracle.matmul(dtype, x[p // top], blocks[e * per:(e + 1) * per], n)
    assert rel_l2(got[0], want) <= 2e-6 and (got[0][experts < 0] == 7.0).all()
