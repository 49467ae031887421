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
