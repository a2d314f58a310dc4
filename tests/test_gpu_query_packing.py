"""Queries packed row after row into a wave's tiles (16-bit in-batch and multi-query
packed scans), or all queries' tokens cut into tiles (split-K in-batch), against the same queries padded with masked tokens to whole tiles, which
takes the kernel with a query per tile: the sums run in the same order, so scores and
tapes are equal bit for bit.  Lengths at both ends of each count of queries per wave,
query counts that leave a wave or a block part filled, documents without a valid token,
documents that share a chunk, and Inf / NaN tokens."""
import ctypes

import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import _lib

pytestmark = pytest.mark.gpu


def _padded(Q, qm):
    B, Tq, dim = Q.shape
    T = (Tq + 31) // 32 * 32
    Qp = torch.zeros(B, T, dim, dtype=Q.dtype, device=Q.device)
    mp = torch.zeros(B, T, dtype=torch.bool, device=Q.device)
    Qp[:, :Tq] = Q
    mp[:, :Tq] = True if qm is None else qm
    return Qp, mp


def _same(x, y):
    return torch.equal(torch.nan_to_num(x, nan=12345.0), torch.nan_to_num(y, nan=12345.0))


def _check(forward, Q, D, qm, *masks):
    Qp, mp = _padded(Q, qm)
    for norm in (False, True):
        S, a = forward(Q, D, qm, *masks, normalize=norm)
        Sp, ap = forward(Qp, D, mp, *masks, normalize=norm)
        assert _same(S, Sp) and torch.equal(a, ap[..., :Q.shape[1]])
        S0, _ = forward(Q, D, qm, *masks, normalize=norm, tape=False)
        assert _same(S, S0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [32, 64, 96, 128])
@pytest.mark.parametrize("Tq", [1, 8, 9, 15, 16, 17, 18, 19, 21, 22, 23, 25, 33, 42])
def test_packed_queries_match_a_query_per_tile(device, dtype, dim, Tq):
    g = torch.Generator(device=device).manual_seed(Tq * 1000 + dim)
    for Bq, Bd, Td in ((1, 1, 1), (33, 90, 50), (130, 40, 33), (7, 700, 180)):
        Q = torch.randn(Bq, Tq, dim, generator=g, device=device).to(dtype)
        D = torch.randn(Bd, Td, dim, generator=g, device=device).to(dtype)
        qm = torch.rand(Bq, Tq, generator=g, device=device) < 0.8
        dm = torch.rand(Bd, Td, generator=g, device=device) < 0.6
        if Bd > 2:
            dm[0] = dm[Bd - 1] = False
        _check(fm.inbatch_forward, Q, D, qm, dm)
        _check(fm.inbatch_forward, Q, D, None, None)
        lens = torch.randint(0, Td + 1, (Bd,), generator=g, device=device)
        cu = torch.ones(Bd + 1, dtype=torch.int32, device=device)
        cu[1:] += lens.cumsum(0).to(torch.int32)
        P = fm.PackedSeq(D.reshape(-1, dim)[:max(1, int(lens.sum()))].contiguous(), cu, int(max(1, lens.max())))
        if int(lens.sum()) > 0:
            _check(fm.packed_multi_forward, Q, P, qm)


@pytest.mark.parametrize("dtype,dim", [(torch.float16, 256), (torch.bfloat16, 768), (torch.bfloat16, 200),
                                       (torch.float32, 128), (torch.float32, 36)])
@pytest.mark.parametrize("Bq,Tq", [(300, 1), (40, 9), (130, 21), (140, 25), (50, 40), (40, 100)])
def test_split_k_tokens_in_one_run(device, dtype, dim, Bq, Tq):
    g = torch.Generator(device=device).manual_seed(Tq * 1000 + dim)
    for Bd, Td in ((1, 1), (37, 70), (200, 200)):
        Q = torch.randn(Bq, Tq, dim, generator=g, device=device).to(dtype)
        D = torch.randn(Bd, Td, dim, generator=g, device=device).to(dtype)
        qm = torch.rand(Bq, Tq, generator=g, device=device) < 0.8
        dm = torch.rand(Bd, Td, generator=g, device=device) < 0.6
        if Bd > 2:
            dm[0] = dm[Bd - 1] = False
        _check(fm.inbatch_forward, Q, D, qm, dm)
        _check(fm.inbatch_forward, Q, D, None, None)


@pytest.mark.parametrize("dtype,dim", [(torch.bfloat16, 256), (torch.float32, 128)])
@pytest.mark.parametrize("Bq,Tq,Bd", [(32, 1, 64), (24, 1, 86), (16, 2, 128), (10, 3, 128), (9, 3, 600),
                                      (33, 1, 128), (17, 2, 128)])
def test_split_k_tokens_in_one_or_two_tiles(device, dtype, dim, Bq, Tq, Bd):
    out = (ctypes.c_int64 * 4)()
    assert _lib.lib().fms_debug_split_rows(Tq, Bq, Bd, out) == 0
    assert list(out) == [1, -(-Bq * Tq // 32), 1, -(-Bq * Tq // 32) * 32 * Bd]  # one run, with room
    g = torch.Generator(device=device).manual_seed(Bq)
    Q = torch.randn(Bq, Tq, dim, generator=g, device=device).to(dtype)
    D = torch.randn(Bd, 70, dim, generator=g, device=device).to(dtype)
    qm = torch.rand(Bq, Tq, generator=g, device=device) < 0.8
    dm = torch.rand(Bd, 70, generator=g, device=device) < 0.6
    dm[0] = dm[Bd - 1] = False
    _check(fm.inbatch_forward, Q, D, qm, dm)
    _check(fm.inbatch_forward, Q, D, None, None)


@pytest.mark.parametrize("dim", [64, 256])
@pytest.mark.parametrize("Tq", [11, 20, 40])
def test_non_finite_tokens(device, Tq, dim):
    g = torch.Generator(device=device).manual_seed(Tq)
    Q = torch.randn(21, Tq, dim, generator=g, device=device).half()
    D = torch.randn(50, 70, dim, generator=g, device=device).half()
    Q[3, Tq - 1, 5], Q[4, 0, 0], Q[20, Tq // 2, 1] = float("nan"), float("inf"), float("-inf")
    D[7, 0, 2], D[8, 30, 2], D[49, 0] = float("nan"), float("inf"), float("-inf")
    _check(fm.inbatch_forward, Q, D, None, None)
    cu = torch.arange(51, dtype=torch.int32, device=device) * 70 + 1
    _check(fm.packed_multi_forward, Q, fm.PackedSeq(D.reshape(-1, dim), cu, 70), None)
