"""The per-document dD kernel of the pullbacks at its edges, against the oracle
(tolerances of test_gpu_backward.py): documents whose sources fit LDS and do
not (2048), shared by few and by many queries, row tiles (1024 rows), one and
several shares of a document's rows, a query with more tokens than the list
holds, and query / document tokens outside every segment."""
import numpy as np
import pytest
import torch

import oracle
from helpers import as_feature, tokens
from test_gpu_backward import DT_ID, DTYPES, _abs, _vals, assert_grad

import flashmaxsim as fm
from flashmaxsim import backward as bw

pytestmark = pytest.mark.gpu


def _dev(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: DT_ID[d])
@pytest.mark.parametrize("B,C,N,Tq,Td,dim,hot", [
    (5, 16, 4, 32, 40, 128, 2),      # 640 sources a document, and none on two
    (9, 60, 30, 32, 33, 64, 3),      # documents past the LDS list among documents without a pair
    (9, 16, 3, 32, 40, 64, 2),       # 1536 sources on average: every document sorted
    (9, 16, 3, 31, 40, 64, 2),       # just below: two documents past the list, one empty
    (2, 64, 2, 32, 1030, 128, 1),    # exactly 4096 sources, two row tiles
    (1, 64, 1, 32, 70, 768, 1),      # exactly 2048: the largest LDS list; two chunks a lane
])
def test_candidates_sources_per_document(device, dtype, B, C, N, Tq, Td, dim, hot):
    rng = np.random.default_rng([B, C, N, Td])
    Qt, Qo, bf = as_feature(tokens(rng, (B, Tq, dim)), dtype)
    Gt, Go, _ = as_feature(tokens(rng, (N, Td, dim)), dtype)
    idx = rng.integers(1, hot + 1, size=(B, C)).astype(np.int64)
    args = rng.integers(0, Td + 2, size=(B, C, Tq)).astype(np.int32)  # 0 and Td + 1: no source
    Dl_t, Dl = _vals(rng, (B, C), dtype, device)
    qm = rng.random((B, Tq)) < (0.9 if N > 2 else 2.0)
    iv_t, iv = _vals(rng, (B,), dtype, device, positive=True)
    want = oracle.candidates_backward(Qo, Go, idx, args, Dl, iv, qm, bf16=bf)
    mag = oracle.candidates_backward(_abs(Qo, bf), _abs(Go, bf), idx, args, np.abs(Dl), iv, qm, bf16=bf)
    dQ, dG = bw.candidates_pullback(Dl_t, Qt.to(device), Gt.to(device), _dev(idx, device),
                                    _dev(qm, device), _dev(args, device), iv_t)
    torch.cuda.synchronize()
    assert_grad(dQ, want[0], mag[0], dtype, "dQ")
    assert_grad(dG, want[1], mag[1], dtype, "dG")


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: DT_ID[d])
@pytest.mark.parametrize("Tq,Td,B", [(2048, 35, 2), (2049, 1100, 2), (3, 1, 700), (33, 257, 300)])
def test_paired_long_queries_and_many_pairs(device, dtype, Tq, Td, B):
    rng = np.random.default_rng([Tq, Td, B])
    dim = 64
    Qt, Qo, bf = as_feature(tokens(rng, (B, Tq, dim)), dtype)
    Dt, Do, _ = as_feature(tokens(rng, (B, Td, dim)), dtype)
    args = rng.integers(0, Td + 2, size=(B, Tq)).astype(np.int32)
    Dl_t, Dl = _vals(rng, (B,), dtype, device)
    want = oracle.paired_backward(Qo, Do, args, Dl, None, None, bf16=bf)
    mag = oracle.paired_backward(_abs(Qo, bf), _abs(Do, bf), args, np.abs(Dl), None, None, bf16=bf)
    dQ, dD = bw.paired_pullback(Dl_t, Qt.to(device), Dt.to(device), None, _dev(args, device))
    torch.cuda.synchronize()
    assert_grad(dQ, want[0], mag[0], dtype, "dQ")
    assert_grad(dD, want[1], mag[1], dtype, "dD")


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: DT_ID[d])
def test_ragged_tokens_outside_every_segment(device, dtype):
    """A device cu is trusted as given: segments that start late, end early or leave
    nothing in between; rows of no segment get zero gradients."""
    rng = np.random.default_rng(5)
    dim, nq, nd = 64, 40, 90
    Qt, Qo, bf = as_feature(tokens(rng, (nq, dim)), dtype)
    Dt, Do, _ = as_feature(tokens(rng, (nd, dim)), dtype)
    cu_q = np.array([4, 9, 9, 30], np.int32)
    cu_d = np.array([6, 40, 41, 70], np.int32)
    max_q = 13  # shorter than the last query segment
    args = rng.integers(1, 3, size=(3, max_q)).astype(np.int32)
    Dl_t, Dl = _vals(rng, (3,), dtype, device)
    P = fm.PackedSeq(Qt.to(device), _dev(cu_q, device), max_q)
    R = fm.PackedSeq(Dt.to(device), _dev(cu_d, device), 34)
    dQ, dD = bw.varlen_pullback(Dl_t, P, R, _dev(args, device))
    q, d = Qt.double().numpy(), Dt.double().numpy()
    wQ, wD = np.zeros_like(q), np.zeros_like(d)
    mQ, mD = np.zeros_like(q), np.zeros_like(d)
    for n in range(3):
        tq, td = min(cu_q[n + 1] - cu_q[n], max_q), cu_d[n + 1] - cu_d[n]
        for t in range(tq):
            u = args[n, t]
            if u <= td:
                i, j = cu_q[n] - 1 + t, cu_d[n] - 1 + u - 1
                wQ[i] += Dl[n] * d[j]
                wD[j] += Dl[n] * q[i]
                mQ[i] += abs(Dl[n] * d[j])
                mD[j] += abs(Dl[n] * q[i])
    torch.cuda.synchronize()
    assert_grad(dQ, wQ, mQ, dtype, "dQ")
    assert_grad(dD, wD, mD, dtype, "dD")
    q1 = Qt[:7].to(device)
    tape = rng.integers(1, 3, size=(3, 7)).astype(np.int32)
    dq, dP = bw.packed_pullback(Dl_t, q1, R, None, _dev(tape, device))
    torch.cuda.synchronize()
    g = dP.float().cpu().numpy()
    assert np.isfinite(g).all() and (g[:5] == 0).all() and (g[69:] == 0).all()
    assert (g[5:7] != 0).any()


def _ragged_want(Qt, Dt, cu_q, cu_d, args, Dl):
    """(dQ, dD, |dQ| terms, |dD| terms) of ragged pairs; cu_q None: one query for all."""
    q, d = Qt.double().numpy(), Dt.double().numpy()
    out = [np.zeros_like(q), np.zeros_like(d), np.zeros_like(q), np.zeros_like(d)]
    n, rows = args.shape
    for i in range(n):
        a, tq = (0, len(q)) if cu_q is None else (cu_q[i] - 1, min(cu_q[i + 1] - cu_q[i], rows))
        u = args[i, :tq].astype(np.int64)
        t = np.flatnonzero((u >= 1) & (u <= cu_d[i + 1] - cu_d[i]))
        r, c = a + t, cu_d[i] - 1 + u[t] - 1
        for k, (dst, src, x) in enumerate(((r, c, d), (c, r, q))):
            np.add.at(out[k], dst, Dl[i] * x[src])
            np.add.at(out[k + 2], dst, np.abs(Dl[i] * x[src]))
    return out


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: DT_ID[d])
@pytest.mark.parametrize("dim", [64, 768])
@pytest.mark.parametrize("lens,before,after", [
    # far from the average length: past what a document's own workgroups take (256 rows
    # here), to the row, in several windows, and next to one another
    ([255, 256, 257, 1, 0, 511, 512, 513, 1300] + [3] * 40, 0, 0),
    ([3] * 30 + [2900] + [3] * 30 + [0, 700], 600, 1025),  # rows of no document on both ends
    ([2000, 2000, 9], 0, 0),  # three documents: shares of long ones, none in a window
])
def test_ragged_long_documents(device, dtype, dim, lens, before, after):
    rng = np.random.default_rng([len(lens), before])
    N, Tq = len(lens), 12
    cu_d = (before + 1 + np.concatenate([[0], np.cumsum(lens)])).astype(np.int32)
    qlens = rng.integers(0, Tq + 1, N)
    qlens[0] = Tq
    cu_q = (1 + np.concatenate([[0], np.cumsum(qlens)])).astype(np.int32)
    nd = before + sum(lens) + after
    Dt, _, _ = as_feature(tokens(rng, (nd, dim)), dtype)
    Qt, _, _ = as_feature(tokens(rng, (int(qlens.sum()), dim)), dtype)
    args = np.stack([rng.integers(0, n + 2, Tq) for n in lens]).astype(np.int32)
    Dl_t, Dl = _vals(rng, (N,), dtype, device)
    P = fm.PackedSeq(Dt.to(device), _dev(cu_d, device), max(lens))
    R = fm.PackedSeq(Qt.to(device), _dev(cu_q, device), Tq)
    dQ, dD = bw.varlen_pullback(Dl_t, R, P, _dev(args, device))
    want = _ragged_want(Qt, Dt, cu_q, cu_d, args, Dl)
    assert_grad(dQ, want[0], want[2], dtype, "dQ")
    assert_grad(dD, want[1], want[3], dtype, "dD")
    q1 = Qt[:Tq].contiguous()
    dq, dP = bw.packed_pullback(Dl_t, q1.to(device), P, None, _dev(args, device))
    want = _ragged_want(q1, Dt, None, cu_d, args, Dl)
    assert_grad(dq, want[0], want[2], dtype, "dq")
    assert_grad(dP, want[1], want[3], dtype, "dP")


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: DT_ID[d])
@pytest.mark.parametrize("dim", [64, 768])
@pytest.mark.parametrize("before,after", [(0, 127), (128, 0), (129, 130), (700, 1100)])
def test_query_rows_of_no_pair_are_zero(device, dtype, dim, before, after):
    """Any number of them: ahead of the first query and past the last (windows of 128 rows),
    and a query segment far longer than max_q."""
    rng = np.random.default_rng([before, after])
    qlens, dlens, max_q = [3, 12, 0, 500, 1, 128, 129, 12], [20] * 8, 12
    cu_q = (before + 1 + np.concatenate([[0], np.cumsum(qlens)])).astype(np.int32)
    cu_d = (1 + np.concatenate([[0], np.cumsum(dlens)])).astype(np.int32)
    Qt, _, _ = as_feature(tokens(rng, (before + sum(qlens) + after, dim)), dtype)
    Dt, _, _ = as_feature(tokens(rng, (sum(dlens), dim)), dtype)
    args = rng.integers(1, 21, size=(8, max_q)).astype(np.int32)
    Dl_t, Dl = _vals(rng, (8,), dtype, device)
    junk = torch.full_like(Qt, float("nan"), device=device)  # what the allocator hands out next
    R = fm.PackedSeq(Qt.to(device), _dev(cu_q, device), max_q)
    P = fm.PackedSeq(Dt.to(device), _dev(cu_d, device), 20)
    tape = _dev(args, device)
    del junk
    dQ, dD = bw.varlen_pullback(Dl_t, R, P, tape)
    want = _ragged_want(Qt, Dt, cu_q, cu_d, args, Dl)
    assert_grad(dQ, want[0], want[2], dtype, "dQ")
    assert_grad(dD, want[1], want[3], dtype, "dD")


def _best_us(fn):
    fn()
    best = float("inf")
    for _ in range(8):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        fn()
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3)
    return best


def test_one_long_document_costs_no_more_than_its_rows(device):
    """1000 documents over 100000 rows, all of 100 rows or one of 90000: the same rows,
    pairs and sources, so about the same time (left to one workgroup, the long one took
    over 20 times as long)."""
    g = torch.Generator(device=device).manual_seed(1)
    tok = torch.randn(100000, 128, generator=g, device=device).bfloat16()
    q = torch.randn(32, 128, generator=g, device=device).bfloat16()
    us = []
    for lens in ([100] * 1000, [10] * 500 + [90009] + [10] * 498 + [11]):
        cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]) + 1, dtype=torch.int32, device=device)
        assert int(cu[-1]) == 100001
        P = fm.PackedSeq(tok, cu, max(lens))
        S, a = fm.packed_forward(q, P)
        us.append(_best_us(lambda: bw.packed_pullback(torch.ones_like(S), q, P, None, a)))
    print("us", us)
    assert us[1] < 6 * us[0]


def test_rows_past_the_last_pair_cost_no_more_than_their_bytes(device):
    """200 pairs in stores with 100000 rows past the last one, against the same rows as 200
    longer pairs (left to one wave, dQ's spare rows took over 10 times as long)."""
    g = torch.Generator(device=device).manual_seed(1)
    q = torch.randn(104000, 128, generator=g, device=device).bfloat16()
    cu_d = torch.arange(201, dtype=torch.int32, device=device) * 100 + 1
    P = fm.PackedSeq(torch.randn(20000, 128, generator=g, device=device).bfloat16(), cu_d, 100)
    us = []
    for n in (520, 20):
        R = fm.PackedSeq(q, torch.arange(201, dtype=torch.int32, device=device) * n + 1, 20)
        S, a = fm.varlen_forward(R, P)
        us.append(_best_us(lambda: bw.varlen_pullback(torch.ones_like(S), R, P, a)))
    print("us", us)
    assert us[1] < 5 * us[0]
