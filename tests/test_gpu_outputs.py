"""The scans write every entry of their output buffers (which the drivers do not
clear), empty documents, masked tokens and rows past the last query included;
and the inverse query lengths against their definition."""
import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import boundary

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _full(S, args):
    assert bool(torch.isfinite(S).all()) and int(args.min()) >= 0


def _nan(device, *shape):
    return torch.full(shape, float("nan"), device=device)


def _neg(device, *shape):
    return torch.full(shape, -9, dtype=torch.int32, device=device)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [128, 96, 40, 256, 768])
@pytest.mark.parametrize("Tq,Td,B", [(24, 70, 5), (32, 180, 33), (45, 33, 600)])
def test_every_output_entry_is_written(device, dtype, dim, Tq, Td, B):
    g = torch.Generator(device=device).manual_seed(dim + Tq)
    Q = torch.randn(B, Tq, dim, generator=g, device=device).to(dtype)
    D = torch.randn(B, Td, dim, generator=g, device=device).to(dtype)
    qm = torch.rand(B, Tq, generator=g, device=device) < 0.8
    dm = torch.rand(B, Td, generator=g, device=device) < 0.7
    qm[0], dm[1], dm[B - 1] = False, False, False
    S, a, p = _nan(device, B), _neg(device, B, Tq), _nan(device, B, Tq)
    boundary.launch_paired_scan(a, p, Q, D, qm, dm, S, True)
    _full(S, a)
    assert bool(torch.isfinite(p).all())
    n = min(B, 40)
    S, a = _nan(device, n, B), _neg(device, n, B, Tq)
    boundary.inbatch_device_scan(S, a, Q[:n], D, qm[:n], dm, True)
    _full(S, a)
    S = _nan(device, n, B)
    boundary.inbatch_device_scan(S, None, Q[:n], D, qm[:n], dm)
    assert bool(torch.isfinite(S).all())
    idx = torch.randint(-1, B + 3, (n, 30), generator=g, device=device)
    S, a = _nan(device, n, 30), _neg(device, n, 30, Tq)
    boundary.launch_candidates_scan(a, None, Q[:n], D, idx, qm[:n], dm, B, S, -2.0)
    _full(S, a)
    lens = torch.randint(0, Td, (B,), generator=g, device=device)
    lens[0] = lens[B - 1] = 0
    cu = torch.ones(B + 1, dtype=torch.int32, device=device)
    cu[1:] += lens.cumsum(0).to(torch.int32)
    tok = D.reshape(-1, dim)[: int(lens.sum())]
    S, a = _nan(device, n, B), _neg(device, n, B, Tq)
    boundary.launch_packed_multi_scan(a, S, Q[:n], tok, cu, qm[:n], int(lens.max()))
    _full(S, a)
    S, a = _nan(device, B), _neg(device, B, Tq)
    boundary.launch_packed_scan(a, None, Q[0], tok, cu, qm[0], S)
    _full(S, a)
    S, a = _nan(device, B), _neg(device, B, Td)
    boundary.launch_varlen_scan(a, None, tok, tok, cu, cu, S, True)
    _full(S, a)


@pytest.mark.parametrize("grouping", ["never", "always", "always_direct_queries"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("dim", [128, 64, 256, 96, 512])
@pytest.mark.parametrize("Tq,Td,B", [(24, 70, 5), (45, 33, 600)])
def test_every_int8_and_grouped_output_entry_is_written(device, dtype, dim, Tq, Td, B, grouping):
    """INT8 pairs and candidates, and candidates of every type in document order."""
    g = torch.Generator(device=device).manual_seed(dim + Tq)
    Q = torch.randn(B, Tq, dim, generator=g, device=device).to(dtype)
    D = torch.randn(B, Td, dim, generator=g, device=device).to(dtype)
    qq, dd = fm.quantize_int8_symmetric(Q), fm.quantize_int8_symmetric(D)
    qm = torch.rand(B, Tq, generator=g, device=device) < 0.8
    dm = torch.rand(B, Td, generator=g, device=device) < 0.7
    qm[0], dm[1], dm[B - 1] = False, False, False
    S, a, p = _nan(device, B), _neg(device, B, Tq), _nan(device, B, Tq)
    boundary.launch_int8_paired_scan(a, p, qq.codes, qq.scales, dd.codes, dd.scales, qm, dm, S)
    _full(S, a)
    assert bool(torch.isfinite(p).all())
    S, a = _nan(device, 1), _neg(device, Tq)
    boundary.launch_int8_pair_scan(a, None, qq.codes[0], qq.scales[0], dd.codes[0], dd.scales[0], qm[0], dm[0], S)
    _full(S, a)
    n = min(B, 40)
    idx = torch.randint(-1, B + 3, (n, 30), generator=g, device=device)
    prev = boundary.candidates_grouping(grouping)
    try:
        S, a, p = _nan(device, n, 30), _neg(device, n, 30, Tq), _nan(device, n, 30, Tq)
        boundary.launch_int8_candidates_scan(a, p, qq.codes[:n], qq.scales[:n], dd.codes, dd.scales, idx, qm[:n],
                                             dm, B, S, -2.0, True)
        _full(S, a)
        assert bool(torch.isfinite(p).all())
        S, a, p = _nan(device, n, 30), _neg(device, n, 30, Tq), _nan(device, n, 30, Tq)
        boundary.launch_candidates_scan(a, p, Q[:n], D, idx, qm[:n], dm, B, S, -2.0, True)
        _full(S, a)
        assert bool(torch.isfinite(p).all())
    finally:
        boundary.candidates_grouping(prev)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [128, 40, 768])
@pytest.mark.parametrize("Tq,Td", [(5, 0), (0, 7), (0, 0)])
def test_empty_sequences_score_zero(device, dtype, dim, Tq, Td):
    junk = [torch.full((4096,), float("nan"), device=device) for _ in range(4)]  # what outputs reuse
    Q = torch.randn(3, Tq, dim, device=device).to(dtype)
    D = torch.randn(3, Td, dim, device=device).to(dtype)
    idx = torch.tensor([[1, 3], [2, 2], [0, 1]], device=device)
    del junk
    for S, a in (fm.pair_forward(Q[0], D[0]), fm.paired_forward(Q, D), fm.inbatch_forward(Q, D),
                 fm.candidates_forward(Q, D, idx, neg=-2.0)):
        assert int(a.abs().sum()) == 0
        if tuple(S.shape) == (3, 2):
            assert float(S[2, 0]) == -2.0
            S[2, 0] = 0.0
        assert float(S.abs().sum()) == 0.0


def test_zero_length_documents_score_zero(device):
    Q = torch.randn(3, 5, 64, device=device)
    S, a = fm.inbatch_forward(Q, Q[:, :0].contiguous())
    assert S.shape == (3, 3) and float(S.abs().sum()) == 0.0 and int(a.abs().sum()) == 0
    assert float(fm.maxsim(Q, Q[:, :0].contiguous(), fm.InBatch()).abs().sum()) == 0.0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,Tq", [(1, 1), (7, 32), (300, 70), (5, 0)])
def test_inverse_counts(device, dtype, n, Tq):
    g = torch.Generator(device=device).manual_seed(n)
    qm = torch.rand(n, Tq, generator=g, device=device) < 0.5
    cu = torch.ones(n + 1, dtype=torch.int32, device=device)
    cu[1:] += torch.randint(0, 50, (n,), generator=g, device=device).cumsum(0).to(torch.int32)
    for mask, c, count in ((qm, None, qm.sum(1)), (None, cu, cu[1:] - cu[:-1]),
                           (None, None, torch.full((n,), Tq, device=device))):
        out = torch.empty(n, dtype=dtype, device=device)
        boundary.inverse_counts(out, mask, c, Tq)
        assert torch.equal(out, (1.0 / count.clamp(min=1).float()).to(dtype))
