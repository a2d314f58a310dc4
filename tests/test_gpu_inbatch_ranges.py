"""The split-K in-batch kernel's chunk list and ranges at their edges, against the
paired scan of the same pairs (16-bit, d = 256: the same k order, so bit for bit):
more documents than one and than several blocks of the list kernel, fewer query groups than XCDs and
many, documents without a valid token at both ends of the list, single valid rows
in late chunks, documents longer than a chunk group, and one K slice per group."""
import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import _lib

pytestmark = pytest.mark.gpu


def _masks(g, B, T, device, p):
    m = torch.rand(B, T, generator=g, device=device) < p
    return m


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Bq,Bd,Tq,Td", [
    (1, 1, 1, 1), (3, 2500, 5, 40), (300, 7, 32, 33), (9, 1025, 33, 31), (70, 60, 32, 225),
    (2, 1024, 8, 64), (17, 300, 40, 400), (2, 5003, 3, 70), (1, 2048, 9, 33)])
def test_ranges_match_the_paired_scan(device, dtype, Bq, Bd, Tq, Td):
    dim = 256
    g = torch.Generator(device=device).manual_seed(Bq * 1000 + Bd)
    Q = torch.randn(Bq, Tq, dim, generator=g, device=device).to(dtype)
    D = torch.randn(Bd, Td, dim, generator=g, device=device).to(dtype)
    qm, dm = _masks(g, Bq, Tq, device, 0.8), _masks(g, Bd, Td, device, 0.5)
    if Bd > 4:
        dm[0] = dm[1] = dm[Bd - 1] = False
        dm[2] = False
        dm[2, Td - 1] = True               # one valid row, in the last chunk
        dm[3] = True
        dm[Bd // 2:Bd // 2 + 2] = False
    assert _lib.lib().fms_debug_inbatch_kernel(1 if dtype == torch.float16 else 2, dim, Tq, Td, Bq, Bd,
                                               Q.data_ptr(), D.data_ptr()) == 2
    for mask in (dm, None):
        S, a = fm.inbatch_forward(Q, D, qm, mask, normalize=True)
        S0, _ = fm.inbatch_forward(Q, D, qm, mask, normalize=True, tape=False)
        assert torch.equal(S, S0)
        n = min(Bq * Bd, 3000)
        pick = torch.randperm(Bq * Bd, generator=g, device=device)[:n]
        i, j = pick // Bd, pick % Bd
        P, ap = fm.paired_forward(Q[i].contiguous(), D[j].contiguous(), qm[i].contiguous(),
                                  None if mask is None else mask[j].contiguous())
        assert torch.equal(a[i, j], ap)
        if Tq <= 32:  # (several tiles per query: summed tile by tile, scaled once)
            P, _ = fm.paired_forward(Q[i].contiguous(), D[j].contiguous(), qm[i].contiguous(),
                                     None if mask is None else mask[j].contiguous(), normalize=True)
            assert torch.equal(S[i, j], P)


@pytest.mark.parametrize("dim", [4, 32, 36, 128])
@pytest.mark.parametrize("Bq,Bd,Tq,Td", [(5, 1100, 7, 35), (66, 20, 32, 130), (1, 3, 64, 97)])
def test_fp32_ranges(device, dim, Bq, Bd, Tq, Td):
    g = torch.Generator(device=device).manual_seed(dim + Bd)
    Q = torch.randn(Bq, Tq, dim, generator=g, device=device)
    D = torch.randn(Bd, Td, dim, generator=g, device=device)
    dm = _masks(g, Bd, Td, device, 0.6)
    dm[Bd - 1] = False
    S, a = fm.inbatch_forward(Q, D, None, dm)
    S0, _ = fm.inbatch_forward(Q, D, None, dm, tape=False)
    assert torch.equal(S, S0) and int(a[:, Bd - 1].abs().sum()) == 0
    sims = (Q.double().reshape(-1, dim) @ D.double().reshape(-1, dim).t()).reshape(Bq, Tq, Bd, Td)
    sims = sims.masked_fill(~dm[None, None], float("-inf")).permute(0, 2, 1, 3)
    best = sims.max(-1).values
    want = torch.where(best.isinf(), torch.zeros_like(best), best)
    # the chosen token reaches the maximum to fp32 rounding: dim products of N(0, 1)
    tol = 1e-6 * (dim ** 0.5 + 1) * 10
    took = torch.gather(sims, 3, (a.long() - 1).clamp(min=0)[..., None])[..., 0]
    assert bool(((took - best)[a > 0].abs() <= tol).all())
    assert bool(((S.double() - want.sum(-1)).abs() <= tol * Tq).all())

