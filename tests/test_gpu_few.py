"""The workgroup-per-pair scan of few pairs against the wave-per-pair scans.

A call of at most 512 pairs (fp32: of any number, from 16-byte aligned arrays)
takes the former, a larger one (fp32: one from other addresses) the latter; the
same pairs must score and choose bit for bit alike in both (every scan
accumulates a dot product in the same k order).  Sizes cover its edges:
one and many chunks per wave, partial chunks and query tiles, rows of one or
several load batches and rows that end inside one, documents with no valid
token, and the first-valid-token rule with NaN and infinite rows.
"""
import numpy as np
import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import boundary

pytestmark = pytest.mark.gpu

MANY = 513  # one more pair than the workgroup-per-pair scan takes


def _moved(x):
    """fp32: the same array 4 bytes past a 16-byte boundary (else the array itself)."""
    if x.dtype != torch.float32:
        return x
    y = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
    y.copy_(x)
    assert y.data_ptr() % 16 == 4
    return y


def _case(dtype, B, Tq, Td, dim, device, seed=0, odd=False):
    g = torch.Generator(device=device).manual_seed(seed)
    Q = torch.randn(B, Tq, dim, generator=g, device=device)
    D = torch.randn(B, Td, dim, generator=g, device=device)
    qm = torch.rand(B, Tq, generator=g, device=device) < 0.9
    dm = torch.rand(B, Td, generator=g, device=device) < 0.8
    dm[0] = False                       # no valid token
    dm[1 % B, : Td // 2] = False        # the first valid token in a later chunk
    if odd:
        first = dm.float().argmax(1)
        D[1 % B, first[1 % B]] = float("nan")           # sticks: the first valid token
        D[2 % B, min(Td - 1, 40)] = float("nan")        # skipped: a later one
        D[3 % B] = -float("inf")                        # nothing above -inf
        Q[3 % B] = Q[3 % B].abs() + 0.1
        D[4 % B, Td - 1] = float("inf")
    return Q.to(dtype), D.to(dtype), qm, dm


def _same(a, b):
    return torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("dtype,dim", [
    (torch.float16, 64), (torch.float16, 128), (torch.bfloat16, 96), (torch.float16, 40),
    (torch.bfloat16, 256), (torch.bfloat16, 384), (torch.float16, 1024), (torch.float32, 64),
    (torch.float32, 128), (torch.float32, 100), (torch.float32, 4), (torch.float32, 768)])
@pytest.mark.parametrize("Tq,Td", [(32, 180), (33, 65), (5, 40), (70, 530)])
def test_paired_matches_the_wave_per_pair_scan(device, dtype, dim, Tq, Td, odd):
    B = 6
    Q, D, qm, dm = _case(dtype, B, Tq, Td, dim, device, odd=odd)
    rep = -(-MANY // B)
    big = [x.repeat(rep, *([1] * (x.dim() - 1))) for x in (Q, D, qm, dm)]
    big[1] = _moved(big[1])
    for norm in (False, True):
        S, args = fm.paired_forward(Q, D, qm, dm, normalize=norm)
        S_b, args_b = fm.paired_forward(*big, normalize=norm)
        assert torch.equal(args, args_b[:B])
        if odd:  # (NaN payloads are not compared)
            assert torch.equal(torch.isnan(S), torch.isnan(S_b[:B]))
            S, S_b = S.nan_to_num(nan=0.0), S_b.nan_to_num(nan=0.0)
        assert _same(S, S_b[:B])
        S2, _ = fm.paired_forward(Q, D, qm, dm, normalize=norm, tape=False)
        assert _same(S2.nan_to_num(nan=0.0) if odd else S2, S)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("dim", [64, 128, 48, 512])
def test_int8_matches_the_wave_per_pair_scan(device, dtype, dim):
    B, Tq, Td = 6, 20, 75
    Q, D, qm, dm = _case(dtype, B, Tq, Td, dim, device)
    rep = -(-MANY // B)
    idx = fm.quantize_int8_symmetric(D)
    big = fm.Int8Index(idx.codes.repeat(rep, 1, 1), idx.scales.repeat(rep, 1))
    S, args = fm.int8_paired_forward(Q, idx, qm, dm)
    S_b, args_b = fm.int8_paired_forward(Q.repeat(rep, 1, 1), big, qm.repeat(rep, 1), dm.repeat(rep, 1))
    assert _same(S, S_b[:B]) and torch.equal(args, args_b[:B])


@pytest.mark.parametrize("idx_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype,dim", [(torch.float16, 128), (torch.float32, 128), (torch.bfloat16, 768)])
def test_candidates_match_the_wave_per_pair_scan(device, dtype, dim, idx_dtype):
    B, C, N, Tq, Td = 3, 17, 9, 24, 130
    _, G, _, dm = _case(dtype, N, Tq, Td, dim, device)
    Q, _, qm, _ = _case(dtype, B, Tq, Td, dim, device, seed=1)
    g = torch.Generator(device=device).manual_seed(2)
    idx = torch.randint(-1, N + 3, (B, C), generator=g, device=device).to(idx_dtype)
    rep = -(-MANY // C)
    prev = boundary.candidates_grouping("never")
    try:
        S, args = fm.candidates_forward(Q, G, idx, qm, dm, neg=-7.0)
        S_b, args_b = fm.candidates_forward(Q, _moved(G), idx.repeat(1, rep), qm, dm, neg=-7.0)
    finally:
        boundary.candidates_grouping(prev)
    assert _same(S, S_b[:, :C]) and torch.equal(args, args_b[:, :C])
    bad = (idx < 1) | (idx > N)
    assert bool((S[bad] == -7.0).all()) and not bool((S[~bad] == -7.0).any())


@pytest.mark.parametrize("dtype,dim", [(torch.bfloat16, 128), (torch.float32, 128), (torch.float16, 1024)])
def test_ragged_layouts_match_the_wave_per_pair_scan(device, dtype, dim):
    rng = np.random.default_rng(3)
    dl = [0, 1, 31, 32, 33, 700, 64, 290]
    ql = [3, 32, 40, 1, 0, 33, 17, 5]
    g = torch.Generator(device=device).manual_seed(4)

    def docs(lens):
        return [torch.randn(n, dim, generator=g, device=device).to(dtype) for n in lens]

    d, q = docs(dl), docs(ql)
    rep = -(-MANY // len(dl))
    q1 = torch.randn(35, dim, generator=g, device=device).to(dtype)
    qm = torch.from_numpy(rng.random(35) < 0.8).to(device)
    S, args = fm.packed_forward(q1, fm.pack_docs(d), qm, normalize=True)
    many = fm.pack_docs(d * rep)
    many.tokens = _moved(many.tokens)
    S_b, args_b = fm.packed_forward(q1, many, qm, normalize=True)
    assert _same(S, S_b[: len(dl)]) and torch.equal(args, args_b[: len(dl)])
    assert float(S[0]) == 0.0 and int(args[0].abs().max()) == 0
    S, args = fm.varlen_forward(*fm.pack_pairs(q, d), normalize=True)
    S_b, args_b = fm.varlen_forward(fm.pack_docs(q * rep), many, normalize=True)
    assert _same(S, S_b[: len(dl)]) and torch.equal(args, args_b[: len(dl)])


@pytest.mark.parametrize("grouping", ["never", "always"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_d96_matches_padded_rows(device, dtype, grouping):
    """d = 96 against the same features padded with zeros to d = 128 (the added products are
    +0), in output order and as document batches, past the sizes of the few-pair scan."""
    B, C, N, Tq, Td = 5, 130, 40, 37, 70
    _, G, _, dm = _case(dtype, N, Tq, Td, 96, device)
    Q, _, qm, _ = _case(dtype, B, Tq, Td, 96, device, seed=1)
    g = torch.Generator(device=device).manual_seed(2)
    idx = torch.randint(0, N + 1, (B, C), generator=g, device=device)
    pad = torch.nn.functional.pad
    prev = boundary.candidates_grouping(grouping)
    try:
        S, a = fm.candidates_forward(Q, G, idx, qm, dm, neg=-7.0)
        S_p, a_p = fm.candidates_forward(pad(Q, (0, 32)), pad(G, (0, 32)), idx, qm, dm, neg=-7.0)
    finally:
        boundary.candidates_grouping(prev)
    assert torch.equal(S, S_p) and torch.equal(a, a_p)


@pytest.mark.parametrize("dim,Td", [(256, 160), (256, 240), (384, 60), (768, 100), (192, 300)])
@pytest.mark.parametrize("layout", ["packed", "varlen"])
def test_wide_rows_past_one_workgroup_per_cu(device, layout, dim, Td):
    """256 and 257 16-bit pairs, documents on both sides of the size up to which the latter
    still take a workgroup each: the same pairs score and choose alike."""
    g = torch.Generator(device=device).manual_seed(dim + Td)
    d = [torch.randn(Td - i % 3, dim, generator=g, device=device).half() for i in range(257)]
    q = [torch.randn(1 + i % 35, dim, generator=g, device=device).half() for i in range(257)]
    out = []
    for n in (256, 257):
        if layout == "packed":
            out.append(fm.packed_forward(q[31], fm.pack_docs(d[:n])))
        else:
            out.append(fm.varlen_forward(*fm.pack_pairs(q[:n], d[:n])))
    (S, a), (S1, a1) = out
    assert _same(S, S1[:256]) and torch.equal(a, a1[:256])
