"""Workspace lent to a call (fms_workspace_lend): results do not depend on it,
whether it holds everything, part or nothing of what the call asks for; loans
are per host thread and end with the call; calls of changing sizes on several
threads and streams use memory that the allocator has given back in between."""
import threading

import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import _lib, boundary

pytestmark = pytest.mark.gpu


def _inputs(device, seed, B=40, Tq=70, Td=90, dim=128, dtype=torch.float16):
    g = torch.Generator(device=device).manual_seed(seed)
    Q = torch.randn(B, Tq, dim, generator=g, device=device).to(dtype)
    D = torch.randn(B + 3, Td, dim, generator=g, device=device).to(dtype)
    return Q, D


@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_any_loan_gives_the_same_results(device, share, dtype):
    Q, D = _inputs(device, 1, dtype=dtype)
    L = _lib.lib()
    B, Bd = Q.shape[0], D.shape[0]
    boundary._wanted.__dict__.clear()
    S0, a0 = fm.inbatch_forward(Q, D)  # nothing lent on a thread's first call
    want = boundary._wanted.__dict__["fms_inbatch_device_scan"]
    assert want > 0
    n = int(want * share)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device=device)
    guard = ws.new_full((4096,), 77)
    S, a = torch.empty_like(S0), torch.empty_like(a0)
    L.fms_workspace_lend(ws.data_ptr(), n)
    st = L.fms_inbatch_device_scan(boundary.dtype_code(Q), S.data_ptr(), a.data_ptr(), Q.data_ptr(),
                                   D.data_ptr(), None, None, Q.shape[2], Q.shape[1], B, D.shape[1],
                                   Bd, 0, boundary.stream_handle(Q.device))
    assert st == 0 and L.fms_workspace_return() == want
    assert L.fms_workspace_return() == 0  # the loan ended
    torch.cuda.synchronize()
    assert torch.equal(S, S0) and torch.equal(a, a0) and bool((guard == 77).all())
    S1, a1 = fm.inbatch_forward(Q, D)  # the driver's own loan
    assert torch.equal(S1, S0) and torch.equal(a1, a0)


def test_loans_on_threads_and_streams(device):
    sizes = [(3, 20), (40, 70), (12, 33), (60, 40)]
    cases = [_inputs(device, k, B=b, Tq=t) for k, (b, t) in enumerate(sizes)]
    want = [fm.inbatch_forward(*c) for c in cases]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        st = torch.cuda.Stream(device)
        with torch.cuda.stream(st):
            for r in range(12):
                i = (k + r) % len(cases)
                S, a = fm.inbatch_forward(*cases[i])
                junk = torch.full((1 << 18,), 255, dtype=torch.uint8, device=device)  # reuses freed memory
                G = torch.ones_like(S)
                dQ, _ = fm.inbatch_pullback(G, *cases[i], None, a)
                st.synchronize()
                if not (torch.equal(S, want[i][0]) and torch.equal(a, want[i][1])
                        and bool(torch.isfinite(dQ).all()) and bool((junk == 255).all())):
                    bad.append((k, r))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_topk_and_grouped_candidates_with_loans(device):
    g = torch.Generator(device=device).manual_seed(3)
    Q = torch.randn(40, 16, 128, generator=g, device=device).half()
    G = torch.randn(500, 40, 128, generator=g, device=device).half()
    idx = torch.randint(0, 501, (40, 500), generator=g, device=device)
    runs = []
    for _ in range(3):  # the first call on the pool, later ones on lent memory
        S, a = fm.candidates_forward(Q, G, idx)
        v, i = fm.topk(torch.cat([S] * 40, 1), 100)
        runs.append((S, a, v, i))
    for r in runs[1:]:
        assert all(torch.equal(x, y) for x, y in zip(r, runs[0]))
