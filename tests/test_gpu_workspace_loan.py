"""Workspace lent to a call (fms_set_workspace_lender): results do not depend on it,
whether what a call asks for is lent or not, and nothing is written beside it; torch
lends each call exactly what it asks for, whatever sizes came before, on every thread;
calls of changing sizes on several threads and streams use memory that the allocator
has given back in between."""
import gc
import threading

import pytest
import torch

import flashmaxsim as fm
from flashmaxsim import _lib, boundary

pytestmark = pytest.mark.gpu


def _inputs(device, seed, B=40, Tq=70, Td=90, dim=128, dtype=torch.float16):
    """Small integers: sums of their products are exact in any order."""
    g = torch.Generator(device=device).manual_seed(seed)
    Q = torch.randint(-3, 4, (B, Tq, dim), generator=g, device=device).to(dtype)
    D = torch.randint(-3, 4, (B + 3, Td, dim), generator=g, device=device).to(dtype)
    return Q, D


class _Lender:
    """Lends the first `pieces` requests of a call from one guarded buffer."""

    GAP, FILL = 4096, 77

    def __init__(self, device, pieces):
        self.buf = torch.full((64 << 20,), self.FILL, dtype=torch.uint8, device=device)
        self.base = -self.buf.data_ptr() % 256 + self.GAP
        self.pieces, self.asked, self.lent = pieces, [], []
        self.fn = _lib.LENDER(self._lend)

    def _lend(self, nbytes, stream):
        self.asked.append(nbytes)
        if len(self.asked) > self.pieces:
            return None
        at = self.lent[-1][1] + self.GAP if self.lent else self.base
        at += -(self.buf.data_ptr() + at) % 256
        assert at + nbytes + self.GAP <= self.buf.numel()
        self.lent.append((at, at + nbytes))
        return self.buf.data_ptr() + at

    def __enter__(self):
        _lib.lib().fms_set_workspace_lender(self.fn)
        return self

    def __exit__(self, *exc):
        _lib.lib().fms_set_workspace_lender(_lib.LENDER(0))
        boundary._this_thread()  # the drivers' lender again
        torch.cuda.synchronize()
        at = 0
        for a, z in self.lent + [(self.buf.numel(), 0)]:
            assert bool((self.buf[at:a] == self.FILL).all()), (self.lent, at)
            at = z


# Each call that needs workspace asks once: the in-batch scans of rows of whole 16-byte
# units, every pullback.
@pytest.mark.parametrize("pieces", [0, 1])
@pytest.mark.parametrize("dtype,dim", [(torch.float16, 128), (torch.float16, 256), (torch.float32, 64),
                                       (torch.float16, 100), (torch.float32, 101)])
def test_any_loan_gives_the_same_results(device, pieces, dtype, dim):
    Q, D = _inputs(device, 1, dim=dim, dtype=dtype)
    L = _lib.lib()
    B, Tq, Bd, Td = Q.shape[0], Q.shape[1], D.shape[0], D.shape[1]
    S0, a0 = fm.inbatch_forward(Q, D)
    G = (torch.arange(B * Bd, device=device).reshape(B, Bd) % 3 - 1).to(dtype)
    dQ0, dD0 = fm.inbatch_pullback(G, Q, D, None, a0)
    S, a, dQ, dD = (torch.empty_like(x) for x in (S0, a0, dQ0, dD0))
    code, stream = boundary.dtype_code(Q), boundary.stream_handle(Q.device)
    scan_asks = 1 if dim * Q.element_size() % 16 == 0 else 0
    with _Lender(device, pieces) as lender:
        assert L.fms_inbatch_device_scan(code, S.data_ptr(), a.data_ptr(), Q.data_ptr(), D.data_ptr(),
                                         None, None, dim, Tq, B, Td, Bd, 0, stream) == 0
        assert len(lender.asked) == scan_asks
    with _Lender(device, pieces) as lender:
        assert L.fms_inbatch_pullback(code, dQ.data_ptr(), dD.data_ptr(), Q.data_ptr(), D.data_ptr(), None,
                                      a.data_ptr(), G.data_ptr(), None, dim, Tq, Td, B, Bd, stream) == 0
        assert len(lender.asked) == 1 and len(lender.lent) == pieces
    for x, y in ((S, S0), (a, a0), (dQ, dQ0), (dD, dD0)):
        assert torch.equal(x, y)
    S1, a1 = fm.inbatch_forward(Q, D)  # the driver's own lender again
    assert torch.equal(S1, S0) and torch.equal(a1, a0)


def _lent_by(call):
    """(torch allocations, most bytes held) of a call, results dropped."""
    gc.collect()
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    n0 = torch.cuda.memory_stats()["allocation.all.allocated"]
    out = call()
    n = torch.cuda.memory_stats()["allocation.all.allocated"] - n0
    peak = torch.cuda.max_memory_allocated() - base
    del out
    return n, peak


def test_torch_lends_what_each_call_needs(device):
    """The scores, the tape and one workspace per call: the first call of a size and of a
    thread as well, and no more for a small call after a large one."""
    sizes = [(4, 20), (90, 70), (4, 20), (40, 33), (90, 70)]
    cases = [_inputs(device, k, B=b, Tq=t, dim=256) for k, (b, t) in enumerate(sizes)]
    seen = {}

    def work(tag):
        seen[tag] = [_lent_by(lambda: fm.inbatch_forward(*c)) for c in cases]

    work("here")
    th = threading.Thread(target=work, args=("there",))
    th.start()
    th.join()
    assert seen["here"] == seen["there"]
    assert [n for n, _ in seen["here"]] == [3] * len(sizes)
    assert seen["here"][0] == seen["here"][2] and seen["here"][1] == seen["here"][4]
    assert seen["here"][2][1] * 20 < seen["here"][1][1]


def test_a_call_outside_the_drivers_is_not_lent_to(device):
    """The library keeps a thread's lender; it declines calls that the drivers do not make."""
    Q, D = _inputs(device, 2)
    S0, a0 = fm.inbatch_forward(Q, D)
    S, a = torch.empty_like(S0), torch.empty_like(a0)
    n0 = torch.cuda.memory_stats()["allocation.all.allocated"]
    assert _lib.lib().fms_inbatch_device_scan(
        boundary.dtype_code(Q), S.data_ptr(), a.data_ptr(), Q.data_ptr(), D.data_ptr(), None, None, Q.shape[2],
        Q.shape[1], Q.shape[0], D.shape[1], D.shape[0], 0, boundary.stream_handle(Q.device)) == 0
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == n0
    assert torch.equal(S, S0) and torch.equal(a, a0)


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
    for _ in range(3):
        S, a = fm.candidates_forward(Q, G, idx)
        v, i = fm.topk(torch.cat([S] * 40, 1), 100)
        runs.append((S, a, v, i))
    for r in runs[1:]:
        assert all(torch.equal(x, y) for x, y in zip(r, runs[0]))
