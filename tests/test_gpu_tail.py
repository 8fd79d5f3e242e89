"""The 128x128 launch that takes the last rows of a 256x256 one: its split of
a long K with every epilogue, and the row maxima it hands to the FFN's second
quantizer, at row counts that end a tile, start one and fill none."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [10753, 10880, 11008, 11001])
@pytest.mark.parametrize("kind", ["none", "gated", "resid", "acc"])
def test_tail_splitk_bitexact(sdq_dev, oracle, M, kind):
    import torch

    import sdq

    K, N = 6144, 3072
    print(f"[tail-splitk] M={M} {kind}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(M)
    A = torch.randn((M, K), generator=g, device=sdq_dev)
    q, s = oracle.quant_rows(oracle.randn(N * K, 3).reshape(N, K) * np.float32(0.02))
    bias, gate = oracle.randn(N, 4), oracle.randn(N, 5)
    w = sdq.Weight.from_host(q, s)
    plan = sdq.qlinear_plan(w, M, kind)
    assert plan[1] == ("qgemm_tail128_splitk", 10752, M - 10752), plan
    t = lambda a: torch.from_numpy(a).to(sdq_dev)  # noqa: E731
    resid = torch.randn((M, N), generator=g, device=sdq_dev)
    kw = {}
    if kind == "acc":
        Y = torch.empty((M, N), dtype=torch.int32, device=sdq_dev)
    elif kind == "none":
        Y = torch.empty((M, N), device=sdq_dev)
        kw = dict(bias=t(bias))
    else:
        Y = resid.clone()
        kw = dict(bias=t(bias), resid=Y, gate=t(gate) if kind == "gated" else None)
    sdq.profile_begin()
    sdq.qlinear(w, A, Y, kind=kind, **kw)
    torch.cuda.synchronize()
    assert "qgemm_tail128_splitk" in sdq.profile_end()
    rows = np.r_[0:3, 10749:10756, M // 2, max(10752, M - 5):M]
    rows = np.unique(rows[rows < M])
    a = A[torch.from_numpy(rows).to(sdq_dev)].cpu().numpy()
    got = Y[torch.from_numpy(rows).to(sdq_dev)].cpu().numpy()
    if kind == "acc":
        aq, _ = oracle.act_quant(a)
        assert_bitexact(got, oracle.qgemm_acc(aq, q), "acc")
    else:
        r = resid[torch.from_numpy(rows).to(sdq_dev)].cpu().numpy()
        want = oracle.linear(a, q, s, bias=bias, epilogue=kind,
                             gate=gate if kind == "gated" else None,
                             resid=r if kind != "none" else None)
        assert_bitexact(got, want, kind)


@pytest.mark.parametrize("M", [2305, 2500, 2560])
def test_ffn_row_maxima_across_the_tail(sdq_dev, oracle, M):
    """sdq_ffn whose fc1 hands its last rows to the narrower tiles: hidden
    state and residual equal, bit for bit, to two separate Linears."""
    import torch

    import sdq

    D, F = 512, 14336
    print(f"[tail-ffn] M={M}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(M)
    q1, s1 = oracle.quant_rows(oracle.randn(F * D, 6).reshape(F, D) * np.float32(0.05))
    q2, s2 = oracle.quant_rows(oracle.randn(D * F, 7).reshape(D, F) * np.float32(0.02))
    w1, w2 = sdq.Weight.from_host(q1, s1), sdq.Weight.from_host(q2, s2)
    assert len(sdq.qlinear_plan(w1, M, "gelu")) == 2
    t = lambda a: torch.from_numpy(a).to(sdq_dev)  # noqa: E731
    b1, b2, gate = t(oracle.randn(F, 8)), t(oracle.randn(D, 9)), t(oracle.randn(D, 10))
    h = torch.randn((M, D), generator=g, device=sdq_dev)
    # the largest hidden values of a row lie anywhere along it, the last columns included
    h *= torch.exp2(torch.randint(-8, 8, (M, 1), generator=g, device=sdq_dev).float())
    x = torch.randn((M, D), generator=g, device=sdq_dev)
    hid, hid2 = torch.empty((M, F), device=sdq_dev), torch.empty((M, F), device=sdq_dev)
    x2 = x.clone()
    sdq.ffn(w1, b1, w2, b2, h, gate, hid, x)
    sdq.qlinear(w1, h, hid2, kind="gelu", bias=b1)
    sdq.qlinear(w2, hid2, x2, kind="gated", bias=b2, gate=gate, resid=x2)
    torch.cuda.synchronize()
    assert torch.equal(hid, hid2)
    assert torch.equal(x, x2)
