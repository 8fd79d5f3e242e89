"""Row norms whose rows stay in registers (up to 3072 columns): layernorm,
rmsnorm + RoPE and the norm + modulation quantizer at the edges of their
workgroups (14 rows), chunks (256 columns; 2, 4, 6, .. 12 held) and limit,
bit-exact against the oracle, with the first shapes past the limit beside
them."""
import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu


def _x(oracle, M, K, seed):
    rng = np.random.default_rng(seed)
    return (oracle.randn(M * K, seed).reshape(M, K) * rng.uniform(0.1, 20, (M, 1))
            + rng.uniform(-9, 9, (M, 1))).astype(np.float32)


@pytest.mark.parametrize("M,K", [(1, 4), (13, 256), (14, 260), (15, 1024), (29, 1028), (3, 2044),
                                 (28, 2048), (16, 2052), (14, 3068), (43, 3072), (15, 3076),
                                 (14, 3074), (29, 508), (14, 512), (1, 516), (15, 1536),
                                 (14, 1540), (43, 2560), (15, 2564)])
def test_rows_bitexact(sdq_dev, oracle, M, K):
    import torch

    import sdq

    print(f"[rowblock] M={M} K={K}", flush=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(sdq_dev)  # noqa: E731
    x = _x(oracle, M, K, M + 3 * K)
    w, b = oracle.randn(K, 11), oracle.randn(K, 12)
    # layernorm: the rows end the allocation; a guard row follows the output
    y = torch.full((M + 1, K), -7.0, device=sdq_dev)
    sdq.layernorm(t(x), y[:M], t(w), t(b), 1e-6)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert_bitexact(got[:M], oracle.layernorm(x, 1e-6, w, b), "layernorm")
    assert (got[M] == -7.0).all()
    # rmsnorm + RoPE of some pairs of each head, two segments of rows inside
    # wider rows, the second with its own row count
    for heads in (1, 2):
        hd = K // heads
        if K % heads or hd % 2:
            continue
        nr = max(1, hd // 2 - 1)
        ang = (np.random.default_rng(5).uniform(-3, 3, (M, nr))).astype(np.float32)
        cs = oracle.rope_cs(ang)
        rows = np.zeros((M, 2 * K + 4), np.float32)
        rows[:, :K], rows[:, K + 4:] = x, x[::-1]
        d = t(rows)
        d2 = t(x[:max(1, M // 2)])
        sdq.rmsnorm_rope_batch([(d, 0, t(w), t(cs)), (d2, 0, t(w), None), (d, K + 4, t(b), t(cs))],
                               K, heads)
        torch.cuda.synchronize()
        got = d.cpu().numpy()

        for c0, src, wt in ((0, x, w), (K + 4, x[::-1], b)):
            assert_bitexact(got[:, c0:c0 + K],
                            oracle.rope(oracle.rmsnorm(src, wt, 1e-6), cs, heads), "rms + rope")
        assert (got[:, K:K + 4] == 0).all()
        assert_bitexact(d2.cpu().numpy(), oracle.rmsnorm(x[:max(1, M // 2)], w, 1e-6), "rmsnorm")
    # norm + modulation + quantizer under a Linear
    N = 132
    q, s = oracle.quant_rows(oracle.randn(N * K, 13).reshape(N, K) * np.float32(0.02))
    shift, scale = oracle.randn(K, 14), oracle.randn(K, 15) * np.float32(0.2)
    Y = torch.full((M, N), -7.0, device=sdq_dev)
    sdq.qlinear_lnmod(sdq.Weight.from_host(q, s), t(x), Y, t(shift), t(scale), 1e-6)
    torch.cuda.synchronize()
    h = oracle.mod_rows(oracle.layernorm(x, 1e-6), shift, scale)
    assert_bitexact(Y.cpu().numpy(), oracle.linear(h, q, s), "lnmod linear")


@pytest.mark.parametrize("v", [0.5, 1.5, 2.5, -0.5, -3.5, 126.5, -126.5, 127.0])
def test_quantizer_rounding(sdq_dev, oracle, v):
    """Ties, signs, NaN, infinities, denormal and huge rows through the
    quantizer, codes bit-exact against the oracle."""
    import torch

    import sdq

    K, N = 256, 128
    print(f"[quant] v={v}", flush=True)
    x = np.zeros((8, K), np.float32)
    x[0, :8] = [127.0, v, -v, v + 1, 0.0, -0.0, 126.49999, -127.0]
    x[1, :4] = [np.nan, 127.0, v, 1.0]
    x[2, :4] = [np.inf, 1.0, v, -1.0]
    x[3, :4] = [1e-42, v * 1e-43, -1e-42, 0.0]
    x[4, :4] = [3e38, v, -3e38, 1e38]
    x[5] = v
    x[6, :3] = [-np.inf, v, np.nan]
    # the identity-like weight shows the codes: column j of the output is code j
    q = np.zeros((N, K), np.int8)
    q[np.arange(N), np.arange(N)] = 1
    s = np.ones(N, np.float32)
    d = torch.from_numpy(np.tile(x, (12, 1))).to(sdq_dev)
    Y = torch.empty((96, N), dtype=torch.int32, device=sdq_dev)
    sdq.qlinear(sdq.Weight.from_host(q, s), d, Y, kind="acc")
    torch.cuda.synchronize()
    codes, _ = oracle.act_quant(x)
    assert_bitexact(Y.cpu().numpy(), np.tile(codes[:, :N].astype(np.int32), (12, 1)), "codes")


def test_rmsnorm_rope_captures_without_warm_up(sdq_dev, oracle):
    """One pass needs no scratch: more rows than any stream has had are
    captured with no call before, and every replay equals the eager call."""
    import torch

    import sdq

    L, C, heads = 300_000, 256, 2
    print(f"[rowblock] capture L={L} C={C}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(3)
    src = torch.randn((L, C), generator=g, device=sdq_dev)
    w = torch.randn(C, generator=g, device=sdq_dev)
    cs = torch.randn((L, 64, 2), generator=g, device=sdq_dev)
    x = src.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        sdq.rmsnorm_rope_batch([(x, 0, w, cs)], C, heads)
    for rep in range(3):
        src.normal_(generator=g)
        x.copy_(src)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = src.clone()
        sdq.rmsnorm_rope_batch([(want, 0, w, cs)], C, heads)
        torch.cuda.synchronize()
        assert torch.equal(x, want), rep


@pytest.mark.parametrize("K", [4, 64])
def test_more_rows_than_one_grid_holds(sdq_dev, oracle, K):
    """Rows beyond one grid of 14-row workgroups: the first, those at its end and
    the last equal a call on them alone (4 columns: the two-kernel form)."""
    import torch

    import sdq

    M, n = 117_440_480 + 45, 99  # one launch's rows (whole 32-row fragments) and some
    print(f"[rowblock] rows M={M} K={K}", flush=True)
    parts = [slice(0, n), slice(117_440_480 - 60, 117_440_480 - 60 + n), slice(M - n, M)]
    x = torch.randn((M, K), device=sdq_dev)
    w, b = torch.randn(K, device=sdq_dev), torch.randn(K, device=sdq_dev)
    q, s = oracle.quant_rows(oracle.randn(4 * K, 13).reshape(4, K))
    lin = sdq.Weight.from_host(q, s)
    Y, Yn = torch.empty((M, 4), device=sdq_dev), torch.empty((n, 4), device=sdq_dev)
    sdq.qlinear_lnmod(lin, x, Y, w, b, 1e-6)
    for r in parts:
        sdq.qlinear_lnmod(lin, x[r].contiguous(), Yn, w, b, 1e-6)
        assert torch.equal(Y[r], Yn)
    del Y
    cs = torch.randn((1, 2, 2), device=sdq_dev).expand(M, 2, 2).contiguous()
    y = torch.empty_like(x)
    sdq.layernorm(x, y, w, b)
    for r in parts:
        want = torch.empty((n, K), device=sdq_dev)
        sdq.layernorm(x[r].contiguous(), want, w, b)
        assert torch.equal(y[r], want)
    y.copy_(x)
    sdq.rmsnorm_rope_batch([(y, 0, w, cs)], K, 1)
    for r in parts:
        want = x[r].clone()
        sdq.rmsnorm_rope_batch([(want, 0, w, cs[:n].contiguous())], K, 1)
        assert torch.equal(y[r], want)


@pytest.mark.parametrize("M,K", [(32768, 4), (32769, 4), (32769, 24), (32769, 28), (32769, 60),
                                 (32769, 64)])
def test_many_narrow_rows(sdq_dev, oracle, M, K):
    """Both sides of the row count and widths where the two-kernel form takes
    over, bit-exact against the oracle."""
    import torch

    import sdq

    print(f"[rowblock] narrow M={M} K={K}", flush=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(sdq_dev)  # noqa: E731
    x = _x(oracle, M, K, K)
    w, b = oracle.randn(K, 11), oracle.randn(K, 12)
    y = torch.empty((M, K), device=sdq_dev)
    sdq.layernorm(t(x), y, t(w), t(b), 1e-6)
    d = t(x)
    cs = oracle.rope_cs(np.random.default_rng(5).uniform(-3, 3, (M, 2)).astype(np.float32))
    sdq.rmsnorm_rope_batch([(d, 0, t(w), t(cs))], K, 1)
    torch.cuda.synchronize()
    assert_bitexact(y.cpu().numpy(), oracle.layernorm(x, 1e-6, w, b), "layernorm")
    assert_bitexact(d.cpu().numpy(), oracle.rope(oracle.rmsnorm(x, w, 1e-6), cs, 1), "rms + rope")
