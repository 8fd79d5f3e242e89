"""sdq_sdpa's packed form at the edges of its key blocks (32), query groups
(256) and key shares, over V's element range, in chunks, and the form without
scratch under graph capture. Bound: 2e-5 of the output scale (the parity bound
of the attention against the oracle), of each output dimension's own scale
where V's magnitudes differ from dimension to dimension or key to key."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(sdq_dev, q, kv, heads, batch=1):
    import torch

    import sdq

    out = torch.full((q.shape[0], heads * 128), float("nan"), device=sdq_dev)
    sdq.sdpa(q, kv, kv, out, heads, kcol=0, vcol=heads * 128, batch=batch)
    torch.cuda.synchronize()
    return out


def _want64(q, kv, heads):
    """softmax(q k^T / sqrt(128)) v in float64, head by head."""
    import torch

    C = heads * 128
    out = torch.empty(q.shape[0], C, dtype=torch.float64, device=q.device)
    for h in range(heads):
        c = slice(128 * h, 128 * h + 128)
        s = q[:, c].double() @ kv[:, c].double().t().contiguous() / 128.0 ** 0.5
        out[:, c] = torch.softmax(s, 1) @ kv[:, C + 128 * h:C + 128 * h + 128].double().contiguous()
    return out


@pytest.mark.parametrize("Lq,Lk,heads", [
    (1, 1, 1), (255, 31, 2), (256, 32, 1), (257, 33, 2), (33, 64, 3), (5, 65, 1),
    (300, 191, 2), (300, 193, 2), (64, 1025, 5), (2900, 200, 24), (2816, 97, 24)])
def test_edges(sdq_dev, oracle, Lq, Lk, heads):
    """Partial last key blocks and query groups, ranges of one to many blocks,
    whole rounds of items with and without a rest cut into shares."""
    import torch

    print(f"[sdpa-packed] Lq={Lq} Lk={Lk} heads={heads}", flush=True)
    rng = np.random.default_rng(Lq + 31 * Lk)
    C = heads * 128
    q = (rng.standard_normal((Lq, C)) * 0.6).astype(np.float32)
    kv = rng.standard_normal((Lk, 2 * C)).astype(np.float32)
    got = _run(sdq_dev, torch.from_numpy(q).to(sdq_dev), torch.from_numpy(kv).to(sdq_dev), heads)
    got = got.cpu().numpy().astype(np.float64)
    want = oracle.sdpa(q, kv[:, :C], kv[:, C:], heads)
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("case", ["rows", "tiny", "huge", "zero_blocks", "far_logits", "inf"])
def test_value_range(sdq_dev, case):
    """V rows of 2^-12..2^12 in one block, V near the ends of float's range,
    blocks of zeros between blocks of small values, logits all far below 0
    (the padding keys of a last block would win if they counted), and an
    infinity, which reaches its own dimension only."""
    import torch

    print(f"[sdpa-packed] range {case}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(5)
    Lq, Lk, heads = 70, 300, 2
    C = heads * 128
    q = torch.randn((Lq, C), generator=g, device=sdq_dev)
    kv = torch.randn((Lk, 2 * C), generator=g, device=sdq_dev)
    v = kv[:, C:]
    bound = 2e-5
    if case == "rows":
        v *= torch.exp2(torch.randint(-12, 13, (Lk, 1), generator=g, device=sdq_dev).float())
    elif case == "tiny":
        v *= 2.0 ** -80
    elif case == "huge":
        v *= 2.0 ** 120
    elif case == "zero_blocks":
        v *= 2.0 ** -40
        v[64:128] = 0.0
        v[290:] = 0.0
    elif case == "far_logits":
        q.abs_()
        kv[:, :C] = -kv[:, :C].abs() * 30.0
        bound = 2e-4  # logits of ~-2000 carry 2^-24 of themselves: 1e-4 of a weight
    want = _want64(q, kv, heads)
    if case == "inf":
        v[17, 5] = float("inf")
    got = _run(sdq_dev, q, kv, heads).double()
    if case == "inf":
        assert not torch.isfinite(got[:, 5]).any()
        got[:, 5] = want[:, 5]
    scale = want.abs().max()
    assert torch.isfinite(got).all()
    err = float((got - want).abs().max() / scale)
    print(f"  max err {err:.3e}", flush=True)
    assert err <= bound


@pytest.mark.parametrize("Lq,Lk", [(70, 300), (70, 1024), (70, 5000), (60, 5000)])
@pytest.mark.parametrize("cut", [True, False])
@pytest.mark.parametrize("case", ["falling", "rising", "far_rows", "light_keys", "ignored",
                                  "outlier_dim", "outlier_element", "short_keys"])
def test_value_magnitudes(sdq_dev, monkeypatch, case, cut, Lq, Lk):
    """V of 2^40 and 2^-90, by halves with blocks of zeros in either order and
    row by row (the small keys count in the softmax's sum all the same); keys
    of 2^-20 of the weight whose V is 2^20 times larger; keys of no weight whose
    V is 2^100; a dimension 2^16 and an element 2^12 above the others; keys 2^30
    shorter than their neighbours, of all the weight. Every output dimension to
    its own scale, with the keys cut into shares and not."""
    import torch

    print(f"[sdpa-packed] magnitudes {case} Lq={Lq} Lk={Lk} cut={cut}", flush=True)
    if not cut:
        monkeypatch.setenv("SDQ_SDPA_SPLIT", "1")
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(9)
    heads = 2
    C = heads * 128
    q = torch.randn((Lq, C), generator=g, device=sdq_dev)
    kv = torch.randn((Lk, 2 * C), generator=g, device=sdq_dev)
    v = kv[:, C:]
    if case in ("falling", "rising"):
        first, second = (40, -90) if case == "falling" else (-90, 40)
        v[:Lk // 2] *= 2.0 ** first
        v[Lk // 2:] *= 2.0 ** second
        v[32:96] = 0.0
    elif case == "far_rows":
        v[0::2] *= 2.0 ** 40
        v[1::2] *= 2.0 ** -90
    elif case in ("light_keys", "ignored"):
        e = -20 if case == "light_keys" else -2000
        q[:, ::128] = 8.0
        kv[:, 0:C:128] = 0.0
        kv[1::3, 0:C:128] = e * np.log(2.0) * 128 ** 0.5 / 8
        v[1::3] *= 2.0 ** (20 if case == "light_keys" else 100)
    elif case == "outlier_dim":
        v[:, 7] *= 2.0 ** 16
    elif case == "short_keys":
        q.abs_()
        kv[1::2, :C] = -kv[1::2, :C].abs() * 2.0 ** 30
        v[32:64] = 0.0
    else:
        v[17, 5] *= 2.0 ** 12
    want = _want64(q, kv, heads)
    got = _run(sdq_dev, q, kv, heads).double()
    assert torch.isfinite(got).all()
    err = ((got - want).abs().amax(0) / want.abs().amax(0)).max()
    print(f"  max err of a dimension {float(err):.3e}", flush=True)
    assert err <= 2e-5


@pytest.mark.parametrize("Lq,Lk,heads", [(1, 4097, 1), (31, 4128, 5), (33, 8191, 3),
                                         (64, 4129, 24), (64, 20001, 2), (65, 4129, 2),
                                         (64, 4096, 2)])
def test_few_queries(sdq_dev, Lq, Lk, heads):
    """At most 64 queries over more than 4096 keys: key ranges that end in a
    partial block, partial and whole query groups, and two stacked sequences
    with the bits of two separate calls. To the packed form's precision."""
    import torch

    print(f"[sdpa-packed] few Lq={Lq} Lk={Lk} heads={heads}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(Lq + Lk)
    q = torch.randn((2 * Lq, 128 * heads), generator=g, device=sdq_dev)
    kv = torch.randn((2 * Lk, 256 * heads), generator=g, device=sdq_dev)
    both = _run(sdq_dev, q, kv, heads, batch=2)
    for b in range(2):
        qs, ks = q[b * Lq:(b + 1) * Lq], kv[b * Lk:(b + 1) * Lk]
        one = _run(sdq_dev, qs, ks, heads)
        assert torch.equal(both[b * Lq:(b + 1) * Lq], one)
        want = _want64(qs, ks, heads)
        err = float((one.double() - want).norm() / want.norm())
        print(f"  err {err:.3e}", flush=True)
        assert err <= 2e-6  # float sums of up to 20001 terms; the two-part products alone 4e-6


def test_chunks(sdq_dev):
    """More keys than one launch's scratch holds for two heads: one launch
    per head; two stacked sequences give the bits of two separate calls."""
    import torch

    L, heads = 1_100_000, 2
    print(f"[sdpa-packed] chunks Lk={L}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(6)
    q = torch.randn((2 * 40, 256), generator=g, device=sdq_dev)
    kv = torch.randn((2 * L, 512), generator=g, device=sdq_dev)
    got = _run(sdq_dev, q, kv, heads, batch=2)
    for b in range(2):
        qs, ks = q[40 * b:40 * b + 40], kv[b * L:(b + 1) * L]
        one = _run(sdq_dev, qs, ks, heads)
        assert torch.equal(got[40 * b:40 * b + 40], one)
        want = _want64(qs, ks, heads)
        assert float((one.double() - want).abs().max() / want.abs().max()) <= 2e-5


def test_ragged_head_chunks(sdq_dev):
    """Heads that the launches' scratch does not divide: the last launch has
    fewer, and its own plan."""
    import torch

    Lq, Lk, heads = 70, 600_000, 5
    print(f"[sdpa-packed] head chunks Lk={Lk} heads={heads}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(8)
    q = torch.randn((Lq, 128 * heads), generator=g, device=sdq_dev)
    kv = torch.randn((Lk, 256 * heads), generator=g, device=sdq_dev)
    got = _run(sdq_dev, q, kv, heads)
    want = _want64(q, kv, heads)
    assert float((got.double() - want).abs().max() / want.abs().max()) <= 2e-5


def test_capture_without_warm_up(sdq_dev):
    """A capture on a stream whose workspace cannot grow any more takes the
    form without scratch; replays see new inputs."""
    import torch

    import sdq

    g = torch.Generator(device=sdq_dev)
    g.manual_seed(7)
    q = torch.randn((300, 256), generator=g, device=sdq_dev)
    kv = torch.randn((500, 512), generator=g, device=sdq_dev)
    out = torch.empty((300, 256), device=sdq_dev)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        sdq.sdpa(q, kv, kv, out, 2, kcol=0, vcol=256)
    for _ in range(3):
        q.copy_(torch.randn((300, 256), generator=g, device=sdq_dev))
        graph.replay()
        torch.cuda.synchronize()
        want = _want64(q, kv, 2)
        assert float((out.double() - want).abs().max() / want.abs().max()) <= 2e-5


def test_fallback_leaves_no_error_text(sdq_dev):
    """A call that does without its scratch (a capture whose workspace would
    have to grow) succeeds, and the thread's last error stays the one before."""
    import torch

    import sdq

    print("[sdpa-packed] error text", flush=True)
    q = torch.zeros((40, 384), device=sdq_dev)
    kv = torch.zeros((120_000, 768), device=sdq_dev)  # more than any stream has had
    out = torch.empty((40, 384), device=sdq_dev)
    torch.cuda.synchronize()
    lib = sdq.load_library()
    assert lib.sdq_add(None, None, -1, None) != 0
    before = lib.sdq_last_error()
    assert before
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        sdq.sdpa(q, kv, kv, out, 3, kcol=0, vcol=384)
    assert lib.sdq_last_error() == before


@pytest.mark.parametrize("shared", [True, False])
def test_threads_on_one_stream(sdq_dev, shared):
    """Four threads with their own inputs on one stream, sizes that grow the
    workspace among them: every result equals the call alone. The same on the
    per-thread stream, one handle for a stream of each thread."""
    import threading

    import torch

    import sdq

    print(f"[sdpa-packed] threads shared={shared}", flush=True)
    g = torch.Generator(device=sdq_dev)
    g.manual_seed(12)
    heads, C = 3, 384
    sizes = [1100, 1500, 2300, 150_000]
    xs = [torch.randn((min(n, 1500), C), generator=g, device=sdq_dev) for n in sizes]
    kvs = [torch.randn((n, 2 * C), generator=g, device=sdq_dev) for n in sizes]
    own = torch.cuda.Stream()
    s = own if shared else 2  # hipStreamPerThread
    torch.cuda.synchronize()
    outs = [[torch.zeros_like(x) for _ in range(8)] for x in xs]
    torch.cuda.synchronize()
    go = threading.Barrier(len(sizes))

    def run(i):
        sdq.init(0)
        go.wait()
        for out in outs[i]:
            sdq.sdpa(xs[i], kvs[i], kvs[i], out, heads, kcol=0, vcol=C, stream=s)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, x in enumerate(xs):
        want = torch.zeros_like(x)
        sdq.sdpa(x, kvs[i], kvs[i], want, heads, kcol=0, vcol=C, stream=own)
        own.synchronize()
        for out in outs[i]:
            assert torch.equal(out, want), sizes[i]
