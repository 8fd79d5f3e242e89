"""sdq_qlinear_host by pieces of rows: row counts that end a piece, leave a
rest of one row and wrap round the slots, every epilogue's extra inputs, a
residual updated in place, and an output that lies on the input, which must be
read whole first. Each result equals the device entry's bit for bit."""
import ctypes

import numpy as np
import pytest

from conftest import assert_bitexact

pytestmark = pytest.mark.gpu

K, N = 1540, 1284


def _device(sdq, dev, w, A, kind, bias=None, gate=None, resid=None):
    import torch

    t = lambda a: None if a is None else torch.from_numpy(a).to(dev)  # noqa: E731
    Y = torch.empty((A.shape[0], w.N), device=dev,
                    dtype=torch.int32 if kind == "acc" else torch.float32)
    sdq.qlinear(w, t(A), Y, kind=kind, bias=t(bias), gate=t(gate), resid=t(resid))
    torch.cuda.synchronize()
    return Y.cpu().numpy()


@pytest.mark.parametrize("M", [1, 92, 93, 97, 385, 1000, 2500])
@pytest.mark.parametrize("kind", ["none", "acc", "gated"])
def test_pieces(sdq_dev, M, kind):
    import sdq

    print(f"[host-pieces] M={M} {kind}", flush=True)
    rng = np.random.default_rng(M)
    q = rng.integers(-127, 128, size=(N, K), dtype=np.int8)
    s = (rng.random(N, dtype=np.float32) * 0.01 + 1e-3).astype(np.float32)
    w = sdq.Weight.from_host(q, s)
    A = rng.standard_normal((M, K)).astype(np.float32)
    kw = {}
    if kind != "acc":
        kw["bias"] = rng.standard_normal(N).astype(np.float32)
    if kind == "gated":
        kw["gate"] = rng.standard_normal(N).astype(np.float32)
        kw["resid"] = rng.standard_normal((M, N)).astype(np.float32)
    want = _device(sdq, sdq_dev, w, A, kind, **kw)
    assert_bitexact(sdq.qlinear_host(w, A, kind=kind, **kw), want, "host")
    if kind == "gated":  # x += in place, over the host array
        x = kw["resid"].copy()
        e = sdq.make_epilogue(kind, kw["bias"], kw["gate"], x, True)
        p = lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
        assert sdq.load_library().sdq_qlinear_host(w.h, p(A), M, K, ctypes.byref(e), p(x)) == 0
        assert_bitexact(x, want, "host in place")


def test_output_over_its_inputs(sdq_dev):
    """Y begins inside A (and inside the residual): rows written early must not
    change rows that are read late."""
    import sdq

    M, D = 1000, 1536
    rng = np.random.default_rng(3)
    q = rng.integers(-127, 128, size=(D, D), dtype=np.int8)
    s = (rng.random(D, dtype=np.float32) * 0.01 + 1e-3).astype(np.float32)
    w = sdq.Weight.from_host(q, s)
    buf = rng.standard_normal((M + 300, D)).astype(np.float32)
    p = lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
    lib = sdq.load_library()
    A = buf[:M].copy()
    want = _device(sdq, sdq_dev, w, A, "none")
    b = buf.copy()
    e = sdq.make_epilogue("none")
    assert lib.sdq_qlinear_host(w.h, p(b), M, D, ctypes.byref(e), p(b[300:])) == 0
    assert_bitexact(b[300:], want, "over A")
    x = buf[:M].copy()
    want = _device(sdq, sdq_dev, w, A, "resid", resid=x)
    b = buf.copy()
    e = sdq.make_epilogue("resid", None, None, b[:M], True)
    assert lib.sdq_qlinear_host(w.h, p(A), M, D, ctypes.byref(e), p(b[300:])) == 0
    assert_bitexact(b[300:], want, "over the residual")
