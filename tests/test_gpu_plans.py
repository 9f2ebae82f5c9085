"""Launch plans of the soft calls (csrc/bcjr_capi.hip): what they cost the host, which
calls run in two halves, and what a workspace that holds part of the batch gives."""
import ctypes
import time

import numpy as np
import pytest
import torch

from conftest import max_rel

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[plans] {msg}", flush=True)


def _query_seconds(lib, prob, op):
    n = ctypes.c_size_t(0)
    t0 = time.perf_counter()
    rc = lib.bcjr_workspace_bytes(ctypes.byref(prob), op, ctypes.byref(n))
    return rc, n.value, time.perf_counter() - t0


def test_shape_whose_halves_do_not_fit_is_planned_once(bcjr_mod, oracle):
    """Backward, L = 15, k = 2, N = 2100: the two-halves state and offsets exceed
    the LDS, so the call runs in one launch.  A second query does no layout search
    (11 to 55 ms), a success leaves the last error alone, and a new N of the same L
    searches nothing again."""
    from bcjr import _lib, ops
    lib = _lib.load()
    L, N, B = 15, 2100, 2
    prob = _lib.Problem(L, 2, 1, B, N, _lib.CODE_1MAD, 9, 0)
    bad = _lib.Problem(L, 3, 1, B, N, _lib.CODE_1MAD, 9, 0)
    _say(f"backward L={L} N={N}: workspace queries")
    assert _query_seconds(lib, prob, 1)[0] == 0
    assert _query_seconds(lib, bad, 1)[0] == _lib.BCJR_EUNSUPPORTED
    said = lib.bcjr_last_error()
    took = []
    for _ in range(3):
        rc, nbytes, dt = _query_seconds(lib, prob, 1)
        assert rc == 0 and nbytes == B * N * (2 << (L - 2)) * 4
        took.append(dt)
    _say(f"repeated query {min(took) * 1e3:.3f} ms")
    assert min(took) < 0.003
    for op, kv4 in ((1, False), (0, False), (0, True)):
        other = [_lib.Problem(L, 4 if kv4 else 2, 1, B, 1000 + i, _lib.CODE_1MAD, 9, 0) for i in range(4)]
        dts = [_query_seconds(lib, p, op)[2] for p in other]
        _say(f"first query of a new N, op {op}, kV {4 if kv4 else 2}: {min(dts[1:]) * 1e3:.3f} ms")
        assert min(dts[1:]) < 0.003
    assert lib.bcjr_last_error() == said

    cb = bcjr_mod.make_1mad_codebook(L, "cuda")
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 2, 1, torch.device("cuda"))
    rng = np.random.default_rng(15)
    x, g = (rng.standard_normal((B, N, 1)).astype(np.float32) for _ in range(2))
    _say(f"backward L={L} N={N}")
    d = ops.backward(spec, torch.tensor(x, device="cuda"), 0.2, table, torch.tensor(g, device="cuda"))
    ref = oracle.bcjr_backward(x, cb.cpu().numpy(), 0.2, L, 2, g)
    assert max_rel(d.cpu().numpy(), ref) < 1e-3  # the parity bound of the gradient
