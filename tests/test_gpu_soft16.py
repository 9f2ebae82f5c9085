"""The kV = 4 soft kernels (csrc/bcjr_soft16.h) at the edges of their launch rules,
against the float64 oracle: every L, odd and tiny N, batches on both sides of
the two-halves rule, and workspaces that hold no transposed table or only part
of the batch.  Tolerances are those of the other parity tests (float32
log-domain recursions: soft 1e-4, gradient 1e-3, log Z 1e-5, entropy 1e-4)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SOFT_TOL, GRAD_TOL, Z_TOL = 1e-4, 1e-3, 1e-5


def _codebook(bcjr, kind, L, V, seed):
    rng = np.random.default_rng(seed)
    if kind == "hyb":
        return bcjr.make_hyb_codebook_gpu(rng.standard_normal((512, 2)).astype(np.float32), 9, L, "cuda")
    if kind == "3inst":
        return bcjr.make_3inst_codebook(L, "cuda")
    if kind == "1mad":
        return bcjr.make_1mad_codebook(L, "cuda")
    return torch.tensor(rng.standard_normal((1 << L, V)).astype(np.float32), device="cuda")


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _check(bcjr, oracle, kind, L, V, N, B, T, rows):
    from bcjr import ops
    k = 4 // V
    cb = _codebook(bcjr, kind, L, V, L + N)
    spec, table = bcjr.codes.resolve_codebook(cb, L, k, V, torch.device("cuda"))
    rng = np.random.default_rng(100 * L + N)
    x = rng.standard_normal((B, N, V)).astype(np.float32)
    g = rng.standard_normal((B, N, V)).astype(np.float32)
    gz = rng.standard_normal(B).astype(np.float32)
    xd = torch.tensor(x, device="cuda")
    soft, logZ = ops.forward(spec, xd, T, table)
    soft_e, logZ_e, H = ops.forward_entropy(spec, xd, T, table)
    d = ops.backward(spec, xd, T, table, torch.tensor(g, device="cuda"), torch.tensor(gz, device="cuda"))
    cb_np, rows = cb.cpu().numpy(), [r for r in rows if r < B]
    s_ref, z_ref = oracle.bcjr_forward(x[rows], cb_np, T, L, 4)
    d_ref = oracle.bcjr_backward(x[rows], cb_np, T, L, 4, g[rows], gz[rows])
    h_ref = oracle.marginal_entropy(x[rows], cb_np, T, L, 4)
    assert _rel(soft.cpu().numpy()[rows], s_ref) < SOFT_TOL
    assert _rel(logZ.cpu().numpy()[rows], z_ref) < Z_TOL
    assert _rel(d.cpu().numpy()[rows], d_ref) < GRAD_TOL
    assert np.abs(H.cpu().numpy()[rows] - h_ref).max() < 1e-4 * max(1.0, h_ref.max())
    assert _rel(soft_e.cpu().numpy()[rows], s_ref) < SOFT_TOL and torch.isfinite(d).all()


@pytest.mark.parametrize("kind,V", [("hyb", 2), ("table", 2), ("table", 1), ("3inst", 1), ("1mad", 1)])
@pytest.mark.parametrize("L,N,T", [(8, 1, 0.3), (9, 2, 0.06), (10, 3, 0.3), (11, 37, 0.1), (12, 16, 0.06), (13, 5, 0.2),
                                   (14, 4, 0.06), (15, 9, 0.1), (16, 1, 0.2), (16, 2, 0.05), (16, 7, 0.1),
                                   (9, 6, 0.06), (10, 4, 0.3), (16, 4, 0.05)])
def test_every_L_and_short_N(bcjr_mod, oracle, kind, V, L, N, T):
    print(f"[soft16] {kind} V={V} L={L} N={N} T={T}", flush=True)
    _check(bcjr_mod, oracle, kind, L, V, N, 3, T, [0, 1, 2])


# 256 CUs: two halves on the wide column-walk workgroup up to 128, on the narrow
# one up to half of what is resident, then one launch.
@pytest.mark.parametrize("kind,V,L,B", [("hyb", 2, 16, 128), ("hyb", 2, 16, 129), ("hyb", 2, 16, 256), ("hyb", 2, 16, 257),
                                        ("hyb", 2, 16, 600), ("table", 2, 16, 128), ("table", 2, 16, 129),
                                        ("3inst", 1, 16, 300), ("hyb", 2, 12, 700), ("table", 1, 10, 2100)])
@pytest.mark.parametrize("T", [0.06, 0.25])
def test_batches_around_the_two_halves_rule(bcjr_mod, oracle, kind, V, L, B, T):
    print(f"[soft16] {kind} L={L} B={B} T={T}", flush=True)
    _check(bcjr_mod, oracle, kind, L, V, 6, B, T, [0, 127, 128, 255, 256, 299, 599, 2099])


@pytest.mark.parametrize("kind,V", [("hyb", 2), ("table", 2)])
def test_short_workspaces(bcjr_mod, oracle, kind, V):
    """One slot only (no room for the meeting vectors or the table copy: whole
    sequences, the table as it is), room for 3 of 8 sequences (three rounds of
    halves, the same bits as one round), and the full workspace; a NaN sequence
    and per-sequence T among them."""
    from bcjr import _lib
    lib = _lib.load()
    L, N, B = 16, 12, 8
    cb = _codebook(bcjr_mod, kind, L, V, 3)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 4 // V, V, torch.device("cuda"))
    rng = np.random.default_rng(5)
    x = rng.standard_normal((B, N, V)).astype(np.float32)
    g = rng.standard_normal((B, N, V)).astype(np.float32)
    T = np.array([0.05, 0.1, 0.2, 0.06, 0.5, 0.1, 0.3, 0.07], np.float32)
    x[5, 3, 0] = np.nan
    xd, gd, Td = (torch.tensor(a, device="cuda") for a in (x, g, T))
    prob = spec.problem(B, N, True)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    nt = 1 << (L - 4)
    outs = []
    for op, st in ((0, 1), (1, 2)):
        full = ctypes.c_size_t(0)
        _lib.check(lib.bcjr_workspace_bytes(ctypes.byref(prob), op, ctypes.byref(full)), "ws")
        slot = N * nt * 4 * st
        per = slot + 2 * nt * 4 * st + 256
        copy = 4 * V << L if kind == "table" else 0
        res = []
        for nbytes in (full.value, copy + 3 * per, slot):
            print(f"[soft16] {kind} op {op} workspace {nbytes}", flush=True)
            ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
            out, z = torch.full((B, N, V), 7.0, device="cuda"), torch.full((B,), 7.0, device="cuda")
            if op == 0:
                rc = lib.bcjr_forward(ctypes.byref(prob), xd.data_ptr(), Td.data_ptr(), _lib.ptr(table), out.data_ptr(),
                                      z.data_ptr(), ws.data_ptr(), nbytes, stream)
            else:
                rc = lib.bcjr_backward(ctypes.byref(prob), xd.data_ptr(), Td.data_ptr(), _lib.ptr(table), None,
                                       gd.data_ptr(), None, out.data_ptr(), ws.data_ptr(), nbytes, stream)
            _lib.check(rc, "call")
            torch.cuda.synchronize()
            assert torch.isnan(out[5]).all()
            res.append(out.cpu().numpy())
        assert np.array_equal(res[0], res[1], equal_nan=True)
        outs.append(res)
    rows = [0, 1, 2, 3, 4, 6, 7]
    cb_np = cb.cpu().numpy()
    for r in rows:
        s_ref, _ = oracle.bcjr_forward(x[r:r + 1], cb_np, float(T[r]), L, 4)
        d_ref = oracle.bcjr_backward(x[r:r + 1], cb_np, float(T[r]), L, 4, g[r:r + 1])
        for i in (0, 2):
            assert _rel(outs[0][i][r], s_ref[0]) < SOFT_TOL and _rel(outs[1][i][r], d_ref[0]) < GRAD_TOL


@pytest.mark.parametrize("kind,k,V,L,N", [("table", 1, 1, 2, 5), ("table", 1, 1, 7, 64), ("table", 1, 1, 11, 33),
                                          ("3inst", 2, 1, 4, 2), ("1mad", 2, 1, 6, 3), ("table", 2, 1, 9, 17),
                                          ("3inst", 2, 1, 12, 40), ("1mad", 2, 1, 13, 21), ("3inst", 2, 1, 14, 8),
                                          ("table", 2, 1, 15, 9), ("3inst", 2, 1, 16, 11), ("1mad", 2, 1, 16, 1),
                                          ("hyb", 1, 2, 8, 7), ("table", 1, 2, 12, 30), ("hyb", 1, 2, 13, 5),
                                          ("table", 1, 2, 15, 4), ("hyb", 1, 2, 16, 6),
                                          # (from the fewest steps that take two halves on)
                                          ("table", 1, 1, 2, 18), ("table", 1, 1, 4, 16), ("3inst", 2, 1, 4, 17),
                                          ("1mad", 2, 1, 6, 16), ("hyb", 1, 2, 8, 23), ("hyb", 1, 2, 13, 17),
                                          ("table", 1, 2, 15, 12), ("table", 2, 1, 16, 8)])
@pytest.mark.parametrize("T", [0.06, 0.2])
def test_small_steps_in_two_halves(bcjr_mod, oracle, kind, k, V, L, N, T):
    """kV <= 2 (csrc/bcjr_halves.h): every L's launch shape, odd and even N, a
    table, hashed codes and the LUT."""
    from bcjr import ops
    print(f"[halves] {kind} k={k} V={V} L={L} N={N} T={T}", flush=True)
    cb = _codebook(bcjr_mod, kind, L, V, L + N)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, k, V, torch.device("cuda"))
    rng, B = np.random.default_rng(L * 7 + N), 3
    x = rng.standard_normal((B, N, V)).astype(np.float32)
    g = rng.standard_normal((B, N, V)).astype(np.float32)
    gz = rng.standard_normal(B).astype(np.float32)
    Tv = np.array([T, 0.5, 0.1], np.float32)
    xd, Td = torch.tensor(x, device="cuda"), torch.tensor(Tv, device="cuda")
    soft, logZ = ops.forward(spec, xd, Td, table)
    _, _, H = ops.forward_entropy(spec, xd, Td, table)
    d = ops.backward(spec, xd, Td, table, torch.tensor(g, device="cuda"), torch.tensor(gz, device="cuda"))
    cb_np = cb.cpu().numpy()
    for r in range(B):
        s_ref, z_ref = oracle.bcjr_forward(x[r:r + 1], cb_np, float(Tv[r]), L, k * V)
        d_ref = oracle.bcjr_backward(x[r:r + 1], cb_np, float(Tv[r]), L, k * V, g[r:r + 1], gz[r:r + 1])
        h_ref = oracle.marginal_entropy(x[r:r + 1], cb_np, float(Tv[r]), L, k * V)
        assert _rel(soft.cpu().numpy()[r], s_ref[0]) < SOFT_TOL and _rel(logZ.cpu().numpy()[r], z_ref[0]) < Z_TOL
        assert _rel(d.cpu().numpy()[r], d_ref[0]) < GRAD_TOL
        assert np.abs(H.cpu().numpy()[r] - h_ref[0]).max() < 1e-4 * max(1.0, h_ref.max())


@pytest.mark.parametrize("B", [128, 129])
def test_sequences_beside_each_other_in_two_halves(bcjr_mod, oracle, B):
    """The largest batch two halves take at L = 16 (one workgroup per CU) and the
    smallest one launch takes: first, middle and last sequence."""
    from bcjr import ops
    print(f"[halves] 3inst L=16 B={B}", flush=True)
    L, N, T = 16, 10, 0.1
    cb = bcjr_mod.make_3inst_codebook(L, "cuda")
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 2, 1, torch.device("cuda"))
    rng = np.random.default_rng(B)
    x, g = (rng.standard_normal((B, N, 1)).astype(np.float32) for _ in range(2))
    xd = torch.tensor(x, device="cuda")
    soft, _ = ops.forward(spec, xd, T, table)
    d = ops.backward(spec, xd, T, table, torch.tensor(g, device="cuda"))
    rows = [0, 64, B - 1]
    assert _rel(soft.cpu().numpy()[rows], oracle.bcjr_forward(x[rows], cb.cpu().numpy(), T, L, 2)[0]) < SOFT_TOL
    assert _rel(d.cpu().numpy()[rows], oracle.bcjr_backward(x[rows], cb.cpu().numpy(), T, L, 2, g[rows])) < GRAD_TOL


@pytest.mark.parametrize("L,k,V,N", [(16, 2, 2, 9), (14, 2, 2, 6), (9, 4, 1, 5)])
def test_viterbi_table_with_and_without_its_copy(bcjr_mod, oracle, L, k, V, N):
    """kV = 4 tables: the full workspace (transposed copy) and one slot (the table
    as it is) give the oracle's walks, with ties (a table of few values), a NaN
    and an infinite weight among the sequences."""
    from bcjr import _lib
    lib = _lib.load()
    B = 5
    rng = np.random.default_rng(L)
    cb_np = np.round(2 * rng.standard_normal((1 << L, V))).astype(np.float32) / 2
    x = np.round(rng.standard_normal((B, N, V)) * 4).astype(np.float32) / 4
    x[3, 1, 0], x[4, 2, V - 1] = np.nan, np.inf
    cb, xd = torch.tensor(cb_np, device="cuda"), torch.tensor(x, device="cuda")
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, k, V, torch.device("cuda"))
    prob = spec.problem(B, N)
    full = ctypes.c_size_t(0)
    _lib.check(lib.bcjr_workspace_bytes(ctypes.byref(prob), 2, ctypes.byref(full)), "ws")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    walk_ref = oracle.viterbi(x[:3], cb_np, L, 4)[0]
    slot = (N * (1 << (L - 4)) + 255) // 256 * 256
    res = []
    for nbytes in (full.value, slot):
        print(f"[viterbi] table L={L} k={k} V={V} workspace {nbytes}", flush=True)
        ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
        walk = torch.full((B, N), -1, dtype=torch.int32, device="cuda")
        mse = torch.zeros(B, device="cuda")
        _lib.check(lib.bcjr_viterbi(ctypes.byref(prob), xd.data_ptr(), _lib.ptr(table), walk.data_ptr(), None, None, None,
                                    mse.data_ptr(), None, ws.data_ptr(), nbytes, stream), "viterbi")
        torch.cuda.synchronize()
        assert np.array_equal(walk.cpu().numpy()[:3], walk_ref)
        assert torch.isnan(mse[3]) and torch.isinf(mse[4])
        res.append(walk.cpu().numpy())
    assert np.array_equal(res[0], res[1]) and res[0].min() >= 0 and res[0].max() < 1 << L


@pytest.mark.parametrize("kind,B,bound", [("hyb", 600, 1.85e-5), ("table", 300, 1.08e-5)])
def test_gradient_keeps_its_precision_beside_a_large_expected_path_value(bcjr_mod, oracle, kind, B, bound):
    """Weights about 2 and upstream gradients about 4: E[F] is about 128, which is
    taken off path values as large, and a rounding of E[F] beyond its last one shows
    in the whole gradient.  Relative error (2-norm) against the float64 oracle; the
    bound lies halfway between float sums of E[F] (2.23e-5 hyb, 1.33e-5 table) and
    sums in double (1.48e-5 and 0.82e-5)."""
    from bcjr import ops
    print(f"[soft16] {kind} B={B}, large E[F]", flush=True)
    L, N, V, T = 16, 8, 2, 0.2
    cb = _codebook(bcjr_mod, kind, L, V, 16)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 2, V, torch.device("cuda"))
    rng = np.random.default_rng(3)
    x = (2 + 0.2 * rng.standard_normal((B, N, V))).astype(np.float32)
    g = (4 + 0.1 * rng.standard_normal((B, N, V))).astype(np.float32)
    d = ops.backward(spec, torch.tensor(x, device="cuda"), T, table, torch.tensor(g, device="cuda"))
    ref = oracle.bcjr_backward(x, cb.cpu().numpy(), T, L, 4, g)
    err = float(np.linalg.norm(d.cpu().numpy() - ref) / np.linalg.norm(ref))
    print(f"[soft16] {kind}: {err:.3e}", flush=True)
    assert err < bound
