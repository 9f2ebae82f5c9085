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


def _codebook(bcjr, kind, L, V):
    if kind == "hyb":
        lut = np.random.default_rng(L).standard_normal((512, 2)).astype(np.float32)
        return bcjr.make_hyb_codebook_gpu(lut, 9, L, "cuda")
    if kind == "1mad":
        return bcjr.make_1mad_codebook(L, "cuda")
    return torch.tensor(np.random.default_rng(L).standard_normal((1 << L, V)).astype(np.float32), device="cuda")


@pytest.mark.parametrize("op", ["forward", "entropy", "backward"])
@pytest.mark.parametrize("kind,L,k,V,N", [("hyb", 16, 2, 2, 12), ("table", 16, 2, 2, 12), ("hyb", 12, 2, 2, 20),
                                          ("1mad", 12, 2, 1, 24), ("1mad", 16, 2, 1, 16), ("table", 10, 1, 1, 32)])
def test_rounds_of_a_short_workspace(bcjr_mod, kind, L, k, V, N, op):
    """8 sequences (one of them NaN, each at its own T and g_logZ): a workspace for
    3 of their halves gives every output of the full one bit for bit, in rounds of
    3, 3 and 2; one of 8 slots, which 7 halves exhaust at most, runs one launch as
    one slot does, bit for bit, and within the tolerances of the parity tests of
    the halves."""
    from bcjr import _lib
    lib = _lib.load()
    B, kV = 8, k * V
    cb = _codebook(bcjr_mod, kind, L, V)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, k, V, torch.device("cuda"))
    rng = np.random.default_rng(L + N)
    x, g = (rng.standard_normal((B, N, V)).astype(np.float32) for _ in range(2))
    x[5, 3, 0] = np.nan
    T = np.array([0.05, 0.1, 0.2, 0.06, 0.5, 0.1, 0.3, 0.07], np.float32)
    gz = rng.standard_normal(B).astype(np.float32)
    xd, gd, Td, gzd = (torch.tensor(a, device="cuda") for a in (x, g, T, gz))
    prob = spec.problem(B, N, True)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    st, nt = (2 if op == "backward" else 1), 1 << (L - kV)
    full = ctypes.c_size_t(0)
    _lib.check(lib.bcjr_workspace_bytes(ctypes.byref(prob), 1 if op == "backward" else 0, ctypes.byref(full)), "ws")
    up = lambda b: (b + 255) // 256 * 256
    slot = up(N * nt * 4 * st)
    halves = slot + up(2 * st * nt * 4) + up(8 * (N + 2))
    copy = 4 * V << L if kind == "table" and kV == 4 else 0
    assert full.value >= copy + B * halves and 8 * slot < 8 * halves
    res = []
    for nbytes in (full.value, copy + 3 * halves, copy + B * slot, copy + slot):
        _say(f"{op} {kind} L={L} kV={kV}: workspace {nbytes}")
        ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
        out, z, H = (torch.full(s, 7.0, device="cuda") for s in ((B, N, V), (B,), (B, N)))
        if op == "backward":
            rc = lib.bcjr_backward(ctypes.byref(prob), xd.data_ptr(), Td.data_ptr(), _lib.ptr(table), None, gd.data_ptr(),
                                   gzd.data_ptr(), out.data_ptr(), ws.data_ptr(), nbytes, stream)
            got = [out]
        elif op == "entropy":
            rc = lib.bcjr_forward_entropy(ctypes.byref(prob), xd.data_ptr(), Td.data_ptr(), _lib.ptr(table), out.data_ptr(),
                                          z.data_ptr(), H.data_ptr(), ws.data_ptr(), nbytes, stream)
            got = [out, z, H]
        else:
            rc = lib.bcjr_forward(ctypes.byref(prob), xd.data_ptr(), Td.data_ptr(), _lib.ptr(table), out.data_ptr(),
                                  z.data_ptr(), ws.data_ptr(), nbytes, stream)
            got = [out, z]
        _lib.check(rc, op)
        torch.cuda.synchronize()
        got = [t.cpu().numpy() for t in got]
        for t in got:
            assert np.isnan(t[5]).all() and np.isfinite(np.delete(t, 5, 0)).all()
        res.append(got)
    for a, b in zip(res[0], res[1]):
        assert np.array_equal(a, b, equal_nan=True)
    for a, b in zip(res[2], res[3]):
        assert np.array_equal(a, b, equal_nan=True)
    tol = [1e-3] if op == "backward" else [1e-4, 1e-5, 1e-4]  # gradient; soft, log Z, entropy: the parity tests' bounds
    for a, b, t in zip(res[0], res[2], tol):
        assert max_rel(np.delete(a, 5, 0), np.delete(b, 5, 0)) < t


@pytest.mark.parametrize("N,B", [(2048, 1), (2048, 2), (256, 8)])
def test_noalloc_holds_its_slots_in_two_halves(bcjr_mod, N, B):
    """L = 16, kV = 2: one slot of 128 MiB, and eight of 16, run as bcjr_forward runs
    them, bit for bit and (8 sequences) in one round: with seven halves in a round it
    took two, about twice as long."""
    from bcjr import _lib
    lib = _lib.load()
    L = 16
    x = torch.randn(B, N, 1, device="cuda", generator=torch.Generator("cuda").manual_seed(N))
    T = torch.full((1,), 0.1, device="cuda")
    prob = _lib.Problem(L, 2, 1, B, N, _lib.CODE_3INST, 9, 0)
    n = ctypes.c_size_t(0)
    _lib.check(lib.bcjr_workspace_bytes(ctypes.byref(prob), 0, ctypes.byref(n)), "ws")
    ws = torch.empty(n.value, dtype=torch.uint8, device="cuda")
    out = [[torch.full_like(x, 7.0), torch.full((B,), 7.0, device="cuda")] for _ in range(2)]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(i):
        args = [ctypes.byref(prob), x.data_ptr(), T.data_ptr(), None, out[i][0].data_ptr(), out[i][1].data_ptr()]
        _lib.check(lib.bcjr_forward_noalloc(*args, stream) if i else
                   lib.bcjr_forward(*args, ws.data_ptr(), ws.numel(), stream), "forward")

    def ms(i):
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            run(i)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    _say(f"noalloc N={N} B={B}")
    run(0), run(1)
    torch.cuda.synchronize()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert torch.isfinite(out[1][0]).all()
    if B == 8:
        with_ws, without = ms(0), ms(1)
        _say(f"8 sequences: {with_ws:.3f} ms with a workspace, {without:.3f} ms without")
        assert without < 1.5 * with_ws


@pytest.mark.parametrize("L", [15, 16])
def test_low_temperature_tables_in_two_halves(bcjr_mod, oracle, L):
    """A table at k = 2, V = 1 and T below the low-temperature line (0.08): the parity
    bounds, and about the time of T = 0.1 (its codewords are held over the sweep
    there too; read again for every unit, forward and entropy took twice as long)."""
    from bcjr import ops
    cb = _codebook(bcjr_mod, "table", L, 1)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 2, 1, torch.device("cuda"))
    rng = np.random.default_rng(L)
    B, N = 4, 16
    x, g = (rng.standard_normal((B, N, 1)).astype(np.float32) for _ in range(2))
    xd, gd = (torch.tensor(a, device="cuda") for a in (x, g))
    for T in (0.06, 0.02):
        _say(f"table L={L} T={T}")
        soft, logZ = ops.forward(spec, xd, T, table)
        H = ops.forward_entropy(spec, xd, T, table)[2]
        d = ops.backward(spec, xd, T, table, gd)
        cb_np = cb.cpu().numpy()
        s_ref, z_ref = oracle.bcjr_forward(x, cb_np, T, L, 2)
        assert max_rel(soft.cpu().numpy(), s_ref) < 1e-4 and max_rel(logZ.cpu().numpy(), z_ref) < 1e-5
        assert max_rel(d.cpu().numpy(), oracle.bcjr_backward(x, cb_np, T, L, 2, g)) < 1e-3
        h_ref = oracle.marginal_entropy(x, cb_np, T, L, 2)
        assert np.abs(H.cpu().numpy() - h_ref).max() < 1e-4 * max(1.0, h_ref.max())

    x = torch.randn(8, 96, 1, device="cuda", generator=torch.Generator("cuda").manual_seed(L))

    def ms(f):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    for name, f in (("forward", ops.forward), ("entropy", ops.forward_entropy)):
        warm, low = ms(lambda: f(spec, x, 0.1, table)), ms(lambda: f(spec, x, 0.06, table))
        _say(f"{name} L={L}: {warm:.3f} ms at T = 0.1, {low:.3f} at T = 0.06")
        assert low < 1.5 * warm


# (k, V, L, code, op, N, sequences per 256 CUs up to which the batch runs in two halves; 0: never)
@pytest.mark.parametrize("k,V,L,code,op,N,top", [
    # a lane per output, 24 waves per CU where one launch fills its waves
    (1, 1, 11, "table", 0, 64, 128), (1, 1, 11, "table", 1, 64, 128), (1, 1, 10, "table", 0, 64, 384),
    (1, 1, 8, "table", 0, 64, 1536), (2, 1, 10, "1mad", 0, 64, 768), (2, 1, 10, "1mad", 1, 64, 768),
    (2, 1, 11, "1mad", 0, 64, 512), (1, 2, 11, "table", 0, 64, 384),
    # whole butterflies, codewords in registers or not
    (1, 2, 12, "table", 0, 64, 384), (1, 2, 12, "table", 1, 64, 384),
    (1, 2, 13, "table", 0, 64, 128), (1, 2, 13, "table", 1, 64, 128), (1, 2, 14, "table", 0, 64, 128),
    (2, 1, 16, "3inst", 0, 64, 128),
    # fewest steps
    (2, 1, 10, "1mad", 0, 15, 0), (2, 1, 10, "1mad", 0, 16, 768), (2, 1, 10, "1mad", 1, 7, 0), (2, 1, 10, "1mad", 1, 8, 768),
    (1, 1, 8, "table", 1, 15, 0), (2, 1, 16, "3inst", 1, 7, 0), (2, 1, 16, "3inst", 0, 8, 128), (4, 1, 14, "1mad", 0, 3, 0),
    (4, 1, 16, "1mad", 1, 4, 128)])
def test_where_two_halves_end(bcjr_mod, k, V, L, code, op, N, top):
    """The largest batch that runs in two halves, from the workspace the call asks
    for (the halves' state beside the slots; the forward's is also the entropy's,
    whose lines lie at or above it): past these lines, or below these steps,
    the halves were slower than one launch."""
    from bcjr import _lib
    lib = _lib.load()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    st, nt = op + 1, 1 << (L - k * V)
    up = lambda b: (b + 255) // 256 * 256
    halves = up(N * nt * 4 * st) + up(2 * st * nt * 4) + up(8 * (N + 2))
    kind = {"table": _lib.CODE_TABLE, "1mad": _lib.CODE_1MAD, "3inst": _lib.CODE_3INST}[code]
    top = top * cus // 256
    for B, expect in ((max(top, 1), top > 0), (top + 1, False)):
        rc, nbytes, _ = _query_seconds(lib, _lib.Problem(L, k, V, B, N, kind, 9, 0), op)
        _say(f"k={k} V={V} L={L} {code} op {op} N={N} B={B}: {nbytes} bytes")
        assert rc == 0 and (nbytes >= B * halves) == expect


@pytest.mark.parametrize("L,top", [(12, 128), (14, 96)])
def test_where_two_halves_end_for_a_table_of_two_components(bcjr_mod, L, top):
    """The plain forward's own line there: a sequence has the bits of a batch far past
    it from one sequence past it on, and not at it."""
    from bcjr import ops
    top = top * torch.cuda.get_device_properties(0).multi_processor_count // 256
    cb = _codebook(bcjr_mod, "table", L, 2)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, 1, 2, torch.device("cuda"))
    x = torch.randn(8 * top, 32, 2, device="cuda", generator=torch.Generator("cuda").manual_seed(L))
    _say(f"table V=2 L={L} forward around {top} sequences")
    far, at, past = (ops.forward(spec, x[:B], 0.1, table)[0][:top] for B in (8 * top, top, top + 1))
    assert torch.equal(far, past) and not torch.equal(far, at)
    assert max_rel(at.cpu().numpy(), far.cpu().numpy()) < 1e-4  # the parity bound of soft


@pytest.mark.parametrize("kind,k,V,L,B,same", [("hyb", 2, 2, 16, 2, True), ("table", 4, 1, 9, 700, True), ("1mad", 2, 1, 14, 4, True),
                                               ("1mad", 2, 1, 12, 1200, True), ("1mad", 2, 1, 14, 160, False)])
def test_diagnostics_give_the_forwards_soft_and_log_z(bcjr_mod, kind, k, V, L, B, same):
    """return_internals: soft and log Z are the plain forward's bit for bit, in two
    halves, at kV = 4 and in one launch below L = 14; from there on (kV = 2, V = 1) the
    plain forward of a large batch runs on twice the threads, and they agree to the
    parity bounds."""
    from bcjr import ops
    cb = _codebook(bcjr_mod, kind, L, V)
    spec, table = bcjr_mod.codes.resolve_codebook(cb, L, k, V, torch.device("cuda"))
    x = torch.randn(B, 16, V, device="cuda", generator=torch.Generator("cuda").manual_seed(B))
    _say(f"diagnostics {kind} L={L} kV={k * V} B={B}")
    soft, logZ = ops.forward(spec, x, 0.2, table)
    got = ops.forward_internals(spec, x, 0.2, table)
    if same:
        assert torch.equal(got[0], soft) and torch.equal(got[1], logZ)
    assert max_rel(got[0].cpu().numpy(), soft.cpu().numpy()) < 1e-4
    assert max_rel(got[1].cpu().numpy(), logZ.cpu().numpy()) < 1e-5
