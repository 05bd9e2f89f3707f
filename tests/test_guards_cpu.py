"""What the decode path refuses on the host, before any kernel is launched."""
import subprocess
import types

import pytest
import torch

from openattention_amd import ops
from openattention_amd.method import RMAX, OursHIP


def test_rows_step_refuses_keys_past_the_cache():
    """A multi-row call over more keys than the index or the cache holds, or over a cache of another
    shape, is refused on the host (the kernels read positions up to n_keys - 1 unchecked)."""
    B, Lmax, Q = 1, 512, 4
    m = OursHIP(types.SimpleNamespace(rho=0.01), B, Lmax, "cpu", n_layers=1)
    q = torch.zeros(B, 32, Q, 128, dtype=torch.bfloat16)
    out = torch.empty_like(q)
    n_dev = torch.zeros(1, dtype=torch.int32)

    def rows(kv, n_keys, v=None):
        K = torch.zeros(kv, dtype=torch.bfloat16)
        return m.rows_step(m.st[0], K, K if v is None else torch.zeros(v, dtype=torch.bfloat16), q, n_dev, n_keys, out)

    for args in (((8, Lmax + 64, 128), Lmax + 1), ((8, 300, 128), 301), ((4, Lmax, 128), 300),
                 ((8, Lmax, 128), 300, (8, Lmax - 1, 128)), ((8, Lmax, 128), 0)):
        with pytest.raises(ValueError, match="n_keys|K, V"):
            rows(*args)
    assert int(n_dev) == 0


def _moved(ns, name):
    """A copy of the namespace with one tensor on the host."""
    t = getattr(ns, name)
    return types.SimpleNamespace(**{**vars(ns), name: torch.empty(t.shape, dtype=t.dtype, device="cpu")})


@pytest.mark.parametrize("rows", [False, True])
def test_step_refuses_tensors_on_another_device(rows):
    """A step whose index, work buffers or row statistics are not on the keys' device raises for each of
    its tensors before a pointer is taken (stand-in device tensors, which have no pointer to take)."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    ns, nl, k, Lmax = 1, 1, 2, 256
    with FakeTensorMode():
        m = OursHIP(types.SimpleNamespace(rho=0.01), 1, Lmax, "cuda", n_layers=1)
        m.TMn = torch.empty_like(m.TM)
        st = types.SimpleNamespace(**vars(m.st[0]))
        w = types.SimpleNamespace(**{f: getattr(m, f) for f in ("limbs", "fexp", "H", "TM", "TMn", "S", "score", "n_t",
                                                                "quota", "qsk", "exp_idx")})
        K = torch.empty(8, Lmax, 128, device="cuda", dtype=torch.bfloat16)
        q = torch.empty(32, 128, device="cuda", dtype=torch.bfloat16)
        sel = torch.empty(32, ns + nl + k, device="cuda", dtype=torch.int32)
        n_dev = torch.empty(1, device="cuda", dtype=torch.int32)
        stats = {f: torch.empty_like(getattr(st, f)) for f in ("nb", "Sk", "Sk2", "Sv")} if rows else {}

        def call(st=st, w=w, stats=stats):
            ops.step(K, K, st, n_dev, q, w, sel, m.out, ns, nl, k, 0.1, m.E, RMAX, update=not rows, later=int(rows),
                     stats=tuple(stats.values()) or None)

        used = ["codes", "U", "scale", "asg", "asg8", "nb", "Sk", "Sk2", "Sv"]
        used += [] if rows else ["W", "colmean", "cent", "reclist", "reccnt"]
        for f in used:
            with pytest.raises(RuntimeError, match="HIP device"):
                call(st=_moved(st, f))
        for f in vars(w):
            with pytest.raises(RuntimeError, match="HIP device"):
                call(w=_moved(w, f))
        for f in stats:
            with pytest.raises(RuntimeError, match="HIP device"):
                call(stats={**stats, f: torch.empty(stats[f].shape, device="cpu")})


def test_step_over_a_cache_longer_than_its_index():
    """One row without an index update over K, V rows longer than the index's capacity passes the checks;
    an update, or question rows, which reach the keys' positions, are refused."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    calls = []
    with FakeTensorMode(), pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, "_stream", lambda dev: 0)
        mp.setattr(ops.lib, "call", lambda name, *a: calls.append(name))
        m = OursHIP(types.SimpleNamespace(rho=0.01), 1, 256, "cuda", n_layers=1)
        st = m.st[0]
        K = torch.empty(8, 320, 128, device="cuda", dtype=torch.bfloat16)
        q = torch.empty(32, 128, device="cuda", dtype=torch.bfloat16)
        sel = torch.empty(32, 4, device="cuda", dtype=torch.int32)
        n_dev = torch.empty(1, device="cuda", dtype=torch.int32)
        stats = (st.nb, st.Sk, st.Sk2, st.Sv)

        def call(**kw):
            ops.step(K, K, st, n_dev, q, m, sel, m.out, 1, 1, 2, 0.1, m.E, RMAX, **kw)

        call(update=False)
        assert calls == ["oa_step"]
        for kw in (dict(update=True), dict(update=False, later=1, stats=stats)):
            with pytest.raises(ValueError, match="asg"):
                call(**kw)


def test_question_rows_are_grouped_where_a_group_holds_two():
    """Rows per launch of a multi-row call: the largest power of two that 1024 query-head rows and the
    call hold; a batch that leaves one row to a launch runs its rows one after the other in place."""
    for B, want in ((1, 5), (2, 4), (3, 3), (8, 2), (16, 1), (17, 0), (32, 0)):
        m = OursHIP(types.SimpleNamespace(rho=0.01), B, 128, "meta", n_layers=1)
        assert m._rows_shift(64) == want
        assert [m._rows_shift(Q) for Q in (1, 2, 3)] == [0, min(want, 1), min(want, 1)]
    for kw in (dict(fused=False), dict(gate_mode="separate")):
        assert OursHIP(types.SimpleNamespace(rho=0.01), 1, 128, "meta", n_layers=1, **kw)._rows_shift(64) == 0

    m = OursHIP(types.SimpleNamespace(rho=0.01), 32, 128, "cpu", n_layers=1)
    ran = []
    m.step = lambda st, K, V, q, n_dev, n, counts, update_index: ran.append(n) or m.out
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, "index_downdate", lambda K, V, st, n_dev: ran.append("back"))
        K = torch.zeros(256, 128, 128, dtype=torch.bfloat16)
        q = torch.zeros(32, 32, 3, 128, dtype=torch.bfloat16)
        m.rows_step(m.st[0], K, K, q, torch.zeros(1, dtype=torch.int32), 128, torch.empty_like(q))
    assert ran == [128, "back", 127, "back", 126]


@pytest.mark.parametrize("rho,Lmax", [(0.01, 32896), (0.10, 32896), (0.01, 131200), (0.10, 131200), (0.01, 262144)])
def test_question_rows_work_buffers_are_bounded(rho, Lmax):
    """What a group of question rows allocates stays within its bound whatever the index's capacity, in
    the largest group that does."""
    from openattention_amd import method as M
    m = OursHIP(types.SimpleNamespace(rho=rho), 1, Lmax, "meta", n_layers=1)
    sh = m._rows_shift(64)
    got = []

    def bytes_of(st, K, V, n_dev, q, w, sel, *a, stats, **kw):
        ts = [t for t in vars(w).values() if t is not None] + list(stats)
        got.append(sum(t.numel() * t.element_size() for t in ts))

    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, "step", lambda K, V, st, *a, **kw: bytes_of(st, K, V, *a, **kw))
        q = torch.empty(1, 32, 64, 128, dtype=torch.bfloat16, device="meta")
        K = torch.empty(8, Lmax, 128, dtype=torch.bfloat16, device="meta")
        m.rows_step(m.st[0], K, K, q, torch.empty(1, dtype=torch.int32, device="meta"), Lmax, torch.empty_like(q))
    small = 32 << sh << 10          # limbs, fexp: under 1 KB a row
    assert max(got) <= M.ROWS_BYTES + small
    assert sh == 5 or 2 * max(got) + small > M.ROWS_BYTES


def test_question_rows_walk_back_a_bounded_number_of_keys():
    """A group's statistics start from those of an earlier group's first row once the walk from the last
    key would be long: the keys a long call's groups walk over grow with its rows, not with their
    square, and each group's count fits the statistics it starts from."""
    from openattention_amd import method as M
    Q, n_keys = 5000, 6000
    m = OursHIP(types.SimpleNamespace(rho=0.01), 1, 6016, "meta", n_layers=1)
    st, n_dev, calls = m.st[0], types.SimpleNamespace(at=[]), []
    n_dev.fill_ = n_dev.at.append
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, "step", lambda K, V, st, *a, qshift, later, **kw: calls.append((st, qshift, later)))
        q = torch.empty(1, 32, Q, 128, dtype=torch.bfloat16, device="meta")
        K = torch.empty(8, n_keys, 128, dtype=torch.bfloat16, device="meta")
        m.rows_step(st, K, K, q, n_dev, n_keys, torch.empty_like(q))
    assert n_dev.at[-1] == n_keys and sum(1 << c[1] for c in calls) == Q
    held, end, last = n_keys, n_keys, st
    for (base, sh, later), n_first in zip(calls, n_dev.at):
        if base is not last:         # copied after the group before, from the row that saw `end` keys
            held, last = end + 1, base
            assert base.codes is st.codes and base.Sk is not st.Sk and base.Sk.shape == st.Sk.shape
        assert n_first + (1 << sh) - 1 + later == held and n_first + (1 << sh) - 1 == end
        end = n_first - 1
        assert later <= M.ROWS_WALK
    assert last is not st


def test_tracers_and_modes_are_noticed():
    """What follows torch's operations (a tracer, make_fx with its dispatch mode before or after
    decomposition, a dispatch or function mode, autocast to another type) is noticed, so that the prefill
    attention stays a torch operation under it; a default device and bf16 autocast are not."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    x, seen = torch.zeros(3), []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    def f(t):
        seen.append(ops._watched())
        return t + 1

    f(x)
    with torch.device("cpu"):
        f(x)
    assert seen == [False, False]
    torch.jit.trace(f, (x,), check_trace=False)
    make_fx(f)(x)
    make_fx(f, pre_dispatch=True)(x)
    with Dispatch():
        seen.append(ops._watched())
    with Function(), torch.device("cpu"):
        seen.append(ops._watched())
    was, dt = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    try:
        torch.set_autocast_enabled("cuda", True)
        torch.set_autocast_dtype("cuda", torch.float16)
        seen.append(ops._watched())
        torch.set_autocast_dtype("cuda", torch.bfloat16)
        assert not ops._watched()
    finally:
        torch.set_autocast_enabled("cuda", was)
        torch.set_autocast_dtype("cuda", dt)
    assert len(seen) == 8 and all(seen[2:])


@pytest.mark.parametrize("abi,want", [(None, "lacks oa_"), (8, "has ABI 8")])
def test_an_older_library_is_refused_with_a_rebuild_message(abi, want, tmp_path, monkeypatch):
    """A kernel library of another ABI version, or of this one without the newer entry points, is refused
    with the message that names it and says to rebuild."""
    from openattention_amd import _build, lib
    src, so = tmp_path / "old.c", tmp_path / "old.so"
    src.write_text(f"int oa_abi_version(void) {{ return {lib.ABI_VERSION if abi is None else abi}; }}\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    monkeypatch.setattr(_build, "lib_path", lambda: str(so))
    monkeypatch.setattr(lib, "_LIB", None)
    with pytest.raises(RuntimeError, match=want) as e:
        lib.load()
    assert "rebuild it" in str(e.value) and str(so) in str(e.value)
