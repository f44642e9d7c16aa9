"""Calls that give their grid as a tuple (``_grid=(...)``, as the reference's matmul examples launch,
examples/matmul_tiled.py:305-402): repeated ones go through one native call, a lifted GEMM planned in it from
its arguments.  Every call must do what the full path does: the same outputs, the same refusals.
"""

from __future__ import annotations

import importlib

import numpy as np
import pytest

import eas
import kernels as K
from oracle import ops

eas_kernel = importlib.import_module("easy_as_amd.kernel")


class _Runtime:
    """Records full-path runs and grid launches; declines grids of one dimension."""

    def __init__(self):
        self.runs, self.fast, self.made = [], [], 0

    def run(self, ck, runtime_args, meta, **opts):
        self.runs.append((dict(runtime_args), opts))

    def grid_launcher(self, ck, names, args, sync):
        self.made += 1

        def launch(call_args, grid):
            if len(grid) == 1:
                return NotImplemented
            self.fast.append((call_args, grid, sync))
            return None

        return launch


def test_which_calls_take_the_grid_launch(monkeypatch):
    rt = _Runtime()
    monkeypatch.setattr(eas_kernel, "get_runtime", lambda *a, **k: rt)
    k = eas.kernel(K.add_kernel.fn)
    a = np.ones(64, np.float32)
    k(a, a, a, 64, BLOCK=64, _grid=(1, 1), _sync=False)  # the full path, which makes the launch
    assert len(rt.runs) == 1 and rt.made == 1 and rt.runs[0][1]["grid"] == (1, 1, 1)
    k(a, a, a, 50, BLOCK=64, _grid=(2, 1), _sync=False)  # another grid and scalar: the same launch
    assert rt.fast == [((a, a, a, 50), (2, 1), False)] and len(rt.runs) == 1
    k(a, a, a, 64, BLOCK=64, _grid=(3,), _sync=False)  # declined: the full path, no second launch made
    assert len(rt.runs) == 2 and rt.runs[1][1]["grid"] == (3, 1, 1) and rt.made == 1
    # other options have their own; a callable or int grid, _shape and _nthreads keep the full path
    k(a, a, a, 64, BLOCK=64, _grid=(1, 1))
    assert rt.made == 2 and len(rt.runs) == 3
    for opts in ({"_grid": lambda meta, args: (1, 1)}, {"_grid": 1}, {"_grid": [1, 1]},
                 {"_grid": (1, 1), "_nthreads": 64}):
        k(a, a, a, 64, BLOCK=64, **opts)
    assert rt.made == 2 and len(rt.runs) == 7 and len(rt.fast) == 1
    # what the full path refuses is refused after a launch was made
    for bad in ({"_grid": (1.5, 1), "_tptg": 3.0}, {"_grid": (1, 1), "_tptg": (64, 1, 1)}):
        with pytest.raises((TypeError, ValueError)):
            k(a, a, a, 64, BLOCK=64, **bad)


def test_one_launch_per_kind_of_arguments(monkeypatch):
    """A launch takes the types it was made for; each kind of arguments keeps its own, or that there is none."""
    class Typed(_Runtime):
        def grid_launcher(self, ck, names, args, sync):
            self.made += 1
            if args[0].dtype == np.float16:
                return None
            launch = super().grid_launcher(ck, names, args, sync)
            self.made -= 1
            kind = type(args[0])
            return lambda call_args, grid: launch(call_args, grid) if type(call_args[0]) is kind else NotImplemented

    rt = Typed()
    monkeypatch.setattr(eas_kernel, "get_runtime", lambda *a, **k: rt)
    k = eas.kernel(K.add_kernel.fn)
    a, h = np.ones(64, np.float32), np.ones(64, np.float16)
    t = eas.tensor(a, device="cpu")

    def call(x, **kw):
        k(x, x, x, 64, BLOCK=64, _grid=(1, 1), **kw)

    for x in (a, t, h):
        call(x)
    assert len(rt.runs) == 3 and rt.made == 3 and not rt.fast
    for x in (a, t, a, t, t):  # in turn: never the full path
        call(x)
    assert len(rt.runs) == 3 and rt.made == 3 and len(rt.fast) == 5
    for _ in range(3):  # no launch for this kind: the full path, and none is made anew
        call(h)
    assert len(rt.runs) == 6 and rt.made == 3 and len(rt.fast) == 5
    k(a, a, a, np.uint32(64), BLOCK=64, _grid=(1, 1))  # a scalar of a type no launch takes
    assert len(rt.runs) == 7 and rt.made == 3
    for i in range(200):  # bounded
        k(a, a, a, 64, BLOCK=64, _grid=(1, 1), _tptg=(1,) + (1,) * (i % 3), _sync=bool(i % 2))
    assert len(k._grid_made) <= 64 and len(k._grid_fast) <= 64


@pytest.mark.parametrize("sync", [1, 0, 1.0, None, np.True_])
def test_a_sync_that_is_no_bool_is_refused_after_one_that_equals_it(monkeypatch, sync):
    rt = _Runtime()
    monkeypatch.setattr(eas_kernel, "get_runtime", lambda *a, **k: rt)
    k = eas.kernel(K.add_kernel.fn)
    a = np.ones(64, np.float32)
    for s in (True, False):
        k(a, a, a, 64, BLOCK=64, _grid=(1, 1), _sync=s)
    with pytest.raises(TypeError, match="_sync must be bool"):
        k(a, a, a, 64, BLOCK=64, _grid=(1, 1), _sync=sync)
    assert len(rt.runs) == 2 and not rt.fast


@pytest.mark.gpu
@pytest.mark.parametrize("sync", [True, False])
@pytest.mark.parametrize("kind", ["mma", "tiled"])
def test_lifted_matmuls(gpu_runtime, monkeypatch, kind, sync):
    import torch

    def call(m, n, a, b, c, grid=None):
        grid = grid or (K.cdiv(n, 32), K.cdiv(m, 32))
        if kind == "mma":
            mma(a, b, c, m, n, BM=32, BN=32, BK=8, K=k, NT=512, _grid=grid, _sync=sync)
        else:
            tiled(a, b, c, m, n, 0, 0, BM=32, BN=32, BK=32, K=k, NT=256, _grid=grid, _sync=sync, _tptg=(256, 1, 1))

    mma, tiled = eas.kernel(K.matmul_mma_kernel.fn), eas.kernel(K.matmul_tiled_kernel.fn)
    k = 72
    dt = torch.float16 if kind == "mma" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(0)

    def operands(m, n):
        a, b = (torch.empty(s, device="cuda").uniform_(-1, 1, generator=g).to(dt) for s in (m * k, k * n))
        return a, b, torch.full((m * n,), float("nan"), device="cuda")

    def check(m, n, a, b, c, rows=None):
        gpu_runtime.synchronize()
        torch.cuda.synchronize()
        got = c.view(m, n)[:rows].cpu().numpy().astype(np.float64)
        want = a.view(m, k).double().cpu().numpy()[:rows] @ b.view(k, n).double().cpu().numpy()
        assert ops.rel_err(got, want) <= 1e-5 * k ** 0.5

    a, b, c = operands(300, 520)
    call(300, 520, a, b, c)
    check(300, 520, a, b, c)
    refused = gpu_runtime.run
    monkeypatch.setattr(gpu_runtime, "run", lambda *x, **y: (_ for _ in ()).throw(AssertionError("the full path ran")))
    for m, n in ((300, 520), (16, 520), (257, 101), (33, 1000)):  # other shapes, entries and operands
        a, b, c = operands(m, n)
        call(m, n, a, b, c)
        check(m, n, a, b, c)
    a, b, c = operands(96, 64)  # a grid over two of three tile rows
    call(96, 64, a, b, c, grid=(2, 2, 1))
    check(96, 64, a, b, c, rows=64)
    assert bool(c.view(96, 64)[64:].isnan().all())
    monkeypatch.setattr(gpu_runtime, "run", refused)
    with pytest.raises(ValueError, match="holds"):  # a short buffer: refused before a launch
        call(300, 520, *operands(96, 64))
    with pytest.raises(TypeError):
        call(96, 64, a.double(), b, c)
    call(96, 64, a, b, c, grid=(0, 2))  # nothing to run
    call(96, 64, a, b, c, grid=(2.0, 3.0))  # as the full path converts it
    check(96, 64, a, b, c)


@pytest.mark.gpu
@pytest.mark.parametrize("sync", [True, False])
def test_kinds_of_arguments_in_turn(gpu_runtime, monkeypatch, sync):
    """f16 and f32 torch tensors and GPU eas.Tensors through one matmul: each on its own specialisation and buffers."""
    import torch

    mma = eas.kernel(K.matmul_mma_kernel.fn)
    k = 72
    g = torch.Generator(device="cuda").manual_seed(1)

    def one(kind, m, n):
        dt = torch.float32 if kind == "f32" else torch.float16
        a, b = (torch.empty(s, device="cuda").uniform_(-1, 1, generator=g).half().to(dt) for s in (m * k, k * n))
        c = torch.full((m * n,), float("nan"), device="cuda")
        args = [eas.tensor(x, device="hip") for x in (a, b, c)] if kind == "eas" else [a, b, c]
        torch.cuda.synchronize()  # eas.Tensors alone go on the default stream
        mma(*args, m, n, BM=32, BN=32, BK=8, K=k, NT=512, _grid=(K.cdiv(n, 32), K.cdiv(m, 32)), _sync=sync)
        gpu_runtime.synchronize()
        torch.cuda.synchronize()
        want = a.view(m, k).double().cpu().numpy() @ b.view(k, n).double().cpu().numpy()
        assert ops.rel_err(c.view(m, n).cpu().numpy().astype(np.float64), want) <= 1e-5 * k ** 0.5

    for kind in ("f16", "f32", "eas"):
        one(kind, 200, 136)
    monkeypatch.setattr(gpu_runtime, "run", lambda *x, **y: (_ for _ in ()).throw(AssertionError("the full path ran")))
    for kind in ("f32", "eas", "f16", "f32", "f16", "eas"):
        one(kind, 200, 136)
        one(kind, 33, 101)
    monkeypatch.undo()
    short = eas.tensor(torch.zeros(8, device="cuda", dtype=torch.float16), device="hip")
    with pytest.raises(ValueError, match="holds"):  # refused before a launch, by the buffer's length
        mma(short, short, eas.tensor(torch.zeros(8, device="cuda"), device="hip"), 64, 64,
            BM=32, BN=32, BK=8, K=k, NT=512, _grid=(2, 2), _sync=sync)


@pytest.mark.gpu
def test_two_dimensional_grids_bit_exact(gpu_runtime, monkeypatch):
    import torch

    mm, add = eas.kernel(K.matmul_kernel.fn), eas.kernel(K.add2d_shape_kernel.fn)
    rng = np.random.default_rng(0)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((37, 50), (50, 130)))
    ta, tb = torch.from_numpy(a.reshape(-1)).cuda(), torch.from_numpy(b.reshape(-1)).cuda()
    tc = torch.empty(37 * 130, device="cuda")
    mm(ta, tb, tc, 37, 130, BLOCK=64, K=50, _grid=(37, 3))
    first = tc.cpu().numpy().copy()
    assert np.allclose(first.reshape(37, 130), a.astype(np.float64) @ b, rtol=1e-5, atol=1e-5)
    x = torch.randn(37 * 130, device="cuda")
    s = torch.empty_like(x)
    add(x, tc, s, 37, 130, BLOCK=64, _grid=(3, 37))
    monkeypatch.setattr(gpu_runtime, "run", lambda *p, **q: (_ for _ in ()).throw(AssertionError("the full path ran")))
    tc.fill_(float("nan"))
    s.fill_(float("nan"))
    mm(ta, tb, tc, 37, 130, BLOCK=64, K=50, _grid=(37, 3))
    add(x, tc, s, 37, 130, BLOCK=64, _grid=(3, 37))
    assert np.array_equal(tc.cpu().numpy(), first)
    assert torch.equal(s, x + tc)
