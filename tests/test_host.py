"""CPU tests: the C ABI library loads and exports every declared symbol, the
host-side mirror of the reference API behaves as the reference does, and the
committed fixtures are reproduced by the oracle."""

from __future__ import annotations

import ctypes
import pathlib
import re

import numpy as np
import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
HEADERS = sorted((ROOT / "include").glob("*.h"))
LIB = ROOT / "pyshocks_amd" / "libpyshocks_amd.so"


def declared_functions() -> list[str]:
    names: list[str] = []
    for h in HEADERS:
        text = h.read_text()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names += re.findall(r"^\s*int\s+(psa_\w+)\s*\(", text, flags=re.M)
    return names


def test_header_declares_entry_points() -> None:
    names = declared_functions()
    assert "psa_ssprk33_steps" in names
    assert "psa_weno_reconstruct" in names
    assert len(names) == len(set(names))


@pytest.mark.skipif(not LIB.exists(), reason="library not built")
def test_library_exports_every_declared_symbol() -> None:
    lib = ctypes.CDLL(str(LIB))
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing


@pytest.mark.skipif(not LIB.exists(), reason="library not built")
def test_binding_covers_header() -> None:
    from pyshocks_amd import _lib

    assert set(declared_functions()) <= set(_lib.SIGNATURES), \
        set(declared_functions()) - set(_lib.SIGNATURES)


@pytest.mark.skipif(not LIB.exists(), reason="library not built")
def test_struct_layouts_and_errors() -> None:
    from pyshocks_amd import _lib

    lib = _lib.load()
    assert lib.psa_control_bytes() == ctypes.sizeof(_lib.PsaControl)
    # argument validation runs before any device work
    assert lib.psa_weno_reconstruct(7, None, None, None, 10, 1e-6, None) == \
        _lib.PSA_ERR_NOT_IMPLEMENTED
    assert "dtype" in _lib.last_error()
    # the ES-WENO entry points validate before any launch
    assert lib.psa_esweno_dissipation(0, None, None, 8, 1e-6, 1e-6, 0, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    assert lib.psa_esweno_dissipation(0, 1, 1, 8, 1e-6, 1e-6, 2, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    assert "weight" in _lib.last_error()
    assert lib.psa_esweno_dissipation(0, 1, 1, 8, 0.0, 1e-6, 0, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    assert lib.psa_flux_divergence(0, 1, None, 1, 8, -1.0, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    assert lib.psa_esweno_advection_flux(0, 1, None, 1, 1, 8, 1e-6, 1e-6, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    assert lib.psa_apply_operator_rec(0, _lib.PSA_FLUX_ESWENO, _lib.PSA_REC_ESWENO32, 1,
                                      None, None, 1, 16, 2, 0.1, 1e-6, None) == \
        _lib.PSA_ERR_INVALID_ARGUMENT
    desc_es = _lib.PsaSolverDesc()
    desc_es.dtype, desc_es.flux, desc_es.n, desc_es.g, desc_es.dx = 0, 5, 16, 2, 1 / 16
    desc_es.rec = _lib.PSA_REC_WENOJS32
    with pytest.raises(ValueError, match="ES-WENO"):
        _lib.check(lib.psa_ssprk33_steps(ctypes.byref(desc_es), None, None, None, None,
                                         None, 1, None))
    # the Koren limiter has no slope form
    assert lib.psa_muscls_reconstruct(0, _lib.PSA_LIMITER_KOREN, None, None, None, 8,
                                      0.1, None) == _lib.PSA_ERR_NOT_IMPLEMENTED
    assert "Koren" in _lib.last_error()
    with pytest.raises(ValueError):
        _lib.check(lib.psa_apply_boundary_periodic(0, None, None, 4, 3, None))
    desc = _lib.PsaSolverDesc()
    desc.dtype = 0
    desc.flux = 0
    desc.n = 16
    desc.g = 2
    desc.dx = 1 / 16
    with pytest.raises(ValueError, match="ghost"):
        _lib.check(lib.psa_ssprk33_steps(ctypes.byref(desc), None, None, None, None,
                                         None, 1, None))


def test_product_refuses_cpu_tensors() -> None:
    import torch

    from pyshocks_amd import make_uniform_cell_grid
    from pyshocks_amd.burgers import Rusanov
    from pyshocks_amd.reconstruction import WENOJS53
    from pyshocks_amd.scalar import PeriodicBoundary
    from pyshocks_amd.schemes import apply_operator

    grid = make_uniform_cell_grid(0.0, 1.0, 16, nghosts=3, device="cpu")
    u = torch.zeros(22, dtype=torch.float64)
    with pytest.raises((ValueError, RuntimeError)):
        apply_operator(Rusanov(rec=WENOJS53(eps=1e-6)), grid, PeriodicBoundary(), 0.0, u)


def test_registries_and_errors() -> None:
    from pyshocks_amd import _lib, advection, burgers
    from pyshocks_amd.reconstruction import WENOJS53, make_reconstruction_from_name

    rec = make_reconstruction_from_name("wenojs53", eps=1e-6, unused=3)
    assert isinstance(rec, WENOJS53) and rec.eps == 1e-6
    assert WENOJS53().eps == 1e-12
    assert rec.order == 3 and rec.stencil_width == 3
    with pytest.raises(ValueError):
        make_reconstruction_from_name("nope")
    with pytest.raises(NotImplementedError):
        make_reconstruction_from_name("ssweno242")

    s = burgers.make_scheme_from_name("rusanov", rec=rec, alpha=0.9, other=1)
    assert isinstance(s, burgers.Rusanov) and s.alpha == 0.9
    assert s.name == "rusanov_wenojs53" and s.order == 3 and s.stencil_width == 3
    with pytest.raises(ValueError):
        burgers.make_scheme_from_name("nope")
    # burgers/__init__.py:62-72: "default" and "lf" are Lax-Friedrichs, a
    # Rusanov subclass with its alpha; "eo" has a fixed omega = 0
    lf = burgers.make_scheme_from_name("default", rec=rec, alpha=0.8)
    assert type(lf) is burgers.LaxFriedrichs and isinstance(lf, burgers.Rusanov)
    assert lf.alpha == 0.8 and lf.name == "laxfriedrichs_wenojs53"
    assert type(burgers.make_scheme_from_name("lf", rec=rec)) is burgers.LaxFriedrichs
    eo = burgers.make_scheme_from_name("eo", rec=rec)
    assert type(eo) is burgers.EngquistOsher and eo.omega == 0
    assert burgers.flux_kind(lf) == _lib.PSA_FLUX_LAX_FRIEDRICHS
    assert burgers.flux_kind(eo) == _lib.PSA_FLUX_ENGQUIST_OSHER
    assert burgers.scheme_ids() == ("default", "godunov", "rusanov", "lf", "eo",
                                    "esweno32")
    with pytest.raises(NotImplementedError):
        burgers.make_scheme_from_name("ssweno242", rec=rec)
    # burgers/schemes.py:214-216: ES-WENO needs its reconstruction
    with pytest.raises(TypeError):
        burgers.make_scheme_from_name("esweno32", rec=rec)
    a = advection.make_scheme_from_name("godunov", rec=rec)
    assert a.velocity is None


def test_checkpoint_semantics() -> None:
    from pyshocks_amd.checkpointing import InMemoryCheckpoint, load, save

    chk = InMemoryCheckpoint(basename="Iteration")
    for i in range(5):
        save(chk, i, {"i": i})
    assert 3 in chk and 7 not in chk
    assert load(chk, 3)["i"] == 3
    assert load(chk, 3, include=("j",)) == {}
    with pytest.raises(KeyError):
        save(chk, 3, {"i": 3})
    with pytest.raises(KeyError):
        load(chk, 9)


@pytest.mark.parametrize("kind", ["npz", "pickle"])
def test_on_disk_checkpoints(tmp_path, kind: str) -> None:
    """``checkpointing.py:149-254``: file names ``<basename>_<i:09d>.npz``, the
    saved dict round-trips (arrays onto the requested device, 0-d values as
    0-d arrays), ``KeyError`` when saving over an existing file or loading a
    missing one, ``include``; the npz files are plain ``numpy.savez`` archives
    in both directions (the reference's ``{m, t, u}`` layout)."""
    import torch

    from pyshocks_amd.checkpointing import NumpyCheckpoint, PickleCheckpoint, load, save

    cls = NumpyCheckpoint if kind == "npz" else PickleCheckpoint
    chk = cls(basename="Iteration", dirname=tmp_path, device="cpu")
    u = torch.linspace(0.0, 1.0, 11, dtype=torch.float64)
    save(chk, 7, {"m": 7, "t": np.float64(0.25), "u": u})
    assert chk.index_to_key(7) == tmp_path / "Iteration_000000007.npz"
    assert 7 in chk and 8 not in chk
    with pytest.raises(KeyError):
        save(chk, 7, {"m": 7})
    with pytest.raises(KeyError):
        load(chk, 8)
    got = load(chk, 7)
    assert int(got["m"]) == 7 and got["m"].ndim == 0 and float(got["t"]) == 0.25
    assert isinstance(got["u"], torch.Tensor) and torch.equal(got["u"], u)
    assert set(load(chk, 7, include=("t",))) == {"t"}
    if kind == "npz":
        with np.load(chk.index_to_key(7), allow_pickle=False) as f:
            assert set(f.files) == {"m", "t", "u"}
            np.testing.assert_array_equal(f["u"], u.numpy())
        np.savez(tmp_path / "Iteration_000000002.npz", m=2, t=0.5, u=np.arange(3.0))
        got = load(chk, 2)
        assert int(got["m"]) == 2 and got["u"].tolist() == [0.0, 1.0, 2.0]


def test_fused_plan_selection() -> None:
    from pyshocks_amd import apply_operator, make_uniform_cell_grid
    from pyshocks_amd.burgers import Godunov, Rusanov
    from pyshocks_amd.reconstruction import WENOJS53
    from pyshocks_amd.scalar import PeriodicBoundary
    from pyshocks_amd.timestepping import (
        SSPRK33,
        FixedTimestep,
        fused_plan,
        make_ssprk33,
    )

    grid = make_uniform_cell_grid(0.0, 1.0, 64, nghosts=3, device="cpu")
    bc = PeriodicBoundary()
    st = make_ssprk33(Rusanov(rec=WENOJS53(eps=1e-6)), grid, bc, theta=1.0)
    plan = fused_plan(st)
    assert plan is not None
    assert plan.cfl_num == 0.5 / 64 and plan.theta == 1.0
    st = make_ssprk33(Godunov(rec=WENOJS53(eps=1e-6)), grid, bc, dt=1e-3)
    plan = fused_plan(st)
    assert plan is not None and plan.fixed_dt == 1e-3

    opaque = SSPRK33(predict_timestep=FixedTimestep(1e-3),
                     source=lambda t, u: apply_operator(st.source.scheme, grid, bc, t, u),
                     checkpoint=None)
    assert fused_plan(opaque) is None


def test_generic_ssprk33_order_on_host() -> None:
    """The generic path of ``step``/``advance`` (any callables) follows the
    reference loop: SSP-RK3 order on u' = exp(-t)
    (``tests/test_timestepping.py:26-99``)."""
    import torch

    from pyshocks_amd.timestepping import SSPRK33, predict_maxit_from_timestep, step

    def source(t, u):
        return torch.tensor([np.exp(-float(t))], dtype=torch.float64)

    tfinal = 4.0
    u0 = torch.tensor([-1.0], dtype=torch.float64)
    hs, errs = [], []
    for n in range(2, 7):
        maxit, dt = predict_maxit_from_timestep(tfinal, 1.0 / 2.0**n)
        st = SSPRK33(predict_timestep=lambda t, u, dt=dt: dt, source=source,
                     checkpoint=None)
        ev = None
        for ev in step(st, u0, maxit=maxit):
            pass
        errs.append(abs(float(ev.u[0]) + np.exp(-tfinal)) / np.exp(-tfinal))
        hs.append(dt)
    from pyshocks_amd.tools import estimate_order_of_convergence

    assert estimate_order_of_convergence(np.array(hs), np.array(errs))[1] >= 2.9


def test_golden_fixtures_reproduced_by_oracle() -> None:
    """Regression of the committed fixtures against the oracle."""
    import subprocess
    import sys
    import tempfile

    golden = ROOT / "tests" / "golden"
    with tempfile.TemporaryDirectory() as tmp:
        script = (golden / "make_golden.py").read_text()
        (pathlib.Path(tmp) / "make_golden.py").write_text(
            script.replace("HERE = pathlib.Path(__file__).resolve().parent",
                           f"HERE = pathlib.Path({tmp!r})").replace(
                "sys.path.insert(0, str(HERE.parents[1]))",
                f"sys.path.insert(0, {str(ROOT)!r})"))
        subprocess.run([sys.executable, str(pathlib.Path(tmp) / "make_golden.py")],
                       check=True, capture_output=True)
        for ref in golden.glob("*.npz"):
            new = np.load(pathlib.Path(tmp) / ref.name)
            old = np.load(ref)
            assert set(new.files) == set(old.files)
            for k in old.files:
                np.testing.assert_allclose(new[k], old[k], rtol=1e-14, atol=1e-300)


def test_c_oracle_matches_numpy_oracle() -> None:
    from oracle import build as oracle_build
    from oracle import exact as E
    from oracle import ref_c
    from oracle import weno_np as W

    if not ref_c.LIB.exists():
        oracle_build.build(verbose=False)
    for kind in ("rusanov", "godunov", "eo", "lf", "advection"):
        n = 200
        grid = W.make_uniform_cell_grid(0.0, 1.0, n, nghosts=3)
        u0 = E.exact_cell_averages(E.large_initial_condition(seed=2), n)
        vel = np.ones(n + 6)
        theta = 0.5 if kind == "advection" else 1.0
        u, dts, t = W.solve(W.Scheme(kind, eps=1e-6, velocity=vel), grid, u0,
                            theta=theta, tfinal=0.05)
        cfl = 1.0 / n if kind == "advection" else 0.5 / n
        uc, tc, it, dtc = ref_c.solve(kind, u0, n=n, g=3, dx=1.0 / n, eps=1e-6,
                                      theta=theta, cfl_num=cfl, tfinal=0.05,
                                      velocity=vel)
        assert it == len(dts)
        np.testing.assert_allclose(dtc, dts, rtol=1e-14, atol=1e-16)
        i = grid.i_
        assert np.linalg.norm(uc[i] - u[i]) / np.linalg.norm(u[i]) < 1e-13
    for rec in ("wenojs32", "esweno32"):
        n = 150
        grid = W.make_uniform_cell_grid(0.0, 1.0, n, nghosts=2)
        u0 = W.apply_boundary_periodic(grid, np.sin(2 * np.pi * grid.x) + 0.3)
        u, dts, t = W.solve(W.Scheme("rusanov", eps=1e-6, rec=rec), grid, u0,
                            theta=1.0, tfinal=0.3)
        uc, tc, it, dtc = ref_c.solve("rusanov", u0, n=n, g=2, dx=1.0 / n, eps=1e-6,
                                      theta=1.0, cfl_num=0.5 / n, tfinal=0.3, rec=rec)
        assert it == len(dts)
        np.testing.assert_allclose(dtc, dts, rtol=1e-14, atol=1e-16)
        i = grid.i_
        assert np.linalg.norm(uc[i] - u[i]) / np.linalg.norm(u[i]) < 1e-13


@pytest.mark.skipif(not LIB.exists(), reason="library not built")
def test_static_solve_limits() -> None:
    """psa_ssprk33_solve_static refuses arrays beyond its static scratch and
    bad arguments before it touches a device."""
    from pyshocks_amd import _lib

    lib = _lib.load()
    assert ctypes.sizeof(_lib.PsaStaticResult) == 32
    desc = _lib.PsaSolverDesc()
    desc.dtype, desc.flux, desc.g, desc.dx, desc.eps = 0, 0, 3, 1.0, 1e-6
    desc.n = _lib.PSA_STATIC_MAX_CELLS - 5  # m = n + 6 > the limit
    st = lib.psa_ssprk33_solve_static(ctypes.byref(desc), 1, 1, 0.0, 1.0, -1,
                                      _lib.PSA_DT_CFL, 1.0, 0.5, 0.0, 1, None, None)
    assert st == _lib.PSA_ERR_WORKSPACE
    assert "PSA_STATIC_MAX_CELLS" in _lib.last_error()
    desc.n = 256
    assert lib.psa_ssprk33_solve_static(ctypes.byref(desc), None, 1, 0.0, 1.0, -1,
                                        _lib.PSA_DT_CFL, 1.0, 0.5, 0.0, 1, None,
                                        None) == _lib.PSA_ERR_INVALID_ARGUMENT
    assert lib.psa_ssprk33_solve_static(ctypes.byref(desc), 1, 1, 0.0, 1.0, -1,
                                        _lib.PSA_DT_CFL, 1.0, 0.5, 0.0, -1, None,
                                        None) == _lib.PSA_ERR_INVALID_ARGUMENT


def test_boundary_fill_plans_and_refusals() -> None:
    """Constant Neumann / Dirichlet boundaries get a fused plan (the
    whole-step kernel fills the ghost cells); callables, mixed sides and
    schemes without the whole-step kernel keep the host loop; every other
    fused entry point refuses the fills before any device work."""
    from pyshocks_amd import _lib, make_uniform_cell_grid
    from pyshocks_amd.burgers import LaxFriedrichs, Rusanov
    from pyshocks_amd.reconstruction import WENOJS53
    from pyshocks_amd.scalar import (DirichletBoundary, NeumannBoundary, TwoSidedBoundary,
                                     make_dirichlet_boundary, make_neumann_boundary)
    from pyshocks_amd.timestepping import fused_plan, make_ssprk33

    grid = make_uniform_cell_grid(0.0, 1.0, 64, nghosts=3, device="cpu")
    sch = Rusanov(rec=WENOJS53(eps=1e-6))
    plan = fused_plan(make_ssprk33(sch, grid, make_neumann_boundary(0.5, -0.25)))
    assert plan is not None and plan.desc.bc == _lib.PSA_BC_NEUMANN
    assert (plan.desc.bc_left, plan.desc.bc_right) == (0.5, -0.25)
    plan = fused_plan(make_ssprk33(sch, grid, make_dirichlet_boundary(1.0, 2.0)))
    assert plan is not None and plan.desc.bc == _lib.PSA_BC_DIRICHLET
    (values,) = [k for k in plan.keepalive if getattr(k, "numel", lambda: 0)() == 6]
    assert values.tolist() == [1.0, 1.0, 1.0, 2.0, 2.0, 2.0]
    assert fused_plan(make_ssprk33(sch, grid, make_neumann_boundary(lambda t: 0.5))) is None
    mixed = TwoSidedBoundary(left=NeumannBoundary(side=-1, g=0.5),
                             right=DirichletBoundary(side=+1, g=1.0))
    assert fused_plan(make_ssprk33(sch, grid, mixed)) is None
    lf = LaxFriedrichs(rec=WENOJS53(eps=1e-6))
    assert fused_plan(make_ssprk33(lf, grid, make_neumann_boundary(0.5))) is None

    lib = _lib.load()
    desc = _lib.PsaSolverDesc()
    desc.dtype, desc.flux, desc.n, desc.g, desc.dx = 0, 0, 64, 3, 1 / 64
    desc.bc = _lib.PSA_BC_NEUMANN
    p = ctypes.c_void_p
    assert lib.psa_ssprk33_stage(ctypes.byref(desc), 1, p(8), p(16), p(24), p(32), None,
                                 None) == _lib.PSA_ERR_NOT_IMPLEMENTED
    assert lib.psa_ssprk33_stage(ctypes.byref(desc), 0, None, p(16), p(24), None, None,
                                 None) == _lib.PSA_ERR_NOT_IMPLEMENTED
    assert lib.psa_ssprk33_advance(ctypes.byref(desc), p(8), p(16), p(24), p(32), p(40),
                                   None) == _lib.PSA_ERR_NOT_IMPLEMENTED
    assert lib.psa_numerical_flux_desc(ctypes.byref(desc), p(8), None, p(16), None) == \
        _lib.PSA_ERR_NOT_IMPLEMENTED
    desc.bc_left = float("inf")
    assert lib.psa_ssprk33_steps(ctypes.byref(desc), p(8), p(16), p(24), p(32), p(40), 1,
                                 None) == _lib.PSA_ERR_INVALID_ARGUMENT
    desc.bc, desc.bc_left = _lib.PSA_BC_DIRICHLET, 0.0
    assert lib.psa_ssprk33_steps(ctypes.byref(desc), p(8), p(16), p(24), p(32), p(40), 1,
                                 None) == _lib.PSA_ERR_INVALID_ARGUMENT
    assert "bc_values" in _lib.last_error()
    desc.bc = _lib.PSA_BC_GIVEN
    assert lib.psa_ssprk33_steps(ctypes.byref(desc), p(8), p(16), p(24), p(32), p(40), 1,
                                 None) == _lib.PSA_ERR_NOT_IMPLEMENTED
    # a Neumann step needs the whole-step kernel: a velocity array rules it out
    desc.bc, desc.flux = _lib.PSA_BC_NEUMANN, _lib.PSA_FLUX_ADVECTION_UPWIND
    desc.velocity, desc.velocity_is_const = 48, 0
    assert lib.psa_ssprk33_steps(ctypes.byref(desc), p(8), p(16), p(24), p(32), p(40), 1,
                                 None) == _lib.PSA_ERR_NOT_IMPLEMENTED


def test_work_teams_balance_the_persistent_grid() -> None:
    """Teams sized by work (cell count squared): the smallest team that
    brings an instance's work per member to the mean work per workgroup,
    within the cap; a balanced batch stays on one workgroup per instance."""
    from pyshocks_amd.batched import work_teams

    assert np.all(work_teams(np.full(1000, 4096), 256, 32) == 1)
    ns = np.array([65536] + [1024] * 300)
    team = work_teams(ns, 256, 32)
    assert team[0] == 32 and np.all(team[1:] == 1)
    rng = np.random.default_rng(3)
    for grid in (256, 512, 1024):
        ns = np.round(np.exp(rng.uniform(np.log(128), np.log(65536), 500))).astype(np.int64)
        cap = np.minimum(32, (ns + 1023) // 1024)
        for share in (1.0, 0.5):
            team = work_teams(ns, grid, cap, share)
            w = ns.astype(np.float64) ** 2
            mean = share * w.sum() / grid
            assert np.all((team >= 1) & (team <= cap))
            uncapped = team < cap
            assert np.all(w[uncapped] / team[uncapped] <= mean * (1 + 1e-12))
            split = team > 1
            assert np.all(w[split] / (team[split] - 1) > mean)
        assert np.all(work_teams(ns, grid, cap, 0.5) >= work_teams(ns, grid, cap, 1.0))


def test_batched_team_size_argument_checked_before_any_allocation() -> None:
    """team_cells takes a cell count >= 0, "work" or None; anything else is
    refused before the solver touches a device."""
    from pyshocks_amd.batched import BatchedSolver

    for bad in (-1, 2.5, True, "cells"):
        with pytest.raises(ValueError, match="team_cells"):
            BatchedSolver([64, 128], team_cells=bad)


def test_evolve_chunk(monkeypatch) -> None:
    """evolve enqueues as many steps at a time as its caller asks for, also where
    one launch would run them all; only by default does it choose itself."""
    import inspect
    import types

    import torch

    from pyshocks_amd import _lib, timestepping

    class Plan:
        np_dtype = np.float64

        def __init__(self, one_launch: bool) -> None:
            self.one_launch, self.calls, self.m = one_launch, [], 0

        def new_control(self, *args):
            return None

        def runs_in_one_launch(self) -> bool:
            return self.one_launch

        def steps(self, u_in, u_out, k1, k2, ctrl, n: int) -> None:
            self.calls.append(n)
            self.m = min(self.m + n, 100)

        def read_progress(self, ctrl):
            return types.SimpleNamespace(t=0.0, dt=1.0, m=self.m, status=_lib.PSA_OK,
                                         active=int(self.m < 100))

    monkeypatch.setattr(_lib, "require_device", lambda *a: None)

    def calls(one_launch: bool, **kwargs) -> list[int]:
        plan = Plan(one_launch)
        monkeypatch.setattr(timestepping, "fused_plan", lambda *a, **k: plan)
        end = timestepping.evolve(None, torch.zeros(10, dtype=torch.float64), tfinal=1.0,
                                  **kwargs)
        assert end.iteration == 100
        return plan.calls

    assert inspect.signature(timestepping.evolve).parameters["chunk"].default == 64
    assert calls(False) == [64, 64]
    assert calls(True) == [timestepping.ONE_LAUNCH_STEPS]
    for one_launch in (False, True):
        assert calls(one_launch, chunk=64) == [64, 64]
        assert calls(one_launch, chunk=40) == [40, 40, 40]
