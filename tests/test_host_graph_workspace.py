"""Captured solver steps and the workspaces they write to, on the CPU: the graphs of a batch are dropped when the operator
replaces a workspace, and the line sweep's partial sinograms are sized for the full angle set beside the subsets."""
import numpy as np
import pytest
import torch

from diffractom_amd import batched
from diffractom_amd.operator import SinglePhaseForwardOperator


class _Op:
    queue = None
    device = "cpu"
    scratch_generation = 3

    def _tables(self, m):
        return None


class _Graph:
    def __init__(self):
        self.replays = 0

    def replay(self):
        self.replays += 1


class _Capture:
    def __init__(self, graph):
        pass

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


@pytest.fixture
def batch(monkeypatch):
    """A BatchedSPDHGPoisson of 3 subsets whose steps are recorded in bat.ran."""
    monkeypatch.setattr(torch.cuda, "CUDAGraph", _Graph)
    monkeypatch.setattr(torch.cuda, "graph", _Capture)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: None)
    monkeypatch.setattr(batched, "SPDHGPoisson", lambda op, **k: type("S", (), {"subsets": [0, 1, 2]})())
    op = _Op()
    op.Nx = op.Ny = op.My = op.N_Omega = op.N_seg = op.K_stride = 4
    op.angles, op.cor_offset, op.batches = np.zeros(4), 0.0, [0]
    op.mfma_batches, op.blk_batches, op.pf_precision = None, [0], "bf16"
    bat = batched.BatchedSPDHGPoisson([op], subsets=3, graphs=True)
    bat._group = lambda forward, m: None
    bat.ran, bat.grow = [], {}
    bat._seq, bat._pos = [0, 1, 2], 0

    def step(next_block=None, full_forward=False, block=None):
        key = (bat._seq[bat._pos] if block is None else block, next_block)
        bat.ran.append(key)
        op.scratch_generation += bat.grow.pop(key, 0)
    bat.step = step
    return bat


def test_replaced_workspace_drops_the_captured_steps(batch):
    assert batch.capture_all() == 6
    graphs = dict(batch._graph_cache)
    batch._run_step(1)
    assert graphs[0, 1].replays == 1
    batch.ops[0].scratch_generation += 1                     # e.g. an eager forward of every angle
    batch.ran.clear()
    batch._run_step(1)
    assert graphs[0, 1].replays == 1 and batch.ran == [(0, 1)] and not batch._graph_cache
    batch._run_step(1)                                       # captured again ...
    batch._run_step(1)                                       # ... and replayed
    assert batch._graph_cache[0, 1].replays == 2


def test_growth_while_capturing_captures_the_earlier_steps_again(batch):
    batch.grow[1, 2] = 1
    assert batch.capture_all() == 6
    assert batch.ran.count((0, 1)) == 2 and batch.ran.count((2, 1)) == 1


def test_growth_in_a_lazy_capture_runs_the_step(batch):
    batch._run_step(1)
    batch.grow[0, 1] = 1
    batch.ran.clear()
    batch._run_step(1)                                       # its capture finds the workspace replaced
    assert batch.ran == [(0, 1), (0, 1)] and not batch._graph_cache


@pytest.mark.parametrize("n,my,n_omega,M,kn", [(128, 131, 90, 5, 256), (99, 103, 60, 6, 128), (99, 103, 180, 10, 576),
                                               (200, 203, 60, 7, 64), (99, 103, 180, 10, 9920)])
def test_partial_sinograms_are_sized_for_every_angle_set(n, my, n_omega, M, kn):
    op = object.__new__(SinglePhaseForwardOperator)
    op.Nx = op.Ny = n
    op.My, op.N_Omega, op.radon_variant, op._lines_caps = my, n_omega, {}, {}
    groups = lambda na: {"sweep_grp_p": np.zeros((-(-na // (512 // -(-my // 2))), 1))}
    op._tables_full = groups(n_omega)
    op.omega_subsets = [np.arange(m, n_omega, M) for m in range(M)]
    op._sub_tables = [groups(len(s)) for s in op.omega_subsets]

    def need(t, na):
        ns = op._lines_variant(t, kn)[0]
        return ns * na * my * kn if ns > 1 else 0
    sets = [(op._tables_full, n_omega)] + [(t, len(s)) for t, s in zip(op._sub_tables, op.omega_subsets)]
    most = max(need(t, na) for t, na in sets)
    for t, na in sets:
        assert op._lines_part(t, na, kn) == most


def test_tuned_line_sweep_keeps_the_rule_for_other_launches():
    """Autotuning on a subset that splits its lines leaves the number of ranges of every other launch to the rule."""
    from diffractom_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("the library is not built")
    n, my, n_omega, M, kn = 99, 103, 180, 10, 576
    op = object.__new__(SinglePhaseForwardOperator)
    op.Nx = op.Ny = n
    op.My, op.N_Omega, op._lines_caps, op.fourier, op.radon_bands = my, n_omega, {}, None, 1
    op.radon_variant = {"fwd": 8 + 256, "bwd": None, "fwd_kernel": None, "bwd_kernel": "table"}

    def tables(na):
        return {"sweep_grp_p": np.zeros((-(-na // 9), 1)), "pairs_ok": True, "mfma_ok": True, "tbase8": torch.zeros(2)}
    op._tables_full, op.omega_subsets = tables(n_omega), [np.arange(m, n_omega, M) for m in range(M)]
    op._sub_tables = [tables(len(s)) for s in op.omega_subsets]
    sub, full = op._sub_tables[0], op._tables_full
    rule = {k: op._lines_variant(full, k) for k in (64, kn, 9920)}
    assert op._lines_variant(sub, kn)[0] > 1 and rule[kn][0] < op._lines_variant(sub, kn)[0]
    op._angle_set = lambda m: (len(op.omega_subsets[m]), None, None, None)
    op._radon_backward = lambda *a, **k: 1.0
    # the line sweep is the fastest, the more ranges the better
    op._radon_forward = lambda *a: (1.0 / op._lines_variant(sub, kn)[0] if op.radon_variant["fwd_kernel"] == "lines"
                                    else 9.0)
    op.tune_projector(0, None, kn, 0, kn, None, None, None, None, lambda f: f())
    assert op.radon_variant["fwd_kernel"] == "lines"
    assert {k: op._lines_variant(full, k)[0] for k in rule} == {k: r[0] for k, r in rule.items()}
