"""GPU tests of the wave-uniform cell lists (cells grouped by the operator types
a kernel reads, each group padded to whole 64-cell waves): the mixed-precision
kernels take their cells from them.  On a planar mesh the lists are there by
default; with PECS_SCHUR_UNIFORM=0 they are not, and the mode is refused.

Every cell is in them, whatever its group's padding (refinement 3 leaves the
groups of the mesh's boundary types partly filled), so a mixed-precision step
depends on the state alone: the old currents, which no kernel reads, may be
NaN, and the same step after one from another state gives the same bits,
where a cell left out would keep its old currents, multiplier data or Schur
right-hand side.  (How far the mode is from FP64 is test_gpu_mixed.py's part.)
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _params(B, seed, r, k=2):
    import pecs_amd
    rng = np.random.default_rng(seed)
    prms = []
    for _ in range(B):
        p = pecs_amd.workload_params(r, k, 5e-4)
        p.update(phi_bi=0.4, phi_app=float(rng.uniform(-0.5, 0.5)), G0=float(10 ** rng.uniform(-1, 1)))
        prms.append(p)
    return prms


@pytest.mark.parametrize("B,r,k", [(1, 3, 2), (1, 5, 2), (4, 4, 2), (1, 3, 1), (3, 3, 3)])
def test_lists_hold_every_cell(B, r, k, seed):
    import pecs_amd
    prms = _params(B, seed, r, k)
    _say(f"[gpu] uniform cell lists, mixed-precision steps: B={B} r={r} k={k} seed={seed}")
    g = pecs_amd.SolarCellGPU(prms if B > 1 else prms[0])
    assert g.uniform_lists() == 31
    g.initial_state()
    start = [g.get_state(i) for i in range(B)]
    g.step(2)  # (FP64: other right-hand sides in every buffer)
    other = [g.get_state(i) for i in range(B)]
    g.set_mixed_precision(True)

    def step_from(states):
        for i, st in enumerate(states):
            st = {c: v.copy() for c, v in st.items()}
            for c in "npro":
                st[c][:2 * len(st[c]) // 3] = np.nan
            g.set_state(st, i)
        g.step(1)
        return [g.get_state(i) for i in range(B)]

    first = step_from(start)
    step_from(other)
    again = step_from(start)
    g.close()
    for i in range(B):
        for c in "nproP":
            assert np.all(np.isfinite(first[i][c])), (i, c)
            assert np.array_equal(first[i][c], again[i][c]), (i, c)


def test_without_lists_mixed_precision_is_refused(seed, monkeypatch):
    import pecs_amd
    _say("[gpu] uniform cell lists switched off")
    monkeypatch.setenv("PECS_SCHUR_UNIFORM", "0")
    g = pecs_amd.SolarCellGPU(_params(1, seed, 3)[0])
    assert g.uniform_lists() == 0
    with pytest.raises(RuntimeError):
        g.set_mixed_precision(True)
    g.close()
