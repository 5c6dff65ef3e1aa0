"""GPU tests of the cell and network kernels at the sizes where their tiles end.

The cell kernels give a workgroup 16 to 64 cells, 256 / (k + 1)^2 cells or 4
instances of a batch: refinements 1 and 2 leave workgroups mostly empty,
batches of 5, 6, 17 and 18 leave remainders, and the boundary-layer mesh takes
the hanging-face variants.  Trajectories are compared with the CPU oracle at
the 1e-10 trajectory bar, the steady residual with the states around its step:
at most 3e4 squares per sum, each exact to 2 roundings, summed in any order,
are off by less than 3e4 eps = 7e-12; the bar is 1e-11.

The network's convolutions run on strips of whole rows where the map divides
into them (up to 64 output channels per workgroup; gradients up to 1152 inputs
times taps) and element by element elsewhere.  FP32 sums of K terms are off by
about sqrt(K) eps of their largest: 4e-6 at K = 1161; bars 1e-5 for values and
1e-4 for gradients, relative to the block's largest.  A hidden value within
1e-6 of its layer's largest (and not zero: no input at all) has no sign in FP32, and the gradient jumps there
(one unit at 2e-8 moves the first decoder's encoder gradients by 6e-4, in FP32
on the CPU likewise): either derivative is right, so the FP64 reference is
taken with each such unit on and off.
"""
import itertools

import numpy as np
import pytest

from oracle.solarcell import OracleSolarCell

pytestmark = pytest.mark.gpu

MESH = {"planar": dict(), "conic": dict(r1=0.5, r2=0.5 + np.tan(np.radians(7.0)), L=1.5),
        "layer": dict(r1=0.3, r2=0.6, L=1.0, local_refine=1, bl=0.1)}


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# (k, refinement, batch, mesh, distinct mobilities)
@pytest.mark.parametrize("k,r,B,mesh,distinct", [
    (1, 1, 1, "planar", False), (1, 3, 18, "layer", False), (2, 2, 1, "conic", True), (2, 2, 6, "layer", True),
    (2, 3, 17, "conic", False), (3, 2, 1, "layer", False), (3, 1, 5, "planar", True), (3, 2, 17, "conic", False)])
def test_cell_kernels_at_tile_ends(k, r, B, mesh, distinct):
    import pecs_amd
    print(f"[gpu] tiles k={k} r={r} B={B} {mesh} distinct={distinct}", flush=True)
    rng = np.random.default_rng(17)
    prms = []
    for _ in range(B):
        p = pecs_amd.workload_params(r, k, 5e-4)
        p.update(MESH[mesh], phi_bi=0.4, phi_app=float(rng.uniform(-0.5, 0.5)), G0=float(10 ** rng.uniform(-1, 1)))
        if distinct:
            p.update(mu_n=1.3, mu_p=0.7, mu_r=2.0, mu_o=0.5)
        prms.append(p)
    g = pecs_amd.SolarCellGPU(prms if B > 1 else prms[0])
    g.initial_state()
    g.step(2)
    old = [g.get_state(i) if B > 1 else g.get_state() for i in range(B)]
    g.step(1)
    res = g.residuals() if B > 1 else [g.residual()]
    for i in range(B):
        st = g.get_state(i) if B > 1 else g.get_state()
        d = np.sqrt(sum(np.sum((st[c] - old[i][c]) ** 2) for c in "nproP"))
        n = np.sqrt(sum(np.sum(old[i][c] ** 2) for c in "nproP"))
        assert abs(res[i] - d / (n * 5e-4)) <= 1e-11 * res[i], (i, res[i], d / (n * 5e-4))
        if i % 4 == 0 or i == B - 1:
            ref = OracleSolarCell(prms[i]).run(3)
            for c in "nproP":
                assert _rel(st[c], ref[c]) < 1e-10, (i, c, _rel(st[c], ref[c]))
    g.close()


def _reference(p, lay, x, y):
    """FP64 outputs, loss and the gradient for each choice at the undecided hidden units."""
    import torch
    q = torch.tensor(p, requires_grad=True)
    y = torch.tensor(y, dtype=torch.float64)

    def run(flips):
        a, und = torch.tensor(x, dtype=torch.float64), []
        for i, L in enumerate(lay["layers"]):
            if not L["conv"]:
                z = a @ q[L["w"]:L["b"]].view(L["nin"], L["nout"]) + q[L["b"]:L["b"] + L["nout"]]
            else:
                if a.dim() == 2:
                    a = a.view(-1, lay["c0"], lay["g0"], lay["g0"])
                if L["up"]:
                    a = a.repeat_interleave(2, 2).repeat_interleave(2, 3)
                z = torch.nn.functional.conv2d(a, q[L["w"]:L["b"]].view(L["cout"], L["cin"], 3, 3),
                                               q[L["b"]:L["b"] + L["cout"]], padding=1)
            if i == len(lay["layers"]) - 1:
                break
            on = z.detach() > 0
            small = (z.detach() != 0) & (z.detach().abs() <= 1e-6 * z.detach().abs().max())
            und += [(i, j) for j in small.flatten().nonzero().flatten().tolist()]
            for l, j in flips:
                if l == i:
                    on.view(-1)[j] ^= True
            a = z * on
        z = z.reshape(len(x), -1)
        loss = ((z - y) ** 2).mean()
        (grad,) = torch.autograd.grad(loss, q)
        return z.detach().numpy(), loss.item(), grad.numpy(), und

    out, loss, grad, und = run(())
    assert len(und) <= 6, len(und)
    return out, loss, [grad] + [run(f)[2] for n in range(1, len(und) + 1) for f in itertools.combinations(und, n)]


# encoder + decoder (nin, nh, nl, c0, g0, stages, batch)
@pytest.mark.parametrize("spec", [
    (4, 16, 1, 64, 8, [(64, 1), (32, 1), (4, 0)], 1),    # strips of every width, few of them
    (3, 16, 1, 20, 4, [(33, 0), (17, 1), (5, 1)], 3),    # channels just past 32 and 16: idle waves, tails in k
    (2, 16, 1, 129, 2, [(3, 1)], 2),                     # weight gradients too wide for registers
    (2, 8, 1, 1, 16, [(1, 1), (49, 0)], 2),              # one channel; 49 outputs: four row blocks
    (2, 8, 1, 2, 32, [(3, 1)], 40),                      # more strips than slices of the weight gradient
    (2, 8, 1, 3, 6, [(4, 1), (2, 0)], 4),                # 12 x 12 maps: no strips
])
def test_convolutions_at_tile_ends(spec):
    import pecs_amd
    from mlp_reference import layout_decoder
    nin, nh, nl, c0, g0, stages, b = spec
    print(f"[gpu] tiles decoder {spec}", flush=True)
    net = pecs_amd.WarmStartNet(nin, nh, nl, 0, seed=5, decoder=(c0, g0, stages))
    lay, _ = layout_decoder(nin, nh, nl, c0, g0, stages)
    rng = np.random.default_rng(23)
    x = rng.normal(size=(b, nin)).astype(np.float32)
    y = rng.normal(size=(b, net.nout)).astype(np.float32)
    p = net.params().astype(np.float64)
    loss, g = net.gradients(x, y)
    yr, rloss, grads = _reference(p, lay, x, y)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss)
    blocks = [b for yl in lay["layers"] for b in
              ((yl["w"], yl["b"]), (yl["b"], yl["b"] + (yl["cout"] if yl["conv"] else yl["nout"])))]
    worst = min(max(np.abs(g[lo:hi] - rg[lo:hi]).max() / (1e-4 * np.abs(rg[lo:hi]).max() + 1e-12) for lo, hi in blocks)
                for rg in grads)
    assert worst <= 1.0, worst
    assert np.abs(net.predict(x, bf16=False) - yr).max() <= 1e-5 * np.abs(yr).max()
    rel = np.abs(net.predict(x, bf16=True) - yr).max() / np.abs(yr).max()
    assert 0 < rel < 3e-2, rel
    net.close()
