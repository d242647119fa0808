"""The learned preconditioner's application, whose convolutions run on the matrix cores with exactly
split FP32 activations (conv3_split_kernel), against the CPU operator in FP64 with the same BF16
weights, at the edges of the kernels' 16 x 8 x 4 tiles and of their bands per workgroup.

Tolerance (largest difference over the band's largest value): 2e-5, the FP32 accumulation bound the
FMA form of the network is tested with (layers of at most 216 terms; the split itself is exact)."""
import numpy as np
import pytest

import cnn_ref as R
import qumasun_amd as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nb", [((16, 8, 4), 1), ((17, 9, 5), 3), ((13, 7, 5), 2), ((32, 16, 12), 9),
                                  ((20, 5, 4), 17), ((15, 24, 9), 4)])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_apply_matches_cpu(gpu, n, nb, prec):
    import torch
    print(f"learned apply {n} {nb} {prec}", flush=True)
    rng = np.random.default_rng(4)
    h = (0.3, 0.35, 0.4)
    g = Q.Grid(*n, *h)
    V = rng.uniform(-2.0, 1.0, g.size)
    H = Q.Hamiltonian(g, V)
    net = Q.LearnedPreconditioner(H, 0.8, max_pairs=0, seed=12)
    net.set_params((rng.standard_normal(R.NPARAM) * 0.3).astype(np.float32))
    P = R.split(torch.from_numpy(net.get_params()).to(torch.bfloat16).to(torch.float64))
    v = torch.from_numpy(R.vnorm(V).reshape(1, 1, n[2], n[1], n[0]))
    T = torch.from_numpy(R.kinetic_symbol(n, h))
    x = rng.standard_normal((nb, g.size)) * 10.0 ** rng.uniform(-5, 3, (nb, 1))
    dt = torch.float32 if prec == "f32" else torch.float64
    r = torch.from_numpy(x).to(gpu).to(dt)
    u = R.kinetic(r.double().cpu().reshape(nb, 1, n[2], n[1], n[0]), T, 0.8)
    ref = (u + R.kinetic(R.net_adj(P, v, R.net(P, v, u)), T, 0.8)).reshape(nb, -1).numpy()
    for again in range(2):      # the second pass finds its plans and workspaces in place
        y = r.clone()
        net.apply(y)
        torch.cuda.synchronize()
        got = y.double().cpu().numpy()
        for b in range(nb):
            assert np.abs(got[b] - ref[b]).max() <= 2e-5 * np.abs(ref[b]).max(), (again, b)


def test_alternating_band_counts(gpu):
    """More band counts and precisions in turn than transform plans are kept."""
    import torch
    n = (16, 12, 10)
    g = Q.Grid(*n, 0.3, 0.3, 0.3)
    rng = np.random.default_rng(5)
    net = Q.LearnedPreconditioner(Q.Hamiltonian(g, rng.uniform(-2, 1, g.size)), 0.8, max_pairs=0, seed=12)
    x = torch.from_numpy(rng.standard_normal((7, g.size))).to(gpu)
    want = {}
    for turn in range(2):
        for nb in (7, 1, 3, 5, 2, 6):
            for dt in (torch.float32, torch.float64):
                y = x[:nb].to(dt).contiguous().clone()
                net.apply(y)
                torch.cuda.synchronize()
                key = (nb, dt)
                if turn == 0:
                    want[key] = y
                else:
                    assert torch.equal(want[key], y), key
