"""Weight gradients over the chunk sizes of k_sur_wgrad: the number of points
decides how many a workgroup sums (128 to 1024 here).  Against the numpy
surrogate oracle with the kernels' roundings, at the bars of its own test:
loss 1e-3, every parameter block 1e-2.
"""

import numpy as np
import pytest

from conftest import rel_l2
from oracle import surrogate as osur

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblk", [1, 33, 64, 128, 256])  # 256-point blocks: chunks 128, 128, 256, 512, 1024
def test_gradient_matches_numpy_at_every_chunk(nblk):
    import torch

    from bldfm_amd import surrogate as sur

    ms = sur.MetSet(sur.sample_met(8, 3))
    mu, sd = sur.met_normalisation(ms)
    net = sur.SurrogateNet(mu, sd, seed=4)
    rng = np.random.default_rng(nblk)
    p = net.params.cpu().numpy().astype(np.float64)
    off, _ = osur.layout()
    p[off["Wo"][0] : off["Wo"][0] + 512] = rng.normal(0.0, 0.05, 512)
    net.params.copy_(torch.from_numpy(p.astype(np.float32)).cuda())
    net.pack()
    gen = torch.Generator(device="cuda").manual_seed(nblk)
    mids, kxy = net.sample_points(ms, nblk, gen)
    g = ms.solve(mids, kxy)
    P = kxy.shape[0]
    ws = torch.zeros(P * net.bytes_per_point, dtype=torch.uint8, device="cuda")
    net.grad.zero_()
    loss = net.grad_step(ms, mids.repeat_interleave(2), kxy, g, ws=ws)
    x0 = ws.view(torch.bfloat16)[: 96 * P].view(96, P).float().cpu().numpy().T.astype(np.float64)
    sm = ms.surmet_host[np.repeat(mids.cpu().numpy(), 256)]
    k = kxy.cpu().numpy()
    L, grad, _ = osur.loss_grad(p, x0, g.cpu().numpy(), osur.phi0(sm, k[:, 0], k[:, 1]), block=128, bf16_mode=True)
    assert abs(float(loss.item()) - L) <= 1e-3 * abs(L)
    got = net.grad.cpu().numpy().astype(np.float64)
    for name, (o, s) in off.items():
        n = int(np.prod(s))
        assert rel_l2(got[o : o + n], grad[o : o + n]) < 1e-2, name
