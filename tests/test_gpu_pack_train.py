"""Both packed operands from one read of the masters equal the separate packs,
and a training step packs anew after an update (needs an MI355X)."""
import pytest
import torch

from hanuman_amd import MoE
from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,F", [(1, 64, 32), (3, 200, 96), (2, 72, 160)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_pack_train_equals_separate_packs(gpu, N, D, F, dtype):
    g = torch.Generator(device="cpu").manual_seed(D)
    wg, wu = (torch.randn(N, D, F, generator=g).to(gpu, dtype) for _ in range(2))
    wd = torch.randn(N, F, D, generator=g).to(gpu, dtype)
    gu, gu_d = K.pack_gate_up_train(wg, wu)
    dn, dn_d = K.pack_down_train(wd)
    torch.cuda.synchronize()
    assert torch.equal(gu, K.pack_gate_up(wg, wu))
    assert torch.equal(gu_d, K.pack_gate_up_dgrad(wg, wu))
    assert torch.equal(dn, K.pack_down(wd))
    assert torch.equal(dn_d, K.pack_down_dgrad(wd))


def test_training_step_repacks_after_update(gpu):
    """Gradients after an in-place update equal those of a fresh layer with the
    updated weights, bit for bit."""
    def layer():
        m = MoE(256, 256, 4, 2, 1, 0.02, 2.5, torch.bfloat16, 3, device=gpu)
        for p in m._params():
            p.requires_grad_(True)
        return m
    x = torch.randn(2, 17, 256, generator=torch.Generator().manual_seed(1)).to(gpu, torch.bfloat16)

    def grads(m):
        out, aux = m(x)
        return torch.autograd.grad(out.square().sum() + aux["router_z_loss"], list(m._params()))
    a, b = layer(), layer()
    g0 = grads(a)
    for m in (a, b):
        with torch.no_grad():
            for p, g in zip(m._params(), g0):
                p.sub_(0.1 * g)
    for u, v in zip(grads(a), grads(b)):
        assert torch.equal(u, v)
