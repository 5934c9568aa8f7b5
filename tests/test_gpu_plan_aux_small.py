"""The one-launch dispatch plan either side of its limits, and the aux
losses' chunks with partial waves (needs an MI355X)."""
import numpy as np
import pytest
import torch

import oracle as O
from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,Kk,N,cap", [(1, 1, 9, 1), (512, 2, 16, 700), (600, 3, 64, 5000),
                                        (4096, 2, 16, 3000), (8192, 1, 64, 8192), (1023, 8, 100, 900)])
def test_plan_one_launch_collapsed_load(gpu, T, Kk, N, cap):
    """Every token on the same experts, at each number of counter arrays (1 to 16)."""
    print(f"plan collapsed {T} {Kk} {N}", flush=True)
    idx = np.tile(np.arange(N - Kk, N, dtype=np.int32), (T, 1))
    ref = O.dispatch_plan(idx, N, cap)
    plan = K.dispatch_plan(torch.from_numpy(idx).to(gpu), N, cap)
    torch.cuda.synchronize()
    for name in ("counts", "offsets", "slot_pos"):
        assert np.array_equal(getattr(plan, name).cpu().numpy(), ref[name]), name
    kept = int(ref["offsets"][-1])
    assert np.array_equal(plan.perm_src.cpu().numpy()[:kept], ref["perm_src"][:kept])


@pytest.mark.parametrize("T,Kk,N,cap", [(1, 1, 1, 1), (512, 2, 7, 130), (513, 2, 7, 130),
                                        (1024, 8, 8, 900), (1025, 8, 8, 900), (2730, 3, 300, 20)])
def test_plan_one_launch_matches_oracle(gpu, T, Kk, N, cap):
    print(f"plan {T} {Kk} {N}", flush=True)
    rng = np.random.default_rng(T)
    idx = np.argsort(rng.random((T, N)) + rng.random(N), axis=1)[:, :Kk].astype(np.int32)
    ref = O.dispatch_plan(idx, N, cap)
    plan = K.dispatch_plan(torch.from_numpy(idx).to(gpu), N, cap)
    torch.cuda.synchronize()
    for name in ("counts", "offsets", "slot_pos"):
        assert np.array_equal(getattr(plan, name).cpu().numpy(), ref[name]), name
    kept = int(ref["offsets"][-1])
    assert np.array_equal(plan.perm_src.cpu().numpy()[:kept], ref["perm_src"][:kept])
    assert (plan.perm_src.cpu().numpy()[kept:] == -1).all()


# waves with none, one, two and four tokens of a chunk
@pytest.mark.parametrize("B,S,N,Kk", [(1, 1, 64, 8), (2, 63, 80, 8), (1, 65, 16, 2), (3, 131, 200, 4),
                                      (5, 1, 256, 8), (2, 18, 80, 8), (1, 34, 64, 8)])
def test_aux_losses_partial_chunks(gpu, B, S, N, Kk):
    """Sums of at most B * S * N float32 terms of one sign or nearly so, in
    another order than the oracle's float64: within 1e-5 relative."""
    print(f"aux {B} {S} {N}", flush=True)
    rng = np.random.default_rng(S)
    logits = rng.standard_normal((B * S, N)).astype(np.float32)
    idx = np.argsort(-logits, axis=1)[:, :Kk].astype(np.int32)
    ref = O.aux_losses(logits, 1 / (1 + np.exp(-logits.astype(np.float64))), idx, B, S, N)
    losses, counts = K.router_aux(torch.from_numpy(logits).to(gpu), torch.from_numpy(idx).to(gpu), B, S)
    torch.cuda.synchronize()
    for got, name in zip(losses.cpu().numpy(), ("router_z_loss", "balance_loss", "mean_entropy")):
        assert abs(got - ref[name]) <= 1e-5 * abs(ref[name]), name
    assert np.array_equal(counts.cpu().numpy(), ref["expert_counts"])
