"""The shared experts' tiles in the routed experts' GEMM launches, bit for bit
against separate launches (needs an MI355X)."""
import ctypes

import pytest
import torch

from hanuman_amd import MoE, _lib
from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # T, K, N, d_model, d_ff, shared experts, capacity factor
    (1, 1, 1, 256, 256, 1, None),        # one row, one expert
    (1, 8, 64, 2048, 1024, 1, None),     # most experts empty
    (33, 2, 16, 256, 384, 3, None),      # one row past a fragment, three shared experts
    (48, 8, 64, 2048, 1024, 2, 1.0),     # rows dropped: the experts' rows end before the shared ones
    (333, 8, 80, 1536, 768, 1, None),    # several row tiles of the shared expert, the last partial
    (300, 3, 7, 512, 128, 2, 0.5),
    (1350, 8, 80, 1536, 768, 2, None),   # the routed GEMMs alone: 256 x 256
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T%d_K%d_N%d_D%d_F%d_S%d_%s" % c)
def test_joined_equal_separate(gpu, case):
    T, Kk, N, D, F, n, cf = case
    print(f"shared joined {case}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(T + N)
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).to(gpu)
    score = torch.rand(T, N, generator=g) + 2.0 * torch.rand(N, generator=g)
    top = score.topk(Kk, dim=1).indices.to(torch.int32).contiguous().to(gpu)
    plan = K.dispatch_plan(top, N, K.capacity(T, Kk, N, cf))
    std = D ** -0.5

    def weights(count):
        wg, wu = (torch.randn(count, D, F, generator=g).to(gpu) * std for _ in range(2))
        wd = torch.randn(count, F, D, generator=g).to(gpu) * std
        return K.pack_gate_up(wg, wu), K.pack_down(wd)
    wgu, wd = weights(N)
    sgu, sdown = weights(n)
    kept = int(plan.offsets[-1])
    ys, shared = K.grouped_swiglu_shared(x, plan, wgu, wd, sgu, sdown)
    torch.cuda.synchronize()
    ref = K.grouped_down(K.grouped_gate_up_gather(x, plan, wgu), plan.offsets, wd)
    assert torch.equal(ys[:kept], ref[:kept])
    off = K.one_group_offsets(T, x.device)
    for i in range(n):
        want = K.grouped_down(K.grouped_gate_up(x, off, sgu[i:i + 1]), off, sdown[i:i + 1])
        assert torch.equal(shared[i], want)


def test_no_joining_where_the_entries_refuse(gpu):
    """The query's 0 for every size that the two entries (host checks, placeholder
    pointers) refuse; 1 for the same sizes put right."""
    lib, p = _lib.lib(), ctypes.c_void_p(16)
    joins = lib.hmoe_grouped_shared_joins
    assert joins(64, 4, 10, 256, 128, 1, None) == 1
    for d, f in ((256, 160), (256, 100), (320, 128), (300, 128), (128, 128), (1 << 22, 128),
                 (256, 1 << 22)):
        rcs = {lib.hmoe_grouped_gate_up_gather_shared(p, 64, 2, p, p, 4, 10, d, f, p, p, 1, p, None)
               if d % 64 or f % 128 or d >= 1 << 22 or f >= 1 << 22 else 0,
               lib.hmoe_grouped_down_shared(p, p, 4, 10, 64, f, d, p, p, 1, p, None)
               if f % 64 or d % 256 or d >= 1 << 22 or f >= 1 << 22 else 0}
        assert rcs != {0}, (d, f)
        assert joins(64, 4, 10, d, f, 1, None) == 0, (d, f)


def test_joining_rule_by_size(gpu):
    """Few rows an expert join; many where the joined launch is clearly the
    shorter one, also where the routed GEMM alone takes 256 x 256 tiles."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the rule's lines are those of 256 CUs")
    joins = _lib.lib().hmoe_grouped_shared_joins
    for tokens, n, k, d, f, shared, want in ((1, 64, 8, 2048, 1024, 1, 1), (333, 80, 8, 1536, 768, 1, 1),
                                             (1350, 80, 8, 1536, 768, 2, 1), (1500, 64, 8, 2048, 1024, 1, 0),
                                             (16384, 64, 8, 2048, 1024, 1, 0)):
        assert joins(tokens, n, tokens * k, d, f, shared, None) == want, (tokens, n, shared)


@pytest.mark.parametrize("shared,d_ff_shared", [(1, None), (2, None), (1, 512)])
def test_module_same_result(gpu, monkeypatch, shared, d_ff_shared):
    """The module with the joined launches, and where they do not apply (another
    d_ff of the shared expert), against its separate launches."""
    taken = []
    rule = K.shared_joins
    monkeypatch.setattr(K, "shared_joins", lambda *a: taken.append(rule(*a)) or taken[-1])
    layer = MoE(512, 256, 16, 4, shared, 0.02, 2.5, torch.bfloat16, 3, d_ff_shared=d_ff_shared)
    x = torch.randn(2, 19, 512, device=gpu, generator=torch.Generator(gpu).manual_seed(1))
    x = x.to(torch.bfloat16)
    with torch.no_grad():
        joined = layer(x)[0]
        assert taken == [d_ff_shared is None]
        monkeypatch.setattr(K, "shared_joins", lambda *a: False)
        assert torch.equal(joined, layer(x)[0])
