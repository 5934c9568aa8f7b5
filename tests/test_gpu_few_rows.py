"""The grouped GEMM's tiles for few rows per expert, bit for bit against the
256 x 256 tiles: the one-launch gate/up + down kernel always uses those and
sums in the same order, so the two-launch results must equal it whichever
tile their sizes choose (needs an MI355X)."""
import numpy as np
import pytest
import torch

from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # T, K, N, d_model, d_ff, the gate/up GEMM's tile
    (1, 1, 1, 256, 256, (32, 64)),       # one row, one segment
    (33, 1, 1, 512, 256, (32, 64)),      # one row past a fragment
    (129, 1, 1, 256, 384, (32, 64)),     # several row tiles of one segment, the last of one row
    (333, 1, 1, 1536, 768, (64, 64)),
    (700, 1, 1, 2048, 1024, (64, 128)),
    (2000, 1, 1, 2048, 1024, (128, 128)),
    (4096, 1, 1, 1536, 768, (128, 256)),
    (3, 2, 16, 256, 256, (32, 64)),      # fewer rows than experts, most experts empty
    (16, 8, 80, 1536, 768, (32, 256)),
    (48, 8, 64, 2048, 1024, (32, 128)),
    (333, 8, 80, 1536, 768, (64, 256)),  # an odd number of 128-byte steps in the down GEMM
    (300, 3, 7, 320, 256, (32, 64)),     # five steps (320 / 64), odd counts
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T%d_K%d_N%d_D%d_F%d" % c[:5])
def test_few_rows_equal_full_tiles(gpu, case):
    T, Kk, N, D, F, tile = case
    print(f"few rows {case}", flush=True)
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert K.grouped_tile(T * Kk, N, 2 * D, 2 * F, cus) == tile
    g = torch.Generator(device="cpu").manual_seed(T + N)
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).to(gpu)
    # a skewed choice of experts, so that segment lengths differ and some are empty
    score = torch.rand(T, N, generator=g) + 2.0 * torch.rand(N, generator=g)
    top = score.topk(Kk, dim=1).indices.to(torch.int32).contiguous().to(gpu)
    plan = K.dispatch_plan(top, N, T * Kk)
    wg, wu = (torch.randn(N, D, F, generator=g) * D ** -0.5 for _ in range(2))
    wd = torch.randn(N, F, D, generator=g) * F ** -0.5
    wgu = K.pack_gate_up(wg.to(gpu), wu.to(gpu))
    h = K.grouped_gate_up_gather(x, plan, wgu)
    h_plain = K.grouped_gate_up(K.permute_rows(x, plan), plan.offsets, wgu)
    torch.cuda.synchronize()
    R = T * Kk
    assert torch.equal(h[:R], h_plain[:R])
    if D % 256 == 0:
        wdp = K.pack_down(wd.to(gpu))
        ys = K.grouped_down(h, plan.offsets, wdp)
        h2, ys2, ws = K.grouped_swiglu_fused(x, plan, wgu, wdp)
        torch.cuda.synchronize()
        assert K.fused_status(ws) == 0
        assert torch.equal(h[:R], h2[:R])
        assert torch.equal(ys[:R], ys2[:R])
    # and the products themselves: float64 on the same bf16 operands, h within
    # the bf16 rounding of g, u and h (three roundings of 2^-9 each, normwise)
    off = plan.offsets.cpu().numpy()
    src = plan.perm_src.cpu().numpy()[:R] // Kk
    e = int(np.argmax(np.diff(off)))
    rows = slice(int(off[e]), int(off[e + 1]))
    xe = x.float().cpu().double()[src[rows]]
    a, b = (w[e].to(torch.bfloat16).double() for w in (wg, wu))
    ref = torch.nn.functional.silu(xe @ a) * (xe @ b)
    err = (h[rows].cpu().double() - ref).norm() / ref.norm()
    assert err < 3 * 2.0 ** -9, err
