"""The router's launch shapes at their edges, bit for bit against the oracle:
chains of 4 and of 16 tokens either side of the switch between them, every
count of expert tiles, token and expert remainders, chunk tails of d_model,
zeros, subnormals and infinities (needs an MI355X)."""
import numpy as np
import pytest
import torch

import oracle as O
from hanuman_amd import _lib
from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # T, D, N, K, x dtype, w dtype
    (1, 8, 1, 1, "bf16", "f32"),          # one chunk, two MFMA steps, one expert
    (3, 264, 16, 4, "f32", "bf16"),       # one tile, chunk tail of 8 (256 + 8)
    (5, 520, 17, 5, "bf16", "f32"),       # two tiles, one lane of the second
    (6144, 136, 16, 4, "bf16", "f32"),    # last token count of the short chains at one tile
    (6145, 136, 16, 4, "bf16", "f32"),    # and the first past it (staged W)
    (6151, 72, 12, 3, "f32", "bf16"),     # W staged by elements (12 % 8), chunk tail of 8 (64 + 8)
    (6200, 264, 7, 2, "bf16", "f32"),
    (4093, 72, 30, 3, "bf16", "bf16"),    # two tiles, 16-token chains, W staged off (30 % 8)
    (3072, 136, 32, 4, "bf16", "f32"),    # last token count of the short chains at two tiles
    (3073, 136, 32, 4, "bf16", "f32"),    # and the first past it (staged W)
    (6, 136, 48, 8, "f32", "f32"),        # three tiles
    (1537, 136, 64, 8, "bf16", "f32"),    # four tiles, first token count of 16-token chains
    (9, 264, 80, 8, "bf16", "f32"),       # five tiles, token remainder
    (1300, 136, 80, 8, "bf16", "bf16"),
    (7, 136, 129, 32, "f32", "bf16"),     # nine tiles
    (500, 136, 256, 8, "bf16", "f32"),    # sixteen
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"T{c[0]}_D{c[1]}_N{c[2]}_{c[4]}_{c[5]}")
def test_router_chains_bit_exact(gpu, case):
    T, D, N, Kk, xd, wd = case
    print(f"router chains {case}", flush=True)
    rng = np.random.default_rng(T + D + N)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = (0.1 * rng.standard_normal((D, N))).astype(np.float32)
    x[rng.random((T, D)) < 0.05] = 0.0
    w[rng.random((D, N)) < 0.05] = 0.0
    x[0, 0] = 1e-40                       # subnormal in both types
    w[D // 2, 0] = -3e-39
    w[D - 1, N - 1] = np.inf              # in the chunk tail; x there is non-zero
    x[:, D - 1] = np.abs(x[:, D - 1]) + 0.5
    if xd == "bf16":
        x = O.bf16_round(x)
    if wd == "bf16":
        w = O.bf16_round(w)
    bias = (0.05 * rng.standard_normal(N)).astype(np.float32)
    logits_ref = O.router_logits(x, w)
    idx_ref, g_ref, _ = O.route_sigmoid(logits_ref, bias, Kk, 2.5)
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}
    logits, idx, g = K.router(torch.from_numpy(x).to(gpu, dt[xd]), torch.from_numpy(w).to(gpu, dt[wd]),
                              torch.from_numpy(bias).to(gpu), Kk, _lib.ROUTE_SIGMOID_BIAS, 2.5)
    torch.cuda.synchronize()
    for name, got, ref in (("logits", logits, logits_ref), ("gates", g, g_ref)):
        assert np.array_equal(got.cpu().numpy().view(np.uint32), ref.view(np.uint32)), name
    assert np.array_equal(idx.cpu().numpy(), idx_ref)


@pytest.mark.parametrize("T,N", [(6145, 16), (6151, 12), (3073, 32), (1537, 64)])
def test_router_with_quantisation_past_the_switch(gpu, T, N):
    """The launch that quantises x beside the router, in the forms for many
    tokens, against the two separate launches."""
    print(f"router quant T{T} N{N}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(T)
    x = torch.randn(T, 264, generator=g).to(gpu, torch.bfloat16)
    w = torch.randn(264, N, generator=g).mul(0.1).to(gpu, torch.bfloat16)
    got = K.router_quant_fp8(x, w, None, 4, _lib.ROUTE_SOFTMAX, 1.0)
    ref = (*K.router(x, w, None, 4, _lib.ROUTE_SOFTMAX, 1.0), *K.quantize_rows_fp8(x))
    torch.cuda.synchronize()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D", [8, 72, 136, 264])
@pytest.mark.parametrize("T,N", [(5, 16), (7000, 16), (5, 30), (4100, 30), (4100, 32), (5, 64),
                                 (1600, 64), (5, 80), (1300, 80), (500, 256)])
@pytest.mark.parametrize("wd", [torch.float32, torch.bfloat16])
def test_rows_behind_w_are_not_read(gpu, T, N, D, wd):
    """W as the front of a larger buffer: what lies behind its last row (NaN, or
    zeros) makes no difference, also where d_model ends inside a chunk."""
    print(f"router W tail T{T} N{N} D{D} {wd}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(T + N + D)
    x = torch.randn(T, D, generator=g).to(gpu, torch.bfloat16)
    w = torch.randn(D, N, generator=g).mul(0.1)
    got = []
    for behind in (0.0, float("nan")):
        buf = torch.full(((D + 256) * N,), behind, dtype=wd, device=gpu)
        buf[:D * N] = w.to(gpu, wd).reshape(-1)
        got.append(K.router(x, buf[:D * N].view(D, N), None, min(4, N), _lib.ROUTE_SOFTMAX, 1.0))
    torch.cuda.synchronize()
    assert torch.isfinite(got[0][0]).all()
    for a, b in zip(*got):
        assert torch.equal(a, b)
