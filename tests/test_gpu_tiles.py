"""Every tile shape of the bf16 and e4m3 grouped GEMMs, forward and data
gradients, bit for bit against each other on the same ragged segments: the
shape is chosen by the number of rows the buffers hold, so longer buffers make
the few rows of the segments run on larger tiles (needs an MI355X)."""
import dataclasses

import pytest
import torch

from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu

T, TOP_K, N = 600, 2, 6


def _problem(gpu, D, F):
    """Routing of 600 tokens to 6 experts, one of them with most rows and one with
    none, x and float32 masters."""
    g = torch.Generator(device="cpu").manual_seed(D + F)
    score = torch.rand(T, N, generator=g) + torch.tensor([1.0, 0.3, 0.2, 0.0, 0.0, -9.0])
    top = score.topk(TOP_K, dim=1).indices.to(torch.int32).contiguous().to(gpu)
    plan = K.dispatch_plan(top, N, T * TOP_K)

    def rnd(*shape, std=1.0):
        return torch.randn(*shape, generator=g).mul(std).to(gpu)
    return plan, rnd


def _longer(t, rows):
    """t with rows more behind its own, which no segment holds."""
    out = torch.full((rows, *t.shape[1:]), 1, dtype=t.dtype, device=t.device)
    out[:t.shape[0]] = t
    return out


def _caps(gpu, k_bytes, ncols):
    """Buffer lengths for each tile shape these sizes take, and the shapes."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    caps = {}
    rows = T * TOP_K
    while rows < 120000:
        caps.setdefault(K.grouped_tile(rows, N, k_bytes, ncols, cus), rows)
        rows += rows // 4
    assert (256, 256) in caps and len(caps) >= 5, caps
    return caps


def _same_bits(gpu, k_bytes, ncols, plan, run):
    kept = int(plan.offsets[-1])
    assert kept == T * TOP_K and int(plan.counts.min()) == 0
    results = {}
    for tile, rows in _caps(gpu, k_bytes, ncols).items():
        print("tile", tile, "rows", rows, flush=True)
        long_plan = dataclasses.replace(plan, rows_cap=rows,
                                        perm_src=_longer(plan.perm_src, rows))
        got = run(long_plan, rows)
        torch.cuda.synchronize()
        results[tile] = [r[:kept] for r in (got if isinstance(got, tuple) else (got,))]
    want = results.pop((256, 256))
    for tile, got in results.items():
        for a, b in zip(got, want):
            assert torch.equal(a, b), tile


# (d_model, d_ff): an even and an odd number of 64-element steps of K
@pytest.mark.parametrize("D,F", [(256, 256), (320, 128)])
@pytest.mark.parametrize("form", ["swiglu", "raw", "dswiglu"])
@pytest.mark.parametrize("gather", [True, False])
def test_bf16_gate_up_forms(gpu, D, F, form, gather):
    plan, rnd = _problem(gpu, D, F)
    x, dh = rnd(T, D).to(torch.bfloat16), rnd(T * TOP_K, F).to(torch.bfloat16)
    w = K.pack_gate_up(rnd(N, D, F, std=0.05), rnd(N, D, F, std=0.05))
    xs = K.permute_rows(x, plan)

    def run(p, rows):
        if form == "dswiglu":
            d = _longer(dh, rows)
            return (K.grouped_gate_up_swiglu_bwd_gather(x, p, w, d) if gather else
                    K.grouped_gate_up_swiglu_bwd(_longer(xs, rows), p.offsets, w, d))
        if form == "raw":
            return (K.grouped_gate_up_raw_gather(x, p, w) if gather else
                    K.grouped_gate_up_raw(_longer(xs, rows), p.offsets, w))
        return (K.grouped_gate_up_gather(x, p, w) if gather else
                K.grouped_gate_up(_longer(xs, rows), p.offsets, w))
    _same_bits(gpu, 2 * D, 2 * F, plan, run)


@pytest.mark.parametrize("form,k", [("down", 256), ("down", 192), ("dgrad_down", 256),
                                    ("dgrad_down", 320), ("dgrad_gate_up", 128),
                                    ("dgrad_gate_up", 160)])
def test_bf16_plain_forms(gpu, form, k):
    """k: d_ff of the down GEMM and of the gate/up one's gradient, d_model of the
    down one's; 256 output columns."""
    plan, rnd = _problem(gpu, 256, k)
    if form == "down":
        a, w, kdim = rnd(T * TOP_K, k), K.pack_down(rnd(N, k, 256, std=0.05)), k
        f = K.grouped_down
    elif form == "dgrad_down":
        a, w, kdim = rnd(T * TOP_K, k), K.pack_down_dgrad(rnd(N, 256, k, std=0.05)), k
        f = K.grouped_dgrad_down
    else:
        a, kdim = rnd(T * TOP_K, 2 * k), 2 * k
        w = K.pack_gate_up_dgrad(rnd(N, 256, k, std=0.05), rnd(N, 256, k, std=0.05))
        f = K.grouped_dgrad_gate_up
    a = a.to(torch.bfloat16)
    _same_bits(gpu, 2 * kdim, 256, plan, lambda p, rows: f(_longer(a, rows), p.offsets, w))


@pytest.mark.parametrize("D,F", [(256, 128), (384, 256)])
@pytest.mark.parametrize("quantised_h", [True, False])
@pytest.mark.parametrize("gather", [True, False])
def test_e4m3_gate_up_forms(gpu, D, F, quantised_h, gather):
    plan, rnd = _problem(gpu, D, F)
    q, s = K.quantize_rows_fp8(rnd(T, D).to(torch.bfloat16))
    w, ws = K.pack_fp8_gate_up(rnd(N, D, F, std=0.05), rnd(N, D, F, std=0.05))
    rows_of = (plan.perm_src // TOP_K).long()
    qs, ss = q[rows_of].contiguous(), s[rows_of].contiguous()

    def run(p, rows):
        if gather:
            f = K.grouped_gate_up_fp8_gather_qh if quantised_h else K.grouped_gate_up_fp8_gather
            return f(q, s, p, w, ws)
        f = K.grouped_gate_up_fp8_qh if quantised_h else K.grouped_gate_up_fp8
        return f(_longer(qs, rows), _longer(ss, rows), p.offsets, w, ws)
    _same_bits(gpu, D, 2 * F, plan, run)


@pytest.mark.parametrize("F", [128, 384])
@pytest.mark.parametrize("block_scaled", [True, False])
def test_e4m3_down_forms(gpu, F, block_scaled):
    D = 256
    plan, rnd = _problem(gpu, D, F)
    w, ws = K.pack_fp8_down(rnd(N, F, D, std=0.05))
    q, s = K.quantize_rows_fp8(rnd(T * TOP_K, F).to(torch.bfloat16))
    e = torch.randint(117, 130, (T * TOP_K, F // 32), dtype=torch.uint8, device=gpu,
                      generator=torch.Generator(gpu).manual_seed(F))
    f, scale = (K.grouped_down_fp8_mx, e) if block_scaled else (K.grouped_down_fp8, s)
    _same_bits(gpu, F, D, plan,
               lambda p, rows: f(_longer(q, rows), _longer(scale, rows), p.offsets, w, ws))
