"""The float32 GEMMs either side of the switch to tiles whose waves split K,
against float64 (needs an MI355X)."""
import pytest
import torch

from hanuman_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # segment lengths, d_model, d_ff: a K of one half chunk, of odd halves, remainders
    ([1], 64, 64),
    ([33, 0, 5], 64, 128),
    ([100, 31, 0, 64], 192, 192),
    ([771], 512, 768),          # gate/up split (156 tiles of 64 x 64)
    ([2048], 256, 512),         # gate/up not (256 tiles), down split
    ([513, 511, 0, 1024, 40, 1, 900, 1107], 256, 512),
    # weight gradients: segments either side of the length from which a sum is
    # split, 40, 120 and 360 rows for one, two and three rounds of workgroups
    ([39, 0, 40, 41], 64, 128),
    ([119, 120, 0, 121, 1, 359, 360, 361], 256, 512),
    # and more 64 x 64 tiles (1536, 3072) than two a CU: never split
    ([37, 0, 64, 65, 1, 16, 100, 17, 31, 48, 2, 80, 15, 128, 33, 3], 512, 768),
]


def test_weight_gradient_cases_take_both_kernels(gpu):
    """The two sides of the switch at two 64 x 64 tiles a CU."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    tiles = [[len(lens) * (D // 64) * (f // 64) for f in (F, 2 * F)] for lens, D, F in CASES]
    assert max(tiles[-2]) <= 2 * cus < min(tiles[-1])
    assert [-(-4 * t // (3 * cus)) for t in tiles[-3] + tiles[-2]] == [1, 1, 2, 3]


@pytest.mark.parametrize("lens,D,F", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_f32_gemms_match_float64(gpu, lens, D, F):
    """Sums of up to 2 F products in float32, in any order: 2e-6 normwise is
    several times sqrt(1536) roundings of 2^-24."""
    print(f"f32 split {lens} {D} {F}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(sum(lens))
    N, R = len(lens), sum(lens)
    off = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(gpu)

    def rnd(*s, std=1.0):
        return (torch.randn(*s, generator=g) * std).to(gpu)
    x, h, dy, dh, dgu = rnd(R, D), rnd(R, F), rnd(R, D), rnd(R, F), rnd(R, 2 * F)
    wg, wu, wd = rnd(N, D, F, std=D ** -0.5), rnd(N, D, F, std=D ** -0.5), rnd(N, F, D, std=F ** -0.5)
    got = {"gu": K.grouped_gate_up_f32(x, off, wg, wu), "down": K.grouped_down_f32(h, off, wd),
           "dh": K.grouped_dgrad_down_f32(dy, off, wd),
           "dgu": K.grouped_gate_up_swiglu_bwd_f32(x, off, wg, wu, dh),
           "dxs": K.grouped_dgrad_gate_up_f32(dgu, off, wg, wu),
           "dwd": K.grouped_wgrad_down_f32(h, dy, off)}
    got["dwg"], got["dwu"] = K.grouped_wgrad_gate_up_f32(x, dgu, off)
    torch.cuda.synchronize()
    ref = {k: torch.zeros_like(v, dtype=torch.float64) for k, v in got.items()}
    r0 = 0
    for e, n in enumerate(lens):
        s = slice(r0, r0 + n)
        r0 += n
        G, U = x[s].double() @ wg[e].double(), x[s].double() @ wu[e].double()
        sg = torch.sigmoid(G)
        ref["gu"][s] = G * sg * U
        ref["down"][s] = h[s].double() @ wd[e].double()
        ref["dh"][s] = dy[s].double() @ wd[e].double().T
        d = dh[s].double()
        ref["dgu"][s] = torch.cat([d * U * sg * (1 + G * (1 - sg)), d * G * sg], 1)
        ref["dxs"][s] = dgu[s, :F].double() @ wg[e].double().T + dgu[s, F:].double() @ wu[e].double().T
        ref["dwd"][e] = h[s].double().T @ dy[s].double()
        ref["dwg"][e] = x[s].double().T @ dgu[s, :F].double()
        ref["dwu"][e] = x[s].double().T @ dgu[s, F:].double()
    for k in got:
        err = ((got[k].double() - ref[k]).norm() / ref[k].norm()).item()
        assert err < 2e-6, (k, err)


@pytest.mark.parametrize("D", [16, 48, 272])
def test_f32_gate_up_odd_half_chunks(gpu, D):
    """d_model an odd multiple of 16: the last half chunk of K."""
    g = torch.Generator(device="cpu").manual_seed(D)
    x = torch.randn(70, D, generator=g).to(gpu)
    wg, wu = (torch.randn(2, D, 64, generator=g).mul(D ** -0.5).to(gpu) for _ in range(2))
    off = torch.tensor([0, 37, 70], dtype=torch.int32, device=gpu)
    h = K.grouped_gate_up_f32(x, off, wg, wu)
    torch.cuda.synchronize()
    for e, s in enumerate((slice(0, 37), slice(37, 70))):
        G, U = x[s].double() @ wg[e].double(), x[s].double() @ wu[e].double()
        ref = torch.nn.functional.silu(G) * U
        assert ((h[s].double() - ref).norm() / ref.norm()).item() < 2e-6
