"""The F32 warp's adjoint where its kernels change path: images narrower than a wave and heights off the
row groups, sources of one row or column, samples that leave the source or lie behind the camera,
homographies whose z leaves the range of the shared reciprocal, and scaled or rotated footprints whose
contributions to dL/dsource do not line up from pixel to pixel.  Reference: float64 autograd.

Tolerances: F32 positions carry about 1e-7 of their coordinate (below 140 here), so a bilinear weight is
off by at most about 2e-5 and a sum of a few such terms by 1e-4 of the largest.  dL/dH is compared as a
vector within 1e-4 plus what cell boundaries allow: the image slope jumps there, by at most 2 for values in
[0, 1], so a sample within 4e-5 px of a boundary (twice the position error) may move its term of dL/dH by
2 |g| / z times its coordinates."""
import pytest
import torch

from mivisionx_amd import align
from test_gpu_warp_adjoint import warp64

pytestmark = pytest.mark.gpu

SIZES = [((1, 1), (1, 1)), ((5, 1), (3, 7)), ((1, 9), (70, 5)), ((2, 2), (63, 4)), ((64, 16), (64, 16)), ((65, 33), (65, 17)),
         ((130, 37), (127, 35)), ((40, 50), (130, 66))]
HOMS = {"near_identity": [1.013, 0.021, 0.37, -0.017, 0.991, -0.43, 1e-4, -2e-4, 1.0],
        "shift_out": [1, 0, 31.3, 0, 1, -12.6, 0, 0, 1],
        "shrink_rotate": [1.9, 0.83, -7.3, -0.77, 2.1, 5.2, 0, 0, 1],
        "enlarge": [0.31, 0.013, 0.7, -0.02, 0.27, 0.4, 0, 0, 1],
        "behind": [1.1, 0.1, 0.3, -0.2, 0.9, 0.6, 0.03, -0.04, 0.21],
        "tiny_z": [1.013e-25, 0.021e-25, 0.37e-25, -0.017e-25, 0.991e-25, -0.43e-25, 0, 0, 1e-25],
        "huge_z": [1.013e25, 0.021e25, 0.37e25, -0.017e25, 0.991e25, -0.43e25, 0, 0, 1e25]}


def _boundary_allowance(H, g):
    """the sum over samples near a cell boundary of 2 |g| / z |(x, y, 1)| |(u, v, 1)|, both images together"""
    n, dh, dw = g.shape
    ys, xs = torch.meshgrid(torch.arange(dh, dtype=torch.float64, device=g.device), torch.arange(dw, dtype=torch.float64, device=g.device),
                            indexing="ij")
    p = torch.stack([xs, ys, torch.ones_like(xs)], -1).reshape(-1, 3)
    q = torch.einsum("nij,pj->npi", H.reshape(n, 3, 3), p)
    z = q[..., 2]
    ok = z > 0
    uv = q[..., :2] / torch.where(ok, z, torch.ones_like(z))[..., None]
    near = ok & ((uv - uv.round()).abs() < 4e-5).any(-1)
    size = torch.linalg.norm(p, dim=-1)[None] * torch.sqrt(1 + (uv * uv).sum(-1))
    return float((2 * g.double().abs().reshape(n, -1) / z * size)[near].sum())


def _check_gH(got, want, H, g, what):
    bound = 1e-4 * float(torch.linalg.norm(want)) + _boundary_allowance(H, g)
    assert float(torch.linalg.norm(got - want)) <= bound, f"{what}: {got}\n{want}\nbound {bound}"


@pytest.mark.parametrize("name", HOMS)
@pytest.mark.parametrize("src_wh,dst_wh", SIZES)
def test_adjoint_paths(gpu, src_wh, dst_wh, name):
    print(f"adjoint {name}: source {src_wh}, destination {dst_wh}", flush=True)
    (sw, sh), (dw, dh) = src_wh, dst_wh
    gen = torch.Generator(device="cuda").manual_seed(7)
    src = torch.rand((2, sh, sw), generator=gen, device="cuda")
    g = torch.rand((2, dh, dw), generator=gen, device="cuda") - 0.3
    g[:, ::3, ::5] = 0.0
    H = torch.tensor([HOMS[name], HOMS[name]], dtype=torch.float64, device="cuda")
    H[1, 2] += 0.21 * H[1, 8]
    s64, H64 = src.double().requires_grad_(True), H.clone().requires_grad_(True)
    out = warp64(s64, H64.reshape(-1, 3, 3), (dh, dw))
    ws, wH = torch.autograd.grad((out * g.double()).sum(), (s64, H64))
    gs, gH = align.warp_adjoint(g, src, H)
    assert float((gs.double() - ws).abs().max()) <= 1e-4 * max(1.0, float(ws.abs().max()))
    _, gH_only = align.warp_adjoint(g, src, H, want_src=False)
    _check_gH(gH, wH, H, g, "dL/dH beside dL/dsource")
    _check_gH(gH_only, wH, H, g, "dL/dH alone")

    # the fused loss: weight * sum (warp - target)^2 and its gradients, accumulated
    l2 = align.L2Grad(src, g)
    loss, gHl = torch.full((2,), 1.5, dtype=torch.float64, device="cuda"), torch.zeros((2, 9), dtype=torch.float64, device="cuda")
    gsl = torch.zeros_like(src)
    l2(H, 0.25, loss, gHl, accumulate=True, gsrc=gsl)
    res = warp64(s64, H64.reshape(-1, 3, 3), (dh, dw)) - g.double()
    want = 0.25 * (res ** 2).sum(dim=(1, 2))
    ws, wH = torch.autograd.grad(want.sum(), (s64, H64))
    assert float((loss - 1.5 - want).abs().max()) <= 1e-4 * max(1.0, float(want.abs().max()))
    assert float((gsl.double() - ws).abs().max()) <= 1e-4 * max(1.0, float(ws.abs().max()))
    _check_gH(gHl, wH, H, 0.5 * res.detach(), "dL/dH of the loss")


@pytest.mark.parametrize("scale,gscale,sscale", [(2.0 ** -133, 2.0 ** -40, 1.0), (2.0 ** -126, 8.0, 2.0 ** -30), (2.0 ** 126, 8.0, 1.0)])
def test_adjoint_z_at_the_ends_of_f32(gpu, scale, gscale, sscale):
    """1 / z, or dL/d(out) / z, outgrows an F32 but dL/d(out) dI/du / z does not.  The shift by (1.5, -2.5) is
    exact in F32, so what is left is the sums' rounding: below 130 * 70 terms of one size, 1e-5 of the largest."""
    print(f"adjoint, z = {scale}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    src = (torch.rand((1, 37, 130), generator=gen, device="cuda") > 0.5).float() * sscale
    src[:, :, 64:] = 0.0                                     # no slope: dL/d(out) / z meets 0
    g = (torch.randint(1, 3, (1, 35, 127), generator=gen, device="cuda")).float() * gscale
    H = torch.tensor([[1, 0, 1.5, 0, 1, -2.5, 0, 0, 1]], dtype=torch.float64, device="cuda") * scale
    s64, H64 = src.double().requires_grad_(True), H.clone().requires_grad_(True)
    out = warp64(s64, H64.reshape(-1, 3, 3), (35, 127))
    ws, wH = torch.autograd.grad((out * g.double()).sum(), (s64, H64))
    for want_src in (True, False):
        gs, gH = align.warp_adjoint(g, src, H, want_src=want_src)
        assert torch.isfinite(gH).all(), f"dL/dH {gH}"
        assert float((gH - wH).abs().max()) <= 1e-5 * float(wH.abs().max()), f"{gH}\n{wH}"
        if want_src:
            assert float((gs.double() - ws).abs().max()) <= 1e-5 * float(ws.abs().max())


# u and v are exact in F32 and no sample lies on a cell boundary: multiples of 1/4 (1/8) plus 1/8 (1/16)
EXACT = {"shift": [1, 0, 3.125, 0, 1, -2.375, 0, 0, 1], "shrink_rotate": [1.5, 0.5, 0.125, -0.75, 1.25, 30.375, 0, 0, 1],
         "enlarge": [0.25, 0, 0.125, 0, 0.375, 0.0625, 0, 0, 1]}


@pytest.mark.parametrize("name", EXACT)
@pytest.mark.parametrize("n,w,h", [(4, 1021, 1003), (350, 130, 37), (704, 63, 83)])
def test_adjoint_batches_of_eight_rows(gpu, n, w, h, name):
    """batches of 2048 tiles and more, whose waves take eight rows each: last row groups cut off, all four kernels.
    Positions and weights are exact, so what is left is the rounding of terms and F32 partial sums (of at most 8
    rows and 64 columns): dL/dH within 1e-6 of the sum of its terms' sizes, a gradient of the source, a sum of at
    most 16 terms below 1, within 1e-5, the loss within 1e-5 of itself."""
    print(f"adjoint of eight-row waves, {name}: {n} images of {w}x{h}", flush=True)
    assert n * -(-w // 64) * -(-h // 32) >= 2048
    gen = torch.Generator(device="cuda").manual_seed(11)
    src = torch.rand((n, h, w), generator=gen, device="cuda")
    g = torch.rand((n, h, w), generator=gen, device="cuda") - 0.3
    g[:, ::3, ::5] = 0.0
    H = torch.tensor([EXACT[name]], dtype=torch.float64, device="cuda").repeat(n, 1)
    H[:, 2] += torch.arange(n, device="cuda") % 7                  # each image its own
    H[:, 5] -= torch.arange(n, device="cuda") % 5
    s64, H64 = src.double().requires_grad_(True), H.clone().requires_grad_(True)
    out = warp64(s64, H64.reshape(-1, 3, 3), (h, w))
    ys, xs = torch.meshgrid(torch.arange(h, dtype=torch.float64, device="cuda"), torch.arange(w, dtype=torch.float64, device="cuda"),
                            indexing="ij")
    u, v = (H[:, k, None, None] * xs + H[:, k + 1, None, None] * ys + H[:, k + 2, None, None] for k in (0, 3))
    inside = (u > -1) & (u < w) & (v > -1) & (v < h)
    terms = (torch.sqrt(1 + xs * xs + ys * ys) * torch.sqrt(1 + u * u + v * v)) * inside

    def close(gH, gs, loss, what, gout):
        wantS, wantH = torch.autograd.grad(loss, (s64, H64), retain_graph=True)
        err, bound = (gH - wantH).abs().amax(1), 1e-6 * (terms * gout.abs()).sum((1, 2))
        print(f"  {what}: {float((err / wantH.abs().amax(1)).max()):.1e} of dL/dH off, bound {float((bound / wantH.abs().amax(1)).max()):.1e}", flush=True)
        assert (err <= bound).all(), f"{what}: image {int((err / bound).argmax())}"
        if gs is not None:
            assert float((gs.double() - wantS).abs().max()) <= 1e-5, what

    for want_src in (True, False):
        gs, gH = align.warp_adjoint(g, src, H, want_src=want_src)
        close(gH, gs, (out * g.double()).sum(), f"dL/dH, dL/dsource {want_src}", g.double())
    res = out - g.double()
    want = 0.25 * (res ** 2).sum(dim=(1, 2))
    l2 = align.L2Grad(src, g)
    for gsrc in (torch.zeros_like(src), None):
        loss, gH = torch.zeros(n, dtype=torch.float64, device="cuda"), torch.zeros((n, 9), dtype=torch.float64, device="cuda")
        l2(H, 0.25, loss, gH, accumulate=False, gsrc=gsrc)
        assert float(((loss - want.detach()) / want.detach()).abs().max()) <= 1e-5
        close(gH, gsrc, want.sum(), f"the loss, dL/dsource {gsrc is not None}", 0.5 * res.detach())
