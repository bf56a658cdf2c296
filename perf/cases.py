"""The measured workloads: what a user of this framework has it do, called as a user's program calls it.

``listed()`` holds twelve cases over the real range of the vision path -- from one small graph, where
launches and the host path count, to a batch of sixteen 4K frames -- and ``draw(rng)`` gives further
cases of the same ranges.  ``prepare`` makes the device inputs and the plans, workspaces or graphs that
a program keeps; ``run`` is one pass through the public entry points and returns every output whole.

Integer paths reproduce the reference CPU's bytes, so their outputs have to be the same bytes; the F32
warp is compared with a tolerance and with plain float64 torch (``exact``).
"""
import ctypes as c
import math

import numpy as np
import torch

from mivisionx_amd import align, kernels, synth
from mivisionx_amd import openvx as vx
from mivisionx_amd.device import Plane, align16, call
from mivisionx_amd.pipelines import (Canny, ChainImage, ChainPlan, Harris, PyrLKTracker, VisionFrame, VisionParams, harris_norm,
                                     pyramid_dims)

DEV = "cuda"
KEYPOINT_BYTES = 28
CORNERS = 16384          # keypoints a caller's array holds
LEVELS = 5               # pyramid levels of the vision graph


def listed():
    return [
        # offline / multi-camera analysis: sixteen resident 4K frames per call of the fused vision graph
        # (luma, half-size image, 5-level Gaussian pyramid, Canny edges, Harris corners)
        dict(name="vision_4k_x16", kind="vision", w=3840, h=2160, frames=16),
        # a live camera: the same graph, one frame per call, a ragged size (tiles cut at both edges)
        dict(name="vision_1284x726_x1", kind="vision", w=1284, h=726, frames=1),
        # the smallest call: a verified OpenVX graph (gradient chain) on a QVGA image, vxProcessGraph
        dict(name="engine_chain_320x240", kind="engine", graph="chain", w=320, h=240),
        # photo collections: 48 images of uneven sizes through the gradient chain in one launch
        dict(name="chain_batch_48", kind="chain_batch", n=48, wmax=4096, hmax=2160, step=16, merged=False),
        # edge detection of one 4K frame with the 5x5 gradient and the L2 norm
        dict(name="canny_4k_g5_l2", kind="canny", w=3840, h=2160, gradient=5, l2=True),
        # corner detection of one 4K frame, FAST with suppression
        dict(name="fast_4k", kind="corners", op="fast", w=3840, h=2160),
        # tracking 10,000 points between two 4K frames, both pyramids built in the pass
        dict(name="lk_4k_10000", kind="lk", w=3840, h=2160, points=10000, window=9),
        # stabilisation / rectification of one 4K frame
        dict(name="warp_perspective_4k", kind="warp", op="perspective", nearest=False, constant=True, w=3840, h=2160),
        # 360-degree stitching: six 1080p cameras into one equirectangular frame
        dict(name="stitch_7680x3840", kind="stitch", w=7680, h=3840, cams=6, sw=1920, sh=1080),
        # a decoded video frame made RGB for display or a network
        dict(name="color_nv12_rgb_1080", kind="color", op="RGB_NV12", w=1920, h=1080),
        # gradient-based alignment: loss and dL/dH of 64 pairs over three pyramid levels
        dict(name="align_l2_64x1024", kind="align", op="l2", n=64, w=1024, h=1024),
        # the differentiable warp inside a training step: forward, then dL/dsource and dL/dH
        dict(name="warp_f32_vjp_8x509x387", kind="align", op="vjp", n=8, w=509, h=387),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vision", "engine", "chain_batch", "canny", "corners", "lk", "warp", "stitch", "color", "align"])
    w, h = _log(rng, 160, 3840), _log(rng, 120, 2160)
    if kind == "vision":
        w, h = w // 4 * 4, h // 2 * 2
        return dict(kind=kind, w=w, h=h, frames=_log(rng, 1, 16))
    if kind == "engine":
        graph = rng.choice(["chain", "filters"])
        return dict(kind=kind, graph=graph, w=w, h=h)
    if kind == "chain_batch":
        return dict(kind=kind, n=_log(rng, 1, 48), wmax=_log(rng, 340, 4096), hmax=_log(rng, 260, 2160), step=rng.choice([2, 16]),
                    merged=rng.random() < 0.3)
    if kind == "canny":
        return dict(kind=kind, w=w, h=h, gradient=rng.choice([3, 5, 7]), l2=rng.random() < 0.5)
    if kind == "corners":
        return dict(kind=kind, op=rng.choice(["fast", "harris"]), w=w, h=h)
    if kind == "lk":
        return dict(kind=kind, w=max(w, 320), h=max(h, 240), points=_log(rng, 100, 10000), window=rng.choice([5, 7, 9, 11]))
    if kind == "warp":
        return dict(kind=kind, op=rng.choice(["affine", "perspective", "remap"]), nearest=rng.random() < 0.3,
                    constant=rng.random() < 0.5, w=w, h=h)
    if kind == "stitch":
        sw = _log(rng, 320, 1920) // 2 * 2
        return dict(kind=kind, w=4 * sw // 8 * 8, h=2 * sw, cams=rng.choice([4, 6, 8]), sw=sw, sh=sw * 9 // 16)
    if kind == "color":
        return dict(kind=kind, op=rng.choice(sorted(_COLOR)), w=w // 2 * 2, h=h // 2 * 2)
    return dict(kind=kind, op=rng.choice(["l2", "vjp"]), n=_log(rng, 1, 16), w=_log(rng, 120, 1024), h=_log(rng, 120, 1024))


# ------------------------------------------------------------------ inputs ---------------------
def _scene(w, h, seed):
    """an image like those the path meets: smooth structure, sharp rectangles, sensor noise"""
    return synth.scene_u8_device(w, h, seed, DEV)


def _plane(img):
    h, w = img.shape
    p = Plane(w, h)
    p.t[:, :w].copy_(img)
    return p


def _zeros(*shape, dtype=torch.uint8):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _ptr(t):
    return c.c_void_p(t.data_ptr())


def _stream():
    return c.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ok(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what} returned {rc}")


# ------------------------------------------------------------------ the fused vision graph -----
def _prepare_vision(case, seed):
    w, h, n = case["w"], case["h"], case["frames"]
    K = kernels()
    K.mvx_VisionGraph_workspace_size.restype = c.c_size_t
    params = VisionParams(w, h, w // 2, h // 2, LEVELS, 80, 100, 0.04, 0.0005, 5.0, CORNERS)
    dims = pyramid_dims(w, h, LEVELS)
    lv = [(align16(a), b) for a, b in dims]
    sstride = align16(w // 2)
    rgb = _zeros(n, h, align16(3 * w))
    for f in range(n):
        for ch in range(3):
            rgb[f, :, ch:3 * w:3].copy_(_scene(w, h, (seed * 16 + f) * 3 + ch))
    pyr = [_zeros(n, b, a) for a, b in lv]
    scaled, edges = _zeros(n, h // 2, sstride), _zeros(n, h, align16(w))
    corners = _zeros(n, CORNERS * KEYPOINT_BYTES)
    items, count = _zeros(n, dtype=torch.int32), _zeros(n, dtype=torch.int64)
    table = (VisionFrame * n)()
    for f in range(n):
        d = table[f]
        d.rgb, d.rgbStride = rgb[f].data_ptr(), align16(3 * w)
        for k, (a, _) in enumerate(lv):
            d.pyramid[k], d.pyramidStride[k] = pyr[k][f].data_ptr(), a
        d.scaled, d.scaledStride = scaled[f].data_ptr(), sstride
        d.edges, d.edgesStride = edges[f].data_ptr(), align16(w)
        d.corners, d.numItems, d.numCorners = corners[f].data_ptr(), items[f].data_ptr(), count[f].data_ptr()
    size = K.mvx_VisionGraph_workspace_size(c.byref(params), n)
    ws = _zeros(max(size, 16))
    _ok(K.mvx_VisionGraph_prepare(_stream(), c.byref(params), table, n, _ptr(ws), c.c_size_t(size)), "mvx_VisionGraph_prepare")
    return dict(K=K, params=params, n=n, ws=ws, size=size, rgb=rgb, table=table,
                out=dict(pyramid=pyr, scaled=scaled, edges=edges, corners=corners, items=items, count=count))


def _run_vision(s):
    _ok(s["K"].mvx_VisionGraph_run(_stream(), c.byref(s["params"]), s["n"], _ptr(s["ws"]), c.c_size_t(s["size"])), "mvx_VisionGraph_run")
    return s["out"]


# ------------------------------------------------------------------ OpenVX graphs --------------
class _Graph:
    """a verified graph over device images the caller owns (VX_MEMORY_TYPE_HIP handles)"""

    def __init__(self):
        self.L = vx.lib()
        self.ctx = self.L.vxCreateContext()
        self.graph = self.L.vxCreateGraph(self.ctx)
        self.planes = []

    def image(self, plane):
        self.planes.append(plane)
        addr = vx.Addressing(plane.width, plane.height, plane.bpp, plane.stride, 1024, 1024, 1, 1, 0)
        return self.L.vxCreateImageFromHandle(self.ctx, vx.DF[plane.fmt], c.byref(addr), (c.c_void_p * 1)(plane.t.data_ptr()),
                                              vx.VX_MEMORY_TYPE_HIP)

    def virtual(self):
        return self.L.vxCreateVirtualImage(self.graph, 0, 0, vx.DF["VIRT"])

    def __del__(self):
        g, ctx = c.c_void_p(self.graph), c.c_void_p(self.ctx)
        self.L.vxReleaseGraph(c.byref(g))
        self.L.vxReleaseContext(c.byref(ctx))


def _prepare_engine(case, seed):
    w, h = case["w"], case["h"]
    g = _Graph()
    L = g.L
    src = g.image(_plane(_scene(w, h, seed)))
    if case["graph"] == "chain":      # Gaussian -> Sobel -> Magnitude and Phase, every result kept
        outs = [Plane(w, h, f) for f in ("S16", "S16", "S16", "U8")]
        o = [g.image(p) for p in outs]
        blur = g.virtual()
        nodes = [L.vxGaussian3x3Node(g.graph, src, blur), L.vxSobel3x3Node(g.graph, blur, o[0], o[1]),
                 L.vxMagnitudeNode(g.graph, o[0], o[1], o[2]), L.vxPhaseNode(g.graph, o[0], o[1], o[3])]
    else:                             # denoise, smooth and shrink: Median, Box, Gaussian -> half size
        outs = [Plane(w, h), Plane(w, h), Plane(max(w // 2, 1), max(h // 2, 1))]
        o = [g.image(p) for p in outs]
        blur = L.vxCreateVirtualImage(g.graph, w, h, vx.DF["U8"])
        nodes = [L.vxMedian3x3Node(g.graph, src, o[0]), L.vxBox3x3Node(g.graph, src, o[1]), L.vxGaussian3x3Node(g.graph, src, blur),
                 L.vxScaleImageNode(g.graph, blur, o[2], vx.VX_INTERPOLATION_BILINEAR)]
    if not all(nodes):
        raise RuntimeError("a node was refused")
    vx.check(L.vxVerifyGraph(g.graph), "vxVerifyGraph")
    return dict(g=g, out=[p.t for p in outs])


def _run_engine(s):
    vx.check(s["g"].L.vxProcessGraph(s["g"].graph), "vxProcessGraph")
    return s["out"]


# ------------------------------------------------------------------ uneven batch ---------------
def _batch_sizes(case):
    """sizes from 320 x 240 up to the case's largest, even numbers in steps of `step`"""
    u = synth.u32(7, 4, 2 * case["n"]).astype(np.float64) / 4294967296.0
    st = case["step"]
    ws = 320 + st * np.floor(u[0::2] * ((case["wmax"] - 320) // st + 1)).astype(np.int64)
    hs = 240 + st * np.floor(u[1::2] * ((case["hmax"] - 240) // st + 1)).astype(np.int64)
    return [(int(a), int(b)) for a, b in zip(ws, hs)]


def _prepare_chain_batch(case, seed):
    K = kernels()
    K.mvx_ChainBatch_workspace_size.restype = c.c_size_t
    sizes = _batch_sizes(case)
    n = len(sizes)
    out = {}
    roles = {"mag": (2, 1), "phase": (1, 1), "half": (1, 2)}
    if not case["merged"]:
        roles.update({"gx": (2, 1), "gy": (2, 1)})
    where = {}
    for role, (bpp, div) in roles.items():
        at, size = [], 0
        for w, h in sizes:
            at.append(size)
            size += (align16(w // div * bpp) * (h // div) + 255) // 256 * 256
        out[role], where[role] = _zeros(size), at
    srcs = [_plane(_scene(w, h, seed * 64 + i)) for i, (w, h) in enumerate(sizes)]
    arr = (ChainImage * n)()
    for i, (w, h) in enumerate(sizes):
        a = {r: (out[r].data_ptr() + where[r][i], align16(w // d * b)) for r, (b, d) in roles.items()}
        gx, gy = a.get("gx", (None, 0)), a.get("gy", (None, 0))
        arr[i] = ChainImage(srcs[i].t.data_ptr(), w, h, srcs[i].stride, gx[0], gx[1], gy[0], gy[1], a["mag"][0], a["mag"][1],
                            a["phase"][0], a["phase"][1], a["half"][0], a["half"][1])
    size = K.mvx_ChainBatch_workspace_size(n)
    ws, plan = _zeros(size), ChainPlan()
    _ok(K.mvx_ChainBatch_prepare(arr, n, 4, 0, _ptr(ws), c.c_size_t(size), c.byref(plan)), "mvx_ChainBatch_prepare")
    return dict(K=K, plan=plan, ws=ws, srcs=srcs, out=out)


def _run_chain_batch(s):
    _ok(s["K"].mvx_ChainBatch_run(_stream(), c.byref(s["plan"])), "mvx_ChainBatch_run")
    return s["out"]


# ------------------------------------------------------------------ Canny ----------------------
def _prepare_canny(case, seed):
    w, h, g = case["w"], case["h"], case["gradient"]
    # thresholds that keep a few percent of the pixels: the 5x5 and 7x7 kernels give larger gradients
    lo, hi = {3: (80, 100), 5: (500, 900), 7: (700, 1400)}[g]
    return dict(canny=Canny(w, h), src=_plane(_scene(w, h, seed)), dst=Plane(w, h), lo=lo, hi=hi,
                sobel=f"CannySobel_U16_U8_{g}x{g}_L{2 if case['l2'] else 1}NORM")


def _run_canny(s):
    k, src, dst = s["canny"], s["src"], s["dst"]
    w, h = k.w, k.h
    call(s["sobel"], w, h, k.mag, k.mag.stride, src, src.stride)
    call("CannySuppThreshold_U8XY_U16_3x3", w, h, dst, dst.stride, k.mag, k.mag.stride, _ptr(k.stack), w * h, s["lo"], s["hi"])
    call("CannyEdgeTrace_U8_U8XY", w, h, dst, dst.stride, _ptr(k.stack), w * h)
    return dst.t


# ------------------------------------------------------------------ corners --------------------
def _prepare_corners(case, seed):
    w, h = case["w"], case["h"]
    src = _plane(_scene(w, h, seed))
    if case["op"] == "harris":
        return dict(harris=Harris(w, h, CORNERS), src=src, norm=harris_norm(3))
    K = kernels()
    K.mvx_FastCorners_workspace_size.restype = c.c_size_t
    size = int(K.mvx_FastCorners_workspace_size(w, h))
    return dict(harris=None, src=src, ws=_zeros(size), size=size, corners=_zeros(CORNERS * KEYPOINT_BYTES),
                items=_zeros(1, dtype=torch.int32), count=_zeros(1, dtype=torch.int64))


def _run_corners(s):
    hr, src = s["harris"], s["src"]
    if hr is not None:
        hr.run(src, 0.04, 0.0005, 5.0, s["norm"])
        return [hr.corners, hr.num_items, hr.count]
    call("FastCorners_XY_U8_Supression", CORNERS, _ptr(s["corners"]), _ptr(s["items"]), _ptr(s["count"]), src.width, src.height, src,
         src.stride, 30.0, _ptr(s["ws"]), c.c_size_t(s["size"]))
    return [s["corners"], s["items"], s["count"]]


# ------------------------------------------------------------------ optical flow ---------------
def _prepare_lk(case, seed):
    w, h = case["w"], case["h"]
    old = _scene(w, h, seed)
    p = synth.uniform01(seed, 600, 2)      # the scene moves by 2 to 8 pixels
    tx, ty = (2 + 6 * p[0]) * math.cos(2 * math.pi * p[1]), (2 + 6 * p[0]) * math.sin(2 * math.pi * p[1])
    ix, iy = math.floor(tx), math.floor(ty)
    fx, fy = tx - ix, ty - iy
    f = old.to(torch.float32)
    sh = [torch.roll(f, (iy + b, ix + a), (0, 1)) for b in (0, 1) for a in (0, 1)]
    new = torch.round((sh[0] * (1 - fx) + sh[1] * fx) * (1 - fy) + (sh[2] * (1 - fx) + sh[3] * fx) * fy).to(torch.uint8)
    dims = pyramid_dims(w, h, 4)
    imgs = [_plane(old), _plane(new)]
    pyrs = [[Plane(a, b) for a, b in dims] for _ in range(2)]
    tr = PyrLKTracker(pyrs[0], pyrs[1], case["points"])
    tr.set_points(synth.lk_keypoints(w, h, case["points"], seed))
    return dict(imgs=imgs, pyrs=pyrs, tr=tr, dims=dims, window=case["window"])


def _run_lk(s):
    dims, tr = s["dims"], s["tr"]
    for img, lv in zip(s["imgs"], s["pyrs"]):
        call("ChannelCopy_U8_U8", dims[0][0], dims[0][1], lv[0], lv[0].stride, img, img.stride)
        for k in range(1, len(dims)):
            call("ScaleGaussianHalf_U8_U8_5x5", dims[k][0], dims[k][1], lv[k], lv[k].stride, dims[k - 1][0], dims[k - 1][1], lv[k - 1],
                 lv[k - 1].stride)
    tr.run(0xF002, 0.01, 20, False, s["window"])
    return [tr.out, tr.out_count] + [p.t for lv in s["pyrs"] for p in lv]


# ------------------------------------------------------------------ warps ----------------------
def _barrel(w, h, k1):
    yy, xx = torch.meshgrid(torch.arange(h, dtype=torch.float64, device=DEV), torch.arange(w, dtype=torch.float64, device=DEV), indexing="ij")
    cx, cy = (w - 1) / 2.0, (h - 1) / 2.0
    rn = math.hypot(cx, cy)
    dx, dy = (xx - cx) / rn, (yy - cy) / rn
    f = 1.0 + k1 * (dx * dx + dy * dy)
    return torch.stack([cx + dx * f * rn, cy + dy * f * rn], -1).to(torch.float32).contiguous()


def _prepare_warp(case, seed):
    w, h, op = case["w"], case["h"], case["op"]
    interp = "Nearest" if case["nearest"] else "Bilinear"
    tail = "_Constant" if case["constant"] else ""
    src, dst = _plane(_scene(w, h, seed)), Plane(w, h)
    s = dict(w=w, h=h, src=src, dst=dst, keep=None)
    if op == "remap":
        fixed, m = _zeros(h, 4 * w), _barrel(w, h, 0.05 + 0.1 * float(synth.uniform01(seed, 900, 1)[0]))
        call("Remap_FixedMap_F32", w, h, _ptr(fixed), 4 * w, _ptr(m), 8 * w, w, h)
        s["keep"] = fixed
        s["name"] = f"Remap_U8_U8_{interp}{tail}"
        whole = [] if case["constant"] and not case["nearest"] else [src.stride * h]   # srcImageBufferSize
        s["args"] = whole + [_ptr(fixed), 4 * w] + ([c.c_uint8(0)] if case["constant"] else [])
    else:
        aff, per = synth.warp_matrices(w, h, seed)
        s["keep"] = np.ascontiguousarray(aff if op == "affine" else per)
        s["name"] = f"Warp{op.capitalize()}_U8_U8_{interp}{tail}"
        s["args"] = [s["keep"].ctypes.data_as(c.c_void_p)]
        if case["constant"]:
            s["args"] += [c.c_uint8(0)] + ([None] if op == "affine" and case["nearest"] else [])
    return s


def _run_warp(s):
    w, h, src, dst = s["w"], s["h"], s["src"], s["dst"]
    tail = [src, src.stride] + s["args"]
    call(s["name"], w, h, dst, dst.stride, w, h, *tail)
    return dst.t


# ------------------------------------------------------------------ stitching ------------------
def _prepare_stitch(case, seed):
    """`cams` pinhole cameras (90 degrees wide) around the vertical axis and Loom's selection maps: a
    group of 8 output pixels takes one camera, or two where their 64-pixel seam ramps overlap"""
    W, H, n, sw, sh = case["w"], case["h"], case["cams"], case["sw"], case["sh"]
    G = W // 8
    f, cx, cy = sw / 2.0, (sw - 1) / 2.0, (sh - 1) / 2.0
    lon = (torch.arange(W, dtype=torch.float64, device=DEV) + 0.5) / W * 2 * math.pi - math.pi
    lat = (math.pi / 2 - (torch.arange(H, dtype=torch.float64, device=DEV) + 0.5) / H * math.pi)[:, None]
    jitter = synth.uniform01(seed, 4100, n)
    cams, used, full = [], [], []
    fixed, weights = _zeros(n * H, 4 * W), _zeros(n * H, W)
    for k in range(n):
        yaw = math.radians(360.0 / n * k - 2 + 4 * float(jitter[k]))
        d = torch.remainder(lon[None, :] - yaw + math.pi, 2 * math.pi) - math.pi
        z = torch.cos(lat) * torch.cos(d)
        zs = torch.where(z > 1e-6, z, torch.ones_like(z))
        mx, my = cx + f * torch.cos(lat) * torch.sin(d) / zs, cy - f * torch.sin(lat) / zs
        inside = (z > 1e-6) & (mx >= 0) & (my >= 0) & (mx <= sw - 1) & (my <= sh - 1)
        m = torch.where(inside[..., None], torch.stack([mx, my], -1), -1.0).to(torch.float32).contiguous()
        call("Remap_FixedMap_F32", W, H, _ptr(fixed[k * H:]), 4 * W, _ptr(m), 8 * W, sw, sh)
        ramp = torch.clamp(0.5 + (math.pi / n - torch.abs(d)) * W / (2 * math.pi) / 64, 0, 1)
        wt = torch.round(ramp * 255).expand(H, W) * inside
        weights[k * H:(k + 1) * H].copy_(wt)
        g = wt.reshape(H, G, 8)
        used.append((g > 0).any(-1))
        full.append((g == 255).all(-1))
        cam = Plane(sw, sh, "RGB")
        for ch in range(3):
            cam.t[:, ch:3 * sw:3].copy_(_scene(sw, sh, (seed * 8 + k) * 3 + ch))
        cams.append(cam)
        del m, mx, my, inside, wt, z, zs
    used, full = torch.stack(used), torch.stack(full)
    count = used.sum(0)
    ids = torch.full((3, H, G), 31, dtype=torch.int32, device=DEV)
    rank = torch.cumsum(used.to(torch.int32), 0) - 1
    for k in range(n):
        for j in range(3):
            ids[j].masked_fill_(used[k] & (rank[k] == j), k)
    single = (count == 1) & (used & full).any(0)
    id0 = torch.where(count == 0, 31, torch.where(single, ids[0], 128 + torch.clamp(count - 2, min=0))).to(torch.uint8).contiguous()
    id1 = (ids[0] | (ids[1] << 5) | (ids[2] << 10)).to(torch.int16).contiguous()
    id2 = torch.full((H, G), 31 | (31 << 5) | (31 << 10), dtype=torch.int16, device=DEV)
    out = Plane(W, H, "RGB")
    args = [W, H, out, out.stride, n, (c.c_void_p * n)(*[p.t.data_ptr() for p in cams]), (c.c_uint32 * n)(*[p.stride for p in cams]),
            sw, sh, _ptr(fixed), 4 * W, _ptr(weights), W, _ptr(id0), G, _ptr(id1), 2 * G, _ptr(id2), 2 * G]
    return dict(out=out, args=args, keep=(cams, fixed, weights, id0, id1, id2))


def _run_stitch(s):
    call("Stitch_Loom_RGB", *s["args"])
    return s["out"].t


# ------------------------------------------------------------------ colour ---------------------
# entry point (destination_source): planes of the destination, then of the source, as (bytes per
# sample, chroma subsampling)
_ONE = {"RGB": [(3, 1)], "RGBX": [(4, 1)], "UYVY": [(2, 1)], "NV12": [(1, 1), (2, 2)], "NV21": [(1, 1), (2, 2)],
        "IYUV": [(1, 1), (1, 2), (1, 2)], "YUV4": [(1, 1), (1, 1), (1, 1)], "Y": [(1, 1)]}
_COLOR = {op: tuple(op.split("_")) for op in ("RGB_NV12", "RGB_IYUV", "RGBX_NV12", "RGB_UYVY", "RGBX_UYVY", "IYUV_RGB", "NV12_RGB",
                                              "YUV4_RGB", "Y_RGB", "RGBX_RGB", "RGB_RGBX", "NV12_UYVY")}


class _Raw:
    """a plane of any sample width in the framework's layout (rows padded to 16 bytes)"""

    def __init__(self, w, h, bpp):
        self.stride = align16(w * bpp)
        self.t = _zeros(h, self.stride)


def _prepare_color(case, seed):
    w, h = case["w"], case["h"]
    dst_f, src_f = _COLOR[case["op"]]
    dst = [_Raw(w // s, h // s, b) for b, s in _ONE[dst_f]]
    src = [_Raw(w // s, h // s, b) for b, s in _ONE[src_f]]
    for k, ((b, s), p) in enumerate(zip(_ONE[src_f], src)):
        for ch in range(b):
            p.t[:, ch:b * (w // s):b].copy_(_scene(w // s, h // s, seed * 16 + 4 * k + ch))
    name = ("FormatConvert_" if case["op"] == "NV12_UYVY" else "ColorConvert_") + case["op"]
    args = [w, h] + [v for p in dst + src for v in (_ptr(p.t), p.stride)]
    return dict(name=name, args=args, dst=dst, src=src)


def _run_color(s):
    call(s["name"], *s["args"])
    return [p.t for p in s["dst"]]


# ------------------------------------------------------------------ F32 warp -------------------
def _align_inputs(case, seed):
    """smooth images in [0, 1], homographies of a few degrees and pixels, and the other image of each
    pair: its mate shifted by a few pixels with sensor noise (l2), or an incoming gradient (vjp)"""
    n, w, h = case["n"], case["w"], case["h"]
    gen = torch.Generator(device=DEV).manual_seed(seed)
    p = torch.rand((n, 6, 4), generator=gen, device=DEV, dtype=torch.float32)
    xs, ys = torch.arange(w, device=DEV, dtype=torch.float32)[None, None, :], torch.arange(h, device=DEV, dtype=torch.float32)[None, :, None]
    src = torch.full((n, h, w), 0.5, device=DEV)
    for k in range(6):
        a, per, th, ph = (p[:, k, j, None, None] for j in range(4))
        fr = 2 * math.pi / (16.0 * torch.exp(per * math.log(32.0)))
        src += 0.08 * a * torch.sin(fr * torch.cos(math.pi * th) * xs + fr * torch.sin(math.pi * th) * ys + 2 * math.pi * ph)
    src = src.clamp_(0, 1)
    noise = torch.randn((n, h, w), generator=gen, device=DEV)
    other = (torch.roll(src, (2, -3), (1, 2)) + 0.01 * noise) if case["op"] == "l2" else noise
    q = align.true_params(n, w, h, 5100 + 64 * (seed % 4096)) * 0.25
    s = w / 2.0
    N = np.array([[1 / s, 0, -1], [0, 1 / s, -(h / 2.0) / s], [0, 0, 1]])
    Hh = np.zeros((n, 9))
    Hh[:, :8] = q
    Hh = np.linalg.inv(N) @ (np.eye(3) + Hh.reshape(n, 3, 3)) @ N
    return src, other.contiguous(), torch.as_tensor(Hh, device=DEV)


def _align_levels(case, src, tgt, Hh):
    """(source, target, homography, weight) per pyramid level: 2x2 means, S H S^-1"""
    out = []
    for lv in range(3 if min(case["w"], case["h"]) >= 64 else 1):
        s = 0.5 ** lv
        S, Si = (torch.diag(torch.tensor([v, v, 1.0], dtype=torch.float64, device=DEV)) for v in (s, 1 / s))
        out.append((src, tgt, (S @ Hh @ Si).reshape(-1, 9).contiguous(), 1.0 / (src.shape[1] * src.shape[2])))
        a, b = src.shape[1] // 2 * 2, src.shape[2] // 2 * 2
        src, tgt = (((t[:, :a:2, :b:2] + t[:, 1:a:2, :b:2]) + (t[:, :a:2, 1:b:2] + t[:, 1:a:2, 1:b:2])).mul(0.25).contiguous() for t in (src, tgt))
    return out


def _prepare_align(case, seed):
    src, other, Hh = _align_inputs(case, seed)
    n = case["n"]
    if case["op"] == "vjp":
        return dict(src=src, grad=other, H=Hh.reshape(n, 9).contiguous())
    lv = _align_levels(case, src, other, Hh)
    return dict(levels=[(align.L2Grad(a, b), Hl, wt, _zeros(n, dtype=torch.float64), _zeros(n, 9, dtype=torch.float64)) for a, b, Hl, wt in lv])


def _run_align(s):
    if "grad" in s:
        out = align.warp(s["src"], s["H"])
        return [out, *align.warp_adjoint(s["grad"], s["src"], s["H"])]
    for l2, Hl, wt, loss, gH in s["levels"]:
        l2(Hl, wt, loss, gH, accumulate=False)
    return [v for _, _, _, loss, gH in s["levels"] for v in (loss, gH)]


def _exact_warp(src, Hm, grad, scatter):
    """one image in float64: (warp, dL/dsrc or None, dL/dH) for dL/d(out) = grad(out)"""
    h, w = src.shape
    yy, xx = torch.meshgrid(torch.arange(h, dtype=torch.float64, device=DEV), torch.arange(w, dtype=torch.float64, device=DEV), indexing="ij")
    m = Hm.tolist()
    X, Y, z = m[0] * xx + m[1] * yy + m[2], m[3] * xx + m[4] * yy + m[5], m[6] * xx + m[7] * yy + m[8]
    ok = z > 0
    zs = torch.where(ok, z, torch.ones_like(z))
    u, v = X / zs, Y / zs
    x0, y0 = torch.floor(u).clamp(-2, w + 1), torch.floor(v).clamp(-2, h + 1)
    fx, fy = torch.where(ok, u - x0, 0 * u), torch.where(ok, v - y0, 0 * u)
    pix, at, val = {}, {}, {}
    for j in (0, 1):
        for i in (0, 1):
            xi, yi = (x0 + i).long(), (y0 + j).long()
            inn = ok & (xi >= 0) & (xi < w) & (yi >= 0) & (yi < h)
            at[i, j] = (yi.clamp(0, h - 1) * w + xi.clamp(0, w - 1)).reshape(-1)
            val[i, j] = inn.to(torch.float64)
            pix[i, j] = src.reshape(-1)[at[i, j]].reshape(h, w) * val[i, j]
    out = (pix[0, 0] * (1 - fx) + pix[1, 0] * fx) * (1 - fy) + (pix[0, 1] * (1 - fx) + pix[1, 1] * fx) * fy
    g = grad(out)
    du = ((pix[1, 0] - pix[0, 0]) * (1 - fy) + (pix[1, 1] - pix[0, 1]) * fy) * g / zs
    dv = ((pix[0, 1] - pix[0, 0]) * (1 - fx) + (pix[1, 1] - pix[1, 0]) * fx) * g / zs
    dz = -(du * u + dv * v)
    gH = torch.stack([(d * q).sum() for d in (du, dv, dz) for q in (xx, yy, torch.ones_like(xx))])
    gsrc = None
    if scatter:
        gsrc = torch.zeros(h * w, dtype=torch.float64, device=DEV)
        for (i, j), idx in at.items():
            wt = (fx if i else 1 - fx) * (fy if j else 1 - fy) * val[i, j]
            gsrc.index_add_(0, idx, (wt * g).reshape(-1))
        gsrc = gsrc.reshape(h, w)
    return out, gsrc, gH


def exact(case, seed):
    """the F32 warp in float64; the integer paths are compared byte for byte instead"""
    if case["kind"] != "align":
        return None
    src, other, Hh = _align_inputs(case, seed)
    if case["op"] == "vjp":
        r = [_exact_warp(src[i].double(), Hh[i].reshape(9), lambda o, i=i: other[i].double(), True) for i in range(case["n"])]
        return [torch.stack([v[k] for v in r]) for k in range(3)]
    out = []
    for a, b, Hl, wt in _align_levels(case, src, other, Hh):
        loss, gH = [], []
        for i in range(case["n"]):
            t = b[i].double()
            o, _, g = _exact_warp(a[i].double(), Hl[i], lambda o, t=t, wt=wt: 2 * wt * (o - t), False)
            loss.append(wt * ((o - t) ** 2).sum())
            gH.append(g)
        out += [torch.stack(loss), torch.stack(gH)]
    return out


# ------------------------------------------------------------------ what a pass needs ----------
def work(case):
    """bytes: each input read and each output written once; flops: the arithmetic of the plain
    formulas (operations per pixel counted once, nothing for borders)"""
    k = case["kind"]
    w, h = case.get("w", 0), case.get("h", 0)
    px = w * h
    if k == "vision":
        pyr = sum(a * b for a, b in pyramid_dims(w, h, LEVELS))
        return {"bytes": case["frames"] * (3 * px + px // 4 + pyr + px), "flops": case["frames"] * 90 * px}
    if k == "engine":
        return {"bytes": px * 8, "flops": px * 40} if case["graph"] == "chain" else {"bytes": px * 3.25, "flops": px * 60}
    if k == "chain_batch":
        bpp = 4.25 if case["merged"] else 8.25
        total = sum(a * b for a, b in _batch_sizes(case))
        return {"bytes": total * bpp, "flops": total * 42}
    if k == "canny":
        return {"bytes": 2 * px, "flops": px * {3: 25, 5: 50, 7: 75}[case["gradient"]]}
    if k == "corners":
        return {"bytes": px, "flops": px * (20 if case["op"] == "fast" else 60)}
    if k == "lk":
        pyr = sum(a * b for a, b in pyramid_dims(w, h, 4))
        win = case["window"] ** 2
        return {"bytes": 2 * (px + pyr) + 2 * KEYPOINT_BYTES * case["points"], "flops": 2 * 14 * (pyr - px) + case["points"] * 4 * win * 60}
    if k == "warp":
        return {"bytes": px * (6 if case["op"] == "remap" else 2), "flops": px * 20}
    if k == "stitch":
        # the cameras, the table entry and the output of each pixel, one selection byte per eight
        return {"bytes": case["cams"] * 3 * case["sw"] * case["sh"] + px * (4 + 3) * 0.6 + px / 8, "flops": px * 20}
    if k == "color":
        return {"bytes": px * sum(b / (s * s) for f in _COLOR[case["op"]] for b, s in _ONE[f]), "flops": px * 10}
    n = case["n"]
    if case["op"] == "vjp":
        return {"bytes": n * px * 4 * 4, "flops": n * px * 90}
    levels = sum((w >> i) * (h >> i) for i in range(3 if min(w, h) >= 64 else 1))
    return {"bytes": n * levels * 8, "flops": n * levels * 60}


def tolerance(case):
    if case["kind"] != "align":
        return "exact"        # the reference CPU's bytes
    # F32 sampling and sums: 4e-6 at most against float64 over the drawn range (dL/dH, whose sums of
    # signed terms cancel); another order of the sums moves it by as much
    return {"rel": 2e-5}


_PREPARE = {"vision": _prepare_vision, "engine": _prepare_engine, "chain_batch": _prepare_chain_batch, "canny": _prepare_canny,
            "corners": _prepare_corners, "lk": _prepare_lk, "warp": _prepare_warp, "stitch": _prepare_stitch, "color": _prepare_color,
            "align": _prepare_align}
_RUN = {"vision": _run_vision, "engine": _run_engine, "chain_batch": _run_chain_batch, "canny": _run_canny, "corners": _run_corners,
        "lk": _run_lk, "warp": _run_warp, "stitch": _run_stitch, "color": _run_color, "align": _run_align}


def prepare(case, seed):
    return dict(kind=case["kind"], s=_PREPARE[case["kind"]](case, seed))


def run(state):
    return _RUN[state["kind"]](state["s"])
