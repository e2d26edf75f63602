"""Timed cases of the renderer: what a program that renders, differentiates and
post-processes particle frames asks of this package, from a thumbnail of a
thousand particles to a 16M-particle frame at 2048^2.

listed() names the cases, draw() makes more of the same ranges, prepare() makes
a case's inputs on the GPU from a seed, run() does one pass through the public
entry points, work() counts what the pass cannot do without, and exact() gives
the pass's outputs from plain torch in double precision.

The particle fields follow the package's synthetic generator (Plummer halos in
a uniform background, log-normal smoothing lengths and intensities, uniform
colour scalars), drawn here on the GPU.
"""
import math

import numpy as np
import torch

import splotch_amd as S
from splotch_amd import synth

DEV = "cuda"
BOX = 100.0


# ------------------------------------------------------------------- the cases

def frame(name, n, xres, yres, mode, hsml=0.3, vector=False, grad=False, host=False):
    """One view: n particles (mode "both": half gas, depth-sorted, half stars,
    additive), the image's size, gas smoothing length, vector colours, whether
    the gradient is taken and whether the records come from host memory."""
    return dict(name=name, kind="frame", n=n, xres=xres, yres=yres, mode=mode, hsml=hsml,
                vector=vector, grad=grad, host=host)


def batch(name, views, n_min, n_max, sides, pick, replay=False):
    """Views of log-uniform particle counts around the box, alternately additive
    and ordered (sides: 256-1024 or 96-256 px squares; pick: the draw of counts,
    sides and cameras), in one call, or captured once and replayed."""
    return dict(name=name, kind="batch", views=views, n_min=n_min, n_max=n_max, sides=sides,
                pick=pick, replay=replay)


def post(name, xres, yres, a_eq_e=True, gamma=1.0, colorbar=False, floats=False):
    return dict(name=name, kind="post", xres=xres, yres=yres, a_eq_e=a_eq_e, gamma=gamma,
                colorbar=colorbar, floats=floats)


def norm(name, n, ptypes, log=False, vector=False):
    return dict(name=name, kind="norm", n=n, ptypes=ptypes, log=log, vector=vector)


def listed():
    return [
        # interactive preview of a small selection: launches and host waits are all there is
        frame("thumb_additive_1k_64", 1000, 64, 64, "additive"),
        # a small depth-sorted frame of odd size
        frame("small_ordered_20k_257x193", 20_000, 257, 193, "ordered"),
        # the plain frame: 1M particles at 800^2
        frame("plain_1M_800", 1_000_000, 800, 800, "additive"),
        # a depth-sorted movie frame, HD size, vector colours (velocity maps)
        frame("ordered_1p3M_1279x719", 1_333_333, 1279, 719, "ordered", vector=True),
        # the headline frame: 8M gas depth-sorted + 8M stars additive at 2048^2
        frame("gas_stars_16M_2048", 16_000_000, 2048, 2048, "both", hsml=0.5),
        # a serving batch: 64 views, 56M particles in one call
        batch("batch_64_views", 64, 1e5, 4e6, "large", 1200),
        # thumbnails of an orbit, captured once and replayed for new particle values
        batch("replay_16_thumbs", 16, 2e3, 5e4, "small", 1300, replay=True),
        # differentiable rendering: forward + backward, both modes
        frame("grad_additive_2M_512", 2_000_000, 512, 512, "additive", grad=True),
        frame("grad_ordered_500k_512", 500_000, 512, 512, "ordered", grad=True),
        # the host renderer's call form: particle records and image in host memory
        frame("host_records_1M_800", 1_000_000, 800, 800, "additive", host=True),
        # the master's epilogue of a 2048^2 frame: tone map and TGA bytes
        post("post_tga_2048", 2048, 2048),
        # the scene maker's normalization before the render, 16M particles of two types
        norm("normalize_16M", 16_000_000, 2),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frame", "frame", "frame", "grad", "host", "batch", "post", "norm"])
    if kind == "frame":
        mode = rng.choice(["additive", "ordered", "both"])
        xres = logu(48, 1600)
        yres = max(33, int(round(xres * rng.uniform(0.5, 1.2))))
        c = frame("", logu(500, 4_000_000), xres, yres, mode,
                  hsml=rng.choice([0.1, 0.2, 0.3, 0.5]), vector=rng.random() < 0.3)
    elif kind == "grad":
        mode = rng.choice(["additive", "ordered"])
        side = logu(64, 640)
        c = frame("", logu(1000, 2_000_000 if mode == "additive" else 500_000), side,
                  max(33, int(round(side * rng.uniform(0.6, 1.0)))), mode,
                  vector=rng.random() < 0.3, grad=True)
    elif kind == "host":
        side = logu(64, 1024)
        c = frame("", logu(1000, 2_000_000), side, side,
                  rng.choice(["additive", "both"]), vector=rng.random() < 0.3, host=True)
    elif kind == "batch":
        if rng.random() < 0.5:
            c = batch("", rng.randint(2, 24), 5e4, 1e6, "large", rng.randrange(1 << 20))
        else:
            c = batch("", rng.randint(2, 48), 1e3, 5e4, "small", rng.randrange(1 << 20),
                      replay=rng.random() < 0.5)
    elif kind == "post":
        xres = logu(64, 4096)
        c = post("", xres, logu(64, 4096), a_eq_e=rng.random() < 0.7,
                 gamma=rng.choice([1.0, 1.0, 0.7]), colorbar=rng.random() < 0.3,
                 floats=rng.random() < 0.5)
    else:
        c = norm("", logu(1000, 16_000_000), rng.randint(1, 3), log=rng.random() < 0.5,
                 vector=rng.random() < 0.3)
    del c["name"]
    return c


# ------------------------------------------------------------------- the inputs

def gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1_000_003 + salt) & ((1 << 62) - 1))
    return g


def plummer(n, seed, salt, hsml, hsml_fixed=None, halo_frac=0.7, n_halos=50):
    """The synthetic field on the GPU: dict of float32 tensors."""
    rng = np.random.default_rng([seed & 0x7FFFFFFF, salt])
    centres = rng.uniform(0.0, BOX, (n_halos, 3))
    scale = np.exp(rng.uniform(math.log(0.2), math.log(2.0), n_halos))
    u = rng.uniform(0.0, 1.0, n_halos)
    mass = (1.0 + u * (1e3 ** -0.9 - 1.0)) ** (-1.0 / 0.9)
    n_halo = int(round(n * halo_frac))
    counts = np.floor(mass / mass.sum() * n_halo).astype(np.int64)
    counts[np.argsort(-mass, kind="stable")[:n_halo - int(counts.sum())]] += 1
    g = gen(seed, salt)
    f64 = dict(dtype=torch.float64, device=DEV)
    rand = lambda m: torch.rand(m, generator=g, **f64)  # noqa: E731
    hid = torch.repeat_interleave(torch.arange(n_halos, device=DEV),
                                  torch.from_numpy(counts).to(DEV))
    a = torch.from_numpy(scale).to(DEV)[hid]
    uu = rand(n_halo).clamp_(1e-12, 1.0 - 1e-12)
    rad = torch.minimum(a / torch.sqrt(uu ** (-2.0 / 3.0) - 1.0), 20.0 * a)
    cth, phi = rand(n_halo) * 2.0 - 1.0, rand(n_halo) * (2.0 * math.pi)
    sth = torch.sqrt(1.0 - cth * cth)
    c = torch.from_numpy(centres).to(DEV)[hid]
    halo = (c[:, 0] + rad * sth * torch.cos(phi), c[:, 1] + rad * sth * torch.sin(phi),
            c[:, 2] + rad * cth)
    d = {}
    for k, h in zip(("x", "y", "z"), halo):
        d[k] = torch.cat([h, rand(n - n_halo) * BOX]).float()
    nrm = lambda m: torch.randn(m, generator=g, **f64)  # noqa: E731
    d["hsml"] = (torch.full((n,), hsml_fixed, **f64) if hsml_fixed is not None
                 else torch.exp(math.log(hsml) + 0.6 * nrm(n))).float()
    d["inten"] = torch.exp(nrm(n)).float()
    d["col"] = rand(n).float()
    return d


def frame_fields(case, seed):
    """Particles, per-type modes and brightness of a frame case."""
    if case["mode"] == "both":
        n_gas = (case["n"] + 1) // 2
        gas = plummer(n_gas, seed, 1, case["hsml"])
        stars = plummer(case["n"] - n_gas, seed, 2, case["hsml"], hsml_fixed=0.05)
        d = {k: torch.cat([gas[k], stars[k]]) for k in gas}
        d["type"] = torch.ones(case["n"], dtype=torch.uint8, device=DEV)
        d["type"][:n_gas] = 0
        modes, bright = [False, True], [0.5, 2.0]
    else:
        d = plummer(case["n"], seed, 3, case["hsml"])
        modes, bright = [case["mode"] == "additive"], [1.0]
    if case["vector"]:
        g = gen(seed, 4)
        for k in ("c1", "c2"):
            d[k] = torch.rand(case["n"], generator=g, device=DEV)
    return d, modes, bright


def batch_views(case, seed):
    """(fields, camera, additive) of each view of a batch case."""
    sides = [256, 512, 768, 1024] if case["sides"] == "large" else [96, 128, 200, 256]
    for j in range(case["views"]):
        rng = np.random.default_rng([case["pick"], j])
        n = int(round(math.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"])))))
        side = int(rng.choice(sides))
        view = synth.orbit_view(rng.uniform(0.0, 2.0 * math.pi),
                                math.asin(rng.uniform(-0.98, 0.98)), 150.0, side)
        yield plummer(n, seed, 100 + j, 0.3), view, j % 2 == 0


def post_image(case, seed):
    """A raw frame: additive (-optical depth) or composited values in [0, 1]."""
    g = gen(seed, 5)
    v = torch.randn(case["xres"] * case["yres"] * 3, generator=g, device=DEV)
    return -torch.exp(v - 2.0) if case["a_eq_e"] else torch.sigmoid(v)


def norm_fields(case, seed):
    d = plummer(case["n"], seed, 6, 0.3)
    d = {k: d[k] for k in ("hsml", "inten", "col")}
    d["col"] = d["col"] * 50.0 + 1.0
    g = gen(seed, 7)
    if case["vector"]:
        for k in ("c1", "c2"):
            d[k] = torch.rand(case["n"], generator=g, device=DEV) * 50.0 + 1.0
    if case["ptypes"] > 1:
        d["type"] = torch.randint(0, case["ptypes"], (case["n"],), generator=g, device=DEV,
                                  dtype=torch.uint8)
    return d


def norm_text(case):
    t = "ptypes=%d\n" % case["ptypes"]
    for k in range(case["ptypes"]):
        if case["log"]:
            t += "intensity_log%d=T\ncolor_log%d=T\n" % (k, k)
        if case["vector"] and k == 0:
            t += "color_is_vector0=T\n"
    return t


# ------------------------------------------------------------------- the passes

_renderer = None


def new_renderer():
    r = S.Renderer(0)
    for t in range(2):
        r.set_palette(t, *synth.default_palette())
    return r


def renderer():
    """The one context that a program keeps for all its frames."""
    global _renderer
    if _renderer is None:
        _renderer = new_renderer()
    return _renderer


def prepare(case, seed):
    if case["kind"] == "frame":
        d, modes, bright = frame_fields(case, seed)
        view = synth.default_view(case["xres"], case["yres"])
        prm = S.params(ptypes=len(modes), a_eq_e=modes, brightness=bright,
                       col_vector=[True, False] if case["vector"] else None)
        st = dict(R=renderer(), cam=S.camera_setup(view), prm=prm, case=case)
        if case["host"]:
            a = np.zeros(case["n"], S.capi.PARTICLE_SIM)
            for k, f in (("x", "x"), ("y", "y"), ("z", "z"), ("r", "hsml"), ("I", "inten"),
                         ("er", "col"), ("eg", "c1"), ("eb", "c2"), ("type", "type")):
                if f in d:
                    a[k] = d[f].cpu().numpy()
            st["aos"] = a
            return st
        st["dev"] = d
        st["pic"] = torch.empty(case["xres"] * case["yres"] * 3, device=DEV)
        if case["grad"]:
            st["g"] = torch.randn(case["xres"] * case["yres"] * 3, generator=gen(seed, 8),
                                  device=DEV)
        return st
    if case["kind"] == "batch":
        views = [(d, S.camera_setup(v), S.params(a_eq_e=add),
                  torch.empty(v.xres * v.yres * 3, device=DEV))
                 for d, v, add in batch_views(case, seed)]
        st = dict(R=new_renderer() if case["replay"] else renderer(), views=views, case=case)
        if case["replay"]:
            st["R"].capture_reserve(views, 1.25)
            torch.cuda.synchronize()
            graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                with torch.cuda.graph(graph, stream=side):
                    st["R"].render_batched(views)
            torch.cuda.synchronize()
            st["graph"] = graph
        return st
    if case["kind"] == "post":
        n = case["xres"] * case["yres"] * 3
        return dict(R=renderer(), case=case, pic=post_image(case, seed),
                    q=S.post(a_eq_e=case["a_eq_e"], gamma=case["gamma"],
                             colorbar=case["colorbar"], ptypes=2),
                    out=torch.empty(n, device=DEV) if case["floats"] else None,
                    rgb8=torch.empty(n, dtype=torch.uint8, device=DEV))
    d = norm_fields(case, seed)
    st = dict(R=renderer(), case=case, q=S.norm_from_par(norm_text(case)), dev=d)
    if case["log"]:  # logs change the values for good: they are taken of a copy
        st["raw"] = {k: d[k].clone() for k in ("inten", "col", "c1", "c2") if k in d}
    return st


def run(st):
    case, R = st["case"], st["R"]
    if case["kind"] == "frame":
        if case["host"]:
            return {"pic": R.render_host(st["aos"], st["cam"], st["prm"])}
        R.render(st["dev"], st["cam"], st["prm"], st["pic"])
        out = {"pic": st["pic"]}
        if case["grad"]:
            out.update(R.backward(st["g"], case["n"], vector=case["vector"]))
        return out
    if case["kind"] == "batch":
        if case["replay"]:
            st["graph"].replay()
            return [v[3] for v in st["views"]]
        return R.render_batched(st["views"])
    if case["kind"] == "post":
        out, rgb8 = R.postprocess(st["pic"], case["xres"], case["yres"], st["q"], st["out"],
                                  st["rgb8"])
        return {"rgb8": rgb8, "image": out} if case["floats"] else {"rgb8": rgb8}
    for k, v in st.get("raw", {}).items():
        st["dev"][k].copy_(v)
    R.normalize(st["dev"], st["q"], ranges=False)
    return {k: st["dev"][k] for k in ("inten", "col", "c1", "c2") if k in st["dev"]}


# ------------------------------------------------------------------- the work

def disc_pixels(case_n, hsml, xres, yres, dist):
    """Expected footprint pixels of log-normal particles of a view (0.75 of the
    projected smoothing length, at least a pixel) that fall into the image."""
    scale = 0.5 * xres / (math.tan(math.radians(15.0)) * dist)
    r2 = (2.0 * scale) ** 2 * hsml * hsml * math.exp(2.0 * 0.6 ** 2) + 1.0
    return case_n * math.pi * 0.5625 * r2 * min(1.0, yres / xres)


def frame_fragments(case):
    n, x, y = case["n"], case["xres"], case["yres"]
    if case["mode"] == "both":
        g = (n + 1) // 2
        scale = 0.5 * x / (math.tan(math.radians(15.0)) * 200.0)
        stars = (n - g) * math.pi * 0.5625 * ((0.1 * scale) ** 2 + 1.0) * min(1.0, y / x)
        return disc_pixels(g, case["hsml"], x, y, 200.0), stars
    f = disc_pixels(n, case["hsml"], x, y, 200.0)
    return (f, 0.0) if case["mode"] == "ordered" else (0.0, f)


def work(case):
    """Bytes: every particle field and image value read or written once.
    Operations: per footprint pixel three channels of the update (additive 2,
    ordered 4 and the exponential's 3) and the Gaussian's product; the gradient
    twice that again."""
    if case["kind"] == "frame":
        n, px = case["n"], case["xres"] * case["yres"]
        per = 24 + (8 if case["vector"] else 0) + (1 if case["mode"] == "both" else 0)
        fo, fa = frame_fragments(case)
        flops = 100.0 * n + 22.0 * fo + 7.0 * fa
        if case["host"]:
            return {"bytes": 36 * n + 12 * px, "flops": flops}
        if case["grad"]:
            return {"bytes": 2 * per * n + 24 * px, "flops": 3.0 * flops}
        return {"bytes": per * n + 12 * px, "flops": flops}
    if case["kind"] == "batch":
        b = f = 0.0
        sides = [256, 512, 768, 1024] if case["sides"] == "large" else [96, 128, 200, 256]
        for j in range(case["views"]):
            rng = np.random.default_rng([case["pick"], j])
            n = int(round(math.exp(rng.uniform(math.log(case["n_min"]),
                                               math.log(case["n_max"])))))
            side = int(rng.choice(sides))
            b += 24 * n + 12 * side * side
            f += 100.0 * n + (7.0 if j % 2 == 0 else 22.0) * disc_pixels(n, 0.3, side, side, 150.0)
        return {"bytes": b, "flops": f}
    if case["kind"] == "post":
        v = 3 * case["xres"] * case["yres"]
        return {"bytes": (9 if case["floats"] else 5) * v, "flops": 6 * v}
    cols = 4 if case["vector"] else 2
    return {"bytes": case["n"] * (8 * cols + 4 + (1 if case["ptypes"] > 1 else 0)),
            "flops": case["n"] * 6 * cols}


# ------------------------------------------------------------------- in 64 bits

H2SIGMA = 0.5 * math.pi ** (-1.0 / 6.0)
BFAK = 0.5 * math.pi ** (-5.0 / 6.0)


def screen64(d, view, bright, vector):
    """Projection and colouring: centre x, y, radius and emission (n, 3) of
    every particle, and its depth; d: leaf tensors in double."""
    v = lambda t: torch.tensor(t, dtype=torch.float64, device=DEV)  # noqa: E731
    cam, look, sky = v(view.campos), v(view.lookat), v(view.sky)
    unit = lambda t: t / torch.linalg.norm(t)  # noqa: E731
    az = unit(cam - look)
    ax = unit(torch.linalg.cross(unit(sky), az))
    ay = torch.linalg.cross(az, ax)
    p = torch.stack([d["x"] - cam[0], d["y"] - cam[1], d["z"] - cam[2]], 1)
    vx, vy, vz = p @ ax, p @ ay, p @ az
    half = 0.5 * view.xres
    scale = -half / (math.tan(math.radians(0.5 * view.fov)) * vz)
    sx, sy = half + vx * scale, 0.5 * view.yres + vy * scale
    r2 = 2.0 * d["hsml"] * scale
    r = torch.sqrt(r2 * r2 + 1.0)
    inten = d["inten"] * (0.5 * BFAK) / d["hsml"] * r2 / r
    if vector:
        rgb = torch.stack([d["col"], d["c1"], d["c2"]], 1)
    else:
        px, prgb = synth.default_palette()
        px, prgb = v(px), v(prgb)
        c = d["col"].clamp(0.0, 1.0)
        i = (torch.searchsorted(px, c.detach()) - 1).clamp(0, len(px) - 2)
        w = ((c - px[i]) / (px[i + 1] - px[i]))[:, None]
        rgb = (1.0 - w) * prgb[i] + w * prgb[i + 1]
    return sx, sy, r, rgb * (inten * bright)[:, None], vz


def splat64(state, xres, yres, additive, grad=None, per=24_000_000):
    """The image of a screen-space state, and with grad (dL/dimage) the
    gradients of its (n, 6) state, in runs of fragments of whole image
    columns.  Additive: P -= e att.  Ordered, particles by ascending z, gray
    absorption 0.2: P = q + (P - q) exp(-e att), summed as every particle's
    own light behind the depth in front of it."""
    sx, sy, r, e, vz = (t.detach() for t in state)
    image = torch.zeros(xres * yres, 3, dtype=torch.float64, device=DEV)
    gs = torch.zeros(len(sx), 6, dtype=torch.float64, device=DEV) if grad is not None else None
    rad = 0.75 * r
    live = (vz < 0) & (sx + rad > 0) & (sx - rad < xres) & (sy + rad > 0) & (sy - rad < yres)
    order = torch.nonzero(live).squeeze(1)
    if not additive:
        order = order[torch.sort(vz[order].float(), stable=True)[1]]
    lo_x = torch.clamp(torch.ceil(sx - rad), 0, xres).long()
    hi_x = torch.clamp(torch.floor(sx + rad) + 1, 0, xres).long()
    lo_y = torch.clamp(torch.ceil(sy - rad), 0, yres).long()
    hi_y = torch.clamp(torch.floor(sy + rad) + 1, 0, yres).long()
    rows = torch.clamp(hi_y - lo_y, min=0)
    step = torch.zeros(xres + 1, dtype=torch.int64, device=DEV)
    step.index_add_(0, lo_x[order], rows[order])
    step.index_add_(0, hi_x[order], -rows[order])
    cost = torch.cumsum(step, 0)[:xres].cpu().tolist()
    xa = 0
    while xa < xres:
        xb, total = xa + 1, cost[xa]
        while xb < xres and total + cost[xb] <= per:
            total += cost[xb]
            xb += 1
        x0, x1 = torch.clamp(lo_x[order], min=xa), torch.clamp(hi_x[order], max=xb)
        cnt = torch.clamp(x1 - x0, min=0) * rows[order]
        keep = torch.nonzero(cnt > 0).squeeze(1)
        if len(keep):
            ids, cnt, x0 = order[keep], cnt[keep], x0[keep]
            w = torch.repeat_interleave(torch.arange(len(ids), device=DEV), cnt)
            k = torch.arange(len(w), device=DEV) - (torch.cumsum(cnt, 0) - cnt)[w]
            h = rows[ids][w]
            X, Y, w = x0[w] + k // h, lo_y[ids][w] + k % h, ids[w]
            ok = (X - sx[w]) ** 2 + (Y - sy[w]) ** 2 <= rad[w] ** 2
            X, Y, w = X[ok], Y[ok], w[ok]
            pix = X * yres + Y
            if not additive:
                pix, at = torch.sort(pix, stable=True)
                X, Y, w = X[at], Y[at], w[at]
                end = torch.searchsorted(pix, pix, right=True) - 1
            leaf = torch.cat([torch.stack([sx[w], sy[w], r[w]], 1), e[w]], 1)
            leaf.requires_grad_(grad is not None)
            dx, dy, sig = X - leaf[:, 0], Y - leaf[:, 1], H2SIGMA * leaf[:, 2]
            att = torch.exp(-(dx * dx + dy * dy) / (sig * sig))
            depth = leaf[:, 3:] * att[:, None]
            if additive:
                part = -depth
            else:
                cum = torch.cumsum(depth, 0)
                part = (leaf[:, 3:] / (leaf[:, 3:] + 0.2) * -torch.expm1(-depth) *
                        torch.exp(cum - cum[end]))
            image.index_add_(0, pix, part.detach())
            if grad is not None:
                (gl,) = torch.autograd.grad((part * grad.view(-1, 3).double()[pix]).sum(), leaf)
                gs.index_add_(0, w, gl)
        xa = xb
    return image, gs


def frame64(case_fields, view, modes, bright, vector, grad=None):
    """Image (and field gradients, for one type) of a frame, in double."""
    image, grads = 0.0, None
    for t, additive in enumerate(modes):
        sel = (case_fields["type"] == t) if "type" in case_fields else slice(None)
        d = {k: v[sel].double().requires_grad_(grad is not None)
             for k, v in case_fields.items() if k != "type"}
        vec = vector and t == 0
        state = screen64(d, view, bright[t], vec)
        img, gs = splat64(state, view.xres, view.yres, additive, grad)
        image = image + img
        if grad is not None:
            s = torch.cat([torch.stack(state[:3], 1), state[3]], 1)
            keys = ["x", "y", "z", "hsml", "inten", "col"] + (["c1", "c2"] if vec else [])
            grads = dict(zip(keys, torch.autograd.grad((s * gs).sum(), [d[k] for k in keys])))
    return image.reshape(-1), grads


def exact(case, seed):
    if case["kind"] == "frame":
        fo, fa = frame_fragments(case)
        if (fo * 4.0 + fa) * (3.0 if case["grad"] else 1.0) > 1.5e9:
            return None  # minutes in double
        d, modes, bright = frame_fields(case, seed)
        view = synth.default_view(case["xres"], case["yres"])
        g = (torch.randn(case["xres"] * case["yres"] * 3, generator=gen(seed, 8), device=DEV)
             if case["grad"] else None)
        image, grads = frame64(d, view, modes, bright, case["vector"], g)
        if case["host"]:
            return {"pic": image.view(case["xres"], case["yres"], 3).cpu().numpy()}
        return {"pic": image, **(grads or {})}
    if case["kind"] == "batch":
        if work(case)["flops"] > 2e9:
            return None
        return [frame64(d, v, [add], [1.0], False)[0] for d, v, add in batch_views(case, seed)]
    if case["kind"] == "post":
        if not case["floats"] or case["colorbar"]:
            return None  # bytes, and bars over the image's last rows
        v = post_image(case, seed).double()
        v = -torch.expm1(v) if case["a_eq_e"] else v
        return {"rgb8": None, "image": v ** case["gamma"] if case["gamma"] != 1.0 else v}
    d = norm_fields(case, seed)
    typ = d.get("type", torch.zeros(case["n"], dtype=torch.uint8, device=DEV))
    out = {k: d[k].double() for k in ("inten", "col", "c1", "c2") if k in d}
    if case["log"]:
        out["inten"], out["col"] = torch.log10(out["inten"]), torch.log10(out["col"])
    for t in range(case["ptypes"]):
        sel = typ == t
        vec = case["vector"] and t == 0
        if vec and case["log"]:
            for k in ("c1", "c2"):
                out[k][sel] = torch.log10(out[k][sel])
        for keys in (("inten",), ("col", "c1", "c2") if vec else ("col",)):
            v = [out[k][sel] for k in keys]
            if v[0].numel():
                lo, hi = min(x.min() for x in v), max(x.max() for x in v)
                for k, x in zip(keys, v):
                    out[k][sel] = (x - lo) / (hi - lo) if hi > lo else torch.ones_like(x)
    return out
