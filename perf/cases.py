"""Workloads of the imaging-and-trigger path, each through a public entry point.

A case is a dict of plain values: ``form`` names the entry point, ``image``,
``tile`` and ``nbl`` (visibilities per snapshot) the shape, ``fill`` the longest
projected baseline as a fraction of the sampling rate 1/cell (0.5 is Nyquist).
The inputs are synthetic observations: a log-radial array on the ground under
earth rotation, a power-law point-source sky with one transient, Gaussian
noise, and each snapshot's uv plane from the principal axes of its baselines.

The arrays and image sizes are those of the repository's benchmark and tests:
64 antennas at 256^2, 128 at 1024^2, 256 at 2048^2, 512 at 4096^2, 1024 at
8192^2, 140 MHz.
"""
import math

import numpy as np
import torch

import fastimagingpipe_amd as F

FREQ_HZ = 140e6
C_LIGHT = 299792458.0
BETA, SUPPORT = 15.3704324328, 8      # the gridding kernel's shape
LATITUDE = math.radians(-26.7)
CHAN_HZ = 1e6                         # channel spacing of the raw form
VIS = {"f32": F.VIS_F32, "bf16": F.VIS_BF16, "f16": F.VIS_F16}
TORCH_VIS = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    def case(name, form, image, nbl, tile=32, fill=0.27, **more):
        return {"name": name, "form": form, "image": image, "nbl": nbl, "tile": tile, "fill": fill, **more}

    return [
        # One trigger decision of a small station, inputs already on the GPU:
        # the call is launches and latency.
        case("device_256_2016bl", "device", 256, 2016, tile=16),
        # The same for growing arrays; the cell shrinks with the longest
        # baseline, so each fills the same part of its grid.
        case("device_1024_8128bl", "device", 1024, 8128),
        case("device_2048_32640bl", "device", 2048, 32640),
        # The benchmark's headline: 512 antennas at 4096^2.
        case("device_4096_130816bl", "device", 4096, 130816),
        # The largest supported image with its 1024-antenna array.
        case("device_8192_523776bl", "device", 8192, 523776),
        # A partly flagged array with long baselines (uv coverage almost to the
        # edge of the grid) and a tile size that does not divide the image.
        case("device_2048_77777bl_t24", "device", 2048, 77777, tile=24, fill=0.46),
        # The drop-in for the reference's call: host arrays in, tLISI out.
        case("host_4096_130816bl", "host", 4096, 130816, vis="f32"),
        # The same with visibilities stored in 16 bits, at a quarter of it.
        case("host_1024_8128bl_f16", "host", 1024, 8128, vis="f16"),
        # The images themselves (source finding, archiving), read back.
        case("image_1024_8128bl", "image", 1024, 8128),
        # A recorded scan: unevenly flagged snapshots resident on the GPU, one
        # trigger per sliding window.
        case("batch_2048_16x32640bl_bf16", "batch", 2048, 32640, snapshots=16, vis="bf16"),
        # Raw correlator output to trigger on the GPU: collapse of two
        # polarisations, projection, imaging; 4 channels of 128 antennas.
        case("raw_1024_4x8128bl", "raw", 1024, 8128, channels=4),
        # A busy live stream: snapshots submitted faster than they are imaged.
        case("serve_2048_12x32640bl", "serve", 2048, 32640, snapshots=12, vis="f32"),
    ]


def draw(rng):
    """One more case: image sizes over the supported range, visibility counts
    from a sparse to a crowded array of that size, odd counts among them."""
    form = rng.choice(["device"] * 4 + ["host", "image", "batch", "raw", "serve"])
    top = {"device": 4096, "host": 4096, "image": 1024, "batch": 2048, "raw": 2048, "serve": 2048}[form]
    image = rng.choice([s for s in (128, 256, 512, 1024, 2048, 4096) if s <= top])
    typical = image * image / 128.0
    nbl = int(math.exp(rng.uniform(math.log(max(300.0, typical / 8)), math.log(max(4000.0, typical * 3)))))
    case = {"form": form, "image": image, "nbl": min(nbl, 400000), "tile": rng.choice([16, 24, 32, 32, 32, 50, 64]),
            "fill": round(rng.uniform(0.15, 0.48), 3)}
    if form == "host":
        case["vis"] = rng.choice(["f32", "f16", "bf16"])
    if form == "batch":
        case["snapshots"] = rng.randint(4, 16)
        case["vis"] = rng.choice(["f32", "bf16"])
    if form == "raw":
        case["channels"] = rng.randint(1, 4)
        case["nbl"] = max(300, case["nbl"] // case["channels"])
    if form == "serve":
        case["snapshots"] = rng.randint(4, 14)
        case["vis"] = rng.choice(["f32", "bf16"])
    return case


# ------------------------------------------------------------------ inputs


def cell_of(case):
    """Pixel size (rad): sizes scale so that the field stays that of 4096 px of 7.27e-6 rad."""
    return float(np.float32(7.2722e-6 * 4096.0 / case["image"]))


def snapshots_of(case):
    return case.get("snapshots", 3)


def principal_axes(d):
    """Rows V0, V1 (principal axes of the baselines, largest entry positive) and V0 x V1."""
    mean = d.mean(0)
    cov = ((d - mean).T @ (d - mean) / (d.shape[0] - 1)).cpu().numpy()
    val, vec = np.linalg.eigh(cov)
    V = vec[:, np.argsort(val)[::-1][:2]].T.copy()
    for r in V:
        if r[np.argmax(np.abs(r))] < 0:
            r *= -1.0
    return np.vstack([V, np.cross(V[0], V[1])])


def observe(case, seed):
    """The observation on the GPU: uvw [S][n][3] metres, noiseless sky as a
    function of (snapshot, frequency), and a generator for what is random."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def uniform(*shape):
        return torch.rand(*shape, generator=gen, device=dev, dtype=torch.float64)

    image, n, cell, S = case["image"], case["nbl"], cell_of(case), snapshots_of(case)
    radius = 0.5 * case["fill"] * C_LIGHT / (FREQ_HZ * cell)
    nant = 2
    while nant * (nant - 1) // 2 < n:
        nant += 1
    r, az = radius * 10.0 ** (-2.0 * (1.0 - uniform(nant))), 2 * math.pi * uniform(nant)
    east, north = r * torch.cos(az), r * torch.sin(az)
    i, j = torch.triu_indices(nant, nant, 1, device=dev)
    if i.numel() > n:   # flagged baselines are dropped
        keep = torch.sort(torch.randperm(i.numel(), generator=gen, device=dev)[:n]).values
        i, j = i[keep], j[keep]
    de, dn = east[j] - east[i], north[j] - north[i]
    x, y, z = -math.sin(LATITUDE) * dn, de, math.cos(LATITUDE) * dn
    sky = uniform(4)
    dec, ha0 = math.radians(-40.0 + 25.0 * float(sky[0])), 0.6 * (float(sky[1]) - 0.5)
    sd, cd = math.sin(dec), math.cos(dec)
    uvw = torch.empty(S, n, 3, device=dev, dtype=torch.float64)
    for s in range(S):
        H = ha0 + 2 * math.pi * s / 86164.0905
        sh, ch = math.sin(H), math.cos(H)
        uvw[s, :, 0] = sh * x + ch * y
        uvw[s, :, 1] = -sd * ch * x + sd * sh * y + cd * z
        uvw[s, :, 2] = cd * ch * x - cd * sh * y + sd * z
    nsrc, fov = 50, 0.4 * image * cell
    l, m = fov * (2 * uniform(nsrc + 1) - 1), fov * (2 * uniform(nsrc + 1) - 1)
    flux = (0.01 ** -0.8 + uniform(nsrc + 1) * (1.0 - 0.01 ** -0.8)) ** (-1.0 / 0.8)
    flux[nsrc] = 0.5   # the transient
    n1 = torch.sqrt(1.0 - l * l - m * m) - 1.0

    def sky_of(s, freq):
        k = nsrc + 1 if s == min(2, S - 1) else nsrc
        d = uvw[s] * (freq / C_LIGHT)
        out = torch.zeros(n, device=dev, dtype=torch.complex128)
        for q in range(k):
            ph = -2 * math.pi * (d[:, 0] * l[q] + d[:, 1] * m[q] + d[:, 2] * n1[q])
            out += flux[q] * torch.polar(torch.ones_like(ph), ph)
        return out

    def noise(count):
        return 0.1 * torch.view_as_complex(torch.randn(count, 2, generator=gen, device=dev, dtype=torch.float64))

    return uvw, sky_of, noise, uniform


def projected(case, seed):
    """vis_re, vis_im [S][n], bin [S][n][2], vin [S][3][3] on the GPU (float),
    and each snapshot's count of valid rows (the batch form's are uneven)."""
    uvw, sky_of, noise, uniform = observe(case, seed)
    S, n = uvw.shape[:2]
    dev = uvw.device
    vr, vi = torch.zeros(S, n, device=dev), torch.zeros(S, n, device=dev)
    b, v = torch.zeros(S, n, 2, device=dev), torch.zeros(S, 3, 3, device=dev)
    nvis = np.full(S, n, np.int32)
    for s in range(S):
        d = uvw[s] * (FREQ_HZ / C_LIGHT)
        V = principal_axes(d)
        vis = sky_of(s, FREQ_HZ) + noise(n)
        bs = d @ torch.from_numpy(V[:2].T.copy()).to(dev)
        if case["form"] == "batch":   # up to 30% of a snapshot's rows are flagged away
            keep = uniform(n) >= 0.3 * float(uniform(1))
            vis, bs = vis[keep], bs[keep]
            nvis[s] = vis.numel()
        k = int(nvis[s])
        vr[s, :k], vi[s, :k], b[s, :k] = vis.real.float(), vis.imag.float(), bs.float()
        v[s] = torch.from_numpy(V).float().to(dev)
    t = TORCH_VIS[case.get("vis", "f32")]
    return vr.to(t), vi.to(t), b, v, nvis


def raw_inputs(case, seed):
    """Raw columns on the GPU: uvw, freqs, two polarisations, flags, weights."""
    uvw, sky_of, noise, uniform = observe(case, seed)
    S, n = uvw.shape[:2]
    nchan = case["channels"]
    freqs = FREQ_HZ - CHAN_HZ * torch.arange(nchan, device=uvw.device, dtype=torch.float64)
    ns = n * nchan
    out = {"uvw": uvw.contiguous(), "freqs": freqs}
    xx = torch.empty(S, ns, device=uvw.device, dtype=torch.complex64)
    yy = torch.empty_like(xx)
    for s in range(S):
        sky = torch.cat([sky_of(s, float(f)) for f in freqs])
        xx[s], yy[s] = sky + noise(ns), sky + noise(ns)
    for name, v in (("xx", xx), ("yy", yy)):
        out[name + "_re"], out[name + "_im"] = v.real.contiguous(), v.imag.contiguous()
    for k in ("0", "3"):
        out["flag" + k] = (uniform(S, ns) < 0.1).to(torch.uint8)
        out["w" + k] = (0.5 + 1.5 * uniform(S, ns)).float()
    return out


def host(t):
    """A host array of a GPU tensor; 16-bit floats as their bit patterns."""
    t = t.contiguous().cpu()
    return t.numpy() if t.dtype == torch.float32 else t.view(torch.int16).numpy().view(np.uint16)


def prepare(case, seed):
    form, un = case["form"], case["image"] // case["tile"]
    state = {"case": case, "cell": cell_of(case), "vis": VIS[case.get("vis", "f32")]}
    if form == "raw":
        state["in"] = raw_inputs(case, seed)
        ns = case["nbl"] * case["channels"]
        state["out"] = torch.zeros(un, un, device="cuda")
        state["bin"], state["vin"] = torch.zeros(3, ns, 2, device="cuda"), torch.zeros(3, 3, 3, device="cuda")
        return state
    vr, vi, b, v, nvis = projected(case, seed)
    if form in ("device", "batch"):
        state["in"], state["nvis"] = (vr, vi, b, v), nvis
        state["out"] = torch.zeros(*((vr.shape[0] - 2,) if form == "batch" else ()), un, un, device="cuda")
    else:
        state["in"] = (host(vr), host(vi), host(b), host(v))
    if form == "serve":
        stream = {"num_baselines": case["nbl"], "image_size": case["image"], "cell_size": state["cell"],
                  "unit_size": case["tile"], "vis_type": state["vis"]}
        state["server"] = F.Server([stream], ring=16, hbm_budget_bytes=16 << 30)
    return state


def run(state):
    case, cell = state["case"], state["cell"]
    form, image, tile, n = case["form"], case["image"], case["tile"], case["nbl"]
    if form == "device":
        vr, vi, b, v = state["in"]
        F.pipe_device(vr.data_ptr(), vi.data_ptr(), b.data_ptr(), v.data_ptr(), state["out"].data_ptr(), n, image, 3,
                      cell, tile)
        return state["out"]
    if form == "batch":
        vr, vi, b, v = state["in"]
        F.batch_device(vr.data_ptr(), vi.data_ptr(), state["vis"], b.data_ptr(), v.data_ptr(), state["nvis"], n,
                       vr.shape[0], n, image, cell, tile, state["out"].data_ptr())
        return state["out"]
    if form == "raw":
        F.pipe_raw_device({k: t.data_ptr() for k, t in state["in"].items()}, n, case["channels"], 3, image, cell, tile,
                          state["out"].data_ptr(), state["bin"].data_ptr(), state["vin"].data_ptr())
        return {"tlisi": state["out"], "bin": state["bin"], "vin": state["vin"]}
    vr, vi, b, v = state["in"]
    if form == "host":
        if case["vis"] == "f32":
            return F.fipipe(vr, vi, b, v, n, image, 3, cell, tile)
        return F.fipipe_lowp(vr, vi, state["vis"], b, v, n, image, 3, cell, tile)
    if form == "image":
        pre, img, top = F.image(vr, vi, b, v, n, image, 3, cell)
        return {"pre": pre, "img": img, "max": top}
    for k in range(vr.shape[0]):
        if not state["server"].submit(0, vr[k], vi[k], b[k], v[k]):
            raise RuntimeError("a snapshot was refused")
    state["server"].drain()
    return state["server"].latest(0)[0]


def work(case):
    """Inputs read once, outputs written once; the taps of the gridding kernel,
    the two FFT axes over the covered columns, the re-projection of each pixel
    and the trigger's terms."""
    image, S, n = case["image"], snapshots_of(case), case["nbl"] * case.get("channels", 1)
    g, un2 = 1.5 * image, (image // case["tile"]) ** 2
    vis = {"f32": 4, "bf16": 2, "f16": 2}[case.get("vis", "f32")]
    bytes_in = S * (n * (2 * vis + 8) + 36)
    bytes_out = 4 * un2
    if case["form"] == "raw":
        bytes_in = S * (case["nbl"] * 24 + n * (4 * 4 + 2 + 8))
        bytes_out += S * (n * 8 + 36)
    if case["form"] == "batch":
        bytes_out = 4 * un2 * (S - 2)
    if case["form"] == "image":
        bytes_out = S * (2 * 4 * image * image + 4)
    columns = min(case["fill"] * g + 5, g / 2 + 1)
    flops = S * (n * (64 * 4 + 16 * 8) + columns * 5 * g * math.log2(g) + image * 2.5 * g * math.log2(g)
                 + 25.0 * image * image)
    windows = {"image": 0, "batch": S - 2, "serve": S - 2}.get(case["form"], 1)
    return {"bytes": float(bytes_in + bytes_out), "flops": float(flops + windows * 9.0 * image * image)}


# ------------------------------------------------------- the same in 64 bits


def kernel64(x):
    return torch.where(x.abs() <= 1, torch.exp(BETA * (torch.sqrt((1 - x * x).clamp(min=0)) - 1)), torch.zeros_like(x))


def correction64(image, g):
    """1 / (c(t) norm), t = 0..image/2: the gridding kernel's transform by 28-point quadrature."""
    x, w = np.polynomial.legendre.leggauss(28)
    t = np.arange(image // 2 + 1)[:, None] / g
    c = 0.5 * (np.exp(BETA * (np.sqrt(1 - x * x) - 1)) * w * np.cos(math.pi * t * SUPPORT * x)).sum(1)
    th, wt = np.polynomial.legendre.leggauss(200)   # norm = 4 int ES, with x = sin(theta)
    th, wt = th * math.pi / 2, wt * math.pi / 2
    norm = 4.0 * float((np.exp(BETA * (np.cos(th) - 1)) * np.cos(th) * wt).sum())
    return torch.from_numpy(1.0 / (c * SUPPORT / norm * norm)).cuda()


def taps64(p, g):
    """The nine candidate cells along one axis and their weights."""
    t = torch.ceil(p - 4)[:, None] + torch.arange(9, device=p.device)
    w = kernel64((t - p[:, None]) / 4)
    w = torch.where((t <= torch.floor(p + 4)[:, None]) & (t >= -(g // 2)) & (t <= g // 2 - 1), w, torch.zeros_like(w))
    return torch.remainder(t, g).long(), w


def image64(vr, vi, b, v, image, cell, norm_n):
    """One snapshot: the corrected image before and after re-projection."""
    g, h = int(math.ceil(1.5 * image)), image // 2
    dev = torch.device("cuda")
    V = v.double().cpu().numpy().reshape(3, 3)
    J = abs(V[0, 0] * V[1, 1] - V[0, 1] * V[1, 0])
    grid = torch.zeros(g * g, 2, device=dev, dtype=torch.float64)
    for k in range(0, vr.numel(), 65536):
        s = slice(k, k + 65536)
        i1, w1 = taps64(b[s, 0].double() * (cell * g), g)
        i2, w2 = taps64(b[s, 1].double() * (cell * g), g)
        val = torch.stack([vr[s].double(), vi[s].double()], -1) / J
        at = (i1[:, :, None] * g + i2[:, None, :]).reshape(-1)
        w = (w1[:, :, None] * w2[:, None, :])[..., None]
        grid.index_add_(0, at, (w * val[:, None, None, :]).reshape(-1, 2))
    d = torch.fft.ifft2(torch.view_as_complex(grid.reshape(g, g, 2)), norm="forward").real
    del grid
    x = torch.arange(image, device=dev) - h
    c = correction64(image, g)[x.abs()]
    at = torch.remainder(x, g)
    pre = d[at][:, at].abs() * c[:, None] * c[None, :]
    del d
    xi, eta, a22 = V[2, 0] / V[2, 2], V[2, 1] / V[2, 2], abs(V[2, 2])
    img = torch.zeros(image * image, device=dev, dtype=torch.float64)
    rows = max(1, (1 << 24) // image)
    col = x.double()[None, :]
    for k in range(0, image, rows):
        row = x[k:k + rows].double()[:, None]
        q1 = (-V[0, 0] * col + V[1, 0] * row) / a22
        q2 = (-V[0, 1] * col + V[1, 1] * row) / a22
        r2 = (cell * (q1 - 1)) ** 2 + (cell * (q2 - 1)) ** 2
        np_ = torch.where(r2 <= 1, r2 / (1 + torch.sqrt((1 - r2).clamp(min=0))), torch.zeros_like(r2))
        o1, o2 = q1 - xi * np_ / cell, q2 + eta * np_ / cell
        ok = (o1.abs() < h - 1) & (o2.abs() < h - 1)
        val = (pre[k:k + rows] / norm_n)[ok]
        o1, o2 = o1[ok], o2[ok]
        f1, f2 = torch.floor(o1), torch.floor(o2)
        a, e = o1 - f1, o2 - f2
        at = ((f2 + h) * image + f1 + h).long()
        # an integer position puts its second weight, zero, on the next pixel
        for off, w in ((0, (1 - a) * (1 - e)), (image, (1 - a) * e), (1, a * (1 - e)), (image + 1, a * e)):
            img.index_add_(0, at + off, w * val)
    return pre, img.reshape(image, image)


def trigger64(d1, d2, d3, tile):
    un = d1.shape[0] // tile
    top = max(0.0, float(d1.max()), float(d2.max()), float(d3.max()))
    dd = ((d1 - d2).abs() - (d2 - d3).abs()).abs()
    s2 = torch.where(d2 <= 0, torch.full_like(d2, float(np.float32(1e-6))), d2)
    ratio = (dd / s2).clamp(max=1.0)

    def tiles(t):
        return t[:un * tile, :un * tile].reshape(un, tile, un, tile).transpose(1, 2).reshape(un, un, -1)

    return 1.0 - tiles(dd).mean(-1) * tiles(dd).amax(-1) * tiles(ratio).mean(-1) / top / top


def raw64(case, seed):
    """Collapsed visibilities, and the projection in its interchange type (float)."""
    r = raw_inputs(case, seed)
    S = r["uvw"].shape[0]
    a = torch.where(r["flag0"] > 0, torch.zeros_like(r["w0"]), r["w0"]).double()
    b = torch.where(r["flag3"] > 0, torch.zeros_like(r["w3"]), r["w3"]).double()
    den = torch.where(a + b > 0, a + b, torch.ones_like(a))
    vr = (r["xx_re"].double() * a + r["yy_re"].double() * b) / den
    vi = (r["xx_im"].double() * a + r["yy_im"].double() * b) / den
    bins, vins = [], []
    for s in range(S):
        d = torch.cat([r["uvw"][s] * (float(f) / C_LIGHT) for f in r["freqs"]])
        V = torch.from_numpy(principal_axes(d)).to(d.device)
        bins.append(d @ V[:2].T)
        vins.append(V)
    return vr, vi, torch.stack(bins), torch.stack(vins)


def exact(case, seed):
    form, cell = case["form"], cell_of(case)
    more = {}
    if form == "raw":
        vr, vi, b, v = raw64(case, seed)
        more = {"bin": b, "vin": v}
        b, v = b.float(), v.float()
        nvis = np.full(vr.shape[0], vr.shape[1])
    else:
        vr, vi, b, v, nvis = projected(case, seed)
    S, norm_n = vr.shape[0], vr.shape[1]
    first = S - 3 if form == "serve" else 0   # a server keeps its latest window
    pres, imgs, tlisi = [], [], []
    for s in range(first, S):
        k = int(nvis[s])
        pre, img = image64(vr[s, :k], vi[s, :k], b[s, :k], v[s], case["image"], cell, norm_n)
        if form == "image":
            pres.append(pre)
        imgs.append(img)
        if form != "image" and len(imgs) > 2:
            tlisi.append(trigger64(*imgs[-3:], case["tile"]))
            imgs = imgs[-2:]
    if form == "image":
        imgs = torch.stack(imgs)
        return {"pre": torch.stack(pres), "img": imgs, "max": imgs.amax((1, 2))}
    out = torch.stack(tlisi) if form == "batch" else tlisi[-1]
    return {"tlisi": out, **more} if form == "raw" else out
