"""Performance cases of the framework: the calls that users of the Monte Carlo,
of its stages and of the surrogate make, over the sizes they make them at.

A case is a dict of plain values; its "kind" names the call:
  mc       Context.run_realizations: a border-count map from scratch;
  stages   the stage methods one by one on the caller's own rasters;
  field    random_field + convolve: the correlated error field alone;
  batch    Batch.run in graph mode: many uneven DEMs at once;
  predict  Surrogate.predict: the border-probability map of one DEM;
  train    Trainer.gradients: loss and parameter gradients of one batch.
Cells are 10 m and the DEMs come from the package's generator, as in the
benchmark and the tests.
"""
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

import cageo_amd as ca
from cageo_amd import surrogate as sg

CELL = 10.0
NODATA = -9999.0
BEVEL = 2


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # one realization of a very small DEM: launches and waits decide
        dict(name="mc_128x96", kind="mc", w=128, h=96, model="gauss", pr=60.0, rmse=1.8, n=1),
        # an ordinary DEM, ragged at every block edge, a few realizations a call
        dict(name="mc_1000x777", kind="mc", w=1000, h=777, model="gauss", pr=60.0, rmse=1.8, n=4),
        # the headline workload
        dict(name="mc_4096", kind="mc", w=4096, h=4096, model="gauss", pr=60.0, rmse=1.8, n=2),
        # a large DEM, one realization at a time (a program that shows progress)
        dict(name="mc_8192", kind="mc", w=8192, h=8192, model="gauss", pr=60.0, rmse=2.5, n=1),
        # the exponential filter in the reference's order
        dict(name="mc_exp_2048", kind="mc", w=2048, h=2048, model="exp", pr=200.0, rmse=1.8, n=1),
        # a program that drives the stages itself and keeps every raster
        dict(name="stages_1536x1100", kind="stages", w=1536, h=1100, model="gauss", pr=100.0,
             rmse=1.8),
        # error fields with the fast convolution: a power-of-two grid, and one that is not
        dict(name="field_fast_4096", kind="field", w=4096, h=4096, model="exp_fast", pr=200.0,
             rmse=2.5),
        dict(name="field_fast_3000x2301", kind="field", w=3000, h=2301, model="exp_fast", pr=200.0,
             rmse=2.5),
        # many uneven DEMs, each with its own error model
        dict(name="batch_12", kind="batch", tiles=12, lo=256, hi=1024, n=2),
        # the surrogate on an odd-sized DEM and at the headline size
        dict(name="predict_1001x700", kind="predict", w=1001, h=700, rmse=1.8, pr=60.0),
        dict(name="predict_4096", kind="predict", w=4096, h=4096, rmse=1.8, pr=60.0),
        # one training batch as the packaged network was trained
        dict(name="train_8x512", kind="train", batch=8, size=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mc", "mc", "mc", "mc_exp", "stages", "field", "field", "batch", "predict",
                       "predict", "train"])
    rmse, pr = round(rng.uniform(0.5, 3.0), 2), round(rng.uniform(30.0, 200.0), 1)
    if kind == "mc":
        w, h = _log(rng, 64, 4096), _log(rng, 64, 4096)
        most = max(1, min(4, (1 << 24) // (w * h)))
        return dict(kind="mc", w=w, h=h, model="gauss", pr=pr, rmse=rmse, n=rng.randint(1, most))
    if kind == "mc_exp":
        return dict(kind="mc", w=_log(rng, 128, 2048), h=_log(rng, 128, 2048), model="exp", pr=pr,
                    rmse=rmse, n=1)
    if kind == "stages":
        return dict(kind="stages", w=_log(rng, 64, 2500), h=_log(rng, 64, 2500), model="gauss",
                    pr=pr, rmse=rmse)
    if kind == "field":
        model = rng.choice(["gauss", "exp_fast", "exp_fast"])
        if rng.random() < 0.4:
            w, h = 1 << rng.randint(7, 12), 1 << rng.randint(7, 12)
        else:
            w, h = _log(rng, 128, 3000), _log(rng, 128, 3000)
        return dict(kind="field", w=w, h=h, model=model, pr=pr, rmse=rmse)
    if kind == "batch":
        lo = _log(rng, 100, 400)
        return dict(kind="batch", tiles=rng.randint(2, 16), lo=lo, hi=lo * rng.randint(2, 3),
                    n=rng.randint(1, 2))
    if kind == "predict":
        return dict(kind="predict", w=_log(rng, 64, 3000), h=_log(rng, 64, 3000), rmse=rmse, pr=pr)
    return dict(kind="train", batch=rng.randint(1, 8), size=8 * rng.randint(8, 64))


# ---- what a program has in hand ------------------------------------------------

def _dem(w, h, seed):
    """DEM and stream rasters on the device; streams start at 2000 cells of
    upstream area, fewer on DEMs too small to have any."""
    threshold = 2000 if w * h >= 1 << 18 else 200
    dem, stream = ca.synth_dem(w, h, seed, CELL, threshold, NODATA)
    return torch.from_numpy(dem).cuda(), torch.from_numpy(stream).cuda()


def _context(case, seed):
    ctx = ca.Context(case["w"], case["h"], torch.cuda.current_stream())
    model = ca.GAUSSIAN if case["model"] == "gauss" else ca.EXPONENTIAL
    r = ca.filter_radius(case["pr"], CELL)
    ctx.set_filter(model, r, ca.create_filter(model, case["pr"], CELL, r))
    if case["model"] == "exp_fast":
        ctx.set_conv_mode(ca.CONV_FAST)
    return ctx


def _f32(h, w):
    return torch.zeros((h, w), dtype=torch.float32, device="cuda")


def _train_shape(case):
    """The tiles are cut from one DEM, two rows of them where they are even."""
    rows = 2 if case["batch"] % 2 == 0 else 1
    return rows, case["batch"] // rows


def _train_inputs(case, seed):
    """Inputs [batch][s][s][4] and Monte Carlo frequencies [batch][s][s]."""
    rows, cols = _train_shape(case)
    s = case["size"]
    h, w = rows * s, cols * s
    rmse, pr = 1.8, 60.0
    dem, stream = _dem(w, h, seed)
    count = _f32(h, w)
    with _context(dict(w=w, h=h, model="gauss", pr=pr), seed) as ctx:
        ctx.mc_setup(dem, stream, NODATA, NODATA, BEVEL, 0.0, rmse)
        ctx.run_realizations(count, 20, seed)
    planes = torch.empty((h, w, 4), dtype=torch.float32, device="cuda")
    planes[..., 0] = (dem - dem.mean()) / dem.std()
    planes[..., 1] = (stream != NODATA).float()
    planes[..., 2] = rmse / 3.0
    planes[..., 3] = pr / 200.0
    x = planes.view(rows, s, cols, s, 4).permute(0, 2, 1, 3, 4).reshape(-1, s, s, 4).contiguous()
    y = (count / 20.0).view(rows, s, cols, s).permute(0, 2, 1, 3).reshape(-1, s, s).contiguous()
    return x, y


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind in ("mc", "stages"):
        dem, stream = _dem(case["w"], case["h"], seed)
        ctx = _context(case, seed)
        s = dict(kind=kind, ctx=ctx, seed=seed, case=case, dem=dem, stream=stream,
                 mc=_f32(case["h"], case["w"]))
        if kind == "mc":
            ctx.mc_setup(dem, stream, NODATA, NODATA, BEVEL, 0.0, case["rmse"])
        else:
            s["z"], s["filled"] = _f32(case["h"], case["w"]), _f32(case["h"], case["w"])
            s["dir"] = torch.zeros((case["h"], case["w"], 2), dtype=torch.int8, device="cuda")
            s["labels"] = torch.zeros((case["h"], case["w"]), dtype=torch.int32, device="cuda")
        return s
    if kind == "field":
        return dict(kind=kind, ctx=_context(case, seed), seed=seed, case=case,
                    field=_f32(case["h"], case["w"]))
    if kind == "batch":
        sides = np.random.default_rng([case["tiles"], case["lo"], case["hi"]])
        shapes = [tuple(int(v) for v in sides.integers(case["lo"], case["hi"] + 1, size=2))
                  for _ in range(case["tiles"])]
        rmse = rng.uniform(0.5, 3.0, len(shapes))
        pr = rng.uniform(30.0, 200.0, len(shapes))
        batch = ca.Batch(shapes)
        for t, (h, w) in enumerate(shapes):
            dem, stream = _dem(w, h, seed + 100 + t)
            batch.setup_tile(t, dem, stream, NODATA, NODATA, BEVEL, ca.GAUSSIAN, float(pr[t]), CELL,
                             0.0, float(rmse[t]), seed + 1000 + t)
        return dict(kind=kind, batch=batch, case=case, mcs=[_f32(h, w) for h, w in shapes])
    if kind == "predict":
        dem, stream = _dem(case["w"], case["h"], seed)
        return dict(kind=kind, net=ca.Surrogate(sg.DEFAULT_WEIGHTS, torch.cuda.current_stream()),
                    case=case, dem=dem, stream=stream, prob=_f32(case["h"], case["w"]))
    x, y = _train_inputs(case, seed)
    folder = tempfile.mkdtemp()
    try:
        path = os.path.join(folder, "init.bin")
        params = _initial_weights(seed)
        sg.save_params(params, path)
        trainer = ca.Trainer(32, init_weights=path, stream=torch.cuda.current_stream())
    finally:
        shutil.rmtree(folder)
    return dict(kind=kind, trainer=trainer, x=x, y=y,
                shapes={k: v.shape for k, v in params.items()})


def run(s):
    kind = s["kind"]
    if kind == "mc":
        s["mc"].zero_()
        s["ctx"].run_realizations(s["mc"], s["case"]["n"], s["seed"])
        return s["mc"]
    if kind == "stages":
        c, ctx = s["case"], s["ctx"]
        s["mc"].zero_()
        ctx.random_field(s["z"], s["seed"], 0, 0, 0.0, c["rmse"])
        ctx.convolve(s["z"])
        ctx.realistic_dem(s["dem"], s["z"], NODATA)
        ctx.stream_burn(s["z"], s["stream"], BEVEL, NODATA, NODATA)
        ctx.pit_fill(s["filled"], s["z"], NODATA)
        ctx.flow_routing(s["dir"], s["filled"], NODATA)
        long_paths = ctx.flow_tracing(s["labels"], s["dir"], s["stream"])
        ctx.catchment_border(s["mc"], s["labels"])
        return dict(z=s["z"], filled=s["filled"], dir=s["dir"], labels=s["labels"], mc=s["mc"],
                    long_paths=long_paths)
    if kind == "field":
        s["ctx"].random_field(s["field"], s["seed"], 0, 0, 0.0, s["case"]["rmse"])
        s["ctx"].convolve(s["field"])
        return s["field"]
    if kind == "batch":
        for m in s["mcs"]:
            m.zero_()
        s["batch"].run(s["mcs"], s["case"]["n"], 0, ca.BATCH_GRAPH)
        return s["mcs"]
    if kind == "predict":
        s["net"].predict(s["dem"], s["stream"], NODATA, NODATA, s["case"]["rmse"], s["case"]["pr"],
                         s["prob"])
        return s["prob"]
    loss = s["trainer"].gradients(s["x"], s["y"])
    out = {k: s["trainer"].read(k, shape, grad=True) for k, shape in s["shapes"].items()}
    out["loss"] = loss
    return out


# ---- what a pass cannot do without -----------------------------------------------

def _realization(w, h, model, pr):
    """Bytes and operations of one realization: the DEM and the streams read,
    the counters read and written; the filter's products and sums."""
    taps = 2 * math.ceil(2.5 * pr / CELL) + 1
    if model == "gauss":
        conv = 4 * taps
    elif model == "exp":
        conv = 2 * taps * taps
    else:
        conv = 5 * math.log2(w * h)
    return 16 * w * h, conv * w * h


# name, input channels (the first layer's four planes), output channels, level
LAYERS = [("enc1a", 4, 32, 0), ("enc1b", 32, 32, 0), ("enc2a", 32, 64, 1), ("enc2b", 64, 64, 1),
          ("enc3a", 64, 128, 2), ("enc3b", 128, 128, 2), ("mida", 128, 256, 3),
          ("midb", 256, 256, 3), ("dec3a", 384, 128, 2), ("dec3b", 128, 128, 2),
          ("dec2a", 192, 64, 1), ("dec2b", 64, 64, 1), ("dec1a", 96, 32, 0), ("dec1b", 32, 32, 0)]


def work(case):
    kind = case["kind"]
    if kind == "mc":
        b, f = _realization(case["w"], case["h"], case["model"], case["pr"])
        return dict(bytes=b * case["n"], flops=f * case["n"])
    if kind == "stages":
        # each stage reads its inputs and writes its outputs: 4, 8, 12, 12, 12, 6, 10 and 12
        # bytes a cell
        cells = case["w"] * case["h"]
        return dict(bytes=76 * cells, flops=_realization(case["w"], case["h"], case["model"],
                                                         case["pr"])[1])
    if kind == "field":
        cells = case["w"] * case["h"]
        return dict(bytes=4 * cells, flops=_realization(case["w"], case["h"], case["model"],
                                                        case["pr"])[1])
    if kind == "batch":
        side = (case["lo"] + case["hi"]) / 2.0
        b, f = _realization(side, side, "gauss", 115.0)
        return dict(bytes=b * case["tiles"] * case["n"], flops=f * case["tiles"] * case["n"])
    pixels = case["w"] * case["h"] if kind == "predict" else case["batch"] * case["size"] ** 2
    macs = pixels * (32 + sum(9 * ci * co / 4 ** lv for _, ci, co, lv in LAYERS))
    weights = sum(9 * ci * co for _, ci, co, _ in LAYERS)
    if kind == "predict":
        return dict(bytes=12 * pixels + 2 * weights, flops=2 * macs)
    # forward, gradient of the inputs (not the first layer's), gradient of the weights
    first = pixels * 9 * 4 * 32
    return dict(bytes=20 * pixels + 6 * weights, flops=2 * (3 * macs - first))


# ---- the same in 64 bits ------------------------------------------------------------

def _mul32(a, b):
    """High and low words of the product of 32-bit words (in int64 tensors)."""
    p = a * b
    return (p >> 32) & 0xffffffff, p & 0xffffffff


def _normal_field(w, h, seed, std):
    """std x N(0, 1), one Philox4x32-10 block per four cells and Box-Muller on
    24-bit uniforms, in float64."""
    blocks = (w * h + 3) // 4
    c0 = torch.arange(blocks, dtype=torch.int64, device="cuda")
    c1, c2 = torch.zeros_like(c0), torch.zeros_like(c0)
    c3 = c0 >> 32
    c0 = c0 & 0xffffffff
    k0, k1 = seed & 0xffffffff, seed >> 32
    for _ in range(10):
        hi0, lo0 = _mul32(c0, 0xD2511F53)
        hi1, lo1 = _mul32(c2, 0xCD9E8D57)
        c0, c1, c2, c3 = hi1 ^ c1 ^ k0, lo1, hi0 ^ c3 ^ k1, lo0
        k0, k1 = (k0 + 0x9E3779B9) & 0xffffffff, (k1 + 0xBB67AE85) & 0xffffffff
    out = []
    for a, b in ((c0, c1), (c2, c3)):
        u1 = ((a >> 8) + 1).double() / 2.0 ** 24
        u2 = (b >> 8).double() / 2.0 ** 24
        r = torch.sqrt(-2.0 * torch.log(u1))
        out += [r * torch.cos(2 * math.pi * u2), r * torch.sin(2 * math.pi * u2)]
    return (torch.stack(out, 1).reshape(-1)[:w * h] * std).reshape(h, w)


def _filter_2d(model, pr):
    """The process-convolution filter: the correlogram's square root in the
    frequency domain (the distances and exponents of the exponential one in
    float32, as the filter is defined)."""
    r = int(np.ceil(np.float32(np.float32(pr) / np.float32(CELL)) * np.float32(2.5)))
    y, x = np.mgrid[-r:r + 1, -r:r + 1]
    d2 = x * x + y * y
    if model == "gauss":
        scale = np.float64(np.float32(np.float32(pr) / np.float32(1.73205080757)) / np.float32(CELL))
        c = np.exp(-d2 / scale ** 2).astype(np.float32)
    else:
        scale = np.float32(np.float32(pr) / np.float32(3.0)) / np.float32(CELL)
        c = np.exp((-np.sqrt(d2.astype(np.float32)) / scale).astype(np.float64)).astype(np.float32)
    k = np.fft.irfft2(np.sqrt(np.abs(np.fft.rfft2(c.astype(np.float64)))), s=c.shape)
    k = np.roll(k, (r, r), axis=(0, 1))
    if model == "gauss":
        u, s, _ = np.linalg.svd(k)
        k = np.outer(u[:, 0], u[:, 0]) * s[0]
    return r, k


def _exact_field(case, seed):
    w, h = case["w"], case["h"]
    field = _normal_field(w, h, seed, float(np.float32(case["rmse"])))
    r, k = _filter_2d(case["model"], case["pr"])
    torus = torch.zeros((h, w), dtype=torch.float64, device="cuda")
    iy = torch.arange(-r, r + 1, device="cuda") % h
    ix = torch.arange(-r, r + 1, device="cuda") % w
    # a filter wider than the grid wraps onto itself
    torus.index_put_((iy[:, None].expand(k.shape), ix[None, :].expand(k.shape)),
                     torch.from_numpy(k).cuda(), accumulate=True)
    spectrum = torch.fft.rfft2(field) * torch.fft.rfft2(torus).conj()
    return torch.fft.irfft2(spectrum, s=(h, w))


def _bf16(a):
    """Nearest bfloat16, ties to even, as float32."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7fff + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


def _initial_weights(seed):
    """Weights as a training run begins with them: He-normal, the
    convolutions' rounded to bfloat16 as a weights file holds them; the first
    layer reads 32 channels, of which four are planes."""
    rng = np.random.default_rng(seed)
    params = {}
    for name, ci, co, _ in LAYERS:
        w = np.zeros((9, co, max(ci, 32)), np.float32)
        w[:, :, :ci] = rng.normal(0.0, math.sqrt(2.0 / (9 * ci)), (9, co, ci))
        params[name + ".w"] = _bf16(w).reshape(w.shape)
        params[name + ".b"] = rng.normal(0.0, 0.05, co).astype(np.float32)
    params["head.w"] = rng.normal(0.0, math.sqrt(1.0 / 32), 32).astype(np.float32)
    params["head.b"] = np.full(1, -2.0, np.float32)  # borders are rare
    return params


def _read_weights(path):
    """Tensors of a weights file: float32, or bfloat16 bit patterns."""
    params = {}
    with open(path, "rb") as f:
        f.read(8)
        _, count = struct.unpack("<ii", f.read(8))
        for _ in range(count):
            name = f.read(struct.unpack("<i", f.read(4))[0]).decode()
            half, ndim = struct.unpack("<ii", f.read(8))
            shape = struct.unpack("<%di" % ndim, f.read(4 * ndim))
            count_of = int(np.prod(shape))
            if half:
                raw = np.frombuffer(f.read(2 * count_of), "<u2").astype(np.uint32) << 16
                params[name] = raw.view(np.float32).reshape(shape)
            else:
                params[name] = np.frombuffer(f.read(4 * count_of), "<f4").reshape(shape)
    return params


def _logits(p, x):
    """The network in float64: x [n][h][w][4], p the parameters as float64
    device tensors."""
    def conv(name, a):
        n, h, w, c = a.shape
        a = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        out = p[name + ".b"]
        for tap in range(9):
            part = a[:, tap // 3:tap // 3 + h, tap % 3:tap % 3 + w].reshape(-1, c)
            out = out + part @ p[name + ".w"][tap, :, :c].t()
        return torch.relu(out).reshape(n, h, w, -1)

    def pool(a):
        n, h, w, c = a.shape
        return a.reshape(n, h // 2, 2, w // 2, 2, c).mean((2, 4))

    def up(a):
        n, h, w, c = a.shape
        return a[:, :, None, :, None].expand(n, h, 2, w, 2, c).reshape(n, 2 * h, 2 * w, c)

    e1 = conv("enc1b", conv("enc1a", x))
    e2 = conv("enc2b", conv("enc2a", pool(e1)))
    e3 = conv("enc3b", conv("enc3a", pool(e2)))
    a = conv("midb", conv("mida", pool(e3)))
    for k, skip in ((3, e3), (2, e2), (1, e1)):
        a = conv("dec%db" % k, conv("dec%da" % k, torch.cat([up(a), skip], -1)))
    return (a * p["head.w"]).sum(-1) + p["head.b"]


def _f64(params):
    return {k: torch.from_numpy(np.array(v, np.float64)).cuda() for k, v in params.items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "field":
        return _exact_field(case, seed)
    if kind == "predict":
        w, h = case["w"], case["h"]
        dem, stream = _dem(w, h, seed)
        d = dem.double()
        # the network halves its input three times: zero planes beyond the raster
        x = torch.zeros((1, h + -h % 8, w + -w % 8, 4), dtype=torch.float64, device="cuda")
        x[0, :h, :w, 0] = (d - d.mean()) / d.std(unbiased=False)
        x[0, :h, :w, 1] = (stream != NODATA).double()
        x[0, :h, :w, 2] = case["rmse"] / 3.0
        x[0, :h, :w, 3] = case["pr"] / 200.0
        with torch.no_grad():
            logits = _logits(_f64(_read_weights(sg.DEFAULT_WEIGHTS)), x)
        return torch.sigmoid(logits)[0, :h, :w].contiguous()
    if kind == "train":
        x, y = (t.double() for t in _train_inputs(case, seed))
        p = {k: v.requires_grad_() for k, v in _f64(_initial_weights(seed)).items()}
        loss = 0.0
        for k in range(case["batch"]):  # one tile at a time: the products' copies are large
            part = torch.nn.functional.binary_cross_entropy_with_logits(
                _logits(p, x[k:k + 1]), y[k:k + 1]) / case["batch"]
            part.backward()
            loss += float(part.detach())
        out = {k: v.grad for k, v in p.items()}
        out["loss"] = loss
        return out
    return None  # counts, directions and labels of a chain of comparisons
