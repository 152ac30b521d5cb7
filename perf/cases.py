# SPDX-License-Identifier: Unlicense
"""The framework's work as measurable cases: single layers through the
generic operations, the matchers' own kernels, and three whole networks.

A case is a dict of plain values with a "kind":

linear     ops_linear, token-major (the transformers' products)
block      a refiner block: roma_dwconv5, then ops_conv1x1
attention  ops_attention_batch on packed q, k, v rows
conv       ops_conv2d_batch, with DISK's input normalisation or without
corr       roma_local_corr
gp         roma_gp_solve
eloftr     an ELoFTR grey pair in device memory, matches out
roma       a RoMa pair's coarse forward in device memory
disk       DISK on a host image, keypoints and descriptors out

Layer cases keep their tensors in torch memory and hand the library views
of it. Network cases keep one loaded network per size; a state is that
network with one pair of images.
"""

import importlib.util
import math
import shutil
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

ROOT = Path(__file__).resolve().parent.parent
ACT_NONE, ACT_GELU, ACT_RELU = 0, 1, 2
WEIGHT_SEED = 20261201


def _package(name="icoreg_amd", part="__init__.py"):
    """The package (its folder is no Python identifier) or a module of it."""
    if name not in sys.modules:
        folder = ROOT / "i.coregistration.opencl_amd"
        spec = importlib.util.spec_from_file_location(name, folder / part)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


_held = {}  # the device, and the networks' weights and loaded networks


def _device():
    if "device" not in _held:
        torch.cuda.init()
        _held["device"] = _package().Device("auto")
    return _held["device"]


def _wrap(t):
    """The library's view of a torch tensor (which the state keeps)."""
    return _package().lib().ocl_wrap(t.data_ptr(), t.numel() * t.element_size())


class _Memory:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": "<f4",
                                         "strides": None, "version": 3}


def _tensor(mem, shape):
    """A library buffer's first floats as a torch tensor."""
    return torch.as_tensor(_Memory(mem.contents.ptr, shape), device="cuda")


# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # ELoFTR's query projection on the 20 x 20 aggregated tokens of a
        # 640 x 640 tile: the smallest product, launch and latency.
        {"name": "linear_agg_400", "kind": "linear", "rows": 400, "cin": 256, "cout": 256, "act": ACT_NONE,
         "bias": False, "residual": False},
        # DINOv2 ViT-L/14's first MLP layer on a 560 x 560 pair's tokens.
        {"name": "linear_vit_fc1", "kind": "linear", "rows": 3202, "cin": 1024, "cout": 4096, "act": ACT_GELU,
         "bias": True, "residual": False},
        # Its attention, and ELoFTR's aggregated attention.
        {"name": "attention_vit", "kind": "attention", "images": 2, "nq": 1601, "nk": 1601, "heads": 16, "d": 64},
        {"name": "attention_agg", "kind": "attention", "images": 2, "nq": 400, "nk": 400, "heads": 8, "d": 32},
        # ELoFTR's backbone at 1/2 of 640 x 640, both images.
        {"name": "conv3_pair_320", "kind": "conv", "images": 2, "k": 3, "stride": 1, "cin": 64, "cout": 64,
         "h": 320, "w": 320, "norm": False},
        # DISK's last layer at 512 x 512.
        {"name": "conv5_norm_512", "kind": "conv", "images": 1, "k": 5, "stride": 1, "cin": 80, "cout": 129,
         "h": 512, "w": 512, "norm": True},
        # A block of RoMa's 1/4 refiner on a 864 x 864 tile.
        {"name": "refiner_block_4", "kind": "block", "c": 572, "h": 216, "w": 216},
        # RoMa's 1/8 refiner's local correlation on the same tile.
        {"name": "local_corr_8", "kind": "corr", "c": 512, "h": 108, "w": 108, "r": 3},
        # The match encoder's Gaussian process at 560 x 560.
        {"name": "gp_solve_1600", "kind": "gp", "n": 1600, "d": 512},
        # The two headline networks and DISK, whole.
        {"name": "eloftr_640", "kind": "eloftr", "h": 640, "w": 640},
        {"name": "roma_coarse_560", "kind": "roma", "coarse": 560},
        {"name": "disk_512", "kind": "disk", "h": 512, "w": 512},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "attention", "attention", "conv", "conv", "block", "corr", "gp",
                       "eloftr", "roma", "disk"])
    if kind == "linear":
        # Channel counts as the networks have them, or any.
        width = lambda: rng.choice([256, 512, 1024, 3072, 4096]) if rng.random() < 0.6 else _log(rng, 64, 4096)  # noqa: E731
        return {"kind": kind, "rows": _log(rng, 16, 4096), "cin": width(), "cout": width(),
                "act": rng.choice([ACT_NONE, ACT_GELU, ACT_RELU]), "bias": rng.random() < 0.7,
                "residual": rng.random() < 0.3}
    if kind == "attention":
        nq = _log(rng, 49, 2304)
        return {"kind": kind, "images": rng.randint(1, 2), "nq": nq,
                "nk": nq if rng.random() < 0.7 else _log(rng, 49, 2304), "heads": rng.choice([4, 8, 16]),
                "d": rng.choice([32, 64, 128])}
    if kind == "conv":
        k = rng.choice([3, 3, 5])
        return {"kind": kind, "images": 1 if k == 5 else rng.randint(1, 2), "k": k,
                "stride": 1 if k == 5 or rng.random() < 0.8 else 2,
                "cin": rng.choice([3, 16, 32, 64, 80, 96, 128, 256]),
                "cout": rng.choice([16, 32, 64, 64, 128, 129, 256]),
                "h": _log(rng, 32, 432), "w": _log(rng, 32, 432), "norm": k == 5 and rng.random() < 0.8}
    if kind == "block":
        return {"kind": kind, "c": rng.choice([144, 572, 1140, rng.randint(33, 600)]),
                "h": _log(rng, 40, 256), "w": _log(rng, 40, 256)}
    if kind == "corr":
        return {"kind": kind, "c": rng.choice([64, 128, 192, 256, 512]), "h": rng.randint(20, 160),
                "w": rng.randint(20, 160), "r": rng.choice([1, 2, 3, 3, 7])}
    if kind == "gp":
        return {"kind": kind, "n": rng.randint(16, 40) ** 2, "d": rng.choice([256, 512])}
    if kind == "eloftr":
        return {"kind": kind, "h": 32 * rng.randint(6, 26), "w": 32 * rng.randint(6, 26)}
    if kind == "roma":
        return {"kind": kind, "coarse": 56 * rng.randint(4, 10)}
    return {"kind": kind, "h": 16 * rng.randint(8, 48), "w": 16 * rng.randint(8, 48)}


# ---- inputs ------------------------------------------------------------------


def _rng(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _blurred(g, shape):
    """Smooth noise in 0..1, as image tiles are."""
    x = torch.rand((1,) + shape, generator=g, device="cuda")
    for _ in range(3):
        x = F.avg_pool2d(x, 5, 1, 2, count_include_pad=False)
    x = x[0]
    return (x - x.min()) / (x.max() - x.min())


def _shifted(g, a, step, reach):
    """a moved by whole steps of up to reach px with zeros behind, and a
    little noise: the second image of a pair."""
    dy, dx = ((torch.randint(-(reach // step), reach // step + 1, (2,), generator=g, device="cuda") * step).tolist())
    h, w = a.shape[-2:]
    b = torch.zeros_like(a)
    b[..., max(dy, 0):h + min(dy, 0), max(dx, 0):w + min(dx, 0)] = \
        a[..., max(-dy, 0):h - max(dy, 0), max(-dx, 0):w - max(dx, 0)]
    return b + 0.01 * torch.randn(a.shape, generator=g, device="cuda")


def _inputs(c, seed):
    g, k = _rng(seed), c["kind"]
    randn = lambda *s, std=1.0: std * torch.randn(s, generator=g, device="cuda")  # noqa: E731
    rand = lambda *s, lo=0.0, hi=1.0: lo + (hi - lo) * torch.rand(s, generator=g, device="cuda")  # noqa: E731
    if k == "linear":
        # Normalised tokens and weights that keep their scale.
        return {"x": randn(c["rows"], c["cin"]), "w": randn(c["cout"], c["cin"], std=c["cin"] ** -0.5),
                "b": rand(c["cout"], lo=-0.05, hi=0.05) if c["bias"] else None,
                "y": randn(c["rows"], c["cout"]) if c["residual"] else None}
    if k == "block":
        n = c["c"]
        return {"x": randn(n, c["h"], c["w"]), "dw": randn(n, 25, std=(2 / 25) ** 0.5), "db": rand(n, lo=-0.1, hi=0.1),
                "pw": randn(n, n, std=(2 / n) ** 0.5), "pb": rand(n, lo=-0.05, hi=0.05)}
    if k == "attention":
        D = c["heads"] * c["d"]
        return {"q": randn(c["images"], c["nq"], D, std=1.4), "kv": randn(c["images"], c["nk"], 2 * D, std=1.4)}
    if k == "conv":
        ci, co, kk = c["cin"], c["cout"], c["k"]
        x = randn(c["images"], ci, c["h"], c["w"])
        d = {"x": x if c["norm"] or ci <= 3 else x.relu_(), "w": randn(co, ci, kk, kk, std=(2 / (ci * kk * kk)) ** 0.5),
             "b": rand(co, lo=-0.1, hi=0.1)}
        if c["norm"]:
            d.update(mean=randn(ci, std=0.1), rstd=rand(ci, lo=0.8, hi=1.25), gate=rand(ci, lo=0.1, hi=0.3))
        return d
    if k == "corr":
        h, w = c["h"], c["w"]
        gy, gx = torch.meshgrid(_centres(h), _centres(w), indexing="ij")
        bend = torch.stack([0.03 * torch.sin(3 * gy + 1), 0.03 * torch.cos(2 * gx)])
        jitter = randn(2, h, w) * torch.tensor([0.5 / w, 0.5 / h], device="cuda")[:, None, None]
        return {"f1": randn(c["c"], h, w), "f2": randn(c["c"], h, w),
                "flow": (torch.stack([gx, gy]) + bend + jitter).float()}
    if k == "gp":
        # The cosine kernel of tokens that share a few directions.
        z = randn(c["n"], 24).double() @ randn(24, 512).double()
        z = z / z.norm(dim=1, keepdim=True)
        return {"K": torch.exp((z @ z.T - 1) / 0.2).float(), "F": torch.cos(3 * randn(c["n"], c["d"]))}
    if k == "eloftr":
        a = rand(c["h"], c["w"])
        return {"a": a, "b": _shifted(g, a, 8, 32)}
    if k == "roma":
        a = _blurred(g, (3, c["coarse"], c["coarse"]))
        pair = torch.stack([a, _shifted(g, a, 1, 20)])
        mean, std = (torch.tensor(v, device="cuda")[None, :, None, None] for v in ((0.485, 0.456, 0.406),
                                                                                  (0.229, 0.224, 0.225)))
        return {"pair": ((pair - mean) / std).contiguous()}
    return {"image": _blurred(g, (3, c["h"], c["w"]))}


def _centres(n):
    return torch.linspace(-1 + 1 / n, 1 - 1 / n, n, device="cuda", dtype=torch.float64)


# ---- the networks ------------------------------------------------------------


def _weights(kind):
    """Seeded random weights, drawn once."""
    synth = _package("icoreg_amd_synth", "synth.py")
    if kind not in _held:
        _held[kind] = {"eloftr": lambda: [synth.eloftr_weights_calibrated(WEIGHT_SEED + 1, 128)],
                       "roma": lambda: [synth.roma_weights(WEIGHT_SEED + 2), synth.dino_weights(WEIGHT_SEED + 2)],
                       "disk": lambda: [synth.disk_weights(WEIGHT_SEED)]}[kind]()
    return _held[kind]


def _network(c):
    """The network of a case's kind and size, loaded from a weights file."""
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if key not in _held:
        ic, synth, folder = _package(), _package("icoreg_amd_synth", "synth.py"), tempfile.mkdtemp()
        try:
            files = [synth.save_safetensors(w, Path(folder) / f"{i}.safetensors")
                     for i, w in enumerate(_weights(c["kind"]))]
            if c["kind"] == "eloftr":
                net = ic.Eloftr(_device(), files[0], c["h"], c["w"])
            elif c["kind"] == "roma":
                net = ic.Roma(_device(), files[0], files[1], c["coarse"], c["coarse"], coarse=c["coarse"])
            else:
                net = ic.Disk(_device(), files[0], c["h"], c["w"], 2048)
        finally:
            shutil.rmtree(folder)
        _held[key] = net
    return _held[key]


# ---- a state and a pass ------------------------------------------------------


def prepare(case, seed):
    c, dev, ic = case, _device(), _package()
    k, t = c["kind"], _inputs(c, seed)
    s = {"kind": k, "case": c, "t": t, "api": dev.api, "dev": dev}
    empty = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if k in ("eloftr", "roma", "disk"):
        net = s["net"] = _network(c)
        if k == "eloftr":
            n, lib = (c["h"] // 8) * (c["w"] // 8), ic.lib()
            s["out"] = {name: _tensor(lib.icoreg_eloftr_buffer(net.m, name.encode()), shape)
                        for name, shape in (("x0", (256, n)), ("x1", (256, n)), ("row_lse", (n,)),
                                            ("fineh0", (64, c["h"] // 2, c["w"] // 2)),
                                            ("fineh1", (64, c["h"] // 2, c["w"] // 2)))}
        elif k == "roma":
            n, lib = (c["coarse"] // 14) ** 2, ic.lib()
            s["out"] = {name: _tensor(lib.icoreg_roma_buffer(net.m, name.encode()), shape)
                        for name, shape in (("g_y", (2, n, 512)), ("t_x", (n, 1024)), ("t_out", (n, 4097)))}
        else:
            s["out"] = {"out": _tensor(ic.lib().icoreg_disk_buffer(net.m, b"out"), (129, c["h"], c["w"]))}
            s["image"] = t["image"].cpu().numpy()
        if k != "disk":
            s["m"] = {name: ic.Buffer(dev, _wrap(v), v.numel() * 4) for name, v in t.items()}
        torch.cuda.synchronize()
        return s
    if k == "linear":
        out = t["y"] if t["y"] is not None else empty(c["rows"], c["cout"])
    elif k == "block":
        out, s["mid"] = empty(c["c"], c["h"], c["w"]), empty(c["c"], c["h"], c["w"])
    elif k == "attention":
        out = empty(c["images"], c["nq"], c["heads"] * c["d"])
    elif k == "conv":
        p, st = c["k"] // 2, c["stride"]
        ho, wo = ((n + 2 * p - c["k"]) // st + 1 for n in (c["h"], c["w"]))
        out, s["geom"] = empty(c["images"], c["cout"], ho, wo), ic.geom(c["k"], c["k"], st, st, p, p, 1, 1, 1)
    elif k == "corr":
        out = empty((2 * c["r"] + 1) ** 2, c["h"], c["w"])
    else:
        out = empty(c["n"], c["d"])
        s["work"] = torch.empty(ic.lib().roma_gp_work_bytes(c["n"], c["d"]), dtype=torch.uint8, device="cuda")
        s["info"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    s["out"] = out
    s["m"] = {name: _wrap(v) for name, v in {**t, "out": out, "mid": s.get("mid"), "work": s.get("work"),
                                             "info": s.get("info")}.items() if v is not None}
    torch.cuda.synchronize()
    return s


def run(s):
    c, k, a, po, m = s["case"], s["kind"], s["api"], s["dev"].po, s.get("m")
    ic = _package()
    if k == "linear":
        a.ops_linear(po, c["rows"], c["cin"], c["cout"], m["x"], 0, m["w"], m.get("b"), m["out"], 0, c["act"], 0.0,
                     int(c["residual"]))
    elif k == "block":
        n = c["h"] * c["w"]
        a.roma_dwconv5(po, m["x"], c["c"], c["h"], c["w"], m["dw"], m["db"], m["mid"])
        a.ops_conv1x1(po, m["mid"], 0, c["c"], n, m["pw"], m["pb"], c["c"], m["out"], 0, ACT_NONE, 0.0)
    elif k == "attention":
        D = c["heads"] * c["d"]
        a.ops_attention_batch(po, c["images"], ic.Opnd(m["q"], 0, D, 0, 0), c["nq"] * D,
                              ic.Opnd(m["kv"], 0, 2 * D, 0, 0), c["nk"] * 2 * D,
                              ic.Opnd(m["kv"], D, 2 * D, 0, 0), c["nk"] * 2 * D,
                              ic.Opnd(m["out"], 0, D, 0, 0), c["nq"] * D, c["nq"], c["nk"], c["heads"], c["d"],
                              c["d"] ** -0.5, None)
    elif k == "conv":
        o = s["out"]
        a.ops_conv2d_batch(po, c["images"], m["x"], c["cin"] * c["h"] * c["w"], c["cin"], c["h"], c["w"], m["w"],
                           m["b"], c["cout"], ic.C.byref(s["geom"]), m.get("mean"), m.get("rstd"), m.get("gate"),
                           ACT_NONE if c["norm"] else ACT_RELU, 0.0, m["out"], o[0].numel())
    elif k == "corr":
        a.roma_local_corr(po, m["f1"], m["f2"], c["c"], c["h"], c["w"], c["r"], m["flow"], m["out"], 0)
    elif k == "gp":
        # The solve is in place: the right-hand side is copied in first, as RoMa's driver does.
        a.ocl_copy(s["dev"].pb, m["F"], 0, m["out"], 0, c["n"] * c["d"] * 4)
        a.roma_gp_solve(po, m["K"], c["n"], 0.1, m["out"], c["d"], m["work"], m["info"])
    elif k == "eloftr":
        s["net"].match_device(m["a"], m["b"])
    elif k == "roma":
        s["net"].coarse_device(m["pair"])
    else:
        s["keypoints"] = s["net"].detect(s["image"])
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------


def _conv_flops(cin, cout, k, cells):
    return 2 * cin * cout * k * k * cells


def work(c):
    k = c["kind"]
    if k == "linear":
        r, i, o = c["rows"], c["cin"], c["cout"]
        return {"bytes": 4 * (r * i + i * o + o * c["bias"] + r * o * (1 + c["residual"])), "flops": 2 * r * i * o}
    if k == "block":
        n, ch = c["h"] * c["w"], c["c"]
        return {"bytes": 4 * (2 * ch * n + ch * ch + 27 * ch), "flops": 2 * n * ch * (ch + 25)}
    if k == "attention":
        D, b = c["heads"] * c["d"], c["images"]
        return {"bytes": 4 * b * D * 2 * (c["nq"] + c["nk"]), "flops": 4 * b * c["nq"] * c["nk"] * D}
    if k == "conv":
        out = c["images"] * (-(-c["h"] // c["stride"])) * (-(-c["w"] // c["stride"]))
        return {"bytes": 4 * (c["images"] * c["cin"] * c["h"] * c["w"] + c["cin"] * c["cout"] * c["k"] ** 2
                              + c["cout"] * (1 + out)), "flops": _conv_flops(c["cin"], c["cout"], c["k"], out)}
    if k == "corr":
        n, win = c["h"] * c["w"], (2 * c["r"] + 1) ** 2
        # Bilinear weights commute with the dot product: one more row and column of products a cell.
        return {"bytes": 4 * n * (2 * c["c"] + 2 + win), "flops": 2 * c["c"] * n * (2 * c["r"] + 2) ** 2}
    if k == "gp":
        n, d = c["n"], c["d"]
        return {"bytes": 4 * (n * n + 2 * n * d), "flops": n ** 3 / 3 + 2 * n * n * d}
    if k == "eloftr":
        return _eloftr_work(c["h"], c["w"])
    if k == "roma":
        return _roma_work(c["coarse"])
    n, cin, cout = c["h"] * c["w"], (3, 16, 32, 64, 64, 128, 128, 96, 80), (16, 32, 64, 64, 64, 64, 64, 64, 129)
    at = (0, 1, 2, 3, 4, 3, 2, 1, 0)
    return {"bytes": 4 * (3 * n + 129 * n + sum(25 * i * o for i, o in zip(cin, cout))),
            "flops": sum(_conv_flops(i, o, 5, n >> (2 * s)) for i, o, s in zip(cin, cout, at))}


def _eloftr_work(h, w):
    hw, n, fl, params, cin = h * w, h * w // 64, 0, 0, 1
    for stage, (blocks, cout, shift) in enumerate(((1, 64, 2), (2, 64, 2), (4, 128, 4), (14, 256, 6))):
        for _ in range(blocks):
            fl += 2 * _conv_flops(cin, cout, 3, hw >> shift)
            params, cin = params + 9 * cin * cout, cout
    na = n // 16
    # Per image and layer, self and cross: projections, attention, the message and the MLP's three parts.
    per = 2 * na * 256 * 256 * 3 + 4 * na * na * 256 + 2 * na * 256 * 512 + 2 * n * 512 * (256 + 256)
    fl += 2 * 8 * per + 2 * n * n * 256
    params += 8 * (3 * 256 * 256 + 512 * 256 + 512 * 256 + 512 * 256)
    for ci, co, k, s in ((256, 256, 1, 6), (128, 256, 1, 4), (256, 256, 3, 4), (256, 128, 3, 4), (64, 128, 1, 2),
                         (128, 128, 3, 2), (128, 64, 3, 2)):
        fl += 2 * _conv_flops(ci, co, k, hw >> s)
        params += ci * co * k * k
    return {"bytes": 4 * (2 * hw + params + 2 * 256 * n + 2 * 64 * (hw // 4) + n), "flops": fl}


def _roma_work(side):
    n, D = (side // 14) ** 2, 1024
    t = n + 1
    block = lambda rows, keys: 24 * rows * D * D + 4 * rows * keys * D  # noqa: E731
    fl = 2 * (2 * n * 588 * D + 24 * block(t, t)) + 2 * 2 * n * D * 512  # the ViT, the projection
    fl += 2 * (2 * n * n * 512) + n ** 3 / 3 + 2 * n * n * 512 + 2 * n * n * 512  # the two kernels, the solve, the mean
    fl += 5 * block(n, n) + 2 * n * D * 4097
    params = 29 * 12 * D * D + 588 * D + D * 512 + D * 4097
    return {"bytes": 4 * (6 * side * side + params + 2 * n * 512 + n * (D + 4097)), "flops": fl}


def tolerance(c):
    # About four times what the paths differ from 64 bits by: sums of 32-bit
    # products, in the local correlation the 32-bit sampling positions, in the
    # networks what their layers pass on.
    return {"linear": {"rel": 4e-6, "max": 2e-4}, "block": {"rel": 2e-6, "max": 1e-4},
            "attention": {"rel": 4e-6, "max": 2e-4}, "conv": {"rel": 6e-6, "max": 3e-4},
            "corr": {"rel": 2e-5, "max": 1e-3}, "gp": {"rel": 5e-7, "max": 1e-5},
            "eloftr": {"rel": 2e-5, "max": 2e-3}, "roma": {"rel": 5e-5, "max": 4e-3},
            "disk": {"rel": 6e-6, "max": 4e-4}}[c["kind"]]


# ---- the same in 64 bits -----------------------------------------------------


def exact(case, seed):
    """run's answer for these inputs from plain torch in 64 bits."""
    c, k = case, case["kind"]
    t = {n: v.double() for n, v in _inputs(c, seed).items() if v is not None}
    if k == "linear":
        y = t["x"] @ t["w"].T + t.get("b", 0.0)
        y = F.gelu(y) if c["act"] == ACT_GELU else y.relu() if c["act"] == ACT_RELU else y
        return y + t.get("y", 0.0)
    if k == "block":
        y = F.pad(t["x"], (2, 2, 2, 2))
        z = sum(t["dw"][:, 5 * i + j, None, None] * y[:, i:i + c["h"], j:j + c["w"]] for i in range(5)
                for j in range(5))
        z = (z + t["db"][:, None, None]).relu().reshape(c["c"], -1)
        return (t["pw"] @ z + t["pb"][:, None]).reshape(c["c"], c["h"], c["w"])
    if k == "attention":
        D = c["heads"] * c["d"]
        return _attend(t["q"], t["kv"][..., :D], t["kv"][..., D:], c["heads"])
    if k == "conv":
        x = t["x"]
        if c["norm"]:
            x = (x - t["mean"][:, None, None]) * t["rstd"][:, None, None]
            x = torch.where(x >= 0, x, t["gate"][:, None, None] * x)
        y = torch.stack([_conv(v, t["w"], t["b"], c["stride"]) for v in x])
        return y if c["norm"] else y.relu()
    if k == "corr":
        return _correlate(t["f1"], t["f2"], t["flow"], c["r"])
    if k == "gp":
        K = t["K"].cpu() + float(np.float32(0.1)) * torch.eye(c["n"], dtype=torch.float64)
        return torch.cholesky_solve(t["F"].cpu(), torch.linalg.cholesky(K))
    w = [{n: torch.from_numpy(v).cuda() for n, v in d.items()} for d in _weights(k)]
    return _eloftr(w[0], t) if k == "eloftr" else _roma(w[0], w[1], t, c["coarse"]) if k == "roma" else \
        {"out": _disk(w[0], t["image"])}


def _conv(x, w, b=None, stride=1, pad=None):
    """(C, H, W) through a k x k convolution, one product a tap."""
    k = w.shape[-1]
    p = k // 2 if pad is None else pad
    x, w = F.pad(x, (p, p, p, p)), w.double()
    h, wd = ((n - k) // stride + 1 for n in x.shape[-2:])
    y = 0
    for i in range(k):
        for j in range(k):
            v = x[:, i:i + (h - 1) * stride + 1:stride, j:j + (wd - 1) * stride + 1:stride]
            y = y + w[:, :, i, j].contiguous() @ v.reshape(x.shape[0], -1)
    return (y if b is None else y + b.double()[:, None]).reshape(-1, h, wd)


def _attend(q, k, v, heads):
    q, k, v = (z.unflatten(-1, (heads, -1)).transpose(-3, -2).contiguous() for z in (q, k, v))
    p = torch.softmax(q @ k.transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5, -1)
    return (p @ v).transpose(-3, -2).flatten(-2)


def _correlate(f1, f2, flow, r):
    C, h, w = f1.shape
    out = []
    for a in range(-r, r + 1):
        for b in range(-r, r + 1):
            at = flow + torch.tensor([2 * b / w, 2 * a / h], device="cuda", dtype=torch.float64)[:, None, None]
            v = F.grid_sample(f2[None], at.permute(1, 2, 0)[None], "bilinear", "zeros", False)[0]
            out.append((f1 * v).sum(0) / math.sqrt(C))
    return torch.stack(out)


def _bn(w, p, y):
    g = w[p + ".weight"].double() / torch.sqrt(w[p + ".running_var"].double() + 1e-5)
    return (y - w[p + ".running_mean"].double()[:, None, None]) * g[:, None, None] + \
        w[p + ".bias"].double()[:, None, None]


def _eloftr(w, t):
    """Efficient LoFTR's coarse features of both images, the row
    log-sum-exp of their scores and the fine maps at half resolution."""
    P, first, half, quarter = "efficientloftr.", [], [], []
    for x in (t["a"][None], t["b"][None]):
        for s, blocks in enumerate((1, 2, 4, 14)):
            for i in range(blocks):
                p, st = f"{P}backbone.stages.{s}.blocks.{i}", (2, 1, 2, 2)[s] if i == 0 else 1
                y = _bn(w, p + ".conv1.norm", _conv(x, w[p + ".conv1.conv.weight"], stride=st)) + \
                    _bn(w, p + ".conv2.norm", _conv(x, w[p + ".conv2.conv.weight"], stride=st))
                if p + ".identity.weight" in w:
                    y = y + _bn(w, p + ".identity", x)
                x = y.relu()
            (half if s == 1 else quarter if s == 2 else first if s == 3 else []).append(x)
    X = first
    ah, aw = X[0].shape[1] // 4, X[0].shape[2] // 4
    # 2-D rotary angles: even pairs turn with the row, odd ones with the column, both from 1.
    f = 10000.0 ** (-2 * torch.arange(64, device="cuda", dtype=torch.float64) / 128)
    row = torch.arange(1, ah + 1, device="cuda", dtype=torch.float64)[:, None, None].expand(ah, aw, 64) * f
    col = torch.arange(1, aw + 1, device="cuda", dtype=torch.float64)[None, :, None].expand(ah, aw, 64) * f
    ang = torch.stack([row, col], -1).reshape(ah * aw, 128)
    cs, sn = ang.cos(), ang.sin()

    def turn(v):
        a, b = v[:, 0::2], v[:, 1::2]
        return torch.stack([a * cs - b * sn, b * cs + a * sn], -1).flatten(1)

    def attend(p, x, y, rope):
        d = lambda n: w[f"{p}.{n}"].double()  # noqa: E731
        win = x.reshape(256, ah, 4, aw, 4)
        q = (win * d("aggregation.q_aggregation.weight").reshape(256, 1, 4, 1, 4)).sum((2, 4)).reshape(256, -1).T
        kv = y.reshape(256, ah, 4, aw, 4).amax((2, 4)).reshape(256, -1).T
        q, kv = (F.layer_norm(v, (256,), d("aggregation.norm.weight"), d("aggregation.norm.bias"), 1e-5)
                 for v in (q, kv))
        q, key, v = (z @ d(f"attention.{n}_proj.weight").T for n, z in (("q", q), ("k", kv), ("v", kv)))
        if rope:
            q, key = turn(q), turn(key)
        m = (_attend(q, key, v, 8) @ d("attention.o_proj.weight").T).T.reshape(1, 256, ah, aw)
        m = F.interpolate(m, scale_factor=4, mode="bilinear", align_corners=False)[0]
        z = F.leaky_relu(d("mlp.fc1.weight") @ torch.cat([x, m]).flatten(1), 0.01)
        z = F.layer_norm((d("mlp.fc2.weight") @ z).T, (256,), d("mlp.layer_norm.weight"), d("mlp.layer_norm.bias"),
                         1e-5)
        return x + z.T.reshape(x.shape)

    for i in range(4):
        p = f"{P}local_feature_transformer.layers.{i}"
        X = [attend(p + ".self_attention", x, x, True) for x in X]
        X[0] = attend(p + ".cross_attention", X[0], X[1], False)
        X[1] = attend(p + ".cross_attention", X[1], X[0], False)
    out = {"x0": X[0].flatten(1), "x1": X[1].flatten(1)}
    out["row_lse"] = torch.logsumexp(out["x0"].T @ out["x1"] / 25.6, 1)
    for i in range(2):
        y = _conv(X[i] / 16, w["refinement_layer.out_conv.weight"])
        for j, skip in enumerate((quarter[i], half[i])):
            p = f"refinement_layer.out_conv_layers.{j}"
            y = F.interpolate(y[None], scale_factor=2, mode="bilinear", align_corners=False)[0]
            y = y + _conv(skip, w[p + ".out_conv1.weight"])
            y = F.leaky_relu(_bn(w, p + ".batch_norm", _conv(y, w[p + ".out_conv2.weight"])), 0.01)
            y = _conv(y, w[p + ".out_conv3.weight"])
        out[f"fineh{i}"] = y
    return out


def _vit_block(w, p, x, heads, eps):
    d = lambda n: w[f"{p}.{n}"].double() if f"{p}.{n}" in w else None  # noqa: E731
    qkv = F.linear(F.layer_norm(x, (1024,), d("norm1.weight"), d("norm1.bias"), eps), d("attn.qkv.weight"),
                   d("attn.qkv.bias"))
    y = F.linear(_attend(*qkv.split(1024, -1), heads), d("attn.proj.weight"), d("attn.proj.bias"))
    x = x + (y if d("ls1.gamma") is None else y * d("ls1.gamma"))
    y = F.gelu(F.linear(F.layer_norm(x, (1024,), d("norm2.weight"), d("norm2.bias"), eps), d("mlp.fc1.weight"),
                        d("mlp.fc1.bias")))
    y = F.linear(y, d("mlp.fc2.weight"), d("mlp.fc2.bias"))
    return x + (y if d("ls2.gamma") is None else y * d("ls2.gamma"))


def _roma(wm, wd, t, side):
    """RoMa's coarse forward: the projected DINOv2 tokens, the decoder's
    tokens and its anchor logits."""
    c16, D = side // 14, 1024
    pos = wd["pos_embed"][0].double()
    grid = F.interpolate(pos[1:].reshape(1, 37, 37, D).permute(0, 3, 1, 2),
                         scale_factor=((c16 + 0.1) / 37, (c16 + 0.1) / 37), mode="bicubic", align_corners=False)
    pos = torch.cat([pos[:1], grid[0].reshape(D, -1).T])
    g = []
    for img in t["pair"]:
        patch = img.reshape(3, c16, 14, c16, 14).permute(1, 3, 0, 2, 4).reshape(c16 * c16, -1)
        x = patch @ wd["patch_embed.proj.weight"].double().reshape(D, -1).T + wd["patch_embed.proj.bias"].double()
        x = torch.cat([wd["cls_token"][0].double(), x]) + pos
        for i in range(24):
            x = _vit_block(wd, f"blocks.{i}", x, 16, 1e-6)
        x = F.layer_norm(x, (D,), wd["norm.weight"].double(), wd["norm.bias"].double(), 1e-6)[1:]
        p = "decoder.proj.16"
        y = x @ wm[p + ".0.weight"].double().reshape(512, D).T + wm[p + ".0.bias"].double()
        g.append(_bn(wm, p + ".1", y.T.reshape(512, c16, c16)).reshape(512, -1).T)

    def kernel(a, b):
        return torch.exp(((a @ b.T) / (a.norm(dim=1)[:, None] * b.norm(dim=1)[None] + 1e-6) - 1) / 0.2)

    gy, gx = torch.meshgrid(_centres(c16), _centres(c16), indexing="ij")
    at = torch.stack([gx, gy], -1).reshape(-1, 2)
    p = "decoder.gps.16.pos_conv"
    basis = torch.cos(8 * math.pi * (at @ wm[p + ".weight"].double().reshape(512, 2).T + wm[p + ".bias"].double()))
    K = kernel(g[1], g[1]).cpu() + 0.1 * torch.eye(c16 * c16, dtype=torch.float64)
    mu = kernel(g[0], g[1]) @ torch.cholesky_solve(basis.cpu(), torch.linalg.cholesky(K)).cuda()
    x = torch.cat([mu, g[0]], 1)
    for i in range(5):
        x = _vit_block(wm, f"decoder.embedding_decoder.blocks.{i}", x, 8, 1e-5)
    p = "decoder.embedding_decoder.to_out"
    return {"g_y": torch.stack(g), "t_x": x,
            "t_out": x @ wm[p + ".weight"].double().T + wm[p + ".bias"].double()}


def _disk(w, img):
    """DISK's 128 descriptor channels and its heatmap."""
    def layer(i, x):
        p = f"unet.path_down.{i}.1" if i < 5 else f"unet.path_up.{i - 5}.conv"
        if i:
            v = x.flatten(1)
            x = (x - v.mean(1)[:, None, None]) / torch.sqrt(v.var(1, unbiased=False) + 1e-5)[:, None, None]
            x = torch.where(x >= 0, x, w[p + ".1.weight"].double()[:, None, None] * x)
        return _conv(x, w[p + ".3.weight"], w[p + ".3.bias"])

    down = [layer(0, img)]
    for i in range(1, 5):
        down.append(layer(i, F.avg_pool2d(down[-1], 2)))
    y = down[4]
    for j in range(4):
        y = F.interpolate(y[None], scale_factor=2, mode="bilinear", align_corners=False)[0]
        y = layer(5 + j, torch.cat([y, down[3 - j]]))
    return y
