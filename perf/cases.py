"""Performance cases of the GroupNorm+SiLU path, the layers around it and the
SOAR model, through the Python binding a user's program calls.

kind "gn"     GroupNorm+SiLU forward and backward (soar_gn.gn_silu_forward /
              gn_silu_backward), with the residual add where a block has one
kind "pw"     a CBA block with a pointwise conv: pw_conv_gn_silu_forward and
              pw_cba_backward
kind "dw"     a CBA block with a depthwise conv (Down.dw, LKR.dw, the Ctx
              branches): dw_conv_gn_silu_forward and dw_cba_backward
kind "predict" / "grad"   whole calls of the model (soar_model.SOAR.predict,
              SOAR.forward_backward with the gradients read back)

All tensors are fp32, the one data type of the framework.  Activations are
written into buffers that the program keeps; the parameter gradients are
fresh zeros that each backward adds into.  Work is the bytes a pass cannot
do without (its inputs read once by each direction, its outputs written
once) and its multiply-adds.
"""
import math
import os
import sys
import tempfile
import zlib

import numpy as np
import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "soar.cpp_amd"))

import soar_gn as gn  # noqa: E402
import soar_model  # noqa: E402

EPS = 1e-5

# width and depth per variant: c0..c17, n2, n4, n6, n8, n11, n13
ARCH = {
    "nano": (16, 32, 32, 64, 64, 128, 128, 256, 256, 256, 128, 128, 64, 64, 32, 32, 16, 16,
             1, 1, 2, 1, 1, 1),
    "small": (24, 48, 48, 96, 96, 192, 192, 384, 384, 384, 192, 192, 96, 96, 48, 48, 24, 24,
              1, 2, 3, 2, 1, 1),
}


def _groups(c):
    """The CBA blocks' group count: the largest divisor of c up to 8."""
    return max(g for g in range(1, min(8, c) + 1) if c % g == 0)


# ---- the cases ---------------------------------------------------------------

def _gn(name, n, c, h, w, g, residual=False):
    return {"name": name, "kind": "gn", "N": n, "C": c, "H": h, "W": w, "G": g,
            "residual": residual}


def _pw(name, n, ci, co, h, w, g, silu=True):
    return {"name": name, "kind": "pw", "N": n, "Ci": ci, "Co": co, "H": h, "W": w, "G": g,
            "silu": silu}


def _dw(name, n, c, h, w, k, stride, dil, g):
    return {"name": name, "kind": "dw", "N": n, "C": c, "H": h, "W": w, "K": k,
            "stride": stride, "dil": dil, "G": g}


def listed():
    return [
        # the deepest Nano layers at a 512^2 image: a call is launches and
        # host work, hardly any data
        _gn("gn_small", 1, 128, 32, 32, 8),
        # a mid-depth layer of a 512^2 - 1024^2 image with the skip added
        _gn("gn_mid_residual", 2, 32, 256, 256, 8, residual=True),
        # a batch whose planes are no multiple of anything
        _gn("gn_odd", 3, 48, 125, 187, 8),
        # the benchmark's headline tensor
        _gn("gn_large", 1, 64, 2048, 2048, 16),
        # LKR.pw1 of the Nano model's stride-16 stage at a 512^2 image
        _pw("pw_small", 1, 128, 256, 32, 32, 8),
        # LKR.pw1 of the XLarge model's stride-8 stage at a 1024^2 image
        _pw("pw_mid", 1, 192, 384, 128, 128, 8),
        # the benchmark's pointwise CBA
        _pw("pw_large", 1, 64, 64, 2048, 2048, 16),
        # LKR.dw of the Nano model's stride-16 stage at a 1024^2 image
        _dw("dw_k7_mid", 1, 128, 64, 64, 7, 1, 1, 8),
        # Down.dw on a plane of odd sides
        _dw("dw_k3s2_odd", 1, 48, 333, 255, 3, 2, 1, 8),
        # the benchmark's depthwise k3 CBA
        _dw("dw_k3_large", 1, 64, 2048, 2048, 3, 1, 1, 16),
        # one image through the deployed model: probabilities and mask
        {"name": "predict_nano", "kind": "predict", "variant": "nano", "H": 1024, "W": 1024},
        # forward, loss and backward of the model on one image
        {"name": "grad_nano", "kind": "grad", "variant": "nano", "H": 1024, "W": 1024},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gn", "gn", "gn", "pw", "pw", "pw", "dw", "dw", "dw", "predict", "grad"])
    if kind in ("predict", "grad"):
        return {"kind": kind, "variant": rng.choice(["nano", "nano", "small"]),
                "H": _spread(rng, 64, 1024), "W": _spread(rng, 64, 1024)}
    while True:
        h, w = _spread(rng, 16, 2048), _spread(rng, 16, 2048)
        if rng.random() < 0.6:  # model planes: sides that are multiples of 8
            h, w = max(16, h // 8 * 8), max(16, w // 8 * 8)
        n = rng.choice([1, 1, 1, 2, 3, 4])
        c = 8 * _spread(rng, 1, 48)
        if kind == "gn":
            g = rng.choice([x for x in (4, 8, 16, 32) if c % x == 0])
            if n * c * h * w <= 1 << 28:
                case = _gn("", n, c, h, w, g, rng.random() < 0.3)
                break
        elif kind == "pw":
            ci, co = c, 8 * _spread(rng, 1, 48)
            if n * max(ci, co) * h * w <= 1 << 26 and n * ci * co * h * w <= 1 << 33:
                case = _pw("", n, ci, co, h, w, _groups(co), rng.random() < 0.6)
                break
        else:
            k, s, d = rng.choice([(3, 1, 1), (3, 2, 1), (5, 1, 1), (7, 1, 1), (7, 1, 1),
                                  (3, 1, 3), (3, 1, 5)])
            if n * c * h * w * k * k <= 1 << 31:
                case = _dw("", n, c, h, w, k, s, d, _groups(c))
                break
    del case["name"]
    return case


# ---- inputs ------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _normal(seed, salt, shape, mean=0.0, std=1.0):
    return torch.empty(shape, device="cuda").normal_(mean, std, generator=_gen(seed, salt))


def _uniform(seed, salt, shape, lo, hi):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=_gen(seed, salt))


def _out_hw(case):
    k, s, d = case["K"], case["stride"], case["dil"]
    pad = d * (k - 1) // 2
    return pad, gn.conv_out_size(case["H"], k, pad, s, d), gn.conv_out_size(case["W"], k, pad, s, d)


def _layer_inputs(case, seed):
    """x, dy and the parameters of a layer case."""
    kind, n, h, w = case["kind"], case["N"], case["H"], case["W"]
    t = {}
    if kind == "pw":
        ci, c = case["Ci"], case["Co"]
        t["x"] = _normal(seed, 1, (n, ci, h, w))
        t["w"] = _uniform(seed, 2, (c, ci), -ci ** -0.5, ci ** -0.5)
        oh, ow = h, w
    else:
        c = case["C"]
        t["x"] = _normal(seed, 1, (n, c, h, w), 0.1 if kind == "gn" else 0.0)
        oh, ow = h, w
        if kind == "dw":
            k = case["K"]
            t["w"] = _uniform(seed, 2, (c, k, k), -1.0 / k, 1.0 / k)
            _, oh, ow = _out_hw(case)
    t["gamma"] = _uniform(seed, 3, (c,), 0.5, 1.5)
    t["beta"] = _normal(seed, 4, (c,), 0.0, 0.1)
    t["dy"] = _normal(seed, 5, (n, c, oh, ow), 0.0, 1e-2)
    return t


def _weight(seed, name, shape):
    """A trained-like value of one model parameter, from its name alone."""
    r = np.random.default_rng([int(seed) & 0x7FFFFFFF, zlib.crc32(name.encode())])
    if name.endswith("norm.weight"):
        v = r.uniform(0.5, 1.5, size=shape)
    elif name.endswith("bias"):
        v = r.normal(0.0, 0.1, size=shape)
    else:
        b = 1.0 / math.sqrt(int(np.prod(shape[1:])))
        v = r.uniform(-b, b, size=shape)
    if name.startswith("l17_head.pred"):
        # the head's four sub-pixel outputs of a trained model nearly agree, so
        # its masks are regions and not noise
        v = 4.0 * v[:1] + 0.02 * v
    return v.astype(np.float32)


def _image(case, seed):
    r = np.random.default_rng([int(seed) & 0x7FFFFFFF, 77])
    h, w = case["H"], case["W"]
    yy, xx = np.mgrid[0:h, 0:w].astype(np.float32)
    cy, cx = r.uniform(0.3, 0.7, 2) * (h, w)
    d = ((yy - cy) / (0.25 * h)) ** 2 + ((xx - cx) / (0.2 * w)) ** 2
    # a bright blob on a dark ground, with the noise of a sensor
    image = 0.2 + 0.6 / (1.0 + np.exp(np.clip(20.0 * (d - 1.0), -30.0, 30.0)))
    image = image + 0.01 * r.standard_normal((h, w), dtype=np.float32)
    return image[None].astype(np.float32), (d < 1.0)[None].astype(np.float32)


def _load(model, seed):
    """Loads the seed's weights into the model from a .soar file."""
    out = [np.array([0x534F4152, 1, soar_model.VARIANT_MAP[model.variant]], "<u4").tobytes()]
    named = model.tensors()
    out.append(np.array([len(named)], "<u4").tobytes())
    for name, shape in named:
        v = _weight(seed, name, shape)
        dims = list(shape) + [1] * (4 - len(shape))
        out += [name.encode().ljust(128, b"\0"), np.array([len(shape)] + dims, "<u4").tobytes(),
                np.array([v.nbytes], "<u8").tobytes(), v.tobytes()]
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "weights.soar")
        with open(path, "wb") as f:
            f.write(b"".join(out))
        model.load_weights(path)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("predict", "grad"):
        model = soar_model.SOAR(1, 1, case["variant"], seed=int(seed))
        _load(model, seed)
        image, mask = _image(case, seed)
        st = {"case": case, "model": model, "image": image, "mask": mask}
        if kind == "grad":
            st["params"] = model.tensors()
        return st
    st = _layer_inputs(case, seed)
    st["case"] = case
    n, h, w, g = case["N"], case["H"], case["W"], case["G"]
    new = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    raw = lambda b: torch.empty(max(int(b), 1), dtype=torch.uint8, device="cuda")  # noqa: E731
    st["y"] = torch.empty_like(st["dy"])
    st["dx"] = torch.empty_like(st["x"])
    st["stats"] = (new(n * g), new(n * g), new(n * g))
    if kind == "gn":
        st["ws"] = gn.workspace(n, case["C"], h * w, g)
    elif kind == "pw":
        ci, co = case["Ci"], case["Co"]
        st["z"] = torch.empty_like(st["dy"])
        st["ws"] = raw(gn.pw_conv_gn_workspace_bytes(n, co, h * w, g))
        st["ws_bwd"] = raw(gn.pw_cba_backward_workspace_bytes(n, ci, co, h * w, g))
    else:
        pad, oh, ow = _out_hw(case)
        geo = (n, case["C"], h, w, oh, ow, case["K"], pad, case["stride"], case["dil"], g)
        st["pad"] = pad
        st["z"] = torch.empty_like(st["dy"])
        st["ws"] = raw(gn.dw_conv_gn_workspace_bytes(*geo))
        st["ws_bwd"] = raw(gn.dw_cba_backward_workspace_bytes(*geo))
    return st


# ---- one pass ----------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "predict":
        probs, mask, _ = st["model"].predict(st["image"])
        return {"probs": probs, "mask": mask}
    if kind == "grad":
        model = st["model"]
        metrics = model.forward_backward(st["image"], st["mask"])
        grads = [model.read(i, grad=True, shape=s).ravel() for i, (_, s) in enumerate(st["params"])]
        return {"loss": metrics["loss"], "grads": np.concatenate(grads)}
    g = case["G"]
    mean, rstd, lo = st["stats"]
    if kind == "gn":
        res = case["residual"]
        y, stats = gn.gn_silu_forward(st["x"], st["gamma"], st["beta"], g, eps=EPS, residual=res,
                                      y=st["y"], mean=mean, rstd=rstd, mean_lo=lo, ws=st["ws"])
        dx, dgamma, dbeta = gn.gn_silu_backward(st["dy"], st["x"], st["gamma"], st["beta"], stats,
                                                g, residual=res, dx=st["dx"], ws=st["ws"])
        return {"y": y, "dx": dx, "dgamma": dgamma, "dbeta": dbeta}
    if kind == "pw":
        z, y, stats = gn.pw_conv_gn_silu_forward(
            st["x"], st["w"], None, st["gamma"], st["beta"], g, eps=EPS, silu=case["silu"],
            z=st["z"], y=st["y"], mean=mean, rstd=rstd, mean_lo=lo, ws=st["ws"])
        dx, dw, dgamma, dbeta = gn.pw_cba_backward(
            st["dy"], z, st["x"], st["w"], st["gamma"], st["beta"], stats, g, silu=case["silu"],
            dx=st["dx"], ws=st["ws_bwd"])
    else:
        k, s, d = case["K"], case["stride"], case["dil"]
        z, y, stats = gn.dw_conv_gn_silu_forward(
            st["x"], st["w"], None, st["gamma"], st["beta"], g, st["pad"], s, d, eps=EPS,
            z=st["z"], y=st["y"], mean=mean, rstd=rstd, mean_lo=lo, ws=st["ws"])
        dx, dw, dgamma, dbeta = gn.dw_cba_backward(
            st["dy"], z, st["x"], st["w"], st["gamma"], st["beta"], stats, g, st["pad"], s, d,
            dx=st["dx"], ws=st["ws_bwd"])
    return {"z": z, "y": y, "dx": dx, "dw": dw, "dgamma": dgamma, "dbeta": dbeta}


# ---- what a pass cannot do without ---------------------------------------------

def _model_work(case):
    """(multiply-adds, activation floats written, parameters) of a forward."""
    tally = {"macs": 0, "floats": 0, "params": 0}

    class Count(_Model):
        def conv(self, name, x, shape, stride=1, dil=1, bias=False):
            n, _, h, w = x.shape
            oh, ow = -(-h // stride), -(-w // stride)
            tally["macs"] += shape[0] * shape[1] * shape[2] * shape[3] * oh * ow
            tally["params"] += int(np.prod(shape)) + (shape[0] if bias else 0)
            tally["floats"] += shape[0] * oh * ow
            return torch.empty((n, shape[0], oh, ow), device="meta")

        def norm(self, name, x, act):
            tally["params"] += 2 * x.shape[1]
            tally["floats"] += x.numel()
            return x

        def param(self, name, shape):
            return torch.empty(shape, device="meta")

    Count(case["variant"], None).forward(torch.empty((1, 1, case["H"], case["W"]), device="meta"))
    return tally


def work(case):
    kind = case["kind"]
    if kind in ("predict", "grad"):
        t = _model_work(case)
        hw = case["H"] * case["W"]
        if kind == "predict":  # each layer's output written and read once
            return {"bytes": 8 * t["floats"] + 4 * t["params"] + 9 * hw, "flops": 2 * t["macs"]}
        # the backward reads each once more and moves as many gradient values
        return {"bytes": 20 * t["floats"] + 8 * t["params"] + 8 * hw, "flops": 6 * t["macs"]}
    p = case["N"] * case["H"] * case["W"]
    if kind == "gn":  # x in, y out; x and dy in, dx out
        return {"bytes": 4 * 5 * case["C"] * p, "flops": 30 * case["C"] * p}
    if kind == "pw":  # x in, z and y out; dy, z and x in, dx out
        ci, co = case["Ci"], case["Co"]
        return {"bytes": 4 * (3 * ci + 4 * co) * p + 8 * ci * co, "flops": 6 * ci * co * p}
    _, oh, ow = _out_hw(case)
    po, c = case["N"] * oh * ow, case["C"]
    return {"bytes": 4 * c * (3 * p + 4 * po), "flops": 6 * case["K"] ** 2 * c * po}


def tolerance(case):
    """fp32 sums, four times the error against float64 that the worst output
    shows.  Of a layer that is the weight gradient, up to 4 million cancelling
    terms (1.2e-6 at 2048^2); in the model a change of rounding travels
    through all layers (probabilities 1.1e-6, gradients 1.8e-6), and a pixel at the threshold may
    change sides."""
    kind = case["kind"]
    if kind == "predict":
        return {"rel": 5e-6, "max": 3e-4, "differ": 2e-5}
    if kind == "grad":
        return {"rel": 8e-6, "max": 2e-3}
    return {"rel": 5e-6, "max": 3e-4}


# ---- the same in 64 bits ---------------------------------------------------------

def _conv64(x, w, stride=1, dil=1):
    """Grouped-by-one ([C,1,K,K]) or dense convolution, "same" padding."""
    k = w.shape[-1]
    if k == 1 and w.shape[1] == x.shape[1]:
        return torch.stack([(w[:, :, 0, 0] @ s.reshape(s.shape[0], -1)).reshape(
            (-1,) + s.shape[1:]) for s in x])
    pad = dil * (k - 1) // 2
    h, wd = x.shape[2:]
    oh = (h + 2 * pad - dil * (k - 1) - 1) // stride + 1
    ow = (wd + 2 * pad - dil * (k - 1) - 1) // stride + 1
    xp = F.pad(x, (pad, pad, pad, pad))
    out = None
    for ky in range(k):
        for kx in range(k):
            v = xp[:, :, ky * dil:ky * dil + (oh - 1) * stride + 1:stride,
                   kx * dil:kx * dil + (ow - 1) * stride + 1:stride]
            # depthwise, or a dense convolution of one input channel
            v = v * w[:, 0, ky, kx][None, :, None, None]
            out = v if out is None else out + v
    return out


def _norm64(x, groups, gamma, beta):
    n, c = x.shape[:2]
    v = x.reshape(n, groups, -1)
    mean = v.mean(dim=2, keepdim=True)
    var = (v - mean).square().mean(dim=2, keepdim=True)
    v = ((v - mean) * (var + EPS).rsqrt()).reshape(x.shape)
    return v * gamma[None, :, None, None] + beta[None, :, None, None]


def _silu64(x):
    return x * torch.sigmoid(x)


class _Model:
    """The SOAR forward over parameters by name, [1,C,H,W] in float64."""

    def __init__(self, variant, param):
        self.a = ARCH[variant]
        self.get = param

    def param(self, name, shape):
        return self.get(name, shape)

    def conv(self, name, x, shape, stride=1, dil=1, bias=False):
        z = _conv64(x, self.param(name + ".weight", shape), stride, dil)
        return z + self.param(name + ".bias", shape[:1])[None, :, None, None] if bias else z

    def norm(self, name, x, act):
        c = x.shape[1:2]
        y = _norm64(x, _groups(c[0]), self.param(name + ".weight", c), self.param(name + ".bias", c))
        return _silu64(y) if act else y

    def cba(self, name, x, co, k=1, stride=1, dil=1, dw=False, act=True):
        shape = (co, 1 if dw else x.shape[1], k, k)
        return self.norm(name + ".norm", self.conv(name + ".conv", x, shape, stride, dil), act)

    def down(self, name, x, co):
        y = self.cba(name + ".dw", x, x.shape[1], 3, 2, dw=True, act=False)
        return self.cba(name + ".pw", y, co)

    def stack(self, base, n, x, k, indexed=False):
        for i in range(n):
            name = base if n == 1 and not indexed else "%s_%d" % (base, i)
            c = x.shape[1]
            y = self.cba(name + ".dw", x, c, k, dw=True, act=False)
            y = self.cba(name + ".pw1", y, max(2 * c, 8))
            x = x + self.cba(name + ".pw2", y, c, act=False)
        return x

    def resize(self, x, like):
        if x.shape[2:] == like.shape[2:]:
            return x
        if x.device.type == "meta":
            return torch.empty(x.shape[:2] + like.shape[2:], device="meta")
        return F.interpolate(x, size=like.shape[2:], mode="bilinear", align_corners=False)

    def fuse(self, name, low, skip, c):
        a = self.cba(name + ".skip", skip, c, act=False)
        b = self.resize(self.cba(name + ".low", low, c, act=False), a)
        g = self.cba(name + ".gate_dw", a + b, c, 3, dw=True, act=False)
        g = torch.sigmoid(self.conv(name + ".gate_conv", g, (c, c, 1, 1), bias=True))
        y = self.cba(name + ".out_dw", g * a + (1 - g) * b, c, 3, dw=True, act=False)
        return self.cba(name + ".out_pw", y, c)

    def ctx(self, name, x, co):
        h = co // 2
        y = self.cba(name + ".cv1", x, h)
        cat = [y] + [self.cba("%s.branch_%d" % (name, i), y, h, 3, 1, d, dw=True, act=False)
                     for i, d in enumerate((1, 3, 5))]
        out = self.cba(name + ".cv2", torch.cat(cat, dim=1), co)
        gate = self.conv(name + ".gate_conv", x.mean(dim=(2, 3), keepdim=True),
                         (co, x.shape[1], 1, 1), bias=True)
        out = out * torch.sigmoid(gate)
        return x + out if x.shape[1] == co else out

    def forward(self, x):
        a = self.a
        h, w = x.shape[2:]
        ph, pw = -h % 32, -w % 32
        if x.device.type == "meta":
            x = torch.empty((1, 1, h + ph, w + pw), device="meta")
        elif ph or pw:
            mode = "reflect" if ph < h and pw < w else "replicate"
            x = F.pad(x, (0, pw, 0, ph), mode=mode)
        n2, n4, n6, n8, n11, n13 = a[18:]
        s2 = self.cba("l0_cba", x, a[0], 3, 2)
        p2 = self.stack("l2_lkr", n2, self.down("l1_down", s2, a[1]), 5)
        p3 = self.stack("l4_lkr", n4, self.down("l3_down", p2, a[3]), 7)
        p4 = self.stack("l6_lkr", n6, self.down("l5_down", p3, a[5]), 7, True)
        p5 = self.stack("l8_lkr", n8, self.down("l7_down", p4, a[7]), 7)
        d16 = self.stack("l11_lkr", n11, self.fuse("l10_fuse", self.ctx("l9_ctx", p5, a[9]),
                                                   p4, a[10]), 7)
        d8 = self.stack("l13_lkr", n13, self.fuse("l12_fuse", d16, p3, a[12]), 7)
        d4 = self.fuse("l14_fuse", d8, p2, a[14])
        p = max(a[15] // 2, 8)
        ys = [self.resize(self.cba("l15_agg.proj_%d" % i, t, p), d4)
              for i, t in enumerate((d4, d8, d16))]
        d2 = self.fuse("l16_fuse", self.cba("l15_agg.fuse", torch.cat(ys, dim=1), a[15]), s2, a[16])
        y = self.cba("l17_head.refine_dw", d2, a[16], 3, dw=True, act=False)
        y = self.cba("l17_head.refine_pw", y, a[17])
        y = self.conv("l17_head.pred", y, (4, a[17], 1, 1), bias=True)
        if y.device.type == "meta":
            return y
        return F.pixel_shuffle(y, 2)[:, :, :h, :w]


def _model_exact(case, seed):
    params = {}

    def param(name, shape):
        v = torch.tensor(_weight(seed, name, tuple(shape)), dtype=torch.float64, device="cuda")
        params[name] = v.requires_grad_(case["kind"] == "grad")
        return params[name]

    image, mask = _image(case, seed)
    image = torch.tensor(image, dtype=torch.float64, device="cuda")[None]
    z = _Model(case["variant"], param).forward(image)
    if case["kind"] == "predict":
        return {"probs": torch.sigmoid(z)[0], "mask": None}
    # 0.5 * BCE (positives weighted 3) + 0.5 * soft Dice
    t = torch.tensor(mask, dtype=torch.float64, device="cuda")[None]
    bce = ((1 - t) * z + (1 + 2 * t) * F.softplus(-z)).mean()
    p = torch.sigmoid(z)
    dice = 1 - (2 * (p * t).sum() + 1) / (p.sum() + t.sum() + 1 + 1e-7)
    loss = 0.5 * bce + 0.5 * dice
    loss.backward()
    # the library's order: parameters of a module by name, then its modules by name
    tree = {}
    for name in params:
        node = tree
        *path, leaf = name.split(".")
        for part in path:
            node = node.setdefault(part, {})
        node[leaf] = params[name]

    def flat(node):
        own = sorted(k for k, v in node.items() if not isinstance(v, dict))
        subs = sorted(k for k, v in node.items() if isinstance(v, dict))
        return [node[k].grad.reshape(-1) for k in own] + [v for k in subs for v in flat(node[k])]

    return {"loss": loss.detach(), "grads": torch.cat(flat(tree))}


def exact(case, seed):
    if case["kind"] in ("predict", "grad"):
        return _model_exact(case, seed)
    t = {k: v.double() for k, v in _layer_inputs(case, seed).items()}
    leaves = [k for k in ("x", "w", "gamma", "beta") if k in t]
    for k in leaves:
        t[k].requires_grad_(True)
    out = {}
    z = t["x"]
    if case["kind"] == "pw":
        z = _conv64(z, t["w"][:, :, None, None])
    elif case["kind"] == "dw":
        z = _conv64(z, t["w"][:, None], case["stride"], case["dil"])
    y = _norm64(z, case["G"], t["gamma"], t["beta"])
    if case.get("silu", True):
        y = _silu64(y)
    if case.get("residual"):
        y = y + t["x"]
    grads = dict(zip(leaves, torch.autograd.grad(y, [t[k] for k in leaves], t["dy"])))
    if case["kind"] != "gn":
        out["z"] = z.detach()
        out["dw"] = grads["w"]
    out.update(y=y.detach(), dx=grads["x"], dgamma=grads["gamma"], dbeta=grads["beta"])
    return out
