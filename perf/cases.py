"""The work that programs have this library do, as cases to be timed and compared.

Every case goes through the C interface (openclipp_amd.ocip) as a C program uses it: images are
created and sent once, an operation is queued on the context's stream, and its map stays on the
GPU for whatever reads it next.  A case is a dict of plain values; its "path" says which entry
points it stands for:

  match      ocip<Op>(Source, Template, Dest): the reference's interface, plain arithmetic of the
             element type; "locate": followed by ocipMaxIndx / ocipMinIndx on the map
  mfma       ocipCrossCorr[_Norm]Ex: a precision chosen by the caller
  batch      ocip{CrossCorr,SqrDistance}_NormBatch: many templates, one image
  gradients  ocipProximityBackwardBatch: both operations' gradients, many images
  fft        ocip{CrossCorr,SqrDistance}FFT_Norm: big templates
  integral   ocip[Sqr]Integral
"""
import ctypes
import math
import random

import numpy as np
import torch

from openclipp_amd import ocip

_context = None
_PRECISION = {"bf16": ocip.PREC_BF16, "f16": ocip.PREC_F16, "bf16x3": ocip.PREC_BF16X3}


def listed():
    return [
        # a crop of a camera frame searched for a small mark, the answer awaited: all latency
        dict(name="locate_f32_160x120_t8", path="match", op="CrossCorr_Norm", type="F32",
             channels=1, w=160, h=120, tw=8, th=8, locate=True),
        # the reference Bench's own size and template, its plain F32 path
        dict(name="ssd_norm_f32_1024_t16", path="match", op="SqrDistance_Norm", type="F32",
             channels=1, w=1024, h=1024, tw=16, th=16, locate=False),
        # the 4096^2 / 64x64 workload through the reference's entry point, F32 arithmetic
        dict(name="ncc_f32_4096_t64", path="match", op="CrossCorr_Norm", type="F32",
             channels=1, w=4096, h=4096, tw=64, th=64, locate=False),
        # 8-bit frames, exact integer sums: the 4096^2 / 32x32 workload
        dict(name="ssd_u8_4096_t32", path="match", op="SqrDistance", type="U8", channels=1,
             w=4096, h=4096, tw=32, th=32, locate=False),
        # an 8-bit video frame with a ragged template, absolute differences
        dict(name="sad_u8_1919x1079_t31x23", path="match", op="AbsDistance", type="U8",
             channels=1, w=1919, h=1079, tw=31, th=23, locate=False),
        # a 16-bit sensor
        dict(name="ncc_u16_2048x1536_t31", path="match", op="CrossCorr_Norm", type="U16",
             channels=1, w=2048, h=1536, tw=31, th=31, locate=False),
        # a colour frame (three channels on the host, four on the device)
        dict(name="ncc_color_u8_1280x960_t24", path="match", op="CrossCorr_Norm", type="U8",
             channels=3, w=1280, h=960, tw=24, th=24, locate=False),
        # the headline: 4096^2, 64x64, BF16 matrix products
        dict(name="ncc_bf16_4096_t64", path="mfma", op="CrossCorr_Norm", precision="bf16",
             w=4096, h=4096, tw=64, th=64),
        # a library of templates of all sizes against one image
        dict(name="batch_bf16_2048_48", path="batch", op="CrossCorr_Norm", precision="bf16",
             w=2048, h=2048, count=48, lo=8, hi=96, mix=4),
        # training a template on a batch of images
        dict(name="gradients_16x1024_t31", path="gradients", count=16, w=1024, h=1024, tw=31,
             th=31),
        # a template too big for the direct path
        dict(name="ncc_fft_4096_t256", path="fft", op="CrossCorr_Norm", w=4096, h=4096, tw=256,
             th=256),
        # window sums of 8-bit images
        dict(name="sqr_integral_u8_4096", path="integral", sqr=True, type="U8", dest="F64",
             w=4096, h=4096),
    ]


# ------------------------------------------------------------------------------ drawn cases
_MOST_TAPS = 4096 * 4096 * 64 * 64       # output pixels times template pixels of the largest case


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _image(rng, lo, hi):
    """A size within lo..hi a side, at most 2:1 either way; odd and ragged as often as not."""
    w = _log(rng, lo, hi)
    h = _log(rng, max(lo, w // 2), min(hi, 2 * w))
    if rng.random() < 0.4:
        w, h = (max(lo, v // 32 * 32) for v in (w, h))
    return w, h


def draw(rng):
    path = rng.choice(["match"] * 6 + ["mfma"] * 2 + ["batch", "gradients", "fft", "integral"])
    if path == "match":
        kind, channels = rng.choice([("F32", 1), ("F32", 1), ("U8", 1), ("U8", 1), ("U8", 3),
                                     ("U16", 1), ("S16", 1)])
        w, h = _image(rng, 96, 4096)
        tw, th = _log(rng, 5, 64), _log(rng, 5, 64)
        # the paths of the 16-bit and colour images cost more per tap than the largest case's
        most = _MOST_TAPS // (1 if kind == "F32" else 8 if channels == 1 else 32)
        while w * h * tw * th > most:
            w, h = max(96, w // 2 + 1), max(96, h // 2 + 1)
        return dict(path=path, op=rng.choice(ocip.PROXIMITY_OPS), type=kind, channels=channels,
                    w=w, h=h, tw=tw, th=th, locate=channels == 1 and rng.random() < 0.3)
    if path == "mfma":
        w, h = _image(rng, 256, 4096)
        return dict(path=path, op=rng.choice(["CrossCorr_Norm", "CrossCorr_Norm", "CrossCorr"]),
                    precision=rng.choice(["bf16", "f16", "bf16x3"]), w=w, h=h,
                    tw=_log(rng, 8, 96), th=_log(rng, 8, 96))
    if path == "batch":
        w, h = _image(rng, 256, 2048)
        return dict(path=path, op=rng.choice(["CrossCorr_Norm", "SqrDistance_Norm"]),
                    precision=rng.choice(["bf16", "bf16", "f16", "bf16x3"]), w=w, h=h,
                    count=rng.randint(2, 48) if w * h < 1 << 20 else rng.randint(2, 16), lo=8,
                    hi=rng.choice([24, 48, 96]), mix=rng.randrange(1 << 20))
    if path == "gradients":
        w, h = _image(rng, 256, 1024)
        t = _log(rng, 7, 31)
        return dict(path=path, count=rng.randint(1, 16), w=w, h=h, tw=t, th=max(5, t - rng.randint(0, 4)))
    if path == "fft":
        w, h = _image(rng, 512, 4096)
        return dict(path=path, op=rng.choice(["CrossCorr_Norm", "SqrDistance_Norm"]), w=w, h=h,
                    tw=_log(rng, 64, 256), th=_log(rng, 64, 256))
    w, h = _image(rng, 256, 4096)
    return dict(path=path, sqr=rng.random() < 0.5, type=rng.choice(["U8", "U16", "F32"]),
                dest=rng.choice(["F32", "F64"]), w=w, h=h)


# ------------------------------------------------------------------------------ inputs
_TYPE = {"U8": np.uint8, "U16": np.uint16, "S16": np.int16, "F32": np.float32,
         "F64": np.float64}
_RANGE = {"U8": (0, 255), "U16": (0, 65535), "S16": (-32768, 32767)}


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _field(g, h, w):
    """Smooth noise over [0, 1], as a blurred scene is: three box blurs of 9 pixels."""
    f = torch.rand((h + 24, w + 24), generator=g, device=g.device)
    for _ in range(3):
        for d in (0, 1):
            n = f.shape[d] - 8
            f = sum(f.narrow(d, k, n) for k in range(9)) / 9
    lo, hi = f.min(), f.max()
    return (f - lo) / (hi - lo)


def _source(g, kind, h, w, channels=1):
    if kind in _RANGE:
        lo, hi = _RANGE[kind]
        v = torch.stack([_field(g, h, w) for _ in range(channels)], dim=-1)
        v = torch.round(lo + v * (hi - lo))
        v = v.squeeze(-1) if channels == 1 else v
        return v.cpu().numpy().astype(_TYPE[kind])
    v = 0.5 + 0.2 * torch.randn((h, w), generator=g, device=g.device)
    return v.clamp_(0, 1).cpu().numpy()


def _crop(rng, src, tw, th):
    """A crop of the image with a little noise: what a template is."""
    y, x = rng.randint(0, src.shape[0] - th), rng.randint(0, src.shape[1] - tw)
    t = src[y:y + th, x:x + tw].astype(np.float64)
    noise = np.random.default_rng(rng.randrange(1 << 30)).standard_normal(t.shape)
    if src.dtype == np.float32:
        return (t * 1.1 + 0.01 * noise).astype(np.float32)
    top = np.iinfo(src.dtype)
    t = t + np.rint(noise * 2 * (top.max - top.min) / 255)
    return np.clip(t, top.min, top.max).astype(src.dtype)


def _inputs(case, seed):
    """The host arrays of a case, by name."""
    g, rng = _generator(seed), random.Random(seed)
    h, w = case["h"], case["w"]
    path = case["path"]
    if path == "gradients":
        n = case["count"]
        return {"src": torch.rand((n, h, w), generator=g, device=g.device).cpu().numpy(),
                "tpl": torch.randn((case["th"], case["tw"]), generator=g, device=g.device).cpu().numpy(),
                "g_ncc": torch.randn((n, h, w), generator=g, device=g.device).cpu().numpy(),
                "g_ssd": torch.randn((n, h, w), generator=g, device=g.device).cpu().numpy()}
    src = _source(g, case.get("type", "F32"), h, w, case.get("channels", 1))
    if path == "integral":
        return {"src": src}
    if path == "batch":
        mix = random.Random(case["mix"])
        lo, hi = case["lo"], case["hi"]
        return {"src": src, "tpl": [_crop(rng, src, mix.randint(lo, hi), mix.randint(lo, hi))
                                    for _ in range(case["count"])]}
    return {"src": src, "tpl": _crop(rng, src, case["tw"], case["th"])}


# ------------------------------------------------------------------------------ a user's program
class Map(torch.Tensor):
    """The map of an ocipImage as a tensor: it stays on the GPU, where a program's next operation
    finds it, and is read back (ocipReadImage) when its values are looked at."""

    @staticmethod
    def of(image):
        m = torch.from_numpy(image.arr).as_subclass(Map)
        m.image = image
        return m

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        with torch._C.DisableTorchFunctionSubclass():
            plain = []
            for a in args:
                if isinstance(a, cls):
                    a.image.read()
                    a = a.as_subclass(torch.Tensor)
                plain.append(a)
            return func(*plain, **(kwargs or {}))


class Program:
    """An ocipProgram, released with its owner."""

    def __init__(self, prepare, *images):
        self.handle = ctypes.c_void_p()
        ocip.check(prepare(ctypes.byref(self.handle), *(i.handle for i in images)), "prepare")

    def __del__(self):
        ocip.lib.ocipReleaseProgram(self.handle)


def _dest(h, w, kind="F32", channels=1):
    return ocip.Image(shape=(h, w), dtype=_TYPE[kind], channels=channels)


def prepare(case, seed):
    global _context
    if _context is None:
        _context = ocip.initialize()
    lib, path = ocip.lib, case["path"]
    h, w = case["h"], case["w"]
    a = _inputs(case, seed)
    if path == "gradients":
        S, G1, G2 = ([ocip.Image(x).send() for x in a[k]] for k in ("src", "g_ncc", "g_ssd"))
        T = ocip.Image(a["tpl"]).send()
        dS = [_dest(h, w) for _ in S]
        dT = _dest(case["th"], case["tw"])
        args = (ocip.handles(S), T.handle, ocip.handles(G1), ocip.handles(G2), ocip.handles(dS),
                dT.handle, len(S))
        return {"call": lib.ocipProximityBackwardBatch, "args": args, "keep": (S, G1, G2, T),
                "out": {"source": [Map.of(d) for d in dS], "template": Map.of(dT)}}
    S = ocip.Image(a["src"]).send()
    if path == "integral":
        D = _dest(h, w, case["dest"])
        P = Program(lib.ocipPrepareIntegral, S)
        return {"call": lib.ocipSqrIntegral if case["sqr"] else lib.ocipIntegral,
                "args": (P.handle, S.handle, D.handle), "keep": (S, P), "out": Map.of(D)}
    if path == "batch":
        T = [ocip.Image(t).send() for t in a["tpl"]]
        D = [_dest(h, w) for _ in T]
        return {"call": getattr(lib, "ocip" + case["op"] + "Batch"),
                "args": (S.handle, ocip.handles(T), ocip.handles(D), len(T),
                         _PRECISION[case["precision"]]),
                "keep": (S, T), "out": [Map.of(d) for d in D]}
    T = ocip.Image(a["tpl"]).send()
    D = _dest(h, w, channels=case.get("channels", 1))
    state = {"call": getattr(lib, "ocip" + case["op"]), "args": (S.handle, T.handle, D.handle),
             "keep": (S, T), "out": Map.of(D)}
    if path == "mfma":
        state["call"] = getattr(lib, "ocip" + case["op"] + "Ex")
        state["args"] += (_PRECISION[case["precision"]],)
    elif path == "fft":
        P = Program(lib.ocipPrepareImageProximityFFT, S, T)
        state["call"] = getattr(lib, "ocip" + case["op"].replace("_", "FFT_"))
        state["args"] = (P.handle,) + state["args"]
        state["keep"] += (P,)
    elif case["locate"]:
        P = Program(lib.ocipPrepareStatistics, D)
        found = (ctypes.c_double(), ctypes.c_int(), ctypes.c_int())
        state["locate"] = lib.ocipMaxIndx if case["op"].startswith("CrossCorr") else lib.ocipMinIndx
        state["locate_args"] = (P.handle, D.handle) + tuple(ctypes.byref(v) for v in found)
        state["found"] = found
        state["keep"] += (P,)
    return state


def run(state):
    ocip.check(state["call"](*state["args"]), "call")
    if "locate" not in state:
        return state["out"]
    ocip.check(state["locate"](*state["locate_args"]), "locate")
    value, x, y = state["found"]
    return {"map": state["out"], "value": value.value, "x": x.value, "y": y.value}


# ------------------------------------------------------------------------------ its work
def work(case):
    w, h, path = case["w"], case["h"], case["path"]
    px = w * h
    if path == "integral":
        size = np.dtype(_TYPE[case["type"]]).itemsize + np.dtype(_TYPE[case["dest"]]).itemsize
        return {"bytes": px * size, "flops": px * (3 if case["sqr"] else 2)}
    if path == "batch":
        mix = random.Random(case["mix"])
        taps = sum(mix.randint(case["lo"], case["hi"]) * mix.randint(case["lo"], case["hi"])
                   for _ in range(case["count"]))
        return {"bytes": 4 * (px * (1 + case["count"]) + taps), "flops": 2 * px * taps}
    taps = case["tw"] * case["th"]
    if path == "gradients":
        # the image, both weights and the gradient of each; per output pixel and tap one
        # multiply-add each for the forward map, the image's and the template's gradient
        return {"bytes": 4 * (4 * case["count"] * px + 2 * taps), "flops": 6 * case["count"] * px * taps}
    if path == "fft":
        # a real transform of the padded image and of the template, and one back
        n = (w + case["tw"]) * (h + case["th"])
        return {"bytes": 4 * (2 * px + taps), "flops": 3 * 2.5 * n * math.log2(n)}
    size, ch = np.dtype(_TYPE[case.get("type", "F32")]).itemsize, case.get("channels", 1)
    per_tap = 2 if case["op"].startswith("CrossCorr") else 3
    return {"bytes": ch * (px * (size + 4) + taps * size), "flops": per_tap * ch * px * taps}


# ------------------------------------------------------------------------------ in 64 bits
def _size(n):
    return (n + 63) // 64 * 64


def _correlate(P, t, h, w):
    """sum over u, v of P[..., y + v, x + u] t[v, u], for y < h and x < w."""
    n = (_size(P.shape[-2]), _size(P.shape[-1]))
    f = torch.fft.rfft2(P, s=n) * torch.fft.rfft2(t, s=n).conj()
    return torch.fft.irfft2(f, s=n)[..., :h, :w]


def _pad(s, tw, th):
    cx, cy = tw // 2, th // 2
    return torch.nn.functional.pad(s, (cx, tw - 1 - cx, cy, th - 1 - cy))


def _box(P, tw, th, h, w):
    rows = sum(P[..., v:v + h, :] for v in range(th))
    return sum(rows[..., u:u + w] for u in range(tw))


def _map(op, src, tpl):
    h, w = src.shape
    th, tw = tpl.shape
    P = _pad(src, tw, th)
    if op == "AbsDistance":
        out = torch.zeros_like(src)
        for v in range(th):
            for u in range(tw):
                out += (P[v:v + h, u:u + w] - tpl[v, u]).abs_()
        return out
    out = _correlate(P, tpl, h, w)
    if op == "CrossCorr":
        return out
    ss, tt = _box(P * P, tw, th, h, w), (tpl * tpl).sum()
    if op.startswith("SqrDistance"):
        out = (ss + tt - 2 * out).clamp_(min=0)
    return out / torch.sqrt(ss * tt) if op.endswith("_Norm") else out


def _wide(a):
    return torch.from_numpy(np.ascontiguousarray(a).astype(np.float64)).to(_device())


def exact(case, seed):
    a, path = _inputs(case, seed), case["path"]
    src = _wide(a["src"])
    if path == "integral":
        f = src * src if case["sqr"] else src
        return f.cumsum(0).cumsum(1).cpu()
    if path == "batch":
        return [_map(case["op"], src, _wide(t)).cpu() for t in a["tpl"]]
    tpl = _wide(a["tpl"])
    if path == "gradients":
        h, w, th, tw = case["h"], case["w"], case["th"], case["tw"]
        dT, dS = torch.zeros_like(tpl), []
        ones = torch.ones_like(tpl)
        for k in range(case["count"]):
            s, t = src[k].requires_grad_(), tpl.detach().requires_grad_()
            P = _pad(s, tw, th)
            c, ss, tt = _correlate(P, t, h, w), _correlate(P * P, ones, h, w), (t * t).sum()
            loss = (_wide(a["g_ncc"][k]) * c / torch.sqrt(ss * tt)).sum() + \
                (_wide(a["g_ssd"][k]) * (ss - 2 * c + tt)).sum()
            ds, dt = torch.autograd.grad(loss, (s, t))
            dS.append(ds.cpu())
            dT += dt
        return {"source": dS, "template": dT.cpu()}
    if case.get("channels", 1) > 1:
        return torch.stack([_map(case["op"], src[..., c].contiguous(), tpl[..., c].contiguous())
                            for c in range(case["channels"])], dim=-1).cpu()
    out = _map(case["op"], src, tpl).cpu()
    if not case.get("locate"):
        return out
    # where two pixels are equally good in fewer bits either may be named: no value for these
    return {"map": out, "value": None, "x": None, "y": None}
