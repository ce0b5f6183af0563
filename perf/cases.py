"""The work that users of this framework have it do, as cases that can be timed.

Each case goes through the library's public entry points (the C-ABI in
include/sexgpu.h, by way of gpu-sextractor_amd/sexgpu.py): whole frames kept on the GPU
(sxg_process_resident), the reference front-end's call order from host memory, catalogue
photometry, weight maps, the FP64 catalogue mode, batches from host memory, the graph
batch as a serving loop, and the allocation-free background.  Frames come from the
repository's own generator with the source densities and flux laws of its workloads.

Sizes are pixels.  Results are bit-exact by contract (integers, bytes and floats alike),
except the FP64 catalogue mode, whose sums may be taken in another order.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "gpu-sextractor_amd"))
import sexgpu  # noqa: E402

CONV3, GAUSS7, MEXHAT11 = "default.conv", "gauss_3.0_7x7.conv", "mexhat_5.0_11x11.conv"
FRAME_VALUES = ("backmean", "backsig", "dthresh", "thresh")
FRAME_COUNTS = ("npix_above", "npix_raw", "nraw", "nobj", "nsurv")
OUTOBJ = np.dtype({"names": [f[0] for f in sexgpu.OutObj._fields_],
                   "formats": [np.dtype((f[1]._type_, f[1]._length_)) if hasattr(f[1], "_length_")
                               else np.dtype(f[1]) for f in sexgpu.OutObj._fields_],
                   "offsets": [getattr(sexgpu.OutObj, f[0]).offset
                               for f in sexgpu.OutObj._fields_],
                   "itemsize": C.sizeof(sexgpu.OutObj)})


def listed():
    def case(name, kind, width, height, mask, density, preset="plain1024", fmin=0.0, back_size=64):
        return {"name": name, "kind": kind, "width": width, "height": height, "mask": mask,
                "density": density, "preset": preset, "fmin": fmin, "back_size": back_size}

    return [
        # a postage stamp cut out around a target: launches and host round trips
        case("stamp_300x260", "resident", 300, 260, CONV3, 3e-3),
        # the ordinary small frame of the tests and the smoke check
        case("plain_1024", "resident", 1024, 1024, CONV3, 3000 / 1024 ** 2),
        # a detector with overscan cut off: no size is a multiple of anything
        case("ragged_2011x1533", "resident", 2011, 1533, CONV3, 3e-3),
        # the headline frame: a crowded field
        case("crowded_4096", "resident", 4096, 4096, GAUSS7, 167000 / 4096 ** 2, "crowded4096"),
        # a globular-cluster-like field: nearly half of the pixels are in blends
        case("dense_2048", "resident", 2048, 2048, GAUSS7, 167000 / 4096 ** 2, "crowded4096",
             3000.0),
        # half of a wide-field plate with its weight map, large filter, large meshes
        case("wide_8192x4096", "weighted", 8192, 4096, MEXHAT11, 400000 / 8192 ** 2,
             "wide8192", 0.0, 128),
        # saturated stars over faint sources, catalogue in FP64
        case("hdr_2048", "precision", 2048, 2048, GAUSS7, 100000 / 4096 ** 2, "hdr4096"),
        # detection plus the catalogue photometry with CLASS_STAR
        case("photometry_2048", "photometry", 2048, 2048, GAUSS7, 167000 / 4096 ** 2,
             "crowded4096"),
        # the reference front-end's thirteen calls on one frame in host memory
        case("drop_in_1024", "drop_in", 1024, 1024, CONV3, 3000 / 1024 ** 2),
        # a night's uneven frames from host memory over the worker contexts
        {"name": "host_batch_8", "kind": "host_batch", "frames": 8, "mix": 2000, "mask": CONV3},
        # a serving loop: new pixels into a resident batch, one graph launch, maps out
        {"name": "graph_batch_12", "kind": "graph_batch", "frames": 12, "mix": 2064,
         "mask": CONV3},
        # background estimation alone, on frames that the caller keeps as tensors
        case("background_4096", "background", 4096, 4096, CONV3, 3e-3),
    ]


def draw(rng):
    kind = rng.choice(["resident"] * 5 + ["drop_in"] * 2 + ["photometry", "weighted", "precision",
                                                         "background", "host_batch",
                                                         "graph_batch"])
    if kind in ("host_batch", "graph_batch"):
        return {"kind": kind, "frames": rng.randint(4, 12), "mix": rng.randint(0, 10 ** 6),
                "mask": rng.choice([CONV3, GAUSS7])}

    def side(lo, hi):
        s = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return rng.choice([s, s | 1, max(64 * (s // 64), 192), s])

    dense = kind == "resident" and rng.random() < 0.25
    most = 2048 if dense or kind in ("drop_in", "photometry", "precision") else 4096
    width, height = side(192, most), side(192, most)
    preset = "plain1024"
    density = 10 ** rng.uniform(-4, -2)
    if kind == "precision":
        preset, density = "hdr4096", 100000 / 4096 ** 2
    elif dense or rng.random() < 0.4:
        preset = "crowded4096"
    return {"kind": kind, "width": width, "height": height,
            "mask": rng.choice([CONV3, GAUSS7, MEXHAT11]), "density": density,
            "preset": preset, "fmin": 3000.0 if dense else 0.0,
            "back_size": rng.choice([32, 64, 64, 64, 128])}


# ---------------------------------------------------------------- inputs ----
def _frame(case, seed):
    w, h = case["width"], case["height"]
    kw = {"width": w, "height": h, "nsrc": max(1, int(round(case["density"] * w * h))),
          "seed": seed}
    if case["fmin"]:
        kw["fmin"] = case["fmin"]
    if case["preset"] == "hdr4096":
        kw["nsat"] = max(1, int(round(200 * w * h / 4096 ** 2)))
    return sexgpu.synth(case["preset"], **kw)


def _batch_shapes(case):
    """(height, width, density) of each frame: the many-frame workload's sizes and
    densities."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["frames"]):
        h, w = sexgpu.BATCH64_SIZES[int(rng.integers(0, len(sexgpu.BATCH64_SIZES)))]
        out.append((h, w, float(10 ** rng.uniform(-4, -2))))
    return out


def _pinned(shape, dtype):
    return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()


def _pin(frame):
    out = _pinned(frame.shape, torch.float32)
    out[...] = frame
    return out


def _params(case):
    return sexgpu.Params(mask=sexgpu.read_conv(case["mask"]),
                         back_size=case.get("back_size", 64))


class _Ctx:
    """A context of the library's, as a program keeps one for each frame in flight: taken
    from the free ones, given back with its frame."""
    free = []

    def __init__(self):
        self.ptr = self.free.pop() if self.free else sexgpu.gpu().sxg_ctx_create()

    def bind(self):
        sexgpu.gpu().sxg_ctx_bind(self.ptr)

    def __del__(self):
        self.free.append(self.ptr)


class _Plane:
    """A W x H float plane of a context's as an array on the GPU; keeps the context."""

    def __init__(self, ctx, ptr, shape):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "version": 2,
                                         "data": (ptr, False)}


def _planes(state):
    """The background-subtracted and the filtered frame, where they are."""
    L = sexgpu.gpu()
    ptrs = (L.sxg_device_frame(0), L.sxg_device_frame(1))
    if state.get("planes_at") != ptrs:
        state["planes_at"] = ptrs
        state["planes"] = [torch.as_tensor(_Plane(state["ctx"], p, state["shape"]), device="cuda")
                           for p in ptrs]
    return state["planes"]


_graph_of = None   # the shapes and filter of the batch that the library holds


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("host_batch", "graph_batch"):
        p = _params(case)
        frames = [_pin(sexgpu.synth("plain1024", width=w, height=h, seed=1000 * seed + i,
                                    nsrc=max(1, int(round(d * w * h)))))
                  for i, (h, w, d) in enumerate(_batch_shapes(case))]
        state = {"kind": kind, "p": p, "frames": frames,
                 "segs": [_pinned(f.shape, torch.int32) for f in frames]}
        if kind == "host_batch":
            state["rows"] = [np.zeros(max(64, f.size // 64), sexgpu.ISOROW_DTYPE) for f in frames]
        else:
            state["key"] = repr((_batch_shapes(case), case["mask"]))
            _hold_batch(state)
        return state
    img = _frame(case, seed)
    h, w = img.shape
    p = _params(case)
    if kind == "background":
        return {"kind": kind, "p": p, "src": torch.from_numpy(img).cuda(),
                "dst": torch.empty((h, w), dtype=torch.float32, device="cuda")}
    cap = max(64, w * h // 64)
    if kind == "drop_in":
        return {"kind": kind, "p": p, "img": _pin(img), "seg": _pinned((h, w), torch.int32),
                "sub": _pinned((h, w), torch.float32), "master": np.zeros(cap, np.uint32),
                "rows": np.zeros(cap, sexgpu.ISOROW_DTYPE)}
    ctx = _Ctx()
    ctx.bind()
    L = sexgpu.gpu()
    wt = None
    if kind == "weighted":
        # 20 % vignetting and 1 % dead columns
        wt = sexgpu.synth_weight(case["preset"], width=w, height=h, seed=seed)
    sexgpu.set_weight(wt, p)
    L.sxg_set_resident_frame(img.ctypes.data, w, h)
    sexgpu.check()
    state = {"kind": kind, "p": p, "ctx": ctx, "shape": (h, w), "native": sexgpu.native_params(p)}
    if kind == "photometry":
        sexgpu.set_photometry()
        state["brain"] = sexgpu.read_nnw("default.nnw")
        state["rows"] = np.zeros(cap, OUTOBJ)
    else:
        state["rows"] = np.zeros(cap, sexgpu.ISOROW_DTYPE)
    return state


def _hold_batch(state):
    """The resident batch and its graph, once for each kind of batch."""
    global _graph_of
    if _graph_of != state["key"]:
        sexgpu.set_batch_frames(state["frames"])
        sexgpu.process_batch_graph(len(state["frames"]), None, state["p"], nworkers=8,
                                   segmaps=False)
        _graph_of = state["key"]


# ------------------------------------------------------------------ a pass ----
def run(state):
    return {"background": _run_background, "drop_in": _run_drop_in, "host_batch": _run_host_batch,
            "graph_batch": _run_graph_batch}.get(state["kind"], _run_resident)(state)


def _fields(rows):
    """The columns of the catalogue rows: the whole buffer, of which the first nsurv (the
    photometry: nobj) rows are written."""
    return {k: rows[k] for k in rows.dtype.names if not k.startswith("_")}


def _run_resident(state):
    L, p = sexgpu.gpu(), state["p"]
    state["ctx"].bind()
    precise = state["kind"] == "precision"
    if precise:
        sexgpu.set_option("precision", 1)
    fi = sexgpu.FrameInfo()
    nobj = L.sxg_process_resident(C.byref(state["native"]), C.byref(fi))
    if precise:
        sexgpu.set_option("precision", 0)
    sexgpu.check()
    rows = state["rows"]
    if state["kind"] == "photometry":
        h, w = state["shape"]
        if nobj > rows.size:
            raise RuntimeError("%d objects" % nobj)
        L.endobject_gpu(None, C.byref(state["brain"]), None, rows.ctypes.data, None, 0, h, w, h,
                        fi.backsig, fi.thresh, p.satur_level, 1.0, 0.0, p.gain, nobj)
    else:
        L.sxg_get_catalog(rows.ctypes.data, rows.size)
    sexgpu.check()
    sub, cd = _planes(state)
    out = {k: getattr(fi, k) for k in FRAME_VALUES + FRAME_COUNTS}
    out.update(sub=sub, cd=cd, rows=_fields(rows))
    return out


def _run_drop_in(state):
    sexgpu.gpu().sxg_ctx_bind(None)
    nobj, nsurv = sexgpu.run_drop_in(state["img"], state["p"], state["seg"], state["sub"],
                                     state["master"], state["rows"])
    return {"nobj": nobj, "nsurv": nsurv, "seg": state["seg"], "sub": state["sub"],
            "master": state["master"], "rows": _fields(state["rows"])}


def _infos(infos):
    out = {k: np.array([getattr(f, k) for f in infos], np.float32) for k in FRAME_VALUES}
    out.update((k, np.array([getattr(f, k) for f in infos], np.int64)) for k in FRAME_COUNTS)
    return out


def _run_host_batch(state):
    infos, _, segs, _ = sexgpu.process_batch_host(state["frames"], state["p"], nworkers=4,
                                                  segs=state["segs"], rows=state["rows"])
    return dict(_infos(infos), segs=segs, rows=[r.view(np.uint8) for r in state["rows"]])


def _run_graph_batch(state):
    L, frames = sexgpu.gpu(), state["frames"]
    _hold_batch(state)
    for i, f in enumerate(frames):
        if L.sxg_batch_update_frame(i, f.ctypes.data) != 0:
            sexgpu.check()
    infos, _, _, _ = sexgpu.process_batch_graph(len(frames), None, state["p"], nworkers=8,
                                                segmaps=False)
    for i, s in enumerate(state["segs"]):
        if L.sxg_batch_segmap(i, s.ctypes.data) != 0:
            sexgpu.check()
    return dict(_infos(infos), segs=state["segs"])


def _run_background(state):
    src, dst, p = state["src"], state["dst"], state["p"]
    h, w = src.shape
    bs = p.back_size
    nbx, nby = (w - 1) // bs + 1, (h - 1) // bs + 1
    mean, sig = C.c_float(), C.c_float()
    if sexgpu.gpu().sxg_back_estimate_noalloc(
            src.data_ptr(), dst.data_ptr(), w, h, bs, 0.0, p.back_fsize if nbx > 1 else 1,
            p.back_fsize if nby > 1 else 1, 0, 0.0, C.byref(mean), C.byref(sig),
            torch.cuda.current_stream().cuda_stream) != 0:
        sexgpu.check()
    return {"backmean": mean.value, "backsig": sig.value, "sub": dst}


# -------------------------------------------------- bounds and tolerances ----
def work(case):
    """The frame read and the subtracted, filtered and segmentation planes written once
    (what each kind has of them), with weights read; two operations for each tap of the
    filter and a few for each pixel of the background."""
    kind = case["kind"]
    if kind in ("host_batch", "graph_batch"):
        n = sum(h * w for h, w, _ in _batch_shapes(case))
    else:
        n = case["width"] * case["height"]
    planes = {"background": 2, "drop_in": 3, "host_batch": 2, "graph_batch": 2,
              "weighted": 5}.get(kind, 4)
    taps = {CONV3: 9, GAUSS7: 49, MEXHAT11: 121}[case["mask"]]
    return {"bytes": 4.0 * planes * n,
            "flops": float(n) * ((0 if kind == "background" else 2 * taps) + 20)}


def tolerance(case):
    if case["kind"] == "precision":
        # FP64 sums in any order (1e-15), rounded to float columns: 6e-8 to 1e-7 seen
        # against long double, angles of round objects 4e-6 degrees
        return {"rel": 2.5e-7, "max": 2e-5, "differ": 0.0}
    return "exact"


# --------------------------------------------------------- 64-bit reference ----
def exact(case, seed):
    """The background in 64 bits, and the frames and values that follow from it.  The
    catalogue has no 64-bit value here: its columns are sums over pixel sets that the
    detection decides."""
    kind = case["kind"]
    if kind in ("host_batch", "graph_batch", "weighted"):
        return None
    if case["width"] * case["height"] > 5e6:
        return None
    img = _frame(case, seed).astype(np.float64)
    mean, sig, back = _background64(img, case["back_size"], 3)
    sub = img - back
    if kind == "background":
        return {"backmean": mean, "backsig": sig, "sub": sub}
    if kind == "drop_in":
        return {"nobj": None, "nsurv": None, "seg": None, "sub": sub, "master": None,
                "rows": None}
    out = {k: None for k in FRAME_COUNTS}
    out.update(backmean=mean, backsig=sig, dthresh=1.5 * sig, thresh=1.5 * sig, sub=sub,
               cd=_correlate64(sub, sexgpu.read_conv(case["mask"]).astype(np.float64)), rows=None)
    return out


def _correlate64(a, mask):
    k = mask.shape[0] // 2
    h, w = a.shape
    pad = np.pad(a, k)
    out = np.zeros_like(a)
    for i in range(mask.shape[0]):
        for j in range(mask.shape[1]):
            out += mask[i, j] * pad[i:i + h, j:j + w]
    return out


def _background64(img, bs, fs):
    """SExtractor's background: clipped mesh statistics, the mode of each mesh's
    histogram, median filtering, natural bicubic splines."""
    h, w = img.shape
    bs = min(bs, w, h)
    nx, ny = (w - 1) // bs + 1, (h - 1) // bs + 1
    back, sigma = np.zeros((ny, nx)), np.zeros((ny, nx))
    for j in range(ny):
        for i in range(nx):
            back[j, i], sigma[j, i] = _mode64(img[j * bs:(j + 1) * bs, i * bs:(i + 1) * bs].ravel())
    fx, fy = (fs if nx > 1 else 1) // 2, (fs if ny > 1 else 1) // 2
    fb, fsig = np.zeros_like(back), np.zeros_like(sigma)
    for j in range(ny):
        dj = min(fy, ny - 1 - j, j)
        for i in range(nx):
            di = min(fx, nx - 1 - i, i)
            at = np.s_[j - dj:j + dj + 1, i - di:i + di + 1]
            fb[j, i], fsig[j, i] = np.median(back[at]), np.median(sigma[at])
    nodes = _spline64(fb, _positions(h, bs, ny))
    full = _spline64(np.ascontiguousarray(nodes.T), _positions(w, bs, nx, centre=True)).T
    return float(np.median(fb)), float(np.median(fsig)), full


def _mode64(v):
    step = math.sqrt(2 / math.pi) * 5 / 4
    mean = v.mean()
    sig = math.sqrt(max((v * v).mean() - mean * mean, 0.0))
    v1 = v[(v >= mean - 2 * sig) & (v <= mean + 2 * sig)]
    mean = v1.mean()
    sig = math.sqrt(max((v1 * v1).mean() - mean * mean, 0.0))
    nlev = min(int(step * v1.size + 1), 4096)
    scale = 10 * sig / nlev if sig > 0 else 1.0
    zero = mean - 5 * sig
    t = v / scale + (0.499999 - zero / scale)
    hist = np.bincount(t[(t > -1) & (t < nlev)].astype(np.int64), minlength=nlev).tolist()
    lo_cut, hi_cut, s, s1, med, mea = 0, nlev - 1, 10.0 * (nlev - 1), 1.0, mean, mean
    n = 100
    while n and s >= 0.1 and abs(s / s1 - 1.0) > 1e-4:
        n -= 1
        s1 = s
        lo, hi, low, high, total, m1, m2 = lo_cut, hi_cut, 0, 0, 0, 0.0, 0.0
        for i in range(lo_cut, hi_cut + 1):
            if low < high:
                low += hist[lo]
                lo += 1
            else:
                high += hist[hi]
                hi -= 1
            total += hist[i]
            m1 += hist[i] * i
            m2 += hist[i] * i * i
        at = lambda k: hist[k] if 0 <= k < nlev else 0  # noqa: E731
        med = hi + 0.5 + (high - low) / (2.0 * max(at(lo), at(hi))) if hi >= 0 else 0.0
        if total:
            mea = m1 / total
            s = math.sqrt(max(m2 / total - mea * mea, 0.0))
        cut = med - 3 * s
        lo_cut = int(cut + 0.5) if cut > 0 else 0
        cut = med + 3 * s
        hi_cut = int(cut + 0.5 if cut > 0 else cut - 0.5) if cut < nlev - 1 else nlev - 1
    if s > 0 and abs((mea - med) / s) < 0.3:
        best = 2.5 * med - 1.5 * mea
    else:
        best = med if s > 0 else mea
    return zero + best * scale, s * scale


def _positions(n, bs, nodes, centre=False):
    """(segment, offset in it) of each pixel among the mesh centres.  Rows sit half a
    pixel below columns, as SExtractor has them; the outermost segments extrapolate."""
    at = (np.arange(n) + (0.5 if centre else 0.0)) / bs - 0.5
    seg = np.clip(np.floor(at).astype(np.int64), 0, max(nodes - 2, 0))
    return seg, at - seg


def _spline64(v, positions):
    """The natural cubic spline through the rows of v (SExtractor's second derivatives,
    over 6), at the given rows."""
    n = v.shape[0]
    seg, d = positions
    if n == 1:
        return np.repeat(v, d.size, 0)
    d2, u = np.zeros_like(v), np.zeros_like(v)
    for k in range(1, n - 1):
        t = -1 / (d2[k - 1] + 4)
        d2[k] = t
        u[k] = t * (u[k - 1] - 6 * (v[k + 1] + v[k - 1] - 2 * v[k]))
    for k in range(n - 2, 0, -1):
        d2[k] = (d2[k] * d2[k + 1] + u[k]) / 6.0
    d2[0] = d2[n - 1] = 0.0
    d = d[:, None]
    c = 1 - d
    return c * v[seg] + d * v[seg + 1] + (c ** 3 - c) * d2[seg] + (d ** 3 - d) * d2[seg + 1]
