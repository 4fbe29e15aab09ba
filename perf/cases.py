"""Performance cases of libapr_amd: what a program that uses this package has it do.

listed() names the cases, draw(rng) gives more of the same ranges, prepare(case, seed) makes what
a program has in hand before a call, and run(state) is one pass through the public entry points on
device-resident data.  exact(case, seed) is the same result in plain torch in 64 bits, for the
passes whose outputs are computed numbers.

The volumes are the package's synthetic ones (Gaussian blobs on a background with shot noise, and
for deconvolution the same blurred by a PSF), at the parameters of the benchmark and the tests.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import libapr_amd as A  # noqa: E402
from libapr_amd import warm_start as W  # noqa: E402

APR_PARAMS = dict(rel_error=0.1, lambda_=3.0, sigma_th=50.0, Ip_th=120.0, grad_th=10.0)
SIDES = (128, 192, 256, 384, 512)   # the batch benchmark's volume sides (z capped at 256)


# ---------------- the cases ----------------

def listed():
    return [
        # conversion (APRConverter.get_apr) with the particles sampled from the same image
        # a small crop, where launches and latency count: the tests' size
        dict(name="convert_crop_u16", op="convert", y=60, x=52, z=36, dtype="uint16"),
        # a microscope stack whose sides are no multiples of anything
        dict(name="convert_ragged_u16", op="convert", y=1001, x=777, z=203, dtype="uint16"),
        # the benchmark's volume
        dict(name="convert_large_u16", op="convert", y=2048, x=2048, z=512, dtype="uint16"),
        # a float image (APRConverter<float>): a preprocessed or normalised stack
        dict(name="convert_f32", op="convert", y=640, x=513, z=250, dtype="float32"),
        # many stacks of uneven sizes through one recorded plan
        dict(name="convert_batch", op="batch", volumes=12, sides=2, odd=False),
        # a filter on a small APR, in the reference's summation order: the benchmark's small volume
        dict(name="filter_small", op="filter", y=256, x=256, z=128, taps=3, dtype="uint16", separable=False),
        # a Gaussian on an ordinary APR of float particles, in the reference's summation order
        dict(name="filter_exact", op="filter", y=1000, x=1024, z=250, taps=5, dtype="float32", separable=False),
        # Richardson-Lucy at the benchmark's size, separable PSF
        dict(name="deconvolve", op="deconvolve", y=1024, x=1024, z=256, taps=9, iterations=4, separable=True),
        # particles back to pixels, for display or a pixel-based tool
        dict(name="reconstruct", op="reconstruct", y=1000, x=1023, z=255, smooth=False),
        # the smooth reconstruction, for display
        dict(name="reconstruct_smooth", op="reconstruct", y=512, x=480, z=200, smooth=True),
        # the trained warm-start network over a reconstructed image
        dict(name="network_apply", op="network", y=512, x=500, z=130),
        # one training step of that network on a batch of tiles
        dict(name="network_train", op="train", tiles=16, side=64),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _volume(rng, voxels):
    """a stack of about `voxels` voxels: uneven sides, z mostly the shortest; every third has a y side that is a multiple of 64"""
    fy, fx, fz = 2 ** rng.uniform(-0.7, 0.7), 2 ** rng.uniform(-0.7, 0.7), 2 ** rng.uniform(-2.5, 0.0)
    f = (voxels / (fy * fx * fz)) ** (1.0 / 3.0)
    y, x, z = (max(24, int(f * v)) for v in (fy, fx, fz))
    if rng.random() < 0.33:
        y = max(64, y // 64 * 64)
    return dict(y=y, x=x, z=z)


def draw(rng):
    op = rng.choice(["convert", "convert", "convert", "batch", "filter", "filter", "deconvolve", "reconstruct", "reconstruct", "network", "train"])
    if op == "convert":
        return dict(op=op, dtype=rng.choice(["uint16", "uint16", "float32"]), **_volume(rng, _log(rng, 60_000, 400_000_000)))
    if op == "batch":
        return dict(op=op, volumes=rng.randint(3, 14), sides=rng.randint(3, 1 << 20), odd=rng.random() < 0.5)
    if op == "filter":
        return dict(op=op, taps=rng.choice([3, 3, 5, 5, 7]), dtype=rng.choice(["uint16", "float32"]), separable=rng.random() < 0.5,
                    **_volume(rng, _log(rng, 500_000, 150_000_000)))
    if op == "deconvolve":
        return dict(op=op, taps=rng.choice([5, 7, 9]), iterations=rng.randint(2, 5), separable=True, **_volume(rng, _log(rng, 1_000_000, 150_000_000)))
    if op == "reconstruct":
        return dict(op=op, smooth=rng.random() < 0.5, **_volume(rng, _log(rng, 500_000, 150_000_000)))
    if op == "network":
        return dict(op=op, **_volume(rng, _log(rng, 500_000, 30_000_000)))
    return dict(op=op, tiles=rng.randint(2, 20), side=rng.choice([32, 48, 64, 64]))


# ---------------- what a program has in hand ----------------

_contexts = {}
_latest = [None]


def _context(case):
    """The program's context (one per convolution mode).  A program works on one kind of data at a time: when the
    case changes, the memory cached for the last one goes back."""
    key = str(sorted((k, v) for k, v in case.items() if k != "name"))
    if _latest[0] != key:
        for c in _contexts.values():
            c.release_cache()
        _latest[0] = key
    sep = bool(case.get("separable", False))
    if sep not in _contexts:
        _contexts[sep] = A.Context(0)
        _contexts[sep].set_conv_mode(A.CONV_SEPARABLE if sep else A.CONV_EXACT)
    return _contexts[sep]


class _Span:
    """device memory of `owner` for torch.as_tensor: no copy, and the owner lives as long as the tensor"""

    def __init__(self, owner, address, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(int(count),), typestr=typestr, data=(int(address), False), version=2)


def _structure(apr):
    """(xz_end_vec, y_vec) of an APR as device tensors (u64 and u16 seen as signed)"""
    xz, yv = apr.device_structure()
    return (torch.as_tensor(_Span(apr, xz, apr.xz_end_size, "<i8"), device="cuda"),
            torch.as_tensor(_Span(apr, yv, apr.total, "<i2"), device="cuda"))


def _room(dims):
    """a program's own buffers for the structure of an APR of these dims: xz_end_vec, and y_vec for as many particles as there are voxels"""
    y, x, z = dims
    top = max(1, int(np.ceil(np.log2(max(dims)))))
    rows = 1 + sum(-(-x // (1 << (top - lv))) * -(-z // (1 << (top - lv))) for lv in range(1, top + 1))
    return torch.zeros(rows, dtype=torch.int64, device="cuda"), torch.zeros(x * y * z, dtype=torch.int16, device="cuda")


def _keep(apr, room):
    """the APR's structure into the program's buffers"""
    A._check(A.lib().aprh_apr_copy_structure(apr.h, None, room[0].data_ptr(), room[1].data_ptr()))
    return [apr.total, room[0], room[1]]


def _blobs(ctx, case, seed):
    y, x, z = case["y"], case["x"], case["z"]
    img = torch.empty(z * x * y, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    A.synth_blobs((z, x, y), seed, max(8, y * x * z // 22 ** 3), sigma=(1.5, 8.0), amp=(300.0, 4000.0), background=100.0, noise=True,
                  out=img.data_ptr(), ctx=ctx)
    return img


def _blurred(ctx, case, seed):
    y, x, z = case["y"], case["x"], case["z"]
    truth = torch.empty(z * x * y, dtype=torch.float32, device="cuda")
    img = torch.empty(z * x * y, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    A.synth_deconv((z, x, y), seed, max(8, y * x * z // 5400), truth.data_ptr(), img.data_ptr(), sigma=(1.0, 4.0), amp=(200.0, 2000.0),
                   background=100.0, psf_sigma=(1.0, 1.0, 2.0), psf_taps=9, ctx=ctx)
    return img, truth


def _converted(ctx, case, img):
    """the APR of a u16 image and its particles"""
    conv = A.APRConverter(ctx)
    conv.par = A.APRParameters(**APR_PARAMS)
    dims = (case["y"], case["x"], case["z"])
    apr = conv.get_apr(img, dims=dims)
    parts = torch.empty(apr.total, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    A.ParticleData().sample_image(apr, img, out=parts, dtype="uint16")
    return apr, parts


def _as_float(parts):
    return (parts.to(torch.int32) & 0xFFFF).to(torch.float32)


def _batch_dims(case):
    rng = np.random.default_rng(case["sides"])
    d = rng.choice(SIDES, size=(case["volumes"], 3))
    d[:, 2] = np.minimum(d[:, 2], 256)
    if case["odd"]:
        d = d - rng.integers(0, 60, size=d.shape)
    return [tuple(int(v) for v in r) for r in d]


def prepare(case, seed):
    ctx = _context(case)
    s = dict(case=case, ctx=ctx)
    op = case["op"]
    seed = int(seed) & 0x7FFFFFFF
    if op == "convert":
        img = _blobs(ctx, case, seed)
        n = img.numel()
        if case["dtype"] == "float32":
            img = _as_float(img)
        s["img"] = img
        # buffers for the most particles that there can be: the rest of them stays as it is
        s["parts"] = torch.zeros(n, dtype=torch.float32 if case["dtype"] == "float32" else torch.int16, device="cuda")
        s["room"] = _room((case["y"], case["x"], case["z"]))
        s["conv"] = A.APRConverter(ctx, image_type=np.dtype(case["dtype"]))
        s["conv"].par = A.APRParameters(**APR_PARAMS)
    elif op == "batch":
        dims = _batch_dims(case)
        s["room"] = [_room(d) for d in dims]
        s["batch"] = A.APRBatch(dims, par=A.APRParameters(**APR_PARAMS), ctx=ctx)
        for i, (y, x, z) in enumerate(dims):
            A.synth_blobs((z, x, y), (seed << 8) + i, max(1, y * x * z // 32 ** 3), sigma=(1.5, 8.0), amp=(300.0, 4000.0), background=100.0,
                          noise=True, out=s["batch"].input_address(i), ctx=ctx)
    elif op == "filter":
        s["apr"], parts = _converted(ctx, case, _blobs(ctx, case, seed))
        s["parts"] = _as_float(parts) if case["dtype"] == "float32" else parts
        k = case["taps"]
        s["stencil"] = A.APRStencil.create_mean_filter((3, 3, 3)) if k == 3 else A.APRStencil.create_gaussian_filter((k / 5.0,) * 3, (k,) * 3, True)
        s["out"] = torch.zeros(case["y"] * case["x"] * case["z"], dtype=torch.float32, device="cuda")
    elif op == "deconvolve":
        img, _ = _blurred(ctx, case, seed)
        s["apr"], s["parts"] = _converted(ctx, case, img)
        k = case["taps"]
        s["psf"] = A.APRStencil.create_gaussian_filter((1.0, 1.0, 2.0), (k, k, k), True)
        s["out"] = torch.zeros(case["y"] * case["x"] * case["z"], dtype=torch.float32, device="cuda")
    elif op == "reconstruct":
        s["apr"], s["parts"] = _converted(ctx, case, _blobs(ctx, case, seed))
        s["out"] = torch.empty((case["z"], case["x"], case["y"]), dtype=torch.float32 if case["smooth"] else torch.int16, device="cuda")
    elif op == "network":
        img, _ = _blurred(ctx, case, seed)
        apr, parts = _converted(ctx, case, img)
        s["img"] = torch.empty((case["z"], case["x"], case["y"]), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        _reconstruct(apr, parts, s["img"], False)
        s["net"] = A.WarmStartCNN.load(W.DEFAULT_WEIGHTS, ctx=ctx)
        s["out"] = torch.empty_like(s["img"])
    else:
        # tiles of a blurred volume and of its ground truth, normalised by the observed mean
        t, S = case["tiles"], case["side"]
        d = dict(y=256, x=256, z=128)
        img, truth = _blurred(ctx, d, seed)
        img = _as_float(img)
        mean = float(img.mean())
        rng = np.random.default_rng(seed)
        org = np.stack([rng.integers(0, n - S + 1, t) for n in (256, 256, 128)], axis=1).astype(np.int32)
        s["x"] = torch.empty((t, S + 8, S + 8, S + 8), dtype=torch.float32, device="cuda")
        s["target"] = torch.empty((t, S, S, S), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        A.extract_tiles(img, (256, 256, 128), org, S, 4, mean, out=s["x"], ctx=ctx)
        A.extract_tiles(truth, (256, 256, 128), org, S, 0, mean, out=s["target"], ctx=ctx)
        s["net"] = A.WarmStartCNN(ctx, seed=0)
    torch.cuda.synchronize()
    return s


def _reconstruct(apr, parts, out, smooth):
    # the array form of `out` is for host arrays: device memory goes in by its address
    if smooth:
        A.APRReconstruction.reconstruct_smooth(apr, parts, out_dtype=np.float32, out=out.data_ptr(), dtype="uint16")
    else:
        A.APRReconstruction.reconstruct_constant(apr, parts, out_dtype=np.float32 if out.dtype == torch.float32 else np.uint16,
                                                 out=out.data_ptr(), dtype="uint16")


# ---------------- one pass ----------------

def run(s):
    case = s["case"]
    op = case["op"]
    if op == "convert":
        dims = (case["y"], case["x"], case["z"])
        if case["dtype"] == "uint16":
            apr, sampled = s["conv"].get_apr_and_sample(s["img"], s["parts"].data_ptr(), s["parts"].numel(), dims=dims)
            if not sampled:
                A.ParticleData().sample_image(apr, s["img"], out=s["parts"], dtype="uint16")
        else:
            apr = s["conv"].get_apr(s["img"], dims=dims)
            A.ParticleData().sample_image(apr, s["img"], out=s["parts"], dtype="float32")
        kept = _keep(apr, s["room"])
        apr.close()
        return kept + [s["parts"]]
    if op == "batch":
        s["batch"].run()
        return [_keep(s["batch"].get(i), s["room"][i]) for i in range(case["volumes"])]
    if op == "filter":
        return A.APRFilter.convolve_pencil(s["apr"], s["stencil"], s["parts"], s["out"], dtype=case["dtype"])
    if op == "deconvolve":
        out, _ = A.APRNumerics.richardson_lucy(s["apr"], s["parts"], s["out"], s["psf"], case["iterations"], dtype="uint16")
        return out
    if op == "reconstruct":
        _reconstruct(s["apr"], s["parts"], s["out"], case["smooth"])
        return s["out"]
    if op == "network":
        return s["net"].apply(s["img"], dims=(case["y"], case["x"], case["z"]), out=s["out"], dtype="float32")
    loss, grads = s["net"].train_step(s["x"].data_ptr(), s["target"].data_ptr(), case["side"], 1e-4, grads=True, T=case["tiles"])
    return [loss, grads]


# ---------------- what a pass cannot do without ----------------

# particles per voxel of the blob volumes and of the blurred ones, as the conversion gives them
FILL, FILL_BLURRED = 0.8, 0.46


def _rows(y, x, z):
    return 4 * x * z // 3 + 16


def work(case):
    op = case["op"]
    if op == "train":
        t, S = case["tiles"], case["side"]
        # read tiles and targets; each layer's products forward, for its weights and (but the first) for its input
        return dict(bytes=4.0 * t * ((S + 8) ** 3 + S ** 3),
                    flops=2.0 * 27 * t * (2 * 16 * (S + 6) ** 3 + 3 * 256 * (S + 4) ** 3 + 3 * 256 * (S + 2) ** 3 + 3 * 16 * S ** 3))
    if op == "batch":
        n = sum(y * x * z for y, x, z in _batch_dims(case))
        return dict(bytes=2.0 * n + 2 * FILL * n + sum(8.0 * _rows(*d) for d in _batch_dims(case)), flops=60.0 * n)
    y, x, z = case["y"], case["x"], case["z"]
    n, r = float(y * x * z), 8.0 * _rows(y, x, z)
    if op == "convert":
        size = 4 if case["dtype"] == "float32" else 2
        return dict(bytes=size * n + (2 + size) * FILL * n + r, flops=60.0 * n)
    if op == "filter":
        size = 4 if case["dtype"] == "float32" else 2
        k = case["taps"]
        return dict(bytes=(2 + size + 4) * FILL * n + r, flops=2.0 * (3 * k if case["separable"] else k ** 3) * FILL * n)
    if op == "deconvolve":
        k = case["taps"]
        return dict(bytes=8 * FILL_BLURRED * n + r, flops=case["iterations"] * FILL_BLURRED * n * (2 * 2 * 3 * k + 2))
    if op == "reconstruct":
        return dict(bytes=4 * FILL * n + r + (4 if case["smooth"] else 2) * n, flops=12.0 * n if case["smooth"] else 1.0)
    return dict(bytes=8 * n, flops=2.0 * 27 * (16 + 256 + 256 + 16) * n)


# Largest relative errors: about four times what the results differ by from exact() below.
# Structures, u16 results and whole numbers are the same in every correct implementation, and
# so are the sampled float means up to their own rounding.
def tolerance(case):
    op = case["op"]
    if op == "batch" or (op == "convert" and case["dtype"] == "uint16") or (op == "reconstruct" and not case["smooth"]):
        return "exact"
    if op == "convert":
        return dict(rel=3e-7, max=3e-6)
    if op == "filter":
        return dict(rel=1e-6, max=1e-5)
    if op == "deconvolve":
        return dict(rel=4e-6, max=1e-4)
    if op == "reconstruct":
        return dict(rel=5e-6, max=1e-3)
    if op == "network":
        return dict(rel=8e-3, max=0.5)
    return dict(rel=1e-2, max=0.5)


# ---------------- the same in 64 bits ----------------

def _levels(apr):
    """per level l_min .. l_max: (dims (z, x, y), first particle, flat cell index of each particle)"""
    xz, yv = _structure(apr)
    y, x, z = apr.org_dims
    out, row = {}, 1   # xz_end_vec[0] is the leading zero; levels 0 .. l_min - 1 have no rows
    first = 0
    for lv in range(apr.l_min, apr.l_max + 1):
        s = 1 << (apr.l_max - lv)
        d = (-(-z // s), -(-x // s), -(-y // s))
        n = d[0] * d[1]
        ends = xz[row:row + n]
        starts = xz[row - 1:row + n - 1]
        counts = (ends - starts).clamp_(min=0)
        rows = torch.repeat_interleave(torch.arange(n, device="cuda"), counts)
        m = rows.numel()
        out[lv] = (d, first, rows * d[2] + (yv[first:first + m].to(torch.int64) & 0xFFFF))
        first += m
        row += n
    return out


def _upsampled(a, d):
    for k in range(3):
        a = a.repeat_interleave(2, dim=k).narrow(k, 0, d[k])
    return a


def _children_mean(v, there):
    """mean of the existing children of each 2x2x2 block, and whether there are any"""
    pad = [0, v.shape[2] & 1, 0, v.shape[1] & 1, 0, v.shape[0] & 1]
    v = torch.nn.functional.pad(torch.where(there, v, torch.zeros_like(v)), pad)
    c = torch.nn.functional.pad(there.to(torch.float64), pad)
    z, x, y = (n // 2 for n in v.shape)
    v, c = (t.view(z, 2, x, 2, y, 2).sum(dim=(1, 3, 5)) for t in (v, c))
    return v / c.clamp(min=1.0), c > 0


def _level_images(levels, parts):
    """the piecewise-constant image at each level: particles, coarser particles, and means of finer ones"""
    lo, hi = min(levels), max(levels)
    own, mask = {}, {}
    up_v = up_m = None
    for lv in range(hi, lo - 1, -1):
        d, first, at = levels[lv]
        v = torch.zeros(d[0] * d[1] * d[2], dtype=torch.float64, device="cuda")
        m = torch.zeros(v.numel(), dtype=torch.bool, device="cuda")
        v[at] = parts[first:first + at.numel()]
        m[at] = True
        v, m = v.view(d), m.view(d)
        if up_v is not None:
            v = torch.where(up_m, up_v, v)
            m = m | up_m
        own[lv], mask[lv] = v, m
        if lv > lo:
            up_v, up_m = _children_mean(v, m)
    img = None
    for lv in range(lo, hi + 1):
        if img is not None:
            own[lv] = torch.where(mask[lv], own[lv], _upsampled(img, own[lv].shape))
        img = own[lv]
    return own


def _stencils(st, n):
    """the stencil at level distances 0 .. n - 1: the area-weighted downsampling of its taps"""
    st = torch.as_tensor(np.asarray(st, np.float64))
    out = [st]
    for d in range(1, max(n, 1)):
        step = 1 << d
        w = st
        for k in range(3):
            m = st.shape[k]
            if m == 1:
                continue
            new = max(2 * (((m - 1) // 2 + step - 1) // step) + 1, 3)
            off = (new // 2) * step - m // 2
            i, j = np.arange(new)[:, None] * step, off + np.arange(m)[None, :]
            over = np.maximum(np.minimum(i + step, j + step) - np.maximum(i, j), 0) / step
            w = torch.movedim(torch.tensordot(torch.as_tensor(over, dtype=torch.float64), torch.movedim(w, k, 0), dims=1), 0, k)
        out.append(w)
    return out


def _reflected(n, h):
    q = torch.arange(-h, n + h, device="cuda").abs()
    q = torch.where(q >= n, 2 * (n - 1) - q, q)
    return q.clamp(0, n - 1)


def _convolved(levels, parts, stencils):
    images = _level_images(levels, parts)
    hi = max(levels)
    out = torch.empty_like(parts)
    for lv, (d, first, at) in levels.items():
        w = stencils[min(hi - lv, len(stencils) - 1)]
        v = images.pop(lv)
        for k in range(3):
            if w.shape[k] > 1:
                v = v.index_select(k, _reflected(d[k], w.shape[k] // 2))
        acc = torch.zeros(d, dtype=torch.float64, device="cuda")
        for i in range(w.shape[0]):
            for j in range(w.shape[1]):
                for k in range(w.shape[2]):
                    acc.add_(v[i:i + d[0], j:j + d[1], k:k + d[2]], alpha=float(w[i, j, k]))
        out[first:first + at.numel()] = acc.view(-1)[at]
        del v, acc
    return out


def _filled(room, values):
    """the values of the particles at the front of a buffer of zeros as large as `room`"""
    out = torch.zeros(room.numel(), dtype=torch.float64, device="cuda")
    out[:values.numel()] = values
    return out


def _smoothed(apr, parts):
    """reconstruct_smooth's adaptive window means (scale 2 per axis) of the constant reconstruction"""
    levels = _levels(apr)
    top = max(levels)
    img = _level_images(levels, parts)[top]
    lev = _level_images(levels, torch.cat([torch.full((levels[k][2].numel(),), float(k), dtype=torch.float64, device="cuda") for k in sorted(levels)]))[top]
    half = torch.floor(torch.exp2(top - lev) / 2.0).to(torch.int64)
    del lev
    for axis in (2, 1, 0):
        n = img.shape[axis]
        if n <= 1:
            continue
        most = min(20, n // 2 - 1)
        off = half.clamp(max=most)
        shape = [1, 1, 1]
        shape[axis] = n
        k = torch.arange(n, device="cuda").view(shape).expand(img.shape)
        sums = torch.cat([torch.zeros_like(img.narrow(axis, 0, 1)), img.cumsum(dim=axis)], dim=axis)
        lo, hi = (k - off).clamp(min=0), (k + off).clamp(max=n - 1)
        if axis == 2:   # along y the low end's means leave out the first sample, but at that sample
            lo = torch.where((k >= 1) & (k < off + 1), torch.ones_like(lo), lo)
        mean = (sums.gather(axis, hi + 1) - sums.gather(axis, lo)) / (hi + 1 - lo)
        if axis == 0:   # along z the low end's condition is on the x position
            x = torch.arange(img.shape[1], device="cuda").view(1, -1, 1)
            mean = torch.where((k < off + 1) & ~((k <= most) & (x < off + 1)), img, mean)
        img = mean
    return img


def _network(p, x):
    """four valid 3x3x3 convolutions, ReLU after the first three, residual: x [t, z, x, y], all in 64 bits"""
    sizes = [27 * 16, 16, 27 * 256, 16, 27 * 256, 16, 27 * 16, 1]
    w1, b1, w2, b2, w3, b3, w4, b4 = torch.split(p, sizes)
    a = x.unsqueeze(-1)
    for w, b, ci, co in ((w1, b1, 1, 16), (w2, b2, 16, 16), (w3, b3, 16, 16), (w4, b4, 16, 1)):
        w = w.view(3, 3, 3, ci, co)
        z, xx, y = (n - 2 for n in a.shape[1:4])
        o = b
        for i in range(3):
            for j in range(3):
                for k in range(3):
                    o = o + a[:, i:i + z, j:j + xx, k:k + y].reshape(-1, ci) @ w[i, j, k]
        a = o.view(a.shape[0], z, xx, y, co)
        if co > 1:
            a = torch.relu(a)
    return x[:, 4:-4, 4:-4, 4:-4] + a.squeeze(-1)


def exact(case, seed):
    op = case["op"]
    if op == "batch" or (op == "convert" and case["dtype"] == "uint16") or (op == "reconstruct" and not case["smooth"]):
        return None   # whole numbers
    s = prepare(case, seed)
    if op == "convert":
        # the particles are the image's means over their cells
        apr = s["conv"].get_apr(s["img"], dims=(case["y"], case["x"], case["z"]))
        levels = _levels(apr)
        img = s["img"].to(torch.float64).view(case["z"], case["x"], case["y"])
        out = torch.empty(apr.total, dtype=torch.float64, device="cuda")
        for lv in sorted(levels, reverse=True):
            d, first, at = levels[lv]
            if lv < max(levels):   # an odd end counts its last sample twice, which is the mean of what exists
                img, _ = _children_mean(img, torch.ones_like(img, dtype=torch.bool))
            out[first:first + at.numel()] = img.reshape(-1)[at]
        return [None, None, None, _filled(s["parts"], out)]
    if op == "network":
        p = torch.as_tensor(s["net"].get_params()).to("cuda", torch.float64)
        img = s["img"].to(torch.float64)
        scale = float(img.mean())
        for k in range(3):
            img = img.index_select(k, _reflected(img.shape[k], 4))
        img = img / scale
        slabs = []
        for z0 in range(0, case["z"], 16):
            slabs.append(_network(p, img[z0:min(z0 + 16, case["z"]) + 8].unsqueeze(0)).squeeze(0))
        return torch.cat(slabs) * scale
    if op == "train":
        p = torch.as_tensor(s["net"].get_params()).to("cuda", torch.float64).requires_grad_(True)
        total, count = 0.0, s["target"].numel()
        for i in range(case["tiles"]):
            d = _network(p, s["x"][i:i + 1].to(torch.float64)) - s["target"][i:i + 1].to(torch.float64)
            loss = d.square().sum() / count
            loss.backward()
            total += float(loss.detach())
        return [total, p.grad]
    parts = s["parts"].to(torch.float64) if s["parts"].dtype == torch.float32 else _as_float(s["parts"]).to(torch.float64)
    if op == "reconstruct":
        return _smoothed(s["apr"], parts)
    levels = _levels(s["apr"])
    n = s["apr"].l_max - s["apr"].l_min
    if op == "filter":
        return _filled(s["out"], _convolved(levels, parts, _stencils(s["stencil"], n)))
    psf, flipped = _stencils(s["psf"], n), _stencils(s["psf"][::-1, ::-1, ::-1], n)
    u = torch.ones_like(parts)
    for _ in range(case["iterations"]):
        u = u * _convolved(levels, parts / _convolved(levels, u, flipped), psf)
    return _filled(s["out"], u)
