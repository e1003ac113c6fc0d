"""Performance cases of the raw-development framework: what its users run,
through the entry points they call.

Families
  plain   one still through the host runtime's graph (pipe.Graph): the drop-in
          path, the node launches replayed over the resident raw, waited for
  batch   many stills of mixed sizes and CFAs in one captured batch
          (batch.Batch, graph replay)
  serve   frames and stills admitted together: a batch created, launched and
          retired, as the serving loop does for each admission
  jpg     an 8-bit rgba image on the device to the bytes of a JPEG file
  lj92    lossless-JPEG raw tiles or strips (compressed DNG) from host bytes to
          the mosaic on the device
  unpack  one bit-packed raw video frame (MLV) from host bytes to the mosaic
  mcraw   one MotionCam frame resident on the device: block offsets, decode

A case is a dict of plain values.  Images are written "WxH" + "b" (Bayer) or
"x" (X-Trans), separated by commas.
"""
import ctypes
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from vkdt_amd import batch, hip, pipe, synth, synth_gpu

DEV = "cuda"
BLACK, WHITE = 512, 16383          # 14-bit stills
FRAME_BLACK, FRAME_WHITE = 256, 4095   # 12-bit video frames


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # a preview or thumbnail source: odd extents, launches dominate
        dict(name="plain-0.7mp-odd", kind="plain", image="1001x667b", hilite=False, noise=1e-3),
        # the drop-in benchmark still
        dict(name="plain-24mp", kind="plain", image="6000x4000b", hilite=False, noise=2e-4),
        # X-Trans through the stock darkroom chain (with highlight inpainting)
        dict(name="plain-26mp-xtrans-hilite", kind="plain", image="6240x4160x", hilite=True, noise=5e-4),
        # a folder of stills from several bodies, a quarter X-Trans
        dict(name="batch-10-stills", kind="batch", hilite=False, noise=5e-4,
             images="4000x3000b,4000x3000b,4000x3000x,6000x4000b,6000x4000b,6000x4000x,6000x4000b,"
                    "8256x5504b,8256x5504x,9504x6336b"),
        # the same chain with hilite, two stills
        dict(name="batch-2-stills-hilite", kind="batch", hilite=True, noise=2e-4, images="6000x4000b,4000x3000x"),
        # one video frame served alone: latency
        dict(name="serve-1-frame", kind="serve", hilite=False, noise=4e-4, images="4096x2160b"),
        # a loaded server: frames of several streams and a still in one admission
        dict(name="serve-4-frames-1-still", kind="serve", hilite=False, noise=4e-4,
             images="4096x2160b,4096x2160b,4096x2160b,4096x2160b,6000x4000b"),
        # full-quality export of a developed still
        dict(name="jpg-24mp-444", kind="jpg", wd=6000, ht=4000, quality=95, hs=1, vs=1),
        # a web-size export
        dict(name="jpg-2mp-420", kind="jpg", wd=1620, ht=1080, quality=85, hs=2, vs=2),
        # a converter's compressed DNG
        dict(name="lj92-24mp-tiles", kind="lj92", wd=6000, ht=4000, tile_wd=256, tile_ht=256, comp=2, bits=14),
        # raw video, uncompressed
        dict(name="unpack-14bit-frame", kind="unpack", wd=3584, ht=1730, bits=14),
        # raw video, phone
        dict(name="mcraw-12mp-frame", kind="mcraw", wd=4096, ht=3072, mean=4.0),
    ]


def _size(rng, lo_mp, hi_mp):
    """an extent of lo..hi megapixels, log-uniform, with the aspect of a sensor"""
    mp = math.exp(rng.uniform(math.log(lo_mp), math.log(hi_mp)))
    aspect = rng.choice([1.0, 4 / 3, 1.5, 16 / 9])
    w = math.sqrt(mp * 1e6 * aspect)
    return max(64, int(w)), max(64, int(w / aspect) + rng.randrange(3))


def draw(rng):
    kind = rng.choice(["plain", "plain", "batch", "batch", "serve", "serve", "jpg", "jpg", "lj92", "unpack", "mcraw"])
    if kind == "plain":
        w, h = _size(rng, 0.3, 26)
        return dict(kind=kind, image=f"{w}x{h}{rng.choice('bbx')}", hilite=rng.random() < 0.4,
                    noise=math.exp(rng.uniform(math.log(1e-4), math.log(1e-3))))
    if kind in ("batch", "serve"):
        total = math.exp(rng.uniform(math.log(2), math.log(200 if kind == "batch" else 50)))
        images = []
        while total > 0.3 and len(images) < 12:
            w, h = _size(rng, 0.3, 61 if kind == "batch" else 24)
            if w * h / 1e6 > total:
                w, h = _size(rng, 0.5 * total, total)
            total -= w * h / 1e6
            images.append(f"{w}x{h}{rng.choice('bbbx')}")
        return dict(kind=kind, images=",".join(images), hilite=rng.random() < 0.3,
                    noise=math.exp(rng.uniform(math.log(1e-4), math.log(1e-3))))
    if kind == "jpg":
        w, h = _size(rng, 0.1, 45)
        quality = rng.randrange(60, 101)
        hs, vs = rng.choice([(1, 1), (2, 1), (2, 2)])
        return dict(kind=kind, wd=w, ht=h, quality=quality, hs=hs, vs=vs)
    if kind == "lj92":
        w, h = _size(rng, 1, 45)
        tw, th = rng.choice([(256, 256), (512, 512), (240, 288), (w + w % 2, 64), (w + w % 2, h)])
        return dict(kind=kind, wd=w, ht=h, tile_wd=tw, tile_ht=th, comp=rng.choice([1, 2, 2]), bits=rng.choice([12, 14, 16]))
    if kind == "unpack":
        w, h = _size(rng, 0.5, 20)
        return dict(kind=kind, wd=w, ht=h, bits=rng.choice([10, 12, 14]))
    w, h = _size(rng, 1, 48)
    return dict(kind=kind, wd=max(64, w // 64 * 64), ht=max(4, h // 4 * 4), mean=rng.uniform(2.5, 7.0))


def _images(case):
    out = []
    for s in (case["image"] if case["kind"] == "plain" else case["images"]).split(","):
        w, h = s[:-1].split("x")
        out.append((int(w), int(h), "xtrans" if s[-1] == "x" else "bayer"))
    return out


def _levels(case):
    return (FRAME_BLACK, FRAME_WHITE) if case["kind"] == "serve" else (BLACK, WHITE)


# ---------------------------------------------------------------------------
# development: state
# ---------------------------------------------------------------------------

def _graph(dng, case):
    na, nb = synth.noise_params(case["noise"], 1e-6, *_levels(case))
    g = pipe.Graph(lines=pipe.raw_graph_cfg(dng, noise_a=na, noise_b=nb, hilite=bool(case["hilite"])))
    g.export("o-pfm", os.path.join(os.path.dirname(dng), "out"))
    return g


_planned = {}


def _describe(W, H, kind, case):
    """the descriptor of a camera's planned graph: kept by a program for all
    the stills and frames of that camera"""
    key = (W, H, kind, case["noise"], bool(case["hilite"]), _levels(case))
    if key not in _planned:
        tmp = tempfile.mkdtemp(prefix="vkdt_cases_")
        dng = os.path.join(tmp, "p.dng")
        black, white = _levels(case)
        synth.write_dng(dng, np.zeros((H, W), np.uint16), kind, black=black, white=white)
        hip.init(0)
        g = _graph(dng, case)
        g.plan()
        _planned[key] = batch.describe(g)
        g.close()
        shutil.rmtree(tmp)
    d = batch.DevelopImage()
    ctypes.memmove(ctypes.byref(d), ctypes.byref(_planned[key]), ctypes.sizeof(d))
    return d


def _mosaic(W, H, kind, case, seed):
    black, white = _levels(case)
    return synth_gpu.mosaic(W, H, seed, kind, a=case["noise"], b=1e-6, black=black, white=white)[0]


class _View:
    """a graph's output buffer as __cuda_array_interface__; the buffer lies in
    the graph's arena, so a tensor made of this keeps the graph"""

    def __init__(self, graph, buf):
        assert buf.pitch == buf.wd and buf.chan == 4
        self.graph = graph
        self.__cuda_array_interface__ = {"shape": (buf.ht, buf.wd, 4), "typestr": "<f4", "data": (buf.ptr, False),
                                         "version": 2, "strides": None}


_stream = None


def _one_stream():
    """the program's stream"""
    global _stream
    if _stream is None:
        _stream = hip.Stream()
    return _stream.ptr


def _prepare_plain(case, seed):
    (W, H, kind), = _images(case)
    hip.init(0)
    cfa = _mosaic(W, H, kind, case, seed).cpu().numpy().view(np.uint16)
    tmp = tempfile.mkdtemp(prefix="vkdt_cases_")
    dng = os.path.join(tmp, "still.dng")
    synth.write_dng(dng, cfa, kind, black=BLACK, white=WHITE)
    g = _graph(dng, case)
    g.set_replay(True)
    g.run(pipe.RUN_ALL & ~pipe.RUN_DOWNLOAD)   # plan, allocate, upload, first pass
    shutil.rmtree(tmp)
    last, = [n for n in g.nodes() if n["module"] == "llap" and n["kernel"] == "colour" and not n["culled"]]
    buf = last["conns"][-1]["buf"]
    out = torch.as_tensor(_View(g, buf), device=DEV)
    assert out.data_ptr() == buf.ptr
    return dict(kind="plain", graph=g, out=out)


def _prepare_images(case, seed):
    hip.init(0)
    descs, mos, outs = [], [], []
    for i, (W, H, kind) in enumerate(_images(case)):
        d = _describe(W, H, kind, case)
        m = _mosaic(d.cfa_wd, d.cfa_ht, kind, case, seed + 1000 * i)
        o = torch.empty((d.ht, d.wd, 4), dtype=torch.float32, device=DEV)
        d.cfa, d.out = m.data_ptr(), o.data_ptr()
        descs.append(d)
        mos.append(m)
        outs.append(o)
    nbytes = batch.scratch_bytes(descs)
    scratch = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    s = dict(kind=case["kind"], descs=descs, mos=mos, outs=outs, scratch=scratch, nbytes=nbytes)
    if case["kind"] == "batch":
        s["batch"] = batch.Batch(descs, scratch.data_ptr(), nbytes)
    return s


# ---------------------------------------------------------------------------
# codecs: state
# ---------------------------------------------------------------------------

def _scene_rgba(W, H, seed):
    """an 8-bit developed image: smooth background, rectangles, fine texture
    and sensor noise, tone curved"""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = (torch.arange(W, device=DEV, dtype=torch.float32) / W)[None, :]
    y = (torch.arange(H, device=DEV, dtype=torch.float32) / H)[:, None]
    ph = rng.uniform(0, 2 * np.pi, 8)
    lum = 0.5 + 0.3 * torch.sin(2.9 * x + ph[0]) * torch.cos(2.2 * y + ph[1]) + 0.15 * (x - y)
    out = torch.empty((H, W, 4), dtype=torch.uint8, device=DEV)
    rects = [(int(rng.uniform(0, 0.8) * W), int(rng.uniform(0, 0.8) * H), int(rng.uniform(0.02, 0.2) * W),
              int(rng.uniform(0.02, 0.2) * H), rng.uniform(0.02, 0.98, 3)) for _ in range(120)]
    tex = 0.02 * torch.sin(x * (0.7 * W) + ph[2]) * torch.sin(y * (0.5 * H) + ph[3])
    for c in range(3):
        v = lum * (0.75 + 0.25 * torch.cos(1.9 * x + 1.1 * y + ph[4 + c]))
        for x0, y0, w, h, col in rects:
            v[y0:y0 + h, x0:x0 + w] = float(col[c])
        v = v + tex + 0.012 * torch.randn((H, W), device=DEV, generator=gen)
        out[..., c] = (v.clamp(0, 1) * 255 + 0.5).to(torch.uint8)
    out[..., 3] = 255
    return out


# an encoder of lossless-JPEG tiles (ITU-T T.81 process 14, predictor 1) on
# the GPU, all tiles at once: the code lengths suit sensor noise
_CODE_LEN = {0: 4, 1: 4, 2: 3, 3: 3, 4: 3, 5: 3, 6: 3, 7: 4, 8: 5, 9: 6, 10: 7, 11: 8, 12: 9, 13: 10, 14: 11, 15: 12, 16: 13}


def _lj92_tiles(mos, tw, th, comp, bits):
    """[bytes] of the row-major tiles of a mosaic (int32 H x W on the GPU),
    edge tiles padded by the last row and column"""
    H, W = mos.shape
    ntx, nty = -(-W // tw), -(-H // th)
    ys = torch.arange(nty * th, device=DEV).clamp(max=H - 1)
    xs = torch.arange(ntx * tw, device=DEV).clamp(max=W - 1)
    t = mos[ys][:, xs].reshape(nty, th, ntx, tw).permute(0, 2, 1, 3).reshape(nty * ntx, th, tw // comp, comp)
    pred = torch.empty_like(t)
    pred[:, :, 1:] = t[:, :, :-1]
    pred[:, 1:, 0] = t[:, :-1, 0]
    pred[:, 0, 0] = 1 << (bits - 1)
    d = ((t - pred + 32768) & 0xffff) - 32768
    d = d.reshape(nty * ntx, -1)
    cat = torch.zeros_like(d)
    for b in range(16):
        cat += d.abs() >= (1 << b)
    lengths = [_CODE_LEN[k] for k in range(17)]
    order = sorted(range(17), key=lambda k: (lengths[k], k))
    codes, code, prev = [0] * 17, 0, 0
    for k in order:
        code <<= lengths[k] - prev
        prev = lengths[k]
        codes[k] = code
        code += 1
    extra_len = torch.where(cat == 16, 0, cat)
    extra = torch.where(d >= 0, d, d - 1) & ((1 << extra_len) - 1)
    clen = torch.tensor(lengths, device=DEV)[cat.long()]
    val = (torch.tensor(codes, device=DEV)[cat.long()] << extra_len) | extra
    n = clen + extra_len
    end = n.cumsum(1)
    words = int((end[:, -1].max().item() + 31) // 32) + 2
    pos = end - n
    row = torch.arange(d.shape[0], device=DEV)[:, None] * words
    w, off = row + (pos >> 5), pos & 31
    both = val << (64 - 1 - off - n)       # bits off.. of a 63-bit window starting at word w
    acc = torch.zeros(d.shape[0] * words, dtype=torch.int64, device=DEV)
    acc.scatter_add_(0, w.reshape(-1), (both >> 31).reshape(-1))
    acc.scatter_add_(0, (w + 1).reshape(-1), ((both & 0x7fffffff) << 1).reshape(-1))
    sh = torch.tensor([24, 16, 8, 0], device=DEV)
    body = ((acc.reshape(d.shape[0], words)[:, :, None] >> sh) & 255).to(torch.uint8).reshape(d.shape[0], -1).cpu().numpy()
    total = end[:, -1].cpu().numpy()
    cnt = [sum(1 for k in range(17) if lengths[k] == l) for l in range(1, 17)]
    head = b"\xff\xd8\xff\xc4" + struct.pack(">HB", 2 + 1 + 16 + 17, 0) + bytes(cnt) + bytes(order)
    head += b"\xff\xc3" + struct.pack(">HBHHB", 8 + 3 * comp, bits, th, tw // comp, comp)
    head += b"".join(bytes([c, 0x11, 0]) for c in range(comp))
    head += b"\xff\xda" + struct.pack(">HB", 6 + 2 * comp, comp) + b"".join(bytes([c, 0]) for c in range(comp)) + bytes([1, 0, 0])
    out = []
    for k in range(d.shape[0]):
        nb = int(total[k] + 7) // 8
        b = body[k, :nb].copy()
        if total[k] % 8:
            b[-1] |= (1 << (8 - int(total[k]) % 8)) - 1
        out.append(head + b.tobytes().replace(b"\xff", b"\xff\0") + b"\xff\xd9")
    return out


def _prepare_lj92(case, seed):
    hip.init(0)
    W, H, tw, th, bits = (case[k] for k in ("wd", "ht", "tile_wd", "tile_ht", "bits"))
    comp = case["comp"] if tw % case["comp"] == 0 else 1
    m = synth_gpu.mosaic(W, H, seed, "bayer", black=2 ** bits // 32, white=min(2 ** bits - 1, 32767))[0].to(torch.int32)
    blob, tiles = hip.lj92_tiles(_lj92_tiles(m, tw, th, comp, bits), tw, th, W, H)
    out = torch.empty((H, W), dtype=torch.int16, device=DEV)
    return dict(kind="lj92", blob=blob, tiles=tiles, out=out, images=[(out.data_ptr(), W, H, W)])


def _prepare_unpack(case, seed):
    hip.init(0)
    W, H, bits = case["wd"], case["ht"], case["bits"]
    m = synth_gpu.mosaic(W, H, seed, "bayer", black=2 ** bits // 16, white=2 ** bits - 1)[0].reshape(-1).to(torch.int64)
    n = m.numel()
    pad = -n % 16
    m = torch.cat([m, m.new_zeros(pad)]).reshape(-1, 16)
    sh = torch.arange(bits - 1, -1, -1, device=DEV)
    bitrow = ((m[:, :, None] >> sh) & 1).reshape(-1, 16)      # 16 samples are `bits` 16-bit words
    w = (bitrow << torch.arange(15, -1, -1, device=DEV)).sum(1).cpu().numpy().astype("<u2")
    out = torch.empty((H, W), dtype=torch.int16, device=DEV)
    return dict(kind="unpack", packed=w.tobytes(), n=n, bits=bits, out=out)


_MC_BYTES = np.array([0, 8, 16, 24, 32, 40, 48, 64, 64, 80, 80, 128, 128, 128, 128, 128])


def _prepare_mcraw(case, seed):
    """counts as a sensor's noise gives them: brighter parts of the frame
    carry more bits, with a spread from block to block"""
    hip.init(0)
    W, H = case["wd"], case["ht"]
    nb = W * H // 64
    rblock = -(-nb // 64) * 64
    rng = np.random.default_rng(seed)
    k = np.arange(nb) // 4
    bx, by = k % (W // 64) / (W // 64), k // (W // 64) / (H // 4)
    smooth = case["mean"] + 1.5 * np.sin(5 * bx + rng.uniform(0, 6)) * np.cos(4 * by + rng.uniform(0, 6))
    cnt = np.zeros(rblock, np.int64)
    cnt[:nb] = np.clip(np.rint(smooth + rng.normal(0, 0.7, nb)), 0, 10)
    cnt = np.where(cnt == 7, 8, np.where(cnt == 9, 10, cnt))
    refs = np.zeros(rblock, np.uint16)
    refs[:nb] = rng.integers(64, 4096, nb)
    size = int(_MC_BYTES[cnt[:nb]].sum())
    cnt8 = cnt.astype(np.uint8)
    t = dict(bits=torch.from_numpy(cnt8[0::2] | (cnt8[1::2] << 4)).to(DEV), ref=torch.from_numpy(refs.view(np.int16)).to(DEV),
             data=torch.from_numpy(rng.integers(0, 256, max(size, 1), dtype=np.uint8)).to(DEV),
             off=torch.empty(rblock, dtype=torch.int32, device=DEV),
             scr=torch.empty((rblock + 511) // 512 + 1, 4, dtype=torch.int32, device=DEV),
             out=torch.empty((H, W), dtype=torch.int16, device=DEV))

    def buf(x, wd, ht, fmt):
        return hip.Buf(x.data_ptr(), wd, ht, wd, 1, fmt, 1, x.numel() * x.element_size())

    b = buf(t["bits"], t["bits"].numel(), 1, hip.FMT_UI8)
    off = buf(t["off"], rblock, 1, hip.FMT_UI32)
    scr = buf(t["scr"], t["scr"].shape[0], 4, hip.FMT_UI32)
    ref = buf(t["ref"], rblock, 1, hip.FMT_UI16)
    dat = buf(t["data"], t["data"].numel(), 1, hip.FMT_UI8)
    out = buf(t["out"], W, H, hip.FMT_UI16)
    pc = np.array([0, 0, W, H], np.int32)
    tok = hip.token
    # the node launches as the graph runtime issues them
    calls = [(tok("i-mcraw"), tok("prefix"), None, 0, None, 0, (hip.Buf * 3)(b, off, scr), 3, (nb + 511) // 512 * 8, 1, 1, None),
             (tok("i-mcraw"), tok("decode"), pc.ctypes.data, pc.nbytes, None, 0, (hip.Buf * 5)(out, b, off, ref, dat), 5,
              nb * 8, 1, 1, None)]
    return dict(kind="mcraw", calls=calls, keep=(t, pc), nb=nb, off=t["off"], out=t["out"])


def prepare(case, seed):
    k = case["kind"]
    if k == "plain":
        return _prepare_plain(case, seed)
    if k in ("batch", "serve"):
        return _prepare_images(case, seed)
    if k == "jpg":
        hip.init(0)
        # the file is written into the program's own buffer, at most 3 bytes a pixel
        return dict(kind=k, rgba=_scene_rgba(case["wd"], case["ht"], seed), case=case, ptr=ctypes.c_void_p(),
                    len=ctypes.c_size_t(), file=np.zeros(case["wd"] * case["ht"] * 3 + 4096, np.uint8))
    return dict(lj92=_prepare_lj92, unpack=_prepare_unpack, mcraw=_prepare_mcraw)[k](case, seed)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    k = state["kind"]
    if k == "plain":
        state["graph"].run(pipe.RUN_RECORD | pipe.RUN_WAIT)
        return state["out"]
    if k == "batch":
        state["batch"].run(_one_stream(), graph=True)
        return state["outs"]
    if k == "serve":
        b = batch.Batch(state["descs"], state["scratch"].data_ptr(), state["nbytes"])
        b.run(_one_stream())
        hip.sync(_one_stream())
        b.close()
        return state["outs"]
    if k == "jpg":
        c, p, n = state["case"], state["ptr"], state["len"]
        hip.check(hip.lib().vkdt_hip_jpg_encode(state["rgba"].data_ptr(), c["wd"], c["ht"], c["wd"], c["quality"], c["hs"], c["vs"],
                                                ctypes.byref(p), ctypes.byref(n), None), "jpg encode")
        assert n.value <= state["file"].nbytes
        ctypes.memmove(state["file"].ctypes.data, p, n.value)
        hip.lib().vkdt_jpg_free(p)
        return n.value, state["file"]
    if k == "lj92":
        hip.lj92_decode(state["blob"], state["tiles"], state["images"])
        return state["out"]
    if k == "unpack":
        hip.unpack_msb16(state["packed"], state["out"].data_ptr(), state["n"], state["bits"])
        return state["out"]
    for c in state["calls"]:
        hip.check(hip.lib().vkdt_hip_node_launch(*c), "i-mcraw")
    return state["off"][:state["nb"]], state["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    k = case["kind"]
    if k in ("plain", "batch", "serve"):
        # the mosaic read, the rgba f32 image written; FP32 operations per
        # site as the graph's kernels write them: covariances, taps, curves
        px = sum(w * h for w, h, _ in _images(case))
        return {"bytes": 18 * px, "flops": 1500 * px}
    px = case["wd"] * case["ht"]
    if k == "jpg":      # rgba in, about 3 bits a pixel out; a separable 8x8 DCT per component
        return {"bytes": 4 * px + px * 3 // 8, "flops": 3 * 16 * px}
    if k == "lj92":     # the compressed bits (about 0.55 of the raw ones) and the mosaic
        return {"bytes": int(0.55 * case["bits"] / 8 * px) + 2 * px, "flops": 0}
    if k == "unpack":
        return {"bytes": px * case["bits"] // 8 + 2 * px, "flops": 0}
    # mcraw: data at `mean` bits a sample, counts, references and offsets, the mosaic
    return {"bytes": int(px * case["mean"] / 8) + px // 64 * 13 // 2 + 2 * px, "flops": 0}


def tolerance(case):
    """Codecs are integer: exact.  A development stores binary16 between its
    nodes and branches on nearly equal float32 values (the choice between two
    covariances, hot pixels, axis snaps), so another correct float32
    evaluation differs by a binary16 step here and there and at isolated
    pixels visibly: contracting the products and sums into FMAs moves these
    images by 1.5e-4 to 1.1e-3, all of them are 0.6e-3 to 3e-3 off float64."""
    if case["kind"] in ("plain", "batch", "serve"):
        return {"rel": 2e-3, "max": 0.9}
    return "exact"


# ---------------------------------------------------------------------------
# the development in float64, without intermediate rounding
# ---------------------------------------------------------------------------

F64 = torch.float64


def _mirror(i, n):
    t = torch.remainder(i, 2 * n)
    return torch.where(t < n, t, 2 * n - 1 - t)


def _ar(n, lo=0):
    return torch.arange(lo, lo + n, device=DEV)


def _pad(img, r):
    """img (.., H, W) with r mirrored rows and columns around it"""
    H, W = img.shape[-2:]
    return img.index_select(-2, _mirror(_ar(H + 2 * r, -r), H)).index_select(-1, _mirror(_ar(W + 2 * r, -r), W))


def _clamp(x, a, b):
    """GLSL clamp: NaN goes to the lower bound"""
    return torch.fmin(torch.fmax(x, torch.tensor(a, dtype=F64, device=DEV)), torch.tensor(b, dtype=F64, device=DEV))


def _smooth(e0, e1, x):
    t = _clamp((x - e0) / (e1 - e0), 0.0, 1.0)
    return t * t * (3 - 2 * t)


LUM = (2.62700212e-01, 6.77998072e-01, 5.93017165e-02)


def _lum(c):
    return LUM[0] * c[0] + LUM[1] * c[1] + LUM[2] * c[2]


def _at(x, y, pat):
    """CFA colour per site for the coordinates y (column) and x (row) vectors"""
    if pat == "bayer":
        return (y & 1)[:, None] + (x & 1)[None, :]
    tx, ty = torch.div(x, 3, rounding_mode="trunc"), torch.div(y, 3, rounding_mode="trunc")
    mx, my = x - 3 * tx, y - 3 * ty
    top = ((tx[None, :] + ty[:, None]) & 1) > 0
    green = ((mx[None, :] + my[:, None]) & 1) == 0
    blue = top ^ (my == 1)[:, None].expand_as(top)
    return torch.where(green, 1, torch.where(blue, 2, 0))


def _evd(a, b, c):
    """eigenvalues and major axis of the symmetric [[a, b], [b, c]]"""
    ph = -0.5 * (a + c)
    root = torch.sqrt((ph * ph - (a * c - b * b)).clamp(min=0))
    e0, e1 = -ph + root, -ph - root
    a0, c0 = a - e0, c - e0
    s0, s1 = a0 * a0 + b * b, b * b + c0 * c0
    pick = s0 > s1
    vx, vy, sl = torch.where(pick, a0, b), torch.where(pick, b, c0), torch.where(pick, s0, s1)
    vx = torch.where(sl == 0, torch.ones_like(vx), vx)
    sl = torch.where(sl == 0, torch.ones_like(sl), sl)
    vx, vy = vx / sl.sqrt(), vy / sl.sqrt()
    return e0, e1, vy, -vx          # minor axis (vx, vy), major axis its perpendicular


def _tensor(taps, offs):
    """the covariance of smaller determinant of two weightings (p, 1/p for
    the means, p^2 and 1/p^2 for the moments) over the taps"""
    best = None
    for mw, sw in ((lambda p: p, lambda p: p * p), (lambda p: 1 / p, lambda p: 1 / (p * p))):
        s = mx = my = 0
        for p, (i, j) in zip(taps, offs):
            w = mw(p)
            s, mx, my = s + w, mx + i * w, my + j * w
        mx, my = mx / s, my / s
        s = xx = xy = yy = 0
        for p, (i, j) in zip(taps, offs):
            w, dx, dy = sw(p), i - mx, j - my
            s, xx, xy, yy = s + w, xx + w * dx * dx, xy + w * dx * dy, yy + w * dy * dy
        cur = (xx / s, xy / s, yy / s)
        if best is None:
            best = cur
        else:
            det = lambda m: m[0] * m[2] - m[1] * m[1]
            use = det(best) < det(cur)
            best = tuple(torch.where(use, u, v) for u, v in zip(best, cur))
    return _evd(*best)


class _Dev:
    """one image's parameters and stages"""

    def __init__(self, d, raw):
        self.d = d
        self.xt = d.filters == 9
        self.b = 3 if self.xt else 2
        self.pat = "xtrans" if self.xt else "bayer"
        self.raw = (raw.to(torch.int32) & 0xffff).to(F64) / 65535.0
        code = lambda v: round(v * 65535.0) / 65535.0     # the UNORM16 level the float32 stands for
        self.black, self.white = [code(v) for v in d.black], [code(v) for v in d.white]
        self.W, self.H = d.wd, d.ht
        e = list(d.dn_params)[4:8]
        self.edge = [2.0 ** (12 * e[k] + e[3]) for k in range(3)]
        self.bs = 2.23607 if self.xt else 1.414213

    def sigma(self, v, ch=1):
        inv = 1.0 / (self.white[ch] - self.black[ch])
        s = torch.sqrt(self.d.noise_a + torch.clamp((v - self.black[ch]) * inv, min=0) * self.d.noise_b)
        return [_clamp(self.edge[k] * s, 1e-3, 1e3) for k in range(3)]

    def blocks(self, m):
        """sites (i, j) of the blocks: a function of column and row offset"""
        b = self.b
        return lambda i, j: m[j::b, i::b][:self.H // b, :self.W // b]

    def half(self, m, white, hilite=False):
        at = self.blocks(m)
        if not self.xt:
            gx, gz = at(0, 1), at(1, 0)
            gx = torch.where(gx >= white, gz, gx)
            gz = torch.where(gz >= white, gx, gz)
            return torch.stack([at(0, 0), (gx + gz) / 2, at(1, 1)])
        c = [at(i, j) for i in range(3) for j in range(3)]
        if hilite:
            for a, b in ((1, 7), (7, 1), (3, 5), (5, 3)):
                c[a] = torch.where(c[a] >= white, c[b], c[a])
            top = torch.stack([c[k] for k in (0, 2, 4, 6, 8)]).amax(0) >= white
            for k in (0, 2, 4, 6, 8):
                c[k] = torch.where(top, torch.ones_like(c[k]), c[k])
        p, q = (c[1] + c[7]) / 2, (c[3] + c[5]) / 2
        odd = ((_ar(p.shape[1])[None, :] + _ar(p.shape[0])[:, None]) & 1) == 1
        return torch.stack([torch.where(odd, p, q), (c[0] + c[2] + c[4] + c[6] + c[8]) / 5, torch.where(odd, q, p)])

    @staticmethod
    def polyphase(img):
        """texel x stored at x/2 + (x & 1) (n + 1)/2"""
        H, W = img.shape[-2:]
        oy, ox = torch.cat([_ar(H)[0::2], _ar(H)[1::2]]), torch.cat([_ar(W)[0::2], _ar(W)[1::2]])
        return img.index_select(-2, oy).index_select(-1, ox)

    def downcov(self, half):
        H, W = half.shape[-2:]
        p = _pad(half, 2)
        win = lambda k, i, j: p[k][j:j + H, i:i + W]
        offs = [(i - 2, j - 2) for j in range(5) for i in range(5)]
        lum = _lum(p)
        taps = [lum[j + 2:j + 2 + H, i + 2:i + 2 + W] for i, j in offs]
        e0, e1, ax, ay = _tensor(taps, offs)
        hot = 2 * sum(taps) / 25
        e0, e1 = _clamp(e0, 0.01, 25.0), _clamp(0.05 * e1, 0.01, 25.0)
        acc, wt = [0, 0, 0], 0
        for i, j in offs:
            u, v = i * ax + j * ay, i * -ay + j * ax
            w = torch.clamp(torch.exp(-0.5 * (u * u / e0 + v * v / e1)), min=1e-9)
            w = torch.where(win(0, i + 2, j + 2) > hot, torch.zeros_like(w), w)
            wt = wt + w
            for k in range(3):
                acc[k] = acc[k] + w * win(k, i + 2, j + 2)
        return self.polyphase(torch.stack(acc) / wt.clamp(min=1e-8))

    def down(self, img, level):
        H, W = img.shape[-2:]
        p = _pad(img, 2)
        win = lambda i, j: p[:, j + 2:j + 2 + H, i + 2:i + 2 + W]
        g = lambda f: torch.where(f < 0, f, f.clamp(min=0) ** 0.8)
        sc = 0.7 ** level / self.bs
        hw = torch.stack([0.5 / (sc * s) for s in self.sigma(img[0])])
        acc, wt = 0.2 * img, torch.full_like(img, 0.2)
        for ox, oy, a, c in ((1, 0, .2, .4), (-2, -1, .8, .6), (0, -2, .4, .8), (-1, 1, .6, .2)):
            t = (win(ox, oy) * (1 - a) + win(ox + 1, oy) * a) * (1 - c) + (win(ox, oy + 1) * (1 - a) + win(ox + 1, oy + 1) * a) * c
            w = _clamp(1 - hw * (g(t) - g(img)).abs(), 0.0, 1.0) * 0.2
            acc, wt = acc + w * t, wt + w
        return self.polyphase(acc / wt)

    def assemble(self, lev):
        H, W = lev[0].shape[-2:]
        down, py, px = [lev[0]], _ar(H), _ar(W)
        for l in range(4):
            py, px = py // 2 + (py & 1) * ((H + 1) // 2), px // 2 + (px & 1) * ((W + 1) // 2)
            down.append(lev[l + 1].index_select(-2, py).index_select(-1, px))
        sig = torch.stack(self.sigma(down[2][0].clamp(min=0)))
        bl = [0.7 ** (l + 1) / self.bs for l in range(4)]
        d = [(down[l] - down[l + 1]) / (sig * bl[l]) for l in range(4)]
        n = [(x * x).sum(0).sqrt() for x in d]
        slope = ((n[3] - n[0]) / 3 + (n[2] - n[1]) + (n[1] - n[0]) + (n[3] - n[2]) + (n[2] - n[0]) / 2 + (n[3] - n[1]) / 2) / 6
        test = _clamp(1.5 * (1 - (-slope).clamp(min=0)).clamp(min=0) ** 16, 0.0, 1.0)
        out = down[4]
        for l in range(3, -1, -1):
            t = torch.where(d[l][0].abs() > 10, 10000.0, self.d.dn_params[0] ** 4)
            ad = d[l].abs()
            m = (ad / (2 * t)).clamp(max=1)
            out = out + sig * bl[l] * torch.sign(d[l]) * ((ad - t).clamp(min=0) * (1 - m) + ad * m)
        to_yuv = (np.array([[.299, .587, .114], [-.147, -.289, .436], [.615, -.515, -.1]]) @
                  np.array([[1.66022677, -0.58754761, -0.07283825], [-0.12455334, 1.13292605, -0.00834963],
                            [-0.01815514, -0.10060303, 1.11899817]]))
        to_rgb = (np.array([[0.62750375, 0.32927542, 0.04330266], [0.06910828, 0.91951916, 0.0113596],
                            [0.01639406, 0.08801125, 0.89538035]]) @
                  np.array([[1.0, -3.94570707e-05, 1.13982797], [1.0, -3.94610164e-01, -5.80500316e-01],
                            [1.0, 2.03199968, -4.81376263e-04]]))
        mul = lambda m, v: [m[j][0] * v[0] + m[j][1] * v[1] + m[j][2] * v[2] for j in range(3)]
        norm = lambda v: [(v[k] - self.black[k]) / (self.white[k] - self.black[k]) * self.d.wb[k] for k in range(3)]
        yuv, y0 = mul(to_yuv, norm(out)), mul(to_yuv, norm(down[0]))[0]
        yuv[0] = y0 * (1 - self.d.dn_params[1]) + yuv[0] * self.d.dn_params[1]
        rgb = mul(to_rgb, yuv)
        return torch.stack([rgb[k] / self.d.wb[k] * (self.white[k] - self.black[k]) + self.black[k] for k in range(3)]), test

    def upsample(self, img):
        """bilinear lookup of (C, h, w) at the centres of the W x H mosaic"""
        def axis(n, full):
            s = (_ar(full).to(F64) + 0.5) / full * n - 0.5
            f = s.floor()
            return _mirror(f.long(), n), _mirror(f.long() + 1, n), s - f
        h, w = img.shape[-2:]
        y0, y1, fy = axis(h, self.H)
        x0, x1, fx = axis(w, self.W)
        r = img.index_select(-1, x0) * (1 - fx) + img.index_select(-1, x1) * fx
        return r.index_select(-2, y0) * (1 - fy)[:, None] + r.index_select(-2, y1) * fy[:, None]

    def doub(self, asm, test, half):
        col = _at(_ar(self.W), _ar(self.H), self.pat)
        pick = lambda t: torch.where(col == 0, t[0], torch.where(col == 1, t[1], t[2]))
        crs, crs1 = pick(self.upsample(asm)), pick(self.upsample(half))
        up = self.upsample(test[None])[0]
        val = self.raw[:self.H, :self.W]
        T, luma, detail = 0.5 * self.d.dn_params[0] * up, self.d.dn_params[1], self.d.dn_params[2]
        if self.xt:
            T = torch.where(col == 1, T, T / up.clamp(min=1e-4))
        blend = 0.5 * (torch.where(col == 1, luma, 1.0) + 1)
        lev = lambda v: pick([torch.full_like(val, v[k]) for k in range(3)])
        black, white = lev(self.black), lev(self.white)
        s = torch.sqrt(self.d.noise_a + torch.clamp((crs - black) / (white - black), min=0) * self.d.noise_b)
        sig = [_clamp(self.edge[k] * s, 1e-3, 1e3) for k in range(3)]
        wav = (val - crs1) / (sig[0] + sig[2]).clamp(min=1e-8)
        tt = (wav / (2 * T).clamp(min=1e-8)).clamp(max=1)
        uw = 1 - (1 - up.clamp(max=1) ** 4) * detail
        aw = wav.abs()
        den = (crs + sig[1] * torch.sign(wav) * ((aw - T).clamp(min=0) * (1 - tt) + aw * tt)).clamp(min=0)
        f = uw * blend
        val = torch.where(val < white, val * (1 - f) + den * f, val)
        return ((val - black) / (white - black)).clamp(min=0)

    def hilite(self, m):
        white, desat, soft = list(self.d.hl_params)
        wb = list(self.d.hl_wb)[:3]
        if not sum(v * v for v in wb) > 1e-3:
            wb = [1.0] * 3
        pos, ds = (white if white > 0 else 1.0), desat * desat
        w5, s5 = [.0625, .25, .375, .25, .0625], [1, 2, 0, -2, -1]
        fine = [(self.half(m, white, True), None)]
        for _ in range(self.d.hl_levels):
            t = fine[-1][0]
            h, w = t.shape[-2:]
            cw = [t[k] * wb[k] for k in range(3)]
            hi, lo = torch.maximum(torch.maximum(cw[0], cw[1]), cw[2]), torch.minimum(torch.minimum(cw[0], cw[1]), cw[2])
            s = _smooth(0.2, 1.0, t.amax(0) / pos)
            tt = _clamp(5 * ds * ds * s * _smooth(0.15, 0.9, (hi - lo) / hi.clamp(min=1e-3)), 0.0, 1.0)
            ok = (t < pos).all(0).to(F64)
            prep = torch.stack([(t[k] * (1 - tt) + (hi + lo) / wb[k] * 0.5 * tt) * ok for k in range(3)] + [ok, _lum(t)])
            p = _pad(prep, 2)
            oh, ow = (h - 1) // 2 + 1, (w - 1) // 2 + 1
            acc, ex, ey = 0, 0, 0
            for j in range(5):
                for i in range(5):
                    q = p[:, j:j + 2 * oh - 1:2, i:i + 2 * ow - 1:2]
                    acc = acc + w5[i] * w5[j] * q[:4]
                    ex, ey = ex + w5[j] * s5[i] * q[4], ey + w5[i] * s5[j] * q[4]
            mean = torch.where(acc[3] == 0, torch.ones_like(acc[:3]), acc[:3] / torch.where(acc[3] == 0, 1.0, acc[3]))
            fine.append((mean, torch.sqrt(ex * ex + ey * ey)))

        def scale(up, v):
            s = [v[k] / up[k].clamp(min=0.001) for k in range(3)]
            w = [torch.exp(up[k] - torch.maximum(up[(k + 1) % 3], up[(k + 2) % 3])) for k in range(3)]
            return sum(a * b for a, b in zip(s, w)) / sum(w)

        def expand(c, h, w):
            def axis(c, n, dim):
                m, i = c.shape[dim], _ar(n)
                at = lambda o: c.index_select(dim, _mirror(i // 2 + o, m))
                odd = (i & 1) == 1
                odd = odd[:, None] if dim == -2 else odd
                return torch.where(odd, (at(0) + at(1)) / 2, (at(-1) + 6 * at(0) + at(1)) / 8)
            return axis(axis(c, w, -1), h, -2)

        crs = fine[-1][0]
        for t, edge in reversed(fine[:-1]):
            up = expand(crs, *t.shape[-2:])
            r = (up * scale(up, t)).clamp(-65535, 65535)
            # the finest level carries alpha 1, the coarser ones their edge term
            e = torch.ones_like(t[0]) if edge is None else edge
            k = torch.where((t >= white).any(0), 1.0, soft)
            k = _clamp(k * (1 - e.clamp(min=0).sqrt()) + e.clamp(min=0).sqrt(), 0.0, 1.0)
            crs = t * (1 - k) + r * k
        out = m.clone()
        at, put = self.blocks(m), self.blocks(out)
        sw = 0.97 * white
        if not self.xt:
            r, g1, g0, b = at(0, 0), at(1, 0), at(0, 1), at(1, 1)
            sc = scale(crs, [r, torch.minimum(g0, g1), b])
            t = _smooth(sw, white, torch.stack([r, g0, g1, b]).amax(0))
            for (i, j), v, k in (((0, 0), r, 0), ((1, 0), g1, 1), ((0, 1), g0, 1), ((1, 1), b, 2)):
                put(i, j).copy_(v * (1 - t) + sc * crs[k] * t)
            return out
        c = [at(i, j) for i in range(3) for j in range(3)]
        even = ((_ar(crs.shape[2])[None, :] + _ar(crs.shape[1])[:, None]) & 1) == 0
        up = [torch.where(even, crs[2], crs[0]), crs[1], torch.where(even, crs[0], crs[2])]
        g = torch.stack([c[k] for k in (0, 2, 4, 6, 8)])
        sc = scale(up, [torch.minimum(c[1], c[7]), g.amin(0), torch.minimum(c[3], c[5])])
        top = torch.stack(c).amax(0)
        t, tg = _smooth(sw, white, top), torch.where(top > sw, _smooth(sw, white, g.amin(0)), 0.0)
        for k in range(9):
            src, f = (up[1], tg) if k % 2 == 0 else (up[0] if k in (1, 7) else up[2], t)
            put(k // 3, k % 3).copy_(c[k] * (1 - f) + src * sc * f)
        return out

    def gauss(self, m):
        b, n0 = self.b, 0 if self.xt else -1
        offs = [(i, j) for j in range(n0, 3) for i in range(n0, 3) if ((i + j) & 1) == (0 if self.xt else 1)]
        qh, qw = self.H // b, self.W // b
        at = lambda i, j: m.index_select(0, _mirror(b * _ar(qh) + j, self.H)).index_select(1, _mirror(b * _ar(qw) + i, self.W))
        e0, e1, ax, ay = _tensor([at(i, j) for i, j in offs], offs)
        one, zero = torch.ones_like(ax), torch.zeros_like(ax)
        if not self.xt:
            horiz = ax.abs() > ay.abs()
            return torch.stack([0.2 * e0, 0.2 * e1, torch.where(horiz, one, zero), torch.where(horiz, zero, one)])
        hor, ver = ax.abs() > 2 * ay.abs(), ay.abs() > 2 * ax.abs()
        none = ~(hor | ver)
        e0, e1 = torch.where(none, 0.1, 0.4 * e0), torch.where(none, 0.1, 0.4 * e1)
        return torch.stack([e0, e1, torch.where(hor, one, torch.where(ver, zero, ax)),
                            torch.where(hor, zero, torch.where(ver, one, ay))])

    def cov_at(self, cov, add):
        """the block covariance at (x + add) / block, zero outside"""
        p = torch.nn.functional.pad(cov, (0, 1, 0, 1))
        y = ((_ar(self.H) + add) // self.b).clamp(max=cov.shape[1])
        x = ((_ar(self.W) + add) // self.b).clamp(max=cov.shape[2])
        return p.index_select(1, y).index_select(2, x)

    @staticmethod
    def weight(cov, e0, e1, i, j, lo):
        u, v = cov[2] * i + cov[3] * j, -cov[3] * i + cov[2] * j
        return _clamp(torch.exp(-0.5 * (u * u / e0 + v * v / e1)), lo, 1.0)

    def splat(self, m, cov):
        c = self.cov_at(cov, 0 if self.xt else 1)
        e0, e1 = _clamp(c[0], 0.01, 25.0), _clamp(c[1], 0.01, 25.0)
        r = 2 if self.xt else 1
        acc = wt = 0
        for j in range(-r, r + 1):
            for i in range(-r, r + 1):
                x, y = _ar(self.W) + i, _ar(self.H) + j
                green = _at(x + 6, y + 6, self.pat) == 1
                wrap = lambda v, n: torch.where(v < 0, v + 6, torch.where(v >= n, v - 6, v))
                col = m.index_select(0, wrap(y, self.H)).index_select(1, wrap(x, self.W))
                w = torch.full_like(col, 666.0) if i == j == 0 else self.weight(c, e0, e1, i, j, 1e-4)
                w = torch.where(green, w, 0.0)
                acc, wt = acc + col * w, wt + w
        return acc / wt.clamp(min=1e-8)

    def fix(self, m, green, cov):
        c = self.cov_at(cov, 1)
        hi, sc, r = (10.0, 3.0, 2) if self.xt else (49.0, 2.0, 1)
        e0, e1 = sc * _clamp(c[0], 1.0, hi), sc * _clamp(c[1], 1.0, hi)
        num, den = [0, 0, 0], [0, 0, 0]
        for j in range(-r, r + 1):
            for i in range(-r, r + 1):
                x, y = _ar(self.W) + i, _ar(self.H) + j
                k = _at(x, y, self.pat) if self.xt else torch.where(
                    ((x[None, :] + y[:, None]) & 1) == 1, 1, torch.where((x & 1) == 0, 0, 2)[None, :].expand(self.H, -1))
                at = lambda t: t.index_select(0, _mirror(y, self.H)).index_select(1, _mirror(x, self.W))
                w = self.weight(c, e0, e1, i, j, 1e-3)
                v = at(m) * (1e-4 + green) / (1e-4 + at(green)) * w
                for q in (0, 2):
                    num[q] = num[q] + torch.where(k == q, v, 0.0)
                    den[q] = den[q] + torch.where(k == q, w, 0.0)
        return torch.stack([num[0] / den[0].clamp(min=1e-8), green, num[2] / den[2].clamp(min=1e-8)])

    def colour(self, c):
        p = np.array(self.d.co_params)
        cam = p[4:16].reshape(3, 4)[:, :3].T
        cat = np.array([[0.401288, 0.650173, -0.051461], [-0.250268, 1.204414, 0.045854], [-0.002079, 0.048952, 0.953127]])
        cati = np.array([[1.86206786, -1.01125463, 0.14918677], [0.38752654, 0.62144744, -0.00897398],
                         [-0.01584150, -0.03412294, 1.04996444]])
        r2x = np.array([[0.636958048301290991, 0.144616903586208406, 0.168880975164172054],
                        [0.26270021201126692, 0.677998071518871148, 0.0593017164698619384],
                        [4.9999999999999999e-17, 0.0280726930490874452, 1.06098505771079066]])
        x2r = np.array([[1.71665119, -0.35567078, -0.25336628], [-0.66668435, 1.61648124, 0.01576855],
                        [0.01763986, -0.04277061, 0.94210312]])
        to = cat @ r2x
        ratio = (to @ p[0:3]) / to.sum(1)
        m = (x2r @ cati) @ np.diag(ratio) @ to @ cam * p[3]
        return torch.stack([(m[j][0] * c[0] + m[j][1] * c[1] + m[j][2] * c[2]).clamp(-65535, 65535) for j in range(3)])

    def filmcurv(self, c):
        light, contrast, bias = list(self.d.fc_params)[:3]
        il, k = max(5e-3, light), max(1e-4, contrast)
        c = c + bias
        o = 1 - torch.exp(-(c.clamp(min=1e-7) * il) ** k)
        # the hue of the input: the middle channel of the output follows the
        # middle channel's place between the input's extremes
        lo, hi = c.argmin(0), c.argmax(0)
        mid = 3 - lo - hi
        get = lambda t, i: t.gather(0, i[None])[0]
        same = lo == hi
        mid = torch.where(same, torch.ones_like(mid), mid)
        f = (get(c, mid) - get(c, lo) + 1e-6) / (get(c, hi) - get(c, lo) + 1e-6)
        v = get(o, lo) * (1 - f) + get(o, hi) * f
        return o.scatter(0, mid[None], torch.where(same, get(o, mid), v)[None])

    def llap(self, c):
        sigma, shadows, highlights, clarity = list(self.d.ll_params)
        G, nl = self.d.ll_numgamma, self.d.ll_levels
        lum = _lum(c.clamp(-1000, 1000))
        gam = [i / (G - 1) for i in range(G)]

        def curve(x, g):
            v = x - g
            s, sh = torch.where(v > 0, sigma, -sigma), torch.where(v > 0, shadows, highlights)
            t = _clamp(v.abs() / (2 * sigma), 0.0, 1.0)
            near = g + s * 2 * (1 - t) * t + t * t * (s + s * sh)
            out = torch.where(v.abs() > 2 * sigma, g + s + sh * (v - s), near)
            return out + clarity * v * torch.exp(-v * v * 3 / (2 * sigma * sigma))

        def reduce(p):
            def axis(p, dim):
                n = p.shape[dim]
                i = 2 * _ar((n - 1) // 2 + 1)
                at = lambda o: p.index_select(dim, _mirror(i + o, n))
                return (at(-1) + 2 * at(0) + at(1)) / 4
            return axis(axis(p, -1), -2)

        def expand(p, h, w):
            def axis(p, n, dim):
                m, i = p.shape[dim], _ar(n)
                at = lambda o: p.index_select(dim, _mirror(i // 2 + o, m))
                odd = ((i & 1) == 1)[:, None] if dim == -2 else (i & 1) == 1
                even = at(-2) / 2 + at(-1) / 2 + at(0) + at(1) / 2 + at(2) / 2
                return torch.where(odd, at(-1) + at(0) / 2 + at(1) / 2 + at(2), even) / 3
            return axis(axis(p, w, -1), h, -2)

        # per curve: its pyramid, and what each level takes from it
        pyr = [lum]
        for _ in range(1, nl):
            pyr.append(reduce(pyr[-1]))
        place = []
        for v in pyr[:-1]:
            hi = torch.ones_like(v, dtype=torch.long)
            for i in range(1, G - 1):
                hi += v >= gam[i]
            g = torch.tensor(gam, dtype=F64, device=DEV)
            place.append((hi, _clamp((v - g[hi - 1]) / (g[hi] - g[hi - 1]), 0.0, 1.0)))
        detail = [torch.zeros_like(v) for v in pyr[:-1]]
        for i in range(G):
            p = curve(lum, gam[i])
            for l in range(nl - 1):
                q = reduce(p)
                hi, al = place[l]
                w = torch.where(hi - 1 == i, 1 - al, torch.where(hi == i, al, 0.0))
                detail[l] += w * (p - expand(q, *p.shape[-2:]))
                p = q
        out = pyr[-1]
        for l in range(nl - 2, -1, -1):
            out = expand(out, *detail[l].shape[-2:]) + detail[l]
        old = _lum(c).clamp(min=1e-8)
        new = torch.where(out < old, old * torch.exp(out - old), out)
        rgb = (c * (new / old)).clamp(min=0)
        return torch.cat([rgb, torch.ones_like(rgb[:1])]).permute(1, 2, 0).contiguous()

    def develop(self):
        half = self.half(self.raw, self.white[1])
        lev = [half, self.downcov(half)]
        for l in range(1, 4):
            lev.append(self.down(lev[-1], l))
        asm, test = self.assemble(lev)
        del lev
        m = self.doub(asm, test, half)
        del asm, test, half
        if self.d.hl_on:
            m = self.hilite(m)
        cov = self.gauss(m)
        c = self.fix(m, self.splat(m, cov), cov)
        del m, cov
        return self.llap(self.filmcurv(self.colour(c)))


def exact(case, seed):
    """What a development returns, in float64 from the raw and the graph's
    parameters; None for the codecs, whose outputs are whole numbers."""
    if case["kind"] not in ("plain", "batch", "serve"):
        return None
    outs = []
    for i, (W, H, kind) in enumerate(_images(case)):
        d = _describe(W, H, kind, case)
        if case["kind"] == "plain":      # the loader cuts the mosaic to whole blocks
            raw = _mosaic(W, H, kind, case, seed)[:d.cfa_ht, :d.cfa_wd]
        else:
            raw = _mosaic(d.cfa_wd, d.cfa_ht, kind, case, seed + 1000 * i)
        outs.append(_Dev(d, raw).develop())
        torch.cuda.empty_cache()
    return outs[0] if case["kind"] == "plain" else outs
