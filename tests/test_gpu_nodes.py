"""HIP node kernels against the oracle, through the C ABI (vkdt_hip_node_launch).

Every node of the raw-development graph runs on the GPU in graph order.
Each node's output is compared with the oracle's float build run on the
*same* inputs (the GPU's own input buffers), which isolates per-node error:
outside the near-tie texels the oracle flags, at most
parity.MAX_NODE_ULP binary16 ulps.  The final rgba is compared with the
oracle's whole-graph run under the end-to-end bound of tests/parity.py.
"""
import pytest

import graphspec as gs
import parity
from vkdt_amd import synth

pytestmark = pytest.mark.gpu

# (kind, W, H, seed, hilite, denoise strength): hilite inserts hilite between
# denoise and demosaic (bin/default-darkroom.i-raw:17-18); strength 0 (the
# param's default) makes denoise one noop node
CASES = [("bayer", 256, 192, 7, False, 0.5), ("xtrans", 258, 198, 11, False, 0.5),
         ("bayer", 256, 192, 17, True, 0.5), ("xtrans", 258, 198, 19, True, 0.5),
         ("bayer", 256, 192, 23, False, 0.0), ("xtrans", 258, 198, 29, False, 0.0)]
# downcov of hashed inputs (test_downcov_rounding): extent, digest of the output
DOWNCOV = [(67, 35, "1a9a005727e35180"), (258, 130, "c313927aa9e01344")]
IDS = [c[0] + ("-hilite" if c[4] else "") + ("-noop" if c[5] <= 0 else "") for c in CASES]


@pytest.fixture(scope="module", params=CASES, ids=IDS)
def graph_run(request, hip):
    kind, W, H, seed, hilite, strength = request.param
    cfa, _ = synth.mosaic(W, H, seed, kind)
    na, nb = synth.noise_params(2e-4, 1e-6)
    wb = (1.8, 1.0, 1.4, 1.0) if hilite else (1.0, 1.0, 1.0, 1.0)
    p = gs.DevelopParams(kind=kind, noise_a=na, noise_b=nb, hilite=hilite, wb=wb, strength=strength)
    bufs, nodes = gs.build(W, H, p)
    print(f"[gpu_nodes] {kind} {W}x{H} seed {seed} hilite {hilite}: {len(nodes)} nodes", flush=True)
    host = parity.run_gpu_graph(hip, bufs, nodes, cfa)
    return kind, W, H, cfa, p, bufs, nodes, host


def test_nodes_vs_oracle32(graph_run):
    kind, W, H, cfa, p, bufs, nodes, host = graph_run
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))


def test_end_to_end(graph_run):
    kind, W, H, cfa, p, bufs, nodes, host = graph_run
    parity.e2e_check(cfa, p, host["final"], log=lambda s: print(s, flush=True), label=f" {kind}")


@pytest.mark.parametrize("kind", ["bayer", "xtrans"])
def test_demosaic_down_node(hip, kind):
    """demosaic/down (down.comp:18-47), the block-mean luminance the module
    wires but gauss never samples (so the graph culls it): run on its own
    through the C ABI against the oracle"""
    import numpy as np
    import oracle_py as op
    blk = 3 if kind == "xtrans" else 2
    W, H = 96 * blk // 2, 66
    W -= W % blk
    rng = np.random.default_rng(31)
    mos = rng.uniform(0, 1, size=(H, W)).astype(np.float16)
    p = gs.DevelopParams(kind=kind)
    pc = gs.mixed_blob([("f", 1.0)] * 4 + [("i", p.filters)])
    bufs = {"raw": (W, H, 1, gs.F16, 1), "out": (W // blk, H // blk, 1, gs.F16, 1)}
    nodes = [dict(module="demosaic", kernel="down", pc=pc, params=gs.mixed_blob([("i", 0), ("i", 0)]),
                  conn=["raw", "out"], wd=W // blk, ht=H // blk, dp=1)]
    host = parity.run_gpu_graph(hip, bufs, nodes, mos)
    rep = parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))
    assert rep[0][2] <= 1


@pytest.mark.parametrize("fmt", [gs.F16, gs.UI16], ids=["f16", "unorm16"])
@pytest.mark.parametrize("W,H", [(6, 6), (96, 24), (291, 75), (294, 78), (297, 123), (390, 99)])
def test_xtrans_tiles(hip, fmt, W, H):
    """splat and fix on X-Trans mosaics of every tile case: smaller than a
    tile of 96x24, no tile inside the image, the first extents with one (96 +
    96 + taps), partial tiles: against the oracle on the same inputs"""
    import numpy as np
    rng = np.random.default_rng(W * H + fmt)
    mos = rng.uniform(0.05, 1, size=(H, W)).astype(np.float16) if fmt == gs.F16 else rng.integers(2000, 65536, (H, W), dtype=np.uint16)
    p = gs.DevelopParams(kind="xtrans")
    pc = gs.mixed_blob([("f", 1.0)] * 4 + [("i", p.filters)])
    par = gs.mixed_blob([("i", 0), ("i", 0)])
    bufs = {"raw": (W, H, 1, fmt, 1), "cov": (W // 3, H // 3, 4, gs.F16, 1), "green": (W, H, 1, gs.F16, 1),
            "out": (W, H, 4, gs.F16, 1)}
    nodes = [dict(module="demosaic", kernel="gauss", pc=pc, params=par, conn=["raw", "raw", "cov"], wd=W // 3, ht=H // 3, dp=1, out=2),
             dict(module="demosaic", kernel="splat", pc=pc, params=par, conn=["raw", "cov", "green"], wd=W, ht=H, dp=1, out=2),
             dict(module="demosaic", kernel="fix", pc=pc, params=par, conn=["raw", "green", "cov", "out"], wd=W, ht=H, dp=1, out=3)]
    host = parity.run_gpu_graph(hip, bufs, nodes, mos)
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))


@pytest.mark.parametrize("kind,W,H,cx,cy", [("bayer", 2, 2, 0, 0), ("bayer", 67, 35, 1, 3), ("bayer", 130, 18, 4, 2),
                                            ("xtrans", 3, 3, 0, 0), ("xtrans", 97, 26, 0, 0), ("xtrans", 100, 25, 6, 3),
                                            ("xtrans", 195, 51, 1, 2)])
def test_doub_blocks(hip, kind, W, H, cx, cy):
    """denoise/doub, a block or a cell's row per thread, where the last ones are cut
    (one and two columns and rows left), the output is one block, and the crop
    moves it over the mosaic's mirrored edge: against the oracle on the same
    inputs"""
    import numpy as np
    rng = np.random.default_rng(W * H + cx)
    raw = rng.integers(500, 16384, (H, W), dtype=np.uint16)
    p = gs.DevelopParams(kind=kind)
    blk = 3 if kind == "xtrans" else 2
    qw, qh = -(-W // blk), -(-H // blk)
    black, white = np.float32(512 / 65535.0), np.float32(16383 / 65535.0)
    rgbc = [("f", 1.0)] * 4 + [("f", black)] * 4 + [("f", white)] * 4 + [("i", v) for v in (cx, cy, W + cx, H + cy)]
    par = gs.mixed_blob([("f", 0.6), ("f", 0.3), ("f", 0.7), ("f", 0.0)] + [("f", 1.0)] * 4 + [("i", 1)])
    bufs = {"raw": (W, H, 1, gs.UI16, 1), "half": (qw, qh, 4, gs.F16, 1), "s0": (qw, qh, 4, gs.F16, 1), "dn": (W, H, 1, gs.F16, 1)}
    lv = rgbc[:12] + [("i", 0)] * 4
    nodes = [dict(module="denoise", kernel="half", pc=gs.mixed_blob(rgbc + [("i", p.filters)]), params=par,
                  conn=["raw", "half"], wd=qw, ht=qh, dp=1, out=1),
             dict(module="denoise", kernel="downcov", pc=gs.mixed_blob(lv + [("f", 1e-4), ("f", 1e-6), ("i", 0), ("i", blk)]),
                  params=par, conn=["half", "s0"], wd=qw, ht=qh, dp=1, out=1),
             dict(module="denoise", kernel="doub",
                  pc=gs.mixed_blob(rgbc + [("i", p.filters), ("f", 1e-4), ("f", 1e-6), ("i", 0)] + [("i", 0)] * 4), params=par,
                  conn=["raw", "s0", "half", "dn"], wd=W, ht=H, dp=1, out=3)]
    host = parity.run_gpu_graph(hip, bufs, nodes, raw)
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))


@pytest.mark.parametrize("W", [5, 67, 1030])
@pytest.mark.parametrize("par", [(0.12, 1.0, 1.0, 0.2), (0.05, 1.6, 0.3, 1.0), (0.5, 0.2, 2.0, 0.0), (0.25, -0.5, -0.5, -0.3)])
def test_llap_curve(hip, par, W):
    """llap/curve over values on the gammas, at the joint of its two parts
    (2 sigma from a gamma), far out and negative; few and many curves, odd
    extents: against the oracle"""
    import numpy as np
    H, ng = 3, 10
    rng = np.random.default_rng(W)
    lum = rng.uniform(-0.2, 1.4, size=(H, W))
    lum[0, ::2] = rng.integers(0, ng, lum[0, ::2].shape) / (ng - 1.0)
    lum[1, ::2] = lum[0, 0] + 2.0 * par[0]
    lum[2, 0], lum[2, 2] = 40.0, -3.0
    raw = np.repeat(lum[:, :, None], 4, axis=2).astype(np.float16)
    bufs = {"raw": (W, H, 4, gs.F16, 1), "pyr0": (W, H, 1, gs.F16, ng + 1)}
    nodes = [dict(module="llap", kernel="curve", pc=gs.mixed_blob([("i", ng)]), params=gs.f32blob(list(par)),
                  conn=["raw", "pyr0"], wd=W, ht=H, dp=1, out=1)]
    host = parity.run_gpu_graph(hip, bufs, nodes, raw)
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))


def _hashed(n, seed):
    """n values of 0..1 from an integer hash: the same wherever they are made"""
    import numpy as np
    u = np.arange(n, dtype=np.uint64) * np.uint64(2654435761) + np.uint64(seed) * np.uint64(40503)
    u = ((u ^ (u >> np.uint64(15))) * np.uint64(2246822519)) & np.uint64(0xffffffff)
    u = ((u ^ (u >> np.uint64(13))) * np.uint64(3266489917)) & np.uint64(0xffffffff)
    return ((u ^ (u >> np.uint64(16))) & np.uint64(0xffff)).astype(np.float64) / 65535


@pytest.mark.parametrize("W", [67, 1030], ids=["scalar", "vector"])
@pytest.mark.parametrize("par", [(0.12, 1.2, 0.8), (0.05, 1.6, 0.3), (0.25, -0.5, -0.5)])
def test_llap_curve_rounding(hip, par, W):
    """llap/curve without clarity uses no transcendental: it equals the
    reference's formula (curve.comp:39-63) in float32, each operation rounded
    once in the order written there, bit for bit"""
    import numpy as np
    f = np.float32
    H, ng = 96, 10
    lum = _hashed(W * H, 5).reshape(H, W) * 1.5 - 0.2
    raw = np.repeat(lum[:, :, None], 4, axis=2).astype(np.float16)
    bufs = {"raw": (W, H, 4, gs.F16, 1), "pyr0": (W, H, 1, gs.F16, ng + 1)}
    nodes = [dict(module="llap", kernel="curve", pc=gs.mixed_blob([("i", ng)]), params=gs.f32blob(list(par) + [0.0]),
                  conn=["raw", "pyr0"], wd=W, ht=H, dp=1, out=1)]
    got = parity.run_gpu_graph(hip, bufs, nodes, raw)["pyr0"].reshape(ng + 1, H, W)
    x, k = raw[..., 0].astype(f), [f(2.62700212e-01), f(6.77998072e-01), f(5.93017165e-02)]
    x = (k[0] * x + k[1] * x) + k[2] * x                      # the luminance of a grey pixel
    sigma, shadows, highlights = (f(v) for v in par)
    for i in range(ng):
        g = f(i) / f(ng - 1)
        c = x - g
        s = np.where(c > 0, sigma, -sigma)
        sh = np.where(c > 0, shadows, highlights)
        far = g + s + sh * (c - s)
        t = np.clip(c * np.where(c > 0, f(1) / (f(2) * sigma), -(f(1) / (f(2) * sigma))), f(0), f(1))
        near = g + s * f(2) * (f(1) - t) * t + t * t * (s + s * sh)
        want = np.where(np.abs(c) > f(2) * sigma, far, near)
        assert want.dtype == np.float32
        nd = int(np.count_nonzero(want.astype(np.float16) != got[i]))
        assert nd == 0, (i, nd)


@pytest.mark.parametrize("W,H,digest", DOWNCOV, ids=[f"{w}x{h}" for w, h, _ in DOWNCOV])
def test_downcov_rounding(hip, W, H, digest):
    """denoise/downcov's bytes as recorded on a gfx950.  Its weighted sums
    feed the wavelet's base level, and a binary16 step there can reach gauss's
    choice between two nearly equal covariances, which changes a pixel visibly:
    a rounding in another place is a change of the developed image"""
    import hashlib
    import numpy as np
    v = _hashed(W * H * 3, 7).reshape(H, W, 3)
    base = 0.02 + 0.5 * (((np.arange(W) // 5)[None, :] + (np.arange(H) // 3)[:, None]) % 4)   # edges of several heights
    raw = np.ones((H, W, 4), np.float16)
    raw[..., :3] = (base[:, :, None] * (0.9 + 0.2 * v)).astype(np.float16)
    lv = [("f", 1.0)] * 4 + [("f", np.float32(512 / 65535.0))] * 4 + [("f", np.float32(16383 / 65535.0))] * 4 + [("i", 0)] * 4
    par = gs.mixed_blob([("f", 0.6), ("f", 0.3), ("f", 0.7), ("f", 0.0)] + [("f", 1.0)] * 4 + [("i", 1)])
    bufs = {"raw": (W, H, 4, gs.F16, 1), "s0": (W, H, 4, gs.F16, 1)}
    nodes = [dict(module="denoise", kernel="downcov", pc=gs.mixed_blob(lv + [("f", 1e-4), ("f", 1e-6), ("i", 0), ("i", 2)]),
                  params=par, conn=["raw", "s0"], wd=W, ht=H, dp=1, out=1)]
    host = parity.run_gpu_graph(hip, bufs, nodes, raw)
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))
    got = hashlib.sha256(np.ascontiguousarray(host["s0"]).tobytes()).hexdigest()[:16]
    print(f"[downcov] {W}x{H} {got}", flush=True)
    assert got == digest


@pytest.mark.parametrize("ng,step", [(2, 1), (10, 1), (10, 16), (32, 1)])
def test_llap_assemble_planes(hip, ng, step):
    """llap/assemble above the extent of the small kernel with tiles that
    select a few of the planes, all of them and more than are held at once,
    on every gamma (where the choice of the plane changes), partial tiles in
    both directions, and both kinds of coarse level: against the oracle"""
    import numpy as np
    rng = np.random.default_rng(ng)
    W, H = 1037, 531
    lum = rng.uniform(-0.1, 1.2, size=(H // step + 1, W // step + 1)).repeat(step, 0).repeat(step, 1)[:H, :W]
    lum[::3, ::5] = np.round(lum[::3, ::5] * (ng - 1)) / (ng - 1)
    raw = np.repeat(lum[:, :, None], 4, axis=2).astype(np.float16)
    w, h = [W], [H]
    for l in range(2):
        w.append((w[-1] - 1) // 2 + 1)
        h.append((h[-1] - 1) // 2 + 1)
    bufs = {"raw": (W, H, 4, gs.F16, 1)}
    for l in range(3):
        bufs[f"pyr{l}"] = (w[l], h[l], 1, gs.F16, ng + 1)
    bufs.update(out0=(W, H, 1, gs.F16, 1), out1=(w[1], h[1], 1, gs.F16, 1), only=(W, H, 1, gs.F16, 1))
    par = gs.f32blob([0.12, 1.2, 0.8, 0.3])
    node = lambda k, pc, conn, wd, ht, dp=1: dict(module="llap", kernel=k, pc=pc, params=par, conn=conn, wd=wd, ht=ht, dp=dp,
                                                  out=len(conn) - 1)
    asm = lambda first: gs.mixed_blob([("i", ng), ("i", first)])
    nodes = [node("curve", gs.mixed_blob([("i", ng)]), ["raw", "pyr0"], W, H),
             node("reduce", None, ["pyr0", "pyr1"], w[1], h[1], ng + 1), node("reduce", None, ["pyr1", "pyr2"], w[2], h[2], ng + 1),
             node("assemble", asm(1), ["pyr0", "pyr1", "pyr2", "out1"], w[1], h[1]),
             node("assemble", asm(0), ["out1", "pyr0", "pyr1", "out0"], W, H),
             node("assemble", asm(1), ["pyr0", "pyr0", "pyr1", "only"], W, H)]
    host = parity.run_gpu_graph(hip, bufs, nodes, raw)
    parity.check_nodes(bufs, nodes, host, log=lambda s: print(s, flush=True))


@pytest.mark.parametrize("W,H", [(96 * 30, 24 * 18 + 6), (96 * 46 + 3, 24 * 46)])
def test_xtrans_tiles_in_parts(hip, W, H):
    """splat and fix above the tile counts at which a tile is cut into nine
    parts, three and none (570 and 2162 tiles; the smaller extents of
    test_xtrans_tiles have nine): the general path's values, which a graph cut
    to a part of the image gives, away from the cut"""
    import numpy as np
    rng = np.random.default_rng(W)
    mos = rng.uniform(0.05, 1, size=(H, W)).astype(np.float16)
    p = gs.DevelopParams(kind="xtrans")
    pc = gs.mixed_blob([("f", 1.0)] * 4 + [("i", p.filters)])
    par = gs.mixed_blob([("i", 0), ("i", 0)])

    def run(m):
        h, w = m.shape
        bufs = {"raw": (w, h, 1, gs.F16, 1), "cov": (w // 3, h // 3, 4, gs.F16, 1), "green": (w, h, 1, gs.F16, 1),
                "out": (w, h, 4, gs.F16, 1)}
        nodes = [dict(module="demosaic", kernel="gauss", pc=pc, params=par, conn=["raw", "raw", "cov"], wd=w // 3, ht=h // 3, dp=1, out=2),
                 dict(module="demosaic", kernel="splat", pc=pc, params=par, conn=["raw", "cov", "green"], wd=w, ht=h, dp=1, out=2),
                 dict(module="demosaic", kernel="fix", pc=pc, params=par, conn=["raw", "green", "cov", "out"], wd=w, ht=h, dp=1, out=3)]
        return parity.run_gpu_graph(hip, bufs, nodes, np.ascontiguousarray(m))

    host = run(mos)
    for y0, x0 in ((0, 0), (6 * (H // 12), 6 * (W // 12)), (H - 132 - H % 6, W - 132 - W % 6)):
        part = run(mos[y0:y0 + 132, x0:x0 + 132])
        for k in ("green", "out"):
            assert np.array_equal(host[k][y0 + 12:y0 + 120, x0 + 12:x0 + 120], part[k][12:120, 12:120]), (k, y0, x0)
