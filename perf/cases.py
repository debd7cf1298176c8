"""The renders whose speed is measured: what programs that use this library
have it do, each through the C ABI with everything a program keeps (genome
structs, image buffers, the render server) made beforehand.

A case is one of five calls:

* still    one flam3_render call: a still from one genome;
* frame    one flam3_render call: an animation frame between two control
           points, with motion blur (temporal samples);
* many     one fl3h_render_many call: a set of preview requests;
* served   a run of animation frames through a render server;
* bbox     one fl3h_estimate_bounding_box call for a candidate genome.

Genomes are the package's seeded synthetic ones (random affines, variation
mixes, palettes), another for every seed.  A frame's random stream is seeded
again for every call, so that a pass can be repeated.
"""
import ctypes
import math

import numpy as np

import flam3_amd as F
from flam3_amd import abi, opcount
from flam3_amd import genome as G
from flam3_amd._lib import fl3h_request

# Variations without parameters from all over the library (beyond the
# fourteen classic ones), for genomes that need the full variation set.
WIDE_VARS = ["bent", "fisheye", "exponential", "cosine", "eyefish", "bubble", "cylinder", "noise", "blur", "arch",
             "tangent", "square", "rays", "blade", "twintrian", "cross", "edisc", "elliptic", "foci", "loonie",
             "polar2", "exp", "sin", "cosh", "linear", "spherical", "swirl", "julia"]

STILL = dict(kind="still", family="flame", supersample=1, radius=9.0, bits=33, bpc=1, nchan=3, earlyclip=0,
             palette="step", opacity=1.0)


def still(**kw):
    return dict(STILL, **kw)


def listed():
    return [
        # The smallest preview a genome search asks for: one call, where the
        # launches and the walkers' serial steps are all the time.
        still(name="preview_64", family="preview", width=64, height=64, quality=10.0),
        # An ordinary preview of the same search, rendered alone.
        still(name="preview_256", family="preview", width=256, height=256, quality=55.0),
        # A quick colour trial: integer accumulator, no density estimation,
        # clipping before the filter (the settings of the colour search).
        still(name="trial_bits32", family="preview", width=400, height=300, quality=8.0, bits=32, radius=0.0,
              earlyclip=1),
        # A page of a genome search: many previews of mixed sizes together.
        dict(name="previews_many", kind="many", count=48, largest=512),
        # The small reference workload: three xforms of contracting maps.
        still(name="still_640x480", family="small", width=640, height=480, quality=50.0),
        # A still of odd size as an editor exports it: linear palette, faded
        # xforms, 16-bit RGBA.
        still(name="still_odd_rgba16", width=1021, height=767, quality=60.0, supersample=2, bpc=2, nchan=4,
              palette="linear", opacity=0.6),
        # Variations from the whole library, post transforms.
        still(name="still_wide", family="wide", width=800, height=600, quality=100.0, supersample=2),
        # The headline still.
        still(name="still_1080p", width=1920, height=1080, quality=500.0, supersample=2),
        # A large still in double precision with xaos and wide density
        # estimation (its histogram exceeds one band of tiles).
        still(name="still_4k_bits64", family="xaos", width=3840, height=2160, quality=120.0, supersample=3,
              radius=15.0, bits=64),
        # One motion-blurred animation frame in one call.
        dict(name="frame_720p", kind="frame", width=1280, height=720, quality=200.0, supersample=2, temporal=100),
        # Consecutive frames of that animation through the render server.
        dict(name="frames_served", kind="served", count=16, width=1280, height=720, quality=200.0, supersample=2,
             temporal=100),
        # The bounding box of one candidate genome (a single trajectory).
        dict(name="bounding_box", kind="bbox", points=20000),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["still"] * 6 + ["many", "many", "frame", "frame", "served", "bbox"])
    if kind == "bbox":
        return dict(kind=kind, points=int(_log(rng, 2000, 20000)))
    if kind == "many":
        return dict(kind=kind, count=int(_log(rng, 2, 64)), largest=rng.choice([64, 100, 128, 256, 333, 512]))
    if kind in ("frame", "served"):
        width = int(_log(rng, 96, 1280))
        c = dict(kind=kind, width=width, height=int(width * rng.uniform(0.5, 0.8)), quality=round(_log(rng, 10, 200), 1),
                 supersample=rng.choice([1, 2]), temporal=rng.choice([5, 16, 60, 100, 117]))
        if kind == "served":
            c["count"] = rng.randrange(3, 17)
        return c
    width = int(_log(rng, 48, 1920))
    c = still(family=rng.choice(["preview", "small", "flame", "flame", "wide", "xaos"]), width=width,
              height=int(width * rng.uniform(0.5, 1.0)), quality=round(_log(rng, 5, 500), 1),
              supersample=rng.choice([1, 1, 2, 2, 3]), radius=rng.choice([0.0, 4.0, 7.0, 9.0, 9.0, 11.0, 15.0]),
              bits=rng.choice([32, 33, 33, 33, 33, 64]), bpc=rng.choice([1, 1, 2]), nchan=rng.choice([3, 3, 4]),
              earlyclip=rng.choice([0, 0, 0, 1]), palette=rng.choice(["step", "step", "step", "linear"]),
              opacity=rng.choice([1.0, 1.0, 1.0, 0.7]))
    most = 3e8 if c["bits"] == 64 else 1e9
    c["quality"] = min(c["quality"], round(most / (c["width"] * c["height"]), 1))
    return c


# ------------------------------------------------------------- genomes

def _wide(seed, width, height, quality, supersample):
    rng = np.random.default_rng(seed)
    xs = [G._mixed_xform(rng, WIDE_VARS, 3, -1.0, 1.0) for _ in range(5)]
    for x in xs[:2]:
        x.post = tuple(float(v) for v in rng.uniform(-0.9, 0.9, 6))
    return G.Genome(width=width, height=height, scale=height / 3.0, quality=quality, supersample=supersample,
                    estimator_radius=9.0, palette=G.hsv_palette(rng), xforms=xs)


def _still_genome(case, seed):
    size = dict(width=case["width"], height=case["height"], quality=case["quality"])
    if case["family"] == "small":
        g = G.synthetic_small(seed=seed, **size)
    elif case["family"] == "preview":
        g = G.synthetic_preview(seed)
        g.width, g.height, g.scale, g.quality = case["width"], case["height"], case["height"] / 3.0, case["quality"]
    elif case["family"] == "xaos":
        g = G.synthetic_8k(seed=seed, supersample=case["supersample"], **size)
    elif case["family"] == "wide":
        g = _wide(seed, supersample=case["supersample"], **size)
    else:
        g = G.synthetic_1080p(seed=seed, supersample=case["supersample"], **size)
    g.supersample = case["supersample"]
    g.estimator_radius = case["radius"]
    g.palette_mode = case["palette"]
    for k, x in enumerate(g.xforms):
        if case["opacity"] != 1.0 and k % 2:
            x.opacity = case["opacity"]
    return g


def _preview_sizes(case):
    """The size and quality of each request of a preview set: the same for
    every seed, spread over 64..largest and 10..100."""
    out = []
    for k in range(case["count"]):
        s = max(48, case["largest"] >> (k % 4))
        out.append((s, 10.0 + 90.0 * ((k * 37) % 50) / 50.0))
    return out


# ------------------------------------------------------------- calls

class State:
    """What a program keeps for its calls; releases it when dropped."""

    def __init__(self):
        self.owned, self.arrays, self.frames, self.images, self.stats = [], [], [], [], []
        self.server = None
        self.pixels = None   # every image, one after another

    def __del__(self):
        if self.server is not None:
            self.server.close()
        for gp in self.owned:
            G.free_struct(gp)

    def add_genomes(self, genomes):
        arr, owned = G.genome_array(genomes)
        self.arrays.append(arr)
        self.owned += owned
        return arr

    def add_images(self, sizes, nchan=3, bpc=1):
        self.pixels = np.zeros(sum(w * h for w, h in sizes) * nchan, np.uint16 if bpc == 2 else np.uint8)
        at = 0
        for w, h in sizes:
            self.images.append(self.pixels[at:at + w * h * nchan].reshape(h, w, nchan))
            self.stats.append(abi.stat_struct())
            at += w * h * nchan

    def frame(self, k, **kw):
        arr = self.arrays[k if len(self.arrays) > 1 else 0]
        return F.make_frame(ctypes.addressof(arr), len(arr), seed="frame-%d" % k, **kw)


def prepare(case, seed):
    s = State()
    s.kind = case["kind"]
    if s.kind == "still":
        s.settings = dict(bits=case["bits"], bpc=case["bpc"], earlyclip=case["earlyclip"])
        s.nchan = case["nchan"]
        s.add_genomes([_still_genome(case, seed)])
        s.add_images([(case["width"], case["height"])], case["nchan"], case["bpc"])
    elif s.kind == "frame" or s.kind == "served":
        s.settings = {}
        s.nchan = 3
        s.add_genomes(G.synthetic_animation(seed=seed, width=case["width"], height=case["height"],
                                            quality=case["quality"], supersample=case["supersample"],
                                            temporal_samples=case["temporal"]))
        s.add_images([(case["width"], case["height"])] * case.get("count", 1))
        if s.kind == "served":
            s.server = F.Server()
    elif s.kind == "many":
        s.settings = {}
        sizes = _preview_sizes(case)
        for k, (size, quality) in enumerate(sizes):
            s.add_genomes([G.synthetic_preview(64 * seed + k, size=size, quality=quality)])
        s.add_images([(size, size) for size, _ in sizes])
    else:
        s.add_genomes([G.synthetic_1080p(seed=seed, width=128, height=72)])
        s.points = case["points"]
        F.lib().fl3h_estimate_bounding_box.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_int, ctypes.c_void_p,
                                                       ctypes.c_void_p, ctypes.c_void_p]
    return s


def _pointer(img):
    return img.ctypes.data_as(ctypes.c_void_p)


def _results(s):
    return s.pixels, np.array([(int(st.num_iters), int(st.badvals)) for st in s.stats])


def run(s):
    L = F.lib()
    if s.kind == "still" or s.kind == "frame":
        f = s.frame(0, **(s.settings if s.kind == "still" else {"time": 41.5}))
        if L.flam3_render(ctypes.byref(f), _pointer(s.images[0]), 0, s.nchan, 0, ctypes.byref(s.stats[0])):
            raise RuntimeError(F.last_error())
        return _results(s)
    if s.kind == "served":
        s.frames = [s.frame(k, time=40.0 + k) for k in range(len(s.images))]
        ids = [L.fl3h_server_submit(s.server._s, ctypes.byref(f), _pointer(img), 0, 3, 0, ctypes.byref(st))
               for f, img, st in zip(s.frames, s.images, s.stats)]
        for i in ids:
            if i < 0 or L.fl3h_server_wait(s.server._s, i, None):
                raise RuntimeError(F.last_error())
        return _results(s)
    if s.kind == "many":
        s.frames = [s.frame(k) for k in range(len(s.images))]
        reqs = (fl3h_request * len(s.images))()
        for r, f, img, st in zip(reqs, s.frames, s.images, s.stats):
            r.frame = ctypes.addressof(f)
            r.out = img.ctypes.data
            r.nchan = 3
            r.stats = ctypes.addressof(st)
        if L.fl3h_render_many(reqs, len(reqs), None):
            raise RuntimeError(F.last_error())
        return _results(s)
    f = s.frame(0)
    lo, hi = np.zeros(2), np.zeros(2)
    bad = L.fl3h_estimate_bounding_box(ctypes.addressof(s.arrays[0][0]), 0.01, s.points, _pointer(lo), _pointer(hi),
                                       ctypes.byref(f.rc))
    if bad < 0:
        raise RuntimeError(F.last_error())
    return lo, hi, bad


# ------------------------------------------------------------- work

def _ops(genome):
    """FP32 operations per plotted sample."""
    try:
        return opcount.ops_per_sample(genome)
    except KeyError:   # variations the count does not cover
        return 100.0


def work(case):
    """The formula operations of every plotted sample; the image bytes."""
    if case["kind"] == "still":
        px = case["width"] * case["height"]
        return {"bytes": px * case["nchan"] * case["bpc"],
                "flops": px * case["quality"] * _ops(_still_genome(case, 2))}
    if case["kind"] in ("frame", "served"):
        px = case["width"] * case["height"] * case.get("count", 1)
        return {"bytes": px * 3, "flops": px * case["quality"] * _ops(G.synthetic_animation(seed=2)[0])}
    if case["kind"] == "many":
        sizes = _preview_sizes(case)
        return {"bytes": sum(s * s * 3 for s, _ in sizes), "flops": sum(s * s * q for s, q in sizes) * 60.0}
    return {"bytes": 32, "flops": case["points"] * 100.0}


def exact(case, seed):
    """None: images are whole numbers drawn from a random trajectory, which
    only the same arithmetic draws again."""
    return None
