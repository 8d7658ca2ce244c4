"""Timed cases of the escape-time engine: what a program that draws MDZ's
pictures with it asks for, through the entry points of mdz_amd.

Every case is a picture (or a set of pictures) of one of the scenes below, at
a size, an arithmetic and a call of its own:

  tile    Context.render        one rectangle of counts
  image   Context.render_image  a frame coloured on the device, aa x aa samples a pixel
  colour  Context.colour        new colours for counts that the program holds
  batch   Context.render_batch  many tiles of mixed scenes in one call
  lines   Frame                 the line-callback adapter under a pool of threads
  serve   Server                a burst of requests to the batching server

The seed moves each view by up to a twentieth of its width in both
directions, as a user pans.  Outputs are the counts, or the colours.
"""
import atexit
import math
import random
import threading
from decimal import Decimal, localcontext

import numpy as np

import mdz_amd as M

MANDEL, SHIP, CELTIC, VARIANT = (M.MANDELBROT, M.BURNING_SHIP, M.GENERALIZED_CELTIC, M.VARIANT)

# name: (fractal, centre re, centre im, width, depth, least precision, share
# of pixels that never escape, mean count of the others, Julia c or None).
# The first group are overviews at double or long double; the others MDZ's own
# saved scenes (their depth, their precision).
SCENES = {
    "set": (MANDEL, "-0.75", "0", "3.0", 1000, 53, 0.224, 6, None),
    "ship": (SHIP, "-1.755", "-0.03", "0.1", 1000, 53, 0.104, 26, None),
    "celtic": (CELTIC, "-0.5", "0", "4.0", 1000, 53, 0.122, 6, None),
    "rabbit": (MANDEL, "0", "0", "3.2", 1000, 53, 0.17, 4, ("-0.123", "0.745")),
    "valley": (MANDEL, "-0.7453", "0.1127", "0.0065", 2000, 53, 0.013, 163, None),
    "dragon": (MANDEL, "0", "0", "3.0", 2000, 53, 0.0, 40, ("-0.8", "0.156")),
    "minibrot": (MANDEL, "-1.74959314765277955385814405", "5.79069164258482514416295749995e-8",
                 "2.29427e-20", 3000, 80, 0.0, 605, None),
    "spiral": (MANDEL, "-0.74629927262353448490391415", "0.102867096643584583649032504867698",
               "1.327438992939e-9", 15000, 80, 0.0, 3040, None),
    "hue": (MANDEL, "-1.7685784531961471818887580974558413943355",
            "0.000916802637614158724519239287523575594361999996", "1.79114641e-31", 15000, 128,
            0.0, 1563, None),
    "banner": (MANDEL, "-1.99637882227229882217371024639011303135139825345684359602",
               "0.000113489705663572276277936233352526077599783317956930040650901",
               "4.325819211026e-36", 3000, 184, 0.0, 265, None),
    "satellite": (MANDEL, "-1.7851051241085002753420456045351336346026922033207689242805998155297725463",
                  "-1.2521208731662081988945007552294152151996027885546e-28", "1.270030101243e-25",
                  3000, 256, 0.0, 1220, None),
    "polyp": (MANDEL, "-1.749852636221530921864626112707956437852134401079226334071448117529664275168011",
              "3.987601201859246553675232798182764960727864940756534873313235004796405626503770e-16",
              "8.882808612185516632985644148025463626949610948719741e-57", 3000, 256, 0.001, 2331,
              None),
    "floral": (VARIANT, "-0.9353291846362110843246385699545115659353215485435407335736624188558665072689353",
               "0.2477033608381219680237587648624873900987680215948408339843037944858307534819688",
               "6.533710181836352997898952342270801258207833449e-48", 3000, 256, 0.0, 2026, None),
    "embedded": (MANDEL, "-1.9990958622795566830287308905472659490583061397701666190958559748388709828114012512346515",
                 "0.0000122514426432526505999592357810253330852566455347285164054457600705420954630245",
                 "3.789514356581e-39", 10000, 320, 0.0, 1255, None),
    "confirm": (MANDEL,
                "-1.9999999991382701187582747629086949883168091366368209595068022727154"
                "7027727918984035447670553861909622481524128059475119256402014495673143"
                "3166126504103",
                "0.00000000000001314895443507637575136247566806505002151700520912095709"
                "5294493435305489940275245944710958864319980774657032331030795428415894"
                "824327300210",
                "2.438973985837e-107", 1000, 512, 0.0, 516, None),
}

# deep zooms at any precision: a Misiurewicz point, where spiral arms repeat
# at every scale, found by Newton's method from its first digits: (first
# digits, preperiod, period, iterations a decade of zoom)
POINTS = {
    "filament": ("-0.10109636384562", "0.95628651080914", 4, 1, 8.1),
    "seahorse": ("-0.7756837680090538", "0.13646736829469", 24, 2, 60.6),
}
DIGITS = 340
_points = {}


def _mul(a, b):
    return a[0] * b[0] - a[1] * b[1], a[0] * b[1] + a[1] * b[0]


def _point(name):
    """The Misiurewicz point to DIGITS digits."""
    if name not in _points:
        re, im, pre, per, _ = POINTS[name]
        with localcontext() as lc:
            lc.prec = DIGITS + 40
            c = (Decimal(re), Decimal(im))
            for _ in range(14):
                z = d = (Decimal(0), Decimal(0))
                for i in range(pre + per):
                    zd = _mul(z, d)
                    d = (2 * zd[0] + 1, 2 * zd[1])
                    zz = _mul(z, z)
                    z = (zz[0] + c[0], zz[1] + c[1])
                    if i == pre - 1:
                        z0, d0 = z, d
                f = (z[0] - z0[0], z[1] - z0[1])
                g = (d[0] - d0[0], d[1] - d0[1])
                n = g[0] * g[0] + g[1] * g[1]
                q = _mul(f, (g[0], -g[1]))
                step = (q[0] / n, q[1] / n)
                c = (c[0] - step[0], c[1] - step[1])
                if abs(step[0]) + abs(step[1]) < Decimal(10) ** -(DIGITS + 10):
                    break
            _points[name] = c
    return _points[name]


def _decades(p):
    """Decades of zoom that a precision is chosen for: 2^-(p - 40) wide."""
    return (p - 40) * math.log10(2.0)


def _scene(name, p):
    """(fractal, re, im, width, depth, share inside, mean count, julia) as numbers."""
    if name in POINTS:
        rate = POINTS[name][4]
        mean = 10 + rate * _decades(p)
        re, im = _point(name)
        return MANDEL, re, im, Decimal(10) ** -int(_decades(p)), int(1.5 * mean), 0.0, mean, None
    fr, re, im, width, depth, _, inside, mean, julia = SCENES[name]
    return fr, Decimal(re), Decimal(im), Decimal(width), depth, inside, mean, julia


def _path(arith):
    return {"double": M.PATH_DOUBLE, "ld": M.PATH_LD, "mpfr": M.PATH_MPFR, "gmp": M.PATH_GMP}[arith]


def _bits(arith, p):
    return 64 if arith in ("double", "ld") else p


def _view(name, arith, p, w, h, aa, depth, rng):
    """A view of a scene, w x h pixels with aa x aa samples each, moved as rng says."""
    fr, re, im, width, d, _, _, julia = _scene(name, _bits(arith, p))
    with localcontext() as lc:
        lc.prec = DIGITS + 20
        re = re + width * Decimal(rng.randint(-500, 500)) / Decimal(10000)
        im = im + width * Decimal(rng.randint(-500, 500)) / Decimal(10000)
        re, im, width = format(re, "e"), format(im, "e"), format(width, "e")
    bits = _bits(arith, p)
    rect = M.rect_from_center(re, im, width, bits, w, h, coords=arith == "gmp")
    return M.make_view(rect, precision=bits, depth=depth or d, width=w * aa, height=h * aa,
                       fractal=fr, path=_path(arith), julia=julia or (None, None),
                       family=M.FAMILY_JULIA if julia else M.FAMILY_MANDEL)


# tiles of the mixed calls: (scene, arithmetic, precision), shallow and deep
MIX = [("set", "double", 64), ("filament", "mpfr", 128), ("rabbit", "ld", 64),
       ("minibrot", "mpfr", 80), ("seahorse", "mpfr", 256), ("celtic", "double", 64),
       ("satellite", "mpfr", 256), ("floral", "gmp", 256), ("ship", "ld", 64),
       ("filament", "mpfr", 512), ("banner", "mpfr", 184), ("filament", "mpfr", 1024)]
SIDES = (64, 128, 96, 256)


def _mixed(n):
    """n tiles: (scene, arithmetic, precision, side)."""
    return [MIX[i % len(MIX)] + (SIDES[(i // 3 + i) % len(SIDES)],) for i in range(n)]


def listed():
    return [
        # a first look at the set in a small window: the call's own cost counts
        dict(name="thumb_double", kind="tile", scene="set", arith="double", p=64,
             w=240, h=180, aa=1, depth=1000),
        # the whole set on a full-HD screen, 2 x 2 samples, in colour
        dict(name="image_double", kind="image", scene="set", arith="double", p=64,
             w=1920, h=1080, aa=2, depth=1000),
        # a Julia set in MDZ's default arithmetic (long double), window size
        dict(name="julia_ld", kind="tile", scene="rabbit", arith="ld", p=64,
             w=800, h=600, aa=1, depth=1000),
        # a saved scene at 80 bits, just past long double, deep orbits, odd size
        dict(name="spiral_80", kind="tile", scene="spiral", arith="mpfr", p=80,
             w=641, h=479, aa=1, depth=0),
        # a saved scene at 128 bits, 15000 iterations, drawn in colour with 2 x 2 samples
        dict(name="hue_128", kind="image", scene="hue", arith="mpfr", p=128,
             w=480, h=360, aa=2, depth=0),
        # MDZ's own render loop: threads that ask for a 176-bit frame line by line
        dict(name="lines_176", kind="lines", scene="seahorse", arith="mpfr", p=176,
             w=480, h=360, aa=1, depth=0),
        # a saved scene in GMP arithmetic, the odd-iteration Celtic hybrid
        dict(name="floral_gmp", kind="tile", scene="floral", arith="gmp", p=256,
             w=480, h=480, aa=1, depth=0),
        # a saved scene at 320 bits close to the real axis
        dict(name="embedded_320", kind="tile", scene="embedded", arith="mpfr", p=320,
             w=480, h=360, aa=1, depth=0),
        # the deepest frames: 1024 bits, 1e-296 wide
        dict(name="deep_1024", kind="tile", scene="filament", arith="mpfr", p=1024,
             w=960, h=540, aa=1, depth=0),
        # one small tile of a deep view, asked for alone: a preview, a repaired corner
        dict(name="corner_512", kind="tile", scene="filament", arith="mpfr", p=512,
             w=64, h=64, aa=1, depth=0),
        # a contact sheet: 36 tiles of uneven size, precision and formula in one call
        dict(name="batch_mixed", kind="batch", n=36),
        # a burst of the same kinds of tiles at the batching server
        dict(name="serve_mixed", kind="serve", n=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Rough cost of a case (multiply-accumulates and a term for each iteration's other work)."""
    return sum(n * (m + 60) for n, m in _iters(case))


MOST = None


def draw(rng):
    global MOST
    if MOST is None:
        MOST = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("tile", "tile", "tile", "image", "image", "lines", "colour", "batch",
                           "serve"))
        if kind in ("batch", "serve"):
            case = dict(kind=kind, n=rng.randint(3, 40))
        elif kind == "colour":
            case = dict(kind=kind, w=_log_int(rng, 240, 1920), h=_log_int(rng, 180, 1080),
                        aa=rng.choice((1, 2, 3)), ip=rng.random() < 0.5)
        else:
            group = rng.choice(("double", "ld", "saved", "saved", "deep", "deep", "gmp"))
            depth, p = 0, 64
            if group in ("double", "ld"):
                scene = rng.choice(("set", "ship", "celtic", "rabbit", "valley", "dragon"))
                arith, depth = group, _log_int(rng, 500, 5000)
            elif group == "saved":
                scene = rng.choice(("minibrot", "spiral", "hue", "banner", "satellite", "polyp",
                                    "embedded", "confirm"))
                arith, p = "mpfr", SCENES[scene][5] + rng.choice((0, 0, 16, 64))
            elif group == "deep":
                scene = rng.choice(("filament", "filament", "seahorse"))
                arith = "mpfr"
                p = rng.choice((128, 192, 256, 384, 512, 768, 1024, _log_int(rng, 65, 1024)))
            else:
                scene = rng.choice(("floral", "hue", "polyp", "filament"))
                arith = "gmp"
                p = rng.choice((128, 256, 512)) if scene == "filament" else SCENES[scene][5]
            case = dict(kind=kind, scene=scene, arith=arith, p=p, w=_log_int(rng, 48, 1280),
                        h=_log_int(rng, 48, 720), aa=rng.choice((1, 2)) if kind == "image" else 1,
                        depth=depth)
        if _cost(case) <= MOST:
            return case


_ctx = None
_srv = None


def _context():
    """The program's one context (a handle that every program keeps)."""
    global _ctx
    if _ctx is None:
        _ctx = M.Context(0)
        atexit.register(_close)
    return _ctx


def _server():
    global _srv
    if _srv is None:
        _srv = M.Server(_context(), hbm_budget=2 << 30)
    return _srv


def _close():
    global _ctx, _srv
    if _srv is not None:
        _srv.close()
        _srv = None
    if _ctx is not None:
        _ctx.close()
        _ctx = None


def _palette(rng, ip):
    a, b, c = (rng.uniform(0.0, 6.28) for _ in range(3))
    cols = [tuple(int(127.5 + 127.5 * math.sin(t * 0.0736 + k)) for k in (a, b, c))
            for t in range(256)]
    return M.make_palette(cols, offset=rng.randint(0, 200), colour_scale=0.08 if ip else 1.0,
                          interpolate=ip)


def prepare(case, seed):
    rng = random.Random(seed)
    s = {"kind": case["kind"], "ctx": _context()}
    if case["kind"] in ("batch", "serve"):
        s["views"] = [_view(sc, ar, p, side, side, 1, 0, rng) for sc, ar, p, side in
                      _mixed(case["n"])]
        if case["kind"] == "serve":
            s["server"] = _server()
        return s
    if case["kind"] == "colour":
        w, h = case["w"] * case["aa"], case["h"] * case["aa"]
        y, x = np.meshgrid(np.linspace(-1.1, 1.1, h, dtype=np.float32),
                           np.linspace(-2.2, 0.8, w, dtype=np.float32), indexing="ij")
        r = np.hypot(x + np.float32(0.5 + rng.uniform(-0.1, 0.1)), y)
        c = np.minimum(np.float32(2.0) / np.maximum(r - np.float32(0.55), np.float32(1e-3)), 1000)
        s.update(counts=np.where(r < 0.55, 0, 1 + c.astype(np.uint32)).astype(np.uint32),
                 aa=case["aa"], pal=_palette(rng, case["ip"]))
        return s
    s["view"] = _view(case["scene"], case["arith"], case["p"], case["w"], case["h"], case["aa"],
                      case["depth"], rng)
    s["aa"] = case["aa"]
    if case["kind"] == "image":
        s["pal"] = _palette(rng, True)
    if case["kind"] == "lines":
        s["raw"] = np.empty((case["h"], case["w"]), dtype=np.int32)
    return s


THREADS = 8    # MDZ starts one a core


def _lines(s):
    """MDZ's line pool: each thread takes the next line until none is left."""
    v, raw = s["view"], s["raw"]
    frame = M.Frame(s["ctx"], v, raw)
    lock = threading.Lock()
    left = iter(range(v.real_height))

    def work():
        while True:
            with lock:
                line = next(left, None)
            if line is None or frame.calculate_line(line) != 1:
                return

    pool = [threading.Thread(target=work) for _ in range(THREADS)]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    frame.close()
    return raw


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "tile":
        return ctx.render(state["view"])[0]
    if kind == "image":
        return ctx.render_image(state["view"], state["aa"], state["pal"])[0]
    if kind == "colour":
        return ctx.colour(state["counts"], state["aa"], state["pal"])
    if kind == "batch":
        return ctx.render_batch([(v, None, None) for v in state["views"]])[0]
    if kind == "lines":
        return _lines(state)
    srv = state["server"]
    return [srv.wait(i)[0] for i in [srv.submit(v) for v in state["views"]]]


def _iters(case):
    """[(iterations of the reference's loop, multiply operations of each)]."""
    if case["kind"] == "colour":
        return [(case["w"] * case["h"] * case["aa"] ** 2, 0)]
    if case["kind"] in ("batch", "serve"):
        parts = [(sc, ar, p, side, side, 1, 0) for sc, ar, p, side in _mixed(case["n"])]
    else:
        parts = [tuple(case[k] for k in ("scene", "arith", "p", "w", "h", "aa", "depth"))]
    out = []
    for sc, ar, p, w, h, aa, depth in parts:
        _, _, _, _, d, inside, mean, _ = _scene(sc, _bits(ar, p))
        depth = depth or d
        n = w * h * aa * aa * (inside * depth + (1 - inside) * min(mean, depth))
        words = -(-_bits(ar, p) // 32)
        out.append((n, 7 if ar == "double" else 2 * words * words + words))
    return out


def work(case):
    """Counts or colours written once and start values read once; the
    arithmetic of the reference's loop, a 32-bit multiply-accumulate as two
    operations, over the iterations that the scene's pixels take (a pixel
    that never escapes: its depth)."""
    flops = sum(n * (m if m == 7 else 2 * m) for n, m in _iters(case))
    if case["kind"] == "colour":
        n = case["w"] * case["h"]
        return {"bytes": 4 * n * (case["aa"] ** 2 + 1), "flops": 0}
    if case["kind"] in ("batch", "serve"):
        parts = [(ar, p, side, side, 1) for _, ar, p, side in _mixed(case["n"])]
    else:
        parts = [tuple(case[k] for k in ("arith", "p", "w", "h", "aa"))]
    nbytes = 0
    for ar, p, w, h, aa in parts:
        per = 16 if ar == "double" else _bits(ar, p) // 8 + 8
        nbytes += 4 * w * h * (1 if case["kind"] == "image" else aa * aa) + (w + h) * aa * per
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    """Counts and colours are whole numbers: compared as they are."""
    return None
