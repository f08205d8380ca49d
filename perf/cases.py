"""The work that users of this framework have it do, as timed cases.

Every case goes through the public binding: decomp_2d_fft_init (FFTEngine,
made as a user makes it, with the default kernels), decomp_2d_fft_3d's
c2c / r2c / c2r, decomp_2d_dtt_3d_r2r, the batch of many grids, the per-rank
stages with the packs and unpacks of their exchanges, and update_halo.

Fields are flat tensors in Fortran order (i fastest), i.e. torch shape
(nz, ny, nx).  A case is a dict of plain values; `kind` names the path:

  c2c    forward then backward complex transform      -> (spectrum, field)
  r2c    r2c then c2r                                 -> (spectrum, field)
  dtt    forward then backward real-to-real transform -> (coefficients, field)
  batch  c2c of many uneven grids as one batch        -> every grid's output
  rank   the forward r2c stages of one rank of a process grid, each reading
         what an exchange delivered and writing what the next one sends
  halo   update_halo of one pencil                    -> the halo array
"""
import importlib
import math

import torch

d2d = importlib.import_module("2decomp-fft_amd")

# lengths that the uneven batches are made of (the multi-grid benchmark's)
BATCH_LENGTHS = (32, 48, 64, 80, 96, 128, 160, 192, 256)
MAX_POINTS = 1 << 28  # drawn grids: a quarter of the largest listed one


def listed():
    return [
        # the reference's own test grid: odd and prime extents, latency alone
        {"name": "c2c_17x13x11", "kind": "c2c", "nx": 17, "ny": 13, "nz": 11, "fmt": 1, "prec": 64},
        # a small periodic box, the pencils of which stay on the chip
        {"name": "c2c_128", "kind": "c2c", "nx": 128, "ny": 128, "nz": 128, "fmt": 1, "prec": 64},
        # a spectral solver's usual box
        {"name": "r2c_512", "kind": "r2c", "nx": 512, "ny": 512, "nz": 512, "fmt": 1, "prec": 64},
        # an uneven mixed-radix box, physical space in the z-pencil
        {"name": "r2c_z_720x540x432", "kind": "r2c", "nx": 720, "ny": 540, "nz": 432, "fmt": 3,
         "prec": 64},
        # extents as a mesh gives them: odd smooth numbers and one with a
        # large prime factor (382 = 2 * 191)
        {"name": "r2c_450x405x382", "kind": "r2c", "nx": 450, "ny": 405, "nz": 382, "fmt": 1,
         "prec": 64},
        # the headline box in the three precisions a plan can have
        {"name": "r2c_1024", "kind": "r2c", "nx": 1024, "ny": 1024, "nz": 1024, "fmt": 1,
         "prec": 64},
        {"name": "r2c_1024_f32", "kind": "r2c", "nx": 1024, "ny": 1024, "nz": 1024, "fmt": 1,
         "prec": 32},
        {"name": "r2c_1024_split", "kind": "r2c", "nx": 1024, "ny": 1024, "nz": 1024, "fmt": 1,
         "prec": 16},
        # a Poisson solver's cosine transforms on a vertex grid
        {"name": "dct2_513", "kind": "dtt", "nx": 513, "ny": 513, "nz": 513, "fmt": 1, "prec": 64,
         "tx": 2, "ty": 2, "tz": 2},
        # many independent grids at once (multi-block use), forward and back
        {"name": "batch_64", "kind": "batch", "grids": 64, "shape_seed": 4, "mode": 0, "prec": 64},
        # one rank's share of the headline box on a 4 x 2 process grid
        {"name": "rank_1024_4x2", "kind": "rank", "nx": 1024, "ny": 1024, "nz": 1024,
         "p_row": 4, "p_col": 2, "row": 1, "col": 1, "prec": 64},
        # ghost cells of a finite-difference code, two levels
        {"name": "halo_512", "kind": "halo", "nx": 512, "ny": 512, "nz": 512, "level": 2,
         "pencil": 1, "prec": 64},
    ]


# ---- more cases of the same ranges ------------------------------------------


def _smooth(n):
    """The number 2^a 3^b 5^c nearest to n (the larger of two as near)."""
    for d in range(n):
        for m in (n + d, n - d):
            k = m
            for p in (2, 3, 5):
                while k > 1 and k % p == 0:
                    k //= p
            if k == 1 and m > 1:
                return m
    return n


def _length(rng, lo, hi):
    """One extent: mostly smooth numbers, some powers of two, some anything."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    u = rng.random()
    if u < 0.5:
        return max(lo, min(hi, _smooth(n)))
    if u < 0.75:
        return max(lo, min(hi, 1 << int(round(math.log2(n)))))
    return n


def _extents(rng, lo, hi, limit):
    while True:
        e = [_length(rng, lo, hi) for _ in range(3)]
        if e[0] * e[1] * e[2] <= limit:
            return e


def draw(rng):
    kind = rng.choice(("c2c", "c2c", "r2c", "r2c", "r2c", "dtt", "dtt", "batch", "rank", "halo"))
    prec = rng.choice((64, 64, 64, 32, 16 if kind in ("c2c", "r2c") else 32))
    if kind == "batch":
        return {"kind": kind, "grids": rng.randint(8, 96), "shape_seed": rng.randint(5, 1 << 20),
                "mode": rng.choice((-1, 0, 1)), "prec": prec}
    if kind == "dtt":
        nx, ny, nz = _extents(rng, 17, 512, MAX_POINTS)
        t = [rng.randint(1, 8) if rng.random() < 0.5 else 2 for _ in range(3)]
        return {"kind": kind, "nx": nx + 1, "ny": ny + 1, "nz": nz + 1,
                "fmt": rng.choice((1, 3)), "prec": prec, "tx": t[0], "ty": t[1], "tz": t[2]}
    if kind == "rank":
        nx, ny, nz = _extents(rng, 64, 1024, 1 << 30)
        p_row, p_col = rng.choice(((2, 2), (4, 2), (2, 4), (3, 2)))
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "p_row": p_row, "p_col": p_col,
                "row": rng.randrange(p_row), "col": rng.randrange(p_col), "prec": prec}
    nx, ny, nz = _extents(rng, 11, 1024, MAX_POINTS)
    if kind == "halo":
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "level": rng.randint(1, 3),
                "pencil": rng.choice((1, 2, 3)), "prec": prec}
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "fmt": rng.choice((1, 3)), "prec": prec}


# ---- inputs and plans ----------------------------------------------------------


def _real_type(case):
    return torch.float64 if case["prec"] == 64 else torch.float32


def _complex_type(case):
    return torch.complex128 if case["prec"] == 64 else torch.complex64


def _noise(shape, dtype, gen, scale=1.0):
    t = torch.empty(shape, dtype=dtype, device="cuda")
    return t.uniform_(-scale, scale, generator=gen)


def _field(case, gen):
    """A real field (nz, ny, nx): a few large waves over broad-band noise."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dt = _real_type(case)
    f = _noise((nz, ny, nx), dt, gen, 0.05)
    par = torch.rand((3, 7), generator=gen, device="cuda").tolist()
    for p in par:
        w = []
        for n, k, ph in ((nz, p[0], p[3]), (ny, p[1], p[4]), (nx, p[2], p[5])):
            a = torch.arange(n, device="cuda", dtype=torch.float64) * (2 * math.pi * int(8 * k) / n)
            w.append(torch.cos(a + 2 * math.pi * ph).to(dt))
        f += (0.2 + p[6]) * (w[0][:, None, None] * w[1][None, :, None]) * w[2][None, None, :]
    return f.reshape(-1)


def _complex_noise(n, case, gen):
    return torch.view_as_complex(_noise((n, 2), _real_type(case), gen))


def _batch_shapes(case):
    g = torch.Generator().manual_seed(case["shape_seed"])
    i = torch.randint(len(BATCH_LENGTHS), (case["grids"], 3), generator=g).tolist()
    return [tuple(BATCH_LENGTHS[k] for k in t) for t in i]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, prec = case["kind"], case["prec"]
    st = {"case": case}
    if kind == "batch":
        st["shapes"] = _batch_shapes(case)
        st["ins"] = [_complex_noise(a * b * c, case, gen) for a, b, c in st["shapes"]]
        st["outs"] = [torch.empty_like(t) for t in st["ins"]]
        st["engines"] = [d2d.decomp_2d_fft_init(d2d.PHYSICAL_IN_X, *s, prec=prec)
                         for s in st["shapes"]]
        st["batch"] = d2d.Batch(st["engines"])
        st["batch"].bind(st["ins"], st["outs"], mode=case["mode"])
        return st
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if kind == "halo":
        st["sizes"] = (nx, ny, nz)
        st["x"] = _field(case, gen)
        h = d2d.halo_shape(st["sizes"], case["level"], case["pencil"])
        st["out"] = torch.zeros(h[0] * h[1] * h[2], dtype=_real_type(case), device="cuda")
        return st
    if kind == "rank":
        st["eng"] = e = d2d.decomp_2d_fft_init(
            d2d.PHYSICAL_IN_X, nx, ny, nz, prec=prec,
            rank=(case["p_row"], case["p_col"], case["row"], case["col"]))
        _, st["sp"] = e.decomps()
        xs, sx, sy, sz = _rank_pencils(case)
        st["x"] = _field({"nx": xs[0], "ny": xs[1], "nz": xs[2], "prec": prec}, gen)
        # what the two exchanges deliver (other ranks' data), and send buffers
        st["recv_y"] = _complex_noise(sy[0] * sy[1] * sy[2], case, gen)
        st["recv_z"] = _complex_noise(sz[0] * sz[1] * sz[2], case, gen)
        ct = _complex_type(case)
        st["send_x"] = torch.empty(sx[0] * sx[1] * sx[2], dtype=ct, device="cuda")
        st["send_y"] = torch.empty(sy[0] * sy[1] * sy[2], dtype=ct, device="cuda")
        st["z"] = torch.empty(sz[0] * sz[1] * sz[2], dtype=ct, device="cuda")
        return st
    if kind == "c2c":
        st["x"] = _complex_noise(nx * ny * nz, case, gen)
        st["spec"] = torch.empty_like(st["x"])
        st["y"] = torch.empty_like(st["x"])
        st["eng"] = d2d.decomp_2d_fft_init(case["fmt"], nx, ny, nz, prec=prec)
        return st
    st["x"] = _field(case, gen)
    st["y"] = torch.empty_like(st["x"])
    if kind == "r2c":
        n = (nx // 2 + 1) * ny * nz if case["fmt"] == 1 else nx * ny * (nz // 2 + 1)
        st["spec"] = torch.empty(n, dtype=_complex_type(case), device="cuda")
        st["eng"] = d2d.decomp_2d_fft_init(case["fmt"], nx, ny, nz, prec=prec)
    else:
        st["spec"] = torch.empty_like(st["x"])
        st["eng"] = d2d.decomp_2d_fft_init(case["fmt"], nx, ny, nz, prec=prec,
                                           opt_DTT=(case["tx"], case["ty"], case["tz"]))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "c2c":
        st["eng"].fft_c2c(st["x"], st["spec"], d2d.FORWARD)
        st["eng"].fft_c2c(st["spec"], st["y"], d2d.BACKWARD)
        return st["spec"], st["y"]
    if kind == "r2c":
        st["eng"].fft_r2c(st["x"], st["spec"])
        st["eng"].fft_c2r(st["spec"], st["y"])
        return st["spec"], st["y"]
    if kind == "dtt":
        st["eng"].dtt_3d_r2r(st["x"], st["spec"], d2d.FORWARD)
        st["eng"].dtt_3d_r2r(st["spec"], st["y"], d2d.BACKWARD)
        return st["spec"], st["y"]
    if kind == "batch":
        st["batch"].launch()
        return tuple(st["outs"])
    if kind == "rank":
        e, sp = st["eng"], st["sp"]
        e.fft_r2c_pack(st["x"], st["send_x"], sp)
        e.exec_1m_unpack_pack("spec_y", st["recv_y"], st["send_y"], d2d.X_TO_Y, d2d.Y_TO_Z, sp,
                              d2d.FORWARD)
        e.exec_1m_unpack("spec_last", st["recv_z"], st["z"], d2d.Y_TO_Z, sp, d2d.FORWARD)
        return st["send_x"], st["send_y"], st["z"]
    d2d.update_halo(d2d.R8 if case["prec"] == 64 else d2d.R4, st["x"], st["out"], st["sizes"],
                    case["level"], case["pencil"], (True, True, True))
    return st["out"]


# ---- what a pass cannot do without ------------------------------------------------


def _fft_flops(n, points):
    """Complex transforms of length n over `points` values in all."""
    return 5.0 * points * math.log2(max(n, 2))


def work(case):
    kind = case["kind"]
    rb = 8 if case["prec"] == 64 else 4
    if kind == "batch":
        both = 2 if case["mode"] == 0 else 1
        pts = [(s, s[0] * s[1] * s[2]) for s in _batch_shapes(case)]
        return {"bytes": sum(2 * 2 * rb * p for _, p in pts),
                "flops": sum(both * sum(_fft_flops(n, p) for n in s) for s, p in pts)}
    if kind == "rank":
        xs, sx, sy, sz = [a * b * c for a, b, c in _rank_pencils(case)]
        return {"bytes": rb * xs + 2 * rb * (sx + 2 * sy + 2 * sz),
                "flops": _fft_flops(case["nx"], xs) / 2 + _fft_flops(case["ny"], sy) +
                _fft_flops(case["nz"], sz)}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    p = nx * ny * nz
    if kind == "halo":
        h = d2d.halo_shape((nx, ny, nz), case["level"], case["pencil"])
        return {"bytes": rb * (p + h[0] * h[1] * h[2]), "flops": 0.0}
    fl = sum(_fft_flops(n, p) for n in (nx, ny, nz))
    if kind == "c2c":  # field -> spectrum, spectrum -> field
        return {"bytes": 4 * 2 * rb * p, "flops": 2 * fl}
    if kind == "r2c":
        n = (nx // 2 + 1) * ny * nz if case["fmt"] == 1 else nx * ny * (nz // 2 + 1)
        return {"bytes": 2 * (rb * p + 2 * rb * n), "flops": fl}
    return {"bytes": 4 * rb * p, "flops": fl}


# ---- the same outputs in 64 bits by plain torch --------------------------------


def _dist(n, p):
    """Block sizes of n points over p ranks (larger blocks last)."""
    return [n // p + (1 if m >= p - n % p else 0) for m in range(p)]


def _rank_pencils(case):
    """Physical x-pencil, spectral x-, y- and z-pencil of the case's rank."""
    nxc = case["nx"] // 2 + 1
    pr, pc, r, c = case["p_row"], case["p_col"], case["row"], case["col"]
    ny_r, ny_c = _dist(case["ny"], pr)[r], _dist(case["ny"], pc)[c]
    nz_c, nx_r = _dist(case["nz"], pc)[c], _dist(nxc, pr)[r]
    return ((case["nx"], ny_r, nz_c), (nxc, ny_r, nz_c), (nx_r, case["ny"], nz_c),
            (nx_r, ny_c, case["nz"]))


def _pack(a, dim, sizes):
    return torch.cat([b.reshape(-1) for b in torch.split(a, sizes, dim)])


def _unpack(flat, shape, dim, sizes):
    out, at = [], 0
    for s in sizes:
        sh = list(shape)
        sh[dim] = s
        n = sh[0] * sh[1] * sh[2]
        out.append(flat[at:at + n].reshape(sh))
        at += n
    return torch.cat(out, dim)


def _r2r(a, kind, dim):
    """Unnormalised DCT-I..IV (1-4), DST-I..IV (5-8) along `dim`, through the
    Fourier transform of the symmetric extension."""
    a = a.movedim(dim, -1)
    n = a.shape[-1]
    f = a.flip(-1)
    if kind == 1:
        e = torch.cat((a, f[..., 1:n - 1]), -1)
        r = torch.fft.rfft(e).real
    elif kind == 5:
        z = torch.zeros_like(a[..., :1])
        e = torch.cat((z, a, z, -f), -1)
        r = -torch.fft.rfft(e).imag[..., 1:n + 1]
    else:
        m = 8 * n if kind in (4, 8) else 4 * n
        e = torch.zeros(a.shape[:-1] + (m,), dtype=a.dtype, device=a.device)
        sg = 1.0 if kind <= 4 else -1.0
        if kind in (2, 4, 6, 8):  # points at odd places, mirrored
            e[..., 1:2 * n:2] = a
            e[..., m - 2 * n + 1::2] = sg * f
        elif kind == 3:
            e[..., :n] = a
            e[..., n + 1:2 * n + 1] = -f
            e[..., 2 * n + 1:3 * n] = -a[..., 1:]
            e[..., 3 * n + 1:] = f[..., :n - 1]
        else:
            e[..., 1:n + 1] = a
            e[..., n + 1:2 * n] = f[..., 1:]
            e[..., 2 * n + 1:3 * n + 1] = -a
            e[..., 3 * n + 1:] = -f[..., 1:]
        s = torch.fft.rfft(e)
        del e
        s = s.real if kind <= 4 else -s.imag
        if kind == 2:
            r = s[..., :n]
        elif kind == 6:
            r = s[..., 1:n + 1]
        elif kind in (3, 7):
            r = 0.5 * s[..., 1:2 * n:2]
        else:
            r = s[..., 1:2 * n:2]
    return r.movedim(-1, dim)


def _dtt_3d(a, case, inverse):
    """Each axis's transform over its default points, the others untouched."""
    inv = {2: 3, 3: 2, 6: 7, 7: 6}
    a = a.clone()
    for dim, t in ((2, case["tx"]), (1, case["ty"]), (0, case["tz"])):
        n = a.shape[dim]
        first = 1 if t in (5, 7) else 0
        cnt = n - (0 if t == 1 else 2 if t == 5 else 1)
        kind = inv.get(t, t) if inverse else t
        v = a.narrow(dim, first, cnt)
        v.copy_(_r2r(v, kind, dim))
    return a


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "batch":
        out = []
        for (nx, ny, nz), t in zip(st["shapes"], st["ins"]):
            a = t.to(torch.complex128).reshape(nz, ny, nx)
            if case["mode"] <= 0:
                a = torch.fft.fftn(a)
            if case["mode"] >= 0:
                a = torch.fft.ifftn(a, norm="forward")
            out.append(a.reshape(-1))
        return tuple(out)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if kind == "halo":
        a = st["x"].reshape(nz, ny, nx)
        for dim, ax in ((2, 1), (1, 2), (0, 3)):
            if ax != case["pencil"]:
                n = a.shape[dim]
                i = torch.arange(-case["level"], n + case["level"], device="cuda") % n
                a = a.index_select(dim, i)
        return a.reshape(-1).double()
    if kind == "rank":
        xs, sx, sy, sz = _rank_pencils(case)
        pr, pc = case["p_row"], case["p_col"]
        x = st["x"].double().reshape(xs[2], xs[1], xs[0])
        send_x = _pack(torch.fft.rfft(x, dim=2), 2, _dist(nx // 2 + 1, pr))
        y = _unpack(st["recv_y"].to(torch.complex128), sy[::-1], 1, _dist(ny, pr))
        send_y = _pack(torch.fft.fft(y, dim=1), 1, _dist(ny, pc))
        z = _unpack(st["recv_z"].to(torch.complex128), sz[::-1], 0, _dist(nz, pc))
        return send_x, send_y, torch.fft.fft(z, dim=0).reshape(-1)
    x = st["x"].reshape(nz, ny, nx)
    del st
    if kind == "c2c":
        s = torch.fft.fftn(x.to(torch.complex128))
        return s.reshape(-1), torch.fft.ifftn(s, norm="forward").reshape(-1)
    if kind == "r2c":
        dim, sz = ((0, 1, 2), (nz, ny, nx)) if case["fmt"] == 1 else ((2, 1, 0), (nx, ny, nz))
        s = torch.fft.rfftn(x.double(), dim=dim).contiguous()
        # unnormalised and the inverse of the above: the field times the points
        return s.reshape(-1), x.reshape(-1).double() * float(nx * ny * nz)
    f = _dtt_3d(x.double(), case, False)
    return f.reshape(-1), _dtt_3d(f, case, True).reshape(-1)
