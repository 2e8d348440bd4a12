"""The framework's work as cases that can be timed: whole Born-scattering simulations.

A case is a dict of plain values: the grid (nx, ny, nz), the number of materials and
energies, the E-angle triple (start, step, end), voxel size, options, precision, and how
the program calls the library (`via`):

  device   cyr_simulate_device, morphology and patterns resident on the GPU
  host     cyr_simulate, numpy morphology in and numpy patterns out
  batch    cyr_simulate_batch over several uneven simulations

prepare() makes what a program holds before the call, run() is one simulation (every
energy and angle), exact() the same patterns from a plain torch pipeline in 64 bits.
"""
import math

import numpy as np
import torch

from cyrsoxs_amd import capi, synthetic

PIPES = {"auto": capi.PIPE_AUTO, "plain": capi.PIPE_PLAIN}
STORES = {"native": capi.STORE_NATIVE, "fp16": capi.STORE_FP16, "bf16": capi.STORE_BF16}

DEFAULTS = dict(via="device", field="bulk", materials=2, energies=1, e0=280.0, estep=1.0, a0=0.0, astep=10.0, a1=170.0,
                phys=2.0, linear=True, hann=False, rotmask=False, material_frame=False, vector=False, bits=32,
                storage="native", pipeline="auto", members=1)


def _case(name, nx, ny, nz, **kw):
    c = dict(DEFAULTS, nx=nx, ny=ny, nz=nz, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's shipped example: a small vector morphology, one energy, one angle,
        # nearest neighbour, from host arrays (a first script, or one step of a fitting loop)
        _case("example_host", 32, 32, 16, via="host", vector=True, phys=5.0, linear=False, a1=0.0, astep=1.0),
        # the 64^3 two-material sphere: 3 energies x 6 angles, nearest neighbour (a form-factor check)
        _case("sphere64", 64, 64, 64, field="sphere", energies=3, e0=284.0, astep=30.0, a1=150.0, phys=5.0,
              linear=False),
        # the same in double precision with linear interpolation and the window (a convergence check)
        _case("sphere64_fp64", 64, 64, 64, field="sphere", energies=3, e0=284.0, astep=30.0, a1=150.0, phys=5.0,
              hann=True, bits=64),
        # realistic bulk morphology at full size: 20 energies x 36 angles
        _case("bulk512", 512, 512, 128, materials=4, energies=20, astep=5.0, a1=175.0, hann=True),
        # the thin-film study: 50 energies x 180 angles on a 2048^2 plane
        _case("film2048", 2048, 2048, 1, field="film", materials=3, energies=50, estep=0.5, astep=2.0, a1=358.0,
              phys=1.0),
        # a smaller film in double precision with the rotation mask
        _case("film512_fp64_mask", 512, 512, 1, field="film", materials=3, energies=10, estep=0.5, astep=5.0, a1=355.0,
              phys=1.0, rotmask=True, bits=64),
        # several uneven morphologies handed over together
        _case("batch_uneven", 384, 384, 48, via="batch", materials=3, energies=16, members=4),
        # one energy of a bulk morphology (a look at one resonance)
        _case("one_energy256", 256, 256, 64, materials=3, e0=285.0, astep=5.0, a1=175.0, hann=True),
        # a grid whose sides are round numbers, not powers of two, not square
        _case("round_200x240x50", 200, 240, 50, materials=3, energies=12, hann=True),
        # a grid cut from measured data: sides of no special form, not square
        _case("cut_101x94x21", 101, 94, 21, materials=2, energies=4, astep=15.0, a1=165.0, hann=True),
        # patterns in the sample's frame, with the rotation mask and 16-bit morphology storage
        _case("sample_frame128", 128, 128, 32, materials=2, energies=6, astep=10.0, a1=170.0, material_frame=True,
              rotmask=True, storage="fp16", hann=True),
        # the reference's per-angle structure, which the Python binding's descriptor selects by default
        _case("per_angle128", 128, 128, 32, materials=2, energies=2, astep=30.0, a1=150.0, pipeline="plain"),
    ]


ANGLES = ((0.0, 1.0, 0.0), (0.0, 30.0, 150.0), (0.0, 15.0, 165.0), (0.0, 10.0, 170.0), (0.0, 5.0, 175.0),
          (0.0, 5.0, 355.0), (0.0, 2.0, 358.0), (0.0, 7.0, 175.0))


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A side length: a power of two, a round number or any number."""
    n = _log(rng, lo, hi)
    how = rng.random()
    if how < 0.35:
        return min(hi, max(lo, 1 << int(round(math.log2(n)))))
    if how < 0.75:
        while not _smooth(n):
            n += 1 if n < hi else -1
    return n


def draw(rng):
    """One more simulation of the ranges above."""
    kind = rng.choice(("small", "bulk", "bulk", "film"))
    c = _case(None, 0, 0, 0)
    if kind == "small":
        c["nx"], c["ny"], c["nz"] = _side(rng, 16, 80), _side(rng, 16, 80), _side(rng, 8, 80)
        c.update(materials=rng.randint(1, 3), energies=rng.randint(1, 5), phys=rng.choice((5.0, 2.0)),
                 via=rng.choice(("host", "device")))
    elif kind == "bulk":
        c["nx"] = _side(rng, 96, 512)
        c["ny"] = c["nx"] if rng.random() < 0.6 else _side(rng, 96, 512)
        c["nz"] = _side(rng, 12, 128)
        c.update(materials=rng.randint(2, 4), energies=_log(rng, 1, 24), phys=rng.choice((5.0, 2.0)))
    else:
        c["nx"] = _side(rng, 128, 2048)
        c["ny"] = c["nx"] if rng.random() < 0.7 else _side(rng, 128, 2048)
        c["nz"] = 1
        c.update(field="film" if c["nx"] == c["ny"] else "bulk", materials=3, energies=_log(rng, 1, 40), phys=1.0)
    c["a0"], c["astep"], c["a1"] = rng.choice(ANGLES)
    c.update(e0=rng.choice((280.0, 284.0)), estep=rng.choice((1.0, 0.5)), linear=rng.random() < 0.75,
             hann=kind != "film" and rng.random() < 0.6, rotmask=rng.random() < 0.25,
             material_frame=rng.random() < 0.15, vector=kind != "film" and rng.random() < 0.25,
             bits=64 if rng.random() < 0.25 else 32)
    if c["bits"] == 32 and rng.random() < 0.15:
        c["storage"] = rng.choice(("fp16", "bf16"))
    sides = (c["nx"], c["ny"], c["nz"])
    if kind == "small" and rng.random() < 0.2:
        c["pipeline"] = "plain"
    # sides of no special form occur on grids of moderate size: fewer energies and angles there
    if not all(_smooth(n) for n in sides):
        v = c["nx"] * c["ny"] * c["nz"]
        while (50e-6 + v * sum(sides) * 24 / 1.5e12 * c["bits"] / 32) * c["energies"] * _angles(c) > 1.0:
            if c["energies"] > 4:
                c["energies"] = c["energies"] // 2
            elif _angles(c) > 12:
                c["astep"], c["a1"] = 15.0, 165.0
            else:
                c["nx"], c["ny"] = c["nx"] * 3 // 4, c["ny"] * 3 // 4
                if c["nx"] != c["ny"]:
                    c["field"] = "bulk"
                sides = (c["nx"], c["ny"], c["nz"])
                v = c["nx"] * c["ny"] * c["nz"]
    return c


# ---- inputs ---------------------------------------------------------------------

def _energies(c):
    return [c["e0"] + c["estep"] * i for i in range(c["energies"])]


def _angles(c):
    return int(round((c["a1"] - c["a0"]) / c["astep"] + 1))


def _members(c):
    """The simulations of a case: itself, or the uneven members of a batch."""
    if c["via"] != "batch":
        return [c]
    grids = [(c["nx"], c["ny"], c["nz"]), (128, 128, 32), (256, 256, 64), (512, 512, 64)]
    out = []
    for i in range(c["members"]):
        nx, ny, nz = grids[i % len(grids)]
        out.append(dict(c, nx=nx, ny=ny, nz=nz, materials=2 + (c["materials"] + i) % 3,
                        energies=max(1, c["energies"] - 3 * i)))
    return out


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rand(shape, gen, normal=False):
    f = torch.randn if normal else torch.rand
    return f(shape, generator=gen, device=gen.device, dtype=torch.float32)


def _morphology(c, seed):
    """[M][V][4] on the GPU: Euler (S, theta, psi, Vfrac) or vector (sx, sy, sz, phi_u)."""
    dt = torch.float64 if c["bits"] == 64 else torch.float32
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 17)
    M, shape = c["materials"], (c["nz"], c["ny"], c["nx"])
    V = c["nx"] * c["ny"] * c["nz"]
    if c["field"] == "film" and c["nx"] == c["ny"] and M == 3:
        return synthetic.thinfilm_morphology(c["nx"], seed=seed, device=dev, dtype=dt)
    out = torch.empty((M, V, 4), dtype=dt, device=dev)
    if c["field"] == "sphere":
        # a sphere near the centre with a radial director and its isotropic complement
        n = c["nx"]
        shift = _rand((4,), gen).double()
        centre = n / 2 + 4 * (shift[:3] - 0.5)
        radius = n * (0.28 + 0.08 * float(shift[3]))
        ax = torch.arange(n, device=dev, dtype=torch.float64)
        rz, ry, rx = torch.meshgrid(ax - centre[2], ax - centre[1], ax - centre[0], indexing="ij")
        r = torch.sqrt(rx * rx + ry * ry + rz * rz).clamp_min(1e-9)
        inside = (r <= radius).double()
        out.zero_()
        out[0, :, 0] = 1.0
        out[0, :, 1] = torch.arccos((rz / r).clamp(-1, 1)).reshape(V).to(dt)
        out[0, :, 2] = torch.atan2(ry, rx).reshape(V).to(dt)
        out[0, :, 3] = inside.reshape(V).to(dt)
        out[1, :, 3] = (1 - inside).reshape(V).to(dt)
        return out
    sigma = min(6.0, min(c["nx"], c["ny"]) / 12)

    def smooth(normal):
        f = _rand(shape, gen, normal)
        f = synthetic.gaussian_filter_periodic(f if c["nz"] > 1 else f[0], sigma).reshape(V)
        return f

    logits = torch.stack([smooth(True) for _ in range(M)])
    logits = (logits - logits.mean(1, keepdim=True)) / (logits.std(1, keepdim=True) + 1e-12)
    vf = torch.softmax(logits, 0)
    for m in range(M):
        s = smooth(False)
        s = (s - s.min()) / (s.max() - s.min() + 1e-12)
        theta = torch.arccos(1 - 2 * _rand((V,), gen))
        psi = 2 * math.pi * _rand((V,), gen)
        if c["vector"]:
            # aligned part along the director with length sqrt(Vfrac S), the rest unaligned
            w = torch.sqrt(vf[m] * s)
            out[m, :, 0] = (w * torch.sin(theta) * torch.cos(psi)).to(dt)
            out[m, :, 1] = (w * torch.sin(theta) * torch.sin(psi)).to(dt)
            out[m, :, 2] = (w * torch.cos(theta)).to(dt)
            out[m, :, 3] = (vf[m] * (1 - s)).to(dt)
        else:
            out[m, :, 0], out[m, :, 1], out[m, :, 2], out[m, :, 3] = s.to(dt), theta.to(dt), psi.to(dt), vf[m].to(dt)
    return out


def _inputs(c, seed):
    """(morphology as the library reads it, optical constants)."""
    vox = _morphology(c, seed)
    if c["storage"] == "fp16":
        vox = vox.to(torch.float16)
    elif c["storage"] == "bf16":
        vox = vox.to(torch.bfloat16)
    if c["field"] == "sphere":
        mats = synthetic.sphere_constants(_energies(c))
    elif c["energies"] > 1:
        mats = synthetic.lorentzian_constants(_energies(c), c["materials"], seed=seed)
    else:
        mats = np.random.default_rng(seed).uniform(1e-4, 3e-3, (1, c["materials"], 4))
        mats[:, :, [0, 2]] = 1 - mats[:, :, [0, 2]]
    return vox, mats


def _sim(c):
    return capi.Sim((c["nx"], c["ny"], c["nz"]), c["materials"], c["phys"], _energies(c), (c["a0"], c["astep"], c["a1"]),
                    morphology_type=int(c["vector"]), reference_frame=0 if c["material_frame"] else 1,
                    interpolation=int(c["linear"]), windowing=int(c["hann"]), rot_mask=int(c["rotmask"]),
                    precision=capi.FP64 if c["bits"] == 64 else capi.FP32, storage=STORES[c["storage"]],
                    pipeline=PIPES[c["pipeline"]])


def prepare(case, seed):
    sims, voxels, mats, outs = [], [], [], []
    for i, c in enumerate(_members(case)):
        sim = _sim(c)
        vox, m = _inputs(c, seed + 101 * i)
        if case["via"] == "host":  # host arrays hold the compute precision, whatever the device storage
            vox = vox.to(torch.float64 if c["bits"] == 64 else torch.float32).cpu().numpy()
            outs.append(None)
        else:
            outs.append(torch.empty((c["energies"], 1, c["ny"], c["nx"]),
                                    dtype=torch.float64 if c["bits"] == 64 else torch.float32, device=_device()))
        sims.append(sim)
        voxels.append(vox)
        mats.append(m)
    return dict(via=case["via"], sims=sims, voxels=voxels, mats=mats, outs=outs)


def run(state):
    if state["via"] == "host":
        return capi.simulate(state["sims"][0], state["voxels"][0], state["mats"][0])
    if state["via"] == "batch":
        capi.simulate_batch(state["sims"], state["voxels"], state["mats"], state["outs"])
        return state["outs"]
    capi.simulate_device(state["sims"][0], state["voxels"][0], state["mats"][0], state["outs"][0])
    return state["outs"][0]


def work(case):
    """Morphology read once and patterns written once; the transforms of the fewer of 5
    complex tensor fields per energy and 7 real fields per material, every pixel's fields
    and intensity per energy, and its bilinear sample per angle."""
    nbytes = flops = 0.0
    for c in _members(case):
        real = c["bits"] // 8
        V, P, E = c["nx"] * c["ny"] * c["nz"], c["nx"] * c["ny"], c["energies"]
        store = 2 if c["storage"] != "native" and c["via"] != "host" else real
        nbytes += 4.0 * c["materials"] * V * store + E * P * real
        flops += 5.0 * V * math.log2(V) * min(5 * E, 3.5 * c["materials"])
        flops += E * P * (7 * 2 * 4 * c["materials"] + 60 + 12.0 * _angles(c))
    return {"bytes": nbytes, "flops": flops}


# ---- the same patterns in 64 bits ------------------------------------------------

def _unshift(n, dev):
    x = torch.arange(n, device=dev)
    m = n // 2
    return torch.where(x <= m, m - x, n + m - x)


def _basis(c, vox, m):
    """Material m in 64 bits: isotropic weights (of b and of c) and s_i s_j weighted by phi_a."""
    v = vox[m].double()
    if c["vector"]:
        s = [v[:, 0], v[:, 1], v[:, 2]]
        pa = torch.ones_like(v[:, 0])
        alpha, beta = s[0] * s[0] + s[1] * s[1] + s[2] * s[2], v[:, 3]
    else:
        st = torch.sin(v[:, 1])
        s = [torch.cos(v[:, 2]) * st, torch.sin(v[:, 2]) * st, torch.cos(v[:, 1])]
        pa = v[:, 3] * v[:, 0]
        alpha, beta = pa, v[:, 3] - pa
    return alpha, beta, [pa * s[i] * s[j] for i, j in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2))]


def _fields(c, vox, mats, e):
    """Spectra of N00, N01, N02, N11, N12 (contrast tensor / 4 pi) of one energy, DC replaced."""
    V = c["nx"] * c["ny"] * c["nz"]
    N = torch.zeros((5, V), dtype=torch.complex128, device=vox.device)
    for m in range(c["materials"]):
        npar, nper = complex(mats[e, m, 0], mats[e, m, 1]), complex(mats[e, m, 2], mats[e, m, 3])
        niso = (npar + 2 * nper) / 3
        alpha, beta, ss = _basis(c, vox, m)
        d = npar * npar - nper * nper
        for j in range(5):
            N[j] += d * ss[j]
        iso = (nper * nper - 1) * alpha + (niso * niso - 1) * beta
        N[0] += iso
        N[3] += iso
    N = N.reshape(5, c["nz"], c["ny"], c["nx"]) / (4 * math.pi)
    if c["hann"]:
        for ax, n in ((1, c["nz"]), (2, c["ny"]), (3, c["nx"])):
            if n > 1:
                w = 0.5 * (1 - torch.cos(2 * math.pi * torch.arange(n, device=vox.device, dtype=torch.float64) / n))
                N *= w.reshape([-1 if a == ax else 1 for a in range(4)])
    for j in range(5):
        N[j] = torch.fft.fftn(N[j])
    near = [N[:, 0, 0, 1], N[:, 0, 0, -1], N[:, 0, 1, 0], N[:, 0, -1, 0]]
    if c["nz"] > 1:
        near += [N[:, 1, 0, 0], N[:, -1, 0, 0]]
    N[:, 0, 0, 0] = sum(near) / len(near)
    return N


def _simulate64(c, vox, mats):
    dev = vox.device
    nx, ny, nz, nE = c["nx"], c["ny"], c["nz"], c["energies"]
    three = nz > 1
    f8 = dict(dtype=torch.float64, device=dev)
    start = -(math.pi / c["phys"])
    dx, dy = (2 * math.pi / c["phys"]) / (nx - 1), (2 * math.pi / c["phys"]) / (ny - 1)
    dz = (2 * math.pi / c["phys"]) / (nz - 1) if three else 0.0
    X, Y = torch.arange(nx, **f8)[None, :], torch.arange(ny, **f8)[:, None]
    px, py = start + X * dx, start + Y * dy
    ix, iy = _unshift(nx, dev), _unshift(ny, dev)
    bins = 2 if three and c["linear"] else 1
    fields, matrices, weight, dead = [], [], [], []
    for e in range(nE):
        k = 2 * math.pi / (1239.84197 / _energies(c)[e])
        val = k * k - px * px - py * py
        bad = (val < 0) | (X == nx - 1) | (Y == ny - 1)
        posz = -k + torch.sqrt(val.clamp_min(0))
        z0, f = torch.zeros((ny, nx), dtype=torch.long, device=dev), torch.zeros((ny, nx), **f8)
        if three:
            t = (posz - start) / dz
            if c["linear"]:
                z0 = torch.trunc(t).long()
                bad = bad | ~(t > -1.0) | (z0 + 1 > nz - 1)
                z0 = z0.clamp(0, nz - 2)
                f = (posz - (start + z0.double() * dz)) / dz
            else:
                r = torch.sign(t) * torch.floor(t.abs() + 0.5)
                bad = bad | (r < 0) | (r > nz - 1)
                z0 = r.clamp(0, nz - 1).long()
        N = _fields(c, vox, mats, e)
        vz0 = start + z0.double() * dz if three else 0.0 * posz
        rows, mats6 = [], []
        for q in range(bins):
            kz = _unshift(nz, dev)[z0 + q] if three else z0
            rows.append(N[:, kz, iy[:, None], ix[None, :]])
            vz = k + vz0 + q * dz
            kk = k * k
            mats6.append(torch.stack([kk - px * px + 0 * vz, -px * py + 0 * vz, -px * vz, kk - py * py + 0 * vz, -py * vz,
                                      kk - vz * vz]))
        del N
        fields.append(torch.stack(rows))
        matrices.append(torch.stack(mats6))
        weight.append(f)
        dead.append(bad)
    F, M6 = torch.stack(fields), torch.stack(matrices)  # [nE][bins][5 | 6][ny][nx]
    weight, dead = torch.stack(weight), torch.stack(dead)
    total, count = torch.zeros((nE, ny, nx), **f8), torch.zeros((nE, ny, nx), **f8)
    nA = _angles(c)
    for a in range(nA):
        th = (c["a0"] + a * c["astep"]) * math.pi / 180
        co, si = math.cos(th), math.sin(th)
        image = torch.zeros((nE, ny, nx), **f8)
        for q in range(bins):
            # E = (cos, sin, 0): p = N E, in the sample's frame R^T p with R the turn by the angle about z
            p = [co * F[:, q, 0] + si * F[:, q, 1], co * F[:, q, 1] + si * F[:, q, 3], co * F[:, q, 2] + si * F[:, q, 4]]
            if c["material_frame"]:
                p = [co * p[0] + si * p[1], -si * p[0] + co * p[1], p[2]]
            m = M6[:, q]
            part = 0
            for i, j, l in ((0, 1, 2), (1, 3, 4), (2, 4, 5)):
                s = m[:, i] * p[0] + m[:, j] * p[1] + m[:, l] * p[2]
                part = part + s.real ** 2 + s.imag ** 2
            image = image + part * (1.0 if bins == 1 else (weight if q else 1 - weight))
        image[dead] = math.nan
        # bilinear turn about (nx/2, ny/2), as the inverse of the forward map
        c2, c5 = (1 - co) * nx / 2 - si * ny / 2, si * nx / 2 + (1 - co) * ny / 2
        det = co * co + si * si
        i00, i01, i10, i11 = co / det, -si / det, si / det, co / det
        sx = i00 * X + i01 * Y + -(i00 * c2 + i01 * c5)
        sy = i10 * X + i11 * Y + -(i10 * c2 + i11 * c5)
        inside = (sx >= 0) & (sx <= nx - 1) & (sy >= 0) & (sy <= ny - 1)
        x0, y0 = torch.floor(sx).clamp(0, nx - 1), torch.floor(sy).clamp(0, ny - 1)
        fx, fy = torch.where(inside, sx - x0, 0.0), torch.where(inside, sy - y0, 0.0)
        x0, y0 = x0.long(), y0.long()
        x1, y1 = (x0 + 1).clamp_max(nx - 1), (y0 + 1).clamp_max(ny - 1)
        flat = image.reshape(nE, -1)
        got = torch.zeros((nE, ny * nx), **f8)
        for yy, xx, w in ((y0, x0, (1 - fx) * (1 - fy)), (y0, x1, fx * (1 - fy)), (y1, x0, (1 - fx) * fy), (y1, x1, fx * fy)):
            w = w.reshape(-1)
            got += torch.where(w != 0, w * flat[:, (yy * nx + xx).reshape(-1)], 0.0)
        got = got.reshape(nE, ny, nx)
        got[:, ~inside] = math.nan
        if c["rotmask"]:
            fine = ~torch.isnan(got)
            total += torch.where(fine, got, 0.0)
            count += fine
        else:
            total += got
    if c["rotmask"]:
        total = torch.where(count > 0, total / count.clamp_min(1), 0.0)
    else:
        total = total / nA
    return total.reshape(nE, 1, ny, nx)


def exact(case, seed):
    outs = []
    for i, c in enumerate(_members(case)):
        vox, mats = _inputs(c, seed + 101 * i)
        if case["via"] == "host" and c["storage"] != "native":
            vox = vox.to(torch.float32)
        outs.append(_simulate64(c, vox, mats))
        torch.cuda.empty_cache()
    if case["via"] == "batch":
        return outs
    return outs[0].cpu().numpy() if case["via"] == "host" else outs[0]
