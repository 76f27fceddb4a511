"""Band-limited states (2/3 filter, zero outside the disk |k| < Nx/3) against
the same states with one negligible mode outside the disk, which sends every
call down the path over all modes: RK4CN and CN-AB4 steps (direct and
graph-replayed), the measures with fluxes, the CFL rate, an ensemble, the
adjoint, a handle that is given both kinds of state in turn, and a state that
blows up.  Used on the CPU emulation and on the GPU (tests/test_band_limited.py).

Both paths do the same arithmetic on the disk's modes; 1e-13 (relative L2)
allows for a rounding of each of a few steps' transforms."""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, os.path.join(ROOT, "2d-navier-stokes_amd"))

import numpy as np  # noqa: E402

import ns2d  # noqa: E402
from ns2d import ics  # noqa: E402

TOL = 1e-13
# the emulation's wave barriers do not follow a wave whose lanes diverge, so its wave maxima are not compared
EMULATED = os.environ.get("NS2D_NO_TORCH") == "1"


def disk(nx, ny):
    kx, ky = ics.wavenumbers(nx, ny)
    return kx * kx + ky * ky < (nx // 3) ** 2


def field(nx, ny, seed):
    """A band-limited state with a non-Hermitian ky = 0 entry, filling the disk."""
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((nx, ny // 2 + 1)) + 1j * rng.standard_normal((nx, ny // 2 + 1))
    w *= disk(nx, ny) * (0.1 * nx * ny)
    w[0, 0] = 0.0
    return w


def outside(w):
    """w with one mode outside the disk too small to change a sum."""
    v = w.copy()
    v[w.shape[0] // 2, 0] = 1e-280
    return v


def close(a, b, what):
    assert np.all(np.isfinite(a)) and np.linalg.norm(a - b) <= TOL * np.linalg.norm(b), what


def cfg(nx, ny, **kw):
    base = dict(Nx=nx, Ny=ny, nu=1e-3, hyper_flag=0, hyper_pow=1.0, filter="23")
    base.update(kw)
    return ns2d.Config(**base)


def steps(c, w, n, kv=None, rv=None, dt=1e-4):
    with ns2d.Solver(c) as s:
        if kv is not None:
            s.set_kpass_variant(kv)
        if rv is not None:
            s.set_rpass_variant(rv)
        s.set_state(w)
        s.spectral_step(dt, n)
        got = s.get_state()
        mx, conv = s.max_vort(), s.cfl_rate()
        m = s.system_measures(with_flux=True)
        s.spectral_step(dt, 1)
        return got, s.get_state(), mx, conv, m


def same(a, b, what):
    for i in (0, 1):
        close(a[i], b[i], (what, i))
    assert EMULATED or (abs(a[2] - b[2]) <= TOL * abs(b[2]) and abs(a[3] - b[3]) <= TOL * abs(b[3])), what
    for k, v in b[4].items():
        if "divergence" in k or "_sbst" in k or "d_" in k:   # sums that vanish up to rounding
            continue
        scale = np.linalg.norm(np.atleast_1d(v))
        if "flux" in k:   # bins of conserved sums: |2 Re(conj(w) K)| <= 2 max(pi (|u|/dx + |v|/dy)) |w|^2
            scale += 2.0 * max(b[3], 1.0) * np.linalg.norm(b[4]["enst_spect"])
        assert np.linalg.norm(np.atleast_1d(a[4][k] - v)) <= 1e-12 * scale, (what, k)


def shapes(nx, ny, kvs, rvs):
    """RK4CN over the given column- and row-pass shapes."""
    w = field(nx, ny, nx + 7 * ny)
    ref = steps(cfg(nx, ny), outside(w), 6)
    m = disk(nx, ny)
    for kv, rv in [(k, None) for k in kvs] + [(None, r) for r in rvs]:
        got = steps(cfg(nx, ny), w, 6, kv, rv)
        same(got, ref, (nx, ny, kv, rv))
        if kv is None or not ns2d.kpass_variants(nx)[kv]["packed_pair"]:
            assert np.all(got[0][~m] == 0.0)


def options(nx, ny):
    """Integrators, quirks and forcing."""
    w = field(nx, ny, 5 * nx + ny)
    kf = max(1, min(2, nx // 3 - 1))
    for kw in (dict(quirks=0), dict(integrator="AB4"),
               dict(integrator="AB4", forcing="KOLM", force_k=kf, force_scale=0.5, alpha=0.01, drag_flag=1, drag_pow=0.0),
               dict(forcing="KOLM", force_k=min(nx // 3, ny // 2), force_scale=0.5),   # outside the disk
               dict(check_every=0, hyper_flag=1, hyper_pow=2.0)):
        c = cfg(nx, ny, **kw)
        same(steps(c, w, 9), steps(c, outside(w), 9), (nx, ny, kw))


def turns(nx, ny):
    """One handle, band-limited and other states in turn; the RHS between steps."""
    w, v = field(nx, ny, 1), ics.random_phase(nx, ny, seed=2, k0=3.0, e0=0.5, filt="none")
    v[nx // 2, :] += 0.3 * np.abs(v).max()
    for kw in (dict(), dict(integrator="AB4")):
        c = cfg(nx, ny, **kw)
        with ns2d.Solver(c) as s:
            for x in (w, v, w, v, w):
                s.set_state(x)
                s.spectral_step(1e-4, 5)
                y = s.get_state()
                close(y, steps(c, outside(x) if x is w else x, 5)[0], (nx, ny, kw))
                m = s.system_measures()
                e = ics.energy(y, nx, ny)
                assert abs(m["energy"] - e) <= 1e-12 * e
            with ns2d.Solver(c) as g:
                g.set_state(outside(y))
                s.set_state(y)
                for _ in range(2):
                    for z in (s, g):
                        z.nonlinear_rhs(v)
                        z.spectral_step(1e-4, 3)
                    close(s.get_state(), g.get_state(), (nx, ny, kw, "rhs"))


def ensembles(nx, ny):
    ws = [field(nx, ny, i) for i in range(3)]
    dts = [1e-4, 2e-4, 1.5e-4]
    refs = [steps(cfg(nx, ny), outside(w), 5, dt=d)[0] for w, d in zip(ws, dts)]
    with ns2d.Ensemble([cfg(nx, ny)] * 3) as e:
        for mixed in (False, True, False):
            for i, (m, w) in enumerate(zip(e.members, ws)):
                m.set_state(outside(w) if mixed and i == 1 else w)
            e.step(dts, 3)
            e.members[0].max_vort()   # a call of a member's own between ensemble steps
            e.step(dts, 2)
            for m, r in zip(e.members, refs):
                close(m.get_state(), r, (nx, ny, mixed))


def adjoint(nx, ny):
    w = field(nx, ny, 3)
    lam = field(nx, ny, 4) + 0.1 * ics.random_phase(nx, ny, seed=6, k0=3.0, e0=0.5, filt="none")
    c = cfg(nx, ny, quirks=0, check_every=0)
    with ns2d.Solver(c) as s, ns2d.Solver(c) as g:
        for ck in (0, 2, 2):
            close(s.vjp(w, 1e-4, 8, lam, ckpt_every=ck), g.vjp(outside(w), 1e-4, 8, lam, ckpt_every=ck), (nx, ny, ck))
        close(s.vjp(outside(w), 1e-4, 8, lam, ckpt_every=2), g.vjp(w, 1e-4, 8, lam, ckpt_every=2), (nx, ny, "swapped"))


def blown_up(nx, ny):
    """A state that overflows leaves NaN in every mode but (0, 0) on both paths."""
    w = field(nx, ny, 8) * 1e160
    for x in (w, outside(w)):
        with ns2d.Solver(cfg(nx, ny)) as s:
            s.set_state(x)
            try:
                s.spectral_step(1.0, 4)
            except ns2d.NS2DError as err:
                assert err.code == ns2d.NS2D_ERR_BLOWUP
            else:
                raise AssertionError("no blow-up reported")
            y = s.get_state()
            y[0, 0] = np.nan
            assert np.all(np.isnan(y.real) | np.isnan(y.imag)), (nx, ny)


def case(nx, ny, every_shape):
    k, r = len(ns2d.kpass_variants(nx)), len(ns2d.rpass_variants(ny))
    shapes(nx, ny, range(k) if every_shape else [0], range(r) if every_shape else [0])
    options(nx, ny)
    turns(nx, ny)
    ensembles(nx, ny)
    adjoint(nx, ny)
    if not EMULATED:
        blown_up(nx, ny)
    print(f"band {nx}x{ny} OK", flush=True)


if __name__ == "__main__":
    for a in sys.argv[1:]:
        x, y = (int(t) for t in a.split("x"))
        case(x, y, True)
    print("BAND OK", flush=True)
