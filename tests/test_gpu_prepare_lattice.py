"""The MIXED preparation's lattice kernels against the FP64 oracle
(orc_prepare_moments_std_f64: Levinson's recursion, in FP64).

Both solve the same Toeplitz system in FP64, so at MESE bias 1e-3 and these
densities (|u|^2 up to ~0.99) multipliers agree to a small multiple of the
conditioning times 2^-53; the bound is 1e-9 of a pixel's largest multiplier
(f32 multipliers: half an ulp more). Every kernel of the dispatch (4, 8 and 16
lanes per pixel, by image size and by moments) at the edges of its width, dense
and in compact images of ragged counts with empty pixels, and moments outside
the moment space, where the |u|^2 >= 1 guard fires and every later coefficient
is 0."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mray_amd import hip  # noqa: E402
from oracle_ffi import Oracle  # noqa: E402


@pytest.fixture(scope="module")
def O():
    hip.init(0)
    return Oracle()


def densities(rng, n, m):
    """Moments of random piecewise-constant densities in [0.03, 0.97], f32."""
    cut = np.sort(rng.uniform(-np.pi, 0, (n, 4)), axis=1)
    phi = np.concatenate([np.full((n, 1), -np.pi), cut, np.zeros((n, 1))], axis=1)
    val = rng.uniform(0.03, 0.97, (n, 5))
    mo = np.empty((n, m))
    mo[:, 0] = ((phi[:, 1:] - phi[:, :-1]) * val).sum(1) / np.pi
    for j in range(1, m):
        s = np.sin(j * phi)
        mo[:, j] = ((s[:, 1:] - s[:, :-1]) * val).sum(1) / (np.pi * j) * np.exp(-0.5 * (0.05 * j) ** 2)
    return mo.astype(np.float32)


def check(O, mo, lag, nm, bias, tol):
    for i in range(len(nm)):
        ref = O.prepare_std_f64(int(nm[i]), mo[i][:nm[i]].astype(np.float64), float(np.float32(bias)))
        assert np.abs(lag[i][:nm[i]] - ref).max() <= tol * np.abs(ref).max(), (i, nm[i])


# The widths of the dispatch, lanes x elements per lane: images of up to 4096,
# up to 8192 and more pixels take 16, 8 and 4 lanes where that many hold the
# moments, else more.
ELEMENTS = {16: (2, 3, 4, 5, 6, 7, 8, 10, 13, 16), 8: (2, 3, 4, 5, 6, 7, 8, 10, 13),
            4: (2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 18, 20, 22, 24, 25)}
BEYOND_FOUR = tuple(8 * c for c in (16, 20, 24)) + (16 * 13, 16 * 16)
SIZES = {16: ((9, 7), (64, 64)), 8: ((65, 64), (128, 64)), 4: ((129, 64),)}


def widths(lanes):
    own = tuple(lanes * c for c in ELEMENTS[lanes])
    return own + tuple(w for w in BEYOND_FOUR if w > own[-1])


def edges(lanes):
    """Each width full, short of one moment, and one past the width before."""
    w = widths(lanes)
    return sorted({m for lo, hi in zip((0,) + w, w) for m in (lo + 1, hi - 1, hi) if m <= 255})


def cases():
    for lanes, sizes in SIZES.items():
        for m in edges(lanes):
            yield sizes[-1] + (m,)
        for size in sizes[:-1]:
            for m in (1, 2, 7, 8, 33, 50, 100, 101, 129, 193, 255):
                yield size + (m,)


def ragged(rng, n, m):
    nm = rng.integers(0, m + 1, n)
    nm[:40] = np.arange(40) % (m + 1)
    nm[-3:] = (0, 1, m)
    return nm


@pytest.mark.parametrize("W,H,m", list(cases()))
def test_dense(O, W, H, m):
    rng = np.random.default_rng(W * 1000 + m)
    few = densities(rng, min(W * H, 64), m)
    mo = few[np.arange(W * H) % len(few)]
    lag = hip.prepare(torch.from_numpy(mo).cuda(), W, H, m, 1e-3, form="mixed64").cpu().numpy().reshape(-1, m)
    pick = np.unique(np.concatenate([np.arange(3), rng.integers(0, W * H, 12), np.arange(W * H - 3, W * H)]))
    check(O, mo[pick], lag[pick], np.full(len(pick), m), 1e-3, 1e-9)
    f32 = hip.prepare(torch.from_numpy(mo).cuda(), W, H, m, 1e-3, form="mixed").cpu().numpy().reshape(-1, m)
    assert np.array_equal(f32, lag.astype(np.float32))


@pytest.mark.parametrize("lanes", [16, 8, 4])
def test_compact_matches_dense(O, lanes):
    """Ragged counts through every kernel of the dispatch: a pixel of n moments
    gets what an image of n moments gives it, up to the padding's zeros."""
    W, H = SIZES[lanes][-1]
    rng = np.random.default_rng(lanes)
    for m in (w for w in widths(lanes) if w <= 255):
        mo = densities(rng, 64, m)[np.arange(W * H) % 64]
        nm = ragged(rng, W * H, m)
        index = np.concatenate([[0], np.cumsum(nm)]).astype(np.int32)
        data = mo[np.arange(m)[None] < nm[:, None]]
        lag = hip.prepare(torch.from_numpy(data).cuda(), W, H, m, 1e-3, form="mixed64",
                          index=torch.from_numpy(index).cuda()).cpu().numpy()
        pick = np.unique(np.concatenate([np.arange(1, 6), rng.integers(0, W * H, 6), np.arange(W * H - 2, W * H)]))
        pick = pick[nm[pick] > 0]
        check(O, mo[pick], [lag[index[i]:index[i + 1]] for i in pick], nm[pick], 1e-3, 1e-9)


@pytest.mark.parametrize("W,H", [(12, 11), (70, 70), (130, 64)])
def test_compact_ragged(O, W, H):
    m = 60
    rng = np.random.default_rng(W)
    mo = densities(rng, W * H, m)
    nm = ragged(rng, W * H, m)
    index = np.concatenate([[0], np.cumsum(nm)]).astype(np.int32)
    data = np.concatenate([mo[i][:nm[i]] for i in range(W * H)])
    lag = hip.prepare(torch.from_numpy(data).cuda(), W, H, m, 1e-3, form="mixed64",
                      index=torch.from_numpy(index).cuda()).cpu().numpy()
    pick = np.unique(np.concatenate([np.arange(48), rng.integers(0, W * H, 40), np.arange(W * H - 3, W * H)]))
    pick = pick[nm[pick] > 0]
    check(O, mo[pick], [lag[index[i]:index[i + 1]] for i in pick], nm[pick], 1e-3, 1e-9)


@pytest.mark.parametrize("W,H", [(8, 8), (80, 64), (130, 64)])
def test_outside_the_moment_space(O, W, H):
    """A valid prefix, then a jump that no density has: the guard fires there in
    every implementation (|u| far above 1), the later coefficients are 0."""
    m = 24
    rng = np.random.default_rng(5)
    mo = densities(rng, W * H, m)
    mo[:, 12] += 3.0
    mo[::3, 5] -= 2.0
    lag = hip.prepare(torch.from_numpy(mo).cuda(), W, H, m, 1e-3, form="mixed64").cpu().numpy().reshape(-1, m)
    pick = rng.integers(0, W * H, 30)
    check(O, mo[pick], lag[pick], np.full(30, m), 1e-3, 1e-9)


def fd_gradient(O, mo, gl, bias, eps=1e-6):
    """Central differences of sum(gl * prepare(mo)) in the FP64 oracle."""
    out = np.empty(len(mo))
    for j in range(len(mo)):
        v = []
        for s in (eps, -eps):
            x = mo.astype(np.float64).copy()
            x[j] += s
            v.append(float(gl.astype(np.float64) @ O.prepare_std_f64(len(mo), x, float(np.float32(bias)))))
        out[j] = (v[0] - v[1]) / (2 * eps)
    return out


# 4, 8 and 16 lanes per pixel (up to 40, 80 and 255 moments), their block edges
@pytest.mark.parametrize("m", [1, 2, 8, 9, 39, 40, 41, 63, 80, 81, 160, 161, 255])
def test_adjoint_against_differences(O, m):
    """dL/dmoments against differences of the FP64 oracle. At MESE bias 0.05 the
    solution's condition number stays below ~1e3, so the differences (step
    1e-6) are good to ~1e-8 of the gradient's norm; the kernel rounds to f32
    once: 1e-5 leaves both a factor of 100."""
    W, H, bias = 3, 7, 0.05
    rng = np.random.default_rng(m)
    mo = densities(rng, W * H, m)
    gl = rng.normal(size=(W * H, m)).astype(np.float32)
    gm = hip.prepare_backward(torch.from_numpy(mo).cuda(), W, H, m, bias, torch.from_numpy(gl).cuda())
    gm = gm.cpu().numpy().reshape(-1, m).astype(np.float64)
    for i in (0, 10, W * H - 1):
        ref = fd_gradient(O, mo[i], gl[i], bias)
        assert np.linalg.norm(gm[i] - ref) <= 1e-5 * np.linalg.norm(ref), (i, np.linalg.norm(gm[i] - ref) / np.linalg.norm(ref))


def test_adjoint_past_the_guard(O):
    """Where the guard fires (order 12 of 24) the later coefficients are constants."""
    W, H, m, bias = 4, 4, 24, 0.05
    rng = np.random.default_rng(9)
    mo = densities(rng, W * H, m)
    mo[:, 12] += 3.0
    gl = rng.normal(size=(W * H, m)).astype(np.float32)
    gm = hip.prepare_backward(torch.from_numpy(mo).cuda(), W, H, m, bias, torch.from_numpy(gl).cuda())
    gm = gm.cpu().numpy().reshape(-1, m).astype(np.float64)
    for i in range(4):
        ref = fd_gradient(O, mo[i], gl[i], bias)
        assert np.linalg.norm(gm[i] - ref) <= 1e-5 * np.linalg.norm(ref)


def test_adjoint_compact_matches_dense(O):
    """Ragged counts with empty pixels, every lane group: a pixel's gradient does
    not depend on the image's largest count (up to FP64 rounding, then f32)."""
    W, H, bias = 9, 8, 0.05
    rng = np.random.default_rng(3)
    nm = rng.integers(0, 41, W * H)
    nm[:5] = (0, 1, 2, 40, 39)
    mo = densities(rng, W * H, 40)
    index = np.concatenate([[0], np.cumsum(nm)]).astype(np.int32)
    data = np.concatenate([mo[i][:nm[i]] for i in range(W * H)])
    gl = rng.normal(size=len(data)).astype(np.float32)
    dev = [torch.from_numpy(a).cuda() for a in (data, gl, index)]
    out = [hip.prepare_backward(dev[0], W, H, m, bias, dev[1], index=dev[2]).cpu().numpy().astype(np.float64)
           for m in (40, 64, 120, 255)]
    for i in np.flatnonzero(nm):
        a = slice(index[i], index[i + 1])
        for o in out[1:]:
            assert np.linalg.norm(o[a] - out[0][a]) <= 1e-6 * np.linalg.norm(out[0][a])
