"""Lengths at the upper end of the kernels of any length, against pocketfft
and the oracle: those whose best schedule would need more rows than a
workgroup has threads (6125 = 5^3 7^2, 5250 points of a real-to-real stage).

Tolerances: those of test_gpu_mixed.py (1e-13 FP64, 5e-6 FP32; real-to-real
1e-13, 2e-6; relative L2)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {64: 1e-13, 32: 5e-6}
RTOL = {64: 1e-13, 32: 2e-6}


def dev(torch, a, dt):
    return torch.from_numpy(np.ascontiguousarray(a.ravel(order="F")).astype(dt)).to("cuda")


def host(t, shape):
    return t.cpu().numpy().reshape(shape, order="F")


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec", [64, 32])
def test_long_lengths(d2d, torch_gpu, axis, prec):
    n = 6125
    shape = [3, 2, 2]
    shape[axis] = n
    shape = tuple(shape)
    rng = np.random.default_rng(axis)
    cdt, rdt = (np.complex128, np.float64) if prec == 64 else (np.complex64, np.float32)
    x = (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(cdt)
    r = np.ascontiguousarray(x.real).astype(rdt)
    for fmt in (1, 3):
        e = d2d.FFTEngine(fmt, *shape, prec=prec)
        xin, rin = dev(torch_gpu, x, cdt), dev(torch_gpu, r, rdt)
        out = torch_gpu.empty_like(xin)
        for sign, want in ((-1, np.fft.fftn(x.astype(np.complex128))),
                           (1, np.fft.ifftn(x.astype(np.complex128)) * x.size)):
            e.fft_c2c(xin, out, sign)
            assert rel_l2(host(out, shape), want) < TOL[prec]
        ss = list(shape)
        ss[0 if fmt == 1 else 2] = ss[0 if fmt == 1 else 2] // 2 + 1
        sp = torch_gpu.empty(int(np.prod(ss)), dtype=out.dtype, device="cuda")
        e.fft_r2c(rin, sp)
        axes = (2, 1, 0) if fmt == 1 else (0, 1, 2)
        assert rel_l2(host(sp, ss), np.fft.rfftn(r.astype(np.float64), axes=axes)) < TOL[prec]
        back = torch_gpu.empty_like(rin)
        e.fft_c2r(sp, back)
        assert rel_l2(host(back, shape) / r.size, r) < TOL[prec]


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("types,n,points", [((2, 3, 6, 7), 5280, 5250), ((1,), 2640, 2626), ((5,), 2640, 2624)])
def test_long_real_to_real(d2d, oracle, torch_gpu, types, n, points, axis, prec):
    """5250 transformed points (types 2, 3, 6, 7), an extension of 5250 points
    (DCT-I of 2626, DST-I of 2624), from the third of the axis on."""
    rdt = np.float64 if prec == 64 else np.float32
    shape = [2, 2, 2]
    shape[axis] = n
    shape = tuple(shape)
    x = np.asfortranarray(np.random.default_rng(n + axis).uniform(-1, 1, shape).astype(rdt))
    for t in types:
        dtt, skip = [2, 2, 2] + [1, 1, 1] + [1, 1, 1] + [1, 1, 1], [True, True, True]
        dtt[axis], dtt[3 + axis], dtt[6 + axis], dtt[9 + axis] = t, 3, n - points, 3
        skip[axis] = False
        e = d2d.FFTEngine(1, *shape, prec=prec, opt_DTT=dtt, skip_xyz=skip)
        xin = dev(torch_gpu, x, rdt)
        out = torch_gpu.empty_like(xin)
        for sign in (-1, 1):
            e.dtt_3d_r2r(xin, out, sign)
            want = oracle.dtt3d(x.astype(np.float64), tuple(dtt), sign, 1, skip=tuple(skip))
            assert rel_l2(host(out, shape), want) < RTOL[prec], (t, sign)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec", [64, 32])
def test_dct4_of_2048_points(d2d, oracle, torch_gpu, axis, prec):
    """DCT-IV and DST-IV of 2048 points run (the general kernel's tile of eight
    times the length does not fit a workgroup), on every specialised kernel."""
    rdt = np.float64 if prec == 64 else np.float32
    shape = [3, 3, 2]
    shape[axis] = 2049
    shape = tuple(shape)
    x = np.asfortranarray(np.random.default_rng(axis).uniform(-1, 1, shape).astype(rdt))
    xin = dev(torch_gpu, x, rdt)
    for t in (4, 8):
        dtt, skip = [2, 2, 2], [True, True, True]
        dtt[axis], skip[axis] = t, False
        e = d2d.FFTEngine(1, *shape, prec=prec, opt_DTT=dtt, skip_xyz=skip)
        for sign, st in ((-1, 7 + axis), (1, 10 + axis)):
            want = oracle.dtt3d(x.astype(np.float64), tuple(dtt), sign, 1, skip=tuple(skip))
            names = [n for n in e.stage_candidates(st) if n != "general"]
            assert len(names) == 2
            for name in [None] + names:
                if name:
                    e.set_stage_kernel(st, name)
                out = torch_gpu.empty_like(xin)
                e.dtt_3d_r2r(xin, out, sign)
                assert rel_l2(host(out, shape), want) < RTOL[prec], (t, sign, name)


@pytest.mark.parametrize("prec", [64, 32])
def test_small_pencils_run_the_compiled_real_to_real_tiles(d2d, torch_gpu, prec):
    """Pencils of less than 16 MB start on the compiled tile of their length,
    in every transform kind; large ones on the any-length kernels where those
    are faster."""
    for n, types in ((65, (2, 3, 6, 7)), (65, (1,)), (257, (4, 8)), (129, (5,))):
        for t in types:
            small = d2d.FFTEngine(1, n, n, 20, prec=prec, opt_DTT=(t, t, 2)).dtt_stage_kernels()
            assert all("mixed" not in small[s] for s in (7, 8, 10, 11)), (n, t, small)
    large = d2d.FFTEngine(1, 257, 257, 3000, prec=prec, opt_DTT=(4, 4, 2)).dtt_stage_kernels()
    assert "mixed" in large[7] and "mixed" in large[8]


def test_defaults_of_small_pencils(d2d, torch_gpu):
    """Pencils below 32 MB start on tiles with a plain exchange, large ones on
    those that take real and imaginary parts apart; r2c columns of 1152 points on
    the compiled tile, of 1000 points on the any-length kernel from 32 MB."""
    small = d2d.FFTEngine(1, 16, 1536, 16).stage_kernels()["c2c_y"]
    large = d2d.FFTEngine(1, 32, 1536, 64).stage_kernels()["c2c_y"]
    assert " xs" not in small and " xs" in large
    for n, nx, mixed in ((1000, 16, False), (1000, 256, True), (1152, 256, False), (1152, 512, False)):
        k = d2d.FFTEngine(3, nx, 32, n).stage_kernels()["r2c"]
        assert ("mixed" in k) == mixed, (n, nx, k)
