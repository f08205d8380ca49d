"""The kernels of any length (csrc/mixed_impl.h): every radix alone, two to
five passes, Bluestein lengths, remainders of the tile (columns, real pairs,
rows past the last butterfly), the three kernel classes, against pocketfft and the
general kernel; the packed y / z stages against stage and pack; grouped
batches against the plans' own calls; the compiled tiles' column pairs and the
default between the two.

Tolerances: those of test_gpu_fft.py (1e-13 FP64, 5e-6 FP32, relative L2); a
transform of n points takes at most log2(n) + 1 rounding steps more than the
sum, here below 14 (28 for a convolution) of 1.1e-16 (6e-8)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {64: 1e-13, 32: 5e-6}
# lengths: each radix, its product with others, 4- and 5-pass schedules,
# lengths whose tile is one column wide; then lengths with a prime factor
# above 17 (two- to four-pass convolutions, the shortest and the longest)
LENGTHS = [2, 3, 5, 7, 9, 11, 13, 15, 16, 17, 18, 25, 34, 49, 63, 81, 121, 143, 169, 187, 243, 289,
           375, 405, 450, 625, 686, 729, 1001, 1210, 1875, 2187, 2401, 3125, 4375,
           19, 23, 29, 41, 62, 107, 191, 247, 382, 509, 638, 1021, 1531, 3067]


def dev(torch, a, dt):
    return torch.from_numpy(np.ascontiguousarray(a.ravel(order="F")).astype(dt)).to("cuda")


def host(t, shape):
    return t.cpu().numpy().reshape(shape, order="F")


def mixed_of(e, stage):
    return [n for n in e.stage_candidates(stage) if "mixed" in n]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec", [64, 32])
def test_mixed_lengths(d2d, torch_gpu, n, axis, prec):
    """c2c both ways, r2c and c2r with length n along each axis, in both
    formats; the columns left over are odd in number."""
    torch = torch_gpu
    shape = [7, 5, 3]
    shape[axis] = n
    shape = tuple(shape)
    rng = np.random.default_rng(n + axis)
    x = rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)
    cdt, rdt = (np.complex128, np.float64) if prec == 64 else (np.complex64, np.float32)
    x = x.astype(cdt)
    r = np.ascontiguousarray(x.real).astype(rdt)
    xin, rin = dev(torch, x, cdt), dev(torch, r, rdt)
    stages = ("c2c_x", "c2c_y", "c2c_z")
    for fmt in (1, 3):
        e = d2d.FFTEngine(fmt, *shape, prec=prec)
        assert len(mixed_of(e, stages[axis])) == 1
        for s in e.STAGES:
            for name in mixed_of(e, s):
                e.set_stage_kernel(s, name)
        out = torch.empty_like(xin)
        e.fft_c2c(xin, out, -1)
        assert rel_l2(host(out, shape), np.fft.fftn(x.astype(np.complex128))) < TOL[prec]
        e.fft_c2c(xin, out, 1)
        assert rel_l2(host(out, shape), np.fft.ifftn(x.astype(np.complex128)) * x.size) < TOL[prec]
        ss = list(shape)
        ss[0 if fmt == 1 else 2] = ss[0 if fmt == 1 else 2] // 2 + 1
        sp = torch.empty(int(np.prod(ss)), dtype=out.dtype, device="cuda")
        e.fft_r2c(rin, sp)
        axes = (2, 1, 0) if fmt == 1 else (0, 1, 2)
        assert rel_l2(host(sp, ss), np.fft.rfftn(r.astype(np.float64), axes=axes)) < TOL[prec]
        back = torch.empty_like(rin)
        e.fft_c2r(sp, back)
        assert rel_l2(host(back, shape) / r.size, r) < TOL[prec]
        # the general kernel on the same data
        for s in e.STAGES:
            e.set_stage_kernel(s, "general")
        out_g = torch.empty_like(out)
        e.fft_c2c(xin, out_g, 1)
        assert rel_l2(host(out, shape), host(out_g, shape)) < TOL[prec]


def test_mixed_aligned_and_unaligned_pairs(d2d, torch_gpu):
    """r2c along z pairs adjacent columns: one load per pair when the pairs
    are aligned, two otherwise (odd strides, an odd base address, an odd
    column count)."""
    torch = torch_gpu
    for nx, ny, off in ((6, 4, 0), (6, 4, 1), (5, 4, 0), (5, 3, 1)):
        shape = (nx, ny, 45)
        buf = torch.rand(nx * ny * 45 + 1, dtype=torch.float64, device="cuda")
        x = buf[off:off + nx * ny * 45]
        e = d2d.FFTEngine(3, *shape)
        e.set_stage_kernel("r2c", mixed_of(e, "r2c")[0])
        sp = torch.empty(nx * ny * 23, dtype=torch.complex128, device="cuda")
        e.fft_r2c(x, sp)
        want = np.fft.rfftn(host(x, shape), axes=(0, 1, 2))
        assert rel_l2(host(sp, (nx, ny, 23)), want) < 1e-13, (nx, ny, off)


@pytest.mark.parametrize("n", [64, 720, 1024, 2048])
@pytest.mark.parametrize("nx,off", [(66, 0), (66, 1), (67, 0), (67, 1)])
@pytest.mark.parametrize("prec", [64, 32])
def test_compiled_column_pairs(d2d, torch_gpu, n, nx, off, prec):
    """r2c and c2r along z on every compiled tile: whole tiles take a pair of
    adjacent real columns in one access, aligned or not (odd row length, odd
    base address); the last tile, with columns left over, one by one."""
    torch = torch_gpu
    rdt, cdt = (torch.float64, torch.complex128) if prec == 64 else (torch.float32, torch.complex64)
    shape, ss = (nx, 1, n), (nx, 1, n // 2 + 1)
    buf = torch.rand(nx * n + 1, dtype=rdt, device="cuda")
    out = torch.full((nx * n + 2,), 7.0, dtype=rdt, device="cuda")
    x, back = buf[off:off + nx * n], out[off:off + nx * n]
    sp = torch.empty(nx * (n // 2 + 1), dtype=cdt, device="cuda")
    e = d2d.FFTEngine(3, *shape, prec=prec)
    want = np.fft.rfftn(host(x, shape).astype(np.float64), axes=(0, 1, 2))
    for r, c in zip(e.stage_candidates("r2c"), e.stage_candidates("c2r")):
        e.set_stage_kernel("r2c", r)
        e.set_stage_kernel("c2r", c)
        e.fft_r2c(x, sp)
        assert rel_l2(host(sp, ss), want) < TOL[prec], r
        e.fft_c2r(sp, back)
        assert rel_l2(host(back, shape) / (nx * n), host(x, shape)) < TOL[prec], c
        assert out[off + nx * n] == 7.0 and (off == 0 or out[0] == 7.0)


def test_default_kernel_by_length_and_size(d2d, torch_gpu):
    """Short lengths start on the any-length kernels only in pencils that do
    not stay in the memory-side cache."""
    small = d2d.FFTEngine(1, 128, 128, 128).stage_kernels()
    large = d2d.FFTEngine(1, 128, 1024, 1024).stage_kernels()
    assert "mixed" not in small["c2c_x"] and "mixed" in large["c2c_x"]
    assert "mixed" not in large["c2c_y"]
    wide = d2d.FFTEngine(1, 1024, 128, 1024).stage_kernels()
    assert "mixed" not in small["c2c_y"] and "mixed" in wide["c2c_y"]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("shape", [(50, 90, 63), (30, 187, 26), (18, 57, 101)])
def test_mixed_packed_stages(d2d, torch_gpu, shape, prec):
    """The default kernels of a rank of a 3 x 2 grid whose lengths have no
    compiled tile: y and z stages fused with pack and unpack equal the stage
    and d2dhip_pack / _unpack bit for bit."""
    torch = torch_gpu
    cdt = torch.complex128 if prec == 64 else torch.complex64
    elem = d2d.C16 if prec == 64 else d2d.C8
    XY, YZ = d2d.X_TO_Y, d2d.Y_TO_Z
    for row, col, even in ((0, 0, False), (2, 1, False), (1, 1, True)):
        e = d2d.FFTEngine(1, *shape, prec=prec, rank=(3, 2, row, col))
        _, sp = e.decomps()
        assert "mixed" in e.stage_kernels()["spec_y"] and "mixed" in e.stage_kernels()["spec_last"]
        ny, nz = int(np.prod(list(sp.ysz))), int(np.prod(list(sp.zsz)))
        recv = torch.randn(max(d2d.pack_buffer_elems(XY, sp, even), ny), dtype=cdt, device="cuda")
        ns = d2d.pack_buffer_elems(YZ, sp, even)
        fused = torch.full((ns,), 7.0, dtype=cdt, device="cuda")
        plain = torch.full((ns,), 7.0, dtype=cdt, device="cuda")
        tmp = torch.empty(ny, dtype=cdt, device="cuda")
        e.exec_1m_unpack_pack("spec_y", recv, fused, XY, YZ, sp, -1, even)
        d2d.unpack(XY, elem, recv, tmp, sp, even)
        e.exec_1m("spec_y", tmp, tmp, -1)
        d2d.pack(YZ, elem, tmp, plain, sp, even)
        assert torch.equal(fused, plain)
        recv = torch.randn(max(ns, nz), dtype=cdt, device="cuda")
        a = torch.empty(nz, dtype=cdt, device="cuda")
        b = torch.empty_like(a)
        e.exec_1m_unpack("spec_last", recv, a, YZ, sp, 1, even)
        d2d.unpack(YZ, elem, recv, b, sp, even)
        e.exec_1m("spec_last", b, b, 1)
        assert torch.equal(a, b)


@pytest.mark.parametrize("prec", [64, 32])
def test_mixed_grouped_batch(d2d, torch_gpu, prec):
    """A grouped batch of grids whose stages run the mixed kernels (one launch
    over tiles of different lengths, block sizes and LDS): the plans' own
    calls bit for bit, replayed from a graph."""
    torch = torch_gpu
    cdt = torch.complex128 if prec == 64 else torch.complex64
    shapes = [(18, 45, 63), (375, 7, 5), (17, 13, 11), (2, 405, 9), (27, 3, 143)]
    engines = [d2d.FFTEngine(1 + 2 * (i % 2), *s, prec=prec) for i, s in enumerate(shapes)]
    ins = [torch.randn(int(np.prod(s)), dtype=cdt, device="cuda") for s in shapes]
    outs = [torch.empty_like(a) for a in ins]
    seq = [torch.empty_like(a) for a in ins]
    for e, a, q in zip(engines, ins, seq):
        e.fft_c2c(a, q, -1)
        e.fft_c2c(q, q, 1)
    b = d2d.Batch(engines)
    b.set_mode(d2d.BATCH_GROUPED)
    b.bind(ins, outs, mode=0)
    b.capture_graph()
    for _ in range(3):
        for o in outs:
            o.zero_()
        b.graph_launch()
        b.check()
        for o, q in zip(outs, seq):
            assert torch.equal(o, q)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n", [18, 32, 33, 46, 64, 65, 91, 100, 123, 244, 405, 482, 513])
def test_mixed_real_to_real(d2d, oracle, torch_gpu, n, axis, prec):
    """Every DCT / DST type along one axis of n points (transformed lengths n, n-1
    and n-2; DFTs of half, once, twice that and Bluestein ones), in place,
    against the oracle's direct sums and the general kernel.  Tolerances:
    test_gpu_dtt.py's (1e-13, 2e-6)."""
    torch = torch_gpu
    tol = 1e-13 if prec == 64 else 2e-6
    shape = [5, 4, 3]
    shape[axis] = n
    shape = tuple(shape)
    rdt = np.float64 if prec == 64 else np.float32
    x = np.asfortranarray(np.random.default_rng(n + axis).uniform(-1, 1, shape).astype(rdt))
    ran = 0
    for t in range(1, 9):
        dtt = [2, 2, 2]
        dtt[axis] = t
        skip = [True, True, True]
        skip[axis] = False
        e = d2d.FFTEngine(1, *shape, prec=prec, opt_DTT=dtt, skip_xyz=skip)
        for sign, st in ((-1, 7 + axis), (1, 10 + axis)):
            want = oracle.dtt3d(x.astype(np.float64), tuple(dtt), sign, 1, skip=tuple(skip))
            for name in [c for c in e.stage_candidates(st) if "mixed" in c]:
                e.set_stage_kernel(st, name)
                buf = dev(torch, x, rdt)
                e.dtt_3d_r2r(buf, buf, sign)
                assert rel_l2(host(buf, shape), want) < tol, (t, sign, name)
                e.set_stage_kernel(st, "general")
                gen = torch.empty_like(buf)
                e.dtt_3d_r2r(dev(torch, x, rdt), gen, sign)
                assert rel_l2(host(buf, shape), host(gen, shape)) < tol, (t, sign, name)
                ran += 1
    assert ran >= 14, ran


def test_refused_lengths_stay_refused(d2d, torch_gpu):
    """Stages whose general-kernel tile does not fit a workgroup are refused
    though a kernel of any length could run them (DCT-IV of 721 points runs on
    the general kernel through 8 * 721 points, padded to 16384)."""
    for dtt in ((4, 2, 2), (8, 2, 2)):
        with pytest.raises(d2d.D2dError):
            d2d.FFTEngine(1, 722, 4, 3, opt_DTT=dtt)
    d2d.FFTEngine(1, 722, 4, 3, opt_DTT=(2, 3, 4))
