"""Fused pack / unpack calls queued one after another with no synchronisation
between them: each stage sees its own block table and descriptor, which are
written on the stream (one block, uneven blocks, as many blocks as a process
grid may have, EVEN padding).  Copies, so results are equal bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
def test_queued_pack_tables(d2d, torch_gpu, prec):
    torch = torch_gpu
    cdt = torch.complex128 if prec == 64 else torch.complex64
    rdt = torch.float64 if prec == 64 else torch.float32
    elem = d2d.C16 if prec == 64 else d2d.C8
    XY, YZ = d2d.X_TO_Y, d2d.Y_TO_Z
    nx, ny, nz = 126, 80, 12
    nxc = nx // 2 + 1
    e = d2d.FFTEngine(1, nx, ny, nz, prec=prec)
    a = torch.randn(nx * ny * nz, dtype=rdt, device="cuda")
    y = torch.randn(nxc * ny * nz, dtype=cdt, device="cuda")
    one = d2d.decomp_info_init(nxc, ny, nz)
    # 1, 3, 64 and 5 blocks of the engine's own x- and y-pencil
    xs = [(d2d.decomp_info_init(nxc, ny * m, nz, m, 1), ev) for m in (1, 3, 64, 5) for ev in (False, True)]
    ys = [(d2d.decomp_info_init(nxc, ny, nz * m, 1, m), ev) for m in (1, 3, 64, 5) for ev in (False, True)]
    outs = []
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    plain = torch.empty(nxc * ny * nz, dtype=cdt, device="cuda")
    py = torch.empty_like(y)
    with torch.cuda.stream(side):
        for d, ev in xs:
            o = torch.full((d2d.pack_buffer_elems(XY, d, ev),), 7.0, dtype=cdt, device="cuda")
            e.fft_r2c_pack(a, o, d, ev)
            outs.append((XY, d, ev, o))
        for d, ev in ys:
            o = torch.full((d2d.pack_buffer_elems(YZ, d, ev),), 7.0, dtype=cdt, device="cuda")
            e.exec_1m_pack("spec_y", y, o, YZ, d, -1, ev)
            outs.append((YZ, d, ev, o))
        e.fft_r2c_pack(a, plain, one)
        e.exec_1m("spec_y", y, py, -1)
    side.synchronize()
    for direction, d, ev, o in outs:
        want = torch.full_like(o, 7.0)
        d2d.pack(direction, elem, plain if direction == XY else py, want, d, ev)
        assert torch.equal(o, want), (direction, d.p_row, d.p_col, ev)
