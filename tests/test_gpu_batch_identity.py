"""A persistent batch equals each plan's own call bit for bit also where the
pencils are large enough for another default kernel (128 MB and more): the plans
as made, untuned and tuned, with no stage kernel set by hand."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,shapes", [(64, [(256, 192, 192), (64, 256, 48), (256, 256, 160)]),
                                         (32, [(256, 256, 256), (32, 96, 128)])])
def test_persistent_batch_equals_default_plans(d2d, torch_gpu, prec, shapes):
    torch = torch_gpu
    cdt = torch.complex128 if prec == 64 else torch.complex64
    engines = [d2d.FFTEngine(1 + 2 * (i % 2), *s, prec=prec) for i, s in enumerate(shapes)]
    ins = [torch.randn(int(np.prod(s)), dtype=cdt, device="cuda") for s in shapes]
    outs = [torch.empty_like(a) for a in ins]
    b = d2d.Batch(engines)
    assert b.persistent_tiles()
    b.bind(ins, outs, mode=0)
    b.launch()
    b.check()
    for e, a, o in zip(engines, ins, outs):
        own = torch.empty_like(a)
        e.fft_c2c(a, own, -1)
        e.fft_c2c(own, own, 1)
        assert torch.equal(own, o), e.stage_kernels()


def test_tuned_plans_of_persistent_batches_run_compiled_tiles(d2d, torch_gpu, tmp_path, monkeypatch):
    monkeypatch.setenv("D2DHIP_TUNE_CACHE", str(tmp_path / "tuning.tsv"))
    for shape in ((128, 64, 96), (256, 192, 192)):
        for _ in range(2):  # raced, then from the cache
            k = d2d.FFTEngine(1, *shape, tune=True).stage_kernels()
            assert all("mixed" not in k[s] for s in ("c2c_x", "c2c_y", "c2c_z")), k
