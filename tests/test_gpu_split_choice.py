"""Calls without positions whose kernels choose, by the direction of the image's
columns, between a strip's waves sharing its pulses and a workgroup per tile:
whatever they choose, the image is the batched launch's bit for bit and that of
the FP64 mode within the double-precision oracle tests' bounds."""
import numpy as np
import pytest

from sar_cambrianaccelerationcard_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["ref", "df"])
@pytest.mark.parametrize("axes", ["xy", "yx", "nan"])
@pytest.mark.parametrize("interp,nx,ny,spacing", [("sinc8", 1000, 400, 0.5), ("linear", 1000, 1000, 0.5)])
def test_plain_is_batch_and_matches_fp64(precision, axes, interp, nx, ny, spacing):
    import torch
    pulses, samples, dr = 70, 4096, 0.1875
    u, v = ([0.0, spacing, 0.0], [spacing, 0.0, 0.0]) if axes == "yx" else ([spacing, 0.0, 0.0], [0.0, spacing, 0.0])
    o = [-0.5 * (u[k] * nx + v[k] * ny) for k in range(3)]
    grid = native.make_grid(o, u, v, nx, ny)
    pos = np.zeros((pulses, 3))
    pos[:, 0], pos[:, 1], pos[:, 2] = np.linspace(-50, 50, pulses), -4000.0, 3000.0
    if axes == "nan":
        pos[pulses // 2] = np.nan  # the pulse that the choice looks at
    gen = torch.Generator(device="cuda").manual_seed(3)
    prof = torch.randn((pulses, samples, 2), device="cuda", generator=gen)
    d_pos = torch.from_numpy(pos).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    ctx = native.Context(0)
    try:
        img = {}
        for prec in (precision, "f64"):
            params = native.make_params(c=299792458.0, fc=9.6e9, r0=5000.0 - 0.5 * samples * dr, dr=dr, n_pulses=pulses,
                                        n_samples=samples, interp=interp, precision=prec, dtype="c64", kaiser_beta=6.0)
            for kind in ("plain", "batch"):
                out = torch.full((ny, nx), 7.0 + 0.0j, dtype=torch.complex64, device="cuda")
                print(f"  {prec} {interp} {nx}x{ny} {axes} {kind}", flush=True)
                if kind == "plain":
                    ctx.backproject(prof.data_ptr(), d_pos.data_ptr(), grid, params, out.data_ptr(), stream)
                else:
                    jb = native.Job()
                    jb.d_profiles, jb.d_pos, jb.d_image = prof.data_ptr(), d_pos.data_ptr(), out.data_ptr()
                    jb.grid, jb.params = grid, params
                    ctx.backproject_batch([jb], stream)
                torch.cuda.synchronize()
                img[prec, kind] = out.cpu().numpy()
        got, ref = img[precision, "plain"], img["f64", "plain"]
        if axes == "nan":  # one pulse's sum is no number: every pixel is one, in both
            assert np.isnan(got).all() and np.isnan(img[precision, "batch"]).all()
            return
        assert np.array_equal(got.view(np.uint64), img[precision, "batch"].view(np.uint64))
        assert np.linalg.norm(got - ref) / np.linalg.norm(ref) <= 3e-5
    finally:
        ctx.close()
