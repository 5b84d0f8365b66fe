"""Antennas a few metres from the pixels, where strips of a tile differ in
whether their bins have a bound: the batched image (a workgroup per tile) is the
plain one (waves per strip) bit for bit, and the double-float mode, which then
works in FP64 per pixel, matches the FP64 oracle."""
import numpy as np
import pytest

from sar_cambrianaccelerationcard_amd import native

import oracle as O

pytestmark = pytest.mark.gpu

DR, SAMPLES, FC = 0.1875, 2048, 9.6e9


def _scene(alt, standoff, pulses, span):
    pos = np.empty((pulses, 3))
    pos[:, 0] = np.linspace(-span, span, pulses)
    pos[:, 1] = -standoff
    pos[:, 2] = alt
    rng = np.random.default_rng(pulses)
    prof = rng.standard_normal((pulses, SAMPLES, 2)).astype(np.float32).view(np.complex64)[..., 0]
    return pos, np.ascontiguousarray(prof)


@pytest.mark.parametrize("precision", ["ref", "df"])
@pytest.mark.parametrize("interp", ["linear", "sinc8"])
# above the image (most strips without a bound, half of them, some), beside it at
# grazing angles; pulses shared out over waves and too few for that
@pytest.mark.parametrize("alt,standoff,spacing,pulses", [
    (0.7, 0.0, 0.25, 128), (3.0, 0.0, 0.25, 128), (5.0, 0.0, 0.25, 40), (8.0, 0.0, 0.25, 128), (3.0, 0.0, 0.25, 20),
    (20.0, 250.0, 1.2, 64), (2.0, 60.0, 0.5, 64),
])
def test_batch_is_plain_and_double_float_matches_oracle(precision, interp, alt, standoff, spacing, pulses):
    import torch
    nx, ny = 70, 45
    pos, prof = _scene(alt, standoff, pulses, 0.25 * nx * spacing)
    o = [-0.5 * nx * spacing, -0.5 * ny * spacing, 0.0]
    g = {"origin": o, "ux": [spacing, 0.0, 0.0], "uy": [0.0, spacing, 0.0], "nx": nx, "ny": ny}
    grid = native.make_grid(o, g["ux"], g["uy"], nx, ny)
    params = native.make_params(c=299792458.0, fc=FC, r0=0.0, dr=DR, n_pulses=pulses, n_samples=SAMPLES,
                                interp=interp, precision=precision, dtype="c64", kaiser_beta=6.0)
    d_prof, d_pos = torch.from_numpy(prof).cuda(), torch.from_numpy(pos).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    ref = O.backproject(prof, pos, g, O.params(299792458.0, FC, 0.0, DR, interp, 6.0))
    ctx = native.Context(0)
    try:
        for h_pos in (None, pos):
            print(f"  {precision} {interp} {alt} m above, {standoff} m off, {spacing} m, {pulses} pulses "
                  f"positions={h_pos is not None}", flush=True)
            plain = torch.zeros((ny, nx), dtype=torch.complex64, device="cuda")
            batch = torch.zeros_like(plain)
            ctx.plan(h_pos, grid, params).execute(d_prof.data_ptr(), d_pos.data_ptr(), plain.data_ptr(), stream)
            jb = native.Job()
            jb.d_profiles, jb.d_pos, jb.d_image = d_prof.data_ptr(), d_pos.data_ptr(), batch.data_ptr()
            jb.h_pos = h_pos.ctypes.data if h_pos is not None else None
            jb.grid, jb.params = grid, params
            ctx.backproject_batch([jb], stream)
            torch.cuda.synchronize()
            got = plain.cpu().numpy()
            assert np.isfinite(got.view(np.float32)).all()
            assert np.array_equal(got.view(np.uint64), batch.cpu().numpy().view(np.uint64))
            if precision == "df":
                # FP32 bins up to 1024: a few roundings of 1.8e-5 bin rms, slope
                # of white samples below 2
                err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
                print(f"    rel_l2={err:.2e}", flush=True)
                assert err <= 1e-4
    finally:
        ctx.close()
