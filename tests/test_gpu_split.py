"""Images of few tiles, whose pulses a strip's waves share out: parity with the
FP64 oracle, and the same bits from the batched launch, which sums the same
parts one after another."""
import numpy as np
import pytest

from sar_cambrianaccelerationcard_amd import device as D
from sar_cambrianaccelerationcard_amd import metrics as M
from sar_cambrianaccelerationcard_amd import native
from sar_cambrianaccelerationcard_amd import scene as S

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene():
    sc = S.make_scene(S.scaled_config(S.load_config("config0"), n_pulses=301, nx=64, ny=64))
    return sc, D.DeviceScene(sc, bf16=True)


# 2 parts (32-pulse sums) up to 8 of them, sums that end inside a setup batch
# or are empty, one pulse; strips that touch more positions than a wave stages
# at once (x along range, wide pixels); ragged edges; every row count
@pytest.mark.parametrize("dtype", ["c64", "bf16x2"])
@pytest.mark.parametrize("interp,pulses,nx,ny,spacing,rows,axes", [
    ("sinc8", 301, 65, 17, 0.5, 4, "xy"), ("sinc8", 33, 64, 16, 0.25, 2, "xy"), ("sinc8", 1, 10, 10, 0.5, 4, "xy"),
    ("sinc8", 289, 100, 35, 0.5, 8, "yx"), ("sinc8", 130, 130, 70, 1.1, 4, "yx"), ("sinc8", 16, 300, 9, 1.0, 4, "xy"),
    ("linear", 301, 65, 17, 0.5, 4, "xy"), ("linear", 40, 200, 64, 2.2, 2, "yx"), ("linear", 31, 64, 64, 0.5, 8, "xy"),
])
def test_split_matches_oracle_and_batch(scene, dtype, interp, pulses, nx, ny, spacing, rows, axes):
    import torch
    sc, ds = scene
    o = sc.grid["origin"]
    u, v = [spacing, 0.0, 0.0], [0.0, spacing, 0.0]
    if axes == "yx":
        u, v = v, u
    grid = native.make_grid(o, u, v, nx, ny)
    prof = D.from_bf16x2(D.to_bf16x2(sc.profiles)) if dtype == "bf16x2" else sc.profiles
    ref = O.backproject(np.ascontiguousarray(prof[:pulses]), np.ascontiguousarray(sc.pos[:pulses]),
                        {"origin": o, "ux": u, "uy": v, "nx": nx, "ny": ny},
                        O.params(sc.c, sc.fc, sc.r0, sc.dr, interp, sc.kaiser_beta))
    pos = np.ascontiguousarray(sc.pos[:pulses])
    stream = torch.cuda.current_stream().cuda_stream
    ctx = native.Context(0)
    try:
        ctx.set_tuning(native.INTERP_NAMES[interp], native.PREC_REF, native.DTYPE_NAMES[dtype], rows, 1, 6)
        for h_pos in (None, pos):
            for add in (0, 1):
                params = sc.native_params(interp=interp, dtype=dtype, accumulate=bool(add))
                params.n_pulses = pulses
                plan = ctx.plan(h_pos, grid, params)
                print(f"  {interp} {pulses}p {nx}x{ny} {spacing} m {rows} rows {axes} {dtype} add={add} {plan.info()}",
                      flush=True)
                plain = torch.full((ny, nx), 2.0 - 1.0j, dtype=torch.complex64, device="cuda")
                batch = plain.clone()
                plan.execute(ds.profiles_ptr(dtype), ds.pos.data_ptr(), plain.data_ptr(), stream)
                jb = native.Job()
                jb.d_profiles, jb.d_pos, jb.d_image = ds.profiles_ptr(dtype), ds.pos.data_ptr(), batch.data_ptr()
                jb.h_pos = pos.ctypes.data if h_pos is not None else None
                jb.grid, jb.params = grid, params
                ctx.backproject_batch([jb], stream)
                torch.cuda.synchronize()
                got = plain.cpu().numpy()
                assert np.array_equal(got.view(np.uint64), batch.cpu().numpy().view(np.uint64))
                # dropped terms 5e-6 rad, FP32 phase 1.2e-5 rad, sinc8 fit 2e-6;
                # the FP32 sum into 2 - j
                err = np.linalg.norm(got - (2.0 - 1.0j) * add - ref) / np.linalg.norm(ref + (2.0 - 1.0j) * add)
                assert err <= 3e-5, err
    finally:
        ctx.close()


# the default launch cuts strips to two rows up to 128 strips of four rows (256
# without positions, sinc8, and to four up to 640): both sides of the lines,
# ragged edges, pixels that take the double-float arithmetic, too few pulses to
# share out
@pytest.mark.parametrize("interp,pulses,nx,ny,spacing", [
    ("sinc8", 301, 100, 250, 0.5), ("sinc8", 301, 100, 260, 0.5), ("sinc8", 64, 640, 256, 0.5), ("sinc8", 64, 640, 260, 0.5), ("sinc8", 40, 129, 300, 0.5), ("sinc8", 20, 65, 17, 1.6),
    ("linear", 150, 128, 256, 0.5), ("linear", 150, 128, 257, 0.5), ("linear", 64, 30, 33, 2.2),
])
def test_small_images_match_oracle_and_batch(scene, interp, pulses, nx, ny, spacing):
    import torch
    sc, ds = scene
    o = sc.grid["origin"]
    g = {"origin": o, "ux": [spacing, 0.0, 0.0], "uy": [0.0, spacing, 0.0], "nx": nx, "ny": ny}
    grid = native.make_grid(o, g["ux"], g["uy"], nx, ny)
    pos = np.ascontiguousarray(sc.pos[:pulses])
    ref = O.backproject(np.ascontiguousarray(sc.profiles[:pulses]), pos, g,
                        O.params(sc.c, sc.fc, sc.r0, sc.dr, interp, sc.kaiser_beta))
    params = sc.native_params(interp=interp)
    params.n_pulses = pulses
    stream = torch.cuda.current_stream().cuda_stream
    ctx = native.Context(0)
    try:
        for h_pos in (None, pos):
            print(f"  {interp} {pulses}p {nx}x{ny} {spacing} m positions={h_pos is not None}", flush=True)
            img = [torch.zeros((ny, nx), dtype=torch.complex64, device="cuda") for _ in range(3)]
            ctx.plan(h_pos, grid, params).execute(ds.profiles_ptr("c64"), ds.pos.data_ptr(), img[0].data_ptr(), stream)
            if h_pos is None:
                ctx.backproject(ds.profiles_ptr("c64"), ds.pos.data_ptr(), grid, params, img[1].data_ptr(), stream)
            jb = native.Job()
            jb.d_profiles, jb.d_pos, jb.d_image = ds.profiles_ptr("c64"), ds.pos.data_ptr(), img[2].data_ptr()
            jb.h_pos = h_pos.ctypes.data if h_pos is not None else None
            jb.grid, jb.params = grid, params
            ctx.backproject_batch([jb], stream)
            torch.cuda.synchronize()
            got = [im.cpu().numpy() for im in img]
            assert M.rel_l2(got[0], ref) <= 5e-5  # bins and phases as in the row polynomials' own tests
            for other in (got[2],) if h_pos is not None else got[1:]:
                assert np.array_equal(other.view(np.uint64), got[0].view(np.uint64))
    finally:
        ctx.close()
