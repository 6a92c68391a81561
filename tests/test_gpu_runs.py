"""Runs through empty and constant bricks where their bounds are tightest: long
axes, transfer functions that fall or do not depend on the value, tables of the
largest size, voxels that are not finite.  Each route against the one that
looks for no runs."""
from __future__ import annotations

import numpy as np
import pytest

from robartsvtk_amd import abi, configs
import helpers as H

pytestmark = pytest.mark.gpu


def _sparse(n, dtype, seed):
    """Mostly empty, a block of noise every 400 voxels along x, constant blocks
    that end next to, on and past the faces of bricks and groups."""
    rng = np.random.default_rng(seed)
    vol = np.zeros(n[::-1], np.float32)
    for x0 in range(40, n[0] - 30, 400):
        vol[:, :, x0:x0 + 30] = rng.uniform(-20.0, 60.0, (n[2], n[1], 30))
    for x0, x1 in ((100, 127), (200, 255), (301, 352), (n[0] - 97, n[0] - 33), (n[0] - 9, n[0])):
        vol[:, :, max(x0, 0):x1] = 35.0
    if dtype == "u8":
        vol = np.maximum(vol, 0.0)
    return np.rint(vol).astype({"u8": np.uint8, "i16": np.int16}[dtype]) if dtype != "f32" else vol


# 4 and 8 thousand samples a ray; 26200 rays put four lanes on a ray, a plan's
# 4 x 26200 two; 2.4 million take two samples in flight, and so do 150-sample
# rays between 100 and 200 thousand.
@pytest.mark.parametrize("n,sp,W,h,step,d", [
    ((4096, 6, 7), (1.0, 40.0, 40.0), 200, 131, 0.7, (1.0, 0.0003, -0.0007)),
    ((4096, 6, 7), (1.0, 40.0, 40.0), 200, 131, 0.7, (-1.0, 0.011, 0.009)),
    ((4095, 9, 4), (1.0, 30.0, 60.0), 1610, 1490, 1.0, (-1.0, 0.0, 0.0)),
    ((4093, 9, 8), (1.0, 30.0, 40.0), 1610, 1490, 1.3, (1.0, 0.02, 0.01)),
    ((131, 100, 90), (1.0, 1.0, 1.0), 400, 300, 1.0, (1.0, 0.6, 0.3))])
@pytest.mark.parametrize("dtype,skip", [("u8", 0), ("i16", 1), ("f32", 0), ("f32", 1)])
def test_runs_on_long_axes_sum_what_the_plain_march_does(gpu_ctx, n, sp, W, h, step, d, dtype, skip):
    """A threshold that no ray reaches gives the plain march.  The same samples
    count, a run's sum is rounded once and lanes add theirs at the end, all in
    f64: L within one ulp of float32."""
    import torch
    ext = max(k * s for k, s in zip(n, sp))
    c, d = configs.volume_center(n, sp), np.asarray(d, float) / np.linalg.norm(d)
    cam = abi.camera(c + 3.0 * ext * d, c, (0, 0, 1), 1.2 * np.degrees(0.5 * max(n[1] * sp[1], n[2] * sp[2]) / ext),
                     (0.5 * ext, 6.0 * ext))
    view = abi.compute_view(cam, W, h, spacing=sp)
    vh = H.gpu_volume(gpu_ctx, _sparse(n, dtype, 3), sp)
    march = configs.march_params({"step_scale": step, "term_T": 0.0, "jitter": 1, "skip_rule": skip})
    drr = [configs.drr_params({"intercept": -1e-5, "slope": 1e-5, "offset": o, "output": abi.DRR_F32_L,
                               "ref_termination": t}) for t, o in ((0, 1.0), (1, 1e30))]
    out = [torch.full((h, W), float("nan"), device="cuda") for _ in range(2)]
    for p, o in zip(drr, out):
        abi.render_drr(gpu_ctx, vh, view, march, p, o)
    got = [out[0].cpu().numpy().ravel()]
    if W < 1000:
        plan = abi.DrrPlan(gpu_ctx, vh, [view] * 4, march, drr[0])
        packed = torch.full((plan.total,), float("nan"), device="cuda")
        plan.render(packed)
        got += [packed[o:o + W * h].cpu().numpy() for o in plan.offsets[:-1]]
        plan.close()
    ref = out[1].cpu().numpy().ravel()
    vh.close()
    assert 0.001 < ref.max() < 50.0 and (ref > 0).mean() > 0.05
    for g in got:
        assert np.all(np.abs(g - ref) <= 2.0 ** -23 * np.abs(ref))


def _no_window(view):
    """A keyhole plane that leaves every ray outside: the window is empty, but
    the view takes the casters that march one lane per ray and no runs."""
    v = abi.View.from_buffer_copy(view)
    v.n_keyhole_planes = 1
    v.keyhole_planes[:4] = [1.0, 0.0, 0.0, -1e6]
    return v


@pytest.mark.parametrize("window", ["rising", "falling", "flat", "narrow"])
@pytest.mark.parametrize("n", [40, 2048])
@pytest.mark.parametrize("finite", [True, False])
@pytest.mark.parametrize("skip", [0, 1])
def test_runs_of_values_without_opacity_composite_as_one_lane(gpu_ctx, window, n, finite, skip):
    """1D (plain and shaded), 2D and dual renders over 10 groups of bricks along
    x, to the byte: tables whose columns fall with the value, do not depend on
    it, or are one bitmap word or 64; infinities and NaN among the voxels."""
    import torch
    dims, sp = (315, 21, 19), (1.0, 1.5, 1.3)
    vol = _sparse(dims, "f32", 5)
    if not finite:
        vol[3, 4, 60], vol[9, 9, 170], vol[12, 2, 260] = np.nan, np.inf, -np.inf
    vh = H.gpu_volume(gpu_ctx, vol, sp)
    vh2 = H.gpu_volume(gpu_ctx, np.ascontiguousarray(vol[::-1]), sp)
    lo, mult = {"rising": (-20.0, 1 / 80.0), "falling": (60.0, -1 / 80.0), "flat": (10.0, 0.0),
                "narrow": (30.0, 1 / 8.0)}[window]
    c = configs.volume_center(dims, sp)
    cam = abi.camera(c + np.array([120.0, 330.0, 150.0]), c, (0, 0, 1), 40.0, (50.0, 700.0))
    view = abi.compute_view(cam, 150, 61, spacing=sp)
    march = configs.march_params({"step_scale": 0.8, "term_T": 0.02, "jitter": 1, "skip_rule": skip})
    u = (np.arange(n) + 0.5) / n
    alpha = np.where((np.abs(u - 0.7) < 0.08) | ((n > 64) & (np.abs(u - 0.2) < 0.4 / n)), 0.1, 0.0).astype(np.float32)
    if window == "flat":
        alpha[0] = 0.02
    rgb = np.random.default_rng(n).uniform(0, 1, (n, 3)).astype(np.float32)
    calls, tfs = [], []
    for params in (abi.Tf1dParams(lo, mult, 0.0, float("inf"), 1.0, 0.0, 0.0, 1.0),
                   abi.Tf1dParams(lo, mult, 0.0, 1 / 60.0, 0.4, 0.6, 0.3, 8.0)):
        tfs.append(abi.TF1D(gpu_ctx, alpha, rgb, params, galpha=np.linspace(0.2, 1, n).astype(np.float32)))
        calls.append(lambda v, o, a, tf=tfs[-1]: abi.render_1d(gpu_ctx, vh, tf, v, march, o, a))
    m = min(n, 600)
    um = (np.arange(m) + 0.5) / m
    full = np.ones((m, m), np.float32)
    col = np.where((np.abs(um - 0.7) < 0.08) | ((window == "flat") & (um < 0.03)), 0.1, 0.0).astype(np.float32)
    t = {"alpha": full * col, "red": 0.9 * full, "green": full * um.astype(np.float32), "blue": 0.2 * full,
         "ambient": 0.4 * full, "diffuse": 0.6 * full, "specular": 0.3 * full, "specular_power": 8.0 * full}
    p2 = configs.tf2d_params(configs.tf2d_params_for(0.0, 1.0, 0.0, 60.0))
    p2.intensity_low, p2.intensity_multiplier = lo, mult
    tfs.append(abi.TF2D(gpu_ctx, t, p2))
    calls.append(lambda v, o, a, tf=tfs[-1]: abi.render_2d(gpu_ctx, vh, tf, v, march, o, False, a))
    dual = abi.DualParams(lo, mult, -20.0, 1 / 80.0)
    calls.append(lambda v, o, a, tf=tfs[-1]: abi.render_dual(gpu_ctx, vh, vh2, tf, dual, v, march, o, a))
    for i, call in enumerate(calls):
        got = []
        for v in (view, _no_window(view)):
            out = torch.full((61, 150, 4), 77, dtype=torch.uint8, device="cuda")
            depth = [torch.full((61, 150), float("nan"), device="cuda") for _ in range(3)]
            call(v, out, abi.AuxOut(*[b.data_ptr() for b in depth]))
            torch.cuda.synchronize()
            got.append([out.cpu().numpy()] + [b.cpu().numpy() for b in depth])
        for a, b in zip(*got):
            np.testing.assert_array_equal(a, b, err_msg=str(i))
        if finite and window != "flat":
            assert (got[0][0][..., 3] > 0).any(), i
    for o in tfs + [vh, vh2]:
        o.close()
