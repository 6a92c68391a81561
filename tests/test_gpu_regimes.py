"""Calls whose fastest route depends on their sizes or data: each takes no
longer than the route it could have had instead, measured in the same process,
with the same results."""
from __future__ import annotations

import numpy as np
import pytest

from robartsvtk_amd import abi, configs
import helpers as H

pytestmark = pytest.mark.gpu


def _us(call) -> float:
    """Microseconds a call: the best of seven runs of about 3 ms each."""
    import torch
    call()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(True), torch.cuda.Event(True)
    best, n = float("inf"), 4
    for _ in range(8):
        e0.record()
        for _ in range(n):
            call()
        e1.record()
        torch.cuda.synchronize()
        us = e0.elapsed_time(e1) * 1000.0 / n
        n = int(min(60, max(4, 3000.0 / us)))
        best = min(best, us)
    return best


def _body(n, seed=0, noise=0.0):
    """int16 CT of an ellipsoid in air; noise: standard deviation of the air's."""
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*[np.linspace(-1, 1, n, dtype=np.float32)] * 3, indexing="ij")
    inside = (x / 0.8) ** 2 + (y / 0.6) ** 2 + (z / 0.85) ** 2 < 1.0
    tissue = rng.standard_normal(x.shape, dtype=np.float32) * 20.0 + 40.0
    air = rng.standard_normal(x.shape, dtype=np.float32) * noise - 1000.0
    return np.rint(np.where(inside, tissue, air)).astype(np.int16)


def _view(n, extent, W, h, sod=2.0):
    """A view that a volume of `extent` mm a side about fills."""
    sp = (extent / n,) * 3
    c = configs.volume_center((n, n, n), sp)
    d = np.array([1.0, 0.4, 0.3]) / np.linalg.norm([1.0, 0.4, 0.3])
    cam = abi.camera(c + sod * extent * d, c, (0, 0, 1), 30.0, (0.9 * extent, 3.1 * extent))
    return sp, abi.compute_view(cam, W, h, spacing=sp)


def _empty_window(view):
    """A keyhole plane that leaves every ray outside: the window is empty, but
    the view takes the casters that march one lane per ray."""
    v = abi.View.from_buffer_copy(view)
    v.n_keyhole_planes = 1
    v.keyhole_planes[:4] = [1.0, 0.0, 0.0, -1e6]
    return v


# A ray of an opaque table ends at its first sample: four lanes per ray took
# 1.4 to 2.0 times one lane's time here.
@pytest.mark.parametrize("caster", ["1d", "1d unshaded", "2d", "2d gradient magnitude", "dual", "inex"])
def test_opaque_tables_on_magnified_volumes_take_one_lane_per_ray(gpu_ctx, caster):
    import torch
    n, W, h, m = 128, 1400, 1100, 256
    sp, view = _view(n, 256.0, W, h)
    vol = _body(n)
    vh, vh2 = H.gpu_volume(gpu_ctx, vol, sp), H.gpu_volume(gpu_ctx, vol[::-1].copy(), sp)
    lo, w = -1024.0, 2500.0
    alpha = (np.arange(m) >= 0.4 * m).astype(np.float32)
    rgb = np.random.default_rng(1).uniform(0, 1, (m, 3)).astype(np.float32)
    out = torch.empty((h, W, 4), dtype=torch.uint8, device="cuda")
    full = np.ones((m, m), np.float32)
    tab = {"alpha": full * alpha, "red": 0.9 * full, "green": 0.5 * full, "blue": 0.2 * full, "ambient": 0.4 * full,
           "diffuse": 0.6 * full, "specular": 0.2 * full, "specular_power": 12.0 * full}
    march, over = (configs.march_params({"step_scale": 1.0, "term_T": t, "jitter": 1, "skip_rule": 1})
                   for t in (1.0 / 64.0, 1.0000001))
    if caster.startswith("1d"):
        p = (abi.Tf1dParams(lo, 1 / w, 0.0, float("inf"), 1.0, 0.0, 0.0, 1.0) if caster.endswith("unshaded") else
             abi.Tf1dParams(lo, 1 / w, 0.0, 1 / w, 0.4, 0.6, 0.2, 10.0))
        tf = abi.TF1D(gpu_ctx, alpha, rgb, p, galpha=full[0])
        call = lambda v, mp: abi.render_1d(gpu_ctx, vh, tf, v, mp, out)
    else:
        tf = abi.TF2D(gpu_ctx, tab, configs.tf2d_params(configs.tf2d_params_for(lo, lo + w, 0.0, 512.0)))
        if caster == "dual":
            dp = abi.DualParams(lo, 1 / w, lo, 1 / w)
            call = lambda v, mp: abi.render_dual(gpu_ctx, vh, vh2, tf, dp, v, mp, out)
        elif caster == "inex":
            tf.set_inex(0.3 * full * alpha)
            call = lambda v, mp: abi.render_2d_inex(gpu_ctx, vh, tf, v, mp, out, False)
        else:
            gm = caster.endswith("magnitude")
            if gm:
                vh.compute_gradmag(0, 512.0)
            call = lambda v, mp: abi.render_2d(gpu_ctx, vh, tf, v, mp, out, gm)
    # the in/ex caster takes one lane for thresholds above 1, the others for a
    # view with keyhole planes
    one = (view, over) if caster == "inex" else (_empty_window(view), march)
    us, ref_us = _us(lambda: call(view, march)), _us(lambda: call(*one))
    call(view, march)
    got = out.clone()
    if caster != "inex":
        call(*one)
        assert torch.equal(got, out)
    assert int((got[..., 3] > 0).sum()) > W * h // 10
    for o in (tf, vh, vh2):
        o.close()
    assert us <= 1.2 * ref_us, (us, ref_us)


# Bricks that are neither empty nor constant, and rays too short for runs:
# looking for runs, two lanes per ray and deals took 1.3 to 1.8 times the plain
# march's time.  A termination threshold that no ray reaches gives the plain
# march, one lane per ray.
@pytest.mark.parametrize("n,W,step,noise", [(256, 1024, 0.5, 20.0), (256, 760, 0.5, None), (64, 460, 1.0, 0.0)])
@pytest.mark.parametrize("skip", [0, 1])
def test_single_views_without_runs_cost_the_plain_march(gpu_ctx, n, W, step, noise, skip):
    import torch
    sp, view = _view(n, 256.0, W, W)
    rng = np.random.default_rng(3)
    vol = (np.rint(rng.standard_normal((n, n, n), dtype=np.float32) * 20.0 + 40.0).astype(np.int16) if noise is None
           else _body(n, noise=noise))
    vh = H.gpu_volume(gpu_ctx, vol, sp)
    march = configs.march_params({"step_scale": step, "term_T": 0.0, "jitter": 1, "skip_rule": skip})
    out = torch.empty((W, W), dtype=torch.float32, device="cuda")
    us, images = [], []
    for term, offset in ((0, 1.0), (1, 1e30)):
        d = abi.DrrParams()
        d.ct_intercept, d.ct_slope, d.ct_offset, d.ref_termination = 0.02, 2e-5, offset, term
        d.output = abi.DRR_F32_EXP_NEG_L
        call = lambda: abi.render_drr(gpu_ctx, vh, view, march, d, out)
        us.append(_us(call))
        images.append(out.clone())
    vh.close()
    assert torch.equal(images[0], images[1])
    assert float(images[0].min()) < 0.9
    assert us[0] <= 1.25 * us[1], us


# ---------------------------------------------------------------------------
# The volume gradient by ray tiles and by voxel bricks
def _grad_plan(ctx, vh, sp, n, views, output=abi.DRR_F32_L):
    march = configs.march_params({"step_scale": 0.6, "term_T": 0.0, "jitter": 1, "skip_rule": 0})
    drr = configs.drr_params({"intercept": 0.0, "slope": 1.0, "offset": 1.0, "output": output, "ref_termination": 0})
    return abi.DrrPlan(ctx, vh, views, march, drr)


def _orbit_view(n, sp, d, w, h, fov=40.0, dist=2.2):
    ext = max(k * s for k, s in zip(n, sp))
    c, d = configs.volume_center(n, sp), np.asarray(d, float) / np.linalg.norm(d)
    cam = abi.camera(c + dist * ext * d, c, (0, 0, 1) if abs(d[2]) < 0.9 else (0, 1, 0), fov / 1.4,
                     (0.5 * ext, (dist + 2.0) * ext))
    return abi.compute_view(cam, w, h, spacing=sp)


@pytest.mark.parametrize("d", [(1, 0.1, 0.05), (-1, 0.05, 0.1), (0.1, 1, 0.1), (0.05, -1, -0.1), (0.05, 0.02, 1),
                               (0.1, 0.1, -1), (0.7, -0.6, -0.5)])
@pytest.mark.parametrize("dtype,keyhole", [("f32", False), ("f32", True), ("i16", False)])
def test_volume_gradient_is_the_same_by_tiles_and_by_bricks(gpu_ctx, d, dtype, keyhole):
    """Copies of a view whose d loss / d image is zero add nothing, but make
    the tiles enough for the route by tiles (1248 against 0.5 * 1248 bricks);
    alone the view goes by bricks.  Rays along every axis in both senses."""
    import torch
    n, sp = (92, 60, 97), (1.0, 1.3, 0.9)
    rng = np.random.default_rng(5)
    vol = np.maximum(rng.uniform(-0.02, 0.04, n[::-1]), 0.0).astype(np.float32)
    vol[:, :20] = 0.0
    if dtype == "i16":
        vol = np.rint(vol * 1e4).astype(np.int16)
    view = _orbit_view(n, sp, d, 150, 131)
    if keyhole:
        view.n_keyhole_planes = 2
        view.keyhole_planes[:8] = [1.0, 0.2, 0.0, -0.3 * n[0], -1.0, 0.0, 0.1, 0.6 * n[0]]
    vh = H.gpu_volume(gpu_ctx, vol, sp)
    grads = []
    for copies in (1, 24):
        plan = _grad_plan(gpu_ctx, vh, sp, n, [view] * copies)
        img = torch.zeros(plan.total, device="cuda")
        plan.render(img)
        dldi = torch.zeros(plan.total, device="cuda")
        dldi[: plan.offsets[1]] = torch.from_numpy(np.random.default_rng(6).uniform(-1, 1, plan.offsets[1])).cuda()
        g = torch.full((vol.size,), float("nan"), device="cuda")
        plan.backward(img, dldi, grad_volume=g)
        torch.cuda.synchronize()
        grads.append(g)
        plan.close()
    vh.close()
    assert torch.equal(grads[0], grads[1])
    assert int((grads[0] != 0).sum()) > vol.size // 20


# One 64x64 view took 1674 us by tiles, a 256x256 one 622.
@pytest.mark.parametrize("n,views", [(256, 1), (128, 4)])
def test_volume_gradient_of_fewer_rays_costs_no_more(gpu_ctx, n, views):
    import torch
    sp = (256.0 / n,) * 3
    vol = np.maximum(1.0 + _body(n) / 1000.0, 0.0).astype(np.float32) * 0.02
    vh = H.gpu_volume(gpu_ctx, vol, sp)
    g = torch.empty(vol.size, device="cuda")
    us = []
    for w in (64, n):
        plan = _grad_plan(gpu_ctx, vh, sp, (n,) * 3,
                          [_orbit_view((n,) * 3, sp, (np.cos(0.7 * i), np.sin(0.7 * i), 0.2), w, w)
                           for i in range(views)])
        img, dldi = torch.zeros(plan.total, device="cuda"), torch.ones(plan.total, device="cuda")
        plan.render(img)
        us.append(_us(lambda: plan.backward(img, dldi, grad_volume=g)))
        plan.close()
    vh.close()
    assert us[0] <= 1.1 * us[1], us


def test_volume_gradient_where_its_sums_do_not_fit(gpu_ctx):
    """8 bytes a voxel for the sums of the route by tiles are not to be had:
    the gradient goes by bricks, with the same bits."""
    import torch
    n, sp = (1024, 1024, 640), (0.25, 0.25, 0.4)
    vol = torch.randint(0, 3, (n[2], n[1], n[0]), device="cuda", dtype=torch.uint8,
                        generator=torch.Generator(device="cuda").manual_seed(1))
    vol[:, 300:] = 0
    vh = abi.Volume(gpu_ctx, n, sp, np.uint8)
    vh.set_frame(0, vol)
    del vol
    view = _orbit_view(n, sp, (0.2, 1.0, 0.3), 1000, 900)
    got, hog = [torch.full((n[0] * n[1] * n[2],), float("nan"), device="cuda") for _ in range(2)], None
    for i in range(2):
        plan = _grad_plan(gpu_ctx, vh, sp, n, [view])
        img, dldi = torch.zeros(plan.total, device="cuda"), torch.ones(plan.total, device="cuda")
        plan.render(img)
        if i == 1:
            torch.cuda.synchronize()
            torch.cuda.empty_cache()
            free = torch.cuda.mem_get_info()[0]
            assert free > 8 * n[0] * n[1] * n[2]
            hog = torch.empty(free - (3 << 30), dtype=torch.uint8, device="cuda")
        plan.backward(img, dldi, grad_volume=got[i])
        torch.cuda.synchronize()
        plan.close()
    del hog
    vh.close()
    same = torch.equal(got[0], got[1])
    live = int((got[0] != 0).sum())
    del got
    torch.cuda.empty_cache()
    assert same and live > n[0] * n[1] * n[2] // 100


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("n_views,w", [(1, 90), (2, 140), (3, 300), (9, 300)])
def test_plan_results_do_not_depend_on_schedule_tile_or_order(gpu_ctx, n_views, w, skip):
    """16, 8, 4 and 2 lanes per ray (views of 8100 to 810000 rays in all):
    images, losses and the registration gradient to the bit."""
    import torch
    n, sp = (60, 52, 47), (1.0, 1.1, 1.2)
    rng = np.random.default_rng(7)
    vol = np.maximum(rng.uniform(-0.01, 0.02, n[::-1]), 0.0).astype(np.float32)
    vol[:, :, :15] = 0.0
    c = configs.volume_center(n, sp)
    views, dms = [], []
    for i in range(n_views):
        cam = configs.drr_camera(c, 0.4 + 0.9 * i, w, sod=300.0, sid=600.0, fov=200.0, half_extent=75.0)
        v, dm = abi.posed_view(cam, [0.05 * i, 0.1, -0.08, 1.0, -2.0, 0.5], c, w, w, spacing=sp, with_derivatives=True)
        views.append(v)
        dms.append(dm)
    march = configs.march_params({"step_scale": 0.15, "term_T": 0.0, "jitter": 1, "skip_rule": skip})
    drr = configs.drr_params({"intercept": 0.0, "slope": 1.0, "offset": 1.0, "output": abi.DRR_F32_EXP_NEG_L,
                              "ref_termination": 0})
    vh = H.gpu_volume(gpu_ctx, vol, sp)
    plan = abi.DrrPlan(gpu_ctx, vh, views, march, drr, dview=np.stack(dms))
    tgt = torch.from_numpy(rng.uniform(0, 1, plan.total).astype(np.float32)).cuda()
    ref = None
    for sched, wps in ((abi.SCHED_GRID, 4), (abi.SCHED_PERSISTENT, 2), (abi.SCHED_PERSISTENT, 8)):
        for shape in (abi.TILE_8X8, abi.TILE_16X4, abi.TILE_4X16):
            for order in (abi.ORDER_VIEWS, abi.ORDER_REGIONS):
                plan.set_schedule(sched, wps)
                plan.set_tile_shape(shape)
                plan.set_work_order(order)
                out, reg = (torch.full((plan.total,), float("nan"), device="cuda") for _ in range(2))
                loss, grad = torch.empty(n_views, device="cuda"), torch.empty(6 * n_views, device="cuda")
                plan.render(out)
                plan.register(reg, tgt, loss, grad)
                torch.cuda.synchronize()
                got = [out, reg, loss, grad]
                if ref is None:
                    ref = got
                assert all(torch.equal(a, b) for a, b in zip(ref, got)), (sched, wps, shape, order)
    assert float(ref[0].min()) < 0.95 and float(ref[3].abs().max()) > 0
    plan.close()
    vh.close()


def test_a_new_plan_reports_the_work_order_it_marches(gpu_ctx):
    """Setting the order that a plan reports leaves its time alone (view by view
    in bands, four poses of one body took 1.6 times as long)."""
    import torch
    n, w = 256, 512
    sp = (1.0,) * 3
    c = configs.volume_center((n,) * 3, sp)
    views = [abi.posed_view(configs.drr_camera(c, 0.02 * i, w, sod=600.0, sid=1000.0, fov=409.6, half_extent=225.0),
                            np.zeros(6), c, w, w, spacing=sp) for i in range(16)]
    march = configs.march_params({"step_scale": 0.5, "term_T": 0.0, "jitter": 1, "skip_rule": 0})
    drr = configs.drr_params({"intercept": 0.02, "slope": 2e-5, "offset": 1.0, "output": abi.DRR_F32_EXP_NEG_L,
                              "ref_termination": 0})
    vh = H.gpu_volume(gpu_ctx, _body(n), sp)
    plan = abi.DrrPlan(gpu_ctx, vh, views, march, drr)
    out = torch.empty(plan.total, device="cuda")
    assert plan.work_order() == abi.ORDER_REGIONS
    before = _us(lambda: plan.render(out))
    plan.set_work_order(plan.work_order())
    after = _us(lambda: plan.render(out))
    plan.close()
    vh.close()
    assert after <= 1.15 * before, (before, after)
