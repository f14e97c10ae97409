"""The C ABI's calls beside the forms the package runs: each against its
replacement on the same inputs, with garbage in the buffers it has to set up.

  tgs_isect_tiles_count / _emit          tgs_isect_tiles_plan / _emit_plan
  tgs_tide_camera_centers, _visibility,  tgs_tide_begin and the _begun calls
    _project_fwd
  tgs_tide_rasterize_fwd / _bwd          the _ordered and _split calls
  tgs_tide_loss                          tgs_tide_loss_summed
  tgs_resident_adam_step / _sophia_step  the _checked calls
"""
import types

import numpy as np
import pytest
import torch

from oracle import raster_ref as R
from tests.gpu_util import announce, rel_l2, to_np
from tidegs_amd import GPUResidentAdam, GPUResidentSophia, scenes
from tidegs_amd import _native as N
from tidegs_amd.tide_step import RANGE_SLOTS, TideStep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,n,packed", [(1, 1, False), (1, 257, False), (3, 5000, False), (3, 5000, True)])
def test_isect_count_and_emit(gpu, C, n, packed):
    announce(f"isect count and emit C={C} n={n} packed={packed}")
    rng = np.random.default_rng(n)
    tw, th = 13, 9
    m2d = rng.uniform(-8, [tw * 16 + 8, th * 16 + 8], size=(C, n, 2)).astype(np.float32)
    radii = rng.integers(-2, 30, size=(C, n)).astype(np.int32)
    m2d[0, 0], radii[0, 0] = 1.0, 3
    depths = rng.uniform(0.2, 50, size=(C, n)).astype(np.float32)
    cam = np.sort(rng.integers(0, C, size=C * n)) if packed else None
    o_tiles, o_ids, o_flat = R.isect_tiles(
        *((a.reshape(-1, 2) if a is m2d else a.reshape(-1)) if packed else a
          for a in (m2d, radii, depths)), 16, tw, th, sort=False, camera_ids=cam)
    m, r, d = (torch.from_numpy(a).to(gpu) for a in (m2d, radii, depths))
    c = None if cam is None else torch.from_numpy(cam).to(gpu)
    lib, s, total = N.load(), N.stream_handle(gpu), C * n
    bits = (tw * th).bit_length()
    tiles = torch.full((total,), -9, dtype=torch.int32, device=gpu)
    cum = torch.empty(total, dtype=torch.int64, device=gpu)
    ws = torch.empty(lib.tgs_scan_workspace_size(total), dtype=torch.uint8, device=gpu)
    N.call("tgs_isect_tiles_count", total, N.ptr(m), N.ptr(r), 16, tw, th, N.ptr(tiles), s)
    N.call("tgs_inclusive_scan_i32_i64", N.ptr(tiles), N.ptr(cum), total, N.ptr(ws), ws.numel(), s)
    count = int(cum[-1])
    assert count == o_ids.size
    np.testing.assert_array_equal(to_np(tiles), o_tiles.reshape(-1))

    plan_c, plan_n = (1, total) if packed else (C, n)
    plan = torch.empty(lib.tgs_isect_tiles_plan_size(plan_c, plan_n), dtype=torch.uint8, device=gpu)
    summary = torch.empty(2 + 2 * plan_c, dtype=torch.int64, device=gpu)
    tiles2 = torch.full_like(tiles, -9)
    N.call("tgs_isect_tiles_plan", plan_c, plan_n, N.ptr(m), N.ptr(r), N.ptr(d), 16, tw, th,
           N.ptr(tiles2), N.ptr(plan), plan.numel(), N.ptr(summary), s)
    assert int(summary[0]) == count and torch.equal(tiles, tiles2)

    out = []
    for form in ("emit", "plan"):
        ids = torch.full((count,), -1, dtype=torch.int64, device=gpu)
        flat = torch.full((count,), -1, dtype=torch.int32, device=gpu)
        if form == "emit":
            N.call("tgs_isect_tiles_emit", total, 0 if packed else n, N.ptr(c), N.ptr(m), N.ptr(r),
                   N.ptr(d), N.ptr(cum), 16, tw, th, bits, N.ptr(ids), N.ptr(flat), s)
        else:
            N.call("tgs_isect_tiles_emit_plan", plan_c, plan_n, N.ptr(c), N.ptr(m), N.ptr(r),
                   N.ptr(d), N.ptr(tiles2), N.ptr(plan), 16, tw, th, bits, N.ptr(ids), N.ptr(flat), s)
        out.append((to_np(ids), to_np(flat)))
    for ids, flat in out:
        np.testing.assert_array_equal(ids, o_ids)
        np.testing.assert_array_equal(flat, o_flat)


def _plain_forms(call, used):
    """N.call with the step's calls replaced by the plain ones: set-up buffers
    filled with garbage where the plain call sets them up itself."""
    def replaced(name, *a):
        s = a[-1]
        if name == "tgs_tide_begin":
            C, vm, campos, visible, projected, totals, _ = a
            for ptr, words in ((visible, 2 * RANGE_SLOTS), (projected, 2 * RANGE_SLOTS), (totals, 2 * C)):
                call("tgs_fill_u32", ptr, words, 0x1234567, s)
            name, a = "tgs_tide_camera_centers", (C, vm, campos, s)
        elif name in ("tgs_tide_visibility_begun", "tgs_tide_project_fwd_begun"):
            name = name[:-len("_begun")]
        elif name == "tgs_tide_rasterize_fwd_ordered":
            name, a = "tgs_tide_rasterize_fwd", a[:13] + a[14:]
        elif name == "tgs_tide_rasterize_fwd_split":
            name, a = "tgs_tide_rasterize_fwd", (*a[:13], None, *a[13:15], s)
        elif name == "tgs_tide_rasterize_bwd_ordered":
            name, a = "tgs_tide_rasterize_bwd", (*a[:15], s)
        elif name == "tgs_tide_rasterize_bwd_split":
            name, a = "tgs_tide_rasterize_bwd", (*a[:15], s)
        elif name == "tgs_tide_loss_summed":
            B, sums = a[0], a[8]
            call("tgs_fill_u32", sums, 4 * B, 0, s)
            name, a = "tgs_tide_loss", (*a[:7], *a[8:])
        used.add(name)
        return call(name, *a)
    return replaced


@pytest.mark.parametrize("n,C,W,H", [(3000, 3, 96, 64),      # split
                                     (4000, 9, 330, 300)])   # ordered, not split (3591 tiles)
def test_plain_step_calls(gpu, monkeypatch, n, C, W, H):
    announce(f"plain step calls n={n} C={C} {W}x{H}")
    sc = scenes.small(seed=4, n=n, n_cams=C, W=W, H=H, log_scale_mu=-2.3)
    ref = TideStep(sc.params.to(gpu).contiguous(), W, H, batch_size=C, keep_isect_ids=True)
    r_touched, r_grads, r_stats = ref.forward_backward(sc.viewmats, sc.Ks, sc.gt)
    used = set()
    monkeypatch.setattr(N, "call", _plain_forms(N.call, used))
    ts = TideStep(sc.params.to(gpu).contiguous(), W, H, batch_size=C, keep_isect_ids=True)
    touched, grads, stats = ts.forward_backward(sc.viewmats, sc.Ks, sc.gt)
    for name in ("camera_centers", "visibility", "project_fwd", "rasterize_fwd", "rasterize_bwd", "loss"):
        assert f"tgs_tide_{name}" in used
    assert not any(name.endswith(("_begun", "_ordered", "_split", "_summed")) for name in used)
    assert ts.depth_sort_repairs == 0  # both ranges were set up
    assert torch.equal(touched, r_touched) and stats.isects_per_camera == r_stats.isects_per_camera
    for key in ("campos", "entries", "splats", "isect_ids", "flatten_ids", "offsets", "images", "alphas",
                "last_ids", "v_images"):
        assert torch.equal(ts.last[key], ref.last[key]), key
    np.testing.assert_allclose(to_np(stats.loss_sums), to_np(r_stats.loss_sums), rtol=1e-12)
    # the backward's sums in another order: float32, as between the raster kernels' forms
    assert rel_l2(to_np(grads), to_np(r_grads)) < 2e-5


@pytest.mark.parametrize("cls", [GPUResidentAdam, GPUResidentSophia])
def test_unchecked_optimizer_step(gpu, monkeypatch, cls):
    announce(f"{cls.__name__} without the check")
    rows, block = 5000, 512
    blocks = -(-rows // block)
    mgr = types.SimpleNamespace(loaded_blocks=list(range(blocks)), local_to_global_idx=torch.empty(0),
                                block_to_gpu_slice={b: slice(b * block, min(rows, (b + 1) * block))
                                                    for b in range(blocks)})
    g = torch.Generator().manual_seed(1)
    init = torch.randn((rows, 59), generator=g)
    ids = torch.sort(torch.randperm(rows, generator=g)[:1700]).values.to(gpu)
    grad = (torch.randn((1700, 59), generator=g) * 1e-2).to(gpu)
    call, used = N.call, set()

    def unchecked(name, *a):
        if name in ("tgs_resident_adam_step_checked", "tgs_resident_sophia_step_checked"):
            name, a = name[:-len("_checked")], (*a[:-2], a[-1])
        used.add(name)
        return call(name, *a)

    out = []
    for wrapper in (call, unchecked):
        monkeypatch.setattr(N, "call", wrapper)
        table = init.to(gpu)
        gs = types.SimpleNamespace(gpu_working_set_manager=mgr, optimizer=types.SimpleNamespace(
            columns_lr=torch.tensor([0.01, 0.02, 0.03, 0.04, 0.05, 0.06]),
            param_groups=[{"betas": (0.9, 0.99), "eps": 1e-12}]))
        grads, c = {}, 0
        for name, attr, w, _ in cls.COMPONENT_SPECS:
            setattr(gs, attr, table[:, c:c + w])
            grads[name] = grad[:, c:c + w]
            c += w
        opt = cls(batch_size=2, block_size=block, device="cuda")
        opt.set_resident_blocks(range(blocks))
        for it in (1, 2, 3):
            opt.step(it, gs, ids, grads)
        out.append((table, opt._exp_avg, opt._exp_avg_sq))
    plain = "tgs_resident_adam_step" if cls is GPUResidentAdam else "tgs_resident_sophia_step"
    assert plain in used and not any(name.endswith("_checked") for name in used)
    for a, b in zip(*out):
        assert torch.equal(a, b)
    assert not torch.equal(out[0][0], init.to(gpu))
