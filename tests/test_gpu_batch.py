"""Batched passes: every scene of a batch must come out exactly as it does alone.

One voxelize / mips / trace call over many scenes of uneven size (different triangle
counts, grids, level counts, G-buffer sizes, precisions, an empty scene) is compared
with the same scenes run one call each: accumulator records, every mip level and the
traced outputs must be identical bit for bit (the kernels do the same integer and float
operations per scene; only the workgroup-to-scene mapping differs). The single-scene
path is itself held to the oracle by the other GPU tests, and the full-size batch (64
scenes of 1k-200k triangles on grids up to 256^3) is checked against the oracle scene by
scene.
"""
import numpy as np
import pytest

from final184_amd import scenegen as sg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _vgi():
    from final184_amd import vgi
    return vgi


def _workloads():
    w = sg.batch_scenes(count=5, median=3000.0, tri_range=(200, 12_000), grids=(16, 32, 64),
                        sides=(24, 40, 64))
    # an empty scene and a scene whose grid is smaller than one bin of 16
    empty = sg.batch_scenes(seed=7, count=1, median=10, tri_range=(1, 1), grids=(8,), sides=(16,))[0]
    empty.positions = empty.positions[:0]
    empty.albedo = empty.albedo[:0]
    w.append(empty)
    # different level counts than the default chain
    w[0].grid["levels"] = 1
    w[1].grid["levels"] = 3
    return w


class Job:
    def __init__(self, ctx, w):
        vgi = _vgi()
        self.w = w
        self.meshes = [vgi.MeshData(ctx, w.positions.reshape(-1, 3), albedo=w.albedo)] \
            if w.num_triangles else []
        self.grid = vgi.make_grid(**w.grid)
        self.lights = vgi.make_lights(w.lights)
        self.gb = vgi.GBufferData(ctx, w.gb_pos, w.gb_nrm, w.width, w.height)
        self.cones = vgi.make_cones(**w.cones)
        self.od = vgi.DeviceArray.empty(ctx, (w.num_pixels, 4), np.float32)
        self.os = vgi.DeviceArray.empty(ctx, (w.num_pixels, 4), np.float32)
        self.scene = ctx.scene()

    def levels(self):
        return [self.scene.read_level(k) for k in range(self.w.grid["levels"])]


def _run_alone(ctx, jobs, precs):
    for j, p in zip(jobs, precs):
        j.scene.voxelize(j.meshes, j.grid)
        j.scene.build_mips(j.lights, p)
        j.scene.trace(j.gb, j.cones, j.od, j.os)
    ctx.sync()


def _run_batch(ctx, jobs, precs, stream=None):
    ctx.voxelize_batch([(j.scene, j.meshes, j.grid) for j in jobs], stream)
    for p in sorted(set(precs)):
        ctx.build_mips_batch([(j.scene, j.lights) for j, q in zip(jobs, precs) if q == p], p, stream)
    ctx.trace_batch([(j.scene, j.gb, j.cones, j.od, j.os) for j in jobs], stream)
    ctx.sync(stream)


def _compare(a, b):
    for ja, jb in zip(a, b):
        name = ja.w.name
        sa, sb = ja.scene.stats(), jb.scene.stats()
        if sa.bin_size == sb.bin_size:  # pair and work counts depend on the bin size, voxels do not
            assert sa.bin_pairs == sb.bin_pairs and sa.work_items == sb.work_items, name
        assert np.array_equal(ja.scene.read_voxels(), jb.scene.read_voxels()), f"{name}: voxels differ"
        for k, (la, lb) in enumerate(zip(ja.levels(), jb.levels())):
            assert np.array_equal(la, lb), f"{name}: level {k} differs"
        assert np.array_equal(ja.od.numpy(), jb.od.numpy()), f"{name}: diffuse differs"
        assert np.array_equal(ja.os.numpy(), jb.os.numpy()), f"{name}: specular differs"


@pytest.mark.parametrize("bin_size,tile,order", [(8, (16, 16), 0), (16, (32, 8), 0), (32, (8, 8), 0),
                                                  (16, (16, 16), 1)])
def test_batch_equals_alone(ctx, bin_size, tile, order):
    """Alone runs use the default screen tiles; the batch runs under each tuning,
    Morton pixel order included: every pixel's result must be the same bits."""
    vgi = _vgi()
    print(f"case batch_equals_alone bin={bin_size} tile={tile} order={order}", flush=True)
    try:
        ws = _workloads()
        precs = [vgi.PREC_FP16, vgi.PREC_FP32, vgi.PREC_FP16X2, vgi.PREC_BF16, vgi.PREC_FP16, vgi.PREC_FP16X2]
        alone = [Job(ctx, w) for w in ws]
        batch = [Job(ctx, w) for w in ws]
        _run_alone(ctx, alone, precs)
        ctx.set_tuning(bin_size=bin_size, chunk_tris=64, tile_w=tile[0], tile_h=tile[1], pixel_order=order)
        _run_batch(ctx, batch, precs)
        _compare(alone, batch)
        # the empty scene holds nothing
        assert not batch[-1].scene.read_voxels().any()
        # a second batch call reuses the workspace and the scenes' allocations
        _run_batch(ctx, batch, precs)
        _compare(alone, batch)
    finally:
        ctx.set_tuning()


@pytest.mark.parametrize("frames", [1, 2, 4, 5, 17])
def test_morton_key_bits(ctx, frames):
    """The sort key holds a frame's number and, in the bits that leaves of 32 (30 at most),
    its pixels' Morton codes: one, two and four frames leave 30, five 29, seventeen 27.
    Pixels in the grid's last cell share the padding's code; others lie outside the grid."""
    vgi = _vgi()
    print(f"case morton_key_bits frames={frames}", flush=True)
    w = sg.batch_scenes(count=1, median=3000.0, tri_range=(2000, 4000), grids=(32,), sides=(64,))[0]
    job = Job(ctx, w)
    _run_alone(ctx, [job], [vgi.PREC_FP16])
    rng = np.random.default_rng(frames)
    sides = [(64, 64), (16, 16), (17, 15), (1, 1), (33, 40)]
    size = np.float32(w.grid["extent"])
    corner = np.asarray(w.grid["origin"], np.float32) + size
    gbs, outs = [], []
    for i in range(frames):
        width, height = sides[i % len(sides)]
        pick = rng.integers(0, w.num_pixels, width * height)
        pos, nrm = w.gb_pos.reshape(-1, 3)[pick].copy(), w.gb_nrm.reshape(-1, 3)[pick]
        pos[rng.random(len(pick)) < 0.2] = corner * np.float32(1 - 1e-6)
        pos[rng.random(len(pick)) < 0.1] += 2 * size
        gbs.append(vgi.GBufferData(ctx, pos, nrm, width, height))

    def run():
        out = [[vgi.DeviceArray.empty(ctx, (g.num_pixels, 4), np.float32) for _ in range(2)] for g in gbs]
        ctx.trace_batch([(job.scene, g, job.cones, d, s) for g, (d, s) in zip(gbs, out)])
        ctx.sync()
        return [[x.numpy() for x in o] for o in out]

    try:
        tiles = run()
        ctx.set_tuning(pixel_order=vgi.ORDER_MORTON)
        for a, b in zip(tiles, run()):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    finally:
        ctx.set_tuning()


def test_batch_two_streams(ctx):
    """Two batches on two streams at once give the same results as one after the other."""
    vgi = _vgi()
    print("case batch_two_streams", flush=True)
    ws = _workloads()
    precs = [vgi.PREC_FP16] * len(ws)
    alone = [Job(ctx, w) for w in ws]
    _run_alone(ctx, alone, precs)
    s1, s2 = ctx.stream_create(), ctx.stream_create()
    try:
        a = [Job(ctx, w) for w in ws[:3]]
        b = [Job(ctx, w) for w in ws[3:]]
        ctx.voxelize_batch([(j.scene, j.meshes, j.grid) for j in a], s1)
        ctx.voxelize_batch([(j.scene, j.meshes, j.grid) for j in b], s2)
        ctx.build_mips_batch([(j.scene, j.lights) for j in a], vgi.PREC_FP16, s1)
        ctx.build_mips_batch([(j.scene, j.lights) for j in b], vgi.PREC_FP16, s2)
        ctx.trace_batch([(j.scene, j.gb, j.cones, j.od, j.os) for j in a], s1)
        ctx.trace_batch([(j.scene, j.gb, j.cones, j.od, j.os) for j in b], s2)
        ctx.sync(s1)
        ctx.sync(s2)
        assert ctx.workspace_bytes() > 0
        _compare(alone, a + b)
    finally:
        ctx.stream_destroy(s1)
        ctx.stream_destroy(s2)


def test_batch_rejects_duplicates(ctx):
    vgi = _vgi()
    w = _workloads()[2]
    j = Job(ctx, w)
    with pytest.raises(vgi.VgiError) as e:
        ctx.voxelize_batch([(j.scene, j.meshes, j.grid), (j.scene, j.meshes, j.grid)])
    assert e.value.code == -1
    j.scene.voxelize(j.meshes, j.grid)
    with pytest.raises(vgi.VgiError):
        ctx.build_mips_batch([(j.scene, j.lights), (j.scene, j.lights)], vgi.PREC_FP16)
    # a scene that is not voxelized cannot join a mips batch
    other = ctx.scene()
    with pytest.raises(vgi.VgiError) as e:
        ctx.build_mips_batch([(j.scene, j.lights), (other, j.lights)], vgi.PREC_FP16)
    assert e.value.code == -5


def test_autotune_picks_a_candidate_and_keeps_results(ctx):
    vgi = _vgi()
    print("case autotune", flush=True)
    ws = _workloads()
    precs = [vgi.PREC_FP16] * len(ws)
    alone = [Job(ctx, w) for w in ws]
    _run_alone(ctx, alone, precs)
    jobs = [Job(ctx, w) for w in ws]
    try:
        r = ctx.autotune_batch([(j.scene, j.meshes, j.grid) for j in jobs],
                               [(j.scene, j.lights) for j in jobs],
                               [(j.scene, j.gb, j.cones, j.od, j.os) for j in jobs],
                               vgi.PREC_FP16, reps=2)
        assert list(r.bin_sizes) == [8, 16, 32]
        assert [tuple(t) for t in r.tiles] == [(8, 8, 0), (16, 16, 0), (32, 8, 0), (16, 16, 1)]
        assert all(v > 0 for v in r.build_ms) and all(v > 0 for v in r.trace_ms)
        t = ctx.get_tuning()
        assert (t.bin_size, t.tile_w, t.tile_h) == (r.best.bin_size, r.best.tile_w, r.best.tile_h)
        best = min(r.frame_ms[b][j] for b in range(3) for j in range(4))
        bb = [8, 16, 32].index(r.best.bin_size)
        bt = [(8, 8, 0), (16, 16, 0), (32, 8, 0), (16, 16, 1)].index(
            (r.best.tile_w, r.best.tile_h, r.best.pixel_order))
        assert r.frame_ms[bb][bt] == best
        print("autotune", r.as_dict(), flush=True)
        _compare(alone, jobs)
    finally:
        ctx.set_tuning()


def _rel_l2(x, y):
    return float(np.linalg.norm(x - y) / max(np.linalg.norm(y), 1e-30))


@pytest.mark.parametrize("order", [1, 0])
def test_full_batch_vs_oracle(ctx, order):
    """The 64-scene batch at its measured size (triangle counts lognormal, median 20k,
    clipped to 1k-200k; grids 32^3-256^3; G-buffers 256^2-1024^2; FP16 mips), voxelized,
    built and traced in one call per stage. Per scene: accumulator bit-exact vs the oracle,
    every FP16 level bit-exact, and a seeded 1024-pixel subset within 1e-3 relative L2 of
    the oracle's FP64 run and within 1e-5 of its FP32 run on the same FP16 levels. Morton
    pixel order (the autotuner's choice for these point-sampled G-buffers) and screen
    tiles."""
    vgi = _vgi()
    print(f"case full batch (64 scenes) order={order}", flush=True)
    ws = sg.batch_scenes()
    assert len(ws) == 64 and max(w.num_triangles for w in ws) <= 200_000
    jobs = [Job(ctx, w) for w in ws]
    try:
        ctx.set_tuning(bin_size=8, chunk_tris=64, tile_w=16, tile_h=16, pixel_order=order)
        _run_batch(ctx, jobs, [vgi.PREC_FP16] * len(jobs))
        worst = 0.0
        for i, j in enumerate(jobs):
            w = j.w
            acc, st = orc.voxelize(w.positions, w.grid, albedo=w.albedo)
            got = j.scene.read_voxels()
            assert np.array_equal(got, acc), f"{w.name}: {(got != acc).any(axis=-1).sum()} voxels differ"
            del got
            ref16 = orc.inject_mips(acc, w.grid, w.lights, "fp16")
            for k in range(w.grid["levels"]):
                assert np.array_equal(j.scene.read_level(k), ref16[k]), f"{w.name}: level {k} differs"
            sub = np.random.default_rng(i).choice(w.num_pixels, 1024, replace=False)
            lv64 = orc.inject_mips(acc, w.grid, w.lights, f64=True)
            d64, s64, _ = orc.trace(lv64, w.grid, w.gb_pos, w.gb_nrm, w.cones, pixels=sub, f64=True)
            d32, s32, _ = orc.trace(ref16, w.grid, w.gb_pos, w.gb_nrm, w.cones, pixels=sub)
            d, s = j.od.numpy()[sub], j.os.numpy()[sub]
            got = np.concatenate([d[:, :3], s[:, :3]], 1)
            e64 = _rel_l2(got, np.concatenate([d64[:, :3], s64[:, :3]], 1))
            e32 = _rel_l2(got, np.concatenate([d32[:, :3], s32[:, :3]], 1))
            assert e64 <= 1e-3, f"{w.name}: {e64:.3e} vs FP64"
            assert e32 <= 1e-5, f"{w.name}: {e32:.3e} vs the oracle's FP32 run"
            worst = max(worst, e64)
            j.scene.release()
        print(f"worst scene rel L2 vs FP64 = {worst:.3e}", flush=True)
    finally:
        ctx.set_tuning()


def test_bin_scan_across_more_workgroups_than_fit_at_once(ctx):
    """Two 512^3 scenes (1024 k_bins workgroups each with 8^3 bins) ahead of a 64^3 soup in
    one voxelize batch: the soup's workgroups come after 2048 others, more than the GPU
    holds at once (8 of them per CU), so its bins' offsets come from a look-back over
    predecessors that ran in earlier waves. The soup's voxels must equal the oracle's,
    and no scene may have taken the per-triangle path."""
    vgi = _vgi()
    big = [sg.random_soup(seed=s, ntri=400, n=512, levels=1, width=8, height=8) for s in (11, 12)]
    small = sg.random_soup(ntri=6000, n=64, width=8, height=8)
    print("case voxelize batch 2 x 512^3 + 64^3 (2050 k_bins workgroups)", flush=True)
    scenes, jobs = [], []
    try:
        ctx.set_tuning(bin_size=8)
        for w in big + [small]:
            s = ctx.scene()
            scenes.append(s)
            jobs.append((s, [vgi.MeshData(ctx, w.positions.reshape(-1, 3), albedo=w.albedo)], vgi.make_grid(**w.grid)))
        ctx.voxelize_batch(jobs)
        for s in scenes:
            assert s.stats().voxelize_fallback == 0
        ref, _ = orc.voxelize(small.positions, small.grid, albedo=small.albedo)
        got = scenes[-1].read_voxels()
        assert np.array_equal(got, ref), f"{(got != ref).any(axis=-1).sum()} voxels differ"
    finally:
        ctx.set_tuning()
        for s in scenes:
            s.release()
