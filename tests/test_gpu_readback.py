"""The readback's canonical order and the upload's counts at the sizes where
their kernels change path, against the oracle's packer, bit for bit (needs a
GPU)."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_parity import f32, oracle_world, say
from tests.test_zz_no_alloc import Hip
from wrach_amd import World, WrachConfig, WrachError, _lib

pytestmark = pytest.mark.gpu


def packed_by_the_oracle(oracle, cfg, pos, vel):
    W, H = cfg.dimensions
    return oracle.pack(pos, vel, (0, 0, W, H), cfg.cell_size)


def assert_packed(got, want, what):
    for a, b, name in zip(got, want, ("indices", "positions", "velocities")):
        assert a.shape == b.shape, f"{what}: {name} shape"
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"{what}: {name} differ"


@pytest.mark.parametrize("m", [1, 2, 3, 16, 63, 64, 65, 128, 257, 703, 704, 705, 2048, 2049])
@pytest.mark.parametrize("shift", [0, 1, 37, 63])
def test_canonical_order_of_a_cell(oracle, m, shift):
    """A cell of m particles that starts at packed index `shift`, one of the
    same size right behind it, then a few lone ones, right after an upload:
    every particle is a run of its own there, in arbitrary order.  Cells
    inside a wavefront, past its end, over several, and those that a block
    sorts (over 704, in LDS and past it)."""
    rng = np.random.default_rng(100 * m + shift)
    n = shift + 2 * m + 5
    cell = np.concatenate([np.arange(shift) % 7, np.full(m, 8), np.full(m, 9), 12 + np.arange(5)])
    pos = f32(np.stack([cell + rng.uniform(0.01, 0.99, n), rng.uniform(0.01, 0.99, n)], 1))
    vel = f32(rng.uniform(-1, 1, (n, 2)))
    order = rng.permutation(n)
    pos, vel = pos[order], vel[order]
    cfg = WrachConfig(dimensions=(96, 64), cell_size=1)
    with World(cfg) as w:
        w.add_particles(pos, vel)
        assert_packed(w.read(), packed_by_the_oracle(oracle, cfg, pos, vel), f"m={m} shift={shift}")


@pytest.mark.parametrize("n", [1, 64, 65, 255, 257, 4000])
def test_upload_counts_with_particles_outside(oracle, n):
    """The inside count of the device binning from its striped count of the
    particles outside: none, some, all of them, and a refused upload's."""
    rng = np.random.default_rng(n)
    cfg = WrachConfig(dimensions=(60, 60), cell_size=3)
    for share in (0.0, 0.3, 1.0):
        pos = f32(rng.uniform(0, 60, (n, 2)))
        out = rng.uniform(0, 1, n) < share
        pos[out] = f32(rng.uniform(70, 90, (int(out.sum()), 2))) * np.where(rng.uniform(0, 1, (int(out.sum()), 1)) < 0.5,
                                                                         np.float32(-1), np.float32(1))
        vel = f32(rng.uniform(-1, 1, (n, 2)))
        say(f"[readback] upload of {n}, {int(out.sum())} outside")
        with World(cfg) as w:
            w.add_particles(pos, vel)
            want = packed_by_the_oracle(oracle, cfg, pos, vel)
            assert w.n_particles == len(want[1])
            assert_packed(w.read(), want, f"n={n} share={share}")
            many = np.tile(np.float32([[30, 30]]), (w.capacity + 1, 1))
            with pytest.raises(WrachError) as e:
                w.add_particles(many, np.zeros_like(many))
            assert e.value.code == _lib.WRACH_E_CAPACITY
            assert_packed(w.read(), want, f"n={n} share={share}, after a refused upload")


@pytest.mark.parametrize("m", [1, 8, 9, 64, 65, 300, 1200])
@pytest.mark.parametrize("offset", [0, 4])
def test_noalloc_frame_of_a_crowded_cell(oracle, m, offset):
    """The allocation-free frame's start: cells of up to 8 particles by their
    own thread, larger ones by their wavefront, more cells than particles and
    the reverse; pairs on the caller's side aligned as float2 and only as
    float; twice in a row, the second from what the first left."""
    hip = Hip()
    rng = np.random.default_rng(m + offset)
    n = m + 40
    pos = f32(np.concatenate([rng.uniform((3, 3), (3.99, 3.99), (m, 2)), rng.uniform(0, 30, (40, 2))]))
    vel = f32(rng.uniform(-1, 1, (n, 2)))
    cfg = WrachConfig(dimensions=(30, 30), cell_size=1, gravity=(0.0, -0.1))
    idx, pos, vel = packed_by_the_oracle(oracle, cfg, pos, vel)
    P = oracle.params(30, 30, 1, n, gravity=cfg.gravity)
    ws = _lib.WorldSettingsC()
    ws.view_dimensions[:] = [30.0, 30.0]
    ws.view_anchor[:] = [0.0, 0.0]
    ws.grid_dimensions[:] = [31, 31]
    ws.cell_size = 1
    ws.particles_in_frame_count = n
    g = (ctypes.c_float * 2)(*cfg.gravity)
    skip = offset // 4
    arrays = [idx, np.concatenate([np.zeros(skip, np.float32), pos.ravel()]),
              np.concatenate([np.zeros(skip, np.float32), vel.ravel()])]
    di, dp, dv = (hip.upload(a) for a in arrays)
    ref = (idx, pos, vel)
    try:
        for call in range(2):
            say(f"[readback] noalloc m={m} offset={offset} call {call}")
            assert _lib.load().wrach_frame_noalloc(ctypes.byref(ws), g, 1.0, di, dp.value + offset, dv.value + offset,
                                                   n, None) == 0
            assert hip.h.hipDeviceSynchronize() == 0
            ref = oracle.step(P, *ref)
            got = (hip.download(di, idx), hip.download(dp, arrays[1])[skip:].reshape(-1, 2),
                   hip.download(dv, arrays[2])[skip:].reshape(-1, 2))
            assert_packed(got, ref, f"m={m} offset={offset} call {call}")
    finally:
        hip.free(di, dp, dv)


@pytest.mark.parametrize("cells", [(2897, 2897), (4096, 2049), (11000, 800)])
def test_grids_just_above_the_large_scan(oracle, cells):
    """Grids of 2^23 cells and a little more (a last chunk that is not whole,
    one that ends with the grid, a row of a fraction of the chunks): offsets
    counted from their chunk's first cell until a readback.  Particles in the
    first and last cells, a crowded one, one chunk alone; read, stepped, read
    again, a world's count, an append, and Mode S passes from such offsets."""
    gx, gy = cells
    rng = np.random.default_rng(gx)
    W, H = gx - 1, gy - 1
    n = 3000
    pos = np.concatenate([rng.uniform((1, 1), (W - 1, 40), (n, 2)),             # the first chunks
                          rng.uniform((W - 60, H - 30), (W - 0.5, H - 0.5), (n, 2)),  # the last
                          rng.uniform((700, 500), (703, 503), (300, 2)),        # crowded, alone
                          [[0.0, 0.0], [W, H], [W, 0.0], [0.0, H]]])
    pos, vel = f32(pos), f32(rng.uniform(-0.4, 0.4, (len(pos), 2)))
    cfg = WrachConfig(dimensions=(W, H), cell_size=1, gravity=(0.0, -0.03))
    P, ref = oracle_world(oracle, cfg, pos, vel)
    say(f"[readback] grid {gx} x {gy}")
    with World(cfg) as w:
        w.add_particles(pos, vel)
        assert_packed(w.read(), ref, "upload")
        for per_lane in (4, 2, 1):  # every scatter of such a grid; 1 is the default
            w.set_tuning(scatter_per_lane=per_lane)
            w.step(1)
            ref = oracle.step(P, *ref, nsteps=1)
            assert_packed(w.read(), ref, f"{per_lane} a lane")
        for frames in (1, 5):
            w.step(frames)
            assert w.world_settings(0).particles_in_frame_count == len(ref[1])
            ref = oracle.step(P, *ref, nsteps=frames)
            assert_packed(w.read(), ref, f"{frames} frames")
        w.step(1)
        ref = oracle.step(P, *ref, nsteps=1)
        w.autotune(2)  # its snapshot holds offsets as the frame left them
        w.step(1)
        ref = oracle.step(P, *ref, nsteps=1)
        assert_packed(w.read(), ref, "after autotune")
        w.step(1)
        ref = oracle.step(P, *ref, nsteps=1)
        w.set_solver("S", 2)  # the offsets of a frame without passes
        w.step(2)
        *ref, st = oracle.step_s(P, *ref, max_passes=2, nsteps=2)
        assert_packed(w.read(), ref, "Mode S")
        assert w.solver_stats() == st
        w.set_solver("R")
        w.step(1)
        more = f32(rng.uniform(0, 30, (50, 2)))
        ref = oracle.step(P, *ref, nsteps=1)
        w.store_write_back()  # the append re-packs where the particles are now
        w.add_particles(more, more * 0)
        got = w.read()
        assert got[0][-1] == len(ref[1]) + 50 and np.all(np.diff(got[0].astype(np.int64)) >= 0)
        cell = np.floor(got[1][:, 1]).astype(np.int64) * gx + np.floor(got[1][:, 0]).astype(np.int64)
        assert np.array_equal(np.bincount(cell, minlength=gx * gy), np.diff(got[0][1:].astype(np.int64)))


@pytest.mark.parametrize("m", [65534, 65535, 70000])
def test_large_grid_with_a_chunk_past_16_bits(oracle, m):
    """A chunk of as many particles as 16-bit offsets hold, and more, beside
    ordinary ones: frames, Mode S passes and the readback."""
    rng = np.random.default_rng(m)
    gx, gy = 4099, 2053
    W, H = gx - 1, gy - 1
    cell = 1024 * 8 + np.arange(m) % 1000
    pos = np.concatenate([np.stack([cell % gx, cell // gx], 1) + rng.uniform(0.01, 0.99, (m, 2)),
                          rng.uniform((1, 20), (W - 1, 90), (2000, 2))])
    pos, vel = f32(pos), f32(rng.uniform(-0.2, 0.2, (m + 2000, 2)))
    cfg = WrachConfig(dimensions=(W, H), cell_size=1, gravity=(0.0, -0.01))
    P, ref = oracle_world(oracle, cfg, pos, vel)
    assert np.diff(ref[0][1:].astype(np.int64))[1024 * 8:1024 * 9].sum() == m
    say(f"[readback] chunk of {m}")
    with World(cfg) as w:
        w.add_particles(pos, vel)
        assert_packed(w.read(), ref, "upload")
        w.set_solver("S", 1)
        for frames in (1, 2):
            w.step(frames)
            *ref, st = oracle.step_s(P, *ref, max_passes=1, nsteps=frames)
            assert w.world_settings(0).particles_in_frame_count == len(ref[1])
            assert_packed(w.read(), ref, f"{frames} frames")
        w.set_solver("R")
        w.step(2)
        ref = oracle.step(P, *ref, nsteps=2)
        w.set_solver("S", 1)  # the offsets of a frame without passes
        w.step(1)
        *ref, st = oracle.step_s(P, *ref, max_passes=1, nsteps=1)
        assert_packed(w.read(), ref, "passes after plain frames")
        assert w.solver_stats() == st


@pytest.mark.parametrize("n", [0, 1, 4000, 180_000, 190_000])
def test_read_through_host_memory_and_by_copies(oracle, n):
    """Readbacks up to 4 MiB are stored to host memory by the kernel, larger
    ones copied (here 1.2 MB of offsets, and the pairs of 180,000 and 190,000
    particles just below and above): all of the triple, parts of it, again
    without a frame between, and the device's own canonical arrays after it."""
    rng = np.random.default_rng(n)
    cfg = WrachConfig(dimensions=(600, 500), cell_size=1, gravity=(0.0, -0.02))
    say(f"[readback] read of {n}")
    with World(cfg) as w:
        done = 0
        for add in (n // 3, n - n // 3):  # a longer readback each time
            pos, vel = f32(rng.uniform(0, 500, (add, 2))), f32(rng.uniform(-1, 1, (add, 2)))
            w.add_particles(pos, vel)
            done += add
            got = w.read()
            assert len(got[1]) == done and got[0][-1] == done
        if n:
            w.step(3)
        first = w.read()
        P = oracle.params(600, 500, 1, n, gravity=cfg.gravity)
        want = got if n == 0 else oracle.step(P, *got, nsteps=3)
        assert_packed(first, want, "read")
        assert_packed(w.read(), want, "read again")
        idx, pos, vel = np.zeros(len(want[0]), np.uint32), np.zeros((max(n, 1), 2), np.float32), np.zeros((max(n, 1), 2), np.float32)
        L, count = _lib.load(), ctypes.c_uint32()
        f32p, u32p = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_uint32)
        assert L.wrach_read(w._h, None, vel.ctypes.data_as(f32p), max(n, 1), None, 0, ctypes.byref(count)) == 0
        assert L.wrach_read(w._h, pos.ctypes.data_as(f32p), None, max(n, 1), idx.ctypes.data_as(u32p), len(idx), None) == 0
        assert count.value == n
        assert_packed((idx, pos[:n], vel[:n]), want, "parts")
        hip = Hip()
        view = w.device_state(canonical=True)
        w.sync()
        assert np.array_equal(hip.download(ctypes.c_void_p(view.indices), idx), want[0])
        if n:
            assert np.array_equal(hip.download(ctypes.c_void_p(view.positions), pos).view(np.uint32),
                                  want[1].view(np.uint32))


@pytest.mark.parametrize("n", [0, 1, 4000, 16384])
def test_small_transfers_without_pinned_memory(oracle, n):
    """Uploads and readbacks small enough for pinned host memory, where there
    is none: before any, and after some was in use."""
    rng = np.random.default_rng(50 + n)
    cfg = WrachConfig(dimensions=(160, 128), cell_size=1, gravity=(0.0, -0.1))
    pos, vel = f32(rng.uniform(0, (160, 128), (n, 2))), f32(rng.uniform(-1, 1, (n, 2)))
    more, still = f32(rng.uniform(0, 100, (50, 2))), np.zeros((50, 2), np.float32)
    P, ref = oracle_world(oracle, cfg, pos, vel)
    say(f"[readback] without pinned memory, {n}")
    for used in (False, True):
        with World(cfg) as w:
            if used:
                w.add_particles(pos, vel)
                assert_packed(w.read(), ref, "with pinned memory")
                w.test_no_staging()
            else:
                w.test_no_staging()
                w.add_particles(pos, vel)
            assert_packed(w.read(), ref, f"used={used}")
            if n:
                w.step(2)
                assert_packed(w.read(), oracle.step(P, *ref, nsteps=2), f"used={used}, after 2 frames")
            w.add_particles(more, still)
            assert_packed(w.read(), packed_by_the_oracle(oracle, cfg, np.concatenate([pos, more]),
                                                         np.concatenate([vel, still])), f"used={used}, appended")


@pytest.mark.parametrize("offset", [0, 4])
@pytest.mark.parametrize("fault", ["start", "end", "past", "descends", "alternates", "last cell", "none filled"])
def test_noalloc_frame_leaves_a_bad_triple(oracle, fault, offset):
    """Offsets that do not ascend from 0 to n: the call's kernels find it and
    the caller's arrays stay as they were; the next call, on the good triple,
    is the frame."""
    hip = Hip()
    rng = np.random.default_rng(60)
    n, W, H = 5000, 90, 70
    cfg = WrachConfig(dimensions=(W, H), cell_size=1, gravity=(0.0, -0.1))
    pos = f32(np.concatenate([rng.uniform((3, 3), (3.99, 3.99), (1500, 2)), rng.uniform(0, (W, H), (n - 1500, 2))]))
    vel = f32(rng.uniform(-1, 1, (n, 2)))
    idx, pos, vel = packed_by_the_oracle(oracle, cfg, pos, vel)
    ws = _lib.WorldSettingsC()
    ws.view_dimensions[:] = [float(W), float(H)]
    ws.view_anchor[:] = [0.0, 0.0]
    ws.grid_dimensions[:] = [W + 1, H + 1]
    ws.cell_size = 1
    ws.particles_in_frame_count = n
    bad = idx.copy()
    if fault == "start":
        bad[1] = 1
    elif fault == "end":
        bad[-1] = n - 1
    elif fault == "past":
        bad[-40:] = n + 7
    elif fault == "descends":
        bad[len(bad) // 2] = 0
    elif fault == "alternates":  # every second cell's range is all of them
        bad[1::2], bad[2::2] = 0, n
    elif fault == "last cell":
        bad[-2] = n + 1
    else:
        bad[:] = 0
    g = (ctypes.c_float * 2)(*cfg.gravity)
    skip = offset // 4
    flat = [np.concatenate([np.zeros(skip, np.float32), a.ravel()]) for a in (pos, vel)]
    say(f"[readback] noalloc, bad offsets: {fault}, offset {offset}")
    for _ in range(2):
        for offsets, want in ((bad, (bad, pos, vel)),
                              (idx, oracle.step(oracle.params(W, H, 1, n, gravity=cfg.gravity), idx, pos, vel))):
            di, dp, dv = (hip.upload(a) for a in (offsets, *flat))
            try:
                assert _lib.load().wrach_frame_noalloc(ctypes.byref(ws), g, 1.0, di, dp.value + offset,
                                                       dv.value + offset, n, None) == 0
                assert hip.h.hipDeviceSynchronize() == 0
                got = (hip.download(di, offsets), hip.download(dp, flat[0])[skip:].reshape(-1, 2),
                       hip.download(dv, flat[1])[skip:].reshape(-1, 2))
                assert_packed(got, want, f"{fault} offset={offset} {'bad' if offsets is bad else 'good'}")
            finally:
                hip.free(di, dp, dv)


def test_autotune_leaves_what_changes_no_launch():
    """A grid that scans by chunks has no scan shape to choose, and a small
    world's grids of queued cells launch the same blocks: the autotuner keeps
    them, whichever trial a clock finds the shortest."""
    rng = np.random.default_rng(70)
    say("[readback] autotune")
    with World(WrachConfig(dimensions=(4096, 2048), cell_size=1)) as w:
        w.add_particles(f32(rng.uniform(0, (4096, 100), (3000, 2))), f32(rng.uniform(-1, 1, (3000, 2))))
        for shape in ((1024, 8), (512, 16), (1024, 64)):
            w.set_tuning(scan_threads=shape[0], scan_items=shape[1])
            got = w.autotune(2)
            assert (got["scan_threads"], got["scan_items"]) == shape
    with World(WrachConfig(dimensions=(512, 512), cell_size=1)) as w:
        w.add_particles(f32(rng.uniform(0, 512, (6000, 2))), f32(rng.uniform(-1, 1, (6000, 2))))
        grid = w.tuning()["cells_grid"]
        assert grid // 2 >= 6000 // 64 + 64  # every candidate launches as many
        for _ in range(4):
            assert w.autotune(2)["cells_grid"] == grid
