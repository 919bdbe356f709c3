"""GPU tests of the neighbour passes' branches against the FP32 twin (bit for
bit): streams of candidates shorter and longer than one segment of row marks
(256 positions) and ones ending on its edges, cells of more than 1,023
particles, smoothing lengths above and at 1 (the clamped kernel serves lengths
up to 1), coincident and almost coincident neighbours, scenes that leave part
of a wave empty."""
import numpy as np
import pytest

import oracle as O
import sphe
from gpu_common import orc_scene_from
from sphe import scenes

pytestmark = pytest.mark.gpu


def _params(h, half, dt=1e-5, centre=0.0):
    return sphe.default_params(h=h, mass=0.02 * (h / 0.0457) ** 3, dt=dt, box_half=half, box_center=(centre,) * 3)


def _compare(p, pos, yz, precision=sphe.FP32, comp=1, steps=2):
    n = len(pos)
    pos = np.ascontiguousarray(pos, dtype=np.float32)
    ctx = sphe.Context(precision)
    ctx.set_yz_split(yz)
    sid = ctx.add_scene(p)
    ctx.set_particles(sid, pos)
    ctx.step(steps)
    gp, gv = ctx.state_f64(sid)
    rho = ctx.density(sid)
    osc = orc_scene_from(p)
    osc.yz = yz
    st = dict(pos=pos.astype(np.float64), vel=np.zeros((n, 3)), sed=np.zeros(n, np.int64))
    for _ in range(steps):
        st = O.orc_step(osc, st["pos"], st["vel"], st["sed"], np.arange(n, dtype=np.int32), real=4, comp=comp)
    assert np.array_equal(gp, st["pos"]) and np.array_equal(gv, st["vel"])
    assert np.array_equal(rho.astype(np.float64), st["rho"])


@pytest.mark.parametrize("yz", [1, 2])
@pytest.mark.parametrize("n,edge", [(1, 0.5), (15, 0.3), (66, 0.5), (255, 0.4), (256, 0.4), (257, 0.4), (273, 0.4),
                                    (512, 0.45), (700, 1.5), (2500, 1.2)])
def test_stream_lengths_bit_exact_twin(n, edge, yz):
    """n particles in a cube of `edge` smoothing lengths: in the small cubes
    every particle is a candidate of every other, so streams have n positions
    (256 and 512 end on a segment's edge); 2,500 fill cells past 1,023."""
    h = 0.0457
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, edge * h, (n, 3)) + 0.013
    _compare(_params(h, 0.2), pos, yz)


@pytest.mark.parametrize("h", [1.0, 1.7, 0.02])
@pytest.mark.parametrize("precision,comp", [(sphe.FP32, 1), (sphe.FP32_NAIVE, 0)])
def test_smoothing_lengths_bit_exact_twin(h, precision, comp):
    """Lengths above 1 take the kernels without the clamp; 1 is its limit."""
    rng = np.random.default_rng(7)
    pos = rng.uniform(-1.6 * h, 1.6 * h, (900, 3))
    _compare(_params(h, 4.0 * h), pos, 2, precision, comp)


@pytest.mark.parametrize("yz", [1, 2])
def test_coincident_neighbours_bit_exact_twin(yz):
    """Neighbours at distance 0, just inside and just outside 1e-4 among
    ordinary ones, at every place of the list's groups of four."""
    h = 0.0457
    rng = np.random.default_rng(3)
    base = rng.uniform(-0.06, 0.06, (300, 3))
    near = np.repeat(base[:40], 3, axis=0)
    near[0::3] += 0.0
    near[1::3, 0] += 9.9e-5
    near[2::3, 1] += 1.02e-4
    pos = np.concatenate([base, near])[rng.permutation(420)]
    _compare(_params(h, 0.2, dt=1e-6), pos, yz)


def _cells(p, yz=2):
    """Cells of a scene's grid (one pad cell not counted)."""
    ctx = sphe.Context()
    ctx.set_yz_split(yz)
    sid = ctx.add_scene(p)
    c = ctx.debug_consts(sid)
    return int(c["dim_x"] * c["dim_y"] * c["dim_z"])


@pytest.mark.parametrize("tiles", [2, 16, 17, 4096, 4097])
def test_scan_forms_give_the_same_steps(tiles):
    """The cell scan takes one launch up to 16 tiles, two up to 4,096, three
    beyond: a scene steps to the same bits beside scenes that bring the
    context to exactly that many tiles (of 2,048 cells)."""
    h = 0.0457
    p = _params(h, 0.2, dt=1e-4)
    rng = np.random.default_rng(11)
    pos = rng.uniform(-0.12, 0.12, (2000, 3)).astype(np.float32)
    alone = sphe.Context()
    s0 = alone.add_scene(p)
    alone.set_particles(s0, pos)
    alone.step(6)
    want = alone.state_f64(s0)

    ctx = sphe.Context()
    ctx.set_scan_tile(11)
    sid = ctx.add_scene(p)
    ctx.set_particles(sid, pos)
    # other scenes, the largest first, while more than a tile is left; a
    # scene's cells are followed by one pad cell, the context's by one more
    left = 2048 * tiles - (_cells(p) + 1) - 1
    for half in (2.9, 0.4, 0.2, 0.1, 0.05, 0.01):
        n = _cells(_params(h, half)) + 1
        while left >= 2048 and n <= left:
            left -= n
            o = ctx.add_scene(_params(h, half, dt=1e-4))
            # three falling particles, so that far tiles fill and empty
            ctx.set_particles(o, np.float32(0.4 * half) * np.array([[1, 1, 1], [-1, 1, 1], [1, -1, 1]], np.float32))
    assert 0 <= left < 2048  # the last tile is partly filled
    ctx.step(6)
    got = ctx.state_f64(sid)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    assert ctx.status() == 0


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP32_NAIVE, sphe.FP64])
def test_inspection_by_list_equals_by_walk(lanes, precision):
    """A record from the neighbour list (in its 32 entries, in the overflow
    chunk, past both) is the stencil walk's bit for bit; new lists, which hold
    nothing until the next step, are not read."""
    rng = np.random.default_rng(3)
    pos = rng.normal(0.0, 0.035, (1500, 3)).astype(np.float32)
    recs = []
    for renewed in (False, True):
        ctx = sphe.Context(precision)
        ctx.set_lanes(lanes)
        sid = ctx.add_scene(_params(0.0457, 0.5))
        ctx.set_particles(sid, pos)
        ctx.set_list_capacity(32)
        counts = ctx.debug_neighbours(sid, csr=False)[0] - 1
        assert (counts <= 32).any() and ((counts > 32) & (counts <= 64)).any() and (counts > 64).any()
        ctx.step(1)
        if renewed:
            ctx.set_list_capacity(1024)
        ids = np.concatenate([np.argsort(counts)[[0, 1, -2, -1]], np.flatnonzero(counts == 32)[:3],
                              np.flatnonzero((counts > 32) & (counts <= 64))[::40], np.arange(0, 1500, 250)])
        recs.append([bytes(ctx.particle(sid, int(i))) for i in ids])
    assert recs[0] == recs[1]


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
def test_small_and_large_reads(precision):
    """Positions, velocities and densities of scenes whose values fit the
    staging buffer (read by the id map) and do not (gathered in device memory),
    beside a scene of sparse ids, after steps, edits and the hooks that sort
    again: the state's own values in id order."""
    rng = np.random.default_rng(8)
    ctx = sphe.Context(precision)
    ids = [None, None, np.arange(700, dtype=np.int32) * 3 + 5, None, None]
    sids = []
    for n, i in zip((1, 1000, 700, 21845, 21846), ids):  # 21,845 positions: 4 bytes below the buffer's size
        pos = rng.uniform(-0.3, 0.3, (n, 3)).astype(np.float32)
        sids.append(ctx.add_scene(_params(0.0457, 0.4)))
        ctx.set_particles(sids[-1], pos, ids=i)

    def check():
        got = [(ctx.positions(s), ctx.velocities(s), ctx.density(s)) for s in sids]
        for s, (pos, vel, rho) in zip(sids, got):
            gp, gv = ctx.state_f64(s)
            assert np.array_equal(pos, gp.astype(np.float32)) and np.array_equal(vel, gv.astype(np.float32))
            if len(rho) in (1, 1000):
                assert rho[-1] == ctx.particle(s, len(rho) - 1).Density and rho[0] == ctx.particle(s, 0).Density
    for steps in (1, 2):
        ctx.step(steps)
        check()
        ctx.step(1)
        ctx.debug_density(sids[1])  # sorts the state again, in other slots than its own
        for s in sids:
            pos, vel = ctx.positions(s), ctx.velocities(s)
            gp, gv = ctx.state_f64(s)
            assert np.array_equal(pos, gp.astype(np.float32)) and np.array_equal(vel, gv.astype(np.float32))
    ctx.set_particles(sids[1], ctx.positions(sids[1])[::-1].copy())
    ctx.step(1)
    check()


@pytest.mark.parametrize("cluster", [1, 255, 256, 257, 300, 512, 513, 1400, 2048, 2100])
def test_reorder_windows_bit_exact_twin(cluster):
    """A cell of `cluster` particles among scattered ones, met at several
    offsets of the blocks of 256 slots: ranked from the block's own words and
    256 on either side, from its cells' words, or from memory."""
    h = 0.0457
    rng = np.random.default_rng(cluster)
    pos = np.concatenate([rng.uniform(-0.19, 0.0, (300 + 37 * (cluster % 5), 3)),
                          0.005 + rng.uniform(0.0, 0.01 * h, (cluster, 3)), rng.uniform(0.06, 0.19, (200, 3))])
    pos = pos[rng.permutation(len(pos))]
    _compare(_params(h, 0.2, dt=1e-9), pos, 2, sphe.FP32, 1, 1)


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
@pytest.mark.parametrize("sizes", [(64,), (63, 65, 2), (128, 64, 192)])
def test_two_phase_sums_in_mixed_batches(sizes, precision):
    """Scenes without erosion, with atomic and with two-phase erosion in one
    context, over terrains of odd and even sizes: every scene's terrain,
    sediment and state are those of the scene alone with atomic erosion (or
    without), and no sum of an earlier step is left over."""
    batch = sphe.Context(precision)
    want, ids = [], []
    for k, T in enumerate(sizes):
        for mode in (sphe.EROSION_TWO_PHASE, sphe.EROSION_ATOMIC, sphe.EROSION_OFF):
            sc = scenes.dam_break_scene(50 + k, 900 + 131 * k, 0.3, T, erosion=mode, steps=4)
            ids.append(batch.add_synthetic(sc))
            alone = scenes.dam_break_scene(50 + k, 900 + 131 * k, 0.3, T, steps=4,
                                           erosion=min(mode, sphe.EROSION_ATOMIC))
            ctx = sphe.Context(precision)
            sid = ctx.add_synthetic(alone)
            ctx.step(19)
            ctx.step(1)
            want.append((ctx.terrain_volume_fx(sid), ctx.sediment_fx(sid)) + ctx.state_f64(sid))
    batch.step(19)
    batch.step(1)
    assert any((w[1] != 0).any() for w in want)
    for sid, w in zip(ids, want):
        got = (batch.terrain_volume_fx(sid), batch.sediment_fx(sid)) + batch.state_f64(sid)
        assert all(np.array_equal(a, b) for a, b in zip(got, w))


@pytest.mark.parametrize("graph", [True, False])
def test_scan_tile_changed_between_steps(graph):
    """The tiles' totals, counted by the step before for the old tile size, are
    counted again for the new one: the states stay those of an unchanged
    context bit for bit."""
    rng = np.random.default_rng(12)
    pos = rng.uniform(-0.9, 0.9, (3000, 3)).astype(np.float32)
    pos[:2000] *= 0.2
    ctxs = []
    for _ in range(2):
        ctx = sphe.Context()
        ctx.use_graph(graph)
        sid = ctx.add_scene(_params(0.0457, 1.0))
        ctx.set_particles(sid, pos)
        ctx.step(2)
        ctxs.append(ctx)
    for log2 in (11, 13, 12, 11):
        ctxs[0].set_scan_tile(log2)
        for ctx in ctxs:
            ctx.step(3)
        assert ctxs[0].status() == 0
        a, b = ctxs[0].state_f64(sid), ctxs[1].state_f64(sid)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("block", [64, 256, 512])
@pytest.mark.parametrize("yz", [1, 2])
@pytest.mark.parametrize("n", [256, 512, 768, 1024])
def test_streams_that_end_with_a_segment(n, yz, block):
    """Every particle is a candidate of every other, so all streams end with a
    segment of row marks, the ones of a block's last group too: the look-up past
    their end finds no marks, and the sums and lists are the twin's."""
    h = 0.0457
    rng = np.random.default_rng(n + yz)
    pos = (rng.uniform(0.0, 0.4 * h, (n, 3)) + 0.013).astype(np.float32)
    p = _params(h, 0.2)
    ctx = sphe.Context()
    ctx.set_yz_split(yz)
    ctx.set_tuning(block, 1)
    sid = ctx.add_scene(p)
    ctx.set_particles(sid, pos)
    ctx.step(1)
    gp, gv = ctx.state_f64(sid)
    osc = orc_scene_from(p)
    osc.yz = yz
    st = O.orc_step(osc, pos.astype(np.float64), np.zeros((n, 3)), np.zeros(n, np.int64),
                    np.arange(n, dtype=np.int32), real=4, comp=1)
    assert np.array_equal(gp, st["pos"]) and np.array_equal(gv, st["vel"])
    assert np.array_equal(ctx.density(sid).astype(np.float64), st["rho"])


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
@pytest.mark.parametrize("n", [600, 22000])
@pytest.mark.parametrize("saved,other", [("sparse", "dense"), ("dense", "sparse"), ("sparse", "shifted")])
def test_restored_state_with_other_ids(saved, other, n, precision):
    """A state restored over the same number of particles of other ids reads as
    in a context that never held those: positions, velocities and densities
    (22,000: past the staging buffer), records, absent ids refused."""
    ids = {"sparse": 2 * np.arange(n, dtype=np.int32), "dense": np.arange(n, dtype=np.int32)}
    ids["shifted"] = ids["sparse"] + 1
    rng = np.random.default_rng(n)
    pos = rng.uniform(-0.3, 0.3, (n, 3)).astype(np.float32)
    ctxs = []
    for replaced in (True, False):
        ctx = sphe.Context(precision)
        sid = ctx.add_scene(_params(0.0457, 0.4))
        ctx.set_particles(sid, pos, ids=ids[saved])
        if replaced:
            ctx.save_state()
            ctx.set_particles(sid, pos[::-1].copy(), ids=ids[other])
            ctx.step(1)
            ctx.positions(sid)
            ctx.particle(sid, int(ids[other][3]))
            ctx.restore_state()
        ctx.step(1)
        ctxs.append(ctx)

    def reads(ctx):
        yield ctx.positions(sid)
        yield ctx.velocities(sid)
        yield ctx.density(sid)
        yield ctx.read(sid, sphe.BUF_ID)
        yield from ctx.state_f64(sid)
    for got, want in zip(reads(ctxs[0]), reads(ctxs[1])):
        assert np.array_equal(got, want)
    present = set(ids[saved].tolist())
    for i in (0, 1, 2, 3, n - 1, n, 2 * n - 2, 2 * n - 1, 2 * n):
        if i in present:
            assert bytes(ctxs[0].particle(sid, i)) == bytes(ctxs[1].particle(sid, i))
        else:
            for ctx in ctxs:
                with pytest.raises(sphe.SpheError):
                    ctx.particle(sid, i)


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
@pytest.mark.parametrize("change", [dict(h=0.0447), dict(h=0.0463), dict(mass=0.021)])
def test_inspection_after_a_change_of_parameters(change, precision):
    """Parameters that reach the device between a step and an inspection (here
    with the mass bookkeeping) make the record one of the new parameters over
    the neighbours they give, whether or not the step's lists are still there."""
    rng = np.random.default_rng(5)
    pos = rng.uniform(-0.15, 0.15, (2500, 3)).astype(np.float32)
    recs = []
    for renewed in (False, True):
        ctx = sphe.Context(precision)
        sid = ctx.add_scene(_params(0.0457, 0.2))
        ctx.set_particles(sid, pos)
        ctx.step(1)
        prm = ctx.get_params(sid)
        for k, v in change.items():
            setattr(prm, k, v)
        ctx.set_params(sid, prm)
        ctx.mass(sid)
        if renewed:
            ctx.set_list_capacity(1024)
        recs.append([bytes(ctx.particle(sid, i)) for i in range(0, 2500, 50)])
    assert recs[0] == recs[1]
    ctx.step(1)
    ctx.particle(sid, 0)


@pytest.mark.parametrize("n,lanes,split,persistent,density,force", [
    (1000, 4, 2, False, 64, 64), (1000, 1, 2, False, 64, 64), (1000, 4, 3, False, 64, 64),
    (1000, 4, 2, True, 256, 256), (1000, 8, 1, True, 256, 256),
    (2 ** 21, 4, 2, False, 64, 64), (2 ** 21 + 1, 4, 2, False, 256, 128), (2 ** 21 + 1, 4, 3, False, 64, 128),
    (2 ** 21 + 1, 2, 1, False, 64, 128), (2 ** 21 + 1, 4, 1, True, 256, 256)])
def test_block_sizes_by_kernel_and_size(n, lanes, split, persistent, density, force):
    """The block sizes in effect until some are set, by the kernels that serve
    the context; one that is set is taken for all."""
    ctx = sphe.Context()
    ctx.set_yz_split(split)
    ctx.set_lanes(lanes)
    ctx.set_persistent(persistent)
    sid = ctx.add_scene(_params(0.0457, 2.0))
    ctx.set_particles(sid, np.linspace(-1.9, 1.9, 3 * n, dtype=np.float32).reshape(n, 3))
    ctx.mass(sid)  # builds the layout; a line of this many particles is not stepped
    assert (ctx.get_tuning()[0], ctx.get_force_block()) == (density, force)
    ctx.set_tuning(512, 1)
    assert (ctx.get_tuning()[0], ctx.get_force_block()) == (512, 512)
    ctx.set_force_block(128)
    assert (ctx.get_tuning()[0], ctx.get_force_block()) == (512, 128)


def test_lists_grow_within_a_call_while_counts_rise():
    """A cluster that contracts (no forces): its counts pass the lists' 32
    entries in the first call of 16 steps and list and overflow chunk (64) in
    the second, more than two steps before its end.  The lists have grown when
    the second call is done, as they do one step at a time."""
    g = np.array([(a, b, c) for a in range(6) for b in range(6) for c in range(6)]) - 2.5
    jitter = np.random.default_rng(21).uniform(-0.05, 0.05, g.shape)
    cluster = (g + jitter) * 0.0235
    # far neighbours, so that the pool has a chunk for every particle of the cluster
    k = np.arange(2048)
    far = np.stack([k // 256 * 0.07, k // 16 % 16 * 0.07, k % 16 * 0.07], 1) + (0.3, -0.5, -0.5)
    pos = np.concatenate([cluster, far]).astype(np.float32)
    vel = np.zeros_like(pos)
    vel[:216] = -0.01 * pos[:216] / 1e-3
    p = sphe.default_params(h=0.0457, mass=0.02, dt=1e-3, box_half=1.0, box_center=(0.0, 0.0, 0.0), stiffness=0.0,
                            visc=0.0, surf_tens=0.0, gravity=(0.0, 0.0, 0.0))

    def context():
        ctx = sphe.Context()
        ctx.set_list_capacity(32)
        sid = ctx.add_scene(p)
        ctx.set_particles(sid, pos, vel)
        return ctx, sid
    single, sid = context()
    most = []
    for _ in range(32):
        single.step(1)
        single.sync()
        most.append(int(single.debug_neighbours(sid, csr=False)[0].max()) - 1)  # at the end of the step
    assert most[0] <= 32 < most[14] and max(most[:15]) <= 64 < min(most[27:])
    ctx, sid = context()
    ctx.step(16)
    ctx.sync()
    assert ctx.get_list_capacity() == 32
    ctx.step(16)
    ctx.sync()
    assert ctx.get_list_capacity() > 64
    for a, b in zip(ctx.state_f64(sid), single.state_f64(sid)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("filler", [0, 2 ** 20])
@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
def test_reads_of_single_scenes_of_a_batch(precision, filler):
    """Scenes of a batch read and inspected one by one, in other orders after
    each step, a scene again before and after another's edit: the values of the
    scene alone.  Among them are one particle, a whole wave, sparse ids, ids
    with a gap and double ids.  The first scene read after a step is mapped by
    itself, the first three in a context of 2^20 particles more, the next one
    with all others."""
    rng = np.random.default_rng(31)
    sizes = (1, 64, 700, 333, 65, 1000)
    ids = [None, None, np.arange(700) * 7, np.r_[0:100, 140:373], np.r_[0:40, 20:45], None]
    poss = [rng.uniform(-0.15, 0.15, (n, 3)).astype(np.float32) for n in sizes]

    def add(ctx, k):
        sid = ctx.add_scene(_params(0.0457, 0.2, dt=1e-4))
        ctx.set_particles(sid, poss[k], ids=None if ids[k] is None else ids[k].astype(np.int32))
        return sid
    batch = sphe.Context(precision)
    sids = [add(batch, k) for k in range(6)]
    if filler:
        o = batch.add_scene(_params(0.0457, 3.0))
        batch.set_particles(o, rng.uniform(-2.9, 2.9, (filler, 3)).astype(np.float32))
    alone = []
    for k in range(6):
        ctx = sphe.Context(precision)
        alone.append((ctx, add(ctx, k)))

    def compare(k):
        ctx, sid = alone[k]
        i = 0 if ids[k] is None else int(ids[k][len(ids[k]) // 2])
        assert bytes(batch.particle(sids[k], i)) == bytes(ctx.particle(sid, i))
        for which in (sphe.BUF_POS, sphe.BUF_VEL, sphe.BUF_DENSITY):
            assert np.array_equal(batch.read(sids[k], which), ctx.read(sid, which))
    for order in ((5, 0, 1, 2), (4, 3, 5, 4), (1, 2, 0, 5, 3)):
        batch.step(2)
        for ctx, _ in alone:
            ctx.step(2)
        for k in order:
            compare(k)
    for ctx, sid in ((batch, sids[1]), alone[1]):
        ctx.set_particles(sid, poss[1][::-1].copy())
        ctx.step(1)
    for k in (0, 2, 3, 4, 5):
        alone[k][0].step(1)
    for k in (3, 1, 5, 2, 0, 4):
        compare(k)


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
def test_reads_at_the_edges_of_the_mapped_memory(precision):
    """Sizes on both sides of what a context holds from its creation (16,128
    bytes: 1,344 positions, 4,032 densities) and of what the first larger read
    takes, the small after the large ones: the state's own values; records
    between them."""
    rng = np.random.default_rng(9)
    ctx = sphe.Context(precision)
    sids = []
    for n in (1344, 1345, 4032, 4033, 21845, 21846):
        sids.append(ctx.add_scene(_params(0.0457, 0.5)))
        ctx.set_particles(sids[-1], rng.uniform(-0.45, 0.45, (n, 3)).astype(np.float32))
    for order in ((0, 2, 1, 3, 4, 5), (5, 4, 3, 2, 1, 0)):
        ctx.step(1)
        got = {}
        for k in order:
            got[k] = [ctx.density(sids[k]), ctx.positions(sids[k]), ctx.velocities(sids[k])]
            p = ctx.particle(sids[k], 1000)
            assert p.Density == got[k][0][1000] and list(p.Position) == got[k][1][1000].tolist()
        for k in order:
            gp, gv = ctx.state_f64(sids[k])
            assert np.array_equal(got[k][1], gp.astype(np.float32)) and np.array_equal(got[k][2], gv.astype(np.float32))


@pytest.mark.parametrize("tiles", [4096, 4097])
def test_marked_tiles_give_the_counted_ones_steps(tiles):
    """Above 2^21 slots the tiles are only marked and their totals added up by
    the scan: a scene of 2^21 - 64 particles, and a small one, step to the same
    bits in such a context (of exactly that many tiles at first, so one launch
    less or more) as alone, where the totals are counted; the tile size changes
    between steps."""
    h = 0.0457
    n = 2 ** 21 - 64
    k = np.arange(n)
    rng = np.random.default_rng(4)
    far = (np.stack([k >> 14, k >> 7 & 127, k & 127], 1) * 0.045 - 2.85).astype(np.float32)
    near = rng.uniform(-0.12, 0.12, (2000, 3)).astype(np.float32)

    def add(ctx, half, pos):
        sid = ctx.add_scene(_params(h, half, dt=1e-4))
        ctx.set_particles(sid, pos)
        return sid
    alone = []
    for half, pos in ((2.9, far), (0.2, near)):
        ctx = sphe.Context()
        alone.append((ctx, add(ctx, half, pos)))
    both = sphe.Context()
    both.set_scan_tile(11)
    sids = [add(both, 2.9, far), add(both, 0.2, near)]
    left = 2048 * tiles - (_cells(_params(h, 2.9)) + 1) - (_cells(_params(h, 0.2)) + 1) - 1
    for half in (0.4, 0.2, 0.1, 0.05, 0.01):
        c = _cells(_params(h, half)) + 1
        while left >= 2048 and c <= left:
            left -= c
            add(both, half, np.float32(0.4 * half) * np.array([[1, 1, 1], [-1, 1, 1], [1, -1, 1]], np.float32))
    assert 0 <= left < 2048  # the last tile is partly filled
    for log2 in (11, 12, 13, 11):
        both.set_scan_tile(log2)
        for ctx in [both] + [c for c, _ in alone]:
            ctx.step(2)
    assert both.status() == 0
    for sid, (ctx, other) in zip(sids, alone):
        for which in (sphe.BUF_POS, sphe.BUF_VEL, sphe.BUF_DENSITY):
            assert np.array_equal(both.read(sid, which), ctx.read(other, which))


@pytest.mark.parametrize("tiles", [4097, 8192, 8193, 16385, 40000])
def test_prefix_of_many_tiles(tiles):
    """More than 4,096 tiles get their prefixes from a launch of its own, which
    reads the totals by lines: 2 lines a thread up to 8,192 tiles, 4 to 16,384,
    then 8 and more.  The same scene over the first cells, the last ones and some
    between steps to the bits of the scene alone, while far tiles fill and empty."""
    h = 0.0457
    p = _params(h, 0.2, dt=1e-4)
    pos = np.random.default_rng(11).uniform(-0.12, 0.12, (2000, 3)).astype(np.float32)
    three = np.array([[1, 1, 1], [-1, 1, 1], [1, -1, 1]], np.float32)

    def probe(ctx):
        sid = ctx.add_scene(p)
        ctx.set_particles(sid, pos)
        return sid
    alone = sphe.Context()
    s0 = probe(alone)
    ctx = sphe.Context()
    ctx.set_scan_tile(11)
    cells = {half: _cells(_params(h, half)) + 1 for half in (2.9, 1.0, 0.4, 0.2, 0.1, 0.05, 0.01)}
    sids = [probe(ctx)]
    left = 2048 * tiles - 1 - 4 * cells[0.2]
    for half in sorted(cells, reverse=True):
        while left >= 2048 and cells[half] <= left:
            left -= cells[half]
            o = ctx.add_scene(_params(h, half, dt=1e-4))
            ctx.set_particles(o, np.float32(0.4 * half) * three)
            if len(sids) < 3 and left < 2048 * tiles // (1 + len(sids)):
                sids.append(probe(ctx))
    while len(sids) < 4:
        sids.append(probe(ctx))
    assert 0 <= left < 2048  # the last tile is partly filled
    for k in (1, 5):
        ctx.step(k)
        alone.step(k)
        for sid in sids:
            for which in (sphe.BUF_POS, sphe.BUF_VEL, sphe.BUF_DENSITY):
                assert np.array_equal(ctx.read(sid, which), alone.read(s0, which))
    assert ctx.status() == 0


@pytest.mark.parametrize("precision", [sphe.FP32, sphe.FP64])
@pytest.mark.parametrize("n", [4096, 4097, 8192, 8193, 20000])
def test_many_particles_a_tile(n, precision):
    """More than 4,096 particles to a scan tile only mark it: a scene over one or
    two tiles steps to the same bits as beside an empty scene of many tiles,
    where the particles are counted; the tile size changes between steps."""
    h = 0.0457
    pos = np.random.default_rng(n).uniform(-0.19, 0.19, (n, 3)).astype(np.float32)
    ctxs = []
    for wide in (False, True):
        ctx = sphe.Context(precision)
        sid = ctx.add_scene(_params(h, 0.2, dt=1e-5))
        ctx.set_particles(sid, pos)
        if wide:
            ctx.add_scene(_params(h, 1.0))
        ctxs.append(ctx)
    for log2 in (12, 11, 13, 12):
        for ctx in ctxs:
            ctx.set_scan_tile(log2)
            ctx.step(3)
    for a, b in zip(ctxs[0].state_f64(sid), ctxs[1].state_f64(sid)):
        assert np.array_equal(a, b)
    assert ctxs[0].status() == 0


def test_contexts_of_several_threads():
    """Threads with a context each, that capture sequences of new lengths while
    others upload, download, grow their lists and inspect: no call fails and
    every state is that of the same calls in one thread."""
    import threading

    def work(i):
        ctx = sphe.Context()
        ctx.set_list_capacity(32)
        sid = ctx.add_synthetic(scenes.dam_break_scene(60 + i, 1500 + 100 * i, 0.3, 64))
        out = []
        ctx.step(20)
        ctx.save_state()
        for k in (3, 4, 5, 3, 4, 5, 40, 7, 40, 7, 9, 9):
            ctx.step(k)
            out += ctx.state_f64(sid)
            ctx.particle(sid, 5)
            out.append(ctx.terrain_heights(sid))
            if k == 7:
                ctx.set_particles(sid, ctx.positions(sid), ctx.velocities(sid))
            if k == 40:
                ctx.restore_state()
        return out
    want = [work(i) for i in range(6)]
    for _ in range(4):
        got, failed = [None] * 6, []

        def run(i):
            try:
                got[i] = work(i)
            except Exception as e:  # noqa: BLE001  (reported below)
                failed.append(e)
        threads = [threading.Thread(target=run, args=(i,)) for i in range(6)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not failed, failed
        for a, b in zip(got, want):
            assert all(np.array_equal(x, y) for x, y in zip(a, b))
