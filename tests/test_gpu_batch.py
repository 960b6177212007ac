"""The one-launch batched path: every map's results equal the oracle's
sequential application of insert -> retrieve -> erase -> clean, and equal the
per-map path's; graph replays repeat the eager result."""
import numpy as np
import pytest
import torch

import oracle as O
from hashinator_amd import _lib, hn_tune
from hashinator_amd import workloads as W
from hashinator_amd.batch import BatchedMaps
from tests.helpers import live_pairs, next_overflow, occupancy, reachable_all

pytestmark = pytest.mark.gpu


def small_batch(key_bits=32, n_maps=96, seed=7):
    rng = np.random.default_rng(seed)
    sps = rng.integers(1, 13, size=n_maps)
    ins, vals, qry, ers = [], [], [], []
    for m, sp in enumerate(sps):
        n = int(rng.uniform(0.3, 0.95) * (1 << int(sp)))
        k = W.unique_keys(n, key_bits, seed * 1000 + m)
        a = W.unique_keys(max(1, n // 2), key_bits, seed * 1000 + m, start=n + 2)
        ins.append(k)
        vals.append(W.values(k, m).astype(k.dtype))
        qry.append(rng.permutation(np.concatenate([k, a])))
        ers.append(rng.choice(k, int(0.25 * n), replace=False) if n else k[:0])
    return sps, ins, vals, qry, ers


def check_against_oracle(bm, wl, key_bits, ops=_lib.HN_BATCH_ALL):
    sps, ins, vals, qry, ers = wl
    for m, sp in enumerate(sps):
        model = O.GpuModel(int(sp), key_bits)
        if ops & _lib.HN_BATCH_INSERT:
            model.insert(ins[m], vals[m])
        if ops & _lib.HN_BATCH_RETRIEVE:
            ev, eh = model.retrieve(qry[m])
            v, h = bm.results(m)
            assert np.array_equal(h, eh), m
            assert np.array_equal(v[h], ev[eh]), m
        if ops & _lib.HN_BATCH_ERASE:
            model.erase(ers[m])
        if ops & _lib.HN_BATCH_CLEAN:
            model.clean_tombstones()
        img = bm.buckets(m)
        info = bm.info(m)
        assert np.array_equal(live_pairs(img, key_bits), live_pairs(model.b, key_bits)), m
        assert np.array_equal(occupancy(img, key_bits), occupancy(model.b, key_bits)), m
        assert info.fill == model.info.fill and info.tombstone_counter == model.info.tombstones, m
        assert info.err == 0, m
        assert reachable_all(img, key_bits, int(sp)), m
        mp = getattr(O.lib(), f"or_gpu{key_bits}_max_probe")(np.ascontiguousarray(img.reshape(-1)).ctypes.data,
                                                              int(sp))
        assert info.current_max_bucket_overflow >= max(64, next_overflow(mp)), m


def check_bulk(bm, wl, key_bits, ops=_lib.HN_BATCH_ALL):
    """check_against_oracle with one download of every device array (many maps)."""
    sps, ins, vals, qry, ers = wl
    nd = np.uint32 if key_bits == 32 else np.uint64
    arena = bm.arena.cpu().numpy().view(nd)
    qv = bm.qry_vals.cpu().numpy().view(nd)
    qh = bm.qry_hit.cpu().numpy().astype(bool)
    infos = bm.all_infos()
    mp_fn = getattr(O.lib(), f"or_gpu{key_bits}_max_probe")
    for m, sp in enumerate(sps):
        sp = int(sp)
        model = O.GpuModel(sp, key_bits)
        if ops & _lib.HN_BATCH_INSERT:
            model.insert(ins[m], vals[m])
        if ops & _lib.HN_BATCH_RETRIEVE:
            ev, eh = model.retrieve(qry[m])
            lo, n = int(bm.qry_off[m]), int(bm.qry_len[m])
            h, v = qh[lo:lo + n], qv[lo:lo + n]
            assert np.array_equal(h, eh), m
            assert np.array_equal(v[h], ev[eh]), m
        if ops & _lib.HN_BATCH_ERASE:
            model.erase(ers[m])
        if ops & _lib.HN_BATCH_CLEAN:
            model.clean_tombstones()
        lo = int(bm.slot_off[m])
        img = np.ascontiguousarray(arena[lo:lo + (1 << sp)])
        fill, ovf, tomb = int(infos[m, 1]), int(infos[m, 2]), int(infos[m, 3])
        err = int(infos[m, 4]) & 0xFFFFFFFF
        assert np.array_equal(live_pairs(img, key_bits), live_pairs(model.b, key_bits)), m
        assert np.array_equal(occupancy(img, key_bits), occupancy(model.b, key_bits)), m
        assert fill == model.info.fill and tomb == model.info.tombstones and err == 0, m
        assert reachable_all(img, key_bits, sp), m
        assert ovf >= max(64, next_overflow(mp_fn(img.reshape(-1).ctypes.data, sp))), m


@pytest.mark.parametrize("key_bits", [32, 64])
@pytest.mark.parametrize("width,block", [(8, 512), (4, 256), (16, 1024), (1, 64)])
def test_batch_all_ops_vs_oracle(gpu, key_bits, width, block):
    wl = small_batch(key_bits, seed=width + block)
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    bm.run(_lib.HN_BATCH_ALL, hn_tune(width, block, 0, 0))
    torch.cuda.synchronize()
    check_against_oracle(bm, wl, key_bits)


@pytest.mark.parametrize("key_bits", [32, 64])
def test_batch_phase_by_phase_and_per_map_agree(gpu, key_bits):
    wl = small_batch(key_bits, n_maps=40, seed=3)
    a = BatchedMaps(*wl, key_bits=key_bits)
    a.init()
    for op in (_lib.HN_BATCH_INSERT, _lib.HN_BATCH_RETRIEVE, _lib.HN_BATCH_ERASE, _lib.HN_BATCH_CLEAN):
        a.run(op)
    b = BatchedMaps(*wl, key_bits=key_bits)
    b.init_per_map()
    b.run_per_map(_lib.HN_BATCH_ALL)
    torch.cuda.synchronize()
    check_against_oracle(a, wl, key_bits)
    for m in range(len(wl[0])):
        va, ha = a.results(m)
        vb, hb = b.results(m)
        assert np.array_equal(ha, hb) and np.array_equal(va[ha], vb[hb])
        assert np.array_equal(live_pairs(a.buckets(m), key_bits), live_pairs(b.buckets(m), key_bits))


def test_batch_velocity_grid_workload_small(gpu):
    wl = W.batched_workload(n_maps=64, sp_lo=8, sp_hi=13, seed=11)
    bm = BatchedMaps(*wl, key_bits=32)
    bm.init()
    bm.run()
    torch.cuda.synchronize()
    check_against_oracle(bm, wl, 32)


def test_batch_velocity_grid_workload_full_size(gpu):
    """The full batched workload: 4,096 u32 maps of 2^8..2^16 slots at LF 0.6
    (35.7 M keys), every map's retrieve results, live set, occupancy and Info
    against the oracle's sequential insert -> retrieve -> erase -> clean."""
    wl = W.batched_workload()
    bm = BatchedMaps(*wl, key_bits=32)
    bm.init()
    bm.run()
    torch.cuda.synchronize()
    assert len(wl[0]) == 4096 and sum(len(k) for k in wl[1]) > 35_000_000
    check_bulk(bm, wl, 32)


@pytest.mark.parametrize("key_bits", [32, 64])
def test_batch_skewed_query_units(gpu, key_bits):
    """One map with 2 M queries (489 retrieve units) among 3,000 maps, most
    with no queries at all: every unit is served once, every map's results
    equal the oracle's."""
    rng = np.random.default_rng(17)
    n_maps = 3000
    sps = np.concatenate([[18], rng.integers(2, 9, size=n_maps - 1)])
    ins, vals, qry, ers = [], [], [], []
    for m, sp in enumerate(sps):
        n = int(0.7 * (1 << int(sp)))
        k = W.unique_keys(n, key_bits, 300 + m)
        ins.append(k)
        vals.append(W.values(k, m).astype(k.dtype))
        if m == 0:
            a = W.unique_keys(n, key_bits, 300 + m, start=n + 2)
            q = np.concatenate([np.tile(k, 8), a])[:2_000_000]
            qry.append(rng.permutation(q))
        elif m % 3 == 0:
            qry.append(rng.permutation(np.concatenate([k, W.unique_keys(5, key_bits, 300 + m, start=n + 2)])))
        else:
            qry.append(k[:0])
        ers.append(k[: n // 5])
    wl = (sps, ins, vals, qry, ers)
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    bm.run()
    torch.cuda.synchronize()
    check_bulk(bm, wl, key_bits)


def test_batch_graph_replays_match_eager(gpu):
    wl = small_batch(32, n_maps=48, seed=5)
    bm = BatchedMaps(*wl, key_bits=32)
    bm.init()
    bm.run()
    torch.cuda.synchronize()
    eager_vals, eager_hit = bm.qry_vals.clone(), bm.qry_hit.clone()
    eager_infos = bm.infos.clone()
    eager_live = [live_pairs(bm.buckets(m), 32) for m in range(len(wl[0]))]
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        bm.init(stream=s)  # warm-up on the capture stream
        bm.run(stream=s)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        bm.init()
        bm.run()
    for rep in range(3):
        bm.qry_vals.zero_()
        bm.qry_hit.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(bm.qry_hit, eager_hit), rep
        assert torch.equal(bm.qry_vals[eager_hit.bool()], eager_vals[eager_hit.bool()]), rep
        inf = bm.infos.cpu().numpy()
        ref = eager_infos.cpu().numpy()
        assert np.array_equal(inf[:, 1], ref[:, 1]) and np.array_equal(inf[:, 3], ref[:, 3]), rep
        for m in range(len(wl[0])):
            assert np.array_equal(live_pairs(bm.buckets(m), 32), eager_live[m]), (rep, m)


def test_batch_clean_without_enough_scratch_fails_cleanly(gpu):
    wl = small_batch(32, n_maps=4, seed=9)
    bm = BatchedMaps(*wl, key_bits=32)
    # shrink the first listed map's scratch capacity below its fill
    raw = bm.descs.cpu().numpy().copy()
    rec = raw[:80].view(np.uint64)
    rec[9] = 0  # scratch_cap
    bm.descs.copy_(torch.from_numpy(raw))
    bm.init()
    bm.run(_lib.HN_BATCH_INSERT | _lib.HN_BATCH_ERASE)
    torch.cuda.synchronize()
    m0 = int(bm.order[0])
    assert bm.info(m0).tombstone_counter > 0  # precondition: there is something to clean
    before = bm.buckets(m0).copy()
    bm.run(_lib.HN_BATCH_CLEAN)
    torch.cuda.synchronize()
    assert np.array_equal(bm.buckets(m0), before)
    assert bm.info(m0).err == 1 and bm.info(m0).tombstone_counter > 0
    for m in range(4):
        if m != m0:
            assert bm.info(m).tombstone_counter == 0


def region_batch(key_bits, lf, seed):
    """Maps of one, two and several 64-KiB regions, most keys' homes spread, one map's crowded at region ends."""
    one = 13 if key_bits == 32 else 12  # size power of a one-region map
    sps = [one + 3, one + 2, one + 1, one + 1, one, one - 1, 2, 1, one + 4]
    ins, vals, qry, ers = [], [], [], []
    rng = np.random.default_rng(seed)
    for m, sp in enumerate(sps):
        n = max(1, int(lf * (1 << sp)))
        if m == 3:  # homes near the end of a region and of the table: probes cross both ends
            pool = W.unique_keys(1 << (sp + 3), key_bits, seed * 100 + m)
            h = O.fibhash(pool, np.full(pool.size, sp), key_bits) & ((1 << sp) - 1)
            near = pool[(h & ((1 << one) - 1)) >= (1 << one) - 700]
            k = near[: min(near.size - 64, 2000)]
            a = near[k.size:]
        else:
            if m == 8:
                n = 1 << (sp - 5)  # a few keys in many regions
            k = W.unique_keys(n, key_bits, seed * 100 + m)
            a = W.unique_keys(max(1, n // 2), key_bits, seed * 100 + m, start=n + 2)
        ins.append(k)
        vals.append(W.values(k, m).astype(k.dtype))
        qry.append(rng.permutation(np.concatenate([k, a])))
        ers.append(rng.choice(k, max(1, k.size // 3), replace=False))
    return np.array(sps), ins, vals, qry, ers


@pytest.mark.parametrize("key_bits", [32, 64])
@pytest.mark.parametrize("lf", [0.5, 0.9, 0.97])
def test_batch_regions_vs_oracle(gpu, key_bits, lf):
    wl = region_batch(key_bits, lf, seed=int(lf * 100))
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    bm.run()
    torch.cuda.synchronize()
    check_against_oracle(bm, wl, key_bits)


@pytest.mark.parametrize("key_bits", [32, 64])
def test_batch_regions_with_tombstones_between(gpu, key_bits):
    """Erase, insert everything again over the TOMBSTONEs, retrieve, then clean: region probes over
    tables that are neither empty nor free of TOMBSTONEs, phase by phase."""
    wl = region_batch(key_bits, 0.7, seed=5)
    sps, ins, vals, qry, ers = wl
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    steps = [_lib.HN_BATCH_INSERT, _lib.HN_BATCH_ERASE, _lib.HN_BATCH_INSERT, _lib.HN_BATCH_RETRIEVE,
             _lib.HN_BATCH_ERASE | _lib.HN_BATCH_CLEAN, _lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE]
    for ops in steps:
        bm.run(ops)
    torch.cuda.synchronize()
    for m, sp in enumerate(sps):
        model = O.GpuModel(int(sp), key_bits)
        for ops in steps:
            if ops & _lib.HN_BATCH_INSERT:
                model.insert(ins[m], vals[m])
            if ops & _lib.HN_BATCH_RETRIEVE:
                ev, eh = model.retrieve(qry[m])
            if ops & _lib.HN_BATCH_ERASE:
                model.erase(ers[m])
            if ops & _lib.HN_BATCH_CLEAN:
                model.clean_tombstones()
        v, h = bm.results(m)
        assert np.array_equal(h, eh) and np.array_equal(v[h], ev[eh]), m
        img, info = bm.buckets(m), bm.info(m)
        assert np.array_equal(live_pairs(img, key_bits), live_pairs(model.b, key_bits)), m
        assert info.fill == model.info.fill and info.tombstone_counter == model.info.tombstones, m
        assert reachable_all(img, key_bits, int(sp)), m


def test_batch_regions_full_and_short_scratch(gpu):
    """A map that cannot take all its keys reports FAIL; a clean whose scratch is too small leaves its map."""
    key_bits, sp = 32, 14
    full = W.unique_keys((1 << sp) + 50, key_bits, 1)
    some = W.unique_keys(9000, key_bits, 2)
    wl = ([sp, sp], [full, some], [full, some], [full[:64], some], [full[:1], some[:4000]])
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    bm.run(_lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE)
    torch.cuda.synchronize()
    assert bm.info(0).err == 1 and bm.info(0).fill == 1 << sp
    assert bm.info(1).err == 0 and bm.info(1).fill == 9000
    assert bm.results(1)[1].all()
    bm.descs.view(torch.int64).view(-1, 10)[:, 9] = 100  # scratch_cap
    bm.run(_lib.HN_BATCH_ERASE)
    torch.cuda.synchronize()
    before = bm.buckets(1).copy()
    bm.run(_lib.HN_BATCH_CLEAN)
    torch.cuda.synchronize()
    assert bm.info(1).err == 1 and bm.info(1).tombstone_counter == 4000
    assert np.array_equal(before, bm.buckets(1))


def plant_copies(img, sp, key_bits, per_map, rng):
    """Second copies of live keys behind EMPTY slots, as an insert leaves them in a table that
    reset_to_empty has made holes in; half of them across a region's end where the map has several.
    Returns the number planted."""
    from tests.helpers import EMPTY, TOMB
    n, one = 1 << sp, 13 if key_bits == 32 else 12
    keys = img[:, 0]
    empty = np.flatnonzero(keys == EMPTY[key_bits])
    ends = (np.arange(1, max(1, n >> one)) << one) - 1
    last = np.searchsorted(empty, ends, side="right") - 1  # the last EMPTY slot before each region's end
    at = np.concatenate([last, rng.permutation(empty.size - 2)[:per_map]])
    planted = 0
    for j in at:
        e, e2 = int(empty[j]), int(empty[j + 1])
        if e == 0 or keys[e - 1] >= TOMB[key_bits] or keys[e2] != EMPTY[key_bits]:
            continue
        img[e2] = img[e - 1]
        planted += 1
    return planted


@pytest.mark.parametrize("key_bits", [32, 64])
def test_batch_clean_keeps_one_copy_of_a_key(gpu, key_bits):
    """clean_tombstones lifts out the keys away from home and inserts them again, so of a key
    that stands in the table twice one copy is left, and the fill counts it once."""
    one = 13 if key_bits == 32 else 12
    sps = [one + 2, one + 1, one, 10, 6]
    ins = [W.unique_keys(int(0.6 * (1 << sp)), key_bits, 50 + m) for m, sp in enumerate(sps)]
    ers = [k[: k.size // 3] for k in ins]
    bm = BatchedMaps(sps, ins, ins, [k[:0] for k in ins], ers, key_bits=key_bits)
    bm.init()
    bm.run(_lib.HN_BATCH_INSERT | _lib.HN_BATCH_ERASE)
    torch.cuda.synchronize()
    rng = np.random.default_rng(3)
    infos = bm.infos.cpu().numpy()
    arena = bm.arena.cpu().numpy().view(ins[0].dtype)
    for m, sp in enumerate(sps):
        lo = int(bm.slot_off[m])
        infos[m, 1] += plant_copies(arena[lo:lo + (1 << sp)], sp, key_bits, ins[m].size // 8, rng)
    assert (infos[:, 1] > bm.infos.cpu().numpy()[:, 1]).all()  # there are copies in every map
    bm.arena.copy_(torch.from_numpy(arena.view(np.int32 if key_bits == 32 else np.int64)))
    bm.infos.copy_(torch.from_numpy(infos))
    bm.run(_lib.HN_BATCH_CLEAN)
    torch.cuda.synchronize()
    for m, sp in enumerate(sps):
        left = np.sort(ins[m][ins[m].size // 3:])
        img, info = bm.buckets(m), bm.info(m)
        assert np.array_equal(live_pairs(img, key_bits), np.stack([left, left], axis=1)), m
        assert (info.fill, info.tombstone_counter, info.err) == (left.size, 0, 0), m
        assert reachable_all(img, key_bits, sp), m


def test_batch_more_maps_than_spill_lists(gpu):
    """4,130 maps of two regions whose keys crowd the regions' ends: the last ones have no list for
    the keys that run past an end, and are found among all of the map's."""
    key_bits, sp, n_maps = 64, 13, 4130
    pool = W.unique_keys(1 << 17, key_bits, 8)
    home = O.fibhash(pool, np.full(pool.size, sp), key_bits) & ((1 << sp) - 1)
    pool = pool[(home & 4095) >= 4096 - 350]
    ins = [pool[(37 * m) % 1000:][:900] for m in range(n_maps)]
    none = [pool[:0]] * n_maps
    bm = BatchedMaps([sp] * n_maps, ins, ins, [k[:200] for k in ins], none, key_bits=key_bits)
    bm.init()
    bm.run(_lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE)
    torch.cuda.synchronize()
    infos = bm.infos.cpu().numpy()
    assert (infos[:, 1] == 900).all() and (infos[:, 4] & 0xFFFFFFFF == 0).all()
    assert bool(bm.qry_hit.bool().all())
    for m in [0, 4095, *range(4096, n_maps)]:
        img = bm.buckets(m)
        k = np.sort(ins[m])
        assert np.array_equal(live_pairs(img, key_bits), np.stack([k, k], axis=1)), m
        assert reachable_all(img, key_bits, sp), m


def scratch_words(bm):
    """ticket, retrieve units, regions and maps without regions, as the call's set-up left them."""
    return bm.scratch[:32].cpu().numpy().view(np.uint64)


@pytest.mark.parametrize("key_bits", [32, 64])
# maps, size power below a one-region map's (negative: above), queries each, whether they go by units
@pytest.mark.parametrize("n_maps,below,nq,units", [(1, 0, 1 << 21, True), (8, 1, 1 << 18, True), (1, 0, 4000, False),
                                                   (1, 1, 30_011, True), (3, -3, 1 << 19, True), (1, -9, 70_001, True),
                                                   (300, 2, 20_000, False), (16, -2, 5000, False), (100, 0, 30_011, True)])
def test_batch_long_query_lists(gpu, key_bits, n_maps, below, nq, units):
    """Query lists much longer than the table go over the whole device in units, those of a size
    with it stay with its regions; the results are the oracle's either way, and a call is not much
    slower than the lookups by units alone, which asking for a launch shape gives."""
    from tests.helpers import race
    sp = (13 if key_bits == 32 else 12) - below
    n = int(0.55 * (1 << sp))
    rng = np.random.default_rng(nq)
    ins = [W.unique_keys(n, key_bits, 40 + m) for m in range(n_maps)]
    pool = [np.concatenate([k, W.unique_keys(n, key_bits, 40 + m, start=n + 2)]) for m, k in enumerate(ins)]
    qry = [p[rng.integers(0, p.size, nq - m)] for m, p in enumerate(pool)]
    wl = ([sp] * n_maps, ins, [(k ^ k.dtype.type(0x33)).astype(k.dtype) for k in ins], qry, [k[: n // 7] for k in ins])
    bm = BatchedMaps(*wl, key_bits=key_bits)
    bm.init()
    bm.run(_lib.HN_BATCH_INSERT)
    shape = hn_tune(4, 512, 0, 0)
    default, asked = race(lambda: bm.run(_lib.HN_BATCH_RETRIEVE), lambda: bm.run(_lib.HN_BATCH_RETRIEVE, shape), reps=9)
    assert default <= 1.5 * asked, (default, asked)
    bm.qry_vals.zero_()
    bm.qry_hit.zero_()
    bm.run(_lib.HN_BATCH_RETRIEVE | _lib.HN_BATCH_ERASE)
    torch.cuda.synchronize()
    assert (int(scratch_words(bm)[1]) > 0) == units
    check_bulk(bm, wl, key_bits, _lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE | _lib.HN_BATCH_ERASE)


def test_batch_query_units_beside_regions(gpu):
    """Maps of every way in one call: one region and several, a few queries and a great many, none at
    all, and a map that is not cut into regions."""
    key_bits, rng = 32, np.random.default_rng(12)
    sps = [16, 13, 13, 12, 10, 8, 3, 1, 15, 13]
    nqs = [300_000, 1_000_000, 9000, 0, 200_000, 1, 700, 3, 20_000, 64]
    ins = [W.unique_keys(max(1, int(0.6 * (1 << sp))), key_bits, 70 + m) for m, sp in enumerate(sps)]
    qry = [np.concatenate([k, W.unique_keys(k.size + 8, key_bits, 70 + m, start=k.size + 2)])[rng.integers(0, 2 * k.size + 8, q)]
           for m, (k, q) in enumerate(zip(ins, nqs))]
    wl = (sps, ins, ins, qry, [rng.choice(k, k.size // 4, replace=False) for k in ins])
    bm = BatchedMaps(*wl, key_bits=key_bits)
    for ops in (_lib.HN_BATCH_ALL, _lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE):
        bm.init()
        bm.qry_vals.zero_()
        bm.run(ops)
        torch.cuda.synchronize()
        check_against_oracle(bm, wl, key_bits, ops)


@pytest.mark.parametrize("key_bits", [32, 64])
# maps, size power below a one-region map's, keys of each phase, load factor, the phases
@pytest.mark.parametrize("n_maps,below,k,lf,ops", [
    (1, 0, 16, 0.6, 1), (1, 5, 4, 0.6, 1), (2000, 0, 16, 0.6, 1), (2000, 3, 16, 0.3, 2), (2000, 0, 4, 0.6, 4), (1, 0, 16, 0.6, 15),
    (300, 1, 64, 0.6, 7), (40, 2, 600, 0.5, 7), (64, 1, 2, 0.89, 6), (64, 2, 40, 0.7, 6), (5, 10, 3, 0.5, 15), (30, -1, 100, 0.6, 7)])
def test_batch_few_keys(gpu, key_bits, n_maps, below, k, lf, ops):
    """Lists much shorter than the tables: the oracle's results, and not much slower than one
    workgroup for each map, which asking for a launch shape gives (8 us are two launches)."""
    from tests.helpers import race
    sp = (13 if key_bits == 32 else 12) - below
    n = max(k, int(lf * (1 << sp)))
    base = [W.unique_keys(n, key_bits, 200 + m % 37) for m in range(n_maps)]
    rng = np.random.default_rng(k)
    vals = [(b ^ b.dtype.type(0x51)).astype(b.dtype) for b in base]
    table = BatchedMaps([sp] * n_maps, base, vals, [b[:0] for b in base], [b[:0] for b in base], key_bits=key_bits)
    table.init()
    table.run(_lib.HN_BATCH_INSERT)
    upd = [rng.choice(b, k, replace=False) for b in base]
    qry = [np.concatenate([rng.choice(b, k - k // 3), W.unique_keys(k // 3, key_bits, 200 + m % 37, start=n + 5)])
           for m, b in enumerate(base)]
    ers = [rng.choice(b, k, replace=False) for b in base]
    bm = BatchedMaps([sp] * n_maps, upd, upd, qry, ers, key_bits=key_bits)
    desc = bm.descs.cpu().numpy().view(np.uint64).reshape(n_maps, 10).copy()  # clean: room for the keys already there
    desc[:, 8], desc[:, 9] = bm.slot_off[bm.order], 1 << sp
    bm.clean_scratch = torch.empty_like(bm.arena)
    bm.descs.copy_(torch.from_numpy(desc.view(np.uint8).reshape(-1)))

    def before():
        bm.arena.copy_(table.arena)
        bm.infos.copy_(table.infos)
    shape = hn_tune(4, 512, 0, 0)
    default, asked = race(lambda: bm.run(ops), lambda: bm.run(ops, shape), before, reps=9)
    assert default <= 1.3 * asked + 8, (default, asked)
    before()
    bm.qry_vals.zero_()
    bm.qry_hit.zero_()
    bm.run(ops)
    torch.cuda.synchronize()
    if ops & _lib.HN_BATCH_INSERT:
        for b, v, u in zip(base, vals, upd):
            v[np.isin(b, u)] = b[np.isin(b, u)]
    check_bulk(bm, ([sp] * n_maps, base, vals, qry, ers), key_bits, ops | _lib.HN_BATCH_INSERT)


@pytest.mark.parametrize("key_bits", [32, 64])
@pytest.mark.parametrize("below,k", [(0, 1), (0, 30), (5, 3)])
def test_batch_few_keys_among_tombstones(gpu, key_bits, below, k):
    """A few keys into, of and out of tables whose slots are nearly all TOMBSTONEs, which every probe
    runs through."""
    from tests.helpers import race
    sp, n_maps = (13 if key_bits == 32 else 12) - below, 40
    n = int(0.97 * (1 << sp))
    pool = [W.unique_keys(n + 2 * k, key_bits, 300 + m) for m in range(n_maps)]
    none = [p[:0] for p in pool]
    table = BatchedMaps([sp] * n_maps, [p[:n] for p in pool], [p[:n] for p in pool], none, [p[5:n] for p in pool], key_bits=key_bits)
    table.init()
    table.run(_lib.HN_BATCH_INSERT | _lib.HN_BATCH_ERASE)
    new, qry = [p[n:n + k] for p in pool], [p[n - 3:] for p in pool]
    ers = [np.concatenate([p[:1], p[n:n + k // 2], p[n + k:]]) for p in pool]
    bm = BatchedMaps([sp] * n_maps, new, new, qry, ers, key_bits=key_bits)

    def before():
        bm.arena.copy_(table.arena)
        bm.infos.copy_(table.infos)
    ops = _lib.HN_BATCH_INSERT | _lib.HN_BATCH_RETRIEVE | _lib.HN_BATCH_ERASE
    default, asked = race(lambda: bm.run(ops), lambda: bm.run(ops, hn_tune(4, 512, 0, 0)), before, reps=3)
    assert default <= 1.3 * asked + 8, (default, asked)
    before()
    bm.run(ops)
    torch.cuda.synchronize()
    for m, p in enumerate(pool):
        model = O.GpuModel(sp, key_bits)
        model.insert(p[:n], p[:n])
        model.erase(p[5:n])
        model.insert(new[m], new[m])
        ev, eh = model.retrieve(qry[m])
        model.erase(ers[m])
        v, h = bm.results(m)
        assert np.array_equal(h, eh) and np.array_equal(v[h], ev[eh]), m
        img, info = bm.buckets(m), bm.info(m)
        assert np.array_equal(live_pairs(img, key_bits), live_pairs(model.b, key_bits)), m
        assert np.array_equal(occupancy(img, key_bits), occupancy(model.b, key_bits)), m
        assert (info.fill, info.tombstone_counter, info.err) == (model.info.fill, model.info.tombstones, 0), m
        assert reachable_all(img, key_bits, sp), m
