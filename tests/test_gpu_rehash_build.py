"""device_rehash into a larger table as one bulk build (hn_rehash_build_*):
the new table's image equals the oracle's fresh insert of the old table's
live pairs followed by its Robin Hood reorder, bit for bit (the reordered
image is a function of the key set), and the Info matches (size power, fill,
overflow, no tombstones, ordered flag, err = SUCCESS).  The map's
device_rehash takes this path when it grows a map of many keys."""
import numpy as np
import pytest
import torch

import oracle as O
from hashinator_amd import Hashmap, to_numpy
from hashinator_amd import _lib
from tests.helpers import EMPTY, NDT, TOMB, fresh_model, keyset, live_pairs, occupancy, reachable_all
from tests.test_gpu_build import concentrated_keys

pytestmark = pytest.mark.gpu

TDT = {32: torch.int32, 64: torch.int64}


def old_map(bits, sp, keys, erase_frac, seed):
    vals = (keys * NDT[bits](7) + NDT[bits](1)).astype(NDT[bits])
    hm = Hashmap(sp, bits, auto_build=0, auto_reorder=0)
    if keys.size:
        hm.insert(keys, vals, targetLF=1.0)
    if erase_frac:
        er = keys[np.random.default_rng(seed).choice(keys.size, int(erase_frac * keys.size), replace=False)]
        hm.erase(er)
    return hm


def rehash_build(bits, hm, new_sp, seed=0):
    """Direct C-ABI call into a table holding garbage; returns (image, info words, rc)."""
    L = _lib.load()
    sfx = "u32" if bits == 32 else "u64"
    old_sp = hm.getSizePower()
    junk = np.random.default_rng(seed).integers(0, 2**62, size=(1 << new_sp) * 2, dtype=np.uint64)
    nb = torch.from_numpy(junk.astype(NDT[bits]).view(np.int32 if bits == 32 else np.int64)).cuda().reshape(-1, 2)
    sb = getattr(L, f"hn_rehash_build_scratch_bytes_{sfx}")(old_sp, new_sp)
    assert sb > 0
    sc = torch.empty(sb, dtype=torch.uint8, device="cuda")
    rc = getattr(L, f"hn_rehash_build_{sfx}")(hm.bucket_ptr(), old_sp, nb.data_ptr(), new_sp, hm.info_ptr(),
                                              sc.data_ptr(), sb, None)
    torch.cuda.synchronize()
    return to_numpy(nb, bits).reshape(-1), hm._info.cpu().numpy(), rc


@pytest.mark.parametrize("bits", [32, 64])
# 2^22 old slots: the first partition pass reads the old table in the 8,192-pair tiles.
@pytest.mark.parametrize("old_sp,new_sp,lf,erase", [(3, 4, 0.75, 0.0), (10, 11, 0.9, 0.25), (12, 14, 0.7, 0.0),
                                                     (14, 15, 0.95, 0.3), (16, 17, 0.85, 0.1), (20, 21, 0.9, 0.25),
                                                     (12, 13, 0.0, 0.0), (22, 23, 0.85, 0.2)])
def test_rehash_build_image_exact(gpu, bits, old_sp, new_sp, lf, erase):
    keys = keyset(int(lf * (1 << old_sp)), bits, seed=old_sp + bits)
    hm = old_map(bits, old_sp, keys, erase, seed=old_sp)
    live = live_pairs(hm.host_buckets(), bits)
    img, inf, rc = rehash_build(bits, hm, new_sp, seed=new_sp)
    assert rc == 0
    m = O.GpuModel(new_sp, bits)
    if live.shape[0]:
        m.insert(live[:, 0].copy(), live[:, 1].copy())
    assert m.reorder() == 1
    assert np.array_equal(img, m.b)
    assert int(inf[0]) == new_sp
    assert int(inf[1]) == live.shape[0] == m.info.fill
    assert int(inf[2]) == m.info.overflow
    assert int(inf[3]) == 0
    assert (int(inf[4]) & 0xFFFFFFFF) == 0  # err = SUCCESS: fill preserved
    assert (int(inf[4]) >> 32) == _lib.HN_INFO_ORDERED


@pytest.mark.parametrize("bits", [32, 64])
def test_rehash_build_overfull_region_falls_back(gpu, bits):
    # 6000 keys homed, at the new size, in one 2048-slot region: over the
    # region capacity, so the new table is filled by the probing insert
    new_sp = 15
    keys = concentrated_keys(bits, new_sp, 6000, 2048, seed=8)
    hm = old_map(bits, 14, keys, 0.0, seed=1)
    live = live_pairs(hm.host_buckets(), bits)
    assert live.shape[0] == keys.size
    img, inf, rc = rehash_build(bits, hm, new_sp, seed=3)
    assert rc == 0
    assert (int(inf[4]) & 0xFFFFFFFF) == 0 and int(inf[1]) == keys.size and int(inf[3]) == 0
    assert (int(inf[4]) >> 32) == 0  # arrival order: not marked ordered
    m = O.GpuModel(new_sp, bits)
    m.insert(live[:, 0].copy(), live[:, 1].copy())
    assert np.array_equal(live_pairs(img, bits), live)
    assert np.array_equal(occupancy(img, bits), occupancy(m.b, bits))
    assert reachable_all(img, bits, new_sp)


@pytest.mark.parametrize("bits", [32, 64])
def test_map_device_rehash_uses_build(gpu, bits):
    sp = 14
    keys = keyset(int(0.85 * (1 << sp)), bits, seed=12)
    vals = (keys ^ NDT[bits](0x55)).astype(NDT[bits])
    hm = Hashmap(sp, bits, build_min_keys=0, auto_build=1.0 / 16)
    hm.insert(keys, vals, targetLF=1.0)
    hm.erase(keys[::5])
    live = live_pairs(hm.host_buckets(), bits)
    hm.device_rehash(sp + 2)
    assert hm.getSizePower() == sp + 2 and hm.ordered()
    m = O.GpuModel(sp + 2, bits)
    m.insert(live[:, 0].copy(), live[:, 1].copy())
    assert m.reorder() == 1
    assert np.array_equal(hm.host_buckets().reshape(-1), m.b)
    i = hm.info()
    assert (i.fill, i.tombstone_counter, i.err) == (live.shape[0], 0, 0)
    _, v, h = hm.retrieve(live[:, 0].copy())
    assert h.cpu().numpy().all() and np.array_equal(to_numpy(v, bits), live[:, 1])
    # a map below the key threshold grows by the probing reinsert (then reordered)
    hm2 = Hashmap(sp, bits)  # build_min_keys = 2^17
    hm2.insert(keys, vals, targetLF=1.0)
    hm2.erase(keys[::5])
    hm2.device_rehash(sp + 2)
    assert np.array_equal(hm2.host_buckets().reshape(-1), m.b)


def test_rehash_build_invalid_args(gpu):
    L = _lib.load()
    for sfx in ("u32", "u64"):
        sb = getattr(L, f"hn_rehash_build_scratch_bytes_{sfx}")
        assert sb(10, 10) == 0 and sb(10, 9) == 0 and sb(0, 4) == 0 and sb(10, 33) == 0
        assert sb(10, 11) > 0 and sb(10, 12) == sb(10, 12)
    hm = Hashmap(10, 64)
    b2 = torch.empty((1 << 11, 2), dtype=torch.int64, device="cuda")
    sb = L.hn_rehash_build_scratch_bytes_u64(10, 11)
    sc = torch.empty(sb, dtype=torch.uint8, device="cuda")
    f = L.hn_rehash_build_u64
    assert f(hm.bucket_ptr(), 10, b2.data_ptr(), 10, hm.info_ptr(), sc.data_ptr(), sb, None) == _lib.HN_EINVAL  # same size
    assert f(hm.bucket_ptr(), 10, b2.data_ptr(), 9, hm.info_ptr(), sc.data_ptr(), sb, None) == _lib.HN_EINVAL  # shrink
    assert f(hm.bucket_ptr(), 10, hm.bucket_ptr(), 11, hm.info_ptr(), sc.data_ptr(), sb, None) == _lib.HN_EINVAL  # overlap
    assert f(hm.bucket_ptr(), 10, b2.data_ptr(), 11, hm.info_ptr(), sc.data_ptr(), sb - 1, None) == _lib.HN_ESCRATCH
    assert f(hm.bucket_ptr(), 10, b2.data_ptr(), 11, None, sc.data_ptr(), sb, None) == _lib.HN_EINVAL
    torch.cuda.synchronize()
    assert hm.getSizePower() == 10 and hm.info().size_power == 10  # nothing ran


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("form", ["soa", "pairs", "index"])
@pytest.mark.parametrize("old_sp,new_sp,n", [(1, 2, 1), (3, 5, 20), (6, 7, 60), (10, 11, 1000), (10, 14, 4096),
                                             (12, 13, 3900), (13, 15, 1), (14, 16, 30000), (17, 19, 200003)])
def test_grow_is_rehash_and_insert(gpu, bits, form, old_sp, new_sp, n):
    """hn_grow_*: the old table's live slots (tombstones among them) and a
    batch of new keys, keys of the table and keys of its own, in one build;
    the image and Info are the oracle's insert of both and reorder."""
    from tests.test_gpu_merge import batch, check_merge
    from tests.test_gpu_build import dev
    from hashinator_amd import _lib, to_numpy
    L, sfx = _lib.load(), f"u{bits}"
    N0, N1 = 1 << old_sp, 1 << new_sp
    old = fresh_model(old_sp, bits)
    ok = keyset(max(1, int(0.6 * N0)), bits, seed=old_sp + bits)
    old.insert(ok, (ok ^ NDT[bits](0x77)).astype(NDT[bits]))
    old.erase(ok[::4])
    img = old.b.reshape(-1, 2)
    live = img[(img[:, 0] != EMPTY[bits]) & (img[:, 0] != TOMB[bits])]
    keys, vals = batch(bits, ok, max(1, int(n / 1.2)), seed=new_sp)
    keys, vals = keys[:n], vals[:n]
    if form == "index":
        vals = np.arange(keys.size).astype(NDT[bits])
    m = fresh_model(new_sp, bits)
    m.insert_pairs(live.reshape(-1).copy())
    assert m.insert(keys, vals) == 0
    assert m.reorder() == 1
    ob = dev(img.copy(), bits)
    inf = torch.from_numpy(np.frombuffer(bytes(old.info), dtype=np.int64).copy()).cuda()
    nb = torch.full((N1, 2), 0x5A5A, dtype=ob.dtype, device="cuda")
    sb = getattr(L, f"hn_grow_scratch_bytes_{sfx}")(old_sp, new_sp, keys.size)
    assert sb > 0
    sc = torch.empty(sb, dtype=torch.uint8, device="cuda")
    tail = (ob.data_ptr(), old_sp, nb.data_ptr(), new_sp, inf.data_ptr(), keys.size, sc.data_ptr(), sb, None)
    if form == "pairs":
        dp = dev(np.stack([keys, vals], axis=1), bits)
        rc = getattr(L, f"hn_grow_pairs_{sfx}")(dp.data_ptr(), *tail)
    else:
        dk, dv = dev(keys, bits), dev(vals, bits)
        rc = getattr(L, f"hn_grow_{sfx}")(dk.data_ptr(), None if form == "index" else dv.data_ptr(), *tail)
    torch.cuda.synchronize()
    assert rc == 0 and int(inf[0]) == new_sp
    check_merge(bits, to_numpy(nb, bits).reshape(-1, 2), inf.cpu().numpy(), m)


@pytest.mark.parametrize("bits", [32, 64])
def test_grow_declines_and_falls_back(gpu, bits):
    """Sizes that do not fit are refused; keys that crowd one region are
    placed by probing, the old table's first: the batch's values win."""
    from tests.test_gpu_build import dev
    from hashinator_amd import _lib, to_numpy
    L, sfx = _lib.load(), f"u{bits}"
    scratch = getattr(L, f"hn_grow_scratch_bytes_{sfx}")
    assert scratch(10, 10, 5) == 0 and scratch(10, 11, 1024) == 0 and scratch(10, 11, 0) == 0 and scratch(10, 33, 5) == 0
    old_sp, new_sp = 12, 14
    cand = keyset(60 * 4096, bits, seed=5)
    home = O.fibhash(cand, new_sp, bits).astype(np.int64) & ((1 << new_sp) - 1)
    crowd = cand[(home >= 2048) & (home < 4096)][:2900]
    ok = crowd[:2000]
    old = fresh_model(old_sp, bits)
    old.insert(ok, ok)
    keys = np.concatenate([crowd[1000:2900], cand[home >= 8192][:3000]])
    vals = (keys ^ NDT[bits](0x11)).astype(NDT[bits])
    m = fresh_model(new_sp, bits)
    m.insert(ok, ok)
    m.insert(keys, vals)
    ob, dk, dv = dev(old.b.reshape(-1, 2).copy(), bits), dev(keys, bits), dev(vals, bits)
    inf = torch.from_numpy(np.frombuffer(bytes(old.info), dtype=np.int64).copy()).cuda()
    nb = torch.empty((1 << new_sp, 2), dtype=ob.dtype, device="cuda")
    sb = scratch(old_sp, new_sp, keys.size)
    sc = torch.empty(sb, dtype=torch.uint8, device="cuda")
    assert getattr(L, f"hn_grow_{sfx}")(dk.data_ptr(), dv.data_ptr(), ob.data_ptr(), old_sp, nb.data_ptr(), new_sp,
                                        inf.data_ptr(), keys.size, sc.data_ptr(), sb, None) == 0
    torch.cuda.synchronize()
    img, after = to_numpy(nb, bits).reshape(-1, 2), inf.cpu().numpy()
    assert np.array_equal(live_pairs(img, bits), live_pairs(m.b, bits)) and reachable_all(img, bits, new_sp)
    assert (int(after[1]), int(after[3]), int(after[4])) == (m.info.fill, 0, 0)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("lf,frac", [(0.9, 1 / 8), (0.9, 1 / 20), (0.8, 1 / 8)])
def test_map_insert_near_full(gpu, bits, lf, frac):
    """Inserts below the merge's share of the table: merged into a map that
    ends at least 87% full, probed otherwise; the bucket array stays."""
    sp = 18
    N = 1 << sp
    n, tot = int(frac * N), int(lf * N)
    keys = keyset(tot, bits, seed=77)
    hm = Hashmap(sp, bits, build_min_keys=1)
    hm.insert(keys[n:], keys[n:], targetLF=1.0)
    at = hm.bucket_ptr()
    again = np.concatenate([keys[:n], keys[n:n + 500]])
    vals = (again + NDT[bits](3)).astype(NDT[bits])
    hm.insert(again, vals, targetLF=1.0)
    assert hm.bucket_ptr() == at and hm.size() == tot and hm.peek_status() == 0
    assert hm.ordered() == (n >= N // 16)
    exp = dict(zip(keys.tolist(), keys.tolist()))
    exp.update(zip(again.tolist(), vals.tolist()))
    rows = live_pairs(hm.host_buckets(), bits)
    assert np.array_equal(rows, np.array(sorted(exp.items()), dtype=NDT[bits]))


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("sp,old,n,grows", [(12, 1500, 1700, True), (12, 3300, 500, False), (12, 2000, 1100, False)])
def test_map_insert_padded_with_empty_keys(gpu, bits, sp, old, n, grows):
    """A batch padded with the EMPTY key: as in the probing insert, the padding
    takes no slot, makes no hole and is not counted, whether the insert grows
    the map, merges into a nearly full one or merges a large batch."""
    keys = keyset(old + n, bits, seed=sp)
    hm = Hashmap(sp, bits, build_min_keys=1)
    hm.insert(keys[:old], keys[:old], targetLF=1.0)
    b = np.full(n + n // 8, EMPTY[bits], dtype=NDT[bits])
    at = np.sort(np.random.default_rng(n).choice(b.size, n, replace=False))
    b[at] = keys[old:]
    hm.insert(b, b, targetLF=0.5 if grows else 1.0)
    assert (hm.getSizePower() > sp) == grows and hm.peek_status() == 0
    img = hm.host_buckets()
    assert hm.size() == keys.size
    assert np.array_equal(live_pairs(img, bits)[:, 0], np.sort(keys))
    assert reachable_all(img, bits, hm.getSizePower())
    _, _, hit = hm.retrieve(keys)
    assert bool(hit.all())


@pytest.mark.parametrize("bits", [32, 64])
def test_map_insert_reads_the_info_once(gpu, bits):
    """An insert of a sixteenth of the slots and more that neither grows the map nor is built
    or merged reads the Info back once at most (not at all where the look at its keys brings it)."""
    sp = 14
    keys = keyset(6000, bits, seed=9)
    hm = Hashmap(sp, bits, build_min_keys=1, auto_build=0)
    hm.insert(keys[:4000], keys[:4000], targetLF=1.0)
    reads, info = [], hm.info
    hm.info = lambda: reads.append(1) or info()
    hm.insert(keys[4000:], keys[4000:], targetLF=1.0)
    assert len(reads) <= 1
    assert hm.size() == 6000 and hm.ordered()
    assert np.array_equal(live_pairs(hm.host_buckets(), bits)[:, 0], np.sort(keys))


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("form", ["soa", "pairs", "index"])
# load before, share of the slots inserted, share of those that is new, merged
@pytest.mark.parametrize("lf,frac,new,merged", [(0.8, 1 / 8, 1.0, True), (0.8, 1 / 8, 0.0, False),
                                                (0.88, 1 / 16, 0.0, False), (0.88, 1 / 16, 0.2, False),
                                                (0.88, 1 / 16, 0.9, True), (0.83, 1 / 12, 0.4, False),
                                                (0.7, 1 / 8, 1.0, False), (0.9, 1 / 20, 1.0, False)])
def test_map_insert_near_full_merges_new_keys(gpu, bits, form, lf, frac, new, merged):
    """A smaller insert is merged where the map ends nearly full of it, not where it updates
    keys that are there (update and new keys alternate in the batch, or stand one part after
    the other); where the reorder follows, the image is the oracle's insert and reorder."""
    sp = 14
    N = 1 << sp
    n, old = int(frac * N), int(lf * N)
    keys = keyset(old + n, bits, seed=31)
    hm = Hashmap(sp, bits, build_min_keys=1)
    hm.insert(keys[:old], keys[:old], targetLF=1.0)
    assert hm.ordered()
    fresh = int(new * n)
    b = np.concatenate([keys[:n - fresh], keys[old:old + fresh]])
    if form != "index":
        b = b[np.random.default_rng(5).permutation(n)]
    vals = np.arange(n).astype(NDT[bits]) if form == "index" else (b ^ NDT[bits](0x55)).astype(NDT[bits])
    m = fresh_model(sp, bits)
    m.insert(keys[:old], keys[:old])
    m.insert(b, vals)
    ran, fn, at = [], hm._fn, hm.bucket_ptr()
    hm._fn = lambda name: ran.append(name) or fn(name)
    if form == "pairs":
        hm.insert(np.stack([b, vals], axis=1), targetLF=1.0)
    elif form == "soa":
        hm.insert(b, vals, targetLF=1.0)
    else:
        hm.insertIndex(b, targetLF=1.0)
    assert any(name.startswith("merge") for name in ran) == merged, ran
    assert hm.bucket_ptr() == at and hm.size() == old + fresh and hm.peek_status() == 0
    assert hm.ordered() == (n >= N // 16)
    img = hm.host_buckets()
    if hm.ordered():
        assert m.reorder() == 1
        occ = occupancy(m.b, bits)
        assert np.array_equal(img[occ], m.b.reshape(-1, 2)[occ]) and np.array_equal(occupancy(img, bits), occ)
    else:
        assert np.array_equal(live_pairs(img, bits), live_pairs(m.b, bits))
