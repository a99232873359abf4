"""Sequences of calls on one forest, and the forms a hash pass or sort takes for them, against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PUTS = {"2phase": "puts_2phase_with_valuehp", "latching": "puts_latching_with_valuehp_v2"}


def _put(t, b, mode="2phase"):
    targets, n = getattr(t, PUTS[mode])(b)
    t.hash_onepass_v2(targets, n)
    return t.get_root_hash()


def _after(oracle, batches):
    o = oracle.OracleMPT()
    for b in batches:
        o.puts(b)
        o.hash()
    return o.root()


def _random_batch(workloads, rng, n):
    flat, lens = workloads.random_values(rng, n, 1, 60)
    return workloads.batch_from_fixed(workloads.unique_random_keys(rng, n, 32), flat, lens)


@pytest.mark.parametrize("between", ["gets", "insert", "latching", "values", "export"])
def test_graph_is_captured_again_after_a_buffer_moved(gmpt, workloads, oracle, between):
    # a capture holds the addresses of the workspaces and pools: a larger call
    # between two rebuilds replaces some of them
    rng = np.random.default_rng(len(between))
    small, large = _random_batch(workloads, rng, 2000), _random_batch(workloads, rng, 150_000)
    want = oracle.root_of(small)
    db = gmpt.DeviceBatch(small, adopt_values=True)
    t = gmpt.MPT(device=0)
    assert t.rebuild_graph(db) is False
    assert t.rebuild_graph(db) is True and t.get_root_hash() == want
    if between == "gets":
        assert (t.gets_parallel(large)[1] == t.gets_parallel(large.subset([0]))[1][0]).all()
    elif between == "values":
        assert t.get_values(large.subset(range(60_000)))[:3] == t.get_values(large.subset(range(3)))
    elif between == "export":
        assert len(t.flush_dirty_nodes(large)) > 0
    else:
        _put(t, large, "latching" if between == "latching" else "2phase")
    # (an export of few nodes has workspaces of its own)
    assert t.rebuild_graph(db) is (between == "export") and t.get_root_hash() == want
    for _ in range(2):
        assert t.rebuild_graph(db) is True and t.get_root_hash() == want
    got, sizes = t.gets_parallel(small)
    assert (sizes == np.diff(small.values_indexs.reshape(-1, 2), axis=1).ravel() + 1).all()
    t.close()
    db.free()


def test_refused_batch_leaves_the_dirty_list_as_it_was(gmpt, workloads, oracle):
    # trie 1 holds a branch below slot 0 and a chain of branches below slot 5;
    # the chain waits for its hash.  A batch with a trie id past the last one is
    # refused: two of its keys end in the branch, either side of the key with
    # the bad id in sorted order (id 9 has trie 1's low three bits).
    rng = np.random.default_rng(9)

    def key(*head):
        return bytes(list(head) + [int(x) for x in rng.integers(1, 15, 64 - len(head))] + [16])

    chain = [key(*[5] * d, 6) for d in range(1, 40)] + [key(*[5] * 41)]
    base = workloads.batch_from_hex([key(0, 1), key(0, 2), key(9)] + chain, [b"%d" % i * 30 for i in range(43)])
    deep = workloads.batch_from_hex([chain[-1]], [b"another value of the chain's last key"])
    bad = workloads.batch_from_hex([key(*[0] * 18), key(3), key(0, 3)], [b"x" * 40, b"y" * 40, b"z" * 40])
    f = gmpt.MPT(device=0, num_tries=5)
    for b in (base, deep, bad):
        b.trie_ids = np.full(b.n, 1, np.int32)
    bad.trie_ids[1] = 9
    _put(f, base)
    f.puts_2phase_with_valuehp(deep)
    with pytest.raises(gmpt.GmptError, match="trie id out of range"):
        f.puts_2phase_with_valuehp(bad)
    f.hash_onepass_v2(None, 0)
    assert f.get_root_hash(1) == _after(oracle, [base, deep])
    assert f.stats()["hashed_nodes"] == 41  # the last key's leaf and the branches at depths 0 .. 39 above it
    bad.trie_ids[1] = 2
    _put(f, bad)
    assert f.get_root_hash(1) == _after(oracle, [base, deep, bad.subset([0, 2])])


@pytest.mark.parametrize("n,tries", [(3000, 1), (3000, 300), (80_000, 1)])
def test_nodes_a_climb_leaves_out_are_hashed_by_levels(gmpt, workloads, oracle, n, tries):
    # every key gets the value it has, and one branch is taken out of the dirty
    # list: its parent then waits for it in vain, the climb (alone, and after
    # row launches) ends without the branches above, and the levels take over
    rng = np.random.default_rng(n + tries)
    b = _random_batch(workloads, rng, n)
    b.trie_ids = np.zeros(n, np.int32)
    b.trie_ids[::3] = tries - 1
    want = [oracle.root_of(b.subset(np.flatnonzero(b.trie_ids == t))) for t in sorted({0, tries - 1})]
    f = gmpt.MPT(device=0, num_tries=tries)
    _put(f, b)
    assert f.stats()["hash_launches"] in (1, 3)
    targets, m = f.puts_2phase_with_valuehp(b)
    listed = np.zeros(m, np.uint32)
    L = gmpt.gmpt.lib()
    assert L.gmpt_memcpy_dtoh(listed.ctypes.data, targets, listed.nbytes) == 0
    branches = np.flatnonzero(listed >> 30 == 1)
    at = int(branches[np.argmax(listed[branches])])  # (the roots come first)
    assert L.gmpt_memcpy_htod(targets + 4 * at, np.zeros(1, np.uint32).ctypes.data, 4) == 0
    f.hash_onepass_v2(targets, m)
    st = f.stats()
    assert st["hash_launches"] > 3 and st["hashed_nodes"] == np.count_nonzero(listed) - 1
    assert [f.get_root_hash(t) for t in sorted({0, tries - 1})] == want
    assert f.puts_2phase_with_valuehp(b.subset([]))[1] == 0  # the dirty list is empty


def _huge_values_in_branches(workloads, rng):
    # stems that end at a branch with a value of 512 MiB (one buffer for all),
    # above a branch of two leaves: the levels' messages exceed any device
    stems = list({bytes(s) for s in rng.integers(0, 16, (640, 8), dtype=np.uint8)})
    keys = [s + bytes([1, c, 7, 16]) for s in stems for c in (2, 3)] + [s + b"\x10" for s in stems]
    b = workloads.batch_from_hex(keys, [b""] * len(keys))
    big = 512 << 20
    b.values_bytes = np.zeros(big, np.uint8)
    b.values_indexs = np.array([(0, 39)] * (2 * len(stems)) + [(0, big - 1)] * len(stems), np.int64).ravel()
    return b


def test_failed_allocation_is_reported_once(gmpt, workloads, oracle):
    rng = np.random.default_rng(511)
    db = gmpt.DeviceBatch(_huge_values_in_branches(workloads, rng), adopt_values=True)
    f = gmpt.MPT(device=0)
    f.set_option("hc_fuse_inner", 0)  # by levels
    targets, m = f.puts_2phase_with_valuehp(db)
    with pytest.raises(gmpt.GmptError, match="workspace allocation failed"):
        f.hash_onepass_v2(targets, m)
    f.clear()
    few = _random_batch(workloads, rng, 500)
    assert _put(f, few) == oracle.root_of(few)
    f.close()
    db.free()


def test_a_hash_pass_that_fails_keeps_its_dirty_list(gmpt, workloads):
    # the leaves are taken out of the dirty list: the climb reaches no branch,
    # and the levels ask for more message memory than the device has
    rng = np.random.default_rng(512)
    b = _huge_values_in_branches(workloads, rng)
    one = workloads.batch_from_hex([b.key(0)], [b"another value of one key, after which no new leaf is recorded"])
    db = gmpt.DeviceBatch(b, adopt_values=True)
    f = gmpt.MPT(device=0)
    f.puts_2phase_with_valuehp(db)
    targets, m = f.puts_2phase_with_valuehp(one)
    listed = np.zeros(m, np.uint32)
    L = gmpt.gmpt.lib()
    assert L.gmpt_memcpy_dtoh(listed.ctypes.data, targets, listed.nbytes) == 0
    listed[listed >> 30 != 1] = 0
    assert L.gmpt_memcpy_htod(targets, listed.ctypes.data, listed.nbytes) == 0
    for _ in range(2):
        with pytest.raises(gmpt.GmptError, match="workspace allocation failed"):
            f.hash_onepass_v2(targets, m)
        assert f.puts_2phase_with_valuehp(one.subset([]))[1] == m  # nothing was hashed, all is still listed
        assert f.get_root_hash() == b""
    f.close()
    db.free()


def test_stats_of_a_replay_hold_no_other_pass(gmpt, workloads):
    # a replay records no times; those of the eager pass before it were not read.
    # Its node counts are the captured pass's
    rng = np.random.default_rng(77)
    db = gmpt.DeviceBatch(_random_batch(workloads, rng, 3000), adopt_values=True)
    t = gmpt.MPT(device=0)
    for replayed in (False, True):
        assert t.rebuild_graph(db) is replayed
        st = t.stats()
        assert st["last_hash_ms"] == st["leaf_perm_ms"] == 0 and st["leaf_nodes"] == 3000
    _put(t, _random_batch(workloads, rng, 5000))
    assert t.rebuild_graph(db) is False  # the insert moved buffers
    assert t.stats()["last_hash_ms"] == 0
    _put(t, _random_batch(workloads, rng, 50))
    assert t.rebuild_graph(db) is True
    again = t.stats()
    keys = ("last_hash_ms", "leaf_perm_ms", "hash_launches", "hashed_nodes", "leaf_nodes", "ext_direct_nodes", "perms")
    assert [again[k] for k in keys] == [st[k] for k in keys]
    t.close()
    db.free()


@pytest.mark.parametrize("mode", [0, 1])
def test_autotune_keeps_what_its_sample_cannot_tell_apart(gmpt, workloads, mode):
    # no inner level of 200 uniform keys passes 256 nodes: every threshold from
    # there on launches the same kernels, and 0 (a state per lane) is the slower
    sample = _random_batch(workloads, np.random.default_rng(200), 200)
    t = gmpt.MPT(device=0)
    for value in (None, 256, 5000, 1 << 30):
        if value is None:
            value = t.get_option("hc_spread_max")
        else:
            t.set_option("hc_spread_max", value)
        assert t.autotune(sample, mode)[0] == value == t.get_option("hc_spread_max")
    t.close()


@pytest.mark.parametrize("tries,n", [(7, 5000), (7, 30_000), (200, 5000), (200, 30_000), (3000, 30_000)])
@pytest.mark.parametrize("shape,fallbacks", [("digits", 0), ("short", 0), ("wide", 0), ("long", 1), ("past", 0), ("past-long", 1)])
def test_keys_of_a_trie_that_tie_beside_the_trie_id(gmpt, workloads, oracle, tries, n, shape, fallbacks):
    # A multi-trie batch's first sort sees the trie id and the leading bits of
    # the 16-nibble window (15, 14 or 13 nibbles for 7, 200 and 3,000 tries), in
    # one workgroup, by buckets and by leading bits.  Keys of one trie that
    # differ only in the window's last nibble or further on, in runs of a few
    # and of hundreds, with repeated keys and keys that end in the run; only
    # long runs whose keys agree in the whole window (all that differ in its last
    # nibble alone do) take the sort by whole keys
    rng = np.random.default_rng(tries + n + len(shape))
    per = 6 if shape in ("digits", "short", "past") else 200
    groups = n // per
    keys, tid = [], []
    for g in range(groups):
        t = int(rng.integers(tries)) if per == 6 else g % 3
        if shape == "digits":  # eight digits that vary
            stem = b"user%018d" % int(rng.integers(10**7))
            some = [stem + b"%d" % c for c in rng.integers(0, 10, per)]
        elif shape == "wide":  # each another value of the window's last two nibbles
            stem = [1] * 10 + [int(x) for x in rng.integers(0, 16, 12)] + [3, 4]
            some = [bytes(stem + [int(x) // 16, int(x) % 16, 9, 16]) for x in rng.permutation(256)[:per]]
        else:
            stem = [1] * 10 + [int(x) for x in rng.integers(0, 16, 12)] + [3, 4, 5]
            more = 1 if shape in ("short", "long") else 9  # 15 or more nibbles of the window in common
            stem = stem + [2] * (more - 1)
            some = [bytes(stem + [int(x) for x in rng.integers(0, 16, int(rng.integers(3, 20)))] + [16]) for _ in range(per)]
            if shape.startswith("past"):
                some[0] = bytes(stem + [16])
        keys += some
        tid += [t] * per
    order = rng.permutation(len(keys))
    vals = [b"%d" % i * (1 + i % 5) for i in range(len(keys))]
    keys = [keys[i] for i in order]
    b = (workloads.batch_from_bytes if shape == "digits" else workloads.batch_from_hex)(keys, vals)
    b.trie_ids = np.array(tid, np.int32)[order]
    f = gmpt.MPT(device=0, num_tries=tries)
    _put(f, b)
    roots = f.get_root_hashes()
    assert f.stats()["fallback_sorts"] == fallbacks
    for t in sorted(set(tid))[:: 1 + len(set(tid)) // 12]:
        assert roots[t] == oracle.root_of(b.subset(np.flatnonzero(b.trie_ids == t))), t
    again = b.subset(range(0, b.n, 2))  # over the loaded tries, from position order and latched
    assert _put(f, again, "latching") == _put(f, again)
    db = gmpt.DeviceBatch(b, adopt_values=True)
    assert f.rebuild_graph(db) is False and f.get_root_hashes() == roots
    # (a capture holds the first sort only; seven tries' 15 nibbles leave runs of 16)
    assert f.rebuild_graph(db) is (per == 6 or (shape == "wide" and tries == 7)) and f.get_root_hashes() == roots
    f.close()
    db.free()


@pytest.mark.parametrize("mode", list(PUTS))
@pytest.mark.parametrize("n_long,n,klen", [(6990, 7200, 36), (7010, 7200, 36), (7010, 12_000, 126), (6990, 30_000, 60),
                                           (7300, 30_000, 126), (45_000, 45_000, 40)])
def test_long_leaves_around_the_line_to_lanes(gmpt, workloads, oracle, mode, n_long, n, klen):
    # leaves the word builder does not take (remainders past 64 nibbles up to the
    # longest key, odd and even): left to the climb up to 7,000 of them, one per
    # lane above, in lists with row launches and without; values of no byte, one
    # (raw and not), and around the ends of one to three blocks, at odd addresses
    rng = np.random.default_rng(n_long + n)
    keys = rng.integers(0, 256, (n, 32), dtype=np.uint8)
    hexes = [b"".join(bytes((x >> 4, x & 15)) for x in k.tobytes()) for k in keys]
    tails = rng.integers(0, 16, (n_long, 2 * klen - 64), dtype=np.uint8)
    hexes = [h + (tails[i].tobytes()[i % 2 and 1:] if i < n_long else b"") + b"\x10" for i, h in enumerate(hexes)]
    lens = rng.choice([0, 1, 1, 2, 31, 55, 56, 70, 90, 100, 135, 136, 137, 200, 272, 273, 400], n)
    b = workloads.batch_from_hex(hexes, [bytes(rng.integers(0, 256, int(k), dtype=np.uint8)) for k in lens])
    t, by_level = gmpt.MPT(device=0), gmpt.MPT(device=0)
    by_level.set_option("hc_fuse_leaves", 0)
    for part in (b, b.subset(range(0, n, 1 if n < 20_000 else 2))):  # new, then over the clean trie
        assert _put(t, part, mode) == oracle.root_of(b) == _put(by_level, part, mode)
        assert t.stats()["hash_launches"] in (1, 3)
        for k in ("perms", "enc_bytes", "leaf_perms", "leaf_bytes", "leaf_nodes", "hashed_nodes"):
            assert t.stats()[k] == by_level.stats()[k], k


def test_long_values_around_the_line_to_lanes(gmpt, workloads, oracle):
    # values past 16 KB, some of them at addresses that are no multiple of 8, of
    # every remainder by a block: from an adopted buffer whose pairs overlap (the
    # host does not expect so many), then from one that holds each
    rng = np.random.default_rng(16)
    n = 7100
    b = _random_batch(workloads, rng, n)
    lens = 16_383 + np.arange(n) % 200
    at = rng.integers(0, 1 << 20, n)
    b.values_bytes = rng.integers(0, 256, (1 << 20) + 20_000, dtype=np.uint8)
    b.values_indexs = np.stack([at, at + lens - 1], 1).astype(np.int64).ravel()
    b.values_indexs[-2:] = len(b.values_bytes) - 16_400, len(b.values_bytes) - 1
    want = oracle.root_of(b)
    db = gmpt.DeviceBatch(b, adopt_values=True)
    db.struct.values_bytes_total = len(b.values_bytes)
    t = gmpt.MPT(device=0)
    assert _put(t, db) == want
    t.clear()
    flat = workloads.batch_from_hex([b.key(i) for i in range(n)], [b.value(i) for i in range(n)])
    assert _put(t, flat) == want and t.stats()["leaf_nodes"] == n
    t.close()
    db.free()


@pytest.mark.parametrize("seed", [61, 62, 63])
def test_latched_inserts_into_larger_tries_split_fresh_nodes(gmpt, workloads, oracle, seed):
    # clusters of keys that share prefixes of random lengths; half of them are in
    # the trie, so the rest is latched, and lanes of a wave split the same fresh
    # short nodes at many depths; keys that end inside others among them
    rng = np.random.default_rng(seed)
    keys = {}
    for _ in range(500):
        base = rng.integers(0, 16, 64)
        for _ in range(int(rng.integers(2, 30))):
            k = base.copy()
            cut = int(rng.integers(1, 64))
            k[cut:] = rng.integers(0, 16, 64 - cut)
            keys[bytes(int(x) for x in k[:int(rng.integers(40, 65))]) + b"\x10"] = None
    keys = list(keys)
    keys = [keys[i] for i in rng.permutation(len(keys))]
    cuts = [0, len(keys) // 2, 3 * len(keys) // 4, len(keys)]
    t, o = gmpt.MPT(device=0), oracle.OracleMPT()
    for k, (lo, hi) in enumerate(zip(cuts, cuts[1:])):
        part = keys[lo:hi] + keys[:lo // 5]
        b = workloads.batch_from_hex(part, [bytes(rng.integers(0, 256, int(rng.integers(0, 90)), dtype=np.uint8)) for _ in part])
        before = t.stats()["pool_bytes_used"]
        _put(t, b, "latching")
        o.puts(b)
        o.hash()
        assert t.get_root_hash() == o.root()
        # a latched key takes one branch, two short nodes and one value (288 bytes), used or not
        if k:
            assert t.stats()["pool_bytes_used"] - before >= 288 * (hi - lo)
    assert t.get_values(b) == o.gets(b)


@pytest.mark.parametrize("spread_max", [0, 8192, 1 << 30])
@pytest.mark.parametrize("fuse_leaves", [0, 1])
@pytest.mark.parametrize("case", ["plain", "block-edge", "tiny-values", "long-keys", "short-keys", "mixed"])
def test_short_lists_by_levels(gmpt, workloads, oracle, spread_max, fuse_leaves, case):
    # "hc_fuse_inner" 0 keeps a short list out of the climb: its levels by the
    # spread and the lane kernels, leaves fused and not
    rng = np.random.default_rng(len(case) + fuse_leaves)
    n, klen, vlo, vhi = {"plain": (5000, 32, 70, 110), "block-edge": (129, 32, 70, 110), "tiny-values": (3000, 32, 0, 2),
                         "long-keys": (2000, 44, 10, 60), "short-keys": (2500, 2, 0, 40), "mixed": (8000, 32, 20, 600)}[case]
    flat, lens = workloads.random_values(rng, n, vlo, vhi)
    b = workloads.batch_from_fixed(workloads.unique_random_keys(rng, n, klen), flat, lens)
    t, climb = gmpt.MPT(device=0), gmpt.MPT(device=0)
    t.set_option("hc_spread_max", spread_max)
    t.set_option("hc_fuse_leaves", fuse_leaves)
    t.set_option("hc_fuse_inner", 0)
    want = oracle.root_of(b)
    for part in (b, b.subset(range(0, n, 3))):
        assert _put(t, part) == want == _put(climb, part)
        assert climb.stats()["hash_launches"] == 1 < t.stats()["hash_launches"]
        for k in ("perms", "enc_bytes", "leaf_perms", "leaf_bytes", "leaf_nodes", "hashed_nodes"):
            assert t.stats()[k] == climb.stats()[k], k


@pytest.mark.parametrize("mode", list(PUTS))
def test_levels_beside_a_clean_long_leaf(gmpt, workloads, oracle, mode):
    # by levels, the deepest small ones on the second stream: a new key beside a
    # clean leaf that the leaf word builder does not take
    rng = np.random.default_rng(81)

    def key(*head):
        return bytes(head) + bytes(rng.integers(0, 256, 32 - len(head), dtype=np.uint8))

    keys = [key(0, 0), key(0, 1)] + [key(int(x)) for x in rng.integers(16, 256, 40)]
    first = workloads.batch_from_bytes(keys, [b"long" * 5000] + [b"w%d" % i for i in range(len(keys) - 1)])
    second = workloads.batch_from_bytes([key(0, 2)], [b"v3"])
    t = gmpt.MPT(device=0)
    t.set_option("hc_fuse_inner", 0)
    assert _put(t, first, mode) == oracle.root_of(first)
    assert _put(t, second, mode) == oracle.root_of(workloads.concat_batches([first, second]))
    assert t.stats()["hash_launches"] > 1


def test_leaves_by_wave_and_by_lane_around_their_line(gmpt, workloads, oracle):
    # dirty lists either side of 16,384 entries
    rng = np.random.default_rng(16384)
    listed = []
    for n in (9200, 9350, 9500, 9650, 9800, 12_000):
        b = _random_batch(workloads, rng, n)
        t = gmpt.MPT(device=0)
        targets, m = t.puts_2phase_with_valuehp(b)
        t.hash_onepass_v2(targets, m)
        assert t.get_root_hash() == oracle.root_of(b) and t.stats()["hash_launches"] == 1
        listed.append(m)
    assert listed[0] <= 16_384 < listed[-1]
