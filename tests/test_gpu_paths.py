"""Edges of the kernels' size and shape rules, bit for bit against the CPU oracle."""
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


@pytest.mark.parametrize("mode", list(PUTS))
@pytest.mark.parametrize("first", [0, 1, 5])
def test_keys_leaving_a_long_leaf_at_every_nibble(gmpt, workloads, oracle, mode, first):
    # a key matched 16 nibbles per word: one key, then keys that differ from it
    # at each nibble (word edges 15, 16, 17, 31, 32, ... among them), its own
    # update, and reads of present, absent and invalid keys
    rng = np.random.default_rng(40 + first)
    base = [int(x) for x in rng.integers(0, 16, 64)]
    hexes = [bytes(base[:first] + base[first:] + [16])]
    one = workloads.batch_from_hex(hexes, [b"first value of the shared leaf"])
    others = []
    for d in range(first, 64):
        k = list(base)
        k[d] = (k[d] + 1 + d % 3) % 16
        others.append(bytes(k + [16]))
    others.append(hexes[0])
    more = workloads.batch_from_hex(others, [b"v%d" % i * (1 + i % 40) for i in range(len(others))])
    t = gmpt.MPT(device=0)
    _put(t, one, mode)
    assert _put(t, more, mode) == _after(oracle, [one, more])
    # a second batch of updates along the same path
    upd = workloads.batch_from_hex(others[::3], [b"w%d" % i * 9 for i in range(len(others[::3]))])
    assert _put(t, upd, mode) == _after(oracle, [one, more, upd])
    assert t.get_values(more)[1] == more.value(1)
    bad = [bytes(base[:20] + [0x10 | base[20]] + base[21:] + [16]), bytes(base[:40] + [16]), bytes(base + [3]),
           bytes(base[:63] + [17, 16]), bytes(base[:15] + [0xF0 | base[15]] + base[16:] + [16])]
    assert t.get_values(workloads.batch_from_hex(bad, [b""] * len(bad))) == [None] * len(bad)
    assert t.get_values(upd) == [upd.value(i) for i in range(upd.n)]


@pytest.mark.parametrize("tries", [1, 3])
@pytest.mark.parametrize("share", [0.5, 0.3, 0.05])
def test_latched_insert_by_the_tries_size(gmpt, workloads, oracle, tries, share):
    # the latched insert runs while the batch has no more keys than the trie
    # (share 0.5: both about equal, the line; below: latched); a batch into
    # empty tries is built by position.  Clustered keys split fresh nodes.
    rng = np.random.default_rng(int(100 * share) + tries)
    keys = []
    for _ in range(250):
        base = rng.integers(0, 256, 32, dtype=np.uint8)
        for _ in range(int(rng.integers(2, 30))):
            k = base.copy()
            k[int(rng.integers(1, 32)):] = rng.integers(0, 256, 1, dtype=np.uint8)
            keys.append(k)
    keys = np.unique(np.array(keys), axis=0)
    keys = keys[rng.permutation(len(keys))]
    cut = int(len(keys) * (1 - share))
    f = gmpt.MPT(device=0, num_tries=tries)
    os_ = [oracle.OracleMPT() for _ in range(tries)]
    for part in (keys[:cut], np.concatenate([keys[cut:], keys[:len(keys) // 20]])):
        flat, lens = workloads.random_values(rng, len(part), 1, 120)
        b = workloads.batch_from_fixed(part, flat, lens)
        b.trie_ids = np.sort(rng.integers(0, tries, len(part))).astype(np.int32)
        _put(f, b, "latching")
        for t in range(tries):
            os_[t].puts(b.subset(np.flatnonzero(b.trie_ids == t)))
            os_[t].hash()
        assert f.get_root_hashes() == [o.root() for o in os_]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,vlen", [(1, 40), (3000, 40), (32768, 40), (32768, 1000)])
def test_root_without_allocation_near_its_region(gmpt, workloads, oracle, mode, n, vlen):
    # the largest batch and, at 1,000-byte values, one whose bound is past the
    # region (the latched insert keeps it)
    rng = np.random.default_rng(n + vlen)
    b = workloads.batch_from_fixed(rng.integers(0, 256, (n, 8), dtype=np.uint8),
                                   rng.integers(0, 256, n * vlen, dtype=np.uint8), np.full(n, vlen))
    assert gmpt.build_root_noalloc(b, mode) == oracle.root_of(b)


@pytest.mark.parametrize("tries,per", [(2, 3000), (3, 4000), (130, 70), (130, 700), (257, 40), (5000, 3)])
@pytest.mark.parametrize("shape", ["uniform", "tied", "one-trie"])
def test_batches_ordered_by_trie_and_path(gmpt, workloads, oracle, tries, per, shape):
    # one sort by the trie id above the window's leading bits: trie counts with
    # 1 to 13 bits, batches of one workgroup and more, tries in random order,
    # keys that tie in the window's kept nibbles, all keys in one trie
    rng = np.random.default_rng(tries + per)
    n = tries * per
    keys = rng.integers(0, 256, (n, 12), dtype=np.uint8)
    if shape == "tied":  # 4 bytes in common after the first, then a long tail in common
        keys[:, 1:5] = 7
        keys[:, 6:9] = rng.integers(0, 2, (n, 3), dtype=np.uint8)
    tid = np.full(n, tries - 1, np.int32) if shape == "one-trie" else rng.integers(0, tries, n).astype(np.int32)
    flat, lens = workloads.random_values(rng, n, 1, 60)
    b = workloads.batch_from_fixed(keys, flat, lens)
    b.trie_ids = tid
    f = gmpt.MPT(device=0, num_tries=tries)
    _put(f, b)
    roots = f.get_root_hashes()
    for t in sorted(set(tid[:: max(1, n // 12)].tolist())):
        assert roots[t] == oracle.root_of(b.subset(np.flatnonzero(tid == t))), t
    assert all(roots[t] == b"" for t in set(range(tries)) - set(tid.tolist()))


COUNTS = ("perms", "enc_bytes", "leaf_perms", "leaf_bytes", "leaf_nodes", "hashed_nodes")


def _mixed_keys(rng, n, kind):
    if kind == "uniform":
        return [bytes(k) for k in rng.integers(0, 256, (n, 32), dtype=np.uint8)]
    if kind == "short":  # keys that are prefixes of others (values in branches), encodings under 32 bytes
        return [bytes(rng.integers(0, 256, int(rng.integers(1, 5)), dtype=np.uint8)) for _ in range(n)]
    # long: remainders past 64 nibbles, extensions of every length
    stems = [bytes(rng.integers(0, 256, int(rng.integers(1, 60)), dtype=np.uint8)) for _ in range(1 + n // 6)]
    return [stems[int(rng.integers(len(stems)))] + bytes(rng.integers(0, 256, int(rng.integers(1, 60)), dtype=np.uint8))
            for _ in range(n)]


@pytest.mark.parametrize("mode", list(PUTS))
@pytest.mark.parametrize("kind,n", [("uniform", 1), ("uniform", 2), ("uniform", 36), ("short", 700), ("long", 700),
                                    ("uniform", 4650), ("uniform", 4850), ("short", 9000), ("long", 6000),
                                    ("uniform", 66_000), ("uniform", 75_000)])
def test_short_dirty_lists_hashed_in_one_climb(gmpt, workloads, oracle, mode, kind, n):
    # list lengths around a block of 64, around the lines to leaves by lane
    # (8,192 entries) and to levels (24,576 inner nodes); empty, 1-byte and many-block
    # values, in leaves and in branches; a second batch hashed over a clean trie;
    # the same root as by levels, and for a build into an empty trie the same
    # work counts (later batches may split a node after listing it, which only
    # the levels hash)
    rng = np.random.default_rng(n + len(kind))
    keys = list(dict.fromkeys(_mixed_keys(rng, n, kind)))
    lens = rng.choice([0, 1, 1, 5, 32, 55, 56, 90, 135, 136, 137, 300, 1000], len(keys))
    lens[:: max(1, n // 3)] = rng.choice([255, 256, 16_382, 16_383, 70_000], len(lens[:: max(1, n // 3)]))
    vals = [bytes(rng.integers(0, 256, int(k), dtype=np.uint8)) for k in lens]
    b = workloads.batch_from_bytes(keys, vals)
    some = rng.permutation(len(keys))[: 1 + n // 8]
    more = workloads.batch_from_bytes([keys[i] for i in some] + [b"\x31" + keys[i][:20] for i in some],
                                      [b"u%d" % i for i in range(2 * len(some))])
    t, by_level = gmpt.MPT(device=0), gmpt.MPT(device=0)
    by_level.set_option("hc_fuse_leaves", 0)
    o = oracle.OracleMPT()
    for part in (b, more):
        nt = getattr(t, PUTS[mode])(part)[1]
        t.hash_onepass_v2(None, nt)
        o.puts(part)
        o.hash()
        assert t.get_root_hash() == o.root()
        st = t.stats()
        if part is b:
            assert (st["hash_launches"] == 1) == (st["hashed_nodes"] - st["leaf_nodes"] <= 24576)
        assert _put(by_level, part, mode) == o.root()
        if part is b:
            assert [t.stats()[k] for k in COUNTS] == [by_level.stats()[k] for k in COUNTS]
    assert _put(t, b, mode) == _after(oracle, [b, more, b])


@pytest.mark.parametrize("modes", [("2phase", "2phase"), ("latching", "latching"), ("2phase", "latching"),
                                   ("latching", "2phase")])
@pytest.mark.parametrize("tries", [1, 7])
def test_dirty_nodes_split_before_they_are_hashed(gmpt, workloads, oracle, modes, tries):
    # two inserts before one hash: the second splits leaves and extensions the
    # first left in the dirty list, at their first nibble and further in
    rng = np.random.default_rng(len(modes[0]) + tries)
    first, second = [], []
    for _ in range(300):
        stem = [int(x) for x in rng.integers(0, 16, int(rng.integers(1, 24)))]
        tail = [int(x) for x in rng.integers(0, 16, 64 - len(stem))]
        first += [bytes(stem + [q] + tail[1:] + [16]) for q in (1, 9)]  # a branch below the stem
        cut = int(rng.integers(0, len(stem)))
        second.append(bytes(stem[:cut] + [(stem[cut] + 1) % 16] + stem[cut + 1:] + tail + [16]))
        second.append(bytes(stem + [1] + tail[1:30] + [(tail[30] + 1) % 16] + tail[31:] + [16]))
    f = gmpt.MPT(device=0, num_tries=tries)
    os_ = [oracle.OracleMPT() for _ in range(tries)]
    for hexes, mode in ((first, modes[0]), (second, modes[1]), (first[::5] + second[::3], modes[0])):
        hexes = list(dict.fromkeys(hexes))
        b = workloads.batch_from_hex(hexes, [b"%d" % i * 9 for i in range(len(hexes))])
        b.trie_ids = np.array([h[0] % tries for h in hexes], np.int32)
        n = getattr(f, PUTS[mode])(b)[1]
        for t in range(tries):
            os_[t].puts(b.subset(np.flatnonzero(b.trie_ids == t)))
    f.hash_onepass_v2(None, n)
    assert f.stats()["hash_launches"] == 1  # no node was left out of the climb
    for o in os_:
        o.hash()
    assert f.get_root_hashes() == [o.root() for o in os_]


@pytest.mark.parametrize("n", [2, 64, 66, 700, 8191, 8192, 8193, 30_000])
@pytest.mark.parametrize("shape", ["digits", "hot", "hot-digits", "field", "ends", "one-key"])
@pytest.mark.parametrize("tries", [1, 200])
def test_sort_by_the_bits_that_vary(gmpt, workloads, oracle, n, shape, tries):
    # one workgroup's capacity (8,192) and the first pass above it; runs up to
    # 64 and longer: decimal digits behind a common prefix, a key repeated in a
    # third of the batch (the last write stands), keys equal but for a few bits
    # at the window's end, all writes to one key
    rng = np.random.default_rng(n + len(shape) + tries)
    if shape in ("digits", "hot-digits"):
        keys = [b"user%019d" % int(x) for x in rng.integers(0, 10 * n, n)]
    elif shape == "field":  # every other byte the same
        k = rng.integers(0, 256, (n, 24), dtype=np.uint8)
        k[:, ::2] = 0x5A
        keys = [bytes(r) for r in k]
    elif shape == "ends":
        keys = [b"\x11" * 6 + int(x).to_bytes(2, "big") + bytes(4) for x in rng.integers(0, min(n, 60_000), n)]
    elif shape == "one-key":
        keys = [b"the only key"] * n
    else:
        keys = [bytes(r) for r in rng.integers(0, 256, (n, 32), dtype=np.uint8)]
    if shape.startswith("hot"):
        for i in rng.choice(n, n // 3, replace=False):
            keys[i] = keys[0]
    b = workloads.batch_from_bytes(keys, [b"%d" % i * (1 + i % 5) for i in range(n)])
    b.trie_ids = np.full(n, tries // 2, np.int32) if tries > 1 and n % 2 else rng.integers(0, tries, n).astype(np.int32)
    f = gmpt.MPT(device=0, num_tries=tries)
    _put(f, b)
    roots = f.get_root_hashes()
    for t in sorted(set(b.trie_ids.tolist()))[:: 1 + tries // 12]:
        assert roots[t] == oracle.root_of(b.subset(np.flatnonzero(b.trie_ids == t))), t
    assert _put(f, b, "latching") == roots[0]


@pytest.mark.parametrize("mode", list(PUTS))
@pytest.mark.parametrize("n", [1, 3900, 4200, 11_000, 22_000, 45_000, 60_000, 90_000])
def test_host_batches_around_the_pinned_packing(gmpt, workloads, oracle, mode, n):
    # host batches whose arrays (8 to 65 bytes a key) pass the 1 MiB packed in
    # pinned memory one after the other, with host pointers and trie ids, and
    # reads whose results (12 bytes a key) fit behind them or do not
    rng = np.random.default_rng(n)
    keys = workloads.unique_random_keys(rng, n, 32)
    flat, lens = workloads.random_values(rng, n, 0, 90)
    b = workloads.batch_from_fixed(keys, flat, lens)
    b.trie_ids = rng.integers(0, 2, n).astype(np.int32)
    hps = rng.integers(1, 1 << 60, n).astype(np.uint64)
    f = gmpt.MPT(device=0, num_tries=2)
    targets, m = getattr(f, PUTS[mode])(b, hps)
    f.hash_onepass_v2(targets, m)
    assert f.get_root_hashes() == [oracle.root_of(b.subset(np.flatnonzero(b.trie_ids == t))) for t in range(2)]
    got, sizes = f.gets_parallel(b)
    assert (got == hps).all() and (sizes == lens).all()
    absent = b.subset(range(n))
    absent.trie_ids = 1 - b.trie_ids
    got, sizes = f.gets_parallel(absent)
    assert (got == 0).all() and (sizes == f.gets_parallel(absent.subset([0]))[1][0]).all()
    assert f.get_values(b.subset(range(0, n, 1 + n // 9)))[0] == b.value(0)


@pytest.mark.parametrize("kind,n", [("uniform", 1), ("uniform", 90), ("short", 800), ("long", 800),
                                    ("uniform", 20_000)])
@pytest.mark.parametrize("tries", [1, 3])
def test_export_of_marked_paths(gmpt, workloads, oracle, kind, n, tries):
    # results of less than one and of several halves of the pinned memory, one
    # value above a half; every key, one, and some with repeats and absent ones;
    # again after the pools (and with them the bitmap) have grown
    rng = np.random.default_rng(n + tries)
    keys = list(dict.fromkeys(_mixed_keys(rng, n, kind)))
    vals = [bytes(rng.integers(0, 256, int(k), dtype=np.uint8)) for k in rng.choice([0, 1, 1, 3, 40, 56, 300], len(keys))]
    vals[0] = bytes(rng.integers(0, 256, 700_000, dtype=np.uint8))
    f = gmpt.MPT(device=0, num_tries=tries)
    os_, kept = [oracle.OracleMPT() for _ in range(tries)], []
    for cut in (slice(0, max(1, n // 3)), slice(0, None)):
        # (new values each time: the oracle exports a leaf that was written again
        # with the value it had as if the value were empty)
        part, pv = keys[cut], [v + b"!" * (1 + len(kept)) for v in vals[cut]]
        b = workloads.batch_from_bytes(part, pv)
        b.trie_ids = np.array([k[0] % tries for k in part], np.int32)
        _put(f, b)
        want = set()
        for t in range(tries):
            kept.append(b.subset(np.flatnonzero(b.trie_ids == t)))  # the oracle refers to the values
            os_[t].puts(kept[-1])
            os_[t].hash()
            want |= {(h + bytes(32 - len(h)), e) for h, e in os_[t].export()}
        every = f.flush_dirty_nodes(b)
        assert set(every) == want
        one = f.flush_dirty_nodes(b.subset([0]))
        order = {x: i for i, x in enumerate(every)}  # references ascend
        assert set(one) <= want and [order[x] for x in one] == sorted(order[x] for x in one)
        some = b.subset([0, len(part) // 2, 0, len(part) - 1])
        some.trie_ids = np.array(some.trie_ids)
        got = f.flush_dirty_nodes(some)
        assert set(one) <= set(got) <= want and len(got) <= len(every)
        gone = workloads.batch_from_bytes([b"\xee" * 40], [b""])
        gone.trie_ids = np.zeros(1, np.int32)
        assert set(f.flush_dirty_nodes(gone)) <= want


@pytest.mark.parametrize("inside", [0, 1, 300, 5000, 32_767 - 54, 32_768 - 54, 40_000])
@pytest.mark.parametrize("tries", [1, 3])
def test_split_extension_around_keys_below_it(gmpt, workloads, oracle, inside, tries):
    # keys that leave an extension midway, ordered before and after its subtree,
    # with new keys and updates below it between them (one group in two runs,
    # far apart), at sizes around those of a block and of the minimum tree's
    # one-workgroup levels
    rng = np.random.default_rng(inside + 7 * tries)
    pre = [int(x) for x in rng.integers(1, 15, 24)]

    def below(n):
        return [bytes(pre + [int(x) for x in k] + [16]) for k in rng.integers(0, 16, (n, 40))]

    old = below(9)
    away = []
    for d in range(24):
        for x in (0, 15):
            away.append(bytes(pre[:d] + [x] + [int(y) for y in rng.integers(0, 16, 63 - d)] + [16]))
    first = workloads.batch_from_hex(old, [b"old%d" % i for i in range(len(old))])
    keys = away + below(inside) + old[:6]
    keys = [keys[i] for i in rng.permutation(len(keys))]
    more = workloads.batch_from_hex(keys, [b"new%d" % i for i in range(len(keys))])
    want = _after(oracle, [first, more])
    t = gmpt.MPT(device=0, num_tries=tries)
    for b in (first, more):
        n = b.n
        b.trie_ids = np.full(n, tries - 1, np.int32) if tries > 1 else None
        _put(t, b)
    assert t.stats()["regroups"] == 1
    assert t.get_root_hash(tries - 1) == want
    assert t.get_values(more)[:50] == [more.value(i) for i in range(50)]


@pytest.mark.parametrize("kind,n,launches", [("uniform", 100_000, 3), ("uniform", 150_000, 3), ("uniform", 154_000, 0),
                                             ("short", 150_000, 3), ("long", 60_000, 3), ("digits", 200_000, 3)])
def test_dirty_lists_hashed_by_rows_then_climb(gmpt, workloads, oracle, kind, n, launches):
    # lists whose many lower inner nodes are hashed a lane each before the
    # climb: leaves of one and of more blocks, embedded children, values in
    # branches, extension chains (decimal keys) and long extensions; around the
    # line to levels (57,344 inner nodes); the same root and work counts as by
    # levels, then a batch over the clean trie
    rng = np.random.default_rng(n)
    if kind == "digits":
        keys = [b"user%019d" % i for i in rng.permutation(2 * n)[:n]]
    else:
        keys = list(dict.fromkeys(_mixed_keys(rng, n, kind)))
    lens = rng.choice([0, 1, 5, 32, 56, 90, 95, 110, 135, 136, 137], len(keys))
    lens[:: n // 5] = 16_383
    vals = [bytes(rng.integers(0, 256, int(k), dtype=np.uint8)) for k in lens]
    b = workloads.batch_from_bytes(keys, vals)
    some = rng.permutation(len(keys))[: n // 3]
    more = workloads.batch_from_bytes([keys[i] for i in some] + [b"\x31" + keys[i][:20] for i in some],
                                      [b"u%d" % i for i in range(2 * len(some))])
    t, by_level = gmpt.MPT(device=0), gmpt.MPT(device=0)
    by_level.set_option("hc_fuse_leaves", 0)
    o = oracle.OracleMPT()
    for part in (b, more):
        o.puts(part)
        o.hash()
        assert _put(t, part) == o.root()
        assert _put(by_level, part) == o.root()
        if part is b:
            st = t.stats()
            assert launches in (0, st["hash_launches"]) and (launches or st["hash_launches"] > 3)
            assert [st[k] for k in COUNTS] == [by_level.stats()[k] for k in COUNTS]


@pytest.mark.parametrize("nibbles", [123, 125, 126, 127, 128, 253])
def test_split_points_near_the_byte_compare_limit(gmpt, workloads, oracle, nibbles):
    # split points are compared four bytes at a time while keys (terminator
    # included) have at most 126 nibbles: branches at every depth up to the last
    # nibble, of an empty trie and then below its leaves, with fan-outs that
    # reach past a block of 16 split points
    rng = np.random.default_rng(nibbles)
    base = [int(x) for x in rng.integers(0, 16, nibbles)]

    def leaving(d, x):
        return bytes(base[:d] + [x] + [int(y) for y in rng.integers(0, 16, nibbles - 1 - d)] + [16])

    def batch(keys, tag):
        keys = [keys[i] for i in rng.permutation(len(keys))]
        return workloads.batch_from_hex(keys, [b"%s%d" % (tag, i) for i in range(len(keys))])

    last = [bytes(base[:-1] + [x, 16]) for x in range(16)]
    every = [leaving(d, (base[d] + 1 + d % 5) % 16) for d in range(nibbles - 1)]
    wide = [leaving(d, x) for d in (0, nibbles // 2, nibbles - 2) for x in range(16) for _ in range(3)]
    first = batch(list(dict.fromkeys(last[:9] + every[::2] + wide[::2])), b"a")
    more = batch(list(dict.fromkeys(last + every + wide)), b"b")
    t = gmpt.MPT(device=0)
    assert _put(t, first) == _after(oracle, [first])
    assert _put(t, more) == _after(oracle, [first, more])
