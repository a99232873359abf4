"""The framework's work as a user's program has it: cases to be timed.

``listed()`` names the cases, ``draw()`` gives more of the same ranges,
``prepare()`` makes what a program holds before the call, ``run()`` is one pass
through the public entry points, ``work()`` the bytes such a pass cannot do
without.  Every output is bytes or whole numbers (root hashes, sizes, node
encodings), so two correct runs give the same values bit for bit.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np


def _package():
    """The repository's package (its folder's name is no identifier)."""
    if "gmpt_amd" not in sys.modules:
        d = os.path.join(os.getcwd(), "gpu-merkle-patricia-trie_amd")
        spec = importlib.util.spec_from_file_location("gmpt_amd", os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["gmpt_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["gmpt_amd"]


def listed():
    return [
        # The transaction (or receipt) trie of one block: RLP-encoded indexes
        # as keys, encoded transactions as values, host batch, nothing
        # allocated: the smallest call, once per block.
        {"name": "block_200", "kind": "block", "n": 200, "mode": 0, "vlo": 100, "vhi": 600},
        # One trie of the batched workload's median size through the plain
        # calls (insert, hash, root).
        {"name": "trie_256", "kind": "build", "n": 256, "mode": 0, "klen": 32, "vlo": 32, "vhi": 32, "where": "device"},
        # 10,000 32-byte keys, 64-byte values: the small bulk build.
        {"name": "build_10k", "kind": "build", "n": 10_000, "mode": 0, "klen": 32, "vlo": 64, "vhi": 64,
         "where": "device"},
        # A latched bulk build of an odd size (the other insert algorithm).
        {"name": "olc_build_100k", "kind": "build", "n": 100_003, "mode": 1, "klen": 32, "vlo": 70, "vhi": 110,
         "where": "device"},
        # 1,000,000 32-byte keys, account-sized values: the headline workload.
        {"name": "build_1m", "kind": "build", "n": 1_000_000, "mode": 0, "klen": 32, "vlo": 70, "vhi": 110,
         "where": "device"},
        # A trie is loaded and takes a block's worth of new keys: the insert
        # into tries that are not empty.
        {"name": "insert_2k", "kind": "insert", "base": 20_000, "n": 2_000, "mode": 0, "vlo": 70, "vhi": 110},
        # Skewed latched writes over a loaded trie: 'user' + decimal keys,
        # Zipf(0.99) ranks, half overwrites and half inserts, 1,000-byte values.
        {"name": "skew_lock", "kind": "skew", "base": 200_000, "n": 100_000, "mode": 1, "vlen": 1000},
        # A block of account updates on a resident trie, from host memory.
        {"name": "update_2k", "kind": "update", "base": 200_000, "n": 2_000, "mode": 0, "vlo": 70, "vhi": 110},
        # Point reads: 20,000 host keys, a tenth of them absent.
        {"name": "gets_20k", "kind": "gets", "base": 200_000, "n": 20_000},
        # The nodes on 2,000 keys' paths, for a caller that stores them.
        {"name": "export_2k", "kind": "export", "base": 200_000, "n": 2_000},
        # 4,096 tries of uneven size inserted and hashed as one batch.
        {"name": "batched_4096", "kind": "batched", "tries": 4096, "median": 256, "sigma": 2.046, "cap": 200_000},
        # A burst of serving requests, each for a trie of its own.
        {"name": "served_48", "kind": "served", "requests": 48, "median": 2000, "lanes": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "build", "build", "build", "insert", "skew", "update", "gets", "export", "batched",
                       "served"])
    vlo, vhi = rng.choice([(32, 32), (64, 64), (70, 110), (1, 40), (100, 600)])
    mode = rng.choice([0, 0, 1])
    if kind == "block":
        return {"kind": kind, "n": _log(rng, 1, 2000), "mode": mode, "vlo": 100, "vhi": rng.choice([200, 600, 1500])}
    if kind == "build":
        n = _log(rng, 16, 1_000_000)
        return {"kind": kind, "n": n, "mode": mode, "klen": rng.choice([20, 32, 32]), "vlo": vlo,
                "vhi": vhi if n < 400_000 else min(vhi, 110), "where": rng.choice(["device", "device", "host"])}
    base = _log(rng, 2_000, 300_000)
    if kind == "insert":
        return {"kind": kind, "base": base, "n": _log(rng, 1, base), "mode": mode, "vlo": vlo, "vhi": vhi}
    if kind == "skew":
        return {"kind": kind, "base": base, "n": _log(rng, 1_000, 200_000), "mode": rng.choice([0, 1, 1]),
                "vlen": rng.choice([100, 1000])}
    if kind == "update":
        return {"kind": kind, "base": base, "n": _log(rng, 1, min(base, 20_000)), "mode": mode, "vlo": vlo, "vhi": vhi}
    if kind == "gets":
        return {"kind": kind, "base": base, "n": _log(rng, 1, 100_000)}
    if kind == "export":
        return {"kind": kind, "base": base, "n": _log(rng, 1, min(base, 5_000))}
    if kind == "batched":
        return {"kind": kind, "tries": _log(rng, 16, 4096), "median": rng.choice([64, 128, 256]), "sigma": 1.5,
                "cap": 50_000}
    return {"kind": "served", "requests": _log(rng, 2, 48), "median": _log(rng, 100, 2000),
            "lanes": rng.choice([1, 2, 4])}


# --- inputs -------------------------------------------------------------------

def _values(rng, n, lo, hi):
    lens = rng.integers(lo, hi + 1, size=n).astype(np.int64)
    return np.frombuffer(rng.bytes(int(lens.sum())), np.uint8), lens


def _uniform(wl, rng, n, klen, lo, hi):
    """n uniform keys (hashed addresses: repeats do not occur) with random values."""
    keys = np.frombuffer(rng.bytes(n * klen), np.uint8).reshape(n, klen)
    return wl.batch_from_fixed(keys, *_values(rng, n, lo, hi))


def _rlp_index(i):
    if i == 0:
        return b"\x80"
    b = i.to_bytes((i.bit_length() + 7) // 8, "big")
    return b if i < 128 else bytes([0x80 + len(b)]) + b


def _pick(wl, b, klen, idx, rng, lo, hi):
    """A batch writing new values under keys idx of b (equal-length keys)."""
    hexs = b.keys_hexs.reshape(b.n, 2 * klen + 1)[idx]
    flat, lens = _values(rng, len(idx), lo, hi)
    return wl.Batch(np.ascontiguousarray(hexs).reshape(-1), wl._index_pairs(np.full(len(idx), 2 * klen + 1), np.int32),
                    flat, wl._index_pairs(lens, np.int64), len(idx))


def _put(t, batch, mode, hps=None):
    fn = t.puts_latching_with_valuehp_v2 if mode else t.puts_2phase_with_valuehp
    targets, n = fn(batch, hps)
    t.hash_onepass_v2(targets, n)


def _bytes(root):
    return np.frombuffer(root, np.uint8).copy()


def prepare(case, seed):
    pkg = _package()
    wl = pkg.workloads
    rng = np.random.Generator(np.random.PCG64(seed))
    kind = case["kind"]
    s = {"kind": kind, "mode": case.get("mode", 0), "pkg": pkg}
    if kind == "block":
        flat, lens = _values(rng, case["n"], case["vlo"], case["vhi"])
        b = wl.batch_from_bytes([_rlp_index(i) for i in range(case["n"])], [])
        s["batch"] = wl.Batch(b.keys_hexs, b.keys_indexs, flat, wl._index_pairs(lens, np.int64), case["n"])
        return s
    if kind == "build":
        b = _uniform(wl, rng, case["n"], case["klen"], case["vlo"], case["vhi"])
        s["batch"] = pkg.DeviceBatch(b, adopt_values=True) if case["where"] == "device" else b
        s["trie"] = pkg.MPT(device=0)
    elif kind == "insert":
        s["base"] = pkg.DeviceBatch(_uniform(wl, rng, case["base"], 32, case["vlo"], case["vhi"]), adopt_values=True)
        s["batch"] = pkg.DeviceBatch(_uniform(wl, rng, case["n"], 32, case["vlo"], case["vhi"]), adopt_values=True)
        s["trie"] = pkg.MPT(device=0)
    elif kind == "skew":
        base, ops = case["base"], case["n"]
        universe = rng.permutation(base + max(base, ops))
        old, new = universe[:base], universe[base:]
        ids = np.where(rng.random(ops) < 0.5, old[wl.zipf_ranks(rng, len(old), 0.99, ops)],
                       new[wl.zipf_ranks(rng, len(new), 0.99, ops)])
        for name, these in (("base", old), ("batch", ids)):
            b = wl.batch_from_fixed(wl.user_keys(these), *_values(rng, len(these), case["vlen"], case["vlen"]))
            s[name] = pkg.DeviceBatch(b, adopt_values=True)
        s["trie"] = pkg.MPT(device=0)
    elif kind in ("update", "gets", "export"):
        lo, hi = case.get("vlo", 70), case.get("vhi", 110)
        b = _uniform(wl, rng, case["base"], 32, lo, hi)
        s["trie"] = t = pkg.MPT(device=0)
        # the caller's handles of the values (host pointers in go-ethereum)
        _put(t, b, 0, np.arange(1, b.n + 1, dtype=np.uint64) if kind == "gets" else None)
        n = case["n"]
        idx = rng.choice(b.n, n, replace=n > b.n)
        s["batch"] = _pick(wl, b, 32, idx, rng, lo, hi)
        if kind == "gets":
            k = s["batch"].keys_hexs.reshape(n, 65)
            k[: n // 10, 8:64] = rng.integers(0, 16, size=(n // 10, 56), dtype=np.uint8)  # absent keys
    elif kind == "batched":
        z = rng.standard_normal(case["tries"])
        sizes = np.clip(np.round(np.exp(math.log(case["median"]) + case["sigma"] * z)), 1, case["cap"])
        sizes = sizes.astype(np.int64)
        # the same number of keys whatever the seed (a fixed workload in new keys)
        total = _batched_keys(case)
        sizes[int(np.argmax(sizes))] += total - int(sizes.sum()) if total > int(sizes.sum()) else 0
        while int(sizes.sum()) > total:
            k = int(np.argmax(sizes))
            sizes[k] -= min(int(sizes[k]) - 1, int(sizes.sum()) - total)
        b = _uniform(wl, rng, int(sizes.sum()), 32, 32, 32)
        b.trie_ids = np.repeat(np.arange(case["tries"], dtype=np.int32), sizes)
        s["batch"] = pkg.DeviceBatch(b, adopt_values=True)
        s["trie"] = pkg.MPT(device=0, num_tries=case["tries"])
    elif kind == "served":
        r = case["requests"]
        sizes = _request_sizes(case)
        tries = rng.permutation(256)[:r]
        s["trie"] = srv = pkg.Server(device=0, num_tries=256, lanes=case["lanes"], mem_budget=48 << 30)
        for t in tries:  # resident tries, already filled
            srv.submit(int(t), _uniform(wl, rng, 2000, 32, 70, 110))
        srv.drain()
        s["batch"] = [(int(t), _uniform(wl, rng, int(k), 32, 70, 110)) for t, k in zip(tries, sizes)]
    else:
        raise ValueError(kind)
    return s


def _batched_keys(case):
    """Expected number of keys of `tries` clipped lognormal sizes."""
    q = (np.arange(100_000) + 0.5) / 100_000
    z = np.sqrt(2) * _erfinv(2 * q - 1)
    m = np.clip(np.exp(math.log(case["median"]) + case["sigma"] * z), 1, case["cap"]).mean()
    return int(m * case["tries"])


def _erfinv(x):
    # Winitzki's closed form (2008), two digits are enough for a mean size
    a = 0.147
    ln = np.log(1 - x * x)
    t = 2 / (math.pi * a) + ln / 2
    return np.sign(x) * np.sqrt(np.sqrt(t * t - ln / a) - t)


def _request_sizes(case):
    """Lognormal request sizes, the same for every seed (new keys each)."""
    q = (np.arange(case["requests"]) + 0.5) / case["requests"]
    z = np.sqrt(2) * _erfinv(2 * q - 1)
    return np.clip(np.round(np.exp(math.log(case["median"]) + z)), 1, 50_000).astype(np.int64)


# --- one pass -----------------------------------------------------------------

def _export(pkg, t, batch):
    """The nodes as the C-ABI hands them over (hash slots, encodings, index pairs)."""
    L = pkg.gmpt.lib()
    h, e, ix = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    num = ctypes.c_uint64()
    if L.gmpt_export_nodes(t._f, ctypes.byref(pkg.gmpt.host_batch(batch)), ctypes.byref(h), ctypes.byref(e),
                           ctypes.byref(ix), ctypes.byref(num)):
        raise pkg.GmptError(L.gmpt_last_error().decode())
    n = num.value

    def arr(p, ctype, count):
        return np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctype)), shape=(count,))

    idx = arr(ix, ctypes.c_int64, 2 * n)
    # copied into buffers of a fixed size, as a caller that stores them has
    out = [np.zeros(32 * (4 * batch.n + 512), np.uint8), np.zeros(1536 * batch.n + 65536, np.uint8),
           np.zeros(2 * (4 * batch.n + 512), np.int64)]
    for to, got in zip(out, (arr(h, ctypes.c_uint8, 32 * n), arr(e, ctypes.c_uint8, int(idx[-1]) + 1), idx)):
        to[:len(got)] = got
    for p in (h, e, ix):
        L.gmpt_free_host(p)
    return out


def run(s):
    kind, pkg = s["kind"], s["pkg"]
    if kind == "block":
        return _bytes(pkg.build_root_noalloc(s["batch"], s["mode"]))
    t = s["trie"]
    if kind == "build":
        t.clear()
        _put(t, s["batch"], s["mode"])
        return _bytes(t.get_root_hash())
    if kind in ("insert", "skew"):
        t.clear()
        _put(t, s["base"], 0)
        before = t.get_root_hash()
        _put(t, s["batch"], s["mode"])
        return [_bytes(before), _bytes(t.get_root_hash())]
    if kind == "update":
        _put(t, s["batch"], s["mode"])
        return _bytes(t.get_root_hash())
    if kind == "gets":
        hps, sizes = t.gets_parallel(s["batch"])
        return [hps.astype(np.int64), sizes]
    if kind == "export":
        return _export(pkg, t, s["batch"])
    if kind == "batched":
        t.clear()
        _put(t, s["batch"], 0)
        return _bytes(b"".join(t.get_root_hashes()))
    ids = [t.submit(trie, b) for trie, b in s["batch"]]
    return _bytes(b"".join(t.wait(i)[0] for i in ids))


# --- what a pass cannot do without --------------------------------------------

_NODES = 64 + 32 + 0.36 * 128  # a key's leaf and value nodes and its share of the branches


def _in(n, vmean, klen=32):
    """Hex key, key index pair, value, value index pair."""
    return n * (2 * klen + 1 + 8 + vmean + 16)


def work(case):
    kind = case["kind"]
    n = case.get("n", 0)
    v = (case.get("vlo", 70) + case.get("vhi", 110)) / 2
    path = lambda m, base: m * max(1.0, math.log(max(base, 16), 16)) * 128  # noqa: E731
    if kind == "block":
        b = _in(n, v, 2) + n * _NODES
    elif kind == "build":
        b = _in(n, v, case["klen"]) + n * _NODES
    elif kind == "insert":
        b = _in(n + case["base"], v) + (n + case["base"]) * _NODES
    elif kind == "skew":
        b = _in(n + case["base"], case["vlen"], 23) + (n + case["base"]) * _NODES
    elif kind == "update":
        b = _in(n, v) + path(n, case["base"])
    elif kind == "gets":
        b = n * (73 + 12) + path(n, case["base"])
    elif kind == "export":
        b = n * 73 + 2 * path(n, case["base"])
    elif kind == "batched":
        k = _batched_keys(case)
        b = _in(k, 32) + k * _NODES
    else:
        k = int(_request_sizes(case).sum())
        b = _in(k, 90) + path(k, 4000)
    return {"bytes": float(b), "flops": 0.0}


def exact(case, seed):
    """Outputs are bytes and whole numbers: there is no rounding to measure."""
    return None
