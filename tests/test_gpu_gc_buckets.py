"""Device GC with many nodes in a bucket: more than a wavefront sorts at once (bit-exact against the oracle),
and more than a bucket holds. There the oracle and the reference stop; the device keeps, in old pointer order,
what fits, takes the others out of their parents and reports it, as the model below does."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_plain import assert_same_pool
from test_oracle_pins import small_cfg
from vkhashdag_amd import workloads as W


def specks(n, res, seed):
    """Boxes of 1 to 3 voxels a side all over the grid: long chains of nodes with one or two children."""
    rng = np.random.default_rng(seed)
    lo = rng.integers(0, res - 4, (n, 3))
    hi = lo + rng.integers(1, 4, (n, 3))
    return W.edits([W.edit(W.AABB_FILL, tuple(map(int, a)), tuple(map(int, b)), colored=False) for a, b in zip(lo, hi)])


def config(res, bits, wbpp, pbpb, crowded=None):
    """bits everywhere, or only at the lowest inner level (crowded: the others' bits)."""
    cfg = small_cfg(res, bits, wbpp, pbpb, 3)
    if crowded is not None:
        b = [crowded] * cfg.node_levels
        b[-2] = bits
        cfg = W.PoolConfig(wbpp, pbpb, b, cfg.color_leaf_level)
    return cfg


def bases(cfg):
    return np.concatenate([[0], np.cumsum([1 << b for b in cfg.bucket_bits])]).astype(np.int64)


def nodes_per_bucket(words, bw, cfg, level):
    wpb, wpp, out = cfg.words_per_bucket, 1 << cfg.word_bits_per_page, []
    for b in range(bases(cfg)[level], bases(cfg)[level + 1]):
        i = n = 0
        while i < bw[b]:
            sz = bin(int(words[b * wpb + i]) & 255).count("1")
            i, n = (i + sz + 1, n + 1) if sz else ((i // wpp + 1) * wpp, n)
        out.append(n)
    return out


def gc_model(words, bw, cfg, roots, filled):
    """(bucket counters, words, roots, filled chain, nodes dropped) that a collection leaves."""
    words, bw = words.copy(), bw.copy()
    L, wpb, wpp, base = cfg.node_levels, cfg.words_per_bucket, 1 << cfg.word_bits_per_page, bases(cfg)
    inside = lambda p, l: base[l] * wpb <= p < base[l + 1] * wpb
    live = [{int(filled[l])} if len(filled) and inside(filled[l], l) else set() for l in range(L)]
    live[0] |= {int(r) for r in roots if inside(r, 0)}
    for l in range(L - 1):
        for p in live[l]:
            k = bin(int(words[p]) & 255).count("1")
            live[l + 1] |= {int(c) for c in words[p + 1: p + 1 + k] if inside(c, l + 1)}
    maps, dropped = [{} for _ in range(L)], 0
    old = words.copy()
    for l in range(L - 1, -1, -1):
        at = np.zeros(base[l + 1] - base[l], np.int64)
        for p in sorted(live[l]):
            if l == L - 1:
                b, node = p // wpb - base[l], old[p: p + 2]
            else:
                bits = [i for i in range(8) if int(old[p]) >> i & 1]
                kids = [maps[l + 1].get(int(c), O.HD_NULL) for c in old[p + 1: p + 1 + len(bits)]]
                left = [(i, c) for i, c in zip(bits, kids) if c != O.HD_NULL]
                if not left:
                    maps[l][p] = O.HD_NULL
                    dropped += 1
                    continue
                k = len(left)
                node = np.array([(int(old[p]) & ~255) | sum(1 << i for i, _ in left)] + [c for _, c in left], np.uint32)
                b = O.olib().hdo_hash_span(node, k + 1) & ((1 << cfg.bucket_bits[l]) - 1)
            n, a = len(node), at[b]
            if a % wpp + n > wpp:
                a = (a // wpp + 1) * wpp
            if a + n > wpb:
                maps[l][p] = O.HD_NULL
                dropped += 1
                continue
            q = (base[l] + b) * wpb
            words[q + at[b]: q + a] = 0
            words[q + a: q + a + n] = node
            at[b] = a + n
            maps[l][p] = int(q + a)
        bw[base[l]: base[l + 1]] = at
    return (bw, words, [maps[0].get(int(r), int(r)) for r in roots],
            [maps[l].get(int(filled[l]), int(filled[l])) for l in range(len(filled))], dropped)


def live_words(words, bw, cfg):
    return np.concatenate([words[b * cfg.words_per_bucket: b * cfg.words_per_bucket + n] for b, n in enumerate(bw)])


@pytest.mark.parametrize("bits,wbpp,pbpb", [(6, 5, 2), (1, 9, 3)])
def test_model_equals_the_oracle_where_nothing_overflows(bits, wbpp, pbpb):
    cfg = config(64, bits, wbpp, pbpb)
    ora = O.OraclePool(cfg)
    ora.edit(specks(60, 64, 3))
    bw, words, roots, filled, dropped = gc_model(ora.read_words(0, cfg.total_words), ora.bucket_words(), cfg, [ora.root],
                                                 ora.filled())
    ora.gc()
    assert dropped == 0 and roots == [ora.root] and np.array_equal(filled, ora.filled())
    assert np.array_equal(bw, ora.bucket_words())
    assert np.array_equal(live_words(words, bw, cfg), ora.live_words()[1])


# nodes in the fullest bucket: more than a wavefront's 1024, in buckets of 4096 and of 16384 words
@pytest.mark.gpu
@pytest.mark.parametrize("res,bits,wbpp,pbpb,crowded,n,nodes", [
    (256, 1, 9, 3, 6, 2400, (1025, 2048)), (256, 0, 9, 5, None, 2400, (2049, 8192)), (256, 1, 9, 5, None, 2900, (1025, 2048)),
    (128, 0, 9, 4, 8, 2200, (1025, 2048)),
    (128, 0, 9, 4, 8, 2400, (2049, 4096))])
def test_gc_of_crowded_buckets(res, bits, wbpp, pbpb, crowded, n, nodes):
    from vkhashdag_amd import capi
    cfg = config(res, bits, wbpp, pbpb, crowded)
    print(f"{res}^3, {1 << bits} buckets of {cfg.words_per_bucket} words", flush=True)
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    e = specks(n, res, 5)
    for part in (e[: n // 2], e[n // 2:]):
        dev.edit(part, capi.MODE_PLAIN)
        ora.edit(part)
        assert ora.overflows() == 0
        assert_same_pool(dev, ora, "edits")
        dev.gc()
        ora.gc()
        assert_same_pool(dev, ora, "gc")
        assert np.array_equal(dev.filled(), ora.filled())
    most = max(nodes_per_bucket(ora.read_words(0, cfg.total_words), ora.bucket_words(), cfg, cfg.node_levels - 2))
    assert nodes[0] <= most <= nodes[1], most


def one_bucket_world(bits, wbpp, pbpb, seed):
    """(cfg, words, bucket counters, roots): a pool of two levels whose upper one is full of different nodes that
    all hash to its bucket 0, spread over all its buckets (as a world's nodes are before their children move)."""
    cfg = W.PoolConfig(wbpp, pbpb, [bits, bits], 0)
    rng = np.random.default_rng(seed)
    wpb, wpp, nb = cfg.words_per_bucket, 1 << wbpp, 1 << bits
    words, bw = np.zeros(cfg.total_words, np.uint32), np.zeros(cfg.total_buckets, np.uint32)
    leaves = nb * wpb + 2 * np.arange(wpb // 2)  # the first leaf bucket, full: packing moves none of them
    words[leaves] = 1 + np.arange(wpb // 2)
    bw[nb] = wpb
    roots, seen = [], set()
    todo = [np.array([1 << (i % 8), p], np.uint32) for i, p in enumerate(leaves)]  # every leaf is some node's
    for b in range(nb):
        while True:
            if todo:
                node = todo.pop()
            else:
                k = int(rng.choice([1, 1, 1, 1, 1, 2, 3, 8]))
                mask = sum(1 << int(i) for i in rng.choice(8, k, replace=False))
                node = np.array([mask, *rng.choice(leaves, k)], np.uint32)
                if O.olib().hdo_hash_span(node, len(node)) & (nb - 1):
                    continue
            if node.tobytes() in seen:
                continue
            at = int(bw[b])
            if at % wpp + len(node) > wpp:
                at = (at // wpp + 1) * wpp
            if at + len(node) > wpb:
                break
            seen.add(node.tobytes())
            words[b * wpb + at: b * wpb + at + len(node)] = node
            bw[b] = at + len(node)
            roots.append(b * wpb + at)
    return cfg, words, bw, roots


# from 16 nodes for a bucket of 8 to more than the wavefront sorts at once for one of 2048
@pytest.mark.gpu
@pytest.mark.parametrize("bits,wbpp,pbpb", [(3, 4, 0), (2, 5, 0), (2, 6, 0), (3, 7, 0), (2, 7, 1), (3, 9, 1), (2, 9, 3)])
def test_gc_of_overfull_buckets_keeps_what_fits_in_pointer_order(bits, wbpp, pbpb):
    from vkhashdag_amd import capi
    cfg, words, bw, roots = one_bucket_world(bits, wbpp, pbpb, 7 + bits)
    print(f"{len(roots)} nodes for a bucket of {cfg.words_per_bucket} words", flush=True)
    want = gc_model(words, bw, cfg, roots, [])
    assert want[4] > len(roots) // 4
    dev = capi.DevicePool(cfg)
    dev.write_live_words(bw, live_words(words, bw, cfg))
    assert list(dev.gc(extra_roots=roots))[1:] == want[2]
    assert np.array_equal(dev.bucket_words(), want[0])
    assert np.array_equal(dev.live_words()[1], live_words(want[1], want[0], cfg))
    assert dev.stats().overflow & 4


def null_children(words, cfg, root):
    """Null pointers under set mask bits below root."""
    level, n = {root} - {O.HD_NULL}, 0
    for l in range(cfg.node_levels - 1):
        kids = [int(c) for p in level for c in words[p + 1: p + 1 + bin(int(words[p]) & 255).count("1")]]
        n += kids.count(O.HD_NULL)
        level = set(kids) - {O.HD_NULL}
    return n


@pytest.mark.gpu
@pytest.mark.parametrize("bits,wbpp,seed", [(3, 6, 3), (5, 6, 8), (4, 6, 2)])
def test_worlds_that_lost_nodes_can_be_traced(bits, wbpp, seed):
    """A terrain that overfills its pool, collected: rays go through what is left of it as the oracle's do through
    the same words."""
    from vkhashdag_amd import capi
    res = 256
    print(f"{1 << bits} buckets of {4 << wbpp} words", flush=True)
    h = W.value_noise_heightmap(res, 3, seed, res // 8, res * 3 // 4)
    cfg = config(res, bits, wbpp, 2)
    dev = capi.DevicePool(cfg, heights=h)
    dev.edit(W.terrain_edit(res, seed=seed, skin=4, colored=False))
    words, filled = dev.full_words(), dev.filled()
    want = gc_model(words, dev.bucket_words(), cfg, [dev.root], filled)
    assert want[4] > 0 and O.HD_NULL not in want[3]
    assert null_children(words, cfg, dev.root) == 0
    for k in range(2):
        dev.gc()
        words = dev.full_words()
        if k == 0:
            assert dev.root == want[2][0]
            assert np.array_equal(dev.bucket_words(), want[0])
            assert np.array_equal(dev.live_words()[1], live_words(want[1], want[0], cfg))
        assert null_children(words, cfg, dev.root) == 0
        rng = np.random.default_rng(seed)
        o = rng.random((5000, 3), np.float32) * 3 - 1
        d = rng.random((5000, 3), np.float32) - o
        hits = dev.traversal(o, d)
        rec = O.march_rays(words, cfg.node_levels, dev.root, o, d)
        assert np.array_equal(hits[:, 3] != 0, rec[:, 3] >> 31 != 0) and hits[:, 3].sum() > 100


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(6))
def test_gc_of_a_filled_chain_without_its_root(seed):
    """A pool that came in with a full root bucket has no filled node of level 0, so nothing holds the chain below
    it: the collection drops those nodes and finds the chain again, as at the start of editing."""
    from vkhashdag_amd import capi
    print(f"seed {seed}", flush=True)
    cfg = W.PoolConfig(5, 0, [0, 1, 3], 0)
    rng = np.random.default_rng(seed)
    words, bw = np.zeros(cfg.total_words, np.uint32), np.zeros(cfg.total_buckets, np.uint32)
    leaves = [(3 + b) * 32 for b in range(8)]
    for p in leaves:
        words[p: p + 2] = rng.integers(1, 1 << 32, 2)
        bw[p // 32] = 2
    for i in range(16):  # 8 nodes in each bucket of level 1, a root above each
        p = 32 + 32 * (i // 8) + 2 * (i % 8)
        words[p: p + 2] = 1 << (i % 8), leaves[int(rng.integers(8))]
        words[2 * i: 2 * i + 2] = 1 << (i % 8), p
    bw[0], bw[1: 3] = 32, 16
    roots = [2 * i for i in rng.permutation(16)]
    dev, ora = capi.DevicePool(cfg), O.OraclePool(cfg)
    dev.write_live_words(bw, live_words(words, bw, cfg))
    dev.edit(W.edit(W.SPHERE_DIG, (1, 1, 1), r2=1))
    assert dev.filled()[0] == O.HD_NULL and O.HD_NULL not in dev.filled()[1:]
    ora.load_state(dev.state())
    for k in range(2):
        roots_d, roots_o = dev.gc(extra_roots=roots), ora.gc(extra_roots=roots)
        assert list(roots_d) == list(roots_o)
        assert np.array_equal(dev.filled(), ora.filled())
        bd, wd = dev.live_words()
        bo, wo = ora.live_words()
        assert np.array_equal(bd, bo) and np.array_equal(wd, wo)
        roots = [int(r) for r in roots_o[1:]]
