"""Segmented open-addressing backend (MGBFS_BACKEND_SEGMENTED) against the
oracle: three rolling banks for inverse-closed graphs, full history for
directed ones, u8 and int64 state rows, forced segment spills, colliding
hashes, and the sorted backend's hand-over when a layer exceeds its limits
(cuda/segmented_history.cu and crates/mgbfs-runtime/src/segmented_history.rs
in the reference; fixtures of tests/generic_visited_gpu.py:40-45)."""
import math
import random

import pytest

from multigpubfs_amd import GraphDefinition, NativeEngine, lrx, run_graph
from oracle import oracle as O

pytestmark = pytest.mark.gpu
COLLIDE, TINY, SORTED_CAP = 2, 128, 256
NAME = "SEGMENTED_OPEN_ADDRESSING_THREE_BANK"

FIXTURES = {
    "lx4": GraphDefinition.permutation([[1, 2, 3, 0], [1, 0, 2, 3]], [0, 1, 2, 3]),
    "lx4_repeated_labels": GraphDefinition.permutation([[1, 2, 3, 0], [1, 0, 2, 3]], [0, 0, 1, 2]),
    "matrix_2x1_mod257": GraphDefinition.matrix(2, 1, [([1, 1, 0, 1], 257)], [256, 2]),
    "matrix_wrap_mod0": GraphDefinition.matrix(1, 1, [([2], 0)], [1]),
    "matrix_mixed_moduli": GraphDefinition.matrix(1, 1, [([2], 5), ([3], 7)], [4]),
    "cycle300": GraphDefinition.permutation([list(range(1, 300)) + [0]], list(range(300))),
}


def layers_of(engine):
    rows = [sorted(map(tuple, engine.sample(0, 1 << 30)))]
    while True:
        status = engine.advance()
        if status == 1:
            break
        assert status == 0, (status, engine.fatal)
        rows.append(sorted(map(tuple, engine.sample(0, 1 << 30))))
    return engine.layer_sizes(), rows


def oracle_layers(graph, bound):
    return [sorted(map(tuple, layer)) for layer in O.c_exact_layers(graph.to_dict(), bound)]


@pytest.mark.parametrize("flags", [0, COLLIDE])
@pytest.mark.parametrize("name", list(FIXTURES))
def test_reference_fixtures_layer_sets(name, flags):
    g = FIXTURES[name]
    with NativeEngine(g, backend="segmented", flags=flags) as e:
        assert e.backend_name == NAME
        sizes, rows = layers_of(e)
    want = oracle_layers(g, 1024)
    assert rows == want and sizes == [len(x) for x in want]


def sl2(p):
    return GraphDefinition.matrix(2, 2, [([1, 1, 0, 1], p), ([1, 0, 1, 1], p), ([1, p - 1, 0, 1], p),
                                         ([1, 0, p - 1, 1], p)], [1, 0, 0, 1])


@pytest.mark.parametrize("p", [5, 7, 11, 13])
def test_sl2_three_banks_layer_sets(p):
    g = sl2(p)
    with NativeEngine(g) as e:  # AUTO: inverse-closed int64 states -> segmented
        assert e.backend_name == NAME
        sizes, rows = layers_of(e)
        assert e.info()["history_layers"] == 3
    assert sum(sizes) == p * (p * p - 1)
    assert rows == oracle_layers(g, p * (p * p - 1))


@pytest.mark.parametrize("flags", [0, TINY, TINY | COLLIDE])
def test_lrx9_packed_states_and_segment_spills(flags):
    ref = O.packed_bfs(9, keep_keys=True)
    with NativeEngine(lrx(9), backend="segmented", flags=flags) as e:
        keys = [sorted(e.layer_keys())]
        while e.advance() == 0:
            keys.append(sorted(e.layer_keys()))
        assert e.status == 1
        sizes = e.layer_sizes()
        spills = e.info()["retries"]
    assert sizes == ref["layers"]
    assert keys == [sorted(k) for k in ref["keys"]]
    if flags & TINY:
        assert spills > 0


def test_degree_16_and_wide_labels():
    # Degree 16 leaves no tag nibble for the packed backends; labels >= 16
    # are outside the packed encoding; labels > 255 need int64 rows.
    n, k = 16, 8
    L = [(i + 1) % k if i < k else i for i in range(n)]
    R = [(i - 1) % k if i < k else i for i in range(n)]
    X = [1, 0] + list(range(2, n))
    for start in (list(range(n)), [3 * i + 1 for i in range(n)], [1000 + 7 * i for i in range(n)]):
        g = GraphDefinition.permutation([L, R, X], start)
        with NativeEngine(g) as e:
            assert e.backend_name == NAME
            sizes, rows = layers_of(e)
        want = oracle_layers(g, math.factorial(k))
        assert sum(sizes) == math.factorial(k) and rows == want


@pytest.mark.parametrize("seed", [41, 42])
@pytest.mark.parametrize("flags", [0, TINY])
def test_directed_full_history(seed, flags):
    rng = random.Random(seed)
    n = 8
    gens = []
    for _ in range(rng.randint(2, 3)):
        g = list(range(n))
        rng.shuffle(g)
        gens.append(g)
    graph = GraphDefinition.permutation(gens, list(range(n)))
    assert not graph.inverse_closed()
    ref = O.packed_bfs(n, gens, keep_keys=True)
    with NativeEngine(graph, backend="segmented", flags=flags) as e:
        keys = [sorted(e.layer_keys())]
        while e.advance() == 0:
            keys.append(sorted(e.layer_keys()))
        assert e.info()["history_layers"] == 0
    assert keys == [sorted(k) for k in ref["keys"]]


@pytest.mark.parametrize("n,flags", [(10, SORTED_CAP), (11, SORTED_CAP), (11, SORTED_CAP | TINY)])
def test_sorted_hands_over_to_segmented_at_its_limits(n, flags):
    # The test flag lowers the sorted backend's limit to 2^18 children per
    # layer: the run starts sorted and finishes on the segmented backend
    # from the sorted backend's last two layers.
    ref = O.packed_bfs(n, keep_keys=(n == 10))
    with NativeEngine(lrx(n), backend="sorted", flags=flags) as e:
        assert e.backend_name == "SORTED_THREE_BANK_LDS_UNIQUE"
        names = set()
        keys = [sorted(e.layer_keys())] if n == 10 else None
        while True:
            s = e.advance()
            names.add(e.backend_name)
            if s != 0:
                break
            if keys is not None:
                keys.append(sorted(e.layer_keys()))
        assert s == 1
        sizes = e.layer_sizes()
        info = e.info()
        prev = e.sample(1, 1000)
    assert NAME in names
    assert sizes == ref["layers"] and info["total_states"] == math.factorial(n)
    assert info["backend"] == 3
    if keys is not None:
        assert keys == [sorted(k) for k in ref["keys"]]
        assert sorted(O.pack(r) for r in prev) == sorted(ref["keys"][-2])


def test_resource_stop_keeps_prefix_and_samples():
    with NativeEngine(sl2(11), backend="segmented", capacity=40) as e:
        statuses = []
        while True:
            s = e.advance()
            statuses.append(s)
            if s != 0:
                break
        assert statuses[-1] == 2
        sizes = e.layer_sizes()
        cur = sorted(map(tuple, e.sample(0, 1000)))
    want = oracle_layers(sl2(11), 1320)
    assert sizes == [len(x) for x in want[:len(sizes)]]
    assert cur == want[len(sizes) - 1]


def test_reset_repeats_and_segmented_memory_backend_through_cli(tmp_path):
    with NativeEngine(sl2(13)) as e:
        first, _ = layers_of(e)
        e.reset()
        second, _ = layers_of(e)
    assert first == second
    report = run_graph(sl2(13), tmp_path / "out", device=0, memory_backend="segmented")
    assert report["layer_sizes"] == first and report["backend"] == NAME
    report = run_graph(lrx(8), tmp_path / "out8", device=0, memory_backend="segmented_hash")
    assert report["layer_sizes"] == O.packed_bfs(8)["layers"] and report["backend"] == NAME


# Graphs whose states fit one packed word run in the sorted backend's banks
# (wide keys): few labels over many positions, and modular matrices.
def closed(gens):
    out = list(gens)
    for g in gens:
        q = [0] * len(g)
        for i, v in enumerate(g):
            q[v] = i
        if q not in out:
            out.append(q)
    return out


def random_closed(n, k, seed):
    rng = random.Random(seed)
    gens = []
    for _ in range(k):
        g = list(range(n))
        rng.shuffle(g)
        gens.append(g)
    return closed(gens)


def unitriangular(m):
    x, y = [1, 1, 0, 0, 1, 0, 0, 0, 1], [1, 0, 0, 0, 1, 1, 0, 0, 1]
    xi, yi = [1, m - 1, 0, 0, 1, 0, 0, 0, 1], [1, 0, 0, 0, 1, m - 1, 0, 0, 1]
    return GraphDefinition.matrix(3, 3, [(g, m) for g in (x, y, xi, yi)], [1, 0, 0, 0, 1, 0, 0, 0, 1])


def vectors(p):
    return GraphDefinition.matrix(2, 1, [(g, p) for g in ([1, 1, 0, 1], [1, 0, 1, 1], [1, p - 1, 0, 1], [1, 0, p - 1, 1])],
                                  [1, 0])


WIDE = {
    "sl2_31": lambda: sl2(31),
    "vectors_257": lambda: vectors(257),
    "unitriangular_11": lambda: unitriangular(11),
    "units_4099": lambda: GraphDefinition.matrix(1, 1, [([2], 4099), ([2050], 4099)], [1]),
    "ring18": lambda: GraphDefinition.permutation(O.lrx_generators(18), [0] * 12 + [1] * 6),
    "three_labels17": lambda: GraphDefinition.permutation(O.lrx_generators(17), [-5] * 14 + [70000] * 2 + [9]),
    "random24": lambda: GraphDefinition.permutation(random_closed(24, 2, 3), [0] * 20 + [1] * 4),
    "eight_generators20": lambda: GraphDefinition.permutation(random_closed(20, 4, 5), [2] * 16 + [3] * 3 + [250]),
}


@pytest.mark.parametrize("flags", [0, 8, 1 | 4, 32])
@pytest.mark.parametrize("name", list(WIDE))
def test_wide_keys_layer_sets(name, flags):
    g = WIDE[name]()
    want = oracle_layers(g, 1 << 20)
    with NativeEngine(g, backend="segmented", flags=flags) as e:
        assert e.backend_name == NAME
        if len(want) < 200:
            sizes, rows = layers_of(e)
            assert rows == want
        e.reset()
        assert e.run() == 1
        sizes = e.layer_sizes()
        info = e.info()
        assert sizes == [len(x) for x in want]
        assert sorted(map(tuple, e.sample(0, 1 << 20))) == want[-1]
        assert sorted(map(tuple, e.sample(1, 1 << 20))) == want[-2]
    assert info["backend"] == 3 and info["history_layers"] == 3
    assert info["candidates"] == sum(sizes) * g.generator_count and info["unique_candidates"] == sum(sizes) - 1


@pytest.mark.parametrize("name", ["sl2_101", "ring22"])
def test_wide_keys_hand_over_to_segmented_tables(name):
    # The lowered limit (2^18 children) sends the widest layers on to the
    # segmented tables: int64 rows, and byte rows with their labels.
    g = sl2(101) if name == "sl2_101" else GraphDefinition.permutation(O.lrx_generators(22), [7] * 11 + [200] * 11)
    with NativeEngine(g, backend="segmented") as e:
        assert e.run() == 1
        want, last = e.layer_sizes(), sorted(map(tuple, e.sample(0, 1000)))
    assert sum(want) == (101 * (101 ** 2 - 1) if name == "sl2_101" else math.comb(22, 11))
    with NativeEngine(g, backend="segmented", flags=128) as e:  # the tables alone
        assert e.run() == 1
        assert e.layer_sizes() == want and sorted(map(tuple, e.sample(0, 1000))) == last
    if name == "sl2_101":
        with NativeEngine(g, backend="segmented", flags=SORTED_CAP) as e:
            for _ in range(2):
                assert e.run() == 1 and e.backend_name == NAME
                assert e.layer_sizes() == want and sorted(map(tuple, e.sample(0, 1000))) == last
                assert e.info()["candidates"] == 4 * sum(want)
                e.reset()


@pytest.mark.parametrize("step", [False, True])
def test_wide_keys_out_of_memory_stop_with_their_layers(step):
    # SL(2, Z_431), 80 million states, in 1.2 GB: the packed layers run out of
    # room, and the last two as tables do not fit beside them.
    p, budget = 431, 1184 << 20
    g = sl2(p)
    with NativeEngine(g, backend="segmented") as e:
        assert e.run() == 1
        full = e.layer_sizes()
    assert sum(full) == p * (p * p - 1)
    with NativeEngine(g, backend="segmented", vram_budget=budget) as e:
        for _ in range(2):
            status = 0
            while step and status == 0:
                status = e.advance()
            assert (status if step else e.run()) == 2
            assert e.fatal or not step
            sizes = e.layer_sizes()
            assert 8 < len(sizes) < len(full) and sizes == full[:len(sizes)]
            for which in (0, 1):
                rows = e.sample(which, 1000)
                assert len({tuple(r) for r in rows}) == 1000
                assert all((r[0] * r[3] - r[1] * r[2]) % p == 1 and 0 <= min(r) and max(r) < p for r in rows)
            info = e.info()
            assert info["device_bytes"] <= budget and info["candidates"] == 4 * sum(sizes[:-1])
            e.reset()


@pytest.mark.parametrize("name,bound", [("sl2", 2000), ("ring", 300)])
def test_layer_beyond_the_declared_bound_stops_the_run(name, bound):
    # Layers of up to 7,030 and 829 states, declared to be fewer in all.
    if name == "sl2":
        full = sl2(31)
        g = GraphDefinition({**full.to_dict(), "expected_max_unique_states": bound})
    else:
        full = GraphDefinition.permutation(O.lrx_generators(18), [0] * 12 + [1] * 6)
        g = GraphDefinition.permutation(O.lrx_generators(18), [0] * 12 + [1] * 6, expected_max_unique_states=bound)
    want = [len(x) for x in oracle_layers(full, 1 << 20)]
    assert max(want) > 1.25 * bound
    with NativeEngine(g, backend="segmented") as e:
        for _ in range(2):
            assert e.run() == 2
            sizes = e.layer_sizes()
            assert sizes == want[:len(sizes)] and max(sizes) <= 1.25 * bound and len(sizes) > 3
            e.reset()


@pytest.mark.parametrize("labels", [(7, 200), (-5, 70000)], ids=["bytes", "int64"])
def test_wide_keys_hand_their_labels_over(labels):
    # Sixteen generators over two labels on 24 places (2.7 million states):
    # layers beyond the lowered limit of 2^18 children go on in the tables.
    g = GraphDefinition.permutation(random_closed(24, 8, 9), [labels[0]] * 12 + [labels[1]] * 12)
    seen = {}
    for flags in (0, 128, SORTED_CAP):  # packed, the tables alone, handed over
        with NativeEngine(g, backend="segmented", flags=flags) as e:
            assert e.run() == 1
            info = e.info()
            last = sorted(map(tuple, e.sample(0, 1 << 22)))
            seen[flags] = [e.layer_sizes(), last, info["candidates"]]
            assert sum(e.layer_sizes()) == math.comb(24, 12) and len(last) == e.layer_sizes()[-1]
            e.reset()
            while sum(e.layer_sizes()) < 200_000:  # after the hand-over: the first 16 places of each state
                assert e.advance() == 0
            assert {v for which in (0, 1) for r in e.sample(which, 1000) for v in r} == set(labels)
            seen[flags].append(sorted(e.layer_keys()))
    assert seen[128] == seen[0] == seen[SORTED_CAP]
