"""Batched multi-instance engine: every instance's layer table must equal the
oracle's (committed golden tables) and the one-at-a-time engine's."""
import json
import math
import random
from pathlib import Path

import pytest

from multigpubfs_amd import GraphDefinition, NativeEngine
from multigpubfs_amd._native import BatchEngine
from multigpubfs_amd.sweep import make_sweep, run_batched, run_sequential
from oracle import oracle as O

pytestmark = pytest.mark.gpu
GOLDEN = json.loads((Path(__file__).parent / "golden" / "sweep256.json").read_text())["instances"]


def test_golden_fixture_matches_generator():
    assert [x["graph"] for x in GOLDEN] == make_sweep(256)


def test_full_sweep_batched_matches_golden_tables():
    tables, seconds, _ = run_batched([x["graph"] for x in GOLDEN])
    assert tables == [x["layer_sizes"] for x in GOLDEN]


@pytest.mark.parametrize("visited", ["bitmap", "hash"])
def test_forced_visited_backends_agree(visited):
    subset = GOLDEN[:24]
    tables, _, _ = run_batched([x["graph"] for x in subset], visited=visited)
    assert tables == [x["layer_sizes"] for x in subset]


def test_sequential_plain_engine_matches_batched():
    subset = GOLDEN[:16]
    seq, _ = run_sequential([x["graph"] for x in subset])
    assert seq == [x["layer_sizes"] for x in subset]


def sl2(p):
    gens = [([1, 1, 0, 1], p), ([1, 0, 1, 1], p), ([1, p - 1, 0, 1], p), ([1, 0, p - 1, 1], p)]
    return GraphDefinition.matrix(2, 2, gens, [1, 0, 0, 1], expected_max_unique_states=p * (p * p - 1))


def test_matrix_instances_in_batch_match_oracle():
    graphs = [sl2(p) for p in (5, 7, 11, 13, 101)]
    tables, _, _ = run_batched([g.to_dict() for g in graphs])
    for g, t in zip(graphs, tables):
        p = g.action["generators"][0]["modulo"]
        assert sum(t) == p * (p * p - 1)
        if p <= 13:
            assert t == [len(x) for x in O.c_exact_layers(g.to_dict(), p * (p * p - 1))]


def test_continuous_admission_results_equal_alone():
    # Jobs admitted while others are mid-BFS get the same tables as alone.
    jobs = [x["graph"] for x in GOLDEN[:12]] + [sl2(7).to_dict(), sl2(11).to_dict()]
    alone = [run_batched([j])[0][0] for j in jobs]
    with BatchEngine(max_slots=8) as b:
        owner, done, queue = {}, {}, list(range(len(jobs)))
        while queue or owner:
            if queue:  # admit one job per step so arrivals interleave with running ones
                slot = b.admit(jobs[queue[0]])
                if slot is not None:
                    owner[slot] = queue.pop(0)
            b.step(2)
            for slot in b.poll():
                sizes, status, error = b.result(slot)
                assert error == 0
                done[owner.pop(slot)] = sizes
                b.release(slot)
    assert [done[i] for i in range(len(jobs))] == alone


def test_memory_reused_before_a_step_starts_empty_for_its_new_owner():
    # A released block, taken again before the next step, still holds the old
    # instance's frontier keys and visited bits (or a pending, never-run
    # instance's nothing); the new owner's hash table or bitmap must start
    # empty all the same, and an instance released before any step must not
    # clear memory someone else now owns.
    first, second, dropped, last = GOLDEN[0], GOLDEN[2], GOLDEN[4], GOLDEN[6]
    with BatchEngine(max_slots=2) as b:
        s = b.admit(first["graph"], visited="bitmap")
        b.run()
        sizes, _, error = b.result(s)
        assert error == 0 and sizes == first["layer_sizes"]
        b.release(s)
        s1 = b.admit(second["graph"], visited="hash")
        s2 = b.admit(dropped["graph"], visited="hash")
        b.release(s2)
        s2 = b.admit(last["graph"], visited="bitmap")
        b.run()
        for slot, want in ((s1, second), (s2, last)):
            sizes, _, error = b.result(slot)
            assert error == 0 and sizes == want["layer_sizes"]


def test_budget_admission_refuses_when_full():
    g = GOLDEN[1]["graph"]  # n = 9 or 10
    with BatchEngine(max_slots=4, vram_budget=1) as b:
        assert b.admit(g) is None
    with BatchEngine(max_slots=2) as b:
        assert b.admit(g) is not None and b.admit(g) is not None
        assert b.admit(g) is None  # no free slot
        nbytes, visited = b.plan(g)
        assert nbytes > 0 and visited in ("bitmap", "hash")


def test_batch_samples_are_last_layer_states():
    g = GraphDefinition.permutation(O.lrx_generators(8), list(range(8)))
    ref = O.packed_bfs(8, keep_keys=True)
    with BatchEngine(max_slots=2) as b:
        slot = b.admit(g.to_dict())
        b.run()
        sizes, status, error = b.result(slot)
        rows = b.sample(slot, 8)
    assert sizes == ref["layers"] and error == 0
    assert sorted(O.pack(r) for r in rows) == sorted(ref["keys"][-1])


def test_autotuned_profile_keeps_tables_exact(tmp_path, monkeypatch):
    from multigpubfs_amd.autotune import DEFAULT, DIMENSIONS, choose_profile
    monkeypatch.setenv("MGBFS_AUTOTUNE_CACHE", str(tmp_path / "tune.json"))
    subset = GOLDEN[:32]
    inst = [x["graph"] for x in subset]
    profile = choose_profile(inst, pilot=8)
    allowed = {k: [DEFAULT[k]] + v for k, v in DIMENSIONS}
    assert all(profile[k] in allowed[k] for k in DEFAULT)
    assert all(t.get("identical", True) for t in profile["trials"])
    tried = {k for t in profile["trials"] for k in DEFAULT if t["profile"][k] != DEFAULT[k]}
    assert {"threads", "grid_per_cu", "layers_per_graph", "visited", "bitmap_bias_permille"} <= tried
    tables, _, _ = run_batched(inst, profile=profile)
    assert tables == [x["layer_sizes"] for x in subset]
    assert choose_profile(inst, pilot=8)["cached"] is True


def test_rolling_three_tables_for_undirected_hash_instances():
    # Forced hash: the inverse-closed half keeps three rolling tables sized
    # at 30% of the state bound, the directed half the full orbit.
    subset = GOLDEN[:24]
    inst = [x["graph"] for x in subset]
    tables, _, info = run_batched(inst, visited="hash", history="rolling")
    assert tables == [x["layer_sizes"] for x in subset]
    closed = sum(GraphDefinition(g).inverse_closed() for g in inst)
    assert 0 < closed < len(inst)
    assert info["modes"] == {"hash/rolling": closed, "hash/full": len(inst) - closed}
    full, _, info = run_batched(inst, visited="hash", history="full")
    assert full == tables and info["modes"] == {"hash/full": len(inst)}
    auto, _, info = run_batched(inst, visited="hash")  # the full orbit fits: no rolling
    assert auto == tables and info["modes"] == {"hash/full": len(inst)}


def test_rolling_tables_when_full_history_does_not_fit():
    # A budget below the full-history footprint but above the rolling one:
    # the automatic policy admits the instance with three rolling tables.
    g = sl2(31).to_dict()
    with BatchEngine(max_slots=2, history="full") as b:
        full_bytes = b.plan(g)[0]
    with BatchEngine(max_slots=2, history="rolling") as b:
        rolling_bytes = b.plan(g)[0]
    assert rolling_bytes < full_bytes
    with BatchEngine(max_slots=2, vram_budget=(rolling_bytes + full_bytes) // 2) as b:
        slot = b.admit(g)
        assert b.instance_info(slot)["history_layers"] == 3
        b.run()
        (done,) = b.poll()
        sizes, status, error = b.result(done)
    assert error == 0 and sizes == [len(x) for x in O.c_exact_layers(g, 31 * (31 * 31 - 1))]


def test_rolling_layer_overflow_restarts_exactly():
    # Rolling tables sized for 1% of the bound: layers outgrow them, and the
    # instances restart with doubled room until their largest layer fits.
    subset = [x for x in GOLDEN[:40] if GraphDefinition(x["graph"]).inverse_closed()][:8]
    inst = [x["graph"] for x in subset]
    tables, _, info = run_batched(inst, visited="hash", history="rolling", layer_pct=1)
    assert tables == [x["layer_sizes"] for x in subset]
    assert info["restarts"] > 0 and info["modes"] == {"hash/rolling": len(inst)}


def test_sl2_rolling_tables_match_oracle_and_report_three_layers():
    graphs = [sl2(p) for p in (5, 7, 11, 13, 31)]
    with BatchEngine(max_slots=8, history="rolling") as b:
        slots = [b.admit(g.to_dict()) for g in graphs]
        infos = [b.instance_info(s) for s in slots]
        b.run()
        results = {s: b.result(s) for s in b.poll()}
    for g, s, info in zip(graphs, slots, infos):
        p = g.action["generators"][0]["modulo"]
        assert info["visited"] == "hash" and info["history_layers"] == 3
        # 30% of the group order, at least 1024 rows, at most the order.
        assert info["layer_capacity"] == min(p * (p * p - 1), max(1024, -(-3 * p * (p * p - 1) // 10)))
        sizes, status, error = results[s]
        assert error == 0
        assert sizes == [len(x) for x in O.c_exact_layers(g.to_dict(), p * (p * p - 1))]


@pytest.mark.parametrize("threads", [128, 512])
def test_block_sizes_agree(threads):
    subset = GOLDEN[:24]
    tables, _, _ = run_batched([x["graph"] for x in subset], threads=threads)
    assert tables == [x["layer_sizes"] for x in subset]


@pytest.mark.parametrize("load", [25, 75])
def test_hash_load_factors_agree(load):
    subset = GOLDEN[:16]
    tables, _, _ = run_batched([x["graph"] for x in subset], visited="hash", hash_load_pct=load)
    assert tables == [x["layer_sizes"] for x in subset]


def test_bitmap_bias_moves_the_per_instance_choice():
    # Full history: an S9/S10 bitmap is 1/128 of the hash table's bytes, so
    # a bias of 5 per mille picks the hash table and 1000 the bitmap.
    g = GOLDEN[0]["graph"]
    for bias, want in ((5, "hash"), (1000, "bitmap")):
        with BatchEngine(max_slots=2, history="full", bitmap_bias_permille=bias) as b:
            assert b.plan(g)[1] == want
            slot = b.admit(g)
            assert b.instance_info(slot)["visited"] == want


def test_batch_options_are_validated():
    for bad in ({"threads": 64}, {"hash_load_pct": 95}, {"layer_pct": 101}):
        with pytest.raises(RuntimeError):
            BatchEngine(max_slots=2, **bad)
    with pytest.raises(ValueError):
        BatchEngine(max_slots=2, history="three")


# Bitmap instances of degree 9 to 12 run by owners of the bitmap: alone and in
# a mix, stopped at a layer limit (one short of the search, its exact length),
# released half way, and with more children in a layer (up to 10 per state of
# the group) than their messages hold at a time.
def test_large_bitmap_instances_by_owners():
    n = 11
    lrx_gens = O.lrx_generators(n)
    rng = random.Random(8)
    many = [rng.sample(range(n), n) for _ in range(14)]
    ref, ref_many, small = O.packed_bfs(n)["layers"], O.packed_bfs(n, many)["layers"], O.packed_bfs(9)["layers"]
    jobs = [(lrx_gens, n, 0), (O.lrx_generators(9), 9, 0), (lrx_gens, n, len(ref) - 1), (many, n, 0),
            (lrx_gens, n, len(ref))]
    with BatchEngine(max_slots=8, vram_budget=16 << 30) as b:
        half = b.admit(GraphDefinition.permutation(lrx_gens, list(range(n))))
        b.step(8)
        b.release(half)
        slots = [b.admit(GraphDefinition.permutation(g, list(range(k))), max_layers=m) for g, k, m in jobs]
        b.step(3)
        assert b.result(slots[0])[0] == ref[:len(b.result(slots[0])[0])]
        done = []
        while len(done) < len(jobs):
            b.step(4)
            done += b.poll()
        results = [b.result(s) for s in slots]
        last = b.sample(slots[0], n)
        infos = [b.instance_info(s) for s in slots]
    assert [r[0] for r in results] == [ref, small, ref[:-1], ref_many, ref]
    assert [bool(r[2]) for r in results] == [False, False, True, False, False]
    assert len(last) == ref[-1] and all(sorted(row) == list(range(n)) for row in last)
    assert all(i["visited"] == "bitmap" and i["restarts"] == 0 and i["history_layers"] == 0 for i in infos)


@pytest.mark.parametrize("n,count,closed,copies", [(8, 3, False, 1), (9, 1, True, 1), (9, 16, False, 1),
                                                   (9, 14, False, 9), (10, 2, False, 1), (10, 5, True, 21)])
def test_owned_instances_match_oracle_layer_by_layer(n, count, closed, copies):
    # 1, 9 and 21 instances: 251, 101 and 53 owners (degree 8: none); back
    # edges named (closed sets up to 14) or not; the current layer's states
    # after every step, whole where the layer is small.
    rng = random.Random(n * count)
    gens = [rng.sample(range(n), n) for _ in range(count)]
    if closed:
        gens += [[g.index(i) for i in range(n)] for g in gens]
    ref = O.packed_bfs(n, gens, keep_keys=True)
    seen = 0
    with BatchEngine(max_slots=32, layers_per_graph=1) as b:
        slots = [b.admit(GraphDefinition.permutation(gens, list(range(n)))) for _ in range(copies)]
        while b.step(1):
            d = len(b.result(slots[-1])[0]) - 1
            rows = [O.pack(r) for r in b.sample(slots[-1], n, 2000)]
            assert len(rows) == min(2000, ref["layers"][d]) == len(set(rows))
            assert set(rows) <= set(ref["keys"][d])
            seen += 1
        assert [b.result(s)[0] for s in slots] == [ref["layers"]] * copies
        assert {O.pack(r) for r in b.sample(slots[0], n, 10**6)} == set(ref["keys"][-1])
    assert seen >= len(ref["layers"]) - 1


# Arena chunks outlive their engine in a bounded cache: later engines (with
# smaller, equal and larger needs, of two threads) find them with the contents
# they were left with, and count them as free memory.
def test_engines_reuse_kept_memory_exactly():
    import threading
    from multigpubfs_amd._native import load
    inst = [x["graph"] for x in GOLDEN[:12]]
    golden = [x["layer_sizes"] for x in GOLDEN[:12]]
    assert run_batched(inst)[0] == golden
    with BatchEngine(vram_budget=8 << 30) as b:
        slot = b.admit(GraphDefinition.permutation(O.lrx_generators(11), list(range(11))), visited="hash")
        b.run()
        assert b.result(slot)[0] == O.packed_bfs(11)["layers"]
    with BatchEngine() as b:
        kept = b.usage()["budget"]
    load().mgbfs_release_cached_memory(0)
    with BatchEngine() as b:
        assert abs(b.usage()["budget"] - kept) < 1 << 30
    out = {}

    def work(k, **options):
        out[k] = [run_batched(inst[k::2], **options)[0] for _ in range(3)]

    threads = [threading.Thread(target=work, args=(0,)),
               threading.Thread(target=work, args=(1,), kwargs={"visited": "hash"})]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == {k: [golden[k::2]] * 3 for k in (0, 1)}


@pytest.mark.parametrize("n,layers,copies", [(8, 9, 1), (9, 12, 1), (10, 3, 1), (10, 14, 1), (10, 14, 9), (10, 14, 21),
                                             (11, 13, 1)])
def test_sample_of_an_instance_stopped_at_its_layer_limit(n, layers, copies):
    # The step that meets the limit has found the next layer already: the
    # sample still holds the last layer of the result, and only it.
    gens = O.lrx_generators(n)
    ref = O.packed_bfs(n, gens, keep_keys=True)
    with BatchEngine(max_slots=32, vram_budget=8 << 30) as b:
        slots = [b.admit(GraphDefinition.permutation(gens, list(range(n))), max_layers=layers) for _ in range(copies)]
        b.run()
        for s in slots:
            sizes, _, error = b.result(s)
            assert error and sizes == ref["layers"][:layers]
            rows = [O.pack(r) for r in b.sample(s, n, 10**7)]
            assert sorted(rows) == sorted(ref["keys"][layers - 1])


# A step of the batch runs one form of instances or both, by what is there:
# degree 10 alone (151, 101, 53 owners for 1, 4 and 21), degree 9 beside it or
# beside degree 11, eight of degree 10 beside smaller ones, and sets that stay
# on the shared bitmap; smaller searches join when some layers are done.
@pytest.mark.parametrize("jobs", [{10: 1}, {10: 4}, {10: 21}, {10: 4, 9: 8}, {11: 1, 9: 4, 8: 2}, {10: 8, 8: 3}, {9: 3},
                                  {10: 1, 8: 1}], ids=str)
def test_forms_of_a_step_match_oracle(jobs):
    rng = random.Random(5)
    sets = {}
    for n in {*jobs, 8}:
        gens = [[(i + 1) % n for i in range(n)], rng.sample(range(n), n), rng.sample(range(n), n)]
        sets[n] = gens, O.packed_bfs(n, gens, keep_keys=n <= 10)
    late = [GraphDefinition.permutation(sets[8][0], list(range(8))), sl2(11), GOLDEN[0]["graph"]]
    with BatchEngine(max_slots=32, layers_per_graph=1, vram_budget=16 << 30) as b:
        slots = [(n, b.admit(GraphDefinition.permutation(sets[n][0], list(range(n)))))
                 for n, count in jobs.items() for _ in range(count)]
        watched = {n: s for n, s in slots}
        steps = 0
        while b.step(1):
            steps += 1
            for n, s in watched.items():
                sizes, ref = b.result(s)[0], sets[n][1]
                assert sizes == ref["layers"][:len(sizes)]
                if n <= 10:
                    rows = [O.pack(r) for r in b.sample(s, n, 500)]
                    assert len(set(rows)) == min(500, sizes[-1]) and set(rows) <= set(ref["keys"][len(sizes) - 1])
            if steps == 3:
                late = [b.admit(g) for g in late]
        for n, s in slots:
            sizes, _, error = b.result(s)
            assert not error and sizes == sets[n][1]["layers"]
        assert b.result(late[0])[0] == sets[8][1]["layers"]
        assert sum(b.result(late[1])[0]) == 11 * 120 and b.result(late[2])[0] == GOLDEN[0]["layer_sizes"]


@pytest.mark.parametrize("copies,bound", [(1, 919200), (4, 916600), (21, 914200)])
def test_overflowing_messages_start_over_on_the_shared_bitmap(copies, bound):
    # A declared state bound far below n! leaves an owner room for some 70
    # messages at a time, of which a step uses two thirds on average: now and then one gets more.
    n = 10
    gens = O.lrx_generators(n)
    ref = O.packed_bfs(n, gens, keep_keys=True)
    graph = GraphDefinition.permutation(gens, list(range(n)), expected_max_unique_states=bound)
    with BatchEngine(max_slots=32, vram_budget=8 << 30) as b:
        slots = [b.admit(graph, visited="bitmap") for _ in range(copies)]
        b.run()
        for s in slots:
            sizes, _, error = b.result(s)
            assert not error and sizes == ref["layers"]
            assert sorted(O.pack(r) for r in b.sample(s, n, 10**6)) == sorted(ref["keys"][-1])
        assert any(b.instance_info(s)["restarts"] for s in slots)


def test_engines_made_beside_other_threads_copies():
    # Batch engines come and go in one thread while another's engines upload
    # their generators and read their states back.
    import threading
    stop, errors, made = threading.Event(), [], [0, 0]

    def others():
        try:
            while not stop.is_set():
                with NativeEngine(sl2(13), backend="segmented", flags=128) as e:
                    assert e.run() == 1 and len(e.sample(0, 1000)) == e.layer_sizes()[-1]
                made[1] += 1
        except Exception as exc:
            errors.append(exc)

    thread = threading.Thread(target=others)
    thread.start()
    try:
        for _ in range(60):
            with BatchEngine(max_slots=2) as b:
                slot = b.admit(sl2(11))
                b.run()
                assert sum(b.result(slot)[0]) == 11 * 120
            made[0] += 1
    finally:
        stop.set()
        thread.join()
    assert not errors and made[0] == 60 and made[1] > 5


@pytest.mark.parametrize("n", [8, 10])
def test_layer_beyond_the_declared_bound_is_an_error(n):
    # Sixteen generators: the widest layer holds more states than the graph
    # declares in all, by owners (degree 10) as over the shared bitmap.
    rng = random.Random(n)
    gens = [rng.sample(range(n), n) for _ in range(16)]
    ref = O.packed_bfs(n, gens)["layers"]
    bound = {8: 5000, 10: 1_000_000}[n]
    assert max(ref) > bound
    with BatchEngine(max_slots=2) as b:
        graph = GraphDefinition.permutation(gens, list(range(n)), expected_max_unique_states=bound)
        slot, free = b.admit(graph, visited="bitmap"), b.admit(GraphDefinition.permutation(gens, list(range(n))))
        b.run()
        sizes, _, error = b.result(slot)
        assert error and sizes == ref[:len(sizes)] and max(sizes) <= bound
        assert b.result(free)[0] == ref and not b.result(free)[2]


def test_kept_memory_is_given_back_on_request():
    import ctypes
    from hip_memory import hip
    from multigpubfs_amd import device_info, release_cached_memory

    def kept():  # counted as free beyond what the device has
        now, total = ctypes.c_size_t(), ctypes.c_size_t()
        counted = device_info()["free_bytes"]
        assert hip().hipMemGetInfo(ctypes.byref(now), ctypes.byref(total)) == 0
        return counted - now.value

    run_batched([x["graph"] for x in GOLDEN[:4]])
    assert 1 << 30 <= kept() <= 16 << 30  # a chunk at least
    release_cached_memory()
    assert kept() == 0
