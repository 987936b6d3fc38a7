"""Kernels at the edges of their size ranges, against the oracle."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("props, atoms", [(7, "dense"), (64, "dense"), (65, "dense"), (130, "reachable"), (512, "dense"), (1000, "dense"),
                                          (130, "lazy"), (1090, "dense")])
def test_search_fingerprint_over_row_widths(props, atoms):
    """Narrow rows (1, 2, 4, 8 and 16 words: nibble tables), wider ones and lazily grown rows (a wave per row): the
    fingerprint does not depend on the slots, so a lazy search has the dense oracle's."""
    from mymyr_amd import gen, search
    from mymyr_amd.task import Task
    from oracle import port

    text = gen.random_strips(props, 4 * props, init_atoms=max(3, props // 8), goal_atoms=2, seed=4)
    kw = dict(max_depth=2, stop_at_goal=False)
    r = search.brfs(Task.from_text(text, atoms), fingerprint=True, **kw)
    p = port.brfs(port.Task(text, "dense"), max_states=1 << 40, **kw)
    assert (r.states, r.fingerprint) == (p["states"], p["fingerprint"])


TASKS = ["blocks__probBLOCKS-8-0", "gripper__prob05", "logistics00__probLOGISTICS-6-1", "miconic__s7-4", "zenotravel__p05",
         "driverlog__p03", "depot__p02", "rovers__p02", "freecell__p02", "pegsol-08-strips__p22", "sokoban-opt08-strips__p14",
         "visitall__visitall_x-6_y-3_r-100", "snake-opt18-strips__p05", "parcprinter-opt11-strips__p03", "pathways__p02",
         "transport-opt08-strips__p23", "noop_switches", "witness_order_0", "gridworld", "transport", "strips"]


@pytest.mark.parametrize("name", TASKS)
def test_counts_after_a_move_equal_a_recount(name, golden):
    """A step brings the successor counts up to date from the move's changed atoms (and the cache row's fingerprint from
    its changed words), and a refresh counts the same states from nothing: the same counts and cache rows, over domains
    whose literals share predicates, repeat objects, are negative, ground or of three and more terms."""
    import torch

    from mymyr_amd import rl
    from mymyr_amd.task import Task

    pool = rl.DeviceEnvPool(Task.from_text_file(golden.task_path(name)), 96, seed=11, max_steps=25)
    pool.reset()
    for k in range(40):
        pool.step()
        count, cache = pool.count.clone(), pool.counts_cache.clone()
        pool.refresh()
        assert torch.equal(count, pool.count), f"{name}: counts at step {k}"
        assert torch.equal(cache, pool.counts_cache), f"{name}: cache rows at step {k}"
    pool.check()


@pytest.mark.parametrize("words", [*range(1, 17), 17, 18, 31, 32, 33, 47, 176, 200, 1025])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 257])
def test_hash_of_wide_rows(words, rows):
    """Rows up to 16 words hashed by a lane each, 64 to a wave, and these few wider ones by a wave each: row counts around a
    wave, widths around a tile, rows whose trimmed length ends anywhere (an empty row included)."""
    import torch

    from mymyr_amd import hip
    from oracle import port

    rng = np.random.default_rng(words * 1000 + rows)
    a = rng.integers(0, 1 << 63, size=(rows, words), dtype=np.uint64)
    for i in range(rows):
        a[i, rng.integers(0, words + 1):] = 0
    a[rows // 2] = 0
    got = hip.hash_rows(torch.from_numpy(a.view(np.int64)).cuda()).cpu().numpy().view(np.uint64)
    assert [int(x) for x in got] == [port.hash_state(r) for r in a]


@pytest.mark.parametrize("words", [17, 33, 127, 128, 129, 176, 300])
@pytest.mark.parametrize("rows", [3, 2048, 2049, 2100])
def test_hash_of_few_and_many_wide_rows(words, rows):
    """Rows above 16 words hashed a wave each (up to 2,048) and a lane each: rows around the line, widths around the 128
    words that a wave reads at once, trimmed lengths of no tile to all, whole waves of short rows."""
    import torch

    from mymyr_amd import hip
    from oracle import port

    rng = np.random.default_rng(words * 1000 + rows)
    a = rng.integers(0, 1 << 63, size=(rows, words), dtype=np.uint64)
    for i in range(0, rows, 3):
        a[i, rng.integers(0, words + 1):] = 0
    a[64:128, 5:] = 0
    a[0] = 0
    got = hip.hash_rows(torch.from_numpy(a.view(np.int64)).cuda()).cpu().numpy().view(np.uint64)
    assert [int(x) for x in got] == [port.hash_state(r) for r in a]


@pytest.mark.parametrize("rows", [1, 64, 1000])
def test_hash_of_rows_without_words(rows):
    """The C ABI takes rows of no words: each hashes as the empty row."""
    import torch

    from mymyr_amd._lib import check, lib
    from oracle import port

    out = torch.zeros(rows, dtype=torch.int64, device="cuda")
    check(lib.mya_hash_rows(out.data_ptr(), rows, 0, out.data_ptr(), None))
    torch.cuda.synchronize()
    assert [int(x) for x in out.cpu().numpy().view(np.uint64)] == [port.hash_state(np.zeros(0, np.uint64))] * rows


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("k", [1, 7, 40])
def test_pad_of_rows_at_any_alignment(k, shift):
    """The padded view of rows of an even width (16 bytes a lane), and of the same rows starting 8 bytes off."""
    import torch

    from mymyr_amd import gen, rl
    from mymyr_amd.task import Task
    from oracle import port

    t = Task.from_text(gen.transport(24, 6, 42, goals=6, seed=2))
    assert t.words % 2 == 0
    pool = rl.DeviceEnvPool(t, 33, seed=3)
    pool.reset()
    pool.step()
    x = rl.expand(t, pool.states, goal=True, hashes=True)
    n = x["succ"].shape[0]
    buf = torch.empty(n * t.words + shift, dtype=torch.int64, device="cuda")
    buf[shift:] = x["succ"].reshape(-1)
    flat = dict(x, succ=buf[shift:].view(n, t.words))
    p = rl.pad(flat, k)
    off = x["offsets"].cpu().numpy()
    succ, bind = x["succ"].cpu().numpy(), x["binding"].cpu().numpy()
    for i in range(33):
        c = min(k, int(off[i + 1] - off[i]))
        row = p["succ"][i].cpu().numpy()
        assert np.array_equal(row[:c], succ[off[i]: off[i] + c]) and not row[c:].any()
        b = p["binding"][i].cpu().numpy()
        assert np.array_equal(b[:c], bind[off[i]: off[i] + c]) and (b[c:] == -1).all()
    assert [int(h) for h in x["succ_hash"].cpu().numpy().view(np.uint64)] == [port.hash_state(r) for r in succ.view(np.uint64)]


@pytest.mark.parametrize("name", TASKS + ["crowded"])
def test_expansion_equals_the_successor_listing(name, golden):
    """The flat expansion lists successors 64 at a time from a list of 128 bindings (crowded: more than 128 successors
    under one word of a first parameter; every arity, effect count and atom layout of the suite's tasks), the successor
    listing enumerates them one by one: the same labels and rows, and the rows' flags follow from them."""
    import torch

    from mymyr_amd import gen, rl
    from mymyr_amd.task import Task

    t = Task.from_text(gen.transport(6, 16, 80, seed=3)) if name == "crowded" else Task.from_text_file(golden.task_path(name))
    pool = rl.DeviceEnvPool(t, 37, seed=5, max_steps=None)
    pool.reset()
    for _ in range(9):
        pool.step()
    s = pool.states.clone()
    x = rl.expand(t, s, goal=True, noops=True, hashes=True)
    cap = int((x["offsets"][1:] - x["offsets"][:-1]).max())
    count, schema, binding, rows = rl.successors(t, s, cap=max(cap, 1))
    assert torch.equal(count, (x["offsets"][1:] - x["offsets"][:-1]))
    live = torch.arange(max(cap, 1), device="cuda")[None, :] < count[:, None]
    assert torch.equal(x["schema"], schema[live]) and torch.equal(x["binding"], binding[live]) and torch.equal(x["succ"], rows[live])
    parent = torch.arange(37, device="cuda", dtype=torch.int32)[:, None].expand(live.shape)[live]
    assert torch.equal(x["parent"], parent)
    assert torch.equal(x["noop"] != 0, (x["succ"] == s[parent.long()]).all(dim=1))
    d = rl.expand(t, s, drop_noops=True, noops=True)
    keep = x["noop"] == 0
    for i in range(37):
        a, b = int(x["offsets"][i]), int(x["offsets"][i + 1])
        if not keep[a:b].any():
            keep[a:b] = True
    assert torch.equal(d["succ"], x["succ"][keep]) and torch.equal(d["schema"], x["schema"][keep])


def test_expansion_of_the_widest_rows():
    """A state of 20,300 words leaves a wave's region in a workgroup's 160 KiB of LDS, but no room for the list of
    bindings beside it: the expansion enumerates the successors one by one."""
    import torch

    from mymyr_amd import rl
    from mymyr_amd.task import Task

    n, preds, items = 64960, 20, 8
    lines = [f"O {n}", f"P {preds + 2}", "S 1 item", *(f"F 1 p{k}" for k in range(preds)), "F 1 never", f"SI {items}",
             *(f"0 {o}" for o in range(items)), "FI 1", "1 9", "G 1", "1 1 5", f"A {preds // 5 + 1}", "set 1", "L 2", "0 1 0", "1 0 0",
             "E 1", "0", "L 0", "F 1", "1 1 0"]
    for k in range(0, preds, 5):  # (every atom can be added, so every object has its slots; never applicable)
        lines += [f"fill{k} 1", "L 1", f"{preds + 1} 1 0", "E 1", "0", "L 0", "F 5", *(f"{k + j + 1} 1 0" for j in range(5))]
    t = Task.from_text("\n".join(lines) + "\n", "dense")
    assert 20300 <= t.words <= 20316
    s = torch.from_numpy(t.initial_state().view(np.int64).copy())[None].repeat(3, 1).cuda()
    s[1, 0] |= 1 << 3
    s[2, -1] |= 1
    x = rl.expand(t, s, goal=True, hashes=True)
    want = [(i, o) for i in range(3) for o in range(items) if not (int(s[i, 0]) >> o) & 1]
    assert x["total"] == len(want) and x["binding"][:, 0].tolist() == [o for _, o in want]
    for j, (i, o) in enumerate(want):
        row = s[i].clone()
        row[0] |= 1 << o
        assert torch.equal(x["succ"][j], row) and int(x["goal"][j]) == (o == 5 or (int(s[i, 0]) >> 5) & 1)
    count, _, binding, rows = rl.successors(t, s, cap=items)
    assert count.tolist() == [8, 7, 8] and torch.equal(x["succ"][:8], rows[0])


@pytest.mark.parametrize("words", [17, 32, 33, 64, 65, 128, 129, 160, 161, 192, 193, 256, 257])
def test_state_set_at_the_lane_group_shapes(words):
    """Rows at the edges of the probe's lane-group shapes, with duplicates inside a batch and across batches: ids are
    first-occurrence ranks."""
    import torch

    from mymyr_amd import hip

    rng = np.random.default_rng(words)
    base = rng.integers(0, 1 << 63, size=(700, words), dtype=np.uint64)
    base[:, -1] &= np.uint64(rng.integers(0, 2))
    pick = rng.integers(0, 700, size=2500)
    rows = base[pick]
    s = hip.StateSet(1024, words, 0.5, batch=1000)
    first, want = {}, []
    for p in pick:
        want.append(first.setdefault(int(p), len(first)))
    dev = torch.from_numpy(rows.view(np.int64)).cuda()
    ids = torch.cat([s.insert(dev[:1700])[1], s.insert(dev[1700:])[1]]).cpu().numpy()
    assert len(s) == len(first) and ids.tolist() == want
    got = torch.from_dlpack(s.rows()).view(torch.int64).cpu().numpy().view(np.uint64)
    order = [p for p, _ in sorted(first.items(), key=lambda x: x[1])]
    assert np.array_equal(got, base[order])


@pytest.mark.parametrize("name", ["gridworld", "gripper__prob05", "noop_switches", "witness_order_0", "blocks__probBLOCKS-8-0",
                                  "sokoban-opt08-strips__p14", "strips"])
def test_searches_by_small_layers_equal_the_launches(name, golden):
    """Layers taken whole by one block and by the launches (a chunk too small for the block's batch): the same counts,
    fingerprints, goal states and plans, with budgets of states, expansions and layers that end a search inside its small
    layers, right after them and past them (layers of 1 to more than 512 parents)."""
    from mymyr_amd import search
    from mymyr_amd.task import Task

    task = Task.from_text_file(golden.task_path(name))
    cases = [dict(), dict(stop_at_goal=False)]
    cases += [dict(stop_at_goal=False, max_states=n) for n in (1, 2, 5, 63, 64, 65, 500, 2000, 9000)]
    cases += [dict(stop_at_goal=False, max_expanded=n) for n in (0, 1, 3, 64, 500, 513, 3000)]
    cases += [dict(stop_at_goal=False, max_depth=n) for n in (0, 1, 3, 9)]
    for kw in cases:
        kw = {"max_states": 60000, **kw}
        a = search.brfs(task, fingerprint=True, **kw)
        b = search.brfs(task, fingerprint=True, chunk=2048, **kw)
        key = lambda r: (r.status, r.states, r.expanded, r.generated, r.layers, r.num_goal_states, r.fingerprint, r.cost,  # noqa: E731
                         [tuple(x) for x in r.layer_counts], [(x.schema, tuple(x.binding)) for x in r.plan])
        assert key(a) == key(b), f"{name}: {kw}"


@pytest.mark.parametrize("props, max_states", [(60, (1 << 21) - 1), (60, (1 << 21) + 1), (200, 3000001), (640, 2500000)])
def test_search_past_the_table_it_starts_on(props, max_states):
    """A search takes its whole table when 2^21 states and a chunk's successors no longer fit half of the slots it started
    on: chunks of several sizes reach that with different states stored, and store the same ones."""
    from mymyr_amd import gen, search
    from mymyr_amd.task import Task

    task = Task.from_text(gen.random_strips(props, 2048, init_atoms=props // 8, seed=9), "dense")
    kw = dict(max_states=max_states, stop_at_goal=False, fingerprint=True)
    whole = search.brfs(task, **kw)
    for chunk in (1 << 16, 1 << 20):
        r = search.brfs(task, chunk=chunk, **kw)
        assert (r.states, r.expanded, r.generated, r.fingerprint, r.layer_counts) == (whole.states, whole.expanded, whole.generated,
                                                                                      whole.fingerprint, whole.layer_counts)
    larger = search.brfs(task, **{**kw, "max_states": 1 << 25, "max_depth": len(whole.layer_counts) - 1})
    assert larger.layer_counts == whole.layer_counts[:-1]


@pytest.mark.parametrize("limit, depth", [(500, 260), (3000, 160)])
def test_layer_cuts_that_fill_the_table(limit, depth):
    """Layers cut by max_next_layer_states leave the entries of the winners past the cut in the table, more in all than the
    2^22 slots a search starts on and than the whole table of a search by small chunks, while few states are stored. The
    table is taken whole, or cleared and its states entered anew: the same search however large it is."""
    from mymyr_amd import gen, search
    from mymyr_amd.task import Task

    task = Task.from_text(gen.random_strips(512, 4096, init_atoms=64, seed=4), "dense")
    kw = dict(max_depth=depth, max_states=limit * depth + 100000, max_next_layer_states=limit, layer_order="in_order", stop_at_goal=False,
              fingerprint=True)
    runs = [search.brfs(task, **kw, **c) for c in ({}, {"chunk": 1 << 21}, {"chunk": 1 << 17}, {"chunk": 1 << 23})]
    assert runs[0].layers == depth and all(new == limit for _, _, new in runs[0].layer_counts[-depth // 2:])
    for r in runs[1:]:
        assert (r.states, r.expanded, r.generated, r.fingerprint, r.layer_counts) == (runs[0].states, runs[0].expanded, runs[0].generated,
                                                                                      runs[0].fingerprint, runs[0].layer_counts)
