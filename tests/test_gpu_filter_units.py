"""Filter programs where the filter kernel's work is cut: stacks around the entries that registers hold
and deeper, programs around the length that is cut into single slices, counters that carry through every
plane; alone, in batches of mixed lengths and in small batches.  Against numpy."""
import numpy as np
import pytest

from test_gpu_rows_groups import plain_table

pytestmark = pytest.mark.gpu


def leaf(rng, x):
    lo = int(rng.integers(0, 1000))
    hi = int(min(999, lo + rng.integers(0, 700)))
    return f"(int_between x {lo} {hi})", (x >= lo) & (x <= hi)


def chain(rng, x, length):
    """and(leaf, or(leaf, not(and(leaf, ...)))): one stack entry a level."""
    text, keep = leaf(rng, x)
    for k in range(length):
        t, m = leaf(rng, x)
        if k % 3 == 2:
            text, keep = f"(not {text})", ~keep
        if k % 2:
            text, keep = f"(and {t} {text})", m & keep
        else:
            text, keep = f"(or {t} {text})", m | keep
    return text, keep


def nof(rng, x, m, levels, exact):
    """n of m, whose first child is another one: planes + 1 entries a level."""
    parts = [nof(rng, x, m, levels - 1, exact) if k == 0 and levels > 1 else leaf(rng, x) for k in range(m)]
    count = np.sum([p[1] for p in parts], axis=0)
    n = int(rng.integers(1, m + 1))
    return f"(nof {n} {int(exact)} " + " ".join(p[0] for p in parts) + ")", count == n if exact else count >= n


def programs(rng, x):
    out = [chain(rng, x, k) for k in (0, 1, 2, 7, 8, 13, 14, 15, 16, 22, 30, 40)]
    out += [nof(rng, x, m, 1, m % 2 == 0) for m in (2, 3, 7, 8, 15, 16, 20, 33, 70)]
    out += [nof(rng, x, 20, levels, levels % 2 == 0) for levels in (2, 3, 4)]
    return out


@pytest.mark.parametrize("sizes", [[1], [4096, 65536, 70], [65536] * 9])
def test_programs(engine, sizes):
    et, ids, x, _ = plain_table(engine, sizes, seed=len(sizes))
    try:
        cases = programs(np.random.default_rng(7), x)
        for text, keep in cases:
            assert np.array_equal(et.filter(text), ids[keep]), text
            assert et.count(text) == int(keep.sum()), text
        many = cases * 12  # long programs and short ones, more units than wavefronts at nine chunks
        with et.batch_submit([{"action": "count", "filter": text} for text, _ in many]) as b:
            assert [b.count(q) for q in range(len(many))] == [int(keep.sum()) for _, keep in many]
    finally:
        et.close()


@pytest.mark.parametrize("chunks,n", [(1, 1), (1, 24), (3, 8), (9, 4), (9, 8), (16, 8), (16, 16)])
def test_small_batches(engine, chunks, n):
    """Batches of n programs around the number of slices up to which the operand stack lies in LDS, for
    shallow stacks (4,096: 16 chunks, 16 programs) and for deeper ones (3,072 to 1,024)."""
    et, _, x, _ = plain_table(engine, [65536] * (chunks - 1) + [4500], seed=chunks)
    try:
        cases = programs(np.random.default_rng(11), x)
        for k in range(0, len(cases), n):
            some = cases[k:k + n]
            with et.batch_submit([{"action": "count", "filter": text} for text, _ in some]) as b:
                assert [b.count(q) for q in range(len(some))] == [int(keep.sum()) for _, keep in some], k
    finally:
        et.close()


@pytest.mark.parametrize("n", [3, 63, 64, 65, 127, 129, 500, 1025, 4095, 4096])
def test_array_containers(engine, n):
    """Array containers around the sizes where a sample stands for one row, or a slice for several rounds:
    spread evenly, at random, crowded at either end, around one slice's edge.  (Rows two apart: no runs.)"""
    from silo_amd import table

    rng = np.random.default_rng(n)
    size = 65536
    sets = [np.arange(n) * (size // n), rng.choice(size // 2, n, replace=False) * 2, np.arange(n) * 2, size - 1 - np.arange(n) * 2,
            8191 + 2 * (np.arange(n) - n // 2)]
    spec = table.TableSpec(chunk_sizes=np.array([size, 700], np.uint32))
    want = []
    for k, rows in enumerate(sets):
        rows = np.unique(np.clip(rows, 0, size - 1))
        ids = np.zeros(size + 700, np.uint32)
        ids[rows] = 1
        spec.dict_columns.append(table.DictColumnData(f"d{k}", ids, np.zeros(size + 700, np.uint8), ["other", "mine"]))
        want.append(rows)
    et = engine.table(spec)
    try:
        for k, rows in enumerate(want):
            assert np.array_equal(et.filter(f'(str_eq d{k} "mine")'), spec.global_ids()[rows]), k
        with et.batch_submit([{"action": "count", "filter": f'(str_eq d{k} "mine")'} for k in range(len(want))]) as b:
            assert [b.count(k) for k in range(len(want))] == [len(rows) for rows in want]
    finally:
        et.close()
