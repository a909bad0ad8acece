"""Row ids and Aggregated groups where their kernels' work is cut: chunks of any size, more quarter
chunks than stamps, results larger than one piece; histograms in copies, in ranges, past the last
range and past the kept ones; symbols at positions stored as bitsets, runs, groups and light entries,
inside and outside the coverage bounds, under missing runs and null rows.  Against numpy."""
import numpy as np
import pytest

from helpers import bitset_table, small_spec

pytestmark = pytest.mark.gpu


def plain_table(engine, sizes, seed=1, values=()):
    """A table of an int column x in [0, 1000) and one dictionary column per count in `values`."""
    from silo_amd import table

    rng = np.random.default_rng(seed)
    sizes = np.asarray(sizes, np.uint32)
    n = int(sizes.sum())
    spec = table.TableSpec(chunk_sizes=sizes)
    x = rng.integers(0, 1000, n).astype(np.int32)
    spec.int_columns.append(table.IntColumnData("x", False, x, np.zeros(n, np.uint8)))
    cols = []
    for k, v in enumerate(values):
        # skewed: most rows share a few values, as country and lineage columns do
        ids = np.minimum(rng.integers(0, v, n), rng.integers(0, v, n) * (rng.random(n) < 0.7)).astype(np.uint32)
        null = (rng.random(n) < 0.01).astype(np.uint8)
        spec.dict_columns.append(table.DictColumnData(f"d{k}", ids, null, [f"v{i:05d}" for i in range(v)]))
        cols.append((ids, null))
    return engine.table(spec), spec.global_ids(), x, cols


@pytest.mark.parametrize("sizes", [[1], [65536, 3, 65536, 0, 40000], [17] * 300, [65536] * 70])
def test_row_ids(engine, sizes):
    """(70 full chunks: more rows than one piece of 2^22.)"""
    et, ids, x, _ = plain_table(engine, sizes)
    try:
        for lo, hi in ((0, 999), (0, 0), (5, 4), (0, 400), (500, 501), (999, 999)):
            want = ids[(x >= lo) & (x <= hi)]
            assert np.array_equal(et.filter(f"(int_between x {lo} {hi})"), want), (lo, hi)
    finally:
        et.close()


@pytest.mark.parametrize("values", [(1,), (3, 50), (63, 63), (64, 63), (70, 80), (200, 180), (500, 490), (600, 600),
                                    (20, 20, 20, 20)])
def test_group_counts(engine, values):
    """Combinations (one more label per column: null) from 2 bins to 361,201: both sides of 4,096
    (copies), 32,768 (one LDS range) and 2^18 (the last range, and the kept histogram)."""
    et, _, x, cols = plain_table(engine, [65536, 30000, 700], seed=sum(values), values=values)
    dims = [f"d{k}" for k in range(len(values))]
    try:
        for expr, keep in (("(true)", x >= 0), ("(int_between x 0 30)", x <= 30), ("(int_between x 7 7)", x == 7)):
            key = np.zeros(len(x), np.int64)
            for (ids, null), v in zip(cols, values):
                key = key * (v + 1) + np.where(null != 0, v, ids)
            found, counts = np.unique(key[keep], return_counts=True)
            want = []
            for f, c in zip(found.tolist(), counts.tolist()):
                parts = []
                for v in reversed(values):
                    parts.append(None if f % (v + 1) == v else f % (v + 1))
                    f //= v + 1
                want.append((tuple(reversed(parts)), c))
            # value order with null last: the order of the combined key
            assert et.aggregate(expr, dims) == want, expr
            assert et.aggregate(expr, dims) == want, expr  # the kept histogram was left clear
            assert et.batch([{"filter": expr, "action": "aggregate", "dims": dims}]) == [want], expr
    finally:
        et.close()


def position_groups(M, null, extra, keep, positions, n_symbols):
    """Groups of (symbol at each position[, extra]) over the rows in `keep`, null group last."""
    key = np.zeros(len(null), np.int64)
    for p in positions:
        key = key * (n_symbols + 1) + np.where(null != 0, n_symbols, M[:, p])
    bases = [n_symbols + 1] * len(positions)
    if extra is not None:
        ids, enull, v = extra
        key = key * (v + 1) + np.where(enull != 0, v, ids)
        bases.append(v + 1)
    found, counts = np.unique(key[keep], return_counts=True)
    out = []
    for f, c in zip(found.tolist(), counts.tolist()):
        parts = []
        for b in reversed(bases):
            parts.append(None if f % b == b - 1 else f % b)
            f //= b
        out.append((tuple(reversed(parts)), c))
    return out


def test_position_groups_of_every_container(engine):
    spec, M, null = bitset_table()
    et = engine.table(spec)
    date = spec.int_columns[0]
    some = (date.values >= 18262) & (date.values <= 18263) & (date.is_null == 0)
    every = np.ones(len(null), bool)
    d = spec.dict_columns[0]
    try:
        for expr, keep in (("(true)", every), ("(date_between date 18262 18263)", some)):
            for positions in ([0], [1], [5], [10], [20], [30], [31], [40], [50], [60], [62], [75], [95], [40, 62],
                              [10, 20, 50], [0, 31, 61, 94]):
                want = position_groups(M, null, None, keep, positions, 16)
                assert et.aggregate(expr, [f"main@{p}" for p in positions]) == want, (expr, positions)
            want = position_groups(M, null, (d.ids, d.is_null, 3), keep, [62], 16)
            assert et.aggregate(expr, ["main@62", "country"]) == want
    finally:
        et.close()


def test_position_groups_with_long_missing_runs(engine):
    """Runs in the buckets before the position's and longer than the longest bucketed run, ragged
    coverage, uneven chunks: a 5,000-position genome against the oracle."""
    from oracle.oracle import OracleTable
    from silo_amd import datagen, table

    spec = datagen.GenSpec(n_rows=3000, genome_length=5000, seed=77, lineage_model=True, n_nodes=30, n_lambda=4.0,
                           n_mean=900.0, null_seq_frac=0.02, null_meta_frac=0.05, n_days=50)
    ts = table.spec_from_dataset(datagen.generate(spec), chunk=700)
    ot, et = OracleTable(ts), engine.table(ts)
    try:
        for p in (0, 1, 255, 256, 1023, 1024, 1025, 2047, 3000, 4998, 4999):
            for expr in ("(true)", "(date_between date 18262 18270)"):
                dims = [f"main@{p}", "country"]
                assert et.aggregate(expr, dims) == ot.aggregate(expr, dims), (p, expr)
    finally:
        et.close()
        ot.close()
