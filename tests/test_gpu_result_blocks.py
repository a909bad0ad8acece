"""Single Mutations queries where the counting and result kernels' work is cut: genomes around the
64-position result blocks and longer than one counting block's LDS totals, tables of one chunk up to
more chunks than groups (tiles shared by several work-groups in between), both methods, both
counter forms; and filter programs too long for the kernel's arguments.  Against the oracle."""
import numpy as np
import pytest

from helpers import ExprGen, small_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,n_rows,chunk", [(20, 50, 64), (63, 300, 128), (64, 700, 64), (65, 1300, 64), (129, 2600, 64),
                                            (1000, 600, 128), (30000, 400, 256), (65000, 150, 100)])
def test_cuts_match_oracle(engine, L, n_rows, chunk):
    from oracle.oracle import OracleTable

    ds, ts = small_spec(seed=L, n_rows=n_rows, L=L, chunk=chunk)
    ot, et = OracleTable(ts), engine.table(ts)
    knobs = {k: engine.get_tuning(k) for k in ("sparse_max_rows", "mutation_packed", "mutation_coop", "mutation_groups")}
    try:
        gen = ExprGen(ds, seed=L)
        exprs = ["(true)", "(false)"] + [gen.expr(2) for _ in range(4)]
        for sparse, packed, coop, groups in ((-1, 0, 1, 0), (1 << 40, 0, 1, 0), (-1, 1, 1, 0), (-1, 0, 0, 0), (-1, 0, 1, 5),
                                             (n_rows // 3, 0, 1, 0)):
            for key, value in zip(knobs, (sparse, packed, coop, groups)):
                engine.set_tuning(key, value)
            for e in exprs:
                assert np.array_equal(et.mutation_counts(e, "main"), ot.mutation_counts(e, "main")), (e, sparse, packed)
                for p in (0.0, 0.05):
                    assert et.mutations_query(e, "main", p) == ot.mutations(e, "main", p), (e, p, sparse, packed, coop)
                with et.bitmap(e) as b:
                    assert b.cardinality == ot.count(e)
                    assert et.mutations(b, "main", 0.3) == ot.mutations(e, "main", 0.3)
    finally:
        for key, value in knobs.items():
            engine.set_tuning(key, value)
        et.close()
        ot.close()


def test_long_programs(engine):
    """Programs around and past the words passed with the kernel's arguments (768: 96 instructions
    less their ranges and prefetch codes) give the same rows as short ones that mean the same."""
    from oracle.oracle import OracleTable

    ds, ts = small_spec(seed=5, n_rows=900, L=200, chunk=256)
    ot, et = OracleTable(ts), engine.table(ts)
    try:
        for n in (1, 40, 46, 47, 48, 49, 50, 95, 200):
            e = "(or " + " ".join(f"(and (has_mut main {k % 200}) (sym_eq main {(k * 7) % 200} A))" for k in range(n)) + ")"
            assert np.array_equal(et.filter(e), ot.filter(e)), n
            assert et.count(e) == ot.count(e)
            assert et.mutations_query(e, "main", 0.05) == ot.mutations(e, "main", 0.05)
    finally:
        et.close()
        ot.close()


def test_columns_take_turns(engine):
    """Queries alternate between a long and a short column (more and fewer result blocks), with both
    methods: what one leaves for the next is as the next needs it."""
    from oracle.oracle import OracleTable

    ds, ts = small_spec(seed=8, n_rows=700, L=900, chunk=256)
    _, short = small_spec(seed=9, n_rows=700, L=70, chunk=256)
    short.seq_columns[0].name = "short"
    ts.seq_columns.append(short.seq_columns[0])
    ot, et = OracleTable(ts), engine.table(ts)
    saved = engine.get_tuning("sparse_max_rows")
    try:
        gen = ExprGen(ds, seed=3)
        exprs = ["(true)"] + [gen.expr(1) for _ in range(5)]
        for k in range(40):
            column = ("main", "short", "short", "main", "main")[k % 5]
            engine.set_tuning("sparse_max_rows", (-1, 1 << 40, 100)[k % 3])
            e = exprs[k % len(exprs)]
            assert et.mutations_query(e, column, 0.0) == ot.mutations(e, column, 0.0), (k, column, e)
    finally:
        engine.set_tuning("sparse_max_rows", saved)
        et.close()
        ot.close()
