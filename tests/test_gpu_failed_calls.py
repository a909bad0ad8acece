"""Calls after one that failed answer as if it had not been made."""
import ctypes

import numpy as np
import pytest

from helpers import bitset_table, small_spec

pytestmark = pytest.mark.gpu


def answers(et, country):
    """Every action on a table, single and batched."""
    expr = f'(and (str_eq country "{country}") (not (has_mut main 17)))'
    out = [et.count(expr), et.filter(expr).tolist(), et.mutation_counts(expr, "main").tolist()]
    for p in (0.0, 0.05):
        out.append(et.mutations_query(expr, "main", p))
    for dims in ([], ["country"], ["main@20", "country"]):
        out.append(et.aggregate(expr, dims))
    out.append(et.batch([{"filter": expr, "action": "mutations", "column": "main", "min_proportion": 0.05},
                         {"filter": expr, "action": "aggregate", "dims": ["country"]},
                         {"filter": expr, "action": "count"}]))
    return out


def test_failed_allocation(engine):
    """A device allocation larger than any GPU's memory fails its own call only: the kernels launched
    next, each action's first and last, are not taken for failed ones."""
    from silo_amd.engine import EngineError

    ds, ts = small_spec(seed=91, n_rows=9000, L=400, chunk=4096)
    et = engine.table(ts)
    try:
        country = ds.country_names[0]
        want = answers(et, country)
        calls = [lambda: et.count("(true)"), lambda: et.mutation_counts("(true)", "main").sum(),
                 lambda: et.mutations_query("(true)", "main", 0.05), lambda: et.aggregate("(true)", ["country"]),
                 lambda: et.batch([{"filter": "(true)", "action": "count"}])]
        for call in calls:
            expected = call()
            with pytest.raises(EngineError) as err:
                engine.read_bandwidth(1 << 50, 1)
            assert err.value.status == "RDB_ENOMEM"
            assert np.array_equal(call(), expected) if not isinstance(expected, list) else call() == expected
        assert answers(et, country) == want
    finally:
        et.close()


@pytest.mark.parametrize("knobs", [{}, {"mutation_packed": 1}, {"mutation_coop": 0}, {"sparse_max_rows": 1 << 40}])
def test_failure_between_kernels(engine, knobs):
    """A query that fails after its counting kernels leaves its sums in the table's scratch: the next
    queries, of the same action and of the others, start from zero all the same, and twice in a row
    (the totals of two Mutations queries take turns)."""
    from silo_amd.engine import EngineError

    ds, ts = small_spec(seed=92, n_rows=9000, L=400, chunk=4096)
    saved = {k: engine.get_tuning(k) for k in knobs}
    et = engine.table(ts)
    try:
        for k, v in knobs.items():
            engine.set_tuning(k, v)
        country = ds.country_names[0]
        want = answers(et, country)
        for call in (lambda: et.mutations_query("(true)", "main", 0.05), lambda: et.mutation_counts("(true)", "main"),
                     lambda: et.aggregate("(true)", ["country"]), lambda: et.aggregate("(true)", ["main@20", "country"])):
            for n in (1, 2):  # fails at once, or after one that succeeds
                engine.set_tuning("query_fail", n)
                for _ in range(n - 1):
                    call()
                with pytest.raises(EngineError) as err:
                    call()
                assert err.value.status == "RDB_EDEVICE" and engine.get_tuning("query_fail") == 0
                if n == 2:  # two failures in a row
                    engine.set_tuning("query_fail", 1)
                    with pytest.raises(EngineError):
                        call()
                assert answers(et, country) == want
                assert answers(et, country) == want
    finally:
        engine.set_tuning("query_fail", 0)
        for k, v in saved.items():
            engine.set_tuning(k, v)
        et.close()


@pytest.mark.parametrize("knobs", [{"sparse_max_rows": 1 << 40}, {"batch_shared_scan": 1}, {"batch_shared_scan": 2}])
def test_lane_job_failure_between_kernels(engine, knobs):
    """A lane job launched kernel by kernel that fails after its Mutations were counted leaves nothing
    to the next job: not the sparse counts, not the shared scans' sums of bitset containers."""
    from silo_amd.engine import EngineError

    spec, _, _ = bitset_table()
    knobs = dict(knobs, batch_graphs=0, batch_lanes=1, batch_max_queries=8)
    saved = {k: engine.get_tuning(k) for k in knobs}
    et = engine.table(spec)
    try:
        for k, v in knobs.items():
            engine.set_tuning(k, v)
        queries = [{"filter": f, "action": "mutations", "column": "main", "min_proportion": 0.0}
                   for f in ("(true)", "(date_between date 18262 18263)", '(str_eq country "c1")')]
        want = [et.mutations_query(q["filter"], "main", 0.0) for q in queries]
        assert et.batch(queries) == want
        engine.set_tuning("batch_fail_job", 1)
        with pytest.raises(EngineError) as err:
            et.batch(queries)
        assert err.value.status == "RDB_EDEVICE" and engine.get_tuning("batch_fail_job") == 0
        assert et.batch(queries) == want
        assert et.batch(queries) == want
    finally:
        engine.set_tuning("batch_fail_job", 0)
        for k, v in saved.items():
            engine.set_tuning(k, v)
        et.close()
