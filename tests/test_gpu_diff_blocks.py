"""The diff of aligned sequences where its kernel's work is cut: rows that start at any byte of an aligned
16, differences and missing runs at the edges of a lane's 16 characters and of a step's 1,024, rows that
differ everywhere, lower case, references with missing positions; an append of 74 MB in one piece, and
appends cut after 2^20 rows whose second piece has more characters than the first or fewer;
the adapted reference at the edges of the blocks of 64 positions that the rule is cut into.  Layouts equal
those of the oracle's diff, uploaded in diff form, byte for byte."""
import numpy as np
import pytest

from test_gpu_ingest import aligned_column, oracle_column

pytestmark = pytest.mark.gpu

SYMBOLS = {0: ("ACGT", "ACGTRYN-acgtnuU", "N"), 1: ("ACDEFGHIKLMNPQRSTVWY", "ACDEFGHIKL*-BZxX", "X")}


def edge_rows(rng, ref: str, alphabet: int, n: int):
    _, chars, missing = SYMBOLS[alphabet]
    L = len(ref)
    edges = [0] + [p for k in (1, 2, 15, 16, 17, 63, 64, 65, 2 * 64) for p in (16 * k - 1, 16 * k, 16 * k + 1) if p < L]
    rows = []
    for i in range(n):
        s = list(ref)
        kind = i % 6
        if kind == 0:  # any length, at any offset
            o = int(rng.integers(0, L))
            m = min(L - o, int(rng.choice([0, 1, 2, 15, 16, 17, 31, 33, 1007, 1008, 1023, 1024, 1025, 1040])))
            rows.append((ref[o:o + m].lower() if i % 4 else ref[o:o + m], o))
            continue
        if kind == 1:  # everything differs
            s = [chars[(chars.index(c) + 1) % 4] if c in chars[:4] else chars[0] for c in s]
        for p in rng.choice(edges, size=4):  # differences and runs at the edges
            if kind == 2:
                s[p] = chars[int(rng.integers(0, len(chars)))]
            if kind == 3:
                e = min(L, p + int(rng.choice([1, 2, 15, 16, 17, 40, 1024, 1100])))
                s[p:e] = (missing if i % 4 else missing.lower()) * (e - p)
        if kind == 4:  # a third of the characters, and a ragged end
            for p in rng.choice(L, size=L // 3, replace=False):
                s[p] = chars[int(rng.integers(0, len(chars)))]
            s = s[:int(rng.integers(1, L + 1))]
        rows.append(("".join(s), 0))
    return rows


@pytest.mark.parametrize("alphabet", [0, 1])
@pytest.mark.parametrize("length", [1, 63, 64, 65, 257, 1024, 2500])
def test_edges(engine, alphabet, length):
    from silo_amd import table

    rng = np.random.default_rng(length + alphabet)
    ref_chars, _, missing = SYMBOLS[alphabet]
    ref = "".join(missing if rng.random() < 0.01 else c for c in rng.choice(list(ref_chars), length))
    rows = edge_rows(rng, ref, alphabet, 180)
    check(engine, table.TableSpec(chunk_sizes=np.array([100, 80], np.uint32)), alphabet, ref, rows, 1, 77)


def test_large_append(engine):
    from silo_amd import table

    rng = np.random.default_rng(5)
    ref = "".join(rng.choice(list("ACGT"), 2500))
    rows = edge_rows(rng, ref, 0, 300)
    copies = 120  # about 74 MB
    sizes = np.array([300 * copies - 1000, 1000], np.uint32)
    check(engine, table.TableSpec(chunk_sizes=sizes), 0, ref, rows, copies, 300 * copies)


@pytest.mark.parametrize("grows", [True, False])
def test_append_of_several_pieces(engine, grows):
    """One append of 2^20 + 30,720 rows: the builder's text buffer goes from one piece to the next, and
    either grows or holds the first piece's characters past the second's end, whose last rows end
    at any byte of an aligned 16."""
    from silo_amd import table

    rng = np.random.default_rng(6 + grows)
    ref = "".join(rng.choice(list("ACGT"), 400))

    def some(lo, hi, n):  # rows of lo .. hi characters somewhere, a few differences and missing runs in each
        rows = []
        for i in range(n):
            m = int(rng.integers(lo, hi + 1))
            o = int(rng.integers(0, 400 - m + 1))
            s = list(ref[o:o + m])
            for p in rng.integers(0, m, size=2 if m else 0):
                s[p] = "ACGTRN-n"[int(rng.integers(0, 8))]
            rows.append((None if i % 97 == 5 else "".join(s), o))
        return rows

    short, long = some(0, 8, 1024), some(300, 400, 1024)
    first, then = (short, long) if grows else (some(9, 40, 1024), short)
    parts = [(first, 1024), (then, 30)]
    n = 1024 * 1054
    sizes = np.array([65536] * (n // 65536) + [n % 65536], np.uint32)
    check_parts(engine, table.TableSpec(chunk_sizes=sizes), 0, ref, parts, n)


def check(engine, spec, alphabet, ref, rows, copies, batch_rows):
    check_parts(engine, spec, alphabet, ref, [(rows, copies)], batch_rows)


def check_parts(engine, spec, alphabet, ref, parts, batch_rows):
    """The rows of each part, as many times as it says."""
    from silo_amd import table

    columns = [(oracle_column("main", alphabet, ref, rows), copies) for rows, copies in parts]

    def times(name):
        return np.concatenate([np.tile(getattr(c, name), copies) for c, copies in columns])

    def ptr_times(name):
        step = np.concatenate([np.tile(np.diff(getattr(c, name).astype(np.int64)), copies) for c, copies in columns])
        return np.concatenate([[0], np.cumsum(step)]).astype(np.uint64)

    host = table.SeqColumnData("main", alphabet, columns[0][0].reference, *map(times, ("is_null", "cov_start", "cov_end")),
                               ptr_times("mut_ptr"), times("mut_pos"), times("mut_sym"), ptr_times("nrun_ptr"),
                               times("nrun_start"), times("nrun_end"))
    rows = [row for part, copies in parts for row in part * copies]
    spec.seq_columns = [aligned_column("main", alphabet, ref, rows, batch_rows)]
    built = engine.table(spec)
    spec.seq_columns = [host]
    engine.set_tuning("index_build_device", 0)
    try:
        want = engine.table(spec)
    finally:
        engine.set_tuning("index_build_device", 1)
    try:
        assert np.array_equal(built.local_reference("main"), want.local_reference("main"))
        assert np.array_equal(built.mutation_counts("(true)", "main"), want.mutation_counts("(true)", "main"))
        assert built.digest("main") == want.digest("main")
    finally:
        built.close()
        want.close()
