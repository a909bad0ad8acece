"""The diff of aligned sequences where its kernel's work is cut: rows that start at any byte of an aligned
16, differences and missing runs at the edges of a lane's 16 characters and of a step's 1,024, rows that
differ everywhere, lower case, references with missing positions; an append of 74 MB;
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


def check(engine, spec, alphabet, ref, rows, copies, batch_rows):
    from silo_amd import table

    c = oracle_column("main", alphabet, ref, rows)
    # the rows `copies` times
    def times(ptr):
        step = np.diff(ptr.astype(np.int64))
        return np.concatenate([[0], np.cumsum(np.tile(step, copies))]).astype(np.uint64)

    host = table.SeqColumnData("main", alphabet, c.reference, *[np.tile(a, copies) for a in (c.is_null, c.cov_start, c.cov_end)],
                               times(c.mut_ptr), np.tile(c.mut_pos, copies), np.tile(c.mut_sym, copies), times(c.nrun_ptr),
                               np.tile(c.nrun_start, copies), np.tile(c.nrun_end, copies))
    spec.seq_columns = [aligned_column("main", alphabet, ref, rows * copies, batch_rows)]
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
