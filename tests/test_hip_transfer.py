"""Rows and variables through the engine's host transfers: single-slot and pipelined sizes, element
counts that allow vector accesses and ones that do not, float32 and float16 streams.  What is
written must come back bit for bit (values that the storage types hold exactly)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine(S, n_entity, n_relation, D, F, rw, dtype, shared=False):
    import poplar_kge as kge

    s = kge.Settings.create_demo()
    s.seed = 3
    s.model.n_shard, s.model.n_entity, s.model.n_relation_type = S, n_entity, n_relation
    s.model.embedding_size, s.model.entity_feature_size = D, F
    s.execution.dtype, s.execution.rw_batch_size, s.execution.shared_table = dtype, rw, shared
    return kge.Engine(s.prepare(), np.full(S, n_entity - 1))


# (S, n_entity, D, F, rows per call): one element, an odd row, less than a slot, a slot and a row,
# several times round the slots (a slot holds 2 MiB)
@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("S,n_entity,D,F,rw", [(1, 2, 1, 0, 1), (2, 45, 7, 4, 16), (2, 300, 20, 8, 128),
                                               (1, 683, 256, 0, 683), (4, 1500, 256, 768, 512)])
def test_rows_round_trip(S, n_entity, D, F, rw, dtype):
    engine = _engine(S, n_entity, S, D, F, rw, dtype)
    rng = np.random.default_rng(5)
    W = 3 * D + F
    rows = rng.integers(-2048, 2048, (S, n_entity, W)).astype(np.float32) / 256  # exact in float16
    for offset in reversed(range(0, n_entity, rw)):  # the last chunk's overflow lands on row 0 first
        chunk = np.zeros((S, rw, W), np.float32)
        live = rows[:, offset:offset + rw]
        chunk[:, :live.shape[1]] = live
        engine.write_entity_raw(offset, chunk)
    for offset in range(0, n_entity, rw):
        np.testing.assert_array_equal(engine.read_entity(offset), rows[:, offset:offset + rw])
    got = engine.read_entity_all()
    assert got.dtype == np.dtype(dtype)
    np.testing.assert_array_equal(got, rows)
    # features as a float16 / float32 stream; embeddings are the seeded generator's, moments zero
    if F:
        feat = rng.integers(-2048, 2048, (S, rw, F)).astype(dtype) / 256
        engine.write_entity(0, feat.astype(dtype))
        live = min(rw, n_entity)
        again = engine.read_entity(0)
        np.testing.assert_array_equal(again[:, 1:live, 3 * D:], feat[:, 1:live])
        assert not again[:, 1:live, D:3 * D].any()
        engine.write_entity(0, feat.astype(dtype))
        np.testing.assert_array_equal(engine.read_entity(0)[:, 1:live, :D], again[:, 1:live, :D])


def test_shared_table_reads_the_same_rows_for_every_shard():
    engine = _engine(3, 50, 5, 6, 0, 64, "float32", shared=True)
    engine.write_entity(0, np.zeros((3, 64, 0), np.float32))
    got = engine.read_entity_all()
    assert got.shape == (3, 50, 18)
    np.testing.assert_array_equal(got, engine.read_entity(0))
    np.testing.assert_array_equal(got[0], got[2])


# widths with and without padding columns; one row, one slot, several slots
@pytest.mark.parametrize("n_relation,D", [(1, 3), (12, 8), (700, 5), (2049, 256), (9001, 255)])
def test_variables_round_trip(n_relation, D):
    engine = _engine(1, 10, n_relation, D, 0, 4, "float32")
    rng = np.random.default_rng(6)
    for name in ("relation_embedding", "relation_embedding/adam_m", "relation_embedding/adam_v"):
        value = rng.normal(size=(n_relation, D)).astype(np.float32)
        engine.write_variable(name, value)
        np.testing.assert_array_equal(engine.read_variable(name), value)
