"""The framework's performance cases: program runs of the training step, prediction sweeps and bulk
entity transfers through ``poplar_kge.Engine``, from the demo preset to the 22.8M-row table.

A training case is one program run (``train_step_loop`` on the host index arrays a batch sampler
hands over) followed by what a program keeps an eye on between program runs: the relation table
and the first ``rw`` rows of every shard, moments and features included.  Under the power law these
are the rows the run updated most often.
"""

import math
import os
import sys

import numpy as np
import torch  # noqa: F401  (brings the HIP runtime that the engine's library binds to)

sys.path.insert(0, os.path.join(os.getcwd(), "distributed-kge-poplar_amd"))

import poplar_kge as kge  # noqa: E402

ZIPF = 1.1  # exponent of the ids' power law: id = rank, as in the framework's synthetic workloads


def _train(name, **kw):
    case = dict(name=name, kind="train", score_fn="TransE", distance_fn="L2", loss="logsigmoid", S=1, n_entity=10_000,
                n_relation=1387, D=256, F=0, B=256, A=64, steps=20, dtype="float32", embedding_dtype="", feature_dtype="",
                scoring_dtype="", shared=True, feature_reg=0.0, layout="raw", uniform=False, lr=2e-5, gamma=10.0, rw=16)
    case.update(kw)
    return case


def _predict(name, **kw):
    case = dict(name=name, kind="predict", score_fn="TransE", distance_fn="L2", S=1, n_entity=1_000_000, n_relation=1000,
                D=256, F=0, queries=128, n_best=100, dtype="float32")
    case.update(kw)
    return case


def _entity_io(name, **kw):
    case = dict(name=name, kind="entity_io", S=16, n_entity=2048, D=256, F=768, rw=512, dtype="float16")
    case.update(kw)
    return case


def listed():
    return [
        # the demo preset: the first thing a new user runs, and what a test suite runs all day
        _train("demo_transe_l1", distance_fn="L1", S=2, n_entity=90, n_relation=12, D=8, F=6, B=6, A=5, steps=5, shared=False,
               layout="sampler", uniform=True, lr=0.1, gamma=2.0, rw=45),
        # a small graph in one block: 10 k entities, uniform ids
        _train("small_transe_l2", n_relation=50, D=64, A=64, uniform=True, rw=256),
        # a mid-size graph: 1M entities, 32 blocks of 256 positives against 256 shared tails
        _train("transe_l2_1m", S=32, n_entity=1_000_000, n_relation=1000, A=8, steps=100),
        # the headline: 22.8M entities, 64 blocks of 256 positives against 512 shared tails
        _train("transe_l2_22m", S=64, n_entity=22_800_000, A=8, steps=100, rw=32),
        # the same blocks with the L1 distance, on a table of 4M rows
        _train("transe_l1_4m", distance_fn="L1", S=64, n_entity=4_000_000, A=8, steps=100, rw=32),
        # one wide DistMult block with projected 768-dim features, softmax and bfloat16 scoring
        _train("distmult_features_bf16", score_fn="DistMult", distance_fn="MatMul", loss="softmax", n_entity=500_000, D=512,
               F=768, B=8192, A=2048, feature_dtype="float16", scoring_dtype="bfloat16", rw=1024),
        # bfloat16 embeddings with float32 moments, for tables that would not fit otherwise
        _train("transe_l2_bf16_rows", S=32, n_entity=8_000_000, B=512, A=16, steps=50, embedding_dtype="bfloat16", rw=32),
        # the WikiKG90Mv2 preset: 16 shards, L1, 768-dim float16 features, softmax, feature regulariser
        _train("wikikg_preset_transe_l1", distance_fn="L1", loss="softmax", S=16, n_entity=20_000, n_relation=1392, F=768,
               B=512, A=96, feature_dtype="float16", shared=False, feature_reg=1e-6, layout="sampler", rw=64),
        # the reference's published run: RotatE, float16 storage, 16 shards, 50 steps per program run
        _train("wikikg_rotate_fp16", score_fn="RotatE", S=16, n_entity=20_000, n_relation=1392, F=768, B=256, A=96, steps=50,
               dtype="float16", shared=False, layout="sampler", rw=64),
        # sizes that fit no tile: ComplEx, D = 100, 4 shards of 200 positives against 268 shared tails
        _train("complex_ragged", score_fn="ComplEx", distance_fn="MatMul", loss="softmax", S=4, n_entity=50_000,
               n_relation=536, D=100, B=200, A=67, shared=False, layout="sampler", rw=256),
        # validation: 128 queries against every row of a 1M-row table, the 100 best
        _predict("predict_l2_1m"),
        # writing and reading back a table of float16 rows with features, in the preset's chunks
        _entity_io("entity_io_fp16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_train(rng):
    while True:
        score_fn = rng.choice(["TransE", "TransE", "TransE", "RotatE", "DistMult", "ComplEx"])
        distance_fn = {"TransE": rng.choice(["L1", "L2"]), "RotatE": rng.choice(["L1", "L2"]), "DistMult": "MatMul",
                       "ComplEx": rng.choice(["MatMul", "L2"])}[score_fn]
        sampler = rng.random() < 0.5
        S = rng.choice([1, 2, 4, 8, 16]) if sampler else _log_int(rng, 1, 64)
        D = rng.choice([64, 128, 256, 256, 512]) if rng.random() < 0.6 else _log_int(rng, 8, 512)
        D += D % 2 if score_fn in ("RotatE", "ComplEx") else 0
        F = 0 if rng.random() < 0.6 else rng.choice([64, 128, 768])
        T = rng.choice([128, 256, 512, 1536]) if rng.random() < 0.5 else _log_int(rng, 10, 2048)
        A = max(2, T // S)
        B = rng.choice([128, 256, 512]) if rng.random() < 0.5 else _log_int(rng, 6, 4096)
        if sampler:
            B = S * max(1, min(B // S, A - 1))
        dtype = rng.choice(["float32", "float32", "float16"])
        scoring = "bfloat16" if score_fn == "DistMult" and rng.random() < 0.3 else ""
        steps, n_entity = _log_int(rng, 5, 100), _log_int(rng, 1_000, 4_000_000 // S if not F else 160_000 // S)
        R = S * (B + S * A)
        if steps * S * B * S * A * D > 8e9 or steps * R * F * D > 5e10 or R > 60_000 or steps * R > 3_000_000 or S * A < 2:
            continue
        # float32 tables in earnest hold 16-bit features; bfloat16 rows serve tables that would not fit
        return _train("", score_fn=score_fn, distance_fn=distance_fn, loss=rng.choice(["logsigmoid", "logsigmoid", "softmax"]),
                      S=S, n_entity=n_entity, n_relation=S * max(1, _log_int(rng, 10, 1400) // S), D=D, F=F, B=B, A=A,
                      steps=steps, dtype=dtype, feature_dtype="float16" if F and dtype == "float32" else "",
                      embedding_dtype="bfloat16" if dtype == "float32" and not F and rng.random() < 0.2 else "",
                      scoring_dtype=scoring, shared=not sampler, layout="sampler" if sampler else "raw",
                      feature_reg=1e-6 if sampler and F and not scoring and rng.random() < 0.5 else 0.0,
                      uniform=rng.random() < 0.3, rw=max(1, min(n_entity, 1024 // S)))


def draw(rng):
    """Another case of the listed ranges, not larger than the largest listed one."""
    pick = rng.random()
    if pick < 0.75:
        case = _draw_train(rng)
    elif pick < 0.9:
        score_fn = rng.choice(["TransE", "TransE", "RotatE", "DistMult"])
        S, F = rng.choice([1, 2, 4]), rng.choice([0, 0, 0, 768])
        case = _predict("", score_fn=score_fn, distance_fn="MatMul" if score_fn == "DistMult" else rng.choice(["L1", "L2"]),
                        S=S, n_entity=_log_int(rng, 2_000, 1_000_000 if not F else 100_000) // S,
                        n_relation=S * (_log_int(rng, 10, 1400) // S + 1), D=2 * _log_int(rng, 32, 128), F=F,
                        queries=_log_int(rng, 4, 128), n_best=rng.choice([10, 11, 100]), dtype=rng.choice(["float32", "float16"]))
    else:
        S, F, D = rng.choice([1, 2, 4, 16]), rng.choice([0, 64, 768]), 4 * _log_int(rng, 4, 64)
        case = _entity_io("", S=S, F=F, D=D, n_entity=_log_int(rng, 64, 32_768) // S, rw=_log_int(rng, 32, 512),
                          dtype=rng.choice(["float32", "float16"]))
    del case["name"]
    return case


# ---- sizes -----------------------------------------------------------------------------------------

def _bytes_of(dtype):
    return 4 if dtype == "float32" else 2


def _row_bytes(c):
    """(embedding, both moments, features) bytes of a table row."""
    emb = _bytes_of(c.get("embedding_dtype") or c["dtype"])
    feat = _bytes_of(c.get("feature_dtype") or c["dtype"])
    return emb * c["D"], 2 * _bytes_of(c["dtype"]) * c["D"], feat * c["F"]


def _distinct(n_rows, n, uniform):
    """Expected distinct ids among n draws from ids 1 .. n_rows - 1."""
    m = n_rows - 1
    if uniform:
        return m * -math.expm1(n * math.log1p(-1.0 / m)) if m > 1 else 1.0
    edge = np.unique(np.floor(np.geomspace(1, m + 1, 4096))).astype(np.float64)  # ids [edge, next edge) together
    below = (1 - edge ** (1 - ZIPF)) / (1 - float(m + 1) ** (1 - ZIPF))
    width = np.diff(edge)
    p = np.minimum(np.diff(below) / width, 1.0)
    with np.errstate(divide="ignore"):
        return float(np.sum(width * -np.expm1(n * np.log1p(-p))))


def _counts(c):
    """Expected per step: distinct table rows, distinct tails per block."""
    S, B, T = c["S"], c["B"], c["S"] * c["A"]
    if c["layout"] == "sampler":  # per shard: B heads and B true tails by popularity, the rest uniform
        pop, neg = 2 * B, S * (c["A"] - B // S)
        rows = S * min(c["n_entity"] - 1, _distinct(c["n_entity"], pop, c["uniform"]) + _distinct(c["n_entity"], neg, True))
        P = B // S
        tails = S * min(c["n_entity"] - 1, _distinct(c["n_entity"], P, c["uniform"]) + _distinct(c["n_entity"], c["A"] - P, True))
        return rows, min(T, tails)
    return _distinct(c["n_entity"], S * (B + T), c["uniform"]), _distinct(c["n_entity"], T, c["uniform"])


def work(case):
    c = case
    emb, mom, feat = _row_bytes(dict(case))
    if c["kind"] == "entity_io":
        rows = c["S"] * c["n_entity"]
        return dict(bytes=float(rows * (2 * feat + (emb + mom) * 2 + feat)), flops=0.0)
    per_pair = 2 if c["distance_fn"] == "MatMul" else 3
    if c["kind"] == "predict":
        rows, Q = c["S"] * (c["n_entity"] - 1), c["S"] * c["queries"]
        return dict(bytes=float(rows * (emb + feat) + Q * c["S"] * c["n_best"] * 8),
                    flops=float(per_pair * rows * Q * c["D"] + 2 * rows * c["F"] * c["D"]))
    rows, tails = _counts(c)
    S, B, D, F = c["S"], c["B"], c["D"], c["F"]
    rel = 4 * c["n_relation"] * (D // 2 if c["score_fn"] == "RotatE" else D)
    step_bytes = (rows * (2 * (emb + mom) + feat) + 4 * (S * (B + S * c["A"]) + S * S * c["A"] + 3 * S * B) + 6 * rel
                  + 24 * F * D)
    step_flops = 3 * per_pair * S * B * tails * D + 4 * rows * F * D
    return dict(bytes=float(c["steps"] * step_bytes), flops=float(c["steps"] * step_flops))


def tolerance(case):
    if case["kind"] == "entity_io":
        return "exact"
    if case["kind"] == "predict":
        return dict(rel=1e-5, max=1e-3, differ=5e-3)  # float32 scores; rows whose scores tie to rounding may swap ranks
    # A program run of Adam steps from zero moments: a gradient element that cancels to rounding moves its
    # parameter by the step size in a direction that rounding decides, and later steps start from there.
    # (The low learning rate, late in the presets' linear decay, keeps that from growing over the steps.)
    if case["scoring_dtype"] == "bfloat16":
        return dict(rel=1e-2, max=0.9)
    if case["distance_fn"] == "L1":  # an L1 gradient is a sum of signs: a difference near zero flips a whole term
        return dict(rel=5e-3 if case["loss"] == "softmax" else 5e-4, max=0.9)
    if case["dtype"] == "float16" or case["embedding_dtype"] == "bfloat16" or case["score_fn"] == "RotatE":
        return dict(rel=5e-4, max=0.1)  # 16-bit storage; RotatE forms its phases' gradient in float16
    return dict(rel=2e-5, max=1e-2)


# ---- a user's program --------------------------------------------------------------------------------

def _ids(rng, n_entity, shape, uniform):
    """Ids 1 .. n_entity - 1, uniform or by the bounded power law (inverse CDF, id = rank)."""
    m = n_entity - 1
    if uniform:
        return rng.integers(1, m + 1, shape, dtype=np.uint32)
    u = rng.random(shape)
    k = (1 - u * (1 - float(m + 1) ** (1 - ZIPF))) ** (1 / (1 - ZIPF))
    return np.clip(k, 1, m).astype(np.uint32)


def _unique_pad(ids):
    """Sorted distinct values of every row padded with 0, and every element's position among them."""
    order = np.argsort(ids, axis=-1, kind="stable")
    srt = np.take_along_axis(ids, order, -1)
    new = np.ones(srt.shape, bool)
    new[..., 1:] = srt[..., 1:] != srt[..., :-1]
    rank = np.cumsum(new, axis=-1, dtype=np.int64) - 1
    padded, slot = np.zeros_like(ids), np.empty(ids.shape, np.uint32)
    np.put_along_axis(padded, rank, srt, -1)
    np.put_along_axis(slot, order, rank.astype(np.uint32), -1)
    return padded, slot


def _batch(c, rng):
    S, B, A, n = c["S"], c["B"], c["A"], c["steps"]
    relation = rng.integers(0, c["n_relation"], (S, n, B), dtype=np.uint32)
    if c["layout"] == "raw":
        # raw ids, repeats included: a block's heads, then the tails its shard contributes
        remote = _ids(rng, c["n_entity"], (S, n, B + S * A), c["uniform"])
        head = np.broadcast_to(np.arange(B, dtype=np.uint32), (S, n, B)).copy()
        a2a = np.broadcast_to((B + np.arange(S * A, dtype=np.uint32)).reshape(S, A), (S, n, S, A)).copy()
        tail = rng.integers(0, S * A, (S, n, B), dtype=np.uint32)
        return kge.Batch(remote=remote, a2a=a2a, head=head, relation=relation, tail=tail)
    # the batch sampler's layout: distinct rows per shard, P true tails and A - P uniform negatives to every shard
    P = B // S
    ids = np.concatenate([_ids(rng, c["n_entity"], (S, n, 2 * B), c["uniform"]),
                          _ids(rng, c["n_entity"], (S, n, S * (A - P)), True)], axis=2)
    remote, slot = _unique_pad(ids)
    a2a = np.concatenate([slot[:, :, B:2 * B].reshape(S, n, S, P), slot[:, :, 2 * B:].reshape(S, n, S, A - P)], axis=3)
    position = (A * np.arange(S)[:, None] + np.arange(P)[None, :]).reshape(B).astype(np.uint32)
    return kge.Batch(remote=remote, a2a=np.ascontiguousarray(a2a), head=np.ascontiguousarray(slot[:, :, :B]),
                     relation=relation, tail=np.ascontiguousarray(np.broadcast_to(position, (S, n, B))))


def _engine(c, seed, rw):
    s = kge.Settings.create_demo()
    s.seed = int(seed)
    m, d, t, e = s.model, s.data, s.training, s.execution
    m.score_fn, m.distance_fn = c.get("score_fn", "TransE"), c.get("distance_fn", "L2")
    m.n_shard, m.n_entity, m.n_relation_type = c["S"], c["n_entity"], c.get("n_relation", c["S"])
    m.embedding_size, m.entity_feature_size, m.gamma = c["D"], c["F"], c.get("gamma", 10.0)
    m.init_scale = math.sqrt(c["D"])  # embeddings ~ N(0, 1 / sqrt(D))
    d.batch_size, d.a2a_size = c.get("B", 2), c.get("A", 2)
    t.learning_rate = c.get("lr", 1e-3)
    t.loss = kge.SoftmaxLoss(correction_weight=1.0) if c.get("loss") == "softmax" else kge.LogSigmoidLoss()
    t.feature_regularisation = kge.NormRegularisation(power=3.0, weight=c.get("feature_reg", 0.0))
    e.dtype, e.shared_table = c["dtype"], c.get("shared", False)
    e.embedding_dtype, e.feature_dtype = c.get("embedding_dtype") or None, c.get("feature_dtype") or None
    e.scoring_dtype = c.get("scoring_dtype") or None
    e.train_steps_per_program_run, e.rw_batch_size = c.get("steps", 1), rw
    e.predict_hr_batch_size, e.predict_n_best = c.get("queries", 2), c.get("n_best", 10)
    s.prepare()
    return kge.Engine(s, np.full(c["S"], c["n_entity"] - 1)), s


def _padded(chunk, live):
    """A chunk of rows with zeros behind the ``live`` ones: those go to the padding row, in no order."""
    if live < chunk.shape[1]:
        chunk = chunk.copy()
        chunk[:, live:] = 0
    return chunk


def _write_rows(engine, s, shared, rng):
    """Random-normal rows and N(0, 1) features over the whole table."""
    m, rw = s.model, s.execution.rw_batch_size
    feat = rng.standard_normal(s.entity_data_w_shape, dtype=np.float32).astype(s.execution.dtype)
    if not shared:
        for offset in range(0, m.n_entity, rw):
            engine.write_entity(offset, _padded(feat, m.n_entity - offset))
        return
    # a shared table: the shards' index rows cover different ranges of it
    feat = feat.view(np.int16) if feat.dtype == np.float16 else feat
    per_call = m.n_shard * rw
    for offset in range(0, m.n_entity, per_call):
        idx = np.arange(offset, offset + per_call, dtype=np.int64)
        idx[idx >= m.n_entity] = 0
        engine.engine.run("write_entity", dict(write_indices=idx.astype(np.uint32).reshape(m.n_shard, rw), write_features=feat))
    idx = np.zeros((m.n_shard, rw), np.uint32)  # row 0 last: what the final call's overflow left there goes
    engine.engine.run("write_entity", dict(write_indices=idx, write_features=np.zeros_like(feat)))
    engine.uninitialized_entity_data[:] = False


def prepare(case, seed):
    c, rng = case, np.random.default_rng(seed)
    if c["kind"] == "entity_io":
        engine, s = _engine(c, seed, c["rw"])
        chunks = []
        block = rng.standard_normal(s.entity_data_w_shape, dtype=np.float32).astype(c["dtype"])
        for k, offset in enumerate(range(0, c["n_entity"], c["rw"])):
            chunks.append((offset, _padded(np.roll(block, k, axis=1), c["n_entity"] - offset)))
        return dict(case=c, engine=engine, chunks=chunks)
    engine, s = _engine(c, seed, c.get("rw", 4096))
    engine.initialise_variables()
    _write_rows(engine, s, c.get("shared", False), rng)
    if c["kind"] == "predict":
        n, S = c["queries"] * c["S"], c["S"]
        query = np.stack([np.arange(n) % S, _ids(rng, c["n_entity"], n, False), rng.integers(0, c["n_relation"], n)], axis=1)
        return dict(case=c, engine=engine, query=query.astype(np.uint32))
    return dict(case=c, engine=engine, batch=_batch(c, rng))


def run(state):
    kind, engine = state["case"]["kind"], state["engine"]
    if kind == "entity_io":
        for offset, features in state["chunks"]:
            engine.write_entity(offset, features)
        return engine.read_entity_all()
    if kind == "predict":
        found = engine.predict(state["query"])
        return dict(shard_idx=found.shard_idx, score=found.score)
    loss, learning_rate = engine.train_step_loop(state["batch"])
    return dict(loss=loss, learning_rate=learning_rate, relation_embedding=engine.read_variable("relation_embedding"),
                entity_data=engine.read_entity(0))
