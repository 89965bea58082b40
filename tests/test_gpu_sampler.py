"""GPU sampling and the `llama` command drop-in, through the C ABI, against
fixtures the compiled reference wrote (tests/golden/gen_golden.c `sample`):
sample_token draws and RNG states (sampler.c:54-143), the device generation
loop (q_llama_generate) and the qllama-cli binary (main.c:624-671) on an LLMQ
checkpoint.  Bar: tokens and RNG states bit-exact."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle_lib as O
import qlib
from conftest import ROOT, golden_json

pytestmark = pytest.mark.gpu
S = golden_json("sample")
TINY = [32000, 288, 6, 6, 2, 48, 768, 256]
CLI = os.path.join(ROOT, "llm-project_amd", "qllama-cli")


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def Q():
    q = qlib.load()
    assert q.lib().qllama_device_count() > 0, "no GPU visible to the HIP library"
    return q


def test_sample_token_matches_reference(Q):
    for ci, c in enumerate(S["sample_cases"]):
        log(f"sample case {ci}: V={c['V']} kind={c['kind']} t={c['t']} k={c['k']} p={c['p']}")
        row = O.sample_row(c["V"], c["tid"], c["sigma"], c["kind"]).reshape(1, -1)
        rng = Q.rng_create(c["seed"])
        toks = [Q.sample_token(row, c["t"], c["k"], c["p"], rng) for _ in range(8)]
        assert toks == c["tokens"], ci
        assert rng.state == int(c["state"], 16), ci


@pytest.mark.parametrize("V,k", [(131072, 64), (131072, 65), (131073, 40), (131073, 64), (50, 60), (50, 10),
                                 (1025, 64), (5000, 1)])
def test_sample_token_paths_match_oracle(Q, V, k):
    """Both device paths (blockwise top-k when top_k <= 64 and V <= 131072, the
    full radix sort otherwise) against the oracle, at and around the switch."""
    for kind in (0, 1):
        row = O.sample_row(V, 40 + kind, 1.0, kind)
        rng = Q.rng_create(11)
        st = O.rng_create(11)
        for _ in range(6):
            t = Q.sample_token(row.reshape(1, -1), 0.9, k, 0.97, rng)
            r, st = O.sample_token(row, 0.9, k, 0.97, st)
            assert t == r and rng.state == st, (V, k, kind)


@pytest.mark.parametrize("V,k,p,kind", [
    (1023, 40, 0.95, 0), (1024, 40, 1.0, 1), (4097, 64, 0.9, 0),          # fewer groups than k, one slice and its edges
    (32000, 40, 0.95, 1), (70000, 1, 0.9, 0),                             # quarter-slice and slice maxima
    (262144, 64, 1.0, 0), (262145, 64, 0.95, 0),                          # the split sum's widest vocabulary, and past it
    (20000, 65, 0.9999, 0), (20000, 0, 1.0, 0), (20000, 0, 0.6, 1), (20000, 200, 1.0, 1)])   # kept lists over a wave
def test_sample_token_split_sum_and_search_match_oracle(Q, V, k, p, kind):
    """The sum over classified slices, the top-k bound from group maxima and the
    search over the kept running sums, at the edges of each: tokens and rng states
    of the oracle, over rows of several spreads and many equal logits (kind 1)."""
    for tid, sigma, t in ((70, 0.3, 1.0), (71, 2.5, 0.8), (72, 8.0, 0.7)):
        row = O.sample_row(V, tid, sigma, kind)
        rng = Q.rng_create(tid)
        st = O.rng_create(tid)
        for _ in range(5):
            g = Q.sample_token(row.reshape(1, -1), t, k, p, rng)
            r, st = O.sample_token(row, t, k, p, st)
            assert g == r and rng.state == st, (V, k, p, tid)


def test_sample_argmax_first_index(Q):
    for tid in range(4):
        row = O.sample_row(128256 if tid % 2 else 32000, 30 + tid, 1.0, 1).reshape(1, -1)
        assert Q.sample_argmax(row) == int(np.argmax(row[0]))
    flat = np.full((1, 5000), -np.inf, np.float32)
    assert Q.sample_argmax(flat) == 0                     # sampler.c:13-14: r[0] when nothing is larger
    two = np.zeros((2, 300), np.float32)
    two[1, 7] = two[1, 250] = 3.0
    assert Q.sample_argmax(two, row=1) == 7


def test_generate_matches_reference_cli_loop(Q):
    cli = S["cli"]
    m = Q.Model.synth(TINY, 10000.0, seed=cli["seed"])
    try:
        rng = Q.rng_create(1234)
        for li, line in enumerate(cli["lines"]):
            log(f"generate line {li}: prompt {len(line['prompt'])}")
            m.reset(0)
            m.prefill(line["prompt"], want_logits=False)
            gen = m.generate(cli["n_new"], 0.8, 40, 0.95, rng)
            assert gen == line["gen"], li
            assert m.pos == len(line["prompt"]) + cli["n_new"]
    finally:
        m.close()


def test_generate_in_pieces_equals_one_call(Q):
    """Generation split over several calls (and decode steps replayed for a short
    prompt) draws the same tokens as one call."""
    m = Q.Model.synth(TINY, 10000.0, seed=1234)
    try:
        prompt = O.prompt(9, 55, TINY[0])
        m.prefill(prompt, want_logits=False)
        a = m.generate(24, 1.1, 0, 0.9, Q.rng_create(5))
        m.reset(0)
        m.prefill(prompt, want_logits=False)
        r = Q.rng_create(5)
        b = m.generate(10, 1.1, 0, 0.9, r) + m.generate(1, 1.1, 0, 0.9, r) + m.generate(13, 1.1, 0, 0.9, r)
        assert a == b
        # top-k 0 sorts the whole vocabulary (the library's radix sort, captured in
        # the sampled step's graph): the oracle's draws
        ref = O.Model(TINY, 10000.0, seed=1234)
        try:
            for t in prompt:
                lg = ref.step(t)
            st = O.rng_create(5)
            c = []
            for _ in range(24):
                t, st = O.sample_token(lg, 1.1, 0, 0.9, st)
                c.append(t)
                lg = ref.step(t)
            assert a == c
        finally:
            ref.close()
        # the same through the captured sampled step (top-k path), with a change of
        # parameters in between (a second capture) and back
        m.reset(0)
        m.prefill(prompt, want_logits=False)
        a = m.generate(24, 0.8, 40, 0.95, Q.rng_create(6))
        m.reset(0)
        m.prefill(prompt, want_logits=False)
        r = Q.rng_create(6)
        b = m.generate(7, 0.8, 40, 0.95, r)
        b += m.generate(5, 0.8, 40, 0.95, r)
        b += m.generate(12, 0.8, 40, 0.95, r)
        assert a == b
        # oracle: the same draws from the oracle's decode steps and sampler
        ref = O.Model(TINY, 10000.0, seed=1234)
        try:
            for t in prompt:
                lg = ref.step(t)
            st = O.rng_create(6)
            c = []
            for _ in range(24):
                t, st = O.sample_token(lg, 0.8, 40, 0.95, st)
                c.append(t)
                lg = ref.step(t)
            assert a == c
        finally:
            ref.close()
        # greedy through the sampler path equals the decode graph's argmax
        m.reset(0)
        m.prefill(prompt, want_logits=False)
        g1 = m.generate(12, 0.0, 40, 0.95, Q.rng_create(1))
        m.reset(0)
        logits = m.prefill(prompt)
        g2 = m.generate_greedy(int(np.argmax(logits)), 11)
        assert g1 == [int(np.argmax(logits))] + g2
    finally:
        m.close()


def test_llmq_load_matches_generator(Q, tmp_path):
    ref = O.Model(TINY, 10000.0, seed=1234)
    try:
        path = str(tmp_path / "tiny.llmq")
        O.write_llmq(ref, path)
        m = Q.Model.load(path)
        try:
            assert m.hash() == ref.hash()
        finally:
            m.close()
    finally:
        ref.close()


def test_cli_matches_reference_llama_command(Q, tmp_path):
    assert os.path.exists(CLI), "qllama-cli is not built (make -C llm-project_amd)"
    cli = S["cli"]
    ref = O.Model(TINY, 10000.0, seed=cli["seed"])
    try:
        path = str(tmp_path / "tiny.llmq")
        O.write_llmq(ref, path)
    finally:
        ref.close()
    lines = cli["lines"]
    stdin = "".join(" ".join(str(t) for t in ln["prompt"]) + "\n" for ln in lines)
    stdin = "﻿" + stdin + "\n" + "5 -3 99999\n"          # BOM, an empty line, out-of-range ids
    expect = []
    for ln in lines:
        expect += [f"t {t}" for t in ln["gen"]]
        expect.append("gen: " + " ".join(str(t) for t in ln["prompt"] + ln["gen"]))
    log("running qllama-cli")
    out = subprocess.run([CLI, "llama", path, str(cli["n_new"])], input=stdin.encode(), capture_output=True,
                         timeout=120)
    assert out.returncode == 0, out.stderr.decode()
    got = out.stdout.decode().splitlines()
    assert got[:len(expect)] == expect
    # the last line (id 5 alone after two skips) continues the same generator
    assert got[len(expect) + cli["n_new"]].startswith("gen: 5 ")
    assert "skip out-of-range id -3" in out.stderr.decode()
    assert "skip out-of-range id 99999" in out.stderr.decode()


def test_save_load_round_trip_and_truncation(Q, tmp_path, capfd):
    """q_llama_model_save writes what the loader (mapped file, staged uploads)
    reads back; a file cut short inside the weights is refused like
    llama.c:650-654."""
    m = Q.Model.synth([1000, 256, 2, 4, 2, 64, 512, 128], 10000.0, seed=9, tied=True)
    try:
        path = tmp_path / "m.llmq"
        m.save(str(path))
        m2 = Q.Model.load(str(path))
        try:
            assert m2.hash() == m.hash()
            ids = O.prompt(20, 3, 1000)
            a = m.prefill(ids).copy()
            b = m2.prefill(ids).copy()
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        finally:
            m2.close()
        data = path.read_bytes()
        cut = tmp_path / "cut.llmq"
        cut.write_bytes(data[:len(data) - 100])
        capfd.readouterr()
        mm = Q.QLlamaModel()
        assert Q.lib().q_llama_model_load(os.fsencode(str(cut)), mm) != 0
        assert "is truncated (bad weights)" in capfd.readouterr().err
    finally:
        m.close()


def _edge_rows():
    r = O.sample_row(5000, 60, 1.0, 0)
    ninf = r.copy()
    ninf[::3] = -np.inf                        # expf(-inf) = 0: never kept by top-p, p = 0 otherwise
    return {
        "V1": np.array([0.25], np.float32),
        "flat": np.full(4096, 1.5, np.float32),     # every probability equal: index order decides
        "plain": r,
        "ninf": ninf,
        "wide": O.sample_row(131072, 61, 3.0, 1),   # top-k path at its widest vocabulary
    }


@pytest.mark.parametrize("case", [
    ("V1", 0.8, 40, 0.95), ("V1", 2.0, 0, 1.0),
    ("flat", 1.0, 0, 0.5), ("flat", 0.7, 64, 0.3), ("flat", 1.0, 4096, 1.0),
    ("plain", 1e-30, 0, 0.9), ("plain", 1e3, 40, 0.95), ("plain", 1.0, 5000, 0.0),
    ("plain", 1.0, 0, 1e-7), ("plain", 1.0, 0, 0.999999), ("plain", 0.9, -3, 2.0),
    ("ninf", 0.8, 40, 0.95), ("ninf", 1.0, 0, 0.99),
    ("wide", 0.8, 40, 0.95), ("wide", 1.1, 0, 0.9),
])
def test_sample_token_edge_cases_match_oracle(Q, case):
    name, t, k, p = case
    row = _edge_rows()[name]
    rng = Q.rng_create(2024)
    st = O.rng_create(2024)
    for _ in range(5):
        g = Q.sample_token(row.reshape(1, -1), t, k, p, rng)
        r, st = O.sample_token(row, t, k, p, st)
        assert g == r and rng.state == st, case
    # and the compiled reference's draws for the same case
    ref = [c for c in S["edge_cases"] if c["row"] == name and np.float32(c["t"]) == np.float32(t)
           and c["k"] == k and np.float32(c["p"]) == np.float32(p)]
    assert len(ref) == 1
    rng = Q.rng_create(2024)
    assert [Q.sample_token(row.reshape(1, -1), t, k, p, rng) for _ in range(5)] == ref[0]["tokens"]
    assert rng.state == int(ref[0]["state"], 16)


def test_int8_nonzero_biases_and_gains_match_oracle(Q, tmp_path):
    """Biases and norm gains other than 1 through the int8 path: an LLMQ file
    written from an oracle model whose biases and gains were set, loaded on the
    GPU, decode steps and a batched prefill bit for bit against the oracle."""
    cfg = [3000, 256, 2, 8, 2, 32, 512, 64]
    ref = O.Model(cfg, 10000.0, seed=32)
    try:
        rng = np.random.default_rng(6)
        m = ref.m
        dm, qd, kvd = cfg[1], cfg[3] * cfg[5], cfg[4] * cfg[5]
        views = [(m.final_norm, dm, True)]
        for l in range(cfg[2]):
            b = m.blocks[l]
            views += [(b.attn_norm, dm, True), (b.ffn_norm, dm, True), (b.b_q, qd, False), (b.b_k, kvd, False),
                      (b.b_v, kvd, False)]
        for ptr, n, gain in views:
            a = np.ctypeslib.as_array(ptr, shape=(n,))
            a[:] = ((1.0 + rng.standard_normal(n) * 0.2) if gain else rng.standard_normal(n) * 0.1).astype(np.float32)
        path = str(tmp_path / "b.llmq")
        O.write_llmq(ref, path)
        g = Q.Model.load(path)
        try:
            ids = O.prompt(20, 9, cfg[0])
            for t in ids[:4]:
                assert np.array_equal(g.step(t).view(np.uint32), ref.step(t).view(np.uint32)), t
            lg = g.prefill(ids[4:]).copy()                 # batched (16 rows) after 4 decode steps
            for t in ids[4:]:
                r = ref.step(t)
            assert np.array_equal(lg.view(np.uint32), r.view(np.uint32))
        finally:
            g.close()
    finally:
        ref.close()
