"""GPU fp32 (LLMA) decode path through the C ABI (llama_kv_create /
llama_decode_step) against the fixtures the compiled reference wrote
(gen_golden e2e_f32) and against the oracle's k-order matmul.  Bar: token
streams and logits bit-exact (north-star tolerance reported too)."""
import sys

import numpy as np
import pytest

import oracle_lib as O
import qlib
from conftest import golden, golden_json

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def Q():
    q = qlib.load()
    assert q.lib().qllama_device_count() > 0, "no GPU visible to the HIP library"
    return q


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def gpu_model(Q, ref, cfg, base):
    return Q.FModel(Q.host_model(cfg, base, 1e-5, ref.tensors()))


@pytest.mark.parametrize("name", ["tiny", "mid"])
def test_f32_decode_matches_reference(Q, name):
    meta = golden_json(f"e2e_f32_{name}")
    ref = O.FModel(meta["cfg"], meta["rope_base"], seed=meta["seed"], tied=bool(meta["tied"]))
    try:
        assert ref.hash() == int(meta["model_hash"], 16)
        g = gpu_model(Q, ref, meta["cfg"], meta["rope_base"])
        try:
            hashes = [int(h, 16) for h in meta["logit_hashes"]]
            P = len(meta["prompt"])
            for i, t in enumerate(meta["prompt"]):
                log(f"{name} prompt step {i}")
                lg = g.step(t)
                assert O.hash_f32(lg) == hashes[i], i
            np.testing.assert_allclose(lg, golden(f"e2e_f32_{name}_logits_prompt_last"), atol=1e-3, rtol=1e-4)
            assert np.array_equal(bits(lg), bits(golden(f"e2e_f32_{name}_logits_prompt_last")))
            for s, t in enumerate(meta["gen"]):
                assert int(np.argmax(lg)) == t, s
                lg = g.step(t)
                assert O.hash_f32(lg) == hashes[P + s], P + s
            assert np.array_equal(bits(lg), bits(golden(f"e2e_f32_{name}_logits_final")))
        finally:
            g.close()
    finally:
        ref.close()


@pytest.mark.parametrize("K", [64, 65, 79, 511, 512, 513, 575, 576, 640, 1023, 1087])
def test_f32_gemv_group_edges_match_oracle(Q, K):
    """The fp32 GEMV where its loop changes form: inputs around whole groups of 64
    k rows, around the eight groups in flight (512) and around tiles of 16, with
    a partial column panel: bit for bit against the oracle."""
    cfg = [33, 48, 1, 3, 1, 16, K, 16]
    ref = O.FModel(cfg, 10000.0, seed=K)
    try:
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            for t in [1, 5, 32]:
                r = ref.step(t).copy()
                assert np.array_equal(bits(g.step(t)), bits(r)), (K, t)
        finally:
            g.close()
    finally:
        ref.close()


@pytest.mark.parametrize("dm,dff", [(1, 16), (63, 48), (1023, 32), (1024, 33), (1025, 1040), (2047, 16), (2048, 64),
                                    (2049, 64), (64, 16384), (64, 16400)])
def test_f32_norm_in_gemv_edges_match_oracle(Q, dm, dff):
    """The decode GEMVs that normalize their row themselves, where that changes
    form: rows of one float, around 1024 (elements a thread) and 2048 (separate
    kernels), gate|up widths that are not whole panels (separate SwiGLU) and
    around 1024 panels: bit for bit against the oracle."""
    cfg = [33, dm, 2, 2, 1, 16, dff, 16]
    ref = O.FModel(cfg, 10000.0, seed=dm + dff)
    try:
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            for t in [1, 5, 32]:
                r = ref.step(t).copy()
                assert np.array_equal(bits(g.step(t)), bits(r)), (dm, dff, t)
        finally:
            g.close()
    finally:
        ref.close()


@pytest.mark.parametrize("K", [1, 17, 48, 80, 200, 288, 513, 768, 1040, 2000])
@pytest.mark.parametrize("pro,mode", [(0, 0), (1, 0), (1, 4), (2, 3)])
def test_f32_gemv_sees_its_own_panels_only(Q, pro, mode, K):
    """Inputs that end inside a group of four tiles, or whose groups are fewer than
    those in flight: with every second 16-column panel of the weights infinite, the
    other panels' outputs are finite and, bit for bit, what they are with finite
    neighbours (pro 0 plain, 1 rmsnorm, 2 LayerNorm; mode 4 SwiGLU, 3 GELU)."""
    import ctypes as C
    lib, N = Q.lib(), 64
    cols = 2 * N if mode == 4 else N
    lib.qllama_dev_alloc.restype = C.c_void_p
    lib.qhip_panels_f32_size.restype = C.c_size_t
    lib.qllama_dev_free.argtypes = [C.c_void_p]
    lib.qllama_h2d.argtypes = lib.qllama_d2h.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t]
    lib.qhip_to_panels_f32.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p]
    lib.qhip_gemv_f32.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    lib.qhip_gemv_f32_norm.argtypes = [C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_float,
                                       C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                       C.c_int, C.c_int]
    bufs = []

    def dev(a):
        p = lib.qllama_dev_alloc(C.c_size_t(a.nbytes))
        assert p and lib.qllama_h2d(p, a.ctypes.data, a.nbytes) == 0
        bufs.append(p)
        return p

    rng = np.random.default_rng(K)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    W = f(K, cols)
    Winf = W.copy()
    Winf[:, (np.arange(cols) // 16) % 2 == 1] = np.inf
    try:
        x, gamma, beta, bias = dev(f(K)), dev(f(K)), dev(f(K)), dev(f(N))
        got = []
        for w in (W, Winf):
            panels = dev(np.zeros(lib.qhip_panels_f32_size(K, cols), np.float32))
            out, dst = np.empty(N, np.float32), dev(np.zeros(N, np.float32))
            assert lib.qhip_to_panels_f32(dev(w), K, cols, panels) == 0
            if pro == 0:
                assert lib.qhip_gemv_f32(mode, 12, x, K, panels, N, dst, bias) == 0
            else:
                assert lib.qhip_gemv_f32_norm(pro, mode, 12, x, K, gamma, beta, 1e-5, panels, N, dst,
                                              None if mode == 4 else bias, None, None, None, 0, 0) == 0
            assert lib.qllama_d2h(out.ctypes.data, dst, out.nbytes) == 0
            got.append(out)
    finally:
        lib.qllama_sync()
        for p in bufs:
            lib.qllama_dev_free(p)
    own = (np.arange(N) // 16) % 2 == 0
    assert np.isfinite(got[1][own]).all()
    assert np.array_equal(bits(got[0][own]), bits(got[1][own]))


@pytest.mark.parametrize("rows,dff,vocab", [(1, 33, 70), (5, 64, 17), (9, 100, 130), (40, 31, 64), (70, 95, 2100),
                                            (300, 66, 16384), (130, 34, 16384), (300, 66, 40001)])
def test_f32_forward_tile_edges_match_oracle(Q, rows, dff, vocab):
    """The many-row fp32 matmul where its tiles end: rows around a wave's and a
    block's (each of the row groups of 1, 2, 4 and 8 is taken by one of these),
    k rows past whole stages, batches and groups of four, column panels cut
    short; and where the head's parts and the staged copies of their logits end
    (a part of one copy and one of two rows, parts of three copies): every row bit for bit the oracle's step."""
    cfg = [vocab, 144, 1, 3, 1, 48, dff, 320]
    ref = O.FModel(cfg, 10000.0, seed=rows)
    try:
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            ids = [(7 * i + 3) % vocab for i in range(rows)]
            got = g.forward(ids)
            for i, t in enumerate(ids):
                assert np.array_equal(bits(got[i]), bits(ref.step(t))), (rows, i)
        finally:
            g.close()
    finally:
        ref.close()


@pytest.mark.parametrize("shape", [(4096, 4096), (14336, 4096), (4096, 1024), (300, 17), (1000, 130), (129, 16)])
def test_f32_gemv_rows_match_oracle(Q, shape):
    """The fp32 GEMV at (K, N) through a one-layer model whose down projection
    has K inputs and whose head has N outputs: every step's logits bit for bit
    against the oracle (k-order chains over partial tiles, partial column
    blocks, the 14336-input down projection of the 8B shape)."""
    K, N = shape
    dm = 16 * ((K + 15) // 16) if K % 16 else K
    cfg = [N if N >= 16 else 16, min(dm, 4096), 1, 4, 2, 32, max(K, 64), 32]
    ref = O.FModel(cfg, 10000.0, seed=7)
    try:
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            for t in [1, 5, 2, 9]:
                r = ref.step(t % cfg[0]).copy()
                o = g.step(t % cfg[0]).copy()
                assert np.array_equal(bits(o), bits(r)), shape
        finally:
            g.close()
    finally:
        ref.close()


def test_two_caches_share_one_device_copy(Q):
    meta = golden_json("e2e_f32_tiny")
    ref = O.FModel(meta["cfg"], meta["rope_base"], seed=meta["seed"])
    try:
        host = Q.host_model(meta["cfg"], meta["rope_base"], 1e-5, ref.tensors())
        a, b = Q.FModel(host), Q.FModel(host)
        try:
            la = [a.step(t).copy() for t in meta["prompt"][:6]]
            a.close()                                    # b keeps the device copy alive
            lb = [b.step(t).copy() for t in meta["prompt"][:6]]
            for x, y in zip(la, lb):
                assert np.array_equal(bits(x), bits(y))
            b.reset(0)
            assert np.array_equal(bits(b.step(meta["prompt"][0])), bits(la[0]))
        finally:
            a.close()
            b.close()
    finally:
        ref.close()


def test_cli_f32_branch_matches_reference(Q, tmp_path):
    """qllama-cli on an LLMA file: the `llama` command's f32 branch (main.c:686-700)
    with decode and sampling on the GPU, against the compiled reference's loop."""
    import os
    import subprocess
    from conftest import ROOT
    cli = os.path.join(ROOT, "llm-project_amd", "qllama-cli")
    S = golden_json("sample")["cli_f32"]
    meta = golden_json("e2e_f32_tiny")
    ref = O.FModel(meta["cfg"], meta["rope_base"], seed=S["seed"])
    try:
        path = str(tmp_path / "tiny.llma")
        ref.write_llma(path)
    finally:
        ref.close()
    stdin = "".join(" ".join(str(t) for t in ln["prompt"]) + "\n" for ln in S["lines"])
    expect = []
    for ln in S["lines"]:
        expect += [f"t {t}" for t in ln["gen"]]
        expect.append("gen: " + " ".join(str(t) for t in ln["prompt"] + ln["gen"]))
    log("running qllama-cli on an LLMA file")
    out = subprocess.run([cli, "llama", path, str(S["n_new"])], input=stdin.encode(), capture_output=True,
                         timeout=120)
    assert out.returncode == 0, out.stderr.decode()
    assert out.stdout.decode().splitlines() == expect


@pytest.mark.parametrize("name", ["tiny", "mid"])
def test_f32_forward_matches_reference(Q, name):
    """llama_model_forward on the GPU against the reference's batched forward rows."""
    meta = golden_json(f"e2e_f32_{name}")
    ref = O.FModel(meta["cfg"], meta["rope_base"], seed=meta["seed"], tied=bool(meta["tied"]))
    try:
        g = gpu_model(Q, ref, meta["cfg"], meta["rope_base"])
        try:
            L = g.forward(meta["prompt"])
            assert [f"{O.hash_f32(r):016x}" for r in L] == meta["forward_hashes"]
            assert g.pos == 0                       # the caller's cache is untouched
        finally:
            g.close()
    finally:
        ref.close()


def perturb(ref, seed):
    """Nonzero q/k/v biases and norm gains other than 1 (llama.c:319-321, rmsnorm.c:18)."""
    rng = np.random.default_rng(seed)
    for name, t in ref.tensors():
        if name in ("b_q", "b_k", "b_v"):
            t[:] = rng.standard_normal(t.shape).astype(np.float32) * np.float32(0.1)
        if name in ("attn_norm", "ffn_norm", "final_norm"):
            t[:] = (1.0 + rng.standard_normal(t.shape) * 0.2).astype(np.float32)


def test_f32_forward_two_passes_match_oracle(Q):
    """The batched forward over 2100 rows, so each layer takes two passes (2048 +
    52 rows) and the second pass attends to the first's cache rows; biases, norm
    gains and an FFN width of 250 (not a multiple of 4: the GEMM's scalar loads).
    Every row bit for bit against the oracle's decode step at that position."""
    cfg = [700, 128, 2, 4, 2, 64, 250, 2112]
    n = 2100
    ref = O.FModel(cfg, 10000.0, seed=41)
    try:
        perturb(ref, 9)
        ids = [int(t) for t in np.random.default_rng(3).integers(0, cfg[0], n)]
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            log("forward of 2100 rows")
            L = g.forward(ids)
        finally:
            g.close()
        for i, t in enumerate(ids):
            r = ref.step(t)
            assert np.array_equal(bits(L[i]), bits(r)), i
    finally:
        ref.close()


def test_f32_forwards_at_once_match_single_calls(Q):
    """Forwards from several threads that overlap, on one model and on another:
    every call's logits are those of the same call made alone."""
    from concurrent.futures import ThreadPoolExecutor
    refs = [O.FModel([2100, 96, 2, 2, 1, 48, 130, 320], 10000.0, seed=s) for s in (61, 62)]
    gs = [gpu_model(Q, r, [2100, 96, 2, 2, 1, 48, 130, 320], 10000.0) for r in refs]
    try:
        work = [(i % 2 if k == 2 else 0, [(11 * j + i) % 2100 for j in range(rows)])
                for k in range(3) for i, rows in enumerate((300, 70, 130, 257))]
        alone = [gs[g].forward(ids).copy() for g, ids in work]
        with ThreadPoolExecutor(4) as pool:
            for _ in range(4):
                got = list(pool.map(lambda w: gs[w[0]].forward(w[1]).copy(), work))
                for a, b in zip(alone, got):
                    assert np.array_equal(bits(a), bits(b))
    finally:
        for x in gs + refs:
            x.close()


def test_f32_forward_keeps_a_bounded_workspace(Q):
    """What a long forward used (here 600 rows of 128256 logits, over 300 MB) is given
    back when it ends, with a cache of the model alive; calls after it still match."""
    import ctypes as C

    def free_bytes():
        f, t = C.c_size_t(), C.c_size_t()
        assert Q.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    cfg = [128256, 48, 1, 1, 1, 48, 32, 640]
    ref = O.FModel(cfg, 10000.0, seed=8)
    try:
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            few = g.forward([3, 128255, 7]).copy()
            before = free_bytes()
            L = g.forward([(97 * i + 3) % cfg[0] for i in range(600)])
            assert before - free_bytes() < (32 << 20)
            r = [ref.step((97 * i + 3) % cfg[0]).copy() for i in range(2)]
            for i in range(2):
                assert np.array_equal(bits(L[i]), bits(r[i]))
            assert np.array_equal(bits(g.forward([3, 128255, 7])), bits(few))
        finally:
            g.close()
    finally:
        ref.close()


def test_f32_forward_past_max_seq_matches_oracle(Q):
    """seq_len above the model's max_seq (the reference's forward has no such
    bound, llama.c:167-186): positions 16 .. 39 take RoPE tables made for the
    call.  Rows against the oracle's decode steps on the same weights with room
    for 64 positions."""
    cfg16 = [500, 192, 2, 6, 2, 48, 320, 16]
    cfg64 = cfg16[:7] + [64]
    ref = O.FModel(cfg64, 10000.0, seed=17)
    try:
        ids = [int(t) for t in np.random.default_rng(4).integers(0, 500, 40)]
        g = gpu_model(Q, ref, cfg16, 10000.0)
        try:
            L = g.forward(ids)
        finally:
            g.close()
        for i, t in enumerate(ids):
            assert np.array_equal(bits(L[i]), bits(ref.step(t))), i
    finally:
        ref.close()


def test_f32_forward_batched_equals_steps(Q, monkeypatch):
    """The batched forward and the decode-step replay (QLLAMA_FORWARD_STEPS=1)
    give the same bits on the mid fixture's model."""
    meta = golden_json("e2e_f32_mid")
    ref = O.FModel(meta["cfg"], meta["rope_base"], seed=meta["seed"], tied=bool(meta["tied"]))
    try:
        g = gpu_model(Q, ref, meta["cfg"], meta["rope_base"])
        try:
            ids = list(meta["prompt"]) * 3
            a = g.forward(ids)
            monkeypatch.setenv("QLLAMA_FORWARD_STEPS", "1")
            b = g.forward(ids)
            assert np.array_equal(bits(a), bits(b))
        finally:
            g.close()
    finally:
        ref.close()


def test_f32_nonzero_biases_and_gains_match_oracle(Q):
    """Biases (Qwen-style checkpoints, llama.c:319-321) and norm gains other than 1
    (rmsnorm.c:18) through the fp32 step, bit for bit against the oracle."""
    cfg = [3000, 256, 2, 8, 2, 32, 512, 64]
    ref = O.FModel(cfg, 10000.0, seed=31)
    try:
        perturb(ref, 5)
        g = gpu_model(Q, ref, cfg, 10000.0)
        try:
            for t in [3, 17, 2999, 0, 42, 7]:
                a = g.step(t).copy()
                b = ref.step(t).copy()
                assert np.array_equal(bits(a), bits(b)), t
        finally:
            g.close()
    finally:
        ref.close()
