"""The resident batch-1 decoder step (k_resident.hip): all layers in one launch, with the bits
of the per-layer launches it stands in for."""
import threading

import numpy as np
import pytest

import malaga_amd as M
import oracle as O
from tests.test_gpu_full_size import argmax_chain_check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d0 = tmp_path_factory.mktemp("resident")
    made = {}

    def get(preset, d, f, layers=3):
        p = d0 / f"{preset}-{d}-{f}.gguf"
        if p not in made:
            cfg = dict(vocab_size=1200, d_model=d, encoder_layers=1, decoder_layers=layers, encoder_heads=d // 64,
                       decoder_heads=d // 64, encoder_ffn=512, decoder_ffn=f, max_position_embeddings=256,
                       max_length=200, scale_embedding=1, bos_token_id=0, pad_token_id=1, eos_token_id=2,
                       decoder_start_token_id=2)
            M.write_synthetic(p, cfg, preset, M.INIT_NORMAL_RICH, seed=d + f, std=0.04, name="resident")
            made[p] = p
        return p

    return get


@pytest.mark.parametrize("preset", ["q4_k_m", "q5_k_m"])
@pytest.mark.parametrize("d,f", [(256, 512), (512, 1536), (1024, 4096), (1024, 2560)])
def test_resident_step_matches_oracle(model, preset, d, f):
    """Every width the kernel takes, FFNs that fill and do not fill the gathering threads, and
    one key, a few and more keys than one round of the 8 waves (64) in both attentions: each
    token is the oracle's argmax after the same prefix, the winning logits within 2e-3."""
    path = model(preset, d, f)
    gpu, orc = M.Translator.load(path), O.Model(path)
    calls = 0
    try:
        for n, new in ((1, 5), (7, 9), (70, 72)):
            src = [np.random.default_rng(n + d).integers(4, 1200, n).tolist()]
            batch = gpu.encode_cross(src)
            toks, top = gpu.greedy_top(batch, 1100, new, eos_mask=True)
            again = gpu.greedy_top(batch, 1100, new, eos_mask=True)  # the captured graph
            eager = gpu.greedy_top(batch, 1100, new, eos_mask=True, graph=False)
            assert again == (toks, top) == eager
            calls += 3
            assert gpu.resident_stats() == {"active": True, "calls": calls, "redone": 0}
            tgt = np.array([[2, 1100] + toks[0][:-1]], np.uint32)
            ref = orc.teacher_forced_logits(src, tgt, kv_f16=True)
            argmax_chain_check(toks, top, ref, tie=4e-3)
    finally:
        gpu.close()


def load(path, monkeypatch, **env):
    """A translator that read these variables at load."""
    with monkeypatch.context() as m:
        for k, v in env.items():
            m.setenv(k, v)
        return M.Translator.load(path)


@pytest.mark.parametrize("preset", ["q4_k_m", "q5_k_m"])
@pytest.mark.parametrize("d,f", [(256, 512), (512, 1536), (1024, 4096), (1024, 2560), (256, 3584)])
def test_resident_step_equals_per_layer_launches(model, monkeypatch, preset, d, f):
    """Tokens and winning logits bit for bit, with one key, keys on both sides of the attention's
    groups of 8 and rounds of 64 in both attentions, and several rounds: the sums have one
    order, so what a call returns does not depend on the launches it gets."""
    path = model(preset, d, f)
    on, off = load(path, monkeypatch), load(path, monkeypatch, MALAGA_RESIDENT_STEP="0")
    try:
        for n, new in ((1, 1), (8, 9), (9, 8), (63, 66), (64, 3), (65, 3), (130, 140), (200, 30)):
            src = [np.random.default_rng(n * d).integers(4, 1200, n).tolist()]
            a = on.greedy_top(on.encode_cross(src), 1100, new, eos_mask=True)
            b = off.greedy_top(off.encode_cross(src), 1100, new, eos_mask=True)
            assert a == b, (n, new)
        assert on.resident_stats() == {"active": True, "calls": 8, "redone": 0}
        assert off.resident_stats() == {"active": False, "calls": 0, "redone": 0}
    finally:
        on.close()
        off.close()


def test_resident_step_off_and_out_of_polls(model, monkeypatch):
    """MALAGA_RESIDENT_STEP=0 and a launch whose waits run out at once (the flag is raised and
    the call decodes again per layer) give the same bits; the next 16 calls do without the
    launch, 32 after the second failure, and once it gets its polls again it decodes again."""
    path = model("q4_k_m", 512, 1536)
    src = [np.random.default_rng(3).integers(4, 1200, 11).tolist()]
    off = load(path, monkeypatch, MALAGA_RESIDENT_STEP="0")
    want = off.greedy_top(off.encode_cross(src), 1100, 20, eos_mask=True)
    off.close()
    gpu = load(path, monkeypatch, MALAGA_RESIDENT_SPINS="0")
    try:
        batch = gpu.encode_cross(src)

        def decode(n=1, graph=True):
            for _ in range(n):
                assert gpu.greedy_top(batch, 1100, 20, eos_mask=True, graph=graph) == want

        def stats(active, calls, redone):
            assert gpu.resident_stats() == {"active": active, "calls": calls, "redone": redone}

        decode()
        stats(False, 0, 1)
        decode(15)
        stats(False, 0, 1)
        decode()
        stats(True, 0, 1)
        decode(graph=False)  # out of polls again, the same state and its words used again
        stats(False, 0, 2)
        decode(32)
        stats(True, 0, 2)
        gpu.lib.mlg_debug_resident_spins(gpu.h, 1 << 16)
        decode(2)
        decode(graph=False)
        stats(True, 3, 2)
    finally:
        gpu.close()


def test_resident_step_after_a_failed_launch(model):
    """The state of a launch that gave up is used again, with words of that launch's tag in it: a
    later launch takes none of them for its own."""
    path = model("q4_k_m", 1024, 2560)
    src = [np.random.default_rng(5).integers(4, 1200, 30).tolist()]
    gpu = M.Translator.load(path)
    try:
        batch = gpu.encode_cross(src)
        want = gpu.greedy_top(batch, 1100, 40, eos_mask=True)
        for failed in range(1, 4):
            gpu.lib.mlg_debug_resident_spins(gpu.h, 0)
            assert gpu.greedy_top(batch, 1100, 40, eos_mask=True) == want
            assert gpu.resident_stats()["redone"] == failed
            gpu.lib.mlg_debug_resident_spins(gpu.h, 1 << 16)
            for _ in range(16):
                assert gpu.greedy_top(batch, 1100, 40, eos_mask=True) == want
            before = gpu.resident_stats()["calls"]
            assert gpu.greedy_top(batch, 1100, 40, eos_mask=True) == want
            assert gpu.resident_stats() == {"active": True, "calls": before + 1, "redone": failed}
    finally:
        gpu.close()


def test_resident_step_from_several_threads(model):
    """Contexts of their own on one device: one call at a time has the resident launch, the
    others decode per layer meanwhile; every call gives the tokens and logits, to the bit, that
    it gives alone."""
    path = model("q4_k_m", 256, 512)
    srcs = [[np.random.default_rng(50 + i).integers(4, 1200, 4 + 5 * i).tolist()] for i in range(3)]

    def decode(t, src):
        return t.greedy_top(t.encode_cross(src), 1100, 30, eos_mask=True)

    ref = M.Translator.load(path)
    want = [decode(ref, s) for s in srcs]
    ref.close()
    ts = [M.Translator.load(path) for _ in srcs]
    done = []

    def work(i):
        done.append((i, all(decode(ts[i], srcs[i]) == want[i] for _ in range(8))))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(ts))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert sorted(done) == [(i, True) for i in range(len(ts))]
    assert sum(t.resident_stats()["calls"] for t in ts) > 0
    for t in ts:
        t.close()
