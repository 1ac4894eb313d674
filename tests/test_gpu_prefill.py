"""GPU: a decode whose prompt goes through the layers as passes over many
positions (bfp_prefill.hip) against the same decode step by step (direct
launches, which never take a pass; the number of steps that ran as passes is
checked on both sides) -- tokens, every layer's output at every
step, the cache rows and the tokens generated from them, bit for bit: at the
edges of the attention's tiles (positions a workgroup, 32-row V blocks,
256-row K blocks), over several passes, for ragged and split head groups, and
at a context where the scores of one position fill the workgroup's LDS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dims, batch, prompt lengths, n_gen)
CASES = {
    "short": (dict(D=192, H_Q=3, H_KV=1, FFN=256, NL=2, MAX_CTX=80, VOCAB=512), 1, (2, 3, 4, 5, 13, 65), 4),
    "two-groups": (dict(D=256, H_Q=4, H_KV=2, FFN=512, NL=2, MAX_CTX=340, VOCAB=512), 3, (2, 63, 257, 331), 3),
    "split-heads-4": (dict(D=256, H_Q=4, H_KV=1, FFN=512, NL=2, MAX_CTX=200, VOCAB=512), 2, (4, 130), 3),
    "split-heads-5": (dict(D=320, H_Q=5, H_KV=1, FFN=336, NL=2, MAX_CTX=140, VOCAB=512), 2, (5, 129), 3),
    "one-head": (dict(D=64, H_Q=1, H_KV=1, FFN=128, NL=1, MAX_CTX=100, VOCAB=256), 5, (17,), 2),
    "several-passes": (dict(D=192, H_Q=3, H_KV=1, FFN=256, NL=2, MAX_CTX=90, VOCAB=512), 40, (81,), 2),
    "no-generation": (dict(D=192, H_Q=3, H_KV=1, FFN=256, NL=2, MAX_CTX=40, VOCAB=512), 2, (30,), 0),
    "width": (dict(D=576, H_Q=9, H_KV=3, FFN=1536, NL=2, MAX_CTX=600, VOCAB=1024), 1, (530,), 8),
    "long": (dict(D=192, H_Q=3, H_KV=1, FFN=256, NL=1, MAX_CTX=4096, VOCAB=256), 1, (2600,), 2),
    "large-weights": (dict(D=192, H_Q=3, H_KV=1, FFN=256, NL=2, MAX_CTX=80, VOCAB=512), 2, (70,), 4),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prompt_pass_equals_steps(gpu, name):
    from bfp import Dims, synth
    from bfp.model import BfpModel
    cfg, batch, lengths, n_gen = CASES[name]
    d = Dims(HD=64, **cfg)
    fm = synth.make_model(d, seed=31)
    if name == "large-weights":   # peaked softmax rows: probabilities that underflow to 0
        for lw in fm.layers:
            lw["Wq"] *= 40
            lw["Wk"] *= 40
    gm = BfpModel(d, max_batch=batch)
    gm.load_fp32(fm)
    rng = np.random.default_rng(5)
    for n_prompt in lengths:
        print(f"[prefill] {name} batch {batch} prompt {n_prompt}", flush=True)
        P = rng.integers(0, d.VOCAB, size=(batch, n_prompt)).astype(np.int32)

        def both(**kw):
            gm.reset_kv()
            toks, (hm, he) = gm.decode(P, n_gen, hist=True, **kw)
            kv = [gm.kv_io(li, b, 0, n_prompt + n_gen) for li in range(d.NL) for b in range(batch)]
            return toks, hm, he, kv

        want = both(graph=False)
        assert gm.prompt_pass_steps() == 0
        got = both()
        # at batch 1 these contexts decode persistently, where a pass is made from 4 positions
        taken = n_prompt >= (4 if gm.decode_path() == "persist" else 2)
        assert gm.prompt_pass_steps() == (n_prompt if taken else 0)
        for a, b in zip(want[:3], got[:3]):
            assert np.array_equal(a, b)
        for (wk, wv), (gk, gv) in zip(want[3], got[3]):
            for a, b in zip((*wk, *wv), (*gk, *gv)):
                assert np.array_equal(a, b)
    gm.close()


@pytest.mark.parametrize("batch", [1, 3, 17])
def test_prompt_steps_without_memory_for_a_pass(gpu, monkeypatch, batch):
    """Where there is no memory for a pass's rows the prompt runs step by
    step: the same tokens, history and cache rows, call after call."""
    from bfp import Dims, synth
    from bfp.model import BfpModel
    d = Dims(D=192, H_Q=3, H_KV=1, HD=64, FFN=256, NL=2, MAX_CTX=40, VOCAB=512)
    fm = synth.make_model(d, seed=7)
    P = np.random.default_rng(batch).integers(0, d.VOCAB, size=(batch, 11)).astype(np.int32)
    got = []
    for held in (True, False):
        monkeypatch.setenv("BFP_OPTIONAL_MEMORY", str(int(held)))
        gm = BfpModel(d, max_batch=batch)
        gm.load_fp32(fm)
        assert gm.prompt_pass_steps() is None
        for _ in range(2):
            gm.reset_kv()
            toks, (hm, he) = gm.decode(P, 5, hist=True)
            assert gm.prompt_pass_steps() == (11 if held else 0)
            assert ("prompt" in gm.optional_memory()) == held
            got.append([toks, hm, he] + [x for li in range(d.NL) for b in range(batch)
                                         for t in gm.kv_io(li, b, 0, 16) for x in t])
        gm.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
