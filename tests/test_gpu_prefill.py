"""GPU: a decode whose prompt goes through the layers as passes over many
positions (bfp_prefill.hip) against the same decode step by step (direct
launches, which never take a pass) -- tokens, every layer's output at every
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
        got = both()
        for a, b in zip(want[:3], got[:3]):
            assert np.array_equal(a, b)
        for (wk, wv), (gk, gv) in zip(want[3], got[3]):
            for a, b in zip((*wk, *wv), (*gk, *gv)):
                assert np.array_equal(a, b)
    gm.close()
