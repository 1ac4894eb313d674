"""GPU parity of one decoder layer against the oracle's
fwd_layer (oracle/bfp_sim.py restating
rtl/vc707/host/gen_smollm_blockfp_full.py:261-293): every one of the 13
stage outputs, bit for bit, at positions 0..7 with the KV cache growing."""
import numpy as np
import pytest

from oracle import bfp_sim as sim

pytestmark = pytest.mark.gpu

SMALL = dict(D=64, H_Q=1, H_KV=1, HD=64, FFN=128, NL=1, MAX_CTX=16, VOCAB=256)
MID = dict(D=192, H_Q=3, H_KV=1, HD=64, FFN=256, NL=1, MAX_CTX=16, VOCAB=256)
FULL = dict(D=576, H_Q=9, H_KV=3, HD=64, FFN=1536, NL=1, MAX_CTX=16, VOCAB=256)
# a KV capacity above 512: the long-context attention form (four workgroups
# per head, each dumping its own 16-dimension tile of the attention output)
FULL_LONG = dict(FULL, MAX_CTX=600)


def _setup(cfg, seed, max_batch=1):
    from bfp import Dims, synth
    from bfp.model import BfpModel
    d = Dims(**cfg)
    fm = synth.make_model(d, seed=seed)
    om = sim.build_model(fm)
    gm = BfpModel(d, max_batch=max_batch)
    gm.load_fp32(fm)
    return d, om, gm


def _check_stages(stages, dump, b, pos, tag):
    for name in sim.STAGES:
        wm, we = sim.tile_quantize(dump[name])
        gm_, ge_ = stages[name]
        assert (ge_[b] == we).all(), f"{tag} pos {pos}: stage {name} exponents differ"
        assert (gm_[b] == wm.reshape(-1)).all(), f"{tag} pos {pos}: stage {name} mantissas differ"


@pytest.mark.parametrize("cfg", [SMALL, MID, FULL, FULL_LONG], ids=["small", "mid", "full", "full-long"])
def test_layer_8_positions(gpu, cfg):
    d, om, gm = _setup(cfg, seed=1)
    print(f"[layer] dims {cfg}", flush=True)
    from bfp import synth
    xs = synth.make_layer_inputs(d, 8, seed=1)
    kv = sim.new_kv(om.dims, d.MAX_CTX)
    for p in range(8):
        h = sim.fp_quantize_vec(xs[p])
        dump = {}
        want = sim.fwd_layer(h, om.layers[0], pos=p, kv=kv, kv_pos=p, dims=om.dims, dump=dump)
        hm, he = sim.tile_quantize(h)
        out_m, out_e, st = gm.layer_step_bfp(0, p, hm.reshape(1, -1), he.reshape(1, -1), dump=True)
        _check_stages(st, dump, 0, p, str(cfg["D"]))
        # the returned tile is the raw quantisation: its values are the reference's
        assert (sim.tile_decode(out_m[0].reshape(-1, 16), out_e[0]) == want).all()
    gm.close()


def test_layer_batched_sequences(gpu):
    """Three independent sequences in one launch: each matches its own
    oracle run (own KV cache)."""
    d, om, gm = _setup(MID, seed=2, max_batch=3)
    rng = np.random.default_rng(5)
    kvs = [sim.new_kv(om.dims, d.MAX_CTX) for _ in range(3)]
    for p in range(5):
        hs = [sim.fp_quantize_vec(rng.standard_normal(d.D) * (1 + b)) for b in range(3)]
        q = [sim.tile_quantize(h) for h in hs]
        hm = np.stack([x[0].reshape(-1) for x in q])
        he = np.stack([x[1] for x in q])
        out_m, out_e, st = gm.layer_step_bfp(0, p, hm, he, dump=True)
        for b in range(3):
            dump = {}
            sim.fwd_layer(hs[b], om.layers[0], pos=p, kv=kvs[b], kv_pos=p, dims=om.dims, dump=dump)
            _check_stages(st, dump, b, p, f"seq{b}")
    gm.close()


@pytest.mark.parametrize("cfg,batch", [(MID, 5), (FULL, 6), (MID, 9), (FULL_LONG, 9), (MID, 16), (MID, 17), (MID, 33),
                                       (FULL, 40), (FULL_LONG, 17)],
                         ids=["seq-mid-b5", "seq-full-b6", "seq-mid-b9", "seq-full-long-b9", "mfma-mid-b16",
                              "mfma-mid-b17", "mfma-mid-b33", "mfma-full-b40", "mfma-full-long-b17"])
def test_layer_multi_sequence_path(gpu, cfg, batch):
    """Several sequences a launch: below 16 the per-sequence kernels, from 16
    on the norm once per sequence and the tile sums on the int8 matrix cores
    in blocks of 16 sequences (16: one whole block; 17, 33: a last block of
    one sequence), with the short and the long attention form: every stage of
    every sequence still equals its own oracle run."""
    d, om, gm = _setup(cfg, seed=7, max_batch=batch)
    rng = np.random.default_rng(9)
    kvs = [sim.new_kv(om.dims, d.MAX_CTX) for _ in range(batch)]
    for p in range(4):
        hs = [sim.fp_quantize_vec(rng.standard_normal(d.D) * (0.5 + b)) for b in range(batch)]
        q = [sim.tile_quantize(h) for h in hs]
        hm = np.stack([x[0].reshape(-1) for x in q])
        he = np.stack([x[1] for x in q])
        out_m, out_e, st = gm.layer_step_bfp(0, p, hm, he, dump=True)
        for b in range(batch):
            dump = {}
            sim.fwd_layer(hs[b], om.layers[0], pos=p, kv=kvs[b], kv_pos=p, dims=om.dims, dump=dump)
            _check_stages(st, dump, b, p, f"seq{b}")
    gm.close()


def test_fwd_layer_float_api(gpu):
    """The reference-named float64 entry point."""
    d, om, gm = _setup(SMALL, seed=3)
    kv = sim.new_kv(om.dims, d.MAX_CTX)
    rng = np.random.default_rng(0)
    for p in range(3):
        h = sim.fp_quantize_vec(rng.standard_normal(d.D))
        want = sim.fwd_layer(h, om.layers[0], pos=p, kv=kv, kv_pos=p, dims=om.dims)
        got = gm.fwd_layer(h, 0, p)
        assert (got == want).all()
    # RoPE position and cache slot apart: slot 2 is overwritten
    want = sim.fwd_layer(h, om.layers[0], pos=3, kv=kv, kv_pos=2, dims=om.dims)
    assert (gm.fwd_layer(h, 0, 3, kv_pos=2) == want).all()
    gm.close()


def test_second_context_keeps_lds_limit(gpu):
    """A context made after a larger one of the same attention form must
    not lower the kernel's dynamic-LDS limit under the first: the first
    still runs at a position past the second's capacity, and matches the
    oracle."""
    from bfp import Dims, synth
    from bfp.model import BfpModel
    d1 = Dims(NL=1, MAX_CTX=2048, VOCAB=256)
    fm = synth.make_model(d1, seed=41)
    om = sim.build_model(fm)
    big = BfpModel(d1)
    big.load_fp32(fm)
    small = BfpModel(Dims(NL=1, MAX_CTX=600, VOCAB=256))
    rng = np.random.default_rng(41)
    kv = sim.new_kv(om.dims, 2048)
    h = sim.fp_quantize_vec(rng.standard_normal(d1.D))
    want = sim.fwd_layer(h, om.layers[0], pos=1500, kv=kv, kv_pos=1500, dims=om.dims)
    hm, he = sim.tile_quantize(h)
    om_, oe_, _ = big.layer_step_bfp(0, 1500, hm.reshape(1, -1), he.reshape(1, -1))
    assert (sim.tile_decode(om_[0].reshape(-1, 16), oe_[0]) == want).all()
    small.close()
    big.close()


@pytest.mark.parametrize("spread", [6, 46, 50, 120])
def test_batched_matvecs_exponent_spreads(gpu, spread):
    """The matrix-core matvecs of a batch (float64 floor accumulation, with
    and without the 47-bit window's test) against the batch-1 kernels'
    64-bit shifts: full-range mantissas (sums to 2^34, -32768 among them),
    weight exponents spread below, across and beyond the window, zero tiles."""
    from bfp import Dims
    from bfp.model import BfpModel
    d = Dims(D=192, H_Q=3, H_KV=1, HD=64, FFN=272, NL=1, MAX_CTX=8, VOCAB=256)
    B = 19   # a full group of 16 and a ragged one
    rng = np.random.default_rng(spread)
    gm = BfpModel(d, max_batch=B)
    for name, (r, c) in {"Wq": (d.D, d.D), "Wk": (d.KV, d.D), "Wv": (d.KV, d.D), "Wo": (d.D, d.D),
                         "Wg": (d.FFN, d.D), "Wu": (d.FFN, d.D), "Wd": (d.D, d.FFN)}.items():
        m = rng.integers(-32768, 32768, size=(r, c // 16, 16)).astype(np.int16)
        m[rng.random((r, c // 16)) < 0.05] = -32768
        e = rng.integers(-spread // 2, spread - spread // 2 + 1, size=(r, c // 16)).astype(np.int8)
        zero = rng.random((r, c // 16)) < 0.02
        m[zero], e[zero] = 0, -127
        gm.load_tensor(name, 0, m=m, e=e)
    for name in ("g1", "g2"):
        gm.load_tensor(name, 0, fp32=(1 + 0.1 * rng.standard_normal(d.D)).astype(np.float32))
    hm = rng.integers(-32768, 32768, size=(B, d.D)).astype(np.int16)
    he = rng.integers(-3, 4, size=(B, d.D // 16)).astype(np.int8)
    om, oe, st = gm.layer_step_bfp(0, 0, hm, he, dump=True)
    for b in range(B):
        wm, we, ws = gm.layer_step_bfp(0, 0, hm[b], he[b], dump=True)
        for name in st:
            assert np.array_equal(st[name][0][b], ws[name][0][0]), (b, name)
            assert np.array_equal(st[name][1][b], ws[name][1][0]), (b, name)
        assert np.array_equal(om[b], wm[0]) and np.array_equal(oe[b], we[0])
    gm.close()


@pytest.mark.parametrize("cfg", [dict(D=576, H_Q=9, H_KV=3, FFN=256, MAX_CTX=2048),
                                 dict(D=768, H_Q=12, H_KV=12, FFN=336, MAX_CTX=513),
                                 dict(D=512, H_Q=8, H_KV=2, FFN=512, MAX_CTX=4096)],
                         ids=["ctx2048", "ctx513", "ctx4096"])
def test_long_attention_forms(gpu, cfg):
    """Capacities past 512: one workgroup per head (past 512 / 4 heads a
    launch, without a stage dump) against four per head (with one, and below
    that), at the edges of the 32-row V blocks, the 64-row wave shares and the
    512-row K blocks, peaked and flat scores, RoPE position and KV slot apart."""
    from bfp import Dims, synth
    from bfp.model import BfpModel
    d = Dims(HD=64, NL=1, VOCAB=256, **cfg)
    B = 128 // d.H_Q + 1
    fm = synth.make_model(d, seed=5)
    gm = BfpModel(d, max_batch=B)
    gm.load_fp32(fm)
    rng = np.random.default_rng(d.MAX_CTX)
    n = d.MAX_CTX
    for b in range(B):
        km = rng.integers(-32768, 32768, size=(n, d.KV)).astype(np.int16)
        ke = rng.integers(-3 if b else -12, 3 if b else 5, size=(n, d.KV // 16)).astype(np.int8)
        gm.kv_io(0, b, 0, n, k=(km, ke), v=(km[::-1], ke[::-1]))
    for pos in (0, 1, 31, 32, 33, 63, 64, 500, 511, 512, 513, 1023, 1024, 1100, n - 1):
        if pos >= n:
            continue
        hm = rng.integers(-20000, 20000, size=(B, d.D)).astype(np.int16)
        he = np.zeros((B, d.D // 16), np.int8)
        want = gm.layer_step_bfp(0, pos + 3, hm, he, kv_pos=pos, dump=True)
        k0 = [gm.kv_io(0, b, pos, 1) for b in range(B)]
        got = gm.layer_step_bfp(0, pos + 3, hm, he, kv_pos=pos)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), pos
        for b in range(B):
            k1 = gm.kv_io(0, b, pos, 1)
            assert all(np.array_equal(x, y) for p, q in zip(k0[b], k1) for x, y in zip(p, q)), pos
        one = gm.layer_step_bfp(0, pos + 3, hm[0], he[0], kv_pos=pos)
        assert np.array_equal(one[0][0], got[0][0]) and np.array_equal(one[1][0], got[1][0]), pos
    gm.close()


@pytest.mark.parametrize("batch", [15, 17])
def test_long_attention_one_workgroup_a_head(gpu, batch):
    """Capacities past 512 without a stage dump, from 512 / 4 heads a launch:
    one workgroup per head (below and on the matrix cores otherwise), against
    the oracle, at the ends of the K and V blocks and with RoPE position and
    slot apart."""
    d, om, gm = _setup(dict(FULL, MAX_CTX=1100), seed=11, max_batch=batch)
    rng = np.random.default_rng(batch)
    seqs = (0, batch // 2, batch - 1)
    kvs = {b: sim.new_kv(om.dims, d.MAX_CTX) for b in seqs}
    for b in range(batch):
        rows = []
        for _ in range(2):
            m, e = sim.tile_quantize(rng.standard_normal(d.MAX_CTX * d.KV) * (0.3 + 0.1 * b))
            rows.append((m.reshape(d.MAX_CTX, d.KV), e.reshape(d.MAX_CTX, d.KV // 16)))
        gm.kv_io(0, b, 0, d.MAX_CTX, k=rows[0], v=rows[1])
        if b in seqs:
            for name, (m, e) in zip("kv", rows):
                kvs[b][name][:] = sim.tile_decode(m.reshape(-1, 16), e.reshape(-1)).reshape(d.MAX_CTX, d.H_KV, d.HD)
    for pos, slot in ((0, 0), (33, 31), (511, 511), (512, 512), (1090, 1099)):
        hs = [sim.fp_quantize_vec(rng.standard_normal(d.D) * (0.5 + b)) for b in range(batch)]
        q = [sim.tile_quantize(h) for h in hs]
        om_, oe_, _ = gm.layer_step_bfp(0, pos, np.stack([x[0].reshape(-1) for x in q]), np.stack([x[1] for x in q]),
                                        kv_pos=slot)
        for b in seqs:
            want = sim.fwd_layer(hs[b], om.layers[0], pos=pos, kv=kvs[b], kv_pos=slot, dims=om.dims)
            assert (sim.tile_decode(om_[b].reshape(-1, 16), oe_[b]) == want).all(), (pos, slot, b)
    gm.close()
