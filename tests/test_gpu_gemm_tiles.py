"""The exact GEMM tiles over the prefill copy (gemm_mid.h, gemm_wide.h) through whole layers: a request alone takes
small tiles, the same request inside a batch larger ones, and every tiling runs the same per-element sequence, so
the logits agree bit for bit at row counts around the tile edges (32, 64, 128 rows) and across the tile rule."""
import numpy as np
import pytest

from parity import assert_bits_equal

pytestmark = pytest.mark.gpu

LENGTHS = (2, 17, 32, 33, 65, 129, 300, 517, 700)


@pytest.mark.parametrize("preset, precision, layers", [
    ("plumbing-f16", 0, 1), ("q8-2048", 0, 1), ("q4km-7b", 0, 1), ("q4km-7b", 2, 1), ("f16-7b", 0, 1),
    ("openthai-0.8b", 0, 4)])
def test_decoder_tilings_agree(lh, preset, precision, layers):
    eng = lh.Engine(lh.Gguf.from_bytes(lh.SynthImage(preset, seed=31, n_layers=layers)), kv_tokens=16384,
                    precision=lh.PREC_KV16 if precision else lh.PREC_EXACT)
    rng = np.random.default_rng(7)
    ids = [rng.integers(0, 1000, n).astype(np.int32) for n in LENGTHS]
    options = np.arange(16, dtype=np.int32)

    def logits(requests):
        seqs = [eng.seq_create() for _ in requests]
        out = eng.batch([(s, r, [len(r) // 2, len(r) - 1]) for s, r in zip(seqs, requests)]).run(options)[0]
        for s in seqs:
            eng.seq_free(s)
        return out

    whole = logits(ids * 2)  # twice: enough work that attention takes its 32-row tiles, alone its 16-row ones
    assert np.isfinite(whole).all()
    assert_bits_equal(whole[:len(whole) // 2], whole[len(whole) // 2:])
    for i, r in enumerate(ids):
        print(f"{preset} {len(r)} tokens alone", flush=True)
        assert_bits_equal(logits([r]), whole[2 * i:2 * i + 2])
    eng.close()


def test_encoder_tilings_agree(lh):
    eng = lh.Engine(lh.Gguf.from_bytes(lh.SynthImage("laya-english", seed=31, n_layers=4)))
    rng = np.random.default_rng(9)
    inputs = [(rng.integers(0, 1000, n).astype(np.int32), [0, n - 1], n % 3) for n in (2, 17, 32, 33, 63, 64, 65, 81, 129, 193, 300, 511)]
    whole = eng.laya_forward(inputs * 8)
    for i, x in enumerate(inputs):
        print(f"encoder {len(x[0])} tokens alone", flush=True)
        (logits, act), = eng.laya_forward([x])
        assert_bits_equal(np.asarray(logits), np.asarray(whole[i][0]))
        assert_bits_equal(np.asarray(act), np.asarray(whole[i][1]))
    eng.close()


def test_long_vocabulary_argmax(lh):
    """Vocabularies of 65,536 entries and more take the argmax in two launches: each decoded token is the first
    maximum of its step's logits, and the next step continues from it (a run equals single steps)."""
    eng = lh.Engine(lh.Gguf.from_bytes(lh.SynthImage("q4km-7b", seed=3, n_layers=1)), kv_tokens=4096)
    ids = np.random.default_rng(3).integers(0, 1000, 70).astype(np.int32)
    runs = []
    for single in (False, True):
        s = eng.seq_create()
        eng.forward(s, ids, [len(ids) - 1], vocab_ids=[0])
        if single:
            tok, toks = 5, []
            for _ in range(6):
                t, logits = eng.decode(s, tok, 1, want_logits=True)
                tok = int(t[-1])
                assert tok == int(np.argmax(logits[0]))
                toks.append(tok)
            runs.append(toks)
        else:
            runs.append([int(t) for t in eng.decode(s, 5, 6)])
        eng.seq_free(s)
    assert runs[0] == runs[1]
    eng.close()


@pytest.mark.parametrize("preset, layers, counts", [
    ("f16-7b", 1, (4 * (528,), 8 * (512,), 8 * (672,), 2 * (1640,))), ("q8-2048", 1, (4 * (410,), 7 * (401, 431), 2 * (1600,))),
    ("q4km-7b", 1, (10 * (440,) + 3 * (131,),)), ("laya-english", 1, (13 * (479,) + 21 * (45,),))])
def test_qkv_rule_rows(lh, preset, layers, counts):
    """Row counts where the rotating q|k|v launch goes from the 64-column tiles to the 256 x 256 ones, or to f32 rows and a RoPE
    pass (1,640 F16 rows alone): a request's bits do not change with the launch that its batch takes."""
    eng = lh.Engine(lh.Gguf.from_bytes(lh.SynthImage(preset, seed=31, n_layers=layers)), kv_tokens=16384)
    rng = np.random.default_rng(11)

    def run(requests):
        if preset.startswith("laya"):
            return [np.concatenate([np.ravel(x) for x in o]) for o in eng.laya_forward([(r, [0, len(r) - 1], 1) for r in requests])]
        seqs = [eng.seq_create() for _ in requests]
        out = eng.batch([(s, r, [len(r) - 1]) for s, r in zip(seqs, requests)]).run(np.arange(16, dtype=np.int32))[0]
        for s in seqs:
            eng.seq_free(s)
        return list(out)

    for lengths in counts:
        ids = [rng.integers(0, 1000, n).astype(np.int32) for n in lengths]
        whole = run(ids)
        for i in (0, len(ids) // 2, len(ids) - 1):
            print(f"{preset} {sum(lengths)} rows, request {i}", flush=True)
            assert_bits_equal(run([ids[i]])[0], whole[i])
    eng.close()


def test_head_dim_64_rows(lh):
    """A head_dim 64 decoder of width 2048: its requests rotate in the q|k|v GEMM, its large batches take the 256 x 256 GEMM and
    a RoPE pass (the rotating epilogue of that kernel is head_dim 128's), with the same bits."""
    from decoder_image import image
    eng = lh.Engine(lh.Gguf.from_bytes(image(2048, 32, 8, 64, 1024, 512, 1024)), kv_tokens=16384)
    rng = np.random.default_rng(5)
    options = np.arange(16, dtype=np.int32)

    def run(requests):
        eng.profile_reset()
        seqs = [eng.seq_create() for _ in requests]
        out = eng.batch([(s, r, [len(r) - 1]) for s, r in zip(seqs, requests)]).run(options)[0]
        for s in seqs:
            eng.seq_free(s)
        return out, eng.profile_read("rope_kv")["launches"]

    eng.profile(True)
    for lengths in (16 * (512,), 9 * (467, 443)):
        ids = [rng.integers(0, 512, n).astype(np.int32) for n in lengths]
        print(f"head_dim 64, {sum(lengths)} rows", flush=True)
        whole, passes = run(ids)
        assert passes == 1
        for i in (0, len(ids) - 1):
            one, passes = run([ids[i]])
            assert passes == 0
            assert_bits_equal(one[0], whole[i])
    eng.close()


@pytest.mark.parametrize("zeroed", [0, 40000])
def test_long_argmax_ties(lh, zeroed):
    """Equal maxima in several of the 64 ranges of a long vocabulary: the first one wins (src/models/openthai/decision.rs:330-335).
    With the rows below 40,000 zeroed, which ends inside a range, it is token 0 or 40,000 by the sign of the others."""
    from decoder_image import image
    V, d = 66048, 256
    head = np.tile(np.random.default_rng(2).standard_normal(d) * 0.05, (V, 1))
    head[:zeroed] = 0
    eng = lh.Engine(lh.Gguf.from_bytes(image(d, 2, 1, 128, 256, V, 256, replace={"output.weight": head})), kv_tokens=512)
    s = eng.seq_create()
    eng.forward(s, [3, 4, 5], [2], [0])
    toks, logits = eng.decode(s, 6, 6, want_logits=True)
    for t, z in zip(toks, logits):
        assert (z[zeroed:] == z[V - 1]).all() and z[V - 1] != 0
        assert int(t) == (zeroed if z[V - 1] > 0 else 0) == int(np.argmax(z))
    eng.close()


def test_long_argmax_non_finite(lh):
    """A long vocabulary whose maximum is infinite has no token: the decode fails and the engine stays usable."""
    from decoder_image import image
    V, d = 66048, 256
    head = np.random.default_rng(3).standard_normal((V, d)) * 0.05
    head[50000, 0], head[50001, 0] = np.inf, -np.inf  # one of the two is +inf whatever the sign of its input
    eng = lh.Engine(lh.Gguf.from_bytes(image(d, 2, 1, 128, 256, V, 256, replace={"output.weight": head})), kv_tokens=512)
    s = eng.seq_create()
    eng.forward(s, [3, 4, 5], [2], [0])
    with pytest.raises(lh.LayaError, match="non-finite model output"):
        eng.decode(s, 6, 3)
    assert eng.seq_len(s) == 3
    assert np.isfinite(eng.forward(s, [7, 8], [1], [1, 2])).all()
    eng.close()


@pytest.mark.parametrize("preset, precision", [("plumbing-f16", 0), ("q8-2048", 2), ("q4km-7b", 0)])
@pytest.mark.parametrize("prefix", [5, 37, 100])
def test_attention_tiles_behind_a_prefix(lh, preset, precision, prefix):
    """Requests behind a cached prefix that ends inside a page and inside a tile: alone they take 16-row attention tiles, in a
    batch 32-row ones, with the same bits."""
    eng = lh.Engine(lh.Gguf.from_bytes(lh.SynthImage(preset, seed=31, n_layers=1)), kv_tokens=32768,
                    precision=lh.PREC_KV16 if precision else lh.PREC_EXACT)
    rng = np.random.default_rng(prefix)
    base = eng.seq_create()
    eng.forward(base, rng.integers(0, 1000, prefix).astype(np.int32), [0], vocab_ids=[0])
    ids = [rng.integers(0, 1000, n).astype(np.int32) for n in (1, 15, 16, 17, 31, 33, 64, 97, 300)]
    options = np.arange(16, dtype=np.int32)

    def run(requests):
        seqs = [eng.seq_fork(base, prefix) for _ in requests]
        out = eng.batch([(s, r, [len(r) // 2, len(r) - 1] if len(r) > 1 else [0]) for s, r in zip(seqs, requests)]).run(options)[0]
        for s in seqs:
            eng.seq_free(s)
        return out

    whole, at = run(ids * 8), 0
    for r in ids:
        n = 2 if len(r) > 1 else 1
        print(f"{preset} {len(r)} tokens behind {prefix}", flush=True)
        assert_bits_equal(run([r]), whole[at:at + n])
        at += n
    eng.close()
