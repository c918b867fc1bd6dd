"""F16 decoder images of any shape, for dispatch edges that no preset reaches (tests only)."""
import numpy as np

import gguf_writer as gw


def image(d, hq, hkv, hd, f, vocab, ctx, layers=1, seed=1, replace=None):
    """GGUF bytes of a decoder with normal F16 matrices (sigma 0.02) and unit norms; `replace` maps a tensor's name to the
    array that takes its place (rows x cols)."""
    rng = np.random.default_rng(seed)
    dims = dict(block_count=layers, embedding_length=d, head_count=hq, head_count_kv=hkv, key_length=hd, feed_forward_length=f,
                vocab_size=vocab, context_length=ctx)
    meta = [("general.architecture", gw.STR, "ggmlc"), ("laya.model_name", gw.STR, "laya-decoder")]
    meta += [("laya.decoder." + k, gw.U32, v) for k, v in dims.items()]
    meta.append(("laya.decoder.layer_norm_rms_epsilon", gw.F32, 1e-5))
    angle = np.arange(ctx)[:, None] * 1e4 ** (-2.0 * (np.arange(hd) % (hd // 2)) / hd)[None, :]
    tensors = [(n, [a.size] if a.ndim == 1 else a.shape[::-1], 0, gw.f32_bytes(a)) for n, a in
               [("cos_full", np.cos(angle)), ("sin_full", np.sin(angle)), ("final_norm.weight", np.ones(d))] +
               [(f"{n}_norm.{i}.weight", np.ones(d)) for i in range(layers) for n in ("attn", "ffn")]]
    shapes = {"tok_emb.weight": (vocab, d), "output.weight": (vocab, d)}
    for i in range(layers):
        shapes.update({f"qkv.{i}.weight": ((hq + 2 * hkv) * hd, d), f"wo.{i}.weight": (d, hq * hd),
                       f"mlp_wi.{i}.weight": (2 * f, d), f"mlp_wo.{i}.weight": (d, f)})
    for name, shape in shapes.items():
        w = (replace or {}).get(name)
        w = rng.standard_normal(shape, dtype=np.float32) * 0.02 if w is None else w
        assert w.shape == shape, name
        tensors.append((name, list(shape[::-1]), 1, gw.f16_bytes(w)))
    return gw.build(meta, tensors)
