"""GPU parity of the wide multi-token attention (prefill_wide_kernels.h) against P sequential
decodes of the oracle, at the edges of its launch forms: blocks in pairs (even and odd counts),
key halves with one and with several key splits, one block per workgroup (many blocks), each with a
window too; ragged lengths, soft-cap, sinks, the output gate, virtual KV heads, partial RoPE,
head_dim 96, and Q8_0 rows.  Each case names the form it is for, and fails if the library's plan takes
another.

Bar: output max-abs <= 1e-4 (and <= 1e-4 + 1e-3*|ref|), the cache bit-identical."""
import numpy as np
import pytest

from llmplayer_amd import _lib
from llmplayer_amd import hip_forward_pass as hfp
from oracle import oracle as orc
from tests import decode_cases as dc
from tests.host_driver import wide_form

pytestmark = pytest.mark.gpu

LLAMA, QWEN3, GEMMA2, GEMMA3 = hfp.ARCH_LLAMA, hfp.ARCH_QWEN3, hfp.ARCH_GEMMA2, hfp.ARCH_GEMMA3
CAP = {"attn_logit_soft_cap": 50.0}

# (hq, hkv, d, arch, extra ModelConfig fields, layer, pos0, P, QK-norm, sinks, gate, form)
CASES = {
    "halves, one split": (24, 8, 128, LLAMA, {}, 0, 0, 1000, False, False, False, "halves"),
    "halves, full grid": (24, 8, 128, LLAMA, {}, 0, 37, 1301, False, False, False, "halves"),
    "pairs, odd block count": (24, 8, 128, LLAMA, {}, 0, 5, 1560, False, False, False, "pairs"),
    "one block per workgroup": (32, 8, 64, LLAMA, {}, 0, 3, 4101, False, False, False, "one"),
    "halves, key splits": (24, 8, 128, LLAMA, {}, 0, 3001, 97, False, False, False, "splits"),
    "group 2, QK-norm, NEOX": (16, 8, 128, QWEN3, {}, 0, 1501, 777, True, False, False, "splits"),
    "group 8, sinks": (64, 8, 64, LLAMA, {}, 0, 61, 701, False, True, False, "pairs"),
    "window, soft-cap": (16, 4, 128, GEMMA2, {"sliding_window": 300, **CAP}, 0, 90, 1403, False, False, False, "halves"),
    "global layer, soft-cap": (16, 4, 128, GEMMA2, {"sliding_window": 300, **CAP}, 1, 90, 1403, False, False, False,
                               "halves"),
    "window shorter than a tile": (32, 8, 64, GEMMA3, {"sliding_window": 60}, 0, 700, 4100, True, False, False, "one"),
    "window, one block per workgroup, soft-cap": (16, 4, 128, GEMMA2, {"sliding_window": 300, **CAP}, 0, 37, 4200, False,
                                                  False, False, "one"),
    "window, pairs, soft-cap": (16, 4, 128, GEMMA2, {"sliding_window": 300, **CAP}, 0, 700, 2400, False, False, False,
                                "pairs"),
    # the last block has one token and fewer key tiles than the light blocks paired with it
    "window, pairs, light block the longer": (16, 16, 128, GEMMA2, {"sliding_window": 300}, 0, 700, 2177, False, False,
                                              False, "pairs"),
    "window, key splits, soft-cap": (24, 8, 128, GEMMA2, {"sliding_window": 1500, **CAP}, 0, 3001, 120, False, False,
                                     False, "splits"),
    "gate, two virtual KV heads": (32, 2, 128, LLAMA, {}, 0, 500, 601, False, False, True, "halves"),
    "gate, sinks, key splits": (24, 8, 128, LLAMA, {}, 0, 2990, 133, False, True, True, "splits"),
    "head_dim 96, NEOX": (32, 32, 96, LLAMA, {"rope_type": _lib.LLMP_ROPE_NEOX}, 0, 0, 1001, False, False, False, "halves"),
    "partial NEOX": (24, 8, 128, LLAMA, {"rope_type": _lib.LLMP_ROPE_NEOX, "rope_dim_count": 40}, 0, 11,
                     900, True, False, False, "halves"),
    "partial pairs": (24, 8, 128, LLAMA, {"rope_dim_count": 52}, 0, 0, 900, False, False, False, "halves"),
}


@pytest.mark.parametrize("name", list(CASES))
def test_wide_prefill_matches_sequential_decodes(name):
    hq, hkv, d, arch, extra, layer, pos0, P, qkn, sinks, gated, form = CASES[name]
    c = hfp.ModelConfig(hq, hkv, d, layer + 1, architecture=arch, rope_freq_base=500000.0, **extra)
    assert wide_form(c, layer, pos0, P) == form
    rng = np.random.default_rng(77 + P)
    max_seq = pos0 + P
    kc = np.zeros((max_seq, c.kv_dim), np.float32)
    vc = np.zeros_like(kc)
    kc[:pos0] = rng.standard_normal((pos0, c.kv_dim), dtype=np.float32)
    vc[:pos0] = rng.standard_normal((pos0, c.kv_dim), dtype=np.float32)
    q, k, v = (rng.standard_normal((P, n), dtype=np.float32) for n in (c.q_dim, c.kv_dim, c.kv_dim))
    qk = tuple(rng.uniform(0.5, 1.5, d).astype(np.float32) for _ in range(2)) if qkn else None
    sk = rng.standard_normal(hq).astype(np.float32) if sinks else None
    gate = rng.uniform(-5, 5, (P, c.q_dim)).astype(np.float32) if gated else None
    with hfp.HipForwardPass(c, max_seq, qk_norm=[qk] * c.block_count if qkn else None,
                            sinks=[sk] * c.block_count if sinks else None) as fp:
        fp.kv.write(layer, 0, kc, vc)
        dc.log(f"[gpu] wide prefill {name}: {hq}/{hkv}/{d} pos0={pos0} P={P}")
        got = fp.prefill(layer, pos0, q, k, v, gate=gate)
        cs, sn = dc.oracle_tables(c, max_seq, layer)
        qw, kw = qk if qk is not None else (None, None)
        want = orc.prefill_sequential(dc.oracle_config(c, max_seq, sk), kc, vc, q, k, v, layer, pos0,
                                      qnorm_w=qw, knorm_w=kw, rope_cos=cs, rope_sin=sn, n_threads=16, gate=gate)
        dc.compare_out(got.reshape(-1), want.reshape(-1), name)
        dc.compare_cache(fp, layer, kc, vc, name + " cache")


def test_wide_prefill_over_q8_rows_equals_dequantised_rows():
    """Q8_0 rows and the same values in an fp32 cache give the same attention: the images hold
    quant * scale either way, and the new rows' values are the quantised ones in both."""
    c = hfp.ModelConfig(24, 8, 128, 1, architecture=LLAMA, rope_freq_base=500000.0)
    pos0, P = 2000, 300
    rng = np.random.default_rng(5)
    nb = c.kv_dim // 32
    qs = [rng.integers(-127, 128, (pos0, c.kv_dim), dtype=np.int8) for _ in range(2)]
    sc = [rng.uniform(0.005, 0.02, (pos0, nb)).astype(np.float32) for _ in range(2)]
    q, k, v = (rng.standard_normal((P, n), dtype=np.float32) for n in (c.q_dim, c.kv_dim, c.kv_dim))
    with hfp.HipForwardPass(c, pos0 + P, kv_dtype=_lib.LLMP_KV_Q8_0) as f8, hfp.HipForwardPass(c, pos0 + P) as f32:
        f8.kv.write_q8(0, 0, qs[0], sc[0], qs[1], sc[1])
        got = f8.prefill(0, pos0, q, k, v)
        kq, ks, vq, vs = f8.kv.read_q8(0, 0, pos0 + P)
        rows = [(a.reshape(-1, nb, 32).astype(np.float32) * s[..., None]).reshape(-1, c.kv_dim)
                for a, s in ((kq, ks), (vq, vs))]
        f32.kv.write(0, 0, *rows)
        # the same queries over the same values, as a shared-KV call: nothing is appended
        dq, do = hfp.DeviceBuffer(q.nbytes), hfp.DeviceBuffer(q.nbytes)
        try:
            dq.upload(q)
            _lib.call("llmp_attn_prefill_shared_f32", f32.kv.handle, 0, 0, pos0, P, dq.ptr, 0, do.ptr, 0)
            want = do.download(np.float32, q.size)
        finally:
            dq.free()
            do.free()
    np.testing.assert_array_equal(got.reshape(-1), want)


def test_wide_prefill_keeps_heads_and_tokens_apart_in_range():
    """Queries of 1e9 in one head, and in some tokens of another, leave the rest of the outputs as
    they are without them.  Bar: 2e-6, outputs of at most ~2 over sums of 2^-22 products; only the
    shared running maxima of a wave may move."""
    c = hfp.ModelConfig(24, 8, 128, 1, architecture=LLAMA, rope_freq_base=500000.0)
    pos0, P, big = 2000, 300, np.float32(1e9)
    rng = np.random.default_rng(1)
    q, k, v = (rng.standard_normal((P, n), dtype=np.float32) for n in (c.q_dim, c.kv_dim, c.kv_dim))
    rows = [rng.standard_normal((pos0, c.kv_dim), dtype=np.float32) for _ in range(2)]
    scaled = np.zeros((P, 24), bool)
    scaled[:, 3] = True
    scaled[::7, 10] = True
    q2 = (q.reshape(P, 24, 128) * np.where(scaled, big, np.float32(1))[..., None]).reshape(P, -1)
    out = []
    for x in (q, q2):
        with hfp.HipForwardPass(c, pos0 + P) as fp:
            fp.kv.write(0, 0, *rows)
            out.append(fp.prefill(0, pos0, x, k, v).reshape(P, 24, 128))
    assert np.isfinite(out[1]).all()
    assert np.abs(out[0] - out[1])[~scaled].max() <= 2e-6
