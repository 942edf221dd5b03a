"""GPU parity of the attention half for a prompt's worth of tokens (llmp_attn_block_batch with the
tiled projections of proj_gemm_kernels.h, from 136 tokens, and the 16-token groups of one launch
below) against sequential oracle calls, at the bars of test_block_batch_gpu: every weight format,
tile edges (rows no multiple of 64, columns no multiple of 128, tokens around a tile of 128),
mixes in one launch, the epilogues, and inputs and weights far from fp16's range."""
import ctypes as C

import numpy as np
import pytest

from llmplayer_amd import _lib
from llmplayer_amd import hip_forward_pass as hfp
from oracle import oracle as orc
from tests import ggml_pack as gp
from tests.test_block_gpu import NAMES, TYPES
from tests import test_block_batch_gpu as tbb
from tests.test_block_batch_gpu import _run_batch

pytestmark = pytest.mark.gpu


def _config(hq=8, hkv=2, d=64, **k):
    return hfp.ModelConfig(hq, hkv, d, 1, architecture=hfp.ARCH_LLAMA, rope_freq_base=500000.0, **k)


@pytest.mark.parametrize("t", TYPES, ids=[NAMES[t] for t in TYPES])
def test_prompt_every_weight_format(t):
    _run_batch(_config(), 512, 160, 3, 137, (t,) * 4, seed=900 + t, what=f"prompt {NAMES[t]}", batched=True)


@pytest.mark.parametrize("K", [136, 255, 256, 257])
def test_prompt_tile_edges_in_tokens(K):
    q4, q6 = gp.GGML_Q4_K, gp.GGML_Q6_K
    _run_batch(_config(), 512, 270, 0, K, (q4, q4, q6, q4), seed=K, what=f"prompt {K} tokens", batched=True)


@pytest.mark.parametrize("t", [gp.GGML_Q8_0, gp.GGML_F32, gp.GGML_BF16], ids=["q8_0", "f32", "bf16"])
def test_prompt_rows_and_columns_off_the_tile(t):
    # 288 projection rows (4.5 tiles of 64), 352 columns (2.75 chunks of 128)
    _run_batch(_config(3, 3, 96), 352, 200, 10, 150, (t,) * 4, seed=41 + t, what="prompt 288 x 352", batched=True)


@pytest.mark.parametrize("types", [(gp.GGML_Q6_K, gp.GGML_Q6_K, gp.GGML_Q4_K, gp.GGML_Q6_K),
                                   (gp.GGML_Q3_K, gp.GGML_Q3_K, gp.GGML_Q5_K, gp.GGML_Q5_K),
                                   (gp.GGML_Q8_0, gp.GGML_Q4_0, gp.GGML_F16, gp.GGML_Q4_K)],
                         ids=["swapped pair", "q3_k_l", "three launches"])
def test_prompt_mixes_biases_post_norm_scale(types):
    _run_batch(_config(), 768, 200, 0, 140, types, seed=sum(types), what="prompt mix", bias=True, post=True,
               rscale=0.7, batched=True)


@pytest.mark.parametrize("K", [31, 33, 64, 130])
def test_groups_of_16_in_one_launch(K):
    q4, q6 = gp.GGML_Q4_K, gp.GGML_Q6_K
    _run_batch(_config(), 512, 160, 7, K, (q4, q4, q6, q4), seed=K, what=f"groups, {K} tokens")


@pytest.mark.parametrize("K", [33, 100])
def test_groups_of_16_in_one_launch_q8_1_input(K):
    _run_batch(_config(), 512, 160, 7, K, (gp.GGML_Q4_K,) * 4, seed=K, what=f"Q8_1 groups, {K} tokens", q8=True)


def test_groups_of_16_in_one_launch_append_what_single_groups_append():
    """The Q8_1 mode at 150 tokens: K and V rows equal, bit for bit, to those of calls of 16."""
    c, dim, K = _config(), 512, 150
    rng = np.random.default_rng(8)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K, gp.GGML_Q4_K, gp.GGML_Q6_K, gp.GGML_Q4_K), rng)
    rows = []
    for step in (K, 16):
        with hfp.HipForwardPass(c, K) as fp:
            fp.setBlockConfig(dim, input_mode=_lib.LLMP_INPUT_Q8_1)
            fp.uploadLayerWeights(0, lw)
            for t in range(0, K, step):
                fp.uploadXBatch(x[t:t + step])
                fp.forwardAttentionBlockBatch(0, t, len(x[t:t + step]))
            rows.append(fp.kv.read(0, 0, K))
    for a, b in zip(*rows):
        np.testing.assert_array_equal(a, b)


def test_prompt_inputs_near_the_largest_float():
    """A token with a value whose product with the norm weight exceeds fp32's range, as its square
    does: its RMSNorm factor is 0 and so are its V rows; those of the others stay bit for bit."""
    c, dim, K = _config(), 512, 140
    rng = np.random.default_rng(2)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    lw.attnNorm = np.full(dim, 1.5, np.float32)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    rows = []
    for big in (1.0, 3e38):
        x[5, 7] = np.float32(big)
        with hfp.HipForwardPass(c, K) as fp:
            fp.setBlockConfig(dim)
            fp.uploadLayerWeights(0, lw)
            fp.uploadXBatch(x)
            fp.forwardAttentionBlockBatch(0, 0, K)
            rows.append(fp.kv.read(0, 0, K)[1])
    assert (rows[1][5] == 0).all()
    np.testing.assert_array_equal(np.delete(rows[0], 5, 0), np.delete(rows[1], 5, 0))


@pytest.mark.parametrize("xs,ws", [(1e6, 1e-6), (1e-20, 1.0), (1.0, 3e4)])
def test_prompt_far_from_fp16_range(xs, ws):
    """F32 projections: y = W x to 2^-18 of sum |W||x| per element, whatever their scales (fp32
    sums of hi/lo products hold ~2^-21)."""
    c = _config()
    dim, K = 512, 140
    rng = np.random.default_rng(3)
    def mat(r, n, s):
        return (rng.standard_normal((r, n)) * s / np.sqrt(n)).astype(np.float32)
    def tensor(w):
        return hfp.GgufTensor(gp.GGML_F32, w.shape[0], w.shape[1], w.view(np.uint8).reshape(-1))
    wv = mat(c.kv_dim, dim, ws)
    zero = np.zeros((c.q_dim, dim), np.float32)
    x = (rng.standard_normal((K, dim)) * xs).astype(np.float32)
    with hfp.HipForwardPass(c, K) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, hfp.TransformerLayerWeights(
            wq=tensor(zero), wk=tensor(zero[:c.kv_dim]), wv=tensor(wv), wo=tensor(mat(dim, c.q_dim, 1.0))))
        fp.uploadXBatch(x)
        fp.forwardAttentionBlockBatch(0, 0, K)
        _, v = fp.kv.read(0, 0, K)
    want = x.astype(np.float64) @ wv.T.astype(np.float64)
    bar = 2.0 ** -18 * (np.abs(x).astype(np.float64) @ np.abs(wv.T).astype(np.float64))
    assert np.isfinite(v).all() and (np.abs(v - want) <= bar).all()


@pytest.mark.parametrize("t", TYPES, ids=[NAMES[t] for t in TYPES])
def test_prompt_projections_are_no_less_precise_than_the_groups(t):
    """V rows (a projection as it is stored) of one tiled call against those of calls of 80 tokens in
    groups of 16: no further from 64 bits (5 % for the spread over 16384 values)."""
    c, dim, K = _config(4, 2, 128), 1024, 160
    rng = np.random.default_rng(50 + t)
    lw, bw = tbb._weights(c, dim, (t,) * 4, rng, pre=False)
    w = orc.dequant_rows(t, bw.wv, c.kv_dim, dim).astype(np.float64)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    want = x.astype(np.float64) @ w.T
    err = []
    for step in (K, K // 2):
        with hfp.HipForwardPass(c, K) as fp:
            fp.setBlockConfig(dim)
            fp.uploadLayerWeights(0, lw)
            for t0 in range(0, K, step):
                fp.uploadXBatch(x[t0:t0 + step])
                fp.forwardAttentionBlockBatch(0, t0, step)
            err.append(np.linalg.norm(fp.kv.read(0, 0, K)[1] - want) / np.linalg.norm(want))
    assert err[0] <= 1.05 * err[1], err


def test_prompt_all_zero_blocks_of_any_exponent():
    """MXFP4 blocks of zeros with the largest finite exponent beside ordinary ones."""
    c, dim, K = _config(), 512, 140
    rng = np.random.default_rng(9)
    lw, bw = tbb._weights(c, dim, (gp.GGML_MXFP4,) * 4, rng, pre=False)
    wb = bw.wv.reshape(c.kv_dim, dim // 32, 17).copy()
    wb[:, 3] = 0
    wb[:, 3, 0] = 254                                    # E8M0 byte, then 16 bytes of codes
    lw.wv = hfp.GgufTensor(gp.GGML_MXFP4, c.kv_dim, dim, wb.reshape(-1))
    w = orc.dequant_rows(gp.GGML_MXFP4, wb.reshape(c.kv_dim, -1), c.kv_dim, dim).astype(np.float64)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    with hfp.HipForwardPass(c, K) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, lw)
        fp.uploadXBatch(x)
        fp.forwardAttentionBlockBatch(0, 0, K)
        v = fp.kv.read(0, 0, K)[1]
    want = x.astype(np.float64) @ w.T
    bar = 2.0 ** -18 * (np.abs(x).astype(np.float64) @ np.abs(w.T))
    assert np.isfinite(v).all() and (np.abs(v - want) <= bar).all()


def test_graph_of_a_short_call_outlives_the_growth_of_the_scratch():
    """A captured 16-token call and a captured 20-token call replay what they computed after a
    call that needs far more scratch and attention workspace."""
    c, dim = _config(), 512
    rng = np.random.default_rng(21)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    x = rng.standard_normal((600, dim)).astype(np.float32)
    with hfp.HipForwardPass(c, 600) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, lw)
        bufs = [hfp.DeviceBuffer(n * dim * 4) for n in (16, 20, 600)]
        try:
            def put():
                for b in bufs:
                    b.upload(x[:b.nbytes // (4 * dim)])
            graphs, want = [], []
            for b, n in ((bufs[0], 16), (bufs[1], 20)):
                put()
                _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, 0, n, b.ptr, 0)
                want.append(b.download(np.float32))
                g = C.c_uint64()
                _lib.call("llmp_graph_begin", 0)
                _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, 0, n, b.ptr, 0)
                _lib.call("llmp_graph_end", 0, C.byref(g))
                graphs.append(g.value)
            _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, 0, 600, bufs[2].ptr, 0)
            for _ in range(3):
                put()
                for g, b, w in zip(graphs, bufs, want):
                    _lib.call("llmp_graph_launch", g, 0)
                    np.testing.assert_array_equal(b.download(np.float32), w)
            for g in graphs:
                _lib.call("llmp_graph_destroy", g)
        finally:
            for b in bufs:
                b.free()


@pytest.mark.parametrize("n,block", [(17, True), (16, True), (33, True), (16, False)],
                         ids=["17 tokens", "16 tokens", "33 tokens", "16 tokens, attention alone"])
def test_graph_outlives_the_growth_of_the_split_workspace(n, block):
    """A captured call after 200 rows (two or three key splits) replays what it computed after
    16-token calls at later positions, whose many splits need larger partials, and after new
    allocations of the partials' size."""
    c, dim, pos0, last = _config(), 512, 200, 3900
    rng = np.random.default_rng(31)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    proj = [rng.standard_normal(n * w).astype(np.float32) for w in (c.q_dim, c.kv_dim, c.kv_dim)]
    with hfp.HipForwardPass(c, last + 16) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, lw)
        fp.kv.write(0, 0, *(rng.standard_normal((last, c.kv_dim)).astype(np.float32) for _ in range(2)))
        qkv = [hfp.DeviceBuffer(a.nbytes) for a in proj]
        buf = hfp.DeviceBuffer(n * max(dim, c.q_dim) * 4)
        fill = []
        try:
            for b, a in zip(qkv, proj):
                b.upload(a)

            def put():
                buf.upload(x if block else np.zeros((n, c.q_dim), np.float32))

            def call(pos, k):
                if block:
                    _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, pos, k, buf.ptr, 0)
                else:
                    _lib.call("llmp_attn_prefill_f32", fp.kv.handle, 0, pos, k, *(b.ptr for b in qkv), 0, buf.ptr, 0)
            put()
            call(pos0, n)
            want = buf.download(np.float32)
            g = C.c_uint64()
            _lib.call("llmp_graph_begin", 0)
            call(pos0, n)
            _lib.call("llmp_graph_end", 0, C.byref(g))
            for later in (900, 2000, last):
                call(later, 16)
                fill.append(hfp.DeviceBuffer(1 << 20))
                fill[-1].upload(np.full(1 << 18, np.nan, np.float32))
                put()
                _lib.call("llmp_graph_launch", g.value, 0)
                np.testing.assert_array_equal(buf.download(np.float32), want)
            _lib.call("llmp_graph_destroy", g.value)
        finally:
            for b in qkv + [buf] + fill:
                b.free()


@pytest.mark.parametrize("first", [(0, 300), (900, 40)])
def test_capture_beyond_the_prepared_workspaces_runs_in_groups(first):
    """A captured call of more tokens, or at a later position, than the eager calls before it had:
    in groups of 16 if a workspace would have to grow, with the eager call's result to rounding."""
    c, dim, pos0, K = _config(), 512, 600, 300
    rng = np.random.default_rng(22)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    with hfp.HipForwardPass(c, 1000) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, lw)
        rows = rng.standard_normal((2, 1000, c.kv_dim)).astype(np.float32)
        fp.kv.write(0, 0, rows[0], rows[1])
        buf = hfp.DeviceBuffer(x.nbytes)
        try:
            def call(pos, n):
                _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, pos, n, buf.ptr, 0)
            buf.upload(x)
            call(*first)
            call(pos0 + K - 16, 16)   # the groups' own workspaces
            fp.kv.write(0, 0, rows[0], rows[1])
            g = C.c_uint64()
            _lib.call("llmp_graph_begin", 0)
            call(pos0, K)
            _lib.call("llmp_graph_end", 0, C.byref(g))
            got = []
            for _ in range(3):
                buf.upload(x)
                _lib.call("llmp_graph_launch", g.value, 0)
                _lib.call("llmp_stream_sync", 0)
                got.append(buf.download(np.float32, x.size))
                buf.upload(x)
                call(pos0, K)
            want = buf.download(np.float32, x.size)
            _lib.call("llmp_graph_destroy", g.value)
        finally:
            buf.free()
    for y in got:   # fp32 sums in another order: the bar of the batched blocks
        assert np.abs(y - want).max() <= 1e-4


@pytest.mark.parametrize("n", [17, 33])
def test_captured_call_with_a_last_group_of_one_token(n):
    """Captured after an eager call of 35 tokens at the same position, where n - 1 tokens take more
    key splits than 35: replays equal to the eager call to rounding (in groups of 16 where the
    larger partials are missing), and to each other."""
    c = hfp.ModelConfig(24, 8, 128, 1, architecture=hfp.ARCH_LLAMA, rope_freq_base=500000.0)
    dim, pos0 = 512, 8000
    rng = np.random.default_rng(6)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    x = rng.standard_normal((35, dim)).astype(np.float32)
    with hfp.HipForwardPass(c, pos0 + 35) as fp:
        fp.setBlockConfig(dim)
        fp.uploadLayerWeights(0, lw)
        fp.kv.write(0, 0, *(rng.standard_normal((pos0, c.kv_dim)).astype(np.float32) for _ in range(2)))
        buf = hfp.DeviceBuffer(x.nbytes)
        try:
            def call(k):
                _lib.call("llmp_attn_block_batch", fp.kv.handle, 0, pos0, k, buf.ptr, 0)
            buf.upload(x)
            call(35)
            g = C.c_uint64()
            _lib.call("llmp_graph_begin", 0)
            call(n)
            _lib.call("llmp_graph_end", 0, C.byref(g))
            buf.upload(x)
            call(n)
            want = buf.download(np.float32, n * dim)
            got = []
            for _ in range(3):
                buf.upload(x)
                _lib.call("llmp_graph_launch", g.value, 0)
                got.append(buf.download(np.float32, n * dim))
                call(35)
            _lib.call("llmp_graph_destroy", g.value)
        finally:
            buf.free()
    assert np.abs(got[0] - want).max() <= 1e-4   # the bar of the batched blocks
    assert np.array_equal(got[1], got[0]) and np.array_equal(got[2], got[0])


def test_a_layer_captured_before_it_ever_ran_takes_the_tiled_projections():
    """Two layers of the same weights: the captured call of the one that never ran replays, bit for
    bit, what the other's eager call computed."""
    c = hfp.ModelConfig(8, 2, 64, 2, architecture=hfp.ARCH_LLAMA, rope_freq_base=500000.0)
    dim, K = 512, 300
    rng = np.random.default_rng(4)
    lw, _ = tbb._weights(c, dim, (gp.GGML_Q4_K,) * 4, rng)
    x = rng.standard_normal((K, dim)).astype(np.float32)
    with hfp.HipForwardPass(c, K) as fp:
        fp.setBlockConfig(dim)
        for layer in (0, 1):
            fp.uploadLayerWeights(layer, lw)
        buf = hfp.DeviceBuffer(x.nbytes)
        try:
            def call(layer):
                _lib.call("llmp_attn_block_batch", fp.kv.handle, layer, 0, K, buf.ptr, 0)
            buf.upload(x)
            call(0)   # the handle's scratch and workspaces
            want = buf.download(np.float32)
            g = C.c_uint64()
            _lib.call("llmp_graph_begin", 0)
            call(1)
            _lib.call("llmp_graph_end", 0, C.byref(g))
            for _ in range(3):
                buf.upload(x)
                _lib.call("llmp_graph_launch", g.value, 0)
                np.testing.assert_array_equal(buf.download(np.float32), want)
                call(0)
            _lib.call("llmp_graph_destroy", g.value)
        finally:
            buf.free()
