"""The grouped GEMMs at the edges of their row tiles: 256 rows, and 128 rows where
the weights are MXFP4 and there are tiles enough; weights read through the caches
and past them (few rows per expert and more than 256 MiB of matrices in the handle);
full, half and quarter column tiles.

Bars as in test_gpu_parity.py: max-abs 2e-2 and rel-L2 1e-3 of the oracle on the
same inputs; the two weight formats, whose tiles differ, bit for bit."""
import numpy as np
import pytest

from gpt_oss_amd import abi, synth
from oracle import binding as ob

pytestmark = pytest.mark.gpu

E = 32
FEW = (1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 255, 256, 257)  # 1823 rows: 57 per expert
MANY = FEW + (288, 383, 384, 385, 512, 513, 640, 800, 1024)  # 6752 rows: 211 per expert


@pytest.mark.parametrize("rows", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("H,IM", [(64, 2048), (128, 2112), (192, 2080)])
def test_row_tiles(rows, H, IM):
    rng = np.random.default_rng(H + len(rows))
    experts = rng.permutation(E)[:len(rows)]
    ids = np.repeat(experts, rows).astype(np.int32)
    T = -(-len(ids) // 4)
    ids = rng.permutation(np.concatenate([ids, np.full(4 * T - len(ids), -1, np.int32)])).reshape(T, 4)
    tv = rng.random((T, 4)).astype(np.float32)
    sh = synth.LayerShape("tiles", T, H, IM, E)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    dx, dti = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(ids)
    dtv, dout = abi.DevBuf.from_numpy(tv), abi.DevBuf(T * H * 4)
    got = []
    many = int((256 << 20) / (3 * H * IM * E * 17 / 32)) + 1  # MXFP4 layers from which the weights are read past the caches
    for fp4, layers in ((True, 1), (False, 1), (True, many), (False, many * 17 // 64 + 1)):
        m = abi.Moe(H, IM, E, max_tokens=T, swiglu_limit=sh.limit, layers=layers)
        for i in range(layers):
            if fp4:
                m.upload_layer_mxfp4(i, wr, br, b1k, s1, b1, b2k, s2, b2)
            else:
                m.upload_layer(i, wr, br, w1, b1, w2, b2)
        dout.memset(0xFF)
        m.experts(0, dx, None, dti, dtv, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
        # stage by stage: the dispatch does not know the layer
        dout.memset(0xFF)
        m.dispatch(dti, None, T)
        m.expert_gemms(0, dx, T)
        m.combine(dtv, None, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
        m.close()
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    # a token of every expert at least, and those of the tiles' last rows
    some = np.unique(np.concatenate([np.nonzero((ids == e).any(1))[0][[0, -1]] for e in experts]))
    want = np.zeros((len(some), H), np.float32)
    for i, t in enumerate(some):
        for k, e in enumerate(ids[t]):
            if e >= 0:
                want[i] += tv[t, k] * ob.expert_token(x[t], w1[e], b1[e], w2[e], b2[e], sh.limit,
                                                      mode=ob.ROUND_ACT_BF16)
    d = got[0][some] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("n_experts,IM,T", [(16, 2880, 735), (16, 2880, 736), (32, 2048, 768), (32, 2048, 769),
                                            (32, 2048, 1280), (32, 2048, 1281), (32, 2048, 2048), (32, 2048, 2049)])
def test_sides_of_the_lines(n_experts, IM, T):
    """Tiles of 128 rows under MXFP4 weights (16 experts, 23 column tiles, 735 and 736
    tokens) and either side of the lines up to which weights that exceed 256 MiB are
    read past the caches (96 rows per expert in tiles of 128, 256 in tiles of 256):
    the two weight formats bit for bit, and the oracle."""
    H = 64
    sh = synth.LayerShape("lines", T, H, IM, n_experts)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    many = int((256 << 20) / (3 * H * IM * n_experts * 17 / 32)) + 1
    got = []
    for fp4, layers in ((True, many), (False, many * 17 // 64 + 1)):
        m = abi.Moe(H, IM, n_experts, max_tokens=T, swiglu_limit=sh.limit, layers=layers)
        for i in range(layers):
            if fp4:
                m.upload_layer_mxfp4(i, wr, br, b1k, s1, b1, b2k, s2, b2)
            else:
                m.upload_layer(i, wr, br, w1, b1, w2, b2)
        got.append(abi.run_layer(m, layers - 1, x, None)["out"])
        m.close()
    assert np.array_equal(got[0], got[1])
    rows = np.arange(0, T, T // 15)
    want = ob.moe_layer(np.ascontiguousarray(x[rows]), None, wr, br, w1, b1, w2, b2, 4, sh.limit,
                        mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
    d = got[0][rows] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("H,IM", [(64, 64), (256, 320), (448, 64), (320, 384), (576, 448)])
def test_reduction_depths(H, IM):
    """Reductions of 1 to 9 double steps of 64, shorter and longer than the rings of
    the loads in front of them, under row tiles of 1 to 8 blocks and full, three-quarter,
    half and quarter column tiles: the weight formats bit for bit, and the oracle."""
    rng = np.random.default_rng(H + IM)
    rows = rng.permutation([1, 33, 65, 97, 129, 161, 193, 225, 256, 300, 385, 15])
    n_experts = len(rows)
    ids = np.repeat(np.arange(n_experts), rows).astype(np.int32)
    T = -(-len(ids) // 4)
    ids = rng.permutation(np.concatenate([ids, np.full(4 * T - len(ids), -1, np.int32)])).reshape(T, 4)
    tv = rng.random((T, 4)).astype(np.float32)
    sh = synth.LayerShape("depths", T, H, IM, n_experts)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    dx, dti = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(ids)
    dtv, dout = abi.DevBuf.from_numpy(tv), abi.DevBuf(T * H * 4)
    got = []
    for fp4 in (True, False):
        m = abi.Moe(H, IM, n_experts, max_tokens=T, swiglu_limit=sh.limit)
        if fp4:
            m.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
        else:
            m.upload_layer(0, wr, br, w1, b1, w2, b2)
        for _ in range(3):
            dout.memset(0xFF)
            m.experts(0, dx, None, dti, dtv, T, dout)
            abi.sync()
            got.append(dout.download((T, H), np.float32))
        m.close()
    # a handle with layers of both formats: the dispatch plans tiles of 256 rows for either
    m = abi.Moe(H, IM, n_experts, max_tokens=T, swiglu_limit=sh.limit, layers=2)
    m.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
    m.upload_layer(1, wr, br, w1, b1, w2, b2)
    for layer in (0, 1):
        dout.memset(0xFF)
        m.dispatch(dti, None, T)
        m.expert_gemms(layer, dx, T)
        m.combine(dtv, None, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
    m.close()
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    some = np.unique(np.concatenate([np.nonzero((ids == e).any(1))[0][[0, -1]] for e in range(n_experts)]))
    want = np.zeros((len(some), H), np.float32)
    for i, t in enumerate(some):
        for k, e in enumerate(ids[t]):
            if e >= 0:
                want[i] += tv[t, k] * ob.expert_token(x[t], w1[e], b1[e], w2[e], b2[e], sh.limit,
                                                      mode=ob.ROUND_ACT_BF16)
    d = got[0][some] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("n_experts,H,IM,T", [(16, 64, 2880, 255), (16, 64, 2880, 256), (8, 64, 2880, 256), (8, 64, 2880, 257),
                                              (8, 512, 512, 1927), (8, 512, 512, 1928), (8, 512, 512, 3856)])
def test_sides_of_the_product_lines(n_experts, H, IM, T):
    """Either side of the lines between the products of the MXFP4 kernels (64 rows per
    expert, and 128 where there is at most a workgroup per CU) and between row tiles of 128
    and 256 rows under bf16 weights: the two weight formats, which cross none of these
    together, bit for bit, stage by stage as well, and the oracle."""
    sh = synth.LayerShape("products", T, H, IM, n_experts)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
    dti, dtv, dout = abi.DevBuf(T * 16), abi.DevBuf(T * 16), abi.DevBuf(T * H * 4)
    got = []
    for fp4 in (True, False):
        m = abi.Moe(H, IM, n_experts, max_tokens=T, swiglu_limit=sh.limit)
        if fp4:
            m.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
        else:
            m.upload_layer(0, wr, br, w1, b1, w2, b2)
        got.append(abi.run_layer(m, 0, x, None)["out"])
        m.router(0, dx, None, T, None, dti, dtv)
        m.dispatch(dti, None, T)
        m.expert_gemms(0, dx, T)
        m.combine(dtv, None, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
        m.close()
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    rows = np.arange(0, T, max(1, T // 15))
    want = ob.moe_layer(np.ascontiguousarray(x[rows]), None, wr, br, w1, b1, w2, b2, 4, sh.limit,
                        mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
    d = got[0][rows] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)
