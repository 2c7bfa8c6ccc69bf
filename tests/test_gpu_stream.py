"""The kernels of the batches in which the weights are a stream (stream.hip) at
the sizes where they can go wrong: one row, a group of 16 rows and one more, a
tile of 32 and one more, an expert with several tiles, with and without a plan;
reductions with fewer steps than slices and with slices of unequal length; an odd
number of column pairs where a wave takes two.

Bars as in test_gpu_parity.py: max-abs 2e-2 and rel-L2 1e-3 of the oracle on the
same bf16 inputs; the two weight formats bit for bit."""
import numpy as np
import pytest

from gpt_oss_amd import abi, synth
from oracle import binding as ob

pytestmark = pytest.mark.gpu

W = ("w_router", "b_router", "w_mlp1", "b_mlp1", "w_mlp2", "b_mlp2")


def past_the_caches(sh, fp4):
    """Layers of this shape from which a handle holds more than 256 MiB of expert
    matrices, which are then read past the caches."""
    return int((256 << 20) / (3 * sh.hidden * sh.inter * sh.experts * (17 / 32 if fp4 else 2))) + 1


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64, 65, 128, 150])
@pytest.mark.parametrize("H,IM", [(64, 64), (192, 320), (704, 64)])
def test_rows_of_an_expert(rows, H, IM):
    """Every token names the experts 2, 30, 31 and 0: each has all the rows."""
    E = 32
    sh = synth.LayerShape("rows", rows, H, IM, E)
    L = {k: (synth.round_bf16(v) if v.dtype == np.float32 else v) for k, v in synth.make_layer(sh, seed=rows).items()}
    m = abi.Moe(H, IM, E, max_tokens=rows, swiglu_limit=sh.limit)
    m.upload_layer(0, *[L[k] for k in W])
    ids = [2, 30, 31, 0]
    ti = np.tile(np.array(ids, np.int32), (rows, 1))
    tv = np.random.default_rng(rows).random((rows, 4)).astype(np.float32)
    want = np.zeros((rows, H), np.float32)
    for t in range(rows):
        for k, e in enumerate(ids):
            want[t] += tv[t, k] * ob.expert_token(L["x"][t], L["w_mlp1"][e], L["b_mlp1"][e], L["w_mlp2"][e],
                                                  L["b_mlp2"][e], sh.limit, mode=ob.ROUND_ACT_BF16)
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"]))
    dti, dtv, dout = abi.DevBuf.from_numpy(ti), abi.DevBuf.from_numpy(tv), abi.DevBuf(rows * H * 4)
    first = None
    for distinct in (True, False):  # up to 64 tokens: without a plan, and with one
        m.set_distinct_ids(distinct)
        dout.memset(0xFF)
        m.experts(0, dx, None, dti, dtv, rows, dout)
        abi.sync()
        got = dout.download((rows, H), np.float32)
        assert np.abs(got - want).max() <= 2e-2 and np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
        first = got if first is None else first
        assert np.array_equal(got, first)
    m.close()


@pytest.mark.parametrize("T", [2, 24, 40, 65])
def test_two_pairs_of_columns_per_wave(T):
    """128 experts and nine pairs of columns: MXFP4 waves take two pairs each
    from 25 tokens on (the last of a row has one), one pair up to 24."""
    sh = synth.LayerShape("pairs", T, 576, 576, 128)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    m4 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=T, swiglu_limit=sh.limit)
    m4.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
    m16 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=T, swiglu_limit=sh.limit)
    m16.upload_layer(0, wr, br, w1, b1, w2, b2)
    a, b = abi.run_layer(m4, 0, x, None), abi.run_layer(m16, 0, x, None)
    assert np.array_equal(a["topk_i"], b["topk_i"]) and np.array_equal(a["out"], b["out"])
    rows = np.arange(min(T, 16))
    want = ob.moe_layer(np.ascontiguousarray(x[rows]), None, wr, br, w1, b1, w2, b2, 4, sh.limit,
                        mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
    got = a["out"][rows]
    assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    m4.close()
    m16.close()


def test_hot_experts_under_a_plan():
    """512 tokens over 128 experts, most rows at a few of them: experts of two and
    of many row blocks, one of them on both sides of the 64th block, single blocks
    between them; column tiles that are no multiple of the eight XCDs, an odd number
    of pairs.  MXFP4 (two pairs per wave) and bf16 (one), through the caches and past
    them, bit for bit, and the oracle at the first and last token of every expert."""
    E, H, IM, T = 128, 704, 384, 512
    counts = {**{e: 33 for e in range(30)}, 30: 290, 31: 1, 32: 16, 33: 17, 34: 32, 35: 64, 100: 138, 127: 500}
    assert sum(counts.values()) == 4 * T
    rng = np.random.default_rng(12)
    ids = rng.permutation(np.repeat(list(counts), list(counts.values())).astype(np.int32)).reshape(T, 4)
    tv = rng.random((T, 4)).astype(np.float32)
    sh = synth.LayerShape("hot", T, H, IM, E)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    dx, dti = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(ids)
    dtv, dout = abi.DevBuf.from_numpy(tv), abi.DevBuf(T * H * 4)
    got = []
    for fp4, layers in ((True, 1), (False, 1), (True, past_the_caches(sh, True)), (False, past_the_caches(sh, False))):
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
        m.close()
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    some = np.unique(np.concatenate([np.nonzero((ids == e).any(1))[0][[0, -1]] for e in counts]))
    want = np.zeros((len(some), H), np.float32)
    for i, t in enumerate(some):
        for k, e in enumerate(ids[t]):
            want[i] += tv[t, k] * ob.expert_token(x[t], w1[e], b1[e], w2[e], b2[e], sh.limit, mode=ob.ROUND_ACT_BF16)
    d = got[0][some] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("E,H,IM", [(32, 1728, 896), (8, 4416, 2240)])
def test_tiles_of_both_formats(E, H, IM):
    """Sizes at which an MXFP4 wave takes two pairs of columns (the down GEMM's last one
    has one) and batches in which experts have one tile of rows, two tiles, and none
    between them; a repeated expert that has 64 rows in a batch of 16 tokens; inactive
    rows.  Without a plan and with one, MXFP4 (through the caches and past them) and
    bf16: the same bits; the oracle at the first and last rows and around the 16th
    and 32nd."""
    sh = synth.LayerShape("both", 64, H, IM, E)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    many = past_the_caches(sh, True)
    assert many > 1 and past_the_caches(sh, False) == 1
    m4, m16 = (abi.Moe(H, IM, E, max_tokens=64, swiglu_limit=sh.limit) for _ in range(2))
    m4s = abi.Moe(H, IM, E, max_tokens=64, swiglu_limit=sh.limit, layers=many)
    m4.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
    for i in range(many):
        m4s.upload_layer_mxfp4(i, wr, br, b1k, s1, b1, b2k, s2, b2)
    m16.upload_layer(0, wr, br, w1, b1, w2, b2)
    rng = np.random.default_rng(E)
    dx, dout = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf(64 * H * 4)

    def skewed(T):  # expert 3 in every token, 5 in most, two of the rest
        ids = np.stack([rng.permutation([e for e in range(E) if e not in (3, 5)])[:4] for _ in range(T)]).astype(np.int32)
        ids[:, 1] = 3
        ids[rng.permutation(T)[:T * 3 // 4], 2] = 5
        return ids

    one = np.full((16, 4), E - 1, np.int32)
    for ids in [skewed(T) for T in (16, 17, 32, 33, 48, 64)] + [one]:
        T = len(ids)
        tv = rng.random((T, 4)).astype(np.float32)
        pos = np.zeros(T, np.int32)
        if T == 48:
            pos[4::7] = -1
        dti, dtv, dpos = (abi.DevBuf.from_numpy(a) for a in (ids, tv, pos))
        first = None
        for m in (m4, m4s, m16):
            for distinct in ((False,) if ids is one else (True, False)):
                m.set_distinct_ids(distinct)
                dout.memset(0xFF)
                m.experts(0, dx, dpos, dti, dtv, T, dout)
                abi.sync()
                got = dout.download((T, H), np.float32)
                first = got if first is None else first
                assert np.array_equal(got, first), (T, distinct)
            m.dispatch(dti, dpos, T)  # with a plan also where moe_experts has none
            m.expert_gemms(0, dx, T)
            dout.memset(0xFF)
            m.combine(dtv, dpos, T, dout)
            abi.sync()
            assert np.array_equal(dout.download((T, H), np.float32), first), T
        assert np.all(first[pos < 0] == 0)
        some = [t for t in sorted({0, 15, 16, 31, 32, T - 1}) if t < T and pos[t] >= 0]
        want = np.zeros((len(some), H), np.float32)
        for i, t in enumerate(some):
            y = {e: ob.expert_token(x[t], w1[e], b1[e], w2[e], b2[e], sh.limit, mode=ob.ROUND_ACT_BF16) for e in set(ids[t])}
            for k, e in enumerate(ids[t]):
                want[i] += tv[t, k] * y[e]
        d = first[some] - want
        assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max())), T
        assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want), T
    for m in (m4, m4s, m16):
        m.close()


def test_activation_past_4_gib():
    """256 experts with fixed slots of 64 rows and an intermediate size at which the
    last slot lies past 4 GiB of the activation: the first and the last expert (all
    have the same matrices) give the oracle's rows.  The down GEMM's sums of 131616
    products are compared at the bars above, which scale with the rows."""
    E, H, IM, T = 256, 32, 131616, 3
    assert (E - 1) * 64 * (IM // 64 * 64 + 64) * 2 > 2**32
    rng = np.random.default_rng(5)

    def codes(rows, cols, exp):
        return (rng.integers(0, 256, (1, rows, cols // 32, 16), dtype=np.uint8),
                rng.integers(exp, exp + 3, (1, rows, cols // 32), dtype=np.uint8))

    (b1k, s1), (b2k, s2) = codes(2 * IM, H, 122), codes(H, IM, 114)
    b1 = synth.round_bf16(rng.standard_normal((1, 2 * IM)).astype(np.float32) * 0.1)
    b2 = synth.round_bf16(rng.standard_normal((1, H)).astype(np.float32) * 0.1)
    x = synth.round_bf16(rng.standard_normal((T, H)).astype(np.float32))

    def each(a):
        return np.repeat(a, E, axis=0)

    m = abi.Moe(H, IM, E, max_tokens=T, swiglu_limit=7.0)
    m.upload_layer_mxfp4(0, np.zeros((E, H), np.float32), np.zeros(E, np.float32), each(b1k), each(s1), each(b1),
                         each(b2k), each(s2), each(b2))
    m.set_distinct_ids(True)
    w1, w2 = ob.mxfp4_dequant(b1k, s1)[0], ob.mxfp4_dequant(b2k, s2)[0]
    rows = np.stack([ob.expert_token(x[t], w1, b1[0], w2, b2[0], 7.0, mode=ob.ROUND_ACT_BF16) for t in range(T)])
    tv = np.array([[0.1, 0.2, 0.3, 0.4]] * T, np.float32)
    dx, dtv, dout = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(tv), abi.DevBuf(T * H * 4)
    got = []
    for ids in ([0, 1, 2, 3], [255, 254, 253, 252], [0, 255, 128, 64]):
        dti = abi.DevBuf.from_numpy(np.array([ids] * T, np.int32))
        dout.memset(0xFF)
        m.experts(0, dx, None, dti, dtv, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
        d = got[-1] - rows
        assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(rows), ids
        assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(rows).max())), ids
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    m.close()
