"""Stage-level parity of the HIP path through the C-ABI: the stage entry points
compose to the whole layer, the SwiGLU's clamp points, adversarial router
inputs (near ties, exact ties, NaN rows), the error bound of the router's first
pass, and repeatability of the large-batch kernels.

Bars as in test_gpu_parity.py: ids, offsets and permutations bit-exact; outputs
within max-abs 2e-2 and rel-L2 1e-3 of the oracle on the same bf16 inputs."""
import numpy as np
import pytest

from gpt_oss_amd import abi, synth
from oracle import binding as ob

pytestmark = pytest.mark.gpu

W = ("w_router", "b_router", "w_mlp1", "b_mlp1", "w_mlp2", "b_mlp2")
BF16_ULP = 2.0 ** -7  # spacing of bf16 values relative to the value, at most


def bf16_layer(shape, tokens=None, seed=0):
    L = synth.make_layer(shape, seed=seed, tokens=tokens)
    return {k: (synth.round_bf16(v) if v.dtype == np.float32 else v) for k, v in L.items()}


def make_moe(shape, L, max_tokens):
    m = abi.Moe(shape.hidden, shape.inter, shape.experts, max_tokens=max_tokens, swiglu_limit=shape.limit)
    m.upload_layer(0, *[L[k] for k in W])
    return m


def next_bf16(a, steps=1):
    """The bf16 value `steps` ulps further from zero."""
    bits = synth.to_bf16_bits(a).astype(np.int32) + steps
    return synth.from_bf16_bits(bits.astype(np.uint16))


# ---------------- stage entry points ----------------

@pytest.mark.parametrize("T", [40, 700, 3000])
def test_stage_entry_points_compose(T):
    """moe_router -> moe_dispatch -> moe_expert_gemms -> moe_combine gives the
    bits of moe_forward, with and without accumulation, and the combine stage is
    the weighted sum of the per-assignment rows in slot order."""
    sh = synth.LayerShape("s", T, 320, 128, 13)
    L = bf16_layer(sh, seed=5)
    m = make_moe(sh, L, T)
    m.set_distinct_ids(True)  # the router's ids are four different experts per token
    pos = np.zeros(T, np.int32)
    pos[3::7] = -1
    base = abi.run_layer(m, 0, L["x"], pos)
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"]))
    dpos = abi.DevBuf.from_numpy(pos)
    dti, dtv = abi.DevBuf(T * 16), abi.DevBuf(T * 16)
    prior = np.random.default_rng(T).standard_normal((T, sh.hidden)).astype(np.float32)
    dout, dacc = abi.DevBuf(T * sh.hidden * 4), abi.DevBuf.from_numpy(prior)
    m.router(0, dx, dpos, T, None, dti, dtv)
    with pytest.raises(abi.MoeError) as e:  # no dispatch of this batch yet
        m.expert_gemms(0, dx, T)
    assert e.value.code == -5
    m.dispatch(dti, dpos, T)
    with pytest.raises(abi.MoeError) as e:  # the GEMMs have not run on this dispatch: y is stale
        m.combine(dtv, dpos, T, dout, accumulate=False)
    assert e.value.code == -5
    m.expert_gemms(0, dx, T)
    m.combine(dtv, dpos, T, dout, accumulate=False)
    m.combine(dtv, dpos, T, dacc, accumulate=True)
    abi.sync()
    assert np.array_equal(dout.download((T, sh.hidden), np.float32), base["out"])
    acc = dacc.download((T, sh.hidden), np.float32)
    assert np.array_equal(acc[pos < 0], prior[pos < 0])
    np.testing.assert_allclose(acc[pos >= 0], prior[pos >= 0] + base["out"][pos >= 0], rtol=0, atol=1e-6)
    # a whole-layer call takes the plan over: the stage calls need a new dispatch
    m.forward(0, dx, dpos, T, dout)
    with pytest.raises(abi.MoeError):
        m.combine(dtv, dpos, T, dout)


@pytest.mark.parametrize("T", [17, 40, 64, 65])
def test_caller_routing_with_distinct_ids(T):
    """moe_set_distinct_ids: with the promise that a token's ids are four
    different experts, moe_experts bounds the rows per expert by T as
    moe_forward does and needs no dispatch pass up to 64 tokens: the bits of
    moe_forward.  Without it the bound is 4 T and the same kernels run on a plan:
    the same bits, too."""
    sh = synth.LayerShape("d", T, 2880, 320, 32)
    L = bf16_layer(sh, seed=8)
    m = make_moe(sh, L, 128)
    pos = np.zeros(T, np.int32)
    pos[2::5] = -1
    base = abi.run_layer(m, 0, L["x"], pos)
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"]))
    dpos = abi.DevBuf.from_numpy(pos)
    dti, dtv = abi.DevBuf.from_numpy(base["topk_i"]), abi.DevBuf.from_numpy(base["topk_v"])
    dout = abi.DevBuf(T * sh.hidden * 4)
    def same(got, distinct):
        assert np.array_equal(got, base["out"]), f"distinct={distinct}"

    for distinct in (False, True, False):
        m.set_distinct_ids(distinct)
        dout.memset(0xFF)
        m.experts(0, dx, dpos, dti, dtv, T, dout)
        abi.sync()
        same(dout.download((T, sh.hidden), np.float32), distinct)
        m.dispatch(dti, dpos, T)
        m.expert_gemms(0, dx, T)
        dout.memset(0xFF)
        m.combine(dtv, dpos, T, dout)
        abi.sync()
        same(dout.download((T, sh.hidden), np.float32), distinct)
    # ids that break the promise must not fault: one expert in all four slots of every token
    m.set_distinct_ids(True)
    bad = np.full((T, 4), 3, np.int32)
    m.experts(0, dx, None, abi.DevBuf.from_numpy(bad), dtv, T, dout)
    abi.sync()


def test_reference_7m_model_shape():
    """The reference's smallest model (export_model_bin/gpt-oss-7m/config.json:
    hidden 32, intermediate 64, 32 experts): sizes that are multiples of 32 but
    not of 64 are padded inside the library.  Whole layer, FFN block and MXFP4
    upload against the oracle; batches on both sides of 64 tokens."""
    for H, IM, E in ((32, 64, 32), (96, 96, 32), (32, 32, 8)):
        for T in (1, 50, 64, 300, 1100):
            sh = synth.LayerShape("7m", T, H, IM, E)
            L = bf16_layer(sh, seed=H + T)
            m = make_moe(sh, L, T)
            pos = np.zeros(T, np.int32)
            pos[1::6] = -1
            for p in (None, pos):
                R = abi.run_layer(m, 0, L["x"], p)
                _, ti, _ = ob.router(L["x"], p, L["w_router"], L["b_router"], 4)
                off, perm, _ = ob.dispatch(ti, p, E)
                case = f"H={H} IM={IM} E={E} T={T} masked={p is not None}"
                assert np.array_equal(R["topk_i"], ti), case
                assert np.array_equal(R["offsets"], off) and np.array_equal(R["perm"][:off[-1]], perm), case
                rows = np.arange(min(T, 48))
                want = ob.moe_layer(np.ascontiguousarray(L["x"][rows]), None if p is None else np.ascontiguousarray(p[rows]),
                                    *[L[k] for k in W], 4, sh.limit, mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
                assert np.abs(R["out"][rows] - want).max() <= 2e-2, case
                assert np.linalg.norm(R["out"][rows] - want) <= 1e-3 * np.linalg.norm(want), case
            # the FFN block in place on the bf16 stream
            rng = np.random.default_rng(T)
            rw = synth.round_bf16((1 + 0.1 * rng.standard_normal(H)).astype(np.float32))
            m.upload_norm(0, rw)
            dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"]))
            m.block_forward(0, dx, abi.DevBuf.from_numpy(pos), T)
            abi.sync()
            got = synth.from_bf16_bits(dx.download((T, H), np.uint16))
            rows = np.arange(min(T, 32))
            want, _ = ob.ffn_block(np.ascontiguousarray(L["x"][rows]), np.ascontiguousarray(pos[rows]), rw,
                                   *[L[k] for k in W], 4, sh.limit, mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
            assert np.all(np.abs(got[rows] - want) <= 2e-2 + 2.0 ** -7 * np.abs(want)), f"block H={H} T={T}"
            assert np.array_equal(got[pos < 0], L["x"][pos < 0])
            m.close()
    # MXFP4 upload at sizes that need padding: bit-identical to uploading the decoded matrices
    sh = synth.LayerShape("7q", 200, 96, 96, 8)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    m4 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=sh.tokens)
    m4.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
    m32 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=sh.tokens)
    m32.upload_layer(0, wr, br, w1, b1, w2, b2)
    for T in (200, 40):
        a, b = abi.run_layer(m4, 0, x[:T], None), abi.run_layer(m32, 0, x[:T], None)
        assert np.array_equal(a["out"], b["out"]) and np.isfinite(a["out"]).all()
    with pytest.raises(abi.MoeError) as e:
        abi.Moe(48, 64, 8, max_tokens=16)  # not a multiple of 32
    assert e.value.code == -2


def test_yardsticks_run():
    """The measured denominators the benchmark reports: a register-resident MFMA
    loop and plain streams through HBM.  Sanity only: positive, below the
    published peaks, zeros no slower than random operands."""
    tf, ghz = abi.yardstick_mfma(256, 2000, data=1)
    tf2, _ = abi.yardstick_mfma(256, 2000, data=2)
    tf0, _ = abi.yardstick_mfma(256, 2000, data=0)
    assert 200 < tf < 2600 and 200 < tf2 < 2600 and 0.5 < ghz < 3.0 and tf0 > 0.9 * tf
    c, r = abi.yardstick_hbm(1 << 28, 3)
    assert 500 < c < 8200 and 500 < r < 8200


def test_swiglu_clamp_points():
    """The clamp points of run.cpp:709-726 through moe_experts: W1 = 0 so the
    biases are the gate and up values, W2 = I so the activation is the output.
    The gate is clamped from above only, the up value on both sides; a very
    negative gate gives ~0 rather than being clamped to -limit."""
    H = IM = 64
    E, T = 4, 40
    w1 = np.zeros((E, 2 * IM, H), np.float32)
    w2 = np.tile(np.eye(H, IM, dtype=np.float32), (E, 1, 1))
    b2 = np.zeros((E, H), np.float32)
    b1 = np.zeros((E, 2 * IM), np.float32)
    b1[0, 0:2] = (9.0, 0.5)     # gate above the limit -> 7
    b1[0, 2:4] = (1.0, 9.0)     # up above the limit -> 7
    b1[0, 4:6] = (1.0, -9.0)    # up below -limit -> -7
    b1[0, 6:8] = (-30.0, 2.0)   # very negative gate: not clamped from below, ~0
    b1[0, 8:10] = (-9.0, 1.0)   # gate below -limit stays -9
    b1[0, 10:12] = (7.0, 7.0)   # exactly at the limit
    b1[0, 12:14] = (6.96875, -7.0)
    m = abi.Moe(H, IM, E, max_tokens=T, swiglu_limit=7.0)
    m.upload_layer(0, np.zeros((E, H), np.float32), np.zeros(E, np.float32), w1, b1, w2, b2)
    x = synth.round_bf16(np.random.default_rng(0).standard_normal((T, H)).astype(np.float32))
    ti = np.tile(np.arange(4, dtype=np.int32), (T, 1))
    tv = np.tile(np.array([1, 0, 0, 0], np.float32), (T, 1))
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
    dout = abi.DevBuf(T * H * 4)
    m.experts(0, dx, None, abi.DevBuf.from_numpy(ti), abi.DevBuf.from_numpy(tv), T, dout)
    abi.sync()
    y = dout.download((T, H), np.float32)
    assert np.array_equal(y, np.tile(y[0], (T, 1)))  # W1 = 0: every token sees the same values
    sig = lambda g: 1.0 / (1.0 + np.exp(-1.702 * g))
    want = [7 * sig(7) * 1.5, 1 * sig(1) * 8.0, 1 * sig(1) * -6.0, None, -9 * sig(-9) * 2.0,
            7 * sig(7) * 8.0, 6.96875 * sig(6.96875) * -6.0]
    for j, wv in enumerate(want):
        if wv is None:
            assert abs(y[0, j]) < 1e-18
        else:  # the activation is rounded to bf16 (matmul.cpp:1427)
            np.testing.assert_allclose(y[0, j], wv, rtol=BF16_ULP)
    assert np.all(y[0, len(want):] == 0)
    # and against the oracle's own expert with the same rounding point
    yo = ob.expert_token(x[0], w1[0], b1[0], w2[0], b2[0], 7.0, mode=ob.ROUND_ACT_BF16)
    np.testing.assert_allclose(y[0], yo, rtol=BF16_ULP, atol=1e-30)


# ---------------- router: adversarial inputs ----------------

def _check_ids(m, L, x, pos, E):
    R = abi.run_layer(m, 0, x, pos)
    score, ti, tv = ob.router(x, pos, L["w_router"], L["b_router"], 4)
    assert np.array_equal(R["topk_i"], ti), "expert ids differ from the oracle"
    np.testing.assert_allclose(R["topk_v"], tv, rtol=0, atol=1e-6)
    act = np.ones(x.shape[0], bool) if pos is None else pos >= 0
    # logits of experts the router did not have to recompute exactly are its
    # first-pass values: 2e-6, or two float steps of the value where that is more
    np.testing.assert_allclose(R["score"][act], score[act], rtol=2.0 ** -22, atol=2e-6)
    return R, score, ti


@pytest.mark.parametrize("E,T", [(32, 2048), (128, 1000), (128, 4111), (256, 300)])
def test_router_near_ties(E, T):
    """Logits one bf16 step of one weight apart, and exactly
    equal ones, at the top of every token's ranking: the first pass of the
    router cannot separate them, the ids must still be the oracle's."""
    H = 2880
    sh = synth.LayerShape("nt", T, H, 64, E)
    L = bf16_layer(sh, seed=11)
    rng = np.random.default_rng(E)
    wr, br = L["w_router"].copy(), L["b_router"].copy()
    base = wr[5].copy()
    group = [1, 5, 6, 9, 17, 20, E - 1, E - 2]
    for n, e in enumerate(group):
        wr[e] = base
        br[e] = 8.0  # lifts the whole group to the top of every token
        if n >= 2:   # experts 1 and 5 stay exactly equal; the others move one weight by one step
            k = int(rng.integers(H))
            wr[e, k] = next_bf16(wr[e, k:k + 1], steps=1 if n % 2 else -1)[0]
    L["w_router"], L["b_router"] = wr, br
    m = make_moe(sh, L, T)
    pos = np.zeros(T, np.int32)
    pos[4::13] = -1
    R, score, ti = _check_ids(m, L, L["x"], pos, E)
    act = pos >= 0
    assert np.isin(ti[act], group).all()  # the test is about the group
    top = np.sort(score[act][:, group], axis=1)[:, ::-1]
    assert np.median(top[:, 0] - top[:, 4]) < 2e-2  # and its members really are that close
    both = np.array([(1 in r) and (5 in r) for r in ti])
    assert both.any()
    for r in ti[both]:
        assert list(r).index(1) < list(r).index(5)  # exact tie: the lower id first


@pytest.mark.parametrize("E", [33, 63, 64, 65, 127, 128, 129, 200, 256])
def test_router_selection_of_many_experts(E):
    """Ranks over a whole wave: plateaus of equal logits at the first and the
    last experts, zeros of either sign, experts at minus infinity, rows of NaN (some NaNs: the next test); in
    moe_router's one launch and in the two of a whole layer (768 columns, from 65 experts on)."""
    H, T = 768, 40
    sh = synth.LayerShape("many", T, H, 64, E)
    L = bf16_layer(sh, seed=E)
    wr, br, x = L["w_router"].copy(), np.zeros(E, np.float32), L["x"].copy()
    x[3] = 0.0               # its logits are the biases
    x[::9] = 0.0
    wr[[0, 1, E - 2, E - 1]] = wr[7]
    wr[E // 2] = 0.0
    br[::3] = -0.0           # equal to 0, whatever the sign
    br[[4, E - 3]] = -np.inf
    x[20] = np.nan
    for bias in (br, np.full(E, -np.inf, np.float32), np.arange(E, dtype=np.float32) // 5):
        L["w_router"], L["b_router"], L["x"] = wr, synth.round_bf16(bias), x
        m = make_moe(sh, L, T)
        R = abi.run_layer(m, 0, x, None)
        _, ti, tv = ob.router(x, None, wr, L["b_router"], 4)
        assert np.array_equal(R["topk_i"], ti)
        np.testing.assert_allclose(R["topk_v"], tv, rtol=0, atol=2e-6)
        want = ob.moe_layer(x, None, wr, L["b_router"], L["w_mlp1"], L["b_mlp1"], L["w_mlp2"], L["b_mlp2"], 4, sh.limit,
                            mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
        assert np.array_equal(np.isnan(R["out"]), np.isnan(want))
        fine = ~np.isnan(want).any(1)
        if fine.any():
            assert np.abs(R["out"][fine] - want[fine]).max() <= 2e-2
            assert np.linalg.norm(R["out"][fine] - want[fine]) <= 1e-3 * np.linalg.norm(want[fine])
        m.close()


@pytest.mark.parametrize("E", [4, 5, 8, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200, 256])
def test_router_selection_beside_nans(E):
    """Some NaNs among a token's logits: one is chosen when every expert before it has been, and at no other time.
    From NaN biases, at the ends, in the middle, at even and odd places, next to experts that every token
    names, and at random; in tokens with an infinity also where its weight is zero.  The ids of moe_router and those
    that a whole layer ran on."""
    H, T = 768, 64
    rng = np.random.default_rng(E)
    sh = synth.LayerShape("nans", T, H, 64, E)
    L = bf16_layer(sh, seed=E)
    x, wr, br = L["x"].copy(), L["w_router"].copy(), L["b_router"]
    wr[::3, 5] = 0.0
    wr[1::3, 6] = 0.0
    x[::11, 5], x[1::11, 6], x[2::11, [5, 6]] = np.inf, -np.inf, np.inf
    sets = [[0], [1], [2], [3], [E - 1], [E // 2], [E // 2 + 1], [E // 3], [0, 1], [0, E - 1], range(0, E, 2), range(1, E, 2),
            range(3, E), range(E - 3), *(np.nonzero(rng.random(E) < p)[0] for p in (0.05, 0.05, 0.2, 0.5, 0.8))]
    L["x"], L["w_router"] = x, wr
    m = abi.Moe(H, 64, E, max_tokens=T, swiglu_limit=sh.limit)
    doff, dperm, dout = abi.DevBuf((E + 1) * 4), abi.DevBuf(T * 16), abi.DevBuf(T * H * 4)
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
    chosen = False
    for lift in (0.0, 64.0):  # 64: the first experts lead every token, in their order
        for nans in sets:
            L["b_router"] = br.copy()
            L["b_router"][:3] += lift * np.arange(3, 0, -1)
            L["b_router"][list(nans)] = np.nan
            L["b_router"] = synth.round_bf16(L["b_router"])
            m.upload_layer(0, *[L[k] for k in W])
            _, score, ti = _check_ids(m, L, x, None, E)
            chosen |= bool(np.isnan(np.take_along_axis(score, ti, 1)[:, 1:]).any())
            m.forward(0, dx, None, T, dout)
            m.get_dispatch(doff, dperm, T)
            abi.sync()
            off, perm, _ = ob.dispatch(ti, None, E)
            assert np.array_equal(doff.download((E + 1,), np.int32), off), (lift, list(nans))
            assert np.array_equal(dperm.download((T * 4,), np.int32), perm), (lift, list(nans))
    m.close()
    assert chosen


def test_router_first_pass_error_bound():
    """The first pass decides a token only when its logits are further apart
    than twice kGamma * |x| * max|w_e|; the scores it reports for experts it did
    not recompute must lie within that bound of the exact ones (they are in
    fact far inside it)."""
    E, T, H = 128, 3000, 2880
    sh = synth.LayerShape("eb", T, H, 64, E)
    L = bf16_layer(sh, seed=3)
    x = synth.round_bf16(L["x"] * np.random.default_rng(1).uniform(0.1, 30.0, (T, 1)).astype(np.float32))
    m = make_moe(sh, L, T)
    R, score, _ = _check_ids_loose(m, L, x, E)
    gamma = 2.0 * 33.0 * 2.0 ** -23  # router_gamma(1): a hand-over to fp64 after every MFMA
    bound = gamma * np.linalg.norm(x.astype(np.float64), axis=1) * np.linalg.norm(
        L["w_router"].astype(np.float64), axis=1).max()
    ratio = np.abs(R["score"].astype(np.float64) - score).max(axis=1) / bound
    print(f"first-pass error / proven bound: max {ratio.max():.3g}, median {np.median(ratio):.3g}")
    assert ratio.max() < 0.5


def _check_ids_loose(m, L, x, E):
    R = abi.run_layer(m, 0, x, None)
    score, ti, tv = ob.router(x, None, L["w_router"], L["b_router"], 4)
    assert np.array_equal(R["topk_i"], ti), "expert ids differ from the oracle"
    np.testing.assert_allclose(R["topk_v"], tv, rtol=0, atol=2e-5)  # rows scaled by up to 30
    return R, score, ti


def test_router_nan_row():
    """A row of NaN activations: every logit is NaN, no comparison succeeds and
    the reference's stable sort leaves the experts in index order (run.cpp:378-421),
    so the row goes to experts 0..3 and its output is NaN, as in the reference;
    the other rows are not disturbed."""
    sh = synth.LayerShape("nan", 100, 320, 128, 32)
    L = bf16_layer(sh, seed=9)
    m = make_moe(sh, L, sh.tokens)
    clean = abi.run_layer(m, 0, L["x"], None)
    x = L["x"].copy()
    x[37] = np.nan
    R = abi.run_layer(m, 0, x, None)
    _, ti, tv = ob.router(x, None, L["w_router"], L["b_router"], 4)
    assert list(ti[37]) == [0, 1, 2, 3] and np.isnan(tv[37]).all()
    assert np.array_equal(R["topk_i"], ti)
    assert np.isnan(R["topk_v"][37]).all() and np.isnan(R["out"][37]).all()
    keep = np.arange(sh.tokens) != 37
    assert np.array_equal(R["out"][keep], clean["out"][keep])
    off, perm, _ = ob.dispatch(ti, None, sh.experts)
    assert np.array_equal(R["offsets"], off) and np.array_equal(R["perm"][:off[-1]], perm)


# ---------------- repeatability of the large-batch kernels ----------------

def test_large_batches_repeat_bit_for_bit():
    """The GEMMs' main loop waits for its operands by counting outstanding loads (loads
    complete in issue order).  Twelve calls in a row must give the same bits, with bf16 and with
    MXFP4 weights: 4096 tokens at the 20B shape, which run every tile height and both narrow
    last column tiles (row split 2 in gate_up, 4 in down); 7168 tokens under Zipf routing (one
    expert with 28 row tiles of 256); 512 and 256 tokens, whose weights go past the caches; 200 tokens
    at 8 experts.  With MXFP4 these are all three of its tile kernels: tiles of 128 rows, two
    workgroups per CU, with either product, and tiles of 256.  So must the FFN block at 48 tokens."""
    sh = synth.CONFIGS["c2"]
    T = sh.tokens
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    m4 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=T, swiglu_limit=sh.limit)
    m4.upload_layer_mxfp4(0, wr, br, b1k, s1, b1, b2k, s2, b2)
    m16 = abi.Moe(sh.hidden, sh.inter, sh.experts, max_tokens=T, swiglu_limit=sh.limit)
    m16.upload_layer(0, wr, br, w1, b1, w2, b2)
    del w1, w2
    x = synth.round_bf16(synth.make_activations(sh, seed=1, tokens=T))
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
    dout = abi.DevBuf(T * sh.hidden * 4)
    first = None
    for m in (m16, m4):
        for i in range(12):
            dout.memset(0xFF)
            m.forward(0, dx, None, T, dout)
            abi.sync()
            got = dout.download((T, sh.hidden), np.float32)
            if first is None:
                first = got
                assert np.isfinite(got).all()
            assert np.array_equal(got, first), f"call {i}: a repeated call gave other bits"
    kernels = set()
    for few in (512, 256):
        for m, fp4 in ((m16, False), (m4, True)):
            kernels.add(abi.batch_kernel(sh.hidden, sh.inter, sh.experts, few, fp4)[:2])
            for i in range(12):
                dout.memset(0xFF)
                m.forward(0, dx, None, few, dout)
                abi.sync()
                got = dout.download((few, sh.hidden), np.float32)
                assert np.array_equal(got, first[:few]), f"{few} tokens, MXFP4 {fp4}, call {i}: other bits"
    # 8 experts: one workgroup per CU
    m8 = abi.Moe(sh.hidden, sh.inter, 8, max_tokens=200, swiglu_limit=sh.limit, layers=2)
    w1, w2 = ob.mxfp4_dequant(b1k[:8], s1[:8]), ob.mxfp4_dequant(b2k[:8], s2[:8])
    m8.upload_layer_mxfp4(0, wr[:8], br[:8], b1k[:8], s1[:8], b1[:8], b2k[:8], s2[:8], b2[:8])
    m8.upload_layer(1, wr[:8], br[:8], w1, b1[:8], w2, b2[:8])
    del w1, w2
    first8 = None
    for layer in (0, 1):
        kernels.add(abi.batch_kernel(sh.hidden, sh.inter, 8, 200, layer == 0, 2)[:2])
        for i in range(12):
            dout.memset(0xFF)
            m8.forward(layer, dx, None, 200, dout)
            abi.sync()
            got = dout.download((200, sh.hidden), np.float32)
            if first8 is None:
                first8 = got
                assert np.isfinite(got).all()
            assert np.array_equal(got, first8), f"8 experts, layer {layer}, call {i}: other bits"
    m8.close()
    assert kernels == {("bf16_gemm_kernel", 256), ("grouped_gemm_kernel", 128), ("grouped_gemm_kernel", 256),
                       ("fp4_gemm_kernel", 128)}
    # 7168 tokens with Zipf routing: up to 28 row tiles on one expert, the deepest XCD ranges
    z = synth.CONFIGS["c3b"]
    T3 = z.tokens
    m4.close()
    mz = abi.Moe(z.hidden, z.inter, z.experts, max_tokens=T3, swiglu_limit=z.limit, layers=2)
    wrz, brz = (synth.round_bf16(a) for a in synth.make_router(z))
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    mz.upload_layer(0, wrz, brz, w1, b1, w2, b2)
    mz.upload_layer_mxfp4(1, wrz, brz, b1k, s1, b1, b2k, s2, b2)
    del w1, w2
    xz = synth.round_bf16(synth.make_activations(z))
    dxz = abi.DevBuf.from_numpy(synth.to_bf16_bits(xz))
    doz = abi.DevBuf(T3 * z.hidden * 4)
    firstz = None
    for i in range(24):
        doz.memset(0xFF)
        mz.forward(i // 12, dxz, None, T3, doz)
        abi.sync()
        got = doz.download((T3, z.hidden), np.float32)
        if firstz is None:
            firstz = got
            assert np.isfinite(got).all()
        assert np.array_equal(got, firstz), f"7168 tokens, Zipf routing, call {i}: other bits"
    mz.close()
    del firstz, got
    rw = synth.round_bf16((1 + 0.1 * np.random.default_rng(2).standard_normal(sh.hidden)).astype(np.float32))
    m16.upload_norm(0, rw)
    ref = None
    for i in range(12):
        dxx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x[:48]))
        m16.block_forward(0, dxx, None, 48)
        abi.sync()
        got = dxx.download((48, sh.hidden), np.uint16)
        if ref is None:
            ref = got
        assert np.array_equal(got, ref), f"FFN block, call {i}: other bits"


# ---------------- HIP-graph replay of the paths added later ----------------

@pytest.mark.parametrize("T", [3, 100])
def test_padded_shape_and_split_reduction_replay_from_a_hip_graph(T):
    """moe_forward at a hidden size that needs padding (one more kernel per call,
    the row widening), at 3 tokens (no dispatch pass, the reductions split over the
    waves of a workgroup) and at 100: captured once, replayed three times with eager
    calls of another size in between, every replay bit-identical to the eager
    result."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")

    def ok(rc):
        assert rc == 0, f"HIP call failed with {rc}"

    sh = synth.LayerShape("g", T, 96, 96, 8)
    L = bf16_layer(sh, seed=13)
    m = make_moe(sh, L, 128)
    H = sh.hidden
    dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"]))
    dout, dref = abi.DevBuf(T * H * 4), abi.DevBuf(T * H * 4)
    stream = C.c_void_p()
    ok(hip.hipStreamCreate(C.byref(stream)))
    m.forward(0, dx, None, T, dref, stream=stream)
    ok(hip.hipStreamSynchronize(stream))
    ref = dref.download((T, H), np.float32)
    want = ob.moe_layer(L["x"], None, *[L[k] for k in W], 4, sh.limit, mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
    assert np.abs(ref - want).max() <= 2e-2 and np.linalg.norm(ref - want) <= 1e-3 * np.linalg.norm(want)
    graph, gexec = C.c_void_p(), C.c_void_p()
    ok(hip.hipStreamBeginCapture(stream, C.c_int(0)))
    m.forward(0, dx, None, T, dout, stream=stream)
    ok(hip.hipStreamEndCapture(stream, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)))
    try:
        for _ in range(3):
            dout.memset(0)
            abi.sync()
            ok(hip.hipGraphLaunch(gexec, stream))
            ok(hip.hipStreamSynchronize(stream))
            assert np.array_equal(dout.download((T, H), np.float32), ref)
            m.forward(0, dx, None, max(T // 2, 1), dref, stream=stream)  # eager work of another size
            ok(hip.hipStreamSynchronize(stream))
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)


@pytest.mark.parametrize("E,H", [(100, 96), (100, 768), (128, 2880), (200, 320), (256, 128)])
def test_split_router_gives_the_same_bits(E, H):
    """More than 64 experts: the router of the whole-layer calls runs its first pass as a launch
    of its own up to 200, 400 or 1024 tokens (split_router_tokens; at 96 columns never), moe_router in one
    kernel; ids, weights and so the layer agree bit for bit, on either side of the line, with
    inactive rows and near ties among the tokens."""
    for T in (1, 6, 17, 64, 200, 201, 400, 401, 1023, 1024, 1025):
        sh = synth.LayerShape("r", T, H, 64, E)
        L = bf16_layer(sh, seed=T)
        L["w_router"][E // 2] = L["w_router"][3]  # two experts that always tie but for the bias
        m = make_moe(sh, L, T)
        m.set_distinct_ids(True)
        pos = np.zeros(T, np.int32)
        pos[2::5] = -1
        base = abi.run_layer(m, 0, L["x"], pos)["out"]
        dx, dpos = abi.DevBuf.from_numpy(synth.to_bf16_bits(L["x"])), abi.DevBuf.from_numpy(pos)
        dti, dtv, dout = abi.DevBuf(T * 16), abi.DevBuf(T * 16), abi.DevBuf(T * H * 4)
        dout.memset(0)
        m.router(0, dx, dpos, T, None, dti, dtv)
        m.experts(0, dx, dpos, dti, dtv, T, dout)
        abi.sync()
        assert np.array_equal(dout.download((T, H), np.float32), base)
        ids = dti.download((T, 4), np.int32)
        assert (ids[pos >= 0] >= 0).all() and (ids[pos < 0] == -1).all()
        m.close()


@pytest.mark.parametrize("H", [32, 480, 512, 544, 1024, 1056, 4096, 4128])
def test_norm_at_the_edges_of_its_threads(H):
    """Rows of the norm at the edges of a wave's and a workgroup's pieces and held registers, and
    token counts that leave a last workgroup short: the router behind it finds the oracle's ids (which
    takes the oracle's normalised rows, but for near ties), the block the oracle's result."""
    rng = np.random.default_rng(H)
    for T in (1, 3, 65, 70) + ((1023, 1026) if H in (544, 1024) else ()):
        sh = synth.LayerShape("n", T, H, 64, 8)
        L = bf16_layer(sh, seed=H + T)
        m = make_moe(sh, L, T)
        x = synth.round_bf16((L["x"] * rng.uniform(0.5, 4.0, (T, 1))).astype(np.float32))
        rw = synth.round_bf16((1 + 0.1 * rng.standard_normal(H)).astype(np.float32))
        pos = np.zeros(T, np.int32)
        pos[2::3] = -1
        m.upload_norm(0, rw)
        dx = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
        m.block_forward(0, dx, abi.DevBuf.from_numpy(pos), T)
        doff, dperm = abi.DevBuf(9 * 4), abi.DevBuf(T * 16)
        m.get_dispatch(doff, dperm, T)
        abi.sync()
        _, ti, _ = ob.router(ob.round_to_bf16(ob.rmsnorm(x, rw)), pos, L["w_router"], L["b_router"], 4)
        off, perm, _ = ob.dispatch(ti, pos, 8)
        assert np.array_equal(doff.download((9,), np.int32), off)
        assert np.array_equal(dperm.download((T * 4,), np.int32)[:off[-1]], perm)
        got = synth.from_bf16_bits(dx.download((T, H), np.uint16))
        rows = np.arange(T)[-70:]
        want, _ = ob.ffn_block(np.ascontiguousarray(x[rows]), np.ascontiguousarray(pos[rows]), rw, *[L[k] for k in W], 4,
                               sh.limit, mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
        assert np.all(np.abs(got[rows] - want) <= 2e-2 + 2.0 ** -7 * np.abs(want)), T  # one bf16 step on top of the layer's bar
        assert np.array_equal(got[pos < 0], x[pos < 0])
        m.close()


def test_yardstick_of_the_other_product_runs():
    """v_mfma_f32_16x16x32_bf16 from registers, as test_yardsticks_run."""
    tf, ghz = abi.yardstick_mfma(256, 2000, data=2, small=True)
    tf0, _ = abi.yardstick_mfma(256, 2000, data=0, small=True)
    assert 200 < tf < 2600 and 0.5 < ghz < 3.0 and tf0 > 0.9 * tf


def test_combine_past_the_caches():
    """Either side of the line from which the combine reads the down GEMM's rows past the caches (128 MiB of
    them: 131072 tokens of 64 columns): a token's sums are the same bits, overwritten, added and in the residual
    stream, and the oracle's."""
    H, IM, E, T = 64, 32, 8, 131073
    sh = synth.LayerShape("combine", T, H, IM, E)
    x = synth.round_bf16(synth.make_activations(sh))
    L = {k: (synth.round_bf16(v) if v.dtype == np.float32 else v)
         for k, v in synth.make_layer(synth.LayerShape("combine", 64, H, IM, E), seed=3).items()}
    w = [L[k] for k in ("w_router", "b_router", "w_mlp1", "b_mlp1", "w_mlp2", "b_mlp2")]
    pos = np.zeros(T, np.int32)
    pos[5::97] = -1
    m = abi.Moe(H, IM, E, max_tokens=T, swiglu_limit=sh.limit)
    m.upload_layer(0, *w)
    m.upload_norm(0, np.ones(H, np.float32))
    dx, dpos, dout = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(pos), abi.DevBuf(T * H * 4)
    got = []
    for n in (T - 1, T):
        for accumulate in (False, True):
            dout.memset(0)
            m.forward(0, dx, dpos, n, dout, accumulate=accumulate)
            abi.sync()
            got.append(dout.download((T, H), np.float32)[:T - 1])
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    streams = []
    for n in (T - 1, T):
        ds = abi.DevBuf.from_numpy(synth.to_bf16_bits(x))
        m.block_forward(0, ds, dpos, n)
        abi.sync()
        streams.append(ds.download((T, H), np.uint16)[:T - 1])
    assert np.array_equal(*streams)
    m.close()
    rows = np.arange(0, T - 1, 4001)
    want = ob.moe_layer(np.ascontiguousarray(x[rows]), pos[rows], *w, 4, sh.limit, mode=ob.ROUND_ACT_BF16 | ob.PAR_TOKENS)
    assert np.abs(got[0][rows] - want).max() <= 2e-2 and np.linalg.norm(got[0][rows] - want) <= 1e-3 * np.linalg.norm(want)
