"""The grouped GEMMs at the edges of their row tiles: of 256 and of 128 rows with either
weight format and, with MXFP4, either product; weights read through the caches and
past them (few rows per expert and more than 256 MiB of matrices in the handle);
full, half and quarter column tiles.  Which kernel a case runs is asserted, so that a
line moved elsewhere cannot empty it.

Bars as in test_gpu_parity.py: max-abs 2e-2 and rel-L2 1e-3 of the oracle on the
same inputs; the two weight formats, whose tiles differ, bit for bit."""
import numpy as np
import pytest

from gpt_oss_amd import abi, synth
from oracle import binding as ob

pytestmark = pytest.mark.gpu

E = 32
FEW = (1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 256, 257)  # 1795 rows: 56 per expert
MANY = FEW + (255, 288, 383, 384, 385, 512, 513, 640, 800, 1024)  # 6979 rows: 218 per expert
LOW = (1, 31, 32, 33, 65, 97, 129, 161, 193, 256)  # 998 rows: 31 per expert
BF16, FP4, FP4_MANY = "bf16_gemm_kernel", "grouped_gemm_kernel", "fp4_gemm_kernel"
# kernel, rows of a tile, past the caches: MXFP4 and bf16 weights that the caches hold, then that they do not
ROUTES = {FEW: [(FP4, 128, False), (BF16, 256, False), (FP4, 128, True), (BF16, 256, True)],
          LOW: [(FP4, 256, False), (BF16, 256, False), (FP4, 256, False), (BF16, 256, True)],
          MANY: [(FP4_MANY, 128, False), (BF16, 128, False), (FP4_MANY, 128, False), (BF16, 256, True)]}


@pytest.mark.parametrize("rows", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("H,IM", [(64, 2048), (128, 2112), (192, 2080)])
def test_row_tiles(rows, H, IM):
    check_row_tiles(rows, H, IM)


@pytest.mark.parametrize("H,IM", [(64, 1024), (128, 1088), (192, 992)])
def test_row_tiles_of_few_rounds(H, IM):
    """Few rows per expert and less than two rounds of tiles: bf16 weights past the caches, the rows
    that the GEMMs store through them (bf16_stores_past)."""
    check_row_tiles(LOW, H, IM)


def check_row_tiles(rows, H, IM):
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
    for (fp4, layers), route in zip(((True, 1), (False, 1), (True, many), (False, many * 17 // 64 + 1)), ROUTES[rows]):
        assert abi.batch_kernel(H, IM, E, T, fp4, layers) == route
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


@pytest.mark.parametrize("n_experts,IM,T,fp4_route,bf16_route", [
    (22, 2880, 300, (FP4, 256, False), (BF16, 256, True)), (23, 2880, 300, (FP4, 128, True), (BF16, 256, True)),
    (32, 2048, 511, (FP4, 128, True), (BF16, 256, True)), (32, 2048, 512, (FP4_MANY, 128, True), (BF16, 256, True)),
    (32, 2048, 768, (FP4_MANY, 128, True), (BF16, 256, True)), (32, 2048, 769, (FP4_MANY, 128, False), (BF16, 256, True)),
    (32, 2048, 2048, (FP4_MANY, 128, False), (BF16, 256, True)), (32, 2048, 2049, (FP4_MANY, 128, False), (BF16, 256, False))])
def test_sides_of_the_lines(n_experts, IM, T, fp4_route, bf16_route):
    """Matrices that exceed 256 MiB, on either side of the lines to tiles of 128 rows under
    MXFP4 weights (512 tiles of one row tile per expert), to the other product (64 rows per
    expert), and up to which weights are read past the caches (96 rows per expert with MXFP4,
    256 with bf16): the two weight formats bit for bit, and the oracle."""
    H = 64
    sh = synth.LayerShape("lines", T, H, IM, n_experts)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(sh))
    b1k, s1, b1, b2k, s2, b2 = synth.make_experts_mxfp4(sh)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(b1k, s1), ob.mxfp4_dequant(b2k, s2)
    many = int((256 << 20) / (3 * H * IM * n_experts * 17 / 32)) + 1
    got = []
    for fp4, layers, route in ((True, many, fp4_route), (False, many * 17 // 64 + 1, bf16_route)):
        assert abi.batch_kernel(H, IM, n_experts, T, fp4, layers) == route
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


@pytest.mark.parametrize("H,IM,n_experts,fp4_route,bf16_rows", [
    (H, IM, n, r, b) for H, IM in ((64, 64), (256, 320), (448, 64), (320, 384), (576, 448))
    for n, r, b in ((12, (FP4_MANY, 128), 128), (32, (FP4, 256), 256)) + (((176, (FP4, 128), 256),) if IM > 64 else ())])
def test_reduction_depths(H, IM, n_experts, fp4_route, bf16_rows):
    """Reductions of 1 to 9 double steps of 64, shorter and longer than the rings of the
    loads in front of them, under full, three-quarter, half and quarter column tiles and
    every height of row tile: 12 experts give tiles of 1 to 4 blocks in either format, 32 of 1 to 8,
    176 of 1 to 4 with MXFP4 under the product of few rows per expert.  The weight
    formats bit for bit, and the oracle."""
    rng = np.random.default_rng(H + IM)
    rows = [1, 33, 65, 97, 129, 161, 193, 225, 256, 300, 385, 15]
    if n_experts == 176:
        rows += [17] * 100
    rows = rng.permutation(rows + [0] * (n_experts - len(rows)))
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
    assert abi.batch_kernel(H, IM, n_experts, T, True)[:2] == fp4_route
    assert abi.batch_kernel(H, IM, n_experts, T, False)[:2] == (BF16, bf16_rows)
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
    # a handle with layers of both formats: the dispatch plans tiles of bf16's height for either
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
    some = np.unique(np.concatenate([np.nonzero((ids == e).any(1))[0][[0, -1]] for e in np.nonzero(rows)[0]]))
    want = np.zeros((len(some), H), np.float32)
    for i, t in enumerate(some):
        for k, e in enumerate(ids[t]):
            if e >= 0:
                want[i] += tv[t, k] * ob.expert_token(x[t], w1[e], b1[e], w2[e], b2[e], sh.limit,
                                                      mode=ob.ROUND_ACT_BF16)
    d = got[0][some] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("n_experts,H,IM,T,fp4_route,bf16_rows", [
    (16, 64, 2880, 255, (FP4, 256), 256), (16, 64, 2880, 256, (FP4_MANY, 128), 256),
    (8, 64, 2880, 256, (FP4, 256), 128), (8, 64, 2880, 257, (FP4_MANY, 128), 128),
    (8, 512, 512, 1927, (FP4_MANY, 128), 128), (8, 512, 512, 1928, (FP4_MANY, 128), 256), (8, 512, 512, 3856, (FP4_MANY, 128), 128)])
def test_sides_of_the_product_lines(n_experts, H, IM, T, fp4_route, bf16_rows):
    """Either side of the lines between the products of the MXFP4 kernels (64 rows per
    expert, and 128 where there is at most a workgroup per CU) and between row tiles of 128
    and 256 rows under bf16 weights: the two weight formats bit for bit, stage by
    stage as well, and the oracle."""
    assert abi.batch_kernel(H, IM, n_experts, T, True)[:2] == fp4_route
    assert abi.batch_kernel(H, IM, n_experts, T, False)[:2] == (BF16, bf16_rows)
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


# H, IM of wide plans at 256 experts (tests/test_host_rules.py holds the rule to them): remainders of 2 column blocks
# in both GEMMs, of 6 in gate_up and 4 in down, of none in gate_up and 8 in down
WIDE = [(1024, 512), (1088, 576), (1216, 640)]


@pytest.mark.parametrize("H,IM", WIDE)
def test_wide_tiles(H, IM):
    """Tiles of ten column blocks (up to 6 row blocks high, weights past the caches; the plan's tiles are counted) beside
    tiles of eight, every height, and their last column tiles: the bits of the MXFP4 kernels, whose tiles have
    eight, stage by stage and with an MXFP4 layer under a wide plan as well, and the oracle."""
    n, kinds = 256, 4  # experts of four kinds
    rng = np.random.default_rng(H)
    rows = [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 191, 192, 193, 224, 225, 256, 257, 321, 385]
    rows = rng.permutation(rows + [2] * (n - len(rows)))
    ids = np.repeat(np.arange(n), rows).astype(np.int32)
    T = n * 4 + 4  # stream.hip has batches of up to 16 rows per expert on average
    assert len(ids) <= 4 * T
    ids = rng.permutation(np.concatenate([ids, np.full(4 * T - len(ids), -1, np.int32)])).reshape(T, 4)
    tv = rng.random((T, 4)).astype(np.float32)
    sh = synth.LayerShape("wide", T, H, IM, kinds)
    x = synth.round_bf16(synth.make_activations(sh))
    wr, br = (synth.round_bf16(a) for a in synth.make_router(synth.LayerShape("wide", T, H, IM, n)))
    kind = synth.make_experts_mxfp4(sh)
    b1k, s1, b1, b2k, s2, b2 = (np.tile(a, (n // kinds,) + (1,) * (a.ndim - 1)) for a in kind)
    b1, b2 = synth.round_bf16(b1), synth.round_bf16(b2)
    w1, w2 = ob.mxfp4_dequant(kind[0], kind[1]), ob.mxfp4_dequant(kind[3], kind[4])
    dx, dti = abi.DevBuf.from_numpy(synth.to_bf16_bits(x)), abi.DevBuf.from_numpy(ids)
    dtv, dout = abi.DevBuf.from_numpy(tv), abi.DevBuf(T * H * 4)
    assert abi.batch_kernel(H, IM, n, T, False) == (BF16, 256, True)
    got = []

    def tiles(tallest, narrow_only=False):
        """of both GEMMs; 10 column blocks where they are up to 6 row blocks high, 8 elsewhere"""
        counts = []
        for nb in (2 * IM // 32, H // 32):
            counts.append(0)
            for b in (-(-r // 32) for r in rows):
                n_mt = -(-b // tallest)
                counts[-1] += n_mt * -(-nb // (8 if narrow_only or -(-b // n_mt) > 6 else 10))
        return counts

    wide = tiles(8)
    assert (wide == tiles(8, narrow_only=True)) == (H == 1024)  # there 10 + 10 + 10 + 2 column blocks for four times 8

    def staged(m, layer, planned):
        dout.memset(0xFF)
        m.dispatch(dti, None, T)
        assert list(m.tile_ranges()[:, 8]) == planned
        m.expert_gemms(layer, dx, T)
        m.combine(dtv, None, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))

    m = abi.Moe(H, IM, n, max_tokens=T, swiglu_limit=sh.limit, layers=2)
    m.upload_layer_mxfp4(1, wr, br, b1k, s1, b1, b2k, s2, b2)
    assert abi.batch_kernel(H, IM, n, T, True)[1] == 128
    staged(m, 1, tiles(4, narrow_only=True))  # no bf16 layer: not a wide plan
    m.upload_layer(0, wr, br, np.tile(w1, (n // kinds, 1, 1)), b1, np.tile(w2, (n // kinds, 1, 1)), b2)
    for _ in range(3):
        dout.memset(0xFF)
        m.experts(0, dx, None, dti, dtv, T, dout)
        abi.sync()
        got.append(dout.download((T, H), np.float32))
        assert list(m.tile_ranges()[:, 8]) == wide
    for layer in (0, 1):
        staged(m, layer, wide)
    few = 4 * n  # 16 rows per expert: no tiles
    m.experts(0, dx, None, dti, dtv, few, dout)
    with pytest.raises(abi.MoeError) as e:
        m.tile_ranges()
    assert e.value.code == -5
    m.close()
    for other in got[1:]:
        assert np.array_equal(got[0], other)
    experts = np.nonzero(np.asarray(rows) > 2)[0]
    some = np.unique(np.concatenate([np.nonzero((ids == e).any(1))[0][[0, -1]] for e in experts]))
    want = np.zeros((len(some), H), np.float32)
    for i, t in enumerate(some):
        for k, e in enumerate(ids[t]):
            if e >= 0:
                want[i] += tv[t, k] * ob.expert_token(x[t], w1[e % kinds], b1[e], w2[e % kinds], b2[e], sh.limit,
                                                      mode=ob.ROUND_ACT_BF16)
    d = got[0][some] - want
    assert np.abs(d).max() <= 2e-2 * max(1.0, float(np.abs(want).max()))
    assert np.linalg.norm(d) <= 1e-3 * np.linalg.norm(want)


def _cut(rows, tile_rb, nb, fixed, slow_part):
    """First tiles of the XCDs' ranges, and the estimated time of the slowest, in fp32 as the plan kernel works it out."""
    f = np.float32
    n_rb = (rows + 31) // 32
    n_mt = -(-n_rb // tile_rb)
    mt, rb, tiles = (np.concatenate([[0], np.cumsum(a)]) for a in (n_mt, n_rb, n_mt * -(-nb // 8)))
    cost, slow = fixed * mt + 8 * rb, slow_part * mt + 8 * rb
    bounds, before = [], []
    for x in range(8):
        lo = int(np.nonzero(cost[:-1] * 8 <= cost[-1] * x)[0][-1])
        c, n = cost[lo + 1] - cost[lo], tiles[lo + 1] - tiles[lo]
        k = min(int(f(cost[-1] * x - cost[lo] * 8) / (f(c) * f(8)) * f(n)), n) if c else 0
        bounds.append(int(tiles[lo] + k))
        before.append(f(slow[lo]) + (f(k) * f(slow[lo + 1] - slow[lo]) / f(n) if n else f(0)))
    bounds.append(int(tiles[-1]))
    before.append(f(slow[-1]))
    time = max([f(-(-n // 32)) * (b - a) / f(n) for n, a, b in zip(np.diff(bounds), before, before[1:]) if n > 0], default=f(0))
    cap = (bounds[8] + 7) // 8 + (bounds[8] + 15) // 16 + 1
    for x in range(1, 8):
        bounds[x] = min(max(bounds[x], bounds[x - 1], bounds[8] - (8 - x) * cap), bounds[x - 1] + cap)
    return bounds, time


@pytest.mark.parametrize("H,IM,past", [(2880, 512, True), (2880, 384, False), (1984, 768, True)])
def test_ranges_of_the_xcds(H, IM, past):
    """The cut of either GEMM's tiles into the XCDs' ranges against the rule in numpy: by cost, and with few
    rounds of tiles by the one of two costs whose slowest XCD is expected to be quicker (by 2 % with weights past the
    caches, by 5 % through them); popularities even and uneven, experts without rows, one expert alone."""
    E, top = 32, 3000
    limit, slow_part, gain = (512, 96, np.float32(0.98)) if past else (768, 64, np.float32(0.95))
    m = abi.Moe(H, IM, E, max_tokens=top)
    z = np.zeros
    m.upload_layer(0, z((E, H)), z(E), z((E, 2 * IM, H), np.float32), z((E, 2 * IM)), z((E, H, IM), np.float32), z((E, H)))
    rng = np.random.default_rng(H + IM)
    chosen = [0, 0]
    for T in (129, 150, 200, 256, 300, 350, 400, 450, 480, 512, 600, 700, 1500, 3000):
        kernel, tile_rows, streams = abi.batch_kernel(H, IM, E, T, False)
        assert kernel == BF16 and streams == (past and 4 * T <= 256 * E)
        if streams != past:
            continue
        for exponent in (0.0, 0.6, 1.2, 1.2, 2.0, None):
            if exponent is None:
                ids = np.full((T, 4), 7, np.int32)
                ids[:, 1:] = -1
            else:
                keys = rng.gumbel(size=(T, E)) + 0.65 / 0.78 * np.log(synth.zipf_popularity(E, exponent))
                ids = np.argsort(-keys, axis=1)[:, :4].astype(np.int32)
            rows = np.bincount(ids[ids >= 0], minlength=E)
            m.dispatch(abi.DevBuf.from_numpy(ids), None, T)
            got = m.tile_ranges()
            for g, nb in enumerate((2 * IM // 32, H // 32)):
                (by_64, slow_64), (by_32, slow_32) = (_cut(rows, tile_rows // 32, nb, fixed, slow_part) for fixed in (64, 32))
                few = by_64[8] <= limit and slow_32 < gain * slow_64
                if abs(slow_32 - gain * slow_64) > 1e-5 * slow_64:
                    assert list(got[g]) == (by_32 if few else by_64), (T, exponent, g)
                    chosen[int(few)] += 1
    m.close()
    assert chosen[0] and chosen[1]
