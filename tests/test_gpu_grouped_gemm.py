"""The grouped GEMMs of the batched path at the sizes where they change their code: buckets of every token count at the edge
of a 16-, 32- and 64-token tile (the selection is given, so the counts are), single-block and ragged contractions, and
blocks whose scale is zero (the K-quant kernel keeps its sums in units of the current block's scale)."""
import numpy as np
import pytest

import helpers as H
import moe4all_amd as M
import oracle as O
from moe4all_amd import DType

from test_gpu_parity import REL_L2_MFMA, _bank_weights, _run_batched, bits, moe_graph, run_moe
from test_zz_no_alloc import _free_device_bytes

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130]


@pytest.fixture(scope="module")
def be():
    b = M.Backend(0)
    yield b
    b.close()


def _zero_some_scales(w, dtype, rng):
    """d = 0 in a tenth of the super-blocks (and in the first ones of some rows): byte offset of d, block bytes."""
    at = {H.Q4K: (0, 144), H.Q6K: (208, 210), H.Q5K: (0, 176), H.IQ4_XS: (0, 136)}.get(dtype)
    if at is None:
        return w
    blk = np.ascontiguousarray(w).reshape(-1, at[1])
    pick = rng.random(len(blk)) < 0.1
    pick[:2] = True
    blk[pick, at[0]:at[0] + 2] = 0
    return blk.reshape(-1)


@pytest.mark.parametrize("gdt,ddt,ne,nff", [
    (H.Q4K, H.Q6K, 512, 256), (H.Q6K, H.Q4K, 256, 768), (H.Q8_0, H.Q8_0, 256, 512), (H.Q4K, H.Q4K, 768, 512),
    (H.Q5K, H.Q6K, 512, 256), (H.IQ4_XS, H.Q5K, 256, 512),
    # rows that end inside a 256-k step (64 and 192 k behind the last whole one)
    (H.Q4_0, H.MXFP4, 320, 448), (H.MXFP4, H.Q4_0, 192, 320), (H.Q8_0, H.Q5_0, 448, 64), (H.Q5_1, H.NVFP4, 320, 192),
])
def test_buckets_at_the_edges_of_the_token_tiles(be, gdt, ddt, ne, nff):
    rng = np.random.default_rng(gdt * 31 + ddt)
    E, rows = len(COUNTS), sum(COUNTS)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    sel = rng.permutation(np.repeat(np.arange(E), COUNTS)).astype(np.int32).reshape(rows, 1)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    data = dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel)
    out, r, b = _run_batched(be, g, ids, data, rows, ne)
    assert np.array_equal(r["idx"], sel)
    assert np.array_equal(np.diff(b["offsets"]), COUNTS)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=1, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt,
                    expert_ids=sel)
    for e in range(E):
        m = sel[:, 0] == e
        if m.any():
            assert H.rel_l2(out[m], ref["dst"][m]) < REL_L2_MFMA / 4, (e, COUNTS[e])
    # a row's bits do not depend on the tile it lands in: another order of the rows
    p = rng.permutation(rows)
    out2, _, _ = _run_batched(be, g, ids, dict(data, x=np.ascontiguousarray(x[p]), expert_ids=np.ascontiguousarray(sel[p])), rows, ne)
    assert np.array_equal(bits(out2), bits(out[p]))


WIDE_COUNTS = [0, 7, 8, 9, 16, 17, 33, 64, 65, 96, 97, 127, 128, 129, 257]


@pytest.mark.parametrize("gdt,ddt,ne,nff", [
    # wide rows take tiles of 128 tokens (small launches of others tiles of 64: the same buckets, the other kernel)
    (H.Q4K, H.Q6K, 4352, 256), (H.Q6K, H.Q4K, 256, 4352), (H.Q5K, H.IQ4_XS, 256, 4352), (H.IQ4_XS, H.Q5K, 4352, 512),
    (H.Q8_0, H.Q8_0, 448, 192), (H.Q8_0, H.Q8_0, 1024, 384), (H.Q8_0, H.Q8_0, 4352, 192), (H.Q8_0, H.Q8_0, 448, 4352),
    # rows that end inside a step
    (H.Q4_0, H.Q4_0, 4416, 192), (H.MXFP4, H.Q4_0, 192, 4160), (H.Q4_0, H.MXFP4, 320, 4288),
])
def test_tiles_of_up_to_128_tokens(be, gdt, ddt, ne, nff):
    """Buckets at the edges of the 8-, 16-, 32-, 64-, 96- and 128-token tiles; the bar is that of the 64-token tiles (f16 operands on
    both sides), and a row's bits are those it has in a tile of another size."""
    rng = np.random.default_rng(gdt * 59 + ddt + ne)
    E, rows = len(WIDE_COUNTS), sum(WIDE_COUNTS)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = np.zeros((E, ne), np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    sel = rng.permutation(np.repeat(np.arange(E), WIDE_COUNTS)).astype(np.int32).reshape(rows, 1)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    data = dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel)
    out, _, b = _run_batched(be, g, ids, data, rows, ne)
    assert np.array_equal(np.diff(b["offsets"]), WIDE_COUNTS)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=1, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt,
                    expert_ids=sel)
    for e in range(E):
        m = sel[:, 0] == e
        if m.any():
            assert H.rel_l2(out[m], ref["dst"][m]) < REL_L2_MFMA / 4, (e, WIDE_COUNTS[e])
    # 40 of the rows alone, in tiles of few tokens
    p = rng.choice(rows, 40, replace=False)
    g, ids = moe_graph(40, ne, E, 1, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    out2, _, _ = _run_batched(be, g, ids, dict(data, x=np.ascontiguousarray(x[p]), expert_ids=np.ascontiguousarray(sel[p])), 40, ne)
    assert np.array_equal(bits(out2), bits(out[p]))


@pytest.mark.parametrize("gdt,ddt,ne,nff,rows,K,residual,up_first,down_scale", [
    (H.Q4K, H.Q6K, 512, 256, 130, 2, True, False, False), (H.Q4K, H.Q6K, 512, 256, 300, 8, False, True, True),
    (H.Q8_0, H.Q8_0, 320, 192, 128, 3, True, True, False), (H.Q5K, H.Q4K, 256, 4352, 333, 1, True, False, True),
    (H.MXFP4, H.IQ4_XS, 192, 256, 257, 4, False, False, False),
])
def test_always_on_expert_in_the_batchs_gemms(be, gdt, ddt, ne, nff, rows, K, residual, up_first, down_scale):
    """An always-on expert beside a batch's MoeFfn joins its GEMMs: no launch of its own is left, the result is the oracle's, and that
    of the separate ops up to the activation (both keep it in f32 until its f16 rounding, with an exponential of 1 ulp here;
    an element in some thousand rounds to the other neighbour, 2^-11 of it)."""
    rng = np.random.default_rng(gdt * 61 + ddt + rows)
    E = 9
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.05).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    sg, su, sd = _bank_weights(rng, 1, nff, ne, gdt, ddt)
    ds = (0.5 + rng.random(E)).astype(np.float32) if down_scale else None

    def graph():
        g = M.Graph()
        t = lambda kind, shape, dt=DType.F32: getattr(g, kind)(M.TensorDesc(list(shape), dt))  # noqa: E731
        ids = {k: t("weight", sh, dt) for k, sh, dt in (
            ("router", (E, ne), DType.F32), ("gate", (E, nff, ne), DType(gdt)), ("up", (E, nff, ne), DType(gdt)),
            ("down", (E, ne, nff), DType(ddt)), ("sg", (nff, ne), DType(gdt)), ("su", (nff, ne), DType(gdt)), ("sd", (ne, nff), DType(ddt)))}
        if down_scale:
            ids["ds"] = t("weight", (E,))
        ids["x"], ids["y"] = t("input", (rows, ne)), t("output", (rows, ne))
        moe, tg, tu, ta, ts = (t("internal", (rows, n)) for n in (ne, nff, nff, nff, ne))
        total = t("internal", (rows, ne)) if residual else ids["y"]
        g.moe_ffn(x=ids["x"], router=ids["router"], gate_exps=ids["gate"], up_exps=ids["up"], down_exps=ids["down"], dst=moe, ne=ne,
                  n_expert=E, n_used=K, n_ff_exp=nff, down_scale=ids.get("ds"))
        for w, dst in [("su", tu), ("sg", tg)] if up_first else [("sg", tg), ("su", tu)]:
            g.linear(x=ids["x"], weight=ids[w], dst=dst, m=rows, in_f=ne, out_f=nff)
        g.gated_act(gate=tg, up=tu, dst=ta, rows=rows, nff=nff)
        g.linear(x=ta, weight=ids["sd"], dst=ts, m=rows, in_f=nff, out_f=ne)
        g.add(a=ts if residual else moe, b=moe if residual else ts, dst=total, n=rows * ne)
        if residual:
            g.add(a=ids["x"], b=total, dst=ids["y"], n=rows * ne)
        return g, ids

    data = dict(x=x, router=router, gate=gate, up=up, down=down, sg=sg, su=su, sd=sd)
    if down_scale:
        data["ds"] = ds
    outs, names = {}, {}
    for off in (False, True):
        b = be if not off else M.Backend(0, disable_op_fusion=True)
        try:
            g, ids = graph()
            b.prof_enable(True)
            keep = []
            outs[off] = M.run_graph(b, g, [(ids[k], v) for k, v in data.items()], ids["y"], rows * ne, keep=keep).reshape(rows, ne)
            names[off] = set(b.prof_read())
            b.prof_enable(False)
        finally:
            if off:
                b.close()
    assert not any(n.startswith(("linear", "gated_act", "add")) for n in names[False]), names[False]
    assert {"linear_grouped", "gated_act", "add"} <= names[True]
    moe = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt, down_scale=ds)["dst"]
    always = O.linear(O.gated_act_rows(O.linear(x, sg, gdt, ne, nff), O.linear(x, su, gdt, ne, nff)), sd, ddt, nff, ne)
    want = np.asarray(moe).reshape(rows, ne) + np.asarray(always).reshape(rows, ne)
    base = x if residual else 0.0
    assert H.rel_l2(outs[False] - base, want) < REL_L2_MFMA / 4
    # 2^-11 for one element in 256 of a row's sum: 2^-11 / 16 = 3e-5
    assert H.rel_l2(outs[False], outs[True]) < 3e-5


@pytest.mark.parametrize("gdt,ddt,ne,nff,rows,used", [
    (H.Q4K, H.Q6K, 256, 256, 64, 24), (H.Q4K, H.Q6K, 512, 256, 200, 17), (H.Q5K, H.Q4K, 256, 512, 448, 5), (H.Q8_0, H.Q8_0, 320, 192, 448, 24),
    (H.MXFP4, H.Q4_0, 192, 64, 150, 9), (H.IQ4_XS, H.IQ4_XS, 256, 256, 65, 1),
])
def test_tiles_dealt_to_the_xcds_in_small_launches(be, gdt, ddt, ne, nff, rows, used):
    """From 32 tiles by the launch's bound on, and up to 384 items, the columns of a tile go to one XCD: 40 experts of which some are
    selected, so that the tiles that there are end anywhere inside an eight, against 24 experts, whose tiles' columns lie side by side."""
    rng = np.random.default_rng(gdt * 71 + rows)
    E, few, K = 40, 24, 1
    assert rows * K // 64 + few < 32 <= rows * K // 128 + E
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    sel = rng.permutation(few)[:used][rng.integers(0, used, (rows, K))].astype(np.int32)
    outs = []
    for n in (E, few):
        cut = lambda w: w.reshape(E, -1)[:n].reshape(-1)  # noqa: E731
        g, ids = moe_graph(rows, ne, n, K, nff, DType(gdt), DType(ddt), with_expert_ids=True)
        outs.append(_run_batched(be, g, ids, dict(x=x, router=np.zeros((n, ne), np.float32), gate=cut(gate), up=cut(up), down=cut(down), expert_ids=sel), rows, ne)[0])
    assert np.array_equal(bits(outs[0]), bits(outs[1]))
    ref = O.moe_ffn(x, np.zeros((E, ne), np.float32), gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt, expert_ids=sel)
    assert H.rel_l2(outs[0], ref["dst"].reshape(rows, ne)) < REL_L2_MFMA / 4


INT_COUNTS = [0, 1, 3, 4, 5, 8, 9]   # tiles of up to 4 and up to 8 tokens


@pytest.mark.parametrize("gdt,ddt,ne,nff", [
    (H.Q4K, H.Q6K, 512, 768), (H.Q6K, H.Q5K, 256, 1280), (H.Q8_0, H.Q4_0, 160, 352), (H.MXFP4, H.Q8_0, 96, 224), (H.Q5K, H.IQ4_XS, 768, 256),
    (H.IQ4_XS, H.MXFP4, 256, 288),
    # down rows in parts of K: whole blocks, and a last part that ends inside a 256-k step
    (H.Q8_0, H.Q6K, 64, 8192), (H.MXFP4, H.Q8_0, 64, 8288), (H.Q4_0, H.Q4_0, 64, 8352),
])
def test_decode_batches_over_expert_buckets(be, gdt, ddt, ne, nff):
    """Below the batched threshold a batch with few distinct experts runs the integer kernels over the buckets, f32-accurate."""
    rng = np.random.default_rng(gdt * 37 + ddt + nff)
    E, rows = len(INT_COUNTS), sum(INT_COUNTS)
    x = (rng.standard_normal((rows, ne)) * np.exp(rng.standard_normal((rows, 1)))).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    sel = rng.permutation(np.repeat(np.arange(E), INT_COUNTS)).astype(np.int32).reshape(rows, 1)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    be.prof_enable(True)
    out, r, b = _run_batched(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel), rows, ne)
    names = set(be.prof_read())
    be.prof_enable(False)
    assert {"moe_gate_up_bucketed", "moe_down_bucketed"} <= names
    assert np.array_equal(np.diff(b["offsets"]), INT_COUNTS)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=1, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt,
                    expert_ids=sel)
    for row in range(rows):
        assert H.rel_l2(out[row], ref["dst"][row]) < 1e-5, (row, sel[row])


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("gdt,ddt,ne,nff", [
    (H.Q4_0, H.MXFP4, 192, 2880), (H.MXFP4, H.Q4_0, 2880, 64), (H.Q5K, H.IQ4_XS, 4096, 256), (H.IQ4_XS, H.Q5K, 256, 4096),
    (H.MXFP4, H.MXFP4, 4096, 1088), (H.Q4_0, H.Q4_0, 64, 4096),
])
def test_decode_rows_of_one_to_sixty_four_lanes(be, gdt, ddt, ne, nff, rows):
    rng = np.random.default_rng(gdt * 41 + ddt + ne)
    E, K = 4, 2
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w, dt in zip(_bank_weights(rng, E, nff, ne, gdt, ddt), (gdt, gdt, ddt)))
    g, ids = moe_graph(rows, ne, E, K, nff, DType(gdt), DType(ddt))
    out, r = run_moe(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down), rows, ne)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt)
    assert np.array_equal(r["idx"], ref["idx"])
    for row in range(rows):
        assert H.rel_l2(out.reshape(rows, ne)[row], ref["dst"].reshape(rows, ne)[row]) < 1e-5, row


@pytest.mark.parametrize("dt,ne,nff", [
    (H.Q8_0, 2048, 352), (H.Q8_0, 160, 1056), (H.Q5K, 1280, 768), (H.Q4_0, 1088, 320), (H.Q4_0, 64, 4032), (H.IQ4_XS, 1280, 768),
    (H.Q4K, 2304, 1280), (H.Q6K, 768, 4096),
])
def test_rows_keep_their_bits_in_a_batch_over_buckets(be, dt, ne, nff):
    """A token row alone and among three (per-token kernels) and among 20 on seven experts (buckets): the same group sums, scaled
    and added up in the same order, for every format and row width that both families take; MXFP4 is left out, whose per-token
    kernel multiplies floats."""
    rng = np.random.default_rng(dt * 43 + ne)
    E, rows = 7, 20
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = (_zero_some_scales(w, dt, rng) for w in _bank_weights(rng, E, nff, ne, dt, dt))
    sel = rng.integers(0, E, (rows, 1)).astype(np.int32)

    def run(pick):
        g, ids = moe_graph(len(pick), ne, E, 1, nff, DType(dt), DType(dt), with_expert_ids=True)
        be.prof_enable(True)
        out, _ = run_moe(be, g, ids, dict(x=np.ascontiguousarray(x[pick]), router=router, gate=gate, up=up, down=down,
                                          expert_ids=np.ascontiguousarray(sel[pick])), len(pick), ne)
        names = set(be.prof_read())
        be.prof_enable(False)
        assert ("moe_down_bucketed" in names) == (len(pick) == rows), names
        return out

    full = run(list(range(rows)))
    assert np.array_equal(bits(run([0, 9, 19])), bits(full[[0, 9, 19]]))
    for r in (0, 9, 19):
        assert np.array_equal(bits(run([r])[0]), bits(full[r])), r


def test_down_rows_in_parts_keep_their_bits_in_any_batch(be):
    """Down rows of more than sixteen 256-k steps go in parts of K, as many at 16 rows (some 12 of 24 experts) as at 31."""
    ne, nff, E, rows, dt = 2048, 4352, 24, 31, H.Q4_0
    rng = np.random.default_rng(5)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = (np.tile(w, E) for w in _bank_weights(rng, 1, nff, ne, dt, dt))
    sel = rng.integers(0, E, (rows, 1)).astype(np.int32)
    outs = []
    for n in (16, rows):
        g, ids = moe_graph(n, ne, E, 1, nff, DType(dt), DType(dt), with_expert_ids=True)
        be.prof_enable(True)
        out, _ = run_moe(be, g, ids, dict(x=np.ascontiguousarray(x[:n]), router=router, gate=gate, up=up, down=down,
                                          expert_ids=np.ascontiguousarray(sel[:n])), n, ne)
        assert "moe_down_bucketed" in set(be.prof_read())
        be.prof_enable(False)
        outs.append(out)
    assert np.array_equal(bits(outs[0]), bits(outs[1][:16]))


def _small_first_weight(w, dtype, gain_rows=None):
    """Element 0 of every group of 32 decodes to zero (IQ4_XS: to its smallest magnitude, the book has no zero), so that an
    outlier there adds nothing to hide behind; the rows of `gain_rows` get sixteen times the scale."""
    b = np.ascontiguousarray(w).reshape(-1, H.BLOCK[dtype][1]).copy()
    d_at = 208 if dtype == H.Q6K else 0
    if dtype in (H.Q4K, H.Q5K):
        b[:, 8:12] = 0                    # minimums of groups 0..3, and the upper bits of 4..7's
        b[:, 12:16] &= 0x0F
        first = 16 if dtype == H.Q4K else 48
        for g in range(8):
            b[:, first + 32 * (g >> 1)] &= 0xF0 if g % 2 == 0 else 0x0F
        if dtype == H.Q5K:
            b[:, 16] = 0
        b[:, 2:4] = 0
    elif dtype == H.Q6K:                  # code 32
        for h in range(2):
            b[:, [64 * h, 64 * h + 32]] = 0
            b[:, 128 + 32 * h] = 0xAA
    elif dtype == H.Q8_0:
        b[:, 2] = 0
    elif dtype == H.MXFP4:
        b[:, 1] &= 0xF0
    elif dtype == H.Q4_0:
        b[:, 2] = (b[:, 2] & 0xF0) | 8
    else:
        assert dtype == H.IQ4_XS
        for g in range(8):
            b[:, 8 + 16 * g] = (b[:, 8 + 16 * g] & 0xF0) | 8
    if gain_rows is not None:
        rows = b.reshape(len(gain_rows), -1, b.shape[1])[gain_rows]
        if dtype == H.MXFP4:
            rows[:, :, 0] += 4
        else:
            rows[:, :, d_at:d_at + 2] = (rows[:, :, d_at:d_at + 2].copy().view(np.float16) * np.float16(16)).view(np.uint8)
        b.reshape(len(gain_rows), -1, b.shape[1])[gain_rows] = rows
    return b.reshape(-1)


@pytest.mark.parametrize("dt,ne,nff,rows,where", [
    (H.Q5K, 1280, 768, 1, "xh"), (H.Q5K, 1280, 768, 20, "xh"), (H.Q4_0, 1088, 320, 1, "xh"), (H.Q4_0, 1088, 320, 20, "xh"),
    (H.IQ4_XS, 1280, 768, 1, "xh"), (H.IQ4_XS, 1280, 768, 20, "xh"), (H.MXFP4, 1088, 320, 1, "xh"), (H.MXFP4, 1088, 352, 20, "xh"),
    # rows too wide for a wavefront of the per-token kernels (h: as down banks behind Q4_0 ones)
    (H.Q8_0, 2080, 320, 20, "x"), (H.Q8_0, 320, 2304, 20, "h"), (H.Q4K, 4352, 256, 20, "x"), (H.Q4K, 256, 4352, 20, "h"),
    (H.Q6K, 4352, 256, 20, "x"), (H.Q6K, 256, 4352, 20, "h"),
])
def test_small_activations_beside_outliers_keep_their_bits(be, dt, ne, nff, rows, where):
    """One element of 32 is some 256 times the others, in x and / or (through sixteen-fold gate and up rows) in the activated row, and
    meets a weight of zero.  An f32 sum then loses nothing; fixed point of 24 bits relative to the group's largest is off by up
    to 256 * 2^-24 = 1.5e-5 of the other elements (and of the result: 1.2e-5 to 3.3e-5).  The bar is what f32 arithmetic
    allows: 2^-24 for each of the some eight roundings of a sum's tree, twice (gate/up, down): 1e-6."""
    rng = np.random.default_rng(dt * 47 + ne + rows)
    E, gdt = 1 if rows == 1 else 3, H.Q4_0 if where == "h" else dt
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    if "x" in where:
        x[:, ::32] *= 256
    router = np.zeros((E, ne), np.float32)
    gain = (np.arange(E * nff) % 32 == 0) & ("h" in where)
    raw = _bank_weights(rng, E, nff, ne, gdt, dt)
    gate, up, down = _small_first_weight(raw[0], gdt, gain), _small_first_weight(raw[1], gdt, gain), _small_first_weight(raw[2], dt)
    sel = rng.integers(0, E, (rows, 1)).astype(np.int32)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(gdt), DType(dt), with_expert_ids=True)
    be.prof_enable(True)
    out, _ = run_moe(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel), rows, ne)
    names = set(be.prof_read())
    be.prof_enable(False)
    assert ("moe_down_bucketed" in names) == (rows > 1), names
    wg, wu, wd = (np.asarray(H.ggml_dequant(d, w), np.float64).reshape(s)
                  for d, w, s in ((gdt, gate, (E, nff, ne)), (gdt, up, (E, nff, ne)), (dt, down, (E, ne, nff))))
    for r in range(rows):
        e = sel[r, 0]
        a, u = wg[e] @ x[r].astype(np.float64), wu[e] @ x[r].astype(np.float64)
        want = wd[e] @ (a / (1 + np.exp(-a)) * u)
        assert np.linalg.norm(out[r] - want) < 1e-6 * np.linalg.norm(want), r


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("dt,nff", [(H.MXFP4, 4096), (H.Q4_0, 4096), (H.Q5K, 4096), (H.Q5K, 2560), (H.IQ4_XS, 2816), (H.Q4K, 4096)])
def test_down_rows_of_eight_ranks_fill_the_lds(be, dt, nff, rows):
    """The per-token down kernel holds the activated row of every rank: eight of 4096 are 144 KiB (112 with three planes)."""
    ne, E, K = 256, 9, 8
    rng = np.random.default_rng(dt * 53 + nff)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.02).astype(np.float32)
    gate, up, down = _bank_weights(rng, E, nff, ne, dt, dt)
    g, ids = moe_graph(rows, ne, E, K, nff, DType(dt), DType(dt))
    be.prof_enable(True)
    out, r = run_moe(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down), rows, ne)
    names = set(be.prof_read())
    be.prof_enable(False)
    assert not any("bucket" in n for n in names), names
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=dt, down_dtype=dt)
    assert np.array_equal(r["idx"], ref["idx"])
    for row in range(rows):
        assert H.rel_l2(out[row], ref["dst"][row]) < 1e-5, row


@pytest.mark.parametrize("gdt,ddt,ne,nff,E,rows,beside,bucketed", [
    (H.Q4K, H.Q6K, 4096, 1536, 64, 8, None, False), (H.Q4K, H.Q6K, 4096, 3072, 64, 8, None, True),
    # a Linear of one output on the same rows is no always-on expert; neither is one that the per-token kernels cannot take along
    (H.Q8_0, H.Q8_0, 2048, 768, 128, 14, None, True), (H.Q8_0, H.Q8_0, 2048, 768, 128, 14, 1, True),
    (H.Q8_0, H.Q8_0, 2048, 768, 128, 14, 768, False), (H.Q8_0, H.Q8_0, 4096, 1536, 64, 2, 1536, True),
])
def test_which_decode_batches_go_over_buckets(be, gdt, ddt, ne, nff, E, rows, beside, bucketed):
    """The plan's choice alone (nothing is allocated for the weights): by the time of the bytes on either side, and 20 or, where
    an always-on expert leaves the per-token kernels for launches of its own, 60 us."""
    g, ids = moe_graph(rows, ne, E, 8, nff, DType(gdt), DType(ddt))
    if beside:
        w = g.weight(M.TensorDesc([beside, ne], DType(gdt)))
        y = g.output(M.TensorDesc([rows, beside], DType.F32))
        g.linear(x=ids["x"], weight=w, dst=y, m=rows, in_f=ne, out_f=beside)
    plan = be.compile(g)
    try:
        if bucketed:
            assert len(be.moe_bucketing(plan, 0)["offsets"]) == E + 1
        else:
            with pytest.raises(M.BackendError):
                be.moe_bucketing(plan, 0)
    finally:
        plan.free()


@pytest.mark.parametrize("gdt,ddt,ne,nff,rows,K", [
    # from 1024 h rows on a wavefront each, with one to four chunks per lane (64 to 2048 elements, the last chunk full or not), with and
    # without group sums behind them (Q4_K, Q5_K down); row counts that are no multiple of a block's four
    (H.Q8_0, H.Q8_0, 64, 64, 343, 3), (H.Q8_0, H.Q4K, 256, 512, 256, 4), (H.Q8_0, H.Q5K, 256, 768, 343, 3), (H.Q8_0, H.Q4K, 256, 1024, 343, 3),
    (H.Q8_0, H.Q5K, 256, 1280, 205, 5), (H.Q8_0, H.Q4K, 256, 1536, 343, 3), (H.Q8_0, H.Q4_0, 64, 1600, 343, 3), (H.Q8_0, H.Q6K, 256, 1792, 342, 3),
    (H.Q8_0, H.Q4K, 256, 2048, 343, 3),
    # a block each: fewer rows, longer ones
    (H.Q8_0, H.Q5K, 256, 768, 341, 3), (H.Q8_0, H.Q4K, 256, 2304, 343, 3),
])
def test_activated_rows_to_f16(be, gdt, ddt, ne, nff, rows, K):
    """Rows of h of any length, among them some of zeros and some a thousand times larger: each has a scale of its own, and the bits
    that it has in a small batch, whose rows take a block each."""
    rng = np.random.default_rng(ddt * 67 + nff)
    E = 7
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    x[::5] = 0.0
    x[1::5] *= 1000.0
    router = np.zeros((E, ne), np.float32)
    gate, up, down = _bank_weights(rng, E, nff, ne, gdt, ddt)
    sel = np.argsort(rng.random((rows, E)), axis=1)[:, :K].astype(np.int32)
    g, ids = moe_graph(rows, ne, E, K, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    data = dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel)
    out, _, _ = _run_batched(be, g, ids, data, rows, ne)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=gdt, down_dtype=ddt,
                    expert_ids=sel)["dst"].reshape(rows, ne)
    for r in range(rows):
        if r % 5 == 0:
            assert not out[r].any()
        else:
            assert H.rel_l2(out[r], ref[r]) < REL_L2_MFMA, r
    p = rng.choice(rows, 40, replace=False)
    g, ids = moe_graph(40, ne, E, K, nff, DType(gdt), DType(ddt), with_expert_ids=True)
    few, _, _ = _run_batched(be, g, ids, dict(data, x=np.ascontiguousarray(x[p]), expert_ids=np.ascontiguousarray(sel[p])), 40, ne)
    assert np.array_equal(bits(few), bits(out[p]))


@pytest.mark.parametrize("rows,K", [(300, 8), (256, 8), (257, 8), (2100, 8), (5000, 4)])
def test_bucketing_of_many_pairs(be, rows, K):
    """Up to 2048 pairs on four wavefronts, more on sixteen, more than 16384 in chunks: the reference's order exactly."""
    ne, nff, E = 64, 64, 61
    rng = np.random.default_rng(rows + K)
    sel = np.argsort(rng.random((rows, E)) + 0.6 * np.arange(E) / E, axis=1)[:, :K].astype(np.int32)   # uneven buckets
    gate, up, down = _bank_weights(rng, E, nff, ne, H.Q8_0, H.Q8_0)
    g, ids = moe_graph(rows, ne, E, K, nff, DType.Q8_0, DType.Q8_0, with_expert_ids=True)
    _, _, b = _run_batched(be, g, ids, dict(x=rng.standard_normal((rows, ne)).astype(np.float32), router=np.zeros((E, ne), np.float32),
                                            gate=gate, up=up, down=down, expert_ids=sel), rows, ne)
    flat = sel.reshape(-1)
    order = np.argsort(flat, kind="stable")
    assert np.array_equal(np.diff(b["offsets"]), np.bincount(flat, minlength=E))
    assert np.array_equal(b["pair_row"], order // K) and np.array_equal(b["pair_rank"], order % K)
    slot = np.empty_like(order)
    slot[order] = np.arange(len(order))
    assert np.array_equal(b["slot_pair"].reshape(-1), slot)


@pytest.mark.parametrize("rows,K,E", [
    (33, 1, 3), (64, 8, 150),                        # fewer pairs than threads; fewer than three pairs per expert
    (2048, 1, 7), (683, 3, 61),                      # 2048 pairs on four wavefronts, 2049 on sixteen
    (2048, 8, 61), (3277, 5, 61),                    # 16384 held in registers, 16385 in chunks
])
def test_bucketing_at_the_edges_of_its_kernels(be, rows, K, E):
    """The reference's order exactly, and token rows that have the bits of small batches (33 rows at a time)."""
    ne, nff = 64, 64
    rng = np.random.default_rng(rows + K + E)
    sel = np.argsort(rng.random((rows, E)) + 0.6 * np.arange(E) / E, axis=1)[:, :K].astype(np.int32)   # uneven buckets
    gate, up, down = _bank_weights(rng, E, nff, ne, H.Q8_0, H.Q8_0)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    data = dict(router=np.zeros((E, ne), np.float32), gate=gate, up=up, down=down)
    g, ids = moe_graph(rows, ne, E, K, nff, DType.Q8_0, DType.Q8_0, with_expert_ids=True)
    out, _, b = _run_batched(be, g, ids, dict(data, x=x, expert_ids=sel), rows, ne)
    flat = sel.reshape(-1)
    order = np.argsort(flat, kind="stable")
    assert np.array_equal(np.diff(b["offsets"]), np.bincount(flat, minlength=E))
    assert np.array_equal(b["pair_row"], order // K) and np.array_equal(b["pair_rank"], order % K)
    slot = np.empty_like(order)
    slot[order] = np.arange(len(order))
    assert np.array_equal(b["slot_pair"].reshape(-1), slot)
    for first in (0, rows - 33):   # the last rows among them: they may share a workgroup of the conversion with none
        part = slice(first, first + 33)
        g, ids = moe_graph(33, ne, E, K, nff, DType.Q8_0, DType.Q8_0, with_expert_ids=True)
        few, _, _ = _run_batched(be, g, ids, dict(data, x=np.ascontiguousarray(x[part]), expert_ids=np.ascontiguousarray(sel[part])), 33, ne)
        assert np.array_equal(bits(few), bits(out[part]))


@pytest.mark.parametrize("rows,E,K", [(40, 32, 8), (40, 64, 4), (33, 128, 8), (40, 129, 15), (33, 256, 16), (40, 257, 15), (70, 512, 15), (90, 600, 12)])
def test_routing_of_a_batch_by_itself(be, rows, E, K):
    """The routing launch of a batch, for every number of experts it has code for: ids and weights of the reference, also in rows whose
    logits are equal in pairs, all equal, or far apart, which the selection on two wavefronts leaves to the complete routine."""
    ne, nff = 64, 64
    rng = np.random.default_rng(rows + E + K)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    x[::5] = 0.0
    x[1::5] *= 300.0
    router = (rng.standard_normal((E, ne)) * 0.3).astype(np.float32)
    router[E // 2:E // 2 + E // 4] = router[:E // 4]
    gate, up, down = _bank_weights(rng, E, nff, ne, H.Q8_0, H.Q8_0)
    g, ids = moe_graph(rows, ne, E, K, nff, DType.Q8_0, DType.Q8_0)
    _, r, _ = _run_batched(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down), rows, ne)
    for i in range(rows):
        probs, idx, w = O.route_row(r["logits"][i], K)
        assert np.array_equal(r["idx"][i], idx) and np.array_equal(bits(r["w"][i]), bits(w)) and np.array_equal(bits(r["probs"][i]), bits(probs)), i


@pytest.mark.parametrize("rows,E,K,units", [(16, 8, 2, False), (16, 64, 2, True), (16, 65, 2, True), (16, 9, 3, False), (17, 8, 1, False),
                                            (16, 1, 1, False), (1, 5, 2, True), (3, 64, 10, True), (3, 64, 11, True), (1, 64, 32, True)])
def test_routing_and_bucketing_of_a_few_rows(be, rows, E, K, units):
    """Up to 16 rows, 32 pairs and 64 experts in one launch, more in two: routing and bucket order exactly, with a selection of the
    router's and with a given one that names experts twice in a row.  (units: the kernels over buckets
    that take a width of no whole 64, here from any row count.)"""
    ne, nff = 256, 96 if units else 64
    rng = np.random.default_rng(100 * rows + E)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = (rng.standard_normal((E, ne)) * 0.2).astype(np.float32)
    gate, up, down = _bank_weights(rng, E, nff, ne, H.Q8_0, H.Q8_0)
    b2 = M.Backend(0, moe_batched_min_rows=1) if units else be
    for given in (False, True):
        sel = rng.integers(0, max(1, E // 2), (rows, K)).astype(np.int32)
        g, ids = moe_graph(rows, ne, E, K, nff, DType.Q8_0, DType.Q8_0, with_expert_ids=given)
        out, r, b = _run_batched(b2, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down, **(dict(expert_ids=sel) if given else {})), rows, ne)
        ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff, gate_dtype=H.Q8_0, down_dtype=H.Q8_0,
                        **(dict(expert_ids=sel) if given else {}))
        idx = np.asarray(r["idx"]).reshape(rows, K)
        assert np.array_equal(idx, sel if given else ref["idx"]) and np.array_equal(bits(r["w"]), bits(ref["w"]))
        order = np.argsort(idx.reshape(-1), kind="stable")
        assert np.array_equal(np.diff(b["offsets"]), np.bincount(idx.reshape(-1), minlength=E))
        assert np.array_equal(b["pair_row"], order // K) and np.array_equal(b["pair_rank"], order % K)
        slot = np.empty_like(order)
        slot[order] = np.arange(len(order))
        assert np.array_equal(b["slot_pair"].reshape(-1), slot)
        assert H.rel_l2(out, ref["dst"].reshape(rows, ne)) < 1e-5   # f32 throughout
    if units:
        b2.close()


@pytest.mark.parametrize("dt", [H.Q8_0, H.F16])
def test_gate_times_up_beyond_f32_beside_a_closed_gate(be, dt):
    """silu(g) is 0 for g below -104; that must hold where g * up is beyond f32 too (block formats and the float kernel)."""
    ne, nff, E, rows = 256, 128, 4, 48
    rng = np.random.default_rng(dt)
    x = (np.abs(rng.standard_normal((rows, ne))) * 1e25).astype(np.float32)
    router = np.zeros((E, ne), np.float32)
    if dt == H.F16:
        gate, up, down = ((0.02 * rng.standard_normal(E * nff * ne)).astype(np.float16) for _ in range(3))
        gate = -np.abs(gate)
        gate, up, down = gate.view(np.uint8), up.view(np.uint8), down.view(np.uint8)
    else:
        gate, up, down = _bank_weights(rng, E, nff, ne, dt, dt)
        blk = np.ascontiguousarray(gate).reshape(-1, 34)
        blk[:, 2:] = (-np.abs(blk[:, 2:].view(np.int8).astype(np.int32))).clip(-127, 0).astype(np.int8).view(np.uint8)
        gate = blk.reshape(-1)
    sel = rng.integers(0, E, (rows, 1)).astype(np.int32)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(dt), DType(dt), with_expert_ids=True)
    out, _, _ = _run_batched(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel), rows, ne)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=1, n_ff_exp=nff, gate_dtype=dt, down_dtype=dt, expert_ids=sel)
    assert not np.asarray(ref["dst"]).any() and not out.any()


@pytest.mark.parametrize("dt,act", [(H.Q8_0, M.Activation.Silu), (H.Q8_0, M.Activation.Gelu), (H.F16, M.Activation.Silu)])
def test_clamped_activation_keeps_a_nan_of_up(be, dt, act):
    """A clamp bounds `up` on both sides and lets a NaN through, as the reference's comparisons do: rows of an expert with a NaN in its
    up matrix are NaN, all others are not."""
    ne, nff, E, rows = 256, 128, 4, 48
    rng = np.random.default_rng(dt)
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    router = np.zeros((E, ne), np.float32)
    if dt == H.F16:
        gate, up, down = ((0.1 * rng.standard_normal(E * nff * ne)).astype(np.float16).view(np.uint8) for _ in range(3))
    else:
        gate, up, down = _bank_weights(rng, E, nff, ne, dt, dt)
    up = np.ascontiguousarray(up).copy()
    row_bytes = len(up) // (E * nff)
    up[(nff + 5) * row_bytes:][:2] = (0x00, 0x7E)   # expert 1, feature 5: the first block's scale, or the first element
    sel = rng.integers(0, E, (rows, 1)).astype(np.int32)
    g, ids = moe_graph(rows, ne, E, 1, nff, DType(dt), DType(dt), with_expert_ids=True, swiglu_clamp=2.0, act=act)
    out, _, _ = _run_batched(be, g, ids, dict(x=x, router=router, gate=gate, up=up, down=down, expert_ids=sel), rows, ne)
    ref = O.moe_ffn(x, router, gate, up, down, ne=ne, n_expert=E, n_used=1, n_ff_exp=nff, gate_dtype=dt, down_dtype=dt, expert_ids=sel,
                    swiglu_clamp=2.0, act=int(act))["dst"].reshape(rows, ne)
    hit = sel[:, 0] == 1
    assert np.isnan(ref[hit]).all() and np.isfinite(ref[~hit]).all()
    assert np.isnan(out[hit]).all()
    assert H.rel_l2(out[~hit], ref[~hit]) < REL_L2_MFMA


@pytest.mark.parametrize("gdt,ddt,ne,nff,rows,K,act,clamp", [
    (H.Q4K, H.Q6K, 512, 256, 300, 2, M.Activation.Silu, None), (H.Q4K, H.Q6K, 256, 4352, 130, 1, M.Activation.Silu, None),
    (H.Q8_0, H.Q8_0, 320, 192, 131, 3, M.Activation.Gelu, None), (H.Q5K, H.Q4K, 256, 256, 129, 2, M.Activation.Sigmoid, None),
    (H.MXFP4, H.IQ4_XS, 192, 256, 257, 4, M.Activation.Silu, 0.75), (H.Q4_0, H.Q8_0, 4416, 192, 128, 2, M.Activation.Gelu, 0.5),
])
def test_always_on_expert_in_the_gemms_keeps_the_bits_of_the_ops(be, gdt, ddt, ne, nff, rows, K, act, clamp):
    """The always-on expert's part of a folded batch, activation included, is what Linear, Linear, GatedAct, Linear, Add give: the
    same bits, on tiles of up to 64 and of up to 128 tokens."""
    rng = np.random.default_rng(gdt * 71 + ddt + rows)
    E = 9
    x = rng.standard_normal((rows, ne)).astype(np.float32)
    x[1::7] *= 40.0                                   # closed and wide open gates
    router = (rng.standard_normal((E, ne)) * 0.05).astype(np.float32)
    gate, up, down = _bank_weights(rng, E, nff, ne, gdt, ddt)
    sg, su, sd = _bank_weights(rng, 1, nff, ne, gdt, ddt)
    outs = {}
    for off in (False, True):
        g = M.Graph()
        t = lambda kind, shape, dt=DType.F32: getattr(g, kind)(M.TensorDesc(list(shape), dt))  # noqa: E731
        xt, out = t("input", (rows, ne)), t("output", (rows, ne))
        ws = [t("weight", sh, dt) for sh, dt in (((E, ne), DType.F32), ((E, nff, ne), DType(gdt)), ((E, nff, ne), DType(gdt)),
                                                 ((E, ne, nff), DType(ddt)), ((nff, ne), DType(gdt)), ((nff, ne), DType(gdt)),
                                                 ((ne, nff), DType(ddt)))]
        moe, tg, tu, ta, ts = (t("internal", (rows, n)) for n in (ne, nff, nff, nff, ne))
        g.moe_ffn(x=xt, router=ws[0], gate_exps=ws[1], up_exps=ws[2], down_exps=ws[3], dst=moe, ne=ne, n_expert=E, n_used=K, n_ff_exp=nff,
                  act=act, swiglu_clamp=clamp)
        g.linear(x=xt, weight=ws[4], dst=tg, m=rows, in_f=ne, out_f=nff)
        g.linear(x=xt, weight=ws[5], dst=tu, m=rows, in_f=ne, out_f=nff)
        g.gated_act(gate=tg, up=tu, dst=ta, rows=rows, nff=nff, act=act, swiglu_clamp=clamp)
        g.linear(x=ta, weight=ws[6], dst=ts, m=rows, in_f=nff, out_f=ne)
        g.add(a=moe, b=ts, dst=out, n=rows * ne)
        b = M.Backend(0, disable_op_fusion=True) if off else be
        try:
            b.prof_enable(True)
            b.prof_read()
            outs[off] = M.run_graph(b, g, list(zip([xt] + ws, [x, router, gate, up, down, sg, su, sd])), out, rows * ne)
            assert any(n.startswith("linear") for n in b.prof_read()) == off
            b.prof_enable(False)
        finally:
            if off:
                b.close()
    assert np.isfinite(outs[False]).all()
    assert np.array_equal(bits(outs[False]), bits(outs[True]))


@pytest.mark.parametrize("follower", ["projection", "gated", "fusion off", "up format"])
def test_scratch_for_an_always_on_expert_only_where_it_joins(be, follower):
    """A Linear that reads the op's input is no always-on expert by itself: a projection beside the op, the gate logit of the gated form,
    fusion switched off, an expert in another format.  Such a plan takes the op's scratch and the other tensors, no room for the expert's
    rows (512 * (2.125 * 2048 + 4 * 4096) bytes would be 10 MB)."""
    ne, nff, E, K, rows = 4096, 2048, 8, 2, 512

    def plan_bytes(b, with_linears):
        g = M.Graph()
        t = lambda kind, shape, dt=DType.F32: getattr(g, kind)(M.TensorDesc(list(shape), dt))  # noqa: E731
        xt, out = t("input", (rows, ne)), t("output", (rows, ne))
        w = lambda *shape: t("weight", shape, DType.Q4K)  # noqa: E731
        g.moe_ffn(x=xt, router=t("weight", (E, ne)), gate_exps=w(E, nff, ne), up_exps=w(E, nff, ne), down_exps=w(E, ne, nff), dst=out,
                  ne=ne, n_expert=E, n_used=K, n_ff_exp=nff)
        if with_linears:
            wide = 1 if follower == "gated" else nff
            wt = t("weight", (wide, ne), DType.Q6K if follower == "up format" else DType.Q4K)
            g.linear(x=xt, weight=wt, dst=t("output", (rows, wide)), m=rows, in_f=ne, out_f=wide)
        b.sync()
        before = _free_device_bytes()
        p = b.compile(g)
        b.sync()
        taken = before - _free_device_bytes()
        p.free()
        return taken

    b = M.Backend(0, disable_op_fusion=True) if follower == "fusion off" else be
    try:
        plan_bytes(b, False)
        alone, beside = plan_bytes(b, False), plan_bytes(b, True)
    finally:
        if b is not be:
            b.close()
    assert alone >= 2 * rows * K * nff * 4
    assert beside - alone <= 4 << 20   # the Linear's table, and the allocator's granule


@pytest.mark.parametrize("dt,in_f", [(H.Q3K, 512), (H.Q4_1, 320), (H.IQ3_S, 256)])
@pytest.mark.parametrize("rows,out_f", [(128, 128), (150, 100), (257, 300), (512, 130), (577, 640), (1100, 129)])
def test_dense_matrix_of_the_unit_decoder(be, dt, in_f, rows, out_f):
    """A Linear in a format of the unit decoder, one to eighteen tiles of 64 rows (groups of one to four of them) times one to five columns:
    every item is worked on once, and a row has the bits it has among fewer rows."""
    rng = np.random.default_rng(dt * 73 + rows)
    x = rng.standard_normal((rows, in_f)).astype(np.float32)
    w = H.centred_weight(dt, out_f * in_f, 5)

    def linear(v):
        g = M.Graph()
        xt, wt = g.input(M.TensorDesc([len(v), in_f], DType.F32)), g.weight(M.TensorDesc([out_f, in_f], DType(dt)))
        y = g.output(M.TensorDesc([len(v), out_f], DType.F32))
        g.linear(x=xt, weight=wt, dst=y, m=len(v), in_f=in_f, out_f=out_f)
        be.prof_enable(True)
        be.prof_read()
        out = M.run_graph(be, g, [(xt, v), (wt, w)], y, len(v) * out_f).reshape(len(v), out_f)
        assert "linear_grouped_units" in be.prof_read()
        be.prof_enable(False)
        return out

    out = linear(x)
    ref = O.linear(x, w, dt, in_f, out_f).reshape(rows, out_f)
    for r in range(rows):
        assert H.rel_l2(out[r], ref[r]) < REL_L2_MFMA, r
    assert np.array_equal(bits(linear(np.ascontiguousarray(x[-128:]))), bits(out[-128:]))
