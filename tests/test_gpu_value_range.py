"""Operands at the edges of float: infinities, NaNs, the largest floats, the smallest ones.  Contractions sum products of
bfloat16 terms, which infinities do not have and the largest floats round out of; their results must be those of float
arithmetic all the same."""

import numpy as np
import pytest

from aspen_amd import api, models as M
from tests import helpers as H

pytestmark = pytest.mark.gpu
FLT_MAX = float(np.finfo(np.float32).max)
QUEUE, ORDERED = 128, 64


@pytest.fixture
def engine_flags():
    def set_flags(flags):
        api.lib().aspen_hip_set_flags(2 | flags)
    yield set_flags
    api.lib().aspen_hip_set_flags(2)


def product(call, A, B, bias, act):
    L = api.lib()
    (m, k), n = A.shape, B.shape[0]
    ldc = -(-m // 4) * 4
    out = np.zeros((n, ldc), dtype=np.float32)
    bufs = [L.aspen_hip_alloc(x.nbytes) for x in (A, B, bias, out)]
    try:
        assert all(bufs)
        for d, h in zip(bufs, (A, B, bias, out)):
            assert L.aspen_hip_h2d(d, h.ctypes.data, h.nbytes) == 0
        assert call(m, n, k, bufs[0], k, bufs[1], k, bufs[3], ldc, bufs[2], act) == 0, L.aspen_hip_last_error()
        assert L.aspen_hip_d2h(out.ctypes.data, bufs[3], out.nbytes) == 0
    finally:
        for b in bufs:
            L.aspen_hip_free(b)
    return out[:, :m]


@pytest.mark.parametrize("entry", ["aspen_hip_sgemm", "aspen_hip_sgemm_static"])
@pytest.mark.parametrize("act", [api.NO_ACTIVATION, api.RELU], ids=["linear", "relu"])
@pytest.mark.parametrize("m,n,k", [(40, 37, 96), (33, 31, 3072), (513, 1025, 64), (1031, 2570, 96)])
def test_products_of_infinite_and_largest_operands(gpu, entry, act, m, n, k):
    """Rows of A and of B with one value of +inf, -inf, NaN, +-FLT_MAX, 0.9985 FLT_MAX (rounds to the largest bfloat16 or to
    infinity, either way) at three K positions; their partners there are ordinary, powers of two (terms m and l zero),
    zero, or such a value themselves.  Expected: the 64-bit sum as a float.  Sums beyond the largest float are infinite,
    nothing lies close to the limit.  Finite ones: at most one rounding of 2^-24 of the sum of magnitudes per K
    position (two when it has to be formed by the single-precision instruction, half of that)."""
    rng = np.random.default_rng(m + n + k + act)
    A, B = rng.uniform(-0.25, 0.25, (m, k)).astype(np.float32), rng.uniform(-0.25, 0.25, (n, k)).astype(np.float32)
    bias = rng.uniform(-1, 1, m).astype(np.float32)
    at = [0, k // 2, k - 1]
    special = [np.inf, -np.inf, np.nan, FLT_MAX, -FLT_MAX, 0.9985 * FLT_MAX, 0.996 * FLT_MAX]
    for X, rows in ((A, m), (B, n)):
        X[5:11, at] = np.array([0.0, 0.25, -0.125, 0.0, 2.0 ** -126, -0.25])[:, None]
        for i, v in enumerate(special):
            X[11 + 2 * i, at[i % 3]] = v
            X[rows - 1 - i, at[(i + 1) % 3]] = v
    got = product(getattr(api.lib(), entry), A, B, bias, act)
    with np.errstate(all="ignore"):
        A64, B64 = A.astype(np.float64), B.astype(np.float64)
        a, b = A64.copy(), B64.copy()
        a[:, at] = 0
        b[:, at] = 0
        exact, scale = b @ a.T + bias, np.abs(b) @ np.abs(a).T + np.abs(bias)
        for i in at:        # (term by term: no library may skip a zero here)
            exact += B64[:, i, None] * A64[None, :, i]
            scale += np.abs(B64[:, i, None] * A64[None, :, i])
        if act == api.RELU:     # (a NaN is not above 0)
            exact, scale = np.where(exact > 0, exact, 0.0), np.where(np.isnan(exact), 0.0, scale)
        want = exact.astype(np.float32)
    assert np.isinf(want).any() and (np.isnan(want).any() or act == api.RELU)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    assert np.all(np.abs(got[fin].astype(np.float64) - exact[fin]) <= (k + 8) * 2.0 ** -24 * np.minimum(scale[fin], 4 * FLT_MAX))


CASES = {   # name: (cfg, batch, tiles wanted, environment, {layer: tile rows, columns})
    "three_channels": ("height=19\nwidth=23\nchannels=3", ["conv 16 3 1"], 5, 16, {}, (64, 64)),
    "table": ("height=10\nwidth=10\nchannels=48", ["conv 64 3 1"], 4, 16, {"ASPEN_GPU_NARROW_TILES": "0"}, (64, 64)),
    "small": ("height=8\nwidth=8\nchannels=64", ["conv 64 3 1"], 4, 16, {"ASPEN_GPU_NARROW_TILES": "0"}, (64, 64)),
    "narrow": ("height=8\nwidth=8\nchannels=64", ["conv 64 3 1"], 4, 16, {"ASPEN_GPU_NARROW_TILES": "1"}, (32, 32)),
    "large": ("height=64\nwidth=64\nchannels=64", ["conv 128 3 1"], 32, 16, {}, (128, 64)),
    "row_groups": ("height=64\nwidth=64\nchannels=64", ["conv 320 1 0"], 32, 2048, {}, (256, 64)),
    "wide": ("height=64\nwidth=64\nchannels=64", ["conv 40 1 0"], 32, 16, {}, (64, 128)),
    "tall": ("height=4\nwidth=4\nchannels=64", ["fc 200"], 9, 4, {"ASPEN_GPU_WEIGHT_STREAM_BYTES": "0"}, (128, 32)),
}


@pytest.mark.parametrize("mode,flags", [(api.MODE_LAYERS, 0), (api.MODE_DATAFLOW, QUEUE), (api.MODE_DATAFLOW, ORDERED)], ids=["layers", "queue", "ordered"])
@pytest.mark.parametrize("name", list(CASES))
def test_layers_over_infinite_and_largest_activations(gpu, engine_flags, monkeypatch, name, mode, flags):
    """Four images with a value of +inf, -inf, NaN and one whose leading term rounds to infinity, through every tile shape and
    operand kind, and through a layer that takes the result on (behind a ReLU, which lets infinities pass and makes NaNs
    0, as the reference's comparison has it): NaNs and infinities where the oracle has them, the rest to the
    tolerance of every other layer."""
    from oracle import cpu
    net_cfg, (first,), batch, tiles, env, shape = CASES[name]
    for key, value in env.items():
        monkeypatch.setenv(key, value)
    engine_flags(flags)
    kind, rows, *window = first.split()
    cfg = f"[net]\n{net_cfg}\n\n"
    if kind == "conv":
        cfg += f"[convolutional]\nfilters={rows}\nsize={window[0]}\nstride=1\npad={window[1]}\nactivation=relu\n\n"
        cfg += "[convolutional]\nfilters=32\nsize=1\nstride=1\npad=0\nactivation=linear\n\n"
    else:
        cfg += f"[connected]\noutput={rows}\nactivation=relu\n\n[connected]\noutput=40\nactivation=linear\n\n"
    layers = M.parse_cfg(cfg)
    tens = [(i, what, (v * np.float32(0.05)).astype(np.float32)) for i, what, v in M.synth_weights(layers, 71, "he")]     # (sums of the largest values stay finite)
    x = (M.synth_input(layers, 71, batch, 0, "token_ids") * 2.0 - 1.0).astype(np.float32)
    px = x.reshape(batch, -1, x.shape[-1])
    px[0, 0, 0] = np.inf
    px[1, -1, 1] = -np.inf
    px[2, 1, 2] = FLT_MAX * 0.999
    px[3, -1, 0] = np.nan
    with np.errstate(all="ignore"):
        outs = cpu.run_network(layers, tens, x, batch, 0)
    net = H.GpuNet(cfg, tens, batch, 0, min_ninst=tiles, mode=mode)
    try:
        net.run(x)
        info = net.nasm.info(1)
        assert (info["tile_H"], info["tile_W"]) == shape, info
        for l in (1, 2):
            got, want = net.layer(l), outs[l].reshape(net.layer(l).shape)
            assert np.array_equal(np.isnan(got), np.isnan(want)), l
            inf = np.isinf(want)
            assert np.array_equal(got[inf], want[inf]) and np.array_equal(np.isinf(got), inf), l
            assert l != 1 or inf.any()
            huge = np.isfinite(want) & (np.abs(want) > 1e30)
            assert huge.any() and np.max(np.abs(got[huge].astype(np.float64) - want[huge])) <= H.REL_L2_TOL * np.max(np.abs(want[huge])), l
            ordinary = np.isfinite(want) & ~huge.any(axis=-1, keepdims=True)        # (next to huge ones: sums of the largest values that have cancelled)
            assert H.rel_l2(got[ordinary], want[ordinary]) <= H.REL_L2_TOL, l
    finally:
        net.close()


@pytest.mark.parametrize("mode,flags", [(api.MODE_LAYERS, 0), (api.MODE_DATAFLOW, QUEUE), (api.MODE_DATAFLOW, ORDERED)], ids=["layers", "queue", "ordered"])
def test_infinite_tokens_stay_in_their_sequence(gpu, engine_flags, monkeypatch, mode, flags):
    """A transformer (layer norms folded into the matmul tiles) over two sequences of which one holds an infinity: that one is
    NaN where the oracle's is, and every value of the other is bit for bit that of a run without the infinity, though
    tiles span both."""
    from oracle import cpu
    engine_flags(flags)
    monkeypatch.setenv("ASPEN_GPU_NARROW_TILES", "0")
    cfg, layers, tens, x, batch, seq = H.build_case(H.micro_cases()["bert_mini_b2_s24"])
    y = x.copy()
    y.reshape(batch, seq, -1)[1, 3, 5] = np.inf
    with np.errstate(all="ignore"):
        outs = cpu.run_network(layers, tens, y, batch, seq)
    api.lib().aspen_keep_layer_outputs(0)
    try:
        net = H.GpuNet(cfg, tens, batch, seq, min_ninst=32, mode=mode)
        try:
            last = net.nasm.num_ldata - 1
            net.run(x)
            clean = net.layer(last).reshape(batch, -1)
            net.run(y)
            got = net.layer(last).reshape(batch, -1)
            assert np.array_equal(got[0], clean[0]) and np.isfinite(clean).all()
            assert np.array_equal(np.isnan(got[1]), np.isnan(outs[-1].reshape(batch, -1)[1])) and np.isnan(got[1]).any()
        finally:
            net.close()
    finally:
        api.lib().aspen_keep_layer_outputs(1)


@pytest.mark.parametrize("m,n,k", [(40, 37, 96), (33, 31, 3072), (513, 1025, 64)])
def test_products_of_the_smallest_operands(gpu, m, n, k):
    """Operands of 2^-126 .. 2^-90 against such of 2^40 .. 2^70: terms below bfloat16's smallest number, 2^-133, do not exist, so an
    operand below 2^-110 enters with an absolute error of up to 2^-134 (and as much again in the last term's own rounding); the rest as
    for any other operand."""
    rng = np.random.default_rng(m + n + k)
    A = (rng.standard_normal((m, k)) * 2.0 ** rng.uniform(-126, -90, (m, k))).astype(np.float32)
    B = (rng.standard_normal((n, k)) * 2.0 ** rng.uniform(40, 70, (n, k))).astype(np.float32)
    for swap in (False, True):
        a, b = (B, A) if swap else (A, B)
        got = product(api.lib().aspen_hip_sgemm, a, b, np.zeros(a.shape[0], dtype=np.float32), 0)
        a, b = a.astype(np.float64), b.astype(np.float64)
        bound = (2 * (k // 16) + 4) * 2.0 ** -24 * (np.abs(b) @ np.abs(a).T)
        lost = 2.0 ** -133 * ((np.abs(a).sum(axis=1)[None, :]) if swap else np.abs(b).sum(axis=1)[:, None])
        err = np.abs(got - b @ a.T)
        print("worst", (m, n, k), swap, np.max(err / (bound + lost)), np.max(err / bound), flush=True)
        assert np.all(err <= bound + lost)


@pytest.mark.parametrize("m,n,k", [(40, 37, 32), (33, 31, 3072), (513, 1025, 64), (1031, 2570, 96)])
def test_products_whose_dropped_terms_add_up(gpu, m, n, k):
    """Operands of one sign whose mantissa leaves the most in the three partial products that are not computed: 0.991 x 2^-24 of
    every product, all in one direction (1 + 2^-8 - 2^-17 + 2^-23 has 0.98), next to one rounding per 16 K positions of the leading sum,
    2^-7 of that for the small sum, and the addition of the two: 2^-24 of the sum each."""
    worst = np.uint32(0x3f807fc0).view(np.float32)
    rng = np.random.default_rng(k)
    A = (worst * 2.0 ** rng.integers(-3, 4, (m, k))).astype(np.float32)
    B = (worst * 2.0 ** rng.integers(-3, 4, (n, k))).astype(np.float32)
    a, b = A.astype(np.float64), B.astype(np.float64)
    exact = b @ a.T
    for entry in (api.lib().aspen_hip_sgemm, api.lib().aspen_hip_sgemm_static):
        error = np.max(np.abs(product(entry, A, B, np.zeros(m, dtype=np.float32), 0) - exact) / exact)
        print("worst", (m, n, k), error * 2.0 ** 24, flush=True)
        assert error <= (k // 16 * (1 + 2.0 ** -7) + 2) * 2.0 ** -24


@pytest.mark.parametrize("mode,flags", [(api.MODE_LAYERS, 0), (api.MODE_DATAFLOW, QUEUE), (api.MODE_DATAFLOW, ORDERED)], ids=["layers", "queue", "ordered"])
@pytest.mark.parametrize("masked", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("hidden,seq", [(64, 1), (128, 63), (128, 64), (64, 65), (128, 130)])
def test_fused_attention_of_infinite_and_largest_operands(gpu, engine_flags, hidden, seq, masked, mode, flags):
    """One block of two heads of 32 or 64 channels (a fused tile: 64 queries and 64 keys at a time) over three sequences.  The first
    is ordinary.  In the second one key has +-3e38 in a channel in which some queries hold the same: scores of -inf, whose
    exponential is zero, and of +inf, whose is infinite.  In the third one token's values are infinite.  Expected: the layer's
    formula in 64 bits over the Query, Key and Value the device computed, scores rounded to float; the three-term products
    and the hardware's exponential (2^-22 of scores of a few units) stay within 1e-5 of the row's largest value."""
    engine_flags(flags)
    cfg = M.bert_cfg(1, hidden, 2, hidden)
    if masked:
        cfg = cfg.replace("[attention_k]", "[attention_k]\nmasked=1")
    layers = M.parse_cfg(cfg)
    a = next(L for L in layers if L["type"] == "attn_k")
    assert bool(a["masked"]) == masked
    qi, ki, vi = a["p0"], a["p1"], layers[a["idx"] + 1]["p1"]
    tens = M.synth_weights(layers, 5, "gpt")
    w = {(i, k): t for i, k, t in tens}
    for i in (qi, ki, vi):
        w[i, "WEIGHT"][:] *= 5
        w[i, "WEIGHT"][:, :3] = 0
    c, t, batch = 7, seq // 3, 3
    w[ki, "WEIGHT"][c] = w[qi, "WEIGHT"][c] = 0
    w[ki, "BIAS"][c] = w[qi, "BIAS"][c] = 0
    w[ki, "WEIGHT"][c, 0] = w[qi, "WEIGHT"][c, 1] = 3e38
    w[vi, "WEIGHT"][5, 2] = 3e38
    x = M.synth_input(layers, 6, batch, seq, "embeddings").reshape(batch, seq, hidden) * 20
    x[:, :, :3] = 0
    x[1, t, 0] = 1
    x[1, seq // 2:, 1] = -1
    x[1, -1, 1] = 1 if seq > 1 else -1
    x[2, t, 2] = 1e30
    api.lib().aspen_keep_layer_outputs(0)
    try:
        net = H.GpuNet(cfg, tens, batch, seq, min_ninst=8, mode=mode)
        try:
            assert net.nasm.info(a["idx"] + 1)["fused_attention"] >= 0
            net.run(np.ascontiguousarray(x, dtype=np.float32))
            q, k, v = (net.layer(i).reshape(batch, seq, 2, hidden // 2).astype(np.float64) for i in (qi, ki, vi))
            got = net.layer(a["idx"] + 1).reshape(batch, seq, 2, hidden // 2)
        finally:
            net.close()
    finally:
        api.lib().aspen_keep_layer_outputs(1)
    with np.errstate(all="ignore"):
        scores = np.einsum("bqhc,bkhc->bhqk", q, k).astype(np.float32)
        if masked:
            scores = np.where(np.arange(seq)[None, :] > np.arange(seq)[:, None], np.float32(-1e10), scores)
        e = np.exp((scores * np.float32(1 / np.sqrt(hidden // 2))).astype(np.float64)).transpose(0, 2, 3, 1)[..., None]
        weighted = e * v[:, None]
        if masked:      # blocks of 64 keys behind all of a tile's queries are not computed
            weighted[:, np.arange(seq)[None, :] // 64 > np.arange(seq)[:, None] // 64] = 0
        want = weighted.sum(2) / e.sum(2)
    assert np.isinf(v).any() and np.isfinite(want[0]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    finite = np.isfinite(want)
    most = np.max(np.abs(np.where(finite, want, 0)), axis=-1, keepdims=True)
    assert np.max(np.abs(np.where(finite, got, 0) - np.where(finite, want, 0)) / np.maximum(most, 1e-30)) <= 1e-5


@pytest.mark.parametrize("mode,flags", [(api.MODE_LAYERS, 0), (api.MODE_DATAFLOW, QUEUE), (api.MODE_DATAFLOW, ORDERED)], ids=["layers", "queue", "ordered"])
@pytest.mark.parametrize("masked", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("hidden,seq", [(64, 1), (128, 16), (128, 64), (64, 65), (128, 130)])
def test_fused_attention_of_small_exponentials(gpu, engine_flags, hidden, seq, masked, mode, flags):
    """Rows whose exponentials are all small: one block of two heads of 32 or 64 channels over five sequences whose scaled scores
    are s = -5, -76, -80, -84 and -86 (exponentials of 2^-7 ... 2^-124; float's smallest is 2^-126).  In the first head the
    scores of a sequence are equal (one channel of the queries and keys is not zero), so that its results are means of the
    values, whatever the exponentials' own error: within S + 3 roundings of 2^-24 (the sums, the quotient, what the terms leave
    out) of the row's largest value.  In the second they vary by some tenths: a score of 86 sqrt (hd) has an error of hd 2^-24 of
    its products' magnitudes and the exponent two roundings of 2^-24 of 125, together less than 2e-4 of an exponential.  A
    sixth sequence has ordinary scores and values of 1e-37 (the products
    that make them lose low bits, which is no matter here)."""
    engine_flags(flags)
    cfg = M.bert_cfg(1, hidden, 2, hidden)
    if masked:
        cfg = cfg.replace("[attention_k]", "[attention_k]\nmasked=1")
    layers = M.parse_cfg(cfg)
    a = next(L for L in layers if L["type"] == "attn_k")
    qi, ki, vi = a["p0"], a["p1"], layers[a["idx"] + 1]["p1"]
    tens = M.synth_weights(layers, 5, "gpt")
    w = {(i, k): t for i, k, t in tens}
    hd, batch = hidden // 2, 6
    for i in (qi, ki, vi):
        w[i, "WEIGHT"][:, :2] = 0
        w[i, "BIAS"][:] = 0
        if i != vi:
            w[i, "WEIGHT"][:hd] = 0
            w[i, "WEIGHT"][hd:] *= 5
            w[i, "WEIGHT"][7] = w[i, "WEIGHT"][hd + 7] = 0
            w[i, "WEIGHT"][7, int(i == ki)] = w[i, "WEIGHT"][hd + 7, int(i == ki)] = 1
    x = M.synth_input(layers, 6, batch, seq, "embeddings").reshape(batch, seq, hidden) * 20
    scaled = [-5.0, -76.0, -80.0, -84.0, -86.0, 0.0]
    x[:, :, 0] = np.array(scaled)[:, None] * np.sqrt(hd) / 8
    x[:, :, 1] = 8
    x[5] = 0
    x[5, :, 2:] = M.synth_input(layers, 7, 1, seq, "embeddings").reshape(seq, hidden)[:, 2:] * 1e-34
    api.lib().aspen_keep_layer_outputs(0)
    try:
        net = H.GpuNet(cfg, tens, batch, seq, min_ninst=8, mode=mode)
        try:
            assert net.nasm.info(a["idx"] + 1)["fused_attention"] >= 0
            net.run(np.ascontiguousarray(x, dtype=np.float32))
            q, k, v = (net.layer(i).reshape(batch, seq, 2, hd).astype(np.float64) for i in (qi, ki, vi))
            got = net.layer(a["idx"] + 1).reshape(batch, seq, 2, hd)
        finally:
            net.close()
    finally:
        api.lib().aspen_keep_layer_outputs(1)
    assert np.isfinite(got).all()
    worst = np.zeros((batch, 2))
    for b in range(batch):
        for h in range(2):
            scores = q[b, :, h] @ k[b, :, h].T / np.sqrt(hd)
            assert np.abs(scores - scaled[b]).max() <= (1e-5 * abs(scaled[b]) if h == 0 else 1.0)
            if masked:
                scores = np.where(np.arange(seq)[None, :] > np.arange(seq)[:, None], -np.inf, scores)
            e = np.exp(scores)
            want = e @ v[b, :, h] / e.sum(-1, keepdims=True)
            worst[b, h] = np.max(np.abs(got[b, :, h] - want) / np.max(np.abs(v[b, :, h])))
    print("worst", (hidden, seq, masked), worst.tolist(), flush=True)
    assert np.all(worst[:, 0] <= (seq + 3) * 2.0 ** -24) and np.all(worst[:, 1] <= 2e-4)
