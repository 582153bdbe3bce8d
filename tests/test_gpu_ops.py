"""GPU parity of the op-level kernels against the CPU oracle, through the C ABI.

Bars: i32 accumulators and int8 codes bit-exact; fp32 outputs within 1e-3
relative (the stated tolerance), and in practice bit-identical because the
kernels evaluate the oracle's canonical operation order — the strict tests
assert that too.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_TOL = 1e-3


@pytest.fixture(scope="module")
def dev(pkg):
    from importlib import import_module

    d = import_module(pkg.__name__ + ".device")
    assert d.device_count() >= 1, "no HIP device visible"
    print(f"device: {d.device_name(0)}", flush=True)
    return d


def rel_err(got, want):
    den = np.maximum(np.abs(want), 1e-6)
    return float(np.max(np.abs(got.astype(np.float64) - want) / den)) if got.size else 0.0


@pytest.mark.parametrize("K,N", [(512, 1536), (512, 512), (512, 2048), (2048, 512), (512, 32000)])
@pytest.mark.parametrize("M", [1, 8, 64, 256, 4096])
def test_q8_linear_sweep(pkg, orc, dev, M, K, N):
    print(f"q8_linear M={M} K={K} N={N}", flush=True)
    a, w, mult, bias = pkg.gemm_inputs(M, K, N)
    y_ref, acc_ref, q_ref, s_ref = orc.linear_forward(a, w, mult, bias, threads=16)
    da, dw, dm, db = (dev.DeviceArray.from_host(x) for x in (a, w, mult, bias))
    di = dev.DeviceArray.zeros((M, N), np.int32)
    df = dev.DeviceArray.zeros((M, N), np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.q8_linear(da, dw, dm, db, di, df, err=err)
    dev.synchronize()
    acc, y = di.host(), df.host()
    assert err.host()[0] == 0
    assert np.array_equal(acc, acc_ref), "i32 accumulators differ"
    assert rel_err(y, y_ref) <= REL_TOL
    assert np.array_equal(y.view(np.uint32), y_ref.view(np.uint32)), "dequant not bit-identical"


@pytest.mark.parametrize("K,N", [(2048, 512), (1536, 384)])
@pytest.mark.parametrize("M", [17, 33, 50, 64])
def test_q8_linear_long_k_row_groups(pkg, orc, dev, M, K, N):
    """fp32-only outputs above 16 rows at K = 1536 or 2048 run the skinny
    kernel with one 16-row group per workgroup (the decode FFN
    down-projection's path); ragged row counts leave a partial last group.
    Bit-identical to the oracle."""
    print(f"q8_linear row groups M={M} K={K} N={N}", flush=True)
    a, w, mult, bias = pkg.gemm_inputs(M, K, N)
    y_ref, _, _, _ = orc.linear_forward(a, w, mult, bias, threads=16)
    da, dw, dm, db = (dev.DeviceArray.from_host(x) for x in (a, w, mult, bias))
    df = dev.DeviceArray.zeros((M, N), np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.q8_linear(da, dw, dm, db, None, df, err=err)
    dev.synchronize()
    assert err.host()[0] == 0
    assert np.array_equal(df.host().view(np.uint32), y_ref.view(np.uint32))


def _dequant_ref(acc, a, mult, bias, relu=False):
    inv = np.float32(1) / (a[:, None] * mult[None, :])
    y = acc.astype(np.float32) * inv + bias[None, :]
    return np.where(y > 0, y, np.float32(0)) if relu else y


@pytest.mark.parametrize("M,K,N", [
    (65, 64, 31), (64 * 3 + 1, 192, 129), (127, 2112, 64),  # 64x64 tiles, odd chunk counts, ragged edges
    (1793, 320, 2047), (1920, 128, 1900),                   # 128x128 tiles: from 224 of them
    (2305, 64, 29057),                                      # 256x128 tiles: from 2048, the last row tile of one row
    (65, 64, (1 << 20) + 8),                                # output rows past the buffer stores' offsets
    (7001, 64, 1001), (3600, 512, 2050),                    # rows stored through the caches: over 26 MB, odd strides
    (20001, 64, 150),                                       # past a round of padded 128x128 tiles: 64x64
    (8321, 704, 1025), (8321, 1088, 1025), (14593, 64, 2300),  # both outputs: 64x64, 128x128 and 256x128 tiles
])
def test_q8_linear_tile_sizes(dev, M, K, N):
    """Every tile size of the many-row GEMM at its edges, bit-identical to the
    integer product (exact in float64) dequantized in fp32; every seventh column and
    one row with a multiplier outside the fast reciprocal's range."""
    print(f"q8_linear tiles M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + N)
    q = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
    w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    a = rng.uniform(20, 60, size=M).astype(np.float32)
    mult = rng.uniform(50, 100, size=N).astype(np.float32)
    if N < 4096:
        mult[3::7] = np.float32(1e-25)
        a[M // 2] = np.float32(3e25)
    bias = rng.standard_normal(N).astype(np.float32)
    # |acc| <= 127^2 K < 2^24 up to K = 1040: exact in fp32 there
    dt = np.float32 if K <= 1040 else np.float64
    acc = (q.astype(dt) @ w.astype(dt).T).astype(np.int32)
    D = dev.DeviceArray
    dq, dw, da, dm, db = (D.from_host(x) for x in (q, w, a, mult, bias))
    di, df = D.zeros((M, N), np.int32), D.zeros((M, N), np.float32)
    for relu in (False, True) if N < 4096 else (False,):
        want = _dequant_ref(acc, a, mult, bias, relu)
        df.fill_bytes(0xFF)
        dev.q8_linear(None, dw, dm, db, None, df, relu=relu, xq=dq, xa=da)
        dev.synchronize()
        assert np.array_equal(df.host().view(np.uint32), want.view(np.uint32)), f"fp32 relu={relu}"
        df.fill_bytes(0xFF)
        di.fill_bytes(0xFF)
        dev.q8_linear(None, dw, dm, db, di, df, relu=relu, xq=dq, xa=da)
        dev.synchronize()
        assert np.array_equal(di.host(), acc)
        assert np.array_equal(df.host().view(np.uint32), want.view(np.uint32)), f"both relu={relu}"
    di.fill_bytes(0xFF)
    dev.q8_linear(None, dw, dm, db, di, None, xq=dq, xa=da)
    dev.synchronize()
    assert np.array_equal(di.host(), acc), "int32 alone"


def test_q8_linear_reciprocals(dev):
    """The dequantization's 1 / (a w) where it is taken without a division: every
    mantissa at both ends of the factors' range and in its middle."""
    M, K, D = 1 << 20, 64, dev.DeviceArray
    q, w = np.zeros((M, K), np.int8), np.zeros((3, K), np.int8)
    q[:, 0], w[:, 0] = 1, 1  # every accumulator is 1
    mult = np.float32(2.0) ** np.array([-62, 0, 61], np.float32)
    dq, dw, dm, db = (D.from_host(v) for v in (q, w, mult, np.zeros(3, np.float32)))
    out = D.zeros((M, 3), np.float32)
    for ea in (-62, 0, 61):
        print(f"reciprocals 2^{ea}", flush=True)
        for first in range(0, 1 << 23, M):
            a = (((ea + 127) << 23) + first + np.arange(M, dtype=np.uint32)).astype(np.uint32).view(np.float32)
            da = D.from_host(a)
            dev.q8_linear(None, dw, dm, db, None, out, xq=dq, xa=da)
            dev.synchronize()
            want = np.float32(1) / (a[:, None] * mult[None, :])
            assert want.dtype == np.float32
            assert np.array_equal(out.host().view(np.uint32), want.view(np.uint32)), (ea, first)


@np.errstate(over="ignore")
def test_reciprocal_factor_limits(dev):
    """Multipliers at the first and last float for which the division is left out,
    and right outside them, in each kernel that does so: IEEE results either side."""
    K, N, D = 64, 64, dev.DeviceArray
    lo, hi = np.float32(2.0) ** np.float32(-62), np.float32(2.0) ** np.float32(62)
    edges = [np.nextafter(lo, np.float32(0)), lo, np.float32(1.7), np.nextafter(hi, np.float32(0)), hi]
    rng = np.random.default_rng(57)
    q = rng.integers(-127, 128, (65, K)).astype(np.int8)
    w = rng.integers(-127, 128, (N, K)).astype(np.int8)
    bias = np.zeros(N, np.float32)
    acc = (q.astype(np.int32) @ w.astype(np.int32).T).astype(np.float32)
    dq, dw, db = (D.from_host(v) for v in (q, w, bias))
    out, tok = D.zeros((65, N), np.float32), D.zeros(65, np.int32)
    for a in edges:
        da = D.from_host(np.full(65, a, np.float32))
        for m in edges:
            dm = D.from_host(np.full(N, m, np.float32))
            want = acc * (np.float32(1) / (np.float32(a) * np.float32(m))) + bias
            dev.q8_linear(None, dw, dm, db, None, out, xq=dq, xa=da)
            dev.synchronize()
            assert np.array_equal(out.host().view(np.uint32), want.view(np.uint32)), ("rows of int8", a, m)
            # fp32 rows that the static multiplier a takes back to q (up to their rounding)
            x = (q.astype(np.float64) / np.float64(a)).astype(np.float32)
            xq = np.clip(np.rint(x * np.float32(a)), -127, 127)
            ws = (xq.astype(np.int32) @ w.astype(np.int32).T).astype(np.float32)
            dev.q8_linear_static(D.from_host(x), float(a), dw, dm, db, None, out)
            dev.synchronize()
            sw = ws * (np.float32(1) / (np.float32(a) * np.float32(m))) + bias
            assert np.array_equal(out.host().view(np.uint32), sw.view(np.uint32)), ("fp32 rows", a, m)
            dev.vocab_argmax(dq, da, dw, dm, db, tok, logits=out)
            dev.synchronize()
            lg = want.copy()
            lg[:, [1, *range(7, 39)]] = -np.inf
            assert np.array_equal(out.host().view(np.uint32), lg.view(np.uint32)), ("vocabulary", a, m)
            assert np.array_equal(tok.host(), lg.argmax(1))


@pytest.mark.parametrize("M,K,N", [
    (1, 64, 33), (16, 448, 100), (17, 512, 96), (64, 1024, 1030), (61, 1536, 384), (3, 2048, 70),  # 16-row groups
    (17, 512, 8200), (64, 64, 9000), (65, 192, 127), (129, 512, 1000),  # row tiles, 128 columns
    (1100, 320, 2300),                                                  # row tiles, 256 columns
    (65, 576, 64), (5000, 512, 2048),                                   # quantized first
    (64, 1536, 2300), (33, 1024, 8100), (16, 2048, 20000),              # quantized first: past one round of workgroups
    (64, 1536, 2048), (32, 1024, 8100), (16, 1984, 20000),              # and not
])
@pytest.mark.parametrize("act", [0.0, 31.75])
def test_q8_linear_from_fp32_rows(dev, M, K, N, act):
    """The layer from fp32 rows (their own multipliers, or a static one that clamps the
    largest values) equals the row quantization followed by the layer on its int8 rows,
    bit for bit: zero rows, a row whose multiplier overflows to infinity, halfway values,
    and the error flag of a non-finite value."""
    print(f"q8_linear fp32 rows M={M} K={K} N={N} act={act}", flush=True)
    rng = np.random.default_rng(M + K + N)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.1, 4, size=(M, 1))).astype(np.float32)
    x[0, :8] = [0.5, 1.5, -0.5, -1.5, 2.5, -2.5, 0.0, -0.0]
    if M > 2:
        x[1] = 0.0
        x[2] = 0.0
        x[2, ::3] = np.float32(1e-38)  # 127 / 1e-38 overflows
    w = rng.integers(-127, 128, size=(N, K)).astype(np.int8)
    mult = rng.uniform(50, 100, size=N).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    D = dev.DeviceArray
    dw, dm, db = (D.from_host(v) for v in (w, mult, bias))
    # The static multiplier on the host, the rows' own by the quantization kernel.
    dx = D.from_host(x)
    if act:
        dq = D.from_host(np.clip(np.rint(x * np.float32(act)), -127, 127).astype(np.int8))
        da = D.from_host(np.full(M, act, np.float32))
    else:
        dq, da = D.zeros((M, K), np.int8), D.zeros(M, np.float32)
        dev.quantize_rows(dx, dq, da)
    for bad in (False, True):
        if bad:
            x[M - 1, K - 1] = np.nan if M % 2 else np.inf
            dx = D.from_host(x)
        for relu, ints in ((False, True), (True, False)):
            wi, gi = (D.zeros((M, N), np.int32) if ints else None for _ in range(2))
            wf, gf = (D.zeros((M, N), np.float32) for _ in range(2))
            err = D.zeros(1, np.int32)
            if act:
                dev.q8_linear_static(dx, act, dw, dm, db, gi, gf, relu=relu, err=err)
            else:
                dev.q8_linear(dx, dw, dm, db, gi, gf, relu=relu, err=err)
            dev.synchronize()
            assert err.host()[0] == int(bad)
            if bad:
                continue
            dev.q8_linear(None, dw, dm, db, wi, wf, relu=relu, xq=dq, xa=da)
            dev.synchronize()
            assert np.array_equal(gf.host().view(np.uint32), wf.host().view(np.uint32))
            if ints:
                assert np.array_equal(gi.host(), wi.host())


class _Part:
    """Elements [first, ...) of a device buffer as an array of its own."""

    def __init__(self, whole, first, shape, dtype):
        self.whole, self.shape, self.dtype = whole, shape, np.dtype(dtype)
        self.ptr = whole.ptr + 4 * first

    def host(self):
        n = int(np.prod(self.shape))
        first = (self.ptr - self.whole.ptr) // 4
        return self.whole.host().reshape(-1).view(self.dtype)[first:first + n].reshape(self.shape)


@pytest.mark.parametrize("act", [0.0, 31.75])
@pytest.mark.parametrize("M,K,N", [(61, 384, 384), (64, 512, 512), (1459, 512, 512), (1459, 512, 1536), (50, 2048, 512)])
def test_q8_linear_outputs_over_the_input(dev, M, K, N, act):
    """Outputs that share memory with the fp32 rows they are computed from (the
    same buffer, the rows' second half, the int32 copy over the rows) equal the
    out-of-place call's, bit for bit, on every call of several."""
    print(f"q8_linear in place M={M} K={K} N={N} act={act}", flush=True)
    rng = np.random.default_rng(M + K)
    D = dev.DeviceArray
    x = rng.standard_normal((M, K)).astype(np.float32)
    dw = D.from_host(rng.integers(-127, 128, size=(N, K)).astype(np.int8))
    dm = D.from_host(rng.uniform(50, 100, size=N).astype(np.float32))
    db = D.from_host(rng.standard_normal(N).astype(np.float32))

    def call(dx, i32, f32):
        if act:
            dev.q8_linear_static(dx, act, dw, dm, db, i32, f32)
        else:
            dev.q8_linear(dx, dw, dm, db, i32, f32)
        dev.synchronize()

    wi, wf = D.zeros((M, N), np.int32), D.zeros((M, N), np.float32)
    call(D.from_host(x), wi, wf)
    size = M * (K + N)
    for first_in, first_out in ((0, 0), (0, M * K // 2), (M * N // 2, 0)):
        for ints in (False, True):
            for _ in range(3):
                whole = np.zeros(size, np.float32)
                whole[first_in:first_in + M * K] = x.reshape(-1)
                buf = D.from_host(whole)
                dx = _Part(buf, first_in, (M, K), np.float32)
                out = _Part(buf, first_out, (M, N), np.int32 if ints else np.float32)
                call(dx, *((out, None) if ints else (None, out)))
                want = wi if ints else wf
                assert np.array_equal(out.host().view(np.uint32), want.host().view(np.uint32)), (first_in, first_out, ints)


@pytest.mark.parametrize("K", [576, 512])
def test_q8_linear_on_two_streams_at_once(pkg, orc, dev, K):
    """The op-level entry points keep their intermediate buffers (here the
    quantized activations of an fp32 input, K = 576) per (device, stream): two
    streams that issue calls at the same time, with different row counts that
    grow on the way and no synchronization between them, each get the oracle's
    result bit for bit.  Rows of K = 512 need no such buffer."""
    N = 512
    shapes = {"a": [300, 2048, 2048, 900], "b": [96, 500, 96, 500]}
    print(f"q8_linear on two streams: K={K} rows {shapes}", flush=True)
    x, w, mult, bias = pkg.gemm_inputs(2 * 2048, K, N, seed=100)
    ref = orc.linear_forward(x, w, mult, bias, threads=16)[0]
    dw, dm, db = (dev.DeviceArray.from_host(v) for v in (w, mult, bias))
    first = {"a": 0, "b": 2048}  # each stream's own rows
    streams = {k: dev.Stream() for k in shapes}
    try:
        din = {k: [dev.DeviceArray.from_host(x[first[k]:first[k] + m]) for m in shapes[k]] for k in shapes}
        outs = {k: [dev.DeviceArray.zeros((m, N), np.float32) for m in shapes[k]] for k in shapes}
        err = dev.DeviceArray.zeros(1, np.int32)
        dev.synchronize()
        for rep in range(4):  # interleaved, never waiting
            for k in shapes:
                dev.q8_linear(din[k][rep], dw, dm, db, None, outs[k][rep], err=err, stream=streams[k].handle)
        for st in streams.values():
            st.sync()
        assert err.host()[0] == 0
        for k in shapes:
            for rep, m in enumerate(shapes[k]):
                want = ref[first[k]:first[k] + m]
                assert np.array_equal(outs[k][rep].host().view(np.uint32), want.view(np.uint32)), (k, rep)
    finally:
        for st in streams.values():
            st.close()


def test_vocab_argmax_on_two_streams_at_once(dev):
    """The argmax partials are such a buffer too: 512 and 40 rows on two streams."""
    K, V = 256, 8000
    rng = np.random.default_rng(51)
    emb = rng.integers(-127, 128, (V, K)).astype(np.int8)
    mult, bias = rng.uniform(50, 100, V).astype(np.float32), rng.standard_normal(V).astype(np.float32)
    D = dev.DeviceArray
    weights = [D.from_host(v) for v in (emb, mult, bias)]
    streams = [dev.Stream() for _ in range(2)]
    try:
        calls = []
        for st, M in zip(streams, (512, 40)):
            xq, xa = rng.integers(-127, 128, (M, K)).astype(np.int8), rng.uniform(1.0, 300.0, M).astype(np.float32)
            acc = (xq.astype(np.float32) @ emb.astype(np.float32).T)  # below 2^24: exact
            ref = acc * (np.float32(1) / (xa[:, None] * mult[None, :])) + bias
            ref[:, [1, *range(7, 39)]] = -np.inf
            calls.append((st, D.from_host(xq), D.from_host(xa), [D.zeros(M, np.int32) for _ in range(8)], ref.argmax(1)))
        dev.synchronize()
        for rep in range(8):
            for st, xq, xa, toks, _ in calls:
                dev.vocab_argmax(xq, xa, *weights, toks[rep], stream=st.handle)
        for st in streams:
            st.sync()
        for _, _, _, toks, want in calls:
            for tok in toks:
                assert np.array_equal(tok.host(), want)
    finally:
        for st in streams:
            st.close()


def test_quantize_rows_matches_oracle(pkg, orc, dev):
    rng = np.random.default_rng(11)
    x = (rng.standard_normal((300, 2048)) * rng.uniform(0.01, 50, size=(300, 1))).astype(np.float32)
    x[5] = 0.0  # all-zero row -> multiplier 1
    x[7, :10] = [0.5, 1.5, -0.5, -1.5, 2.5, -2.5, 126.5, 3.0, 0.0, -0.0]
    q_ref, a_ref = orc.quantize_rows(x)
    dx = dev.DeviceArray.from_host(x)
    dq = dev.DeviceArray.zeros(x.shape, np.int8)
    da = dev.DeviceArray.zeros(300, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.quantize_rows(dx, dq, da, err)
    dev.synchronize()
    assert np.array_equal(dq.host(), q_ref) and np.array_equal(da.host(), a_ref)
    assert err.host()[0] == 0
    # a non-finite activation raises the error flag (the reference rejects it)
    x[3, 17] = np.inf
    dx2 = dev.DeviceArray.from_host(x)
    dev.quantize_rows(dx2, dq, da, err)
    dev.synchronize()
    assert err.host()[0] == 1


def test_q8_linear_edges(pkg, orc, dev):
    rng = np.random.default_rng(12)
    # column tail (N not a multiple of 16/64), odd M on both kernels, ReLU,
    # full-range weights including -128 (exact in the int8 matrix core); the
    # last two are wide grids (more than 64 column tiles) whose tiles go in
    # groups of eight row tiles, with a partial group and ragged edges
    for M, K, N in [(3, 64, 100), (77, 128, 130), (200, 192, 65), (130, 64, 1), (200, 64, 4170),
                    (610, 128, 4500)]:
        print(f"edge M={M} K={K} N={N}", flush=True)
        a = rng.standard_normal((M, K)).astype(np.float32)
        w = rng.integers(-128, 128, size=(N, K)).astype(np.int8)
        mult = rng.uniform(50, 100, size=N).astype(np.float32)
        bias = rng.standard_normal(N).astype(np.float32)
        y_ref, acc_ref, _, _ = orc.linear_forward(a, w, mult, bias, relu=True)
        dw = dev.DeviceArray.from_host(w)
        di = dev.DeviceArray.zeros((M, N), np.int32)
        df = dev.DeviceArray.zeros((M, N), np.float32)
        dev.q8_linear(dev.DeviceArray.from_host(a), dw, dev.DeviceArray.from_host(mult),
                      dev.DeviceArray.from_host(bias), di, df, relu=True)
        dev.synchronize()
        assert np.array_equal(di.host(), acc_ref)
        assert np.array_equal(df.host(), y_ref)
    # K not a multiple of 64 is rejected on the host
    with pytest.raises(RuntimeError):
        dev.q8_linear(dev.DeviceArray.zeros((2, 100), np.float32), dev.DeviceArray.zeros((4, 100), np.int8),
                      dev.DeviceArray.zeros(4, np.float32), dev.DeviceArray.zeros(4, np.float32),
                      dev.DeviceArray.zeros((2, 4), np.int32), None)


def test_residual_layer_norm_matches_oracle(pkg, orc, dev):
    rng = np.random.default_rng(13)
    for d in (512, 384):
        y = rng.standard_normal((257, d)).astype(np.float32)
        r = (rng.standard_normal((257, d)) * 3).astype(np.float32)
        g = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
        b = (0.1 * rng.standard_normal(d)).astype(np.float32)
        ref = orc.residual_layer_norm(y, r, g, b)
        q_ref, a_ref = orc.quantize_rows(ref)
        out = dev.DeviceArray.zeros(y.shape, np.float32)
        q = dev.DeviceArray.zeros(y.shape, np.int8)
        a = dev.DeviceArray.zeros(257, np.float32)
        dev.residual_layer_norm(dev.DeviceArray.from_host(y), dev.DeviceArray.from_host(r),
                                dev.DeviceArray.from_host(g), dev.DeviceArray.from_host(b), out, q, a)
        dev.synchronize()
        assert np.array_equal(out.host(), ref)
        assert np.array_equal(q.host(), q_ref) and np.array_equal(a.host(), a_ref)


@pytest.mark.parametrize("d,rows", [(64, 2560), (192, 2561), (256, 7168), (256, 7171), (384, 7169), (384, 9473),
                                    (640, 2563), (960, 2561), (1024, 2562),
                                    (512, 7405), (256, 8193), (384, 9471)])  # one row per wave
def test_residual_layer_norm_many_rows(pkg, orc, dev, d, rows):
    """Several rows per wave at every lane layout (512 and a few row counts keep one
    row per wave): a last wave with fewer rows, rows that start at any float, and
    non-finite rows."""
    print(f"residual_layer_norm {rows} x {d}", flush=True)
    rng = np.random.default_rng(29)
    y = rng.standard_normal((rows, d)).astype(np.float32)
    r = (rng.standard_normal((rows, d)) * 3).astype(np.float32)
    y[0], r[0] = 0.0, -0.0
    y[rows - 1, d - 1], y[rows - 2, 0] = np.inf, np.nan
    g = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    b = (0.1 * rng.standard_normal(d)).astype(np.float32)
    ref = orc.residual_layer_norm(y, r, g, b)
    q_ref, a_ref = orc.quantize_rows(ref[: rows - 2])

    class Shifted:  # the buffer one element past its start
        def __init__(self, host):
            self.whole = dev.DeviceArray.from_host(np.concatenate([host.reshape(-1)[:1], host.reshape(-1)]))
            self.shape, self.ptr = host.shape, self.whole.ptr + host.itemsize

    out, q = Shifted(np.zeros_like(y)), Shifted(np.zeros(y.shape, np.int8))
    a = dev.DeviceArray.zeros(rows, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.residual_layer_norm(Shifted(y), Shifted(r), Shifted(g), Shifted(b), out, q, a, err=err)
    dev.synchronize()
    got = out.whole.host()[1:].reshape(rows, d)
    fin = slice(0, rows - 2)
    assert np.array_equal(got[fin].view(np.uint32), ref[fin].view(np.uint32))
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and err.host()[0] == 1
    assert np.array_equal(q.whole.host()[1:].reshape(rows, d)[fin], q_ref)
    assert np.array_equal(a.host()[fin], a_ref)


def _ln_edge_rows(rng, d=512):
    """Rows whose sequential sums stress the speculative folds (chunks of 64
    or 128):
    prefixes cancelling to near zero at the chunk boundaries (the candidate
    windows miss and chunks are refolded), exact zeros and negative zeros,
    constants, wide and tiny magnitudes."""
    rows = []
    for _ in range(8):  # cancellation at every 64-element chunk boundary
        z = rng.standard_normal(d).astype(np.float32) * np.float32(rng.uniform(0.5, 20))
        for k in range(64, d, 64):
            s = np.float32(-0.0)
            for v in z[:k - 1]:
                s = np.float32(s + v)
            z[k - 1] = -s + np.float32(rng.standard_normal() * 1e-5)
        rows.append(z)
    rows.append(np.zeros(d, np.float32))
    rows.append(np.full(d, -0.0, np.float32))
    rows.append(np.full(d, 0.3, np.float32))
    rows.append((rng.standard_normal(d) * 1e17).astype(np.float32))
    rows.append((rng.standard_normal(d) * 1e-39).astype(np.float32))  # subnormal
    alt = np.where(np.arange(d) % 2 == 0, 1e4, -1e4).astype(np.float32)
    rows.append(alt + (rng.standard_normal(d) * 1e-3).astype(np.float32))
    return np.stack(rows)


@pytest.mark.parametrize("d", [256, 384, 512])
def test_residual_layer_norm_single_wave_speculative_edges(pkg, orc, dev, d):
    """Rows of 256, 384 and 512 fold as two, three or four speculative
    128-element chunks inside one wave (the LayerNorms of both graphs):
    chunk boundaries where the prefix cancels to near zero force refolds; the
    result is the sequential fold's, bit for bit, and non-finite rows keep
    their NaN positions."""
    rng = np.random.default_rng(23 + d)
    z = np.concatenate([_ln_edge_rows(rng, d), rng.standard_normal((21, d)).astype(np.float32) * 3])
    y = (z * np.float32(0.75)).astype(np.float32)
    r = (z - y).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    b = (0.1 * rng.standard_normal(d)).astype(np.float32)
    ref = orc.residual_layer_norm(y, r, g, b)
    q_ref, a_ref = orc.quantize_rows(ref)
    out = dev.DeviceArray.zeros(y.shape, np.float32)
    q = dev.DeviceArray.zeros(y.shape, np.int8)
    a = dev.DeviceArray.zeros(y.shape[0], np.float32)
    dev.residual_layer_norm(dev.DeviceArray.from_host(y), dev.DeviceArray.from_host(r),
                            dev.DeviceArray.from_host(g), dev.DeviceArray.from_host(b), out, q, a)
    dev.synchronize()
    assert np.array_equal(out.host().view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(q.host(), q_ref) and np.array_equal(a.host(), a_ref)
    y2 = y[:3].copy()
    y2[0, 130] = np.nan
    y2[1, 257 % d] = np.inf
    y2[2, 5] = -np.inf
    ref2 = orc.residual_layer_norm(y2, r[:3], g, b)
    out2 = dev.DeviceArray.zeros(y2.shape, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.residual_layer_norm(dev.DeviceArray.from_host(y2), dev.DeviceArray.from_host(r[:3]),
                            dev.DeviceArray.from_host(g), dev.DeviceArray.from_host(b), out2, err=err)
    dev.synchronize()
    got2 = out2.host()
    assert np.array_equal(np.isnan(got2), np.isnan(ref2))
    fin = ~np.isnan(ref2)
    assert np.array_equal(got2[fin], ref2[fin])
    assert err.host()[0] == 1


def test_residual_layer_norm_few_rows_edge_cases(pkg, orc, dev):
    """Rows of width 512 (four speculative 128-element chunks in one wave):
    the edge rows among ordinary ones, with their quantization."""
    rng = np.random.default_rng(17)
    z = _ln_edge_rows(rng)
    base = rng.standard_normal((48, 512)).astype(np.float32) * 2
    z = np.concatenate([z, base])
    y = (z * np.float32(0.75)).astype(np.float32)
    r = (z - y).astype(np.float32)  # y + r rounds back near z; the oracle sees the same y, r
    g = (1 + 0.1 * rng.standard_normal(512)).astype(np.float32)
    b = (0.1 * rng.standard_normal(512)).astype(np.float32)
    ref = orc.residual_layer_norm(y, r, g, b)
    q_ref, a_ref = orc.quantize_rows(ref)
    out = dev.DeviceArray.zeros(y.shape, np.float32)
    q = dev.DeviceArray.zeros(y.shape, np.int8)
    a = dev.DeviceArray.zeros(y.shape[0], np.float32)
    dev.residual_layer_norm(dev.DeviceArray.from_host(y), dev.DeviceArray.from_host(r),
                            dev.DeviceArray.from_host(g), dev.DeviceArray.from_host(b), out, q, a)
    dev.synchronize()
    got = out.host()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))  # bit for bit, signed zeros too
    assert np.array_equal(q.host(), q_ref) and np.array_equal(a.host(), a_ref)
    # non-finite inputs: the same positions turn NaN / infinite, and the flag is set
    y2 = y[:4].copy()
    y2[0, 100] = np.nan
    y2[1, 300] = np.inf
    y2[2, 5] = -np.inf
    ref2 = orc.residual_layer_norm(y2, r[:4], g, b)
    out2 = dev.DeviceArray.zeros(y2.shape, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.residual_layer_norm(dev.DeviceArray.from_host(y2), dev.DeviceArray.from_host(r[:4]),
                            dev.DeviceArray.from_host(g), dev.DeviceArray.from_host(b), out2, err=err)
    dev.synchronize()
    got2 = out2.host()
    assert np.array_equal(np.isnan(got2), np.isnan(ref2))
    fin = ~np.isnan(ref2)
    assert np.array_equal(got2[fin], ref2[fin])
    assert err.host()[0] == 1


def _attention_case(pkg, orc, dev, q, k, v, cu, heads, bf16):
    T = q.shape[0]
    lens = np.diff(cu.astype(np.int64))
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    if bf16:
        qh, kh, vh = (pkg.synthetic.bf16_round(x) for x in (q, k, v))
        q, k, v = (pkg.synthetic.bf16_to_f32(x) for x in (qh, kh, vh))
        dq, dk, dv = (dev.DeviceArray.from_host(x) for x in (qh, kh, vh))
    else:
        dq, dk, dv = (dev.DeviceArray.from_host(x) for x in (q, k, v))
    ref = orc.attention(q, k, v, cu, cu, heads)
    dseq, dcu = dev.DeviceArray.from_host(seq), dev.DeviceArray.from_host(cu)
    # packed_self: the key-staging kernel (ranges up to 256 keys); otherwise
    # one wave per (row, head).
    for packed in (True, False):
        out = dev.DeviceArray.zeros((T, heads * 64), np.float32)
        dev.attention(dq, dk, dv, dseq, dcu, out, heads=heads, max_keys=int(lens.max()), bf16=bf16,
                      packed_self=packed)
        dev.synchronize()
        got = out.host()
        assert rel_err(got, ref) <= REL_TOL or np.max(np.abs(got - ref)) < 1e-5
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
            f"attention not bit-identical (packed_self={packed})"


@pytest.mark.parametrize("bf16", [False, True])
def test_varlen_attention_full_workload(pkg, orc, dev, bf16):
    q, k, v, cu = pkg.attention_inputs()
    print(f"attention T={q.shape[0]} bf16={bf16}", flush=True)
    _attention_case(pkg, orc, dev, q, k, v, cu, 8, bf16)


@pytest.mark.parametrize("bf16", [False, True])
def test_cross_attention_decode_shape(pkg, orc, dev, bf16):
    """The 256-sentence attention workload as cross-attention: one query per
    sentence (cu_q != cu_k) over that sentence's packed keys and values."""
    q, k, v, cu = pkg.attention_inputs()
    B = len(cu) - 1
    lens = np.diff(cu.astype(np.int64))
    qc = np.ascontiguousarray(q[cu[:-1].astype(np.int64)])
    if bf16:
        qh, kh, vh = (pkg.synthetic.bf16_round(x) for x in (qc, k, v))
        qc, k, v = (pkg.synthetic.bf16_to_f32(x) for x in (qh, kh, vh))
        dq, dk, dv = (dev.DeviceArray.from_host(x) for x in (qh, kh, vh))
    else:
        dq, dk, dv = (dev.DeviceArray.from_host(x) for x in (qc, k, v))
    cu_q = np.arange(B + 1, dtype=np.uint32)
    ref = orc.attention(qc, k, v, cu_q, cu, 8)
    print(f"cross-attention B={B} T={k.shape[0]} bf16={bf16}", flush=True)
    out = dev.DeviceArray.zeros((B, 512), np.float32)
    dev.attention(dq, dk, dv, dev.DeviceArray.from_host(np.arange(B, dtype=np.int32)),
                  dev.DeviceArray.from_host(cu), out, heads=8, max_keys=int(lens.max()), bf16=bf16,
                  packed_self=False)
    dev.synchronize()
    got = out.host()
    assert rel_err(got, ref) <= REL_TOL
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), "cross-attention not bit-identical"


def test_attention_edges(pkg, orc, dev):
    rng = np.random.default_rng(14)
    # single key, 64/65 keys (chunk boundary), a 1000-key row (large variant),
    # and the reference's masking KAT shape at head_dim 64
    lens = np.array([1, 64, 65, 2, 1000, 3], np.int64)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    T = int(cu[-1])
    q, k, v = (rng.standard_normal((T, 128)).astype(np.float32) for _ in range(3))
    print("attention edges", flush=True)
    _attention_case(pkg, orc, dev, q, k, v, cu, 2, False)
    # ranges of 1..256 keys around the staging kernel's batch and chunk edges
    lens = np.array([1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 2],
                    np.int64)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    T = int(cu[-1])
    q, k, v = (rng.standard_normal((T, 512)).astype(np.float32) for _ in range(3))
    print("attention edges up to 256 keys", flush=True)
    _attention_case(pkg, orc, dev, q, k, v, cu, 8, False)


@pytest.mark.parametrize("heads,head_dim,bf16,lens", [
    # every class of sequence length (up to 16, 32 and 64 m rows) and its edges, few rows and many
    (8, 64, False, [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 96, 97, 128, 129, 192, 193, 255, 256, 7]),
    (8, 64, False, [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 96, 97, 128, 129, 192, 193, 255, 256, 7] * 3),
    (8, 48, True, [256, 1, 33, 100, 16, 32]),
    (8, 48, True, [256, 1, 33, 100, 16, 32] * 12),
    # few rows: one long sequence among short ones, odd and even numbers of query tiles
    (8, 64, False, [256] + [20] * 31), (8, 64, True, [5] * 9 + [239] + [33] * 6), (4, 48, False, [20] * 30 + [512, 1]),
    # heads that leave a shared workgroup's last places empty
    (3, 64, True, [5, 16, 20, 32, 40, 130] * 50),
    (5, 48, False, [16, 17, 64, 65] * 50),
    # 257 to 512 keys: the variants that hold 512 scores a query
    (4, 64, False, [257, 320, 321, 511, 512, 3, 30]),
    (4, 64, False, [257, 320, 321, 511, 512, 3, 30] * 3),
    (4, 48, True, [400, 17, 449] * 8),
    # few long rows: one wave per (row, head), and right past that
    (1, 64, False, [300, 3, 500, 7]), (2, 48, True, [400, 200, 9, 100]), (2, 64, False, [400, 300, 60, 9]),
    # more sequences than one pass of the lookup, and more than it takes
    (4, 64, False, [1 + (7 * i) % 50 for i in range(600)]),
    (2, 64, False, [1 + (11 * i) % 70 for i in range(1030)]),
])
def test_packed_attention_units(pkg, orc, dev, heads, head_dim, bf16, lens):
    """Packed self-attention against the oracle, bit for bit, with row strides
    wider than the rows and infinite and NaN elements."""
    print(f"packed attention heads={heads} head_dim={head_dim} bf16={bf16} n={len(lens)}", flush=True)
    rng = np.random.default_rng(41)
    lens = np.array(lens, np.int64)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    T, d = int(cu[-1]), heads * head_dim
    ld = (d + 15) // 8 * 8
    wide = [rng.standard_normal((T, ld)).astype(np.float32) for _ in range(3)]
    wide[0][:: 3] *= 40.0  # scores far apart: exponentials down to denormals and zero
    # an infinite key element (scores of either sign, by the query's), a NaN one and an
    # infinite value, each in a head and sequence of its own
    wide[1][int(cu[1]), 0] = np.inf
    wide[1][int(cu[3]) - 1, head_dim] = np.nan
    wide[2][int(cu[3]), 2] = -np.inf
    if bf16:
        dev_in = [dev.DeviceArray.from_host(pkg.synthetic.bf16_round(x)) for x in wide]
        wide = [pkg.synthetic.bf16_to_f32(pkg.synthetic.bf16_round(x)) for x in wide]
    else:
        dev_in = [dev.DeviceArray.from_host(x) for x in wide]
    q, k, v = (np.ascontiguousarray(x[:, :d]) for x in wide)
    with np.errstate(all="ignore"):
        ref = orc.attention(q, k, v, cu, cu, heads)
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    out = dev.DeviceArray.zeros((T, d + 1), np.float32)
    dev.attention(*dev_in, dev.DeviceArray.from_host(seq), dev.DeviceArray.from_host(cu), out, heads=heads,
                  max_keys=int(lens.max()), bf16=bf16, head_dim=head_dim)
    dev.synchronize()
    got = out.host()
    assert np.all(got[:, d] == 0.0)
    got = np.ascontiguousarray(got[:, :d])
    nan = np.isnan(ref)
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(np.where(nan, 0, got).view(np.uint32), np.where(nan, 0, ref).view(np.uint32))


@pytest.mark.parametrize("heads,head_dim,lens", [(8, 64, [200, 3, 31] * 12), (8, 64, [17, 200]), (4, 48, [500, 40])])
def test_packed_attention_products(pkg, orc, dev, heads, head_dim, lens):
    """The products come from the matrix cores.  With one non-zero value row per
    sequence an output is one product, rounded by itself: values of every bit
    pattern (denormal, infinite, NaN, both zeros) times probabilities down to
    denormals, bit for bit against the oracle."""
    print(f"packed attention products heads={heads} lens={len(lens)}", flush=True)
    rng = np.random.default_rng(53)
    d, T = heads * head_dim, sum(lens)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    q, k = (rng.standard_normal((T, d)).astype(np.float32) * np.float32(s) for s in (6.0, 3.0))
    v = np.zeros((T, d), np.float32)
    at = cu[:-1].astype(np.int64) + rng.integers(0, lens)
    v[at] = rng.integers(0, 1 << 32, (len(lens), d), dtype=np.uint32).view(np.float32)
    v[at, ::5] = rng.integers(0, 1 << 24, (len(lens), v[0, ::5].size), dtype=np.uint32).view(np.float32)  # small
    v[at, 1::9], v[at, 2::9], v[at, 3::9] = np.inf, -0.0, np.nan
    with np.errstate(all="ignore"):
        ref = orc.attention(q, k, v, cu, cu, heads)
    out = dev.DeviceArray.zeros((T, d), np.float32)
    dev.attention(*(dev.DeviceArray.from_host(x) for x in (q, k, v)), dev.DeviceArray.from_host(seq),
                  dev.DeviceArray.from_host(cu), out, heads=heads, max_keys=max(lens), head_dim=head_dim)
    dev.synchronize()
    got, nan = out.host(), np.isnan(ref)
    small = (ref != 0) & (np.abs(ref) < np.finfo(np.float32).tiny)
    print(f"{ref.size} products, {int(small.sum())} denormal, {int(nan.sum())} NaN", flush=True)
    assert small.any() and nan.any() and np.isinf(ref).any()
    assert np.array_equal(nan, np.isnan(got))
    assert np.array_equal(np.where(nan, 0, got).view(np.uint32), np.where(nan, 0, ref).view(np.uint32))


class _Rows:
    """n rows of d elements, ld elements apart, the first at element `first` of a
    buffer that holds `size` elements; the bytes between the rows are 0xFF (NaN)."""

    def __init__(self, dev, rows, ld, size, first):
        self.whole = dev.DeviceArray(size, rows.dtype)
        self.whole.fill_bytes(0xFF)
        self.shape = (rows.shape[0], ld)  # the row stride, as the calls take it
        item = rows.dtype.itemsize
        self.ptr = self.whole.ptr + first * item
        for i, row in enumerate(np.ascontiguousarray(rows)):
            at = first + i * ld
            assert 0 <= at and at + rows.shape[1] <= size
            dev._lib.check(self.whole._lib.marian_hip_memcpy_h2d(self.ptr + i * ld * item, row.ctypes.data,
                                                                 row.nbytes), "h2d")


@pytest.mark.parametrize("heads,head_dim,bf16,lens,ldq,ldkv,shift", [
    # key rows whose 64-row chunk, query rows whose 4-row group spans more than 2^32 bytes
    (2, 64, False, [70, 3], None, 33 << 19, 0), (2, 48, True, [70, 3], None, 33 << 20, 0),
    (2, 64, False, [3, 5], 3 << 27, None, 0), (1, 64, True, [3, 5], 3 << 28, None, 0),
    # the widest strides of the path that addresses them by 32 bits
    (2, 64, False, [66], None, (1 << 24) - 8, 0), (2, 64, False, [3, 5], (1 << 26) - 8, None, 0),
    # one row for every key or query, rows that overlap, rows that go backwards
    (4, 64, False, [5, 20, 70], 0, 0, 0), (4, 48, True, [5, 20, 70], 0, 0, 0),
    (4, 64, False, [16, 9, 33, 257], None, 8, 0), (3, 48, True, [16, 9, 33], None, 136, 0),
    (4, 64, False, [16, 9, 33, 130], -256, -264, 0), (4, 64, True, [16, 9, 33, 130], -264, -256, 0),
    # buffers that start at an odd element
    (4, 64, True, [16, 9, 33, 130], None, None, 1), (4, 64, False, [16, 9, 33, 130], None, None, 1),
    (2, 64, True, [1 + (11 * i) % 70 for i in range(1030)], None, None, 1),
])
def test_packed_attention_row_strides(pkg, orc, dev, heads, head_dim, bf16, lens, ldq, ldkv, shift):
    """Any row stride that is a multiple of 8 elements and any element alignment:
    bit-identical to the oracle on the rows that the strides name."""
    print(f"packed attention heads={heads} head_dim={head_dim} bf16={bf16} ldq={ldq} ldkv={ldkv}", flush=True)
    rng = np.random.default_rng(43)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    T, d = int(cu[-1]), heads * head_dim

    def rows(ld):
        ld = d if ld is None else ld
        if abs(ld) >= d:
            x = rng.standard_normal((T, d)).astype(np.float32)
        else:  # overlapping rows of one array
            flat = rng.standard_normal((T - 1) * ld + d).astype(np.float32)
            x = np.lib.stride_tricks.as_strided(flat, (T, d), (4 * ld, 4)).copy()
        enc = pkg.synthetic.bf16_round(x) if bf16 else x
        first = shift + (T - 1) * -ld if ld < 0 else shift
        got = _Rows(dev, enc, ld, shift + (T - 1) * abs(ld) + d, first)
        return got, pkg.synthetic.bf16_to_f32(enc) if bf16 else x

    (dq, q), (dk, k), (dv, v) = rows(ldq), rows(ldkv), rows(ldkv)
    ref = orc.attention(q, k, v, cu, cu, heads)
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    out = dev.DeviceArray.zeros((T, d), np.float32)
    dev.attention(dq, dk, dv, dev.DeviceArray.from_host(seq), dev.DeviceArray.from_host(cu), out, heads=heads,
                  max_keys=int(max(lens)), bf16=bf16, head_dim=head_dim)
    dev.synchronize()
    assert np.array_equal(out.host().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("heads,head_dim,bf16,lens,max_keys", [
    (4, 64, False, [150, 40, 16, 3], 100), (4, 48, True, [150, 40, 16, 256], 1), (2, 64, False, [500, 3, 300], 300),
    (8, 64, False, [200] * 30, 100), (4, 48, True, [40, 200] * 50, 20),
    (2, 64, False, [1 + (11 * i) % 70 for i in range(1030)], 20),
    # longer than the launch holds scores for: the first 256 (512) keys
    (4, 64, False, [300, 20, 257], 200), (8, 48, True, [300, 20] * 20, 200), (2, 64, True, [600, 20], 400),
    (4, 64, False, [600, 20] * 16, 400),
    # far above the lengths: launches of many workgroups without a query
    (8, 64, False, [3, 17] * 120, 256), (8, 48, True, [1, 40] * 45, 512), (4, 64, False, [1, 4, 7] * 400, 256),
    (8, 48, True, [1, 40] * 30, 512), (4, 64, False, [1, 4, 7] * 400, 128),
])
def test_packed_attention_max_keys_off_the_lengths(pkg, orc, dev, heads, head_dim, bf16, lens, max_keys):
    """Sequences longer than max_keys (every row is written, over all its keys up to
    256, or 512 with max_keys above 256) or much shorter: bit-identical to the oracle."""
    print(f"packed attention heads={heads} head_dim={head_dim} bf16={bf16} max_keys={max_keys}", flush=True)
    rng = np.random.default_rng(47)
    d, T = heads * head_dim, sum(lens)
    hold = 256 if max_keys <= 256 else 512
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    first = np.arange(T) - cu[seq].astype(np.int64) < hold  # keys that count
    cu_k = np.concatenate([[0], np.cumsum(np.minimum(lens, hold))]).astype(np.uint32)
    q, k, v = (rng.standard_normal((T, d)).astype(np.float32) for _ in range(3))
    if bf16:
        enc = [pkg.synthetic.bf16_round(x) for x in (q, k, v)]
        q, k, v = (pkg.synthetic.bf16_to_f32(x) for x in enc)
    else:
        enc = [q, k, v]
    ref = orc.attention(q, np.ascontiguousarray(k[first]), np.ascontiguousarray(v[first]), cu, cu_k, heads)
    out = dev.DeviceArray(ref.shape, np.float32)
    out.fill_bytes(0xFF)
    dev.attention(*(dev.DeviceArray.from_host(x) for x in enc), dev.DeviceArray.from_host(seq),
                  dev.DeviceArray.from_host(cu), out, heads=heads, max_keys=max_keys, bf16=bf16, head_dim=head_dim)
    dev.synchronize()
    assert np.array_equal(out.host().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("M", [1, 64, 130])
def test_vocab_argmax_matches_oracle(pkg, orc, dev, full_model, M):
    """Up to 64 rows one row group; 130 rows run three 64-row groups side
    by side, the last one holding two rows."""
    m = full_model
    rng = np.random.default_rng(15 + M)
    x = rng.standard_normal((M, 512)).astype(np.float32)
    q_ref, a_ref = orc.quantize_rows(x)
    logits_ref, _, _, _ = orc.linear_forward(x, m.embedding, m.embedding_mult, m.output_bias)
    masked = np.zeros(m.geometry.vocab, bool)
    masked[1] = True
    masked[7:39] = True
    lm = np.where(masked[None, :], -np.inf, logits_ref).astype(np.float32)
    tok_ref = np.argmax(lm, axis=1)  # first maximum = lowest id
    dq, da = dev.DeviceArray.from_host(q_ref), dev.DeviceArray.from_host(a_ref)
    demb, dmult, dbias = (dev.DeviceArray.from_host(t) for t in
                          (m.embedding, m.embedding_mult, m.output_bias))
    tok = dev.DeviceArray.zeros(M, np.int32)
    logits = dev.DeviceArray.zeros((M, m.geometry.vocab), np.float32)
    dev.vocab_argmax(dq, da, demb, dmult, dbias, tok, logits)
    dev.synchronize()
    assert np.array_equal(tok.host(), tok_ref)
    got = logits.host()
    assert np.array_equal(got, lm)


def test_vocab_argmax_ties_pick_lowest_id(pkg, dev):
    V, K = 4096, 64
    emb = np.zeros((V, K), np.int8)
    emb[:, 0] = 1
    emb[[5, 700, 3000, 4095], 0] = 9  # four equal maxima
    mult = np.ones(V, np.float32)
    bias = np.zeros(V, np.float32)
    xq = np.zeros((3, K), np.int8)
    xq[:, 0] = 127
    xa = np.ones(3, np.float32)
    tok = dev.DeviceArray.zeros(3, np.int32)
    args = [dev.DeviceArray.from_host(t) for t in (xq, xa, emb, mult, bias)]
    dev.vocab_argmax(*args, tok)
    dev.synchronize()
    assert tok.host().tolist() == [5, 5, 5]
    emb[5, 0] = 1
    emb[700, 0] = 1
    args = [dev.DeviceArray.from_host(t) for t in (xq, xa, emb, mult, bias)]
    dev.vocab_argmax(*args, tok)
    dev.synchronize()
    assert tok.host().tolist() == [3000, 3000, 3000]
    # a masked id never wins (id 20 is in 7..38) unless the mask is off
    emb[20, 0] = 100
    args = [dev.DeviceArray.from_host(t) for t in (xq, xa, emb, mult, bias)]
    dev.vocab_argmax(*args, tok)
    dev.synchronize()
    assert tok.host().tolist() == [3000, 3000, 3000]
    dev.vocab_argmax(*args, tok, flags=pkg.FLAG_NO_GENERATION_MASK)
    dev.synchronize()
    assert tok.host().tolist() == [20, 20, 20]


@pytest.mark.gpu
def test_vocab_argmax_nonfinite_logits_follow_strict_scan(pkg, dev):
    """The reference scores with a strict '>' scan from -inf that starts at the
    first unmasked id (q8_engine.rs:749-790): NaN never wins, a row whose
    logits are all -inf or NaN yields its first candidate, and -0.0 ties with
    +0.0.  Zero activations make every logit equal to its bias."""
    V, K = 4096, 64
    emb = np.zeros((V, K), np.int8)
    mult = np.ones(V, np.float32)
    xq = np.zeros((2, K), np.int8)
    xa = np.ones(2, np.float32)

    def run(bias):
        tok = dev.DeviceArray.zeros(2, np.int32)
        args = [dev.DeviceArray.from_host(t) for t in (xq, xa, emb, mult, bias)]
        dev.vocab_argmax(*args, tok)
        dev.synchronize()
        return tok.host().tolist()

    b = np.full(V, -np.inf, np.float32)
    b[[0, 2, 900]] = np.nan
    assert run(b) == [0, 0]          # only -inf / NaN: first candidate (id 0)
    b[0] = -np.inf
    b[[3, 4]] = np.nan
    assert run(b) == [0, 0]
    b[3000] = -5.0
    b[3001] = np.nan
    assert run(b) == [3000, 3000]    # the one finite logit wins over NaN
    b = np.full(V, -1.0, np.float32)
    b[50] = -0.0
    b[100] = 0.0
    assert run(b) == [50, 50]        # -0.0 == +0.0: the lower id
    b[50] = 0.0
    b[100] = -0.0
    assert run(b) == [50, 50]


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,V", [(1, 64, 40), (17, 512, 130), (64, 384, 4097), (70, 512, 300), (200, 256, 1000),
                                   (3, 64, 33000)])
@pytest.mark.parametrize("scale", [0, 70, -90])
def test_vocab_argmax_ties_and_factors(pkg, dev, M, K, V, scale):
    """Logits and tokens against IEEE float32 arithmetic: multipliers within the
    short reciprocal's exponents and, scaled by 2^scale in one column, outside
    them; duplicate columns, so equal logits must keep the lowest id across
    lanes, column tiles, waves and workgroups."""
    print(f"vocab_argmax M={M} K={K} V={V} scale={scale}", flush=True)
    rng = np.random.default_rng(7)
    emb = rng.integers(-127, 128, (V, K)).astype(np.int8)
    emb[V // 2:] = emb[: V - V // 2]  # every column at least twice
    mult = np.full(V, 37.5, np.float32)
    bias = np.full(V, 0.25, np.float32)
    mult[V - 1] *= np.float32(2.0) ** scale
    xq = rng.integers(-127, 128, (M, K)).astype(np.int8)
    xa = rng.uniform(1.0, 300.0, M).astype(np.float32)
    acc = (xq.astype(np.int32) @ emb.astype(np.int32).T).astype(np.float32)
    ref = acc * (np.float32(1) / (xa[:, None] * mult[None, :])) + bias
    assert ref.dtype == np.float32
    ids = np.arange(V)
    ref[:, (ids == 1) | ((ids >= 7) & (ids <= 38))] = -np.inf
    tok, logits = dev.DeviceArray.zeros(M, np.int32), dev.DeviceArray.zeros((M, V), np.float32)
    dev.vocab_argmax(*(dev.DeviceArray.from_host(t) for t in (xq, xa, emb, mult, bias)), tok, logits=logits)
    dev.synchronize()
    assert np.array_equal(logits.host().view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(tok.host(), np.argmax(ref, axis=1).astype(np.int32))


# ---- static activation multiplier (the reference's Q8 models) ---------------------
@pytest.mark.parametrize("K,N", [(512, 1536), (2048, 512), (512, 32000)])
@pytest.mark.parametrize("M", [1, 8, 64, 256])
def test_q8_linear_static_matches_oracle(pkg, orc, dev, M, K, N):
    a, w, mult, bias = pkg.gemm_inputs(M, K, N, seed=9)
    act = float(np.float32(127) / np.float32(np.abs(a).max() * 0.75))  # a few saturate
    print(f"q8_linear_static M={M} K={K} N={N} act_mult={act:.4f}", flush=True)
    y_ref, acc_ref, _ = orc.linear_forward_static(a, w, mult, bias, act, threads=16)
    da, dw, dm, db = (dev.DeviceArray.from_host(x) for x in (a, w, mult, bias))
    di = dev.DeviceArray.zeros((M, N), np.int32)
    df = dev.DeviceArray.zeros((M, N), np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.q8_linear_static(da, act, dw, dm, db, di, df, err=err)
    dev.synchronize()
    assert err.host()[0] == 0
    assert np.array_equal(di.host(), acc_ref), "i32 accumulators differ"
    assert np.array_equal(df.host().view(np.uint32), y_ref.view(np.uint32))


def test_q8_linear_static_reference_kat(pkg, dev, kats):
    """q8_gemm.rs:620-668 on the GPU: K padded to 64 with zero activations
    and weights (quantized to 0, so the accumulators are unchanged)."""
    k = kats["linear_integer_oracle"]
    w = np.zeros((2, 64), np.int8)
    w[:, :4] = np.array(k["weights_out_in"], np.int8)
    mult = np.full(2, k["weight_mult"], np.float32)
    bias = np.array(k["bias"], np.float32)
    dw, dm, db = (dev.DeviceArray.from_host(x) for x in (w, mult, bias))
    for rows in k["inputs"]:
        x = np.zeros((len(rows), 64), np.float32)
        x[:, :4] = np.array(rows, np.float32)
        q = np.clip(np.rint(x * 4.0), -127, 127).astype(np.int64)
        expected = (q @ w.T.astype(np.int64)).astype(np.float32) / np.float32(32.0) + bias
        dx = dev.DeviceArray.from_host(x)
        df = dev.DeviceArray.zeros((len(rows), 2), np.float32)
        dev.q8_linear_static(dx, k["activation_mult"], dw, dm, db, None, df)
        dev.synchronize()
        assert np.array_equal(df.host(), expected)


@pytest.mark.parametrize("d", [64, 384, 512])
@pytest.mark.parametrize("rows", [1, 7, 300])
def test_ssru_layer_norm_matches_oracle(pkg, orc, dev, rows, d):
    rng = np.random.default_rng(rows * 1000 + d)
    c, f, s, r = (rng.standard_normal((rows, d)).astype(np.float32) * 2 for _ in range(4))
    f[0, :8] = [np.inf, -np.inf, 0.0, -0.0, 88.7, -88.7, 104.0, -104.0]  # gate saturation edges
    s[0, 8:12] = [-0.0, 0.0, -1e-30, 1e-30]
    g = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    b = (0.1 * rng.standard_normal(d)).astype(np.float32)
    out_ref, st_ref = orc.ssru_layer_norm(c, f, s, r, g, b)
    q_ref, a_ref = orc.quantize_rows(out_ref)
    print(f"ssru rows={rows} d={d}", flush=True)
    dc, dfg, ds, dr, dg, dbb = (dev.DeviceArray.from_host(x) for x in (c, f, s, r, g, b))
    out = dev.DeviceArray.zeros((rows, d), np.float32)
    q = dev.DeviceArray.zeros((rows, d), np.int8)
    a = dev.DeviceArray.zeros(rows, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.ssru_layer_norm(dc, dfg, ds, dr, dg, dbb, out, q=q, a=a, err=err)
    dev.synchronize()
    assert err.host()[0] == 0
    assert np.array_equal(ds.host().view(np.uint32), st_ref.view(np.uint32)), "state differs"
    assert np.array_equal(out.host().view(np.uint32), out_ref.view(np.uint32)), "output differs"
    assert np.array_equal(q.host(), q_ref) and np.array_equal(a.host(), a_ref)


# ---- lexical shortlist: scoring only the candidate ids ----------------------------
def test_candidate_argmax_matches_oracle(pkg, orc, dev, full_model):
    import importlib

    sl = importlib.import_module(pkg.__name__ + ".shortlist")
    m = full_model
    V, K = m.geometry.vocab, m.geometry.dim
    rng = np.random.default_rng(33)
    # a synthetic shortlist: 100 source ids, 40 targets each, firstNum 100
    src_v = 100
    offs_t = np.arange(0, 40 * src_v + 1, 40, dtype=np.int64)
    targets = rng.integers(0, V, size=40 * src_v).astype(np.uint32)
    short = sl.LexicalShortlist.from_bytes(sl.LexicalShortlist.to_bytes(100, offs_t, targets), src_v, V)
    lists = [short.candidates(rng.integers(0, src_v, size=n)) for n in (3, 17, 60, 1)]
    lists.append(sl.LexicalShortlist.from_bytes(None, src_v, V).candidates([]))  # the full vocabulary
    M = len(lists)
    xq = rng.integers(-127, 128, size=(M, K)).astype(np.int8)
    xa = rng.uniform(1.0, 50.0, size=M).astype(np.float32)
    flat, offs, mx = sl.pack_candidates(lists)
    tok_ref, lg_ref = orc.candidate_argmax(xq, xa, m.embedding, m.embedding_mult, m.output_bias,
                                           flat, offs)
    print(f"candidate_argmax: {M} rows, list lengths {np.diff(offs).tolist()}", flush=True)
    d = {k: dev.DeviceArray.from_host(v) for k, v in dict(
        xq=xq, xa=xa, emb=m.embedding, mult=m.embedding_mult, bias=m.output_bias, cand=flat,
        offs=offs).items()}
    tok = dev.DeviceArray.zeros(M, np.int32)
    lg = dev.DeviceArray.zeros(flat.size, np.float32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.candidate_argmax(d["xq"], d["xa"], d["emb"], d["mult"], d["bias"], d["cand"], d["offs"], mx,
                         tok, logits=lg, err=err)
    dev.synchronize()
    assert err.host()[0] == 0
    assert np.array_equal(tok.host(), tok_ref)
    assert np.array_equal(lg.host().view(np.uint32), lg_ref.view(np.uint32))
    # the full-vocabulary list scores like the vocabulary kernel (masked ids excluded)
    dt = dev.DeviceArray.zeros(1, np.int32)
    dev.vocab_argmax(dev.DeviceArray.from_host(xq[-1:]), dev.DeviceArray.from_host(xa[-1:]),
                     d["emb"], d["mult"], d["bias"], dt)
    dev.synchronize()
    assert dt.host()[0] == tok.host()[-1]


def test_candidate_argmax_ties_and_bad_ids(pkg, orc, dev):
    rng = np.random.default_rng(35)
    V, K = 300, 64
    emb = rng.integers(-127, 128, size=(V, K)).astype(np.int8)
    emb[201] = emb[200]
    mult = np.full(V, 100.0, np.float32)
    bias = np.zeros(V, np.float32)
    xq = emb[200:201].copy()
    xa = np.ones(1, np.float32)
    cand = np.array([0, 5, 200, 201, 250], np.uint32)
    offs = np.array([0, 5], np.uint32)
    tok_ref, _ = orc.candidate_argmax(xq, xa, emb, mult, bias, cand, offs)
    assert tok_ref[0] == 200
    D = dev.DeviceArray.from_host
    tok = dev.DeviceArray.zeros(1, np.int32)
    err = dev.DeviceArray.zeros(1, np.int32)
    dev.candidate_argmax(D(xq), D(xa), D(emb), D(mult), D(bias), D(cand), D(offs), 5, tok, err=err)
    dev.synchronize()
    assert tok.host()[0] == 200 and err.host()[0] == 0
    bad = np.array([0, 5, 200, V + 7, 201], np.uint32)
    dev.candidate_argmax(D(xq), D(xa), D(emb), D(mult), D(bias), D(bad), D(offs), 5, tok, err=err)
    dev.synchronize()
    assert err.host()[0] == 1 and tok.host()[0] == 200


@pytest.mark.parametrize("packed", [True, False])
def test_attention_head_dim_48(pkg, orc, dev, packed):
    """Heads of width 48 (the reference's 384-wide, 8-head model): packed
    self-attention (key-staging kernel, ranges up to 256 keys) and the
    one-wave-per-(row, head) kernel, against the oracle bit for bit."""
    rng = np.random.default_rng(48)
    lens = np.array([1, 5, 47, 64, 65, 130, 256, 3], np.int64)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    T = int(cu[-1])
    q, k, v = (rng.standard_normal((T, 384)).astype(np.float32) for _ in range(3))
    ref = orc.attention(q, k, v, cu, cu, 8)
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    D = dev.DeviceArray.from_host
    out = dev.DeviceArray.zeros((T, 384), np.float32)
    dev.attention(D(q), D(k), D(v), D(seq), D(cu), out, heads=8, max_keys=int(lens.max()),
                  packed_self=packed, head_dim=48)
    dev.synchronize()
    assert np.array_equal(out.host().view(np.uint32), ref.view(np.uint32))
    # cross-attention shape: one query per sequence
    B = len(lens)
    qc = np.ascontiguousarray(q[cu[:-1].astype(np.int64)])
    refc = orc.attention(qc, k, v, np.arange(B + 1, dtype=np.uint32), cu, 8)
    outc = dev.DeviceArray.zeros((B, 384), np.float32)
    dev.attention(D(qc), D(k), D(v), D(np.arange(B, dtype=np.int32)), D(cu), outc, heads=8,
                  max_keys=int(lens.max()), packed_self=False, head_dim=48)
    dev.synchronize()
    assert np.array_equal(outc.host().view(np.uint32), refc.view(np.uint32))
