"""GPU parity of the activation-quantised FP8 linear (fp8.py:111-193) at the
adjacent projections' shapes (l42_reference.py:89-102) and of the group-128
activation quant that feeds it (l42_reference.py:390-403).

EXACT is compared bit for bit with the oracle's s14o_fp8_linear (k
ascending inside each 128-k group, then acc += partial).  FAST (MFMA) is
compared with the same oracle within the reference's own tolerance for this
function (test_primitives.py:109: rtol 2e-5), taken relative to the row's
sum of |products| so that cancellation in a row cannot hide or fake an
error."""

from __future__ import annotations

import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from colormlm_amd import s14  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = {"wq_b": (32768, 1024), "wkv": (512, 4096), "wo_a": (8192, 4096), "wo_b": (4096, 8192)}


# The tests below that name a kernel, with the shapes that reach it: test_linear_plan.py
# holds each to that kernel by the library's own rule.  (m, n, k[, f32 scales])
EXACT_MFMA = [(2, 300, 384), (3, 64, 128), (5, 4160, 1152), (13, 1000, 640), (17, 8192, 256), (31, 2000, 1536),
              (33, 16450, 512), (65, 700, 2176), (97, 8200, 384), (160, 12288, 256), (52, 4160, 640), (132, 1000, 640),
              (12, 8192, 2048), (65, 8192, 2048), (9, 1967, 3200), (23, 7239, 1664), (65, 9982, 1152),
              (52, 4131, 640), (33, 16450, 640), (40, 32768, 1024)]
EXACT_TILE_CHUNKS = [(40, 32768, 1024, True), (7, 129, 4096, False)]
FAST_PROMPT = [(9, 33000, 1024, False), (31, 8192, 1536, True), (33, 4099, 4096, False), (64, 1030, 8192, True),
               (65, 8200, 1024, False), (200, 512, 4096, False), (333, 700, 2560, True), (129, 32768, 1024, False),
               (512, 32768, 1024, False)]
FAST_LAUNCHES = [(1100, 2, 131072, False), (1060, 2, 131072, True)]


def say(msg: str) -> None:
    print(f"[gpu-test] {msg}", file=sys.stderr, flush=True)


def dev(a: np.ndarray) -> "torch.Tensor":
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t) -> np.ndarray:
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = s14.Context(0)
    yield c
    torch.cuda.synchronize()
    c.destroy()


def codes(rng, shape) -> np.ndarray:
    c = rng.integers(0, 256, shape, dtype=np.uint8)
    c[(c & 0x7F) == 0x7F] = 0x7E  # no NaN codes (the caller's to reject)
    return c


def weight(n, k, seed):
    rng = np.random.default_rng(seed)
    return codes(rng, (n, k)), rng.integers(114, 122, (-(-n // 128), -(-k // 128)), dtype=np.uint8)


def decoded(oracle, c, scales, row_group):
    n, k = c.shape
    lut = np.array([oracle.e4m3fn(i) for i in range(256)], np.float64)
    s = scales.astype(np.float64) if scales.dtype == np.float32 else np.exp2(scales.astype(np.float64) - 127)
    s = np.repeat(np.repeat(s, row_group, 0), 128, 1)[:n, :k]
    return lut[c] * s


def check_fast(oracle, got, want, x, xs, w, ws, what, l1=None):
    """|fast - oracle| <= 2e-6 * sum_k |x_k w_k| of the row (f32 summation
    error; measured <= 3.2e-7)."""
    if l1 is None:
        l1 = np.abs(decoded(oracle, x, xs, 1)) @ np.abs(decoded(oracle, w, ws, 128)).T
    err = np.abs(got.astype(np.float64) - want)
    ratio = float(np.max(err / np.maximum(l1, 1e-30)))
    say(f"  {what}: fast max |err| / row L1 = {ratio:.3g}")
    assert np.all(np.isfinite(got)) and ratio <= 2e-6


def test_act_quant_group128_bit_exact(ctx, oracle):
    say("act quant, groups of 128 (and 64, 32)")
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((5, 8192)) * np.exp(rng.uniform(-8, 8, (5, 8192)))).astype(np.float32)
    x[0, :128] *= 1e-9  # below the 1e-4 amax floor
    x[1, 5] = 1e30  # saturating group
    x[2, 7] = np.nan  # ignored by the amax scan
    for group in (128, 64, 32):
        q, s = torch.empty((5, 8192), dtype=torch.uint8, device="cuda"), torch.empty(
            (5, 8192 // group), dtype=torch.uint8, device="cuda")
        s14.act_quant_e4m3(ctx, dev(x), q, s, group=group)
        qo, so = oracle.requant_e4m3(x, group=group)
        assert np.array_equal(host(q), qo) and np.array_equal(host(s), so), group


@pytest.mark.parametrize("rows,k", [(1, 128), (3, 384), (7, 1152)])
def test_act_quant_alignment_and_odd_sizes(ctx, oracle, rows, k):
    """The float4 kernel (shift 0) and the one-thread-per-group kernel that
    takes an x or q off its alignment, at sizes that leave a workgroup partly
    filled: both equal the oracle, and each other where a group holds an
    infinity (whose scale the oracle does not define)."""
    say(f"act quant rows={rows} k={k}")
    rng = np.random.default_rng(rows * k)
    x = (rng.standard_normal((rows, k)) * np.exp(rng.uniform(-6, 6, (rows, k)))).astype(np.float32)
    x[0, 3], x[-1, -1], x[0, 64] = 1e30, -np.nan, 0.0
    xi = x.copy()
    xi[0, 5], xi[-1, k // 2] = np.inf, -np.inf

    def quant(v, shift, group):
        flat = torch.zeros(rows * k + 4, dtype=torch.float32, device="cuda")
        xd = flat[shift:shift + rows * k].view(rows, k)
        xd.copy_(dev(v))
        qf = torch.zeros(rows * k + 4, dtype=torch.uint8, device="cuda")
        q = qf[shift:shift + rows * k].view(rows, k)
        s = torch.empty((rows, k // group), dtype=torch.uint8, device="cuda")
        s14.act_quant_e4m3(ctx, xd, q, s, group=group)
        assert not host(qf)[shift + rows * k:].any() and not host(qf)[:shift].any()
        return host(q), host(s)

    for group in (128, 64, 32):
        want = oracle.requant_e4m3(x, group=group)
        for shift in (0, 1, 2):
            got = quant(x, shift, group)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), (group, shift)
        a, b = quant(xi, 0, group), quant(xi, 1, group)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), group


@pytest.mark.parametrize("group", [32, 64, 128])
def test_act_quant_conversion_range(ctx, oracle, group):
    """Group maxima on both sides of 2^100, where the codes leave the
    hardware's conversion, up to the largest f32 and down to zero, of and just
    past 448 times a power of two (where the scale steps), with NaNs beside
    them: codes and scales equal the oracle's."""
    say(f"act quant conversion range group={group}")
    rng = np.random.default_rng(group)
    f = np.float32
    tops = [f(2.0**100), np.nextafter(f(2.0**100), f(np.inf)), f(3.4028235e38), f(1e-4), f(9e-5), f(1e-40), f(0.0)]
    for e in (-20, 0, 60, 95):
        t = f(448.0 * 2.0**e)
        tops += [t, np.nextafter(t, f(np.inf)), np.nextafter(t, f(0.0))]
    x = (rng.uniform(-1, 1, (len(tops), 128)) * np.exp2(rng.integers(-18, 1, (len(tops), 128)))).astype(f)
    x *= np.array(tops, f)[:, None]
    x[:, ::group] = np.array(tops, f)[:, None]
    x[::2, 5], x[1::3, 7] = np.nan, -np.nan
    q = torch.empty(x.shape, dtype=torch.uint8, device="cuda")
    s = torch.empty((x.shape[0], 128 // group), dtype=torch.uint8, device="cuda")
    s14.act_quant_e4m3(ctx, dev(x), q, s, group=group)
    want = oracle.requant_e4m3(x, group=group)
    assert np.array_equal(host(s), want[1]) and np.array_equal(host(q), want[0])


@pytest.mark.parametrize("m", [1, 4])
@pytest.mark.parametrize("name", list(SHAPES))
def test_fp8_linear_projection_shapes(ctx, oracle, name, m):
    n, k = SHAPES[name]
    say(f"fp8_linear {name} [{n}, {k}] m={m}")
    w, ws = weight(n, k, seed=list(SHAPES).index(name))
    rng = np.random.default_rng(m)
    xf = rng.standard_normal((m, k)).astype(np.float32)
    q = torch.empty((m, k), dtype=torch.uint8, device="cuda")
    qs = torch.empty((m, k // 128), dtype=torch.uint8, device="cuda")
    s14.act_quant_e4m3(ctx, dev(xf), q, qs, group=128)
    xq, xs = host(q), host(qs)
    want = oracle.fp8_linear(xq, xs, w, ws)
    wd, wsd = dev(w), dev(ws)
    y = torch.empty((m, n), dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, q, qs, wd, wsd, y, mode=s14.EXACT)
    assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32)), "exact"
    y.fill_(np.nan)
    s14.fp8_linear(ctx, q, qs, wd, wsd, y, mode=s14.FAST)
    fast = host(y)
    check_fast(oracle, fast, want, xq, xs, w, ws, name)
    # a second FAST launch (split-K counters reset by the first) gives the same bits
    s14.fp8_linear(ctx, q, qs, wd, wsd, y, mode=s14.FAST)
    assert np.array_equal(host(y).view(np.uint32), fast.view(np.uint32))


def test_fp8_linear_reference_known_answer_shape(ctx, oracle):
    """test_primitives.py:97-109's shapes and scales (x [2, 130], w [129, 130],
    ragged last group and row tile): both modes run the EXACT kernel here."""
    say("fp8_linear reference KAT shape")
    torch.manual_seed(7)
    raw_x = torch.randint(0, 255, (2, 130), dtype=torch.uint8)
    raw_w = torch.randint(0, 255, (129, 130), dtype=torch.uint8)
    raw_x[raw_x == 0x7F] = 0x7E
    raw_w[raw_w == 0x7F] = 0x7E
    sa = np.array([[127, 128], [126, 127]], np.uint8)
    sw = np.array([[127, 128], [126, 127]], np.uint8)
    want = oracle.fp8_linear(raw_x.numpy(), sa, raw_w.numpy(), sw)
    y = torch.empty((2, 129), dtype=torch.float32, device="cuda")
    for mode in (s14.EXACT, s14.FAST):
        s14.fp8_linear(ctx, raw_x.cuda(), dev(sa), raw_w.cuda(), dev(sw), y, mode=mode)
        assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32)), mode


@pytest.mark.parametrize("m", [1, 3])
def test_fp8_linear_f32_scales_bias_bf16(ctx, oracle, m):
    """f32 scales (fp8.py:37-46's float form), a bias and the official bf16
    output rounding, at wkv's shape (one token: the single-token kernels)."""
    say(f"fp8_linear f32 scales + bias + bf16 output, m={m}")
    n, k = 512, 4096
    rng = np.random.default_rng(9)
    w = codes(rng, (n, k))
    ws = rng.uniform(1e-3, 4e-3, (n // 128, k // 128)).astype(np.float32)
    x = codes(rng, (m, k))
    xs = rng.uniform(1e-2, 3e-2, (m, k // 128)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    y = torch.empty((m, n), dtype=torch.float32, device="cuda")
    for rb in (False, True):
        want = oracle.fp8_linear(x, xs, w, ws, bias=b, round_bf16=rb)
        s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, bias=dev(b), round_bf16=rb, mode=s14.EXACT)
        assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32)), rb
    want = oracle.fp8_linear(x, xs, w, ws, bias=b)
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, bias=dev(b), mode=s14.FAST)
    got = host(y) - b
    check_fast(oracle, got, (want - b).astype(np.float64), x, xs, w, ws, "f32 scales")


@pytest.mark.parametrize("m,n,k", [(33, 100, 1536), (1, 4000, 512), (8, 96, 16384), (2, 300, 1024), (8, 4096, 8192),
                                   (3, 130, 16384), (1, 4099, 2048), (4, 1000, 4096)])
def test_fp8_linear_fast_edges(ctx, oracle, m, n, k):
    """Row tiles cut by n, two token blocks (m = 33), 12 groups (chunks per
    wavefront 4 or 12), one group-chunk round (k = 512), k = 16384, two
    tokens, and eight tokens at wo_b's shape; for the few-token GEMV, three
    tokens over k = 16384 (two batches of eight chunks) with rows cut by n,
    a last four-row group cut by n, and four tokens at a short n."""
    say(f"fp8_linear fast edges m={m} n={n} k={k}")
    rng = np.random.default_rng(n)
    w, ws = codes(rng, (n, k)), rng.integers(114, 122, (-(-n // 128), k // 128), dtype=np.uint8)
    x, xs = codes(rng, (m, k)), rng.integers(120, 128, (m, k // 128), dtype=np.uint8)
    want = oracle.fp8_linear(x, xs, w, ws)
    y = torch.empty((m, n), dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.EXACT)
    assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32))
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.FAST)
    check_fast(oracle, host(y), want, x, xs, w, ws, f"m={m} n={n} k={k}")


@pytest.mark.parametrize("k", [1024, 2048, 8192])
def test_fp8_linear_exact_one_token_extreme_scales(ctx, oracle, k):
    """The single-token EXACT kernel at each of its four k (4,096 in the
    shape tests) with UE8M0 codes 0..12 mixed with ordinary ones, so that
    products fall to subnormals or zero (the kernel's separate-multiply
    branch; the top of the code range would overflow to inf and NaN, whose
    payloads the CPU and the GPU form differently), rows cut by n; bit for
    bit."""
    say(f"fp8_linear exact m=1 extreme scales k={k}")
    n = 777
    rng = np.random.default_rng(k)
    w, x = codes(rng, (n, k)), codes(rng, (1, k))
    ends = np.arange(0, 13).astype(np.uint8)
    ws = rng.integers(118, 124, (-(-n // 128), k // 128), dtype=np.uint8)
    xs = rng.integers(118, 124, (1, k // 128), dtype=np.uint8)
    sel = rng.random(ws.shape) < 0.4
    ws[sel] = rng.choice(ends, size=int(sel.sum()))
    sel = rng.random(xs.shape) < 0.4
    xs[sel] = rng.choice(ends, size=int(sel.sum()))
    want = oracle.fp8_linear(x, xs, w, ws)
    y = torch.empty((1, n), dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.EXACT)
    got = host(y)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.count_nonzero(got != want)


@pytest.mark.parametrize("m,n,k", EXACT_MFMA)
def test_fp8_linear_exact_mfma_plans(ctx, oracle, m, n, k):
    """The f32-MFMA EXACT kernel with every plan (4, 8, 16 and 32 tokens per
    workgroup; 4, 8 and 16 wavefronts; m = 65 at k = 2,048 in two launches),
    each also over several rounds of groups with a ragged last one: rows cut
    inside a 64-row tile, tokens cut inside a block, fewer groups than
    wavefronts; then UE8M0 codes that leave the MFMA's window (0..12, so that
    products fall to subnormals or zero), a bias and bf16 outputs; bit for
    bit."""
    say(f"fp8_linear exact mfma m={m} n={n} k={k}")
    rng = np.random.default_rng(m * n + k)
    w, x = codes(rng, (n, k)), codes(rng, (m, k))
    b = rng.standard_normal(n).astype(np.float32)
    for extreme in (False, True):
        ws = rng.integers(114, 122, (-(-n // 128), k // 128), dtype=np.uint8)
        xs = rng.integers(118, 128, (m, k // 128), dtype=np.uint8)
        if extreme:
            for a in (ws, xs):
                sel = rng.random(a.shape) < 0.2
                a[sel] = rng.integers(0, 13, int(sel.sum()), dtype=np.uint8)
        y = torch.full((m, n), np.nan, dtype=torch.float32, device="cuda")
        kw = {"bias": dev(b), "round_bf16": True} if extreme else {}
        s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.EXACT, **kw)
        want = oracle.fp8_linear(x, xs, w, ws, **({"bias": b, "round_bf16": True} if extreme else {}))
        got = host(y)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (extreme, np.count_nonzero(got != want))


@pytest.mark.parametrize("f32", [False, True])
def test_fp8_linear_exact_upper_scales(ctx, oracle, f32):
    """Scale codes at the upper ends of the windows, UE8M0 on both sides: the
    codes' sum on both sides of 356 (f32 MFMA, 5 tokens) and of 364 (one token),
    a code on both sides of 246; e4m3 codes below 2^-1 keep every product and sum
    finite.  The same values as f32 scales on the tiles.  Bit for bit."""
    say(f"fp8_linear exact, upper scale codes, f32={f32}")
    n, k = 200, 1024
    rng = np.random.default_rng(4)
    w, x = rng.integers(0, 0x30, (n, k), dtype=np.uint8), rng.integers(0, 0x30, (5, k), dtype=np.uint8)
    w, x = w | rng.choice(np.array([0, 0x80], np.uint8), w.shape), x | rng.choice(np.array([0, 0x80], np.uint8), x.shape)
    for m, top in ((5, 356), (1, 364)):
        for step in range(-2, 3):
            for cw in (top - 246 - 1, top - 246, 178, 246, 247):
                ws = np.full((2, k // 128), 120, np.uint8)
                xs = np.full((m, k // 128), 120, np.uint8)
                g = int(rng.integers(k // 128))
                ws[:, g], xs[:, g] = cw, top + step - cw
                xs[0, g] -= step > 0  # one token inside beside others outside
                if f32:
                    ws, xs = (np.exp2(a.astype(np.float32) - 127) for a in (ws, xs))
                want = oracle.fp8_linear(x[:m], xs, w, ws)
                assert np.isfinite(want).all()
                y = torch.full((m, n), np.nan, dtype=torch.float32, device="cuda")
                s14.fp8_linear(ctx, dev(x[:m]), dev(xs), dev(w), dev(ws), y, mode=s14.EXACT)
                assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32)), (m, step, cw)


@pytest.mark.parametrize("m,n,k,f32", EXACT_TILE_CHUNKS)
def test_fp8_linear_exact_token_chunks(ctx, oracle, m, n, k, f32):
    """The tiled EXACT kernel keeps every group partial of a launch in the
    context's 32 MiB workspace: at wq_b's shape with f32 scales (8 groups x
    32768 rows x 4 bytes per token) 40 tokens take two launches, 32 tokens then
    8.  And UE8M0 scales where few rows and tokens bring the call to the tiles."""
    say(f"fp8_linear exact tiles: m={m} n={n} k={k} f32={f32}")
    w, ws = weight(n, k, seed=11)
    rng = np.random.default_rng(12)
    x, xs = codes(rng, (m, k)), rng.integers(120, 128, (m, k // 128), dtype=np.uint8)
    if f32:
        ws = rng.uniform(1e-3, 4e-3, ws.shape).astype(np.float32)
        xs = rng.uniform(1e-2, 3e-2, xs.shape).astype(np.float32)
    want = oracle.fp8_linear(x, xs, w, ws)
    y = torch.empty((m, n), dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.EXACT)
    assert np.array_equal(host(y).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("m,n,k,f32", FAST_PROMPT)
def test_fp8_linear_fast_prompt_tiles(ctx, oracle, m, n, k, f32):
    """The prompt-tile FAST kernel: 32- and 64-token workgroups, rows cut by n
    inside a wavefront's and a workgroup's rows (and n not a multiple of 4:
    the scalar stores), tokens cut inside a block, K in one range and in
    several (ragged ones too); f32 scales with a bias, and bf16 outputs."""
    say(f"fp8_linear fast prompt tiles m={m} n={n} k={k} f32={f32}")
    rng = np.random.default_rng(m + n)
    w, x = codes(rng, (n, k)), codes(rng, (m, k))
    if f32:
        ws = rng.uniform(1e-3, 4e-3, (-(-n // 128), k // 128)).astype(np.float32)
        xs = rng.uniform(1e-2, 3e-2, (m, k // 128)).astype(np.float32)
    else:
        ws = rng.integers(114, 122, (-(-n // 128), k // 128), dtype=np.uint8)
        xs = rng.integers(120, 128, (m, k // 128), dtype=np.uint8)
    b = rng.standard_normal(n).astype(np.float32) if f32 else np.zeros(n, np.float32)
    want = oracle.fp8_linear(x, xs, w, ws, bias=b)
    y = torch.full((m, n), np.nan, dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, bias=dev(b), mode=s14.FAST)
    got = host(y)
    check_fast(oracle, got - b, (want - b).astype(np.float64), x, xs, w, ws, f"m={m} n={n} k={k}")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, bias=dev(b), round_bf16=True, mode=s14.FAST)
    assert np.array_equal(host(y), torch.from_numpy(got).bfloat16().float().numpy())


@pytest.mark.parametrize("m,n,k,f32", FAST_LAUNCHES)
def test_fp8_linear_fast_token_blocks_in_several_launches(ctx, oracle, m, n, k, f32):
    """k_linear_fast over a long k: 256 K splits a token block, so the 32 MiB
    workspace holds the partials of 32 blocks and more tokens take two launches
    (18 blocks of 35 and 17 of 34 each): x, scale and y offsets and the counters
    between them.  Every token's row matches the oracle."""
    say(f"fp8_linear fast m={m} n={n} k={k} f32={f32} (several launches)")
    rng = np.random.default_rng(m)
    w, x = codes(rng, (n, k)), codes(rng, (m, k))
    if f32:
        ws = rng.uniform(1e-3, 4e-3, (1, k // 128)).astype(np.float32)
        xs = rng.uniform(1e-2, 3e-2, (m, k // 128)).astype(np.float32)
    else:
        ws = rng.integers(114, 122, (1, k // 128), dtype=np.uint8)
        xs = rng.integers(120, 128, (m, k // 128), dtype=np.uint8)
    want = oracle.fp8_linear(x, xs, w, ws)
    l1 = oracle.fp8_linear(x & 0x7F, xs, w & 0x7F, ws)  # the sum of |products|, to f32 rounding
    y = torch.full((m, n), np.nan, dtype=torch.float32, device="cuda")
    s14.fp8_linear(ctx, dev(x), dev(xs), dev(w), dev(ws), y, mode=s14.FAST)
    check_fast(oracle, host(y), want, x, xs, w, ws, f"m={m} n={n} k={k}", l1=l1)
