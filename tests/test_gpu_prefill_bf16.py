"""BF16 prefill projections over Q4_K 0x020D (cuda/prefill.cu:510-779)
through the C-ABI: projections against the oracle (float64 sums of the rebuilt
BF16 operands), epilogues, token-count invariance, the paired SwiGLU, the BF16
RMS producer (bit-exact) and the whole MLP stage by stage."""
import numpy as np
import pytest

import oracle
from _fix import normal, random_q4k

pytestmark = pytest.mark.gpu


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _weight(ops, wl):
    co, mo = wl.physical(oracle.LAYOUT_Q4K_SEQ)
    return ops.PrefillWeight.from_bytes(co, mo, oracle.LAYOUT_Q4K_SEQ, wl.n, wl.k)


def _ref(wl, xb, rows=None):
    """float64 reference [tokens][n or len(rows)] from BF16 bits xb [tokens][k]."""
    sub = wl if rows is None else oracle.Q4K(wl.codes[rows], wl.meta[rows], len(rows), wl.k)
    return np.stack([oracle.q4k_bf16_gemv(sub, xb[t]) for t in range(xb.shape[0])])


def _check(y, ref, label):
    ok, ma, mr = oracle.parity_ok(y, ref)
    ok_ref = np.all(np.abs(y - ref) <= 1e-3 + 1e-4 * np.abs(ref))
    print(f"{label}: max_abs/rms={ma:.3g} mean_rel={mr:.3g}", flush=True)
    assert ok and ok_ref, label


@pytest.mark.parametrize("n,k,m", [(136, 256, 1), (136, 512, 17), (1000, 2560, 130),
                                   (5120, 5120, 64)])
def test_project_vs_oracle(torch_gpu, n, k, m):
    torch = torch_gpu
    import qw38_amd.ops as ops
    wl = random_q4k(n, k, n + k + m)
    w = _weight(ops, wl)
    xb = oracle.fp32_to_bf16(normal((m, k), m + 1))
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.prefill_project(w, _dev(torch, xb.view(np.int16)), m, y, ops.DECODE_STORE_FP32)
    got = y.cpu().numpy()
    rows = None if n * k <= 2_600_000 else np.sort(
        np.random.Generator(np.random.PCG64(n)).choice(n, 256, replace=False))
    ref = _ref(wl, xb, rows)
    _check(got if rows is None else got[:, rows], ref, f"prefill n={n} k={k} m={m}")


def test_epilogues_and_token_invariance(torch_gpu):
    torch = torch_gpu
    import qw38_amd.ops as ops
    n, k, m = 264, 1024, 70
    wl = random_q4k(n, k, 9)
    w = _weight(ops, wl)
    xb = oracle.fp32_to_bf16(normal((m, k), 10))
    x = _dev(torch, xb.view(np.int16))
    f32 = torch.empty(m, n, device="cuda")
    ops.prefill_project(w, x, m, f32, ops.DECODE_STORE_FP32)
    base = f32.cpu().numpy()
    b16 = torch.empty(m, n, dtype=torch.int16, device="cuda")
    ops.prefill_project(w, x, m, b16, ops.DECODE_STORE_BF16)
    assert np.array_equal(b16.cpu().numpy().view(np.uint16), oracle.fp32_to_bf16(base))
    res = normal((m, n), 11)
    out = torch.empty(m, n, device="cuda")
    ops.prefill_project(w, x, m, out, ops.DECODE_RESIDUAL_ADD_FP32, residual=_dev(torch, res))
    assert np.array_equal(out.cpu().numpy(), (res + base).astype(np.float32))
    # each token's row is independent of how many tokens share the launch
    one = torch.empty(1, n, device="cuda")
    ops.prefill_project(w, x[37:38].contiguous(), 1, one, ops.DECODE_STORE_FP32)
    assert np.array_equal(one.cpu().numpy()[0], base[37])
    # unaligned (2-byte) input span: same results through the narrow-load path
    xu = torch.empty(m * k + 1, dtype=torch.int16, device="cuda")
    xu[1:] = x.flatten()
    ops.prefill_project(w, xu[1:], m, f32, ops.DECODE_STORE_FP32)
    assert np.array_equal(f32.cpu().numpy(), base)


def test_tail_split_bitwise(torch_gpu):
    """M=512 over 34816 rows makes 272 tiles of 256 x 256: one round of them
    and a tail on ring tiles (rows 32768 on at 256 CUs). Every row, head or tail,
    equals a 64-token call's result for the same token bitwise, and
    sampled rows match the oracle. The BF16 and residual epilogues and
    2-byte-aligned activations give the same values."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    n, k, m = 34816, 256, 512
    wl = random_q4k(n, k, 77)
    w = _weight(ops, wl)
    xb = oracle.fp32_to_bf16(normal((m, k), 78))
    x = _dev(torch, xb.view(np.int16))
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.prefill_project(w, x, m, y, ops.DECODE_STORE_FP32)
    got = y.cpu().numpy()
    small = torch.full((64, n), float("nan"), device="cuda")
    ops.prefill_project(w, x[448:].contiguous(), 64, small, ops.DECODE_STORE_FP32)
    assert np.array_equal(got[448:], small.cpu().numpy())
    rows = np.concatenate([np.arange(0, 64), np.arange(32700, 32830), np.arange(n - 64, n)])
    _check(got[::16][:, rows], _ref(wl, xb[::16], rows), "prefill split n=34816 m=512")
    # the other epilogues, and 2-byte-aligned activations
    b16 = torch.empty(m, n, dtype=torch.int16, device="cuda")
    ops.prefill_project(w, x, m, b16, ops.DECODE_STORE_BF16)
    assert np.array_equal(b16.cpu().numpy().view(np.uint16), oracle.fp32_to_bf16(got))
    res = normal((m, n), 79)
    out = torch.empty(m, n, device="cuda")
    ops.prefill_project(w, x, m, out, ops.DECODE_RESIDUAL_ADD_FP32, residual=_dev(torch, res))
    assert np.array_equal(out.cpu().numpy(), (res + got).astype(np.float32))
    xu = torch.empty(m * k + 1, dtype=torch.int16, device="cuda")
    xu[1:] = x.flatten()
    ops.prefill_project(w, xu[1:], m, y, ops.DECODE_STORE_FP32)
    assert np.array_equal(y.cpu().numpy(), got)


def test_paired_swiglu(torch_gpu):
    torch = torch_gpu
    import qw38_amd.ops as ops
    n, k, m = 520, 1536, 33
    gl, ul = random_q4k(n, k, 21), random_q4k(n, k, 22)
    g, u = _weight(ops, gl), _weight(ops, ul)
    x = _dev(torch, oracle.fp32_to_bf16(normal((m, k), 23)).view(np.int16))
    ga, ua = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda")
    ops.prefill_project(g, x, m, ga, ops.DECODE_STORE_FP32)
    ops.prefill_project(u, x, m, ua, ops.DECODE_STORE_FP32)
    sw = torch.empty(m, n, dtype=torch.int16, device="cuda")
    ops.prefill_paired_swiglu(g, u, x, sw, m)
    gd, ud = ga.cpu().numpy().astype(np.float64), ua.cpu().numpy().astype(np.float64)
    ref = oracle.bf16_to_fp32(oracle.fp32_to_bf16((gd / (1 + np.exp(-gd)) * ud).astype(np.float32)))
    got = oracle.bf16_to_fp32(sw.cpu().numpy().view(np.uint16))
    ulp = np.abs(ref.view(np.int32).astype(np.int64) - got.view(np.int32).astype(np.int64))
    assert np.all(ulp <= 65536)


def test_paired_big_tile_bitwise(torch_gpu):
    """17408 features at M=512 run the paired 256 x 256 tile (128 gate + 128
    up rows per block) over whole rounds and a 128 x 64 paired tail: every
    feature equals the 128 x 64 paired kernel's output for the same token
    bitwise, and stays within 1 BF16 ulp of SiLU(g) * u from the separate
    projections."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    n, k, m = 17408, 256, 512
    gl, ul = random_q4k(n, k, 31), random_q4k(n, k, 32)
    g, u = _weight(ops, gl), _weight(ops, ul)
    x = _dev(torch, oracle.fp32_to_bf16(normal((m, k), 33)).view(np.int16))
    sw = torch.full((m, n), -1, dtype=torch.int16, device="cuda")
    ops.prefill_paired_swiglu(g, u, x, sw, m)
    small = torch.full((64, n), -1, dtype=torch.int16, device="cuda")
    ops.prefill_paired_swiglu(g, u, x[448:].contiguous(), small, 64)
    got = sw.cpu().numpy()
    assert np.array_equal(got[448:], small.cpu().numpy())
    ga, ua = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda")
    ops.prefill_project(g, x, m, ga, ops.DECODE_STORE_FP32)
    ops.prefill_project(u, x, m, ua, ops.DECODE_STORE_FP32)
    gd, ud = ga.cpu().numpy().astype(np.float64), ua.cpu().numpy().astype(np.float64)
    ref = oracle.bf16_to_fp32(oracle.fp32_to_bf16((gd / (1 + np.exp(-gd)) * ud).astype(np.float32)))
    val = oracle.bf16_to_fp32(got.view(np.uint16))
    ulp = np.abs(ref.view(np.int32).astype(np.int64) - val.view(np.int32).astype(np.int64))
    assert np.all(ulp <= 65536)


def test_hidden_rms_bf16_bit_exact(torch_gpu):
    torch = torch_gpu
    import qw38_amd.ops as ops
    m = 5
    res = (normal((m, 5120), 31) * 4).astype(np.float32)
    res[2] = 0.0
    gamma = oracle.fp32_to_bf16(normal(5120, 32, 0.1))
    out = torch.empty(m, 5120, dtype=torch.int16, device="cuda")
    ops.hidden_rms_bf16(_dev(torch, res), _dev(torch, gamma.view(np.int16)), 1e-6, m, out)
    _, bf = oracle.rms_q8(res, gamma, 1e-6)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), bf)


def test_prefill_mlp(torch_gpu):
    torch = torch_gpu
    import qw38_amd.ops as ops
    m = 40
    gl, ul, dl = random_q4k(17408, 5120, 41), random_q4k(17408, 5120, 42), random_q4k(5120, 17408, 43)
    g, u, d = _weight(ops, gl), _weight(ops, ul), _weight(ops, dl)
    gamma = oracle.fp32_to_bf16(normal(5120, 44, 0.1))
    h = normal((m, 5120), 45)
    dh, dg = _dev(torch, h), _dev(torch, gamma.view(np.int16))
    ws = torch.zeros(ops.prefill_mlp_workspace_bytes(m), dtype=torch.uint8, device="cuda")
    out = torch.full((m, 5120), float("nan"), device="cuda")
    ops.prefill_mlp(g, u, d, dh, dg, 1e-6, out, m, ws)
    b = ws.cpu().numpy()
    norm = b[:m * 5120 * 2].view(np.uint16).reshape(m, 5120)
    sw = b[m * 5120 * 2:m * 5120 * 2 + m * 17408 * 2].view(np.uint16).reshape(m, 17408)
    _, bf = oracle.rms_q8(h, gamma, 1e-6)
    assert np.array_equal(norm, bf), "RMS -> BF16 stage"
    sw2 = torch.empty(m, 17408, dtype=torch.int16, device="cuda")
    ops.prefill_paired_swiglu(g, u, _dev(torch, norm.view(np.int16)), sw2, m)
    assert np.array_equal(sw, sw2.cpu().numpy().view(np.uint16)), "SwiGLU stage"
    rows = np.sort(np.random.Generator(np.random.PCG64(46)).choice(5120, 128, replace=False))
    ref = _ref(dl, sw, rows)
    _check(out.cpu().numpy()[:, rows] - h[:, rows], ref, "prefill mlp down")


def _rows_agree(torch, run, n, ms, label):
    """Runs every token count and compares each token's row, bit for bit, with
    the largest call's; a guard row after the last token stays untouched."""
    full = None
    for m in ms:
        print(f"{label} n={n} m={m}", flush=True)
        y = run(m)
        assert torch.all(y[m] == 7), "token past the last is not written"
        full = y if full is None else full
        assert torch.equal(y[:m].view(torch.int32 if y.dtype == torch.float32 else torch.int16),
                           full[:m].view(torch.int32 if y.dtype == torch.float32 else torch.int16)), f"{label} m={m}"
    return full


@pytest.mark.parametrize("n,ms", [(1030, (1000, 512, 300, 64, 1)), (8200, (1000, 512, 400)), (16384, (512, 17))],
                         ids=lambda v: str(v))
def test_tiles_agree(torch_gpu, n, ms):
    """Every tile of the projection chains the same MFMAs per output: a
    token's row is bitwise the same in a call of any size (each size here
    takes another tile, with partial row and token blocks and, at K = 768, fewer
    super-blocks than some rings hold), and sampled rows meet the oracle."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    k = 768
    wl = random_q4k(n, k, n)
    w = _weight(ops, wl)
    xb = oracle.fp32_to_bf16(normal((ms[0], k), n + 1))
    x = _dev(torch, xb.view(np.int16))

    def run(m):
        y = torch.full((m + 1, n), 7.0, device="cuda")
        ops.prefill_project(w, x[:m].contiguous(), m, y, ops.DECODE_STORE_FP32)
        return y

    y = _rows_agree(torch, run, n, ms, "prefill tiles").cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(0, n, 97), np.arange(n - 9, n)]))
    toks = np.array([0, 15, ms[0] - 1])
    _check(y[toks][:, rows], _ref(wl, xb[toks], rows), f"prefill tiles n={n}")


@pytest.mark.parametrize("n,ms", [(2058, (1000, 700, 128, 64, 1)), (8200, (256, 32)), (8192, (512,))],
                         ids=lambda v: str(v))
def test_paired_tiles_agree(torch_gpu, n, ms):
    """The same for the gate/up tiles, whose values are within 1 BF16 ulp of
    SiLU(g) * u from the separate projections."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    k = 768
    g, u = (_weight(ops, random_q4k(n, k, n + i)) for i in (1, 2))
    x = _dev(torch, oracle.fp32_to_bf16(normal((ms[0], k), n + 3)).view(np.int16))

    def run(m):
        y = torch.full((m + 1, n), 7, dtype=torch.int16, device="cuda")
        ops.prefill_paired_swiglu(g, u, x[:m].contiguous(), y, m)
        return y

    got = _rows_agree(torch, run, n, ms, "paired tiles")[:ms[0]].view(torch.bfloat16).double()
    ga, ua = torch.empty(ms[0], n, device="cuda"), torch.empty(ms[0], n, device="cuda")
    ops.prefill_project(g, x, ms[0], ga, ops.DECODE_STORE_FP32)
    ops.prefill_project(u, x, ms[0], ua, ops.DECODE_STORE_FP32)
    want = ga.double() * torch.sigmoid(ga.double()) * ua.double()
    # BF16 rounding is within 2^-8 relative; one more ulp for the FP32 SiLU's ties
    assert torch.all((got - want).abs() <= want.abs() * 2.0**-7 + 1e-30)


@pytest.mark.parametrize("n,k,m", [(8200, 512, 2040), (16384, 256, 1024)])
def test_big_tile_rounds(torch_gpu, n, k, m):
    """Whole rounds of 256 x 256 tiles, with ring tiles for the rows behind them
    and without: every epilogue gives the bits of 16-token calls."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    g = torch.Generator(device="cuda").manual_seed(n + m)
    codes = torch.randint(0, 256, (n * k // 2,), generator=g, device="cuda", dtype=torch.uint8)
    meta = torch.randint(0, 256, (n * k // 256, 16), generator=g, device="cuda", dtype=torch.uint8)
    meta[:, 1] = meta[:, 3] = 0x24  # d and dmin in [2^-6, 2^-5)
    w = ops.PrefillWeight(codes, meta.view(-1), oracle.LAYOUT_Q4K_SEQ, ops.QUANTIZER_Q4K, n, k, n, k)
    x = torch.randn(m, k, generator=g, device="cuda").bfloat16().view(torch.int16)
    res = torch.randn(m, n, generator=g, device="cuda")
    y, r = torch.full((m, n), float("nan"), device="cuda"), torch.full((m, n), float("nan"), device="cuda")
    h = torch.zeros(m, n, dtype=torch.int16, device="cuda")
    ops.prefill_project(w, x, m, y, ops.DECODE_STORE_FP32)
    ops.prefill_project(w, x, m, r, ops.DECODE_RESIDUAL_ADD_FP32, residual=res)
    ops.prefill_project(w, x, m, h, ops.DECODE_STORE_BF16)
    assert torch.isfinite(y).all()
    assert torch.equal(r, res + y) and torch.equal(h.view(torch.bfloat16), y.bfloat16())
    for t0 in (0, 240, m // 2, m - 16):
        y16 = torch.empty(16, n, device="cuda")
        ops.prefill_project(w, x[t0:t0 + 16].contiguous(), 16, y16, ops.DECODE_STORE_FP32)
        assert torch.equal(y[t0:t0 + 16], y16), t0


def _plan(paired, aligned, n, m):
    """What the dispatch takes: "all" / "whole" (256-row tiles on all rows, or on
    the rows of whole rounds) and the tile of the rows behind them."""
    import ctypes
    from qw38_amd._lib import lib
    p = (ctypes.c_uint32 * 3)()
    assert lib().qw38_gemm_plan(3 + paired + 2 * (not aligned), n, m, 256, p) == 0
    if p[0] * (128 if paired else 256) >= n:
        return {"all"}, p[2]
    return ({"whole"} if p[0] else set()) | {p[1]}, p[2]


def _weight_bytes(torch, g, n, k):
    """Random codes, metadata with d and dmin in [2^-6, 2^-5)."""
    pn = (n + 7) // 8 * 8
    codes = torch.randint(0, 256, (pn * k // 2,), generator=g, device="cuda", dtype=torch.uint8)
    meta = torch.randint(0, 256, (pn * k // 256, 16), generator=g, device="cuda", dtype=torch.uint8)
    meta[:, 1] = meta[:, 3] = 0x24
    return codes, meta.view(-1)


def _weight_of(ops, codes, meta, n, k):
    return ops.PrefillWeight(codes, meta, oracle.LAYOUT_Q4K_SEQ, ops.QUANTIZER_Q4K, n, k, (n + 7) // 8 * 8, k)


# Ragged sizes that take each plan on 256 CUs, with spans that are 16-byte aligned.
PLANS = {False: [(2568, 3000), (1506, 2690), (1290, 2600), (16632, 130), (1030, 1000), (1030, 700), (1030, 300),
                 (264, 521), (5128, 2570), (4104, 4000)],
         True: [(6706, 450), (4104, 700), (1030, 1000), (1030, 500), (264, 1030), (1030, 1), (2568, 3000),
                (2568, 4090)]}


@pytest.mark.parametrize("paired", [False, True])
def test_every_plan(torch_gpu, paired):
    """Every ring tile, the 256-row tiles on all rows (a partly filled last round,
    a ragged last block) and on whole rounds with ring tiles behind: each token's
    rows have the bits of a 16-token call, in every epilogue."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    k, seen = 512, set()
    for n, m in PLANS[paired]:
        taken, tiles = _plan(paired, True, n, m)
        seen |= taken
        print(f"prefill plan paired={paired} n={n} m={m}: {taken}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(n + m)
        w = [_weight_of(ops, *_weight_bytes(torch, g, n, k), n, k) for _ in range(2)]
        x = torch.randn(max(m, 16), k, generator=g, device="cuda").bfloat16().view(torch.int16)

        def call(xs, epilogue=ops.DECODE_STORE_FP32, residual=None):
            t = xs.shape[0]
            half = paired or epilogue == ops.DECODE_STORE_BF16
            y = torch.full((t + 1, n), 7, device="cuda", dtype=torch.int16 if half else torch.float32)
            if paired:
                ops.prefill_paired_swiglu(*w, xs, y, t)
            else:
                ops.prefill_project(w[0], xs, t, y, epilogue, residual)
            assert torch.all(y[t] == 7), "token past the last is not written"
            return y[:t]

        y = call(x[:m].contiguous())
        for t0 in {0, max(0, m // 2 - 8), max(0, m - 16)}:
            assert torch.equal(y[t0:t0 + 16], call(x[t0:t0 + 16].contiguous())[:m]), (n, m, t0)
        if not paired:
            assert torch.isfinite(y).all()
            res = torch.randn(m, n, generator=g, device="cuda")
            assert torch.equal(call(x[:m].contiguous(), ops.DECODE_RESIDUAL_ADD_FP32, res), res + y)
            assert torch.equal(call(x[:m].contiguous(), ops.DECODE_STORE_BF16).view(torch.bfloat16), y.bfloat16())
    assert seen == set(range(tiles)) | {"all", "whole"}


# The same for spans that are not.
PLANS_UNALIGNED = {False: [(6458, 1167)] + PLANS[False][1:], True: [(3234, 1167)] + PLANS[True][1:]}


@pytest.mark.parametrize("paired", [False, True])
def test_every_plan_unaligned(torch_gpu, paired):
    """Spans of 2-byte alignment (the entries' minimum) take the same range of
    tiles, and give the bits of aligned ones: the input, the codes and the metadata
    shifted in turn."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    k, seen = 512, set()

    def shifted(t):
        by = 2 // t.element_size()
        s = torch.empty(t.numel() + by, dtype=t.dtype, device="cuda")[by:]
        s.copy_(t.flatten())
        assert s.data_ptr() % 16 == 2
        return s.view(t.shape)

    for n, m in PLANS_UNALIGNED[paired]:
        taken, tiles = _plan(paired, False, n, m)
        seen |= taken
        print(f"prefill unaligned plan paired={paired} n={n} m={m}: {taken}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(n + m)
        raw = [_weight_bytes(torch, g, n, k) for _ in range(2)]
        x = torch.randn(m, k, generator=g, device="cuda").bfloat16().view(torch.int16)

        def call(weights, xs):
            w = [_weight_of(ops, c, s, n, k) for c, s in weights]
            y = torch.full((m + 1, n), 7, device="cuda", dtype=torch.int16 if paired else torch.float32)
            if paired:
                ops.prefill_paired_swiglu(*w, xs, y, m)
            else:
                ops.prefill_project(w[0], xs, m, y)
            assert torch.all(y[m] == 7), "token past the last is not written"
            return y

        y = call(raw, x)
        for weights, xs in ((raw, shifted(x)), ([(shifted(c), s) for c, s in raw], x),
                            ([(c, shifted(s)) for c, s in raw], x)):
            assert torch.equal(call(weights, xs), y), (n, m)
    assert seen == set(range(tiles)) | {"all", "whole"}


@pytest.mark.parametrize("n,m", [(4102, 1000), (8708, 521)])
def test_single_super_block(torch_gpu, n, m):
    """K of one super-block, where the 256 x 128 big tile stands in for the 256 x 112
    ring tile, with stores of rows one by one (n % 4) and as vectors: each token's
    rows have the bits of a 16-token call, in every epilogue."""
    torch = torch_gpu
    import qw38_amd.ops as ops
    k = 256
    assert _plan(False, True, n, m)[0] == {1}
    g = torch.Generator(device="cuda").manual_seed(n)
    w = _weight_of(ops, *_weight_bytes(torch, g, n, k), n, k)
    x = torch.randn(m, k, generator=g, device="cuda").bfloat16().view(torch.int16)
    y = torch.full((m + 1, n), 7.0, device="cuda")
    ops.prefill_project(w, x, m, y)
    assert torch.all(y[m] == 7) and torch.isfinite(y).all()
    y = y[:m]
    for t0 in (0, m // 2, m - 16):
        small = torch.empty(16, n, device="cuda")
        ops.prefill_project(w, x[t0:t0 + 16].contiguous(), 16, small)
        assert torch.equal(y[t0:t0 + 16], small), t0
    res = torch.randn(m, n, generator=g, device="cuda")
    out = torch.empty(m, n, device="cuda")
    ops.prefill_project(w, x, m, out, ops.DECODE_RESIDUAL_ADD_FP32, res)
    assert torch.equal(out, res + y)
    half = torch.empty(m, n, dtype=torch.int16, device="cuda")
    ops.prefill_project(w, x, m, half, ops.DECODE_STORE_BF16)
    assert torch.equal(half.view(torch.bfloat16), y.bfloat16())
