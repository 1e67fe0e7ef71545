"""The prefill kernel of the formats whose scaled weights are exact in f16 (Q4_K; oxq_gemm_prefill.hip): many token
rows x Q4_K weights on the f16 matrix cores with the 6-bit sub-block scale inside the weight operand
(reference: gemm = m fused matvecs, crates/oxillama-quant/src/reference/q4_k.rs:186-201, 218-333).

Bars: the matrix core's result per (token, row, 32-weight sub-block) is sc * I exactly, compared == with the
scale decoded here from the raw block bytes (decode_scales_mins, q4_k.rs:27-49) times the oracle's integer group
sum; fp32 within 1e-5 * |y|_inf of the oracle's fused matvec per token row (tolerance of the path; the kernel
applies d and dmin once per super-block, the reference once per sub-block)."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from oxillama_amd import capi, linear, synth

pytestmark = pytest.mark.gpu
FP32_REL_TOL = 1e-5


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def q4k_sub_block_scales(w, n, k):
    """sc[row][sub-block] of Q4_K rows (decode_scales_mins, reference/q4_k.rs:27-49), from the raw bytes."""
    blocks = w.reshape(n, k // 256, 144)
    s = blocks[:, :, 4:16].astype(np.int32)
    sc = np.empty((n, k // 256, 8), np.int32)
    for j in range(4):
        sc[:, :, j] = s[:, :, j] & 63
        sc[:, :, j + 4] = (s[:, :, j + 8] & 15) | ((s[:, :, j] >> 6) << 4)
    return sc.reshape(n, k // 32)


def last_launch():
    import ctypes
    buf = ctypes.create_string_buffer(256)
    capi.load().oxq_last_launch(buf, 256)
    return buf.value.decode()


def oracle_rows(ref, t, w, acts, n, k, rows):
    arb = k // 32 * 34
    return np.stack([ref.matvec_q8_fused_mt(t, w, acts[r * arb:(r + 1) * arb], n, k, 16) for r in rows])


@pytest.mark.parametrize("shape", [(1, 32, 256), (33, 100, 1024), (96, 128, 256), (128, 160, 512), (200, 257, 1024),
                                   (130, 129, 2048), (384, 520, 4096)], ids=lambda s: "x".join(map(str, s)))
def test_prefill_f16_kernel(hip, ref, tuning, shape):
    m, n, k = shape
    t = O.Q4_K
    say("prefill f16", shape)
    tuning("gemm_variant", 300)  # this kernel for any number of token rows
    tuning("gemm_tile_min_rows", 1)  # (a handful of rows would otherwise go to the GEMV launches)
    w = synth.weights(t, 900 + m, n, k)
    x = synth.normal_f32(901 + n, m * k)
    x[:k] *= 300.0  # a token with large activations: its block sums' products need all three bf16 pieces
    acts = ref.quantize_q8_0(x)
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    dy = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw, da, dy, m, n, k, accumulate=False, workspace=ws)
    torch.cuda.synchronize()
    assert "gemm_prefill_q4k" in last_launch(), last_launch()
    y = dy.cpu().numpy()
    y_ref = oracle_rows(ref, t, w, acts, n, k, range(m))
    for r in range(m):  # per token row: the bar of the batch-1 matvec
        err, scale = np.abs(y[r] - y_ref[r]).max(), np.abs(y_ref[r]).max()
        assert err <= FP32_REL_TOL * scale, f"token {r}: max err {err:.3e} vs |y|inf {scale:.3e}"
    # accumulate adds the same values to what is there
    dy2 = dy.clone()
    kern.gemm_q8_dev(dw, da, dy2, m, n, k, accumulate=True, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(dy2, dy + dy)
    # the matrix core's results: sc * I exactly, and the dump launch gives the product launch's bits
    dsum = torch.empty((m, n, k // 32), dtype=torch.int32, device="cuda")
    dy3 = torch.empty_like(dy)
    kern.gemm_scaled_sums_dev(dw, da, dy3, dsum, m, n, k, ws)
    torch.cuda.synchronize()
    sc = q4k_sub_block_scales(w, n, k)
    arb = k // 32 * 34
    got = dsum.cpu().numpy()
    for r in range(m):
        want = sc * ref.block_sums(t, w, acts[r * arb:(r + 1) * arb], n, k)
        assert np.array_equal(got[r], want), f"token {r}"
    assert torch.equal(dy3, dy)


def test_prefill_f16_kernel_is_the_default_where_it_fills_the_chip(hip, ref):
    """Without any knob: a Q4_K matmul whose 128-token x 256-row work groups fill 7/8 of the compute units takes this
    kernel (also with 96 of a tile's 128 token rows in use); one that fills 40 % of them, one with 64 token rows (half
    of every work group's token tile empty), and any Q6_K matmul, stay on the int8 tile kernel."""
    cus = hip.device_info()["compute_units"]
    k = 256
    for t, m, n, expect in ((O.Q4_K, 128, 256 * (cus * 7 // 8), True), (O.Q4_K, 128, 256 * (cus * 2 // 5), False),
                            (O.Q4_K, 96, 256 * (cus * 7 // 8), True), (O.Q4_K, 64, 256 * (cus * 7 // 8), False),
                            (O.Q6_K, 128, 256 * (cus * 7 // 8), False)):
        say("default kernel", O.NAMES[t], m, n, k)
        w = synth.weights(t, 5, n, k)
        acts = ref.quantize_q8_0(synth.normal_f32(6, m * k))
        kern = hip.HipKernel(t)
        ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
        dy = torch.empty((m, n), dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda(), dy, m, n, k, accumulate=False,
                         workspace=ws)
        torch.cuda.synchronize()
        assert ("gemm_prefill_q4k" in last_launch()) == expect, (O.NAMES[t], m, n, last_launch())
        rows = [0, 1, 63, m - 1]
        y_ref = oracle_rows(ref, t, w, acts, n, k, rows)
        assert np.abs(dy.cpu().numpy()[rows] - y_ref).max() <= FP32_REL_TOL * np.abs(y_ref).max()


@pytest.mark.parametrize("shape", [(1, 32, 512), (33, 100, 1024), (65, 127, 768), (128, 257, 512), (129, 130, 2304), (200, 300, 4096)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K], ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("variant", [301, 302])
def test_f16_kernel_on_raw_rows(hip, ref, tuning, variant, t, shape):
    """The f16 kernel that takes the Q8_0 rows as they are, both shapes: tiles' edges in tokens and rows, an odd number of
    super-blocks (the halves of k differ by one), two of them.  Weights with every scale and quant value the format has
    (random block bytes); fp32 within the bar of the batch-1 matvec per token row."""
    m, n, k = shape
    say("f16 raw rows", variant, O.NAMES[t], shape)
    tuning("gemm_variant", variant)
    tuning("gemm_tile_min_rows", 1)
    w = O.random_blocks(t, 40 + m, n, k)
    x = synth.normal_f32(41 + n, m * k)
    x[:k] *= 300.0
    acts = ref.quantize_q8_0(x)
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    dy = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw, da, dy, m, n, k, accumulate=False, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_f16_kernel"), last_launch()
    y = dy.cpu().numpy()
    assert np.all(y[m] == 7.0)
    y_ref = oracle_rows(ref, t, w, acts, n, k, range(m))
    for r in range(m):
        err, scale = np.abs(y[r] - y_ref[r]).max(), np.abs(y_ref[r]).max()
        assert err <= FP32_REL_TOL * scale, f"token {r}: max err {err:.3e} vs |y|inf {scale:.3e}"
    dy2 = dy.clone()
    kern.gemm_q8_dev(dw, da, dy2, m, n, k, accumulate=True, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(dy2[:m], dy[:m] + dy[:m])


@pytest.mark.parametrize("k", [256, 512, 768])
@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K], ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("variant", [301, 302])
def test_f16_kernel_is_exact_in_whole_numbers(hip, ref, tuning, variant, t, k):
    """Weights that are whole numbers (d = dmin = 1, every scale and quant value of the format, the largest among them)
    against tokens with one sub-block of whole numbers over 8: a result is at most 2^24 eighths, so that every step of the
    kernel is exact if its operands are (Q6_K's two pieces, P's three), and == is the bar.  k = 256: the small shape's
    second half of k has nothing to do."""
    m, n = 37, 96
    say("f16 exact", variant, O.NAMES[t], k)
    tuning("gemm_variant", variant)
    tuning("gemm_tile_min_rows", 1)
    bb = O.BLOCK[t][1]
    w = O.random_blocks(t, 81, n, k).reshape(n, k // 256, bb)
    for off in O.F16_FIELDS[t]:
        w[:, :, off:off + 2] = [0x00, 0x3C]  # 1.0
    if t == O.Q6_K:  # rows of scale -128 and -127 against the lowest and the highest quant value
        w[0, :, :192], w[0, :, 192:208] = 0, 0x80
        w[1, :, :192], w[1, :, 192:208] = 0, 0x81
        w[2, :, :192], w[2, :, 192:208] = 0xFF, 0x80
    else:  # the largest of everything
        w[0, :, 4:] = 0xFF
    rng = np.random.default_rng(82)
    a = np.zeros((m, k // 32, 32), np.int64)
    for r in range(m):
        v = rng.integers(-127, 128, 32)
        if r < 6:
            v[:] = (-128, 127)[r % 2]
        a[r, (5 * r) % (k // 32)] = v
    acts = np.zeros((m, k // 32, 34), np.uint8)
    acts[:, :, :2] = [0x00, 0x30]  # 1 / 8
    acts[:, :, 2:] = a.astype(np.int8).view(np.uint8)
    want = a.reshape(m, k) @ ref.dequant_rows(t, w.reshape(-1), n, k).reshape(n, k).astype(np.int64).T
    assert np.abs(want).max() <= 1 << 24
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    dy = torch.empty((m, n), dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(torch.from_numpy(w.reshape(-1)).cuda(), torch.from_numpy(acts.reshape(-1)).cuda(), dy, m, n, k,
                     accumulate=False, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_f16_kernel"), last_launch()
    assert np.array_equal(dy.cpu().numpy().astype(np.float64) * 8, want)


@pytest.mark.parametrize("n", [160, 161])
@pytest.mark.parametrize("t", [O.Q4_K, O.Q6_K], ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("variant", [301, 302])
def test_f16_kernel_adds_the_bias(hip, ref, tuning, variant, t, n):
    """The bias is one fp32 addition behind the sum: bit for bit result + bias, in the stores of four rows and of one (rows
    not a multiple of four, an output or a bias off the 16-byte grid)."""
    m, k = 70, 512
    say("f16 bias", variant, O.NAMES[t], n)
    tuning("gemm_variant", variant)
    tuning("gemm_tile_min_rows", 1)
    kern = hip.HipKernel(t)
    dw = torch.from_numpy(O.random_blocks(t, 91, n, k)).cuda()
    da = torch.from_numpy(ref.quantize_q8_0(synth.normal_f32(92, m * k))).cuda()
    bias = torch.from_numpy(synth.normal_f32(93, n + 1)).cuda()
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    y = torch.empty((m, n), dtype=torch.float32, device="cuda")
    linear.linear_forward_batch_dev(t, dw, da, y, m, n, k, workspace=ws)
    assert last_launch().startswith("gemm_f16_kernel"), last_launch()
    for o_off, b_off in ((0, 0), (1, 0), (0, 1)):
        buf = torch.full((m * n + 2,), 7.0, dtype=torch.float32, device="cuda")
        out, b = buf[o_off:o_off + m * n], bias[b_off:b_off + n]
        linear.linear_forward_batch_dev(t, dw, da, out, m, n, k, d_bias=b, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(out.view(m, n), y + b)
        assert (buf[:o_off] == 7.0).all() and (buf[o_off + m * n:] == 7.0).all()


LARGE, SMALL = "4,8,1", "2,4,2"


@pytest.mark.parametrize("t,m,n,k,shape", [
    (O.Q6_K, 128, 256 * 164, 1024, LARGE),  # 164 of 256 large tiles in one round
    (O.Q6_K, 128, 256 * 163, 1024, None),
    (O.Q6_K, 128, 256 * 164, 768, None),    # (short rows)
    (O.Q6_K, 128, 128 * 103, 1024, SMALL),  # 206 small tiles
    (O.Q6_K, 128, 128 * 102, 1024, None),
    (O.Q6_K, 80, 128 * 103, 1024, None),    # (token tiles a quarter empty and more)
    (O.Q6_K, 384, 128 * 69, 1024, None),    # two rounds of small tiles, 414 and 420 of 512
    (O.Q6_K, 384, 128 * 70, 1024, SMALL),
    (O.Q6_K, 448, 128 * 55, 1024, SMALL),   # 385 of 512 behind 384 rows
    (O.Q6_K, 448, 128 * 54, 1024, None),
    (O.Q5_K, 128, 256 * 246, 1024, LARGE),
    (O.Q5_K, 128, 256 * 245, 1024, None),
    (O.Q5_K, 448, 128 * 36, 1024, SMALL),
    (O.Q5_K, 448, 128 * 35, 1024, None),
    (O.Q4_K, 448, 128 * 36, 1024, SMALL),
    (O.Q4_K, 384, 128 * 42, 1024, None),
])
def test_f16_kernel_by_default(hip, ref, t, m, n, k, shape):
    """Which calls take the f16 kernel on raw rows, and in which shape, on both sides of the lines; results of a few tokens
    against the oracle."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the tile counts are of 256 compute units")
    say("f16 default", O.NAMES[t], m, n, k)
    w = O.random_blocks(t, 95, n, k)
    acts = ref.quantize_q8_0(synth.normal_f32(96, m * k))
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    dy = torch.empty((m, n), dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda(), dy, m, n, k, accumulate=False, workspace=ws)
    torch.cuda.synchronize()
    if shape:
        assert last_launch().startswith(f"gemm_f16_kernel<{O.NAMES[t]},{shape}"), last_launch()
    else:
        assert not last_launch().startswith("gemm_f16_kernel"), last_launch()
    rows = [0, 63, 64, m - 1]
    y_ref = oracle_rows(ref, t, w, acts, n, k, rows)
    assert np.abs(dy.cpu().numpy()[rows] - y_ref).max() <= FP32_REL_TOL * np.abs(y_ref).max()


@pytest.mark.parametrize("t,variant", [(O.Q4_K, 300), (O.Q4_K, 301), (O.Q4_K, 302), (O.Q5_K, 301), (O.Q5_K, 302),
                                       (O.Q6_K, 301), (O.Q6_K, 302)])
def test_f16_kernels_on_infinite_block_scales(hip, ref, tuning, t, variant):
    """Activations beyond the range of a block's f16 scale (the quantizer's scale is an infinity there): infinities of the
    same sign and NaNs where the int8 tile kernel has them, and every other token as without them.  (Q6_K: no number; the
    tile kernel adds the two halves of a sub-block as infinities, this one before the scale, the oracle has NaNs.)"""
    m, n, k = 70, 160, 768
    w = O.random_blocks(t, 71, n, k)
    acts = ref.quantize_q8_0(synth.normal_f32(72, m * k)).reshape(m, k // 32, 34)
    clean = acts.copy()
    acts[3, 5, :2] = [0x00, 0x7C]   # +inf in one block of token 3
    acts[66, :, :2] = [0x00, 0x7C]  # in all of token 66
    acts[40, 23, :2] = [0x00, 0x7E]  # a NaN
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    dw = torch.from_numpy(w).cuda()
    tuning("gemm_tile_min_rows", 1)

    def product(a, v):
        tuning("gemm_variant", v)
        dy = torch.empty((m, n), dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, torch.from_numpy(a.reshape(-1)).cuda(), dy, m, n, k, accumulate=False, workspace=ws)
        torch.cuda.synchronize()
        return dy.cpu().numpy()

    y, y_tile, y_clean = product(acts, variant), product(acts, 99), product(clean, variant)
    assert np.isinf(y_tile[3]).any() and np.isnan(y_tile[40]).all()
    for r in (3, 66, 40):
        if t == O.Q6_K:
            assert not np.isfinite(y[r]).any()
            continue
        assert np.array_equal(np.isnan(y[r]), np.isnan(y_tile[r])), r
        assert np.array_equal(np.sign(y[r][np.isinf(y[r])]), np.sign(y_tile[r][np.isinf(y_tile[r])])), r
    rest = [r for r in range(m) if r not in (3, 66, 40)]
    assert np.array_equal(y[rest], y_clean[rest])


def test_scaled_sums_errors(hip):
    kern = hip.HipKernel(O.Q6_K)
    z = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    with pytest.raises(hip.UnsupportedShape):
        kern.gemm_scaled_sums_dev(z, z, z, z, 4, 32, 256, z)
    kern = hip.HipKernel(O.Q4_K)
    with pytest.raises(hip.BufferTooSmall):
        kern.gemm_scaled_sums_dev(z, z, z, z, 4, 32, 256, z[:256])


@pytest.mark.parametrize("shape", [(130, 300, 16384), (97, 1030, 14336), (257, 1283, 4608), (40, 256 * 288 - 3, 2048)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K], ids=lambda t: O.NAMES[t])
def test_f16_kernel_on_an_even_deal(hip, ref, tuning, t, shape):
    """Runs of (tile, super-block) units: a unit each (4 tiles of 64 to 256 work groups), runs that cross tiles, a whole tile
    before the run; tokens and rows past the edges.  The bars of the kernel's other shapes, the bias and accumulation bit for
    bit, and too little room for the sums (or too few units) takes another kernel."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the runs are those of 256 compute units")
    m, n, k = shape
    say("f16 even deal", O.NAMES[t], shape)
    tuning("gemm_variant", 303)
    w = O.random_blocks(t, 40 + m, n, k)
    x = synth.normal_f32(41 + n, m * k)
    x[:k] *= 300.0
    acts = ref.quantize_q8_0(x)
    kern = hip.HipKernel(t)
    ws = torch.full((64 << 20,), 255, dtype=torch.uint8, device="cuda")  # (NaNs wherever nothing is stored)
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    dy = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw, da, dy, m, n, k, accumulate=False, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_f16_deal_kernel"), last_launch()
    y = dy.cpu().numpy()
    assert np.all(y[m] == 7.0)
    rows = range(m) if n < 2000 else [0, 1, 31, 32, m - 1]
    y_ref = oracle_rows(ref, t, w, acts, n, k, rows)
    for r, want in zip(rows, y_ref):
        err, scale = np.abs(y[r] - want).max(), np.abs(want).max()
        assert err <= FP32_REL_TOL * scale, f"token {r}: max err {err:.3e} vs |y|inf {scale:.3e}"
    dy2 = dy.clone()
    kern.gemm_q8_dev(dw, da, dy2, m, n, k, accumulate=True, workspace=ws)
    bias = torch.from_numpy(synth.normal_f32(93, n + 1)).cuda()
    dy3 = torch.empty(m * n + 1, dtype=torch.float32, device="cuda")
    for off in (0, 1):
        linear.linear_forward_batch_dev(t, dw, da, dy3[off:off + m * n], m, n, k, d_bias=bias[off:off + n], workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(dy3[off:off + m * n].view(m, n), dy[:m] + bias[off:off + n])
    assert torch.equal(dy2[:m], dy[:m] + dy[:m])
    for small, width in ((ws[:-256], n), (ws, 100)):
        kern.gemm_q8_dev(dw, da, dy2, m, width, k, accumulate=False, workspace=small)
        assert not last_launch().startswith("gemm_f16_deal_kernel"), last_launch()
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", [(258, 256 * 96 - 3, 2048), (130, 256 * 170 - 3, 1024), (130, 256 * 128, 512)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K], ids=lambda t: O.NAMES[t])
def test_f16_even_deal_behind_whole_tiles(hip, ref, tuning, t, shape):
    """A whole tile to each work group before its run, of two and three token tiles: runs of a unit, runs that cross tiles, and no
    run at all (256 tiles, no second launch).  The large shape's bits where a tile is one work group's, nothing past the rows, 1e-5 of the
    oracle for tokens of every token tile."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the whole tiles are those of 256 compute units")
    m, n, k = shape
    say("f16 even deal behind whole tiles", O.NAMES[t], shape)
    w = O.random_blocks(t, 50 + m, n, k)
    acts = ref.quantize_q8_0(synth.normal_f32(51, m * k))
    kern = hip.HipKernel(t)
    ws = torch.full((64 << 20,), 255, dtype=torch.uint8, device="cuda")  # (NaNs wherever nothing is stored)
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    dy, whole = (torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda") for _ in range(2))
    for y, variant, name in ((dy, 303, "gemm_f16_deal_kernel"), (whole, 301, "gemm_f16_kernel")):
        tuning("gemm_variant", variant)
        kern.gemm_q8_dev(dw, da, y, m, n, k, accumulate=False, workspace=ws)
        assert last_launch().startswith(name), last_launch()
    torch.cuda.synchronize()
    assert bool((dy[m] == 7.0).all())
    m_tiles = (m + 127) // 128
    own = torch.zeros((m, n), dtype=torch.bool)  # the tiles before the runs: 256, the token tiles of a set of weight rows together
    for tile in range(256):
        own[tile % m_tiles * 128:(tile % m_tiles + 1) * 128, tile // m_tiles * 256:(tile // m_tiles + 1) * 256] = True
    own = own.cuda()
    assert torch.equal(dy[:m][own], whole[:m][own])
    rows = sorted({0, 127, 128, 129, m // 2, m - 1})
    y, want = dy[rows].cpu().numpy(), oracle_rows(ref, t, w, acts, n, k, rows)
    assert (np.abs(y - want).max(axis=1) <= FP32_REL_TOL * np.abs(want).max(axis=1)).all()


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K], ids=lambda t: O.NAMES[t])
def test_f16_even_deal_on_infinite_block_scales(hip, ref, tuning, t):
    """Infinite and NaN block scales in runs that several work groups share: infinities and NaNs where whole tiles have them,
    every other token as without them."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the runs are those of 256 compute units")
    m, n, k = 130, 300, 16384
    say("f16 even deal, infinite scales", O.NAMES[t])
    w = O.random_blocks(t, 73, n, k)
    acts = ref.quantize_q8_0(synth.normal_f32(74, m * k)).reshape(m, k // 32, 34)
    clean = acts.copy()
    acts[3, 5, :2] = [0x00, 0x7C]    # +inf in one block of token 3
    acts[7, 300, :2] = [0x00, 0xFC]  # -inf in another run of token 7
    acts[129, :, :2] = [0x00, 0x7C]  # in all of token 129
    acts[40, 511, :2] = [0x00, 0x7E]  # a NaN
    kern = hip.HipKernel(t)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    dw = torch.from_numpy(w).cuda()

    def product(a, v, name):
        tuning("gemm_variant", v)
        dy = torch.empty((m, n), dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, torch.from_numpy(a.reshape(-1)).cuda(), dy, m, n, k, accumulate=False, workspace=ws)
        torch.cuda.synchronize()
        assert last_launch().startswith(name), last_launch()
        return dy.cpu().numpy()

    deal, whole = product(acts, 303, "gemm_f16_deal_kernel"), product(acts, 301, "gemm_f16_kernel")
    y_clean = product(clean, 303, "gemm_f16_deal_kernel")
    for r in (3, 7, 40, 129):
        assert not np.isfinite(whole[r]).any(), r
        assert np.array_equal(np.isnan(deal[r]), np.isnan(whole[r])), r
        assert np.array_equal(np.sign(deal[r][np.isinf(deal[r])]), np.sign(whole[r][np.isinf(whole[r])])), r
    rest = [r for r in range(m) if r not in (3, 7, 40, 129)]
    assert np.array_equal(deal[rest], y_clean[rest]) and np.isfinite(y_clean).all()


@pytest.mark.parametrize("t,m,n,k,deal", [
    (O.Q4_K, 333, 4096, 14336, True), (O.Q4_K, 333, 4096, 4096, False), (O.Q5_K, 65, 28672, 4096, True),
    (O.Q5_K, 64, 28672, 4096, False), (O.Q6_K, 200, 4096, 4096, False), (O.Q6_K, 200, 4096, 11008, True),
    (O.Q6_K, 512, 14336, 4096, False)])
def test_f16_even_deal_by_default(hip, ref, t, m, n, k, deal):
    """Which calls take the even deal; with a workspace that has no room for it, of the size without it, another kernel
    serves; the static scratch gives the workspace form's bits though its limit counts no such room."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the lines are of 256 compute units")
    say("f16 even deal by default", O.NAMES[t], m, n, k)
    kern = hip.HipKernel(t)
    need = kern.gemm_workspace_bytes(m, n, k)
    assert (need == 64 << 20) == deal
    w = O.random_blocks(t, 95, n, k)
    acts = ref.quantize_q8_0(synth.normal_f32(96, m * k))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    dy, other = (torch.empty((m, n), dtype=torch.float32, device="cuda") for _ in range(2))
    kern.gemm_q8_dev(dw, da, dy, m, n, k, accumulate=False, workspace=ws)
    assert last_launch().startswith("gemm_f16_deal_kernel") == deal, last_launch()
    kern.gemm_q8_static_dev(dw, da, other, m, n, k)
    torch.cuda.synchronize()
    assert torch.equal(other, dy)
    if deal:
        least = ((k // 32) * ((m + 127) // 128 * 128 + 128) * 74 + 255) // 256 * 256
        kern.gemm_q8_dev(dw, da, other, m, n, k, accumulate=False, workspace=ws[:least])
        assert not last_launch().startswith("gemm_f16_deal_kernel"), last_launch()
    torch.cuda.synchronize()
    rows = [0, 63, 64 % m, m - 1]
    y_ref = oracle_rows(ref, t, w, acts, n, k, rows)
    for got in (dy, other):
        assert np.abs(got.cpu().numpy()[rows] - y_ref).max() <= FP32_REL_TOL * np.abs(y_ref).max()


def test_workspaces_of_a_shape_on_the_even_deal(hip, ref):
    """What a call must have and what it runs best with: refused below the first with that size, on the other kernels below the
    second, on the deal from there on, without a workspace, and in a captured graph."""
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the lines are of 256 compute units")
    t, m, n, k = O.Q4_K, 333, 4096, 14336
    say("workspaces of the even deal")
    kern = hip.HipKernel(t)
    least, best = kern.gemm_least_workspace_bytes(m, n, k), kern.gemm_workspace_bytes(m, n, k)
    assert least <= capi.load().oxq_gemm_q8_static_max_workspace_bytes() < best == 64 << 20
    acts = ref.quantize_q8_0(synth.normal_f32(98, m * k))
    dw, da = torch.from_numpy(O.random_blocks(t, 97, n, k)).cuda(), torch.from_numpy(acts).cuda()
    ws = torch.empty(best, dtype=torch.uint8, device="cuda")
    want, got = (torch.empty((m, n), dtype=torch.float32, device="cuda") for _ in range(2))
    with pytest.raises(hip.BufferTooSmall) as e:
        kern.gemm_q8_dev(dw, da, got, m, n, k, workspace=ws[:least - 256])
    assert (e.value.needed, e.value.available) == (least, least - 256)
    for size, deal in ((least, False), (best - 256, False), (best, True)):
        kern.gemm_q8_dev(dw, da, want, m, n, k, workspace=ws[:size])
        assert last_launch().startswith("gemm_f16_deal_kernel") == deal, (size, last_launch())
    for call in (lambda: kern.gemm_q8_dev(dw, da, got, m, n, k), lambda: kern.gemm_q8_static_dev(dw, da, got, m, n, k)):
        got.zero_()
        call()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kern.gemm_q8_dev(dw, da, got, m, n, k, workspace=ws)
    for _ in range(3):
        got.zero_()
        ws.fill_(255)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    big = 1100  # (more than the static form's limit, though its array would hold the sums)
    with pytest.raises(hip.BufferTooSmall) as e:
        kern.gemm_q8_static_dev(dw, da, got, big, n, k)
    assert (e.value.needed, e.value.available) == (kern.gemm_least_workspace_bytes(big, n, k), 16 << 20)


@pytest.mark.parametrize("variant", [16, 23])
@pytest.mark.parametrize("t,k", [(O.Q4_K, 1024), (O.Q6_K, 768), (O.Q4_0, 1056), (O.IQ4_XS, 1280)], ids=lambda v: str(v))
def test_tiles_of_at_most_32_rows(hip, ref, tuning, t, k, variant):
    """The 64-token tiles of the tile kernel compute one token tile of 32 where they hold no more rows: the bits of full
    tiles (a token's sums do not depend on its neighbours), plain and in expert groups, nothing past the rows, 1e-5 of the oracle."""
    n, groups = 193, [1, 32, 33, 0, 64, 65, 96, 97]
    offsets = np.concatenate([[0], np.cumsum(groups)]).astype(np.int32)
    m = int(offsets[-1])
    say("short tiles", O.NAMES[t], k, variant)
    tuning("gemm_variant", variant)
    tuning("gemm_tile_min_rows", 1)
    w = O.random_blocks(t, 70 + variant, n, k).reshape(-1)
    acts = ref.quantize_q8_0(synth.normal_f32(71, m * k)).reshape(-1)
    kern, row = hip.HipKernel(t), k // 32 * 34
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    full = torch.empty((448, n), dtype=torch.float32, device="cuda")  # (whole tiles: the rows past m are zeros)
    da_full = torch.zeros(448 * row, dtype=torch.uint8, device="cuda")
    da_full[:m * row] = da
    ws = torch.empty(max(kern.gemm_workspace_bytes(448, n, k), kern.moe_gemm_workspace_bytes(m, n, k)), dtype=torch.uint8, device="cuda")
    kern.gemm_q8_dev(dw, da_full, full, 448, n, k, accumulate=False, workspace=ws)
    assert last_launch().startswith("gemm_tile_kernel"), last_launch()
    for rows in (1, 31, 32, 33, 65, 95, 96, 97):
        y = torch.full((rows + 1, n), 7.0, dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, da, y, rows, n, k, accumulate=False, workspace=ws)
        assert last_launch().startswith("gemm_tile_kernel"), last_launch()
        assert torch.equal(y[:rows], full[:rows]) and bool((y[rows] == 7.0).all()), rows
    d_off = torch.from_numpy(offsets).cuda()
    y = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    experts = dw.repeat(len(groups))
    kern.moe_gemm_q8_dev(experts, w.nbytes, len(groups), da, d_off, m, max(groups), y, n, k, ws)
    assert last_launch().startswith("gemm_tile_kernel"), last_launch()
    assert torch.equal(y[:m], full[:m]) and bool((y[m] == 7.0).all())
    rows = [0, 31, 32, m - 1]
    want = oracle_rows(ref, t, w, acts, n, k, rows)
    assert np.abs(full.cpu().numpy()[rows] - want).max() <= FP32_REL_TOL * np.abs(want).max()


@pytest.mark.parametrize("variant", [16, 23])
@pytest.mark.parametrize("t", [O.Q4_K, O.Q6_K, O.Q8_0], ids=lambda t: O.NAMES[t])
def test_short_tiles_of_many_experts(hip, ref, tuning, t, variant):
    """150 experts of 0 to 130 rows (three scans of 64), their tiles of at most 32 rows behind the others or not: every row is the
    plain matmul's, bit for bit, and nothing is stored past the last."""
    n, k, e = 129, 256, 150
    say("short tiles of many experts", O.NAMES[t], variant)
    rng = np.random.default_rng(7 + variant)
    groups = rng.permutation(np.concatenate([rng.integers(0, 131, e - 12), [0, 1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129]]))
    offsets = np.concatenate([[0], np.cumsum(groups)]).astype(np.int32)
    m = int(offsets[-1])
    tuning("gemm_variant", variant)
    tuning("gemm_tile_min_rows", 1)
    w = O.random_blocks(t, 79, n, k).reshape(-1)
    acts = ref.quantize_q8_0(synth.normal_f32(80, m * k))
    kern = hip.HipKernel(t)
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    want = torch.empty((m, n), dtype=torch.float32, device="cuda")
    ws = torch.empty(max(kern.gemm_workspace_bytes(m, n, k), kern.moe_gemm_workspace_bytes(m, n, k)), dtype=torch.uint8, device="cuda")
    kern.gemm_q8_dev(dw, da, want, m, n, k, accumulate=False, workspace=ws)
    y = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    kern.moe_gemm_q8_dev(dw.repeat(e), w.nbytes, e, da, torch.from_numpy(offsets).cuda(), m, int(groups.max()), y, n, k, ws)
    assert last_launch().startswith("gemm_tile_kernel"), last_launch()
    assert torch.equal(y[:m], want) and bool((y[m] == 7.0).all())


@pytest.mark.parametrize("variant,n", [(23, 5600), (16, 22400)])
@pytest.mark.parametrize("t", [O.Q4_K, O.Q4_0], ids=lambda t: O.NAMES[t])
def test_short_tiles_behind_the_others(hip, ref, tuning, t, variant, n):
    """Grids of more tiles than the chip holds at a time (175 sets of weight rows, which the XCDs do not share evenly) launch a
    third, short token tile last: the bits of full tiles, every tile once, nothing past the rows, 1e-5 of the oracle."""
    k = 256
    say("short tiles last", O.NAMES[t], n, variant)
    tuning("gemm_variant", variant)
    w = O.random_blocks(t, 75, n, k).reshape(-1)
    acts = ref.quantize_q8_0(synth.normal_f32(76, 192 * k)).reshape(-1)
    kern = hip.HipKernel(t)
    dw, da = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda()
    full = torch.empty((192, n), dtype=torch.float32, device="cuda")
    ws = torch.empty(kern.gemm_workspace_bytes(192, n, k), dtype=torch.uint8, device="cuda")
    kern.gemm_q8_dev(dw, da, full, 192, n, k, accumulate=False, workspace=ws)
    grids = {last_launch()}
    for rows in (129, 142, 160, 161):
        y = torch.full((rows + 1, n), 7.0, dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, da, y, rows, n, k, accumulate=False, workspace=ws)
        grids.add(last_launch())
        assert torch.equal(y[:rows], full[:rows]) and bool((y[rows] == 7.0).all()), rows
    if hip.device_info()["compute_units"] < 260:
        assert len(grids) == 2, grids  # (161 and 192 rows: three whole tiles)
    rows = [0, 63, 128, 191]
    want = oracle_rows(ref, t, w, acts, n, k, rows)
    assert np.abs(full.cpu().numpy()[rows] - want).max() <= FP32_REL_TOL * np.abs(want).max()
