"""The kernel whose weights go straight from memory into the matrix core's registers and whose tokens stay there (oxq_gemm_direct.hpp), on
one matrix and up to 512 token rows, against the CPU oracle: fp32 within 1e-5 * |y_ref|_inf, the integer sums of its debug dump bit-exact."""
import numpy as np
import pytest

import oracle as O
from oxillama_amd import synth
from test_gpu_gemm_skinny import last_launch, off_16_bytes, ref_sums, sum_groups, weights
from test_gpu_parity import assert_close, canonical_ref, say

pytestmark = pytest.mark.gpu

FORMATS = [O.Q4_K, O.Q5_K, O.Q6_K, O.IQ4_XS, O.Q4_0, O.Q8_0]

# (rows, n, k).  512..1024: four parts of k, two row tiles at a time (two, three and four super-blocks: parts without work);
# 1280..2048: eight parts (five and eight super-blocks); 2304..4096: sixteen (nine, fifteen, sixteen), for 17 to 32 rows eight
# of two (the last of them with one super-block or none); longer: each wave its own run (17: runs of two and three; 33; 43).
# Row tiles with rows to spare (18 rows, not one: the bar is 1e-5 of the largest of a token's results, and a single result can be far
# smaller than its terms), an odd number of tiles, more tiles than work groups; odd super-blocks put every second row
# of Q6_K off a dword.
SHAPES = [(16, 33, 512), (1, 18, 768), (7, 20, 1024), (16, 4129, 512), (13, 100, 1280), (5, 8300, 2048), (9, 4113, 2304), (16, 40, 3840),
          (16, 17, 4096), (3, 4099, 4096), (17, 33, 768), (32, 100, 1280), (21, 4131, 2048), (18, 50, 2304), (32, 35, 3840), (25, 8210, 4096),
          (16, 35, 4352), (2, 16, 8448), (11, 4099, 11008)]
# More than 32 rows: token tiles in one run and several, full and not; three and four of them to a work group (33 rows of 4128 weight rows and more: few
# enough row tiles are dealt to more work groups with fewer tokens), resident and streamed; row tiles more than work groups.
WIDE = [(33, 4130, 512), (64, 4128, 1024), (77, 8200, 1280), (130, 4118, 2048), (49, 18, 768), (512, 50, 512), (333, 100, 2048),
        (35, 4100, 2304), (65, 2100, 4096), (40, 2080, 4352), (64, 4113, 5120), (100, 33, 8448), (115, 2050, 11008), (17, 4099, 4352)]


@pytest.mark.parametrize("t", FORMATS, ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_direct_kernel(hip, ref, tuning, t, shape):
    import torch
    from oxillama_amd import linear
    m, n, k_ = shape
    say("direct", O.NAMES[t], shape)
    w = weights(t, 171, n, k_)
    acts = ref.quantize_q8_0(synth.normal_f32(172 + m, m * k_)).reshape(m, k_ // 32 * 34)
    bias = synth.normal_f32(173, n)
    kern = hip.HipKernel(t)
    dw, da, db = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda(), torch.from_numpy(bias).cuda()
    tuning("gemm_tile_min_rows", 1)
    tuning("gemm_variant", 207)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    dy = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw, da, dy, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_direct_kernel<"), last_launch()
    y = dy.cpu().numpy()
    assert (y[m:] == 7.0).all()
    for r in sorted({0, m // 2, min(15, m - 1), m - 1}):
        assert_close(y[r], canonical_ref(ref, t, w, acts[r], n, k_), f"{shape} row {r}")
    dy2 = dy[:m].clone()
    kern.gemm_q8_dev(dw, da, dy2, m, n, k_, accumulate=True, workspace=ws)
    dy3 = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    linear.linear_forward_batch_dev(t, dw, da, dy3, m, n, k_, d_bias=db, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(dy2, dy[:m] + dy[:m]) and torch.equal(dy3, dy[:m] + db[None, :])
    # the dump: the same bits, the oracle's integers
    dy4 = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    dsum = torch.full((m, n, sum_groups(t, k_)), -1, dtype=torch.int32, device="cuda")
    kern.gemm_block_sums_dev(dw, da, dy4, dsum, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_direct_kernel<"), last_launch()
    assert torch.equal(dy4, dy[:m])
    for r in (0, m - 1):
        assert (dsum[r].cpu().numpy() == ref_sums(ref, t, w, acts[r], n, k_)).all(), f"integer sums of row {r}"


@pytest.mark.parametrize("t,m,n,k_,direct", [
    (O.Q4_K, 5, 2560, 2560, True), (O.Q4_K, 4, 2560, 2560, False), (O.IQ4_XS, 3, 2560, 4096, True), (O.Q4_K, 33, 2560, 2560, True),
    (O.Q6_K, 16, 4096, 5120, True), (O.Q6_K, 16, 4112, 5120, False), (O.Q6_K, 17, 4096, 5120, True), (O.Q6_K, 17, 4112, 5120, False), (O.Q8_0, 16, 1024, 5120, False),
    (O.Q8_0, 16, 1536, 5120, True), (O.Q4_0, 16, 48, 33024, False), (O.Q4_0, 77, 8960, 1536, True), (O.Q4_K, 64, 4096, 14336, False), (O.Q6_K, 64, 4096, 14336, True),
    (O.Q4_K, 128, 14336, 4096, True), (O.Q6_K, 80, 14336, 4096, False), (O.Q8_0, 512, 1024, 2048, True), (O.Q4_K, 513, 256, 2048, False), (O.Q4_1, 16, 2560, 2560, False),
    # long rows: the chain against the few-token kernel's split of k, alone on its compute units and not, up to eight rows and up to 32
    (O.Q4_K, 16, 2048, 13312, True), (O.Q4_K, 16, 2048, 14336, True), (O.Q4_K, 16, 2048, 15360, False), (O.Q4_K, 8, 2048, 15360, True), (O.IQ4_XS, 16, 2048, 15360, True), (O.Q5_K, 16, 2048, 14336, False), (O.Q4_K, 8, 2048, 20480, True), (O.Q4_K, 8, 2048, 22528, False), (O.Q4_K, 16, 4096, 26624, True),
    (O.Q5_K, 16, 4096, 26624, True), (O.Q5_K, 16, 4096, 27648, False), (O.Q4_0, 16, 2048, 11264, False), (O.Q8_0, 16, 2048, 7168, True), (O.Q8_0, 16, 2048, 8192, False),
    (O.Q8_0, 16, 4096, 14336, True), (O.Q8_0, 32, 2048, 14336, True), (O.Q8_0, 32, 2048, 16384, False), (O.Q6_K, 32, 1024, 32512, True),
    (O.Q6_K, 32, 1024, 32768, False), (O.Q4_K, 32, 2560, 16384, True), (O.Q4_K, 32, 2560, 17408, False), (O.Q4_0, 5, 256, 6144, False),
    (O.IQ4_XS, 5, 256, 6144, True), (O.Q6_K, 96, 1024, 32768, False)],
    ids=lambda v: O.NAMES.get(v, str(v)) if isinstance(v, int) and not isinstance(v, bool) else str(v))
def test_direct_kernel_by_default(hip, ref, t, m, n, k_, direct):
    """The library's own choice on both sides of each bound (16 x 256 compute units; 4097 to 32768 columns; the first row counts
    at which GEMV launches end)."""
    import torch
    if hip.device_info()["compute_units"] != 256:
        pytest.skip("the bounds above are those of 256 compute units")
    w = weights(t, 181, n, k_)
    acts = ref.quantize_q8_0(synth.normal_f32(182, m * k_)).reshape(m, k_ // 32 * 34)
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    dy = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda(), dy, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_direct_kernel<") == direct, last_launch()
    assert_close(dy[m - 1].cpu().numpy(), canonical_ref(ref, t, w, acts[m - 1], n, k_, threads=16), f"m={m}")


@pytest.mark.parametrize("t", [O.Q4_K, O.Q8_0], ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("which", ["weights", "tokens"])
@pytest.mark.parametrize("m", [6, 16, 77])
def test_pointers_off_their_boundary_take_the_other_kernels(hip, ref, t, which, m):
    """Weights off a dword, tokens off 16 bytes: accepted as before, by the kernels that served such calls."""
    import torch
    n, k_ = 200, 1024
    w = weights(t, 191, n, k_)
    acts = ref.quantize_q8_0(synth.normal_f32(192, m * k_)).reshape(m, k_ // 32 * 34)
    off_w, off_a = (2, 0) if which == "weights" else (0, 4)
    dw = torch.zeros(w.nbytes + 16, dtype=torch.uint8, device="cuda")
    da = torch.zeros(acts.nbytes + 16, dtype=torch.uint8, device="cuda")
    dw[off_w:off_w + w.nbytes] = torch.from_numpy(w.reshape(-1)).cuda()
    da[off_a:off_a + acts.nbytes] = torch.from_numpy(acts.reshape(-1)).cuda()
    kern = hip.HipKernel(t)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    dy = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw[off_w:off_w + w.nbytes], da[off_a:off_a + acts.nbytes], dy, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert not last_launch().startswith("gemm_direct_kernel<"), last_launch()
    for r in (0, m - 1):
        assert_close(dy[r].cpu().numpy(), canonical_ref(ref, t, w, acts[r], n, k_), f"row {r}")


@pytest.mark.parametrize("t", FORMATS, ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("shape", WIDE, ids=lambda s: "x".join(map(str, s)))
def test_direct_kernel_on_more_token_tiles(hip, ref, tuning, t, shape):
    import torch
    from oxillama_amd import linear
    m, n, k_ = shape
    say("direct wide", O.NAMES[t], shape)
    w = weights(t, 271, n, k_)
    acts = ref.quantize_q8_0(synth.normal_f32(272 + m, m * k_)).reshape(m, k_ // 32 * 34)
    bias = synth.normal_f32(273, n)
    kern = hip.HipKernel(t)
    dw, da, db = torch.from_numpy(w).cuda(), torch.from_numpy(acts).cuda(), torch.from_numpy(bias).cuda()
    tuning("gemm_tile_min_rows", 1)
    tuning("gemm_variant", 207)
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    dy = torch.full((m + 1, n), 7.0, dtype=torch.float32, device="cuda")
    kern.gemm_q8_dev(dw, da, dy, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_direct_kernel<"), last_launch()
    assert (dy[m:] == 7.0).all()
    rows = [r for r in (0, 15, 16, 31, 32, 47, 48, 63, 64, m // 2, m - 1) if r < m]
    for r in sorted(set(rows)):
        assert_close(dy[r].cpu().numpy(), canonical_ref(ref, t, w, acts[r], n, k_, threads=16), f"{shape} row {r}")
    # every row: the same bits as in a call of its tile alone, which takes one token tile, where k is dealt to the waves alike
    if k_ <= 2048:
        for r0 in range(0, m, 16):
            part = min(16, m - r0)
            one = torch.zeros((part, n), dtype=torch.float32, device="cuda")
            kern.gemm_q8_dev(dw, da[r0:r0 + part].contiguous(), one, part, n, k_, workspace=ws)
            assert torch.equal(one, dy[r0:r0 + part]), f"rows from {r0}"
    dy2 = dy[:m].clone()
    kern.gemm_q8_dev(dw, da, dy2, m, n, k_, accumulate=True, workspace=ws)
    dy3 = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    linear.linear_forward_batch_dev(t, dw, da, dy3, m, n, k_, d_bias=db, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(dy2, dy[:m] + dy[:m]) and torch.equal(dy3, dy[:m] + db[None, :])
    # the dump (two token tiles at most): the same bits, the oracle's integers
    dy4 = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    dsum = torch.full((m, n, sum_groups(t, k_)), -1, dtype=torch.int32, device="cuda")
    kern.gemm_block_sums_dev(dw, da, dy4, dsum, m, n, k_, workspace=ws)
    torch.cuda.synchronize()
    assert last_launch().startswith("gemm_direct_kernel<") and torch.equal(dy4, dy[:m]), last_launch()
    assert (dsum[m - 1].cpu().numpy() == ref_sums(ref, t, w, acts[m - 1], n, k_)).all()


@pytest.mark.parametrize("t", FORMATS, ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("shape", [(13, 100, 1024), (16, 50, 4096), (21, 60, 2304), (77, 4130, 512), (16, 40, 5120), (40, 2080, 4352)],
                         ids=lambda s: "x".join(map(str, s)))
def test_direct_kernel_on_infinite_block_scales(hip, ref, tuning, t, shape):
    """Tokens with infinite block scales (activations beyond f16's range) and a NaN among them: infinities of the same sign and NaNs
    where the tile kernel has them (where a sub-block is one term, the oracle), and every other token as without them.  Four,
    sixteen and eight parts of k in registers, streamed, one to four token tiles."""
    import torch
    m, n, k_ = shape
    say("direct, infinite scales", O.NAMES[t], shape)
    w = weights(t, 371, n, k_)
    clean = ref.quantize_q8_0(synth.normal_f32(372, m * k_)).reshape(m, k_ // 32, 34)
    acts = clean.copy()
    acts[3, 5, :2] = [0x00, 0x7C]                 # +inf in one block
    acts[6, k_ // 32 - 1, :2] = [0x00, 0xFC]      # -inf in the last one
    acts[9, :, :2] = [0x00, 0x7C]                 # in all of a token
    acts[m - 1, k_ // 64, :2] = [0x00, 0x7E]      # a NaN
    kern = hip.HipKernel(t)
    dw = torch.from_numpy(w).cuda()
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    tuning("gemm_tile_min_rows", 1)

    def product(a, variant):
        tuning("gemm_variant", variant)
        dy = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, torch.from_numpy(a.reshape(-1)).cuda(), dy, m, n, k_, workspace=ws)
        torch.cuda.synchronize()
        assert last_launch().startswith("gemm_direct_kernel<" if variant == 207 else "gemm_tile_kernel<"), last_launch()
        return dy.cpu().numpy()

    y, tile, y_clean = product(acts, 207), product(acts, 99), product(clean, 207)
    odd = (3, 6, 9, m - 1)
    assert np.isfinite(y_clean).all() and not np.isfinite(tile[3]).any() and np.isnan(tile[m - 1]).all()
    # (where there is a zero-point term, it and the block's product are mostly infinities of opposite signs; Q4_0 has one in the
    # tile kernel, not in this one)
    assert t in (O.Q4_K, O.Q5_K, O.Q4_0) or np.isinf(tile[3]).any()
    expected = [(tile, odd)] if t != O.Q4_0 else []
    if t in (O.IQ4_XS, O.Q8_0, O.Q4_0):  # (the zero-point terms of the others, and the halves of Q6_K, are infinities of their own)
        want = np.zeros_like(y)
        for r in odd:
            want[r] = canonical_ref(ref, t, w, acts[r].reshape(-1), n, k_)
        expected.append((want, odd))
    for want, rows in expected:
        for r in rows:
            assert np.array_equal(np.isnan(y[r]), np.isnan(want[r])), r
            assert np.array_equal(np.isinf(y[r]), np.isinf(want[r])), r
            assert np.array_equal(y[r][np.isinf(y[r])], want[r][np.isinf(want[r])]), r
    rest = [r for r in range(m) if r not in odd]
    assert np.array_equal(y[rest], y_clean[rest])


@pytest.mark.parametrize("t", FORMATS, ids=lambda t: O.NAMES[t])
@pytest.mark.parametrize("shape", [(16, 512, 1024), (77, 512, 1536), (16, 2352, 14336), (40, 200, 8704)], ids=lambda s: "x".join(map(str, s)))
def test_direct_kernel_is_no_further_from_64_bits(hip, ref, tuning, t, shape):
    """The same terms in another order than the kernels that serve tokens off 16 bytes: no larger an error against 64 bits.  Both
    round each term once and each partial sum; over all results the 2-norms of that noise are within 3 % of a ratio (m * n
    independent values of it, 8000 and more), and orders as short as these differ by a few percent: bar 1.1."""
    import torch
    m, n, k_ = shape
    say("direct, error against 64 bits", O.NAMES[t], shape)
    w = weights(t, 471, n, k_)
    acts = ref.quantize_q8_0(synth.normal_f32(472, m * k_)).reshape(m, k_ // 32, 34)
    a64 = acts[:, :, :2].copy().view(np.float16).astype(np.float64) * acts[:, :, 2:].view(np.int8)
    want = a64.reshape(m, k_) @ ref.dequant_rows(t, w, n, k_).astype(np.float64).T
    kern = hip.HipKernel(t)
    dw = torch.from_numpy(w).cuda()
    ws = torch.empty(kern.gemm_workspace_bytes(m, n, k_), dtype=torch.uint8, device="cuda")
    error = []
    for da, direct in ((torch.from_numpy(acts).cuda(), True), (off_16_bytes(acts), False)):
        dy = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        kern.gemm_q8_dev(dw, da, dy, m, n, k_, workspace=ws)
        torch.cuda.synchronize()
        assert last_launch().startswith("gemm_direct_kernel<") == direct, last_launch()
        error.append(np.linalg.norm(dy.cpu().numpy() - want) / np.linalg.norm(want))
    say(f"  {error[0]:.2e} against {error[1]:.2e}")
    assert error[0] <= 1.1 * error[1]
