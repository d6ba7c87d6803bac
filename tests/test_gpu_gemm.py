"""GPU parity of the Q4_K/Q6_K x Q8_1 GEMM.

Reference value: the product gemm_q4k.cu:103-112, 164-166 computes (mo_gemm_q8_1: exact
integer sub-block sums scaled by d*sc*d8, minus dmin*m*ds for Q4_K).  Contract bar: relative
L2 <= 1e-3.  The kernel sums each sub-block exactly and rescales in fp32, so the
tests hold it to 1e-5.  Small shapes against the fp64 C oracle; the benchmark shapes against
the fp64 torch restatement (tests/torch_ref.py, pinned against the oracle on the CPU) plus
size-independent properties."""
import numpy as np
import pytest
import torch

from mnemocuda_amd import synth
from tests.conftest import rel_l2
from tests import torch_ref
from tests.gpu_util import case, dev, host

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _run(gpu, type_id, wd, actd, M, K, N):
    out = torch.full((N, M), float("nan"), device="cuda")
    gpu.ops.gemm(wd, type_id, actd, out, M, K, N)
    return out


@pytest.mark.parametrize("type_id,M,K,N", [(12, 256, 1024, 128), (12, 100, 512, 37), (14, 130, 768, 9),
                                           (12, 1, 256, 1), (14, 64, 1536, 200),
                                           # ragged tiles with K in 8 slices
                                           (12, 200, 4096, 100), (14, 36, 2048, 68),
                                           # 9 super-blocks: uneven slices of K
                                           (12, 384, 2304, 130)])
def test_gemm_vs_oracle(gpu, oracle, type_id, M, K, N):
    rng = np.random.default_rng(M * N + K)
    w = synth.weights(rng, type_id, M, K)
    act = oracle.quantize_q8_1(rng.standard_normal((N, K)).astype(np.float32))
    case(f"gemm type={type_id} M={M} K={K} N={N}")
    out = _run(gpu, type_id, dev(w), dev(act), M, K, N)
    got, ref = host(out), oracle.gemm(type_id, w, act, M, K, N)
    err = rel_l2(got, ref)
    print(f"rel_l2={err:.2e}")
    if M * N >= 64:
        assert err < TOL
    else:
        # too few outputs for a relative L2 to concentrate: the forward error bound of the
        # fp32 rescale, one rounding per sub-block plus the scale ratios, sum_k |w_k a_k| *
        # (K/32) * 2^-22
        wa = np.abs(oracle.dequant(type_id, w, M, K)).astype(np.float64)
        aa = np.abs(oracle.dequant_q8_1(act, K, N)).astype(np.float64)
        bound = (aa @ wa.T) * (K / 32 * 2.0**-22) + 1e-30
        assert np.all(np.abs(got - ref) <= bound)


# Each workgroup shape with ragged rows and tokens (an M that is no multiple of 4 stores single
# values), and K below, at and above its slices: slices of no super-block, of unequal length, of more
# than one 1024-value window.  Which shape a size takes is the launch rule's; tests/test_gemm_plan.py
# checks that the sizes below reach all of them, for both types.
RAGGED = [
    (33, 256, 17), (31, 2304, 1), (1001, 1280, 15), (4099, 2304, 16), (513, 3328, 65), (1000, 4096, 97),
    (1537, 1536, 201), (2801, 4096, 63), (4093, 1280, 130), (1533, 4352, 510), (4095, 2816, 333), (8191, 1024, 201),
    (6001, 2304, 513), (2047, 4352, 1027), (8190, 1280, 1025), (4093, 5376, 2047),
    # at most one super-block per slice
    (8197, 256, 197), (8263, 512, 195), (8307, 256, 68), (8603, 256, 33), (8201, 768, 33), (4131, 1280, 17),
    (8917, 256, 1), (4109, 256, 1), (5551, 256, 130), (10883, 256, 325), (8311, 512, 338), (2097, 768, 33),
    # more than four
    (33, 8448, 1), (33, 8704, 2070), (8219, 4352, 1), (8455, 4352, 33), (9395, 4864, 34), (8395, 2304, 34),
    (5409, 2304, 337), (8225, 2304, 65), (8401, 2304, 104), (33, 16640, 1), (4123, 8448, 1), (4245, 8704, 17),
    (4655, 4352, 34), (199, 4352, 2157), (8993, 2304, 129),
]


@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("M,K,N", RAGGED)
def test_gemm_shapes_ragged(gpu, type_id, M, K, N):
    rng = np.random.default_rng(M + K + N)
    w = dev(synth.weights(rng, type_id, M, K))
    x = torch.randn((N, K), device="cuda", generator=torch.Generator("cuda").manual_seed(M))
    act = torch.zeros(N * (K // 128) * 144, dtype=torch.uint8, device="cuda")
    case(f"gemm ragged type={type_id} M={M} K={K} N={N}")
    gpu.ops.quantize_q8_1(x, act, K, N)
    out = _run(gpu, type_id, w, act, M, K, N)
    assert torch.equal(out, _run(gpu, type_id, w, act, M, K, N))  # no atomics: the same every time
    ref = torch_ref.gemm(type_id, w, act, M, K, N)
    assert rel_l2(host(out), ref.cpu().numpy()) < TOL


# Roundings of a sum: within a super-block one per sub-block at the running sum's magnitude, which
# grows as the square root of its length (8 / 2 of the block's sum in the mean of squares); then one
# per super-block of a slice (half of them, likewise), log2 for the tree over the slices, one each for
# the min term and the store.  A rounding is 2^-24 / sqrt(3) relative in the root mean square, at
# most (mantissas near 1); a tenth on top for the inputs' draw.
@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("M,K,N", [(64, 256, 300), (512, 4096, 300), (64, 16384, 64), (512, 16384, 300)])
def test_gemm_rounds_once_per_sub_block(gpu, type_id, M, K, N):
    case(f"gemm rounding type={type_id} M={M} K={K} N={N}")
    rng = np.random.default_rng(M + K + N)
    w = dev(synth.weights(rng, type_id, M, K))
    x = torch.randn((N, K), device="cuda", generator=torch.Generator("cuda").manual_seed(M))
    act = torch.zeros(N * (K // 128) * 144, dtype=torch.uint8, device="cuda")
    gpu.ops.quantize_q8_1(x, act, K, N)
    out = _run(gpu, type_id, w, act, M, K, N)
    slices = min(8, K // 256)
    roundings = 8 / 2 + (K // 256 // slices) / 2 + np.log2(slices) + 2
    bar = 1.1 * 2.0**-24 * (roundings / 3) ** 0.5
    err = rel_l2(host(out), torch_ref.gemm(type_id, w, act, M, K, N).cpu().numpy())
    print(f"rel_l2={err:.3e} bar {bar:.3e}")
    assert err < bar


# Wide tiles keep one running sum per slice.  Per sub-block Q6_K's is rounded once (an fma), Q4_K's
# twice, and the scale ratio carries a rounding of its own; one more per super-block (the row's
# scale), all at the running sum's magnitude (half of them, as above); two at the end.  The root mean square over
# mantissas in [1, 2) is 0.74 of a rounding's 2^-24 / sqrt(3); 15 % on top.
@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("M,K,N", [(8192, 4096, 512), (4096, 8192, 1999)])
def test_gemm_wide_tiles_rounding(gpu, type_id, M, K, N):
    from tests.test_gemm_plan import plan
    case(f"gemm wide rounding type={type_id} M={M} K={K} N={N}")
    shape, _, _, slices, *_ = plan(type_id, M, K, N)
    assert shape < 2
    rng = np.random.default_rng(M + K + N)
    w = dev(synth.weights(rng, type_id, M, K))
    x = torch.randn((N, K), device="cuda", generator=torch.Generator("cuda").manual_seed(M))
    act = torch.zeros(N * (K // 128) * 144, dtype=torch.uint8, device="cuda")
    gpu.ops.quantize_q8_1(x, act, K, N)
    out = _run(gpu, type_id, w, act, M, K, N)
    sub = K // 32 / slices
    roundings = (3 if type_id == 12 else 2) * sub / 2 + sub / 8 / 2 + 2
    bar = 1.15 * 0.74 * 2.0**-24 * (roundings / 3) ** 0.5
    err = rel_l2(host(out), torch_ref.gemm(type_id, w, act, M, K, N).cpu().numpy())
    print(f"rel_l2={err:.3e} bar {bar:.3e}")
    assert err < bar


@pytest.mark.parametrize("type_id", [12, 14])
def test_gemm_zero_scales_and_range(gpu, oracle, type_id):
    """Zero weight blocks (d = 0 with nonzero quants), zero activation sub-blocks and sub-blocks
    six decades apart inside one row: the running scale carries across them."""
    M, K, N = 96, 2048, 40
    rng = np.random.default_rng(17 + type_id)
    w = synth.weights(rng, type_id, M, K)
    bb = 144 if type_id == 12 else 210
    wb = w.reshape(M, K // 256, bb)
    dpos = slice(0, 2) if type_id == 12 else slice(208, 210)
    wb[::5, 1, dpos] = 0          # d = 0: the block's main part is zero
    wb[3, :, dpos] = 0            # a whole row of d = 0
    x = rng.standard_normal((N, K)).astype(np.float32)
    # sub-block scales over four decades (the Q8_1 ds field, d * sum x, must stay inside the
    # f16 range: gemm_q4k.cu takes the min term from it)
    x *= np.float32(10.0) ** rng.integers(-3, 2, (N, K // 32)).astype(np.float32).repeat(32, axis=1)
    x[:, 32:64] = 0.0             # a zero sub-block in every row
    x[7, :] = 0.0                 # an all-zero row
    x[9, :512] = 0.0              # zero leading sub-blocks
    x[5, 96:128] *= np.float32(1e-7)  # d = amax/127 rounds to f16 zero, the quants stay +-127
    act = oracle.quantize_q8_1(x)
    case(f"gemm zero scales type={type_id}")
    out = _run(gpu, type_id, dev(wb.reshape(-1)), dev(act), M, K, N)
    got, ref = host(out), oracle.gemm(type_id, wb.reshape(-1), act, M, K, N)
    assert np.all(np.isfinite(got))
    assert np.all(got[7] == 0.0)
    for j in range(N):
        if j != 7:
            assert rel_l2(got[j], ref[j]) < TOL, j


@pytest.mark.parametrize("type_id,M,K,N", [(12, 8192, 4096, 512), (12, 1536, 4096, 512), (14, 4096, 1536, 512),
                                           # 9 super-blocks per slice: three 1024-value windows, the last
                                           # of one super-block
                                           (12, 2048, 4608, 1152)])
def test_gemm_baseline_shapes(gpu, oracle, type_id, M, K, N):
    rng = np.random.default_rng(M + N)
    w = synth.weights(rng, type_id, M, K)
    x = rng.standard_normal((N, K)).astype(np.float32)
    actd = torch.zeros(N * (K // 128) * 144, dtype=torch.uint8, device="cuda")
    case(f"gemm baseline type={type_id} M={M} K={K} N={N}")
    gpu.ops.quantize_q8_1(dev(x), actd, K, N)
    out = _run(gpu, type_id, dev(w), actd, M, K, N)
    ref = torch_ref.gemm(type_id, dev(w), actd, M, K, N)
    err = rel_l2(host(out), ref.cpu().numpy())
    print(f"rel_l2={err:.2e}")
    assert err < TOL
    # linearity in the activation scale: doubling every d8 and ds (both scale with x)
    # doubles the output exactly
    a2 = actd.view(N, K // 128, 144).clone()
    ds = a2[:, :, :16].contiguous().view(torch.float16).clone()
    ds *= 2
    a2[:, :, :16] = ds.view(torch.uint8).reshape(N, K // 128, 16)
    out2 = _run(gpu, type_id, dev(w), a2.reshape(-1), M, K, N)
    assert rel_l2(host(out2), 2 * host(out)) < 1e-6


@pytest.mark.parametrize("type_id", [12, 14])
def test_gemm_large_activations(gpu, oracle, type_id):
    """Rows of very different magnitude (seven decades, |x| up to ~250: beyond that the Q8_1
    block's f16 ds = d8 * sum x, from which the reference takes the min term, overflows)."""
    M, K, N = 192, 1024, 48
    rng = np.random.default_rng(11 + type_id)
    w = synth.weights(rng, type_id, M, K)
    x = rng.standard_normal((N, K)).astype(np.float32)
    x *= np.logspace(-5, 1.9, N, dtype=np.float32)[:, None]
    act = oracle.quantize_q8_1(x)
    case(f"gemm large activations type={type_id}")
    out = _run(gpu, type_id, dev(w), dev(act), M, K, N)
    got, ref = host(out), oracle.gemm(type_id, w, act, M, K, N)
    assert np.all(np.isfinite(got))
    # per token row: rows span 9 decades, so compare each on its own scale
    for j in range(N):
        assert rel_l2(got[j], ref[j]) < TOL, j


def test_gemm_rows_over_4_gib(gpu):
    """17 Q6_K rows of 275 MB: even the smallest tile's rows would span more than a 32-bit offset."""
    from tests.test_gemm_plan import plan
    M, K, N = 17, 5 << 26, 1
    _, _, _, slices, rows1, _ = plan(14, M, K, N)
    assert rows1 < M  # two launches
    nsb = K // 256
    gen = torch.Generator("cuda").manual_seed(3)
    w = torch.randint(0, 256, (M, nsb, 210), dtype=torch.uint8, device="cuda", generator=gen)
    w[:, :, 208:] = torch.tensor([0.01], dtype=torch.float16).view(torch.uint8).cuda()
    act = torch.randint(0, 256, (N, K // 128, 144), dtype=torch.uint8, device="cuda", generator=gen)
    act[:, :, :16] = torch.tensor([0.01, 0.0] * 4, dtype=torch.float16).view(torch.uint8).cuda()
    case(f"gemm long rows M={M} K={K} N={N}")
    out = _run(gpu, 14, w.view(-1), act.view(-1), M, K, N)
    rows = [0, 1, 7, rows1 - 1, rows1, 14, 15, 16]  # the first and last of both launches among them
    ref = torch.zeros((N, len(rows)), dtype=torch.float64, device="cuda")
    var = torch.zeros_like(ref)
    w = w[rows]
    step = 8192  # super-blocks at a time
    for b in range(0, nsb, step):
        n = min(step, nsb - b)
        part = torch_ref.gemm(14, w[:, b:b + n].reshape(-1), act[:, 2 * b:2 * (b + n)].reshape(-1), len(rows), 256 * n, N)
        ref += part
        var += part * part
    # A slice sums n super-blocks of either sign, one rounding each (2^-24 / sqrt(3) of the sum
    # so far at most): the sum's square grows evenly to the slice's share of var, so the error's square is
    # n / 2 * 2^-48 / 3 of var on average.  Over 8 outputs it is spread like a chi-square of 8 degrees
    # (half of it): twice the error is six spreads.  A row read 4 GiB away is an error of the result's
    # size, 10^5 times that.
    err = float((out[:, rows].double() - ref).norm() / var.sum().sqrt())
    bar = 2 * 2.0**-24 * (nsb / slices / 6) ** 0.5
    print(f"err={err:.2e} bar {bar:.2e}")
    assert err < bar


@pytest.mark.parametrize("type_id", [12, 14])
@pytest.mark.parametrize("M,K,N", [(33, 2304, 1), (130, 1280, 70), (2047, 2304, 513), (4099, 1280, 1025)])
def test_gemm_any_weight_address(gpu, type_id, M, K, N):
    """Weights may start at any byte, activation blocks at any multiple of 4."""
    rng = np.random.default_rng(M + K)
    w = dev(synth.weights(rng, type_id, M, K))
    act = torch.zeros(N * (K // 128) * 144, dtype=torch.uint8, device="cuda")
    gpu.ops.quantize_q8_1(torch.randn((N, K), device="cuda", generator=torch.Generator("cuda").manual_seed(M)), act, K, N)
    case(f"gemm alignment type={type_id} M={M} K={K} N={N}")
    ref = _run(gpu, type_id, w, act, M, K, N)
    for off, aoff in ((1, 0), (2, 4), (3, 8), (8, 12)):
        wu = torch.zeros(w.numel() + 16, dtype=torch.uint8, device="cuda")[off:off + w.numel()]
        au = torch.zeros(act.numel() + 16, dtype=torch.uint8, device="cuda")[aoff:aoff + act.numel()]
        wu.copy_(w)
        au.copy_(act)
        assert torch.equal(_run(gpu, type_id, wu, au, M, K, N), ref), (off, aoff)
