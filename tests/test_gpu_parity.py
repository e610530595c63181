"""GPU parity: the HIP kernels, called through the C ABI (ctypes), against the CPU oracle on
the same seeded inputs.  Integer / dequant results must be bit-exact; GEMM outputs must be
within a relative Frobenius error of 2e-3 of the float64 product of the fp16 inputs and the
pinned fp16 weights (TOL below), max-abs error printed."""
import os

import numpy as np
import pytest
import torch

from oracle import awq_ref

pytestmark = pytest.mark.gpu
TOL = 2e-3
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _np_case(M, K, N, G, seed):
    rng = np.random.default_rng(seed)
    g = K if G <= 0 else G
    w = rng.integers(0, 16, (K, N))
    z = rng.integers(0, 16, (K // g, N))
    s = (rng.random((K // g, N)) * 0.019 + 0.001).astype(np.float16)
    x = rng.normal(0, 1, (M, K)).astype(np.float16)
    return x, awq_ref.pack_awq(w), s, awq_ref.pack_awq(z)


def _dev(dev, *arrs):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in arrs]


def _check_gemm(sba, dev, x, qw, s, qz, G, split_k=0, tag="", variant=None):
    ref = awq_ref.gemm_wide(x, qw, s, qz, G)
    xd, qwd, sd, qzd = _dev(dev, x, qw, s, qz)
    y = sba.awq_gemm(xd, qwd, sd, qzd, force_split_k=split_k, _dev_variant=variant)
    torch.cuda.synchronize()
    yh = y.cpu().numpy()
    err = awq_ref.rel_frobenius(yh, ref)
    maxabs = float(np.max(np.abs(yh.astype(np.float64) - ref)))
    print(f"[gemm {tag} M={x.shape[0]} K={x.shape[1]} N={qw.shape[1] * 8} G={G} split={split_k}] "
          f"rel_fro={err:.2e} max_abs={maxabs:.3e}", flush=True)
    assert np.isfinite(yh).all()
    assert err <= TOL
    return yh


# ------------------------------------------------------------------ dequantize (bit-exact)

@pytest.mark.parametrize("K,N,G", [(256, 64, 128), (4096, 4096, 128), (128, 8, 32), (96, 40, 24),
                                   (64, 2056, 64), (384, 128, -1), (30, 16, 3), (512, 264, 256)])
def test_dequantize_bit_exact(sba, gpu, K, N, G):
    _, qw, s, qz = _np_case(1, K, N, G, seed=K + N)
    want = awq_ref.dequantize(qw, s, qz, G)
    qwd, sd, qzd = _dev(gpu, qw, s, qz)
    got = sba.awq_dequantize(qwd, sd, qzd, 0, 0, 0).cpu().numpy()
    assert got.shape == want.shape
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


def test_dequantize_exhaustive_and_fixture(sba, gpu):
    h = np.arange(65536, dtype=np.uint16).view(np.float16)
    with np.errstate(invalid="ignore"):
        finite = h[np.isfinite(h)]
    # every finite fp16 scale (subnormal results included) x every (w, z) pair
    S = finite.size
    N = 16 * S
    N8 = (N + 7) // 8 * 8
    w = np.repeat(np.arange(16)[:, None], N8, axis=1)
    z = np.zeros((1, N8), np.int64)
    s = np.ones((1, N8), np.float16)
    for zz in range(16):
        z[0, zz * S:(zz + 1) * S] = zz
        s[0, zz * S:(zz + 1) * S] = finite
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    with np.errstate(over="ignore"):
        want = ((w - z).astype(np.float64) * s.astype(np.float64)).astype(np.float16)
    got = sba.awq_dequantize(*_dev(gpu, qw, s, qz), 0, 0, 0).cpu().numpy()
    gb, wb = got.view(np.uint16), want.view(np.uint16)
    same = (gb == wb) | (((gb | wb) & 0x7FFF) == 0)     # +0 / -0 both fine
    assert same.all(), np.argwhere(~same)[:5]

    fx = np.load(os.path.join(GOLDEN, "awq_small.npz"))
    got = sba.awq_dequantize(*_dev(gpu, fx["qweight"], fx["scales"], fx["qzeros"]), 0, 0, 0).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), fx["w_dequant_bits"])


# ------------------------------------------------------------------ decode GEMM (M <= 16)

@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("M", [1, 4, 8, 16])
def test_gemm_decode_small(sba, gpu, M, variant):
    x, qw, s, qz = _np_case(M, 1024, 512, 128, seed=10 + M)
    for split in (0, 1, 2, 3, 8):
        _check_gemm(sba, gpu, x, qw, s, qz, 128, split, tag=f"v{variant}", variant=variant)


@pytest.mark.parametrize("K,N,G", [(256, 128, 32), (256, 264, 64), (512, 136, 256), (384, 8, -1),
                                   (128, 2048, 128), (640, 1000, 128)])
def test_gemm_decode_groups_and_ragged_n(sba, gpu, K, N, G):
    x, qw, s, qz = _np_case(5, K, N, G, seed=K * 3 + N)
    g = K if G <= 0 else G
    for split in (0, 1, 2):
        _check_gemm(sba, gpu, x, qw, s, qz, g, split)


@pytest.mark.parametrize("K,N,split,M", [(640, 256, 1, 16), (1152, 512, 1, 3), (1152, 512, 2, 16),
                                         (4736, 256, 8, 1), (4736, 264, 8, 16), (29568, 256, 8, 7)])
def test_gemm_decode_left_over_chunks_step_by_step(sba, gpu, K, N, split, M):
    """Chunk counts that leave L chunks over after each of the 4 x split waves got the same
    number, with 4 L <= waves: the left-over chunks are taken one 32-row step per wave (all
    waves, some of them, or - N = 264 - in the one-word-per-lane form that never does).  Checked
    against the oracle, against the whole-chunk form (development variant bit 1 << 23) within tolerance, and
    exactly with one-hot activations that sit inside the left-over chunks."""
    x, qw, s, qz = _np_case(M, K, N, 128, seed=K + N + split)
    y = _check_gemm(sba, gpu, x, qw, s, qz, 128, split, tag="tail steps")
    y_whole = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), force_split_k=split, _dev_variant=1 << 23).cpu().numpy()
    assert awq_ref.rel_frobenius(y, y_whole.astype(np.float64)) <= 1e-3
    W = awq_ref.dequantize(qw, s, qz, 128)
    nchunks, parts = K // 128, 4 * split
    first_left = (nchunks // parts) * parts * 128          # first row of the left-over chunks
    ks = [0, first_left - 1, first_left, first_left + 31, first_left + 32, first_left + 100, K - 33, K - 1]
    xo = np.zeros((len(ks), K), np.float16)
    for m, k in enumerate(ks):
        xo[m, k] = 1
    yo = sba.awq_gemm(*_dev(gpu, xo, qw, s, qz), force_split_k=split).cpu().numpy()
    for m, k in enumerate(ks):
        assert np.array_equal(yo[m].view(np.uint16), W[k].view(np.uint16)), (m, k)


@pytest.mark.parametrize("M", [17, 24, 32, 33, 48, 64])
def test_gemm_mid_m_skinny_passes(sba, gpu, M):
    """17 .. 32 rows with a set K split run one pass of the skinny kernel (two row blocks share every unpacked weight),
    without one a tile of 32 rows; more rows ignore the split and run tiles; the skinny kernel's passes of up to 32 rows over
    all of them by development variant bit 1 << 18."""
    from server_benchmark_amd import _lib
    form = _lib.load().awqmi_dev_last_gemm_form
    x, qw, s, qz = _np_case(M, 1024, 512, 128, seed=200 + M)
    for split in (0, 1, 4):
        _check_gemm(sba, gpu, x, qw, s, qz, 128, split, tag="mid-M")
        assert form() == (_lib.FORM_SKINNY if split and M <= 32 else _lib.FORM_FUSED)
        _check_gemm(sba, gpu, x, qw, s, qz, 128, split, tag="mid-M skinny", variant=1 << 18)
        assert form() == _lib.FORM_SKINNY
    x, qw, s, qz = _np_case(M, 512, 264, 64, seed=300 + M)      # ragged N, G = 64
    _check_gemm(sba, gpu, x, qw, s, qz, 64, 0, tag="mid-M")


@pytest.mark.parametrize("M,K,N,G,split", [(17, 4096, 272, 128, 1), (32, 3072, 2048, 64, 1), (24, 12288, 512, 128, 4),
                                           (32, 8192, 256, 1024, 2), (24, 3072, 33280, 32, 0)])
def test_gemm_32_row_pass_with_lds_weight_ring(sba, gpu, M, K, N, G, split):
    """17 .. 32 rows over long wave ranges (24 chunks of 128 rows a part and more) keep the weight ring in LDS; the
    register-ring form (development variant bit 4096) must give the same bits.  Every case runs the skinny kernel: two words a
    lane, and a set split or groups that no tile takes."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + K)
    assert K // 128 >= 24 * (split or lib.awqmi_gemm_auto_split_k(M, K, N, G))
    y = _check_gemm(sba, gpu, x, qw, s, qz, G, split, tag="32-row lds ring")
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_SKINNY
    y_reg = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), force_split_k=split, _dev_variant=4096).cpu().numpy()
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_SKINNY
    assert np.array_equal(y.view(np.uint16), y_reg.view(np.uint16))


@pytest.mark.parametrize("K,N,G,split", [
    (128, 16, 128, 0),        # one chunk: three waves of four without work
    (640, 272, 32, 0),        # ragged last column block, five chunks on four waves, a group per step
    (768, 528, 64, 3),        # K split with more parts than chunks a part
    (1024, 1040, 256, 2),
    (2048, 512, -1, 4),
    (128 * 41, 256, 128, 8),  # uneven ranges
])
@pytest.mark.parametrize("M", [33, 48, 49, 64])
def test_mid_kernel_edges(sba, gpu, M, K, N, G, split):
    """The one-pass kernel of 33 .. 64 rows (development variant bit 1 << 28 takes it on layers of any
    size), with and without a K split, against the oracle; the result with a K split does not depend
    on the workspace's contents."""
    from server_benchmark_amd import _lib
    x, qw, s, qz = _np_case(M, K, N, G if G > 0 else K, seed=K + M)
    sba.ops.get_workspace(gpu, 32 << 20)     # room for the partial tiles of any split here
    y = _check_gemm(sba, gpu, x, qw, s, qz, G if G > 0 else K, split, tag="one-pass", variant=1 << 28)
    assert _lib.load().awqmi_dev_last_gemm_form() == _lib.FORM_MID
    sba.ops.get_workspace(gpu, 32 << 20)[65536:].fill_(255)
    y2 = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), force_split_k=split, _dev_variant=1 << 28)
    assert np.array_equal(y2.cpu().numpy(), y)


@pytest.mark.parametrize("M,K,N,G,split", [(33, 768, 528, 64, 3), (64, 1024, 1040, 256, 2), (48, 2048, 512, 32, 4),
                                           (49, 128 * 41, 256, 128, 8)])
def test_mid_kernel_split_writes_its_partial_tiles(sba, gpu, M, K, N, G, split):
    """A K split of the one-pass kernel takes place: the partial tiles of every part, column block and
    16-row block in use are written, those behind them are not."""
    x, qw, s, qz = _np_case(M, K, N, G, seed=K + M)
    ws = sba.ops.get_workspace(gpu, 32 << 20)
    ws[65536:].fill_(255)                    # a NaN in every fp32 value
    _check_gemm(sba, gpu, x, qw, s, qz, G, split, tag="one-pass split", variant=1 << 28)
    ncb, mb = (N + 255) // 256, (M + 15) // 16
    part = ws[65536:].view(torch.float32)[:(split + 1) * ncb * 64 * 256].view(split + 1, ncb, 4, 16 * 256)
    assert torch.isfinite(part[:split, :, :mb]).all()
    assert torch.isnan(part[:split, :, mb:]).all() and torch.isnan(part[split]).all()


@pytest.mark.parametrize("M,K,N,pad,mid", [(64, 5120, 8192, True, False), (33, 5120, 8192, False, False), (48, 16384, 2560, False, False),
                                           (64, 8192, 40960, True, True), (33, 32768, 10240, False, True)])
def test_mid_kernel_by_default_on_large_layers(sba, gpu, M, K, N, pad, mid):
    """The largest layers take the one-pass kernel at 33 .. 64 rows, others one row of tiles, with padded rows of qweight too;
    without room for the partial tiles of a K split both run unsplit."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    form = _lib.FORM_MID if mid else _lib.FORM_FUSED
    g = torch.Generator(device=gpu).manual_seed(M)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    q, qz = words(K, N // 8), words(K // 128, N // 8)
    s = (torch.rand((K // 128, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    qw = sba.ops.pad_qweight_rows(q) if pad else q
    y = sba.awq_gemm(x, qw, s, qz, 0)
    assert lib.awqmi_dev_last_gemm_form() == form
    ref = x.float() @ sba.awq_dequantize(q, s, qz, 0, 0, 0).float()
    assert float((y.float() - ref).norm() / ref.norm()) <= TOL
    small = torch.zeros(65536, dtype=torch.uint8, device=gpu)
    y1 = torch.empty_like(y)
    st = lib.awqmi_gemm_f16(x.data_ptr(), q.data_ptr(), s.data_ptr(), qz.data_ptr(), y1.data_ptr(),
                            small.data_ptr(), small.numel(), M, K, N, 128, 0, torch.cuda.current_stream().cuda_stream)
    assert st == 0 and lib.awqmi_dev_last_gemm_form() == form
    assert float((y1.float() - ref).norm() / ref.norm()) <= TOL


@pytest.mark.parametrize("M,K,N,G,mid", [
    (64, 768, 58368, 128, False),
    (33, 1920, 24576, 64, False),
    (64, 4096, 12288, 128, False),
    (64, 4096, 12288, 64, False),
    (64, 4096, 12288, 32, False),
    (33, 4096, 12288, 32, False),
    (64, 4096, 20480, 32, False),
    (64, 3584, 12288, 128, False),
    (64, 4096, 11776, 128, False),
    (40, 4096, 22272, 64, False),
    (40, 4096, 22784, 64, False),
    (64, 4096, 22784, 64, False),
    (64, 4096, 24832, 64, False),
    (40, 4096, 28432, 128, False),
    (40, 4096, 28944, 128, False),
    (40, 5120, 20736, 128, False),
    (40, 2560, 29184, 128, False),
    (40, 2560, 33024, 128, False),
    (48, 10880, 4112, 32, False),
    (48, 11008, 4112, 32, False),
    (64, 8064, 5376, 128, False),
    (64, 8320, 5120, 128, False),
    (64, 13184, 5632, 128, False),
    (64, 13312, 5632, 128, False),
    (64, 13312, 5648, 128, False),
    (64, 16384, 5648, 128, False),
    # both sides of 320 Mi weights, of whole 16 columns and 128 rows, of 256 column blocks and their multiples
    (33, 8192, 40960, 128, True),
    (64, 8192, 40960, 64, True),
    (49, 8192, 40960, 32, True),
    (64, 8192, 40944, 128, False),
    (65, 8192, 40960, 128, False),
    (48, 65536, 5120, 32, True),
    (40, 2560, 131072, 64, True),
    (40, 1920, 196608, 128, False),
    (40, 4096, 82176, 128, False),
    (64, 8192, 40968, 128, False),
    (40, 8256, 40960, 64, False),
])
def test_one_pass_kernel_rule(sba, gpu, M, K, N, G, mid):
    """Which layers take the one-pass kernel at 33 .. 64 rows, on both sides of every line of the rule (the first ones, of up to
    113 Mi weights, are on both sides of where it stopped beating an earlier tile kernel), and their products against the
    dequantised weights."""
    from server_benchmark_amd import _lib
    g = torch.Generator(device=gpu).manual_seed(K + N)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    qw, qz = words(K, N // 8), words(K // G, N // 8)
    s = (torch.rand((K // G, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    y = sba.awq_gemm(x, qw, s, qz, 0)
    assert _lib.load().awqmi_dev_last_gemm_form() == (_lib.FORM_MID if mid else _lib.FORM_FUSED)
    ref = x.float() @ sba.awq_dequantize(qw, s, qz, 0, 0, 0).float()
    assert float((y.float() - ref).norm() / ref.norm()) <= TOL


@pytest.mark.parametrize("split", [1, 8, 64])
@pytest.mark.parametrize("M,K,N,mid", [(64, 5120, 8192, False), (64, 8192, 40960, True), (64, 32768, 10240, True)])
def test_one_pass_kernel_ignores_split_k(sba, gpu, M, K, N, mid, split):
    """More than 32 rows ignore split_k, with a workspace and without one of the caller's: the same bits
    from the same kernel as the library's own choice (64 partial tiles a column block would not fit the
    static scratch array, and a split of 1 would leave most of the chip idle)."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    form = _lib.FORM_MID if mid else _lib.FORM_FUSED
    g = torch.Generator(device=gpu).manual_seed(1)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    qw, qz = words(K, N // 8), words(K // 128, N // 8)
    s = (torch.rand((K // 128, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    y = sba.awq_gemm(x, qw, s, qz, 0)
    assert lib.awqmi_dev_last_gemm_form() == form
    y1 = sba.awq_gemm(x, qw, s, qz, 0, force_split_k=split)
    y2 = sba.ops.awq_gemm_noalloc(x, qw, s, qz, torch.empty_like(y), force_split_k=split)
    assert lib.awqmi_dev_last_gemm_form() == form
    assert torch.equal(y, y1) and torch.equal(y, y2)


@pytest.mark.parametrize("M", [32, 33, 48, 64])
def test_gemm_wide_layer_mid_m(sba, gpu, M):
    """More than 128 column tiles: 32, 48 and 64 rows run as one row of tiles of their height, unsplit."""
    x, qw, s, qz = _np_case(M, 256, 32768 + 512, 128, seed=M)
    _check_gemm(sba, gpu, x, qw, s, qz, 128, 0, tag="wide-mid-M")


def test_gemm_one_hot_is_exact_and_zero_weights(sba, gpu):
    K, N, G = 512, 256, 128
    _, qw, s, qz = _np_case(1, K, N, G, seed=77)
    W = awq_ref.dequantize(qw, s, qz, G)
    rows = [0, 1, 127, 128, 300, 511, 37, 64, 200, 255, 256, 383, 384, 385, 450, 9]
    x = np.zeros((16, K), np.float16)
    for m, k in enumerate(rows):
        x[m, k] = 1
    for split in (1, 4):
        y = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), force_split_k=split).cpu().numpy()
        for m, k in enumerate(rows):
            assert np.array_equal(y[m].view(np.uint16), W[k].view(np.uint16)), (split, m, k)
    # w == z everywhere: the reference gives exact zeros.  The skinny kernel sums x * w on the
    # matrix core and subtracts z * sum(x) through a separate MFMA, so what is left is fp32
    # cancellation noise: bound it by 2^-18 of the magnitude a full-scale weight would give
    # (|x|_1 * 15 * s_max), four orders of magnitude inside the 2e-3 tolerance.
    zfull = np.repeat(awq_ref.unpack_awq(qz), G, axis=0)
    xr = np.random.default_rng(0).normal(0, 1, (16, K)).astype(np.float16)
    y = sba.awq_gemm(*_dev(gpu, xr, awq_ref.pack_awq(zfull), s, qz), 0).cpu().numpy()
    bound = np.abs(xr.astype(np.float64)).sum(axis=1, keepdims=True) * 15 * float(s.max()) * 2.0 ** -18
    print(f"[w == z] max |y| = {np.abs(y).max():.3e}, bound {bound.min():.3e}", flush=True)
    assert np.all(np.abs(y.astype(np.float64)) <= bound)
    # the tile kernel unpacks to exact fp16 zeros first: exact zeros there
    xl = np.random.default_rng(1).normal(0, 1, (80, K)).astype(np.float16)
    assert not sba.awq_gemm(*_dev(gpu, xl, awq_ref.pack_awq(zfull), s, qz), 0).cpu().numpy().any()


@pytest.mark.parametrize("K,N,G,M", [(4096, 256, -1, 5), (4096, 512, 128, 16), (1024, 264, 1024, 3), (2048, 256, 256, 32)])
def test_gemm_decode_large_mean_and_outlier_activations(sba, gpu, K, N, G, M):
    """The skinny kernel takes the zero point out through a lane's running sum of x fed to the
    matrix core as fp16 pieces: activations with a large mean (sums of tens of thousands per lane
    and group, more with one group over all of K) or massive outliers must neither overflow that
    sum nor cost accuracy.  Checked against the float64 product with a max-abs bound next to the
    relative Frobenius one."""
    rng = np.random.default_rng(K + N + M)
    g = K if G <= 0 else G
    w = rng.integers(0, 16, (K, N))
    z = rng.integers(0, 16, (K // g, N))
    s = (rng.random((K // g, N)) * 0.019 + 0.001).astype(np.float16)
    qw, qz = awq_ref.pack_awq(w), awq_ref.pack_awq(z)
    cases = {
        "mean 100": rng.normal(100.0, 1.0, (M, K)),
        "mean -3000": rng.normal(-3000.0, 10.0, (M, K)),
        "outliers": rng.normal(0.0, 1.0, (M, K)),
    }
    cases["outliers"][:, rng.integers(0, K, 6)] = 30000.0
    cases["outliers"][:, rng.integers(0, K, 6)] = -28000.0
    for name, x in cases.items():
        x = x.astype(np.float16)
        ref = awq_ref.gemm_wide(x, qw, s, qz, g)
        if np.abs(ref).max() >= 60000:      # keep the true result inside fp16
            x = (x.astype(np.float32) * (30000.0 / np.abs(ref).max())).astype(np.float16)
            ref = awq_ref.gemm_wide(x, qw, s, qz, g)
        y = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0).cpu().numpy().astype(np.float64)
        assert np.isfinite(y).all(), name
        err = awq_ref.rel_frobenius(y, ref)
        maxabs = float(np.abs(y - ref).max())
        scale = float(np.abs(ref).max())
        print(f"[gemm {name} M={M} K={K} N={N} G={g}] rel_fro={err:.2e} max_abs={maxabs:.3e} of {scale:.3e}", flush=True)
        assert err <= TOL, name
        assert maxabs <= 2e-3 * scale, name


def test_gemm_config0(sba, gpu):
    c = sba.workloads.config0()
    x, qw, s, qz = (t.numpy() for t in (c.x, c.qweight, c.scales, c.qzeros))
    y16 = _check_gemm(sba, gpu, x, qw, s, qz, 128, 0, tag="config0")
    # row 0 alone (M = 1) equals row 0 of the M = 16 run: the kernel does not depend on M
    y1 = sba.awq_gemm(*_dev(gpu, x[:1], qw, s, qz), 0).cpu().numpy()
    assert awq_ref.rel_frobenius(y1[0], y16[0]) < 1e-3
    W = sba.awq_dequantize(*_dev(gpu, qw, s, qz)).cpu().numpy()
    assert np.array_equal(W.view(np.uint16), awq_ref.dequantize(qw, s, qz, 128).view(np.uint16))


def test_gemm_workspace_counters_stay_zero(sba, gpu):
    from server_benchmark_amd import ops
    x, qw, s, qz = _np_case(16, 1024, 512, 128, seed=3)
    d = _dev(gpu, x, qw, s, qz)
    for _ in range(3):
        sba.awq_gemm(*d, force_split_k=4)
    torch.cuda.synchronize()
    ws = ops.get_workspace(gpu, 1)
    assert int(ws[:65536].view(torch.int32).abs().sum().item()) == 0


def test_split_k_exchange_is_stable_over_many_launches_and_two_streams(sba, gpu):
    """The split-K hand-off (partial tiles + arrival counters in the workspace) over a few thousand
    launches: shapes alternate on one stream and share its workspace, a second stream with a
    workspace of its own runs the same calls at the same time, and every result must carry the bits
    of the first one."""
    cases = []
    for M, K, N, seed in ((16, 4096, 2048, 1), (1, 8192, 1024, 2), (7, 2048, 264, 3), (32, 4096, 512, 4)):
        x, qw, s, qz = _np_case(M, K, N, 128, seed=seed)
        cases.append(_dev(gpu, x, qw, s, qz))
    first = [sba.awq_gemm(*c, 0).clone() for c in cases]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    outs = {0: [], 1: []}
    for it in range(400):
        for i, c in enumerate(cases):
            outs[0].append((i, sba.awq_gemm(*c, 0)))
            with torch.cuda.stream(side):
                outs[1].append((i, sba.awq_gemm(*c, 0)))
        if it % 50 == 49:               # compare in batches, so that launches queue up back to back
            torch.cuda.synchronize()
            for k in (0, 1):
                for i, y in outs[k]:
                    assert torch.equal(y, first[i]), (it, k, i)
                outs[k].clear()
    torch.cuda.synchronize()


def test_workspace_reset_zeroes_the_counters(sba, gpu):
    """A workspace whose counters were left non-zero (a call cut short) gives wrong split-K sums
    until it is reset; awqmi_workspace_reset puts it back."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    x, qw, s, qz = _np_case(16, 1024, 512, 128, seed=4)
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    nbytes = lib.awqmi_gemm_workspace_bytes(16, 1024, 512, 4)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=gpu)
    y = torch.empty((16, 512), dtype=torch.float16, device=gpu)
    st = torch.cuda.current_stream().cuda_stream

    def call():
        rc = lib.awqmi_gemm_f16(xd.data_ptr(), qwd.data_ptr(), sd.data_ptr(), qzd.data_ptr(), y.data_ptr(),
                                ws.data_ptr(), ws.numel(), 16, 1024, 512, 128, 4, st)
        assert rc == 0
        torch.cuda.synchronize()
        return y.clone()

    good = call()
    ws[:65536].view(torch.int32).fill_(-7)      # what a launch that died half-way could leave behind
    assert lib.awqmi_workspace_reset(ws.data_ptr(), ws.numel(), st) == 0
    torch.cuda.synchronize()
    assert int(ws[:65536].view(torch.int32).abs().sum().item()) == 0
    assert torch.equal(call(), good)


# ------------------------------------------------------------------ prefill GEMM (M > 16) and fallback

@pytest.mark.parametrize("M,K,N,G", [(17, 256, 256, 128), (64, 512, 512, 128), (300, 1024, 520, 128),
                                     (512, 2048, 1024, 128), (257, 192, 264, 32), (40, 256, 128, 64),
                                     (33, 384, 256, -1)])
def test_gemm_prefill(sba, gpu, M, K, N, G):
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + K)
    _check_gemm(sba, gpu, x, qw, s, qz, K if G <= 0 else G, 0, tag="prefill")


@pytest.mark.parametrize("M,K,N,G", [(65, 512, 512, 128), (100, 1024, 520, 128), (128, 2048, 1024, 128),
                                     (96, 192, 264, 32), (127, 384, 256, -1), (128, 1024, 8192 + 256, 128),
                                     (129, 512, 512, 128), (160, 1024, 520, 64), (192, 2048, 1024, 128),
                                     (190, 512, 8192 + 256, 128)])
def test_gemm_half_tile(sba, gpu, M, K, N, G):
    """65 .. 192 rows on the tiles that the library picks (ragged rows / columns, K split included);
    two runs agree bit for bit."""
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + K + 1)
    g = K if G <= 0 else G
    y1 = _check_gemm(sba, gpu, x, qw, s, qz, g, 0, tag="half-tile")
    y2 = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0).cpu().numpy()
    assert np.array_equal(y1.view(np.uint16), y2.view(np.uint16))


@pytest.mark.parametrize("M,K,N,G,rows", [(257, 2048, 520, 128, None), (320, 1024, 2560, 128, None),
                                          (384, 512, 10240, 64, None), (640, 1024, 1280, 128, None),
                                          (700, 256, 264, 32, None),
                                          (300, 1024, 1032, 128, 64), (300, 1024, 1032, 128, 128),
                                          (500, 1024, 1032, 128, 192), (100, 1024, 1032, 128, 256)])
def test_gemm_several_row_tiles_of_every_size(sba, gpu, M, K, N, G, rows):
    """Mid-sized batches: the library picks the height of the tiles per launch and runs
    several row tiles of it (ragged last tile, ragged columns, K split of the last round);
    rows forces a height through the development entry point."""
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + N)
    variant = None if rows is None else (rows // 64) << 20
    y1 = _check_gemm(sba, gpu, x, qw, s, qz, G, 0, tag=f"row-tiles {rows}", variant=variant)
    y2 = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0, _dev_variant=variant).cpu().numpy()
    assert np.array_equal(y1.view(np.uint16), y2.view(np.uint16))


# fused tiles of every height: variant -> rows
TILE_HEIGHTS = {1 << 20: 64, 5 << 20: 80, 6 << 20: 96, 7 << 20: 112, 2 << 20: 128, 1 << 29: 160, 3 << 20: 192,
                2 << 29: 208, 3 << 29: 224, 4 << 20: 256}


@pytest.mark.parametrize("K,N,G", [
    (64, 256, 64),            # one stage
    (128, 8, 8),              # one word, eight groups a stage
    (192, 264, 32),           # an odd number of stages, a ragged column tile, two groups a stage
    (320, 288, 16),           # four groups a stage
    (448, 544, 64),           # whole 32 columns, seven stages
    (1152, 1000, 128),        # K split, ragged columns
    (1600, 512, -1),          # one group over an odd number of stages
    (2304, 256, 192),         # three stages a group
])
@pytest.mark.parametrize("variant", TILE_HEIGHTS)
def test_fused_tile_heights(sba, gpu, variant, K, N, G):
    """Every height of the fused kernel's tile, full and with a ragged last tile, against the oracle; without room
    for the partial tiles of a K split it runs unsplit."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    rows, g = TILE_HEIGHTS[variant], K if G <= 0 else G
    # two workspaces: room for every split, and none
    sba.ops.get_workspace(gpu, 80 << 20)[65536:].fill_(255)
    for M in (rows, rows + 17 if rows > 64 else 81):
        x, qw, s, qz = _np_case(M, K, N, g, seed=K + M)
        y = _check_gemm(sba, gpu, x, qw, s, qz, g, 0, tag=f"tile {rows}", variant=variant | (1 << 25))
        assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
        xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
        y1 = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
        assert lib.awqmi_dev_gemm_f16(xd.data_ptr(), qwd.data_ptr(), sd.data_ptr(), qzd.data_ptr(), y1.data_ptr(), 0, 0, M, K, N, g,
                                      0, torch.cuda.current_stream().cuda_stream, variant | (1 << 25)) == 0
        assert awq_ref.rel_frobenius(y1.cpu().numpy(), y) <= TOL


@pytest.mark.parametrize("M", [33, 47, 48, 49])
@pytest.mark.parametrize("K,N,G", [(64, 256, 64), (128, 8, 8), (192, 264, 32), (320, 288, 16), (448, 544, 64), (1152, 1000, 128),
                                   (1600, 512, -1), (2304, 256, 192), (4096, 4112, 128)])
def test_fused_tile_of_48_rows(sba, gpu, M, K, N, G):
    """33 .. 48 rows run on a tile of 48, with a K split and (no workspace) without."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    g = K if G <= 0 else G
    sba.ops.get_workspace(gpu, 80 << 20)[65536:].fill_(255)
    x, qw, s, qz = _np_case(M, K, N, g, seed=K + M)
    y = _check_gemm(sba, gpu, x, qw, s, qz, g, 0, tag="tile 48")
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    y1 = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
    assert lib.awqmi_gemm_f16(xd.data_ptr(), qwd.data_ptr(), sd.data_ptr(), qzd.data_ptr(), y1.data_ptr(), 0, 0, M, K, N, g, 0,
                              torch.cuda.current_stream().cuda_stream) == 0
    assert awq_ref.rel_frobenius(y1.cpu().numpy(), y) <= TOL


@pytest.mark.parametrize("M", [33, 64, 65, 80, 81, 128, 257])
@pytest.mark.parametrize("N,G", [(264, 8), (264, 16), (264, 32), (256, 32), (264, 64), (264, 128)])
def test_fused_tile_groups_of_a_stage(sba, gpu, N, G, M):
    """The tile kernel's three forms by the groups of a 64-row stage (eight; two, which ragged columns take too) over more stages
    than its ring holds, on tiles of every ring depth: against the oracle, and on one-hot rows the dequantised weights themselves."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    K = 1152
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + G)
    _check_gemm(sba, gpu, x, qw, s, qz, G, 0, tag="groups of a stage")
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
    W = awq_ref.dequantize(qw, s, qz, G)
    for k0 in range(0, K, M):                     # every row of W comes out once: a group misplaced shows
        rows = min(M, K - k0)
        one = np.zeros((M, K), np.float16)
        one[np.arange(rows), k0 + np.arange(rows)] = 1
        y = sba.awq_gemm(*_dev(gpu, one, qw, s, qz), 0).cpu().numpy()
        assert np.array_equal(y[:rows], W[k0:k0 + rows])


@pytest.mark.parametrize("M", [17, 31, 32])
@pytest.mark.parametrize("K,N,G", [(128, 32, 64), (128, 256, 128), (384, 288, 64), (640, 544, 128), (1152, 1024, 128), (1920, 800, 64),
                                   (4096, 4128, 128), (16384, 256, 128)])
def test_fused_tile_of_32_rows(sba, gpu, M, K, N, G):
    """17 .. 32 rows on the tile whose group sums are scaled in fp32: full and ragged column tiles, odd numbers of pairs of
    stages, K splits; as near to the 64-bit product as the skinny kernel, whose launch a set split_k still takes."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    sba.ops.get_workspace(gpu, 80 << 20)[65536:].fill_(255)
    x, qw, s, qz = _np_case(M, K, N, G, seed=K + M)
    y = _check_gemm(sba, gpu, x, qw, s, qz, G, 0, tag="tile 32")
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
    skinny = _check_gemm(sba, gpu, x, qw, s, qz, G, 1, tag="skinny")
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_SKINNY
    W = (awq_ref.unpack_awq(qw).astype(np.float64) - awq_ref.unpack_awq(qz).astype(np.float64).repeat(G, 0)) \
        * s.astype(np.float64).repeat(G, 0)
    exact = x.astype(np.float64) @ W
    # both round once, to fp16: 2 % for the noise of that rounding over the fewest outputs here (17 x 32)
    assert awq_ref.rel_frobenius(y, exact) <= 1.02 * awq_ref.rel_frobenius(skinny, exact)


@pytest.mark.parametrize("M,K,N,G,tile", [
    (16, 1024, 1024, 128, False), (17, 1024, 1024, 128, True), (33, 1024, 1024, 128, True), (24, 1024, 1024, 32, False),
    (24, 1024, 1040, 128, False), (24, 1024, 1024, 256, False), (24, 8192, 16352, 128, True), (24, 8192, 16384, 128, False),
    (24, 8192, 16384, 64, True), (25, 8192, 16384, 128, True), (32, 16384, 16384, 64, False),
])
def test_tile_rule_up_to_32_rows(sba, gpu, M, K, N, G, tile):
    """Which calls of up to 32 rows take the tile, on both sides of every line, and their products."""
    from server_benchmark_amd import _lib
    g = torch.Generator(device=gpu).manual_seed(M + K)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    qw, qz = words(K, N // 8), words(K // G, N // 8)
    s = (torch.rand((K // G, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    y = sba.awq_gemm(x, qw, s, qz, 0)
    assert _lib.load().awqmi_dev_last_gemm_form() == (_lib.FORM_FUSED if tile else _lib.FORM_SKINNY)
    ref = x.float() @ sba.awq_dequantize(qw, s, qz, 0, 0, 0).float()
    assert float((y.float() - ref).norm() / ref.norm()) <= TOL


@pytest.mark.parametrize("M,K,N", [(512, 1024, 1280), (300, 2048, 520), (2048, 512, 5120), (768, 1536, 8192 + 256)])
def test_gemm_prefill_partial_rounds(sba, gpu, M, K, N):
    """Tile counts that are not a multiple of the CU count, ragged last row / column tiles;
    two runs must agree bit for bit."""
    x, qw, s, qz = _np_case(M, K, N, 128, seed=M + N)
    y1 = _check_gemm(sba, gpu, x, qw, s, qz, 128, 0, tag="prefill-rounds")
    y2 = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0).cpu().numpy()
    assert np.array_equal(y1.view(np.uint16), y2.view(np.uint16))      # deterministic


@pytest.mark.parametrize("M,K,N,G", [(300, 1024, 520, 128), (512, 2048, 1024, 128), (257, 192, 264, 32),
                                     (700, 256, 264, 64), (1024, 512, 1280, 128), (2048, 512, 5120, 128),
                                     (768, 1536, 8192 + 256, 128), (1500, 384, 2056, -1), (4100, 320, 776, 64)])
def test_gemm_dequantise_once_form(sba, gpu, M, K, N, G):
    """The many-row form (weights dequantised once into a panel in the workspace, then the dense
    kernel fed by direct-to-LDS loads), forced through the development entry point at small
    shapes: ragged rows and columns, stage counts that are not a multiple of the ring length,
    a K split of a sparse last round, groups of 32 / 64 / 128 / K.  Checked against the oracle, and
    bit for bit against the fused kernel with 256-row tiles (same k-step order, same split)."""
    from server_benchmark_amd import _lib, ops
    lib = _lib.load()
    g = K if G <= 0 else G
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + 3 * N)
    y_dense = _check_gemm(sba, gpu, x, qw, s, qz, g, 0, tag="dense form", variant=ops.DEV_VARIANT_DENSE)
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_DENSE
    y_fused = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0, _dev_variant=ops.DEV_VARIANT_NO_DENSE | (4 << 20)).cpu().numpy()
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
    assert np.array_equal(y_dense.view(np.uint16), y_fused.view(np.uint16))
    y_again = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0, _dev_variant=ops.DEV_VARIANT_DENSE).cpu().numpy()
    assert np.array_equal(y_dense.view(np.uint16), y_again.view(np.uint16))


def test_gemm_dequantise_once_default_rule_and_small_workspace(sba, gpu):
    """Fewer than 512 weight rows, from 2048 rows on a wide layer and from 4096 on a narrow one: the public entry point takes the
    dequantise-once form when the workspace holds the panel (a row-padded qweight included) and the tile kernel when it does
    not; the same bits here, where neither splits K."""
    from server_benchmark_amd import _lib, ops
    lib = _lib.load()
    M, K, N, G = 2048, 256, 1024 * 8, 128
    x, qw, s, qz = _np_case(M, K, N, G, seed=11)
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    y = sba.awq_gemm(xd, qwd, sd, qzd, 0)
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_DENSE
    padded = ops.pad_qweight_rows(qwd)
    assert not padded.is_contiguous()
    y_pad = sba.awq_gemm(xd, padded, sd, qzd, 0)
    assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_DENSE
    assert torch.equal(y, y_pad)
    # a workspace without room for the panel: the same call runs the fused kernel
    small = torch.zeros(lib.awqmi_gemm_workspace_bytes(1024, K, N, 0), dtype=torch.uint8, device=gpu)
    y_small = torch.empty_like(y)
    st = lib.awqmi_gemm_f16(xd.data_ptr(), qwd.data_ptr(), sd.data_ptr(), qzd.data_ptr(), y_small.data_ptr(),
                            small.data_ptr(), small.numel(), M, K, N, G, 0, torch.cuda.current_stream().cuda_stream)
    assert st == 0 and lib.awqmi_dev_last_gemm_form() == _lib.FORM_FUSED
    torch.cuda.synchronize()
    assert torch.equal(y, y_small)
    ref = awq_ref.gemm_wide(x[:64], qw, s, qz, G)
    assert awq_ref.rel_frobenius(y[:64].cpu().numpy(), ref) <= TOL
    # the same row count on a narrow layer (64 tiles of 256 x 256): the tile kernel; from 4096 rows on the form is taken again
    for rows, form in ((2048, _lib.FORM_FUSED), (4096, _lib.FORM_DENSE)):
        xn, qwn, sn, qzn = _np_case(rows, K, 2048, G, seed=12)
        xnd, qwnd, snd, qznd = _dev(gpu, xn, qwn, sn, qzn)
        yn = sba.awq_gemm(xnd, qwnd, snd, qznd, 0)
        assert lib.awqmi_dev_last_gemm_form() == form
        refn = awq_ref.gemm_wide(xn[-64:], qwn, sn, qzn, G)
        assert awq_ref.rel_frobenius(yn[-64:].cpu().numpy(), refn) <= TOL


def test_gemm_dequantise_once_form_replays_from_a_graph(sba, gpu):
    """The many-row form is three plain launches (panel pass, dense kernel, K-split sum) on the
    caller's stream and workspace: captured once, every replay -- with new activations and with
    eager calls of other shapes on the same stream in between -- equals the eager result."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    M, K, N, G = 2304, 320, 1032 * 8, 64          # 9 x 33 tiles: a sparse last round, split in K; ragged N
    x, qw, s, qz = _np_case(M, K, N, G, seed=21)
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        eager = sba.awq_gemm(xd, qwd, sd, qzd, 0)            # sizes this stream's workspace
        assert lib.awqmi_dev_last_gemm_form() == _lib.FORM_DENSE
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            y = sba.awq_gemm(xd, qwd, sd, qzd, 0)
        for rep in range(3):
            if rep:
                xd.copy_(torch.randn((M, K), device=gpu, generator=torch.Generator(device=gpu).manual_seed(rep)).half())
                eager = sba.awq_gemm(xd, qwd, sd, qzd, 0)
            sba.awq_gemm(xd[:5], qwd, sd, qzd, 0)           # a skinny call on the same workspace in between
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager)
    torch.cuda.current_stream().wait_stream(st)
    ref = awq_ref.gemm_wide(xd[:32].cpu().numpy(), qw, s, qz, G)
    assert awq_ref.rel_frobenius(y[:32].cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("M,K,N,dense", [
    (2048, 448, 8192, True), (2048, 512, 8192, False), (4096, 512, 1024, False), (6143, 2048, 520, False),
    (6144, 2048, 520, True), (6144, 1984, 520, False), (2048, 8192, 8192, True), (2049, 8192, 8192, False),
])
def test_dequantise_once_rule(sba, gpu, M, K, N, dense):
    """Which many-row calls take the dequantise-once form, on both sides of every line, and their products."""
    from server_benchmark_amd import _lib
    g = torch.Generator(device=gpu).manual_seed(M + K)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    qw, qz = words(K, N // 8), words(K // 64, N // 8)
    s = (torch.rand((K // 64, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    y = sba.awq_gemm(x, qw, s, qz, 0)
    assert _lib.load().awqmi_dev_last_gemm_form() == (_lib.FORM_DENSE if dense else _lib.FORM_FUSED)
    ref = x.float() @ sba.awq_dequantize(qw, s, qz, 0, 0, 0).float()
    assert float((y.float() - ref).norm() / ref.norm()) <= TOL


@pytest.mark.parametrize("M,K,N", [(2048, 13824, 5120), (2048, 16384, 4096), (2048, 8192, 8192), (2048, 448, 2048), (4096, 448, 1024),
                                   (6143, 2048, 520), (6144, 2048, 520), (6144, 1984, 520),
                                   (17, 8192, 5120), (32, 384, 32), (300, 2048, 520), (64, 8192, 1024)])
def test_spare_workspace_changes_nothing(sba, gpu, M, K, N):
    """The workspace of a stream only grows: a call runs the same kernel, bit for bit, in exactly the room that the query
    asks for and in room for any form."""
    from server_benchmark_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device=gpu).manual_seed(M + K)
    words = lambda *shape: torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=gpu, generator=g)
    qw, qz = words(K, N // 8), words(K // 64, N // 8)
    s = (torch.rand((K // 64, N), device=gpu, generator=g) * 0.019 + 0.001).half()
    x = torch.randn((M, K), device=gpu, generator=g).half()
    got = []
    need = lib.awqmi_gemm_workspace_bytes(M, K, N, 0)
    for nbytes in (need, max(need, lib.awqmi_dev_gemm_dense_workspace_bytes(M, K, N)) + (64 << 20)):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=gpu)
        y = torch.empty((M, N), dtype=torch.float16, device=gpu)
        assert lib.awqmi_gemm_f16(x.data_ptr(), qw.data_ptr(), s.data_ptr(), qz.data_ptr(), y.data_ptr(), ws.data_ptr(), ws.numel(),
                                  M, K, N, 64, 0, torch.cuda.current_stream().cuda_stream) == 0
        got.append((lib.awqmi_dev_last_gemm_form(), y))
    assert got[0][0] == got[1][0]
    assert torch.equal(got[0][1].view(torch.int16), got[1][1].view(torch.int16))


@pytest.mark.parametrize("M,K,N,G", [(3, 96, 40, 32), (20, 100, 16, 50), (2, 24, 8, 8)])
def test_gemm_generic_fallback(sba, gpu, M, K, N, G):
    x, qw, s, qz = _np_case(M, K, N, G, seed=5)
    _check_gemm(sba, gpu, x, qw, s, qz, G, 0, tag="generic")


def test_more_rows_than_one_grid_dimension_holds(sba, gpu):
    """Shapes whose row count exceeds 65535, the limit of a grid's second dimension: the
    dequantize launch (one row per slab when the group size is odd) and the any-shape GEMM
    run as consecutive slabs."""
    _, qw, s, qz = _np_case(1, 70001, 8, 1, seed=11)
    want = awq_ref.dequantize(qw, s, qz, 1)
    got = sba.awq_dequantize(*_dev(gpu, qw, s, qz), 0, 0, 0).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
    x, qw, s, qz = _np_case(70001, 24, 8, 8, seed=12)
    _check_gemm(sba, gpu, x, qw, s, qz, 8, 0, tag="generic-tall")


def test_bad_arguments_raise_without_launch(sba, gpu):
    x, qw, s, qz = _dev(gpu, *_np_case(2, 256, 64, 128, seed=1))
    with pytest.raises(ValueError):
        sba.awq_gemm(x[:, :128].contiguous(), qw, s, qz, 0)
    with pytest.raises(ValueError):
        sba.awq_gemm(x.float(), qw, s, qz, 0)
    with pytest.raises(ValueError):
        sba.awq_gemm(x.cpu(), qw, s, qz, 0)
    with pytest.raises(ValueError):
        sba.awq_dequantize(qw, s[:, :32].contiguous(), qz)


def test_linear_method_apply(sba, gpu):
    cfg = sba.AWQConfig.from_config({"w_bit": 4, "q_group_size": 128, "zero_point": True})
    layer = torch.nn.Module()
    m = cfg.get_quant_method(layer, "model.layers.0.mlp.down_proj")
    m.create_weights(layer, 512, [128, 128], 512, 256, torch.float16, device=gpu)
    x, qw, s, qz = _np_case(6, 512, 256, 128, seed=9)
    sd = {"qweight": torch.from_numpy(qw), "qzeros": torch.from_numpy(qz), "scales": torch.from_numpy(s)}
    layer.load_state_dict(sd)
    m.process_weights_after_loading(layer)
    xin = torch.from_numpy(x).to(gpu).reshape(2, 3, 512)
    bias = torch.linspace(-1, 1, 256, dtype=torch.float16, device=gpu)
    y = m.apply(layer, xin, bias)
    assert y.shape == (2, 3, 256)
    ref = awq_ref.gemm_wide(x, qw, s, qz, 128) + bias.cpu().numpy().astype(np.float64)
    assert awq_ref.rel_frobenius(y.reshape(6, 256).cpu().numpy(), ref) <= TOL


def test_gemm_random_shapes_across_dispatch_boundaries(sba, gpu):
    """Seeded random (M, K, N, G) around every boundary of the kernel choice (16 / 32 / 48 / 64 /
    128 / 192 / 256 rows, odd word counts, ragged tiles, K-split on and off), against the oracle."""
    rng = np.random.default_rng(2024)
    ms = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 100, 127, 128, 129, 191, 192, 193, 255, 256, 257, 300]
    worst = 0.0
    for case in range(40):
        M = int(ms[case % len(ms)]) if case < len(ms) else int(rng.integers(1, 320))
        G = int(rng.choice([32, 64, 128, 256]))
        K = int(rng.integers(1, 9)) * 256
        N = int(rng.integers(1, 150)) * 8
        x, qw, s, qz = _np_case(M, K, N, G, seed=1000 + case)
        y = sba.awq_gemm(*_dev(gpu, x, qw, s, qz), 0).cpu().numpy()
        ref = awq_ref.gemm_wide(x, qw, s, qz, G)
        err = awq_ref.rel_frobenius(y, ref)
        assert err <= TOL, f"M={M} K={K} N={N} G={G}: rel_fro={err:.3e}"
        worst = max(worst, err)
    print(f"[random shapes] worst rel_fro={worst:.2e}", flush=True)


def _with_pitch(qw_dev, extra_words):
    """The same qweight as a view of a buffer whose rows are extra_words further apart; the pad
    holds a pattern that would show up in the result if it were ever read."""
    K, NW = qw_dev.shape
    width = (NW + extra_words + 3) // 4 * 4          # a row pitch must keep 16-byte groups whole
    buf = torch.full((K, width), 0x5A5A5A5A, dtype=torch.int32, device=qw_dev.device)
    v = buf[:, :NW]
    v.copy_(qw_dev)
    return v


@pytest.mark.parametrize("M,K,N,G,pitch,split", [
    (1, 1024, 2048, 128, 32, 0), (16, 1024, 2048, 128, 32, 0), (5, 4096, 2048, 128, 32, 3),     # skinny, tail form
    (16, 2048, 264, 64, 4, 0), (3, 512, 136, 256, 12, 2), (7, 256, 8, 32, 36, 0),                 # other groups, one word per lane
    (24, 12288, 512, 128, 32, 4), (32, 3072, 2048, 64, 32, 1),                                   # 32-row passes, LDS ring
    (24, 12288, 512, 128, 32, 0), (48, 1024, 2048, 128, 32, 0),                                  # one row of tiles
    (64, 512, 2048, 128, 32, 0), (100, 1024, 520, 128, 8, 0), (300, 2048, 2048, 128, 32, 0),
    (700, 1024, 2064, 32, 4, 0), (512, 1024, 4096, 128, 32, 0),
    (3, 96, 40, 32, 4, 0), (20, 100, 16, 50, 8, 0)])                                              # generic kernel
def test_qweight_with_a_row_pitch(sba, gpu, M, K, N, G, pitch, split):
    """qweight rows `pitch` words further apart than a row is long (what
    AWQLinearMethod.process_weights_after_loading hands over for rows that are a multiple of 1 KiB):
    awq_gemm on every kernel and awq_dequantize give the bits of the contiguous tensor, and match
    the oracle; the pad is never read."""
    x, qw, s, qz = _np_case(M, K, N, G, seed=M + K + N)
    g = K if G <= 0 else G
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    qwp = _with_pitch(qwd, pitch)
    assert not qwp.is_contiguous() and qwp.stride(0) >= N // 8 + pitch
    y0 = sba.awq_gemm(xd, qwd, sd, qzd, force_split_k=split)
    y1 = sba.awq_gemm(xd, qwp, sd, qzd, force_split_k=split)
    assert torch.equal(y0.view(torch.int16), y1.view(torch.int16))
    ref = awq_ref.gemm_wide(x, qw, s, qz, g)
    assert awq_ref.rel_frobenius(y1.cpu().numpy(), ref) <= TOL
    W0 = sba.awq_dequantize(qwd, sd, qzd)
    W1 = sba.awq_dequantize(qwp, sd, qzd)
    assert torch.equal(W0.view(torch.int16), W1.view(torch.int16))
    Wref = awq_ref.dequantize(qw, s, qz, g)
    assert np.array_equal(W1.cpu().numpy().view(np.uint16), Wref.view(np.uint16))


def test_qweight_pitch_is_validated(sba, gpu):
    x, qw, s, qz = _np_case(4, 256, 256, 128, seed=1)
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    bad = torch.zeros((256, 34), dtype=torch.int32, device=gpu)[:, :32]      # pitch not a multiple of 4 words
    with pytest.raises(ValueError):
        sba.awq_gemm(xd, bad, sd, qzd)
    with pytest.raises(ValueError):
        sba.awq_gemm(xd, qwd.t().contiguous().t(), sd, qzd)      # column-major


def test_linear_method_pads_kib_rows_and_matches_contiguous(sba, gpu):
    """A layer whose packed rows are 32 lines: process_weights_after_loading re-pitches qweight,
    apply gives the bits of awq_gemm on the contiguous tensor at decode and prefill sizes."""
    cfg = sba.AWQConfig(4, 128, True)
    m = sba.AWQLinearMethod(cfg)
    layer = torch.nn.Module()
    m.create_weights(layer, 512, [8192], 512, 8192, torch.float16, device=gpu)
    x, qw, s, qz = _np_case(300, 512, 8192, 128, seed=77)
    layer.load_state_dict({"qweight": torch.from_numpy(qw), "qzeros": torch.from_numpy(qz),
                           "scales": torch.from_numpy(s)})
    m.process_weights_after_loading(layer)
    assert layer.qweight.stride() == (1056, 1)
    xd, qwd, sd, qzd = _dev(gpu, x, qw, s, qz)
    for rows in (1, 16, 40, 300):
        y = m.apply(layer, xd[:rows].contiguous())
        y0 = sba.awq_gemm(xd[:rows].contiguous(), qwd, sd, qzd)
        assert torch.equal(y.view(torch.int16), y0.view(torch.int16))
