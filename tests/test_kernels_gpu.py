"""Parity of every HIP kernel (through the C ABI) with the CPU oracle on identical seeded inputs.

Tolerances (relative Frobenius error): Kronecker factors 1e-5 for fp32 inputs, 5e-3 for bf16 inputs
(the oracle is fed the same bf16-rounded values upcast to fp32; fp32 accumulation leaves only
summation-order differences, so the bf16 cases are in fact held to 1e-5 as well); damped inverses
1e-4 against the fp32 oracle where the matrix is well conditioned, otherwise both are compared with
an fp64 inverse; preconditioned gradients 1e-3.
"""
import time

import numpy as np

import pytest
import torch
import torch.nn as nn

from oracle import cpu_ref as R

pytestmark = pytest.mark.gpu

TOL_FACTOR_F32 = 1e-5
TOL_FACTOR_BF16 = 5e-3
TOL_INV = 1e-4
TOL_PRECOND = 1e-3


def relerr(a, b):
    a = a.detach().double().cpu()
    b = b.detach().double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


@pytest.fixture(scope='module')
def K():
    from asdl_amd import kernels
    return kernels


def _inputs(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(*shape, generator=g)
    if dtype == torch.bfloat16:
        x = x.to(torch.bfloat16)
    return x


# ------------------------------------------------------------------ syrk_tn (Linear A / B, Shampoo G^T G)
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('M,d', [(128, 784), (128, 512), (128, 10), (1, 5), (37, 129), (1000, 300), (4096, 64),
                                 (70000, 40), (513, 1024)])
def test_syrk_tn_matches_oracle(K, dtype, M, d):
    x = _inputs((M, d), dtype, seed=M * 7 + d)
    ref = R.linear_cov_kron_A(x.float().double())
    print(f'syrk_tn dtype={dtype} M={M} d={d}', flush=True)
    out = K.syrk_tn(x.cuda())
    torch.cuda.synchronize()
    tol = TOL_FACTOR_F32 if dtype == torch.float32 else TOL_FACTOR_BF16
    assert relerr(out, ref) < min(tol, 1e-5)
    assert torch.equal(out, out.T)


def test_syrk_tn_alpha_beta_ema_and_strided_rows(K):
    x = _inputs((300, 200), torch.float32, 3)
    xs = x[:, :150]                                    # ldx = 200 > d = 150
    C0 = _inputs((150, 150), torch.float32, 4)
    C0 = C0 + C0.T
    ref = 0.7 * C0.double() + 0.3 / 64 * R.linear_cov_kron_A(xs.double())
    out = C0.cuda().clone()
    K.syrk_tn(x.cuda()[:, :150], out=out, alpha=0.3 / 64, beta=0.7)
    assert relerr(out, ref) < TOL_FACTOR_F32
    # beta == 0 must not read the destination
    out = torch.full((150, 150), float('nan'), device='cuda')
    K.syrk_tn(x.cuda()[:, :150], out=out, alpha=1.0, beta=0.0)
    assert relerr(out, R.linear_cov_kron_A(xs.double())) < TOL_FACTOR_F32


def test_syrk_tn_3d_input_rows_flatten(K):
    x = _inputs((4, 9, 33), torch.bfloat16, 5)
    ref = R.linear_cov_kron_A(x.float().double())
    out = K.syrk_tn(x.cuda().flatten(end_dim=1))
    assert relerr(out, ref) < 1e-5


def test_cpu_tensor_is_refused(K):
    with pytest.raises(RuntimeError):
        K.syrk_tn(torch.randn(4, 4))


# ------------------------------------------------------------------ conv_syrk (fused unfold)
CONV_CASES = [
    # N, C, H, W, k, s, p
    (2, 5, 4, 4, (2, 2), (1, 1), (0, 0)),          # the reference's test CNN
    (3, 4, 4, 3, (2, 2), (1, 1), (0, 0)),
    (4, 3, 32, 32, (3, 3), (1, 1), (1, 1)),        # CIFAR stem
    (2, 16, 16, 16, (3, 3), (2, 2), (1, 1)),
    (2, 3, 30, 30, (7, 7), (2, 2), (3, 3)),        # ImageNet stem geometry
    (3, 64, 7, 7, (3, 3), (1, 1), (1, 1)),         # 7x7 maps, ragged rows
    (2, 32, 14, 14, (1, 1), (1, 1), (0, 0)),       # 1x1 conv: flattened
    (2, 32, 14, 14, (1, 1), (2, 2), (0, 0)),       # 1x1 stride 2 (downsample)
    (2, 6, 9, 6, (3, 2), (2, 1), (0, 1)),          # asymmetric everything
    (1, 150, 8, 8, (3, 3), (1, 1), (1, 1)),        # d = 1350: many tiles
    (2, 20, 5, 70, (3, 3), (1, 1), (1, 1)),        # W_out > 64: column chunks
    (2, 4, 10, 10, (3, 3), (3, 3), (0, 0)),        # stride 3: generic gather path
]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('case', CONV_CASES, ids=[str(c) for c in CONV_CASES])
def test_conv_syrk_matches_oracle(K, dtype, case):
    N, C, H, W, k, s, p = case
    x = _inputs((N, C, H, W), dtype, seed=N + 10 * C + H)
    ref = R.conv_cov_kron_A(x.float().double(), k, s, p)
    out_size = ((H + 2 * p[0] - k[0]) // s[0] + 1) * ((W + 2 * p[1] - k[1]) // s[1] + 1)
    print(f'conv_syrk dtype={dtype} case={case}', flush=True)
    out = K.conv_syrk(x.cuda(), k, s, p, alpha=1.0 / out_size)
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5
    assert torch.equal(out, out.T)


WINDOW_CASES = [
    # N, C, H, W, kernel, stride, padding: layers with C*kh*kw <= 160, taken by the LDS-window kernel
    (2, 3, 64, 64, (7, 7), (2, 2), (3, 3)),        # ImageNet stem geometry, d = 147 (15 tiles, two per wave)
    (3, 3, 37, 29, (7, 7), (2, 2), (3, 3)),        # odd sizes: last strip shorter than the others
    (2, 40, 9, 9, (2, 2), (1, 1), (0, 0)),         # d = 160: the largest it takes
    (2, 1, 28, 28, (5, 5), (1, 1), (2, 2)),        # one channel, d = 25: one tile, eight position slices
    (2, 7, 12, 10, (3, 3), (1, 1), (1, 1)),        # d = 63: three tiles, two position slices
    (2, 10, 12, 10, (3, 3), (2, 1), (1, 0)),       # d = 90: six tiles
    (2, 13, 8, 8, (3, 3), (1, 1), (1, 1)),         # d = 117: ten tiles, idle waves
    (700, 3, 6, 6, (3, 3), (1, 1), (1, 1)),        # more strips than work groups
    (2, 3, 8, 40, (3, 5), (1, 8), (1, 2)),         # stride wider than the kernel, few output columns
    (1, 2, 5, 3, (5, 3), (1, 1), (0, 0)),          # a single output position
    (2, 3, 224, 224, (7, 7), (2, 2), (3, 3)),      # the ImageNet stem at its size: 112 positions per output row
    (2, 4, 20, 45, (3, 3), (3, 3), (0, 0)),        # stride 3, 15 positions per row: a full and a ragged group of 8
]


@pytest.mark.parametrize('layout', ['nchw', 'channels_last'])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, 'f32_as_bf16'])
@pytest.mark.parametrize('case', WINDOW_CASES, ids=[str(c) for c in WINDOW_CASES])
def test_conv_syrk_window_kernel_matches_oracle(K, dtype, layout, case):
    """fp32 input: fp32 matrix instructions; bf16 input, and fp32 input that the kernel rounds to bf16 as it reads
    it (round_bf16: what the reference's matmul does to it inside a bf16 autocast region), the bf16 ones.  The
    oracle gets the rounded values: the sums are fp32 in every case."""
    N, C, H, W, k, s, p = case
    rounded = dtype == 'f32_as_bf16'
    x = _inputs((N, C, H, W), torch.float32 if rounded else dtype, seed=N + 10 * C + H)
    out_size = ((H + 2 * p[0] - k[0]) // s[0] + 1) * ((W + 2 * p[1] - k[1]) // s[1] + 1)
    seen = x.bfloat16() if rounded else x
    ref = R.conv_cov_kron_A(seen.float().double(), k, s, p) * out_size      # the plain sum over positions
    print(f'conv_syrk window dtype={dtype} layout={layout} case={case}', flush=True)
    xg = x.cuda()
    if layout == 'channels_last':
        xg = xg.contiguous(memory_format=torch.channels_last)
    out = K.conv_syrk(xg, k, s, p, alpha=0.5, round_bf16=rounded)
    torch.cuda.synchronize()
    assert relerr(out, 0.5 * ref) < 1e-5
    assert torch.equal(out, out.T)
    if rounded and N * out_size <= 4096:     # not the statistic of the unrounded input: the rounding is really applied
        assert relerr(out, 0.5 * R.conv_cov_kron_A(x.double(), k, s, p) * out_size) > 1e-5
    # accumulation: out <- beta * out + alpha * stat
    K.conv_syrk(xg, k, s, p, out=out, alpha=0.25, beta=2.0, round_bf16=rounded)
    torch.cuda.synchronize()
    assert relerr(out, 1.25 * ref) < 1e-5
    assert torch.equal(out, out.T)


NHWC_CASES = [
    # N, C, H, W, kernel, stride, padding
    (2, 8, 6, 6, (3, 3), (1, 1), (1, 1)),          # smallest channel count the gather path takes
    (2, 64, 12, 12, (3, 3), (1, 1), (1, 1)),       # d = 576
    (3, 64, 7, 7, (3, 3), (1, 1), (1, 1)),         # 7x7 maps: k-tiles straddle rows and images
    (2, 128, 14, 14, (3, 3), (2, 2), (1, 1)),      # stride 2
    (2, 32, 14, 14, (1, 1), (1, 1), (0, 0)),       # 1x1 conv: plain rows
    (2, 32, 14, 14, (1, 1), (2, 2), (0, 0)),       # 1x1 stride 2 (downsample)
    (2, 16, 9, 6, (3, 2), (2, 1), (0, 1)),         # asymmetric everything
    (1, 152, 8, 8, (3, 3), (1, 1), (1, 1)),        # d = 1368: edge tiles, C not a power of two
    (2, 24, 5, 70, (5, 5), (1, 1), (2, 2)),        # 25 taps
    (5, 40, 33, 35, (3, 3), (1, 1), (1, 1)),       # M = 5775: split-K with a ragged last split
    (2, 176, 12, 12, (3, 3), (1, 1), (1, 1)),      # d = 1584: 256-wide tiles with an edge tile
    (2, 12, 6, 6, (3, 3), (1, 1), (1, 1)),         # C % 8 != 0: falls back to the NCHW kernel
]


@pytest.mark.parametrize('case', NHWC_CASES, ids=[str(c) for c in NHWC_CASES])
def test_conv_syrk_channels_last_matches_oracle(K, case):
    N, C, H, W, k, s, p = case
    x = _inputs((N, C, H, W), torch.bfloat16, seed=N + 10 * C + H)
    ref = R.conv_cov_kron_A(x.float().double(), k, s, p)
    out_size = ((H + 2 * p[0] - k[0]) // s[0] + 1) * ((W + 2 * p[1] - k[1]) // s[1] + 1)
    print(f'conv_syrk channels_last case={case}', flush=True)
    xg = x.cuda().contiguous(memory_format=torch.channels_last)
    out = K.conv_syrk(xg, k, s, p, alpha=1.0 / out_size)
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5
    assert torch.equal(out, out.T)
    # same bits as the NCHW kernel is not required, same statistic is
    out2 = K.conv_syrk(x.cuda(), k, s, p, alpha=1.0 / out_size)
    assert relerr(out, out2.double()) < 1e-5


CORR_CASES = [
    # N, C, H, W: 3 x 3 windows, stride 1, padding 1, a multiple of 64 channels: the shifted-correlation form
    (2, 64, 5, 7),          # 64-wide tiles, one tile per shift
    (3, 128, 8, 8),         # 128-wide tiles
    (2, 256, 4, 6),         # two row tiles of 128
    (2, 512, 7, 7),         # 256-wide tiles of 8 waves
    (1, 64, 1, 1),          # a single pixel: only the centre tap sees it
    (2, 64, 2, 3),          # the first and the last image row are neighbours
    (2, 64, 1, 9),          # one image row: both row corrections remove the same pixels
    (3, 192, 6, 5),         # 64-wide tiles, three per shift
    (16, 64, 28, 28),       # 12544 pixels: row splits; image rows of 14 ... 64 pixels: the main product on windows
    (5, 128, 33, 35),       # windows of 48 + 16 pixels, ragged last split
    (4, 64, 14, 14),        # three image rows per pipeline stage
    (2, 128, 56, 56),       # windows of 64 + 16 pixels
    (3, 64, 3, 16),         # W a multiple of 16: no padding pixels; three image rows per sample
    (1, 192, 17, 64),       # the widest image row the windows take
    (2, 256, 14, 14),       # 32 units of (row channels, column channels)
    (5, 64, 20, 30),        # 100 image rows: splits of unequal length
    (7, 64, 5, 65),         # one pixel too wide for the windows: tiles again
]


@pytest.mark.parametrize('case', CORR_CASES, ids=[str(c) for c in CORR_CASES])
def test_conv_syrk_shifted_correlations_match_oracle(K, case):
    """3 x 3 / stride 1 / padding 1 factors of channels-last bf16 inputs are assembled from 13 shifted correlations of
    the input and 16 border corrections (csrc/conv_corr.hip) instead of the unfolded matrix: same statistic
    (asdl/operations/conv.py:80-88), checked against the oracle's unfolded product in fp64, exact symmetry, and
    accumulation into an existing factor."""
    N, C, H, W = case
    from asdl_amd import _lib
    assert _lib.load().ak_conv_syrk_nhwc_ws_bytes(N, C, H, W, 3, 3, 1, 1, 1, 1) > 0
    x = _inputs((N, C, H, W), torch.bfloat16, seed=N + 10 * C + H)
    ref = R.conv_cov_kron_A(x.float().double(), (3, 3), (1, 1), (1, 1))
    print(f'conv_syrk shifted correlations case={case}', flush=True)
    xg = x.cuda().contiguous(memory_format=torch.channels_last)
    out = K.conv_syrk(xg, (3, 3), (1, 1), (1, 1), alpha=1.0 / (H * W))
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5, relerr(out, ref)
    assert torch.equal(out, out.T)
    # every 9C x 9C block against its own norm: a wrong correction of one border block must not hide in the total
    blocks = (out.double().cpu() - ref).reshape(C, 9, C, 9).permute(1, 3, 0, 2)
    ref_blocks = ref.reshape(C, 9, C, 9).permute(1, 3, 0, 2)
    for t1 in range(9):
        for t2 in range(9):
            if float(ref_blocks[t1, t2].norm()) > 0:
                assert float(blocks[t1, t2].norm() / ref_blocks[t1, t2].norm()) < 1e-5, (t1, t2)
            else:
                assert float(blocks[t1, t2].abs().max()) < 1e-6 * float(ref.abs().max()), (t1, t2)
    K.conv_syrk(xg, (3, 3), (1, 1), (1, 1), out=out, alpha=0.25 / (H * W), beta=2.0)
    torch.cuda.synchronize()
    assert relerr(out, 2.25 * ref) < 1e-5
    assert torch.equal(out, out.T)


CORR_F32_CASES = [(2, 64, 5, 7), (3, 128, 8, 8), (2, 256, 4, 6), (1, 512, 7, 7), (4, 64, 16, 16), (2, 192, 6, 5),
                  (8, 64, 32, 32)]


@pytest.mark.parametrize('case', CORR_F32_CASES, ids=[str(c) for c in CORR_F32_CASES])
def test_conv_syrk_fp32_nchw_shifted_correlations_match_oracle(K, case):
    """fp32 NCHW inputs of 3 x 3 / stride 1 / padding 1 layers: the input is split exactly into three bf16 planes
    (channels-last, 3 C channels), the shifted correlations run on the bf16 matrix cores, and the plane pairs are
    folded before the assembly.  The result has to be the fp32 statistic (asdl/operations/conv.py:80-88) to 1e-5,
    not a bf16-rounded one: inputs with a wide dynamic range inside every patch."""
    N, C, H, W = case
    g = torch.Generator().manual_seed(7 * N + C + H)
    x = torch.randn(N, C, H, W, generator=g) * torch.exp(2 * torch.randn(N, C, H, W, generator=g))
    ref = R.conv_cov_kron_A(x.double(), (3, 3), (1, 1), (1, 1))
    print(f'conv_syrk fp32 nchw shifted correlations case={case}', flush=True)
    xg = x.cuda()
    out = K.conv_syrk(xg, (3, 3), (1, 1), (1, 1), alpha=1.0 / (H * W))
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5, relerr(out, ref)
    assert torch.equal(out, out.T)
    # not the statistic of the bf16-rounded input
    assert relerr(out, R.conv_cov_kron_A(x.bfloat16().double(), (3, 3), (1, 1), (1, 1))) > 1e-4
    K.conv_syrk(xg, (3, 3), (1, 1), (1, 1), out=out, alpha=0.25 / (H * W), beta=2.0)
    torch.cuda.synchronize()
    assert relerr(out, 2.25 * ref) < 1e-5
    assert torch.equal(out, out.T)


@pytest.mark.parametrize('layout', ['nchw', 'channels_last'])
def test_round_bf16_outside_the_window_kernel_is_a_cast(K, layout):
    """round_bf16 for operands the window kernel does not take (many channels, 1x1 windows, plain rows): the wrappers
    cast to bf16 and use the bf16 kernels; the C entry points answer AK_ERR_UNSUPPORTED to AK_F32_AS_BF16 there."""
    import ctypes
    from asdl_amd import _lib
    x = _inputs((2, 32, 10, 10), torch.float32, seed=5)
    xg = x.cuda().contiguous(memory_format=torch.channels_last) if layout == 'channels_last' else x.cuda()
    for k, s, p in (((3, 3), (1, 1), (1, 1)), ((1, 1), (1, 1), (0, 0))):
        ref = R.conv_cov_kron_A(x.bfloat16().double(), k, s, p)
        out_size = ((10 + 2 * p[0] - k[0]) // s[0] + 1) ** 2
        out = K.conv_syrk(xg, k, s, p, alpha=1.0 / out_size, round_bf16=True)
        assert relerr(out, ref) < 1e-5
        assert relerr(out, R.conv_cov_kron_A(x.double(), k, s, p)) > 1e-5
    rows = _inputs((300, 48), torch.float32, seed=6)
    out = K.syrk_tn(rows.cuda(), round_bf16=True)
    assert relerr(out, R.linear_cov_kron_A(rows.bfloat16().double())) < 1e-5
    assert relerr(out, R.linear_cov_kron_A(rows.double())) > 1e-5
    # the C ABI itself: the third dtype code is the window kernel's only
    A = torch.empty(288, 288, device='cuda')
    lib = _lib.load()
    args = (ctypes.c_void_p(xg.data_ptr()), K.AK_F32_AS_BF16, 2, 32, 10, 10, 3, 3, 1, 1, 1, 1, 1.0, 0.0,
            ctypes.c_void_p(A.data_ptr()), 288, ctypes.c_void_p(0), 0, ctypes.c_void_p(0))
    fn = lib.ak_conv_syrk_nhwc if layout == 'channels_last' else lib.ak_conv_syrk
    assert fn(*args) == K.AK_ERR_UNSUPPORTED
    torch.cuda.synchronize()


def test_conv_syrk_channels_last_ema_accumulate(K):
    x = _inputs((4, 16, 10, 10), torch.bfloat16, 1)
    x2 = _inputs((4, 16, 10, 10), torch.bfloat16, 2)
    A0 = R.conv_cov_kron_A(x.float(), (3, 3), (1, 1), (1, 1))
    ref = 0.9 * A0.double() + 0.1 * R.conv_cov_kron_A(x2.float().double(), (3, 3), (1, 1), (1, 1))
    out = A0.cuda().clone()
    K.conv_syrk(x2.cuda().contiguous(memory_format=torch.channels_last), (3, 3), (1, 1), (1, 1), out=out,
                alpha=0.1 / 100, beta=0.9)
    assert relerr(out, ref) < TOL_FACTOR_F32


@pytest.mark.parametrize('C,H', [(64, 14), (16, 12)])     # shifted correlations; the gathered kernel
def test_remembered_direct_launch_repeats_the_factor_call(K, C, H):
    """kernels.DirectCall: a hook remembers the library call its factor function made and repeats it on the tensor
    of the next pass (another address, other values) without going through conv_syrk(): the same factor as a fresh
    call bit for bit, and no launch at all for a tensor that would not give the same call."""
    xs = [_inputs((4, C, H, H), torch.bfloat16, seed).cuda().contiguous(memory_format=torch.channels_last) for seed in (3, 4)]
    out = torch.empty(9 * C, 9 * C, device='cuda')
    K.GroupedCall.begin()
    K.conv_syrk(xs[0], (3, 3), (1, 1), (1, 1), out=out, alpha=0.25, beta=0.0)
    assert K.DirectCall.remember(xs[0].clone(), out, 'same') is None         # not the tensor the call read
    K.GroupedCall.begin()
    K.conv_syrk(xs[0], (3, 3), (1, 1), (1, 1), out=out, alpha=0.25, beta=0.0)
    assert K.DirectCall.remember(xs[0], torch.empty_like(out), 'same') is None      # not the buffer it wrote
    K.GroupedCall.begin()
    K.conv_syrk(xs[0], (3, 3), (1, 1), (1, 1), out=out, alpha=0.25, beta=0.0)
    rec = K.DirectCall.remember(xs[0], out, 'same')
    assert rec is not None and K.DirectCall.remember(xs[0], out, 'same') is None    # a note is taken once
    first = out.clone()
    assert rec.again(xs[1], 'same')
    fresh = K.conv_syrk(xs[1], (3, 3), (1, 1), (1, 1), alpha=0.25)
    assert torch.equal(out, fresh) and not torch.equal(out, first)
    out.fill_(-1.0)
    assert not rec.again(xs[1], 'other')                                       # the caller's own state differs
    assert not rec.again(xs[1][:2], 'same')                                    # another shape
    assert not rec.again(xs[1].float(), 'same')                                # another type
    assert not rec.again(xs[1].contiguous(), 'same')                           # other strides (NCHW)
    assert float(out.min()) == -1.0 and float(out.max()) == -1.0               # none of them launched anything
    assert rec.again(xs[0], 'same') and torch.equal(out, first)


@pytest.mark.parametrize('M,d,ld', [(4096, 64, 64), (20000, 64, 64), (3000, 1000, 1000), (777, 256, 320),
                                    (100000, 128, 128), (33, 2048, 2048), (3000, 1600, 1600), (1500, 2560, 2568)])
def test_syrk_tn_bf16_split_k_and_strided(K, M, d, ld):
    """Shapes that exercise split-K, ragged last splits, edge tiles and a row stride larger than d."""
    x = _inputs((M, ld), torch.bfloat16, seed=M % 97)
    ref = x[:, :d].float().double().T @ x[:, :d].float().double()
    print(f'syrk_tn bf16 M={M} d={d} ld={ld}', flush=True)
    out = K.syrk_tn(x.cuda()[:, :d])
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5
    assert torch.equal(out, out.T)


@pytest.mark.parametrize('N,C,H,k,s,p', [(8, 64, 28, 3, 1, 1),      # G = 32, 9 taps
                                         (8, 24, 28, 3, 1, 1),      # G = C = 24 (not a multiple of 32)
                                         (8, 32, 20, 5, 1, 2),      # 25 taps: four channels per column block
                                         (8, 40, 24, 2, 2, 0),      # 4 taps, G = 40
                                         (16, 8, 40, 5, 1, 2),      # G = 8 (few channels, but more than 160 columns)
                                         (64, 256, 14, 3, 1, 1)])   # 8 channel groups: blocks right of the diagonal
def test_gathered_factor_reduction_pass_variants(K, N, C, H, k, s, p):
    """Split gathered factors end in a reduction pass that permutes the working column order (c/G, tap, c%G) into
    the result order (c, tap), staged through the LDS in blocks of a few channels.  Shapes with different group
    sizes G, tap counts and block counts, all of them split along the rows (their workspace query is non-zero),
    against the fp64 product of the unfolded input; alpha and beta (the EMA form) included."""
    import torch.nn.functional as F
    from asdl_amd import _lib
    assert _lib.load().ak_conv_syrk_nhwc_ws_bytes(N, C, H, H, k, k, s, s, p, p) > 0, 'this case should be split'
    torch.manual_seed(C + k)
    x = torch.randn(N, C, H, H, device='cuda').to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
    d = C * k * k
    u = F.unfold(x.double(), k, padding=p, stride=s).transpose(1, 2).reshape(-1, d)
    old = torch.randn(d, d, device='cuda')
    old = old + old.T
    ref = 0.25 * (u.T @ u) + 0.5 * old.double()
    out = old.clone()
    print(f'gathered reduction N={N} C={C} H={H} k={k} s={s} p={p}', flush=True)
    K.conv_syrk(x, (k, k), (s, s), (p, p), out=out, alpha=0.25, beta=0.5)
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5
    assert torch.equal(out, out.T)


def _group_cases():
    """(kind, args): plain [M, d] operands (with a row stride, ragged sizes, a result with a wide row stride) and
    channels-last convolution inputs (3x3, strided 1x1, 5x5 with padding), small and at the benchmark's sizes."""
    plain = [(64, 128, 128), (777, 264, 264), (333, 1000, 1000), (3000, 64, 64), (4096, 512, 520), (12544, 1024, 1024),
             (3136, 2048, 2048), (50176, 256, 256), (100, 136, 136), (1500, 1600, 1608)]
    conv = [(2, 32, 9, 9, 3, 1, 1), (4, 64, 14, 14, 3, 2, 1), (3, 24, 11, 11, 3, 1, 0), (8, 128, 28, 28, 3, 1, 1),
            (2, 16, 13, 13, 5, 2, 2), (16, 64, 56, 56, 3, 1, 1), (4, 256, 14, 14, 1, 2, 0), (8, 256, 14, 14, 3, 1, 1)]
    return plain, conv


def test_factor_group_matches_the_single_launches_and_fp64(K):
    """kernels.FactorGroup: the factors of many layers in one grouped launch per tile class.  Every result has to
    agree with the fp64 product of the rounded operand to 1e-5 and to be exactly symmetric; alpha / beta (the EMA
    form) and a second contribution to the same result (which forces a flush in between) are covered.  The layers
    that the library computes from shifted correlations are launched at once and checked with the others."""
    import torch.nn.functional as F
    plain, conv = _group_cases()
    torch.manual_seed(3)
    xs, outs, refs = [], [], []
    grp = K.FactorGroup(torch.device('cuda'))
    K._group.active = grp
    try:
        for i, (M, d, ld) in enumerate(plain):
            x = torch.randn(M, ld, device='cuda').to(torch.bfloat16)[:, :d]
            alpha, beta = (0.5, 0.0) if i % 3 else (0.25, 0.75)
            out = torch.full((d, d + 8), 2.0, device='cuda')[:, :d] if i % 4 == 0 else torch.full((d, d), 2.0, device='cuda')
            ref = alpha * (x.double().T @ x.double()) + beta * out.double()
            r = K.syrk_tn(x, out=out, alpha=alpha, beta=beta)
            assert r is out
            xs.append(x); outs.append(out); refs.append(ref)
        for (N, C, H, W, k, s, p) in conv:
            x = torch.randn(N, C, H, W, device='cuda').to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
            d = C * k * k
            u = F.unfold(x.double(), k, padding=p, stride=s).transpose(1, 2).reshape(-1, d)
            out = torch.zeros(d, d, device='cuda')
            K.conv_syrk(x, (k, k), (s, s), (p, p), out=out, alpha=2.0)
            xs.append(x); outs.append(out); refs.append(2.0 * (u.T @ u))
        # 3x3 stride-1 padding-1 layers of whole 64-channel tiles run at once as shifted correlations of the input
        at_once = [c for c in conv if c[4:] == (3, 1, 1) and c[1] % 64 == 0]
        assert len(at_once) == 3
        assert len(grp) == len(plain) + len(conv) - len(at_once), 'every other case should have been taken by the group'
        assert float(outs[1].abs().max()) == 2.0, 'nothing may be written before the flush'
        # a second contribution to the first result: the group has to flush before it takes it
        M, d, _ = plain[0]
        x2 = torch.randn(M, d, device='cuda').to(torch.bfloat16)
        refs[0] = refs[0] + (x2.double().T @ x2.double())
        K.syrk_tn(x2, out=outs[0], alpha=1.0, beta=1.0)
        assert len(grp) == 1
        grp.flush()
        assert len(grp) == 0
    finally:
        K._group.active = None
    torch.cuda.synchronize()
    for i, (out, ref) in enumerate(zip(outs, refs)):
        assert relerr(out, ref) < 1e-5, (i, relerr(out, ref))
        assert torch.equal(out, out.T), i
    # the same calls one by one give the same factors up to the summation order
    for i, (M, d, ld) in enumerate(plain[:4]):
        single = K.syrk_tn(xs[i], alpha=1.0)
        assert single.shape == (d, d)


def test_factor_group_leaves_ineligible_calls_alone(K):
    """fp32 operands, rows that are not 16-byte aligned, the few-channel stem and factors of 3456 columns and more are
    launched at once even while a group is active."""
    grp = K.FactorGroup(torch.device('cuda'))
    K._group.active = grp
    try:
        x = torch.randn(300, 40, device='cuda')
        out = K.syrk_tn(x)
        assert len(grp) == 0 and relerr(out, x.double().T @ x.double()) < 1e-5
        xb = torch.randn(300, 44, device='cuda').to(torch.bfloat16)        # 88-byte rows
        out = K.syrk_tn(xb)
        assert len(grp) == 0 and relerr(out, xb.double().T @ xb.double()) < 1e-5
        stem = torch.randn(2, 3, 32, 32, device='cuda').to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
        K.conv_syrk(stem, (7, 7), (2, 2), (3, 3))
        assert len(grp) == 0
        wide = torch.randn(1, 512, 7, 7, device='cuda').to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
        K.conv_syrk(wide, (3, 3), (1, 1), (1, 1))
        assert len(grp) == 0
    finally:
        K._group.active = None


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('N,C,hw', [(2, 4, (3, 3)), (8, 64, (7, 7)), (4, 130, (14, 14)), (2, 1000, (1, 1)),
                                    (3, 17, (28, 28)), (1, 257, (5, 9))])
def test_conv_B_factor_matches_oracle(K, dtype, N, C, hw):
    g = _inputs((N, C, *hw), dtype, seed=C)
    ref = R.conv_cov_kron_B(g.float().double())
    print(f'conv B dtype={dtype} N={N} C={C} hw={hw}', flush=True)
    out = K.syrk_nt(g.cuda().flatten(start_dim=2))
    torch.cuda.synchronize()
    assert relerr(out, ref) < 1e-5


def test_conv_syrk_ema_accumulate(K):
    x = _inputs((2, 8, 6, 6), torch.float32, 1)
    A0 = R.conv_cov_kron_A(x, (3, 3), (1, 1), (1, 1))
    x2 = _inputs((2, 8, 6, 6), torch.float32, 2)
    ref = 0.9 * A0.double() + 0.1 * R.conv_cov_kron_A(x2.double(), (3, 3), (1, 1), (1, 1))
    out = A0.cuda().clone()
    K.conv_syrk(x2.cuda(), (3, 3), (1, 1), (1, 1), out=out, alpha=0.1 / 36, beta=0.9)
    assert relerr(out, ref) < TOL_FACTOR_F32


# ------------------------------------------------------------------ damping
def test_kron_damping_matches_oracle(K):
    torch.manual_seed(0)
    pairs = []
    for dA, dB in [(6, 3), (200, 17), (5, 5), (4, 4), (3, 2), (1000, 64)]:
        X = torch.randn(2 * dA, dA)
        Y = torch.randn(2 * dB, dB) * 0.1
        pairs.append((X.T @ X, Y.T @ Y))
    pairs[2] = (pairs[2][0], torch.zeros(5, 5))                      # pi = inf
    pairs[3] = (torch.zeros(4, 4), pairs[3][1])                      # pi = 0
    offdiag = torch.zeros(3, 3)
    offdiag[0, 2] = offdiag[2, 0] = 1.0                              # zero diagonal, non-zero matrix
    pairs[4] = (offdiag, pairs[4][1])
    lam, nz = K.kron_damping([a.cuda() for a, _ in pairs], [b.cuda() for _, b in pairs], 1e-3)
    lam, nz = lam.cpu(), nz.cpu()
    for i, (A, B) in enumerate(pairs):
        ra, rb = R.kron_damping(A, B, 1e-3)
        assert abs(float(lam[i, 0]) - ra) <= 1e-5 * abs(ra), (i, lam[i], ra)
        assert abs(float(lam[i, 1]) - rb) <= 1e-5 * abs(rb), (i, lam[i], rb)
        assert bool(nz[i, 0]) == (not bool(torch.all(A == 0)))
        assert bool(nz[i, 1]) == (not bool(torch.all(B == 0)))


# ------------------------------------------------------------------ damped inverse
@pytest.mark.parametrize('d', [1, 2, 10, 63, 64, 65, 128, 147, 200, 512, 576, 1000, 1152])
def test_chol_inv_matches_oracle(K, d):
    g = torch.Generator().manual_seed(d)
    X = torch.randn(2 * d + 3, d, generator=g)
    A = X.T @ X / (2 * d + 3)
    lam = 0.05
    ref32 = R.cholesky_inv(A, lam)
    ref64 = torch.linalg.inv(A.double() + lam * torch.eye(d, dtype=torch.float64))
    print(f'chol_inv d={d}', flush=True)
    Ag = A.cuda()
    out = K.cholesky_inv(Ag, lam)
    torch.cuda.synchronize()
    assert torch.equal(Ag.cpu(), A), 'input must be left unchanged'
    assert relerr(out, ref32) < TOL_INV
    assert relerr(out, ref64) < TOL_INV
    resid = (A.double() + lam * torch.eye(d, dtype=torch.float64)) @ out.double().cpu() - torch.eye(d, dtype=torch.float64)
    assert float(resid.abs().max()) < 1e-4
    assert torch.equal(out, out.T)


def test_chol_inv_rank_deficient_vs_fp64(K):
    # d > M: conditioning, not the algorithm, limits accuracy; both fp32 results are judged against fp64
    g = torch.Generator().manual_seed(11)
    d, M = 384, 96
    X = torch.randn(M, d, generator=g)
    A = X.T @ X / M
    lam = 1e-3
    ref64 = torch.linalg.inv(A.double() + lam * torch.eye(d, dtype=torch.float64))
    e_ref = relerr(R.cholesky_inv(A, lam), ref64)
    e_hip = relerr(K.cholesky_inv(A.cuda(), lam), ref64)
    print(f'rank deficient: oracle fp32 err {e_ref:.3e}, hip err {e_hip:.3e}', flush=True)
    # cond(A + lam I) ~ 1e4: eps * cond ~ 1e-3 is the fp32 floor for any algorithm
    assert e_hip < max(8 * e_ref, 1e-4)


def test_chol_inv_batched_skip_and_info(K):
    g = torch.Generator().manual_seed(5)
    d = 96
    mats = []
    for _ in range(4):
        X = torch.randn(200, d, generator=g)
        mats.append((X.T @ X / 200).cuda())
    mats[2] = -torch.eye(d).cuda()                                   # not positive definite
    lam = torch.tensor([0.1, 0.2, 0.3, 0.4], device='cuda')
    active = torch.tensor([1, 0, 1, 1], dtype=torch.int32, device='cuda')
    outs = [torch.full((d, d), 7.0, device='cuda') for _ in range(4)]
    info = K.chol_inv_batched(mats, outs, lam, active=active).cpu()
    assert info[0] == 0 and info[3] == 0
    assert info[2] == 1                                              # first leading minor fails
    assert torch.all(outs[1] == 7.0)                                 # skipped: untouched
    for b in (0, 3):
        assert relerr(outs[b], R.cholesky_inv(mats[b].cpu(), float(lam[b]))) < TOL_INV
    with pytest.raises(torch.linalg.LinAlgError):
        K.cholesky_inv(mats[2], 0.5)
    # failure in a later block is reported with its global index
    A = torch.eye(100)
    A[70, 70] = -5.0
    info = K.chol_inv_batched([A.cuda()], [torch.empty(100, 100, device='cuda')], torch.zeros(1, device='cuda')).cpu()
    assert int(info[0]) == 71


def _spd(d, seed, rows=None):
    g = torch.Generator().manual_seed(seed)
    rows = 2 * d + 3 if rows is None else rows
    X = torch.randn(rows, d, generator=g)
    return X.T @ X / rows


def test_chol_inv_grouped_mixed_sizes_match_oracle(K):
    # one call for matrices of many sizes (ragged, not multiples of 4, single-leaf and multi-level ones)
    dims = [1, 2, 10, 63, 64, 65, 128, 147, 200, 256, 384, 512, 576, 640, 1000, 1152, 129, 64, 256, 512]
    mats = [_spd(d, 100 + i) for i, d in enumerate(dims)]
    lams = [0.05 + 0.01 * (i % 5) for i in range(len(dims))]
    print(f'chol_inv_grouped dims={dims}', flush=True)
    dev = [m.cuda() for m in mats]
    outs = [torch.full_like(m, 7.0) for m in dev]
    info = K.chol_inv_grouped(dev, outs, torch.tensor(lams, device='cuda'))
    torch.cuda.synchronize()
    assert torch.all(info == 0)
    for A, Ag, out, lam, d in zip(mats, dev, outs, lams, dims):
        assert torch.equal(Ag.cpu(), A), 'input must be left unchanged'
        ref64 = torch.linalg.inv(A.double() + lam * torch.eye(d, dtype=torch.float64))
        assert relerr(out, R.cholesky_inv(A, lam)) < TOL_INV, d
        assert relerr(out, ref64) < TOL_INV, d
        assert torch.equal(out, out.T), d


@pytest.mark.parametrize('d', [3, 15, 16, 17, 31, 33, 48, 100, 127, 129, 260])
def test_chol_inv_at_the_edges_of_the_leaf_tiles(K, d):
    """Diagonal blocks that end inside, at and behind a 16 x 16 tile, both entry points, against fp64; and the first
    non-positive pivot on either side of every tile boundary of the block."""
    A, lam = _spd(d, 300 + d), 0.05
    ref = torch.linalg.inv(A.double() + lam * torch.eye(d, dtype=torch.float64))
    lam_dev = torch.tensor([lam], device='cuda')
    for call in (K.chol_inv_batched, K.chol_inv_grouped):
        out = torch.empty(d, d, device='cuda')
        assert int(call([A.cuda()], [out], lam_dev).cpu()) == 0
        assert relerr(out, ref) < 2e-6, (call.__name__, relerr(out, ref))
        for bad in sorted({1, 4, 5, 16, 17, d} & set(range(1, d + 1))):
            B = A.clone()
            B[bad - 1, bad - 1] = -5.0
            assert int(call([B.cuda()], [out], lam_dev).cpu()) == bad, (call.__name__, bad)


@pytest.mark.parametrize('dims', [(127, 255, 2), (129, 257, 1), (383, 384, 385), (1151, 513, 640, 10), (2049, 127), (2700, 2700), (3073,)])
def test_chol_inv_grouped_block_sweep_edges(K, dims):
    """Groups of matrices that end just before, at and behind a block of 128 columns and leave the sweep at different
    steps; the last three need more tiles than the device has CUs.  Against fp64, full-rank and rank-deficient."""
    for rank in (2, 1 / 8):
        mats = [_spd(d, 900 + i, rows=max(1, int(rank * d))) for i, d in enumerate(dims)]
        lam = [0.05 * float(m.diagonal().max()) for m in mats]
        outs = [torch.empty(d, d, device='cuda') for d in dims]
        info = K.chol_inv_grouped([m.cuda() for m in mats], outs, torch.tensor(lam, device='cuda'))
        assert torch.all(info == 0)
        for m, l, out in zip(mats, lam, outs):
            W = m.cuda().double() + l * torch.eye(m.shape[0], device='cuda', dtype=torch.float64)
            assert relerr(out, torch.linalg.inv(W)) < 2e-5, (m.shape, relerr(out, torch.linalg.inv(W)))
            assert torch.equal(out, out.T)


# The chain: groups that end after one, two, three and four blocks and inside one, tiles in the step's launch and (many rows) in
# launches of their own, one matrix and many of other sizes beside it; a skipped matrix and one that is not positive definite.
@pytest.mark.parametrize('dims', [(4225,), (4097, 130, 5), (3500, 2900, 2561), (1100,) * 24 + (3,), (1537,) * 12 + (300,), (641,) * 40, (513,) * 60])
def test_chol_inv_grouped_chain(K, dims):
    plan = K.chol_group_plan(list(dims))
    assert plan.launches != max((d + 127) // 128 for d in dims) + 1, 'the block sweep: one launch per block column'
    print(f'chain {len(dims)} x {dims[0]}', flush=True)
    g = torch.Generator('cuda').manual_seed(len(dims))
    mats = []
    for d in dims:
        x = torch.randn(d + 40, d, device='cuda', generator=g)
        mats.append(x.T @ x / (d + 40))
    lam = torch.full((len(dims),), 1e-2, device='cuda')
    bad, skip = (len(dims) - 2, len(dims) - 1) if len(dims) > 1 else (None, None)
    active = torch.ones(len(dims), dtype=torch.int32, device='cuda')
    if bad is not None:
        mats[bad][100, 100] = -1.0
        mats[bad][0, 1:].fill_(float('nan'))             # above the diagonal: not read
        active[skip] = 0
    outs = [torch.full_like(m, 7.0) for m in mats]
    info = K.chol_inv_grouped(mats, outs, lam, active=active).cpu()
    for i, (a, o) in enumerate(zip(mats, outs)):
        if i == skip:
            assert bool((o == 7.0).all())
        elif i == bad:
            assert int(info[i]) == 101
        else:
            assert int(info[i]) == 0 and torch.equal(o, o.T)
            if i in (0, len(dims) - 3):
                d = a.shape[0]
                full = torch.tril(a.double()) + torch.tril(a.double(), -1).T + 1e-2 * torch.eye(d, device='cuda', dtype=torch.float64)
                inv = o.double()
                for _ in range(2):                       # two Newton steps in 64 bits: the residual to its fourth power
                    residual = 2 * torch.eye(d, device='cuda', dtype=torch.float64) - full @ inv
                    assert float((residual - torch.eye(d, device='cuda', dtype=torch.float64)).norm()) < 0.05
                    inv = inv @ residual
                # rounding 2^-22 of the operands, condition up to 4.2 / 1e-2 (Marchenko-Pastur edge over the damping)
                assert relerr(o, inv) < 420 * 2.0 ** -22, (i, d)


@pytest.mark.parametrize('lam_rel', [1e-2, 1e-6])
@pytest.mark.parametrize('dims', [(4136,), (4136, 2084, 1060), (4700, 4136, 1060, 20), (1064,) * 24, (1092,) * 20 + (552,) * 10, (2100, 2068, 1044) * 4])
def test_chol_inv_grouped_products_beside_the_steps(K, dims, lam_rel):
    """Groups that end inside a block (40 ... 108 columns of 128), matrices that are done before others (their last products go along with
    the others' steps), on fp16 pieces and (a / lam beyond 2^16) on three bf16 pieces: every inverse against 64 bits, to what 22 bits
    and the condition a d / lam allow at most, and the same bits wherever in the group a matrix stands."""
    plan = K.chol_group_plan(list(dims))
    assert plan.launches != max((d + 127) // 128 for d in dims) + 1, 'the block sweep: one launch per block column'
    print(f'chain products {len(dims)} x {dims[0]} {lam_rel}', flush=True)
    g = torch.Generator('cuda').manual_seed(3)
    made = {}
    for d in dims:
        if d not in made:
            x = torch.randn(2 * d, d, device='cuda', generator=g)
            made[d] = x.T @ x / (2 * d)
    mats = [made[d] for d in dims]
    lam = torch.tensor([lam_rel * float(m.diagonal().max()) for m in mats], device='cuda')
    outs = [torch.full_like(m, float('nan')) for m in mats]
    info = K.chol_inv_grouped(mats, outs, lam).cpu()
    assert int(info.abs().max()) == 0
    for d, A in made.items():
        same = [i for i, m in enumerate(mats) if m is A]
        for i in same[1:]:
            assert torch.equal(outs[i], outs[same[0]]), (d, i)
        o = outs[same[0]]
        full = (torch.tril(A).double() + torch.tril(A, -1).double().T + float(lam[same[0]]) * torch.eye(d, device='cuda', dtype=torch.float64)).cpu()
        exact = torch.cholesky_inverse(torch.linalg.cholesky(full))
        assert torch.equal(o, o.T)
        # eigenvalues within (0.29^2 ... 1.71^2) + lam: condition below 35
        assert relerr(o, exact) < 35 * 2.0 ** -22, (d, relerr(o, exact))


@pytest.mark.parametrize('dims', [(4133,), (2051, 2049, 2046, 1409, 1405, 641, 639) * 2, (641,) * 40 + (1023, 1281) * 6])
def test_chol_inv_grouped_takes_the_first_updates_from_the_matrices(K, dims):
    """Groups on the chain, whose first products read the matrices themselves (rows of any length, a last block of one to three columns,
    behind which zeros and a diagonal stand): the same bits from matrices with anything above their diagonals, in memory that ends with
    them, next to one that is left out."""
    plan = K.chol_group_plan(list(dims))
    assert plan.launches != max((d + 127) // 128 for d in dims) + 1, 'the block sweep: one launch per block column'
    g = torch.Generator('cuda').manual_seed(5)
    mats = []
    for d in dims:
        x = torch.randn(2 * d, d, device='cuda', generator=g)
        mats.append(x.T @ x / (2 * d))
    lam = torch.full((len(dims),), 0.03, device='cuda')
    outs, junk = [torch.empty_like(m) for m in mats], [torch.empty_like(m) for m in mats]
    assert int(K.chol_inv_grouped(mats, outs, lam).abs().max()) == 0
    dirty = [torch.tril(m) + torch.triu(torch.full_like(m, float('nan')), 1) for m in mats]
    active = torch.ones(len(dims), dtype=torch.int32, device='cuda')
    if len(dims) > 1:
        active[1] = 0
        junk[1].fill_(7.0)
    K.chol_inv_grouped(dirty, junk, lam, active=active)
    for i, (d, A) in enumerate(zip(dims, mats)):
        if active[i] == 0:
            assert bool((junk[i] == 7).all())
            continue
        assert torch.equal(junk[i], outs[i]), (i, d)
        if i < 8:
            full = torch.tril(A).double() + torch.tril(A, -1).double().T + 0.03 * torch.eye(d, device='cuda', dtype=torch.float64)
            # (A + lam I) X = I up to the condition, below 35, of what 22 bits hold
            assert float((full @ outs[i].double() - torch.eye(d, device='cuda', dtype=torch.float64)).norm()) < 35 * 2.0 ** -22 * d ** 0.5


@pytest.mark.parametrize('case', ['chain', 'chain of many', 'sweep', 'by size', 'low rank', 'low rank one by one'])
def test_sums_of_the_framework_beside_inverses_on_a_side_stream(K, monkeypatch, case):
    """Deferred inverses run on side streams beside whatever the caller enqueues next, the loss backward pass in a step.  Its sums over
    the rows of bf16 matrices, the bias gradients, give the bits that they give alone: 16-bit matrix instructions of another
    kernel on their CUs take values from them."""
    from asdl_amd import symmatrix
    from asdl_amd.symmatrix import Kron, batched_update_inv
    monkeypatch.setattr(symmatrix, 'INLINE_MICROSECONDS', 0)      # (beside the current stream at all sizes)
    monkeypatch.setattr(symmatrix, 'GROUPED_INVERSE', case != 'by size')
    g = torch.Generator('cuda').manual_seed(1)

    def factor(d, rows):
        x = torch.randn(rows, d, device='cuda', generator=g)
        return x if rows < d else x.t() @ x / rows
    sizes = {'chain': [(4096, 5000)] * 2, 'chain of many': [(1100, 1500)] * 24, 'sweep': [(2000, 2500)] * 2, 'by size': [(4096, 5000)] * 2,
             'low rank': [(2304, 128)] * 8, 'low rank one by one': [(4608, 600)] * 4}[case]
    mats = [factor(d, rows) for d, rows in sizes]
    krons = [Kron(mats[i], mats[i + 1]) for i in range(0, len(mats), 2)]
    if case in ('chain', 'chain of many', 'sweep'):
        assert (K.chol_group_plan([d for d, _ in sizes]).launches == max((d + 127) // 128 for d, _ in sizes) + 1) == (case == 'sweep')
    wide = torch.randn(8192, 4096, device='cuda', generator=g).bfloat16()
    low = torch.randn(1024, 3072, device='cuda', generator=g).bfloat16()
    alone = wide.sum(0), low.sum(0)
    for _ in range(10):
        pending = batched_update_inv(krons, 1e-2, defer=True)
        beside = [(wide.sum(0), low.sum(0)) for _ in range(20)]
        pending.finish()
        for got in beside:
            for x, y in zip(got, alone):
                assert torch.equal(x, y), f'{int((x != y).sum())} of {x.numel()} sums differ'


@pytest.mark.parametrize('sizes', [[4096] * 2, [4608, 4608, 2304, 2304, 1152, 1152, 576, 512, 256, 128, 64, 27]])
def test_inverses_on_a_side_stream_beside_products_of_the_framework(K, monkeypatch, sizes):
    """The same the other way round: the inverses have the bits that they have alone, whatever runs beside them."""
    from asdl_amd import symmatrix
    from asdl_amd.symmatrix import Kron, batched_update_inv
    monkeypatch.setattr(symmatrix, 'INLINE_MICROSECONDS', 0)
    g = torch.Generator('cuda').manual_seed(3)
    mats = []
    for d in sizes:
        x = torch.randn(d + 100, d, device='cuda', generator=g).relu()
        mats.append(x.t() @ x / d)
    krons = [Kron(mats[i], mats[i + 1]) for i in range(0, len(mats), 2)]
    batched_update_inv(krons, 1e-3)
    alone = [m.clone() for k in krons for m in (k.A_inv, k.B_inv)]
    wide = torch.randn(4096, 4096, device='cuda', generator=g).bfloat16()
    for i in range(24):
        for k in krons:
            k.A_inv.fill_(float('nan'))
            k.B_inv.fill_(float('nan'))
        pending = batched_update_inv(krons, 1e-3, defer=True)
        for _ in range(8):
            wide @ wide
            wide.float().softmax(1)
        pending.finish()
        for m, (x, y) in enumerate(zip((m for k in krons for m in (k.A_inv, k.B_inv)), alone)):
            assert torch.equal(x, y), f'round {i}, matrix {m}: {int((x != y).sum())} elements differ'


def test_sums_of_the_framework_beside_statistics_on_a_side_stream(K):
    """The same of the factors' products, where they are queued on a side stream."""
    g = torch.Generator('cuda').manual_seed(2)
    rows, wide = torch.randn(8192, 1024, device='cuda', generator=g).bfloat16(), torch.randn(8192, 4096, device='cuda', generator=g).bfloat16()
    alone, factor, out = wide.sum(0), K.syrk_tn(rows), torch.empty(1024, 1024, device='cuda')
    stream = K.FactorStream('cuda')
    for _ in range(10):
        for _ in range(2 * K.FACTOR_STREAM_BATCH):
            stream.run(lambda: K.syrk_tn(rows, out=out), rows, out)
        beside = [wide.sum(0) for _ in range(20)]
        stream.join()
        for got in beside:
            assert torch.equal(got, alone), f'{int((got != alone).sum())} of {got.numel()} sums differ'
        assert torch.equal(out, factor)


def test_chol_inv_grouped_reads_the_lower_triangle_only(K):
    d = 300
    A = _spd(d, 7)
    junk = A.clone()
    junk[torch.triu(torch.ones(d, d, dtype=torch.bool), diagonal=1)] = float('nan')
    out = torch.empty(d, d, device='cuda')
    info = K.chol_inv_grouped([junk.cuda()], [out], torch.tensor([0.1], device='cuda'))
    assert int(info.cpu()[0]) == 0
    assert relerr(out, R.cholesky_inv(A, 0.1)) < TOL_INV


def test_chol_inv_grouped_skip_and_info(K):
    dims = [96, 300, 96, 140, 520]
    mats = [_spd(d, 40 + i).cuda() for i, d in enumerate(dims)]
    mats[2] = -torch.eye(96).cuda()                                  # not positive definite at the first pivot
    bad = torch.eye(520)
    bad[400, 400] = -5.0                                             # fails in a later diagonal block
    mats[4] = bad.cuda()
    lam = torch.tensor([0.1, 0.2, 0.3, 0.4, 0.0], device='cuda')
    active = torch.tensor([1, 0, 1, 1, 1], dtype=torch.int32, device='cuda')
    outs = [torch.full_like(m, 7.0) for m in mats]
    info = K.chol_inv_grouped(mats, outs, lam, active=active).cpu()
    assert info[0] == 0 and info[3] == 0
    assert info[2] == 1 and info[4] == 401
    assert torch.all(outs[1] == 7.0)                                 # skipped: untouched
    for b in (0, 3):
        assert relerr(outs[b], R.cholesky_inv(mats[b].cpu(), float(lam[b]))) < TOL_INV
    # strided lam / flags, and the same call twice (the plan and the workspace are reused)
    lam2 = torch.zeros(5, 2, device='cuda')
    lam2[:, 1] = lam
    info = K.chol_inv_grouped(mats[:2], outs[:2], lam2[:, 1], lam_stride=2).cpu()
    assert info[0] == 0 and info[1] == 0
    assert relerr(outs[1], R.cholesky_inv(mats[1].cpu(), 0.2)) < TOL_INV


@pytest.mark.parametrize('scale,lam_rel', [(1e-8, 1e-2), (1e6, 1e-2), (1.0, 1e-4), (1e-3, 3e-5), (1.0, 1e-6), (3e-5, 1e-8), (1.0, 1e-12), (1e4, 0.0)])
def test_chol_inv_grouped_operand_scaling(K, scale, lam_rel):
    """The products of the grouped inverse run on fp16 pieces of operands scaled by powers of two that come from the
    diagonal maximum and the damping; matrices whose bound a / lam exceeds 2^16 (or lam = 0) keep the bf16 three-piece
    products.  Factors of very different magnitudes (1e-8 ... 1e6) and dampings from 1e-2 down to 1e-12 of the diagonal,
    full-rank and rank-deficient, against fp64: the error has to stay at the level conditioning allows in fp32
    (a few eps * cond), and nothing may overflow."""
    d = 640
    mats, lams = [], []
    for rows, seed in ((2 * d, 1), (d // 4, 2)):                 # full rank; rank 160 of 640
        A = _spd(d, 400 + seed, rows=rows) * scale
        mats.append(A.cuda())
        lams.append(lam_rel * float(A.diagonal().max()))
    lam = torch.tensor(lams, device='cuda')
    outs = [torch.empty_like(m) for m in mats]
    print(f'chol_inv_grouped scaling scale={scale} lam_rel={lam_rel}', flush=True)
    info = K.chol_inv_grouped(mats, outs, lam).cpu()
    eye = torch.eye(d, dtype=torch.float64, device='cuda')
    for i, (A, o) in enumerate(zip(mats, outs)):
        W = A.double() + lams[i] * eye
        ref = torch.linalg.inv(W)
        cond = float(torch.linalg.cond(W))
        try:                                  # what the reference's fp32 Cholesky makes of the same matrix
            e_ref = relerr(R.cholesky_inv(A.cpu(), lams[i]), ref)
        except torch.linalg.LinAlgError:
            e_ref = None
        if e_ref is None or not np.isfinite(e_ref) or e_ref > 1e-2:
            # eps * cond >= 1: beyond what fp32 can factor; LAPACK's unblocked potrf may get through with a result
            # that is wrong in the first digit where the blocked recursion here reports the lost definiteness
            print(f'  matrix {i}: cond {cond:.1e} is out of reach of fp32 (oracle: {e_ref}; info here {int(info[i])})',
                  flush=True)
            continue
        assert int(info[i]) == 0, (i, cond, int(info[i]), e_ref)
        assert torch.isfinite(o).all()
        e = relerr(o, ref)
        print(f'  matrix {i}: cond {cond:.1e}, relative error {e:.1e} (fp32 oracle {e_ref:.1e})', flush=True)
        # Explicit inverses are taken of the 128 x 128 diagonal blocks only (LAPACK solves with the factor itself):
        # measured 1.4-1.7 times the error of potrf + potri on the rank-deficient matrices, 1.3-1.6 on the full-rank
        # ones.  The contract for inverses is 1e-4; beyond the conditioning that allows it, at most twice the oracle.
        assert e < max(1e-4, 2 * e_ref), (i, cond, e, e_ref)


@pytest.mark.parametrize('scale,lam_rel', [(1e-8, 1e-2), (1e6, 1e-2), (1.0, 1e-4), (1e-3, 3e-5), (1.0, 1.4e-5), (1.0, 1e-6), (3e-5, 1e-8), (1.0, 1e-12), (1e4, 0.0)])
def test_chol_inv_grouped_operand_scaling_on_the_chain(K, scale, lam_rel):
    """The same for a group of the chain (csrc/chol_chain.hpp), whose products at the end of four blocks are those on fp16 pieces, or
    on three bf16 pieces where a / lam exceeds 2^16 or lam = 0; 640 columns above are on the block sweep, which has none."""
    d, count = 1100, 24                                          # three groups of blocks: every kind of product, the last ones ragged
    assert K.chol_group_plan([d] * count).launches != (d + 127) // 128 + 1, 'the block sweep: one launch per block column'
    distinct = [_spd(d, 400 + seed, rows=rows) * scale for rows, seed in ((2 * d, 1), (d // 4, 2), (d - 100, 3))]      # full rank; ranks 275, 1000
    lams = [lam_rel * float(A.diagonal().max()) for A in distinct]
    mats = [distinct[i % 3].cuda() for i in range(count)]
    lam = torch.tensor([lams[i % 3] for i in range(count)], device='cuda')
    outs = [torch.empty_like(m) for m in mats]
    print(f'chol_inv_grouped chain scale={scale} lam_rel={lam_rel}', flush=True)
    info = K.chol_inv_grouped(mats, outs, lam).cpu()
    for i, A in enumerate(distinct):
        assert all(int(v) == int(info[i]) for v in info[i::3])
        try:
            ref = torch.linalg.inv(A.cuda().double() + lams[i] * torch.eye(d, dtype=torch.float64, device='cuda'))
            e_ref = relerr(R.cholesky_inv(A, lams[i]), ref)
        except torch.linalg.LinAlgError:
            e_ref = None
        if e_ref is None or not np.isfinite(e_ref) or e_ref > 1e-2:      # beyond what fp32 can factor, as above
            print(f'  matrix {i}: out of reach of fp32 (oracle: {e_ref}; info here {int(info[i])})', flush=True)
            continue
        assert int(info[i]) == 0 and torch.isfinite(outs[i]).all()
        for o in outs[i + 3::3]:
            assert torch.equal(o, outs[i])
        e = relerr(outs[i], ref)
        print(f'  matrix {i}: relative error {e:.1e} (fp32 oracle {e_ref:.1e})', flush=True)
        assert e < max(1e-4, 2 * e_ref), (i, e, e_ref)


@pytest.mark.parametrize('d', [2048, 2304, 4096, 4608])
def test_chol_inv_large_matches_fp32_oracle_and_fp64(K, d):
    # the sizes of the largest ResNet factors: deepest recursion, every level on the split-bf16 tile kernel
    A = _spd(d, d, rows=2 * d)
    lam = 0.05
    eye = torch.eye(d, dtype=torch.float64)
    ref64 = torch.linalg.inv(A.double() + lam * eye)
    ref32 = R.cholesky_inv(A, lam)
    print(f'chol_inv large d={d}', flush=True)
    out_g = torch.empty(d, d, device='cuda')
    info = K.chol_inv_grouped([A.cuda()], [out_g], torch.tensor([lam], device='cuda'))
    out_b = K.cholesky_inv(A.cuda(), lam)
    torch.cuda.synchronize()
    assert int(info.cpu()[0]) == 0
    for name, out in (('grouped', out_g), ('batched', out_b)):
        e32, e64 = relerr(out, ref32), relerr(out, ref64)
        print(f'  {name}: vs fp32 oracle {e32:.2e}, vs fp64 {e64:.2e} (oracle vs fp64 {relerr(ref32, ref64):.2e})', flush=True)
        assert e32 < TOL_INV and e64 < TOL_INV
        assert torch.equal(out, out.T)


@pytest.mark.parametrize('count', [1, 24, 25])
def test_kron_precond_deep_sizes_units_and_fail_word(K, count):
    """Sizes at, below and behind the 64-wide tiles and the 16 rows of a bias work group, more modules than one launch
    takes, unaligned gradients; against fp64.  A fail word that is set leaves everything as it was."""
    g = torch.Generator().manual_seed(3)
    shapes = [(1, 1), (10, 17), (64, 64), (65, 63), (16, 129), (130, 257)]
    scale, mods, units = 0.5, [], []
    for i in range(count):
        dB, dA = shapes[i % len(shapes)]
        flat = torch.randn(dB * dA + 1, generator=g).cuda()
        mods.append((_spd(dB, i).cuda(), _spd(dA, 50 + i).cuda(), flat[1:].view(dB, dA), torch.randn(dB, generator=g).cuda() if i % 2 else None))
        units.append((torch.randn(5 + 256 * (i % 2), 2, 2, generator=g).cuda(), torch.randn(5 + 256 * (i % 2), generator=g).cuda(),
                      torch.randn(5 + 256 * (i % 2), generator=g).cuda()))
    items, unit_items = [], []
    for B, A, w, b in mods:
        items += (B.data_ptr(), A.data_ptr(), w.data_ptr(), 0 if b is None else b.data_ptr(), B.shape[0], A.shape[0])
    for inv, w, b in units:
        unit_items += (inv.data_ptr(), w.data_ptr(), b.data_ptr(), w.numel())
    written = [t for m in mods for t in m[2:] if t is not None] + [t for u in units for t in u[1:]]
    before = [t.clone() for t in written]
    expected = []
    for B, A, w, b in mods:
        expected.append(scale * B.double() @ w.double() @ A.double())
        if b is not None:
            expected.append(scale * B.double() @ b.double())
    for inv, w, b in units:
        v = scale * torch.stack([w, b], 1).double()
        expected += list((inv.double() @ v[:, :, None]).squeeze(2).t())
    words = torch.tensor([0, 1], dtype=torch.int32, device='cuda')
    dev = written[0].device
    assert K.kron_precond_deep(items, unit_items, scale, dev, (words.data_ptr(), words.data_ptr() + 4), only_if_faster=False)
    assert all(torch.equal(a, b) for a, b in zip(written, before))
    assert K.kron_precond_deep(items, unit_items, scale, dev, (words.data_ptr(),), only_if_faster=False)
    for got, want in zip(written, expected):
        assert relerr(got, want) < 2e-6
    big = torch.empty(1, device='cuda').data_ptr()
    assert not K.kron_precond_deep([big, big, big, 0, 8192, 8192], [], 1.0, dev)      # the split products are faster: nothing is launched


@pytest.mark.parametrize('shapes', [[(1, 2)], [(64, 65), (63, 577), (8, 27)], [(65, 512), (128, 513), (129, 1200)], [(16, 40 + i) for i in range(25)]])
def test_smw_inv_grouped_matches_fp64(K, shapes):
    """Tile edges of the Gram matrices and of the results, slices of the long side, more factors than one launch takes."""
    g = torch.Generator().manual_seed(11)
    xs = [torch.randn(n, d, generator=g).cuda() for n, d in shapes]
    lam = torch.rand(len(xs), generator=g).cuda() * 0.2 + 0.05
    outs = [torch.full((d, d), 7.0, device='cuda') for _, d in shapes]
    info = torch.full((len(xs),), -1, dtype=torch.int32, device='cuda')
    K.smw_inv_grouped(xs, [lam.data_ptr() + 4 * i for i in range(len(xs))], outs, info)
    assert torch.all(info == 0)
    for x, l, out in zip(xs, lam.double(), outs):
        n, d = x.shape
        ref = torch.linalg.inv(x.double().t() @ x.double() / n + l * torch.eye(d, device='cuda', dtype=torch.float64))
        assert relerr(out, ref) < 1e-5, ((n, d), relerr(out, ref))
        assert torch.equal(out, out.t())


@pytest.mark.parametrize('warm', [True, False])
def test_grouped_products_in_a_captured_graph(K, warm):
    """Address tables under a stream capture, found (the call ran before) or made inside it: every replay, with other tables made and
    memory reused in between, gives the eager result."""
    g = torch.Generator('cuda').manual_seed(2)
    problems, expected = [], []
    for n in (96, 200):
        A, B = torch.randn(n, 64, device='cuda', generator=g), torch.randn(64, n, device='cuda', generator=g)
        problems.append((A, B, torch.zeros(n, n, device='cuda'), False, False, 1.0))
        expected.append((A.double() @ B.double()).float())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        if warm:
            K.gemm_grouped(problems)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side, capture_error_mode='thread_local'):
            K.gemm_grouped(problems)
    torch.cuda.synchronize()
    K._tables.clear()
    for _ in range(4):
        for i in range(20):
            K.device_ints(tuple(range(i, i + 40)), torch.device('cuda'))
            torch.full((512,), -1, dtype=torch.int64).pin_memory()
        for p in problems:
            p[2].zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for p, want in zip(problems, expected):
            assert relerr(p[2], want) < 1e-5


# ------------------------------------------------------------------ sampling
@pytest.mark.parametrize('shape', [(1, 2), (5, 10), (64, 1000), (3, 1023), (9, 1024), (4, 1025), (2, 3, 5001)])
def test_sample_categorical_draws_what_torch_draws(K, shape):
    """One wave per row, one work group per row, vector and scalar loads: the classes torch draws from the same seed."""
    logits = 3 * torch.randn(shape, device='cuda', generator=torch.Generator('cuda').manual_seed(1))
    torch.manual_seed(5)
    ours = K.sample_categorical(logits)
    torch.manual_seed(5)
    theirs = torch.distributions.Categorical(torch.softmax(logits, -1), validate_args=False).sample()
    assert ours.shape == theirs.shape and torch.equal(ours, theirs)


@pytest.mark.parametrize('offset', [0.0, 1e4, -1e5, 1e6])
@pytest.mark.parametrize('rows,classes', [(20000, 50), (4000, 1027)])
def test_sample_categorical_with_an_offset_of_the_logits(K, offset, rows, classes):
    """An offset that all logits of a row share changes no draw of softmax.  Against the same comparison in 64 bits of the same
    float32 logits and random numbers; only rows whose best two classes are closer than the rounding of the 32-bit terms (log q
    and the differences stay below 64 in size: 4 roundings of 2^-19) may differ."""
    g = torch.Generator('cuda').manual_seed(3)
    logits = 3 * torch.randn(rows, classes, device='cuda', generator=g) + offset
    torch.manual_seed(7)
    ours = K.sample_categorical(logits)
    torch.manual_seed(7)
    q = torch.empty_like(logits).exponential_()
    score = logits.double() - q.double().log()
    best, theirs = score.topk(2, dim=1)
    clear = best[:, 0] - best[:, 1] > 4 * 2 ** -19
    assert int(clear.sum()) > 0.99 * rows
    assert torch.equal(ours[clear], theirs[clear, 0])


def test_sample_categorical_leaves_masked_classes_out(K):
    logits = torch.randn(500, 300, device='cuda', generator=torch.Generator('cuda').manual_seed(1))
    logits[:, ::2] = float('-inf')
    logits[:, 1::4] = torch.finfo(torch.float32).min
    assert torch.all(K.sample_categorical(logits) % 4 == 3)


@pytest.mark.parametrize('classes', [7, 300, 1025, 2052])
@pytest.mark.parametrize('kind', ['nan', 'inf', 'all -inf'])
def test_sample_categorical_refuses_rows_without_a_distribution(K, classes, kind):
    """As torch.multinomial does, wherever in the row and in whichever row the value stands."""
    for at in (0, classes // 2, classes - 1):
        logits = torch.randn(70, classes, device='cuda', generator=torch.Generator('cuda').manual_seed(1))
        if kind == 'all -inf':
            logits[at % 70] = float('-inf')
        else:
            logits[(7 * at) % 70, at] = float(kind)
        with pytest.raises(RuntimeError, match='probability tensor contains'):
            K.sample_categorical(logits)
        targets, drawn = K.sample_categorical(logits, late=True)
        with pytest.raises(RuntimeError, match='probability tensor contains'):
            drawn.check()
        assert int(targets.min()) >= 0 and int(targets.max()) < classes
        assert drawn.check() == []
    K.sample_categorical(torch.zeros(70, classes, device='cuda'))       # the word is clear again


@pytest.mark.parametrize('f', [1, 256, 300])
def test_unit_wise_keep_grouped(K, f):
    """Modules whose blocks are all zero keep their previous inverse or get the identity; the others are left alone."""
    blocks = [torch.rand(f, 2, 2, device='cuda') + torch.eye(2, device='cuda'), torch.zeros(f, 2, 2, device='cuda'),
              torch.zeros(f, 2, 2, device='cuda')]
    previous = [None, torch.rand(f, 2, 2, device='cuda'), None]
    invs, flags = K.unit_wise_inv_grouped(blocks, [0.1] * 3)
    expected = [invs[0].clone(), previous[1], torch.eye(2, device='cuda').expand(f, 2, 2)]
    K.unit_wise_keep_grouped(invs, previous, flags)
    assert all(torch.equal(a, b) for a, b in zip(invs, expected))


# ------------------------------------------------------------------ products
@pytest.mark.parametrize('tA', [False, True])
@pytest.mark.parametrize('tB', [False, True])
@pytest.mark.parametrize('M,N,K_', [(5, 7, 3), (130, 257, 65), (512, 384, 1000)])
def test_gemm_matches_fp64(K, tA, tB, M, N, K_):
    g = torch.Generator().manual_seed(M + N)
    A = torch.randn((K_, M) if tA else (M, K_), generator=g)
    B = torch.randn((N, K_) if tB else (K_, N), generator=g)
    C0 = torch.randn(M, N, generator=g)
    ref = 0.5 * (A.double().T if tA else A.double()) @ (B.double().T if tB else B.double()) - 2.0 * C0.double()
    out = C0.cuda().clone()
    K.gemm(A.cuda(), B.cuda(), out=out, transA=tA, transB=tB, alpha=0.5, beta=-2.0)
    assert relerr(out, ref) < 1e-5


@pytest.mark.parametrize('tA', [False, True])
@pytest.mark.parametrize('tB', [False, True])
@pytest.mark.parametrize('M,N,K_', [(1, 1, 1), (64, 64, 128), (63, 65, 127), (66, 62, 129), (33, 130, 257)])
def test_gemm_at_the_edges_of_the_deep_tiles(K, tA, tB, M, N, K_):
    """Tiles of 64 x 64 and chunks of 128 k that end before, at and behind a boundary; rows of an odd stride (loads of 16
    bytes at 4-byte alignment)."""
    g = torch.Generator().manual_seed(7 * M + N + K_)

    def rows(r, c):
        return torch.randn(r, c + 3, generator=g)[:, 1:1 + c]
    A = rows(K_, M) if tA else rows(M, K_)
    B = rows(N, K_) if tB else rows(K_, N)
    ref = (A.double().T if tA else A.double()) @ (B.double().T if tB else B.double())
    wide = [torch.zeros(t.shape[0], t.shape[1] + 3, device='cuda') for t in (A, B)]
    views = []
    for w, t in zip(wide, (A, B)):
        v = w[:, 1:1 + t.shape[1]]
        v.copy_(t)
        views.append(v)
    assert relerr(K.gemm(views[0], views[1], transA=tA, transB=tB), ref) < 2e-6


@pytest.mark.parametrize('pieces,tol', [(3, 2e-6), (2, 3e-5)])
@pytest.mark.parametrize('tA', [False, True])
@pytest.mark.parametrize('tB', [False, True])
@pytest.mark.parametrize('M,N,K_', [(256, 256, 128), (384, 640, 1000), (1100, 520, 516)])
def test_gemm_split_matches_fp64(K, pieces, tol, tA, tB, M, N, K_):
    """fp32 product on the bf16 matrix cores: 3 pieces have to be as good as the fp32 MFMA kernel."""
    torch.manual_seed(M + N)
    A = torch.randn((K_, M) if tA else (M, K_)) * torch.logspace(-3, 3, K_ if not tA else M)[None, :]
    B = torch.randn((N, K_) if tB else (K_, N))
    ref = (A.T if tA else A).double() @ (B.T if tB else B).double()
    print(f'gemm split pieces={pieces} tA={tA} tB={tB} M={M} N={N} K={K_}', flush=True)
    out = K.gemm(A.cuda(), B.cuda(), transA=tA, transB=tB, pieces=pieces)
    out32 = K.gemm(A.cuda(), B.cuda(), transA=tA, transB=tB)
    torch.cuda.synchronize()
    e, e32 = relerr(out, ref), relerr(out32, ref)
    assert e < tol, (e, e32)
    if pieces == 3:
        assert e < 4 * e32 + 1e-7, (e, e32)
    # accumulate form
    C0 = torch.randn(M, N)
    out2 = K.gemm(A.cuda(), B.cuda(), out=C0.cuda().clone(), transA=tA, transB=tB, alpha=0.5, beta=-2.0, pieces=pieces)
    assert relerr(out2, 0.5 * ref - 2.0 * C0.double()) < tol


def test_unit_wise_grouped_kernels_match_the_single_ones(K):
    """Grouped inverse and grouped block-vector product of many modules against the per-module kernels (bit for
    bit: same arithmetic per feature), including an all-zero module and a singular block."""
    torch.manual_seed(9)
    sizes = [64, 256, 300, 1, 2048, 512]
    blocks = []
    for F_ in sizes:
        g = torch.randn(F_, 2, 2, device='cuda')
        blocks.append((g @ g.transpose(1, 2)).contiguous())
    blocks[3].zero_()                                   # all-zero module: flag 0
    blocks[2][7] = torch.tensor([[-0.5, 0.0], [0.0, -0.5]], device='cuda')      # + damping 0.5 -> singular
    dampings = [0.5] * len(sizes)
    invs, flags = K.unit_wise_inv_grouped(blocks, dampings)
    flags = flags.cpu().tolist()
    for b, inv, fl in zip(blocks, invs, flags):
        ref_inv, ref_fl = K.unit_wise_inv(b, 0.5)
        assert fl == ref_fl.cpu().tolist()
        assert torch.equal(torch.nan_to_num(inv, posinf=7.0, neginf=-7.0), torch.nan_to_num(ref_inv, posinf=7.0, neginf=-7.0))
    assert flags[3][0] == 0 and flags[2][1] == 8 and flags[0] == [1, 0x7fffffff]
    # grouped product through the plan
    ws = [torch.randn(F_, device='cuda') for F_ in sizes]
    bs = [torch.randn(F_, device='cuda') for F_ in sizes]
    refs = []
    for inv, w, b in zip(invs, ws, bs):
        rw, rb = w.clone(), b.clone()
        K.unit_wise_mvp(inv, rw, rb, 0.25)
        refs.append((rw, rb))
    K.KronPrecondPlan([], 0.25, unit_items=list(zip(invs, ws, bs))).launch()
    torch.cuda.synchronize()
    for i, ((rw, rb), w, b) in enumerate(zip(refs, ws, bs)):
        if i == 2:
            continue        # holds the singular block (inf / nan entries)
        assert torch.equal(w, rw) and torch.equal(b, rb)


def test_gemm_grouped_matches_fp64(K):
    """Products of very different sizes in one launch, each against its fp64 product; edge tiles, transposes,
    strided rows, a scale per product."""
    torch.manual_seed(5)
    shapes = [(64, 576, 64, False, False), (512, 4608, 512, False, False), (512, 4608, 4608, False, True),
              (1000, 2048, 1000, False, False), (132, 260, 516, True, False), (256, 64, 2048, True, True),
              (4, 8, 12, False, False)]
    for pieces, tol in [(3, 2e-6), (2, 3e-5)]:
        problems, refs = [], []
        for i, (M, N, K_, tA, tB) in enumerate(shapes):
            A = torch.randn((K_, M) if tA else (M, K_), device='cuda')
            B = torch.randn(N, K_ + 8, device='cuda')[:, :K_] if tB else torch.randn(K_, N, device='cuda')   # strided rows
            C = torch.full((M, N), float('nan'), device='cuda')
            alpha = 0.25 * (i + 1)
            problems.append((A, B, C, tA, tB, alpha))
            refs.append(alpha * (A.T if tA else A).double() @ (B.T if tB else B).double())
        print(f'grouped gemm pieces={pieces}', flush=True)
        K.gemm_grouped(problems, pieces=pieces)
        torch.cuda.synchronize()
        for (A, B, C, tA, tB, alpha), ref in zip(problems, refs):
            assert relerr(C, ref) < tol, (tuple(C.shape), A.shape, relerr(C, ref))
    # accumulate form and symmetric products (lower tiles, mirrored) through the raw table
    for pieces in (3, 0):          # 0: the grouped kernel with true fp32 products
        G = torch.randn(260, 516, device='cuda')
        S0 = torch.randn(260, 260, device='cuda'); S0 = S0 + S0.T
        S1 = torch.randn(516, 516, device='cuda'); S1 = S1 + S1.T
        r0 = 0.3 * G.double() @ G.double().T + 0.7 * S0.double()
        r1 = 0.3 * G.double().T @ G.double() + 0.7 * S1.double()
        g = G.data_ptr()
        K.gemm_grouped_raw([(g, 516, g, 516, S0.data_ptr(), 260, 260, 260, 516, 0, 1, 0.3, 0.7, True),
                            (g, 516, g, 516, S1.data_ptr(), 516, 516, 516, 260, 1, 0, 0.3, 0.7, True)], G.device,
                           pieces=pieces)
        torch.cuda.synchronize()
        assert relerr(S0, r0) < 2e-6 and relerr(S1, r1) < 2e-6, pieces
        assert torch.equal(S0, S0.T) and torch.equal(S1, S1.T), pieces
    with pytest.raises(ValueError):
        K.gemm_grouped([(torch.randn(6, 6, device='cuda'), torch.randn(6, 6, device='cuda'),
                         torch.empty(6, 6, device='cuda'), False, False, 1.0)])       # extents not multiples of 4


def test_kron_precond_grouped_matches_fp64(K):
    """All modules in three launches: against B_inv G A_inv and B_inv b in fp64, and against the per-module kernel."""
    torch.manual_seed(6)
    dims = [(64, 576, False), (512, 4608, False), (1000, 2048, True), (64, 64, True), (256, 1152, False),
            (128, 128, True), (2048, 512, False), (8, 12, True), (64, 576, 'cl'), (128, 1152, 'cl'), (16, 100, 'cl5')]
    items, refs, singles = [], [], []
    for dB, dA, bias in dims:
        Bi = torch.randn(dB, dB, device='cuda'); Bi = Bi @ Bi.T / dB
        Ai = torch.randn(dA, dA, device='cuda'); Ai = Ai @ Ai.T / dA
        G = torch.randn(dB, dA, device='cuda')
        if isinstance(bias, str):          # a convolution gradient in the channels-last layout (3x3 or 5x5 window)
            k = 5 if bias == 'cl5' else 3
            G = G.view(dB, dA // (k * k), k, k).contiguous(memory_format=torch.channels_last)
            assert not G.is_contiguous()
            bias = False
        b = torch.randn(dB, device='cuda') if bias else None
        assert K.kron_precond_groupable(Bi, Ai, G, b)
        refs.append((0.5 * Bi.double() @ G.double().reshape(dB, dA) @ Ai.double(),
                     0.5 * Bi.double() @ b.double() if bias else None))
        Gs, bs = G.contiguous().clone(), (b.clone() if bias else None)
        K.kron_precond(Bi, Ai, Gs, bs, grad_scale=0.5)
        singles.append((Gs, bs))
        items.append((Bi, Ai, G, b))
    print('grouped precondition', flush=True)
    K.kron_precond_grouped(items, grad_scale=0.5)
    torch.cuda.synchronize()
    for (Bi, Ai, G, b), (rw, rb), (Gs, bs) in zip(items, refs, singles):
        assert relerr(G.reshape(rw.shape), rw) < 5e-6, (tuple(G.shape), relerr(G.reshape(rw.shape), rw))
        assert relerr(G.reshape(rw.shape), Gs.double().reshape(rw.shape)) < 5e-6
        if b is not None:
            assert relerr(b, rb) < 1e-5
    assert not K.kron_precond_groupable(torch.eye(6, device='cuda'), torch.eye(8, device='cuda'),
                                        torch.zeros(6, 8, device='cuda'))
    assert not K.kron_precond_groupable(torch.eye(8, device='cuda'), torch.eye(8, device='cuda'),
                                        torch.zeros(8, 8, device='cuda', dtype=torch.float64))


@pytest.mark.parametrize('dB,dA,bias', [(4, 5, True), (10, 784, True), (512, 512, True), (64, 147, False),
                                        (300, 1152, False)])
def test_kron_precond_matches_oracle(K, dB, dA, bias):
    g = torch.Generator().manual_seed(dB * 3 + dA)
    Bi = torch.randn(dB, dB, generator=g)
    Bi = Bi @ Bi.T / dB
    Ai = torch.randn(dA, dA, generator=g)
    Ai = Ai @ Ai.T / dA
    G = torch.randn(dB, dA, generator=g)
    b = torch.randn(dB, generator=g) if bias else None
    if bias:
        rw, rb = R.kron_mvp(Ai.double(), Bi.double(), G.double(), b.double())
    else:
        rw, rb = R.kron_mvp(Ai.double(), Bi.double(), G.double()), None
    Gg = G.cuda()
    bg = b.cuda() if bias else None
    K.kron_precond(Bi.cuda(), Ai.cuda(), Gg, bg, grad_scale=1.0)
    assert relerr(Gg, rw) < TOL_PRECOND
    assert relerr(Gg, rw) < 1e-5
    if bias:
        assert relerr(bg, rb) < 1e-5
    # conv-shaped gradient and grad_scale
    if dA % 9 == 0:
        G4 = G.view(dB, dA // 9, 3, 3).contiguous().cuda()
        K.kron_precond(Bi.cuda(), Ai.cuda(), G4, None, grad_scale=0.5)
        assert relerr(G4.view(dB, dA), 0.5 * rw) < 1e-5


# ------------------------------------------------------------------ unit-wise blocks (BatchNorm / LayerNorm)
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('kind,shape', [('bn2d', (6, 16, 7, 5)), ('bn2d_cl', (6, 16, 7, 5)), ('bn2d', (3, 70, 14, 14)),
                                        ('bn2d_cl', (3, 70, 14, 14)), ('bn2d_cl', (2, 8, 33, 40)), ('bn1d', (300, 12)),
                                        ('ln', (5, 37, 48)), ('ln', (200, 768))])
def test_unit_wise_stats_matches_oracle(K, dtype, kind, shape):
    torch.manual_seed(len(shape) + shape[1])
    if kind.startswith('bn2d'):
        m = nn.BatchNorm2d(shape[1])
    elif kind == 'bn1d':
        m = nn.BatchNorm1d(shape[1])
    else:
        m = nn.LayerNorm(shape[-1])
    with torch.no_grad():
        m.weight.uniform_(0.5, 1.5)
        m.bias.uniform_(-0.5, 0.5)
    y = _inputs(shape, dtype, seed=1)
    g = _inputs(shape, dtype, seed=2) * 0.1
    ref = R.norm_cov_unit_wise(m.double(), y.float().double(), g.float().double())
    yg, gg = y.cuda(), g.cuda()
    if kind == 'bn2d_cl':
        yg = yg.contiguous(memory_format=torch.channels_last)
        gg = gg.contiguous(memory_format=torch.channels_last)
    if kind == 'ln':
        yg, gg = yg.reshape(-1, shape[-1]), gg.reshape(-1, shape[-1])
    print(f'unit_wise_stats {kind} {shape} {dtype}', flush=True)
    w, b = m.weight.detach().float().cuda(), m.bias.detach().float().cuda()
    out = K.unit_wise_stats(yg, gg, w, b, alpha=0.25)
    torch.cuda.synchronize()
    assert relerr(out, 0.25 * ref) < 1e-5
    # accumulate form
    out2 = K.unit_wise_stats(yg, gg, w, b, out=out.clone(), alpha=0.5, beta=2.0)
    assert relerr(out2, 1.0 * ref) < 1e-5


@pytest.mark.parametrize('ydt,gdt', [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                     (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize('N,F', [(1, 4), (29, 12), (64, 256), (97, 260), (333, 768), (130, 770)])
def test_unit_wise_stats_of_rows(K, ydt, gdt, N, F):
    """Rows of features in fours and not, chunks of rows that end anywhere, rows with gaps between them and operands that no load of
    four elements is aligned to."""
    torch.manual_seed(N + F)
    wide_y, wide_g = torch.randn(N, F + 8).to(ydt).cuda(), torch.randn(N, F + 9).to(gdt).cuda()
    w, b = (torch.rand(F) + 0.5).cuda(), torch.randn(F).cuda()
    for y, g in ((wide_y[:, :F].contiguous(), wide_g[:, :F].contiguous()), (wide_y[:, 4:F + 4], wide_g[:, :F]), (wide_y[:, 1:F + 1], wide_g[:, 4:F + 4]),
                 (wide_y[:, :F].contiguous(), wide_g[:1, :F].contiguous().expand(N, F))):
        gd = g.double()
        gw = (y.double() - b.double()) / w.double() * gd
        ref = torch.stack([(gw * gw).sum(0), (gw * gd).sum(0), (gw * gd).sum(0), (gd * gd).sum(0)], 1).view(F, 2, 2)
        out = K.unit_wise_stats(y, g, w, b)
        # a product's factors round three times, a chain is 8 rows, the joins 8 waves and the chunks: below 40 roundings of sums of N terms
        size = ((gw * gw).sum(0) * (gd * gd).sum(0)).sqrt().clamp_min(1e-30)
        err = (out.double() - ref).abs()
        assert float((err[:, 0, 0] / ref[:, 0, 0]).max()) < 40 * 2.0 ** -24 and float((err[:, 1, 1] / ref[:, 1, 1]).max()) < 40 * 2.0 ** -24
        assert float((err[:, 0, 1] / size).max()) < 40 * 2.0 ** -24 and torch.equal(out[:, 0, 1], out[:, 1, 0])


def test_unit_wise_inv_and_mvp_match_oracle(K):
    torch.manual_seed(3)
    v = torch.randn(1000, 2, 3)
    blocks = v @ v.transpose(1, 2)
    inv, flags = K.unit_wise_inv(blocks.cuda(), 0.05)
    ref = R.unit_wise_inv(blocks.double(), 0.05)
    assert relerr(inv, ref) < 1e-5
    assert flags.cpu().tolist() == [1, 0x7fffffff]
    _, flags0 = K.unit_wise_inv(torch.zeros(5, 2, 2).cuda(), 0.05)
    assert flags0.cpu().tolist()[0] == 0
    _, flags_bad = K.unit_wise_inv(torch.zeros(5, 2, 2).cuda(), 0.0)
    assert flags_bad.cpu().tolist()[1] == 1                           # first singular block, 1-based
    w, b = torch.randn(1000), torch.randn(1000)
    rw, rb = R.unit_wise_mvp(ref, w.double(), b.double())
    gw, gb = K.unit_wise_mvp(inv, w.cuda(), b.cuda(), scale=2.0)
    assert relerr(gw, 2 * rw) < 1e-5 and relerr(gb, 2 * rb) < 1e-5


# ------------------------------------------------------------------------------ saved factors (bit-exact)
@pytest.mark.parametrize('d', [1, 3, 64, 257, 1000, 4608])
def test_tril_pack_unpack_bit_exact(K, d):
    import numpy as np
    g = torch.Generator().manual_seed(d)
    mat = torch.randn(d, d, generator=g)
    packed = K.tril_pack(mat.cuda())
    rows, cols = np.tril_indices(d)
    assert np.array_equal(packed.cpu().numpy(), mat.numpy()[rows, cols])
    if d <= 257:
        assert torch.equal(packed.cpu(), R.matrix_to_tril(mat))
        assert torch.equal(K.tril_unpack(packed, d).cpu(), R.tril_to_matrix(R.matrix_to_tril(mat)))
    full = K.tril_unpack(packed, d).cpu()
    assert torch.equal(full, full.T) and torch.equal(torch.tril(full), torch.tril(mat))
    # a row stride larger than d (a view of a wider buffer)
    wide = torch.zeros(d, d + 5)
    wide[:, :d] = mat
    assert torch.equal(K.tril_pack(wide.cuda()[:, :d]), packed)


def test_symmatrix_save_load_files(K, tmp_path):
    """File names, dictionary keys and contents as written by asdl/symmatrix.py:226-269, 471-491, 672-680: float32
    .npy, Kronecker factors as packed lower triangles, unit-wise blocks whole."""
    import numpy as np
    from asdl_amd.symmatrix import Kron, SymMatrix, UnitWise, matrix_to_tril, tril_to_matrix
    g = torch.Generator().manual_seed(5)
    a = torch.randn(40, 23, generator=g)
    b = torch.randn(40, 7, generator=g)
    A, B = a.T @ a, b.T @ b
    A, B = (A + A.T) / 2, (B + B.T) / 2     # bit-exact symmetry, so that equality below is exact
    unit = torch.randn(9, 2, 2, generator=g)
    full = torch.randn(11, 11, generator=g)
    full = full + full.T
    sm = SymMatrix(data=full.cuda(), kron=Kron(A.cuda(), B.cuda()), unit=UnitWise(data=unit.cuda()))
    paths = sm.save(str(tmp_path), 'fisher_emp/layer1')
    assert paths == {'tril': 'fisher_emp/layer1/tril.npy',
                     'kron': {'A_tril': 'fisher_emp/layer1/kron/A_tril.npy',
                              'B_tril': 'fisher_emp/layer1/kron/B_tril.npy'},
                     'unit_wise': 'fisher_emp/layer1/unit_wise.npy'}
    on_disk = np.load(tmp_path / paths['kron']['A_tril'])
    assert on_disk.dtype == np.float32 and on_disk.ndim == 1
    assert np.array_equal(on_disk, A.numpy()[np.tril_indices(23)])
    assert np.array_equal(np.load(tmp_path / paths['unit_wise']), unit.numpy())
    assert np.array_equal(np.load(tmp_path / paths['tril']), R.matrix_to_tril(full).numpy())

    back = SymMatrix()
    back.load(path=str(tmp_path / paths['tril']),
              kron_path={k: str(tmp_path / v) for k, v in paths['kron'].items()},
              unit_path=str(tmp_path / paths['unit_wise']))
    assert back.kron.A.is_cuda and torch.equal(back.kron.A.cpu(), A) and torch.equal(back.kron.B.cpu(), B)
    assert torch.equal(back.unit.data.cpu(), unit) and torch.equal(back.data.cpu(), full)
    assert back.kron.A_dim == 23 and back.kron.B_dim == 7

    # a file written the reference's way (numpy only) loads to the same factor
    ref_file = tmp_path / 'ref_A_tril.npy'
    np.save(ref_file, R.matrix_to_tril(A).numpy().astype('float32'))
    k2 = Kron(None, None)
    k2.load(str(ref_file), str(ref_file))
    assert torch.equal(k2.A.cpu(), A)
    assert torch.equal(tril_to_matrix(matrix_to_tril(B.cuda())).cpu(), B)
    with pytest.raises(RuntimeError):
        k2.load(str(ref_file), str(ref_file), device='cpu')
    with pytest.raises(ValueError):
        matrix_to_tril(torch.zeros(3, device='cuda'))


# ------------------------------------------------------------------------------ low-rank (swift) factors
@pytest.mark.parametrize('layout', ['nchw', 'channels_last'])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('case', [(3, 4, 6, 5, (3, 3), (2, 1), (1, 0)), (5, 70, 9, 9, (3, 3), (1, 1), (1, 1)),
                                  (2, 3, 20, 20, (7, 7), (2, 2), (3, 3)), (4, 130, 7, 7, (1, 1), (1, 1), (0, 0))])
def test_conv_patch_sum_matches_oracle(K, dtype, layout, case):
    N, C, H, W, k, s, p = case
    x = _inputs((N, C, H, W), dtype, seed=N + C)
    want = torch.nn.functional.unfold(x.double(), k, padding=p, stride=s).sum(-1)
    xg = x.cuda()
    if layout == 'channels_last':
        xg = xg.contiguous(memory_format=torch.channels_last)
    print(f'conv_patch_sum dtype={dtype} layout={layout} case={case}', flush=True)
    out = K.conv_patch_sum(xg, k, s, p, alpha=0.5)
    torch.cuda.synchronize()
    assert out.shape == (N, C * k[0] * k[1]) and relerr(out, 0.5 * want) < 1e-5
    K.conv_patch_sum(xg, k, s, p, out=out, alpha=0.25, beta=2.0)
    assert relerr(out, 1.25 * want) < 1e-5


def test_patch_sum_of_rows_and_positions(K):
    g = torch.Generator().manual_seed(2)
    a = torch.randn(7, 300, generator=g).to(torch.bfloat16)
    assert torch.equal(K.conv_patch_sum(a.cuda(), alpha=1.0).cpu(), a.float())          # Linear: a float32 copy
    gr = torch.randn(5, 33, 49, generator=g)                                              # [n, c, positions]
    assert relerr(K.conv_patch_sum(gr.cuda()), gr.double().sum(-1)) < 1e-6


@pytest.mark.parametrize('n,d,lam', [(8, 27, 1e-2), (64, 576, 3e-2), (3, 300, 0.5), (16, 1100, 1e-1)])
def test_smw_inv_matches_oracle(K, n, d, lam):
    g = torch.Generator().manual_seed(n + d)
    x = torch.randn(n, d, generator=g)
    dense = torch.linalg.inv(x.double().T @ x.double() / n + lam * torch.eye(d, dtype=torch.float64))
    out, info = K.smw_inv(x.cuda(), torch.tensor([lam], device='cuda'))
    assert int(info[0]) == 0
    assert relerr(out, dense) < TOL_INV and relerr(out, R.smw_inv(x, lam)) < TOL_INV


def test_kron_damping_with_row_matrices(K):
    g = torch.Generator().manual_seed(9)
    a_rows, b_sq = torch.randn(6, 40, generator=g), torch.randn(30, 12, generator=g)
    b_sq = b_sq.T @ b_sq
    a_sq = torch.randn(50, 9, generator=g)
    a_sq = a_sq.T @ a_sq
    b_rows = torch.randn(4, 21, generator=g)
    zero = torch.zeros(3, 17)
    pairs = [(a_rows, b_sq), (a_sq, b_rows), (a_rows, b_rows), (zero, b_sq)]
    lam, nz = K.kron_damping([p[0].cuda() for p in pairs], [p[1].cuda() for p in pairs], 1e-2,
                             eig_scale=[(1.0, 4.0), (0.25, 1.0), (1.0, 1.0), (1.0, 1.0)])
    lam, nz = lam.cpu(), nz.cpu()
    for i, ((A, B), (sa, sb)) in enumerate(zip(pairs, [(1.0, 4.0), (0.25, 1.0), (1.0, 1.0), (1.0, 1.0)])):
        want = R.swift_kron_damping(A * (sa if A.shape[0] == A.shape[1] else sa ** 0.5),
                                    B * (sb if B.shape[0] == B.shape[1] else sb ** 0.5), 1e-2)
        assert abs(float(lam[i, 0]) - want[0]) < 1e-5 * want[0] and abs(float(lam[i, 1]) - want[1]) < 1e-5 * want[1]
    assert nz.tolist() == [[1, 1], [1, 1], [1, 1], [0, 1]]


# Positions are summed per plane: sizes around one lane's share, a wave's and a work group's, both windows, strides with
# elements that no window takes, planes that are slices of wider ones, and an infinity that only some taps see.
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('case', [(3, 5, 1, 1, 1, 1, 0), (2, 7, 4, 4, 3, 1, 1), (3, 33, 5, 7, 3, 2, 1), (2, 3, 16, 16, 3, 1, 1), (2, 5, 17, 15, 3, 3, 0),
                                  (1, 3, 45, 46, 3, 1, 2), (2, 2, 64, 33, 3, 2, 1), (5, 4, 9, 9, 1, 2, 0), (1, 2, 1024, 3, 3, 1, 1), (1, 2, 1025, 3, 3, 1, 1)])
def test_patch_sum_of_planes(K, dtype, case):
    N, C, H, W, k, s, p = case
    wide = _inputs((N, C, H, W + 3), dtype, seed=H * W)
    x = wide[..., 1:W + 1]
    want = torch.nn.functional.unfold(x.double(), k, padding=p, stride=s).sum(-1)
    size = torch.nn.functional.unfold(x.double().abs(), k, padding=p, stride=s).sum(-1)
    print(f'patch_sum dtype={dtype} case={case}', flush=True)
    out = K.conv_patch_sum(wide.cuda()[..., 1:W + 1], (k, k), (s, s), (p, p))
    # a chain of additions of a lane and a tree over the lanes: 64 additions at most, 2^-24 of the sum of magnitudes each
    assert bool(((out.double().cpu() - want).abs() <= 64 * 2.0 ** -24 * size + 1e-30).all())
    x[0, 0, 0, 0] = float('inf')
    sees = torch.isinf(torch.nn.functional.unfold(x.double(), k, padding=p, stride=s)).any(-1)
    assert torch.equal(torch.isinf(K.conv_patch_sum(wide.cuda()[..., 1:W + 1], (k, k), (s, s), (p, p))).cpu(), sees)


@pytest.mark.parametrize('rows,d', [(1, 2), (3, 1365), (64, 512), (64, 513), (5, 8193)])
def test_kron_damping_of_row_matrices_at_any_alignment(K, rows, d):
    g = torch.Generator().manual_seed(d)
    flat = torch.randn(rows * d + 1, generator=g)
    b = torch.eye(d + rows + 1) * 2
    for skip in (0, 1):
        a = flat[skip:skip + rows * d].view(rows, d)
        lam, nz = K.kron_damping([flat.cuda()[skip:skip + rows * d].view(rows, d)], [b.cuda()], 1e-2)
        pi = ((a.double() ** 2).sum() / d / 2).sqrt()
        assert nz.tolist() == [[1, 1]]
        assert abs(float(lam[0, 0]) - 0.1 * float(pi)) < 1e-5 * 0.1 * float(pi) and abs(float(lam[0, 1]) - 0.1 / float(pi)) < 1e-5 * 0.1 / float(pi)
    last = torch.zeros(rows, d)
    last[-1, -1] = 1e-30
    assert K.kron_damping([last.cuda()], [b.cuda()], 1e-2)[1].tolist() == [[1, 1]]
    assert K.kron_damping([torch.zeros(rows, d).cuda()], [b.cuda()], 1e-2)[1].tolist() == [[0, 1]]


# Split counts around the limits of the reduction's slices (4 | 5, 63 | 64), one tile and several, one-tile windows
@pytest.mark.parametrize('N,C,hw,beta', [(1, 64, 40 * 8, 0.0), (3, 64, 41 * 8, 0.5), (63, 64, 256, 0.0), (64, 60, 256, 0.5), (70, 128, 512, 0.0), (40, 130, 256, 0.5), (9, 500, 64, 0.0)])
def test_split_reductions_match_fp64(K, N, C, hw, beta):
    x = _inputs((N, C, hw // 8, 8), torch.float32, N + C)
    rows = x.double().permute(0, 2, 3, 1).reshape(-1, C)
    old = torch.ones(C, C)
    out = old.cuda()
    K.conv_syrk(x.cuda(), (1, 1), (1, 1), (0, 0), out=out, alpha=0.5, beta=beta)
    assert relerr(out, 0.5 * rows.T @ rows + beta * old.double()) < TOL_FACTOR_F32 and torch.equal(out, out.T)


@pytest.mark.parametrize("M,d,pad", [(1, 1, 0), (1, 63, 1), (15, 64, 0), (16, 65, 3), (17, 127, 0), (63, 128, 5), (64, 129, 0), (129, 300, 1),
                                     (1023, 40, 0), (2100, 500, 4), (5003, 129, 0)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_fp32_rows_straight_to_the_matrix_instruction(K, M, d, pad, beta):
    x = _inputs((M, d + pad), torch.float32, M + d)
    x[:, d:] = float("nan")                 # columns between the rows are not read
    rows = x[:, :d].double()
    out = torch.ones(d, d).cuda()
    K.syrk_tn(x.cuda()[:, :d], out=out, alpha=0.5, beta=beta)
    assert relerr(out, 0.5 * rows.T @ rows + beta) < TOL_FACTOR_F32 and torch.equal(out, out.T)


@pytest.mark.parametrize("N,C,h,w,offset", [(1, 1, 1, 8, 0), (1, 63, 2, 4, 0), (3, 64, 1, 8, 0), (5, 65, 1, 24, 0), (2, 129, 8, 8, 0), (7, 300, 2, 20, 0),
                                            (1, 200, 1, 1000, 0), (130, 33, 4, 4, 0), (3, 65, 1, 8, 1), (3, 65, 3, 3, 0)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_fp32_runs_straight_to_the_matrix_instruction(K, N, C, h, w, offset, beta):
    # the last two go the staged way: a base that is no multiple of 16 bytes, runs that are no multiple of 8
    flat = _inputs((N * C * h * w + offset,), torch.float32, N + C + w)
    x = flat[offset:].reshape(N, C, h, w)
    rows = x.double().permute(0, 2, 3, 1).reshape(-1, C)
    out = torch.ones(C, C).cuda()
    K.conv_syrk(flat.cuda()[offset:].reshape(N, C, h, w), (1, 1), (1, 1), (0, 0), out=out, alpha=0.5, beta=beta)
    assert relerr(out, 0.5 * rows.T @ rows + beta) < TOL_FACTOR_F32 and torch.equal(out, out.T)


@pytest.mark.parametrize("d,k", [(512, 784), (10, 512), (300, 2000), (64, 8), (65, 72), (33, 24), (767, 3072), (1, 136)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_fp32_statistics_in_a_fixed_order(K, d, k, beta):
    # a base that is no multiple of 16 bytes, and rows 2^24 elements and more apart, take the staged kernels: the same bits
    flat = _inputs((d * k + 1,), torch.float32, d + k).cuda()
    x = flat[1:].reshape(d, k)
    old = torch.ones(d, d, device="cuda")
    a, b = old.clone(), old.clone()
    K.syrk_nt(x.clone(), out=a, alpha=0.5, beta=beta, in_order=True)
    K.conv_syrk(x[None, :, None], (1, 1), (1, 1), (0, 0), out=b, alpha=0.5, beta=beta, in_order=True)
    assert torch.equal(a, b) and torch.equal(a, a.T)
    rows = x.double().cpu()
    assert relerr(a, 0.5 * rows @ rows.T + beta) < TOL_FACTOR_F32
    if k <= 136:
        wide = torch.empty((k - 1) * ((1 << 24) + 4) + d, device="cuda").as_strided((k, d), ((1 << 24) + 4, 1))
        wide.copy_(x.T)
        c = old.clone()
        a = old.clone()
        K.syrk_tn(wide, out=c, alpha=0.5, beta=beta, in_order=True)
        K.syrk_tn(x.T.contiguous(), out=a, alpha=0.5, beta=beta, in_order=True)
        assert torch.equal(a, c) and relerr(a, 0.5 * rows @ rows.T + beta) < TOL_FACTOR_F32


@pytest.mark.parametrize("d,k", [(64, 8192), (65, 2560), (300, 4096), (512, 3072), (30, 60000)])
def test_fp32_statistics_in_a_fixed_order_add_their_splits_one_by_one(K, d, k):
    """Nonzero columns 320 apart, farther than a split is long, with products that fp32 holds exactly: the result has the bits of their
    sum from first to last, however many splits there are."""
    g = torch.Generator().manual_seed(d)
    x = torch.zeros(d, k)
    cols = torch.arange(7, k, 320)
    x[:, cols] = torch.randint(-2047, 2048, (d, len(cols)), generator=g) * torch.exp2(torch.randint(-6, 7, (1, len(cols)), generator=g).float())
    ref = torch.zeros(d, d)
    for c in cols:
        ref += x[:, c, None] * x[None, :, c]
    assert torch.equal(K.syrk_nt(x.cuda(), in_order=True).cpu(), ref)
    assert torch.equal(K.syrk_tn(x.T.contiguous().cuda(), in_order=True).cpu(), ref)


@pytest.mark.parametrize("transA", [False, True])
@pytest.mark.parametrize("transB", [False, True])
@pytest.mark.parametrize("Kd", [16, 24])
def test_short_contractions_sum_on_two_accumulators(K, Kd, transA, transB):
    """A matrix instruction adds two products, rounding twice.  Emulated in float32 for zero-mean operands: 7.4e-8 (16 k) and 7.3e-8 (24) on
    one accumulator per 16 k, 6.1e-8 and 6.2e-8 on two."""
    g = torch.Generator().manual_seed(Kd)
    a, b = torch.randn(512, Kd, generator=g), torch.randn(Kd, 512, generator=g)
    out = K.gemm((a.T if transA else a).contiguous().cuda(), (b.T if transB else b).contiguous().cuda(), transA=transA, transB=transB)
    assert relerr(out, a.double() @ b.double()) < 6.7e-8


@pytest.mark.parametrize("M,N,Kd", [(1, 1, 1), (1, 65, 17), (65, 1, 200), (64, 64, 16), (63, 66, 15), (129, 33, 127), (2, 130, 128), (200, 129, 143),
                                    (577, 75, 300), (65, 64, 1153), (31, 700, 2049), (1100, 1100, 300)])
@pytest.mark.parametrize("transA", [False, True])
@pytest.mark.parametrize("transB", [False, True])
def test_fp32_products_straight_to_the_matrix_instruction(K, M, N, Kd, transA, transB):
    # rows of the operands end where the memory of others begins (NaN): nothing beyond an edge may reach a result
    a = torch.full((Kd if transA else M, (M if transA else Kd) + 3), float("nan"))
    b = torch.full((N if transB else Kd, (Kd if transB else N) + 1), float("nan"))
    A, B = a[:, :-3], b[:, :-1]
    A.copy_(_inputs(tuple(A.shape), torch.float32, M + Kd))
    B.copy_(_inputs(tuple(B.shape), torch.float32, N + Kd))
    old = _inputs((M, N), torch.float32, M + N)
    ref = 0.5 * (A.double().T if transA else A.double()) @ (B.double().T if transB else B.double())
    Ag, Bg = a.cuda()[:, :-3], b.cuda()[:, :-1]
    for beta in (0.0, 1.5):
        out = old.cuda()
        K.gemm(Ag, Bg, out=out, transA=transA, transB=transB, alpha=0.5, beta=beta)
        assert relerr(out, ref + beta * old.double()) < TOL_FACTOR_F32


@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_grouped_half_pieces_in_tall_tiles_have_the_same_bits(K, transA, transB):
    # alone, every product stays below the number of tiles from which a launch takes two tile rows per work group
    sizes = [(4100, 3972, 100), (128, 128, 32), (260, 132, 4), (388, 516, 64), (64, 1000, 36), (2052, 260, 96)]
    A = [_inputs((k, m) if transA else (m, k), torch.float32, m + k).cuda() for m, n, k in sizes]
    B = [_inputs((n, k) if transB else (k, n), torch.float32, n + k).cuda() for m, n, k in sizes]

    def run(which):
        mx = torch.zeros(len(sizes), 3, device="cuda")
        out = [torch.full((m, n), 0.25, device="cuda") for m, n, k in sizes]
        specs = []
        for i in which:
            m, n, k = sizes[i]
            mx[i, 0], mx[i, 1] = A[i].abs().max(), B[i].abs().max()
            w = mx.data_ptr() + 12 * i
            specs.append((A[i].data_ptr(), A[i].stride(0), B[i].data_ptr(), B[i].stride(0), out[i].data_ptr(), n, m, n, k,
                          transA, transB, 0.5, 2.0 if i == 3 else 0.0, False, w, w + 4, w + 8))
        K.gemm_grouped_raw(specs, torch.device("cuda"), pieces=22)
        return out, mx[:, 2]
    together, largest = run(range(len(sizes)))
    for i, (m, n, k) in enumerate(sizes):
        if i == 0:
            pieces = []
            for half in (0, 1):                     # 33 x 32 tiles in two launches of fewer than 1024
                sl = slice(0, 2048) if half == 0 else slice(2048, m)
                a = A[0][:, sl] if transA else A[0][sl]
                o, mx = torch.empty(sl.stop - sl.start, n, device="cuda"), torch.zeros(3, device="cuda")
                mx[0], mx[1] = A[0].abs().max(), B[0].abs().max()
                K.gemm_grouped_raw([(a.data_ptr(), a.stride(0), B[0].data_ptr(), B[0].stride(0), o.data_ptr(), n, o.shape[0], n, k,
                                     transA, transB, 0.5, 0.0, False, mx.data_ptr(), mx.data_ptr() + 4, 0)], o.device, pieces=22)
                pieces.append(o)
            alone = torch.cat(pieces)
        else:
            alone = run([i])[0][i]
        assert torch.equal(together[i], alone)
        assert float(largest[i]) == float(alone.abs().max())


@pytest.mark.parametrize("N,C,H,W,kernel,stride,padding", [
    (1, 20, 3, 3, (3, 3), (1, 1), (1, 1)), (3, 64, 9, 7, (3, 3), (2, 2), (1, 1)), (2, 33, 5, 12, (3, 2), (1, 2), (0, 1)), (5, 12, 16, 16, (5, 5), (1, 1), (2, 2)),
    (70, 40, 9, 9, (3, 3), (2, 1), (1, 1)), (4, 65, 7, 7, (1, 1), (2, 2), (0, 0)), (9, 129, 5, 5, (1, 1), (1, 1), (0, 0)), (2, 30, 4, 4, (4, 8), (3, 1), (2, 4)),
    (300, 24, 6, 6, (3, 3), (2, 2), (1, 1)), (2, 18, 70, 65, (3, 3), (1, 1), (1, 1)), (2, 10, 6, 6, (6, 6), (1, 1), (0, 0))])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_fp32_windows_straight_to_the_matrix_instruction(K, N, C, H, W, kernel, stride, padding, beta):
    # (the last window has more than the 32 taps of a mask: the staged kernel)
    memory = torch.full((N * C * H * W + 256,), float("nan"))
    memory[128:-128] = _inputs((N * C * H * W,), torch.float32, N + C + H)
    x = memory[128:-128].view(N, C, H, W)
    rows = nn.functional.unfold(x.double(), kernel, 1, padding, stride).permute(0, 2, 1).reshape(-1, C * kernel[0] * kernel[1])
    d = rows.shape[1]
    out = torch.ones(d, d).cuda()
    K.conv_syrk(memory.cuda()[128:-128].view(N, C, H, W), kernel, stride, padding, out=out, alpha=0.5, beta=beta)
    assert relerr(out, 0.5 * rows.T @ rows + beta) < TOL_FACTOR_F32 and torch.equal(out, out.T)


def test_fp32_few_channels_add_their_partial_sums_in_pairs(K):
    """89 images, one partial sum each.  Every rounding of a sum of positive terms is 2.8e-8 (rms) of its own magnitude: 16 slices of
    5 or 6 partials added in pairs have 2.0 squares of the result's magnitude, one after the other 6.0, four running sums 3.4."""
    x = torch.randn(89, 16, 6, 6, generator=torch.Generator().manual_seed(3)).relu()
    rows = nn.functional.unfold(x.double(), 3, 1, 1, 1).permute(0, 2, 1).reshape(-1, 144)
    assert relerr(K.conv_syrk(x.cuda(), (3, 3), (1, 1), (1, 1)), rows.T @ rows) < 2.8e-8 * 3.4 ** 0.5


@pytest.mark.parametrize("N,C,H,W", [(82, 64, 5, 5), (64, 128, 6, 6), (3, 256, 27, 29), (100, 192, 5, 5), (9, 512, 15, 17), (2050, 64, 1, 1)])
def test_fp32_correlations_of_channels_of_any_scale(K, N, C, H, W):
    """2048 pixels and more: channels scaled by powers of two of their own, from 1e-17 to 1e17, one of them zero."""
    g = torch.Generator().manual_seed(N + C)
    x = torch.randn(N, C, H, W, generator=g).relu() * torch.exp(torch.linspace(-39, 39, C)[torch.randperm(C, generator=g)])[None, :, None, None]
    x[:, 5] = 0
    x[:, 7, 0, 0] *= 1e-3
    rows = nn.functional.unfold(x.double(), 3, 1, 1, 1).permute(0, 2, 1).reshape(-1, 9 * C)
    ref = rows.T @ rows
    xg = x.cuda()
    out = K.conv_syrk(xg, (3, 3), (1, 1), (1, 1))
    # every entry against the norms of its two channels (sums over all pixels, from which the border's are taken away): the
    # accumulation of up to 2050 terms in chunks
    scale = x.double().pow(2).sum(dim=(0, 2, 3)).sqrt().clamp_min(1e-30).repeat_interleave(9)
    assert float(((out.double().cpu() - ref) / scale / scale[:, None]).abs().max()) < 4e-6
    assert torch.equal(out, out.T)
    # a channel that is not finite spoils its own entries only
    bad = xg.clone()
    bad[0, 3, 0, 0], bad[1, 9, 0, 0] = float("inf"), float("nan")
    spoiled = K.conv_syrk(bad, (3, 3), (1, 1), (1, 1)).view(C, 9, C, 9)
    keep = [c for c in range(C) if c not in (3, 9)]
    assert torch.equal(spoiled[keep][:, :, keep], out.view(C, 9, C, 9)[keep][:, :, keep])
    assert not bool(torch.isfinite(spoiled[3, 4, 3, 4])) and bool(torch.isnan(spoiled[9, 4, 9, 4]))


@pytest.mark.parametrize("N,C,H,W", [(82, 64, 5, 5), (64, 128, 6, 6), (40, 256, 8, 8), (128, 64, 32, 32)])
def test_fp32_correlations_hold_all_24_bits(K, N, C, H, W):
    """One pixel that is not zero: every entry is one product of two operands with all 24 bits of their significands in
    use, so that nothing but the product's own roundings (the sum of its pieces, two at 2^-24) may show."""
    g = torch.Generator().manual_seed(C)
    x = torch.zeros(N, C, H, W)
    units = 2 * torch.randint(1024, 2048, (C,), generator=g) + 1        # odd, beyond what 11 + 11 bits hold
    x[N // 2, :, H // 2, W // 2] = (1 + units * 2.0 ** -23) * (2 * torch.randint(0, 2, (C,), generator=g) - 1)
    rows = nn.functional.unfold(x.double(), 3, 1, 1, 1).permute(0, 2, 1).reshape(-1, 9 * C)
    out = K.conv_syrk(x.cuda(), (3, 3), (1, 1), (1, 1))
    assert float((out.double().cpu() - rows.T @ rows).abs().max()) <= 2.0 ** -23


@pytest.mark.parametrize("N,C,H,W", [(1, 64, 1, 1), (15, 128, 1, 1), (17, 64, 1, 3), (1, 128, 1, 33), (5, 192, 4, 1), (3, 320, 7, 2), (33, 384, 2, 3), (1, 64, 31, 64),
                                     (129, 64, 2, 2), (2, 1024, 5, 5)])
def test_fp32_correlations_of_small_and_odd_images(K, N, C, H, W):
    """Images smaller than the window (every shift ends in the frame of zeros), pixels that fill no stage, column tiles that end behind
    the last tap (64, 192 and 320 channels), tiles below the diagonal that are left out (1024); several splits and one."""
    g = torch.Generator().manual_seed(N + C + H + W)
    x = torch.randn(N, C, H, W, generator=g)
    rows = nn.functional.unfold(x.double(), 3, 1, 1, 1).permute(0, 2, 1).reshape(-1, 9 * C)
    ref = rows.T @ rows
    guard = torch.full((9 * C + 2, 9 * C), 7.0, device='cuda')
    out = K.conv_syrk(x.cuda(), (3, 3), (1, 1), (1, 1), out=guard[1:-1])
    # sums of at most 2048 products, against the norms of their channels: a chain of 32 sums of 16 products and the joins after it
    # round at most 2^-24 of a partial sum each, and so do the three corrections of an entry
    scale = x.double().pow(2).sum(dim=(0, 2, 3)).sqrt().clamp_min(1e-30).repeat_interleave(9)
    assert float(((out.double().cpu() - ref) / scale / scale[:, None]).abs().max()) < 64 * 2.0 ** -24
    assert torch.equal(out, out.T)
    assert bool((guard[0] == 7).all()) and bool((guard[-1] == 7).all())


WINDOWS_ON_PLANES = [(128, 24, 32, 32, (3, 3), (1, 1), (1, 1)), (65, 64, 32, 31, (3, 3), (2, 2), (1, 1)), (130, 100, 14, 13, (3, 3), (2, 1), (1, 0)),
                     (37, 70, 21, 20, (5, 3), (1, 2), (2, 0)), (128, 256, 8, 8, (3, 3), (2, 2), (1, 1)), (33, 200, 15, 15, (2, 3), (1, 2), (0, 1)),
                     (90, 60, 17, 30, (5, 5), (3, 3), (4, 4)), (301, 96, 3, 5, (3, 3), (1, 1), (1, 1)), (2, 130, 40, 67, (1, 7), (1, 1), (0, 3))]


@pytest.mark.parametrize("N,C,H,W,k,s,p", WINDOWS_ON_PLANES)
def test_fp32_windows_on_bf16_planes(K, N, C, H, W, k, s, p):
    """Strided and other windows of an fp32 input on its three bf16 planes: channels that fill no 32, frames that cut the image off or
    reach beyond it, several splits and one."""
    from asdl_amd import _lib
    g = torch.Generator().manual_seed(N + C)
    d = C * k[0] * k[1]
    assert _lib.load().ak_conv_syrk_planes_ws_bytes(N, C, H, W, *k, *s, *p) > 0
    scale = torch.exp(torch.linspace(-20, 20, C)[torch.randperm(C, generator=g)])[None, :, None, None]
    x = torch.randn(N, C, H, W, generator=g).relu().cuda() * scale.cuda()
    rows = nn.functional.unfold(x.double(), k, 1, p, s).permute(0, 2, 1).reshape(-1, d)
    ref = rows.T @ rows
    guard = torch.full((d + 2, d + 3), 7.0, device='cuda')
    out = K.conv_syrk(x, k, s, p, out=guard[1:-1, 1:-2])
    # against the norms of the channels: 16 sums of 16 products round at most 2^-24 of their partial sum each, and so does the result; the
    # pieces left out are below 2^-24 of a product
    norm = x.double().pow(2).sum(dim=(0, 2, 3)).sqrt().clamp_min(1e-30).repeat_interleave(k[0] * k[1])
    bound = 24 * 2.0 ** -24
    assert float(((out.double() - ref) / norm / norm[:, None]).abs().max()) < bound
    assert torch.equal(out, out.T)
    before = out.clone()
    K.conv_syrk(x, k, s, p, out=guard[1:-1, 1:-2], alpha=0.5, beta=2.0)
    assert float(((out.double() - 2.5 * ref) / norm / norm[:, None]).abs().max()) < 3 * bound
    assert bool((guard[0] == 7).all()) and bool((guard[-1] == 7).all()) and bool((guard[:, 0] == 7).all()) and bool((guard[:, -2:] == 7).all())
    # a channel that is not finite spoils its own entries only
    x[0, 3, H // 2, W // 2], x[1, 9, H // 2, W // 2] = float("inf"), float("nan")
    spoiled = K.conv_syrk(x, k, s, p).view(C, -1, C, k[0] * k[1])
    keep = [c for c in range(C) if c not in (3, 9)]
    assert torch.equal(spoiled[keep][:, :, keep], before.view(C, -1, C, k[0] * k[1])[keep][:, :, keep])
    assert not bool(torch.isfinite(spoiled[3, :, 3]).all()) and bool(torch.isnan(spoiled[9, :, 9]).any())


@pytest.mark.parametrize("N,C,H", [(128, 64, 32), (128, 128, 16), (128, 256, 8)])
def test_fp32_correlations_are_as_close_as_one_rounding_of_the_result(K, N, C, H):
    """Sums over 8192 to 131072 pixels of ReLU outputs: their accumulators round at the magnitude of a split, and the factor ends
    within 2^-23 of the product in 64 bits (one split per place of the device: 1.3 to 1.5e-7)."""
    x = torch.randn(N, C, H, H, generator=torch.Generator().manual_seed(C)).relu().cuda()
    u = nn.functional.unfold(x.double(), 3, padding=1).transpose(1, 2).reshape(-1, 9 * C)
    out = K.conv_syrk(x, (3, 3), (1, 1), (1, 1)).double()
    ref = u.T @ u
    assert float((out - ref).norm() / ref.norm()) < 2.0 ** -23
