"""FP8 block-scaled linear on the GPU (nanovllm/kernels/fp8_linear.py:11-139)
against the oracle.

Activation quantisation is byte-exact (codes and bf16 scales).  The GEMM is
bit-exact where every step is exact (small-integer codes, power-of-two
scales).  Otherwise it is within one output ulp of the oracle's fp32
accumulator plus 2^-11 of the sum of absolute terms: the oracle sums each
128-wide block exactly, while gfx950's FP8 MFMA sums a block's products
aligned to the largest one in a window of 14 bits (a term more than 2^13
below the block's largest product is dropped: measured with cancelling
448 x 448 products beside one small term), the same kind of reduced-width
FP8 dot product NVIDIA's tensor cores compute for the reference, which is why
the reference promotes to fp32 every 128 elements.  On random codes the
largest error seen is 2^-15 of the sum of absolute terms; a misplaced or
missing K block errs by about 2^-3.5 of it.

Shapes are chosen so that on a 256-CU MI355X the library picks each of its
kernels: the 256x256 and 256x128 tiles whose two wave groups take turns, the
128x64, 128x32 and 64x16 tiles (features x tokens), the 96x192 tile with a
4-stage ring for 33 to 192 tokens with at least a CU's worth of 96-feature tiles
(tiles straddle the 128-row weight blocks, so fragments take their own scales;
K shorter than the ring), the small-M kernel for products of at most 256 tokens
whose tile grid would leave CUs idle and whose rows are long enough to share out
(K split over workgroups with fp32 partials added in split order when the
workspace allows), and the kernel for at most 32 tokens that streams the weights
without barriers.
"""
import numpy as np
import pytest
import torch

from gpu_util import announce
from oracle import fp8
from oracle import fp8_linear as ol
from nanovllm_amd.kernels.fp8_linear import fp8_block_linear
from nanovllm_amd import _native

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


def _codes(g, shape):
    c = torch.randint(0, 256, shape, generator=g, dtype=torch.int32).to(torch.uint8)
    return torch.where((c & 0x7F) == 0x7F, c ^ 0x01, c)   # no NaN codes


def _scales(g, shape, lo=-4, hi=1):
    return (10.0 ** torch.empty(shape).uniform_(lo, hi, generator=g)).to(torch.bfloat16)


# tolerance of the GEMM against the oracle's fp32 accumulator (module docstring)
ABS_TOL = 2.0 ** -11


def _gemm_gpu(xq, x_scale, w, w_scale, out_dtype=torch.bfloat16, w_stride=None, out_stride=None, ws_bytes=None):
    """Calls nvamd_fp8_block_gemm on device copies; optional padded row
    strides; ws_bytes: the workspace given (default: the size the library
    asks for)."""
    M, K = xq.shape
    N = w.shape[0]
    lib = _native.load()
    xq_d = xq.cuda().contiguous()
    xs_d = x_scale.cuda().contiguous()
    ws = w_stride or K
    w_buf = torch.zeros(N, ws, dtype=torch.uint8, device="cuda")
    w_buf[:, :K] = w.cuda()
    os_ = out_stride or N
    out_buf = torch.full((max(M, 1), os_), float("nan"), dtype=out_dtype, device="cuda")
    wsc = w_scale.cuda().contiguous()
    code = 0 if out_dtype == torch.bfloat16 else 1
    if ws_bytes is None:
        ws_bytes = lib.nvamd_fp8_block_gemm_workspace_bytes(M, N, K)
    gws = torch.full((max(ws_bytes, 16),), 0x7F, dtype=torch.uint8, device="cuda")  # NaN-filled partials
    st = lib.nvamd_fp8_block_gemm(xq_d.data_ptr(), xs_d.data_ptr(), w_buf.data_ptr(), ws, wsc.data_ptr(),
                                  out_buf.data_ptr(), os_, code, M, N, K, gws.data_ptr() if ws_bytes else None,
                                  ws_bytes, torch.cuda.current_stream().cuda_stream)
    _native.check(st, "fp8_block_gemm")
    torch.cuda.synchronize()
    if out_stride:
        assert torch.isnan(out_buf[:M, N:].float()).all(), "wrote past the row"
    return out_buf[:M, :N].cpu()


def _f64(xq, x_scale, w, w_scale):
    t = torch.from_numpy(fp8.dequant_table().astype(np.float64))
    xd = t[xq.long()] * x_scale.double().repeat_interleave(128, 1)
    wd = t[w.long()] * w_scale.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return xd @ wd.T, xd.abs() @ wd.abs().T


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_act_quant_byte_exact(dtype):
    announce(f"fp8 linear: activation quant {dtype}")
    g = torch.Generator().manual_seed(21)
    M, K = 77, 2048
    lo, hi = (-30, 30) if dtype == torch.bfloat16 else (-5, 4)
    mag = 10.0 ** torch.empty(M, K // 128, 1).uniform_(lo, hi, generator=g)
    x = (torch.randn(M, K // 128, 128, generator=g) * mag).reshape(M, K)
    x[3, :128] = 0.0                    # zero group
    x[4, 128:256] = -1.25               # constant group
    x[5, 256:384] = 0.0
    x[5, 300] = 3.0                     # single non-zero element
    x = x.to(dtype)
    xq_ref, xs_ref, _ = ol.act_quant(x)
    lib = _native.load()
    xd = x.cuda()
    xq = torch.empty(M, K, dtype=torch.uint8, device="cuda")
    xs = torch.empty(M, K // 128, dtype=torch.bfloat16, device="cuda")
    _native.check(lib.nvamd_fp8_act_quant(xd.data_ptr(), K, 0 if dtype == torch.bfloat16 else 1, xq.data_ptr(),
                                          xs.data_ptr(), M, K, torch.cuda.current_stream().cuda_stream), "act_quant")
    torch.cuda.synchronize()
    assert np.array_equal(xq.cpu().numpy(), xq_ref)
    assert np.array_equal(_bits(xs), xs_ref)


def test_act_quant_unit_scale_all_patterns_and_strided_rows():
    """Every finite bf16 value with |x| <= 448 in groups holding 448 (scale
    exactly 1), read through a row stride wider than K."""
    announce("fp8 linear: activation quant, all bf16 patterns at scale 1, strided rows")
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    vals = fp8.bf16_bits_to_f32(bits)
    vals = vals[np.isfinite(vals) & (np.abs(vals) <= 448.0)]
    groups = -(-len(vals) // 127)
    groups += groups % 2
    x = np.full((groups, 128), 448.0, dtype=np.float32)
    flat = np.zeros(groups * 127, dtype=np.float32)
    flat[:len(vals)] = vals
    x[:, 1:] = flat.reshape(groups, 127)
    x = torch.from_numpy(x.reshape(groups // 2, 256)).to(torch.bfloat16)
    M, K = x.shape
    wide = torch.zeros(M, K + 64, dtype=torch.bfloat16)
    wide[:, :K] = x
    xq_ref, xs_ref, _ = ol.act_quant(x)
    lib = _native.load()
    wd = wide.cuda()
    xq = torch.empty(M, K, dtype=torch.uint8, device="cuda")
    xs = torch.empty(M, K // 128, dtype=torch.bfloat16, device="cuda")
    _native.check(lib.nvamd_fp8_act_quant(wd.data_ptr(), K + 64, 0, xq.data_ptr(), xs.data_ptr(), M, K,
                                          torch.cuda.current_stream().cuda_stream), "act_quant")
    torch.cuda.synchronize()
    assert np.array_equal(xq.cpu().numpy(), xq_ref)
    assert np.array_equal(_bits(xs), xs_ref)


# (M, N, K): tile chosen on 256 CUs -> 256x256: (4096, 4096, 640) with an odd number of K blocks (a token
# row's scale then sits in either half of its x_scale dword); 256x128: (249, 24576, 1408); 128x64: (1024, 2048,
# 256), (4096, 4096, 256); 128x32: (1024, 1024, 128); 64x16: (300, 128, 256), (77, 2048, 1664), (130, 512, 3200)
TILE_SHAPES = [(4096, 4096, 256), (4096, 4096, 640), (1024, 2048, 256), (1024, 1024, 128), (300, 128, 256),
               (249, 24576, 1408)]
# at most 256 tokens: the Qwen3-8B qkv and down products at 192 tokens take the small-M kernel (down with K
# split over workgroups), gate/up the 96x192 ring tile; 256 tokens (16 token fragments), ragged token counts and
# odd K block counts on the small-M kernel; one token and 24 on the kernel for few tokens
SKINNY_SHAPES = [(192, 6144, 4096), (192, 24576, 4096), (192, 4096, 12288), (256, 1024, 4096), (1, 4096, 4096),
                 (24, 256, 512), (1, 128, 128), (77, 2048, 1664), (130, 512, 3200), (256, 1024, 6144),
                 (77, 2048, 2688), (130, 512, 4224), (33, 512, 2176)]
# the 96x192 ring tile: ragged tokens with an odd number of K blocks, K shorter than the ring (2 and 1 blocks),
# 65 tokens (its lower bound)
RING_SHAPES = [(100, 24576, 640), (150, 24576, 256), (192, 24576, 128), (65, 24576, 1024)]


@pytest.mark.parametrize("M,N,K", TILE_SHAPES + SKINNY_SHAPES + RING_SHAPES)
def test_gemm_exact_integer_case(M, N, K):
    """Small-integer codes, power-of-two scales: every fp32 step is exact, so
    the GPU must equal the oracle bit for bit (a transposed operand, a wrong
    K pairing between the MFMA operands or a misplaced scale fails)."""
    announce(f"fp8 linear: exact GEMM M={M} N={N} K={K}")
    g = torch.Generator().manual_seed(M + N + K)
    ints = torch.tensor([-4.0, -3.0, -2.0, -1.0, 0.0, 1.0, 2.0, 3.0, 4.0])
    xq = ints[torch.randint(0, 9, (M, K), generator=g)].to(torch.float8_e4m3fn).view(torch.uint8)
    w = ints[torch.randint(0, 9, (N, K), generator=g)].to(torch.float8_e4m3fn).view(torch.uint8)
    x_scale = (2.0 ** torch.randint(-3, 4, (M, K // 128), generator=g).float()).to(torch.bfloat16)
    w_scale = (2.0 ** torch.randint(-3, 4, (N // 128, K // 128), generator=g).float()).to(torch.bfloat16)
    got = _gemm_gpu(xq, x_scale, w, w_scale)
    want, _ = ol.block_gemm(xq.numpy(), _bits(x_scale), w.numpy(), _bits(w_scale))
    assert np.array_equal(_bits(got), want)


@pytest.mark.parametrize("M,N,K,out_dtype", [(4000, 4096, 384, torch.bfloat16), (1000, 2048, 512, torch.bfloat16),
                                             (77, 1024, 1024, torch.float16), (5, 384, 4096, torch.bfloat16),
                                             (130, 256, 12288, torch.bfloat16), (160, 24576, 768, torch.bfloat16),
                                             (96, 24576, 512, torch.float16)])
def test_gemm_matches_oracle(M, N, K, out_dtype):
    """Random codes (all finite E4M3FN values) and scales over five decades
    (two for the fp16 output, which must stay below 65504); ragged M, K up to
    12,288 (96 scale blocks)."""
    announce(f"fp8 linear: GEMM M={M} N={N} K={K} {out_dtype}")
    g = torch.Generator().manual_seed(M * 3 + N + K)
    xq, w = _codes(g, (M, K)), _codes(g, (N, K))
    lo, hi = (-4, 1) if out_dtype == torch.bfloat16 else (-4, -2)
    x_scale, w_scale = _scales(g, (M, K // 128), lo, hi), _scales(g, (N // 128, K // 128), lo, hi)
    got = _gemm_gpu(xq, x_scale, w, w_scale, out_dtype).double()
    _, acc = ol.block_gemm(xq.numpy(), _bits(x_scale), w.numpy(), _bits(w_scale),
                           "bf16" if out_dtype == torch.bfloat16 else "fp16")
    _, absum = _f64(xq, x_scale, w, w_scale)
    acc = torch.from_numpy(acc).double()
    ulp = 2.0 ** -7 if out_dtype == torch.bfloat16 else 2.0 ** -10
    bad = (got - acc).abs() > ulp * acc.abs() + ABS_TOL * absum
    assert not bad.any(), f"{int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


def test_gemm_large_tile_long_k_against_torch_fp32():
    """The 256x256 tile at the Qwen3-8B down-projection depth (K = 12,288, 96
    scale blocks; 4,000 tokens, ragged against the tile), against the same
    block-scaled sum in torch fp32 on the GPU (per K block an fp32 matmul of
    the dequantised codes, times x_scale * w_scale), at the oracle's
    tolerance.  The full-size oracle would take minutes on the host."""
    announce("fp8 linear: GEMM 4000 x 4096 x 12288 (256x256 tile) vs torch fp32")
    g = torch.Generator().manual_seed(12288)
    M, N, K = 4000, 4096, 12288
    xq, w = _codes(g, (M, K)), _codes(g, (N, K))
    x_scale, w_scale = _scales(g, (M, K // 128)), _scales(g, (N // 128, K // 128))
    got = _gemm_gpu(xq, x_scale, w, w_scale).cuda().double()
    t = torch.from_numpy(fp8.dequant_table().astype(np.float32)).cuda()
    xd, wd = t[xq.cuda().long()], t[w.cuda().long()]
    xs, ws = x_scale.cuda().float(), w_scale.cuda().float().repeat_interleave(128, 0)
    acc = torch.zeros(M, N, device="cuda")
    absum = torch.zeros(M, N, device="cuda")
    for kc in range(K // 128):
        xb, wb = xd[:, 128 * kc:128 * (kc + 1)], wd[:, 128 * kc:128 * (kc + 1)].T.contiguous()
        s = xs[:, kc:kc + 1] * ws[:, kc][None, :]
        acc += torch.matmul(xb, wb) * s
        absum += torch.matmul(xb.abs(), wb.abs()) * s
    bad = (got - acc.double()).abs() > 2.0 ** -7 * acc.double().abs() + ABS_TOL * absum.double()
    assert not bad.any(), f"{int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


def test_gemm_strided_weight_and_output_rows():
    """Weight rows with a padded stride, output rows with a padded stride (the
    padding must stay untouched)."""
    announce("fp8 linear: GEMM with strided weight and output rows")
    g = torch.Generator().manual_seed(9)
    M, N, K = 40, 384, 640
    xq, w = _codes(g, (M, K)), _codes(g, (N, K))
    x_scale, w_scale = _scales(g, (M, K // 128)), _scales(g, (N // 128, K // 128))
    got = _gemm_gpu(xq, x_scale, w, w_scale, w_stride=K + 128, out_stride=N + 8).double()
    _, acc = ol.block_gemm(xq.numpy(), _bits(x_scale), w.numpy(), _bits(w_scale))
    _, absum = _f64(xq, x_scale, w, w_scale)
    acc = torch.from_numpy(acc).double()
    assert not ((got - acc).abs() > 2.0 ** -7 * acc.abs() + ABS_TOL * absum).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fp8_block_linear_matches_oracle(dtype):
    """The drop-in fp8_block_linear (quant + GEMM) against the oracle's
    block_linear at K = 4096 (Qwen3-8B hidden size) with 300 tokens."""
    announce(f"fp8 linear: fp8_block_linear {dtype}")
    g = torch.Generator().manual_seed(4)
    M, N, K = 300, 1024, 4096
    x = (torch.randn(M, K, generator=g) * 3).to(dtype)
    w = _codes(g, (N, K))
    w_scale = (torch.rand(N // 128, K // 128, generator=g) * 2e-3).to(torch.bfloat16)
    got = fp8_block_linear(x.cuda(), w.cuda().view(torch.float8_e4m3fn), w_scale.cuda())
    torch.cuda.synchronize()
    assert got.dtype == dtype and got.shape == (M, N)
    xq, xs, _ = ol.act_quant(x)
    _, acc = ol.block_gemm(xq, xs, w.numpy(), _bits(w_scale), "bf16" if dtype == torch.bfloat16 else "fp16")
    _, absum = _f64(torch.from_numpy(xq), torch.from_numpy(xs.view(np.int16)).view(torch.bfloat16), w, w_scale)
    acc = torch.from_numpy(acc).double()
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert not ((got.cpu().double() - acc).abs() > ulp * acc.abs() + ABS_TOL * absum).any()


def test_skinny_gemm_split_repeatable_and_without_workspace():
    """The Qwen3-8B down projection at 192 tokens (K = 12,288 split over
    workgroups): random codes and scales against the oracle, the same bits on
    a second call (partials added in split order), and the unsplit product
    (no workspace) within the same tolerance."""
    announce("fp8 linear: small-M GEMM 192 x 4096 x 12288, split and unsplit")
    lib = _native.load()
    g = torch.Generator().manual_seed(192)
    M, N, K = 192, 4096, 12288
    assert lib.nvamd_fp8_block_gemm_workspace_bytes(M, N, K) > 0, "this product splits K"
    xq, w = _codes(g, (M, K)), _codes(g, (N, K))
    x_scale, w_scale = _scales(g, (M, K // 128)), _scales(g, (N // 128, K // 128))
    got = _gemm_gpu(xq, x_scale, w, w_scale)
    again = _gemm_gpu(xq, x_scale, w, w_scale)
    assert torch.equal(got.view(torch.int16), again.view(torch.int16)), "split sums differ between calls"
    unsplit = _gemm_gpu(xq, x_scale, w, w_scale, ws_bytes=0)
    _, acc = ol.block_gemm(xq.numpy(), _bits(x_scale), w.numpy(), _bits(w_scale))
    _, absum = _f64(xq, x_scale, w, w_scale)
    acc = torch.from_numpy(acc).double()
    for name, out in (("split", got), ("unsplit", unsplit)):
        bad = (out.double() - acc).abs() > 2.0 ** -7 * acc.abs() + ABS_TOL * absum
        assert not bad.any(), f"{name}: {int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("M,N,K,out_dtype", [(192, 6144, 4096, torch.bfloat16), (256, 2048, 4096, torch.float16),
                                             (33, 1024, 2048, torch.bfloat16), (256, 2048, 6144, torch.float16),
                                             (33, 1024, 3072, torch.bfloat16)])
def test_skinny_gemm_matches_oracle(M, N, K, out_dtype):
    """Random codes and scales over five decades (two for fp16 outputs) on the
    small-M kernel, against the oracle's accumulator."""
    announce(f"fp8 linear: small-M GEMM M={M} N={N} K={K} {out_dtype}")
    g = torch.Generator().manual_seed(M * 7 + N + K)
    xq, w = _codes(g, (M, K)), _codes(g, (N, K))
    lo, hi = (-4, 1) if out_dtype == torch.bfloat16 else (-4, -2)
    x_scale, w_scale = _scales(g, (M, K // 128), lo, hi), _scales(g, (N // 128, K // 128), lo, hi)
    got = _gemm_gpu(xq, x_scale, w, w_scale, out_dtype).double()
    _, acc = ol.block_gemm(xq.numpy(), _bits(x_scale), w.numpy(), _bits(w_scale),
                           "bf16" if out_dtype == torch.bfloat16 else "fp16")
    _, absum = _f64(xq, x_scale, w, w_scale)
    acc = torch.from_numpy(acc).double()
    ulp = 2.0 ** -7 if out_dtype == torch.bfloat16 else 2.0 ** -10
    bad = (got - acc).abs() > ulp * acc.abs() + ABS_TOL * absum
    assert not bad.any(), f"{int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(128, 128), (256, 1024), (384, 1152), (1024, 3072), (4224, 640), (4352, 2176),
                                 (512, 12288), (4224, 5248), (256, 4096), (128, 5120), (4224, 4096), (256, 7168),
                                 (512, 8192), (4096, 8192), (256, 16384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_tokens(M, N, K, dtype):
    """Calls of at most 32 tokens: one K block to several chunks of eight per
    wave with a short last one, one to eight waves, one workgroup a CU or more,
    activations quantised in the kernel (up to 2 or 4 tokens; three with eight
    waves, which with four would need more LDS than there is) and read
    quantised, strided activation rows.  Random codes against the oracle; the
    same call on activations quantised beforehand adds the same products in
    the same order, so it gives the same bits."""
    g = torch.Generator().manual_seed(M + 3 * N + K)
    wide = (torch.randn(M, K + 72, generator=g) * 3).to(dtype)
    wide[0, :128] = 0.0                        # a group of zeros, with both signs
    wide[0, 1:128:2] = -0.0
    w, w_scale = _codes(g, (N, K)), (torch.rand(N // 128, K // 128, generator=g) * 2e-3).to(torch.bfloat16)
    announce(f"fp8 linear: few tokens M={M} N={N} K={K} {dtype}")
    x = wide.cuda()[:, :K]
    got = fp8_block_linear(x, w.cuda().view(torch.float8_e4m3fn), w_scale.cuda())
    torch.cuda.synchronize()
    xq, xs, _ = ol.act_quant(wide[:, :K].contiguous())
    xq, xs = torch.from_numpy(xq), torch.from_numpy(xs.view(np.int16)).view(torch.bfloat16)
    pre = _gemm_gpu(xq, xs, w, w_scale, dtype)
    assert torch.equal(got.cpu().view(torch.int16), pre.view(torch.int16)), "in-kernel quantisation differs"
    _, acc = ol.block_gemm(xq.numpy(), _bits(xs), w.numpy(), _bits(w_scale), "bf16" if dtype == torch.bfloat16 else "fp16")
    _, absum = _f64(xq, xs, w, w_scale)
    acc = torch.from_numpy(acc).double()
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    bad = (got.cpu().double() - acc).abs() > ulp * acc.abs() + ABS_TOL * absum
    assert not bad.any(), f"{int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_act_quant_edge_groups(dtype):
    """Groups at the ends of the range the reciprocal form of the division
    covers: signed zeros, subnormal values, the largest and smallest amax of
    the type, a single value beside its smallest ones."""
    announce(f"fp8 linear: activation quant, edge groups {dtype}")
    info = torch.finfo(dtype)
    tiny = info.smallest_normal * info.eps                   # the smallest subnormal
    rows = [torch.zeros(128), -torch.zeros(128), torch.full((128,), tiny), torch.linspace(-1, 1, 128) * info.max,
            torch.linspace(-1, 1, 128) * info.smallest_normal, torch.arange(128.0) * tiny]
    if dtype == torch.bfloat16:                              # scales on both sides of 2^-100 and 2^100
        rows += [torch.linspace(-1, 1, 128) * 448.0 * 2.0 ** e for e in (-101, -100, -99, 99, 100, 101)]
    x = torch.stack([r.to(dtype) for r in rows] * 2)
    x[len(rows):, 5] = info.max                              # ... beside the largest value
    x = x.reshape(len(rows) * 2 // 2, 256)
    xq_ref, xs_ref, _ = ol.act_quant(x)
    lib = _native.load()
    xd = x.cuda()
    M, K = x.shape
    xq = torch.empty(M, K, dtype=torch.uint8, device="cuda")
    xs = torch.empty(M, K // 128, dtype=torch.bfloat16, device="cuda")
    _native.check(lib.nvamd_fp8_act_quant(xd.data_ptr(), K, 0 if dtype == torch.bfloat16 else 1, xq.data_ptr(),
                                          xs.data_ptr(), M, K, torch.cuda.current_stream().cuda_stream), "act_quant")
    torch.cuda.synchronize()
    assert np.array_equal(xq.cpu().numpy(), xq_ref)
    assert np.array_equal(_bits(xs), xs_ref)


@pytest.mark.parametrize("kernel,M,N,K", [
    (1, 4001, 4096, 128), (1, 4096, 4096, 256), (1, 3850, 4096, 384), (0, 8000, 2048, 1152), (1, 1889, 4096, 128),
    (1, 1900, 4096, 256), (1, 2048, 4096, 384), (1, 1800, 4096, 512), (1, 1793, 4096, 1152),
    (0, 2017, 24576, 384), (0, 3850, 4096, 512), (0, 3481, 4096, 640), (0, 1346, 8192, 1152), (0, 1773, 6144, 1280),
    (5, 126, 51200, 1152), (5, 980, 8192, 1280), (5, 249, 24576, 1408), (5, 65, 51200, 1536), (5, 1793, 4096, 1664)])
def test_group_swap_tiles(kernel, M, N, K):
    """The 256 x 256 and 256 x 128 tiles whose two wave groups take turns, from
    the fewest K blocks that are given to them (3 and 9: every phase of the two
    and three buffers) on, and the calls of 128 x 64 tiles beside them; ragged
    last tiles.  Against the block-scaled sum in torch fp32."""
    announce(f"fp8 linear: GEMM {M} x {N} x {K}, wave groups in turn")
    assert _native.load().nvamd_fp8_linear_kernel(M, N, K, 1, None) == kernel
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    xq = torch.randint(0, 256, (M, K), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    w = torch.randint(0, 256, (N, K), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    xq, w = (torch.where((c & 0x7F) == 0x7F, c ^ 0x01, c) for c in (xq, w))
    x_scale = (torch.rand(M, K // 128, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    w_scale = (torch.rand(N // 128, K // 128, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    got = _gemm_gpu(xq, x_scale, w, w_scale).cuda().double()
    t = torch.from_numpy(fp8.dequant_table().astype(np.float32)).cuda()
    xd, wd = t[xq.long()], t[w.long()]
    acc, absum = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
    for kc in range(K // 128):
        xb, wb = xd[:, 128 * kc:128 * (kc + 1)], wd[:, 128 * kc:128 * (kc + 1)].T.contiguous()
        s = x_scale[:, kc:kc + 1].float() * w_scale[:, kc].float().repeat_interleave(128)[None, :]
        acc += torch.matmul(xb, wb) * s
        absum += torch.matmul(xb.abs(), wb.abs()) * s
    bad = (got - acc.double()).abs() > 2.0 ** -7 * acc.double().abs() + ABS_TOL * absum.double()
    assert not bad.any(), f"{int(bad.sum())} outputs off, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("kernel,M,N,K", [(0, 3851, 4096, 512), (5, 249, 24576, 1408), (1, 1001, 2048, 512),
                                          (3, 77, 2048, 1664), (4, 100, 24576, 640), (6, 77, 2048, 2688),
                                          (7, 9, 512, 1152)])
def test_weights_in_the_last_columns_of_a_wider_matrix(kernel, M, N, K):
    """Weights that are the last K columns of a matrix with longer rows: the
    last row ends with the matrix, so no kernel may read past its K bytes (the
    matrix is the tail of one allocation).  Same bits as on contiguous
    weights."""
    announce(f"fp8 linear: GEMM {M} x {N} x {K}, weights in a wider matrix's last columns")
    lib = _native.load()
    assert lib.nvamd_fp8_linear_kernel(M, N, K, 1, None) == kernel
    g = torch.Generator(device="cuda").manual_seed(K)
    wide = torch.randint(0, 120, (N, K + 256), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    xq = torch.randint(0, 120, (M, K), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    xs = (torch.rand(M, K // 128, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    ws = (torch.rand(N // 128, K // 128, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    need = lib.nvamd_fp8_block_gemm_workspace_bytes(M, N, K)
    work = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    outs = []
    for w in (wide[:, 256:], wide[:, 256:].contiguous()):
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        _native.check(lib.nvamd_fp8_block_gemm(xq.data_ptr(), xs.data_ptr(), w.data_ptr(), w.stride(0), ws.data_ptr(),
                                               out.data_ptr(), N, 0, M, N, K, work.data_ptr() if need else None, need,
                                               torch.cuda.current_stream().cuda_stream), "fp8_block_gemm")
        outs.append(out.view(torch.int16))
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,N,K", [(1, 256, 1152), (2, 4352, 1152), (4, 256, 1664), (9, 256, 1152), (20, 512, 128),
                                   (40, 256, 2176)])
def test_infinite_weight_scale_in_the_last_block(M, N, K):
    """A weight scale of +inf in the last K block (K not a multiple of the
    chunks that kernels work in): the block's features are infinite with the
    sign of the block's sum, the others finite."""
    announce(f"fp8 linear: infinite scale in the last block, {M} x {N} x {K}")
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.rand(M, K, generator=g) + 0.5).to(torch.bfloat16)
    w = (torch.rand(N, K, generator=g) + 0.5).to(torch.float8_e4m3fn)
    w[5] = -w[5].float()
    w_scale = torch.full((N // 128, K // 128), 0.01, dtype=torch.bfloat16)
    w_scale[0, -1] = float("inf")
    got = fp8_block_linear(x.cuda(), w.cuda(), w_scale.cuda()).float().cpu()
    want = torch.full((M, 128), float("inf"))
    want[:, 5] = -float("inf")
    assert torch.equal(got[:, :128], want), got[:, :8]
    assert torch.isfinite(got[:, 128:]).all()


@pytest.mark.parametrize("kernel,M,N,K", [
    (0, 3481, 4096, 640), (0, 2017, 24576, 384), (1, 1001, 2048, 512), (2, 1000, 1024, 128), (3, 301, 128, 256),
    (3, 77, 2048, 1664), (4, 191, 24576, 640), (4, 67, 24576, 384), (5, 249, 24576, 1408), (5, 1793, 4096, 1664),
    (6, 77, 2048, 2688), (6, 191, 4096, 12288), (6, 255, 1024, 6272), (6, 33, 512, 4224), (7, 9, 512, 1152),
    (7, 31, 4096, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layer_equals_its_two_steps(kernel, M, N, K, dtype):
    """The layer quantises into a layout by K block ([K/128, M, 128] and
    [K/128, M]), the two C entry points by row ([M, K] and [M, K/128]): the
    same kernel on the same numbers in the same order, so the same bits; on
    every kernel, with odd token counts (a scale is then either half of its
    dword from block to block) and ragged last tiles (their rows past M would
    be the next block's)."""
    announce(f"fp8 linear: layer against its two steps, {M} x {N} x {K} {dtype}")
    lib = _native.load()
    assert lib.nvamd_fp8_linear_kernel(M, N, K, 0, None) == kernel
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g, device="cuda") * 3).to(dtype)
    x *= 10.0 ** torch.empty(M, 1, device="cuda").uniform_(-1, 1, generator=g)
    w = torch.randint(0, 256, (N, K), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    w = torch.where((w & 0x7F) == 0x7F, w ^ 0x01, w)
    w_scale = (torch.rand(N // 128, K // 128, generator=g, device="cuda") * 2e-4 + 1e-4).to(torch.bfloat16)
    got = fp8_block_linear(x, w.view(torch.float8_e4m3fn), w_scale)
    xq = torch.empty(M, K, dtype=torch.uint8, device="cuda")
    xs = torch.empty(M, K // 128, dtype=torch.bfloat16, device="cuda")
    _native.check(lib.nvamd_fp8_act_quant(x.data_ptr(), K, 0 if dtype == torch.bfloat16 else 1, xq.data_ptr(),
                                          xs.data_ptr(), M, K, torch.cuda.current_stream().cuda_stream), "act_quant")
    want = _gemm_gpu(xq, xs, w, w_scale, dtype)
    assert torch.isfinite(want.float()).all() and float(want.float().abs().max()) > 0
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16))


def test_layer_beyond_32_bit_block_offsets():
    """2^31 quantised bytes and more: the layer keeps its activations by row.
    Its first and last rows have the bits of the same rows in a call of their
    own (by K block; every tile adds the blocks in the same order)."""
    M, N, K = (1 << 19) + 77, 128, 4096
    announce(f"fp8 linear: layer of {M} x {K} activations, by row")
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.empty(M, K, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    w = torch.randint(0, 120, (N, K), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    w, w_scale = w.view(torch.float8_e4m3fn), torch.full((1, K // 128), 1e-3, dtype=torch.bfloat16, device="cuda")
    got = fp8_block_linear(x, w, w_scale)
    for rows in (slice(0, 4096), slice(M - 4099, M)):
        assert torch.equal(got[rows].view(torch.int16), fp8_block_linear(x[rows], w, w_scale).view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_act_quant_every_significand_pair(dtype):
    """The quantisation's division as a product with the reciprocal and one
    correction: every significand of the group's maximum against every
    significand of a value beside it, from the maximum's binade down to below
    half of the smallest E4M3 value; in bf16 also with scales next to 2^-100
    and 2^100, the ends of its range.  Codes and scales equal the oracle's IEEE
    divisions."""
    announce(f"fp8 linear: activation quant, every pair of significands {dtype}")
    bits = 7 if dtype == torch.bfloat16 else 10
    sig = 1.0 + torch.arange(2 ** bits, dtype=torch.float64) / 2 ** bits
    tops = [13] if dtype == torch.float16 else [0, -93, -92, 107]  # scales from 2^(top - 7.8) to 2^(top - 6.8)
    for top in tops:
        down = sig[None, :] * 2.0 ** (top - torch.arange(0, 21, dtype=torch.float64))[:, None]
        values = down.reshape(-1)                                          # 21 binades x all significands
        groups = -(-len(values) // 127)
        padded = torch.zeros(groups * 127, dtype=torch.float64)
        padded[:len(values)] = values
        for maxima in (sig * 2.0 ** (top + 1)).split(256):
            x = torch.empty(len(maxima), groups, 128, dtype=torch.float64)
            x[:, :, 1:] = padded.view(1, groups, 127)
            x[:, :, 0] = maxima[:, None]
            x[:, 1::2] *= -1.0
            x = x.reshape(len(maxima), groups * 128).to(dtype)
            xq_ref, xs_ref, _ = ol.act_quant(x)
            lib = _native.load()
            M, K = x.shape
            xd = x.cuda()
            xq = torch.empty(M, K, dtype=torch.uint8, device="cuda")
            xs = torch.empty(M, K // 128, dtype=torch.bfloat16, device="cuda")
            _native.check(lib.nvamd_fp8_act_quant(xd.data_ptr(), K, 0 if dtype == torch.bfloat16 else 1, xq.data_ptr(),
                                                  xs.data_ptr(), M, K, torch.cuda.current_stream().cuda_stream), "quant")
            torch.cuda.synchronize()
            assert np.array_equal(xq.cpu().numpy(), xq_ref)
            assert np.array_equal(_bits(xs), xs_ref)
