"""The GEMM kernel for any block size, ragged K and unaligned rows (fp16 MFMAs on
converted codes), at the sizes where its tiles, chunks and row ends can go
wrong."""
import pytest
import torch

from hf_kernels_helion_amd import _native
from hf_kernels_helion_amd import deep_gemm_helion, finegrained_fp8_helion as fp8
from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic

pytestmark = pytest.mark.gpu


def _offset_rows(t, pad, shift, dev):
    """t as rows of a wider buffer, `shift` elements from its start."""
    M, K = t.shape
    buf = torch.zeros(M * (K + pad) + shift, dtype=torch.uint8, device=dev)
    rows = buf.view(torch.float8_e4m3fn)[shift:].as_strided((M, K), (K + pad, 1))
    rows.copy_(t.to(dev))
    return rows


def _exact(A, B, As, Bs, bn, bk):
    """The formula in 64 bits, and the sum of its terms' magnitudes."""
    K = A.shape[1]
    a = A.double() * As.double().repeat_interleave(bk, 1)[:, :K]
    b = B.double() * Bs.double().repeat_interleave(bn, 0)[:B.shape[0]].repeat_interleave(bk, 1)[:, :K]
    return a @ b.t(), a.abs() @ b.abs().t()


# Edges of the tile shapes (M 16 | 17, 32 | 33, few and many tiles), K one
# byte around a 16-byte piece, a 128-byte chunk and a K-block, K below 16,
# K-blocks of several chunks (block_k 256, 300), shorter than a piece
# (block_k 8) and not a multiple of 16 (block_k 40), columns that share a
# scale by 16 and not (block_n 128, 32, 24, 1), more waves than K-blocks.
CASES = [(1, 1, 1, 128, 128), (3, 33, 15, 128, 128), (16, 40, 17, 128, 128),
         (17, 65, 129, 128, 128), (16, 300, 1376, 128, 128), (33, 130, 255, 32, 128),
         (40, 64, 300, 24, 64), (5, 70, 200, 1, 40), (20, 50, 90, 128, 8),
         (64, 96, 1000, 1, 256), (31, 100, 700, 64, 300), (777, 4096, 1376, 128, 128),
         (513, 8200, 143, 1, 128), (1030, 4100, 200, 48, 128), (9, 8225, 150, 128, 128),
         (32, 4099, 385, 1, 128), (100, 3000, 333, 128, 128), (7, 100, 14, 16, 4),
         # one chunk and K < 16, on 32x32 tiles and (many tiles) 64x128 ones
         (100, 130, 100, 1, 128), (33, 70, 128, 64, 128), (513, 8300, 13, 128, 128),
         (1500, 3000, 11, 1, 4), (2000, 1300, 100, 24, 300), (700, 6000, 16, 1, 128)]


@pytest.mark.parametrize("M,N,K,bn,bk", CASES)
@pytest.mark.parametrize("pad,shift", [(0, 0), (3, 5), (16, 16)])
def test_generic_gemm_keeps_fp32_sums(M, N, K, bn, bk, pad, shift, dev):
    """fp32 output against 64 bits: every product is exact and every sum is in
    fp32, so the error of a result is below (terms of a rounding chain) x
    2^-24 of the sum of its terms' magnitudes: 8 roundings per 32 columns
    inside a K-block, four per K-block for the fold. bf16 and fp16 outputs are
    the fp32 ones rounded. Rows at any byte offset give the same bits."""
    print(f"generic gemm {M}x{N}x{K} blocks {bn}x{bk} pad {pad} shift {shift}", flush=True)
    A, B, As, Bs = synthetic.harness_operands(M, N, K, seed=M + N + K, block_n=bn, block_k=bk)
    A, B = _offset_rows(A, pad, shift, dev), _offset_rows(B, pad, 2 * shift, dev)
    As, Bs = As.to(dev), Bs.to(dev)
    out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, bk], torch.float32)
    ref, mag = _exact(A, B, As, Bs, bn, bk)
    chain = 8 * (min(bk, K) / 32 + 1) + 4 * (-(-K // bk))
    if K % 128 or (bn, bk) not in ((128, 128), (1, 128)) or shift % 16 or pad % 16:
        assert ((out.double() - ref).abs() <= chain * 2.0 ** -24 * mag).all()
    for dtype in (torch.bfloat16, torch.float16):
        assert torch.equal(fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, bk], dtype),
                           out.to(dtype))
    if shift:
        same = fp8.w8a8_block_fp8_matmul(A.contiguous(), B.contiguous(), As, Bs, [bn, bk],
                                         torch.float32)
        assert torch.equal(same, out)
    if bn == 1:
        assert torch.equal(deep_gemm_helion.gemm_fp8_fp8_bf16_nt(A, B, As, Bs, bk),
                           out.to(torch.bfloat16))


# Aligned rows on a grid of at least 192 tiles of 128x128: the partial K-block
# alone (K 16, 112), in the first four K-blocks (200, 496) and in the fifth,
# sixth and twentieth (528, 640 + 16, 2544), K off a 16-byte piece on padded
# rows (1001, 1337), edges of the last row and column tile, per-row scales.
ALIGNED = [(1500, 2100, 16, 128, 0), (1500, 2100, 112, 128, 0), (777, 4096, 200, 128, 0),
           (777, 4096, 496, 1, 0), (300, 8192, 528, 128, 0), (1300, 4000, 656, 1, 16),
           (100, 28673, 144, 128, 0), (1000, 3100, 2544, 128, 32), (700, 5000, 1001, 128, 7),
           (65, 25000, 1337, 1, 7), (1025, 3000, 17, 128, 15)]


@pytest.mark.parametrize("M,N,K,bn,pad", ALIGNED)
def test_ragged_k_on_128_tiles(M, N, K, bn, pad, dev):
    """gemm_pipe128_kernel's fp16 form: the error bound above against 64 bits,
    16-bit outputs the fp32 one rounded, the bits of the kernel that unaligned
    rows of the same operands take, column-major scales included."""
    print(f"ragged 128 tiles {M}x{N}x{K} bn={bn} pad {pad}", flush=True)
    if pad == 0 and K % 16 == 0 and _native.gemm_plan(M, N, K, block_n=bn)["cu_count"] == 256:
        assert _native.gemm_plan(M, N, K, block_n=bn)["kernel"] == "gemm_pipe128_f16_kernel"
    A, B, As, Bs = synthetic.harness_operands(M, N, K, seed=M + N + K, block_n=bn)
    A, B = _offset_rows(A, pad, 16, dev), _offset_rows(B, pad, 32, dev)
    As, Bs = As.to(dev), Bs.to(dev)
    out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, 128], torch.float32)
    ref, mag = _exact(A, B, As, Bs, bn, 128)
    chain = 8 * (min(128, K) / 32 + 1) + 4 * (-(-K // 128))
    assert ((out.double() - ref).abs() <= chain * 2.0 ** -24 * mag).all()
    for dtype in (torch.bfloat16, torch.float16):
        assert torch.equal(fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, 128], dtype),
                           out.to(dtype))
    As_t, Bs_t = As.t().contiguous().t(), Bs.t().contiguous().t()
    assert torch.equal(fp8.w8a8_block_fp8_matmul(A, B, As_t, Bs_t, [bn, 128], torch.float32), out)
    off = fp8.w8a8_block_fp8_matmul(_offset_rows(A, 3, 1, dev), B, As, Bs, [bn, 128],
                                    torch.float32)
    if -(-M // 64) * -(-N // 128) >= 256:
        assert torch.equal(off, out)  # both walk K in order
    A.view(torch.uint8)[M - 1, K - 1] = 0x7F
    bad = ~torch.isfinite(fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, 128], torch.float32))
    assert bad[M - 1].all() and not bad[:M - 1].any()


# gemm_generic_kernel's tile rules and gemm_pipe128_kernel's fp16 form, with
# scales shared by 16 columns and per column.
@pytest.mark.parametrize("M,N,K,bn,bk", [(7, 40, 12, 128, 128), (16, 100, 200, 128, 128),
                                         (9, 8225, 150, 1, 128), (200, 300, 333, 24, 64),
                                         (777, 4096, 1001, 64, 128), (777, 4096, 208, 128, 128),
                                         (777, 4096, 208, 1, 128)])
@pytest.mark.parametrize("ea,eb,code", [(84, 45, 2.0 ** -8), (-100, -45, 256.0)])
def test_scale_products_outside_fp32(M, N, K, bn, bk, ea, eb, code, dev):
    """(sum * As) * Bs, the reference's order: each factor and the result are
    normal fp32 numbers where As * Bs is infinite or subnormal, and a zero sum
    stays zero. Against 64 bits, with the error bound above."""
    print(f"extreme scales {M}x{N}x{K} blocks {bn}x{bk} 2^{ea} 2^{eb}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    signs = lambda *s: torch.randint(0, 2, s, generator=g).float() * 2 - 1
    A = (signs(M, K) * code).to(torch.float8_e4m3fn).to(dev)
    B = (signs(N, K) * code).to(torch.float8_e4m3fn).to(dev)
    A.view(torch.uint8)[M - 1] = 0
    As = ((1 + torch.rand(M, -(-K // bk), generator=g)) * 2.0 ** ea).to(dev)
    Bs = ((1 + torch.rand(-(-N // bn), -(-K // bk), generator=g)) * 2.0 ** eb).to(dev)
    out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, bk], torch.float32)
    ref, mag = _exact(A, B, As, Bs, bn, bk)
    chain = 8 * (min(bk, K) / 32 + 1) + 4 * (-(-K // bk))
    assert ((out.double() - ref).abs() <= chain * 2.0 ** -24 * mag).all()
    assert not out[M - 1].any()


@pytest.mark.parametrize("M,N,K,bn,bk", [(5, 70, 600, 128, 256), (33, 130, 700, 1, 300),
                                         (16, 8300, 384, 128, 257), (300, 6000, 512, 64, 512),
                                         (700, 5000, 1000, 1, 256)])
@pytest.mark.parametrize("exponent", [0, 112])
def test_long_k_blocks_are_summed_before_scaling(M, N, K, bn, bk, exponent, dev):
    """A K-block longer than 128 is one sum, scaled once: its halves cancel
    exactly here but for the first column, with As * Bs so large at exponent 112
    that either half scaled by itself is infinite."""
    print(f"long K-blocks {M}x{N}x{K} blocks {bn}x{bk} 2^{exponent}", flush=True)
    A = torch.full((M, K), 448.0)
    k = torch.arange(K)
    blk = k // bk * bk
    size = torch.minimum(blk + bk, torch.tensor(K)) - blk
    A[:, k - blk >= (size + 1) // 2] = -448.0
    A[:, ((k - blk) == size // 2) & (size % 2 == 1)] = 0.0
    A[:, 0] = 416.0
    A = A.to(torch.float8_e4m3fn).to(dev)
    B = torch.full((N, K), 448.0).to(torch.float8_e4m3fn).to(dev)
    KB = -(-K // bk)
    As = torch.full((M, KB), 2.0 ** (exponent // 2), device=dev)
    Bs = torch.full((-(-N // bn), KB), 2.0 ** (exponent - exponent // 2), device=dev)
    out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [bn, bk], torch.float32)
    assert (out == -32.0 * 448.0 * 2.0 ** exponent).all()


def test_generic_gemm_every_code_and_nan(dev):
    """Each of the 256 codes against 1.0 comes back exactly (NaN as NaN), and
    a NaN row, column or scale reaches only its own results."""
    codes = torch.arange(256, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    A = codes.view(256, 1).contiguous()
    B = torch.ones(3, 1, device=dev).to(torch.float8_e4m3fn)
    one = torch.ones(256, 1, device=dev)
    out = fp8.w8a8_block_fp8_matmul(A, B, one, torch.ones(1, 1, device=dev), [128, 128],
                                    torch.float32)
    torch.testing.assert_close(out, codes.float().view(256, 1).expand(256, 3), rtol=0, atol=0,
                               equal_nan=True)
    A, B, As, Bs = [t.to(dev) for t in synthetic.harness_operands(40, 70, 143, seed=1)]
    A.view(torch.uint8)[7, 142] = 0x7F
    As[9, 1] = float("nan")
    As[11, 0] = float("inf")
    out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [128, 128], torch.float32)
    bad = ~torch.isfinite(out)
    assert bad[[7, 9, 11]].all() and not bad[[i for i in range(40) if i not in (7, 9, 11)]].any()
