"""Tile grids whose tile count 8 does not divide (the runs of tiles per XCD have
two lengths): every tile of every kernel that walks such a grid, with and
without K splits and a tail launch, comes out once and in its place."""
import pytest
import torch

from hf_kernels_helion_amd import _native, deep_gemm_helion as dg, finegrained_fp8_helion as fp8

pytestmark = pytest.mark.gpu


def _place_operands(M, N, K, dev):
    """A[m,0] and B[n,1] ones, A[m,1] and B[n,0] small integers of m and n: each
    result row and column is told apart, exactly."""
    A = torch.zeros(M, K, device=dev)
    B = torch.zeros(N, K, device=dev)
    m, n = torch.arange(M, device=dev), torch.arange(N, device=dev)
    A[:, 0] = 1.0
    A[:, 1] = (m % 15).float()
    A[:, K - 1] = ((m // 15) % 15).float()
    B[:, 0] = (n % 13).float()
    B[:, 1] = 1.0
    B[:, K - 1] = ((n // 13) % 13).float()
    return A.to(torch.float8_e4m3fn), B.to(torch.float8_e4m3fn)


@pytest.mark.parametrize("M,N,K,bn", [
    (1, 17, 256, 128), (40, 1000, 2048, 128), (200, 2100, 2048, 128),    # small-grid tiles
    (777, 1536, 14336, 128), (777, 1536, 8192, 1), (900, 2500, 4096, 128),  # 128x128, split
    (777, 3000, 7168, 128), (1100, 4100, 8192, 128), (1500, 13900, 512, 1),
    (3001, 5000, 2048, 128), (900, 11008, 4096, 128), (4100, 4200, 1024, 128),
    (2999, 28000, 512, 128)])
def test_every_tile_in_its_place(M, N, K, bn, dev):
    p = _native.gemm_plan(M, N, K, block_n=bn)
    print(f"ragged grid {M}x{N}x{K} bn={bn}: {p['kernel']} {p['workgroups']} tail "
          f"{p['tail_kernel']} {p['tail_workgroups']} splits {p['splits']}", flush=True)
    A, B = _place_operands(M, N, K, dev)
    As = torch.ones(M, K // 128, device=dev)
    Bs = torch.ones(N if bn == 1 else -(-N // 128), K // 128, device=dev)
    ref = (A[:, [0, 1, K - 1]].float() @ B[:, [0, 1, K - 1]].float().t())
    if bn == 1:
        out = dg.gemm_fp8_fp8_bf16_nt(A, B, As, Bs)
        assert torch.equal(out, ref.to(torch.bfloat16))
    else:
        out = fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [128, 128], torch.float32)
        assert torch.equal(out, ref)


# K-block counts: every number of stages in flight (up to 10), the ends of a
# scale window (8) and of the 64 weight scales a register of the 256x128 kernel
# holds, and odd and even totals of the 128x128 kernel's two register sets.
K_BLOCKS = [*range(1, 11), 17, 63, 64, 65, 66, 130]


@pytest.mark.parametrize("N,kernel", [(3900, "gemm_pipe256x128_kernel"),
                                      (2000, "gemm_pipe128_kernel")])
@pytest.mark.parametrize("bn", [128, 1])
@pytest.mark.parametrize("KB", K_BLOCKS)
def test_stages_any_k_block_count(KB, bn, N, kernel, dev):
    """The pipelined 256x128 and 128x128 kernels over any number of K-blocks,
    scales in either layout: random small integers, other ones in every row and
    K-block, so that a fragment of another K-block, stage or row shows, and
    power-of-two scales, other ones in every K-block. Every sum is a whole number
    far below 2^24, which fp32 holds exactly in any order."""
    M, K = 2000, 128 * KB
    p = _native.gemm_plan(M, N, K, block_n=bn)
    print(f"{M}x{N} KB={KB} bn={bn}: {p['kernel']} splits {p['splits']}", flush=True)
    if p["cu_count"] == 256 and not (N == 2000 and KB == 130):  # (split 256x128 tiles)
        assert (p["kernel"], p["splits"]) == (kernel, 1), p
    g = torch.Generator().manual_seed(KB)
    ints = lambda rows: torch.randint(-4, 5, (rows, K), generator=g).float()
    A, B = ints(M).to(dev), ints(N).to(dev)
    As = torch.exp2(torch.randint(0, 4, (M, KB), generator=g).float()).to(dev)
    Bs = torch.exp2(torch.randint(0, 4, (-(-N // bn), KB), generator=g).float()).to(dev)
    x = (A * As.repeat_interleave(128, 1)).double()
    w = (B * Bs.repeat_interleave(bn, 0)[:N].repeat_interleave(128, 1)).double()
    ref = x @ w.t()
    assert ref.abs().max() < 2 ** 22
    A8, B8 = A.to(torch.float8_e4m3fn), B.to(torch.float8_e4m3fn)
    for As_l, Bs_l in ((As, Bs), (As.t().contiguous().t(), Bs.t().contiguous().t())):
        out = fp8.w8a8_block_fp8_matmul(A8, B8, As_l, Bs_l, [bn, 128], torch.float32)
        assert torch.equal(out.double(), ref)
