"""The quantiser of any group size, ragged K and unaligned rows, at the sizes
where its chunks and row ends can go wrong."""
import numpy as np
import pytest
import torch

import oracle
from hf_kernels_helion_amd import finegrained_fp8_helion as fp8
from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,group,pad,shift", [(1, 1, 128, 0, 0), (3, 7, 32, 1, 1),
                                                 (5, 129, 128, 0, 0), (7, 1376, 128, 0, 0),
                                                 (9, 1001, 64, 3, 5), (300, 264, 256, 0, 8),
                                                 (4, 512, 32, 0, 0), (33, 384, 256, 8, 1)])
def test_act_quant_any_group_and_alignment(dtype, M, K, group, pad, shift, dev):
    """Codes and scales equal the oracle's for groups of 32 to 256, row ends
    inside a group and a chunk, and rows at any element offset, with an all-zero
    group, an infinity and a NaN among the rows."""
    print(f"act_quant any {dtype} {M}x{K} group {group} pad {pad} shift {shift}", flush=True)
    x = synthetic.activations(M, K, seed=M + K, outlier_frac=0.01).float()
    x[0, :min(group, K)] = 0
    if M > 4:
        x[2, K - 1] = float("inf")
        x[3, K // 2] = float("nan")
    x = x.to(dtype)
    buf = torch.zeros(M * (K + pad) + shift, dtype=dtype, device=dev)
    rows = buf[shift:].as_strided((M, K), (K + pad, 1))
    rows.copy_(x.to(dev))
    q, s = fp8.act_quant(rows, group)
    if dtype == torch.bfloat16:
        qo, so = oracle.act_quant(x.view(torch.int16).numpy().view(np.uint16), group)
    else:
        qo, so = oracle.act_quant_f32(x.float().numpy(), group)
    np.testing.assert_array_equal(q.cpu().view(torch.uint8).numpy(), qo)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
