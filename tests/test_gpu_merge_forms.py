"""The up-projecting merge on both sides of the lines between its forms (csrc/merge_rule.h), against float64."""
import pytest
import torch

import test_gpu_edges as edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hkv,S,live,dv,d_out", [
    (1, 32, 8, 16, 16, 256, 128), (1, 32, 8, 15, 15, 256, 128),     # splits dealt out from 4096 values of a head on
    (4, 32, 8, 16, 9, 512, 128), (4, 33, 11, 16, 16, 512, 128),     # as many workgroups as CUs; three heads a kv head, more workgroups
    (1, 32, 8, 128, 127, 512, 128), (1, 32, 8, 129, 129, 512, 128),   # up to 65536 values of a head in one kernel
    (4, 32, 8, 7, 7, 512, 128), (5, 32, 8, 7, 3, 512, 128),         # few splits: one head a workgroup, or four
    (1, 5, 1, 1, 1, 70, 24), (1, 24, 2, 2, 2, 64, 200),             # ... of one kv head with rows that are no packets; four column blocks
    (1, 5, 1, 65, 63, 64, 8),          # 16 lanes a split, one packet of columns
    (1, 6, 2, 33, 31, 320, 72),        # six groups of 80 lanes, a partial column block
    (2, 3, 1, 60, 60, 70, 24),         # rows that are no packets
    (1, 16, 1, 128, 1, 512, 512),      # one live split, eight column blocks
    (1, 40, 1, 40, 40, 256, 512),      # more heads than a kv head may have
    (8, 16, 1, 32, 32, 256, 512), (8, 32, 8, 32, 30, 512, 128),     # a chip that the heads fill: 32768 and 65536 values a workgroup
    (8, 32, 8, 33, 33, 512, 128),      # ... and beyond: rows first
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_merge_forms(dev, dtype, b, hq, hkv, S, live, dv, d_out):
    edges.test_merge(dev, dtype, b, hq, hkv, S, live, dv, d_out)
