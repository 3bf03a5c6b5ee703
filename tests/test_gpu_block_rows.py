"""The fp32 projections at the row counts where the rows per workgroup change
with the model's KV heads: every stage's result as in test_gpu_block."""
import pytest

import tests.test_gpu_block as block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nh,nkv,ctx", [
    (2048, 32, 8, 30),    # q/k/v 3072 rows: 12 a workgroup
    (2048, 32, 32, 9),    # 6144: 12, two workgroups per CU
    (2048, 16, 1, 20),    # 2304: 10, the last workgroup short
    (3072, 24, 24, 33),   # 9216: 12, three per CU; wo 3072: 12
    (4096, 32, 2, 21),    # 4608: 6
    (5120, 40, 10, 12),   # 7680: 6; wo 5120: 5
    (8192, 64, 4, 7),     # 9216: 5 or 4
])
def test_block_rows_per_workgroup(hip_device, dim, nh, nkv, ctx):
    block.test_block_matches_oracle(hip_device, dim, nh, nkv, ctx)
