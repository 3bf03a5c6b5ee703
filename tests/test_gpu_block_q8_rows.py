"""The int8 projections at row counts between the compiled sizes: workgroups
with idle row slots, waves with unequal rows, several workgroups per CU and a
ragged last workgroup.  Every stage is checked as in test_gpu_block_q8 (the
int8 products bitwise)."""
import numpy as np
import pytest

from tests.helpers import normal, rng_for
from tests.test_gpu_block_q8 import _check_stages, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nh,nkv,ctx,gs", [
    (2048, 16, 1, 40, 64),    # q/k/v 2304 rows: 9 a workgroup, 5 waves of 2 rows
    (2048, 32, 8, 17, 32),    # 3072: 12 of 16 slots
    (2048, 32, 32, 9, 128),   # 6144: 24, 8 waves of 3
    (3072, 24, 24, 33, 64),   # 9216: 36, 12 waves of 3
    (4096, 32, 4, 21, 64),    # 5120: 20 of 24 slots
    (5120, 40, 10, 12, 64),   # 7680: 30 of 60 slots
    (8192, 64, 16, 5, 128),   # 12288: 48, two workgroups per CU
])
def test_q8_block_between_compiled_sizes(hip_device, dim, nh, nkv, ctx, gs):
    hd = dim // nh
    att, orc, w = _setup(dim, nh, nkv, ctx, 1, [0], gs, 15)
    rms, w8 = w[0]
    with att:
        pos = ctx - 1
        rng = rng_for(dim, nkv, ctx, gs, 16)
        k_rows, v_rows = normal(rng, (pos, nkv * hd), hd), normal(rng, (pos, nkv * hd), hd)
        att.kv_upload(0, 0, 0, k_rows, v_rows)
        orc.key_cache[0, :pos], orc.value_cache[0, :pos] = k_rows, v_rows
        x = rng.standard_normal(dim).astype(np.float32)
        got = att.block(0, pos, x)
        _check_stages(att, orc, 0, pos, x, got, rms, w8, gs, f"dim {dim} kv heads {nkv}")
