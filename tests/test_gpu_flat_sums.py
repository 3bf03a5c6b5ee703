"""Long runs of a flat launch sum thousands of equal terms.  A plain fp32 chain
of n equal terms c rounds the same way at every addition of a binade, an error
of up to n 2^-26 of the sum (3.8e-6 measured at 256); in parts of four passes it
is a quarter of that.  All but every sixteenth row of a sequence have one score,
a little under the sixteenth's, and v is 1: the output is 1, whatever the
scores, up to the rounding of the sums of p and of p v."""
import math

import numpy as np
import pytest

from tests.test_launch_rules import flat_workgroups

CALL = (32, 8, 128, 90001, 6, 6, 90000)
LENGTHS = [90000, 61003, 52001, 50009, 40013, 30011]


def test_the_batch_takes_the_flat_launch():
    assert flat_workgroups([CALL + (sum(LENGTHS),)])[0] == 32


@pytest.mark.gpu
def test_long_runs_of_equal_scores(hip_device):
    import torch
    from leap_amd.attention import HipAttention

    class Rows:
        def __init__(self, ptr, shape):
            self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}

    nh, nkv, hd, seq_len, n, _, max_T = CALL
    with HipAttention(nh, nkv, hd, seq_len, max_batch=n) as att:
        K, V = (torch.as_tensor(Rows(p, (n, seq_len, nkv, hd)), device="cuda") for p in att.kv_device_ptr(0, 0))
        V.fill_(1.0)
        # q = 0 but for the pair that turns slowest, along which k = (a, 0) at every row: a score a q0 cos(pos w)
        w = hd - 2
        K.zero_()
        K[..., w] = 1.0
        K[:, ::16, :, w] = 2.0
        q = torch.zeros(n, nh, hd, device="cuda")
        # p = 2^-d of the many rows, another d for every head and sequence
        d = torch.linspace(0.3, 6.0, n * nh, device="cuda").reshape(n, nh)
        q[..., w] = d * math.sqrt(hd) * math.log(2.0)
        k, v = torch.zeros(n, nkv * hd, device="cuda"), torch.ones(n, nkv * hd, device="cuda")
        out = torch.empty(n, nh * hd, device="cuda")
        pos = torch.tensor([t - 1 for t in LENGTHS], dtype=torch.int32, device="cuda")
        att.step_batched_async(0, n, pos.data_ptr(), max_T - 1, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                               torch.cuda.current_stream().cuda_stream, total_rows=sum(LENGTHS))
        torch.cuda.synchronize()
        err = (out.double() - 1.0).abs().max().item()
    passes = sum(LENGTHS) * nkv / 8 / 32 / 64  # of a run: 158
    # two sums in parts of four passes: passes/4 + 4 additions of 2^-26, and the combine's and merge's few
    bound = 2 * (passes / 4 + 4 + 16) * 2.0 ** -26
    assert err <= bound, f"{err:.2e} > {bound:.2e}"
