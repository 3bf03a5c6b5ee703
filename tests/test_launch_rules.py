"""The host's rules that route a launch: every call they send to a flat launch
has a kernel and a workspace, and batches on both sides of their lines take the
route that measured faster, on the CPU over many shapes and handles; on the
device, calls of a part of a handle's sequences."""
import atexit
import functools
import os
import shutil
import subprocess
import tempfile

import numpy as np
import pytest

from tests.helpers import assert_close, normal, rng_for
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def _program():
    """The check program's path: the host side from its source, the kernel tables from the built library."""
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not found")
    from leap_amd.attention import load_library
    load_library()
    lib = os.path.join(ROOT, "leap_amd")
    tmp = tempfile.mkdtemp()
    atexit.register(shutil.rmtree, tmp, ignore_errors=True)
    exe = os.path.join(tmp, "launch_rules_check")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", "-Xclang", "-target-feature",
                        "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "leap_amd", "csrc"), "-I",
                        os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "launch_rules_check.cpp"), "-o", exe,
                        "-L", lib, "-lleap_hip_attention", f"-Wl,-rpath,{lib}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def flat_workgroups(calls):
    """Workgroups per XCD of the flat launch of each call, 0 for a uniform one: calls are (q heads, KV heads,
    head_dim, seq_len, max_batch, sequences, longest, all rows or 0)."""
    r = subprocess.run([_program(), "route"], input="\n".join(" ".join(map(str, c)) for c in calls), capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return [int(x) for x in r.stdout.split()]


def test_flat_launches_have_kernels_workspace_and_measured_lines():
    r = subprocess.run([_program()], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


# Handles of more sequences than a call serves, whose small batches run as
# twin launch groups: the batch's lengths, the handle's max_batch, and whether
# the call gives its row count.
PARTIAL = [
    (32, 4, 64, [3000, 2000], 8, True),
    (32, 4, 64, [4500, 4500], 3, False),
    (64, 8, 128, [4096], 2, False),
    (64, 8, 128, [5000], 4, False),
    (32, 4, 128, [3000, 2000], 4, True),
    (16, 2, 128, [3000, 2000, 2500, 1500], 8, True),
    (8, 1, 128, [2500, 2011, 3000, 1, 2700, 2900, 2600, 2300], 16, True),
    (32, 4, 64, [300, 200], 8, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,hd,Ts,max_batch,rows_given", PARTIAL)
def test_part_of_a_handle_meets_the_oracle(hip_device, nh, nkv, hd, Ts, max_batch, rows_given):
    import torch
    from leap_amd.attention import HipAttention
    rng = rng_for(83, nh, nkv, hd, len(Ts), max(Ts))
    theta = 10000.0 if hd == 64 else 500000.0
    n = len(Ts)
    with HipAttention(nh, nkv, hd, max(Ts) + 1, max_batch=max_batch, rope_theta=theta) as att:
        rows = []
        for s, T in enumerate(Ts):
            rows.append((normal(rng, (T - 1, nkv * hd), hd), normal(rng, (T - 1, nkv * hd), hd)))
            if T > 1:
                att.kv_upload(s, 0, 0, *rows[s])
        pos = torch.tensor([T - 1 for T in Ts], dtype=torch.int32, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        for rep in range(2):
            q = normal(rng, (n, nh * hd), hd)
            k, v = normal(rng, (n, nkv * hd), hd), normal(rng, (n, nkv * hd), hd)
            d = [torch.from_numpy(a).cuda() for a in (q, k, v)]
            out = torch.zeros(n, nh * hd, device="cuda")
            att.step_batched_async(0, n, pos.data_ptr(), max(Ts) - 1, *(t.data_ptr() for t in d), out.data_ptr(), st,
                                   total_rows=sum(Ts) if rows_given else 0)
            torch.cuda.synchronize()
            out = out.cpu().numpy()
            for s, T in enumerate(Ts):
                orc = O.Oracle(1, nh, nkv, hd, T, theta=theta)
                orc.key_cache[0, :T - 1], orc.value_cache[0, :T - 1] = rows[s]
                want, _ = orc.step(0, T - 1, q[s], k[s], v[s])
                assert_close(out[s], want, what=f"sequence {s} of {T} rows, launch {rep}")
                kr, vr = att.kv_download(s, 0, T - 1, T)
                assert np.array_equal(kr[0], orc.key_cache[0, T - 1])
                assert np.array_equal(vr[0], orc.value_cache[0, T - 1])
