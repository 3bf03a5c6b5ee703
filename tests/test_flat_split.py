"""Flat launches: a batch whose groups do not cut evenly over the CUs, its
rows laid end to end and cut into equal runs (decode_attention_flat_kernel).
The split is checked on the host, and that the batches here take the flat
launch by the host's rule, at the edges of its runs, segments and items; on the
device they meet the oracle (or, where it is slow, the uniform chunks of
set_split)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.helpers import assert_close, normal, rng_for
from tests.test_launch_rules import flat_workgroups
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_flat_segments_cover_every_row_once(tmp_path):
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not found")
    exe = tmp_path / "flat_split_check"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "leap_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-o", str(exe),
                    os.path.join(ROOT, "tests", "flat_split_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def _filled(nh, nkv, hd, seq_len, Ts, rng):
    """A handle whose sequences hold T - 1 rows each, and those rows."""
    from leap_amd.attention import HipAttention
    att = HipAttention(nh, nkv, hd, seq_len, max_batch=len(Ts), rope_theta=10000.0 if hd == 64 else 500000.0)
    rows = []
    for s, T in enumerate(Ts):
        rows.append((normal(rng, (T - 1, nkv * hd), hd), normal(rng, (T - 1, nkv * hd), hd)))
        if T > 1:
            att.kv_upload(s, 0, 0, *rows[s])
    return att, rows


CASES = [
    # (32, 8, 128): eight items per XCD, runs of 64 rows and up; one-row, run-sized and one-over items
    (32, 8, 128, [1, 700, 63, 1200, 64, 65, 900, 1203]),
    (24, 8, 128, [1203, 1, 1, 700, 192, 900, 1200, 63]),
    (16, 8, 64, [700, 1200, 1300, 1, 900, 65]),
    (32, 8, 64, [2000, 1, 900, 65]),                                # 46 rows a run
    (64, 8, 128, [2000, 1, 1500, 129, 1100, 700, 512, 400]),       # 8 q heads per KV head, two-level merges
    (32, 4, 64, [1700, 1, 1300] + [700 + 7 * i for i in range(13)]),  # four KV heads: an XCD has every other sequence
    (128, 8, 128, [2600, 1100]),                                    # 16 q heads per KV head (two launch groups)
    (32, 8, 128, [40 + (37 * i) % 71 for i in range(64)]),          # 64 items per XCD, the most
    # equal lengths that do not divide the CUs
    (32, 8, 128, [1000] * 3),
    (8, 8, 128, [300] * 12),
    (64, 8, 128, [333] * 12),
    # equal lengths cut at the sequences' ends (a start counts as no rows)
    (32, 4, 64, [1920] * 8),
    (32, 4, 64, [241] * 64),
]


LONG = (32, 8, 128, [20000, 17, 9000, 130])
# a position that the launch cannot serve, by sequence
BAD = (32, 8, 128, [900, 300, 1000, 700, 350, 950, 1000, 600])
BAD_AT = {1: -1, 3: 5000, 6: 1001}


# a captured launch whose positions move between replays, sized for an upper bound and without a row count
MOVING = (32, 8, 128, 1600, 8, 6, 1600, 0)


def test_the_batches_here_take_the_flat_launch():
    calls = [(nh, nkv, hd, max(Ts) + 1, len(Ts), len(Ts), max(Ts), sum(Ts)) for nh, nkv, hd, Ts in CASES + [LONG]]
    calls.append((32, 8, 128, 1200, 8, 8, 1001, sum(BAD[3])))
    calls.append(MOVING)
    assert all(n > 0 for n in flat_workgroups(calls)), list(zip(calls, flat_workgroups(calls)))


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,hd,Ts", CASES)
def test_flat_batch_meets_the_oracle(hip_device, nh, nkv, hd, Ts):
    rng = rng_for(77, nh, nkv, hd, len(Ts), max(Ts))
    n, seq_len = len(Ts), max(Ts) + 1
    att, rows = _filled(nh, nkv, hd, seq_len, Ts, rng)
    with att:
        for rep in range(2):  # twice: the second launch finds the workspace as the first left it
            q = normal(rng, (n, nh * hd), hd)
            k, v = normal(rng, (n, nkv * hd), hd), normal(rng, (n, nkv * hd), hd)
            out = att.step_batched(0, [T - 1 for T in Ts], q, k, v)
            for s, T in enumerate(Ts):
                orc = O.Oracle(1, nh, nkv, hd, T, theta=10000.0 if hd == 64 else 500000.0)
                orc.key_cache[0, :T - 1], orc.value_cache[0, :T - 1] = rows[s]
                want, _ = orc.step(0, T - 1, q[s], k[s], v[s])
                assert_close(out[s], want, what=f"sequence {s} of {T} rows, launch {rep}")
                kr, vr = att.kv_download(s, 0, T - 1, T)
                assert np.array_equal(kr[0], orc.key_cache[0, T - 1])
                assert np.array_equal(vr[0], orc.value_cache[0, T - 1])


@pytest.mark.gpu
def test_flat_batch_matches_uniform_chunks_at_long_contexts(hip_device):
    """Runs of many passes and merges of more than 40 chunks.  Both splits are
    fp32 sums of the same products in another order: each within 6e-7 of 64
    bits in the 2-norm at these lengths, so within 1e-5 of the largest value
    of each other."""
    nh, nkv, hd, Ts = LONG
    rng = rng_for(78, 1)
    att, _ = _filled(nh, nkv, hd, max(Ts), Ts, rng)
    with att:
        q = normal(rng, (4, nh * hd), hd)
        k, v = normal(rng, (4, nkv * hd), hd), normal(rng, (4, nkv * hd), hd)
        flat = att.step_batched(0, [T - 1 for T in Ts], q, k, v)
        att.set_split(256)
        uniform = att.step_batched(0, [T - 1 for T in Ts], q, k, v)
        for s in range(4):
            assert_close(flat[s], uniform[s], rel=1e-5, what=f"sequence {s}")


@pytest.mark.gpu
def test_flat_batch_bad_positions_write_nan_rows(hip_device):
    """A position outside the launch: its output row reads NaN, its cache rows
    stay, and the other sequences' results do not change."""
    import torch
    (nh, nkv, hd, Ts), bad = BAD, BAD_AT
    rng = rng_for(79, 1)
    att, rows = _filled(nh, nkv, hd, 1200, Ts, rng)
    with att:
        q = normal(rng, (8, nh * hd), hd)
        k, v = normal(rng, (8, nkv * hd), hd), normal(rng, (8, nkv * hd), hd)
        pos = torch.tensor([bad.get(s, T - 1) for s, T in enumerate(Ts)], dtype=torch.int32, device="cuda")
        d = [torch.from_numpy(a).cuda() for a in (q, k, v)]
        out = torch.zeros(8, nh * hd, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        att.step_batched_async(0, 8, pos.data_ptr(), 1000, *(t.data_ptr() for t in d), out.data_ptr(), st,
                               total_rows=sum(Ts))
        torch.cuda.synchronize()
        out = out.cpu().numpy()
        for s, T in enumerate(Ts):
            if s in bad:
                assert np.isnan(out[s]).all()
                kr, _ = att.kv_download(s, 0, 0, T - 1)
                assert np.array_equal(kr, rows[s][0])
                continue
            orc = O.Oracle(1, nh, nkv, hd, T)
            orc.key_cache[0, :T - 1], orc.value_cache[0, :T - 1] = rows[s]
            want, _ = orc.step(0, T - 1, q[s], k[s], v[s])
            assert_close(out[s], want, what=f"sequence {s}")


@pytest.mark.gpu
def test_flat_launch_replays_at_moving_positions(hip_device):
    """One captured flat launch, replayed as the sequences grow: every replay
    gives the eager launch's output and cache rows at those positions."""
    import torch
    nh, nkv, hd, seq_len, max_batch, n, max_T, rows = MOVING
    from leap_amd.attention import HipAttention
    with HipAttention(nh, nkv, hd, seq_len, max_batch=max_batch) as att:
        att.kv_fill_normal(31, 0.1)
        g = torch.Generator(device="cuda").manual_seed(32)
        q = torch.randn(n, nh * hd, device="cuda", generator=g)
        k, v = (torch.randn(n, nkv * hd, device="cuda", generator=g) for _ in range(2))
        out = torch.zeros(n, nh * hd, device="cuda")
        pos = torch.tensor([0, 700, 63, 1300, 64, 900], dtype=torch.int32, device="cuda")

        def step(stream):
            att.step_batched_async(0, n, pos.data_ptr(), max_T - 1, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                   out.data_ptr(), stream, total_rows=rows)

        s = torch.cuda.Stream()
        step(s.cuda_stream)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            step(torch.cuda.current_stream().cuda_stream)
        for grow in (0, 1, 63, 130):
            pos += grow
            torch.cuda.synchronize()
            step(s.cuda_stream)
            torch.cuda.synchronize()
            want, at = out.clone(), pos.tolist()
            want_kv = [att.kv_download(i, 0, p, p + 1) for i, p in enumerate(at)]
            for rep in range(2):
                for i, p in enumerate(at):
                    att.kv_upload(i, 0, p, np.zeros((1, nkv * hd), np.float32), np.zeros((1, nkv * hd), np.float32))
                out.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, want), f"positions {at}, replay {rep}"
                for (wk, wv), i, p in zip(want_kv, range(n), at):
                    gk, gv = att.kv_download(i, 0, p, p + 1)
                    assert np.array_equal(gk, wk) and np.array_equal(gv, wv), f"sequence {i}"
