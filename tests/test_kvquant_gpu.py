"""GPU quantizer parity: bit-exact with the reference's vectors and with the oracle.

Restates the int8 parts of the reference's ``tests/test_kvquant.py`` (226-249) and
``tests/test_kvattn.py::test_pack_matches_quantizer`` (168-175) against the HIP kernels.
"""

from __future__ import annotations

from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import kvquant as okq
from tests.helpers import bench_outliers, npy, randn

pytestmark = pytest.mark.gpu

GOLD = Path(__file__).resolve().parent / "golden"
QUANT_FILES = sorted(GOLD.glob("quant_*.npz"))


def _eq16(a: torch.Tensor, b: np.ndarray) -> bool:
    return np.array_equal(npy(a).view(np.uint16), np.asarray(b).view(np.uint16))


@pytest.mark.parametrize("path", QUANT_FILES, ids=[p.stem for p in QUANT_FILES])
def test_gpu_quantizer_matches_reference_vectors(path):
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    z = np.load(path)
    gs, axis = int(z["group"]), str(z["axis"])
    print(f"case {path.stem} shape={z['x'].shape} group={gs} axis={axis}", flush=True)
    x = torch.from_numpy(z["x"]).cuda()
    q, mn, st = quantize_int8(x, gs, axis)
    assert np.array_equal(npy(q), z["q"])
    assert _eq16(mn, z["mins"]) and _eq16(st, z["steps"])
    deq = dequantize_int8(torch.from_numpy(z["q"]).cuda(), torch.from_numpy(z["mins"]).cuda(),
                          torch.from_numpy(z["steps"]).cuda(), gs, axis)
    assert _eq16(deq, z["deq"])


@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 200, 2048])
def test_token_axis_matches_oracle(n):
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    x = randn((1, 8, n, 128), n, 1.0)
    x = bench_outliers(x, n)
    q, mn, st = quantize_int8(x.cuda(), 64, "token")
    rq, rm, rs = okq.quantize_int8_token(npy(x), 64)
    assert np.array_equal(npy(q), rq)
    assert _eq16(mn, rm) and _eq16(st, rs)
    deq = dequantize_int8(q, mn, st, 64, "token")
    assert _eq16(deq, okq.dequantize_int8_token(rq, rm, rs, 64))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_other_input_dtypes_match_oracle(dtype):
    """The reference upcasts any float input to fp32 first; bf16 and fp32 inputs follow."""
    from nova_amd.kvquant import quantize_int8

    x = (torch.randn(1, 4, 130, 128, generator=torch.Generator().manual_seed(3)) * 2).to(dtype)
    q, mn, st = quantize_int8(x.cuda(), 64, "token")
    rq, rm, rs = okq.quantize_int8_token(x.float().numpy(), 64)
    assert np.array_equal(npy(q), rq)
    assert _eq16(mn, rm) and _eq16(st, rs)


def test_strided_slices_into_cache_match_contiguous():
    """``quantize_int8_into`` writes straight into slices of larger cache buffers."""
    from nova_amd.kvquant import quantize_int8, quantize_int8_into

    src = randn((1, 8, 300, 128), 11).cuda()
    qbuf = torch.full((1, 8, 512, 128), 7, dtype=torch.uint8, device="cuda")
    mbuf = torch.zeros((1, 8, 8, 128), dtype=torch.float16, device="cuda")
    sbuf = torch.zeros_like(mbuf)
    quantize_int8_into(src[:, :, :256], 64, qbuf[:, :, :256], mbuf[:, :, :4], sbuf[:, :, :4])
    q, mn, st = quantize_int8(src[:, :, :256].contiguous(), 64, "token")
    assert torch.equal(qbuf[:, :, :256], q)
    assert torch.equal(mbuf[:, :, :4], mn) and torch.equal(sbuf[:, :, :4], st)
    assert (qbuf[:, :, 256:] == 7).all() and not mbuf[:, :, 4:].any()


def test_constant_and_shapes():
    """``tests/test_kvquant.py:243-249``: constant tensors round-trip exactly, shapes return."""
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    const = torch.full((1, 2, 8, 128), 3.5, dtype=torch.float16, device="cuda")
    for axis, gs in (("channel", 32), ("token", 4)):
        q, mins, steps = quantize_int8(const, gs, axis)
        assert q.shape == const.shape
        assert torch.equal(dequantize_int8(q, mins, steps, gs, axis), const)


def test_error_bounds_against_int4_like_channel_axis():
    """``tests/test_kvquant.py:226-240`` (int8 half): token-axis rulers beat channel-axis
    ones under a channel outlier, and the relative error stays below 0.02."""
    from nova_amd.kvquant import roundtrip_int8

    g = torch.Generator().manual_seed(7)
    x = torch.randn(1, 2, 256, 128, generator=g, dtype=torch.float16)
    x[:, :, :, 7] *= 40
    xc = x.cuda()
    e_chan = (roundtrip_int8(xc, 32, "channel").float() - xc.float()).norm() / xc.float().norm()
    e_tok = (roundtrip_int8(xc, 64, "token").float() - xc.float()).norm() / xc.float().norm()
    assert float(e_chan) < 0.02
    assert float(e_tok) <= float(e_chan)


def test_pack_matches_quantizer():
    from nova_amd.kvattn import GROUP_T, pack_int8_kv
    from nova_amd.kvquant import quantize_int8

    k = randn((1, 8, 200, 128), 5).cuda()
    v = randn((1, 8, 200, 128), 6).cuda()
    kq, kmn, kst, vq, vmn, vst = pack_int8_kv(k, v)
    for got, want in zip((kq, kmn, kst), quantize_int8(k, GROUP_T, "token")):
        assert torch.equal(got, want.contiguous())
    for got, want in zip((vq, vmn, vst), quantize_int8(v, GROUP_T, "token")):
        assert torch.equal(got, want.contiguous())


def test_full_size_prefill_quantize_properties():
    """A 32768-token, 8-head prefill: codes bit-exact with the oracle, and every
    non-degenerate group holds both a 0 and a 255 code."""
    from nova_amd.kvquant import quantize_int8

    x = bench_outliers(randn((1, 8, 32768, 128), 42, 1.0), 43)
    q, mn, st = quantize_int8(x.cuda(), 64, "token")
    rq, rm, rs = okq.quantize_int8_token(npy(x), 64)
    assert np.array_equal(npy(q), rq)
    assert _eq16(mn, rm) and _eq16(st, rs)
    qg = q.view(1, 8, 512, 64, 128)
    assert int(qg.amin(dim=3).max()) == 0 and int(qg.amax(dim=3).min()) == 255


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("axis,group,n,dim", [
    ("token", 4, 9, 128), ("token", 8, 17, 64), ("token", 9, 30, 136), ("token", 64, 65, 200),
    ("token", 0, 65, 128), ("token", 100, 333, 128), ("token", 0, 1500, 8),
    ("channel", 8, 3, 128), ("channel", 16, 65, 48), ("channel", 32, 129, 160), ("channel", 64, 64, 64),
    ("channel", 128, 1, 128), ("channel", 0, 70, 128), ("channel", 24, 66, 72), ("channel", 4, 5, 8),
])
def test_every_quantizer_route_matches_oracle(axis, group, n, dim, dtype):
    """Each split of the quantizers and the dequantizer at its edges (groups of one wave, four and
    sixteen, tails of tokens and channels, channel groups of lanes and the general ones): whole
    numbers, so the same bits."""
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    print(f"case {axis} group={group} n={n} dim={dim} {dtype}", flush=True)
    x = (torch.randn(2, 3, n, dim, generator=torch.Generator().manual_seed(n + dim)) * 2).to(dtype)
    x[..., 3] *= 8
    if axis == "token":
        rq, rm, rs = okq.quantize_int8_token(x.float().numpy(), group)
        want = okq.dequantize_int8_token(rq, rm, rs, group)
    else:
        rq, rm, rs = okq.quantize_int8_channel(x.float().numpy(), group)
        want = okq.dequantize_int8_channel(rq, rm, rs, group)
    for src in (x.cuda(), torch.zeros(2, 3, n + 5, dim, dtype=dtype).cuda()[:, :, :n].copy_(x)):
        q, mn, st = quantize_int8(src, group, axis)
        assert np.array_equal(npy(q), rq)
        assert _eq16(mn, rm) and _eq16(st, rs)
    assert _eq16(dequantize_int8(q, mn, st, group, axis), want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("rows,n,group", [
    (3, 9, 0), (3, 32, 64), (1024, 16, 0), (1025, 16, 0), (1025, 17, 32), (1025, 32, 0), (3, 33, 0), (700, 64, 0),
    (5, 65, 0), (5, 96, 100), (5, 97, 0), (512, 65, 0), (512, 96, 0), (512, 97, 0), (512, 192, 0), (512, 384, 0),
    (512, 385, 0),
])
def test_token_groups_over_the_splits_match_oracle(rows, n, group, dtype):
    """The waves that a group gets follow its tokens and the number of groups: at the edges of each, the
    oracle's codes and rulers."""
    from nova_amd.kvquant import quantize_int8

    print(f"case rows={rows} n={n} group={group} {dtype}", flush=True)
    x = (torch.randn(rows, n, 8, generator=torch.Generator().manual_seed(n + rows)) * 2).to(dtype)
    rq, rm, rs = okq.quantize_int8_token(x.float().numpy(), group)
    q, mn, st = quantize_int8(x.cuda(), group, "token")
    assert np.array_equal(npy(q), rq)
    assert _eq16(mn, rm) and _eq16(st, rs)


def _graph_us(fn, inner=10, reps=10):
    """GPU time of a call: the least of several replays of a captured run of them."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(inner):
            fn()
    best = float("inf")
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / inner)
    return best


def test_short_slabs_do_not_pay_for_long_groups():
    """A group longer than its slab is the slab: the time is that of a group of its length (it took a
    workgroup of sixteen waves for three tokens, 5.5 times as long)."""
    from nova_amd.kvquant import quantize_int8

    x = torch.randn(1000, 3, 512, dtype=torch.float16, device="cuda")
    short, long = (_graph_us(lambda: quantize_int8(x, g, "token")) for g in (3, 128))
    print(f"group 3 {short:.1f} us, group 128 {long:.1f} us", flush=True)
    assert long < 2 * short


@pytest.mark.parametrize("axis,group,rows,n,dim", [
    ("token", 8, 6, 17, 8), ("token", 9, 6, 30, 24), ("token", 64, 5, 70, 40), ("token", 0, 3, 3, 56), ("token", 8, 6, 17, 64),
    ("token", 8, 6, 17, 72), ("token", 64, 3, 180001, 8), ("channel", 8, 5, 30, 24), ("channel", 8, 6, 17, 40),
    ("channel", 16, 3, 70, 16), ("channel", 32, 5, 9, 32), ("channel", 64, 5, 33, 64), ("channel", 8, 3, 180001, 8),
    ("channel", 4, 4, 33, 24), ("channel", 24, 3, 11, 72),
])
def test_narrow_rows_match_oracle(axis, group, rows, n, dim):
    """Rows of at most 64 channels lie over a workgroup as one sequence over the slabs: slabs that do not end
    on a group, few rows and many, and inputs inside longer slabs."""
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    print(f"case {axis} group={group} rows={rows} n={n} dim={dim}", flush=True)
    x = (torch.randn(rows, n, dim, generator=torch.Generator().manual_seed(n + dim)) * 2).half()
    quantize, dequantize = ((okq.quantize_int8_token, okq.dequantize_int8_token) if axis == "token" else
                            (okq.quantize_int8_channel, okq.dequantize_int8_channel))
    rq, rm, rs = quantize(x.float().numpy(), group)
    for src in (x.cuda(), torch.zeros(rows, n + 5, dim, dtype=x.dtype).cuda()[:, :n].copy_(x)):
        q, mn, st = quantize_int8(src, group, axis)
        assert np.array_equal(npy(q), rq)
        assert _eq16(mn, rm) and _eq16(st, rs)
    assert _eq16(dequantize_int8(q, mn, st, group, axis), dequantize(rq, rm, rs, group))


@pytest.mark.parametrize("axis,group", [("token", 64), ("channel", 8)])
def test_narrow_rows_keep_their_lanes_busy(axis, group):
    """As many bytes in rows of 8 channels as in rows of 128 take about as long (three to four times, with
    15 of 16 lanes idle)."""
    from nova_amd.kvquant import dequantize_int8, quantize_int8

    times = []
    for n, dim in ((32768, 8), (2048, 128)):
        x = torch.randn(8, n, dim, dtype=torch.float16, device="cuda")
        q, mn, st = quantize_int8(x, group, axis)
        times.append((_graph_us(lambda: dequantize_int8(q, mn, st, group, axis)),
                      _graph_us(lambda: quantize_int8(x, group, axis))))
    (d8, q8), (d128, q128) = times
    print(f"dequantize {d8:.1f} / {d128:.1f} us, quantize {q8:.1f} / {q128:.1f} us", flush=True)
    assert d8 < 2 * d128
    if axis == "channel":
        assert q8 < 2.5 * q128
