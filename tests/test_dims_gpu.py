"""The matrix-core kernels of other head dims and float32 (mla_decode_dims.hip):
head_dim_v 64 to 512 and rope_dim 16 to 64 with 16-byte aligned rows, balanced
(num_splits=None: here one tile a worker; straddling ranges and longer pieces
with given worker counts) and uniform (float32 with a split count keeps the general
form, checked all the same), against the float64 oracle and, through the
C ABI, against the general forms that the same call takes when its output
rows are not 16-byte aligned.

Bars as in test_generic_gpu.py: out atol = rtol = 1e-2 for bf16 / fp16, 1e-4
for float32; lse 1e-3 / 1e-4. The general and the new form differ by the order
of float32 sums and the rounding of the probabilities (both round each once to
the element type), so two of their results lie within twice the bar.
"""

import numpy as np
import pytest
import torch

import oracle
from conftest import bits
from test_generic_gpu import NAME, TOL, _as_oracle, _paged

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32

# head_dim_v, rope_dim, dtype, heads, page size (0: dense): head-block edges
# (16, 32, 33, 128, 130), every dims class, pages that hold whole sub-tiles
# (32, 64, 128), parts of one (16) and neither (48)
CASES = [
    (64, 16, BF, 8, 0), (64, 64, HF, 130, 48), (128, 32, BF, 33, 16), (128, 64, HF, 32, 128),
    (256, 16, HF, 128, 32), (256, 32, BF, 128, 64), (256, 64, BF, 20, 16), (512, 16, BF, 64, 0),
    (512, 32, HF, 129, 64), (512, 64, F32, 16, 64), (512, 64, F32, 33, 16), (512, 16, F32, 32, 0),
    (256, 32, F32, 17, 48), (128, 64, F32, 16, 32), (64, 32, F32, 40, 64), (64, 16, F32, 1, 0),
]
# empty, one token, the edges of 16-, 32- and 64-token steps, long enough for
# several workers
LENS = [0, 1, 15, 16, 17, 31, 33, 63, 64, 65, 129, 1000, 0, 2500]


def _inputs(dv, dr, dtype, heads, page, seed, q_scale=1.0):
    g = torch.Generator().manual_seed(seed)
    lens = torch.tensor(LENS, dtype=torch.int32)
    q = (torch.randn(len(LENS), heads, dv + dr, generator=g) * q_scale).to(dtype)
    kv = torch.randn(len(LENS), max(LENS), dv + dr, generator=g).to(dtype)
    bt = None
    if page:
        kv, bt = _paged(kv, page, g)
    return q, kv, lens, bt


def _check(out, lse, q, kv, lens, bt, dv, scale, dtype):
    ref_out, ref_lse = oracle.mla_decode_ref(_as_oracle(q), _as_oracle(kv), lens.numpy(),
                                             None if bt is None else bt.numpy(), dv, scale, dtype=NAME[dtype])
    otol, ltol = TOL[dtype]
    torch.testing.assert_close(out.float().cpu(), torch.from_numpy(ref_out), atol=otol, rtol=otol)
    some = lens > 0
    torch.testing.assert_close(lse.cpu()[some], torch.from_numpy(ref_lse)[some], atol=ltol, rtol=ltol)
    assert torch.all(out.cpu()[~some] == 0) and torch.all(torch.isneginf(lse.cpu()[~some]))
    row = kv[1, 0] if bt is None else kv[bt[1, 0].long(), 0]  # one token: the row itself
    assert torch.equal(out[1].cpu(), row[:dv].expand(out.shape[1], dv))


@pytest.mark.parametrize("splits", [None, 1, 5])
@pytest.mark.parametrize("dv,dr,dtype,heads,page", CASES)
def test_dims_match_oracle(gpu, dv, dr, dtype, heads, page, splits):
    from triton_mla import mla_decode

    print(f"dims {dv}+{dr} {NAME[dtype]} heads={heads} page={page} splits={splits}", flush=True)
    q, kv, lens, bt = _inputs(dv, dr, dtype, heads, page, dv + dr + heads)
    for scale in ((dv + dr) ** -0.5, -0.25):  # (a spread that moves the reference max late, and negative)
        out, lse = mla_decode(q.to(gpu), kv.to(gpu), lens.to(gpu), None if bt is None else bt.to(gpu), head_dim_v=dv,
                              softmax_scale=scale, num_splits=splits, return_lse=True)
        torch.cuda.synchronize()
        _check(out, lse, q, kv, lens, bt, dv, scale, dtype)


def _balanced(lib, gpu, q, kv, lens, bt, dv, dr, scale, workers):
    """tmla_mla_decode_generic_balanced with a given worker count."""
    from triton_mla import _native

    batch, heads, dtype = q.shape[0], q.shape[1], q.dtype
    gq, gkv, gl, gbt = q.to(gpu), kv.to(gpu), lens.to(gpu), None if bt is None else bt.to(gpu)
    out = torch.full((batch, heads, dv), 7.0, dtype=dtype, device=gpu)
    lse = torch.full((batch, heads), 7.0, device=gpu)
    ws = torch.empty(lib.tmla_generic_balanced_workspace_bytes(batch, heads, dv, workers), dtype=torch.uint8, device=gpu)
    _native.check(lib.tmla_mla_decode_generic_balanced(
        gq.data_ptr(), gq.stride(0), gq.stride(1), gkv.data_ptr(), gkv.stride(0), gkv.stride(1),
        gkv.shape[1] if bt is None else gkv.shape[0], 1 if bt is None else gkv.shape[1],
        None if bt is None else gbt.data_ptr(), 0 if bt is None else gbt.stride(0), 1 if bt is None else gbt.shape[1],
        gl.data_ptr(), batch, heads, dv, dr, _native.DTYPE_CODE[dtype], scale, workers, out.data_ptr(), out.stride(0),
        out.stride(1), lse.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "balanced")
    torch.cuda.synchronize()
    return out, lse


# every kernel class (16 bits up to 256 dims and at 512, float32 with 16 and
# 32 heads a workgroup), a dense cache, pages of whole sub-tiles and smaller
SEGMENT_CASES = [
    (64, 16, HF, 33, 0), (128, 64, BF, 130, 16), (256, 32, BF, 128, 64), (256, 64, HF, 20, 48), (512, 32, BF, 64, 32),
    (512, 16, HF, 129, 0), (512, 64, F32, 16, 64), (256, 32, F32, 40, 16), (64, 16, F32, 33, 0),
]


@pytest.mark.parametrize("workers,snapped", [(5, False), (1, False), (30, True)])
@pytest.mark.parametrize("dv,dr,dtype,heads,page", SEGMENT_CASES)
def test_dims_ranges_across_sequences(gpu, dv, dr, dtype, heads, page, workers, snapped):
    """Ranges over several sequences (the next segment reuses the ring, Q and
    the merge area in LDS, and starts mid-range on the partition's line), empty
    ones between them, and snapped pieces of several tiles."""
    from triton_mla import _native

    q, kv, lens, bt = _inputs(dv, dr, dtype, heads, page, 3 * dv + heads)
    tiles = [-(-n // 64) for n in lens.tolist()]
    chunk = -(-sum(tiles) // workers)
    assert chunk > 1 and (sum(-(-t // chunk) for t in tiles) <= workers) == snapped
    print(f"segments {dv}+{dr} {NAME[dtype]} heads={heads} page={page} workers={workers}", flush=True)
    out, lse = _balanced(_native.load(), gpu, q, kv, lens, bt, dv, dr, 0.2, workers)
    _check(out, lse, q, kv, lens, bt, dv, 0.2, dtype)


@pytest.mark.parametrize("dtype", [BF, F32])
def test_dims_many_sequences(gpu, dtype):
    """More than 64 sequences (each lane of the partition takes several):
    snapped and straddling ranges."""
    from triton_mla import _native

    g = torch.Generator().manual_seed(21)
    dv, dr, heads, batch = 128, 32, 17, 150
    lens = torch.randint(0, 300, (batch,), generator=g, dtype=torch.int32)
    lens[[1, 3, 70]] = torch.tensor([1, 0, 64], dtype=torch.int32)
    q = torch.randn(batch, heads, dv + dr, generator=g).to(dtype)
    kv, bt = _paged(torch.randn(batch, 300, dv + dr, generator=g).to(dtype), 64, g)
    for workers in (600, 40):
        print(f"150 sequences {NAME[dtype]} workers={workers}", flush=True)
        out, lse = _balanced(_native.load(), gpu, q, kv, lens, bt, dv, dr, 0.2, workers)
        _check(out, lse, q, kv, lens, bt, dv, 0.2, dtype)


@pytest.mark.parametrize("dtype", [BF, F32])
def test_dims_strided_rows_and_cut_lengths(gpu, dtype):
    """q and the cache as slices of wider tensors, a table with spare columns
    and ids past the cache, and lengths beyond what the cache holds (cut to
    it), as the general forms take them."""
    from triton_mla import mla_decode

    g = torch.Generator().manual_seed(11)
    dv, dr, heads, page = 256, 32, 24, 64
    d = dv + dr
    wide_q = torch.randn(3, 2 * heads, d + 32, generator=g).to(dtype)
    wide_kv = torch.randn(12, page, d + 64, generator=g).to(dtype)
    table = torch.randperm(12, generator=g).view(3, 4).int()
    q, kv = wide_q[:, ::2, :d], wide_kv[:, :, :d]
    lens = torch.tensor([256, 100000, 130], dtype=torch.int32)
    cut = torch.tensor([256, 256, 130], dtype=torch.int32)
    gq, gkv = wide_q.to(gpu)[:, ::2, :d], wide_kv.to(gpu)[:, :, :d]
    print(f"strided {NAME[dtype]}", flush=True)
    out, lse = mla_decode(gq, gkv, lens.to(gpu), table.to(gpu), head_dim_v=dv, softmax_scale=0.1, return_lse=True)
    torch.cuda.synchronize()
    ref_out, ref_lse = oracle.mla_decode_ref(_as_oracle(q), _as_oracle(kv), cut.numpy(), table.numpy(), dv, 0.1,
                                             dtype=NAME[dtype])
    otol, ltol = TOL[dtype]
    torch.testing.assert_close(out.float().cpu(), torch.from_numpy(ref_out), atol=otol, rtol=otol)
    torch.testing.assert_close(lse.cpu(), torch.from_numpy(ref_lse), atol=ltol, rtol=ltol)


@pytest.mark.parametrize("dv,dr,dtype,heads,page", CASES[1:9:2])
def test_dims_agree_with_general_form(gpu, dv, dr, dtype, heads, page):
    """The same C ABI call with a 16-byte aligned output (these kernels) and
    with output rows one element off (the general forms)."""
    from triton_mla import _native

    lib = _native.load()
    q, kv, lens, bt = _inputs(dv, dr, dtype, heads, page, 5)
    gq, gkv, gl = q.to(gpu), kv.to(gpu), lens.to(gpu)
    gbt = None if bt is None else bt.to(gpu)
    batch, splits = len(LENS), 3
    ws = torch.empty(lib.tmla_generic_workspace_bytes(batch, heads, dv, splits), dtype=torch.uint8, device=gpu)
    print(f"general {dv}+{dr} {NAME[dtype]} heads={heads} page={page}", flush=True)
    outs = []
    for pad in (0, 1):
        out = torch.zeros(batch, heads, dv + pad, dtype=dtype, device=gpu)
        lse = torch.zeros(batch, heads, dtype=torch.float32, device=gpu)
        _native.check(lib.tmla_mla_decode_generic(
            gq.data_ptr(), gq.stride(0), gq.stride(1), gkv.data_ptr(), gkv.stride(0), gkv.stride(1),
            gkv.shape[0] if page else gkv.shape[1], page or 1, None if gbt is None else gbt.data_ptr(),
            0 if gbt is None else gbt.stride(0), 1 if gbt is None else gbt.shape[1], gl.data_ptr(), batch, heads, dv, dr,
            _native.DTYPE_CODE[dtype], 0.11, splits, out.data_ptr(), out.stride(0), out.stride(1), lse.data_ptr(),
            ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "generic")
        torch.cuda.synchronize()
        outs.append((out[..., :dv].float().cpu(), lse.cpu()))
    otol, ltol = TOL[dtype]
    torch.testing.assert_close(outs[0][0], outs[1][0], atol=2 * otol, rtol=2 * otol)
    some = lens > 0
    torch.testing.assert_close(outs[0][1][some], outs[1][1][some], atol=2 * ltol, rtol=2 * ltol)


def test_dims_graph_replay(gpu):
    """The balanced form captured in a HIP graph and replayed with new
    contents gives the eager results."""
    from triton_mla import mla_decode

    q, kv, lens, bt = (t.to(gpu) for t in _inputs(256, 32, BF, 32, 64, 3))
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        mla_decode(q, kv, lens, bt, head_dim_v=256)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out = mla_decode(q, kv, lens, bt, head_dim_v=256)
    for k in range(3):
        lens.copy_(torch.roll(lens, 1))
        kv.mul_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, mla_decode(q, kv, lens, bt, head_dim_v=256))
