"""The Voduvik design on the GPU, mechanism by mechanism and end to end, against the plain restatement (oracle/voduvik.py, float64).

float32 runs of the kernels are compared tightly: there a wrong key, position, page or state shows at once.  bfloat16 runs are
compared within what rounding explains, and with inputs that make one key stand out where an average would hide it."""
from __future__ import annotations

import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import voduvik as plain
from tests import tile_cases, voduvik_cases as cases

pytestmark = pytest.mark.gpu
REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BOTH = [torch.float32, torch.bfloat16]


def dev():
    return torch.device("cuda:0")


def i32(v):
    return torch.as_tensor(np.asarray(v), dtype=torch.int32).to(dev())


def close(got, want, dtype, tol32=2e-5, tol16=2e-2):
    got, want = got.double().cpu(), want.double().cpu()
    scale = float(want.abs().max()) + 1e-6
    err = float((got - want).abs().max()) / scale
    assert err <= (tol32 if dtype == torch.float32 else tol16), f"max|d| / max = {err:.3e}"


def layout(counts, ctx, tables, page, slots=None, flips=None, pos_slots=True):
    """A StepLayout for portions of `counts` tokens behind `ctx` ones."""
    from vllmini_amd import hybrid_ops as ops

    counts, ctx = np.asarray(counts), np.asarray(ctx)
    starts = np.cumsum(counts) - counts
    seq = np.repeat(np.arange(len(counts)), counts)
    pos = np.arange(counts.sum()) - np.repeat(starts, counts) + np.repeat(ctx, counts)
    tables = np.asarray(tables)
    slot = tables[seq, pos // page] * page + pos % page if pos_slots else np.full(len(seq), -1)
    f = dict(tok_seq=i32(seq), tok_pos=i32(pos), tok_slot=i32(slot), q_start=i32(starts), q_len=i32(counts), ctx=i32(ctx),
             state_slot=i32(range(len(counts)) if slots is None else slots), flip=i32([0] * len(counts) if flips is None else flips),
             table=i32(tables))
    if (counts > 1).any():
        per = -(-counts // ops.CHUNK_ROWS)
        f["chunk_start"] = i32(np.cumsum(per) - per)
        f["chunks"] = i32([(b, 16 * c) for b in range(len(counts)) for c in range(per[b])])
    spans = bool((starts // ops.ROW_TILE != (starts + counts - 1) // ops.ROW_TILE).any())
    return ops.StepLayout(f, int(counts.sum()), len(counts), page, bool((counts == 1).all()), spans, int(counts.max()),
                          int((ctx + counts).max()))


@pytest.mark.parametrize("ints,n", [(4, 1), (1028, 0), (1 << 15, 300)])
def test_a_steps_inputs_arrive(ints, n):
    from vllmini_amd import hybrid_ops as ops
    from vllmini_amd.staging import PinnedBuffer

    buf, ids = PinnedBuffer(4 * ints + 64), torch.arange(7, 7 + n, device=dev())
    for turn in (1, 2):
        buf.wait()
        buf.tensor.copy_(torch.randint(0, 255, buf.tensor.shape, dtype=torch.uint8, generator=torch.Generator().manual_seed(turn)))
        to, out = torch.zeros(ints, dtype=torch.int32, device=dev()), torch.full((n + 2,), -1, dtype=torch.int64, device=dev())
        ops.step_inputs(buf, to, ids, out)
        assert torch.equal(to.cpu(), buf.tensor[: 4 * ints].view(torch.int32)) and out.tolist() == [*range(7, 7 + n), -1, -1]
    with pytest.raises(RuntimeError):
        ops.step_inputs(buf, torch.zeros(ints + 20, dtype=torch.int32, device=dev()), ids, out)


# ---- linear layers ---------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("M", [1, 5, 17, 40, 130])
@pytest.mark.parametrize("N,K", [(32, 32), (96, 288), (352, 800), (1056, 1312)])
def test_linear_kinds(dtype, M, N, K):
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator().manual_seed(M * N + K)
    rnd = lambda *s: torch.randn(*s, generator=g)      # noqa: E731
    x, w = rnd(M, K).to(dtype).to(dev()), (rnd(N, K) / K ** 0.5).to(torch.bfloat16).to(dev())
    t = ops.MatrixTiles(w, dtype)
    W = w.double()
    bias = rnd(N).to(dev())
    close(ops.linear(x, t, bias=bias), x.double() @ W.T + bias.double(), dtype)
    base = rnd(M, N).to(dev())
    close(ops.linear(x, t, residual=True, out=base.clone()), base.double() + x.double() @ W.T, dtype, tol16=1e-3)
    # normalised rows, with a mean far from zero and a ragged true length
    n = K - 13
    xf, nw = (rnd(M, K) * 3 + 40).to(dev()), torch.zeros(K, device=dev())
    xf[:, n:] = 0
    nw[:n] = 1 + 0.5 * rnd(n).to(dev())
    h = torch.zeros(M, K, dtype=torch.float64, device=dev())
    h[:, :n] = plain.layer_norm(xf[:, :n].double(), nw[:n].double(), 1e-5)
    close(ops.linear(xf, t, norm=(nw, n, 1e-5)), h @ W.T, dtype, tol32=1e-4)
    rows = torch.tensor([M - 1, 0, M // 2], dtype=torch.int32, device=dev())
    cols = N - 5
    close(ops.linear(xf, t, norm=(nw, n, 1e-5), rows=rows, float_out=(cols, 0.3)), (h @ W.T)[rows.long(), :cols] * 0.3, dtype, tol32=1e-4)
    y = h @ W.T
    gate, up = y[:, 0::2].clamp(max=0.8), y[:, 1::2].clamp(-0.8, 0.8)
    close(ops.linear(xf, t, norm=(nw, n, 1e-5), glu=ops.GatedUnit.clamped(0.8)), gate * torch.sigmoid(1.702 * gate) * (up + 1), dtype, tol32=1e-4, tol16=3e-2)
    if K % 64 == 0:
        a, b = rnd(M, K // 2).to(dev()), rnd(M, K // 2).to(dev())
        close(ops.linear(a, t, x2=b, float_out=(N, 1.0)), torch.cat([a, b], 1).double() @ W.T, dtype)


@pytest.mark.parametrize("M,N,K", [(1, 32, 32), (16, 96, 224), (17, 160, 288), (3, 2048, 1024), (50, 512, 1056), (64, 1024, 2048), (33, 64, 512)])
def test_few_rows_behind_a_norm_split_k_over_the_waves(M, N, K):
    """rows_kernel where its waves have unequal parts of K, or none; row tiles that are not full; several of them."""
    _norm_products(M, N, K)


@pytest.mark.parametrize("M,N,K", [(1, 16 * 530, 256), (2, 16 * 600, 288), (3, 16 * 514, 1024), (5, 32, 4096), (8, 16 * 1030, 320), (16, 16 * 258, 2080), (17, 16 * 512, 256),
                                   (12, 512, 4096), (32, 16 * 515, 1024), (31, 16 * 600, 2048)])
def test_rows_behind_a_norm_stay_in_lds(M, N, K):
    """resident_kernel at the edges of what it deals out: rows over waves, k-steps over waves, slabs over workgroups (fewer, one more than a round,
    several), one and two places for partial tiles."""
    from vllmini_amd import hybrid_ops as ops

    t = _norm_products(M, ops.pad32(N), K)
    assert ops.linear_resident(M, t) and not ops.linear_resident(33, t)


@pytest.mark.parametrize("M,N,K", [(9, 32, 4096), (16, 16384, 4096), (12, 1024, 4128), (17, 4128, 4096), (32, 8192, 4096), (33, 64, 4096), (47, 4128, 4128), (70, 256, 4096)])
def test_rows_are_normed_once_before_the_product(M, N, K):
    """norm_first: at its borders, and kept to bfloat16 on one group (the same bound: one rounding of the normed rows either way)."""
    from vllmini_amd import hybrid_ops as ops

    asks = lambda m, n, k, groups=1, dtype=torch.bfloat16: bool(ops.load().vmi_hy_linear_normed(m, n, k, groups, ops.DTYPES[dtype]))      # noqa: E731
    assert asks(M, N, K) and not asks(M, N, K, 2) and not asks(M, N, K, 1, torch.float32)
    assert not asks(8, N, K) and not asks(16, 4 * 4096 + 16, 4096) and not asks(32, 8192, 4064) and asks(32, 24576, 4096)
    _norm_products(M, ops.pad32(N), K)


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("M,N,K", [(12, 512, 4096), (12, 512, 512), (3, 64, 9216)])
def test_columns_behind_the_norm_do_not_count(M, N, K, rms):
    """The norm is over its first columns, wherever it happens (before the product, in rows_kernel, in linear_kernel): what the rows hold behind them
    (the weight is zero there) changes no bit, and add_norm leaves them out of its mean too."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M + K)
    n, x = K - 28, torch.randn(M, K, generator=g, device=dev())
    t = ops.MatrixTiles((torch.randn(N, K, generator=g, device=dev()) / K ** 0.5).to(torch.bfloat16), torch.bfloat16)
    nw = torch.zeros(K, device=dev())
    nw[:n] = 1
    clean, dirty = x.clone(), x.clone()
    clean[:, n:], dirty[:, n:] = 0, 1000
    a, b = (ops.linear(v, t, norm=(nw, n, 1e-5, rms)) for v in (clean, dirty))
    assert torch.equal(a, b)
    a, b = (ops.add_norm(v, None, (nw, n, 1e-5, rms), torch.bfloat16) for v in (clean, dirty))
    assert torch.equal(a[:, :n], b[:, :n])


@pytest.mark.parametrize("stride", [0, 4096])
def test_groups_behind_a_norm_read_the_same_rows_normed_once_or_not(stride):
    """vmi_hy_linear of two groups behind a norm: x_gstride means nothing there, with room for normed rows or without."""
    import ctypes

    from vllmini_amd import hybrid_ops as ops

    M, N, K = 12, 64, 4096
    g = torch.Generator(device=dev()).manual_seed(stride)
    x, w = torch.randn(M, K, generator=g, device=dev()), torch.randn(2 * N, K, generator=g, device=dev()) / K ** 0.5
    t = [ops.MatrixTiles(w[i * N:(i + 1) * N].to(torch.bfloat16), torch.bfloat16).tiles.flatten() for i in range(2)]
    tiles, nw = torch.cat(t), torch.ones(K, device=dev())
    normed = torch.full((M, K), 7.0, dtype=torch.bfloat16, device=dev())
    got = []
    for room in (None, normed.data_ptr()):
        y = torch.zeros(M, 2 * N, dtype=torch.bfloat16, device=dev())
        a = ops.LinearArgs(x=x.data_ptr(), norm_w=nw.data_ptr(), w=tiles.data_ptr(), y=y.data_ptr(), normed=room, ldx=K, ldy=2 * N, x_gstride=stride, y_gstride=N, M=M,
                           N=N, K=K, groups=2, norm_n=K, eps=1e-5, x_kind=1, epilogue=0, dtype=ops.DTYPES[torch.bfloat16])
        assert ops.load().vmi_hy_linear(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
        got.append(y)
    h = torch.nn.functional.layer_norm(x.double(), (K,), nw.double(), None, 1e-5) @ w.to(torch.bfloat16).double().T
    for y in got:
        close(y, h, torch.bfloat16)


@pytest.mark.parametrize("M,N,K", [(16, 6144, 3072), (12, 16 * 1026, 4096), (9, 16 * 1540, 4096), (17, 16 * 514, 256), (24, 8192, 1024), (32, 16384, 1536), (20, 16 * 1538, 3072),
                                   (16, 16 * 1026, 512), (16, 16 * 2046, 544)])
def test_rows_behind_a_norm_stay_in_lds_and_are_not_normed_first(M, N, K):
    """resident_kernel where no rule stands in front of it: one workgroup a compute unit with one row tile and with two, and just past the lines at which
    linear_kernel takes over."""
    from vllmini_amd import hybrid_ops as ops

    t = _norm_products(M, N, K)
    assert ops.linear_resident(M, t) and not ops.linear_normed_first(M, t)


@pytest.mark.parametrize("M,N,K", [(16, 16 * 1024, 512), (9, 16 * 2048, 256), (9, 16 * 3072, 512), (17, 16 * 512, 512), (25, 8192, 1024), (32, 16 * 1024, 992), (17, 16 * 1536, 1280)])
def test_rows_that_could_stay_in_lds_but_are_few_and_short(M, N, K):
    _norm_products(M, N, K)


@pytest.mark.parametrize("M,N,K", [(31, 16 * 1542, 1024), (32, 16 * 1536, 2048)])
def test_many_columns_leave_the_rows_in_lds(M, N, K):
    _norm_products(M, N, K)


@pytest.mark.parametrize("M,N,K,slabs", [(7, 16 * 515, 1024, 3), (33, 16 * 387, 1024, 6), (17, 16 * 389, 1024, 4), (64, 16 * 130, 1024, 3), (40, 16 * 510, 1024, 6), (3, 16 * 257, 2048, 2),
                                         (31, 16 * 129, 2048, 2), (18, 16 * 254, 1536, 2), (5, 16 * 99, 1536, 1), (50, 16 * 129, 768, 4), (40, 16 * 254, 512, 4), (90, 16 * 85, 256, 4),
                                         (21, 16 * 200, 96, 2), (35, 16 * 330, 992, 4), (9, 16 * 255, 1056, 1), (20, 16 * 201, 1152, 2), (33, 16 * 77, 1280, 1), (64, 16 * 127, 1792, 2),
                                         (1, 16 * 511, 1888, 2), (47, 32, 2016, 1)])
def test_few_rows_behind_a_norm_take_several_slabs_a_workgroup(M, N, K, slabs):
    """norm_rows_kernel with one to six slabs of 16 columns a workgroup, the last workgroup's not all there, for every length of a row it is built for, shared
    out evenly and not."""
    from vllmini_amd import hybrid_ops as ops

    w = _norm_products(M, ops.pad32(N), K)
    assert ops.linear_slabs(M, w) == slabs and not ops.linear_normed_first(M, w)


@pytest.mark.parametrize("M,N,K", [(9, 16 * 513, 2048), (16, 16 * 1030, 2048), (32, 16 * 770, 2048), (33, 16 * 400, 2048), (64, 16 * 514, 2048), (50, 16 * 770, 1024), (12, 16 * 258, 4096),
                                   (40, 16 * 514, 4096), (33, 32, 3072), (50, 16 * 258, 3072), (40, 16 * 34, 3072), (64, 16 * 514, 3072), (16, 16 * 386, 4096), (32, 16 * 770, 4096)])
def test_rows_normed_once_are_held_in_registers(M, N, K):
    """held_rows_kernel: one and two row tiles, row blocks, slabs that the workgroups do not share evenly, several chunks of K a slab and one."""
    from vllmini_amd import hybrid_ops as ops

    assert ops.linear_normed_first(M, _norm_products(M, ops.pad32(N), K))


@pytest.mark.parametrize("M,K,wgs,slabs", [(3, 1024, 512, (4, 5, 6, 7, 8)), (16, 2048, 256, (3, 4, 5, 6)), (5, 2048, 512, (2, 3, 4)), (1, 4096, 512, (1, 2)), (20, 1024, 512, (2, 4, 5, 6, 7)),
                                           (32, 2048, 256, (2, 3, 4, 5)), (50, 1024, 128, (4, 5, 6, 7, 8, 9)), (40, 3072, 128, (1, 2, 3, 4))])
def test_every_number_of_slabs_behind_the_rings_last_round(M, K, wgs, slabs):
    """resident_kernel and held_rows_kernel over whole chunks of K: `slabs` of a workgroup's are all that the longest walks have, one workgroup's; the others' are one less."""
    for n in slabs:
        _norm_products(M, 16 * (wgs * (n - 1) + 2), K)


@pytest.mark.parametrize("M", [1, 16, 33, 64])
@pytest.mark.parametrize("N,K", [(48, 32), (16 * 130, 128), (32, 224), (16 * 133, 480), (16 * 131, 992), (64, 1024), (16 * 129, 2016), (32, 2080), (96, 3072), (32, 4064), (48, 4576), (32, 4640),
                                 (16 * 130, 4640), (48, 9248), (16 * 386, 96), (16 * 258, 1056), (16 * 514, 2080), (16 * 386, 8224)])
def test_few_rows_as_they_are(M, N, K):
    """plain_rows_kernel: K in one chunk a wave and in several, waves with unequal parts or none, one and two row tiles a workgroup; the rows of a wider matrix; linear_kernel past
    the line between them."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M * K + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    N = ops.pad32(N)
    w = (rnd(N, K) / K ** 0.5).to(torch.bfloat16)
    t, x, bias, base = ops.MatrixTiles(w, torch.bfloat16), rnd(M, K + 8).to(torch.bfloat16)[:, :K], rnd(N), rnd(M, N)
    y = x.double() @ w.double().T
    close(ops.linear(x, t, bias=bias), y + bias, torch.bfloat16)
    close(ops.linear(x, t, residual=True, out=base.clone()), base.double() + y, torch.bfloat16, tol16=1e-3)


@pytest.mark.parametrize("K", [6144, 8192, 12288])
@pytest.mark.parametrize("M,slabs", [(1, 3), (2, 512), (3, 130), (8, 514), (9, 66), (16, 384), (17, 96), (32, 128), (50, 6)])
def test_rows_as_they_are_over_whole_chunks(M, slabs, K):
    """plain_rows_kernel's form for waves of whole chunks, with requests for two, eight and sixteen rows, and linear_kernel past its line; gated by a column as well."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M * K + slabs)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    N = 16 * slabs
    w = (rnd(ops.pad32(N), K) / K ** 0.5).to(torch.bfloat16)
    t, x, bias, base, gate = ops.MatrixTiles(w, torch.bfloat16), rnd(M, K + 8).to(torch.bfloat16)[:, :K], rnd(len(w)), rnd(M, len(w)), rnd(M, 1).to(torch.bfloat16)
    y = x.double() @ w.double().T
    close(ops.linear(x, t, bias=bias), y + bias, torch.bfloat16)
    close(ops.linear(x, t, residual=True, out=base.clone()), base.double() + y, torch.bfloat16, tol16=1e-3)
    close(ops.linear(x, t, gate=gate), y * torch.sigmoid(gate.double()), torch.bfloat16)


@pytest.mark.parametrize("groups,K,N,pad", [(2, 64, 32, 0), (3, 128, 512, 64), (16, 192, 96, 8), (5, 512, 128, 16), (4, 96, 64, 0), (2, 320, 4096, 0)])
@pytest.mark.parametrize("M", [65, 130, 400, 1100])
def test_groups_of_many_rows(groups, K, N, pad, M):
    """group_tiles_kernel, linear_kernel past its line (K no whole chunks of 64, short K): groups whose columns of x overlap, stored
    with a bias and gated, into columns of a wider matrix.  (The list of tiles: test_each_tile_by_itself_over_a_group.)"""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M * K + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    step, wide = K // 2 + pad, N + 32
    w = (rnd(groups, N, K) / K ** 0.5).to(torch.bfloat16)
    t, x = ops.MatrixTiles(w, torch.bfloat16), rnd(M, (groups - 1) * step + K + 8).to(torch.bfloat16)
    gate, bias = rnd(M, groups).to(torch.bfloat16), rnd(N)
    cols = torch.stack([x[:, i * step:i * step + K] for i in range(groups)]).double()
    want = torch.bmm(cols, w.double().transpose(1, 2).contiguous())      # [groups, M, N]
    for kind in ("bias", "gate"):
        out = torch.full((M, groups * wide), 7.0, dtype=torch.bfloat16, device=dev())
        ops.linear(x, t, x_gstride=step, y_gstride=wide, out=out, **({"bias": bias} if kind == "bias" else {"gate": gate}))
        y = out.view(M, groups, wide)
        close(y[..., :N].transpose(0, 1), want + bias if kind == "bias" else want * torch.sigmoid(gate.double()).T[..., None], torch.bfloat16)
        assert (y[..., N:] == 7).all()


@pytest.mark.parametrize("M", [1, 2, 3, 8, 9, 16, 17])
@pytest.mark.parametrize("N,K", [(48, 64), (128, 448), (16 * 30, 1024), (96, 1984), (64, 2112), (16 * 70, 4608), (32, 6144), (16 * 20, 8192), (48, 12288), (64, 10240)])
def test_few_rows_side_by_side(M, N, K):
    """plain_rows_kernel over two float32 halves: waves whose parts lie in one and in both, K in one chunk a wave and in several, linear_kernel past its lines; some of the columns, scaled."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M * K + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    a, b, w = rnd(M, K // 2 + 8)[:, :K // 2], rnd(M, K // 2 + 8)[:, :K // 2], (rnd(ops.pad32(N), K) / K ** 0.5).to(torch.bfloat16)
    want = torch.cat([a, b], 1).to(torch.bfloat16).double() @ w.double().T
    got = ops.linear(a, ops.MatrixTiles(w, torch.bfloat16), x2=b, float_out=(N - 3, 0.5))
    close(got, 0.5 * want[:, :N - 3], torch.bfloat16, tol16=1e-5)      # (products of 16 bits are exact in 32: what is left is the order of a float32 sum)


@pytest.mark.parametrize("K", [10240, 14336, 16384])
@pytest.mark.parametrize("M,slabs", [(1, 3), (2, 512), (8, 130), (9, 66), (16, 384), (17, 96)])
def test_rows_as_they_are_over_every_number_of_whole_chunks(M, slabs, K):
    """As above over the other multiples of 2048 up to 16 384; two float32 halves side by side too."""
    from vllmini_amd import hybrid_ops as ops

    test_rows_as_they_are_over_whole_chunks(M, slabs, K)
    g = torch.Generator(device=dev()).manual_seed(M + K)
    a, b, w = (torch.randn(*s, generator=g, device=dev()) for s in ((M, K // 2), (M, K // 2), (16 * slabs + 16 * (slabs & 1), K)))
    w = (w / K ** 0.5).to(torch.bfloat16)
    want = torch.cat([a, b], 1).to(torch.bfloat16).double() @ w.double().T
    close(ops.linear(a, ops.MatrixTiles(w, torch.bfloat16), x2=b, float_out=(16 * slabs, 1.0)), want[:, :16 * slabs], torch.bfloat16, tol16=1e-5)


def _norm_products(M, N, K):
    """Every epilogue behind a norm against float64, the norm over fewer columns than there are; returns the weights."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M * K + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    t = ops.MatrixTiles((rnd(N, K) / K ** 0.5).to(torch.bfloat16), torch.bfloat16, dense=True)
    n, x, bias = K - 13, rnd(M + 2, K + 8)[:, :K] * 3 + 40, rnd(N)
    nw = torch.zeros(K, device=dev())
    nw[:n] = 1 + 0.5 * rnd(n)
    x[:, n:] = 0
    for rms in (False, True):
        d = x[:, :n].double()
        h = torch.zeros(M + 2, K, dtype=torch.float64, device=dev())
        h[:, :n] = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * nw[:n] if rms else plain.layer_norm(d, nw[:n].double(), 1e-5)
        y, norm = h @ t.dense.double().T, (nw, n, 1e-5, rms)
        close(ops.linear(x[:M], t, norm=norm, bias=bias), y[:M] + bias, torch.bfloat16)
        rows = torch.arange(M + 1, 1, -1, dtype=torch.int32, device=dev())
        close(ops.linear(x, t, norm=norm, rows=rows, float_out=(N - 5, 0.3)), y[rows.long(), : N - 5] * 0.3, torch.bfloat16)
        gate, up = y[:M, 0::2].clamp(max=0.8), y[:M, 1::2].clamp(-0.8, 0.8)
        close(ops.linear(x[:M], t, norm=norm, glu=ops.GatedUnit.clamped(0.8)), gate * torch.sigmoid(1.702 * gate) * (up + 1), torch.bfloat16, tol16=3e-2)
        split, rest = 16 * (N // 32), torch.empty((M, (N - 16 * (N // 32)) // 2), dtype=torch.bfloat16, device=dev())
        close(ops.linear(x[:M], t, norm=norm, glu=ops.SILU_UNIT, glu_from=split, glu_out=rest), y[:M, :split], torch.bfloat16)
        close(rest, F.silu(y[:M, split::2]) * y[:M, split + 1::2], torch.bfloat16, tol16=3e-2)
    return t


@pytest.mark.parametrize("M,N,K,split", [(1, 16, 64, 0), (17, 96, 128, 32), (300, 3088, 320, 16), (1063, 5408, 192, 5408 - 32), (770, 5392, 128, 0), (1442, 6160, 128, 4096), (641, 5920, 576, 48),
                                         (323, 5424, 832, 0), (481, 5392, 64, 2048), (130, 5472, 768, 0), (129, 5552, 1984, 64), (2100, 768, 3072, 256)])
def test_many_rows_in_tiles_with_the_gated_unit_behind(M, N, K, split):
    """vmi_hy_linear_tiles: rows and columns left over, one chunk of K, two, an odd number of them and many; the line between columns as they
    are and gated ones inside tiles; outputs that are columns of wider tensors, whose others stay as they were.  (The list of tiles: test_each_tile_by_itself.)"""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M + N + K)
    x, w = (torch.randn(*s, generator=g, device=dev()) for s in ((M, K), (N, K)))
    N = ops.pad32(N)
    t = ops.MatrixTiles(w / K ** 0.5, torch.bfloat16, dense=True)
    x = torch.cat([x, x], 1).to(torch.bfloat16)[:, K:]
    y = x.double() @ t.dense.double().T
    for unit in (ops.SILU_UNIT, ops.GatedUnit.clamped(0.7)):
        wide = torch.full((M, (N - split) // 2 + 24), 7.0, dtype=torch.bfloat16, device=dev())
        out = ops.linear_tiles(x, t, unit, split, wide[:, 8:-16])
        # as glu() over the rounded product, which is another only where a sum in another order rounds the other way (K products in float32: one in hundreds)
        other = ops.glu(y[:, split:].to(torch.bfloat16).contiguous(), unit)
        differ = wide[:, 8:-16] != other
        assert float(differ.float().mean()) <= 0.02
        a, b = y[:, split::2].clamp(max=unit.limit), y[:, split + 1::2].clamp(-unit.limit, unit.limit)
        want = a * torch.sigmoid(unit.alpha * a) * (b + unit.up)
        # (half a unit of bfloat16 in the gate, in up and in the result; the unit's slope in the gate is at most 1.2 alpha^0 (b + up), its value at most the gate's)
        bound = 2.0 ** -8 * (want.abs() + 1.2 * a.abs() * (b + unit.up).abs() + a.abs() * y[:, split + 1::2].abs()) + 1e-4
        assert bool(((wide[:, 8:-16].double() - want).abs() <= bound).all())
        assert bool((wide[:, :8] == 7).all()) and bool((wide[:, -16:] == 7).all())
        if split:
            assert out.shape == (M, split) and bool(((out.double() - y[:, :split]).abs() <= 2.0 ** -8 * y[:, :split].abs() + 1e-3).all())


@pytest.mark.parametrize("M,N,K", [(2029, 6560, 768), (2507, 7232, 256), (1859, 3232, 512), (963, 5920, 1152), (2026, 4416, 128), (321, 7552, 128), (269, 6560, 512),
                                   (257, 6560, 1152), (769, 7616, 128), (391, 6560, 1536), (195, 7104, 128), (199, 7008, 256), (130, 6752, 640), (70, 5472, 512),
                                   (66, 5984, 640), (1, 32, 384), (5, 32, 512), (1, 160, 1152), (1, 160, 64)])
def test_products_of_many_rows_alone(M, N, K):
    """vmi_hy_product_tiles: rows, columns and chunks of K left over, rows of a wider tensor; in bfloat16 with a bias in 32 bits (half a unit of the result) and in
    32 bits (K products summed in another order).  Beside the result nothing is written."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M + N + K)
    x, w, b = (torch.randn(*s, generator=g, device=dev()) for s in ((M, 2 * K), (N, K), (N,)))
    t = ops.MatrixTiles(w / K ** 0.5, torch.bfloat16, dense=True)
    x = x.to(torch.bfloat16)[:, K:]
    y = x.double() @ t.dense.double().T
    err = 2.0 ** -24 * K ** 0.5 * 8 * (x.double().abs() @ t.dense.double().abs().T) / K ** 0.5
    got = ops.product_tiles(x, t, float_out=True)
    assert got.dtype == torch.float32 and bool(((got.double() - y).abs() <= err + 1e-6).all())
    for bias in (None, b):
        want = y if bias is None else y + b.double()
        got = ops.product_tiles(x, t, bias)
        assert got.dtype == torch.bfloat16 and bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + err + 1e-6).all())


@pytest.mark.parametrize("kind", ["alone", "gated", "some gated"])
@pytest.mark.parametrize("tile,left", tile_cases.places())
def test_each_tile_by_itself(tile, left, kind):
    """Each tile of the list with each kind of end, so many chunks of K left behind two rounds of its walk or more: the size is looked up, so the tile runs whatever the costs it is picked by."""
    M, N, K, _ = tile_cases.size_for(tile, left)
    if kind == "alone":
        test_products_of_many_rows_alone(M, N, K)
    else:
        test_many_rows_in_tiles_with_the_gated_unit_behind(M, N, K, 0 if kind == "gated" else N // 32 * 16)


@pytest.mark.parametrize("tile", range(len(tile_cases.tiles())))
def test_each_tile_by_itself_over_a_group(tile):
    """The same of group_tiles_kernel."""
    M, N, K, groups = tile_cases.size_for(tile, tile_cases.tiles()[tile][2], (2, 3, 8, 16, 32))
    test_groups_of_many_rows(groups, K, N, 8, M)


@pytest.mark.parametrize("M,N,K,split", [(66, 96, 192, 0), (300, 3104, 320, 1552), (770, 5408, 128, 0), (1063, 2080, 576, 64), (2100, 1568, 1024, 1024)])
def test_results_of_tiles_in_rows_that_are_not_whole_pieces(M, N, K, split):
    """lines_out: rows of outputs that begin anywhere and are no multiple of sixteen bytes long hold, bit for bit, what aligned ones do, and nothing beside them is written."""
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev())      # noqa: E731
    t, x = ops.MatrixTiles(rnd(N, K) / K ** 0.5, torch.bfloat16), rnd(M, K).to(torch.bfloat16)
    n = (N - split) // 2
    whole, wide = torch.empty((M, n), dtype=torch.bfloat16, device=dev()), torch.full((M, n + 10), 7.0, dtype=torch.bfloat16, device=dev())
    a, b = ops.linear_tiles(x, t, ops.SILU_UNIT, split, whole), ops.linear_tiles(x, t, ops.SILU_UNIT, split, wide[:, 2:-8])
    assert torch.equal(wide[:, 2:-8], whole) and bool((wide[:, :2] == 7).all()) and bool((wide[:, -8:] == 7).all())
    assert not split or torch.equal(a, b)
    groups = ops.MatrixTiles(rnd(3, N, K) / K ** 0.5, torch.bfloat16)
    for gate in (None, rnd(M, 3).to(torch.bfloat16)):
        whole, wide = torch.empty((M, 3 * N), dtype=torch.bfloat16, device=dev()), torch.full((M, 3 * (N + 4)), 7.0, dtype=torch.bfloat16, device=dev())
        ops.linear(x, groups, x_gstride=0, y_gstride=N, out=whole, gate=gate)
        ops.linear(x, groups, x_gstride=0, y_gstride=N + 4, out=wide, gate=gate)
        y = wide.view(M, 3, N + 4)
        assert torch.equal(y[..., :N].reshape(M, 3 * N), whole) and bool((y[..., N:] == 7).all())


def test_products_of_many_rows_alone_refuse_what_is_not_built():
    from vllmini_amd import hybrid_ops as ops

    x, t = torch.zeros((64, 128), dtype=torch.bfloat16, device=dev()), ops.MatrixTiles(torch.zeros((64, 128), device=dev()), torch.bfloat16)
    odd = ops.MatrixTiles(torch.zeros((64, 96), device=dev()), torch.bfloat16)
    wide = torch.zeros((64, 136), dtype=torch.bfloat16, device=dev())
    for bad in (lambda: ops.product_tiles(x.float(), t), lambda: ops.product_tiles(x[:, :96], t), lambda: ops.product_tiles(x[:, :96], odd), lambda: ops.product_tiles(wide[:, 4:132], t),
                lambda: ops.product_tiles(x, t, torch.zeros(64, dtype=torch.bfloat16, device=dev())), lambda: ops.product_tiles(x, t, torch.zeros(64, device=dev()), True),
                lambda: ops.product_tiles(torch.zeros((64, 132), dtype=torch.bfloat16, device=dev())[:, :128], t), lambda: ops.product_tiles(x, t, torch.zeros(32, device=dev()))):
        with pytest.raises(RuntimeError):
            bad()
    assert ops.product_tiles_pay(x, t) and not ops.product_tiles_pay(x[:, :96], odd) and not ops.product_tiles_pay(wide[:, 4:132], t) and not ops.product_tiles_pay(x.float(), t)


@pytest.mark.parametrize("split", [0, 64])
def test_gated_rows_past_what_one_launch_takes_go_in_parts(split, monkeypatch):
    """Without the vendor's layout rows of 4 GiB and more are cut in two until a launch takes them: the same bits."""
    from vllmini_amd import hybrid_layers as hl, hybrid_ops as ops

    g = torch.Generator(device=dev()).manual_seed(split)
    w, x = hl.gated_matrix(torch.randn((192, 128), generator=g, device=dev()) / 11, torch.bfloat16, split), torch.randn((333, 128), generator=g, device=dev()).to(torch.bfloat16)
    runs, pay = [], ops.linear_tiles_pay
    assert w.dense is None
    for most in (10 ** 9, 50):
        monkeypatch.setattr(ops, "linear_tiles_pay", lambda M, w, split=0: M <= most and pay(M, w, split))
        out = torch.zeros((333, 200), dtype=torch.bfloat16, device=dev())[:, 8:8 + (192 - split) // 2]
        runs.append((hl.gated_product(x, w, ops.SILU_UNIT, split, out), hl.gated_product(x, w, ops.SILU_UNIT, split), out))
    assert all(torch.equal(a, b) for a, b in zip(*runs)) and bool(runs[0][2].any())
    assert hl.gated_product(x[:0], w, ops.SILU_UNIT, split).shape == (0, split or 96)


def test_many_rows_in_tiles_refuse_what_is_not_built():
    from vllmini_amd import hybrid_ops as ops

    x, t = torch.zeros((64, 128), dtype=torch.bfloat16, device=dev()), ops.MatrixTiles(torch.zeros((64, 128), device=dev()), torch.bfloat16)
    for bad in (lambda: ops.linear_tiles(x.float(), t, ops.SILU_UNIT), lambda: ops.linear_tiles(x[:, :96], t, ops.SILU_UNIT), lambda: ops.linear_tiles(x, t, ops.SILU_UNIT, 8),
                lambda: ops.linear_tiles(x[:, :96], ops.MatrixTiles(torch.zeros((64, 96), device=dev()), torch.bfloat16), ops.SILU_UNIT),
                lambda: ops.linear_tiles(x, t, ops.SILU_UNIT, 32, x[:, :32]), lambda: ops.linear_tiles(x, ops.MatrixTiles(torch.zeros((64, 128), device=dev()), torch.float32), ops.SILU_UNIT)):
        with pytest.raises(RuntimeError):
            bad()
    assert not ops.linear_tiles_pay(300, ops.MatrixTiles(torch.zeros((64, 96)), torch.bfloat16)) and not ops.linear_tiles_pay(300, ops.MatrixTiles(torch.zeros((64, 128)), torch.float32))


@pytest.mark.parametrize("dtype", BOTH)
def test_products_that_are_not_built_are_refused(dtype):
    """Inputs and epilogues that vmi_hy_linear has no kernel for: an error and nothing written, whether or not there is room for normed rows."""
    import ctypes

    from vllmini_amd import hybrid_ops as ops

    M, N, K = 12, 64, 4096
    lib, t = ops.load(), ops.MatrixTiles(torch.ones(N, K, dtype=dtype, device=dev()), dtype)
    x, xt = torch.ones(M, K, device=dev()), torch.ones(M, K, dtype=dtype, device=dev())
    nw, y, y2, normed = torch.ones(K, device=dev()), torch.full((M, N), 7.0, device=dev()), torch.full((M, N), 7.0, device=dev()), torch.full_like(xt, 7.0)
    assert all(b.is_cuda for b in (t.tiles, x, xt, nw, y, y2, normed))
    built = {0: {0, 1, 4}, 1: {0, 2, 3, 5}, 2: {2}}      # x_kind: epilogues
    for kind, epi in ((a, b) for a in range(3) for b in range(6) if b not in built[a]):
        for room in (None, normed):
            a = ops.LinearArgs(x=(xt if kind == 0 else x).data_ptr(), x2=x.data_ptr(), norm_w=nw.data_ptr(), w=t.tiles.data_ptr(), gate=xt.data_ptr(), y=y.data_ptr(),
                               y2=y2.data_ptr(), normed=None if room is None else room.data_ptr(), ldx=K, ldy=N, ldg=K, ldy2=N, M=M, N=N, K=K, groups=1, norm_n=K,
                               n_out=N, n_split=32, eps=1e-5, scale=1.0, x_kind=kind, epilogue=epi, dtype=ops.DTYPES[dtype])
            assert lib.vmi_hy_linear(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 1, (kind, epi)
            assert b"not built" in lib.vmi_hybrid_last_error()
    assert all(bool((b == 7.0).all()) for b in (y, y2, normed))


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("M", [3, 70])
def test_linear_groups_and_head_gate(dtype, M):
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator().manual_seed(M)
    G, N, K, gap = 5, 64, 96, 160
    x = torch.randn(M, G * gap, generator=g).to(dtype).to(dev())
    w = (torch.randn(G, N, K, generator=g) / 10).to(torch.bfloat16).to(dev())
    gate = torch.randn(M, 32, generator=g).to(dtype).to(dev())
    out = torch.zeros(M, G * 80, dtype=dtype, device=dev())
    ops.linear(x, ops.MatrixTiles(w, dtype), x_gstride=gap, y_gstride=80, gate=gate[:, 3:], out=out)
    for i in range(G):
        want = x[:, i * gap:i * gap + K].double() @ w[i].double().T * torch.sigmoid(gate[:, 3 + i].double())[:, None]
        close(out[:, i * 80:i * 80 + N], want, dtype)
        assert not out[:, i * 80 + N:(i + 1) * 80].any()


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("n", [50, 96, 1500, 9001])
def test_elementwise_ends(dtype, n):
    from vllmini_amd import hybrid_ops as ops

    g = torch.Generator().manual_seed(n)
    ld = ops.pad32(n)
    x = torch.zeros(7, ld, device=dev())
    x[:, :n] = (torch.randn(7, n, generator=g) * 2 - 30).to(dev())
    add, w = torch.zeros(7, ld, dtype=dtype, device=dev()), torch.zeros(ld, device=dev())
    add[:, :n] = torch.randn(7, n, generator=g).to(dtype).to(dev())
    w[:n] = torch.randn(n, generator=g).to(dev())
    want = x.double() + add.double()
    h = ops.add_norm(x, add, (w, n, 1e-6), dtype)
    close(x, want, torch.float32)
    close(h[:, :n], plain.layer_norm(want[:, :n], w[:n].double(), 1e-6), dtype, tol32=1e-4)
    assert not h[:, n:].any()
    v = (torch.randn(7, 2 * ld, generator=g) * 2).to(dtype).to(dev())
    gate, up = v[:, 0::2].double().clamp(max=1.25), v[:, 1::2].double().clamp(-1.25, 1.25)
    close(ops.glu(v, ops.GatedUnit.clamped(1.25)), gate * torch.sigmoid(1.702 * gate) * (up + 1), dtype)
    table = torch.zeros(40, ld, dtype=torch.bfloat16, device=dev())
    table[:, :n] = torch.randn(40, n, generator=g).to(dev())
    ids = torch.tensor([0, 39, 7], device=dev())
    assert torch.equal(ops.embed(ids, table, n, 2.5), table[ids].float() * 2.5)
    lg = torch.randn(6, n, generator=g).to(dev())
    lg[2, 5] = lg[2, 31] = 9.0
    assert ops.argmax(lg).tolist() == lg.argmax(-1).tolist() and ops.argmax(lg)[2] == 5


# ---- the recurrent block ---------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("ld", [32, 1024, 1056, 2080, 4096, 4128, 8192, 8224])
def test_rows_of_every_width_added_normed_and_merged(dtype, ld):
    """What a workgroup keeps of a row by its length, and what is read again behind it; columns that are not normed hold numbers for the sum alone."""
    from vllmini_amd import hybrid_ops as ops

    n, T = ld - 8, 3
    g = torch.Generator().manual_seed(ld)
    x, a, b, c = (torch.randn(T, ld, generator=g).to(dev()) for _ in range(4))
    a, b, c = (t.to(dtype) for t in (a, b, c))
    w, u = ((1 + 0.3 * torch.randn(ld, generator=g)).to(dev()) for _ in range(2))
    w[n:] = u[n:] = 0
    for rms in (False, True):
        y = x.clone()
        h = ops.add_norm(y, a, (w, n, 1e-5, rms), dtype)
        want = x.double() + a.double()
        close(y, want, torch.float32, tol32=1e-6)
        d = want[:, :n] - (0 if rms else want[:, :n].mean(-1, keepdim=True))
        close(h[:, :n], d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * w[:n].double(), dtype, tol16=6e-3)
        assert not h[:, n:].any()
    a[:, n:] = b[:, n:] = 0
    for add in (None, c):
        y = x.clone()
        ops.merge(y, a, w, b, u, add, n=n, eps=1e-5, scale=0.5)
        unit = [t.double() / torch.sqrt((t.double() ** 2).sum(-1, keepdim=True) / n + 1e-5) * v.double() for t, v in ((a, w), (b, u))]
        close(y, x.double() + 0.5 * (unit[0] + unit[1]) + (0 if add is None else c.double()), torch.float32, tol32=2e-6)


def _rglru_weights(width, blocks, taps, seed):
    c = cases.config([cases.rglru(width, blocks, taps)], width=width)
    return cases.tensors(c, seed)


class _Rglru:
    """The kernel's operands for a width / block count, and the plain result for a whole sequence."""

    def __init__(self, width, blocks, taps, dtype, slots, seed=0):
        from vllmini_amd.hybrid_layers import Norm, RGLRU

        w = {k: v.to(dev()) for k, v in _rglru_weights(width, blocks, taps, seed).items()}
        self.w = {k[len("l0.mix."):]: v for k, v in w.items() if k.startswith("l0.mix.")}
        n = self.w
        self.layer = RGLRU(width=width, size=width, blocks=blocks, taps=taps, norm=Norm(w["l0.norm1"], (width + 31) // 32 * 32, 1e-5),
                           y=n["y"], y_b=n["y.b"], x=n["x"], x_b=n["x.b"], conv=n["conv"], conv_b=n["conv.b"], ra=n["ra"],
                           ra_b=n["ra.b"], ri=n["ri"], ri_b=n["ri.b"], lam=n["lam"], o=n["o"], dtype=dtype)
        self.width, self.blocks, self.dtype = width, blocks, dtype
        bw, bp = width // blocks, self.layer.width // blocks
        self.idx = (torch.arange(blocks)[:, None] * bp + torch.arange(bw)[None]).reshape(-1).to(dev())
        (s, _), (t, _) = self.layer.state_shapes()
        self.state = torch.full((slots, *s), 7.0, device=dev())              # what former owners left must not matter
        self.tail = torch.full((slots, *t), 5.0, dtype=dtype, device=dev())

    def inputs(self, T, seed):
        g = torch.Generator().manual_seed(seed)
        y, x = (torch.randn(T, self.width, generator=g).to(self.dtype).to(dev()) for _ in range(2))
        yx = torch.zeros(T, 2 * self.layer.width, dtype=self.dtype, device=dev())
        yx[:, self.idx], yx[:, self.layer.width + self.idx] = y, x
        return y, x, yx

    def plain(self, y, x):
        n = {k: v.double() for k, v in self.w.items()}
        u = plain.causal_conv(x.double(), n["conv"], n["conv.b"])
        if self.dtype == torch.bfloat16:
            u = u.to(torch.bfloat16).double()
        S, _ = plain.rglru_scan(u, plain.rglru_gate(u, n["ra"], n["ra.b"]), plain.rglru_gate(u, n["ri"], n["ri.b"]), n["lam"])
        return S * plain.gelu_tanh(y.double())

    def run(self, yx, step):
        from vllmini_amd import hybrid_ops as ops

        L = self.layer
        return ops.rglru(yx, step, conv_w=L.conv_w, conv_b=L.conv_b, gates=L.gates, gate_b=L.gate_b, decay=L.decay, blocks=L.blocks,
                         state=self.state, tail=self.tail)[:, self.idx]


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,blocks,taps", [(96, 3, 4), (40, 2, 1), (150, 1, 2), (600, 2, 7), (66, 11, 3)])
def test_recurrence_over_portions_of_every_size(dtype, width, blocks, taps):
    """Three sequences cut differently — whole, portions around the 64-row tile, two and three tokens, single tokens — in shared
    steps, the state in slots whose former contents are garbage."""
    T = 210
    k = _Rglru(width, blocks, taps, dtype, slots=5)
    seqs = [k.inputs(T, 10 + i) for i in range(3)]
    cuts = [[210], [63, 2, 64, 3, 1, 1, 65, 2, 9], [1] * 9 + [2, 3, 70, 1, 2, 123]]
    slots, at, flips = [4, 0, 2], [0] * 3, [0] * 3
    out = [[] for _ in range(3)]
    while any(at[i] < T for i in range(3)):
        live = [i for i in range(3) if at[i] < T]
        n = [cuts[i].pop(0) for i in live]
        yx = torch.cat([seqs[i][2][at[i]:at[i] + c] for i, c in zip(live, n)])
        step = layout(n, [at[i] for i in live], [[0]] * len(live), 64, [slots[i] for i in live], [flips[i] for i in live], pos_slots=False)
        got = k.run(yx, step)
        for i, c, g in zip(live, n, got.split(n)):
            out[i].append(g)
            at[i] += c
            flips[i] ^= 1
    for i in range(3):
        close(torch.cat(out[i]), k.plain(*seqs[i][:2]), dtype, tol32=3e-5, tol16=1.5e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,blocks", [(512, 2), (320, 2), (192, 3), (600, 1)])
def test_recurrence_over_portions_in_wide_blocks(dtype, width, blocks):
    """Four taps, rows taken together: blocks of one and two shares of a workgroup's channels (the second not all there), and of several chunks."""
    test_recurrence_over_portions_of_every_size(dtype, width, blocks, 4)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("lens", [[64 * 9 + 1], [30, 64 * 63 + 34], [30, 64 * 63 + 35]])
def test_recurrence_over_long_portions(dtype, lens):
    """Carries over more tiles than a request holds, one that ends with its tile, and one tile more than run in one launch; a second portion takes the state up."""
    k = _Rglru(64, 2, 4, dtype, slots=2)
    seqs = [k.inputs(n + 3, 40 + i) for i, n in enumerate(lens)]
    got = []
    for at, counts in ((0, lens), (1, [3] * len(lens))):
        step = layout(counts, [0] * len(lens) if at == 0 else lens, [[0]] * len(lens), 64, flips=[at] * len(lens), pos_slots=False)
        got.append(k.run(torch.cat([s[2][:n] if at == 0 else s[2][n:] for s, n in zip(seqs, lens)]), step).split(counts))
    for i, s in enumerate(seqs):
        close(torch.cat([got[0][i], got[1][i]]), k.plain(*s[:2]), dtype, tol32=3e-5, tol16=1.5e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,blocks", [(512, 2), (96, 3)])
def test_portions_that_share_rows_taken_together_with_padding(dtype, width, blocks):
    """Portions of one to nine tokens, so that the eight (four) rows of a thread hold several starts, and rows behind them that are no token's and hold NaN."""
    from vllmini_amd import hybrid_ops as ops

    counts = [1, 2, 3, 9, 5, 1, 7, 64, 4, 2]
    k, T, pad = _Rglru(width, blocks, 4, dtype, slots=len(counts)), sum(counts), 5
    seqs = [k.inputs(n, 90 + i) for i, n in enumerate(counts)]
    step = layout(counts, [0] * len(counts), [[0]] * len(counts), 64, pos_slots=False)
    f = dict(step.fields)
    f["tok_seq"], f["tok_pos"], f["tok_slot"] = (torch.cat([f[n], i32([v] * pad)]) for n, v in (("tok_seq", -1), ("tok_pos", 0), ("tok_slot", -1)))
    yx = torch.cat([s[2] for s in seqs] + [torch.full((pad, 2 * k.layer.width), float("nan"), dtype=dtype, device=dev())])
    got = k.run(yx, ops.StepLayout(f, T + pad, len(counts), 64, False, True, max(counts), max(counts)))
    assert not got[T:].any()
    for s, g in zip(seqs, got[:T].split(counts)):
        close(g, k.plain(*s[:2]), dtype, tol32=3e-5, tol16=1.5e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,blocks,taps", [(512, 2, 4), (96, 3, 4), (66, 11, 3)])
@pytest.mark.parametrize("bad,value", [(0, float("nan")), (1, float("inf")), (3, float("nan")), (3, float("-inf")), (4, None)])
def test_portions_that_are_no_numbers_leave_the_others_alone(dtype, width, blocks, taps, bad, value):
    """A NaN or an infinity in one portion's inputs, or (None) in the state it takes up, in front of others in its row tile and across the tile's end: every bit of the others' results, states
    and tails is as it is without."""
    counts, ctx = [5, 40, 3, 100, 9, 20], [0, 7, 0, 0, 7, 0]
    k = _Rglru(width, blocks, taps, dtype, slots=len(counts))
    g = torch.Generator().manual_seed(width)
    state, tail = (torch.randn(t.shape, generator=g).to(t.dtype).to(dev()) for t in (k.state, k.tail))
    yx, at = torch.cat([k.inputs(n, 60 + i)[2] for i, n in enumerate(counts)]), sum(counts[:bad])
    rest = torch.tensor([i for i in range(len(counts)) if i != bad], device=dev())
    got = []
    for poison in (False, True):
        k.state.copy_(state), k.tail.copy_(tail)
        rows = yx.clone()
        if poison and value is None:
            k.state[bad] = float("nan")
        elif poison:
            rows[at + counts[bad] // 3, k.layer.width:] = value
        out = k.run(rows, layout(counts, ctx, [[0]] * len(counts), 64, pos_slots=False))
        got.append((torch.cat([o for i, o in enumerate(out.split(counts)) if i != bad]), k.state[rest].clone(), k.tail[rest].clone()))
        assert poison == (not bool(torch.isfinite(out[at: at + counts[bad]].float()).all()))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(torch.isfinite(got[1][0].float()).all())


@pytest.mark.parametrize("dtype", BOTH)
def test_recurrence_decodes_like_it_prefills_and_skips_padding_rows(dtype):
    from vllmini_amd import hybrid_ops as ops

    k = _Rglru(96, 2, 4, dtype, slots=20)
    T, B = 20, 19
    seqs = [k.inputs(T, 50 + i) for i in range(B)]
    want = [k.plain(*s[:2]) for s in seqs]
    untouched = k.state[B].clone()
    for t in range(T):
        step = layout([1] * B, [t] * B, [[0]] * B, 64, flips=[t & 1] * B, pos_slots=False)
        f = dict(step.fields)
        f["tok_seq"] = torch.cat([f["tok_seq"], i32([-1, -1])])      # two padding rows, as a padded decode batch has
        f["tok_pos"], f["tok_slot"] = torch.cat([f["tok_pos"], i32([0, 0])]), torch.cat([f["tok_slot"], i32([-1, -1])])
        pad = ops.StepLayout(f, B + 2, B, 64, True, False, 1, t + 1)
        yx = torch.cat([s[2][t:t + 1] for s in seqs] + [torch.full((2, 2 * k.layer.width), float("nan"), dtype=dtype, device=dev())])
        got = k.run(yx, pad)
        assert not got[B:].any()
        for i in range(B):
            close(got[i], want[i][t], dtype, tol32=1e-4, tol16=3e-2)
    assert torch.equal(k.state[B], untouched)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("width,blocks,taps", [(96, 3, 4), (1536, 2, 4), (288, 9, 6)])
def test_entries_of_padding_rows_name_no_state(dtype, width, blocks, taps):
    """Single tokens among padding rows whose entries hold a slot, a context and a flip that are none: zeros come out, and no state and no tail is read or written for them."""
    k = _Rglru(width, blocks, taps, dtype, slots=4)
    from vllmini_amd import hybrid_ops as ops

    at = [1, 4, 18]      # rows of the three sequences, of twenty
    seqs = [k.inputs(2, 70 + i) for i in range(3)]
    for t in range(2):
        step = layout([1] * 20, [-1] * 20, [[0]] * 20, 64, slots=[-1 - 1000 * i for i in range(20)], flips=[-5] * 20, pos_slots=False)
        f = dict(step.fields)
        f["tok_seq"] = torch.full_like(f["tok_seq"], -1)
        for i, row in enumerate(at):
            f["tok_seq"][row], f["ctx"][row], f["state_slot"][row], f["flip"][row] = row, t, i, t & 1
        yx = torch.full((20, 2 * k.layer.width), float("nan"), dtype=dtype, device=dev())
        for i, row in enumerate(at):
            yx[row] = seqs[i][2][t]
        tail = k.tail[3].clone()
        got = k.run(yx, ops.StepLayout(f, 20, 20, 64, True, False, 1, t + 1))
        for i, row in enumerate(at):
            close(got[row], k.plain(*seqs[i][:2])[t], dtype, tol32=1e-4, tol16=3e-2)
        assert not got[[r for r in range(20) if r not in at]].any()
        assert bool((k.state[3] == 7).all()) and torch.equal(k.tail[3], tail)


@pytest.mark.parametrize("width,blocks,taps,B", [(96, 1, 4, 1), (2560, 10, 4, 16), (2112, 3, 4, 70), (1536, 2, 4, 33), (288, 9, 6, 40), (4096, 16, 4, 70)])
def test_single_tokens_share_a_gate_block_over_waves_and_workgroups(width, blocks, taps, B):
    """rglru_step_kernel with one, two and four tiles of channels a workgroup (the last one's not all there), blocks of fewer and more channels than its waves take at
    a time, beside rglru_tile_kernel where there are more tiles: two steps, whose tokens come in another order than their entries in the second."""
    k = _Rglru(width, blocks, taps, torch.bfloat16, slots=B)
    seqs = [k.inputs(2, 90 + i) for i in range(B)]
    for t in range(2):
        order = list(range(B)) if t == 0 else list(range(B))[::-1]
        step = layout([1] * B, [t] * B, [[0]] * B, 64, flips=[t & 1] * B, pos_slots=False)
        step.fields["tok_seq"].copy_(i32(order))
        step.fields["q_start"].copy_(i32(order))
        got = k.run(torch.cat([seqs[i][2][t:t + 1] for i in order]), step)
        for at, i in enumerate(order):
            close(got[at], k.plain(*seqs[i][:2])[t], torch.bfloat16, tol32=1e-4, tol16=3e-2)


def test_recurrence_keeps_a_long_memory_in_fp32():
    """Decays near one: after a thousand tokens without input the first token's trace is still there, to fp32 accuracy."""
    k = _Rglru(64, 2, 1, torch.bfloat16, slots=1)
    k.layer.decay.fill_(-1e-4)
    T = 1000
    yx = torch.zeros(T, 2 * k.layer.width, dtype=torch.bfloat16, device=dev())
    yx[:, k.idx] = 1.0
    yx[0, k.layer.width + k.idx] = 4.0
    k.layer.conv_b.zero_()
    k.layer.conv_w.fill_(1.0)
    k.layer.gate_b.zero_()
    k.layer.gates.zero_()
    got = k.run(yx, layout([T], [0], [[0]], 64, pos_slots=False)).double().cpu()
    a = np.exp(-1e-4 * 0.5)
    want = 4.0 * 0.5 * np.sqrt(1 - a * a) * a ** np.arange(T) * float(plain.gelu_tanh(torch.tensor(1.0, dtype=torch.float64)))
    assert np.abs(got.numpy() / want[:, None] - 1).max() < 5e-3          # (one bfloat16 rounding of the output)
    S = float(k.state[0, 0])
    assert S == pytest.approx(2.0 * np.sqrt(1 - a * a) * a ** (T - 1), rel=2e-5)


# ---- latent attention --------------------------------------------------------------------------------------------------------------
def _attend(dtype, H, rank, rot, counts, ctx, page, row_tiles=None, splits=1, spike=None, seed=0):
    from vllmini_amd import hybrid_ops as ops

    D, B = rank + rot, len(counts)
    g = torch.Generator().manual_seed(seed)
    total = [c + n for c, n in zip(ctx, counts)]
    per = [-(-t // page) for t in total]
    pages = torch.randperm(sum(per) + 3, generator=g).numpy()
    cache = torch.randn(len(pages), page, D, generator=g).to(dtype).to(dev())
    tables = np.zeros((B, max(per)), dtype=np.int64)
    at = 0
    for b in range(B):
        tables[b, :per[b]] = pages[at:at + per[b]]
        at += per[b]
    q = torch.randn(sum(counts), H, D, generator=g).to(dtype).to(dev())
    scale = 1.7 * D ** -0.5
    flat = cache.view(-1, D)
    row = lambda b, p: int(tables[b, p // page]) * page + p % page      # noqa: E731
    if spike is not None:      # query `t` of entry b meets a key of its own direction at position p: that score stands far out
        for b, t, p in spike:
            u = torch.randn(D, generator=g)
            u = u / u.norm()
            q[sum(counts[:b]) + t] = (u * (14 / scale) ** 0.5).to(dtype).to(dev())
            flat[row(b, p)] = (u * (14 / scale) ** 0.5).to(dtype).to(dev())
    step = layout(counts, ctx, tables, page)
    rt = ops.latent_row_tiles(D, row_tiles or 4, dtype)
    tiles = [(b, r) for b in range(B) for r in range(0, counts[b] * H, 16 * rt)]
    tiles.insert(1, (-1, -1))
    out = ops.latent_attention(q.view(-1, H * D), cache, step, i32(tiles), heads=H, rank=rank, rot=rot, scale=scale, row_tiles=rt,
                               splits=splits).view(-1, H, rank)
    want, at = [], 0
    for b in range(B):
        keys = flat[[row(b, p) for p in range(total[b])]].double()
        for t in range(counts[b]):
            s = q[at].double() @ keys[: ctx[b] + t + 1].T * scale
            want.append(torch.softmax(s, -1) @ keys[: ctx[b] + t + 1, :rank])
            at += 1
    return out, torch.stack(want)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("H,rank,rot,page", [(1, 32, 32, 16), (3, 64, 32, 64), (7, 128, 32, 64), (20, 256, 64, 32), (16, 512, 64, 64),
                                             (5, 608, 32, 64), (40, 160, 96, 8)])
def test_latent_attention_over_pages(dtype, H, rank, rot, page):
    for counts, ctx in (([1], [0]), ([1, 1, 1], [63, 64, 200]), ([70, 1, 2], [0, 130, 62]), ([33], [95])):
        for rt in (1, 2, 4) if dtype == torch.bfloat16 else (1,):
            for sp in (1, 2, 5):
                got, want = _attend(dtype, H, rank, rot, counts, ctx, page, rt, sp)
                close(got, want, dtype, tol32=2e-5, tol16=1.5e-2)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("H,rank,rot", [(3, 32, 32), (2, 160, 32), (1, 512, 64), (2, 608, 32)])
def test_parts_of_any_number_add_up(dtype, H, rank, rot):
    """combine_kernel: groups of 4, 8 and 16 parts, whole and not, up to all 128; parts without keys (of the short contexts most); one wave of columns and several."""
    for sp in (2, 4, 5, 8, 9, 16, 17, 64, 65, 128):
        got, want = _attend(dtype, H, rank, rot, [1, 1, 2], [40, 700, 8300], 64, 1, sp, seed=sp)
        close(got, want, dtype, tol32=2e-5, tol16=1.5e-2)


@pytest.mark.parametrize("dtype", BOTH)
def test_latent_attention_sees_the_far_key_and_never_the_next_one(dtype):
    """One score stands out: at the very first token, at page borders, at the query's own position — and one past it, where it must
    not be seen."""
    n, ctx = 5, 700
    for p in (0, 1, 63, 64, 65, 127, 128, 447, 639, 640, ctx + 1, ctx + 2):
        got, want = _attend(dtype, 4, 64, 32, [n], [ctx], 64, splits=4, spike=[(0, 2, p)], seed=p)
        close(got, want, dtype)
        assert float(want[2].abs().max()) > 0.5
    got, want = _attend(dtype, 4, 64, 32, [n], [ctx], 64, splits=4, spike=[(0, 2, ctx + 3)], seed=1)      # the next token's key
    close(got, want, dtype)


@pytest.mark.parametrize("dtype", BOTH)
def test_latent_prep_normalises_rotates_and_writes_the_cache(dtype):
    from vllmini_amd import hybrid_ops as ops

    heads, dim, rot, rank, rot_n, rank_n, rot_true = 3, 32, 32, 64, 10, 50, 20
    g = torch.Generator().manual_seed(4)
    counts, ctx, page = [3, 1], [4000, 77], 16
    T = sum(counts)
    tables = np.arange(2 * 251).reshape(2, 251)[:, ::-1].copy()
    step = layout(counts, ctx, tables, page)
    ldp = heads * (dim + rot) + rank + rot + 32
    proj = torch.zeros(T, ldp)
    for h in range(heads + 1):
        at = h * (dim + rot) + dim if h < heads else heads * (dim + rot) + rank
        proj[:, at:at + rot_true] = torch.randn(T, rot_true, generator=g)
    proj[:, heads * (dim + rot):heads * (dim + rot) + rank_n] = 5 * torch.randn(T, rank_n, generator=g)
    proj = proj.to(dtype).to(dev())
    q = torch.full((T, heads * (rank + rot)), 3.0, dtype=dtype, device=dev())
    cache = torch.full((502, page, rank + rot), 9.0, dtype=dtype, device=dev())
    w = torch.zeros(rank, device=dev())
    w[:rank_n] = 1 + 0.3 * torch.randn(rank_n, generator=g).to(dev())
    freq = (500.0 ** (-2.0 * torch.arange(rot_n // 2, dtype=torch.float64) / rot_n)).to(dev())
    ops.latent_prep(proj, q, cache, step, norm_w=w, freq=freq, heads=heads, dim=dim, rot=rot, rank=rank, rot_n=rot_n, rank_n=rank_n, eps=1e-5)
    flat, P = cache.view(-1, rank + rot), proj.double().cpu()
    used = []
    for t in range(T):
        b, pos = (0, 4000 + t) if t < 3 else (1, 77)
        r = int(tables[b, pos // page]) * page + pos % page
        used.append(r)
        lat = heads * (dim + rot)
        close(flat[r, :rank_n], plain.rms_norm(P[t, lat:lat + rank_n], w[:rank_n].double().cpu(), 1e-5), dtype, tol16=6e-3)
        assert not flat[r, rank_n:rank].any()
        close(flat[r, rank:], plain.rotate(P[t, lat + rank:lat + rank + rot], pos, 500.0, rot_n), dtype, tol16=6e-3)
        for h in range(heads):
            s = h * (dim + rot) + dim
            close(q[t, h * (rank + rot) + rank:(h + 1) * (rank + rot)], plain.rotate(P[t, s:s + rot], pos, 500.0, rot_n), dtype, tol16=6e-3)
            assert (q[t, h * (rank + rot):h * (rank + rot) + rank] == 3).all()
    rest = torch.ones(flat.shape[0], dtype=torch.bool, device=dev())
    rest[used] = False
    assert (flat[rest] == 9).all()


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("T", [1, 16, 17, 50, 64, 65])
@pytest.mark.parametrize("heads,dim,rank", [(3, 32, 64), (16, 128, 512), (2, 160, 96), (1, 512, 32), (2, 544, 32)])
def test_latent_in_is_the_product_and_the_preparation(dtype, T, heads, dim, rank):
    """Every bit of the two launches it stands for, a padding row and rows past the last one left alone; sizes on both sides of what goes into one launch."""
    from vllmini_amd import hybrid_ops as ops

    rot, rot_n, page = 32, 20, 16
    g = torch.Generator().manual_seed(T + dim)
    step = layout([1] * T, list(range(5, 5 + T)), np.arange(T * 6).reshape(T, 6), page)
    f = dict(step.fields)
    f["tok_seq"] = torch.cat([f["tok_seq"][: T - 1], i32([-1])]) if T > 1 else f["tok_seq"]
    step = ops.StepLayout(f, T, T, page, True, False, 1, T + 5)
    proj = torch.randn(T, heads * (dim + rot) + rank + rot + 32, generator=g).to(dtype).to(dev())
    w = ops.MatrixTiles((torch.randn(heads, rank, dim, generator=g) * dim ** -0.5).to(dev()), dtype)
    names = dict(norm_w=torch.rand(rank, generator=g).to(dev()), freq=(500.0 ** (-2.0 * torch.arange(rot_n // 2, dtype=torch.float64) / rot_n)).to(dev()), heads=heads, dim=dim, rot=rot,
                 rank=rank, rot_n=rot_n, rank_n=rank, eps=1e-5)
    qs = [torch.full((T + 2, heads * (rank + rot)), 3.0, dtype=dtype, device=dev()) for _ in range(2)]
    caches = [torch.full((T * 6, page, rank + rot), 9.0, dtype=dtype, device=dev()) for _ in range(2)]
    ops.linear(proj, w, x_gstride=dim + rot, y_gstride=rank + rot, out=qs[0][:T])
    ops.latent_prep(proj, qs[0][:T], caches[0], step, **names)
    ops.latent_in(proj, w, qs[1][:T], caches[1], step, **names)
    assert torch.equal(*qs) and torch.equal(*caches)


@pytest.mark.parametrize("dim,rot,rank,rot_n,lens", [(128, 64, 512, 64, [64, 1, 65, 16]), (128, 32, 64, 16, [130, 63]), (64, 64, 128, 32, [15, 200, 17]), (64, 32, 192, 32, [321])])
def test_latent_prompt_matches_plain_attention_and_leaves_the_caches_rows(dim, rot, rank, rot_n, lens):
    """A step whose entries have no past: the cache rows, bytes, that latent_prep writes, and plain attention over them in float64.  Rounded to bfloat16 (2^-8 of it at most) are a
    key, a value, a probability and the result; the scores of keys off by 2^-9 in the mean, of |score| up to about 4, move a probability by 1 per cent."""
    from vllmini_amd import hybrid_ops as ops

    H, page, T, D, bf = 3, 32, sum(lens), rank + rot, torch.bfloat16
    g = torch.Generator().manual_seed(T + dim)
    hd, scale = dim + rot, (dim + rot) ** -0.5
    proj = torch.randn(T, H * hd + D + 32, generator=g).to(bf).to(dev())
    up = (torch.randn(H, 2 * dim, rank, generator=g) * rank ** -0.5).to(bf).to(dev())
    w = (1 + 0.3 * torch.randn(rank, generator=g)).to(dev())
    freq = (500.0 ** (-2.0 * torch.arange(rot_n // 2, dtype=torch.float64) / rot_n)).to(dev())
    per = [-(-n // page) for n in lens]
    tables = np.zeros((len(lens), max(per)), dtype=np.int64)
    for i, n in enumerate(per):
        tables[i, :n] = sum(per) - sum(per[:i]) - np.arange(n)
    step = layout(lens, [0] * len(lens), tables, page)
    step.fresh = True
    caches = [torch.full((sum(per) + 1, page, D), 9.0, dtype=bf, device=dev()) for _ in range(2)]
    q = torch.zeros((T, H * D), dtype=bf, device=dev())
    names = dict(norm_w=w, freq=freq, heads=H, dim=dim, rot=rot, rank=rank, rot_n=rot_n, rank_n=rank, eps=1e-5)
    ops.latent_prep(proj, q, caches[0], step, **names)
    out = ops.latent_prompt(proj.clone(), ops.MatrixTiles(up.reshape(-1, rank), bf), caches[1], step, vdim=dim, scale=scale, gate=proj[:, H * hd + D:], **names)
    assert torch.equal(caches[0], caches[1])
    rows = caches[0].view(-1, D).double().cpu()
    at = 0
    for i, n in enumerate(lens):
        c = rows[[int(tables[i, t // page]) * page + t % page for t in range(n)]]
        hide = torch.full((n, n), float("-inf"), dtype=torch.float64).triu(1)
        for h in range(H):
            own = proj[at: at + n, h * hd: h * hd + dim].double().cpu()
            turned = q[at: at + n].view(n, H, D)[:, h, rank:].double().cpu()
            kv = c[:, :rank] @ up[h].double().cpu().T
            p = torch.softmax((own @ kv[:, :dim].T + turned @ c[:, rank:].T) * scale + hide, dim=-1)
            gate = torch.sigmoid(proj[at: at + n, H * hd + D + h].double().cpu())[:, None]
            close(out[at: at + n, h * dim: (h + 1) * dim], p @ kv[:, dim:] * gate, bf, tol16=1.2e-2)
        at += n


@pytest.mark.parametrize("lens", [[60], [90, 3, 40, 1]])
def test_prompts_over_keys_and_over_latents_lead_to_the_same_decoder(lens, monkeypatch):
    """Heads that latent_prompt is built for: prompts in one step, in one of its own and with the kernel over latents, and the tokens behind them, against the plain model."""
    from vllmini_amd import hybrid_ops as ops
    from vllmini_amd.hybrid_decoder import HybridDecoder
    from vllmini_amd.voduvik import VoduvikConfig, build_model

    c = cases.config([cases.attention(2, 64, 32, 64, 128, 0.1, mlp=cases.dense(64, 1.0)), cases.rglru(64, 1)], width=64)
    w, took, prompt = cases.tensors(c), [], ops.latent_prompt
    m = build_model(VoduvikConfig.from_json(c), w, torch.bfloat16, dev())
    monkeypatch.setattr(ops, "latent_prompt", lambda *a, **k: took.append(1) or prompt(*a, **k))
    toks = [cases.tokens(c, n + 2, i) for i, n in enumerate(lens)]
    want = [plain.forward(c, w, t)[0] for t in toks]
    for keys in (True, False):
        if not keys:
            monkeypatch.setattr(ops, "latent_prompt_pays", lambda step: False)
        took.clear()
        d = HybridDecoder(m, m.make_pool(640, 4, 16))
        ids = list(range(len(lens)))
        got = [d.prefill_batch(ids, [list(t[:n]) for t, n in zip(toks, lens)])]
        assert bool(took) == keys
        for k in range(2):
            got.append(d.decode(ids, torch.tensor([int(t[n + k]) for t, n in zip(toks, lens)])))
        for i, n in enumerate(lens):
            logits_close(torch.stack([x[i] for x in got]), want[i][n - 1: n + 2], torch.bfloat16)


@pytest.mark.parametrize("dim,rot,rank", [(128, 64, 512), (64, 32, 64)])
@pytest.mark.parametrize("counts,ctx", [([70], [0]), ([1, 70, 1], [40, 0, 3]), ([130, 5, 2, 1], [0, 17, 0, 0]), ([64, 1, 65], [0, 0, 0]), ([1] * 60 + [3], [7] * 60 + [0]),
                                        ([1, 9, 1, 1], [90, 0, 4, 64])])
def test_a_prompt_comes_to_the_same_whatever_shares_its_step(dim, rot, rank, counts, ctx):
    """The layer over a step of prompts and other portions against the same entries in two steps, the prompts' and the others': every bit of the results and of the cache."""
    from vllmini_amd import hybrid_layers as layers, hybrid_ops as ops
    from vllmini_amd.hybrid_decoder import HybridDecoder

    H, page, bf = 3, 32, torch.bfloat16
    g, D, hd, B = torch.Generator().manual_seed(dim + len(counts)), rank + rot, dim + rot, len(counts)
    w = lambda *s: torch.randn(s, generator=g).mul(s[-1] ** -0.5).to(bf).to(dev())      # noqa: E731
    layer = layers.LatentAttention(width=32, heads=H, dim=dim, rot=rot, vdim=dim, rank=rank, scale=hd ** -0.5, rot_base=500.0, rot_dims=rot, norm=layers.Norm(torch.ones(32, device=dev()), 32, 1e-5),
                                   q=w(H * hd, 32), dkv=w(D, 32), dkv_norm=torch.ones(rank, device=dev()), uk=w(H * dim, rank), uv=w(H * dim, rank), g=w(H, 32), o=w(32, H * dim), dtype=bf)
    counts, ctx = np.asarray(counts), np.asarray(ctx)
    T, at = int(counts.sum()), np.cumsum(counts) - counts
    proj = torch.randn(T, layer.w_in.N, generator=g).to(bf).to(dev())
    per = -(-(ctx + counts) // page)
    tables = np.zeros((B, per.max()), dtype=np.int64)
    for b in range(B):
        tables[b, :per[b]] = per[:b].sum() + np.arange(per[b])
    pages = torch.randn(int(per.sum()), page, D, generator=g).to(bf).to(dev())
    d = object.__new__(HybridDecoder)
    d.model, d._kinds = type("Model", (), {"dtype": bf}), [layer.tiling()]

    def run(own, splits=None, listed=False):
        """(the rows of the entries `own`, the cache) of a step of these entries alone; listed: with the prompts' tiles as a list."""
        n, c = counts[own], ctx[own]
        tok = np.concatenate([np.arange(at[b], at[b] + counts[b]) for b in own])
        a = {"entry": np.repeat(np.arange(len(own)), n), "pos": tok, "slots": [tok], "ctx": c, "state_slot": n * 0, "parity": n * 0, "tables": tables[own][None]}
        sec, _, _, plans = d._layout(a, n, np.arange(1), len(tok), len(own), tables.shape[1], int((c + n).max()))
        rt, sp, nt, spans = plans[0]
        assert "prompts" not in sec
        tiles = i32([(e, m) for e in np.flatnonzero(c == 0) for m in range(0, n[e] + 64, 64)]).view(-1, 2) if listed else None      # (one more than there are, each)
        plan = layers.AttentionPlan(i32(sec["tiles0"]).view(nt, 2), rt, splits or sp, None if spans is None else ops.PromptTiles(tiles, *spans))
        cache, rows, step = pages.clone(), [], layout(n, c, tables[own], page)
        res = type("Residual", (), {"branch_in": lambda self, *a: proj[torch.as_tensor(tok, device=dev())].clone(), "branch_out": lambda self, o, *a: rows.append(o)})()
        layer.run(res, step, {layer.tiling(): plan}, [cache])
        return rows[0], cache, plan

    prompts, others = np.flatnonzero(ctx == 0), np.flatnonzero(ctx > 0)
    got, cache, plan = run(np.arange(B))
    assert plan.prompts is not None
    again, pages_again, _ = run(np.arange(B), listed=True)
    assert torch.equal(got, again) and torch.equal(cache, pages_again)
    for own in (prompts, others):
        if len(own):
            want, alone, part = run(own, plan.splits if own is others else None)
            assert (part.prompts is not None) == (own is prompts) and (own is prompts or part.row_tiles == plan.row_tiles)
            for b, rows in zip(own, want.split(counts[own].tolist())):
                assert torch.equal(got[at[b]: at[b] + counts[b]], rows), b
                assert torch.equal(cache[tables[b, :per[b]]], alone[tables[b, :per[b]]])


def test_the_parts_of_latent_prompts_by_themselves():
    """The C entries for a step without a past, preparation and attention with a product between them, against the one call that has all three: every bit."""
    import ctypes

    from vllmini_amd import hybrid_ops as ops

    H, dim, rot, rank, lens, page, bf = 2, 128, 32, 128, [70, 1, 130], 16, torch.bfloat16
    g, T, D = torch.Generator(device=dev()).manual_seed(5), sum(lens), rank + rot
    proj = torch.randn(T, H * (dim + rot) + D + 32, generator=g, device=dev()).to(bf)
    w = ops.MatrixTiles(torch.randn(H * 2 * dim, rank, generator=g, device=dev()) * rank ** -0.5, bf)
    step = layout(lens, [0] * 3, np.arange(3 * 9).reshape(3, 9), page)
    step.fresh = True
    names = dict(norm_w=torch.ones(rank, device=dev()), freq=torch.rand(rot // 2, generator=g, dtype=torch.float64, device=dev()), heads=H, dim=dim, rot=rot, rank=rank, rot_n=rot, rank_n=rank, eps=1e-5)
    gate, caches = proj[:, H * (dim + rot) + D:], [torch.zeros((27, page, D), dtype=bf, device=dev()) for _ in range(2)]
    want = ops.latent_prompt(proj.clone(), w, caches[0], step, vdim=dim, scale=0.1, gate=gate, **names)
    own, rows, got, lib = proj.clone(), torch.empty((T, D), dtype=bf, device=dev()), torch.zeros_like(want), ops.load()
    stream = torch.cuda.current_stream().cuda_stream
    a = ops.PrepArgs(proj=own.data_ptr(), cache=caches[1].data_ptr(), norm_w=names["norm_w"].data_ptr(), freq=names["freq"].data_ptr(), ldp=own.stride(0), heads=H, dim=dim, rot=rot, rank=rank,
                     rot_n=rot, rank_n=rank, eps=1e-5, dtype=ops.DTYPES[bf], device=0)
    assert lib.vmi_hy_latent_prompt_prep(ctypes.byref(a), rows.data_ptr(), step.ref, stream) == 0
    kv = ops.product_tiles(rows[:, :rank], w)
    assert lib.vmi_hy_latent_prompt(own.data_ptr(), own.stride(0), kv.data_ptr(), kv.stride(0), rows.data_ptr(), gate.data_ptr(), gate.stride(0), got.data_ptr(), got.stride(0), H, dim, rot, dim,
                                    rank, max(lens), 0.1, ops.DTYPES[bf], 0, step.ref, stream) == 0
    assert torch.equal(got, want) and torch.equal(*caches)


def test_prompts_of_more_places_than_a_launch_has_workgroups():
    """Entries of one token each under a longest one of 65 535: places, entries and heads come to more than 2^24, and a token alone attends to its own value."""
    from vllmini_amd import hybrid_ops as ops

    H, dim, rot, rank, T, bf = 3, 64, 32, 64, 5500, torch.bfloat16
    g = torch.Generator(device=dev()).manual_seed(1)
    proj = torch.randn(T, H * (dim + rot) + rank + rot + 32, generator=g, device=dev()).to(bf)
    up = (torch.randn(H, 2 * dim, rank, generator=g, device=dev()) * rank ** -0.5).to(bf)
    step = layout([1] * T, [0] * T, np.arange(T)[:, None], 1)
    step.fresh, step.max_len = True, 65535
    assert H * T * -(-step.max_len // 64) >= 1 << 24
    cache, gate = torch.zeros((T, 1, rank + rot), dtype=bf, device=dev()), proj[:, H * (dim + rot) + rank + rot:]
    out = ops.latent_prompt(proj.clone(), ops.MatrixTiles(up.reshape(-1, rank), bf), cache, step, vdim=dim, scale=0.1, gate=gate, norm_w=torch.ones(rank, device=dev()),
                            freq=torch.ones(rot // 2, dtype=torch.float64, device=dev()), heads=H, dim=dim, rot=rot, rank=rank, rot_n=rot, rank_n=rank, eps=1e-5)
    value = cache[:, 0, :rank].float() @ up[:, dim:].reshape(-1, rank).float().T
    close(out, value.view(T, H, dim).mul(torch.sigmoid(gate[:, :H].float())[:, :, None]).reshape(T, -1), bf, tol16=8e-3)      # (two roundings to bfloat16)


# ---- the whole decoder -------------------------------------------------------------------------------------------------------------
_PLAIN = {}


def expected(name, toks):
    """Plain logits of a configuration's sequence (cached: several tests ask for prefixes of the same ones)."""
    key = (name, tuple(toks))
    if key not in _PLAIN:
        c = cases.CONFIGS[name]
        _PLAIN[key] = plain.forward(c, cases.tensors(c), toks)
    return _PLAIN[key]


def decoder(name, dtype, max_tokens=640, max_seqs=4, page=16, **kw):
    from vllmini_amd.hybrid_decoder import HybridDecoder
    from vllmini_amd.voduvik import VoduvikConfig, build_model

    c = cases.CONFIGS[name]
    m = build_model(VoduvikConfig.from_json(c), cases.tensors(c), dtype, dev())
    d = HybridDecoder(m, m.make_pool(max_tokens, max_seqs, page), **kw)
    g = torch.Generator(device=dev()).manual_seed(3)
    for t in d.pool.row_pages + d.pool.state:          # stale contents must never matter
        t.copy_(torch.empty(t.shape, device=dev()).uniform_(-4, 4, generator=g))
    return d


def logits_close(got, want, dtype, tol32=2e-4, tol16=0.12):
    got, want = got.double().cpu(), want.double().cpu()
    d = got - want
    d = d - d.mean(-1, keepdim=True)
    err = float((d.pow(2).mean(-1).sqrt() / want.std()).max())
    assert err <= (tol32 if dtype == torch.float32 else tol16), f"rms error / spread = {err:.3e}"


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("name", sorted(cases.CONFIGS))
def test_whole_prompt_and_the_stream_after_every_run(name, dtype):
    toks = cases.tokens(cases.CONFIGS[name], 90, 1)
    want, streams = expected(name, toks)
    d = decoder(name, dtype)
    d.pool.open(0)
    d.tap = []
    got = d.step([0], [toks], [list(range(90))])
    logits_close(got, want, dtype)
    assert len(d.tap) == len(streams)
    for a, b in zip(d.tap, streams):
        close(a, b, dtype, tol32=1e-4, tol16=8e-2)


def test_ids_come_from_the_host_from_the_device_or_from_both():
    """Prompts as lists, tensors of the host, tensors of the device, mixed in one step: the same logits; what is no token is refused as it was."""
    name = sorted(cases.CONFIGS)[0]
    a, b, c = ([int(t) for t in cases.tokens(cases.CONFIGS[name], n, s)] for n, s in ((7, 1), (1, 2), (20, 3)))
    got = []
    for form in (lambda k, t: t, lambda k, t: torch.tensor(t), lambda k, t: torch.tensor(t).to(dev()), lambda k, t: t if k == 1 else torch.tensor(t, dtype=torch.int32).to(dev())):
        d = decoder(name, torch.bfloat16)
        for k in range(3):
            d.pool.open(k)
        got.append(d.step([0, 1, 2], [form(k, t) for k, t in enumerate((a, b, c))]))
        got.append(d.decode([0, 1, 2], [5, 6, 7] if len(got) % 4 == 1 else torch.tensor([5, 6, 7]), use_graph=len(got) > 4))
    for g, h in zip(got[2:], got):
        assert torch.equal(g, h)
    for bad, kind in (([[d.model.vocab_size]], ValueError), ([[-1]], ValueError), ([[1 << 70]], RuntimeError), ([[]], IndexError)):
        with pytest.raises(kind):
            d.step([0], bad)


@pytest.mark.parametrize("name", sorted(cases.CONFIGS))
def test_many_tokens_take_the_dense_path_to_the_same_logits(name, monkeypatch):
    from vllmini_amd import hybrid_layers

    monkeypatch.setattr(hybrid_layers, "DENSE_MIN_TOKENS", 1)
    toks = cases.tokens(cases.CONFIGS[name], 90, 1)
    for dtype in BOTH:
        d = decoder(name, dtype)
        d.pool.open(0)
        logits_close(d.step([0], [toks], [list(range(90))]), expected(name, toks)[0], dtype)


@pytest.mark.parametrize("dtype", BOTH)
@pytest.mark.parametrize("name", sorted(cases.CONFIGS))
def test_portions_single_tokens_and_neighbours_do_not_change_the_logits(name, dtype):
    """Unequal requests cut in every way, pages and slots given back and used again, requests left out of steps."""
    c = cases.CONFIGS[name]
    lens = [90, 40, 3, 1, 66, 90]
    toks = [cases.tokens(c, 90, 1)[:n] for n in lens]       # prefixes of one sequence: one plain run checks all of them
    want = expected(name, cases.tokens(c, 90, 1))[0]
    d = decoder(name, dtype, max_tokens=16 * 14, max_seqs=3)
    rng = np.random.default_rng(5)
    sizes = [[90], [2, 3, 2, 31, 2], [1, 2], [1], [64, 2], [17] + [2] * 20 + [1] * 33]
    waiting, live, at, rows = list(range(6)), [], {}, {i: [] for i in range(6)}
    while waiting or live:
        while waiting and len(live) < 3 and len(d.pool.free_blocks) >= sum(-(-lens[i] // 16) for i in live) + -(-lens[waiting[0]] // 16) - \
                sum(len(d.pool.allocated_blocks[i]) for i in live):
            i = waiting.pop(0)
            d.pool.open(i)
            live.append(i)
            at[i] = 0
        now = [i for i in live if len(live) == 1 or rng.random() < 0.8] or live[:1]
        n = [sizes[i].pop(0) if sizes[i] else lens[i] - at[i] for i in now]
        got = d.step(now, [toks[i][at[i]:at[i] + k] for i, k in zip(now, n)], [list(range(k)) for k in n])
        for i, k, g in zip(now, n, got.split(n)):
            rows[i].append(g.cpu())
            at[i] += k
            if at[i] == lens[i]:
                d.pool.free(i)
                live.remove(i)
    for i in range(6):
        logits_close(torch.cat(rows[i]), want[: lens[i]], dtype)
    assert len(d.pool.free_blocks) == 14 and d.pool.free_state_slots == 3


@pytest.mark.parametrize("dtype", BOTH)
def test_long_decoding_from_one_token(dtype):
    name, n = "mixed", 330
    toks = cases.tokens(cases.CONFIGS[name], n, 9)
    want = expected(name, toks)[0]
    d = decoder(name, dtype, page=32)
    first = d.prefill(0, toks[:1])
    got = torch.cat([first[None]] + [d.decode([0], torch.tensor([t], device=dev())).clone() for t in toks[1:]])
    logits_close(got, want, dtype, tol32=5e-4)


@pytest.mark.parametrize("vendor", [False, True], ids=["streaming", "vendor"])
def test_graph_replay_equals_eager_steps(vendor, monkeypatch):
    """Both ways a layer's products may run, captured; eager steps run between the replays."""
    from vllmini_amd import hybrid_layers

    if vendor:
        monkeypatch.setattr(hybrid_layers, "DENSE_MIN_TOKENS", 1)
    name = "mixed"
    c = cases.CONFIGS[name]
    a, b = decoder(name, torch.bfloat16, pad_batch_to=4), decoder(name, torch.bfloat16)
    prompts = [cases.tokens(c, n, n) for n in (5, 30, 100)]
    la, lb = a.prefill_batch([0, 1, 2], prompts), b.prefill_batch([0, 1, 2], prompts)
    for i in range(40):      # every replay against the eager step; the batch shrinks once, contexts cross a split bucket
        ids = [0, 1, 2] if i < 25 else [0, 2]
        tok = b.greedy(lb[: len(ids)] if i != 25 else lb[[0, 2]])
        la, lb = a.decode(ids, tok, use_graph=True).clone(), b.decode(ids, tok).clone()
        logits_close(la, lb, torch.bfloat16, tol16=2e-2)
    assert len(a._sets) >= 1 and all(s["graph"] is not None for s in a._sets.values())
    assert torch.isfinite(la).all()


def test_step_refuses_what_does_not_fit():
    d = decoder("no_loop", torch.float32, max_tokens=64, max_seqs=2)
    d.pool.open(0)
    with pytest.raises(ValueError, match="token id"):
        d.step([0], [[1, 130]])
    with pytest.raises(ValueError, match="wanted places"):
        d.step([0], [[1, 2]], [[2]])
    with pytest.raises(RuntimeError, match="free blocks|blocks per layer"):
        d.step([0], [[1] * 65])
    assert d.pool.seq_len(0) == 0 and d.step([0], [[1, 2]], [[]]) is None
    with pytest.raises(RuntimeError):
        d.prefill_batch([1], [[1] * 100])
    assert 1 not in d.pool.allocated_blocks and d.pool.free_state_slots == 1


# ---- generation through the framework's entry points ----------------------------------------------------------------------------------
def _plain_greedy(name, prompt, n):
    c = cases.CONFIGS[name]
    w, seq = cases.tensors(c), list(prompt)
    for _ in range(n):
        seq.append(int(plain.forward(c, w, seq)[0][-1].argmax()))
    return seq


@pytest.fixture(scope="module")
def greedy_case():
    name = "mixed"
    prompts = [cases.tokens(cases.CONFIGS[name], n, 40 + n) for n in (1, 19, 34)]
    return name, prompts, [_plain_greedy(name, p, 12) for p in prompts]


@pytest.mark.parametrize("kw", [{}, {"use_graph": True}, {"prefill_chunk": 7}, {"prefill_chunk": 16, "use_graph": True}, {"preempt_after": 4}],
                         ids=["plain", "graph", "chunks", "chunks+graph", "preempted"])
def test_greedy_generation_through_the_scheduler(kw, greedy_case):
    from vllmini_amd.scheduler import BatchScheduler

    name, prompts, want = greedy_case
    kw, blocks = dict(kw), 12
    after = kw.pop("preempt_after", 0)
    d = decoder(name, torch.float32, max_tokens=16 * blocks, max_seqs=3)
    sch = BatchScheduler(d, max_length=46, eos_token_id=-1, max_batch=3, sampler=lambda lg, generator=None: d.greedy(lg), **kw)
    ids = [sch.submit(p, max_new_tokens=12) for p in prompts]
    if after:                                          # a victim leaves for the host in mid-run and comes back by itself
        sch.run(max_steps=after)
        assert sch._make_room(exclude=()) and len(sch.swapped) == 1
    sch.run(max_steps=500)
    assert [sch.sequences[i] for i in ids] == want and not sch.pending() and not sch.rejected
    assert sch.stats["resumes"] == (1 if after else 0)
    assert len(d.pool.free_blocks) == blocks and d.pool.free_state_slots == 3


def test_swapped_out_sequences_continue_where_they_were():
    name = "mixed"
    c = cases.CONFIGS[name]
    d = decoder(name, torch.float32)
    toks = cases.tokens(c, 90, 1)
    want = expected(name, toks)[0]
    d.prefill(0, toks[:50])
    d.prefill(1, toks[:33])
    d.pool.swap_out(0)
    d.prefill(2, cases.tokens(c, 60, 8))               # takes the blocks and the slot that came free
    d.pool.free(1)
    assert d.pool.swap_in(0)
    got = torch.cat([d.step([0], [toks[50:70]], [list(range(20))])] + [d.decode([0], [t]) for t in toks[70:80]])
    logits_close(got, want[50:80], torch.float32)


def test_sampling_from_float_logits_stays_inside_the_top_k():
    from vllmini_amd.scheduler import sample_top_k

    lg = torch.randn(6, 203, device=dev())
    g = torch.Generator(device=dev()).manual_seed(0)
    top = lg.topk(4, -1).indices
    for _ in range(20):
        t = sample_top_k(lg, 4, 0.7, generator=g)
        assert ((top == t[:, None]).any(-1)).all()


def test_command_line_generation_and_trace_replay(tmp_path, greedy_case):
    name, prompts, want = greedy_case
    c = cases.CONFIGS[name]
    folder = cases.write_model(tmp_path / "model", c, cases.tensors(c))
    args = [a for p in prompts for a in ("--prompt-ids", ",".join(map(str, p)))]
    r = subprocess.run([sys.executable, "-m", "vllmini_amd", "generate", "--model", folder, "--dtype", "float32", "--max-new-tokens", "12",
                        "--prefill-chunk", "9", *args], capture_output=True, text=True, cwd=REPO, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    got = [json.loads(x) for x in r.stdout.splitlines()]
    assert [g["prompt"] + g["generated"] for g in got] == want
    out = tmp_path / "out"
    out.mkdir()
    toks = cases.tokens(c, 90, 1)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": toks[:40], "want": [0, 39]}, {"id": "b", "tokens": toks[:2], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": toks[2:3], "want": []}], "end": ["a"]},
             {"step": 2, "entries": [{"id": "b", "tokens": toks[3:70], "want": [66]}, {"id": "c", "tokens": toks[:1], "want": [0]}], "end": ["b", "c"]}]
    r = subprocess.run([os.path.join(REPO, "bin", "trace_run"), "--model", folder, "--dtype", "float32", "--out", str(out), "--max-tokens", "256"],
                       input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split("\n")[:3] == ["done 0", "done 1", "done 2"], r.stderr[-2000:]
    assert not (out / "1.f32").exists()
    ref = expected(name, toks)[0]
    read = lambda n: torch.from_numpy(np.fromfile(out / n, "<f4").reshape(-1, c["vocab"]))      # noqa: E731
    logits_close(read("0.f32"), ref[[0, 39]], torch.float32)
    logits_close(read("2.f32"), ref[[69, 0]], torch.float32)
