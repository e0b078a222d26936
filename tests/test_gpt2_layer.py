"""The decode harness's own library (include/vmi_gpt2_layer.h): CPU checks of its C-ABI, GPU checks of
the linear-layer kernels against a torch fp32 restatement of the module chain they replace (vllmini/model/gpt2.py:14-15,
117-128, 130-135) with the chain's own rounding points, and of the harness that runs on them."""
from __future__ import annotations

import ctypes
import os
import re
import subprocess
from types import SimpleNamespace

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests import tile_cases

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    src = open(os.path.join(REPO, "include", "vmi_gpt2_layer.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(vmi_gpt2_[a-z0-9_]+)\s*\(", src)))


def test_layer_library_exports_its_header_and_nothing_else():
    from vllmini_amd import build, gpt2_layer

    path = build.build_layer()
    declared = _declared()
    assert "vmi_gpt2_linear_f16" in declared and set(declared) == set(gpt2_layer.SIGNATURES)
    r = subprocess.run(["nm", "-D", "--defined-only", path], capture_output=True, text=True, check=True)
    funcs = {ln.split()[-1] for ln in r.stdout.splitlines() if ln.strip() and ln.split()[-2] in "TtWw"}
    assert funcs == set(declared), funcs ^ set(declared)
    lib = gpt2_layer.load()
    assert lib.vmi_gpt2_layer_abi_version() == gpt2_layer.ABI_VERSION == 1
    assert lib.vmi_gpt2_layer_target_arch() == b"gfx950"


def test_layer_entry_refuses_bad_arguments_without_touching_a_device():
    from vllmini_amd import gpt2_layer

    lib = gpt2_layer.load()
    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf) // 16 * 16 + 16
    call = lambda x, w, y, M, N, K, epi, res=None: lib.vmi_gpt2_linear_f16(x, K, w, None, None, None, 0.0, res, N, y, N, M, N, K,  # noqa: E731
                                                                           epi, 0, 0, None)
    assert call(None, p, p, 1, 16, 32, 0) == 1                      # null x
    assert call(p, p, p, 1, 16, 32, 3) == 1                         # unknown epilogue
    assert call(p, p, p, 1, 16, 32, 2) == 1                         # residual epilogue without a residual
    assert b"residual" in lib.vmi_gpt2_layer_last_error()
    assert call(p, p, p, 1, 16, 48, 0) == 2                         # K % 32
    assert call(p, p, p, 1, 24, 32, 0) == 2                         # N % 16
    assert call(p, p, p, 1, 16, 4640, 0) == 2                       # row tile past a CU's LDS
    assert b"K % 32" in lib.vmi_gpt2_layer_last_error()
    assert not gpt2_layer.supports(4, 24, 32) and gpt2_layer.supports(4, 384, 128)
    assert gpt2_layer.kernel_name(4, 64, 2080, True) is None and gpt2_layer.kernel_name(4, 64, 2080, False) is not None


def test_layer_picks_for_the_gpt2_small_decode_step():
    """The four launches of a layer at batch 256: 32-row tiles where that leaves workgroups for most of the chip, 16-row
    tiles otherwise, the K range of a slab over two waves from 48 k-steps on."""
    from vllmini_amd import gpt2_layer as gl

    assert gl.kernel_name(256, 2304, 768, True, gl.EPI_BIAS) == "bm32_nw4_ks1_r2_ln_bias"
    assert gl.kernel_name(256, 768, 768, False, gl.EPI_BIAS_RESIDUAL) == "bm16_nw4_ks1_r2_residual"
    assert gl.kernel_name(256, 3072, 768, True, gl.EPI_BIAS_GELU) == "bm32_nw4_ks1_r2_ln_gelu"
    assert gl.kernel_name(256, 768, 3072, False, gl.EPI_BIAS_RESIDUAL) == "bm16_nw4_ks2_r4_residual"
    assert gl.kernel_name(3, 384, 128, True, gl.EPI_BIAS) == "bm16_nw4_ks1_r2_ln_bias"
    # few rows (one sequence per step) x a long K: 16-column workgroups with the K range over their four waves
    assert gl.kernel_name(1, 768, 3072, False, gl.EPI_BIAS_RESIDUAL) == "bm16_nw1_ks4_r2_residual"
    assert gl.kernel_name(64, 768, 3072, False, gl.EPI_BIAS_RESIDUAL) == "bm16_nw1_ks4_r2_residual"
    assert gl.kernel_name(64, 768, 768, False, gl.EPI_BIAS_RESIDUAL) == "bm16_nw4_ks1_r2_residual"


@pytest.mark.parametrize("L,E,mb", [(4, 768, 134), (12, 768, 247), (12, 256, 45)])
def test_pages_go_past_the_caches_where_they_and_the_weights_leave_them(L, E, mb):
    """The rule of a decode step, in the sizes of GPT-2 and smaller: by the tokens whose pages no longer fit beside the weights."""
    from vllmini_amd import ops
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder

    def holds(numel):
        return SimpleNamespace(numel=lambda: numel, element_size=lambda: 2)

    d, names = object.__new__(GPT2PagedDecoder), ops.variant_names()
    d.dims, d._cold = GPT2Dims(n_embd=E, n_head=E // 64, n_layer=L), None
    d.pool = SimpleNamespace(key_cache=torch.empty(0, dtype=torch.float16), kv_cache_dtype="auto", block_size=16)
    d._step_weights = GPT2PagedDecoder.step_weights({"lm_head.weight": holds(50257 * E), "transformer.wte.weight": holds(50257 * E), "transformer.wpe.weight": holds(1024 * E), **{f"transformer.h.{i}": holds(12 * E * E) for i in range(L)}})
    assert abs(d._step_weights / 1e6 - mb) < 2
    fits = ((248 << 20) - d._step_weights) // (4 * L * E)
    assert not d._pages_leave_the_cache(fits) and d._pages_leave_the_cache(fits + 1)
    at = {n: i + 1 for i, n in enumerate(names)}
    for name, B, to in (("d64_h1_w16_u2_nt0", 1, "d64_h1_w16_u1_nt1"), ("d64_h1_w8_u1_nt0", 32, "d64_h1_w8_u1_nt1"), ("d64_h1_w4_u2_nt0", 1, "d64_h1_w4_u2_nt0"), ("d64_h1_w4_u2_nt0", 48, "d64_h1_w4_u1_nt1"),
                        ("d64_h1_w8_u1_nt1", 64, "d64_h1_w8_u1_nt1")):
        assert names[d._past_caches(at[name], B) - 1] == to
    d._step_weights = (256 << 20) + 1
    assert names[d._past_caches(at["d64_h1_w4_u2_nt0"], 48) - 1] == "d64_h1_w4_u2_nt0" and names[d._past_caches(at["d64_h1_w16_u2_nt0"], 48) - 1] == "d64_h1_w16_u1_nt1"


def test_pinned_memory_that_cannot_be_waited_for_is_not_given_back(monkeypatch):
    """PinnedBuffer: a launch may still read what nobody holds any more.  Waited for where that is possible; while a stream of the thread is captured, and where waiting fails, the memory is kept until its event says that the launch has run."""
    from vllmini_amd import staging

    class Event:
        waited, done, fails = 0, False, False

        def record(self):
            pass

        def synchronize(self):
            if self.fails:
                raise RuntimeError("not now")
            Event.waited += 1

        def query(self):
            return self.done

    empty = torch.empty
    monkeypatch.setattr(staging.torch, "empty", lambda n, dtype, pin_memory: empty(n, dtype=dtype))
    monkeypatch.setattr(staging.torch.cuda, "Event", Event)
    capturing = [False]
    monkeypatch.setattr(staging.torch.cuda, "is_current_stream_capturing", lambda: capturing[0])

    def dropped(fails, captured):
        b = staging.PinnedBuffer(64)
        b.read()
        event, at = b._read, b.tensor.data_ptr()
        event.fails, capturing[0] = fails, captured
        del b
        capturing[0] = False
        return event, at

    assert not staging._kept
    dropped(False, False)
    assert Event.waited == 1 and not staging._kept
    for fails, captured in ((True, False), (False, True)):
        event, at = dropped(fails, captured)
        assert Event.waited == 1 and [t.data_ptr() for _, t in staging._kept] == [at]
        staging.PinnedBuffer(64)
        assert len(staging._kept) == 1
        event.done = True
        staging.PinnedBuffer(64)
        assert not staging._kept


def test_linears_of_few_rows_past_1536_columns_count_the_rounds_of_a_die():
    """Where a workgroup has a compute unit to itself, the kernels for few rows end when the die with the most column blocks does: three of its rounds are behind one of tiles, two are level, and as the widths go these lie at
    other numbers of rows."""
    from vllmini_amd import gpt2_layer as gl

    def slabs(M, N, K, ln=False, epi=None):
        return gl.load().vmi_gpt2_linear_slabs(M, N, K, int(ln), gl.EPI_BIAS_RESIDUAL if epi is None else epi)

    for N, K, few, tiles in ((640, 2560, 336, 352), (576, 2304, 336, 352), (896, 3584, 144, 160), (704, 2816, 320, 352)):
        assert slabs(few, N, K) and not slabs(tiles, N, K), (N, K)
    assert slabs(448, 640, 2560) == 2 and slabs(384, 768, 3072) == 2 and slabs(128, 1152, 4608) == 1 and not slabs(160, 1152, 4608)
    assert slabs(512, 3072, 768, True, gl.EPI_BIAS_GELU) == 6 and slabs(512, 768, 768) == 2 and not slabs(1040, 768, 768) and not slabs(8, 768, 768, True)


# ---- GPU ---------------------------------------------------------------------------------------------------------------

def _chain(x, w, b, ln=None, gelu=False, residual=None):
    """The torch module chain in fp32 with ITS rounding points: layer_norm -> half, linear (fp32 sums) + bias -> half,
    GELU (erf) -> half | residual add -> half."""
    xf = x.float()
    if ln is not None:
        xf = F.layer_norm(xf, (x.shape[1],), ln[0].float(), ln[1].float(), ln[2]).half().float()
    y = xf.double() @ w.double().t()
    if b is not None:
        y = y + b.double()
    y = y.float().half()
    if gelu:
        y = F.gelu(y.float()).half()
    if residual is not None:
        y = (residual.float() + y.float()).half()
    return y


def _close(got, ref, what):
    g, r = got.float().cpu().numpy().astype(np.float64), ref.float().cpu().numpy().astype(np.float64)
    assert np.isfinite(g).all(), what
    # fp32 sums in another order may cross a rounding boundary of the half output: one half ulp of the value (2^-10 relative),
    # twice over for the second rounding of the GELU / residual epilogues
    tol = 2e-3 * np.abs(r) + 2e-3 * max(1e-3, np.abs(r).max()) * 0.25 + 1e-4
    bad = np.abs(g - r) > tol
    assert not bad.any(), (what, int(bad.sum()), float(np.abs(g - r).max()))


SHAPES = [  # (N, K, ln, epi)    GPT-2 small's four layers, the tiny fixture's, and shapes that leave partial tiles
    (2304, 768, True, "bias"), (768, 768, False, "res"), (3072, 768, True, "gelu"), (768, 3072, False, "res"),
    (384, 128, True, "bias"), (128, 128, False, "res"), (512, 128, True, "gelu"), (128, 512, False, "res"),
    (80, 96, True, "gelu"), (128, 2048, False, "gelu"), (16, 32, False, "bias"), (208, 1568, False, "res"), (2320, 800, True, "bias"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 5, 16, 33, 100, 256, 300])
def test_linear_kernels_match_the_module_chain(M):
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(M)
    for N, K, ln, epi in SHAPES:
        x = (torch.randn(M, K, generator=g) * 1.5 + 0.3).half().to(dev)
        w = (torch.randn(N, K, generator=g) * (0.6 / K ** 0.5)).half().to(dev)
        b = (torch.randn(N, generator=g) * 0.1).half().to(dev)
        lnp = ((1 + 0.2 * torch.randn(K, generator=g)).half().to(dev), (0.1 * torch.randn(K, generator=g)).half().to(dev), 1e-5) \
            if ln else None
        res = torch.randn(M, N, generator=g).half().to(dev) if epi == "res" else None
        got = gl.linear(x, w, b, ln=lnp, gelu=epi == "gelu", residual=res)
        ref = _chain(x, w, b, lnp, epi == "gelu", res)
        _close(got, ref, (M, N, K, ln, epi, gl.kernel_name(M, N, K, ln)))
        # the packed weight form holds the same values in another order: the same sums in the same order, the same bits
        assert torch.equal(gl.linear(x, gl.pack_weight(w), b, ln=lnp, gelu=epi == "gelu", residual=res), got), (M, N, K)
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_linear_layout_is_not_transposed_anywhere():
    """x = one-hot rows and a weight whose entry names its (n, k): every output element must be the entry its row's hot k and
    its column n select — a swapped row/column map of the MFMA result, or a k-group permutation, cannot pass."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    for M, N, K in ((48, 64, 64), (256, 768, 3072), (40, 2304, 768)):
        hot = (torch.arange(M) * 37 + 5) % K
        x = torch.zeros(M, K, dtype=torch.float16)
        x[torch.arange(M), hot] = 1
        n, k = torch.meshgrid(torch.arange(N), torch.arange(K), indexing="ij")
        w = (((n * 7 + k * 13) % 1024).float() / 64 - 8).half()       # exactly representable, asymmetric in (n, k)
        got = gl.linear(x.to(dev), w.to(dev), None).cpu()
        assert torch.equal(got, w[:, hot].t().contiguous()), (M, N, K)
        assert torch.equal(gl.linear(x.to(dev), gl.pack_weight(w.to(dev)), None).cpu(), got), (M, N, K)


@pytest.mark.gpu
def test_linear_in_place_residual_strided_input_no_bias_and_graph_replay():
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(3)
    M, E = 64, 768
    qkv = torch.randn(M, 3 * E, generator=g).half().to(dev)
    w = (torch.randn(E, E, generator=g) * 0.02).half().to(dev)
    b = (torch.randn(E, generator=g) * 0.1).half().to(dev)
    x0 = torch.randn(M, E, generator=g).half().to(dev)
    xs = qkv[:, E:2 * E]                                  # rows 3E apart
    ref = _chain(xs, w, b, residual=x0)
    x = x0.clone()
    assert gl.linear(xs, w, b, residual=x, out=x) is x    # out aliases the residual
    _close(x, ref, "in place")
    _close(gl.linear(xs, w, None), _chain(xs, w, None), "no bias")
    with pytest.raises(RuntimeError, match="alternative"):
        gl.linear(xs, w, b, gelu=True, residual=x0)
    with pytest.raises(RuntimeError, match="must not alias x"):
        gl.linear(x0, w, b, out=x0)
    with pytest.raises(RuntimeError, match="K % 32"):
        gl.linear(qkv[:, :48], w[:, :48].contiguous(), b)
    with pytest.raises(RuntimeError, match="no CPU path"):
        gl.linear(x0.cpu(), w.cpu(), b.cpu())
    # captured in a hipGraph: replays give the eager bits
    s = torch.cuda.Stream(dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    y = torch.empty(M, E, dtype=torch.float16, device=dev)
    with torch.cuda.stream(s):
        gl.linear(xs, w, b, residual=x0, out=y)
    torch.cuda.current_stream(dev).wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        gl.linear(xs, w, b, residual=x0, out=y)
    y.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, x)


@pytest.mark.gpu
def test_gpt2_small_decode_on_native_layers_tracks_the_torch_modules():
    """GPT-2 small, random weights, 24 sequences: the step on the native layer kernels against the same step on torch modules
    (same pools, same tokens): logits agree to fp16 GEMM rounding, the argmax wherever the top-2 gap is not tiny; and the
    hipGraph replay of the native step gives the eager native bits."""
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dev = torch.device("cuda:0")
    dims = GPT2Dims()
    sd = random_state_dict(dims, dev, seed=1)
    B = 24

    def make(native):
        pool = PagedKVPool(B * dims.n_layer * 4 + 8, dims.n_head, dims.head_size, 16, 5, dims.n_layer, device=dev, max_seqs=B)
        dec = GPT2PagedDecoder(dims, sd, pool, native_layers=native)
        for s in range(B):
            dec.prefill(s, [(7 * s + j) % dims.vocab_size for j in range(1 + s % 13)])
        return dec

    nat, ref, rep = make(True), make(False), make(True)
    assert nat.native_layers and not ref.native_layers
    rng = np.random.default_rng(0)
    ids = list(range(B))
    for step in range(6):
        toks = rng.integers(0, dims.vocab_size, B).tolist()
        a = nat.decode(ids, toks).float()
        b = ref.decode(ids, toks).float()
        c = rep.decode(ids, toks, use_graph=True).float()
        assert torch.equal(a, c)
        err = (a - b).abs().max().item()
        assert err <= 2e-2 + 1e-2 * b.abs().max().item(), err
        top2 = b.topk(2, dim=1).values
        decisive = (top2[:, 0] - top2[:, 1]) > 5e-2
        assert (a.argmax(1) == b.argmax(1))[decisive].all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,H,D,BS", [(1, 12, 64, 16), (37, 12, 64, 16), (256, 12, 64, 16), (20, 2, 64, 16), (9, 4, 128, 8)])
def test_qkv_projection_with_the_cache_write_leaves_reshape_and_caches_bytes(M, H, D, BS):
    """vmi_gpt2_linear_qkv_cache_f16 = linear() + cache_ops.reshape_and_cache on its k / v views: the same qkv bits, the same
    cache bytes (rows with a negative slot skipped, everything else in the caches untouched)."""
    from vllmini_amd import cache_ops, gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(M + D)
    E = H * D
    K = E
    NB = max(4, (M + BS - 1) // BS * 3)
    x = torch.randn(M, K, generator=g).half().to(dev)
    w = (torch.randn(3 * E, K, generator=g) * (0.6 / K ** 0.5)).half().to(dev)
    b = (torch.randn(3 * E, generator=g) * 0.1).half().to(dev)
    lnp = ((1 + 0.2 * torch.randn(K, generator=g)).half().to(dev), (0.1 * torch.randn(K, generator=g)).half().to(dev), 1e-5)
    kc0 = torch.randn(NB, H, D // 8, BS, 8, generator=g).half().to(dev)
    vc0 = torch.randn(NB, H, D, BS, generator=g).half().to(dev)
    slots = torch.randperm(NB * BS, generator=g)[:M].to(torch.int64)
    if M > 4:
        slots[3] = -1
    slots = slots.to(dev)
    for weight in (w, gl.pack_weight(w)):
        ref_qkv = gl.linear(x, weight, b, ln=lnp)
        kr, vr = kc0.clone(), vc0.clone()
        k, v = (ref_qkv[:, j * E:(j + 1) * E].view(M, H, D) for j in (1, 2))
        cache_ops.reshape_and_cache(k, v, kr, vr, slots, "auto", 1.0)
        kg, vg = kc0.clone(), vc0.clone()
        got = gl.linear_qkv_cache(x, weight, b, kg, vg, slots, H, ln=lnp)
        torch.cuda.synchronize()
        assert torch.equal(got, ref_qkv)
        assert torch.equal(kg.view(torch.int16), kr.view(torch.int16)) and torch.equal(vg.view(torch.int16), vr.view(torch.int16))
        assert not torch.equal(kg, kc0)
    with pytest.raises(RuntimeError, match="float16 caches"):
        gl.linear_qkv_cache(x, w, b, kc0.to(torch.uint8), vc0.to(torch.uint8), slots, H, ln=lnp)


@pytest.mark.gpu
def test_decoder_with_the_scatter_in_c_attn_is_bit_identical_to_the_call_pair(golden_dir):
    """The harness with reshape_and_cache's copy folded into the q / k / v projection: same logits, same caches, bit for bit,
    as with the reference's call pair — eager and replayed from a hipGraph."""
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dev = torch.device("cuda:0")
    dims = GPT2Dims()
    sd = random_state_dict(dims, dev, seed=2)
    B = 9

    def make(scatter):
        pool = PagedKVPool(B * dims.n_layer * 4 + 8, dims.n_head, dims.head_size, 16, 5, dims.n_layer, device=dev, max_seqs=B)
        dec = GPT2PagedDecoder(dims, sd, pool, scatter_in_c_attn=scatter)
        for s in range(B):
            dec.prefill(s, [(11 * s + j) % dims.vocab_size for j in range(1 + (5 * s) % 17)])
        return dec

    pair, scat, scat_g = make(False), make(True), make(True)
    rng = np.random.default_rng(1)
    ids = list(range(B))
    for step in range(8):
        toks = rng.integers(0, dims.vocab_size, B).tolist()
        a = pair.decode(ids, toks)
        b = scat.decode(ids, toks)
        c = scat_g.decode(ids, toks, use_graph=True)
        assert torch.equal(a, b) and torch.equal(a, c)
    assert torch.equal(pair.pool.key_cache, scat.pool.key_cache) and torch.equal(pair.pool.value_cache, scat.pool.value_cache)
    assert torch.equal(pair.pool.key_cache, scat_g.pool.key_cache)
    with pytest.raises(ValueError, match="scatter_in_c_attn"):
        GPT2PagedDecoder(dims, sd, pair.pool, scatter_in_c_attn=True, fused_append=True)


@pytest.mark.gpu
def test_linear_kernels_over_random_shapes():
    """Every pick — 32 / 16-row tiles, K over one, two or four waves, two- and four-chunk rings, partial chunks, partial row and
    column tiles — on 80 random (M, N, K, LayerNorm, epilogue) against the module chain, plain and packed weights."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    rng = np.random.default_rng(5)
    g = torch.Generator(device="cpu").manual_seed(5)
    seen = set()
    for case in range(80):
        M = int(rng.choice([1, 2, 7, 16, 17, 31, 32, 33, 63, 64, 100, 129, 255, 256, 257, 400, 600]))
        N = 16 * int(rng.integers(1, 200))
        ln = bool(rng.integers(0, 2))
        K = 32 * int(rng.integers(1, (2048 if ln else 4608) // 32 + 1))
        epi = ["bias", "gelu", "res"][int(rng.integers(0, 3))]
        x = (torch.randn(M, K, generator=g) * 1.5 + 0.3).half().to(dev)
        w = (torch.randn(N, K, generator=g) * (0.6 / K ** 0.5)).half().to(dev)
        b = (torch.randn(N, generator=g) * 0.1).half().to(dev) if rng.integers(0, 4) else None
        lnp = ((1 + 0.2 * torch.randn(K, generator=g)).half().to(dev), (0.1 * torch.randn(K, generator=g)).half().to(dev), 1e-5) \
            if ln else None
        res = torch.randn(M, N, generator=g).half().to(dev) if epi == "res" else None
        name = gl.kernel_name(M, N, K, ln)
        seen.add(name.rsplit("_", 1)[0])
        got = gl.linear(x, w, b, ln=lnp, gelu=epi == "gelu", residual=res)
        _close(got, _chain(x, w, b, lnp, epi == "gelu", res), (case, M, N, K, ln, epi, name))
        assert torch.equal(gl.linear(x, gl.pack_weight(w), b, ln=lnp, gelu=epi == "gelu", residual=res), got), (case, M, N, K)
    torch.cuda.synchronize()
    assert len(seen) >= 6, seen      # the draw reached most of the kernel family


@pytest.mark.gpu
def test_embed_and_argmax_equal_torch():
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(9)
    V, P, E = 50257, 1024, 768
    wte = torch.randn(V, E, generator=g).half().to(dev)
    wpe = torch.randn(P, E, generator=g).half().to(dev)
    for T in (1, 5, 256):
        ids = torch.randint(0, V, (T,), generator=g).to(dev)
        pos = torch.randint(0, P, (T,), generator=g).to(dev)
        assert torch.equal(gl.embed(ids, pos, wte, wpe), wte[ids] + wpe[pos])
    # argmax: rows of 50 257 halves start at every alignment; ties go to the first maximum; a row slice of a wider tensor
    for B in (1, 3, 9, 256):
        logits = torch.randn(B, V, generator=g).half().to(dev)
        assert torch.equal(gl.argmax(logits), logits.argmax(-1))
    tie = torch.zeros(4, V, dtype=torch.float16, device=dev)
    tie[0, 777] = tie[0, 40000] = 3.0
    tie[1, V - 1] = 1.0
    tie[2, 0] = tie[2, 1] = 2.0
    tie[3] = -5.0
    assert gl.argmax(tie).tolist() == [777, V - 1, 0, 0]
    wide = torch.randn(6, V + 37, generator=g).half().to(dev)
    assert torch.equal(gl.argmax(wide[:, 5:5 + 1000]), wide[:, 5:5 + 1000].argmax(-1))
    small = torch.randn(7, 13, generator=g).half().to(dev)
    assert torch.equal(gl.argmax(small), small.argmax(-1))
    with pytest.raises(RuntimeError, match="half logits"):
        gl.argmax(logits.float())


@pytest.mark.gpu
def test_graph_replay_across_a_pick_threshold_keeps_one_graph_per_launch_geometry():
    """32 sequences whose contexts grow from 505 to 520 tokens cross a threshold of the attention pick (the variant id is baked
    into a captured step): the harness keeps ONE graph per variant and switches between them — never a capture in the middle of
    a run once both exist — and the replayed logits are the eager ones."""
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dev = torch.device("cuda:0")
    dims = GPT2Dims(n_layer=2)
    sd = random_state_dict(dims, dev, seed=4)
    B, ctx = 32, 505

    def make():
        pool = PagedKVPool(B * dims.n_layer * 34 + 8, dims.n_head, dims.head_size, 16, 35, dims.n_layer, device=dev, max_seqs=B,
                           multi_block_prefill=True)
        dec = GPT2PagedDecoder(dims, sd, pool)
        for s in range(B):
            dec.prefill(s, [(3 * s + j) % dims.vocab_size for j in range(ctx)])
        return dec

    eager, graph = make(), make()
    rng = np.random.default_rng(2)
    ids = list(range(B))
    variants = []
    for step in range(15):
        toks = rng.integers(0, dims.vocab_size, B).tolist()
        a = eager.decode(ids, toks)
        b = graph.decode(ids, toks, use_graph=True)
        variants.append(graph._static["variant"])
        assert torch.equal(a, b), step
    assert len(set(variants)) == len(graph._graph)
    captured = dict(graph._graph)
    for step in range(3):      # more steps on variants already seen: the same graph objects, nothing captured
        toks = rng.integers(0, dims.vocab_size, B).tolist()
        assert torch.equal(eager.decode(ids, toks), graph.decode(ids, toks, use_graph=True))
    assert all(graph._graph[v][0] is captured[v][0] for v in captured)


@pytest.mark.gpu
def test_top_k_sampling_kernel_draws_from_the_reference_distribution():
    """vmi_gpt2_sample_top_k_f16 against the torch chain the reference spells out (scheduler.py:144-153): the k survivors are
    torch.topk's, the draw at a given uniform number is the inverse CDF over their softmax in descending order, ties go to the
    smaller index, rows of equal logits (the block-wide path) work, and the frequencies of many draws match the probabilities."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(11)
    V = 50257
    for B, k, temp in ((1, 50, 1.0), (7, 50, 0.7), (256, 50, 1.0), (5, 1, 1.0), (4, 64, 1.3), (3, 13, 1.0)):
        logits = (torch.randn(B, V, generator=g) * 2).half().to(dev)
        vals, idx = torch.topk(logits.float() / temp, k, dim=-1)
        cdf = torch.softmax(vals, -1).double().cumsum(-1)
        for u in (0.0, 0.173, 0.5, 0.9371, 0.999999):
            uu = torch.full((B,), u, dtype=torch.float32, device=dev)
            got = gl.sample_top_k(logits, k, temp, uniform=uu)
            j = (cdf >= u * cdf[:, -1:]).int().argmax(-1)                       # first survivor whose cumulative mass reaches u
            want = idx.gather(-1, j[:, None]).squeeze(-1)
            # (a draw that sits within float rounding of a CDF step may land on the neighbour: compare there by mass)
            bad = got != want
            if bad.any():
                pos = (idx == got[:, None]).int().argmax(-1)
                assert ((idx == got[:, None]).any(-1))[bad].all()
                near = (cdf.gather(-1, pos[:, None]).squeeze(-1) - u * cdf[:, -1]).abs() < 1e-5
                near |= (cdf.gather(-1, (pos - 1).clamp(min=0)[:, None]).squeeze(-1) - u * cdf[:, -1]).abs() < 1e-5
                assert near[bad].all(), (B, k, u)
    # ties: equal logits everywhere -> the k smallest indices, equal mass each; a few equal maxima -> smaller index first
    flat = torch.zeros(3, V, dtype=torch.float16, device=dev)
    for u, want in ((0.0, 0), (0.51, 25), (0.999, 49)):
        assert gl.sample_top_k(flat, 50, 1.0, uniform=torch.full((3,), u, device=dev)).tolist() == [want] * 3
    peaks = torch.full((2, V), -4.0, dtype=torch.float16, device=dev)
    peaks[:, 40000] = peaks[:, 123] = peaks[:, 9999] = 6.0
    assert gl.sample_top_k(peaks, 3, 1.0, uniform=torch.tensor([0.1, 0.5], device=dev)).tolist() == [123, 9999]
    small = torch.randn(4, 37, generator=g).half().to(dev)           # fewer columns than threads, top_k larger than the row
    got = gl.sample_top_k(small, 50, 1.0, uniform=torch.zeros(4, device=dev))
    assert torch.equal(got, small.argmax(-1))
    # frequencies: 20 000 draws of one row against its top-8 probabilities
    row = (torch.randn(1, V, generator=g) * 3).half().to(dev)
    vals, idx = torch.topk(row.float(), 8, dim=-1)
    p = torch.softmax(vals, -1)[0].cpu().numpy()
    gen = torch.Generator(device=dev).manual_seed(3)
    draws = gl.sample_top_k(row.expand(20000, V).contiguous(), 8, 1.0, generator=gen).cpu().numpy()
    freq = np.array([(draws == int(i)).mean() for i in idx[0].cpu().numpy()])
    assert abs(freq.sum() - 1) < 1e-9 and np.abs(freq - p).max() < 0.012, (freq, p)
    # the scheduler's sampler takes this path for the decoder's half logits
    from vllmini_amd.scheduler import sample_top_k
    out = sample_top_k(row.expand(64, V).contiguous(), generator=torch.Generator(device=dev).manual_seed(1))
    assert out.dtype == torch.int64 and set(out.tolist()) <= set(torch.topk(row.float(), 50).indices[0].tolist())



@pytest.mark.gpu
@pytest.mark.parametrize("H,D,lens,tile_rows", [(3, 64, [1, 15, 16, 17], 64), (2, 64, [63, 64, 65, 130], 64), (5, 64, [400], 64), (2, 128, [31, 257], 64),
                                                (1, 128, [127, 128, 129, 1], 64), (1, 128, [127, 128, 129, 1], 128), (3, 128, [300, 17], 128)])
def test_prompt_attention_matches_plain_attention_and_leaves_reshape_and_caches_bytes(H, D, lens, tile_rows):
    """One launch over whole prompts against plain attention in float64, and its cache writes against cache_ops.reshape_and_cache: the
    same bytes at the prompts' slots, nothing anywhere else.  A probability is rounded to half (2^-11 of it) and so is the result:
    |error| <= 2^-11 sum p |v| + 2^-11 |out|, and as much again for float32 sums and exponentials."""
    from vllmini_amd import cache_ops, gpt2_layer as gl

    dev, E, T = torch.device("cuda:0"), H * D, sum(lens)
    g = torch.Generator(device=dev).manual_seed(T * H + D)
    wide = torch.randn((T, 3 * E + 8), generator=g, device=dev, dtype=torch.float32).half()
    qkv = wide[:, : 3 * E]                                # (rows of a stride of their own)
    per = [-(-n // 16) for n in lens]
    blocks = torch.randperm(sum(per) + 3, generator=g, device=dev).to(torch.int32)
    table = torch.full((len(lens), max(per) + 1), -1, dtype=torch.int32, device=dev)
    slots, at = [], 0
    for i, n in enumerate(lens):
        table[i, : per[i]] = blocks[at: at + per[i]]
        at += per[i]
        pos = torch.arange(n, device=dev)
        slots.append(table[i, pos // 16].long() * 16 + pos % 16)
    kc = torch.randn((sum(per) + 3, H, D // 8, 16, 8), generator=g, device=dev).half()
    vc = torch.randn((sum(per) + 3, H, D, 16), generator=g, device=dev).half()
    kw, vw = kc.clone(), vc.clone()
    q, k, v = (qkv[:, i * E:(i + 1) * E].view(T, H, D) for i in range(3))
    cache_ops.reshape_and_cache(k, v, kw, vw, torch.cat(slots), "auto", 1.0)
    tiles = torch.tensor([[i, sum(lens[:i]), a, n] for i, n in enumerate(lens) for a in range(0, n, tile_rows)], dtype=torch.int32, device=dev)
    out = gl.prompt_attention(qkv, tiles, tile_rows, kc, vc, table, H, D ** -0.5)
    assert torch.equal(kc, kw) and torch.equal(vc, vw)
    at = 0
    for n in lens:
        a, b, c = (t[at: at + n].double().cpu().transpose(0, 1) for t in (q, k, v))
        s = (a @ b.transpose(1, 2).contiguous()) * D ** -0.5 + torch.full((n, n), float("-inf"), dtype=torch.float64).triu(1)
        w = torch.softmax(s, dim=-1)
        want, size = (w @ c).transpose(0, 1), (w @ c.abs()).transpose(0, 1)
        got = out[at: at + n].view(n, H, D).double().cpu()
        assert bool(((got - want).abs() <= 2 * 2.0 ** -11 * (size + want.abs())).all())
        at += n


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("D,tile_rows,lens,at", [(64, 64, [3, 50, 20], 30), (64, 64, [150], 149), (64, 64, [200], 64), (128, 64, [70], 1), (128, 128, [300], 190)])
def test_prompt_attention_keeps_values_that_are_not_numbers_from_queries_that_do_not_see_them(D, tile_rows, lens, at, bad):
    """A value of inf or NaN at one position (of the prompt that holds it) shows in the rows from that position on and in no other: the
    rows in front of it, which share tiles with it, and the other prompts are what plain attention gives (bound as above)."""
    from vllmini_amd import gpt2_layer as gl

    dev, H, T = torch.device("cuda:0"), 2, sum(lens)
    E, which = H * D, int(np.argmax(lens))
    g = torch.Generator(device=dev).manual_seed(T + D)
    qkv = torch.randn((T, 3 * E), generator=g, device=dev).half()
    first = sum(lens[:which])
    qkv[first + at, 2 * E + D + 7] = bad                  # head 1, column 7
    per = [-(-n // 16) for n in lens]
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32, device=dev)
    for i, n in enumerate(per):
        table[i, :n] = torch.arange(sum(per[:i]), sum(per[:i]) + n, device=dev)
    kc, vc = torch.zeros((sum(per), H, D // 8, 16, 8), device=dev).half(), torch.zeros((sum(per), H, D, 16), device=dev).half()
    tiles = torch.tensor([[i, sum(lens[:i]), a, n] for i, n in enumerate(lens) for a in range(0, n, tile_rows)], dtype=torch.int32, device=dev)
    out = gl.prompt_attention(qkv, tiles, tile_rows, kc, vc, table, H, D ** -0.5).view(T, H, D).double().cpu()
    q, k, v = (qkv[:, i * E:(i + 1) * E].view(T, H, D).double().cpu() for i in range(3))
    hit = torch.zeros(T, H, D, dtype=torch.bool)
    hit[first + at: first + lens[which], 1, 7] = True
    assert bool((~torch.isfinite(out))[hit].all()) and bool(torch.isfinite(out)[~hit].all())
    v[first + at, 1, 7] = 0
    for i, n in enumerate(lens):
        a, b, c = (t[sum(lens[:i]): sum(lens[:i]) + n].transpose(0, 1) for t in (q, k, v))
        w = torch.softmax((a @ b.transpose(1, 2).contiguous()) * D ** -0.5 + torch.full((n, n), float("-inf"), dtype=torch.float64).triu(1), dim=-1)
        rows = slice(sum(lens[:i]), sum(lens[:i]) + n)
        want, size = (w @ c).transpose(0, 1), (w @ c.abs()).transpose(0, 1)
        ok = ((out[rows] - want).abs() <= 2 * 2.0 ** -11 * (size + want.abs())) | hit[rows]
        assert bool(ok.all())


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,T", [(1, 64, 1200), (3, 64, 1217), (1, 128, 1263), (12, 64, 1249), (12, 64, 2900)])
def test_prompts_of_many_rows_take_tiles_and_agree_with_the_entries_one_by_one(H, D, T):
    """vmi_gpt2_prompts_f16 from 1200 rows on (rows and chunks left over; norms and tiles at width 768, the few-row kernels below) against its entries called one by one.
    Both round in the same five places (normed rows, q / k / v, attention, hidden, stream); a sum in another order may fall on the other side,
    2^-10 of a value each, and the two products behind one another pass that on."""
    from vllmini_amd import gpt2_layer as gl

    dev, E = torch.device("cuda:0"), H * D
    g = torch.Generator(device=dev).manual_seed(T + E)
    rnd = lambda *s, std=1.0: (torch.randn(s, generator=g, device=dev) * std).half()      # noqa: E731
    lens = [16] * (T // 16 - 1) + [16 + T % 16]
    w = {"ln_1": (1 + rnd(E, std=0.2), rnd(E, std=0.2)), "ln_2": (1 + rnd(E, std=0.2), rnd(E, std=0.2)), "ln_f": (1 + rnd(E, std=0.2), rnd(E, std=0.2))}
    for name, n, k in (("c_attn", 3 * E, E), ("attn_proj", E, E), ("c_fc", 4 * E, E), ("mlp_proj", E, 4 * E)):
        w[name] = (gl.pack_weight(rnd(n, k, std=k ** -0.5)), rnd(n, std=0.2))
    wte, wpe = rnd(50, E), rnd(40, E)
    ids = torch.randint(0, 50, (T,), generator=g, device=dev)
    pos = torch.cat([torch.arange(n, device=dev) for n in lens])
    last = (torch.tensor(lens, device=dev).cumsum(0) - 1).int()
    per = [-(-n // 16) for n in lens]
    table = torch.full((1, len(lens), max(per)), -1, dtype=torch.int32, device=dev)
    at = 0
    for i, n in enumerate(per):
        table[0, i, :n] = torch.arange(at, at + n, device=dev)
        at += n
    kc, vc = rnd(at, H, D // 8, 16, 8), rnd(at, H, D, 16)
    k2, v2 = kc.clone(), vc.clone()
    rows = 64
    tiles = torch.tensor([[i, sum(lens[:i]), a, n] for i, n in enumerate(lens) for a in range(0, n, rows)], dtype=torch.int32, device=dev)
    flat = []
    for name in ("ln_1", "c_attn", "attn_proj", "ln_2", "c_fc", "mlp_proj"):
        flat += [getattr(w[name][0], "tiles", w[name][0]), w[name][1]]
    got = gl.prompts(flat, (wte, wpe, *w["ln_f"]), ids, pos, last, tiles, rows, table, kc, vc, H, D, 1e-5, D ** -0.5)
    x = gl.embed(ids, pos, wte, wpe)
    qkv = gl.linear(x, *w["c_attn"], ln=(*w["ln_1"], 1e-5))
    a = gl.prompt_attention(qkv, tiles, rows, k2, v2, table[0], H, D ** -0.5)
    x = gl.linear(a, *w["attn_proj"], residual=x)
    h = gl.linear(x, *w["c_fc"], gelu=True, ln=(*w["ln_2"], 1e-5))
    x = gl.linear(h, *w["mlp_proj"], residual=x)
    want = torch.nn.functional.layer_norm(x[last.long()].float(), (E,), w["ln_f"][0].float(), w["ln_f"][1].float(), 1e-5)
    assert float((got.float() - want).abs().max()) <= 10 * 2.0 ** -10 * float(want.abs().max())
    for new, old in ((kc, k2), (vc, v2)):
        assert float((new.float() - old.float()).abs().max()) <= 4 * 2.0 ** -10 * float(old.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,T", [(1, 64, 6099), (3, 64, 2035), (1, 128, 3049), (12, 64, 508), (16, 64, 381), (9, 128, 339), (18, 64, 1201)])
def test_prompts_take_tiles_from_fewer_rows_the_wider_they_are(H, D, T):
    """As above at T E = 390 000 and a little more, at widths from 64 to 1152: tiles past a width of 192 (vmi_gpt2_prompts_in_tiles), the few-row kernels up to there."""
    from vllmini_amd import gpt2_layer as gl

    assert gl.load().vmi_gpt2_prompts_in_tiles(T, H * D) == (H * D > 192)
    assert 390000 <= T * H * D
    test_prompts_of_many_rows_take_tiles_and_agree_with_the_entries_one_by_one(H, D, T)


def test_how_many_tokens_one_native_call_takes_depends_on_the_width():
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    for E, most in ((64, 8192), (768, 4747), (1152, 2109)):
        dims = GPT2Dims(vocab_size=8, n_positions=8, n_embd=E, n_layer=1, n_head=E // 64)
        pool = PagedKVPool(4, dims.n_head, 64, 16, 4, 1, device="cpu", allocate_tensors=False)
        assert GPT2PagedDecoder(dims, random_state_dict(dims, torch.device("cpu")), pool).NATIVE_PROMPT_MAX_TOKENS == most


def test_what_the_prompt_kernels_read_by_address():
    from vllmini_amd import gpt2_layer as gl

    flat = torch.zeros(64, dtype=torch.float16)
    off = -(flat.data_ptr() // 2) % 8
    ok = flat[off: off + 16]
    assert gl.takes_weights([ok, flat[off + 8: off + 24]])
    for bad in (flat[off + 1: off + 17], flat[off + 4: off + 20], flat[off: off + 32: 2], ok.float(), ok.to("meta")):
        assert not gl.takes_weights([ok, bad])


def test_weights_of_other_shapes_or_places_are_not_read_by_address():
    from vllmini_amd import gpt2_layer as gl
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dims = GPT2Dims(vocab_size=50, n_positions=128, n_embd=64, n_layer=2, n_head=1)
    dec = GPT2PagedDecoder(dims, random_state_dict(dims, torch.device("cpu")), PagedKVPool(24, 1, 64, 16, 10, 2, device="cpu", allocate_tensors=False))
    dec.native_layers = True
    assert dec._find_prompt_tensors()
    weights, ends = dec._prompt_tensors
    assert [tuple(t.shape) for t in ends] == [(50, 64), (128, 64), (64,), (64,)]
    assert all(weights[12 + j] is dec.sd["transformer.h.1." + k] for j, k in enumerate(gl.LAYER_WEIGHTS))
    for key, bad in (("ln_f.bias", torch.zeros(63).half()), ("h.1.attn.c_attn.bias", torch.zeros(64).half()), ("h.0.mlp.c_fc.weight", torch.zeros(64, 256).half()),
                     ("wte.weight", torch.zeros(50, 72).half()), ("h.1.ln_2.weight", torch.zeros(65).half()[1:]), ("wpe.weight", torch.zeros(128, 64)), ("h.0.ln_1.bias", None)):
        was = dec.sd["transformer." + key]
        dec.sd["transformer." + key] = bad
        assert not dec._find_prompt_tensors(), key
        dec.sd["transformer." + key] = was
    assert dec._find_prompt_tensors()


def test_prompt_tiles_cover_every_position_once():
    from vllmini_amd import gpt2_layer as gl

    for lens, heads, dim in (([5], 12, 64), ([1, 64, 65, 128, 900], 12, 128), (list(range(1, 120)), 16, 64), (list(range(1, 140)), 16, 128)):
        tiles, rows = gl.prompt_tiles(lens, heads, dim)
        assert rows == (128 if dim == 128 and sum(-(-n // 128) for n in lens) * heads >= 512 else 64)
        seen = sorted((int(i), int(r) + q) for i, r, a, n in tiles for q in range(a, min(n, a + rows)))
        assert seen == [(i, sum(lens[:i]) + q) for i, n in enumerate(lens) for q in range(n)]
        assert all(int(n) == lens[i] for i, _, _, n in tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("E", [8, 64, 520, 768, 1032, 2048, 4096])
@pytest.mark.parametrize("M", [1, 4, 7])
def test_add_norm_is_the_add_and_the_layer_norm(M, E):
    """Against torch's add (the same rounding: equal) and layer_norm in float32 on the rounded stream: one rounding of the result (2^-11
    of it), and as much again for the float32 steps before it."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(E + M)
    x, y = ((torch.randn((M, E), generator=g, device=dev) * 3 + 1).half() for _ in range(2))
    ln = (torch.randn(E, generator=g, device=dev).half(), torch.randn(E, generator=g, device=dev).half(), 1e-5)

    def close(got, rows):
        want = F.layer_norm(rows.double(), (E,), ln[0].double(), ln[1].double(), ln[2])
        size = want.abs() + ln[0].double().abs() * 4 + ln[1].double().abs()      # (terms that may cancel)
        assert bool(((got.double() - want).abs() <= 2.0 ** -10 * size).all())

    z = x.clone()
    close(gl.add_norm(z, ln, y), x + y)
    assert torch.equal(z, x + y)
    rows = torch.tensor([M - 1, 0], dtype=torch.int32, device=dev)
    close(gl.add_norm(z, ln, rows=rows), z[rows.long()])
    assert torch.equal(z, x + y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (16, 48, 224), (17, 144, 288), (3, 2304, 768), (47, 768, 1056), (33, 320, 2048), (112, 768, 3072), (5, 80, 4096), (1, 832, 3328), (17, 48, 3616), (64, 96, 4128), (352, 640, 2560)])
def test_few_rows_split_k_over_the_waves(M, N, K):
    """rows_kernel where its waves have unequal parts of K, or none; row tiles that are not full; more of them than XCDs: against the module chain,
    for every epilogue it has, both weight layouts to the same bits."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    x, w, b, res = (rnd(M, K + 8) * 1.5 + 0.3).half()[:, :K], (rnd(N, K) * 0.6 / K ** 0.5).half(), (rnd(N) * 0.1).half(), rnd(M, N).half()
    ln = ((1 + 0.2 * rnd(K)).half(), (0.1 * rnd(K)).half(), 1e-5)
    for kw in ({"ln": ln}, {"ln": ln, "gelu": True}, {"residual": res}):
        if kw.get("ln") and K > 2048:
            continue
        got = gl.linear(x, w, b, **kw)
        _close(got, _chain(x, w, b, kw.get("ln"), kw.get("gelu", False), kw.get("residual")), (M, N, K, sorted(kw)))
        assert torch.equal(gl.linear(x, gl.pack_weight(w), b, **kw), got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 2320, 768), (70, 2320, 768), (90, 2320, 768), (123, 2320, 768), (40, 3088, 1152), (50, 2064, 2048), (200, 784, 768), (20, 48, 4608),
                                   (9, 256, 1504)])
def test_few_rows_of_several_slabs_a_workgroup(M, N, K):
    """norm_rows_kernel with 2, 3, 4 and 6 slabs a workgroup and rows_kernel with two, the last workgroup's not all there; K that its waves do not divide evenly."""
    test_few_rows_split_k_over_the_waves(M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(1, 768), (17, 768), (33, 96), (5, 1056), (12, 2048), (200, 768), (700, 768), (640, 1024), (900, 224)])
def test_the_norm_in_front_holds_rows_whose_mean_is_far_from_zero(M, K):
    """Rows of mean 300 and deviation 0.5 (a half holds these to 0.25) through both kernels' norms: identity weights, so a result is one normed
    value.  The sum and the squares are float32 sums of a few dozen terms a lane: the mean is off by at most 8 roundings (2^-24 of 300) and so is
    the deviation, relatively; the result is rounded once to half (2^-11 of it)."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + K)
    x = (torch.randn((M, K), generator=g, device=dev) * 0.5 + 300).half()
    x[0] = (x[0].float() - 600).half()
    gamma, beta = (1 + 0.2 * torch.randn(K, generator=g, device=dev)).half(), (0.1 * torch.randn(K, generator=g, device=dev)).half()
    got = gl.linear(x, gl.pack_weight(torch.eye(K, device=dev).half()), torch.zeros(K, device=dev).half(), ln=(gamma, beta, 1e-5)).double()
    d = x.double()
    dev_, off = d.std(-1, unbiased=False, keepdim=True), d.mean(-1, keepdim=True).abs()
    t = (d - d.mean(-1, keepdim=True)) / torch.sqrt(dev_ ** 2 + 1e-5) * gamma.double()
    want = t + beta.double()
    bound = 2.0 ** -11 * want.abs() + 8 * 2.0 ** -24 * (off / dev_ * gamma.double().abs() + t.abs()) + 2.0 ** -24
    assert bool(((got - want).abs() <= 1.01 * bound).all()), float(((got - want).abs() / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (17, 80, 128), (300, 3088, 320), (1063, 5408, 192), (770, 5392, 128), (1442, 6160, 128), (641, 5920, 576), (323, 5424, 832),
                                   (481, 5392, 64), (130, 5472, 768), (129, 5552, 1984), (2100, 768, 3072)])
def test_products_of_many_rows_in_tiles(M, N, K):
    """tiles_kernel: rows and columns left over, one chunk of K, two, an odd number of them and many; every epilogue.  (Which tile runs is the rule's: test_each_tile_by_itself goes
    through their list.)"""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    x, w, b, res = (rnd(M, K) * 1.5 + 0.3).half(), (rnd(N, K) * 0.6 / K ** 0.5).half(), (rnd(N) * 0.1).half(), rnd(M, N).half()
    for bias, kw in ((None, {}), (b, {"gelu": True}), (b, {"residual": res})):
        _close(gl.linear_tiles(x, gl.pack_weight(w), bias, **kw), _chain(x, w, bias, None, kw.get("gelu", False), kw.get("residual")), (M, N, K, sorted(kw)))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 272, 320), (300, 3088, 320), (770, 768, 3072), (2100, 768, 768), (2029, 6544, 768)])
def test_residuals_that_begin_anywhere(M, N, K):
    """tiles_kernel: residuals aligned to eight bytes, not to sixteen, give what aligned ones do, also where they are added in place of themselves."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    x, w, b, flat = rnd(M, K).half(), gl.pack_weight((rnd(N, K) / K ** 0.5).half()), rnd(N).half(), rnd(M * N + 8).half()
    want = gl.linear_tiles(x, w, b, residual=flat[4:-4].clone().view(M, N))
    assert torch.equal(gl.linear_tiles(x, w, b, residual=flat[4:-4].view(M, N)), want)
    before = flat.clone()
    for at in (0, 4):
        flat.copy_(before)
        y, res = flat[at: at + M * N].view(M, N), flat[at: at + M * N].clone().view(M, N)
        gl._check(gl.load().vmi_gpt2_linear_tiles_f16(x.data_ptr(), w.tiles.data_ptr(), b.data_ptr(), y.data_ptr(), y.data_ptr(), M, N, K, gl.EPI_BIAS_RESIDUAL, 0,
                                                      torch.cuda.current_stream().cuda_stream))
        assert torch.equal(y, gl.linear_tiles(x, w, b, residual=res)) and torch.equal(flat[:at], before[:at]) and torch.equal(flat[at + M * N:], before[at + M * N:])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2029, 6544, 768), (2024, 6576, 704), (2507, 7216, 256), (2517, 7216, 192), (1859, 3232, 512), (866, 6624, 832), (963, 5920, 1152),
                                   (1375, 4368, 448), (2026, 4400, 128), (2068, 4368, 64), (321, 7536, 128), (354, 6800, 64), (269, 6544, 512), (263, 6688, 832),
                                   (257, 6544, 1152), (259, 6576, 448), (769, 7600, 128), (778, 7568, 64), (391, 6560, 1536), (386, 6560, 1216), (195, 7088, 128),
                                   (193, 7056, 64), (199, 7008, 256), (132, 6624, 576), (130, 6736, 640), (194, 7136, 192), (70, 5456, 512), (67, 5456, 576), (66, 5968, 640),
                                   (68, 5536, 448), (1, 32, 384), (8, 16, 64), (5, 32, 512), (1, 112, 576), (1, 160, 1152), (16, 16, 448), (1, 160, 64), (40, 272, 320)])
def test_every_tile_with_every_number_of_chunks_left(M, N, K):
    """tiles_kernel, rows, columns and chunks of K left over, fewer chunks than are in flight among them.  A chunk that is none adds nothing where the last one holds an infinity: the row that
    has one is infinite or, where the weight is zero, NaN, and no other row is touched."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    x, w, b, res = (rnd(M, K) * 1.5 + 0.3).half(), (rnd(N, K) * 0.6 / K ** 0.5).half(), (rnd(N) * 0.1).half(), rnd(M, N).half()
    w[N // 3, -1] = 0
    packed = gl.pack_weight(w)
    for bias, kw in ((None, {}), (b, {"gelu": True}), (b, {"residual": res})):
        _close(gl.linear_tiles(x, packed, bias, **kw), _chain(x, w, bias, None, kw.get("gelu", False), kw.get("residual")), (M, N, K, sorted(kw)))
    before, row = gl.linear_tiles(x, packed), M // 2
    x[row, -1] = float("inf")
    after = gl.linear_tiles(x, packed)
    rest = torch.arange(M, device=dev) != row
    assert torch.equal(after[rest], before[rest])
    want = torch.where(w[:, -1] == 0, float("nan"), torch.sign(w[:, -1]) * float("inf")).half()
    assert bool(((after[row] == want) | (after[row].isnan() & want.isnan())).all()) and bool(after[row, N // 3].isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("tile,left", tile_cases.places())
def test_each_tile_by_itself(tile, left):
    """As above, the tile of the list with so many chunks of K left behind two rounds of its walk or more: the size is looked up, so the tile runs whatever the costs it is picked by."""
    M, N, K, _ = tile_cases.size_for(tile, left)
    test_every_tile_with_every_number_of_chunks_left(M, N, K)


@pytest.mark.gpu
def test_gelu_of_every_half():
    """The exact GELU of all 65536 halves, as biases under rows of zeros: within half a unit in the last place of v Phi(v) in 64 bits, up to the float's own error
    (2^-11 of a unit, some twenty roundings); infinity stays, minus infinity
    (times a zero) and NaN are NaN, as 0.5 v (1 + erf) has them."""
    from vllmini_amd import gpt2_layer as gl

    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    x = torch.zeros((1, 64), dtype=torch.float16, device="cuda:0")
    w = gl.pack_weight(torch.zeros((4096, 64), dtype=torch.float16, device="cuda:0"))
    got = torch.cat([gl.linear(x, w, part.cuda(), gelu=True)[0] for part in v.split(4096)]).cpu()
    fin, d = torch.isfinite(v), v.double()
    want = d * torch.special.ndtr(d)
    unit = 2.0 ** (want.abs().clamp_min(2.0 ** -14).log2().floor() - 10)
    assert bool((((got.double() - want) / unit).abs()[fin] <= 0.5 + 2.0 ** -11).all())
    assert bool((got[v == float("inf")] == float("inf")).all()) and bool(got[~fin & (v != float("inf"))].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,T", [(12, 64, 391), (14, 64, 179), (18, 64, 139), (6, 128, 400), (8, 64, 587)])
def test_prompts_take_tiles_from_fewer_rows_still_past_a_width_of_768(H, D, T):
    """As test_prompts_of_many_rows_..., at T E = 300 000 up to a width of 768 and 160 000 beyond."""
    from vllmini_amd import gpt2_layer as gl

    assert gl.load().vmi_gpt2_prompts_in_tiles(T, H * D)
    test_prompts_of_many_rows_take_tiles_and_agree_with_the_entries_one_by_one(H, D, T)


LINES = [(128, 4800), (192, 3200), (256, 1760), (320, 912), (384, 768), (448, 656), (512, 576), (576, 448), (640, 400), (704, 368), (768, 336), (832, 144), (896, 144), (960, 128),
         (1024, 128), (1088, 112), (1152, 112)]      # width, the most tokens that the few-row kernels are measured ahead or level for


def test_prompts_take_tiles_where_the_few_row_kernels_fall_behind():
    """The rule against both sides as measured: the line, and points of either side that a line over T E alone has got wrong."""
    from vllmini_amd import gpt2_layer as gl

    tiles = gl.load().vmi_gpt2_prompts_in_tiles
    for E, T in LINES:
        assert not tiles(T, E) and tiles(T + 16, E), (E, T)
    for T, E in ((1600, 256), (2400, 192), (4000, 128), (120, 960), (124, 1024), (100, 1152)):
        assert not tiles(T, E), (T, E)
    for T, E in ((1100, 320), (850, 384), (500, 576), (450, 640), (160, 832), (130, 960), (130, 1024), (128, 1088)):
        assert tiles(T, E), (T, E)
    assert not tiles(8192, 64) and not tiles(4000, 800) and not tiles(4000, 1216) and not tiles(0, 768)


@pytest.mark.gpu
@pytest.mark.parametrize("E,T", [(E, T + d) for E, T in LINES if E in (192, 256, 512, 640, 768, 896, 1024, 1152) for d in (0, 1)])
def test_prompts_on_both_sides_of_the_line_to_tiles(E, T):
    """As test_prompts_of_many_rows_..., where the kernels change."""
    test_prompts_of_many_rows_take_tiles_and_agree_with_the_entries_one_by_one(E // 64, 64, T)


@pytest.mark.gpu
@pytest.mark.parametrize("head,rows,ld,used,n", [(0, 0, 0, 0, 1), (16, 3, 5, 5, 0), (4080, 1, 64, 1, 0), (4096, 384, 64, 13, 32), (48, 7, 9, 0, 300), (1 << 20, 1000, 33, 32, 5)])
def test_a_steps_inputs_go_where_its_launches_read_them(head, rows, ld, used, n):
    """step_inputs: the head, the columns that count and the ids arrive, everything else stays; the pinned memory may be written again after wait()."""
    from vllmini_amd import gpt2_layer as gl
    from vllmini_amd.staging import PinnedBuffer

    dev = torch.device("cuda:0")
    buf, size = PinnedBuffer(head + rows * ld * 4 + 16), head + rows * ld * 4 + 16
    ids = torch.arange(100, 100 + n, device=dev)
    for turn in (1, 2):
        buf.wait()
        buf.tensor.copy_(torch.randint(0, 255, (size,), dtype=torch.uint8, generator=torch.Generator().manual_seed(turn)))
        to, out = torch.full((size,), 255, dtype=torch.uint8, device=dev), torch.full((n + 2,), -1, dtype=torch.int64, device=dev)
        gl.step_inputs(buf, to, head, rows, ld, used, ids if n else None, out)
        want = torch.full((size,), 255, dtype=torch.uint8)
        want[:head] = buf.tensor[:head]
        want[head:head + rows * ld * 4].view(rows, ld * 4)[:, : used * 4] = buf.tensor[head:head + rows * ld * 4].view(rows, ld * 4)[:, : used * 4]
        assert torch.equal(to.cpu(), want) and out.tolist() == [*range(100, 100 + n), -1, -1]
    with pytest.raises(RuntimeError):
        gl.step_inputs(buf, to, head + 32, rows, ld, used, None, out)
    with pytest.raises(RuntimeError):
        gl.step_inputs(buf, to, head, rows, ld, used, ids.int() if n else out.int(), out)


@pytest.mark.gpu
@pytest.mark.parametrize("M,V,E", [(1, 50257, 768), (16, 50257, 768), (15, 33000, 32), (16, 1003, 1152), (5, 15, 416), (16, 4096, 384), (3, 32784, 1536), (2, 100001, 64), (9, 70001, 800)])
@pytest.mark.parametrize("norm", [True, False])
def test_logits_of_few_rows(M, V, E, norm):
    """head(): fewer slabs than waves and several a wave, the last one cut, one to three chunks of K, rows with a stride, an odd number of columns."""
    from vllmini_amd import gpt2_layer as gl

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + V + E)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    x, w = (rnd(M, E + 8) * 2 + 0.5).half()[:, :E], (rnd(V, E) / E ** 0.5).half()
    ln = ((1 + 0.2 * rnd(E)).half(), (0.1 * rnd(E)).half(), 1e-5) if norm else None
    assert gl.head_fits(M, E)
    got = gl.head(x, gl.pack_head(w), ln)
    h = torch.nn.functional.layer_norm(x.float(), (E,), ln[0].float(), ln[1].float(), 1e-5).half() if norm else x
    want = h.double() @ w.double().T
    # half a unit in the last place of the result, the float32 sum, and (norm) rows that round the other way: one in thousands of them, 2^-10 of its product
    bound = 2.0 ** -11 * want.abs() + 2.0 ** -20 * E ** 0.5 + (2.0 ** -10 * 4 / E ** 0.5 if norm else 0) + 2.0 ** -24
    assert got.shape == (M, V) and bool(((got.double() - want).abs() <= 1.01 * bound).all()), float(((got.double() - want).abs() / bound).max())
    assert gl.HEAD_MAX_ROWS == 16 and not gl.head_fits(17, E) and not gl.head_fits(M, 1568)
    with pytest.raises(RuntimeError):
        gl.head(x.float(), gl.pack_head(w), ln)


@pytest.mark.gpu
def test_the_vocabulary_is_kept_once_more_unless_the_caller_declines():
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dims, dev = GPT2Dims(vocab_size=203, n_layer=2), torch.device("cuda:0")
    sd, got = random_state_dict(dims, dev), []
    for native_head in (None, True, False):
        pool = PagedKVPool(64, dims.n_head, dims.head_size, 16, 8, dims.n_layer, device=dev, max_seqs=2)
        d = GPT2PagedDecoder(dims, sd, pool, native_head=native_head)
        assert (d._head is None) == (native_head is False)
        d.prefill_batch([0, 1], [list(range(20)), list(range(5, 12))])
        got.append(d.decode([0, 1], [1, 2]))
    assert torch.equal(got[0], got[1])
    _close(got[2], got[0], "torch's lm_head beside gpt2_layer.head")
    odd = {**sd, "lm_head.weight": sd["lm_head.weight"].t().contiguous().t()}
    with pytest.raises(RuntimeError, match="native_head"):
        GPT2PagedDecoder(dims, odd, pool, native_head=True)
    assert GPT2PagedDecoder(dims, odd, pool)._head is None


@pytest.mark.gpu
def test_logits_of_a_vocabulary_of_more_than_sixteen_million():
    from vllmini_amd import gpt2_layer as gl

    dev, V = torch.device("cuda:0"), (1 << 24) + 37
    g = torch.Generator(device=dev).manual_seed(7)
    x, w = torch.randn((2, 32), generator=g, device=dev).half(), torch.randn((V, 32), generator=g, device=dev, dtype=torch.float16)
    got, want = gl.head(x, gl.pack_head(w)), (w.float() @ x.float().T).T
    assert got.shape == (2, V) and bool(((got.float() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-4).all())


@pytest.mark.gpu
@pytest.mark.parametrize("B,ctx,switch", [(32, 100, False), (16, 200, True), (1, 800, True), (4, 300, False), (12, 250, True)])
def test_steps_read_their_pages_past_the_caches_with_the_same_results(B, ctx, switch, monkeypatch):
    """_past_caches, in a cache that holds the weights and nothing else: where a step takes another variant than the operators would (where two blocks a wave and few heads are not left to them, nor pages non-temporal as they
    are), it is the same split of a head over waves without a temporal load, and logits and caches agree (to the bit where a wave takes its blocks one by one in both)."""
    from vllmini_amd import ops
    from vllmini_amd.gpt2_decode import GPT2Dims, GPT2PagedDecoder, random_state_dict
    from vllmini_amd.kv_pool import PagedKVPool

    dims, dev = GPT2Dims(vocab_size=200, n_layer=2), torch.device("cuda:0")
    sd = random_state_dict(dims, dev)
    names, got = ops.variant_names(), []
    for past in (True, False):
        if not past:
            monkeypatch.setattr(GPT2PagedDecoder, "_past_caches", lambda self, variant, B: variant)
        pool = PagedKVPool(B * dims.n_layer * 64 + 8, dims.n_head, dims.head_size, 16, 64, dims.n_layer, device=dev, max_seqs=B, multi_block_prefill=True)
        d = GPT2PagedDecoder(dims, sd, pool)
        monkeypatch.setattr(d, "INFINITY_CACHE", d._step_weights)
        d.prefill_batch(list(range(B)), [[(7 * s + j) % 200 for j in range(ctx - s % 5)] for s in range(B)])
        out = [d.decode(list(range(B)), torch.full((B,), 3 + i, device=dev), use_graph=True).clone() for i in range(3)]
        got.append((names[d._static["variant"] - 1], out, pool.key_cache.clone(), pool.value_cache.clone()))
    (a, x, ka, va), (b, y, kb, vb) = got
    assert (a != b) == switch, (a, b)
    if a != b:
        assert a.endswith("_u1_nt1") and b.endswith("_nt0") and a.rsplit("_u", 1)[0] == b.rsplit("_u", 1)[0]
    if a.replace("nt1", "nt0") == b.replace("nt1", "nt0"):
        assert all(torch.equal(p, q) for p, q in zip(x, y)) and torch.equal(ka, kb) and torch.equal(va, vb)
    for p, q in zip(x, y):
        assert float((p.float() - q.float()).norm() / q.float().norm()) <= 2e-3
