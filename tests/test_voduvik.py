"""The Voduvik design on the CPU: the plain restatement against itself, configuration and checkpoint reading, the pool's portions
and state slots, portions of prompts in the scheduler, and the C-ABI of libvmi_hybrid.so."""
from __future__ import annotations

import ctypes
import os
import re
import subprocess
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import voduvik as plain
from tests import voduvik_cases as cases

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---- the oracle's own mechanisms, checked on their defining properties ---------------------------------------------------------
def test_plain_rotation_turns_pairs_and_keeps_relative_angles():
    g = torch.Generator().manual_seed(0)
    q, k = (torch.randn(24, generator=g, dtype=torch.float64) for _ in range(2))
    dot = lambda p, j: float(plain.rotate(q, p, 700.0, 16) @ plain.rotate(k, j, 700.0, 16))      # noqa: E731
    assert dot(9, 4) == pytest.approx(dot(105, 100)) and dot(9, 4) != pytest.approx(dot(9, 5))
    assert torch.equal(plain.rotate(q, 31, 700.0, 16)[16:], q[16:]) and torch.equal(plain.rotate(q, 0, 700.0, 16), q)


def test_plain_convolution_and_recurrence_against_closed_forms():
    g = torch.Generator().manual_seed(1)
    x, w, b = torch.randn(9, 3, generator=g), torch.randn(3, 4, generator=g), torch.randn(3, generator=g)
    ref = torch.nn.functional.conv1d(torch.nn.functional.pad(x.t()[None], (3, 0)), w[:, None], b, groups=3)[0].t()
    assert torch.allclose(plain.causal_conv(x, w, b), ref, atol=1e-5)
    u, r, i = torch.ones(5, 2, dtype=torch.float64), torch.full((5, 2), 0.5, dtype=torch.float64), torch.ones(5, 2, dtype=torch.float64)
    lam = torch.tensor([-4.0, 1.0], dtype=torch.float64)
    a = torch.exp(-4 * torch.nn.functional.softplus(lam))
    S, last = plain.rglru_scan(u, r, i, lam)
    want = torch.stack([torch.sqrt(1 - a * a) * (1 - a ** n) / (1 - a) for n in range(1, 6)])
    assert torch.allclose(S, want) and torch.equal(last, S[-1])
    half, mid = plain.rglru_scan(u[:2], r[:2], i[:2], lam)
    rest, _ = plain.rglru_scan(u[2:], r[2:], i[2:], lam, state=mid)
    assert torch.allclose(torch.cat([half, rest]), S)


@pytest.mark.parametrize("name", sorted(cases.CONFIGS))
def test_plain_forward_is_causal_and_its_faults_show(name):
    c = cases.CONFIGS[name]
    w, toks = cases.tensors(c), cases.tokens(c, 24)
    full, streams = plain.forward(c, w, toks)
    assert streams.shape[0] == len(plain.layer_runs(c)) and torch.isfinite(full).all()
    part, _ = plain.forward(c, w, toks[:15])
    assert torch.allclose(part, full[:15], atol=1e-9)
    other, _ = plain.forward(c, w, [toks[0] ^ 1] + toks[1:])       # the first token still matters at the end: a lost state or key
    assert float((other[-1] - full[-1]).abs().max()) > 1e-3        # would show
    for planted in ("lam", "dkv.norm", "conv.b", "norm1", "mlp.gate", "loop.in"):       # so would any weight that is left out
        hit = [k for k in w if k.endswith(planted)]
        if hit:
            bad = dict(w)
            bad[hit[0]] = bad[hit[0]] * 0.5
            assert float((plain.forward(c, bad, toks)[0] - full).abs().max()) > 1e-2, planted


# ---- configuration, checkpoints, registry ----------------------------------------------------------------------------------------
@pytest.mark.parametrize("name", sorted(cases.CONFIGS))
def test_config_reads_every_size_and_orders_the_runs(name):
    from vllmini_amd.voduvik import VoduvikConfig

    c = cases.CONFIGS[name]
    cfg = VoduvikConfig.from_json(c)
    assert cfg.order() == plain.layer_runs(c)
    assert cfg.tensor_shapes() == cases.shapes(c)


def test_config_refuses_what_the_design_does_not_have():
    from vllmini_amd.voduvik import VoduvikConfig

    c = cases.config([{"type": "sliding", "mixer": {}, "mlp": None}])
    with pytest.raises(ValueError, match="unknown mixer"):
        VoduvikConfig.from_json(c)
    with pytest.raises(ValueError, match="feed-forward"):
        VoduvikConfig.from_json(cases.config([cases.rglru(32, 1, mlp={"kind": "experts", "ff": 8, "limit": 1.0})]))
    with pytest.raises(ValueError, match="loop"):
        VoduvikConfig.from_json(cases.config([cases.rglru(32, 1)], loop=(0, 2, 2)))


def test_safetensors_reader_round_trip_and_bounds(tmp_path):
    from vllmini_amd.weights import load_checkpoint, read_safetensors

    named = {"a": torch.randn(3, 5).to(torch.bfloat16), "b.c": torch.arange(7, dtype=torch.int32), "s": torch.randn(2, 1, 2)}
    cases.write_safetensors(tmp_path / "x.safetensors", named)
    got = load_checkpoint(str(tmp_path))
    assert set(got) == set(named)
    for k in named:
        assert got[k].dtype == named[k].dtype and torch.equal(got[k], named[k])
    raw = (tmp_path / "x.safetensors").read_bytes()
    (tmp_path / "cut.safetensors").write_bytes(raw[:-4])
    with pytest.raises(ValueError, match="extent"):
        read_safetensors(str(tmp_path / "cut.safetensors"))
    (tmp_path / "bad.safetensors").write_bytes((1 << 40).to_bytes(8, "little") + raw[8:])
    with pytest.raises(ValueError, match="header"):
        read_safetensors(str(tmp_path / "bad.safetensors"))


def test_registry_names_the_architecture_and_refuses_unknown_ones(tmp_path):
    from vllmini_amd import registry

    assert {"Voduvik", "GPT2LMHeadModel"} <= set(registry.architectures())
    assert registry.architecture_of({"architecture": "Voduvik"}) == "Voduvik"
    assert registry.architecture_of({"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2"}) == "GPT2LMHeadModel"
    with pytest.raises(ValueError, match="no known architecture"):
        registry.architecture_of({"architecture": "Somethingelse"})
    folder = cases.write_model(tmp_path / "m", cases.CONFIGS["mixed"], cases.tensors(cases.CONFIGS["mixed"]))
    with pytest.raises(registry.UnsupportedDtype):
        registry.load_decoder(folder, dtype="float16", max_tokens=64, max_seqs=1, device="cpu")


def test_builder_refuses_missing_and_misshapen_tensors():
    from vllmini_amd.voduvik import VoduvikConfig, build_model

    c = cases.CONFIGS["no_loop"]
    w = cases.tensors(c)
    cfg = VoduvikConfig.from_json(c)
    with pytest.raises(KeyError, match="l1.mix.lam"):
        build_model(cfg, {k: v for k, v in w.items() if k != "l1.mix.lam"}, torch.float32, "cpu")
    with pytest.raises(ValueError, match="head"):
        build_model(cfg, {**w, "head": w["head"][:-1]}, torch.float32, "cpu")
    m = build_model(cfg, w, torch.float32, "cpu")
    assert len(m.runs) == 3 and m.head.w.N % 32 == 0


def test_padded_layouts_keep_the_products():
    """Tiles and padding only rearrange: the padded input projection of a latent-attention layer, read back, is the checkpoint's."""
    from vllmini_amd.voduvik import VoduvikConfig, build_model

    c = cases.CONFIGS["mixed"]
    w = cases.tensors(c)
    a = build_model(VoduvikConfig.from_json(c), w, torch.float32, "cpu").runs[1].mixer
    d = a.w_in.dense
    H, dim, rot, rank, E = 3, 20, 12, 40, c["width"]
    q = d[: H * (a.dim + a.rot), :E].view(H, a.dim + a.rot, E)
    assert torch.equal(q[:, :dim], w["l1.mix.q"].float().view(H, dim + rot, E)[:, :dim])
    assert torch.equal(q[:, a.dim:a.dim + rot], w["l1.mix.q"].float().view(H, dim + rot, E)[:, dim:])
    assert not q[:, dim:a.dim].any() and not q[:, a.dim + rot:].any() and not d[:, E:].any()
    at = H * (a.dim + a.rot)
    assert torch.equal(d[at:at + rank, :E], w["l1.mix.dkv"].float()[:rank])
    assert torch.equal(d[at + a.rank:at + a.rank + rot, :E], w["l1.mix.dkv"].float()[rank:])
    assert torch.equal(d[a.gate_at:a.gate_at + H, :E], w["l1.mix.g"].float())
    t = a.w_in.tiles[0]                                        # [N / 16][K / 32][kc][r][e]
    back = t.permute(0, 3, 1, 2, 4).reshape(a.w_in.N, a.w_in.K)
    assert torch.equal(back, d)


# ---- the pool ---------------------------------------------------------------------------------------------------------------------
def _pool(blocks=6, page=4, slots=2, per_seq=6):
    from vllmini_amd.kv_pool import PagedKVPool

    return PagedKVPool(blocks, 1, 8, page, per_seq, 1, device="cpu", page_rows=[8, 16], page_dtype=torch.float32,
                       state=[((5,), torch.float32)], state_slots=slots)


def test_pool_append_hands_out_positions_slots_and_parities():
    p = _pool()
    p.open(7)
    a = p.append([7], [3])
    assert a["ctx"].tolist() == [0] and a["pos"].tolist() == [0, 1, 2] and a["slots"][0].tolist() == [0, 1, 2] and a["parity"].tolist() == [0]
    p.open(9)
    b = p.append([9, 7], [5, 2])                             # 9 takes two blocks, 7 crosses into a second one
    assert b["ctx"].tolist() == [0, 3] and b["entry"].tolist() == [0] * 5 + [1] * 2 and b["pos"].tolist() == [0, 1, 2, 3, 4, 3, 4]
    assert b["slots"][0].tolist() == [4, 5, 6, 7, 8, 3, 12] and b["parity"].tolist() == [0, 1]
    assert b["state_slot"].tolist() == [1, 0] and p.seq_len(7) == 5 and p.free_state_slots == 0
    with pytest.raises(RuntimeError, match="free blocks"):
        p.open(11)
    assert 11 not in p.allocated_blocks
    before = (list(p.free_blocks), p._tables.copy(), p._seq_len.copy(), p._parity.copy())
    with pytest.raises(RuntimeError, match="No free blocks"):      # 9: 5 -> 17 tokens needs 3 blocks, 2 are left
        p.append([7, 9], [1, 12])
    assert list(p.free_blocks) == before[0] and all(np.array_equal(x, y) for x, y in zip(before[1:], (p._tables, p._seq_len, p._parity)))
    with pytest.raises(RuntimeError, match="blocks per layer"):
        p.append([7], [40])
    p.free(9)
    p.open(11)                                                 # pages and slots come round again
    c = p.append([11], [9])
    assert c["state_slot"].tolist() == [1] and set(p.allocated_blocks[11]) & {1, 2}
    with pytest.raises(ValueError):
        p.append([7, 7], [1, 1])
    assert p.row_pages[0].shape == (6, 4, 8) and p.row_pages[1].shape == (6, 4, 16) and p.state[0].shape == (2, 5)


def test_pool_append_agrees_with_the_decode_step_of_the_key_value_layout():
    from vllmini_amd.kv_pool import PagedKVPool

    a, b = (PagedKVPool(40, 2, 8, 4, 8, 3, device="cpu", allocate_tensors=False) for _ in range(2))
    a.allocate_for_prefill(0, 6)
    b.allocate_for_prefill(0, 6)
    for _ in range(7):
        ta, sa, la = a.decode_step_batch([0])
        r = b.append([0], [1])
        assert np.array_equal(ta, r["tables"]) and np.array_equal(sa, r["slots"]) and la.tolist() == (r["ctx"] + 1).tolist()


# ---- portions of prompts in the scheduler --------------------------------------------------------------------------------------------
class _Stand:
    """A decoder whose next token is a hash of the sequence: whatever the schedule, a request's tokens must come out the same."""

    def __init__(self, pool, vocab=50):
        self.pool, self.vocab, self.seen, self.steps = pool, vocab, {}, []

    def _logits(self, seq):
        out = torch.zeros(self.vocab)
        out[(sum((i + 1) * t for i, t in enumerate(seq)) * 31 + len(seq)) % self.vocab] = 1.0
        return out

    def step(self, ids, tokens, want):
        a = self.pool.append(ids, [len(t) for t in tokens])
        self.steps.append([len(t) for t in tokens])
        rows = []
        for s, t, w, ctx in zip(ids, tokens, want, a["ctx"]):
            seq = ([] if ctx == 0 else self.seen[s]) + [int(x) for x in t]
            assert len(seq) == ctx + len(t)
            self.seen[s] = seq
            rows += [self._logits(seq[: ctx + k + 1]) for k in w]
        return torch.stack(rows) if rows else None

    def prefill_batch(self, ids, prompts):
        for i in ids:
            self.pool.open(i)
        return self.step(ids, prompts, [[len(p) - 1] for p in prompts])

    paged_prefill = True

    def prefill(self, i, p):
        return self.prefill_batch([i], [p])[0]

    def decode(self, ids, tokens):
        return self.step(ids, [[int(t)] for t in tokens], [[0]] * len(ids))


def _generate(prompts, new, blocks, chunk, max_batch=3, slots=3):
    from vllmini_amd.kv_pool import PagedKVPool
    from vllmini_amd.scheduler import BatchScheduler, sample_greedy

    pool = PagedKVPool(blocks, 1, 8, 4, 40, 1, device="cpu", page_rows=[8], page_dtype=torch.float32, state_slots=slots,
                       allocate_tensors=False, host_blocks=100)
    dec = _Stand(pool)
    sch = BatchScheduler(dec, max_length=120, eos_token_id=-1, max_batch=max_batch, sampler=sample_greedy, prefill_chunk=chunk)
    ids = [sch.submit(p, max_new_tokens=n) for p, n in zip(prompts, new)]
    sch.run(max_steps=2000)
    assert not sch.pending() and len(pool.free_blocks) == blocks and pool.free_state_slots == slots
    return [sch.sequences[i] for i in ids], sch, dec


@pytest.mark.parametrize("chunk", [2, 5, 16])
@pytest.mark.parametrize("blocks", [60, 14])
def test_scheduler_runs_portions_beside_single_tokens(chunk, blocks):
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, 50, n).tolist() for n in (21, 1, 9, 30, 4, 17)]
    new = [6, 9, 3, 5, 12, 7]
    want, _, _ = _generate(prompts, new, 200, 0, max_batch=6, slots=6)
    got, sch, dec = _generate(prompts, new, blocks, chunk)
    assert got == want and not sch.rejected and not sch.evicted
    assert any(1 in s and max(s) > 1 for s in dec.steps), "no step mixed a portion with single tokens"
    assert max(sum(n for n in s if n > 1) for s in dec.steps) <= chunk


def test_scheduler_rejects_a_prompt_no_pool_can_hold_and_aborts_unfinished_ones():
    got, sch, _ = _generate([[1] * 90, [2, 3, 4]], [2, 2], 10, 8)
    assert list(sch.rejected) == [0] and len(got[1]) == 5
    from vllmini_amd.kv_pool import PagedKVPool
    from vllmini_amd.scheduler import BatchScheduler, sample_greedy

    pool = PagedKVPool(30, 1, 8, 4, 40, 1, device="cpu", page_rows=[8], state_slots=2, allocate_tensors=False)
    sch = BatchScheduler(_Stand(pool), max_length=100, eos_token_id=-1, sampler=sample_greedy, prefill_chunk=4)
    i = sch.submit([5] * 20, max_new_tokens=3)
    sch.step()
    assert sch.prefilling == {i: 4} and sch.abort(i) and len(pool.free_blocks) == 30 and not sch.pending()
    with pytest.raises(ValueError, match="step"):
        BatchScheduler(object(), max_length=4, eos_token_id=0, prefill_chunk=4)


# ---- the library's boundary ------------------------------------------------------------------------------------------------------
def test_hybrid_library_exports_its_header_and_nothing_else():
    from vllmini_amd import build, hybrid_ops

    path = build.build_hybrid()
    src = re.sub(r"/\*.*?\*/", "", open(os.path.join(REPO, "include", "vmi_hybrid.h")).read(), flags=re.S)
    declared = set(re.findall(r"\b(vmi_hy(?:brid)?_[a-z0-9_]+)\s*\(", src))
    assert declared == set(hybrid_ops.SIGNATURES)
    r = subprocess.run(["nm", "-D", "--defined-only", path], capture_output=True, text=True, check=True)
    funcs = {ln.split()[-1] for ln in r.stdout.splitlines() if ln.strip() and ln.split()[-2] in "TtWw"}
    assert funcs == declared, funcs ^ declared
    lib = hybrid_ops.load()
    assert lib.vmi_hybrid_abi_version() == hybrid_ops.ABI_VERSION and lib.vmi_hybrid_target_arch() == b"gfx950"


@pytest.mark.parametrize("module,error", [("hybrid_ops", "HybridLibraryError"), ("gpt2_layer", "LayerLibraryError")])
def test_a_library_of_older_sources_is_named_with_what_to_do(module, error, monkeypatch, tmp_path):
    """One of the same version that lacks an entry which came since (its struct layouts are right), and one of another version."""
    import importlib

    from vllmini_amd import build

    m = importlib.import_module(f"vllmini_amd.{module}")
    version = next(n for n in m.SIGNATURES if n.endswith("abi_version"))
    late = sorted(set(m.SIGNATURES) - {version})
    for left_out, number, words in ((late[-1], m.ABI_VERSION, f"does not export {late[-1]}"), (None, m.ABI_VERSION + 1, f"expected {m.ABI_VERSION}")):
        src, lib = tmp_path / f"{number}.c", tmp_path / f"{number}.so"
        src.write_text("".join(f"int {n}(void) {{ return {number if n == version else 0}; }}\n" for n in m.SIGNATURES if n != left_out))
        subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
        monkeypatch.setattr(build, "HYBRID_LIB_PATH" if module == "hybrid_ops" else "LAYER_LIB_PATH", str(lib))
        monkeypatch.setattr(m, "_lib", None)
        with pytest.raises(getattr(m, error), match=words) as e:
            m.load()
        assert "python -m vllmini_amd.build" in str(e.value) and str(lib) in str(e.value)


def test_the_structs_layouts_belong_to_their_version(tmp_path):
    """A caller knows a struct by its version number alone: a field that comes or moves takes a new one (3: `normed` in vmi_hy_linear_args).  The sizes as
    the C header has them, as the ctypes side has them, and as recorded for the version."""
    from vllmini_amd import hybrid_ops as h

    layouts = {2: {"linear_args": 184, "step": 112, "rglru_args": 136, "latent_prep_args": 88, "latent_attention_args": 80, "state_args": 216, "kv_prep_args": 64,
                   "attention_args": 128}}
    layouts[3] = {**layouts[2], "linear_args": 192}
    src = open(os.path.join(REPO, "include", "vmi_hybrid.h")).read()
    names = re.findall(r"^} vmi_hy_([a-z_]+);", src, flags=re.M)
    (tmp_path / "s.c").write_text('#include <stdio.h>\n#include "vmi_hybrid.h"\nint main(void) {\n' + "".join(
        f'printf("{n} %zu\\n", sizeof(vmi_hy_{n}));\n' for n in names) + "return 0; }\n")
    subprocess.run(["gcc", "-I", os.path.join(REPO, "include"), str(tmp_path / "s.c"), "-o", str(tmp_path / "s")], check=True)
    lines = subprocess.run([str(tmp_path / "s")], capture_output=True, text=True, check=True).stdout.split()
    sizes = dict(zip(lines[::2], map(int, lines[1::2])))
    assert sizes == layouts[h.ABI_VERSION]
    py = {"linear_args": h.LinearArgs, "step": h.StepArgs, "rglru_args": h.RglruArgs, "latent_prep_args": h.PrepArgs, "latent_attention_args": h.AttentionArgs,
          "state_args": h.StateArgs, "kv_prep_args": h.KvPrepArgs, "attention_args": h.GqaArgs}
    assert {n: ctypes.sizeof(c) for n, c in py.items()} == sizes


def test_gated_products_go_to_tiles_but_where_the_library_is_ahead():
    """The rule against both sides as measured: in the mean of its sizes the library with the unit behind it is ahead in two places past K 7168 only."""
    from vllmini_amd import hybrid_ops as h

    pay, only = h.load().vmi_hy_linear_tiles_pay, h.load().vmi_hy_linear_tiles_only
    for M, N, K in ((420, 20480, 8192), (1200, 8192, 16384), (742, 16384, 8192), (76, 2048, 16384), (61, 2816, 8192), (55, 1152, 8960)):
        assert not pay(M, N, K, 0, h.DTYPES[torch.bfloat16]), (M, N, K)
    for M, N, K in ((300, 6144, 1024), (4500, 6144, 1024), (948, 40960, 4096), (64, 2048, 6144), (420, 20512, 8192), (300, 16384, 8192), (2773, 8192, 8192), (130, 2048, 16384)):
        assert pay(M, N, K, 0, h.DTYPES[torch.bfloat16]), (M, N, K)
    for split in (0, 4096):
        assert only(20480, 4096, split, 0) and not only(20480, 8192, split, 0) and not only(20480, 4096, split, 1) and not only(20480, 96, split, 0)
    assert not only(4096, 4096, 4096, 0) and not pay(1 << 20, 4096, 2048, 0, 0) and not pay(0, 4096, 2048, 0, 0)


def test_products_alone_go_to_tiles_but_where_the_library_is_ahead():
    """The rule against both sides as measured."""
    from vllmini_amd import hybrid_ops as h

    pay = lambda M, N, K: h.load().vmi_hy_product_tiles_pay(M, N, K, K, h.DTYPES[torch.bfloat16])      # noqa: E731
    for M, N, K in ((7455, 2048, 1024), (5251, 3072, 1536), (3985, 6400, 1728), (4000, 6400, 1024), (4500, 2048, 6144), (2400, 4096, 2048), (64, 2048, 6144), (300, 4096, 8192), (48, 64, 16384)):
        assert not pay(M, N, K), (M, N, K)
    for M, N, K in ((3719, 2048, 1024), (3564, 2048, 1024), (7455, 2080, 1024), (5274, 1792, 768), (2300, 2048, 2048), (2400, 2080, 3072), (1300, 2048, 6144), (48, 512, 512)):
        assert pay(M, N, K), (M, N, K)


def test_whole_columns_over_a_long_k_go_to_tiles_by_what_is_left_of_the_librarys_turns():
    """Both sides as measured, 2 % and more apart: how full the library's tiles and ours leave the chip, not how many results there are."""
    from vllmini_amd import hybrid_ops as h

    pay = lambda M, N, K: h.load().vmi_hy_product_tiles_pay(M, N, K, K, h.DTYPES[torch.bfloat16])      # noqa: E731
    for M, N, K in ((3417, 2048, 3584), (1751, 5120, 3584), (2604, 3072, 4096), (3906, 2048, 4608), (3662, 2048, 5120), (3173, 2048, 6144), (3568, 2048, 6144), (3906, 2048, 6144), (1464, 5120, 6144), (1057, 6144, 5120)):
        assert not pay(M, N, K), (M, N, K)
    for M, N, K in ((2744, 2048, 3584), (1953, 3072, 4096), (2744, 2048, 5120), (4379, 2048, 4608), (1660, 5120, 4608), (1829, 3072, 5120), (914, 6144, 5120), (2744, 2048, 6144), (4379, 2048, 6144), (3125, 2560, 3072)):
        assert pay(M, N, K), (M, N, K)


def test_groups_go_to_tiles_but_where_all_run_at_once_over_a_short_k():
    """The rule against both sides as measured."""
    from vllmini_amd import hybrid_ops as h

    pick = h.load().vmi_hy_tiles_pick
    for M, N, K, groups in ((2260, 128, 512, 8), (879, 128, 512, 16), (366, 128, 512, 32), (1312, 160, 448, 10), (1628, 96, 192, 16), (900, 4096, 192, 2), (97, 512, 128, 16)):
        assert pick(M, N, K, groups) >= 0, (M, N, K, groups)
    for M, N, K, groups in ((177, 512, 128, 32), (354, 2048, 64, 4), (1365, 1024, 128, 2), (220, 4096, 192, 2), (864, 256, 64, 12), (1100, 512, 128, 3), (64, 512, 128, 16), (300, 512, 96, 16), (300, 520, 128, 16)):
        assert pick(M, N, K, groups) == -1, (M, N, K, groups)


@pytest.mark.parametrize("width,dtype,kept", [(64, torch.bfloat16, False), (96, torch.bfloat16, True), (64, torch.float32, True), (7168, torch.bfloat16, True)])
def test_gated_matrices_keep_the_librarys_layout_only_where_it_is_asked_for(width, dtype, kept):
    from vllmini_amd import hybrid_layers as hl

    w = torch.randn((48, width), generator=torch.Generator().manual_seed(width))
    for m in (hl.gated_matrix(w, dtype), hl.gated_matrix(w, dtype, 16)):
        assert (m.dense is not None) == kept and (m.N, m.K) == (64, width)
    norm = hl.Norm(torch.ones(width), width, 1e-5)
    ff = hl.ClampedGLU(width=width, limit=7.0, norm=norm, gate=w, up=w, down=w.t(), dtype=dtype)
    assert (ff.w_in.dense is not None) == kept and ff.w_out.dense is not None


def test_hybrid_entries_refuse_bad_arguments_without_touching_a_device():
    from vllmini_amd import hybrid_ops as h

    lib = h.load()
    assert lib.vmi_hy_linear(ctypes.byref(h.LinearArgs()), None) == 1
    buf = (ctypes.c_char * 256)()
    p = (ctypes.addressof(buf) + 15) & ~15
    a = h.LinearArgs(x=p, w=p, y=p, M=1, N=16, K=40, groups=1, ldx=40, ldy=16)
    assert lib.vmi_hy_linear(ctypes.byref(a), None) == 2 and b"K % 32" in lib.vmi_hybrid_last_error()
    a = h.LinearArgs(x=p, w=p, y=p, norm_w=p, normed=p + 8, M=1, N=16, K=32, groups=1, ldx=32, ldy=16, norm_n=32, x_kind=1)
    assert lib.vmi_hy_linear(ctypes.byref(a), None) == 2 and b"16-byte aligned" in lib.vmi_hybrid_last_error()
    assert lib.vmi_hy_rglru(ctypes.byref(h.RglruArgs()), ctypes.byref(h.StepArgs()), None) == 1
    assert lib.vmi_hy_latent_attention(ctypes.byref(h.AttentionArgs()), ctypes.byref(h.StepArgs()), None) == 1
    assert lib.vmi_hy_latent_prep(ctypes.byref(h.PrepArgs()), ctypes.byref(h.StepArgs()), None) == 1
    with pytest.raises(RuntimeError, match="no CPU path"):
        h.argmax(torch.zeros(1, 4))
    # what a workgroup can hold: never more row tiles than fit beside 64 keys, fp32 one
    assert [h.latent_row_tiles(576, n, torch.bfloat16) for n in (1, 2, 4)] == [1, 2, 4]
    assert h.latent_row_tiles(576, 4, torch.float32) == 1 and h.latent_row_tiles(640, 4, torch.bfloat16) == 2
    assert h.latent_row_tiles(1000, 4, torch.bfloat16) == 1


def test_large_products_stay_with_the_library_unless_their_rows_stay_in_lds():
    """dense(): 17 to 47 tokens and a large matrix go to the library, but for those behind a norm whose kernel keeps the rows in LDS; a product that
    norms its rows first is not that kernel (17 tokens, 8192 x 4096)."""
    from types import SimpleNamespace

    from vllmini_amd import hybrid_layers, hybrid_ops as h

    def of(N, K, groups=1, dtype=torch.bfloat16):
        return SimpleNamespace(N=N, K=K, groups=groups, tiles=torch.empty(0, dtype=dtype))

    assert not hybrid_layers.dense(32, of(22528, 2048), True) and hybrid_layers.dense(32, of(22528, 2048)) and not hybrid_layers.dense(17, of(24576, 4096), True)
    for M, N, K in ((17, 8192, 4096), (18, 24560, 4096), (19, 24576, 4096)):
        assert hybrid_layers.dense(M, of(N, K), True), (M, N, K)
    assert not hybrid_layers.dense(16, of(8192, 4096), True) and h.linear_normed_first(17, of(8192, 4096)) and not h.linear_normed_first(17, of(8192, 4096, 2))


@pytest.mark.parametrize("heads,row,tokens,keys,tiles", [(16, 576, 256, 4000, 1), (32, 576, 1, 1000, 1), (32, 576, 16, 400, 1), (32, 576, 16, 4000, 2), (32, 576, 64, 1000, 2), (32, 576, 128, 400, 1), (32, 576, 256, 400, 2),
                                                         (128, 576, 1, 4000, 1), (128, 576, 16, 400, 1), (128, 576, 16, 4000, 4), (128, 576, 256, 1000, 4), (32, 544, 16, 1000, 2), (64, 288, 16, 1000, 1)])
def test_single_tokens_take_a_row_tile_each_while_they_or_their_keys_are_few(heads, row, tokens, keys, tiles):
    """The tiles of a step of single tokens, of latent attention; grouped queries of as many rows take as many as fit, however many tokens there are."""
    from vllmini_amd.hybrid_decoder import HybridDecoder
    from vllmini_amd.hybrid_layers import QueryTiling

    d, at = object.__new__(HybridDecoder), np.arange(tokens)
    d.model = SimpleNamespace(dtype=torch.bfloat16)
    d._kinds = [QueryTiling("latent", heads, 1, row, sizes=(row,)), QueryTiling("grouped", heads, 1, 128, sizes=(128, 128))]
    a = {"entry": at, "pos": at, "slots": [at], "ctx": np.full(tokens, keys - 1), "state_slot": at, "parity": at * 0, "tables": np.zeros((1, tokens, 1), dtype=np.int32)}
    _, _, _, plans = d._layout(a, np.ones(tokens, dtype=np.int64), at, tokens, tokens, 1, keys)
    assert [p[0] for p in plans] == [tiles, 4 if heads > 16 else 1]
    assert plans[0][2] == tokens * -(-heads // (16 * tiles))


def test_portions_over_keys_and_values_by_the_portion_alone():
    """Which portions of a step go through latent_prompt, between which tokens and entries they and the others lie, and their tiles where others stand among them and the places are many;
    the others keep the latents, and captured steps have none."""
    from vllmini_amd.hybrid_decoder import HybridDecoder
    from vllmini_amd.hybrid_layers import QueryTiling

    d = object.__new__(HybridDecoder)
    d.model = SimpleNamespace(dtype=torch.bfloat16)
    d._kinds = [QueryTiling("latent", 16, 1, 576, sizes=(576,)), QueryTiling("latent", 16, 1, 576, sizes=(576,), prompts=True)]
    many = [1] * 100 + [2] * 60 + [1200]
    for ctx, counts, tiles, span, own in (
            ([9, 0, 30, 0, 0], [1, 130, 70, 1, 64], None, (1, 266, 0, 201, 1, 5), {0, 2}), ([0, 0], [2, 65], None, (0, 67, 0, 0, 0, 2), set()),
            ([5, 8], [1, 1], None, None, {0, 1}), ([5, 0], [1, 1], None, (1, 2, 0, 1, 1, 2), {0}), ([64, 0], [64, 300], None, (64, 364, 0, 64, 1, 2), {0}),
            ([3] * 100 + [0] * 61, many, None, (100, 1420, 0, 100, 100, 161), set(range(100))),
            ([0] + [3] * 99 + [0] * 61, [2] + many[1:], [(160, 64 * i) for i in range(18, 0, -1)] + [(i, 0) for i in (0, *range(100, 161))], (0, 1421, 2, 101, 0, 161), set(range(1, 100)))):
        ctx, counts = np.asarray(ctx), np.asarray(counts)
        n, T = len(counts), int(counts.sum())
        a = {"entry": np.repeat(np.arange(n), counts), "pos": np.zeros(T), "slots": [np.zeros(T)], "ctx": ctx, "state_slot": counts * 0, "parity": counts * 0, "tables": np.zeros((1, n, 1), dtype=np.int32)}
        sec, _, _, plans = d._layout(a, counts, np.arange(n), T, n, 1, int((ctx + counts).max()))
        assert plans[0][3] is None and set(sec["tiles0"][::2]) == set(range(n))
        assert plans[1][3] == span and set(sec["tiles1"][::2]) == own
        assert d._layout(a, counts, np.arange(n), T, n, 1, int((ctx + counts).max()), captured=True)[3][1][3] is None
        assert ("prompts" in sec) == (tiles is not None) and (tiles is None or list(map(tuple, sec["prompts"].reshape(-1, 2).tolist())) == tiles)


def test_products_behind_a_norm_of_few_rows_and_columns_share_one_kernel_whatever_their_width():
    """Up to 2048 columns, up to 64 rows, one workgroup a compute unit with one slab of 16 columns each: no width among them goes to kernels for more."""
    from vllmini_amd import hybrid_ops as h

    for K in range(32, 2049, 32):
        for M in (1, 12, 16, 17, 33, 47, 64):
            for N in (32, 512, 16 * (256 // -(-M // 16))):
                assert h.load().vmi_hy_linear_slabs(M, N, K, 0) > 0 and not h.load().vmi_hy_linear_normed(M, N, K, 1, 0), (M, N, K)
    assert h.load().vmi_hy_linear_slabs(12, 512, 2080, 0) == h.load().vmi_hy_linear_slabs(12, 512, 1024, 1) == h.load().vmi_hy_linear_slabs(12, 512, 1000, 0) == 0


def test_rows_normed_once_are_held_at_every_multiple_of_1024_columns():
    """Whole chunks of K a wave are what the kernel that holds its rows in registers asks for, and few columns of long rows are left to kernels that share a slab's K out."""
    from vllmini_amd import hybrid_ops as h

    held, normed = h.load().vmi_hy_linear_held, h.load().vmi_hy_linear_normed
    for K in (1024, 2048, 3072):
        assert held(40, 50272, K, 0) and normed(40, 50272, K, 1, 0) and not held(65, 50272, K, 0) and not held(8, 50272, K, 0)
    assert held(33, 512, 3072, 0) and held(9, 50272, 2048, 0) and not held(32, 50272, 3072, 0) and not held(40, 50272, 2560, 0) and not held(40, 50272, 4096, 0)
    rows = h.load().vmi_hy_linear_holds
    for M, N, stored, want in ((16, 4096, 1, 0), (16, 6144, 1, 1), (32, 8192, 1, 0), (32, 12288, 0, 1), (40, 512, 1, 0), (40, 512, 0, 1), (64, 4096, 1, 1)):
        assert rows(M, N, 4096, stored, 0) == want, (M, N, stored)


def test_products_of_few_rows_over_many_columns_read_their_rows_once():
    """The kernel whose every workgroup brings the rows again is for a workgroup a compute unit, or for rows that are few or short."""
    from vllmini_amd import hybrid_ops as h

    plain = h.load().vmi_hy_linear_plain
    for K in (128, 512, 1024, 2048, 4096, 4608):
        assert all(plain(M, 16 * (256 // g), K, g, 0) for M in (1, 16, 32, 64) for g in (1, 8))
        assert plain(16, 8192, K, 1, 0) and not plain(65, 512, K, 1, 0)
    for M, N, K, groups in ((47, 16384, 2048, 1), (24, 16384, 1280, 1), (64, 8192, 768, 1), (16, 16384, 4096, 1), (32, 6144, 4096, 1), (1, 6144, 5120, 1), (16, 1024, 5120, 1), (64, 16384, 128, 1),
                            (64, 128, 512, 64), (47, 512, 128, 64), (64, 128, 256, 128)):
        assert not plain(M, N, K, groups, 0), (M, N, K, groups)
    assert plain(47, 576, 128, 64, 0) and plain(64, 6144, 12288, 1, 0) and not plain(1, 512, 128, 1, 1)


def test_command_line_lists_models_and_parses_requests(capsys):
    from vllmini_amd.__main__ import _parser, main

    assert main(["models"]) == 0 and "Voduvik" in capsys.readouterr().out
    a = _parser().parse_args(["generate", "--model", "x", "--prompt-ids", "1,2", "--prompt-ids", "3", "--prefill-chunk", "8"])
    assert a.prompt_ids == ["1,2", "3"] and a.prefill_chunk == 8
    r = subprocess.run([os.path.join(REPO, "bin", "trace_run"), "--help"], capture_output=True, text=True)
    assert r.returncode == 0 and "--max-tokens" in r.stdout
