"""GPU parity of the wide kernels (a slot's dispatch rows in passes of up to 32
over the whole of K) against the oracle, where their tiles can go wrong: one row,
15 / 16 / 17 rows (a column tile and its edge), 31 / 32 / 33 (a pass and its edge),
an intermediate that fills its last block of row tiles in part, and, from 128
tokens, slots on both sides of the rows the GEMM tiles take over at."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import dsk_moe
from oracle import layer as L
from oracle import synth
from conftest import assert_layer_close
from test_gpu_layer import to_bank, to_shared

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(spec, T, hot, seed, label, shared=True, f32=False):
    print(f"wide {label} T={T} hot={hot}", flush=True)
    d = synth.make_layer(spec, seed, T)
    if f32:
        d["x"] = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(seed))
    if hot:
        d["gate_b"] = d["gate_b"].clone()
        d["gate_b"][:hot] += 10.0          # every token goes to experts 0 .. hot - 1
    r = L.moe_forward(d["x"], d["gate_w"], d["gate_b"], d["bank"], d["shared"] if shared else None, spec)
    idx = torch.empty((T, spec.k), dtype=torch.int32, device=DEV)
    layer = dsk_moe.MoELayer(d["gate_w"].to(DEV), d["gate_b"].to(DEV), to_bank(d["bank"]),
                             to_shared(d["shared"]) if shared else None, spec.k)
    x = d["x"].to(DEV)
    out = layer(x, idx=idx)
    again = layer(x)
    assert torch.equal(out, again)
    np.testing.assert_array_equal(idx.cpu().numpy(), r["idx"])
    c, rel = assert_layer_close(out.cpu().float(), r["y_ref"])
    if f32:        # hi / lo pairs hold 2^-17, h and x each: well inside 1e-4 of the largest output
        assert rel < 1e-4
    print(f"cos={c:.9f} rel={rel:.2e} rows {sorted(set(int(v) for v in r['counts']))}", flush=True)
    return r


@pytest.mark.parametrize("T,hot", [(9, 0), (15, 4), (16, 4), (17, 4), (31, 4), (32, 4), (33, 4), (127, 4)])
def test_wide_rows_of_a_slot(T, hot):
    _check(L.LayerSpec(H=1024, E=24, k=4, I=512, I_shared=256), T, hot, 310 + T, "rows")


@pytest.mark.parametrize("T,hot,H,I", [(3, 0, 1024, 512), (9, 0, 512, 256), (17, 4, 1024, 768), (70, 0, 5120, 256),
                                       (127, 4, 1024, 512)])
def test_wide_float32_pairs(T, hot, H, I):
    """float32 x: passes of 16 rows and a part of one, the shared expert over one and two
    groups of 64 tokens, the decode pipeline's form (3 tokens)."""
    _check(L.LayerSpec(H=H, E=16, k=4, I=I, I_shared=256), T, hot, 370 + T, f"f32 H {H} I {I}", f32=True)


@pytest.mark.parametrize("T,hot,H,I", [(1, 0, 1024, 640), (2, 0, 4096, 512), (4, 0, 512, 512), (9, 4, 1024, 640), (16, 4, 768, 768), (17, 4, 1024, 896),
                                       (40, 4, 5120, 512), (150, 0, 1024, 768), (300, 4, 512, 1024)])
def test_wide_q3(T, hot, H, I):
    """q3: sets of eight rows and a part of one, passes of sixteen, one to three blocks
    after the last superblock, the decode pipeline's form (1, 2, 4 tokens), and from 128
    tokens GEMM tiles alone (more than 16 rows a slot on average)."""
    _check(L.LayerSpec(H=H, E=16, k=4, I=I, I_shared=256, quant=L.QUANT_Q3), T, hot, 410 + T, f"q3 H {H} I {I}")


@pytest.mark.parametrize("T", [4, 7])
def test_wide_in_the_decode_pipeline(T):
    _check(L.LayerSpec(H=1024, E=32, k=4, I=512, I_shared=256), T, 0, 390 + T, "decode")
    _check(L.LayerSpec(H=1024, E=32, k=4, I=512, I_shared=256), T, 0, 390 + T, "decode, no shared", shared=False)


@pytest.mark.parametrize("H,I,Is", [(1024, 256, 128), (5120, 768, 384), (2048, 2304, 0)])
def test_wide_shapes(H, I, Is):
    """Two K steps, an odd number of them, and rows of scales of 8-byte pieces."""
    _check(L.LayerSpec(H=H, E=6, k=2, I=I, I_shared=Is or 128), 20, 0, 330, f"H {H} I {I}", shared=Is > 0)


@pytest.mark.parametrize("T,E,k", [(128, 64, 4), (150, 16, 4), (300, 24, 4), (520, 64, 2)])
def test_wide_slots_beside_gemm_tiles(T, E, k):
    """From 128 tokens: slots of up to 32 rows beside GEMM tiles of 64 and 128 columns,
    the shared expert in the wide kernels (up to 512 tokens) and in GEMM tiles."""
    r = _check(L.LayerSpec(H=1024, E=E, k=k, I=768, I_shared=256), T, 0, 350, f"E {E} k {k}")
    assert int(r["counts"].min()) <= 32 or E == 24


@pytest.mark.parametrize("T,hot,E", [(130, 0, 64), (150, 40, 64), (150, 0, 40), (513, 0, 256)])
def test_wide_q3_prefill_slots(T, hot, E):
    """q3 from 128 tokens: from 32 slots of at most 16 rows these and (up to 512 tokens)
    the shared expert on the wide kernels beside GEMM tiles (64 and 256 experts), with
    fewer all on GEMM tiles (40 experts)."""
    _check(L.LayerSpec(H=512, E=E, k=4, I=2048, I_shared=256, quant=L.QUANT_Q3), T, hot, 470 + T, f"q3 E {E}")


@pytest.mark.parametrize("quant,H,I,T,k", [("fp4", 1024, 512, 1, 8), ("fp4", 1024, 512, 3, 12), ("fp4", 1024, 768, 20, 4),
                                           ("fp4", 3072, 512, 127, 2), ("q3", 1024, 640, 1, 8), ("q3", 1024, 640, 5, 12),
                                           ("q3", 1024, 640, 24, 4)])
def test_wide_repeated_experts(quant, H, I, T, k):
    """A caller's routing that names an expert several times in a row: slots of more
    rows than the call has tokens (1 to 16 tokens: the LDS of one column tile, with
    more than 16 rows; more tokens: of two)."""
    from dsk_moe.layer import experts_forward
    print(f"wide repeated {quant} H={H} I={I} T={T} k={k}", flush=True)
    spec = L.LayerSpec(H=H, E=16, k=k, I=I, I_shared=256, quant=L.QUANT_Q3 if quant == "q3" else L.QUANT_FP4)
    d = synth.make_layer(spec, 450 + T, T)
    rng = np.random.default_rng(T)
    idx = np.where(np.arange(k) < k - k // 4, 3, rng.integers(0, spec.E, (T, k))).astype(np.int32)
    w = (rng.random((T, k), dtype=np.float32) + 0.5) / k
    r = L.moe_forward(d["x"], None, None, d["bank"], d["shared"], spec, routing=(idx, w, None, None))
    assert int(r["counts"].max()) > T
    out = experts_forward(d["x"].to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV),
                          to_bank(d["bank"]), to_shared(d["shared"]))
    c, rel = assert_layer_close(out.cpu().float(), r["y_ref"])
    print(f"cos={c:.9f} rel={rel:.2e} rows {int(r['counts'].max())}", flush=True)


@pytest.mark.parametrize("quant,H,I,T,E,k", [
    ("fp4", 1024, 512, 20, 16, 4), ("fp4", 5120, 768, 4, 16, 4), ("fp4", 1024, 768, 200, 16, 4),
    ("fp4", 2560, 768, 200, 64, 2), ("fp4", 384, 128, 9, 8, 2), ("q3", 1024, 640, 20, 16, 4), ("q3", 4096, 512, 10, 16, 4),
    ("q3", 512, 2048, 130, 64, 4), ("q3", 1024, 640, 300, 16, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_not_finite_activations(quant, H, I, T, E, k, dtype):
    """A row of x with an infinity or a NaN comes out as NaN throughout (as the oracle
    gives it), on FP8 planes, bf16 pairs and factored sums alike; other rows are untouched."""
    from dsk_moe.layer import experts_forward
    print(f"not finite {quant} H={H} I={I} T={T} {dtype}", flush=True)
    spec = L.LayerSpec(H=H, E=E, k=k, I=I, I_shared=128, quant=L.QUANT_Q3 if quant == "q3" else L.QUANT_FP4)
    d = synth.make_layer(spec, 480, T)
    rng = np.random.default_rng(T)
    idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    w = (rng.random((T, k), dtype=np.float32) + 0.5) / k
    clean = d["x"].to(dtype)
    x = clean.clone()
    bad = [0, T // 2, T - 1]
    for t, v in zip(bad, (float("inf"), float("-inf"), float("nan"))):
        x[t, (77 * (t + 1)) % H] = v
    r = L.moe_forward(x, None, None, d["bank"], None, spec, routing=(idx, w, None, None))
    assert torch.isnan(r["y_ref"][bad]).all()
    bank = to_bank(d["bank"])
    run = lambda v: experts_forward(v.to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), bank).cpu()
    out, ok = run(x), np.setdiff1d(np.arange(T), bad)
    assert torch.isnan(out[bad]).all()
    assert torch.equal(out[ok], run(clean)[ok])
    assert_layer_close(out[ok].float(), r["y_ref"][ok])


def _experts(quant, H, I, Is, T, E, k, seed, label, idx=None, f32=False):
    """experts_forward of a random routing (no expert twice in a row) against the oracle."""
    from dsk_moe.layer import experts_forward
    print(f"wide {label} {quant} H={H} I={I} Is={Is} T={T} E={E} k={k}", flush=True)
    spec = L.LayerSpec(H=H, E=E, k=k, I=I, I_shared=Is or 128, quant=L.QUANT_Q3 if quant == "q3" else L.QUANT_FP4)
    d = synth.make_layer(spec, seed, T)
    rng = np.random.default_rng(seed)
    if idx is None:
        idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    w = (rng.random((T, k), dtype=np.float32) + 0.5) / k
    shared = d["shared"] if Is else None
    if f32:
        d["x"] = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(seed))
    r = L.moe_forward(d["x"], None, None, d["bank"], shared, spec, routing=(idx, w, None, None))
    run = lambda: experts_forward(d["x"].to(DEV), torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV),
                                  to_bank(d["bank"]), to_shared(shared))
    out = run()
    assert torch.equal(out, run())
    c, rel = assert_layer_close(out.cpu().float(), r["y_ref"])
    if f32:
        assert rel < 1e-4       # (see _check)
    print(f"cos={c:.9f} rel={rel:.2e} rows {sorted(set(int(v) for v in r['counts']))}", flush=True)


@pytest.mark.parametrize("quant,H,I,Is,T", [("fp4", 1024, 2048, 384, 3), ("fp4", 5120, 768, 256, 7), ("fp4", 5120, 768, 256, 8),
                                            ("fp4", 2048, 1024, 2304, 8), ("fp4", 1024, 2048, 384, 9), ("q3", 1024, 640, 256, 1),
                                            ("q3", 1024, 640, 384, 8), ("q3", 1024, 640, 256, 9)])
def test_wide_shared_expert_of_few_tokens(quant, H, I, Is, T):
    """The shared expert beside wide slots: column tiles up to eight tokens (of as many
    rows as the LDS of half a CU holds), the wide walk from there."""
    _experts(quant, H, I, Is, T, 16, 4, 520 + T, "shared")


@pytest.mark.parametrize("H,I,Is,T,k", [(1024, 512, 256, 1, 4), (1024, 512, 256, 8, 4), (1024, 512, 256, 9, 4), (4096, 256, 0, 16, 2),
                                        (4096, 256, 0, 17, 2), (1024, 2048, 256, 1, 8), (1024, 2048, 256, 2, 8), (1024, 2048, 0, 2, 8), (8192, 256, 0, 20, 2),
                                        (1024, 4096, 0, 4, 1), (1024, 4096, 0, 5, 1)])
def test_wide_little_work(H, I, Is, T, k):
    """Both sides of the work up to which FP4 slots stay with the column tiles (positions x
    I of 16384, from H 4096 of 8192; two tokens with a shared expert), and a hidden size
    past the wide kernels'."""
    _experts("fp4", H, I, Is, T, 16, k, 540 + T, "little work")


@pytest.mark.parametrize("T,I,shared", [(4, 1280, True), (5, 1536, False), (8, 768, True)])
def test_wide_decode_pipeline_sizes(T, I, shared):
    """The decode pipeline's wide form (four tokens and more work than the column tiles keep)."""
    _check(L.LayerSpec(H=1024, E=32, k=4, I=I, I_shared=256), T, 0, 560 + T, f"decode I {I}", shared=shared)


@pytest.mark.parametrize("H,I,Is,T,k", [(5120, 256, 0, 16, 4), (1024, 768, 256, 16, 4), (5120, 2304, 0, 1, 2), (1024, 1280, 0, 9, 4),
                                        (7168, 256, 128, 12, 6), (2048, 2304, 0, 7, 4)])
def test_wide_few_rows(H, I, Is, T, k):
    """Slots of one, two, three and four rows beside each other where the slots are many
    for the rows (K ranges of one step and none, of an odd number of steps; blocks that
    fill less than half the CUs, more than all of them, and between)."""
    idx = np.arange(T * k).reshape(T, k)
    for first, rows in ((0, 4), (4, 3), (7, 2)):          # rows that share their first expert
        if first + rows <= T:
            idx[first:first + rows, 0] = idx[first, 0]
    _experts("fp4", H, I, Is, T, 72, k, 580 + T, "few rows", idx=idx.astype(np.int32))


@pytest.mark.parametrize("H,I,Is,T,k", [(1024, 512, 256, 8, 4), (1024, 512, 256, 9, 4), (1024, 512, 0, 4, 4), (1024, 512, 0, 5, 4),
                                        (512, 2048, 128, 1, 8), (512, 2048, 0, 1, 8)])
def test_wide_float32_little_work(H, I, Is, T, k):
    """Both sides of the work up to which float32 calls stay with the general kernels."""
    _experts("fp4", H, I, Is, T, 16, k, 600 + T, "float32 little work", f32=True)


@pytest.mark.parametrize("T,E,k,hot,I", [(820, 64, 3, 2, 768), (820, 128, 3, 2, 768), (810, 24, 2, 1, 1024), (600, 64, 3, 2, 768)])
def test_skewed_fp4_prompt(T, E, k, hot, I):
    """Skewed prompts: too few narrow slots for the wide kernels (left to the GEMM tiles),
    enough of them, and, up to 800 tokens, whatever their number beside the shared expert."""
    r = _check(L.LayerSpec(H=512, E=E, k=k, I=I, I_shared=128), T, hot, 640 + E, "skewed prompt")
    narrow = int(((r["counts"] > 0) & (r["counts"] <= 32)).sum())
    need = -(-2 * 256 * 128 // I)
    assert (r["counts"][:hot] == T).all()
    assert narrow >= need if E == 128 else narrow < need


def test_tile_list_of_the_dispatch():
    """The tile list written by the multi-block dispatch (8192 positions and more) is the
    one that the entry point with a routing of its own makes: the same rows."""
    from dsk_moe.layer import experts_forward
    print("tile list", flush=True)
    spec = L.LayerSpec(H=512, E=40, k=4, I=512, I_shared=128)
    for T in (2080, 700):
        d = synth.make_layer(spec, 660, T, zipf_s=0.5)
        bank, shared, x = to_bank(d["bank"]), to_shared(d["shared"]), d["x"].to(DEV)
        idx, w = torch.empty((T, spec.k), dtype=torch.int32, device=DEV), torch.empty((T, spec.k), device=DEV)
        layer = dsk_moe.MoELayer(d["gate_w"].to(DEV), d["gate_b"].to(DEV), bank, shared, spec.k)
        out = layer(x, idx=idx, w=w)
        assert torch.equal(out, experts_forward(x, idx, w, bank, shared))
        r = L.moe_forward(d["x"], None, None, d["bank"], d["shared"], spec, routing=(idx.cpu().numpy(), w.cpu().numpy(), None, None))
        assert_layer_close(out.cpu().float(), r["y_ref"])


@pytest.mark.parametrize("role,T", [("w1", 150), ("w2", 150), ("w3", 600)])
def test_prompt_with_arrays_at_eight_bytes(role, T):
    """FP4 codes of one role off 16-byte alignment: the register-staged GEMM loop takes
    every slot, narrow ones too, beside the shared expert's wide blocks."""
    print(f"arrays at eight bytes {role} T={T}", flush=True)
    spec = L.LayerSpec(H=1024, E=48, k=2, I=768, I_shared=256)
    d = synth.make_layer(spec, 680, T)
    r = L.moe_forward(d["x"], d["gate_w"], d["gate_b"], d["bank"], d["shared"], spec)
    bank = to_bank(d["bank"])
    codes, scales = bank.roles[role]
    raw = torch.empty(codes.numel() + 8, dtype=torch.uint8, device=DEV)
    off = raw[8:].view(codes.shape)
    off.copy_(codes)
    assert off.data_ptr() % 16 == 8
    roles = dict(bank.roles)
    roles[role] = (off, scales)
    layer = dsk_moe.MoELayer(d["gate_w"].to(DEV), d["gate_b"].to(DEV), dsk_moe.ResidentBank("fp4", roles),
                             to_shared(d["shared"]), spec.k)
    out = layer(d["x"].to(DEV)).cpu()
    assert_layer_close(out.float(), r["y_ref"])


@pytest.mark.parametrize("T", [23, 24, 27, 28])
def test_wide_q3_down_beside_column_tiles(T):
    """H 4096: column tiles to 23 tokens, the wide gate/up with the tiles' down to 27, then
    both wide."""
    _check(L.LayerSpec(H=4096, E=12, k=3, I=512, I_shared=128, quant=L.QUANT_Q3), T, 1, 700 + T, "q3 down")


@pytest.mark.parametrize("T,hot,wide", [(130, 0, True), (130, 1, True), (200, 4, False)])
def test_wide_q3_prompt_after_the_last_superblock(T, hot, wide):
    """q3 from 128 tokens with two blocks of H and three of I after their last superblock:
    enough slots of at most 16 rows (the wide kernels, beside GEMM tiles for the hot
    expert), and too few."""
    spec = L.LayerSpec(H=768, E=64, k=4, I=1408, I_shared=128, quant=L.QUANT_Q3)
    r = _check(spec, T, hot, 720 + T, f"q3 prompt hot={hot}")
    narrow = int(((r["counts"] > 0) & (r["counts"] <= 16)).sum())
    assert T * spec.k <= 16 * spec.E
    assert (narrow >= -(-2 * 256 * 128 // spec.I)) == wide
    assert not hot or int(r["counts"].max()) > 16
