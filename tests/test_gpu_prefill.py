"""GPU parity of the prefill path (activation quantisation and grouped GEMMs)."""

from __future__ import annotations

import ctypes
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle
from oracle import synth
from oracle.numerics import bf16_round
from freetoken_amd import _lib, ops

from _helpers import bf16_dev, to_device_bank, to_np
from conftest import COS_TOL, MAX_REL_TOL, cosine, max_rel

pytestmark = pytest.mark.gpu

BLOCKS_HELPER = Path(__file__).resolve().parent / "gpu_helpers" / "libprefillblocks.so"
_FMT_CODE = {"bf16": _lib.FMT_BF16, "fp8": _lib.FMT_FP8_B128, "mxfp4": _lib.FMT_MXFP4}


def _block(fmt, M, k, rows, H, I):
    """Routes per tile of a prefill call (the launch's own rule)."""
    if not BLOCKS_HELPER.exists():
        from tests.gpu_helpers import build_helpers  # built by __graft_entry__.build(); rebuilt if absent

        build_helpers.build()
    return ctypes.CDLL(str(BLOCKS_HELPER)).prefill_blocks(_FMT_CODE[fmt], M, k, rows, H, I)


@pytest.mark.parametrize("rows,K", [(1, 128), (37, 1024), (513, 7168)])
def test_act_quant_fp8_exact(dev, rows, K):
    rng = np.random.default_rng(rows)
    x = bf16_round(synth.activations(rng, rows, K) * np.float32(rng.uniform(0.01, 30)))
    x[0, :128] = 0.0  # all-zero group: amax clamp
    q_ref, s_ref = oracle.experts.per_token_group_quant_fp8(x)
    q, s = ops.act_quant_fp8(bf16_dev(x, dev), 0)
    np.testing.assert_array_equal(to_np(s), s_ref)
    np.testing.assert_array_equal(to_np(q), q_ref)


@pytest.mark.parametrize("rows,K", [(3, 256), (129, 2048)])
def test_act_quant_ue8m0_exact(dev, rows, K):
    rng = np.random.default_rng(rows + 1)
    x = bf16_round(synth.activations(rng, rows, K) * np.float32(3.0))
    x[1, 128:256] = bf16_round(np.float32(1e-6))  # below the 1e-4 amax floor
    q_ref, c_ref = oracle.experts.act_quant_ue8m0(x)
    q, c = ops.act_quant_fp8(bf16_dev(x, dev), 1)
    np.testing.assert_array_equal(to_np(c), c_ref)
    np.testing.assert_array_equal(to_np(q), q_ref)


def _prefill_case(fmt, E, H, I, M, k, shared, seed, grouped=True):
    rng = np.random.default_rng(seed)
    bank = synth.make_bank(fmt, E, H, I, rng)
    sh = synth.make_bank(fmt, 1, H, I, rng) if shared else None
    x = synth.activations(rng, M, H)
    if grouped:
        lg = synth.normal(rng, (M, E)) + synth.zipf_bias(rng, E)[None, :]
        w, ids = oracle.routing.grouped_sigmoid_topk(lg, synth.normal(rng, (E,), 0.05), 8, 4, k, True, 2.5)
    else:
        lg = synth.normal(rng, (M, E))
        w, ids = oracle.routing.softmax_topk(lg, k, True)
    return bank, sh, x, w, ids


PREFILL_CASES = [
    ("fp8_shared", "fp8", 32, 1024, 256, 512, 8, True),
    ("mxfp4_shared", "mxfp4", 32, 1024, 256, 512, 8, True),
    ("fp8_noshared_small", "fp8", 16, 512, 384, 37, 8, False),
    ("bf16", "bf16", 16, 512, 256, 300, 2, False),
    # every token on 8 of 16 experts: experts of up to 10 M blocks, so the
    # tile schedule's chunks of 8 (FP8 gate_up) and 2 (down) run full and
    # with a remainder
    ("fp8_hot_experts", "fp8", 16, 512, 256, 2560, 8, True),
    ("mxfp4_hot_experts", "mxfp4", 16, 512, 256, 2560, 8, False),
]


@pytest.mark.parametrize("case", PREFILL_CASES, ids=[c[0] for c in PREFILL_CASES])
def test_prefill_parity(dev, case):
    name, fmt, E, H, I, M, k, shared = case
    bank, sh, x, w, ids = _prefill_case(fmt, E, H, I, M, k, shared, seed=len(name), grouped=(E % 8 == 0 and k == 8))
    y_ref = oracle.experts.moe_layer("prefill", x, w, ids, bank, sh)
    y = ops.experts_prefill(bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev),
                            to_device_bank(bank, dev), to_device_bank(sh, dev) if sh else None)
    got = to_np(y)
    assert max_rel(got, y_ref) <= MAX_REL_TOL, (name, max_rel(got, y_ref))
    assert cosine(got, y_ref) >= COS_TOL, (name, cosine(got, y_ref))


def test_prefill_skipped_ids_and_sentinel(dev):
    bank, sh, x, w, ids = _prefill_case("fp8", 16, 512, 256, 64, 4, True, seed=3, grouped=False)
    ids[0, 0] = -1
    ids[5, 2] = 16  # == num_experts: the align sentinel bucket, no expert
    ids[7, 1] = 99
    y_ref = oracle.experts.moe_layer("prefill", x, w, ids, bank, sh)
    y = ops.experts_prefill(bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev),
                            to_device_bank(bank, dev), to_device_bank(sh, dev))
    got = to_np(y)
    assert max_rel(got, y_ref) <= MAX_REL_TOL
    assert cosine(got, y_ref) >= COS_TOL


def test_prefill_deterministic(dev):
    bank, sh, x, w, ids = _prefill_case("fp8", 32, 1024, 256, 256, 8, True, seed=4)
    args = (bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev),
            to_device_bank(bank, dev), to_device_bank(sh, dev))
    a = ops.experts_prefill(*args).clone()
    b = ops.experts_prefill(*args)
    assert torch.equal(a, b)


def test_decode_and_prefill_agree_on_bf16(dev):
    """The two regimes compute the same bf16 math (reference decode-vs-grouped
    check, tests/moe/test_fused_moe.py:101-156, tolerance 2e-2)."""
    bank, _, x, w, ids = _prefill_case("bf16", 16, 512, 256, 24, 4, False, seed=5, grouped=False)
    args = (bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev), to_device_bank(bank, dev))
    a = to_np(ops.experts_prefill(*args))
    b = to_np(ops.experts_decode(*args))
    assert max_rel(a, b) <= 2e-2 and cosine(a, b) >= COS_TOL


@pytest.mark.parametrize("activation", ["gelu", "gelu_tanh"])
@pytest.mark.parametrize("fmt", ["fp8", "mxfp4", "bf16"])
def test_prefill_activation_variants(dev, fmt, activation):
    """The gelu forms of the gate/up epilogue (reference kernel/triton/
    activation.py:99-109), which takes the runtime-kind branch of the
    quantised GEMMs' epilogue (SiLU has its own straight-line code)."""
    bank, sh, x, w, ids = _prefill_case(fmt, 16, 512, 256, 300, 4, fmt != "bf16", seed=11, grouped=False)
    y_ref = oracle.experts.moe_layer("prefill", x, w, ids, bank, sh, activation=activation)
    y = ops.experts_prefill(bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev),
                            to_device_bank(bank, dev), to_device_bank(sh, dev) if sh else None, activation=activation)
    got = to_np(y)
    assert max_rel(got, y_ref) <= MAX_REL_TOL, (fmt, activation, max_rel(got, y_ref))
    assert cosine(got, y_ref) >= COS_TOL, (fmt, activation, cosine(got, y_ref))
    y_silu = oracle.experts.moe_layer("prefill", x, w, ids, bank, sh)
    assert max_rel(y_silu, y_ref) > 4 * MAX_REL_TOL


def _bank_rows(bank, rows):
    """The device bank's rows in turn, `rows` of them."""
    def take(t):
        idx = torch.arange(rows, device=bank.gate_up.device) % t.shape[0]
        return t.view(torch.uint8)[idx].view(t.dtype)

    return ops.ExpertBank(bank.fmt, *(take(t) if t is not None else None
                                      for t in (bank.gate_up, bank.down, bank.gate_up_scale, bank.down_scale)))


@pytest.mark.parametrize("H,I", [(640, 384), (128, 1152), (1024, 128)])
@pytest.mark.parametrize("fmt,block,n,E,E2", [
    ("fp8", 64, 2, 16, 3), ("fp8", 128, 1, 4, 16), ("fp8", 256, 24, 4, 128),
    ("mxfp4", 64, 2, 16, 3), ("mxfp4", 128, 1, 4, 16), ("mxfp4", 256, 24, 4, 128),
    ("bf16", 64, 2, 16, 3), ("bf16", 128, 1, 4, 16), ("bf16", 256, 24, 4, 128),
])
def test_prefill_block_sizes(dev, fmt, block, n, E, E2, H, I):
    """Every routes-per-tile variant of the GEMMs at its edges: one expert with
    n full blocks, one with a route more, one with a single route, the rest
    empty (the mean over the E bank rows picks the variant); K of 1, 3, 5, 8 and
    9 blocks of 128: shorter than the copies run ahead, whole and partial groups
    of scales.  The tiling does not enter an output's arithmetic, so the same
    call over E2 rows, which takes another variant, gives the same bits.
    The oracle is held by its 2-norm: with these short K a single activation
    whose bf16 rounding, and with it its e4m3 code, falls the other way (the
    sums differ in their last bit) moves one output row by up to 1/16 of that
    product, which the maximum over few outputs would show as 2-3%."""
    rng = np.random.default_rng(block + H)
    flat = np.repeat(np.arange(3, dtype=np.int32), [n * block, n * block + 1, 1])
    ids = rng.permutation(flat).reshape(-1, 2)
    M = ids.shape[0]
    assert _block(fmt, M, 2, E, H, I) == block != _block(fmt, M, 2, E2, H, I)
    w = rng.uniform(0.1, 1.0, size=ids.shape).astype(np.float32)
    bank, sh = synth.make_bank(fmt, 16, H, I, rng), synth.make_bank(fmt, 1, H, I, rng)
    x = synth.activations(rng, M, H)
    y_ref = oracle.experts.moe_layer("prefill", x, w, ids, bank, sh)
    y, y2 = (ops.experts_prefill(bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev),
                                 _bank_rows(to_device_bank(bank, dev), r), to_device_bank(sh, dev)) for r in (E, E2))
    assert torch.equal(y, y2)
    got = to_np(y).astype(np.float64)
    assert np.linalg.norm(got - y_ref) <= 1e-2 * np.linalg.norm(y_ref)
    assert cosine(got, y_ref) >= COS_TOL, cosine(got, y_ref)


@pytest.mark.parametrize("hb,ib,shared", [(5, 1, True), (6, 2, False), (7, 3, True), (9, 4, False), (1, 6, True),
                                          (2, 5, False), (3, 7, False), (4, 9, True)])
@pytest.mark.parametrize("fmt", ["fp8", "mxfp4", "bf16"])
def test_prefill_many_tiles_per_workgroup(dev, fmt, hb, ib, shared):
    """The persistent GEMMs with several tiles for every workgroup, where copies,
    scale groups, route lists and router weights run on from tile to tile: K of
    1 to 9 blocks of 128 in both GEMMs (shorter than the copies run ahead, up to
    twice that, every remainder of the groups of four).  One routing over 60
    experts; more bank rows take a smaller tile, with the same bits; tokens taken
    at random are held against the oracle (by the 2-norm, as above)."""
    H, I, E, k = 128 * hb, 128 * ib, 60, 8
    rng = np.random.default_rng(100 * hb + ib)
    distinct = 7  # weights that repeat over the bank's rows: no neighbour has its expert's
    bank, sh = synth.make_bank(fmt, distinct, H, I, rng), synth.make_bank(fmt, 1, H, I, rng) if shared else None
    M = 330 * E // k
    x = synth.activations(rng, M, H)
    w, ids = oracle.routing.softmax_topk(synth.normal(rng, (M, E)), k, True)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    counts = np.bincount(ids.ravel(), minlength=E)
    dbank, dsh = to_device_bank(bank, dev), to_device_bank(sh, dev) if shared else None
    args = (bf16_dev(x, dev), torch.from_numpy(w).to(dev), torch.from_numpy(ids).to(dev))
    outs = {}
    for rows in (E, 200, 1000):
        bm = _block(fmt, M, k, rows, H, I)
        blocks = int(np.sum(-(-counts // bm))) + (-(-M // bm) if shared else 0)
        assert max(blocks * ib, blocks * -(-H // 256)) > cus  # gate_up, down
        outs[bm] = ops.experts_prefill(*args, _bank_rows(dbank, rows), dsh)
    assert set(outs) == {64, 128, 256}
    y = outs[64]
    for other in outs.values():
        assert torch.equal(y, other)
    s = rng.choice(M, size=24, replace=False)
    y_ref = oracle.experts.moe_layer("prefill", x[s], w[s], ids[s] % distinct, bank, sh)
    got = to_np(y)[s].astype(np.float64)
    assert np.linalg.norm(got - y_ref) <= 1e-2 * np.linalg.norm(y_ref)
    assert cosine(got, y_ref) >= COS_TOL, cosine(got, y_ref)


@pytest.mark.parametrize("fmt", ["fp8", "mxfp4", "bf16"])
def test_prefill_bank_rows_up_to_the_limit(dev, fmt):
    """Banks of 511, 512 and 1023 rows, whose per-expert list fills the LDS beside
    the largest tiles: the same routes over fewer rows, in another tile, give the
    same bits."""
    H, I, k = 256, 384, 8
    rng = np.random.default_rng(7)
    bank = to_device_bank(synth.make_bank(fmt, 7, H, I, rng), dev)
    r = 330 if fmt == "bf16" else 130
    for rows in (511, 512, 1023):
        M = r * rows // k + 1
        g = torch.Generator(device=dev).manual_seed(rows)
        x = torch.randn((M, H), generator=g, device=dev).to(torch.bfloat16)
        w, ids = ops.route_softmax_topk(torch.randn((M, 16), generator=g, device=dev), k, True)
        ids += rows - 16  # the last rows of the bank: nothing lands on the others
        assert _block(fmt, M, k, rows, H, I) == 256
        y = ops.experts_prefill(x, w, ids, _bank_rows(bank, rows))
        # the same experts as rows 0 to 15 of a bank that puts the weights in the same places
        few = _bank_rows(bank, rows)
        few = ops.ExpertBank(few.fmt, *(t[rows - 16:].contiguous() if t is not None else None
                                        for t in (few.gate_up, few.down, few.gate_up_scale, few.down_scale)))
        h = 200  # so few tokens a call that it takes 64 or 128 routes per tile
        assert _block(fmt, h, k, 16, H, I) < 256
        part = ops.experts_prefill(x[:h].contiguous(), w[:h].contiguous(), (ids[:h] - (rows - 16)).contiguous(), few)
        assert torch.equal(y[:h], part), rows


@pytest.mark.parametrize("offset", [1, 2, 4])
@pytest.mark.parametrize("M", [1, 33])
def test_bf16_operands_at_any_element(dev, M, offset):
    """bf16 tokens and weights that start at any element of their allocation (2,
    4 and 8 bytes past a 16-byte line): the same bits as aligned ones."""
    E, H, I, k = 8, 512, 256, 2
    g = torch.Generator(device=dev).manual_seed(M)

    def at(t):
        buf = torch.zeros(t.numel() + offset, dtype=t.dtype, device=dev)
        buf[offset:] = t.reshape(-1)
        return buf[offset:].view(t.shape)

    gu = (torch.randn((E, 2 * I, H), generator=g, device=dev) * 0.05).to(torch.bfloat16)
    dn = (torch.randn((E, H, I), generator=g, device=dev) * 0.05).to(torch.bfloat16)
    x = torch.randn((M, H), generator=g, device=dev).to(torch.bfloat16)
    w, ids = ops.route_softmax_topk(torch.randn((M, E), generator=g, device=dev), k, True)
    for fn in (ops.experts_decode, ops.experts_prefill):
        y = fn(x, w, ids, ops.ExpertBank("bf16", gu, dn))
        assert torch.equal(y, fn(at(x), w, ids, ops.ExpertBank("bf16", at(gu), at(dn))))


def test_prefill_bf16_beyond_2gib(dev):
    """A bf16 call whose activations pass the 31-bit offsets of the LDS-DMA GEMM
    takes the register-staged one: equal to the same tokens in two calls that
    fit, within the rounding of bf16 sums taken in another order."""
    M, k, E, H, I = 60000, 8, 16, 128, 2048
    assert M * (k + 1) * I * 2 > 2**31 > M // 2 * (k + 1) * I * 2
    g = torch.Generator(device=dev).manual_seed(3)
    gu = (torch.randn((E, 2 * I, H), generator=g, device=dev) * 0.05).to(torch.bfloat16)
    dn = (torch.randn((E, H, I), generator=g, device=dev) * 0.02).to(torch.bfloat16)
    x = torch.randn((M, H), generator=g, device=dev).to(torch.bfloat16)
    w, ids = ops.route_softmax_topk(torch.randn((M, E), generator=g, device=dev), k, True)
    bank = ops.ExpertBank("bf16", gu, dn)
    y = ops.experts_prefill(x, w, ids, bank)
    h = M // 2
    halves = torch.cat([ops.experts_prefill(x[s].contiguous(), w[s].contiguous(), ids[s].contiguous(), bank)
                        for s in (slice(0, h), slice(h, M))])
    err = (y.double() - halves.double()).norm() / halves.double().norm()
    assert float(err) <= 4e-3  # one bf16 rounding (2^-9 relative) on each side


@pytest.mark.parametrize("fmt", ["fp8", "bf16"])
def test_prefill_token_of_route_many_choices(dev, fmt):
    """The token of a route (route / k) where k times the route index passes
    2^32: k = 4369 divides 2^32 - 1, so a rounded-up 32-bit reciprocal is one
    too large for the last choice of every token from 225 on.  Only the last
    choice has weight: the sums hold one term and equal a top-1 call's."""
    M, k, H, I = 320, 4369, 128, 128
    rng = np.random.default_rng(11)
    bank = to_device_bank(synth.make_bank(fmt, 4, H, I, rng), dev)
    x = bf16_dev(synth.activations(rng, M, H), dev)
    ids = torch.from_numpy(rng.integers(0, 4, size=(M, k)).astype(np.int32)).to(dev)
    w = torch.zeros((M, k), device=dev)
    w[:, -1] = 1.0
    y = ops.experts_prefill(x, w, ids, bank)
    y1 = ops.experts_prefill(x, w[:, -1:].contiguous(), ids[:, -1:].contiguous(), bank)
    assert torch.equal(y, y1)


def test_prefill_bf16_silu_is_the_decode_one(dev):
    """bf16 SwiGLU over gates of -88.5 to 88.5, where the reciprocal of
    1 + exp(-gate) passes from subnormal to 1: the products of every weight with
    a one or a zero are exact, so prefill and decode give the same bits, and the
    64-bit value within one bf16 rounding (8 significant bits: 2^-8) on top of
    the exponential's (its argument, up to 88, rounded to 24 bits)."""
    n, M = 1024, 12
    gate = torch.linspace(-88.5, 88.5, n).to(torch.bfloat16)
    gu = torch.zeros((1, 2 * n, n), dtype=torch.bfloat16)
    gu[0, :n, 0] = gate
    gu[0, n:, 1] = 1.0
    x = torch.zeros((M, n), dtype=torch.bfloat16)
    x[:, 0] = 1.0
    x[:, 1] = 2.0 ** torch.arange(0, 10 * M, 10)  # the up values: large enough for the smallest products to be normal
    bank = ops.ExpertBank("bf16", gu.to(dev), torch.eye(n, dtype=torch.bfloat16)[None].to(dev))
    args = (x.to(dev), torch.ones((M, 1), device=dev), torch.zeros((M, 1), dtype=torch.int32, device=dev), bank)
    y, yd = ops.experts_prefill(*args).cpu(), ops.experts_decode(*args).cpu()
    assert torch.equal(y, yd)
    g = gate.double()
    ref = (g / (1 + torch.exp(-g)))[None, :] * x[:, 1:2].double()
    seen = ref.abs() > 2.0 ** -120
    assert float(((y.double() - ref).abs() / ref.abs())[seen].max()) <= 2.0 ** -8 + 88.5 * 2.0 ** -23
