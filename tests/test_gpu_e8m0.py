"""F4: experts of the E8M0 block-32 contract (W4A8 routed, W8A8 32x32-block shared expert) in exact arithmetic, through
the C ABI, bit-equal to the oracle's restatement of kernels/q38_contract.cuh:53-101,153-170 and
kernels/moe_ffn.cu:601-700 (pinned on the CPU against rational arithmetic and closed forms)."""
import numpy as np
import pytest
import torch

import oracle as orc
from flyingfish_amd import capi, synth
from flyingfish_amd.ops import E8m0DecodeOps, ExpertTable, PrefillOps
from helpers import assert_close_with_rare_outliers, assert_close_bf16, bits

pytestmark = pytest.mark.gpu
# Values behind two composed stages (end to end) or behind a twice-rounded product (activations of the matrix-core paths):
# the per-stage bars are 2 steps; here the relative-L2 bar holds on the tensor, no element lies beyond a loose bound, and
# the share of elements beyond 2 steps must stay below these (small shapes: a cancelled output behind one activation that
# rounded the other way moves by several of its own steps).
E2E_RARE = 5e-3
ACT_RARE = 2e-3
DEV = "cuda"


def rand_bf16(shape, std, seed):
    return synth.normal(shape, std, seed).to(torch.bfloat16)


def _tables(experts, hidden, inter, shared_inter, seed):
    routed = ExpertTable.allocate(capi.FMT_E2M1_E8M0, experts, hidden, inter, DEV)
    ref = []
    for e in range(experts):
        v = routed.expert_views(e)
        mats = []
        for i, shape in enumerate([(inter, hidden), (inter, hidden), (hidden, inter)]):
            codes, scales = synth.quant_e2m1_e8m0(synth.normal(shape, 0.05, seed * 1000 + e * 3 + i))
            v[2 * i].copy_(codes); v[2 * i + 1].copy_(scales)
            mats += [codes.numpy(), scales.numpy()]
        ref.append(mats)
    sh_table = ExpertTable.allocate(capi.FMT_E4M3_E8M0_32, 1, hidden, shared_inter, DEV)
    v = sh_table.expert_views(0)
    sh_ref = []
    for i, shape in enumerate([(shared_inter, hidden), (shared_inter, hidden), (hidden, shared_inter)]):
        codes, scales = synth.quant_e4m3_e8m0_block32(synth.normal(shape, 0.05, seed * 1000 + 900 + i))
        v[2 * i].copy_(codes); v[2 * i + 1].copy_(scales)
        sh_ref += [codes.numpy(), scales.numpy()]
    return routed, ref, sh_table, sh_ref


def test_act_quant_e8m0_bit_exact():
    x = (synth.normal((5, 256), 1.0, 3) * torch.exp(synth.normal((5, 1), 3.0, 4))).to(torch.bfloat16)
    x[2, 32:64] = 0  # an all-zero group takes the amax floor
    codes, scales = E8m0DecodeOps.act_quant(x.to(DEV))
    torch.cuda.synchronize()
    oc, os_ = orc.act_quant_e8m0(bits(x))
    assert np.array_equal(codes.cpu().numpy(), oc) and np.array_equal(scales.cpu().numpy(), os_)


@pytest.mark.parametrize("hidden,inter,shared_inter,rows,top_k", [(256, 128, 128, 1, 2), (512, 256, 384, 3, 3), (1024, 512, 512, 2, 4)])
def test_e8m0_experts_bit_exact(hidden, inter, shared_inter, rows, top_k):
    experts, limit = 6, 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, shared_inter, 41 + rows)
    sh = sh_table.shared_struct(0)
    x = rand_bf16((rows, hidden), 1.0, 5 + rows)
    g = synth.generator(6 + rows)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(rows)]).to(torch.int32)
    wt = torch.rand((rows, top_k), generator=g) * 0.5 + 0.05
    active = torch.ones((rows, top_k), dtype=torch.int32)
    if rows > 1:
        active[1, 0] = 0
    op = E8m0DecodeOps(routed, sh, rows, top_k, limit)
    op.contributions.zero_()
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV), active.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    for r in range(rows):
        for c in range(top_k):
            if not active[r, c]:
                assert not got[r, c].any()
                continue
            want = orc.expert_ffn_e8m0(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))
            assert np.array_equal(got[r, c], want), (r, c)
        assert np.array_equal(got_sh[r], orc.expert_ffn_e8m0(0, xb[r], *sh_ref, limit, 1.0)), r
    assert np.array_equal(op.done.cpu().numpy(), active.numpy())


@pytest.mark.parametrize("seed", range(10))
@pytest.mark.parametrize("exact", [True, False])
def test_e8m0_experts_seeded_sweep(seed, exact):
    """Bit equality at widths the fixed cases do not visit (any multiple of 32 from 64 to 1024, shared expert of another
    width, 1..5 rows, 1..6 choices, activations scaled over several binades), in the exact arithmetic and in the
    FP32-chain variant."""
    rng = np.random.default_rng(8000 + seed)
    hidden = 32 * int(rng.integers(2, 33))
    inter = 32 * int(rng.integers(2, 17))
    shared_inter = 32 * int(rng.integers(2, 17))
    experts = int(rng.integers(2, 8))
    top_k = int(rng.integers(1, min(6, experts) + 1))
    rows = int(rng.choice([1, 2, 5]))
    limit = float(rng.choice([0.5, 7.0]))
    print("hidden=%d inter=%d shared_inter=%d experts=%d top_k=%d rows=%d limit=%g exact=%d" %
          (hidden, inter, shared_inter, experts, top_k, rows, limit, exact), flush=True)
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, shared_inter, 8100 + seed)
    x = (synth.normal((rows, hidden), 1.0, 8200 + seed) * float(rng.choice([0.01, 1.0, 30.0]))).to(torch.bfloat16)
    g = synth.generator(8300 + seed)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(rows)]).to(torch.int32)
    wt = torch.rand((rows, top_k), generator=g) * 0.5 + 0.05
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), rows, top_k, limit, exact=exact)
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    ffn = orc.expert_ffn_e8m0 if exact else orc.expert_ffn_e8m0_f32
    for r in range(rows):
        for c in range(top_k):
            assert np.array_equal(got[r, c], ffn(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))), (r, c)
        assert np.array_equal(got_sh[r], ffn(0, xb[r], *sh_ref, limit, 1.0)), r


def _down_exact(packed, act_bits, down, sdown):
    """The contract's down projection of one BF16 activation row: quantize per 32, exact dots, BF16."""
    hq, hs = orc.act_quant_e8m0(act_bits[None, :])
    return np.array([orc.scaled_dot_exact(packed, down[d], sdown[d] if packed else sdown[d // 32], hq[0], hs[0])[1]
                     for d in range(down.shape[0])], dtype=np.uint16)


@pytest.mark.parametrize("rows,top_k,experts,hidden,inter,shared_inter", [(40, 3, 6, 256, 128, 128), (130, 2, 3, 384, 256, 128), (5, 4, 9, 128, 128, 256)])
def test_e8m0_prefill_on_the_mx_matrix_cores(rows, top_k, experts, hidden, inter, shared_inter):
    """Cohorts of the W4A8 / W8A8 contract through ffmoe_prefill_contribute: the same quantized operands and stage
    boundaries as the exact decode entry, the dots on v_mfma_scale_f32_16x16x128_f8f6f4 (block scales applied by the
    matrix core, FP32 accumulation in its own order). Checked per stage against the exact oracle: activations, then the
    down projection of the device's own activations."""
    limit = 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, shared_inter, 500 + rows)
    x = rand_bf16((rows, hidden), 1.0, 510 + rows)
    g = synth.generator(520 + rows)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(rows)]).to(torch.int32)
    wt = torch.rand((rows, top_k), generator=g) * 0.5 + 0.05
    active = torch.ones((rows, top_k), dtype=torch.int32)
    active[1, 0] = 0
    op = PrefillOps(routed, rows, top_k, swiglu=capi.SWIGLU_CLAMPED_ONCE, swiglu_limit=limit, routed_weight=capi.WEIGHT_BEFORE_DOWN_F32,
                    weights_f32=True, shared=sh_table.shared_struct(0), act_mode=capi.ACT_E4M3_E8M0_32)
    op.contributions.zero_()
    got = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV), active=active.to(DEV))
    torch.cuda.synchronize()
    assert np.array_equal(op.done.cpu().numpy() != 0, active.numpy() != 0)
    v = op.scratch_views()
    n_live = int(active.sum())
    assert int(v["totals"][3].item()) == n_live
    perm = v["perm"].cpu().numpy()[:n_live]
    act = bits(v["act"])[:n_live]
    g2 = bits(got).reshape(rows * top_k, -1)
    xb = bits(x)
    flat_ids, flat_w = ids.reshape(-1).numpy(), wt.reshape(-1).numpy()
    want_act = np.zeros_like(act)
    want_down = np.zeros((n_live, hidden), dtype=np.uint16)
    want_full = np.zeros((n_live, hidden), dtype=np.uint16)
    for pos, a in enumerate(perm):
        m = ref[int(flat_ids[a])]
        want_full[pos], want_act[pos] = orc.expert_ffn_e8m0(1, xb[a // top_k], *m, limit, float(flat_w[a]), return_act=True)
        want_down[pos] = _down_exact(1, act[pos], m[4], m[5])
    assert_close_with_rare_outliers(act, want_act, "activations", loose=3, rare=ACT_RARE)
    assert_close_bf16(g2[perm], want_down, "down projection of the device activations")
    assert orc.rel_l2(g2[perm], want_full) <= 5e-2
    assert not g2[np.flatnonzero(active.reshape(-1).numpy() == 0)].any()
    so, sh_act = bits(op.shared_out), bits(v["sh_act"])
    want_sa = np.zeros_like(sh_act)
    want_sd = np.zeros_like(so)
    for r in range(rows):
        want_sa[r] = orc.expert_ffn_e8m0(0, xb[r], *sh_ref, limit, 1.0, return_act=True)[1]
        want_sd[r] = _down_exact(0, sh_act[r], sh_ref[4], sh_ref[5])
    assert_close_with_rare_outliers(sh_act, want_sa, "shared activations", loose=3, rare=ACT_RARE)
    assert_close_bf16(so, want_sd, "shared down projection of the device activations")


@pytest.mark.parametrize("rows,hidden,shared_inter", [(3, 128, 128), (65, 384, 256), (200, 256, 384), (300, 1280, 128)])
def test_e8m0_shared_expert_tile_kernel_equals_the_row_group_kernel_bitwise(rows, hidden, shared_inter, monkeypatch):
    routed, _, sh_table, _ = _tables(2, hidden, 128, shared_inter, 700 + rows)
    x = rand_bf16((rows, hidden), 1.0, 710 + rows).to(DEV)
    ids = torch.zeros((rows, 1), dtype=torch.int32, device=DEV)
    wt = torch.ones((rows, 1), device=DEV)
    out = []
    for switch in ("0", "1"):
        monkeypatch.setenv("FFMOE_W8A8_TILE", switch)
        op = PrefillOps(routed, rows, 1, swiglu=capi.SWIGLU_CLAMPED_ONCE, swiglu_limit=7.0, routed_weight=capi.WEIGHT_BEFORE_DOWN_F32, weights_f32=True,
                        shared=sh_table.shared_struct(0), act_mode=capi.ACT_E4M3_E8M0_32)
        op.contribute(x, ids, wt)
        torch.cuda.synchronize()
        out.append(op.shared_out.clone())
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("rows,hidden,inter", [(16, 128, 384), (33, 1280, 128), (65, 384, 640), (150, 768, 256)])
def test_e8m0_prefill_rows_do_not_depend_on_their_group_bitwise(rows, hidden, inter):
    """Groups of one to 64 rows, contractions of one to five stages with and without a last half, columns past the end of a
    tile: every row equals itself in a cohort of its own."""
    routed, _, _, _ = _tables(4, hidden, inter, 128, 800 + rows)
    x = rand_bf16((rows, hidden), 1.0, 810 + rows).to(DEV)
    g = synth.generator(820 + rows)
    ids = torch.stack([torch.multinomial(torch.tensor([0.6, 0.3, 0.07, 0.03]), 2, generator=g) for _ in range(rows)]).to(torch.int32).to(DEV)
    wt = (torch.rand((rows, 2), generator=g) * 0.5 + 0.05).to(DEV)

    def op(n):
        return PrefillOps(routed, n, 2, swiglu=capi.SWIGLU_CLAMPED_ONCE, swiglu_limit=7.0, routed_weight=capi.WEIGHT_BEFORE_DOWN_F32, weights_f32=True,
                          act_mode=capi.ACT_E4M3_E8M0_32)
    whole = op(rows)
    got = whole.contribute(x, ids, wt)
    one = op(1)
    want = torch.stack([one.contribute(x[r:r + 1], ids[r:r + 1], wt[r:r + 1])[0].clone() for r in range(rows)])
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert int(whole.done.min()) == 1


def test_e8m0_entry_checks_its_contract():
    routed, _, sh_table, _ = _tables(2, 64, 32, 32, 9)
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), 1, 1, 7.0)
    op.limit = 0.0  # the contract clamps: a limit is required
    x = rand_bf16((1, 64), 1.0, 1).to(DEV)
    ids = torch.zeros((1, 1), dtype=torch.int32, device=DEV)
    with pytest.raises(capi.FfmoeError):
        op.contribute(x, ids, torch.ones((1, 1), device=DEV))


def test_e8m0_rows_whose_scales_span_many_binades_take_the_ordered_path():
    """Block scales spread over ~100 binades: partial sums round, so only the reference's group order gives its bits."""
    experts, hidden, inter, rows, top_k, limit = 3, 256, 128, 2, 2, 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, inter, 77)
    g = synth.generator(78)
    for e in range(experts):
        v = routed.expert_views(e)
        for i in (1, 3, 5):
            wild = torch.randint(70, 175, v[i].shape, generator=g, dtype=torch.uint8)
            v[i].copy_(wild)
            ref[e][i] = wild.numpy()
    v = sh_table.expert_views(0)
    for i in (1, 3, 5):
        wild = torch.randint(90, 150, v[i].shape, generator=g, dtype=torch.uint8)
        v[i].copy_(wild)
        sh_ref[i] = wild.numpy()
    x = rand_bf16((rows, hidden), 1.0, 79)
    ids = torch.tensor([[0, 2], [1, 0]], dtype=torch.int32)
    wt = torch.tensor([[0.3, 0.2], [0.4, 0.1]])
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), rows, top_k, limit)
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    for r in range(rows):
        for c in range(top_k):
            assert np.array_equal(got[r, c], orc.expert_ffn_e8m0(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))), (r, c)
        assert np.array_equal(got_sh[r], orc.expert_ffn_e8m0(0, xb[r], *sh_ref, limit, 1.0)), r


@pytest.mark.parametrize("hidden,inter,shared_inter,rows,top_k", [(256, 128, 128, 1, 2), (1024, 512, 384, 3, 3)])
def test_e8m0_fp32_chain_variant_bit_exact(hidden, inter, shared_inter, rows, top_k):
    """act_mode FFMOE_ACT_E4M3_E8M0_32_F32: the reference's 32-lane FP32 kernels, reproduced lane for lane."""
    experts, limit = 5, 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, shared_inter, 141 + rows)
    x = rand_bf16((rows, hidden), 1.0, 15 + rows)
    g = synth.generator(16 + rows)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(rows)]).to(torch.int32)
    wt = torch.rand((rows, top_k), generator=g) * 0.5 + 0.05
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), rows, top_k, limit, exact=False)
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    for r in range(rows):
        for c in range(top_k):
            want = orc.expert_ffn_e8m0_f32(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))
            assert np.array_equal(got[r, c], want), (r, c)
        assert np.array_equal(got_sh[r], orc.expert_ffn_e8m0_f32(0, xb[r], *sh_ref, limit, 1.0)), r
    assert np.all(op.done.cpu().numpy() == 1)


@pytest.mark.parametrize("hidden,inter,shared_inter,rows,top_k", [
    (128, 128, 128, 1, 1),    # one K block: waves without work, half a line of codes per row
    (384, 128, 256, 2, 2),    # an odd number of K blocks, two tokens per instruction
    (256, 640, 128, 5, 3),    # a ragged last block of output columns, an unpaired token
    (1152, 384, 640, 1, 6),
    (2304, 896, 384, 3, 2),
])
def test_e8m0_matrix_core_tiles_bit_exact_on_any_code(hidden, inter, shared_inter, rows, top_k):
    """The matrix-core kernels of the exact arithmetic at the edges of their tiles, on weight codes drawn uniformly (every E2M1
    nibble, both zeros; every finite E4M3 code, so products over the whole exponent range) and on activations whose groups
    mix the largest with the smallest E4M3 magnitudes, some groups all zero. The outputs are BF16 behind a SwiGLU, so a lost last bit
    shows only beside a tie here; test_e8m0_sums_that_cancel_to_their_last_bit isolates it."""
    rng = np.random.default_rng(9000 + hidden + rows)
    experts, limit = max(6, top_k), 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, shared_inter, 9100 + rows)
    for e in range(experts):
        v = routed.expert_views(e)
        for i in range(3):
            codes = rng.integers(0, 256, tuple(v[2 * i].shape), dtype=np.uint8)
            scales = rng.integers(116, 122, tuple(v[2 * i + 1].shape), dtype=np.uint8)
            codes[0, :16] = 0  # an all-zero group with a scale of its own
            scales[0, 0] = 3
            v[2 * i].copy_(torch.from_numpy(codes)); v[2 * i + 1].copy_(torch.from_numpy(scales))
            ref[e][2 * i], ref[e][2 * i + 1] = codes, scales
    v = sh_table.expert_views(0)
    for i in range(3):
        codes = rng.integers(0, 256, tuple(v[2 * i].shape), dtype=np.uint8)
        codes[(codes & 127) == 127] = 0x7e
        scales = rng.integers(108, 111, tuple(v[2 * i + 1].shape), dtype=np.uint8)
        v[2 * i].copy_(torch.from_numpy(codes)); v[2 * i + 1].copy_(torch.from_numpy(scales))
        sh_ref[2 * i], sh_ref[2 * i + 1] = codes, scales
    mag = np.exp2(rng.uniform(-16, 0, (rows, hidden))) * rng.choice([-1.0, 1.0], (rows, hidden))
    mag[:, ::32] = 1.0
    mag[0, 32:64] = 0.0
    x = torch.from_numpy(mag.astype(np.float32)).to(torch.bfloat16)
    ids = torch.from_numpy(np.stack([rng.permutation(experts)[:top_k] for _ in range(rows)]).astype(np.int32))
    wt = torch.from_numpy(rng.uniform(0.05, 0.5, (rows, top_k)).astype(np.float32))
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), rows, top_k, limit)
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    for r in range(rows):
        for c in range(top_k):
            assert np.array_equal(got[r, c], orc.expert_ffn_e8m0(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))), (r, c)
        assert np.array_equal(got_sh[r], orc.expert_ffn_e8m0(0, xb[r], *sh_ref, limit, 1.0)), r
    assert np.all(op.done.cpu().numpy() == 1)


def _single_expert(hidden, inter, codes, scales):
    """A table of one routed expert with these six tensors, gate codes, gate scales, up .., down .."""
    routed = ExpertTable.allocate(capi.FMT_E2M1_E8M0, 1, hidden, inter, DEV)
    for v, a in zip(routed.expert_views(0), [t for pair in zip(codes, scales) for t in pair]):
        v.copy_(torch.from_numpy(a))
    return routed


def _pack(nibbles):
    """[.., K] E2M1 nibbles to [.., K / 2] codes, low nibble first."""
    return (nibbles[..., 0::2] | (nibbles[..., 1::2] << 4)).astype(np.uint8)


def _one_choice(routed, x, weight=1.0, shared=None):
    rows = x.shape[0]
    op = E8m0DecodeOps(routed, shared, rows, 1, 7.0)
    ids = torch.zeros((rows, 1), dtype=torch.int32, device=DEV)
    contrib, shared_out = op.contribute(x.to(DEV), ids, torch.full((rows, 1), weight, device=DEV))
    torch.cuda.synchronize()
    return bits(contrib)[:, 0], None if shared is None else bits(shared_out)


def _identity_down(n):
    """Down projection that hands the (quantized) activations through: 1.0 on the diagonal."""
    return _pack(2 * np.eye(n, dtype=np.uint8)), np.full((n, n // 32), 127, dtype=np.uint8)


def test_e8m0_group_sums_at_the_ends_of_the_fp32_range():
    """Two groups of 32 x 448 x 6.0 x 2^(code sum - 254) that cancel, or nearly do: from a code sum of 366 on one alone is
    beyond FP32, while the contract's FP64 total is 0 or an ordinary multiple. Row j has weight scale 358 - 239 + j / 4 on a
    token whose scale codes are 239; every second pair of rows leaves one product standing. Below, small sums: FP32 results
    around the smallest normal number, which a large routing weight brings back to the output."""
    n = 128
    for xexp, first, weight in ((112, 119, 1.0), (-14, 0, 2.0 ** 120)):  # token codes 239 and 113; sums 358 .. 389 and 113 .. 144
        x = np.zeros((3, n), dtype=np.float32)
        x[:, :32] = 448.0
        x[:, 32:64] = -448.0
        xb = torch.from_numpy(x * np.float32(2.0 ** xexp)).to(torch.bfloat16)
        up = np.zeros((n, n), dtype=np.uint8)
        up[:, :64] = 7  # 6.0
        up[2::4, 5] = 6   # one product of the pair stands: negative
        up[3::4, 40] = 6  # positive
        gate = np.zeros((n, n), dtype=np.uint8)
        gate[:, :32] = 7
        sup = np.repeat((first + np.arange(n) // 4).astype(np.uint8)[:, None], n // 32, 1)
        sgate = np.full((n, n // 32), 127, dtype=np.uint8)
        down, sdown = _identity_down(n)
        m = [_pack(gate), sgate, _pack(up), sup, down, sdown]
        got, _ = _one_choice(_single_expert(n, n, m[0::2], m[1::2]), xb, weight)
        for r in range(3):
            want = orc.expert_ffn_e8m0(1, bits(xb)[r], *m, 7.0, weight)
            assert np.array_equal(got[r], want), (xexp, r, np.flatnonzero(got[r] != want))


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("code", [253, 254, 255])
def test_e8m0_all_zero_group_adds_nothing_whatever_its_scale(code, rows):
    """A weight group of zeros (of both signs) under the largest scales, and under the reserved code, on ordinary and on huge
    activations: the result is that of any other scale."""
    n = 128
    rng = np.random.default_rng(code + rows)
    _, ref, _, _ = _tables(1, n, n, n, 600)
    m = [a.copy() for a in ref[0]]
    for i in range(3):
        m[2 * i][:, 16:32] = rng.choice(np.array([0x00, 0x08, 0x80, 0x88], dtype=np.uint8), (n, 16))
        m[2 * i + 1][:, 1] = 100
    x = rand_bf16((rows, n), 1.0, 601)
    x[1:, 32:64] *= 2.0 ** 119
    plain, _ = _one_choice(_single_expert(n, n, m[0::2], m[1::2]), x)
    for r in range(rows):
        assert np.array_equal(plain[r], orc.expert_ffn_e8m0(1, bits(x)[r], *m, 7.0, 1.0))
    for i in range(3):
        m[2 * i + 1][:, 1] = code
    got, _ = _one_choice(_single_expert(n, n, m[0::2], m[1::2]), x)
    assert np.array_equal(got, plain)


def test_e8m0_call_larger_than_one_grid_dimension_bitwise():
    """65535 rows, the most the entry takes, whose blocks hold more threads than one dimension of a launch counts: equal to the
    same rows in four calls."""
    hidden, inter, rows, top_k = 128, 512, 65535, 8
    routed, _, sh_table, _ = _tables(16, hidden, inter, inter, 660)
    sh = sh_table.shared_struct(0)
    x = synth.normal((rows, hidden), 1.0, 661, device=DEV).to(torch.bfloat16)
    ids = torch.stack([torch.arange(rows, device=DEV) % 9 + c for c in range(top_k)], 1).to(torch.int32)
    wt = torch.linspace(0.05, 0.5, rows * top_k, device=DEV).view(rows, top_k)
    op = E8m0DecodeOps(routed, sh, rows, top_k, 7.0)
    contrib, shared_out = op.contribute(x, ids, wt)
    part = 16384
    for r0 in range(0, rows, part):
        n = min(part, rows - r0)
        few = E8m0DecodeOps(routed, sh, n, top_k, 7.0)
        c, s = few.contribute(x[r0:r0 + n].contiguous(), ids[r0:r0 + n].contiguous(), wt[r0:r0 + n].contiguous())
        assert torch.equal(c.view(torch.int16), contrib[r0:r0 + n].view(torch.int16)), r0
        assert torch.equal(s.view(torch.int16), shared_out[r0:r0 + n].view(torch.int16)), r0
    assert int(op.done.min()) == 1


@pytest.mark.parametrize("rows,hidden,inter", [(9, 384, 256), (150, 640, 128)])
def test_e8m0_prefill_takes_scales_at_any_address_bitwise(rows, hidden, inter):
    """Scale bytes that start anywhere: the slots of a table promise 16-byte alignment of the codes only."""
    routed, _, sh_table, _ = _tables(3, hidden, inter, 128, 680 + rows)
    x = rand_bf16((rows, hidden), 1.0, 681).to(DEV)
    g = synth.generator(682)
    ids = torch.stack([torch.multinomial(torch.tensor([0.7, 0.2, 0.1]), 2, generator=g) for _ in range(rows)]).to(torch.int32).to(DEV)
    wt = (torch.rand((rows, 2), generator=g) * 0.5 + 0.05).to(DEV)
    moved = [[torch.empty(v.numel() + 16, dtype=torch.uint8, device=DEV) for v in routed.expert_views(e)[1::2]] for e in range(3)]
    out = []
    for shift in (0, 1, 2, 3, 4):
        slots = routed.slots.tolist()
        for e in range(3):
            for i, (v, m) in enumerate(zip(routed.expert_views(e)[1::2], moved[e])):
                m[shift:shift + v.numel()].copy_(v.reshape(-1))
                slots[e][2 * i + 1] = m.data_ptr() + shift
        table = ExpertTable(routed.format, 3, hidden, inter, routed.storage, torch.tensor(slots, dtype=torch.int64, device=DEV), None)
        op = PrefillOps(table, rows, 2, swiglu=capi.SWIGLU_CLAMPED_ONCE, swiglu_limit=7.0, routed_weight=capi.WEIGHT_BEFORE_DOWN_F32, weights_f32=True,
                        act_mode=capi.ACT_E4M3_E8M0_32)
        op.contribute(x, ids, wt)
        torch.cuda.synchronize()
        out.append(bits(op.contributions))
    assert out[0].any()
    for shift in range(1, 5):
        assert np.array_equal(out[shift], out[0]), shift


@pytest.mark.parametrize("hidden,inter,rows,top_k", [
    (128, 128, 2, 3), (384, 256, 5, 3), (640, 384, 9, 2),
    (7168, 128, 3, 1),   # two tokens' planes beyond 64 KB of LDS
    (7680, 128, 2, 2),   # the longest rows that pair
    (7936, 128, 3, 1),   # one token at a time: two do not leave room for a second block
    (15872, 128, 2, 1),  # the longest rows the entry takes
    (128, 128, 700, 6),  # more assignments than the grouping launch holds
])
@pytest.mark.parametrize("pairs", ["0", "1"])
def test_e8m0_launch_regimes_bit_exact(hidden, inter, rows, top_k, pairs, monkeypatch):
    """Rows one at a time and in pairs, at the lengths where the one takes over from the other."""
    monkeypatch.setenv("FFMOE_E8M0_PAIRS", pairs)
    experts, limit = 7, 7.0
    routed, ref, sh_table, sh_ref = _tables(experts, hidden, inter, inter, 650 + rows)
    x = rand_bf16((rows, hidden), 1.0, 651)
    g = synth.generator(652)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(rows)]).to(torch.int32)
    wt = torch.rand((rows, top_k), generator=g) * 0.5 + 0.05
    op = E8m0DecodeOps(routed, sh_table.shared_struct(0), rows, top_k, limit)
    contrib, shared_out = op.contribute(x.to(DEV), ids.to(DEV), wt.to(DEV))
    torch.cuda.synchronize()
    got, got_sh, xb = bits(contrib), bits(shared_out), bits(x)
    for r in range(0, rows, max(1, rows // 20)):
        for c in range(top_k):
            assert np.array_equal(got[r, c], orc.expert_ffn_e8m0(1, xb[r], *ref[int(ids[r, c])], limit, float(wt[r, c]))), (r, c)
        assert np.array_equal(got_sh[r], orc.expert_ffn_e8m0(0, xb[r], *sh_ref, limit, 1.0)), r
    assert np.all(op.done.cpu().numpy() == 1)


_E4M3_INT = np.array([0 if c & 127 == 127 else ((8 + (c & 7)) << ((c >> 3 & 15) - 1) if c & 0x78 else c & 7) * (-1 if c & 128 else 1) for c in range(256)], dtype=np.int64)
_E2M1_INT = np.array([0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12], dtype=np.int64)


@pytest.mark.parametrize("pairs", ["0", "1"])
@pytest.mark.parametrize("weights", ["routed", "shared, small codes", "shared, large codes"])
@pytest.mark.parametrize("low,high", [(1, 240), (1, 960), (9 << 5, 15 << 9), (9 << 7, 14 << 14), (9 << 10, 14 << 14)])
def test_e8m0_sums_that_cancel_to_their_last_bit(weights, low, high, pairs, monkeypatch):
    """Every dot is one smallest product of an exponent class (9 or 1 units times 1 or 3, or 9 or 11) beside large ones that cancel
    exactly, anywhere in their group of 32 or (odd rows, sums of one sign) against the next group: a single bit lost from a
    product or a sum changes the result outright. The parameters are the smallest and largest activation in units of 2^-9: the
    exponent classes of the routed experts' tokens (bit 6 of the code) and of the shared expert's (0 .. 5, 6 .. 10, 11 .. 15). Three
    rows, the second with every sign but the gate's turned, one at a time and two per instruction."""
    monkeypatch.setenv("FFMOE_E8M0_PAIRS", pairs)
    n = 128
    packed = weights == "routed"
    rng = np.random.default_rng(low + high + len(weights))
    table = _E2M1_INT if packed else _E4M3_INT
    code_of = {int(table[c]): c for c in reversed(range(len(table)))}
    large, small = ([12, 8, 6], [1, 3]) if packed else ([960, 480, 832], [1, 3]) if "small" in weights else ([14 << 14, 15 << 13, 9 << 14], [9 << 7, 11 << 7])
    ints = np.unique(np.abs(_E4M3_INT))
    # groups 0 and 1: 448, which gives the group scale 1 and meets a zero weight, 26 large values in pairs, 5 small ones, the same
    # magnitudes in both groups; group 2: 448, for the gate
    pairs = np.repeat(rng.choice(ints[(ints >= high // 2) & (ints <= high)], 13), 2)
    av, kind = np.zeros(n, dtype=np.int64), np.zeros(n, dtype=np.int64)  # kind: 0 zero weight, 1 .. 13 a pair, 14 small
    for g in (0, 32):
        order = rng.permutation(32)
        av[g:g + 32] = (np.concatenate([[448 << 9], pairs, [low] * 5]) * rng.choice([-1, 1], 32))[order]
        kind[g:g + 32] = np.concatenate([[0], np.repeat(np.arange(13) + 1, 2), [14] * 5])[order]
    av[64] = 448 << 9
    turn = np.where(np.arange(n) == 64, 1, -1)
    x = torch.from_numpy((np.stack([av, av * turn, av]) * 2.0 ** -9).astype(np.float32)).to(torch.bfloat16)
    codes, scales = orc.act_quant_e8m0(bits(x))
    assert np.array_equal(_E4M3_INT[codes[0]], av) and np.all(scales[0, :3] == 127)
    sign = np.sign(av)
    w = np.zeros((n, n), dtype=np.int64)
    for j in range(n):
        if j % 2:
            v = large[j // 2 % 3]
            w[j, :64] = np.where((kind[:64] > 0) & (kind[:64] < 14), v * sign[:64], 0)
            w[j, 32:64] *= -1
        else:
            for i in range(1, 14):
                a, b = np.flatnonzero(kind[:32] == i)
                v = int(rng.choice(large)) * int(rng.choice([-1, 1]))
                w[j, a], w[j, b] = v * sign[a], -v * sign[b]
        w[j, rng.choice(np.flatnonzero(kind[:32] == 14))] = int(rng.choice(small)) * int(rng.choice([-1, 1]))
    total = w @ av
    assert np.all(total != 0) and np.abs(total).max() <= 11 * low * max(small)
    shift = int(np.floor(np.log2(float(np.abs(total).max()) * 2.0 ** (-10 if packed else -18))))  # the largest total lies between 1 and 2
    up = np.vectorize(lambda v: code_of[int(v)], otypes=[np.uint8])(w)
    gate = np.zeros((n, n), dtype=np.uint8)
    gate[:, 64] = code_of[12 if packed else 960]
    if packed:
        down, sdown = _identity_down(n)
        m = [_pack(gate), np.full((n, n // 32), 120, dtype=np.uint8), _pack(up), np.full((n, n // 32), 127 - shift, dtype=np.uint8), down, sdown]
        got, _ = _one_choice(_single_expert(n, n, m[0::2], m[1::2]), x)
    else:
        blocks = lambda c: np.full((n // 32, n // 32), c, dtype=np.uint8)
        m = [gate, blocks(120), up, blocks(127 - shift), (0x38 * np.eye(n)).astype(np.uint8), blocks(127)]
        routed, _, sh_table, _ = _tables(1, n, n, n, 900)
        for v, a in zip(sh_table.expert_views(0), m):
            v.copy_(torch.from_numpy(a))
        _, got = _one_choice(routed, x, shared=sh_table.shared_struct(0))
    for r in range(3):
        want = orc.expert_ffn_e8m0(packed, bits(x)[r], *m, 7.0, 1.0)
        assert np.count_nonzero(want & 0x7fff) == n  # every total survives to the output
        assert np.array_equal(got[r], want), (r, np.flatnonzero(got[r] != want))


@pytest.mark.parametrize("up", [0, 6, 8, 14, 30])
def test_e8m0_activations_over_many_binades_bit_exact(up):
    """Group scales from the quantizer's floor up to 2^`up` times an ordinary token's: FP64 sums of any order, or the ordered chain
    where those would round. Up to 25 binades, which tokens with near-silent and with outlying channels reach, a call takes about
    as long as any other (the ordered chain is a hundred times slower)."""
    experts, hidden, inter, rows = 2, 7168, 256, 2
    routed, ref, _, _ = _tables(experts, hidden, inter, inter, 690)
    rng = np.random.default_rng(691 + up)
    f = np.exp2(up - rng.uniform(0, up + 14, (rows, hidden // 32, 1)))
    f[:, 0], f[:, 1] = 2.0 ** up, 2.0 ** -14
    x = torch.from_numpy((rng.standard_normal((rows, hidden // 32, 32)) * f).reshape(rows, hidden).astype(np.float32)).to(torch.bfloat16)
    _, scales = orc.act_quant_e8m0(bits(x))
    assert np.all(scales.max(1).astype(int) - scales.min(1) >= up + 14)
    op = E8m0DecodeOps(routed, None, rows, 1, 7.0)
    ids, wt = torch.tensor([[0], [1]], dtype=torch.int32, device=DEV), torch.ones((rows, 1), device=DEV)

    def us(x):
        op.contribute(x, ids, wt)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(20):
            op.contribute(x, ids, wt)
        b.record()
        b.synchronize()
        return a.elapsed_time(b) * 50
    plain = us(rand_bf16((rows, hidden), 1.0, 692).to(DEV))
    wide = us(x.to(DEV))
    got = bits(op.contributions)[:, 0]
    for r in range(rows):
        assert np.array_equal(got[r], orc.expert_ffn_e8m0(1, bits(x)[r], *ref[r], 7.0, 1.0)), r
    print("up=%d: %.1f us against %.1f" % (up, wide, plain))
    if up <= 8:
        assert wide < 8 * plain
