"""Fused dense-stack forward on the GPU (through the C ABI) against the NumPy oracle.
Bar: policy within a relative Frobenius error of 3e-3 of the f32 oracle evaluated on the rounded
inputs; sampled actions bit-exact given the kernel's own policy and the same uniforms."""
import numpy as np
import pytest
import torch

from oracle import gemm as ogemm, layers as olayers, row_ops as orow
from gpu_util import announce, dev, host

pytestmark = pytest.mark.gpu

TORCH = {"f16": torch.float16, "bf16": torch.bfloat16}
HEAD_CODE = {"softmax": olayers.HEAD_SOFTMAX, "regret_matching": olayers.HEAD_REGRET_MATCHING,
             "softmax_regret_matching": olayers.HEAD_SOFTMAX_RM, None: olayers.HEAD_NONE}


@pytest.fixture(scope="module")
def LY():
    from ml import layers
    return layers


def make_problem(rng, batch, dims, dtype):
    x = (rng.random((batch, dims[0])) < 0.2).astype(np.float32)
    ws = [ogemm.round_to(olayers.weight_init(rng, o, i), dtype) for i, o in zip(dims[:-1], dims[1:])]
    u = (1 - rng.random(batch, dtype=np.float32)).astype(np.float32)
    return x, ws, u


def check(LY, x, ws, u, dtype, head="softmax_regret_matching", mask=0, biases=None, packed=False):
    t = TORCH[dtype]
    bd = None if biases is None else [dev(b) if b is not None else None for b in biases]
    wd = [dev(w, t) for w in ws]
    pk = None
    if packed:
        pk = LY.pack_weights(wd)
        assert pk is not None and pk.buffer.numel() == LY.packed_bytes([x.shape[1]] + [w.shape[0] for w in ws])
    policy, action, logits = LY.mlp_forward(dev(x, t), wd, bd, head, dev(u), mask, True, packed=pk)
    policy, action, logits = host(policy), host(action), host(logits)
    want_p, _, want_l = olayers.mlp_forward(x, ws, biases, HEAD_CODE[head], u, None, mask or None)
    # hidden activations are rounded to the storage dtype before they feed the next MFMA: f16 keeps
    # 11 significant bits, bf16 only 8 (2^-9 relative rounding per activation and layer), so the raw
    # last-layer outputs of a bf16 stack get a looser bound; the policy keeps the 3e-3 contract
    assert ogemm.rel_frobenius(logits, want_l) < (3e-3 if dtype == "f16" else 1e-2)
    assert ogemm.rel_frobenius(policy, want_p) < 3e-3
    # against the oracle that rounds hidden activations to the storage dtype like the kernel does:
    # only summation order differs, which now and then flips a rounded activation by one ulp
    tight_p, _, tight_l = olayers.mlp_forward(x, ws, biases, HEAD_CODE[head], u, dtype, mask or None)
    assert ogemm.rel_frobenius(logits, tight_l) < 2e-4
    assert ogemm.rel_frobenius(policy, tight_p) < 2e-4
    # bit-exact action given the kernel's policy and the same uniforms
    if head is not None:
        assert (action == orow.discrete_sampling(policy, u)).all()
        assert (np.take_along_axis(policy, action[:, None].astype(np.int64), 1) > 0).all()
        if mask:
            assert (action < mask).all() and (policy[:, mask:] == 0).all()
        assert np.abs(policy.sum(axis=1) - 1).max() < 1e-5
    return policy, action


def test_config3_leduc_policy(LY):
    """The benchmark's policy-network workload: batch 16384, 32 -> 256 -> 256 -> 256 -> 3, f16, softmax head, regret-matching sampling."""
    announce("mlp config 3")
    rng = np.random.default_rng(3)
    x, ws, u = make_problem(rng, 16384, [32, 256, 256, 256, 3], "f16")
    policy, action = check(LY, x, ws, u, "f16")
    counts = np.bincount(action, minlength=3) / len(action)
    assert np.abs(counts - policy.mean(axis=0)).max() < 0.02   # sampled frequencies follow the policy


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch", [1, 100, 640])
def test_ragged_batches_and_dtypes(LY, dtype, batch):
    announce("mlp ragged batch=%d %s" % (batch, dtype))
    rng = np.random.default_rng(batch)
    x, ws, u = make_problem(rng, batch, [32, 256, 256, 256, 3], dtype)
    check(LY, x, ws, u, dtype)


@pytest.mark.parametrize("dims,head,mask", [([128, 64, 64], "regret_matching", 3), ([64, 64, 64], "softmax", 3),
                                            ([16, 32, 8], "softmax", 0), ([256, 256, 64], None, 0),
                                            ([32, 96, 160, 5], "softmax_regret_matching", 0), ([48, 3], "softmax", 0)])
def test_other_stacks(LY, dims, head, mask):
    """Shapes of the reference's real models: Leduc input(128) -> 64 -> 64 (3 valid) with a masked
    regret-matching head (game/leduc/model_cem.spi:47-63)."""
    announce("mlp stack %s head=%s mask=%d" % (dims, head, mask))
    rng = np.random.default_rng(len(dims) * 100 + dims[0])
    x, ws, u = make_problem(rng, 300, dims, "f16")
    if head is None:
        t = TORCH["f16"]
        policy, _, logits = LY.mlp_forward(dev(x, t), [dev(w, t) for w in ws], None, None, None, 0, True)
        want = olayers.mlp_forward(x, ws, head=olayers.HEAD_NONE, act_dtype="f16")[2]
        assert ogemm.rel_frobenius(host(policy), want) < 2e-4 and (host(policy) == host(logits)).all()
    else:
        check(LY, x, ws, u, "f16", head, mask)


@pytest.mark.parametrize("dims,head,mask,batch,dtype,with_bias", [
    ([48, 256, 256, 17], "softmax", 0, 300, "f16", True),                 # K0 not a multiple of 64, ragged head
    ([128, 256, 256, 256, 64], "softmax_regret_matching", 40, 200, "bf16", True),   # four first-layer chunks, widest head
    ([256, 256, 8], "regret_matching", 5, 130, "f16", False),             # no hidden 256 -> 256 layer at all
    ([64, 256, 256, 3], "softmax_regret_matching", 0, 20000, "f16", False),  # more rows than 4-wave workgroups cover: 8 waves
    ([16, 256, 256, 256, 256, 256, 256, 256, 4], "softmax", 0, 64, "f16", True),  # the deepest stack
    # up to one 64-row workgroup per compute unit and at most 16 outputs: hidden layers split by output features
    ([128, 256, 256, 256, 10], "softmax", 7, 300, "f16", True),           # four first-layer chunks, head staged in LDS
    ([48, 256, 256, 16], "regret_matching", 0, 130, "bf16", False),       # K0 in (32, 64], not a multiple of 32; 16 outputs
    ([32, 256, 256, 256, 256, 5], "softmax_regret_matching", 0, 16384, "bf16", True),   # every compute unit busy
])
def test_stacks_with_256_wide_hidden_layers(LY, dims, head, mask, batch, dtype, with_bias):
    """The shapes served by the two kernels for stacks whose hidden layers are all 256 wide."""
    announce("mlp h256 %s head=%s mask=%d batch=%d %s bias=%s" % (dims, head, mask, batch, dtype, with_bias))
    rng = np.random.default_rng(sum(dims) + batch)
    x, ws, u = make_problem(rng, batch, dims, dtype)
    biases = None
    if with_bias:
        biases = [rng.standard_normal(d, dtype=np.float32) * np.float32(0.1) for d in dims[1:]]
        biases[0] = None
    check(LY, x, ws, u, dtype, head, mask, biases)


def test_bias_extension(LY):
    announce("mlp biases")
    rng = np.random.default_rng(9)
    dims = [32, 64, 64, 3]
    x, ws, u = make_problem(rng, 200, dims, "bf16")
    biases = [rng.standard_normal(d, dtype=np.float32) * np.float32(0.1) for d in dims[1:]]
    biases[1] = None
    check(LY, x, ws, u, "bf16", biases=biases)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,dims,head,mask", [(16384, [32, 256, 256, 256, 64], "softmax", 3),
                                                  (1000, [128, 256, 256, 64], "regret_matching", 3),
                                                  (333, [32, 256, 256, 256, 64], "softmax_regret_matching", 11),
                                                  (40000, [32, 256, 256, 32], "softmax", 16),
                                                  (257, [64, 256, 256, 6], "softmax", 5)])
def test_masked_head_without_logits(LY, dtype, batch, dims, head, mask):
    """Without the logits output a masked head is computed for its valid columns only and the rest of every policy
    row is written as zeros (a 64-wide layer with 3 valid columns is the reference's shape for a 3-action game).
    The policy must match the oracle and the run that does write the logits, the masked columns must be exact zeros
    inside a buffer of sentinels, and the action must be the one the kernel's own policy and the uniforms give."""
    announce("mlp masked head, no logits: %s %s batch=%d mask=%d %s" % (dims, head, batch, mask, dtype))
    rng = np.random.default_rng(batch + mask)
    x, ws, u = make_problem(rng, batch, dims, dtype)
    t = TORCH[dtype]
    xd, wd, ud = dev(x, t), [dev(w, t) for w in ws], dev(u)
    n = dims[-1]
    buf = torch.full((64 + batch * n + 64,), -9.0, dtype=torch.float32, device="cuda")
    policy_t = buf[64:64 + batch * n].view(batch, n)
    action_t = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    LY.mlp_forward(xd, wd, None, head, ud, mask, False, policy_out=policy_t, action_out=action_t)
    raw = host(buf)
    assert (raw[:64] == -9).all() and (raw[-64:] == -9).all()
    policy, action = raw[64:-64].reshape(batch, n), host(action_t)
    full_p, full_a, _ = LY.mlp_forward(xd, wd, None, head, ud, mask, True)
    want_p, _, _ = olayers.mlp_forward(x, ws, None, HEAD_CODE[head], u, dtype, mask)
    assert (policy[:, mask:] == 0).all() and np.abs(policy.sum(axis=1) - 1).max() < 1e-5
    assert ogemm.rel_frobenius(policy, want_p) < 2e-4 and ogemm.rel_frobenius(policy, host(full_p)) < 2e-4
    assert (action == orow.discrete_sampling(policy, u)).all() and (action < mask).all() and (action >= 0).all()


@pytest.mark.parametrize("dims,head,mask", [([32, 64, 9], "softmax", 0), ([16, 96, 16], "regret_matching", 0),
                                            ([64, 32, 17], "softmax_regret_matching", 11), ([48, 160, 32], "softmax", 0),
                                            ([32, 64, 33], "softmax", 0)])
def test_head_widths_of_other_stacks(LY, dims, head, mask):
    """The widths at which the head of the kernel for any hidden width changes its instance."""
    announce("mlp head width %s head=%s mask=%d" % (dims, head, mask))
    x, ws, u = make_problem(np.random.default_rng(dims[-1]), 70, dims, "f16")
    check(LY, x, ws, u, "f16", head, mask)


@pytest.mark.parametrize("dims,mask,batch,with_bias", [
    ([16, 3], 0, 1, True), ([16, 32, 4], 0, 17, False),                   # one layer; waves without a tile of their own
    ([144, 96, 5], 0, 16, True), ([256, 128, 96, 64], 60, 33, False),     # K that ends in mid-step; inputs on both planes; a wide mask
    ([48, 32, 32, 32, 32, 32, 32, 32, 33], 0, 50, True),                  # eight layers
    ([80, 192, 192, 24], 0, 100, True), ([256, 224, 256, 256, 64], 0, 65, False),      # sixteen waves; more units than slots
    ([64, 160, 64, 16], 0, "16+1", True), ([64, 128, 7], 0, "32+1", False), ([64, 64, 192, 2], 0, "64", True),    # 32 and 64 rows a workgroup
    ([256, 64, 128, 9], 0, "64+1", True), ([48, 96, 3], 0, "64+33", True), ([16, 3], 0, "65", False),     # rows shared out
    ([128, 160, 64], 5, "64+1", False), ([64, 256, 40], 0, "64+1", True), ([64, 32, 12], 2, "66", False),
    ([64, 192, 192, 192, 3], 0, "128+1", True), ([128, 128, 128, 128, 128, 128, 20], 0, "128+40", False),     # and weights that do not fit
    ([256, 224, 256, 256, 64], 0, "129", False)])
def test_stacks_of_any_width_at_the_edges_of_their_kernels(LY, dims, mask, batch, with_bias):
    """Widths and batches around every rule of the kernels for any hidden width; batches as "rows per compute unit + rows"."""
    announce("mlp any width %s mask=%d batch=%s bias=%s" % (dims, mask, batch, with_bias))
    if isinstance(batch, str):
        per_cu, _, more = batch.partition("+")
        batch = int(per_cu) * torch.cuda.get_device_properties(0).multi_processor_count + int(more or 0)
    rng = np.random.default_rng(sum(dims))
    dtype = "bf16" if len(dims) % 2 else "f16"
    x, ws, u = make_problem(rng, batch, dims, dtype)
    biases = [rng.standard_normal(o).astype(np.float32) * 0.1 for o in dims[1:]] if with_bias else None
    if biases is not None and len(biases) > 1:
        biases[0] = None
    check(LY, x, ws, u, dtype, "softmax", mask, biases)


@pytest.mark.parametrize("dims,head,mask,batch,dtype", [([128, 64, 64], "regret_matching", 3, 64, "bf16"),
                                                        ([48, 96, 128, 10], "softmax", 4, 37, "f16"),      # rows of no whole pieces
                                                        ([16, 32, 12], "softmax_regret_matching", 7, 130, "bf16"),
                                                        ([32, 64, 160, 64], "softmax", 1, 20000, "f16")])  # 128 rows a workgroup
def test_masked_head_of_other_stacks_without_logits(LY, dims, head, mask, batch, dtype):
    """The same for hidden widths other than 256: bit for bit what the run that writes the logits (and computes every
    column) gives, a row of NaNs among them."""
    announce("mlp masked head, no logits: %s %s batch=%d mask=%d %s" % (dims, head, batch, mask, dtype))
    rng = np.random.default_rng(batch + mask)
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    x = rng.standard_normal((batch, dims[0])).astype(np.float32)
    x[batch // 2] = np.nan
    xd = dev(x, t)
    wd = [dev((rng.standard_normal((o, i)) / np.sqrt(i)).astype(np.float32), t) for i, o in zip(dims[:-1], dims[1:])]
    ud = dev((1 - rng.random(batch)).astype(np.float32))
    policy_t = torch.full((batch, dims[-1]), 7.0, device="cuda")
    _, action = LY.mlp_forward(xd, wd, None, head, ud, mask, False, policy_out=policy_t)
    full_p, full_a, _ = LY.mlp_forward(xd, wd, None, head, ud, mask, True)
    assert torch.equal(policy_t.view(torch.int32), full_p.view(torch.int32)) and torch.equal(action, full_a)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("dims,mask,rows_per_unit", [([128, 64, 64], 3, 0), ([64, 96, 160, 10], 0, 0), ([80, 192, 192, 24], 0, 0), ([64, 128, 64], 3, 65),
                                                     ([64, 128, 40], 0, 65), ([48, 192, 64], 11, 65), ([128] * 7 + [20], 0, 129), ([64, 256, 128, 64], 3, 65)])
def test_a_hidden_sum_that_is_no_number_becomes_zero(LY, dims, mask, rows_per_unit, dtype):
    """relu is max(0, x) as in the reference.  Features with a NaN for a bias, of either sign, are zeros, as those with a bias far below
    every sum are, bit for bit.  In a row with a NaN, of either sign, or inf - inf in every sum, the first hidden layer is zeros, hence the
    outputs are without biases, and the head falls to the even distribution of the valid columns."""
    announce("mlp hidden nan %s mask=%d %s" % (dims, mask, dtype))
    batch = 50 if rows_per_unit == 0 else rows_per_unit * torch.cuda.get_device_properties(0).multi_processor_count
    rng = np.random.default_rng(sum(dims))
    t = TORCH[dtype]
    x = rng.standard_normal((batch, dims[0])).astype(np.float32)
    odd = [0, 7, batch // 2, batch - 1]
    x[odd[0]], x[odd[1], 3], x[odd[2], 2:], x[odd[2], :2], x[odd[3]] = np.nan, -np.nan, 0, [np.inf, -np.inf], -np.nan
    wd = [dev(rng.standard_normal((o, i)).astype(np.float32) / np.float32(np.sqrt(i)), t) for i, o in zip(dims[:-1], dims[1:])]
    wd[0][:, :2] = wd[0][:, :2].abs() + 0.5                # (inf times the one minus inf times the other, in every feature)
    bias = [rng.standard_normal(o).astype(np.float32) for o in dims[1:]]
    none, low = [b.copy() for b in bias], [b.copy() for b in bias]
    for l in range(len(dims) - 2):
        off = rng.choice(dims[l + 1], 5, replace=False)
        none[l][off], low[l][off] = [np.nan, -np.nan, np.nan, -np.nan, np.nan], -1e30
    un = (1 - rng.random(batch)).astype(np.float32)
    u, xd, valid = dev(un), dev(x, t), mask or dims[-1]
    for head in ("softmax", "regret_matching", "softmax_regret_matching"):
        got = LY.mlp_forward(xd, wd, [dev(b) for b in none], head, u, mask)
        want = LY.mlp_forward(xd, wd, [dev(b) for b in low], head, u, mask)
        assert all(torch.equal(g, w) for g, w in zip(got, want)) and torch.isfinite(got[0]).all()
        for want_logits in (False, True):
            policy, action = (host(o) for o in LY.mlp_forward(xd, wd, None, head, u, mask, want_logits)[:2])
            assert np.isfinite(policy).all() and (action == orow.discrete_sampling(policy, un)).all()
            assert np.abs(policy[odd, :valid] * valid - 1).max() < 1e-6 and (policy[odd, valid:] == 0).all()


@pytest.mark.parametrize("dims,mask,few,many", [([32, 256, 4], 0, "64", "128+1"), ([64, 256, 64], 4, "64+1", "129"), ([80, 256, 3], 0, "64", "64+1"),
                                                ([128, 256, 2], 0, "128", "128+1"), ([256, 256, 4], 0, "64+1", "130"), ([16, 256, 8], 0, "64", "64+1"),
                                                ([144, 256, 8], 5, "3", "140"), ([112, 256, 7], 0, "16", "16+1"), ([64, 256, 64], 8, "64", "200"), ([64, 256, 12], 9, "64", "129")])
def test_a_single_hidden_layer_of_256_on_both_sides_of_its_lines(LY, dims, mask, few, many):
    """Which kernel such a stack runs on goes by the outputs, the inputs and the rows per compute unit: the rows of a batch in front of a
    line give the bits they give as part of one behind it, with and without biases, against the oracle."""
    announce("mlp one hidden layer %s mask=%d rows %s / %s" % (dims, mask, few, many))
    units = torch.cuda.get_device_properties(0).multi_processor_count
    few, many = (int(r.partition("+")[0]) * units + int(r.partition("+")[2] or 0) for r in (few, many))
    rng = np.random.default_rng(sum(dims) + few)
    for dtype, with_bias in (("f16", True), ("bf16", False)):
        x, ws, u = make_problem(rng, many, dims, dtype)
        biases = [rng.standard_normal(o).astype(np.float32) for o in dims[1:]] if with_bias else None
        t = TORCH[dtype]
        xd, wd, ud = dev(x, t), [dev(w, t) for w in ws], dev(u)
        bd = [dev(b) for b in biases] if with_bias else None
        for head in ("softmax", "softmax_regret_matching"):
            part = LY.mlp_forward(xd[:few].contiguous(), wd, bd, head, ud[:few].contiguous(), mask)
            whole = LY.mlp_forward(xd, wd, bd, head, ud, mask)
            assert all(torch.equal(p, w[:few]) for p, w in zip(part, whole))
            assert (host(whole[1]) == orow.discrete_sampling(host(whole[0]), u)).all()
        want, _, _ = olayers.mlp_forward(x, ws, biases, HEAD_CODE[head], u, dtype, mask or None)
        assert ogemm.rel_frobenius(host(whole[0]), want) < 2e-4          # (the bound of the other stacks: order of sums, flipped roundings)


@pytest.mark.parametrize("dims,mask", [([48, 256, 256, 32, 64], 4), ([48, 256, 256, 32, 64], 9), ([64, 256, 224, 128, 6], 0), ([128, 192, 192, 192, 12], 5),
                                       ([128, 256, 256, 32], 0), ([112, 256, 256, 256, 24], 17), ([128, 256, 256, 64], 20), ([128] * 7 + [30], 0),
                                       ([256, 256, 16], 0), ([32, 64, 64, 64, 10], 0), ([128, 64, 64], 3), ([256, 192, 10], 0), ([32, 64, 64, 5], 0),
                                       ([48, 128, 16], 7)])
def test_a_round_of_128_rows_per_unit(LY, dims, mask):
    """Between 64 and 128 rows per compute unit other forms run than below and above: the rows of a batch just behind the first line and
    just in front of the second give the bits they give as part of one behind it, a row of NaNs among them, with biases and without, and
    nothing outside the policy is written."""
    announce("mlp round of 128 rows %s mask=%d" % (dims, mask))
    units = torch.cuda.get_device_properties(0).multi_processor_count
    many = 128 * units + 77
    rng = np.random.default_rng(sum(dims) + mask)
    for dtype, with_bias, head in (("f16", True, "softmax"), ("bf16", False, "softmax_regret_matching")):
        x, ws, u = make_problem(rng, many, dims, dtype)
        x[5], x[17, 3] = np.nan, np.inf
        t, n = TORCH[dtype], dims[-1]
        xd, wd, ud = dev(x, t), [dev(w, t) for w in ws], dev(u)
        biases = [rng.standard_normal(o).astype(np.float32) for o in dims[1:]] if with_bias else None
        bd = [dev(b) for b in biases] if with_bias else None
        whole = LY.mlp_forward(xd, wd, bd, head, ud, mask)
        for rows in (64 * units, 64 * units + 1, 100 * units + 3, 128 * units):
            buf = torch.full((64 + rows * n + 64,), -9.0, device="cuda")
            policy = buf[64:64 + rows * n].view(rows, n)
            _, action = LY.mlp_forward(xd[:rows].contiguous(), wd, bd, head, ud[:rows].contiguous(), mask, policy_out=policy)
            assert torch.equal(policy.nan_to_num(7), whole[0][:rows].nan_to_num(7)) and torch.equal(action, whole[1][:rows])
            assert (buf[:64] == -9).all() and (buf[-64:] == -9).all()
        plain = np.ones(many, bool)
        plain[[5, 17]] = False
        want, _, _ = olayers.mlp_forward(x[plain], ws, biases, HEAD_CODE[head], u[plain], dtype, mask or None)
        got = host(whole[0])[plain]
        assert ogemm.rel_frobenius(got, want) < 2e-4 and (host(whole[1])[plain] == orow.discrete_sampling(got, u[plain])).all()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("mask", [1, 3, 13, 16])
def test_past_a_narrow_mask_are_zeros_behind_a_256_wide_layer(LY, mask, dtype):
    """... whatever the valid columns are: in a row whose hidden sums are infinite those are NaN and there is no action."""
    announce("mlp 64-256-64 nan rows mask=%d %s" % (mask, dtype))
    rng = np.random.default_rng(mask)
    t = TORCH[dtype]
    wd = [dev(rng.standard_normal((o, i)).astype(np.float32) / np.float32(np.sqrt(i)), t) for i, o in ((64, 256), (256, 64))]
    units = torch.cuda.get_device_properties(0).multi_processor_count
    for batch in (20, 64 * units + 9):
        x = rng.standard_normal((batch, 64)).astype(np.float32)
        x[3, 0] = np.inf
        x[batch - 2, 1] = -np.inf
        u = dev((1 - rng.random(batch)).astype(np.float32))
        policy, action = LY.mlp_forward(dev(x, t), wd, None, "softmax", u, mask)
        policy, action = host(policy), host(action)
        for row in (3, batch - 2):
            assert np.isnan(policy[row, :mask]).all() and action[row] == 2147483647
        assert (policy[:, mask:] == 0).all()


@pytest.mark.parametrize("dims,mask", [([64, 128, 64], 5), ([64, 128, 64], 11), ([64, 128, 64], 32), ([64, 128, 64], 40), ([48, 96, 40], 20), ([32, 160, 63], 13),
                                       ([128, 192, 256, 192, 64], 17), ([128, 192, 256, 192, 64], 3), ([128, 192, 256, 192, 64], 47)])
@pytest.mark.parametrize("rows", ["40", "66", "130"])
def test_masked_columns_of_rows_wider_than_the_head(LY, dims, mask, rows):
    """Without logits the valid columns alone are computed and the rest of a row, of whole 16-byte pieces or not, follows: bit for bit the
    policy and the actions of the call that writes the logits, in every kernel (rows per compute unit from 66 up), in front of and behind
    nothing, and the oracle's."""
    announce("mlp masked rows %s mask=%d rows %s" % (dims, mask, rows))
    batch = int(rows) if rows == "40" else int(rows) * torch.cuda.get_device_properties(0).multi_processor_count + 5
    rng = np.random.default_rng(sum(dims) + mask)
    for dtype, head in (("f16", "regret_matching"), ("bf16", "softmax_regret_matching"), ("f16", "softmax")):
        x, ws, u = make_problem(rng, batch, dims, dtype)
        t, n = TORCH[dtype], dims[-1]
        xd, wd, ud = dev(x, t), [dev(w, t) for w in ws], dev(u)
        buf = torch.full((64 + batch * n + 64,), -9.0, device="cuda")
        policy = buf[64:64 + batch * n].view(batch, n)
        _, action = LY.mlp_forward(xd, wd, None, head, ud, mask, policy_out=policy)
        full_p, full_a, _ = LY.mlp_forward(xd, wd, None, head, ud, mask, True)
        assert torch.equal(policy, full_p) and torch.equal(action, full_a)
        assert (buf[:64] == -9).all() and (buf[-64:] == -9).all() and (policy[:, mask:] == 0).all()
        want, _, _ = olayers.mlp_forward(x, ws, None, HEAD_CODE[head], u, dtype, mask)
        assert ogemm.rel_frobenius(host(policy), want) < 2e-4          # (the bound of the other stacks)
        assert (host(action) == orow.discrete_sampling(host(policy), u)).all()


@pytest.mark.parametrize("dims,mask", [([64, 128, 4], 0), ([32, 64, 64], 3), ([64, 128, 16], 0), ([32, 160, 64], 0), ([48, 64, 64], 40), ([128, 192, 256, 192, 4], 0),
                                       ([128, 192, 256, 192, 64], 0), ([128, 192, 256, 192, 64], 21), ([64, 256, 4], 0)])
@pytest.mark.parametrize("rows", [2, 66, 132])
def test_heads_of_any_width_draw_their_own_uniforms(LY, dims, mask, rows):
    """A Philox stream in place of the tensor of uniforms in every kernel of these stacks: the policy's bits and the actions of the run that
    reads what sp_philox_uniforms hands out for the rows."""
    from ml import _lib, primitives
    announce("mlp philox any width %s mask=%d rows %d" % (dims, mask, rows))
    batch = rows * torch.cuda.get_device_properties(0).multi_processor_count - 32
    rng = np.random.default_rng(sum(dims) + mask + rows)
    x, ws, _ = make_problem(rng, batch, dims, "bf16")
    xd, wd = dev(x, torch.bfloat16), [dev(w, torch.bfloat16) for w in ws]
    for cfg in (primitives.philox(_lib.PHILOX_LAYER, blocks_per_grid=32, rows_per_block=batch // 32, offset=8), primitives.philox(_lib.PHILOX_GRID, blocks_per_grid=24)):
        u = primitives.philox_uniforms(cfg, batch, dims[-1])
        assert u.unique().numel() > batch // 2
        for head in ("regret_matching", "softmax"):
            want = LY.mlp_forward(xd, wd, None, head, u, mask)
            got = LY.mlp_forward(xd, wd, None, head, None, mask, rng=cfg)
            assert all(torch.equal(g, w) for g, w in zip(got, want))
    assert (host(got[1]) == orow.discrete_sampling(host(got[0]), host(u))).all()


@pytest.mark.parametrize("dims,head,mask,batch,dtype,with_bias", [
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 16384, "f16", False),     # the benchmark's policy network
    ([32, 256, 256, 256, 3], "softmax", 0, 1, "bf16", False),                        # a single row
    ([32, 256, 256, 3], "softmax_regret_matching", 0, 100, "f16", True),             # three layers
    ([32, 256, 256, 256, 256, 5], "softmax_regret_matching", 0, 333, "bf16", True),  # five layers: refills into both register sets
    ([48, 256, 256, 16], "regret_matching", 0, 130, "bf16", False),                  # two first-layer k-steps, K0 not a multiple of 32
    ([64, 256, 256, 256, 256, 9], "softmax", 7, 640, "f16", True),                   # two first-layer k-steps, five layers, masked head with logits
    ([128, 256, 256, 256, 10], "softmax", 7, 300, "f16", True),                      # eight first-layer k-steps (zero-padded K0)
    ([256, 256, 256, 8], "regret_matching", 5, 130, "f16", False),                   # a full-width first layer, three layers
    ([256, 256, 256, 256, 256, 16], "softmax", 0, 64, "bf16", True),                 # full-width first layer, five layers, widest head
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 20000, "f16", False),     # more workgroups than compute units
    ([32, 256, 256, 256, 3], "softmax", 0, 200, "f16", "all"),                        # a bias on every layer
    ([256, 256, 256, 256, 256, 12], "softmax", 0, 200, "bf16", "all"),
    ([64, 256, 256, 256, 4], "regret_matching", 0, 77, "f16", "only1"),               # a bias on the second layer alone
])
def test_packed_weights_kernel(LY, dims, head, mask, batch, dtype, with_bias):
    """The kernel that streams pre-packed weights straight into registers (sp_mlp_pack_weights +
    sp_mlp_forward_packed) against the oracle, and against sp_mlp_forward on the row-major weights."""
    announce("mlp packed %s head=%s mask=%d batch=%d %s bias=%s" % (dims, head, mask, batch, dtype, with_bias))
    rng = np.random.default_rng(sum(dims) + batch + 1)
    x, ws, u = make_problem(rng, batch, dims, dtype)
    biases = None
    if with_bias:
        biases = [rng.standard_normal(d, dtype=np.float32) * np.float32(0.1) for d in dims[1:]]
        if with_bias == "only1":
            biases = [b if l == 1 else None for l, b in enumerate(biases)]
        elif with_bias != "all":
            biases[1] = None
    policy, action = check(LY, x, ws, u, dtype, head, mask, biases, packed=True)
    t = TORCH[dtype]
    bd = None if biases is None else [dev(b) if b is not None else None for b in biases]
    plain_p, plain_a = LY.mlp_forward(dev(x, t), [dev(w, t) for w in ws], bd, head, dev(u), mask)
    assert ogemm.rel_frobenius(policy, host(plain_p)) < 2e-4
    assert (action != host(plain_a)).mean() < 1e-3      # same uniforms, policies equal to rounding


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_packed_masked_head_without_logits(LY, dtype):
    """A 64-wide output layer under a 3-column mask (the reference's shape for a 3-action game) on the packed
    kernel: only the valid columns are computed, the rest of each policy row is exact zeros inside sentinels."""
    announce("mlp packed masked head, no logits " + dtype)
    batch, dims, mask = 4100, [32, 256, 256, 256, 64], 3
    rng = np.random.default_rng(77)
    x, ws, u = make_problem(rng, batch, dims, dtype)
    t = TORCH[dtype]
    xd, wd, ud = dev(x, t), [dev(w, t) for w in ws], dev(u)
    pk = LY.pack_weights(wd)
    buf = torch.full((64 + batch * 64 + 64,), -9.0, dtype=torch.float32, device="cuda")
    policy_t = buf[64:64 + batch * 64].view(batch, 64)
    action_t = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    LY.mlp_forward(xd, None, None, "softmax", ud, mask, False, policy_out=policy_t, action_out=action_t, packed=pk)
    raw = host(buf)
    assert (raw[:64] == -9).all() and (raw[-64:] == -9).all()
    policy, action = raw[64:-64].reshape(batch, 64), host(action_t)
    want_p, _, _ = olayers.mlp_forward(x, ws, None, HEAD_CODE["softmax"], u, dtype, mask)
    assert (policy[:, mask:] == 0).all() and np.abs(policy.sum(axis=1) - 1).max() < 1e-5
    assert ogemm.rel_frobenius(policy, want_p) < 2e-4
    assert (action == orow.discrete_sampling(policy, u)).all() and (action < mask).all() and (action >= 0).all()
    # the logits of a wide masked layer are more than the packed kernel computes: the call says so
    from ml import _lib
    with pytest.raises(_lib.SpiralError, match="UNSUPPORTED"):
        LY.mlp_forward(xd, None, None, "softmax", ud, mask, True, packed=pk)


def test_packing_is_refused_for_other_stacks(LY):
    announce("mlp packed: unsupported stacks")
    t = torch.float16
    mk = lambda dims: [torch.zeros((o, i), dtype=t, device="cuda") for i, o in zip(dims[:-1], dims[1:])]
    assert LY.pack_weights(mk([32, 64, 64, 3])) is None                  # hidden width other than 256
    assert LY.pack_weights(mk([32, 256, 3])) is None                     # two layers
    assert LY.pack_weights(mk([32] + [256] * 6 + [3])) is None           # deeper than the packed kernel goes
    assert LY.packed_bytes([32, 256, 256, 256, 3]) == 4 * 4096 + 2 * 131072 + 8192


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("dims,mask,with_bias", [([32, 256, 256, 256, 3], 0, False), ([32, 256, 256, 256, 64], 3, False),
                                                 ([256, 256, 256, 16], 0, True), ([64, 128, 96, 8], 0, False)])
def test_results_do_not_change_from_run_to_run(LY, dims, mask, with_bias, packed):
    """Three launches on the same inputs give the same bits, for every fused kernel (hand-issued MFMAs and loads
    counted by hand: a wait that is one short, or a register overwritten too early, shows up as results that
    differ between launches)."""
    announce("mlp run-to-run dims=%s packed=%s" % (dims, packed))
    rng = np.random.default_rng(23)
    x, ws, u = make_problem(rng, 16384, dims, "f16")
    wd = [dev(w, torch.float16) for w in ws]
    bd = [dev(rng.standard_normal(w.shape[0], dtype=np.float32)) for w in ws] if with_bias else None
    pk = LY.pack_weights(wd) if packed else None
    if packed and pk is None:
        pytest.skip("this stack has no packed form")
    xd, ud = dev(x, torch.float16), dev(u)
    logits = not (packed and mask)        # the packed kernel computes a masked head for its valid columns only
    first = [t.clone() for t in LY.mlp_forward(xd, wd, bd, "softmax_regret_matching", ud, mask, logits, packed=pk) if t is not None]
    for _ in range(2):
        again = [t for t in LY.mlp_forward(xd, wd, bd, "softmax_regret_matching", ud, mask, logits, packed=pk) if t is not None]
        assert len(first) == len(again)
        for a, b in zip(first, again):
            assert torch.equal(a, b)



@pytest.mark.parametrize("dims,mask,batch,want_logits,packed,mode", [
    ([32, 96, 160, 8], 0, 24 * 13, False, False, "layer"),               # the general kernel
    ([128, 256, 256, 64], 40, 24 * 9, True, False, "layer"),             # 256-wide hidden layers, wide head
    ([32, 256, 256, 256, 64], 3, 16384, False, False, "layer"),          # feature-split kernel, head of 3 valid columns of 64
    ([32, 256, 256, 256, 64], 3, 16384, False, True, "layer"),           # the same on packed weights
    ([32, 256, 256, 256, 4], 0, 1000, False, True, "block"),             # packed, plain head, the block-level stream
    ([64, 256, 256, 16], 0, 40000, False, False, "grid"),                # more rows than one round of workgroups
])
def test_head_draws_its_own_uniforms(LY, dims, mask, batch, want_logits, packed, mode):
    """A head given a Philox stream instead of a tensor of uniforms (the reference seeds one generator per thread
    and the sampling node draws in the kernel, ml/layers.spi:339-344): every row must use exactly the uniform
    sp_philox_uniforms hands out for it -- same policy bits, same actions as the run that reads those uniforms
    from a tensor -- and those uniforms are the stream the golden sampled indices pin."""
    from ml import _lib, primitives
    from oracle import philox as ophilox
    announce("mlp philox head dims=%s mask=%d batch=%d packed=%s mode=%s" % (dims, mask, batch, packed, mode))
    rng = np.random.default_rng(sum(dims) + batch)
    x, ws, _ = make_problem(rng, batch, dims, "f16")
    xd, wd = dev(x, torch.float16), [dev(w, torch.float16) for w in ws]
    pk = LY.pack_weights(wd) if packed else None
    cols = dims[-1]
    if mode == "layer":
        q = 24 if batch % 24 == 0 else 32
        cfg = primitives.philox(_lib.PHILOX_LAYER, blocks_per_grid=q, rows_per_block=batch // q, offset=8)
        want_u = ophilox.row_uniforms_layer(q, batch // q, cols, offset=8)
    elif mode == "block":
        cfg = primitives.philox(_lib.PHILOX_BLOCK)
        want_u = ophilox.row_uniforms_block(batch, cols)
    else:
        cfg = primitives.philox(_lib.PHILOX_GRID, blocks_per_grid=24)
        want_u = ophilox.row_uniforms_grid(batch, cols, blocks=24)
    u = primitives.philox_uniforms(cfg, batch, cols)
    assert (host(u) == np.asarray(want_u, dtype=np.float32).reshape(-1)).all()
    head = "softmax_regret_matching"
    with_u = LY.mlp_forward(xd, wd, None, head, u, mask, want_logits, packed=pk)
    with_rng = LY.mlp_forward(xd, wd, None, head, None, mask, want_logits, packed=pk, rng=cfg)
    for a, b in zip(with_u, with_rng):
        assert torch.equal(a, b)
    assert (host(with_rng[1]) == orow.discrete_sampling(host(with_rng[0]), host(u))).all()


@pytest.mark.parametrize("dims,head,mask,batch,dtype,with_bias,packed", [
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 100000, "f16", False, True),   # the benchmark's network, ragged last pair
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 133000, "f16", False, False),  # ... from the row-major weights
    ([32, 256, 256, 256, 3], "softmax", 0, 300000, "bf16", "all", True),                  # 18 tiles per compute unit
    ([16, 256, 256, 4], "softmax_regret_matching", 0, 132000, "f16", True, False),        # three layers, a 16-wide first layer
    ([48, 256, 256, 256, 16], "softmax", 0, 131100, "bf16", True, False),                 # two first-layer k-steps, K0 not a multiple of 32, 16 outputs
    ([64, 256, 256, 12], "softmax", 7, 98400, "f16", "only1", True),                      # masked head with logits, head staged in LDS
    ([32, 256, 256, 256, 2], "softmax_regret_matching", 0, 98304 + 65, "bf16", False, True),   # one row in the second tile of the last pair
    ([64, 256, 256, 256, 4], "softmax_regret_matching", 0, 131072 + 31, "f16", "all", False),  # pipelined form: two first-layer k-steps, every bias, row-major
    ([48, 256, 256, 256, 8], "softmax", 3, 99000, "bf16", True, True),                          # pipelined form: 3 of 8 columns valid, zeros behind them
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 98304 + 32 * 256 * 9 + 5, "f16", False, True),  # a last head pass of one tile on some units
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 65536 + 7, "f16", False, True),      # the smallest batch the pipelined form takes, packed
    ([32, 256, 256, 256, 3], "softmax_regret_matching", 0, 81920 + 33, "f16", False, False),    # ... and from row-major weights
])
def test_weights_resident_in_registers(LY, dims, head, mask, batch, dtype, with_bias, packed):
    """Batches of several 64-row tiles per compute unit run on the kernels that load the weights once and keep them in
    registers while they walk over their tiles (from six tiles per unit with packed weights, from eight with row-major
    ones; the pipelined form of four-layer stacks from four and five): against the oracle like every other kernel, and against the per-tile packed kernel run on the same rows in
    slices small enough to stay on that kernel (same operand layout; the same order of the sums except in the output
    layer of the pipelined form)."""
    announce("mlp resident %s head=%s mask=%d batch=%d %s bias=%s packed=%s" % (dims, head, mask, batch, dtype, with_bias, packed))
    rng = np.random.default_rng(sum(dims) + batch + 7)
    x, ws, u = make_problem(rng, batch, dims, dtype)
    biases = None
    if with_bias:
        biases = [rng.standard_normal(d, dtype=np.float32) * np.float32(0.1) for d in dims[1:]]
        if with_bias == "only1":
            biases = [b if l == 1 else None for l, b in enumerate(biases)]
        elif with_bias != "all":
            biases[1] = None
    policy, action = check(LY, x, ws, u, dtype, head, mask, biases, packed=packed)
    t = TORCH[dtype]
    wd = [dev(w, t) for w in ws]
    bd = None if biases is None else [dev(b) if b is not None else None for b in biases]
    pk = LY.pack_weights(wd)
    # four-layer stacks with at most 4 outputs take the pipelined form, whose output layer adds its k-steps slice by
    # slice: equal to the per-tile kernel to rounding; the others add in the per-tile kernel's order: equal bit for bit
    pipelined = len(dims) == 5 and (mask or dims[-1]) <= 4
    # the call that asks for no logits is another instance of the kernel: the same bits -- unless only that call can
    # leave the masked columns out of the output layer and so comes to run on the pipelined form
    p, a = LY.mlp_forward(dev(x, t), wd, bd, head, dev(u), mask, packed=pk if packed else None)
    if pipelined and mask:
        assert ogemm.rel_frobenius(policy, host(p)) < 2e-5 and (host(a) != action).mean() < 1e-3
        assert (host(a) == orow.discrete_sampling(host(p), u)).all() and (host(p)[:, mask:] == 0).all()
    else:
        assert (host(p) == policy).all() and (host(a) == action).all()
    step = 16384
    for lo in range(0, batch, step):
        hi = min(batch, lo + step)
        p, a = LY.mlp_forward(dev(x[lo:hi], t), None, bd, head, dev(u[lo:hi]), mask, packed=pk)
        if pipelined:
            assert ogemm.rel_frobenius(policy[lo:hi], host(p)) < 2e-5, lo
            assert (host(a) != action[lo:hi]).mean() < 1e-3, lo
        else:
            assert (host(p) == policy[lo:hi]).all() and (host(a) == action[lo:hi]).all(), lo


def test_resident_kernel_run_to_run_and_philox(LY):
    """The resident kernel gives the same bits on every launch, and with a Philox stream in place of the uniforms tensor
    it draws for every tile of its walk what sp_philox_uniforms hands out for those rows."""
    from ml import _lib, primitives
    announce("mlp resident run-to-run + philox")
    rng = np.random.default_rng(41)
    batch, dims = 24 * 5632, [32, 256, 256, 256, 64]
    x, ws, _ = make_problem(rng, batch, dims, "f16")
    xd, wd = dev(x, torch.float16), [dev(w, torch.float16) for w in ws]
    pk = LY.pack_weights(wd)
    cfg = primitives.philox(_lib.PHILOX_LAYER, blocks_per_grid=24, rows_per_block=5632)
    u = primitives.philox_uniforms(cfg, batch, 64)
    for packed in (pk, None):
        first = [t.clone() for t in LY.mlp_forward(xd, wd, None, "softmax", u, 3, packed=packed)]
        for _ in range(2):
            again = LY.mlp_forward(xd, wd, None, "softmax", u, 3, packed=packed)
            assert all(torch.equal(a, b) for a, b in zip(first, again))
        drawn = LY.mlp_forward(xd, wd, None, "softmax", None, 3, packed=packed, rng=cfg)
        assert all(torch.equal(a, b) for a, b in zip(first, drawn))
        assert (host(first[1]) == orow.discrete_sampling(host(first[0]), host(u))).all()


@pytest.mark.parametrize("members,batch,dims,head,mask,sample", [
    (32, 6144, [128, 64, 64], "regret_matching", 3, None),      # the reference's Leduc policy: 3 valid of 64 columns, no sampling
    (5, 1000, [128, 64, 64], "softmax", 3, "u"),                 # ragged last tile, uniforms from a tensor
    (3, 4100, [64, 64, 4], "softmax_regret_matching", 0, "u"),   # a head 4 wide, no mask: dense rows
    (7, 777, [24, 64, 6], "regret_matching", 2, "philox"),       # K0 not a multiple of 32, row width not a multiple of 4
    (300, 64, [8, 64, 64], "softmax", 4, "philox"),              # more members than compute units
])
def test_ensemble_forward(LY, members, batch, dims, head, mask, sample):
    """sp_mlp_forward_ensemble -- every member's relu(x.W1^T).W2^T + head in one launch -- against the oracle's
    forward of each member on its own (f32: relative Frobenius error below 1e-5, the f32 bar), zeros behind the
    mask, and actions bit-exact given the kernel's own policy and the member's uniforms."""
    from ml import _lib, primitives
    from oracle import philox as ophilox
    announce("mlp ensemble members=%d batch=%d dims=%s head=%s mask=%d sample=%s" % (members, batch, dims, head, mask, sample))
    rng = np.random.default_rng(members * 1000 + batch)
    x = rng.standard_normal((batch, dims[0]), dtype=np.float32)
    w1 = rng.standard_normal((members, dims[1], dims[0]), dtype=np.float32) * np.float32(1 / np.sqrt(dims[0]))
    w2 = rng.standard_normal((members, dims[2], dims[1]), dtype=np.float32) * np.float32(1 / np.sqrt(dims[1]))
    u, cfg = None, None
    if sample == "u":
        u = (1 - rng.random((members, batch), dtype=np.float32)).astype(np.float32)
    elif sample == "philox":
        # the stacked rows of the members, each member a run of its own `member_draws` further into every thread's stream
        cols = dims[2] if dims[2] % 4 == 0 else 8
        cfg = primitives.philox(_lib.PHILOX_LAYER, blocks_per_grid=1, rows_per_block=batch, member_rows=batch, member_draws=12)
        u = host(primitives.philox_uniforms(cfg, members * batch, cols)).reshape(members, batch)
        if dims[2] % 4 != 0:
            sample = "u"          # (a Philox stream needs 16-byte rows: such a head takes the same numbers as a tensor)
    out = LY.mlp_forward_ensemble(dev(x), (dev(w1), dev(w2)), head, dev(u) if sample == "u" else None, mask,
                                  rng=cfg if sample == "philox" else None)
    policy, action = (host(out[0]), host(out[1])) if sample else (host(out), None)
    assert policy.shape == (members, batch, dims[2])
    for e in range(members):
        want, _, _ = olayers.mlp_forward(x, [w1[e], w2[e]], None, HEAD_CODE[head], None, None, mask or None)
        assert ogemm.rel_frobenius(policy[e], want) < 1e-5, e
        if mask:
            assert (policy[e][:, mask:] == 0).all()
        assert np.abs(policy[e].sum(axis=1) - 1).max() < 1e-5
        if sample:
            assert (action[e] == orow.discrete_sampling(policy[e], u[e])).all(), e
    if sample:
        assert len(np.unique(action)) > 1


def test_ensemble_rejects_what_it_does_not_take(LY):
    from ml import _lib
    x = torch.zeros((64, 128), dtype=torch.float32, device="cuda")
    w1 = torch.zeros((2, 64, 128), dtype=torch.float32, device="cuda")
    with pytest.raises(_lib.SpiralError) as err:      # 64 computed outputs: left to the node-by-node pass
        LY.mlp_forward_ensemble(x, (w1, torch.zeros((2, 64, 64), dtype=torch.float32, device="cuda")), "softmax")
    assert err.value.code == -2
    with pytest.raises(_lib.SpiralError) as err:      # a hidden layer of another width
        LY.mlp_forward_ensemble(x, (torch.zeros((2, 32, 128), dtype=torch.float32, device="cuda"),
                                    torch.zeros((2, 4, 32), dtype=torch.float32, device="cuda")), "softmax")
    assert err.value.code == -2


@pytest.mark.parametrize("k0", [32, 40, 56, 64, 72, 104, 120, 128, 136, 248, 256])
def test_ensemble_weights_of_every_row_length(LY, k0):
    """The first layer's weights come through LDS, in pieces whose row follows from a multiplication: weights that are one
    in one column (feature, or output, i in column 5 i + 3 mod k0) hand that column of the inputs on, exactly."""
    announce("ensemble weights k0=%d" % k0)
    members, batch = 3, 33
    x = (torch.randn((batch, k0), generator=torch.Generator().manual_seed(k0)) + 0.25).cuda()

    def one_each(rows, e):
        w = torch.zeros((rows, k0))
        col = (5 * torch.arange(rows) + 3 + 7 * e) % k0
        w[torch.arange(rows), col] = 1
        return w, col

    picked = [one_each(32, e) for e in range(members)]
    got = LY.ensemble_binarize(x, torch.stack([w for w, _ in picked]).cuda(), 1 << 31).cpu()
    for e, (_, col) in enumerate(picked):
        want = orow.binarize(x.cpu()[:, col].numpy(), 1 << 31)
        assert (host(got[e]).view(np.uint32) == want).all(), e
    picked = [one_each(4, e) for e in range(members)]             # one layer under a head: four rows, straight or through LDS
    got = LY.mlp_forward_ensemble(x, (torch.stack([w for w, _ in picked]).cuda(),), None)
    for e, (_, col) in enumerate(picked):
        assert torch.equal(got[e].cpu(), x.cpu()[:, col])
    if k0 > 128:
        return                     # (two layers: up to 128 inputs)
    picked = [one_each(64, e) for e in range(members)]
    w2 = torch.zeros((members, 4, 64))
    feature = torch.tensor([0, 21, 42, 63])
    w2[:, torch.arange(4), feature] = 1
    got = LY.mlp_forward_ensemble(x, (torch.stack([w for w, _ in picked]).cuda(), w2.cuda()), "regret_matching").cpu()
    for e, (_, col) in enumerate(picked):
        y = x.cpu()[:, col[feature]].clamp(min=0).numpy()
        want, _, _ = olayers.mlp_forward(y, [np.eye(4, dtype=np.float32)], None, HEAD_CODE["regret_matching"], None, None, None)
        assert np.abs(got[e].numpy() - want).max() < 1e-6, e     # (a sum of four, a division: a few ulp of at most one)


@pytest.mark.parametrize("members,batch,k0,n,head,mask,sample", [
    (4, 6144, 128, 64, "regret_matching", 3, None),     # the reference's hold'em CEM policy: one layer, 3 valid of 64 columns
    (6, 1000, 256, 64, "softmax", 4, "u"),              # the widest input, a ragged last tile, sampling
    (3, 333, 40, 3, "softmax_regret_matching", 0, "u"),  # input width not a multiple of 32, a dense 3-wide head
])
def test_single_layer_ensemble_forward(LY, members, batch, k0, n, head, mask, sample):
    """sp_mlp_forward_ensemble with ONE layer per member (policy[e] = head(x . W[e]^T), only the head's valid columns
    computed) against the oracle's forward of each member (f32 bar 1e-5), zeros behind the mask, actions exact given
    the kernel's policy."""
    announce("ensemble single layer members=%d batch=%d k0=%d n=%d head=%s mask=%d" % (members, batch, k0, n, head, mask))
    rng = np.random.default_rng(members + batch + k0)
    x = rng.standard_normal((batch, k0), dtype=np.float32)
    w = rng.standard_normal((members, n, k0), dtype=np.float32) * np.float32(1 / np.sqrt(k0))
    u = (1 - rng.random((members, batch), dtype=np.float32)).astype(np.float32) if sample else None
    out = LY.mlp_forward_ensemble(dev(x), (dev(w),), head, dev(u) if sample else None, mask)
    policy, action = (host(out[0]), host(out[1])) if sample else (host(out), None)
    for e in range(members):
        want, _, _ = olayers.mlp_forward(x, [w[e]], None, HEAD_CODE[head], None, None, mask or None)
        assert ogemm.rel_frobenius(policy[e], want) < 1e-5, e
        if mask:
            assert (policy[e][:, mask:] == 0).all()
        if sample:
            assert (action[e] == orow.discrete_sampling(policy[e], u[e])).all(), e


@pytest.mark.parametrize("members,batch,k0,n,modulo", [
    (4, 6144, 128, 128, 1 << 12),     # the reference's CFR models: 128 outputs hashed into 4096 worlds
    (5, 1001, 256, 20, 1000003),      # fewer than 32 columns, a modulus that is not a power of two, a ragged last tile
    (3, 64, 24, 40, 1 << 31),         # every one of the 32 counted bits kept
])
def test_ensemble_binarize(LY, members, batch, k0, n, modulo):
    """sp_ensemble_binarize (one ensemble layer + the hash head, the product never written) against the oracle's
    binarize of the oracle's product.  A bit can only differ where an output is so close to zero that the order of the
    sum decides its sign: such entries are left out of the comparison (and are counted: there must be next to none)."""
    from ml import primitives
    announce("ensemble binarize members=%d batch=%d k0=%d n=%d modulo=%d" % (members, batch, k0, n, modulo))
    rng = np.random.default_rng(members * 7 + batch + n)
    x = rng.standard_normal((batch, k0), dtype=np.float32)
    w = rng.standard_normal((members, n, k0), dtype=np.float32)
    got = host(LY.ensemble_binarize(dev(x), dev(w), modulo)).view(np.uint32)
    assert got.shape == (members, batch)
    close = 0
    for e in range(members):
        y = ogemm.gemm_abt(x, w[e])
        want = orow.binarize(y, modulo)
        sure = (np.abs(y[:, :32]) > 1e-4).all(axis=1)       # rows whose counted outputs are all clear of zero
        close += int((~sure).sum())
        assert (got[e][sure] == want[sure]).all(), e
        # and exactly the node-by-node result on the same product computed by the library's own GEMM
    assert close < 0.02 * members * batch
    # the row kernel on the library's own product gives the same words wherever the signs are not in question
    from ml import matmul
    y0 = matmul.matmul_abt(dev(x), dev(w[0]))
    node = host(primitives.binarize(y0, modulo)).view(np.uint32)
    sure0 = (np.abs(host(y0)[:, :32]) > 1e-4).all(axis=1)
    assert (node[sure0] == got[0][sure0]).all()


# The ensemble on the bf16 pipe, and calls on the other side of its rule: rounds of 1, 2, ... 9 tiles of 32 rows, a ragged last tile, widths of
# a step of 16 and odd halves of one, rows of 4, 16, 20 and 64 columns, 1 to 4 outputs, a width that is no multiple of 4
@pytest.mark.parametrize("members,batch,dims,head,mask,sample", [
    (3, 31, [8, 64, 4], "softmax", 0, True), (4, 32 * 256 + 1, [16, 64, 16], "regret_matching", 2, False),
    (5, 32 * 128 * 3, [24, 64, 20], "softmax", 3, False), (5, 32 * 128 * 4 - 17, [40, 64, 64], "softmax_regret_matching", 4, True),
    (6, 32 * 128 * 5 + 9, [64, 64, 64], "regret_matching", 3, False), (7, 32 * 128 * 2 + 32, [72, 64, 6], "softmax", 1, True),
    (4, 32 * 256 * 6 + 33, [128, 64, 8], "none", None, False), (9, 32 * 85 * 7 + 40, [120, 64, 64], "regret_matching", 4, False),
    (9, 32 * 85 * 8, [128, 64, 64], "softmax", 3, True), (256, 200, [48, 64, 12], "regret_matching", 3, False),
    (4, 32 * 1024 + 1, [16, 64, 16], "regret_matching", 2, False), (7, 32 * 600 - 5, [24, 64, 20], "softmax", 3, True),
    (6, 32 * 690 + 9, [64, 64, 64], "regret_matching", 3, False), (300, 32 * 17 + 1, [40, 64, 12], "softmax", 4, True),
    (768, 1, [128, 64, 64], "softmax", 3, True), (800, 31, [8, 64, 4], "softmax", 0, True), (1021, 64, [24, 64, 16], "regret_matching", 2, False),
    (900, 96, [104, 64, 20], "softmax", 3, False), (513, 129, [64, 64, 64], "softmax_regret_matching", 4, True),
    (900, 160, [16, 64, 6], "softmax", 1, True), (777, 224, [120, 64, 8], "none", None, False), (900, 265, [32, 64, 64], "softmax", 3, True)])
def test_ensemble_in_three_parts(LY, members, batch, dims, head, mask, sample):
    """Against float64: the hidden layer no further off than f32 sums are, so the f32 bar of the head holds row by row wherever the
    head itself is not the quotient of two small numbers; exact zeros behind the mask; actions given the kernel's own policy."""
    announce("ensemble parts members=%d batch=%d dims=%s head=%s mask=%s" % (members, batch, dims, head, mask))
    if head == "none":
        dims = dims[:2] + [4]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(batch)
    x = torch.randn((batch, dims[0]), generator=gen, device="cuda")
    w1 = torch.randn((members, 64, dims[0]), generator=gen, device="cuda") / dims[0] ** 0.5
    w2 = torch.randn((members, dims[2], 64), generator=gen, device="cuda") / 8
    u = 1 - torch.rand((members, batch), generator=gen, device="cuda") if sample else None
    out = LY.mlp_forward_ensemble(x, (w1, w2), head, u, mask or 0)
    policy, action = out if sample else (out, None)
    cols = mask or dims[2]
    assert (policy[:, :, cols:] == 0).all()
    for e in range(members):
        z = torch.relu(x.double() @ w1[e].double().T) @ w2[e, :cols].double().T
        if head in ("softmax", "softmax_regret_matching"):
            z = torch.softmax(z, 1)
        got = policy[e, :, :cols].double()
        if head == "regret_matching":
            z = torch.relu(z)
            total = z.sum(1, keepdim=True)
            clear = (total > 0.01).squeeze(1)
            assert clear.any()
            z, got = (z / total)[clear], got[clear]
        assert ((got - z).norm() / z.norm()).item() < 1e-5, e
        if sample:
            assert (host(action[e]) == orow.discrete_sampling(host(policy[e]), host(u[e]))).all(), e


def test_ensemble_in_three_parts_keeps_what_parts_cannot_hold(LY):
    """Members 0 and 1 of four on the bf16 pipe against the same two alone on the f32 kernel, hidden features as they are: inputs and
    weights with infinities, NaN, values whose bf16 is infinite and values above 2^60, weights below 2^-94.  Infinities where the
    f32 kernel has them, the rest to f32 sums of 128 terms, either of which is off by less than 16 roundings of the row's norm."""
    announce("ensemble parts, special values")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    batch = 65536
    x = torch.randn((batch, 128), generator=gen, device="cuda")
    w1 = torch.randn((4, 64, 128), generator=gen, device="cuda") / 11
    w2, features = hidden_features(4)
    x[3, 5] = float("inf")
    x[40, 7] = float("-inf")
    x[100, 0] = float("nan")
    x[200] *= 2.0 ** -125
    x[300] = 0.0
    x[300, 9] = 3.4028234e38
    x[batch - 1] *= 2.0 ** 90
    for scale, poison in ((1.0, None), (1.0, float("inf")), (2.0 ** -118, None), (2.0 ** 70, None)):
        w = w1.clone()
        w[1] *= scale
        if poison is not None:
            w[1, features[1][2], 3] = poison
        four = LY.mlp_forward_ensemble(x, (w, w2), "none")
        two = LY.mlp_forward_ensemble(x, (w[:2].contiguous(), w2[:2].contiguous()), "none")
        a, b = four[:2].double(), two.double()
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
        for e in range(2):
            norms = x.double().norm(dim=1, keepdim=True) * w[e, features[e]].double().norm(dim=1)
            ok = b[e].isfinite() & norms.isfinite()
            assert ok.sum().item() > (0.9 if poison is None else 0.3) * ok.numel()       # (a feature that is infinite makes all four NaN: 0 x inf)
            assert ((a[e] - b[e]).abs()[ok] <= 32 * 2.0 ** -24 * norms[ok] + 128 * 2.0 ** -149).all()
            assert (a[e][ok] != 0).any()


def few(gen, m, k, terms):
    at = torch.rand((m, k), generator=gen, device="cuda").topk(terms).indices
    return torch.zeros((m, k), device="cuda").scatter_(1, at, torch.randn((m, terms), generator=gen, device="cuda"))


PARTS_INPUTS = {
    "normal": lambda gen, m, k: torch.randn((m, k), generator=gen, device="cuda"),
    "uniform": lambda gen, m, k: torch.rand((m, k), generator=gen, device="cuda"),
    "relu": lambda gen, m, k: torch.randn((m, k), generator=gen, device="cuda").relu(),
    "features": lambda gen, m, k: (torch.rand((m, k), generator=gen, device="cuda") < 0.2).float(),
    "lognormal": lambda gen, m, k: torch.randn((m, k), generator=gen, device="cuda") * torch.exp(2 * torch.randn((m, k), generator=gen, device="cuda")),
    "eight": lambda gen, m, k: few(gen, m, k, 8), "two": lambda gen, m, k: few(gen, m, k, 2), "one": lambda gen, m, k: few(gen, m, k, 1)}


def hidden_features(members):
    """Second layers that pass features (11 e + 17 o) % 64, o < 4, of member e on as they are, and those features."""
    features = [[(11 * e + 17 * o) % 64 for o in range(4)] for e in range(members)]
    w2 = torch.zeros((members, 4, 64), device="cuda")
    for e in range(members):
        w2[e, torch.arange(4), torch.tensor(features[e])] = 1.0
    return w2, features


@pytest.mark.parametrize("inputs", sorted(PARTS_INPUTS))
@pytest.mark.parametrize("k0", [16, 64, 120])
def test_ensemble_in_three_parts_is_no_further_off_than_in_f32(LY, k0, inputs):
    """Six members on the bf16 pipe against two of them alone, which f32 MFMAs take: the error of the hidden layer against float64
    (2-norm) is no larger.  A single product is rounded once: to the nearest but for 3 in 1000, and those within 2^-7 of that."""
    announce("ensemble parts error k0=%d %s" % (k0, inputs))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(k0)
    x = PARTS_INPUTS[inputs](gen, 65536, k0)
    w1 = torch.randn((6, 64, k0), generator=gen, device="cuda") / k0 ** 0.5
    w2, features = hidden_features(6)
    parts = LY.mlp_forward_ensemble(x, (w1, w2), "none")[:2]
    f32 = LY.mlp_forward_ensemble(x, (w1[:2].contiguous(), w2[:2].contiguous()), "none")
    want = torch.stack([torch.relu(x.double() @ w1[e, features[e]].double().T) for e in range(2)])
    assert (parts.double() - want).norm() <= 1.005 * (f32.double() - want).norm()
    if inputs == "one":
        assert (parts != want.float()).double().mean().item() < 3e-3
        assert ((parts.double() - want).abs() <= 2.0 ** -24 * (1 + 2.0 ** -7) * want).all()


@pytest.mark.parametrize("x_exp,w_exp", [(-60, 0), (-105, 50), (-126, 58), (-149, 58), (58, -93), (58, -110), (40, -130), (-70, -66)])
def test_ensemble_in_three_parts_of_tiny_numbers(LY, x_exp, w_exp):
    """Inputs down to the smallest subnormal and weights down to 2^-94 are held by their parts, smaller weights send their member
    through f32 MFMAs: in every row as close as f32 sums are, also where the lowest parts are subnormal bf16 or (the last case)
    the products subnormal f32, which are rounded to multiples of 2^-149."""
    announce("ensemble parts, tiny numbers 2^%d 2^%d" % (x_exp, w_exp))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    k0 = 128
    x = torch.randint(-2 ** 20, 2 ** 20, (65536, k0), generator=gen, device="cuda").float() * 2.0 ** (-20 if x_exp > -149 else 0)
    x = (x.double() * 2.0 ** x_exp).float()
    w1 = torch.randn((6, 64, k0), generator=gen, device="cuda")
    w1[1] *= 2.0 ** w_exp
    w1[2] = (w1[2].double() * 2.0 ** w_exp).float()
    w2, features = hidden_features(6)
    got = LY.mlp_forward_ensemble(x, (w1, w2), "none")
    for e in (1, 2):
        w = w1[e, features[e]].double()
        want, scale = torch.relu(x.double() @ w.T), x.double().norm(dim=1, keepdim=True) * w.norm(dim=1)
        off = (got[e].double() - want).abs()
        assert (off <= 2.0 ** -24 * 16 * scale + 2.0 ** -149 * k0).all()
        assert x_exp + w_exp < -120 or (off.norm() / want.norm()).item() < 2.0 ** -24 * (k0 / 2) ** 0.5 + 1e-7


@pytest.mark.parametrize("k0", [32, 64, 128])
def test_ensemble_in_three_parts_keeps_rows_and_members_their_own(LY, k0):
    """Rows with inputs that parts cannot hold, and a member with such weights, change nothing in other rows and members; and where
    rows and members lie does not matter either: all to the last bit."""
    announce("ensemble parts, rows and members of their own k0=%d" % k0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(k0)
    batch = 65536
    x = torch.randn((batch, k0), generator=gen, device="cuda")
    w1, w2 = torch.randn((6, 64, k0), generator=gen, device="cuda") / 8, torch.randn((6, 16, 64), generator=gen, device="cuda") / 8
    w1[4, 60, 1] = 0.0
    clean, _ = LY.mlp_forward_ensemble(x, (w1, w2), "softmax", torch.ones((6, batch), device="cuda"), mask_size=3)
    odd = x.clone()
    odd[3, 5], odd[40, 7], odd[100, 0], odd[20000] = float("inf"), float("-inf"), float("nan"), 1e20
    odd[300], odd[batch - 1] = odd[300] * 2.0 ** -130, odd[batch - 1] * 2.0 ** 90
    w = w1.clone()
    w[1, 9, 3] = float("inf")
    w[4, 60, 1] = 1e-35
    policy = LY.mlp_forward_ensemble(odd, (w, w2), "softmax", mask_size=3)
    rest = torch.ones(batch, dtype=torch.bool, device="cuda")
    rest[[3, 40, 100, 300, 20000, batch - 1]] = False
    for e in (0, 2, 3, 5):
        assert torch.equal(policy[e, rest], clean[e, rest])
    assert torch.allclose(policy[4, rest], clean[4, rest], rtol=0, atol=1e-5)
    rows, members = torch.randperm(batch, generator=gen, device="cuda"), torch.randperm(6, generator=gen, device="cuda")
    moved = LY.mlp_forward_ensemble(x[rows], (w1[members].contiguous(), w2[members].contiguous()), "softmax", mask_size=3)
    assert torch.equal(moved, clean[members][:, rows])


@pytest.mark.parametrize("name", ["mlp_forward_ensemble_parts", "mlp_forward_ensemble_parts_action"])
def test_the_parts_ensemble_kernels_are_named(name):
    announce("kernel info " + name)
    from ml import _lib
    info = _lib.kernel_info(name)
    assert info["threads_per_block"] == 512 and 0 < info["vgprs"] <= 256
