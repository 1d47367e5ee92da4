"""sp_stack_forward_f32 on the launch shapes a graph of ordinary size does not reach: several tiles per wave (inputs read
ahead, one draw for four tiles, the scratch used again), eight waves a workgroup, every instance of the kernel, uniforms given or
drawn.  Probabilities against float64 (f32 sums of up to 128 terms in up to three layers and an exponential to 1e-6: 1e-5 in the
Frobenius norm); sampled indices bit for bit given the kernel's own probabilities and the uniforms."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import philox as ophilox, row_ops as orow
from gpu_util import announce, dev, host

pytestmark = pytest.mark.gpu

ACT = {"copy": 0, "relu": 1, "tanh": 2, "sigmoid": 3}
LN = 0x100


@pytest.fixture(scope="module")
def S():
    from ml import _lib
    return _lib


def forward(S, x, ws, acts, head, mask=0, u=None, rng=None, sample=True):
    members, rows, n = ws[0].shape[0], x.shape[0], ws[-1].shape[1]
    policy = torch.full((members, rows, n), 7.0, device="cuda")
    action = torch.full((members, rows), -7, dtype=torch.int32, device="cuda") if sample else None
    k, dims = len(ws), [x.shape[1]] + [w.shape[1] for w in ws]
    codes = [sum(ACT.get(part, LN) for part in act.split("+")) for act in acts] + [0]
    S.check(S.lib.sp_stack_forward_f32(S.ptr(x), k, (C.c_void_p * k)(*[S.ptr(w) for w in ws]), (C.c_int32 * (k + 1))(*dims),
                                       (C.c_int32 * k)(*codes), members, S.ptr(u), C.byref(rng) if rng is not None else None,
                                       S.ptr(policy), S.ptr(action), rows, head, mask, S.stream_ptr()))
    return policy, action


def probabilities(x, ws, acts, regret, mask):
    """In float64, a member at a time."""
    out = []
    for e in range(ws[0].shape[0]):
        h = x.double()
        for w, act in zip(ws, acts + [""]):
            h = h @ w[e].double().T
            for part in [p for p in act.split("+") if p]:
                if part == "ln":
                    s = (h * h).sum(-1, keepdim=True)
                    h = torch.where(s != 0, h / s, torch.zeros_like(h))
                else:
                    h = {"copy": lambda t: t, "relu": torch.relu, "tanh": torch.tanh, "sigmoid": torch.sigmoid}[part](h)
        valid = torch.arange(h.shape[-1], device=h.device) < (mask or h.shape[-1])
        if regret:
            p = torch.where(valid, torch.relu(h), torch.zeros_like(h))
            s = p.sum(-1, keepdim=True)
            p = torch.where(s != 0, p / s, valid.double() / valid.sum())
        else:
            p = torch.softmax(torch.where(valid, h, torch.full_like(h, -np.inf)), -1)
        out.append(p)
    return torch.stack(out)


def make(rng, members, rows, widths, scale=0.3):
    x = dev(rng.standard_normal((rows, widths[0]), dtype=np.float32))
    return x, [dev(rng.standard_normal((members, o, i), dtype=np.float32) * np.float32(scale / np.sqrt(i / 16)))
               for i, o in zip(widths[:-1], widths[1:])]


def check(S, x, ws, acts, head, mask, u, rng):
    """u: (members * rows,) uniforms the run is to use, given as they are (rng None) or drawn on the device."""
    members, rows, n = ws[0].shape[0], x.shape[0], ws[-1].shape[1]
    policy, action = forward(S, x, ws, acts, head, mask, dev(u) if rng is None else None, rng)
    want = probabilities(x, ws, acts, head in (S.ROW_REGRET_MATCHING, S.ROW_MASKED_REGRET_MATCHING), mask)
    assert float((policy.double() - want).norm() / want.norm()) < 1e-5
    p, a = host(policy).reshape(-1, n), host(action).reshape(-1)
    assert (p[:, mask or n:] == 0).all()
    assert (a == orow.discrete_sampling(p, u, order="wave")).all()
    again, none = forward(S, x, ws, acts, head, mask, sample=False)
    assert torch.equal(again, policy) and none is None


def uniforms(rng, n):
    return (1 - rng.random(n, dtype=np.float32)).astype(np.float32)


# 64 wide stacks: 512 workgroups of eight waves, 16 rows a wave and turn; 128 wide ones: 256 workgroups
@pytest.mark.parametrize("members,rows,widths,acts,head,mask", [
    (1, 5 * 65536 + 37, (64, 64, 64, 64), "ln+relu", "ROW_SOFTMAX", 0),                 # six turns, the last tile of five rows
    (3, 8 * 21888 + 3, (64, 64, 16), "relu", "ROW_SOFTMAX", 0),                         # nine turns a member: two refills of the draws
    (16, 16384, (64, 64, 64, 64), "ln+relu", "ROW_MASKED_SOFTMAX", 17),                 # eight waves, two tiles a wave
    (1, 5 * 32768 + 9, (128, 128, 64), "ln+tanh", "ROW_SOFTMAX", 0),                    # full_product of 128 x 128 and 128 x 64
    (2, 40000, (128, 128, 64), "sigmoid", "ROW_REGRET_MATCHING", 0),
    (5, 33000, (36, 48, 96, 24), "relu", "ROW_SOFTMAX", 0)])                            # narrow layers, several turns
def test_many_tiles_per_wave(S, members, rows, widths, acts, head, mask):
    announce("stack, many tiles: %d x %d rows %s %s" % (members, rows, widths, head))
    rng = np.random.default_rng(rows)
    x, ws = make(rng, members, rows, widths)
    check(S, x, ws, [acts] * (len(widths) - 2), getattr(S, head), mask, uniforms(rng, members * rows), None)


@pytest.mark.parametrize("widths,head,mask", [
    ((64, 64, 64, 64), "ROW_SOFTMAX", 0), ((52, 64, 64), "ROW_REGRET_MATCHING", 0),      # full, the second with a part of a K-block
    ((64, 64, 20), "ROW_MASKED_REGRET_MATCHING", 9), ((4, 16, 4), "ROW_SOFTMAX", 0),     # a narrow head behind full layers; not full
    ((128, 128, 64), "ROW_MASKED_SOFTMAX", 64), ((116, 128, 48), "ROW_REGRET_MATCHING", 0), ((128, 64), "ROW_SOFTMAX", 0),
    ((100, 32, 128, 40), "ROW_MASKED_SOFTMAX", 33), ((128, 16, 16, 16, 16, 16, 16, 16, 8), "ROW_SOFTMAX", 0)])
@pytest.mark.parametrize("rows", [1, 16, 47])
def test_every_instance(S, rows, widths, head, mask):
    announce("stack instance %s %s rows=%d" % (widths, head, rows))
    rng = np.random.default_rng(rows + widths[0])
    x, ws = make(rng, 3, rows, widths)
    check(S, x, ws, ["ln+relu", "tanh", "copy", "ln+sigmoid", "ln+copy", "sigmoid", "relu"][:len(widths) - 2], getattr(S, head), mask,
          uniforms(rng, 3 * rows), None)


@pytest.mark.parametrize("members,tiles_per_unit,short,widths,acts,head,mask", [
    (1, 1, 5, (64, 64, 64, 64), "ln+relu", "ROW_SOFTMAX", 0), (1, 1, 0, (108, 64, 32), "tanh", "ROW_MASKED_SOFTMAX", 3),
    (4, 1, 15, (4, 16, 4), "ln+copy", "ROW_REGRET_MATCHING", 0), (1, 2, 17, (116, 128, 96, 64), "ln+sigmoid", "ROW_SOFTMAX", 0),
    (2, 2, 7, (80, 112, 20), "relu", "ROW_MASKED_REGRET_MATCHING", 17), (1, 2, 1, (36, 16, 128, 16, 16, 16, 16, 16, 48), "ln+relu", "ROW_SOFTMAX", 0)])
def test_rows_of_few_are_those_of_many(S, members, tiles_per_unit, short, widths, acts, head, mask):
    """Up to a tile of 16 rows per compute unit (two of wide layers) the waves share the features, beyond that the rows: a row's
    result is the same bit for bit, at the last batch before the rule's line and, as part of a larger one, behind it."""
    announce("stack, few rows %d x %d tiles per unit %s %s" % (members, tiles_per_unit, widths, head))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    few = 16 * tiles_per_unit * cus // members - short
    many = 16 * (2 * cus + 16)
    rng = np.random.default_rng(few)
    x, ws = make(rng, members, many, widths)
    u = dev(uniforms(rng, members * many).reshape(members, many))
    names = [acts] * (len(widths) - 2)
    p, a = forward(S, x[:few].contiguous(), ws, names, getattr(S, head), mask, u[:, :few].contiguous())
    want_p, want_a = forward(S, x, ws, names, getattr(S, head), mask, u)
    assert torch.equal(p, want_p[:, :few]) and torch.equal(a, want_a[:, :few])
    check(S, x[:few].contiguous(), ws, names, getattr(S, head), mask, host(u[:, :few].contiguous()).reshape(-1), None)


@pytest.mark.parametrize("members,blocks,rows_per_block,widths", [(3, 24, 9101, (64, 64, 64)), (2, 7, 5, (128, 128, 16)), (1, 24, 13655, (32, 64, 8))])
def test_uniforms_drawn_on_the_device(S, members, blocks, rows_per_block, widths):
    """A run per member (member_rows), later in the stream each, and one run over all members' rows."""
    from ml import primitives as P
    rows, n = blocks * rows_per_block, widths[-1]
    announce("stack draws: %d x %d rows %s" % (members, rows, widths))
    rng = np.random.default_rng(rows)
    x, ws = make(rng, members, rows, widths)
    draws = ophilox.draws_per_sampling_node(rows_per_block, n)
    layer = P.philox(S.PHILOX_LAYER, blocks_per_grid=blocks, rows_per_block=rows_per_block, offset=4, member_rows=rows, member_draws=draws)
    u = np.concatenate([ophilox.row_uniforms_layer(blocks, rows_per_block, n, offset=4 + e * draws) for e in range(members)])
    check(S, x, ws, ["relu"] * (len(widths) - 2), S.ROW_SOFTMAX, 0, u, layer)
    grid = P.philox(S.PHILOX_GRID, blocks_per_grid=24)
    check(S, x, ws, ["relu"] * (len(widths) - 2), S.ROW_SOFTMAX, 0, ophilox.row_uniforms_grid(members * rows, n), grid)


def test_rows_of_nan_and_infinity_stay_their_own(S):
    announce("stack, NaN and infinite rows")
    rng = np.random.default_rng(1)
    x, ws = make(rng, 2, 100, (64, 64, 64, 16))
    u = dev(uniforms(rng, 200))
    clean, picks = forward(S, x, ws, ["ln+relu", "ln+relu"], S.ROW_SOFTMAX, 0, u)
    bad = x.clone()
    bad[17], bad[40, 3], bad[99] = float("nan"), float("inf"), float("-inf")
    policy, action = forward(S, bad, ws, ["ln+copy", "ln+copy"], S.ROW_SOFTMAX, 0, u)
    mixed, mixed_picks = forward(S, bad, ws, ["ln+relu", "ln+relu"], S.ROW_SOFTMAX, 0, u)
    rest = [r for r in range(100) if r not in (17, 40, 99)]
    assert torch.equal(mixed[:, rest], clean[:, rest]) and torch.equal(mixed_picks[:, rest], picks[:, rest])
    assert bool(policy[:, [17, 40, 99]].isnan().all()) and bool((action[:, [17, 40, 99]] == 2147483647).all())


# ---- full 64 wide stacks of enough rows: the products as three bf16 parts ----
@pytest.mark.parametrize("members,rows,widths,acts,head,mask", [
    (1, 65521, (64, 64, 64), "ln+relu", "ROW_SOFTMAX", 0),                              # the fewest tiles, the last of one row
    (1, 131057, (52, 64), "", "ROW_REGRET_MATCHING", 0),                                # one layer, a part of a K-block
    (5, 30011, (64, 64, 64, 60), "tanh", "ROW_MASKED_SOFTMAX", 49),                     # workgroups that do not divide the units; masked
    (200, 330, (56, 64, 64), "ln+sigmoid", "ROW_SOFTMAX", 0),                           # (f32: half of the turns without a tile)
    (300, 500, (64, 64, 64), "relu", "ROW_SOFTMAX", 0),                                 # (f32: units idle)
    (200, 500, (56, 64, 64), "ln+sigmoid", "ROW_SOFTMAX", 0),                           # a workgroup a member
    (450, 500, (64, 64, 64), "relu", "ROW_SOFTMAX", 0),                                 # more members than units, the fewest tiles
    (300, 500, (64, 64, 64, 64, 64), "relu", "ROW_MASKED_REGRET_MATCHING", 50)])        # four layers
def test_parts(S, members, rows, widths, acts, head, mask):
    announce("stack in parts: %d x %d rows %s %s" % (members, rows, widths, head))
    rng = np.random.default_rng(rows)
    x, ws = make(rng, members, rows, widths)
    check(S, x, ws, [acts] * (len(widths) - 2), getattr(S, head), mask, uniforms(rng, members * rows), None)


@pytest.mark.parametrize("what", ["rows", "weights"])
def test_numbers_that_parts_cannot_hold(S, what):
    """Infinities and numbers above 2^60 in some rows of the input or in a member's weights, and tiny numbers, under heads that make
    them matter (regret matching does not see a row's scale): such rows as the f32 kernel gives them alone (few rows take that
    one), the same bits where every layer's inputs are out of range, and the other rows as they are without them."""
    announce("stack in parts, %s out of range" % what)
    rng = np.random.default_rng(3)
    rows = 32768
    x, ws = make(rng, 2, rows, (64, 64, 64))
    acts, head = ["relu"], S.ROW_REGRET_MATCHING
    clean, _ = forward(S, x, ws, acts, head, sample=False)
    if what == "rows":
        odd = [17, 18, 40, 5000, rows - 1]
        x[17, 3], x[18, 60], x[40, 0] = float("inf"), float("-inf"), float("nan")
        x[5000] *= 2.0 ** -125
        x[rows - 1] *= 2.0 ** 100
        policy, _ = forward(S, x, ws, acts, head, sample=False)
        alone, _ = forward(S, x[odd].contiguous(), ws, acts, head, sample=False)
        assert torch.equal(policy[:, odd[:3]].isnan(), alone[:, :3].isnan())
        assert torch.equal(policy[:, odd[4]], alone[:, 4])
        assert float((policy[:, 5000] - clean[:, 5000]).norm() / clean[:, 5000].norm()) < 1e-6
        rest = torch.ones(rows, dtype=torch.bool, device="cuda")
        rest[odd] = False
        assert torch.equal(policy[:, rest], clean[:, rest])
    else:
        scaled = [w.clone() for w in ws]
        scaled[0][1] *= 2.0 ** 70
        scaled[1][1] *= 2.0 ** -115
        policy, _ = forward(S, x, scaled, acts, head, sample=False)
        alone, _ = forward(S, x[:300].contiguous(), scaled, acts, head, sample=False)
        assert torch.equal(policy[1, :300], alone[1]) and torch.equal(policy[0], clean[0])
        assert float((policy[1] - clean[1]).norm() / clean[1].norm()) < 1e-5
        scaled[0][1], scaled[1][1] = ws[0][1] * 2.0 ** -115, ws[1][1] * 2.0 ** 20
        policy, _ = forward(S, x, scaled, acts, head, sample=False)
        assert torch.equal(policy[0], clean[0])
        assert float((policy[1] - clean[1]).norm() / clean[1].norm()) < 1e-6
        ws[0][1, 5, 7], ws[1][1, 63, 0] = 1e-37, float("-inf")
        policy, _ = forward(S, x, ws, acts, head, sample=False)
        alone, _ = forward(S, x[:300].contiguous(), ws, acts, head, sample=False)
        assert torch.equal(policy[1, :300].isnan(), alone[1].isnan()) and torch.equal(policy[1, :300].nan_to_num(), alone[1].nan_to_num())
        assert torch.equal(policy[0], clean[0])


@pytest.mark.parametrize("inputs", ["normal", "uniform", "relu", "features", "eight", "two", "one"])
@pytest.mark.parametrize("widths,acts", [((64, 64), []), ((56, 64, 64), ["relu"]), ((64, 64, 64, 64), ["tanh", "ln+relu"])])
def test_parts_are_no_further_off_than_f32(S, widths, acts, inputs):
    """All rows at once in parts against a sixteenth of them at a time, which f32 MFMAs take: the error of the probabilities against
    float64 (2-norm) is no larger, whatever the inputs."""
    announce("stack in parts, error %s %s" % (widths, inputs))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(len(widths))
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    rows, k = 131072, widths[0]
    if inputs in ("one", "two", "eight"):
        terms = {"one": 1, "two": 2, "eight": 8}[inputs]
        x = torch.zeros((rows, k), device="cuda").scatter_(1, normal(rows, k).topk(terms).indices, normal(rows, terms))
    else:
        x = {"normal": lambda: normal(rows, k), "uniform": lambda: normal(rows, k).abs().frac(), "relu": lambda: normal(rows, k).relu(),
             "features": lambda: (normal(rows, k) > 0.84).float()}[inputs]()
    ws = [normal(1, b, a) / a ** 0.5 for a, b in zip(widths[:-1], widths[1:])]
    for head in (S.ROW_SOFTMAX, S.ROW_REGRET_MATCHING):
        want = probabilities(x, ws, acts, head == S.ROW_REGRET_MATCHING, 0)
        parts, _ = forward(S, x, ws, acts, head, sample=False)
        f32 = torch.cat([forward(S, part.contiguous(), ws, acts, head, sample=False)[0] for part in x.chunk(16)], dim=1)
        assert not torch.equal(parts, f32)
        assert (parts.double() - want).norm() <= 1.005 * (f32.double() - want).norm()


@pytest.mark.parametrize("x_exp,w_exp", [(-60, 0), (-105, 0), (-140, 58), (-70, -50), (58, -93), (58, -110), (40, -125)])
def test_parts_of_tiny_numbers(S, x_exp, w_exp):
    """A layer and regret matching, which does not see a common factor: inputs down to subnormal numbers are held by their parts,
    and weights down to 2^-94 (smaller ones send their member through f32 MFMAs)."""
    announce("stack in parts, tiny numbers 2^%d 2^%d" % (x_exp, w_exp))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    x = torch.randint(-511, 512, (131072, 64), generator=gen, device="cuda").double() * 2.0 ** (x_exp - 9)
    w = torch.randn((1, 64, 64), generator=gen, device="cuda").double() * 2.0 ** w_exp
    x, ws = x.float(), [w.float()]
    got, _ = forward(S, x, ws, [], S.ROW_REGRET_MATCHING, sample=False)
    want = probabilities(x, ws, [], True, 0)
    assert (got.double() - want).norm() <= 4 * 2.0 ** -24 * want.norm()
    assert ((got.double() - want).norm(dim=2) <= 32 * 2.0 ** -24 * want.norm(dim=2)).all()


@pytest.mark.parametrize("name", ["stack_forward_f32_parts", "stack_forward_f32_parts_regret"])
def test_the_instances_in_parts_are_named(S, name):
    announce("kernel info " + name)
    info = S.kernel_info(name)
    assert info["threads_per_block"] == 1024 and 0 < info["vgprs"] <= 128
