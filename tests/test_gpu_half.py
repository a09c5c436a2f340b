"""fp32 through two fp16 parts per operand (c6_half.h), and the boards that it leaves to three bf16 parts (c6_split.h): at
either side of every line between them, alone, in teams and among others."""
import pytest
import torch

import connect6_amd as c6
from connect6_amd import _lib
from connect6_amd.model import run_forward
from connect6_amd.synthetic import gen_boards, gen_uniform
from oracle import torch_ref as R
from tests.test_gpu_team import _team
from tests.util import rel_l2

pytestmark = pytest.mark.gpu
PREC = _lib.PREC_F32S


def _model(cuda, st):
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(st)
    return model


def _parts(packed, layer):
    """The three parts of a 3x3 layer's weights, [part, cout, cin, tap], as float64."""
    cin, cout = (32, 32, 64, 64, 64, 96, 96)[layer - 1], (32, 64, 64, 64, 96, 96, 96)[layer - 1]
    at = 105 + sum((9 * i // 16) * (o // 32) for i, o in zip((32, 32, 64, 64, 64, 96, 96)[:layer - 1], (32, 64, 64, 64, 96, 96, 96)[:layer - 1]))
    n = 9 * cin // 16 * (cout // 32)
    w = packed.cpu()[3 * 1024 * at:3 * 1024 * (at + n)].view(torch.int16)
    # fragment (tap, 16 channels, cout tile), part, lane (half, row), 8 channels
    w = w.view(9, cin // 16, cout // 32, 3, 2, 32, 8).permute(3, 2, 5, 1, 4, 6, 0)
    return w.reshape(3, cout, cin, 9)


def _units(packed):
    """What each layer's sums are multiplied by (0: the set goes through three parts)."""
    one = (packed.numel() - 208) // 2          # (the set of three parts lies behind it, 256-byte aligned)
    return packed.cpu()[one - 4 * (8 + 544):one - 4 * 544].view(torch.float32).double()


def _factors(packed):
    return 1.0 / _units(packed) / torch.tensor([1.0] + [16.0] * 7).double()


@pytest.mark.parametrize("size", [1.0, 1e-7, 1e-12, 1e5])
@pytest.mark.parametrize("layer", [1, 3, 5, 7])
def test_parts_of_weights(cuda, layer, size):
    """hi + lo / 2048, which is what a 3x3 layer reads, is its weights times a power of two to three units of lo's last bit, and what they
    leave adds up to nothing over a channel's taps; whatever the size of the layer's weights."""
    st = R.init_state(3, "reference")
    w = st[f"convs.{layer}.weight"]
    w[0, 0] = torch.tensor([[1e-3, -1e-4, 1e-6], [0.0, 0.1, -0.05], [1e-9, -1e-12, 3e-13]])
    w *= size
    packed = _model(cuda, st).packed_weights(PREC)
    factor = _factors(packed)[layer]
    want = w.flatten(2).double() * factor
    assert 2.0 ** 14 <= float(want.abs().max()) < 2.0 ** 15 and float(factor.log2()) % 1 == 0
    hi, lo, _ = _parts(packed, layer).view(torch.float16).double().unbind(0)
    left = want - hi - lo / 2048.0
    # half a unit of lo each, a whole one where it is rounded the other way for the sum, and the sum of nine such in one of them
    step = (lo.abs().amax(2, keepdim=True) * 2.0 ** -10 + 2.0 ** -24) / 2048.0   # one unit of the largest lo's last bit
    assert bool((left.abs() <= 3 * step).all())
    assert float((left.sum(2, keepdim=True).abs() / step).mean()) <= 0.02
    # ... and over an output's weights: half a unit of 2^-22 of a weight, at random
    assert bool((left.flatten(1).norm(dim=1) <= 2.0 ** -23 * want.flatten(1).norm(dim=1)).all())


@pytest.mark.parametrize("size", [1.0, 1e-7, 1e-12, 1e5])
def test_parts_of_the_first_layer(cuda, size):
    """... of which all three are read: to 2^-33 of a weight, or half of the third's smallest number."""
    st = R.init_state(3, "reference")
    st["convs.0.weight"] *= size
    packed = _model(cuda, st).packed_weights(PREC)
    factor = _factors(packed)[0]
    w = st["convs.0.weight"].double() * -1.4426950408889634 * factor                # [32, 3, 23, 23]
    assert 2.0 ** 14 / 1.5 <= float(w.abs().max()) < 2.0 ** 15
    rows = torch.zeros(32, 70, 24, dtype=torch.float64)                             # 35 K rows per lane half, (ky, plane)
    rows[:, :69, :23] = w.permute(0, 2, 1, 3).reshape(32, 69, 23)
    # fragment (row, 8 columns), part, lane (half, output), 8 columns
    got = packed.cpu()[:105 * 3 * 1024].view(torch.float16).double().view(35, 3, 3, 2, 32, 8).permute(2, 4, 3, 0, 1, 5).reshape(3, 32, 70, 24)
    off = (got[0] + (got[1] + got[2]) / 2048.0 - rows).abs()
    assert bool((off <= rows.abs() * 2.0 ** -33 + 2.0 ** -36).all())


def _scale_kernel(st, layer, share):
    """One input of one output: its largest weight to `share` of that output's."""
    w = st[f"convs.{layer}.weight"]
    w[5, 9] *= share * w[5].abs().max() / w[5, 9].abs().max()


def _scale_output(st, layer, share):
    w = st[f"convs.{layer}.weight"]
    factor = share * w.abs().max() / w[5].abs().max()
    w[5] *= factor
    st[f"convs.{layer}.bias"][5] *= factor


def _set(st, layer, index, value):
    st[f"convs.{layer}.weight"][index] = value


@pytest.mark.parametrize("layer", [0, 1, 4, 7])
@pytest.mark.parametrize("change,held", [
    (lambda st, l: None, True),
    (lambda st, l: _set(st, l, slice(None), 0.0), True),                            # a layer, an output of zeros
    (lambda st, l: _set(st, l, 3, 0.0), True),
    (lambda st, l: _set(st, l, (3, 1, 1, 1), 1e-38), True),                         # one weight that nothing depends on
    (lambda st, l: st[f"convs.{l}.weight"].mul_(1e-13), True),
    (lambda st, l: st[f"convs.{l}.weight"].mul_(1e20), True),
    (lambda st, l: st[f"convs.{l}.weight"].mul_(1e-15), False),
    (lambda st, l: st[f"convs.{l}.weight"].mul_(1e25), False),
    (lambda st, l: _scale_output(st, l, 2.0 ** -9.9), True),
    (lambda st, l: _scale_output(st, l, 2.0 ** -10.1), False),
    (lambda st, l: st[f"convs.{l}.weight"][5, 1].mul_(2.0 ** -6.1 * st[f"convs.{l}.weight"][5].abs().max() / st[f"convs.{l}.weight"][5, 1].abs().max()), False),
    (lambda st, l: st[f"convs.{l}.weight"][5, 1].mul_(2.0 ** -5.9 * st[f"convs.{l}.weight"][5].abs().max() / st[f"convs.{l}.weight"][5, 1].abs().max()), True),
    (lambda st, l: _set(st, l, (3, 1), 0.0), False),
    (lambda st, l: _set(st, l, (3, 1, 1, 1), float("inf")), False),
    (lambda st, l: _set(st, l, (3, 1, 1, 1), float("nan")), False),
    (lambda st, l: _set(st, l, (3, 1, 1, 1), 1e5), False),
])
def test_which_weights_two_parts_hold(cuda, layer, change, held):
    st = R.init_state(3, "reference")
    change(st, layer)
    units = _units(_model(cuda, st).packed_weights(PREC))
    assert ((units != 0) == torch.tensor([held or l != layer for l in range(8)])).all()


# (name, what it does to the parameters or the planes): on this side of the line, beyond it
_LINES = [
    ("weights", 2047.0, 2e5), ("an input", 2.0 ** -5.9, 2.0 ** -6.1), ("an output", 2.0 ** -9.9, 2.0 ** -10.1),
    ("activations", 1350.0, 1500.0), ("activations", 1e5, 1e30),
    ("small layer", 2e-2, 5e-3), ("planes", 32768.0, 32800.0), ("small planes", 0.2, 0.05), ("zero", 0.0, 0.0),
]


def _case(name, size):
    st, x = R.init_state(7, "torch_default"), gen_boards(40, 200, 3)[0]
    if name == "an input":
        _scale_kernel(st, 4, size)
    elif name == "an output":
        _scale_output(st, 4, size)
    elif name == "weights":          # one of them, with an input of the same channel that is zero but for a bias
        st["convs.4.weight"][5, 9] = 0.0
        st["convs.4.weight"][5, 9, 1, 1] = size
        st["convs.3.bias"][9] = 1e-3
        st["convs.3.weight"][9] *= 1e-3
    elif name == "activations":      # one channel, of which the next layer takes little (less than two parts hold beside the others, the second line)
        st["convs.4.bias"][11] = size
        st["convs.4.weight"][11] = 0.0
        st["convs.5.weight"][:, 11] *= 1.0 / 8 if size < 1e4 else 1.0 / size
    elif name == "small layer":      # a layer of small numbers, blown up again behind it
        st["convs.4.weight"] *= size
        st["convs.4.bias"] *= size
        st["convs.5.weight"] *= 1.0 / max(size, 1e-3)
    elif name == "planes":
        x[1::2] *= size
    elif name == "small planes":     # (0.1 is no fp16 number)
        x[1::2] *= 0.1 * size
    elif name == "zero":
        st, x = R.init_state(7, "reference"), x * 0.0
    return st, x


@pytest.mark.parametrize("name,within,beyond", _LINES)
@pytest.mark.parametrize("side", [0, 1])
def test_either_side_of_a_line(cuda, name, within, beyond, side):
    """As near to float64 as the fp32 instructions, boards that take different ways among one another, and every board the
    same alone, in teams of any size and with one workgroup."""
    st, x = _case(name, (within, beyond)[side])
    model = _model(cuda, st)
    l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x.double())
    xd = torch.cat([x] * 4).to(cuda)
    with torch.inference_mode():
        plain = run_forward(xd[:40], model.packed_weights(_lib.PREC_F32), _lib.PREC_F32, 1, 40)
        packed = model.packed_weights(PREC)
        want = run_forward(xd, packed, PREC, 1, 160)       # (one workgroup each)
        for n in (1, 2, 30, 60, 100):
            got = run_forward(xd[:n], packed, PREC, 1, n)
            assert torch.equal(got[0], want[0][:n]) and torch.equal(got[1], want[1][:n]), n
        # outputs that are not asked for: the others carry on
        value = run_forward(xd[:40], packed, PREC, 1, 40, want_logits=False)[1] if name == "planes" else want[1][:40]
        assert torch.equal(value, want[1][:40])
    if name == "zero":
        assert int(want[0].count_nonzero()) == 0 and int(want[1].count_nonzero()) == 0
        return
    for rows in (slice(0, 40, 2), slice(1, 40, 2)):
        was, now = rel_l2(plain[0][rows].double().cpu(), l64[rows]), rel_l2(want[0][:40][rows].double().cpu(), l64[rows])
        # (one network and twenty boards: either's error scatters; and half an ulp of the logits themselves, where little cancels)
        assert now <= 2 * was + 3e-8, (was, now)
    assert float((want[1][:40].double().cpu() - v64).abs().max()) <= 2 * float((plain[1].double().cpu() - v64).abs().max()) + 1e-7


@pytest.mark.parametrize("boards", [3, 160])
def test_draws_alone_of_boards_that_take_either_way(cuda, boards):
    """Neither logits nor values asked for: the draw is the output that says which boards are left over."""
    st, x = _case("planes", 40000.0)
    model = _model(cuda, st)
    xd, u = torch.cat([x] * 4)[:boards].to(cuda), gen_uniform(boards, 3).to(cuda)
    lib = c6.load()
    packed = model.packed_weights(PREC)
    with torch.inference_mode():
        want = run_forward(xd, packed, PREC, 1, boards, mask_mode=_lib.MASK_INPUT, u=u, want_logprob=True)
        actions = torch.full((boards,), -7, dtype=torch.int64, device=cuda)
        logprob = torch.empty(boards, device=cuda)
        rc = lib.c6_forward(xd.data_ptr(), 0, 1, boards, packed.data_ptr(), packed.numel(), PREC, None, None, _lib.MASK_INPUT, None,
                            0.0, u.data_ptr(), 1.0, actions.data_ptr(), logprob.data_ptr(), _lib.stream_ptr(cuda))
        _lib.check(rc, "c6_forward")
        assert torch.equal(actions, want[2]) and torch.equal(logprob, want[3])


def test_a_rest_behind_whole_rounds_takes_either_way(cuda):
    """The boards with a workgroup each and the rest in teams, half of either beyond the line, in one call."""
    st, x = _case("planes", 40000.0)
    packed = _model(cuda, st).packed_weights(PREC)
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rows = torch.arange(cus + 41) % 40
    with torch.inference_mode():
        want = run_forward(x.to(cuda), packed, PREC, 1, 40)
        got = run_forward(x[rows].to(cuda), packed, PREC, 1, len(rows))
    assert torch.equal(got[0], want[0][rows]) and torch.equal(got[1], want[1][rows])


@pytest.mark.parametrize("per", [1, 2, 3])
@pytest.mark.parametrize("outputs", ["all", "value", "actions"])
def test_boards_with_a_workgroup_each_take_either_way(cuda, per, outputs):
    """One board for each workgroup, which does it again itself, and more, which leave it to the next launch; the last workgroups
    have fewer or none."""
    st, x = _case("planes", 40000.0)
    packed = _model(cuda, st).packed_weights(PREC)
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    for boards in (per * cus, per * cus - 3):
        rows = torch.arange(boards) % 40
        u = gen_uniform(40, 5)
        with torch.inference_mode():
            want = run_forward(x.to(cuda), packed, PREC, 1, 40, mask_mode=_lib.MASK_INPUT, u=u.to(cuda))
            if outputs == "actions":
                got = run_forward(x[rows].to(cuda), packed, PREC, 1, boards, mask_mode=_lib.MASK_INPUT, u=u[rows].to(cuda),
                                  want_logits=False, want_value=False)
                assert torch.equal(got[2], want[2][rows])
                continue
            got = run_forward(x[rows].to(cuda), packed, PREC, 1, boards, mask_mode=_lib.MASK_INPUT, want_logits=outputs == "all")
        assert torch.equal(got[1], want[1][rows])
        if outputs == "all":
            assert torch.equal(got[0], want[0][rows])


def _against_float64(cuda, st, x, boards=(None,)):
    """Errors of logits and values against a float64 forward: the fp32 instructions', and this for each number of boards."""
    model = _model(cuda, st)
    l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x.double())
    xd = x.to(cuda)

    def errors(prec, n):
        rows = torch.arange(n) % len(x)
        with torch.inference_mode():
            lg, vg, _, _ = run_forward(xd[rows], model.packed_weights(prec), prec, 1, n)
        return rel_l2(lg.double().cpu(), l64[rows]), float((vg.double().cpu() - v64[rows]).abs().max())

    return errors(_lib.PREC_F32, len(x)), [errors(PREC, n or len(x)) for n in boards]


@pytest.mark.parametrize("factors", [{0: 1e-5, 1: 1e3, 2: 1e2}, {0: 1e-6, 1: 1e3, 2: 1e3}, {0: 1e-7, 1: 1e3, 2: 1e4}])
def test_small_weights_of_the_first_layer(cuda, factors):
    """Whichever way these boards go, their weights are those of the caller to 24 bits."""
    st, x = R.init_state(5, "reference"), gen_boards(6, 200, 3)[0]
    for layer, factor in factors.items():
        st[f"convs.{layer}.weight"] *= factor
    was, now = _against_float64(cuda, st, x, (6, 60, 200, 600))
    for n in now:
        assert n[0] <= 2 * was[0] + 3e-8 and n[1] <= 2 * was[1] + 1e-7, (was, now)


def _channels(st, layer, channels, factor):
    """Outputs of a layer times factor, and what the next takes of them divided by it."""
    st[f"convs.{layer}.weight"][channels] *= factor
    st[f"convs.{layer}.bias"][channels] *= factor
    st[f"convs.{layer + 1}.weight"][:, channels] /= factor


@pytest.mark.parametrize("factors", [
    {3: 300, 4: 1e-6, 5: 1e3}, {3: 300, 4: 1e-7, 5: 1e3}, {3: 300, 4: 5e-8, 5: 3e3}, {3: 1e3, 4: 1.6e-8, 5: 3e3}, {3: 1e3, 4: 5e-9, 5: 3e3},
    {1: 1e-4, 6: 1e4}, {2: 1e3, 3: 1e-9, 4: 1e4, 5: 1e2},
    (3, slice(5, 6), 1e-5), (3, slice(5, 6), 1e-8), (3, slice(0, 32), 1e-3), (3, slice(0, 32), 1e-6), (3, slice(0, 63), 1e-6), (5, slice(0, 95), 1e-8),
    (3, slice(0, 32), 2.0 ** -5), (3, slice(0, 63), 2.0 ** -3),
])
def test_small_weights_behind_large_activations(cuda, factors):
    """Layers of small weights between others, and outputs of a layer that are small where the next layer's weights for them are large:
    as near to float64 as the fp32 instructions."""
    st, x = R.init_state(5, "reference"), gen_boards(6, 200, 3)[0]
    if isinstance(factors, tuple):
        _channels(st, *factors)
    else:
        for layer, factor in factors.items():
            st[f"convs.{layer}.weight"] *= factor
    was, now = _against_float64(cuda, st, x, (6, 60, 200, 600))
    for n in now:
        assert n[0] <= 2 * was[0] + 3e-8 and n[1] <= 2 * was[1] + 1e-7, (was, now)


@pytest.mark.parametrize("per", [1, 5, 150, 300, 700])
def test_sets_that_go_either_way_in_one_call(cuda, per):
    """Weight sets of which every other is beyond two parts: teams, one board and several for each workgroup, runs of boards of both."""
    states = [R.init_state(20 + i, "reference") for i in range(4)]
    for st in states[1::2]:
        _scale_output(st, 4, 2.0 ** -12)
    packed = [_model(cuda, st).packed_weights(PREC) for st in states]
    assert [bool((_units(p) != 0).all()) for p in packed] == [True, False, True, False]
    x = gen_boards(4 * 30, 200, 9)[0][torch.arange(4 * per) % 120].to(cuda)
    u = gen_uniform(4 * per, 5).to(cuda)
    with torch.inference_mode():
        got = run_forward(x, torch.stack(packed), PREC, 4, per, mask_mode=_lib.MASK_INPUT, u=u, want_logprob=True)
        for i in range(4):
            rows = slice(i * per, (i + 1) * per)
            want = run_forward(x[rows], packed[i], PREC, 1, per, mask_mode=_lib.MASK_INPUT, u=u[rows], want_logprob=True)
            assert all(torch.equal(g[rows].flatten(), w.flatten()) for g, w in zip(got, want)), i


@pytest.mark.parametrize("boards", [1, 7, 30, 60, 100])
@pytest.mark.parametrize("case", [("planes", 40000.0), ("an output", 2.0 ** -12)])
def test_a_team_without_all_its_members_does_a_board_again(cuda, boards, case):
    """Boards of either kind, and those of a set that two parts do not hold, in teams whose waits run out at once, so that members leave
    before the verdict or come late, and in ordinary ones."""
    st, x = _case(*case)
    packed = _model(cuda, st).packed_weights(PREC)
    xd = x[(torch.arange(boards) + 1) % 40].to(cuda)
    flags = torch.zeros(boards * 256, dtype=torch.int32, device=cuda)
    with torch.inference_mode():
        want = run_forward(torch.cat([xd] * (300 // boards + 1)), packed, PREC, 1, boards * (300 // boards + 1))
        for tag, polls in ((1, 1), (2, 2), (3, 5), (4, 0), (5, 1)):
            lg, vg = _team(PREC, xd, packed, tag, flags, polls)
            assert torch.equal(lg, want[0][:boards]) and torch.equal(vg, want[1][:boards]), polls


@pytest.mark.parametrize("boards", [20, 300, 600])
@pytest.mark.parametrize("case", [("planes", 40000.0), ("an output", 2.0 ** -12)])
def test_graphs_of_boards_that_take_either_way(cuda, boards, case):
    st, x = _case(*case)
    model = _model(cuda, st)
    xs = [x[(torch.arange(boards) + i) % 40].to(cuda) for i in range(3)]
    with torch.inference_mode():
        want = [model(v) for v in xs]
        static = xs[0].clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(static)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(static)
        for i in (0, 1, 2, 1, 0):
            static.copy_(xs[i])
            graph.replay()
            model(xs[2])                       # eager work in between
            torch.cuda.synchronize()
            assert torch.equal(out[0], want[i][0]) and torch.equal(out[1], want[i][1]), i
