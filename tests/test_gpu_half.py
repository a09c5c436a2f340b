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


@pytest.mark.parametrize("layer", [1, 3, 5, 7])
def test_parts_of_weights(cuda, layer):
    """16 w = hi + (lo + rest / 2048) / 2048, in fp16 each: exactly where hi is a normal number, but for the tap that takes in what the
    others of its channel leave; and hi and lo leave nothing of the sum over a channel's taps."""
    st = R.init_state(3, "reference")
    w = st[f"convs.{layer}.weight"]
    w[0, 0] = torch.tensor([[1e-3, -1e-4, 1e-6], [0.0, 2000.0, -2047.9], [1e-9, -1e-12, 3e-13]])
    w[1, 1, 0] = torch.tensor([2049.0, -3e38, float("nan")])
    w[1, 1, 1] = torch.tensor([2e-13, -1e-30, 0.0])
    bits = _parts(_model(cuda, st).packed_weights(PREC), layer)
    want = w.flatten(2).double()
    marked = torch.zeros_like(want, dtype=torch.bool)
    marked[1, 1, :5] = True
    assert bool(((bits[0] == 0x7fff) == marked).all())
    raw = (bits[1][marked].int() & 0xffff) | (bits[2][marked].int() << 16)
    assert torch.equal(raw, w.flatten(2)[marked].view(torch.int32))
    hi, lo, rest = bits.view(torch.float16).double().masked_fill(marked, 0.0).unbind(0)
    rest = rest / 2048.0
    off = ((hi + (lo + rest) / 2048.0) / 16.0 - want).abs().masked_fill(marked, 0.0)
    largest = want.masked_fill(marked, 0.0).abs().amax(2, keepdim=True)
    # that tap's third part is the others' rest with the sign changed, up to three units of lo's last bit (2^-21 of the largest), to
    # half a unit of its own
    assert bool((off <= 3 * largest * 2.0 ** -33 + 2.0 ** -51).all())
    inexact = (off != 0) & (want.abs() >= 2.0 ** -18)
    assert int(inexact.sum(2).max()) <= 1
    step = lo.abs().amax(2, keepdim=True) * 2.0 ** -10 + 2.0 ** -24   # one unit of the largest lo's last bit
    plain = ~marked.any(2)
    assert bool((rest.abs() <= 3 * step)[plain].all())
    assert float((rest.sum(2, keepdim=True).abs() / step)[plain].mean()) <= 0.02


# (name, what it does to the parameters or the planes): on this side of the line, beyond it
_LINES = [
    ("weights", 2047.0, 2049.0), ("activations", 1350.0, 1500.0), ("activations", 1e5, 1e30),
    ("small layer", 2e-5, 1e-6), ("planes", 32768.0, 32800.0), ("small planes", 2e-4, 1e-5), ("zero", 0.0, 0.0),
]


def _case(name, size):
    st, x = R.init_state(7, "torch_default"), gen_boards(40, 200, 3)[0]
    if name == "weights":            # ... with an input of the same channel that is zero but for a bias
        st["convs.4.weight"][5, 9] = 0.0
        st["convs.4.weight"][5, 9, 1, 1] = size
        st["convs.3.bias"][9] = 1e-3
        st["convs.3.weight"][9] *= 1e-3
    elif name == "activations":      # one channel, of which the next layer takes little
        st["convs.4.bias"][11] = size
        st["convs.4.weight"][11] = 0.0
        st["convs.5.weight"][:, 11] *= 1.0 / size
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


@pytest.mark.parametrize("boards", [1, 7, 30, 60, 100])
def test_a_team_without_all_its_members_does_a_board_again(cuda, boards):
    """Boards of either kind in teams whose waits run out at once, so that members leave before the verdict or come late, and in
    ordinary ones."""
    st, x = _case("planes", 40000.0)
    packed = _model(cuda, st).packed_weights(PREC)
    xd = x[(torch.arange(boards) + 1) % 40].to(cuda)
    flags = torch.zeros(boards * 256, dtype=torch.int32, device=cuda)
    with torch.inference_mode():
        want = run_forward(torch.cat([xd] * (300 // boards + 1)), packed, PREC, 1, boards * (300 // boards + 1))
        for tag, polls in ((1, 1), (2, 2), (3, 5), (4, 0), (5, 1)):
            lg, vg = _team(PREC, xd, packed, tag, flags, polls)
            assert torch.equal(lg, want[0][:boards]) and torch.equal(vg, want[1][:boards]), polls


@pytest.mark.parametrize("boards", [20, 300])
def test_graphs_of_boards_that_take_either_way(cuda, boards):
    st, x = _case("planes", 40000.0)
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
