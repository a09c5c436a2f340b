"""Two workgroups per CU (more boards than CUs, plain 16-bit modes) against one workgroup per board:
the same bits at batch sizes around whole rounds, for every input form, mask and output type, and
the cascade's lists."""
import ctypes

import pytest
import torch

import connect6_amd as c6
from connect6_amd import _lib
from connect6_amd.model import run_forward
from connect6_amd.synthetic import gen_boards, gen_uniform
from oracle import torch_ref as R

pytestmark = pytest.mark.gpu
PIECE = 100   # boards of a call that one workgroup per board serves


def _model(cuda, seed=11):
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(R.init_state(seed, "torch_default"))
    return model


def _inputs(n):
    x, legal = gen_boards(n, 200, 77)
    x[3::5, 2] = (torch.rand(19, 19, generator=torch.Generator().manual_seed(1)) > 0.5).float()   # a varying third plane
    x[4::5] *= 0.3                                                                                # not exact in 16 bits
    return x, legal


def _pieces(call, n):
    """call(slice) over pieces of the batch, outputs joined."""
    outs = [call(slice(i, min(i + PIECE, n))) for i in range(0, n, PIECE)]
    return [torch.cat(t) if t[0] is not None else None for t in zip(*outs)]


def _same(got, want):
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        assert a is None or torch.equal(a, b)


@pytest.mark.parametrize("prec", [_lib.PREC_BF16, _lib.PREC_F16])
def test_same_bits_as_one_workgroup_per_board(cuda, prec):
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    most = 4 * cus + 3
    model, (x, legal) = _model(cuda), _inputs(most)
    x, legal, u = x.to(cuda), legal.to(cuda), gen_uniform(most, 5).to(cuda)
    packed = model.packed_weights(prec)

    def call(s):
        n = x[s].shape[0]
        return run_forward(x[s], packed, prec, 1, n, mask_mode=_lib.MASK_LEGAL, legal=legal[s], u=u[s], temperature=0.8,
                           want_logprob=True)

    with torch.inference_mode():
        want = _pieces(call, most)
        for n in (cus + 1, 300, 2 * cus - 1, 2 * cus, 2 * cus + 1, 3 * cus + 9, 4 * cus, most):
            _same(call(slice(0, n)), [w[:n] for w in want])
        for kw in (dict(), dict(mask_mode=_lib.MASK_INPUT, fill=-3.0), dict(want_value=False)):
            for t in (x, x.half(), x.bfloat16()):
                part = lambda s: run_forward(t[s], packed, prec, 1, t[s].shape[0], **kw)
                _same(part(slice(0, 777)), _pieces(part, 777))


@pytest.mark.parametrize("prec", [_lib.PREC_BF16, _lib.PREC_F16])
def test_weight_sets_and_board_state(cuda, prec):
    sets, per = 3, 259
    models = [_model(cuda, 20 + i) for i in range(sets)]
    x = _inputs(sets * per)[0].to(cuda)
    packed = torch.stack([m.packed_weights(prec) for m in models])
    with torch.inference_mode():
        logits, value, _, _ = run_forward(x, packed, prec, sets, per)
        for i in range(sets):
            part = lambda s: run_forward(x[i * per:(i + 1) * per][s], packed[i], prec, 1, len(range(per)[s]))
            want = _pieces(part, per)
            assert torch.equal(logits[i * per:(i + 1) * per], want[0])
            assert torch.equal(value[i * per:(i + 1) * per], want[1])
        # int8 state, rows picked (some outside: they are clamped), every board symmetry
        g = torch.Generator().manual_seed(3)
        boards = torch.randint(-1, 2, (700, 19, 19), generator=g, dtype=torch.int8).to(cuda)
        player = (torch.randint(0, 2, (700,), generator=g, dtype=torch.int8) * 2 - 1).to(cuda)
        left = torch.randint(1, 3, (700,), generator=g, dtype=torch.int8).to(cuda)
        index = torch.randint(-5, 710, (613,), generator=g).to(cuda)
        models[0].precision = "bf16" if prec == _lib.PREC_BF16 else "fp16"
        for view in range(8):
            part = lambda s: models[0].forward_boards(boards, player, left, index=index[s], view=view)
            _same(part(slice(0, 613)), _pieces(part, 613))


@pytest.mark.parametrize("rounds", [1, 2, 3, 4])
@pytest.mark.parametrize("prec", [_lib.PREC_BF16, _lib.PREC_F16])
def test_rest_in_teams_beside_whole_rounds(cuda, prec, rounds):
    """A few boards beyond whole rounds go to teams in the same launch: sizes on either side of a change of the
    team's size and of the most that are shared, also when no workgroup waits for another for long."""
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    most = rounds * cus + cus * 5 // 16 + 1
    model, (x, legal) = _model(cuda), _inputs(most)
    x, legal, u = x.to(cuda), legal.to(cuda), gen_uniform(most, 5).to(cuda)
    packed = model.packed_weights(prec)

    def call(s):
        return run_forward(x[s], packed, prec, 1, x[s].shape[0], mask_mode=_lib.MASK_LEGAL, legal=legal[s], u=u[s],
                           temperature=0.8, want_logprob=True)

    with torch.inference_mode():
        want = _pieces(call, most)
        for rest in (1, 2, cus // 12, cus // 12 + 1, cus * 5 // 32, cus * 5 // 32 + 1, cus * 5 // 16, cus * 5 // 16 + 1):
            n = rounds * cus + rest
            _same(call(slice(0, n)), [w[:n] for w in want])
        # through the C ABI, each workgroup looking at a flag once only
        lib, n = c6.load(), rounds * cus + cus * 5 // 32
        ws, fl = ctypes.c_size_t(), ctypes.c_size_t()
        assert lib.c6_team_bytes(prec, n, ctypes.byref(ws), ctypes.byref(fl)) == 0 and ws.value > 0
        work = torch.full((ws.value,), 255, dtype=torch.uint8, device=cuda)
        flags = torch.zeros(fl.value // 4, dtype=torch.int32, device=cuda)
        raw = run_forward(x, packed, prec, 1, most)
        for tag in (1, 2):
            logits, value = torch.empty(n, 361, device=cuda), torch.empty(n, device=cuda)
            rc = lib.c6_forward_team(x.data_ptr(), 0, 1, n, packed.data_ptr(), packed.numel(), prec, logits.data_ptr(),
                                     value.data_ptr(), 0, None, 0.0, None, 1.0, None, None, work.data_ptr(), ws.value,
                                     flags.data_ptr(), flags.numel() * 4, tag, 1, _lib.stream_ptr(x.device))
            _lib.check(rc, "c6_forward_team")
            _same((logits, value), (raw[0][:n], raw[1][:n]))


@pytest.mark.parametrize("rounds,rest", [(1, 9), (2, 30), (3, 60)])   # twelve, six and three workgroups per board
@pytest.mark.parametrize("precision", ["bf16", "fp16"])
def test_board_state_of_a_rest(cuda, precision, rounds, rest):
    """int8 states, rows picked (some outside: they are clamped), every board symmetry, where a rest goes to teams."""
    n = rounds * torch.cuda.get_device_properties(cuda).multi_processor_count + rest
    model = _model(cuda, 20)
    model.precision = precision
    g = torch.Generator().manual_seed(3)
    boards = torch.randint(-1, 2, (700, 19, 19), generator=g, dtype=torch.int8).to(cuda)
    player = (torch.randint(0, 2, (700,), generator=g, dtype=torch.int8) * 2 - 1).to(cuda)
    left = torch.randint(1, 3, (700,), generator=g, dtype=torch.int8).to(cuda)
    index, u = torch.randint(-5, 710, (n,), generator=g).to(cuda), gen_uniform(n, 6).to(cuda)
    with torch.inference_mode():
        for view in range(8):
            part = lambda s: model.forward_boards(boards, player, left, index=index[s], view=view)
            _same(part(slice(0, n)), _pieces(part, n))
            part = lambda s: model.selfplay_step_boards(boards, player, left, u[s], 0.7, index=index[s], view=view)
            _same(part(slice(0, n)), _pieces(part, n))


@pytest.mark.parametrize("rounds,rest", [(1, 9), (2, 30), (3, 60)])
@pytest.mark.parametrize("precision", ["bf16", "fp16", "bf16c"])
def test_graphs_and_streams_of_a_rest(cuda, precision, rounds, rest):
    """A rest in teams: a graph replayed behind eager work, and calls on three streams at once."""
    n = rounds * torch.cuda.get_device_properties(cuda).multi_processor_count + rest
    model = _model(cuda)
    model.precision = precision
    x = _inputs(n)[0]
    xs = [torch.roll(x, 100 * i, 0).to(cuda) for i in range(3)]
    with torch.inference_mode():
        want = [_pieces(lambda s: model(v[s]), n) for v in xs]
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
            _same(out, want[i])
        streams = [torch.cuda.Stream() for _ in range(3)]
        torch.cuda.synchronize()
        got = []
        for _ in range(4):
            for i, s in enumerate(streams):
                with torch.cuda.stream(s):
                    got.append((i, model(xs[i])))
        torch.cuda.synchronize()
        for i, answer in got:
            _same(answer, want[i])


@pytest.mark.parametrize("prec", [_lib.PREC_BF16, _lib.PREC_F16])
def test_one_board_behind_many_rounds_is_not_shared(cuda, prec):
    """Teams gain nothing there: they take a rest of more than one board for every sixteen rounds, here at the edges of that
    rule.  (Exchange memory is what tells which way a batch goes.)  The same bits on either side."""
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    model, lib = _model(cuda), c6.load()
    packed = model.packed_weights(prec)
    ws, fl = ctypes.c_size_t(), ctypes.c_size_t()
    for rounds, rest, shared in ((15, 1, True), (16, 1, False), (16, 2, True), (31, 2, True), (32, 2, False), (32, 3, True),
                                 (63, 3, False), (63, 4, True), (63, 80, True)):
        assert lib.c6_team_bytes(prec, rounds * cus + rest, ctypes.byref(ws), ctypes.byref(fl)) == 0
        assert (ws.value > 0) == shared and (fl.value > 0) == shared, (rounds, rest)
    x = _inputs(399)[0].to(cuda)
    with torch.inference_mode():
        part = run_forward(x[:100], packed, prec, 1, 100)
        for n in (15 * cus + 1, 16 * cus + 1, 16 * cus + 2):
            pick = torch.arange(n, device=cuda) % 100
            got = run_forward(x[pick], packed, prec, 1, n)
            assert torch.equal(got[0], part[0][pick]) and torch.equal(got[1], part[1][pick]), n


@pytest.mark.parametrize("boards", [257, 336, 513, 1400, 1576, 4096, 4097, 4098])
def test_cascade_lists_the_same_boards(cuda, boards):
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(R.init_state(5, "reference"))
    model.precision = "bf16c"
    x = gen_boards(boards, 200, 9)[0].to(cuda)
    listed = []

    def call(s):
        out = model.forward_masked(x[s])
        listed.append(model.cascade_stats["second_pass"].clone())
        return out

    with torch.inference_mode():
        got = call(slice(0, boards))
        whole = int(listed.pop())
        want = _pieces(call, boards)
    _same(got, want)
    assert whole == sum(int(n) for n in listed) > 0
