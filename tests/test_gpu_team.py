"""Several workgroups per board (c6_forward_team) against the one-workgroup kernels: the same bits at
every batch size on either side of a change of the team's size, also when no workgroup waits for
another for long (each then computes what it misses), in graphs and on two streams at once."""
import ctypes

import pytest
import torch

import connect6_amd as c6
from connect6_amd import _lib
from connect6_amd.model import run_forward
from connect6_amd.synthetic import gen_boards, gen_uniform
from oracle import torch_ref as R

pytestmark = pytest.mark.gpu
MODES = [_lib.PREC_F32S, _lib.PREC_BF16, _lib.PREC_F16, _lib.PREC_BF16F6, _lib.PREC_BF16F6W]


def _model(cuda, seed=11):
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(R.init_state(seed, "torch_default"))
    return model


def _inputs(n):
    x, legal = gen_boards(n, 200, 77)
    x[3::5, 2] = (torch.rand(19, 19, generator=torch.Generator().manual_seed(1)) > 0.5).float()   # a varying third plane
    x[4::5] *= 0.3                                                                                # not exact in bf16
    return x, legal


def _team(prec, x, packed, tag, flags, polls=0, **kw):
    """c6_forward_team through the C ABI: logits, value."""
    lib, b = c6.load(), x.shape[0]
    ws, fl = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.c6_team_bytes(prec, b, ctypes.byref(ws), ctypes.byref(fl)) == 0 and ws.value > 0
    assert flags.numel() * 4 >= fl.value
    work = torch.full((ws.value,), 255, dtype=torch.uint8, device=x.device)
    logits, value = torch.empty(b, 361, device=x.device), torch.empty(b, device=x.device)
    rc = lib.c6_forward_team(x.data_ptr(), 0, 1, b, packed.data_ptr(), packed.numel(), prec, logits.data_ptr(),
                             value.data_ptr(), 0, None, 0.0, None, 1.0, None, None, work.data_ptr(), ws.value,
                             flags.data_ptr(), flags.numel() * 4, tag, polls, _lib.stream_ptr(x.device))
    _lib.check(rc, "c6_forward_team")
    return logits, value


@pytest.mark.parametrize("prec", MODES)
def test_same_bits_as_one_workgroup_per_board(cuda, prec):
    model, (x, legal) = _model(cuda), _inputs(300)
    xd, ld, u = x.to(cuda), legal.to(cuda), gen_uniform(300, 5).to(cuda)
    packed = model.packed_weights(prec)
    with torch.inference_mode():
        kw = dict(mask_mode=_lib.MASK_LEGAL, u=u, temperature=0.8, want_logprob=True)
        want = run_forward(xd, packed, prec, 1, 300, legal=ld, **kw)
        for n in (1, 2, 5, 20, 21, 22, 41, 42, 43, 72, 73, 74, 84, 85, 86):
            kw["u"] = u[:n]
            got = run_forward(xd[:n], packed, prec, 1, n, legal=ld[:n], **kw)
            for a, b in zip(got, want):
                assert torch.equal(a, b[:n]), n
        raw = run_forward(xd, packed, prec, 1, 300)
        for n in (1, 40):
            got = run_forward(xd[7:7 + n], packed, prec, 1, n)
            assert torch.equal(got[0], raw[0][7:7 + n]) and torch.equal(got[1], raw[1][7:7 + n])
        # several weight sets, and board states through a view and an index
        sets = torch.cat([packed, _model(cuda, 12).packed_weights(prec)])
        a = run_forward(xd[:6], sets, prec, 2, 3)
        assert torch.equal(a[0][:3], raw[0][:3])
        assert torch.equal(a[0][3:], run_forward(xd[3:6], sets[packed.numel():], prec, 1, 3)[0])


@pytest.mark.parametrize("prec", [_lib.PREC_F32S, _lib.PREC_BF16F6, _lib.PREC_BF16F6W])
def test_boards_beyond_whole_rounds(cuda, prec):
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    most = {_lib.PREC_F32S: cus // 3, _lib.PREC_BF16F6W: cus * 2 // 7}.get(prec, cus // 6)
    total = 2 * cus + most + 1
    model, (x, legal) = _model(cuda), _inputs(total)
    xd, ld, u = x.to(cuda), legal.to(cuda), gen_uniform(total, 5).to(cuda)
    packed = model.packed_weights(prec)

    def call(a, b, x=xd, groups=1, weights=packed):
        return run_forward(x[a:b], weights, prec, groups, (b - a) // groups, mask_mode=_lib.MASK_LEGAL, legal=ld[a:b],
                           u=u[a:b], temperature=0.8, want_logprob=True)

    with torch.inference_mode():
        # (a hundred boards: one workgroup each)
        want = [torch.cat(t) for t in zip(*[call(i, min(i + 100, total)) for i in range(0, total, 100)])]
        for n in (cus, cus + 1, cus + most // 4, cus + most // 2 + 1, cus + most, cus + most + 1, 2 * cus, total - 1, total):
            for a, b in zip(call(0, n), want):
                assert torch.equal(a, b[:n]), n
        # the shared ones in a weight set of their own
        sets = torch.cat([packed, _model(cuda, 12).packed_weights(prec)])
        n = 2 * (cus // 2 + 3)
        got, other = call(0, n, groups=2, weights=sets), call(n // 2, n, weights=sets[packed.numel():])
        for a, b, c in zip(got, want, other):
            assert torch.equal(a[:n // 2], b[:n // 2]) and torch.equal(a[n // 2:], c)


# (boards up to what the mode shares at all: 21 between twelve workgroups, 42 between six, 73 or 85 between three)
@pytest.mark.parametrize("prec,boards", [(p, b) for p in MODES for b in (1, 7, 30, 60)
                                         if b <= {_lib.PREC_F32S: 85, _lib.PREC_BF16F6W: 73, _lib.PREC_BF16F6: 42}.get(p, 21)])
def test_a_workgroup_that_waited_long_enough_does_the_work_itself(cuda, prec, boards):
    model, (x, _) = _model(cuda), _inputs(boards)
    xd = x.to(cuda)
    packed = model.packed_weights(prec)
    flags = torch.zeros(boards * 256, dtype=torch.int32, device=cuda)
    with torch.inference_mode():
        want = run_forward(torch.cat([xd] * (300 // boards + 1)), packed, prec, 1, boards * (300 // boards + 1))
        for tag, polls in ((1, 0), (2, 1), (3, 2), (4, 5)):
            lg, vg = _team(prec, xd, packed, tag, flags, polls)
            assert torch.equal(lg, want[0][:boards]) and torch.equal(vg, want[1][:boards]), polls


@pytest.mark.parametrize("prec", [_lib.PREC_BF16C, _lib.PREC_BF16C6])
def test_cascade_with_few_listed_boards(cuda, prec):
    model, (x, legal) = _model(cuda), gen_boards(1100, 200, 31)
    xd, ld, u = x.to(cuda), legal.to(cuda), gen_uniform(1100, 5).to(cuda)
    packed = model.packed_weights(prec)
    with torch.inference_mode():
        # the margin that about every tenth board is under: the listed ones are few enough for teams
        # of every size, or too many, depending on the batch
        for threshold in (0.0, 0.004, 0.3, -1.0):
            kw = dict(mask_mode=_lib.MASK_LEGAL, temperature=0.8, want_logprob=True, threshold=threshold)
            stats = {}
            want = run_forward(xd, packed, prec, 1, 1100, legal=ld, u=u, stats=stats, **kw)
            for n in (1, 7, 21, 22, 42, 43, 85, 86, 257, 277, 278, 298, 299, 300, 329, 330, 512, 530, 1024):
                got = run_forward(xd[:n], packed, prec, 1, n, legal=ld[:n], u=u[:n], stats=stats, **kw)
                for a, b in zip(got, want):
                    assert torch.equal(a, b[:n]), (threshold, n, int(stats["second_pass"]))
                if threshold in (0.0, -1.0):
                    assert int(stats["second_pass"]) == (0 if threshold == 0.0 else n)


@pytest.mark.parametrize("prec,sizes", [(_lib.PREC_F32S, (86, 100, 127, 128, 129, 342, 384, 385)), (_lib.PREC_BF16, (22, 40, 41)),
                                        (_lib.PREC_F16, (23, 39, 40, 41))])
def test_edges_of_the_smallest_teams(cuda, prec, sizes):
    model, (x, legal) = _model(cuda), _inputs(385)
    xd, ld, u = x.to(cuda), legal.to(cuda), gen_uniform(385, 5).to(cuda)
    packed = model.packed_weights(prec)
    kw = dict(mask_mode=_lib.MASK_LEGAL, temperature=0.8, want_logprob=True)
    with torch.inference_mode():
        # (200 boards: one workgroup each)
        want = [torch.cat(t) for t in zip(*[run_forward(xd[a:a + 200], packed, prec, 1, 200, legal=ld[a:a + 200], u=u[a:a + 200], **kw)
                                            for a in (0, 185)])]
        want = [torch.cat([t[:185], t[200:]]) for t in want]
        for n in sizes:
            for a in (0, 385 - n):
                got = run_forward(xd[a:a + n], packed, prec, 1, n, legal=ld[a:a + n], u=u[a:a + n], **kw)
                for p, q in zip(got, want):
                    assert torch.equal(p, q[a:a + n]), (n, a)


@pytest.mark.parametrize("prec", [_lib.PREC_BF16C, _lib.PREC_BF16C6])
def test_both_passes_in_one_launch(cuda, prec):
    """At most 21 boards (of 256 CUs) go through c6_forward_cascade_team in one launch; also when nobody waits for long."""
    model, (x, _) = _model(cuda), _inputs(21)
    xd, lib = x.to(cuda), c6.load()
    packed = model.packed_weights(prec)
    flags = torch.zeros(2 * 21 * 256, dtype=torch.int32, device=cuda)
    cw, tag = ctypes.c_size_t(), 1
    with torch.inference_mode():
        for threshold in (0.0, 0.02, 0.3, -1.0):
            big = {}
            want = run_forward(torch.cat([xd] * 4), packed, prec, 1, 84, threshold=threshold, stats=big)
            counts = []
            for b in (1, 2, 16, 17, 21):
                for polls in (0, 1, 3):
                    ws, fl = ctypes.c_size_t(), ctypes.c_size_t()
                    assert lib.c6_team_bytes(prec, b, ctypes.byref(ws), ctypes.byref(fl)) == 0
                    assert 0 < fl.value <= flags.numel() * 4
                    assert lib.c6_cascade_workspace_bytes(b, ctypes.byref(cw)) == 0
                    work = torch.full((ws.value,), 255, dtype=torch.uint8, device=cuda)
                    cascade = torch.full((cw.value // 4,), -7, dtype=torch.int32, device=cuda)
                    lg, vg = torch.empty(b, 361, device=cuda), torch.empty(b, device=cuda)
                    rc = lib.c6_forward_cascade_team(xd.data_ptr(), 0, 1, b, packed.data_ptr(), packed.numel(), prec,
                                                     lg.data_ptr(), 0, vg.data_ptr(), 0, None, 0.0, None, 1.0, None, None,
                                                     threshold, cascade.data_ptr(), cw.value, work.data_ptr(), ws.value,
                                                     flags.data_ptr(), flags.numel() * 4, tag, polls,
                                                     _lib.stream_ptr(cuda))
                    _lib.check(rc, "c6_forward_cascade_team")
                    tag += 2
                    assert torch.equal(lg, want[0][:b]) and torch.equal(vg, want[1][:b]), (threshold, b, polls)
                    counts.append(int(cascade[0]))
                assert counts[-1] == counts[-2] == counts[-3] and 0 <= counts[-1] <= b
            assert int(big["second_pass"]) == 4 * counts[-1]
            assert threshold != 0.0 or counts[-1] == 0
            assert threshold != -1.0 or counts[-1] == 21


@pytest.mark.parametrize("prec", [_lib.PREC_BF16C, _lib.PREC_BF16C6])
@pytest.mark.parametrize("boards", [22, 42, 43, 73, 74, 255, 256, 257, 298, 299, 329, 330, 513])
def test_second_pass_of_whole_rounds_and_a_rest(cuda, prec, boards):
    """Every board listed: none, one or two whole rounds of one workgroup per board, and a rest at the edges of what
    teams take, twice on the same stream; the bits and the count of the second pass's own mode."""
    net = c6.PolicyValueNet().to(cuda).eval()
    x = gen_boards(boards, 120, 3)[0].to(cuda)
    alone = _lib.PREC_BF16F6W if prec == _lib.PREC_BF16C else _lib.PREC_BF16F6
    with torch.inference_mode():
        want = run_forward(torch.cat([x, x[:1].expand(600, -1, -1, -1)])[:512], net.packed_weights(alone), alone, 1, 512)
        for _ in range(2):
            stats = {}
            got = run_forward(x, net.packed_weights(prec), prec, 1, boards, threshold=-1.0, stats=stats)
            assert int(stats["second_pass"]) == boards
            n = min(boards, 512)
            assert torch.equal(got[0][:n], want[0][:n]) and torch.equal(got[1][:n], want[1][:n])


@pytest.mark.parametrize("prec", [_lib.PREC_BF16, _lib.PREC_F16, _lib.PREC_BF16C, _lib.PREC_BF16C6])
def test_a_rest_behind_an_odd_number_of_rounds(cuda, prec):
    """Two workgroups per CU, and teams for a rest beside them: the bits and the listed boards of batches that have no team, at
    the edges of the rule (teams of twelve, six and three; at two rounds of the first two only)."""
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    most, three = cus * 5 // 32, cus * 5 // 16
    total = 11 * cus + three + 1
    x, legal = gen_boards(400, 200, 31)
    pick = torch.arange(total) % 399
    xd, ld, u = x[pick].to(cuda), legal[pick].to(cuda), gen_uniform(total, 5).to(cuda)
    packed = _model(cuda).packed_weights(prec)
    cascade = prec in _lib.CASCADES
    with torch.inference_mode():
        for threshold in (0.0, 0.02, -1.0) if cascade else (None,):
            def call(a, b):
                stats = {}
                out = run_forward(xd[a:b], packed, prec, 1, b - a, mask_mode=_lib.MASK_LEGAL, legal=ld[a:b], u=u[a:b],
                                  temperature=0.8, want_logprob=True, threshold=threshold, stats=stats)
                return out, int(stats["second_pass"]) if cascade else 0
            parts = [call(i, min(i + 100, total)) for i in range(0, total, 100)]
            want = [torch.cat(t) for t in zip(*[p[0] for p in parts])]
            for n in (2 * cus + 9, 2 * cus + most, 2 * cus + most + 1, 3 * cus, 3 * cus + 1, 3 * cus + 2, 3 * cus + 9,
                      3 * cus + most, 3 * cus + most + 1, 3 * cus + three, 3 * cus + three + 1, 4 * cus + 9, 5 * cus + 21,
                      11 * cus + 5, 11 * cus + 6, total - 1, total):
                got, listed = call(0, n)
                for a, b in zip(got, want):
                    assert torch.equal(a, b[:n]), (threshold, n)
                tail = call(n // 100 * 100, n)[1] if n % 100 else 0
                assert listed == sum(p[1] for p in parts[:n // 100]) + tail, (threshold, n)


def test_boards_states_views_and_index(cuda):
    model, (x, _) = _model(cuda), gen_boards(300, 200, 5)
    boards = (x[:, 0] - x[:, 1]).to(torch.int8).to(cuda)
    player = torch.where(torch.arange(300) % 3 == 0, -1, 1).to(torch.int8).to(cuda)
    left = torch.where(torch.arange(300) % 2 == 0, 1, 2).to(torch.int8).to(cuda)
    u = gen_uniform(300, 6).to(cuda)
    index = torch.randperm(300, generator=torch.Generator().manual_seed(3)).to(cuda)
    with torch.inference_mode():
        la, va = model.forward_boards(boards, player, left, index=index, view=6)
        lb, vb = model.forward_boards(boards, player, left, index=index[:20], view=6)
        assert torch.equal(la[:20], lb) and torch.equal(va[:20], vb)
        a = model.selfplay_step_boards(boards, player, left, u, 0.7, index=index, view=3)
        b = model.selfplay_step_boards(boards, player, left, u[:50], 0.7, index=index[:50], view=3)
        for p, q in zip(a, b):
            assert torch.equal(p[:50], q)


@pytest.mark.parametrize("precision", ["fp32", "bf16c"])
def test_graphs_and_streams(cuda, precision):
    model, (x, _) = _model(cuda), _inputs(20)
    model.precision = precision
    model.cascade_threshold = 0.3      # (several boards go twice)
    xs = [torch.roll(x, i, 0).to(cuda) for i in range(3)]
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
        streams = [torch.cuda.Stream() for _ in range(3)]
        torch.cuda.synchronize()
        got = []
        for r in range(6):
            for i, s in enumerate(streams):
                with torch.cuda.stream(s):
                    got.append((i, model(xs[i])))
        torch.cuda.synchronize()
        for i, (lg, vg) in got:
            assert torch.equal(lg, want[i][0]) and torch.equal(vg, want[i][1])
