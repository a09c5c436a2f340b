"""fp32 through 16-bit parts of its operands (C6_PREC_F32S) against a float64 forward: no further from
it than fp32 arithmetic, whatever the input planes hold.  Ordinary boards go through two fp16 parts (inputs that are exact in
fp16 are staged once and others in two parts, a constant third plane is contracted through a table), those with infinities and
the ends of fp32's range through three bf16 parts; test_gpu_half.py has the lines between the two."""
import pytest
import torch

import connect6_amd as c6
from connect6_amd import _lib
from connect6_amd.model import run_forward
from connect6_amd.synthetic import gen_boards, gen_uniform
from oracle import torch_ref as R
from tests.util import rel_l2

pytestmark = pytest.mark.gpu


def _planes(kind, n):
    g = torch.Generator().manual_seed(4)
    x, _ = gen_boards(n, 200, 3)
    if kind == "randn":
        x = torch.randn(n, 3, 19, 19, generator=g)
    elif kind == "varying":
        x[:, 2] = (torch.rand(n, 19, 19, generator=g) > 0.5).float()
    elif kind == "inexact constant":
        x[:, 2] = 0.3
    elif kind == "one inexact square":       # only one thread of the workgroup sees it
        x[:, 2, 17, 3] = 0.3
    elif kind == "large":
        x = x * 300.0
    return x


@pytest.mark.parametrize("init", ["reference", "torch_default"])
@pytest.mark.parametrize("kind", ["boards", "randn", "varying", "inexact constant", "one inexact square", "large"])
def test_no_further_from_float64_than_fp32(cuda, kind, init):
    st = R.init_state(5, init)
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(st)
    x = _planes(kind, 33)
    l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x.double())
    err = {}
    with torch.inference_mode():
        for prec in (_lib.PREC_F32, _lib.PREC_F32S):
            lg, vg, _, _ = run_forward(x.to(cuda), model.packed_weights(prec), prec, 1, 33)
            err[prec] = (rel_l2(lg.double().cpu(), l64), rel_l2(vg.double().cpu(), v64))
    # Eight layers of fp32 sums: each of the two results is within a few 2^-24 per layer of float64
    # (logits 0.3 to 0.55 of the other's error); the value, a mean that nearly cancels, scatters over 33
    # boards of one network (over many networks: the test below).
    assert err[_lib.PREC_F32S][0] <= err[_lib.PREC_F32][0], err
    assert err[_lib.PREC_F32S][1] <= err[_lib.PREC_F32][1] + 1e-6, err


@pytest.mark.parametrize("init", ["reference", "torch_default"])
def test_value_and_logits_of_many_networks(cuda, init):
    """Against a float64 forward no larger an error than the fp32 instructions', neither in size nor in its
    mean over a network's boards (what rounds the same way in every square stays in the value, a mean over
    them)."""
    nets, boards = 64, 12
    err = {p: {"value": [], "logits": []} for p in (_lib.PREC_F32, _lib.PREC_F32S)}
    for s in range(nets):
        st = R.init_state(1000 + s, init)
        model = c6.PolicyValueNet().to(cuda).eval()
        model.load_state_dict(st)
        x, _ = gen_boards(boards, 200, 5000 + s)
        l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x.double())
        xd = x.to(cuda)
        with torch.inference_mode():
            for prec, e in err.items():
                lg, vg, _, _ = run_forward(xd, model.packed_weights(prec), prec, 1, boards)
                e["value"].append(vg.double().cpu() - v64)
                e["logits"].append((lg.double().cpu() - l64) / l64.pow(2).mean().sqrt())
            one, v1 = model(xd[s % boards: s % boards + 1])   # (a board on its own: the same bits)
            assert torch.equal(one[0], lg[s % boards]) and torch.equal(v1[0], vg[s % boards])
    # Measured over 24 networks, this against the fp32 instructions: value 0.21 (PyTorch's initialisation 0.69) of the error,
    # logits 0.28 (0.20).
    was, now = [{k: torch.stack(v) for k, v in err[p].items()} for p in (_lib.PREC_F32, _lib.PREC_F32S)]
    for name, of in (("value", lambda e: e["value"]), ("mean of the value's", lambda e: e["value"].mean(1)),
                     ("logits", lambda e: e["logits"])):
        a, b = of(was).pow(2).mean().sqrt(), of(now).pow(2).mean().sqrt()
        assert b <= a, (name, float(a), float(b))
    # The mean of a network's logit errors holds what its scaled parameters are rounded to: 0.6e-9 by the weights
    # (24 bits; 0.7e-9 the error of the fp32 instructions, which have them unscaled), 2.3e-9 by biases in fp32
    # (float64 forwards with rounded parameters).  Medians; together 0.9e-9, measured 1.1e-9.
    a, b = [e["logits"].flatten(1).mean(1).abs().median() for e in (was, now)]
    assert b <= 2 * a, (float(a), float(b))


_INF, _NAN = float("inf"), float("nan")
_EXTREMES = [  # (where, index, value); "x": board 1 of three
    ("x", (1, 0, 9, 9), _INF), ("x", (1, 1, 0, 0), -_INF), ("x", (1, 0, 3, 3), _NAN), ("x", (1, 2), _INF),
    ("x", (1, 0, 9, 9), 3.4e38), ("x", (1, 2), -1e38), ("x", (1, 2, 4, 4), 3.39e38), ("x", (1, 0, 5, 7), 1.7e-30),
    ("convs.0.weight", (3, 0, 11, 11), _INF), ("convs.0.weight", (3, 0, 11, 11), 1e38),
    ("convs.3.weight", (3, 0, 1, 1), -_INF), ("convs.7.weight", (5, 3, 1, 1), _INF),
    ("convs.7.weight", (5, 3, 1, 1), -_INF), ("convs.7.weight", (5, 3, 1, 1), 3.4e38),
    ("convs.0.bias", 5, -1e34), ("convs.3.bias", 5, -2e38), ("convs.6.bias", 5, 2e36), ("convs.6.bias", 5, _INF),
    ("convs.7.bias", 5, _INF), ("convs.7.bias", 5, -_INF), ("convs.7.bias", 5, -2.3e38), ("convs.7.bias", 5, _NAN),
    ("policy_output.weight", (0, 5, 0, 0), _INF), ("policy_output.bias", 0, -_INF),
    ("value_output.weight", (0, 5, 0, 0), _NAN), ("value_output.bias", 0, -_INF),
]


@pytest.mark.parametrize("where,index,value", _EXTREMES)
def test_infinities_and_the_ends_of_the_range_as_in_fp32(cuda, where, index, value):
    """What the fp32 instructions make of an infinity, a NaN or a number near the end of fp32.  (Sums and activations
    up to 2.3e38: they carry a factor of 1.44.)"""
    st, x = R.init_state(5, "torch_default"), gen_boards(3, 200, 3)[0]
    (x if where == "x" else st[where])[index] = value
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(st)
    xd = torch.cat([x] * 30).to(cuda)          # one workgroup per board; three boards: several
    with torch.inference_mode():
        want = run_forward(xd[:3], model.packed_weights(_lib.PREC_F32), _lib.PREC_F32, 1, 3)[:2]
        packed = model.packed_weights(_lib.PREC_F32S)
        for n in (3, 90):
            got = run_forward(xd[:n], packed, _lib.PREC_F32S, 1, n)[:2]
            for a, b in zip(want, got):
                a, b = a.double().cpu(), b[:3].double().cpu()
                assert torch.equal(a.isnan(), b.isnan()), n
                ends = a.isinf() | b.isinf()
                assert torch.equal(a[ends], b[ends]), n
                fine = a.isfinite()
                # (either's error is 1e-6 to 2e-6 of a board's logits as a whole; ten times that for the worst square)
                size = a.where(fine, torch.zeros_like(a)).abs().flatten(1).amax(1, keepdim=True) if a.ndim > 1 else a.abs()
                assert bool(((a - b).abs()[fine] <= (2e-5 * size).expand_as(a)[fine]).all()), n


def test_fp32_batches_draws_masks_and_states(cuda):
    st = R.init_state(11, "reference")
    model = c6.PolicyValueNet().to(cuda).eval()
    model.load_state_dict(st)
    x, legal = gen_boards(600, 200, 77)
    xd, ld, u = x.to(cuda), legal.to(cuda), gen_uniform(600, 5).to(cuda)
    boards = (x[:, 0] - x[:, 1]).to(torch.int8).to(cuda)
    player = torch.ones(600, dtype=torch.int8, device=cuda)
    left = (x[:, 2, 0, 0] == 1).to(torch.int8).to(cuda)
    with torch.inference_mode():
        lg, vg = model.forward_masked(xd, ld)
        ag, pg, _ = model.selfplay_step(xd, u, 0.8, legal=ld)
        assert torch.equal(lg == torch.finfo(torch.float32).min, ~ld)
        assert bool(ld.gather(1, ag.view(-1, 1)).all())
        lb, vb = model.forward_boards(boards, player, left)
        assert torch.equal(lb, lg) and torch.equal(vb, vg)
        for n in (1, 2, 37, 255, 257, 513):
            l, v = model.forward_masked(xd[:n], ld[:n])
            a, p, _ = model.selfplay_step(xd[:n], u[:n], 0.8, legal=ld[:n])
            assert torch.equal(l, lg[:n]) and torch.equal(v, vg[:n]), n
            assert torch.equal(a, ag[:n]) and torch.equal(p, pg[:n]), n
