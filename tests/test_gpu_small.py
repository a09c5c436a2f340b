"""One-launch forward of small networks (c6_forward_generic_packed) against the oracle, at the sizes
where its layout changes: boards of one square to 19 x 19, channels around multiples of 8 and 16,
wide and 1x1 kernels, one to many boards per workgroup, several weight sets."""
import ctypes

import pytest
import torch

import connect6_amd as c6
from connect6_amd import _lib
from connect6_amd.model import pack_generic, run_forward_generic, run_packed_generic, architecture_bytes
from connect6_amd.synthetic import gen_boards
from oracle import torch_ref as R
from tests.util import rel_l2

pytestmark = pytest.mark.gpu


def _inputs(batch, board, seed):
    x = torch.randn(batch, 3, board, board, generator=torch.Generator().manual_seed(seed))
    x[:, :2] = (x[:, :2] > 0.7).float()
    return x


@pytest.mark.parametrize("board,kernels,channels,batch", [
    (1, [1], [1], 70), (2, [3, 1], [8, 9], 33), (5, [3, 3, 3], [8, 8, 16], 1), (5, [3, 3, 3], [8, 8, 16], 3000),
    (7, [7, 5], [17, 48], 300), (9, [5, 3, 3], [16, 32, 32], 1024), (9, [5, 3, 3], [16, 32, 32], 2),
    (11, [11, 1, 3], [33, 7, 40], 65), (13, [3, 3, 5, 1], [24, 32, 16, 47], 301), (19, [3, 3], [32, 48], 5),
    (19, [7, 3, 3], [32, 32, 32], 259),
])
def test_fits_and_matches_the_oracle(cuda, board, kernels, channels, batch):
    st = R.init_state(7, "torch_default", kernels=kernels, channels=channels)
    model = c6.PolicyValueNet(board_size=board, kernels=kernels, channels=channels).to(cuda).eval()
    model.load_state_dict(st)
    assert _lib.generic_packed_bytes(board, kernels, channels, _lib.PREC_F32) > 0
    x = _inputs(batch, board, 3)
    xd = x.to(cuda)
    legal = ((x[:, 0] == 0) & (x[:, 1] == 0)).flatten(1)
    dev_state = {k: v.to(cuda) for k, v in st.items()}
    with torch.inference_mode():
        lo, vo = R.forward(st, x)
        lg, vg = model(xd)
        # fp32 sums of at most 9 x 48 x 9 products and sigmoids to 2^-22: the oracle's own order of
        # summation moves these networks by 1e-6
        assert rel_l2(lg, lo) <= 5e-6 and rel_l2(vg, vo) <= 5e-6
        # the same weights straight from the tensors: the same values, bit for bit
        lr, vr = run_forward_generic(xd, dev_state, kernels, channels, _lib.PREC_F32)
        assert torch.equal(lg, lr) and torch.equal(vg, vr)
        # a board's result does not depend on how many share its workgroup
        one, vone = model(xd[batch - 1:])
        assert torch.equal(one, lg[batch - 1:]) and torch.equal(vone, vg[batch - 1:])
        lm, _ = model.forward_masked(xd, legal.to(cuda))
        assert torch.equal(lm.cpu(), R.mask_logits(lg.cpu(), legal))
        for name, tol in (("bf16", 2e-3), ("fp16", 2e-3)):
            model.precision = name
            lb, _ = model(xd)
            want = R.forward_bf16_emulated(st, x)[0] if name == "bf16" else lo
            # bf16: the emulation's roundings in another order of summation (a few fall the other way);
            # fp16: half an ulp (2^-12) at every operand of two to four layers
            assert rel_l2(lb, want) <= tol, (name, rel_l2(lb, want))


def _fp32_chain(st, x, layers):
    """The forward with every output one chain of fp32 multiply-adds, as fp32 arithmetic gives it (products exact,
    each sum rounded once): float64 operations, rounded."""
    import torch.nn.functional as F

    a = x
    for i in range(layers):
        w, b = st[f"convs.{i}.weight"], st[f"convs.{i}.bias"]
        k = w.shape[2]
        cols = F.unfold(a.double(), k, padding=k // 2)
        acc = b.view(1, -1, 1).expand(x.shape[0], -1, cols.shape[2])
        for j, col in enumerate(cols.unbind(1)):
            acc = (acc.double() + w.flatten(1)[:, j].double().view(1, -1, 1) * col.unsqueeze(1)).float()
        a = F.silu(acc).view(x.shape[0], -1, *x.shape[2:])
    f = a.flatten(2)
    heads = []
    for name in ("policy_output", "value_output"):
        acc = st[f"{name}.bias"].view(1, 1).expand(x.shape[0], f.shape[2]) if name == "policy_output" else torch.zeros_like(f[:, 0])
        for c in range(f.shape[1]):
            acc = (acc.double() + st[f"{name}.weight"].flatten()[c].double() * f[:, c].double()).float()
        heads.append(acc)
    return heads[0], torch.tanh(heads[1].mean(1) + st["value_output.bias"])


@pytest.mark.parametrize("init", ["reference", "torch_default"])
@pytest.mark.parametrize("board,kernels,channels", [(9, [5, 3, 3], [16, 32, 32]), (13, [7, 5, 5, 5, 5], [32] * 5)])
def test_no_further_from_float64_than_fp32(cuda, board, kernels, channels, init):
    nets, boards = 16, 16
    err = {"here": [], "chain": []}
    for s in range(nets):
        st = R.init_state(300 + s, init, kernels=kernels, channels=channels)
        model = c6.PolicyValueNet(board_size=board, kernels=kernels, channels=channels).to(cuda).eval()
        model.load_state_dict(st)
        x, _ = gen_boards(boards, board * board // 2, 900 + s, board_size=board)
        l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x.double())
        with torch.inference_mode():
            outs = {"here": model(x.to(cuda)),
                    "chain": _fp32_chain({k: v.to(cuda) for k, v in st.items()}, x.to(cuda), len(kernels))}
        for name, (l, v) in outs.items():
            err[name].append(((l.double().cpu() - l64) / l64.pow(2).mean().sqrt(), v.double().cpu() - v64))
    logits, value = [{n: torch.stack([e[i] for e in es]) for n, es in err.items()} for i in (0, 1)]

    def rms(t):
        return float(t.pow(2).mean().sqrt())
    # Measured against the layer-by-layer kernel, a chain as above: logits 0.3 to 0.5 of its error, the value 0.5
    # and its mean over a network's boards 0.25 to 0.5.  (PyTorch's initialisation makes the value so large that
    # rounding it once is most of either error, and its mean one of sixteen roundings.)
    assert rms(logits["here"]) <= 0.75 * rms(logits["chain"])
    assert rms(value["here"]) <= rms(value["chain"])
    if init == "reference":
        assert rms(value["here"].mean(1)) <= rms(value["chain"].mean(1))


def test_weight_sets_and_an_architecture_without_packed_form(cuda):
    board, kernels, channels = 9, [3, 3], [16, 24]
    states = [R.init_state(20 + i, "torch_default", kernels=kernels, channels=channels) for i in range(3)]
    stacked = {k: torch.stack([s[k] for s in states]).to(cuda) for k in states[0]}
    x = _inputs(3 * 11, board, 5).to(cuda)
    arch = architecture_bytes(kernels, channels)
    for prec in (_lib.PREC_F32, _lib.PREC_BF16C, _lib.PREC_BF16, _lib.PREC_F16):
        packed = pack_generic(stacked, board, kernels, channels, prec, cuda, groups=3)
        lg, vg = run_packed_generic(x, packed, arch, prec, groups=3)
        lr, vr = run_forward_generic(x, stacked, kernels, channels, prec, groups=3)
        assert torch.equal(lg, lr) and torch.equal(vg, vr)
        for i in range(3):
            one, v1 = run_packed_generic(x[11 * i:11 * i + 11], packed[i:i + 1], arch, prec)
            assert torch.equal(one, lg[11 * i:11 * i + 11]) and torch.equal(v1, vg[11 * i:11 * i + 11])
    for kernels, channels in (([3], [49]), ([3, 7], [48, 8])):   # too many channels; too large for the LDS
        assert _lib.generic_packed_bytes(19, kernels, channels, _lib.PREC_F32) == 0
        st = R.init_state(3, "torch_default", kernels=kernels, channels=channels)
        model = c6.PolicyValueNet(board_size=19, kernels=kernels, channels=channels).to(cuda).eval()
        model.load_state_dict(st)
        xb = _inputs(4, 19, 9)
        with torch.inference_mode():
            lo, vo = R.forward(st, xb)
            lg, vg = model(xb.to(cuda))
        assert rel_l2(lg, lo) <= 5e-6 and rel_l2(vg, vo) <= 5e-6


@pytest.mark.parametrize("precision", ["fp32", "bf16c", "fp16"])
def test_parameters_are_read_on_every_call(cuda, precision):
    """Edits that no version counter shows (an average of weights kept through ``p.data``), replaced parameters,
    other types: what the module holds at the call is what answers."""
    board, kernels, channels = 9, [5, 3, 3], [16, 32, 24]
    model = c6.PolicyValueNet(board_size=board, kernels=kernels, channels=channels).to(cuda).eval()
    model.load_state_dict(R.init_state(31, "torch_default", kernels=kernels, channels=channels))
    model.precision = precision
    x = _inputs(37, board, 5).to(cuda)

    def check():
        other = c6.PolicyValueNet(board_size=board, kernels=kernels, channels=channels).to(cuda).eval()
        other.load_state_dict(model.state_dict())
        other.precision = precision
        with torch.inference_mode():
            got, want = model(x), other(x)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        return got[0]

    seen = [check()]
    model.convs[1].weight.data.mul_(0.5)
    seen.append(check())
    model.policy_output.bias.data.add_(1.0)
    seen.append(check())
    model.convs[2].bias = torch.nn.Parameter(torch.ones(24, device=cuda))
    seen.append(check())
    for a, b in zip(seen, seen[1:]):
        assert not torch.equal(a, b)
    model.convs[1].weight = torch.nn.Parameter(model.convs[1].weight.detach().cpu().double())   # converted on the way
    assert torch.equal(check(), seen[-1])
    static = x.clone()                     # ... and in every replay of a graph
    model.convs[1].to(cuda, torch.float32)
    with torch.inference_mode():
        model(static)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, _ = model(static)
        for factor in (1.0, 2.0, 0.25):
            model.convs[1].weight.data.mul_(factor)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, model(x)[0]), factor


@pytest.mark.parametrize("board,kernels,channels,batch", [(5, [3, 3], [8, 17], 3), (9, [5, 3, 3], [16, 32, 48], 70), (19, [7, 1], [33, 8], 9)])
@pytest.mark.parametrize("prec", [_lib.PREC_F32, _lib.PREC_BF16, _lib.PREC_BF16F6])
def test_weights_packed_for_the_call_or_read_as_they_are(cuda, board, kernels, channels, batch, prec):
    """The same bits; inputs that are exact in bf16 and inputs that are not, one of them in a batch of the other."""
    st = {k: v.to(cuda) for k, v in R.init_state(9, "torch_default", kernels=kernels, channels=channels).items()}
    arch = architecture_bytes(kernels, channels)
    x = _inputs(batch, board, 8)
    x[:, 2] = 1.0
    for inexact in (False, True):
        if inexact:
            x[batch // 2, 1] *= 0.3
        with torch.inference_mode():
            weights = pack_generic(st, board, kernels, channels, prec, cuda)
            packed = run_packed_generic(x.to(cuda), weights, arch, prec)
            raw = run_forward_generic(x.to(cuda), st, kernels, channels, prec, static_workspace=True)
            alone = run_packed_generic(x[:1].to(cuda), weights, arch, prec)
        assert torch.equal(packed[0], raw[0]) and torch.equal(packed[1], raw[1])
        assert torch.equal(packed[0][:1], alone[0]) and torch.equal(packed[1][:1], alone[1])


@pytest.mark.parametrize("groups", [1, 3])
@pytest.mark.parametrize("prec", [_lib.PREC_F32, _lib.PREC_BF16])
def test_the_workspace_of_a_one_launch_network_is_left_alone(cuda, groups, prec):
    """Calls on several streams may share it, however large it is."""
    board, kernels, channels, batch = 9, [5, 3, 3], [16, 32, 32], 20
    states = [R.init_state(50 + i, "torch_default", kernels=kernels, channels=channels) for i in range(groups)]
    st = {k: torch.stack([s[k] for s in states]).to(cuda) for k in states[0]}
    x = _inputs(groups * batch, board, 4).to(cuda)
    ints, ptrs, lib = ctypes.c_int * 3, ctypes.c_void_p * 3, _lib.load()
    ks, cs = ints(*kernels), ints(*channels)
    need = ctypes.c_size_t(0)
    _lib.check(lib.c6_generic_workspace_bytes(groups * batch, board, 3, cs, ctypes.byref(need)), "c6_generic_workspace_bytes")
    size = need.value + groups * _lib.generic_packed_bytes(board, kernels, channels, prec)
    workspace = torch.full((size,), 0xA5, dtype=torch.uint8, device=cuda)
    logits, value = torch.empty(groups * batch, board * board, device=cuda), torch.empty(groups * batch, device=cuda)
    rc = lib.c6_forward_generic_grouped(
        x.data_ptr(), _lib.DT_F32, groups, batch, board, 3, ks, cs, ptrs(*[st[f"convs.{i}.weight"].data_ptr() for i in range(3)]),
        ptrs(*[st[f"convs.{i}.bias"].data_ptr() for i in range(3)]), *[st[f"{h}_output.{k}"].data_ptr() for h in ("policy", "value")
                                                                      for k in ("weight", "bias")],
        prec, workspace.data_ptr(), size, logits.data_ptr(), value.data_ptr(), _lib.MASK_NONE, None, 0.0, _lib.stream_ptr(cuda))
    _lib.check(rc, "c6_forward_generic_grouped")
    assert bool((workspace == 0xA5).all())
    packed = pack_generic(st, board, kernels, channels, prec, cuda, groups=groups)
    want = run_packed_generic(x, packed, architecture_bytes(kernels, channels), prec, groups=groups)
    assert torch.equal(logits, want[0]) and torch.equal(value, want[1])


@pytest.mark.parametrize("board,kernels,channels,batch", [(1, [1], [1], 70), (9, [3], [48], 300), (19, [5], [17], 40)])
def test_one_layer_with_inputs_that_are_not_exact_in_bf16(cuda, board, kernels, channels, batch):
    """A network without a layer behind its first: with a value head, and packed without one (the heads then store
    zeros where the inputs' exactness was noted).  Weights read as they are take every part of an input always."""
    states = [R.init_state(40 + i, "torch_default", kernels=kernels, channels=channels) for i in range(2)]
    x = torch.randn(2 * batch, 3, board, board, generator=torch.Generator().manual_seed(6))
    xd, arch = x.to(cuda), architecture_bytes(kernels, channels)
    model = c6.PolicyValueNet(board_size=board, kernels=kernels, channels=channels).to(cuda).eval()
    stacked = {k: torch.stack([s[k] for s in states]).to(cuda) for k in states[0]}
    policy_only = pack_generic(stacked, board, kernels, channels, _lib.PREC_F32, cuda, groups=2, want_value=False)
    with torch.inference_mode():
        sets, _ = run_packed_generic(xd, policy_only, arch, _lib.PREC_F32, groups=2, want_value=False)
        for i, st in enumerate(states):
            model.load_state_dict(st)
            part = slice(i * batch, (i + 1) * batch)
            raw = run_forward_generic(xd[part], {k: v.to(cuda) for k, v in st.items()}, kernels, channels, _lib.PREC_F32,
                                      static_workspace=True)
            lg, vg = model(xd[part])
            assert torch.equal(lg, raw[0]) and torch.equal(vg, raw[1])
            assert torch.equal(sets[part], raw[0])
            lo, vo = R.forward(st, x[part])
            # fp32 sums of at most 25 x 3 and 48 products; one part of the inputs alone would be off by 2^-9
            assert rel_l2(lg, lo) <= 5e-6 and rel_l2(vg, vo) <= 5e-6


@pytest.mark.parametrize("board,kernels,channels,batch", [
    (18, [7] * 8, [48] * 8, 3), (16, [9] * 15, [48] * 15, 2), (11, [17, 17], [48, 48], 1), (19, [11] * 16, [32] * 16, 300)])
def test_networks_that_fill_the_lds(cuda, board, kernels, channels, batch):
    """No room beside the activations for a copy of the biases and head weights: one launch all the same."""
    states = [R.init_state(60 + i, "torch_default", kernels=kernels, channels=channels) for i in range(2)]
    stacked = {k: torch.stack([s[k] for s in states]).to(cuda) for k in states[0]}
    x, arch = _inputs(2 * batch, board, 7).to(cuda), architecture_bytes(kernels, channels)
    for prec in (_lib.PREC_F32, _lib.PREC_BF16F6):
        packed = pack_generic(stacked, board, kernels, channels, prec, cuda, groups=2)
        lg, vg = run_packed_generic(x, packed, arch, prec, groups=2)
        for i, st in enumerate(states):
            part = slice(i * batch, (i + 1) * batch)
            raw = run_forward_generic(x[part], {k: v.to(cuda) for k, v in st.items()}, kernels, channels, prec)
            assert torch.equal(lg[part], raw[0]) and torch.equal(vg[part], raw[1])
            if prec == _lib.PREC_F32 and batch <= 3:
                l64, v64 = R.forward({k: v.double() for k, v in st.items()}, x[part].double().cpu())
                # sixteen layers at most, each a sum of at most 17 x 17 x 48 products rounded to fp32 (2^-24)
                assert rel_l2(lg[part], l64) <= 1e-5 and rel_l2(vg[part], v64) <= 1e-5


def test_board_size_set_after_construction(cuda):
    """The network is fully convolutional: the same module on boards of another size."""
    for kernels, channels, first, second in ((None, None, 19, 9), ([3, 3], [8, 16], 7, 13)):
        model = c6.PolicyValueNet(board_size=first, kernels=kernels, channels=channels).to(cuda).eval()
        for board in (first, second, first):
            model.board_size, model.action_size = board, board * board
            assert model.is_default_architecture == (kernels is None and board == 19)
            x = _inputs(3, board, 2)
            with torch.inference_mode():
                lo, vo = R.forward({k: v.cpu() for k, v in model.state_dict().items()}, x)
                lg, vg = model(x.to(cuda))
            assert rel_l2(lg, lo) <= 1e-5 and rel_l2(vg, vo) <= 1e-4


@pytest.mark.parametrize("where,index,value", [
    ("x", (1, 0, 4, 4), float("inf")), ("x", (1, 0, 4, 4), float("nan")), ("x", (1, 0, 4, 4), 3.4e38), ("x", (1, 2), -3.39e38),
    ("convs.2.weight", (5, 3, 1, 1), float("inf")), ("convs.0.weight", (3, 0, 2, 2), 3.38e38), ("convs.0.bias", 5, -1e34),
    ("convs.1.bias", 5, -3.4e38), ("convs.1.bias", 5, 3.38e38), ("convs.1.bias", 5, float("inf")),
    ("convs.2.bias", 5, -float("inf")), ("convs.2.bias", 5, 3.4e38)])
def test_infinities_and_the_ends_of_the_range_as_in_fp32(cuda, where, index, value):
    kernels, channels = [5, 3, 3], [16, 32, 32]
    st = R.init_state(31, "torch_default", kernels=kernels, channels=channels)
    x = _inputs(3, 9, 5)
    (x if where == "x" else st[where])[index] = value
    model = c6.PolicyValueNet(board_size=9, kernels=kernels, channels=channels).to(cuda).eval()
    model.load_state_dict(st)
    dev = {k: v.to(cuda) for k, v in st.items()}
    with torch.inference_mode():
        want = _fp32_chain(dev, x.to(cuda), 3)
        got = model(x.to(cuda))
    for a, b in zip(want, got):
        a, b = a.double().cpu(), b.double().cpu()
        assert torch.equal(a.isnan(), b.isnan())
        ends = a.isinf() | b.isinf()
        assert torch.equal(a[ends], b[ends])
        fine = a.isfinite()
        size = a.where(fine, torch.zeros_like(a)).abs().flatten(1).amax(1, keepdim=True) if a.ndim > 1 else a.abs()
        assert bool(((a - b).abs()[fine] <= (2e-5 * size).expand_as(a)[fine]).all())
