"""Win check of c6_env_step on crowded boards: runs of every length in every direction, across the
number of neighbours a lane asks for at once (eight), against the oracle."""
import pytest
import torch

import connect6_amd as c6
from oracle import env_ref as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("board,win", [(19, 1), (19, 2), (19, 6), (19, 9), (19, 10), (19, 17), (19, 18), (5, 9), (33, 20)])
def test_long_runs_match_oracle(cuda, board, win):
    num, gen = 1003, torch.Generator().manual_seed(win)
    st = E.new_state(num, board, win)
    density = torch.rand(num, 1, 1, generator=gen) * 0.12 + 0.88          # of the mover's stones
    mine = torch.rand(num, board, board, generator=gen) < density
    st.current_player[:] = (torch.randint(0, 2, (num,), generator=gen) * 2 - 1).to(torch.int8)
    other = (torch.randint(-1, 1, (num, board, board), generator=gen)).to(torch.int8)   # free or the other side's
    st.boards[:] = torch.where(mine, torch.ones_like(other), other) * st.current_player.view(-1, 1, 1)
    env = c6.VectorConnect6(num, board, win, device=cuda)
    for name in ("boards", "current_player", "stones_left", "empty_count", "move_count"):
        getattr(env, name).copy_(getattr(st, name))
    actions = torch.randint(0, board * board, (num,), generator=gen)
    want, got = E.step(st, actions), env.step(actions.to(cuda))
    assert torch.equal(got.reward.cpu(), want.reward) and torch.equal(got.winner.cpu(), want.winner)
    assert torch.equal(got.done.cpu(), want.done) and torch.equal(env.boards.cpu(), st.boards)
    assert torch.equal(got.transition_sign.cpu(), want.transition_sign)
    assert win < 3 or board == 5 or 0 < int(want.reward.sum()) < num
