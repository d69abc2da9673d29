"""The autotuner's choices on a stand-in context (no GPU): the library's own
block length is among the default candidates and wins when it is the fastest;
it stays when the group is skipped; otherwise the fastest length is set."""
from types import SimpleNamespace

import pytest

from btrc_amd import _abi
from btrc_amd.autotune import autotune


class StandIn:
    def __init__(self, seconds):
        self.seconds, self.tuning = seconds, dict(graph_bounces=0)

    def set_tuning(self, **kw):
        self.tuning.update(kw)

    def get_tuning(self):
        return dict(self.tuning)

    def render(self, p):
        return SimpleNamespace(stage_ms=[1.0] * 8, seconds=self.seconds(self.tuning["graph_bounces"], p.state_count))


@pytest.mark.parametrize("fastest", [0, 2, 4, 8])
def test_block_length(fastest):
    ctx = StandIn(lambda g, pool: 1.0 if g == fastest else 2.0)
    best, _, table = autotune(ctx, _abi.RenderParams(state_count=1 << 20), waves=(), stage_blocks=())
    assert best["graph_bounces"] == ctx.tuning["graph_bounces"] == fastest
    assert {v[1] for k, v, _ in table if k == "pool_and_graph"} == {0, 2, 4, 8}


def test_skipped_group_keeps_the_library_choice():
    ctx = StandIn(lambda g, pool: pool)
    best, pool, _ = autotune(ctx, _abi.RenderParams(), waves=(), stage_blocks=(), graph_bounces=(),
                             pools=(1 << 20, 1 << 18))
    assert pool == 1 << 18 and best["graph_bounces"] == ctx.tuning["graph_bounces"] == 0
