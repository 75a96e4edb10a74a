"""An env's result does not depend on the envs or the steps around it, at any
batch size and rollout length: the kernel follows from the topology and the
launch settings alone."""

import numpy as np
import pytest
import torch

from brax_amd import systems as S
from brax_amd.generalized import autotune, pipeline

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("name,n", [("quadruped", 32769), ("quadruped", 65537), ("ant", 40000),
                                    ("humanoid", 5000)])
def test_long_rollout_of_a_large_batch(name, n):
  """Six env steps of five substeps in one rollout, in two of three, and of
  40 of the envs alone: the same bits."""
  sys = S.ant() if name == "ant" else getattr(S, name)(0)
  gen = torch.Generator(device=DEV)
  gen.manual_seed(n)
  q = torch.tensor(sys.init_q, device=DEV, dtype=torch.float32) + 0.2 * (
      torch.rand(n, sys.q_size(), device=DEV, generator=gen) - 0.5)
  qd = 0.1 * torch.randn(n, sys.qd_size(), device=DEV, generator=gen)
  scale = 0.4 if name == "humanoid" else 1.0
  acts = scale * (2 * torch.rand(6, n, sys.act_size(), device=DEV, generator=gen) - 1)

  def roll(q, qd, acts):
    st, _ = pipeline.rollout(sys, pipeline.State(q=q, qd=qd, x=None, xd=None), acts, 5,
                             frames=False)
    return st.q, st.qd
  whole = roll(q, qd, acts)
  halves = roll(*roll(q, qd, acts[:3]), acts[3:])
  some = torch.arange(0, n, n // 39, device=DEV)
  few = roll(q[some], qd[some], acts[:, some])
  bits = lambda t: t.view(torch.int32)  # noqa: E731
  for k in range(2):
    assert torch.equal(bits(whole[k]), bits(halves[k]))
    assert torch.equal(bits(whole[k][some]), bits(few[k]))


def test_lanes_in_use():
  """The launch query names the kernel that runs: a lane per leg by default,
  one thread per env when asked for or when a tile is chosen."""
  sys = S.quadruped(0)
  m = pipeline.device_model(sys, DEV)
  assert autotune.get_launch(m, autotune.LANES) == 4
  try:
    autotune.set_launch(m, autotune.TILE, 6)
    assert autotune.get_launch(m, autotune.LANES) == 1
    autotune.set_launch(m, autotune.LANES, 4)
    assert autotune.get_launch(m, autotune.LANES) == 4
    autotune.set_launch(m, autotune.TILE, 0)
    autotune.set_launch(m, autotune.LANES, 1)
    assert autotune.get_launch(m, autotune.LANES) == 1
  finally:
    autotune.set_launch(m, autotune.TILE, 0)
    autotune.set_launch(m, autotune.LANES, 0)
  assert np.isin(autotune.get_launch(m, autotune.TILE), autotune.tiles(sys))
