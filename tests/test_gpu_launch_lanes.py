"""Launch settings of topologies with a multi-lane kernel: the one-thread
kernel's launch shapes, asked for with one lane per env, and tuners that leave
the choice of the kernel alone."""

import contextlib

import numpy as np
import pytest
import torch

from brax_amd import systems as S
from brax_amd.generalized import autotune, pipeline

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _inputs(sys, n, T, seed, drop=0.0):
  rng = np.random.default_rng(seed)
  q = sys.init_q + rng.uniform(-0.1, 0.1, (n, sys.q_size()))
  q[:, 2] -= drop
  t = lambda x: torch.tensor(np.asarray(x, np.float32), device=DEV)  # noqa: E731
  return (t(q), t(0.1 * rng.standard_normal((n, sys.qd_size()))),
          t(rng.uniform(-1, 1, (T, n, sys.act_size()))))


@contextlib.contextmanager
def _settings(m, **settings):
  kinds = {"step": autotune.STEP, "tile": autotune.TILE, "lanes": autotune.LANES}
  try:
    for k, v in settings.items():
      autotune.set_launch(m, kinds[k], v)
    yield
  finally:
    for kind in kinds.values():
      autotune.set_launch(m, kind, 0)


def _rollout(sys, q, qd, acts):
  st, (qt, qdt) = pipeline.rollout(sys, pipeline.State(q=q, qd=qd, x=None, xd=None), acts, 5,
                                   trajectory=True)
  return [t.cpu().numpy() for t in (qt, qdt, st.q, st.qd, st.x.pos, st.xd.vel, st.status)]


@pytest.mark.parametrize("name,n", [("quadruped", 200), ("ant", 65), ("humanoid", 70)])
def test_one_thread_rollout_bitwise_across_envs_per_workgroup(name, n):
  """A ragged batch over 3 env steps: the same bits for 64, 16, 4 and 1 envs
  per workgroup of the one-thread kernel."""
  sys = S.ant() if name == "ant" else getattr(S, name)(0)
  q, qd, acts = _inputs(sys, n, 3, seed=3)
  m = pipeline.device_model(sys, DEV)
  out = []
  for epw in (64, 16, 4, 1):
    with _settings(m, lanes=1, step=epw):
      assert autotune.get_launch(m, autotune.LANES) == 1
      out.append(_rollout(sys, q, qd, acts))
  for other in out[1:]:
    for a, b in zip(out[0], other):
      np.testing.assert_array_equal(a, b)


def test_tuners_leave_the_lanes_alone():
  """Tuned for a batch, a four-legged model steps a small batch on the same
  kernel to the same bits; the tile is tuned only where one thread per env
  runs, by the horizon that it is timed over."""
  sys = S.quadruped(0)
  m = pipeline.device_model(sys, DEV)
  q, qd, acts = _inputs(sys, 700, 6, seed=5, drop=0.2)
  small = _inputs(sys, 3, 2, seed=6, drop=0.2)
  with _settings(m):
    before = _rollout(sys, *small)
    assert autotune.tune_tile(sys, q, qd, acts, 5) in autotune.tiles(sys)
    assert autotune.tune_step(sys, q, qd, acts[:2], 5) in autotune.CANDIDATES
    assert autotune.get_launch(m, autotune.LANES) == 4
    for a, b in zip(before, _rollout(sys, *small)):
      np.testing.assert_array_equal(a, b)
  with _settings(m, lanes=1):
    for T in (1, 6):
      k = autotune.tune_tile(sys, q, qd, acts[:T], 5)
      assert k in autotune.tiles(sys) and autotune.get_launch(m, autotune.TILE) == k
      assert autotune.tune_tile(sys, q, qd, acts[:T], 5) == k
    assert autotune.get_launch(m, autotune.LANES) == 1
