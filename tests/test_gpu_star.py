"""The lane-per-leg kernel (a free root with four equal legs: quadruped, ant)
against the one-thread kernel and the float64 oracle, at batch sizes around a
wavefront's 16 envs.

Tolerance: the parity band |gpu - ref| <= 1e-5 + 1e-4 |ref|."""

import numpy as np
import pytest
import torch

from brax_amd import systems as S
from brax_amd.generalized import autotune, pipeline
from oracle.generalized import Oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"
SYSTEMS = {"quadruped": S.quadruped(0), "ant": S.ant()}


def _ratio(a, ref):
  a, ref = np.asarray(a, np.float64), np.asarray(ref, np.float64)
  return (np.abs(a - ref) / (1e-5 + 1e-4 * np.abs(ref))).max()


def _t(x):
  return torch.tensor(np.asarray(x, np.float32), device=DEV)


def _inputs(name, n, height):
  sys = SYSTEMS[name]
  rng = np.random.default_rng(n)
  q = np.array(sys.init_q) + rng.uniform(-0.1, 0.1, (n, 15))
  q[:, 2] += height
  q[:, 3:7] /= np.linalg.norm(q[:, 3:7], axis=1, keepdims=True)
  qd = 0.1 * rng.standard_normal((n, 14))
  return sys, q.astype(np.float32), qd.astype(np.float32), rng


def _both(sys, fn):
  """fn() on the lane-per-leg kernel and on the one-thread kernel."""
  m = pipeline.device_model(sys, torch.device(DEV))
  assert autotune.get_launch(m, autotune.LANES) == 4
  star = fn()
  autotune.set_launch(m, autotune.LANES, 1)
  try:
    return star, fn()
  finally:
    autotune.set_launch(m, autotune.LANES, 0)


@pytest.mark.parametrize("name", ["quadruped", "ant"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 65])
def test_flight_rollout_matches_one_thread(name, n):
  """Two env steps off the ground: trajectory, final state, frames, status."""
  sys, q, qd, rng = _inputs(name, n, 5.0)
  acts = _t(rng.uniform(-0.2, 0.2, (2, n, 8)))

  def fn():
    st = pipeline.State(q=_t(q), qd=_t(qd), x=None, xd=None)
    st, (qt, qdt) = pipeline.rollout(sys, st, acts, 5, trajectory=True)
    return [x.cpu().numpy() for x in (qt, qdt, st.q, st.qd, st.x.pos, st.x.rot, st.xd.ang,
                                      st.xd.vel)], st.status.cpu().numpy()
  (a, sa), (b, sb) = _both(sys, fn)
  np.testing.assert_array_equal(sa, sb)
  for x, y in zip(a, b):
    assert _ratio(x, y) <= 1.0


@pytest.mark.parametrize("n", [1, 17, 65])
def test_floor_substep_matches_the_oracle(n):
  """One substep of quadrupeds sunk to 0.06-0.3 m: up to every candidate of a
  leg in contact; qf_smooth, contacts and status as the one-thread kernel's."""
  sys, q, qd, rng = _inputs("quadruped", n, 0.0)
  q[:, 2] = rng.uniform(0.06, 0.3, n)
  act = rng.uniform(-1, 1, (n, 8)).astype(np.float32)

  def fn():
    st = pipeline.State(q=_t(q), qd=_t(qd), x=None, xd=None)
    pr = pipeline.probe(sys, st, _t(act), 1)
    st = pipeline.pipeline_step(sys, st, _t(act), 1)
    return {k: v.cpu().numpy() for k, v in pr.items()}, st
  (a, sa), (b, sb) = _both(sys, fn)
  np.testing.assert_array_equal(a["n_contacts"], b["n_contacts"])
  np.testing.assert_array_equal(sa.status.cpu().numpy(), sb.status.cpu().numpy())
  assert _ratio(a["qf_smooth"], b["qf_smooth"]) <= 1.0
  o = Oracle(sys, torch.float64, inverse="exact")
  ref = o.step(o.init(q.astype(np.float64), qd.astype(np.float64)), act.astype(np.float64))
  assert _ratio(sa.q.cpu(), ref.q) <= 1.0
  assert _ratio(sa.qd.cpu(), ref.qd) <= 1.0


@pytest.mark.parametrize("name", ["quadruped", "ant"])
def test_env_does_not_depend_on_its_wavefront(name):
  """An env on the floor steps to the same bits alone and among others."""
  sys, q, qd, rng = _inputs(name, 33, -0.1)
  act = _t(rng.uniform(-1, 1, (33, 8)))
  whole = pipeline.pipeline_step(sys, pipeline.State(q=_t(q), qd=_t(qd), x=None, xd=None), act, 2)
  for i in (0, 16, 31, 32):
    one = pipeline.pipeline_step(
        sys, pipeline.State(q=_t(q[i:i + 1]), qd=_t(qd[i:i + 1]), x=None, xd=None),
        act[i:i + 1], 2)
    np.testing.assert_array_equal(one.q.cpu().numpy(), whole.q[i:i + 1].cpu().numpy())
    np.testing.assert_array_equal(one.qd.cpu().numpy(), whole.qd[i:i + 1].cpu().numpy())
