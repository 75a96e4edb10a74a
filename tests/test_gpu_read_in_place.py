"""Steps, rollouts and init read the caller's state where it lies: any strides
give the result of a contiguous copy, the state is left as it was, and a launch
on a given stream reads what the returned State keeps."""

import numpy as np
import pytest
import torch

from brax_amd import systems as S
from brax_amd.generalized import pipeline

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
N = 37
SYSTEMS = {
    "quadruped": lambda: S.quadruped(0),
    "humanoid": lambda: S.humanoid(0),
    "chain": lambda: pipeline.SystemBatch([S.chain(5, i) for i in range(N)]),
}


def _state(sys):
  one = sys.systems[0] if isinstance(sys, pipeline.SystemBatch) else sys
  rng = np.random.default_rng(7)
  t = lambda x: torch.tensor(np.asarray(x, np.float32), device=DEV)  # noqa: E731
  q = t(one.init_q + rng.uniform(-0.05, 0.05, (N, one.q_size())))
  qd = t(0.1 * rng.standard_normal((N, one.qd_size())))
  return q, qd, t(rng.uniform(-0.4, 0.4, (3, N, one.act_size())))


def _laid_out(x, layout):
  """x's values with other strides."""
  if layout == "columns of a wider array":
    wide = torch.full((N, x.shape[1] + 3), float("nan"), device=DEV)
    wide[:, 2:2 + x.shape[1]] = x
    return wide[:, 2:2 + x.shape[1]]
  if layout == "transposed":
    return x.t().contiguous().t()
  if layout == "every other row":
    wide = torch.full((2 * N, x.shape[1]), float("nan"), device=DEV)
    wide[::2] = x
    return wide[::2]
  return x


def _outputs(sys, q, qd, acts):
  out = []
  st = pipeline.init(sys, q, qd)
  out += [st.q, st.qd, st.x.pos, st.xd.vel]
  start = pipeline.State(q=q, qd=qd, x=None, xd=None)
  st = pipeline.pipeline_step(sys, start, acts[0], 2)
  out += [st.q, st.qd, st.x.pos, st.xd.vel, st.status]
  st, (qt, qdt) = pipeline.rollout(sys, start, acts, 2, trajectory=True)
  return out + [st.q, st.qd, st.x.rot, st.status, qt, qdt]


@pytest.mark.parametrize("layout", ["columns of a wider array", "transposed", "every other row"])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_strided_states(name, layout):
  sys = SYSTEMS[name]()
  q, qd, acts = _state(sys)
  want = _outputs(sys, q, qd, acts)
  ql, qdl = _laid_out(q, layout), _laid_out(qd, layout)
  assert not ql.is_contiguous()
  for a, b in zip(want, _outputs(sys, ql, qdl, acts)):
    assert torch.equal(a, b)
  assert torch.equal(ql, q) and torch.equal(qdl, qd)


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_state_is_left_and_not_shared(name):
  """The caller's arrays keep their values and are none of the results'."""
  sys = SYSTEMS[name]()
  q, qd, acts = _state(sys)
  kept = q.clone(), qd.clone()
  out = _outputs(sys, q, qd, acts)
  assert torch.equal(q, kept[0]) and torch.equal(qd, kept[1])
  mine = {t.data_ptr() for t in (q, qd)}
  assert not mine & {t.data_ptr() for t in out}


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_rollout_on_another_stream(name):
  """The handle of the stream that is current: copied, then read there."""
  sys = SYSTEMS[name]()
  q, qd, acts = _state(sys)
  start = pipeline.State(q=q, qd=qd, x=None, xd=None)
  want, _ = pipeline.rollout(sys, start, acts, 2)
  side = torch.cuda.Stream(device=DEV)
  torch.cuda.synchronize()
  q2, qd2 = _laid_out(q, "transposed"), _laid_out(qd, "transposed")
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    st, _ = pipeline.rollout(sys, pipeline.State(q=q2, qd=qd2, x=None, xd=None), acts, 2,
                             stream=side.cuda_stream)
  side.synchronize()
  for a, b in ((want.q, st.q), (want.qd, st.qd), (want.x.pos, st.x.pos)):
    assert torch.equal(a, b)
