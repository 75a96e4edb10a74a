"""Line-search decisions of the contact solver where a trial step ties.

The search accepts a trial where f(x+) - f(y) <= g.d + |d|^2 / (2 eta); at a
tie, 32 bits decide, and the other decision moves a robot's velocities by
0.01 to 0.3.  Every kernel of a topology is to decide as the one whose steps
the adjoint tapes.

tests/golden/humanoid_ties.npz: ten humanoids on the floor with such a tie
that the test on f decides as 64 bits do, and the same test written as
|A d|^2 against |d|^2 / eta does not.
tests/golden/ant_ties.npz: ten ants for which the two tests part the other
way, so that states by one and a tape by the other give a gradient that is off
by 0.2 to 13%."""

import os

import numpy as np
import torch
import pytest

from brax_amd import systems as S
from brax_amd.generalized import autotune, pipeline
from oracle.generalized import Oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
# between what rounding moves (4e-4 at most) and what a decision moves (1e-2)
TIE_ATOL = 1e-3
# between what rounding makes of these gradients (1e-6) and a decision (2e-3)
GRAD_TIE_RTOL = 3e-4


def _t(x):
  return torch.tensor(np.asarray(x, np.float32), device=DEV)


def test_humanoid_ties_are_decided_as_in_64_bits():
  """One substep of the ten: velocities as the float64 oracle's, and as many
  solver iterations and trials as one thread per env takes."""
  sys = S.humanoid(0)
  g = np.load(os.path.join(GOLDEN, "humanoid_ties.npz"))
  m = pipeline.device_model(sys, DEV)
  st = pipeline.State(q=_t(g["q"]), qd=_t(g["qd"]), x=None, xd=None)
  probes = []
  for lanes in (0, 1):
    autotune.set_launch(m, autotune.LANES, lanes)
    try:
      probes.append(pipeline.probe(sys, st, _t(g["act"]), 1))
      new = pipeline.pipeline_step(sys, st, _t(g["act"]), 1)
    finally:
      autotune.set_launch(m, autotune.LANES, 0)
    o = Oracle(sys, torch.float64, inverse="exact")
    ref = o.step(o.init(g["q"].astype(np.float64), g["qd"].astype(np.float64)),
                 g["act"].astype(np.float64))
    off = np.abs(new.qd.double().cpu().numpy() - ref.qd.numpy()).max(1)
    print(f"\nlanes {lanes}: qd off 64 bits by {np.array2string(off, precision=1)}", flush=True)
    assert off.max() <= TIE_ATOL
  for key in ("iters", "trials"):
    np.testing.assert_array_equal(probes[0][key].cpu().numpy(), probes[1][key].cpu().numpy())


def _loss(qd, act):
  return -qd[:, 0].sum() + 1e-3 * (act * act).sum()


@pytest.mark.parametrize("call", ["rollout_grad", "pipeline_step"])
def test_ant_gradient_takes_the_steps_of_its_states(call):
  """One substep of the ten ants: velocities, and the gradient to actions and
  velocities, as the float64 oracle's autograd gives them."""
  sys = S.ant()
  g = np.load(os.path.join(GOLDEN, "ant_ties.npz"))
  q, qd, act = _t(g["q"]), _t(g["qd"]).requires_grad_(True), _t(g["act"]).requires_grad_(True)
  if call == "rollout_grad":
    _, qdt, _ = pipeline.rollout_grad(sys, q, qd, act[None], 1, 1)
    new = qdt[0]
  else:
    new = pipeline.pipeline_step(sys, pipeline.State(q=q, qd=qd, x=None, xd=None), act, 1).qd
  got = torch.cat(torch.autograd.grad(_loss(new, act), (qd, act)), 1).double().cpu().numpy()
  o = Oracle(sys, torch.float64, inverse="exact")
  qd64 = torch.tensor(g["qd"], dtype=torch.float64, requires_grad=True)
  act64 = torch.tensor(g["act"], dtype=torch.float64, requires_grad=True)
  ref = o.step(o.init(torch.tensor(g["q"], dtype=torch.float64), qd64), act64)
  want = torch.cat(torch.autograd.grad(_loss(ref.qd, act64), (qd64, act64)), 1).numpy()
  off = np.abs(new.detach().double().cpu().numpy() - ref.qd.detach().numpy()).max()
  rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
  print(f"\n{call}: qd off by {off:.1e}, gradient by {np.array2string(rel, precision=1)}",
        flush=True)
  assert off <= TIE_ATOL
  assert rel.max() <= GRAD_TIE_RTOL


@pytest.mark.parametrize("name", ["quadruped", "ant"])
@pytest.mark.parametrize("n", [1, 17, 65])
def test_backward_pass_repeats_the_states_of_rollout_grad(name, n):
  """The states of bgx_rollout_primal are those of one thread per env, which
  the tape is written by: over 4 env steps on the floor, bit for bit, from a
  state that is left as it was."""
  sys = S.quadruped(0) if name == "quadruped" else S.ant()
  rng = np.random.default_rng(n)
  q = sys.init_q + rng.uniform(-0.1, 0.1, (n, 15))
  q[:, 2] -= 0.1
  q, qd = _t(q), _t(0.1 * rng.standard_normal((n, 14)))
  acts = _t(rng.uniform(-1, 1, (4, n, 8)))
  kept = q.clone(), qd.clone()
  qt, qdt, _ = pipeline.rollout_grad(sys, q, qd, acts, 5, 2)
  m = pipeline.device_model(sys, DEV)
  autotune.set_launch(m, autotune.LANES, 1)
  try:
    _, (q1, qd1) = pipeline.rollout(sys, pipeline.State(q=q, qd=qd, x=None, xd=None), acts, 5,
                                    trajectory=True)
  finally:
    autotune.set_launch(m, autotune.LANES, 0)
  assert torch.equal(qt, q1) and torch.equal(qdt, qd1)
  assert torch.equal(q, kept[0]) and torch.equal(qd, kept[1])
