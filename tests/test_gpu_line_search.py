"""Line-search decisions of the contact solver where a trial step ties.

The search accepts a trial where f(x+) - f(y) <= g.d + |d|^2 / (2 eta); at a
tie, 32 bits decide, and the other decision moves a robot's velocities by
0.01 to 0.3.  Every kernel of a topology is to decide as the one whose steps
the adjoint tapes.

tests/golden/humanoid_ties.npz: ten humanoids on the floor with such a tie
that the test on f decides as 64 bits do, and the same test written as
|A d|^2 against |d|^2 / eta does not."""

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
