"""One substep of ants on the floor, the lane-per-leg kernel whose contact rows
live in registers, against the float64 oracle and the one-thread kernel, at
batch sizes around a wavefront's 16 envs.

Tolerance: the parity band |gpu - ref| <= 1e-5 + 1e-4 |ref|, but for robots
where the float32 oracle leaves it too (a line-search step that rounding
decides), at most one in eight."""

import numpy as np
import pytest
import torch

from brax_amd import systems as S
from brax_amd.generalized import autotune, pipeline
from oracle.generalized import Oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _t(x):
  return torch.tensor(np.asarray(x, np.float32), device=DEV)


def _ratio(a, ref):
  a, ref = np.asarray(a, np.float64), np.asarray(ref, np.float64)
  return (np.abs(a - ref) / (1e-5 + 1e-4 * np.abs(ref))).max(1)


@pytest.mark.parametrize("n", [1, 17, 65])
def test_ant_floor_substep(n):
  """Feet in the floor on one to four legs, hips and ankles past their limits
  on some."""
  sys = S.ant()
  rng = np.random.default_rng(n)
  q = np.array(sys.init_q) + rng.uniform(-0.1, 0.1, (n, 15))
  q[:, 7:] = np.array([0.0, 0.9, 0.0, -0.9, 0.0, -0.9, 0.0, 0.9]) + rng.uniform(
      -0.65, 0.65, (n, 8))
  q[:, 2] = rng.uniform(0.35, 0.6, n)
  q[:, 3:7] /= np.linalg.norm(q[:, 3:7], axis=1, keepdims=True)
  q = q.astype(np.float32)
  qd = (0.1 * rng.standard_normal((n, 14))).astype(np.float32)
  act = rng.uniform(-1, 1, (n, 8)).astype(np.float32)
  st = pipeline.State(q=_t(q), qd=_t(qd), x=None, xd=None)
  pr = pipeline.probe(sys, st, _t(act), 1)
  new = pipeline.pipeline_step(sys, st, _t(act), 1)
  m = pipeline.device_model(sys, DEV)
  autotune.set_launch(m, autotune.LANES, 1)
  try:
    one = pipeline.probe(sys, st, _t(act), 1)
  finally:
    autotune.set_launch(m, autotune.LANES, 0)
  np.testing.assert_array_equal(pr["n_contacts"].cpu().numpy(), one["n_contacts"].cpu().numpy())
  lo, hi = (np.asarray(x)[6:] for x in sys.dof.limit)
  limits = (q[:, 7:] < lo) | (q[:, 7:] > hi)
  if n > 1:
    assert pr["n_contacts"].max() >= 2 and limits.any() and not limits.all()

  def oracle(dtype):
    o = Oracle(sys, dtype, inverse="exact")
    s = o.step(o.init(torch.tensor(q, dtype=dtype), torch.tensor(qd, dtype=dtype)),
               torch.tensor(act, dtype=dtype))
    return s.q.double().numpy(), s.qd.double().numpy()
  q64, qd64 = oracle(torch.float64)
  q32, qd32 = oracle(torch.float32)
  ok = np.maximum(_ratio(q32, q64), _ratio(qd32, qd64)) <= 1.0
  r = np.maximum(_ratio(new.q.cpu(), q64), _ratio(new.qd.cpu(), qd64))
  print(f"\nants {n}: {int(limits.any(1).sum())} at limits, contacts "
        f"{float(pr['n_contacts'].mean()):.1f}, worst ratio {r[ok].max():.3f}, float32 oracle "
        f"outside the band {int((~ok).sum())}", flush=True)
  assert (~ok).sum() <= n // 8
  assert r[ok].max() <= 1.0
