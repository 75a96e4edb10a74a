"""Workloads of the physics step, and what they return in 64 bits.

Each case is one call (or one forward and backward pass) that programs on
this framework make: single substeps and env steps of a batch, rollouts in one
launch, batches of different robots, gradients, and the frames of a reset.

States follow the environments' resets: the model's pose with uniform noise on
every coordinate, normal velocities, uniform actions.  Two things are kept away
from what 32 bits cannot decide, so that results can be compared at all:
  * batches on the floor take one or two substeps: over more of them the
    solver's line search reaches steps that 32 bits accept or halve by their
    last bits, and a contact then lands on either side;
  * no contact starts within MARGIN of touching, no joint within MARGIN of a
    limit.
Longer rollouts are the flight phase of a jump, under small actions.
"""

import functools
import math

import numpy as np
import torch

from brax_amd import systems
from brax_amd.generalized import hetero, pipeline

MARGIN = 2e-5
MODELS = ("quadruped", "ant", "humanoid")
# dofs, links, contact candidates and limit rows: what work() counts
SIZES = {"quadruped": (14, 9, 17, 8), "ant": (14, 9, 4, 8), "humanoid": (23, 10, 13, 17)}
# constraint rows active on the floor and solver iterations, for work()
ROWS = {"quadruped": 4.3, "ant": 8.1, "humanoid": 15.0}
ITERATIONS = {"quadruped": 4, "ant": 4, "humanoid": 8}
ENV_STEP = 5  # substeps of an env step
CHAIN_SEEDS = 4  # chains of one length in a mixed batch


def listed():
  return [
      # one robot, one substep: a controller in a loop, all latency
      {"name": "substep, one quadruped", "kind": "substep", "model": "quadruped", "n": 1,
       "frames": 1},
      # the training batch the benchmark is quoted on
      {"name": "substep, 65536 quadrupeds", "kind": "substep", "model": "quadruped", "n": 65536,
       "frames": 1},
      # a small training batch that fills no wavefront evenly
      {"name": "two substeps, 3001 quadrupeds", "kind": "substep", "model": "quadruped",
       "n": 3001, "frames": 2},
      # the ant task's batch
      {"name": "substep, 4096 ants", "kind": "substep", "model": "ant", "n": 4096, "frames": 1},
      # the humanoid task on its feet
      {"name": "substep, 1000 humanoids", "kind": "substep", "model": "humanoid", "n": 1000,
       "frames": 1},
      # data collection: a rollout in one launch, with its trajectory
      {"name": "flight, 8192 quadrupeds", "kind": "flight", "model": "quadruped", "n": 8192,
       "steps": 8},
      {"name": "flight, 16384 humanoids", "kind": "flight", "model": "humanoid", "n": 16384,
       "steps": 2},
      # a curriculum of different robots stepped together
      {"name": "mixed batch, 4096 robots", "kind": "mixed", "n": 4096, "steps": 2},
      # analytic policy gradients on the floor, the benchmark's batch
      {"name": "gradient, 4096 quadrupeds", "kind": "gradient", "model": "quadruped", "n": 4096,
       "steps": 2, "frames": 1, "every": 1},
      # and through a jump, over several checkpoint segments
      {"name": "gradient in flight, 1024 quadrupeds", "kind": "gradient", "model": "quadruped",
       "n": 1024, "steps": 16, "frames": ENV_STEP, "every": 8},
      # the frames of a reset batch
      {"name": "reset, 65536 quadrupeds", "kind": "reset", "model": "quadruped", "n": 65536},
  ]


def _log_int(rng, low, high):
  return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
  kind = rng.choice(["substep", "substep", "substep", "flight", "flight", "mixed", "gradient",
                     "gradient", "reset"])
  model = rng.choice(["quadruped", "quadruped", "ant", "humanoid"])
  if kind == "substep":
    frames = rng.choice([1, 1, 2]) if model == "quadruped" else 1
    top = {"quadruped": 65536 if frames == 1 else 8192, "ant": 6000, "humanoid": 1500}[model]
    return {"kind": kind, "model": model, "n": _log_int(rng, 1, top), "frames": frames}
  if kind == "flight":
    top = 16384 if model == "humanoid" else 32768
    return {"kind": kind, "model": model, "n": _log_int(rng, 32, top),
            "steps": rng.randint(1, 2 if model == "humanoid" else 8)}
  if kind == "mixed":
    return {"kind": kind, "n": _log_int(rng, 256, 4096), "steps": rng.randint(1, 2)}
  if kind == "gradient":
    model = "ant" if model == "ant" else "quadruped"
    if rng.random() < 0.5:
      return {"kind": kind, "model": model, "n": _log_int(rng, 64, 4096),
              "steps": rng.randint(1, 2), "frames": 1, "every": rng.randint(1, 2)}
    steps = rng.randint(3, 12)
    return {"kind": kind, "model": model, "n": _log_int(rng, 32, 1024), "steps": steps,
            "frames": ENV_STEP, "every": rng.randint(2, steps)}
  return {"kind": kind, "model": model, "n": _log_int(rng, 64, 65536)}


# ---------------------------------------------------------------------------
# inputs


@functools.lru_cache(maxsize=None)
def _system(model):
  return systems.ant() if model == "ant" else getattr(systems, model)(0)


@functools.lru_cache(maxsize=None)
def _chain(links, seed):
  return systems.chain(links, seed)


def _pose(model):
  """The pose a batch starts around: legs and arms bent, off their limits."""
  s = _system(model)
  q = np.array(s.init_q, np.float64)
  if model == "ant":
    q[7:] = [0.0, 0.9, 0.0, -0.9, 0.0, -0.9, 0.0, 0.9]
    q[2] -= 0.05
  if model == "humanoid":
    lo, hi = np.asarray(s.dof.limit[0])[6:], np.asarray(s.dof.limit[1])[6:]
    room = np.minimum(0.3, 0.5 * (hi - lo))
    q[7:] = np.minimum(np.maximum(0.0, lo + room), hi - room)
  return q


def _device():
  return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _uniform(gen, shape, low, high):
  return low + (high - low) * torch.rand(shape, generator=gen, device=gen.device,
                                         dtype=torch.float64)


def _states(model, n, gen, flight):
  """(q, qd) of a reset batch, float32."""
  s = _system(model)
  ref = _reference(model, str(gen.device))
  pose = torch.tensor(_pose(model), device=gen.device)
  noise = 0.05 if model == "humanoid" else 0.1
  q = None
  for _ in range(20):
    new = pose + _uniform(gen, (n, s.q_size()), -noise, noise)
    if flight:
      new[:, 2] += 5.0 + noise
    elif model == "humanoid":
      new[:, 2] -= 0.05
    new[:, 3:7] /= new[:, 3:7].norm(dim=1, keepdim=True)
    new = new.float()
    q = new if q is None else torch.where(close[:, None], new, q)
    close = ref.clearance(q.double()) < MARGIN
    if not bool(close.any()):
      break
  qd = 0.1 * torch.randn((n, s.qd_size()), generator=gen, device=gen.device)
  return q, qd


def _mixed_systems(n):
  """Half chains of 2 to 32 links, half quadrupeds, in that order."""
  lengths = [2 + i % 31 for i in range(n // 2)]
  seen = {}
  chains = []
  for k in sorted(lengths):
    seen[k] = seen.get(k, -1) + 1
    chains.append((k, seen[k] % CHAIN_SEEDS))
  return chains, n - n // 2


def prepare(case, seed):
  gen = torch.Generator(device=_device())
  gen.manual_seed(int(seed))
  kind, n = case["kind"], case["n"]
  if kind == "mixed":
    chains, quads = _mixed_systems(n)
    batch = hetero.HeteroBatch([_chain(*c) for c in chains] + [_system("quadruped")] * quads)
    dofs = sum(k for k, _ in chains)
    q, qd = _states("quadruped", quads, gen, False)
    acts = _uniform(gen, (case["steps"], dofs + quads * 8), -1.0, 1.0).float()
    return {"case": case, "batch": batch, "acts": acts,
            "q": torch.cat([_uniform(gen, (dofs,), -0.3, 0.3).float(), q.flatten()]),
            "qd": torch.cat([_uniform(gen, (dofs,), -0.3, 0.3).float(), qd.flatten()])}
  s = _system(case["model"])
  flight = kind == "flight" or (kind == "gradient" and case["frames"] > 1)
  q, qd = _states(case["model"], n, gen, flight)
  state = {"case": case, "sys": s, "q": q, "qd": qd}
  if kind == "reset":
    return state
  limit = 0.4 if case["model"] == "humanoid" else 1.0
  if flight:
    limit = 0.1 if case["model"] == "humanoid" else 0.02 if case["steps"] > 8 else 0.05
  steps = () if kind == "substep" else (case["steps"],)
  state["acts"] = _uniform(gen, steps + (n, s.act_size()), -limit, limit).float()
  if kind == "gradient":
    state["qd"].requires_grad_(True)
    state["acts"].requires_grad_(True)
  else:
    state["start"] = pipeline.State(q=q, qd=qd, x=None, xd=None)
  return state


# ---------------------------------------------------------------------------
# one pass


def _frames(st):
  return {"x_pos": st.x.pos, "x_rot": st.x.rot, "xd_ang": st.xd.ang, "xd_vel": st.xd.vel}


def run(state):
  case = state["case"]
  kind = case["kind"]
  if kind == "substep":
    st = pipeline.pipeline_step(state["sys"], state["start"], state["acts"], case["frames"])
    return {"q": st.q, "qd": st.qd, "status": st.status, **_frames(st)}
  if kind == "flight":
    st, (q, qd) = pipeline.rollout(state["sys"], state["start"], state["acts"], ENV_STEP,
                                   trajectory=True)
    return {"q": q, "qd": qd, "status": st.status, **_frames(st)}
  if kind == "mixed":
    q, qd = state["q"].clone(), state["qd"].clone()
    status, q_traj, qd_traj = state["batch"].rollout(q, qd, state["acts"], case["steps"], 1,
                                                     trajectory=True)
    return {"q": q_traj, "qd": qd_traj, "status": status}
  if kind == "gradient":
    q, qd, status = pipeline.rollout_grad(state["sys"], state["q"], state["qd"], state["acts"],
                                          case["frames"], ckpt_every=case["every"])
    loss = _loss(qd, state["acts"])
    g_act, g_qd = torch.autograd.grad(loss, (state["acts"], state["qd"]))
    return {"q": q.detach(), "qd": qd.detach(), "status": status, "g_act": g_act, "g_qd": g_qd}
  st = pipeline.init(state["sys"], state["q"], state["qd"])
  return {"q": st.q, "qd": st.qd, **_frames(st)}


def _loss(qd, acts):
  """Forward speed against effort, as a locomotion task pays it."""
  return -qd[:, :, 0].sum() + 1e-3 * (acts * acts).sum()


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _substep_flops(dofs, links, contacts, limits, rows, iterations):
  """One substep of one robot: kinematics, bias and COM terms per link, the
  mass matrix and its factor, contact geometry, and per solver iteration two
  products with the active rows (a multiply-add is two)."""
  tree = 720 * links + 190 * dofs
  mass = 5.5 * dofs * (dofs + 1) + 36 * dofs + dofs ** 3 / 3 + 4 * dofs ** 2
  contact = contacts * 60 + limits * 10
  solve = rows * dofs ** 2 + iterations * 20 * rows * (dofs + 1)
  return tree + mass + contact + solve


def work(case):
  kind, n = case["kind"], case["n"]
  if kind == "mixed":
    chains, quads = _mixed_systems(n)
    one = _substep_flops(*SIZES["quadruped"], ROWS["quadruped"], ITERATIONS["quadruped"])
    flops = quads * one + sum(_substep_flops(k, k, 0, 0, 0, 0) for k, _ in chains)
    dofs = sum(k for k, _ in chains)
    floats = 2 * dofs + quads * 29 + case["steps"] * (3 * dofs + quads * 37) + n
    return {"bytes": 4 * floats, "flops": case["steps"] * flops}
  dofs, links, contacts, limits = SIZES[case["model"]]
  acts = 17 if case["model"] == "humanoid" else 8
  state = 2 * dofs + 1
  frames = 13 * links
  if kind == "reset":
    return {"bytes": 4 * n * (2 * state + frames), "flops": n * links * 150}
  flight = kind == "flight" or (kind == "gradient" and case["frames"] > 1)
  rows = 0 if flight else ROWS[case["model"]]
  one = _substep_flops(dofs, links, 0 if flight else contacts, 0 if flight else limits, rows,
                       ITERATIONS[case["model"]])
  if kind == "substep":
    return {"bytes": 4 * n * (2 * state + acts + frames + 1), "flops": n * case["frames"] * one}
  if kind == "flight":
    return {"bytes": 4 * n * (state + frames + 1 + case["steps"] * (state + acts)),
            "flops": n * case["steps"] * ENV_STEP * (one + links * 30)}
  # a gradient costs about three times the function, after the function itself
  return {"bytes": 4 * n * (state + dofs + 1 + case["steps"] * (2 * state + 2 * acts)),
          "flops": 4 * n * case["steps"] * case["frames"] * one}


# ---------------------------------------------------------------------------
# the same in 64 bits: dense matrices over world-frame motion vectors


def _qmul(a, b):
  w, v = a[..., :1], a[..., 1:]
  x, u = b[..., :1], b[..., 1:]
  return torch.cat([w * x - (v * u).sum(-1, keepdim=True), w * u + x * v + _cross(v, u)], -1)


def _cross(a, b):
  a, b = torch.broadcast_tensors(a, b)
  return torch.linalg.cross(a, b)


def _mat(q):
  """Rotation matrix of a quaternion, times its length squared."""
  w, x, y, z = q.unbind(-1)
  return torch.stack([
      w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y),
      2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x),
      2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z], -1).reshape(
          q.shape[:-1] + (3, 3))


def _apply(m, v):
  return (m @ v[..., None])[..., 0]


def _unit(v):
  return v / v.norm(dim=-1, keepdim=True)


def _turn(axis, angle):
  """The quaternion of a turn about a unit axis."""
  half = 0.5 * angle[..., None]
  return torch.cat([torch.cos(half), torch.sin(half) * axis], -1)


def _motion_cross(a, b):
  """a x b of motions (angular, linear at the world's origin)."""
  w, v = a[..., :3], a[..., 3:]
  return torch.cat([_cross(w, b[..., :3]), _cross(v, b[..., :3]) + _cross(w, b[..., 3:])], -1)


def _force_cross(a, f):
  """a x* f of a motion and a force (moment about the origin, force)."""
  w, v = a[..., :3], a[..., 3:]
  return torch.cat([_cross(w, f[..., :3]) + _cross(v, f[..., 3:]), _cross(w, f[..., 3:])], -1)


class _Reference:
  """The step of one System, or of several of one structure, one each env."""

  def __init__(self, many, device):
    s = self.s = many[0]
    f = lambda get: torch.tensor(np.stack([np.asarray(get(x), np.float64) for x in many]),  # noqa: E731
                                 device=device)
    self.links, self.dofs = len(s.link_types), s.qd_size()
    self.tpos, self.trot = f(lambda x: x.link.transform.pos), f(lambda x: x.link.transform.rot)
    self.jpos = f(lambda x: x.link.joint.pos)
    self.ipos = f(lambda x: x.link.inertia.transform.pos)
    self.irot = f(lambda x: x.link.inertia.transform.rot)
    self.inertia, self.mass = f(lambda x: x.link.inertia.i), f(lambda x: x.link.inertia.mass)
    self.axis = f(lambda x: x.dof.motion.ang)
    self.armature, self.stiffness = f(lambda x: x.dof.armature), f(lambda x: x.dof.stiffness)
    self.damping = f(lambda x: x.dof.damping)
    self.gravity = f(lambda x: x.gravity)
    a = s.actuator
    self.act_q, self.act_d = [torch.tensor(np.asarray(i), device=device) for i in (a.q_id, a.qd_id)]
    self.ctrl, self.force = f(lambda x: x.actuator.ctrl_range), f(lambda x: x.actuator.force_range)
    self.gain, self.gear = f(lambda x: x.actuator.gain), f(lambda x: x.actuator.gear)
    self.bias_q, self.bias_qd = f(lambda x: x.actuator.bias_q), f(lambda x: x.actuator.bias_qd)
    self.dt = float(s.opt.timestep)
    # joint coordinates: q and dof index of every hinge, first ones per link
    self.q_at, self.d_at, nq, nd = [], [], 0, 0
    self.hinge_q, self.hinge_d = [], []
    for t in s.link_types:
      self.q_at.append(nq)
      self.d_at.append(nd)
      if t != "f":
        self.hinge_q += range(nq, nq + int(t))
        self.hinge_d += range(nd, nd + int(t))
      nq, nd = nq + (7 if t == "f" else int(t)), nd + (6 if t == "f" else int(t))
    # ancestors[l, d]: dof d moves link l
    anc = np.zeros((self.links, self.dofs))
    for l, (t, p) in enumerate(zip(s.link_types, s.link_parents)):
      if p >= 0:
        anc[l] = anc[p]
      anc[l, self.d_at[l]:self.d_at[l] + (6 if t == "f" else int(t))] = 1
    self.ancestors = torch.tensor(anc, device=device)
    self.device = device
    limit = s.dof.limit
    if limit is not None:
      row = lambda x: torch.tensor(np.asarray(x, np.float64), device=device)  # noqa: E731
      d = self.hinge_d
      self.lo, self.hi = row(limit[0])[d], row(limit[1])[d]
      self.lim_weight = row(s.dof.invweight)[d]
      self.lim_solver = row(s.dof.solver_params)[d]
    self.limited = limit is not None
    self.points = []  # (pair, end of the capsule)
    for p in s.contact_pairs():
      self.points += [(p, e) for e in ((0.0,) if int(s.geom_type[p.geom2]) == 2 else (1.0, -1.0))]

  def tree(self, q):
    """World quaternions and positions of the links, motions of the dofs."""
    s, n = self.s, q.shape[0]
    rot, pos, motion = [], [], []
    wide = lambda x: x.expand(n, *x.shape[1:])  # noqa: E731
    for l, (t, p) in enumerate(zip(s.link_types, s.link_parents)):
      x = q[:, self.q_at[l]:]
      if t == "f":  # its quaternion as it is: a length off 1 scales what hangs on it
        r, at = x[:, 3:7], x[:, :3]
      else:
        r, at = wide(self.trot[:, l]), wide(self.tpos[:, l])
        if p >= 0:
          r, at = _qmul(rot[p], r), pos[p] + _apply(_mat(rot[p]), at)
        at = at + _apply(_mat(r), wide(self.jpos[:, l]))
        for k in range(int(t)):
          r = _qmul(r, _turn(wide(self.axis[:, self.d_at[l] + k]), x[:, k]))
        at = at - _apply(_mat(r), wide(self.jpos[:, l]))
      rot.append(r)
      pos.append(at)
    rot = [_unit(r) for r in rot]
    zero = torch.zeros(n, 3, dtype=q.dtype, device=q.device)
    unit = torch.eye(3, dtype=q.dtype, device=q.device)
    for l, (t, p) in enumerate(zip(s.link_types, s.link_parents)):
      if t == "f":
        m, at = _mat(rot[l]), pos[l]
        motion += [torch.cat([zero, unit[k].expand(n, 3)], -1) for k in range(3)]
        motion += [torch.cat([m[:, :, k], _cross(at, m[:, :, k])], -1) for k in range(3)]
        continue
      r, at = wide(self.trot[:, l]), wide(self.tpos[:, l])
      if p >= 0:
        r, at = _qmul(rot[p], r), pos[p] + _apply(_mat(rot[p]), at)
      at = at + _apply(_mat(r), wide(self.jpos[:, l]))
      for k in range(int(t)):
        axis = wide(self.axis[:, self.d_at[l] + k])
        a = _apply(_mat(r), axis)
        motion.append(torch.cat([a, _cross(at, a)], -1))
        r = _qmul(r, _turn(axis, q[:, self.q_at[l] + k]))
    return torch.stack(rot, 1), torch.stack(pos, 1), torch.stack(motion, 1)

  def frames(self, q, qd):
    """The links' world frames and their velocities, a link's own turn left
    out of its linear velocity."""
    s = self.s
    rot, pos, _ = self.tree(q)
    ang, vel = [], []
    for l, (t, p) in enumerate(zip(s.link_types, s.link_parents)):
      w = qd[:, self.d_at[l]:]
      if t == "f":
        ang.append(_apply(_mat(rot[:, l]), w[:, 3:6]))
        vel.append(w[:, :3])
        continue
      own = sum(self.axis[:, self.d_at[l] + k] * w[:, k:k + 1] for k in range(int(t)))
      a = _apply(_mat(rot[:, l]), own)
      ang.append(a if p < 0 else ang[p] + a)
      vel.append(torch.zeros_like(a) if p < 0 else
                 vel[p] + _cross(ang[p], pos[:, l] - pos[:, p]))
    return {"x_pos": pos, "x_rot": rot, "xd_ang": torch.stack(ang, 1),
            "xd_vel": torch.stack(vel, 1)}

  def contacts(self, rot, pos):
    """Distance, point and frame of every contact candidate with the floor
    (the plane z = 0, normal up)."""
    s, dist, point, tangent = self.s, [], [], []
    up = torch.tensor([0.0, 0.0, 1.0], dtype=pos.dtype, device=pos.device)
    side = torch.tensor([0.0, 1.0, 0.0], dtype=pos.dtype, device=pos.device)
    for p, end in self.points:
      l, g = int(s.geom_bodyid[p.geom2]) - 1, p.geom2
      at = lambda x: torch.tensor(np.asarray(x, np.float64), device=pos.device)  # noqa: E731
      c = pos[:, l] + _apply(_mat(rot[:, l]), at(s.geom_pos[g]).expand(pos.shape[0], 3))
      t = side.expand_as(c)
      if end:
        axis = _mat(_qmul(rot[:, l], at(s.geom_quat[g]).expand(pos.shape[0], 4)))[:, :, 2]
        c = c + axis * (end * float(s.geom_size[g][1]))
        flat = axis * torch.tensor([1.0, 1.0, 0.0], dtype=pos.dtype, device=pos.device)
        length = (flat * flat).sum(-1, keepdim=True)
        lies = length >= 0.25
        t = torch.where(lies, flat / torch.where(lies, length, 1.0).sqrt(), t)
      radius = float(s.geom_size[g][0])
      d = c[:, 2] - radius
      dist.append(d)
      point.append(c - up * (radius + 0.5 * d)[:, None])
      tangent.append(t)
    return torch.stack(dist, 1), torch.stack(point, 1), torch.stack(tangent, 1), up

  def clearance(self, q):
    """How near each state's nearest contact or limit is to becoming active."""
    rot, pos, _ = self.tree(q)
    near = torch.full((q.shape[0],), math.inf, dtype=q.dtype, device=q.device)
    if self.points:
      near = self.contacts(rot, pos)[0].abs().amin(1)
    if self.limited:
      x = q[:, self.hinge_q]
      near = torch.minimum(near, torch.minimum((x - self.lo).abs(), (self.hi - x).abs()).amin(1))
    return near

  @staticmethod
  def _impedance(solver, x):
    """Impedance, damping and stiffness of a constraint violated by x."""
    tc, ratio, low, high, width, mid, power = solver.unbind(-1)
    y = x.abs() / width
    below = y.clamp(max=1.0) ** power / mid ** (power - 1)
    above = 1 - (1 - y).clamp(min=0.0) ** power / (1 - mid) ** (power - 1)
    imp = low + torch.where(y < mid, below, above) * (high - low)
    imp = torch.where(y > 1, high, torch.minimum(torch.maximum(imp, low), high))
    return imp, 2 / (high * tc), 1 / (high * tc * ratio) ** 2

  def rows(self, q, qd, rot, pos, motion):
    """Constraint rows: Jacobian, diagonal, reference acceleration; zero where
    the constraint is not active."""
    s, jac, diag, ref = self.s, [], [], []
    if self.points:
      dist, point, t1, up = self.contacts(rot, pos)
      link = [int(s.geom_bodyid[p.geom2]) - 1 for p, _ in self.points]
      solver = torch.tensor(np.stack([np.concatenate([p.solref, p.solimp])
                                      for p, _ in self.points]), device=q.device)
      mu = torch.tensor([float(p.friction[0]) for p, _ in self.points], device=q.device,
                        dtype=q.dtype)
      weight = torch.tensor(np.asarray(s.link.invweight, np.float64)[link], device=q.device)
      on = dist < 0
      depth = torch.where(on, dist, 0.0)
      imp, b, k = self._impedance(solver, depth)
      t2 = _cross(up.expand_as(t1), t1)
      # velocity of the contact point by dof, on the dofs that move its link
      moved = (motion[:, None, :, 3:] + _cross(motion[:, None, :, :3], point[:, :, None]))
      moved = moved * self.ancestors[link][None, :, :, None]
      for way in (t1, -t1, t2, -t2):
        j = (moved * (up + mu[:, None] * way)[:, :, None]).sum(-1) * on[..., None]
        jac.append(j)
        diag.append(on * (weight * (1 + mu * mu) * 2 * mu * mu * (1 - imp) / (imp + 1e-8)))
        ref.append(-b * (j @ qd[..., None])[..., 0] - on * (k * imp * depth))
    if self.limited:
      x = q[:, self.hinge_q]
      low, high = x - self.lo, self.hi - x
      gap = torch.minimum(torch.minimum(low, high), torch.zeros_like(x))
      on = gap < 0
      imp, b, k = self._impedance(self.lim_solver, gap)
      sign = torch.where(low < high, 1.0, -1.0) * on
      j = torch.zeros(q.shape[0], len(self.hinge_d), self.dofs, dtype=q.dtype, device=q.device)
      j[:, range(len(self.hinge_d)), self.hinge_d] = sign.to(q.dtype)
      jac.append(j)
      diag.append(on * self.lim_weight * (1 - imp) / (imp + 1e-8))
      ref.append(-b * sign * qd[:, self.hinge_d] - on * (k * imp * gap))
    return torch.cat(jac, 1), torch.cat(diag, 1), torch.cat(ref, 1)

  def solve(self, a, b):
    """Accelerated projected gradient with a backtracking line search on
    |a x + b|^2 / 2 over x >= 0, from zero, a fixed number of iterations."""
    times = lambda v: (a @ v[..., None])[..., 0]  # noqa: E731
    x = y = torch.zeros_like(b)
    one = torch.ones(b.shape[0], dtype=b.dtype, device=b.device)
    eta, t, err = one, one, one * math.inf
    slack, tol = float(np.finfo(np.float32).eps), 1e-3
    alive = (b != 0).any(1)
    for _ in range(int(self.s.solver_iterations)):
      alive = alive & (err > tol)
      if not bool(alive.any()):
        break
      r = times(y) + b
      g = times(r)
      fy = 0.5 * (r * r).sum(1)
      step, go = eta, alive
      for k in range(int(self.s.solver_maxls) + 1):
        if k:
          step = torch.where(go, 0.5 * step, step)
        new = (y - step[:, None] * g).clamp(min=0.0)
        rx, d = times(new) + b, new - y
        fx = 0.5 * (rx * rx).sum(1)
        go = go & (step * (fx - fy) > step * (d * g).sum(1) + 0.5 * (d * d).sum(1) + slack)
        if not bool(go.any()):
          break
      away = ((new - times(rx)).clamp(min=0.0) - new).detach().norm(dim=1)
      t_new = 0.5 * (1 + (1 + 4 * t * t).sqrt())
      y_new = new + ((t - 1) / t_new)[:, None] * (new - x)
      on = alive[:, None]
      x, y = torch.where(on, new, x), torch.where(on, y_new, y)
      eta = torch.where(alive, torch.where(step <= 1e-6, 1.0, 2 * step), eta)
      t, err = torch.where(alive, t_new, t), torch.where(alive, away, err)
    return x

  def step(self, q, qd, act):
    """One substep."""
    n = q.shape[0]
    rot, pos, motion = self.tree(q)
    # spatial inertia of each link about the world's origin
    m = _mat(rot)
    com = pos + _apply(m, self.ipos.expand(n, -1, 3))
    r = m @ _mat(self.irot)
    c = torch.zeros(n, self.links, 3, 3, dtype=q.dtype, device=q.device)
    c[..., 0, 1], c[..., 0, 2], c[..., 1, 2] = -com[..., 2], com[..., 1], -com[..., 0]
    c = c - c.transpose(-1, -2)
    mc = self.mass[..., None, None] * c
    eye = self.mass[..., None, None] * torch.eye(3, dtype=q.dtype, device=q.device)
    inertia = torch.cat([
        torch.cat([r @ self.inertia @ r.transpose(-1, -2) - mc @ c, mc], -1),
        torch.cat([-mc, eye.expand_as(mc)], -1)], -2)
    jac = self.ancestors[None, :, :, None] * motion[:, None]  # (n, links, dofs, 6)
    heavy = jac @ inertia  # inertias are symmetric
    mass = torch.einsum("nlax,nlbx->nab", heavy, jac) + torch.diag_embed(self.armature)
    # velocities, and the accelerations that they alone cause
    speed = motion * qd[..., None]
    before = []
    for l, (t, p) in enumerate(zip(self.s.link_types, self.s.link_parents)):
      d = self.d_at[l]
      v = torch.zeros_like(speed[:, 0]) if p < 0 else self.ancestors[p] @ speed
      for k in range(6 if t == "f" else int(t)):
        if t == "f":  # translations keep their directions
          before.append(speed[:, d:d + 3].sum(1) if k >= 3 else torch.zeros_like(v))
        else:
          before.append(v + speed[:, d:d + k].sum(1))
    turned = _motion_cross(torch.stack(before, 1), motion) * qd[..., None]
    v = torch.einsum("ld,ndx->nlx", self.ancestors, speed)
    acc = torch.einsum("ld,ndx->nlx", self.ancestors, turned)
    acc = acc - torch.cat([torch.zeros_like(self.gravity), self.gravity], -1)[:, None]
    f = _apply(inertia, acc) + _force_cross(v, _apply(inertia, v))
    force = -torch.einsum("nldx,nlx->nd", jac, f) - self.damping * qd
    spring = torch.zeros_like(qd)
    spring[:, self.hinge_d] = self.stiffness[:, self.hinge_d] * q[:, self.hinge_q]
    force = force - spring
    if len(self.act_q):
      u = torch.minimum(torch.maximum(act, self.ctrl[..., 0]), self.ctrl[..., 1])
      u = self.gain * u + self.gear * (q[:, self.act_q] * self.bias_q +
                                       qd[:, self.act_d] * self.bias_qd)
      u = torch.minimum(torch.maximum(u, self.force[..., 0]), self.force[..., 1]) * self.gear
      force = force.index_add(1, self.act_d, u)
    chol = torch.linalg.cholesky(mass)
    free = torch.cholesky_solve(force[..., None], chol)
    qdd = free[..., 0]
    if self.points or self.limited:
      j, diag, ref = self.rows(q, qd, rot, pos, motion)
      back = torch.cholesky_solve(j.transpose(-1, -2), chol)
      x = self.solve(j @ back + torch.diag_embed(diag), (j @ free)[..., 0] - ref)
      qdd = qdd + (back @ x[..., None])[..., 0]
    qd = qd + self.dt * qdd
    parts = []
    for l, t in enumerate(self.s.link_types):
      i, d = self.q_at[l], self.d_at[l]
      if t != "f":
        parts.append(q[:, i:i + int(t)] + self.dt * qd[:, d:d + int(t)])
        continue
      w = qd[:, d + 3:d + 6]
      rate = (w * w).sum(-1).clamp(min=1e-30).sqrt() + 1e-8
      turn = _turn(w / rate[:, None], self.dt * rate)
      parts += [q[:, i:i + 3] + self.dt * qd[:, d:d + 3], _unit(_qmul(q[:, i + 3:i + 7], turn))]
    return torch.cat(parts, 1), qd

  def roll(self, q, qd, acts, frames):
    """States after every step of `frames` substeps."""
    qs, qds = [], []
    for act in acts:
      for _ in range(frames):
        q, qd = self.step(q, qd, act)
      qs.append(q)
      qds.append(qd)
    return torch.stack(qs), torch.stack(qds)


@functools.lru_cache(maxsize=None)
def _reference(model, device):
  return _Reference([_system(model)], device)


def _by_part(n, size, fn):
  """fn(slice) over parts of a batch, joined: the dense rows fill memory."""
  parts = [fn(slice(i, min(i + size, n))) for i in range(0, n, size)]
  return {k: torch.cat([p[k] for p in parts], 0 if parts[0][k].dim() < 3 or k[0] == "x" else 1)
          for k in parts[0]}


def exact(case, seed):
  state = prepare(case, seed)
  kind, n = case["kind"], case["n"]
  if kind == "mixed":
    return _exact_mixed(case, state)
  ref = _reference(case["model"], str(state["q"].device))
  q, qd = state["q"].detach().double(), state["qd"].detach().double()
  if kind == "reset":
    return {"q": q, "qd": qd, **ref.frames(q, qd)}
  acts = state["acts"].detach().double()
  if kind == "substep":
    def part(i):
      a, b = ref.roll(q[i], qd[i], [acts[i]], case["frames"])
      return {"q": a[0], "qd": b[0], **ref.frames(a[0], b[0])}
    return {**_by_part(n, 8192, part), "status": None}
  if kind == "flight":
    def part(i):
      a, b = ref.roll(q[i], qd[i], acts[:, i], ENV_STEP)
      return {"q": a, "qd": b, **ref.frames(a[-1], b[-1])}
    return {**_by_part(n, 4096, part), "status": None}

  def part(i):
    act, speed = acts[:, i].clone().requires_grad_(True), qd[i].clone().requires_grad_(True)
    a, b = ref.roll(q[i], speed, act, case["frames"])
    g_act, g_qd = torch.autograd.grad(_loss(b, act), (act, speed))
    return {"q": a.detach(), "qd": b.detach(), "g_act": g_act, "g_qd": g_qd}
  return {**_by_part(n, 1024, part), "status": None}


def _exact_mixed(case, state):
  chains, quads = _mixed_systems(case["n"])
  qs, qds = [], []
  at = act_at = 0  # a chain has a coordinate, a dof and a motor each link
  groups = {}
  for k, seed in chains:
    groups.setdefault(k, []).append(seed)
  device = str(state["q"].device)
  parts = [(_Reference([_chain(k, x) for x in v], device), len(v), k, k, k)
           for k, v in groups.items()]
  parts.append((_reference("quadruped", device), quads, 15, 14, 8))
  dat = 0
  for ref, n, nq, nv, nu in parts:
    q = state["q"][at:at + n * nq].double().reshape(n, nq)
    qd = state["qd"][dat:dat + n * nv].double().reshape(n, nv)
    acts = state["acts"][:, act_at:act_at + n * nu].double().reshape(-1, n, nu)
    a, b = ref.roll(q, qd, acts, 1)
    qs.append(a.flatten(1))
    qds.append(b.flatten(1))
    at, dat, act_at = at + n * nq, dat + n * nv, act_at + n * nu
  return {"q": torch.cat(qs, 1), "qd": torch.cat(qds, 1), "status": None}
