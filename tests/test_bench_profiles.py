"""The bench line quotes HBM traffic only from a committed profile of the
kernel that runs, and names a profile only where it quotes one."""

import os

import pytest

import bench


@pytest.mark.parametrize("key", sorted(bench.PROFILED, key=str))
def test_every_named_profile_is_committed(key):
  name, _ = key
  n = bench.WORKLOADS[name][1]
  path = os.path.join(bench.ROOT, bench.profile_path(bench.PROFILED[key], name, n))
  steps = [int(line.split("env_steps=")[1].split()[0]) for line in open(path)
           if line.startswith("traffic_per_launch:")]
  for k in steps:
    t = bench.roofline_traffic(*key, n, k)
    assert t["traffic"] > 0 and os.path.basename(path) in t["traffic_source"]
  # the workload's own length among them
  if key != ("humanoid", 1):
    assert bench.DEFAULT_STEPS[name] in steps


@pytest.mark.parametrize("args", [("quadruped", 4, 65536, 7), ("quadruped", 4, 1024, 1000),
                                  ("quadruped", 1, 65536, 1000), ("hetero", None, 4096, 500)])
def test_no_profile_no_source(args):
  assert bench.roofline_traffic(*args) == {"traffic": None, "traffic_source": None}
