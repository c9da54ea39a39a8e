"""bench.py times the searches that a user runs: never one with the per-kernel
accounting on, which has the host drive the single-root search's levels."""
import argparse
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

PLAIN_MS, ACCOUNTED_MS, NEDGE = 2.0, 1000.0, 4_000_000
STATS = {"ms": 1.0, "launches": 2, "bytes": 3e6, "edges": 4}


class Engine:
    """What bench.py uses of the engines, with times that tell how they ran."""

    def __init__(self, graph):
        self.accounted = False
        self.seen = 0

    def run(self, root, codec=False):
        self.seen += self.accounted
        return 7, ACCOUNTED_MS if self.accounted else PLAIN_MS

    def profile(self, enable=True):
        self.accounted = enable

    def kernel_stats(self):
        assert self.accounted and self.seen == 64
        return {"k_expand": dict(STATS), "k_bottom_up": dict(STATS, ms=5.0)}

    def stats(self):
        return {"k_pull_wave": dict(STATS)}

    def nedge(self):
        return NEDGE

    def times(self):
        return PLAIN_MS, 0.5

    def bins(self):
        return [1, 2, 3]

    def maps(self):
        return None, None, None, True

    def free(self):
        pass


class Batched(Engine):
    def nedge(self):
        return np.full(64, NEDGE)


class Graph:
    nglobal, n_rows, nnz = 1 << 16, 1 << 16, 1 << 20

    @classmethod
    def kronecker(cls, scale):
        return cls()

    def select_roots(self, vertices, n=64):
        return np.arange(n)

    def free(self):
        pass


class Library:
    Graph, BFS, MSBFS = Graph, Engine, Batched

    @staticmethod
    def lib():
        return argparse.Namespace(g5_device_sync=lambda: 0)


ARGS = dict(scale=16, roots=64, steps=2, warmup=1, validate="off", autotune="off", place=0, levels=False,
            cpu_baseline="off", subconfigs="off")


@pytest.mark.parametrize("config", ["c1", "c2", "c4"])
def test_timed_searches_run_without_accounting(config):
    args = argparse.Namespace(**ARGS)
    if config == "c4":
        out = bench.bench_c4(args, Library, None, None, None)
        assert out["single_root_mean_ms"] == PLAIN_MS
        assert out["single_root_hmean_gteps"] == pytest.approx(NEDGE / PLAIN_MS / 1e6)
        assert out["single_root_kernel"]["k_bottom_up"]["avg_launch_ms"] == 2.5
    else:
        out = getattr(bench, "bench_" + config)(args, Library)
        assert out["value"] == pytest.approx(NEDGE / PLAIN_MS / 1e6)
        assert out["roofline"]["kernel"] == "k_bottom_up"
