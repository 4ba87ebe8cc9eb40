"""The executor's idle streams: runs that ask for more distinct CU masks than
the pool keeps, repeated and from two threads at once, give the results of a
first run."""

import os
import threading

import numpy as np
import pytest

from kernrelay_amd import dag_bench, libapi, schedule, workloads
from tests.conftest import announce

pytestmark = pytest.mark.gpu

M, K, N = 256, 128, 256


def run(path, out, mode):
    with dag_bench._stdout_to_stderr():
        r = libapi.plan_run(path, mode=mode, iters=1, warmup=0, out_json=out)
    assert r["_rc"] == 0 and r["ok"], r
    return r["checksum"]


def test_runs_share_idle_streams(gpu, tmp_path):
    inputs = workloads.write_inputs(str(tmp_path), M, K, N, 3)
    dag = schedule.dag_from_dict(workloads.mm_consumers_dag("fanout", M, K, N, ("softmax", "gelu", "cast"),
                                                            inputs=inputs))
    path = schedule.dump_schedule(workloads.variants(dag, 2)["split"], tmp_path / "schedule.json")
    announce("stream pool: five CU masks, twice, two modes")
    sums = []
    try:
        for cus in ("0", "1", "2", "3", "4") * 2:  # the pool keeps four idle streams
            os.environ["KR_CONSUMER_CUS_PER_XCD"] = cus
            sums += [run(path, tmp_path / "o.json", m) for m in ("direct", "graph_per_stream")]
    finally:
        del os.environ["KR_CONSUMER_CUS_PER_XCD"]
    assert len(set(sums)) == 1 and np.isfinite(sums[0])
    announce("stream pool: two threads")
    got, errors = [], []

    def work(i):
        try:
            for _ in range(3):
                r = libapi.plan_run(path, mode="direct", iters=1, warmup=0, out_json=tmp_path / ("t%d.json" % i))
                assert r["_rc"] == 0 and r["ok"], r
                got.append(r["checksum"])
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and set(got) == {sums[0]}
