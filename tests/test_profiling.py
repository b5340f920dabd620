"""The profile summaries that the benchmark reads."""

import os

import bench
from o_o_solver_amd import profiling


def test_traffic_per_launch_of_one_kernel_and_of_all_of_a_form(tmp_path):
    path = tmp_path / "traffic.txt"
    path.write_text("# kernel dispatches fetch write bytes\n"
                    "  triangleInverseKernel<double,false>   30   1.0   1.0   100\n"
                    "  triangleInverseKernel<double,true>    10   1.0   1.0   500\n"
                    "  triangleInverseKernel<float,true>     10   1.0   1.0   900\n")
    assert profiling.read_traffic(path, "triangleInverseKernel<double,true>") == 500.0
    assert profiling.read_traffic(path, "triangleInverseKernel<double,*>") == 200.0
    assert profiling.read_traffic(path, "triangleInverseKernel<double>") is None
    assert profiling.read_traffic(tmp_path / "absent.txt", "triangleInverseKernel<double,*>") is None


def test_every_kind_of_the_benchmark_is_in_the_committed_summary():
    # The kernels of the kinds whose launches the benchmark's workload makes, named as the trace names them: a kernel
    # that was renamed leaves the benchmark's traffic out.
    assert os.path.exists(bench.TRAFFIC_SUMMARY)
    missing = [kind for kind, name in bench.KIND_KERNELS.items()
               if any(profiling.read_traffic(bench.TRAFFIC_SUMMARY, name.format(T=t)) is None
                      for t in ("double", "float"))]
    assert missing == []
