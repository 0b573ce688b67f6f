"""The benchmark's HBM traffic comes from a measurement of the kernel and the tree that it reports, or is left out."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_is_of_the_kernel_and_tree(tmp_path):
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    f = tmp_path / "traffic.txt"
    f.write_text("text: 1\nbytes_per_launch_m2l_learned: 123 k_m2l 1000\nbytes_per_launch_near_learned: 5\n")
    assert bench.read_traffic("m2l_learned", "k_m2l", 1000, f) == 123
    assert bench.read_traffic("m2l_learned", "k_translate", 1000, f) is None
    assert bench.read_traffic("m2l_learned", "k_m2l", 1001, f) is None
    assert bench.read_traffic("near_learned", "k_near", 1000, f) is None
    assert bench.read_traffic("m2l_fp64", "k_m2l", 1000, f) is None
    assert bench.read_traffic("m2l_fp64", "k_m2l", 1000, tmp_path / "none") is None
    for pair in bench.TRAFFIC_KEYS.values():  # the committed file: well formed, of kernels that exist
        for key, kernel in zip(pair, ("k_m2l", "k_near")):
            line = [v for v in open(bench.TRAFFIC_FILE) if v.startswith(f"bytes_per_launch_{key}:")]
            assert len(line) == 1
            nbytes, name, boxes = line[0].partition(":")[2].split()
            assert name == kernel and bench.read_traffic(key, kernel, int(boxes)) == int(nbytes)
