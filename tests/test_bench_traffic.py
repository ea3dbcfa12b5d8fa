"""bench.py shows a kernel's measured HBM traffic beside its compulsory bytes
only when the summary was taken of a launch of the same bytes."""
import glob
import os

import bench
from conftest import ROOT


def test_committed_summaries_name_their_launch():
    files = glob.glob(os.path.join(ROOT, "profiles", "traffic_k_?_fast_debye256_*.txt"))
    assert len(files) == 4
    for f in files:
        kernel, prec = os.path.basename(f)[len("traffic_"):-len(".txt")].split("_debye256_")
        vals = dict(x.split() for x in open(f) if len(x.split()) == 2 and x[0] != "#")
        of = int(vals["algorithmic_bytes"])
        got = bench._traffic(kernel, prec, of)
        # no launch moves less than its bytes, and the sweeps' tiles not much more
        assert of <= got <= 1.25 * of
        assert bench._traffic(kernel, prec, of - 2) is None


def test_summary_without_its_launch_is_not_shown(tmp_path, monkeypatch):
    (tmp_path / "profiles").mkdir()
    f = tmp_path / "profiles" / "traffic_k_e_fast_debye256_fp32.txt"
    f.write_text("kernel k_e_fast\ntraffic_bytes_per_launch 599627141\n")
    monkeypatch.setattr(bench, "HERE", str(tmp_path))
    assert bench._traffic("k_e_fast", "fp32", 594450288) is None
    assert bench._traffic("k_e_fast", "fp64", 594450288) is None
    f.write_text("kernel k_e_fast\nalgorithmic_bytes 594450288\ntraffic_bytes_per_launch 651145168\n")
    assert bench._traffic("k_e_fast", "fp32", 594450288) == 651145168
