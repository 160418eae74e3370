"""bench.py --traffic-summary on a run of the direct solve: bytes per evaluation of its
kernels, the factorisation's together, as the roofline line reads them back."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench


def test_traffic_summary_of_a_direct_run(tmp_path, capsys, monkeypatch):
    copy = {"FETCH_SIZE": 524288.0, "WRITE_SIZE": 1048576.0}   # KiB read for the 1 GiB copy: factors 2 and 1
    kernels = {"void jsso::k_front_small<512>(jsso::DirectDev)": 100.0, "jsso::k_front_cb(jsso::DirectDev)": 30.0,
               "void jsso::k_solve_fwd<1>(jsso::DirectDev)": 7.0, "void jsso::ell_assemble_kernel(long)": 50.0}
    for counter in copy:
        d = tmp_path / counter
        d.mkdir()
        rows = ["Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value", f"1,copyBuffer,{counter},{copy[counter]}"]
        for solve in range(2):
            rows += [f"{2 + len(rows)},\"{k}\",{counter},{v * (1 + solve)}" for k, v in kernels.items()]
        (d / "run_counter_collection.csv").write_text("\n".join(rows) + "\n")
    log = tmp_path / "bench.log"
    log.write_text(json.dumps({"roofline": {"kernel": bench.FRONT_KERNELS}, "solve_log": {"solves": [[1, 0, 0]] * 2}}))
    bench.traffic_summary(str(tmp_path / "FETCH_SIZE"), str(tmp_path / "WRITE_SIZE"), str(log))
    out = capsys.readouterr().out
    kib = 1024 * 3 / 2   # both counters, three times a kernel's value over two evaluations
    assert f"direct_traffic k_front_small<512>: fetch {int(100 * kib * 2)} write {int(100 * kib)}" in out
    assert f"direct_traffic k_solve_fwd<1>: fetch {int(7 * kib * 2)}" in out
    assert f"assembly_traffic ell_assemble_kernel: fetch {int(50 * kib * 2)}" in out
    os.makedirs(tmp_path / "profiles")
    (tmp_path / "profiles" / "t.txt").write_text(out)
    monkeypatch.setattr(bench, "HERE", str(tmp_path))
    assert bench._measured_traffic("t.txt", bench.FRONT_KERNELS) == (int(130 * kib * 3), "profiles/t.txt")
