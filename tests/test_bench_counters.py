"""bench.py's counter summaries on a small CSV: the calibration copies are found by their kernel's name without template
arguments, and traffic is scaled by them."""
import importlib
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
bench = importlib.import_module("bench")

ROW = '%d,"void tsn::(anonymous namespace)::%s(float const*, float*, unsigned long)",%s,%g,1000,2000\n'


def _csv(path, rows):
    path.write_text("Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value,Start_Timestamp,End_Timestamp\n" +
                    "".join(ROW % ((i,) + r) for i, r in enumerate(rows)))
    return str(path)


def test_calibration_copy_is_found(tmp_path):
    kib = bench.CAL_COPY_FLOATS * 4 / 1024.0
    for name in ("copy_kernel", "copy_kernel<true>"):
        f = _csv(tmp_path / "f.csv", [(name, "FETCH_SIZE", kib / 2), ("other_kernel", "FETCH_SIZE", 8)])
        w = _csv(tmp_path / "w.csv", [(name, "WRITE_SIZE", kib), ("other_kernel", "WRITE_SIZE", 4)])
        line = [x for x in bench.pmc_summary(f, w, "cmd").split("\n") if x.startswith("other_kernel")][0]
        assert float(line.split()[-1]) == 8 * 1024 * 2 + 4 * 1024
        sq = _csv(tmp_path / "s.csv", [("other_kernel", c, 64.0) for c in (
            "SQ_VALU_MFMA_BUSY_CYCLES", "SQ_INSTS_VALU", "SQ_INSTS_MFMA", "SQ_INSTS_VALU_MFMA_MOPS_F16", "SQ_INSTS_LDS",
            "SQ_WAVES", "GRBM_GUI_ACTIVE")])
        dr = _csv(tmp_path / "d.csv", [(k, c, v) for k, v in ((name, kib * 8), ("other_kernel", 1000.0))
                                       for c in ("TCC_EA0_RDREQ_DRAM_sum", "TCC_EA0_WRREQ_DRAM_sum")])
        line = [x for x in bench.pmc_util_summary(sq, dr, "t", "c").split("\n") if x.startswith("other_kernel")][0]
        assert abs(float(line.split()[-2]) - 2 * 1000 * 128 / 1e6) < 0.01   # DRAM MB at 128 bytes a request
