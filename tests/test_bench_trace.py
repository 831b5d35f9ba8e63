"""bench.py's kernel-trace summary: the decode phase is the longest run of dispatches with no launch of a block step's or
panel's GEMM, also where the context was built in panels of more dispatches than the decode steps."""
import csv
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import bench  # noqa: E402


def test_decode_phase_of_a_run_with_panels(tmp_path):
    names = ["k_embed"] * 5
    for _ in range(6):
        names += ["k_panel_split", "void k_panel_gemm<4, 4>(PanelGemmArgs)", "k_panel_epi"] * 10
    names += ["k_gemv_xm", "k_attn_mfma", "k_finish"] * 20
    names += ["k_gemv_mt", "k_block_epi"] * 8
    path, out = tmp_path / "trace.csv", tmp_path / "out.md"
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, ["Kernel_Name", "Start_Timestamp", "End_Timestamp", "Grid_Size_X", "Grid_Size_Y"])
        w.writeheader()
        for i, n in enumerate(names):
            w.writerow(dict(Kernel_Name=n, Start_Timestamp=1000 * i, End_Timestamp=1000 * i + 500, Grid_Size_X=256, Grid_Size_Y=1))
    bench.trace_summary(str(path), str(out))
    text = out.read_text()
    decode = text.split("### other")[0]
    assert "### decode: 61 dispatches" in decode  # (the last panel's epilogue among them)
    assert "`k_gemv_xm` | 20" in decode and "k_panel_gemm" not in decode
    assert "`k_panel_gemm<4, 4> grid 256x1` | 60" in text.split("### other")[1]
