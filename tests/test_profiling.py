"""CPU: the profile summaries name the kernels that the frames launch."""
import csv

from helios_amd import profiling

CONV = "_ZN2hh2dn9k_conv3x3ILi48ELi2ELi32ELi32ELi5ENS0_9ConvLargeEEEvPKDF16bS4_S4_PKfS4_PvjjjNS0_9ConvExtraE"


def write(path, rows):
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, rows[0].keys())
        w.writeheader()
        w.writerows(rows)
    return path


def test_convolution_names_keep_their_shape():
    assert profiling.demangle(CONV) == "hh::dn::k_conv3x3<48, 2, 32, 32, 5, ConvLarge>"
    assert profiling.demangle("_ZN2hh2dn12k_conv_wgradILi32ELi1ELi0ELi32ELi2ELi2EEEvPKDF16b") == \
        "hh::dn::k_conv_wgrad<32, 1, 0, 32, 2, 2>"
    assert profiling.demangle("_ZN2hh2dn14k_reduce_gradsENS0_10GradSlicesE") == "hh::dn::k_reduce_grads"


def test_passes_list_shared_launches(tmp_path):
    names = ["k_generate<64>", "k_extend_packet<4, 64>", "k_shade<64>", "k_shadow<4, 64, 0, false>", "k_extend<4, 64, 0, false>",
             "k_shade<64>", "k_trace<4, 64, 0>", "k_shade<64>", "k_trace<4, 64, 0>", "k_extend<4, 256, 0, true>"]
    rows = [dict(Kernel_Name=f"void hh::{n}(hh::SceneGPU const*)", Start_Timestamp=1000 * i, End_Timestamp=1000 * i + 500,
                 Queue_Id=1) for i, n in enumerate(names)]
    text = profiling.passes_md(write(tmp_path / "t.csv", rows))
    assert "| 1 | hh::k_generate<64> | 2 | 0.5 | 2 | 0.5 | 1 | 0.5 |" in text


def test_issue_table_holds_the_shared_launch(tmp_path):
    rows = [dict(Kernel_Name=f"void hh::{k}(hh::SceneGPU const*)", Counter_Name=c, Counter_Value=8.0)
            for k in ("k_trace<4, 64, 0>", "k_extend<4, 64, 0, false>", "k_extend<4, 256, 0, true>")
            for c in profiling.ISSUE_COUNTERS]
    out = profiling.issue(write(tmp_path / "p.csv", rows), "cmd")["kernels"]
    assert set(out) == {"k_trace", "k_extend"}
    assert out["k_trace"]["dispatches"] == 1
