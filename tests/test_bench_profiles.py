"""bench.py's summaries of rocprofv3 results, on counter files of two calls:
bytes per launch are per call, whichever ordering the calls took, and every
layer's contraction has its phase in each of its launch shapes."""
import csv

import pytest

import bench

LARGE = ["k_decode", "k_rs_hist", "k_pscan<24, 48, true, true>", "k_outt<24, 48, 2, 1, 3>",
         "k_pscan<48, 48, false, true>", "k_outt<48, 48, 1, 3, 1>", "k_pscan<48, 96, true, false>",
         "k_outt<48, 96, 1, 3, 1>", "k_pscan<96, 96, false, false>", "k_outt<96, 96, 1, 3, 1>",
         "k_head", "k_emit<128>"]
SMALL = ["k_small_order<{}>", "k_pscan<24, 48, true, true>", "k_outt<24, 48, 1, 9, 1>",
         "k_pscan<48, 48, false, true>", "k_outt<48, 48, 1, 9, 1>", "k_pscan<48, 96, true, false>",
         "k_outt<48, 96, 1, 9, 1>", "k_pscan<96, 96, false, false>", "k_outt<96, 96, 1, 3, 1>",
         "k_head_linear", "k_emit<8>"]
PHASES = {"order", "L4.proj", "L4.out", "L5.proj", "L5.out", "L6.proj", "L6.out", "L7.proj",
          "L7.out", "head", "emit"}


def _counters(d, kernels, calls, kib):
    d.mkdir()
    with open(d / "c_counter_collection.csv", "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Dispatch_Id", "Kernel_Name", "Counter_Value"])
        for i, k in enumerate(kernels * calls):
            w.writerow([i, f"void ssla::(anonymous namespace)::{k}(int, float*)", kib])
    return str(d)


@pytest.mark.parametrize("kernels", [LARGE, [k.format("true") for k in SMALL],
                                     [k.format("false") for k in SMALL]])
@pytest.mark.parametrize("calls", [1, 2])          # (exact shares)
def test_bytes_are_per_call(tmp_path, kernels, calls):
    fetch = _counters(tmp_path / "f", kernels, calls, 4)
    write = _counters(tmp_path / "w", kernels, calls, 2)
    copy = _counters(tmp_path / "c", ["copy"], 1, 8)          # 8 KiB read as 8 KiB: scale 1
    res = bench.pmc_summary(fetch, write, copy, copy, 8 * 1024, "cmd")
    assert set(res["launches"]) == PHASES
    for ph, r in res["launches"].items():
        launches = 2 if ph == "order" and kernels is LARGE else 1
        assert r == {"fetch_bytes": launches * 4096, "write_bytes": launches * 2048,
                     "hbm_bytes": launches * 6144}, ph


def test_no_call_is_an_error(tmp_path):
    fetch = _counters(tmp_path / "f", ["k_batch_drain"], 2, 4)
    copy = _counters(tmp_path / "c", ["copy"], 1, 8)
    with pytest.raises(ValueError, match="no whole-ring drain"):
        bench.pmc_summary(fetch, fetch, copy, copy, 8 * 1024, "cmd")


def test_committed_profiles_are_of_the_default_call_only():
    """The committed traffic and trace are of 200,000 records at 80x64: no
    other call's roofline line takes its traffic or launch time from them."""
    per, flops, byts, iface = {"L5.proj": 1.9}, {"L5.proj": 1e11}, {"L5.proj": 4e9}, {"L5.proj": 8e8}
    own = bench._roofline(per, flops, byts, iface, "L5.proj", True)
    assert own["traffic"] and own["avg_launch_ms_kernel_trace"] and "frac_kernel_trace" in own
    other = bench._roofline(per, flops, byts, iface, "L5.proj", False)
    assert other["traffic"] is None
    assert "frac_kernel_trace" not in other and "avg_launch_ms_kernel_trace" not in other
    assert other["frac"] == own["frac"]
