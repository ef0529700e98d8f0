"""bench.py's command-line contract that can be checked without a GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                          timeout=120)
    assert proc.returncode != 0
    assert "one GPU" in proc.stderr and proc.stdout.strip() == ""


def test_counter_file_of_the_profiler_is_read_per_kernel(tmp_path):
    """bench.py takes its live traffic figure from rocprofv3's counter_collection.csv: median over the copy
    kernel's dispatches, the yardstick kernel apart, other kernels and counters ignored."""
    sys.path.insert(0, ROOT)
    import bench
    rows = [("copy_uniform_kernel<1, 4, 1>(x)", "A", 10.0), ("copy_uniform_kernel<1, 4, 1>(x)", "A", 30.0),
            ("copy_uniform_kernel<1, 4, 1>(x)", "A", 20.0), ("copy_uniform_kernel<1, 4, 1>(x)", "B", 7.0),
            ("void at::native::vectorized_elementwise_kernel<4, at::native::CUDAFunctorOnSelf_add<int>, a>(b)", "A", 5.0),
            ("void at::native::vectorized_elementwise_kernel<4, at::native::CUDAFunctorOnSelf_add<int>, a>(b)", "A", 6.0),
            ("void at::native::vectorized_elementwise_kernel<4, at::native::CUDAFunctorOnSelf_add<int>, a>(b)", "B", 2.0),
            ("some_other_kernel(y)", "A", 1e9), ("copy_uniform_kernel<1, 4, 1>(x)", "C", 1e9)]
    path = tmp_path / "t_counter_collection.csv"
    with open(path, "w") as f:
        f.write('"Dispatch_Id","Kernel_Name","Counter_Name","Counter_Value"\n')
        for i, (k, c, v) in enumerate(rows):
            f.write(f'{i},"{k}","{c}",{v}\n')
    kernel, yard, n = bench.counter_samples(str(path), ["A", "B"])
    assert kernel == {"A": 20.0, "B": 7.0} and yard == {"A": 6.0, "B": 2.0} and n == 3
    assert bench.counter_samples(str(path), ["A", "D"]) is None


def test_phase_timers_are_read_from_the_debug_lines():
    """bench.py's breakdown of a request made through prepXfer comes from the debug lines of the
    agent and of the plugin: one entry per request and phase, other lines ignored."""
    sys.path.insert(0, ROOT)
    import bench
    text = "\n".join([
        "[nixl D] backend HIP: prepared 524288 descriptors into 1 strides",
        "[nixl D] makeXferReq: merged 65536 indices into 65536 descriptors in 128.5 us",
        "[nixl D] HIP backend: prepXfer of 65536 descriptors (blocks): block pass 124.525 us, plan from records 8.03 us, "
        "rest (general lowering, event, stream) 0.611 us",
        "[nixl D] makeXferReq: merged 65536 indices into 65472 descriptors in 1.3e+02 us",
        "[nixl D] HIP backend: prepXfer of 65472 descriptors (general): block pass 0 us, plan from records 0 us, "
        "rest (general lowering, event, stream) 2500.5 us"])
    phases, paths = bench.parse_prep_debug_lines(text)
    assert phases == {"agent_expand_index_pairs": [128.5, 130.0], "plugin_block_pass": [124.525, 0.0],
                      "plugin_plan_from_records": [8.03, 0.0], "plugin_rest": [0.611, 2500.5]}
    assert paths == ["blocks", "general"]


def test_counter_file_is_read_for_several_kernels_at_once(tmp_path):
    """The expert-parallel traffic figures: medians per kernel tag from one counter file, a tag
    without samples left out, the yardstick apart."""
    sys.path.insert(0, ROOT)
    import bench
    rows = [("void (anonymous namespace)::ll_bits_kernel<false, 1>(a)", "A", 3.0),
            ("void (anonymous namespace)::ll_bits_kernel<true, 4>(a)", "A", 100.0),
            ("void (anonymous namespace)::ll_dispatch_kernel<true>(a)", "A", 10.0),
            ("void (anonymous namespace)::ll_dispatch_kernel<true>(a)", "A", 30.0),
            ("void (anonymous namespace)::ll_dispatch_kernel<true>(a)", "A", 20.0),
            ("void at::native::vectorized_elementwise_kernel<4, at::native::CUDAFunctorOnSelf_add<int>, a>(b)", "A", 8.0)]
    path = tmp_path / "t_counter_collection.csv"
    with open(path, "w") as f:
        f.write('"Dispatch_Id","Kernel_Name","Counter_Name","Counter_Value"\n')
        for i, (k, c, v) in enumerate(rows):
            f.write(f'{i},"{k}","{c}",{v}\n')
    medians, yard = bench.counter_medians(str(path), ["A"], ["ll_bits_kernel<false", "ll_dispatch_kernel<true>", "ll_scales_kernel"])
    assert medians == {"ll_bits_kernel<false": {"A": 3.0}, "ll_dispatch_kernel<true>": {"A": 20.0}} and yard == {"A": 8.0}


def test_a_kernel_that_is_not_launched_costs_no_call_its_traffic():
    """The receive-side counts of normal mode share the scan's launch up to a number of tokens, so that their own kernel may have no
    samples: every call keeps its figure, and a call that lacks one of its kernels is the only one without."""
    sys.path.insert(0, ROOT)
    import bench
    from nixl_amd import ep_bench
    classes = {"A": 128, "B": 64}
    names = {k for ks in ep_bench.CALL_KERNELS.values() for k in ks}
    read = {k: {"A": 10.0, "B": 2.0} for k in names}
    written = {k: {"WRITE_SIZE": 3.0} for k in names}
    one = 10 * 128 + 2 * 64 + 3 * 1024 * 2
    got = bench.ep_call_traffic(read, written, classes, 2.0)
    assert {c: v["traffic"] for c, v in got.items()} == {c: one * len(ks) for c, ks in ep_bench.CALL_KERNELS.items()}
    for side, value in ((read, {"A": 1.0, "B": 0.0}), (written, {"WRITE_SIZE": 1.0})):
        side["ht_prefix_kernel"] = value
    assert bench.ep_call_traffic(read, written, classes, 2.0)["ht_dispatch"]["traffic"] == 2 * one + 128 + 2048
    del read["ll_scales_kernel"]
    got = bench.ep_call_traffic(read, written, classes, 2.0)
    assert got["ll_dispatch"]["traffic"] is None and "ll_scales_kernel" in got["ll_dispatch"]["traffic_live_error"]
    assert got["ll_combine"]["traffic"] == one


def test_the_kernels_whose_traffic_is_counted_exist():
    """Every kernel that the traffic figures name is one of the sources' (a renamed one would have no samples), and no
    name stands for two of a call's kernels."""
    import re
    from nixl_amd import ep_bench
    kernels = os.path.join(ROOT, "nixl_amd", "csrc", "kernels")
    defined = {name for f in os.listdir(kernels) if f.endswith(".hip")
               for name in re.findall(r"^(\w+_kernel)\(", open(os.path.join(kernels, f)).read(), re.M)}
    for calls in (ep_bench.CALL_KERNELS, ep_bench.CALL_KERNELS_IF_LAUNCHED):
        for names in calls.values():
            assert all(len([d for d in defined if name.split("<")[0] in d]) == 1 for name in names), names
