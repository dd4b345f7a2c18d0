"""What the host classes queue, wait for and refuse, on a runtime that only keeps count (tests/native/fake_hip.cpp, linked
in front of HIP's): no GPU is used, kernels do not run.  Each scenario of tests/native/stream_order.cpp is a process of its own."""
import os
import subprocess
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
NATIVE = os.path.join(HERE, "native")
PKG = os.path.join(os.path.dirname(HERE), "grape_amd")
FAKE, EXE = os.path.join(NATIVE, "libfake_hip.so"), os.path.join(NATIVE, "stream_order")


@pytest.fixture(scope="module")
def program():
    src = [os.path.join(NATIVE, f) for f in ("fake_hip.cpp", "stream_order.cpp")]
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", FAKE, src[0]])
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-Wno-class-memaccess", "-o", EXE, src[1],
                           "-Wl,--no-as-needed", "-L" + NATIVE, "-lfake_hip", "-L" + os.path.join(PKG, "host"), "-lgrape_host", "-L" + PKG, "-lgrape_hip",
                           "-Wl,-rpath,$ORIGIN/../../grape_amd/host", "-Wl,-rpath,$ORIGIN/../../grape_amd", "-Wl,-rpath,$ORIGIN"])
    return EXE


@pytest.mark.parametrize("scenario", ["refused_lookup", "proof_after_a_refused_one", "mapping_objects", "carried_lookups", "the_longest_indexed_range", "where_padding_is_free", "a_mapping_with_another_r", "lookups_without_a_weighted_term",
                                      "weights_that_are_read", "tensor_memory_is_idle", "sparse_commitment_table",
                                      "scaled_tables_that_grow", "operands_at_any_address", "element_products_that_carry", "a_tensor_times_itself", "padded_openings", "verify_with_more_variables",
                                      "single_rows_without_memory", "single_row_table_gives_way", "tables_of_single_rows", "a_sum_behind_a_failed_one", "verify_with_another_generator", "blocks_of_two_devices",
                                      "default_order_blocks", "short_copies"])
def test_scenario(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
