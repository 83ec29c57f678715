"""The library's host code on the CPU (tests/cpp/api_host_test.cpp): what its entries hand to the launchers, whom they
share memory with, and what they do when the machine refuses something."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.mark.parametrize("name", [
    "partials_and_words_fit",
    "batched_calls_share_nothing",
    "calls_on_the_per_thread_stream_take_turns",
    "host_slices_follow_the_current_device",
    "the_prefill_plan_deals_as_the_kernel_does",
    "a_tiles_lds_has_one_writer",
    "gradients_that_share_memory_take_turns",
    "wide_gradients_read_the_workspace",
    "a_chunks_keys_are_cut_as_its_tests_say",
    "wide_heads_take_the_form_that_pays",
    "a_chunk_of_unknown_lengths_keeps_the_short_walk",
    "no_thread_spins_through_the_kernel",
    "a_host_without_threads_copies_by_itself",
    "a_host_without_memory_is_an_error",
])
def test_host_code(name):
    subprocess.check_call(["make", "-s", "-C", CPP, "api_host_test"])
    r = subprocess.run([os.path.join(CPP, "api_host_test"), name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("ok")
