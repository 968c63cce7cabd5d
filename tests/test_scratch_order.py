"""Order of the calls that share the static scratch, on a runtime that only
keeps account (scratch_order.cpp): every call waits for the last one before
it, whatever the stream's handle says, since handles do not name streams
(hipStreamPerThread is one value for every thread's own stream, and a new
stream can get a destroyed one's). Needs no GPU.
"""

import subprocess
from pathlib import Path

import pytest

from gfx906_amd import build

HERE = Path(__file__).parent


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("scratch") / "scratch_order"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__=1",
                    "-D__align__(n)=__attribute__((aligned(n)))", "-DHIP_SYMBOL(x)=x",
                    f"-I{build.ROCM / 'include'}", f"-I{build.CSRC}", "-x", "c++",
                    str(build.CSRC / "scratch.hip"), str(HERE / "scratch_order.cpp"),
                    "-o", str(exe), "-pthread"], check=True)
    return exe


def lines(program, what):
    return subprocess.run([str(program), what], check=True, capture_output=True,
                          text=True).stdout.splitlines()


def test_equal_handles_are_ordered(program):
    assert lines(program, "same handle") == [
        "call s2", "record s2 e1", "wait s2 e1", "call s2", "record s2 e1",
        "wait s2 e1", "call s2", "record s2 e1"]


def test_two_streams_are_ordered(program):
    assert lines(program, "two streams") == [
        "call s7", "record s7 e1", "wait s8 e1", "call s8", "record s8 e1",
        "wait s7 e1", "call s7", "record s7 e1"]


def test_captured_calls_neither_wait_nor_record(program):
    assert lines(program, "capture") == [
        "call s7", "record s7 e1", "call s8", "wait s9 e1", "call s9", "record s9 e1"]


def test_a_failed_call_is_waited_for(program):
    """A call whose merge cannot be launched leaves a kernel queued."""
    assert lines(program, "failed call") == [
        "launch s7", "record s7 e1", "wait s8 e1", "call s8", "record s8 e1"]


def test_a_failed_record_waits_on_the_host(program):
    assert lines(program, "failed record") == [
        "call s7", "synchronize s7", "not released", "call s8", "record s8 e1"]
