"""Order of the calls that share the static scratch, on a runtime that only
keeps account (scratch_order.cpp). A call waits for the last ones that used its
pieces of the scratch, whatever their stream's handle says, since handles do
not name streams (a new stream can get a destroyed one's; hipStreamPerThread is
one value for every thread's own stream). Streams and threads get pieces of
their own while these last and do not wait for each other. Needs no GPU.

A line "call s8 3+2" is a call on stream 8 with pieces 3 and 4; piece n's event
is e(n + 1).
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
        "call s7 0+1", "record s7 e1", "wait s7 e1", "call s7 0+1", "record s7 e1",
        "wait s7 e1", "call s7 0+1", "record s7 e1"]


def test_streams_do_not_wait_for_each_other(program):
    assert lines(program, "two streams") == [
        "call s7 0+1", "record s7 e1", "call s8 1+1", "record s8 e2",
        "wait s7 e1", "call s7 0+1", "record s7 e1"]


def test_threads_do_not_wait_for_each_other(program):
    assert lines(program, "threads") == [
        "call s2 0+1", "record s2 e1", "wait s2 e1", "call s2 0+1", "record s2 e1",
        "call s2 1+1", "record s2 e2", "wait s2 e2", "call s2 1+1", "record s2 e2"]


def test_calls_that_share_pieces_are_ordered(program):
    assert lines(program, "full") == [
        "call s7 0+10", "record s7 e1",
        "wait s8 e1", "call s8 0+10", "record s8 e1",
        "call s9 10+6", "record s9 e11",
        "wait s7 e1", "call s7 0+10", "record s7 e1",
        "wait s9 e11", "call s9 10+1", "record s9 e11",
        "wait s8 e1", "wait s8 e11", "call s8 0+16", "record s8 e1",
        "wait s7 e1", "call s7 0+1", "record s7 e1"]


def test_a_new_record_covers_the_old_one(program):
    """Stream 7's second call records the event that guards pieces 1-7 too: the
    next call's wait for it covers both."""
    assert lines(program, "guards") == [
        "call s7 0+8", "record s7 e1", "call s8 8+8", "record s8 e9",
        "wait s7 e1", "call s7 0+1", "record s7 e1",
        "wait s9 e1", "wait s9 e9", "call s9 0+16", "record s9 e1", "1"]


def test_captured_calls_neither_wait_nor_record(program):
    assert lines(program, "capture") == [
        "call s7 0+1", "record s7 e1", "call s8 0+1", "call s9 1+1", "record s9 e2"]


def test_a_failed_call_is_waited_for(program):
    """A call whose merge cannot be launched leaves a kernel queued."""
    assert lines(program, "failed call") == [
        "launch s7", "record s7 e1", "wait s8 e1", "call s8 0+1", "record s8 e1"]


def test_a_failed_record_waits_on_the_host(program):
    assert lines(program, "failed record") == [
        "call s7 0+1", "synchronize s7", "not released", "call s8 0+1", "record s8 e1"]
