"""The host transfers (rhyme_amd/csrc/rhy_transfer.hip) compiled for the host
against a runtime of plain memory copies (tests/hostrt) that counts what it is
asked for: which copies are staged, and what happens to the staging memory and
its threads where a device run cannot easily bring it about."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rhyme_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfers") / "transfers")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(HERE, "hostrt"),
                    "-I", CSRC, os.path.join(HERE, "hostrt", "transfers.cpp"), "-o", exe],
                   check=True)
    return exe


def call(program, *args):
    r = subprocess.run([program] + [str(a) for a in args], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, (args, r.returncode, r.stdout, r.stderr)
    return {k: int(v) for k, v in re.findall(r"(\w+) (\d+)", r.stdout)}


# the sizes (KiB of device values) on both sides of each measured crossover:
# a copy in one piece up to it, in chunks from it on
@pytest.mark.parametrize("kind,way,least", [("same", "up", 32 << 10), ("same", "down", 8 << 10),
                                            ("mixed", "up", 8 << 10), ("mixed", "down", 4 << 10)])
def test_staged_only_where_it_is_faster(program, kind, way, least):
    for kib, staged in ((1 << 10, False), (3 << 10, False), (least - 1, False), (least, True),
                        (2 * least + 1, True)):
        got = call(program, "route", kib, kind, way)
        assert (got["copies"] > 1) == staged, (kib, kind, way, got)
        assert got["events"] == 0 and got["pinned"] == 0  # all given back


def test_pinned_caller_memory_is_copied_directly(program):
    assert call(program, "pinned")["copies"] == 2


def test_box_on_another_device_than_the_current_one(program):
    assert call(program, "device")["current"] == 1


def test_no_memory_on_the_way(program):
    """Whichever allocation fails, the copy is made, in one piece or in chunks."""
    got = call(program, "memory")
    assert got["events"] == 0 and got["pinned"] == 0


def test_short_lived_objects_do_not_pay_for_staging(program):
    assert call(program, "short")["asked"] == 0
    got = call(program, "long")
    assert got["asked"] == 1 and got["held"] == 1 and got["pinned"] == 0


def test_refused_pinned_memory_is_asked_for_once(program):
    got = call(program, "refused")
    assert got["asked"] == 1 and got["copies"] == 10


def test_a_copy_whose_caller_waits_does_not_wait_too(program):
    got = call(program, "wait")
    assert got["unwaited"] == 0 and got["waited"] == 1
