"""The host's end of the scalar mailbox (cl2qcd_amd/csrc/cl2_mailbox.hpp), compiled for the CPU with transfers that the
test delivers itself: a transfer whose wait failed and that arrives late must not pass for the next one."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "cl2_mailbox.hpp"
#include <cstdio>

static cl2_mailbox box{};
static void deliver(uint64_t number, double v)
{
    box.value[0] = v;
    __atomic_store_n(&box.number, number, __ATOMIC_RELEASE);
}

int main()
{
    cl2_mail_reader reader;
    // the box is asked for until there is one, and then no more
    if (reader.open([] { return (cl2_mailbox*)nullptr; })) return 6;
    if (!reader.open([] { return &box; }) || !reader.open([] { return (cl2_mailbox*)nullptr; })) return 7;
    double got = 0.;
    // one that comes at once, and one that comes while the stream is waited for
    if (reader.read(&got, 1, [](uint64_t k) { deliver(k, 1.); return 0; }, [] { return 9; }) != 0 || got != 1.) return 1;
    uint64_t sent = 0;
    auto send = [&](uint64_t k) { sent = k; return 0; };
    if (reader.read(&got, 1, send, [&] { deliver(sent, 2.); return 0; }) != 0 || got != 2.) return 2;
    // a wait that fails, then the next read: the failed transfer arrives before its own
    uint64_t failed = 0;
    if (reader.read(&got, 1, [&](uint64_t k) { failed = k; return 0; }, [] { return 7; }) != 7 || got != 2.) return 3;
    if (reader.read(&got, 1, [&](uint64_t k) { deliver(failed, 3.); sent = k; return 0; },
                    [&] { deliver(sent, 4.); return 0; }) != 0 || got != 4.) return 4;
    // what could not be enqueued is an error at once
    if (reader.read(&got, 1, [](uint64_t) { return 5; }, [] { return 0; }) != 5 || got != 4.) return 5;
    return 0;
}
"""


def test_late_transfer_does_not_pass_for_the_next(tmp_path):
    src, exe = tmp_path / "mail.cpp", tmp_path / "mail"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "cl2qcd_amd", "csrc"), str(src), "-o",
                    str(exe), "-pthread"], check=True)
    assert subprocess.run([str(exe)], timeout=20).returncode == 0
