"""What is set on a device before a kernel's first launch there (its LDS limit) is set on every device, not once a process. Runs without a GPU."""
import glob
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mimir_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "once_a_device.h"
int main() {
    mimir::OnceADevice once;
    int calls = 0;
    auto set = [&](int status) { return [&calls, status] { calls++; return status; }; };
    auto expect = [&](int device, int status, int returned, int total) {
        if (once(device, set(status)) != returned || calls != total) { std::printf("device %d: %d calls\n", device, calls); return false; }
        return true;
    };
    bool ok = expect(0, 0, 0, 1) && expect(0, 0, 0, 1);       // once on a device
    ok = ok && expect(1, 0, 0, 2) && expect(1, 0, 0, 2);      // and on the next
    ok = ok && expect(7, 5, 5, 3) && expect(7, 0, 0, 4) && expect(7, 5, 0, 4);  // a failure is returned and tried again
    ok = ok && expect(63, 0, 0, 5) && expect(63, 0, 0, 5) && expect(64, 0, 0, 6) && expect(64, 0, 0, 7);
    mimir::OnceADevice shared;
    std::vector<std::thread> threads;
    std::atomic<int> sets{0}, before{0};
    for (int t = 0; t < 8; t++)
        threads.emplace_back([&] {
            for (int i = 0; i < 1000; i++)
                if (shared(i % 4, [&] { sets++; return 0; }) != 0) before++;
        });
    for (auto& t : threads) t.join();
    ok = ok && before == 0 && sets >= 4 && sets <= 32;
    return ok ? 0 : 1;
}
"""


def test_once_on_every_device_and_again_after_a_failure(tmp_path):
    src, out = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", CSRC, str(src), "-o", str(out)], check=True)
    assert subprocess.run([str(out)]).returncode == 0


def test_no_limit_is_kept_for_the_process():
    """Every kernel's limit is raised through LdsLimit, or on each call; a flag of the process's own would leave the other devices without."""
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        text = open(path).read()
        found += len(re.findall(r"\bstatic LdsLimit\b", text))
        assert not re.search(r"atomic<bool>\s+raised", text), path
        for at in re.finditer(r"hipFuncSetAttribute\(", text):
            assert "call_once" not in text[max(0, at.start() - 120):at.start()], path
    assert found >= 14
