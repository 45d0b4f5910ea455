"""Tuned cluster layouts are remembered safely from several threads.

Eight threads look up and keep layouts of their own keys and of shared ones, as
sessions created at the same time do.  Built with the compiler's thread checker where
it works (an unlocked map is reported as a race and ends the program), else run as it
is: every layout kept is found again.
"""
import shutil
import subprocess

import pytest

from test_cluster_layout_cpu import compile_driver

DRIVER = r'''
#include <thread>
#include "cluster_layout.hpp"
using namespace mp_host;
int main()
{
    LayoutCache cache;
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&cache, t] {
            for (int i = 0; i < 500; ++i) {
                ClusterLayout l, shared;
                l.block = 64 * (1 + i % 8);
                cache.keep(LayoutKey{t, i, 1, 0, 0}, l);
                if (!cache.find(LayoutKey{99, i, 1, 0, 0}, shared)) cache.keep(LayoutKey{99, i, 1, 0, 0}, l);
            }
        });
    for (auto &t : threads) t.join();
    for (int t = 0; t < 8; ++t)
        for (int i = 0; i < 500; ++i) {
            ClusterLayout l;
            if (!cache.find(LayoutKey{t, i, 1, 0, 0}, l) || l.block != 64 * (1 + i % 8)) return 3;
        }
    return 0;
}
'''


def checker(tmp):
    """Flags of the thread checker, none where a clean program does not run under it."""
    flags = ["-fsanitize=thread", "-g"]
    (tmp / "c.cpp").write_text("#include <thread>\nint main(){std::thread([]{}).join();}")
    try:
        subprocess.run([shutil.which("g++") or "g++", *flags, str(tmp / "c.cpp"), "-pthread", "-o",
                        str(tmp / "c")], check=True, capture_output=True)
        subprocess.run([str(tmp / "c")], check=True, capture_output=True, timeout=60)
    except (OSError, subprocess.SubprocessError):
        return []
    return flags


@pytest.mark.parametrize("checked", [False, True])
def test_threads_share_the_cache(tmp_path, checked):
    flags = checker(tmp_path) if checked else []
    if checked and not flags:
        pytest.skip("the thread checker does not run here")
    compile_driver(tmp_path, DRIVER, "-pthread", *flags, "-o", str(tmp_path / "t"))
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
