"""FairShare (fair_share.h): a part that needs everything is not passed over by small ones that ask later."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "fair_share.h"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <string>
#include <thread>
#include <vector>

using namespace mm;

int main()
{
  ShareGate g;
  std::string order;
  std::mutex mu;
  const auto asked = [&](unsigned long long n) {
    for (;;) {
      {
        std::lock_guard<std::mutex> lk(g.mu);
        if (g.next == n) return;
      }
      std::this_thread::yield();
    }
  };
  const auto take = [&](char name, long long part) {
    FairShare s(g, part, 10);
    std::lock_guard<std::mutex> lk(mu);
    order += name;
  };
  std::vector<std::thread> ts;
  {
    FairShare first(g, 3, 10);
    ts.emplace_back(take, 'B', 10);  // waits for everything
    asked(2);
    for (int i = 0; i < 4; i++) {  // would fit beside the first
      ts.emplace_back(take, 's', 1);
      asked(3 + i);
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    std::lock_guard<std::mutex> lk(mu);
    if (!order.empty()) return 1;
  }
  for (auto &t : ts) t.join();
  printf("%s\n", order.c_str());
  // many threads, parts of all sizes: never more than the whole
  std::atomic<long long> held{0}, most{0};
  std::vector<std::thread> many;
  for (int i = 0; i < 8; i++)
    many.emplace_back([&, i] {
      for (int k = 0; k < 200; k++) {
        const long long part = 1 + (7 * i + 3 * k) % 10;
        FairShare s(g, part, 10);
        const long long now = held += part;
        if (now > most) most = now;
        held -= part;
      }
    });
  for (auto &t : many) t.join();
  return order == "Bssss" && most <= 10 && g.used == 0 ? 0 : 2;
}
"""


def test_in_the_order_of_asking(tmp_path):
    src, exe = tmp_path / "share.cpp", tmp_path / "share"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "madmax_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], timeout=60, capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
