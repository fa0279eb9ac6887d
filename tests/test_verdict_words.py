"""Words of checked dequantisation calls (``csrc/verdict_words.h``, host code), in a small C++ program."""

import shutil
import subprocess

import pytest

from loraforge_amd import _build

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "verdict_words.h"

int main() {
  lf::VerdictWords words;
  bool taken[lf::VerdictWords::kWords] = {};
  for (int i = 0; i < lf::VerdictWords::kWords; ++i) {
    const int w = words.take();
    if (w < 0 || w >= lf::VerdictWords::kWords || taken[w]) return 1;  // distinct while in use
    taken[w] = true;
  }
  if (words.take() != -1) return 2;  // none left
  words.give(200);
  words.give(3);
  const int a = words.take(), b = words.take();
  if (!((a == 3 && b == 200) || (a == 200 && b == 3)) || words.take() != -1) return 3;  // only what came back
  for (int i = 0; i < lf::VerdictWords::kWords; ++i) words.give(i);
  // Threads: a word is in one hand at a time.
  static int owner[lf::VerdictWords::kWords] = {};
  bool shared = false;
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; ++t)
    threads.emplace_back([&] {
      for (int i = 0; i < 20000; ++i) {
        const int w = words.take();
        if (w < 0 || __atomic_add_fetch(&owner[w], 1, __ATOMIC_SEQ_CST) != 1) shared = true;
        if (w < 0) continue;
        __atomic_sub_fetch(&owner[w], 1, __ATOMIC_SEQ_CST);
        words.give(w);
      }
    });
  for (auto& t : threads) t.join();
  return shared ? 4 : 0;
}
"""


def test_a_word_belongs_to_one_call_at_a_time(tmp_path):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    source, program = tmp_path / "words.cpp", tmp_path / "words"
    source.write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-pthread", f"-I{_build.CSRC}", str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)]).returncode == 0
