"""Which of a context's assemblies are launched, recorded and replayed (csrc/graph_rule.hpp), on the CPU:
a program around the header walks through sequences of assemblies as the library does and prints
each step."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fem_2d_amd", "csrc")

# a Domain is a letter; a capital one has row groups of the block path. Whether it has is not known
# before its first assembly, which launches that path's kernels in any case.
PROGRAM = r"""
#include <cctype>
#include <cstdio>
#include <map>
#include "graph_rule.hpp"
int main(int, char** argv) {
  fem2d::GraphRule rule;
  std::map<char, int> large;
  for (const char* p = argv[1]; *p; ++p) {
    fem2d::GraphKey key;
    key.domain = (unsigned char)*p;
    key.capacity = 1;
    key.precision = 0;
    key.run_large = !large.count(*p) || large[*p] != 0;
    const auto step = rule.step(key);
    if (step == fem2d::GraphRule::kRecord) {
      rule.forget();
      rule.made(key);
    }
    rule.came(key);
    large[*p] = std::isupper((unsigned char)*p) ? 1 : 0;
    rule.learned(large[*p] != 0);
    std::putchar(step == fem2d::GraphRule::kLaunch ? 'l' : step == fem2d::GraphRule::kRecord ? 'r' : 'p');
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("graph_rule")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{CSRC}", str(d / "main.cpp"), "-o",
                    str(d / "main")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("domains,steps", [
    ("AAAA", "lrpp"),
    ("aaaa", "lrpp"),  # recorded the second time in a row, though the first one launched more kernels
    ("abab", "llll"),
    ("aabaa", "lrlpp"),  # a recording stays until another is made
    ("aabbaa", "lrlrlr"),
    ("aAaaA", "lllrl"),
])
def test_steps(program, domains, steps):
    out = subprocess.run([program, domains], check=True, capture_output=True, text=True).stdout
    assert out == steps
