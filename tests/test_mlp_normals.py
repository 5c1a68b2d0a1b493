"""The normal deviates of a network's initial weights (normals.h) are those of std::normal_distribution<float>, so that
networks of a seed stay the same."""
import os
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "clode_amd", "csrc", "mlp", "normals.h")

MAIN = r"""
#include "%s"
#include <cstdio>
#include <cstring>
int main()
{
    unsigned long long different = 0;
    for (unsigned long long seed : {0ull, 1ull, 13ull, 12345ull, 1ull << 40, ~0ull})
        for (int k = 0; k < 20; ++k) {
            clode::Normals mine(seed + 977 * k);
            std::mt19937_64 rng(seed + 977 * k);
            std::normal_distribution<float> theirs(0.f, 1.f);
            for (int i = 0; i < 20001; ++i) {
                const float a = mine(), b = theirs(rng);
                different += std::memcmp(&a, &b, 4) != 0;
            }
        }
    std::printf("%%llu\n", different);
}
"""


def test_deviates_are_those_of_the_standard_library(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O2", str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    out = subprocess.run([str(tmp_path / "main")], capture_output=True, text=True, check=True, timeout=120).stdout
    assert out.strip() == "0"
