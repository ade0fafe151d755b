"""What a kernel is told before its first launch (neura_amd/csrc/once_a_device.hpp): once on each device, again where it failed, and every
time on devices past the 64 the word counts."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_device_is_told_once(tmp_path):
    source, program = tmp_path / "once.cpp", tmp_path / "once"
    source.write_text('#include "%s"\n#include <cstdio>\nint main() {\n    static nh::OnceADevice one, other;\n    int calls = 0, answer = 1;\n'
                      '    auto tell = [&] { calls++; return answer; };\n    auto ask = [&](nh::OnceADevice &of, int device) { std::printf("%%d ", of(device, tell)); std::printf("%%d\\n", calls); };\n'
                      '    ask(one, 0);\n    answer = 0;\n    ask(one, 0), ask(one, 0), ask(one, 7), ask(one, 7), ask(one, 63), ask(one, 63), ask(one, 64), ask(one, 64), ask(other, 0);\n}\n'
                      % os.path.join(ROOT, "neura_amd", "csrc", "once_a_device.hpp"))
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-o", str(program), str(source)], check=True)
    said = subprocess.run([str(program)], capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
    assert said == ["1 1", "0 2", "0 2", "0 3", "0 3", "0 4", "0 4", "0 5", "0 6", "0 7"]
