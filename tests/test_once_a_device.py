"""What a process does once for each of its GPUs (csrc/once_a_device.h), compiled for the host."""
import os
import subprocess

from arle_amd.kernels import build

PROGRAM = """
#include "once_a_device.h"
#include <cstdio>
static arle::OnceADevice made;
int main() {
  const int devices[] = {0, 1, 5, 63, 64, 200, -1};
  for (int device : devices) std::printf("%d", made.done(device));
  for (int device : devices) {
    made.mark(device);
    std::printf(" ");
    for (int other : devices) std::printf("%d", made.done(other));
  }
  return 0;
}
"""


def test_a_device_is_remembered_by_itself(tmp_path):
    source, program = tmp_path / "once.cpp", tmp_path / "once"
    source.write_text(PROGRAM)
    subprocess.run([build.find_host_compiler(), "-std=c++17", "-Wall", "-Werror", f"-I{build.CSRC_DIR}", str(source), "-o", str(program)], check=True)
    said = subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split(" ")
    assert said == ["0000000", "1000000", "1100000", "1110000", "1111000", "1111000", "1111000", "1111000"]


def test_no_launcher_asks_for_lds_once_a_process():
    """The attribute belongs to a device: every launcher goes through the helper that remembers devices."""
    for name in sorted(os.listdir(build.CSRC_DIR)):
        if name.endswith((".hip", ".h")):
            with open(os.path.join(build.CSRC_DIR, name)) as fh:
                text = fh.read()
            assert text.count("hipFuncSetAttribute(") == (1 if name == "common.h" else 0), name
