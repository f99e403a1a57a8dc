"""Which large batches of short rows run as one launch of the grid form (csrc/paged_attention_policy.h), compiled for the host:
batches that were timed both ways on 256 compute units keep the form that was faster."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash_attention_factory_amd", "csrc")

# head size, sequences, kv heads, extended, kv heads side by side -> time of the grid form over that of sub-batches
TIMED = [
    (64, 150, 1, True, False, 0.44), (64, 200, 8, True, False, 0.61), (64, 264, 8, False, True, 0.61), (64, 340, 8, True, False, 0.47),
    (64, 509, 16, False, True, 0.79), (64, 552, 16, True, True, 0.66), (64, 634, 16, True, True, 0.77), (64, 132, 32, False, True, 0.77),
    (64, 169, 32, True, True, 0.83), (64, 260, 32, True, True, 0.87),
    (64, 384, 24, True, True, 1.20), (64, 218, 64, True, True, 1.51), (64, 214, 32, True, False, 1.03), (64, 224, 32, True, True, 1.13), (64, 225, 32, False, True, 1.14), (64, 248, 32, True, True, 1.17),
    (64, 252, 32, True, True, 1.32), (64, 291, 32, True, True, 1.14), (64, 302, 32, True, True, 1.24), (64, 307, 32, True, True, 1.37),
    (64, 325, 32, False, True, 1.10), (64, 335, 32, True, True, 1.46), (64, 421, 32, True, False, 1.07), (64, 544, 32, True, True, 1.18),
    (64, 591, 32, False, True, 1.45), (64, 216, 32, False, False, 0.84), (64, 325, 32, False, False, 0.72), (64, 448, 32, False, False, 0.74),
    (128, 148, 1, False, False, 0.46), (128, 481, 2, True, True, 0.6), (128, 182, 4, True, False, 0.81), (128, 268, 4, True, True, 0.76),
    (128, 288, 4, True, False, 0.85), (128, 228, 4, False, True, 0.76), (128, 254, 5, False, False, 0.77), (128, 147, 8, True, True, 0.78),
    (128, 204, 4, True, False, 1.06), (128, 211, 4, True, True, 1.06), (128, 215, 4, True, True, 1.10), (128, 244, 4, True, True, 1.06),
    (128, 247, 4, True, False, 1.05), (128, 173, 5, True, True, 1.03),
    (128, 161, 8, False, False, None), (128, 150, 32, False, False, None),  # more than five rows a unit
]


def test_timed_batches_keep_the_faster_form(tmp_path):
    calls = "".join(f"  printf(\"%d\\n\", fa::short_rows_run_as_grid({d}, {s}, 128, {hk}, 256, {int(e)}, {int(a)}));\n"
                    for d, s, hk, e, a, _ in TIMED)
    src, exe = tmp_path / "policy.cpp", tmp_path / "policy"
    src.write_text(f'#include <cstdio>\n#include "paged_attention_policy.h"\nint main() {{\n{calls}}}\n')
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    got = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    for (*batch, ratio), grid in zip(TIMED, got):
        assert grid == str(int(ratio is not None and ratio < 1)), (batch, ratio)
    assert len(got) == len(TIMED)
