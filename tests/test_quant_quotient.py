"""The FP8 quantization's two-operation quotient against the division, on the
host: same FP8 codes for every scale that takes it (tests/quant_quotient_check.cpp)."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]


def test_quotient_gives_the_codes_of_the_division(tmp_path):
    exe = tmp_path / "quant_quotient_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                    f"-I{REPO / 'kvx_amd' / 'csrc'}",
                    str(REPO / "tests" / "quant_quotient_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=300)
    lines = dict(line.split(" ", 1) for line in out.stdout.splitlines())
    assert set(lines) == {"quotient", "rule"}
    for name, rest in lines.items():
        assert rest.startswith("0 of "), (name, rest, out.stderr)
