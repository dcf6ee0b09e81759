"""The code-book quantizer's lookup without a quotient (csrc/code_book_cells.h), on the CPU."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_lookup_without_a_quotient_is_the_search_on_the_ieee_quotient(tmp_path):
    """For each book and 20,000 scales from 1e-6 to 2^61 (all mantissa bits, 8, 11 and few): dividends next to every step
    and cell end, 16-bit dividends around the steps and random ones, with reciprocals two ulps to either side.  For stochastic
    rounding the entry below a quotient against the search, and the fraction of the gap against the division for every
    significand and gap."""
    binary = tmp_path / "check_book_quotients"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-o", str(binary),
                    str(ROOT / "tests" / "native" / "check_book_quotients.cpp")], check=True)
    done = subprocess.run([str(binary), "20000"], capture_output=True, text=True, timeout=600)
    assert done.returncode == 0, done.stdout
    lines = done.stdout.splitlines()
    assert lines[-1] == "MISMATCHES 0" and int(lines[-2].split()[1]) > 6 * 10 ** 8
