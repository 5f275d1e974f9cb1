"""CPU replay of the base conversion fused with its targets' column pass (tests/emu/
conv_cols_emu.cpp): the sources' bounds, clipped digits beside full ones, 50-, 60- and 40-bit primes
on either side, the extremes of the single-quotient sums, N = 2^12 .. 2^16, against the oracle."""
import subprocess

from test_emu import _build


def test_replay_of_the_fused_conversion_equals_the_oracle():
    r = subprocess.run([_build("conv_cols_emu")], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "EMU OK" in r.stdout
    assert len([l for l in r.stdout.splitlines() if l.endswith("exact")]) == 17
