"""CPU replay of the narrow passes (tests/emu/narrow_emu.cpp): transforms at every ring size they serve and the
key switch's fused stages, over prime sizes, digit counts, permutations and addends, against the oracle, with
every LDS access checked for a race."""
import subprocess

from test_emu import _build


def test_replay_of_the_narrow_passes_equals_the_oracle():
    r = subprocess.run([_build("narrow_emu")], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "EMU OK" in r.stdout
    assert len([l for l in r.stdout.splitlines() if l.endswith("narrow passes exact")]) == 5
