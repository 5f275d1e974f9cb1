"""CPU replay of the row passes with their LDS exchanges ordered inside one wave of 64 threads only
(tests/emu/wave_emu.cpp), and the same replay with waves of 32 as a planted mistake that it has to catch."""
import subprocess

import pytest

from test_emu import _build


@pytest.fixture(scope="module")
def wave_bin():
    return _build("wave_emu")


def test_row_exchanges_stay_inside_one_wave(wave_bin):
    r = subprocess.run([wave_bin], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "EMU OK" in r.stdout
    assert len([x for x in r.stdout.splitlines() if x.endswith("row exchanges inside one wave")]) == 10


def test_exchanges_across_waves_are_caught(wave_bin):
    r = subprocess.run([wave_bin, "32"], capture_output=True, text=True, timeout=300)
    assert r.returncode != 0 and "LDS slot shared by two waves" in r.stderr
