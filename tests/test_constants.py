"""CPU: coefficients of the format that the device code and the oracle each
write out are the same decimal, not only the same binary32 value."""
import re
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_dc_smoothing_coefficients():
    """src/codec/dc_smoothing.cpp's side and corner weights."""
    device = (ROOT / "gjxl_amd" / "csrc" / "aq.hip").read_text()
    oracle = (ROOT / "oracle" / "aq.c").read_text()
    number = r"(\d+\.\d+)f"
    found = re.findall(rf"kSide = {number}, kCorner = {number}", device)
    assert len(found) == 1
    assert found == re.findall(rf"side = {number}, corner = {number}", oracle)
