"""CPU: bench.py's counter summary finds the evaluations and comparisons of a
run in its dispatches, as the path launches them now."""
import re
from pathlib import Path

import pytest

import bench

ROOT = Path(__file__).resolve().parents[1]

FRONT = ["SrgbKernel", "OpsinDynamicsKernel", "BlurKernel<16, 512, LowPlanes, 3>", "MaskKernel",
         "Symmetric5Kernel", "InitialCflKernel", "CandidateCostKernel<5>", "SearchKernel",
         "ResetStatsKernel", "AnchorLayoutKernel", "AnchorDctKernel"]
SELECTION = {"small": ["QuantizerKernel"], "large": ["SelectPassKernel"] * 6 + ["RawQuantKernel"]}
CODE = ["FinalCflKernel", "CodeTransformKernel"]
DECODE = ["DcQuantKernel", "BlockFieldsKernel", "ReconstructKernel", "LoopFilterKernel<true>"]
COMPARE = ["OpsinDynamicsKernel"] + ["BlurKernel<16, 512, LowPlanes, 3>"] * 4 + [
    "DifferencesKernel<false>", "ComposeKernel"]
TOKENS = ["FillKernel", "FillWordsKernel", "AnchorLayoutKernel", "FrameStatisticsKernel",
          "TokenCountKernel", "TokenEmitKernel"]


def _mixed(a, b):
    """b's dispatches among a's, as two streams' are."""
    out = []
    for i, name in enumerate(a):
        out.append(name)
        out += b[i::len(a)]
    return out


@pytest.mark.parametrize("size", ["small", "large"])
def test_stage_dispatches(size):
    evaluate = SELECTION[size] + CODE + DECODE
    update = ["ReduceKernel", "AqUpdateKernel"]
    image = FRONT + (evaluate + COMPARE + update) * 2 + SELECTION[size] + CODE + _mixed(
        DECODE + COMPARE, TOKENS) + ["ReduceKernel"]
    names = [f"void gjxl_amd::(anonymous namespace)::{n}(Args)" for n in image * 2]
    spans = bench._stage_dispatches(names)
    bare = [(image * 2)[i] for i in range(len(names))]
    assert [[bare[i] for i in s] for s in spans["aq_evaluate"]] == [evaluate] * 6
    assert [[bare[i] for i in s] for s in spans["butteraugli_compare"]] == [COMPARE] * 6


def test_stage_kernels_exist():
    """Every kernel that the summary looks for is one that the library has."""
    sources = "\n".join(p.read_text() for p in (ROOT / "gjxl_amd" / "csrc").glob("*.hip"))
    kernels = set(re.findall(r"__global__[^;{]*?void\s+(\w+Kernel)\s*\(", sources))
    wanted = {k for names in bench.STAGE_KERNELS.values() for k in names}
    assert wanted | set(bench.TRAFFIC_KERNELS) <= kernels


def test_stages_are_whole():
    """Every kernel that an evaluation or a comparison launches is counted."""
    csrc = ROOT / "gjxl_amd" / "csrc"

    def launched(path, *functions):
        text = (csrc / path).read_text()
        out = set()
        for f in functions:
            body = text[re.search(rf"^GJXLResult {f}\(", text, re.M).start():]
            body = body[:re.search(r"^}", body, re.M).start()]
            out |= set(re.findall(r"hipLaunchKernelGGL\(\(?(\w+)", body))
        return out

    evaluate = launched("aq.hip", "LaunchQuantizer", "LaunchFinalCfl", "LaunchCodeCoefficients",
                        "LaunchReconstruct") | launched("filters.hip", "LaunchLoopFiltersAndColor")
    compare = launched("butteraugli.hip", "Psycho", "MaskActivity", "Differences",
                       "ButteraugliCompare")
    assert evaluate == set(bench.STAGE_KERNELS["aq_evaluate"])
    assert compare == set(bench.STAGE_KERNELS["butteraugli_compare"])
