"""The schedules that the size rules choose, against the explicit gather-GEMM oracle, on both sides of their lines: ragged channel
counts and row counts around the tiles' edges, for every tile shape and K split that the rules answer with."""
import pytest
import torch

from flexgemm_amd.workloads import reference_test_shell
from test_gpu_conv import _run_and_check, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype, res, ci, co", [
    (torch.float32, 8, 24, 40), (torch.float32, 24, 320, 96), (torch.float32, 32, 33, 512), (torch.float32, 64, 96, 24), (torch.float32, 100, 7, 33),
    (torch.float16, 16, 80, 200), (torch.bfloat16, 16, 300, 136), (torch.float16, 32, 320, 16), (torch.bfloat16, 40, 40, 72),
    (torch.float16, 8, 768, 256), (torch.bfloat16, 32, 768, 256), (torch.float16, 40, 72, 512), (torch.bfloat16, 24, 256, 768), (torch.float16, 48, 24, 384), (torch.bfloat16, 60, 128, 96), (torch.float16, 64, 264, 56), (torch.float16, 100, 48, 24), (torch.bfloat16, 100, 40, 200),
])
def test_rule_schedules_match_oracle(gpu_device, dtype, res, ci, co):
    coords = reference_test_shell(res)
    shape = torch.Size([1, ci, res, res, res])
    _say(f"rule schedule res={res} {ci}->{co} {dtype}")
    _run_and_check(coords, shape, ci, co, dtype, gpu_device, seed=res + ci)
