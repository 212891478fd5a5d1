"""The benchmark's times by operation count every call that a part makes into the kernel library."""
import glob
import os
import re
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402

# what parts ask the library without a launch
QUESTIONS = {"attention_long_col_tiles", "attention_long_span_tile", "attention_tokens_per_tile", "check_attention_sizes", "fixed_decay_chunk", "gated_kind",
             "latent_attention_on_matrix_cores", "latent_tile_tokens", "pack_gate_up", "plain_kind", "rope_in_launch"}


def test_every_operation_of_a_part_has_its_cost():
    called = set()
    for path in glob.glob(os.path.join(ROOT, "yalis_amd", "parts", "*.py")):
        with open(path) as f:
            called |= set(re.findall(r"\bops\.(\w+)\(", f.read()))
    assert "linear" in called
    assert called - QUESTIONS <= set(bench._op_costs(None, None))


def test_a_product_with_its_activation_costs_what_the_product_does():
    costs = bench._op_costs(None, None)
    x, w = torch.empty(300, 64, dtype=torch.bfloat16), torch.empty(128, 64, dtype=torch.bfloat16)
    y = torch.empty(300, 128, dtype=torch.bfloat16)
    assert costs["linear_act"]((x, w, "silu", y.dtype), {}, y) == costs["linear"]((x, w, y.dtype), {}, y)
    assert costs["linear_act"]((x, w, "silu", y.dtype), {}, y)[0] == 2.0 * 300 * 128 * 64
