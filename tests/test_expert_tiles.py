"""How a step's (token, choice) pairs are cut into row tiles, on both sides of every line."""
import types

import torch

from servelab_amd.kernels.recurrent_ops import ExpertMatrices, RecurrentOps


class Table(RecurrentOps):
    act_dtype = torch.bfloat16


def last_narrow(experts, ff, width, gated=True):
    """The most rows an expert may have on average for tiles of 16 rows."""
    w = ExpertMatrices(None, (experts, 2 * ff if gated else ff, width), True)
    rows = next(n for n in range(1, 200) if Table().expert_tile_rows(n * experts, w, gated) == 128) - 1
    assert Table().expert_tile_rows(rows * experts + experts - 1, w, gated) == 16
    return rows


def test_lines_of_the_row_tiles():
    assert last_narrow(64, 1024, 2048) == 11 and last_narrow(64, 1024, 2048, gated=False) == 11
    assert last_narrow(64, 1024, 2080) == 47                          # rows of 65 times 32 values
    assert last_narrow(4, 4096, 1024) == 95                           # few experts
    assert last_narrow(8, 1024, 4096) == 11 and last_narrow(8, 896, 4096) == 95       # 64 and 56 workgroups with a tile an expert
    assert last_narrow(8, 1024, 4128) == 47 and last_narrow(8, 896, 4128) == 95
    wide = ExpertMatrices(None, (64, 2048, 2048), True)
    assert type("Float", (Table,), {"act_dtype": torch.float32})().expert_tile_rows(1 << 20, wide) == 16


def test_the_part_asks_for_them():
    from servelab_amd.parts.routed import RoutedExperts
    part = RoutedExperts(64, 8, 2, 32)
    seen = []
    ops = types.SimpleNamespace(linear=lambda *a, **k: "logits", expert_tile_rows=lambda *a: seen.append(a) or 128,
                                route_tokens=lambda *a, **k: seen.append((a, k)), routed_experts=lambda *a: "rows")
    part.rt, part.w_router, part.b_router, part.w_gate_up, part.w_down = types.SimpleNamespace(ops=ops), None, None, "first", "down"
    assert part.forward(torch.zeros(5, 64)) == "rows"
    assert seen == [(10, "first", True), (("logits", 8, 2), {"tile_rows": 128})]
