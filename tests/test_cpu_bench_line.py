"""The line that bench.py prints: short enough for a reader that keeps the last 8 KB of the output."""

from __future__ import annotations

import json

import bench


def _record() -> dict:
    engine = {k: 1234.567890123456 for k in bench.BRIEF_LEG[:-1]} | {f"counter_{i}": 1e9 / 7 for i in range(60)}
    plain = {"s_per_it": 0.123456789012345, "peak_device_bytes": 1 << 37, "s_per_it_rounds": [0.1] * 4}
    refused = {"skipped": "needs 172.9 GiB of pinned host memory per step (one pin per save), over the 55 GiB cap"}
    legs = {name: {"saves": 168, "none": plain, "engine": engine, "reference": refused}
            for name in ("A", "B", "BR", "AH", "A4", "B4", "B4R", "C5U", "C5P")}
    legs["AH"]["engine_hipdma"] = engine
    parity = {name: {mode: {k: 1.2345678901234567e-5 for k in ("loss_rel", "grad_rel", "worst_tensor_grad_rel")}
                     for mode in ("engine", "reference")} for name in ("A", "B", "B16")}
    micro = {k: 1234.567890123456 for k in bench.BRIEF_MICRO} | {f"counter_{i}": 1e9 / 7 for i in range(20)}
    return {"regimes": legs, "link": {"dma_d2h": 55.98}, "parity": parity, "micro": micro,
            "int8_gemm": {"shapes": {"qkvo": [1.0] * 300}, "block_ms": {"hip": 8.065}}}


def test_the_printed_detail_is_short_and_keeps_each_leg() -> None:
    record = _record()
    kept = bench.brief(record)
    # the line's other keys take 2 KB, most of it the two rooflines
    assert len(json.dumps(kept)) < 5500
    assert kept["regimes"].keys() == record["regimes"].keys()
    assert kept["regimes"]["B"]["engine"]["s_per_it"] == 1234.6
    assert kept["regimes"]["B"]["reference"] == record["regimes"]["B"]["reference"]
    assert kept["parity"] == record["parity"] and "shapes" not in kept["int8_gemm"]


def test_the_whole_record_goes_to_a_file(tmp_path) -> None:
    path = tmp_path / "new" / "detail.json"
    bench.write_detail(str(path), {"detail": _record()})
    assert json.loads(path.read_text())["detail"] == _record()
    bench.write_detail(str(tmp_path), {})  # a folder: said in the log, nothing raised
