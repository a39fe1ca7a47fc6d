"""Tuned values per thread and lines per column tile (no GPU)."""
import fftz


def test_tuned_widths_are_used():
    """Tuned values per thread and lines per column tile override the rules for rows of
    256 threads and for whole-LDS tiles in complex128."""
    fftz.tune_clear()
    try:
        assert fftz.tune_parse("p8:0:0:0:0|4095,1,1;|1024,4095,4095; 0 0 0 0 e=8\n") == 1
        assert fftz.plan_json([(4095, 1, 1)], [(1024, 4095, 4095)], "d")["launches"][0]["TL"] == 512
        assert fftz.tune_parse("p8:0:0:0:0|1024,100,100;|100,1,1;20,102400,102400; 0 8 0 0\n") == 1
        geo = [(1024, 100, 100)], [(100, 1, 1), (20, 102400, 102400)]
        assert fftz.plan_json(*geo, "d")["launches"][0]["C"] == 8
    finally:
        fftz.tune_clear()
