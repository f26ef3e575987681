"""What bench.py prints: one line on stdout, short enough for a reader of the last few kilobytes of a log."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_one_short_line(capsys):
    record = {"metric": "m", "value": 1.0, "config": {"workload": "w"}, "roofline": {"note": "n" * 1700}}
    others = [dict(record, metric=f"form {i}") for i in range(2)], [dict(record, metric=f"workload {i}") for i in range(7)]
    bench.report(dict(record, other_forms=others[0], secondary=others[1]))
    out, err = capsys.readouterr()
    assert out.count("\n") == 1 and len(out) < 4096 and json.loads(out) == record
    assert [json.loads(line) for line in err.splitlines()] == [{"other_forms": o} for o in others[0]] + [{"secondary": o} for o in others[1]]
