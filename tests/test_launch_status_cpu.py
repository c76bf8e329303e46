"""A launcher clears the error it returns, so a caller that drops it reports success with nothing computed: every call of
one in the library's sources keeps the status."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "v.1.1_amd" / "csrc"


def test_every_launch_status_is_kept():
    calls = 0
    for path in sorted(CSRC.glob("*.hip")):
        for number, line in enumerate(path.read_text().splitlines(), 1):
            for m in re.finditer(r"mpsk::launch_\w+\(", line):
                calls += 1
                before = line[:m.start()].rstrip()
                assert before.endswith("=") or re.search(r"(\breturn|CHK\(\w+,)$", before), f"{path.name}:{number}: {line.strip()}"
    assert calls > 20
