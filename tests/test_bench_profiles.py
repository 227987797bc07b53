"""The profile summaries that bench.py quotes are there, with the keys it reads."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_profile_value_has_its_file():
    with open(os.path.join(ROOT, "bench.py")) as f:
        named = re.findall(r'profile_value\(\s*"([^"]+)",\s*"([^"]+)"\)', f.read())
    assert named
    for name, key in named:
        with open(os.path.join(ROOT, "profiles", name)) as f:
            assert any(re.match(key + r" = \d", line) for line in f), (name, key)
