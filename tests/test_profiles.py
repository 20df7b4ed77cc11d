"""The committed rocprof traffic summaries (profiles/traffic_*.json) belong to
the kernel sources in the tree: each lists the files it was measured on with
their SHA-256, and every listed file still has that hash.  (bench.py reports
no rocprof traffic for a summary whose sources changed; this test makes the
change visible where it happens.)  The summaries that the bench and the
documents use are there."""

import glob
import hashlib
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# what bench.py reports of its kernels, and the tables in the documents
REQUIRED = [f"traffic_{kernel}_C{config}.json" for config in (3, 4, 5)
            for kernel in ("forward", "backward", "scene_prep")] + [
    "traffic_render_C3.json", "traffic_certify_C3.json", "traffic_batch_gather_fetch.json"]


def test_summaries_are_there():
    for name in REQUIRED:
        assert os.path.exists(os.path.join(ROOT, "profiles", name)), name


def test_documents_name_profiles_that_exist():
    import re

    for doc in ("DESIGN.md", "README.md"):
        with open(os.path.join(ROOT, doc)) as f:
            for name in set(re.findall(r"profiles/([A-Za-z0-9_]+\.(?:json|md))", f.read())):
                assert os.path.exists(os.path.join(ROOT, "profiles", name)), (doc, name)


def test_traffic_summaries_match_the_sources():
    paths = sorted(glob.glob(os.path.join(ROOT, "profiles", "traffic_*.json")))
    assert paths
    for path in paths:
        with open(path) as f:
            c = json.load(f)
        name = os.path.basename(path)
        assert c.get("sources"), f"{name} lists no sources"
        assert c.get("hbm_bytes_per_launch", 0) > 0, name
        for rel, sha in c["sources"].items():
            with open(os.path.join(ROOT, rel), "rb") as f:
                got = hashlib.sha256(f.read()).hexdigest()
            assert got == sha, f"{name}: {rel} changed since it was profiled"
