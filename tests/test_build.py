"""The device code as the compiler's own machine verifier sees it (no GPU)."""
from resolve2d_amd import build


def test_machine_verifier_passes(tmp_path):
    refused = build.verify(str(tmp_path))
    assert not refused, [(src, err[-2000:]) for src, err in refused]
