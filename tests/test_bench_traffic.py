"""bench.py reports counted HBM traffic only where the committed counters are of
the present k_step: the figure of a kernel that is gone belongs to no kernel."""
import bench


def _profile(monkeypatch, tmp_path, text):
    f = tmp_path / "traffic.md"
    f.write_text(text)
    monkeypatch.setattr(bench, "TRAFFIC_PROFILE", str(f))


def test_traffic_of_the_present_kernel(monkeypatch, tmp_path):
    _profile(monkeypatch, tmp_path,
             f"text\n\ntraffic_bytes_per_launch: 123456789\ntraffic_kernel: {bench.k_step_fingerprint()}\n")
    assert bench.measured_traffic(512) == 123456789
    assert bench.measured_traffic(256) is None


def test_no_traffic_of_another_kernel(monkeypatch, tmp_path):
    for text in ("traffic_bytes_per_launch: 355697667\n",
                 "traffic_bytes_per_launch: 355697667\ntraffic_kernel: 0123456789abcdef\n"):
        _profile(monkeypatch, tmp_path, text)
        assert bench.measured_traffic(512) is None
    monkeypatch.setattr(bench, "TRAFFIC_PROFILE", str(tmp_path / "none.md"))
    assert bench.measured_traffic(512) is None


def test_fingerprint_follows_the_code_alone(monkeypatch, tmp_path):
    import os
    src = open(os.path.join(bench.ROOT, "ipglasma_amd", "csrc", "kernels_evolve.hip")).read()
    d = tmp_path / "ipglasma_amd" / "csrc"
    d.mkdir(parents=True)
    want = bench.k_step_fingerprint()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    a = src.index("void k_step(")
    for text, same in ((src, True), (src[:a] + src[a:].replace("{", "{  // a comment\n", 1), True),
                       (src[:a] + src[a:].replace("{", "{ if (it < 0) return;", 1), False)):
        (d / "kernels_evolve.hip").write_text(text)
        assert (bench.k_step_fingerprint() == want) is same
