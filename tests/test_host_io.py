"""The host-buffer calls' host code on a stand-in for the HIP runtime
(fake_hip.cpp; no GPU): a call whose results did not come back leaves the
caller's buffers as they were, and a call that is refused leaves nothing on
the stream."""
import pytest

import fake_hip


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return fake_hip.build(tmp_path_factory.mktemp("hip"))


@pytest.mark.parametrize("check", ["failed_copies", "refused_calls"])
def test_host_calls(runtime, check):
    assert fake_hip.run(runtime, "host_io_check.py", check) == "ok"
