"""Test set-up of the whole tree: a tests folder that comes without its built
clients (a checkout of its sources, or one put in the place of another) gets
them before the tests run."""
import os

ROOT = os.path.dirname(os.path.abspath(__file__))


def pytest_sessionstart(session):
    if hasattr(session.config, "workerinput"):  # a worker of another session
        return
    cpp = os.path.join(ROOT, "tests", "cpp")
    missing = [c for c in ("client", "client_asan") if not os.path.exists(os.path.join(cpp, c))]
    built = os.path.exists(os.path.join(ROOT, "mgpu_old_amd", "lib", "noalloc.o"))
    if missing and built and os.path.exists(os.path.join(cpp, "client.cpp")):
        import __graft_entry__
        __graft_entry__.build_clients()
