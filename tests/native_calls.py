"""Which entry points of the kernel libraries a call reaches."""
import contextlib


@contextlib.contextmanager
def counted(ops, module, *entries, defines=()):
    """The names of ``entries`` of ``module`` in the order in which ``ops`` calls them inside the block."""
    lib, calls = ops.lib(module, defines), []

    class Counted:
        def __getattr__(self, name):
            entry = getattr(lib, name)
            if name not in entries:
                return entry

            def call(*args):
                calls.append(name)
                return entry(*args)
            return call

    ops._libs[(module, defines)] = Counted()
    try:
        yield calls
    finally:
        ops._libs[(module, defines)] = lib
