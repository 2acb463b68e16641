"""build() compiles before the package is imported: importing it loads the libraries (CPU)."""

import subprocess
import sys

from tests.conftest import ROOT


def test_builder_leaves_the_package_unloaded():
    code = ("import sys, __graft_entry__ as entry\n"
            "builder = entry._builder()\n"
            "assert 'hilberta_amd' not in sys.modules\n"
            "assert str(builder.LIB).startswith(entry.ROOT) and builder.CSRC.is_dir()\n")
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True)
