"""The build collects its compilers' output without waiting on them: more
sources than compilers at a time, each printing more than a pipe holds."""
import subprocess
import sys


def test_compilers_that_print_much_do_not_block(tmp_path):
    cc = tmp_path / "cc"
    # as a compiler: 256 KB of warnings, then the object or library after -o
    cc.write_text("#!/bin/sh\nhead -c 262144 /dev/zero | tr '\\0' 'w'\n"
                  'while [ "$1" != -o ]; do shift; done\n: > "$2"\n')
    cc.chmod(0o755)
    code = ("import sys\nfrom aiimage_amd import build as b\n"
            "b.HERE, b.LIB, b.hipcc = sys.argv[1], sys.argv[1] + '/lib.so', lambda: sys.argv[1] + '/cc'\n"
            "assert len(b.SOURCES) > 4\nb.build(verbose=False, jobs=4)\n")
    subprocess.run([sys.executable, "-c", code, str(tmp_path)], check=True, timeout=100,
                   stdout=subprocess.DEVNULL)
    assert (tmp_path / "lib.so").exists()
