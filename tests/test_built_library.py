"""The library that is loaded was built from the sources that are here."""
import glob
import hashlib
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_is_built_from_these_sources():
    # its build id is the digest of what the Makefile compiles, in the Makefile's order: a source that no longer compiles, or was
    # changed after the last build, leaves a library with another one
    pkg = os.path.join(ROOT, "grab-anns_amd")
    files = sorted(sum((glob.glob(os.path.join(pkg, "csrc", "*" + e)) for e in (".hip", ".cpp", ".hpp")), []))
    files += [os.path.join(ROOT, "include", "grab_anns.h"), os.path.join(pkg, "Makefile")]
    digest = hashlib.sha1(b"".join(open(f, "rb").read() for f in files)).digest()
    lib = open(os.path.join(pkg, "libgrab_anns.so"), "rb").read()
    note = b"\x14\x00\x00\x00\x03\x00\x00\x00GNU\x00"  # length of the id, NT_GNU_BUILD_ID, the owner's name
    at = lib.find(note)
    assert at >= 0 and lib[at + len(note):at + len(note) + 20] == digest, "run `make -C grab-anns_amd`"
