"""The words workgroups of the decode loop wait for (csrc/exchange_word.h): a producer never stores the empty
pattern, whatever NaN it computed, and nothing but the empty pattern reads as empty.  A word that did would
hold the loop until its 2 s limit.  Host only; the driver goes through every NaN."""
import os
import subprocess

from conftest import ROOT


def test_filled_and_empty_over_every_nan():
    exe = os.path.join(ROOT, "tests", "cpp", "exchange_word")
    assert os.path.exists(exe), f"{exe} missing: run __graft_entry__.build()"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout) > 2 * (1 << 23)


def test_every_store_of_a_waited_for_word_is_filled():
    """Stores to hx and ppx in the device code take filled() values or empty4()."""
    with open(os.path.join(ROOT, "parakeet.cpp_amd", "csrc", "pk_device.h")) as f:
        src = f.read()
    stores = []
    for head in ("st_coh(p.hx", "st4_coh(B.hx", "st4_coh(B.ppx"):
        at = src.find(head)
        while at >= 0:
            stores.append(src[at:src.index(";", at)])
            at = src.find(head, at + 1)
    # h of layer 0, h of the later layers, the new prediction output and the emptied old one, the copy
    # from the slots and the other half it empties, the emptied h
    assert len(stores) == 7, stores
    for st in stores:
        assert "empty4()" in st or st.count("filled(") in (1, 4), st
