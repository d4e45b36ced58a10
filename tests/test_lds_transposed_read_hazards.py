"""The hand-placed transposing LDS reads of the weight gradient (ds_read_b64_tr_b16) follow the protocol of the
ds_read_b128 ones: no instruction touches a destination between a read and the wait that covers it, nothing is in flight
at a loop edge.  The checker of those reads runs on the same assembly with the other mnemonic in its place."""
import os
import re
import subprocess

import test_lds_read_hazards as H


def _functions():
    subprocess.run(["make", "-C", H.CSRC, "isa"], check=True, stdout=subprocess.DEVNULL)
    current = None
    with open(os.path.join(H.CSRC, "build", "conv_igemm.s")) as f:
        for no, raw in enumerate(f, 1):
            m = re.match(r"^(_Z\w+):\s*(;.*)?$", raw)
            if m:
                name, current = m.group(1), []
            elif raw.startswith(".Lfunc_end") and current is not None:
                yield name, current
                current = None
            elif current is not None:
                current.append((no, raw))


def test_weight_gradient_reads():
    kernels, problems, total = 0, [], 0
    for name, lines in _functions():
        if "wgrad" not in name or not any("ds_read_b64_tr_b16" in raw for _, raw in lines):
            continue
        seen, bad = H.check_function(name, [(no, raw.replace("ds_read_b64_tr_b16", "ds_read_b128")) for no, raw in lines])
        kernels, total = kernels + 1, total + seen
        problems += bad
    assert kernels >= 10 and total >= 1000, (kernels, total)
    assert not problems, "\n".join(problems[:20])
