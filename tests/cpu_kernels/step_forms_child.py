"""Child process of tests/test_whole_step.py: every form of tests/step_forms.py
on the host copy of the kernels (see replay.py), one JSON line per form."""

import json
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
sys.path.insert(0, os.path.dirname(HERE))

import replay  # noqa: E402
import step_forms  # noqa: E402


def main():
    replay.load()
    for arg in [a for a in sys.argv[1:] if not a.startswith("--")]:
        name, backend = arg.split("/")
        compare = step_forms.form_differences if "--half" in sys.argv else step_forms.differences
        if "--gradient" in sys.argv:
            compare = step_forms.gradient_differences
        bad = compare(replay.fdtd, name, backend)
        print(json.dumps({"form": arg, "bad": bad}), flush=True)


if __name__ == "__main__":
    main()
