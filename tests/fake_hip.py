"""libzen_hip.so on a HIP runtime without a device (fake_hip.cpp), in a process of its own: run as
`fake_hip.py FAKE LIBRARY`, calls are read as lines of JSON ([name, fail_at, arguments]) and answered with
[return code, log].  An argument is a number, null, or a list of numbers that stands for the address of such int64s;
"host" is the address of the thread's answer words."""
import ctypes
import json
import sys


def main():
    fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    fake.fake_log.restype = ctypes.c_char_p
    L = ctypes.CDLL(sys.argv[2])
    words = (ctypes.c_int64 * 4096)()
    for line in sys.stdin:
        name, fail_at, args = json.loads(line)
        keep, given = [], []
        for a in args:
            if isinstance(a, list):
                keep.append((ctypes.c_int64 * len(a))(*a))
                a = ctypes.addressof(keep[-1])
            elif a == "host":
                a = ctypes.addressof(words)
            given.append(ctypes.c_void_p(a))  # every argument takes a 64-bit register or stack slot
        fake.fake_reset(fail_at)
        rc = getattr(L, name)(*given)
        print(json.dumps([rc, fake.fake_log().decode().splitlines()]), flush=True)


if __name__ == "__main__":
    main()
