import ctypes


def tiles_run(bh):
    """Launches of the matrix products whose tile an estimate picks, by tile."""
    n = bh.buddy_hip_tile_report(None, 0)
    buf = ctypes.create_string_buffer(n)
    bh.buddy_hip_tile_report(buf, n)
    return {name: int(hits) for name, hits in
            (line.split("\t") for line in buf.value.decode().splitlines())}
