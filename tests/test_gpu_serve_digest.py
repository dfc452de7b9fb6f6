"""The served requests' digest at row lengths around the 16 lanes that share a row, and at particle counts that leave
part of a workgroup without a row: the same 64-bit sum as on the host over a plain pipeline's keys, counts and rows."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def mix64(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def host_digest(keys, counts, rows):
    n, ngmax = rows.shape
    i = np.arange(n, dtype=np.uint64)
    with np.errstate(over="ignore"):
        total = np.sum(mix64(i * np.uint64(0x9E3779B97F4A7C15) ^ keys), dtype=np.uint64)
        total += np.sum(mix64((i << np.uint64(32)) | counts.astype(np.uint64)), dtype=np.uint64)
        k = np.arange(ngmax, dtype=np.uint64)[None, :]
        d = mix64((rows.astype(np.uint64) << np.uint64(20)) ^ (k << np.uint64(52)) ^ i[:, None])
        total += np.sum(np.where(k < counts[:, None], d, np.uint64(0)), dtype=np.uint64)
    return int(total)


@pytest.mark.parametrize("n,ngmax", [(1, 1), (15, 15), (17, 16), (1000, 17), (4097, 31), (5000, 150)])
def test_digest_row_lengths(hip, n, ngmax):
    print(f"digest n {n} ngmax {ngmax}", flush=True)
    rng = np.random.RandomState(n)
    p = [rng.uniform(-1, 1, n).astype(np.float32) for _ in range(3)]
    p.append(np.full(n, 0.5 * (60.0 / n) ** (1.0 / 3.0), np.float32))
    req = {"id": 0, "cloud": 0, "kind": hip.SERVE_BUILD, "n": n, "arrival_s": 0.0, "seed": 1,
           **dict(zip("xyzh", p))}
    res, _ = hip.serve_run([req], slots=1, ngmax=ngmax, realtime=False, digests=True)
    pipe = hip.Pipeline(curve=hip.HILBERT, key_bits=64, real_bits=32, bucket_size=64, ngmax=ngmax)
    nb, nc = hip.DeviceArray(n * ngmax, np.uint32), hip.DeviceArray(n, np.uint32)
    pipe.sync(*[hip.DeviceArray.from_numpy(a) for a in p], n, hip.make_box(-1.0, 1.0, np.float32), full_build=True,
              neighbors=nb, counts=nc)
    assert res[0]["digest"] == host_digest(pipe.arrays()["keys"], nc.download(), nb.download().reshape(n, ngmax))
