"""Batched geometric and bi-objective tracking (the lockstep launches, and a
workgroup per pair for many small ones) against the single-pair tracker and
the oracle, on a mixed-size batch (160x120 .. 640x480), and against each other.

- The batch's keyframe and current clouds of every level equal the FP32
  oracle's bit for bit.
- The coarsest level's ICP selection count and Student-t variance, formed
  under the initial pose before any update, equal the oracle's bit for bit.
- Every pair's tracked pose agrees with the single-pair tracker and with the
  FP32 oracle tracker, both started from the same pose, within 1e-5 rad /
  1e-2 mm; the error against the FP64 oracle is printed."""
import numpy as np
import pytest

import oracle
from recon_amd import BIOBJECTIVE, GEOMETRIC, synth
from recon_amd.hip import DeviceBuffer
from recon_amd.tracker import BatchTracker, PhotoTracker

pytestmark = pytest.mark.gpu

SIZES = [(160, 120), (320, 240), (480, 360), (640, 480)]
ITERS = (1, 3, 10, 5)
N = 8192


def _pairs(n, seed):
    out = []
    for i in range(n):
        W, H = SIZES[i % 4]
        g0, d0, g1, d1, Tgt = synth.make_pair(seed + i, W, H, 3.0, 50.0)
        init = synth.sample_motion(seed * 5 + i, 1.0, 15.0) @ Tgt
        bufs = [DeviceBuffer.from_array(a) for a in (g0, d0, g1, d1)]
        out.append(dict(ref_gray=bufs[0].ptr, ref_depth=bufs[1].ptr, cur_gray=bufs[2].ptr, cur_depth=bufs[3].ptr,
                        width=W, height=H, calib=synth.calib_block_np(W, H), host=(g0, d0, g1, d1), bufs=bufs,
                        init=init, gt=Tgt))
    return out


@pytest.mark.parametrize("mode", [BIOBJECTIVE, GEOMETRIC])
def test_batch_icp_matches_single_and_oracle(mode):
    print(f"case batch icp mode {mode}", flush=True)
    pairs = _pairs(8, 1200 + 10 * mode)
    bt = BatchTracker(len(pairs), 640, 480, mode=mode, n_select=N, iters=ITERS, lam=0.5)
    Trel, _, rms, st = bt.track(pairs, init=[p["init"] for p in pairs])
    assert np.all(st == 0)
    from tests._oracle_steps import Steps
    for i, p in enumerate(pairs):
        W, H = p["width"], p["height"]
        L = 4 if W == 640 else 3
        g0, d0, g1, d1 = p["host"]
        # clouds of every level, bit for bit
        stp = Steps(W, H, L, p["calib"], g0, d0, g1, d1, nselect=N, dtype=np.float32)
        stp.clouds()
        for l in range(L):
            nl = (W >> l) * (H >> l)
            rc = bt.debug_read(i, "REF_CLOUD", l, np.float32, 8 * nl)
            pos, nrm = rc[:4 * nl].reshape(nl, 4), rc[4 * nl:].reshape(nl, 4)
            R = stp.rpts[l].reshape(nl, 6)
            assert np.array_equal(pos[:, :3], R[:, :3]) and np.array_equal(nrm[:, :3], R[:, 3:]), (i, l)
            assert np.array_equal(pos[:, 3] != 0, stp.rmask[l].astype(bool)), (i, l)
            cp = bt.debug_read(i, "CUR_CLOUD", l, np.float32, 4 * nl).reshape(nl, 4)
            C = stp.cpts[l].reshape(nl, 6)
            assert np.array_equal(cp[:, :3], C[:, :3]) and np.array_equal(cp[:, 3] != 0, stp.cmask[l].astype(bool))
        # the coarsest level's selection under the initial pose, bit for bit
        o = stp.icp_select(L - 1, p["init"].astype(np.float32))
        cnt = bt.debug_read(i, "ICP_COUNT", 0, np.int32, 4)
        var = bt.debug_read(i, "ICP_VAR", L - 1, np.float32, 3)
        assert cnt[L - 1] == o["n"], (i, cnt, o["n"])
        assert var[2] / np.float32(o["n"]) == o["sigma2"], (i, var, o["sigma2"])
        # poses: single-pair tracker and the oracles from the same start
        tr = PhotoTracker(W, H, p["calib"], mode=mode, n_select=N, iters=ITERS, lam=0.5)
        tr.set_reference_points(g0, d0, mode=mode, lam=0.5, force=True)
        tr.set_current_image(g1, d1)
        tr.track_from(np.linalg.inv(p["init"]))
        Ts = tr.trel().astype(np.float64)
        tr.close()
        res = {}
        for dt in (np.float32, np.float64):
            ot = oracle.Tracker(W, H, p["calib"], mode=mode, levels=L, iters=ITERS, nselect=N, lam=0.5, dtype=dt)
            ot.set_reference(g0, d0); ot.set_current(g1, d1); ot.prepare(); ot.set_trel(p["init"]); ot.track()
            res[dt] = ot.poses()[0]
        es = synth.pose_error(Trel[i], Ts)
        e32 = synth.pose_error(Trel[i], res[np.float32])
        e64 = synth.pose_error(Trel[i], res[np.float64])
        et = synth.pose_error(Trel[i], p["gt"])
        print(f"  pair {i} {W}x{H}: vs single {es[0]:.2e} deg {es[1]:.2e} mm; vs FP32 oracle {e32[0]:.2e} deg "
              f"{e32[1]:.2e} mm; vs FP64 oracle {e64[0]:.2e} deg {e64[1]:.2e} mm; vs truth {et[0]:.3f} deg "
              f"{et[1]:.2f} mm; ICP points {list(cnt[:L])}", flush=True)
        assert np.radians(es[0]) < 1e-5 and es[1] < 1e-2, i
        assert np.radians(e32[0]) < 1e-5 and e32[1] < 1e-2, i
    bt.close()


def _variant(mode):
    import ctypes
    from recon_amd import lib
    info, v = (ctypes.c_int * 6)(), 0
    while lib().rt_batch_variant_info(v, info) == 0 and info[5] != mode:
        v += 1
    return v


@pytest.mark.parametrize("mode,N,iters", [(BIOBJECTIVE, 8192, ITERS), (BIOBJECTIVE, 256, (2, 0, 3, 1)),
                                          (GEOMETRIC, 8192, ITERS), (GEOMETRIC, 2048, (0, 1, 0, 2)),
                                          (BIOBJECTIVE, 2048, (0, 0, 0, 0))])
def test_lockstep_equals_the_persistent_kernel(mode, N, iters, monkeypatch):
    """The geometric modes' two ways, a launch per pass over all pairs and a
    workgroup per pair, take the same sums in the same order: the same poses,
    RMS, counts and variances bit for bit, on mixed sizes."""
    print(f"case batch icp ways mode {mode} N {N} iters {iters}", flush=True)
    pairs = _pairs(5, 1500)
    res = []
    for force in (None, _variant(mode)):
        monkeypatch.delenv("RT_BATCH_VARIANT", raising=False)
        if force is not None:
            monkeypatch.setenv("RT_BATCH_VARIANT", str(force))
        bt = BatchTracker(len(pairs), 640, 480, mode=mode, n_select=N, iters=iters, lam=0.5)
        out = list(bt.track(pairs, init=[p["init"] for p in pairs]))
        out += list(bt.retrack(init=out[0].reshape(-1, 16), n=len(pairs)))
        for i, p in enumerate(pairs):
            L = 4 if p["width"] == 640 else 3
            for l in range(L):
                if iters[L - 1 - l]:
                    out.append(bt.debug_read(i, "ICP_COUNT", 0, np.int32, 4)[l:l + 1])
                    out.append(bt.debug_read(i, "ICP_VAR", l, np.float32, 3))
        bt.close()
        res.append(out)
    for x, y in zip(*res):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("mode,W,H,n", [(GEOMETRIC, 160, 120, 200), (BIOBJECTIVE, 160, 120, 200), (BIOBJECTIVE, 224, 168, 260)])
def test_many_small_pairs_equal_few(mode, W, H, n):
    """Batches past the line to a workgroup per pair against the same pairs in
    a batch before it."""
    print(f"case batch icp many {n} {W}x{H} mode {mode}", flush=True)
    kinds, pairs, keep = 4, [], []
    for i in range(kinds):
        g0, d0, g1, d1, Tgt = synth.make_pair(1600 + i, W, H, 3.0, 50.0)
        bufs = [DeviceBuffer.from_array(a) for a in (g0, d0, g1, d1)]
        keep.append(bufs)
        pairs.append(dict(ref_gray=bufs[0].ptr, ref_depth=bufs[1].ptr, cur_gray=bufs[2].ptr, cur_depth=bufs[3].ptr,
                          width=W, height=H, calib=synth.calib_block_np(W, H)))
    few = BatchTracker(kinds, W, H, mode=mode, n_select=2048, iters=ITERS, lam=0.5).track(pairs)
    many = BatchTracker(n, W, H, mode=mode, n_select=2048, iters=ITERS, lam=0.5).track([pairs[i % kinds] for i in range(n)])
    for x, y in zip(few, many):
        for i in range(n):
            assert np.array_equal(x[i % kinds], y[i]), i


@pytest.mark.parametrize("mode,W,H,L,N", [(GEOMETRIC, 904, 580, 3, 2048), (BIOBJECTIVE, 904, 580, 3, 8192),
                                          (BIOBJECTIVE, 320, 240, 3, 16384), (BIOBJECTIVE, 192, 144, 2, 256),
                                          (GEOMETRIC, 192, 144, 1, 256)])
def test_batch_icp_at_the_ends_of_its_sizes(mode, W, H, L, N):
    """The most pixels of a pair (513 blocks of 1024), more points than a
    round's 8192, few points and levels: three pairs against the FP32 oracle
    from the same start."""
    print(f"case batch icp mode {mode} {W}x{H} levels {L} N {N}", flush=True)
    iters = (2, 4, 3, 0)
    pairs, host = [], []
    for i in range(3):
        g0, d0, g1, d1, Tgt = synth.make_pair(1400 + i, W, H, 3.0, 50.0)
        bufs = [DeviceBuffer.from_array(a) for a in (g0, d0, g1, d1)]
        host.append((g0, d0, g1, d1, bufs, synth.sample_motion(7000 + i, 1.0, 15.0) @ Tgt))
        pairs.append(dict(ref_gray=bufs[0].ptr, ref_depth=bufs[1].ptr, cur_gray=bufs[2].ptr, cur_depth=bufs[3].ptr,
                          width=W, height=H, calib=synth.calib_block_np(W, H)))
    bt = BatchTracker(3, W, H, mode=mode, n_select=N, iters=iters, lam=0.5, levels=L)
    Trel, _, rms, st = bt.track(pairs, init=[h[5] for h in host])
    assert np.all(st == 0)
    for i, (g0, d0, g1, d1, _, init) in enumerate(host):
        ot = oracle.Tracker(W, H, pairs[i]["calib"], mode=mode, levels=L, iters=iters, nselect=N, lam=0.5, dtype=np.float32)
        ot.set_reference(g0, d0); ot.set_current(g1, d1); ot.prepare(); ot.set_trel(init); ot.track()
        e = synth.pose_error(Trel[i], ot.poses()[0])
        print(f"  pair {i}: vs FP32 oracle {e[0]:.2e} deg {e[1]:.2e} mm", flush=True)
        assert np.radians(e[0]) < 1e-5 and e[1] < 1e-2, i
    bt.close()


@pytest.mark.parametrize("mode,iters", [(BIOBJECTIVE, (-1, 3, 2, 1)), (GEOMETRIC, (2, -7, 1, -1)),
                                        (GEOMETRIC, (-1, -1, -1, -1))])
def test_negative_iteration_counts_are_levels_without_iterations(mode, iters):
    print(f"case batch icp mode {mode} iters {iters}", flush=True)
    pairs = _pairs(4, 1300)
    res = []
    for it in (iters, [max(0, k) for k in iters]):
        bt = BatchTracker(len(pairs), 640, 480, mode=mode, n_select=2048, iters=it, lam=0.5)
        res.append(bt.track(pairs, init=[p["init"] for p in pairs]))
        bt.close()
    for x, y in zip(*res):
        assert np.array_equal(x, y)
