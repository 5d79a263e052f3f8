"""Host-side bounds model of the batched path, on the CPU.

The library's own descriptor builder (rt_batch_layout: the code rt_batch_prepare
runs, reporting offsets instead of touching a device) places every pair's
buffers in the arena, and rt_batch_lock_layout places the lockstep launches'
arrays; this model replays the launch grids of the preparation and tracking
launches (launch_prep, launch_track, launch_lockstep in rt_batch.hip) for them
and forms the indices the kernels form, from their code, asserting that each
lies inside its buffer. It runs on the 256-pair mixed-size batch of
the mixed-size workload (160x120 .. 640x480, 8192 points), the 4096-pair
640x480 batch of the headline and small mixed batches."""
import ctypes

import numpy as np
import pytest

from recon_amd import RtPair, lib
from recon_amd.tracker import default_params

SIZES = [(160, 120), (320, 240), (480, 360), (640, 480)]
FIELDS = 40
BINS_TILE_H = 32
NW_BINS = ((64 + 8) // 4) * (BINS_TILE_H + 4)   # words of the kb_bins tile (TWW * TH)


def _align(x):
    return (x + 255) & ~255


def _layout(sizes, N, max_w=640, max_h=480, mode=1):
    n = len(sizes)
    arr = (RtPair * n)()
    cal = np.zeros(96, np.float32)
    cal[43], cal[45], cal[47], cal[48], cal[62], cal[63] = -525.0, 319.5, 525.0, 239.5, 500.0, 4000.0
    cal[26:42] = np.eye(4, dtype=np.float32).ravel()
    cal[64:80] = np.eye(4, dtype=np.float32).ravel()
    cal[0:9] = cal[43:52]
    for i, (W, H) in enumerate(sizes):
        # frame pointers are never dereferenced by the layout: distinct dummies
        arr[i].ref_gray, arr[i].ref_depth = 0x1000 + 16 * i, 0x2000 + 16 * i
        arr[i].cur_gray, arr[i].cur_depth = 0x3000 + 16 * i, 0x4000 + 16 * i
        arr[i].width, arr[i].height = W, H
        arr[i].calib = cal.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
    f = np.zeros(n * FIELDS, np.int64)
    order = np.zeros(n, np.int32)
    maxes = np.zeros(3, np.int32)
    prm = default_params(n_select=N, mode=mode)
    rc = lib().rt_batch_layout(ctypes.byref(prm), max_w, max_h, n, arr, f.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                               order.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                               maxes.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
    assert rc == 0, lib().rt_last_error()
    return f.reshape(n, FIELDS), order, maxes


def _buffers(p, max_w, max_h):
    """{name: (offset, bytes)} of one pair's arena buffers, sized by what the
    kernels may address: the level images by the pair's own size, the other
    buffers by their slots."""
    W, H, L, N = (int(x) for x in p[:4])
    b = {}
    for f in range(2):
        for l in range(1, 4):
            o = int(p[4 + l + 3 * f])
            if l < L:
                b[f"gray{f}_{l}"] = (o, (W >> l) * (H >> l) * 4)
            else:
                assert o == -1
    b["bins"] = (int(p[11]), W * H)
    b["zblk"] = (int(p[37]), W * ((H + 7) // 8 * 8) * 2)
    b["ghist"] = (int(p[12]), 256 * 4)
    b["sel"] = (int(p[13]), N * 4)
    b["pts"] = (int(p[14]), N * 16)
    for l in range(4):
        b[f"jac{l}"] = (int(p[15 + l]), N * 28)
    if p[21] >= 0:   # geometric buffers, sized by the pair's own levels
        for l in range(4):
            nl = (W >> l) * (H >> l)
            for k, name in enumerate(("rpos", "rnrm", "cpos")):
                b[f"{name}{l}"] = (int(p[21 + 3 * l + k]), nl * 16)
        b["isel"] = (int(p[33]), W * H * 4)
        b["ir2"] = (int(p[34]), W * H * 4)
        b["icnt"] = (int(p[35]), 16)
        b["ivar"] = (int(p[36]), 48)
        assert p[36] == p[35] + 16
    else:
        assert np.all(p[21:37] == -1)
    return b


def _check_layout(f, order, maxes, max_w, max_h, N, icp=False):
    n = len(f)
    slot = int(f[0, 20])
    npx = max_w * max_h
    want = 2 * _align(npx * 4 // 3 + 64) + _align(npx) + _align(max_w * ((max_h + 7) // 8 * 8) * 2) + \
        _align(1024) + _align(N * 4) + _align(N * 16) + 4 * _align(N * 28)
    if icp:
        want += sum(3 * _align((npx >> (2 * l)) * 16) for l in range(4)) + 2 * _align(npx * 4) + _align(64)
    assert slot == want
    assert sorted(order.tolist()) == list(range(n))         # the work queue hands out every pair once
    assert maxes[0] == f[:, 0].max() and maxes[1] == f[:, 1].max() and maxes[2] == f[:, 3].max()
    for i in range(n):
        p = f[i]
        assert p[19] == i * slot and p[20] == slot
        bufs = sorted(_buffers(p, max_w, max_h).values())
        for (o, sz) in bufs:
            assert p[19] <= o and o + sz <= p[19] + slot, (i, o, sz)
        for (o1, s1), (o2, s2) in zip(bufs, bufs[1:]):
            assert o1 + s1 <= o2, (i, o1, s1, o2)                # disjoint


def _kb_pyramid(W, H, L, maxW, maxH):
    """kb_pyramid / convert_pyramid_block<3>: 16x16 threads of 4x4 pixels per
    64x64 block; largest element index of each access, per buffer."""
    bx, by, t = np.meshgrid(np.arange((maxW + 63) // 64), np.arange((maxH + 63) // 64), np.arange(256), indexing="ij")
    live = (bx * 64 < W) & (by * 64 < H)
    tx, ty = t & 15, t >> 4
    x0, y0 = (bx * 16 + tx) * 4, (by * 16 + ty) * 4
    inside = live & (x0 < W) & (y0 < H)
    x0, y0 = x0[inside], y0[inside]
    out = {"g8": ((y0 + 3) * W + x0 + 3).max()}                  # uchar4 rows y0..y0+3
    if L > 1:
        out["gray_1"] = ((y0 // 2 + 1) * (W >> 1) + x0 // 2 + 1).max()
    if L > 2:
        out["gray_2"] = ((y0 // 4) * (W >> 2) + x0 // 4).max()
    if L > 3:
        ev = ((t & 15)[inside] % 2 == 0) & ((t >> 4)[inside] % 2 == 0)
        out["gray_3"] = ((y0[ev] // 8) * (W >> 3) + x0[ev] // 8).max()
        assert ((t & 15)[inside][ev] + 1).max() <= 15 and ((t >> 4)[inside][ev] + 1).max() <= 15  # l2tile[16][17]
    # the current frame's depth copy into 8x8 blocks and the network's inputs:
    # 4 threads per 8x8 cell, two columns each, columns clamped to px <= W - 2,
    # rows one by one to <= H - 1; block rows stored while below H
    assert W % 8 == 0
    cell, part = t[live] >> 2, t[live] & 3
    cx = bx[live] * 8 + (cell & 7)
    cy = by[live] * 8 + (cell >> 3)
    px = np.minimum(cx * 8 + 2 * part, W - 2)
    rows = np.minimum(cy[:, None] * 8 + np.arange(8)[None, :], H - 1)
    out["g8_feat"] = (rows.max(axis=1) * W + px + 1).max()        # two gray bytes
    out["d16_feat"] = (rows.max(axis=1) * W + px + 1).max()       # two depths
    # LDS assembly: word cell * 32 + 4r + part of 64 * 32; stores: thread t writes
    # words w .. w + 7 (w = 8 (t % 32)) of cell row t // 32, as two 16-byte stores
    lds = (t[live] >> 2)[:, None] * 32 + 4 * np.arange(8)[None, :] + (t[live] & 3)[:, None]
    assert lds.max() < 64 * 32
    tt = t[live]
    w = (tt & 31) * 8
    bcx, bcy = bx[live] * 8 + (w >> 5), by[live] * 8 + (tt >> 5)
    st = (bcx < W // 8) & (bcy < (H + 7) // 8)
    words = 32 * (bcy * (W // 8) + bcx) + (w & 31) + 7
    assert np.all(((32 * (bcy * (W // 8) + bcx) + (w & 31)) * 4) % 16 == 0)   # 16-byte aligned stores
    out["zblk_words"] = words[st].max()
    if W % 8 == 0 and H % 8 == 0:
        ok = (cx < W // 8) & (cy < H // 8)
        out["feat"] = (4 * (cy[ok] * (W // 8) + cx[ok]) + 3).max()    # channels 2, 3
    return out


def _kb_bins(W, H, maxW, maxH):
    """kb_bins: 64 x BINS_TILE_H tiles, lane = column, BINS_TILE_H / 4 rows
    per wave; the clamped depth and gray-word loads, the bin writes, the LDS
    tile and the keyframe pyramid levels built from it."""
    bx, by = np.meshgrid(np.arange((maxW + 63) // 64), np.arange((maxH + BINS_TILE_H - 1) // BINS_TILE_H),
                         indexing="ij")
    live = (bx * 64 < W) & (by * BINS_TILE_H < H)
    bx, by = bx[live], by[live]
    lane = np.arange(64)
    x = (bx[:, None] * 64 + lane[None, :]).ravel()
    yb = by[:, None].repeat(64, 1).ravel() * BINS_TILE_H
    out = {}
    xc = np.minimum(x, W - 1)
    ys = np.concatenate([yb + r for r in range(BINS_TILE_H)])
    out["d16"] = (np.tile(xc, BINS_TILE_H) + np.minimum(ys, H - 1) * W).max()
    e = np.arange(NW_BINS)
    gx = (bx[:, None] * 64 - 4) + 4 * (e[None, :] % ((64 + 8) // 4))
    gy = (by[:, None] * BINS_TILE_H - 2) + e[None, :] // ((64 + 8) // 4)
    o = np.clip(gx, 0, W - 4) + np.clip(gy, 0, H - 1) * W
    out["g8_words"] = (o + 3).max()
    xs = np.tile(x, BINS_TILE_H)
    keep = (xs < W) & (ys < H)
    out["bins"] = (xs[keep] + ys[keep] * W).max()
    # taps of the gradient: in_bounds keeps the projected point in
    # [10, W - 10) x [10, H - 10); the taps are xdi - 1 .. xdi + 2, ydi - 1 .. ydi + 2
    out["gray_taps"] = (H - 11 + 2) * W + (W - 11 + 2)
    # keyframe pyramid: level-1 value (i, j) averages tile entries rows
    # 2 + 2j .. 3 + 2j, columns 4 + 2i .. 5 + 2i of the (64 + 8) x (T + 4) tile
    T = BINS_TILE_H
    j1, i1 = np.meshgrid(np.arange(T // 2), np.arange(32), indexing="ij")
    assert (3 + 2 * j1).max() < T + 4 and (5 + 2 * i1).max() < 64 + 8
    for lq, (nx, ny) in enumerate([(32, T // 2), (16, T // 4), (8, T // 8)], start=1):
        X = (bx[:, None] * nx + np.arange(nx)[None, :]).ravel()
        Y = (by[:, None] * ny + np.arange(ny)[None, :]).ravel()
        Xg, Yg = np.meshgrid(X, Y, indexing="ij")
        ok = (Xg < (W >> lq)) & (Yg < (H >> lq))
        if ok.any():
            out[f"gray_{lq}"] = (Xg[ok] + Yg[ok] * (W >> lq)).max()
    return out


SEL_WAVES, SEL_U = 8, 2


def _select_parts(n):
    parts = 1
    while parts < 16 and 2 * parts * n <= 2048:
        parts *= 2
    return parts


def _kb_select(W, H, N, n):
    npix = W * H
    Pn = npix // 512
    assert Pn >= 1 and (Pn * 512) <= npix
    # the segments that the workgroups of a pair count and scatter: each of the
    # 512 once (wave + 16 k + 8 u inside a workgroup's range)
    parts = _select_parts(n)
    per = 512 // parts
    g, wave, k, u = np.meshgrid(np.arange(parts), np.arange(SEL_WAVES), np.arange(0, per, SEL_WAVES * SEL_U),
                                np.arange(SEL_U), indexing="ij")
    live = wave + k < per                                   # the loops' condition, before u is added
    seg = (per * g + wave + k + SEL_WAVES * u)[live]
    assert np.array_equal(np.sort(seg), np.arange(512))
    # packed counts: both below 2^16; split, they wait in the pair's points (512 words)
    assert Pn < 1 << 16
    out = {"counts": 4 * 511 + 3 if parts > 1 else -1}
    # last byte a segment load may touch: clamped to the segment's last byte
    # (byte path) or an 8-byte load at min(base, end - 8) (only when Pn % 8 == 0)
    last = 512 * Pn - 1
    if Pn % 8 == 0:
        assert Pn >= 8
    out.update(bins=last, sel=N - 1)
    return out


def _ref_points_blocks(n, chunks):
    """kb_ref_points' XCD-aware grid: workgroup b -> (pair, chunk), pairs of
    one XCD (b % 8) together; returns the (pair, chunk) of every live block."""
    b = np.arange(8 * ((n + 7) // 8) * chunks)
    k = b >> 3
    pair, chunk = (b & 7) + 8 * (k // chunks), k % chunks
    assert np.all(pair % 8 == b % 8)
    live = pair < n
    return pair[live], chunk[live]


@pytest.mark.parametrize("n", [1, 2, 64, 128, 129, 256, 257, 512, 513, 1024, 1025, 4096])
def test_selection_splits_cover_each_segment_once(n):
    """Any number of pairs, at the fewest points (whose records hold the counts)."""
    assert _kb_select(160, 120, 256, n)["counts"] < 16 * 256


@pytest.mark.parametrize("n,chunks", [(1, 1), (3, 32), (8, 32), (13, 7), (4096, 32), (257, 5)])
def test_ref_points_grid_covers_each_chunk_once(n, chunks):
    pair, chunk = _ref_points_blocks(n, chunks)
    key = pair * chunks + chunk
    assert key.size == n * chunks and np.array_equal(np.sort(key), np.arange(n * chunks))


def _kb_ref_points(W, H, L, N):
    out = {"sel": N - 1, "pts": N - 1, "jac_bytes": 28 * N - 1}
    for lq in range(1, L):
        out[f"gray_{lq}"] = (W >> lq) * (H >> lq) - 1         # taps clamped into the level image
    return out


def _kb_track(W, H, L, N, maxN, pc):
    out = {}
    for layer in range(L):
        wl, hl = W >> layer, H >> layer
        # bilinear taps at xdi .. xdi + 1, ydi .. ydi + 1 with 0 <= xdi < wl - 1, 0 <= ydi < hl - 1
        out[f"img_{layer}"] = (wl - 2) + (hl - 2) * wl + 1 + wl
        assert out[f"img_{layer}"] <= wl * hl - 1
    # the depth tap reads the current depth map in 8x8 blocks (kb_pyramid's copy):
    # pixel (x, y) at ((y // 8) * (W // 8) + x // 8) * 64 + (y % 8) * 8 + x % 8, 0 <= x < W, 0 <= y < H
    x, y = np.meshgrid(np.arange(W), np.arange(H), indexing="ij")
    blk = ((y // 8) * (W // 8) + x // 8) * 64 + (y % 8) * 8 + x % 8
    out["zblk_tap"] = blk.max()
    assert np.unique(blk).size == W * H                  # a distinct element per pixel
    assert N <= maxN                                     # LDS residuals: maxN entries
    assert min(N, pc) <= min(maxN, pc)                   # point cache: min(maxN, capacity) entries
    return out


def _geometric(W, H, L):
    """kb_clouds and the ICP terms: largest element index per buffer (float4
    clouds, isel / ir2)."""
    out = {}
    # kb_clouds: 16x16 pixel tiles; the normal's four neighbours only for
    # 1 <= x <= W - 2, 1 <= y <= H - 2
    out["depth"] = max((W - 1) + (H - 1) * W, (W - 2 + 1) + (H - 2) * W, (W - 2) + (H - 2 + 1) * W)
    out["cloud0"] = W * H - 1
    # cloud_tile_levels: level l of a tile from level l - 1 in LDS (256 + 64 + 16
    # + 4 records), stored inside the level's image; a pixel's four taps lie in
    # the tile and, the sizes being multiples of 2^(L-1), in the image
    src, dst = 0, 256
    for l in range(1, L):
        Wl, Hl, side = W >> l, H >> l, 16 >> l
        assert (W >> (l - 1)) == 2 * Wl and (H >> (l - 1)) == 2 * Hl
        t = np.arange(side * side)
        x, y = t & (side - 1), t // side
        o = src + 2 * x + 4 * y * side
        taps = np.stack([o, o + 1, o + 2 * side, o + 2 * side + 1])
        assert taps.min() >= src and taps.max() < dst and np.unique(taps).size == 4 * t.size
        assert dst + t.max() < 256 + 64 + 16 + 4
        gx = (np.arange((W + 15) // 16)[:, None] * side + np.arange(side)[None, :]).ravel()
        gy = (np.arange((H + 15) // 16)[:, None] * side + np.arange(side)[None, :]).ravel()
        gx, gy = gx[gx < Wl], gy[gy < Hl]
        assert np.array_equal(gx, np.arange(Wl)) and np.array_equal(gy, np.arange(Hl))     # every pixel once
        out[f"level{l}"] = (gx.max() + gy.max() * Wl, Wl * Hl - 1)
        src, dst = dst, dst + side * side
    for l in range(L):
        w, h = W >> l, H >> l
        # mask / system taps: 0 <= xdi < w - 1, 0 <= ydi < h - 1, taps o2 .. o2 + w + 1
        out[f"taps{l}"] = ((w - 2) + (h - 2) * w + w + 1, w * h - 1)
        out[f"isel{l}"] = (w * h - 1, W * H - 1)               # at most w*h selected points
        assert w * h < 1 << 28                                 # 32-bit byte offsets of the records (ldo)
    return out


def _check_kernels(f, maxes, max_w, max_h, pcs=(0, 5120, 5632, 8192)):
    maxW, maxH, maxN = (int(x) for x in maxes)
    for p in {tuple(int(v) for v in r[:4]) for r in f}:
        W, H, L, N = p
        bufsz = {"g8": W * H, "d16": W * H, "bins": W * H, "sel": N, "pts": N}
        for l in range(1, L):
            bufsz[f"gray_{l}"] = (W >> l) * (H >> l)
        bufsz.update(g8_feat=W * H, d16_feat=W * H, feat=4 * (W // 8) * (H // 8),
                     zblk_words=W * ((H + 7) // 8 * 8) // 2)
        pyr = _kb_pyramid(W, H, L, maxW, maxH)
        for k, v in pyr.items():
            assert v < bufsz[k], (p, "kb_pyramid", k, v)
        bins = _kb_bins(W, H, maxW, maxH)
        assert bins["d16"] < W * H and bins["g8_words"] < W * H and bins["bins"] < W * H
        assert bins["gray_taps"] < W * H
        for k, v in bins.items():
            if k.startswith("gray_") and k != "gray_taps" and int(k[5:]) < L:
                assert v < bufsz[k], (p, "kb_bins", k, v)
        sel = _kb_select(W, H, N, len(f))
        assert sel["bins"] < W * H and sel["sel"] < N and sel["counts"] < 16 * N
        ref = _kb_ref_points(W, H, L, N)
        for k, v in ref.items():
            if k.startswith("gray_"):
                assert v < bufsz[k]
        assert ref["jac_bytes"] < 28 * N
        for pc in pcs:
            tr = _kb_track(W, H, L, N, maxN, pc)
            assert tr["zblk_tap"] < W * ((H + 7) // 8 * 8)
            for layer in range(1, L):
                assert tr[f"img_{layer}"] < bufsz[f"gray_{layer}"]
            assert tr["img_0"] < W * H
        if f[0, 21] >= 0:
            g = _geometric(W, H, L)
            assert g["depth"] < W * H and g["cloud0"] < W * H
            for k, v in g.items():
                if isinstance(v, tuple):
                    assert v[0] <= v[1], (p, k, v)


def _lock_layout(max_w, max_h, N, mode):
    off = np.zeros(10, np.int64)
    prm = default_params(n_select=N, mode=mode)
    assert lib().rt_batch_lock_layout(ctypes.byref(prm), max_w, max_h,
                                      off.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))) == 0
    names = ("wsum", "hist", "cnt", "bsum0", "bsum1", "bsum2", "rz", "bits", "rfull", "end")
    return dict(zip(names, (int(v) for v in off)))


def _check_lockstep(W, H, L, N, off, mode):
    """Largest byte that the kl_* launches touch in each of a pair's arrays,
    against the start of the next one."""
    names = list(off)
    end = {a: off[b] for a, b in zip(names, names[1:])}
    used = {"wsum": 4 * (512 + 32 * 15 + 31), "hist": 4 * (256 + 255), "rz": 8 * (N - 1) + 4}
    if mode != 1:
        for layer in range(L):
            npix = (W >> layer) * (H >> layer)
            blocks = (npix + 1023) // 1024              # kl_icp_mask, kl_icp_compact: one per 1024 pixels
            assert blocks <= 1024                       # wave_student_total's reach, and cnt[t], t < g
            used["cnt"] = max(used.get("cnt", 0), 4 * (blocks - 1))
            used["bits"] = max(used.get("bits", 0), 8 * (16 * (blocks - 1) + 15))   # the words of every wave
            used["rfull"] = max(used.get("rfull", 0), 4 * (npix - 1))
            for r in range(3):                          # a block sum per 1024 of at most npix points
                used[f"bsum{r}"] = max(used.get(f"bsum{r}", 0), 4 * (blocks - 1))
    # kl_terms' grid is kb_ref_points': _ref_points_blocks' test covers it
    for k, last in used.items():
        elem = 8 if k == "bits" else 4
        assert off[k] % (8 if k in ("bits", "rz") else 4) == 0
        assert off[k] + last + elem <= end[k], (W, H, L, N, k, last, off[k], end[k])


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("W,H,levels", [(160, 120, 0), (640, 480, 0), (904, 580, 3), (1024, 512, 4), (656, 799 // 8 * 8, 4),
                                        (32, 32, 1)])
def test_lockstep_launches_stay_in_bounds(W, H, levels, mode):
    """Up to the most pixels that a preparation admits (524,799: 904x580 is
    513 blocks of 1024), each array's last element lies before the next one."""
    N = min(8192, W * H // 2 // 256 * 256)
    L = levels or (4 if W == 640 else 3)
    prm = default_params(n_select=N, mode=mode, levels=levels)
    f, order, maxes = np.zeros(FIELDS, np.int64), np.zeros(1, np.int32), np.zeros(3, np.int32)
    cal = np.ones(96, np.float32)
    p = RtPair(ref_gray=0x1000, ref_depth=0x2000, cur_gray=0x3000, cur_depth=0x4000, width=W, height=H,
               calib=cal.ctypes.data_as(ctypes.POINTER(ctypes.c_float)))
    assert lib().rt_batch_layout(ctypes.byref(prm), W, H, 1, ctypes.byref(p),
                                 f.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                                 order.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                 maxes.ctypes.data_as(ctypes.POINTER(ctypes.c_int))) == 0
    _check_lockstep(W, H, L, N, _lock_layout(W, H, N, mode), mode)


def _mixed_256():
    """The mixed-size workload's 256 pairs: sizes drawn by rng(3)."""
    rng = np.random.default_rng(3)
    return [SIZES[k] for k in rng.integers(0, 4, 256)]


@pytest.mark.parametrize("name,sizes,N,mode", [
    ("mixed 256 pairs", _mixed_256(), 8192, 1),
    ("640x480 x 4096", [(640, 480)] * 4096, 8192, 1),
    ("mixed 8 pairs", SIZES * 2, 2048, 1),
    ("mixed 6 pairs 12288", [(320, 240), (480, 360), (640, 480)] * 2, 12288, 1),
    ("mixed 64 pairs bi-objective", SIZES * 16, 8192, 2),
    ("mixed 8 pairs geometric", SIZES * 2, 2048, 0),
])
def test_batch_launches_stay_in_bounds(name, sizes, N, mode):
    f, order, maxes = _layout(sizes, N, mode=mode)
    _check_layout(f, order, maxes, 640, 480, N, icp=mode != 1)
    _check_kernels(f, maxes, 640, 480)


def test_layout_rejects_what_the_kernels_cannot_take():
    """Sizes the kernels' indexing does not cover are refused at preparation."""
    for sizes, N in ([[(648, 480)], 2048], [[(100, 120)], 2048], [[(160, 120)], 16384], [[(20, 20)], 256]):
        f = np.zeros(FIELDS, np.int64)
        n = len(sizes)
        arr = (RtPair * n)()
        cal = np.zeros(96, np.float32)
        for i, (W, H) in enumerate(sizes):
            arr[i].ref_gray = arr[i].ref_depth = arr[i].cur_gray = arr[i].cur_depth = 0x1000
            arr[i].width, arr[i].height = W, H
            arr[i].calib = cal.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
        order = np.zeros(n, np.int32)
        maxes = np.zeros(3, np.int32)
        prm = default_params(n_select=N, mode=1)
        rc = lib().rt_batch_layout(ctypes.byref(prm), 640, 480, n, arr, f.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                                   order.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                   maxes.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
        assert rc == -1, (sizes, N)
