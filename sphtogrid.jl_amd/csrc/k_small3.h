// k_small3.h -- index arithmetic of the windowed 3D small scatter, in plain
// C++ so that it can be checked on the host.
#pragma once

namespace s2g {

// 3D: footprint box side <= 8 voxels goes to the scatter path.
constexpr int kSmallSide3D = 8;
// side of the windowed 3D scatter's tiles
constexpr int kST3 = 9;
// its LDS window, the tile and the largest box; strides with one voxel of
// padding against bank conflicts
constexpr int kSW3 = kST3 + kSmallSide3D - 1;
constexpr int kSW3y = kSW3 + 1, kSW3x = kSW3 * kSW3y;

// Of a box of iw x jw x kw voxels, iw, jw, kw <= kSmallSide3D: a wave's 64
// lanes take R = small3_planes(jw kw) x planes of jw x kw voxels per step.
constexpr int small3_planes(int jk)
{
    const int r = (int)(64.5f * (1.0f / (float)jk));
    return r < kSmallSide3D ? r : kSmallSide3D;
}

// Lane ln's voxel of step 0: (ri, dj, dk) of the box; at step st it has (ri +
// st R, dj, dk), which is a voxel of the box while st R < left.  A lane past
// the R planes (left 0) or past the box's last plane has none, and deposits
// nothing whatever the particle's scale: its weight is 0, but 0 times an
// infinite scale is not.
struct Small3Lane {
    int ri, dj, dk, left;
};
constexpr Small3Lane small3_lane(int ln, int iw, int jw, int kw)
{
    const int jk = jw * kw;
    const int ri = (int)(((float)ln + 0.5f) * (1.0f / (float)jk)), rem = ln - ri * jk;
    const int dj = (int)(((float)rem + 0.5f) * (1.0f / (float)kw));
    return Small3Lane{ri, dj, rem - dj * kw, ri < small3_planes(jk) ? iw - ri : 0};
}

}  // namespace s2g
