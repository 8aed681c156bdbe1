// Device geometry shared by the FP64 and mixed-precision kernels: rotated pixel position,
// trilinear cell and interpolated model value, as slice_gen3d (dragonfly/src/model.c:11-59).
#pragma once

#include <cfloat>

#include "emc_common.h"
#include "emc_kernels.h"

namespace emc {

// ---- geometry ------------------------------------------------------------------------

// Rotated voxel position of a pixel and its trilinear cell, as slice_gen3d / slice_merge3d
// (dragonfly/src/model.c:19-45 and :184-207): p = R q + center, cell = trunc(p).
// Cell coordinates are 32-bit: truncation toward zero (v_cvt_i32_f64, which saturates far
// outside the grid, where the range test fails either way).
struct Cell {
    int x, y, z;
    double fx, fy, fz;
};

__device__ __forceinline__ bool locate(const double *rot, double q0, double q1, double q2,
                                       double center, long size, Cell &c) {
    double p0 = rot[0] * q0 + rot[1] * q1 + rot[2] * q2 + center;
    double p1 = rot[3] * q0 + rot[4] * q1 + rot[5] * q2 + center;
    double p2 = rot[6] * q0 + rot[7] * q1 + rot[8] * q2 + center;
    c.x = __double2int_rz(p0);
    c.y = __double2int_rz(p1);
    c.z = __double2int_rz(p2);
    const int hi = (int)size - 2;
    c.fx = p0 - c.x;
    c.fy = p1 - c.y;
    c.fz = p2 - c.z;
    // one unsigned comparison an axis (a negative cell is a large one); hi < 0: no cell
    return hi >= 0 && (unsigned)c.x <= (unsigned)hi && (unsigned)c.y <= (unsigned)hi && (unsigned)c.z <= (unsigned)hi;
}

// Two neighbouring voxels along z, read with one 16-byte load from any 8-byte boundary.
typedef double VoxelPair __attribute__((ext_vector_type(2), aligned(8)));

// Interpolated model value times corr, DBL_MIN outside the grid (model.c:35-57). No branch
// around the loads: a pixel outside the grid reads the corners of cell (0, 0, 0) and returns
// DBL_MIN, so the loads of several calls can be in flight at once. The reference wraps the far
// corner, (x + 1) % size, but cells stop at size - 2, so the wrap never happens: the far
// corners are at fixed distances from the near one and the two corners of each z edge are one
// 16-byte load (models have 3 voxels an axis or more, so those of cell (0, 0, 0) are inside). Without
// the three 64-bit remainders and four of the eight loads the FP64 expand of 25,680 orientations x 66,820
// pixels on 251^3 took 16.0 ms instead of 19.4.
__device__ __forceinline__ double slice_value(const double *__restrict__ model, long size,
                                              const double *rot, double q0, double q1, double q2,
                                              double corr, double center) {
    Cell c;
    const bool ok = locate(rot, q0, q1, q2, center, size, c);
    const int sz = (int)size;
    const long at = (long)(int)((unsigned)c.x * (unsigned)sz + (unsigned)c.y) * sz + c.z;
    const double *__restrict__ m = model + (ok ? at : 0);
    const long s2 = (long)sz * sz;
    const VoxelPair m00 = *(const VoxelPair *)m, m01 = *(const VoxelPair *)(m + sz);
    const VoxelPair m10 = *(const VoxelPair *)(m + s2), m11 = *(const VoxelPair *)(m + s2 + sz);
    const double cx = 1. - c.fx, cy = 1. - c.fy, cz = 1. - c.fz;
    const double fx = c.fx, fy = c.fy, fz = c.fz;
    const double v = cx * cy * cz * m00.x + cx * cy * fz * m00.y + cx * fy * cz * m01.x + cx * fy * fz * m01.y +
                     fx * cy * cz * m10.x + fx * cy * fz * m10.y + fx * fy * cz * m11.x + fx * fy * fz * m11.y;
    return ok ? v * corr : DBL_MIN;
}

// FP64 model copy in bricks of 4 x 4 x 4 trilinear cells: 16 rows (x % 4, y % 4) of the five voxels
// that four cells along z touch, 640 bytes a brick. A compact detector patch rotated into the
// volume touches a few whole lines of it at any orientation, where lines of 16 voxels along z give
// a patch across z one or two voxels each.
struct BrickLayout {
    int nb, nbz;  // bricks along x and y, and along z
    __host__ __device__ explicit BrickLayout(long size) : nb((int)((size + 3) / 4)), nbz((int)((size + 2) / 4)) {}
    static constexpr int kVoxels = 80;
    __host__ __device__ size_t elems() const { return (size_t)nb * nb * nbz * kVoxels; }
};

// slice_value from the brick copy: the same values and operations (a copy is below 2^31 elements).
__device__ __forceinline__ double slice_value(const BrickVoxel *__restrict__ model, long size, const double *rot,
                                              double q0, double q1, double q2, double corr, double center) {
    Cell c;
    const bool ok = locate(rot, q0, q1, q2, center, size, c);
    const BrickLayout b(size);
    const int x = ok ? (int)c.x : 0, y = ok ? (int)c.y : 0, z = ok ? (int)c.z : 0;
    const int row = b.nbz * BrickLayout::kVoxels, slab = b.nb * row;  // a brick further along y, along x
    const int at = (x >> 2) * slab + (y >> 2) * row + (z >> 2) * BrickLayout::kVoxels + (x & 3) * 20 + (y & 3) * 5 + (z & 3);
    const int dx = (x & 3) == 3 ? slab - 60 : 20, dy = (y & 3) == 3 ? row - 15 : 5;
    const double *__restrict__ m = &model->v;
    const VoxelPair m00 = *(const VoxelPair *)(m + (unsigned)at), m01 = *(const VoxelPair *)(m + (unsigned)(at + dy));
    const VoxelPair m10 = *(const VoxelPair *)(m + (unsigned)(at + dx)),
                    m11 = *(const VoxelPair *)(m + (unsigned)(at + dx + dy));
    const double cx = 1. - c.fx, cy = 1. - c.fy, cz = 1. - c.fz;
    const double fx = c.fx, fy = c.fy, fz = c.fz;
    const double v = cx * cy * cz * m00.x + cx * cy * fz * m00.y + cx * fy * cz * m01.x + cx * fy * fz * m01.y +
                     fx * cy * cz * m10.x + fx * cy * fz * m10.y + fx * fy * cz * m11.x + fx * fy * fz * m11.y;
    return ok ? v * corr : DBL_MIN;
}

// FP32 model copy in bricks of 4 x 4 x 4 trilinear cells: brick (X/4, Y/4, Z/4) of an nb^3
// grid (nb = (size - 2) / 4 + 1, the cells x <= size - 2 of the grid) holds the 5 x 5 x 5
// corners of its cells (shared faces are stored twice), padded to 128 floats, z fastest. The
// eight corners of any cell are then at fixed offsets {0, 1, 5, 6, 25, 26, 30, 31} from one
// address, all within the brick's 512 bytes: one index computation per interpolation, and a
// compact detector patch rotated into the volume at any orientation touches few cache lines.
constexpr int kModelBrick = 4;
constexpr int kHaloBrickFloats = 128;  // 5^3 = 125 corners, padded
__host__ __device__ __forceinline__ int model_bricks(long size) { return (int)((size - 2) / kModelBrick + 1); }
__device__ __forceinline__ long halo_index(int nb, int x, int y, int z) {
    return ((long)((x >> 2) * nb + (y >> 2)) * nb + (z >> 2)) * kHaloBrickFloats + ((x & 3) * 25 + (y & 3) * 5 + (z & 3));
}

// Interpolated value of the FP32 brick copy at the rotated position of a pixel times the
// pixel's corr, all in FP32: the position R q + center, the truncated cell (toward zero, as
// model.c:31-33) and its fractions, then the trilinear value as three rounds of linear
// interpolation (z, y, x), each a fused multiply-add a + f (b - a). rot: the rotation as 9
// floats; q: the pixel's q-vector in FP32. -inf outside the grid (x, y or z outside
// [0, size - 2]), where the reference takes DBL_MIN.
__device__ __forceinline__ float slice_value_f32h(const float *__restrict__ model, int size, int nb, const float *rot,
                                                  float q0, float q1, float q2, float corr, float center) {
    const float p0 = __builtin_fmaf(rot[0], q0, __builtin_fmaf(rot[1], q1, __builtin_fmaf(rot[2], q2, center)));
    const float p1 = __builtin_fmaf(rot[3], q0, __builtin_fmaf(rot[4], q1, __builtin_fmaf(rot[5], q2, center)));
    const float p2 = __builtin_fmaf(rot[6], q0, __builtin_fmaf(rot[7], q1, __builtin_fmaf(rot[8], q2, center)));
    const int x = (int)p0, y = (int)p1, z = (int)p2;  // truncation toward zero
    const int hi = size - 2;
    const bool ok = hi >= 0 && (unsigned)x <= (unsigned)hi && (unsigned)y <= (unsigned)hi && (unsigned)z <= (unsigned)hi;
    const float fx = p0 - (float)x, fy = p1 - (float)y, fz = p2 - (float)z;
    // the cell, not the index, is selected: a branch here would serialise the loads of a wave's values
    const float *b = model + halo_index(nb, ok ? x : 0, ok ? y : 0, ok ? z : 0);
    const float m000 = b[0], m001 = b[1], m010 = b[5], m011 = b[6];
    const float m100 = b[25], m101 = b[26], m110 = b[30], m111 = b[31];
    const float a00 = __builtin_fmaf(fz, m001 - m000, m000), a01 = __builtin_fmaf(fz, m011 - m010, m010);
    const float a10 = __builtin_fmaf(fz, m101 - m100, m100), a11 = __builtin_fmaf(fz, m111 - m110, m110);
    const float b0 = __builtin_fmaf(fy, a01 - a00, a00), b1 = __builtin_fmaf(fy, a11 - a10, a10);
    const float v = __builtin_fmaf(fx, b1 - b0, b0);
    return ok ? v * corr : -INFINITY;
}

}  // namespace emc
