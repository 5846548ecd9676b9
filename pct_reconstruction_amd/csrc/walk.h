// walk.h — the voxel walk along a straight line with a z slope (take_3D_step_GPU, DS.cu:11392; the same steps
// in find_MLP_endpoints_GPU :7581), one axis per step.
//
// A step moves along the axis whose next voxel edge is nearest along the line, and forms the position on the
// other two axes from the position on that one and the line's slopes.  The edge in front of a lane is kept for
// each axis, as the value that edge_coordinate_GPU (:11322) gives: the position of a step and both distances that
// it leaves are then one operation away, and only the moved axis' edge is formed again.  Every value is the one of
// the step's own formulas, operation by operation, and none is accumulated: a state follows from the voxel, the
// last axis and the line, so a walk can be taken up at any voxel of it.
#pragma once
#include "devmath.h"

struct Walk3 {
    // the line: start, slopes, directions
    double xs, ys, zs;
    double dy_dx, dz_dx, dz_dy, dx_dy, dx_dz, dy_dz;
    int xm, ym, zm;
    int ax, ay, az, at;  // what a step along each axis adds to the address `at`; the caller's to set
    // the state: voxel, distances to the next edges, those edges as multiples of the voxel size, their coordinates
    int vx, vy, vz;
    double xt, yt, zt;
    int kx, ky, kz;
    double ex, ey, ez;
    double passed;  // the edge passed by the last step

    __device__ __forceinline__ void edges(const DevGeom& g)
    {
        const int nx = vx + xm, ny = vy - ym, nz = vz - zm;  // next voxels
        kx = xm == PCT_X_INC ? nx : nx + 1;
        ky = -(ym == PCT_Y_INC ? ny : ny + 1);
        kz = -(zm == PCT_Z_INC ? nz : nz + 1);
        ex = g.X0 + kx * g.VW;
        ey = g.Y0 + ky * g.VH;
        ez = g.Z0 + kz * g.VT;
    }
    // the state at the line's start
    __device__ __forceinline__ void begin(const DevGeom& g)
    {
        edges(g);
        xt = fabs(ex - xs);
        yt = fabs(ey - ys);
        zt = fabs(ez - zs);
    }
    // the state after a step along `axis` (0 x, 1 y, 2 z) into the current voxel; bit k of `full`: the distance on
    // axis k was zero and became the whole voxel
    __device__ __forceinline__ void resume(const DevGeom& g, int axis, int full)
    {
        edges(g);
        // the edge that was passed is one voxel behind the next one
        if (axis == 0) move_x(g, g.X0 + (kx - xm) * g.VW);
        else if (axis == 1) move_y(g, g.Y0 + (ky - ym) * g.VH);
        else move_z(g, g.Z0 + (kz - zm) * g.VT);
        if (full & 1) xt = g.VW;
        if (full & 2) yt = g.VH;
        if (full & 4) zt = g.VT;
    }
    // the distances once an edge at p was passed
    __device__ __forceinline__ void move_x(const DevGeom& g, double p)
    {
        passed = p;
        const double d = p - xs;
        xt = g.VW;
        yt = fabs(ey - (dy_dx * d + ys));
        zt = fabs(ez - (dz_dx * d + zs));
    }
    __device__ __forceinline__ void move_y(const DevGeom& g, double p)
    {
        passed = p;
        const double d = p - ys;
        xt = fabs(ex - (dx_dy * d + xs));
        yt = g.VH;
        zt = fabs(ez - (dz_dy * d + zs));
    }
    __device__ __forceinline__ void move_z(const DevGeom& g, double p)
    {
        passed = p;
        const double d = p - zs;
        xt = fabs(ex - (dx_dz * d + xs));
        yt = fabs(ey - (dy_dz * d + ys));
        zt = g.VT;
    }
    // the position after a step along `axis`
    __device__ __forceinline__ void position(int axis, double* x, double* y, double* z) const
    {
        if (axis == 0) {
            *x = passed;
            *y = dy_dx * (passed - xs) + ys;
            *z = dz_dx * (passed - xs) + zs;
        } else if (axis == 1) {
            *x = dx_dy * (passed - ys) + xs;
            *y = passed;
            *z = dz_dy * (passed - ys) + zs;
        } else {
            *x = dx_dz * (passed - zs) + xs;
            *y = dy_dz * (passed - zs) + ys;
            *z = passed;
        }
    }
    // One step; the axis moved along.  *full as in resume, *clamped: the z voxel fell below 0 and stays at 0
    // (`at` is then for the caller to set).
    __device__ __forceinline__ int step(const DevGeom& g, int* full, bool* clamped)
    {
        const double x_ext = fabs(dz_dx) * xt, y_ext = fabs(dz_dy) * yt;
        int axis;
        if (zt <= x_ext && zt <= y_ext) {
            const double p = ez;
            vz -= zm;
            kz += zm;
            at += az;
            ez = g.Z0 + kz * g.VT;
            move_z(g, p);
            axis = 2;
        } else if (x_ext <= y_ext) {
            const double p = ex;
            vx += xm;
            kx += xm;
            at += ax;
            ex = g.X0 + kx * g.VW;
            move_x(g, p);
            axis = 0;
        } else {
            const double p = ey;
            vy -= ym;
            ky += ym;
            at += ay;
            ey = g.Y0 + ky * g.VH;
            move_y(g, p);
            axis = 1;
        }
        *full = 0;
        *clamped = false;
        if (xt == 0 || yt == 0 || zt == 0 || vz < 0) {  // rare
            if (xt == 0) { xt = g.VW; vx += xm; at += ax; *full |= 1; }
            if (yt == 0) { yt = g.VH; vy -= ym; at += ay; *full |= 2; }
            if (zt == 0) { zt = g.VT; vz -= zm; at += az; *full |= 4; }
            if (vz < 0) { vz = 0; *clamped = true; }
            edges(g);
        }
        return axis;
    }
};
