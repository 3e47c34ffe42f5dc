// pm_mesh.h -- tile and sub-tile densities cut from one mesh of the whole
// image per resolution (pm_mesh.hip).
#pragma once
#include "pm.h"

namespace cube {

// The image's mesh at w mesh cells per coarse cell: n = nc w points per dim.
struct MeshGeo {
  int n, w, sh;  // sh: coordinate bits below the mesh cell (B - log2 w)
  int nc, nt, nnt, nte, ncb;
};
MeshGeo mesh_geo(const Geo& g, int w, int bits);
// Windows of whole coarse cells at w = 4 or 8 with a power-of-two scale.
bool pm_mesh_applies(const Geo& g, const PMLevel& L);

// Every physical particle into the image's mesh (n^3 floats).
void pm_mesh_deposit(int izipx, const MeshGeo& M, const void* xp, const int32_t* rhoc, const int64_t* cell_off,
                     float* mesh, float mass, hipStream_t s);
// The outermost layers of the windows: faces, 6 n^2 floats per box.
void pm_mesh_faces(int izipx, const MeshGeo& M, const PMLevel& L, const PMBox* boxes_dev, int nbox, const void* xp,
                   const int32_t* rhoc, const int64_t* cell_off, float* faces, float mass, hipStream_t s);
// A box's window in the image's mesh: its first point per axis, in [0, n).
int4 mesh_origin(const MeshGeo& M, const PMLevel& L, const PMBox& B);
// The windows (n points per dim, origins on the device) written out as cubes.
void pm_mesh_window(const MeshGeo& M, int n, const int4* org_dev, int nbox, const float* mesh, const float* faces,
                    float* out, hipStream_t s);
// *bad = 1 unless every buffer cell holds the coordinates of the physical
// cell it is the periodic image of, in the same order.
void mesh_check_images(int izipx, const Geo& g, const void* xp, const int32_t* rhoc, const int64_t* cell_off,
                       int32_t* bad, hipStream_t s);

}  // namespace cube
