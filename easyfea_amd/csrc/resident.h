// The plan of a resident solve (resident.hip), as include/efea.h describes it.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include "efea.h"

namespace efea {

typedef efea_resident_plan ResidentPlan;

int resident_shape(int dof_n, int max_neighbours, int min_passes, int* lanes, int* slots, int* passes);
int resident_fits(const ResidentPlan& P);
int resident_bisect(int Nn, const double* coord, int parts, int* order, int* part_ptr);
int resident_neighbours(int Nn, const int* node_ptr, const int* node_cols, int lanes, int slots, int passes, int nblk,
                        const int* rows, unsigned short* lidx, int* halo_ptr, int* halo_ex, int halo_room, int* pub,
                        int* pub_ptr, int* pub_pos, int* self, int* nex, int* max_halo);
size_t resident_workspace_bytes(int Nnode, int dof_n, const ResidentPlan& P);
int solve_resident(const ResidentPlan& P, int Nnode, const int* node_ptr, const double* vals,
                   const unsigned char* known, const double* Minv, const double* rel, const double* Ainv, int ld,
                   const double* b, double* x, void* ws, double tol_r, double tol_A, int maxit, int first_check,
                   double wait_ms, hipStream_t s, double* info, int phase, int* resumed);

}  // namespace efea
