// Random-torsion conformers on the device (conformers.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace cdk {

// U[0, 1) from a counter-based stream; the same on host and device.
__host__ __device__ double torsion_uniform(unsigned long long seed, int trial, int rotor);

// Trials first .. first + ntrial - 1: coords [natom][3]; rotors [nrotor][4];
// moving [ceil(nrotor / 64)][natom], bit r % 64 of word r / 64 of an atom set
// when rotor r moves it; exclude [natom][ceil(natom / 64)], bits of the atoms
// the steric filter does not test an atom against; out [ntrial][natom][3]
// (written for passing trials); ok [ntrial] (1 = no clash).
hipError_t launch_conformers(hipStream_t st, int natom, const double* coords, int nrotor, const int* rotors,
                             const unsigned long long* moving, const unsigned long long* exclude, int first,
                             int ntrial, unsigned long long seed, double clash_dist, double* out, int* ok);
// The first max_keep passing trials of such a launch, packed in trial order:
// kept [count][natom][3], trial [count]; list [min(max_keep, ntrial)] is
// scratch.
hipError_t launch_keep_conformers(hipStream_t st, int natom, int first, int ntrial, const int* ok, const double* all,
                                  int max_keep, int* list, int* count, double* kept, int* trial);

}  // namespace cdk
