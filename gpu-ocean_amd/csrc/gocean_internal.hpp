// gocean_internal.hpp -- declarations shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>

#include "../../include/gocean.h"
#include "cdklm16_tile.hpp"

namespace gocean {

struct TileConfig {
    int bw, bh, nt;
    const char* name;
};

extern const TileConfig kTileConfigs[];
extern const int kNumTileConfigs;
extern const int kDefaultTileConfig;
extern const int kMarchAutoConfig;
// Tiles of the rotated and per-cell modes (they ignore the configuration), and
// the choice among them for a mode and n domains
constexpr TileConfig kGeneralTiles[] = {{32, 14, 512, "32x14/512"}, {16, 16, 256, "16x16/256"}, {32, 8, 256, "32x8/256"}};
int general_tile(int mode, const int* nx, const int* ny, int n);
// configurations kFirstMarchConfig .. kNumTileConfigs-1 are column marching
constexpr int kFirstMarchConfig = 7;
// configuration used when the caller passes -1
int default_tile_config(int nx, int ny);

int set_error(int code, const char* fmt, ...);
void clear_error();
const char* last_error();
int check_launch(const char* what);
int validate_domain(const gocean_domain_t* d);
void fill_args(const gocean_domain_t* d, SubstepArgs& A);
// the low part l of div_k's reciprocal r + l of a divisor d, and whether the two
// instructions then divide every float by d correctly rounded (searched and
// checked once per value of d, on the host)
struct DivisorLow {
    float low;
    bool exact;
};
DivisorLow divisor_low(float d);
// the substep's FAST arithmetic is exact for these constants: two-instruction
// division by dx, dy and 2g, whose low parts it writes to D, and the Newton
// square root of g h for h above the depth cutoff
bool fast_arith(float g, float dx, float dy, float cutoff, SubstepDerived& D);
// the column-marching kernels' 32-bit plane offsets cover a domain of this
// height and pitches
bool march_fits(int ny, int pitch, int hi_pitch);
// column-marching launch shape: waves the device holds at once for a kernel,
// and the rows per strip that fill whole rounds of them
int compute_units();
int resident_waves(const void* kernel);
int march_stage(int rk_order, int rk_step, float r);
int march_rows(const int* strips, const int* ny, int n, int resident, int least);
int launch_substep(const SubstepArgs& A, int cfg, bool field, hipStream_t s);
// zero-rotation substep that also writes the branch record (A.tape_*)
int launch_substep_tape(SubstepArgs A, hipStream_t s);
int periodic_bc(const gocean_domain_t* d, float* e, float* u, float* v, hipStream_t s);
// CFL reduction: out[0..1] as gocean_max_dt, partial minima (one per
// reduction workgroup, max_dt_partials(d) <= kMaxDtPartials of them) in
// `partial`; max_dt keeps them in out[2..]
constexpr int kMaxDtPartials = 1024;
int max_dt_partials(const gocean_domain_t* d);
int max_dt_into(const gocean_domain_t* d, const float* eta, const float* hu, const float* hv,
                const float* Hm, float courant, float* partial, float* out, hipStream_t s, float* host = nullptr);
int max_dt(const gocean_domain_t* d, const float* eta, const float* hu, const float* hv,
           const float* Hm, float courant, float* out, hipStream_t s);
// substep-adjoint kernel of the reverse entry points (0 tile, 1 marching)
// and the marching kernel's rows per strip for domains of these sizes
extern int g_adj_kernel;
int adj_march_rows(const int* nx, const int* ny, int n);
// the reverse kernel for a launch over this many cells: column marching
// (true) or tile, by g_adj_kernel
bool adj_use_march(long long cells);

}  // namespace gocean
