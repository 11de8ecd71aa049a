// gctf_internal.hpp -- shared device structures and kernel launchers of
// libgctf_hip.so.  Not part of the public C-ABI (include/gctf_hip.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gctf_fft.hpp"

namespace gctf {

// Candidate-stage kinds of the 2D search (CFindDefocus2D.cpp:153-361).
enum StageKind : int {
	ST_NONE = 0,
	ST_INIT = 2,     // mIterate's first mCorrelate
	ST_ASTIG = 3,    // mFindAstig grid
	ST_ASTMAG = 4,   // mRefineAstMag
	ST_ASTANG = 5,   // mRefineAstAng
	ST_DFMEAN = 6,   // mRefineDfMean
	ST_PHASE = 7,    // mRefinePhase
};

// Largest candidate count of one stage: the 51 x 51 astigmatism grid.
constexpr int kMaxCands = 2601;
// Pixel chunks the 2D correlation is split into (partial sums per chunk).
constexpr int kPixChunks = 8;
// Partial sums of one image's stage; its buffer holds two stages (a launch
// reads the previous stage's sums and writes its own).
constexpr long long kPartStages = 2;
constexpr long long kPartStage = (long long)kMaxCands * kPixChunks;
constexpr long long kPartStride = kPartStages * kPartStage;
// Parts of a ring spectrum's FP64 energy.
constexpr int kRingParts = 16;

// Per-plan CTF constants in pixel units (CCTFTheory.cpp:77-78,
// GCalcCTF2D.cu:88-97).
struct CtfConsts {
	float wl;         // wavelength / pixel
	float cs;         // Cs / pixel
	float amp_phase;  // atanf(ac / sqrtf(1 - ac^2))
	float pix;        // working pixel size (A)
};

// Candidate counts of the 2D search program.  The plain program is the
// reference's (CFindDefocus2D.cpp:153-361): a 51 x 51 astigmatism grid, then
// 19 rounds of 21 / 51 / 31 candidates, defocus step floor 20 A.  The
// learned path runs a smaller program inside the proposal's window and
// ends with a fine defocus stage.
struct SearchProgram {
	int n_ast, n_ang;     // mFindAstig grid
	int n_mag, n_angl;    // mRefineAstMag / mRefineAstAng candidates
	int n_df;             // mRefineDfMean candidates
	int iters;            // mIterate's iIterations
	float df_minstep;     // mRefineDfMean step floor (A)
	int fine_n;           // final defocus stage (0: none)
	float fine_step;      // its step (A)
};

__host__ __device__ constexpr SearchProgram plain_program()
{
	return SearchProgram{51, 51, 21, 51, 31, 20, 20.0f, 0, 0.0f};
}

// Per-micrograph search state; mirrors the fields of CFindCtfBase,
// CFindDefocus1D and CFindDefocus2D (CFindCTFInc.h:480-562).
struct SearchState {
	// CFindCtfBase outputs (degrees, A)
	float df_min, df_max, ast_ang, ext_phase, score, ctf_res;
	// CFindCtfBase::SetPhase range (degrees); ext_phase above holds the
	// current CFindCtfBase::m_fExtPhase
	float phase_range;
	// CFindDefocus2D
	float dfmean, ast, ang, phase, ccmax, oldcc;
	float dfrange[2], astrange[2], angrange[2], phrange[2];
	float tot_df, tot_ast, tot_ang;
	int done;
	int iter;
	// pending candidate stage
	int st_kind;
	int st_n;        // number of candidates
	int st_nast;     // astig grid: candidates per angle row
	float st_a0, st_astep;   // first value / step (ast for ASTIG)
	float st_b0, st_bstep;   // angle grid for ASTIG
	float st_lo, st_hi;      // phase window for ST_PHASE
	float st_old;            // mRefineDfMean: the df before the stage
	int lowpassed;           // a12 gate outcome
	SearchProgram pg;        // candidate counts of the running 2D program
	int skip;                // 1: the image sits out the running search pass
	int fallback;            // learned path: 1 when the plain search must decide
	float conf;              // learned path: proposal confidence
	// pending 1D stage (CFindDefocus1D::mBrutalForceSearch): candidate
	// i = iph * s1_ndf + idf at defocus s1_df0 + idf s1_dfstep A and phase
	// s1_ph0 + iph s1_phstep degrees (clamped to [0, 150]); s1_stage 0 is
	// CFindCtf1D::mFindDefocus, 1 mRefineDefocus
	float s1_df0, s1_dfstep, s1_ph0, s1_phstep;
	int s1_ndf, s1_n, s1_stage;
};

__host__ __device__ __forceinline__ void step_program(SearchProgram& d, const SearchProgram& s)
{
	d.n_ast = s.n_ast; d.n_ang = s.n_ang; d.n_mag = s.n_mag; d.n_angl = s.n_angl;
	d.n_df = s.n_df; d.iters = s.iters; d.df_minstep = s.df_minstep;
	d.fine_n = s.fine_n; d.fine_step = s.fine_step;
}

// The fields of a state that a transition reads or writes, one by one (a
// struct assignment would keep the copy in memory instead of registers).
__host__ __device__ __forceinline__ void step_fields(SearchState& d, const SearchState& s)
{
	d.df_min = s.df_min; d.df_max = s.df_max; d.ast_ang = s.ast_ang; d.ext_phase = s.ext_phase; d.score = s.score;
	d.phase_range = s.phase_range;
	d.dfmean = s.dfmean; d.ast = s.ast; d.ang = s.ang; d.phase = s.phase; d.ccmax = s.ccmax; d.oldcc = s.oldcc;
#pragma unroll
	for (int i = 0; i < 2; ++i) {
		d.dfrange[i] = s.dfrange[i]; d.astrange[i] = s.astrange[i];
		d.angrange[i] = s.angrange[i]; d.phrange[i] = s.phrange[i];
	}
	d.tot_df = s.tot_df; d.tot_ast = s.tot_ast; d.tot_ang = s.tot_ang;
	d.done = s.done; d.iter = s.iter; d.skip = s.skip;
	d.st_kind = s.st_kind; d.st_n = s.st_n; d.st_nast = s.st_nast;
	d.st_a0 = s.st_a0; d.st_astep = s.st_astep; d.st_b0 = s.st_b0; d.st_bstep = s.st_bstep;
	d.st_lo = s.st_lo; d.st_hi = s.st_hi; d.st_old = s.st_old;
	step_program(d.pg, s.pg);
}

// The other fields: a transition only carries them over.
__host__ __device__ __forceinline__ void step_kept(SearchState& d, const SearchState& s)
{
	d.ctf_res = s.ctf_res;
	d.lowpassed = s.lowpassed;
	d.fallback = s.fallback; d.conf = s.conf;
	d.s1_df0 = s.s1_df0; d.s1_dfstep = s.s1_dfstep; d.s1_ph0 = s.s1_ph0; d.s1_phstep = s.s1_phstep;
	d.s1_ndf = s.s1_ndf; d.s1_n = s.s1_n; d.s1_stage = s.s1_stage;
}

// The new state s of a transition from `in` into `out` (which may be `in`) by
// the lanes of one wavefront.  One lane stores every field, once and by its
// name: lanes have no order among themselves, and neither have stores to one
// address through different types.
__host__ __device__ __forceinline__ void step_store(SearchState* out, const SearchState* in, const SearchState& s,
	int lane)
{
	if (lane != 0) return;
	step_fields(*out, s);
	if (out != in) step_kept(*out, *in);
}

// Per-plan 2D-ring tables in structure-of-arrays form (device pointers).
struct RingTables {
	int n;                 // ring pixel count
	const int* idx;        // y * cmpx + x
	const float4* abcs;    // a = (pi'/pi) * wl * s^2 (chi/pi per unit df), b = (pi'/pi) * 0.5 * wl^3 * s^4 * Cs,
	                       // cos(2 theta), sin(2 theta)
	const float* w;        // exp(-16 s^2)
};

// Per-micrograph search plan (device array indexed by image): the CTF
// constants at the micrograph's working pixel size, its correlation ring and
// its 1D bin range.  Micrographs of one batch may differ in all three.
struct ImgPlan {
	CtfConsts cc;
	RingTables ring;
	float lo1d, hi1d;
};

}  // namespace gctf
