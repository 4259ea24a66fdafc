// What the kernels for dense contractions share: operand modes, arguments, tile arithmetic.
#pragma once

#include "common.h"

namespace nh {

typedef float f32x16 __attribute__( ( ext_vector_type( 16 ) ) );

// AM_Conv1x1 runs the same code as AM_Conv; the separate value gives 1x1 convolutions their own kernel symbols, so
// that profiles tell them apart from the 3x3 ones
// AM_ConvRows serves channel counts that are not a multiple of 4 (grey and RGB inputs): the reduction index runs
// over Fh filter rows of RowPitch = ceil4( Fw * Cin ) values each. The Fw * Cin values that one filter row meets are
// contiguous in a channels-last image (no dilation along the width), so they are fetched as 128-bit runs however
// Cin divides; the 1-3 padding values per row are masked to zero on both operands.
// AM_ConvClasses: the gradient by the input of a strided convolution, one stride-1 convolution per residue class of the
// input pixels (blockIdx.y = class): AM_Conv whose geometry, filter and output rows come from args.Class[class].
// AM_ConvTaps: AM_Conv for channel counts that are a multiple of the K step, without the strided gradient's exact-division
// test: a step never straddles two taps, the reduction ends on a step, and everything that is only needed otherwise is
// compiled out of the loop ( the 3x3 convolutions of the image networks ).
enum TAMode { AM_RowsK = 0, AM_RowsM = 1, AM_Conv = 2, AM_Conv1x1 = 3, AM_ConvRows = 4, AM_ConvClasses = 5, AM_ConvTaps = 6 };
// BM_ConvN: B is the im2col view of an N,H,W,C image read N-major: row k = output pixel, column n = ( kh, kw, ci ).
// With A = the gradient by the convolution's output read M-major this is the gradient by the filter.
enum TBMode { BM_RowsK = 0, BM_RowsN = 1, BM_ConvN = 2 };

// One residue class ( ( hi + pad ) mod stride, same along the width ) of the input pixels of a strided convolution. Only
// the filter taps kh with kh * dilation in the same class reach its pixels, Fh x Fw of them, and through them the
// class is a stride-1 convolution over the output gradient. Its result rows are the pixels
// ( OutH0 + j * strideH, OutW0 + i * strideW ), j < Ho, i < Wo, of every image.
struct CConvClass {
	int K, Fh, Fw, PadH, PadW, Ho, Wo, M, OutH0, OutW0;
	long long BOffset; // of the class's filter [N][Fh][Fw][Cin] inside B, in floats
};

constexpr int MaxConvClasses = 4;
constexpr int MaxProductGroup = 3;

struct CMatMulArgs {
	const float* A;
	const float* B;
	float* C;
	const float* Bias; // per column n, may be null
	int M, N, K;
	int Lda, Ldb, Ldc;
	long long BatchStrideA, BatchStrideB, BatchStrideC;
	int Accumulate; // C += instead of C =
	int SplitK;     // number of K slices (grid z); > 1: partial products are added to C with atomics
	int StepsPerSplit;
	int TilesM, TilesN;
	// convolution geometry (AM_Conv only): A is the image, M = batch * Ho * Wo
	int H, W, Cin, Ho, Wo, Fh, Fw, PadH, PadW, StrideH, StrideW, DilH, DilW;
	int RowK, RowPitch; // AM_ConvRows: Fw * Cin and its round-up to a multiple of 4; K = Fh * RowPitch
	int AFloats, BFloats; // AM_ConvRows: sizes of the image and of the filter, the limit of a 128-bit load that reads past a run
	// AM_Conv as the gradient by the input of a strided convolution: the tap's source coordinate is
	// ( ho * StrideH - PadH + kh * DilH ) / UpH and only exists where that division is exact (values <= 1: no division)
	int UpH, UpW;
	int ManySlices; // the reduction is far longer than the output is large: as many K slices as fill the device
	// Tail mode (FullTiles > 0, grid z = 1): the first FullTiles workgroups compute one whole tile each; the workgroups
	// behind them share the TailTiles remaining tiles, TailSplit slices of TailSteps K steps per tile, and meet in C
	// through atomic adds like the K slices above
	int FullTiles, TailTiles, TailSplit, TailSteps;
	// K slices that meet without atomics (Partials != null): every slice leaves its accumulators in Partials
	// [ sliced tile ][ slice ][ 4096 ] and counts itself in Counters[ sliced tile ]; the slice that counts last adds
	// them up in slice order, runs the ordinary epilogue and sets the counter back to zero for the next launch.
	float* Partials;
	unsigned* Counters;
	// AM_ConvClasses: the dense result is [images][OutH][OutW][Ldc], DenseM pixels in all
	int OutH, OutW, OutUpH, OutUpW, DenseM;
	CConvClass Class[MaxConvClasses];
	// products of one A ( grid y ): each with its own B, free term and result
	int Group;
	const float* GroupB[MaxProductGroup];
	const float* GroupBias[MaxProductGroup];
	float* GroupC[MaxProductGroup];
	// C = x * gate with gate = sigmoid( x * *GateScale ), x = A * B + bias, the gates stored too ( C's layout; null: none ): a GELU taken along
	float* Gate;
	const float* GateScale;
	int SmallTile; // smallProductKernel: 0: 16 x 16, 1: 16 x 32, 2: 32 x 32
	// epilogue of the fused blocks: C = act( A * B + bias ) + Residual; Residual has C's layout, may be C itself
	CFusedActivation Act;
	const float* Residual;
	// floor( 2^32 / divisor ) for the divisions of the prologue ( pixel -> image, row, column; workgroup -> tile ): a
	// multiplication and one correction instead of the twenty-odd instructions of a division by a run-time value
	unsigned WoMagic, HoMagic, TilesNMagic;
	// size of C in bytes when its rows can be addressed by 32-bit offsets from its start ( 0: they cannot ): the
	// epilogue then stores through a buffer descriptor of that size, which drops the rows of a last tile that lie
	// beyond the matrix by itself
	unsigned CBytes;
};

// floor( 2^32 / d ), capped: with it q = mulhi( x, magic ) is floor( x / d ) or one less for every x < 2^32
inline unsigned divisionMagic( int d )
{
	return d <= 1 ? 0xFFFFFFFFu : static_cast<unsigned>( 0x100000000ULL / static_cast<unsigned>( d ) );
}

__device__ __forceinline__ void fastDivMod( int x, int d, unsigned magic, int& quotient, int& remainder )
{
	unsigned q = __umulhi( static_cast<unsigned>( x ), magic );
	unsigned r = static_cast<unsigned>( x ) - q * static_cast<unsigned>( d );
	const bool low = r >= static_cast<unsigned>( d );
	quotient = static_cast<int>( low ? q + 1 : q );
	remainder = static_cast<int>( low ? r - static_cast<unsigned>( d ) : r );
}

constexpr int Threads = 256;

#ifndef NH_KSTEP
#define NH_KSTEP 16
#endif

// ( gemm_split.hip ) C = act( A * B^T + bias ) (+ C, + residual) for operands that are K-major ( args as the fp32 kernels take
// them ). true: launched, *rc is the launch's code; false: not one that it is for.
bool trySplitProduct( hipStream_t stream, const CMatMulArgs& args, int batch, bool vec, int* rc );

// A meeting place handed in by the caller instead of the stream's block: the launch neither allocates nor looks the
// stream up, and fails when the place is too small.
struct CSliceMeeting {
	float* Partials;
	size_t PartialFloats;
	unsigned* Counters;
	size_t CounterCount;
};

// The counters of such a place are whatever the last call left there: cleared on the stream in front of each launch.
void clearCounters( hipStream_t stream, unsigned* counters, size_t count );

// ( gemm_small.hip ) the same for results of a few tiles; A also as the im2col view of an image whose channel count is a multiple
// of 16. fixedMeeting: where its slices meet ( none if they would not fit ) instead of the stream's block.
constexpr int MaxSmallSlices = 16;
bool trySmallProduct( hipStream_t stream, const CMatMulArgs& args, bool convolution, int batch, bool vec, int* rc,
	const CSliceMeeting* fixedMeeting = nullptr );

// The stream's block of partial tiles and arrival counters for reductions that are cut into slices ( the counters are zero
// between launches ). false: none to be had ( a capturing stream, a shared stream handle, no memory ).
bool sliceMeetingPlace( hipStream_t stream, size_t partialFloats, size_t counterCount, float** partials, unsigned** counters );

} // namespace nh
