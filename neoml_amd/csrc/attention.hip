// The core of an attention layer as one launch: scores, their factor, softmax over rows, the weighted sum of the values.
#include "gemm.h"
#include <float.h>

namespace nh {

typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

struct CAttentionArgs {
	const float* Q;       // [batch][M][K]
	const float* KT;      // [batch][K][N]
	const float* V;       // [batch][N][D]
	const float* Scale;   // a device scalar, may be null
	float* Scores;        // [batch][M][N]
	float* Weights;       // [batch][M][N]
	float* Context;       // [batch][M][D]
	float* Transposed;    // [batch / Heads][M][Heads][D], may be null
	int M, N, K, D, Heads, Strips, Pitch;
};

// A workgroup owns 16 rows of one product and keeps their scores in LDS. Its wavefronts deal the columns of the scores, 16 at a
// time, among themselves, then the rows of the softmax, then the columns of the result, with v_mfma_f32_16x16x4_f32 and operands
// that lie N-major in memory ( the transposed keys, the values ) fetched by 64 bytes a row straight into registers, the next block's on
// their way while one is multiplied.
// All four results are written, as the separate calls leave them, but scores and weights are not read back. For many heads the matrix
// pipe ( 31 us of the 71 for 256 heads of 256 x 256 ), the softmax's arithmetic and the stores bound it, for few the launch. us, the four or
// five separate launches and this one: 8 heads of 37 16.1 and 5.2, 32 of 128 19.5 and 7.5, 32 of 333 56 and 25, 256 of 256 87 and 71, 1024 of
// 32 27 and 17; 128 of 512 162 and 168, see attentionTakes. 32 rows to a workgroup: 7.5, 10.8, 33, 76, 18.
// NJ: columns of the scores are at most 64 NJ.
template<int NJ>
__global__ __launch_bounds__( 256 )
void attentionKernel( const CAttentionArgs args )
{
	extern __shared__ float4 attentionLds[];
	float* queries = reinterpret_cast<float*>( attentionLds ); // [16][64 + 4]
	float* scores = queries + 16 * 68;                         // [16][Pitch]
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane( tid >> 6 );
	const int l16 = lane & 15, quad = lane >> 4;
	const int id = xcdSwizzle( blockIdx.x, gridDim.x ); // the strips of one product share keys and values: same XCD, same L2
	const int batch = id / args.Strips;
	const int m0 = ( id % args.Strips ) * 16;
	const int M = args.M, N = args.N, K = args.K, D = args.D, pitch = args.Pitch;
	const int rows = min( 16, M - m0 );
	const float alpha = args.Scale != nullptr ? *args.Scale : 1.f;

	const float* Q = args.Q + ( static_cast<long long>( batch ) * M + m0 ) * K;
	const __amdgpu_buffer_rsrc_t bufQ = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( Q ), 0, static_cast<unsigned>( rows * K ) * 4u, 0x00020000 );
	const __amdgpu_buffer_rsrc_t bufK = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( args.KT + static_cast<long long>( batch ) * K * N ), 0,
		static_cast<unsigned>( K * N ) * 4u, 0x00020000 );
	const __amdgpu_buffer_rsrc_t bufV = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( args.V + static_cast<long long>( batch ) * N * D ), 0,
		static_cast<unsigned>( N * D ) * 4u, 0x00020000 );

	// scores: this wavefront's blocks of 16 columns; lane ( column, quad ) holds k = 16 quad + s of step s ( what lies behind the last row or
	// column is out of range: zeros )
	const int blocks = ( N + 15 ) / 16;
	auto loadKeys = [&]( int block, float ( &to )[16] ) {
		// ( K is a multiple of 16: a lane's sixteen rows are inside or outside together )
		const int n = block * 16 + l16;
		const unsigned at = n < N && quad * 16 < K ? ( static_cast<unsigned>( quad * 16 ) * static_cast<unsigned>( N ) + static_cast<unsigned>( n ) ) * 4u : OutOfRange;
#pragma unroll
		for( int s = 0; s < 16; ++s ) {
			to[s] = __uint_as_float( __builtin_amdgcn_raw_buffer_load_b32( bufK, at, static_cast<unsigned>( s * N ) * 4u, 0 ) );
		}
	};
	float keys[2][16];
	loadKeys( wave, keys[0] );
	{
		const int row = tid >> 4, k = ( tid & 15 ) * 4;
		*reinterpret_cast<float4*>( queries + row * 68 + k ) = bufferLoad4( bufQ, row < rows && k < K ? static_cast<unsigned>( row * K + k ) * 4u : OutOfRange );
	}
	__syncthreads();
	f32x4 q[4];
#pragma unroll
	for( int s = 0; s < 4; ++s ) {
		q[s] = *reinterpret_cast<const f32x4*>( queries + l16 * 68 + quad * 16 + s * 4 );
	}
	auto scoresOf = [&]( int block, const float ( &k )[16] ) {
		f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
		for( int s = 0; s < 16; ++s ) {
			acc = __builtin_amdgcn_mfma_f32_16x16x4f32( q[s >> 2][s & 3], k[s], acc, 0, 0, 0 );
		}
		// lane ( column, quad ): rows 4 quad .. + 3
		if( block * 16 + l16 < N ) {
#pragma unroll
			for( int r = 0; r < 4; ++r ) {
				scores[( quad * 4 + r ) * pitch + block * 16 + l16] = acc[r] * alpha;
			}
		}
	};
	for( int block = wave; block < blocks; block += 8 ) {
		loadKeys( block + 4, keys[1] );
		scoresOf( block, keys[0] );
		if( block + 4 < blocks ) {
			loadKeys( block + 8, keys[0] );
			scoresOf( block + 4, keys[1] );
		}
	}

	// the values' first block for the product behind the softmax: lane ( column, quad ) holds k = 16 g + 4 quad + j
	const int column = wave * 16 + l16;
	const unsigned valueAt = column < D ? static_cast<unsigned>( quad * 4 * D + column ) * 4u : OutOfRange;
	auto loadValues = [&]( int g, float ( &to )[4] ) {
#pragma unroll
		for( int j = 0; j < 4; ++j ) {
			to[j] = __uint_as_float( __builtin_amdgcn_raw_buffer_load_b32( bufV, valueAt + static_cast<unsigned>( g * 16 + j ) * static_cast<unsigned>( D ) * 4u, 0, 0 ) );
		}
	};
	constexpr int Ahead = 4;
	float values[Ahead][4];
#pragma unroll
	for( int g = 0; g < Ahead; ++g ) {
		loadValues( g, values[g] );
	}
	__syncthreads();

	// softmax, four rows to a wavefront, side by side; exp( x - max ) * ( 1 / sum ) as softmaxRowsKernel has it
	const int padded = blocks * 16;
	{
		const int row0 = wave * 4;
		float v[4][NJ], mx[4], sum[4];
#pragma unroll
		for( int r = 0; r < 4; ++r ) {
			mx[r] = -FLT_MAX;
#pragma unroll
			for( int j = 0; j < NJ; ++j ) {
				const int n = lane + j * 64;
				v[r][j] = n < N ? scores[( row0 + r ) * pitch + n] : -FLT_MAX;
				mx[r] = fmaxf( mx[r], v[r][j] );
			}
		}
#pragma unroll
		for( int r = 0; r < 4; ++r ) {
			mx[r] = waveReduceMax( mx[r] );
		}
#pragma unroll
		for( int r = 0; r < 4; ++r ) {
			const bool inside = row0 + r < rows;
			float* to = args.Scores + ( static_cast<long long>( batch ) * M + m0 + row0 + r ) * N;
			sum[r] = 0.f;
#pragma unroll
			for( int j = 0; j < NJ; ++j ) {
				const int n = lane + j * 64;
				if( inside && n < N ) {
					to[n] = v[r][j];
				}
				v[r][j] = n < N ? expf( v[r][j] - mx[r] ) : 0.f;
				sum[r] += v[r][j];
			}
		}
#pragma unroll
		for( int r = 0; r < 4; ++r ) {
			sum[r] = waveReduceSum( sum[r] );
		}
#pragma unroll
		for( int r = 0; r < 4; ++r ) {
			const bool inside = row0 + r < rows;
			const float inv = 1.f / sum[r];
			float* to = args.Weights + ( static_cast<long long>( batch ) * M + m0 + row0 + r ) * N;
#pragma unroll
			for( int j = 0; j < NJ; ++j ) {
				const int n = lane + j * 64;
				const float weight = v[r][j] * inv;
				if( n < padded ) {
					scores[( row0 + r ) * pitch + n] = n < N ? weight : 0.f; // ( up to whole blocks: what is multiplied by no value )
				}
				if( inside && n < N ) {
					to[n] = weight;
				}
			}
		}
	}
	__syncthreads();

	// the result: 16 columns to a wavefront, two chains of sums
	if( wave * 16 >= D ) {
		return;
	}
	f32x4 acc[2] = { { 0.f, 0.f, 0.f, 0.f }, { 0.f, 0.f, 0.f, 0.f } };
	for( int g0 = 0; g0 < blocks; g0 += Ahead ) {
#pragma unroll
		for( int u = 0; u < Ahead; ++u ) {
			const int g = g0 + u;
			// ( groups behind the last: values out of range, and weights that are not there )
			const f32x4 w = g < blocks ? *reinterpret_cast<const f32x4*>( scores + l16 * pitch + g * 16 + quad * 4 ) : f32x4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
			for( int j = 0; j < 4; ++j ) {
				acc[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32( w[j], values[u][j], acc[j & 1], 0, 0, 0 );
			}
			loadValues( g + Ahead, values[u] );
		}
	}
	if( column >= D ) {
		return;
	}
#pragma unroll
	for( int r = 0; r < 4; ++r ) {
		const int row = quad * 4 + r;
		if( row < rows ) {
			const float v = acc[0][r] + acc[1][r];
			args.Context[( static_cast<long long>( batch ) * M + m0 + row ) * D + column] = v;
			if( args.Transposed != nullptr ) {
				const int image = batch / args.Heads, head = batch - image * args.Heads;
				args.Transposed[( ( static_cast<long long>( image ) * M + m0 + row ) * args.Heads + head ) * D + column] = v;
			}
		}
	}
}

constexpr int MaxAttentionColumns = 512;
constexpr long long MaxWorkgroups = ( 1 << 24 ) - 1; // a launch has fewer than 2^32 threads

// Whether it takes the core of this layer. Scores of more than 256 columns only where the kernel for batches of products does not
// have enough strips of 64 rows to take the two products by itself.
bool attentionTakes( int batch, int M, int N, int K, int D, const float* q )
{
	return batch > 0 && M > 0 && N > 0 && N <= MaxAttentionColumns && K > 0 && K <= 64 && K % 16 == 0 && D > 0 && D <= 64 && isAligned16( q )
		&& ( N <= 256 || static_cast<long long>( ceilDiv( M, 64 ) ) * batch < 512 ) && static_cast<long long>( ceilDiv( M, 16 ) ) * batch <= MaxWorkgroups;
}

int launchAttention( hipStream_t stream, const CPendingAttention& a )
{
	CAttentionArgs args = { a.Q, a.KT, a.V, a.Scale, a.Scores, a.Weights, a.Context, a.Transposed, a.M, a.N, a.K, a.D, a.Heads, ceilDiv( a.M, 16 ),
		ceilDiv( a.N, 16 ) * 16 + 4 };
	const dim3 grid( static_cast<unsigned>( static_cast<long long>( args.Strips ) * a.Batch ) );
	const size_t lds = static_cast<size_t>( 16 ) * ( 68 + args.Pitch ) * sizeof( float );
	if( a.N <= 64 ) {
		hipLaunchKernelGGL( attentionKernel<1>, grid, dim3( 256 ), lds, stream, args );
	} else if( a.N <= 128 ) {
		hipLaunchKernelGGL( attentionKernel<2>, grid, dim3( 256 ), lds, stream, args );
	} else if( a.N <= 256 ) {
		hipLaunchKernelGGL( attentionKernel<4>, grid, dim3( 256 ), lds, stream, args );
	} else {
		hipLaunchKernelGGL( attentionKernel<8>, grid, dim3( 256 ), lds, stream, args );
	}
	NH_LAUNCH_CHECK();
	return NH_OK;
}

} // namespace nh
