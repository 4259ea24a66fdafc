// fp32 products and convolutions whose result is a few hundred 32 x 32 tiles or less: one picture, one short sequence.
#include "gemm.h"
#include <type_traits>

namespace nh {

typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

// C[M x N] = act( A * B^T + bias ) (+ C, + residual), A rows of K values or the im2col view of an image whose channel count is
// a multiple of 16, B rows of K values.
// What bounds such a product is latency: a chain of K steps, each with a barrier, on a few workgroups.
// So a workgroup is one 32 x 32 tile whose reduction is dealt to its WAVES wavefronts and, where the tiles leave compute
// units idle, to several workgroups. A wavefront fetches its share straight into operand registers, 16 k at a time: lane
// ( row, quad ) holds k = 16 g + 4 quad .. + 3 of its rows, so that four lanes cover 64 bytes of a row, for 2 x 2 blocks of
// v_mfma_f32_16x16x4_f32; eight such groups are in flight. It meets no barrier until its share is done. The shares are
// summed through LDS in the order of k, the slices through scratch memory by the one that arrives last, which fetches the
// others' tiles all at once.
template<int AMODE, int WAVES>
__global__ __launch_bounds__( 64 * WAVES, 2 )
void smallProductKernel( const CMatMulArgs args )
{
	constexpr bool IsTaps = ( AMODE == AM_ConvTaps );
	static_assert( IsTaps || AMODE == AM_RowsK, "operands that are K-major" );
	constexpr int T = 64 * WAVES;
	constexpr int Batch = 2, Sets = 4; // groups of 16 k to a register set, sets
	constexpr int PerThread = 1024 / T; // elements of the tile that a thread sums and writes
	__shared__ float lds[WAVES][16][64];
	__shared__ unsigned arrived;

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane( tid >> 6 );
	const int l16 = lane & 15, quad = lane >> 4;
	const int tile = xcdSwizzle( blockIdx.x, gridDim.x );
	int tileM, tileN;
	fastDivMod( tile, args.TilesN, args.TilesNMagic, tileM, tileN );
	const int m0 = tileM * 32, n0 = tileN * 32;
	const int batch = blockIdx.y, slice = blockIdx.z;
	const int M = args.M, N = args.N, K = args.K;
	const float* baseA = args.A + batch * args.BatchStrideA;
	const float* baseB = args.B + batch * args.BatchStrideB;

	// this wavefront's groups
	const int groups = ( K + 15 ) / 16;
	const int firstGroup = ( slice * WAVES + wave ) * args.StepsPerSplit;
	const int lastGroup = min( firstGroup + args.StepsPerSplit, groups );

	// the lane's two rows of A and of B
	unsigned offA[2], offB[2];
	unsigned baseOfA[2] = {}; // in floats, of tap ( 0, 0 ): unsigned arithmetic, it may lie in front of the image
	int imageH0[2] = {}, imageW0[2] = {};
	int tapCi = 0, tapKh = 0, tapKw = 0;
	auto tapOffsets = [&]() {
		const int dh = tapKh * args.DilH, dw = tapKw * args.DilW; // ( scalar )
		const unsigned tapFloats = ( static_cast<unsigned>( dh ) * static_cast<unsigned>( args.W ) + static_cast<unsigned>( dw ) )
			* static_cast<unsigned>( args.Cin );
#pragma unroll
		for( int i = 0; i < 2; ++i ) {
			const bool ok = tapKh < args.Fh && static_cast<unsigned>( imageH0[i] + dh ) < static_cast<unsigned>( args.H )
				&& static_cast<unsigned>( imageW0[i] + dw ) < static_cast<unsigned>( args.W );
			offA[i] = ok ? ( baseOfA[i] + tapFloats ) * 4u : OutOfRange;
		}
	};
#pragma unroll
	for( int i = 0; i < 2; ++i ) {
		const int n = n0 + i * 16 + l16, m = m0 + i * 16 + l16;
		offB[i] = n < N ? ( static_cast<unsigned>( n ) * static_cast<unsigned>( args.Ldb ) + quad * 4u ) * 4u : OutOfRange;
		if constexpr( IsTaps ) {
			int t, wo, image, ho;
			fastDivMod( m, args.Wo, args.WoMagic, t, wo );
			fastDivMod( t, args.Ho, args.HoMagic, image, ho );
			imageH0[i] = m < M ? ho * args.StrideH - args.PadH : -0x40000000;
			imageW0[i] = wo * args.StrideW - args.PadW;
			baseOfA[i] = static_cast<unsigned>( image * args.H * args.W * args.Cin ) + ( static_cast<unsigned>( imageH0[i] )
				* static_cast<unsigned>( args.W ) + static_cast<unsigned>( imageW0[i] ) ) * static_cast<unsigned>( args.Cin ) + quad * 4u;
		} else {
			offA[i] = m < M ? ( static_cast<unsigned>( m ) * static_cast<unsigned>( args.Lda ) + quad * 4u ) * 4u : OutOfRange;
		}
	}
	if constexpr( IsTaps ) {
		const int tap = firstGroup * 16 / args.Cin;
		tapCi = firstGroup * 16 - tap * args.Cin;
		tapKh = tap / args.Fw;
		tapKw = tap - tapKh * args.Fw;
		tapOffsets();
	}

	float4 a[Sets][Batch][2], b[Sets][Batch][2];
	// ( a group behind the share's last is asked of a descriptor of size zero: zeros, no memory access )
	auto load = [&]( int group, int set ) {
#pragma unroll
		for( int g = 0; g < Batch; ++g ) {
			const unsigned range = group + g < lastGroup ? BufferBytes : 0u;
			const __amdgpu_buffer_rsrc_t bufA = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( baseA ), 0, range, 0x00020000 );
			const __amdgpu_buffer_rsrc_t bufB = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( baseB ), 0, range, 0x00020000 );
			const unsigned uniB = static_cast<unsigned>( group + g ) * 64u;
			const bool inK = IsTaps || ( group + g ) * 16 + quad * 4 < K; // ( K is a multiple of 4 )
#pragma unroll
			for( int i = 0; i < 2; ++i ) {
				a[set][g][i] = bufferLoad4( bufA, inK ? offA[i] : OutOfRange, IsTaps ? static_cast<unsigned>( tapCi ) * 4u : uniB );
				b[set][g][i] = bufferLoad4( bufB, inK ? offB[i] : OutOfRange, uniB );
			}
			if constexpr( IsTaps ) {
				tapCi += 16;
				if( tapCi >= args.Cin ) {
					tapCi = 0;
					if( ++tapKw == args.Fw ) {
						tapKw = 0;
						++tapKh;
					}
					tapOffsets();
				}
			}
		}
	};
	f32x4 acc[2][2];
#pragma unroll
	for( int r = 0; r < 16; ++r ) {
		acc[r >> 3][( r >> 2 ) & 1][r & 3] = 0.f;
	}
	auto multiply = [&]( int set ) {
#pragma unroll
		for( int g = 0; g < Batch; ++g ) {
			auto product = [&]( auto partOf ) {
#pragma unroll
				for( int mi = 0; mi < 2; ++mi ) {
#pragma unroll
					for( int ni = 0; ni < 2; ++ni ) {
						acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32( partOf( a[set][g][mi] ), partOf( b[set][g][ni] ), acc[mi][ni], 0, 0, 0 );
					}
				}
			};
			product( []( const float4& v ) { return v.x; } );
			product( []( const float4& v ) { return v.y; } );
			product( []( const float4& v ) { return v.z; } );
			product( []( const float4& v ) { return v.w; } );
		}
	};
	auto step = [&]( int group, auto setOf ) {
		constexpr int set = decltype( setOf )::value;
		multiply( set );
		__builtin_amdgcn_sched_barrier( 0 );
		load( group + Sets * Batch, set );
		__builtin_amdgcn_sched_barrier( 0 );
	};
	if( firstGroup < lastGroup ) {
		load( firstGroup, 0 );
		load( firstGroup + Batch, 1 );
		load( firstGroup + 2 * Batch, 2 );
		load( firstGroup + 3 * Batch, 3 );
		for( int group = firstGroup; group < lastGroup; group += Sets * Batch ) {
			step( group, std::integral_constant<int, 0>() );
			if( group + Batch < lastGroup ) {
				step( group + Batch, std::integral_constant<int, 1>() );
			}
			if( group + 2 * Batch < lastGroup ) {
				step( group + 2 * Batch, std::integral_constant<int, 2>() );
			}
			if( group + 3 * Batch < lastGroup ) {
				step( group + 3 * Batch, std::integral_constant<int, 3>() );
			}
		}
	}

#pragma unroll
	for( int r = 0; r < 16; ++r ) {
		lds[wave][r][lane] = acc[r >> 3][( r >> 2 ) & 1][r & 3];
	}
	__syncthreads();
	// from here on a thread owns elements ( r = wave + i WAVES, lane ) of the tile
	float sum[PerThread];
#pragma unroll
	for( int i = 0; i < PerThread; ++i ) {
		sum[i] = 0.f;
#pragma unroll
		for( int w = 0; w < WAVES; ++w ) {
			sum[i] += lds[w][wave + i * WAVES][lane];
		}
	}
	const int slices = args.SplitK;
	if( slices > 1 ) {
		// Values cross between the L2 caches of the XCDs through agent-scope atomic accesses, which go past them; a wave's
		// stores are complete before the barrier in front of the count, and the reads come behind the barrier that follows it.
		unsigned* first = reinterpret_cast<unsigned*>( args.Partials ) + static_cast<long long>( tile ) * slices * 1024 + tid;
#pragma unroll
		for( int i = 0; i < PerThread; ++i ) {
			__hip_atomic_store( first + slice * 1024 + i * T, __float_as_uint( sum[i] ), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
		}
		__builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt( 0 ): this wave's stores have been acknowledged
		__syncthreads();
		if( tid == 0 ) {
			arrived = __hip_atomic_fetch_add( args.Counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
		}
		__syncthreads();
		if( arrived != static_cast<unsigned>( slices - 1 ) ) {
			return;
		}
		unsigned v[MaxSmallSlices][PerThread];
#pragma unroll
		for( int s = 0; s < MaxSmallSlices; ++s ) {
#pragma unroll
			for( int i = 0; i < PerThread; ++i ) {
				v[s][i] = s < slices ? __hip_atomic_load( first + s * 1024 + i * T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) : 0u;
			}
		}
#pragma unroll
		for( int i = 0; i < PerThread; ++i ) {
			sum[i] = 0.f;
#pragma unroll
			for( int s = 0; s < MaxSmallSlices; ++s ) {
				sum[i] += __uint_as_float( v[s][i] );
			}
		}
		if( tid == 0 ) {
			__hip_atomic_store( args.Counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
		}
	}
	// element ( r, lane ): block ( r / 8, r / 4 % 2 ), of it column lane % 16 of row 4 ( lane / 16 ) + r % 4
	float* C = args.C + batch * args.BatchStrideC;
	const CFusedActivation act = withParam( args.Act );
#pragma unroll
	for( int i = 0; i < PerThread; ++i ) {
		const int r = wave + i * WAVES;
		const int row = m0 + ( r >> 3 ) * 16 + quad * 4 + ( r & 3 ), n = n0 + ( ( r >> 2 ) & 1 ) * 16 + l16;
		if( row < M && n < N ) {
			const long long at = static_cast<long long>( row ) * args.Ldc + n;
			float v = sum[i] + ( args.Bias != nullptr ? args.Bias[n] : 0.f );
			if( args.Accumulate ) {
				v += C[at];
			}
			v = applyActivation( v, act );
			if( args.Residual != nullptr ) {
				v += args.Residual[batch * args.BatchStrideC + at];
			}
			C[at] = v;
		}
	}
}

// What this kernel is expected to take, in microseconds, with shares of so many groups. Fitted to some 1700 launches over
// 478 products and convolutions of up to 256 tiles, K from 128 to 8196, as all figures here are.
static double smallCost( int waves, int share, int slices, long long tiles )
{
	// ( the groups that all compute units have to do, to each: loads and matrix instructions share what there is )
	const double fill = static_cast<double>( tiles ) * slices * share / 256;
	const double meeting = slices > 1 ? 1.2 + 0.05 * slices : 0.0;
	return waves == 8 ? 4.6 + 0.25 * share + 0.83 * ( ( share + 1 ) / 2 ) + 0.45 * fill + meeting : 4.4 + 0.27 * share + 0.2 * fill + meeting;
}

// What the 64 x 64 tiles take: chains of steps below 32 steps, slices of them from there on.
static double tilesCost( int steps, long long tiles64, bool convolution )
{
	if( steps < 32 ) {
		return 3.3 + 0.256 * steps + ( convolution ? 0.6 : 0.0 );
	}
	return 6.7 + steps * ( 0.033 + 0.0008 * static_cast<double>( tiles64 ) ) + ( convolution ? 0.3 : 0.0 );
}

bool trySmallProduct( hipStream_t stream, const CMatMulArgs& given, bool convolution, int batch, bool vec, int* rc )
{
	if( !vec || batch > 65535 || given.K < 128 || ( convolution && given.Cin % 16 != 0 ) ) {
		return false;
	}
	const long long tilesM = ceilDiv( given.M, 32 ), tilesN = ceilDiv( given.N, 32 );
	const long long tiles = tilesM * tilesN * batch;
	if( tiles > 256 ) { // ( a second workgroup on a compute unit waits for the first )
		return false;
	}
	const int groups = ceilDiv( given.K, 16 );
	const int waves = groups >= 16 ? 8 : 4;
	// as many slices as are expected to pay, up to a workgroup for every compute unit
	int slices = 0;
	double cost = 0;
	for( int s = 1; s <= ( batch == 1 ? MaxSmallSlices : 1 ) && tiles * s <= 256; ++s ) {
		const int share = ceilDiv( groups, static_cast<long long>( s ) * waves );
		if( ceilDiv( groups, static_cast<long long>( share ) * waves ) != s ) {
			continue; // ( fewer slices have the same share )
		}
		const double c = smallCost( waves, share, s, tiles );
		if( slices == 0 || c < cost ) {
			slices = s;
			cost = c;
		}
	}
	// Of the 478 one was slower so ( 196 x 384 x 512 8.0 -> 8.2 us ); all together take 0.856 of the tiles' time, the faster kernel with
	// the best count of slices 0.850. us: 1 x 1000 x 1280 10.8 -> 7.7, 37 x 512 x 400 9.7 -> 6.9, 196 x 96 x 576 8.2 -> 7.8, 37 x 512 x 768
	// 8.4 -> 8.1, x 2048 11.7 -> 8.9, 49 x 160 x 960 9.4 -> 7.7, 100 x 512 x 960 9.8 -> 8.4, 1024 x 256 x 256 7.3 -> 6.7; convolutions of
	// 7 x 7 x 512 17.2 -> 12.3, 14 x 14 x 256 13.3 -> 11.7, 30 x 30 x 48 10.4 -> 6.8. Not 512 x 512 x 768 ( 10.3 and 10.5 ) or
	// 9 x 6 x 7 x 512 ( 26 and 35 ).
	if( cost > tilesCost( groups, static_cast<long long>( ceilDiv( given.M, 64 ) ) * ceilDiv( given.N, 64 ) * batch, convolution ) ) {
		return false;
	}
	CMatMulArgs args = given;
	args.StepsPerSplit = ceilDiv( groups, static_cast<long long>( slices ) * waves );
	if( slices > 1 && !sliceMeetingPlace( stream, static_cast<size_t>( tiles ) * slices * 1024, static_cast<size_t>( tiles ), &args.Partials, &args.Counters ) ) {
		return false;
	}
	args.SplitK = slices;
	args.TilesM = static_cast<int>( tilesM );
	args.TilesN = static_cast<int>( tilesN );
	args.TilesNMagic = divisionMagic( args.TilesN );
	args.WoMagic = divisionMagic( args.Wo );
	args.HoMagic = divisionMagic( args.Ho );
	const dim3 grid( static_cast<unsigned>( tilesM * tilesN ), batch, slices );
	auto launch = [&]( auto modeOf ) {
		constexpr int Mode = decltype( modeOf )::value;
		if( waves == 8 ) {
			hipLaunchKernelGGL( ( smallProductKernel<Mode, 8> ), grid, dim3( 512 ), 0, stream, args );
		} else {
			hipLaunchKernelGGL( ( smallProductKernel<Mode, 4> ), grid, dim3( 256 ), 0, stream, args );
		}
	};
	if( convolution ) {
		launch( std::integral_constant<int, AM_ConvTaps>() );
	} else {
		launch( std::integral_constant<int, AM_RowsK>() );
	}
	const hipError_t err = hipGetLastError();
	if( err != hipSuccess ) {
		setLastError( "small product: launch failed: %s", hipGetErrorString( err ) );
		*rc = NH_ERR_HIP;
	} else {
		*rc = NH_OK;
	}
	return true;
}

} // namespace nh
