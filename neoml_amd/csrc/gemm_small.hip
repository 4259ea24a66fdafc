// fp32 products and convolutions whose result is a few hundred 32 x 32 tiles or less: one picture, one short sequence.
#include "gemm.h"
#include <type_traits>

namespace nh {

typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

// C[M x N] = act( A * B^T + bias ) (+ C, + residual), A rows of K values or the im2col view of an image whose channel count is
// a multiple of 16, B rows of K values.
// What bounds such a product is latency: a chain of K steps, each with a barrier, on a few workgroups, and the instructions in
// front of its first load and behind its last sum ( a launch by itself takes 1.6 us, a few hundred instructions of a wavefront 1 us ).
// So a workgroup is one tile of 16 MB x 16 NB whose reduction is dealt to its WAVES wavefronts and, where the tiles leave compute
// units idle, to several workgroups. A wavefront fetches its share into registers, 16 k at a time with DEPTH such groups in flight,
// turns them round in its own part of LDS ( pass, below ) and multiplies MB x NB blocks by v_mfma_f32_16x16x4_f32, one group behind
// what it turns. It meets no barrier until its share is done. The shares are summed through LDS in the order of k, the
// slices through scratch memory by the one that arrives last, which fetches the others' tiles all at once.
// us, for operands loaded straight into the matrix instructions' layout and 32 x 32 tiles only, and now: 37 x 512 x 512 7.5 -> 3.9,
// x 2048 x 512 8.1 -> 5.2, x 512 x 2048 9.2 -> 7.1, 49 x 160 x 960 7.6 -> 5.0, 196 x 64 x 384 7.6 -> 3.1, 1 x 1000 x 1280 7.7 -> 4.9;
// 3 x 3 convolutions of 56 x 56 x 64 9.8 -> 6.7, 28 x 28 x 128 12.0 -> 7.1, 14 x 14 x 256 12.0 -> 7.9, 7 x 7 x 512 12.6 -> 10.2.
template<int AMODE, int WAVES, int MB, int NB, int DEPTH>
__device__ __forceinline__ void smallProductTile( const CMatMulArgs& args, float* lds, unsigned* arrived )
{
	constexpr bool IsTaps = ( AMODE == AM_ConvTaps );
	static_assert( IsTaps || AMODE == AM_RowsK, "operands that are K-major" );
	static_assert( MB * NB <= MB + NB && MB + NB <= 4, "the sums take the place of the operands in LDS" );
	constexpr int T = 64 * WAVES;
	constexpr int Regs = 4 * MB * NB; // accumulators of a lane
	constexpr int Elements = 64 * Regs;
	constexpr int Stage = ( MB + NB ) * 256; // floats of LDS that a wavefront stages its operands in
	constexpr int PerThread = ( Elements + T - 1 ) / T; // elements of the tile that a thread sums and writes

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane( tid >> 6 );
	const int l16 = lane & 15, quad = lane >> 4; // of the matrix instructions' operands
	const int loadRow = lane >> 2, loadQuad = lane & 3; // of the loads
	const int tile = xcdSwizzle( blockIdx.x, gridDim.x );
	int tileM, tileN;
	fastDivMod( tile, args.TilesN, args.TilesNMagic, tileM, tileN );
	const int m0 = tileM * 16 * MB, n0 = tileN * 16 * NB;
	const int batch = blockIdx.y, slice = blockIdx.z;
	const int M = args.M, N = args.N, K = args.K;
	const float* baseA = args.A + batch * args.BatchStrideA;
	const bool group = !IsTaps && args.Group != 0;
	const float* baseB = group ? args.GroupB[batch] : args.B + batch * args.BatchStrideB;
	const float* freeTerm = group ? args.GroupBias[batch] : args.Bias;

	// this wavefront's groups
	const int groups = ( K + 15 ) / 16;
	const int firstGroup = ( slice * WAVES + wave ) * args.StepsPerSplit;
	const int lastGroup = min( firstGroup + args.StepsPerSplit, groups );

	// the lane's rows of A and of B
	unsigned offA[MB], offB[NB];
	unsigned baseOfA[MB] = {}; // in floats, of tap ( 0, 0 ): unsigned arithmetic, it may lie in front of the image
	int imageH0[MB] = {}, imageW0[MB] = {};
	int tapCi = 0, tapKh = 0, tapKw = 0;
	auto tapOffsets = [&]() {
		const int dh = tapKh * args.DilH, dw = tapKw * args.DilW; // ( scalar )
		const unsigned tapFloats = ( static_cast<unsigned>( dh ) * static_cast<unsigned>( args.W ) + static_cast<unsigned>( dw ) )
			* static_cast<unsigned>( args.Cin );
#pragma unroll
		for( int i = 0; i < MB; ++i ) {
			const bool ok = tapKh < args.Fh && static_cast<unsigned>( imageH0[i] + dh ) < static_cast<unsigned>( args.H )
				&& static_cast<unsigned>( imageW0[i] + dw ) < static_cast<unsigned>( args.W );
			offA[i] = ok ? ( baseOfA[i] + tapFloats ) * 4u : OutOfRange;
		}
	};
#pragma unroll
	for( int i = 0; i < NB; ++i ) {
		const int n = n0 + i * 16 + loadRow;
		offB[i] = n < N ? ( static_cast<unsigned>( n ) * static_cast<unsigned>( args.Ldb ) + loadQuad * 4u ) * 4u : OutOfRange;
	}
#pragma unroll
	for( int i = 0; i < MB; ++i ) {
		const int m = m0 + i * 16 + loadRow;
		if constexpr( IsTaps ) {
			int t, wo, image, ho;
			fastDivMod( m, args.Wo, args.WoMagic, t, wo );
			fastDivMod( t, args.Ho, args.HoMagic, image, ho );
			imageH0[i] = m < M ? ho * args.StrideH - args.PadH : -0x40000000;
			imageW0[i] = wo * args.StrideW - args.PadW;
			baseOfA[i] = static_cast<unsigned>( image * args.H * args.W * args.Cin ) + ( static_cast<unsigned>( imageH0[i] )
				* static_cast<unsigned>( args.W ) + static_cast<unsigned>( imageW0[i] ) ) * static_cast<unsigned>( args.Cin ) + loadQuad * 4u;
		} else {
			offA[i] = m < M ? ( static_cast<unsigned>( m ) * static_cast<unsigned>( args.Lda ) + loadQuad * 4u ) * 4u : OutOfRange;
		}
	}
	if constexpr( IsTaps ) {
		const int tap = firstGroup * 16 / args.Cin;
		tapCi = firstGroup * 16 - tap * args.Cin;
		tapKh = tap / args.Fw;
		tapKw = tap - tapKh * args.Fw;
		tapOffsets();
	}

	// what the thread adds behind the sums, asked for in front of them: columns of its elements e = tid + i T ( see below )
	float free[PerThread] = {};
	const CFusedActivation act = withParam( args.Act );
	const float gateScale = args.Gate != nullptr ? *args.GateScale : 0.f;
	if( freeTerm != nullptr ) {
		const __amdgpu_buffer_rsrc_t bias = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( freeTerm ), 0, N * 4u, 0x00020000 );
#pragma unroll
		for( int i = 0; i < PerThread; ++i ) {
			free[i] = bufferLoad1( bias, ( n0 + ( ( wave + i * WAVES ) / 4 % NB ) * 16 + l16 ) * 4u );
		}
	}

	const __amdgpu_buffer_rsrc_t bufA = makeBuffer( baseA ), bufB = makeBuffer( baseB );
	float4 a[DEPTH][MB], b[DEPTH][NB];
	unsigned uniform = static_cast<unsigned>( firstGroup ) * 64u; // of the next group, in bytes
	const unsigned ragged = !IsTaps && ( K & 15 ) != 0 ? static_cast<unsigned>( groups - 1 ) * 64u : OutOfRange;
	auto load = [&]( int set ) {
		if( !IsTaps && uniform == ragged ) { // the last group of all: some quads lie behind K ( a multiple of 4 )
			const bool inK = static_cast<int>( uniform >> 2 ) + loadQuad * 4 < K;
#pragma unroll
			for( int i = 0; i < MB; ++i ) {
				offA[i] = inK ? offA[i] : OutOfRange;
			}
#pragma unroll
			for( int i = 0; i < NB; ++i ) {
				offB[i] = inK ? offB[i] : OutOfRange;
			}
		}
#pragma unroll
		for( int i = 0; i < MB; ++i ) {
			a[set][i] = bufferLoad4( bufA, offA[i], IsTaps ? static_cast<unsigned>( tapCi ) * 4u : uniform );
		}
#pragma unroll
		for( int i = 0; i < NB; ++i ) {
			b[set][i] = bufferLoad4( bufB, offB[i], uniform );
		}
		uniform += 64u;
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
	};
	// ( a block of its own has two accumulators, of the even and the odd quarters: a matrix instruction waits for the one whose sum
	// it continues )
	constexpr int Chains = MB * NB == 1 ? 2 : 1;
	f32x4 acc[Chains][MB][NB];
#pragma unroll
	for( int c = 0; c < Chains; ++c ) {
#pragma unroll
		for( int mi = 0; mi < MB; ++mi ) {
#pragma unroll
			for( int ni = 0; ni < NB; ++ni ) {
				acc[c][mi][ni] = f32x4{ 0.f, 0.f, 0.f, 0.f };
			}
		}
	}
	// A wavefront's operands pass through its own part of LDS ( instructions of one wavefront are executed there in their order: no
	// barrier, one buffer ): asked for with four lanes to a row and read back with rows across lanes, as the matrix instructions
	// want them. Where consecutive lanes ask for 16 bytes of different rows the memory unit delivers 16 bytes a clock, where four
	// lanes ask for 64 neighbouring bytes 64 ( 288 KB by one workgroup in 9.2 and 4.1 us ). The quads of a row are dealt so that
	// 16 lanes of a read meet all banks.
	float4* stage = reinterpret_cast<float4*>( lds + wave * Stage ); // blocks of 16 rows x 64 bytes
	float4* stageWrite = stage + loadRow * 4 + ( loadQuad ^ ( ( loadRow >> 2 ) & 3 ) );
	const float4* stageRead = stage + l16 * 4 + ( quad ^ ( ( l16 >> 2 ) & 3 ) );
	struct COperands { float4 X[MB], Y[NB]; } even, odd; // of this step and the next
	auto pass = [&]( int set, COperands& to ) {
#pragma unroll
		for( int i = 0; i < MB; ++i ) {
			stageWrite[i * 64] = a[set][i];
		}
#pragma unroll
		for( int i = 0; i < NB; ++i ) {
			stageWrite[( MB + i ) * 64] = b[set][i];
		}
		__builtin_amdgcn_wave_barrier();
		asm volatile( "" ::: "memory" );
#pragma unroll
		for( int i = 0; i < MB; ++i ) {
			to.X[i] = stageRead[i * 64];
		}
#pragma unroll
		for( int i = 0; i < NB; ++i ) {
			to.Y[i] = stageRead[( MB + i ) * 64];
		}
		__builtin_amdgcn_wave_barrier();
		asm volatile( "" ::: "memory" );
	};
	auto multiply = [&]( const COperands& of ) {
		auto product = [&]( int chain, auto partOf ) {
#pragma unroll
			for( int mi = 0; mi < MB; ++mi ) {
#pragma unroll
				for( int ni = 0; ni < NB; ++ni ) {
					acc[chain][mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32( partOf( of.X[mi] ), partOf( of.Y[ni] ), acc[chain][mi][ni], 0, 0, 0 );
				}
			}
		};
		product( 0, []( const float4& v ) { return v.x; } );
		product( Chains - 1, []( const float4& v ) { return v.y; } );
		product( 0, []( const float4& v ) { return v.z; } );
		product( Chains - 1, []( const float4& v ) { return v.w; } );
	};
	static_assert( DEPTH % 2 == 0, "steps alternate" );
	const int sets = lastGroup - firstGroup;
	if( sets > 0 ) {
#pragma unroll
		for( int u = 0; u < DEPTH; ++u ) {
			if( u < sets ) {
				load( u );
			}
		}
		pass( 0, even );
		// ( no condition inside: a wait counts the loads behind the awaited one, which all paths to it must have asked for )
		int left = sets;
		for( ; left >= 2 * DEPTH; left -= DEPTH ) {
#pragma unroll
			for( int u = 0; u < DEPTH; u += 2 ) {
				__builtin_amdgcn_sched_barrier( 0 );
				load( u );
				pass( u + 1, odd );
				__builtin_amdgcn_sched_barrier( 0 );
				multiply( even );
				__builtin_amdgcn_sched_barrier( 0 );
				load( u + 1 );
				pass( ( u + 2 ) % DEPTH, even );
				__builtin_amdgcn_sched_barrier( 0 );
				multiply( odd );
			}
		}
		if( left >= DEPTH ) {
			left -= DEPTH;
#pragma unroll
			for( int u = 0; u < DEPTH; u += 2 ) {
				if( u < left ) {
					load( u );
				}
				pass( u + 1, odd );
				multiply( even );
				if( u + 1 < left ) {
					load( u + 1 );
				}
				pass( ( u + 2 ) % DEPTH, even ); // ( of the last step, where nothing is left: values that are not used )
				multiply( odd );
			}
		}
#pragma unroll
		for( int u = 0; u + 1 < DEPTH; u += 2 ) {
			if( u < left ) {
				pass( u + 1, odd );
				multiply( even );
			}
			if( u + 1 < left ) {
				if( u + 2 < DEPTH ) {
					pass( u + 2, even );
				}
				multiply( odd );
			}
		}
	}

#pragma unroll
	for( int r = 0; r < Regs; ++r ) {
		float v = acc[0][r / ( 4 * NB )][( r / 4 ) % NB][r & 3];
		if constexpr( Chains == 2 ) {
			v += acc[1][0][0][r & 3];
		}
		lds[wave * Stage + r * 64 + lane] = v;
	}
	__syncthreads();
	// from here on a thread owns elements e = tid + i T of the tile: of register e / 64 of lane e % 64
	float sum[PerThread];
	const bool owns = Elements % T == 0 || tid < Elements;
#pragma unroll
	for( int i = 0; i < PerThread; ++i ) {
		sum[i] = 0.f;
		if( owns ) {
#pragma unroll
			for( int w = 0; w < WAVES; ++w ) {
				sum[i] += lds[w * Stage + tid + i * T];
			}
		}
	}
	const int slices = args.SplitK;
	if( slices > 1 ) {
		// Values cross between the L2 caches of the XCDs through agent-scope atomic accesses, which go past them; a wave's
		// stores are complete before the barrier in front of the count, and the reads come behind the barrier that follows it.
		unsigned* first = reinterpret_cast<unsigned*>( args.Partials ) + static_cast<long long>( tile ) * slices * Elements + tid;
		if( owns ) {
#pragma unroll
			for( int i = 0; i < PerThread; ++i ) {
				__hip_atomic_store( first + slice * Elements + i * T, __float_as_uint( sum[i] ), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
			}
		}
		__builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt( 0 ): this wave's stores have been acknowledged
		__syncthreads();
		if( tid == 0 ) {
			*arrived = __hip_atomic_fetch_add( args.Counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
		}
		__syncthreads();
		if( *arrived != static_cast<unsigned>( slices - 1 ) ) {
			return;
		}
		unsigned v[MaxSmallSlices][PerThread];
#pragma unroll
		for( int s = 0; s < MaxSmallSlices; ++s ) {
#pragma unroll
			for( int i = 0; i < PerThread; ++i ) {
				v[s][i] = s < slices && owns ? __hip_atomic_load( first + s * Elements + i * T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) : 0u;
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
	if( !owns ) {
		return;
	}
	// element ( r, lane ): block ( r / ( 4 NB ), r / 4 % NB ), of it column lane % 16 of row 4 ( lane / 16 ) + r % 4
	float* C = group ? args.GroupC[batch] : args.C + batch * args.BatchStrideC;
	const float* residual = args.Residual != nullptr ? args.Residual + batch * args.BatchStrideC : nullptr;
#pragma unroll
	for( int i = 0; i < PerThread; ++i ) {
		const int r = wave + i * WAVES;
		const int row = m0 + ( r / ( 4 * NB ) ) * 16 + quad * 4 + ( r & 3 ), n = n0 + ( ( r / 4 ) % NB ) * 16 + l16;
		if( row < M && n < N ) {
			const long long at = static_cast<long long>( row ) * args.Ldc + n;
			float v = sum[i] + free[i];
			if( args.Accumulate ) {
				v += C[at];
			}
			if( args.Gate != nullptr ) {
				const float gate = sigmoidOf( v * gateScale );
				args.Gate[at] = gate;
				v *= gate;
			} else if( residual != nullptr ) {
				const float r = residual[at];
				v = act.BehindResidual != 0 ? applyActivation( v + r, act ) : applyActivation( v, act ) + r;
			} else {
				v = applyActivation( v, act );
			}
			C[at] = v;
		}
	}
}

// The tile is chosen per launch ( CMatMulArgs::SmallTile ).
template<int AMODE, int WAVES>
__global__ __launch_bounds__( 64 * WAVES, 2 )
void smallProductKernel( const CMatMulArgs args )
{
	__shared__ float lds[WAVES * 1024];
	__shared__ unsigned arrived;
	if( args.SmallTile == 0 ) {
		smallProductTile<AMODE, WAVES, 1, 1, 6>( args, lds, &arrived );
	} else if( args.SmallTile == 1 ) {
		smallProductTile<AMODE, WAVES, 1, 2, 4>( args, lds, &arrived );
	} else {
		smallProductTile<AMODE, WAVES, 2, 2, 4>( args, lds, &arrived );
	}
}

constexpr int SmallTiles = 3;
constexpr int SmallTileM[SmallTiles] = { 16, 16, 32 }, SmallTileN[SmallTiles] = { 16, 32, 32 };
constexpr int MaxSmallWorkgroups = 384;

// What this kernel is expected to take, in microseconds. Fitted to 2177 launches over 302 products and convolutions ( 1 to 17000
// rows, 16 to 2500 columns, K from 28 to 4608 ), standard deviation 9 %.
static double smallCost( int tile, int waves, int share, int slices, long long tiles, bool convolution )
{
	struct CFit {
		double Launch, Group, GroupMore, GroupFill, More, Convolution, Eight, Meeting, MeetingSlice, MeetingTile;
	};
	static const CFit fits[SmallTiles] = { { 2.27, 0.196, 0.226, 0.131, 0.31, 0.22, 0.43, 1.09, 0.141, 1.32 },
		{ 2.57, 0.352, 0.352, 0.167, 0.43, 0.13, 0.15, 0.76, 0.167, 1.68 }, { 2.87, 0.556, 0.557, 0.283, 0.48, 0.28, 0.02, 1.03, 0.136, 0.96 } };
	const CFit& f = fits[tile];
	const double x = share * waves / 8.0; // groups to be done, two wavefronts to a matrix pipe
	const double fill = static_cast<double>( tiles ) * slices / 256;
	const double more = ceilDiv( tiles * slices, 256 ) - 1; // further workgroups on the fullest compute unit
	return f.Launch + f.Group * x + f.GroupMore * x * more + f.GroupFill * x * fill + f.More * more + ( convolution ? f.Convolution : 0.0 )
		+ ( waves == 8 ? f.Eight : 0.0 ) + ( slices > 1 ? f.Meeting + f.MeetingSlice * slices + f.MeetingTile * static_cast<double>( tiles ) / 256 : 0.0 );
}

// What the other kernels take for the same, standard deviation 4 % below K = 512 ( one workgroup to a tile ) and 7 % from there on.
static double tilesCost( int M, int N, int K, int batch, bool convolution )
{
	const double steps = ceilDiv( K, 16 );
	const double fill = static_cast<double>( batch ) * ( N > 32 ? static_cast<double>( ceilDiv( M, 64 ) ) * ceilDiv( N, 64 ) : ceilDiv( M, 128 ) ) / 256;
	if( K < 512 ) {
		return 2.57 + 0.291 * steps + 1.08 * fill + ( convolution ? 0.54 : 0.0 );
	}
	return 6.59 + 0.034 * steps + 0.166 * steps * fill + 3.42 * fill + ( convolution ? 0.43 : 0.0 );
}

// The tile and as many slices as are expected to pay; tile < 0: none. Of the 302 none was slower than without this kernel, all
// together take 0.556 of that time ( 0.549 with the best tile and count of slices for each ). Beyond 384 workgroups the larger tiles
// of the other kernels win: 9 x 12 x 14 x 256 3 x 3 22 and 26 us, 410 x 1121 x 832 14.7 and 16.9.
static void chooseSmall( const CMatMulArgs& args, bool convolution, int batch, int waves, int maxSlices, int& tile, int& slices )
{
	const int perWave = ceilDiv( ceilDiv( args.K, 16 ), waves );
	tile = -1;
	double cost = tilesCost( args.M, args.N, args.K, batch, convolution );
	for( int t = 0; t < SmallTiles; ++t ) {
		const long long tiles = static_cast<long long>( ceilDiv( args.M, SmallTileM[t] ) ) * ceilDiv( args.N, SmallTileN[t] ) * batch;
		// ( a slice's share in groups to each of its wavefronts; beyond perWave slices some would have none )
		for( int s = 1; s <= maxSlices && s <= perWave && tiles * s <= MaxSmallWorkgroups; ++s ) {
			const int share = ( perWave + s - 1 ) / s;
			if( ( perWave + share - 1 ) / share != s ) {
				continue; // ( fewer slices have the same share )
			}
			const double c = smallCost( t, waves, share, s, tiles, convolution );
			if( c < cost ) {
				tile = t;
				slices = s;
				cost = c;
			}
		}
	}
}

bool trySmallProduct( hipStream_t stream, const CMatMulArgs& given, bool convolution, int batch, bool vec, int* rc,
	const CSliceMeeting* fixedMeeting )
{
	if( !vec || batch > 65535 || given.K < 16 || ( convolution && given.Cin % 16 != 0 ) ) {
		return false;
	}
	const int groups = ceilDiv( given.K, 16 );
	const int waves = groups >= 16 ? 8 : 4;
	CMatMulArgs args = given;
	int tile = -1, slices = 1;
	chooseSmall( given, convolution, batch, waves, batch == 1 ? MaxSmallSlices : 1, tile, slices );
	if( tile >= 0 && slices > 1 ) {
		const size_t tiles = static_cast<size_t>( ceilDiv( given.M, SmallTileM[tile] ) ) * ceilDiv( given.N, SmallTileN[tile] );
		const size_t floats = tiles * slices * SmallTileM[tile] * SmallTileN[tile];
		bool place;
		if( fixedMeeting != nullptr ) {
			place = floats <= fixedMeeting->PartialFloats && tiles <= fixedMeeting->CounterCount;
			args.Partials = fixedMeeting->Partials;
			args.Counters = fixedMeeting->Counters;
			if( place ) {
				clearCounters( stream, args.Counters, tiles );
			}
		} else {
			place = sliceMeetingPlace( stream, floats, tiles, &args.Partials, &args.Counters );
		}
		if( !place ) { // ( under capture, at a pool's limit )
			chooseSmall( given, convolution, batch, waves, 1, tile, slices );
		}
	}
	if( tile < 0 ) {
		return false;
	}
	const long long tilesM = ceilDiv( given.M, SmallTileM[tile] ), tilesN = ceilDiv( given.N, SmallTileN[tile] );
	args.StepsPerSplit = ceilDiv( groups, static_cast<long long>( slices ) * waves );
	args.SplitK = slices;
	args.SmallTile = tile;
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
