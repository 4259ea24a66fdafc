// fp32 matrix products on the bf16 matrix instructions, each operand as the sum of three bf16 values.
//
// An fp32 value is exactly hi + mid + lo, where hi is the value rounded to bf16, mid what is left rounded to bf16, and lo
// the rest: 8 significant bits each, signs of their own. Of the nine products of two such sums six are multiplied, down to
// 2^-16 of the largest. The three that are left out ( mid lo, lo mid, lo lo ) come to 2^-24 of the product at most ( 1 + 2^-8 - 2^-17
// squared: 0.99 of that ) and to 2^-27 as a rule. What that and the instruction's own roundings leave is measured at the
// kernel: less than the fp32 instructions do.
#include "gemm.h"
#include <algorithm>
#include <type_traits>

namespace nh {

typedef __bf16 bf16x2 __attribute__( ( ext_vector_type( 2 ) ) );
typedef __bf16 bf16x8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef float f32x2 __attribute__( ( ext_vector_type( 2 ) ) );

// values ( x, y ) -> their three bf16 parts, packed
__device__ __forceinline__ void splitPair( float x, float y, unsigned& hi, unsigned& mid, unsigned& lo )
{
	const f32x2 v = { x, y };
	const bf16x2 h = __builtin_convertvector( v, bf16x2 );
	hi = __builtin_bit_cast( unsigned, h );
	const f32x2 r = { x - __uint_as_float( hi << 16 ), y - __uint_as_float( hi & 0xffff0000u ) };
	const bf16x2 m = __builtin_convertvector( r, bf16x2 );
	mid = __builtin_bit_cast( unsigned, m );
	const f32x2 q = { r.x - __uint_as_float( mid << 16 ), r.y - __uint_as_float( mid & 0xffff0000u ) };
	lo = __builtin_bit_cast( unsigned, __builtin_convertvector( q, bf16x2 ) );
}

constexpr int SplitStep = 16; // k per matrix instruction and per step

// The lowest bit of a value is 2^-23 of its power of two: below 2^-103 some of its parts lie under the smallest normal number, 2^-126,
// and are lost, whatever the value is multiplied by. So operands are split times 2^24, which every normal value's parts bear and
// which the sums are relieved of again as they are added up. ( Denormal values count as zero, here as in the fp32 instructions. )
constexpr float OperandScale = 0x1p24f, SumScale = 0x1p-48f;

// C[M x N] = act( A * B^T + bias ) (+ C, + residual), A and B rows of K values.
// What bounds it: the instructions of a SIMD's one or two wavefronts, which a barrier a step keeps together ( 8192 x 2048 x 512: the
// matrix pipe busy 52 % of the cycles, the vector instructions that split the operands another 36 % ), and the card's power ( back
// to back the clock is 1.9 GHz; on zeros 2.4, 69 us instead of 90 ). So the tiles are as large as the registers allow: a wavefront
// reads 2 x 2 blocks of fragments for 24 matrix instructions. Measured against the fp32 instructions, us: 8192 x 2048 x 512
// 130 -> 93 ( 185 TFLOP/s ), 8192 x 512 x 2048 125 -> 94, 8192 x 512 x 512 37.4 -> 27.2, 8192 x 1024 x 256 37.2 -> 28.0.
// Error against 64 bits ( 2-norm ), K from 132 to 2064: 1.2e-7 to 1.8e-7 where the fp32 instructions have 2.9e-7 to 8.5e-7.
// WGM x WGN wavefronts, each MI x NI blocks of 32 x 32; WPE: wavefronts per SIMD the registers must leave room for; RAGGED: K is not a multiple of the step.
template<int WGM, int WGN, int MI, int NI, int WPE, bool RAGGED>
__global__ __launch_bounds__( 64 * WGM * WGN, WPE )
void splitProductKernel( const CMatMulArgs args )
{
	constexpr int KS = SplitStep;
	constexpr int T = 64 * WGM * WGN;
	constexpr int BM = 32 * WGM * MI, BN = 32 * WGN * NI;
	// A tile's k step in LDS: three planes ( hi, mid, lo ) of [32-row block][k half][row][8 values], the order in which the
	// lanes of a matrix instruction take their 16 bytes. The rows of the second half are rotated by eight, so that the 32
	// lanes that store together, 8 rows of 4 quads, meet every bank once.
	constexpr int AUnits = BM * 4, BUnits = BN * 4; // quads of k: a quarter of a tile row's step
	constexpr int ASlots = ( AUnits + T - 1 ) / T, BSlots = ( BUnits + T - 1 ) / T;
	constexpr int Plane = ( BM + BN ) * 32; // bytes
	__shared__ __attribute__( ( aligned( 16 ) ) ) unsigned char lds[2][3 * Plane];

	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane( tid >> 6 );
	const int waveM = wave / WGN, waveN = wave % WGN;
	const int l32 = lane & 31, half = lane >> 5;

	const int batch = blockIdx.y;
	const int M = args.M, N = args.N, K = args.K;
	const float* baseA = args.A + batch * args.BatchStrideA;
	const float* baseB = args.B + batch * args.BatchStrideB;
	float* C = args.C + batch * args.BatchStrideC;
	const int totalSteps = ( K + KS - 1 ) / KS;

	const int tile = xcdSwizzle( blockIdx.x, gridDim.x );
	int tileM, tileN;
	fastDivMod( tile, args.TilesN, args.TilesNMagic, tileM, tileN );
	const int m0 = tileM * BM, n0 = tileN * BN;

	// ---- this thread's quads: quad tid % 4 of tile rows tid / 4 + i T / 4, four lanes cover the 64 bytes of a row's step
	unsigned offA[ASlots], offB[BSlots];
	const unsigned quad = tid & 3;
	const int tileRow = tid >> 2;
	constexpr int RowsPerSlot = T / 4;
#pragma unroll
	for( int i = 0; i < ASlots; ++i ) {
		const int row = tileRow + i * RowsPerSlot;
		const int m = m0 + row;
		offA[i] = ( AUnits % T == 0 || row < BM ) && m < M
			? ( static_cast<unsigned>( m ) * static_cast<unsigned>( args.Lda ) + quad * 4u ) * 4u : OutOfRange;
	}
#pragma unroll
	for( int i = 0; i < BSlots; ++i ) {
		const int row = tileRow + i * RowsPerSlot;
		const int n = n0 + row;
		offB[i] = ( BUnits % T == 0 || row < BN ) && n < N
			? ( static_cast<unsigned>( n ) * static_cast<unsigned>( args.Ldb ) + quad * 4u ) * 4u : OutOfRange;
	}

	// A matrix instruction rounds its accumulator twice, a step twelve times, and not to nearest: the errors lean to one side,
	// which a sum over many results ( the gradient by a filter, over 200704 pixels ) adds up: 7e-6 of it where the single
	// results are off by 2e-7. So the reduction is cut into an even number of chunks of up to eight steps. Each begins from
	// zero and is added to the totals, and every other one is computed with A negated and subtracted. Most roundings are then of short
	// sums ( the error of 576 k falls from 3.6e-7 to 1.5e-7, of 2304 k from 7.2e-7 to 1.8e-7; the fp32 instructions: 4.2e-7 and
	// 8.3e-7 ) and lean to both sides alike, for 2 - 4 % of the time. A chunk is a number of pairs of steps, so that it begins on
	// LDS buffer 0; the numbers differ by one at most, and the longer chunks are the last ones, where a step may be missing.
	// ( Mean error in 264, 288, 640, 1152 k: 3e-10, 1e-9 ( two of eighteen steps more with one sign ), 1e-10, 1e-10; with an odd number
	// of chunks 4e-9, 5e-9, 4e-9, 3e-9. )
	constexpr int LongestChunk = 8;
	const int chunks = ( totalSteps + 2 * LongestChunk - 1 ) / ( 2 * LongestChunk ) * 2;
	const int pairsOfSteps = ( totalSteps + 1 ) >> 1;
	const int chunkPairs = pairsOfSteps / chunks, firstLonger = chunks - ( pairsOfSteps - chunkPairs * chunks );
	auto chunkSteps = [&]( int index ) -> int { return ( chunkPairs + ( index < firstLonger ? 0 : 1 ) ) * 2; };

	float4 regA[ASlots], regB[BSlots];
	// Requests the quads of a step. A step behind the last is asked of a descriptor of size zero ( zeros, no memory
	// access ): every step runs the same code.
	auto load = [&]( int step ) {
		const unsigned range = step < totalSteps ? BufferBytes : 0u;
		const __amdgpu_buffer_rsrc_t bufA = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( baseA ), 0, range, 0x00020000 );
		const __amdgpu_buffer_rsrc_t bufB = __builtin_amdgcn_make_buffer_rsrc( const_cast<float*>( baseB ), 0, range, 0x00020000 );
		const unsigned uni = static_cast<unsigned>( step ) * ( KS * 4u );
		// the last step of a K that is not a multiple of the step ( it is one of 4 )
		const bool masked = RAGGED && step * KS + static_cast<int>( quad ) * 4 >= K;
#pragma unroll
		for( int i = 0; i < ASlots; ++i ) {
			regA[i] = bufferLoad4( bufA, masked ? OutOfRange : offA[i], uni );
		}
#pragma unroll
		for( int i = 0; i < BSlots; ++i ) {
			regB[i] = bufferLoad4( bufB, masked ? OutOfRange : offB[i], uni );
		}
	};
	const int quadAt = static_cast<int>( quad >> 1 ) * 512 + static_cast<int>( quad & 1 ) * 8;
	auto unitAt = [&]( int row ) -> int {
		return ( row >> 5 ) * 1024 + quadAt + ( ( row + static_cast<int>( quad >> 1 ) * 8 ) & 31 ) * 16;
	};
	auto storeUnit = [&]( int buf, int at, const float4& v ) {
		uint2 hi, mid, lo;
		splitPair( v.x, v.y, hi.x, mid.x, lo.x );
		splitPair( v.z, v.w, hi.y, mid.y, lo.y );
		*reinterpret_cast<uint2*>( &lds[buf][at] ) = hi;
		*reinterpret_cast<uint2*>( &lds[buf][at + Plane] ) = mid;
		*reinterpret_cast<uint2*>( &lds[buf][at + 2 * Plane] ) = lo;
	};
	auto store = [&]( int buf, float scaleOfA ) {
#pragma unroll
		for( int i = 0; i < ASlots; ++i ) {
			if( AUnits % T == 0 || tileRow + i * RowsPerSlot < BM ) {
				const float4 v = regA[i];
				storeUnit( buf, unitAt( tileRow + i * RowsPerSlot ),
					make_float4( v.x * scaleOfA, v.y * scaleOfA, v.z * scaleOfA, v.w * scaleOfA ) );
			}
		}
#pragma unroll
		for( int i = 0; i < BSlots; ++i ) {
			if( BUnits % T == 0 || tileRow + i * RowsPerSlot < BN ) {
				const float4 v = regB[i];
				storeUnit( buf, BM * 32 + unitAt( tileRow + i * RowsPerSlot ),
					make_float4( v.x * OperandScale, v.y * OperandScale, v.z * OperandScale, v.w * OperandScale ) );
			}
		}
	};

	f32x16 acc[MI][NI];
	auto clear = [&]() {
#pragma unroll
		for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
			for( int ni = 0; ni < NI; ++ni ) {
#pragma unroll
				for( int r = 0; r < 16; ++r ) {
					acc[mi][ni][r] = 0.f;
				}
			}
		}
	};
	clear();

	const int fragLane = half * 512 + ( ( l32 + half * 8 ) & 31 ) * 16;
	const int fragA = waveM * MI * 1024 + fragLane, fragB = BM * 32 + waveN * NI * 1024 + fragLane;
	struct CFrag {
		bf16x8 A[3][MI], B[3][NI];
	};
	CFrag frag[2];
	auto readFrag = [&]( int buf, CFrag& f ) {
#pragma unroll
		for( int p = 2; p >= 0; --p ) {
#pragma unroll
			for( int mi = 0; mi < MI; ++mi ) {
				f.A[p][mi] = *reinterpret_cast<const bf16x8*>( &lds[buf][p * Plane + fragA + mi * 1024] );
			}
#pragma unroll
			for( int ni = 0; ni < NI; ++ni ) {
				f.B[p][ni] = *reinterpret_cast<const bf16x8*>( &lds[buf][p * Plane + fragB + ni * 1024] );
			}
		}
	};
	auto products = [&]( const CFrag& f ) {
		auto product = [&]( int pa, int pb ) {
#pragma unroll
			for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
				for( int ni = 0; ni < NI; ++ni ) {
					acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16( f.A[pa][mi], f.B[pb][ni], acc[mi][ni], 0, 0, 0 );
				}
			}
		};
		product( 2, 0 );
		product( 0, 2 );
		product( 1, 1 );
		product( 1, 0 );
		product( 0, 1 );
		product( 0, 0 );
	};

	// Step s multiplies the fragments that step s - 1 read. Under its matrix instructions the fragments of step s + 1 are read
	// from LDS buffer ( s + 1 ) % 2 and the values of step s + 2 are split and stored to buffer s % 2, whose last readers
	// were in step s - 1; one barrier ends the step. Reads, stores and vector instructions are dealt evenly over the step.
	load( 0 );
	store( 0, OperandScale );
	load( 1 );
	store( 1, OperandScale );
	load( 2 );
	__syncthreads();
	readFrag( 0, frag[0] );
	__syncthreads();
	constexpr int Products = 6 * MI * NI; // matrix instructions of a step
	constexpr int SplitVector = ( ASlots + BSlots ) * 26; // vector instructions of a step's quads, about
	auto step = [&]( int s, float scaleOfStored, auto curOf ) {
		constexpr int cur = decltype( curOf )::value, nxt = cur ^ 1;
		__builtin_amdgcn_sched_barrier( 0 );
		readFrag( nxt, frag[nxt] );
		store( cur, scaleOfStored );
		products( frag[cur] );
#pragma unroll
		for( int i = 0; i < Products; ++i ) {
			__builtin_amdgcn_sched_group_barrier( 0x008, 1, 0 ); // a matrix instruction
			__builtin_amdgcn_sched_group_barrier( 0x100, ( 3 * ( MI + NI ) + Products - 1 ) / Products, 0 ); // LDS reads
			__builtin_amdgcn_sched_group_barrier( 0x002, ( SplitVector + Products - 1 ) / Products, 0 ); // vector instructions under it
			__builtin_amdgcn_sched_group_barrier( 0x200, ( 3 * ( ASlots + BSlots ) + Products - 1 ) / Products, 0 ); // LDS stores
		}
		__builtin_amdgcn_sched_barrier( 0 );
		load( s + 3 );
		__syncthreads();
	};
	f32x16 total[MI][NI] = {};
	int s = 0, end = 0;
	for( int chunk = 0; chunk < chunks; ++chunk ) {
		end = min( end + chunkSteps( chunk ), totalSteps );
		const float scale = chunk & 1 ? -OperandScale : OperandScale;
		for( ; s + 1 < end; s += 2 ) {
			const float scaleOfStored = s + 2 < end ? scale : -scale; // ( the last pair stores the next chunk's first )
			step( s, scaleOfStored, std::integral_constant<int, 0>() );
			step( s + 1, scaleOfStored, std::integral_constant<int, 1>() );
		}
		if( s < end ) {
			step( s, scale, std::integral_constant<int, 0>() );
			++s;
		}
		const float sign = chunk & 1 ? -SumScale : SumScale;
#pragma unroll
		for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
			for( int ni = 0; ni < NI; ++ni ) {
#pragma unroll
				for( int r = 0; r < 16; ++r ) {
					total[mi][ni][r] = __builtin_fmaf( acc[mi][ni][r], sign, total[mi][ni][r] );
				}
			}
		}
		clear();
	}
#pragma unroll
	for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
		for( int ni = 0; ni < NI; ++ni ) {
			acc[mi][ni] = total[mi][ni];
		}
	}

	// An operand that is infinite or NaN, or that times its factor rounds to infinity, has no finite parts: infinity - infinity makes
	// all it meets NaN. And a sum beyond 2^80 overflows times the factors. Either shows in the totals: such a wavefront multiplies its
	// blocks again with the fp32 instructions, operands straight from memory.
	float notFinite = 0.f;
#pragma unroll
	for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
		for( int ni = 0; ni < NI; ++ni ) {
#pragma unroll
			for( int r = 0; r < 16; ++r ) {
				notFinite = __builtin_fmaf( acc[mi][ni][r], 0.f, notFinite );
			}
		}
	}
	const bool again = notFinite != notFinite;
	if( __builtin_amdgcn_ballot_w64( again ) != 0 ) {
		clear();
		const __amdgpu_buffer_rsrc_t bufA = makeBuffer( baseA ), bufB = makeBuffer( baseB );
		#pragma unroll 1
		for( int k0 = 0; k0 < K; k0 += 8 ) {
			const bool inK = k0 + half * 4 < K;
			float4 a[MI], b[NI];
#pragma unroll
			for( int mi = 0; mi < MI; ++mi ) {
				const int m = m0 + ( waveM * MI + mi ) * 32 + l32;
				a[mi] = bufferLoad4( bufA, inK && m < M
					? ( static_cast<unsigned>( m ) * static_cast<unsigned>( args.Lda ) + static_cast<unsigned>( k0 + half * 4 ) ) * 4u : OutOfRange );
			}
#pragma unroll
			for( int ni = 0; ni < NI; ++ni ) {
				const int n = n0 + ( waveN * NI + ni ) * 32 + l32;
				b[ni] = bufferLoad4( bufB, inK && n < N
					? ( static_cast<unsigned>( n ) * static_cast<unsigned>( args.Ldb ) + static_cast<unsigned>( k0 + half * 4 ) ) * 4u : OutOfRange );
			}
#pragma unroll
			for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
				for( int ni = 0; ni < NI; ++ni ) {
					acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32( a[mi].x, b[ni].x, acc[mi][ni], 0, 0, 0 );
					acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32( a[mi].y, b[ni].y, acc[mi][ni], 0, 0, 0 );
					acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32( a[mi].z, b[ni].z, acc[mi][ni], 0, 0, 0 );
					acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32( a[mi].w, b[ni].w, acc[mi][ni], 0, 0, 0 );
				}
			}
		}
	}

	// C through a buffer descriptor that ends with the matrix: rows beyond it are dropped by the range check. A row adds a
	// multiple of the row pitch to the lane's offset, in a scalar register where the tile lies inside the matrix.
	const __amdgpu_buffer_rsrc_t bufC = __builtin_amdgcn_make_buffer_rsrc( C, 0, args.CBytes, 0x00020000 );
	const float* residual = args.Residual != nullptr ? args.Residual + batch * args.BatchStrideC : nullptr;
	const float actParam = withParam( args.Act ).Param; // ( the threshold may live in device memory )
	const float reluTop = actParam > 0.f ? actParam : __builtin_inff();
	const bool behind = args.Act.BehindResidual != 0;
	constexpr int GateType = -1; // ( beside the activations: the gates of a GELU )
	const float gateScale = args.Gate != nullptr ? *args.GateScale : 0.f;
	const __amdgpu_buffer_rsrc_t bufGate = __builtin_amdgcn_make_buffer_rsrc( args.Gate != nullptr ? args.Gate : C, 0, args.CBytes, 0x00020000 );
	const unsigned pitchBytes = static_cast<unsigned>( args.Ldc ) * 4u;
	auto write = [&]( auto typeOf, auto extraOf, auto insideOf ) {
		constexpr int Type = decltype( typeOf )::value;
		constexpr bool Extra = decltype( extraOf )::value; // accumulate and / or residual
		constexpr bool Inside = decltype( insideOf )::value;
#pragma unroll
		for( int ni = 0; ni < NI; ++ni ) {
			const int n = n0 + ( waveN * NI + ni ) * 32 + l32;
			const float bias = ( args.Bias != nullptr && n < N ) ? args.Bias[n] : 0.f;
			const int rowBase = m0 + waveM * MI * 32 + half * 4;
			const unsigned laneOffset = n < N ? static_cast<unsigned>( rowBase ) * pitchBytes + static_cast<unsigned>( n ) * 4u : OutOfRange;
#pragma unroll
			for( int mi = 0; mi < MI; ++mi ) {
#pragma unroll
				for( int r = 0; r < 16; ++r ) {
					const int row = mi * 32 + ( r >> 2 ) * 8 + ( r & 3 );
					// ( an offset that was out of range stays so: what is added is below 2^31 )
					const unsigned groupOffset = laneOffset + static_cast<unsigned>( row & ~3 ) * pitchBytes;
					const unsigned rowBytes = static_cast<unsigned>( row & 3 ) * pitchBytes;
					float v = acc[mi][ni][r] + bias;
					if constexpr( Type == GateType ) {
						const float gate = sigmoidOf( v * gateScale );
						v *= gate;
						if constexpr( Inside ) {
							__builtin_amdgcn_raw_buffer_store_b32( __float_as_uint( gate ), bufGate, groupOffset, rowBytes, 0 );
						} else {
							__builtin_amdgcn_raw_buffer_store_b32( __float_as_uint( gate ), bufGate, groupOffset + rowBytes, 0, 0 );
						}
					} else if constexpr( Extra ) {
						const bool ok = n < N && rowBase + row < M;
						const long long at = static_cast<long long>( rowBase + row ) * args.Ldc + n;
						if( args.Accumulate && ok ) {
							v += C[at];
						}
						const float r = residual != nullptr && ok ? residual[at] : 0.f;
						v = behind ? applyActivationOf<Type>( v + r, reluTop ) : applyActivationOf<Type>( v, reluTop ) + r;
					} else {
						v = applyActivationOf<Type>( v, reluTop );
					}
					if constexpr( Inside ) {
						__builtin_amdgcn_raw_buffer_store_b32( __float_as_uint( v ), bufC, groupOffset, rowBytes, 0 );
					} else {
						__builtin_amdgcn_raw_buffer_store_b32( __float_as_uint( v ), bufC, groupOffset + rowBytes, 0, 0 );
					}
				}
			}
		}
	};
	auto writeAs = [&]( auto typeOf ) {
		if( args.Accumulate || residual != nullptr ) {
			write( typeOf, std::true_type(), std::false_type() );
		} else if( m0 + BM <= M ) {
			write( typeOf, std::false_type(), std::true_type() );
		} else {
			write( typeOf, std::false_type(), std::false_type() );
		}
	};
	if( args.Gate != nullptr ) {
		if( m0 + BM <= M ) {
			write( std::integral_constant<int, GateType>(), std::false_type(), std::true_type() );
		} else {
			write( std::integral_constant<int, GateType>(), std::false_type(), std::false_type() );
		}
	} else if( args.Act.Type == NH_ACT_RELU ) {
		writeAs( std::integral_constant<int, NH_ACT_RELU>() );
	} else if( args.Act.Type == NH_ACT_HSWISH ) {
		writeAs( std::integral_constant<int, NH_ACT_HSWISH>() );
	} else {
		writeAs( std::integral_constant<int, NH_ACT_NONE>() );
	}
}

// What a launch is expected to take, in microseconds, and its tiles.
struct CSplitPlan {
	double Cost;
	int TilesM, TilesN;
};

// A launch takes what the compute unit with the most tiles takes, or, where the matrix instructions of all units together draw more
// power than there is, what the card's rate leaves: the longer of the two. Fitted to 443 products of 0.3 to 40 GFLOP, K from 128 to
// 4092, one or up to 64 of them, repeated until the clock had settled ( fitted over measured, 5th and 95th percentile: 0.90 and 1.10
// for the largest tiles, 0.86 and 1.12, 0.82 and 1.15 ). A step of a tile takes
//   256 x 128 tiles: 0.84 us, one workgroup to a unit; the card 213 TFLOP/s;
//   128 x 128 tiles by eight wavefronts of 64 x 32: 0.525 us, 188 TFLOP/s ( by four of 64 x 64: 33.2 us instead of 29.5 for
//   8192 x 512 x 512, 116 instead of 113 for 8192 x 512 x 2048 );
//   128 x 64 tiles: 0.46 us, 0.39 us for each of several side by side ( three to a unit ), 166 TFLOP/s;
// and a tile costs what its prologue and epilogue take on top.
enum TSplitShape { SS_256x128, SS_128x128, SS_128x64, SS_Count };

static CSplitPlan splitPlan( int shape, const CMatMulArgs& a, int batch )
{
	const int bm = shape == SS_256x128 ? 256 : 128;
	const int bn = shape == SS_128x64 ? 64 : 128;
	const double steps = ceilDiv( a.K, SplitStep );
	CSplitPlan plan = {};
	plan.TilesM = ceilDiv( a.M, bm );
	plan.TilesN = ceilDiv( a.N, bn );
	const long long tiles = static_cast<long long>( plan.TilesM ) * plan.TilesN * batch;
	const double deepest = static_cast<double>( ( tiles + 255 ) / 256 );
	const double megaflops = static_cast<double>( tiles ) * steps * ( 2e-6 * SplitStep * bm * bn );
	switch( shape ) {
		case SS_256x128: plan.Cost = std::max( deepest * steps * 0.84, megaflops / 213 ) + deepest * 8; break;
		case SS_128x128: plan.Cost = std::max( deepest * steps * 0.525, megaflops / 188 ) + deepest * 3.5 + 1.9; break;
		default: plan.Cost = std::max( steps * std::max( 0.46, 0.39 * deepest ), megaflops / 166 ) + deepest * 0.5 + 3.5; break;
	}
	return plan;
}

template<int WGM, int WGN, int MI, int NI, int WPE>
static void launchSplit( hipStream_t stream, const CMatMulArgs& args, const dim3& grid )
{
	const dim3 threads( 64 * WGM * WGN );
	if( args.K % SplitStep != 0 ) {
		hipLaunchKernelGGL( ( splitProductKernel<WGM, WGN, MI, NI, WPE, true> ), grid, threads, 0, stream, args );
	} else {
		hipLaunchKernelGGL( ( splitProductKernel<WGM, WGN, MI, NI, WPE, false> ), grid, threads, 0, stream, args );
	}
}

// Products, a pointwise convolution's among them. 3x3 convolutions would be done in 0.66 to 0.9 of the time ( us: 65536 pixels,
// 1152 -> 256, 282 -> 190; 64 x 28 x 28 x 128, 116 -> 83; 64 x 56 x 56 x 64, 119 -> 104 ), but the ReLU behind one decides by a
// value's sign what a training step's gradients are made of. Another rounding, also a smaller one, moves a value next to zero to the
// other side, and with each such value of the 1.3e7 of 64 x 56 x 56 x 64 a residual block's gradients move by 3e-4, where the sums
// differ by 4e-7. A convolution cannot know what it is computed for, and its size says nothing about it: they stay on the fp32
// instructions at every size.
bool trySplitProduct( hipStream_t stream, const CMatMulArgs& given, int batch, bool vec, int* rc )
{
	CMatMulArgs args = given;
	if( !vec || batch > 65535 || args.M < 128 || args.N < 48 || args.K < 128 ) {
		return false;
	}
	const long long cBytes = ( static_cast<long long>( args.M - 1 ) * args.Ldc + args.N ) * 4;
	if( args.Ldc < args.N || cBytes >= 0x7fffff00LL || args.Ldc > 0x1000000 ) {
		return false;
	}
	int shape = 0;
	CSplitPlan plan = {};
	for( int s = 0; s < SS_Count; ++s ) {
		const CSplitPlan p = splitPlan( s, args, batch );
		if( s == 0 || p.Cost < plan.Cost ) {
			plan = p;
			shape = s;
		}
	}
	// The fp32 instructions at their best on such sizes: 130 TFLOP/s, three steps' time for the ends of a tile, 3 us. What is taken is
	// what is expected to be faster. Of the 443 products one was slower so, 15265 x 128 x 1048 with 43.9 us instead of 42.7; all together
	// take 0.881 of the time of the fp32 instructions, the faster kernel every time would take 0.864. ( 1792 x 1024 x 512 20.2 -> 17.3,
	// 4096 x 512 x 256 12.2 -> 10.9, 4096 x 768 x 128 12.0 -> 9.8; not 1024 x 512 x 512, 10.5 and 16.3, or 6272 x 160 x 960, 23 and 32. )
	const double steps = ceilDiv( args.K, SplitStep );
	const double flops = 2.0 * args.M * args.N * args.K * batch;
	if( plan.Cost > flops / 130e6 * ( steps + 3 ) / steps + 3 ) {
		return false;
	}
	args.TilesM = plan.TilesM;
	args.TilesN = plan.TilesN;
	args.TilesNMagic = divisionMagic( args.TilesN );
	args.CBytes = static_cast<unsigned>( cBytes );
	const dim3 grid( static_cast<unsigned>( plan.TilesM ) * plan.TilesN, batch );
	switch( shape ) {
		case SS_256x128: launchSplit<4, 2, 2, 2, 2>( stream, args, grid ); break;
		case SS_128x128: launchSplit<2, 4, 2, 1, 2>( stream, args, grid ); break;
		default: launchSplit<2, 2, 2, 1, 3>( stream, args, grid ); break;
	}
	const hipError_t err = hipGetLastError();
	if( err != hipSuccess ) {
		setLastError( "split product: launch failed: %s", hipGetErrorString( err ) );
		*rc = NH_ERR_HIP;
	} else {
		*rc = NH_OK;
	}
	return true;
}

} // namespace nh
